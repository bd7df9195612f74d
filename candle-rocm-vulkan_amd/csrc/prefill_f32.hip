// Flash attention of f32 queries at prefill shapes (flash_attn with f32 q and out over f32, f16, bf16
// or E4M3 K / V; the reference's fa{2,3}_d*_f32_* kernels, candle-core/kernels/flash_attn_impl.h:330-443)
// on the bf16 matrix units with f32 precision.
//
// Every f32 operand is the exact sum of three bf16 parts x = x0 + x1 + x2 (8 significant bits each,
// rounded to nearest), so a product is x0 y0 + (x0 y1 + x1 y0) + (x0 y2 + x1 y1 + x2 y0) plus terms
// below 2^-25 of it. The six products are exact on v_mfma_f32_32x32x16_bf16 and summed in f32: fewer
// roundings than the f32 MFMA's one per four terms, at 16 / 6 of its rate. In K Q^T the five small ones
// of a dot product come first in the one accumulator, so that the sums at full magnitude are one
// rounding per 16 dims; in V^T P^T they have an accumulator per tile, added once. Probabilities are
// f32 and split the same way.
// 2048 causal tokens, 2 sequences, 12 / 4 heads, D = 128, call: 341 us in fa32_kernel's column mode (f32
// MFMA, K / V read by every wavefront) -> 182 us; relative error against float64 4.9e-7 -> 3.1e-7. Equal
// ranges (1024 x 4096, 64 heads) run at 216 TFLOP/s, 1.3 PFLOP/s of bf16 products, what a large bf16
// matrix product reaches on this card (matrix units 73 % busy at 1.7 GHz).
//
//  * prefill_f32_stage_kernel writes each 32-key tile of a (sequence, kv head) plane as the image the
//    attention keeps in LDS: three parts of K (rows of keys) and of V^T (rows of head dims, keys of
//    each 16 in the order of the S^T registers), 16-byte chunks XOR-swizzled as the reads want them.
//  * prefill_f32_kernel: 8 (or 4) wavefronts of 32 columns ((query, head of the group) pairs). Images stream
//    through LDS rings of three K and V^T stages (144 KB at D = 128) by asynchronous copies, one
//    barrier per tile. With 96 products of 32 cycles a tile and wavefront against some 400 vector
//    instructions and 48 operand reads, the matrix units are the bound.
//  * Non-finite queries and keys: the whole value goes into part 2, whose only product is with the
//    other side's part 0, so an infinity meets neither another infinity's remainder nor a zero part.
//    Non-finite V elements are zeros in the image, since a matrix product would carry them, times a
//    zero probability, into all 32 columns of a tile; the rows that see their keys get them after the
//    loop (x3_bad_values; nothing is done there where the wavefront's tiles hold none).
//  * Inputs below about 2^-110 lose their last parts (bf16 has f32's exponent range).
#include <algorithm>
#include <utility>

#include "cqkv_device.h"
#include "cqkv_host.h"
#include "flash_plain.h"
#include "prefill_split.h"

namespace cqkv {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kX3Bk = 32;  // keys of a tile

// Bytes of a part of K or V^T of a tile, and of the whole image.
template <int D>
constexpr int x3_part() { return 2 * kX3Bk * D; }
template <int D>
constexpr int x3_image() { return 6 * x3_part<D>(); }

// 16-byte chunk swizzles: K rows of 2 D bytes, V^T rows of 64 bytes (conflict-free over the 16 rows of
// one ds_read_b128 pass).
template <int D>
__device__ inline int x3_swz_k(int r) {
    if constexpr (D == 128) return ((r & 7) << 1) | ((r >> 3) & 1);
    else return (r >> 1) & 7;
}
__device__ inline int x3_swz_v(int d) { return (d >> 2) & 3; }

struct X3Args {
    FaArgs f;
    uint8_t *img;     // (batch, kv head, tiles) images
    uint32_t *bad;    // (batch, kv head, tiles): the tile's keys with a non-finite value (null: not kept)
    int32_t tiles;    // images per plane
    int32_t q_blocks;
    int32_t piece_tiles, max_pieces;
    int32_t nc;       // columns of a workgroup
    uint32_t group_m;
};

// Split dense calls: (column block << 4 | piece) of each workgroup of a plane by falling size, in the
// launch's arguments (n 0: the order of the ids). The blocks of a causal prompt fall in size, their
// last pieces do not: handed out by block, the CUs ended after 43 steps of 28 on average.
constexpr int kX3Jobs = 1024;
struct X3Order {
    int32_t n;
    uint16_t job[kX3Jobs];
};

// Two values to bf16 pairs of their three parts (word p: part p of a in the low half, of b high).
__device__ inline uint32_t x3_pack(float a, float b) {
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}
// finite values whose rounding stays finite (probabilities)
__device__ inline void x3_split_finite(float a, float b, uint32_t *w) {
    w[0] = x3_pack(a, b);
    const float ra = a - __uint_as_float(w[0] << 16), rb = b - __uint_as_float(w[0] & 0xffff0000u);
    w[1] = x3_pack(ra, rb);
    w[2] = x3_pack(ra - __uint_as_float(w[1] << 16), rb - __uint_as_float(w[1] & 0xffff0000u));
}
// part 0 of any value: 0 for non-finite ones, truncated where rounding would overflow
__device__ inline float x3_head(float x) {
    const float r = (float)(__bf16)x;
    if (__builtin_fabsf(r) < __builtin_inff()) return r;
    return __builtin_fabsf(x) < __builtin_inff() ? __uint_as_float(__float_as_uint(x) & 0xffff0000u) : 0.0f;
}
__device__ inline void x3_split(float a, float b, uint32_t *w) {
    const float ha = x3_head(a), hb = x3_head(b);
    const bool fa = __builtin_fabsf(a) < __builtin_inff(), fb = __builtin_fabsf(b) < __builtin_inff();
    w[0] = x3_pack(ha, hb);
    const float ra = fa ? a - ha : 0.0f, rb = fb ? b - hb : 0.0f;
    w[1] = x3_pack(ra, rb);
    const float ta = ra - __uint_as_float(w[1] << 16), tb = rb - __uint_as_float(w[1] & 0xffff0000u);
    w[2] = x3_pack(fa ? ta : a, fb ? tb : b);
}

// Four consecutive elements of a K / V row as f32.
template <int KV>
__device__ inline f32x4 x3_load4(const uint16_t *base, int64_t at) {
    if constexpr (KV == CQKV_F32) {
        return *(const f32x4 *)((const float *)base + at);
    } else if constexpr (KV == kKvE4M3) {
        const uint32_t w = *(const uint32_t *)((const uint8_t *)base + at);
        const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
        return f32x4{lo.x, lo.y, hi.x, hi.y};
    } else {
        const u32x2 w = *(const u32x2 *)(base + at);
        if constexpr (KV == CQKV_F16)
            return f32x4{f16_bits_to_f32(w.x & 0xffffu), f16_bits_to_f32(w.x >> 16),
                         f16_bits_to_f32(w.y & 0xffffu), f16_bits_to_f32(w.y >> 16)};
        else
            return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                         __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
    }
}

// One workgroup per tile of a plane: K and V rows of 32 keys (zeros past the sequence's keys and past
// head_dim) to the tile's image. Bound by the bytes: 4 (2) read and 6 written per element.
template <int KV, int D>
__global__ __launch_bounds__(256) void prefill_f32_stage_kernel(X3Args x) {
    const FaArgs &a = x.f;
    constexpr int CPR = D / 8, IT = kX3Bk * CPR / 256, ROW = D + 4;
    __shared__ __attribute__((aligned(16))) float vt[kX3Bk * ROW];
    __shared__ uint32_t rows_bad[4 * IT];
    const int tile = blockIdx.x, plane = blockIdx.y;
    const int b = plane / a.kv_heads, hk = plane % a.kv_heads;
    const FaSeq sq = fa_sequence(a, b);
    if (tile * kX3Bk >= sq.lk) return;  // (no workgroup reads the tile)
    uint8_t *img = x.img + ((int64_t)plane * x.tiles + tile) * x3_image<D>();
    const int64_t k0 = sq.k0 + (int64_t)hk * a.k_sh, v0 = sq.v0 + (int64_t)hk * a.v_sh;
    f32x4 kr[IT][2], vr[IT][2];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int id = threadIdx.x + 256 * i, row = id / CPR, c = id % CPR;
        const int key = tile * kX3Bk + row;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            kr[i][h] = vr[i][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (key < sq.lk && 8 * c < a.head_dim) {
                kr[i][h] = x3_load4<KV>(a.k, k0 + (int64_t)key * a.k_st + 8 * c + 4 * h);
                vr[i][h] = x3_load4<KV>(a.v, v0 + (int64_t)key * a.v_st + 8 * c + 4 * h);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int id = threadIdx.x + 256 * i, row = id / CPR, c = id % CPR;
        if (x.bad) {
            bool any = false;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = vr[i][e >> 2][e & 3];
                const bool fin = __builtin_fabsf(v) < __builtin_inff();
                any |= !fin;
                vr[i][e >> 2][e & 3] = fin ? v : 0.0f;
            }
            // this wavefront's 64 / CPR rows
            const uint64_t lanes = __ballot(any);
            uint32_t w = 0;
#pragma unroll
            for (int r = 0; r < 64 / CPR; ++r)
                w |= (lanes >> (r * CPR) & ((1u << CPR) - 1) ? 1u : 0u) << r;
            if ((threadIdx.x & 63) == 0) rows_bad[4 * i + (threadIdx.x >> 6)] = w << (row & 31);
        }
        *(f32x4 *)&vt[row * ROW + 8 * c] = vr[i][0];
        *(f32x4 *)&vt[row * ROW + 8 * c + 4] = vr[i][1];
        uint32_t w[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x3_split(kr[i][e >> 1][2 * (e & 1)], kr[i][e >> 1][2 * (e & 1) + 1], w[e]);
#pragma unroll
        for (int p = 0; p < 3; ++p)
            *(u32x4 *)(img + p * x3_part<D>() + row * 2 * D + ((c ^ x3_swz_k<D>(row)) << 4)) =
                u32x4{w[0][p], w[1][p], w[2][p], w[3][p]};
    }
    __syncthreads();
    if (x.bad && threadIdx.x == 0) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4 * IT; ++i) w |= rows_bad[i];
        x.bad[(int64_t)plane * x.tiles + tile] = w;
    }
    // V^T: chunk j of row d holds keys 8j .. 8j+7 in the order of the S^T registers
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int id = threadIdx.x + 256 * i, d = id % D, j = id / D;
        uint32_t w[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int p0 = 8 * j + 2 * e;  // position -> key: bits 2 and 3 swapped
            const int key = (p0 & ~12) | ((p0 & 4) << 1) | ((p0 & 8) >> 1);
            x3_split(vt[key * ROW + d], vt[(key + 1) * ROW + d], w[e]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
            *(u32x4 *)(img + (3 + p) * x3_part<D>() + d * 64 + ((j ^ x3_swz_v(d)) << 4)) =
                u32x4{w[0][p], w[1][p], w[2][p], w[3][p]};
    }
}

__device__ inline f32x16 x3_mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// the products beside the largest: parts (i, j) of the two sides with 0 < i + j <= 2
__device__ inline f32x16 x3_small(const u32x4 *a, const u32x4 *b, f32x16 c) {
    c = x3_mfma(a[0], b[2], c);
    c = x3_mfma(a[2], b[0], c);
    c = x3_mfma(a[1], b[1], c);
    c = x3_mfma(a[0], b[1], c);
    return x3_mfma(a[1], b[0], c);
}

__device__ inline float x3_max_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float x3_sum_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int D>
struct X3State {
    u32x4 q[D / 16][3];  // Q^T operands: parts of this lane's column, 16-dim steps
    f32x16 acc[D / 32];  // O^T
    float m_run, l_run, negm;
    int qlo, qhi, pos;   // visible keys and key position of the lane's query
    float scale_log2, cap2, slope2;
    // this lane's LDS read offsets: row and swizzled chunk h of K and V^T; chunk 2 i + h is at
    // row + (chunk ^ (i << 5)). Made opaque every step: left alone, the compiler keeps a register per
    // chunk and stage and spills.
    uint32_t krow, kchunk, vrow, vchunk;
};

// Scores of a key tile (exp2 units, masked): S^T = K Q^T, the small products first, so that the sums
// at full magnitude are one rounding per 16 dims.
template <int D>
__device__ __attribute__((always_inline)) inline void x3_scores(const X3State<D> &st, float *s,
                                                                const uint8_t *kt, int k0, bool masked,
                                                                bool terms, int lane) {
    constexpr int PART = x3_part<D>();
    const int h = lane >> 5;
    f32x16 sum = {};
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
        u32x4 k[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
            k[p] = *(const u32x4 *)(kt + (st.krow + (st.kchunk ^ (ks << 5))) + p * PART);
        sum = x3_small(k, st.q[ks], sum);
    }
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
        sum = x3_mfma(*(const u32x4 *)(kt + (st.krow + (st.kchunk ^ (ks << 5)))), st.q[ks][0], sum);
    // lane (qr, h), register j: key k0 + 8 (j / 4) + 4 h + j % 4 of this lane's column
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = sum[j] * st.scale_log2;
    if (terms) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
            s[j] = fa_logit2(s[j], st.cap2, st.slope2, st.pos - (k0 + 8 * (j >> 2) + 4 * h + (j & 3)));
    }
    if (masked) {
        int u = k0 + 4 * h - st.qlo;
        asm volatile("" : "+v"(u));
        const uint32_t w = (uint32_t)(st.qhi - st.qlo);
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if ((uint32_t)(u + 8 * (j >> 2) + (j & 3)) >= w) s[j] = -__builtin_inff();
    }
}

// The softmax of a tile's scores: the P^T operands (16-key steps, parts).
template <int D>
__device__ __attribute__((always_inline)) inline void x3_softmax(X3State<D> &st, u32x4 (*pp)[3], const float *s) {
    float mx = s[0], mx1 = s[1];
#pragma unroll
    for (int j = 2; j < 16; j += 2) {
        mx = fmaxf(mx, s[j]);
        mx1 = fmaxf(mx1, s[j + 1]);
    }
    mx = x3_max_halves(fmaxf(mx, mx1));
    // the maximum moves at a row's first visible key and when exceeded by 2^8
    const bool need = mx > (st.m_run == -__builtin_inff() ? -__builtin_inff() : st.m_run + 8.0f);
    if (__any(need)) {
        const float m_new = need ? mx : st.m_run;
        const float alpha = need ? __builtin_amdgcn_exp2f(st.m_run - m_new) : 1.0f;
#pragma unroll
        for (int md = 0; md < D / 32; ++md) st.acc[md] *= alpha;
        st.l_run *= alpha;
        st.m_run = m_new;
        st.negm = m_new == -__builtin_inff() ? 0.0f : -m_new;
    }
    float l0 = 0.0f, l1 = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
        uint32_t w[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float p0 = __builtin_amdgcn_exp2f(s[8 * kk + 2 * e] + st.negm);
            const float p1 = __builtin_amdgcn_exp2f(s[8 * kk + 2 * e + 1] + st.negm);
            l0 += p0;
            l1 += p1;
            x3_split_finite(p0, p1, w[e]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) pp[kk][p] = u32x4{w[0][p], w[1][p], w[2][p], w[3][p]};
    }
    st.l_run += l0 + l1;
}

// O^T += V^T P^T of a key tile; the small products of a block are summed apart and added once.
template <int D>
__device__ __attribute__((always_inline)) inline void x3_pv(X3State<D> &st, const u32x4 (*pp)[3],
                                                            const uint8_t *vt) {
    constexpr int PART = x3_part<D>();
#pragma unroll
    for (int md = 0; md < D / 32; ++md) {
        f32x16 rest = {};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            u32x4 v[3];
#pragma unroll
            for (int p = 0; p < 3; ++p)
                v[p] = *(const u32x4 *)(vt + (st.vrow + (st.vchunk ^ (kk << 5))) + (p * PART + 32 * 64 * md));
            rest = x3_small(v, pp[kk], rest);
            st.acc[md] = x3_mfma(v[0], pp[kk][0], st.acc[md]);
        }
        st.acc[md] += rest;
    }
}

// Non-finite V elements of the wavefront's n tiles from tile kt of the plane on: each is added to the rows that see its key, times the key's weight there, which only has to be zero
// (0 times infinity is NaN, as in plain attention) or not.
template <int D>
__device__ __attribute__((always_inline)) inline void x3_bad_values(X3State<D> &st, const X3Args &x, int plane,
                                                                    int kt, int n, int lane) {
    const FaArgs &a = x.f;
    const int h = lane >> 5, b = plane / a.kv_heads;
    const int64_t tile0 = (int64_t)plane * x.tiles + kt;
    const uint32_t *flags = x.bad + tile0;
    const uint8_t *images = x.img + tile0 * x3_image<D>();
    for (int i0 = 0; i0 < n; i0 += 64) {
        const uint32_t m = i0 + lane < n ? flags[i0 + lane] : 0u;
        for (uint64_t left = __ballot(m != 0); left; left &= left - 1) {
            const int i = __builtin_ctzll(left);
            for (uint32_t keys = __builtin_amdgcn_readlane(m, i); keys; keys &= keys - 1) {
                const int r = __builtin_ctz(keys), key = (kt + i0 + i) * kX3Bk + r;
                const uint8_t *kimg = images + (int64_t)(i0 + i) * x3_image<D>() + r * 2 * D;
                float dot = 0.0f;
#pragma unroll
                for (int ks = 0; ks < D / 16; ++ks) {
                    f32x4 ka[2] = {}, qa[2] = {};
#pragma unroll
                    for (int p = 2; p >= 0; --p) {
                        asm volatile("" : "+v"(st.q[ks][p]));  // (or their sums are kept over the loop)
                        const u32x4 w = *(const u32x4 *)(kimg + p * x3_part<D>() + (((2 * ks + h) ^ x3_swz_k<D>(r)) << 4));
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const int sh = e & 1;
                            ka[e >> 2][e & 3] += __uint_as_float(sh ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16);
                            qa[e >> 2][e & 3] += __uint_as_float(sh ? st.q[ks][p][e >> 1] & 0xffff0000u
                                                                    : st.q[ks][p][e >> 1] << 16);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) dot += ka[e >> 2][e & 3] * qa[e >> 2][e & 3];
                    __builtin_amdgcn_sched_barrier(0);  // (few registers are left beside q and acc)
                }
                const float s = fa_logit2(x3_sum_halves(dot) * st.scale_log2, st.cap2, st.slope2, st.pos - key);
                if (key >= st.qlo && key < st.qhi) {
                    const float p = __builtin_amdgcn_exp2f(s + st.negm);
                    const int64_t at = fa_sequence(a, b).v0 + (plane - b * a.kv_heads) * a.v_sh +
                                       (int64_t)key * a.v_st + 4 * h;
#pragma unroll
                    for (int md = 0; md < D / 32; ++md)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int d = 32 * md + 8 * j;
                            if (d >= a.head_dim) continue;
                            const f32x4 v = a.kv_dtype == CQKV_F32    ? x3_load4<CQKV_F32>(a.v, at + d)
                                            : a.kv_dtype == CQKV_F16  ? x3_load4<CQKV_F16>(a.v, at + d)
                                            : a.kv_dtype == CQKV_BF16 ? x3_load4<CQKV_BF16>(a.v, at + d)
                                                                      : x3_load4<kKvE4M3>(a.v, at + d);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (!(__builtin_fabsf(v[e]) < __builtin_inff())) st.acc[md][4 * j + e] += p * v[e];
                            __builtin_amdgcn_sched_barrier(0);
                        }
                }
            }
        }
    }
}

#define X3_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 15) | (((n) >> 4) << 14)) | 0x0f70)

// W wavefronts of 32 columns: 8 (two per SIMD), or 4 where blocks of 256 columns would leave CUs idle
// (a step of a lone wavefront per SIMD takes 2.1 us, of two 3.4 to 5 us).
template <int D, bool SPLIT, int W>
__global__ __launch_bounds__(W * 64, W / 4) void prefill_f32_kernel(X3Args x, X3Order order) {
    const FaArgs &a = x.f;
    // half an image (K or V^T of a tile) and the 1 KB copies of it per wavefront (at D = 64, W = 8 the last
    // four wavefronts' second copies repeat the first four's, so that all have the same count in flight)
    constexpr int IMG = x3_image<D>(), HALF = IMG / 2, UNITS = HALF / 1024, CP = (UNITS + W - 1) / W, NC = 32 * W;
    // distinct arrays, so the compiler can tell a copy into one stage from the reads of another
    __shared__ __attribute__((aligned(1024))) uint8_t ks0[HALF];
    __shared__ __attribute__((aligned(1024))) uint8_t ks1[HALF];
    __shared__ __attribute__((aligned(1024))) uint8_t ks2[HALF];
    __shared__ __attribute__((aligned(1024))) uint8_t vs0[HALF];
    __shared__ __attribute__((aligned(1024))) uint8_t vs1[HALF];
    __shared__ __attribute__((aligned(1024))) uint8_t vs2[HALF];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qr = lane & 31, h = lane >> 5;

    // planes first (a plane's workgroups on one XCD), blocks with the most key tiles first; split key
    // ranges by the order table, or the whole pieces of every block, then the last ones
    const int nplanes = a.kv_heads * a.batch;
    const int rest = (int)blockIdx.x / nplanes, plane = (int)blockIdx.x % nplanes;
    const int whole = SPLIT ? x.max_pieces - 1 : 0;
    const bool listed = SPLIT && order.n > 0, last_slot = !SPLIT || rest >= x.q_blocks * whole;
    const int qb = listed ? order.job[rest] >> 4
                          : x.q_blocks - 1 - (last_slot ? rest - x.q_blocks * whole : rest / whole);
    const int b = plane / a.kv_heads, hk = plane % a.kv_heads;
    const FaSeq sq = fa_sequence(a, b);
    const int lq = sq.lq, lk = sq.lk;
    const int64_t ncols = (int64_t)lq * a.group, c0 = (int64_t)qb * NC;
    if (c0 >= ncols) return;
    const int q0 = (int)(c0 / a.group), cr0 = (int)(c0 - (int64_t)q0 * a.group);
    const int ncol = (int)min((int64_t)NC, ncols - c0);
    int kt;
    int ntiles = pf_block_tiles(q0, q0 + pf_div_group(cr0 + ncol - 1, a.group, x.group_m), lq, lk, a.wl,
                                a.wr, kX3Bk, kt);
    const int pieces = SPLIT ? pf_pieces(ntiles, x.piece_tiles, x.max_pieces) : 1;
    const int piece = listed ? order.job[rest] & 15 : last_slot ? pieces - 1 : rest % whole;
    if (piece >= pieces - (listed || last_slot ? 0 : 1)) return;
    if (SPLIT && pieces > 1) {
        kt += piece * x.piece_tiles;
        ntiles = piece == pieces - 1 ? ntiles - piece * x.piece_tiles : x.piece_tiles;
    }
    // this wavefront's tiles and the keys that all its columns see
    const bool wave_live = 32 * wave < ncol;
    int lo, hi, lo_last, hi_first;
    pf_key_range(q0 + pf_div_group(cr0 + min(32 * wave, ncol - 1), a.group, x.group_m), lq, lk, a.wl, a.wr,
                 lo, hi_first);
    pf_key_range(q0 + pf_div_group(cr0 + min(32 * wave + 32, ncol) - 1, a.group, x.group_m), lq, lk, a.wl,
                 a.wr, lo_last, hi);
    const int wtiles = wave_live ? min(max((hi + kX3Bk - 1) / kX3Bk - kt, 0), ntiles) : 0;

    // whether its tiles hold non-finite values (x3_bad_values), read beside the queries
    uint32_t bad = 0;
    if (x.bad)
        for (int i = lane; i < wtiles; i += 64) bad |= x.bad[(int64_t)plane * x.tiles + kt + i];

    X3State<D> st;
    const int c = cr0 + min(32 * wave + qr, ncol - 1);
    const int qc = pf_div_group(c, a.group, x.group_m), head = hk * a.group + (c - qc * a.group);
    const bool ok = 32 * wave + qr < ncol;
    {
        const float *row = (const float *)a.q + sq.q0 + (int64_t)head * a.q_sh + (int64_t)(q0 + qc) * a.q_st;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
            f32x4 v[2] = {};
            if (ok && 16 * ks + 8 * h < a.head_dim) {
                v[0] = *(const f32x4 *)(row + 16 * ks + 8 * h);
                v[1] = *(const f32x4 *)(row + 16 * ks + 8 * h + 4);
            }
            uint32_t w[4][3];
#pragma unroll
            for (int e = 0; e < 4; ++e) x3_split(v[e >> 1][2 * (e & 1)], v[e >> 1][2 * (e & 1) + 1], w[e]);
#pragma unroll
            for (int p = 0; p < 3; ++p) st.q[ks][p] = u32x4{w[0][p], w[1][p], w[2][p], w[3][p]};
        }
    }
    if (ok) pf_key_range(q0 + qc, lq, lk, a.wl, a.wr, st.qlo, st.qhi);
    else st.qlo = st.qhi = 0;
    st.pos = q0 + qc + lk - lq;
    st.scale_log2 = a.scale_log2 * (a.q_mul_dev ? a.q_mul_dev[0] : 1.0f);
    st.cap2 = a.softcap2;
    st.slope2 = a.alibi ? a.alibi[(int64_t)b * a.alibi_bs + head] * kLog2e : 0.0f;
    const bool terms = a.softcap2 > 0.0f || a.alibi;
    st.krow = qr * 2 * D;
    st.kchunk = (h ^ x3_swz_k<D>(qr)) << 4;
    st.vrow = qr * 64;
    st.vchunk = (h ^ x3_swz_v(qr)) << 4;
    st.m_run = -__builtin_inff();
    st.l_run = st.negm = 0.0f;
#pragma unroll
    for (int md = 0; md < D / 32; ++md) st.acc[md] = f32x16{};

    const uint8_t *images = x.img + ((int64_t)plane * x.tiles + kt) * IMG;
    X3_WAIT_VMCNT(0);  // the loads above must not be counted by the copy waits below
    const bool any_bad = __any(bad != 0);
    // Step t works on the scores of tile t and on P V of tile t - 1. The two wavefronts of a SIMD (w and
    // w + 4) order them so that one's softmax runs beside the other's products: the first takes P V
    // of tile t - 1, scores and softmax of tile t, the second the softmax and P V of tile t - 1, then the
    // scores of tile t (64 heads of 1024 x 4096: 844 us with both in the same order, 821 us so).
    // K(t) and V(t) live in stage t % 3 of their rings. Step t copies K(t + 2) and V(t + 1) behind its
    // barrier, into the stages of K(t - 1) and V(t - 2), which step t - 1 read last; they are waited
    // for two barriers later. Tiles outside the range are copied with a zero-size resource (no memory
    // access, zeros into a stage nobody reads), which keeps the count of copies in flight.
    const auto issue = [&](uint8_t *stage, int t, int half) {
        const bool valid = t >= 0 && t < ntiles;
        const uint64_t p = (uint64_t)(images + (int64_t)(valid ? t : 0) * IMG + half * HALF);
        const uint32_t plo = __builtin_amdgcn_readfirstlane((uint32_t)p);
        const uint32_t phi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
        const rsrc_t r = make_rsrc((const void *)(((uint64_t)phi << 32) | plo),
                                   __builtin_amdgcn_readfirstlane(valid ? (uint32_t)HALF : 0u));
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            const int unit = wave + W * i < UNITS ? wave + W * i : wave + W * i - UNITS;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t *)(stage + unit * 1024), 16,
                                                     unit * 1024 + 16 * lane, 0, 0, 0);
        }
    };
    issue(ks0, 0, 0);
    issue(vs2, -1, 1);
    issue(ks1, 1, 0);
    issue(vs0, 0, 1);
    u32x4 pp[2][3];
    float s[16];
#define X3_SCORES(K)                                                                         \
    if (t < wtiles) {                                                                        \
        const int k0 = (kt + t) * kX3Bk;                                                     \
        x3_scores<D>(st, s, K, k0, !(k0 >= lo_last && k0 + kX3Bk <= hi_first), terms, lane); \
    }
#define X3_STEP(K, KNEXT, VPREV, VNEXT, ORDER)                                               \
    {                                                                                        \
        if (t > ntiles) break;                                                               \
        X3_WAIT_VMCNT(2 * CP); /* all but the copies of the step before */                   \
        __builtin_amdgcn_s_barrier();                                                        \
        issue(KNEXT, t + 2, 0);                                                              \
        issue(VNEXT, t + 1, 1);                                                              \
        asm volatile("" : "+v"(st.krow), "+v"(st.kchunk), "+v"(st.vrow), "+v"(st.vchunk));   \
        const bool prev = t > 0 && t <= wtiles;                                              \
        ORDER(K, VPREV)                                                                      \
        __builtin_amdgcn_sched_barrier(0);                                                   \
        ++t;                                                                                 \
    }
#define X3_EARLY(K, VPREV)                                                                   \
    if (prev) x3_pv<D>(st, pp, VPREV);                                                       \
    X3_SCORES(K)                                                                             \
    if (t < wtiles) x3_softmax<D>(st, pp, s);
#define X3_LATE(K, VPREV)                                                                    \
    if (prev) {                                                                              \
        x3_softmax<D>(st, pp, s);                                                            \
        x3_pv<D>(st, pp, VPREV);                                                             \
    }                                                                                        \
    X3_SCORES(K)
#define X3_LOOP(ORDER)                                                                       \
    for (int t = 0;;) {                                                                      \
        X3_STEP(ks0, ks2, vs2, vs1, ORDER)                                                   \
        X3_STEP(ks1, ks0, vs0, vs2, ORDER)                                                   \
        X3_STEP(ks2, ks1, vs1, vs0, ORDER)                                                   \
    }
    if (W == 4 || wave < 4) X3_LOOP(X3_EARLY)
    else X3_LOOP(X3_LATE)
#undef X3_LOOP
#undef X3_LATE
#undef X3_EARLY
#undef X3_SCORES
#undef X3_STEP
    X3_WAIT_VMCNT(0);

    if (any_bad) {
        // Values that were zeros in the images. Arguments and plane are read anew: kept over the loop they
        // cost it registers (2 x 2048 causal tokens, 12 / 4 heads, D = 128: 162 us, 158.4 without this).
        typedef const __attribute__((address_space(4))) X3Args kernarg_t;
        uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
        uint32_t id = blockIdx.x;
        asm volatile("" : "+s"(at), "+s"(id));
        const X3Args &y = *(const X3Args *)(kernarg_t *)at;
        x3_bad_values<D>(st, y, (int)(id % (uint32_t)(y.f.kv_heads * y.f.batch)), kt, wtiles, lane);
    }
    // lane (qr, h): head dims 32 md + 8 (j / 4) + 4 h + j % 4 of column qr
    if (!ok) return;
    const float l = x3_sum_halves(st.l_run);
    const bool part = SPLIT && pieces > 1;
    const float inv = l == 0.0f ? 0.0f : (part ? 1.0f : a.o_mul * (a.o_mul_dev ? a.o_mul_dev[0] : 1.0f)) / l;
    float *orow;
    if (part) {
        const int64_t row = ((int64_t)piece * nplanes + plane) * ((int64_t)a.q_len * a.group) + c0 + 32 * wave + qr;
        if (h == 0) a.part_lse[row] = pf_piece_lse(st.m_run, l);
        orow = a.part_o + row * D;
    } else {
        orow = (float *)a.out + sq.o0 + (int64_t)(q0 + qc) * a.o_st + (int64_t)head * a.o_sh;
    }
#pragma unroll
    for (int md = 0; md < D / 32; ++md)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d = 32 * md + 8 * j + 4 * h;
            if (!part && d >= a.head_dim) continue;
            *(f32x4 *)(orow + d) = f32x4{st.acc[md][4 * j] * inv, st.acc[md][4 * j + 1] * inv,
                                         st.acc[md][4 * j + 2] * inv, st.acc[md][4 * j + 3] * inv};
        }
}

// Merges the pieces of split column blocks (prefill_combine_kernel's form, f32 rows).
template <int D>
__global__ __launch_bounds__(256) void prefill_f32_combine_kernel(X3Args x) {
    const FaArgs &a = x.f;
    constexpr int L = D / 4;  // lanes per column
    const int li = threadIdx.x % L, plane = blockIdx.y;
    const int b = plane / a.kv_heads, hk = plane % a.kv_heads;
    const int64_t col = (int64_t)blockIdx.x * (256 / L) + threadIdx.x / L;
    const FaSeq sq = fa_sequence(a, b);
    const int64_t ncols = (int64_t)sq.lq * a.group;
    if (col >= ncols) return;
    const int64_t c0 = col / x.nc * x.nc;
    int begin;
    const int n = pf_block_tiles((int)(c0 / a.group), (int)((min(c0 + x.nc, ncols) - 1) / a.group), sq.lq,
                                 sq.lk, a.wl, a.wr, kX3Bk, begin);
    const int pieces = pf_pieces(n, x.piece_tiles, x.max_pieces);
    if (pieces <= 1) return;
    const int64_t rows = (int64_t)a.q_len * a.group, step = rows * a.kv_heads * a.batch;
    float r[4];
    pf_merge_pieces<D>(a.part_o, a.part_lse, plane * rows + col, step, pieces, li,
                       a.o_mul * (a.o_mul_dev ? a.o_mul_dev[0] : 1.0f), r);
    if (4 * li >= a.head_dim) return;
    const int qi = (int)(col / a.group), g = (int)(col % a.group);
    float *o = (float *)a.out + sq.o0 + (int64_t)qi * a.o_st + (int64_t)(hk * a.group + g) * a.o_sh + 4 * li;
    *(f32x4 *)o = f32x4{r[0], r[1], r[2], r[3]};
}

// ---- host ----
// The plan of a call and its workgroups: the smaller estimate of 8 and 4 wavefronts.
struct X3Plan {
    PfPlan split;
    int waves;
};
static X3Plan x3_plan(int dk, const FaArgs &a, int wl, int wr) {
    const PfShape g8 = dk == 64 ? PfShape{256, kX3Bk, 64, 1.8, 0.7, 2, 128, true}
                                : PfShape{256, kX3Bk, 128, 3.4, 1.5, 2, 128, true};
    const PfShape g4 = dk == 64 ? PfShape{128, kX3Bk, 64, 1.1, 0.4, 2, 128, true}
                                : PfShape{128, kX3Bk, 128, 2.1, 0.8, 2, 128, true};
    const PfPlan p8 = pf_plan(g8, a.batch, a.q_len, a.kv_len, a.q_heads, a.kv_heads, wl, wr);
    const PfPlan p4 = pf_plan(g4, a.batch, a.q_len, a.kv_len, a.q_heads, a.kv_heads, wl, wr);
    if (p4.us > 0.0 && p4.us < p8.us) return {p4, 4};
    return {p8, 8};
}
static int x3_dk(int head_dim) { return head_dim <= 64 ? 64 : 128; }
static size_t x3_images(const FaArgs &a) {
    const size_t image = x3_dk(a.head_dim) == 64 ? x3_image<64>() : x3_image<128>();
    return (size_t)a.batch * a.kv_heads * ((a.kv_len + kX3Bk - 1) / kX3Bk) * image;
}

// Bytes of the image region and of the flags behind it; the partials follow.
static size_t x3_images_end(const FaArgs &a) { return (x3_images(a) + 255) / 256 * 256; }
static size_t x3_flags(const FaArgs &a) {
    return ((size_t)a.batch * a.kv_heads * ((a.kv_len + kX3Bk - 1) / kX3Bk) * 4 + 255) / 256 * 256;
}

// Key tiles (of bk keys) of a group of n columns, the mean over the groups of a plane (up to 32 of
// them, evenly spaced) and the largest.
static double x3_mean_tiles(const FaArgs &a, int wl, int wr, int n, int bk, int *most) {
    const int64_t cols = (int64_t)a.q_len * a.group, groups = (cols + n - 1) / n, k = std::min<int64_t>(groups, 32);
    double sum = 0.0;
    *most = 0;
    for (int64_t i = 0; i < k; ++i) {
        const int64_t c0 = (k > 1 ? i * (groups - 1) / (k - 1) : 0) * n;
        int begin;
        const int t = pf_block_tiles((int)(c0 / a.group), (int)((std::min(c0 + n, cols) - 1) / a.group), a.q_len,
                                     a.kv_len, wl, wr, bk, begin);
        *most = std::max(*most, t);
        sum += t;
    }
    return sum / k;
}

// Whether a call takes this path: where its estimate is 5 % below fa32_kernel's. Both are fitted to 800
// calls of 17 to 1400 columns, 96 to 5000 keys, 1 to 96 planes, f32 and bf16 K / V, each measured on
// both paths (the mean call is 0.6 % off the faster one; by column and plane counts alone, 14 %).
//  * Here: the three launches, the plan's estimate (with more than two blocks per CU, the chip's rate),
//    and the images written and the K / V read: within 10 % of the time of 90 % of the calls.
//  * fa32_kernel: 1.5 us per 16-key tile of a wavefront's 16 columns (0.7 at D = 64), one wavefront a
//    SIMD at a time, the longest split where the chip is not full, and the combine, a serial chain over
//    the splits (0.4 us each) besides its traffic: within 15 %.
// Short key ranges and few columns stay on fa32_kernel: 8 planes of 195 columns and 196 keys, D = 128:
// 30.7 us here, 18.1 there; 16 planes of 300 columns and 300 keys: 33 and 21; up to 128 keys nothing was
// faster here. 8 planes of 300 columns and 2780 keys: 73 and 53; 4 planes of 2800 columns and 2100 keys at
// D = 64: 29 and 53.
static bool x3_sizes(const FaArgs &a, int wl, int wr, const X3Plan &plan) {
    const int64_t cols = (int64_t)a.q_len * a.group, planes = (int64_t)a.batch * a.kv_heads;
    const int dk = x3_dk(a.head_dim);
    const bool d64 = dk == 64;
    int most;
    double us = plan.split.us;
    if (us == 0.0)
        us = (double)planes * ((cols + 255) / 256) / 256 * (d64 ? 2.5 : 4.9) *
             (x3_mean_tiles(a, wl, wr, 256, kX3Bk, &most) + 2);
    const double mb = (double)planes * a.kv_len * dk * 2 * (6 + fa_kv_esz(a.kv_dtype)) / 1e6;
    const double here = d64 ? 8.5 + 1.12 * us + 0.15 * mb : 11.3 + 1.05 * us + 0.13 * mb;
    const double per_simd = (double)planes * ((cols + 15) / 16) / 1024 * x3_mean_tiles(a, wl, wr, 16, 16, &most);
    const double longest = (d64 ? 0.4 : 0.8) * std::min(most, 2 * a.tiles_per_split);
    const double parts = a.splits > 1 ? (double)a.splits * cols * planes * dk * 8 / 8e6 : 0.0;
    const double there = d64 ? 10.7 + 0.72 * std::max(per_simd, longest) + 0.40 * a.splits + 2.6 * parts
                             : 8.4 + 1.49 * std::max(per_simd, longest) + 0.43 * a.splits + 2.9 * parts;
    return here < 0.95 * there;
}
// What it can take at all.
static bool x3_can(const FaArgs &a) {
    return a.dtype == CQKV_F32 && a.head_dim <= 128 && a.head_dim % 8 == 0 && a.kv_len > 128 &&
           (int64_t)a.q_len * a.group > 16 && (int64_t)a.batch * a.kv_heads <= 65535 &&
           x3_images(a) <= ((size_t)2 << 30);
}

// a: sizes, dtypes and the splits that fa32_kernel would take; 0 where neither a causal nor a full mask
// takes this path.
size_t prefill_f32_workspace(const FaArgs &a) {
    if (!x3_can(a)) return 0;
    const int dk = x3_dk(a.head_dim);
    size_t parts = 0;
    bool any = false;
    for (int wr = -1; wr <= 0; ++wr) {
        const X3Plan p = x3_plan(dk, a, -1, wr);
        any |= x3_sizes(a, -1, wr, p);
        parts = std::max(parts, p.split.bytes);
    }
    return any ? x3_images_end(a) + x3_flags(a) + parts : 0;
}

template <int D, int W>
static void x3_launch(const X3Args &x, hipStream_t st) {
    const FaArgs &a = x.f;
    const unsigned planes = (unsigned)(a.batch * a.kv_heads);
    const dim3 sg((unsigned)x.tiles, planes);
    if (a.kv_dtype == CQKV_F32)
        hipLaunchKernelGGL((prefill_f32_stage_kernel<CQKV_F32, D>), sg, dim3(256), 0, st, x);
    else if (a.kv_dtype == CQKV_F16)
        hipLaunchKernelGGL((prefill_f32_stage_kernel<CQKV_F16, D>), sg, dim3(256), 0, st, x);
    else if (a.kv_dtype == CQKV_BF16)
        hipLaunchKernelGGL((prefill_f32_stage_kernel<CQKV_BF16, D>), sg, dim3(256), 0, st, x);
    else
        hipLaunchKernelGGL((prefill_f32_stage_kernel<kKvE4M3, D>), sg, dim3(256), 0, st, x);
    X3Order order;
    order.n = 0;
    if (x.max_pieces <= 1) {
        hipLaunchKernelGGL((prefill_f32_kernel<D, false, W>), dim3((unsigned)x.q_blocks * planes), dim3(W * 64),
                           0, st, x, order);
        return;
    }
    unsigned rows = (unsigned)(x.q_blocks * x.max_pieces);
    if (!a.cu_q && rows <= kPfMaxWgs) {
        std::pair<int, int> jobs[kPfMaxWgs];  // (-tiles, block << 4 | piece)
        unsigned count = 0;
        for (int qb = x.q_blocks - 1; qb >= 0; --qb) {
            const int64_t c0 = (int64_t)qb * x.nc, cols = (int64_t)a.q_len * a.group;
            int begin;
            const int n = pf_block_tiles((int)(c0 / a.group), (int)((std::min(c0 + x.nc, cols) - 1) / a.group),
                                         a.q_len, a.kv_len, a.wl, a.wr, kX3Bk, begin);
            const int pieces = pf_pieces(n, x.piece_tiles, x.max_pieces);
            for (int p = 0; p < pieces; ++p)
                jobs[count++] = {p + 1 < pieces ? -x.piece_tiles : p * x.piece_tiles - n, qb << 4 | p};
        }
        if (count <= kX3Jobs && x.q_blocks <= 4096) {
            std::stable_sort(jobs, jobs + count,
                             [](const auto &l, const auto &r) { return l.first < r.first; });
            for (unsigned i = 0; i < count; ++i) order.job[i] = (uint16_t)jobs[i].second;
            order.n = (int)count;
            rows = count;
        }
    }
    hipLaunchKernelGGL((prefill_f32_kernel<D, true, W>), dim3(rows * planes), dim3(W * 64), 0, st, x,
                       order);
    constexpr int cpw = 256 / (D / 4);
    const int64_t cols = (int64_t)a.q_len * a.group;
    hipLaunchKernelGGL(prefill_f32_combine_kernel<D>, dim3((unsigned)((cols + cpw - 1) / cpw), planes),
                       dim3(256), 0, st, x);
}

// Runs the call here when its sizes and alignment allow and the workspace, or without one the free
// memory, holds it; *taken says whether it did. plain_bytes: the partials of fa32_kernel's plan. (q /
// out rows 16-byte aligned; K / V rows are in whole 4-element pieces by fa_plain_run's check.)
int prefill_f32_run(const FaArgs &f, const char *who, void *workspace, size_t workspace_bytes,
                    size_t plain_bytes, hipStream_t st, bool *taken) {
    *taken = false;
    if (!x3_can(f) || !f.q_vec || !f.o_vec) return CQKV_OK;
    const int dk = x3_dk(f.head_dim);
    const X3Plan choice = x3_plan(dk, f, f.wl, f.wr);
    const size_t images = x3_images_end(f), parts_off = images + x3_flags(f);
    // (a workspace that holds the images but not the other kernel's partials serves the call here)
    const bool only_here = workspace && workspace_bytes >= images && workspace_bytes < plain_bytes;
    if (!only_here && !x3_sizes(f, f.wl, f.wr, choice)) return CQKV_OK;
    PfPlan plan = choice.split;
    if (workspace && workspace_bytes < images) return CQKV_OK;
    if (workspace && workspace_bytes < parts_off + plan.bytes) plan = PfPlan{};
    X3Args x = {};
    x.f = f;
    x.tiles = (f.kv_len + kX3Bk - 1) / kX3Bk;
    x.nc = 32 * choice.waves;
    x.q_blocks = (int)(((int64_t)f.q_len * f.group + x.nc - 1) / x.nc);
    if ((int64_t)x.q_blocks * f.batch * f.kv_heads * plan.pieces > 0x7fffffff) return CQKV_OK;
    x.piece_tiles = plan.tiles;
    x.max_pieces = plan.pieces;
    x.group_m = pf_group_m(f.group);
    void *ws = workspace;
    if (!ws) ws = scratch_or_null(parts_off + plan.bytes, st);
    if (!ws) return CQKV_OK;  // no memory for the images: the other kernel needs none
    *taken = true;
    x.img = (uint8_t *)ws;
    // (in the images alone, non-finite values stay in them and reach the other rows of their tiles)
    if (!workspace || workspace_bytes >= parts_off) x.bad = (uint32_t *)((char *)ws + images);
    if (plan.pieces > 1) {
        const size_t rows = (size_t)plan.pieces * f.batch * f.q_heads * f.q_len;
        x.f.part_o = (float *)((char *)ws + parts_off);
        x.f.part_lse = (float *)((char *)x.f.part_o + (rows * dk * 4 + 255) / 256 * 256);
    }
    if (dk == 64) choice.waves == 4 ? x3_launch<64, 4>(x, st) : x3_launch<64, 8>(x, st);
    else choice.waves == 4 ? x3_launch<128, 4>(x, st) : x3_launch<128, 8>(x, st);
    hipError_t e = hipGetLastError();
    if (!workspace) {
        const hipError_t fe = hipFreeAsync(ws, st);
        if (e == hipSuccess) e = fe;
    }
    if (e != hipSuccess) return fail(CQKV_ERR_HIP, "%s: launch failed: %s", who, hipGetErrorString(e));
    return CQKV_OK;
}

}  // namespace cqkv
