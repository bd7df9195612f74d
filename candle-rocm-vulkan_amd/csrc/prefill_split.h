// Column blocks, key tiles and the split of key ranges over idle CUs, shared by the MFMA prefill
// (prefill_attn.hip) and its f32 form (prefill_f32.hip). A column is one (query, query head) pair of
// a kv head, query-major; a column block is the columns of one workgroup.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "cqkv_device.h"

namespace cqkv {

// ceil(2^32 / group) for group 2 .. 32768, else 0: c / group of the columns of a workgroup
// (c < group + 256) is one multiplication instead of a division's dependent chain in the prologue
// (exact, as c * (m * group - 2^32) < 2^32).
inline uint32_t pf_group_m(int group) {
    return group > 1 && group <= 32768 ? (uint32_t)(0x100000000ull / group + (0x100000000ull % group != 0)) : 0;
}
__device__ inline int pf_div_group(int c, int group, uint32_t m) {
    return group == 1 ? c : m ? (int)__umulhi((uint32_t)c, m) : c / group;
}

// visible keys [lo, hi) of query position i (bottom-right aligned)
__host__ __device__ inline void pf_key_range(int i, int lq, int lk, int wl, int wr, int &lo, int &hi) {
    const int pos = i + lk - lq;
    lo = wl >= 0 ? max(pos - wl, 0) : 0;
    hi = wr >= 0 ? min(pos + wr + 1, lk) : lk;
    lo = min(lo, lk);
    hi = max(hi, lo);
}

// Pieces that n key tiles are cut into: whole pieces of piece_tiles and a last one of up to a
// quarter more (the rest up to a quarter is not worth a workgroup and its partials).
__host__ __device__ inline int pf_pieces(int n, int piece_tiles, int max_pieces) {
    const int rest = n - piece_tiles / 4;
    return max_pieces <= 1 || rest <= piece_tiles ? 1 : min((rest + piece_tiles - 1) / piece_tiles, max_pieces);
}
// Key tiles (of bk keys) of the column block whose queries are q0 .. q1: first tile and count.
__host__ __device__ inline int pf_block_tiles(int q0, int q1, int lq, int lk, int wl, int wr, int bk,
                                              int &begin) {
    int lo, hi, lo1;
    pf_key_range(q0, lq, lk, wl, wr, lo, hi);
    pf_key_range(q1, lq, lk, wl, wr, lo1, hi);
    begin = lo / bk;
    return max((hi + bk - 1) / bk - begin, 0);
}

constexpr int kPfMaxPieces = 16;

// log2-sum-exp of a piece's row from its running maximum and sum: -inf marks a row that sees no key
// of the piece (l 0), and only that: a NaN sum (a NaN key or query, a score of +inf) stays NaN.
__device__ inline float pf_piece_lse(float m, float l) {
    return l == 0.0f ? -__builtin_inff() : m + __builtin_amdgcn_logf(l);
}

// Merges the pieces of one column's row: o = sum_p w_p o_p / sum_p w_p with w_p = 2^(lse_p - max lse)
// (tq_combine_impl's formula, candle-core/kernels/turbo_quant_impl.h:659-685), times o_mul. Called by
// the D / 4 lanes of a column, lane li with head dims 4 li .. 4 li + 3; row: the column's first
// partial, step: rows of a piece. Lane p of each 16 loads piece p's lse (at most kPfMaxPieces = 16),
// so the weights cost one load's latency. Pieces without a visible key are skipped; all others
// count, also where the weight underflows or is NaN, so that non-finite rows come out as the unsplit
// kernel's do.
template <int D>
__device__ inline void pf_merge_pieces(const float *part_o, const float *part_lse, int64_t row,
                                       int64_t step, int pieces, int li, float o_mul, float *o) {
    static_assert((D / 4) % kPfMaxPieces == 0, "whole groups of one lane per piece");
    const int pl = li % kPfMaxPieces;
    const float e = pl < pieces ? part_lse[row + pl * step] : -__builtin_inff();
    float M = e;  // (NaN is passed over)
#pragma unroll
    for (int k = 1; k < kPfMaxPieces; k <<= 1) M = fmaxf(M, __shfl_xor(M, k, kPfMaxPieces));
    const bool empty = e == -__builtin_inff();
    const float w = empty ? -1.0f : __builtin_amdgcn_exp2f(e - M);  // -1: skipped
    float sum = empty ? 0.0f : w;
#pragma unroll
    for (int k = 1; k < kPfMaxPieces; k <<= 1) sum += __shfl_xor(sum, k, kPfMaxPieces);
    const float *po = part_o + row * D + 4 * li;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int p0 = 0; p0 < pieces; p0 += 4) {  // four pieces' rows in flight
        f32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *(const f32x4 *)(po + min(p0 + i, pieces - 1) * step * D);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float wp = __shfl(w, p0 + i, kPfMaxPieces);  // -1 past the last piece
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] += wp < 0.0f ? 0.0f : wp * v[i][k];
        }
    }
    const float inv = sum == 0.0f ? 0.0f : o_mul / sum;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = acc[k] * inv;
}

// How a call's key ranges are split: column blocks of more than `tiles` key tiles in up to `pieces`
// pieces (1: not at all), and the bytes of the partials.
struct PfPlan {
    int tiles = 1 << 30, pieces = 1;
    size_t bytes = 0;
    double us = 0.0;  // the estimate (0: not planned, more than two blocks per CU)
};
// A CU holds one workgroup, so a call of few column blocks leaves CUs idle: one 300-token chunk of a
// 32 / 8-head model over 7000 keys is 40 blocks of 110 tiles on 256 CUs (157 -> 54 us per call in 6
// pieces). The count with the smallest estimate is taken:
//  * steps: key tiles that the last CU to end works through, a workgroup costing some tiles beside
//    its own (its queries, the first tiles' latency, the output). Up to 256 workgroups: the longest;
//    more: the mean per CU and half a workgroup (8 % where the pieces are handed out
//    by size).
//  * a step takes lo us on an idle chip and up to hi us more the fuller it is (clocks, caches: at
//    D = 128, 1.3 us with 40 workgroups, 1.86 us with 200), so t = lo * steps + hi * mean tiles per CU.
//  * the combine: 3 us, and its partials written and read, mostly cached, at 8 TB/s (6.8 us for 9600
//    rows of 5 pieces).
// A causal prompt of about as many blocks as CUs keeps them whole: its mean is half of its longest,
// but the rate rises as CUs fall idle, and the partials cost what is left (2048 tokens, 32 / 8 heads:
// 62.6 us whole, 66.2 us in halves; 3000 tokens: 91.7 and 110.2). Whole pieces have at least
// min_keys (512 in the 16-bit prefill), so shorter key ranges are never split; the last piece of a block
// may be anything above a quarter of a whole one (pf_pieces).
struct PfShape {
    int nc, bk, head_dim;  // columns of a block, keys of a tile, head dim of the partials
    double lo, hi;         // step time, us: lo idle, lo + hi with every CU busy
    int setup, min_keys;   // tiles' worth of a workgroup's setup, smallest piece
    bool sorted;           // pieces are handed out by size: the CUs end together
};
constexpr int kCus = 256;  // gfx950 (MI355X); a part with fewer would only be planned less well
constexpr int kPfMaxBlocks = 2 * kCus, kPfMaxWgs = 8 * kCus;  // planned (a plane's) and split into (a call's)
inline PfPlan pf_plan(const PfShape &g, int batch, int q_len, int kv_len, int q_heads, int kv_heads,
                      int wl, int wr) {
    const int nc = g.nc, bk = g.bk, min_tiles = g.min_keys / bk, group = q_heads / kv_heads;
    const double lo = g.lo, hi = g.hi;
    const int64_t planes = (int64_t)batch * kv_heads, cols = (int64_t)q_len * group;
    const int64_t blocks = (cols + nc - 1) / nc;
    PfPlan best;
    if (planes * blocks > kPfMaxBlocks || kv_len <= g.min_keys) return best;
    int n[kPfMaxBlocks];  // key tiles, in the order the blocks are handed out
    int most = 0;
    for (int64_t i = 0; i < blocks; ++i) {
        const int64_t c0 = (blocks - 1 - i) * nc;
        int begin;
        n[i] = pf_block_tiles((int)(c0 / group), (int)((std::min(c0 + nc, cols) - 1) / group), q_len,
                              kv_len, wl, wr, bk, begin);
        most = std::max(most, n[i]);
    }
    double &best_us = best.us;
    for (int p = 1; p <= kPfMaxPieces; ++p) {
        const int tiles = (most + p - 1) / p;
        if (p > 1 && (tiles < min_tiles || planes * blocks * p > kPfMaxWgs)) break;
        int64_t wgs = 0, total = 0, split_cols = 0;
        int longest = 0;
        for (int64_t i = 0; i < blocks; ++i) {
            const int k = pf_pieces(n[i], tiles, p);
            const int last = n[i] - (k - 1) * tiles;
            longest = std::max(longest, k > 1 ? std::max(last, tiles) : last);
            wgs += planes * k;
            total += planes * (n[i] + (int64_t)k * g.setup);
            if (k > 1) split_cols += k * nc;
        }
        const double mean = (double)total / kCus;
        double steps = longest + g.setup;
        if (wgs > kCus) steps = std::max(steps, g.sorted ? 1.08 * mean : mean + 0.5 * total / wgs);
        double t = lo * steps + hi * mean;
        if (p > 1) t += 3.0 + (double)planes * split_cols * g.head_dim * 8 / 8e6;
        if (p == 1 || t < (best.pieces == 1 ? 0.92 : 0.97) * best_us) {
            best_us = t;
            best.tiles = tiles;
            best.pieces = p;
        }
    }
    if (best.pieces > 1)
        best.bytes = ((size_t)best.pieces * planes * cols * g.head_dim * 4 + 255) / 256 * 256 +
                     (size_t)best.pieces * planes * cols * 4;
    return best;
}

}  // namespace cqkv
