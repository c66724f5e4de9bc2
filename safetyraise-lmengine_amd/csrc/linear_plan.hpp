// Which kernels a linear call takes and how it is cut (linear_kernels.hip).
// Host code only, so that it is tested without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "safetyraise_kernel.h"

namespace sr {

constexpr int kLinTile = 16;   // rows and outputs per workgroup
constexpr int kLinWaves = 4;   // waves splitting K
constexpr uint32_t kLinMaxSplits = 8;  // K splits per tile at most
constexpr uint32_t kLinBlock = 32;      // k per block (8 MFMAs)
constexpr uint32_t kLinMinSplitK = 512;  // K per split at least (4 blocks per wave)

// linear_rows_kernel: outputs per workgroup
constexpr int kRowsWaves = 8;
constexpr int kRowsBN = kLinTile * kRowsWaves;  // 128 outputs per workgroup

// linear_gemm_wide_kernel
constexpr uint32_t kGemmK = 64;  // K granularity: stages in pairs
constexpr uint32_t kWideMinOutputs = 2048;
constexpr int kWideWM = 2, kWideWN = 2;           // waves over rows, over outputs
constexpr int kWideRT = 4, kWideCT = 4;           // 16 x 16 tiles per wave
constexpr int kWideBM = 16 * kWideRT * kWideWM;   // 128 rows per workgroup
constexpr int kWideBN = 16 * kWideCT * kWideWN;   // 128 outputs per workgroup

// How a call is cut: T output tiles per wave, W waves per workgroup and K
// split over `splits` workgroups per tile (their partial sums are added by
// a second kernel, in split order), never more workgroups than CUs (one
// 8-wave workgroup fills a CU: one more would take a second round).  T = 3
// or, for bf16 weights, 4 (x read once per 48 or 64 outputs, 8 waves: two
// per SIMD; wider weights take more registers than a wave has) when its
// workgroups cover 7/8 of the CUs without a split, or with one when the
// weight is large enough (kLinSplitTElems) that the second kernel's few
// microseconds are small against the stream; otherwise one tile per wave
// and 4 waves, K split until the CUs are covered.  max_splits: what the
// scratch for partial sums holds.
constexpr uint64_t kLinSplitTElems = (uint64_t)32 << 20;
struct LinPlan {
    uint32_t T, W, splits;
};
inline LinPlan linear_plan(uint32_t M, uint32_t N, uint32_t K, uint32_t dtype, int num_cus,
                           uint64_t max_splits = kLinMaxSplits) {
    const uint64_t cus = (uint64_t)(num_cus > 0 ? num_cus : 1);
    const uint64_t mt = (M + kLinTile - 1) / kLinTile;
    auto splits_for = [&](uint64_t tiles) -> uint32_t {
        if (tiles == 0 || tiles >= cus) return 1;
        uint64_t s = cus / tiles;
        s = std::min<uint64_t>(s, K / kLinMinSplitK);
        s = std::min<uint64_t>(s, std::min<uint64_t>(max_splits, kLinMaxSplits));
        return s < 1 ? 1u : (uint32_t)s;
    };
    const uint32_t t_max = dtype == SAFETYRAISE_KERNEL_DTYPE_BF16 ? 4 : 3;
    for (uint32_t T = 3; T <= t_max; ++T) {
        const uint64_t t = (uint64_t)((N + T * kLinTile - 1) / (T * kLinTile)) * mt;
        const uint32_t s = splits_for(t);
        if (t * s * 8 >= cus * 7 && (s == 1 || (uint64_t)N * K >= kLinSplitTElems)) {
            return {T, 8, s};
        }
    }
    const uint64_t t1 = (uint64_t)((N + kLinTile - 1) / kLinTile) * mt;
    return {1, kLinWaves, splits_for(t1)};
}

constexpr uint32_t kMaxRows = 65535u * kLinTile;  // grid y limit of one row-tile launch

// Which kernels a call takes.  All of it rests on cold-weight timings of
// 13 shapes (K, N of 256 .. 12288) at 17 .. 3000 rows; the figures are us.
enum class LinRoute {
    kTile,  // linear_kernel, 16 rows per workgroup (linear_plan)
    kPair,  // linear_kernel, 32 rows per workgroup
    kRows,  // linear_rows_kernel
    kWide,  // split x + linear_gemm_wide_kernel
};
struct LinChoice {
    LinRoute route;
    LinPlan plan;     // kTile's
    uint32_t splits;  // of K over grid z (kTile, kRows)
    size_t scratch;   // bytes the route uses
};

// Split x of a tiled-product call: whole row tiles x K x 3 bf16 parts.
inline size_t split_x_bytes(uint32_t M, uint32_t K) {
    return (size_t)((M + kLinTile - 1) / kLinTile) * kLinTile * K * 3 * sizeof(uint16_t);
}

// K splits of linear_rows_kernel: the least of stages x time per stage (one
// workgroup on a CU, two sharing it, or several rounds of two) plus, with a
// split, the second launch and the partial sums' traffic.  Reproduces the best
// measured split or one within 5 % of it, e.g. 512 rows of 3072 x 1024: 1
// (17.6; 2: 25.7), 1024 of 1024 x 4096: 4 (35.1; 1: 55.4, 3: 40.3).
struct RowsSplit {
    uint32_t splits;
    double us;
};
inline RowsSplit rows_splits(uint32_t M, uint32_t N, uint32_t units, uint32_t base, bool two_tiles,
                             uint64_t cus, size_t scratch) {
    const double one = two_tiles ? 1.1 : 0.86, two = two_tiles ? 1.9 : 1.5;  // us per stage
    const uint64_t outputs = (uint64_t)M * N;
    RowsSplit best{1, 0.0};
    for (uint32_t s = 1; s <= kLinMaxSplits && s <= units; ++s) {
        if (s > 1 && (outputs > UINT32_MAX || outputs * s > scratch / sizeof(float))) break;
        const uint64_t wgs = (uint64_t)base * s;
        const uint64_t rounds = wgs / (2 * cus), rest = wgs % (2 * cus);
        double us = (double)((units + s - 1) / s) *
                    ((double)rounds * two + (rest == 0 ? 0.0 : rest <= cus ? one : two));
        if (s > 1) us += 3.0 + (double)(outputs * (2 * s + 1) * sizeof(float)) / 5e6;
        if (s == 1 || us < best.us) best = {s, us};
    }
    return best;
}

// linear_kernel on a bf16 weight, unsplit, in us: 5 and 0.034 per 16 x 16 x 32
// block of the product and CU.  Of 180 timings from 6 to 1300 us half lie within
// 15 %; calls of 17 to 64 rows, which wait for the weight, take up to 2.6 times
// that.
inline double tile_us(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    return 5.0 + 0.034 / (double)cus * ((double)((M + kLinTile - 1) / kLinTile) * N / kLinTile) *
                     ((double)K / kLinBlock);
}

// scratch: the bytes that are there (SIZE_MAX: as many as the call likes).  No
// route needs any: without it K is not split, and kWide's calls take kRows.
// split_rows: kRows may use it.
inline LinChoice linear_choice(uint32_t M, uint32_t N, uint32_t K, uint32_t dtype, int num_cus,
                               bool x_aligned, size_t scratch, bool split_rows) {
    const uint64_t cus = (uint64_t)(num_cus > 0 ? num_cus : 1);
    const size_t split_bytes = (size_t)M * N * sizeof(float);  // partial sums of one split
    const LinPlan plan = linear_plan(M, N, K, dtype, num_cus, split_bytes ? scratch / split_bytes : 1);
    const LinChoice tile = {LinRoute::kTile, plan, plan.splits,
                            plan.splits > 1 ? plan.splits * split_bytes : 0};
    if (dtype != SAFETYRAISE_KERNEL_DTYPE_BF16 || M <= (uint32_t)kLinTile || M > kMaxRows) return tile;
    const uint64_t weight = (uint64_t)N * K, work = weight * M;
    // nearly two 128 x 128 output tiles per CU or more: 2048 rows of 12288 x
    // 4096 (1536 tiles) 476 against 540 with kRows, of 4096 x 4096 (512) 185 / 210;
    // with fewer kRows, which can split K: 1500 rows of it (384) 173 / 160, 1024
    // (256) 160 / 106.  From 1.5 tiles per CU to there kWide would be up to a fifth
    // faster (1664 rows of 4096 x 1024, 416 tiles, 51 / 61; of 4096 x 192 18.4 / 22.8),
    // and with one stage of K from one tile on (1528 rows of 2752 x 64 11.7 / 13.4),
    // but its one chain of all three parts of x rounds more (relative error at K =
    // 4096 7.0e-7 / 1.4e-7), so it stays with the calls that it had.  Not with fewer
    // outputs than 2048 (k/v projections): there kRows is the faster one too (7168
    // rows of 1024 x 4096 246 / 210, of 1024 x 12288 727 / 628).
    const uint64_t tiles = (uint64_t)((M + kWideBM - 1) / kWideBM) * ((N + kWideBN - 1) / kWideBN);
    if (M > 64 && N >= kWideMinOutputs && K % kGemmK == 0 && K > 0 &&
        4 * tiles >= 7 * cus && split_x_bytes(M, K) <= scratch) {
        return {LinRoute::kWide, {}, 1, split_x_bytes(M, K)};
    }
    const bool pair = M <= 2 * kLinTile;
    // 32 rows, one workgroup of three output tiles on nearly every CU: 12288 x
    // 4096 25.1 against 34.8 (kTile) and 28.2 (kRows, its best split)
    if (pair && x_aligned && K % 8 == 0 && 8 * ((uint64_t)(N + 3 * kLinTile - 1) / (3 * kLinTile)) >= 7 * cus) {
        return {LinRoute::kPair, {}, 1, 0};
    }
    const uint32_t stage = pair ? 4 * kLinBlock : 2 * kLinBlock;
    if (K == 0 || K % stage != 0) return tile;
    // Where the stages and the second launch cost less than reading the
    // weight once per 16 rows: 32 rows of 4096 x 4096 12.8 against 19.2, of
    // 2048 x 6144 13.0 / 15.2, but 2048 x 2048 8.3 / 6.7 and, where kTile
    // covers the CUs without a split, 6144 x 2048 13.0 / 10.0; 64 rows of
    // 2048 x 6144 17.8 / 27.2, 1024 x 4096 13.2 / 10.8, 33 of 6144 x 2048 15.0 /
    // 13.8; 100 of 2048 x 2048 12.5 / 15.7, 512 of 512 x 2048 13.6 / 15.3, but
    // 333 of it 12.3 / 8.8 and 65 (two row blocks, one nearly empty) of 6144 x
    // 2048 20.6 / 19.6; short K: 256 of 3072 x 1024 16.5 / 15.8, 300 of it 17.9 /
    // 18.8.  However short K is, a call of many rows or outputs pays a workgroup
    // per 16 x 16 of them: with a 128 x 128 tile for every other CU, 3840 rows of
    // 1024 x 64 9.7 against 81, 237 of 9088 x 128 9.9 / 50, 17384 of 64 x 576 20 / 48.
    bool pays;
    if (M >= 64 && 2 * tiles >= cus) {
        pays = true;
    } else if (pair) {
        pays = weight >= (12u << 20) && (plan.T < 3 || plan.splits > 1 || weight >= (24u << 20));
    } else if (M <= 64) {
        pays = weight >= (K < 4096 ? 16u << 20 : 12u << 20);
    } else if (M <= 80 && K < 4096) {
        pays = work >= 1000000000u;
    } else {
        pays = work >= (K < 2048 ? 850000000u : N < 1024 ? 500000000u : 300000000u);
    }
    if (!pays) return tile;
    const uint32_t rows = pair ? 2 * kLinTile : 4 * kLinTile;
    const uint32_t base = ((N + kRowsBN - 1) / kRowsBN) * ((M + rows - 1) / rows);
    const RowsSplit liked = rows_splits(M, N, K / stage, base, pair, cus, SIZE_MAX);
    const RowsSplit split = rows_splits(M, N, K / stage, base, pair, cus, split_rows ? scratch : 0);
    // Without the split it likes, a few workgroups walk all of K: 32 rows of 4096
    // x 4096 35.5 (13.1 split) against 20.9 with kTile, 64 of it 57 / 29, 512 of
    // 1024 x 12288 163 / 104, but 200 of 4096 x 4096 57 / 71
    if (split.splits < liked.splits && split.us + 2.0 > tile_us(M, N, K, cus)) return tile;
    return {LinRoute::kRows, {}, split.splits, split.splits > 1 ? split.splits * split_bytes : 0};
}

}  // namespace sr
