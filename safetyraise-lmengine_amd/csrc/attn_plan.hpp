// How a split-K attention launch (attn_verify_kernel in attn_prefill.hip) is
// cut.  Host code only, so that it is tested without a GPU.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "sr_internal.hpp"

namespace sr {

constexpr int kKeyTile = 64;  // keys per LDS stage of the prefill and split-K kernels

// LDS entries for the page ids of one partition (a partition never spans more
// pages)
constexpr uint32_t kVerifyPageSlots = 2048;

// Floats of a partition record: m, l, 2 unused, o[head_dim] (16-byte aligned).
constexpr uint32_t record_stride(uint32_t head_dim) { return head_dim + 4; }

// Bytes to reserve for records when `have` are there and `need` are not: 8 MiB
// at least, then at least twice what was there, up to the records' usual limit.
// A context that grows by a few keys a call replaces the buffer a few times and
// not every few partitions (32 rows of 32 / 8 x 128 take another 1.1 MB every
// 512 keys; each replacement is a wait for the stream and 0.3 ms).  First pass
// of a 16 K prompt by 32 rows, 17.2 ms once warm: 18.6, grown by 1 MB 21.4.
inline size_t grown_bytes(size_t have, size_t need) {
    constexpr size_t kLeast = (size_t)8 << 20;
    return std::max(need, std::min(std::max(2 * have, kLeast), kAttnScratchBytes));
}

struct SplitShape {
    uint32_t heads, kv_heads;  // of the grid: at most 8 query heads per KV head
    uint32_t head_dim, page_tokens;
    int num_cus;
};

// Sequences of 16 or more rows that may take the split-K kernel.  The prefill
// kernels run one workgroup per row block and KV head down the whole context,
// so a chunk of few rows leaves most CUs idle: 32 rows of 32 / 8 x 128 at 4096
// keys 90 us, split 25; at 16 K keys 323 / 38.  Below these lengths the second
// launch and the records cost what the split gives (32 rows at 320 keys 18 / 17
// us, 256 rows at 640 keys 31 / 24 but four such sequences 32 / 58).  Head_dim
// 256 has no kernel but the lock-step one, 10 us per 64 keys (32 rows of 16 / 2
// at 1 K keys 206 us, split 28; 1024 rows 364 / 88, four such 668 / 292).
inline bool split_candidate(const SplitShape &a, const SeqMeta &m) {
    const uint32_t g = a.heads / a.kv_heads;
    const uint64_t keys = (uint64_t)m.ctx + m.rows;
    if (a.head_dim > 128) return keys > 256;
    return keys > (m.rows * g <= 128 && m.rows <= 64 ? 320u : 1024u);
}

// Which of a call's sequences of 16 or more rows take the split-K kernel: the
// candidates, where that makes the call faster by a margin of a tenth, or none.
// Times in us, fitted to calls of one and four sequences of 16 to 1024 rows at
// 128 to 16 K keys: the prefill kernels take a start and a time per 64-key tile
// of the longest workgroup (more with every CU busy), the split form a start, a
// time per tile of an equal share per CU, and the merge of the records.  32 / 8 x
// 128, estimated (measured): 512 rows at 4096 keys 125 (105) / 78 (65), 1024 rows
// at 16 K 534 (373) / 400 (346), four sequences of 512 rows at 4096 keys 150 (144)
// / 233 (243).  The sequences that are no candidates run the prefill kernels
// beside or after them: 808 rows and 165 after 1351 keys (16 / 4 x 128) 49 us in
// one launch, 60 with the second sequence split; 23 sequences of 23 to 1212 rows
// (8 / 8 x 64) 48 / 77; 118 rows after 142 keys and 135 after 100 (16 / 2 x 256) 105 /
// 127.  At head_dim 256 any candidate on its own gains.
inline void choose_split(const SplitShape &a, const SeqMeta *seqs, int nseq, uint8_t *split) {
    int candidates = 0;
    for (int i = 0; i < nseq; ++i) {
        split[i] = split_candidate(a, seqs[i]);
        candidates += split[i];
    }
    if (candidates == 0) return;
    struct Times {
        double block, start, tile, tile_busy;          // prefill kernels; query vectors a block
        double slice, split_start, split_tile, record;  // split form; query vectors a slice
    };
    const Times t = a.head_dim == 64    ? Times{256, 6, 1.43, 0.05, 128, 11, 0.95, 0.0004}
                    : a.head_dim == 128 ? Times{256, 12, 1.22, 0.7, 128, 17, 1.4, 0.0004}
                                        : Times{128, 60, 9, 0, 64, 22, 2.8, 0};
    const uint32_t g = a.heads / a.kv_heads;
    const double cus = std::max(a.num_cus, 1);
    auto tiles = [&](int i) { return ((double)seqs[i].ctx + seqs[i].rows) / kKeyTile; };
    // the prefill kernels over all the sequences, or those that are no candidates
    auto whole = [&](bool all) {
        double wgs = 0, total = 0, longest = 0;
        for (int i = 0; i < nseq; ++i) {
            if (split[i] && !all) continue;
            const double blocks = std::ceil((double)seqs[i].rows * g / t.block) * a.kv_heads;
            wgs += blocks;
            total += blocks * tiles(i);
            longest = std::max(longest, tiles(i));
        }
        return wgs == 0 ? 0.0
                        : t.start + (t.tile + t.tile_busy * std::min(1.0, wgs / cus)) *
                                        std::max(longest, total / cus);
    };
    double share = 0, records = 0;
    for (int i = 0; i < nseq; ++i) {
        if (!split[i]) continue;
        const double vectors = (double)seqs[i].rows * g;
        share += std::ceil(vectors / t.slice) * a.kv_heads * (tiles(i) - 0.5 * seqs[i].rows / kKeyTile);
        records += vectors * a.kv_heads;
    }
    const double parts =
        t.split_start + t.split_tile * std::max(share / cus, 2.0) + t.record * records + whole(false);
    if (parts * 1.1 >= whole(true)) std::fill(split, split + nseq, (uint8_t)0);
}

struct SplitPlan {
    bool all_tiles;             // each consumer wave takes both tiles of a step
    bool direct;                // every (row, head) has one record: the output itself
    uint32_t rows_per_slice;    // query rows per workgroup
    uint32_t records_per_part;  // per (row, head): one per tile of a step
    uint32_t part_keys;
    uint64_t record_bytes;
};

// Keys per partition, a multiple of the 64-key tile, of sequences in descending
// order of their keys.  A workgroup has a CU to itself and costs its keys plus
// a start and end worth about 5 tiles, so the candidates are one to four
// workgroups per CU, each with the smallest partition of at least 256 keys that
// keeps to that number, and, with one record per partition, no split and no
// merge pass: the first sequence's workgroups in whole rounds, those of shorter
// ones after what is before them.
//
// A candidate whose records take more than record_limit bytes has its
// partitions enlarged until they fit; with a partition for every KV head's
// whole context there is nothing larger, and if that takes too much as well the
// plan is the first candidate (one workgroup per CU) as it was, with
// record_bytes above the limit.  64 sequences of 16 K keys and 8 rows each (64 /
// 8 x 128): four workgroups per CU took 69 MB of records, one takes 35.
inline SplitPlan split_plan(const SplitShape &a, const SeqMeta *seqs, int nseq,
                            uint64_t record_limit) {
    const uint64_t kvv = a.kv_heads, group = a.heads / a.kv_heads;
    const uint64_t cus = std::max(a.num_cus, 1);
    constexpr uint64_t kEnds = 5 * kKeyTile;
    constexpr uint64_t kMerge = 3 * kKeyTile;
    auto up = [](uint64_t x, uint64_t unit) { return (x + unit - 1) / unit; };
    SplitPlan plan{};
    uint64_t max_rows = 0;
    uint64_t total[kMetaPerLaunch], slices[kMetaPerLaunch];  // keys, row slices
    for (int i = 0; i < nseq; ++i) {
        max_rows = std::max<uint64_t>(max_rows, seqs[i].rows);
        total[i] = (uint64_t)seqs[i].ctx + seqs[i].rows;
    }
    // query vectors per workgroup: 64 in the pair mode; at D <= 128 a call
    // with more takes the all-tiles form (128 vectors over its four consumer
    // waves), rows beyond run as further slices of the rows
    plan.all_tiles = a.head_dim <= 128 && max_rows * group > 64;
    plan.rows_per_slice = (uint32_t)((plan.all_tiles ? 128 : 64) / group);
    plan.records_per_part = (a.head_dim <= 128 && !plan.all_tiles) ? 2 : 1;
    for (int i = 0; i < nseq; ++i) slices[i] = up(seqs[i].rows, plan.rows_per_slice);
    auto direct = [&](uint64_t part) { return plan.records_per_part == 1 && total[0] <= part; };
    auto bytes = [&](uint64_t part) -> uint64_t {
        if (direct(part)) return 0;
        uint64_t n = 0;
        for (int i = 0; i < nseq; ++i) n += up(total[i], part) * seqs[i].rows;
        return n * plan.records_per_part * a.heads * record_stride(a.head_dim) * sizeof(float);
    };
    // a partition starting mid-page touches at most part/page_tokens + 2 pages
    const uint64_t max_part = std::min<uint64_t>(
        ((uint64_t)(kVerifyPageSlots - 2) * a.page_tokens) / kKeyTile * kKeyTile, 1u << 30);
    const uint64_t longest = up(total[0], kKeyTile) * kKeyTile;
    const uint64_t most = std::min(longest, max_part);
    uint64_t keys = 0, unsplit = 0, before = 0;
    for (int i = 0; i < nseq; ++i) {
        const uint64_t n = slices[i] * kvv;
        // (a slice sees the context and the rows up to its own last)
        keys += n * seqs[i].ctx +
                kvv * (seqs[i].rows + plan.rows_per_slice * (slices[i] - 1)) * slices[i] / 2;
        unsplit = std::max(unsplit, i == 0 ? up(n, cus) * (total[i] + kEnds)
                                           : (before + n * (total[i] + kEnds)) / cus + total[i]);
        before += n * (total[i] + kEnds);
    }
    uint64_t best = 0, best_time = ~0ull, first = 0;
    if (longest <= max_part && bytes(longest) <= record_limit) {
        best = longest;
        best_time = unsplit + (plan.records_per_part > 1 ? kMerge : 0);
    }
    for (uint64_t per = 1; per <= 4; ++per) {
        uint64_t part = std::max<uint64_t>(256, up(keys, per * cus * kKeyTile) * kKeyTile);
        // (each sequence's last partition is short: a few steps up until they fit)
        for (int step = 0; step < 32 && part < longest; ++step) {
            uint64_t n = 0;
            for (int i = 0; i < nseq; ++i) n += up(total[i], part) * slices[i];
            if (n * kvv <= per * cus) break;
            part += up(part, 32 * kKeyTile) * kKeyTile;
        }
        part = std::min(part, most);
        if (per == 1) first = part;
        while (part < most && bytes(part) > record_limit) {
            part = std::min(most, part + up(part, 8 * kKeyTile) * kKeyTile);
        }
        if (part >= longest || bytes(part) > record_limit) continue;
        const uint64_t time = per * (part + kEnds) + kMerge;
        if (time < best_time) {
            best_time = time;
            best = part;
        }
    }
    if (best == 0) best = first;
    plan.part_keys = (uint32_t)best;
    plan.direct = direct(best);
    plan.record_bytes = bytes(best);
    return plan;
}

}  // namespace sr
