"""How a split-K attention launch is cut (csrc/attn_plan.hpp), without a GPU.

split_plan is host code: a small program compiled from the header answers for
calls written to its standard input.
"""
import random
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS = 256
REGION = 64 << 20  # the no-allocation entry point's scratch

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "attn_plan.hpp"
int main(int argc, char **argv) {
    if (argc == 3) {
        printf("%zu\n", sr::grown_bytes(strtoull(argv[1], nullptr, 10), strtoull(argv[2], nullptr, 10)));
        return 0;
    }
    unsigned heads, kv, dim, page, n;
    unsigned long long limit;
    const bool choose = argc == 2;
    while (scanf("%u %u %u %u %llu %u", &heads, &kv, &dim, &page, &limit, &n) == 6) {
        sr::SeqMeta m[64] = {};
        for (unsigned i = 0; i < n; ++i) {
            if (scanf("%u %u", &m[i].ctx, &m[i].rows) != 2) return 1;
        }
        if (choose) {
            uint8_t split[64];
            sr::choose_split({heads, kv, dim, page, 256}, m, (int)n, split);
            for (unsigned i = 0; i < n; ++i) printf("%d ", (int)split[i]);
            printf("\n");
            continue;
        }
        const sr::SplitPlan p = sr::split_plan({heads, kv, dim, page, 256}, m, (int)n, limit);
        printf("%u %llu %u %u %d\n", p.part_keys, (unsigned long long)p.record_bytes,
               p.rows_per_slice, p.records_per_part, (int)p.direct);
    }
}
"""


@pytest.fixture(scope="session")
def plans(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'safetyraise-lmengine_amd' / 'csrc'}", str(where / "plan.cpp"),
                    "-o", str(where / "plan")], check=True)

    def run(calls, *args):
        text = "".join(f"{h} {kv} {d} {p} {lim} {len(seqs)} "
                       + " ".join(f"{c} {r}" for c, r in seqs) + "\n"
                       for h, kv, d, p, lim, seqs in calls)
        return subprocess.run([str(where / "plan"), *args], input=text, capture_output=True,
                              text=True, check=True).stdout.splitlines()

    def ask(calls):
        """calls: (heads, kv_heads, head_dim, page_tokens, limit, [(ctx, rows), ...]), the
        sequences in descending order of their keys."""
        return [dict(zip(("part", "bytes", "rows_per_slice", "per_part", "direct"),
                         map(int, line.split()))) for line in run(calls)]

    ask.chosen = lambda heads, kv, dim, seqs: list(
        map(int, run([(heads, kv, dim, 64, 0, seqs)], "choose")[0].split()))
    ask.grown = lambda have, need: int(subprocess.run(
        [str(where / "plan"), str(have), str(need)], capture_output=True, text=True,
        check=True).stdout)
    return ask


def up(x, unit):
    return -(-x // unit)


def rope_bytes(dim, seqs):
    return up(sum(r for _, r in seqs) * (dim // 2) * 8, 256) * 256


def one_workgroup_per_cu(heads, kv, dim, page, seqs):
    """Record bytes of the plan with one workgroup per CU over the whole call: partitions of
    an equal share of every slice's keys, at least 256."""
    group, most = heads // kv, max(r for _, r in seqs)
    wide = dim <= 128 and most * group > 64
    slices = up(most, (128 if wide else 64) // group)
    part = up(sum(c + r for c, r in seqs) * kv * slices, CUS)
    part = min(max(256, up(part, 64) * 64), 2046 * page // 64 * 64)
    per_part = 2 if dim <= 128 and not wide else 1
    return sum(up(c + r, part) * r for c, r in seqs) * per_part * heads * (dim + 4) * 4


def batch(rng):
    heads, kv, dim = rng.choice([(64, 8, 128), (32, 8, 128), (16, 2, 256), (14, 2, 64), (8, 8, 128)])
    seqs = [(int(2 ** rng.uniform(0, 17)), rng.randint(2, 15)) for _ in range(rng.randint(1, 64))]
    if rng.random() < 0.3:
        seqs = [seqs[0]] * len(seqs)
    return heads, kv, dim, rng.choice([16, 64, 256]), sorted(seqs, key=sum, reverse=True)


def test_draft_rows_fit_the_fixed_scratch_wherever_one_workgroup_per_cu_does(plans):
    rng = random.Random(5)
    calls = [(64, 8, 128, 16, [(16384, 8)] * 64), (64, 8, 128, 16, [(25669, 8)] * 18),
             (16, 2, 256, 16, [(68790, 8)] * 46)] + [batch(rng) for _ in range(3000)]
    limits = [max(0, REGION - rope_bytes(d, s)) for _, _, d, _, s in calls]
    got = plans([(*c[:4], lim, c[4]) for c, lim in zip(calls, limits)])
    assert len(got) == len(calls)
    fitted = 0
    for c, lim, p in zip(calls, limits, got):
        if one_workgroup_per_cu(*c) <= lim:
            fitted += 1
            assert p["bytes"] <= lim, (c, lim, p)
    assert fitted > 2000


def test_plans_are_whole_and_a_limit_only_enlarges_partitions(plans):
    rng = random.Random(6)
    calls = [batch(rng) for _ in range(1000)]
    free = plans([(*c[:4], 2 ** 63, c[4]) for c in calls])
    tight = plans([(*c[:4], p["bytes"] // 2, c[4]) for c, p in zip(calls, free)])
    for (heads, kv, dim, page, seqs), p, q in zip(calls, free, tight):
        for plan in (p, q):
            part = plan["part"]
            assert part % 64 == 0 and part >= 64
            # a partition starting mid-page touches at most 2048 pages
            assert up(part, page) + 1 <= 2048
            longest = sum(seqs[0])
            assert plan["direct"] == (plan["per_part"] == 1 and longest <= part)
            records = sum(up(c + r, part) * r for c, r in seqs) * plan["per_part"]
            assert plan["bytes"] == (0 if plan["direct"] else records * heads * (dim + 4) * 4)
        if q["bytes"] <= p["bytes"] // 2:
            assert q["part"] >= p["part"]


@pytest.mark.parametrize("heads,kv,dim", [(32, 8, 128), (16, 2, 256)])
def test_a_prompt_in_small_chunks_replaces_its_records_a_few_times(plans, heads, kv, dim):
    # 32-row chunks up to 32 K keys: each replacement waits for the stream
    chunks = [(heads, kv, dim, 64, REGION, [(c, 32)]) for c in range(0, 32768, 32)]
    needs = sorted({p["bytes"] for p in plans(chunks)})
    assert len(needs) >= 16
    have, grown = 0, 0
    for need in needs:
        if need > have:
            have = up(plans.grown(have, need), 1 << 20) << 20
            grown += 1
            assert need <= have <= max(need + (1 << 20), REGION)
    assert grown <= 3
    # a single need above the usual limit is met and no more
    assert plans.grown(REGION, REGION + 5) == REGION + 5


# (context, rows) of each sequence; us of a call in one launch of the prefill
# kernels, and with the sequences that are long enough split beside it
@pytest.mark.parametrize("heads,kv,dim,seqs,expected", [
    (32, 8, 128, [(4064, 32)], [1]),                               # 90 / 25
    (32, 8, 128, [(3584, 512)], [1]),                              # 105 / 65
    (32, 8, 128, [(3584, 512)] * 4, [0] * 4),                      # 144 / 243
    (16, 4, 128, [(0, 808), (1351, 165)], [0, 0]),                 # 49 / 60
    (14, 2, 64, [(790, 566), (714, 197), (0, 184), (1712, 52)], [0] * 4),  # 53 / 60
    (8, 8, 64, [(0, 1212)] + [(3, 600)] * 22, [0] * 23),           # 48 / 77 (such a call)
    (32, 8, 128, [(16352, 32), (0, 64)], [1, 0]),                  # 323 / 50
    (16, 2, 256, [(142, 118), (100, 135)], [0, 0]),                # 105 / 127
    (16, 2, 256, [(1000, 32)], [1]),                               # 206 / 28
    (16, 2, 256, [(1000, 1024)] * 4, [1] * 4),                     # 668 / 292
    (8, 2, 256, [(640, 96), (300, 40), (200, 48)], [1, 1, 0]),
    (16, 2, 256, [(100, 40), (0, 200)], [0, 0]),                   # no candidate
])
def test_sequences_are_split_where_the_whole_call_gains(plans, heads, kv, dim, seqs, expected):
    assert plans.chosen(heads, kv, dim, seqs) == expected
