"""Which kernels a linear call takes (csrc/linear_plan.hpp), without a GPU.

linear_choice is host code: a small program compiled from the header answers
for shapes written to its standard input.
"""
import random
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS = 256
F32, F16, BF16 = 1, 2, 3
TILE, PAIR, ROWS, WIDE = range(4)
ANY = 2 ** 64 - 1  # as much scratch as a call likes

PROGRAM = r"""
#include <cstdio>
#include "linear_plan.hpp"
int main() {
    unsigned m, n, k, dtype, aligned, split;
    unsigned long long scratch;
    while (scanf("%u %u %u %u %u %u %llu", &m, &n, &k, &dtype, &aligned, &split, &scratch) == 7) {
        const sr::LinChoice c = sr::linear_choice(m, n, k, dtype, 256, aligned != 0,
                                                  (size_t)scratch, split != 0);
        printf("%d %u %zu\n", (int)c.route, c.splits, c.scratch);
    }
}
"""


@pytest.fixture(scope="session")
def choose(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'safetyraise-lmengine_amd' / 'csrc'}", str(where / "plan.cpp"),
                    "-o", str(where / "plan")], check=True)

    def ask(shapes, scratch=ANY, dtype=BF16, aligned=True, split_rows=True):
        """(route, K splits, scratch bytes) of each (rows, outputs, columns)."""
        text = "".join(f"{m} {n} {k} {dtype} {int(aligned)} {int(split_rows)} {scratch}\n"
                       for m, n, k in shapes)
        out = subprocess.run([str(where / "plan")], input=text, capture_output=True, text=True,
                             check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return ask


def up(x, unit):
    return -(-x // unit)


def shapes(seed, count, cols=64):
    """(rows, outputs, columns), columns a multiple of `cols`."""
    rng = random.Random(seed)

    def spread(lo, hi):
        return int(2 ** rng.uniform(lo, hi))

    return [(spread(0, 17), spread(4, 14), up(spread(4, 14), cols) * cols) for _ in range(count)]


def tiles(m, n):
    return up(m, 128) * up(n, 128)


def test_short_columns_do_not_send_many_rows_to_the_row_tiles(choose):
    # a 128 x 128 output tile for every other CU, however little there is to add up
    many = [s for s in shapes(1, 6000) if s[0] >= 64 and 2 * tiles(s[0], s[1]) >= CUS]
    many += [(3840, 1024, 64), (237, 9088, 128), (64, 16384, 64), (17384, 64, 576)]
    assert len(many) > 1000
    for shape, (route, _, _) in zip(many, choose(many)):
        assert route in (ROWS, WIDE), shape


def test_calls_of_few_outputs_sum_the_parts_of_x_in_two_chains(choose):
    # the tiled product adds the three parts of x in one chain: not below 2048 outputs
    few = [s for s in shapes(2, 6000) if s[1] < 2048 and 4 * tiles(s[0], s[1]) >= 7 * CUS]
    few += [(7168, 1024, 4096), (3840, 1920, 12288), (60000, 1024, 64)]
    assert len(few) > 200
    for shape, (route, _, _) in zip(few, choose(few)):
        assert route == ROWS, shape


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("scratch", [0, 1 << 20, 40 << 20])
def test_no_call_needs_more_scratch_than_there_is(choose, dtype, aligned, scratch):
    calls = shapes(3, 3000, cols=8) + [(1, 1024, 4096), (9, 4096, 12288), (2048, 4096, 4096)]
    liked = choose(calls, dtype=dtype, aligned=aligned)
    got = choose(calls, scratch=scratch, dtype=dtype, aligned=aligned)
    short = 0
    for call, like, have in zip(calls, liked, got):
        short += like[2] > scratch
        assert have[2] <= scratch, call
        assert have[1] <= like[1] or like[0] != have[0], call
        if like[2] <= scratch:
            assert have == like, call
    assert short > 0 or dtype != BF16


# without a K split; us of the row tiles and of linear_rows_kernel
@pytest.mark.parametrize("shape,route", [
    ((32, 4096, 4096), TILE),     # 21 / 36
    ((64, 4096, 4096), TILE),     # 29 / 57
    ((256, 1024, 4096), TILE),    # 25 / 56
    ((512, 1024, 12288), TILE),   # 104 / 163
    ((200, 4096, 4096), ROWS),    # 71 / 57
    ((400, 2048, 6144), ROWS),    # 106 / 83
    ((1024, 1024, 12288), ROWS),  # 186 / 162
])
def test_a_call_that_cannot_split_takes_the_faster_kernel(choose, shape, route):
    liked, splits, _ = choose([shape])[0]
    assert liked == ROWS and splits > 1
    for got in (choose([shape], split_rows=False), choose([shape], scratch=0)):
        assert got[0][0] == route and got[0][1] == 1
