"""csrc/attn_plan.h, how attention tiles are dealt to several work-groups: plain C++, compiled here and run on the CPU."""
import ctypes as C
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "async-grpo-nccl_amd", "csrc")
MAX_PARTS = 8

SOURCE = r"""
#include "attn_plan.h"
using namespace fgrpo;
extern "C" {
int inside(int np, int first, int skip, int stride, int grid) { return attn_parts_inside(np, first, skip, stride, grid); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("attn_plan")
    src, lib = str(where / "plan.cpp"), str(where / "plan.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{CSRC}", src, "-o", lib], check=True)
    return C.CDLL(lib)


def test_merges_follow_no_entry_out_of_the_launch(plan):
    """Whatever an unwritten table entry holds, an accepted one reads inside the launch; every entry that a launch of so many
    work-groups can write is accepted.  The smallest launches are those of the shortest batches, of one work-group an XCD
    and few more, which eight parts do not fit."""
    rng = random.Random(1)
    wild = [0, 1, 2, 8, 9, -1, -2 ** 31, 2 ** 31 - 1, 0x7f7f7f7f]
    accepted = 0
    for _ in range(20000):
        nb = rng.choice((1, 1, 2, 3, 16))
        stride, grid = 8 * nb, 8 * rng.choice((nb, nb + 1, 4 * nb + 3, 300))
        skip, np = 8 * rng.randrange(nb), rng.choice(wild + list(range(2, 9)))
        first = rng.choice(wild + [rng.randrange(grid), grid - 1, grid, grid + 7])
        reads = [first + skip + j * stride for j in range(np)] if 1 < np <= MAX_PARTS else []
        ok = bool(reads) and first >= 0 and max(reads) < grid
        assert bool(plan.inside(np, first, skip, stride, grid)) == ok, (np, first, skip, stride, grid)
        accepted += ok
    assert 1000 < accepted < 19000
