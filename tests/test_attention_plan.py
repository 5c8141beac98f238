"""csrc/attn_plan.h, how attention tiles are dealt to several work-groups: plain C++, compiled here and run on the CPU."""
import ctypes as C
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "async-grpo-nccl_amd", "csrc")
MAX_PARTS = 8

SOURCE = r"""
#include <math.h>
#include <vector>
#include "attn_plan.h"
using namespace fgrpo;

// The numbering of attn_deal on one XCD, with whole-number divisions: 0, or what is wrong.  `seen` counts the parts of a tile and head
// (of all XCDs), of which each part must cover its share of the steps.
static int deal(const std::vector<int>& steps, const std::vector<int>& what, int xcd, int width, const SplitPlan& s, int grid, std::vector<int>& seen) {
  auto quotient = [](int n, int d) { return n / d; };
  const int slots = (int)steps.size(), budget = slots * width + s.extra;
  long long sum = 0;
  for (int x : steps) sum += x > 0 ? x : 0;
  sum *= width;
  if (sum >= 1LL << 31) return 1;
  auto parts_at = [&](int i, int per) { return steps[i] < 0 ? 0 : attn_parts(steps[i], s.parts, per, quotient); };
  const int per = attn_part_steps((int)sum, budget, s.extra, s.per, s.deal, [&](int x) {
    int n = 0;
    for (int i = 0; i < slots; ++i) n += parts_at(i, x);
    return n * width;
  });
  if (per < 1) return 2;
  int base = 0;
  for (int i = 0; i < slots; ++i) {
    const int np = parts_at(i, per);
    if (np == 0) continue;
    if (np > kAttnMaxParts || steps[i] + per - 1 >= 1 << 21 || steps[i] * np >= 1 << 21) return 3;      // the range of the quotients by reciprocal
    for (int u = 0; u < width; ++u)
      if (np > 1 && !attn_parts_inside(np, 8 * base + xcd, 8 * u, 8 * width, grid)) return 4;
    int walked = 0;
    for (int j = 0; j < np; ++j) walked += steps[i] * (j + 1) / np - steps[i] * j / np;
    if (walked != steps[i]) return 5;
    seen[what[i]] += 1;
    base += np * width;
  }
  return base > budget || 8 * (budget - 1) + xcd >= grid ? 6 : 0;
}

extern "C" {
int inside(int np, int first, int skip, int stride, int grid) { return attn_parts_inside(np, first, skip, stride, grid); }

// A launch over the segments cu[0 .. n]: which (0: forward, 1: dQ, 2: dK/dV); order: a permutation of its tiles (128-key tiles for 2).
// Negative: it is left whole; 0: divided, as it has to be; else what is wrong.
int launch(int cus, int heads, int which, const int* cu, int n, int max_len, int Hq, int Hkv, int D, int causal, int merged, const int* order) {
  const int T = cu[n];
  std::vector<int> first(T), end(T);
  for (int i = 0; i < n; ++i)
    for (int t = cu[i]; t < cu[i + 1]; ++t) first[t] = cu[i], end[t] = cu[i + 1];
  const SplitPlan s = which == 2 ? plan_key_split(cus, 0, T, n, max_len, Hq, Hkv, D, causal)
                                 : plan_query_split(cus, heads, 0, T, n, max_len, Hq, Hkv, D, causal, which == 0, merged);
  if (s.parts <= 1) return -1;
  if (s.extra < 1 || s.deal < 1 || s.per < 1 || s.parts > kAttnMaxParts) return 10;
  const size_t sums = which == 2 ? key_sums_bytes(s, D) : query_sums_bytes(s, D), rows = which == 2 ? 2 * attn_keyside_keys(D) : 128;
  if (sums < (size_t)s.grid * rows * D * 4 || sums % 256) return 11;
  const int hb = attn_heads_per_group(heads, Hq / Hkv, T, n), rb = 128 / hb, nb = (Hq / Hkv + hb - 1) / hb, keys = attn_keyside_keys(D);
  const int size = which == 2 ? keys : rb, ntile = (T + size - 1) / size, width = which == 2 ? 1 : nb;
  const int blocks = which == 2 ? attn_keyside_blocks(D, T, Hkv) : attn_query_blocks(hb, T, Hq, Hkv), slots = blocks / 8 / width;
  if (s.grid != blocks + 8 * s.extra || slots * width * 8 != blocks || slots > kAttnDealSlots) return 12;
  std::vector<int> seen(ntile * Hkv);
  for (int xcd = 0; xcd < 8; ++xcd) {
    std::vector<int> steps(slots, -1), what(slots, -1);
    for (int slot = 0; slot < slots; ++slot) {
      const int unit = 8 * slot + xcd;
      int tile = -1, head = 0;
      if (which == 2) {
        const KeyPick pick = attn_key_pick(unit, (T + 127) / 128, 128 / keys, Hkv);
        if (pick.rank >= 0) tile = order[pick.rank] * (128 / keys) + pick.piece, head = pick.head;
        if (tile >= ntile) tile = -1;
      } else if (unit < ntile * Hkv) {
        tile = order[unit / Hkv], head = unit % Hkv;
      }
      if (tile < 0) continue;
      const int a = tile * size, b = a + size < T ? a + size : T;
      what[slot] = tile * Hkv + head;
      if (which == 2) steps[slot] = ((end[b - 1] - (causal ? a : first[a]) + kDkv3Rows - 1) / kDkv3Rows * (Hq / Hkv) + 3) / 4;
      else steps[slot] = ((causal ? b : end[b - 1]) - first[a] + kAttnBK - 1) / kAttnBK;
    }
    const int rc = deal(steps, what, xcd, width, s, s.grid, seen);
    if (rc) return rc;
  }
  for (int x : seen)
    if (x != 1) return 13;
  return 0;
}

int divided(int which, int T, int n, int max_len, int Hq, int Hkv, int D) {
  return (which == 2 ? plan_key_split(256, 0, T, n, max_len, Hq, Hkv, D, 1) : plan_query_split(256, 0, 0, T, n, max_len, Hq, Hkv, D, 1, which == 0, 0)).parts > 1;
}
unsigned long long sums(int which, int T, int n, int max_len, int Hq, int Hkv, int D, int causal) {
  const SplitPlan s = which == 2 ? plan_key_split(256, 0, T, n, max_len, Hq, Hkv, D, causal) : plan_query_split(256, 0, 0, T, n, max_len, Hq, Hkv, D, causal, which == 0, 1);
  return s.parts <= 1 ? 0 : which == 2 ? key_sums_bytes(s, D) : query_sums_bytes(s, D);
}
int heads(int wanted, int G, int T, int n) { return attn_heads_per_group(wanted, G, T, n); }

// n / d by reciprocal, with the reciprocal one unit in the last place off either way
int quotients(int n, int d) {
  const float r = 1.0f / (float)d, off[3] = {r, nextafterf(r, 0.0f), nextafterf(r, 2.0f)};
  for (float x : off)
    if ((int)(((float)n + 0.5f) * x) != n / d) return 0;
  return 1;
}
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("attn_plan")
    src, lib = str(where / "plan.cpp"), str(where / "plan.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{CSRC}", src, "-o", lib], check=True)
    lib = C.CDLL(lib)
    lib.sums.restype = C.c_ulonglong
    return lib


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


def test_quotients_by_reciprocal(plan):
    """Exact below 2^21, whatever the last bit of the reciprocal: at the numbers next to a multiple, where they could go wrong."""
    rng = random.Random(2)
    for d in list(range(1, 200)) + [rng.randrange(200, 2 ** 21) for _ in range(2000)]:
        most = (2 ** 21 - 1) // d
        for k in {0, 1, 2, most - 1, most, rng.randint(0, most), rng.randint(0, most)}:
            for n in (k * d - 1, k * d, k * d + 1):
                assert not 0 <= n < 2 ** 21 or plan.quotients(n, d), (n, d)


def _segments(rng, T):
    kind, out, at = rng.randrange(4), [0], 0
    while at < T:
        k = T if kind == 0 else rng.randint(1, T) if kind == 1 else rng.randint(1, 700) if kind == 2 else rng.choice((1, 2, 31, 64, T))
        at = min(at + k, T)
        out.append(at)
    return out


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("causal", [0, 1])
def test_every_tile_gets_its_parts_and_no_launch_more_than_it_has(plan, which, causal):
    """Divided launches of any shape: on every XCD the parts fit the work-groups of the launch, every tile and head is taken exactly once,
    its parts cover its steps, the merge finds them inside the launch and the workspace holds them.  With the length of the longest segment
    named, wrong or left out, the tiles in any order, K/V heads that do not divide eight."""
    rng = random.Random(10 * which + causal)
    divided = 0
    for _ in range(8000):
        T = int(2 ** rng.uniform(4, 14))
        cu = _segments(rng, T)
        n = len(cu) - 1
        Hkv, G, D = rng.choice((1, 2, 3, 4, 5, 6, 8)), rng.choice((1, 2, 3, 4, 6, 7, 8, 12)), rng.choice((64, 128))
        heads, longest = rng.choice((0, 0, 0, 1, 2, 4)), max(b - a for a, b in zip(cu, cu[1:]))
        length = rng.choice((longest, longest, 0, 1, T, rng.randint(1, T)))
        size = 128 if which == 2 else {1: 128, 2: 64, 4: 32}[plan.heads(heads, G, T, n)]
        order = list(range((T + size - 1) // size))
        rng.shuffle(order)
        rc = plan.launch(rng.choice((256, 256, 304, 64)), heads, which, (C.c_int * (n + 1))(*cu), n, length, G * Hkv, Hkv, D, causal, rng.randrange(2),
                         (C.c_int * len(order))(*order))
        assert rc <= 0, (rc, which, T, n, length, G * Hkv, Hkv, D, causal, heads)
        divided += rc == 0
    assert divided > 200


@pytest.mark.parametrize("T,n,longest,Hq,Hkv,D,divided", [
    (7359, 1, 7359, 28, 4, 128, False), (15330, 1, 15330, 12, 2, 128, False), (32768, 1, 32768, 4, 1, 128, False),
    (28241, 14, 7263, 14, 2, 64, False), (32768, 30, 5808, 14, 2, 64, False), (12345, 22, 1821, 28, 4, 128, False),
    (777, 1, 777, 12, 2, 128, True), (5000, 1, 5000, 28, 4, 128, True), (6000, 13, 1694, 16, 4, 128, True),
    (9000, 14, 2048, 12, 2, 128, True), (2000, 1, 2000, 14, 2, 64, True), (7472, 7, 3821, 16, 4, 128, True),
    (9178, 12, 3889, 28, 4, 128, True), (2730, 2, 1772, 40, 8, 128, True), (11848, 25, 928, 12, 2, 128, True)])
def test_tiles_of_several_rounds_are_dealt_out_where_one_is_long(plan, T, n, longest, Hq, Hkv, D, divided):
    """dQ + dK/dV of these took 3 to 9 % longer dealt out, or, where the launch is divided, at least as much longer whole."""
    assert bool(plan.divided(2, T, n, longest, Hq, Hkv, D)) == divided


@pytest.mark.parametrize("causal", [0, 1])
def test_partial_sums_of_a_launch_stay_within_256_mib(plan, causal):
    """As they are allocated, by whole work-groups: the heads of a group that do not fill one (5 as 8) count.  A backward has two such
    launches, and small tables beside the sums."""
    rng = random.Random(7 + causal)
    most = 0
    for _ in range(60000):
        T, Hkv, G = int(2 ** rng.uniform(8, 17)), rng.choice((1, 2, 3, 4, 8)), rng.choice((1, 2, 3, 5, 6, 7, 9, 13))
        n, D, which = rng.choice((1, 1, 2, 3, 4, 8)), rng.choice((64, 128)), rng.randrange(3)
        b = plan.sums(which, T, n, rng.choice((0, T, -(-T // n))), G * Hkv, Hkv, D, causal)
        assert b <= 256 << 20, (which, T, n, G * Hkv, Hkv, D)
        most = max(most, b)
    assert most > (200 if causal else 80) << 20
