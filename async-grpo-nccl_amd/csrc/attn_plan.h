// How attention tiles are dealt to several work-groups: what host and kernels agree on.  Plain C++ (constexpr functions run on
// either side), so that a test can compile it by itself.
#pragma once
#include <math.h>
#include <stddef.h>

namespace fgrpo {

constexpr int kAttnBQ = 128;          // tokens per work-group (32 per wavefront)
constexpr int kAttnBK = 64;           // tokens of the other side per step
constexpr int kDkv3Rows = 32;         // queries of an item of the dK/dV kernel
constexpr int kAttnMaxParts = 8;      // parts of a tile at most
constexpr int kAttnDealSlots = 256;   // tiles an XCD can deal out
constexpr size_t kAttnSplitMaxBytes = 256u << 20;      // partial sums of a launch at most: a backward has two, and tables beside them

// Query heads per work-group of the query-side kernels (tile = 128 / heads tokens).  Short segments gain from short
// tiles (less masked work on the diagonal and at segment boundaries) as long as the heads of a group fill the
// work-group; long ones do not care, and a lone head per K/V head has nothing to share.
inline int attn_heads_per_group(int wanted, int G, int T, int n_seq) {      // wanted: Tuning::attn_heads
  if (wanted == 1 || wanted == 2 || wanted == 4) return wanted;
  if (G <= 1 || (long long)T >= 8192LL * n_seq) return 1;      // measured: -10..-22 % up to 2048-token segments, +1 % at 8192
  if (G % 4 == 0) return 4;
  if (G % 2 == 0) return 2;
  return G >= 3 ? 4 : 1;
}

inline int attn_query_blocks(int hb, int T, int Hq, int Hkv) {      // work-groups of an undivided launch: (tile, K/V head) units by eight, times the heads of a group
  const int rb = 128 / hb, G = Hq / Hkv;
  const long long units = (long long)((T + rb - 1) / rb) * Hkv;
  return (int)((units + 7) / 8 * 8 * ((G + hb - 1) / hb));
}

// Which 128-key tile, K/V head and piece (of kPer128 a tile is dealt in) work-group `bid` takes.  Work-groups go to the 8
// XCDs round-robin (work-group b runs on XCD b % 8, each with its own L2).  All pieces of a tile and head run on one XCD, one
// behind the other: they read the same Q and dO rows; and where the K/V heads divide eight, an XCD stays with one head.
// The units (tile, head) that no longer go round the eight are dealt to all of them piece by piece.
// With the pieces of a tile on several XCDs each row came through several L2s; dQ + dK/dV, before -> after: 32768 tokens
// in segments of 128..512, 14 / 2 heads of 64 181 -> 148 us; 36000 in 128..2048, 16 / 4 heads of 128 654 -> 639; 9000 in
// 128..1024, 28 / 4 heads 216.5 -> 213.7; 4 x 8192, 28 / 4 heads 5.70 -> 5.50 ms; 32 / 8 heads of 64 unchanged (the
// same order as before).  Runs of neighbouring tiles on one XCD (256 .. 4096 tokens) were no better, and worse where they
// disturbed the order by work; so were XCDs taken in alternating direction, which mixes the heads.
struct KeyPick {
  int rank, head, piece;       // rank: place in the launch order; negative: no work
};
constexpr KeyPick attn_key_pick(int bid, int ntile, int pieces, int Hkv) {
  const int xcd = bid & 7, slot = bid >> 3, units = ntile * Hkv, rounds = units / 8;
  int u = slot / pieces * 8 + xcd, piece = slot % pieces;
  if (slot >= rounds * pieces) {
    const int i = (slot - rounds * pieces) * 8 + xcd;
    u = rounds * 8 + i / pieces, piece = i % pieces;
    if (u >= units) return KeyPick{-1, 0, 0};
  }
  return KeyPick{u / Hkv, u % Hkv, piece};
}
inline long long attn_key_blocks(long long ntile, int pieces, int Hkv) {      // work-groups of a launch (or of one share): whole rows of eight
  const long long units = ntile * Hkv, rounds = units / 8;
  return 8 * (rounds * pieces + ((units - 8 * rounds) * pieces + 7) / 8);
}
inline int attn_keyside_keys(int D) { return D == 128 ? 64 : 32; }      // keys of a tile of the dK/dV kernel
inline int attn_keyside_blocks(int D, int T, int Hkv) { return (int)attn_key_blocks((T + 127) / 128, 128 / attn_keyside_keys(D), Hkv); }      // every 128-key tile, in pieces

// Parts of a tile of `steps` steps where a part is to walk `per`; div(n, d) is n / d of whole numbers, in the form the caller has
// at hand.
template <class Div>
constexpr int attn_parts(int steps, int parts, int per, Div div) {
  const int n = div(steps + per - 1, per), some = n > 1 ? n : 1;
  return some < parts ? some : parts;
}
// Steps a part of an XCD's tiles walks: `least`, or what shares `sum` steps (of all work-groups of the tiles) among the `deal`
// work-groups meant for them, or more until the parts, parts_with(per) of them, fit `budget` work-groups, `extra` more than tiles.
template <class Parts>
constexpr int attn_part_steps(int sum, int budget, int extra, int least, int deal, Parts parts_with) {
  int per = least;
  if (sum > per * deal) per = (sum + deal - 1) / deal;
  if (sum > per * extra) {
    const int sure = (sum + extra - 1) / extra;                // with it the parts fit: each tile rounds up by less than one
    do {
      const int n = parts_with(per);
      if (n <= budget) break;
      const int longer = (int)((long long)per * n / budget), next = longer > per + 1 ? longer : per + 1;
      per = next < sure ? next : sure;
    } while (per < sure);
  }
  return per;
}

// The merge launches read from a table how many parts a tile has and which work-group took the first; the others' lie `stride`
// behind one another, and what is read starts `skip` behind (the heads of a query tile that further work-groups take).  An entry
// is written by the work-group of the tile's first part: of a tile that an order list of the caller's leaves out it is whatever
// the workspace held.  Only an entry whose work-groups all are in the launch is followed; the sums of any other would be read
// from outside the workspace.
constexpr bool attn_parts_inside(int np, int first, int skip, int stride, int grid) {
  return np > 1 && np <= kAttnMaxParts && first >= 0 && first <= grid - 1 - skip - (np - 1) * stride;
}

// Whether the tiles of a launch are dealt to several work-groups, and to how many at most (the kernels then go by the true
// lengths, see attn_deal).  A launch of few tiles ends when its longest chain of steps does, however idle the device is;
// sharing a chain costs fp32 sums through memory and mostly one more launch.  Both sides are estimated, in us, from what was
// measured: `step` for a step of a work-group alone on its CU, half as much again where two share one, `open` steps to
// open and close a work-group.  Decided by shapes and the length that the caller gives for the longest segment; where it
// gives none, that of four or more is taken to be 1.75 means long (lengths spread evenly).  A wrong length costs time, and
// another division means another order of the fp32 sums: the results are as good, not the same bits.
// Guessed | told, forward and backward, us: 6000 tokens in 13 segments, one of 1694, 16 / 4 heads 47.2, 149 | 40.7, 114; 1500 in 2,
// one of 997, 14 / 2 heads of 64 20.3, 33.7 | 16.5, 33.2.  Where the guess is wrong because segments are equal it costs up to a fifth: forward of
// 3052 tokens in five, 16 / 4 heads, 22.9 whole and 27.7 dealt out; a guess that spares these (the mean's estimate asked too) loses
// more on uneven ones, up to 1.75 times.
// Whole | dealt out, merge launch included, 12 / 2 heads of 128: one segment of 777 tokens, forward 22.6 | 17.1 us, backward 81.4 | 37.9; of 2000
// 50.5 | 32.5 and 181 | 75.
struct SplitPlan {
  int parts = 1, per = 1;                // most parts of a tile, steps a part walks at least
  int extra = 0, deal = 1;               // see AttnParams
  int grid = 0;                          // work-groups of the launch
};
inline double shared_step(int cus, double step, int per_cu, double n) {      // step time with n work-groups in flight
  const double over = per_cu > 1 ? n / cus - 1.0 : 0.0;
  return step * (1.0 + 0.5 * (over < 0.0 ? 0.0 : over > 1.0 ? 1.0 : over));
}
// Without the mask: the tiles of a segment have equal chains.  Parts of a steps' count of their own; 4 us for the merge, 3 TB/s for the sums, written and read.
inline SplitPlan plan_even(int cus, long long wgs, int blocks, int per_cu, double chain, double step, size_t bytes_a_part) {
  SplitPlan best;
  const double slots = (double)cus * per_cu;
  auto shared = [&](double n) { return shared_step(cus, step, per_cu, n); };
  const double load = (double)wgs * chain / slots * shared(2.0 * slots);
  const double whole = chain * shared((double)wgs) > load ? chain * shared((double)wgs) : load;
  double least = 0.85 * whole;
  for (int n = 2; n <= kAttnMaxParts; ++n) {
    const int per = (int)(chain / n) + 1;
    if ((size_t)n * bytes_a_part > kAttnSplitMaxBytes || per < 2) break;
    const double x = chain / per;          // parts of a tile
    const double walk = per * shared(wgs * x);
    const double cost = (walk > load ? walk : load) + 4.0 + x * (double)bytes_a_part * 2.0 / 3.0e6;
    if (cost >= least) continue;
    least = cost;
    const int parts = (int)(2.0 * x) + 1, fit = (int)(kAttnSplitMaxBytes / bytes_a_part);
    best.parts = parts < kAttnMaxParts ? parts : kAttnMaxParts;
    if (best.parts > fit) best.parts = fit;
    best.per = per;
  }
  best.extra = blocks / 8 * (best.parts - 1), best.deal = blocks / 8 * best.parts;
  return best;
}
// Under the causal mask the tiles of a segment walk 0 .. chain steps, evenly; `sum` steps of all tiles, `longest` steps a tile could have at most.
// Either every part is in flight at once - the steps go by the work-groups the tiles leave over, of one a CU or of all - or, with about
// as many tiles as the device holds or more, the long tiles are cut to one and a half times a work-group's share, 40 steps
// at most.  A first part that waits for a CU costs more than its own steps: launches order work-groups by shader engine, so 260 parts
// on 256 CUs took 120 us where 250 took 100 (dK/dV of 3000 tokens in 4 segments, 12 / 2 heads of 128).  Sums are taken at 6 TB/s, most
// of them leaving while others still walk; a part is no shorter than its own are worth at 3 (`worth` times, `at_most`: measured at
// 2 .. 12 steps).  dK/dV whole | dealt out, dQ and
// merge included: 6000 tokens in 13 segments, 16 / 4 heads 149 | 114; 4000 in 6, 28 / 4 heads 139 | 119; 5000 in one, 28 / 4
// heads 663 | 620; 12345 in 23, 14 / 2 heads of 64 87 | 94 and 4000 in 5, 32 / 8 heads of 64 83 | 96, both refused.
// A launch of more than one round of tiles ends with its longest tile or with its load, and dealing out takes off only what that tile
// walks beyond the load; the more rounds, the less of it the tiles in their order leave.  So the longest has to be
// 1 + `rounds` * (rounds of tiles) times the load (key side; on the query side the estimate holds).  dQ + dK/dV whole | dealt out: one segment of 7359 tokens,
// 28 / 4 heads 1183 | 1272, of 15330, 12 / 2 heads 2107 | 2288; 28241 in 14, 14 / 2 heads of 64 721 | 790, all three 1.1 to 1.3 times.  Over 2177
// launches of one to three rounds dealing out was worth it from 1.5 times the load on at 1.75 rounds, 1.75 at 3 (head dimension 64: 1.75 and 2.3);
// by this line they take 0.6 % longer than with the better of both each, all whole 2.6 %, all dealt out 2.4.
inline SplitPlan plan_uneven(int cus, long long wgs, int blocks, int per_cu, double chain, double sum, double longest, double step, double open, double bytes_a_part, double worth, double at_most, double merge, double rounds) {
  SplitPlan s;
  const double slots = (double)cus * per_cu, load = sum / slots;
  auto shared = [&](double n) { return shared_step(cus, step, per_cu, n); };
  auto most = [](double a, double b) { return a > b ? a : b; };
  // more tiles than CUs, one a CU: 1.15 to 1.25 of what the longest tile or the load comes to, for the order by shader engine
  // (dK/dV of 6000 tokens in 12 segments, 28 / 4 heads 99 us, of 9000 in 14 173; both dealt out, with dQ, 152 -> 140 and 276 -> 270)
  const double whole = most((chain + open) * shared((double)wgs), (sum + wgs * open) / slots * shared(2.0 * slots)) * (per_cu == 1 && wgs > slots ? 1.15 : 1.0);
  const double sums = bytes_a_part * 2.0 / 3.0e6, even = worth * sqrt(sum * sums / step), least = floor(most(even < at_most ? even : at_most, 1.5) + 0.5);
  const double cap = most(least, chain / kAttnMaxParts);
  auto parts = [&](double per) { return per < chain ? sum / per + 0.5 * wgs : (double)wgs; };
  double per = most(1.5 * load < 40.0 ? 1.5 * load : 40.0, cap), room = 0.0;
  const double spare = 1.0 - wgs / slots;
  double walk = (load + parts(per) * open / slots + 0.5 * per + (spare < 0.0 ? 0.0 : spare < 0.25 ? 8.0 * spare : 2.0) * open) * shared(2.0 * slots);
  for (double r = cus; r <= slots; r += cus) {
    if (wgs >= r) continue;
    const double x = most(most(sum / (r - 0.5 * wgs), chain * (2.0 - r / wgs)), cap), t = (x + open) * shared(parts(x));
    if (t < walk) walk = t, per = x, room = r;
  }
  if (walk + merge + most(parts(per) - 0.5 * wgs, 0.0) * sums * 0.5 >= whole) return s;
  if (room == 0.0 && wgs > slots && chain < load * (1.0 + rounds * wgs / slots)) return s;
  s.per = (int)least;
  s.extra = room > 0.0 ? ((int)room - blocks) / 8 : (int)(load / per * slots / 8) + 1;
  s.deal = room > 0.0 ? ((int)room - blocks / 2) / 8 : s.extra;
  const int ways = (int)(longest / least) + 1, bound = blocks / 8 * ((ways < kAttnMaxParts ? ways : kAttnMaxParts) - 1);
  if (s.extra > bound) s.extra = bound;
  if (s.extra >= 1 && (blocks + 8 * s.extra) * bytes_a_part <= kAttnSplitMaxBytes) s.parts = kAttnMaxParts;
  return s;
}
// queries or keys that a token's segment has, and the longest segment
struct SegmentGuess {
  double longest, seen;
};
inline SegmentGuess guess_segments(int T, int n_seq, int max_len) {
  const double mean = (double)T / n_seq;
  if (n_seq == 1 || (max_len <= 0 && n_seq < 4)) return SegmentGuess{mean, mean};
  double longest = max_len > 0 ? max_len : 1.75 * mean;
  longest = longest < mean ? mean : longest > T ? T : longest;
  const double rest = T - longest;
  return SegmentGuess{longest, (longest * longest + rest * rest / (n_seq - 1)) / T};
}
inline SplitPlan plan_query_split(int cus, int heads, int form, int T, int n_seq, int max_len, int Hq, int Hkv, int D, int causal, bool forward, bool merged) {
  if (form == 1 || (!forward && form == 3)) return SplitPlan();
  const int hb = attn_heads_per_group(heads, Hq / Hkv, T, n_seq), rb = 128 / hb, nb = (Hq / Hkv + hb - 1) / hb;
  const int blocks = attn_query_blocks(hb, T, Hq, Hkv);
  const long long wgs = (long long)((T + rb - 1) / rb) * Hkv * nb;
  if (blocks / nb > 8 * kAttnDealSlots) return SplitPlan();
  const double step = D == 128 ? 1.6 : forward ? 1.15 : 1.3;
  SplitPlan s;
  if (!causal) {
    s = plan_even(cus, wgs, blocks, 2, (double)T / n_seq / kAttnBK, step, (size_t)T * Hq * (D * 4 + (forward ? 8 : 0)));
  } else {
    const SegmentGuess g = guess_segments(T, n_seq, max_len);
    const double sum = wgs * (g.seen * 0.5 + 32 + (n_seq > 1 ? rb : 0)) / kAttnBK;      // steps begun; tiles that reach into the next segment
    s = plan_uneven(cus, wgs, blocks, 2, g.longest / kAttnBK, sum, (double)T / kAttnBK, step, 1.5, 128.0 * D * 4, 1.35, 7.0, merged ? 0.5 : 4.0, 0.0);
  }
  s.grid = blocks + 8 * s.extra;
  return s;
}
inline SplitPlan plan_key_split(int cus, int form, int T, int n_seq, int max_len, int Hq, int Hkv, int D, int causal) {
  if (form == 1 || form == 2) return SplitPlan();
  const int keys = attn_keyside_keys(D), blocks = attn_keyside_blocks(D, T, Hkv), per_cu = D == 128 ? 1 : 2;
  const long long wgs = (long long)((T + keys - 1) / keys) * Hkv;
  if (blocks > 8 * kAttnDealSlots) return SplitPlan();
  const double items = (Hq / Hkv) / 4.0 / 32;           // of one of the four wavefronts, a token
  SplitPlan s;
  if (!causal) {
    s = plan_even(cus, wgs, blocks, per_cu, (double)T / n_seq * items, D == 128 ? 1.3 : 0.65, (size_t)T * Hkv * D * 8);
  } else {
    const SegmentGuess g = guess_segments(T, n_seq, max_len);
    const double sum = wgs * (g.seen * 0.5 + 16 + (n_seq > 1 ? keys : 0)) * items;
    s = plan_uneven(cus, wgs, blocks, per_cu, g.longest * items, sum, T * items, D == 128 ? 1.4 : 0.65, D == 128 ? 6.0 : 4.0, keys * D * 8.0, 1.0, 1e30, 4.0, D == 128 ? 0.25 : 0.45);
  }
  s.grid = blocks + 8 * s.extra;
  return s;
}
inline size_t align256(size_t n) { return (n + 255) / 256 * 256; }
inline size_t query_sums_bytes(const SplitPlan& s, int D) { return align256((size_t)s.grid * 128 * D * 4); }
inline size_t query_info_bytes(int T, int Hkv) { return align256((size_t)((T + 31) / 32) * Hkv * 8); }
inline size_t query_split_bytes(const SplitPlan& s, int T, int Hkv, int D, bool forward) {
  return s.parts <= 1 ? 0 : query_sums_bytes(s, D) + query_info_bytes(T, Hkv) + (forward ? align256((size_t)s.grid * 128 * 8) : 0);
}
inline size_t key_sums_bytes(const SplitPlan& s, int D) { return align256((size_t)s.grid * attn_keyside_keys(D) * D * 8); }
inline size_t key_split_bytes(const SplitPlan& s, int T, int Hkv, int D) {
  const int keys = attn_keyside_keys(D);
  return s.parts <= 1 ? 0 : key_sums_bytes(s, D) + align256((size_t)((T + keys - 1) / keys) * Hkv * 8);
}

}  // namespace fgrpo
