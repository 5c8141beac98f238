// Packed variable-length attention: C entry points, argument checks and launches (kernels in attn_kernels.h).
#include <math.h>
#include <string.h>

#include "host_common.h"
#include "attn_kernels.h"
#include "attn_route.h"

using namespace fgrpo;

namespace fgrpo {
constexpr size_t kAttnSplitMaxBytes = 256u << 20;
int launch_attn_dkv3(int D, const AttnParams& p, hipStream_t st);      // launch_attn_keyside.hip
int attn_keyside_keys(int D);
int attn_keyside_blocks(int D, int T, int Hkv);
int launch_attn_merge_bwd(int D, const AttnParams& p, int rb, hipStream_t st);
}

namespace {
// Query heads per work-group of the query-side kernels (tile = 128 / heads tokens).  Short segments gain from short
// tiles (less masked work on the diagonal and at segment boundaries) as long as the heads of a group fill the
// work-group; long ones do not care, and a lone head per K/V head has nothing to share.
int attn_heads_per_group(const Tuning& tn, int G, int T, int n_seq) {
  if (tn.attn_heads == 1 || tn.attn_heads == 2 || tn.attn_heads == 4) return tn.attn_heads;
  if (G <= 1 || (long long)T >= 8192LL * n_seq) return 1;      // measured: -10..-22 % up to 2048-token segments, +1 % at 8192
  if (G % 4 == 0) return 4;
  if (G % 2 == 0) return 2;
  return G >= 3 ? 4 : 1;
}

int attn_query_blocks(int hb, int T, int Hq, int Hkv) {                      // work-groups of an undivided launch: (tile, K/V head) units by eight, times the heads of a group
  const int rb = 128 / hb, G = Hq / Hkv;
  const long long units = (long long)((T + rb - 1) / rb) * Hkv;
  return (int)((units + 7) / 8 * 8 * ((G + hb - 1) / hb));
}

template <template <int, int> class Launcher>
int launch_query_side(int form, int D, int hb, AttnParams& p, int T, int Hq, int Hkv, int32_t* bounds_ws, hipStream_t st) {
  p.order_q = bounds_ws + attn_order_offset(T, hb == 1 ? 1 : hb == 2 ? 2 : 3);
  p.blocks_q = attn_query_blocks(hb, T, Hq, Hkv);
  const dim3 grid((unsigned)(p.blocks_q + (p.parts_q > 1 ? 8 * p.extra_q : 0)));
  if (D == 128) {
    if (hb == 1) Launcher<128, 1>::run(form, grid, st, p);
    else if (hb == 2) Launcher<128, 2>::run(form, grid, st, p);
    else Launcher<128, 4>::run(form, grid, st, p);
  } else {
    if (hb == 1) Launcher<64, 1>::run(form, grid, st, p);
    else if (hb == 2) Launcher<64, 2>::run(form, grid, st, p);
    else Launcher<64, 4>::run(form, grid, st, p);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}
template <int HD, int HB>
struct FwdLauncher {
  static void run(int form, dim3 grid, hipStream_t st, const AttnParams& p) {
    if (form == 1) hipLaunchKernelGGL((varlen_attn_fwd_kernel<HD, HB>), grid, dim3(256), 0, st, p);
    else if (p.parts_q > 1) hipLaunchKernelGGL((varlen_attn_fwd2_kernel<HD, HB, true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((varlen_attn_fwd2_kernel<HD, HB>), grid, dim3(256), 0, st, p);
  }
};
template <int HD, int HB>
struct DqLauncher {
  static void run(int form, dim3 grid, hipStream_t st, const AttnParams& p) {
    if (form == 1 || form == 3) hipLaunchKernelGGL((varlen_attn_dq_kernel<HD, HB>), grid, dim3(256), 0, st, p);
    else if (p.parts_q > 1) hipLaunchKernelGGL((varlen_attn_dq2_kernel<HD, HB, true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((varlen_attn_dq2_kernel<HD, HB>), grid, dim3(256), 0, st, p);
  }
};
// Whether the tiles of a launch are dealt to several work-groups, and to how many at most (the kernels then go by the true
// lengths, see attn_deal).  A launch of few tiles ends when its longest chain of steps does, however idle the device is;
// sharing a chain costs fp32 sums through memory and mostly one more launch.  Both sides are estimated, in us, from what was
// measured: `step` for a step of a work-group alone on its CU, half as much again where two share one, `open` steps to
// open and close a work-group.  Decided by shapes and the length that the caller gives for the longest segment; where it
// gives none, that of four or more is taken to be 1.75 means long (lengths spread evenly).  A wrong length costs time, nothing else.
// Guessed | told, forward and backward, us: 6000 tokens in 13 segments, one of 1694, 16 / 4 heads 47.1, 148 | 39.7, 115; 1500 in 2,
// one of 997, 14 / 2 heads of 64 20.1, 33.1 | 16.2, 32.8; 2000 in 3, one of 970, 12 / 2 heads 27.1, 57.5 | 23.3, 53.5.  Whole | dealt out, merge launch included, 12 / 2 heads of 128: one segment of 777
// tokens, forward 22.5 | 16.5 us, backward 77.8 | 36.7; of 2000 50.0 | 31.8 and 147 | 74.
struct SplitPlan {
  int parts = 1, per = 1;                // most parts of a tile, steps a part walks at least
  int extra = 0, deal = 1;               // see AttnParams
  int grid = 0;                          // work-groups of the launch
};
double shared_step(double step, int per_cu, double n) {      // step time with n work-groups in flight
  const double over = per_cu > 1 ? n / num_cus() - 1.0 : 0.0;
  return step * (1.0 + 0.5 * (over < 0.0 ? 0.0 : over > 1.0 ? 1.0 : over));
}
// Without the mask: the tiles of a segment have equal chains.  Parts of a steps' count of their own; 4 us for the merge, 3 TB/s for the sums, written and read.
SplitPlan plan_even(long long wgs, int blocks, int per_cu, double chain, double step, size_t bytes_a_part) {
  SplitPlan best;
  const double slots = (double)num_cus() * per_cu;
  auto shared = [&](double n) { return shared_step(step, per_cu, n); };
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
// merge included: 6000 tokens in 13 segments, 16 / 4 heads 150 | 123; 4000 in 6, 28 / 4 heads 124 | 115; 5000 in one, 28 / 4
// heads 645 | 609; 12345 in 23, 14 / 2 heads of 64 87 | 94 and 4000 in 5, 32 / 8 heads of 64 83 | 96, both refused.
SplitPlan plan_uneven(long long wgs, int blocks, int per_cu, double chain, double sum, double longest, double step, double open, double bytes_a_part, double worth, double at_most, double merge) {
  SplitPlan s;
  const double cus = num_cus(), slots = cus * per_cu, load = sum / slots;
  auto shared = [&](double n) { return shared_step(step, per_cu, n); };
  auto most = [](double a, double b) { return a > b ? a : b; };
  // more tiles than CUs, one a CU: 1.15 to 1.25 of what the longest tile or the load comes to, for the order by shader engine
  // (dK/dV of 6000 tokens in 12 segments, 28 / 4 heads 99 us, of 9000 in 14 173; both dealt out, with dQ, 154 -> 139 and 270 -> 267)
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
SegmentGuess guess_segments(int T, int n_seq, int max_len) {
  const double mean = (double)T / n_seq;
  if (n_seq == 1 || (max_len <= 0 && n_seq < 4)) return SegmentGuess{mean, mean};
  double longest = max_len > 0 ? max_len : 1.75 * mean;
  longest = longest < mean ? mean : longest > T ? T : longest;
  const double rest = T - longest;
  return SegmentGuess{longest, (longest * longest + rest * rest / (n_seq - 1)) / T};
}
SplitPlan plan_query_split(const Tuning& tn, int form, int T, int n_seq, int max_len, int Hq, int Hkv, int D, int causal, bool forward, bool merged) {
  if (form == 1 || (!forward && form == 3)) return SplitPlan();
  const int hb = attn_heads_per_group(tn, Hq / Hkv, T, n_seq), rb = 128 / hb, nb = (Hq / Hkv + hb - 1) / hb;
  const int blocks = attn_query_blocks(hb, T, Hq, Hkv);
  const long long wgs = (long long)((T + rb - 1) / rb) * Hkv * nb;
  if (blocks / nb > 8 * kAttnDealSlots) return SplitPlan();
  const double step = D == 128 ? 1.6 : forward ? 1.15 : 1.3;
  SplitPlan s;
  if (!causal) {
    s = plan_even(wgs, blocks, 2, (double)T / n_seq / kAttnBK, step, (size_t)T * Hq * (D * 4 + (forward ? 8 : 0)));
  } else {
    const SegmentGuess g = guess_segments(T, n_seq, max_len);
    const double sum = wgs * (g.seen * 0.5 + 32 + (n_seq > 1 ? rb : 0)) / kAttnBK;      // steps begun; tiles that reach into the next segment
    s = plan_uneven(wgs, blocks, 2, g.longest / kAttnBK, sum, (double)T / kAttnBK, step, 1.5, 128.0 * D * 4, 1.35, 7.0, merged ? 0.5 : 4.0);
  }
  s.grid = blocks + 8 * s.extra;
  return s;
}
SplitPlan plan_key_split(int form, int T, int n_seq, int max_len, int Hq, int Hkv, int D, int causal) {
  if (form == 1 || form == 2) return SplitPlan();
  const int keys = attn_keyside_keys(D), blocks = attn_keyside_blocks(D, T, Hkv), per_cu = D == 128 ? 1 : 2;
  const long long wgs = (long long)((T + keys - 1) / keys) * Hkv;
  if (blocks > 8 * kAttnDealSlots) return SplitPlan();
  const double items = (Hq / Hkv) / 4.0 / 32;           // of one of the four wavefronts, a token
  SplitPlan s;
  if (!causal) {
    s = plan_even(wgs, blocks, per_cu, (double)T / n_seq * items, D == 128 ? 1.3 : 0.65, (size_t)T * Hkv * D * 8);
  } else {
    const SegmentGuess g = guess_segments(T, n_seq, max_len);
    const double sum = wgs * (g.seen * 0.5 + 16 + (n_seq > 1 ? keys : 0)) * items;
    s = plan_uneven(wgs, blocks, per_cu, g.longest * items, sum, T * items, D == 128 ? 1.4 : 0.65, D == 128 ? 6.0 : 4.0, keys * D * 8.0, 1.0, 1e30, 4.0);
  }
  s.grid = blocks + 8 * s.extra;
  return s;
}
size_t align256(size_t n) { return (n + 255) / 256 * 256; }
size_t query_sums_bytes(const SplitPlan& s, int D) { return align256((size_t)s.grid * 128 * D * 4); }
size_t query_info_bytes(int T, int Hkv) { return align256((size_t)((T + 31) / 32) * Hkv * sizeof(int2)); }
size_t query_split_bytes(const SplitPlan& s, int T, int Hkv, int D, bool forward) {
  return s.parts <= 1 ? 0 : query_sums_bytes(s, D) + query_info_bytes(T, Hkv) + (forward ? align256((size_t)s.grid * 128 * sizeof(float2)) : 0);
}
size_t key_sums_bytes(const SplitPlan& s, int D) { return align256((size_t)s.grid * attn_keyside_keys(D) * D * 8); }
size_t key_split_bytes(const SplitPlan& s, int T, int Hkv, int D) {
  const int keys = attn_keyside_keys(D);
  return s.parts <= 1 ? 0 : key_sums_bytes(s, D) + align256((size_t)((T + keys - 1) / keys) * Hkv * sizeof(int2));
}
}  // namespace

extern "C" {

// ---- packed variable-length attention ------------------------------------------------------------------
namespace {
int check_attn(const char* who, const void* q, const void* k, const void* v, long long q_st, long long q_sh,
               long long k_st, long long k_sh, long long v_st, long long v_sh, const int32_t* cu, int n_seq, int T,
               int Hq, int Hkv, int D, float scale, const int32_t* bounds_ws) {
  if (!q || !k || !v || !cu || !bounds_ws) return fail(FGRPO_ERR_BAD_ARG, "%s: null argument", who);
  if (T <= 0 || n_seq <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0)
    return fail(FGRPO_ERR_BAD_ARG, "%s: T=%d n_seq=%d Hq=%d Hkv=%d", who, T, n_seq, Hq, Hkv);
  if (D != 128 && D != 64) return fail(FGRPO_ERR_BAD_ARG, "%s: head dimension %d not supported (128 or 64)", who, D);
  if (!(scale > 0.f)) return fail(FGRPO_ERR_BAD_ARG, "%s: softmax scale must be positive", who);
  if (!aligned16(q) || !aligned16(k) || !aligned16(v)) return fail(FGRPO_ERR_ALIGN, "%s: q/k/v must be 16-byte aligned", who);
  const long long st[6] = {q_st, q_sh, k_st, k_sh, v_st, v_sh};
  for (int i = 0; i < 6; ++i)
    if (st[i] <= 0 || st[i] % 8 != 0) return fail(FGRPO_ERR_ALIGN, "%s: strides must be positive multiples of 8 elements", who);
  return 0;
}

void fill_attn(AttnParams& p, const void* q, const void* k, const void* v, long long q_st, long long q_sh,
               long long k_st, long long k_sh, long long v_st, long long v_sh, int T, int Hq, int Hkv, float scale,
               int causal, int32_t* bounds_ws) {
  memset(&p, 0, sizeof(p));
  p.q = (const bf16_t*)q;
  p.k = (const bf16_t*)k;
  p.v = (const bf16_t*)v;
  p.q_st = q_st, p.q_sh = q_sh, p.k_st = k_st, p.k_sh = k_sh, p.v_st = v_st, p.v_sh = v_sh;
  p.seg_start = bounds_ws;
  p.seg_end = bounds_ws + T;
  p.order_k = bounds_ws + attn_order_offset(T, 0);
  p.order_q = bounds_ws + attn_order_offset(T, 1);      // the query-side launches pick the list of their tile size
  p.T = T, p.Hq = Hq, p.Hkv = Hkv;
  p.scale = scale;
  p.causal = causal != 0;
}
}  // namespace

int fgrpo_varlen_attn_bounds(const int32_t* cu, int n_seq, int T, int causal, int32_t* bounds_ws, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  if (!cu || !bounds_ws || T <= 0 || n_seq <= 0) return fail(FGRPO_ERR_BAD_ARG, "varlen_attn_bounds: bad argument");
  hipLaunchKernelGGL(segment_bounds_kernel, dim3((T + 255) / 256), dim3(256), 0, st, cu, n_seq, T, bounds_ws, bounds_ws + T);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(attn_tile_order_kernel, dim3(4, kAttnOrderSlices), dim3(1024), 0, st, bounds_ws, bounds_ws + T, T, causal != 0, bounds_ws);
  HIP_TRY(hipGetLastError());
  return 0;
}

size_t fgrpo_varlen_attn_workspace(int T, int n_seq, int Hq, int Hkv, int D, int causal, int backward) {
  return fgrpo_varlen_attn_workspace_len(T, n_seq, 0, Hq, Hkv, D, causal, backward);
}

size_t fgrpo_varlen_attn_workspace_len(int T, int n_seq, int max_len, int Hq, int Hkv, int D, int causal, int backward) {
  if (T <= 0 || n_seq <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || (D != 128 && D != 64)) return 0;
  const Tuning tn = g_tune;
  const SplitPlan sk = backward ? plan_key_split(tn.attn_dkv, T, n_seq, max_len, Hq, Hkv, D, causal) : SplitPlan();
  const SplitPlan sq = plan_query_split(tn, tn.attn_qside, T, n_seq, max_len, Hq, Hkv, D, causal, !backward, sk.parts > 1);
  return query_split_bytes(sq, T, Hkv, D, !backward) + key_split_bytes(sk, T, Hkv, D);
}

int fgrpo_varlen_attn_fwd(const void* q, const void* k, const void* v, long long q_st, long long q_sh, long long k_st,
                          long long k_sh, long long v_st, long long v_sh, const int32_t* cu, int n_seq, int T, int Hq,
                          int Hkv, int D, float scale, int causal, void* out, float* lse, int32_t* bounds_ws,
                          int bounds_valid, void* stream) {
  return fgrpo_varlen_attn_fwd_ws(q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, T, Hq, Hkv, D, scale, causal, out,
                                  lse, bounds_ws, bounds_valid, nullptr, 0, stream);
}

int fgrpo_varlen_attn_fwd_ws(const void* q, const void* k, const void* v, long long q_st, long long q_sh, long long k_st,
                          long long k_sh, long long v_st, long long v_sh, const int32_t* cu, int n_seq, int T, int Hq,
                          int Hkv, int D, float scale, int causal, void* out, float* lse, int32_t* bounds_ws,
                          int bounds_valid, void* ws, size_t ws_bytes, void* stream) {
  return fgrpo_varlen_attn_fwd_len(q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, 0, T, Hq, Hkv, D, scale, causal, out,
                                   lse, bounds_ws, bounds_valid, ws, ws_bytes, stream);
}

int fgrpo_varlen_attn_fwd_len(const void* q, const void* k, const void* v, long long q_st, long long q_sh, long long k_st,
                          long long k_sh, long long v_st, long long v_sh, const int32_t* cu, int n_seq, int max_len, int T, int Hq,
                          int Hkv, int D, float scale, int causal, void* out, float* lse, int32_t* bounds_ws,
                          int bounds_valid, void* ws, size_t ws_bytes, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  int rc = check_attn("varlen_attn_fwd", q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, T, Hq, Hkv, D, scale, bounds_ws);
  if (rc) return rc;
  if (!out || !lse) return fail(FGRPO_ERR_BAD_ARG, "varlen_attn_fwd: null output");
  if (!aligned16(out)) return fail(FGRPO_ERR_ALIGN, "varlen_attn_fwd: out must be 16-byte aligned");
  AttnParams p;
  fill_attn(p, q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, T, Hq, Hkv, scale, causal, bounds_ws);
  p.out = (bf16_t*)out;
  p.lse = lse;
  if (!bounds_valid) {   // else bounds_ws still holds what an earlier call with the same segments wrote
    rc = fgrpo_varlen_attn_bounds(cu, n_seq, T, causal, bounds_ws, stream);
    if (rc) return rc;
  }
  const Tuning tn = g_tune;   // one reading of the tuning state per call: the kernel launched is the one the split was planned for
  const int form = attn_query_form(tn.attn_qside, q_st, k_st, v_st, Hq, D), hb = attn_heads_per_group(tn, Hq / Hkv, T, n_seq);
  SplitPlan sp = plan_query_split(tn, form, T, n_seq, max_len, Hq, Hkv, D, causal, true, false);
  const size_t need = query_split_bytes(sp, T, Hkv, D, true);
  if (!ws || need == 0) sp = SplitPlan();
  else if (ws_bytes < need) return fail(FGRPO_ERR_WORKSPACE, "varlen_attn_fwd: workspace %zu < %zu", ws_bytes, need);
  else if (!aligned16(ws)) return fail(FGRPO_ERR_ALIGN, "varlen_attn_fwd: workspace must be 16-byte aligned");
  p.parts_q = sp.parts, p.per_q = sp.per, p.extra_q = sp.extra, p.deal_q = sp.deal;
  p.part_q = (float*)ws;
  p.query_info = (int2*)((char*)ws + query_sums_bytes(sp, D));
  p.part_ml = (float2*)((char*)ws + query_sums_bytes(sp, D) + query_info_bytes(T, Hkv));
  rc = launch_query_side<FwdLauncher>(form, D, hb, p, T, Hq, Hkv, bounds_ws, st);
  if (rc || sp.parts <= 1) return rc;
  const unsigned blocks = (unsigned)((T + 31) / 32) * (unsigned)Hq;
  if (D == 128) hipLaunchKernelGGL(attn_merge_fwd_kernel<128>, dim3(blocks), dim3(256), 0, st, p, 128 / hb);
  else hipLaunchKernelGGL(attn_merge_fwd_kernel<64>, dim3(blocks), dim3(256), 0, st, p, 128 / hb);
  HIP_TRY(hipGetLastError());
  return 0;
}

int fgrpo_varlen_attn_bwd(const void* dout, const void* q, const void* k, const void* v, const void* out, const float* lse,
                          long long q_st, long long q_sh, long long k_st, long long k_sh, long long v_st, long long v_sh,
                          const int32_t* cu, int n_seq, int T, int Hq, int Hkv, int D, float scale, int causal, void* dq,
                          void* dk, void* dv, float* delta_ws, int32_t* bounds_ws, int bounds_valid, void* stream) {
  return fgrpo_varlen_attn_bwd_ws(dout, q, k, v, out, lse, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, T, Hq, Hkv, D, scale, causal, dq, dk, dv, delta_ws,
                                  bounds_ws, bounds_valid, nullptr, 0, stream);
}

int fgrpo_varlen_attn_bwd_ws(const void* dout, const void* q, const void* k, const void* v, const void* out, const float* lse,
                          long long q_st, long long q_sh, long long k_st, long long k_sh, long long v_st, long long v_sh,
                          const int32_t* cu, int n_seq, int T, int Hq, int Hkv, int D, float scale, int causal, void* dq,
                          void* dk, void* dv, float* delta_ws, int32_t* bounds_ws, int bounds_valid, void* ws,
                             size_t ws_bytes, void* stream) {
  return fgrpo_varlen_attn_bwd_len(dout, q, k, v, out, lse, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, 0, T, Hq, Hkv, D, scale, causal, dq, dk,
                                   dv, delta_ws, bounds_ws, bounds_valid, ws, ws_bytes, stream);
}

int fgrpo_varlen_attn_bwd_len(const void* dout, const void* q, const void* k, const void* v, const void* out, const float* lse,
                          long long q_st, long long q_sh, long long k_st, long long k_sh, long long v_st, long long v_sh,
                          const int32_t* cu, int n_seq, int max_len, int T, int Hq, int Hkv, int D, float scale, int causal, void* dq,
                          void* dk, void* dv, float* delta_ws, int32_t* bounds_ws, int bounds_valid, void* ws,
                             size_t ws_bytes, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  int rc = check_attn("varlen_attn_bwd", q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu, n_seq, T, Hq, Hkv, D, scale, bounds_ws);
  if (rc) return rc;
  if (!dout || !out || !lse || !dq || !dk || !dv || !delta_ws) return fail(FGRPO_ERR_BAD_ARG, "varlen_attn_bwd: null argument");
  if (!aligned16(dout) || !aligned16(out) || !aligned16(dq) || !aligned16(dk) || !aligned16(dv))
    return fail(FGRPO_ERR_ALIGN, "varlen_attn_bwd: dout/out/dq/dk/dv must be 16-byte aligned");
  AttnParams p;
  fill_attn(p, q, k, v, q_st, q_sh, k_st, k_sh, v_st, v_sh, T, Hq, Hkv, scale, causal, bounds_ws);
  p.lse = const_cast<float*>(lse);
  p.dout = (const bf16_t*)dout;
  p.delta = delta_ws;
  p.out_fwd = (const bf16_t*)out;
  p.dq = (bf16_t*)dq;
  p.dk = (bf16_t*)dk;
  p.dv = (bf16_t*)dv;
  if (!bounds_valid) {   // else bounds_ws still holds what an earlier call with the same segments wrote
    rc = fgrpo_varlen_attn_bounds(cu, n_seq, T, causal, bounds_ws, stream);
    if (rc) return rc;
  }
  const Tuning tn = g_tune;   // one reading of the tuning state per call: the kernel launched is the one the split was planned for
  const int form = attn_query_form(tn.attn_qside, q_st, k_st, v_st, Hq, D), hb = attn_heads_per_group(tn, Hq / Hkv, T, n_seq);
  const int key_form = attn_key_form(tn.attn_dkv, q_st, k_st, v_st, T, Hq, Hkv, D, attn_keyside_keys(D));
  SplitPlan sk = plan_key_split(key_form, T, n_seq, max_len, Hq, Hkv, D, causal), sq = plan_query_split(tn, form, T, n_seq, max_len, Hq, Hkv, D, causal, false, sk.parts > 1);
  const size_t need_q = query_split_bytes(sq, T, Hkv, D, false), need = need_q + key_split_bytes(sk, T, Hkv, D);
  if (!ws || need == 0) sq = sk = SplitPlan();
  else if (ws_bytes < need) return fail(FGRPO_ERR_WORKSPACE, "varlen_attn_bwd: workspace %zu < %zu", ws_bytes, need);
  else if (!aligned16(ws)) return fail(FGRPO_ERR_ALIGN, "varlen_attn_bwd: workspace must be 16-byte aligned");
  if (key_form != 3) sq = sk = SplitPlan();
  p.parts_q = sq.parts, p.per_q = sq.per, p.extra_q = sq.extra, p.deal_q = sq.deal;
  p.parts_k = sk.parts, p.per_k = sk.per, p.extra_k = sk.extra, p.deal_k = sk.deal;
  p.part_q = (float*)ws;
  p.query_info = (int2*)((char*)ws + query_sums_bytes(sq, D));
  p.part_k = (float*)((char*)ws + need_q);
  p.key_info = (int2*)((char*)ws + need_q + key_sums_bytes(sk, D));
  rc = launch_query_side<DqLauncher>(form, D, hb, p, T, Hq, Hkv, bounds_ws, st);
  if (rc) return rc;
  if (key_form == 3) {
    rc = launch_attn_dkv3(D, p, st);
    if (rc || (sq.parts <= 1 && sk.parts <= 1)) return rc;
    return launch_attn_merge_bwd(D, p, 128 / hb, st);
  }
  const dim3 grid_k(Hkv, (T + kAttnBQ - 1) / kAttnBQ);
  if (key_form == 1) {
    if (D == 128) hipLaunchKernelGGL(varlen_attn_dkv_kernel<128>, grid_k, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(varlen_attn_dkv_kernel<64>, grid_k, dim3(256), 0, st, p);
  } else if (D == 128) {
    rc = raise_lds<varlen_attn_dkv2_kernel<128>>(kAttnDkv2Lds<128>);
    if (rc) return rc;
    hipLaunchKernelGGL(varlen_attn_dkv2_kernel<128>, grid_k, dim3(512), kAttnDkv2Lds<128>, st, p);
  } else {
    rc = raise_lds<varlen_attn_dkv2_kernel<64>>(kAttnDkv2Lds<64>);
    if (rc) return rc;
    hipLaunchKernelGGL(varlen_attn_dkv2_kernel<64>, grid_k, dim3(512), kAttnDkv2Lds<64>, st, p);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

}  // extern "C"
