// Packed variable-length attention: C entry points, argument checks and launches (kernels in attn_kernels.h).
#include <string.h>

#include "host_common.h"
#include "attn_kernels.h"
#include "attn_route.h"

using namespace fgrpo;

namespace fgrpo {
int launch_attn_dkv3(int D, const AttnParams& p, hipStream_t st);      // launch_attn_keyside.hip
int launch_attn_merge_bwd(int D, const AttnParams& p, int rb, hipStream_t st);
}

namespace {
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
  const SplitPlan sk = backward ? plan_key_split(num_cus(), tn.attn_dkv, T, n_seq, max_len, Hq, Hkv, D, causal) : SplitPlan();
  const SplitPlan sq = plan_query_split(num_cus(), tn.attn_heads, tn.attn_qside, T, n_seq, max_len, Hq, Hkv, D, causal, !backward, sk.parts > 1);
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
  const int form = attn_query_form(tn.attn_qside, q_st, k_st, v_st, Hq, D), hb = attn_heads_per_group(tn.attn_heads, Hq / Hkv, T, n_seq);
  SplitPlan sp = plan_query_split(num_cus(), tn.attn_heads, form, T, n_seq, max_len, Hq, Hkv, D, causal, true, false);
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
  const int form = attn_query_form(tn.attn_qside, q_st, k_st, v_st, Hq, D), hb = attn_heads_per_group(tn.attn_heads, Hq / Hkv, T, n_seq);
  const int key_form = attn_key_form(tn.attn_dkv, q_st, k_st, v_st, T, Hq, Hkv, D, attn_keyside_keys(D));
  SplitPlan sk = plan_key_split(num_cus(), key_form, T, n_seq, max_len, Hq, Hkv, D, causal), sq = plan_query_split(num_cus(), tn.attn_heads, form, T, n_seq, max_len, Hq, Hkv, D, causal, false, sk.parts > 1);
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
