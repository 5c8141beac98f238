// Key-side attention backward, barrier-free form (attn_keyside.h): a translation unit of its own, compiled so that the
// matrix instructions the compiler schedules keep their results in ordinary vector registers.
#include "host_common.h"
#include "attn_keyside.h"

namespace fgrpo {

template <int HD, int KB>
static int launch(const AttnParams& p, hipStream_t st) {
  AttnParams a = p;
  a.blocks_k = attn_keyside_blocks(HD, p.T, p.Hkv);
  if (p.parts_k > 1) {
    const int rc = raise_lds<varlen_attn_dkv3_kernel<HD, KB, true>>(kDkv3Lds<HD, KB>);
    if (rc) return rc;
    hipLaunchKernelGGL((varlen_attn_dkv3_kernel<HD, KB, true>), dim3((unsigned)(a.blocks_k + 8 * p.extra_k)), dim3(256), (kDkv3Lds<HD, KB>), st, a);
  } else {
    const int rc = raise_lds<varlen_attn_dkv3_kernel<HD, KB, false>>(kDkv3Lds<HD, KB>);
    if (rc) return rc;
    hipLaunchKernelGGL((varlen_attn_dkv3_kernel<HD, KB, false>), dim3((unsigned)a.blocks_k), dim3(256), (kDkv3Lds<HD, KB>), st, a);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Head dimension 128 takes two key blocks a wavefront (its accumulators fill the file either way, and a fragment
// serves two products); 64 takes one, which leaves room for a second work-group on the CU: same box, backward of
// 12345 tokens with 14 / 2 heads 112 -> 99 us, of one 8192-token segment 483 -> 405, of 1237 tokens with 32 / 8 heads
// 57 -> 48; two blocks were slower at every size.
int launch_attn_dkv3(int D, const AttnParams& p, hipStream_t st) {
  return D == 128 ? launch<128, 2>(p, st) : launch<64, 1>(p, st);
}

int launch_attn_merge_bwd(int D, const AttnParams& params, int rb, hipStream_t st) {
  AttnParams p = params;
  p.blocks_k = attn_keyside_blocks(D, p.T, p.Hkv);
  const int nq = p.parts_q > 1 ? (p.T + 31) / 32 * p.Hq : 0;
  const long long nk = p.parts_k > 1 ? (long long)p.T * p.Hkv * (D / 8) : 0;
  const dim3 grid((unsigned)(nq + (2 * nk + 255) / 256));
  if (D == 128) hipLaunchKernelGGL((attn_merge_bwd_kernel<128, 64>), grid, dim3(256), 0, st, p, rb, nq, nk);
  else hipLaunchKernelGGL((attn_merge_bwd_kernel<64, 32>), grid, dim3(256), 0, st, p, rb, nq, nk);
  HIP_TRY(hipGetLastError());
  return 0;
}

}  // namespace fgrpo
