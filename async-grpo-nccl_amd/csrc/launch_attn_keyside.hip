// Key-side attention backward, barrier-free form (attn_keyside.h): a translation unit of its own, compiled so that the
// matrix instructions the compiler schedules keep their results in ordinary vector registers.
#include "host_common.h"
#include "attn_keyside.h"

namespace fgrpo {

int launch_attn_dkv3(int D, const AttnParams& p, hipStream_t st) {
  const long long ranks = (long long)((p.T + 127) / 128) * 2;          // every 128-key tile of the launch order, as two of 64
  const dim3 grid((unsigned)(ranks * p.Hkv));
  int rc;
  if (D == 128) {
    rc = raise_lds<varlen_attn_dkv3_kernel<128>>(kDkv3Lds<128>);
    if (rc) return rc;
    hipLaunchKernelGGL(varlen_attn_dkv3_kernel<128>, grid, dim3(256), kDkv3Lds<128>, st, p);
  } else {
    rc = raise_lds<varlen_attn_dkv3_kernel<64>>(kDkv3Lds<64>);
    if (rc) return rc;
    hipLaunchKernelGGL(varlen_attn_dkv3_kernel<64>, grid, dim3(256), kDkv3Lds<64>, st, p);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

}  // namespace fgrpo
