// Key-side attention backward, barrier-free form (attn_keyside.h): a translation unit of its own, compiled so that the
// matrix instructions the compiler schedules keep their results in ordinary vector registers.
#include "host_common.h"
#include "attn_keyside.h"

namespace fgrpo {

template <int HD, int KB>
static int launch(const AttnParams& p, hipStream_t st) {
  const long long ranks = (long long)((p.T + 127) / 128) * (4 / KB);          // every 128-key tile of the launch order, in pieces of 32 KB keys
  const int rc = raise_lds<varlen_attn_dkv3_kernel<HD, KB>>(kDkv3Lds<HD, KB>);
  if (rc) return rc;
  hipLaunchKernelGGL((varlen_attn_dkv3_kernel<HD, KB>), dim3((unsigned)(ranks * p.Hkv)), dim3(256), (kDkv3Lds<HD, KB>), st, p);
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

}  // namespace fgrpo
