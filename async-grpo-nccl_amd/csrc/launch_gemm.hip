// Instantiations and launches of the plain GEMM with store epilogue: every tile configuration with K-contiguous
// operands, and the 256x256x64 tile with contraction-major operands (the gradient GEMMs that read dLogits,
// hidden and W where they lie).
#include "host_common.h"

namespace fgrpo {
namespace {
template <class C>
int launch_store(const StoreParams& p, hipStream_t st) {
  return launch_tile_kernel<gemm_store_kernel<C, false, false>, C>(p, p.nblocks, st);
}
}  // namespace

int launch_store_variant(int variant, const StoreParams& p, hipStream_t st) {
  int rc = 0;
  DISPATCH_VARIANT(variant, launch_store, p, st);
  return rc;
}

int launch_store_splitk(const StoreParams& p, hipStream_t st) {
  // Pieces of one column chunk walk the same rows of W; from the fifth device round on, work-groups that replace others have
  // lost step with each other, and the longer lead lets them stay apart.  Longer | shorter lead, ms: H = 5120, T = 8192, five
  // rounds 10.3 | 9.6; H = 3584, T = 16384, seven 13.1 | 12.9; T = 8192, seven 6.74 | 6.75; four rounds at most: H = 3584, T = 8975
  // 6.70 | 7.02, T = 2000 1.76 | 1.85; H = 1536, T = 8192 2.72 | 2.79.
  if (p.nblocks > 4 * num_cus()) return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true, true, false>, Cfg8>(p, p.nblocks, st);
  return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true, true>, Cfg8>(p, p.nblocks, st);
}

int launch_small_split(const SmallSplitPair& p, int nblocks, hipStream_t st) {
  return launch_tile_kernel<gemm_small_split_kernel<Cfg4>, Cfg4>(p, nblocks, st);
}

int launch_store_kmajor(bool akm, bool bkm, const StoreParams& p, hipStream_t st) {
  const int nb = p.nblocks;
  if (akm && bkm) return launch_tile_kernel<gemm_store_kernel<Cfg8, true, true>, Cfg8>(p, nb, st);
  if (akm) return launch_tile_kernel<gemm_store_kernel<Cfg8, true, false>, Cfg8>(p, nb, st);
  if (bkm) return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true>, Cfg8>(p, nb, st);
  return fail(FGRPO_ERR_BAD_ARG, "gemm(k-major): no k-major operand");
}

}  // namespace fgrpo
