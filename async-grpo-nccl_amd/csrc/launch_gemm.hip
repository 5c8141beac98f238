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

// dHidden's lead (AHEAD, see early_barrier_pipeline16): work-groups walk the same rows of W, and the longer lead lets those that have
// lost step with each other stay apart.  They lose it along long contractions and when they replace others, so those take the
// shorter one.  Before the longer lead existed | longer | shorter, ms: whole tiles over the vocabulary (numerators of the whole batch
// kept): H = 5120, T = 16384 18.7 | 20.4 | 18.5, 12288 14.6 | 15.5 | 14.7; H = 3584, T = 32768 26.6 | 27.4 | 26.3; H = 1536 11.2 | 11.4 | 10.9;
// H = 896 .. 2048 and 8192 the same or up to 3 % better with the shorter; two pieces: H = 5120, T = 4500 5.66 | 6.02 | 5.75, 4800 5.79 | 6.13
// | 5.91.  Panels of the recomputing backward, a quarter of the vocabulary, keep the longer (H = 3584, T = 10400 10.5 | 11.1, longer |
// shorter), and so do three pieces or more (H = 3584, T = 4500 3.68 | 3.77; H = 6144, T = 4000 5.84 | 5.93) up to four device rounds of
// them (H = 3584, T = 8975 6.70 | 7.02; H = 1536, T = 8192 2.72 | 2.79; from the fifth on H = 5120, T = 8192 10.3 | 9.6).
constexpr int kLongContraction = 60000;
int launch_store_splitk(const StoreParams& p, hipStream_t st) {
  if (p.nblocks > 4 * num_cus() || p.kchunk >= kLongContraction)
    return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true, true, false>, Cfg8>(p, p.nblocks, st);
  return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true, true>, Cfg8>(p, p.nblocks, st);
}

int launch_small_split(const SmallSplitPair& p, int nblocks, hipStream_t st) {
  return launch_tile_kernel<gemm_small_split_kernel<Cfg4>, Cfg4>(p, nblocks, st);
}

int launch_store_kmajor(bool akm, bool bkm, const StoreParams& p, hipStream_t st) {
  const int nb = p.nblocks;
  // dW of the recomputing backward: the shorter lead as well.  Before the longer one existed | longer | shorter, ms: H = 1536, T =
  // 8192 2.91 | 3.02 | 2.97, 24000 8.62 | 8.94 | 8.74, 32768 11.9 | 12.4 | 12.2; H = 3584, T = 32768 28.9 | 30.0 | 29.6; H = 5120, T = 16384
  // 20.3 | 21.1 | 20.8; H = 1536, T = 4500 1.71 | 1.59 | 1.59.  dW of the kept numerators gains from the longer one (H = 1536, four
  // chunks of 8192 12.0 | 11.6 | 11.7).
  if (akm && bkm) return launch_tile_kernel<gemm_store_kernel<Cfg8, true, true, false, false>, Cfg8>(p, nb, st);
  if (akm) return launch_tile_kernel<gemm_store_kernel<Cfg8, true, false>, Cfg8>(p, nb, st);
  if (bkm && p.g.seg[0].K >= kLongContraction) return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true, false, false>, Cfg8>(p, nb, st);
  if (bkm) return launch_tile_kernel<gemm_store_kernel<Cfg8, false, true>, Cfg8>(p, nb, st);
  return fail(FGRPO_ERR_BAD_ARG, "gemm(k-major): no k-major operand");
}

}  // namespace fgrpo
