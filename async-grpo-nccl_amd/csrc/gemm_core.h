// bf16 GEMM main loops for gfx950 (CDNA4): D[m,n] = sum_k A[m,k] * B[n,k] on v_mfma_f32_32x32x16_bf16
// (lane l supplies row l % 32 and the eight k values 8*(l/32) .. 8*(l/32)+7 of each operand) or, on the
// 8-wavefront 256x256x64 tile every large problem takes (kMi16 below), on v_mfma_f32_16x16x32_bf16
// (lane l supplies row l % 16 and the eight k values 8*(l/16) .. 8*(l/16)+7).
//
// Work-group tile BM x BN, K step BK, WM x WN wavefronts (64 lanes each), every wavefront owning a
// (BM/WM) x (BN/WN) sub-tile made of 32x32 MFMA blocks kept in fp32 accumulators.  Four loops, chosen by the
// tile configuration (run_mainloop) or by the caller:
//   gemm_mainloop      global -> registers -> LDS, padded LDS rows, two buffers (small tiles, fp32 split path);
//   gemm_mainloop_dma  global -> LDS directly (buffer_load ... lds), swizzled LDS rows; with two buffers (of operand A three on
//                      16x16x32 MFMAs) it runs the early-barrier schedule below (the default for large problems), with
//                      three a plain prefetch loop;
//   gemm_mainloop_la   direct-to-LDS with four or more BK=32 buffers and one K step of fragment look-ahead;
//   gemm_mainloop_km   operands whose contraction index is the ROW index as stored (read through
//                      ds_read_b64_tr_b16), early-barrier schedule.
// Operands are K-contiguous (X[m][k]) unless a loop says otherwise.
//
// A contraction may be the sum of up to three (A_s, B_s, K_s) segments sharing
// the leading dimensions; the fp32 path uses that for the bf16 hi/lo split
// a*b ~= a_hi*b_hi + a_hi*b_lo + a_lo*b_hi.
//
// Contract checked by the host launchers: every K_s is a positive multiple of
// BK, every operand base is 16-byte aligned, lda/ldb are multiples of 8
// elements, rows past M (or N) are never read (row indices are clamped) and a
// tile's rows span less than 4 GiB.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include <utility>

// Every fragment read must stay consumed by an MFMA: the two-buffer loops issue their LDS reads as inline
// assembly, and a read whose result is dead lets the register allocator reuse its destination while the
// data is still in flight (a build that dropped the MFMAs corrupted load addresses that way).
#define FGRPO_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16((a), (b), (c), 0, 0, 0)

#define FGRPO_LDFRAG(ptr) (*(const bf16x8_t*)(ptr))

namespace fgrpo {

typedef uint16_t bf16_t;  // storage type of a bfloat16
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;  // one 16-byte chunk

struct GemmSeg {
  const bf16_t* A;
  const bf16_t* B;
  int K;
};

struct GemmOperands {
  GemmSeg seg[3];
  int nseg;
  long long lda, ldb;  // elements
  int M, N;
  // K-major operands only (gemm_mainloop_km): rows k >= ka_valid / kb_valid do not exist in memory
  // and read as zero (buffer bounds).  0 = every row of K exists.
  int ka_valid, kb_valid;
  // Column-blocked A (direct-to-LDS two/three-buffer loops and gemm_mainloop_km only): when a_blk != 0 the
  // logical matrix X[r][c] (r = row as stored, c = contiguous index) is kept as 256-column blocks,
  // X[r][c] at A + (c / 256) * a_blk + r * 256 + (c % 256) elements (lda must be 256).  A tile that walks
  // down the rows of one block (K-major use) then reads one sequential stream, and a tile that walks along
  // the columns (K-contiguous use) reads 128 KiB contiguous pieces.
  long long a_blk;
  // gemm_mainloop_km with a K-major A only: the contraction may skip whole K steps (64 rows each) that
  // are known to contribute nothing.  k_runs (device memory, written by an earlier launch on the stream) =
  // {number of runs R, K steps in all runs, start_0 .. start_{kRunCap-1}, end_0 .. end_{kRunCap-1}}: run r covers
  // the K steps start_r <= k < end_r, runs ascending and disjoint.  Null = every K step.
  const int* k_runs;
};
constexpr int kRunCap = 4096;   // runs a k_runs list can hold (more live/dead alternations than that: pass null)

template <int BM_, int BN_, int BK_, int WM_, int WN_, int OCC_, int NST_ = 2, bool DMA_ = false>
struct TileCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, OCC = OCC_;
  static constexpr bool DMA = DMA_;             // global -> LDS directly (no register staging)
  static constexpr int NW = WM * WN;            // wavefronts per work-group
  static constexpr int NT = NW * 64;            // threads per work-group
  static constexpr int WTM = BM / WM;           // wavefront tile rows
  static constexpr int WTN = BN / WN;           // wavefront tile cols
  static constexpr int TM = WTM / 32;           // 32x32 blocks per wavefront, rows
  static constexpr int TN = WTN / 32;           // 32x32 blocks per wavefront, cols
  static constexpr int CPR = BK / 8;            // 16-byte chunks per tile row
  static constexpr int RPP = NT / CPR;          // tile rows covered by one load pass of the work-group
  static constexpr int PA = BM / RPP;           // load passes for A (per thread)
  static constexpr int PB = BN / RPP;           // load passes for B (per thread)
  static constexpr int RPI = 64 / CPR;          // tile rows covered by one wavefront-wide 16-byte load
  static constexpr int ROWB = DMA ? BK * 2 : BK * 2 + 16;  // LDS row bytes (register path pads, DMA path swizzles)
  static constexpr int STAGE = (BM + BN) * ROWB;
  static constexpr int NSTAGE = NST_;
  static constexpr bool MI16 = DMA && NST_ == 2 && NW == 8 && BK == 64 && TM == 4 && TN == 2;   // see kMi16
  // the 16x16x32 schedule keeps a third buffer for operand A (early_barrier_pipeline16)
  static constexpr int LDS_BYTES = STAGE * NSTAGE + (MI16 ? BM * ROWB : 0);
  static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "tile/wave shape");
  static_assert(BK % 16 == 0 && NT % CPR == 0 && BM % RPP == 0 && BN % RPP == 0, "loader shape");
  static_assert(!DMA || (CPR == 4 || CPR == 8), "DMA path supports BK = 32 or 64");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

// Accumulator element (i, j, r) of lane `lane` in wavefront (wm, wn) sits at
//   row = wm*WTM + i*32 + 8*(r/4) + 4*(lane/32) + (r%4)
//   col = wn*WTN + j*32 + (lane%32)
// relative to the tile origin.
template <class C>
__device__ __forceinline__ int acc_row(int wm, int i, int r, int lane) {
  return wm * C::WTM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}
template <class C>
__device__ __forceinline__ int acc_col(int wn, int j, int lane) {
  return wn * C::WTN + j * 32 + (lane & 31);
}

// The 256x256x64 two-buffer direct-to-LDS loops of the 8-wavefront tile can run on v_mfma_f32_16x16x32_bf16 instead
// of 32x32x16 (kMi16): same flops per cycle, half the fp32 accumulator registers read and written per flop - on this
// power-limited part the same kernels run 5 % faster with it.  A 32x32 block (i, j) of a wavefront is then four
// 16x16 blocks (rh, ch), each one MFMA per 32-wide K slice, and the block's sixteen accumulator registers are
//   element e = 4*(2*rh + ch) + r :  row = wm*WTM + i*32 + 16*rh + 4*(lane/16) + r
//                                   col = wn*WTN + j*32 + 16*ch + (lane%16)
// relative to the tile origin.
template <class C>
constexpr bool kMi16 = C::MI16;
template <class C>
__device__ __forceinline__ int acc16_row(int wm, int i, int e, int lane) {
  return wm * C::WTM + i * 32 + 16 * (e >> 3) + 4 * (lane >> 4) + (e & 3);
}
template <class C>
__device__ __forceinline__ int acc16_col(int wn, int j, int e, int lane) {
  return wn * C::WTN + j * 32 + 16 * ((e >> 2) & 1) + (lane & 15);
}
// Sub-tile (wm, wn) of a wavefront.  Wavefronts w and w + 4 share a SIMD.  CROSSED (the contraction-major gradient
// products): the two lie in different row halves AND different column halves, so that a tile with one half outside
// the matrix (rows or columns) leaves every SIMD one wavefront that computes and one that only loads (wave_is_live).
template <class C, bool CROSSED>
__device__ __forceinline__ void wave_coords(int wave, int& wm, int& wn) {
  if constexpr (CROSSED) {
    static_assert(C::WM == 2 && C::WN == 4, "wavefront grid");
    wm = (wave ^ (wave >> 2)) & 1;
    wn = wave >> 1;
  } else {
    wm = wave / C::WN;
    wn = wave % C::WN;
  }
}
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
// acc<registers 4Q .. 4Q+3> += a (16 rows x 32 k) * b (16 columns x 32 k)
template <int Q>
__device__ __forceinline__ void mfma16_slice(bf16x8_t a, bf16x8_t b, f32x16_t& c) {
  f32x4_t t = __builtin_shufflevector(c, c, 4 * Q, 4 * Q + 1, 4 * Q + 2, 4 * Q + 3);
  t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, t, 0, 0, 0);
  c[4 * Q] = t[0];
  c[4 * Q + 1] = t[1];
  c[4 * Q + 2] = t[2];
  c[4 * Q + 3] = t[3];
}

template <class C>
__device__ __forceinline__ void zero_acc(f32x16_t (&acc)[C::TM][C::TN]) {
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// acc += A[row0 : row0+BM, :] * B[col0 : col0+BN, :]^T over all segments.
// Must be called by every thread of the work-group (it contains barriers).  On
// return all LDS reads have completed and a barrier has been passed, so the
// caller may reuse `smem`.  klen > 0: only the range [k0, k0 + klen) of every segment.
template <class C>
__device__ __forceinline__ void gemm_mainloop(const GemmOperands& g, int row0, int col0, char* smem,
                                              f32x16_t (&acc)[C::TM][C::TN], int k0 = 0, int klen = 0) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int lrow = tid / C::CPR, lchk = tid % C::CPR;

  uint32_t aoff[C::PA], boff[C::PB];
  const int amax = g.M - 1 - row0, bmax = g.N - 1 - col0;
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    int r = lrow + i * C::RPP;
    r = r < amax ? r : amax;
    aoff[i] = (uint32_t)((long long)r * g.lda * 2 + lchk * 16);
  }
#pragma unroll
  for (int i = 0; i < C::PB; ++i) {
    int r = lrow + i * C::RPP;
    r = r < bmax ? r : bmax;
    boff[i] = (uint32_t)((long long)r * g.ldb * 2 + lchk * 16);
  }
  // LDS byte offsets of this thread's staging stores and fragment reads.
  const int st_a = lrow * C::ROWB + lchk * 16;
  const int st_b = C::BM * C::ROWB + st_a;
  const int fr_a = (wm * C::WTM + (lane & 31)) * C::ROWB + (lane >> 5) * 16;
  const int fr_b = C::BM * C::ROWB + (wn * C::WTN + (lane & 31)) * C::ROWB + (lane >> 5) * 16;

  for (int s = 0; s < g.nseg; ++s) {
    const char* Ab = (const char*)(g.seg[s].A + (long long)row0 * g.lda + k0);
    const char* Bb = (const char*)(g.seg[s].B + (long long)col0 * g.ldb + k0);
    const int nk = (klen > 0 ? klen : g.seg[s].K) / C::BK;

    u32x4_t ra[C::PA], rb[C::PB];
#pragma unroll
    for (int i = 0; i < C::PA; ++i) ra[i] = *(const u32x4_t*)(Ab + aoff[i]);
#pragma unroll
    for (int i = 0; i < C::PB; ++i) rb[i] = *(const u32x4_t*)(Bb + boff[i]);
#pragma unroll
    for (int i = 0; i < C::PA; ++i) *(u32x4_t*)(smem + st_a + i * C::RPP * C::ROWB) = ra[i];
#pragma unroll
    for (int i = 0; i < C::PB; ++i) *(u32x4_t*)(smem + st_b + i * C::RPP * C::ROWB) = rb[i];
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
      const int cur = (kt & 1) * C::STAGE;
      const bool more = (kt + 1 < nk);
      if (more) {
        Ab += C::BK * 2;
        Bb += C::BK * 2;
#pragma unroll
        for (int i = 0; i < C::PA; ++i) ra[i] = *(const u32x4_t*)(Ab + aoff[i]);
#pragma unroll
        for (int i = 0; i < C::PB; ++i) rb[i] = *(const u32x4_t*)(Bb + boff[i]);
      }
#pragma unroll
      for (int kk = 0; kk < C::BK / 16; ++kk) {
        bf16x8_t af[C::TM], bf[C::TN];
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
          af[i] = *(const bf16x8_t*)(smem + cur + fr_a + i * 32 * C::ROWB + kk * 32);
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
          bf[j] = *(const bf16x8_t*)(smem + cur + fr_b + j * 32 * C::ROWB + kk * 32);
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
          for (int j = 0; j < C::TN; ++j)
            acc[i][j] = FGRPO_MFMA(af[i], bf[j], acc[i][j]);
      }
      if (more) {
        const int nxt = C::STAGE - cur;
#pragma unroll
        for (int i = 0; i < C::PA; ++i) *(u32x4_t*)(smem + nxt + st_a + i * C::RPP * C::ROWB) = ra[i];
#pragma unroll
        for (int i = 0; i < C::PB; ++i) *(u32x4_t*)(smem + nxt + st_b + i * C::RPP * C::ROWB) = rb[i];
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// Direct-to-LDS variant.  global_load_lds_dwordx4 writes lane l's 16 bytes at
// (wave-uniform LDS base) + 16*l, so one wavefront-wide load fills RPI whole
// tile rows of BK*2 bytes without padding.  Bank conflicts of the fragment
// reads are avoided by an XOR swizzle of the 16-byte chunk index with a
// function of the row, applied on the *global* side (each lane fetches the
// chunk that belongs at its LDS slot).  NSTAGE LDS buffers keep NSTAGE-1 K
// steps of loads in flight; completion is tracked with explicit vmcnt waits and
// one s_barrier per K step.
// ---------------------------------------------------------------------------
#define FGRPO_DMA_AUX 0   // cache-policy bits of the direct-to-LDS loads
#define FGRPO_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define FGRPO_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

// Raw buffer descriptor over [base, base + bytes): offsets past `bytes` read as zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// s_waitcnt that waits only for the vector-memory counter to drop to n (n < 64).
#define FGRPO_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | (((n) >> 4) << 14))
// same, and also wait for every outstanding LDS read (lgkmcnt = 0)
#define FGRPO_WAIT_VMCNT_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (0 << 8) | (((n) >> 4) << 14))

template <class C, bool MI16 = false>
__device__ __forceinline__ int lds_swizzle(int row) {
  // Chosen with SQ_LDS_BANK_CONFLICT on the real kernels and a read-rate microbenchmark.  32x32x16 fragment read:
  // lane l -> row l%32, chunk l/32 + 2*kk.  16x16x32 fragment read: lane l -> row l%16, chunk l/16 + 4*k2; under the
  // 32-row swizzle these reads run at half rate (two-way conflicts), under row%8 at the full rate.
  if constexpr (C::CPR == 4)
    return (row >> 2) & 3;                       // 64-byte rows
  else if constexpr (MI16)
    return row & 7;                              // 128-byte rows, 16-row fragments
  else
    return (row + ((row >> 3) & 1)) & 7;         // 128-byte rows, 32-row fragments
}

__device__ __forceinline__ void wg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The fragment reads of the two-buffer direct-to-LDS loops are written as inline assembly: for an LDS access it can see, the
// compiler waits (vmcnt) for every direct-to-LDS load in flight, which would serialise the prefetch of the
// next K step behind each fragment read.  The price: the compiler does not count these reads either, so
// the loop waits for them itself (s_waitcnt lgkmcnt(n); LDS operations return in order).
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t lds_addr(const char* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
template <int OFF0, int OFF1>
__device__ __forceinline__ bf16x8_t lds_read_tr_pair(uint32_t addr) {
  static_assert(OFF0 >= 0 && OFF1 < 65536, "DS offset field");
  u32x2_t lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
               : "=&v"(lo), "=&v"(hi)
               : "v"(addr), "i"(OFF0), "i"(OFF1));
  const u32x4_t v = {lo.x, lo.y, hi.x, hi.y};
  return __builtin_bit_cast(bf16x8_t, v);
}
// 8-byte LDS store the compiler does not see either (an epilogue patch written while direct-to-LDS loads of the
// next tile are in flight would otherwise wait for them)
template <int OFF = 0>
__device__ __forceinline__ void lds_write_b64_asm(uint32_t addr, uint32_t lo, uint32_t hi) {
  static_assert(OFF >= 0 && OFF < 65536, "DS offset field");
  const u32x2_t v = {lo, hi};
  asm volatile("ds_write_b64 %0, %1 offset:%2" : : "v"(addr), "v"(v), "i"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ bf16x8_t lds_read_b128_asm(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "DS offset field");
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(OFF));
  return __builtin_bit_cast(bf16x8_t, v);
}

// ---------------------------------------------------------------------------
// Two-buffer schedule shared by the direct-to-LDS loops ("barrier one sub-step early").
// The barrier of step kt sits before its LAST 16-wide sub-step: by then every
// wavefront has its last fragments of buffer `cur` in registers and the loads of
// step kt+1 have landed, so (a) the first fragments of step kt+1 are fetched right
// after the barrier and arrive under the MFMAs of the last sub-step (no LDS
// latency is exposed), and (b) buffer `cur` is free from that point: the loads of
// step kt+2 start into it at once, spread one by one over the MFMA groups of the
// next EB_PHASES sub-steps, which leaves them the rest of the step to land.
//   issue_one(stage, idx): load idx (0 .. LPT-1) of the next K step into `stage`;
//                          idx == LPT-1 also advances the source cursor.
//   load_a/load_b(stage_ptr, block, kk): one MFMA operand from LDS.
// On entry the loads of step 0 have been issued into buffer 0 (if nk_total > 0).
// ---------------------------------------------------------------------------
constexpr int kLoadPhases = 2;   // sub-steps over which one K step's loads are issued (1 and 3 measured slower)
// compile-time loop: f(std::integral_constant<int, 0>{}) ... f(std::integral_constant<int, N-1>{})
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

//   load_a/load_b(stage_ptr, I, KK): one MFMA operand from LDS (I, KK are std::integral_constant), issued as
//   RA / RB inline-assembly LDS instructions that the compiler does not count: this function places every
//   s_waitcnt lgkmcnt(n) itself (LDS operations return in order).
// The fragments of the following sub-step are requested between the MFMA row groups of the current one, in the
// order a0, b0 .. b(TN-1), a1 .. a(TM-1) (row group 0 needs a0 and every b), so that the LDS sees a steady
// trickle of reads next to the direct-to-LDS stream instead of a burst per sub-step (a burst measured equal or
// slower).
template <int N>
__device__ __forceinline__ void wait_lgkm() {
  static_assert(N >= 0, "wait count");
  __builtin_amdgcn_s_waitcnt(0xC07F | ((N > 15 ? 15 : N) << 8));   // vmcnt / expcnt untouched
}

template <class C, int LPT, int RA, int RB, class IssueOne, class LoadA, class LoadB>
__device__ __forceinline__ void early_barrier_pipeline(int nk_total, char* smem, f32x16_t (&acc)[C::TM][C::TN],
                                                       IssueOne&& issue_one, LoadA&& load_a, LoadB&& load_b) {
  constexpr int KK = C::BK / 16;
  constexpr int TM = C::TM, TN = C::TN, NR = TM + TN;
  static_assert(KK % 2 == 0 && KK >= kLoadPhases + 1, "sub-steps per K step");
  constexpr int NSLOT = kLoadPhases * TM;         // MFMA groups over which one step's loads are spread
  // fragment order and bookkeeping (all compile time)
  struct Ord {
    static constexpr int cum(int i) { return (i * NR + TM - 1) / TM; }  // entries requested before row group i ends.. starts
    static constexpr int instrs(int n) {              // LDS instructions of the first n entries
      int c = 0;
      for (int e = 0; e < n; ++e) c += (e == 0 || e > TN) ? RA : RB;
      return c;
    }
    static constexpr int need(int i) { return i == 0 ? TN : TN + i; }   // last entry row group i waits for
    // instructions that may still be outstanding when row group i starts
    static constexpr int allowed(int i, bool issuing) {
      return instrs(NR) - instrs(need(i) + 1) + (issuing ? instrs(cum(i)) : 0);
    }
  };
  FGRPO_WAIT_VMCNT(0);
  wg_barrier();                                       // step 0 is in buffer 0
  int steps_issued = nk_total > 0 ? 1 : 0;
  bool active = steps_issued < nk_total;              // a step is being loaded
  int tgt = 1;                                        // ... into this buffer
  if (active) {
    ++steps_issued;
    static_for<LPT>([&](auto q) {
      if constexpr (decltype(q)::value * NSLOT / LPT < TM) issue_one(1, decltype(q)::value);  // phase 0's share
    });
  }
  bf16x8_t af[2][TM], bf[2][TN];
  // entry e of the request order, for sub-step KN of the buffer at `base`, into register buffer BUF
  auto request = [&](const char* base, auto ec, auto knc, auto bufc) {
    constexpr int e = decltype(ec)::value, buf = decltype(bufc)::value;
    if constexpr (e == 0)
      af[buf][0] = load_a(base, std::integral_constant<int, 0>{}, knc);
    else if constexpr (e <= TN)
      bf[buf][e - 1] = load_b(base, std::integral_constant<int, e - 1>{}, knc);
    else
      af[buf][e - TN] = load_a(base, std::integral_constant<int, e - TN>{}, knc);
  };
  static_for<NR>([&](auto e) { request(smem, e, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}); });
  int cur = 0;
  // One K step.  STEADY: at least two more steps follow, so a next step exists and a further one is always
  // there to be loaded; the body then carries no conditionals at all.
  auto step = [&](int kt, auto steady_c) {
    constexpr bool STEADY = decltype(steady_c)::value;
    const char* st = smem + cur * C::STAGE;
    const char* sn = smem + (cur ^ 1) * C::STAGE;
    const bool next = STEADY || kt + 1 < nk_total;
    static_for<KK>([&](auto kkc) {
      constexpr int kk = decltype(kkc)::value;
      constexpr bool last = (kk == KK - 1);
      constexpr int kn = last ? 0 : kk + 1, nbuf = (kk + 1) & 1;
      const char* src = last ? sn : st;
      const bool issuing = STEADY || !last || next;
      if constexpr (last) {
        if (next) {
          FGRPO_WAIT_VMCNT_LGKM0(0);                  // my loads of step kt+1 landed; my reads of `cur` returned
          wg_barrier();
          active = STEADY || steps_issued < nk_total; // loads of step kt+2 go into the buffer just freed
          tgt = cur;
          if (active) ++steps_issued;
        }
      }
      // phase of the load spreading this sub-step belongs to: 0 = last sub-step, then 1, 2 .. from the top
      constexpr int phase = last ? 0 : kk + 1;
      const bool loads_here = STEADY || (active && phase < kLoadPhases && (phase > 0 || next));
      __builtin_amdgcn_sched_barrier(0);
      static_for<TM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (!last) {
          wait_lgkm<Ord::allowed(i, true)>();
        } else {
          if (next) wait_lgkm<Ord::allowed(i, true)>(); else wait_lgkm<Ord::allowed(i, false)>();
        }
        __builtin_amdgcn_sched_barrier(0);
        {
          // the group's fragment requests and loads go BETWEEN its MFMAs (after MFMA j the extras x with
          // x*TN/X == j): an MFMA keeps the matrix pipe busy for 32 cycles but issues in 4, so whatever is
          // issued right behind it is free - what is issued after the last one delays the next group.
          constexpr int R = Ord::cum(i + 1) - Ord::cum(i);
          constexpr int slot = phase * TM + i;
          constexpr int q_lo = (phase < kLoadPhases) ? (slot * LPT + NSLOT - 1) / NSLOT : 0;
          constexpr int q_hi = (phase < kLoadPhases) ? ((slot + 1) * LPT + NSLOT - 1) / NSLOT : 0;   // loads q_lo .. q_hi-1
          constexpr int X = R + (q_hi - q_lo);
          static_for<TN>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            acc[i][j] = FGRPO_MFMA(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
            static_for<X>([&](auto xc) {
              constexpr int x = decltype(xc)::value;
              if constexpr (x * TN / (X > 0 ? X : 1) == j) {
                if constexpr (x < R) {
                  if (issuing)
                    request(src, std::integral_constant<int, Ord::cum(i) + x>{}, std::integral_constant<int, kn>{},
                            std::integral_constant<int, nbuf>{});
                } else {
                  if (loads_here) issue_one(tgt, q_lo + (x - R));
                }
              }
            });
            __builtin_amdgcn_sched_barrier(0);
          });
        }
      });
    });
    cur ^= 1;
  };
  int kt = 0;
  for (; kt + 2 < nk_total; ++kt) step(kt, std::true_type{});
  for (; kt < nk_total; ++kt) step(kt, std::false_type{});
  wg_barrier();                                       // LDS may be reused by the caller
}

// The same schedule on 16x16x32 MFMAs (kMi16 tiles: TM = 4, TN = 2, BK = 64).  A K step is still four sub-steps of
// equal length: sub-step kk works on the 32-wide K slice k2 = kk/2 and on the row half rh = kk%2 of every 32x32
// block - 16 MFMAs: for each block row i the fragment a(i, rh) (16 rows x 32 k) against the four fragments
// b(j, ch) (16 columns x 32 k) of the slice.  The b fragments of a slice are fetched once, before its first
// sub-step, and serve both; so the fragment requests alternate between 4 (a only, before an odd sub-step) and
// 8 (a0, the four b, a1 .. a3, before an even one).
// Operand A (the streamed one in every use: W in the LM-head kernels, the [T x V] buffer in the gradient products) has
// three LDS buffers and operand B two.  AHEAD: A is requested almost two K steps before it is needed,
//   B of step kt + 1 behind the barrier of step kt - 1 (its buffer was freed there), A of step kt + 2 in the next sub-step,
// and the barrier of step kt waits for all but that youngest A.  With one step of lead for both, as it was, a request that
// missed the L2 was waited for in every step.  But such waits also keep the work-groups of an XCD together: the first to
// ask for a slice waits, those behind it find it in the L2.  With the longer lead nothing held them (forward of 40000
// tokens, H = 5120: past the L2s 36.7 -> 71.8 GB, 6 % fewer cycles at a lower clock, 35.6 -> 36.9 ms); so every
// kStrictEvery-th step waits for the youngest A as well (33.9 ms; every second step 34.0, every eighth 34.9).  !AHEAD: the
// one step of lead, for dHidden over the whole vocabulary or in many device rounds (launch_store_splitk, launch_store_kmajor), where
// the drift adds up.  Before -> after, one box each: forward that keeps the numerators, T = 8192, H = 1536: 3.28 -> 3.09 ms, H =
// 3584, T = 16384: 13.14 -> 12.78; dW of 8192 tokens, H = 1536: 3.04 -> 2.98; dHidden of 777 tokens 0.409 -> 0.388.
//   issue_a(lds, idx) / issue_b(lds, idx): load idx of the next K step of that operand into the buffer at `lds`; the
//   last one of A (the first one of B, but for step 0's) advances the operand's cursor;
//   load_a(lds, I, KK): fragment a(I, KK % 2) of slice KK / 2;  load_b(lds, JC, K2): fragment b(JC/2, JC%2).
// NB: 16-column blocks of operand B a wavefront multiplies, 4 or, on tiles 64 NB columns wide (the forward's narrow last token tile), fewer.
// On entry B of step 0 and A of steps 0 and 1 have been issued, in this order (as far as they exist).  DRAIN: wait for
// all of it (the caller has issued something else since), not just for step 0.
constexpr int kStrictEvery = 4;                      // a power of two
template <class C>
constexpr int kOpBytes = C::BM * C::ROWB;            // one buffer of one operand (32 KiB)
// of step's B, in kOpBytes; A's is step % 3, so that buffers 2 and 3 are free between tiles
__device__ __forceinline__ constexpr int mi16_b_buf(int step) { return 4 - (step & 1); }
template <class C, int NB, int RA, int RB, bool DRAIN, bool AHEAD, class IssueA, class IssueB, class LoadA, class LoadB>
__device__ __forceinline__ void early_barrier_pipeline16(int nk_total, char* smem, f32x16_t (&acc)[C::TM][C::TN],
                                                         bool live, IssueA&& issue_a, IssueB&& issue_b, LoadA&& load_a,
                                                         LoadB&& load_b) {
  constexpr int KK = 4;
  constexpr int TM = C::TM;                           // a fragments per sub-step; NB: b fragments per K slice
  constexpr int PA = C::PA, PB = NB, OP = kOpBytes<C>;
  static_assert(kMi16<C> && C::BK == 64 && PA == TM && C::PB == 4 && NB >= 1 && NB <= 4, "16x16x32 schedule: 8-wavefront 256x256x64 tile, one load per row group");
  // request list of a sub-step by its parity P (0: a0, b0 .. b(NB-1), a1 ..; 1: a0 .. a(TM-1)), all compile time
  struct Ord {
    static constexpr int nr(int P) { return P == 0 ? TM + NB : TM; }
    static constexpr int cost(int P, int e) { return P == 0 ? ((e == 0 || e > NB) ? RA : RB) : RA; }
    static constexpr int instrs(int P, int n) {
      int c = 0;
      for (int e = 0; e < n; ++e) c += cost(P, e);
      return c;
    }
    static constexpr int cum(int P, int i) { return (i * nr(P) + TM - 1) / TM; }     // entries requested before row group i starts
    static constexpr int need(int P, int i) { return P == 0 ? (i == 0 ? NB : NB + i) : i; }   // last entry row group i waits for
    // LDS instructions that may still be outstanding when row group i of a sub-step of parity P starts
    static constexpr int allowed(int P, int i, bool issuing) {
      return instrs(P, nr(P)) - instrs(P, need(P, i) + 1) + (issuing ? instrs(1 - P, cum(1 - P, i)) : 0);
    }
  };
  if (DRAIN || nk_total < 2) FGRPO_WAIT_VMCNT(0);
  else FGRPO_WAIT_VMCNT(PA);
  wg_barrier();                                       // step 0 is in LDS
  if (AHEAD && nk_total > 1) static_for<PB>([&](auto q) { issue_b(smem + mi16_b_buf(1) * OP, decltype(q)::value); });
  char *a0 = smem, *a1 = smem + OP, *a2 = smem + 2 * OP;                                    // A of steps kt, kt + 1, kt + 2
  char *b0 = smem + mi16_b_buf(0) * OP, *b1 = smem + mi16_b_buf(1) * OP;                    // B of steps kt, kt + 1
  auto rotate = [&]() {
    char* t = a0;
    a0 = a1, a1 = a2, a2 = t;
    t = b0;
    b0 = b1, b1 = t;
  };
  if (!live || nk_total <= 0) {
    // a sub-tile outside the matrix: this wavefront's share of the loads and every barrier, nothing else
    for (int kt = 0; kt + 1 < nk_total; ++kt) {
      const bool more = kt + 2 < nk_total;
      if constexpr (AHEAD) {
        if (more) static_for<PA>([&](auto q) { issue_a(a2, decltype(q)::value); });
      } else {
        static_for<PB>([&](auto q) { issue_b(b1, decltype(q)::value); });
      }
      FGRPO_WAIT_VMCNT(0);
      wg_barrier();                                   // the one inside step kt: step kt + 1 is in LDS, the buffers of step kt are free
      if (more) {
        if constexpr (AHEAD) static_for<PB>([&](auto q) { issue_b(b0, decltype(q)::value); });
        else static_for<PA>([&](auto q) { issue_a(a2, decltype(q)::value); });
      }
      rotate();
    }
    wg_barrier();
    return;
  }
  bf16x8_t af[2][TM], bfr[2][NB];
  // entry e of the request list of sub-step KN, read from the buffers at `ba` and `bb`
  auto request = [&](const char* ba, const char* bb, auto ec, auto knc) {
    constexpr int e = decltype(ec)::value, kn = decltype(knc)::value;
    if constexpr ((kn & 1) == 1) {
      af[1][e] = load_a(ba, ec, knc);
    } else if constexpr (e == 0) {
      af[0][0] = load_a(ba, std::integral_constant<int, 0>{}, knc);
    } else if constexpr (e <= NB) {
      bfr[(kn >> 1) & 1][e - 1] = load_b(bb, std::integral_constant<int, e - 1>{}, std::integral_constant<int, (kn >> 1)>{});
    } else {
      af[0][e - NB] = load_a(ba, std::integral_constant<int, e - NB>{}, knc);
    }
  };
  static_for<Ord::nr(0)>([&](auto e) { request(a0, b0, e, std::integral_constant<int, 0>{}); });
  // One K step.  STEADY: at least two more steps follow; the body then carries no conditionals at all.
  auto step = [&](int kt, auto steady_c) {
    constexpr bool STEADY = decltype(steady_c)::value;
    constexpr bool more = STEADY;                     // step kt + 2 is loaded during this one
    const bool next = STEADY || kt + 1 < nk_total;
    static_for<KK>([&](auto kkc) {
      constexpr int kk = decltype(kkc)::value;
      constexpr bool last = (kk == KK - 1);
      constexpr int kn = last ? 0 : kk + 1;
      constexpr int P = kk & 1, k2 = kk >> 1;
      const char *src_a = last ? a1 : a0, *src_b = last ? b1 : b0;
      const bool issuing = STEADY || !last || next;
      if constexpr (last) {
        if (next) {
          // my loads of step kt + 1 landed (of step kt + 2 the A loads may be in flight); my reads of step kt returned
          if (!AHEAD || !more || (NB == 4 && (kt & (kStrictEvery - 1)) == 0)) FGRPO_WAIT_VMCNT_LGKM0(0);
          else FGRPO_WAIT_VMCNT_LGKM0(PA);
          wg_barrier();                               // the buffers of step kt are free
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<TM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (!last) {
          wait_lgkm<Ord::allowed(P, i, true)>();
        } else {
          if (next) wait_lgkm<Ord::allowed(P, i, true)>(); else wait_lgkm<Ord::allowed(P, i, false)>();
        }
        __builtin_amdgcn_sched_barrier(0);
        {
          // the row group's load: one operand's in the first sub-step, the other's behind the barrier
          constexpr bool load_here = (AHEAD ? kk == 0 : last) || ((AHEAD ? last : kk == 0) && i < PB);
          constexpr int R = Ord::cum(1 - P, i + 1) - Ord::cum(1 - P, i);
          constexpr int X = R + (load_here ? 1 : 0);
          static_for<NB>([&](auto jcc) {
            constexpr int jc = decltype(jcc)::value;       // b fragment (j, ch) = (jc / 2, jc % 2)
            mfma16_slice<2 * P + (jc & 1)>(af[P][i], bfr[k2 & 1][jc], acc[i][jc >> 1]);
            static_for<X>([&](auto xc) {
              constexpr int x = decltype(xc)::value;
              if constexpr (x * NB / (X > 0 ? X : 1) == jc) {
                if constexpr (x < R) {
                  if (issuing) request(src_a, src_b, std::integral_constant<int, Ord::cum(1 - P, i) + x>{}, std::integral_constant<int, kn>{});
                } else if constexpr (!AHEAD && !last) {
                  if (next) issue_b(b1, i);
                } else if constexpr (more) {
                  if constexpr (AHEAD && last) issue_b(b0, i);
                  else issue_a(a2, i);
                }
              }
            });
            __builtin_amdgcn_sched_barrier(0);
          });
        }
      });
    });
    rotate();
  };
  int kt = 0;
  for (; kt + 2 < nk_total; ++kt) step(kt, std::true_type{});
  for (; kt < nk_total; ++kt) step(kt, std::false_type{});
  wg_barrier();                                       // LDS may be reused by the caller
}

// Whether a wavefront's sub-tile holds anything of the matrix.  Those that do not skip the matrix instructions and LDS
// reads of the main loop (their accumulators stay zero).  In the contraction-major gradient products only: the LM-head
// kernels keep their statistics in registers across the loop and would spill.
template <class C>
__device__ __forceinline__ bool wave_is_live(const GemmOperands& g, int row0, int col0, int wm, int wn) {
  return row0 + wm * C::WTM < g.M && col0 + wn * C::WTN < g.N;
}

// MODE 0: the whole contraction.  MODE 2: only issue the first loads and return (the caller does something else, e.g. the
// epilogue of the previous tile, while they fly): K step 0 into buffer 0 of two, or on the 16x16x32 schedule B of step 0 and A
// of steps 0 and 1 into operand buffers 4, 0 and 1 (the caller may use what lies between: 64 KiB from C::STAGE on).  MODE 1: the contraction, given that
// a MODE 2 call for the same tile has been made since the last MODE 0/1 call returned.  Modes 1 and 2 exist for
// the two-buffer schedule only (kSplitPrologue).
template <class C>
constexpr bool kSplitPrologue = C::DMA && C::NSTAGE == 2 && (C::BK / 16) % 2 == 0;

// gemm_mainloop_dma on the 16x16x32 schedule.  MODE 2 requests what early_barrier_pipeline16 expects on entry and
// leaves operand buffers 2 and 3 to the caller until the MODE 1 call.
// NB < 4: the tile is 64 NB columns wide, 16 NB of them a wavefront's.
template <class C, int MODE, int NB = 4>
__device__ __forceinline__ void gemm_mainloop_dma16(const GemmOperands& g, int row0, int col0, char* smem,
                                                    f32x16_t (&acc)[C::TM][C::TN]) {
  static_assert(kMi16<C>, "16x16x32 MFMAs: 8-wavefront 256x256x64 two-buffer tile only");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));                 // the per-lane offsets are formed anew per call (see gemm_mainloop_dma)
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int lrow = lane / C::CPR, lpc = lane % C::CPR;
  uint32_t aoff[C::PA], boff[NB];
  const int amax = g.M - 1 - row0, bmax = g.N - 1 - col0;
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;
    const int r = rt < amax ? rt : amax;
    aoff[i] = (uint32_t)((long long)r * g.lda * 2 + ((lpc ^ lds_swizzle<C, true>(rt)) * 16));
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;
    const int r = rt < bmax ? rt : bmax;
    boff[i] = (uint32_t)((long long)r * g.ldb * 2 + ((lpc ^ lds_swizzle<C, true>(rt)) * 16));
  }
  const int dst_w = wave * C::RPI * C::ROWB;

  int nk_total = 0;
  for (int s = 0; s < g.nseg; ++s) nk_total += g.seg[s].K / C::BK;

  // One cursor over (segment, k) per operand: A runs a K step ahead of B.
  int sa = 0, la = g.seg[0].K / C::BK, sb = 0, lb = la;
  const char* Abase = (const char*)(g.seg[0].A + (long long)row0 * g.lda);
  __amdgpu_buffer_rsrc_t rsa = make_rsrc(Abase, 0xffffffffu);
  __amdgpu_buffer_rsrc_t rsb = make_rsrc(g.seg[0].B + (long long)col0 * g.ldb, 0xffffffffu);
  uint32_t ka = 0, kb = 0;
  constexpr int kStepsPerBlk = 256 / C::BK;
  const long long a_blk_bytes = g.a_blk * 2;
  int ablk_left = kStepsPerBlk;
  auto advance_a = [&]() {
    ka += C::BK * 2;
    if (--ablk_left == 0) {
      ablk_left = kStepsPerBlk;
      if (a_blk_bytes != 0) {                          // next column block of A: re-base the descriptor
        Abase += a_blk_bytes;
        rsa = make_rsrc(Abase, 0xffffffffu);
        ka = 0;
      }
    }
    if (--la == 0 && sa + 1 < g.nseg) {
      ++sa;
      la = g.seg[sa].K / C::BK;
      Abase = (const char*)(g.seg[sa].A + (long long)row0 * g.lda);
      rsa = make_rsrc(Abase, 0xffffffffu);
      ka = 0;
      ablk_left = kStepsPerBlk;
    }
  };
  auto advance_b = [&]() {
    kb += C::BK * 2;
    if (--lb == 0 && sb + 1 < g.nseg) {
      ++sb;
      lb = g.seg[sb].K / C::BK;
      rsb = make_rsrc(g.seg[sb].B + (long long)col0 * g.ldb, 0xffffffffu);
      kb = 0;
    }
  };
  auto load_lds = [&](const __amdgpu_buffer_rsrc_t& rs, char* lds, int idx, uint32_t off, uint32_t k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, FGRPO_LDS_PTR(lds + dst_w + idx * C::NW * C::RPI * C::ROWB), 16, (int)off, (int)k, 0, FGRPO_DMA_AUX);
  };
  auto issue_a = [&](char* lds, int idx) {
    load_lds(rsa, lds, idx, aoff[idx], ka);
    if (idx == C::PA - 1) advance_a();
  };
  auto issue_b = [&](char* lds, int idx) {
    if (idx == 0) advance_b();
    load_lds(rsb, lds, idx, boff[idx], kb);
  };
  if constexpr (MODE == 1) {                    // the MODE 2 call issued these
    if (nk_total > 0) advance_a();
    if (nk_total > 1) advance_a();
  } else {
    if constexpr (MODE == 0) FGRPO_WAIT_VMCNT(0);      // the caller's own loads must not be mistaken for ours
    if (nk_total > 0) {
      static_for<NB>([&](auto q) { load_lds(rsb, smem + mi16_b_buf(0) * kOpBytes<C>, decltype(q)::value, boff[decltype(q)::value], 0); });
      static_for<C::PA>([&](auto q) { issue_a(smem, decltype(q)::value); });
    }
    if (nk_total > 1) static_for<C::PA>([&](auto q) { issue_a(smem + kOpBytes<C>, decltype(q)::value); });
    if constexpr (MODE == 2) return;
  }

  // fragments: lane l reads row (l % 16) of a 16-row block and the 16-byte chunk 4*k2 + l/16 of its 64-wide K slice (16
  // consecutive rows at one chunk index: conflict-free under the swizzle)
  const int sw16 = lds_swizzle<C, true>(lane & 15);
  const int fa16 = (wm * C::WTM + (lane & 15)) * C::ROWB, fb16 = (wn * 16 * NB + (lane & 15)) * C::ROWB;
  int fc16[2];
#pragma unroll
  for (int k2 = 0; k2 < 2; ++k2) fc16[k2] = ((4 * k2 + (lane >> 4)) ^ sw16) * 16;
  early_barrier_pipeline16<C, NB, 1, 1, MODE == 1, true>(
      nk_total, smem, acc, true, issue_a, issue_b,
      [&](const char* st, auto i, auto kk) {
        constexpr int kkv = decltype(kk)::value;
        return lds_read_b128_asm<(decltype(i)::value * 32 + 16 * (kkv & 1)) * C::ROWB>(lds_addr(st) + fa16 + fc16[kkv >> 1]);
      },
      [&](const char* st, auto jc, auto k2) {
        constexpr int jcv = decltype(jc)::value;
        return lds_read_b128_asm<16 * jcv * C::ROWB>(lds_addr(st) + fb16 + fc16[decltype(k2)::value]);
      });
}

template <class C, int MODE = 0, bool MI16 = false, int NB = 4>
__device__ __forceinline__ void gemm_mainloop_dma(const GemmOperands& g, int row0, int col0, char* smem,
                                                  f32x16_t (&acc)[C::TM][C::TN]) {
  static_assert(MODE == 0 || kSplitPrologue<C>, "split prologue needs the two-buffer schedule");
  if constexpr (MI16) {
    gemm_mainloop_dma16<C, MODE, NB>(g, row0, col0, smem, acc);
    return;
  }
  constexpr int D = C::NSTAGE - 1;              // K steps of loads in flight
  constexpr int LPT = C::PA + C::PB;            // loads per thread per K step
  static_assert(D >= 1 && D <= 4 && LPT * (D - 1) < 64, "pipeline depth");
  // The per-lane offsets below are cheap to derive and expensive to keep: a caller that runs this loop once per
  // tile with an epilogue in between would otherwise carry two dozen loop-invariant registers through that
  // epilogue.  The empty asm makes the thread id opaque, so they are recomputed per call.
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wavefront-uniform: LDS targets stay scalar
  const int wm = wave / C::WN, wn = wave % C::WN;

  // loader: instruction i of this wavefront covers tile rows (i*NW + wave)*RPI ..
  const int lrow = lane / C::CPR, lpc = lane % C::CPR;
  uint32_t aoff[C::PA], boff[C::PB];
  const int amax = g.M - 1 - row0, bmax = g.N - 1 - col0;
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;            // row inside the tile (decides the swizzle)
    const int r = rt < amax ? rt : amax;                          // row actually read
    aoff[i] = (uint32_t)((long long)r * g.lda * 2 + ((lpc ^ lds_swizzle<C>(rt)) * 16));
  }
#pragma unroll
  for (int i = 0; i < C::PB; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;
    const int r = rt < bmax ? rt : bmax;
    boff[i] = (uint32_t)((long long)r * g.ldb * 2 + ((lpc ^ lds_swizzle<C>(rt)) * 16));
  }
  const int dst_a = wave * C::RPI * C::ROWB;                      // + i * NW*RPI*ROWB, wave-uniform
  const int dst_b = C::BM * C::ROWB + dst_a;
  // fragment reads
  const int sw = lds_swizzle<C>(lane & 31);
  const int fr_a = (wm * C::WTM + (lane & 31)) * C::ROWB;
  const int fr_b = C::BM * C::ROWB + (wn * C::WTN + (lane & 31)) * C::ROWB;
  int fr_c[C::BK / 16];
#pragma unroll
  for (int kk = 0; kk < C::BK / 16; ++kk) fr_c[kk] = ((kk * 2 + (lane >> 5)) ^ sw) * 16;

  int nk_total = 0;
  for (int s = 0; s < g.nseg; ++s) nk_total += g.seg[s].K / C::BK;

  // Issue cursor over (segment, k).  The loads are buffer loads: a 128-bit descriptor per operand (base = first
  // row of the tile in the current segment / column block), the lane's constant byte offset in a VGPR and the
  // running K offset in an SGPR, so that issuing a load costs two scalar instructions and no vector arithmetic.
  int iseg = 0, ileft = g.seg[0].K / C::BK;
  const char* Abase = (const char*)(g.seg[0].A + (long long)row0 * g.lda);
  const char* Bbase = (const char*)(g.seg[0].B + (long long)col0 * g.ldb);
  __amdgpu_buffer_rsrc_t rsa = make_rsrc(Abase, 0xffffffffu);
  __amdgpu_buffer_rsrc_t rsb = make_rsrc(Bbase, 0xffffffffu);
  uint32_t ka = 0, kb = 0;                            // byte offset of the K slice being issued
  // after the last load of a K step: next K slice, next 256-column block of a blocked A, next segment
  constexpr int kStepsPerBlk = 256 / C::BK;
  const long long a_blk_bytes = g.a_blk * 2;
  int ablk_left = kStepsPerBlk;
  auto advance = [&]() {
    ka += C::BK * 2;
    kb += C::BK * 2;
    if (--ablk_left == 0) {
      ablk_left = kStepsPerBlk;
      if (a_blk_bytes != 0) {                          // next column block of A: re-base the descriptor
        Abase += a_blk_bytes;
        rsa = make_rsrc(Abase, 0xffffffffu);
        ka = 0;
      }
    }
    if (--ileft == 0 && iseg + 1 < g.nseg) {
      ++iseg;
      ileft = g.seg[iseg].K / C::BK;
      Abase = (const char*)(g.seg[iseg].A + (long long)row0 * g.lda);
      Bbase = (const char*)(g.seg[iseg].B + (long long)col0 * g.ldb);
      rsa = make_rsrc(Abase, 0xffffffffu);
      rsb = make_rsrc(Bbase, 0xffffffffu);
      ka = kb = 0;
      ablk_left = kStepsPerBlk;
    }
  };
  // One load of the current issue step (idx < PA: operand A, else B); the last one advances the cursor.
  auto issue_one = [&](int stage, int idx) {
    char* base = smem + stage * C::STAGE;
    if (idx < C::PA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, FGRPO_LDS_PTR(base + dst_a + idx * C::NW * C::RPI * C::ROWB), 16,
                                               (int)aoff[idx], (int)ka, 0, FGRPO_DMA_AUX);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, FGRPO_LDS_PTR(base + dst_b + (idx - C::PA) * C::NW * C::RPI * C::ROWB),
                                               16, (int)boff[idx - C::PA], (int)kb, 0, FGRPO_DMA_AUX);
    if (idx == LPT - 1) advance();
  };
  auto issue = [&](int stage) {
#pragma unroll
    for (int i = 0; i < LPT; ++i) issue_one(stage, i);
  };

  int issued = 0;
  if constexpr (MODE == 1) {                    // step 0 is already on its way into buffer 0
    if (nk_total > 0) {
      advance();
      issued = 1;
    }
  } else {
    // loads issued before this call (by the caller's epilogue) must not be mistaken for ours
    FGRPO_WAIT_VMCNT(0);
    for (; issued < D && issued < nk_total; ++issued) issue(issued);
    if constexpr (MODE == 2) return;
  }

  if constexpr (C::NSTAGE == 2 && (C::BK / 16) % 2 == 0) {
    early_barrier_pipeline<C, LPT, 1, 1>(
        nk_total, smem, acc, issue_one,
        [&](const char* st, auto i, auto kk) {
          return lds_read_b128_asm<decltype(i)::value * 32 * C::ROWB>(lds_addr(st) + fr_a + fr_c[decltype(kk)::value]);
        },
        [&](const char* st, auto j, auto kk) {
          return lds_read_b128_asm<decltype(j)::value * 32 * C::ROWB>(lds_addr(st) + fr_b + fr_c[decltype(kk)::value]);
        });
    return;
  }

  // The loads of a step are interleaved with its MFMAs (a burst right after the barrier would keep
  // every wavefront busy issuing addresses, about 40 cycles per load, before its first MFMA).
  // With three or more LDS buffers they are spread over the whole step; with two buffers over the
  // first half, so that the last one still has half a step to land.
  constexpr int kGroups = (C::BK / 16) * C::TM;                                  // MFMA groups (TN MFMAs each) per step
  constexpr int kSpreadG = (C::NSTAGE >= 3) ? kGroups : (kGroups / 2 > 0 ? kGroups / 2 : 1);
  constexpr int kPer = (LPT + kSpreadG - 1) / kSpreadG;                          // loads after each group
  constexpr bool kSpread = true;
  constexpr int KK = C::BK / 16;

  int cur = 0, nxt = D % C::NSTAGE;
  for (int kt = 0; kt < nk_total; ++kt) {
    const int rem = nk_total - 1 - kt;          // K steps after this one
    // wait until this step's loads have landed: at most min(rem, D-1) younger steps may stay in flight
    if (rem >= D - 1) {
      FGRPO_WAIT_VMCNT(LPT * (D - 1));
    } else if (D >= 3 && rem == 2) {
      FGRPO_WAIT_VMCNT(LPT * 2);
    } else if (D >= 2 && rem == 1) {
      FGRPO_WAIT_VMCNT(LPT * 1);
    } else {
      FGRPO_WAIT_VMCNT(0);
    }
    wg_barrier();   // everyone's part of step kt is in LDS; everyone is done reading step kt-1
    const bool more = issued < nk_total;
    if (more) ++issued;
    if (!kSpread && more) issue(nxt);
    const char* st = smem + cur * C::STAGE;
    bf16x8_t af[2][C::TM], bf[2][C::TN];
#pragma unroll
    for (int i = 0; i < C::TM; ++i) af[0][i] = FGRPO_LDFRAG(st + fr_a + i * 32 * C::ROWB + fr_c[0]);
#pragma unroll
    for (int j = 0; j < C::TN; ++j) bf[0][j] = FGRPO_LDFRAG(st + fr_b + j * 32 * C::ROWB + fr_c[0]);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if (kk + 1 < KK) {   // next sub-step's fragments fly while this one multiplies
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
          af[(kk + 1) & 1][i] = FGRPO_LDFRAG(st + fr_a + i * 32 * C::ROWB + fr_c[kk + 1]);
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
          bf[(kk + 1) & 1][j] = FGRPO_LDFRAG(st + fr_b + j * 32 * C::ROWB + fr_c[kk + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < C::TM; ++i) {
#pragma unroll
        for (int j = 0; j < C::TN; ++j) acc[i][j] = FGRPO_MFMA(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
        if (kSpread && more) {
#pragma unroll
          for (int q = 0; q < kPer; ++q)
            if ((kk * C::TM + i) * kPer + q < LPT) issue_one(nxt, (kk * C::TM + i) * kPer + q);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    cur = (cur + 1 == C::NSTAGE) ? 0 : cur + 1;
    nxt = (nxt + 1 == C::NSTAGE) ? 0 : nxt + 1;
  }
  wg_barrier();   // LDS may be reused by the caller
}

// ---------------------------------------------------------------------------
// Direct-to-LDS main loop with one K step of look-ahead (NSTAGE >= 4).
// The barrier that opens step kt also guarantees that step kt+1 is complete in
// LDS, so the first fragments of step kt+1 are read *before* the next barrier,
// while the last MFMAs of step kt run: no LDS latency is exposed after a
// barrier.  Per step: fragments double-buffered in registers, the loads of step
// kt+NSTAGE-1 spread one per TN MFMAs, one vmcnt wait + one s_barrier.
// ---------------------------------------------------------------------------
template <class C>
__device__ __forceinline__ void gemm_mainloop_la(const GemmOperands& g, int row0, int col0, char* smem,
                                                 f32x16_t (&acc)[C::TM][C::TN]) {
  constexpr int NST = C::NSTAGE;
  constexpr int LPT = C::PA + C::PB;            // loads per thread per K step
  constexpr int KK = C::BK / 16;
  static_assert(NST >= 4 && NST <= 6, "look-ahead pipeline needs 4..6 LDS buffers");
  static_assert(LPT <= KK * C::TM, "one load slot per TN MFMAs");
  static_assert(LPT * (NST - 3) < 64, "vmcnt range");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WN, wn = wave % C::WN;

  const int lrow = lane / C::CPR, lpc = lane % C::CPR;
  uint32_t aoff[C::PA], boff[C::PB];
  const int amax = g.M - 1 - row0, bmax = g.N - 1 - col0;
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;
    const int r = rt < amax ? rt : amax;
    aoff[i] = (uint32_t)((long long)r * g.lda * 2 + ((lpc ^ lds_swizzle<C>(rt)) * 16));
  }
#pragma unroll
  for (int i = 0; i < C::PB; ++i) {
    const int rt = (i * C::NW + wave) * C::RPI + lrow;
    const int r = rt < bmax ? rt : bmax;
    boff[i] = (uint32_t)((long long)r * g.ldb * 2 + ((lpc ^ lds_swizzle<C>(rt)) * 16));
  }
  const int dst_a = wave * C::RPI * C::ROWB;
  const int dst_b = C::BM * C::ROWB + dst_a;
  const int sw = lds_swizzle<C>(lane & 31);
  const int fr_a = (wm * C::WTM + (lane & 31)) * C::ROWB;
  const int fr_b = C::BM * C::ROWB + (wn * C::WTN + (lane & 31)) * C::ROWB;
  int fr_c[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) fr_c[kk] = ((kk * 2 + (lane >> 5)) ^ sw) * 16;

  // segment table in registers (no scalar memory traffic inside the loop)
  const char* segA[3];
  const char* segB[3];
  int segN[3];
  int nk_total = 0;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const bool on = s < g.nseg;
    segA[s] = on ? (const char*)(g.seg[s].A + (long long)row0 * g.lda) : nullptr;
    segB[s] = on ? (const char*)(g.seg[s].B + (long long)col0 * g.ldb) : nullptr;
    segN[s] = on ? g.seg[s].K / C::BK : 0;
    nk_total += segN[s];
  }
  int iseg = 0, ileft = segN[0];
  const char* Ai = segA[0];
  const char* Bi = segB[0];
  auto issue_one = [&](int stage, int idx) {
    char* base = smem + stage * C::STAGE;
    if (idx < C::PA)
      __builtin_amdgcn_global_load_lds(FGRPO_GLOBAL_PTR(Ai + aoff[idx]),
                                       FGRPO_LDS_PTR(base + dst_a + idx * C::NW * C::RPI * C::ROWB), 16, 0, FGRPO_DMA_AUX);
    else
      __builtin_amdgcn_global_load_lds(FGRPO_GLOBAL_PTR(Bi + boff[idx - C::PA]),
                                       FGRPO_LDS_PTR(base + dst_b + (idx - C::PA) * C::NW * C::RPI * C::ROWB), 16, 0,
                                       FGRPO_DMA_AUX);
    if (idx == LPT - 1) {
      Ai += C::BK * 2;
      Bi += C::BK * 2;
      if (--ileft == 0) {
        ++iseg;
        const bool s1 = (iseg == 1);
        ileft = s1 ? segN[1] : segN[2];
        Ai = s1 ? segA[1] : segA[2];
        Bi = s1 ? segB[1] : segB[2];
      }
    }
  };
  // At most `tiles` K steps of this thread's loads stay in flight.  The look-ahead fragment reads
  // issued half a step earlier are certainly back by now; saying so (lgkmcnt 0) lets the compiler
  // start the next step's MFMAs without waiting for the reads it issues at the top of that step.
  auto wait_allow = [&](int tiles) {
    if (tiles >= NST - 3) {
      FGRPO_WAIT_VMCNT_LGKM0(LPT * (NST - 3));
    } else if (NST >= 6 && tiles == 2) {
      FGRPO_WAIT_VMCNT_LGKM0(LPT * 2);
    } else if (NST >= 5 && tiles == 1) {
      FGRPO_WAIT_VMCNT_LGKM0(LPT * 1);
    } else {
      FGRPO_WAIT_VMCNT_LGKM0(0);
    }
  };

  FGRPO_WAIT_VMCNT(0);   // the caller's own loads must not be mistaken for ours
  int issued = 0;
  for (; issued < NST - 1 && issued < nk_total; ++issued) {
#pragma unroll
    for (int idx = 0; idx < LPT; ++idx) issue_one(issued, idx);
  }
  // steps 0 and 1 must be in LDS before the first barrier
  {
    int allow = issued - 2;
    wait_allow(allow < 0 ? 0 : allow);
  }
  wg_barrier();

  bf16x8_t af[2][C::TM], bf[2][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i) af[0][i] = FGRPO_LDFRAG(smem + fr_a + i * 32 * C::ROWB + fr_c[0]);
#pragma unroll
  for (int j = 0; j < C::TN; ++j) bf[0][j] = FGRPO_LDFRAG(smem + fr_b + j * 32 * C::ROWB + fr_c[0]);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): enter the loop with these fragments in registers

  int cur = 0;                 // stage of step kt
  int nst = (NST - 1) % NST;   // stage that the loads issued during step kt go to (= stage of step kt-1)
  for (int kt = 0; kt < nk_total; ++kt) {
    const bool more = issued < nk_total;       // a step to issue during this one
    const bool has_next = kt + 1 < nk_total;
    const char* st = smem + cur * C::STAGE;
    const int nx = (cur + 1 == NST) ? 0 : cur + 1;
    const char* sn = smem + nx * C::STAGE;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int b = kk & 1;
      // fragments of the next sub-step (or of the next K step's first sub-step) fly under these MFMAs
      if (kk + 1 < KK) {
#pragma unroll
        for (int i = 0; i < C::TM; ++i) af[b ^ 1][i] = FGRPO_LDFRAG(st + fr_a + i * 32 * C::ROWB + fr_c[kk + 1]);
#pragma unroll
        for (int j = 0; j < C::TN; ++j) bf[b ^ 1][j] = FGRPO_LDFRAG(st + fr_b + j * 32 * C::ROWB + fr_c[kk + 1]);
      } else if (has_next) {
#pragma unroll
        for (int i = 0; i < C::TM; ++i) af[b ^ 1][i] = FGRPO_LDFRAG(sn + fr_a + i * 32 * C::ROWB + fr_c[0]);
#pragma unroll
        for (int j = 0; j < C::TN; ++j) bf[b ^ 1][j] = FGRPO_LDFRAG(sn + fr_b + j * 32 * C::ROWB + fr_c[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < C::TM; ++i) {
#pragma unroll
        for (int j = 0; j < C::TN; ++j) acc[i][j] = FGRPO_MFMA(af[b][i], bf[b][j], acc[i][j]);
        if (kk * C::TM + i < LPT) {
          if (more) issue_one(nst, kk * C::TM + i);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    static_assert(KK % 2 == 0, "fragment buffer parity must return to 0 every K step");
    if (more) ++issued;
    // before the next step starts, step kt+2 must be complete (step kt+1 already is)
    {
      int allow = issued - (kt + 3);
      wait_allow(allow < 0 ? 0 : allow);
    }
    wg_barrier();
    cur = nx;
    nst = (nst + 1 == NST) ? 0 : nst + 1;
  }
}

// ---------------------------------------------------------------------------
// Main loop for operands stored "K-major" (the contraction index is the ROW
// index: X[k][m], m contiguous), as dLogits [token][vocab], hidden [token][H] and
// W [vocab][H] are when the contraction runs over tokens or vocabulary.  No
// transposed copy is made: the tile goes to LDS as it lies in memory (two k rows
// of 256 columns per wavefront-wide direct-to-LDS load) and the MFMA operand is
// assembled by ds_read_b64_tr_b16, which hands lane i of every 16-lane group the
// i-th column of a 4 (k) x 16 (m) block whose rows are addressed by lanes
// 4e .. 4e+3.  Two such reads give the eight consecutive k values of a
// 32x32x16 operand.  16-byte chunks of a row are XOR-swizzled with 4*(k%4) so
// that the four rows one read touches fall into different banks.
// Either operand may instead be K-contiguous (X[m][k]) and is then handled as in
// gemm_mainloop_dma.  One segment, BM = BN = 256, BK = 64, two LDS buffers.
// ---------------------------------------------------------------------------
// Chunk-index XOR of k row `kr` of a K-major LDS tile (512-byte rows).  The transposing reads of a 16-lane group take
// rows k .. k+3: 4*(k%4) spreads the four; two groups of a pass read the same columns of rows k and k + 8: bit 3 of k
// moves them 32 bytes apart.
__device__ __forceinline__ int km_swizzle(int kr) { return ((kr & 3) << 2) | (((kr >> 3) & 1) << 1); }
template <class C, bool AKM, bool BKM, bool AHEAD = true>
__device__ __forceinline__ void gemm_mainloop_km(const GemmOperands& g, int row0, int col0, char* smem,
                                                 f32x16_t (&acc)[C::TM][C::TN]) {
  static_assert(kMi16<C> && C::BM == 256 && C::BN == 256, "K-major loop: the 8-wavefront 256x256x64 tile");
  constexpr int KROWB = 512;                    // bytes of one k row of a K-major tile (256 columns)
  constexpr int OP = kOpBytes<C>;               // bytes of one operand's buffer (32 KiB either way)
  static_assert(C::ROWB == 128 && OP == C::BK * KROWB, "buffer size");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wavefront-uniform
  int wm, wn;
  wave_coords<C, true>(wave, wm, wn);

  // ---- loader ------------------------------------------------------------------------------
  uint32_t aoff[C::PA], boff[C::PB];            // per-lane byte offset of each load inside the step's slice
  {
    const int lrow = lane / C::CPR, lpc = lane % C::CPR;
    const int amax = g.M - 1 - row0, bmax = g.N - 1 - col0;
#pragma unroll
    for (int i = 0; i < C::PA; ++i) {
      if constexpr (AKM) {
        const int kr = (i * C::NW + wave) * 2 + (lane >> 5);
        aoff[i] = (uint32_t)((long long)kr * g.lda * 2) + (uint32_t)((((lane & 31) ^ km_swizzle(kr))) * 16);
      } else {
        const int rt = (i * C::NW + wave) * C::RPI + lrow;
        const int r = rt < amax ? rt : amax;
        aoff[i] = (uint32_t)((long long)r * g.lda * 2 + ((lpc ^ lds_swizzle<C, true>(rt)) * 16));
      }
    }
#pragma unroll
    for (int i = 0; i < C::PB; ++i) {
      if constexpr (BKM) {
        const int kr = (i * C::NW + wave) * 2 + (lane >> 5);
        boff[i] = (uint32_t)((long long)kr * g.ldb * 2) + (uint32_t)((((lane & 31) ^ km_swizzle(kr))) * 16);
      } else {
        const int rt = (i * C::NW + wave) * C::RPI + lrow;
        const int r = rt < bmax ? rt : bmax;
        boff[i] = (uint32_t)((long long)r * g.ldb * 2 + ((lpc ^ lds_swizzle<C, true>(rt)) * 16));
      }
    }
  }
  // Buffer loads: the lane's constant byte offset travels in a VGPR, everything that moves is scalar.
  //  * K-contiguous operand: descriptor on the tile's first row, K offset in an SGPR (re-based per 256-column
  //    block when A is column-blocked);
  //  * K-major operand: descriptor re-based on the first k row of every step, with num_records = the bytes of
  //    the k rows that exist from there on, so rows past the end of the contraction read as zero.
  // K-major A kept in 256-column blocks: tile column block row0/256 is one [K][256] matrix of its own
  const char* Ap = AKM ? (const char*)(g.seg[0].A + (g.a_blk ? (long long)(row0 >> 8) * g.a_blk : (long long)row0))
                       : (const char*)(g.seg[0].A + (long long)row0 * g.lda);
  const char* Bp = BKM ? (const char*)(g.seg[0].B + col0) : (const char*)(g.seg[0].B + (long long)col0 * g.ldb);
  const long long lda2 = g.lda * 2, ldb2 = g.ldb * 2;
  long long a_rem = (AKM && g.ka_valid > 0) ? g.ka_valid : (1LL << 40);   // k rows of A that exist from Ap on
  long long b_rem = (BKM && g.kb_valid > 0) ? g.kb_valid : (1LL << 40);
  // bytes from a descriptor's base (first k row of the step, first column of the tile) to the end of the operand:
  // `rows` k rows of ld2 bytes, less the tile's column offset - the last tile of a row width that is not a multiple
  // of 256 reads past the end of every row, which must not carry past the end of the last one
  auto bytes_of = [](long long rows, long long ld2, long long col_bytes) -> uint32_t {
    if (rows <= 0) return 0u;
    const long long bts = rows * ld2 - col_bytes;
    if (bts <= 0) return 0u;
    return (rows > (1LL << 31) || bts > 0xffffffffLL) ? 0xffffffffu : (uint32_t)bts;
  };
  const long long a_col = (AKM && g.a_blk == 0) ? (long long)row0 * 2 : 0, b_col = BKM ? (long long)col0 * 2 : 0;
  __amdgpu_buffer_rsrc_t rsa = make_rsrc(Ap, AKM ? bytes_of(a_rem, lda2, a_col) : 0xffffffffu);
  __amdgpu_buffer_rsrc_t rsb = make_rsrc(Bp, BKM ? bytes_of(b_rem, ldb2, b_col) : 0xffffffffu);
  uint32_t ka = 0, kb = 0;                      // running K byte offset of a K-contiguous operand
  const int dst_w = wave * 1024;                // both layouts: one load fills 1 KiB, loads i are NW KiB apart

  // run list (A K-major; B either way): the cursors walk the listed K steps; the compute side never
  // knows, it consumes LDS buffers in the order they were filled
  const int* runs = AKM ? g.k_runs : nullptr;
  const int n_runs = runs ? runs[0] : 0;
  const int nk_total = runs ? runs[1] : g.seg[0].K / C::BK;
  int run_idx = 0, run_left = 0, cur_step = 0;
  auto skip_a = [&](long long steps) {           // A's cursor that many K steps on (A K-major)
    Ap += steps * C::BK * lda2;
    a_rem -= steps * C::BK;
    rsa = make_rsrc(Ap, bytes_of(a_rem, lda2, a_col));
  };
  auto skip_b = [&](long long steps) {
    if constexpr (BKM) {
      Bp += steps * C::BK * ldb2;
      b_rem -= steps * C::BK;
      rsb = make_rsrc(Bp, bytes_of(b_rem, ldb2, b_col));
    } else {
      kb += (uint32_t)steps * C::BK * 2;
    }
  };
  if (runs != nullptr && n_runs > 0) {
    cur_step = runs[2];
    run_left = runs[2 + kRunCap] - cur_step;
    skip_a(cur_step);
    skip_b(cur_step);
  }
  const long long a_blk_bytes = (!AKM) ? g.a_blk * 2 : 0;
  int ablk_left = 256 / C::BK;
  int jump_a = 1, jump_b = 1;                    // K steps from the step A's cursor came from to where it is, and from the one before it
  auto load_lds = [&](const __amdgpu_buffer_rsrc_t& rs, char* lds, int idx, uint32_t off, uint32_t k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, FGRPO_LDS_PTR(lds + dst_w + idx * C::NW * 1024), 16, (int)off, (int)k, 0, FGRPO_DMA_AUX);
  };
  auto issue_a = [&](char* lds, int idx) {
    load_lds(rsa, lds, idx, aoff[idx], ka);
    if (idx == C::PA - 1) {                      // next K step
      if constexpr (AKM) {
        int jump = 1;
        if (runs != nullptr && --run_left == 0 && run_idx + 1 < n_runs) {   // this run is done: on to the next
          ++run_idx;
          const int s = runs[2 + run_idx];
          jump = s - cur_step;
          run_left = runs[2 + kRunCap + run_idx] - s;
        }
        cur_step += jump;
        jump_b = jump_a;                         // B follows a step behind
        jump_a = jump;
        skip_a(jump);
      } else {
        ka += C::BK * 2;
        if (--ablk_left == 0) {
          ablk_left = 256 / C::BK;
          if (a_blk_bytes != 0) {                // K-contiguous A kept in 256-column blocks: next block
            Ap += a_blk_bytes;
            rsa = make_rsrc(Ap, 0xffffffffu);
            ka = 0;
          }
        }
      }
    }
  };
  auto issue_b = [&](char* lds, int idx) {
    if (idx == 0) skip_b(AKM ? jump_b : 1);
    load_lds(rsb, lds, idx, boff[idx], kb);
  };

  // ---- fragment addressing -------------------------------------------------------------------
  // K-contiguous operand: row l % 16 of a 16-row block, chunk 4*k2 + l/16.  K-major operand:
  // lane l = 16*g + j supplies row k = 32*k2 + 8*g + 4*r + j/4 (r = 0, 1: the two transposing reads) and the 8 bytes
  // at column 4*(j%4) of the 16-column block; every 16-lane group gets its own eight k values of the slice.
  const int sw16 = lds_swizzle<C, true>(lane & 15);
  const int fa16 = (wm * C::WTM + (lane & 15)) * C::ROWB, fb16 = (wn * C::WTN + (lane & 15)) * C::ROWB;
  int fc16[2];
#pragma unroll
  for (int k2 = 0; k2 < 2; ++k2) fc16[k2] = ((4 * k2 + (lane >> 4)) ^ sw16) * 16;
  const int j4 = (lane & 15) >> 2, g16 = lane >> 4;
  const int k16_row = (8 * g16 + j4) * KROWB;                      // + (32*k2 + 4*r) * KROWB
  const int k16_sw = (j4 << 2) | ((g16 & 1) << 1);                 // km_swizzle of the lane's rows
  const int k16_cl = (lane & 3) >> 1;                              // chunk of the lane's column inside a 16-column block
  auto km16_off = [&](int block_col0) { return ((((block_col0 >> 3) + k16_cl) ^ k16_sw) << 4) + (lane & 1) * 8; };
  int fka16[C::TM][2], fkb16[2 * C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int rh = 0; rh < 2; ++rh) fka16[i][rh] = k16_row + km16_off(wm * C::WTM + i * 32 + 16 * rh);
#pragma unroll
  for (int jc = 0; jc < 2 * C::TN; ++jc) fkb16[jc] = k16_row + km16_off(wn * C::WTN + (jc >> 1) * 32 + 16 * (jc & 1));

  FGRPO_WAIT_VMCNT(0);
  if (nk_total > 0) {
    static_for<C::PB>([&](auto q) { load_lds(rsb, smem + mi16_b_buf(0) * OP, decltype(q)::value, boff[decltype(q)::value], kb); });
    static_for<C::PA>([&](auto q) { issue_a(smem, decltype(q)::value); });
  }
  if (nk_total > 1) static_for<C::PA>([&](auto q) { issue_a(smem + OP, decltype(q)::value); });
  early_barrier_pipeline16<C, 4, AKM ? 2 : 1, BKM ? 2 : 1, false, AHEAD>(
      nk_total, smem, acc, wave_is_live<C>(g, row0, col0, wm, wn), issue_a, issue_b,
      [&](const char* st, auto ic, auto kc) -> bf16x8_t {
        constexpr int i = decltype(ic)::value, kk = decltype(kc)::value, k2 = kk >> 1, rh = kk & 1;
        if constexpr (AKM)
          return lds_read_tr_pair<(32 * k2) * KROWB, (32 * k2 + 4) * KROWB>(lds_addr(st) + fka16[i][rh]);
        else
          return lds_read_b128_asm<(i * 32 + 16 * rh) * C::ROWB>(lds_addr(st) + fa16 + fc16[k2]);
      },
      [&](const char* st, auto jcc, auto k2c) -> bf16x8_t {
        constexpr int jc = decltype(jcc)::value, k2 = decltype(k2c)::value;
        if constexpr (BKM)
          return lds_read_tr_pair<(32 * k2) * KROWB, (32 * k2 + 4) * KROWB>(lds_addr(st) + fkb16[jc]);
        else
          return lds_read_b128_asm<((jc >> 1) * 32 + 16 * (jc & 1)) * C::ROWB>(lds_addr(st) + fb16 + fc16[k2]);
      });
}

template <class C>
__device__ __forceinline__ void run_mainloop(const GemmOperands& g, int row0, int col0, char* smem,
                                             f32x16_t (&acc)[C::TM][C::TN]) {
  if constexpr (C::DMA && C::NSTAGE >= 4)
    gemm_mainloop_la<C>(g, row0, col0, smem, acc);
  else if constexpr (C::DMA)
    gemm_mainloop_dma<C>(g, row0, col0, smem, acc);
  else
    gemm_mainloop<C>(g, row0, col0, smem, acc);
}

// Work-groups are handed to the 8 XCDs round-robin (block b runs on XCD b % 8)
// and each XCD has a private L2.  Remap so that every XCD walks one contiguous
// range of logical tile ids; neighbouring logical ids share operand panels.
__device__ __forceinline__ int xcd_contiguous_id(int bid, int nblocks) {
  const int q = nblocks >> 3, rem = nblocks & 7;
  const int xcd = bid & 7, idx = bid >> 3;
  return xcd * q + (xcd < rem ? xcd : rem) + idx;
}

}  // namespace fgrpo
