// dK / dV of the packed attention with one wavefront per SIMD and no barrier in its loop (head dimension HD = 128 or
// 64).  A work-group owns 64 keys of one K/V head (32 at HD = 64, where two
// work-groups then share a CU); its four wavefronts deal the work on those keys among themselves -
// item n = (32 queries, query head) goes to wavefront n % 4 - and each walks its items alone: it brings the item's
// Q / dO rows into two LDS buffers of its own (global -> LDS, two items ahead), waits for nothing but its own loads,
// and keeps both accumulators for all 64 keys (256 accumulation registers at HD = 128).  The four accumulator sets are
// added in a fixed order at the end, through LDS: bit-reproducible, no atomics.
//
// Why this shape.  The paired kernel (varlen_attn_dkv2_kernel) tiles 128 keys with eight wavefronts that share every
// Q / dO tile: a barrier of all eight and three LDS round trips per 32 queries, 0.40 of the matrix pipe at its clock,
// and 512 threads x 128 keys x all query heads of a group is a coarse unit: at 12345 tokens and 2 K/V heads it is 194
// work-groups on 256 CUs, each a chain of (query heads x steps).  Here every fragment read from LDS feeds TWO matrix
// instructions (64 keys), so LDS carries half the bytes per product, the chain of a work-group is dealt to four
// independent wavefronts, and units of 64 keys fill the device four times as finely.  The price is that a
// wavefront's tile serves only itself: 32 queries x 64 keys per 16 KiB through the L2, 32 B/clk and CU at full matrix
// rate, of the ~70 that direct-to-LDS loads sustain.
//
// Measured, dQ + dK/dV, paired kernel -> this one on one box: 4 segments of 8192 tokens, 28 / 4 heads of 128:
// 7.20 -> 6.00 ms; 32768 tokens in segments of 128..1024, 12 / 2 heads of 128: 442 -> 393 us; 12345 such tokens, 14 / 2
// heads of 64: 245 -> 99 us; one segment of 8192 tokens, 14 / 2 heads of 64: 1222 -> 617 us.  It was faster
// at every size tried, so no rule picks between the two.  Counters at the long shape: matrix pipe 0.61 busy at 1.81
// GHz, the power limit; at the short ones the clock is 2.4 GHz and the pipe 0.38 busy: opening and closing a
// work-group and the masked items weigh there.
//
// Orientation and register permutation as in attn_kernels.h (S = Q K^T: a lane owns a key).  One item, with the
// vector work of one stage behind the matrix instructions of the next (a 32x32x16 instruction hides about 20 cycles
// of it):
//   S of key block 0             |
//   S of key block 1             | P = exp2(S c - lse) of key block 0
//   dP of both                   | P of key block 1
//   dV += P^T dO   (rows 0..7 of each lane's 16)  | dS = P (dP - delta) of rows 0..7
//   dK += dS^T Q   (rows 0..7)   | dS of rows 8..15
//   dK             (rows 8..15)  | Q loads of the item after next, into the rows just read
//   dV             (rows 8..15)  | its dO loads; first Q fragments of the next item on their way
// -delta enters as the addend of dP's first instruction.  K lives in registers (64 keys x HD), V in LDS, shared by
// the four wavefronts (both in registers would exceed the file beside the accumulators).
#pragma once
#include "attn_kernels.h"

#ifndef FGRPO_MFMA_VGPR_FORM
#error "compile this unit with -mllvm -amdgpu-mfma-vgpr-form=1 -DFGRPO_MFMA_VGPR_FORM=1: else the compiler overwrites the accumulators below"
#endif

#define FGRPO_LDS_AT(a) ((__attribute__((address_space(3))) void*)(uint32_t)(a))      // LDS pointer from a byte address

namespace fgrpo {

template <int HD>
constexpr int kDkv3Buf = 2 * kDkv3Rows * HD * 2 + 512;                 // Q | dO | lse | -delta of 32 queries
template <int HD>
constexpr int kDkv3SumStride = HD * 4 + 32;                            // fp32 row of the closing sum: the two lane halves (rows 4 apart) hit different banks
template <int HD, int KB>
constexpr int kDkv3LoopLds = 4 * 2 * kDkv3Buf<HD> + 32 * KB * HD * 2;
template <int HD, int KB>
constexpr int kDkv3Lds = kDkv3LoopLds<HD, KB> > 4 * 32 * KB * kDkv3SumStride<HD> ? kDkv3LoopLds<HD, KB> : 4 * 32 * KB * kDkv3SumStride<HD>;

// The accumulators live in fixed accumulation registers, a[16 n : 16 n + 15] for block n, named in the instructions:
// at HD = 128 they are all 256 of them, and a register allocator that may move or copy a block has nowhere to put it
// (left to it, the loop spilled 260 registers).  Every instruction lists the whole range as clobbered, so that the
// compiler keeps nothing of its own there across one of them; that it puts nothing there in between (a clobber does not
// reserve a register) takes -amdgpu-mfma-vgpr-form, and the build reads in the compiler's assembly that it did not.
// The compiler's hazard table does not see these instructions: the first one behind vector arithmetic that formed an
// operand carries two wait states, and two instructions on one block, KB * DB matrix instructions apart (eight at HD = 128,
// two at HD = 64), accumulate into the identical register range, an order the hardware keeps by itself.
#define FGRPO_DKV3_CLOBBER_64 \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
  "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
  "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
  "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63"
#define FGRPO_DKV3_CLOBBER_128 \
  FGRPO_DKV3_CLOBBER_64, \
  "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
  "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
  "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
  "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127"
#define FGRPO_DKV3_CLOBBER_256 \
  FGRPO_DKV3_CLOBBER_128, \
  "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
  "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
  "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
  "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", \
  "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
  "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", \
  "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
  "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
// NACC accumulation registers in use; FIRST: behind vector arithmetic
template <int NACC, int BLK, bool FIRST>
__device__ __forceinline__ void dkv3_mfma(u32x4_t a, u32x4_t b) {
  constexpr int r0 = 16 * BLK, r1 = r0 + 15;
  static_assert(r1 < NACC && (NACC == 64 || NACC == 128 || NACC == 256), "accumulator block");
#define FGRPO_DKV3_MFMA(clobber)                                                                                            \
  if constexpr (FIRST) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : clobber); \
  else asm volatile("v_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : clobber)
  if constexpr (NACC == 256) { FGRPO_DKV3_MFMA(FGRPO_DKV3_CLOBBER_256); }
  else if constexpr (NACC == 128) { FGRPO_DKV3_MFMA(FGRPO_DKV3_CLOBBER_128); }
  else { FGRPO_DKV3_MFMA(FGRPO_DKV3_CLOBBER_64); }
#undef FGRPO_DKV3_MFMA
}
template <int NACC, int REG>
__device__ __forceinline__ void dkv3_acc_clear() {
  if constexpr (NACC == 256) asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(REG) : FGRPO_DKV3_CLOBBER_256);
  else if constexpr (NACC == 128) asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(REG) : FGRPO_DKV3_CLOBBER_128);
  else asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(REG) : FGRPO_DKV3_CLOBBER_64);
}
template <int REG, int OFF>
__device__ __forceinline__ void dkv3_acc_to_lds(uint32_t addr) {       // LDS instructions take their data from these registers directly
  static_assert(OFF >= 0 && OFF < 65536, "DS offset field");
  asm volatile("ds_write_b32 %0, a[%1] offset:%2" : : "v"(addr), "n"(REG), "n"(OFF) : "memory");
}

// Items of a key tile: 32-query blocks from q_begin on x query heads of the group
__device__ __forceinline__ int attn_key_items(int q_begin, int q_end, int G) {
  return q_end > q_begin ? (q_end - q_begin + kDkv3Rows - 1) / kDkv3Rows * G : 0;
}

// What a work-group walks: queries [q_begin, q_end) for the keys of `tile`
struct KeyWork {
  int tile, head, share, np;       // part `share` of the tile's np (see attn_deal); tile < 0: no work
  int q_begin, q_end, one_segment; // one segment holds every key of the tile
};
template <int kKeys>
__device__ __forceinline__ void attn_key_bounds(const AttnParams& p, int k0, int& q_begin, int& q_end, int& one_segment) {
  const int klast = min(k0 + kKeys, p.T) - 1, s0 = p.seg_start[k0];
  q_begin = max(p.causal ? k0 : s0, 0);                        // inside [0, T]
  q_end = min(p.seg_end[klast], p.T);
  one_segment = s0 == p.seg_start[klast];
}
// SPLIT launches: tiles in the order of attn_key_pick
template <int kKeys>
__device__ __forceinline__ KeyWork attn_key_deal(const AttnParams& p, int bid) {
  constexpr int kPer128 = 128 / kKeys, N = kAttnDealSlots / 64;
  const int lane = threadIdx.x & 63, xcd = bid & 7, slots = p.blocks_k >> 3;
  const int ntile = (p.T + kKeys - 1) / kKeys, n128 = (p.T + 127) / 128;
  int tile[N], head[N], q_begin[N], q_end[N], one_segment[N], items[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    tile[i] = items[i] = -1, head[i] = q_begin[i] = q_end[i] = one_segment[i] = 0;
    const int slot = 64 * i + lane;
    if (slot < slots) {
      const KeyPick pick = attn_key_pick(8 * slot + xcd, n128, kPer128, p.Hkv);
      const int t = pick.rank < 0 ? ntile : min(max(p.order_k[pick.rank], 0), n128 - 1) * kPer128 + pick.piece;
      if (t < ntile) {
        attn_key_bounds<kKeys>(p, t * kKeys, q_begin[i], q_end[i], one_segment[i]);
        tile[i] = t, head[i] = pick.head, items[i] = (attn_key_items(q_begin[i], q_end[i], p.Hq / p.Hkv) + 3) / 4;
      }
    }
  }
  const AttnDeal d = attn_deal(items, bid >> 3, slots, 1, p.extra_k, p.parts_k, p.per_k, p.deal_k);
  KeyWork out{-1, 0, d.share, d.np, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (d.slot >= 0 && d.slot / 64 == i) {
      const int l = d.slot % 64;
      out.tile = __builtin_amdgcn_readlane(tile[i], l), out.head = __builtin_amdgcn_readlane(head[i], l);
      out.q_begin = __builtin_amdgcn_readlane(q_begin[i], l), out.q_end = __builtin_amdgcn_readlane(q_end[i], l);
      out.one_segment = __builtin_amdgcn_readlane(one_segment[i], l);
    }
  return out;
}

// KB key blocks of 32 (2: one wavefront per SIMD; 1, head dimension 64: two).  SPLIT: a tile's items are dealt to the
// wavefronts of several work-groups (attn_key_deal), item n to wavefront n % (4 np) of them.
template <int HD, int KB, bool SPLIT>
__global__ __launch_bounds__(256, KB == 2 ? 1 : 2) void varlen_attn_dkv3_kernel(AttnParams p) {
  constexpr int kKeys = 32 * KB;
  constexpr int KS = HD / 16, DB = HD / 32, RB = HD * 2, kT = kDkv3Rows * RB, kBuf = kDkv3Buf<HD>;
  constexpr int QG = KS / 2, NG = KS / 2;              // row fragments of a half of S; groups of two k steps of dP
  constexpr int kSc = 2 * kT;                          // per-query scalars inside a buffer
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = lds_addr(smem);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = p.Hq / p.Hkv;
  KeyWork w{-1, 0, 0, 1, 0, 0, 0};
  if constexpr (SPLIT) {
    w = attn_key_deal<kKeys>(p, blockIdx.x);
    if (w.tile < 0) return;
    if (w.share == 0 && threadIdx.x == 0) p.key_info[w.tile * p.Hkv + w.head] = make_int2(w.np, blockIdx.x);
  } else {
    constexpr int kPer128 = 128 / kKeys;
    const int ntile = (p.T + kKeys - 1) / kKeys, n128 = (p.T + 127) / 128;
    const KeyPick pick = attn_key_pick(blockIdx.x, n128, kPer128, p.Hkv);
    if (pick.rank < 0) return;
    w.head = pick.head;
    w.tile = min(max(p.order_k[pick.rank], 0), n128 - 1) * kPer128 + pick.piece;      // clamped: the list may come from the caller
    if (w.tile >= ntile) return;
    attn_key_bounds<kKeys>(p, w.tile * kKeys, w.q_begin, w.q_end, w.one_segment);
  }
  const int hkv = w.head, share = w.share, np = w.np, k0 = w.tile * kKeys, klast = min(k0 + kKeys, p.T) - 1;
  const int q_begin = __builtin_amdgcn_readfirstlane(w.q_begin), q_end = __builtin_amdgcn_readfirstlane(w.q_end);
  // where one segment holds every key of the tile, queries from `q_full` on that are complete blocks see all of it
  const bool one_segment = __builtin_amdgcn_readfirstlane(w.one_segment);
  const int q_full = !one_segment ? 0x7fffffff : p.causal ? k0 + kKeys - 1 : q_begin;
  const int nqb = q_end > q_begin ? (q_end - q_begin + kDkv3Rows - 1) / kDkv3Rows : 0;
  const int NI = nqb * G;
  const int first = wave + 4 * share, stride = 4 * np;          // this wavefront's items
  const int stride_g = SPLIT ? stride % G : 4, stride_b = SPLIT ? stride / G : 0;      // ... in heads and query blocks

  // per-lane LDS addresses, this wavefront's buffer base included (see AttnLane)
  const uint32_t base_w = lds0 + wave * 2 * kBuf;
  const uint32_t v_delta = lds0 + 4 * 2 * kBuf - base_w;       // V tile minus the wavefront's base
  uint32_t rowc[KS], tr[DB][2];
  {
    const AttnLane<HD> L = attn_lane<HD>(lane);
#pragma unroll
    for (int st = 0; st < KS; ++st) rowc[st] = base_w + (uint32_t)L.rowc[st];
#pragma unroll
    for (int nb = 0; nb < DB; ++nb)
#pragma unroll
      for (int rd = 0; rd < 2; ++rd) tr[nb][rd] = base_w + (uint32_t)L.tr[nb][rd];
  }
  const uint32_t scl = base_w + kSc + h * 16;                  // + array * 128 + row group * 32

  const float c = p.scale * kLog2e;

  // accumulator blocks: dV[kb][nb] = kb DB + nb, dK behind them
  constexpr int kAccV = 0, kAccK = KB * DB, NACC = 2 * KB * DB * 16;

  // ---- loads of an item.  Instruction i of a tile fills its KiB i: RPI rows; lane l lands at 16 l of it, i.e. row
  // i RPI + l / (HD/8), chunk slot l % (HD/8), and fetches the chunk the swizzle puts there (four or two patterns).
  // Two items are in flight: a buffer's Q rows (with the per-query scalars) are free when the item's last Q^T
  // fragments have been read, three quarters through it, its dO rows an eighth later, and the item after next takes
  // them at once.
  constexpr int RPI = 1024 / RB, NLD = kDkv3Rows / RPI, NPAT = HD == 128 ? 4 : 2;
  const long long do_st = (long long)p.Hq * HD;
  uint32_t foq[NPAT], fod[NPAT];
#pragma unroll
  for (int i = 0; i < NPAT; ++i) {
    const int row = lane / (HD / 8), ch = (lane % (HD / 8)) ^ attn_swz<HD>(i * RPI + row);
    foq[i] = (uint32_t)((row * p.q_st + ch * 8) * 2);
    fod[i] = (uint32_t)((row * do_st + ch * 8) * 2);
  }
  const int sq = (int)(RPI * p.q_st * 2), sd = (int)(RPI * do_st * 2);
  // The walk goes from the last queries to the first, heads inside: work-groups on the same segment start at the same
  // rows and pass over them together, so that one L2 serves them all.  A step of it is a few additions.
  int g_f = first % G, qb_f = q_begin + (nqb - 1 - first / G) * kDkv3Rows;      // the item the loads are at
  const char* f_qp = (const char*)(p.q + (long long)(hkv * G + g_f) * p.q_sh + (long long)qb_f * p.q_st);
  const char* f_dp = (const char*)(p.dout + (long long)(hkv * G + g_f) * HD + (long long)qb_f * do_st);
  long long f_qb = ((long long)q_end - qb_f - 1) * p.q_st * 2 + RB;           // bytes to the end of the head's last row
  long long f_db = ((long long)q_end - qb_f - 1) * do_st * 2 + RB;
  // per-query scalars: the descriptors end with the queries of the head the item reads (the scalar offset counts in the
  // range check), so that rows past them, another segment's, read as zero like their Q and dO: those may be NaN
  const uint32_t los = (lane & 31) * 4;
  const float *lse_g = p.lse + (long long)hkv * G * p.T, *delta_g = p.delta + (long long)hkv * G * p.T;
  __amdgpu_buffer_rsrc_t rsq, rsd, rsl, rsx;
  const long long h_q = p.q_sh * 2, r_q = (long long)kDkv3Rows * p.q_st * 2, r_d = (long long)kDkv3Rows * do_st * 2;
  auto fetch_setup = [&](bool more) {      // without an item the loads go out all the same: to an empty range (zeros), the last item's scalars
    long long bq = more ? f_qb : 0, bd = more ? f_db : 0;
    if (bq > 0xffffffffLL) bq = 0xffffffffLL;
    if (bd > 0xffffffffLL) bd = 0xffffffffLL;
    rsq = make_rsrc(f_qp, (uint32_t)bq);
    rsd = make_rsrc(f_dp, (uint32_t)bd);
    const uint32_t bs = (uint32_t)(g_f * p.T + q_end) * 4;
    rsl = make_rsrc(lse_g, bs);
    rsx = make_rsrc(delta_g, bs);
  };
  auto fetch_advance = [&]() {             // `stride` items on
    if constexpr (SPLIT) {
      int dg = stride_g, db = stride_b;
      if (g_f + dg >= G) dg -= G, ++db;
      g_f += dg, qb_f -= db * kDkv3Rows;
      f_qp += dg * h_q - db * r_q, f_dp += (long long)dg * HD * 2 - db * r_d;
      f_qb += db * r_q, f_db += db * r_d;
      return;
    }
    g_f += 4;
    f_qp += 4 * h_q, f_dp += 4 * HD * 2;
    while (g_f >= G) {
      g_f -= G, qb_f -= kDkv3Rows;
      f_qp -= G * h_q + r_q, f_dp -= (long long)G * HD * 2 + r_d;
      f_qb += r_q, f_db += r_d;
    }
  };
  auto fetch_q = [&](auto ic, uint32_t buf, int step) {                   // NLD + 2 instructions: Q rows, scalars
    constexpr int i = decltype(ic)::value;
    if constexpr (i < NLD) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsq, FGRPO_LDS_AT(buf + i * 1024), 16, (int)foq[i % NPAT], i * step, 0, 0);
    else if constexpr (i == NLD) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsl, FGRPO_LDS_AT(buf + kSc), 4, (int)los, (g_f * p.T + qb_f) * 4, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsx, FGRPO_LDS_AT(buf + kSc + 256), 4, (int)los, (g_f * p.T + qb_f) * 4, 0, 0);
  };
  auto fetch_d = [&](auto ic, uint32_t buf, int step) {                   // NLD instructions: dO rows
    constexpr int i = decltype(ic)::value;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsd, FGRPO_LDS_AT(buf + kT + i * 1024), 16, (int)fod[i % NPAT], i * step, 0, 0);
  };
  auto fence = []() { __builtin_amdgcn_sched_barrier(0); };

  // What a work-group needs before it can start, all of it under way at once: the V tile, the K tile (both shared; K stays in
  // wavefront 0's second buffer until every wavefront has read its operands) and the first items.  Read with each lane on
  // its own row, K was 16 instructions a wavefront of which each touches 32 rows: 5.8 us from the segment bounds to the first
  // item, of 46 a work-group took at segments of 128..1024 tokens; now 3.7.
  constexpr uint32_t kStage = kBuf;
  {
    const int row = wave * RPI + lane / (HD / 8), ch = (lane % (HD / 8)) ^ attn_swz<HD>(row);      // 4 RPI rows a step: the same swizzle
    auto shared_tile = [&](const bf16_t* first, long long st, uint32_t lds) {
      const uint32_t off = (uint32_t)((row * st + ch * 8) * 2);
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(first, (uint32_t)min((klast - k0) * st * 2 + RB, 0xffffffffLL));
#pragma unroll
      for (int i = 0; i < kKeys / RPI / 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, FGRPO_LDS_AT(lds + wave * 1024 + i * 4096), 16, (int)off, (int)(i * 4 * RPI * st * 2), 0, 0);
    };
    shared_tile(p.k + (long long)hkv * p.k_sh + (long long)k0 * p.k_st, p.k_st, lds0 + kStage);
    shared_tile(p.v + (long long)hkv * p.v_sh + (long long)k0 * p.v_st, p.v_st, lds0 + 4 * 2 * kBuf);
  }
  static_assert(kKeys * RB <= kBuf && kKeys % (4 * RPI) == 0, "the K tile fits a buffer, in whole instructions of every wavefront");
  int g_c = g_f, qb = qb_f;                                    // the item being computed
  constexpr int kItemLoads = 2 * NLD + 2;
  auto fetch_item = [&](auto bc) {
    constexpr int b = decltype(bc)::value;
    const bool more = first + stride * b < NI;
    if (b == 1 && more) fetch_advance();
    fetch_setup(more);
    static_for<NLD + 2>([&](auto ic) { fetch_q(ic, base_w + b * kBuf, sq); });
    static_for<NLD>([&](auto ic) { fetch_d(ic, base_w + b * kBuf, sd); });
  };
  if (first < NI) fetch_item(std::integral_constant<int, 0>{});
  static_for<NACC>([&](auto rc) { dkv3_acc_clear<NACC, decltype(rc)::value>(); });      // under the loads
  // the queries that see the lane's key: key_n of them, from the key itself (causal) or its segment's start on; kept
  // relative to the lane's first row of a query block
  int key_lo[KB];
  uint32_t key_n[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int key = k0 + 32 * kb + (lane & 31), kc = min(key, p.T - 1);
    const int lo = p.causal ? kc : p.seg_start[kc];
    key_lo[kb] = lo - 4 * h;
    key_n[kb] = key < p.T ? (uint32_t)max(min(p.seg_end[kc], q_end) - lo, 0) : 0u;
    asm volatile("" : "+v"(key_lo[kb]), "+v"(key_n[kb]));
  }
  FGRPO_WAIT_VMCNT(0);
  wg_barrier();                                                // the whole K and V tiles are there
  u32x4_t kf[KB][KS];                                          // K rows of the key blocks as operands
  {
    const uint32_t ka = lds0 + kStage - base_w;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      kf[0][st] = lds_read_u128_asm<0>(rowc[st] + ka);
      if constexpr (KB == 2) kf[KB - 1][st] = lds_read_u128_asm<32 * RB>(rowc[st] + ka);
    }
  }
  wait_lgkm<0>();
  fence();
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int st = 0; st < KS; ++st) attn_settle(kf[kb][st]);
  wg_barrier();                                                // K has been read: the second item may have the buffer
  if (first < NI) fetch_item(std::integral_constant<int, 1>{});

  u32x4_t qf[KS];                                              // Q rows of the item; the first half is requested by the item before
  auto req_q = [&](auto offc, auto stc) { qf[decltype(stc)::value] = lds_read_u128_asm<decltype(offc)::value>(rowc[decltype(stc)::value]); };
  auto item = [&](auto curc, int n) {
    constexpr int cur = decltype(curc)::value, qt = cur * kBuf, dot = qt + kT, sct = cur * kBuf, nxt = (cur ^ 1) * kBuf;
    const bool masked = qb < q_full || qb + kDkv3Rows > q_end;
    u32x4_t fo[2][2], fv[2][2][KB], nd[4], l4[4];
    AttnTr ta[DB], tb[DB];
    f32x16_t s[KB], dp[KB];
    u32x4_t pp[KB][2], ds[KB][2];                               // P, dS as operands: [key block][rows 8 s2 ..]
    auto req_dp = [&](auto gc) {                               // dP group: k steps 2 g, 2 g + 1: dO rows, V rows of both key blocks
      constexpr int g = decltype(gc)::value;
      static_for<2>([&](auto ic) {
        constexpr int i = decltype(ic)::value, st = 2 * g + i;
        fo[g % 2][i] = lds_read_u128_asm<dot>(rowc[st]);
        const uint32_t va = rowc[st] + v_delta;
        fv[g % 2][i][0] = lds_read_u128_asm<0>(va);
        if constexpr (KB == 2) fv[g % 2][i][KB - 1] = lds_read_u128_asm<32 * RB>(va);
      });
    };
    auto req_tr = [&](auto offc, AttnTr (&t)[DB]) {
      static_for<DB>([&](auto dc) {
        constexpr int db = decltype(dc)::value;
        t[db] = attn_rd_tr_asm<decltype(offc)::value>(tr[db][0], tr[db][1]);
      });
    };
    auto e_el = [&](auto kbc, auto rc) {                       // P in place of S
      constexpr int kb = decltype(kbc)::value, r = decltype(rc)::value;
      s[kb][r] = fast_exp2(__builtin_fmaf(s[kb][r], c, -__uint_as_float(l4[r / 4][r % 4])));
      asm volatile("" : "+v"(s[kb][r]));
    };
    auto f_el = [&](auto ec, auto halfc) {                     // dS in place of dP: element e of a half is key block e % KB, row 8 half + e / KB
      constexpr int e = decltype(ec)::value, half = decltype(halfc)::value, kb = e % KB, r = 8 * half + e / KB;
      dp[kb][r] = s[kb][r] * dp[kb][r];
      asm volatile("" : "+v"(dp[kb][r]));
    };
    auto pack = [&](const f32x16_t& x, int half) {
      const u32x4_t v = {pack_bf16x2(x[8 * half], x[8 * half + 1]), pack_bf16x2(x[8 * half + 2], x[8 * half + 3]),
                         pack_bf16x2(x[8 * half + 4], x[8 * half + 5]), pack_bf16x2(x[8 * half + 6], x[8 * half + 7])};
      return v;
    };
    // P of a hidden pair is zero, whatever its query's lse is (a NaN row of another segment in the same block must not
    // reach this key); a branch of its own around the selects
    auto hide = [&](auto kbc) {
      constexpr int kb = decltype(kbc)::value;
      int qv = qb;
      asm volatile("" : "+s"(qv));                             // formed here: hoisted, it would be computed for every item
      const uint32_t q0 = (uint32_t)(qv - key_lo[kb]);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = q0 + (uint32_t)(8 * (r >> 2) + (r & 3)) < key_n[kb] ? s[kb][r] : 0.f;
    };
    // vector work w = 0 .. N - 1 dealt evenly to instructions m = M0 .. M1 - 1 of a run
    auto deal = [&](auto nc, auto mc, auto m0c, auto m1c, auto&& side) {
      constexpr int N = decltype(nc)::value, m = decltype(mc)::value - decltype(m0c)::value, M = decltype(m1c)::value - decltype(m0c)::value;
      if constexpr (m >= 0 && m < M)
        static_for<N>([&](auto wc) {
          constexpr int w = decltype(wc)::value;
          if constexpr (w >= N * m / M && w < N * (m + 1) / M) side(wc);
        });
    };
#define FGRPO_IC(x) std::integral_constant<int, (x)>{}
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;

    // ---- S of key block 0
    static_for<QG>([&](auto ic) { req_q(FGRPO_IC(qt), FGRPO_IC(QG + decltype(ic)::value)); });
    static_for<4>([&](auto gc) { l4[decltype(gc)::value] = lds_read_u128_asm<sct + 32 * decltype(gc)::value>(scl); });
    wait_lgkm<QG + 4>();
    fence();
    auto s_mma = [&](auto kbc, auto stc) {
      constexpr int kb = decltype(kbc)::value, st = decltype(stc)::value;
      if constexpr (kb == 0) attn_settle(qf[st]);
      if constexpr (st == 0) s[kb] = attn_mfma(qf[st], kf[kb][st], f32x16_t{0.f});
      else s[kb] = attn_mfma(qf[st], kf[kb][st], s[kb]);
      fence();
    };
    static_for<QG>([&](auto ic) { s_mma(H0{}, ic); });
    wait_lgkm<0>();
    fence();
    static_for<QG>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      s_mma(H0{}, FGRPO_IC(QG + i));
      deal(FGRPO_IC(4), ic, FGRPO_IC(0), FGRPO_IC(QG), [&](auto gc) {
        constexpr int gr = decltype(gc)::value;
        attn_settle(l4[gr]);
#pragma unroll
        for (int e = 0; e < 4; ++e) l4[gr][e] = __float_as_uint(__uint_as_float(l4[gr][e]) * kLog2e);
        attn_settle(l4[gr]);
      });
      fence();
    });
    constexpr int GD = 2 + 2 * KB;                             // LDS reads of a dP group
    auto open_dp = [&]() {                                     // -delta and the first group on their way
      static_for<4>([&](auto gc) { nd[decltype(gc)::value] = lds_read_u128_asm<sct + 256 + 32 * decltype(gc)::value>(scl); });
      FGRPO_WAIT_VMCNT(kItemLoads);                            // this item's dO rows: later loads are the next item's
      req_dp(H0{});
      fence();
    };
    // ---- S of key block 1 | P of key block 0
    if constexpr (KB == 2) {
      static_for<KS>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        s_mma(FGRPO_IC(KB - 1), ic);
        deal(FGRPO_IC(16), ic, FGRPO_IC(1), FGRPO_IC(KS), [&](auto rc) { e_el(H0{}, rc); });
        fence();
        if constexpr (i == KS / 2 - 1) open_dp();
      });
      if (masked) hide(H0{});
    } else {
      open_dp();
    }
    // ---- dP, starting from -delta | P of the last key block
    static_for<NG>([&](auto gc) {
      constexpr int g = decltype(gc)::value;
      if constexpr (g + 1 < NG) req_dp(FGRPO_IC(g + 1));
      else req_tr(FGRPO_IC(dot), ta);
      wait_lgkm<(g + 1 < NG ? GD : 2 * DB)>();
      fence();
      static_for<2>([&](auto ic) {
        constexpr int i = decltype(ic)::value, st = 2 * g + i;
        attn_settle(fo[g % 2][i]);
        static_for<KB>([&](auto kbc) {
          constexpr int kb = decltype(kbc)::value, m = KB * (2 * g + i) + kb;
          attn_settle(fv[g % 2][i][kb]);
          if constexpr (st == 0) {
            f32x16_t ndelta;
#pragma unroll
            for (int gr = 0; gr < 4; ++gr) {
              if constexpr (kb == 0) attn_settle(nd[gr]);
#pragma unroll
              for (int e = 0; e < 4; ++e) ndelta[4 * gr + e] = __uint_as_float(nd[gr][e]);
            }
            dp[kb] = attn_mfma(fo[0][0], fv[0][0][kb], ndelta);
          } else {
            dp[kb] = attn_mfma(fo[g % 2][i], fv[g % 2][i][kb], dp[kb]);
          }
          fence();
          deal(FGRPO_IC(16), FGRPO_IC(m), FGRPO_IC(1), FGRPO_IC(KB * KS), [&](auto rc) { e_el(FGRPO_IC(KB - 1), rc); });
          fence();
        });
      });
    });
    if (masked) hide(FGRPO_IC(KB - 1));
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) pp[kb][0] = pack(s[kb], 0);
    // ---- dV and dK in quarters of NQ instructions
    constexpr int NQ = KB * DB, EH = 8 * KB;                   // EH: elements of half the rows
    static_assert(NQ >= 2, "two instructions on one accumulator block never follow each other directly");
    auto quarter = [&](AttnTr (&t)[DB], u32x4_t (&op)[KB][2], auto s2c, auto accc, auto&& side) {
      constexpr int s2 = decltype(s2c)::value, acc = decltype(accc)::value;
      static_for<DB>([&](auto dc) {
        constexpr int db = decltype(dc)::value;
        const u32x4_t b = attn_settle_tr(t[db]);
        static_for<KB>([&](auto kbc) {
          constexpr int kb = decltype(kbc)::value;
          dkv3_mfma<NACC, acc + kb * DB + db, db == 0>(op[kb][s2], b);
          fence();
          side(FGRPO_IC(KB * db + kb));
          fence();
        });
      });
    };
    // dV, rows 0..7 | P of the other rows packed, dS of rows 0..7
    req_tr(FGRPO_IC(qt), tb);
    wait_lgkm<2 * DB>();
    fence();
    quarter(ta, pp, H0{}, FGRPO_IC(kAccV), [&](auto mc) {
      deal(FGRPO_IC(KB), mc, FGRPO_IC(0), FGRPO_IC(KB), [&](auto kbc) { pp[decltype(kbc)::value][1] = pack(s[decltype(kbc)::value], 1); });
      deal(FGRPO_IC(EH), mc, FGRPO_IC(1), FGRPO_IC(NQ), [&](auto ec) { f_el(ec, H0{}); });
    });
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) ds[kb][0] = pack(dp[kb], 0);
    // dK, rows 0..7 | dS of the other rows
    req_tr(FGRPO_IC(qt + 16 * RB), ta);
    wait_lgkm<2 * DB>();
    fence();
    quarter(tb, ds, H0{}, FGRPO_IC(kAccK), [&](auto mc) {
      deal(FGRPO_IC(EH), mc, FGRPO_IC(0), FGRPO_IC(NQ), [&](auto ec) { f_el(ec, H1{}); });
    });
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) ds[kb][1] = pack(dp[kb], 1);
    // dK, rows 8..15 | the Q rows and scalars of the item after next
    const bool more2 = n + 2 * stride < NI;
    // destinations and row offsets are formed here: held across the loop they would fill the scalar registers
    uint32_t bufs = base_w;
    int sqv = sq, sdv = sd;
    asm volatile("" : "+s"(bufs), "+s"(sqv), "+s"(sdv));
    if (more2) fetch_advance();
    fetch_setup(more2);
    req_tr(FGRPO_IC(dot + 16 * RB), tb);
    wait_lgkm<2 * DB>();                                       // everything of this item's Q rows and scalars has been read
    fence();
    quarter(ta, ds, H1{}, FGRPO_IC(kAccK), [&](auto mc) {
      deal(FGRPO_IC(NLD + 2), mc, FGRPO_IC(0), FGRPO_IC(NQ), [&](auto ic) { fetch_q(ic, bufs + qt, sqv); });
    });
    // dV, rows 8..15 | its dO rows; the first Q rows of the next item on their way
    FGRPO_WAIT_VMCNT(kItemLoads);                              // the next item's Q rows: later loads are its dO rows and the Q rows just requested
    static_for<QG>([&](auto ic) { req_q(FGRPO_IC(nxt), ic); });
    wait_lgkm<QG>();                                           // everything of this item's dO rows has been read
    fence();
    if constexpr (SPLIT) {
      g_c += stride_g, qb -= stride_b * kDkv3Rows;
      if (g_c >= G) g_c -= G, qb -= kDkv3Rows;
    } else {
      g_c += 4;
      while (g_c >= G) g_c -= G, qb -= kDkv3Rows;
    }
    quarter(tb, pp, H1{}, FGRPO_IC(kAccV), [&](auto mc) {
      deal(FGRPO_IC(NLD), mc, FGRPO_IC(0), FGRPO_IC(NQ), [&](auto ic) { fetch_d(ic, bufs + qt, sdv); });
    });
  };
  if (first < NI) {
    static_for<QG>([&](auto ic) { req_q(FGRPO_IC(0), ic); });
    for (int n = first; n < NI; n += 2 * stride) {
      item(FGRPO_IC(0), n);
      if (n + stride < NI) item(FGRPO_IC(1), n + stride);
    }
    wait_lgkm<0>();
#pragma unroll
    for (int i = 0; i < QG; ++i) attn_settle(qf[i]);
    FGRPO_WAIT_VMCNT(0);                                       // the loads that brought nothing: the buffers are about to be reused
  }
#undef FGRPO_IC
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");           // the last matrix instructions have written their accumulators

  // ---- the four sets of accumulators, added in wavefront order; 16-byte stores of eight columns
  // (lane and thread index formed anew: held across the loop they would cost registers it does not have)
  constexpr int SS = kDkv3SumStride<HD>;
  const int lane_e = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), tid_e = wave * 64 + lane_e;
  auto sum_store = [&](auto accc, float mul, bf16_t* out, int which) {
    constexpr int acc = decltype(accc)::value;
    wg_barrier();                                              // the tiles / the previous sums are no longer read
    const uint32_t w0 = lds0 + wave * (kKeys * SS) + (4 * (lane_e >> 5)) * SS + (lane_e & 31) * 4;
    static_for<KB>([&](auto kbc) {
      static_for<DB>([&](auto nbc) {
        static_for<16>([&](auto rc) {
          constexpr int kb = decltype(kbc)::value, nb = decltype(nbc)::value, r = decltype(rc)::value;
          dkv3_acc_to_lds<16 * (acc + kb * DB + nb) + r, (32 * kb + 8 * (r / 4) + r % 4) * SS + nb * 128>(w0);
        });
      });
    });
    wait_lgkm<0>();
    wg_barrier();
#pragma unroll
    for (int i = 0; i < kKeys * HD / 8 / 256; ++i) {
      const int piece = tid_e + 256 * i, row = piece / (HD / 8), col = piece % (HD / 8);
      const uint32_t a = lds0 + row * SS + col * 32;
      u32x4_t part[4][2];
      static_for<4>([&](auto wc) {
        constexpr int w = decltype(wc)::value;
        const uint32_t aw = a + w * (kKeys * SS);
        part[w][0] = lds_read_u128_asm<0>(aw);
        part[w][1] = lds_read_u128_asm<16>(aw);
      });
      wait_lgkm<0>();
      fence();
      float x[8];
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j % 4 == 0) attn_settle(part[w][j / 4]);
          x[j] = (w == 0 ? 0.f : x[j]) + __uint_as_float(part[w][j / 4][j % 4]);
        }
      const int kk = k0 + row;
      const bool partial = SPLIT && np > 1;
      if (SPLIT && partial && kk < p.T) {
        float4* dst = (float4*)(p.part_k + (((long long)blockIdx.x * 2 + which) * kKeys + row) * HD + col * 8);
        dst[0] = make_float4(x[0], x[1], x[2], x[3]);
        dst[1] = make_float4(x[4], x[5], x[6], x[7]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= mul;
      if (kk < p.T && !partial) __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, attn_pack8(x)), (u32x4_t*)(out + ((long long)kk * p.Hkv + hkv) * HD + col * 8));
    }
    wait_lgkm<0>();
  };
  sum_store(std::integral_constant<int, kAccK>{}, p.scale, p.dk, 0);
  sum_store(std::integral_constant<int, kAccV>{}, 1.f, p.dv, 1);
}

__device__ __forceinline__ void attn_load8(const float* src, float (&v)[8]) {
  const float4 a = *(const float4*)src, b = *(const float4*)(src + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
// Sums of the parts, in part order, of dQ (the first nq work-groups, see attn_merge_query_tile) and of dK and dV (key tiles of
// kKeys): eight columns of one row a thread.  Rows of tiles that were not dealt out are already in place.
template <int HD, int kKeys>
static __global__ __launch_bounds__(256) void attn_merge_bwd_kernel(AttnParams p, int RB, int nq, long long nk) {
  if ((int)blockIdx.x < nq) {
    attn_merge_query_tile<HD, false>(p, RB, blockIdx.x);
    return;
  }
  long long idx = (long long)((int)blockIdx.x - nq) * 256 + threadIdx.x;
  if (idx >= 2 * nk) return;
  const int which = idx >= nk;
  if (which) idx -= nk;
  const int col = (int)(idx % (HD / 8)) * 8;
  const long long row = idx / (HD / 8);                        // key * Hkv + head
  const int kk = (int)(row / p.Hkv), head = (int)(row % p.Hkv);
  const int2 info = p.key_info[kk / kKeys * p.Hkv + head];
  const int np = info.x, first = info.y;                       // parts, the work-group of the first (the others' 8 apart)
  if (!attn_parts_inside(np, first, 0, 8, p.blocks_k + 8 * p.extra_k)) return;
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = 0.f;
  constexpr int slice = 2 * kKeys * HD;
  const float* src = p.part_k + (long long)first * slice + (which * kKeys + kk % kKeys) * HD + col;
#pragma unroll
  for (int j0 = 0; j0 < kAttnMaxParts; j0 += kAttnMergeWide) {
    if (j0 >= np) break;
    float v[kAttnMergeWide][8];
#pragma unroll
    for (int u = 0; u < kAttnMergeWide; ++u) attn_load8(src + (j0 + u < np ? j0 + u : 0) * (8LL * slice), v[u]);
#pragma unroll
    for (int u = 0; u < kAttnMergeWide; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = j0 + u < np ? x[e] + v[u][e] : x[e];
  }
  const float mul = which ? 1.f : p.scale;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] *= mul;
  *(bf16x8_t*)((which ? p.dv : p.dk) + row * HD + col) = attn_pack8(x);
}

}  // namespace fgrpo
