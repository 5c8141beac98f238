// dK / dV of the packed attention with one wavefront per SIMD and no barrier in its loop (head dimension HD = 128 or
// 64).  A work-group owns 64 keys of one K/V head; its four wavefronts deal the work on those keys among themselves -
// item n = (32 queries, query head) goes to wavefront n % 4 - and each walks its items alone: it brings the item's
// Q / dO rows into two LDS buffers of its own (global -> LDS, an item ahead), waits for nothing but its own loads,
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
// 7.20 -> 6.17 ms; 32768 tokens in segments of 128..1024, 12 / 2 heads of 128: 442 -> 409 us; 12345 such tokens, 14 / 2
// heads of 64: 245 -> 143 us; 6535 tokens, 12 / 2 heads of 128: 160 -> 101 us.  It was faster at every size tried, so
// no rule picks between the two.  Counters at the long shape: matrix pipe 0.58 busy, a fifth of the time waiting
// for tiles (with every load aimed at one tile: 5.38 ms).
//
// Orientation and register permutation as in attn_kernels.h (S = Q K^T: a lane owns a key).  One item, with the
// vector work of one stage behind the matrix instructions of the next (a 32x32x16 instruction hides about 20 cycles
// of it):
//   S(both key blocks)            | loads of the next item issued between the instructions
//   dP                            | P = exp2(S c - lse) of rows 0..7 of each lane's 16, packed to bf16
//   dV += P^T dO   (rows 0..7)    | P of rows 8..15
//   dV             (rows 8..15)   | dS = P (dP - delta) of rows 0..7
//   dK += dS^T Q   (rows 0..7)    | dS of rows 8..15
//   dK             (rows 8..15)   | first Q fragments of the next item on their way
// -delta enters as the addend of dP's first instruction.  K lives in registers (64 keys x HD), V in LDS, shared by
// the four wavefronts (both in registers would exceed the file beside the accumulators).
#pragma once
#include "attn_kernels.h"

namespace fgrpo {

constexpr int kDkv3Keys = 64, kDkv3Rows = 32;
template <int HD>
constexpr int kDkv3Buf = 2 * kDkv3Rows * HD * 2 + 512;                 // Q | dO | lse, delta | seg_start, seg_end of 32 queries
template <int HD>
constexpr int kDkv3SumStride = HD * 4 + 32;                            // fp32 row of the closing sum: the two lane halves (rows 4 apart) hit different banks
template <int HD>
constexpr int kDkv3LoopLds = 4 * 2 * kDkv3Buf<HD> + kDkv3Keys * HD * 2;
template <int HD>
constexpr int kDkv3Lds = kDkv3LoopLds<HD> > 4 * kDkv3Keys * kDkv3SumStride<HD> ? kDkv3LoopLds<HD> : 4 * kDkv3Keys * kDkv3SumStride<HD>;

// The accumulators live in fixed accumulation registers, a[16 n : 16 n + 15] for block n, named in the instructions:
// at HD = 128 they are all 256 of them, and a register allocator that may move or copy a block has nowhere to put it
// (left to it, the loop spilled 260 registers).  Every instruction lists the whole range as clobbered, so that the
// compiler keeps nothing of its own there; the build checks that the kernel spills nothing.
// The compiler's hazard table does not see these instructions: the first one behind vector arithmetic that formed an
// operand carries two wait states, instructions on one block are at least four matrix instructions apart.
#define FGRPO_DKV3_CLOBBER_128 \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
  "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
  "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
  "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
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
template <int HD, int BLK, bool FIRST>
__device__ __forceinline__ void dkv3_mfma(u32x4_t a, u32x4_t b) {
  constexpr int r0 = 16 * BLK, r1 = r0 + 15;
  if constexpr (HD == 128) {
    if constexpr (FIRST) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : FGRPO_DKV3_CLOBBER_256);
    else asm volatile("v_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : FGRPO_DKV3_CLOBBER_256);
  } else {
    if constexpr (FIRST) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : FGRPO_DKV3_CLOBBER_128);
    else asm volatile("v_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(r0), "n"(r1) : FGRPO_DKV3_CLOBBER_128);
  }
}
template <int HD, int REG>
__device__ __forceinline__ void dkv3_acc_clear() {
  if constexpr (HD == 128) asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(REG) : FGRPO_DKV3_CLOBBER_256);
  else asm volatile("v_accvgpr_write_b32 a[%0], 0" : : "n"(REG) : FGRPO_DKV3_CLOBBER_128);
}
template <int REG>
__device__ __forceinline__ float dkv3_acc_read() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(REG));
  return x;
}

template <int HD>
__global__ __launch_bounds__(256, 1) void varlen_attn_dkv3_kernel(AttnParams p) {
  constexpr int KS = HD / 16, DB = HD / 32, RB = HD * 2, kT = kDkv3Rows * RB, kBuf = kDkv3Buf<HD>;
  constexpr int QG = KS / 2, NG = KS / 2;              // row fragments of a half of S; groups of two k steps of dP
  constexpr int kSc = 2 * kT;                          // per-query scalars inside a buffer
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = lds_addr(smem);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = p.Hq / p.Hkv;
  const int hkv = blockIdx.x % p.Hkv, rank = blockIdx.x / p.Hkv;
  const int ntile = (p.T + kDkv3Keys - 1) / kDkv3Keys, n128 = (p.T + 127) / 128;
  const int tile = min(max(p.order_k[rank >> 1], 0), n128 - 1) * 2 + (rank & 1);      // clamped: the list may come from the caller
  if (tile >= ntile) return;
  const int k0 = tile * kDkv3Keys, klast = min(k0 + kDkv3Keys, p.T) - 1;
  const int q_begin = max(__builtin_amdgcn_readfirstlane(p.causal ? k0 : p.seg_start[k0]), 0);      // inside [0, T]
  const int q_end = min(__builtin_amdgcn_readfirstlane(p.seg_end[klast]), p.T);
  // one segment holds every key of the tile: queries from `q_full` on that are complete blocks see all of it
  const bool one_segment = __builtin_amdgcn_readfirstlane(p.seg_start[k0]) == __builtin_amdgcn_readfirstlane(p.seg_start[klast]);
  const int q_full = !one_segment ? 0x7fffffff : p.causal ? k0 + kDkv3Keys - 1 : q_begin;
  const int nqb = q_end > q_begin ? (q_end - q_begin + kDkv3Rows - 1) / kDkv3Rows : 0;
  const int NI = nqb * G;

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

  // V tile -> LDS by the whole work-group; rows past the end of the keys read as zero
  {
    const uint32_t fvo = attn_dma_lane_offset<HD>(wave, lane, p.v_st);
    attn_dma_tile<HD>(p.v + (long long)hkv * p.v_sh, p.v_st, k0, klast + 1, fvo, smem + 4 * 2 * kBuf + wave * 1024);
  }
  // K rows of the two key blocks as operands
  u32x4_t kf[2][KS];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    bf16x8_t f[KS];
    const int key = k0 + 32 * kb + (lane & 31);
    attn_row_operand(f, p.k + (long long)min(key, p.T - 1) * p.k_st + (long long)hkv * p.k_sh, key < p.T, h);
#pragma unroll
    for (int st = 0; st < KS; ++st) kf[kb][st] = __builtin_bit_cast(u32x4_t, f[st]);
  }
  const float c = p.scale * kLog2e;

  // accumulator blocks: dV[kb][nb] = kb DB + nb, dK behind them
  constexpr int kAccV = 0, kAccK = 2 * DB;
  static_for<4 * DB * 16>([&](auto rc) { dkv3_acc_clear<HD, decltype(rc)::value>(); });

  // ---- loads of an item.  Instruction i of a tile fills its KiB i: RPI rows; lane l lands at 16 l of it, i.e. row
  // i RPI + l / (HD/8), chunk slot l % (HD/8), and fetches the chunk the swizzle puts there (four or two patterns)
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
  // lanes 0..31 bring lse and seg_start of the 32 queries, lanes 32..63 delta and seg_end
  const float* sc0 = h ? p.delta : p.lse;
  const int* sc1 = h ? p.seg_end : p.seg_start;
  const uint32_t T = (uint32_t)p.T;
  // the walk goes from the last queries to the first, heads inside: work-groups on the same segment start at the same
  // rows and pass over them together, so that one L2 serves them all
  int g_n = wave % G, qb_n = q_begin + (nqb - 1 - wave / G) * kDkv3Rows;      // the item the next loads bring
  __amdgpu_buffer_rsrc_t rsq, rsd;
  const float* l_p0 = nullptr;
  const int* l_p1 = nullptr;
  auto fetch_setup = [&](bool more) {      // without a next item the loads go out all the same, to an empty range (zeros) and the last scalars
    const int hq = hkv * G + g_n;
    const long long rows = (long long)q_end - qb_n;            // >= 1
    long long bq = more ? (rows - 1) * p.q_st * 2 + RB : 0, bd = more ? (rows - 1) * do_st * 2 + RB : 0;
    if (bq > 0xffffffffLL) bq = 0xffffffffLL;
    if (bd > 0xffffffffLL) bd = 0xffffffffLL;
    rsq = make_rsrc(p.q + (long long)hq * p.q_sh + (long long)qb_n * p.q_st, (uint32_t)bq);
    rsd = make_rsrc(p.dout + (long long)hq * HD + (long long)qb_n * do_st, (uint32_t)bd);
    const uint32_t row = (uint32_t)min(qb_n + (lane & 31), q_end - 1);
    l_p0 = sc0 + ((unsigned long long)hq * T + row);
    l_p1 = sc1 + row;
  };
  auto fetch_piece = [&](auto ic, char* buf) {                 // 2 NLD + 2 instructions
    constexpr int i = decltype(ic)::value;
    if constexpr (i < NLD) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsq, FGRPO_LDS_PTR(buf + i * 1024), 16, (int)foq[i % NPAT], i * sq, 0, 0);
    else if constexpr (i < 2 * NLD)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsd, FGRPO_LDS_PTR(buf + i * 1024), 16, (int)fod[i % NPAT], (i - NLD) * sd, 0, 0);
    else if constexpr (i == 2 * NLD) __builtin_amdgcn_global_load_lds(FGRPO_GLOBAL_PTR(l_p0), FGRPO_LDS_PTR(buf + kSc), 4, 0, 0);
    else __builtin_amdgcn_global_load_lds(FGRPO_GLOBAL_PTR(l_p1), FGRPO_LDS_PTR(buf + kSc + 256), 4, 0, 0);
  };
  auto advance = [&]() {
    g_n += 4;
    while (g_n >= G) g_n -= G, qb_n -= kDkv3Rows;
  };
  char* buf_w = smem + wave * 2 * kBuf;
  auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int st = 0; st < KS; ++st) asm volatile("" : "+v"(kf[kb][st]));      // complete before the loop

  int qb = qb_n;                                               // the item being computed
  if (wave < NI) {
    fetch_setup(true);
    static_for<2 * NLD + 2>([&](auto ic) { fetch_piece(ic, buf_w); });
    if (wave + 4 < NI) advance();
  }
  FGRPO_WAIT_VMCNT(0);
  wg_barrier();                                                // the V tile is there too

  u32x4_t qa[QG];                                              // first half of the Q fragments, carried across items
  auto req_rows = [&](auto offc, auto stc, u32x4_t& f) { f = lds_read_u128_asm<decltype(offc)::value>(rowc[decltype(stc)::value]); };
  auto item = [&](auto curc, int n) {
    constexpr int cur = decltype(curc)::value, qt = cur * kBuf, dot = qt + kT, sct = cur * kBuf, nxt = (cur ^ 1) * kBuf;
    const bool more = n + 4 < NI;
    const bool masked = qb < q_full || qb + kDkv3Rows > q_end;
    char* nbuf = buf_w + nxt;
    u32x4_t qh[QG], fo[2][2], fv[2][2][2], nd[4], l4[2][2];
    AttnTr ta[DB], tb[DB];
    f32x16_t s[2], dp[2];
    u32x4_t pp[2][2], ds[2][2];                                // P, dS as operands: [key block][rows 8 s2 ..]
    auto req_dp = [&](auto gc) {                               // dP group: k steps 2 g, 2 g + 1: dO rows, V rows of both key blocks
      constexpr int g = decltype(gc)::value;
      static_for<2>([&](auto ic) {
        constexpr int i = decltype(ic)::value, st = 2 * g + i;
        fo[g % 2][i] = lds_read_u128_asm<dot>(rowc[st]);
        const uint32_t va = rowc[st] + v_delta;
        fv[g % 2][i][0] = lds_read_u128_asm<0>(va);
        fv[g % 2][i][1] = lds_read_u128_asm<32 * RB>(va);
      });
    };
    auto req_tr = [&](auto offc, AttnTr (&t)[DB]) {
      static_for<DB>([&](auto dc) {
        constexpr int db = decltype(dc)::value;
        t[db] = attn_rd_tr_asm<decltype(offc)::value>(tr[db][0], tr[db][1]);
      });
    };
    auto e_el = [&](auto ec) {                                 // element e of a half: key block e % 2, row 8 half + e / 2
      return [&](auto halfc) {
        constexpr int e = decltype(ec)::value, half = decltype(halfc)::value, kb = e % 2, r = 8 * half + e / 2;
        s[kb][r] = fast_exp2(__builtin_fmaf(s[kb][r], c, -__uint_as_float(l4[half][(e / 2) / 4][(e / 2) % 4])));
        asm volatile("" : "+v"(s[kb][r]));
      };
    };
    auto f_el = [&](auto ec, auto halfc) {
      constexpr int e = decltype(ec)::value, half = decltype(halfc)::value, kb = e % 2, r = 8 * half + e / 2;
      dp[kb][r] = s[kb][r] * dp[kb][r];
      asm volatile("" : "+v"(dp[kb][r]));
    };
    auto pack = [&](const f32x16_t& x, int half) {
      const u32x4_t v = {pack_bf16x2(x[8 * half], x[8 * half + 1]), pack_bf16x2(x[8 * half + 2], x[8 * half + 3]),
                         pack_bf16x2(x[8 * half + 4], x[8 * half + 5]), pack_bf16x2(x[8 * half + 6], x[8 * half + 7])};
      return v;
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    using AV = std::integral_constant<int, kAccV>;
    using AK = std::integral_constant<int, kAccK>;

    // ---- S, first half of the k steps; the next item's loads go out between the instructions
    fetch_setup(more);
    static_for<QG>([&](auto ic) { req_rows(std::integral_constant<int, qt>{}, std::integral_constant<int, QG + decltype(ic)::value>{}, qh[decltype(ic)::value]); });
    wait_lgkm<QG>();
    fence();
    constexpr int NF = 2 * NLD + 2, PF = (NF + 2 * KS - 1) / (2 * KS);      // loads behind each S instruction
    auto s_mma = [&](u32x4_t& f, auto stc) {
      constexpr int st = decltype(stc)::value;
      attn_settle(f);
      static_for<2>([&](auto kbc) {
        constexpr int kb = decltype(kbc)::value;
        if constexpr (st == 0) s[kb] = attn_mfma(f, kf[kb][st], f32x16_t{0.f});
        else s[kb] = attn_mfma(f, kf[kb][st], s[kb]);
        fence();
        static_for<PF>([&](auto jc) {
          constexpr int i = (2 * st + kb) * PF + decltype(jc)::value;
          if constexpr (i < NF) fetch_piece(std::integral_constant<int, i>{}, nbuf);
        });
        fence();
      });
    };
    static_for<QG>([&](auto ic) { s_mma(qa[decltype(ic)::value], ic); });
    // ---- second half; -delta and the first dP group are on their way
    static_for<4>([&](auto gc) { nd[decltype(gc)::value] = lds_read_u128_asm<sct + 128 + 32 * decltype(gc)::value>(scl); });
    req_dp(H0{});
    wait_lgkm<4 + 6>();
    fence();
    static_for<QG>([&](auto ic) { s_mma(qh[decltype(ic)::value], std::integral_constant<int, QG + decltype(ic)::value>{}); });
    if (masked) {      // hidden pairs become -inf; a branch of its own around the selects
      const int key0 = k0 + (lane & 31);
      static_for<4>([&](auto gc) {
        constexpr int gr = decltype(gc)::value;
        u32x4_t lo4 = lds_read_u128_asm<sct + 256 + 32 * gr>(scl), en4 = lds_read_u128_asm<sct + 384 + 32 * gr>(scl);
        wait_lgkm<0>();
        fence();
        attn_settle(lo4);
        attn_settle(en4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int q = qb + 8 * gr + 4 * h + e;
          const int hi = q < q_end ? (p.causal ? q : (int)en4[e] - 1) : -1;
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            const int key = key0 + 32 * kb;
            s[kb][4 * gr + e] = ((int)(key >= (int)lo4[e]) & (int)(key <= hi)) ? s[kb][4 * gr + e] : -INFINITY;
          }
        }
      });
      fence();
    }
    // ---- dP: groups of two k steps, P of rows 0..7 behind all but the first
    f32x16_t ndelta;
    static_for<NG>([&](auto gc) {
      constexpr int g = decltype(gc)::value;
      if constexpr (g + 1 < NG) req_dp(std::integral_constant<int, g + 1>{});
      if constexpr (g == 0) static_for<2>([&](auto ic) { l4[0][decltype(ic)::value] = lds_read_u128_asm<sct + 32 * decltype(ic)::value>(scl); });
      if constexpr (g + 1 == NG) {
        static_for<2>([&](auto ic) { l4[1][decltype(ic)::value] = lds_read_u128_asm<sct + 64 + 32 * decltype(ic)::value>(scl); });
        req_tr(std::integral_constant<int, dot>{}, ta);
      }
      wait_lgkm<(g + 1 < NG ? 6 : 0) + (g == 0 ? 2 : 0) + (g + 1 == NG ? 2 + 2 * DB : 0)>();
      fence();
      if constexpr (g == 0) {
#pragma unroll
        for (int gr = 0; gr < 4; ++gr) {
          attn_settle(nd[gr]);
#pragma unroll
          for (int e = 0; e < 4; ++e) ndelta[4 * gr + e] = -__uint_as_float(nd[gr][e]);
        }
      }
      if constexpr (g == 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          attn_settle(l4[0][i]);
#pragma unroll
          for (int e = 0; e < 4; ++e) l4[0][i][e] = __float_as_uint(__uint_as_float(l4[0][i][e]) * kLog2e);
        }
      }
      static_for<2>([&](auto ic) {
        constexpr int i = decltype(ic)::value, st = 2 * g + i;
        attn_settle(fo[g % 2][i]);
        static_for<2>([&](auto kbc) {
          constexpr int kb = decltype(kbc)::value, m = 4 * (g - 1) + 2 * i + kb, M = 4 * (NG - 1);
          attn_settle(fv[g % 2][i][kb]);
          dp[kb] = attn_mfma(fo[g % 2][i], fv[g % 2][i][kb], st == 0 ? ndelta : dp[kb]);
          fence();
          if constexpr (g >= 1)
            static_for<16>([&](auto ec) {
              constexpr int e = decltype(ec)::value;
              if constexpr (e >= 16 * m / M && e < 16 * (m + 1) / M) e_el(ec)(H0{});
            });
          fence();
        });
      });
    });
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) pp[kb][0] = pack(s[kb], 0);
    // ---- dV and dK in quarters of 2 DB instructions
    constexpr int NQ = 2 * DB, EPI = 16 / NQ;                  // vector elements behind each instruction
    auto quarter = [&](AttnTr (&t)[DB], u32x4_t (&op)[2][2], auto s2c, auto accc, auto&& side) {
      constexpr int s2 = decltype(s2c)::value, acc = decltype(accc)::value;
      static_for<DB>([&](auto dc) {
        constexpr int db = decltype(dc)::value;
        const u32x4_t b = attn_settle_tr(t[db]);
        static_for<2>([&](auto kbc) {
          constexpr int kb = decltype(kbc)::value;
          dkv3_mfma<HD, acc + kb * DB + db, db == 0>(op[kb][s2], b);
          fence();
          static_for<EPI>([&](auto jc) { side(std::integral_constant<int, (2 * db + kb) * EPI + decltype(jc)::value>{}); });
          fence();
        });
      });
    };
    req_tr(std::integral_constant<int, dot + 16 * RB>{}, tb);
    wait_lgkm<2 * DB>();
    fence();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      attn_settle(l4[1][i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) l4[1][i][e] = __float_as_uint(__uint_as_float(l4[1][i][e]) * kLog2e);
    }
    quarter(ta, pp, H0{}, AV{}, [&](auto ec) { e_el(ec)(H1{}); });
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) pp[kb][1] = pack(s[kb], 1);
    req_tr(std::integral_constant<int, qt>{}, ta);
    wait_lgkm<2 * DB>();
    fence();
    quarter(tb, pp, H1{}, AV{}, [&](auto ec) { f_el(ec, H0{}); });
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) ds[kb][0] = pack(dp[kb], 0);
    req_tr(std::integral_constant<int, qt + 16 * RB>{}, tb);
    wait_lgkm<2 * DB>();
    fence();
    quarter(ta, ds, H0{}, AK{}, [&](auto ec) { f_el(ec, H1{}); });
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) ds[kb][1] = pack(dp[kb], 1);
    FGRPO_WAIT_VMCNT(0);                                       // the next item is in its buffer
    static_for<QG>([&](auto ic) { req_rows(std::integral_constant<int, nxt>{}, ic, qa[decltype(ic)::value]); });
    wait_lgkm<QG>();
    fence();
    qb = qb_n;
    if (n + 8 < NI) advance();                                 // else the walk stays on the last item there is
    quarter(tb, ds, H1{}, AK{}, [](auto) {});
  };
  if (wave < NI) {
    static_for<QG>([&](auto ic) { req_rows(std::integral_constant<int, 0>{}, ic, qa[decltype(ic)::value]); });
    for (int n = wave; n < NI; n += 8) {
      item(std::integral_constant<int, 0>{}, n);
      if (n + 4 < NI) item(std::integral_constant<int, 1>{}, n + 4);
    }
    wait_lgkm<0>();
#pragma unroll
    for (int i = 0; i < QG; ++i) attn_settle(qa[i]);
  }
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");           // the last matrix instructions have written their accumulators

  // ---- the four sets of accumulators, added in wavefront order; 16-byte stores of eight columns
  constexpr int SS = kDkv3SumStride<HD>;
  auto sum_store = [&](auto accc, float mul, bf16_t* out) {
    constexpr int acc = decltype(accc)::value;
    wg_barrier();                                              // the tiles / the previous sums are no longer read
    const uint32_t w0 = lds0 + wave * (kDkv3Keys * SS) + (4 * h) * SS + (lane & 31) * 4;
    static_for<2>([&](auto kbc) {
      static_for<DB>([&](auto nbc) {
        static_for<16>([&](auto rc) {
          constexpr int kb = decltype(kbc)::value, nb = decltype(nbc)::value, r = decltype(rc)::value;
          lds_write_u32_asm<(32 * kb + 8 * (r / 4) + r % 4) * SS + nb * 128>(w0, __float_as_uint(dkv3_acc_read<16 * (acc + kb * DB + nb) + r>()));
        });
      });
    });
    wait_lgkm<0>();
    wg_barrier();
#pragma unroll
    for (int i = 0; i < kDkv3Keys * HD / 8 / 256; ++i) {
      const int piece = threadIdx.x + 256 * i, row = piece / (HD / 8), col = piece % (HD / 8);
      const uint32_t a = lds0 + row * SS + col * 32;
      float x[8];
      static_for<4>([&](auto wc) {
        constexpr int w = decltype(wc)::value;
        const uint32_t aw = a + w * (kDkv3Keys * SS);
        u32x4_t lo = lds_read_u128_asm<0>(aw), hi = lds_read_u128_asm<16>(aw);
        wait_lgkm<0>();
        fence();
        attn_settle(lo);
        attn_settle(hi);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[j] = (w == 0 ? 0.f : x[j]) + __uint_as_float(lo[j]);
          x[4 + j] = (w == 0 ? 0.f : x[4 + j]) + __uint_as_float(hi[j]);
        }
      });
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= mul;
      const int kk = k0 + row;
      if (kk < p.T) *(bf16x8_t*)(out + ((long long)kk * p.Hkv + hkv) * HD + col * 8) = attn_pack8(x);
    }
    wait_lgkm<0>();
  };
  sum_store(std::integral_constant<int, kAccK>{}, p.scale, p.dk);
  sum_store(std::integral_constant<int, kAccV>{}, 1.f, p.dv);
}

}  // namespace fgrpo
