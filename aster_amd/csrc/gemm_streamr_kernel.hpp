// Stream kernel with unequal tile sides, 16-bit and fp8 operands: C[M,N] = epi(A[M,K] * B[N,K]^T)
// on 256 x 128 and 192 x 128 tiles (fp8 also 128 x 128), one eight-wave workgroup per CU.  What it
// measured against the square tiles stands at the rules of selection (unequal_tile_of,
// unequal_split_pays).
//
// What bounds it: 16-bit operands the matrix cores, at the clock the power limit leaves (busy 73 % of a
// busy CU's cycles on 333 x 14336 x 4096, 84 % on 800 x 8192 x 8192, at 1.65 of 2.4 GHz; 34-36 bytes of
// operands per CU and clock from L2, above what the square kernels draw), and the CUs without a tile or on
// padding rows (224 of 256 busy, 333 of 384 rows); fp8 the operand bytes from L2 (25-29 per CU and clock,
// matrix cores busy 52-60 %).  A 256 x 128 tile brings in 384 rows for 32768 outputs, two 128 x 128 tiles
// 512 rows for the same; where a problem has too few 256 x 256 tiles to fill the chip these are the shapes
// between.
//
// LDS is a ring of NS stages, each one whole K-step (128 bytes of every row of A's and B's tile):
// three of 48 KiB, four of 40 KiB or five of 32 KiB.  Unlike the ring of gemm_stream_body, whose halves trade
// places and must be equal, a stage is refilled as a whole: when K-step k is in registers its stage
// is requested for K-step k + NS, so NS - 1 K-steps are on their way at any time.  Swizzle, staging
// plan, fragment order and epilogue are those of gemm_stream_body.  As AUTO runs it the K loops of different XCDs
// start at different steps (first_step_of_xcd), by name at step 0 with the bits of gemm_stream_body: bf16
// 333x14336x4096 50.5 -> 47.9 us, 1400x4096x14336 161 -> 144, 333x4096x14336 (split K) 63.1 -> 58.3, 136x28672x4096
// 59.7 -> 52.3, fp8 200x28672x4096 44.5 -> 40.9; on buffers that no kernel has read yet as much.
#pragma once
#include "gemm_stream_kernel.hpp"

namespace astergemm {
namespace {

template <int DT, int OUT, int BM, int BN, int WM, int WN, int NS, bool K8>
__device__ __forceinline__ void gemm_streamr_body(const GemmArgs& p, int bid) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM / 16;
  constexpr int TN = BN / WN / 16;
  using PlanA = StreamLoadPlan<BM, NW>;  // the staging as cooperative load plans (stream_load_plan.inc)
  using PlanB = StreamLoadPlan<BN, NW>;
  constexpr int LA = PlanA::LH, LB = PlanB::LH, L = LA + LB;  // 1 KiB transfers per wave and K-step
  constexpr int B_AT = BM * kRowBytes;                        // B's rows behind A's in a stage
  constexpr int STAGE = (BM + BN) * kRowBytes;
  constexpr int NF = TM + TN;                                 // fragments per substep
  constexpr int NMF = TM * TN;                                // MFMAs per substep
  static_assert(PlanA::TILE_ROWS == 8 && PlanA::TILE_LDS_BYTES == 8 * kRowBytes, "transfer tile");
  static_assert(DT == ASTERGEMM_BF16 || DT == ASTERGEMM_F16, "16-bit operands");
  static_assert(NS * STAGE <= 160 * 1024, "LDS of a CU");
  static_assert(LA * 8 * NW == BM && LB * 8 * NW == BN, "whole transfers");
  static_assert((8 * NW) % 16 == 0, "swizzle phase must not depend on the transfer index");
  static_assert(LB + NF <= NMF && NF + LA <= NMF, "one side instruction per MFMA");
  static_assert((NS - 1) * L <= 63, "vmcnt field");

  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int tile_m, tile_n;
  map_tile(bid, p.tiles_m, p.tiles_n, p.group_m, tile_m, tile_n);
  const int row0 = tile_m * BM, col0 = tile_n * BN;

  // ---- global -> LDS: 128-byte rows, granule index XOR ((row >> 1) & 7) ----------------------
  const int lrow = lane >> 3;
  const int g_lane = (lane & 7) ^ (((wave * 8 + lrow) >> 1) & 7);
  const unsigned a_off = (unsigned)(lrow * (int)p.lda_bytes + g_lane * 16);
  const unsigned b_off = K8 ? lane * 16 : (unsigned)(lrow * (int)p.ldb_bytes + g_lane * 16);
  const uint8_t* a_base[LA];
  const uint8_t* b_base[LB];
  constexpr int B_STEP = K8 ? 16 * kRowBytes : kRowBytes;  // from one K-step of B to the next
  group_bases<PlanA>(p.A, p.lda_bytes, row0, wave, p.M, a_base);
  if constexpr (K8) block_bases<PlanB>(p.B, p.ldb_bytes, col0, wave, p.N, b_base);
  else group_bases<PlanB>(p.B, p.ldb_bytes, col0, wave, p.N, b_base);
  const int nk = p.ksteps - (p.tail_granules ? 1 : 0);  // whole 128-byte steps

  const int first = K8 && DT == ASTERGEMM_FP8_E4M3 ? 0 : first_step_of_xcd(p, nk);
  auto g2s = [&](const uint8_t* base, unsigned voff, uint8_t* dst) {
    const unsigned m0v = (unsigned)(size_t)AG_LDS(dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0v), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  auto issue_a1 = [&](int k, int stage, int j) {
    g2s(a_base[j] + (int64_t)step_from(first, k, nk) * kRowBytes, a_off, lds + stage * STAGE + PlanA::lds_offset(wave, j));
  };
  auto issue_b1 = [&](int k, int stage, int j) {
    g2s(b_base[j] + (int64_t)step_from(first, k, nk) * B_STEP, b_off,
        lds + stage * STAGE + B_AT + PlanB::lds_offset(wave, j));
  };

  // ---- LDS -> fragments: I < TN is B tile I, else A tile I - TN ------------------------------
  const int li = lane & 15, lq = lane >> 4;
  unsigned rd_off[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    rd_off[s] = (unsigned)(li * kRowBytes + (((s * 4 + lq) ^ (li >> 1)) << 4));
  unsigned rd_b[2];  // K8: a block of 16 rows is 2 KiB, lane for lane the fragments of its two halves
#pragma unroll
  for (int s = 0; s < 2; ++s) rd_b[s] = K8 ? (unsigned)(s * 1024 + lane * 16) : rd_off[s];
  const unsigned a_rd = (unsigned)(wm * TM * 16 * kRowBytes);
  const unsigned b_rd = (unsigned)(B_AT + wn * TN * 16 * kRowBytes);
  i32x4 fa[2][TM], fb[2][TN];
  auto read_one = [&](auto stage, auto sub, auto idx) {
    constexpr int S = decltype(sub)::value;
    constexpr int I = decltype(idx)::value;
    const uint8_t* st = lds + decltype(stage)::value * STAGE;
    if constexpr (I < TN) fb[S][I] = *(const i32x4*)(st + b_rd + I * 16 * kRowBytes + rd_b[S]);
    else fa[S][I - TN] = *(const i32x4*)(st + a_rd + (I - TN) * 16 * kRowBytes + rd_off[S]);
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  // ---- prologue: K-steps 0 ... NS - 1 requested; K-step 0 in registers, its first substep done
  static_for<0, NS>([&](auto ic) {
    constexpr int I = decltype(ic)::value;
    if (nk > I) {
#pragma unroll
      for (int j = 0; j < LB; ++j) issue_b1(I, I, j);
#pragma unroll
      for (int j = 0; j < LA; ++j) issue_a1(I, I, j);
    }
  });
  {
    const int behind = (nk < NS ? nk : NS) - 1;  // K-steps requested behind K-step 0
    static_for<0, NS>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      if (behind == I) __builtin_amdgcn_s_waitcnt(waitcnt_imm(I * L, 15));
    });
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_for<0, NF>([&](auto ic) { read_one(S0{}, S0{}, ic); });
  static_for<0, NF>([&](auto ic) { read_one(S0{}, S1{}, ic); });
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) stream_mma<DT, false>(fb[0][n], fa[0][m], acc[m][n]);
  __builtin_amdgcn_sched_barrier(0);

  // ---- K loop --------------------------------------------------------------------------------
  // Trip k finishes K-step k and starts K-step k + 1, like the trip of gemm_stream_body.  It begins
  // with a wait and a barrier: K-step k + 1 has landed for everybody (k + 2 ... k + NS - 1 may be
  // in flight) and every fragment of K-step k is in registers, which frees its stage for k + NS.
  auto trip = [&](int k, auto kmod, auto steady) {
    constexpr int KM = decltype(kmod)::value;
    constexpr bool STEADY = decltype(steady)::value;
    using KN = std::integral_constant<int, (KM + 1) % NS>;
    // the count holds while all of k + 2 ... k + NS - 1 were requested
    if (STEADY || k + NS - 1 < nk) __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * L, 0));
    else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bool do_ld = STEADY || k + NS < nk;
    static_for<0, NMF>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      stream_mma<DT, false>(fb[1][I / TM], fa[1][I % TM], acc[I % TM][I / TM]);
      if constexpr (I < LB) {
        if (do_ld) issue_b1(k + NS, KM, I);
      }
      if constexpr (I >= LB && I < LB + NF) read_one(KN{}, S0{}, std::integral_constant<int, I - LB>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    static_for<0, NMF>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      stream_mma<DT, false>(fb[0][I / TM], fa[0][I % TM], acc[I % TM][I / TM]);
      if constexpr (I < NF) read_one(KN{}, S1{}, std::integral_constant<int, I>{});
      if constexpr (I >= NF && I < NF + LA) {
        if (do_ld) issue_a1(k + NS, KM, I - NF);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  int k = 0;
  // steady: K-steps up to k + (NS - 1) + NS exist for the whole group of NS trips
  for (; k + 2 * NS <= nk; k += NS)
    static_for<0, NS>([&](auto ic) { trip(k + decltype(ic)::value, ic, std::true_type{}); });
  for (; k + 1 < nk; k += NS)
    static_for<0, NS>([&](auto ic) {
      if (k + decltype(ic)::value + 1 < nk) trip(k + decltype(ic)::value, ic, std::false_type{});
    });
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) stream_mma<DT, false>(fb[1][n], fa[1][m], acc[m][n]);

  if (p.tail_granules) stream_k_tail<DT, BM, BN, WM, WN>(p, acc, wave, row0, col0, nk);
  stream_epilogue<OUT, BM, BN, WM, WN, NS * STAGE>(p, acc, lds, wave, row0, col0);
}

// The same for fp8 e4m3.  A K-step is one v_mfma_scale_f32_16x16x128_f8f6f4 per 16 x 16 tile with
// 32 bytes of each operand per lane (granules lq and 4 + lq, as in gemm_stream8_body, so the bits
// are the same).  64 accumulators leave room for two whole sets of fragments (2 x 64 registers), so
// trip k multiplies set k mod 2 and reads K-step k + 1 into the other one.  The stage is a scalar that
// rotates from trip to trip: unrolled over six trips (both sets, three stages) it spilled 400 dwords.
template <int DT, int OUT, int BM, int BN, int WM, int WN, int NS, bool K8>
__device__ __forceinline__ void gemm_stream8r_body(const GemmArgs& p, int bid) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM / 16;
  constexpr int TN = BN / WN / 16;
  using PlanA = StreamLoadPlan<BM, NW>;
  using PlanB = StreamLoadPlan<BN, NW>;
  constexpr int LA = PlanA::LH, LB = PlanB::LH, L = LA + LB;
  constexpr int B_AT = BM * kRowBytes;
  constexpr int STAGE = (BM + BN) * kRowBytes;
  constexpr int NF = TM + TN;
  constexpr int NMF = TM * TN;
  constexpr int RPM = (2 * NF + NMF - 1) / NMF;               // 16-byte LDS reads behind each MFMA
  static_assert(PlanA::TILE_ROWS == 8 && PlanA::TILE_LDS_BYTES == 8 * kRowBytes, "transfer tile");
  static_assert(DT == ASTERGEMM_FP8_E4M3, "fp8 operands");
  static_assert(NS * STAGE <= 160 * 1024, "LDS of a CU");
  static_assert(LA * 8 * NW == BM && LB * 8 * NW == BN, "whole transfers");
  static_assert((8 * NW) % 16 == 0, "swizzle phase must not depend on the transfer index");
  static_assert(L <= NMF, "at most one transfer per MFMA");
  static_assert((NS - 1) * L <= 63, "vmcnt field");

  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int tile_m, tile_n;
  map_tile(bid, p.tiles_m, p.tiles_n, p.group_m, tile_m, tile_n);
  const int row0 = tile_m * BM, col0 = tile_n * BN;

  const int lrow = lane >> 3;
  const int g_lane = (lane & 7) ^ (((wave * 8 + lrow) >> 1) & 7);
  const unsigned a_off = (unsigned)(lrow * (int)p.lda_bytes + g_lane * 16);
  const unsigned b_off = K8 ? lane * 16 : (unsigned)(lrow * (int)p.ldb_bytes + g_lane * 16);
  const uint8_t* a_base[LA];
  const uint8_t* b_base[LB];
  constexpr int B_STEP = K8 ? 16 * kRowBytes : kRowBytes;  // from one K-step of B to the next
  group_bases<PlanA>(p.A, p.lda_bytes, row0, wave, p.M, a_base);
  if constexpr (K8) block_bases<PlanB>(p.B, p.ldb_bytes, col0, wave, p.N, b_base);
  else group_bases<PlanB>(p.B, p.ldb_bytes, col0, wave, p.N, b_base);
  const int nk = p.ksteps - (p.tail_granules ? 1 : 0);

  const int first = K8 && DT == ASTERGEMM_FP8_E4M3 ? 0 : first_step_of_xcd(p, nk);
  auto g2s = [&](const uint8_t* base, unsigned voff, uint8_t* dst) {
    const unsigned m0v = (unsigned)(size_t)AG_LDS(dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0v), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  // transfer j (0 ... L - 1) of K-step k: B's rows first, then A's
  auto issue1 = [&](int k, int stage, auto jc) {
    constexpr int J = decltype(jc)::value;
    if constexpr (J < LB)
      g2s(b_base[J] + (int64_t)step_from(first, k, nk) * B_STEP, b_off,
          lds + stage * STAGE + B_AT + PlanB::lds_offset(wave, J));
    else
      g2s(a_base[J - LB] + (int64_t)step_from(first, k, nk) * kRowBytes, a_off,
          lds + stage * STAGE + PlanA::lds_offset(wave, J - LB));
  };

  const int li = lane & 15, lq = lane >> 4;
  unsigned rd_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    rd_off[h] = (unsigned)(li * kRowBytes + (((h * 4 + lq) ^ (li >> 1)) << 4));
  unsigned rd_b[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) rd_b[h] = K8 ? (unsigned)(h * 1024 + lane * 16) : rd_off[h];
  const unsigned a_rd = (unsigned)(wm * TM * 16 * kRowBytes);
  const unsigned b_rd = (unsigned)(B_AT + wn * TN * 16 * kRowBytes);
  i32x8 fa[2][TM], fb[2][TN];
  // read I: half I & 1 of fragment I / 2 (below TN a B tile, else an A tile) into set S
  auto read_half = [&](int stage, auto set, auto idx) {
    constexpr int S = decltype(set)::value;
    constexpr int F = decltype(idx)::value / 2, H = decltype(idx)::value % 2;
    const unsigned at = F < TN ? b_rd + F * 16 * kRowBytes : a_rd + (F - TN) * 16 * kRowBytes;
    const i32x4 v = *(const i32x4*)(lds + stage * STAGE + at + (F < TN ? rd_b[H] : rd_off[H]));
    i32x8* f;
    if constexpr (F < TN) f = &fb[S][F];
    else f = &fa[S][F - TN];
#pragma unroll
    for (int e = 0; e < 4; ++e) (*f)[H * 4 + e] = v[e];
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  static_for<0, NS>([&](auto ic) {
    constexpr int I = decltype(ic)::value;
    if (nk > I) static_for<0, L>([&](auto jc) { issue1(I, I, jc); });
  });
  {
    const int behind = (nk < NS ? nk : NS) - 1;  // K-steps requested behind K-step 0
    static_for<0, NS>([&](auto ic) {
      constexpr int I = decltype(ic)::value;
      if (behind == I) __builtin_amdgcn_s_waitcnt(waitcnt_imm(I * L, 15));
    });
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_for<0, 2 * NF>([&](auto ic) { read_half(0, std::integral_constant<int, 0>{}, ic); });
  __builtin_amdgcn_sched_barrier(0);

  // Trip k: K-step k + 1 has landed (k + 2 ... k + NS - 1 may be in flight) and K-step k is in
  // registers for everybody, which frees its stage for k + NS.
  int stage = 0;  // k mod NS
  auto trip = [&](int k, auto set, auto steady) {
    constexpr int S = decltype(set)::value;
    const int next = stage + 1 == NS ? 0 : stage + 1;
    constexpr bool STEADY = decltype(steady)::value;
    const bool do_rd = STEADY || k + 1 < nk;
    if (do_rd) {
      if (STEADY || k + NS - 1 < nk) __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * L, 0));
      else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    const bool do_ld = STEADY || k + NS < nk;
    static_for<0, NMF>([&](auto mc) {
      constexpr int I = decltype(mc)::value;
      constexpr int n = I / TM, m = I % TM;
      // cbsz = blgp = 0: both operands OCP e4m3; zero scale operands select the unscaled form
      acc[m][n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[S][n], fa[S][m], acc[m][n], 0, 0,
                                                                   0, 0, 0, 0);
      if constexpr (I < L) {
        if (do_ld) issue1(k + NS, stage, mc);
      }
      if (do_rd)
        static_for<I * RPM, (I + 1) * RPM>([&](auto rc) {
          if constexpr (decltype(rc)::value < 2 * NF)
            read_half(next, std::integral_constant<int, S ^ 1>{}, rc);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
    stage = next;
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  int k = 0;
  // steady: K-step k + 1 + NS exists for the second trip of a pair
#pragma unroll 1
  for (; k + 2 + NS <= nk; k += 2) {
    trip(k, S0{}, std::true_type{});
    trip(k + 1, S1{}, std::true_type{});
  }
#pragma unroll 1
  for (; k < nk; k += 2) {
    trip(k, S0{}, std::false_type{});
    if (k + 1 < nk) trip(k + 1, S1{}, std::false_type{});
  }
  __builtin_amdgcn_sched_barrier(0);

  if (p.tail_granules) stream_k_tail<DT, BM, BN, WM, WN>(p, acc, wave, row0, col0, nk);
  stream_epilogue<OUT, BM, BN, WM, WN, NS * STAGE>(p, acc, lds, wave, row0, col0);
}

template <int DT, int OUT, int BM, int BN, int WM, int WN, int NS, bool K8 = false>
__global__ __launch_bounds__(WM* WN * 64) void gemm_streamr_kernel(const GemmArgs p) {
  if constexpr (DT == ASTERGEMM_FP8_E4M3) gemm_stream8r_body<DT, OUT, BM, BN, WM, WN, NS, K8>(p, blockIdx.x);
  else gemm_streamr_body<DT, OUT, BM, BN, WM, WN, NS, K8>(p, blockIdx.x);
}

// Split K (see gemm_stream_splitk_kernel): copy s of the tile grid multiplies K steps
// [s * p.ksteps, (s + 1) * p.ksteps) into plane s of the fp32 workspace.
template <int DT, int BM, int BN, int WM, int WN, int NS>
__global__ __launch_bounds__(WM* WN * 64) void gemm_streamr_splitk_kernel(const GemmArgs p) {
  const int tiles = p.tiles_m * p.tiles_n;
  const int ks = blockIdx.x / tiles;
  const int bid = blockIdx.x - ks * tiles;
  GemmArgs q = p;
  q.A = p.A + (int64_t)ks * p.ksteps * kRowBytes;
  q.B = p.B + (int64_t)ks * p.ksteps * kRowBytes;
  q.C = p.workspace + (int64_t)ks * p.M * p.N;
  if constexpr (DT == ASTERGEMM_FP8_E4M3) gemm_stream8r_body<DT, ASTERGEMM_F32, BM, BN, WM, WN, NS, false>(q, bid);
  else gemm_streamr_body<DT, ASTERGEMM_F32, BM, BN, WM, WN, NS, false>(q, bid);
}

}  // namespace
}  // namespace astergemm
