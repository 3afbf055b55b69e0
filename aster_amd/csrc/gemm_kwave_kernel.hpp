// K split over the waves of a workgroup: C[M,N] = epi(A[M,K] * B[N,K]^T) for problems with at most about
// one small output tile per CU -- decoding (M <= 64 rows against a whole weight matrix) and small products.
// Which shape runs what, and what each measured, stands at the rules in gemm_kwave.hip.
//
// What bounds these problems is how early and how evenly the operands arrive, not the matrix cores: a CU
// needs its rows once, from HBM (decoding) or L2 (small products), and 128 bytes of every row are gone
// in a few MFMAs.  So:
//   * the WK wave groups of a workgroup take the 128-byte K-steps round robin.  Each group stages its own
//     steps, 8 rows x 128 bytes per transfer, straight into its part of an LDS ring of S stages and
//     multiplies the whole BM x BN tile with them; the groups' sums are added once, through LDS, at the
//     end.  A group of one wave (WM = WN = 1) waits for nobody: no barrier in the loop, only its own
//     transfers' counter.  Up to 160 KiB of operands are on their way at any time.
//   * nothing of A is kept from one weight row to the next (decode kernels that hold the activations in
//     registers need rows of whole slices, and K ranges with a second kernel for long ones): any row length
//     of whole 16-byte granules is one launch.
//   * workgroups start their K loop at different K-steps (`rot`).  In step, all CUs ask for the same
//     columns of every weight row, and with rows a multiple of a few KiB apart those are few HBM channels:
//     bf16 8x8192x8192 28.3 us in step, 21.4 rotated; 64x14336x4096 25.3 -> 22.9; 64x28672x4096 49.3 -> 37.7;
//     fp8 8x8192x8192 17.6 -> 11.2.
//   * K8: weights pre-shuffled (ASTERGEMM_OPERAND_DIRECT_B_K8), staged as they lie: 16 rows x 128 bytes are 2 KiB in
//     one piece, lane for lane the operands of the 16 x 16 tile, so a transfer is 1 KiB of consecutive bytes and a
//     fragment read 1 KiB of consecutive LDS.  MXFP4: both scale planes in lane order, whose bytes a lane reads
//     are its own: two tiles' bytes are a dword per lane.
// Sums: a K-step's products in MFMA order, a group's steps in rotated order, the groups in index order: the
// same bits on every run of a config.
#pragma once
#include "gemm_tile_kernel.hpp"

namespace astergemm {
namespace {

// What PackedArgs::form says: weight rows of a workgroup (a multiple of 8, at most BN), K ranges (1: the result;
// more: fp32 planes in the workspace), output type, whether weights are fetched past the last-level cache, whether the
// tile rows of a panel are on one XCD (else tile after tile, whatever the XCD), and with K ranges the workgroups of
// one.
struct KwaveForm32 {
  int per, ranges, out, nt, by_panel, blocks;
  __host__ __device__ uint32_t bits() const {
    return (uint32_t)(per >> 3) | (uint32_t)ranges << 5 | (uint32_t)out << 10 | (uint32_t)nt << 13 |
           (uint32_t)by_panel << 14 | (uint32_t)(ranges > 1 ? blocks : 0) << 16;
  }
  __host__ __device__ static KwaveForm32 of(uint32_t b) {
    return KwaveForm32{(int)(b & 31) << 3, (int)(b >> 5 & 31), (int)(b >> 10 & 7), (int)(b >> 13 & 1),
                       (int)(b >> 14 & 1), (int)(b >> 16)};
  }
};

// 32-row transfers of e8m0 bytes per K-step (K8: of each operand by itself)
constexpr int kwave_scale_loads(int dt, bool k8, int bm, int bn) {
  return dt != ASTERGEMM_MXFP4 ? 0 : k8 ? (bm + 31) / 32 + (bn + 31) / 32 : (bm + bn + 31) / 32;
}
constexpr int kwave_step_bytes(int dt, bool k8, int bm, int bn) {  // LDS of one K-step of a wave group
  return (bm + bn) * kRowBytes + kwave_scale_loads(dt, k8, bm, bn) * 256;
}

template <int DT, bool K8, int BM, int BN, int WM, int WN, int WK, int S>
__global__ __launch_bounds__(WM* WN* WK * 64) void gemm_kwave_kernel(const PackedArgs args) {
  constexpr int GW = WM * WN;                   // waves of a group
  constexpr int NW = GW * WK;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int GA = BM / 8, G = GA + BN / 8;   // 8-row transfers of a K-step, A's first
  constexpr bool FP4 = DT == ASTERGEMM_MXFP4;
  constexpr int NSX = kwave_scale_loads(DT, K8, BM, BN);
  constexpr int LG = G / GW, LS = (NSX + GW - 1) / GW, L = LG + LS;  // transfers per wave and stage
  constexpr int B_AT = BM * kRowBytes, SCALES = (BM + BN) * kRowBytes;
  constexpr int STEP = kwave_step_bytes(DT, K8, BM, BN), STAGE = STEP * WK;
  constexpr int NT = (BM / 16) * (BN / 16);     // 16 x 16 tiles of the workgroup
  constexpr int TPW = (NT + NW - 1) / NW;       // of them finished by one wave
  static_assert(G % GW == 0, "whole transfers per wave");
  static_assert(S >= 2 && (S - 2) * L <= 63, "the counted wait fits the vmcnt field");
  static_assert(S * STAGE <= 160 * 1024 && WK * NT * 1024 <= S * STAGE, "LDS of a CU");

  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const GemmArgs p = unpack_args<DT>(args);
  const KwaveForm32 q = KwaveForm32::of(args.form);
  const int tiles_m = (p.M + BM - 1) / BM;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave / GW, wv = wave % GW, wm = wv / WN, wn = wv % WN;

  // block b runs on XCD b % 8: the tile rows of a weight panel side by side on one XCD, the panels round
  // robin over the XCDs (runs of neighbouring panels per XCD: fp8 8x8192x8192 11.0 -> 15.5 us, the panels
  // that start at the same K-step are then a large power of two apart)
  int range = 0, bid = blockIdx.x, range_steps = p.ksteps;
  if (q.ranges > 1) {
    range = bid / q.blocks;
    bid -= range * q.blocks;
    range_steps = (p.ksteps + q.ranges - 1) / q.ranges;
  }
  const int idx = q.by_panel ? bid >> 3 : bid, panel = idx / tiles_m;
  const int tile_m = idx - panel * tiles_m, tile_n = q.by_panel ? panel * 8 + (bid & 7) : panel;
  if ((int64_t)tile_n * q.per >= p.N) return;
  const int row0 = tile_m * BM, col0 = tile_n * q.per;
  const int col1 = (col0 + q.per) < p.N ? (col0 + q.per) : p.N;
  const int k0 = range * range_steps;
  const int k1 = (k0 + range_steps) < p.ksteps ? (k0 + range_steps) : p.ksteps;
  const int kwhole = p.tail_granules && k1 == p.ksteps ? k1 - 1 : k1;  // steps of 128 bytes
  const int nst = (k1 - k0 + WK - 1) / WK;
  const int rot = panel % nst;

  // ---- global -> LDS: 128-byte rows, granule index XOR ((row >> 1) & 7) ----------------------
  // Rows past the end repeat the last valid one (the same lines); their products are never stored.
  const uint8_t* a_base = p.A + (int64_t)row0 * p.lda_bytes;
  const uint8_t* b_base = p.B + (int64_t)col0 * p.ldb_bytes;
  unsigned off[LG];
  int gran[LG];
#pragma unroll
  for (int j = 0; j < LG; ++j) {
    const int t = wv + j * GW;
    const bool is_a = t < GA;
    int r = (is_a ? t : t - GA) * 8 + (lane >> 3);
    gran[j] = (lane & 7) ^ ((r >> 1) & 7);
    const int last = is_a ? p.M - 1 - row0 : col1 - 1 - col0;
    r = r < last ? r : last;
    off[j] = (unsigned)(r * (int)(is_a ? p.lda_bytes : p.ldb_bytes) + gran[j] * 16);
    if (K8 && !is_a) {  // half (t - GA) & 1 of a block of 16 rows (ranges of whole blocks: past the end the last one)
      const int blk = (t - GA) >> 1, last_blk = ((col1 - col0) >> 4) - 1;
      off[j] = (unsigned)((blk < last_blk ? blk : last_blk) * 16 * (int)p.ldb_bytes + ((t - GA) & 1) * 1024 + lane * 16);
    }
  }
  constexpr int B_STEP = K8 ? 16 * kRowBytes : kRowBytes;  // from one K-step of B to the next
  const uint8_t* s_src[LS ? LS : 1];            // e8m0: 8 bytes per row and K-step, A's rows first
  int s_step[K8 && FP4 ? LS : 1];
  if constexpr (FP4 && K8) {
    // lane order: tiles t, t + 1 (t even) of lane L are 4 bytes at 16 L + 2 t of A's 128-row group (1 KiB per
    // K-step), at 8 L + 2 t of B's 64-row group (512 bytes); pairs of tiles, A's first
    constexpr int PA = (BM + 31) / 32;
#pragma unroll
    for (int j = 0; j < LS; ++j) {
      int x = wv + j * GW;
      x = x < NSX ? x : NSX - 1;                // a surplus transfer repeats the last one: the same bytes
      if (x < PA) {
        // pairs past the last group of A's plane, whose rows are never stored, repeat its last
        int t = ((row0 >> 4) & ~1) + 2 * x;
        const int last = ((p.M - 1) >> 7) * 8 + 6;
        t = t < last ? t : last;
        s_src[j] = p.mx_a + (int64_t)(t >> 3) * p.ksteps * 1024 + lane * 16 + (t & 7) * 2;
        s_step[j] = 1024;
      } else {
        int t = ((col0 >> 4) & ~1) + 2 * (x - PA);
        const int last = (p.N >> 4) - 2;
        t = t < last ? t : last;
        s_src[j] = p.mx_b + (int64_t)(t >> 2) * p.ksteps * 512 + lane * 8 + (t & 3) * 2;
        s_step[j] = 512;
      }
    }
  } else if constexpr (FP4) {
#pragma unroll
    for (int j = 0; j < LS; ++j) {
      int x = wv + j * GW;
      x = x < NSX ? x : NSX - 1;                // a surplus transfer repeats the last one: the same bytes
      int r = x * 32 + (lane >> 1);
      r = r < BM + BN ? r : BM + BN - 1;
      const bool is_a = r < BM;
      r = is_a ? row0 + r : col0 + r - BM;
      const int last = is_a ? p.M - 1 : col1 - 1;
      r = r < last ? r : last;
      s_src[j] = (is_a ? p.mx_a : p.mx_b) + (int64_t)r * p.mx_ld + (lane & 1) * 4;
    }
  }
  auto m0_of = [&](const uint8_t* dst) { return (unsigned)(size_t)AG_LDS(dst); };
  auto g2s = [&](const uint8_t* base, unsigned voff, const uint8_t* dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0_of(dst)), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  auto g2s_nt = [&](const uint8_t* base, unsigned voff, const uint8_t* dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(m0_of(dst)), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  auto g2s_lane = [&](const uint8_t* src, const uint8_t* dst) {  // from an address per lane
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(m0_of(dst)), "v"(src)
                 : "memory", "m0");
  };
  auto g2s_dword = [&](const uint8_t* src, const uint8_t* dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                 :
                 : "s"(m0_of(dst)), "v"(src)
                 : "memory", "m0");
  };
  auto s_stride = [&](int j) {
    if constexpr (K8 && FP4) return s_step[j];
    else return 8;
  };
  auto issue = [&](int st, int slot) {          // this group's K-step of stage st
    int sr = st + rot;
    sr = sr < nst ? sr : sr - nst;
    const int k = k0 + sr * WK + wk;
    const uint8_t* d = lds + slot * STAGE + wk * STEP;
    const uint8_t* ga = a_base + (int64_t)k * kRowBytes;
    const uint8_t* gb = b_base + (int64_t)k * B_STEP;
    auto dst = [&](int j) {
      const int t = wv + j * GW;
      return d + (t < GA ? t * 1024 : B_AT + (t - GA) * 1024);
    };
    if (k >= kwhole) {
      // the last, partial step of a row, or none at all: granules past the end come from a block of zeros
      const int live = k < k1 ? p.tail_granules : 0;
#pragma unroll
      for (int j = 0; j < LG; ++j)
        g2s_lane(gran[j] < live ? (wv + j * GW < GA ? ga : gb) + off[j] : g_zero16, dst(j));
    } else if (q.nt) {
#pragma unroll
      for (int j = 0; j < LG; ++j) {
        if (wv + j * GW < GA) g2s(ga, off[j], dst(j));
        else g2s_nt(gb, off[j], dst(j));
      }
    } else {
#pragma unroll
      for (int j = 0; j < LG; ++j) g2s(wv + j * GW < GA ? ga : gb, off[j], dst(j));
    }
    if constexpr (FP4) {
#pragma unroll
      for (int j = 0; j < LS; ++j) {
        int x = wv + j * GW;
        x = x < NSX ? x : NSX - 1;
        g2s_dword(k < k1 ? s_src[j] + (int64_t)k * s_stride(j) : g_zero16, d + SCALES + x * 256);
      }
    }
  };

  // ---- what the epilogue needs from memory, requested ahead of everything else ---------------
  const int li = lane & 15, lq = lane >> 4;
  float scale = 1.0f;
  f32x4 bias_v[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    bias_v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int t = wave + i * NW;
    if (p.bias && q.ranges == 1 && t < NT) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int col = col0 + (t % (BN / 16)) * 16 + 4 * lq + e;
        bias_v[i][e] = p.bias[col < p.N ? col : p.N - 1];
      }
    }
  }
  if (p.scale_a && q.ranges == 1) scale *= *p.scale_a;
  if (p.scale_b && q.ranges == 1) scale *= *p.scale_b;

  // ---- LDS -> fragments: lane (li, lq) has row li, granule 4 s + lq (16-bit, fp4) or 2 lq + s (fp8)
  unsigned rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    rd[s] = (unsigned)(li * kRowBytes + (((DT == ASTERGEMM_FP8_E4M3 ? 2 * lq + s : 4 * s + lq) ^ (li >> 1)) << 4));
  unsigned rd_b[2];  // K8: granule g of row li of a block is at (g / 4) KiB, lane 16 (g mod 4) + li
#pragma unroll
  for (int s = 0; s < 2; ++s)
    rd_b[s] = !K8 ? rd[s]
              : DT == ASTERGEMM_FP8_E4M3 ? (unsigned)((lq >> 1) * 1024 + (((lq & 1) * 2 + s) * 16 + li) * 16)
                                         : (unsigned)(s * 1024 + lane * 16);
  f32x4 acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int st = 0; st < S - 1; ++st)
    if (st < nst) issue(st, st);

  int slot = 0, slot_ld = S - 1;  // stage st is in slot st mod S; the next transfers go to slot_ld
  auto trip = [&](int st) {
    // the group's stage st is complete, and stage st - 1 is in its registers
    if constexpr (GW > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (st + S - 1 < nst) issue(st + S - 1, slot_ld);
    const uint8_t* sp = lds + slot * STAGE + wk * STEP;
    i32x4 af[2][TM], bf[2][TN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int m = 0; m < TM; ++m) af[s][m] = *(const i32x4*)(sp + (wm * TM + m) * 16 * kRowBytes + rd[s]);
#pragma unroll
      for (int n = 0; n < TN; ++n)
        bf[s][n] = *(const i32x4*)(sp + B_AT + (wn * TN + n) * 16 * kRowBytes + rd_b[s]);
    }
    i32x2 sa[FP4 ? TM : 1], sb[FP4 ? TN : 1];
    if constexpr (FP4 && K8) {
      // bytes 0, 1 of a word: substeps 0, 1 of the pair's first tile, bytes 2, 3 of its second
      constexpr int PA = (BM + 31) / 32;
      const int ta = ((row0 >> 4) & 1) + wm * TM, tb = ((col0 >> 4) & 1) + wn * TN;
#pragma unroll
      for (int m = 0; m < TM; ++m)
        sa[m][0] = *(const int*)(sp + SCALES + ((ta + m) >> 1) * 256 + lane * 4) >> (((ta + m) & 1) * 16);
#pragma unroll
      for (int n = 0; n < TN; ++n)
        sb[n][0] = *(const int*)(sp + SCALES + (PA + ((tb + n) >> 1)) * 256 + lane * 4) >> (((tb + n) & 1) * 16);
    } else if constexpr (FP4) {
#pragma unroll
      for (int m = 0; m < TM; ++m) sa[m] = *(const i32x2*)(sp + SCALES + ((wm * TM + m) * 16 + li) * 8);
#pragma unroll
      for (int n = 0; n < TN; ++n) sb[n] = *(const i32x2*)(sp + SCALES + (BM + (wn * TN + n) * 16 + li) * 8);
    }
    if constexpr (DT == ASTERGEMM_FP8_E4M3) {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          const i32x4 b[2] = {bf[0][n], bf[1][n]}, a[2] = {af[0][m], af[1][m]};
          acc[m][n] = mfma_step<DT>(b, a, acc[m][n], 0, 0);
        }
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n) {
            int xa = 0, xb = 0;
            if constexpr (FP4 && K8) {
              xa = (int)((unsigned)sa[m][0] >> (8 * s));
              xb = (int)((unsigned)sb[n][0] >> (8 * s));
            } else if constexpr (FP4) {
              xa = (int)((unsigned)sa[m][s] >> (8 * lq));
              xb = (int)((unsigned)sb[n][s] >> (8 * lq));
            }
            acc[m][n] = mfma_step<DT>(&bf[s][n], &af[s][m], acc[m][n], xb, xa);
          }
    }
    slot = slot == S - 1 ? 0 : slot + 1;
    slot_ld = slot_ld == S - 1 ? 0 : slot_ld + 1;
  };
  int st = 0;
  for (; st + S - 2 < nst; ++st) {  // S - 2 younger stages have been requested
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 2) * L, 0));
    trip(st);
  }
  for (; st < nst; ++st) {          // the last S - 2: nothing left to request
    const int younger = nst - 1 - st;
    static_for_stages<0, S - 2>([&](auto c) {
      constexpr int n = decltype(c)::value;
      if (younger == n) __builtin_amdgcn_s_waitcnt(waitcnt_imm(n * L, 0));
    });
    trip(st);
  }

  // ---- the groups' sums, added in index order; scale, bias, cast, store ----------------------
  __syncthreads();                  // everybody has left the ring
  f32x4* red = (f32x4*)lds;
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n)
      red[(wk * NT + (wm * TM + m) * (BN / 16) + wn * TN + n) * 64 + lane] = acc[m][n];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int t = wave + i * NW;
    if (t >= NT) break;
    f32x4 v = red[t * 64 + lane];
#pragma unroll
    for (int g = 1; g < WK; ++g) v += red[(g * NT + t) * 64 + lane];
    const int row = row0 + (t / (BN / 16)) * 16 + li, col = col0 + (t % (BN / 16)) * 16 + 4 * lq;
    if (row >= p.M || col >= col1) continue;
    const int ncols = (col1 - col) < 4 ? (col1 - col) : 4;
    if (q.ranges > 1) {
      store4<ASTERGEMM_F32>(p.C, ((int64_t)range * p.M + row) * p.N + col, v, ncols);
      continue;
    }
    v *= scale;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += bias_v[i][e];
    const int64_t idx = (int64_t)row * p.ldc + col;
    if (q.out == ASTERGEMM_F32) store4<ASTERGEMM_F32>(p.C, idx, v, ncols);
    else if (q.out == ASTERGEMM_BF16) store4<ASTERGEMM_BF16>(p.C, idx, v, ncols);
    else store4<ASTERGEMM_F16>(p.C, idx, v, ncols);
  }
}

}  // namespace
}  // namespace astergemm
