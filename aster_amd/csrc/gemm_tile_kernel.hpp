// LDS-staged MFMA tile kernels for gfx950 (CDNA4): C[M,N] = epi(A[M,K] * B[N,K]^T).
//
// One kernel body serves four operand encodings because they share one byte
// geometry: a K-step is 128 bytes of an operand row (64 bf16/f16, 128 fp8,
// 256 fp4), which the matrix core consumes in 32 cycles per 16x16 tile pair in
// every encoding (2 x 16x16x32 for 16-bit, 1 x 16x16x128 for fp8, 2 x 16x16x128
// for fp4).
//
// What the reference does for the same job, as generated AMDGCN:
//   * global -> LDS with `buffer_load_dwordx4 ... lds`, XOR-swizzled through the
//     global source address because the LDS side of that instruction is linear
//     (python/aster/dialects/kernel_builder_with_layouts.py:371-481,
//      contrib/kittens/test/test_102_gemm_python_multitile_g2s_lds_cdna4.py:142);
//   * LDS -> VGPR MFMA fragments (contrib/kittens/library/lds_mfma_16x64_b.mlir);
//   * v_mfma_f32_16x16x32_f16 inner loop over (k, m, n) tiles with AGPR
//     accumulators (test_102_..._g2s_directb_cdna4.py:296-306);
//   * row-major workgroup -> (m, n) tile mapping (same file :201-203).
// Here: 128-byte LDS rows, 16-byte granule index XOR ((row >> 1) & 7) so that a
// ds_read_b128 of 16 rows x one granule touches 16 distinct 16-byte bank groups;
// fragments are read with ds_read_b128; accumulators are computed transposed
// (srcA = B rows, srcB = A rows) so each lane owns 4 consecutive columns of one
// C row and the epilogue stores 8/16-byte vectors.
#pragma once
#include <type_traits>

#include "astergemm_internal.h"

namespace astergemm {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

#define AG_LDS(p) ((__attribute__((address_space(3))) void*)(p))
#define AG_GLOBAL(p) ((const __attribute__((address_space(1))) void*)(p))

constexpr int kRowBytes = 128;  // bytes of one operand row per K-step

// Source of the 16-byte transfers that lie past the end of a row.
__device__ __attribute__((aligned(16))) const uint8_t g_zero16[16] = {0};

// s_waitcnt immediate for gfx9: vmcnt[3:0]|[15:14], expcnt[6:4], lgkmcnt[11:8].
constexpr int waitcnt_imm(int vm, int lgkm) {
  return (vm & 0xF) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 0xF) << 8);
}

__device__ __forceinline__ float bf16_bits_to_f32(unsigned short b) {
  return __builtin_bit_cast(float, (unsigned)b << 16);
}

// fp32 -> bf16 round-to-nearest-even, NaN kept quiet.
// Four fp32 values to four 16-bit outputs, round to nearest even, with the hardware
// converters (v_cvt_pk_bf16_f32 / v_cvt_f16_f32): the integer bf16 rounding sequence is six
// VALU operations per element, which made the epilogue of a 256x256 tile VALU bound.
template <int OUT>
__device__ __forceinline__ u16x4 cast4_16(f32x4 v) {
  if constexpr (OUT == ASTERGEMM_BF16) {
    typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(u16x4, __builtin_convertvector(v, bf16x4_t));
  } else {
    typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(u16x4, __builtin_convertvector(v, f16x4_t));
  }
}

// Hardware hands workgroup b to XCD b % 8.  Give each XCD one contiguous run of
// the logical tile order, then walk that order in groups of `group_m` tile rows
// (column-major inside a group) so the 32 workgroups resident on an XCD share
// A and B panels through that XCD's L2.
__device__ __forceinline__ void map_tile(int bid, int tiles_m, int tiles_n,
                                         int group_m, int& tm, int& tn) {
  if (group_m < 0) {
    // band order (tiles_m % 8 == 0, tiles_n % 8 == 0): all eight XCDs work on the same band of
    // eight tile rows, XCD x on its own tiles_n / 8 tile columns of it, so that a band of A is
    // fetched from HBM once and reaches the other seven XCDs from the last-level cache
    const int xcd = bid & 7, idx = bid >> 3;
    const int cols = tiles_n >> 3;               // tile columns of an XCD
    const int per_band = 8 * cols;               // tiles of an XCD in one band
    const int band = idx / per_band, j = idx - band * per_band;
    tm = band * 8 + (j & 7);
    tn = xcd * cols + (j >> 3);
    return;
  }
  const int total = tiles_m * tiles_n;
  const int q = total >> 3, rem = total & 7;
  const int xcd = bid & 7, idx = bid >> 3;
  const int logical = xcd * q + (xcd < rem ? xcd : rem) + idx;
  const int gsz = group_m * tiles_n;
  const int g = logical / gsz;
  const int first_m = g * group_m;
  const int rows = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
  const int r = logical - g * gsz;
  tm = first_m + r % rows;
  tn = r / rows;
}

// Workgroup b of `ranges` copies of a grid of `tiles` output tiles -> its K range and its number in the tile grid
// (what map_tile takes).  A range is on as few XCDs as there are for it (8 / ranges of them, two ranges on each for
// 16; where its tiles do not divide among them, or the ranges are no power of two, on all).  Its tiles lie side by
// side there and the XCD's L2 holds the range's rows once for all of them, where with every range on every XCD each
// reads all of A.  Every range on every XCD / this, us, 128 x 128 tiles: f16 1391x1024x8192 40.6 / 35.1, bf16
// 900x1024x8192 29.0 / 25.2, 634x1024x8192 25.7 / 23.9, 240x4096x11008 43.8 / 42.7, fp8 558x1024x8192 29.5 / 27.9.
// Not for MXFP4 (700x1024x8192 20.5 / 22.2, 162x4096x14336 22.7 / 23.3) and not on 256 x 128 tiles, whose XCDs then
// stream weights a quarter of the row apart from memory: bf16 324x8192x28672 198 / 211, 333x4096x14336 59.1 / 62.1
// (weights in the last-level cache: 54.2 / 54.3).
__device__ __forceinline__ void place_range(int b, int tiles, int ranges, int& range, int& bid) {
  const int xcds = ranges < 8 ? 8 / ranges : 1;  // XCDs of a range
  const int share = tiles / xcds;                // tiles of a range on one of them
  if (ranges > 16 || (ranges & (ranges - 1)) != 0 || share * xcds != tiles) {
    range = b / tiles;
    bid = b - range * tiles;
    return;
  }
  const int xcd = b & 7, i = b >> 3, second = i / share;
  range = ranges == 16 ? xcd * 2 + second : xcd / xcds;
  const int logical = (xcd & (xcds - 1)) * share + i - second * share;
  // map_tile gives XCD x the logical tiles from x * q + min(x, rem) on
  const int q = tiles >> 3, rem = tiles & 7, head = rem * (q + 1);
  const int x = logical < head ? logical / (q + 1) : rem + (logical - head) / q;
  bid = ((logical - x * q - (x < rem ? x : rem)) << 3) + x;
}

// What a packed kernel argument says, apart from the tile grid and the workspace.
template <int DT>
__device__ __forceinline__ GemmArgs unpack_args(const PackedArgs& q) {
  GemmArgs a = {};
  auto ptr = [&](int i) {  // by way of a global pointer: loads and stores stay global ones
    return (uint8_t*)(__attribute__((address_space(1))) uint8_t*)((uint64_t)q.hi[i] << 32 | q.lo[i]);
  };
  a.A = ptr(0);
  a.B = ptr(1);
  a.C = ptr(2);
  a.bias = (const float*)ptr(3);
  if constexpr (DT == ASTERGEMM_MXFP4) {
    a.mx_a = ptr(4);
    a.mx_b = ptr(5);
    a.mx_ld = q.K >> 5;
  } else {
    a.scale_a = (const float*)ptr(4);
    a.scale_b = (const float*)ptr(5);
  }
  a.M = q.M, a.N = q.N, a.K = q.K;
  a.lda_bytes = (int64_t)(q.lda & 0x7FFFF) << 4;
  a.ldb_bytes = (int64_t)(q.ldb & 0x7FFFF) << 4;
  a.ldc = (int64_t)((uint64_t)(q.ldb >> 19) << 45 | (uint64_t)(q.lda >> 19) << 32 | q.ldc);
  const unsigned rb = DT == ASTERGEMM_MXFP4 ? (unsigned)q.K >> 1 : DT == ASTERGEMM_FP8_E4M3 ? (unsigned)q.K
                                                                                       : (unsigned)q.K * 2;
  a.ksteps = (int)((rb + 127) >> 7);
  a.tail_granules = (int)((rb & 127) >> 4);
  return a;
}

template <int DT>
struct Enc {
  // MFMA k-substeps per 128-byte row chunk and 16-byte granules per fragment.
  static constexpr int kSub = (DT == ASTERGEMM_FP8_E4M3) ? 1 : 2;
  static constexpr int kGran = (DT == ASTERGEMM_FP8_E4M3) ? 2 : 1;
  static constexpr int kElemsPerStep =
      (DT == ASTERGEMM_FP8_E4M3) ? 128 : (DT == ASTERGEMM_MXFP4 ? 256 : 64);
};

// One MFMA: acc += srcA(16 x k) * srcB(k x 16), operands as raw dwords.
template <int DT>
__device__ __forceinline__ f32x4 mfma_step(const i32x4* a, const i32x4* b, f32x4 c,
                                           int sa, int sb) {
  if constexpr (DT == ASTERGEMM_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a[0]), __builtin_bit_cast(bf16x8, b[0]), c, 0, 0, 0);
  } else if constexpr (DT == ASTERGEMM_F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(f16x8, a[0]), __builtin_bit_cast(f16x8, b[0]), c, 0, 0, 0);
  } else if constexpr (DT == ASTERGEMM_FP8_E4M3) {
    i32x8 av = {a[0].x, a[0].y, a[0].z, a[0].w, a[1].x, a[1].y, a[1].z, a[1].w};
    i32x8 bv = {b[0].x, b[0].y, b[0].z, b[0].w, b[1].x, b[1].y, b[1].z, b[1].w};
    // cbsz = blgp = 0: both operands OCP e4m3; zero scale operands select the
    // unscaled form of the instruction.
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 0, 0, 0);
  } else {
    i32x8 av = {a[0].x, a[0].y, a[0].z, a[0].w, 0, 0, 0, 0};
    i32x8 bv = {b[0].x, b[0].y, b[0].z, b[0].w, 0, 0, 0, 0};
    // cbsz = blgp = 4: both operands e2m1; byte 0 of sa / sb is the e8m0 scale
    // of this lane's 32 K-elements.
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 4, 4, 0, sa, 0, sb);
  }
}

template <int I, int N, class Fn>
__device__ __forceinline__ void static_for_stages(Fn&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_stages<I + 1, N>(f);
  }
}

// C[row][col .. col + ncols) = cast(v): one vector store where all four columns exist (the vector
// memory path takes any element alignment, so an odd row pitch costs nothing extra).
template <int OUT>
__device__ __forceinline__ void store4(void* C, int64_t idx, f32x4 v, int ncols) {
  typedef f32x4 f32x4_el __attribute__((aligned(4)));
  typedef u16x4 u16x4_el __attribute__((aligned(2)));
  if constexpr (OUT == ASTERGEMM_F32) {
    float* p = (float*)C + idx;
    if (ncols == 4) {
      *(f32x4_el*)p = v;
    } else {
      for (int r = 0; r < ncols; ++r) p[r] = v[r];
    }
  } else {
    const u16x4 h = cast4_16<OUT>(v);
    unsigned short* p = (unsigned short*)C + idx;
    if (ncols == 4) {
      *(u16x4_el*)p = h;
    } else {
      for (int r = 0; r < ncols; ++r) p[r] = h[r];
    }
  }
}

// K loop: LDS is a ring of S stages (A and B rows of one K-step, MXFP4: and their scale bytes).
// While K-step k is multiplied, the transfers of k + 1 .. k + S - 1 are in flight: with the two
// stages this kernel had before, every K-step waited for its own transfers, about 0.7 us of memory
// latency per 128 bytes of row, whatever the tile.  A trip starts with the wait for stage k (the
// younger ones stay outstanding), one barrier -- stage k is complete for everybody and everybody
// has stage k - 1 in registers -- and the transfers of k + S - 1 into the slot of k - 1.  Transfers
// are inline assembly, so that the compiler does not wait for them on its own; nothing else that
// counts in vmcnt is issued inside the loop.
template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
__device__ __forceinline__ void gemm_tile_body(const GemmArgs& p) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM / 16;  // 16-row MFMA tiles per wave along M
  constexpr int TN = BN / WN / 16;
  constexpr bool FP4 = DT == ASTERGEMM_MXFP4;
  constexpr int SCALES = (BM + BN) * kRowBytes;  // offset of the scale bytes in a stage (MXFP4)
  constexpr int STAGE = SCALES + (FP4 ? (BM + BN) * 8 : 0);
  constexpr int LA = BM / 8 / NW;  // 1 KiB (8-row) global->LDS transfers per wave
  constexpr int LB = BN / 8 / NW;
  // scale transfers: 4 bytes per lane, 32 rows each, round robin over the waves
  constexpr int NSX = (BM + BN) / 32;
  constexpr int LS = FP4 ? (NSX + NW - 1) / NW : 0;
  constexpr int L = LA + LB + LS;
  constexpr int KSUB = Enc<DT>::kSub;
  constexpr int KGRAN = Enc<DT>::kGran;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile rows per wave");
  static_assert((8 * NW) % 16 == 0, "swizzle phase must not depend on the transfer index");
  static_assert(S >= 2 && (S - 2) * L <= 63, "the counted wait fits the vmcnt field");
  static_assert(BM % 32 == 0 && BN % 32 == 0, "scale transfers cover 32 rows");

  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  int tile_m, tile_n;
  map_tile(blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, tile_m, tile_n);
  const int row0 = tile_m * BM, col0 = tile_n * BN;

  // ---- global -> LDS addressing -------------------------------------------
  // Transfer j of this wave fills tile rows [j*8*NW + wave*8, +8): lane i writes
  // LDS slot (row = i/8, granule slot = i%8) and therefore fetches the global
  // granule (slot ^ ((row >> 1) & 7)) of that row.  Rows past M / N are clamped
  // to the last valid row; their products are never stored.
  const uint8_t* a_base = p.A + (int64_t)row0 * p.lda_bytes;
  const uint8_t* b_base = p.B + (int64_t)col0 * p.ldb_bytes;
  unsigned a_off[LA], b_off[LB];
  int g_lane;  // K granule (0..7) of a row that this lane moves; same for every transfer
  {
    const int lrow = lane >> 3, slot = lane & 7;
    g_lane = slot ^ (((wave * 8 + lrow) >> 1) & 7);
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int r = j * 8 * NW + wave * 8 + lrow;
      const int rr = (row0 + r < p.M) ? r : (p.M - 1 - row0);
      a_off[j] = (unsigned)(rr * (int)p.lda_bytes + g_lane * 16);
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int r = j * 8 * NW + wave * 8 + lrow;
      const int rr = (col0 + r < p.N) ? r : (p.N - 1 - col0);
      b_off[j] = (unsigned)(rr * (int)p.ldb_bytes + g_lane * 16);
    }
  }
  // MX scales: 8 bytes per row and K-step at [row][8], A rows first
  const uint8_t* s_base[LS ? LS : 1];
  unsigned s_off[LS ? LS : 1];
  unsigned s_dst[LS ? LS : 1];
  if constexpr (FP4) {
#pragma unroll
    for (int j = 0; j < LS; ++j) {
      int x = wave + j * NW;
      x = x < NSX ? x : NSX - 1;  // a surplus transfer repeats the last one: the same bytes
      const bool is_a = x < BM / 32;
      const int first = is_a ? row0 : col0, rows = is_a ? p.M : p.N;
      int r = (is_a ? x : x - BM / 32) * 32 + (lane >> 1);
      r = (first + r < rows) ? r : (rows - 1 - first);
      s_base[j] = (is_a ? p.mx_a : p.mx_b) + (int64_t)first * p.mx_ld;
      s_off[j] = (unsigned)(r * p.mx_ld + (lane & 1) * 4);
      s_dst[j] = (unsigned)(SCALES + x * 256);
    }
  }
  auto m0_of = [&](const uint8_t* dst) { return (unsigned)(size_t)AG_LDS(dst); };
  // 64 lanes x 16 bytes from (scalar base + lane offset) to LDS at M0 + lane * 16
  auto g2s = [&](const uint8_t* base, unsigned voff, const uint8_t* dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0_of(dst)), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  auto g2s_lane = [&](const uint8_t* src, const uint8_t* dst) {  // the same from an address per lane
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(m0_of(dst)), "v"(src)
                 : "memory", "m0");
  };
  auto g2s_dword = [&](const uint8_t* base, unsigned voff, const uint8_t* dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(m0_of(dst)), "v"(voff), "s"(base)
                 : "memory", "m0");
  };
  auto issue = [&](int kt, int slot) {
    const uint8_t* ga = a_base + (int64_t)kt * kRowBytes;
    const uint8_t* gb = b_base + (int64_t)kt * kRowBytes;
    const uint8_t* la = lds + slot * STAGE + wave * 8 * kRowBytes;
    const uint8_t* lb = la + BM * kRowBytes;
    if (p.tail_granules != 0 && kt == p.ksteps - 1) {
      // Last K-step of a row that does not fill 128 bytes: granules past the end of
      // the row are fetched from a block of zeros instead, so they add nothing.
      const bool live = g_lane < p.tail_granules;
#pragma unroll
      for (int j = 0; j < LA; ++j) g2s_lane(live ? ga + a_off[j] : g_zero16, la + j * 8 * NW * kRowBytes);
#pragma unroll
      for (int j = 0; j < LB; ++j) g2s_lane(live ? gb + b_off[j] : g_zero16, lb + j * 8 * NW * kRowBytes);
    } else {
#pragma unroll
      for (int j = 0; j < LA; ++j) g2s(ga, a_off[j], la + j * 8 * NW * kRowBytes);
#pragma unroll
      for (int j = 0; j < LB; ++j) g2s(gb, b_off[j], lb + j * 8 * NW * kRowBytes);
    }
    if constexpr (FP4) {
#pragma unroll
      for (int j = 0; j < LS; ++j) g2s_dword(s_base[j] + kt * 8, s_off[j], lds + slot * STAGE + s_dst[j]);
    }
  };

  // ---- what the epilogue needs from memory, requested ahead of everything else ---------------
  const int li = lane & 15, lq = lane >> 4;
  constexpr bool EARLY = TM * TN <= 16;  // the big tiles have no registers to spare for it
  float scale = 1.0f;
  f32x4 bias_v[TN];
  auto load_bias = [&](int n) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (p.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int col = col0 + (wn * TN + n) * 16 + 4 * lq + e;
        v[e] = p.bias[col < p.N ? col : p.N - 1];
      }
    }
    return v;
  };
  if constexpr (EARLY) {
#pragma unroll
    for (int n = 0; n < TN; ++n) bias_v[n] = load_bias(n);
  }
  if (p.scale_a) scale *= *p.scale_a;
  if (p.scale_b) scale *= *p.scale_b;

  // ---- LDS -> fragment addressing ------------------------------------------
  // Lane (li = lane%16, lq = lane/16) owns row li of a 16-row tile and, for
  // k-substep s, granule s*4+lq (16-bit, fp4) or granules 2*lq, 2*lq+1 (fp8).
  unsigned rd_off[KSUB][KGRAN];
#pragma unroll
  for (int s = 0; s < KSUB; ++s)
#pragma unroll
    for (int h = 0; h < KGRAN; ++h) {
      const int g = (KGRAN == 2) ? (2 * lq + h) : (s * 4 + lq);
      rd_off[s][h] = (unsigned)(li * kRowBytes + ((g ^ (li >> 1)) << 4));
    }
  const unsigned a_rd = (unsigned)(wm * TM * 16 * kRowBytes);
  const unsigned b_rd = (unsigned)((BM + wn * TN * 16) * kRowBytes);
  const unsigned sa_rd = (unsigned)(SCALES + (wm * TM * 16 + li) * 8);
  const unsigned sb_rd = (unsigned)(SCALES + (BM + wn * TN * 16 + li) * 8);

  f32x4 acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk = p.ksteps;
#pragma unroll
  for (int k = 0; k < S - 1; ++k)
    if (k < nk) issue(k, k);

  int slot = 0, slot_ld = S - 1;  // stage k is in slot k mod S; the next transfers go to slot_ld
  auto trip = [&](int kt) {
    // behind the barrier: stage kt complete, stage kt - 1 in everybody's registers
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + S - 1 < nk) issue(kt + S - 1, slot_ld);
    const uint8_t* st = lds + slot * STAGE;
    i32x2 sa[FP4 ? TM : 1], sb[FP4 ? TN : 1];
    if constexpr (FP4) {
#pragma unroll
      for (int m = 0; m < TM; ++m) sa[m] = *(const i32x2*)(st + sa_rd + m * 128);
#pragma unroll
      for (int n = 0; n < TN; ++n) sb[n] = *(const i32x2*)(st + sb_rd + n * 128);
    }
    i32x4 af[KSUB][TM][KGRAN], bf[KSUB][TN][KGRAN];
    auto read_frags = [&](int s) {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int h = 0; h < KGRAN; ++h)
          af[s][m][h] = *(const i32x4*)(st + a_rd + m * 16 * kRowBytes + rd_off[s][h]);
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int h = 0; h < KGRAN; ++h)
          bf[s][n][h] = *(const i32x4*)(st + b_rd + n * 16 * kRowBytes + rd_off[s][h]);
    };
#pragma unroll
    for (int s = 0; s < KSUB; ++s) {
      read_frags(s);
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) {
          int xa = 0, xb = 0;
          if constexpr (FP4) {
            xa = (int)((unsigned)(s ? sa[m].y : sa[m].x) >> (8 * lq));
            xb = (int)((unsigned)(s ? sb[n].y : sb[n].x) >> (8 * lq));
          }
          acc[m][n] = mfma_step<DT>(bf[s][n], af[s][m], acc[m][n], xb, xa);
        }
    }
    slot = slot == S - 1 ? 0 : slot + 1;
    slot_ld = slot_ld == S - 1 ? 0 : slot_ld + 1;
  };
  int kt = 0;
  for (; kt + S - 2 < nk; ++kt) {  // S - 2 younger stages have been requested
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((S - 2) * L, 0));
    trip(kt);
  }
  for (; kt < nk; ++kt) {          // the last S - 2: nothing left to request
    const int younger = nk - 1 - kt;
    static_for_stages<0, S - 2>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if (younger == g) __builtin_amdgcn_s_waitcnt(waitcnt_imm(g * L, 0));
    });
    trip(kt);
  }

  // ---- epilogue: scale, bias, cast, vector store ----------------------------
  // row by row: the 16-column pieces of a row leave one behind the other and meet in L2 as whole lines
  // (column by column, 256 x 256 tiles: f16 -> f32 1269x22135x312 60.8 us and, on buffers that no kernel has
  // read yet, 96.8; row by row 38.5 and 53.6; bf16 4096x4097x256 48.2 / 53.9 -> 45.4 / 46.7; 64 x 64 level)
  if constexpr (!EARLY) {
#pragma unroll
    for (int n = 0; n < TN; ++n) bias_v[n] = load_bias(n);
  }
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = row0 + (wm * TM + m) * 16 + li;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int col = col0 + (wn * TN + n) * 16 + 4 * lq;
      if (row < p.M && col < p.N) {
        f32x4 v = acc[m][n] * scale;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bias_v[n][e];
        store4<OUT>(p.C, (int64_t)row * p.ldc + col, v, (p.N - col) < 4 ? (p.N - col) : 4);
      }
    }
  }
}


template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
__global__ __launch_bounds__(WM* WN * 64) void gemm_tile_kernel(const GemmArgs p) {
  gemm_tile_body<DT, OUT, BM, BN, WM, WN, S>(p);
}

// The same with its arguments in one line (gemm_tile.hip says which of the two a launch takes).
template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
__global__ __launch_bounds__(WM* WN * 64) void gemm_tile_packed_kernel(const PackedArgs q) {
  GemmArgs p = unpack_args<DT>(q);
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  p.group_m = tile_order(p.tiles_m, p.tiles_n);
  gemm_tile_body<DT, OUT, BM, BN, WM, WN, S>(p);
}

}  // namespace
}  // namespace astergemm
