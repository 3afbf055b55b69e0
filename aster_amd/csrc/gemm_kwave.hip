// Shapes, rules and launches of the kernels that split K over the waves of a workgroup
// (device code: gemm_kwave_kernel.hpp).  Compiled once per operand type (AG_KWAVE_DT) and order of the weights
// (AG_KWAVE_K8); the unit of f16 operands and row-major weights also holds what all of them share.
#include "gemm_kwave.h"
#include "gemm_kwave_kernel.hpp"

namespace astergemm {

// Tiles, waves (tile rows x tile columns x K) and stages; the second number of stages is MXFP4's, whose
// scale bytes share the ring.  X(index, BM, BN, WM, WN, WK, S, S of MXFP4)
#define AG_KWAVE_SHAPES(X)       \
  X(0, 16, 16, 1, 1, 8, 5, 4)    \
  X(1, 16, 32, 1, 1, 8, 3, 3)    \
  X(2, 16, 48, 1, 1, 4, 5, 4)    \
  X(3, 16, 64, 1, 1, 4, 4, 3)    \
  X(4, 16, 16, 1, 1, 4, 4, 3)    \
  X(5, 32, 16, 2, 1, 4, 6, 6)    \
  X(6, 32, 32, 1, 2, 4, 4, 4)    \
  X(7, 32, 64, 1, 2, 4, 3, 3)    \
  X(8, 32, 128, 2, 2, 2, 4, 3)   \
  X(9, 64, 32, 2, 1, 4, 3, 3)    \
  X(10, 64, 48, 2, 1, 2, 5, 5)   \
  X(11, 64, 64, 2, 2, 2, 3, 3)   \
  X(12, 64, 128, 2, 2, 2, 3, 3)  \
  X(13, 96, 64, 2, 2, 2, 4, 3)   \
  X(14, 128, 64, 2, 2, 2, 3, 3)  \
  X(15, 128, 128, 2, 4, 1, 5, 4)

struct KwaveShape {
  int bm, bn, wm, wn, wk, stages, lds;
  const void* func;
  int (*launch)(const PackedArgs& q, int grid, hipStream_t s);
};
constexpr int kKwaveShapes = 16;
template <int DT, bool K8>
const KwaveShape* kwave_shapes();

namespace {

template <int DT, bool K8, int BM, int BN, int WM, int WN, int WK, int S>
int launch_kwave(const PackedArgs& q, int grid, hipStream_t s) {
  constexpr int lds = S * WK * kwave_step_bytes(DT, K8, BM, BN);
  AG_LAUNCH_KERNEL((gemm_kwave_kernel<DT, K8, BM, BN, WM, WN, WK, S>), dim3(grid), dim3(WM * WN * WK * 64), lds, s,
                   q);
  return (int)hipGetLastError();
}

template <int DT, bool K8, int BM, int BN, int WM, int WN, int WK, int S>
constexpr KwaveShape kwave_shape() {
  return KwaveShape{BM, BN, WM, WN, WK, S, S * WK * kwave_step_bytes(DT, K8, BM, BN),
                    (const void*)gemm_kwave_kernel<DT, K8, BM, BN, WM, WN, WK, S>,
                    launch_kwave<DT, K8, BM, BN, WM, WN, WK, S>};
}

#define AG_KWAVE_ENTRY(I, BM, BN, WM, WN, WK, S, S4) \
  kwave_shape<AG_KWAVE_DT, AG_KWAVE_K8 != 0, BM, BN, WM, WN, WK, AG_KWAVE_DT == ASTERGEMM_MXFP4 ? S4 : S>(),
const KwaveShape kShapes[kKwaveShapes] = {AG_KWAVE_SHAPES(AG_KWAVE_ENTRY)};

}  // namespace

template <>
const KwaveShape* kwave_shapes<AG_KWAVE_DT, AG_KWAVE_K8 != 0>() { return kShapes; }

#if AG_KWAVE_DT == 0 && !AG_KWAVE_K8
template <> const KwaveShape* kwave_shapes<ASTERGEMM_F16, true>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_BF16, false>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_BF16, true>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_FP8_E4M3, false>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_FP8_E4M3, true>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_MXFP4, false>();
template <> const KwaveShape* kwave_shapes<ASTERGEMM_MXFP4, true>();

namespace {

template <bool K8>
const KwaveShape* shapes_of(int dt) {
  switch (dt) {
    case ASTERGEMM_F16: return kwave_shapes<ASTERGEMM_F16, K8>();
    case ASTERGEMM_BF16: return kwave_shapes<ASTERGEMM_BF16, K8>();
    case ASTERGEMM_FP8_E4M3: return kwave_shapes<ASTERGEMM_FP8_E4M3, K8>();
    default: return kwave_shapes<ASTERGEMM_MXFP4, K8>();
  }
}
const KwaveShape* shapes_of(int dt, bool k8) { return k8 ? shapes_of<true>(dt) : shapes_of<false>(dt); }

// Weight rows of a workgroup when `tiles_m` tile rows share the chip: one round, groups of 8 rows.  The tile
// rows of a panel are on one XCD, so a round is what fits every XCD's eighth of the CUs (a few panels more
// put a second round on some XCDs: bf16 400x4096x4096 26.7 -> 41.4 us).
int rows_per(int64_t N, int tiles_m, int cus, int unit = 8) {
  const int per_xcd = cus / 8 / tiles_m, panels = per_xcd > 0 ? per_xcd * 8 : 1;
  return (int)(((N + panels - 1) / panels + unit - 1) / unit * unit);
}

// Workgroups of a K range: by panels on one XCD each, in whole groups of 8 panels, while that is one round;
// else tile after tile.
int kwave_blocks(int tiles_m, int tiles_n, int cus, int* by_panel) {
  const int64_t grouped = (int64_t)tiles_m * ((tiles_n + 7) & ~7);
  *by_panel = grouped <= cus;
  return *by_panel ? (int)grouped : tiles_m * tiles_n;
}

}  // namespace

// Decoding: the tile that brings the fewest operand rows into a CU while one round covers all of N (a
// workgroup's panel is N / CUs rows in groups of 8, not the tile's), within two limits:
//   * panels of more than 64 rows with up to 16 activation rows stay with the resident kernels, whose
//     activations are then read once for many weight rows (bf16 16x28672x4096 37.3 us against 40.2 for
//     16 x 128 tiles, fp8 21.6 / 23.4, MXFP4 11.5 / 13.2); MXFP4 on rows that the resident kernel takes
//     without K ranges already from 32 on (16x14336x4096 7.3 / 7.5), with more than 16 activation rows from
//     40 on: ahead while the weights are found in the last-level cache, behind where they are not
//     (64x14336x4096 11.6 / 9.4 and 11.9 / 14.1, 32x28672x4096 14.3 / 12.3 and 14.6 / 17.6).
//   * a workgroup's own rows over all of K, (bm + per) * rb bytes, come from L2 at about 60 GB/s.  Where K
//     ranges on 64-row panels take half a megabyte off that (two ranges, whose planes weigh more: three
//     quarters), they pay for the planes and the kernel that adds them: bf16 64x4096x14336 37.2 -> 28.4
//     (resident 32.9), 32x4096x11008 22.7 -> 20.2, fp8 64x8192x28672 54.6 -> 48.5 (55.9); behind: fp8
//     64x4096x14336 14.3 / 17.5, bf16 64x8192x8192 29.4 / 30.7.  MXFP4 of more than 48 rows on such
//     rows stays resident (64x8192x28672 39.6 / 42.2).
// Resident kernel / this, us, over rotating weights (three sets):
//   M       bf16 4096x4096  14336x4096   28672x4096   4096x14336   4096x11008   8192x8192    1024x8192
//   8       8.1 / 7.4       19.8 / 18.7  resident     24.4 / 19.8  19.5 / 16.8  28.6 / 21.9  10.0 / 6.9
//   16      8.4 / 7.4       20.1 / 18.9  resident     25.4 / 22.8  20.0 / 18.3  28.7 / 21.9  10.3 / 7.4
//   32      11.6 / 8.0      22.5 / 19.6  40.2 / 36.6  28.0 / 24.0  22.6 / 20.2  30.7 / 22.9  13.7 / 7.6
//   64      15.1 / 8.9      27.7 / 23.4  50.7 / 38.3  32.9 / 28.4  28.7 / 24.2  34.1 / 29.4  13.2 / 8.9
//   fp8 16  6.1 / 5.4       12.3 / 11.1  resident     15.0 / 11.3  28.0 / 10.0  19.4 / 12.1  6.9 / 5.6
//   fp8 64  9.4 / 6.7       17.6 / 12.3  26.9 / 22.2  21.8 / 14.3  28.7 / 12.5  18.2 / 13.2  9.7 / 6.1
//   fp4 16  4.8 / 4.6       resident     resident     10.9 / 7.4   14.6 / 7.4   10.2 / 7.9   5.9 / 4.7
//   fp4 64  6.5 / 5.4       resident     resident     16.9 / 11.0  17.0 / 9.1   14.5 / 10.9  8.6 / 4.8
// (fp8 and MXFP4 4096x11008, no whole 512 bytes: against the tile kernels.)
// The byte limits are what one of 256 CUs reads in the time the other side's extra launch or planes take on this
// chip: another CU count moves `per` with it, the limits were measured at this one only.
KwaveForm kwave_decode_form(int dt, int64_t M, int64_t N, int64_t K, int cus, int max_ranges) {
  KwaveForm f;
  const int64_t rb = row_bytes(dt, K);
  if (cus <= 0 || M < 1 || M > 64 || N < 1 || N > INT32_MAX / 2 || rb % 16 != 0) return f;
  const int t16 = (int)((M + 15) / 16), per = rows_per(N, 1, cus);
  auto take = [&](int shape, int bm, int rows) {
    const int64_t t64 = (N + 63) / 64;
    int r = (int)(cus / t64);
    r = r > 4 ? 4 : r;
    r = r > max_ranges ? max_ranges : r;
    const int64_t own = (bm + rows) * rb, cut = r > 1 ? (bm + 64) * rb / r : own;
    if (M > 16 && own - cut > (r == 2 ? 768 << 10 : 512000)) {
      f.shape = M <= 32 ? 7 : 11;
      f.per = 64;
      f.ranges = r;
    } else if (!(dt == ASTERGEMM_MXFP4 && M > 48 && own > 1300000)) {
      f.shape = shape;
      f.per = rows;
    }
    return f;
  };
  if (const int p16 = rows_per(N, t16, cus); p16 <= 16) return take(0, 16, p16);
  if (M <= 16) {
    const bool resident = dt == ASTERGEMM_MXFP4 && (K == 4096 || K == 8192 || K == 16384);
    if (per > (resident ? 32 : 64)) return f;
    return per <= 32 ? take(1, 16, per) : per <= 48 ? take(2, 16, per) : take(3, 16, per);
  }
  if (per > 128 || (dt == ASTERGEMM_MXFP4 && (K == 4096 || K == 8192) && per > 40)) return f;
  if (M <= 32)
    return per <= 16 ? take(5, 32, per) : per <= 32 ? take(6, 32, per) : per <= 64 ? take(7, 32, per)
                                                                                  : take(8, 32, per);
  if (const int half = rows_per(N, 2, cus); half <= 32) return take(6, 32, half);
  return per <= 32 ? take(9, 64, per) : per <= 48 ? take(10, 64, per) : per <= 64 ? take(11, 64, per)
                                                                                 : take(12, 64, per);
}

// Rows the resident kernels do not take (K a multiple of 32 below 2048, or no whole 512 bytes), one round of
// 16 x 16 tiles: against gemm_skinny_kernel, us: bf16 16x1000x1504 6.0 -> 3.8, 40x300x1984 15.8 -> 4.0,
// 64x1000x992 9.9 -> 3.7, 62x592x352 5.5 -> 3.8 (3.7 is what a launch takes here).
KwaveForm kwave_small_decode_form(int dt, int64_t M, int64_t N, int64_t K, int cus) {
  KwaveForm f;
  if (cus <= 0 || M < 1 || M > 64 || N < 1 || N > INT32_MAX / 2 || row_bytes(dt, K) % 16 != 0) return f;
  const int per = rows_per(N, (int)((M + 15) / 16), cus);
  if (per <= 16) f.shape = 4, f.per = per;
  return f;
}

namespace {

// The tile and panel that bring the fewest operand rows into a CU in one round, among those of a tile's
// exact rows or less; shape -1 where none covers N.
KwaveForm fewest_rows(int64_t M, int64_t N, int cus, int* rows) {
  static const struct { int bm, bn, shape; } kTiles[] = {{32, 16, 5}, {32, 32, 6}, {32, 64, 7}, {64, 32, 9},
                                                         {64, 48, 10}, {64, 64, 11}, {64, 128, 12},
                                                         {96, 64, 13}, {128, 64, 14}, {128, 128, 15}};
  KwaveForm f;
  int bm = 0, best = INT32_MAX;
  for (const auto& t : kTiles) {
    const int64_t tm = (M + t.bm - 1) / t.bm;
    if (tm > cus / 8 || t.bm == bm) continue;  // (the first panel that fits a tile height is its best)
    const int per = rows_per(N, (int)tm, cus);
    if (per > t.bn) continue;
    bm = t.bm;
    // one tile row reads every weight once: worth a sixteenth (bf16 128x14336x4096, 184 rows on 128 x 64 tiles
    // 32.5 us, 176 on 64 x 128 33.9)
    // and a panel of less than three quarters of the tile pays for those
    const int loaded = t.bm + (per * 4 > t.bn * 3 ? per : t.bn * 3 / 4);
    const int cost = loaded - (tm == 1 ? loaded / 16 : 0);
    if (cost < best) best = cost, *rows = t.bm + per, f.shape = t.shape, f.per = per;
  }
  return f;
}

// Whether that is ahead of 128 x 128 tiles past 512 rows, by what either takes, us: one round of small tiles a wave's
// share of the tile's loads and MFMAs over the row, and what all workgroups bring through the L2s; split K a range's
// loads and the fp32 planes, to memory and back, one K loop the loads of a whole row, which few columns have in cache.
// With few columns the planes weigh nothing, and tall tiles, of which 32 rows cover M, leave most CUs without one.
// Fitted to 1342 sizes of 513 ... 4096 rows on 256 CUs, mean errors 5 % and 3 %.  Of the 1149 of them where K is
// split 602 are taken, 16 of those by mistake (behind by 1 ... 5 %, one by 9), and 31 left where this was ahead by
// 3 ... 11 %; by the bytes of the rows alone, 503 of those taken were behind, by up to 111 %.  Tiles of 128 rows are
// left: behind, or ahead by no more than 15 %.
bool ahead_past_512_rows(int dt, int64_t M, int64_t N, int64_t K, const KwaveForm& f) {
  const bool mx = dt == ASTERGEMM_MXFP4;
  const KwaveShape& t = shapes_of(dt, false)[f.shape];
  if (t.bm >= 128) return false;
  const int64_t rb = row_bytes(dt, K), g128 = (M + 127) / 128 * ((N + 127) / 128);
  const int64_t tiles = (M + t.bm - 1) / t.bm * ((N + f.per - 1) / f.per);
  // (the conditions of check_stream_splitk)
  const bool splits = rb % kRowBytes == 0 && rb >= (mx ? 32 : 64) * kRowBytes && (!mx || K % 512 == 0) &&
                      (M % 8 == 0 || g128 >= 8);
  const int S = splits ? stream_split_of(g128, rb / kRowBytes, mx) : 0;
  if (!mx && S == 0) return false;
  const double rows = rb * 1e-6, tile = (double)t.bm * rows, all = (double)tiles * (t.bm + f.per) * rows;
  const double own = mx ? 3.81 + 13.6 * tile + 0.206 * t.bn * tile + 0.0352 * all
                        : 8.45 + 3.3 * tile + 0.118 * t.bn * tile + 0.0211 * all;
  const double planes = (double)S * M * N * 4e-6;
  const double other = S == 0 ? (N <= 128 ? 5100 : 6500) * rows
                     : mx     ? 7.01 + 19.95 * 256 * rows / S + 0.389 * planes
                              : 10.57 + 12.08 * 256 * rows / S + 0.298 * planes;
  return own < 0.95 * other;
}

}  // namespace

// Prompts of a few hundred tokens, 128 x 128 tiles (split K, or one K loop) / this, us:
//   M          bf16 4096x4096  14336x4096   11008x4096   8192x8192    28672x4096
//   80         14.8 / 11.3     41.7 / 28.0  33.9 / 22.6  42.5 / 36.9  57.8 / 49.4
//   128        16.4 / 11.8     44.0 / 32.5  37.2 / 27.0  45.4 / 41.6  59.2 / 53.5
//   256        19.4 / 16.8     46.6 / 45.2  42.0 / 40.6  53.3 / 54.1  80.1 / 87.2
//   512        27.3 / 24.4     72.8 / 81.1  52.0 / 79.0  77.2 / 82.4
//   fp8 128    11.0 / 7.9      -            -            21.7 / 19.5  34.2 / 29.8
//   MXFP4 128  13.8 / 6.8      14.6 / 12.5  14.4 / 11.7  17.1 / 13.5  15.6 / 17.7
//   MXFP4 256  14.1 / 8.3      15.1 / 17.3  14.6 / 16.7  23.2 / 19.8  21.3 / 32.3
// The lines, measured on 256 CUs: operand rows per CU times their bytes, against tiles that read 256 rows or
// split K further
// (bf16 128x4096x14336, 2.8 MB here: 37.4 / 50.0; fp8 200x4096x14336 24.8 / 30.2; MXFP4 333x8192x8192 24.3 / 26.8).
// More than 512 rows, operands of bytes (ahead_past_512_rows):
//   fp8   560x1024x8192 19.6 / 17.1, 900x1024x8192 21.1 / 17.4, 1194x1024x8192 25.6 / 21.5, 1500x1024x8192 26.3 / 22.5,
//         700x2048x8192 25.9 / 21.8; behind: 3000x512x8192 26.6 / 32.2 (nothing below 1024 columns is taken),
//         1100x1024x16384 (2.6 MB) 32.2 / 37.7, 631x1904x9216 23.9 / 27.7, 762x1256x9216 21.9 / 25.0
//   MXFP4 560x1024x8192 16.4 / 12.3, 1194x1024x8192 21.1 / 18.3, 2047x1024x8192 23.2 / 21.5, 600x2048x4096 14.2 / 10.6,
//         1000x1024x4096 14.6 / 9.0, 3000x512x8192 21.9 / 20.3; behind: 800x4096x4096 (216 rows) 14.4 / 17.9,
//         3000x64x14336 14.4 / 29.5, 4096x64x8192 13.7 / 23.6, 2047x256x14336 16.6 / 21.2, 4096x64x4096 11.0 / 14.6
// 16-bit ones are behind from 700 rows on (1194x1024x8192 32.9 / 34.9).
KwaveForm kwave_prompt_form(int dt, int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t rb = row_bytes(dt, K);
  if (cus <= 0 || M <= 64 || N < 1 || N > INT32_MAX / 2 || rb % 16 != 0) return KwaveForm{};
  if (M > 512 && dt != ASTERGEMM_MXFP4 && (dt != ASTERGEMM_FP8_E4M3 || N < 1024)) return KwaveForm{};
  int rows = 0;
  const KwaveForm f = fewest_rows(M, N, cus, &rows);
  if (!f) return f;
  const int64_t own = rows * rb;
  bool pays;
  if (dt == ASTERGEMM_MXFP4) pays = rows <= 192 && own <= 800000;
  else if (dt == ASTERGEMM_FP8_E4M3)
    pays = M <= 128 ? own <= 1400000 : M <= 512 ? rows <= 128 && own <= 900000 : rows <= 160 && own <= 1350000;
  else pays = M <= 128 ? own <= 2200000 : rows <= 192 && own <= 1600000;
  return pays && (M <= 512 || ahead_past_512_rows(dt, M, N, K, f)) ? f : KwaveForm{};
}

// Small products, general 64 x 64 tile kernel / this, us: bf16 300x300x2048 10.0 / 5.4 (32 x 32),
// 500x500x1024 6.7 / 4.6, 207x28x1440 8.0 / 3.9 (16 x 16), 600x600x2056 12.2 / 10.1 (32 x 64), 600x600x4104
// 21.0 / 17.2, 2000x200x1032 7.5 / 7.1; fp8 300x300x4096 11.1 / 6.4, 600x600x4096 11.3 / 9.2.  The 64 x 64 form is
// for configs that name the kernel.
KwaveForm kwave_tile_form(int64_t M, int64_t N, int cus) {
  static const struct { int shape, bm, bn; } kOrder[] = {{0, 16, 16}, {6, 32, 32}, {7, 32, 64}};
  KwaveForm f;
  f.shape = 11;
  f.per = 64;
  for (const auto& t : kOrder)
    if (((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) <= cus) {
      f.shape = t.shape, f.per = t.bn;
      break;
    }
  return f;
}

// Tiles of up to 32 x 64 fit one round.  Up to 32 x 32 whatever the row, 16-bit operands: a launch is most of the
// time, and a K-step per wave group takes less of it than a chain of K-steps in 64 x 64 tiles (general kernel / this,
// captured and replayed, us: f16 256x256x256 3.7 / 2.75, bf16 17x26x40 2.9 / 2.6, 100x100x384 4.1 / 2.7, 512x500x40
// 3.1 / 3.1, 512x500x520 4.9 / 3.7).  32 x 64 from three K-steps on (500x1000x40 3.3 / 3.5, x136 3.8 / 3.5, x384 4.35
// / 3.85, 2000x200x384 4.3 / 3.8), from nine to sixteen of them only with the tile rows of a panel on one XCD
// (256x2000x800 5.9 / 4.9; not 800x600x800 5.96 / 6.14).  fp8 on 32 x 32 from nine K-steps on, 32 x 64 from sixteen
// (600x600x1040 with the quantiser before it 13.1 / 14.3).  Past one round, with 64 x 64 tiles of its own, it is
// behind on short rows (bf16 777x1001x1032 8.0 / 8.8, 1200x640x1024 6.8 / 7.8, fp8 1200x640x2064 8.4 / 9.7, ahead:
// bf16 777x1001x4096 17.5 / 16.3).
bool kwave_small_product(int dt, int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t m32 = (M + 31) / 32, n64 = (N + 63) / 64, rb = row_bytes(dt, K);
  if (dt == ASTERGEMM_MXFP4 || m32 * n64 > cus) return false;
  const bool small = m32 * ((N + 31) / 32) <= cus;
  if (dt == ASTERGEMM_FP8_E4M3) return rb > (small ? 8 * 128 : 2047);
  return small || rb > 2047 || (rb > 2 * 128 && (rb <= 8 * 128 || m32 * ((n64 + 7) & ~7) <= cus));
}

KwaveForm kwave_variant_form(bool split, int dt, int64_t M, int64_t N, int64_t K, int cus) {
  if (!split && kwave_small_product(dt, M, N, K, cus)) return kwave_tile_form(M, N, cus);
  KwaveForm f = kwave_decode_form(dt, M, N, K, cus, 1);
  if (!f) f = kwave_prompt_form(dt, M, N, K, cus);
  return f ? f : kwave_tile_form(M, N, cus);
}

// Pre-shuffled weights (K8): the tile that brings the fewest operand rows into a CU in one round, panels of whole
// 16-row blocks (MXFP4: of pairs of them, whose scale bytes are fetched together).
KwaveForm kwave_k8_form(int dt, int64_t M, int64_t N, int cus, int* rows) {
  static const struct { int bm, bn, shape; } kTiles[] = {
      {16, 16, 0},  {16, 32, 1},  {16, 48, 2},  {16, 64, 3},   {32, 16, 5},  {32, 32, 6},  {32, 64, 7}, {32, 128, 8},
      {64, 32, 9},  {64, 48, 10}, {64, 64, 11}, {64, 128, 12}, {96, 64, 13}, {128, 64, 14}, {128, 128, 15}};
  KwaveForm f;
  if (cus < 8 || M < 1 || M > 512 || N < 16 || N % 16 != 0 || N > INT32_MAX / 2) return f;
  int bm = 0, best = INT32_MAX;
  for (const auto& t : kTiles) {
    const int64_t tm = (M + t.bm - 1) / t.bm;
    if (tm > cus / 8 || t.bm == bm) continue;  // (the first panel that fits a tile height is its best)
    const int per = rows_per(N, (int)tm, cus, dt == ASTERGEMM_MXFP4 && t.bn > 16 ? 32 : 16);
    if (per > t.bn) continue;
    bm = t.bm;
    const int loaded = t.bm + (per * 4 > t.bn * 3 ? per : t.bn * 3 / 4);
    const int cost = loaded - (tm == 1 ? loaded / 16 : 0);
    if (cost < best) best = cost, *rows = t.bm + per, f.shape = t.shape, f.per = per, f.k8 = true;
  }
  return f;
}

int kwave_ready(int dt, bool k8) {
  static std::atomic<uint64_t> all[8], devs[8][kKwaveShapes];
  int dev = 0;
  if (current_device(&dev) != hipSuccess) return (int)hipGetLastError();
  const uint64_t bit = (uint64_t)1 << (dev & 63);
  const int set = (dt & 3) + (k8 ? 4 : 0);
  if (all[set].load(std::memory_order_acquire) & bit) return 0;
  const KwaveShape* shapes = shapes_of(dt, k8);
  for (int i = 0; i < kKwaveShapes; ++i) {
    if (shapes[i].lds <= 65536) continue;  // within the default limit
    if (int e = lds_attr_once(devs[set][i], shapes[i].func, shapes[i].lds)) return e;
  }
  all[set].fetch_or(bit, std::memory_order_release);
  return 0;
}

int kwave_launch(int dt, int out, const GemmArgs& a, const KwaveForm& f, hipStream_t s) {
  const KwaveShape& sh = shapes_of(dt, f.k8)[f.shape];
  const int tiles_m = (a.M + sh.bm - 1) / sh.bm, tiles_n = (a.N + f.per - 1) / f.per;
  KwaveForm32 q;
  q.per = f.per;
  q.ranges = f.ranges;
  q.out = out;
  // Past the last-level cache where that is no use: a matrix of more than 64 MiB is not found there again
  // after a few others; with few activation rows for the panel's the loop is the weight stream and little
  // else, from 30 MiB on.  Through the cache / past it, us, three sets in turn and sets that no kernel has
  // read for 700 MB: bf16 8x4096x11008 16.8 / 16.6 and 19.3 / 17.4, 64x14336x4096 25.9 / 23.3 and 26.5 / 24.2,
  // fp8 16x14336x4096 11.1 / 10.8 and 13.1 / 11.4; the other side: fp8 16x4096x14336 11.3 / 12.8 and 14.5 / 13.3,
  // 64x14336x4096 12.3 / 14.1 and 16.7 / 14.7, 16x1024x8192 5.7 / 6.5 and 5.8 / 6.9.  Not where two tile rows
  // share a panel in L2 (bf16 64x4096x4096 8.9 / 11.8 and 12.5 / 12.2).
  const int64_t mib = (int64_t)a.N * row_bytes(dt, a.K) >> 20;
  q.nt = a.M <= 64 && tiles_m == 1 && (mib > 64 || (mib >= 30 && (a.M <= 8 || (a.M <= 16 && f.per >= 48))));
  q.blocks = kwave_blocks(tiles_m, tiles_n, device_cus(), &q.by_panel);
  const int grid = q.blocks * f.ranges;
  if (f.ranges == 1) return sh.launch(pack_args(a, q.bits(), a.C), grid, s);
  std::unique_lock<std::mutex> order(splitk_order());
  GemmArgs g = a;
  if (!g.workspace)
    if (int rc = splitk_workspace_for((size_t)f.ranges * a.M * a.N * sizeof(float), s, &g.workspace)) return rc;
  if (int e = sh.launch(pack_args(g, q.bits(), g.workspace), grid, s)) return e;
  return splitk_reduce(out, g, f.ranges, s);
}

void kwave_describe(int dt, const KwaveForm& f, int64_t M, int64_t N, int cus, LaunchForm* o) {
  const KwaveShape& sh = shapes_of(dt, f.k8)[f.shape];
  int by_panel;
  o->grid = kwave_blocks((int)((M + sh.bm - 1) / sh.bm), (int)((N + f.per - 1) / f.per), cus, &by_panel) * f.ranges;
  o->tile_m = sh.bm;
  o->tile_n = sh.bn;
  o->waves_m = sh.wm;
  o->waves_n = sh.wn * sh.wk;
  o->stages = sh.stages;
  o->lds_bytes = sh.lds;
  o->threads = sh.wm * sh.wn * sh.wk * 64;
  o->func = sh.func;
}

bool kwave_prompt_describe(const astergemm_config& c, int cus, LaunchForm* o) {
  const KwaveForm f = kwave_prompt_form(c.dtype_ab, c.M, c.N, c.K, cus);
  if (f) kwave_describe(c.dtype_ab, f, c.M, c.N, cus, o);
  return (bool)f;
}
bool kwave_decode_describe(const astergemm_config& c, int cus, int max_ranges, LaunchForm* o) {
  const KwaveForm f = kwave_decode_form(c.dtype_ab, c.M, c.N, c.K, cus, max_ranges);
  if (f) kwave_describe(c.dtype_ab, f, c.M, c.N, cus, o);
  return (bool)f;
}
bool kwave_small_decode_describe(const astergemm_config& c, int cus, LaunchForm* o) {
  const KwaveForm f = kwave_small_decode_form(c.dtype_ab, c.M, c.N, c.K, cus);
  if (f) kwave_describe(c.dtype_ab, f, c.M, c.N, cus, o);
  return (bool)f;
}
#endif  // AG_KWAVE_DT == 0 && !AG_KWAVE_K8

}  // namespace astergemm
