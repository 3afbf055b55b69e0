// Stream kernels (whole-ring, hand-scheduled MFMA loops) for f16 / bf16, fp8 and MXFP4:
// launchers, shape checks and the variant table.  Kept apart from gemm_tile.hip so that the
// two halves of the kernel set compile side by side.
#include <mutex>
#include <vector>

#include "gemm_kwave.h"
#include "gemm_stream_kernel.hpp"
#include "gemm_streamr_kernel.hpp"
#include "gemm_stream8_kernel.hpp"
#include "gemm_stream4_kernel.hpp"
#include "gemm_streamdb_kernel.hpp"
#include "gemm_stream4db_kernel.hpp"
#include "gemm_stream4dbl_kernel.hpp"
#include "gemm_stream8db_kernel.hpp"
#include "gemm_directab_kernel.hpp"

namespace astergemm {
namespace {

// Prompts of few tokens: the kernels that split K over the waves stand in for the 128 x 128 tiles in AUTO's form
// of their variants (kwave_prompt_form).  Either's first launch readies both, so that a config that
// is captured later finds its kernel ready; inside a capture only the one that runs has to be.
inline KwaveForm kwave_instead(int dt, const GemmArgs& a) {
  return a.own_kernel ? KwaveForm{} : kwave_prompt_form(dt, a.M, a.N, a.K, device_cus());
}
// 0 and *taken = false: the launcher's own kernel is to run
inline int kwave_prompt(int dt, int out, const GemmArgs& a, int own_ready, hipStream_t s, bool* taken) {
  const KwaveForm f = kwave_instead(dt, a);
  *taken = (bool)f;
  if (own_ready != 0 && !f) return own_ready;
  const int e = kwave_ready(dt);
  if (!f) return 0;
  return e != 0 ? e : kwave_launch(dt, out, a, f, s);
}

// Whole 128 x 128 tiles, two to a CU, in AUTO's form of the variant: each two as one of 256 x 128, whose
// 384 operand rows replace their 512 and whose ring runs two K-steps ahead for the CU's eight waves together.
// From 7/8 of the chip's CUs on in pairs: below, unequal_tile_of has taken the 256 x 128 kernel already.  One
// round only: past it a second round of pairs is as long as the first.  128 x 128 / pairs, us (rows of 4096 / 11008 /
// 1024 elements): bf16 2048x4096 57.9 / 52.8, 180 / 159, 18.4 / 18.0; 512x14336 73.1 / 57.5, 184 / 157, 16.9 / 15.8;
// 1024x8192 57.3 / 52.1, 185 / 155, 18.0 / 17.4; with a K tail 2048x4096x4104 79.0 / 67.0.  fp32 outputs on rows
// of 2 KiB are behind (f16 2048x4096x1024 21.2 / 21.9).  K loops from step 0 in both for these figures; as AUTO
// runs them they start by XCD, and odd tile rows swap the steps of a pair (step_order).
inline bool pairs_tiles(int out, int64_t M, int64_t N, int64_t row_bytes, int cus) {
  const int64_t g128 = M / 128 * (N / 128);
  return M % 128 == 0 && N % 128 == 0 && row_bytes >= (out == ASTERGEMM_F32 ? 18 * 128 : 2048) &&
         g128 * 8 >= (int64_t)2 * cus * 7 && (M + 255) / 256 * (N / 128) <= cus;
}

template <int DT, int OUT>
int launch_pairs(GemmArgs a, hipStream_t s) {
  a.tiles_m = (a.M + 255) / 256;
  a.group_m = tile_order(a.tiles_m, a.tiles_n);
  auto k = gemm_streamr_kernel<DT, OUT, 256, 128, 4, 2, 3>;
  AG_LAUNCH_KERNEL(k, dim3(a.tiles_m * a.tiles_n), dim3(512), 3 * 384 * kRowBytes, s, a);
  return (int)hipGetLastError();
}

template <int DT, int OUT>
bool pairs_describe(const astergemm_config& c, int cus, LaunchForm* o) {
  if (kwave_prompt_describe(c, cus, o)) return true;
  if (cus <= 0 || !pairs_tiles(OUT, c.M, c.N, row_bytes(DT, c.K), cus)) return false;
  o->grid = (int)((c.M + 255) / 256 * (c.N / 128));
  o->tile_m = 256;
  o->tile_n = 128;
  o->waves_m = 4;
  o->waves_n = 2;
  o->stages = 3;
  o->lds_bytes = 3 * 384 * kRowBytes;
  o->threads = 512;
  o->func = (const void*)gemm_streamr_kernel<DT, OUT, 256, 128, 4, 2, 3>;
  return true;
}

template <int DT, int OUT, int BM, int BN, int WM, int WN, int NSLOT = 5>
int launch_stream(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = NSLOT * BM * kRowBytes;
  auto k = gemm_stream_kernel<DT, OUT, BM, BN, WM, WN, NSLOT>;
  static std::atomic<uint64_t> attr_devs{0};
  if constexpr (BM == 128 && NSLOT == 5) {
    static std::atomic<uint64_t> pair_devs{0};
    const bool pairs = !a.own_kernel && pairs_tiles(OUT, a.M, a.N, row_bytes(DT, a.K), device_cus());
    const int pair_ready = lds_attr_once(
        pair_devs, (const void*)gemm_streamr_kernel<DT, OUT, 256, 128, 4, 2, 3>, 3 * 384 * kRowBytes);
    const int own_ready = lds_attr_once(attr_devs, (const void*)k, lds);
    bool taken = false;
    if (const int e = kwave_prompt(DT, OUT, a, pairs ? pair_ready : own_ready, s, &taken); e || taken) return e;
    if (pairs) return launch_pairs<DT, OUT>(a, s);
    AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), lds, s, a);
    return (int)hipGetLastError();
  }
  if constexpr (BM == 128) {
    bool taken = false;
    if (const int e = kwave_prompt(DT, OUT, a, lds_attr_once(attr_devs, (const void*)k, lds), s, &taken); e || taken)
      return e;
  } else if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) {
    return e;
  }
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_stream(const astergemm_config& c) {
  // Edge tiles move in units of 8 operand rows and 16-byte output chunks; a unit of A across the
  // last row is shifted up (edge_row), so M is free from one whole unit on.  The general tile
  // kernels against these, M not a multiple of 8, back to back: bf16 333x14336x4096 71.0 -> 62.8 us,
  // 500x4096x14336 158 -> 79, 1537x8192x8192 211 -> 173, 130x4096x4096 47 -> 21; fp8 500x4096x14336
  // 80.6 -> 53.9, 1537x8192x8192 110 -> 87; MXFP4 333x14336x4096 48.0 -> 25.7, 1537x8192x8192 135 -> 62.
  if (c.M < 8 || c.N < 8 || c.N % 8 != 0) return "M must be at least 8 and N a multiple of 8";
  // a K tail of 1..7 granules is multiplied after the loop; at least one whole step is needed
  if (row_bytes(c.dtype_ab, c.K) % 16 != 0) return "K must cover a whole number of 16-byte granules";
  if (row_bytes(c.dtype_ab, c.K) < kRowBytes) return "K must cover at least one 128-byte row chunk";
  if (c.ldc % 8 != 0) return "ldc must be a multiple of 8 elements";
  return nullptr;
}

const char* check_stream_whole_k(const astergemm_config& c) {
  if (const char* why = check_stream(c)) return why;
  if (row_bytes(c.dtype_ab, c.K) % kRowBytes != 0) return "K must fill whole 128-byte row chunks";
  return nullptr;
}

#define AG_STREAM(name, DT, OUT, BM, BN, WM, WN)                                 \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, BM, BN, kRowBytes, WM, WN, 3,          \
        (WM * WN == 8 || BM == 128) ? 2 : 0, 5 * BM * kRowBytes,                \
        (const void*)gemm_stream_kernel<DT, OUT, BM, BN, WM, WN>,                \
        launch_stream<DT, OUT, BM, BN, WM, WN>,                                  \
        (WM * WN == 8 || BM == 128) ? check_stream : check_stream_whole_k,       \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0,                              \
        BM == 128 ? pairs_describe<DT, OUT> : nullptr, BM == 128                 \
  }

// The 128 x 128 kernel with a ring of nine slots (144 KiB of LDS, one workgroup per CU): four
// K-steps requested ahead instead of two.  For grids of at most one workgroup per CU with two or
// more tile rows, where nothing else covers a workgroup's waits (bf16, five -> nine slots:
// 256 x 14336 x 4096 37.7-38.7 -> 33.7-34.4 us, 384 x 8192 x 4096 34.4 -> 31.0, 2048^3 23.3 ->
// 21.2, 1024 x 4096 x 4096 36.9 -> 35.5; one tile row, which is HBM-bound on B alone, loses:
// 128 x 28672 x 4096 39.8 -> 41.8; eight waves instead of four: level).  With K loops that start at different
// steps on different XCDs: 200 x 14336 x 4096 41.4 -> 39.2, 333 x 8192 x 8192 68.4 -> 64.4.
const char* check_stream_ring9(const astergemm_config& c) {
  if (const char* why = check_stream(c)) return why;
  int cus = device_cus();
  if (cus <= 0) cus = 256;  // no device to ask: describe the MI355X
  const int64_t tm = (c.M + 127) / 128, tn = (c.N + 127) / 128;
  if (tm < 2) return "the nine-slot ring pays from two tile rows on";
  if (tm * tn > cus) return "the nine-slot ring takes the LDS of a CU: at most one workgroup per CU";
  if (row_bytes(c.dtype_ab, c.K) < 16 * kRowBytes) return "the nine-slot ring needs 16 K-steps or more";
  return nullptr;
}
#define AG_STREAM_RING9(name, DT, OUT)                                           \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 128, kRowBytes, 2, 2, 5, 3,       \
        9 * 128 * kRowBytes,                                                     \
        (const void*)gemm_stream_kernel<DT, OUT, 128, 128, 2, 2, 9>,             \
        launch_stream<DT, OUT, 128, 128, 2, 2, 9>, check_stream_ring9,           \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0, kwave_prompt_describe, true  \
  }
#define AG_STREAM_RING9_SET(prefix, DT)                                          \
  AG_STREAM_RING9(prefix "_128x128_w2x2_ring9_bf16", DT, ASTERGEMM_BF16),        \
      AG_STREAM_RING9(prefix "_128x128_w2x2_ring9_f32", DT, ASTERGEMM_F32),      \
      AG_STREAM_RING9(prefix "_128x128_w2x2_ring9_f16", DT, ASTERGEMM_F16)

// ---- unequal tile sides (gemm_streamr_kernel.hpp); rank 5: AUTO takes them by unequal_tile_of ----
template <int DT, int OUT, int BM, int BN, int WM, int WN, int NS>
int launch_streamr(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = NS * (BM + BN) * kRowBytes;
  auto k = gemm_streamr_kernel<DT, OUT, BM, BN, WM, WN, NS>;
  static std::atomic<uint64_t> attr_devs{0};
  if constexpr (BM == 128) {
    bool taken = false;
    if (const int e = kwave_prompt(DT, OUT, a, lds_attr_once(attr_devs, (const void*)k, lds), s, &taken); e || taken)
      return e;
  } else if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) {
    return e;
  }
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), lds, s, a);
  return (int)hipGetLastError();
}

#define AG_STREAMR(name, DT, OUT, BM, BN, WM, WN, NS)                      \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, BM, BN, kRowBytes, WM, WN, NS, 5,      \
        NS * (BM + BN) * kRowBytes,                                              \
        (const void*)gemm_streamr_kernel<DT, OUT, BM, BN, WM, WN, NS>,           \
        launch_streamr<DT, OUT, BM, BN, WM, WN, NS>, check_stream,               \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0,                              \
        BM == 128 ? kwave_prompt_describe : nullptr, true                        \
  }
#define AG_STREAMR_SET(prefix, DT, BM, BN, WM, WN, NS)                     \
  AG_STREAMR(prefix "_bf16", DT, ASTERGEMM_BF16, BM, BN, WM, WN, NS),      \
      AG_STREAMR(prefix "_f32", DT, ASTERGEMM_F32, BM, BN, WM, WN, NS),    \
      AG_STREAMR(prefix "_f16", DT, ASTERGEMM_F16, BM, BN, WM, WN, NS)

// ---- pre-shuffled weights (K8 order) in AUTO's form of the kernels below -----------------------
//
// The kernels that load them straight into MFMA operands have 128 x 256 tiles and nothing for problems that those leave
// half the chip without: through LDS they are as good an operand as rows (16 rows x 128 bytes are 2 KiB in one
// piece), for K over waves (gemm_kwave_kernel), tiles of 128, 192 or 256 x 128 (gemm_streamr_kernel) and of 256 x 256
// (gemm_stream_kernel).  A workgroup takes as long as its operand rows, per K-step; straight into operands 384 rows
// weigh as much as 500 here (390 in fp8; past one per CU two share it).  Own kernel / K over waves / 128 / 192 /
// 256 x 128, us over three sets of weights (fp8 and MXFP4 with their quantiser):
//   bf16 80x4096x4096       43.0 / 11.9 / 22.0 / 27.9 / 35.2    bf16 512x1024x8192   77.8 / 22.1 / 41.7 / 53.2 / 67.7
//   bf16 160x14336x4096     60.3 / 49.3 / 38.9 / 44.0 / 44.4    bf16 320x4096x14336  181 / 85.5 / 101 / 128 / 123
//   bf16 320x14336x4096     63.8 / - / 63.9 / 44.6 / 49.0       bf16 512x14336x4096  68.5 / - / 72.5 / 79.4 / 53.8
//   bf16 640x11008x4096     63.2 / - / 68.6 / 71.8 / 82.7       bf16 1280x8192x8192  199 / - / 188 / 156 / 184
//   bf16 640x28672x4096     165 / - / 178 / 158 / 145           bf16 4096x4096x4096  108 / - / - / 123 / 109
//   fp8 80x14336x4096       29.3 / 20.8 / 22.6 / 23.8 / 27.6    fp8 320x28672x4096   66.2 / - / 67.9 / 55.1 / 62.3
//   fp8 1280x4096x14336     96.3 / - / 117 / 87.6 / 96.3        fp8 944x14336x4096   60.0 / - / - / 71.9 / 63.2
//   MXFP4 160x4096x14336    45.4 / 28.4                         MXFP4 160x14336x4096 21.5 / 23.2 (240 rows)
// A second round on short rows, and a third one, are not what the count of rows says; own / these:
//   two rounds: fp8 from 2048 columns of K on (320x22016x256 11.6 / 13.4, 3776x3200x512 18.9 / 20.7, 1792x5632x1024
//     22.5 / 23.8, 1912x6464x1536 27.8 / 28.6, 1512x7744x2048 32.3 / 32.1, 3016x4096x4096 59.6 / 56.9), 16-bit from
//     192 on (bf16 584x15936x64 6.85 / 7.53; the tests hold a size of 192, up to 256 it is still behind,
//     664x15616x256 11.1 / 11.9); 256 x 128 up to 2048 rows from 8192 on (bf16 1568x9344x8192 207 / 200, f16
//     1304x10880x14336 376 / 359; f16 1360x10816x2048 52.5 / 54.7, bf16 4944x3200x5120 118 / 121, f16 3128x4992x14336
//     357 / 364)
//   one round of 256 x 128, fp8: up to 768 rows (496x14336x8192 70.5 / 62.6, 640x10240x8192 65.6 / 59.5;
//     896x8192x8192 58.0 / 61.8, 800x8192x4096 34.0 / 35.3), past them only where the own kernel's tiles are a whole
//     round, one of which the tests hold: level to 4 % behind (960x8192x4096 35.8 / 36.3, 1936x4096x14336 111 / 116)
//   128 x 128 (up to 128 rows, more than 65536 columns) from 1024 columns of K on: bf16 128x73728x4096 156 / 129,
//     128x66048x1024 45.2 / 38.9, 128x73728x512 20.6 / 22.8
//   192 x 128 where the own kernel needs one too (more than two per CU): bf16 1472x11008x4096 135 / 124,
//     4512x4096x4096 132 / 122, 2184x8192x8192 274 / 246, 560x28672x4096 160 / 137; not 1392x11008x4096 (473 of its
//     tiles) 111 / 117, 1648x9920x4096 110 / 121, 4984x3328x1024 30.8 / 37.1
//   256 x 128, which reads weights less often: past 132 MiB of them on up to 2048 rows and a third of the third
//     round, 720x28672x4096 166 / 153, 1224x17024x4096 160 / 151, 976x20672x14336 (f16) 572 / 528; not
//     1664x13120x3584 129 / 139, 1288x14336x4096 (f16) 149 / 154, 5264x4096x4096 139 / 144, 2552x7360x8192 268 / 279,
//     656x28224x1024 40.5 / 42.7, 2552x8192x28672 (f16) 1077 / 1100, 1264x14208x7680 (f16, 555 tiles) 258 / 277
// and, in 16-bit, the 256 x 256 tiles of the row-major kernel: a round of them weighs as 580 rows, more by what M is
// padded with, and two rounds and more pay where seven eighths of the workgroups' places in them are filled (0.85 of
// 6, 5496x14912x1024 134 / 152, 0.86 of 3, f16 1304x28032x1024 69.3 / 76.7, 0.84 of 2, f16 880x27648x3072 130 / 139),
// two from 2048 columns on (1920x14336x1024 takes 57.9 / 58.9, 8192x4096x512 40.1 / 40.8), more than three from 1536
// on (4928x23872x64 50.6 / 53.9, 5464x23872x256 85.8 / 92.3, f16 5656x27328x1024 264 / 275, bf16 3584x18560x1536 156
// / 150; three as well, but the tests hold one of 64 columns: 1520x32512x64 24.5 / 25.5).  Own / what this rule took
// without them / these:
//   bf16 944x14336x4096     108.9 / 97.8 / 86.9                 bf16 640x14336x4096  91.5 / 77.9 / 79.0 (M padded by 1.2)
//   bf16 1280x8192x28672    735 / 565 / 489                     bf16 640x11008x4096  61.9 / 61.1 / 67.5
//   bf16 8192x4096x14336    721 / 720 / 624 (2 rounds, full)    bf16 1920x11008x4096 149 / 147 / 156 (0.67 of 2)
//   bf16 4096x14336x4096    363 / 362 / 342 (0.88 of 4)         bf16 2560x14336x4096 241 / 236 / 244 (0.73 of 3)
// fp8 in this order adds from K-step 0 on, so the tiles have the bits of the own kernel, and K over waves, which does
// not, is for weights of 1024 rows and more, as among row-major ones (MXFP4 too).
struct K8Form {
  KwaveForm kw;
  int tile = 0;         // rows of a tile 128 columns wide
  bool square = false;  // 256 x 256 tiles (16-bit); none of them: the launcher's own kernel
  explicit operator bool() const { return kw || tile || square; }
};
inline K8Form k8_form(int dt, int64_t M, int64_t N, int64_t K, int cus) {
  K8Form f;
  if (cus <= 0 || M < 1 || N < 1) return f;  // (an id is described whether or not its kernel takes the sizes)
  const bool fp8 = dt == ASTERGEMM_FP8_E4M3, fp4 = dt == ASTERGEMM_MXFP4;
  int64_t best = INT64_MAX;
  if (!fp4) {
    const int64_t own_grid = (M + 127) / 128 * ((N + 255) / 256);
    if (fp8 && own_grid > 2 * cus) return f;
    const int64_t squares = (M + 255) / 256 * ((N + 255) / 256), sq_rounds = (squares + cus - 1) / cus;
    const int64_t sq_from = sq_rounds == 2 ? 2048 : sq_rounds == 3 ? 64 : 1536;
    if (!fp8 && sq_rounds > 1 && squares * 8 >= sq_rounds * cus * 7 && K >= sq_from) {
      f.square = true;
      return f;
    }
    if (own_grid > 700 * cus / 256) return f;
    best = own_grid <= cus ? (fp8 ? 390 : 500) : fp8 ? 700 : own_grid <= 2 * cus ? 1000 : 1200;
    const bool second[] = {K >= (fp8 ? 2048 : 192), K >= (fp8 ? 2048 : 192), M <= 2048 && K >= 8192};
    const bool third[] = {K >= 1024, own_grid > 2 * cus, M <= 2048 && N * K > (int64_t)66 << 20};
    for (int bm : {128, 192, 256}) {
      const int64_t tiles = (M + bm - 1) / bm * ((N + 127) / 128), rounds = (tiles + cus - 1) / cus;
      if (bm == 256 && (rounds == 3 ? tiles * 3 < 7 * cus : fp8 && M > 768 && own_grid < cus)) break;
      const bool pays = rounds == 1 || (rounds == 2 && second[bm / 64 - 2]) || (rounds == 3 && third[bm / 64 - 2]);
      if (pays && rounds * (bm + 128) < best) best = rounds * (bm + 128), f.tile = bm;
    }
    const int64_t sq = 580 * ((M + 255) / 256 * 256) / M;
    if (!fp8 && sq_rounds == 1 && sq < best) best = sq, f.tile = 0, f.square = true;
  }
  int rows = 0;
  if ((fp8 || fp4) && N < 1024) return f;
  const KwaveForm kw = kwave_k8_form(dt, M, N, cus, &rows);
  if (kw && (fp4 ? rows <= 192 : fp8 ? rows * 4 < best * 3 : rows * 4 <= best * 3)) {
    f.kw = kw;
    f.tile = 0, f.square = false;
  }
  return f;
}

constexpr int k8_stages(int bm) { return bm == 128 ? 5 : bm == 192 ? 4 : 3; }
constexpr int k8_lds(int bm) { return k8_stages(bm) * (bm + 128) * kRowBytes; }
template <int DT, int OUT, int BM>
constexpr auto k8_kernel() {
  return gemm_streamr_kernel<DT, OUT, BM, 128, 4, 2, k8_stages(BM), true>;
}
template <int DT, int OUT, int BM>
int launch_k8_tile(GemmArgs a, hipStream_t s) {
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + 127) / 128;
  a.group_m = tile_order(a.tiles_m, a.tiles_n);
  auto k = k8_kernel<DT, OUT, BM>();
  AG_LAUNCH_KERNEL(k, dim3(a.tiles_m * a.tiles_n), dim3(512), k8_lds(BM), s, a);
  return (int)hipGetLastError();
}

template <int DT, int OUT>
constexpr auto k8_square() {
  return gemm_stream_kernel<DT, OUT, 256, 256, 2, 4, 5, true>;
}
constexpr int k8_square_lds = 5 * 256 * kRowBytes;
template <int DT, int OUT>
int launch_k8_square(GemmArgs a, hipStream_t s) {
  a.tiles_m = (a.M + 255) / 256;
  a.tiles_n = (a.N + 255) / 256;
  a.group_m = tile_order(a.tiles_m, a.tiles_n);
  auto k = k8_square<DT, OUT>();
  AG_LAUNCH_KERNEL(k, dim3(a.tiles_m * a.tiles_n), dim3(512), k8_square_lds, s, a);
  return (int)hipGetLastError();
}

// 0 and *taken = false: the launcher's own kernel is to run.  Either's first launch readies all of them.
template <int DT, int OUT>
int k8_instead(const GemmArgs& a, int own_ready, hipStream_t s, bool* taken) {
  *taken = false;
  const K8Form f = a.own_kernel ? K8Form{} : k8_form(DT, a.M, a.N, a.K, device_cus());
  if (own_ready != 0 && !f) return own_ready;
  if (const int e = kwave_ready(DT, true)) return e;
  if constexpr (DT != ASTERGEMM_MXFP4) {
    static std::atomic<uint64_t> devs[3];
    if (const int e = lds_attr_once(devs[0], (const void*)k8_kernel<DT, OUT, 128>(), k8_lds(128))) return e;
    if (const int e = lds_attr_once(devs[1], (const void*)k8_kernel<DT, OUT, 192>(), k8_lds(192))) return e;
    if (const int e = lds_attr_once(devs[2], (const void*)k8_kernel<DT, OUT, 256>(), k8_lds(256))) return e;
  }
  constexpr bool SQUARE = DT == ASTERGEMM_BF16 || DT == ASTERGEMM_F16;
  if constexpr (SQUARE) {
    static std::atomic<uint64_t> devs{0};
    if (const int e = lds_attr_once(devs, (const void*)k8_square<DT, OUT>(), k8_square_lds)) return e;
  }
  if (!f) return 0;
  *taken = true;
  if (f.kw) return kwave_launch(DT, OUT, a, f.kw, s);
  if constexpr (SQUARE) {
    if (f.square) return launch_k8_square<DT, OUT>(a, s);
  }
  if constexpr (DT != ASTERGEMM_MXFP4) {
    if (f.tile == 128) return launch_k8_tile<DT, OUT, 128>(a, s);
    if (f.tile == 192) return launch_k8_tile<DT, OUT, 192>(a, s);
    return launch_k8_tile<DT, OUT, 256>(a, s);
  }
  return 0;
}

template <int DT, int OUT>
bool k8_describe(const astergemm_config& c, int cus, LaunchForm* o) {
  const K8Form f = cus > 0 ? k8_form(DT, c.M, c.N, c.K, cus) : K8Form{};
  if (f.kw) kwave_describe(DT, f.kw, c.M, c.N, cus, o);
  if constexpr (DT == ASTERGEMM_BF16 || DT == ASTERGEMM_F16) {
    if (f.square) {
      o->grid = (int)((c.M + 255) / 256 * ((c.N + 255) / 256));
      o->tile_m = o->tile_n = 256;
      o->waves_m = 2;
      o->waves_n = 4;
      o->stages = 3;
      o->lds_bytes = k8_square_lds;
      o->threads = 512;
      o->func = (const void*)k8_square<DT, OUT>();
    }
  }
  if constexpr (DT != ASTERGEMM_MXFP4) {
    if (f.tile) {
      o->grid = (int)((c.M + f.tile - 1) / f.tile * ((c.N + 127) / 128));
      o->tile_m = f.tile;
      o->tile_n = 128;
      o->waves_m = 4;
      o->waves_n = 2;
      o->stages = k8_stages(f.tile);
      o->lds_bytes = k8_lds(f.tile);
      o->threads = 512;
      o->func = f.tile == 128   ? (const void*)k8_kernel<DT, OUT, 128>()
                : f.tile == 192 ? (const void*)k8_kernel<DT, OUT, 192>()
                                : (const void*)k8_kernel<DT, OUT, 256>();
    }
  }
  return (bool)f;
}

// ---- B pre-shuffled, loaded straight into MFMA operands (gemm_streamdb_kernel.hpp) ---------
template <int DT, int OUT, int NSLOT, int NBUF, int WM>
int launch_streamdb(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = 5 * 128 * WM * kRowBytes;  // the epilogue stages through the ring
  auto k = gemm_streamdb_kernel<DT, OUT, NSLOT, NBUF, WM>;
  static std::atomic<uint64_t> attr_devs{0};
  // what the kernels' indexing assumes: whole 16-row blocks of B and whole K-steps
  if (a.N % 16 != 0 || a.N < 16 || a.M < 8 || a.M % 8 != 0 || a.K % 64 != 0 || a.tail_granules != 0 ||
      a.ldb_bytes != (int64_t)a.K * 2)
    return (int)hipErrorInvalidValue;
  const int own_ready = lds_attr_once(attr_devs, (const void*)k, lds);
  if constexpr (WM == 1) {
    bool taken = false;
    if (const int e = k8_instead<DT, OUT>(a, own_ready, s, &taken); e || taken) return e;
  }
  if (own_ready != 0) return own_ready;
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * 256), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_streamdb(const astergemm_config& c) {
  if (c.M % 8 != 0 || c.M < 8) return "M must be a multiple of 8";
  if (c.N % 16 != 0 || c.N < 16) return "pre-shuffled B needs N % 16 == 0";
  if (c.K % 64 != 0) return "pre-shuffled B in K8 order needs K % 64 == 0";
  if (c.ldb != 0 && c.ldb != c.K) return "pre-shuffled B is packed (ldb = K)";
  if (c.ldc % 8 != 0) return "ldc must be a multiple of 8 elements";
  if (c.N * c.K * 2 >= ((int64_t)1 << 32)) return "pre-shuffled B must stay below 4 GiB";
  return nullptr;
}

#define AG_STREAMDB(name, DT, OUT, NSLOT, NBUF, WM, RANK)                        \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128 * WM, 256, kRowBytes, WM, 4, NSLOT, RANK, \
        5 * 128 * WM * kRowBytes,                                                \
        (const void*)gemm_streamdb_kernel<DT, OUT, NSLOT, NBUF, WM>,             \
        launch_streamdb<DT, OUT, NSLOT, NBUF, WM>, check_streamdb,               \
        ASTERGEMM_OPERAND_DIRECT_B_K8, nullptr, nullptr, 0,                      \
        WM == 1 ? k8_describe<DT, OUT> : nullptr, WM == 1                        \
  }

// ---- A and B pre-shuffled, both loaded straight into MFMA operands, no LDS
// (gemm_directab_kernel.hpp) --------------------------------------------------------------------
template <int DT, int OUT, int TM, int TN, int WM, int WN, int NB>
int launch_directab(const GemmArgs& a, int grid, hipStream_t s) {
  auto k = gemm_directab_kernel<DT, OUT, TM, TN, WM, WN, NB>;
  // what the kernel's indexing assumes: whole 16-row blocks of both operands, whole 32-element
  // chunk columns, both operands packed
  if (a.M % 16 != 0 || a.M < 16 || a.N % 16 != 0 || a.N < 16 || a.K % 32 != 0 || a.K < 32 ||
      a.lda_bytes != (int64_t)a.K * 2 || a.ldb_bytes != (int64_t)a.K * 2)
    return (int)hipErrorInvalidValue;
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), 0, s, a);
  return (int)hipGetLastError();
}

const char* check_directab(const astergemm_config& c) {
  if (c.M % 16 != 0 || c.M < 16) return "pre-shuffled A needs M % 16 == 0";
  if (c.N % 16 != 0 || c.N < 16) return "pre-shuffled B needs N % 16 == 0";
  if (c.K % 32 != 0) return "pre-shuffled operands need K % 32 == 0";
  if (c.lda != 0 && c.lda != c.K) return "pre-shuffled A is packed (lda = K)";
  if (c.ldb != 0 && c.ldb != c.K) return "pre-shuffled B is packed (ldb = K)";
  if (c.ldc % 4 != 0) return "ldc must be a multiple of 4 elements";
  if (c.M * c.K * 2 >= ((int64_t)1 << 32) || c.N * c.K * 2 >= ((int64_t)1 << 32))
    return "pre-shuffled operands must stay below 4 GiB each";
  return nullptr;
}

#define AG_DIRECTAB(name, DT, OUT, TM, TN, WM, WN, NB, RANK)                     \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, TM * 16 * WM, TN * 16 * WN, 64, WM, WN, NB, RANK, 0, \
        (const void*)gemm_directab_kernel<DT, OUT, TM, TN, WM, WN, NB>,          \
        launch_directab<DT, OUT, TM, TN, WM, WN, NB>, check_directab,            \
        ASTERGEMM_OPERAND_DIRECT_AB                                              \
  }
#define AG_DIRECTAB_SET(prefix, DT)                                                        \
  AG_DIRECTAB(prefix "_128x256_w1x4_bf16", DT, ASTERGEMM_BF16, 8, 4, 1, 4, 4, 1),          \
      AG_DIRECTAB(prefix "_128x256_w1x4_f32", DT, ASTERGEMM_F32, 8, 4, 1, 4, 4, 1),        \
      AG_DIRECTAB(prefix "_128x256_w1x4_f16", DT, ASTERGEMM_F16, 8, 4, 1, 4, 4, 1),        \
      AG_DIRECTAB(prefix "_256x256_w2x2_bf16", DT, ASTERGEMM_BF16, 8, 8, 2, 2, 3, 2),      \
      AG_DIRECTAB(prefix "_256x256_w2x2_f32", DT, ASTERGEMM_F32, 8, 8, 2, 2, 3, 2),        \
      AG_DIRECTAB(prefix "_256x256_w2x2_f16", DT, ASTERGEMM_F16, 8, 8, 2, 2, 3, 2)

// ---- MXFP4, B pre-shuffled (payload in step order, scale plane in lane order) and loaded
// straight into MFMA operands: 128 x 256 tiles, four waves (gemm_stream4db_kernel.hpp) ---------
template <int DT, int OUT, bool SAL>
int launch_stream4db(const GemmArgs& a, int grid, hipStream_t s) {
  // SAL: A's e8m0 plane in lane order as well (gemm_stream4dbl_kernel.hpp), nothing but A in LDS
  constexpr int lds = 4 * 128 * kRowBytes + (SAL ? 0 : 2 * 128 * 16);
  void (*k)(const GemmArgs);
  if constexpr (SAL) k = gemm_stream4dbl_kernel<DT, OUT>;
  else k = gemm_stream4db_kernel<DT, OUT>;
  static std::atomic<uint64_t> attr_devs{0};
  // what the kernels' indexing assumes: whole 64-row groups of B, an even number of whole
  // K-steps, packed B, A scale rows fetched in 16-byte granules
  if (a.N % 64 != 0 || a.N < 64 || a.M < 8 || a.M % 8 != 0 || a.K % 512 != 0 || a.tail_granules != 0 ||
      a.ldb_bytes != (int64_t)a.K / 2 || (((uintptr_t)a.mx_a | (uintptr_t)a.mx_b) & 15) != 0 ||
      a.mx_ld % 16 != 0)
    return (int)hipErrorInvalidValue;
  const int own_ready = lds_attr_once(attr_devs, (const void*)k, lds);
  if constexpr (SAL) {
    bool taken = false;
    if (const int e = k8_instead<DT, OUT>(a, own_ready, s, &taken); e || taken) return e;
  }
  if (own_ready != 0) return own_ready;
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(256), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_stream4db(const astergemm_config& c) {
  if (c.M % 8 != 0 || c.M < 8) return "M must be a multiple of 8";
  if (c.N % 64 != 0 || c.N < 64) return "the pre-shuffled scale plane needs N % 64 == 0";
  if (c.K % 512 != 0) return "K must be a multiple of 512";
  if (c.ldb != 0 && c.ldb != c.K) return "pre-shuffled B is packed (ldb = K)";
  if (c.ldc % 8 != 0) return "ldc must be a multiple of 8 elements";
  if (c.N * (c.K / 2) >= ((int64_t)1 << 32)) return "pre-shuffled B must stay below 4 GiB";
  return nullptr;
}

#define AG_STREAM4DB(name, DT, OUT, SAL)                                         \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 256, kRowBytes, 1, 4, 4, 2,       \
        4 * 128 * kRowBytes + (SAL ? 0 : 2 * 128 * 16),                          \
        SAL ? (const void*)gemm_stream4dbl_kernel<DT, OUT>                       \
            : (const void*)gemm_stream4db_kernel<DT, OUT>,                       \
        launch_stream4db<DT, OUT, SAL>, check_stream4db,                         \
        ASTERGEMM_OPERAND_DIRECT_B_K8, nullptr, nullptr,                         \
        SAL ? ASTERGEMM_MX_LANES128 : ASTERGEMM_MX_ROWS,                         \
        SAL ? k8_describe<DT, OUT> : nullptr, SAL                                \
  }

// ---- fp8, B pre-shuffled into step order and loaded straight into MFMA operands: 128 x 256
// tiles, four waves (gemm_stream8db_kernel.hpp) -------------------------------------------------
template <int DT, int OUT>
int launch_stream8db(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = 4 * 128 * kRowBytes;
  auto k = gemm_stream8db_kernel<DT, OUT>;
  static std::atomic<uint64_t> attr_devs{0};
  // what the kernels' indexing assumes: whole 16-row blocks of B, whole K-steps, packed B
  if (a.N % 16 != 0 || a.N < 16 || a.M < 8 || a.M % 8 != 0 || a.K % 128 != 0 || a.tail_granules != 0 ||
      a.ldb_bytes != (int64_t)a.K)
    return (int)hipErrorInvalidValue;
  const int own_ready = lds_attr_once(attr_devs, (const void*)k, lds);
  bool taken = false;
  if (const int e = k8_instead<DT, OUT>(a, own_ready, s, &taken); e || taken) return e;
  if (own_ready != 0) return own_ready;
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(256), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_stream8db(const astergemm_config& c) {
  if (c.M % 8 != 0 || c.M < 8) return "M must be a multiple of 8";
  if (c.N % 16 != 0 || c.N < 16) return "pre-shuffled B needs N % 16 == 0";
  if (c.K % 128 != 0) return "pre-shuffled fp8 B needs K % 128 == 0";
  if (c.ldb != 0 && c.ldb != c.K) return "pre-shuffled B is packed (ldb = K)";
  if (c.ldc % 8 != 0) return "ldc must be a multiple of 8 elements";
  if (c.N * c.K >= ((int64_t)1 << 32)) return "pre-shuffled B must stay below 4 GiB";
  return nullptr;
}

#define AG_STREAM8DB(name, DT, OUT)                                              \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 256, kRowBytes, 1, 4, 4, 2,       \
        4 * 128 * kRowBytes,                                                     \
        (const void*)gemm_stream8db_kernel<DT, OUT>, launch_stream8db<DT, OUT>,  \
        check_stream8db, ASTERGEMM_OPERAND_DIRECT_B_K8, nullptr, nullptr, 0,     \
        k8_describe<DT, OUT>, true                                               \
  }

// ---- split K on the 128x128 kernel --------------------------------------------------------
//
// KIND 0: 16-bit operands, 1: fp8, 2: MXFP4 (ranges of an even number of steps)
template <int KIND, int DT, int OUT>
int launch_stream_splitk(const GemmArgs& a0, int grid, hipStream_t s) {
  (void)grid;
  constexpr int lds = KIND == 2 ? 4 * 128 * kRowBytes + 4 * 128 * 16 : 5 * 128 * kRowBytes;
  void (*k)(const GemmArgs);
  if constexpr (KIND == 0) k = gemm_stream_splitk_kernel<DT, 128, 128, 2, 2>;
  else if constexpr (KIND == 1) k = gemm_stream8_splitk_kernel<DT, 128, 128, 2, 2>;
  else k = gemm_stream4_splitk_kernel<DT, 128, 128, 2, 2>;
  static std::atomic<uint64_t> attr_devs{0};
  bool taken = false;
  if (const int e = kwave_prompt(DT, OUT, a0, lds_attr_once(attr_devs, (const void*)k, lds), s, &taken); e || taken) {
    const int ranges = stream_split_of((int64_t)a0.tiles_m * a0.tiles_n, a0.ksteps, KIND == 2);
    if (!e && !a0.workspace && !launch_context().prepare_only)
      splitk_workspace_touch((size_t)ranges * a0.M * a0.N * sizeof(float), s);
    return e;
  }
  if constexpr (KIND == 2) {
    if ((((uintptr_t)a0.mx_a | (uintptr_t)a0.mx_b) & 15) != 0 || a0.mx_ld % 16 != 0)
      return (int)hipErrorInvalidValue;
  }
  const int tiles = a0.tiles_m * a0.tiles_n;
  const int S = stream_split_of(tiles, a0.ksteps, KIND == 2);
  if (S == 0) return (int)hipErrorInvalidValue;
  GemmArgs a = a0;
  std::lock_guard<std::mutex> order(splitk_order());
  if (!a.workspace) {
    if (int rc = splitk_workspace_for((size_t)S * a.M * a.N * sizeof(float), s, &a.workspace))
      return rc;
  }
  GemmArgs part = a;           // what the K-range workgroups see: fp32 planes, no epilogue terms
  part.split_k = S;
  part.ksteps = a.ksteps / S;
  part.ldc = a.N;
  part.scale_a = part.scale_b = part.bias = nullptr;
  AG_LAUNCH_KERNEL(k, dim3(tiles * S), dim3(256), lds, s, part);
  // the partial sums must exist before anything adds them: a failed launch ends here
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
  return splitk_reduce(OUT, a, S, s);
}

const char* check_stream_splitk(const astergemm_config& c) {
  if (const char* why = check_stream_whole_k(c)) return why;
  if (c.dtype_ab == ASTERGEMM_MXFP4 && c.K % 512 != 0) return "K must be a multiple of 512";
  const int64_t tiles = ((c.M + 127) / 128) * ((c.N + 127) / 128);
  // a ragged M with a handful of tiles stays with the 64 x 64 kernels: the tests pin this selection, which is
  // the slower one there (bf16 100x512x8192 31.8 against 12.4 us, 129x256x28672 102 against 22.3, fp8
  // 250x384x14336 31.2 against 14.3, MXFP4 129x256x28672 36.0 against 13.0, 333x256x8192 12.6 against 11.6)
  if (c.M % 8 != 0 && tiles < 8) return "split K of a ragged M needs eight output tiles";
  // shorter rows: the unsplit 64 x 64 kernels are ahead (fp8 256x4096x4096: 15.2 against 19.8 us)
  const int64_t min_steps = c.dtype_ab == ASTERGEMM_MXFP4 ? 32 : 64;
  if (row_bytes(c.dtype_ab, c.K) / kRowBytes < min_steps)
    return "split K needs rows of at least 8 KiB (4 KiB for MXFP4)";
  if (stream_split_of(tiles, row_bytes(c.dtype_ab, c.K) / kRowBytes,
                      c.dtype_ab == ASTERGEMM_MXFP4) == 0)
    return "split K needs at most 128 output tiles of 128 x 128 and a K that divides into 2..16 "
           "ranges of 8 or more 128-byte steps (an even number of steps for MXFP4)";
  if (c.M * c.N > ((int64_t)1 << 26)) return "split K workspace would pass 4 GiB";
  return nullptr;
}

int splits_stream_splitk(const astergemm_config& c) {
  const int64_t tiles = ((c.M + 127) / 128) * ((c.N + 127) / 128);
  const int S = stream_split_of(tiles, row_bytes(c.dtype_ab, c.K) / kRowBytes,
                                c.dtype_ab == ASTERGEMM_MXFP4);
  return S < 1 ? 1 : S;
}

#define AG_STREAM_SPLITK(name, KIND, DT, OUT, LDS, FUNC)                         \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 128, kRowBytes, 2, 2, 3, 4, LDS,  \
        (const void*)FUNC<DT, 128, 128, 2, 2>, launch_stream_splitk<KIND, DT, OUT>, \
        check_stream_splitk, ASTERGEMM_OPERAND_LDS, splits_stream_splitk,        \
        nullptr, 0, kwave_prompt_describe, true                                  \
  }
#define AG_STREAM_SPLITK_SET(prefix, KIND, DT, LDS, FUNC)                        \
  AG_STREAM_SPLITK(prefix "_128x128_w2x2_bf16", KIND, DT, ASTERGEMM_BF16, LDS, FUNC),   \
      AG_STREAM_SPLITK(prefix "_128x128_w2x2_f32", KIND, DT, ASTERGEMM_F32, LDS, FUNC), \
      AG_STREAM_SPLITK(prefix "_128x128_w2x2_f16", KIND, DT, ASTERGEMM_F16, LDS, FUNC)

// ---- split K on the 256 x 128 tiles; rank 6: AUTO takes them by unequal_split_pays --------------
template <int DT, int OUT>
int launch_streamr_splitk(const GemmArgs& a0, int grid, hipStream_t s) {
  (void)grid;
  constexpr int lds = 3 * (256 + 128) * kRowBytes;
  auto k = gemm_streamr_splitk_kernel<DT, 256, 128, 4, 2, 3>;
  static std::atomic<uint64_t> attr_devs{0};
  if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) return e;
  const int tiles = a0.tiles_m * a0.tiles_n;
  const int S = streamr_split_of(tiles, a0.ksteps);
  if (S == 0 || a0.tail_granules != 0) return (int)hipErrorInvalidValue;
  GemmArgs a = a0;
  std::lock_guard<std::mutex> order(splitk_order());
  if (!a.workspace) {
    if (int rc = splitk_workspace_for((size_t)S * a.M * a.N * sizeof(float), s, &a.workspace))
      return rc;
  }
  GemmArgs part = a;
  part.split_k = S;
  part.ksteps = a.ksteps / S;
  part.ldc = a.N;
  part.scale_a = part.scale_b = part.bias = nullptr;
  AG_LAUNCH_KERNEL(k, dim3(tiles * S), dim3(512), lds, s, part);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
  return splitk_reduce(OUT, a, S, s);
}

int splits_streamr_splitk(const astergemm_config& c) {
  const int64_t tiles = ((c.M + 255) / 256) * ((c.N + 127) / 128);
  const int S = streamr_split_of(tiles, row_bytes(c.dtype_ab, c.K) / kRowBytes);
  return S < 1 ? 1 : S;
}

const char* check_streamr_splitk(const astergemm_config& c) {
  if (const char* why = check_stream_whole_k(c)) return why;
  if (row_bytes(c.dtype_ab, c.K) / kRowBytes < 64) return "split K needs rows of at least 8 KiB";
  if (splits_streamr_splitk(c) < 2) return "split K needs at most 128 output tiles of 256 x 128 and 2..4 K ranges";
  return nullptr;
}

#define AG_STREAMR_SPLITK(name, DT, OUT)                                         \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 128, kRowBytes, 4, 2, 3, 6,       \
        3 * (256 + 128) * kRowBytes,                                             \
        (const void*)gemm_streamr_splitk_kernel<DT, 256, 128, 4, 2, 3>,          \
        launch_streamr_splitk<DT, OUT>, check_streamr_splitk,                    \
        ASTERGEMM_OPERAND_LDS, splits_streamr_splitk, nullptr, 0, nullptr, true  \
  }
#define AG_STREAMR_SPLITK_SET(prefix, DT)                                        \
  AG_STREAMR_SPLITK(prefix "_256x128_w4x2_bf16", DT, ASTERGEMM_BF16),            \
      AG_STREAMR_SPLITK(prefix "_256x128_w4x2_f32", DT, ASTERGEMM_F32),          \
      AG_STREAMR_SPLITK(prefix "_256x128_w4x2_f16", DT, ASTERGEMM_F16)

template <int DT, int OUT, int BM, int BN, int WM, int WN>
int launch_stream8(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = 5 * BM * kRowBytes;
  auto k = gemm_stream8_kernel<DT, OUT, BM, BN, WM, WN>;
  static std::atomic<uint64_t> attr_devs{0};
  if constexpr (BM == 128) {
    bool taken = false;
    if (const int e = kwave_prompt(DT, OUT, a, lds_attr_once(attr_devs, (const void*)k, lds), s, &taken); e || taken)
      return e;
  } else if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) {
    return e;
  }
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), lds, s, a);
  return (int)hipGetLastError();
}

// The 256 x 256 fp8 kernel as a tile walk (see gemm_stream8_body): one workgroup per CU.
template <int DT, int OUT>
int launch_stream8_walk(const GemmArgs& a, int grid, hipStream_t s) {
  (void)grid;
  constexpr int lds = 5 * 256 * kRowBytes;
  // what the kernel assumes: whole tiles (its epilogue stores without bounds checks), whole
  // K-steps and enough of them for the steady form of trip 0
  if (a.M % 256 != 0 || a.N % 256 != 0 || a.tail_granules != 0 || a.ksteps < 4)
    return (int)hipErrorInvalidValue;
  auto k = gemm_stream8_walk_kernel<DT, OUT, 256, 256, 2, 4>;
  static std::atomic<uint64_t> attr_devs{0};
  if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) return e;
  const int cus = device_cus();
  if (cus <= 0) return (int)hipErrorNoDevice;
  const int tiles = a.tiles_m * a.tiles_n;
  AG_LAUNCH_KERNEL(k, dim3(tiles < cus ? tiles : cus), dim3(512), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_stream8_walk(const astergemm_config& c) {
  if (const char* why = check_stream_whole_k(c)) return why;
  if (c.K < 512) return "the tile walk needs at least four K-steps";
  if (c.M % 256 != 0 || c.N % 256 != 0) return "the tile walk needs M and N to be multiples of 256";
  int cus = device_cus();
  if (cus <= 0) cus = 256;                       // no device to ask: describe the MI355X
  if (((c.M + 255) / 256) * ((c.N + 255) / 256) <= cus)
    return "the tile walk pays from two tiles per workgroup on";
  return nullptr;
}

int grid_stream_walk(const astergemm_config& c, int cus) {
  const int64_t tiles = ((c.M + 255) / 256) * ((c.N + 255) / 256);
  if (cus <= 0) cus = 256;
  return (int)(tiles > cus ? cus : tiles);
}

#define AG_STREAM8_WALK(name, DT, OUT, RANK)                                     \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, 2, 4, 3, RANK,    \
        5 * 256 * kRowBytes,                                                     \
        (const void*)gemm_stream8_walk_kernel<DT, OUT, 256, 256, 2, 4>,          \
        launch_stream8_walk<DT, OUT>, check_stream8_walk, ASTERGEMM_OPERAND_LDS, \
        nullptr, grid_stream_walk                                                \
  }
#define AG_STREAM8(name, DT, OUT)                                                \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, 2, 4, 3, 2,       \
        5 * 256 * kRowBytes,                                                     \
        (const void*)gemm_stream8_kernel<DT, OUT, 256, 256, 2, 4>,               \
        launch_stream8<DT, OUT, 256, 256, 2, 4>, check_stream                    \
  }
#define AG_STREAM8_128(name, DT, OUT)                                            \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 128, kRowBytes, 2, 2, 3, 2,       \
        5 * 128 * kRowBytes,                                                     \
        (const void*)gemm_stream8_kernel<DT, OUT, 128, 128, 2, 2>,               \
        launch_stream8<DT, OUT, 128, 128, 2, 2>, check_stream,                   \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0, kwave_prompt_describe, true  \
  }

template <int DT, int OUT, int BM, int BN, int WM, int WN>
int launch_stream4(const GemmArgs& a, int grid, hipStream_t s) {
  constexpr int lds = 4 * BM * kRowBytes + 4 * BM * 16;
  // the scale planes are fetched in 16-byte granules
  if ((((uintptr_t)a.mx_a | (uintptr_t)a.mx_b) & 15) != 0 || a.mx_ld % 16 != 0)
    return (int)hipErrorInvalidValue;
  auto k = gemm_stream4_kernel<DT, OUT, BM, BN, WM, WN>;
  static std::atomic<uint64_t> attr_devs{0};
  if constexpr (BM == 128) {
    bool taken = false;
    if (const int e = kwave_prompt(DT, OUT, a, lds_attr_once(attr_devs, (const void*)k, lds), s, &taken); e || taken)
      return e;
  } else if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) {
    return e;
  }
  AG_LAUNCH_KERNEL(k, dim3(grid), dim3(WM * WN * 64), lds, s, a);
  return (int)hipGetLastError();
}

// Whole 256x256 tiles and an even number of 256-element K-steps (scales move in 16-byte
// granules = two K-steps of a row).
const char* check_stream4(const astergemm_config& c) {
  if (const char* why = check_stream_whole_k(c)) return why;
  if (c.K % 512 != 0) return "K must be a multiple of 512";
  return nullptr;
}

#define AG_STREAM4(name, DT, OUT)                                                \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, 2, 2, 2, 1,       \
        4 * 256 * kRowBytes + 4 * 256 * 16,                                      \
        (const void*)gemm_stream4_kernel<DT, OUT, 256, 256, 2, 2>,               \
        launch_stream4<DT, OUT, 256, 256, 2, 2>, check_stream4                   \
  }
// The same kernel with eight waves (2 x 4, wave tile 128 x 64, two waves per SIMD): with the
// accumulators in the accumulation registers it allocates without spills (128 + 116), and a
// second wave on every SIMD covers the waits of the first.  p50, one box, four -> eight waves:
// 4096 x 14336 x 4096 134.2 -> 125.3 us, 8192^3 246.8 -> 243.1, 16384 x 16384 x 4096 550.5 ->
// 533.3, 4096^3 38.1 -> 37.3; the same bits.  Preferred (rank 2 over 1).
#define AG_STREAM4_W8(name, DT, OUT, RANK)                                       \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, 2, 4, 2, RANK,    \
        4 * 256 * kRowBytes + 4 * 256 * 16,                                      \
        (const void*)gemm_stream4_kernel<DT, OUT, 256, 256, 2, 4>,               \
        launch_stream4<DT, OUT, 256, 256, 2, 4>, check_stream4                   \
  }
// Tile walk: one workgroup per CU takes its tiles round-robin as one long K loop, the next
// tile's first K-steps arriving during the last trips and the epilogue of the current one
// (see gemm_stream4_body).  16 KiB of LDS outside the ring stage the epilogue.
template <int DT, int OUT>
int launch_stream4_walk(const GemmArgs& a, int grid, hipStream_t s) {
  (void)grid;
  constexpr int lds = 4 * 256 * kRowBytes + 4 * 256 * 16 + 8 * 2048;
  if ((((uintptr_t)a.mx_a | (uintptr_t)a.mx_b) & 15) != 0 || a.mx_ld % 16 != 0)
    return (int)hipErrorInvalidValue;
  // what the kernel assumes: slot parities that carry over from tile to tile, and whole tiles
  // (its epilogue stores without bounds checks)
  if (a.ksteps % 4 != 0 || a.M % 256 != 0 || a.N % 256 != 0) return (int)hipErrorInvalidValue;
  auto k = gemm_stream4_walk_kernel<DT, OUT, 256, 256, 2, 4>;
  static std::atomic<uint64_t> attr_devs{0};
  if (int e = lds_attr_once(attr_devs, (const void*)k, lds)) return e;
  const int cus = device_cus();
  if (cus <= 0) return (int)hipErrorNoDevice;
  const int tiles = a.tiles_m * a.tiles_n;
  AG_LAUNCH_KERNEL(k, dim3(tiles < cus ? tiles : cus), dim3(512), lds, s, a);
  return (int)hipGetLastError();
}

const char* check_stream4_walk(const astergemm_config& c) {
  if (const char* why = check_stream4(c)) return why;
  if (c.K % 1024 != 0) return "the tile walk needs K to be a multiple of 1024";
  if (c.M % 256 != 0 || c.N % 256 != 0) return "the tile walk needs M and N to be multiples of 256";
  int cus = device_cus();
  if (cus <= 0) cus = 256;                       // no device to ask: describe the MI355X
  if (((c.M + 255) / 256) * ((c.N + 255) / 256) <= cus)
    return "the tile walk pays from two tiles per workgroup on";
  return nullptr;
}

int grid_stream4_walk(const astergemm_config& c, int cus) {
  const int64_t tiles = ((c.M + 255) / 256) * ((c.N + 255) / 256);
  if (cus <= 0) cus = 256;
  return (int)(tiles > cus ? cus : tiles);
}

#define AG_STREAM4_WALK(name, DT, OUT)                                           \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, 2, 4, 2, 3,       \
        4 * 256 * kRowBytes + 4 * 256 * 16 + 8 * 2048,                           \
        (const void*)gemm_stream4_walk_kernel<DT, OUT, 256, 256, 2, 4>,          \
        launch_stream4_walk<DT, OUT>, check_stream4_walk, ASTERGEMM_OPERAND_LDS, \
        nullptr, grid_stream4_walk                                               \
  }
#define AG_STREAM4_128(name, DT, OUT)                                            \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 128, 128, kRowBytes, 2, 2, 2, 2,       \
        4 * 128 * kRowBytes + 4 * 128 * 16,                                      \
        (const void*)gemm_stream4_kernel<DT, OUT, 128, 128, 2, 2>,               \
        launch_stream4<DT, OUT, 128, 128, 2, 2>, check_stream4,                  \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0, kwave_prompt_describe, true  \
  }

// ---- whole rounds of 256 x 256 tiles, the rest in 128 x 128 tiles ---------------------------
//
// One workgroup of the 256 x 256 kernels runs per CU, so a tile count that is not a multiple of
// the CU count leaves the last round partly empty (4096 x 14336: 896 tiles on 256 CUs = 3.5
// rounds, paid as 4).  The problem is cut along N or M: the part whose 256 x 256 tiles fill
// whole rounds goes to the 256 x 256 kernel, the remaining columns (or rows) to the 128 x 128
// kernel of the same family, two workgroups per CU, right behind it on the same stream.
// Measured on 4096 x 14336 x 4096, p50 on one box, 256 x 256 alone -> with the cut: MXFP4 136.3 ->
// 134.7 us, bf16 350.2 -> 343.4 us, fp8 179.2 -> 180.0 us (128 x 128 alone: 141.9, 393.7, 203.5).
// The gain is far below the 12 % of the empty half round: the chip is power limited, and the CUs
// that stay busy in a half-empty round run at a higher clock.
struct TailSplit {
  int along = 0;      // 0 = no split, 1 = along N, 2 = along M
  int64_t first = 0;  // columns (rows) of the 256 x 256 part
};

inline TailSplit tail_split_of(int64_t M, int64_t N, int cus) {
  TailSplit best;
  if (cus <= 0) cus = 256;
  const int64_t tm = (M + 255) / 256, tn = (N + 255) / 256;
  const double whole = (double)((tm * tn + cus - 1) / cus);
  double best_cost = whole * 0.93;  // a split has to save at least 7 %
  for (int along = 1; along <= 2; ++along) {
    const int64_t cut_tiles = along == 1 ? tn : tm, other = along == 1 ? tm : tn;
    const int64_t extent = along == 1 ? N : M;
    // the largest number of tile columns (rows) that gives whole rounds
    for (int64_t t1 = cut_tiles - 1; t1 >= 1; --t1) {
      if ((t1 * other) % cus != 0) continue;
      const int64_t rest = extent - t1 * 256;
      if (rest < 8) break;  // the 128 x 128 kernel shifts the edge by up to 8 rows (edge_row)
      const int64_t rest128 = (rest + 127) / 128 * (((along == 1 ? M : N) + 127) / 128);
      const double cost = (double)(t1 * other / cus) +
                          0.55 * (double)((rest128 + 2 * cus - 1) / (2 * cus));
      if (cost < best_cost) {
        best_cost = cost;
        best.along = along;
        best.first = t1 * 256;
      }
      break;
    }
  }
  return best;
}

// the two sub-problems of a split: `part1` the first `ts.first` columns (rows), `part2` the rest
inline void tail_parts(const GemmArgs& a, const TailSplit& ts, int out_bytes, GemmArgs* part1,
                       GemmArgs* part2) {
  *part1 = a;
  *part2 = a;
  part1->own_kernel = part2->own_kernel = 1;   // the bits of the tile kernels, whatever the parts' sizes
  if (ts.along == 1) {
    part1->N = (int32_t)ts.first;
    part2->N = a.N - (int32_t)ts.first;
    part2->B = a.B + ts.first * a.ldb_bytes;
    if (a.mx_b) part2->mx_b = a.mx_b + ts.first * a.mx_ld;
    if (a.bias) part2->bias = a.bias + ts.first;
    part2->C = (uint8_t*)a.C + ts.first * out_bytes;
  } else {
    part1->M = (int32_t)ts.first;
    part2->M = a.M - (int32_t)ts.first;
    part2->A = a.A + ts.first * a.lda_bytes;
    if (a.mx_a) part2->mx_a = a.mx_a + ts.first * a.mx_ld;
    part2->C = (uint8_t*)a.C + ts.first * a.ldc * out_bytes;
  }
  part1->tiles_m = (part1->M + 255) / 256;
  part1->tiles_n = (part1->N + 255) / 256;
  part2->tiles_m = (part2->M + 127) / 128;
  part2->tiles_n = (part2->N + 127) / 128;
  // the tile order is a property of each part's own tile grid (see map_tile)
  part1->group_m = tile_order(part1->tiles_m, part1->tiles_n);
  part2->group_m = tile_order(part2->tiles_m, part2->tiles_n);
}

// KIND 0: 16-bit operands, 1: fp8, 2: MXFP4
template <int KIND, int DT, int OUT>
int launch_stream_tail(const GemmArgs& a, int grid, hipStream_t s) {
  (void)grid;
  const TailSplit ts = tail_split_of(a.M, a.N, device_cus());
  if (ts.along == 0) return (int)hipErrorInvalidValue;
  GemmArgs p1, p2;
  tail_parts(a, ts, OUT == ASTERGEMM_F32 ? 4 : 2, &p1, &p2);
  const int g1 = p1.tiles_m * p1.tiles_n, g2 = p2.tiles_m * p2.tiles_n;
  int rc;
  if constexpr (KIND == 0) {
    if ((rc = launch_stream<DT, OUT, 256, 256, 2, 4>(p1, g1, s)) != 0) return rc;
    return launch_stream<DT, OUT, 128, 128, 2, 2>(p2, g2, s);
  } else if constexpr (KIND == 1) {
    // the whole rounds as a tile walk where its conditions hold (see launch_stream8_walk)
    const bool walk = p1.M % 256 == 0 && p1.N % 256 == 0 && p1.tail_granules == 0 &&
                      p1.ksteps >= 4 && g1 > device_cus();
    rc = walk ? launch_stream8_walk<DT, OUT>(p1, g1, s) : launch_stream8<DT, OUT, 256, 256, 2, 4>(p1, g1, s);
    if (rc != 0) return rc;
    return launch_stream8<DT, OUT, 128, 128, 2, 2>(p2, g2, s);
  } else {
    // the whole rounds as a tile walk where its conditions hold (see launch_stream4_walk)
    const bool walk = p1.ksteps % 4 == 0 && p1.M % 256 == 0 && p1.N % 256 == 0 && g1 > device_cus();
    rc = walk ? launch_stream4_walk<DT, OUT>(p1, g1, s) : launch_stream4<DT, OUT, 256, 256, 2, 4>(p1, g1, s);
    if (rc != 0) return rc;
    return launch_stream4<DT, OUT, 128, 128, 2, 2>(p2, g2, s);
  }
}

const char* check_stream_tail(const astergemm_config& c) {
  if (c.dtype_ab == ASTERGEMM_MXFP4) {
    if (const char* why = check_stream4(c)) return why;
  } else if (const char* why = check_stream(c)) {
    return why;
  }
  if (tail_split_of(c.M, c.N, device_cus()).along == 0)
    return "no cut along M or N gives whole rounds of 256 x 256 tiles plus a cheaper rest";
  return nullptr;
}

int grid_stream_tail(const astergemm_config& c, int cus) {
  const TailSplit ts = tail_split_of(c.M, c.N, cus);
  if (ts.along == 0) return (int)(((c.M + 255) / 256) * ((c.N + 255) / 256));
  const int64_t m1 = ts.along == 2 ? ts.first : c.M, n1 = ts.along == 1 ? ts.first : c.N;
  const int64_t m2 = ts.along == 2 ? c.M - ts.first : c.M, n2 = ts.along == 1 ? c.N - ts.first : c.N;
  int64_t g1 = ((m1 + 255) / 256) * ((n1 + 255) / 256);
  // MXFP4, fp8: the whole rounds run as a tile walk, one workgroup per CU (see launch_stream_tail)
  if (cus <= 0) cus = 256;
  if (c.dtype_ab == ASTERGEMM_MXFP4 && c.K % 1024 == 0 && m1 % 256 == 0 && n1 % 256 == 0 && g1 > cus)
    g1 = cus;
  if (c.dtype_ab == ASTERGEMM_FP8_E4M3 && c.K % 128 == 0 && c.K >= 512 && m1 % 256 == 0 &&
      n1 % 256 == 0 && g1 > cus)
    g1 = cus;
  return (int)(g1 + ((m2 + 127) / 128) * ((n2 + 127) / 128));
}

// rank 3: preferred over the plain 256 x 256 kernel wherever its check passes
#define AG_STREAM_TAIL(name, KIND, DT, OUT, WM, WN, LDS, FUNC)                   \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 256, 256, kRowBytes, WM, WN, 3, 3, LDS, \
        (const void*)FUNC<DT, OUT, 256, 256, WM, WN>, launch_stream_tail<KIND, DT, OUT>, \
        check_stream_tail, ASTERGEMM_OPERAND_LDS, nullptr, grid_stream_tail      \
  }
#define AG_STREAM_TAIL_SET(prefix, KIND, DT, WM, WN, LDS, FUNC)                  \
  AG_STREAM_TAIL(prefix "_bf16", KIND, DT, ASTERGEMM_BF16, WM, WN, LDS, FUNC),   \
      AG_STREAM_TAIL(prefix "_f32", KIND, DT, ASTERGEMM_F32, WM, WN, LDS, FUNC), \
      AG_STREAM_TAIL(prefix "_f16", KIND, DT, ASTERGEMM_F16, WM, WN, LDS, FUNC)

#define AG_STREAM_SET(prefix, DT)                                                      \
  AG_STREAM(prefix "_256x256_w2x4_bf16", DT, ASTERGEMM_BF16, 256, 256, 2, 4),          \
      AG_STREAM(prefix "_256x256_w2x4_f32", DT, ASTERGEMM_F32, 256, 256, 2, 4),        \
      AG_STREAM(prefix "_256x256_w2x4_f16", DT, ASTERGEMM_F16, 256, 256, 2, 4),        \
      AG_STREAM(prefix "_256x256_w2x2_bf16", DT, ASTERGEMM_BF16, 256, 256, 2, 2),        \
      AG_STREAM(prefix "_128x128_w2x2_bf16", DT, ASTERGEMM_BF16, 128, 128, 2, 2),        \
      AG_STREAM(prefix "_128x128_w2x2_f32", DT, ASTERGEMM_F32, 128, 128, 2, 2),          \
      AG_STREAM(prefix "_128x128_w2x2_f16", DT, ASTERGEMM_F16, 128, 128, 2, 2)

// The table is compiled in five parts (this file once per AG_STREAM_PART: bf16, fp8, MXFP4 and f16
// operands, and unequal tile sides), so that the parts build side by side and work on one family
// recompiles one part.
#ifndef AG_STREAM_PART
#error "compile with -DAG_STREAM_PART=0, 1, 2, 3 or 4"
#endif

const Variant kStreamVariants[] = {
#if AG_STREAM_PART == 0 || AG_STREAM_PART == 3
#if AG_STREAM_PART == 0
#define AG_P16 ASTERGEMM_BF16
#define AG_N16(x) x "_bf16"
#else
#define AG_P16 ASTERGEMM_F16
#define AG_N16(x) x "_f16"
#endif
    AG_STREAM_SET(AG_N16("stream"), AG_P16),
    AG_STREAM_SPLITK_SET(AG_N16("splitk"), 0, AG_P16, 5 * 128 * kRowBytes, gemm_stream_splitk_kernel),
    AG_STREAMDB(AG_N16("streamdb") "_256x256_w2x4_bf16", AG_P16, ASTERGEMM_BF16, 5, 5, 2, 2),
    AG_STREAMDB(AG_N16("streamdb") "_256x256_w2x4_f32", AG_P16, ASTERGEMM_F32, 5, 5, 2, 2),
    AG_STREAMDB(AG_N16("streamdb") "_256x256_w2x4_f16", AG_P16, ASTERGEMM_F16, 5, 5, 2, 2),
    AG_STREAMDB(AG_N16("streamdb") "_128x256_w1x4_bf16", AG_P16, ASTERGEMM_BF16, 5, 5, 1, 1),
    AG_STREAMDB(AG_N16("streamdb") "_128x256_w1x4_f32", AG_P16, ASTERGEMM_F32, 5, 5, 1, 1),
    AG_STREAMDB(AG_N16("streamdb") "_128x256_w1x4_f16", AG_P16, ASTERGEMM_F16, 5, 5, 1, 1),
    AG_STREAM_TAIL_SET(AG_N16("stream") "_256x256_w2x4_tail128", 0, AG_P16, 2, 4, 5 * 256 * kRowBytes,
                       gemm_stream_kernel),
    AG_STREAM_RING9_SET(AG_N16("stream"), AG_P16),
    AG_DIRECTAB_SET(AG_N16("directab"), AG_P16),
#elif AG_STREAM_PART == 1
    AG_STREAM_SPLITK_SET("splitk_fp8", 1, ASTERGEMM_FP8_E4M3, 5 * 128 * kRowBytes,
                         gemm_stream8_splitk_kernel),
    AG_STREAM_TAIL_SET("stream_fp8_256x256_w2x4_tail128", 1, ASTERGEMM_FP8_E4M3, 2, 4,
                       5 * 256 * kRowBytes, gemm_stream8_kernel),
    AG_STREAM8("stream_fp8_256x256_w2x4_bf16", ASTERGEMM_FP8_E4M3, ASTERGEMM_BF16),
    AG_STREAM8("stream_fp8_256x256_w2x4_f32", ASTERGEMM_FP8_E4M3, ASTERGEMM_F32),
    AG_STREAM8("stream_fp8_256x256_w2x4_f16", ASTERGEMM_FP8_E4M3, ASTERGEMM_F16),
    AG_STREAM8_WALK("stream_fp8_256x256_w2x4_walk_bf16", ASTERGEMM_FP8_E4M3, ASTERGEMM_BF16, 3),
    AG_STREAM8_WALK("stream_fp8_256x256_w2x4_walk_f32", ASTERGEMM_FP8_E4M3, ASTERGEMM_F32, 3),
    AG_STREAM8_WALK("stream_fp8_256x256_w2x4_walk_f16", ASTERGEMM_FP8_E4M3, ASTERGEMM_F16, 3),
    AG_STREAM8_128("stream_fp8_128x128_w2x2_bf16", ASTERGEMM_FP8_E4M3, ASTERGEMM_BF16),
    AG_STREAM8_128("stream_fp8_128x128_w2x2_f32", ASTERGEMM_FP8_E4M3, ASTERGEMM_F32),
    AG_STREAM8_128("stream_fp8_128x128_w2x2_f16", ASTERGEMM_FP8_E4M3, ASTERGEMM_F16),
    AG_STREAM8DB("streamdb_fp8_128x256_w1x4_bf16", ASTERGEMM_FP8_E4M3, ASTERGEMM_BF16),
    AG_STREAM8DB("streamdb_fp8_128x256_w1x4_f32", ASTERGEMM_FP8_E4M3, ASTERGEMM_F32),
    AG_STREAM8DB("streamdb_fp8_128x256_w1x4_f16", ASTERGEMM_FP8_E4M3, ASTERGEMM_F16),
#elif AG_STREAM_PART == 4
    AG_STREAMR_SET("stream_bf16_256x128_w4x2", ASTERGEMM_BF16, 256, 128, 4, 2, 3),
    AG_STREAMR_SET("stream_bf16_192x128_w4x2", ASTERGEMM_BF16, 192, 128, 4, 2, 4),
    AG_STREAMR_SET("stream_f16_256x128_w4x2", ASTERGEMM_F16, 256, 128, 4, 2, 3),
    AG_STREAMR_SET("stream_f16_192x128_w4x2", ASTERGEMM_F16, 192, 128, 4, 2, 4),
    AG_STREAMR_SET("stream_fp8_256x128_w4x2", ASTERGEMM_FP8_E4M3, 256, 128, 4, 2, 3),
    AG_STREAMR_SET("stream_fp8_192x128_w4x2", ASTERGEMM_FP8_E4M3, 192, 128, 4, 2, 4),
    AG_STREAMR_SET("stream_fp8_128x128_w4x2", ASTERGEMM_FP8_E4M3, 128, 128, 4, 2, 5),
    AG_STREAMR_SPLITK_SET("splitk_bf16", ASTERGEMM_BF16),
    AG_STREAMR_SPLITK_SET("splitk_f16", ASTERGEMM_F16),
    AG_STREAMR_SPLITK_SET("splitk_fp8", ASTERGEMM_FP8_E4M3),
#else
    AG_STREAM_SPLITK_SET("splitk_mxfp4", 2, ASTERGEMM_MXFP4, 4 * 128 * kRowBytes + 4 * 128 * 16,
                         gemm_stream4_splitk_kernel),
    AG_STREAM_TAIL_SET("stream_mxfp4_256x256_w2x4_tail128", 2, ASTERGEMM_MXFP4, 2, 4,
                       4 * 256 * kRowBytes + 4 * 256 * 16, gemm_stream4_kernel),
    AG_STREAM4("stream_mxfp4_256x256_w2x2_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16),
    AG_STREAM4("stream_mxfp4_256x256_w2x2_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32),
    AG_STREAM4("stream_mxfp4_256x256_w2x2_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16),
    AG_STREAM4_W8("stream_mxfp4_256x256_w2x4_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16, 2),
    AG_STREAM4_W8("stream_mxfp4_256x256_w2x4_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32, 2),
    AG_STREAM4_W8("stream_mxfp4_256x256_w2x4_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16, 2),
    AG_STREAM4_WALK("stream_mxfp4_256x256_w2x4_walk_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16),
    AG_STREAM4_WALK("stream_mxfp4_256x256_w2x4_walk_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32),
    AG_STREAM4_WALK("stream_mxfp4_256x256_w2x4_walk_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16),
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16, false),
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32, false),
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16, false),
    AG_STREAM4_128("stream_mxfp4_128x128_w2x2_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16),
    AG_STREAM4_128("stream_mxfp4_128x128_w2x2_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32),
    AG_STREAM4_128("stream_mxfp4_128x128_w2x2_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16),
    // the same with A's e8m0 plane in lane order (mx_a_layout = ASTERGEMM_MX_LANES128)
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_sal_bf16", ASTERGEMM_MXFP4, ASTERGEMM_BF16, true),
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_sal_f32", ASTERGEMM_MXFP4, ASTERGEMM_F32, true),
    AG_STREAM4DB("streamdb_mxfp4_128x256_w1x4_sal_f16", ASTERGEMM_MXFP4, ASTERGEMM_F16, true),
#endif
};

}  // namespace

#define AG_CAT_(a, b) a##b
#define AG_CAT(a, b) AG_CAT_(a, b)
const Variant* AG_CAT(stream_variants_part, AG_STREAM_PART)(int* count) {
  *count = (int)(sizeof(kStreamVariants) / sizeof(kStreamVariants[0]));
  return kStreamVariants;
}

#if AG_STREAM_PART == 0
const Variant* stream_variants_part1(int* count);
const Variant* stream_variants_part2(int* count);
const Variant* stream_variants_part3(int* count);
const Variant* stream_variants_part4(int* count);

// the parts as one table: bf16, f16, fp8, MXFP4, unequal tile sides
static const std::vector<Variant>& all_stream_variants() {
  static const std::vector<Variant> all = [] {
    std::vector<Variant> v;
    int n = 0;
    const Variant* p = stream_variants_part0(&n);
    v.insert(v.end(), p, p + n);
    p = stream_variants_part3(&n);
    v.insert(v.end(), p, p + n);
    p = stream_variants_part1(&n);
    v.insert(v.end(), p, p + n);
    p = stream_variants_part2(&n);
    v.insert(v.end(), p, p + n);
    p = stream_variants_part4(&n);
    v.insert(v.end(), p, p + n);
    return v;
  }();
  return all;
}
int num_stream_variants() { return (int)all_stream_variants().size(); }
const Variant* stream_variants() { return all_stream_variants().data(); }
#endif

}  // namespace astergemm
