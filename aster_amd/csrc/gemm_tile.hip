// Variant table and launchers of the LDS-staged MFMA tile kernels
// (device code: gemm_tile_kernel.hpp).
#include "gemm_tile_kernel.hpp"
#include "gemm_kwave.h"

namespace astergemm {
namespace {

// ---- host side: variant table ------------------------------------------------
constexpr int tile_lds_bytes(int dt, int bm, int bn, int stages) {
  return stages * (bm + bn) * (kRowBytes + (dt == ASTERGEMM_MXFP4 ? 8 : 0));
}

// 64 x 64 tiles, operands of bytes: the arguments in one line whatever the size (in one line / as GemmArgs, us: MXFP4
// 512x512x1024 4.28 / 4.6, 256x256x4096 7.50 / 7.95, fp8 512x512x512 with the quantiser 10.5 / 11.2).  16-bit ones
// where a launch is as long as the kernel (bf16 500x1000x40 3.34 / 3.8, f16 1200x1200x64, 361 tiles, 3.69 / 4.35;
// bf16 1000x1000x256, 256 tiles of 4 K-steps, level at 4.5); past that the launch is hidden and unpacking stands in
// front of the K loop (f16 1100x1003x200, 288 tiles of 4, 5.00 / 4.83, bf16 391x6864x288 6.50 / 6.43, 777x1001x1032
// 8.11 / 8.07). Larger tiles have no such sizes: GemmArgs (bf16 1269x22136x312 49.3 / 48.8).
template <int DT, int BM>
constexpr bool kTileAlwaysPacks = BM == 64 && (DT == ASTERGEMM_FP8_E4M3 || DT == ASTERGEMM_MXFP4);
inline bool packs_16_bit(int64_t grid, int ksteps) { return ksteps <= 4 && grid <= 512 && grid * ksteps <= 1024; }

template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
constexpr auto tile_kernel() {
  if constexpr (kTileAlwaysPacks<DT, BM>) return gemm_tile_packed_kernel<DT, OUT, BM, BN, WM, WN, S>;
  else return gemm_tile_kernel<DT, OUT, BM, BN, WM, WN, S>;
}

template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
int tile_ready() {
  static std::atomic<uint64_t> attr_devs{0}, packed_devs{0};
  constexpr int lds = tile_lds_bytes(DT, BM, BN, S);
  if constexpr (BM == 64)
    if (int e = lds_attr_once(packed_devs, (const void*)gemm_tile_packed_kernel<DT, OUT, BM, BN, WM, WN, S>, lds))
      return e;
  if constexpr (!kTileAlwaysPacks<DT, BM>)
    return lds_attr_once(attr_devs, (const void*)gemm_tile_kernel<DT, OUT, BM, BN, WM, WN, S>, lds);
  return 0;
}

template <int DT, int OUT, int BM, int BN, int WM, int WN, int S>
int launch_tile(const GemmArgs& a, int grid, hipStream_t s) {
  if (int e = tile_ready<DT, OUT, BM, BN, WM, WN, S>()) return e;
  // the kernels that stand in for this one on small grids: a config captured later finds either ready
  if constexpr (BM == 64) (void)kwave_ready(DT);
  constexpr int lds = tile_lds_bytes(DT, BM, BN, S);
  if constexpr (BM == 64) {
    if (kTileAlwaysPacks<DT, BM> || packs_16_bit(grid, a.ksteps)) {
      AG_LAUNCH_KERNEL((gemm_tile_packed_kernel<DT, OUT, BM, BN, WM, WN, S>), dim3(grid), dim3(WM * WN * 64), lds, s,
                       pack_args(a, 0, a.C));
      return (int)hipGetLastError();
    }
  }
  if constexpr (!kTileAlwaysPacks<DT, BM>)
    AG_LAUNCH_KERNEL((gemm_tile_kernel<DT, OUT, BM, BN, WM, WN, S>), dim3(grid), dim3(WM * WN * 64), lds, s, a);
  return (int)hipGetLastError();
}

// K split over the waves (gemm_kwave.h): SPLIT = false for small products, true for decoding on byte
// rows that the kernels with resident activations do not take.
template <int DT, int OUT, bool SPLIT>
int launch_kwave_tile(const GemmArgs& a, int grid, hipStream_t s) {
  (void)grid;
  (void)tile_ready<DT, OUT, 64, 64, 2, 2, 4>();
  if (int e = kwave_ready(DT)) return e;
  const int cus = device_cus();
  if (cus <= 0) return (int)hipErrorNoDevice;
  return kwave_launch(DT, OUT, a, kwave_variant_form(SPLIT, DT, a.M, a.N, a.K, cus), s);
}

const char* check_tile(const astergemm_config& c) {
  const int64_t kb = row_bytes(c.dtype_ab, c.K);
  if (c.dtype_ab == ASTERGEMM_MXFP4) {
    if (kb % kRowBytes != 0) return "MXFP4 needs K % 256 == 0";
  } else if (kb % 16 != 0) {
    return "K must cover a whole number of 16-byte granules";
  }
  return nullptr;
}

#define AG_TILE1(name, DT, OUT, BM, BN, WM, WN, S)                               \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, BM, BN, kRowBytes, WM, WN, S, 1,       \
        tile_lds_bytes(DT, BM, BN, S),                                           \
        (const void*)tile_kernel<DT, OUT, BM, BN, WM, WN, S>(),                  \
        launch_tile<DT, OUT, BM, BN, WM, WN, S>, check_tile                      \
  }
#define AG_TILE(name, DT, BM, BN, WM, WN, S)                                     \
  AG_TILE1(name "_bf16", DT, ASTERGEMM_BF16, BM, BN, WM, WN, S),                 \
      AG_TILE1(name "_f32", DT, ASTERGEMM_F32, BM, BN, WM, WN, S),               \
      AG_TILE1(name "_f16", DT, ASTERGEMM_F16, BM, BN, WM, WN, S)

// Stages of LDS (the last number).  64 x 64 on grids of up to two workgroups per CU (past that: two stages,
// see tile64_stages_of), S = 2
// (every K-step waits for its own transfers) / 3 / 4 / 5: bf16 777x1001x1032 12.4 / 8.1 / 8.1 / 8.3 us,
// 130x4096x4096 47 / 25.5 / 19.0 / 17.8, MXFP4 300x4096x11008 45 / 32.3 / 32.7 / 41.8 (five stages: one
// workgroup per CU).  The larger tiles are taken from 448 workgroups on, where two (128 x 128) and three
// (128 x 64) workgroups share a CU only with two stages: the two-stage kernel before / S = 3 / 4 / 2, back to
// back, 128 x 128 bf16 2048x4097x4096 107 / 120 / 120 / 96.7, 700x10007x4096 66.6 / 81.7 / 80.6 / 61.2, fp8
// 700x10007x4096 40.3 / 47.7 / 47.5 / 33.5, MXFP4 2048x4096x11008 87.2 / 72.9 / 71.6 / 64.8; 128 x 64, S = 3 / 2,
// bf16 1500x4001x4096 61.7 / 63.2 / 57.4, 509x8245x8192 102 / 114 / 96.2, fp8 434x8749x8192 58.7 / 61.9 / 54.6
// (behind on rows of 512-2048 bytes, bf16 408x8089x2048 26.3 / 22.3 / 22.4).  256 x 256 has room for two.
#define AG_TILE_SET(prefix, DT)                                                  \
  AG_TILE(prefix "_256x256_w2x4", DT, 256, 256, 2, 4, 2),                        \
      AG_TILE(prefix "_128x128_w2x2", DT, 128, 128, 2, 2, 2),                    \
      AG_TILE(prefix "_128x64_w2x2", DT, 128, 64, 2, 2, 2),                      \
      AG_TILE(prefix "_64x64_w2x2", DT, 64, 64, 2, 2, 4)
template <bool SPLIT>
bool kwave_variant_describe(const astergemm_config& c, int cus, LaunchForm* o) {
  kwave_describe(c.dtype_ab, kwave_variant_form(SPLIT, c.dtype_ab, c.M, c.N, c.K, cus), c.M, c.N, cus, o);
  return true;
}

#define AG_KWAVE1(name, DT, OUT, SPLIT, RANK)                                    \
  Variant {                                                                      \
    name, ASTERGEMM_KERNEL_TILE, DT, OUT, 64, 64, kRowBytes, 2, 4, 3, RANK,      \
        0, nullptr, launch_kwave_tile<DT, OUT, SPLIT>, check_tile,               \
        ASTERGEMM_OPERAND_LDS, nullptr, nullptr, 0,                              \
        kwave_variant_describe<SPLIT>                                            \
  }
#define AG_KWAVE(name, DT, SPLIT, RANK)                                          \
  AG_KWAVE1(name "_bf16", DT, ASTERGEMM_BF16, SPLIT, RANK),                      \
      AG_KWAVE1(name "_f32", DT, ASTERGEMM_F32, SPLIT, RANK),                    \
      AG_KWAVE1(name "_f16", DT, ASTERGEMM_F16, SPLIT, RANK)
#define AG_TILE_RING2(prefix, DT)                                                \
  AG_TILE(prefix "_64x64_w2x2_ring2", DT, 64, 64, 2, 2, 2)

const Variant kTileVariants[] = {
    AG_TILE_SET("tile_bf16", ASTERGEMM_BF16),
    AG_TILE_SET("tile_f16", ASTERGEMM_F16),
    AG_TILE_SET("tile_fp8", ASTERGEMM_FP8_E4M3),
    AG_TILE_SET("tile_mxfp4", ASTERGEMM_MXFP4),
    AG_TILE_RING2("tile_bf16", ASTERGEMM_BF16),
    AG_TILE_RING2("tile_f16", ASTERGEMM_F16),
    AG_TILE_RING2("tile_fp8", ASTERGEMM_FP8_E4M3),
    AG_TILE_RING2("tile_mxfp4", ASTERGEMM_MXFP4),
    AG_KWAVE("tile_bf16_kwave", ASTERGEMM_BF16, false, 8),
    AG_KWAVE("tile_f16_kwave", ASTERGEMM_F16, false, 8),
    AG_KWAVE("tile_fp8_kwave", ASTERGEMM_FP8_E4M3, false, 8),
    AG_KWAVE("splitk_fp8_kwave", ASTERGEMM_FP8_E4M3, true, 7),
    AG_KWAVE("tile_mxfp4_kwave", ASTERGEMM_MXFP4, true, 7),
};

}  // namespace

int num_tile_variants() { return (int)(sizeof(kTileVariants) / sizeof(kTileVariants[0])); }
const Variant* tile_variants() { return kTileVariants; }

}  // namespace astergemm
