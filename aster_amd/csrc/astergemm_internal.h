// Internal declarations shared by the HIP translation units of libastergemm.
#pragma once
#include <atomic>
#include <mutex>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "astergemm.h"

namespace astergemm {

// Arguments of every GEMM kernel (passed by value as one kernarg struct).
struct GemmArgs {
  const uint8_t* A;      // [M, lda_bytes]
  const uint8_t* B;      // [N, ldb_bytes]
  void* C;               // [M, ldc] elements of the output type
  const float* scale_a;  // per-tensor scales (device) or nullptr
  const float* scale_b;
  const float* bias;     // [N] or nullptr
  const uint8_t* mx_a;   // e8m0 [M, mx_ld] or nullptr
  const uint8_t* mx_b;   // e8m0 [N, mx_ld]
  int64_t lda_bytes, ldb_bytes;
  int64_t ldc;           // elements
  int32_t mx_ld;         // bytes per row of the e8m0 planes (= K/32)
  int32_t M, N, K;       // K in elements
  int32_t ksteps;        // K-loop trip count (128 bytes of a row per step)
  int32_t tail_granules; // valid 16-byte granules of the last step, 0 = all 8
  int32_t tiles_m, tiles_n;
  int32_t group_m;       // tile rows per rasterisation group; < 0: band order (see map_tile)
  int32_t split_k;       // skinny path: K slices per output row block
  int32_t own_kernel;    // not AUTO's form: the launcher's own kernel, K loops from step 0 (Variant::auto_form)
  float* workspace;      // fp32 partials [split_k][M][N] when a row is cut into K ranges; set by
                         // the caller of a launcher = use this buffer, null = the library's own
};

// Tile order (map_tile): groups of 8 tile rows inside one contiguous run per XCD; where the tile grid divides, band order
// instead (all XCDs on one band of 8 tile rows, 8 x 4 tiles per XCD and round as before): 8192^3 bf16 +0.5 %, fp8
// +1.3 %, 16384 x 16384 x 4096 fp8 +1.2 %, MXFP4 +1.5 %, bf16 -0.1 %, same process.
__host__ __device__ inline int tile_order(int tiles_m, int tiles_n) {
  return (tiles_m % 8 == 0 && tiles_n % 32 == 0) ? -1 : 8;
}

// Bytes of one operand row covering `k` elements.
__host__ __device__ inline int64_t row_bytes(int dtype, int64_t k) {
  switch (dtype) {
    case ASTERGEMM_F16:
    case ASTERGEMM_BF16: return k * 2;
    case ASTERGEMM_FP8_E4M3: return k;
    case ASTERGEMM_MXFP4: return k / 2;
    default: return k * 4;
  }
}

// The same in one 64-byte line, for the kernels of products that a launch is a good part of.  A launch writes its
// arguments to device memory, across PCIe: one line costs the host 2.9 us, two 3.5, the 144 bytes of GemmArgs 3.6
// (empty kernels).  Addresses have 48 bits and C's pitch 58 (build_args refuses others), row pitches of A and B 23
// (validate_problem), in units of 16 bytes 19, with bits 32 ... 57 of C's above them; everything else follows from M,
// N and K.
struct PackedArgs {
  uint32_t lo[6];       // A, B, C (K ranges: the workspace), bias, scale_a or mx_a, scale_b or mx_b
  uint16_t hi[6];
  int32_t M, N, K;
  uint32_t lda, ldb, ldc;
  uint32_t form;        // the kernel's own
};
static_assert(sizeof(PackedArgs) == 64, "one line");
inline PackedArgs pack_args(const GemmArgs& a, uint32_t form, const void* c) {
  const void* ptr[6] = {a.A, a.B, c, a.bias, a.mx_a ? a.mx_a : (const void*)a.scale_a,
                        a.mx_b ? a.mx_b : (const void*)a.scale_b};
  PackedArgs q;
  for (int i = 0; i < 6; ++i) {
    q.lo[i] = (uint32_t)(uintptr_t)ptr[i];
    q.hi[i] = (uint16_t)((uintptr_t)ptr[i] >> 32);
  }
  q.M = a.M, q.N = a.N, q.K = a.K;
  q.lda = (uint32_t)(a.lda_bytes >> 4) | (uint32_t)((uint64_t)a.ldc >> 32 & 0x1FFF) << 19;
  q.ldb = (uint32_t)(a.ldb_bytes >> 4) | (uint32_t)((uint64_t)a.ldc >> 45 & 0x1FFF) << 19;
  q.ldc = (uint32_t)a.ldc;
  q.form = form;
  return q;
}

inline int out_elt_bytes(int dtype) { return dtype == ASTERGEMM_F32 ? 4 : 2; }

// What a launcher with several kernels launches for one problem.
struct LaunchForm {
  int grid = 0, tile_m = 0, tile_n = 0, waves_m = 0, waves_n = 0, stages = 0, lds_bytes = 0;
  int threads = 0;
  const void* func = nullptr;
};

// One entry of the variant table (filled in by gemm_tile.hip / gemm_skinny.hip).
struct Variant {
  const char* name;
  int family;
  int dtype_ab;      // -1 = any 16-bit float (F16 and BF16 share a kernel body)
  int dtype_c;
  int tile_m, tile_n, tile_k_bytes;
  int waves_m, waves_n;
  int stages;
  int rank;          // preference among variants of equal tile size (higher wins)
  int lds_bytes;
  const void* func;  // device function symbol, for hipFuncGetAttributes
  // Launches the kernel; returns a hipError_t as int.
  int (*launch)(const GemmArgs& a, int grid, hipStream_t s);
  // Host-side shape check: nullptr when ok, else a reason.
  const char* (*check)(const astergemm_config& c);
  // B operand form this variant reads (astergemm_operand_path); plain row-major by default.
  int operand_path = 0;
  // K ranges the launcher cuts the rows of this problem into (1 = none): the launch then needs
  // splits * M * N * 4 bytes of fp32 workspace.  nullptr = never splits.
  int (*splits)(const astergemm_config& c) = nullptr;
  // Grid the launcher uses when it is not the number of output tiles (persistent kernels);
  // `cus` = compute units of the current device.  nullptr = tiles (times splits).
  int (*grid)(const astergemm_config& c, int cus) = nullptr;
  // Layout of A's e8m0 plane this variant reads (astergemm_mx_layout); row-major by default.
  int mx_a_layout = 0;
  // Launchers with a second kernel for some problems: its description when this one is among them
  // (`cus` as for grid; 0 = no device, nothing is known to fill it).  splits() stays an upper bound then.
  bool (*form)(const astergemm_config& c, int cus, LaunchForm* o) = nullptr;
  // Where AUTO takes this variant the launcher may run another kernel (form) or start its K loops elsewhere
  // (first_step_of_xcd).  AUTO's form has an id and a name of its own, behind those of the table, which are the
  // launcher's own kernel: a plan of either gives the bits of what reported the id.  false: one form, `form`
  // if set.
  bool auto_form = false;
};

// Compute units of the current device (0 when there is none), cached per device ordinal.
int device_cus();

// State of the launcher call in progress on this thread, set by the entry points in
// astergemm_api.hip: the stream the kernels go to, and whether this is astergemm_prepare (every
// one-time step of the launcher runs, the kernels themselves are not launched).
struct LaunchContext {
  hipStream_t stream = nullptr;
  bool prepare_only = false;
  int dev = -1;  // the thread's device for the length of the call; -1: not asked for
};
LaunchContext& launch_context();
// The current device: asked for once by an entry point that has set it in the context (50 ns a time, and a call
// needs it in half a dozen places).
inline hipError_t current_device(int* dev) {
  if (const int d = launch_context().dev; d >= 0) {
    *dev = d;
    return hipSuccess;
  }
  return hipGetDevice(dev);
}

// Every GEMM kernel launch of the library goes through this macro.
#define AG_LAUNCH_KERNEL(...)                                                   \
  do {                                                                          \
    if (!::astergemm::launch_context().prepare_only) hipLaunchKernelGGL(__VA_ARGS__); \
  } while (0)

// Raises a kernel's dynamic-LDS limit once per device; `devs` is a static of the launcher with
// one bit per device ordinal.  Returns 0 or a hipError_t.  Changing a function attribute is not
// a stream operation: when the kernel's first launch on a device arrives while the stream is
// being captured into a graph, the launcher refuses (hipErrorStreamCaptureUnsupported) instead
// of touching the runtime from inside the capture; astergemm_prepare does this step ahead of time.
inline int lds_attr_once(std::atomic<uint64_t>& devs, const void* func, int lds_bytes) {
  int dev = 0;
  if (current_device(&dev) != hipSuccess) return (int)hipGetLastError();
  const uint64_t bit = (uint64_t)1 << (dev & 63);
  if (devs.load(std::memory_order_acquire) & bit) return 0;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(launch_context().stream, &st) != hipSuccess ||
      st != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return (int)hipErrorStreamCaptureUnsupported;
  }
  const hipError_t e = hipFuncSetAttribute(func, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (e != hipSuccess) return (int)e;
  devs.fetch_or(bit, std::memory_order_release);
  return 0;
}

int num_tile_variants();
const Variant* tile_variants();
int num_stream_variants();
const Variant* stream_variants();
int num_skinny_variants();
const Variant* skinny_variants();

// K ranges for `tiles` output tiles and rows of `ksteps` 128-byte steps: the largest divisor
// S of ksteps (2..16, ranges of at least 8 steps) with tiles * S <= 256, one workgroup per CU
// of a 256-CU part; 0 if there is none.  Measured on MI355X (bf16 and fp8, 32 to 128 tiles,
// 64 to 224 steps): filling the CUs once beats filling them twice by 5-15 % (32 tiles x 224
// steps: 32.3 us with 8 ranges, 37.4 with 16, 61.3 with 2; unsplit 103), and split K is ahead
// of the best unsplit kernel wherever this returns a value and rows are 8 KiB or longer.
inline int stream_split_of(int64_t tiles, int64_t ksteps, bool even_ranges = false) {
  int best = 0;
  for (int S = 2; S <= 16; ++S) {
    if (ksteps % S != 0 || ksteps / S < 8 || tiles * S > 256) continue;
    if (even_ranges && (ksteps / S) % 2 != 0) continue;
    best = S;
  }
  // ranges of 64 steps and more: twice as many, two workgroups per CU, is ahead (128 tiles x
  // 224 steps: 64.8 us with 4 ranges, 67-77 with 2)
  if (best && ksteps / best >= 64 && best * 2 <= 16 && ksteps % (best * 2) == 0 &&
      tiles * best * 2 <= 512 && !(even_ranges && (ksteps / (best * 2)) % 2 != 0))
    best *= 2;
  return best;
}

// K ranges of the split-K kernel on 256 x 128 tiles: the largest divisor up to 4 that leaves at most
// one workgroup per CU; 0 if there is none.
inline int streamr_split_of(int64_t tiles, int64_t ksteps) {
  int best = 0;
  for (int S = 2; S <= 4; ++S)
    if (ksteps % S == 0 && ksteps / S >= 8 && tiles * S <= 256) best = S;
  return best;
}

// Split-K support shared by the decode and the tile kernels (gemm_skinny.hip): the fp32
// workspace of a (device, stream), and the kernel that adds `splits` planes [M][N] of
// a.workspace in index order, applies a's scales and bias and stores a.C in `out_dtype`.
int splitk_workspace_for(size_t bytes, hipStream_t stream, float** out);
// A launcher whose K ranges another kernel stands in for: the stream's buffer is made as large as the ranges
// would have, so that a later capture finds it (never inside a capture; a failure is nobody's).
void splitk_workspace_touch(size_t bytes, hipStream_t stream);
// Held by a launcher from the lookup of the workspace to the launch of the kernel that adds it up, whoever
// owns that memory (the library's buffer of the stream, the built-in scratch, the caller): two host threads
// on one stream that share it would otherwise enqueue product, product, sum, sum.
std::mutex& splitk_order();
// Frees the workspace of a (synchronised) stream that is about to be destroyed.
void splitk_workspace_release(hipStream_t stream);
int splitk_reduce(int out_dtype, const GemmArgs& a, int splits, hipStream_t stream);

void set_error(const char* fmt, ...);
int hip_fail(hipError_t e, const char* what, const char* file, int line);

#define AG_HIP(expr)                                                   \
  do {                                                                 \
    hipError_t _e = (expr);                                            \
    if (_e != hipSuccess) return hip_fail(_e, #expr, __FILE__, __LINE__); \
  } while (0)

}  // namespace astergemm
