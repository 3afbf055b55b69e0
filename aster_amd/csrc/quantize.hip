// Operand quantisers for the fp8 and MXFP4 GEMM paths: fp32 / bf16 / f16 -> OCP e4m3 with a
// per-tensor absmax scale, and -> MXFP4 (e2m1 nibbles + one e8m0 byte per 32 elements).
//
// These produce, on the device, exactly the bytes the GEMM kernels consume (operand
// layouts of astergemm_config: row-major, e2m1 low nibble first, scales [rows, K/32]).
// The e4m3 rounding follows the converter the reference's tests hold
// (f32_to_fp8_e4m3(val, fnuz=False), test/integration/test_conversion_pack_e2e.py:91-167:
// bias 7, round to nearest even with carry into the exponent, saturation to 0x7E = 448,
// NaN and infinities to S|0x7F, signed zero), with the subnormal range rounded to nearest
// even as the hardware converter does.  The MX block format is the one the scaled MFMA
// expects (v_mfma_scale_f32_16x16x128_f8f6f4, e8m0 scale per 32 K-elements).
// Both are HBM-bound byte work: one pass over the source, for the per-tensor scale where the register files hold it and
// the launch is not captured, two elsewhere.
#include <type_traits>

#include "astergemm_internal.h"

namespace astergemm {
namespace {

// Kernels take the size of their grid as an argument: asking for it costs 256 bytes of hidden ones, and a launch
// writes its arguments to device memory line by line (PackedArgs).
typedef float f32x4 __attribute__((ext_vector_type(4)));
// Vector elements are passed by value (__float_as_uint) before their bits are taken: a bit
// cast applied to the element expression itself read element 0 for every index.

// fp32 -> e4m3 code, round to nearest even, saturating: |x| > 448 -> 0x7E, NaN / inf -> 0x7F.
// Normal range (|x| >= 2^-6): round the fp32 bit pattern to 3 fraction bits in integer
// arithmetic (a carry out of the fraction flows into the exponent) and re-bias 127 -> 7.
// Below that the codes are multiples of 2^-9: adding 2^14 makes the fp32 adder round |x| to
// that grid, ties to even, and leaves the code in the low bits of the sum.
__device__ __forceinline__ unsigned e4m3_rne_sat(float x) {
  const unsigned b = __float_as_uint(x);
  const unsigned s = (b >> 24) & 0x80u;
  const unsigned m = b & 0x7FFFFFFFu;
  unsigned code;
  if (m >= 0x3C800000u) {  // 2^-6
    code = ((m + 0x7FFFFu + ((m >> 20) & 1u)) >> 20) - ((127u - 7u) << 3);
    code = code > 0x7Eu ? 0x7Eu : code;
    code = m >= 0x7F800000u ? 0x7Fu : code;
  } else {
    code = __float_as_uint(__uint_as_float(m) + 16384.0f) & 0xFu;
  }
  return s | code;
}

// fp32 -> e2m1 code (0..15): nearest value of {0, .5, 1, 1.5, 2, 3, 4, 6}, ties to the code
// with an even index, saturation to 6, NaN -> S|7.  Same two tricks: one fraction bit kept
// for |x| >= 1, the grid of 0.5 below (2^22 has an ulp of 0.5).
__device__ __forceinline__ unsigned e2m1_rne_sat(float x) {
  const unsigned b = __float_as_uint(x);
  const unsigned s = (b >> 28) & 0x8u;
  const unsigned m = b & 0x7FFFFFFFu;
  unsigned code;
  if (m >= 0x3F800000u) {  // 1.0
    code = ((m + 0x1FFFFFu + ((m >> 22) & 1u)) >> 22) - ((127u - 1u) << 1);
    code = code > 7u ? 7u : code;
  } else {
    code = __float_as_uint(__uint_as_float(m) + 4194304.0f) & 0x3u;
  }
  return s | code;
}

__global__ void zero_u32_kernel(unsigned* p) { *p = 0u; }

// Source element types: fp32, or the 16-bit types a GEMM of this library writes (both widen
// to fp32 exactly, so quantising them equals quantising the widened values).  The kernels move the
// source in 16-byte groups of kPer elements, one group per lane and load.
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_a4 __attribute__((aligned(4)));  // fp8 destinations are 4-byte aligned
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

template <int SRC>
struct Src {
  static constexpr int kBytes = SRC == ASTERGEMM_F32 ? 4 : 2;
  static constexpr int kPer = 16 / kBytes;
};
template <int SRC>
__device__ __forceinline__ float widen(unsigned short h) {
  if constexpr (SRC == ASTERGEMM_BF16) return __uint_as_float((unsigned)h << 16);
  else return (float)__builtin_bit_cast(_Float16, h);
}
template <int SRC>
__device__ __forceinline__ float load1(const void* base, int64_t i) {
  if constexpr (SRC == ASTERGEMM_F32) return ((const float*)base)[i];
  else return widen<SRC>(((const unsigned short*)base)[i]);
}
// element e of a group as fp32
template <int SRC>
__device__ __forceinline__ float element(const i32x4& raw, int e) {
  if constexpr (SRC == ASTERGEMM_F32) return __builtin_bit_cast(f32x4, raw)[e];
  else return widen<SRC>(__builtin_bit_cast(u16x8, raw)[e]);
}

// max over |x| as unsigned bits (non-negative floats order like their bit patterns; NaNs
// compare above infinity and so survive the maximum, as they do in numpy's max), in the bits of
// the source type: two elements per packed 16-bit maximum.
template <int SRC>
struct AbsMax {
  u16x2 m2 = {0, 0};
  unsigned m = 0;
  __device__ __forceinline__ void fold(const i32x4& raw) {
    if constexpr (SRC == ASTERGEMM_F32) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned b = (unsigned)raw[e] & 0x7FFFFFFFu;
        m = b > m ? b : m;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m2 = __builtin_elementwise_max(m2, __builtin_bit_cast(u16x2, (unsigned)raw[e] & 0x7FFF7FFFu));
    }
  }
  // fp32 bits of the maximum (widening keeps the order)
  __device__ __forceinline__ unsigned bits() const {
    if constexpr (SRC == ASTERGEMM_F32) return m;
    else return __float_as_uint(widen<SRC>(m2[0] > m2[1] ? m2[0] : m2[1]));
  }
};

__device__ __forceinline__ unsigned wave_max64(unsigned m) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned o = (unsigned)__shfl_xor((int)m, off, 64);
    m = o > m ? o : m;
  }
  return m;
}
// maximum over a workgroup of NW waves, known to every thread
template <int NW>
__device__ __forceinline__ unsigned block_max(unsigned m) {
  __shared__ unsigned wave_max[NW];
  m = wave_max64(m);
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
  __syncthreads();
  m = wave_max[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = wave_max[w] > m ? wave_max[w] : m;
  return m;
}

// This thread's share of max |src[0..n)|: groups first, first + stride, ..., U loads in flight,
// and the elements behind the last whole group.  BATCHED: what is left of less than U groups is requested together
// too (one by one each waits for the one before: bf16 500 x 4096 10.8 -> 9.9 us for the two launches, 333 x 4096
// 9.7 -> 8.7); a workgroup that reads the whole of a small tensor has U groups or few (16 x 4096 3.56 against
// 3.62 us) and does without.
template <int SRC, int U, bool BATCHED>
__device__ __forceinline__ unsigned absmax_share(const void* __restrict__ src, int64_t n, int64_t first,
                                                 int64_t stride) {
  constexpr int NE = Src<SRC>::kPer;
  const i32x4* g = (const i32x4*)src;
  const int64_t ng = n / NE;
  AbsMax<SRC> am;
  int64_t i = first;
  for (; i + (U - 1) * stride < ng; i += U * stride) {
    i32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = g[i + u * stride];
#pragma unroll
    for (int u = 0; u < U; ++u) am.fold(v[u]);
  }
  if constexpr (!BATCHED) {
    for (; i < ng; i += stride) am.fold(g[i]);
  } else if (i < ng) {
    i32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = i32x4{0, 0, 0, 0};
      if (i + u * stride < ng) v[u] = g[i + u * stride];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) am.fold(v[u]);
  }
  unsigned m = am.bits();
  for (int64_t j = ng * NE + first; j < n; j += stride) {
    const unsigned b = __float_as_uint(load1<SRC>(src, j)) & 0x7FFFFFFFu;
    m = b > m ? b : m;
  }
  return m;
}

// One atomic per workgroup; the atomics of all workgroups go to one address, which the memory
// system takes one at a time (2048 workgroups: 20 us of a 30 us call; 256: 3 us).
template <int SRC>
__global__ __launch_bounds__(1024) void absmax_kernel(const void* __restrict__ src, int64_t n,
                                                      unsigned* __restrict__ out, int grid) {
  const unsigned m = block_max<16>(absmax_share<SRC, 4, false>(
      src, n, blockIdx.x * (int64_t)1024 + threadIdx.x, (int64_t)grid * 1024));
  if (threadIdx.x == 0 && m != 0) atomicMax(out, m);
}

// ---- e4m3 with one scale per tensor ----------------------------------------------------------
//
// scale = absmax / 448 in fp32, 1.0 when absmax is zero (or NaN).  For a finite tensor whose
// scale is in [2^-60, 2^60] every quotient is at most 448 in magnitude and the converter
// instruction (nearest even, like the integer form above) needs no saturation; the quotient is the
// correctly rounded one by two residual corrections with the correctly rounded reciprocal
// (Markstein's theorem: q' = RN(q + r * RN(1/s)), r = RN(x - q s), is RN(x / s) when q is within
// one unit in the last place, which the first correction ensures).  x below 2^-11 s encodes to
// zero whatever its last bits are; anything above keeps r far from the subnormal range.
struct Fp8Scale {
  float s, rcp;
  bool plain;
  __device__ __forceinline__ explicit Fp8Scale(unsigned amax_bits) {
    const float a = __uint_as_float(amax_bits);
    s = (a > 0.0f) ? a / 448.0f : 1.0f;
    rcp = 1.0f / s;
    plain = amax_bits < 0x7F800000u && s >= 0x1p-60f && s <= 0x1p60f;
  }
  __device__ __forceinline__ float quotient(float x) const {
    float q = x * rcp;
    q = fmaf(fmaf(-q, s, x), rcp, q);
    return copysignf(fmaf(fmaf(-q, s, x), rcp, q), x);  // a correction by +0 turns -0 into +0
  }
  __device__ __forceinline__ unsigned code(float x) const { return e4m3_rne_sat(x / s); }
};

// the codes of four elements, first one in the low byte
template <int SRC>
__device__ __forceinline__ unsigned fp8_codes4(const i32x4& raw, int e0, const Fp8Scale& sc) {
  if (sc.plain) {
    int w = 0;
    w = __builtin_amdgcn_cvt_pk_fp8_f32(sc.quotient(element<SRC>(raw, e0)),
                                        sc.quotient(element<SRC>(raw, e0 + 1)), w, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(sc.quotient(element<SRC>(raw, e0 + 2)),
                                        sc.quotient(element<SRC>(raw, e0 + 3)), w, true);
    return (unsigned)w;
  }
  unsigned w = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) w |= sc.code(element<SRC>(raw, e0 + e)) << (8 * e);
  return w;
}
// group i of the source to its place in dst
template <int SRC>
__device__ __forceinline__ void fp8_store_group(const i32x4& raw, int64_t i, const Fp8Scale& sc,
                                                uint8_t* __restrict__ dst) {
  if constexpr (SRC == ASTERGEMM_F32) {
    ((unsigned*)dst)[i] = fp8_codes4<SRC>(raw, 0, sc);
  } else {
    ((u32x2_a4*)dst)[i] = u32x2{fp8_codes4<SRC>(raw, 0, sc), fp8_codes4<SRC>(raw, 4, sc)};
  }
}

// Small tensors (the activations of a decode step) in one launch: every workgroup reads the whole
// source for the maximum -- from L2, all of it in flight at once -- and encodes its own part.
template <int SRC>
__global__ __launch_bounds__(1024) void quantize_fp8_small_kernel(const void* __restrict__ src, int n,
                                                                  uint8_t* __restrict__ dst,
                                                                  float* __restrict__ scale) {
  constexpr int NE = Src<SRC>::kPer;
  const int ng = n / NE;
  const int i = blockIdx.x * 1024 + threadIdx.x;
  i32x4 mine = {0, 0, 0, 0};
  if (i < ng) mine = ((const i32x4*)src)[i];
  const Fp8Scale sc(block_max<16>(absmax_share<SRC, 8, false>(src, n, threadIdx.x, 1024)));
  if (i == 0) *scale = sc.s;
  if (i < ng) fp8_store_group<SRC>(mine, i, sc, dst);
  if (blockIdx.x == 0)
    for (int j = ng * NE + threadIdx.x; j < n; j += 1024) dst[j] = (uint8_t)sc.code(load1<SRC>(src, j));
}

// Larger ones inside a capture, and on devices of fewer than kFp8Slots CUs, in two launches (elsewhere:
// quantize_fp8_once_kernel below).  The first leaves one maximum per workgroup in the first 4 * gridDim.x bytes of dst
// (written over by the codes in the end) and clears the counters of the second: *scale, and kFp8Counters of them behind
// the partial maxima.
constexpr int kFp8Counters = 16, kFp8CounterPitch = 32;  // a counter every 128 bytes of dst
constexpr int kFp8CounterBytes = kFp8Counters * kFp8CounterPitch * 4;

template <int SRC>
__global__ __launch_bounds__(256) void fp8_absmax_kernel(const void* __restrict__ src, int64_t n,
                                                         unsigned* __restrict__ partial,
                                                         unsigned* __restrict__ counter, int grid) {
  if (blockIdx.x == 0 && threadIdx.x < kFp8Counters) partial[grid + threadIdx.x * kFp8CounterPitch] = 0u;
  const unsigned m = block_max<4>(absmax_share<SRC, 8, true>(
      src, n, blockIdx.x * (int64_t)256 + threadIdx.x, (int64_t)grid * 256));
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = m;
    if (blockIdx.x == 0) *counter = 0u;
  }
}

// Every workgroup takes the maximum of the `np` partial ones, counts itself in and encodes its
// part of the tensor behind the place of the partial maxima and counters; the last one to have counted itself
// in -- everybody has read the partial maxima by then -- encodes that place and stores the scale over
// the counter there.  Nobody waits for anybody.  Atomics on one address are taken one at a time (one counter for 256
// workgroups kept the kernel 1.3 us longer than its bytes: bf16 500 x 4096 10.8 -> 8.0 us for the two launches,
// 500 x 14336 13.5 -> 12.4, 4096 x 4096 20.8 -> 19.5), so past 64 workgroups each adds to one of 16 counters, a line
// of dst apart, and the last of each of them to the one in *scale; up to 64 one counter is level or ahead (64 x 4096
// 6.1 against 6.3).
template <int SRC>
__global__ __launch_bounds__(1024) void quantize_fp8_kernel(const void* __restrict__ src, int64_t n, int np,
                                                           uint8_t* __restrict__ dst,
                                                           float* __restrict__ scale, int grid) {
  constexpr int NE = Src<SRC>::kPer, U = 4;
  __shared__ bool last;
  const i32x4* g = (const i32x4*)src;
  const bool two_levels = grid > 4 * kFp8Counters;
  const int64_t ng = n / NE, head = ((int64_t)np * 4 + (two_levels ? kFp8CounterBytes : 0)) / NE;
  const int64_t stride = (int64_t)grid * 1024;
  int64_t i = head + blockIdx.x * (int64_t)1024 + threadIdx.x;
  i32x4 v[U];
  auto fetch = [&]() {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * stride < ng) v[u] = __builtin_nontemporal_load(g + i + u * stride);
  };
  fetch();  // in flight while the maximum is found
  unsigned m = 0;
  for (int j = threadIdx.x; j < np; j += 1024) {
    const unsigned o = ((const unsigned*)dst)[j];
    m = o > m ? o : m;
  }
  const Fp8Scale sc(block_max<16>(m));  // its barrier: the workgroup's reads of dst are over
  const unsigned c = blockIdx.x % kFp8Counters;
  unsigned ticket = 0;  // looked at in the end: nobody waits for the atomic
  if (threadIdx.x == 0)
    ticket = atomicAdd(two_levels ? (unsigned*)dst + np + c * kFp8CounterPitch : (unsigned*)scale, 1u);
  while (i < ng) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * stride < ng) fp8_store_group<SRC>(v[u], i + u * stride, sc, dst);
    i += U * stride;
    fetch();
  }
  for (int64_t j = ng * NE + blockIdx.x * (int64_t)1024 + threadIdx.x; j < n; j += stride)
    dst[j] = (uint8_t)sc.code(load1<SRC>(src, j));
  if (threadIdx.x == 0) {
    const unsigned of_c = (grid - c + kFp8Counters - 1) / kFp8Counters;
    last = two_levels ? ticket == of_c - 1 && atomicAdd((unsigned*)scale, 1u) == kFp8Counters - 1
                      : ticket == (unsigned)grid - 1;
  }
  __syncthreads();
  if (!last) return;
  for (int64_t j = threadIdx.x; j < head; j += 1024) fp8_store_group<SRC>(g[j], j, sc, dst);
  if (threadIdx.x == 0) *scale = sc.s;
}

// Larger ones outside a capture, on a device of kFp8Slots CUs or more (kFp8OneLaunchUncaptured): one launch, the
// source read once and kept in registers from the maximum to the codes (a tensor of up to 128 MB is held whole; of a
// larger one 112 MB are, and the rest is read twice).  What bounds it is the way of the maxima through memory, about
// 2 us, and from 4 M elements on the bytes.  bf16, two launches -> this, back to back: 64 x 4096 7.3 -> 4.8 us,
// 500 x 8192 8.7 -> 7.4, 500 x 14336 12.1 -> 9.6, 4096 x 4096 19.5 -> 16.1, 8192 x 4096 31.4 -> 24.5, 8192 x 8192
// 70.6 -> 54.2, 8192 x 28672 240 -> 214.  Every workgroup leaves its maximum, with the tag of this launch beside it in
// the same 8 bytes, in a slot of its own and reads everybody else's (agent scope: past the L2s, which differ from XCD
// to XCD; a slot says all there is to know, so nothing has to be ordered with it).  No wait depends on another workgroup
// being there: one that has not seen all slots after `patience` looks up the missing shares in the source itself, one
// after the other from a place that each workgroup draws for itself, and leaves what it finds in the slot of the share
// (what the share's owner will store there).  So where other work holds CUs, the workgroups that run read the shares of
// those that do not less than one and a half times between them, and those that come later find every slot filled
// (beside a product of 2.8 ms on 224 CUs, two launches / this: 500 x 14336 60 / 73 us, 4096 x 4096 92 / 143, 8192 x
// 8192 290 / 550; each workgroup for itself: until the product ends).
//
// The slots are kFp8SlotSets sets that launches take in turn.  Nothing is cleared: a tag is used once in 2^33
// launches, and if two launches that run at the same time should ever share a set, what the one writes over of the
// other's is looked up in the source as well.  A captured launch would repeat its tag at every replay, so
// captures get the two launches above.
constexpr int kFp8Slots = 256, kFp8SlotSets = 64;
// Ticks of the 100 MHz counter before a workgroup gives up: 5 us, and half as long as a CU takes for its share at the
// rate of a large copy (200 bytes a tick).  With the chip to itself the last maximum is 1 to 6 us behind the first.
constexpr unsigned fp8_patience(int64_t src_bytes) { return 500 + (unsigned)(src_bytes / (kFp8Slots * 400)); }
constexpr uint64_t kFp8Tags = ((uint64_t)1 << 33) - 1;
__device__ uint64_t fp8_slots[kFp8SlotSets][kFp8Slots];

template <int SRC, int T, int U, bool MORE>
__global__ __launch_bounds__(T) void quantize_fp8_once_kernel(const void* __restrict__ src, int64_t n,
                                                              uint8_t* __restrict__ dst,
                                                              float* __restrict__ scale, int grid, int set,
                                                              uint64_t tag, unsigned patience) {
  constexpr int NE = Src<SRC>::kPer;
  static_assert(T >= kFp8Slots, "a thread per slot");
  const i32x4* g = (const i32x4*)src;
  using index = std::conditional_t<MORE, int64_t, int>;
  const index ng = (index)(n / NE), stride = grid * T, i = blockIdx.x * T + threadIdx.x;
  const int tid = threadIdx.x;
  i32x4 v[U];
  AbsMax<SRC> am;
  if constexpr (MORE) {
    constexpr int B = 6;  // in flight
    for (index k = i + U * stride; k < ng; k += B * stride) {
      i32x4 r[B];
#pragma unroll
      for (int b = 0; b < B; ++b) r[b] = g[k + b * stride < ng ? k + b * stride : ng - 1];
#pragma unroll
      for (int b = 0; b < B; ++b) am.fold(r[b]);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const index k = i + u * stride;  // past the end: the last group once more, which leaves the maximum as it is
    v[u] = __builtin_nontemporal_load(g + (k < ng ? k : ng - 1));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) am.fold(v[u]);
  unsigned m = am.bits();
  const int64_t j = (int64_t)ng * NE + tid;  // elements behind the last whole group: workgroup 0's
  if (blockIdx.x == 0 && j < n) {
    const unsigned b = __float_as_uint(load1<SRC>(src, j)) & 0x7FFFFFFFu;
    m = b > m ? b : m;
  }
  uint64_t* slots = fp8_slots[set];
  m = block_max<T / 64>(m);
  if (tid == 0)
    __hip_atomic_store(slots + blockIdx.x, tag << 31 | m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  bool seen = true;
  auto look = [&]() {
    const uint64_t s = __hip_atomic_load(slots + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (s >> 31 != tag) return;
    const unsigned o = (unsigned)s & 0x7FFFFFFFu;
    m = o > m ? o : m;
    seen = true;
  };
  if (tid < kFp8Slots) {
    const uint64_t began = wall_clock64();
    seen = tid >= grid || tid == (int)blockIdx.x;
    while (true) {
      if (!seen) look();
      if (__all(seen) || wall_clock64() - began >= patience) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (__builtin_amdgcn_readfirstlane(__syncthreads_or(!seen))) {
    __shared__ int nearest;
    unsigned mix = blockIdx.x * 0x9E3779B1u;
    while (true) {
      const int first = (int)__umulhi(mix, (unsigned)grid);  // another place for each workgroup and share
      mix = (mix ^ mix >> 15) * 0x85EBCA6Bu + 0x9E3779B1u;
      if (tid == 0) nearest = grid;
      __syncthreads();
      if (!seen) look();
      if (!seen) atomicMin(&nearest, (tid - first + grid) % grid);
      __syncthreads();
      const int d = __builtin_amdgcn_readfirstlane(nearest);
      if (d == grid) break;
      const int w = (first + d) % grid;
      constexpr int B = MORE ? 8 : U;  // in flight
      AbsMax<SRC> of_w;
      for (index k = w * T + tid; k < ng; k += B * stride) {
        i32x4 r[B];
#pragma unroll
        for (int b = 0; b < B; ++b) r[b] = g[k + b * stride < ng ? k + b * stride : ng - 1];
#pragma unroll
        for (int b = 0; b < B; ++b) of_w.fold(r[b]);
      }
      unsigned o = of_w.bits();
      if (w == 0 && j < n) {
        const unsigned e = __float_as_uint(load1<SRC>(src, j)) & 0x7FFFFFFFu;
        o = e > o ? e : o;
      }
      o = block_max<T / 64>(o);
      m = o > m ? o : m;
      if (tid == 0) __hip_atomic_store(slots + w, tag << 31 | o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (tid == w) seen = true;
    }
    // The loads above have the registers of v, which is fetched again, from places that the compiler does not know: it
    // would keep the first values or their addresses all the same.
    const i32x4* again = g;
    index at = i;
    asm volatile("" : "+s"(again), "+v"(at));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const index k = at + u * stride;
      v[u] = again[k < ng ? k : ng - 1];
    }
  }
  const Fp8Scale sc(block_max<T / 64>(m));
  if (sc.plain) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      asm volatile("" : "+v"(v[u]));  // widened here: the fp32 values of all groups do not fit
      if (i + u * stride < ng) fp8_store_group<SRC>(v[u], i + u * stride, sc, dst);
    }
  } else {
    for (index k = i; k < ng && k < i + U * stride; k += stride) fp8_store_group<SRC>(g[k], k, sc, dst);
  }
  if constexpr (MORE) {
    constexpr int B = 4;
    for (index k = i + U * stride; k < ng; k += B * stride) {
      i32x4 r[B];
#pragma unroll
      for (int b = 0; b < B; ++b)
        r[b] = __builtin_nontemporal_load(g + (k + b * stride < ng ? k + b * stride : ng - 1));
#pragma unroll
      for (int b = 0; b < B; ++b)
        if (k + b * stride < ng) fp8_store_group<SRC>(r[b], k + b * stride, sc, dst);
    }
  }
  if (blockIdx.x != 0) return;
  if (j < n) dst[j] = (uint8_t)sc.code(load1<SRC>(src, j));
  if (tid == 0) *scale = sc.s;
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for_pairs(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_pairs<N, I + 1>(f);
  }
}

// ---- MXFP4 -----------------------------------------------------------------------------------
//
// A 32-element block is kPB neighbouring lanes with one 16-byte group each: the block maximum goes
// round them by lane permutes inside the row, every lane encodes its group (the converter
// instruction divides by the power of two, rounds to nearest even and saturates) and the block's
// scale byte is known to all of them.
template <int SRC>
struct Mx4Group {
  static constexpr int kPB = 32 / Src<SRC>::kPer;  // lanes per block: 4, or 8 for fp32
  unsigned w;       // the group's nibbles: 4 bytes, or 2 for fp32
  uint8_t scale;    // the block's e8m0 byte
};
template <int SRC>
__device__ __forceinline__ Mx4Group<SRC> mx4_encode(const i32x4& raw) {
  constexpr int NE = Src<SRC>::kPer;
  AbsMax<SRC> am;
  am.fold(raw);
  unsigned mb = am.bits();
  auto with = [&](unsigned o) { mb = o > mb ? o : mb; };
  with((unsigned)__builtin_amdgcn_mov_dpp((int)mb, 0xB1, 0xF, 0xF, true));   // lane ^ 1
  with((unsigned)__builtin_amdgcn_mov_dpp((int)mb, 0x4E, 0xF, 0xF, true));   // lane ^ 2
  if constexpr (Mx4Group<SRC>::kPB == 8)
    with((unsigned)__builtin_amdgcn_mov_dpp((int)mb, 0x141, 0xF, 0xF, true));  // 7 - lane of eight
  // shared exponent = floor(log2(absmax)) - 2; an all-zero block gets exponent 0, a block
  // holding NaN / inf gets scale byte 0xFF and its elements are scaled by 2^2
  const bool bad = mb >= 0x7F800000u;
  int fl;
  if (mb == 0 || bad) fl = bad ? 0 : 2;                    // -> shared 0 (zero) / -2 (bad)
  else if (mb >= 0x00800000u) fl = (int)(mb >> 23) - 127;  // normal
  else fl = -149 + (31 - __builtin_clz(mb));               // fp32 subnormal
  int sbyte = (fl - 2) + 127;
  sbyte = sbyte < 0 ? 0 : (sbyte > 254 ? 254 : sbyte);
  Mx4Group<SRC> r;
  r.scale = bad ? (uint8_t)0xFF : (uint8_t)sbyte;
  r.w = 0;
  if (!bad && sbyte >= 1) {
    const float s = __uint_as_float((unsigned)sbyte << 23);
    static_for_pairs<NE / 2>([&](auto P) {
      constexpr int e = decltype(P)::value;
      r.w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r.w, element<SRC>(raw, 2 * e),
                                                     element<SRC>(raw, 2 * e + 1), s, e);
    });
  } else {
    const int shift = -(sbyte - 127);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      // exact scaling by a power of two in two steps (|shift| can exceed the fp32 exponent
      // range of a single factor)
      const float q = ldexpf(ldexpf(element<SRC>(raw, e), shift / 2), shift - shift / 2);
      r.w |= e2m1_rne_sat(q) << (4 * e);
    }
  }
  return r;
}
template <int SRC>
__device__ __forceinline__ void mx4_store(uint8_t* packed, int64_t group, unsigned w) {
  if constexpr (SRC == ASTERGEMM_F32) *(unsigned short*)(packed + group * 2) = (unsigned short)w;
  else *(unsigned*)(packed + group * 4) = w;
}

// Scale bytes row-major: the source as one run of blocks, U 16-byte groups in flight per lane.  What bounds it
// is a load, an encoding and a store one behind the other where the chip is not full, then the bytes; more
// groups per lane lengthen that chain.  bf16, captured and replayed, U = 4 / 2 / 1: 16 x 4096 2.44 / 2.02 /
// 1.92 us, 64 x 14336 2.5 / 2.2 / 2.0, 500 x 4096 2.8 / 2.4 / 2.2, 500 x 14336 4.7 / 4.1 / 4.1, 4096 x 4096 9.1
// / 8.0 / 8.3, 8192 x 8192 33.2 / 29.1 / 29.3 (a large copy's rate): one while 2048 workgroups hold the source,
// past that two, or four (mx4_four_groups).  CONTIG: ld == K, so block t sits at element 32 t and no (row, column)
// split is needed.
template <int SRC, bool CONTIG, int U>
__global__ __launch_bounds__(256) void quantize_mxfp4_kernel(const void* __restrict__ src,
                                                             int64_t nblocks, unsigned bpr,
                                                             int64_t ld,
                                                             uint8_t* __restrict__ packed,
                                                             uint8_t* __restrict__ scales, int grid) {
  constexpr int PB = Mx4Group<SRC>::kPB;
  const int64_t ngroups = nblocks * PB;
  const int64_t step = (int64_t)grid * 256;
  for (int64_t base = blockIdx.x * (int64_t)256 + threadIdx.x; base < ngroups; base += U * step) {
    i32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // a lane past the end repeats its first group: the lanes of a block stay together (blocks
      // are whole and both bounds are multiples of kPB), nothing of it is stored
      const int64_t t = base + u * step < ngroups ? base + u * step : base;
      int64_t off;
      if (CONTIG) {
        off = t * Src<SRC>::kPer;
      } else {
        const unsigned blk = (unsigned)(t / PB), r = blk / bpr, c = blk - r * bpr;
        off = (int64_t)r * ld + (int64_t)c * 32 + (t % PB) * Src<SRC>::kPer;
      }
      v[u] = __builtin_nontemporal_load((const i32x4*)((const uint8_t*)src + off * Src<SRC>::kBytes));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = base + u * step;
      const Mx4Group<SRC> q = mx4_encode<SRC>(v[u]);
      if (t < ngroups) {
        mx4_store<SRC>(packed, t, q.w);
        if (t % PB == 0) scales[t / PB] = q.scale;
      }
    }
  }
}

// Scale bytes in lane order (astergemm_shuffle_scales_e8m0_lanes128): a workgroup takes 128 rows x 256
// elements, whose scale bytes are one KiB of the plane, collects them in LDS and stores them as whole lines;
// written where they fall they are single bytes 256 apart (bf16 4096 x 4096 17.6 -> 10.9 us, 8192 x 8192 60.5
// -> 32.0).  T threads, which for the same reason are many: 256 / 512 / 1024, captured and replayed, 333 x 4096
// 5.5 / 4.0 / 3.6, 1024 x 4096 5.9 / 4.2 / 3.8, 1024 x 8192 7.5 / 5.7 / 5.6, 4096 x 4096 10.8 / 9.1 / 9.4, 4096
// x 14336 27.4 / 27.4 / 27.1, 8192 x 8192 32.6 / 30.2 / 31.9.  Up to 48 rows (fp32: 32) 256: rows past the end are
// loaded and encoded too, those of the whole tile with more threads (fp32 1 x 4096 3.4 / - / 4.6, 32 x 4096 3.9 / - /
// 4.8, 40 x 4096 5.3 / - / 4.8; bf16 1 x 4096 3.6 / - / 3.7, 64 x 4096 4.3 / - / 4.2).
template <int SRC, int T>
__global__ __launch_bounds__(T) void quantize_mxfp4_lanes_kernel(const void* __restrict__ src, int rows,
                                                                   unsigned bpr, int64_t ld,
                                                                   uint8_t* __restrict__ packed,
                                                                   uint8_t* __restrict__ scales) {
  constexpr int NE = Src<SRC>::kPer, PB = Mx4Group<SRC>::kPB;
  constexpr int LPR = 256 / NE;                  // lanes per row of the tile
  constexpr int RPI = T / LPR;                   // rows per trip of the workgroup
  constexpr int U = 128 / RPI < 8 ? 128 / RPI : 8;
  __shared__ __attribute__((aligned(16))) uint8_t sc[1024];
  const unsigned steps = bpr >> 3;               // 256-element steps of a row
  const unsigned grp = blockIdx.x / steps, st = blockIdx.x - grp * steps;
  const int row0 = (int)grp * 128;
  const int live = rows - row0 < 128 ? rows - row0 : 128;
  const int lr = threadIdx.x / LPR, lc = threadIdx.x % LPR;
  const int c = lc / PB;                         // block 0..7 of the step
  for (int r0 = 0; r0 < live; r0 += U * RPI) {
    i32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int r = r0 + u * RPI + lr;
      r = r < live ? r : live - 1;               // nothing of it is stored
      const int64_t off = (int64_t)(row0 + r) * ld + (int64_t)st * 256 + lc * NE;
      v[u] = __builtin_nontemporal_load((const i32x4*)((const uint8_t*)src + off * Src<SRC>::kBytes));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = r0 + u * RPI + lr;
      const Mx4Group<SRC> q = mx4_encode<SRC>(v[u]);
      if (r < live) {
        mx4_store<SRC>(packed, ((int64_t)(row0 + r) * bpr + st * 8) * PB + lc, q.w);
        // (q, i, tile, h): block c = 4 h + q, row 16 tile + i
        if (lc % PB == 0) sc[((c & 3) * 16 + (r & 15)) * 16 + (r >> 4) * 2 + (c >> 2)] = q.scale;
      }
    }
  }
  __syncthreads();
  uint8_t* dst = scales + (int64_t)blockIdx.x * 1024 + threadIdx.x * 16;
  if (threadIdx.x < 64) {
    if (live == 128) {
      *(i32x4*)dst = *(const i32x4*)(sc + threadIdx.x * 16);
    } else {                                     // bytes of rows past the end stay as they are
      for (int b = 0; b < 16; ++b)
        if ((b >> 1) * 16 + (int)(threadIdx.x & 15) < live) dst[b] = sc[threadIdx.x * 16 + b];
    }
  }
}

// Past one group per lane: four where a trip of all workgroups is more than three fifths full with them, rows with
// gaps between them, which would otherwise take two trips with half of their loads in flight (bf16, two / four,
// replayed: 3000 x 4096 of pitch 4104 8.3 / 7.25 us, 1000 x 14336 of 14344 8.7 / 8.3; fp32 4096 x 4096 of 4224 16.1 /
// 14.7; emptier: bf16 2500 x 8192 of 8200 12.3 / 13.8, fp32 700 x 28672 of 28680 19.0 / 20.5), up to four trips
// (8192 x 8192 of 8200 and 6000 x 14336 of 14344 level).  Rows without gaps only where two groups leave half of a
// second trip empty (bf16 3000 x 4096 7.4 / 7.1; 1000 x 14336 7.8 / 8.05).
bool mx4_four_groups(int64_t groups, bool contig) {
  const int64_t trip = 4 * 256 * 2048, rest = groups % trip;
  if (contig) return groups > trip * 59 / 100 && groups <= trip * 78 / 100;
  return groups <= 4 * trip && (rest == 0 || rest > trip * 3 / 5);
}

// workgroups of 256 threads for `work_items` thread-items, at most 8 per compute unit
int blocks_for(int64_t work_items) {
  const int64_t b = (work_items + 255) / 256, cap = 256 * 8;
  return (int)(b < 1 ? 1 : (b > cap ? cap : b));
}

// Up to this many elements every workgroup reads the whole source for the maximum: against two launches (bf16, back to
// back: 65536 elements 4.1 / 6.8 us, 229376 7.5 / 6.8), and against quantize_fp8_once_kernel, which captures do not
// get (with the product behind it: 65536 elements, 16x14336x4096, 14.5 / 15.0).  Between 98304 and 114688 either is
// ahead, by the product behind it (12x8192x8192, 98304, 17.4 / 16.5; 7x4096x14336, 100352, 15.5 / 16.1); past the line
// that form was at each size measured (31x14336x4096 17.7 / 16.0, 9x4096x14336 17.4 / 15.7, 16x8192x8192 17.1 / 16.6).
constexpr int64_t kFp8OneLaunch = 131072, kFp8OneLaunchUncaptured = 114688;

}  // namespace
}  // namespace astergemm

using namespace astergemm;

namespace {
bool src_ok(int dt) { return dt == ASTERGEMM_F32 || dt == ASTERGEMM_BF16 || dt == ASTERGEMM_F16; }

// Calls f with the source type as a compile-time constant.
template <class F>
void with_src(int dt, F&& f) {
  switch (dt) {
    case ASTERGEMM_F32: f(std::integral_constant<int, ASTERGEMM_F32>{}); break;
    case ASTERGEMM_BF16: f(std::integral_constant<int, ASTERGEMM_BF16>{}); break;
    default: f(std::integral_constant<int, ASTERGEMM_F16>{}); break;
  }
}

std::atomic<uint64_t> g_fp8_launches{0};  // of every source type: they share the sets

// That form for any tensor of a whole group: workgroups of 512 threads with up to 16 groups each (of 256
// or 1024: 500 x 4096 6.1 and 6.8 against 6.4 us, 500 x 14336 10.0 and 9.7 against 9.6), of 1024 where that
// does not hold the tensor (16 groups at 2^25 16-bit elements; the rest beyond is read twice).
template <int SRC>
void launch_fp8_once(const void* src, int64_t n, uint8_t* dst, float* scale, unsigned patience, hipStream_t s) {
  const uint64_t l = g_fp8_launches.fetch_add(1, std::memory_order_relaxed);
  const int64_t ng = n / Src<SRC>::kPer;
  auto go = [&](auto T, auto U, auto more) {
    const int64_t need = (ng + T * U - 1) / (T * U);
    const int grid = (int)(need < 1 ? 1 : need < kFp8Slots ? need : kFp8Slots);
    hipLaunchKernelGGL((quantize_fp8_once_kernel<SRC, T, U, more>), dim3((unsigned)grid), dim3((unsigned)T), 0, s, src,
                       n, dst, scale, grid, (int)(l % kFp8SlotSets), 1 + l % kFp8Tags, patience);
  };
  constexpr std::integral_constant<int, 512> half;
  constexpr std::integral_constant<int, 1024> full;
  constexpr std::false_type whole;
  const int64_t per = (ng + kFp8Slots * 512 - 1) / (kFp8Slots * 512);
  if (per <= 1) go(half, std::integral_constant<int, 1>{}, whole);
  else if (per <= 2) go(half, std::integral_constant<int, 2>{}, whole);
  else if (per <= 4) go(half, std::integral_constant<int, 4>{}, whole);
  else if (per <= 8) go(half, std::integral_constant<int, 8>{}, whole);
  else if (per <= 16) go(half, std::integral_constant<int, 16>{}, whole);
  else if (per <= 24) go(full, std::integral_constant<int, 12>{}, whole);
  else if (per <= 32) go(full, std::integral_constant<int, 16>{}, whole);
  else go(full, std::integral_constant<int, 14>{}, std::true_type{});
}
}  // namespace

extern "C" int astergemm_absmax(const void* dSrc, int src_dtype, int64_t n, float* dAbsmax,
                                void* stream) {
  if ((!dSrc && n > 0) || !dAbsmax || n < 0 || (((uintptr_t)dSrc) & 15) || !src_ok(src_dtype)) {
    set_error("astergemm_absmax: bad argument (source F32, BF16 or F16, 16-byte aligned)");
    return ASTERGEMM_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();  // only this call's launches are reported below
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, s, (unsigned*)dAbsmax);
  if (n > 0)
    with_src(src_dtype, [&](auto T) {
      constexpr int SRC = decltype(T)::value;
      const int64_t b = (n / Src<SRC>::kPer + 4 * 1024) / (4 * 1024);
      hipLaunchKernelGGL(absmax_kernel<SRC>, dim3((unsigned)(b < 256 ? b : 256)), dim3(1024), 0, s, dSrc,
                         n, (unsigned*)dAbsmax, (int)(b < 256 ? b : 256));
    });
  AG_HIP(hipGetLastError());
  return 0;
}

extern "C" int astergemm_quantize_fp8_tensor(const void* dSrc, int src_dtype, int64_t n,
                                             uint8_t* dDst, float* dScale, void* stream) {
  if ((!dSrc && n > 0) || (!dDst && n > 0) || !dScale || n < 0 || (((uintptr_t)dSrc) & 15) ||
      (((uintptr_t)dDst) & 3) || !src_ok(src_dtype)) {
    set_error("astergemm_quantize_fp8_tensor: bad argument (source F32, BF16 or F16, 16-byte "
              "aligned; dDst 4-byte aligned)");
    return ASTERGEMM_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();
  with_src(src_dtype, [&](auto T) {
    constexpr int SRC = decltype(T)::value, NE = Src<SRC>::kPer;
    const int64_t ng = n / NE;
    const bool once = n > kFp8OneLaunchUncaptured && device_cus() >= kFp8Slots && !is_capturing(s);
    if (n <= kFp8OneLaunch && !once) {
      const unsigned b = (unsigned)((ng + 1023) / 1024);
      hipLaunchKernelGGL(quantize_fp8_small_kernel<SRC>, dim3(b ? b : 1), dim3(1024), 0, s, dSrc, (int)n,
                         dDst, dScale);
      return;
    }
    if (once) {
      launch_fp8_once<SRC>(dSrc, n, dDst, dScale, fp8_patience(n * Src<SRC>::kBytes), s);
      return;
    }
    // one partial maximum per workgroup, a multiple of 32 of them (128 bytes of dst), 1024 at most
    int64_t np = ((ng + 4 * 256 - 1) / (4 * 256) + 31) & ~(int64_t)31;
    if (np > 1024) np = 1024;
    hipLaunchKernelGGL(fp8_absmax_kernel<SRC>, dim3((unsigned)np), dim3(256), 0, s, dSrc, n,
                       (unsigned*)dDst, (unsigned*)dScale, (int)np);
    // a workgroup per CU, two from 2^25 elements on (bf16, one / two: 4096 x 4096 19.5 / 20.4 us, 4096 x 14336
    // 57.5 / 55.7)
    const int64_t b = (ng + 1023) / 1024, cap = n < ((int64_t)1 << 25) ? 256 : 512;
    hipLaunchKernelGGL(quantize_fp8_kernel<SRC>, dim3((unsigned)(b < cap ? b : cap)), dim3(1024), 0, s,
                       dSrc, n, (int)np, dDst, dScale, (int)(b < cap ? b : cap));
  });
  AG_HIP(hipGetLastError());
  return 0;
}

extern "C" int astergemm_diag_quantize_fp8(const void* dSrc, int src_dtype, int64_t n, uint8_t* dDst, float* dScale,
                                           unsigned patience, void* stream) {
  if (!dSrc || !dDst || !dScale || n <= kFp8OneLaunchUncaptured || (((uintptr_t)dSrc) & 15) || (((uintptr_t)dDst) & 3) ||
      !src_ok(src_dtype) || is_capturing((hipStream_t)stream)) {
    set_error("astergemm_diag_quantize_fp8: bad argument (more than %lld elements, no capture, otherwise as for "
              "astergemm_quantize_fp8_tensor)", (long long)kFp8OneLaunchUncaptured);
    return ASTERGEMM_EINVAL;
  }
  (void)hipGetLastError();
  with_src(src_dtype, [&](auto T) {
    launch_fp8_once<decltype(T)::value>(dSrc, n, dDst, dScale, patience, (hipStream_t)stream);
  });
  AG_HIP(hipGetLastError());
  return 0;
}

extern "C" int astergemm_quantize_mxfp4_ex(const void* dSrc, int src_dtype, int64_t rows, int64_t K,
                                           int64_t ld_src, uint8_t* dPacked, uint8_t* dScales,
                                           int scales_layout, void* stream) {
  if (ld_src == 0) ld_src = K;
  const bool lanes = scales_layout == ASTERGEMM_MX_LANES128;
  if (rows < 0 || K < 0 || K % 32 != 0 || ld_src < K || ld_src % 8 != 0 || !src_ok(src_dtype) ||
      ((rows > 0 && K > 0) && (!dSrc || !dPacked || !dScales)) || (((uintptr_t)dSrc) & 15) ||
      (((uintptr_t)dPacked) & 15) || (!lanes && scales_layout != ASTERGEMM_MX_ROWS) ||
      (lanes && (K % 256 != 0 || (((uintptr_t)dScales) & 15)))) {
    set_error("astergemm_quantize_mxfp4: need a source of F32, BF16 or F16, K %% 32 == 0, "
              "ld_src >= K, ld_src %% 8 == 0, dSrc and dPacked 16-byte aligned; scales in lane "
              "order: K %% 256 == 0 and dScales 16-byte aligned");
    return ASTERGEMM_EINVAL;
  }
  if (rows == 0 || K == 0) return 0;
  const int64_t nblocks = rows * (K / 32);
  if (nblocks >= (int64_t)1 << 31) {
    set_error("astergemm_quantize_mxfp4: more than 2^31 blocks");
    return ASTERGEMM_EINVAL;
  }
  (void)hipGetLastError();
  with_src(src_dtype, [&](auto T) {
    constexpr int SRC = decltype(T)::value;
    const unsigned bpr = (unsigned)(K / 32);
    hipStream_t st = (hipStream_t)stream;
    if (lanes) {
      const unsigned grid = (unsigned)((rows + 127) / 128 * (K / 256));
      auto go = [&](auto kern, int threads) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), 0, st, dSrc, (int)rows, bpr, ld_src, dPacked, dScales);
      };
      if (rows <= (SRC == ASTERGEMM_F32 ? 32 : 48)) go(quantize_mxfp4_lanes_kernel<SRC, 256>, 256);
      else if (rows * K <= (int64_t)1 << 22) go(quantize_mxfp4_lanes_kernel<SRC, 1024>, 1024);
      else go(quantize_mxfp4_lanes_kernel<SRC, 512>, 512);
      return;
    }
    const int64_t groups = nblocks * Mx4Group<SRC>::kPB;
    auto go = [&](auto kern, int per) {
      const dim3 grid(blocks_for((groups + per - 1) / per));
      hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, dSrc, nblocks, bpr, ld_src, dPacked, dScales, (int)grid.x);
    };
    const bool contig = ld_src == K;
    if (groups <= (int64_t)2048 * 256) {
      if (contig) go(quantize_mxfp4_kernel<SRC, true, 1>, 1);
      else go(quantize_mxfp4_kernel<SRC, false, 1>, 1);
    } else if (mx4_four_groups(groups, contig)) {
      if (contig) go(quantize_mxfp4_kernel<SRC, true, 4>, 4);
      else go(quantize_mxfp4_kernel<SRC, false, 4>, 4);
    } else {
      if (contig) go(quantize_mxfp4_kernel<SRC, true, 2>, 2);
      else go(quantize_mxfp4_kernel<SRC, false, 2>, 2);
    }
  });
  AG_HIP(hipGetLastError());
  return 0;
}

extern "C" int astergemm_quantize_mxfp4(const void* dSrc, int src_dtype, int64_t rows, int64_t K,
                                        int64_t ld_src, uint8_t* dPacked, uint8_t* dScales,
                                        void* stream) {
  return astergemm_quantize_mxfp4_ex(dSrc, src_dtype, rows, K, ld_src, dPacked, dScales,
                                     ASTERGEMM_MX_ROWS, stream);
}

// ---- pre-shuffle of weights on the device ----------------------------------------------------
//
// Every pre-shuffled layout is a permutation of fixed-size units inside blocks of 16 (64) rows:
// thread t writes destination unit t, fetched from where the host functions of the same name
// take it.  MODE 0: 16-bit, the reference's shuffle_weight order (units of 8 bytes);
// 1: 16-bit, K8 order (16 bytes); 2: byte rows in step order (16 bytes); 3: e8m0 plane in
// step order (8 bytes); 4: e8m0 plane in lane order (1 byte).
namespace astergemm {
namespace {

template <int MODE>
__global__ __launch_bounds__(256) void preshuffle_kernel(const uint8_t* __restrict__ src,
                                                         uint8_t* __restrict__ dst, int64_t units,
                                                         int64_t rb) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= units) return;
  if constexpr (MODE == 0) {
    // dst (nb, kb, g, n, kh) <- src (nb, n, kb, kh, g), units of 4 elements
    const int64_t kblocks = rb / 64;
    const int kh = (int)(t & 1), n = (int)((t >> 1) & 15), g = (int)((t >> 5) & 3);
    const int64_t kb = (t >> 7) % kblocks, nb = (t >> 7) / kblocks;
    *(uint2*)(dst + t * 8) = *(const uint2*)(src + (nb * 16 + n) * rb + kb * 64 + kh * 32 + g * 8);
  } else if constexpr (MODE == 1) {
    // dst (nb, kb, g, n) <- src (nb, n, kb, g), units of 8 elements
    const int64_t kblocks = rb / 64;
    const int n = (int)(t & 15), g = (int)((t >> 4) & 3);
    const int64_t kb = (t >> 6) % kblocks, nb = (t >> 6) / kblocks;
    *(uint4*)(dst + t * 16) = *(const uint4*)(src + (nb * 16 + n) * rb + kb * 64 + g * 16);
  } else if constexpr (MODE == 2) {
    // dst (nb, step, u, q, n) <- src (nb, n, step, 4u + q), units of 16 bytes
    const int64_t steps = rb / 128;
    const int n = (int)(t & 15), q = (int)((t >> 4) & 3), u = (int)((t >> 6) & 1);
    const int64_t st = (t >> 7) % steps, nb = (t >> 7) / steps;
    *(uint4*)(dst + t * 16) = *(const uint4*)(src + (nb * 16 + n) * rb + st * 128 + (4 * u + q) * 16);
  } else if constexpr (MODE == 3) {
    // dst (nb, step, n) <- src (nb, n, step), units of 8 bytes; rb = K / 32 bytes
    const int64_t steps = rb / 8;
    const int n = (int)(t & 15);
    const int64_t st = (t >> 4) % steps, nb = (t >> 4) / steps;
    *(uint2*)(dst + t * 8) = *(const uint2*)(src + (nb * 16 + n) * rb + st * 8);
  } else if constexpr (MODE == 4) {
    // dst (nb4, step, q, i, tile, h) <- src (nb4, tile, i, step, 4h + q), bytes; rb = K / 32 bytes
    const int64_t steps = rb / 8;
    const int h = (int)(t & 1), tl = (int)((t >> 1) & 3), i = (int)((t >> 3) & 15), q = (int)((t >> 7) & 3);
    const int64_t st = (t >> 9) % steps, nb4 = (t >> 9) / steps;
    dst[t] = src[(nb4 * 64 + tl * 16 + i) * rb + st * 8 + 4 * h + q];
  }
}

// A's plane into lane order in groups of 128 rows: dst (g, step, q, i, tile, h) <- src (g, tile, i,
// step, 4h + q), one byte per thread; rows past `rows` get 127 (scale 1)
__global__ __launch_bounds__(256) void preshuffle_scales_a_kernel(const uint8_t* __restrict__ src,
                                                                  uint8_t* __restrict__ dst,
                                                                  int64_t units, int64_t rb, int64_t rows) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= units) return;
  const int64_t steps = rb / 8;
  const int h = (int)(t & 1), tl = (int)((t >> 1) & 7), i = (int)((t >> 4) & 15), q = (int)((t >> 8) & 3);
  const int64_t st = (t >> 10) % steps, g = (t >> 10) / steps;
  const int64_t row = g * 128 + tl * 16 + i;
  dst[t] = row < rows ? src[row * rb + st * 8 + 4 * h + q] : (uint8_t)127;
}

template <int MODE>
int preshuffle_launch(const void* src, void* dst, int64_t bytes, int unit, int64_t row_bytes_,
                      hipStream_t s) {
  const int64_t units = bytes / unit;
  if (units == 0) return 0;
  if ((units + 255) / 256 >= (int64_t)1 << 31) {
    set_error("astergemm_preshuffle: matrix too large");
    return ASTERGEMM_EINVAL;
  }
  (void)hipGetLastError();
  hipLaunchKernelGGL(preshuffle_kernel<MODE>, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s,
                     (const uint8_t*)src, (uint8_t*)dst, units, row_bytes_);
  AG_HIP(hipGetLastError());
  return 0;
}

}  // namespace
}  // namespace astergemm

extern "C" int astergemm_preshuffle(int dtype_ab, int operand_path, int64_t N, int64_t K,
                                    const void* dSrc, void* dDst, const uint8_t* dMxSrc,
                                    uint8_t* dMxDst, void* stream) {
  using namespace astergemm;
  const bool is16 = dtype_ab == ASTERGEMM_F16 || dtype_ab == ASTERGEMM_BF16;
  const bool fp4 = dtype_ab == ASTERGEMM_MXFP4;
  if (!is16 && !fp4 && dtype_ab != ASTERGEMM_FP8_E4M3) {
    set_error("astergemm_preshuffle: dtype_ab must be F16, BF16, FP8_E4M3 or MXFP4");
    return ASTERGEMM_EINVAL;
  }
  // DIRECT_AB: one call per operand (A [M, K] or B [N, K]), both in DIRECT_B's 16-bit order
  if (operand_path == ASTERGEMM_OPERAND_DIRECT_AB && is16) operand_path = ASTERGEMM_OPERAND_DIRECT_B;
  if (operand_path != ASTERGEMM_OPERAND_DIRECT_B && operand_path != ASTERGEMM_OPERAND_DIRECT_B_K8) {
    set_error("astergemm_preshuffle: operand_path must be DIRECT_B, DIRECT_B_K8 or (16-bit "
              "operands) DIRECT_AB");
    return ASTERGEMM_EINVAL;
  }
  const bool k8 = operand_path == ASTERGEMM_OPERAND_DIRECT_B_K8;
  const int64_t rb = row_bytes(dtype_ab, K);
  const int64_t rows_mod = (fp4 && k8) ? 64 : 16;
  if (N < 0 || K < 0 || N % rows_mod != 0 || (is16 ? K % 32 != 0 : rb % 128 != 0) ||
      (N > 0 && K > 0 && (!dSrc || !dDst || dSrc == dDst)) || ((((uintptr_t)dSrc) | ((uintptr_t)dDst)) & 15) ||
      (fp4 && N > 0 && K > 0 && (!dMxSrc || !dMxDst || dMxSrc == dMxDst ||
                                 ((((uintptr_t)dMxSrc) | ((uintptr_t)dMxDst)) & 7)))) {
    set_error("astergemm_preshuffle: need N %% %d == 0, rows of whole %s, distinct 16-byte aligned "
              "source and destination (MXFP4: and distinct 8-byte aligned scale planes)",
              (int)rows_mod, is16 ? "32-element blocks" : "128-byte steps");
    return ASTERGEMM_EINVAL;
  }
  if (N == 0 || K == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  int rc;
  if (is16) rc = k8 ? preshuffle_launch<1>(dSrc, dDst, N * rb, 16, rb, s)
                    : preshuffle_launch<0>(dSrc, dDst, N * rb, 8, rb, s);
  else rc = preshuffle_launch<2>(dSrc, dDst, N * rb, 16, rb, s);
  if (rc != 0 || !fp4) return rc;
  return k8 ? preshuffle_launch<4>(dMxSrc, dMxDst, N * (K / 32), 1, K / 32, s)
            : preshuffle_launch<3>(dMxSrc, dMxDst, N * (K / 32), 8, K / 32, s);
}

extern "C" int astergemm_preshuffle_scales_a(int64_t M, int64_t K, const uint8_t* dMxSrc,
                                             uint8_t* dMxDst, void* stream) {
  using namespace astergemm;
  if (M < 0 || K < 0 || K % 256 != 0 || (M > 0 && K > 0 && (!dMxSrc || !dMxDst || dMxSrc == dMxDst)) ||
      ((((uintptr_t)dMxSrc) | ((uintptr_t)dMxDst)) & 15)) {
    set_error("astergemm_preshuffle_scales_a: need K %% 256 == 0 and distinct 16-byte aligned planes");
    return ASTERGEMM_EINVAL;
  }
  const int64_t units = astergemm_mx_lanes128_bytes(M, K);
  if (units == 0) return 0;
  if ((units + 255) / 256 >= (int64_t)1 << 31) {
    set_error("astergemm_preshuffle_scales_a: plane too large");
    return ASTERGEMM_EINVAL;
  }
  (void)hipGetLastError();
  hipLaunchKernelGGL(preshuffle_scales_a_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, dMxSrc, dMxDst, units, K / 32, M);
  AG_HIP(hipGetLastError());
  return 0;
}
