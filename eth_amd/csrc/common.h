// Shared helpers for the eth_amd HIP kernels (gfx950 / CDNA4 only).
//
// Every exported entry point returns an int status (ETH_OK on success) and
// records a message retrievable through eth_last_error().  Kernels are
// launched on the caller's stream; nothing here allocates device memory on a
// hot path.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string>

#include "../../include/eth_amd.h"

namespace eth {

void set_error(const char* fmt, ...);

#define ETH_CHECK_ARG(cond, ...)              \
  do {                                        \
    if (!(cond)) {                            \
      ::eth::set_error(__VA_ARGS__);          \
      return ETH_ERR_INVALID;                 \
    }                                         \
  } while (0)

#define ETH_CHECK_LAUNCH(what)                                              \
  do {                                                                      \
    hipError_t _e = hipGetLastError();                                      \
    if (_e != hipSuccess) {                                                 \
      ::eth::set_error("%s: launch failed: %s", what, hipGetErrorString(_e)); \
      return ETH_ERR_HIP;                                                   \
    }                                                                       \
  } while (0)

typedef uint16_t bf16_t;
typedef _Float16 f16_t;

// float -> bfloat16, round to nearest even (v_cvt_pk_bf16_f32; denormals are
// kept, NaN stays NaN).
__device__ __forceinline__ bf16_t f2bf(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
// two floats -> packed bf16 pair (lo in bits 0-15), one conversion instruction
typedef float eth_f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 eth_bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2bf_pair(float lo, float hi) {
  const eth_f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, eth_bf16x2_t));
}
// two floats -> packed fp16 pair (lo in bits 0-15), each rounded to nearest
// even from its fp32 value.  The empty asm pins the fp32 values in
// registers: otherwise the compiler may fold the multiply that produced them
// into a mixed-precision fma with a +0 addend (v_fma_mixlo_f16), which
// rounds the exact product once and turns a -0 product into +0.
typedef _Float16 eth_f16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2h_pair(float lo, float hi) {
  eth_f32x2_t v = {lo, hi};
  asm volatile("" : "+v"(v));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, eth_f16x2_t));
}
// the same rounding for one value, returned as fp32
__device__ __forceinline__ float round_to_f16(float f) {
  asm volatile("" : "+v"(f));
  return (float)(_Float16)f;
}
__device__ __forceinline__ float bf2f(bf16_t h) {
  return __uint_as_float(((uint32_t)h) << 16);
}
// float -> fp16 bits, rounded to nearest even from the fp32 value (pinned
// in a register for the reason given at f2h_pair)
__device__ __forceinline__ uint16_t f2h_bits(float f) {
  asm volatile("" : "+v"(f));
  return __builtin_bit_cast(uint16_t, (f16_t)f);
}
__device__ __forceinline__ float h2f_bits(uint16_t b) {
  f16_t h = *reinterpret_cast<f16_t*>(&b);
  return (float)h;
}

// Load/store one element of a tensor whose dtype is chosen at run time.
__device__ __forceinline__ float load_elem(const void* p, int64_t i, int dtype) {
  if (dtype == ETH_F32) return reinterpret_cast<const float*>(p)[i];
  uint16_t b = reinterpret_cast<const uint16_t*>(p)[i];
  return dtype == ETH_BF16 ? bf2f(b) : h2f_bits(b);
}
__device__ __forceinline__ void store_elem(void* p, int64_t i, int dtype, float v) {
  if (dtype == ETH_F32) {
    reinterpret_cast<float*>(p)[i] = v;
  } else {
    reinterpret_cast<uint16_t*>(p)[i] = dtype == ETH_BF16 ? f2bf(v) : f2h_bits(v);
  }
}

// Sum over the wavefront, in every lane.  Called with all 64 lanes active.
// Pairs 32, 16, 8, 4, 2 and 1 lanes apart are added in that order, all within
// the VALU: the two halves and the pairs of rows by lane swaps, then
// data-parallel-primitive moves inside a row of 16 (a rotation by 8 or 4 meets
// the same pairs as the exchange, whose sums repeat with that period).  The
// same tree by lane exchanges goes through LDS six times, which a row's
// LayerNorm waits for twice in a chain (LayerNorm backward of [8192, 2048]
// 32.4 -> 30.7 us, of [4096, 5120] 46.5 -> 43.8 us).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  // each swap turns (v, v) into the two addends of every lane
  u32x2 p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p.x) + __uint_as_float(p.y);
  p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p.x) + __uint_as_float(p.y);
  v = dpp_add<0x128>(v);     // row_ror:8
  v = dpp_add<0x124>(v);     // row_ror:4
  v = dpp_add<0x4e>(v);      // quad_perm:[2,3,0,1]
  return dpp_add<0xb1>(v);   // quad_perm:[1,0,3,2]
}

// Block-wide sum for blockDim.x == NT (multiple of 64).  `red` must hold
// NT/64 floats of shared memory.  Every thread receives the total.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

// out[c] (+)= sum_g part[g*ld + c] for c < cols (cols % 4 == 0, part and ld
// 16-byte aligned): 64 columns per workgroup, one round trip of float4 loads
// per lane, fixed summation order (deterministic).  With gridDim.y == 2 the
// second slab (columns [cols, 2 cols) of each partial row) goes to out1.
__global__ void reduce_partials_kernel(const float* __restrict__ part, int groups, int cols, int64_t ld,
                                       float* __restrict__ out0, float* __restrict__ out1, int accumulate);
inline dim3 reduce_partials_grid(int cols, int slabs = 1) { return dim3((cols + 63) / 64, slabs); }
constexpr int kReducePartialsThreads = 256;

// 32-bit mix of (seed, index): element `idx` is kept when
//   z = seed + G (idx + 1), z = (z ^ z>>30) C1, z = (z ^ z>>27) C2,
//   (z ^ z>>31) >> 32  >=  p * 2^32
// Shared by every kernel that applies or replays a dropout mask, so they all
// draw the same one.  The 64-bit products are most of such a kernel's VALU
// time (a 32-bit multiply issues at a quarter of the rate), so eight
// consecutive elements share the first, of the last only the upper half is
// formed, and nothing branches per element: dropout's backward over
// [8192, 2048] 15.7 -> 13.9 us, bias-dropout-add + LayerNorm with p = 0.1 26.7
// -> 24.0 us (without a mask 21.3).
constexpr uint64_t kMixG = 0x9E3779B97F4A7C15ull, kMixC1 = 0xBF58476D1CE4E5B9ull, kMixC2 = 0x94D049BB133111EBull;
__device__ __forceinline__ uint32_t mix_u32(uint64_t z) {
  z = (z ^ (z >> 30)) * kMixC1;
  z ^= z >> 27;
  const uint32_t lo = (uint32_t)z, hi = (uint32_t)(z >> 32);
  const uint32_t h = __umulhi(lo, (uint32_t)kMixC2) + lo * (uint32_t)(kMixC2 >> 32) + hi * (uint32_t)kMixC2;
  return h ^ (h >> 31);
}
// v[j] of elements idx .. idx + 7: scaled where kept, else 0
__device__ __forceinline__ void dropout8(float (&v)[8], uint64_t seed, uint64_t idx, uint32_t thresh, float scale) {
  const uint64_t z = seed + kMixG * (idx + 1);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = mix_u32(z + kMixG * (uint64_t)j) >= thresh ? v[j] * scale : 0.f;
}

// Host side of the dropout mask: keep threshold (0 when p == 0, no mask) and
// the 1/(1-p) scale of kept elements.
inline void dropout_params(float p, uint32_t& thresh, float& scale) {
  thresh = p <= 0.f ? 0u : (uint32_t)fmin(4294967295.0, (double)p * 4294967296.0);
  scale = p <= 0.f ? 1.f : (float)(1.0 / (1.0 - (double)p));
}

inline int dtype_size(int dtype) { return dtype == ETH_F32 ? 4 : 2; }
inline bool valid_dtype(int dtype) {
  return dtype == ETH_F32 || dtype == ETH_F16 || dtype == ETH_BF16;
}

}  // namespace eth
