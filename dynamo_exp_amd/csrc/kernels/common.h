// Shared helpers for the gfx950 (CDNA4, MI355X) kernels.
//
// Conventions used by every kernel in this directory:
//   * wave64 everywhere (never 32-lane warp idioms);
//   * bf16 activations/KV, fp32 accumulation;
//   * global loads/stores are 16-byte vectors (dwordx4) wherever the layout
//     allows (guide G13: scalar bf16 loads cost 2-2.5x);
//   * launchers take a hipStream_t and never allocate / synchronise, so every
//     launch is hipGraph-capturable.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define DX_WAVE 64

typedef uint16_t bf16_t;  // raw bf16 bits
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

struct __attribute__((aligned(16))) u16x8 {
  uint32_t w[4];
};

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
  return __uint_as_float(((uint32_t)v) << 16);
}
// low / high bf16 of a packed u32 -> f32 (one VALU op each)
__device__ __forceinline__ float bf16lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// f32 -> bf16, round-to-nearest-even; the plain cast lowers to v_cvt_pk_bf16_f32
// on gfx950 which keeps NaNs NaN (microarch "Correctness boundaries").
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  __bf16 b = (__bf16)f;
  return __builtin_bit_cast(bf16_t, b);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  // one v_cvt_pk_bf16_f32 for the pair (RNE)
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// raw v_exp_f32 (2^x) without the denormal range fix-up exp2f() adds; inputs
// here are <= 0 softmax exponents where flushing tiny results to 0 is exact
// enough (|err| < 2^-126)
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- tiles on their way to LDS by DMA, and fragments read transposed from them
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
// (a function of its own: the compiler then knows that the read is of what p names, and does not wait in front of it for the
// DMA of the next tile, which goes to the other buffer)
__device__ __forceinline__ i16x4 read_tr16(const lds_i16x4* __restrict__ p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p);
}
// 16 bytes a lane from `off` bytes behind `from` to LDS; zeros from `bytes` on.  (global_load_lds would count as an LDS access
// as well, and every wait for an LDS read become one for all of them.)  NT 2: a nontemporal read.
template <int NT = 0>
__device__ __forceinline__ void dma16(const void* from, int bytes, int off, lds_void* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)from, 0, bytes, 0x00020000), to, 16, off, 0, 0, NT);
}
// every wave is done with a tile, and the DMA of the next has landed
__device__ __forceinline__ void landed() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
}

// over a wave, every lane with the lane 32, 16, 8, 4, 2 and 1 from it, by exchanges in registers (all lanes on): the six LDS
// permutes of __shfl_xor took some 700 cycles, a part of every small kernel's time (a launch of 3 to 5 us)
template <int CTRL> __device__ __forceinline__ float row_dpp(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), CTRL, 0xf, 0xf, false));
}
template <typename F> __device__ __forceinline__ float over_halves(float v, F f) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename F> __device__ __forceinline__ float over_row_pairs(float v, F f) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_max(float v) {
  return over_halves(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float halves_sum(float v) {
  return over_halves(v, [](float a, float b) { return a + b; });
}
// (N: aligned groups of so many lanes, 16 or more)
template <int N, typename F> __device__ __forceinline__ float over_lanes(float v, F f) {
  static_assert(N == 16 || N == 32 || N == 64, "whole rows of lanes");
  if constexpr (N == 64) v = over_halves(v, f);
  if constexpr (N >= 32) v = over_row_pairs(v, f);
  v = f(v, row_dpp<0x128>(v));  // row_ror:8
  v = f(v, row_dpp<0x124>(v));  // row_ror:4 (4 or 12 lanes on, which hold the same by now)
  v = f(v, row_dpp<0x4E>(v));   // quad_perm
  return f(v, row_dpp<0xB1>(v));
}
__device__ __forceinline__ float wave_reduce_sum(float v) {
  return over_lanes<64>(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_reduce_max(float v) {
  return over_lanes<64>(v, [](float a, float b) { return fmaxf(a, b); });
}

// Block-wide sum for blockDim.x <= 1024 (16 waves). `red` must hold >= 16 floats.
__device__ __forceinline__ float block_reduce_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_reduce_sum(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float r = (threadIdx.x < (unsigned)nw) ? red[threadIdx.x] : 0.f;
  if (wid == 0) r = wave_reduce_sum(r);
  if (threadIdx.x == 0) red[0] = r;
  __syncthreads();
  r = red[0];
  __syncthreads();
  return r;
}

#define DX_CHECK_LAUNCH() (void)hipGetLastError()
