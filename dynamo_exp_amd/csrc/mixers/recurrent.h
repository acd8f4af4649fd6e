// Shared by the kernels with per-sequence state: element access, activations,
// sums over lane groups by DPP exchanges, 16-byte vector access, dispatch over
// the activation element.
#pragma once
#include <climits>

#include "../kernels/common.h"

namespace {

constexpr int kRows = 16;  // state rows per thread
constexpr int kTok = 8;    // tokens per staged block

template <typename T> __device__ __forceinline__ float ldf(const T* p, int64_t i);
template <> __device__ __forceinline__ float ldf<bf16_t>(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
template <> __device__ __forceinline__ float ldf<float>(const float* p, int64_t i) { return p[i]; }
template <typename T> __device__ __forceinline__ void stf(T* p, int64_t i, float v);
template <> __device__ __forceinline__ void stf<bf16_t>(bf16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }
template <> __device__ __forceinline__ void stf<float>(float* p, int64_t i, float v) { p[i] = v; }

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + expf(-z)); }

// the same from the hardware's exp2 and reciprocal (relative error a few 1e-7): per-element gates of wide rows
__device__ __forceinline__ float fast_sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.f + fast_exp2(z * -1.4426950408889634f));
}

// Four neighbours of a state matrix, read and written once a step.  ONCE: nontemporally, for a decode step whose states
// no cache could hold for the next one anyway (state_once).
template <bool ONCE> __device__ __forceinline__ f32x4 load_state(const float* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
  else return *reinterpret_cast<const f32x4*>(p);
}
template <bool ONCE> __device__ __forceinline__ void store_state(float* p, f32x4 v) {
  if constexpr (ONCE) __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
  else *reinterpret_cast<f32x4*>(p) = v;
}
// One layer's repeated step, kept / not, us: state-space duality, 128 heads, 64 / 88 / 128 MB 33.8 / 39.7, 45.2 / 49.3, 67.7 / 59.8;
// delta rule, 32 heads, 64 / 88 / 128 MB 29.2 / 33.4, 42.2 / 41.9, 66.5 / 55.2; gated linear attention 72 / 96 / 128 MB 39.1 / 40.2,
// 52.3 / 49.0, 69.5 / 57.4.  Behind the states of other layers nothing of this one's is left when its next step comes, and
// the line lies lower.  Eight layers with their other launches, a layer, kept / not, us: state-space duality 46 / 67 / 101 MB
// 30.8 / 27.1, 40.7 / 36.1, 53.7 / 46.9; delta rule 46 / 84 / 126 MB 29.4 / 22.7, 43.0 / 36.2, 59.9 / 50.5; gated linear attention
// 50 / 84 MB 30.4 / 26.5, 44.6 / 39.9; 24 layers of the smallest the same.  (Only read or only written nontemporally: nothing.)
inline bool state_once(int n_seq, int H, int dk, int dv, int layers) {
  return (int64_t)n_seq * H * dk * dv * 4 >= (layers > 1 ? 44 : 128) << 20;
}

template <int CTRL> __device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
// sum over the R lanes of an aligned lane group (R <= 16), the result in every lane of the group:
// neighbours within a quad, the other pair of the quad, the other quad of a half row (half-row
// mirror: the quads already hold one value each), the other half of a row of 16 (row mirror)
template <int R> __device__ __forceinline__ float group_sum(float v) {
  if constexpr (R >= 2) v += dpp_f<0xB1>(v);
  if constexpr (R >= 4) v += dpp_f<0x4E>(v);
  if constexpr (R >= 8) v += dpp_f<0x141>(v);
  if constexpr (R >= 16) v += dpp_f<0x140>(v);
  return v;
}

// The sequence of a workgroup that is the k-th to go out: the k-th longest of those with `least` rows and more, so that the
// longest does not start when a short one's place is free.  Where more than `most` have as many rows, they go as they
// come: they even out by themselves, and every wave pays for comparing their lengths (some ten instructions a length, in the
// workgroup of a decode row more than its work).  Behind them, if asked for, the `others`, as they come.  n = 0: there is none.  The lanes' loads are all asked for at once:
// where a launch is short, one that waits for another is a hundredth of it.
struct SeqRows {
  int r0, n, slot, s;
};
template <bool ALL>  // all sequences count, whatever their length
__device__ __forceinline__ SeqRows by_length(const int* seq_rows, const int* slots, int n_seq, int k, int least, int most,
                                             bool others = false) {
  if (n_seq > (ALL ? most : 64)) return SeqRows{seq_rows[k], seq_rows[k + 1] - seq_rows[k], slots[k], k};
  const int lane = threadIdx.x & 63, at = min(lane, n_seq - 1);
  const int r0 = seq_rows[at], end = seq_rows[at + 1], slot = slots[at];
  const int len = lane < n_seq ? end - r0 : INT_MIN;
  const uint64_t any = __builtin_amdgcn_ballot_w64(len >= least);
  const int count = __builtin_popcountll(any);
  if (count <= k) {  // behind them the others as they come
    const uint64_t rest = ~any & (n_seq == 64 ? ~0ull : (1ull << n_seq) - 1);
    if (ALL || !others || k - count >= __builtin_popcountll(rest)) return SeqRows{0, 0, 0, 0};
    const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(rest >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)rest, 0));
    const int s = __builtin_ctzll(__builtin_amdgcn_ballot_w64(before == k - count) & rest);
    return SeqRows{__builtin_amdgcn_readlane(r0, s), __builtin_amdgcn_readlane(len, s), __builtin_amdgcn_readlane(slot, s), s};
  }
  int rank = 0;
  if (!ALL && count > most) {
    rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0));
  } else {
    for (uint64_t left = any; left; left &= left - 1) {
      const int j = __builtin_ctzll(left), other = __builtin_amdgcn_readlane(len, j);
      rank += other > len || (other == len && j < lane);
    }
  }
  const int s = __builtin_ctzll(__builtin_amdgcn_ballot_w64(rank == k) & any);
  return SeqRows{__builtin_amdgcn_readlane(r0, s), __builtin_amdgcn_readlane(len, s), __builtin_amdgcn_readlane(slot, s), s};
}

// Barrier for what the waves exchange in LDS: __syncthreads() would also wait for every load of the next chunk and
// for the results' way to memory.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename T, int V> struct VecIO;
template <> struct VecIO<bf16_t, 8> {
  __device__ static __forceinline__ void ld(const bf16_t* p, float* o) {
    const u16x8 a = *reinterpret_cast<const u16x8*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[2 * i] = bf16lo(a.w[i]), o[2 * i + 1] = bf16hi(a.w[i]);
  }
  __device__ static __forceinline__ void st(bf16_t* p, const float* v) {
    u16x8 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a.w[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    *reinterpret_cast<u16x8*>(p) = a;
  }
};
// 16 raw bytes as floats
typedef uint32_t raw_u32x4 __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ void chunk_to_f32(const raw_u32x4& c, float* o);
template <> __device__ __forceinline__ void chunk_to_f32<bf16_t>(const raw_u32x4& c, float* o) {
#pragma unroll
  for (int i = 0; i < 4; ++i) o[2 * i] = bf16lo(c[i]), o[2 * i + 1] = bf16hi(c[i]);
}
template <> __device__ __forceinline__ void chunk_to_f32<float>(const raw_u32x4& c, float* o) {
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(c[i]);
}
template <> struct VecIO<float, 4> {
  __device__ static __forceinline__ void ld(const float* p, float* o) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p);
    o[0] = a[0], o[1] = a[1], o[2] = a[2], o[3] = a[3];
  }
  __device__ static __forceinline__ void st(float* p, const float* v) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  }
};

}  // namespace

#define DISPATCH_T(f32, ...)          \
  if (f32) {                          \
    using T = float;                  \
    __VA_ARGS__;                      \
  } else {                            \
    using T = bf16_t;                 \
    __VA_ARGS__;                      \
  }
