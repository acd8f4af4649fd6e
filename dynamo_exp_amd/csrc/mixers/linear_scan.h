// Shared by the token-by-token and the chunked form of the linear recurrences
// (linear_scan.hip, chunk_scan.hip): arguments, decays, step sizes.
#pragma once
#include "recurrent.h"

enum ScanMode { kFixed = 0, kStep = 1, kChannel = 2 };

struct ScanArgs {
  float* out;    // [T, H * dv]
  float* state;  // [slots, H, dv, dk]
  const void *q, *k, *v;
  int64_t qs, ks, vs;  // row strides (elements)
  float q_scale, k_scale;
  int qk_rep;          // heads that share a q / k head
  const float* decay;  // kFixed: [H]
  const void* g;       // kStep: step logits [T, H]; kChannel: decay logits [T, H * dk]
  int64_t gs;
  const float* g_bias;  // [H] / [H * dk] or null
  const float* rate;    // kStep: [H]
  const float* skip;    // [H] or null
  float inv_tau;        // kChannel
  const int64_t* pos;
  const int* seq_rows;  // null: row i is sequence i
  const int* slots;
  int n_slots, T, H, dk, dv;
  int min_rows, max_rows;  // sequences with fewer / more rows in the step are another launch's
  int sorted;              // chunked kernels: workgroups take the sequences by length
  int all;                 // chunked kernels: sequences of fewer rows than min_rows too, token by token
  int layers;              // of the step (state_once)
};

__device__ __forceinline__ float softplusf_(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// sigmoid(z)^(1 / tau) = exp(-softplus(-z) / tau).  Only the exponent's absolute error matters, so the
// plain log of 1 + e serves (its error is below 1e-7 where log1p would return e itself).
__device__ __forceinline__ float channel_decay(float z, float inv_tau) {
  const float sp = fmaxf(-z, 0.f) + __logf(1.f + __expf(-fabsf(z)));
  return __expf(-sp * inv_tau);
}

// step size of one (row, head)
template <typename T> __device__ __forceinline__ float step_size(const ScanArgs& g, int64_t row, int h) {
  return softplusf_(ldf<T>((const T*)g.g, row * g.gs + h) + (g.g_bias ? g.g_bias[h] : 0.f));
}

// step size and decay of one (row, head)
template <typename T> __device__ __forceinline__ float2 step_terms(const ScanArgs& g, int64_t row, int h) {
  const float u = step_size<T>(g, row, h);
  return float2{u, expf(-g.rate[h] * u)};
}

// The same for key widths dk = 16 R and 16-byte aligned operands: nothing in the token loop is
// conditional.  Lane r of a column's group owns the four row quads 4 (r + R qd) .. + 3, qd < 4, so
// a group's 128-bit LDS reads of a row vector are neighbouring chunks and the state is read and
// written as 16-byte runs.  The next block's eight tokens (q, k, decay logits of the head, v of the
// workgroup's columns) are fetched into registers as 16-byte chunks while the current block's chain runs.
// The first block is asked for in front of the state and staged while the state is on its way (its barriers wait for LDS
// only), and the state in front of the position that says whether it counts, so that a decode step is one latency, not three
// (four layers of gated linear attention, 16 heads, 5 sequences 38.9 -> 37.6 us with the latter).  Bound by memory: two layers with their other launches in a graph, us:
// state-space duality, 128 heads of 64 columns, 2 / 12 / 64 sequences 32 / 70 / 239 -> 30 / 64 / 204 (the last with
// ONCE, 230 without); gated linear attention, 32 heads of 128 columns, 12 / 64: 39 / 139 -> 38 / 112 (135 without).
template <int DK, int MODE, int COLS> struct ScanLds {
  __attribute__((aligned(16))) float q[kTok * DK];
  __attribute__((aligned(16))) float k[kTok * DK];
  __attribute__((aligned(16))) float a[MODE == kChannel ? kTok * DK : 4];
  __attribute__((aligned(16))) float v[kTok * COLS];
  float2 u[kTok];
};

// rows r0 .. r1 - 1 (of one sequence, whose state is in `slot`) of columns col0 .. + COLS - 1 of head h, by a workgroup of NT
// threads, COLS R of which own columns; hq: its q / k head (a division, which the caller has done beside its loads); ONCE: the
// state's lines are not kept (state_once)
template <typename T, int R, int MODE, int COLS, int NT, bool ONCE = false>
__device__ __forceinline__ void scan_tokens(const ScanArgs& g, ScanLds<16 * R, MODE, COLS>& lds, int r0, int r1, int h, int hq, int slot,
                                            int col0) {
  constexpr int dk = 16 * R, cols = COLS, VEC = 16 / (int)sizeof(T);
  constexpr int QC = dk / VEC, VC = cols / VEC;  // chunks per token row
  constexpr int QK_CH = kTok * QC, V_CH = kTok * VC;
  constexpr int N_ROWS = MODE == kChannel ? 3 : 2;  // row vectors of dk staged per token
  constexpr int N_CH = N_ROWS * QK_CH + V_CH;
  constexpr int PER = (N_CH + NT - 1) / NT;
  float *qs_ = lds.q, *ks_ = lds.k, *as_ = lds.a, *vs_ = lds.v;
  float2* us_ = lds.u;
  static_assert(NT >= COLS * R, "a column's lanes");
  const int tid = threadIdx.x, r = tid % R;
  const bool owner = NT == COLS * R || tid < COLS * R;
  const int cl = owner ? tid / R : 0, j = col0 + cl;
  const int64_t ow = (int64_t)g.H * g.dv;
  float* sp = g.state + (((int64_t)slot * g.H + h) * g.dv + j) * dk;
  const float fixed = MODE == kFixed ? g.decay[h] : 0.f, skip = g.skip ? g.skip[h] : 0.f;
  const T* q = (const T*)g.q + (int64_t)hq * dk;
  const T* k = (const T*)g.k + (int64_t)hq * dk;
  const T* gl = (const T*)g.g + (int64_t)h * dk;
  const T* v = (const T*)g.v + (int64_t)h * g.dv + col0;
  raw_u32x4 pf[PER];
  // kChannel: a thread's chunks Z0 .. Z1 - 1 may be decays, and have biases
  constexpr int Z0 = 2 * QK_CH / NT, Z1 = (3 * QK_CH + NT - 1) / NT;
  float zb[MODE == kChannel ? Z1 - Z0 : 1][VEC] = {};
  // kStep: token tid's step logit as loaded (its terms are formed in commit(): here they would wait for the load)
  T logit{};
  bool stepped = false;
  const float g_bias = MODE == kStep && g.g_bias ? g.g_bias[h] : 0.f, rate = MODE == kStep ? g.rate[h] : 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NT;
      const T* src = nullptr;
      if (c < QK_CH) {
        const int tt = c / QC;
        if (t0 + tt < r1) src = q + (int64_t)(t0 + tt) * g.qs + (c % QC) * VEC;
      } else if (c < 2 * QK_CH) {
        const int c2 = c - QK_CH, tt = c2 / QC;
        if (t0 + tt < r1) src = k + (int64_t)(t0 + tt) * g.ks + (c2 % QC) * VEC;
      } else if (MODE == kChannel && c < 3 * QK_CH) {
        const int c2 = c - 2 * QK_CH, tt = c2 / QC;
        if (t0 + tt < r1) src = gl + (int64_t)(t0 + tt) * g.gs + (c2 % QC) * VEC;
      } else if (c < N_CH) {
        const int c2 = c - N_ROWS * QK_CH, tt = c2 / VC;
        if (t0 + tt < r1) src = v + (int64_t)(t0 + tt) * g.vs + (c2 % VC) * VEC;
      }
      pf[i] = src ? *reinterpret_cast<const raw_u32x4*>(src) : raw_u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (MODE == kStep) {
      stepped = tid < kTok && t0 + tid < r1;
      if (stepped) logit = ((const T*)g.g)[(int64_t)(t0 + tid) * g.gs + h];
    }
  };
  auto commit = [&]() {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + i * NT;
      float f[VEC];
      chunk_to_f32<T>(pf[i], f);
      float* dst = nullptr;
      if (c < QK_CH) {
        dst = qs_ + c * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] *= g.q_scale;
      } else if (c < 2 * QK_CH) {
        dst = ks_ + (c - QK_CH) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] *= g.k_scale;
      } else if (MODE == kChannel && c < 3 * QK_CH) {
        dst = as_ + (c - 2 * QK_CH) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = channel_decay(f[e] + zb[i >= Z0 && i < Z1 ? i - Z0 : 0][e], g.inv_tau);
      } else if (c < N_CH) {
        dst = vs_ + (c - N_ROWS * QK_CH) * VEC;
      }
      if (dst) {
#pragma unroll
        for (int e = 0; e < VEC; e += 4) *reinterpret_cast<f32x4*>(dst + e) = f32x4{f[e], f[e + 1], f[e + 2], f[e + 3]};
      }
    }
    if constexpr (MODE == kStep) {
      if (tid < kTok) {
        const float u = softplusf_(ldf<T>(&logit, 0) + g_bias);
        us_[tid] = stepped ? float2{u, expf(-rate * u)} : float2{0.f, 1.f};
      }
    }
  };
  fetch(r0);  // (in front of the state, which it does not wait for)
  // The biases of the thread's decays, the same for every token.  (Asked for where the rows go to LDS they were a latency more:
  // decode steps with their norms in a graph, 32 heads of 128 columns, four layers of 4 / 16 sequences 39.3 -> 37.6, 78 -> 67
  // us, two of 40 71 -> 64.  Only by the waves that hold decays, and where there are biases: asked for by all, with the state for
  // missing ones, three layers without biases of 8 sequences 28.6 -> 27.3 us, of 400 of 64 / 64 columns 264 -> 257, with them
  // 264 -> 257 and of 8 of 128 / 128 28.7 -> 27.8; 256 / 128 columns, 64 prompts of 30 rows without 549 -> 533.)
  if constexpr (MODE == kChannel) {
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const float* from = g.g_bias + h * dk;
#pragma unroll
    for (int i = Z0; i < Z1; ++i) {
      const int c2 = tid + i * NT - 2 * QK_CH;
      if (g.g_bias && c2 >= 0 && c2 < QK_CH) {
#pragma unroll
        for (int e = 0; e < VEC; e += 4) {
          const f32x4 b = *reinterpret_cast<const f32x4_a4*>(from + c2 % QC * VEC + e);
          zb[i - Z0][e] = b[0], zb[i - Z0][e + 1] = b[1], zb[i - Z0][e + 2] = b[2], zb[i - Z0][e + 3] = b[3];
        }
      }
    }
  }
  // (asked for before it is known whether it counts: at position 0 the state is zero, whatever the slot held)
  float S[16];
#pragma unroll
  for (int qd = 0; qd < 4; ++qd) *reinterpret_cast<f32x4*>(S + 4 * qd) = load_state<ONCE>(sp + 4 * (r + R * qd));
  const bool fresh = g.pos[r0] == 0;
  for (int t0 = r0; t0 < r1; t0 += kTok) {
    const int nt = r1 - t0 < kTok ? r1 - t0 : kTok;
    lds_barrier();  // the previous block's reads are done
    commit();
    lds_barrier();
    if (fresh && t0 == r0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) S[i] = 0.f;
    }
    if (t0 + kTok < r1) fetch(t0 + kTok);
    for (int tt = 0; tt < nt; ++tt) {
      const float vj = vs_[tt * cols + cl];
      float uv = vj, dec = fixed;
      if constexpr (MODE == kStep) {
        const float2 u = us_[tt];
        uv = vj * u.x;
        dec = u.y;
      }
      float acc = 0.f;
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const f32x4 kk = *reinterpret_cast<const f32x4*>(ks_ + tt * dk + 4 * (r + R * qd));
        const f32x4 qq = *reinterpret_cast<const f32x4*>(qs_ + tt * dk + 4 * (r + R * qd));
        f32x4 aa;
        if constexpr (MODE == kChannel) aa = *reinterpret_cast<const f32x4*>(as_ + tt * dk + 4 * (r + R * qd));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // (written out: every instance rounds alike, whichever launch a sequence is in)
          S[4 * qd + e] = fmaf(MODE == kChannel ? aa[e] : dec, S[4 * qd + e], kk[e] * uv);
          acc = fmaf(qq[e], S[4 * qd + e], acc);
        }
      }
      acc = group_sum<R>(acc);
      if (r == 0 && owner) g.out[(int64_t)(t0 + tt) * ow + h * g.dv + j] = fmaf(skip, vj, acc);
    }
  }
  if (!owner) return;
#pragma unroll
  for (int qd = 0; qd < 4; ++qd)
    store_state<ONCE>(sp + 4 * (r + R * qd), f32x4{S[4 * qd], S[4 * qd + 1], S[4 * qd + 2], S[4 * qd + 3]});
}

// a sequence with at least this many rows in the step goes through the chunked kernels
constexpr int kChunkMinRows = 8;

bool chunk_scan_ok(int mode, const ScanArgs& g);
// true: it takes the shorter sequences as well
bool launch_chunk_scan(int mode, const ScanArgs& g, int n_seq, hipStream_t st);
