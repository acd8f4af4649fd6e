// Linear recurrences over a running matrix for gfx950: per (sequence, head) a
// matrix S [dk, dv], without softmax and without a denominator,
//     S_t = D_t S_(t-1) + (k_scale k_t) (u_t v_t)^T,   o_t = S_t^T (q_scale q_t) + skip_h v_t
// in three forms of the decay D_t and the step u_t (kMode):
//   kFixed    D_t = decay_h, u_t = 1                                         (retention)
//   kStep     u_t = softplus(g_t,h + bias_h), D_t = exp(-rate_h u_t)         (state-space duality)
//   kChannel  D_t = diag(sigmoid(g_t,h,i + bias_h,i)^(1 / tau)), u_t = 1     (gated linear attention)
// Query head h reads the q / k head h / qk_rep (state-space groups share them).
//
// Columns of S are independent: R neighbouring lanes share a column (up to
// kRows rows each, in registers) and join their partial q^T S by DPP lane
// exchanges; a workgroup owns blockDim / R columns of one (sequence, head).
// Tokens are staged through LDS kTok at a time.  State layout [slots, H, dv,
// dk]: a column's rows are contiguous.  This file scans token by token (any
// sizes, decode steps, fp32); chunk_scan.hip has the matrix-core form for prompt
// portions in bf16.  Slots, seq_rows and the reset at position 0 as in
// recurrent.hip.  Decays, step sizes, the state and all sums
// are fp32 whatever the activation element is.
#include "linear_scan.h"

namespace {

constexpr int kMaxKey = 512;

// Any sizes: rows and columns beyond dk / dv are guarded one by one.  Lane r of a column's group owns
// rows r, r + R, ...
template <typename T, int R, int MODE, int ROWS = kRows>
__global__ void __launch_bounds__(256) scan_kernel(ScanArgs g) {
  extern __shared__ float scan_lds[];
  const int s = blockIdx.x, h = blockIdx.y, hq = h / g.qk_rep;
  const int tid = threadIdx.x, cols = blockDim.x / R;
  const int cl = tid / R, r = tid % R;
  const int col0 = blockIdx.z * cols, j = col0 + cl;
  const int r0 = g.seq_rows ? g.seq_rows[s] : s, r1 = g.seq_rows ? g.seq_rows[s + 1] : s + 1;
  if (r1 <= r0 || r0 < 0 || r1 > g.T || r1 - r0 > g.max_rows) return;
  const bool colok = j < g.dv;
  const int slot = g.slots[s];
  const int64_t ow = (int64_t)g.H * g.dv;
  if (slot < 0 || slot >= g.n_slots) {  // a padding row: zeros out, no state touched
    for (int t = r0; t < r1; ++t)
      if (r == 0 && colok) g.out[(int64_t)t * ow + h * g.dv + j] = 0.f;
    return;
  }
  float* qs_ = scan_lds;
  float* ks_ = qs_ + kTok * g.dk;
  float* vs_ = ks_ + kTok * g.dk;
  float* gs_ = vs_ + kTok * cols;  // kStep: (step, decay) per token; kChannel: [kTok][dk] decays
  float* sp = g.state + (((int64_t)slot * g.H + h) * g.dv + (colok ? j : 0)) * g.dk;
  const bool fresh = g.pos[r0] == 0;
  float S[ROWS];
#pragma unroll
  for (int ii = 0; ii < ROWS; ++ii) {
    const int i = r + R * ii;
    S[ii] = (!fresh && colok && i < g.dk) ? sp[i] : 0.f;
  }
  const float fixed = MODE == kFixed ? g.decay[h] : 0.f, skip = g.skip ? g.skip[h] : 0.f;
  const T* q = (const T*)g.q;
  const T* k = (const T*)g.k;
  const T* v = (const T*)g.v;
  for (int t0 = r0; t0 < r1; t0 += kTok) {
    const int nt = r1 - t0 < kTok ? r1 - t0 : kTok;
    __syncthreads();  // the previous block's reads are done
    for (int e = tid; e < nt * g.dk; e += blockDim.x) {
      const int tt = e / g.dk, i = e - tt * g.dk;
      qs_[e] = ldf<T>(q, (int64_t)(t0 + tt) * g.qs + hq * g.dk + i) * g.q_scale;
      ks_[e] = ldf<T>(k, (int64_t)(t0 + tt) * g.ks + hq * g.dk + i) * g.k_scale;
      if constexpr (MODE == kChannel)
        gs_[e] = channel_decay(ldf<T>((const T*)g.g, (int64_t)(t0 + tt) * g.gs + h * g.dk + i) +
                                   (g.g_bias ? g.g_bias[h * g.dk + i] : 0.f), g.inv_tau);
    }
    for (int e = tid; e < nt * cols; e += blockDim.x) {
      const int tt = e / cols, c = e - tt * cols;
      vs_[e] = col0 + c < g.dv ? ldf<T>(v, (int64_t)(t0 + tt) * g.vs + h * g.dv + col0 + c) : 0.f;
    }
    if constexpr (MODE == kStep) {
      if (tid < nt) {
        const float2 st = step_terms<T>(g, t0 + tid, h);
        gs_[2 * tid] = st.x;
        gs_[2 * tid + 1] = st.y;
      }
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float vj = vs_[tt * cols + cl];
      const float uv = MODE == kStep ? vj * gs_[2 * tt] : vj;
      const float dec = MODE == kStep ? gs_[2 * tt + 1] : fixed;
      const float* qt = qs_ + tt * g.dk;
      const float* kt = ks_ + tt * g.dk;
      const float* gt = gs_ + tt * g.dk;
      float acc = 0.f;
#pragma unroll
      for (int ii = 0; ii < ROWS; ++ii) {
        const int i = r + R * ii;
        if (i < g.dk) {
          S[ii] = (MODE == kChannel ? gt[i] : dec) * S[ii] + kt[i] * uv;
          acc += qt[i] * S[ii];
        }
      }
      acc = group_sum<R>(acc);
      if (r == 0 && colok) g.out[(int64_t)(t0 + tt) * ow + h * g.dv + j] = acc + skip * vj;
    }
  }
  if (colok) {
#pragma unroll
    for (int ii = 0; ii < ROWS; ++ii) {
      const int i = r + R * ii;
      if (i < g.dk) sp[i] = S[ii];
    }
  }
}

// scan_tokens for every sequence of a step
template <typename T, int R, int MODE, bool ONCE>
__global__ void __launch_bounds__(256) scan_fast_kernel(ScanArgs g) {
  constexpr int cols = 256 / R;
  __shared__ ScanLds<16 * R, MODE, cols> lds;
  const int s = blockIdx.x, h = blockIdx.y, hq = h / g.qk_rep, col0 = blockIdx.z * cols;
  const int slot = g.slots[s];
  const int r0 = g.seq_rows ? g.seq_rows[s] : s, r1 = g.seq_rows ? g.seq_rows[s + 1] : s + 1;
  if ((r1 <= r0) | (r0 < 0) | (r1 > g.T) | (r1 - r0 > g.max_rows)) return;  // (bitwise: one wait for all of them)
  if (slot < 0 || slot >= g.n_slots) {  // a padding row: zeros out, no state touched
    for (int t = r0; t < r1; ++t)
      if (threadIdx.x % R == 0) g.out[(int64_t)t * g.H * g.dv + h * g.dv + col0 + threadIdx.x / R] = 0.f;
    return;
  }
  scan_tokens<T, R, MODE, cols, 256, ONCE>(g, lds, r0, r1, h, hq, slot, col0);
}

// whether the unconditional kernel serves the launch: dk = 16 R exactly, whole column blocks,
// 16-byte aligned rows and sections
template <typename T, int R, int MODE>
bool scan_fast_ok(const ScanArgs& g) {
  constexpr int VEC = 16 / (int)sizeof(T), cols = 256 / R;
  auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  return g.dk == 16 * R && g.dv % cols == 0 && cols % VEC == 0 && g.qs % VEC == 0 && g.ks % VEC == 0 &&
         g.vs % VEC == 0 && al(g.q) && al(g.k) && al(g.v) && al(g.state) &&
         (MODE != kChannel || (g.gs % VEC == 0 && al(g.g)));
}

template <typename T, int R, int MODE, int ROWS = kRows>
void launch_scan(const ScanArgs& g, int n_seq, hipStream_t st) {
  if constexpr (ROWS == kRows) {
    if (scan_fast_ok<T, R, MODE>(g)) {
      auto kern = state_once(n_seq, g.H, g.dk, g.dv, g.layers) ? scan_fast_kernel<T, R, MODE, true> : scan_fast_kernel<T, R, MODE, false>;
      hipLaunchKernelGGL(kern, dim3(n_seq, g.H, g.dv / (256 / R)), dim3(256), 0, st, g);
      return;
    }
  }
  int nt = (R * g.dv + 63) / 64 * 64;
  nt = nt > 256 ? 256 : nt;
  const int cols = nt / R;
  const size_t lds = (size_t)((MODE == kChannel ? 3 : 2) * kTok * g.dk + kTok * cols + 2 * kTok) * sizeof(float);
  hipLaunchKernelGGL((scan_kernel<T, R, MODE, ROWS>), dim3(n_seq, g.H, (g.dv + cols - 1) / cols), dim3(nt), lds, st, g);
}

template <typename T, int MODE>
void dispatch_rows(const ScanArgs& g, int n_seq, hipStream_t st) {
  const int need = (g.dk + kRows - 1) / kRows;
  if (need <= 1) launch_scan<T, 1, MODE>(g, n_seq, st);
  else if (need <= 2) launch_scan<T, 2, MODE>(g, n_seq, st);
  else if (need <= 4) launch_scan<T, 4, MODE>(g, n_seq, st);
  else if (need <= 8) launch_scan<T, 8, MODE>(g, n_seq, st);
  else if (need <= 16) launch_scan<T, 16, MODE>(g, n_seq, st);
  else launch_scan<T, 16, MODE, kMaxKey / 16>(g, n_seq, st);
}

}  // namespace

extern "C" int dxm_linear_scan(int mode, float* out, float* state, int n_slots, const void* q, int64_t qs, const void* k,
                               int64_t ks, const void* v, int64_t vs, float q_scale, float k_scale, int qk_rep,
                               const float* decay, const void* gate, int64_t gs, const float* g_bias, const float* rate,
                               const float* skip, float inv_tau, const int64_t* pos, const int* seq_rows,
                               const int* slots, int n_seq, int T_, int H, int dk, int dv, int f32, int layers,
                               hipStream_t st) {
  if (n_seq <= 0 || T_ <= 0) return 0;
  if (H < 1 || dk < 1 || dv < 1 || n_slots < 1 || H > 65535 || (int64_t)T_ * H * dv > 0x7fffffffffffLL) return 1;
  if (dk > kMaxKey) return 2;  // wider keys need more rows per lane than instantiated
  if (!out || !state || !pos || !slots || !q || !k || !v) return 3;
  if (!seq_rows && n_seq != T_) return 4;
  if (qk_rep < 1 || H % qk_rep) return 5;
  ScanArgs g{out, state, q, k, v, qs, ks, vs, q_scale, k_scale, qk_rep, decay, gate, gs, g_bias, rate, skip, inv_tau,
             pos, seq_rows, slots, n_slots, T_, H, dk, dv, 1, 0x7fffffff, 0, 0, layers};
  // prompt portions in bf16: matrix-core chunks where the sizes fit; shorter runs of a sequence
  // (decode tokens among them) stay with the token scan
  if (!f32 && seq_rows && n_seq <= 65535 && T_ >= kChunkMinRows + n_seq - 1 && chunk_scan_ok(mode, g)) {
    if ((mode == kFixed && !decay) || (mode == kStep && (!gate || !rate)) || (mode == kChannel && !gate)) return 6;
    g.min_rows = kChunkMinRows;
    if (launch_chunk_scan(mode, g, n_seq, st) || n_seq == 1) {
      DX_CHECK_LAUNCH();
      return 0;
    }
    g.max_rows = kChunkMinRows - 1;
  }
  if (mode == kFixed) {
    if (!decay) return 6;
    DISPATCH_T(f32, (dispatch_rows<T, kFixed>(g, n_seq, st)));
  } else if (mode == kStep) {
    if (!gate || !rate) return 6;
    DISPATCH_T(f32, (dispatch_rows<T, kStep>(g, n_seq, st)));
  } else if (mode == kChannel) {
    if (!gate) return 6;
    DISPATCH_T(f32, (dispatch_rows<T, kChannel>(g, n_seq, st)));
  } else {
    return 7;
  }
  DX_CHECK_LAUNCH();
  return 0;
}
