// The generalized delta rule token by token (recurrent.hip), as a function: its chunked form (delta_chunk.hip) takes short
// sequences, and values that are not finite, through the same arithmetic.
#pragma once
#include "recurrent.h"

namespace {

struct DeltaArgs {
  float* out;    // [T, H * dv]
  float* state;  // [slots, H, dv, dk]
  const void *r, *k, *v;
  int64_t rs, ks, vs;  // row strides (elements)
  const float* prep;   // [T, H, 3, dk]: unit key, decay, removal rate * unit key
  const int64_t* pos;
  const int* seq_rows;  // null: row i is sequence i
  const int* slots;
  int n_slots, T, H, dk, dv;
  // what `prep` is formed from, where delta_tokens does it (SELF)
  const void *a, *w;
  int64_t as, wst;
  const float *a_bias, *w_bias;
  float decay_scale, key_eps;
  int layers;  // of the step (state_once)
};

// u = k / sqrt(sum k^2 + key_eps), w = exp(-decay_scale sigmoid(wl + w_bias)), a u with a = sigmoid(al + a_bias); a wave
// holds the sum of its lanes' squares
__device__ __forceinline__ float delta_key_scale(float ss, float key_eps) { return rsqrtf(wave_reduce_sum(ss) + key_eps); }
__device__ __forceinline__ float delta_decay(float wl, float wb, float decay_scale) {
  return expf(-decay_scale * sigmoidf_(wl + wb));
}
__device__ __forceinline__ float delta_removal(float al, float ab, float u) { return sigmoidf_(al + ab) * u; }

// One token on a thread's rows of CT columns: b is the unit key, the decay, removal rate * unit key, the key and the read-out.
// (Its multiply-adds are written out: a row's result is the same bits in every kernel that takes it token by token.  The sign
// is where it leaves the state's old value in its register: with it on the product the compiler copied the tile first, 32
// sequences of one to 27 rows, 32 heads, 50.0 us instead of 46.6.)
template <int R, int CT>
__device__ __forceinline__ void delta_step(float (*S)[kRows], const float (*b)[kRows], const float* vj, float* o_) {
  float us[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    float a_ = 0.f;
#pragma unroll
    for (int q = 0; q < kRows; ++q) a_ = fmaf(b[0][q], S[c][q], a_);
    us[c] = group_sum<R>(a_);
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    float a_ = 0.f;
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      S[c][q] = fmaf(b[3][q], vj[c], -fmaf(-S[c][q], b[1][q], b[2][q] * us[c]));
      a_ = fmaf(b[4][q], S[c][q], a_);
    }
    o_[c] = group_sum<R>(a_);
  }
}

// kTok tokens' row vectors and the workgroup's values
template <int R, int NT, int CT> struct DeltaLds {
  __attribute__((aligned(16))) float r[kTok][kRows * R], k[kTok][kRows * R], u[kTok][kRows * R], w[kTok][kRows * R],
      a[kTok][kRows * R], v[kTok][NT / R * CT];
};

// Rows r0 .. r0 + n - 1 of one sequence and head, columns from col0 on (NT / R * CT of them, those below col_end).
// SELF: the row vectors are formed here instead of read from g.prep, and tokens run in a plain loop (few registers).
template <typename T, int R, int NT, int CT, bool SELF>
__device__ __forceinline__ void delta_tokens(const DeltaArgs& g, DeltaLds<R, NT, CT>& lds, int r0, int n, int h, int slot,
                                             int col0, int col_end) {
  constexpr int kCols = CT;
  constexpr int kGroups = NT / R;            // column tiles per workgroup
  constexpr int kWgCols = kGroups * kCols;   // columns per workgroup
  constexpr int kDkp = kRows * R;            // padded key width
  constexpr int kE = (kTok * kDkp + NT - 1) / NT;  // staged elements per thread and array
  constexpr int kEv = (kTok * kWgCols + NT - 1) / NT;
  constexpr int kWaves = NT / 64;
  static_assert(!SELF || (kDkp == 128 && kTok % kWaves == 0), "two channels a lane");
  auto &sr = lds.r, &sk = lds.k, &su = lds.u, &sw = lds.w, &sa = lds.a;
  auto& sv = lds.v;
  const int tid = threadIdx.x, part = tid % R, grp = tid / R, j0 = col0 + grp * kCols;
  const int wave = tid >> 6, lane = tid & 63;
  // The thread's 16 rows are four quads, quad m at row (m * R + part) * 4: for one m the R lanes of a
  // group read R consecutive 16-byte pieces of a row vector, so a wave's LDS read touches every bank once
  // (16 consecutive rows per lane would put lanes 0, 2, 4, .. on the same banks).
  float* sp = g.state + (((int64_t)slot * g.H + h) * g.dv) * g.dk;  // + column * dk + row
  const bool fresh = g.pos[r0] == 0;
  int rq[kRows / 4];
#pragma unroll
  for (int m = 0; m < kRows / 4; ++m) rq[m] = (m * R + part) * 4;
  float S[kCols][kRows];
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
#pragma unroll
    for (int q = 0; q < kRows; ++q) S[c][q] = 0.f;
    if (fresh || j0 + c >= col_end) continue;
    const float* spc = sp + (int64_t)(j0 + c) * g.dk;
#pragma unroll
    for (int m = 0; m < kRows / 4; ++m) {
      if (g.dk % 4 == 0 && rq[m] + 4 <= g.dk) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(spc + rq[m]);
        S[c][4 * m] = x[0], S[c][4 * m + 1] = x[1], S[c][4 * m + 2] = x[2], S[c][4 * m + 3] = x[3];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (rq[m] + e < g.dk) S[c][4 * m + e] = spc[rq[m] + e];
      }
    }
  }
  const T* pr = (const T*)g.r + (int64_t)h * g.dk;
  const T* pk = (const T*)g.k + (int64_t)h * g.dk;
  const float* pp = g.prep + (int64_t)h * 3 * g.dk;
  const T* pv = (const T*)g.v + (int64_t)h * g.dv + col0;
  float ab[2], wb[2];
  const T *pa = nullptr, *pw = nullptr;
  if constexpr (SELF) {
    pa = (const T*)g.a + (int64_t)h * g.dk;
    pw = (const T*)g.w + (int64_t)h * g.dk;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      ab[c] = g.a_bias ? g.a_bias[h * g.dk + lane + 64 * c] : 0.f;
      wb[c] = g.w_bias ? g.w_bias[h * g.dk + lane + 64 * c] : 0.f;
    }
  }
  float fr[kE], fk[kE], fu[kE], fa[kE], fw[kE], fv[kEv];
  auto fetch = [&](int t0) {
    if constexpr (SELF) {  // a wave per token, two channels a lane
#pragma unroll
      for (int e = 0; e < kE; ++e) {
        const int tt = wave + e / 2 * kWaves, ch = lane + 64 * (e & 1);
        const bool ok = t0 + tt < n;
        const int64_t row = r0 + t0 + tt;
        fr[e] = ok ? ldf<T>(pr, row * g.rs + ch) : 0.f;
        fk[e] = ok ? ldf<T>(pk, row * g.ks + ch) : 0.f;
        fa[e] = ok ? ldf<T>(pa, row * g.as + ch) : 0.f;
        fw[e] = ok ? ldf<T>(pw, row * g.wst + ch) : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < (SELF ? 0 : kE); ++e) {
      const int idx = tid + e * NT, tt = idx / kDkp, ch = idx % kDkp;
      const bool ok = idx < kTok * kDkp && t0 + tt < n && ch < g.dk;
      const int64_t row = r0 + t0 + tt;
      const float* pq = pp + row * g.H * 3 * g.dk + ch;
      fr[e] = ok ? ldf<T>(pr, row * g.rs + ch) : 0.f;
      fk[e] = ok ? ldf<T>(pk, row * g.ks + ch) : 0.f;
      fu[e] = ok ? pq[0] : 0.f;
      fw[e] = ok ? pq[g.dk] : 0.f;
      fa[e] = ok ? pq[2 * g.dk] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < kEv; ++e) {
      const int idx = tid + e * NT, tt = idx / kWgCols, cc = idx % kWgCols;
      const bool ok = idx < kTok * kWgCols && t0 + tt < n && col0 + cc < col_end;
      fv[e] = ok ? ldf<T>(pv, (int64_t)(r0 + t0 + tt) * g.vs + cc) : 0.f;
    }
  };
  fetch(0);
  float* outp = g.out + (int64_t)r0 * g.H * g.dv + h * g.dv + j0;
  const bool out4 = g.dv % 4 == 0 && j0 + kCols <= col_end;
  for (int t0 = 0; t0 < n; t0 += kTok) {
    __syncthreads();  // the previous block's tokens are consumed
    if constexpr (SELF) {
#pragma unroll
      for (int e = 0; e < kE; e += 2) {
        const int tt = wave + e / 2 * kWaves;
        const float inv = delta_key_scale(fmaf(fk[e + 1], fk[e + 1], fk[e] * fk[e]), g.key_eps);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int ch = lane + 64 * c;
          const float u = fk[e + c] * inv;
          sr[tt][ch] = fr[e + c];
          sk[tt][ch] = fk[e + c];
          su[tt][ch] = u;
          sw[tt][ch] = delta_decay(fw[e + c], wb[c], g.decay_scale);
          sa[tt][ch] = delta_removal(fa[e + c], ab[c], u);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < (SELF ? 0 : kE); ++e) {
      const int idx = tid + e * NT, tt = idx / kDkp, ch = idx % kDkp;
      if (idx < kTok * kDkp) {
        sr[tt][ch] = fr[e];
        sk[tt][ch] = fk[e];
        su[tt][ch] = fu[e];
        sw[tt][ch] = fw[e];
        sa[tt][ch] = fa[e];
      }
    }
#pragma unroll
    for (int e = 0; e < kEv; ++e) {
      const int idx = tid + e * NT;
      if (idx < kTok * kWgCols) sv[idx / kWgCols][idx % kWgCols] = fv[e];
    }
    __syncthreads();
    if (t0 + kTok < n) fetch(t0 + kTok);
    const int nt = n - t0 < kTok ? n - t0 : kTok;
    // the five row vectors of a token (unit key, decay, removal, key, read-out) and its values
    auto load = [&](int tt, float (*b)[kRows], float* vj) {
#pragma unroll
      for (int q = 0; q < kRows; q += 4) {
        *reinterpret_cast<f32x4*>(b[0] + q) = *reinterpret_cast<const f32x4*>(&su[tt][rq[q / 4]]);
        *reinterpret_cast<f32x4*>(b[1] + q) = *reinterpret_cast<const f32x4*>(&sw[tt][rq[q / 4]]);
        *reinterpret_cast<f32x4*>(b[2] + q) = *reinterpret_cast<const f32x4*>(&sa[tt][rq[q / 4]]);
        *reinterpret_cast<f32x4*>(b[3] + q) = *reinterpret_cast<const f32x4*>(&sk[tt][rq[q / 4]]);
        *reinterpret_cast<f32x4*>(b[4] + q) = *reinterpret_cast<const f32x4*>(&sr[tt][rq[q / 4]]);
      }
#pragma unroll
      for (int c = 0; c < kCols; ++c) vj[c] = sv[tt][grp * kCols + c];
    };
    auto step = [&](const float (*b)[kRows], const float* vj, float* o_) { delta_step<R, kCols>(S, b, vj, o_); };
    auto store = [&](int tt, const float* o_) {
      float* op = outp + (int64_t)(t0 + tt) * g.H * g.dv;
      if constexpr (kCols == 4) {
        if (out4) *reinterpret_cast<f32x4*>(op) = f32x4{o_[0], o_[1], o_[2], o_[3]};
      }
      if (kCols != 4 || !out4) {
#pragma unroll
        for (int c = 0; c < kCols; ++c)
          if (j0 + c < col_end) op[c] = o_[c];
      }
    };
    if (!SELF && kCols <= 2 && nt == kTok) {
      // a whole block of the narrow tile (the wide one has no registers to spare), unrolled in one basic
      // block: the next token's vectors are read from LDS while the current token's chain runs, and the
      // outputs are stored once at the end
      float b0[5][kRows], b1[5][kRows], v0[kCols], v1[kCols], ob[kTok][kCols];
      load(0, b0, v0);
#pragma unroll
      for (int tt = 0; tt < kTok; tt += 2) {
        load(tt + 1, b1, v1);
        step(b0, v0, ob[tt]);
        if (tt + 2 < kTok) load(tt + 2, b0, v0);
        step(b1, v1, ob[tt + 1]);
      }
      if (part == 0) {
#pragma unroll
        for (int tt = 0; tt < kTok; ++tt) store(tt, ob[tt]);
      }
    } else {
      for (int tt = 0; tt < nt; ++tt) {
        float b0[5][kRows], v0[kCols], o_[kCols];
        load(tt, b0, v0);
        step(b0, v0, o_);
        if (part == 0) store(tt, o_);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    if (j0 + c >= col_end) continue;
    float* spc = sp + (int64_t)(j0 + c) * g.dk;
#pragma unroll
    for (int m = 0; m < kRows / 4; ++m) {
      if (g.dk % 4 == 0 && rq[m] + 4 <= g.dk) {
        *reinterpret_cast<f32x4*>(spc + rq[m]) = f32x4{S[c][4 * m], S[c][4 * m + 1], S[c][4 * m + 2], S[c][4 * m + 3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (rq[m] + e < g.dk) spc[rq[m] + e] = S[c][4 * m + e];
      }
    }
  }
}

}  // namespace
