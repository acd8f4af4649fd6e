// Grouped GEMM of few rows per expert (a decode step of a mixture of experts), for gfx950: the experts'
// weights stream from HBM once, straight into matrix-core fragments; the handful of activation rows comes
// from L2.  Same meaning as grouped_gemm (moe.hip): for expert e, rows r of its run offsets[e] ..
// offsets[e + 1],
//     out[dst(r), :] = a[src(r), :] @ w[e]^T        src(r) = order[r] / top (gather) or r, dst(r) = order[r] (scatter) or r
// and with glu (weights in blocks of 32 gate rows and their 32 up rows) out = silu(gate) * up, [R, N / 2].
//
// A workgroup (2 or 4 waves) takes 32 weight rows of one expert -- 16 gate and their 16 up rows with glu -- and
// all rows of the expert, 64 at a time; the waves share the width in pieces of 64 and their partial
// sums are added in LDS in wave order.  v_mfma_f32_16x16x32_bf16 with the weights as A (lane: one weight row,
// 32 contiguous bytes of each piece: four lanes read a whole line) and the activations as B in the same
// order, so nothing is shuffled; two pieces are in flight per wave.  More in flight is slower (three pieces
// by a tenth, eight or sixteen waves by 6 to 50 %): HBM likes the few long runs of lines better.
//
// Bound by HBM.  A line is read by two loads, 16 bytes of each lane's 32 at a time, so the lines have to stay:
// as nontemporal loads (before, and for steps of one or two rows) part of them come from memory twice.  16 experts of 3584, 24 tokens, gate-up /
// down: 169 / 93 us -> 144 / 75, 6.3 TB/s.  A pass takes 16, 32 or 64 rows, whichever holds the rest: a pass of
// 16 leaves out the products and loads of the second tile (24 tokens: 148 / 77 us without), one of 64 reads the
// weights once where two of 32 read them twice (8 experts of 2048, 100 tokens: 56 / 26 us -> 39 / 23).
#include "../kernels/common.h"

namespace {

typedef uint32_t gs_raw4 __attribute__((ext_vector_type(4)));
typedef __bf16 gs_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kMT = 4, kDepth = 2;

struct StreamGemmArgs {
  bf16_t* out;
  const bf16_t* a;
  int64_t a_stride;
  const bf16_t* w;  // [E, N, K]
  const int* order;
  const int* offsets;
  int N, K, top, gather, scatter;
};

// MT: 16-row activation tiles, NW: waves, NT: the weights' lines are not kept in L2
template <int MT, int NW, bool NT, bool GLU>
__device__ __forceinline__ void stream_pass(const StreamGemmArgs& g, int e, int lo, int rows, int j, f32x4* red) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c16 = lane & 15, g4 = lane >> 4;
  // first weight rows of the two 16-row tiles
  const int n0 = GLU ? 64 * (j >> 1) + 16 * (j & 1) : 32 * j;
  const int n1 = GLU ? n0 + 32 : n0 + 16;
  const bf16_t* wp[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int n = (t ? n1 : n0) + c16;
    wp[t] = g.w + ((int64_t)e * g.N + (n < g.N ? n : 0)) * g.K + 16 * g4 + 64 * wave;
  }
  const bf16_t* ap[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int r = lo + min(16 * m + c16, rows - 1);  // rows past the last repeat it and are not stored
    ap[m] = g.a + (int64_t)(g.gather ? g.order[r] / g.top : r) * g.a_stride + 16 * g4 + 64 * wave;
  }
  f32x4 C[2][MT];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) C[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int D = kDepth;
  gs_raw4 W[D][2][2], A[D][MT][2];
  const int np = (g.K / 64 - wave + NW - 1) / NW;  // this wave's pieces: wave, wave + NW, ...
  auto fetch = [&](int s, int p) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const gs_raw4* q = reinterpret_cast<const gs_raw4*>(wp[t] + (int64_t)p * (64 * NW) + 8 * h);
        if constexpr (NT) W[s][t][h] = __builtin_nontemporal_load(q);
        else W[s][t][h] = *q;
      }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) A[s][m][h] = *reinterpret_cast<const gs_raw4*>(ap[m] + (int64_t)p * (64 * NW) + 8 * h);
  };
  auto use = [&](int s) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          C[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gs_bf16x8, W[s][t][h]),
                                                            __builtin_bit_cast(gs_bf16x8, A[s][m][h]), C[t][m], 0, 0, 0);
  };
  if (np > 0) {
    // workgroups start at different pieces: rows a power of two apart would otherwise meet on the same channels
    const int skew = (j * 5 + e * 3) % np;
    auto at = [&](int p) {
      p = min(p, np - 1) + skew;
      return p < np ? p : p - np;
    };
#pragma unroll
    for (int s = 0; s < D; ++s) fetch(s, at(s));
    for (int p = 0; p < np; p += D) {  // a slot is refilled as it is used (at the end: with the last piece again)
#pragma unroll
      for (int s = 0; s < D; ++s) {
        if (p + s < np) use(s);
        fetch(s, at(p + D + s));
      }
    }
  }
  // C[t][m]: weight rows n_t + 4 g4 .. + 3 of activation row 16 m + c16
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((wave * 2 + t) * MT + m) * 64 + lane] = C[t][m];
  __syncthreads();
  constexpr int kFrags = GLU ? MT : 2 * MT;
  for (int f = wave; f < kFrags; f += NW) {
    const int t = GLU ? 0 : f / MT, m = GLU ? f : f - t * MT;
    auto total = [&](int tt) {
      f32x4 s = red[(tt * MT + m) * 64 + lane];
#pragma unroll
      for (int wv = 1; wv < NW; ++wv) s += red[((wv * 2 + tt) * MT + m) * 64 + lane];
      return s;
    };
    f32x4 v = total(t);
    int n = (t ? n1 : n0) + 4 * g4, No = g.N;
    if constexpr (GLU) {
      const f32x4 u = total(1);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.f + __expf(-v[i])) * u[i];
      n = 16 * j + 4 * g4;
      No = g.N / 2;
    }
    const int r = 16 * m + c16;
    if (r >= rows || n >= No) continue;
    const int64_t dst = g.scatter ? g.order[lo + r] : lo + r;
    *reinterpret_cast<uint2*>(g.out + dst * No + n) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
  __syncthreads();  // (red is free again)
}

template <int NW, bool NT, bool GLU>
__global__ void __launch_bounds__(64 * NW, 2) stream_grouped_gemm_kernel(StreamGemmArgs g) {
  __shared__ __attribute__((aligned(16))) f32x4 red[NW * 2 * kMT * 64];
  const int e = blockIdx.y, j = blockIdx.x;
  const int lo = g.offsets[e], hi = g.offsets[e + 1];
  for (int r = lo; r < hi; r += 16 * kMT) {
    if (hi - r <= 16) stream_pass<1, NW, NT, GLU>(g, e, r, hi - r, j, red);
    else if (hi - r <= 32) stream_pass<2, NW, NT, GLU>(g, e, r, hi - r, j, red);
    else stream_pass<kMT, NW, NT, GLU>(g, e, r, min(hi - r, 16 * kMT), j, red);
  }
}

}  // namespace

extern "C" {

// 1 when stream_grouped_gemm takes the shape: whole 64-wide pieces, whole 32-row blocks of weights
int dxm_stream_grouped_ok(int N, int K) { return N >= 32 && N % 32 == 0 && K >= 64 && K % 64 == 0; }

int dxm_stream_grouped_gemm(void* out, const void* a, int64_t a_stride, const void* w, const int* order,
                            const int* offsets, int R, int E, int N, int K, int top, int gather, int scatter, int glu,
                            hipStream_t st) {
  if (R <= 0) return 0;
  if (E < 1 || E > 65535 || top < 1 || !dxm_stream_grouped_ok(N, K) || (glu && N % 64)) return 1;
  if (!out || !a || !w || !order || !offsets || a_stride % 8 || (uintptr_t)a % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)out % 8)
    return 2;
  const StreamGemmArgs g{(bf16_t*)out, (const bf16_t*)a, a_stride, (const bf16_t*)w, order, offsets, N, K, top, gather, scatter};
  const dim3 grid((unsigned)(N / 32), (unsigned)E);
  // Two waves where four would have no more than eight pieces each: 2048 wide, 8 experts, gate-up + down, 3 / 16 / 40
  // tokens, us: 33.2 / 45.8 / 48.5 with four, 29.0 / 44.8 / 46.2 with two; 4096 and 3584 wide, 16 experts, 6 / 24 tokens:
  // 125.6 / 223.1 with four, 141.7 / 237.3 with two.  Between them, 16 experts as wide as the model, two layers, 2 / 6 / 24 / 60
  // tokens: 2304 80 / 143 / 204 / 222 with four, 86 / 146 / 209 / 223 with two; 2560 76 / 140 / 242 / 264, 95 / 158 / 262 / 283.
  const bool two = K <= 2048;
  // Of one or two rows in all little comes through the caches, and what a step of many layers reads is not there the next time:
  // 24 layers of 8 experts of 2048 (nothing of 0.4 to 1.2 GB is left), a layer, kept / not, us, one row 21.7 / 20.4, two (one
  // token's at two each) 25.0 / 24.3, two tokens' at one each 24.9 / 24.6, four 31.4 / 34.3 (two tokens') and 33.3 / 37.1 (one
  // token's); experts of 1792 20.9 / 19.6, 25.0 / 25.5, 24.6 / 25.1, 30.3 / 34.0 and 32.2 / 36.7.  (Steps that fit the last cache lose:
  // eight layers of 2048, one row 17.7 / 20.8, two 25.1 / 24.2.)
  const bool nt = two && R <= 2;
  auto kern = nt    ? (glu ? stream_grouped_gemm_kernel<2, true, true> : stream_grouped_gemm_kernel<2, true, false>)
              : two ? (glu ? stream_grouped_gemm_kernel<2, false, true> : stream_grouped_gemm_kernel<2, false, false>)
                    : (glu ? stream_grouped_gemm_kernel<4, false, true> : stream_grouped_gemm_kernel<4, false, false>);
  // LDS that is not used keeps four-wave workgroups at two a CU.  Few experts with rows are few workgroups, and the
  // dispatcher would pile four on one CU and leave others idle: 4 experts, down (512 workgroups): 29.6 us -> 23.3.
  hipLaunchKernelGGL(kern, grid, dim3(two ? 128 : 256), two ? 0 : 32 * 1024, st, g);
  DX_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
