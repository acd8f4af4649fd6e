// The generalized delta rule (recurrent.hip) over prompt rows in chunks of 16 tokens, for gfx950; keys of 128 channels,
// everything in true fp32 on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32).
//
//     S_t = diag(w_t) S_(t-1) - b_t (u_t^T S_(t-1)) + k_t v_t^T,    o_t = S_t^T r_t,      b_t = a_t * u_t
//
// Within a chunk let P_t be the product of the decays up to token t (P_0 = 1) and S the state in front of it.  With
//     U_t = u_t P_(t-1),  R_t = r_t P_t,  B_t = b_t / P_t,  K_t = k_t / P_t        (per channel; rows of [16, 128])
// the removed rows X_t = u_t^T S_(t-1) solve a lower triangular system of 16 rows, and everything is linear in S and V:
//     X = U' S + G V       U' = (I + tril(U B^T, -1))^-1 U,        G = (I + tril(U B^T, -1))^-1 tril(U K^T, -1)
//     O = R' S + H V       R' = R - tril(R B^T) U',                H = tril(R K^T) - tril(R B^T) G
//     S <- diag(P_16) S + K''^T V - B''^T X                        K'' = K P_16, B'' = B P_16
// delta_form_kernel makes U', R', K'', B'', G, H and P_16 of every (chunk, head) of the sequences long enough (kLong) -- no
// chunk needs another's -- and delta_chunk_kernel runs the chunks of a sequence in order: per (sequence, head, 16 columns of S) four waves that
// own 32 channels each, S in their accumulators.  A wave's accumulators are the second operand of its part of U' S and
// R' S as they lie; the parts of X and O join in LDS, one barrier a chunk.  The other sequences run in the same launch,
// token by token, beside the long ones' chains.
//
// P_t shrinks by at most exp(-16 |decay_scale|) in a chunk: 1e-7, and 1 / P 1e7, at the largest the host sends here (1), so
// that only values within 1e7 of fp32's ends leave its range on the way.  A chunk's dependent chain is 50 matrix
// instructions and a barrier instead of 16 tokens' chains of lane sums.
// Its rounding: the products of decays come from sums of logarithms in fp64, the sums run in an order that keeps them
// small and through short chains; relative to 64 bits 1.28e-7 in o and 6.90e-8 in S where the token-by-token form has
// 1.32e-7 and 6.91e-8 (900 to 4001 tokens; 1.9e-7 and 1.2e-7 with running products and one chain per sum).
// A value that is not finite, or that 1 / P makes so, would reach other rows of its chunk than its own and later ones (zero
// factors times it).  It shows in the rows or stays in the state, and a workgroup that meets one takes its columns again,
// token by token.
// 4001 tokens in three prompts, 32 heads: 1287 us token by token + 85 us for its elementwise pass -> 211 + 99 us, each
// profiled by itself (in a row, with the layer's norm of 24: 314); a prompt of 600 beside 30 single tokens 704 -> 89, the
// layer without its norm.  Bound by the chain of the longest prompt's chunks: 125 of them at 3700 cycles where three
// workgroups share a CU, 1088 of a wave's matrix instructions each, so that the matrix cores are busy 59 % of the time (a
// chain alone: 2400 cycles a chunk); 162 us with the loads taken out.
#include <algorithm>

#include "delta_tokens.h"

namespace {

constexpr int kC = 16;    // tokens per chunk
// A sequence with at least this many rows in the step goes in chunks, a shorter one (a decode row beside a prompt among
// them) token by token, whatever else is in the step: what shares a step does not change a sequence's arithmetic.
// From 32 rows on the chunks are no slower: one prompt of 32 rows 23 us either way, 63 36 token by token and 22 in chunks;
// 16 prompts of 32 78 and 75; 600 rows beside 30 decode rows 704 all token by token, 138 all in chunks, 102 like this.
constexpr int kLong = 32;
constexpr int kD = 128;   // key channels
constexpr int kPad = 4;   // floats of padding per LDS row
constexpr int kMat = kC * kD;
// Floats per (chunk, head): U', R', K''^T, B''^T, G, H, P_16.  The matrices lie as the chunk kernel's lanes take them, 16
// bytes a lane and 1 KiB an instruction in a row: U' and R' [channel / 16][channel / 4 % 4][row][channel % 4], K''^T and
// B''^T [channel / 16][row / 4][channel % 16][row % 4], G and H [column % 4][column / 4][row].  In rows of 128 channels
// neighbouring lanes lay 512 bytes apart, every lane a cache line of its own, and the chains waited for the vector cache's
// tags: 298 us of the case below (163 with the loads taken out), 228 like this.
constexpr int kChunkFloats = 4 * kMat + 2 * kC * kC + kD;

struct FormArgs {
  float* ws;  // [chunks, H, kChunkFloats]
  const bf16_t *r, *k, *a, *w;
  int64_t rs, ks, as, wst;  // row strides (elements)
  const float *a_bias, *w_bias;
  const int* seq_rows;
  const int* slots;
  float decay_scale, key_eps;
  int n_seq, n_slots, T, H;
};

// A long sequence s has the chunks first_chunk(s) and up.  The second term grows by one at least with every long sequence,
// so no two share a chunk; the step's rows bound it as its sequences do.
__device__ __forceinline__ int first_chunk(const int* seq_rows, int s) {
  return (seq_rows[s] >> 4) + min(s, seq_rows[s] / kLong);
}

// Where token t stands in U' (row), G (row and column), H (column), K''^T and B''^T (column): instruction i of the chunk
// kernel's sums over tokens then takes tokens 4 i .. 4 i + 3.  In the order of the tokens, later ones decayed less, the
// partial sums stay small until the end and little is rounded away.
__device__ __forceinline__ int place(int t) { return 4 * (t & 3) + (t >> 2); }

__device__ __forceinline__ f32x4 mma1(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Reads and writes through descriptors: a uniform base and a size for the rows of a chunk, lane offsets that stay the same
// from chunk to chunk.  Behind the size reads are 0 and nothing is written.
typedef __amdgpu_buffer_rsrc_t Range;
__device__ __forceinline__ Range range(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
}
__device__ __forceinline__ f32x4 get4(Range r, uint32_t off, int at) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, at, 0));
}
__device__ __forceinline__ float get1(Range r, uint32_t off, int at) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, at, 0));
}
__device__ __forceinline__ uint32_t get_half(Range r, uint32_t off, int at) {
  return __builtin_amdgcn_raw_buffer_load_b16(r, off, at, 0);
}
__device__ __forceinline__ void put1(Range r, uint32_t off, int at, float x) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), r, off, at, 0);
}

// 1 / (1 + exp(-z)) with the exponential's argument in two parts and a Newton step behind the reciprocal: half the
// instructions of 1.f / (1.f + expf(-z)), and nearer to 64 bits (largest relative error over 2^24 arguments of |z| < 1, 8 and
// 30: 1.3e-7, 1.6e-7 and 2.1e-7; that one's 1.3e-7, 4.5e-7 and 1.4e-6).
__device__ __forceinline__ float sigmoid1(float z) {
  const float hi = -1.44269504f * z, lo = fmaf(-1.44269504f, z, -hi) - 1.92596300e-8f * z;
  const float p = __builtin_amdgcn_exp2f(hi);
  const bool in = fabsf(hi) < 126.f;
  const float d = 1.f + (in ? fmaf(p, 0.69314718f * lo, p) : p);
  const float q = __builtin_amdgcn_rcpf(d);
  return in ? fmaf(fmaf(-d, q, 1.f), q, q) : q;  // (at either end, and of NaN, 1 / (1 + p) as it is)
}

// The even lane's value, in both lanes of a pair
__device__ __forceinline__ double of_even(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_mov_dpp((int)b, 0xa0, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xa0, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// 2^-(hi + lo)
__device__ __forceinline__ float exp2m(float hi, float lo) {
  const float p = __builtin_amdgcn_exp2f(-hi);
  return fmaf(p, -0.69314718f * lo, p);
}

// Bound by its elementwise instructions (900 a wave with the sums in fp64, 53 matrix instructions), four workgroups a CU: 144
// -> 99 us at 4001 tokens of 32 heads, 281 MB written.  The sums went through two of the four waves, as did the
// substitution, one column a thread with its factors handed out lane by lane (1450 instructions in those two waves).
__global__ void __launch_bounds__(256, 4) delta_form_kernel(FormArgs g) {
  constexpr int LD = kD + kPad;
  // four workgroups fit a CU's LDS
  __shared__ __attribute__((aligned(16))) float m[4][kC][LD];            // U (then U'), R, B, K
  __shared__ __attribute__((aligned(16))) float gram[4][kC][kC + kPad];  // U B^T, U K^T (below the diagonal; then G), R B^T, R K^T
  __shared__ __attribute__((aligned(16))) float p16[kD];
  float(*pw)[LD] = m[3];  // minus the decays' logarithms
  const int tid = threadIdx.x, h = blockIdx.x % g.H, ci = blockIdx.x / g.H;
  int s = 0;
  for (int lo = 0, hi = g.n_seq; lo < hi;) {  // the last sequence that starts at or before the chunk
    const int mid = (lo + hi) >> 1;
    if (first_chunk(g.seq_rows, mid) <= ci) s = mid, lo = mid + 1;
    else hi = mid;
  }
  const int t0 = (ci - first_chunk(g.seq_rows, s)) * kC, r0 = g.seq_rows[s] + t0, n = g.seq_rows[s + 1] - r0;
  const int slot = g.slots[s];
  if (t0 < 0 || n <= 0 || t0 + n < kLong || g.seq_rows[s] < 0 || g.seq_rows[s + 1] > g.T || slot < 0 || slot >= g.n_slots)
    return;
  // ---- a thread per token and eight channels
  const int t = tid >> 4, c0 = (tid & 15) * 8;
  float u[8], b[8], kk[8], rr[8];
  if (t < n) {
    const int64_t row = r0 + t, col = (int64_t)h * kD + c0;
    float al[8], wl[8], ss = 0.f;
    VecIO<bf16_t, 8>::ld(g.k + row * g.ks + col, kk);
    VecIO<bf16_t, 8>::ld(g.r + row * g.rs + col, rr);
    VecIO<bf16_t, 8>::ld(g.a + row * g.as + col, al);
    VecIO<bf16_t, 8>::ld(g.w + row * g.wst + col, wl);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += kk[e] * kk[e];
    const float inv = rsqrtf(group_sum<16>(ss) + g.key_eps);
    const Range abr = range(g.a_bias, g.a_bias ? 4 * kD * g.H : 0), wbr = range(g.w_bias, g.w_bias ? 4 * kD * g.H : 0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const f32x4 ab = get4(abr, 4 * (uint32_t)col, 16 * q), wb = get4(wbr, 4 * (uint32_t)col, 16 * q);  // (0 without a bias)
      f32x4 dec;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e = 4 * q + i;
        u[e] = kk[e] * inv;
        b[e] = sigmoid1(al[e] + ab[i]) * u[e];
        dec[i] = g.decay_scale * sigmoid1(wl[e] + wb[i]);
      }
      *reinterpret_cast<f32x4*>(&pw[t][c0 + 4 * q]) = dec;
    }
  } else {  // behind the sequence's end: nothing read, nothing removed, nothing added
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u[e] = b[e] = kk[e] = rr[e] = 0.f;
      pw[t][c0 + e] = 0.f;
    }
  }
  __syncthreads();
  // Every product of decays is 2^-(a difference of sums), its sums hi + lo: rounded once.  Products of rounded decays
  // would drift token by token, and the form would be less exact than the one that takes the tokens in order.
  {
    const int c = tid >> 1, first = tid & 1 ? 8 : 0;  // two threads a channel, eight tokens each
    double sum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double x = pw[first + i][c];
      sum[i] = i ? fma(x, 1.4426950408889634, sum[i - 1]) : x * 1.4426950408889634;
    }
    const double half = of_even(sum[7]), before = first ? half : 0.0;  // (every lane asks: one that is off answers nothing)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sum[i] += before;
      const float hi = (float)sum[i];
      m[0][first + i][c] = hi;
      m[1][first + i][c] = (float)(sum[i] - (double)hi);
      if (i == 7 && first) p16[c] = exp2m(hi, (float)(sum[i] - (double)hi));
    }
  }
  __syncthreads();
  float k2[8], b2[8];  // K'' and B''
  f32x4 x[4][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = c0 + 4 * j;
    auto at = [&](int half, int i) { return *reinterpret_cast<const f32x4*>(&m[half][i][c]); };
    const f32x4 hi = at(0, t), lo = at(1, t), hi0 = at(0, max(t - 1, 0)), lo0 = at(1, max(t - 1, 0));
    const f32x4 end = at(0, kC - 1), endl = at(1, kC - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = 4 * j + i;
      const float ip = exp2m(-hi[i], -lo[i]), dh = end[i] - hi[i];
      // (what the difference of the his rounds off, exactly)
      const float q = exp2m(dh, ((end[i] - dh) - hi[i]) + (endl[i] - lo[i]));
      x[0][j][i] = t ? u[e] * exp2m(hi0[i], lo0[i]) : u[e];
      x[1][j][i] = rr[e] * exp2m(hi[i], lo[i]);
      x[2][j][i] = b[e] * ip;
      x[3][j][i] = kk[e] * ip;
      k2[e] = kk[e] * q;
      b2[e] = b[e] * q;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 2; ++e) *reinterpret_cast<f32x4*>(&m[i][t][c0 + 4 * e]) = x[i][e];
  __syncthreads();
  // ---- the four products of 16 x 16 over the channels, one a wave (slot g of instruction (cb, i): channel 16 cb + 4 g + i)
  const int w = tid >> 6, lane = tid & 63, l16 = lane & 15, g4 = lane >> 4;
  {
    const float(*A)[LD] = m[w >> 1];
    const float(*B)[LD] = m[2 + (w & 1)];
    f32x4 acc[8];  // short chains: the longer the chain the more of its sum is rounded away
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cb = 0; cb < kD / 16; ++cb) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&A[l16][16 * cb + 4 * g4]);
      const f32x4 y = *reinterpret_cast<const f32x4*>(&B[l16][16 * cb + 4 * g4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i + 4 * (cb & 1)] = mma1(x[i], y[i], acc[i + 4 * (cb & 1)]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += acc[i + 4];
    acc[0] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tt = 4 * g4 + i;  // row tt, column l16
      gram[w][tt][l16] = l16 < tt || (w >= 2 && l16 == tt) ? acc[0][i] : 0.f;
    }
  }
  __syncthreads();
  float* o = g.ws + ((int64_t)ci * g.H + h) * kChunkFloats;
  // ---- K'' and B'' by channel (through the places of B and K, which are done): four tokens a thread, neighbouring
  // threads on neighbouring pieces
#pragma unroll
  for (int e = 0; e < 8; e += 4) {
    *reinterpret_cast<f32x4*>(&m[2][t][c0 + e]) = f32x4{b2[e], b2[e + 1], b2[e + 2], b2[e + 3]};
    *reinterpret_cast<f32x4*>(&m[3][t][c0 + e]) = f32x4{k2[e], k2[e + 1], k2[e + 2], k2[e + 3]};
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int it = tid + 256 * (k & 1), ch = (it >> 6) * 16 + l16, q = g4;
    const float(*src)[LD] = m[3 - (k >> 1)];
    *reinterpret_cast<f32x4*>(o + (2 + (k >> 1)) * kMat + 4 * it) =
        f32x4{src[q][ch], src[4 + q][ch], src[8 + q][ch], src[12 + q][ch]};
  }
  if (tid < kD) o[4 * kMat + 2 * kC * kC + tid] = p16[tid];
  // ---- [U | G] to [U' | G]: forward substitution by blocks of 16 columns, the waves' own to the end: blocks w and w + 4 of
  // U, G wave 0's.  Tokens 4 p .. 4 p + 3 lie in the lanes with g4 = p, which take them from each other; the rows behind lose
  // them in one matrix instruction, its factors below the block of four only.
  f32x4 low[3], take;
#pragma unroll
  for (int i = 0; i < 3; ++i) low[i] = *reinterpret_cast<const f32x4*>(&gram[0][4 * g4 + 1 + i][4 * g4]);
#pragma unroll
  for (int p = 0; p < 3; ++p) take[p] = l16 > 4 * p + 3 ? -gram[0][l16][4 * p + g4] : 0.f;
  // R' and H: what tril(R B^T) takes of U' and G (slot g of instruction i: token 4 g + i)
  const f32x4 rb = -*reinterpret_cast<const f32x4*>(&gram[2][l16][4 * g4]);
  auto solve = [&](float* at, int ld, f32x4 r) __attribute__((always_inline)) {  // at: the block, r: its rows of R or H
    f32x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = at[(4 * g4 + i) * ld + l16];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (g4 == p) {
        y[1] = fmaf(-low[0][0], y[0], y[1]);
        y[2] = fmaf(-low[1][1], y[1], fmaf(-low[1][0], y[0], y[2]));
        y[3] = fmaf(-low[2][2], y[2], fmaf(-low[2][1], y[1], fmaf(-low[2][0], y[0], y[3])));
#pragma unroll
        for (int i = 0; i < 4; ++i) at[(4 * p + i) * ld + l16] = y[i];
      }
      asm volatile("" ::: "memory");  // (a wave's LDS accesses go in order; other lanes read what this one wrote)
      if (p < 3) y = mma1(take[p], at[(4 * p + g4) * ld + l16], y);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) r = mma1(at[(4 * g4 + i) * ld + l16], rb[i], r);
    return r;
  };
#pragma unroll
  for (int cb = w; cb < kD / 16; cb += 4) {
    const f32x4 r = solve(&m[0][0][16 * cb], LD, *reinterpret_cast<const f32x4*>(&m[1][l16][16 * cb + 4 * g4]));
    float* to = o + 4 * (64 * cb + lane);
    *reinterpret_cast<f32x4*>(to) = *reinterpret_cast<const f32x4*>(&m[0][place(l16)][16 * cb + 4 * g4]);
    *reinterpret_cast<f32x4*>(to + kMat) = r;
  }
  if (w == 0) {
    const f32x4 r = solve(&gram[1][0][0], kC + kPad, *reinterpret_cast<const f32x4*>(&gram[3][l16][4 * g4]));
    float* to = o + 4 * kMat + 64 * g4 + l16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      to[16 * i] = gram[1][place(l16)][4 * g4 + i];
      to[kC * kC + 16 * i] = r[i];
    }
  }
}

struct ChunkArgs {
  DeltaArgs tok;  // the same rows token by token
  float* out;     // [T, H * dv]
  float* state;  // [slots, H, dv, 128]
  const float* ws;
  const bf16_t* v;
  int64_t vs;
  const int64_t* pos;
  const int* seq_rows;
  const int* slots;
  int n_seq, n_slots, T, H, dv;
};

template <int NB> struct Frags {
  f32x4 u[2], r[2], k[2], b[2], p[2];
  float g, h;
  uint32_t v[NB][4];  // rows g4, 4 + g4, 8 + g4 and 12 + g4 of V; bf16 bits as loaded: a conversion here would wait for the load
};

// NB: blocks of 16 columns per workgroup; CT: columns per thread of the sequences that go token by token
template <int NB, int CT>
__global__ void __launch_bounds__(256, NB == 1 ? 3 : 2) delta_chunk_kernel(ChunkArgs g) {
  struct Parts {
    __attribute__((aligned(16))) f32x4 x[2][4][NB][64];  // parts of X
    float o[2][4][NB][4][64];                            // parts of O, by accumulator register
  };
  __shared__ union {
    Parts parts;
    DeltaLds<8, 256, CT> tok;
  } lds;
  auto& px = lds.parts.x;
  auto& po = lds.parts.o;
  const int nb = g.dv / (16 * NB);
  // the column blocks of a (sequence, head) read the same chunks: neighbours on one XCD (blocks go out round robin)
  const int id = blockIdx.x, sh = id / (8 * nb) * 8 + id % 8, blk = id / 8 % nb;
  if (sh >= g.n_seq * g.H) return;
  const int h = sh % g.H;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // In order up to 16 sequences: 20 tokens beside 31 decode rows 45 us as they come and 57 in order, 24 prompts of 40 122 and
  // 140, four of 2000 together beside 20 decode rows 180 and 193.
  const auto [r0, n, slot, s] = by_length<true>(g.seq_rows, g.slots, g.n_seq, sh / g.H, 1, 16);
  if (n <= 0 || r0 < 0 || r0 + n > g.T) return;
  const int col0 = h * g.dv + blk * 16 * NB;
  if (slot < 0 || slot >= g.n_slots) {  // padding rows: a defined result, no state
    for (int i = threadIdx.x; i < n * 16 * NB; i += 256)
      g.out[(int64_t)(r0 + i / (16 * NB)) * g.H * g.dv + col0 + i % (16 * NB)] = 0.f;
    return;
  }
  if (n < kLong) {
    // as many columns as the threads take at once, and other workgroups of every sequence and head: they are dealt out to
    // the chip in turn, and every fourth of them would lie in a quarter of it
    constexpr int W = 32 * CT;
    const int c0 = (blk + sh / 8) % nb * W;
    if (c0 < g.dv) delta_tokens<bf16_t, 8, 256, CT, true>(g.tok, lds.tok, r0, n, h, slot, c0, min(g.dv, c0 + W));
    return;
  }
  // S: channels 32 w + 16 cb + 4 g4 + i of column l16 of every block
  float* sp = g.state + (((int64_t)slot * g.H + h) * g.dv + blk * 16 * NB + l16) * kD + 32 * w + 4 * g4;
  f32x4 S[NB][2];
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
      S[q][cb] = g.pos[r0] != 0 ? *reinterpret_cast<const f32x4*>(sp + q * 16 * kD + 16 * cb) : f32x4{0.f, 0.f, 0.f, 0.f};
  // uniform bases and 32-bit lane offsets: the chain of a chunk has no time for 64-bit address arithmetic
  const int64_t stride = (int64_t)g.H * kChunkFloats * 4;
  const char* wp = (const char*)(g.ws + ((int64_t)first_chunk(g.seq_rows, s) * g.H + h) * kChunkFloats);
  const char* vp = (const char*)(g.v + (int64_t)r0 * g.vs + col0);
  const uint32_t f_off = 16u * (128 * w + lane), p_off = 4u * (32 * w + 4 * g4), sq_off = 4u * (64 * w + lane), vs2 = 2u * (uint32_t)g.vs;
  const int nc = (n + kC - 1) / kC;
  const uint32_t mine[4] = {w == 0 ? ~0u : 0u, w == 1 ? ~0u : 0u, w == 2 ? ~0u : 0u, w == 3 ? ~0u : 0u};  // the wave's quarter
  uint32_t v_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v_off[i] = (g4 + 4 * i) * vs2 + 2u * l16;
  auto load = [&](Frags<NB>& f, int c) {
    const Range p = range(wp + c * stride, kChunkFloats * 4);
    const Range vr = range(vp + (int64_t)c * kC * vs2, (uint32_t)(min(n - c * kC, kC) - 1) * vs2 + 32 * NB);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      f.u[cb] = get4(p, f_off, 1024 * cb);
      f.r[cb] = get4(p, f_off, 4 * kMat + 1024 * cb);
      f.k[cb] = get4(p, f_off, 8 * kMat + 1024 * cb);
      f.b[cb] = get4(p, f_off, 12 * kMat + 1024 * cb);
      f.p[cb] = get4(p, p_off, 16 * kMat + 8 * kC * kC + 64 * cb);
    }
    f.g = get1(p, sq_off, 16 * kMat);
    f.h = get1(p, sq_off, 16 * kMat + 4 * kC * kC);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < NB; ++q) f.v[q][i] = get_half(vr, v_off[i], 32 * q);
  };
  char* op = (char*)(g.out + (int64_t)r0 * g.H * g.dv + col0);
  const uint32_t out_row = 4u * (uint32_t)(g.H * g.dv), o_off = (4 * g4 + w) * out_row + 4u * l16;
  bool finite = true;
  // The wave's row of each group of four, from the parts that the last chunk's end left
  auto finish = [&](int c, int buf) {
    const Range o4 = range(op + (int64_t)c * kC * out_row, (uint32_t)(min(n - c * kC, kC) - 1) * out_row + 64 * NB);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const float o = (po[buf][0][q][w][lane] + po[buf][1][q][w][lane]) + (po[buf][2][q][w][lane] + po[buf][3][q][w][lane]);
      put1(o4, o_off, 64 * q, o);
      finite = finite && fabsf(o) < INFINITY;
    }
  };
  auto step = [&](const Frags<NB>& f, int c, Frags<NB>& next, int cn) {
    const int buf = c & 1;
    __builtin_amdgcn_sched_barrier(0);  // (a load's first use may not move in front of the step that it is for)
    load(next, min(cn, nc - 1));  // (always a load, the last chunk again: the waits stay counts)
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    float v[NB][4], vw[NB];
    f32x4 X[NB][2], O[NB][2], N[NB][2];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[q][i] = bf16lo(f.v[q][i]);
      vw[q] = __uint_as_float(__float_as_uint(v[q][0]) & mine[0] | __float_as_uint(v[q][1]) & mine[1] |
                              __float_as_uint(v[q][2]) & mine[2] | __float_as_uint(v[q][3]) & mine[3]);
      X[q][0] = X[q][1] = O[q][0] = O[q][1] = zero;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int q = 0; q < NB; ++q) X[q][cb] = mma1(f.u[cb][i], S[q][cb][i], X[q][cb]);
#pragma unroll
    for (int q = 0; q < NB; ++q) X[q][0] = mma1(f.g, vw[q], X[q][0]);  // a quarter of G V each wave, the larger part last
#pragma unroll
    for (int q = 0; q < NB; ++q) px[buf][w][q][lane] = X[q][0] + X[q][1];
#pragma unroll
    for (int i = 0; i < 8 * NB; ++i) {  // a load or two issue while the matrix instruction in front of them runs
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();  // (a buffer is written again two chunks on, when its readers have met another barrier)
    f32x4 xp[NB][4];
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) xp[q][k] = px[buf][k][q][lane];
    finish(max(c - 1, 0), 1 - buf);  // (in front of the second chunk zeros, which the first chunk's rows replace)
    __builtin_amdgcn_sched_group_barrier(0x100, 4 * NB, 0);
    // the products that need no other wave's part, while theirs arrive
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          N[q][cb] = mma1(f.k[cb][i], v[q][i], i ? N[q][cb] : zero);
          O[q][cb] = mma1(f.r[cb][i], S[q][cb][i], O[q][cb]);
        }
#pragma unroll
    for (int q = 0; q < NB; ++q) O[q][0] = mma1(f.h, vw[q], O[q][0]);
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) N[q][cb][i] = fmaf(S[q][cb][i], f.p[cb][i], N[q][cb][i]);
    f32x4 xn[NB], M[NB][2];  // (sums of their own: into diag(P) S they would be rounded at its size at every token)
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) xn[q][i] = (xp[q][0][i] + xp[q][1][i]) + (xp[q][2][i] + xp[q][3][i]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int q = 0; q < NB; ++q) M[q][cb] = mma1(f.b[cb][i], xn[q][i], i ? M[q][cb] : zero);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
#pragma unroll
      for (int i = 0; i < 4; ++i) po[buf][w][q][i][lane] = O[q][0][i] + O[q][1][i];  // (joined behind the next barrier)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[q][cb][i] = N[q][cb][i] - M[q][cb][i];
    }
  };
  Frags<NB> f0, f1;  // (two chunks ahead: a workgroup fewer per CU, 1 to 4 % slower)
  load(f0, 0);
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) po[1][w][q][i][lane] = 0.f;
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): what is pending here the compiler would wait for in every turn
  for (int c = 0; c < nc; c += 2) {
    step(f0, c, f1, c + 1);
    if (c + 1 < nc) step(f1, c + 1, f0, c + 2);
  }
  lds_barrier();
  finish(nc - 1, (nc - 1) & 1);
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) finite = finite && fabsf(S[q][cb][i]) < INFINITY;
  if (__syncthreads_or(!finite)) {  // (also waits for the rows stored above)
    delta_tokens<bf16_t, 8, 256, CT, true>(g.tok, lds.tok, r0, n, h, slot, blk * 16 * NB, (blk + 1) * 16 * NB);
    return;
  }
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) *reinterpret_cast<f32x4*>(sp + q * 16 * kD + 16 * cb) = S[q][cb];
}

}  // namespace

extern "C" {

// Floats of workspace of the chunked form for these rows (named by seq_rows), 0 where the token-by-token form takes all of
// them: bf16 rows, enough for a long sequence (a decode step has no seq_rows at all), keys of 128 channels, whole blocks of
// 16 value columns, decays whose product over a chunk stays far inside fp32, 16-byte aligned rows (`ptrs`, `strides`: those
// of r, k, a, w and the state's pointer, or-ed), a chunk's rows of v and of the result within 32-bit byte offsets (`vs`: v's
// row stride).
int64_t dxm_delta_chunk_floats(int T_, int n_seq, int H, int dk, int dv, int f32, float decay_scale, int64_t ptrs,
                               int64_t strides, int64_t vs) {
  if (vs < 0 || vs > (1 << 27) || (int64_t)H * dv > (1 << 26)) return 0;
  if (f32 || dk != kD || dv % 16 || dv < 16 || ptrs % 16 || strides % 8 || !(decay_scale >= -1.f && decay_scale <= 1.f))
    return 0;
  const int64_t chunks = T_ / kC + std::min(n_seq, T_ / kLong);
  if (T_ < kLong || chunks * H > 0x7fffffff || H > 65535 ||
      (int64_t)n_seq * H * (dv / 16) > (1 << 30))
    return 0;
  return chunks * H * kChunkFloats;
}

int dxm_delta_chunk(float* out, float* state, int n_slots, float* ws, const void* r, int64_t rs, const void* k, int64_t ks,
                    const void* v, int64_t vs, const void* a, int64_t as, const void* w, int64_t wst, const float* a_bias,
                    const float* w_bias, float decay_scale, float key_eps, const int64_t* pos, const int* seq_rows,
                    const int* slots, int n_seq, int T_, int H, int dv, hipStream_t st) {
  if (n_seq <= 0 || T_ <= 0) return 0;
  if (H < 1 || n_slots < 1 || !out || !state || !ws || !pos || !slots || !seq_rows) return 3;
  const int64_t ptrs = (int64_t)(uintptr_t)r | (int64_t)(uintptr_t)k | (int64_t)(uintptr_t)a | (int64_t)(uintptr_t)w |
                       (int64_t)(uintptr_t)state | (int64_t)(uintptr_t)ws;
  if (!dxm_delta_chunk_floats(T_, n_seq, H, kD, dv, 0, decay_scale, ptrs, rs | ks | as | wst, vs)) return 2;
  FormArgs f{ws, (const bf16_t*)r, (const bf16_t*)k, (const bf16_t*)a, (const bf16_t*)w, rs, ks, as, wst, a_bias, w_bias,
             seq_rows, slots, decay_scale, key_eps, n_seq, n_slots, T_, H};
  hipLaunchKernelGGL(delta_form_kernel, dim3((unsigned)((T_ / kC + std::min(n_seq, T_ / kLong)) * H)), dim3(256), 0, st, f);
  DeltaArgs d{};
  d.out = out, d.state = state, d.r = r, d.k = k, d.v = v, d.rs = rs, d.ks = ks, d.vs = vs, d.pos = pos;
  d.seq_rows = seq_rows, d.slots = slots, d.n_slots = n_slots, d.T = T_, d.H = H, d.dk = kD, d.dv = dv;
  d.a = a, d.w = w, d.as = as, d.wst = wst, d.a_bias = a_bias, d.w_bias = w_bias;
  d.decay_scale = decay_scale, d.key_eps = key_eps;
  ChunkArgs c{d, out, state, ws, (const bf16_t*)v, vs, pos, seq_rows, slots, n_seq, n_slots, T_, H, dv};
  const int64_t heads = ((int64_t)n_seq * H + 7) / 8 * 8;
  // Long sequences gain nothing from two column blocks a workgroup (one / two, us, whole layer of 32 heads: three prompts of
  // 12003 tokens together 904 / 1095, four of 3000 238 / 256, six of 5000 385 / 381); short ones in great numbers do, in tiles
  // of four columns a thread by four times fewer workgroups (32 prompts of 16 tokens 131 / 116, 64 of them 249 / 196, one of
  // 600 beside 100 decode rows 203 / 195).  Up to about a thousand (sequence, head) there are too few of them for that: 600
  // tokens beside 12, 30 and 48 decode rows 72 / 93, 102 / 103 and 128 / 128, three 20-token prompts beside 12 40 / 52, 16
  // prompts of 16 tokens 64 / 66.
  if (dv % 32 == 0 && heads >= 1024)
    hipLaunchKernelGGL((delta_chunk_kernel<2, 4>), dim3((unsigned)(heads * (dv / 32))), dim3(256), 0, st, c);
  else
    hipLaunchKernelGGL((delta_chunk_kernel<1, 1>), dim3((unsigned)(heads * (dv / 16))), dim3(256), 0, st, c);
  DX_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
