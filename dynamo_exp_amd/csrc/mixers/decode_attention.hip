// Attention of decode rows (one token a row) over pages of whole 32-key tiles, for gfx950: heads of 128 columns with
// values of 128, pairs of maps with values of 256, or one shared row of 256 columns per key that is key and value (its
// first 192 columns, or all).  Every score form of tile_attention.hip.  Scores and sums are fp32, weights enter the value
// product as the sum of two bf16 numbers.
//
// A workgroup (4 waves) serves one (row, key / value group, part of the keys): up to 16 query vectors of the group (a
// shared row: 16 QB) are the columns of 16x16x32 products.  Both maps of a two-map layer are in one workgroup, so their
// common values are read once.  The waves take the part's tiles in turn and run on their own: a wave brings its tiles
// into LDS of its own by DMA (buffer loads: with global_load_lds no wait for an LDS read can be partial) and waits for its
// own loads only, so there is no barrier until the end, where the four partial results are joined in LDS.  Fragments are
// asked for six to eight ahead.  Keys and values have a buffer each, refilled as soon as its product is done; a
// shared row has two buffers in turn.  V^T fragments come from the row-major image by ds_read_b64_tr_b16.
// One part: the result goes out finished; several: partials to the workspace that merge_parts joins.
// Bound by memory at many rows and by latency at few (position, block table, first tile, join: 7 us of a launch with one
// tile a wave).  Two layers in a graph with their joins, us: two maps, window 1024 + 64, 48 rows 98 -> 86 nontemporally -> 84.5,
// shared row 256 / 192 causal to 4000, 33 rows 53 with fragments read one product ahead -> 49.5 -> 44.5, to 2500, 100 rows 79 ->
// 70.5 -> 63; 256 / 256 window 1024, 20 rows 41 -> 37.4 -> 33.8; two maps, 2 rows of 142 25.3 -> 24.2 (the last step each time:
// accumulators that are not copied between the two kinds of registers, a build option; the join's reads all at once instead of
// column block by column block, 3400 cycles before; both blocks of query vectors through the softmax side by side).  Parts dealt out by the rows' lengths
// instead of equally: 33 rows the same (memory is as busy while the short rows last), 41 rows of up to 281 keys 60 -> 64.
// (The one-wave forms it took over from, register-staged group_decode, stream_decode, latent_decode: 270 and 92.)
#include <algorithm>
#include <type_traits>

#include "stream_attention.h"

namespace {

struct DecodeArgs {
  void* out;  // [rows, n_qh, DV]
  float* ws;  // parts > 1: [rows, n_qh, parts, 2 + DV]
  const bf16_t* q;
  int64_t q_stride;
  const bf16_t* kc;
  const bf16_t* vc;
  const int64_t* pos;
  const int* seq;  // null: row i is sequence i
  const int* bt;
  int bt_stride, bs_shift;
  int n_qh, maps, group;
  int Wk, Wv;
  float scale;
  int mask, size, parts;
  float softcap;    // 0: none
  const float* r1;  // [n_qh], null: no distance penalty
  const float* r2;
  const float* hbias;
  const bf16_t* gate;
  int64_t gate_stride;
  int keep;
  const float* sink;
  int out_f32;
  int kept_tiles;  // a row of more tiles does not keep its lines
};

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
// A launch that reads more of the cache than this asks for it nontemporally: each line is read once, whole, and behind so
// many no cache holds much of it for the next step.  Less is kept.  Of a single layer that is repeated: each row takes the
// others to be as long as itself, which a window's mostly are; other rows' lengths differ, so their line lies higher.  One
// layer's repeated launch, kept / not, us: plain heads, 51 / 85 / 128 MB 20.0 / 21.1, 26.5 / 26.9, 37.3 / 33.6; capped,
// window 1024, 84 / 126 / 200 MB 27.5 / 27.8, 34.4 / 31.8, 50.1 / 42.8; rows in chunks of 2048, the longest 131 of 67 MB
// 23.5 / 26.3.  Two launches of other layers: two maps, 190 MB 97.4 / 86.5; plain heads, 300 MB 137 / 122 (5.0 TB/s).  In a
// step of several layers nothing of one is left when it comes round again: eight layers, a layer, two maps, 62 / 89 MB 24.9
// / 23.8, 28.6 / 27.3; capped, 64 / 85 MB 20.5 / 18.7, 26.3 / 24.1; plain heads, 65 / 120 MB 16.9 / 16.5, 24.7 / 22.8.  A
// shared row (one cache for all heads) gains nothing: 46.9 / 48.2 and 64.9 / 62.8 for two launches of 40 and 100 rows.
constexpr int64_t kKeptWindow = 96 << 20, kKept = 160 << 20, kKeptLayers = 48 << 20;
constexpr int kTile = 32;       // keys per tile
constexpr float kDefer = 8.f;   // log2 units that a score may exceed the running maximum by (weights are bf16 pairs)
enum { kPlain = 0, kTerms = 1, kSigmoid = 2 };
// metadata that no kernel in flight writes: scalar loads
typedef const __attribute__((address_space(4))) int* scalar_int;
typedef const __attribute__((address_space(4))) int64_t* scalar_long;

// the wave's own DMA: all but the newest N instructions have landed.  (The builtin, which the compiler counts itself:
// behind a wait it does not know it would put a full one in front of the next LDS read.)
template <int N> __device__ __forceinline__ void dma_wait() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));  // vmcnt alone
  asm volatile("" ::: "memory");
}
// every LDS read issued so far has returned: its buffer may be refilled
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// over the four 16-lane groups of a wave
__device__ __forceinline__ float groups_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float groups_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// D: key columns, DV: value columns, MAPS: maps a workgroup serves, SAME: the value is the first DV columns of the
// key's row, QB: blocks of 16 query vectors, LONG: some rows may not keep their lines (both forms of the body: a choice at each
// tile costs 3 to 6 %; rows that are known to be short take the instance without it, 1 %)
template <int D, int DV, int MAPS, bool SAME, int MODE, int QB, bool LONG>
__global__ void __launch_bounds__(256, SAME || MAPS == 2 ? 1 : 2) decode_attention_kernel(DecodeArgs a) {
  constexpr int KS = D / 32, NC = DV / 16, KB = 2 * D * MAPS, VB = SAME ? KB : 2 * DV;  // row bytes of the images
  constexpr int KN = kTile * KB / 1024, VN = SAME ? KN : kTile * VB / 1024;             // DMA instructions per tile
  constexpr int GR = MAPS == 2 ? 8 : 16;  // columns per map
  static_assert(!SAME || (MAPS == 1 && D == 256), "one shared row");
  // a wave's keys and values; a shared row: its tiles with even / odd turn
  constexpr int kImg = kTile * (KB + VB), kVal = kTile * KB;
  __shared__ __attribute__((aligned(16))) char img[4][kImg];
  __shared__ float ml[2][4][QB][16];
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.y, part = blockIdx.z;
  const int p = (int)((scalar_long)a.pos)[row];
  const int lo = first_key(p, a.mask, a.size);
  const int keep = a.mask == 1 ? a.keep : 0, keeplo = min(keep, lo);  // (kept keys in front of the window)
  // tiles in order: those of the kept keys, then the mask's
  const int first = lo / kTile, kept = min((keep + kTile - 1) / kTile, first), total = kept + p / kTile - first + 1;
  // at least two tiles a wave, four of a long context: shorter parts cost more in the join than they gain
  const int tpp = max((total + a.parts - 1) / a.parts, max(8, min(16, total / 12))), i0 = part * tpp, i1 = min(i0 + tpp, total);
  const scalar_int bt = (scalar_int)(a.bt + (int64_t)(a.seq ? ((scalar_int)a.seq)[row] : row) * a.bt_stride);
  auto tile = [&](int i) { return i < kept ? i : first + i - kept; };
  // K head of the workgroup (of the first map), its key / value group
  const int gm = SAME ? 0 : MAPS == 2 ? 2 * blockIdx.x : blockIdx.x, g = SAME ? 0 : gm / a.maps, m = gm - g * a.maps;
  int qh[QB];
  bool okh[QB];
  float r1[QB], r2[QB], hb[QB];
  bf16x8_t qf[QB][KS];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int hi_ = SAME ? (int)blockIdx.x * 16 * QB + 16 * qb + c16 : c16 % GR;
    okh[qb] = hi_ < a.group;
    qh[qb] = (g * a.group + (okh[qb] ? hi_ : 0)) * a.maps + (MAPS == 2 ? c16 / GR : m);
    r1[qb] = MODE != kPlain && a.r1 ? a.r1[qh[qb]] : 0.f;
    r2[qb] = MODE != kPlain && a.r1 ? a.r2[qh[qb]] : 0.f;
    hb[qb] = MODE == kSigmoid && a.hbias ? a.hbias[qh[qb]] * kLog2e : 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const raw_u32x4 zero{0u, 0u, 0u, 0u};
      qf[qb][ks] = __builtin_bit_cast(bf16x8_t, okh[qb] ? *reinterpret_cast<const raw_u32x4*>(
          a.q + (int64_t)row * a.q_stride + (int64_t)qh[qb] * D + 32 * ks + 8 * g4) : zero);
    }
  }
  if (i0 >= i1 && part > 0) {  // a part without a key: sum 0
    if (w == 0 && g4 == 0)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        if (okh[qb]) {
          float* ws = a.ws + (((int64_t)row * a.n_qh + qh[qb]) * a.parts + part) * (2 + DV);
          ws[0] = MODE == kSigmoid ? 0.f : -INFINITY;
          ws[1] = 0.f;
        }
    return;
  }
  const bf16_t* kc = a.kc + (int64_t)gm * D;
  const bf16_t* vc = a.vc + (int64_t)g * DV;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)&img[w][0];
  // Fragment addresses: step ks of the keys is an XOR with 64 ks away from the first (pieces 16 and up of a row: + 256
  // bytes), block cb of the values one with 32 cb; values 16 rows further: + 16 rows.
  uint32_t koff[4], voff_[8];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) koff[ks] = base + image_off<KB>(c16, 4 * ks + g4);
#pragma unroll
  for (int cb = 0; cb < 8; ++cb)
    voff_[cb] = base + (SAME ? 0 : kVal) + image_off<VB>(4 * g4 + (c16 >> 2), 2 * cb + ((lane & 3) >> 1)) + 8 * (lane & 1);
  // The DMA: source of an image's k-th KB, from the tile's first row.  Rows behind the query hold stale values, which must
  // not meet a zero weight: they lie outside the descriptor and arrive as zeros.
  auto source = [&](auto rb, int k, int width) {
    constexpr int CH = decltype(rb)::value / 16;
    const int r = k * (64 / CH) + lane / CH;
    return 2 * (r * width + 8 * ((lane % CH) ^ piece_xor(r)));
  };
  int ksrc[KN], vsrc[SAME ? 1 : VN];
#pragma unroll
  for (int k = 0; k < KN; ++k) ksrc[k] = source(std::integral_constant<int, KB>{}, k, a.Wk);
  if constexpr (!SAME)
#pragma unroll
    for (int k = 0; k < VN; ++k) vsrc[k] = source(std::integral_constant<int, VB>{}, k, a.Wv);
  auto slot = [&](int t) __attribute__((always_inline)) {
    const int j = t * kTile;
    return ((uint32_t)bt[j >> a.bs_shift] << a.bs_shift) + (j & ((1 << a.bs_shift) - 1));
  };
  auto body = [&](auto nt) __attribute__((always_inline)) {
    constexpr int NT = decltype(nt)::value ? 2 : 0;
    auto fetch_k = [&](uint32_t dst, int i) __attribute__((always_inline)) {
      const int t = tile(i), rows = min(p - t * kTile, kTile - 1);  // whole rows in front of the last one
      const bf16_t* from = kc + (uint64_t)slot(t) * (uint32_t)a.Wk;
#pragma unroll
      for (int k = 0; k < KN; ++k) dma16<NT>(from, 2 * rows * a.Wk + KB, ksrc[k], base + dst + k * 1024);
    };
    auto fetch_v = [&](int i) __attribute__((always_inline)) {
      const int t = tile(i), rows = min(p - t * kTile, kTile - 1);
      const bf16_t* from = vc + (uint64_t)slot(t) * (uint32_t)a.Wv;
      if constexpr (!SAME)
#pragma unroll
        for (int k = 0; k < VN; ++k) dma16<NT>(from, 2 * rows * a.Wv + VB, vsrc[k], base + kVal + k * 1024);
    };

    const float cap = a.softcap, inv_cap = MODE != kPlain && cap > 0.f ? 1.f / cap : 0.f;
    const bool terms = MODE != kPlain && (cap > 0.f || a.r1);
    const float sc = terms ? 1.f : a.scale * kLog2e;  // scores to log2 units
    float mx[QB], lsum[QB];
    f32x4 O[QB][NC];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      mx[qb] = -INFINITY;
      lsum[qb] = 0.f;
#pragma unroll
      for (int cb = 0; cb < NC; ++cb) O[qb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    f32x4 S[QB][2];  // scores: lane column = query vector, rows = keys 16 kb + 4 g4 + r
    constexpr int KF = 2 * KS * MAPS, KA = KF < 8 ? KF : 8;  // key fragments of a tile, of them asked for ahead
    constexpr int VA = NC < 6 ? NC : 6;                        // value fragments asked for ahead
    auto scores = [&](auto buf) __attribute__((always_inline)) {
      constexpr int at = decltype(buf)::value;
      auto kread = [&](int f) {  // fragment f: step f / (2 MAPS), 16 keys kb, map
        const int ks = f / (2 * MAPS), kb = f / MAPS % 2, mp = f % MAPS;
        return lds_frag(koff[ks & 3] + (at + kb * 16 * KB + 256 * (ks >> 2) + 256 * mp));
      };
      bf16x8_t kf[KA];
      f32x4 S1[2];
#pragma unroll
      for (int f = 0; f < KA; ++f) kf[f] = kread(f);
      __builtin_amdgcn_sched_group_barrier(0x100, KA, 0);
#pragma unroll
      for (int f = 0; f < KF; ++f) {
        const int ks = f / (2 * MAPS), kb = f / MAPS % 2;
        const bf16x8_t k = kf[f % KA];
        if (f + KA < KF) kf[f % KA] = kread(f + KA);
        const f32x4 zero{0.f, 0.f, 0.f, 0.f};
        if (f % MAPS == 0) {
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) S[qb][kb] = mma(k, qf[qb][ks], ks ? S[qb][kb] : zero);
          __builtin_amdgcn_sched_group_barrier(0x008, QB, 0);
        } else {
          S1[kb] = mma(k, qf[0][ks], ks ? S1[kb] : zero);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        if (f + KA < KF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      if constexpr (MAPS == 2) {  // every column keeps its own map's product
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[0][kb][r] = c16 < GR ? S[0][kb][r] : S1[kb][r];
      }
    };
    bf16x8_t Ph[QB], Pl[QB];
    auto softmax = [&](int t) __attribute__((always_inline)) {
      const int kt = t * kTile;
      // (bitwise: of the two ways of a || the compiler counts the longer one's instructions as a wait for the scores' last product)
      const bool edge = (kt + kTile - 1 > p) | ((kt < lo) & (kt + kTile > keep));
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        if (MODE != kPlain && terms) {  // final scores in log2 units
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float x = S[qb][kb][r] * a.scale;
              // cap * tanh(x / cap): tanh(y) = 1 - 2 / (1 + e^(2 y))
              x = cap > 0.f ? cap * kLog2e * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + fast_exp2(x * (2.f * kLog2e) * inv_cap)))
                            : x * kLog2e;
              if (a.r1) {
                const int dist = p - (kt + 16 * kb + 4 * g4 + r);
                x -= r1[qb] * __builtin_amdgcn_logf(1.f + r2[qb] * (float)max(dist, 0));
              }
              S[qb][kb][r] = x;
            }
        }
        if (edge) {
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int j = kt + 16 * kb + 4 * g4 + r;  // (bitwise: a compare and a select, no branches)
              const bool seen = ((unsigned)(j - lo) <= (unsigned)(p - lo)) | (j < keeplo);
              S[qb][kb][r] = seen ? S[qb][kb][r] : -INFINITY;
            }
        }
      }
      // (all blocks of query vectors behind one branch: with one for each their chains ran one after the other)
      float mu[QB], mn[QB];
      bool moved = false;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        mu[qb] = 0.f;
        if constexpr (MODE != kSigmoid) {
          float mloc = S[qb][0][0];
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, S[qb][kb][r]);
          const float tm = groups_max(mloc) * sc;  // (every tile holds a visible key)
          mn[qb] = tm > mx[qb] + kDefer ? tm : mx[qb];
          mu[qb] = mn[qb] == -INFINITY ? 0.f : mn[qb];
          moved |= mn[qb] != mx[qb];
        }
      }
      if (MODE != kSigmoid && __any(moved)) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          const float alpha = fast_exp2(mx[qb] - mu[qb]);
          lsum[qb] *= alpha;
#pragma unroll
          for (int cb = 0; cb < NC; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) O[qb][cb][r] *= alpha;
          mx[qb] = mn[qb];
        }
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        raw_u32x4 ph, pl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float wt[2];
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const float v = S[qb][e / 2][2 * (e % 2) + x];
            if constexpr (MODE == kSigmoid)  // an invisible key (-inf) weighs 0
              wt[x] = __builtin_amdgcn_rcpf(1.f + fast_exp2(-fmaf(v, sc, hb[qb])));
            else
              wt[x] = fast_exp2(fmaf(v, sc, -mu[qb]));
          }
          lsum[qb] += wt[0] + wt[1];
          ph[e] = pack_bf16x2(wt[0], wt[1]);
          pl[e] = pack_bf16x2(wt[0] - bf16lo(ph[e]), wt[1] - bf16hi(ph[e]));
        }
        Ph[qb] = __builtin_bit_cast(bf16x8_t, ph);
        Pl[qb] = __builtin_bit_cast(bf16x8_t, pl);
      }
    };
    bf16x8_t vf[VA];
    auto vread = [&](int at, int cb) __attribute__((always_inline)) {
      const uint32_t vp = voff_[cb & 7] + (at + 256 * (cb >> 3));
      const i16x4 l4 = read_tr16((const lds_i16x4*)(uintptr_t)vp);
      const i16x4 u4 = read_tr16((const lds_i16x4*)(uintptr_t)(vp + 16 * VB));
      return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(l4, u4, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto ahead = [&](auto buf) __attribute__((always_inline)) {  // the first value fragments
#pragma unroll
      for (int cb = 0; cb < VA; ++cb) vf[cb] = vread(decltype(buf)::value, cb);
    };
    auto values = [&](auto buf) __attribute__((always_inline)) {
#pragma unroll
      for (int cb = 0; cb < NC; ++cb) {
        const bf16x8_t v = vf[cb % VA];
        if (cb + VA < NC) vf[cb % VA] = vread(decltype(buf)::value, cb + VA);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          O[qb][cb] = mma(v, Ph[qb], O[qb][cb]);
          O[qb][cb] = mma(v, Pl[qb], O[qb][cb]);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * QB, 0);
        if (cb + VA < NC) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
    };
    typedef std::integral_constant<int, 0> K0;
    typedef std::integral_constant<int, kVal> K1;  // a shared row's second image
    int i = i0 + w;
    // (the loops hold no conditional DMA: the compiler's count of what is in flight stays exact, see dma_wait)
    if constexpr (SAME) {
      auto turn = [&](auto buf, int i) __attribute__((always_inline)) {
        scores(buf);
        ahead(buf);
        softmax(tile(i));
        values(buf);
        lds_wait();
      };
      if (i < i1) fetch_k(0, i);
      for (; i + 8 < i1; i += 8) {
        fetch_k(kVal, i + 4);
        dma_wait<KN>();
        turn(K0{}, i);
        fetch_k(0, i + 8);
        dma_wait<KN>();
        turn(K1{}, i + 4);
      }
      if (i + 4 < i1) {
        fetch_k(kVal, i + 4);
        dma_wait<KN>();
        turn(K0{}, i);
        dma_wait<0>();
        turn(K1{}, i + 4);
      } else if (i < i1) {
        dma_wait<0>();
        turn(K0{}, i);
      }
    } else if (i < i1) {
      // Score terms take so long that the values arrive meanwhile: their wait comes behind them.  Four layers with cap and penalty,
      // window 1024, us, in front / behind: 40 rows to 4000 171 / 163, 8 to 4594 61.5 / 57.9, 16 to 600 56.7 / 53.5 (with sigmoid
      // weights 40 rows 164 either way).  Not so for a wave's only tile, when nothing else is on its way: one row of 90 keys 23.5
      // in front, 24.2 behind.
      constexpr bool kLate = MODE == kTerms;
      fetch_k(0, i);
      fetch_v(i);
      for (; i + 4 < i1; i += 4) {
        dma_wait<VN>();  // the keys; the values may still fly
        scores(K0{});
        lds_wait();
        fetch_k(0, i + 4);
        if constexpr (kLate) softmax(tile(i));
        dma_wait<KN>();
        ahead(K0{});
        if constexpr (!kLate) softmax(tile(i));
        values(K0{});
        lds_wait();
        fetch_v(i + 4);
      }
      dma_wait<VN>();
      scores(K0{});
      const bool late = kLate && i != i0 + w;
      if (!late) {
        dma_wait<0>();
        ahead(K0{});
      }
      softmax(tile(i));
      if (late) {
        dma_wait<0>();
        ahead(K0{});
      }
      values(K0{});
    }
    // ---- join the waves
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float l = groups_sum(lsum[qb]);
      if (g4 == 0) {
        ml[0][w][qb][c16] = mx[qb];
        ml[1][w][qb][c16] = l;
      }
    }
    __syncthreads();  // (also: every wave is done with its images)
    float mt[QB], lt[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      mt[qb] = fmaxf(fmaxf(ml[0][0][qb][c16], ml[0][1][qb][c16]), fmaxf(ml[0][2][qb][c16], ml[0][3][qb][c16]));
      if (MODE == kSigmoid) mt[qb] = 0.f;
      lt[qb] = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {  // a wave without a tile: sum 0, maximum -inf (a NaN stays one)
        const float l = ml[1][v][qb][c16];
        lt[qb] += MODE == kSigmoid ? l : l != 0.f ? l * fast_exp2(ml[0][v][qb][c16] - mt[qb]) : 0.f;
      }
    }
    constexpr int kSlab = QB * NC * 64;  // f32x4 of a wave
    static_assert(4 * kSlab * 16 <= (int)sizeof(img), "partial results fit the images");
    auto slab = [&](int v) { return reinterpret_cast<f32x4*>(&img[0][0]) + v * kSlab; };
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float f = MODE == kSigmoid ? 1.f : mx[qb] == -INFINITY ? 0.f : fast_exp2(mx[qb] - mt[qb]);
#pragma unroll
      for (int cb = 0; cb < NC; ++cb)
        slab(w)[(qb * NC + cb) * 64 + lane] = f32x4{O[qb][cb][0] * f, O[qb][cb][1] * f, O[qb][cb][2] * f, O[qb][cb][3] * f};
    }
    __syncthreads();
    // the wave's blocks of 16 columns, every fourth: all reads on their way together
    constexpr int CW = NC / 4;
    f32x4 o[QB][CW];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int j = 0; j < CW; ++j) {
        const int at = (qb * NC + 4 * j + w) * 64 + lane;
        o[qb][j] = slab(0)[at];
#pragma unroll
        for (int v = 1; v < 4; ++v) o[qb][j] += slab(v)[at];
      }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      if (!okh[qb]) continue;
      float inv = 1.f;
      if (a.parts == 1) {
        if constexpr (MODE != kSigmoid) {
          float l = lt[qb];
          if (a.sink) l += fast_exp2(a.sink[qh[qb]] * kLog2e - mt[qb]);  // (finite: a row sees itself)
          inv = 1.f / l;
        }
        if (a.gate) inv /= 1.f + __expf(-bf16_to_f32(a.gate[(int64_t)row * a.gate_stride + qh[qb] / a.maps]));
      }
      const int64_t vrow = (int64_t)row * a.n_qh + qh[qb];
      float* ws = a.parts == 1 ? nullptr : a.ws + (vrow * a.parts + part) * (2 + DV);
      if (ws && w == 0 && g4 == 0) {
        ws[0] = mt[qb] * kLn2;
        ws[1] = MODE == kSigmoid ? 1.f : lt[qb];
      }
#pragma unroll
      for (int j = 0; j < CW; ++j) {
        const f32x4 x = o[qb][j];
        const int c = (4 * j + w) * 16 + 4 * g4;
        if (ws) {
          *reinterpret_cast<float2*>(ws + 2 + c) = float2{x[0], x[1]};
          *reinterpret_cast<float2*>(ws + 4 + c) = float2{x[2], x[3]};
        } else if (a.out_f32) {
          *reinterpret_cast<f32x4*>((float*)a.out + vrow * DV + c) = f32x4{x[0] * inv, x[1] * inv, x[2] * inv, x[3] * inv};
        } else {
          *reinterpret_cast<uint2*>((bf16_t*)a.out + vrow * DV + c) = uint2{pack_bf16x2(x[0] * inv, x[1] * inv),
                                                                            pack_bf16x2(x[2] * inv, x[3] * inv)};
        }
      }
    }
  };
  if constexpr (!LONG) body(std::false_type{});
  else if (total > a.kept_tiles) body(std::true_type{});
  else body(std::false_type{});
}

}  // namespace

extern "C" {

// 1 when the kernel has an instance for the heads; `same`: keys and values are one cache
int dxm_decode_attention_ok(int d, int dv, int n_qh, int maps, int group, int bs, int same, int terms, int sigmoid) {
  if (bs < kTile || (bs & (bs - 1)) || group < 1) return 0;
  if (same) return d == 256 && (dv == 192 || dv == 256) && maps == 1 && group == n_qh && !terms && !sigmoid;
  if (d == 128 && dv == 256) return maps == 2 && group <= 8 && !terms && !sigmoid;
  return d == 128 && dv == 128 && group <= 16;
}

// workgroups per row and part
static int decode_units(int n_qh, int group, int same, int dv) {
  if (same) return (n_qh + (n_qh > 16 ? 31 : 15)) / (n_qh > 16 ? 32 : 16);
  return n_qh / group / (dv == 256 ? 2 : 1);
}

// Parts worth launching.  Values of more than 128 columns fill a CU's LDS with one workgroup: as many as fit the chip
// at once, a second round costs more than a longer first one.  Heads of 128: two workgroups a CU, at least one each.
int dxm_decode_attention_parts(int rows, int n_qh, int group, int same, int dv) {
  const int units = std::max(1, rows * decode_units(n_qh, group, same, dv));
  return std::max(1, dv > 128 ? 256 / units : (512 + units - 1) / units);
}

int dxm_decode_attention(void* out, float* ws, const void* q, int64_t q_stride, const void* kc, const void* vc,
                         const int64_t* pos, const int* seq, const int* bt, int bt_stride, int bs, int rows, int n_qh,
                         int maps, int group, int d, int dv, int Wk, int Wv, float scale, int mask, int size, float softcap,
                         const float* r1, const float* r2, int wfn, const float* hbias, const void* gate,
                         int64_t gate_stride, int keep, const float* sink, int parts, int out_f32, int layers, hipStream_t st) {
  if (rows <= 0) return 0;
  const bool same = kc == vc, terms = softcap > 0.f || r1;
  if (softcap < 0.f || (r1 && !r2) || wfn < 0 || wfn > 1 || keep < 0 || (keep && mask != 1)) return 6;
  if (!dxm_decode_attention_ok(d, dv, n_qh, maps, group, bs, same, terms, wfn)) return 2;
  if (n_qh < 1 || maps < 1 || n_qh % maps || (n_qh / maps) % group || rows > 65535) return 1;
  if (mask < 0 || mask > 2 || (mask && size < 1) || parts < 1 || parts > 65535 || !(scale > 0.f)) return 3;
  if (!out || (parts > 1 && !ws) || Wk % 8 || Wv % 8 || q_stride % 8 || (uintptr_t)q % 16 || (uintptr_t)kc % 16 ||
      (uintptr_t)vc % 16 || (uintptr_t)out % 16 || (uintptr_t)ws % 8)
    return 4;
  // tiles a row may have at most (a window and the keys kept in front of it may each reach into two more), and of how many
  // rows still keep their lines
  const int64_t most = mask ? ((int64_t)size + keep) / kTile + 4 : (int64_t)bt_stride * bs / kTile;
  const int64_t kept = (layers > 1 ? kKeptLayers : mask == 1 ? kKeptWindow : kKept) / (2 * kTile * ((int64_t)Wk + Wv) * rows);
  const bool many = most > kept;
  DecodeArgs a{out, ws, (const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, pos, seq, bt, bt_stride,
               __builtin_ctz((unsigned)bs), n_qh, maps, group, Wk, Wv, scale, mask, size, parts, softcap, r1, r2, hbias,
               (const bf16_t*)gate, gate_stride, keep, sink, out_f32,
               (int)std::min<int64_t>(kept, INT32_MAX)};
  const dim3 grid(decode_units(n_qh, group, same, dv), rows, parts);
#define DECODE(...) hipLaunchKernelGGL((decode_attention_kernel<__VA_ARGS__>), grid, dim3(256), 0, st, a)
  if (same && dv == 192) {
    if (n_qh > 16) DECODE(256, 192, 1, true, kPlain, 2, false);
    else DECODE(256, 192, 1, true, kPlain, 1, false);
  } else if (same) {
    if (n_qh > 16) DECODE(256, 256, 1, true, kPlain, 2, false);
    else DECODE(256, 256, 1, true, kPlain, 1, false);
  } else if (dv == 256) {
    if (many) DECODE(128, 256, 2, false, kPlain, 1, true);
    else DECODE(128, 256, 2, false, kPlain, 1, false);
  } else if (wfn) {
    if (many) DECODE(128, 128, 1, false, kSigmoid, 1, true);
    else DECODE(128, 128, 1, false, kSigmoid, 1, false);
  } else if (terms) {
    if (many) DECODE(128, 128, 1, false, kTerms, 1, true);
    else DECODE(128, 128, 1, false, kTerms, 1, false);
  } else {
    if (many) DECODE(128, 128, 1, false, kPlain, 1, true);
    else DECODE(128, 128, 1, false, kPlain, 1, false);
  }
#undef DECODE
  DX_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
