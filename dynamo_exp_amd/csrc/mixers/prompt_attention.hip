// Attention of prompt rows over pages of whole 64-key tiles, for gfx950: heads of 128 columns (values of 128 or 256),
// or one shared row of 256 columns per key that is key and value (the first 192 or all of them the value).  Every
// score form of tile_attention.hip: causal, window (with kept first keys) and chunk masks, a tanh cap, a log-distance
// penalty, sigmoid weights, a sink, a gate per head.  Scores, weights and sums are fp32.
//
// A workgroup is four waves: HPW heads that share a key / value head times 4 / HPW blocks of 32 rows, a wave
// per (head, block).  Two or three workgroups fit a CU and are at different places of their tiles: one's softmax runs
// beside another's products (eight waves with one barrier went through both in step, and a last round of workgroups
// that filled a CU each left a quarter of the card idle).  Products are v_mfma_f32_32x32x16_bf16, swapped (S^T = K Q^T, O^T = V^T P^T), so a query row
// sits on a lane and the score accumulator is the second product's operand.
//   * Tiles go from the caches to LDS by DMA (buffer loads, 16 bytes a lane) into a double buffer; the 16-byte
//     pieces of a row are permuted on the source side, so that both kinds of fragment reads below hit different banks.
//   * Fragments are asked for three or four products ahead and waited for by count.  For that the DMA may not be
//     global_load_lds, which counts as an LDS access too and makes every wait for an LDS read one for all of them, and
//     the transposed reads have to say what they read (read_tr16), or each waits for the DMA on its way.  With both, and
//     every fragment read right in front of its product, the LDS's latency stood before two products of three.
//   * V^T fragments are read from the row-major image by ds_read_b64_tr_b16: no value passes through registers on
//     its way in, and where one row is key and value one image serves both products.
//   * Weights enter the value product as one bf16, or (FINE) as the sum of two.  FINE: the running maximum moves only
//     when a tile's exceeds it by 2^8, so the accumulators are rescaled on few tiles; a single bf16 holds a row's
//     largest weight exactly when that weight is 1, so there the maximum follows every tile.
//   * Wide shared rows (256 value columns): the upper half of the queries stays in LDS, the accumulators need its
//     registers.
//   * Tiles of 64 keys, or of 32 where that lets more workgroups onto a CU: values of 256 columns, and the forms with
//     score terms or sigmoid weights, whose vector work hides behind three waves a SIMD rather than two.  Shared rows of 192
//     value columns take 32 for their exactness: with 64 they are 8 % faster (half as many tiles raise a maximum, which
//     costs a multiplication of each accumulator: 4203 rows 107.5 -> 98.8 us, 600 23.8 -> 21.7), but half as many hold a weight
//     that is 1, and the error against 64 bits grows by 0.5 % (1.919e-3 -> 1.927e-3, 1.928e-3 -> 1.938e-3).
//   * Between the products of a tile's scores the next tile's DMA goes out; all four waves' at once behind the barrier
//     stood in each other's way.
//   * Score terms: the tanh cap is a polynomial of degree 5 or 7 where a tile's scores are small against the cap (|x / cap| <
//     0.17 or 0.36, relative error 2.3e-7; exp2 and reciprocal elsewhere), and where a row sees at most 1216 keys back the
//     log-distance penalty is a table of the distance in LDS: of four transcendentals a score one is left.  The keys
//     stay in order: with the newest first the maximum soon stands and 4500 rows of a window of 1024 take 91 us rather than 98,
//     but the largest weight of most tiles is no longer 1, and the error against 64 bits grows by 0.5 to 2 %.
//   * Few rows behind a long context leave most of the chip idle, and a workgroup alone on its CU takes 0.5 to 1 us for 32
//     keys, whatever it does with them: there the keys go out in parts (dxm_prompt_attention_parts, grid z), whose sums
//     merge_parts joins.  One prompt of 16 rows behind 2000 keys, 32 heads, us of the GPU: causal 41 -> 13, two maps in
//     chunks of 2048 68 -> 23, shared row 256 / 192 60 -> 17, cap + penalty in a window of 1024 39 -> 14; two of 300
//     together behind 1500: 35 -> 26, 62 -> 44, 51 -> 36, 41 -> 27.
// What bounds it: two waves a SIMD in softmax and products in turn (two maps: the matrix cores busy 45 % of the time;
// forming a tile's scores between the weights of the one in front needs 16 registers more than there are, and spills:
// 1.25 x slower), and a wave's issue where there are score terms.  32 heads, ragged prompts of about 4000 tokens, us,
// before -> now: two maps with values of 256, window 1024 + 64, 5003 rows beside 16 decode rows, with the combine: 288 -> 270;
// shared row 256 / 192 causal 125 -> 113 (870 TFLOP/s); cap + penalty, window 1024, degree 7 -> 5, 4500 rows 99 -> 97, 3000 of
// 16 heads 52.1 -> 50.5, 600 rows behind 2000 cached, window 512, 25.6 -> 25.3 (its error against 64 bits unchanged);
// sigmoid 85 -> 78.  (The register-staged 16x16x32 forms
// of tile_attention.hip, stream and latent prefill, which it took over from: two maps and their combine 776, 242, 313.)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "stream_attention.h"

namespace {

struct PromptArgs {
  void* out;  // [T, n_qh, DV]
  const bf16_t* q;
  int64_t q_stride;
  const bf16_t* kc;
  const bf16_t* vc;
  const int64_t* pos;
  const int* seq;
  const int* bt;
  int bt_stride, bs_shift;
  const int* tiles;  // [n, 2]: first row, rows (up to 128) of one sequence, consecutive positions
  int subs;          // workgroups per entry of tiles
  int n_qh, maps, group;
  int Wk, Wv;
  float scale;
  int mask, size;
  float softcap;    // 0: none
  const float* r1;  // [n_qh], null: no distance penalty
  const float* r2;
  const float* hbias;  // [n_qh] (sigmoid weights only)
  const bf16_t* gate;  // [rows, gate_stride] logits per head
  int64_t gate_stride;
  int keep;           // window mask: the first `keep` keys stay visible
  const float* sink;  // [n_qh], softmax only
  float* ws;          // parts > 1: [rows, n_qh, parts, 2 + DV]
  int parts, rows, whole;  // up to `whole` keys are not cut
};

constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
constexpr int kLeastTiles = 4;  // of a part, of several
// kTable: cap and / or penalty where a row sees at most kTableKeys keys back: the penalty is a table of the distance in LDS
enum { kPlain = 0, kTerms = 1, kSigmoid = 2, kTable = 3 };
constexpr int kTableKeys = 1216;  // what three workgroups of a CU have room for beside their tiles
constexpr int kTablePad = 64;     // entries for keys of a tile that a row does not see, on both sides

// tanh(y) / y = sum kTanh[i] y^(2 i) for |y| <= kTanhMax (minimax, fitted in 64 bits; relative error of these floats 6.2e-8, of
// the scaled scores that the kernel forms with them 2.3e-7), of scores as large as kNearMax at most: beyond, their powers and
// those of scale / cap would leave the number range
constexpr float kTanhMax = 0.36f, kNearMax = 0x1p18f;
constexpr float kTanh[4] = {0.99999996f, -0.33332261f, 0.13291534f, -0.04868792f};
// the same for |y| <= kTanhMin, to 6.2e-8 with a term less
constexpr float kTanhMin = 0.17f, kTanhFew[3] = {0.99999994f, -0.33330771f, 0.13098775f};

__device__ __forceinline__ void opaque(int& x) { asm("" : "+v"(x)); }
// One v_maximum3, which hands a NaN on (fmaxf() would quiet every operand first).  The compiler's own: in front of inline
// assembly it does not wait for the matrix product that an operand comes from.
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float max3(float a, float b, float c) { return max2(max2(a, b), c); }
// a number that is the same in every lane, in a scalar register
__device__ __forceinline__ float uniform(float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); }

// D: key columns, DV: value columns, SAME: the value is the first DV columns of the key's row
// HPW: heads per workgroup, NW: waves, SUBS: blocks of 32 keys per tile
// PARTS: the keys of a workgroup that sees enough of them go out in parts (an instance of its own: the others' loop is 2 %
// slower with what is kept for it)
template <int D, int DV, bool SAME, int MODE, bool FINE, typename OutT, int HPW, int NW, int SUBS, bool PARTS>
__global__ void __launch_bounds__(64 * NW, SUBS == 1 && DV == 128 ? 3 : 2) prompt_attention_kernel(PromptArgs a) {
  constexpr int RT = NW / HPW, ROWS = 32 * RT, KT = 32 * SUBS, SH = SUBS == 2 ? 6 : 5;
  constexpr int KS = D / 16, NC = DV / 32, KB = 2 * D, VB = SAME ? KB : 2 * DV;  // row bytes of the images
  constexpr int kKey = KT * KB, kStage = kKey + (SAME ? 0 : KT * VB);
  constexpr int KP = KT * KB / 1024 / NW, VP = SAME ? 0 : KT * VB / 1024 / NW;  // 1-KB pieces per wave
  constexpr int QR = SAME && DV == 256 ? 8 : KS;                      // query fragments in registers
  constexpr int KA = MODE == kPlain ? 4 : 3, VA = FINE ? 3 : MODE == kPlain ? 4 : 2;  // fragments asked for ahead of their products
  // Forms whose vector work is the longer part: a wave that is at it goes first, products fill what it leaves.  Not for the
  // others: raised value products of shared rows, vector work of two maps, products of sigmoid weights are 2 to 9 % faster at
  // some sizes and 2 to 5 % slower at others, and neither rows nor workgroups tell which.  us, without / with:
  // 256 / 192 causal, 3000 rows of 32 heads 136 / 126, 2500 in two prompts 63.6 / 66.7, 4000 of 16 heads 132 / 140; two maps, 4000
  // rows in chunks 180 / 175, 3000 in three prompts 99 / 103; sigmoid, 3000 rows 54.9 / 51.9, 2500 of 16 heads 28.2 / 29.4.
  constexpr bool kEager = MODE == kTerms || MODE == kTable;
  constexpr float kDefer = 8.f;  // pairs of products: log2 units that a score may exceed the running maximum by
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int yi = gridDim.y - 1 - blockIdx.y;  // later rows see more keys: hand them out first
  const int ti = yi / a.subs, off = (yi - ti * a.subs) * ROWS;
  const int n = a.tiles[2 * ti + 1] - off;
  if (n <= 0) return;
  const int row0 = a.tiles[2 * ti] + off;
  const int p0 = __builtin_amdgcn_readfirstlane((int)a.pos[row0]);
  const int* bt = a.bt + (int64_t)__builtin_amdgcn_readfirstlane(a.seq[row0]) * a.bt_stride;
  const int per = a.group / HPW, gm = blockIdx.x / per, g = gm / a.maps;  // key head, key / value group
  const int head = g * a.group + (blockIdx.x - gm * per) * HPW + wid % HPW;
  const int qh = head * a.maps + (gm - g * a.maps);
  const int rw = 32 * (wid / HPW);  // the wave's first row
  const int hi = p0 + min(n, ROWS) - 1;
  const int first = first_key(p0, a.mask, a.size) >> SH, last = hi >> SH;
  const int kept = a.mask == 1 ? min((a.keep + KT - 1) >> SH, first) : 0;  // tiles of kept keys in front of the window's
  // tiles in order: the kept ones, then the window's; of them this part's
  const int total = kept + last - first + 1, part = PARTS ? blockIdx.z : 0;
  const bool cut = PARTS && total * KT > a.whole;
  const int per_part = cut ? max((total + a.parts - 1) / a.parts, kLeastTiles) : total;
  const int i0 = part * per_part, i1 = min(i0 + per_part, total);
  // rows beyond n repeat the last one and are not stored
  const int myrow = min(rw + r, n - 1), my = p0 + myrow, mylo = first_key(my, a.mask, a.size);
  const int wlo = p0 + min(rw, n - 1), whi = p0 + min(rw + 31, n - 1);  // the wave's first and last position
  const int wfirst = first_key(wlo, a.mask, a.size), wlast = first_key(whi, a.mask, a.size);
  const int keep = a.mask == 1 ? a.keep : 0;
  float* const ws = PARTS ? a.ws + (((int64_t)(row0 + myrow) * a.n_qh + qh) * a.parts + part) * (2 + DV) : nullptr;
  if (PARTS && i0 >= i1) {  // (never the first part) no tile: sum 0
    if (cut && rw + r < n && row0 + myrow < a.rows && h == 0) *reinterpret_cast<float2*>(ws) = float2{MODE == kSigmoid ? 0.f : -INFINITY, 0.f};
    return;
  }
  bf16x8_t qf[QR];
  const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)smem;
  const uint32_t ql = base + 2 * kStage + (wid * (KS - QR) * 64 + lane) * 16;  // the lane's own pieces
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bf16x8_t f = frag16(a.q + (int64_t)(row0 + myrow) * a.q_stride + (int64_t)qh * D + 16 * ks + 8 * h);
    if (ks < QR) qf[ks < QR ? ks : 0] = f;
    else *(lds_u32x4*)(uintptr_t)(ql + (ks - QR) * 1024) = __builtin_bit_cast(raw_u32x4, f);
  }
  // Fragment addresses: step ks of the keys is an XOR with 32 ks away from the first (piece 16 and up of a row: + 256
  // bytes), block dt of the values one with 64 dt, and the rows 8 further one with 32.
  const int k_off = base + image_off<KB>(r, h);
  const int v_off = base + image_off<VB>(4 * h + ((lane & 15) >> 2), 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 8 * (lane & 1);
  const bf16_t* kc = a.kc + (int64_t)gm * D;
  const bf16_t* vc = a.vc + (int64_t)g * DV;
  // Source of the k-th 1-KB piece of a wave, from the tile's first row.  Rows behind the last query, whose values are stale,
  // are left out and arrive as zeros.
  auto source = [&](auto rb, int per_wave, int k, int width) {
    constexpr int RB = decltype(rb)::value, CH = RB / 16;
    const int row = (per_wave * wid + k) * (1024 / RB) + lane / CH;
    return 2 * (row * width + 8 * ((lane % CH) ^ piece_xor(row)));
  };
  int ksrc[KP], vsrc[VP ? VP : 1];
#pragma unroll
  for (int k = 0; k < KP; ++k) ksrc[k] = source(std::integral_constant<int, KB>{}, KP, k, a.Wk);
#pragma unroll
  for (int k = 0; k < VP; ++k) vsrc[k] = source(std::integral_constant<int, VB>{}, VP, k, a.Wv);
  // 64 entries of the block table at a time, a lane each: a load per tile would be waited for in front of its DMA
  int page0 = -64, pages = 0;
  // where the next tile lies: found in front of a tile's scores, its DMA goes out between their products (all four waves'
  // at once behind the barrier stood in each other's way)
  const bf16_t *knext = kc, *vnext = vc;
  int kbytes = 0, vbytes = 0;
  auto find = [&](int t) {
    const int j = t << SH, page = j >> a.bs_shift;
    if (page - page0 >= 64 || page < page0) {
      page0 = page;
      pages = bt[min(page0 + lane, hi >> a.bs_shift)];
      __builtin_amdgcn_s_waitcnt(0x0f70);  // (here and now: behind the branch it would be waited for, and the DMA, at every tile)
    }
    const uint32_t slot = ((uint32_t)__builtin_amdgcn_readlane(pages, page - page0) << a.bs_shift) + (j & ((1 << a.bs_shift) - 1));
    const int rows = min(hi - j, KT - 1);  // whole rows in front of the last one
    knext = kc + (uint64_t)slot * (uint32_t)a.Wk;
    kbytes = 2 * (rows * a.Wk + D);
    vnext = vc + (uint64_t)slot * (uint32_t)a.Wv;
    vbytes = 2 * (rows * a.Wv + DV);
  };
  auto fetch = [&](uint32_t buf, int k) {
    if (k < KP) dma16(knext, kbytes, ksrc[k < KP ? k : 0], buf + (KP * wid + k) * 1024);
    else dma16(vnext, vbytes, vsrc[k < KP ? 0 : k - KP], buf + kKey + (VP * wid + k - KP) * 1024);
  };
  constexpr int ND = KP + VP;  // DMA instructions of a wave and tile
  const int table_len = a.size + 2 * kTablePad;  // kTable: floats per head, entry kTablePad + d is the penalty at distance d
  const uint32_t table = base + 2 * kStage + (wid % HPW) * table_len * 4;  // of the wave's head
  if constexpr (MODE == kTable) {  // the waves of a head share its table
    const float p1 = a.r1[qh], p2 = a.r2[qh];
    for (int i = lane + 64 * (wid / HPW); i < table_len; i += 64 * RT)
      *(lds_float*)(uintptr_t)(table + 4 * i) = i >= kTablePad ? p1 * __builtin_amdgcn_logf(fmaf(p2, (float)(i - kTablePad), 1.f)) : 0.f;
  }
  const float cap = a.softcap, capl = uniform(cap * kLog2e);
  const float cape = uniform(MODE != kPlain && cap > 0.f ? a.scale * (2.f * kLog2e) / cap : 0.f);
  const bool terms = MODE != kPlain && (cap > 0.f || a.r1);
  // the polynomial on scores as the product leaves them, and how far it holds
  const float y1 = terms && cap > 0.f ? a.scale / cap : 0.f, y2 = y1 * y1, near = uniform(y1 > 0.f ? fminf(kTanhMax / y1, kNearMax) : 0.f);
  const float t0 = uniform(a.scale * kLog2e * kTanh[0]), t1 = uniform(a.scale * kLog2e * kTanh[1] * y2),
              t2 = uniform(a.scale * kLog2e * kTanh[2] * y2 * y2), t3 = uniform(a.scale * kLog2e * kTanh[3] * y2 * y2 * y2);
  const float nearer = near * (kTanhMin / kTanhMax), u0 = uniform(a.scale * kLog2e * kTanhFew[0]),
              u1 = uniform(a.scale * kLog2e * kTanhFew[1] * y2), u2 = uniform(a.scale * kLog2e * kTanhFew[2] * y2 * y2);
  const bool logs = MODE != kPlain && MODE != kTable && a.r1;
  const float r1 = uniform(logs ? a.r1[qh] : 0.f), r2 = uniform(logs ? a.r2[qh] : 0.f);
  const float sc = terms ? 1.f : a.scale * kLog2e;  // scores to log2 units
  const float hb = MODE == kSigmoid && a.hbias ? a.hbias[qh] * kLog2e : 0.f;
  float m_i = -INFINITY, l_i = 0.f;
  f32x16 O[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) O[i] = f32x16{};

  auto vread = [&](uint32_t vb, int v_at, int f) {  // columns 32 (f % NC) .. + 31 of keys 16 (f / NC) .. + 15
    const uint32_t vp = vb + f / NC * 16 * VB + 256 * (f % NC >> 2);
    const i16x4 lo = read_tr16((const lds_i16x4*)(uintptr_t)(vp + (v_at ^ 64 * (f % NC & 3))));
    const i16x4 up = read_tr16((const lds_i16x4*)(uintptr_t)(vp + 8 * VB + (v_at ^ 64 * (f % NC & 3) ^ 32)));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto step = [&](auto bufc, int t) {
    constexpr uint32_t kb = decltype(bufc)::value * kStage, vb = SAME ? kb : kb + kKey;  // from the front
    constexpr uint32_t other = (1 - decltype(bufc)::value) * kStage;                     // the next tile's
    const int kt = t << SH;
    const bool kept_tile = kt + KT <= keep;  // wholly of kept keys
    if constexpr (RT > 1) {
#pragma unroll
      for (int k = 0; k < ND; ++k) fetch(base + other, k);
      if (rw >= n || kt > whi || (kt + KT - 1 < wfirst && kt >= keep)) return;  // nothing the wave's rows see
    }
    f32x16 s[SUBS] = {};
    int k_at = k_off, v_at = v_off;
    if constexpr (MODE != kPlain) opaque(k_at), opaque(v_at);  // (three waves a SIMD: no registers to keep them all)
    {
      auto kread = [&](int ks, int sub) {
        return lds_frag((k_at ^ 32 * (ks & 7)) + (kb + 256 * (ks >> 3) + sub * 32 * KB));
      };
      bf16x8_t kf[KA][SUBS];
#pragma unroll
      for (int ks = 0; ks < KA; ++ks)
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub) kf[ks][sub] = kread(ks, sub);
      __builtin_amdgcn_sched_group_barrier(0x100, KA * SUBS, 0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8_t qk = ks < QR ? qf[ks < QR ? ks : 0] : lds_frag(ql + (ks - QR) * 1024);
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub) {
          const bf16x8_t f = kf[ks % KA][sub];
          if (ks + KA < KS) kf[ks % KA][sub] = kread(ks + KA, sub);
          s[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, qk, s[sub], 0, 0, 0);
        }
        if (RT == 1 && ks < ND) fetch(base + other, ks);
        __builtin_amdgcn_sched_group_barrier(0x008, SUBS, 0);
        if (RT == 1 && ks < ND) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, SUBS + (QR < KS), 0);
      }
    }
    if (MODE != kPlain && terms) {  // final scores in log2 units
      // penalties of the lane's keys
      const uint32_t pen = table + 4 * (kTablePad - 31 + my - kt - 4 * h);
      auto penalty = [&](int sub, int i) {
        return MODE == kTable ? *(const lds_float*)(uintptr_t)(pen + 4 * (31 - (32 * sub + (i & 3) + 8 * (i >> 2)))) : 0.f;
      };
      if (cap > 0.f) {  // cap * tanh(x / cap)
        float far = fabsf(s[0][0]);
#pragma unroll
        for (int i = 1; i < 16 * SUBS - 1; i += 2) far = max3(far, fabsf(s[i >> 4][i & 15]), fabsf(s[(i + 1) >> 4][(i + 1) & 15]));
        far = max2(far, fabsf(s[SUBS - 1][15]));
        if (__builtin_amdgcn_ballot_w64(!(far <= nearer)) == 0) {
#pragma unroll
          for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float t = s[sub][i] * s[sub][i];
              s[sub][i] = fmaf(s[sub][i], fmaf(t, fmaf(t, u2, u1), u0), -penalty(sub, i));
            }
        } else if (__builtin_amdgcn_ballot_w64(!(far <= near)) == 0) {
#pragma unroll
          for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float t = s[sub][i] * s[sub][i];
              s[sub][i] = fmaf(s[sub][i], fmaf(t, fmaf(t, fmaf(t, t3, t2), t1), t0), -penalty(sub, i));
            }
        } else {  // tanh(y) = 1 - 2 / (1 + e^(2 y))
#pragma unroll
          for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              s[sub][i] = fmaf(-2.f * capl, __builtin_amdgcn_rcpf(1.f + fast_exp2(s[sub][i] * cape)), capl) - penalty(sub, i);
        }
      } else {
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[sub][i] = fmaf(s[sub][i], a.scale * kLog2e, -penalty(sub, i));
      }
      if (logs) {  // (keys behind the row: their argument may be anything, they are masked below)
        // the distance first, which is exact: r2 times the lane's distance less r2 times the key's place would cancel
        const float d0 = (float)(my - kt - 4 * h);
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[sub][i] = fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, d0 - (float)(32 * sub + (i & 3) + 8 * (i >> 2)), 1.f)), s[sub][i]);
      }
    }
    bf16x8_t vf[VA];
#pragma unroll
    for (int f = 0; f < VA; ++f) vf[f] = vread(vb, v_at, f);
    // Some key is not seen by some row.  (Bitwise: of the two ways of a || behind the scores' last product the compiler counts the
    // longer one's instructions as waited for, and on the shorter one the scores are read too early)
    if ((kt + KT - 1 > wlo) | ((kt < wlast) & !kept_tile)) {
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = kt + 32 * sub + (i & 3) + 8 * (i >> 2) + 4 * h;
          const bool seen = ((unsigned)(j - mylo) <= (unsigned)(my - mylo)) | (j < min(keep, mylo));  // (bitwise: no branches)
          s[sub][i] = seen ? s[sub][i] : -INFINITY;
        }
    }
    float mu = 0.f;
    if constexpr (MODE != kSigmoid) {
      float ta, tb;
      if constexpr (SUBS == 2) {
        ta = max2(s[0][0], s[SUBS - 1][0]), tb = max2(s[0][1], s[SUBS - 1][1]);
#pragma unroll
        for (int i = 2; i < 16; i += 2) {
          ta = max3(ta, s[0][i], s[SUBS - 1][i]);
          tb = max3(tb, s[0][i + 1], s[SUBS - 1][i + 1]);
        }
      } else {
        ta = max2(s[0][0], s[0][1]), tb = max2(s[0][2], s[0][3]);
#pragma unroll
        for (int i = 4; i < 16; i += 4) {
          ta = max3(ta, s[0][i], s[0][i + 1]);
          tb = max3(tb, s[0][i + 2], s[0][i + 3]);
        }
      }
      // both halves of a row see the same maximum and take the same decision
      const float tm = halves_max(fmaxf(ta, tb)) * sc;
      const float mn = tm > (FINE ? m_i + kDefer : m_i) ? tm : m_i;
      mu = mn == -INFINITY ? 0.f : mn;  // a row that has seen nothing yet
      if (__builtin_amdgcn_ballot_w64(mn != m_i)) {
        const float alpha = fast_exp2(m_i - mu);
        l_i *= alpha;
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) O[i][e] *= alpha;
      }
      m_i = mn;
    }
    // the weights of 16 keys (group f / NC of the tile) as they enter the product
    raw_u32x4 ph[2], pl[2];
    auto weigh = [&](int k16) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float w[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const float v = s[k16 >> 1][8 * (k16 & 1) + 2 * e + x];
          if constexpr (MODE == kSigmoid)  // sigmoid(s + bias); an invisible key (s = -inf) weighs 0
            w[x] = __builtin_amdgcn_rcpf(1.f + fast_exp2(-fmaf(v, sc, hb)));
          else
            w[x] = fast_exp2(fmaf(v, sc, -mu));
        }
        if constexpr (MODE != kSigmoid) l_i += w[0] + w[1];
        ph[k16 & 1][e] = pack_bf16x2(w[0], w[1]);
        if constexpr (FINE) pl[k16 & 1][e] = pack_bf16x2(w[0] - bf16lo(ph[k16 & 1][e]), w[1] - bf16hi(ph[k16 & 1][e]));
      }
    };
    constexpr int NF = 2 * SUBS * NC;  // value fragments of the tile
    weigh(0);
    if constexpr (kEager) __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int k16 = f / NC, dt = f % NC;
      // (blocks of rows behind one another: what the later rows' own values hold must not meet this one's zero weights)
      if (RT > 1 && SUBS == 2 && f == NF / 2 && kt + 32 > whi) break;
      if (dt == 0 && k16 + 1 < 2 * SUBS) weigh(k16 + 1);
      const bf16x8_t cur = vf[f % VA];
      if (f + VA < NF) vf[f % VA] = vread(vb, v_at, f + VA);
      O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur, __builtin_bit_cast(bf16x8_t, ph[k16 & 1]), O[dt], 0, 0, 0);
      if constexpr (FINE)
        O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur, __builtin_bit_cast(bf16x8_t, pl[k16 & 1]), O[dt], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, FINE ? 2 : 1, 0);
      if (f + VA < NF) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    if constexpr (kEager) __builtin_amdgcn_s_setprio(1);
  };
  auto tile = [&](int i) { return i < kept ? i : first + i - kept; };
  static_assert(ND <= KS, "a DMA instruction beside a product at most");
  find(tile(i0));
#pragma unroll
  for (int k = 0; k < ND; ++k) fetch(base, k);
  landed();
  for (int i = i0; i < i1; i += 2) {  // (behind the last tile it is fetched again: no branch among the products)
    find(tile(min(i + 1, i1 - 1)));
    step(std::integral_constant<int, 0>{}, tile(i));
    landed();
    if (i + 1 < i1) {
      find(tile(min(i + 2, i1 - 1)));
      step(std::integral_constant<int, 1>{}, tile(i + 1));
      landed();
    }
  }

  const bool ok = rw + r < n;
  const bool kept_row = PARTS && ok && row0 + myrow < a.rows;
  if (PARTS && !cut && kept_row && h == 0) *reinterpret_cast<float2*>(ws) = float2{0.f, -1.f};  // the join's sign to leave the row
  if (cut) {  // sums as they are: gate, sink and denominator come with the join
    if (!kept_row) return;
    const float l = MODE == kSigmoid ? 1.f : halves_sum(l_i);
    if (h == 0) *reinterpret_cast<float2*>(ws) = float2{MODE == kSigmoid ? 0.f : m_i * kLn2, l};
#pragma unroll
    for (int dt = 0; dt < NC; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        float* o = ws + 2 + dt * 32 + 8 * g4 + 4 * h;
        *reinterpret_cast<float2*>(o) = float2{O[dt][4 * g4], O[dt][4 * g4 + 1]};
        *reinterpret_cast<float2*>(o + 2) = float2{O[dt][4 * g4 + 2], O[dt][4 * g4 + 3]};
      }
    return;
  }
  float inv = 1.f;
  if constexpr (MODE != kSigmoid) {
    float l = halves_sum(l_i);
    if (a.sink) l += fast_exp2(a.sink[qh] * kLog2e - m_i);  // (finite: a row sees itself)
    inv = 1.f / l;
  }
  if (a.gate) inv /= 1.f + __expf(-bf16_to_f32(a.gate[(int64_t)(row0 + myrow) * a.gate_stride + head]));
  OutT* o = (OutT*)a.out + ((int64_t)(row0 + myrow) * a.n_qh + qh) * DV;
  // lane (r, h) holds columns 8 g4 + 4 h .. + 3 of each block of 32
#pragma unroll
  for (int dt = 0; dt < NC; ++dt) {
    if constexpr (sizeof(OutT) == 4) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        if (ok)
          *reinterpret_cast<f32x4*>(o + dt * 32 + 8 * g4 + 4 * h) =
              f32x4{O[dt][4 * g4] * inv, O[dt][4 * g4 + 1] * inv, O[dt][4 * g4 + 2] * inv, O[dt][4 * g4 + 3] * inv};
    } else {  // two neighbouring groups swap halves: 16 bytes a lane
#pragma unroll
      for (int g4 = 0; g4 < 4; g4 += 2) {
        const uint32_t ax = pack_bf16x2(O[dt][4 * g4] * inv, O[dt][4 * g4 + 1] * inv);
        const uint32_t ay = pack_bf16x2(O[dt][4 * g4 + 2] * inv, O[dt][4 * g4 + 3] * inv);
        const uint32_t bx = pack_bf16x2(O[dt][4 * g4 + 4] * inv, O[dt][4 * g4 + 5] * inv);
        const uint32_t by = pack_bf16x2(O[dt][4 * g4 + 6] * inv, O[dt][4 * g4 + 7] * inv);
        const auto sx = __builtin_amdgcn_permlane32_swap(ax, bx, false, false);
        const auto sy = __builtin_amdgcn_permlane32_swap(ay, by, false, false);
        if (ok) *reinterpret_cast<raw_u32x4*>(o + dt * 32 + 8 * g4 + 8 * h) = raw_u32x4{sx[0], sy[0], sx[1], sy[1]};
      }
    }
  }
}

template <int D, int DV, bool SAME, int MODE, bool FINE, typename OutT, int HPW, int NW, int SUBS, bool PARTS>
int launch_prompt_as(const PromptArgs& a0, int n_tiles, hipStream_t st) {
  PromptArgs a = a0;
  a.subs = 128 / (32 * (NW / HPW));
  constexpr int tiles = 2 * 32 * SUBS * 2 * (D + (SAME ? 0 : DV)) + (SAME && DV == 256 ? NW * (D / 16 - 8) * 1024 : 0);
  constexpr int most = tiles + (MODE == kTable ? HPW * (kTableKeys + 2 * kTablePad) * 4 : 0);
  const int lds = tiles + (MODE == kTable ? HPW * (a.size + 2 * kTablePad) * 4 : 0);
  auto kern = prompt_attention_kernel<D, DV, SAME, MODE, FINE, OutT, HPW, NW, SUBS, PARTS>;
  static bool raised = false;  // once per instance
  if (most > 48 * 1024 && !raised) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess) return 7;
    raised = true;
  }
  const int step = 65535 / a.subs;
  for (int t0 = 0; t0 < n_tiles; t0 += step) {
    a.tiles = a0.tiles + 2 * t0;
    const int nt = n_tiles - t0 < step ? n_tiles - t0 : step;
    hipLaunchKernelGGL(kern, dim3(a.n_qh / HPW, nt * a.subs, a.parts), dim3(64 * NW), lds, st, a);
  }
  DX_CHECK_LAUNCH();
  return 0;
}

template <int D, int DV, bool SAME, int MODE, bool FINE, typename OutT, int HPW, int NW, int SUBS>
int launch_prompt(const PromptArgs& a, int n_tiles, hipStream_t st) {
  return a.parts > 1 ? launch_prompt_as<D, DV, SAME, MODE, FINE, OutT, HPW, NW, SUBS, true>(a, n_tiles, st)
                     : launch_prompt_as<D, DV, SAME, MODE, FINE, OutT, HPW, NW, SUBS, false>(a, n_tiles, st);
}

// (tiles of 32 / 64 keys, us, launches back to back: cap + penalty 157 / 153, sigmoid 91 / 99, shared row 256 / 256
// 128 / 182, 256 / 192 causal 120 / 113 and of 600 rows 24.5 / 22.0 (less exact: above), two maps 265 / 350, plain of 5000 149 / 154 and of 40 behind
// 2900 cached 94 / 83, fine 179 / 186)
template <int D, int DV, bool SAME, int MODE, bool FINE, typename OutT>
int prompt_heads(const PromptArgs& a, int n_tiles, hipStream_t st) {
  constexpr int SUBS = DV == 128 && MODE == kPlain ? 2 : 1;
  if (a.group % 4 == 0) return launch_prompt<D, DV, SAME, MODE, FINE, OutT, 4, 4, SUBS>(a, n_tiles, st);
  return launch_prompt<D, DV, SAME, MODE, FINE, OutT, 2, 4, SUBS>(a, n_tiles, st);
}

}  // namespace

extern "C" {

// 1 when the kernel has an instance for the heads and the kind of result; `same`: keys and values are one cache
int dxm_prompt_attention_ok(int d, int dv, int n_qh, int maps, int group, int bs, int same, int terms, int sigmoid,
                            int out_f32, int fine) {
  if (bs < 64 || (bs & (bs - 1)) || group < 1) return 0;
  if (group % 2) return 0;
  if (same) return d == 256 && (dv == 192 || dv == 256) && maps == 1 && group == n_qh && !terms && !sigmoid && !out_f32 && !fine;
  if (d == 128 && dv == 256) return out_f32 && !terms && !sigmoid;
  return d == 128 && dv == 128 && !out_f32 && !(fine && (terms || sigmoid));
}

// Parts that the keys of `rows` prompt rows in n_tiles tiles are cut into, `keys` of them visible to a row's workgroup at
// most; *whole: a workgroup that sees no more keys than that takes them in one.  (The host knows a bound only, beside decode
// rows of long contexts a high one.  Prompts of 60 to 300 rows with nothing cached beside 8 to 30 decode rows to 5000: 1 us
// of 29 to 69 for the join that finds them done.)
// A workgroup alone on its CU goes from tile to tile at the pace of its loads (0.5 to 1 us for 32 keys); one that shares it
// takes a fifth longer, of three to a CU each takes nearly twice as long.  Against that stand the join and every part's sums
// on their way through memory.  Terms in us, fitted to one to six prompts of 16 to 1000 rows together at 16 and 32 heads,
// behind 0 to 3000 cached keys: gains above 2 all hold there.  The rule asks for 4, which is what the second launch costs on
// the host (it counts where steps are so small that the host is behind).
static int prompt_parts(int rows, int n_tiles, int keys, int n_qh, int group, int dv, bool terms, bool sigmoid, bool fine, int* whole) {
  const int tall = group % 4 ? 2 : 1, blocks = std::min(n_tiles * (4 / tall), n_tiles + rows / (32 * tall));
  const double wgs = (double)blocks * n_qh * tall / 4, floats = (double)rows * n_qh * (2 + dv);
  const double key = (sigmoid ? 1.4 : dv > 128 || terms ? 2.0 : fine ? 1.2 : 1.0) / 64;  // of a workgroup alone
  double best = 4.0;
  int parts = 1;
  *whole = 0;
  for (int p = 2; p <= 8 && (p - 1) * kLeastTiles * 32 < keys; p *= 2) {
    const double saved = key * (1.0 - std::max(1.0, 0.6 * std::ceil(wgs * p / 256)) / p), cost = 6.5 + floats * p * 1.25e-6;
    if (saved * keys - cost > best) best = saved * keys - cost, parts = p, *whole = (int)(cost / saved);
  }
  return parts;
}

int dxm_prompt_attention_parts(int rows, int n_tiles, int keys, int n_qh, int maps, int group, int d, int dv, int bs, int same,
                               int terms, int sigmoid, int out_f32, int fine, int* whole) {
  *whole = 0;
  if (rows < 1 || n_tiles < 1 || !dxm_prompt_attention_ok(d, dv, n_qh, maps, group, bs, same, terms, sigmoid, out_f32, fine)) return 1;
  return prompt_parts(rows, n_tiles, keys, n_qh, group, dv, terms, sigmoid, fine, whole);
}

int dxm_prompt_attention(void* out, const void* q, int64_t q_stride, const void* kc, const void* vc, const int64_t* pos,
                         const int* seq, const int* bt, int bt_stride, int bs, const int* tiles, int n_tiles, int n_qh,
                         int maps, int group, int d, int dv, int Wk, int Wv, float scale, int mask, int size,
                         float softcap, const float* r1, const float* r2, int wfn, const float* hbias, const void* gate,
                         int64_t gate_stride, int keep, const float* sink, int out_f32, int fine, float* ws, int parts,
                         int rows, int whole, hipStream_t st) {
  if (n_tiles <= 0) return 0;
  const bool same = kc == vc, terms = softcap > 0.f || r1;
  if (softcap < 0.f || (r1 && !r2) || wfn < 0 || wfn > 1 || keep < 0 || (keep && mask != 1)) return 6;
  if (!dxm_prompt_attention_ok(d, dv, n_qh, maps, group, bs, same, terms, wfn, out_f32, fine)) return 2;
  if (n_qh < 1 || maps < 1 || n_qh % maps || (n_qh / maps) % group || n_qh > 65535) return 1;
  if (mask < 0 || mask > 2 || (mask && size < 1) || !(scale > 0.f) || parts < 1 || parts > 64) return 3;
  if (!out || (parts > 1 && (!ws || (uintptr_t)ws % 8)) || !seq || !tiles || Wk % 8 || Wv % 8 || q_stride % 8 || (uintptr_t)q % 16 || (uintptr_t)kc % 16 ||
      (uintptr_t)vc % 16 || (uintptr_t)out % 16)
    return 4;
  PromptArgs a{out, (const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, pos, seq, bt, bt_stride,
               __builtin_ctz((unsigned)bs), tiles, 1, n_qh, maps, group, Wk, Wv, scale, mask, size, softcap, r1, r2, hbias,
               (const bf16_t*)gate, gate_stride, keep, sink, ws, parts, rows, whole};
  if (same && dv == 256) return prompt_heads<256, 256, true, kPlain, false, bf16_t>(a, n_tiles, st);
  if (same) return prompt_heads<256, 192, true, kPlain, false, bf16_t>(a, n_tiles, st);
  if (dv == 256) return prompt_heads<128, 256, false, kPlain, true, float>(a, n_tiles, st);
  if (wfn) return prompt_heads<128, 128, false, kSigmoid, false, bf16_t>(a, n_tiles, st);
  // Every row sees keys within `size` of it.  Table / logarithms, us, at 1216 / 1217 keys, 4500 rows of 32 heads 115 / 117, 5000
  // of 16 62 / 82 (of 1024 keys, 4500 rows of 32 heads: 97)
  if (r1 && mask && !keep && size <= kTableKeys) return prompt_heads<128, 128, false, kTable, false, bf16_t>(a, n_tiles, st);
  if (terms) return prompt_heads<128, 128, false, kTerms, false, bf16_t>(a, n_tiles, st);
  if (fine) return prompt_heads<128, 128, false, kPlain, true, bf16_t>(a, n_tiles, st);
  return prompt_heads<128, 128, false, kPlain, false, bf16_t>(a, n_tiles, st);
}

}  // extern "C"
