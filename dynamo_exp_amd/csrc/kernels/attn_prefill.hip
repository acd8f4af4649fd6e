// Paged-KV causal prefill attention (varlen, with cached prefix) for gfx950.
//
// Flash-attention forward on MFMA v_mfma_f32_32x32x16_bf16:
//   * workgroup = 8 or 4 waves; every wave owns 32 query rows of ONE query head.
//     The waves of a workgroup share one KV head (GQA group: 4 heads x 2 or 1
//     32-token tiles), so every K/V tile staged in LDS is reused by all of them;
//     32-row K sub-blocks that lie entirely above a wave's causal diagonal are
//     skipped (no MFMA, no softmax work);
//   * K/V tiles of 64 tokens are gathered from the paged cache (block table)
//     by LDS-DMA (16-byte buffer loads, no staging registers; rows past the
//     context arrive as zeros) into a double-buffered, XOR-swizzled LDS image
//     (the swizzle is chosen on the source side), the next tile in flight
//     while the current one computes;
//   * S^T = K . Q^T ("swapped" product): the query row sits on the lane, so the
//     online softmax is lane-local (+1 cross-half exchange) and the S
//     accumulator is directly the B operand of the P.V product
//     O^T = V^T . P^T (guide section 3, "accumulator tile as next operand");
//   * V^T fragments come from the same swizzled image via ds_read_b64_tr_b16
//     (guide T10), K fragments via ds_read_b128; both conflict-free;
//   * fragments are asked for four products ahead and waited for by count.
//     With global_load_lds, which the compiler counts as an LDS access too, and
//     transposed reads that do not say what they read, each was waited for
//     right in front of its product (and the first of a tile's values for the
//     next tile's DMA): 32 / 8 heads, us, then -> now: two prompts of 5000
//     tokens together 132 -> 123, one of 2000 53.5 -> 48.6, 300 rows behind
//     2900 cached 71 -> 65, six of 3000 with 16 / 4 heads 26.1 -> 24.4.
//
// Q is read straight from the fused QKV buffer (row stride q_stride) after the
// rope kernel rotated it in place; the new tokens' K/V are already in the paged
// cache, so prefix and new tokens are handled uniformly.
#include "common.h"

#include <type_traits>

namespace {

constexpr int D = 128;
constexpr int BQ = 32;   // query rows per wave
constexpr int BKV = 64;  // kv rows per tile
constexpr int kTileBytes = BKV * D * 2;  // 16 KiB

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
// byte offset of 16-B chunk `ch` (0..15) of row `row` inside a [64][128] bf16 tile
__device__ __forceinline__ int tile_off(int row, int ch) { return row * 256 + 16 * (ch ^ swz(row)); }

__device__ __forceinline__ bf16x8_t as_frag(const u16x8& v) { return __builtin_bit_cast(bf16x8_t, v); }

// ---------------------------------------------------------------------------
// The kernel: NW waves (8: 4 heads x 64 query tokens per workgroup sharing each
// K/V tile; 4: 32 tokens), K/V staged by LDS-DMA into a double-buffered
// swizzled image, with the per-tile vector work cut down -- the loop is
// issue-bound, not MFMA-bound, at 2 waves/SIMD.  (Earlier register-staged
// 4/8-wave, 4-wave x 2 q-block and 3-stage-DMA variants measured 322-794
// TFLOP/s vs 592-875 for this one: profiles/r1_prefill_attn_*.json; removed.)
// (each MFMA holds the SIMD's vector issue for 8 of its 32 cycles; v_exp 8,
// everything else 4 cycles of issue, MI355X_MICROARCH constants table):
//   * LDS fragment addresses are per-lane constants (the XOR swizzle only
//     depends on row bits 0..3, so +32 rows / +16 rows / the other buffer are
//     immediate offsets): the loop is unrolled over the two buffers;
//   * with block_size >= 64 a full tile lies in one KV block, so the DMA source
//     is a scalar base (from 64 block-table entries in a register) + a
//     per-lane constant;
//   * masking only on diagonal / ragged tiles, by select (no branches);
//     softmax with the scale folded into the FMA; the row
//     max as two v_max3 chains; the row sum l as ones . P^T on the matrix
//     pipe (the exact sum of the bf16 P the P.V product uses: with the
//     deferred max, profiles/r4_prefill_attn_variants.txt).
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr float kRescaleLog2 = 8.0f;  // deferred-max threshold (log2 units)

// PLS: max / sum over the two halves of a wave by one v_permlane32_swap (halves_max, halves_sum: VALU) instead of a
// ds_bpermute round trip through LDS in the softmax's dependent chain
// V: 0 = the first loop (kept for A/B), 1 = deferred rescale, row
// sum on the matrix pipe, v_max3 row max, raised priority (step), widened epilogue.
// (Ping-pong wave halves, two tiles per barrier and a software-pipelined QK /
// softmax measured slower, as did 4-wave workgroups where there are enough of
// 8: profiles/r4_prefill_attn_variants.txt.)
template <bool BS64, bool PLS, int V, int NW>
__global__ void __launch_bounds__(64 * NW, 2) prefill_attn_v2_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ cu_seqlens_q, const int* __restrict__ ctx_lens, const int* __restrict__ work,
    int n_q_heads, int n_kv_heads, int bs_shift, int heads_per_wg, float scale_log2e, int causal) {
  constexpr int kBuf = 2 * kTileBytes;  // one (K, V) stage
  constexpr bool kMfmaSum = V == 1;  // row sum l on the matrix pipe
  __shared__ __attribute__((aligned(16))) char smem[2 * kBuf];
  const int block_size = 1 << bs_shift;
  const int G = n_q_heads / n_kv_heads;
  const int head_groups = G / heads_per_wg;
  // grid = (head groups, work items): x fastest in dispatch order, so every
  // work item (heaviest first) goes out for all heads before the next one --
  // a global longest-first schedule -- and consecutive workgroups land on
  // consecutive XCDs, i.e. with 8 KV-head groups each XCD's L2 serves one KV
  // head's tiles for all work items.
  const int kvh = __builtin_amdgcn_readfirstlane(blockIdx.x / head_groups);
  const int hg = blockIdx.x % head_groups;
  const int token_tiles = NW / heads_per_wg;
  // a work item is the rows of eight waves; its later rows see more keys and go first
  const int item = blockIdx.y / (8 / NW), sub = 8 / NW - 1 - blockIdx.y % (8 / NW);
  // (the same for every lane, and known as such: a descriptor in vector registers would be read out lane by lane)
  const int seq = __builtin_amdgcn_readfirstlane(work[2 * item]);
  const int tok0 = __builtin_amdgcn_readfirstlane(work[2 * item + 1]) + sub * token_tiles * BQ;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q_start = __builtin_amdgcn_readfirstlane(cu_seqlens_q[seq]);
  const int qlen = __builtin_amdgcn_readfirstlane(cu_seqlens_q[seq + 1]) - q_start;
  const int ctx = __builtin_amdgcn_readfirstlane(ctx_lens[seq]);
  const int pos0 = ctx - qlen;
  if (tok0 >= qlen) return;
  const int r = lane & 31, h = lane >> 5;

  const int head = kvh * G + hg * heads_per_wg + (wid % heads_per_wg);
  const int wtok0 = tok0 + (wid / heads_per_wg) * BQ;
  const bool row_valid = wtok0 + r < qlen;
  // causal 0 (bidirectional, e.g. a vision tower): every query sees the whole
  // context -- only the ragged last tile is masked
  const int my_pos = causal ? pos0 + wtok0 + r : ctx - 1;
  const int wave_min_pos = causal ? pos0 + wtok0 : ctx - 1;
  const int wave_max_pos = causal ? pos0 + min(wtok0 + BQ, qlen) - 1 : ctx - 1;
  const int wg_last_tok = min(tok0 + token_tiles * BQ, qlen) - 1;
  const int kv_end = causal ? min(ctx, pos0 + wg_last_tok + 1) : ctx;
  const int n_tiles = (kv_end + BKV - 1) / BKV;

  u16x8 qf[8];
  {
    const bf16_t* qp = q + (int64_t)(q_start + wtok0 + r) * q_stride + (int64_t)head * D + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      qf[ks] = row_valid ? *reinterpret_cast<const u16x8*>(qp + 16 * ks) : u16x8{{0, 0, 0, 0}};
  }

  // ---- per-lane constant LDS offsets ----
  int koff[8];  // K fragment row r (+32 for the second half: +8192 B), chunk 2ks+h
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) koff[ks] = tile_off(r, 2 * ks + h);
  int voff[4][2];  // V^T fragments: rows 4h+qq and 4h+qq+8 (+16 s2, +32 sub: immediates)
  {
    const int g16 = (lane >> 4) & 1, qq = (lane & 15) >> 2, pp = lane & 3;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const int ch = dt * 4 + 2 * g16 + (pp >> 1);
      voff[dt][0] = tile_off(4 * h + qq, ch) + 8 * (pp & 1);
      voff[dt][1] = tile_off(4 * h + qq + 8, ch) + 8 * (pp & 1);
    }
  }
  // ---- DMA slots: instruction k of this wave fills tile rows 4*(KPW*wid+k) .. +3 ----
  constexpr int KPW = 16 / NW;  // 1-KB pieces of a 16-KB K (or V) tile per wave
  const int* bt = block_tables + (int64_t)seq * bt_stride;
  const int64_t head_stride = (int64_t)block_size * D;
  int src_off[KPW];  // bytes from the tile's first row
#pragma unroll
  for (int k = 0; k < KPW; ++k) {
    const int row = (KPW * wid + k) * 4 + (lane >> 4);
    src_off[k] = 2 * (row * D + ((lane & 15) ^ swz(row)) * 8);
  }
  // 64 entries of the block table at a time, a lane each: a load per tile would be waited for in front of its DMA
  int page0 = -64, pages = 0;
  const int last_page = (ctx - 1) >> bs_shift;
  auto block = [&](int j) __attribute__((always_inline)) {  // the first of 64 keys' block, or a later one of theirs
    return __builtin_amdgcn_readlane(pages, min(j >> bs_shift, last_page) - page0);
  };
  auto issue = [&](char* kb, int j0) __attribute__((always_inline)) {
    char* vb = kb + kTileBytes;
    if (min((j0 + BKV - 1) >> bs_shift, last_page) - page0 >= 64) {
      page0 = j0 >> bs_shift;
      pages = bt[min(page0 + lane, last_page)];
      __builtin_amdgcn_s_waitcnt(0x0f70);  // (here and now: behind the branch it would be waited for at every tile)
    }
    if (BS64) {  // one block; rows past the context arrive as zeros
      const int64_t base = ((int64_t)block(j0) * n_kv_heads + kvh) * head_stride + (int64_t)(j0 & (block_size - 1)) * D;
      const int bytes = 2 * D * min(ctx - j0, BKV);
#pragma unroll
      for (int k = 0; k < KPW; ++k) {
        dma16(k_cache + base, bytes, src_off[k], (lds_void*)(kb + (KPW * wid + k) * 1024));
        dma16(v_cache + base, bytes, src_off[k], (lds_void*)(vb + (KPW * wid + k) * 1024));
      }
    } else {
#pragma unroll
      for (int k = 0; k < KPW; ++k) {  // a piece's four rows lie in one block (block_size % 4 == 0)
        const int at = 4 * (KPW * wid + k), j = __builtin_amdgcn_readfirstlane(j0 + at);
        const int64_t base = ((int64_t)block(j) * n_kv_heads + kvh) * head_stride + (int64_t)(j & (block_size - 1)) * D;
        const int bytes = __builtin_amdgcn_readfirstlane(2 * D * max(min(ctx - j, 4), 0));
        dma16(k_cache + base, bytes, src_off[k] - 2 * D * at, (lds_void*)(kb + (KPW * wid + k) * 1024));
        dma16(v_cache + base, bytes, src_off[k] - 2 * D * at, (lds_void*)(vb + (KPW * wid + k) * 1024));
      }
    }
  };

  f32x16 o_acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o_acc[i] = f32x16{};
  float m_i = -1e30f, l_i = 0.f;
  f32x16 l_acc = f32x16{};  // V1: every row of the 32 x 32 tile = l of the lane's query column
  const bf16x8_t kOnes = __builtin_bit_cast(bf16x8_t, u16x8{{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u}});
  const f32x2 sc2 = {scale_log2e, scale_log2e};

  constexpr int kAhead = 4;  // fragments asked for ahead of their products
  auto vread = [&](const char* vb, int i) __attribute__((always_inline)) {  // columns 32 (i % 4) .. + 31 of keys 16 (i / 4) .. + 15
    const i16x4 lo = read_tr16((const lds_i16x4*)(vb + i / 4 * 4096 + voff[i % 4][0]));
    const i16x4 hi = read_tr16((const lds_i16x4*)(vb + i / 4 * 4096 + voff[i % 4][1]));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // segment 1 of a tile: S^T = K . Q^T, mask, online softmax -> this wave's
  // bf16 P fragments (and the O / l rescale); false: nothing of the tile is
  // at or below this wave's diagonal
  auto qk_sm = [&](const char* kb, int t, u16x8 (&pf)[2][2], bool& live1, bf16x8_t (&vf)[kAhead]) __attribute__((always_inline)) -> bool {
    const int j0 = t * BKV;
    live1 = j0 + 32 <= wave_max_pos;
    if (j0 > wave_max_pos) return false;
    f32x16 s0 = f32x16{}, s1 = f32x16{};
    bf16x8_t kf[kAhead];
    auto kread = [&](int i) __attribute__((always_inline)) { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kb + 8192 * (i >> 3) + koff[i & 7])); };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) kf[i] = kread(i);
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8_t f = kf[ks % kAhead];
      kf[ks % kAhead] = kread(ks + kAhead);
      s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, as_frag(qf[ks]), s0, 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if (live1) {
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const bf16x8_t f = kf[ks % kAhead];
        if (ks + kAhead < 8) kf[ks % kAhead] = kread(8 + ks + kAhead);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, as_frag(qf[ks]), s1, 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (ks + kAhead < 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
#pragma unroll
    for (int f = 0; f < kAhead; ++f) vf[f] = vread(kb + kTileBytes, f);
    if ((j0 + BKV - 1 > wave_min_pos) || (j0 + BKV > ctx)) {  // diagonal / ragged tile
      const int lim = min(my_pos, ctx - 1) - j0 - 4 * h;  // keep kv row j0 + 4h + off <= lim + j0 + 4h
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int off = (i & 3) + 8 * (i >> 2);
        s0[i] = off > lim ? -INFINITY : s0[i];
        s1[i] = off + 32 > lim ? -INFINITY : s1[i];
      }
    }
    // (!live1 implies a diagonal tile: the select above already set every
    // valid row's second half to -inf, and its P.V half is skipped below)
    float tmax;
    if constexpr (kMfmaSum) {  // two independent v_max3 chains (the file is built for scores that are no NaN: nothing is quieted first)
      float ta = fmaxf(s0[0], s1[0]), tb = fmaxf(s0[1], s1[1]);
#pragma unroll
      for (int i = 2; i < 16; i += 2) {
        ta = fmaxf(fmaxf(ta, s0[i]), s1[i]);
        tb = fmaxf(fmaxf(tb, s0[i + 1]), s1[i + 1]);
      }
      tmax = halves_max(fmaxf(ta, tb));
    } else {
      float ta = -INFINITY, tb = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        ta = fmaxf(ta, fmaxf(s0[i], s1[i]));
        tb = fmaxf(tb, fmaxf(s0[i + 1], s1[i + 1]));
      }
      tmax = fmaxf(ta, tb);
      tmax = PLS ? halves_max(tmax) : fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    }
    // deferred rescale (guide T13): the running max moves only when the
    // tile's max exceeds it by more than kRescaleLog2, so P = 2^(s - m) stays
    // <= 2^kRescaleLog2 (exact enough in bf16 / fp32) and the O / l rescale
    // below is skipped on almost every tile; both halves of a row (lanes r,
    // r + 32) see the same tmax, so they always take the same decision
    const float t_s = tmax * scale_log2e;
    const float m_new = t_s > m_i + (V == 1 ? kRescaleLog2 : 0.f) ? t_s : m_i;
    const float alpha = fast_exp2(m_i - m_new);
    m_i = m_new;
    const f32x2 nm2 = {-m_new, -m_new};
    f32x2 rs2 = {0.f, 0.f};
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int i = 8 * s2 + 2 * w;
        const f32x2 a0 = f32x2{s0[i], s0[i + 1]} * sc2 + nm2;
        const f32x2 a1 = f32x2{s1[i], s1[i + 1]} * sc2 + nm2;
        const f32x2 p0 = {fast_exp2(a0.x), fast_exp2(a0.y)};
        const f32x2 p1 = {fast_exp2(a1.x), fast_exp2(a1.y)};
        pf[0][s2].w[w] = pack_bf16x2(p0.x, p0.y);
        pf[1][s2].w[w] = pack_bf16x2(p1.x, p1.y);
        if constexpr (!kMfmaSum) rs2 += p0 + p1;  // V1: l_acc below
      }
    if constexpr (!kMfmaSum) {
      float rs = rs2.x + rs2.y;
      rs = PLS ? halves_sum(rs) : rs + __shfl_xor(rs, 32, 64);
      l_i = l_i * alpha + rs;
    }
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o_acc[dt] *= alpha;
      if constexpr (kMfmaSum) l_acc *= alpha;
    }
    return true;
  };
  // segment 2: O^T += V^T . P^T (+ l on the matrix pipe)
  auto pv = [&](const char* vb, bool live1, const u16x8 (&pf)[2][2], bf16x8_t (&vf)[kAhead]) __attribute__((always_inline)) {
    // O^T[d][q] += V^T[d][kv] . P^T[kv][q]
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      if (sub == 0 || live1) {
#pragma unroll
        for (int i = 8 * sub; i < 8 * sub + 8; ++i) {
          const bf16x8_t p = as_frag(pf[sub][(i >> 2) & 1]), f = vf[i % kAhead];
          if (i + kAhead < 16) vf[i % kAhead] = vread(vb, i + kAhead);
          o_acc[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, p, o_acc[i & 3], 0, 0, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i + kAhead < 16) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          // l += ones . P^T: the row sum of exactly the bf16 P the P.V product
          // used (O / l stays an exact weighted mean of V rows under the
          // deferred max), on the matrix pipe instead of 16 packed adds + a
          // cross-half exchange on the issue-bound VALU
          if constexpr (kMfmaSum)
            if ((i & 3) == 3) l_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kOnes, p, l_acc, 0, 0, 0);
        }
      }
    }
  };

  {
    // Two waves of one workgroup share a SIMD: scores and softmax at raised priority, the value products fill what they leave.
    // (Three of 2000 together 141 -> 137 us with waves 4-7 raised throughout before.  Two workgroups of four waves lose 4 to 6 %.)
    constexpr bool kRaised = NW == 8 && V != 0;
    auto step = [&](auto bufc, int t) __attribute__((always_inline)) {
      constexpr int BUF = decltype(bufc)::value;
      char* kb = smem + BUF * kBuf;
      if (t + 1 < n_tiles) issue(smem + (BUF ^ 1) * kBuf, t * BKV + BKV);
      u16x8 pf[2][2];
      bf16x8_t vf[kAhead];
      bool live1;
      if (qk_sm(kb, t, pf, live1, vf)) {
        if constexpr (kRaised) __builtin_amdgcn_s_setprio(0);
        pv(kb + kTileBytes, live1, pf, vf);
        if constexpr (kRaised) __builtin_amdgcn_s_setprio(1);
      }
      landed();
    };
    if (n_tiles > 0) issue(smem, 0);
    landed();
    for (int t = 0; t < n_tiles; t += 2) {
      step(std::integral_constant<int, 0>{}, t);
      if (t + 1 < n_tiles) step(std::integral_constant<int, 1>{}, t + 1);
    }
  }

  // epilogue, widened (guide T21): lane (r, h) holds columns 8 g + 4 h .. + 3
  // of each 8-column group g; one v_permlane32_swap per dword pairs groups
  // (g, g + 1) so each lane stores 16 contiguous bytes: half the stores
  if constexpr (kMfmaSum) l_i = l_acc[0];
  const float inv_l = l_i > 0.f ? 1.f / l_i : 0.f;
  bf16_t* op = out + ((int64_t)(q_start + wtok0 + r) * n_q_heads + head) * D;
  if constexpr (V == 0) {  // A/B baseline: 8-byte stores
    if (!row_valid) return;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        uint2 v;
        v.x = pack_bf16x2(o_acc[dt][4 * g4 + 0] * inv_l, o_acc[dt][4 * g4 + 1] * inv_l);
        v.y = pack_bf16x2(o_acc[dt][4 * g4 + 2] * inv_l, o_acc[dt][4 * g4 + 3] * inv_l);
        *reinterpret_cast<uint2*>(op + dt * 32 + 8 * g4 + 4 * h) = v;
      }
    return;
  }
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; g4 += 2) {
      uint2 a, b;
      a.x = pack_bf16x2(o_acc[dt][4 * g4 + 0] * inv_l, o_acc[dt][4 * g4 + 1] * inv_l);
      a.y = pack_bf16x2(o_acc[dt][4 * g4 + 2] * inv_l, o_acc[dt][4 * g4 + 3] * inv_l);
      b.x = pack_bf16x2(o_acc[dt][4 * g4 + 4] * inv_l, o_acc[dt][4 * g4 + 5] * inv_l);
      b.y = pack_bf16x2(o_acc[dt][4 * g4 + 6] * inv_l, o_acc[dt][4 * g4 + 7] * inv_l);
      const auto sx = __builtin_amdgcn_permlane32_swap(a.x, b.x, false, false);
      const auto sy = __builtin_amdgcn_permlane32_swap(a.y, b.y, false, false);
      a.x = sx[0];
      b.x = sx[1];
      a.y = sy[0];
      b.y = sy[1];
      if (row_valid)  // after the swaps: every lane takes part in them
        *reinterpret_cast<uint4*>(op + dt * 32 + 8 * g4 + 8 * h) = make_uint4(a.x, a.y, b.x, b.y);
    }
}


}  // namespace

extern "C" int dx_prefill_attention(void* out, const void* q, int64_t q_stride, const void* k_cache,
                                    const void* v_cache, const int* block_tables, int bt_stride,
                                    const int* cu_seqlens_q, const int* ctx_lens, const int* work, int n_work,
                                    int n_q_heads, int n_kv_heads, int head_dim, int block_size, float scale,
                                    int causal, int n_waves, hipStream_t stream) {
  if (head_dim != D || n_q_heads % n_kv_heads) return -1;
  const int G = n_q_heads / n_kv_heads;
  const int hpw = G >= 4 ? 4 : G;
  if (G % hpw || (hpw != 1 && hpw != 2 && hpw != 4)) return -2;
  if (n_work == 0) return 0;
  const int bs_shift = __builtin_ctz((unsigned)block_size);
  if (block_size < 4 || (1 << bs_shift) != block_size) return -3;
  // Workgroups of eight waves stage every K/V tile once for all of them; of four, two to a CU, out of step with each other
  // and with half as much work in the last and the longest of them.  32 / 8 heads, us, eight / four: one prompt of 2000 61.9 /
  // 54.8 (256 workgroups of eight), six of 3000 together 32.2 / 29.7 (392), 300 rows behind 2900 cached 92.7 / 71.0 (40),
  // two of 5000 136.3 / 138.2 (632), three of 6151 152.4 / 151.2 (776).
  // n_waves 92 selects the first loop, of eight waves (A/B runs: tools/attn_ab.py, tools/attn_accuracy.py)
  const bool r3 = n_waves == 92;
  const bool four = !r3 && (int64_t)n_kv_heads * (G / hpw) * n_work < 512;
  const dim3 grid(n_kv_heads * (G / hpw), n_work * (four ? 2 : 1));
  const float sl2e = scale * 1.4426950408889634f;
#define DX_PA_LAUNCH(BS, VV, NW)                                                                                     \
  prefill_attn_v2_kernel<BS, true, VV, NW><<<grid, 64 * NW, 0, stream>>>(                                            \
      (bf16_t*)out, (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables,        \
      bt_stride, cu_seqlens_q, ctx_lens, work, n_q_heads, n_kv_heads, bs_shift, hpw, sl2e, causal)
#define DX_PA(BS)                    \
  do {                               \
    if (r3) DX_PA_LAUNCH(BS, 0, 8);  \
    else if (four) DX_PA_LAUNCH(BS, 1, 4); \
    else DX_PA_LAUNCH(BS, 1, 8);     \
  } while (0)
  if (block_size >= 64) DX_PA(true);
  else DX_PA(false);
#undef DX_PA
#undef DX_PA_LAUNCH
  return (int)hipGetLastError();
}

// query tokens per work item (the Python work list must use the same value)
extern "C" int dx_prefill_tile_tokens(int n_q_heads, int n_kv_heads, int n_waves) {
  const int G = n_q_heads / n_kv_heads;
  const int hpw = G >= 4 ? 4 : G;
  (void)n_waves;
  return (8 / hpw) * BQ;  // 8 waves x 32 query rows over hpw heads
}
