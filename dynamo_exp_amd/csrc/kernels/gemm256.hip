// Large-M projection GEMM for gfx950 (prefill token counts), three epilogues:
//   EPI_STORE:  y[M, N]   = x[M, K] . w[N, K]^T
//   EPI_SILU:   y[M, N/2] = silu(g) * u, where the N weight rows are the MLP's
//               gate and up projections interleaved in blocks of 32 rows
//               (g0..g31, u0..u31, g32..g63, u32..u63, ...; ops.interleave_gate_up):
//               the SwiGLU of the Llama MLP fused into the gate_up GEMM, so the
//               [M, 2F] intermediate is never written or re-read and the
//               separate silu_and_mul launch disappears.
//   EPI_ADD:    y[M, N]  += x[M, K] . w[N, K]^T, for a residual stream behind a
//               long sum (the MLP's down projection)
// bf16 in / out, fp32 accumulation.
//
// Design (CDNA4 guide §5 "256² 8-phase template", re-derived here):
//   * 256 x 256 output tile per workgroup, K in 64-deep tiles, 8 waves as
//     2 (tokens) x 4 (weight rows); each wave owns 128 tokens x 64 weight rows
//     = 8 x 4 tiles of v_mfma_f32_16x16x32_bf16 (128 accumulator registers).
//     Operands are swapped (A = weight rows, B = token rows) so that every lane
//     ends up holding 4 consecutive output columns of one token: 8-byte stores,
//     and the gate tile and its up tile sit in the same lanes and registers.
//   * Both operands are staged HBM -> LDS by LDS-DMA (global_load_lds_dwordx4,
//     no staging registers), two 64-KB buffers (x tile + w tile each).  The
//     image is lane-linear (8 rows x 128 B per wave instruction) and XOR-
//     swizzled by choosing each lane's SOURCE chunk: slot s of row r holds
//     chunk s ^ ((r >> 1) & 7), which makes every 16-lane group of the
//     ds_read_b128 fragment reads hit 16 distinct bank slots.
//   * Each K-tile runs in 2 phases, half of the wave's accumulators per phase
//     (32 MFMAs); a phase reads only the fragments it newly needs (the w
//     fragments stay in registers for the whole tile: 24 ds_read_b128 per wave
//     and K-tile):   p1: w + x-half 0 -> Q(x0, w)     p2: x-half 1 -> Q(x1, w)
//     The four "parts" of a buffer (x rows of half 0 / 1, w rows of half
//     0 / 1; 16 KB each) are refilled one phase after their last read.
//   * Waves 4-7 run one barrier (half a phase) behind waves 0-3 (two barriers
//     per phase), so the two waves of each SIMD alternate between their LDS-read
//     segment and their MFMA segment (guide §5 8-phase template, microarch "two
//     waves per SIMD" item 9).  Hazards under that stagger: every wave retires
//     its reads (lgkmcnt(0)) BEFORE the phase's first barrier, so the leading
//     group's refill one phase later cannot overtake the lagging group's reads;
//     the DMA waits sit at the end of each phase and cover the parts read two
//     phases later (one barrier before the lagging group reads them).
//   * Grouped mode (mixture of experts): the token rows are sorted by expert
//     (order / offsets, built on the device), an expert's run of rows is cut
//     into row tiles against that expert's weight matrix w[e] (w is
//     [E, N, K]), x rows are gathered per lane (the DMA takes any row address)
//     and y rows scattered by the same map.  The tiles of an expert are as many
//     as 256 rows each need, all of one height (a multiple of 32: 312 rows are
//     2 x 160, not 256 + 56), half of a tile's 16-row blocks in each phase; the
//     blocks that a lower tile does not have are neither read nor multiplied.
//     The host does not know the experts' row counts, so the workgroups count
//     the tiles before they split them.  Bound by the weights' way from HBM up to
//     some 300 rows per expert, above by the matrix cores.  Expert part of a
//     layer, 16 experts of width 3584, 2 a token, model width 4096, us: 300
//     tokens 421 -> 307 (1.41 GB of weights: 4.6 TB/s), 1000 462 -> 390, 2500
//     667 -> 539, 4000 854 -> 754; 8 experts of 2048, width 2048, 2500: 186 -> 186.
//   * EPI_ADD with a last round that fills at most half of the CUs: its tiles are
//     cut along K into as many pieces as there are CUs for (16 at most), the
//     pieces' fp32 sums go through a workspace (256 pieces, 67 MB at most) to a kernel that
//     adds them in order.  One more round costs 230 to 320 us at K 14336, whatever
//     it holds; a sixteenth of one costs 20 and the way through the workspace 30:
//     4150 x 4096 520 -> 365 us, 1000 x 4096 227 -> 104.  Where it fills somewhat more,
//     half as many tiles as there are CUs go out in two pieces each and the others in
//     as many as fit beside each other, three at least (512 pieces, 134 MB at most), if K
//     is long enough for that (kWorth): a round is cut to half of one and a third or less.
//     K 14336: 6151 x 4096 575 -> 534 us, 6500 583 -> 554, 6800 598 -> 579, 12492 x 2048
//     606 -> 530; K 28672: 3100 x 8192 1132 -> 1055.
//     (In full rounds the
//     card's power is the bound, not the schedule: the matrix cores are busy
//     80 % of the cycles, and the clock is 1.75 GHz where launches stand alone,
//     1.5 in a prompt step: profiles/step_case_counters.txt.)  A row's sum is
//     cut or not by the tile it lies in, so equal rows of a step may differ by
//     a rounding, as they do with the library at most of these sizes.
//   * Blocks are remapped so that each XCD walks a contiguous range of tiles
//     (bijective for any grid size), in bands of group_m token tiles: the ~32
//     workgroups resident on one XCD then share group_m x tiles and
//     32 / group_m weight tiles through that XCD's L2.
#include "common.h"

#include <algorithm>
#include <cstdlib>

namespace {

constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kTile = 256 * 128;   // one operand tile: 256 rows x 64 bf16
constexpr int kBuf = 2 * kTile;    // x tile + w tile
constexpr int kLds = 2 * kBuf;     // double buffered: 128 KB

// EPI_SILU_RS: EPI_SILU whose input rows carry a deferred RMSNorm: g and u
// are scaled by rs[token] (1 / rms of the row) before the activation -- the
// norm's weight is folded into the weight columns (models/llama.py)
// EPI_ADD: y += x . w^T (one rounding), the tiles of an incomplete last round split along K (Split)
enum { EPI_STORE = 0, EPI_SILU = 1, EPI_SILU_RS = 2, EPI_ADD = 3 };

// EPI_ADD: tiles 0 .. full - 1 are whole; each of the rest[0] behind them is segs[0] pieces of K, and each of the rest[1]
// behind those segs[1].  Their fp32 sums go to part[piece * rest + tile][block (i, j) of the wave][thread] (the second kind's
// behind all of the first one's) and are joined by gemm256_join_kernel.
struct Split {
  f32x4* part;
  int full, rest[2], segs[2];
};
// Two kinds of pieces: the least K times the part of K that they save.  The pieces' way to
// the workspace and back is 134 MB each way whatever K is.  6151 / 6500 / 6800 / 7100 / 7300 x 4096 (16, 8, 5, 4, 3 pieces of the second kind), time over that of whole
// tiles: K 10240 1.05 1.02 1.04 1.04 1.06, 11520 1.00 1.01 1.03 1.04 1.03, 12288 0.98 0.99 1.00 1.00 1.02, 14336 0.93 0.95 0.97
// 0.99 1.00, 18432 0.91 0.94 0.95 0.97 0.99, 28672 0.89 0.92 0.93 0.96 0.98; 3100 / 3500 x 8192 (8, 4) K 12288 1.01 1.04, 14336
// 0.98 1.02, 28672 0.93 0.98; N 2048 gains from K 10240 on.  What loses anywhere lies below 59e6 (K 16384, 4 pieces: 67e6, 0.97).
constexpr int64_t kWorth = 60000000;

__device__ __forceinline__ float silu_f(float g) { return g / (1.f + __expf(-g)); }

// Grouped mode: sorted row r (offsets[e] <= r < offsets[e + 1] belongs to expert e)
// reads x row order[r] / top (gather) or r, and writes y row order[r] (scatter) or r.
struct GroupMap {
  const int* order;
  const int* offsets;
  int E, top, gather, scatter;
};

// four bf16 plus four sums, rounded once
__device__ __forceinline__ uint2 add_bf16x4(uint2 a, f32x4 v) {
  return uint2{pack_bf16x2(bf16lo(a.x) + v[0], bf16hi(a.x) + v[1]), pack_bf16x2(bf16lo(a.y) + v[2], bf16hi(a.y) + v[3])};
}

// tile lid -> (token tile, weight tile): bands of group_m token tiles across all weight tiles, token tile fastest
__device__ __forceinline__ void tile_of(int lid, int mtn, int ntn, int group_m, int& mt, int& nt) {
  const int band = lid / (group_m * ntn), first_m = band * group_m;
  const int gsz = min(mtn - first_m, group_m), in_band = lid - band * group_m * ntn;
  mt = first_m + in_band % gsz;
  nt = in_band / gsz;
}

template <int EPI, bool GRP>
__global__ void __launch_bounds__(512) gemm256_kernel(bf16_t* __restrict__ y, int64_t ldy,
                                                      const bf16_t* __restrict__ x, int64_t ldx,
                                                      const bf16_t* __restrict__ w, int M, int N, int K,
                                                      int group_m, const float* __restrict__ rs, GroupMap gm,
                                                      Split sp) {
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int l15 = lane & 15, lq = lane >> 4;

  // ---- persistent, XCD-aware tile order: the workgroups on one XCD (blocks
  // b, b + 8, ...) walk one contiguous range of logical tiles, stride = their
  // count, so the ~32 tiles in flight on an XCD are always neighbours
  // grouped: the experts' row tiles are counted here (the host only knows a bound, and tiles that do not exist would
  // leave the XCDs they fall to without work: they lie behind the others, and with a bound of
  // 36 row tiles for 32 the last XCD had a ninth of the others' work)
  int mtn = (M + kBM - 1) / kBM;
  if constexpr (GRP) {
    int n = 0;
    for (int e = lane; e < gm.E; e += 64) n += (gm.offsets[e + 1] - gm.offsets[e] + kBM - 1) / kBM;
    for (int d = 32; d; d >>= 1) n += __shfl_xor(n, d);
    mtn = __builtin_amdgcn_readfirstlane(n);
  }
  const int ntn = N / kBN, nwg = EPI == EPI_ADD ? sp.full : mtn * ntn;
  const int G = gridDim.x, bid = blockIdx.x, xcd = bid & 7;
  const int gq = G >> 3, gr8 = G & 7;                 // workgroups on this XCD: gq (+1)
  const int per_xcd = xcd < gr8 ? gq + 1 : gq;
  const int q = nwg >> 3, rr = nwg & 7;               // logical tiles owned by this XCD
  const int t_begin = xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q;
  const int t_end = t_begin + (xcd < rr ? q + 1 : q);

  // ---- DMA sources: part P (0 = x half 0, 1 = x half 1, 2 = w half 0, 3 = w half 1),
  // instruction i of this wave covers part rows pr = 16 wave + 8 i + (lane >> 3)
  int prow[4][2];  // part row of this lane's source
  int goff[4][2];
  int loff[4][2];
#pragma unroll
  for (int P = 0; P < 4; ++P)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int pr0 = 16 * wave + 8 * i;
      const int pr = pr0 + (lane >> 3);
      const int h = P & 1;
      int row, row0;
      if (P < 2) {
        row = (pr >> 6) * 128 + h * 64 + (pr & 63);
        row0 = (pr0 >> 6) * 128 + h * 64 + (pr0 & 63);
      } else {
        row = (pr >> 5) * 64 + h * 32 + (pr & 31);
        row0 = (pr0 >> 5) * 64 + h * 32 + (pr0 & 31);
      }
      const int ch = (lane & 7) ^ ((row >> 1) & 7);
      prow[P][i] = row;
      goff[P][i] = (P < 2 ? 0 : row * K) + ch * 8;  // x rows: + clamped row * ldx per tile
      loff[P][i] = (P < 2 ? 0 : kTile) + row0 * 128;
    }
  const int nkt = K / kBK;
  const bf16_t* xb = x;
  const bf16_t* wb = w;
  int xoff[2][2];  // per tile: x part offsets (rows past M re-read row M-1)
  int kbase = 0, nk = nkt;  // K tiles of this unit of work
  auto issue = [&](int P, int kt, int buf) {
    kt = min(kt, nk - 1) + kbase;  // past the end: harmless reload into a buffer that is not read again
    const bf16_t* src = (P < 2 ? xb : wb) + kt * kBK;
    char* dst = smem + buf * kBuf;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(src + (P < 2 ? xoff[P][i] : goff[P][i]), (lds_void*)(dst + loff[P][i]), 16,
                                       0, 0);
  };

  // ---- fragment read addresses (row = 16-row tile base + l15; the XOR term of
  // a 16-aligned base is (l15 >> 1))
  const int c0 = (lq ^ (l15 >> 1)) << 4, c1 = ((4 + lq) ^ (l15 >> 1)) << 4;
  const int fx = (wr * 128 + l15) * 128, fw = kTile + (wc * 64 + l15) * 128;

  f32x4 acc[4][8];
  bf16x8_t xf[4][2], wf[4][2];

  // grouped: 16-row blocks of this tile that each wave owns, in the two phases
  int n1 = 4, n2 = 4;
  auto read_x = [&](const char* b, int xh) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (GRP && j >= (xh ? n2 : n1)) break;
      const char* p = b + fx + (xh * 4 + j) * 2048;
      xf[j][0] = *reinterpret_cast<const bf16x8_t*>(p + c0);
      xf[j][1] = *reinterpret_cast<const bf16x8_t*>(p + c1);
    }
  };
  auto read_w = [&](const char* b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const char* p = b + fw + i * 2048;
      wf[i][0] = *reinterpret_cast<const bf16x8_t*>(p + c0);
      wf[i][1] = *reinterpret_cast<const bf16x8_t*>(p + c1);
    }
  };
  // Two 32-MFMA phases per K-tile (one barrier hand-off per phase and wave
  // group; four 16-MFMA phases measured 4-7 % slower, profiles/r2_gemm256.txt):
  //   p1: all w + x-half 0 -> Q(x0, w)    p2: x-half 1 -> Q(x1, w)
  // x half 1 of tile t+1 is refilled in p1 of tile t (its buffer's last read
  // was p2 of tile t-1), the other three parts of tile t+2 in p2; reads of
  // phase q are covered by the wait at the end of phase q-2 (stagger rule).
  auto mma2 = [&](int xh) {
    if constexpr (GRP) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= (xh ? n2 : n1)) break;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[i][xh * 4 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][s], xf[j][s], acc[i][xh * 4 + j], 0, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][xh * 4 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][s], xf[j][s], acc[i][xh * 4 + j], 0, 0, 0);
  };
  auto compute2 = [&](int xh, int vm) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    mma2(xh);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    if (vm == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");  // tile t+1's x0 / w landed
    if (vm == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  // tile t+1's x1 landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto ktile2 = [&](int t, int buf) {
    const char* b = smem + buf * kBuf;
    read_w(b);
    read_x(b, 0);
    issue(1, t + 1, buf ^ 1);
    compute2(0, 2);
    read_x(b, 1);
    issue(0, t + 2, buf);
    issue(2, t + 2, buf);
    issue(3, t + 2, buf);
    compute2(1, 6);
  };

  // (tile_of) the ~32 workgroups resident on an XCD
  // cover group_m x (32 / group_m) tiles (8 x 4: 12 KB of new operand bytes per
  // workgroup and K-step through the XCD's L2 instead of 33 KB for one weight
  // tile x 32 token tiles)
  int mt = 0, nt = 0;
  int row0 = 0, rend = 0;  // grouped: this tile's first sorted row and its expert's end
  auto select = [&](int lid) {
    tile_of(lid, mtn, ntn, group_m, mt, nt);
    if constexpr (GRP) {
      int e = 0, rem = mt, lo = 0, hi = 0;
      for (; e < gm.E; ++e) {
        lo = gm.offsets[e];
        hi = gm.offsets[e + 1];
        const int n = (hi - lo + kBM - 1) / kBM;
        if (rem < n) break;
        rem -= n;
      }
      // the expert's rows in tiles of one height, in 32s
      const int blocks = (hi - lo + 31) >> 5, tiles = (hi - lo + kBM - 1) / kBM, nj = (blocks + tiles - 1) / tiles;
      n1 = (nj + 1) >> 1;
      n2 = nj - n1;
      row0 = lo + rem * 32 * nj;  // (before hi: a tile fewer would not hold the rows at 8 blocks each)
      rend = min(row0 + 32 * nj, hi);
      xb = x;
      wb = w + ((int64_t)e * N + (int64_t)nt * kBN) * K;
#pragma unroll
      for (int P = 0; P < 2; ++P)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int in = prow[P][i] & 63;  // (a part's rows behind its blocks: one row for all of them)
          const int r = in < 16 * (P ? n2 : n1) ? min(row0 + (prow[P][i] >> 7) * 16 * nj + P * 16 * n1 + in, rend - 1) : row0;
          const int src = gm.gather ? gm.order[r] / gm.top : r;
          xoff[P][i] = src * (int)ldx + goff[P][i];
        }
      return;
    }
    xb = x + (int64_t)mt * kBM * ldx;
    wb = w + (int64_t)nt * kBN * K;
#pragma unroll
    for (int P = 0; P < 2; ++P)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        xoff[P][i] = (min(mt * kBM + prow[P][i], M - 1) - mt * kBM) * (int)ldx + goff[P][i];
  };
  // prologue of a tile: tile 0 of K, then K-tile 1 without its x half 1 (issued in p1 of K-tile 0)
  auto prologue = [&]() {
    issue(0, 0, 0);
    issue(2, 0, 0);
    issue(3, 0, 0);
    issue(1, 0, 0);
    issue(0, 1, 1);
    issue(2, 1, 1);
    issue(3, 1, 1);
  };

  int pieces = 0, slot = 0;  // EPI_ADD: kinds of pieces of K that this workgroup has come to (it takes number `unit` of each)
  const int unit = (xcd < gr8 ? xcd * (gq + 1) : gr8 * (gq + 1) + (xcd - gr8) * gq) + (bid >> 3);
  auto begin = [&](int lid) -> bool {
    if (lid < t_end) {
      select(lid);
      return true;
    }
    if constexpr (EPI == EPI_ADD) {
      // the workgroups of an XCD take the same piece of neighbouring tiles
      const int first = sp.rest[0] * sp.segs[0];
      if (pieces == 0 && unit >= first) ++pieces;
      if (pieces == 2 || (pieces == 1 && unit >= sp.rest[1] * sp.segs[1])) return false;
      const int rest = pieces ? sp.rest[1] : sp.rest[0], segs = pieces ? sp.segs[1] : sp.segs[0];
      const int c = unit / rest, pairs = nkt / 2;
      kbase = pairs * c / segs * 2;
      nk = pairs * (c + 1) / segs * 2 - kbase;
      select(sp.full + (pieces ? sp.rest[0] : 0) + unit - c * rest);
      slot = (pieces ? first : 0) + unit;
      ++pieces;
      return true;
    }
    return false;
  };
  int lid = t_begin + (bid >> 3);
  if (!begin(lid)) return;
  prologue();
  for (;;) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // K-tile 0 landed (the stores of the previous tile, issued after this
    // prologue, are in flight underneath: the wait covers them as well)
    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (wave >= 4) __builtin_amdgcn_s_barrier();  // start the lagging group one barrier late
    __builtin_amdgcn_sched_barrier(0);
    for (int t = 0; t < nk; t += 2) {
      ktile2(t, 0);
      ktile2(t + 1, 1);
    }
    if (wave < 4) __builtin_amdgcn_s_barrier();  // balance the barrier count: every LDS read of this tile is done
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped tail reloads landed before the buffers are refilled

    const int cmt = mt, cnt = nt;
    const int tok0 = (GRP ? row0 + wr * 16 * (n1 + n2) : cmt * kBM + wr * 128) + l15;
    const int c1n = GRP ? n1 : 4, cn = GRP ? n1 + n2 : 8;  // (the next tile's select changes n1 and n2)
    // accumulator column j: block j of phase one, block j - 4 of phase two
    auto block = [&](int j) { return GRP ? (j < 4 ? j : c1n + j - 4) : j; };
    auto absent = [&](int j) { return GRP && (j < 4 ? j >= c1n : c1n + j - 4 >= cn); };
    const int tok_end = GRP ? rend : M;
    // grouped + scatter: the 8 destination rows, loaded and retired like the row scales below
    int dstv[8];
    if constexpr (GRP) {
#pragma unroll
      for (int j = 0; j < 8; ++j) dstv[j] = gm.scatter ? gm.order[min(tok0 + 16 * block(j), tok_end - 1)] : tok0 + 16 * block(j);
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" ::"v"(dstv[j]));
    }
    // EPI_SILU_RS: the 8 row scales this lane needs, loaded in one batch and
    // retired BEFORE the next tile's prologue DMA is queued (the empty asm
    // consumes them): vmcnt retires in order, and the compiler otherwise
    // waits with vmcnt(0) in the epilogue -- for the whole prologue too (the
    // first version: 15 % slower per GEMM, profiles/r6_fold_pmc.txt)
    float scv[8];
    if (EPI == EPI_SILU_RS) {
#pragma unroll
      for (int j = 0; j < 8; ++j) scv[j] = rs[min(tok0 + 16 * j, M - 1)];
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" ::"v"(scv[j]));
    }

    // the next tile's first K-tiles go out before this tile's stores
    if constexpr (EPI == EPI_ADD) {
      // (in front of the next unit's prologue: its DMA would retire before the loads of y)
      const bool piece = pieces > 0;
      if (piece) {
        f32x4* o = sp.part + (int64_t)slot * (kBM * kBN / 4) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j) o[(i * 8 + j) * 512] = acc[i][j];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int tok = tok0 + 16 * j;
        if (piece || tok >= tok_end) continue;
        bf16_t* yr = y + (int64_t)tok * ldy + cnt * kBN + wc * 64 + 4 * lq;
        uint2 was[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) was[i] = *reinterpret_cast<const uint2*>(yr + 16 * i);
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(yr + 16 * i) = add_bf16x4(was[i], acc[i][j]);
      }
    }
    lid += per_xcd;
    const bool more = begin(lid);
    if (more) prologue();

    // ---- epilogue: acc[i][j] register r = (weight row wc*64 + 16 i + 4 lq + r, token 16 j + l15)
    if (EPI == EPI_ADD) {
      // done above
    } else if (EPI == EPI_STORE) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int tok = tok0 + 16 * block(j);
        if (absent(j) || tok >= tok_end) continue;
        bf16_t* yr = y + (int64_t)(GRP ? dstv[j] : tok) * ldy + cnt * kBN + wc * 64 + 4 * lq;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint2 pk;
          pk.x = pack_bf16x2(acc[i][j][0], acc[i][j][1]);
          pk.y = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
          *reinterpret_cast<uint2*>(yr + 16 * i) = pk;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int tok = tok0 + 16 * block(j);
        if (absent(j) || tok >= tok_end) continue;
        bf16_t* yr = y + (int64_t)(GRP ? dstv[j] : tok) * ldy + cnt * (kBN / 2) + wc * 32 + 4 * lq;
        const float sc = EPI == EPI_SILU_RS ? scv[j] : 1.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          f32x4 g = acc[i][j], u = acc[2 + i][j];
          if (EPI == EPI_SILU_RS) {
            g *= sc;
            u *= sc;
          }
          uint2 pk;
          pk.x = pack_bf16x2(silu_f(g[0]) * u[0], silu_f(g[1]) * u[1]);
          pk.y = pack_bf16x2(silu_f(g[2]) * u[2], silu_f(g[3]) * u[3]);
          *reinterpret_cast<uint2*>(yr + 16 * i) = pk;
        }
      }
    }
    if (!more) break;
  }
}

// y += the pieces of K of the tiles that EPI_ADD split.  grid (2 * 8, tiles), block 256: the 16 rows j of half of the
// tile's waves
__global__ void __launch_bounds__(256) gemm256_join_kernel(bf16_t* __restrict__ y, int64_t ldy, int M, int N, int group_m,
                                                           Split sp) {
  const int j = blockIdx.x & 7, thread = (blockIdx.x >> 3) * 256 + threadIdx.x, wave = thread >> 6;
  const int wr = wave >> 2, wc = wave & 3, l15 = thread & 15, lq = (thread & 63) >> 4;
  int mt, nt;
  tile_of(sp.full + blockIdx.y, (M + kBM - 1) / kBM, N / kBN, group_m, mt, nt);
  const int tok = mt * kBM + wr * 128 + 16 * j + l15;
  if (tok >= M) return;
  bf16_t* yr = y + (int64_t)tok * ldy + nt * kBN + wc * 64 + 4 * lq;
  uint2 was[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) was[i] = *reinterpret_cast<const uint2*>(yr + 16 * i);
  f32x4 sum[4] = {};
  const int kind = (int)blockIdx.y >= sp.rest[0], rest = kind ? sp.rest[1] : sp.rest[0], segs = kind ? sp.segs[1] : sp.segs[0];
  const f32x4* p = sp.part + ((int64_t)(kind ? sp.rest[0] * (sp.segs[0] - 1) : 0) + blockIdx.y) * (kBM * kBN / 4) + j * 512 + thread;
  for (int c = 0; c < segs; ++c, p += (int64_t)rest * (kBM * kBN / 4))
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] += p[i * 8 * 512];
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(yr + 16 * i) = add_bf16x4(was[i], sum[i]);
}

// one resident workgroup per CU (128 KB of LDS): a grid of min(tiles, CUs)
// workgroups walks all tiles
int num_cus() {
  static int n = 0;
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    // DX_GEMM256_CUS: persistent grid for a CU-masked stream (study knob; profiles/r4_mixed_split_cu_mask.txt)
    if (const char* e = getenv("DX_GEMM256_CUS")) n = std::max(1, atoi(e));
  }
  return n;
}

template <int EPI>
void launch(bf16_t* y, int64_t ldy, const bf16_t* x, int64_t ldx, const bf16_t* w, int M, int N, int K, int gm,
            int persistent, hipStream_t st, const float* rs) {
  const int tiles = ((M + kBM - 1) / kBM) * (N / kBN);
  const int grid = persistent ? std::min(tiles, num_cus()) : tiles;
  hipLaunchKernelGGL((gemm256_kernel<EPI, false>), dim3(grid), dim3(512), 0, st, y, ldy, x, ldx, w, M, N, K, gm, rs,
                     GroupMap{nullptr, nullptr, 0, 1, 0, 0}, Split{});
}

template <int EPI>
void launch_grouped(bf16_t* y, int64_t ldy, const bf16_t* x, int64_t ldx, const bf16_t* w, int R, int N, int K, int gm,
                    hipStream_t st, const GroupMap& map) {
  const int tiles = ((R + kBM - 1) / kBM + map.E) * (N / kBN);
  hipLaunchKernelGGL((gemm256_kernel<EPI, true>), dim3(std::min(tiles, num_cus())), dim3(512), 0, st, y, ldy, x, ldx, w,
                     R, N, K, gm, nullptr, map, Split{});
}

}  // namespace

// epi: 0 = store y[M, N]; 1 = SwiGLU y[M, N/2] over 32-row interleaved gate/up weights;
// 2 = SwiGLU with the rows' deferred-RMSNorm scales rs[M] (fp32) applied first.
// group_m: token tiles per L2 band.  Requirements: N % 256 == 0, K % 128 == 0,
// 16-byte aligned x / w, x row stride % 8 == 0, y row stride % 4 == 0, y 8-byte aligned.
extern "C" int dx_gemm256(void* y, int64_t ldy, const void* x, int64_t ldx, const void* w, int M, int N, int K,
                          int epi, int group_m, hipStream_t st, const float* rs) {
  if (M < 1) return 0;
  const int persistent = group_m < 1000;  // A/B switch: group_m + 1000 launches one workgroup per tile
  if (!persistent) group_m -= 1000;
  if (group_m < 1) return 7;
  if (N % kBN != 0 || K % (2 * kBK) != 0 || K < 2 * kBK) return 3;
  if ((ldx & 7) || (ldy & 3) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(w) & 15) ||
      (reinterpret_cast<uintptr_t>(y) & 7))
    return 5;
  if ((int64_t)N * K >= (1ll << 31) || (int64_t)kBM * ldx >= (1ll << 31)) return 6;  // 32-bit DMA offsets
  auto* Y = static_cast<bf16_t*>(y);
  auto* X = static_cast<const bf16_t*>(x);
  auto* W = static_cast<const bf16_t*>(w);
  if (epi == EPI_STORE) launch<EPI_STORE>(Y, ldy, X, ldx, W, M, N, K, group_m, persistent, st, nullptr);
  else if (epi == EPI_SILU) launch<EPI_SILU>(Y, ldy, X, ldx, W, M, N, K, group_m, persistent, st, nullptr);
  else if (epi == EPI_SILU_RS && rs != nullptr) launch<EPI_SILU_RS>(Y, ldy, X, ldx, W, M, N, K, group_m, persistent, st, rs);
  else return 2;
  DX_CHECK_LAUNCH();
  return 0;
}

// How dx_gemm256_add splits its tiles.  A last round that fills at most half of the CUs is cut along K into as many pieces
// as there are CUs for.  A fuller one: half as many tiles as CUs in two pieces each, then what is left like that, where this
// saves enough of K, (1 - 1 / 2 - 1 / pieces) K, for the way of 512 pieces through the workspace (kWorth).
static Split add_split(int M, int N, int K) {
  const int tiles = (M + kBM - 1) / kBM * (N / kBN), cus = num_cus(), left = tiles % cus, half = cus / 2;
  auto pieces = [&](int n) { return std::min(std::min(cus / n, 16), K / (2 * kBK)); };
  Split sp{nullptr, tiles, {0, 0}, {0, 0}};
  if (left == 0) return sp;
  if (2 * left <= cus) {
    sp.full = tiles - left, sp.rest[0] = left, sp.segs[0] = pieces(left);
  } else if (const int n = pieces(left - half); n > 2 && (int64_t)K * K * (n - 2) >= 2 * kWorth * n) {
    sp.full = tiles - left, sp.rest[0] = half, sp.segs[0] = 2, sp.rest[1] = left - half, sp.segs[1] = n;
  }
  return sp;
}

// fp32 workspace (floats) of dx_gemm256_add
extern "C" int64_t dx_gemm256_add_floats(int M, int N, int K) {
  if (M < 1 || N < kBN || N % kBN || K < 2 * kBK || K % (2 * kBK)) return 0;
  const Split sp = add_split(M, N, K);
  return (int64_t)(sp.rest[0] * sp.segs[0] + sp.rest[1] * sp.segs[1]) * kBM * kBN;
}

// y[M, N] += x[M, K] . w[N, K]^T, each element rounded once; ws: dx_gemm256_add_floats floats, 16-byte aligned.  Same
// requirements as dx_gemm256.
extern "C" int dx_gemm256_add(void* y, int64_t ldy, const void* x, int64_t ldx, const void* w, int M, int N, int K,
                              int group_m, float* ws, hipStream_t st) {
  if (M < 1) return 0;
  if (group_m < 1) return 7;
  if (N < kBN || N % kBN != 0 || K % (2 * kBK) != 0 || K < 2 * kBK) return 3;
  if ((ldx & 7) || (ldy & 3) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(w) & 15) ||
      (reinterpret_cast<uintptr_t>(y) & 7) || (reinterpret_cast<uintptr_t>(ws) & 15))
    return 5;
  if ((int64_t)N * K >= (1ll << 31) || (int64_t)kBM * ldx >= (1ll << 31)) return 6;  // 32-bit DMA offsets
  Split sp = add_split(M, N, K);
  sp.part = reinterpret_cast<f32x4*>(ws);
  if (sp.rest[0] && !ws) return 5;
  const int grid = std::max({std::min(sp.full, num_cus()), sp.rest[0] * sp.segs[0], sp.rest[1] * sp.segs[1]});
  auto* Y = static_cast<bf16_t*>(y);
  hipLaunchKernelGGL((gemm256_kernel<EPI_ADD, false>), dim3(grid), dim3(512), 0, st, Y, ldy, static_cast<const bf16_t*>(x),
                     ldx, static_cast<const bf16_t*>(w), M, N, K, group_m, nullptr, GroupMap{nullptr, nullptr, 0, 1, 0, 0}, sp);
  if (sp.rest[0])
    hipLaunchKernelGGL(gemm256_join_kernel, dim3(16, sp.rest[0] + sp.rest[1]), dim3(256), 0, st, Y, ldy, M, N, group_m, sp);
  DX_CHECK_LAUNCH();
  return 0;
}

// Grouped GEMM over the rows of each expert: w [E, N, K]; order [R] / offsets [E + 1]
// sort the R rows by expert (see GroupMap).  epi 0: y[dst, N]; epi 1: SwiGLU over 32-row
// interleaved gate/up rows of every w[e], y[dst, N/2].  x_rows: rows of x (its row
// addresses must fit 32-bit element offsets).  Same shape requirements as dx_gemm256.
extern "C" int dx_gemm256_grouped(void* y, int64_t ldy, const void* x, int64_t ldx, int64_t x_rows, const void* w,
                                  const int* order, const int* offsets, int R, int E, int N, int K, int top,
                                  int gather, int scatter, int epi, int group_m, hipStream_t st) {
  if (R < 1) return 0;
  if (E < 1 || top < 1 || group_m < 1 || !order || !offsets) return 7;
  if (N % kBN != 0 || K % (2 * kBK) != 0 || K < 2 * kBK) return 3;
  if ((ldx & 7) || (ldy & 3) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(w) & 15) ||
      (reinterpret_cast<uintptr_t>(y) & 7))
    return 5;
  if ((int64_t)N * K >= (1ll << 31) || x_rows * ldx >= (1ll << 31)) return 6;  // 32-bit DMA offsets
  const GroupMap map{order, offsets, E, top, gather, scatter};
  auto* Y = static_cast<bf16_t*>(y);
  auto* X = static_cast<const bf16_t*>(x);
  auto* W = static_cast<const bf16_t*>(w);
  if (epi == EPI_STORE) launch_grouped<EPI_STORE>(Y, ldy, X, ldx, W, R, N, K, group_m, st, map);
  else if (epi == EPI_SILU) launch_grouped<EPI_SILU>(Y, ldy, X, ldx, W, R, N, K, group_m, st, map);
  else return 2;
  DX_CHECK_LAUNCH();
  return 0;
}
