// Kernel templates of the segmented LoRA pass, bf16 on v_mfma_f32_16x16x32_bf16 (fp32 accumulate), instantiated by
// kernels_mfma.hip (rank up to 64) and kernels_rank128.hip.
//
// All of these kernels stream activations from HBM: the matrix cores are used
// because the vector ALUs could not keep up with 8 TB/s at these ranks, not
// because anything is compute bound.  Everything is laid out so that each
// wave-wide load covers whole 128-byte lines and every activation byte crosses
// HBM once per pass.
//
//   k_shrink_pair / k_shrink_dl / k_shrink_oct / k_shrink_finish    h = scale * x A^T (split over column slices when x is wide)
//   k_expand_mfma / k_expand_multi                     y += h B^T in place (rank <= 16 / above)
//   k_wgrad_pipe / k_wgrad_coop                        dA, dB: contraction over the rows of a chunk (rank <= 16 / above)
//   transpose_weights_job                              B^T, A^T copies for the backward shrink / expand
//
// MFMA operand layout used below (l = lane, 64 lanes):
//   A operand: lane l holds A[i = l % 16][k = 8 * (l / 16) .. + 8]   (8 bf16 = 16 B)
//   B operand: lane l holds B[k = 8 * (l / 16) .. + 8][j = l % 16]
//   D        : lane l holds D[i = 4 * (l / 16) + v][j = l % 16], v = 0..3
// The contraction index k may be permuted freely as long as A and B agree, and
// the output indices i, j may be mapped to any rows / columns: both freedoms
// are used to make the global accesses contiguous.
#pragma once

#include <algorithm>

#include <type_traits>

#include "tk_mfma.h"

// depths of the software pipelines of k_dy_fused<1>, k_dy_fused<2> (one tile: with two blocks of accumulators a second
// tile in registers leaves one wave per SIMD), k_wgrad_pipe<1, S> and k_wgrad_coop<NB, S> (tiles in registers per wave)
#ifndef TK_DY_STAGES
#define TK_DY_STAGES 2
#endif
#ifndef TK_DY_STAGES2
#define TK_DY_STAGES2 1
#endif
#ifndef TK_COOP_STAGES
#define TK_COOP_STAGES 3
#endif
#ifndef TK_WGRAD_STAGES
#define TK_WGRAD_STAGES 3
#endif

// pairs of waves per block of k_wgrad_coop (see wgrad_coop_body)
#ifndef TK_COOP_PAIRS
#define TK_COOP_PAIRS 2
#endif

// h operands of k_expand_multi through LDS (once per block) or straight from memory (once per wave)
#ifndef TK_EXPAND_LDS_H
#define TK_EXPAND_LDS_H 1
#endif

// block renumbering of the rank > 16 expand (contiguous runs of tiles per XCD)
#ifndef TK_XCD_MAP
#define TK_XCD_MAP(b, n) xcd_contiguous(b, n)
#endif

namespace tk {

namespace {

// Scales, rounds and writes one tile of h from `planes` partial planes in LDS ([plane][32][RP + 1]):
// slot-major (hrow) and rank-major (hT); padding slots (row >= cnt) get exact zeros.
template <int RP, int THREADS>
__device__ inline void shrink_epilogue(const float* part, int planes, const PassArgs& a, bf16_t* __restrict__ hrow,
                                       int slot0, int cnt, float sc) {
  constexpr int PR = RP + 1;
  const int tid = threadIdx.x;
  bf16_t* hT = (bf16_t*)a.hT;
  // slot-major copy: consecutive threads -> consecutive rank indices of one slot
  for (int idx = tid; idx < kTileRows * RP; idx += THREADS) {
    const int row = idx / RP, n = idx % RP;
    float sum = 0.f;
    for (int w = 0; w < planes; ++w) sum += part[(w * kTileRows + row) * PR + n];
    hrow[(int64_t)(slot0 + row) * RP + n] = row < cnt ? (bf16_t)(pack_bf16(sum * sc, 0.f) & 0xffffu) : (bf16_t)0;
  }
  // rank-major copy: consecutive threads -> consecutive slots of one rank index
  for (int idx = tid; idx < kTileRows * RP; idx += THREADS) {
    const int n = idx >> 5, row = idx & 31;
    float sum = 0.f;
    for (int w = 0; w < planes; ++w) sum += part[(w * kTileRows + row) * PR + n];
    hT[(int64_t)n * a.ldh + slot0 + row] = row < cnt ? (bf16_t)(pack_bf16(sum * sc, 0.f) & 0xffffu) : (bf16_t)0;
  }
}

// ---------------------------------------------------------------------------
// Shrink: h[slot][n] = scale_g * sum_k src[row(slot)][k] * W1_g[n][k].
//
// Work item = (two consecutive tiles of 32 padded slots, slice of 512*NW source columns), one block of
// NW waves; the slices of a tile pair are consecutive blocks, so neighbouring waves read neighbouring
// 1 KB pieces of the same rows.  The grid is thousands of short independent streams: the hardware
// dispatcher keeps every CU equally loaded, which a tile-per-workgroup split does not (2.03 workgroups
// per CU leaves most CUs waiting for the few that got 3).  A wave takes 64-column steps, interleaved
// with the other waves of its block, keeps its partial h[32][rank] of both tiles in MFMA accumulators
// and issues the loads of two steps before the first MFMA of the batch.  Every weight operand feeds both
// tiles: at rank 64 a step has 8 weight loads for 4 source loads per tile, and with one tile per block the
// load pipeline, not memory, set the pace (rank 64: 129 -> 87 us; rank 16: 2 us).  Consecutive tiles
// almost always belong to the same group; a pair that straddles a group boundary is done one tile at a
// time.  The waves' partials meet in LDS; if the source is wider than one block the block sums go to
// a global buffer and k_shrink_finish adds the slices in slice order (a device-scope fence per block,
// the alternative, costs a cache write-back on this multi-die part).  Summation order is fixed
// throughout: results are bitwise repeatable.  The result is scaled, rounded to bf16 and written
// twice: slot-major (hrow, the expand kernel's A operand) and rank-major (hT, read by the
// weight-gradient kernels); padding slots get exact zeros.
// ---------------------------------------------------------------------------
// PF: steps whose loads are issued together
template <int NB, int NW, int TT, int PF = 2>
__device__ inline void shrink_tiles(const PassArgs& a, bf16_t* __restrict__ hrow, const int32_t* __restrict__ slot_rows,
                                    const int (&tiles)[TT], int g, int ks, float (*part)[kTileRows][16 * NB + 1]) {
  constexpr int RP = 16 * NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const bf16_t* src = (const bf16_t*)a.src;
  const bf16_t *xa[TT], *xb[TT];
  int cnt[TT];
#pragma unroll
  for (int u = 0; u < TT; ++u) {
    const int slot0 = tiles[u] * kTileRows;
    int ra = slot_rows[slot0 + li], rb = slot_rows[slot0 + 16 + li];
    // padding is always at the end of a tile: count the valid slots
    cnt[u] = __popcll(__ballot(ra >= 0) & 0xffffull) + __popcll(__ballot(rb >= 0) & 0xffffull);
    ra = min(max(ra, 0), a.src_rows - 1);
    rb = min(max(rb, 0), a.src_rows - 1);
    xa[u] = src + (int64_t)ra * a.ld_src + 16 * kb;
    xb[u] = src + (int64_t)rb * a.ld_src + 16 * kb;
  }
  const int r = class_rank(a.rank[g], a.rank_lo, RP);
  if (a.class_mode && r <= 0) return;  // a group of another rank class (uniform over the block): nothing is requested
  const bf16_t* W1 = group_weight<bf16_t>(a.w_shrink, a.w_shrink_base, a.shrink_group_stride, g);
  const bf16_t* wp[NB];
  bool wv[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = 16 * nb + li;
    wv[nb] = n < r;
    wp[nb] = W1 + (int64_t)(wv[nb] ? n : 0) * a.ld_shrink + 16 * kb;
  }
  f32x4 acc[TT][2][NB];
#pragma unroll
  for (int u = 0; u < TT; ++u)
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[u][tt][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nsteps = a.width_src >> 6;
  const int s_first = ks * (kShrinkSteps * NW) + wave;
#pragma unroll
  for (int b = 0; b < kShrinkSteps / PF; ++b) {
    uint4 x0[PF][TT][2], x1[PF][TT][2], w0[PF][NB], w1[PF][NB];
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int s = s_first + (b * PF + j) * NW;
      const bool ok = s < nsteps;  // wave-uniform
      const int c = (ok ? s : 0) << 6;
#pragma unroll
      for (int u = 0; u < TT; ++u) {
        x0[j][u][0] = ld16(xa[u] + c);
        x1[j][u][0] = ld16(xa[u] + c + 8);
        x0[j][u][1] = ld16(xb[u] + c);
        x1[j][u][1] = ld16(xb[u] + c + 8);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        w0[j][nb] = (wv[nb] && ok) ? ld16(wp[nb] + c) : zero4();
        w1[j][nb] = (wv[nb] && ok) ? ld16(wp[nb] + c + 8) : zero4();
      }
    }
    if constexpr (PF == kShrinkSteps) __builtin_amdgcn_sched_barrier(0);  // (or the loads are spread over the products)
#pragma unroll
    for (int j = 0; j < PF; ++j)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int u = 0; u < TT; ++u)
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) {
            acc[u][tt][nb] = mfma16(x0[j][u][tt], w0[j][nb], acc[u][tt][nb]);
            acc[u][tt][nb] = mfma16(x1[j][u][tt], w1[j][nb], acc[u][tt][nb]);
          }
  }
  if (r <= 0) return;  // adapter not live on this layer (uniform over the block)
  const float sc = a.scale[g];
#pragma unroll
  for (int u = 0; u < TT; ++u) {
    __syncthreads();  // the previous tile's sums have been read
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[wave][16 * tt + 4 * kb + v][16 * nb + li] = acc[u][tt][nb][v];
    __syncthreads();
    if (a.kslices > 1) {
      // the source is wider than one block: leave this block's sums for k_shrink_finish
      float* mine = a.hpart + ((int64_t)tiles[u] * a.kslices + ks) * (kTileRows * RP);
      for (int idx = tid; idx < kTileRows * RP; idx += NW * 64) {
        const int row = idx / RP, n = idx % RP;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += part[w][row][n];
        mine[idx] = sum;
      }
    } else {
      shrink_epilogue<RP, NW * 64>(&part[0][0][0], NW, a, hrow, tiles[u] * kTileRows, cnt[u], sc);
    }
  }
}

template <int NB, int NW>
__device__ __forceinline__ void shrink_pair_body(const PassArgs& a, bf16_t* __restrict__ hrow,
                                                 const int32_t* __restrict__ tile_group,
                                                 const int32_t* __restrict__ slot_rows, int max_tiles, int item) {
  __shared__ float part[NW][kTileRows][16 * NB + 1];
  const int nth = item / a.kslices, ks = item - nth * a.kslices;
  const int pair = work_item(a.wl_pairs, nth);
  if (pair < 0) return;  // past the end of this rank class's list (uniform over the block)
  const int t0 = 2 * pair, t1 = t0 + 1;
  if (t0 >= max_tiles) return;
  const int g0 = checked_group(tile_group[t0], a.tb);
  const int g1 = t1 < max_tiles ? checked_group(tile_group[t1], a.tb) : -1;
  if (g0 >= 0 && g1 == g0) {
    const int tiles[2] = {t0, t1};
    shrink_tiles<NB, NW, 2>(a, hrow, slot_rows, tiles, g0, ks, part);
    return;
  }
  if (g0 >= 0) {
    const int tiles[1] = {t0};
    shrink_tiles<NB, NW, 1>(a, hrow, slot_rows, tiles, g0, ks, part);
  }
  if (g1 >= 0) {
    const int tiles[1] = {t1};
    shrink_tiles<NB, NW, 1>(a, hrow, slot_rows, tiles, g1, ks, part);
  }
}

template <int NB, int NW>
__global__ __launch_bounds__(NW * 64) void k_shrink_pair(PassArgs a, bf16_t* __restrict__ hrow,
                                                         const int32_t* __restrict__ tile_group,
                                                         const int32_t* __restrict__ slot_rows, int max_tiles) {
  shrink_pair_body<NB, NW>(a, hrow, tile_group, slot_rows, max_tiles, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Shrink with the weights shared through LDS, for groups of many tiles.  In k_shrink_pair every wave fetches the
// weight columns of its own steps, 16 * NB rank indices for 64 rows: at rank 64 as many bytes of weights (from L2)
// as of activations (from memory), and the two share the path between L2 and the CUs, which is what sets the pace
// (measured at rank 64: 536 MB of L2 reads for 268 MB of activations, 7.6 TB/s together).  Here a block of eight
// waves owns (eight consecutive tiles, slice of columns): wave w takes tile w through all steps of 128 columns, and
// the weight block of a step (16 * NB x 128) is fetched once per block, 16 B per thread and piece, into a
// double-buffered LDS tile from which every wave reads its MFMA operands.  One LDS-only barrier per step: a buffer is
// overwritten one step after the barrier behind its last reader.  The eight tiles are taken in runs of equal group
// (almost always one run); waves whose tile lies outside the run still help to stage the weights.  What bounds it is
// memory latency: a wave keeps S - 1 steps (8 KB each: 256 contiguous bytes of 32 rows) in flight and the weights are
// requested two steps ahead.  (k_shrink_quad in kernels_mfma.hip is the same with four waves of two tiles and 64 columns a
// step: see oct_blocks for which is faster where.)  Every block leaves its sums as one slice of the split-shrink buffer
// (k_shrink_finish follows); each entry is the sum of one wave's MFMA chain in column order, in either kernel, so results
// do not depend on timing or on the choice.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void shrink_oct_body(const PassArgs& a, const int32_t* __restrict__ tile_group,
                                                const int32_t* __restrict__ slot_rows, int max_tiles, int item) {
  constexpr int RP = 16 * NB;
  constexpr int WS = 136;             // row stride of a staged weight block in bf16 (272 B: conflict-free)
  constexpr int NLD = RP * 16 / 512;  // 16-byte pieces of a weight block per thread
  constexpr int S = NB >= 4 ? 2 : 4;  // steps of activations in registers (three at rank 64: 0.4 % slower on 32768 rows)
  constexpr int WD = 2;               // steps the weights are requested ahead
  static_assert(NB >= 2 && S % WD == 0, "the loop's unrolling names the weight registers");
  __shared__ __attribute__((aligned(16))) bf16_t wbuf[2][RP * WS];
  __shared__ int32_t gts[8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int nth = item / a.kslices, ks = item - nth * a.kslices;
  const int set = work_item(a.wl_octs, nth);
  if (set < 0) return;  // past the end of this rank class's list (uniform over the block)
  const int t_first = set * 8;
  if (tid < 8) gts[tid] = t_first + tid < max_tiles ? checked_group(tile_group[t_first + tid], a.tb) : -1;
  const int s0 = ks * a.set_steps;                                 // in 64-column steps
  const int n64 = min(a.set_steps, (a.width_src >> 6) - s0);       // >= 1 for every slice
  const int ns = (n64 + 1) >> 1;                                   // steps of 128 columns, the last perhaps half
  // this wave's tile
  const bf16_t* x_row[2];
  {
    const int t = min(t_first + wave, max_tiles - 1);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const int row = min(max(slot_rows[t * kTileRows + 16 * tt + li], 0), a.src_rows - 1);
      x_row[tt] = (const bf16_t*)a.src + (int64_t)row * a.ld_src + 16 * kb + (int64_t)s0 * 64;
    }
  }
  __syncthreads();
  for (int j = 0; j < 8;) {
    const int g = gts[j];
    int e = j + 1;
    while (e < 8 && gts[e] == g) ++e;
    const int lo = j, hi = e;  // the run: tiles t_first + lo .. t_first + hi - 1, all of group g
    j = e;
    if (g < 0) continue;
    const int r = class_rank(a.rank[g], a.rank_lo, RP);
    if (r <= 0) continue;  // adapter not live on this layer, or a group of another rank class
    const bool active = wave >= lo && wave < hi;  // wave-uniform
    const bf16_t* W1 = group_weight<bf16_t>(a.w_shrink, a.w_shrink_base, a.shrink_group_stride, g) + (int64_t)s0 * 64;
    // staging: piece p = tid + 512 i is columns 8 (p % 16) .. + 8 of rank index p / 16
    auto stage_load = [&](int s, uint4 (&wr)[NLD]) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int p = tid + 512 * i, n = p >> 4, c = (s << 7) + 8 * (p & 15);
        wr[i] = (n < r && c < (n64 << 6)) ? ld16(W1 + (int64_t)n * a.ld_shrink + c) : zero4();
      }
    };
    auto stage_store = [&](int buf, const uint4 (&wr)[NLD]) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int p = tid + 512 * i;
        st16(&wbuf[buf][(p >> 4) * WS + 8 * (p & 15)], wr[i]);
      }
    };
    struct Step {
      uint4 x[2][2][2];  // [half of 64 columns][piece][16 rows]
    };
    auto issue = [&](int s, Step& X) {
      // (steps past the slice repeat its last one, a half past its end the half in front: requested and not used)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const int c = min(2 * s + hf, n64 - 1) << 6;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int p = 0; p < 2; ++p) X.x[hf][p][tt] = ld16(x_row[tt] + c + 8 * p);
      }
    };
    f32x4 acc[2][NB];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 wr[WD][NLD];
    // (w_cur: the weights of step s + 1, w_next: where those of step s + WD go)
    auto step = [&](int s, const Step& X, Step& Xnext, const uint4 (&w_cur)[NLD], uint4 (&w_next)[NLD]) {
      lds_barrier();  // block s is complete; the other buffer has been read by everyone
      stage_load(s + WD, w_next);
      if (active) {
        issue(s + S - 1, Xnext);
        const bf16_t* wb = wbuf[s & 1] + li * WS + 16 * kb;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          if (hf && 2 * s + 1 >= n64) break;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              const uint4 w = ld16(wb + 16 * nb * WS + 64 * hf + 8 * p);
#pragma unroll
              for (int tt = 0; tt < 2; ++tt) acc[tt][nb] = mfma16(X.x[hf][p][tt], w, acc[tt][nb]);
            }
          __builtin_amdgcn_sched_barrier(0);  // (reading the weights further ahead costs registers: spills)
        }
      }
      stage_store((s + 1) & 1, w_cur);  // block s + 1 (zeros past the slice), visible behind the next barrier
    };
    Step T[S];
    stage_load(0, wr[0]);
    stage_load(1, wr[1]);
    if (active) {
#pragma unroll
      for (int i = 0; i < S - 1; ++i) issue(i, T[i]);
    }
    stage_store(0, wr[0]);
    int s = 0;
    for (; s + S <= ns; s += S) {
#pragma unroll
      for (int i = 0; i < S; ++i) step(s + i, T[i], T[(i + S - 1) % S], wr[(i + 1) % WD], wr[i % WD]);
    }
#pragma unroll
    for (int i = 0; i < S - 1; ++i)
      if (s + i < ns) step(s + i, T[i], T[(i + S - 1) % S], wr[(i + 1) % WD], wr[i % WD]);  // block-uniform
    lds_barrier();  // the next run's first block goes into buffer 0
    if (!active) continue;
    float* out = a.hpart + ((int64_t)(t_first + wave) * a.kslices + ks) * (kTileRows * RP) + 4 * kb * RP + li;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v) out[(16 * tt + v) * RP + 16 * nb] = acc[tt][nb][v];
  }
}

template <int NB>
__global__ __launch_bounds__(512) void k_shrink_oct(PassArgs a, const int32_t* __restrict__ tile_group,
                                                    const int32_t* __restrict__ slot_rows, int max_tiles) {
  shrink_oct_body<NB>(a, tile_group, slot_rows, max_tiles, blockIdx.x);
}

// ---------------------------------------------------------------------------
// The same work as k_shrink_oct, item by item and sum by sum, with the operands going from memory straight into LDS: no
// registers hold loads in flight, so three stages of 64 columns (x 32 KB, weights RP x 128 B) are on their way per CU where
// the registers held one or two steps, which is what the time of a step was.  A wave's tile goes through a window of its own
// (no barrier for it), the weights are shared: one barrier a step, behind a wait for the wave's loads of that step; the
// stage read before it takes the loads two steps ahead.  Rows of 128 B, 16-byte chunk c of row r at position c ^ (r & 7): a
// load covers whole lines, an operand read eight different bank groups.
// Source under 4 GB (32-bit row offsets); the weights of a matrix that is not 16-byte aligned go through registers.
// Shrink with its slice sums, eight adapters, oct or quad / here, us: rank 128 8192 x 4096 49.6 / 39.3, 32768 x 4096 126 /
// 104; rank 64 8192 x 4096 32.6 / 28.2, 32768 x 4096 86 / 76; rank 32 8192 x 4096 28.7 / 23.6, 2048 x 1024 20.1 / 14.1: faster
// at every size from 2048 x 1024 to 32768 x 4096, rows packed or shuffled.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void shrink_dl_body(const PassArgs& a, const int32_t* __restrict__ tile_group,
                                               const int32_t* __restrict__ slot_rows, int max_tiles, int item) {
  constexpr int RP = 16 * NB, NW = NB > 4 ? NB / 4 : 1;  // NW: weight loads of a wave per step (8 rank indices each)
  __shared__ __attribute__((aligned(1024))) bf16_t X0[256 * 64], X1[256 * 64], X2[256 * 64];
  __shared__ __attribute__((aligned(1024))) bf16_t W0[RP * 64], W1[RP * 64], W2[RP * 64];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nth = item / a.kslices, ks = item - nth * a.kslices;
  const int set = work_item(a.wl_octs, nth);
  if (set < 0) return;  // past the end of this rank class's list (uniform over the block)
  const int t_first = set * 8;
  const int my_tile = t_first + (lane & 7);
  const int gts = my_tile < max_tiles ? checked_group(tile_group[my_tile], a.tb) : -1;  // lane j: group of tile j
  const int s0 = ks * a.set_steps;
  const int ns = min(a.set_steps, (a.width_src >> 6) - s0);  // >= 1 for every slice
  const int lrow = lane >> 3, chunk = (lane & 7) ^ lrow;
  uint32_t xoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = min(t_first + wave, max_tiles - 1);
    const int row = min(max(slot_rows[t * kTileRows + 8 * i + lrow], 0), a.src_rows - 1);
    xoff[i] = (uint32_t)row * (uint32_t)(a.ld_src * 2) + (uint32_t)(s0 * 128 + chunk * 16);
  }
  const int64_t xbytes = ((int64_t)(a.src_rows - 1) * a.ld_src + a.width_src) * 2;
  const uint32_t rd = (uint32_t)((2 * kb) ^ (li & 7)) * 16u;  // this lane's chunk 2 kb of a row; chunk 2 kb + 1: ^ 16
  for (int j = 0; j < 8;) {
    const int g = __builtin_amdgcn_readlane(gts, j);
    int e = j + 1;
    while (e < 8 && __builtin_amdgcn_readlane(gts, e) == g) ++e;
    const int lo = j, hi = e;  // the run: tiles t_first + lo .. t_first + hi - 1, all of group g
    j = e;
    if (g < 0) continue;
    const int r = class_rank(a.rank[g], a.rank_lo, RP);
    if (r <= 0) continue;  // adapter not live on this layer, or a group of another rank class
    const bool active = wave >= lo && wave < hi;
    const bf16_t* W = group_weight<bf16_t>(a.w_shrink, a.w_shrink_base, a.shrink_group_stride, g) + (int64_t)s0 * 64;
    const bf16_t* wp[NW];
    uint32_t wlive[NW];
    int wrow[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      wrow[i] = 8 * (NB >= 4 ? wave + 8 * i : wave & (2 * NB - 1));  // (rank 32: two waves bring the same rows)
      const int n = wrow[i] + lrow;
      wlive[i] = n < r ? ~0u : 0u;
      wp[i] = n < r ? W + (int64_t)n * a.ld_shrink + 8 * chunk : reinterpret_cast<const bf16_t*>(kernel_zeros);
    }
    auto fetch_x = [&](int s, bf16_t* X) __attribute__((always_inline)) {
      const Buffer xbuf = buffer_of(a.src, active && s < ns ? xbytes : 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) buffer16_to_lds(xbuf, xoff[i], (uint32_t)s * 128u, X + (32 * wave + 8 * i) * 64);
    };
    auto fetch_w = [&](int s, bf16_t* Ws, auto direct) __attribute__((always_inline)) {
      const uint32_t at = (uint32_t)min(s, ns - 1) * 128u;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        if constexpr (decltype(direct)::value) {
          load16_to_lds(wp[i], at & wlive[i], Ws + wrow[i] * 64);
        } else {
          st16(Ws + wrow[i] * 64 + 8 * lane,
               ld16(reinterpret_cast<const bf16_t*>(reinterpret_cast<const char*>(wp[i]) + (at & wlive[i]))));
        }
      }
    };
    f32x4 acc[2][NB];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const bf16_t* X, const bf16_t* Ws) __attribute__((always_inline)) {
      const char* xr = reinterpret_cast<const char*>(X) + (32 * wave + li) * 128;
      const char* wr = reinterpret_cast<const char*>(Ws) + li * 128;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t at = rd ^ (16u * p);
        uint4 fx[2], fw[NB];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) fx[tt] = *reinterpret_cast<const uint4*>(xr + 2048 * tt + at);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) fw[nb] = *reinterpret_cast<const uint4*>(wr + 2048 * nb + at);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) acc[tt][nb] = mfma16(fw[nb], fx[tt], acc[tt][nb]);
      }
    };
    auto run = [&](auto direct) __attribute__((always_inline)) {
      fetch_x(0, X0);
      fetch_w(0, W0, direct);
      fetch_x(1, X1);
      fetch_w(1, W1, direct);
      auto step = [&](int s, const bf16_t* X, const bf16_t* Ws, bf16_t* Xn, bf16_t* Wn) __attribute__((always_inline)) {
        if constexpr (decltype(direct)::value) loads_landed_barrier<4 + NW>();
        else loads_landed_barrier<4>();  // (the younger step's weights have been waited for on their way)
        fetch_x(s + 2, Xn);
        fetch_w(s + 2, Wn, direct);
        if (active && s < ns) compute(X, Ws);
      };
      for (int s = 0; s < ns; s += 3) {
        step(s, X0, W0, X2, W2);
        step(s + 1, X1, W1, X0, W0);
        step(s + 2, X2, W2, X1, W1);
      }
    };
    if ((reinterpret_cast<uintptr_t>(W) & 15u) == 0) run(std::integral_constant<bool, true>{});
    else run(std::integral_constant<bool, false>{});
    if (active) {
      float* out = a.hpart + ((int64_t)(t_first + wave) * a.kslices + ks) * (kTileRows * RP) + li * RP + 4 * kb;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          *reinterpret_cast<float4*>(out + 16 * tt * RP + 16 * nb) =
              make_float4(acc[tt][nb][0], acc[tt][nb][1], acc[tt][nb][2], acc[tt][nb][3]);
    }
    loads_landed_barrier<0>();  // the stages are the next run's, or the next block's
  }
}

template <int NB>
__global__ __launch_bounds__(512) void k_shrink_dl(PassArgs a, const int32_t* __restrict__ tile_group,
                                                   const int32_t* __restrict__ slot_rows, int max_tiles) {
  shrink_dl_body<NB>(a, tile_group, slot_rows, max_tiles, blockIdx.x);
}

// whether k_shrink_dl runs: sources of 32-bit offsets, and see set_narrow
inline bool shrink_dl_applies(const PassArgs& a) { return !a.set_narrow && ((int64_t)a.src_rows * a.ld_src) * 2 < (1ll << 32); }

// Adds the slices of a split shrink in slice order and writes h (one block per tile).
template <int NB>
__device__ __forceinline__ void shrink_finish_body(const PassArgs& a, bf16_t* __restrict__ hrow,
                                                   const int32_t* __restrict__ tile_group,
                                                   const int32_t* __restrict__ slot_rows, int nth) {
  constexpr int RP = 16 * NB, PR = RP + 1;
  __shared__ float part[kTileRows][PR];
  const int tid = threadIdx.x;
  const int tile_id = checked_tile(work_item(a.wl_tiles, nth), a.tb);
  if (tile_id < 0) return;  // past the end of this rank class's list
  const int slot0 = tile_id * kTileRows;
  // independent loads first: group id, this tile's row indices, the slices themselves
  const int g = checked_group(tile_group[tile_id], a.tb);
  // (with several rank classes most tiles belong to another launch: look before reading their slices)
  if (a.class_mode && (g < 0 || class_rank(a.rank[g], a.rank_lo, RP) <= 0)) return;
  const int my_row = slot_rows[slot0 + (tid & 31)];
  const float* tile_part = a.hpart + (int64_t)tile_id * a.kslices * (kTileRows * RP);
  constexpr int NI = (kTileRows * RP + 255) / 256;
  float sums[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) sums[i] = 0.f;
  // eight slices are requested together (their latencies overlap) and added in slice order
  for (int k0 = 0; k0 < a.kslices; k0 += 8) {
    float v[NI][8];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int idx = tid + 256 * i;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[i][k] = (idx < kTileRows * RP && k0 + k < a.kslices) ? tile_part[(int64_t)(k0 + k) * (kTileRows * RP) + idx] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int k = 0; k < 8; ++k) sums[i] += v[i][k];
  }
  const int gg = max(g, 0);
  const int rk = class_rank(a.rank[gg], a.rank_lo, RP);
  const float sc = a.scale[gg];
  if (g < 0 || rk <= 0) return;
  const int cnt = __popcll(__ballot(my_row >= 0) & 0xffffffffull);  // padding is at the end of a tile
#pragma unroll
  for (int i = 0; i < (kTileRows * RP + 255) / 256; ++i) {
    const int idx = tid + 256 * i;
    if (idx < kTileRows * RP) part[idx / RP][idx % RP] = sums[i];
  }
  __syncthreads();
  shrink_epilogue<RP, 256>(&part[0][0], 1, a, hrow, slot0, cnt, sc);
}

// The same above rank 16: a block takes 32 of a tile's rank indices (blockIdx.y), a thread four of them of one slot, so that
// eight 16-byte loads are in flight per thread, there are RP / 32 blocks for a tile and h leaves in 8-byte pieces.
// Bound by the latency of those loads and their number per CU.  One block per tile with 4-byte loads before, us: rank 128,
// 8192 rows, 8 slices (33 MB) 11.5 -> 8.4; rank 64, 32768 rows 10.3 -> 9.2, 6000 rows 6.4 -> 5.0.
template <int NB>
__device__ __forceinline__ void shrink_finish_wide(const PassArgs& a, bf16_t* __restrict__ hrow,
                                                   const int32_t* __restrict__ tile_group,
                                                   const int32_t* __restrict__ slot_rows) {
  constexpr int RP = 16 * NB;
  __shared__ __attribute__((aligned(16))) bf16_t turn[32][kTileRows + 4];  // [rank index][slot]
  const int tile_id = checked_tile(work_item(a.wl_tiles, blockIdx.x), a.tb);
  if (tile_id < 0) return;
  const int slot0 = tile_id * kTileRows, n0 = 32 * blockIdx.y, tid = threadIdx.x;
  const int g = checked_group(tile_group[tile_id], a.tb);
  if (a.class_mode && (g < 0 || class_rank(a.rank[g], a.rank_lo, RP) <= 0)) return;
  const int my_row = slot_rows[slot0 + (tid & 31)];
  const int slot = tid >> 3, n = 4 * (tid & 7);
  const float* p = a.hpart + (int64_t)tile_id * a.kslices * (kTileRows * RP) + slot * RP + n0 + n;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < a.kslices; k0 += 8) {
    float4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v[k] = k0 + k < a.kslices ? *reinterpret_cast<const float4*>(p + (int64_t)(k0 + k) * (kTileRows * RP))
                                : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      sum[0] += v[k].x;
      sum[1] += v[k].y;
      sum[2] += v[k].z;
      sum[3] += v[k].w;
    }
  }
  const int gg = max(g, 0);
  const int rk = class_rank(a.rank[gg], a.rank_lo, RP);
  const float sc = a.scale[gg];
  if (g < 0 || rk <= 0) return;  // (uniform over the block, like the returns above)
  const int cnt = __popcll(__ballot(my_row >= 0) & 0xffffffffull);  // padding is at the end of a tile
  uint2 o = make_uint2(0u, 0u);
  if (slot < cnt) o = make_uint2(pack_bf16(sum[0] * sc, sum[1] * sc), pack_bf16(sum[2] * sc, sum[3] * sc));
  *reinterpret_cast<uint2*>(hrow + (int64_t)(slot0 + slot) * RP + n0 + n) = o;
  turn[n][slot] = (bf16_t)(o.x & 0xffffu);
  turn[n + 1][slot] = (bf16_t)(o.x >> 16);
  turn[n + 2][slot] = (bf16_t)(o.y & 0xffffu);
  turn[n + 3][slot] = (bf16_t)(o.y >> 16);
  __syncthreads();
  const int rn = tid >> 3, s4 = 4 * (tid & 7);
  *reinterpret_cast<uint2*>((bf16_t*)a.hT + (int64_t)(n0 + rn) * a.ldh + slot0 + s4) =
      *reinterpret_cast<const uint2*>(&turn[rn][s4]);
}

template <int NB>
__global__ __launch_bounds__(256) void k_shrink_finish(PassArgs a, bf16_t* __restrict__ hrow,
                                                       const int32_t* __restrict__ tile_group,
                                                       const int32_t* __restrict__ slot_rows) {
  if constexpr (NB == 1) shrink_finish_body<NB>(a, hrow, tile_group, slot_rows, blockIdx.x);
  else shrink_finish_wide<NB>(a, hrow, tile_group, slot_rows);
}

template <int NB>
inline dim3 shrink_finish_grid(const SegLayout& L) { return dim3((unsigned)L.max_tiles, (unsigned)std::max(NB / 2, 1)); }

// ---------------------------------------------------------------------------
// Expand: dst[row(slot)][c] += sum_n h[slot][n] * W2_g[c][n], read-modify-write
// in place.  Work is flat: one wave owns one 128-column group of one tile and
// nothing is shared between waves, so the grid is thousands of independent
// streams.  Column c0 + 8 j + q of a group is output column j of MFMA q, which
// makes each lane's 8 results of one row 16 contiguous bytes and each wave-wide
// access 4 rows x 256 B.  Row indices, h and the group id are addressed from the
// work-item number alone, so the destination loads are one dependent step away
// from the start of the wave.  (Used for padded rank 16; above that
// k_expand_multi shares the weight block between tiles.)
// ---------------------------------------------------------------------------
// FIN: the slices of a split shrink are added here, by every wave for its tile (NB = 1), and the wave of the first
// columns writes h: for launches of few tiles (see kFewFinishReads).  Same sums, same rounding as k_shrink_finish.
template <int NB, bool FIN = false>
__device__ __forceinline__ void expand_flat_body(const PassArgs& a, const bf16_t* __restrict__ hrow,
                                                 const int32_t* __restrict__ tile_group,
                                                 const int32_t* __restrict__ slot_rows,
                                                 const int32_t* __restrict__ tile_walk, int num_items, int block) {
  constexpr int RP = 16 * NB;
  constexpr int NKS = (RP + 31) / 32;  // contraction steps of the MFMAs
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int ngroups = a.width_dst >> 7;
  const int item = block * 4 + wave;
  if (item >= num_items) return;
  // Items are numbered tile by tile; with a walk order the n-th tile taken is tile_walk[n], the tiles sorted by their
  // first row.  The table itself is group-major and a group's tiles are spread over all rows, so in table order the
  // waves in flight at any moment touch rows all over the destination; in walk order they touch neighbouring rows,
  // and the in-place update runs faster (probe: 43 us against 54 us for 256 MB touched in tiles of 32 random rows
  // taken from windows of 512 rows instead of from all 16384).
  const int nth = item / ngroups;
  // (one of several rank classes: the class's own list of tiles, which is in the same walk order)
  const int tile_id = checked_tile(a.wl_tiles.ids ? work_item(a.wl_tiles, nth) : (tile_walk ? tile_walk[nth] : nth), a.tb);
  if (tile_id < 0) return;
  const int c0 = (item - nth * ngroups) << 7;
  const int slot0 = tile_id * kTileRows;
  // independent first loads: group id, row indices, h operand (nothing branches before the
  // destination loads are in flight)
  const int g_raw = checked_group(tile_group[tile_id], a.tb);
  // rows this lane updates: slots 16 tt + 4 kb + v
  const int4 r0 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 4 * kb);
  const int4 r1 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 16 + 4 * kb);
  uint4 hop[2][NKS];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int n0 = 32 * ks + 8 * kb;
      if constexpr (!FIN) hop[tt][ks] = n0 < RP ? ld16(hrow + (int64_t)(slot0 + 16 * tt + li) * RP + n0) : zero4();
    }
  const int g = max(g_raw, 0);
  if constexpr (FIN) {
    static_assert(NB == 1, "one operand step");
    const int r = g_raw < 0 ? 0 : class_rank(a.rank[g], a.rank_lo, RP);
    const float sc = a.scale[g];
    const bool first = item - nth * ngroups == 0;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const int slot = slot0 + 16 * tt + li;
      const bool real = kb < 2 && r > 0 && slot_rows[slot] >= 0;
      const float* p = a.hpart + (int64_t)tile_id * a.kslices * (kTileRows * RP) + (16 * tt + li) * RP + 8 * (kb & 1);
      float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int k0 = 0; k0 < a.kslices; k0 += 4) {  // four slices are requested together and added in slice order
        float4 v[4][2];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int q = 0; q < 2; ++q)
            v[k][q] = real && k0 + k < a.kslices
                          ? *reinterpret_cast<const float4*>(p + (int64_t)(k0 + k) * (kTileRows * RP) + 4 * q)
                          : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            sum[4 * q] += v[k][q].x;
            sum[4 * q + 1] += v[k][q].y;
            sum[4 * q + 2] += v[k][q].z;
            sum[4 * q + 3] += v[k][q].w;
          }
      }
      hop[tt][0] = real ? make_uint4(pack_bf16(sum[0] * sc, sum[1] * sc), pack_bf16(sum[2] * sc, sum[3] * sc),
                                     pack_bf16(sum[4] * sc, sum[5] * sc), pack_bf16(sum[6] * sc, sum[7] * sc))
                        : zero4();
      if (first && kb < 2 && r > 0) {
        st16(const_cast<bf16_t*>(hrow) + (int64_t)slot * RP + 8 * kb, hop[tt][0]);
        const uint32_t w[4] = {hop[tt][0].x, hop[tt][0].y, hop[tt][0].z, hop[tt][0].w};
#pragma unroll
        for (int i = 0; i < 8; ++i)
          ((bf16_t*)a.hT)[(int64_t)(8 * kb + i) * a.ldh + slot] = (bf16_t)(w[i >> 1] >> (16 * (i & 1)));
      }
    }
  }
  const int rows[2][4] = {{r0.x, r0.y, r0.z, r0.w}, {r1.x, r1.y, r1.z, r1.w}};
  bool rok[2][4];
  bf16_t* yp[2][4];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      rok[tt][v] = g_raw >= 0 && checked_row(rows[tt][v], a.tb) >= 0;
      yp[tt][v] = (bf16_t*)a.dst + (int64_t)(rok[tt][v] ? rows[tt][v] : 0) * a.ld_dst + 8 * li + c0;
    }
  const int r = g_raw < 0 ? 0 : class_rank(a.rank[g], a.rank_lo, RP);
  if (a.class_mode && r <= 0) return;  // a tile of another rank class: its rows are not even requested
  const bf16_t* W2 = group_weight<bf16_t>(a.w_expand, a.w_expand_base, a.expand_group_stride, g);
  uint4 y[2][4];
  uint4 bq[8][NKS];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int v = 0; v < 4; ++v) y[tt][v] = rok[tt][v] && !a.dst_store ? ld16_nt(yp[tt][v]) : zero4();
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int n0 = 32 * ks + 8 * kb;
      const int wrow = a.expand_swizzled ? c0 + 16 * q + li : c0 + 8 * li + q;
      bq[q][ks] = n0 < r ? keep_first(ld16(W2 + (int64_t)wrow * a.ld_expand + n0), r - n0) : zero4();
    }
  if (r <= 0) {  // unused tile, or adapter not live on this layer (uniform over the wave)
    if (a.dst_store && !a.class_mode) {  // (several classes: launch_zero_rows)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (checked_row(rows[tt][v], a.tb) >= 0)
            st16_nt((bf16_t*)a.dst + (int64_t)rows[tt][v] * a.ld_dst + 8 * li + c0, zero4());
    }
    return;
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    f32x4 d[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      d[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) d[q] = mfma16(hop[tt][ks], bq[q][ks], d[q]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (!rok[tt][v]) continue;
      const uint4 yy = y[tt][v];
      uint4 o;
      o.x = pack_bf16(bf16_lo(yy.x) + d[0][v], bf16_hi(yy.x) + d[1][v]);
      o.y = pack_bf16(bf16_lo(yy.y) + d[2][v], bf16_hi(yy.y) + d[3][v]);
      o.z = pack_bf16(bf16_lo(yy.z) + d[4][v], bf16_hi(yy.z) + d[5][v]);
      o.w = pack_bf16(bf16_lo(yy.w) + d[6][v], bf16_hi(yy.w) + d[7][v]);
      st16_nt(yp[tt][v], o);
    }
  }
}

template <int NB, bool FIN>
__global__ __launch_bounds__(256) void k_expand_mfma(PassArgs a, const bf16_t* __restrict__ hrow,
                                                     const int32_t* __restrict__ tile_group,
                                                     const int32_t* __restrict__ slot_rows,
                                                     const int32_t* __restrict__ tile_walk, int num_items) {
  expand_flat_body<NB, FIN>(a, hrow, tile_group, slot_rows, tile_walk, num_items, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Expand for padded ranks above 16.  There a wave's block of W2 (128 columns x rank) is as large as
// its piece of a 32-row tile (16 KB at rank 64), so re-reading it for every tile doubles the traffic
// between L2 and the CUs.  Here a wave keeps the block in registers and walks TPI consecutive tiles:
// work item = (TPI tiles, 128 columns).  Consecutive tiles almost always belong to the same group;
// where the group changes inside an item the wave reloads the block.  The next tile's rows, h operand
// and destination rows are requested before the current tile is consumed.
// ---------------------------------------------------------------------------
// CLS: the launch serves one of several rank classes (work list of sets, ranks outside the class skipped).  A
// compile-time switch because this kernel's schedule is touchy: with the two forms in one body the single-class
// launch measured 10 % slower (config 5's q projection: 116 against 106 us).
// STORE: dst_store, for the same reason.
template <int NB, int TPI, bool CLS, bool STORE>
__global__ __launch_bounds__(256) void k_expand_multi(PassArgs a, const bf16_t* __restrict__ hrow,
                                                      const int32_t* __restrict__ tile_group,
                                                      const int32_t* __restrict__ slot_rows,
                                                      const int32_t* __restrict__ set_walk,
                                                      const SegHeader* __restrict__ header,
                                                      const uint8_t* __restrict__ round_moved, int sort_blocks,
                                                      int max_tiles) {
  static_assert(TPI == kSetTiles, "the segment table's set order is built for sets of kSetTiles tiles");
  constexpr int RP = 16 * NB;
  constexpr int NKS = (RP + 31) / 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int ngroups = a.width_dst >> 7;
  const int nbt = (ngroups + 3) >> 2;  // blocks per tile set: column block fastest
  // Gathered rows whose groups interleave: the sets of tiles in the order of their first row, so that neighbouring
  // rows are in flight together (measured at config 3: 2.5 % of the step).  Rows in segment order, or a table built
  // from keys that came in order (then that order is the identity): contiguous runs of sets per XCD, whose L2 then
  // fetches the weights of few groups (1.2 % at config 5's q projection; combining the two loses the first gain).
  // Whether the keys came in order is in the builder's flags, one byte per 64 rows, eight per lane here.
  // (the flags and the order entry are requested together: one round trip in front of the tile's first loads)
  int swept_set = 0;
  bool sweep = false;
  if constexpr (CLS) {
    // the class's list of sets, already in the order to take them in
    swept_set = work_item(a.wl_sets, blockIdx.x / nbt);
    if (swept_set < 0) return;
    sweep = true;
  } else if (set_walk != nullptr) {
    swept_set = set_walk[blockIdx.x / nbt];
    uint2 moved = make_uint2(0u, 0u);
    if (lane < sort_blocks) moved = reinterpret_cast<const uint2*>(round_moved)[lane];
    sweep = header->identity_order == 0 && __ballot((moved.x | moved.y) != 0u) != 0ull;
  }
  const int block = sweep ? (int)blockIdx.x : TK_XCD_MAP(blockIdx.x, gridDim.x);
  const int cb = block % nbt, set = block / nbt;
  const int tile0 = (sweep ? swept_set : set) * TPI;
  const int cg = cb * 4 + wave;
  if ((unsigned)tile0 >= (unsigned)max_tiles) return;  // (uniform over the block)
  const int nt = min(TPI, max_tiles - tile0);
  int gt[TPI];
#pragma unroll
  for (int t = 0; t < TPI; ++t) gt[t] = t < nt ? checked_group(tile_group[tile0 + t], a.tb) : -1;
#if TK_EXPAND_LDS_H
  // The block's four waves multiply the same tiles' h operands with their own columns' weights: the operands (one
  // contiguous run of hrow, nt x 32 slots x RP) are fetched once per block into LDS instead of once per wave.  Row
  // stride RP + 8 elements: operand reads without bank conflicts.
  constexpr int HS = RP + 8;
  __shared__ __attribute__((aligned(16))) bf16_t h_s[TPI * kTileRows * HS];
  {
    constexpr int PPR = RP / 8, PIECES = TPI * kTileRows * PPR, PER = (PIECES + 255) / 256;
    const bf16_t* hp = hrow + (int64_t)tile0 * kTileRows * RP;
    uint4 v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 256 * i;
      v[i] = e < nt * kTileRows * PPR ? ld16(hp + 8 * e) : zero4();
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 256 * i;
      if (e < PIECES) st16(&h_s[(e / PPR) * HS + 8 * (e % PPR)], v[i]);
    }
  }
  __syncthreads();
#endif
  if (cg >= ngroups) return;  // a column group past the width
  const int c0 = cg << 7;
  bf16_t* dst = (bf16_t*)a.dst + c0 + 8 * li;

  struct Tile {
    int rows[2][4];
#if !TK_EXPAND_LDS_H
    uint4 hop[2][NKS];
#endif
    uint4 y[2][4];
    int t;
  };
  auto issue = [&](int t, Tile& T) {
    const bool tok = t < nt;  // wave-uniform
    const unsigned row_limit = tok ? (unsigned)a.tb.rows : 0u;  // rows of the table are in [0, rows): see TableBounds
    const int slot0 = (tile0 + (tok ? t : 0)) * kTileRows;
    const int4 r0 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 4 * kb);
    const int4 r1 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 16 + 4 * kb);
    const int rr[2][4] = {{r0.x, r0.y, r0.z, r0.w}, {r1.x, r1.y, r1.z, r1.w}};
    T.t = tok ? t : 0;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#if !TK_EXPAND_LDS_H
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int n0 = 32 * ks + 8 * kb;
        T.hop[tt][ks] = (tok && n0 < RP) ? ld16(hrow + (int64_t)(slot0 + 16 * tt + li) * RP + n0) : zero4();
      }
#endif
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        T.rows[tt][v] = (unsigned)rr[tt][v] < row_limit ? rr[tt][v] : -1;
        T.y[tt][v] = T.rows[tt][v] >= 0 && !STORE ? ld16_nt(dst + (int64_t)T.rows[tt][v] * a.ld_dst) : zero4();
      }
    }
  };
  uint4 bq[8][NKS];
  int r = 0;
  // Above rank 64 adapters may lie at any element address: a piece that the rank cuts may then reach past the matrix's
  // last row, behind which there need be nothing to read, so the rows q = 7 are read element by element.  (Copies inside
  // a workspace, the only weights of the writing form, are aligned: there a piece ends where an aligned 16 bytes end.)
  auto load_cut_weights = [&](const bf16_t* W2) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int n0 = 32 * ks + 8 * kb;
      const bf16_t* p = W2 + (int64_t)(c0 + 8 * li) * a.ld_expand + n0;
#pragma unroll
      for (int q = 0; q < 7; ++q) bq[q][ks] = n0 < r ? keep_first(ld16(p + q * a.ld_expand), r - n0) : zero4();
      uint64_t lo = 0, hi = 0;
#pragma unroll 1
      for (int i = min(r - n0, 8) - 1; i >= 0; --i) {
        hi = (hi << 16) | (lo >> 48);
        lo = (lo << 16) | p[7 * a.ld_expand + i];
      }
      bq[7][ks] = make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
    }
  };
  auto load_weights = [&](int g) {  // this wave's block of W2 for group g
    r = CLS ? class_rank(a.rank[g], a.rank_lo, RP) : min(a.rank[g], RP);
    const bf16_t* W2 = group_weight<bf16_t>(a.w_expand, a.w_expand_base, a.expand_group_stride, g);
    if constexpr (NB == 8 && !STORE) {
      if ((r & 7) && (reinterpret_cast<uintptr_t>(W2) & 15u) && c0 + 128 == a.width_dst) {  // (uniform over the wave)
        load_cut_weights(W2);
        return;
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int n0 = 32 * ks + 8 * kb;
        bq[q][ks] = n0 < r ? keep_first(ld16(W2 + (int64_t)(c0 + 8 * li + q) * a.ld_expand + n0), r - n0) : zero4();
      }
  };
  auto consume = [&](const Tile& T) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#if TK_EXPAND_LDS_H
      uint4 hop[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        hop[ks] = 32 * ks + 8 * kb < RP ? ld16(h_s + (T.t * kTileRows + 16 * tt + li) * HS + 32 * ks + 8 * kb) : zero4();
#endif
      f32x4 d[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        d[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#if TK_EXPAND_LDS_H
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) d[q] = mfma16(hop[ks], bq[q][ks], d[q]);
#else
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) d[q] = mfma16(T.hop[tt][ks], bq[q][ks], d[q]);
#endif
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (T.rows[tt][v] < 0) continue;
        const uint4 yy = T.y[tt][v];
        uint4 o;
        o.x = pack_bf16(bf16_lo(yy.x) + d[0][v], bf16_hi(yy.x) + d[1][v]);
        o.y = pack_bf16(bf16_lo(yy.y) + d[2][v], bf16_hi(yy.y) + d[3][v]);
        o.z = pack_bf16(bf16_lo(yy.z) + d[4][v], bf16_hi(yy.z) + d[5][v]);
        o.w = pack_bf16(bf16_lo(yy.w) + d[6][v], bf16_hi(yy.w) + d[7][v]);
        st16_nt(dst + (int64_t)T.rows[tt][v] * a.ld_dst, o);
      }
    }
  };
  // the rows of a tile that has no live group (one class: nobody else writes them)
  auto zero_tile = [&](int t) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = checked_row(slot_rows[(tile0 + t) * kTileRows + 8 * kb + i], a.tb);
      if (row >= 0) st16_nt(dst + (int64_t)row * a.ld_dst, zero4());
    }
  };
  if constexpr (STORE && !CLS) {
#pragma unroll
    for (int t = 0; t < TPI; ++t)
      if (t < nt && gt[t] < 0) zero_tile(t);
  }
  // tiles past the last one of the table carry -1 and come last
  bool uniform = true;
#pragma unroll
  for (int t = 1; t < TPI; ++t) uniform = uniform && (gt[t] == gt[0] || gt[t] < 0);
  Tile A, B;
  if (uniform) {  // the usual case: one group, one block of W2, loads pipelined over the tiles
    if (gt[0] < 0) return;
    int nv = 0;
#pragma unroll
    for (int t = 0; t < TPI; ++t) nv += gt[t] >= 0;
    load_weights(gt[0]);
    if (r <= 0) {  // adapter not live on this layer
      if constexpr (STORE && !CLS)
        for (int t = 0; t < nv; ++t) zero_tile(t);
      return;
    }
    issue(0, A);
    for (int t = 0; t < nv; t += 2) {
      issue(t + 1 < nv ? t + 1 : nt, B);
      consume(A);
      if (t + 1 < nv) {
        issue(t + 2 < nv ? t + 2 : nt, A);
        consume(B);
      }
    }
    return;
  }
  for (int t = 0; t < nt; ++t) {  // a group boundary inside the item: tile by tile
    if (gt[t] < 0) continue;
    load_weights(gt[t]);
    if (r <= 0) {
      if constexpr (STORE && !CLS) zero_tile(t);
      continue;
    }
    issue(t, A);
    consume(A);
  }
}

// 8 x 8 block of bf16 transposed inside a lane: in[i] holds 8 consecutive elements of row i, out[q] the 8 rows'
// q-th elements (v_perm_b32 picks the low or the high halves of a register pair).
__device__ inline void transpose8x8(const uint4 (&in)[8], uint4 (&out)[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int d = q >> 1;
    const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w[4] = {in[i].x, in[i].y, in[i].z, in[i].w};
      e[i] = w[d];
    }
    out[q].x = __builtin_amdgcn_perm(e[1], e[0], sel);
    out[q].y = __builtin_amdgcn_perm(e[3], e[2], sel);
    out[q].z = __builtin_amdgcn_perm(e[5], e[4], sel);
    out[q].w = __builtin_amdgcn_perm(e[7], e[6], sel);
  }
}

// Eight consecutive weights as bf16, from a bf16 or an fp32 matrix (element index e, a multiple of 8 for the
// vector form; fp32 is rounded to nearest even).
__device__ inline uint4 load8_weights(const void* base, int64_t e, bool f32) {
  if (!f32) return ld16((const bf16_t*)base + e);
  const float4 lo = *reinterpret_cast<const float4*>((const float*)base + e);
  const float4 hi = *reinterpret_cast<const float4*>((const float*)base + e + 4);
  return make_uint4(pack_bf16(lo.x, lo.y), pack_bf16(lo.z, lo.w), pack_bf16(hi.x, hi.y), pack_bf16(hi.z, hi.w));
}
__device__ inline uint32_t load_weight(const void* base, int64_t e, bool f32) {
  return f32 ? (pack_bf16(((const float*)base)[e], 0.f) & 0xffffu) : (uint32_t)((const bf16_t*)base)[e];
}

// Transposed weight copies (see TransposeJob).  A work unit is an 8 x 8 block: eight 16-byte loads along the
// source's contiguous dimension, a transpose inside the lane, eight 16-byte stores along the copy's contiguous
// dimension; consecutive threads take neighbouring blocks so that a wave's accesses cover whole rows (128 bytes and
// more).  A source whose row stride or address rules out 16-byte loads is gathered element by element.
__device__ inline void transpose_weights_job(const TransposeJob& t, const int32_t* __restrict__ rank, int rpad,
                                             int64_t thread, int64_t threads) {
  const int m8 = t.out_features >> 3, n8 = rpad >> 3, k8 = t.in_features >> 3;
  const int64_t units_b = t.bT ? (int64_t)t.groups * m8 * n8 : 0;  // (g, m-octet, n-octet), n-octet fastest
  const int64_t units_a = (int64_t)t.groups * n8 * k8;              // (g, k-octet, n-octet), n-octet fastest
  const bool f32 = t.src_f32 != 0;
  const int ld_mask = f32 ? 3 : 7;  // row strides that keep every row 16-byte aligned
  for (int64_t u = thread; u < units_b + units_a; u += threads) {
    uint4 in[8], out[8];
    if (u < units_b) {
      // bT[g][n][m] = B_g[m][n]: rows m of B hold the rank index contiguously
      const int no = (int)(u % n8);
      const int64_t q = u / n8;
      const int mo = (int)(q % m8), g = (int)(q / m8);
      const int r = class_rank(rank[g], t.rank_lo, rpad);
      if (8 * no >= r && t.skip_dead) continue;
      const void* B = t.lora_B[g];
      const int64_t b0 = (int64_t)(8 * mo) * t.ldb + 8 * no;
      const bool vec = (t.ldb & ld_mask) == 0 && 8 * no + 8 <= t.ldb && (reinterpret_cast<uintptr_t>(B) & 15u) == 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (8 * no >= r) {
          in[i] = zero4();
        } else if (vec) {
          in[i] = keep_first(load8_weights(B, b0 + (int64_t)i * t.ldb, f32), r - 8 * no);
        } else {
          uint32_t e[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) e[j] = 8 * no + j < r ? load_weight(B, b0 + (int64_t)i * t.ldb + j, f32) : 0;
          in[i] = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
        }
      }
      transpose8x8(in, out);
      bf16_t* o = (bf16_t*)t.bT + ((int64_t)g * rpad + 8 * no) * t.out_features + 8 * mo;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (8 * no + j < r || !t.skip_dead) st16(o + (int64_t)j * t.out_features, out[j]);
    } else {
      // aT[g][k][n] = A_g[n][k]: rows n of A hold the input features contiguously
      // rank octet fastest: the threads that hold the octets of one column of A are neighbours, so a wave-wide
      // store covers whole rows of the copy (a row is rpad elements), and a wave-wide load still covers 128-byte
      // runs of A's rows (eight neighbouring column octets per rank octet)
      const int64_t v = u - units_b;
      const int no = (int)(v % n8);
      const int64_t q = v / n8;
      const int ko = (int)(q % k8), g = (int)(q / k8);
      const int r = class_rank(rank[g], t.rank_lo, rpad);
      if (8 * no >= r && t.skip_dead) continue;
      const void* A = t.lora_A[g];
      const int64_t a0 = (int64_t)(8 * no) * t.lda + 8 * ko;
      const bool vec = (t.lda & ld_mask) == 0 && (reinterpret_cast<uintptr_t>(A) & 15u) == 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (8 * no + i >= r) {
          in[i] = zero4();
        } else if (vec) {
          in[i] = load8_weights(A, a0 + (int64_t)i * t.lda, f32);
        } else {
          uint32_t e[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) e[j] = load_weight(A, a0 + (int64_t)i * t.lda + j, f32);
          in[i] = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
        }
      }
      transpose8x8(in, out);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = 8 * ko + j;  // column of A; which row of aT holds it:
        const int kd = t.swizzle_a ? ((k & ~127) | ((k & 7) << 4) | ((k >> 3) & 15)) : k;
        st16((bf16_t*)t.aT + ((int64_t)g * t.in_features + kd) * rpad + 8 * no, out[j]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Weight gradient: out_g[n][c] = sum over the rows of group g of hT[n][slot] * src[row(slot)][c].
//
// Work item = (chunk of one group, 128 source columns), one wave.  The wave walks all tiles of
// the chunk with an S-stage software pipeline: the source rows of tile t+S-1 are requested before tile t
// is consumed, so a wave has S-1 tiles (8 KB each) in flight; the chunk's row indices wait in LDS, where
// reading them does not have to wait for the tile loads in flight.  A grid of (chunks x 128-column
// blocks) is small next to the chip, so the depth of the pipeline, not the number of resident waves, is
// what keeps enough bytes in flight.  A lane loads 16 B of eight rows, transposes the 8x8 block in registers
// (v_perm_b32) and feeds it as the MFMA A operand with the rows as contraction index.  The result is
// staged in LDS in [n][column] order and leaves as whole 512-byte rows: into the chunk's slot of the
// partial buffer (groups that span several chunks; k_wgrad_reduce adds the chunks in order) or straight
// into the gradient (single-chunk groups).  No atomics: the result is bitwise repeatable.
//
// This one-wave form serves padded rank 16; above it two waves share the tiles (k_wgrad_coop below).
// ---------------------------------------------------------------------------
template <int NB, int S>
__global__ __launch_bounds__(64) void k_wgrad_pipe(WgradArgs a, const ChunkInfo* __restrict__ chunks,
                                                        const int32_t* __restrict__ slot_rows) {
  constexpr int OS = kWgradStageStride;
  __shared__ __attribute__((aligned(16))) float lds[16 * NB * OS];
  extern __shared__ __attribute__((aligned(16))) int32_t rows_s[];  // the chunk's row indices
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  if ((int)blockIdx.y < a.tr.y_blocks) {  // side job: the first rows of the grid transpose the adapter weights
    transpose_weights_job(a.tr, a.rank, a.rpad, ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 64 + tid,
                          (int64_t)a.tr.y_blocks * gridDim.x * 64);
    return;
  }
  // column block fastest: blocks that run together read neighbouring pieces of the same rows
  const int c0 = blockIdx.x * 128;
  const int cidx = work_item(a.wl_chunks, blockIdx.y - a.tr.y_blocks);
  if (cidx < 0) return;  // past the end of this rank class's list
  const ChunkInfo ci = checked_chunk(chunks[cidx], a.tb);
  const int g = ci.group;
  if (g < 0) return;
  const int r = class_rank(a.rank[g], a.rank_lo, 16 * NB);
  if (r <= 0) return;
  const int nt = ci.ntiles;
  for (int i = tid; i < nt * kTileRows; i += 64) rows_s[i] = slot_rows[ci.tile0 * kTileRows + i];
  __syncthreads();

  const bf16_t* src = (const bf16_t*)a.src + c0 + 8 * li;
  const bf16_t* hT = (const bf16_t*)a.hT + (int64_t)li * a.ldh + (int64_t)ci.tile0 * kTileRows + 8 * kb;
  f32x4 acc[8][NB];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[q][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The loop body below is straight-line code: every load is unconditional (tiles past the end re-read the
  // last tile, padding slots read row 0) and what must not count is zeroed when it is consumed.  With no
  // branch between a load and its use the compiler can wait for exactly the loads it needs and leave the
  // younger ones in flight.
  struct Tile {
    uint4 x[8];
    uint4 h[NB];
    uint32_t live;  // bit q: row q of this lane is a real row of a tile inside the chunk
  };
  auto issue = [&](int t, Tile& T) {
    const int tc = min(t, nt - 1);
    const int4 ra = *reinterpret_cast<const int4*>(rows_s + tc * kTileRows + 8 * kb);
    const int4 rb = *reinterpret_cast<const int4*>(rows_s + tc * kTileRows + 8 * kb + 4);
    const int rows[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
    T.live = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int row = checked_row(rows[q], a.tb);
      T.x[q] = ld16(src + (int64_t)max(row, 0) * a.ld_src);
      T.live |= (t < nt && row >= 0) ? (1u << q) : 0u;
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) T.h[nb] = ld16(hT + (int64_t)(16 * nb) * a.ldh + tc * kTileRows);
  };
  auto consume = [&](const Tile& T) {
    // 8x8 transpose inside the lane: tr holds column q of the 8 rows
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int d = q >> 1;
      const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
      uint32_t e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t wsrc[4] = {T.x[i].x, T.x[i].y, T.x[i].z, T.x[i].w};
        e[i] = (T.live >> i) & 1u ? wsrc[d] : 0u;
      }
      uint4 tr;
      tr.x = __builtin_amdgcn_perm(e[1], e[0], sel);
      tr.y = __builtin_amdgcn_perm(e[3], e[2], sel);
      tr.z = __builtin_amdgcn_perm(e[5], e[4], sel);
      tr.w = __builtin_amdgcn_perm(e[7], e[6], sel);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[q][nb] = mfma16(tr, T.h[nb], acc[q][nb]);
    }
  };
  Tile T[S];
#pragma unroll
  for (int i = 0; i < S - 1; ++i) issue(i, T[i]);
  int t = 0;
  for (; t + S <= nt; t += S) {  // every tile consumed in here exists (the youngest requests may lie past the end)
#pragma unroll
    for (int i = 0; i < S; ++i) {
      issue(t + i + S - 1, T[(i + S - 1) % S]);
      consume(T[i]);
    }
  }
  // drain: fewer than S tiles are left, all requested already (tiles past the end count as zeros)
#pragma unroll
  for (int i = 0; i < S - 1; ++i) consume(T[i]);
  wgrad_store<NB>(acc, lds, a, ci, g, r, c0, lane);
}

// ---------------------------------------------------------------------------
// Weight gradient above rank 16: (chunk, 128 columns), two waves (four at padded rank 128), each owning half of the rank
// indices and both needing every tile of the source (one wave with all of them would hold 64 or 128
// accumulator registers next to its tiles in flight: measured 49 against 41 us at rank 32, one wave per SIMD
// at rank 64).  Two independent readers of a tile drift apart and the later one misses the CU's cache
// (measured at rank 64: 1.66 x the source bytes fetched from memory), so here the tile crosses the
// memory system once: each wave requests half of it (4 of the 8 rows of every lane's 8 x 8 block), S - 1
// tiles ahead, the halves meet in a double-buffered LDS tile behind an LDS-only barrier (global loads stay
// in flight), and every wave reads the whole tile back in the operand layout.  Padding rows are zeroed when
// they are written to LDS.  One barrier per tile: a wave overwrites a buffer two tiles later, after the
// barrier that every reader of it has passed.
// ---------------------------------------------------------------------------
// PAIRS: pairs of waves per block (1 or 2).  Two pairs take neighbouring column blocks of the same chunk: they load
// the same h operands at about the same time, so the second pair's come from the CU's cache instead of from L2
// (every 128-column block of a chunk re-reads the chunk's h: a third of this kernel's L2 reads at rank 64).
// NB = 8 (rank 128): four waves share a tile, each with a quarter of the rank indices and of the tile's rows, so that the
// accumulators stay at 64 registers per wave; the result is staged 16 rank indices at a time.
template <int NB, int S, int PAIRS = 1>
__device__ __forceinline__ void wgrad_coop_body(const WgradArgs& a, const ChunkInfo* __restrict__ chunks,
                                                const int32_t* __restrict__ slot_rows, int bx, int by, int nx) {
  constexpr int RS = NB == 8 ? 4 : 2, NBW = NB / RS, PR = 8 / RS;  // waves per tile, rank blocks and rows of each
  constexpr int NBS = NB == 8 ? 1 : NBW;  // rank blocks a wave stages together
  constexpr int OS = kWgradStageStride;
  constexpr int XS = 136;  // row stride of a staged tile in bf16 (272 B)
  // the tile buffers are dead when the result is staged: one array serves both
  constexpr int kLdsFloats = 16 * RS * NBS * OS > kTileRows * XS ? 16 * RS * NBS * OS : kTileRows * XS;  // >= two staged bf16 tiles
  __shared__ __attribute__((aligned(16))) float lds_all[PAIRS * kLdsFloats];
  float* const lds = lds_all + (PAIRS > 1 ? (threadIdx.x >> 7) * kLdsFloats : 0);
  extern __shared__ __attribute__((aligned(16))) int32_t rows_s[];  // the chunk's row indices (same for both pairs)
  static_assert(PAIRS == 1 || RS == 2, "");
  const int tid = threadIdx.x & (64 * RS - 1), lane = tid & 63, li = lane & 15, kb = lane >> 4, rs = tid >> 6;
  if (by < a.tr.y_blocks) {  // side job: the first rows of the grid transpose the adapter weights
    transpose_weights_job(a.tr, a.rank, a.rpad, ((int64_t)by * nx + bx) * (RS * 64) + tid,
                          (int64_t)a.tr.y_blocks * nx * (RS * 64));
    return;
  }
  const int c0 = bx * 128;
  const int cidx = work_item(a.wl_chunks, by - a.tr.y_blocks);
  if (cidx < 0) return;  // past the end of this rank class's list
  const ChunkInfo ci = checked_chunk(chunks[cidx], a.tb);
  const int g = ci.group;
  if (g < 0) return;
  int nt = ci.ntiles;
  if (a.pair_chunks) {  // (the neighbours' entries do not depend on ci: three loads side by side)
    const ChunkInfo none{-1, 0, 0, -1};
    const ChunkInfo before = cidx > 0 ? checked_chunk(chunks[cidx - 1], a.tb) : none;
    const ChunkInfo after = cidx + 1 < a.tb.max_chunks ? checked_chunk(chunks[cidx + 1], a.tb) : none;
    if (chunk_follows(before, ci)) return;  // the block of the chunk in front takes this one's tiles
    if (chunk_follows(ci, after)) nt += after.ntiles;
  }
  const int r = class_rank(a.rank[g], a.rank_lo, 16 * NB);
  if (r <= 0) return;
  for (int i = tid; i < nt * kTileRows; i += RS * 64) rows_s[i] = slot_rows[ci.tile0 * kTileRows + i];
  __syncthreads();
  const int n_base = rs * NBW * 16;   // first rank index of this wave
  const bool mine = r > n_base;       // a wave without live rank indices still carries its half of every tile

  bf16_t* tiles = reinterpret_cast<bf16_t*>(lds);
  const bf16_t* src = (const bf16_t*)a.src + c0 + 8 * li;
  const bf16_t* hT = (const bf16_t*)a.hT + (int64_t)(n_base + li) * a.ldh + (int64_t)ci.tile0 * kTileRows + 8 * kb;
  f32x4 acc[8][NBW];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) acc[q][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Piece {
    uint4 x[PR];     // rows 8 kb + PR rs + i of the tile, columns 8 li .. 8 li + 7
    uint4 h[NBW];
    uint32_t live;
  };
  auto issue = [&](int t, Piece& P) {
    const int tc = min(t, nt - 1);
    int rows[PR];
    __builtin_memcpy(rows, __builtin_assume_aligned(rows_s + tc * kTileRows + 8 * kb + PR * rs, 4 * PR), 4 * PR);
    P.live = 0;
#pragma unroll
    for (int i = 0; i < PR; ++i) {
      const int row = checked_row(rows[i], a.tb);
      P.x[i] = ld16(src + (int64_t)max(row, 0) * a.ld_src);
      P.live |= row >= 0 ? (1u << i) : 0u;
    }
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) P.h[nb] = ld16(hT + (int64_t)(16 * nb) * a.ldh + tc * kTileRows);
  };
  auto consume = [&](int t, const Piece& P) {
    bf16_t* buf = tiles + (t & 1) * (kTileRows * XS);
#pragma unroll
    for (int i = 0; i < PR; ++i)
      st16(buf + (8 * kb + PR * rs + i) * XS + 8 * li, (P.live >> i) & 1u ? P.x[i] : zero4());
    lds_barrier();
    if (!mine) return;
    uint4 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = ld16(buf + (8 * kb + i) * XS + 8 * li);
    // 8x8 transpose inside the lane: tr holds column q of the 8 rows
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int d = q >> 1;
      const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
      uint32_t e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t wsrc[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
        e[i] = wsrc[d];
      }
      uint4 tr;
      tr.x = __builtin_amdgcn_perm(e[1], e[0], sel);
      tr.y = __builtin_amdgcn_perm(e[3], e[2], sel);
      tr.z = __builtin_amdgcn_perm(e[5], e[4], sel);
      tr.w = __builtin_amdgcn_perm(e[7], e[6], sel);
#pragma unroll
      for (int nb = 0; nb < NBW; ++nb) acc[q][nb] = mfma16(tr, P.h[nb], acc[q][nb]);
    }
  };
  Piece T[S];
#pragma unroll
  for (int i = 0; i < S - 1; ++i) issue(i, T[i]);
  int t = 0;
  for (; t + S <= nt; t += S) {  // every tile consumed in here exists (the youngest requests may lie past the end)
#pragma unroll
    for (int i = 0; i < S; ++i) {
      issue(t + i + S - 1, T[(i + S - 1) % S]);
      consume(t + i, T[i]);
    }
  }
  // fewer than S tiles are left, all of them requested already; both waves take the same trips (barriers inside)
#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (t + i < nt) consume(t + i, T[i]);
  __syncthreads();  // the last tile has been read everywhere: its buffer becomes the staging area
  if constexpr (NBS == NBW) {
    if (mine) wgrad_store<NBW>(acc, lds + n_base * OS, a, ci, g, r, c0, lane, n_base);
  } else {
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) {
      if (r <= n_base + 16 * nb) break;
      f32x4 one[8][1];
#pragma unroll
      for (int q = 0; q < 8; ++q) one[q][0] = acc[q][nb];
      wgrad_store<1>(one, lds + rs * 16 * OS, a, ci, g, r, c0, lane, n_base + 16 * nb);
    }
  }
}

template <int NB, int S, int PAIRS>
__global__ __launch_bounds__((NB == 8 ? 256 : 128) * PAIRS) void k_wgrad_coop(WgradArgs a, const ChunkInfo* __restrict__ chunks,
                                                              const int32_t* __restrict__ slot_rows) {
  wgrad_coop_body<NB, S, PAIRS>(a, chunks, slot_rows, blockIdx.x * PAIRS + (PAIRS > 1 ? threadIdx.x >> 7 : 0), blockIdx.y,
                                gridDim.x * PAIRS);
}

// The expand above rank 16: written or added, one class or several.
template <int NB>
inline void launch_expand_multi(const PassArgs& a, const bf16_t* hrow, const SegView& seg, const SegLayout& L, hipStream_t s) {
  constexpr int TPI = kSetTiles;
  const int64_t blocks = ceil_div(L.max_tiles, TPI) * ceil_div(a.width_dst >> 7, 4);
  const auto kernel = a.dst_store ? (a.wl_sets.ids ? k_expand_multi<NB, TPI, true, true> : k_expand_multi<NB, TPI, false, true>)
                                  : (a.wl_sets.ids ? k_expand_multi<NB, TPI, true, false> : k_expand_multi<NB, TPI, false, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, s, a, hrow, seg.tile_group, seg.slot_table(a.map_rows),
                     seg.set_walk(a.map_rows), seg.header, seg.round_moved, (int)std::min<int64_t>(L.sort_blocks, 64),
                     (int)L.max_tiles);
}

}  // namespace

}  // namespace tk
