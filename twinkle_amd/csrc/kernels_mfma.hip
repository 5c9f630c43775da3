// bf16 launches of the segmented LoRA pass (kernel templates: lora_kernels.h), and the bf16-only kernels:
//
//   k_shrink_few        h of few tiles at rank <= 16
//   k_shrink_quad       h at rank 17 to 64 with many tiles
//   k_dy_fused<NB>      backward, rank <= 32: dB and the slices of dh from one pass over dy
//   k_transpose_job     B^T, A^T copies for the backward shrink / expand
//   *_multi             the same bodies for several projections in one launch
#include <algorithm>

#include "lora_kernels.h"

namespace tk {

namespace {

// Work item `item` of projection p out of nproj that read the same rows: blocks go to the eight XCDs (each with an
// L2 of its own) round-robin by block number, so the items are numbered in runs of eight per projection: blocks
// 8 (g nproj + p) + j, j < 8, are items 8 g + j of projection p.  The nproj blocks that read the same piece of the
// source then lie eight apart, run on the same XCD at about the same time, and the piece comes from memory once and
// from that L2 afterwards.
__device__ inline void shared_source_item(int block, int nproj, int& p, int& item) {
  const int run = block >> 3;
  p = run % nproj;
  item = ((run / nproj) << 3) + (block & 7);
}

// The shrink of up to kMaxShared projections of one padded rank that read the same source, in one launch: the
// bodies of k_shrink_pair, every piece of the source crossing memory once (see shared_source_item).
template <int NB, int NW>
__global__ __launch_bounds__(NW * 64) void k_shrink_pair_multi(PassJobs jobs, int nproj, int items,
                                                               const int32_t* __restrict__ tile_group,
                                                               const int32_t* __restrict__ slot_rows, int max_tiles) {
  int p, item;
  shared_source_item(blockIdx.x, nproj, p, item);
  if (item >= items) return;
  const PassArgs& a = jobs.p[p];
  shrink_pair_body<NB, NW>(a, (bf16_t*)a.hT + (int64_t)a.rpad * a.ldh, tile_group, slot_rows, max_tiles, item);
}

// The same for up to kMaxShared projections that read the same source (see shared_source_item).
template <int NB>
__global__ __launch_bounds__(512) void k_shrink_oct_multi(PassJobs jobs, int nproj, int items,
                                                           const int32_t* __restrict__ tile_group,
                                                           const int32_t* __restrict__ slot_rows, int max_tiles) {
  int p, item;
  shared_source_item(blockIdx.x, nproj, p, item);
  if (item >= items) return;
  shrink_oct_body<NB>(jobs.p[p], tile_group, slot_rows, max_tiles, item);
}

// The same for up to kMaxShared projections of padded rank 16 in one launch: blockIdx.y selects the projection.
__global__ __launch_bounds__(256) void k_shrink_finish_multi(PassJobs jobs, const int32_t* __restrict__ tile_group,
                                                             const int32_t* __restrict__ slot_rows) {
  const PassArgs& a = jobs.p[blockIdx.y];
  shrink_finish_body<1>(a, (bf16_t*)a.hT + (int64_t)a.rpad * a.ldh, tile_group, slot_rows, blockIdx.x);
}

// Up to kMaxShared projections of padded rank 16 in one launch: blockIdx.y selects the projection; the grid
// is as wide as the widest projection needs.
__global__ __launch_bounds__(256) void k_expand_mfma_multi(PassJobs jobs, const int32_t* __restrict__ tile_group,
                                                           const int32_t* __restrict__ slot_rows,
                                                           const int32_t* __restrict__ tile_walk, int max_tiles) {
  const PassArgs& a = jobs.p[blockIdx.y];
  expand_flat_body<1>(a, (const bf16_t*)a.hT + (int64_t)a.rpad * a.ldh, tile_group, slot_rows, tile_walk,
                      max_tiles * (a.width_dst >> 7), blockIdx.x);
}

// The transposed copies as a launch of their own (backward paths whose first kernel cannot carry them as a side job).
__global__ __launch_bounds__(256) void k_transpose_job(TransposeJob t, const int32_t* __restrict__ rank, int rpad) {
  transpose_weights_job(t, rank, rpad, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
}

// The same contraction for up to kMaxShared projections that read the same source (dA_p = dh_p^T x for the
// projections of one input): one launch, the bodies of k_wgrad_coop, every tile of the source crossing memory
// once (see shared_source_item).  Work item = (chunk, 128 columns), column block fastest.
template <int NB, int S>
__global__ __launch_bounds__(128) void k_wgrad_coop_multi(SharedWgradArgs jobs, int items, int nx,
                                                            const ChunkInfo* __restrict__ chunks,
                                                            const int32_t* __restrict__ slot_rows) {
  int p, item;
  shared_source_item(blockIdx.x, jobs.nproj, p, item);
  if (item >= items) return;
  wgrad_coop_body<NB, S>(jobs.w[p], chunks, slot_rows, item % nx, item / nx, nx);
}

// ---------------------------------------------------------------------------
// Backward, both uses of dy in one pass (rank <= 16 NB, NB = 1 or 2; width a multiple of 512): a block of four waves owns
// (chunk of one group, 512 columns), wave w the columns [128 w, 128 w + 128) of it.
// Per tile a wave loads its 32 x 128 piece once, in the weight-gradient layout (a lane holds 8 rows x 8
// columns), and uses it twice:
//   dB:  the piece, transposed in registers, is the MFMA A operand with the rows as contraction index,
//        accumulated over the chunk's tiles exactly like k_wgrad_pipe does;
//   dh:  the piece goes through a per-wave LDS buffer to come back in the row-major operand layout and
//        is multiplied with the wave's 128 x rank block of B (loaded once per chunk, straight from the
//        adapter's [out][r] layout); the four waves' partial dh[32][rank] meet in LDS after a block
//        barrier and one of them writes the sum as slice `blockIdx.x` of the split-shrink buffer, which
//        k_shrink_finish turns into dh like after a separate shrink.
// dy crosses the memory system once instead of twice.  Sums are formed in a fixed order.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void dy_fused_body(const WgradArgs& a, const void* const* __restrict__ lora_B, int64_t ldb,
                                              float* __restrict__ hpart, int kslices,
                                              const ChunkInfo* __restrict__ chunks,
                                              const int32_t* __restrict__ slot_rows, int bx, int by, int x_blocks) {
  constexpr int RP = 16 * NB;
  constexpr int SS = 136;     // row stride of the staged piece in bf16 (272 B)
  constexpr int PR = RP + 1;  // row stride of the partial dh in floats
  extern __shared__ int32_t rows_s[];  // the chunk's row indices (chunk_tiles x 32)
  __shared__ __attribute__((aligned(16))) bf16_t stage[4][kTileRows * SS];
  __shared__ float part[2][4][kTileRows * PR];
  static_assert(sizeof(bf16_t) * kTileRows * SS >= sizeof(float) * 16 * kWgradStageStride, "stage holds a dB block too");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  if (by < a.tr.y_blocks) {  // side job: the first rows of the grid transpose the adapter weights
    transpose_weights_job(a.tr, a.rank, a.rpad, ((int64_t)by * x_blocks + bx) * 256 + tid,
                          (int64_t)a.tr.y_blocks * x_blocks * 256);
    return;
  }
  const int cidx = work_item(a.wl_chunks, by - a.tr.y_blocks);
  if (cidx < 0) return;  // past the end of this rank class's list
  const ChunkInfo ci = checked_chunk(chunks[cidx], a.tb);
  const int g = ci.group;
  if (g < 0) return;
  const int r = class_rank(a.rank[g], a.rank_lo, RP);
  if (r <= 0) return;
  const int slab = bx;
  const int c0 = slab * 512 + wave * 128;
  const int nt = ci.ntiles;
  for (int i = tid; i < nt * kTileRows; i += 256) rows_s[i] = slot_rows[ci.tile0 * kTileRows + i];
  // this wave's block of B as MFMA B operand: lane (n = 16 nb + li, kb) holds B[c0 + 32 s + 8 kb + i][n], i = 0..7
  uint4 wB[NB][4];
  const void* Bsrc = lora_B[g];
  const bool b_f32 = a.grad_f32 != 0;  // fp32 adapters: converted as they are loaded
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = 16 * nb + li;
    const int64_t b0 = (int64_t)(c0 + 8 * kb) * ldb + (n < r ? n : 0);
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      uint32_t e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)  // (the address is valid for every lane: loads first, masks after)
        e[i] = load_weight(Bsrc, b0 + (int64_t)(32 * s4 + i) * ldb, b_f32);
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = n < r ? e[i] : 0;
      wB[nb][s4] = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
    }
  }
  __syncthreads();

  const bf16_t* src = (const bf16_t*)a.src + c0 + 8 * li;
  const bf16_t* hT = (const bf16_t*)a.hT + (int64_t)li * a.ldh + (int64_t)ci.tile0 * kTileRows + 8 * kb;
  bf16_t* my_stage = stage[wave];
  f32x4 acc[8][NB];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[q][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // loads are unconditional (tiles past the end re-read the last one, padding slots read row 0) and what
  // must not count is zeroed when it is consumed: no branch between a load and its use
  auto issue = [&](int t, uint4 (&x)[8], uint4 (&h)[NB], uint32_t& live) {
    const int tc = min(t, nt - 1);
    const int4 ra = *reinterpret_cast<const int4*>(rows_s + tc * kTileRows + 8 * kb);
    const int4 rb = *reinterpret_cast<const int4*>(rows_s + tc * kTileRows + 8 * kb + 4);
    const int rows[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
    live = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int row = checked_row(rows[q], a.tb);
      x[q] = ld16(src + (int64_t)max(row, 0) * a.ld_src);
      live |= (t < nt && row >= 0) ? (1u << q) : 0u;
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) h[nb] = ld16(hT + (int64_t)(16 * nb) * a.ldh + tc * kTileRows);
  };
  auto consume = [&](int t, uint4 (&x)[8], const uint4 (&h)[NB], uint32_t live) {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (!((live >> q) & 1u)) x[q] = zero4();
    // the piece in row-major order for the dh product
#pragma unroll
    for (int q = 0; q < 8; ++q) st16(my_stage + (8 * kb + q) * SS + 8 * li, x[q]);
    // dB: 8x8 transpose inside the lane, rows become the contraction index
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
      for (int nb = 0; nb < NB; ++nb) acc[q][nb] = mfma16(tr, h[nb], acc[q][nb]);
    }
  };
  // dh of tile t from the staged piece: partial over this wave's 128 columns (LDS operations of one wave complete
  // in order); needs no register of the tile any more
  auto consume_dh = [&](int t) {
    float* mine = part[t & 1][wave];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      f32x4 d[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) d[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const uint4 piece = ld16(my_stage + (16 * tt + li) * SS + 32 * s4 + 8 * kb);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) d[nb] = mfma16(piece, wB[nb][s4], d[nb]);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v) mine[(16 * tt + 4 * kb + v) * PR + 16 * nb + li] = d[nb][v];
    }
    lds_barrier();
    if (wave == (t & 3)) {
      float* o = hpart + ((int64_t)(ci.tile0 + t) * kslices + slab) * (kTileRows * RP);
#pragma unroll
      for (int i = 0; i < 8 * NB; ++i) {
        const int idx = lane + 64 * i, row = idx / RP, n = idx % RP;
        float sum = part[t & 1][0][row * PR + n];
        sum += part[t & 1][1][row * PR + n];
        sum += part[t & 1][2][row * PR + n];
        sum += part[t & 1][3][row * PR + n];
        o[idx] = sum;
      }
    }
  };

  constexpr int S = NB == 1 ? TK_DY_STAGES : TK_DY_STAGES2;  // software pipeline: S - 1 tiles in flight while one is consumed
  struct Tile {
    uint4 x[8];
    uint4 h[NB];
    uint32_t live;
  };
  Tile T[S];
  if constexpr (S == 1) {
    // one tile in registers: its successor is requested as soon as the dB products have used it up, and is in
    // flight during the dh half of the iteration
    issue(0, T[0].x, T[0].h, T[0].live);
    for (int t = 0; t < nt; ++t) {
      consume(t, T[0].x, T[0].h, T[0].live);
      issue(t + 1, T[0].x, T[0].h, T[0].live);
      consume_dh(t);
    }
  } else {
#pragma unroll
    for (int i = 0; i < S - 1; ++i) issue(i, T[i].x, T[i].h, T[i].live);
    int t = 0;
    for (; t + S <= nt; t += S) {  // every tile consumed in here exists (the youngest requests may lie past the end)
#pragma unroll
      for (int i = 0; i < S; ++i) {
        Tile& Y = T[(i + S - 1) % S];
        issue(t + i + S - 1, Y.x, Y.h, Y.live);
        consume(t + i, T[i].x, T[i].h, T[i].live);
        consume_dh(t + i);
      }
    }
    // fewer than S tiles are left, all of them requested already
#pragma unroll
    for (int i = 0; i < S - 1; ++i)
      if (t + i < nt) {
        consume(t + i, T[i].x, T[i].h, T[i].live);
        consume_dh(t + i);
      }
  }
  // every wave has its own 128 columns of dB; they leave 16 rank indices at a time through the wave's stage
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    if (16 * nb >= r) break;
    f32x4 one[8][1];
#pragma unroll
    for (int q = 0; q < 8; ++q) one[q][0] = acc[q][nb];
    wgrad_store<1>(one, reinterpret_cast<float*>(my_stage), a, ci, g, r, c0, lane, 16 * nb);
  }
}

template <int NB>
__global__ __launch_bounds__(256) void k_dy_fused(WgradArgs a, const void* const* __restrict__ lora_B, int64_t ldb,
                                                  float* __restrict__ hpart, int kslices,
                                                  const ChunkInfo* __restrict__ chunks,
                                                  const int32_t* __restrict__ slot_rows) {
  dy_fused_body<NB>(a, lora_B, ldb, hpart, kslices, chunks, slot_rows, blockIdx.x, blockIdx.y, gridDim.x);
}

// Up to kMaxShared projections in one launch: a narrow projection alone has too few (chunk, 512 columns)
// blocks to fill the chip.  The jobs' column slabs lie side by side along blockIdx.x, so that the blocks of
// all projections are dispatched interleaved and run next to each other.
__global__ __launch_bounds__(256) void k_dy_fused_multi(DyFusedJobs jobs, const ChunkInfo* __restrict__ chunks,
                                                        const int32_t* __restrict__ slot_rows, int max_chunks) {
  int p = 0;
#pragma unroll
  for (int i = 1; i < kMaxShared; ++i) p += (i < jobs.n && (int)blockIdx.x >= jobs.x_first[i]) ? 1 : 0;
  const DyFusedJob& j = jobs.j[p];
  if ((int)blockIdx.y >= j.a.tr.y_blocks + max_chunks) return;
  dy_fused_body<1>(j.a, j.lora_B, j.ldb, j.hpart, j.kslices, chunks, slot_rows, blockIdx.x - jobs.x_first[p],
                   blockIdx.y, j.x_blocks);
}

// ---------------------------------------------------------------------------
// k_shrink_oct (lora_kernels.h) with four waves instead of eight: a block of four waves owns (eight consecutive tiles,
// slice of columns), wave w takes tiles 2 w and 2 w + 1 through all steps of 64 columns, and the weight block of a step
// (16 * NB x 64) is fetched once per block, 16 B per thread, into a double-buffered LDS tile.  Two such blocks fit a CU
// where one of eight waves does (registers), and a block that waits leaves the other one running, which is what counts
// once the chip is full (see oct_blocks).  Activations: two or three steps in registers per wave.
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ void shrink_quad_body(const PassArgs& a, const int32_t* __restrict__ tile_group,
                                                 const int32_t* __restrict__ slot_rows, int max_tiles, int item) {
  constexpr int RP = 16 * NB;
  constexpr int WS = 72;                    // row stride of a staged weight block in bf16 (144 B: conflict-free)
  constexpr int NLD = (RP * 8 + 255) / 256;  // 16-byte pieces of a weight block per thread
  constexpr int S = NB == 4 ? 2 : 3;  // steps of activations in registers (rank 64: the accumulators take the room)
  __shared__ __attribute__((aligned(16))) bf16_t wbuf[2][RP * WS];
  __shared__ int32_t gts[8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int nth = item / a.kslices, ks = item - nth * a.kslices;
  const int set = work_item(a.wl_octs, nth);
  if (set < 0) return;  // past the end of this rank class's list (uniform over the block)
  const int t_first = set * 8;
  if (tid < 8) gts[tid] = t_first + tid < max_tiles ? checked_group(tile_group[t_first + tid], a.tb) : -1;
  const int nsteps = a.width_src >> 6;
  const int s0 = ks * a.set_steps;
  const int ns = min(a.set_steps, nsteps - s0);  // >= 1 for every slice
  // this wave's two tiles
  const bf16_t* src = (const bf16_t*)a.src;
  const bf16_t *xa[2], *xb[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = min(t_first + 2 * wave + u, max_tiles - 1);
    int ra = slot_rows[t * kTileRows + li], rb = slot_rows[t * kTileRows + 16 + li];
    ra = min(max(ra, 0), a.src_rows - 1);
    rb = min(max(rb, 0), a.src_rows - 1);
    xa[u] = src + (int64_t)ra * a.ld_src + 16 * kb + (int64_t)s0 * 64;
    xb[u] = src + (int64_t)rb * a.ld_src + 16 * kb + (int64_t)s0 * 64;
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
    bool mine[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) mine[u] = 2 * wave + u >= lo && 2 * wave + u < hi;
    const bool active = mine[0] || mine[1];  // wave-uniform
    const bf16_t* W1 = group_weight<bf16_t>(a.w_shrink, a.w_shrink_base, a.shrink_group_stride, g) + (int64_t)s0 * 64;
    // staging: piece p = tid + 256 i is columns 8 (p % 8) .. + 8 of rank index p / 8
    auto stage_load = [&](int s, uint4 (&wr)[NLD]) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int p = tid + 256 * i, n = p >> 3;
        wr[i] = (n < r && s < ns) ? ld16(W1 + (int64_t)n * a.ld_shrink + (s << 6) + 8 * (p & 7)) : zero4();
      }
    };
    auto stage_store = [&](int buf, const uint4 (&wr)[NLD]) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int p = tid + 256 * i, n = p >> 3;
        if (n < RP) st16(&wbuf[buf][n * WS + 8 * (p & 7)], wr[i]);
      }
    };
    struct Step {
      uint4 x0[2][2], x1[2][2];
    };
    auto issue = [&](int s, Step& X) {
      const int c = min(s, ns - 1) << 6;  // requests past the slice repeat its last step and are not used
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        X.x0[u][0] = ld16(xa[u] + c);
        X.x1[u][0] = ld16(xa[u] + c + 8);
        X.x0[u][1] = ld16(xb[u] + c);
        X.x1[u][1] = ld16(xb[u] + c + 8);
      }
    };
    f32x4 acc[2][2][NB];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[u][tt][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 wr[NLD];
    auto step = [&](int s, const Step& X, Step& Xnext) {
      lds_barrier();  // block s is complete; the other buffer has been read by everyone
      stage_load(s + 1, wr);
      if (active) issue(s + S - 1, Xnext);
      if (active) {
        const bf16_t* wb = wbuf[s & 1] + li * WS + 16 * kb;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const uint4 w0 = ld16(wb + 16 * nb * WS), w1 = ld16(wb + 16 * nb * WS + 8);
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
              acc[u][tt][nb] = mfma16(X.x0[u][tt], w0, acc[u][tt][nb]);
              acc[u][tt][nb] = mfma16(X.x1[u][tt], w1, acc[u][tt][nb]);
            }
        }
      }
      stage_store((s + 1) & 1, wr);  // block s + 1 (zeros past the slice), visible behind the next barrier
    };
    Step T[S];
    stage_load(0, wr);
    if (active) {
#pragma unroll
      for (int i = 0; i < S - 1; ++i) issue(i, T[i]);
    }
    stage_store(0, wr);
    int s = 0;
    for (; s + S <= ns; s += S) {
#pragma unroll
      for (int i = 0; i < S; ++i) step(s + i, T[i], T[(i + S - 1) % S]);
    }
#pragma unroll
    for (int i = 0; i < S - 1; ++i)
      if (s + i < ns) step(s + i, T[i], T[(i + S - 1) % S]);  // block-uniform
    lds_barrier();  // the next run's first block goes into buffer 0
    if (!active) continue;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (!mine[u]) continue;
      float* out = a.hpart + ((int64_t)(t_first + 2 * wave + u) * a.kslices + ks) * (kTileRows * RP) + 4 * kb * RP + li;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int v = 0; v < 4; ++v) out[(16 * tt + v) * RP + 16 * nb] = acc[u][tt][nb][v];
    }
  }
}

template <int NB>
__global__ __launch_bounds__(256, 2) void k_shrink_quad(PassArgs a, const int32_t* __restrict__ tile_group,
                                                     const int32_t* __restrict__ slot_rows, int max_tiles) {
  shrink_quad_body<NB>(a, tile_group, slot_rows, max_tiles, blockIdx.x);
}

// The same for up to kMaxShared projections that read the same source (see shared_source_item).
template <int NB>
__global__ __launch_bounds__(256, 2) void k_shrink_quad_multi(PassJobs jobs, int nproj, int items,
                                                           const int32_t* __restrict__ tile_group,
                                                           const int32_t* __restrict__ slot_rows, int max_tiles) {
  int p, item;
  shared_source_item(blockIdx.x, nproj, p, item);
  if (item >= items) return;
  shrink_quad_body<NB>(jobs.p[p], tile_group, slot_rows, max_tiles, item);
}

// The shrink of few tiles at padded rank 16: one wave per (tile, slice) requests its whole slice, eight steps, at once.
// There are too few blocks to cover latencies with each other, so the launch takes as long as one block, and that as
// many memory latencies as it has batches (five with k_shrink_pair's).  Same products in the same order: same bits.
__global__ __launch_bounds__(64) void k_shrink_few(PassArgs a, bf16_t* __restrict__ hrow,
                                                   const int32_t* __restrict__ tile_group,
                                                   const int32_t* __restrict__ slot_rows) {
  __shared__ float part[1][kTileRows][17];
  const int nth = blockIdx.x / a.kslices, ks = blockIdx.x - nth * a.kslices;
  const int tile = checked_tile(work_item(a.wl_tiles, nth), a.tb);
  if (tile < 0) return;
  const int g = checked_group(tile_group[tile], a.tb);
  if (g < 0) return;
  const int tiles[1] = {tile};
  shrink_tiles<1, 1, 1, kShrinkSteps>(a, hrow, slot_rows, tiles, g, ks, part);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Few tiles at padded rank 16: k_shrink_few up to seven waves per CU.  Forward with few / pair, us (4096 columns unless
// said): 1024 rows 13.5 / 14.8, 4096 (1160 blocks) 21.2 / 21.9, 6144 (1672) 23.9 / 24.4, 8192 (2184) 29.0 / 28.1, 12288
// 36.4 / 34.9, 16 adapters; 12288 x 2048 (1572) 25.8 / 26.5; 14336 columns: 1024 rows 21.9 / 22.8, 2048 (1932) 27.7 / 26.5.
// (Tiles that may hold rows count: 256 rows of a decode step over 512 expert groups are 256, and the empty ones cost little.)
constexpr int64_t kFewShrinkBlocks = 7 * 256;  // (tile, slice) pairs
// The expand of few tiles adds the slices itself: a launch less against every wave's reading of its tile's slices (2 KB
// each, from L2; nothing is read for padding slots, so tiles of few rows are cheap).  GPU time of a forward with / without:
//   up to 4 slices (2048 columns)  32 x 2048 -> 2048 9.7 / 10.9, 512 x 1024 -> 14336 13.9 / 14.8 (4700 readings),
//                                  3072 x 2048 -> 2048 17.5 / 17.3 (6460), 2048 x 2048 -> 4096 18.6 / 17.5 (10370)
//   8 slices, 4096 -> 4096         16 adapters: 32 rows 10.7 / 11.2, 128 11.1 / 11.6, 256 12.5 / 12.1;
//                                  one adapter: 8 rows 10.5 / 10.7, 32 12.3 / 11.7 (a full tile)
//   28 slices, 14336 -> 4096       4 adapters: 8 rows 14.7 / 13.2, 64 18.1 / 13.7 us
// An eager call saves 1 to 2.5 us of host time besides (a decode step of 32 rows takes 30 us instead of 33; 256 rows of 16
// adapters, eight slices, one after the other: 13.1 instead of 15.1), so there eight slices count as few at any row count.
constexpr int64_t kFewFinishReads = 6400;
inline bool finish_in_expand(const PassArgs& a, const SegLayout& L, hipStream_t s) {
  if (a.kslices <= 1 || a.kslices > 8 || L.max_tiles * (a.width_dst >> 7) * a.kslices > kFewFinishReads) return false;
  return a.kslices <= 4 || L.rows <= 8 * (int64_t)L.groups || !stream_is_capturing(s);
}

template <int NB>
void launch_pass(const PassArgs& a, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  bf16_t* hrow = (bf16_t*)a.hT + (int64_t)a.rpad * a.ldh;  // second half of the h buffer
  const int32_t* rows = seg.slot_table(a.map_rows);
  constexpr int NW = NB == 1 ? 1 : (NB == 2 ? 2 : 4);  // shrink_waves(16 * NB)
  if (phases & 1) {
    if (NB > 1 && a.set_steps > 0 && shrink_dl_applies(a))
      hipLaunchKernelGGL((k_shrink_dl<NB == 1 ? 2 : NB>), dim3((unsigned)(ceil_div(L.max_tiles, 8) * a.kslices)), dim3(512), 0,
                         s, a, seg.tile_group, rows, (int)L.max_tiles);
    else if (NB > 1 && a.set_steps > 0)  // see shrink_plan
      hipLaunchKernelGGL((a.set_waves == 8 ? k_shrink_oct<NB == 1 ? 2 : NB> : k_shrink_quad<NB == 1 ? 2 : NB>),
                         dim3((unsigned)(ceil_div(L.max_tiles, 8) * a.kslices)), dim3(64 * a.set_waves), 0, s, a,
                         seg.tile_group, rows, (int)L.max_tiles);
    else if (NB == 1 && L.live_tiles() * a.kslices <= kFewShrinkBlocks)
      hipLaunchKernelGGL(k_shrink_few, dim3((unsigned)(L.max_tiles * a.kslices)), dim3(64), 0, s, a, hrow, seg.tile_group,
                         rows);
    else
      hipLaunchKernelGGL((k_shrink_pair<NB, NW>), dim3((unsigned)(ceil_div(L.max_tiles, 2) * a.kslices)),
                         dim3(NW * 64), 0, s, a, hrow, seg.tile_group, rows, (int)L.max_tiles);
  }
  const bool fin = NB == 1 && (phases & 5) && (phases & 2) && a.dst && !a.class_mode && finish_in_expand(a, L, s);
  if ((phases & 5) && a.kslices > 1 && !fin)
    hipLaunchKernelGGL((k_shrink_finish<NB>), shrink_finish_grid<NB>(L), dim3(256), 0, s, a, hrow, seg.tile_group,
                       rows);
  if (!a.dst || !(phases & 2)) return;
  if constexpr (NB > 1) {
    launch_expand_multi<NB>(a, hrow, seg, L, s);
  } else {
    const int64_t items = L.max_tiles * (a.width_dst >> 7);
    const auto kernel = fin ? k_expand_mfma<NB, true> : k_expand_mfma<NB, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(items, 4)), dim3(256), 0, s, a, hrow, seg.tile_group, rows,
                       seg.tile_walk(a.map_rows), (int)items);
  }
}

template <int NB, int S>
void launch_wgrad_pipe(const WgradArgs& a0, const SegView& seg, const SegLayout& L, hipStream_t s) {
  WgradArgs a = a0;
  a.tr.y_blocks = 0;
  if (a.tr.aT) {  // about four 16-byte outputs per thread of the side job
    const int64_t units = (int64_t)a.tr.groups * a.rpad * ((a.tr.out_features + a.tr.in_features) / 64);
    a.tr.y_blocks = (int)std::min<int64_t>(64, std::max<int64_t>(1, units / (2 * (a.width / 128) * 64)));
  }
  const dim3 grid((unsigned)(a.width / 128), (unsigned)(L.max_chunks + a.tr.y_blocks));
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);  // a chunk's row indices
  hipLaunchKernelGGL((k_wgrad_pipe<NB, S>), grid, dim3(64), dyn, s, a, seg.chunks,
                     seg.slot_table(a.map_rows));
}

template <int NB>
void launch_wgrad_coop(const WgradArgs& a0, const SegView& seg, const SegLayout& L, hipStream_t s) {
  constexpr int S = TK_COOP_STAGES;
  WgradArgs a = a0;
  a.tr.y_blocks = 0;
  if (a.tr.aT) {
    const int64_t units = (int64_t)a.tr.groups * a.rpad * ((a.tr.out_features + a.tr.in_features) / 64);
    a.tr.y_blocks = (int)std::min<int64_t>(64, std::max<int64_t>(1, units / (2 * (a.width / 128) * 128)));
  }
  const int nx = a.width / 128;
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t) * (a.pair_chunks ? 2 : 1);
  // Two pairs per block only where that still leaves every CU several blocks (the grid counts every chunk slot of
  // the table): measured at config 3 (65 chunk slots x 112 / 32 column blocks) 2.4 % of the step; at config 5's
  // q projection (41 x 32) the coarser blocks balance worse over the CUs and cost 13 %.
  if (TK_COOP_PAIRS == 2 && nx % 2 == 0 && (int64_t)nx * L.max_chunks >= 8 * 256) {
    const dim3 grid((unsigned)(nx / 2), (unsigned)(L.max_chunks + a.tr.y_blocks));
    hipLaunchKernelGGL((k_wgrad_coop<NB, S, 2>), grid, dim3(256), dyn, s, a, seg.chunks, seg.slot_table(a.map_rows));
  } else {
    const dim3 grid((unsigned)nx, (unsigned)(L.max_chunks + a.tr.y_blocks));
    hipLaunchKernelGGL((k_wgrad_coop<NB, S, 1>), grid, dim3(128), dyn, s, a, seg.chunks, seg.slot_table(a.map_rows));
  }
}

}  // namespace

bool dy_fused_supported(const WgradArgs& a, int kslices) {
  return (a.rpad == 16 || a.rpad == 32) && a.width % 512 == 0 && kslices >= 2 && kslices == a.width / 512 &&
         wgrad_mfma_supported(a);
}

int launch_dy_fused(const WgradArgs& a0, const void* const* lora_B, int64_t ldb, float* hpart, int kslices,
                    const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  WgradArgs a = a0;
  a.tr.y_blocks = 0;
  if (a.tr.aT) {
    const int64_t units = (int64_t)a.tr.groups * a.rpad * ((a.tr.bT ? a.tr.out_features : 0) + a.tr.in_features) / 64;
    a.tr.y_blocks = (int)std::min<int64_t>(64, std::max<int64_t>(1, units / (2 * (a.width / 512) * 256)));
  }
  const dim3 grid((unsigned)(a.width / 512), (unsigned)(L.max_chunks + a.tr.y_blocks));
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);  // a chunk's row indices
  if (a.rpad == 16)
    hipLaunchKernelGGL(k_dy_fused<1>, grid, dim3(256), dyn, s, a, lora_B, ldb, hpart, kslices, seg.chunks,
                       seg.slot_table(a.map_rows));
  else
    hipLaunchKernelGGL(k_dy_fused<2>, grid, dim3(256), dyn, s, a, lora_B, ldb, hpart, kslices, seg.chunks,
                       seg.slot_table(a.map_rows));
  return check_launch();
}

int launch_dy_fused_multi(const DyFusedJob* jobs, int n, const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0 || n == 0) return TK_OK;
  DyFusedJobs J{};
  J.n = n;
  int gy = 0;
  for (int p = 0; p < n; ++p) {
    DyFusedJob& j = J.j[p];
    j = jobs[p];
    j.x_blocks = j.a.width / 512;
    j.a.tr.y_blocks = 0;
    if (j.a.tr.aT) {
      const int64_t units =
          (int64_t)j.a.tr.groups * j.a.rpad * ((j.a.tr.bT ? j.a.tr.out_features : 0) + j.a.tr.in_features) / 64;
      j.a.tr.y_blocks = (int)std::min<int64_t>(64, std::max<int64_t>(1, units / (2 * j.x_blocks * 256)));
    }
    J.x_first[p + 1] = J.x_first[p] + j.x_blocks;
    gy = std::max(gy, (int)L.max_chunks + j.a.tr.y_blocks);
  }
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);
  hipLaunchKernelGGL(k_dy_fused_multi, dim3((unsigned)J.x_first[n], (unsigned)gy), dim3(256), dyn, s, J, seg.chunks,
                     seg.slot_table(J.j[0].a.map_rows), (int)L.max_chunks);
  return check_launch();
}

// Finish and / or flat expand of several projections of padded rank 16 (phases: 4 finish, 2 expand).
int launch_pass_multi(const PassArgs* a, int n, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  if (L.rows == 0 || n == 0) return TK_OK;
  PassJobs J{};
  int64_t widest = 0;
  for (int p = 0; p < n; ++p) {
    J.p[p] = a[p];
    widest = std::max<int64_t>(widest, a[p].width_dst >> 7);
  }
  const int32_t* rows = seg.slot_table(a[0].map_rows);
  if (phases & 4)
    hipLaunchKernelGGL(k_shrink_finish_multi, dim3((unsigned)L.max_tiles, (unsigned)n), dim3(256), 0, s, J,
                       seg.tile_group, rows);
  if (phases & 2)
    hipLaunchKernelGGL(k_expand_mfma_multi, dim3((unsigned)ceil_div(L.max_tiles * widest, 4), (unsigned)n), dim3(256), 0,
                       s, J, seg.tile_group, rows, seg.tile_walk(a[0].map_rows), (int)L.max_tiles);
  return check_launch();
}

// B^T / A^T copies for the MFMA shrink and expand of a backward pass (bf16, out_features a multiple of 8).
// Entries at and beyond a group's rank are left unwritten: those kernels never read them.
int launch_transpose_job(const TransposeJob& t0, const int32_t* rank, int rpad, hipStream_t s) {
  if (t0.groups == 0) return TK_OK;
  TransposeJob t = t0;
  t.skip_dead = 1;
  const int64_t units = (int64_t)t.groups * rpad * ((t.bT ? t.out_features : 0) + t.in_features) / 64;  // 8 x 8 blocks
  const int64_t blocks = std::min<int64_t>(8192, std::max<int64_t>(1, units / 256));
  hipLaunchKernelGGL(k_transpose_job, dim3((unsigned)blocks), dim3(256), 0, s, t, rank, rpad);
  return check_launch();
}

// Shrink (with the slice sums) of n projections of one padded rank above 16 that read the same source.
int launch_shrink_multi(const PassArgs* a, int n, const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0 || n == 0) return TK_OK;
  PassJobs J{};
  for (int p = 0; p < n; ++p) J.p[p] = a[p];
  const int32_t* rows = seg.slot_table(a[0].map_rows);
  const bool set = a[0].set_steps > 0;
  const int items = (int)(ceil_div(L.max_tiles, set ? 8 : 2) * a[0].kslices);
  const dim3 grid((unsigned)(ceil_div(items, 8) * 8 * n));
  if (set) {  // (same sums and same bits as the single-projection launch, whichever kernel either takes)
    const auto kernel = a[0].set_waves == 8 ? (a[0].rpad <= 32 ? k_shrink_oct_multi<2> : k_shrink_oct_multi<4>)
                                            : (a[0].rpad <= 32 ? k_shrink_quad_multi<2> : k_shrink_quad_multi<4>);
    hipLaunchKernelGGL(kernel, grid, dim3(64 * a[0].set_waves), 0, s, J, n, items, seg.tile_group, rows, (int)L.max_tiles);
  } else if (a[0].rpad <= 32) {
    hipLaunchKernelGGL((k_shrink_pair_multi<2, 2>), grid, dim3(128), 0, s, J, n, items, seg.tile_group, rows,
                       (int)L.max_tiles);
  } else {
    hipLaunchKernelGGL((k_shrink_pair_multi<4, 4>), grid, dim3(256), 0, s, J, n, items, seg.tile_group, rows,
                       (int)L.max_tiles);
  }
  if (a[0].kslices > 1) {
    for (int p = 0; p < n; ++p) {
      bf16_t* hrow = (bf16_t*)a[p].hT + (int64_t)a[p].rpad * a[p].ldh;
      if (a[0].rpad <= 32)
        hipLaunchKernelGGL(k_shrink_finish<2>, shrink_finish_grid<2>(L), dim3(256), 0, s, a[p], hrow,
                           seg.tile_group, rows);
      else
        hipLaunchKernelGGL(k_shrink_finish<4>, shrink_finish_grid<4>(L), dim3(256), 0, s, a[p], hrow,
                           seg.tile_group, rows);
    }
  }
  return check_launch();
}

// Row contractions of n projections of one padded rank above 16 over the same source (see k_wgrad_coop_multi).
int launch_wgrad_coop_multi(const SharedWgradArgs& a0, const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0 || a0.nproj == 0) return TK_OK;
  SharedWgradArgs a = a0;
  for (int p = 0; p < a.nproj; ++p) a.w[p].tr = TransposeJob{};
  const int nx = a.w[0].width / 128;
  const int items = nx * (int)L.max_chunks;
  const dim3 grid((unsigned)(ceil_div(items, 8) * 8 * a.nproj));
  size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);
  for (int p = 0; p < a.nproj; ++p)
    if (a.w[p].pair_chunks) dyn = 2 * (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);
  const int32_t* rows = seg.slot_table(a.w[0].map_rows);
  if (a.w[0].rpad <= 32)
    hipLaunchKernelGGL((k_wgrad_coop_multi<2, TK_COOP_STAGES>), grid, dim3(128), dyn, s, a, items, nx, seg.chunks, rows);
  else
    hipLaunchKernelGGL((k_wgrad_coop_multi<4, TK_COOP_STAGES>), grid, dim3(128), dyn, s, a, items, nx, seg.chunks, rows);
  return check_launch();
}

bool pass_mfma_supported(const PassArgs& a) {
  if (a.width_src % 64 != 0 || a.ld_src % 8 != 0 || !aligned16(a.src)) return false;
  if (a.dst && (a.width_dst % 128 != 0 || a.ld_dst % 8 != 0 || !aligned16(a.dst))) return false;
  if (a.ld_shrink % 8 != 0 || a.ld_expand % 8 != 0 || a.ldh % 8 != 0) return false;
  if (a.w_shrink_base && !aligned16(a.w_shrink_base)) return false;
  if (a.w_expand_base && !aligned16(a.w_expand_base)) return false;
  return true;
}

int launch_pass_mfma(const PassArgs& a, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  if (a.rpad <= 16) launch_pass<1>(a, seg, L, phases, s);
  else if (a.rpad <= 32) launch_pass<2>(a, seg, L, phases, s);
  else if (a.rpad <= 64) launch_pass<4>(a, seg, L, phases, s);
  else return launch_pass_rank128(a, seg, L, phases, s);
  return check_launch();
}

bool wgrad_mfma_supported(const WgradArgs& a) {
  if (a.width % 128 != 0 || a.ld_src % 8 != 0 || a.ldh % 8 != 0 || !aligned16(a.src) || !aligned16(a.hT)) return false;
  return true;
}

int launch_wgrad_mfma(const WgradArgs& a, const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  if (a.rpad <= 16) launch_wgrad_pipe<1, TK_WGRAD_STAGES>(a, seg, L, s);
  else if (a.rpad <= 32) launch_wgrad_coop<2>(a, seg, L, s);
  else if (a.rpad <= 64) launch_wgrad_coop<4>(a, seg, L, s);
  else return launch_wgrad_rank128(a, seg, L, s);
  return check_launch();
}

}  // namespace tk
