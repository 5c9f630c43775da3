// Kernels of the segmented LoRA pass for fp32 and for every shape the kernels of lora_kernels.h do not take (odd
// widths, strides that are no multiple of 16 bytes): any width / stride / rank <= 128, on the matrix cores, fp32
// accumulation.  They share all buffers and tables with those kernels, so the two families are interchangeable per
// launch.
//
// One body serves both types because it counts in pieces of 16 bytes, E = 8 bf16 or 4 fp32 elements.  A piece per lane
// is one operand of v_mfma_f32_16x16x32_bf16, or of four v_mfma_f32_16x16x4_f32 (exact fp32 products and sums, the
// operand components taken one after the other); either way 16 lanes are 16 rows or columns and the four lane groups
// kb = lane / 16 are consecutive pieces of the contraction index, 4 E in all.  Pieces are loaded from any element
// address (global loads need no 16-byte alignment on this part); where the width ends inside a piece its elements are
// loaded one by one, so nothing past a row's end is touched.
#include <algorithm>
#include <type_traits>

#include "tk_mfma.h"

namespace tk {

namespace {

template <typename T>
struct Piece {
  static constexpr int E = 16 / (int)sizeof(T);  // elements of a piece
};

// E consecutive elements from an address that is a multiple of the element size only
typedef u32x4_t u32x4_any __attribute__((aligned(2)));
template <typename T>
__device__ inline uint4 ld_piece(const T* p) {
  // (weights are reached through pointers read from memory: said to be global, or the loads would be flat)
  const u32x4_t v = *(const __attribute__((address_space(1))) u32x4_any*)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
// the same for data that is touched once per pass (see ld16_nt)
template <typename T>
__device__ inline uint4 ld_piece_nt(const T* p) {
  const u32x4_t v = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4_any*)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <typename T>
__device__ inline void st_piece_nt(T* p, uint4 v) {
  const u32x4_t w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, (__attribute__((address_space(1))) u32x4_any*)p);
}
// the first `keep` of them (zeros behind); nothing past them is read
template <typename T>
__device__ inline uint4 ld_piece(const T* p, int keep) {
  constexpr int E = Piece<T>::E;
  if (keep >= E) return ld_piece(p);
  uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < E; ++i)
    if (i < keep) {
      if constexpr (sizeof(T) == 4) w[i] = __builtin_bit_cast(uint32_t, p[i]);
      else w[i >> 1] |= (uint32_t)p[i] << (16 * (i & 1));
    }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// A piece cut by the end of its row, without a load per element: it is loaded as the last E elements of the row (column
// min(c, width - E)) and this drops the `drop` = c - that column elements in front, zeros behind.  drop >= E: all zeros.
// The one wave at the end of a row set the pace of its whole launch while it loaded element by element: bf16, 3001 x 1000
// and x 1500 at rank 24, shrink 10.7 -> 8.5 us, expand 15.5 -> 10.6, row contraction 20.0 -> 9.3 (means of the two widths).
// Rows, or in the expand ranks, shorter than a piece have nothing to move back into and keep the loads with a guard each.
template <typename T>
__device__ inline uint4 drop_front(const uint4& v, int drop) {
  constexpr int H = 8 / (int)sizeof(T);  // elements of half a piece
  uint64_t lo = v.x | ((uint64_t)v.y << 32), hi = v.z | ((uint64_t)v.w << 32);
  if (drop >= H) { lo = hi; hi = 0; }
  const int bits = (drop & (H - 1)) * 8 * (int)sizeof(T);
  lo = (lo >> bits) | ((hi << 1) << (63 - bits));
  hi >>= bits;
  if (drop >= 2 * H) lo = hi = 0;
  return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

__device__ inline float part_f32(const uint4& v, int i) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  return __uint_as_float(w[i]);
}

// acc += A B over the 4 E contraction indices of one piece per lane
template <typename T>
__device__ inline f32x4 mma_piece(const uint4& a, const uint4& b, f32x4 acc) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(part_f32(a, i), part_f32(b, i), acc, 0, 0, 0);
    return acc;
  } else {
    return mfma16(a, b, acc);
  }
}

// h of one tile from its sums (element (row, n) from `sum`): slot-major and rank-major copies; exact zeros in padding
// slots and at rank indices past the group's rank, so that the row contractions and the expand need no masks there
template <typename T, typename Sum>
__device__ inline void write_h(const PassArgs& a, int slot0, int cnt, int r, float sc, int n0, int nn, const Sum& sum) {
  T* hT = (T*)a.hT;
  T* hrow = hT + (int64_t)a.rpad * a.ldh;
  for (int idx = threadIdx.x; idx < kTileRows * nn; idx += 256) {
    const int row = idx / nn, n = idx % nn;
    T v;
    from_f32(row < cnt && n0 + n < r ? sum(row, n) * sc : 0.f, &v);
    hrow[(int64_t)(slot0 + row) * a.rpad + n0 + n] = v;
  }
  for (int idx = threadIdx.x; idx < kTileRows * nn; idx += 256) {
    const int row = idx & 31, n = idx >> 5;
    T v;
    from_f32(row < cnt && n0 + n < r ? sum(row, n) * sc : 0.f, &v);
    hT[(int64_t)(n0 + n) * a.ldh + slot0 + row] = v;
  }
}

// ---------------------------------------------------------------------------
// Shrink: h[slot][n] = scale_g * sum_k src[row(slot)][k] * W_g[n][k].  A block of four waves owns (tile of 32 slots,
// slice of the source columns); its waves take steps of 8 E columns (128 bytes of every row) in turn, so a slice is a
// few memory latencies long, and their sums meet in LDS.  (The form on the vector ALUs before it walked all columns in
// one block, 64 at a time behind two barriers each: 4096 rows x 4096 columns of fp32 at rank 16 took 1010 us against
// 20 + 4 for the slice sums, 3.4 TB/s; 3001 x 1000 bf16 at rank 24 390 against 13.)  With several slices (the plan of the split shrink, whose
// buffer lies behind h) the block leaves its sums for k_shrink_any_finish.
// ---------------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_shrink_any(PassArgs a, int slice_cols, const int32_t* __restrict__ tile_group,
                                                    const int32_t* __restrict__ slot_rows) {
  constexpr int E = Piece<T>::E, RP = 16 * NB;
  constexpr int NBS = NB < 4 ? NB : 4;  // rank blocks that leave through LDS together
  constexpr int PF = NB == 1 && sizeof(T) == 4 ? 4 : (NB <= 2 ? 2 : 1);  // a slice of 512 columns in one go
  __shared__ float part[4][kTileRows][16 * NBS + 1];
  const int nth = blockIdx.x / a.kslices, ks = blockIdx.x - nth * a.kslices;
  const int tile_id = checked_tile(work_item(a.wl_tiles, nth), a.tb);
  if (tile_id < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int slot0 = tile_id * kTileRows;
  const int g = checked_group(tile_group[tile_id], a.tb);
  int ra = checked_row(slot_rows[slot0 + li], a.tb), rb = checked_row(slot_rows[slot0 + 16 + li], a.tb);
  if (g < 0) return;
  const int r = class_rank(a.rank[g], a.rank_lo, RP);
  if (r <= 0) return;  // (uniform over the block, like the returns above)
  const int cnt = __popcll(__ballot(ra >= 0) & 0xffffull) + __popcll(__ballot(rb >= 0) & 0xffffull);
  const T* src = (const T*)a.src;
  const T* xr[2] = {src + (int64_t)max(ra, 0) * a.ld_src, src + (int64_t)max(rb, 0) * a.ld_src};
  const T* W = group_weight<T>(a.w_shrink, a.w_shrink_base, a.shrink_group_stride, g);
  const T* wr[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) wr[nb] = W + (int64_t)min(16 * nb + li, r - 1) * a.ld_shrink;  // (masked below)
  f32x4 acc[2][NB];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int k0 = ks * slice_cols, k1 = min(a.width_src, k0 + slice_cols);
  constexpr int STEP = 8 * E;
  int c = k0 + wave * STEP;
  // whole steps: loads of PF steps side by side, no guards
  for (; c + (PF - 1) * 4 * STEP + STEP <= k1; c += PF * 4 * STEP) {
    uint4 x[PF][2][2], w[PF][NB][2];
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int cc = c + 4 * j * STEP + 2 * E * kb;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int p = 0; p < 2; ++p) x[j][tt][p] = ld_piece(xr[tt] + cc + p * E);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int p = 0; p < 2; ++p) w[j][nb][p] = ld_piece(wr[nb] + cc + p * E);
    }
    __builtin_amdgcn_sched_barrier(0);  // (left alone the compiler pairs each load with its use, one latency each)
#pragma unroll
    for (int j = 0; j < PF; ++j)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int p = 0; p < 2; ++p) acc[tt][nb] = mma_piece<T>(x[j][tt][p], w[j][nb][p], acc[tt][nb]);
  }
  // The steps left, the last of them perhaps cut by the width (a slice ends at a whole step or there): the two pieces of
  // a lane are moved back into the row and shifted, unless a row is shorter than a piece.  One loop for both: with a loop
  // each the compiler kept a second set of accumulators, and at rank 128 one wave per SIMD where two fit (8192 x 4096 fp32
  // at rank 128, forward 294 us against 274).  Not unrolled and laid out as the rare case: fp32 at rank 96 to 112, 300 x
  // 4096, shrink 60 us otherwise, 53 so, although its whole steps never come here.
  const bool wide = a.width_src >= E;
#pragma clang loop unroll(disable)
  for (; __builtin_expect(c < k1, 0); c += 4 * STEP) {
    const int cc = c + 2 * E * kb;
    uint4 x[2][2], w[NB][2];
    if (wide) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int col = min(cc + p * E, a.width_src - E);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) x[tt][p] = ld_piece(xr[tt] + col);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) w[nb][p] = ld_piece(wr[nb] + col);
      }
    } else {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int col = cc + p * E, keep = k1 - col;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) x[tt][p] = ld_piece(xr[tt] + col, keep);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) w[nb][p] = ld_piece(wr[nb] + col, keep);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (wide && c + STEP > k1) {  // (uniform)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int drop = max(0, cc + p * E - (a.width_src - E));
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) x[tt][p] = drop_front<T>(x[tt][p], drop);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) w[nb][p] = drop_front<T>(w[nb][p], drop);
      }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) acc[tt][nb] = mma_piece<T>(x[tt][p], w[nb][p], acc[tt][nb]);
  }
  const float sc = a.scale[g];
#pragma unroll
  for (int b = 0; b < NB; b += NBS) {
    if (b) __syncthreads();
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int nb = 0; nb < NBS; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[wave][16 * tt + 4 * kb + v][16 * nb + li] = acc[tt][b + nb][v];
    __syncthreads();
    auto sum = [&](int row, int n) { return ((part[0][row][n] + part[1][row][n]) + part[2][row][n]) + part[3][row][n]; };
    if (a.kslices > 1) {
      float* mine = a.hpart + ((int64_t)tile_id * a.kslices + ks) * (kTileRows * RP) + 16 * b;
      for (int idx = tid; idx < kTileRows * 16 * NBS; idx += 256) {
        const int row = idx / (16 * NBS), n = idx % (16 * NBS);
        mine[row * RP + n] = sum(row, n);
      }
    } else {
      write_h<T>(a, slot0, cnt, r, sc, 16 * b, 16 * NBS, sum);
    }
  }
}

// Adds the slices in slice order and writes h: a block per (tile, 16 rank indices).
template <typename T>
__global__ __launch_bounds__(256) void k_shrink_any_finish(PassArgs a, const int32_t* __restrict__ tile_group,
                                                           const int32_t* __restrict__ slot_rows) {
  __shared__ float part[kTileRows][17];
  const int tile_id = checked_tile(work_item(a.wl_tiles, blockIdx.x), a.tb);
  if (tile_id < 0) return;
  const int tid = threadIdx.x, slot0 = tile_id * kTileRows, n0 = 16 * blockIdx.y;
  const int g = checked_group(tile_group[tile_id], a.tb);
  const int my_row = checked_row(slot_rows[slot0 + (tid & 31)], a.tb);
  if (g < 0) return;
  const int r = class_rank(a.rank[g], a.rank_lo, a.rpad);
  if (r <= 0) return;
  const int cnt = __popcll(__ballot(my_row >= 0) & 0xffffffffull);  // padding is at the end of a tile
  const int64_t slice = (int64_t)kTileRows * a.rpad;
  const float* p = a.hpart + (int64_t)tile_id * a.kslices * slice + n0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i, row = idx >> 4, n = idx & 15;
    const float* q = p + row * a.rpad + n;
    float s = 0.f;
    for (int k0 = 0; k0 < a.kslices; k0 += 8) {  // eight slices are requested together and added in slice order
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = k0 + k < a.kslices ? q[(k0 + k) * slice] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
    part[row][n] = s;
  }
  __syncthreads();
  write_h<T>(a, slot0, cnt, r, a.scale[g], n0, 16, [&](int row, int n) { return part[row][n]; });
}

// ---------------------------------------------------------------------------
// Expand: dst[row(slot)][c] += sum_n h[slot][n] * W_g[c][n].  A wave owns (tile, 16 E columns): column c0 + E li + q is
// output column li of the q-th product, so a lane updates E consecutive columns of eight rows, 16 bytes each, and a
// wave-wide access covers four rows of 256 bytes.  The rows are requested before the contraction starts; its operands
// (h of the tile, 16 E rows of W) come from L2.  4096 x 4096 fp32 at rank 16: 245 -> 29 us (4.6 TB/s of y).
// ---------------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_expand_any(PassArgs a, const int32_t* __restrict__ tile_group,
                                                    const int32_t* __restrict__ slot_rows,
                                                    const int32_t* __restrict__ tile_walk, int num_items) {
  constexpr int E = Piece<T>::E, RP = 16 * NB;
  constexpr int NKS = (RP + 4 * E - 1) / (4 * E);  // contraction steps
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kb = lane >> 4;
  const int ngroups = (a.width_dst + 16 * E - 1) / (16 * E);
  const int item = blockIdx.x * 4 + wave;
  if (item >= num_items) return;
  const int nth = item / ngroups;
  const int tile_id = checked_tile(a.wl_tiles.ids ? work_item(a.wl_tiles, nth) : (tile_walk ? tile_walk[nth] : nth), a.tb);
  if (tile_id < 0) return;
  const int slot0 = tile_id * kTileRows;
  const int g = checked_group(tile_group[tile_id], a.tb);
  const int4 r0 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 4 * kb);
  const int4 r1 = *reinterpret_cast<const int4*>(slot_rows + slot0 + 16 + 4 * kb);
  const int r = g < 0 ? 0 : class_rank(a.rank[g], a.rank_lo, RP);
  const int rows[2][4] = {{r0.x, r0.y, r0.z, r0.w}, {r1.x, r1.y, r1.z, r1.w}};
  const int c = (item - nth * ngroups) * (16 * E) + E * li;  // this lane's columns
  const int keep = min(E, a.width_dst - c);                  // <= 0: none
  T* dst = (T*)a.dst + c;
  if (r <= 0) {
    // no live group: zeros (several classes: launch_zero_rows), 16 bytes a lane like the results (fp32 8192 x 4096, no row
    // with an adapter: the backward takes 46 us, 82 with a store per element)
    if (a.dst_store && !a.class_mode) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = checked_row(rows[tt][v], a.tb);
          if (row < 0) continue;
          T* o = dst + (int64_t)row * a.ld_dst;
          if (keep == E) {
            st_piece_nt(o, zero4());
          } else {
            for (int q = 0; q < keep; ++q) o[q] = (T)0;
          }
        }
    }
    return;
  }
  const T* W = group_weight<T>(a.w_expand, a.w_expand_base, a.expand_group_stride, g);
  const T* h = (const T*)a.hT + (int64_t)a.rpad * a.ldh + (int64_t)slot0 * RP;
  uint4 y[2][4];
  f32x4 d[2][E];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int q = 0; q < E; ++q) d[tt][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  // 2, whole: every lane has its E columns and the rank is whole pieces, so that nothing is guarded (rows of padding
  // slots read row 0, rank indices past the rank read index 0 and are zeroed).  1, cut: the pieces at the end of the
  // width or the rank are moved back into their row and shifted, columns past the width read the last one's weights.
  // 0: a row or a rank shorter than a piece, an element at a time.
  // Cut pieces go through the caches and are shifted only where something is cut off: rows off the 16-byte pieces share
  // their lines with the items beside them (8192 x 4001 fp32 at rank 13, us: an element at a time 64, non-temporal 75, so
  // 59; bf16 71 / 56 / 46; 4096 columns, where only the rank is cut, fp32 54 / 58 / 49).
  const int back = c - min(c, a.width_dst - E);
  const bool columns = (c - E * li) + 16 * E <= a.width_dst;  // every lane has its E columns (uniform over the wave)
  auto body = [&](auto form) {
    constexpr bool whole = form == 2, cut = form == 1;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T* row = dst + (int64_t)max(checked_row(rows[tt][v], a.tb), 0) * a.ld_dst;
        y[tt][v] = a.dst_store ? zero4() : (whole ? ld_piece_nt(row) : (cut ? ld_piece(row - back) : ld_piece(row, keep)));
      }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int n0 = 4 * E * ks + E * kb;
      if (ks && 4 * E * ks >= r) break;  // (uniform over the block)
      uint4 hop[2], w[E];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) hop[tt] = n0 < RP ? ld_piece(h + (16 * tt + li) * RP + n0) : zero4();
#pragma unroll
      for (int q = 0; q < E; ++q) {
        if constexpr (whole) {
          w[q] = ld_piece(W + (int64_t)(c + q) * a.ld_expand + (n0 < r ? n0 : 0));
        } else if constexpr (cut) {
          w[q] = ld_piece(W + (int64_t)min(c + q, a.width_dst - 1) * a.ld_expand + min(n0, r - E));
        } else {
          w[q] = q < keep ? ld_piece(W + (int64_t)(c + q) * a.ld_expand + n0, r - n0) : zero4();
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < E; ++q) {
        if (whole && n0 >= r) w[q] = zero4();
        if constexpr (cut) {
          if (4 * E * (ks + 1) > r) w[q] = drop_front<T>(w[q], max(0, n0 - (r - E)));  // (uniform over the block)
        }
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) d[tt][q] = mma_piece<T>(hop[tt], w[q], d[tt][q]);
      }
    }
    if constexpr (cut) {
      if (!columns) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int v = 0; v < 4; ++v) y[tt][v] = drop_front<T>(y[tt][v], back);
      }
    }
  };
  if (columns && r % E == 0) body(std::integral_constant<int, 2>{});
  else if (a.width_dst >= E && r >= E) body(std::integral_constant<int, 1>{});
  else body(std::integral_constant<int, 0>{});
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = checked_row(rows[tt][v], a.tb);
      if (row < 0 || keep <= 0) continue;
      T* o = dst + (int64_t)row * a.ld_dst;
      T e[E];
      __builtin_memcpy(e, &y[tt][v], 16);
#pragma unroll
      for (int q = 0; q < E; ++q) from_f32(to_f32(e[q]) + d[tt][q][v], &e[q]);
      if (keep == E) {
        uint4 out;
        __builtin_memcpy(&out, e, 16);
        st_piece_nt(o, out);
      } else {
#pragma unroll
        for (int q = 0; q < E; ++q)
          if (q < keep) o[q] = e[q];
      }
    }
}

// Zeros in the rows whose group is not live, next to the expands of several rank classes that write the others instead
// of adding onto them (with one class the expand does it).  A block owns (tile, 256 pieces of 16 bytes of its rows) and
// its stores do not wait for each other.  A backward of 16384 x 4096 bf16, four rank classes and no row with an adapter:
// 87 -> 75 us (an element per thread and one row after the other before); half of the rows: 151 -> 126.
template <typename T>
__global__ __launch_bounds__(256) void k_zero_rows(T* dst, int64_t ld, int width, const int32_t* __restrict__ rank,
                                                   int max_rank, TableBounds tb, const int32_t* __restrict__ tile_group,
                                                   const int32_t* __restrict__ slot_rows) {
  constexpr int E = Piece<T>::E;
  const int g = checked_group(tile_group[blockIdx.x], tb);
  if (g >= 0 && class_rank(rank[g], 0, max_rank) > 0) return;
  const int c = (blockIdx.y * 256 + threadIdx.x) * E, keep = min(E, width - c);
#pragma unroll 8
  for (int i = 0; i < kTileRows; ++i) {
    const int row = checked_row(slot_rows[blockIdx.x * kTileRows + i], tb);
    if (row < 0) continue;
    T* o = dst + (int64_t)row * ld + c;
    if (keep == E) {
      st_piece_nt(o, zero4());
    } else {
      for (int q = 0; q < keep; ++q) o[q] = (T)0;
    }
  }
}

template <typename T>
__device__ inline void store_grad(const WgradArgs& a, int g, int n, int c, float v) {
  if (sizeof(T) != 4 && a.grad_f32) {  // fp32 gradient next to bf16 activations
    store_grad<float>(a, g, n, c, v);
    return;
  }
  T* gp = grad_of<T>(a, g);
  T* o = a.transposed ? gp + (int64_t)c * a.ld_grad + n : gp + (int64_t)n * a.ld_grad + c;
  if (a.accumulate) v += to_f32(*o);
  from_f32(v, o);
}

// ---------------------------------------------------------------------------
// Row contraction: out[n][c] = sum over the slots of a chunk of hT[n][slot] * src[row(slot)][c].  A wave owns (chunk,
// 16 E columns, 16 NB rank indices) and walks the chunk's tiles, the next tile's rows in flight while one is consumed.
// A lane loads a piece (E columns) of eight rows 8 kb .. 8 kb + 7; column c0 + E li + q is row li of the q-th product.
// In fp32 component q of the eight pieces is that product's operand as it stands (row 8 kb + i in step i); in bf16 the
// 8 x 8 block is transposed inside the lane first.  The sums leave through LDS as whole rows (16-byte
// stores of 64 separate rows instead: 36 against 25 us).  4096 x 4096 fp32 at rank 16: 81 -> 25 us.
// ---------------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_wgrad_any(WgradArgs a, const ChunkInfo* __restrict__ chunks,
                                                   const int32_t* __restrict__ slot_rows) {
  constexpr int E = Piece<T>::E, HP = 8 / E;  // pieces of a lane's eight slots of hT
  constexpr int CW = 16 * E, SS = CW + 4;  // columns of a wave, row stride of its staged sums
  __shared__ __attribute__((aligned(16))) float stage[4][16 * SS];
  extern __shared__ __attribute__((aligned(16))) int32_t rows_s[];  // the chunk's row indices
  // column blocks of one chunk are neighbours (they read neighbouring pieces of the same rows and the same h), the
  // blocks of one column range and other rank indices too (they read the same pieces)
  const int nz = a.rpad / (16 * NB), ncb = (a.width + 4 * CW - 1) / (4 * CW);
  const int z = blockIdx.x % nz, cb = (blockIdx.x / nz) % ncb;
  const int cidx = work_item(a.wl_chunks, blockIdx.x / (nz * ncb));
  if (cidx < 0) return;
  const ChunkInfo ci = checked_chunk(chunks[cidx], a.tb);
  const int g = ci.group;
  if (g < 0) return;
  const int r = class_rank(a.rank[g], a.rank_lo, a.rpad);
  const int nb0 = 16 * NB * z;  // first rank index of this block
  if (r <= nb0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int nt = ci.ntiles;
  for (int i = tid; i < nt * kTileRows; i += 256) rows_s[i] = checked_row(slot_rows[ci.tile0 * kTileRows + i], a.tb);
  __syncthreads();
  const int c0 = (cb * 4 + wave) * CW;
  if (c0 >= a.width) return;  // (no barrier follows)
  const int c = c0 + E * li;
  const int keep = min(E, a.width - c);  // <= 0: none
  // lanes past the width's last whole piece load that piece and shift it (drop_front), unless a row is shorter than one
  const bool wide = a.width >= E;
  const int drop = wide ? max(0, c - (a.width - E)) : 0;
  const T* src = (const T*)a.src + (c - drop);
  const T* hT = (const T*)a.hT + (int64_t)(nb0 + li) * a.ldh + (int64_t)ci.tile0 * kTileRows + 8 * kb;
  const bool full = c0 + CW <= a.width;  // every lane has its E columns (uniform over the wave)
  struct Tile {
    uint4 x[8], h[NB][HP];
    uint32_t live;  // bit i: row i of this lane is a real row
  };
  auto issue = [&](int t, Tile& t_) {
    const int4 ra = *reinterpret_cast<const int4*>(rows_s + t * kTileRows + 8 * kb);
    const int4 rb = *reinterpret_cast<const int4*>(rows_s + t * kTileRows + 8 * kb + 4);
    const int rows[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
    t_.live = 0;
    if (wide) {
#pragma unroll
      for (int i = 0; i < 8; ++i) t_.x[i] = ld_piece(src + (int64_t)max(rows[i], 0) * a.ld_src);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) t_.x[i] = ld_piece(src + (int64_t)max(rows[i], 0) * a.ld_src, keep);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) t_.live |= rows[i] >= 0 ? (1u << i) : 0u;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int p = 0; p < HP; ++p) t_.h[nb][p] = ld_piece(hT + (int64_t)(16 * nb) * a.ldh + t * kTileRows + E * p);
  };
  f32x4 acc[E][NB];
#pragma unroll
  for (int q = 0; q < E; ++q)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[q][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto consume = [&](Tile& t_) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!((t_.live >> i) & 1u)) t_.x[i] = zero4();
    if (!full) {
#pragma unroll
      for (int i = 0; i < 8; ++i) t_.x[i] = drop_front<T>(t_.x[i], drop);
    }
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int q = 0; q < E; ++q)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[q][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(part_f32(t_.x[i], q), part_f32(t_.h[nb][i >> 2], i & 3),
                                                             acc[q][nb], 0, 0, 0);
    } else {
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
        uint32_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t w[4] = {t_.x[i].x, t_.x[i].y, t_.x[i].z, t_.x[i].w};
          e[i] = w[q >> 1];
        }
        const uint4 tr = make_uint4(__builtin_amdgcn_perm(e[1], e[0], sel), __builtin_amdgcn_perm(e[3], e[2], sel),
                                    __builtin_amdgcn_perm(e[5], e[4], sel), __builtin_amdgcn_perm(e[7], e[6], sel));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[q][nb] = mfma16(tr, t_.h[nb][0], acc[q][nb]);
      }
    }
  };
  Tile A, B;
  if (nt > 0) issue(0, A);
  for (int t = 0; t < nt; t += 2) {
    if (t + 1 < nt) issue(t + 1, B);
    consume(A);
    if (t + 1 >= nt) break;
    if (t + 2 < nt) issue(t + 2, A);
    consume(B);
  }
  // 16 rank indices at a time through the wave's stage, [n][column], so that whole rows leave
  float* st = stage[wave];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n_first = nb0 + 16 * nb;
    if (n_first >= r) break;
    if (nb) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int q = 0; q < E; q += 4)
        *reinterpret_cast<float4*>(st + li * SS + E * (4 * kb + v) + q) =
            make_float4(acc[q][nb][v], acc[q + 1][nb][v], acc[q + 2][nb][v], acc[q + 3][nb][v]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    if (ci.partial >= 0) {  // (columns past the width lie inside the buffer's blocks of 128)
      float* p = a.partial + partial_index(ci.partial, n_first, c0, a.rpad, a.width);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int idx = lane + 64 * i, n = idx / (CW / 4), cc = 4 * (idx % (CW / 4));
        if (n_first + n < r) *reinterpret_cast<float4*>(p + n * 128 + cc) = *reinterpret_cast<const float4*>(st + n * SS + cc);
      }
    } else if (a.transposed) {
      for (int idx = lane; idx < 16 * CW; idx += 64) {
        const int cc = idx >> 4, n = idx & 15;
        if (n_first + n < r && c0 + cc < a.width) store_grad<T>(a, g, n_first + n, c0 + cc, st[n * SS + cc]);
      }
    } else {
      for (int idx = lane; idx < 16 * CW; idx += 64) {
        const int n = idx / CW, cc = idx % CW;
        if (n_first + n < r && c0 + cc < a.width) store_grad<T>(a, g, n_first + n, c0 + cc, st[n * SS + cc]);
      }
    }
  }
}

// Groups with several chunks: sum their partials in chunk order.  Groups with
// no rows: clear the live block when overwriting.  One (group, 8 rank
// indices, 256 columns) per block, a thread owns one column of the eight, so
// that a transposed gradient ([width][r], dB) leaves as 16-byte pieces instead
// of single elements; blockIdx.z >= rpad / 8 selects the second argument set,
// so that the reductions of dA and dB share one launch.
// PAIRED: chunks were taken in pairs (WgradArgs::pair_chunks), so only some slots hold sums.  A compile-time switch:
// the kernel's time is the chain from its first loads to its stores, and the slot arithmetic in that chain cost the
// unpaired launch 1 us of its 10.
template <typename T, bool PAIRED>
__device__ __forceinline__ void wgrad_reduce_body(const WgradArgs& a, int n0, const int32_t* __restrict__ chunk_first,
                                                  const int32_t* __restrict__ partial_first) {
  if (a.grad == nullptr) return;
  const int g = blockIdx.x;
  // independent loads first
  const int rk = a.rank[g], cf0 = chunk_first[g], cf1 = chunk_first[g + 1], pf = partial_first[g];
  const int r = class_rank(rk, a.rank_lo, a.rpad);
  const int nchunk = cf1 - cf0;
  // (table entries are compared with the table's bounds before they index: see TableBounds)
  if (nchunk < 0 || (nchunk > 1 && (pf < 0 || pf > a.tb.max_partials - nchunk))) return;
  if (nchunk == 1) return;
  if (nchunk == 0 && a.accumulate) return;
  // paired chunks (WgradArgs::pair_chunks): only every other slot behind the first holds a sum
  const int nlive = PAIRED && nchunk > 0 ? live_partials(nchunk, pf) : nchunk;  // (no chunks: zeros are written)
  auto slot = [&](int m) { return PAIRED ? live_partial(m, pf) : m; };
  const int64_t stride = partial_slot_floats(a.rpad, a.width);
  T* const gt = grad_of<T>(a, g);
  if (a.transposed && (a.ld_grad & (sizeof(T) == 2 ? 7 : 3)) == 0 && (reinterpret_cast<uintptr_t>(gt) & 15u) == 0 &&
      (r & 7) == 0) {
    // A transposed gradient ([width][r], dB) whose rows are whole 16-byte pieces.  With a thread per column and an
    // octet of rank indices per block every 128-byte line of it was written in up to eight partial stores from eight
    // blocks (measured at 14336 columns, rank 64: 40 of the kernel's 79 us).  Here a block owns all octets of its
    // columns: it reads the partial sums with neighbouring threads on neighbouring columns (whole lines of the
    // partial buffer), turns the sums over in LDS and writes with neighbouring threads on neighbouring octets,
    // i.e. whole rows of the gradient.  The blocks of a group are renumbered: block (y, octet z) takes the columns
    // [b cpb, b cpb + cpb), b = y * (rpad / 8) + z, cpb = 256 / octets per column.
    __shared__ __attribute__((aligned(16))) float turn[256 * 8];
    if (r == 0) return;
    int noct = 1;
    while (8 * noct < r) noct <<= 1;  // octets per column, padded to a power of two
    const int cpb = 256 / noct, tid = threadIdx.x;
    const int col0 = (blockIdx.y * (a.rpad >> 3) + (n0 >> 3)) * cpb;
    if (col0 >= a.width) return;  // (block-uniform, like every return above)
    {
      const int oct = tid / cpb, cl = tid % cpb, c = col0 + cl;
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = 0.f;
      if (c < a.width && 8 * oct < r) {
        const float* p = a.partial + partial_index(pf, 8 * oct, c, a.rpad, a.width);
        for (int j0 = 0; j0 < nlive; j0 += 2) {
          float v[2][8];
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] = j0 + j < nlive ? p[slot(j0 + j) * stride + i * 128] : 0.f;
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] += v[j][i];
        }
      }
      float4* o = reinterpret_cast<float4*>(turn + (cl * noct + oct) * 8);
      o[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
      o[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
    __syncthreads();
    const int oct = tid & (noct - 1), c = col0 + tid / noct;
    if (c >= a.width || 8 * oct >= r) return;
    const float4 lo = *reinterpret_cast<const float4*>(turn + tid * 8), hi = *reinterpret_cast<const float4*>(turn + tid * 8 + 4);
    float acc[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    if constexpr (sizeof(T) == 4) {  // fp32 gradient: the octet is two 16-byte pieces
      float4* of = reinterpret_cast<float4*>(gt + (int64_t)c * a.ld_grad + 8 * oct);
      if (a.accumulate) {
        const float4 o0 = of[0], o1 = of[1];
        acc[0] += o0.x; acc[1] += o0.y; acc[2] += o0.z; acc[3] += o0.w;
        acc[4] += o1.x; acc[5] += o1.y; acc[6] += o1.z; acc[7] += o1.w;
      }
      of[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
      of[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
      return;
    }
    uint4* o = reinterpret_cast<uint4*>(gt + (int64_t)c * a.ld_grad + 8 * oct);
    if (a.accumulate) {
      const uint4 old = *o;
      const uint32_t w[4] = {old.x, old.y, old.z, old.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] += __uint_as_float(w[i] << 16);
        acc[2 * i + 1] += __uint_as_float(w[i] & 0xffff0000u);
      }
    }
    uint16_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) from_f32(acc[i], &h[i]);
    *o = make_uint4(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16),
                    h[6] | ((uint32_t)h[7] << 16));
    return;
  }
  if (n0 >= r) return;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= a.width) return;
  const float* p = a.partial + partial_index(pf, n0, c, a.rpad, a.width);
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  // two chunks (16 loads) are requested together; every sum adds its chunks in chunk order
  for (int j0 = 0; j0 < nlive; j0 += 2) {
    float v[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[j][i] = (j0 + j < nlive && n0 + i < r) ? p[slot(j0 + j) * stride + i * 128] : 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += v[j][i];
  }
  T* gp = grad_of<T>(a, g);
  if (sizeof(T) == 2 && a.transposed && n0 + 8 <= r && (a.ld_grad & 7) == 0 &&
      (reinterpret_cast<uintptr_t>(gp) & 15u) == 0) {
    uint4* o = reinterpret_cast<uint4*>(gp + (int64_t)c * a.ld_grad + n0);
    if (a.accumulate) {
      const uint4 old = *o;
      const uint32_t w[4] = {old.x, old.y, old.z, old.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] += __uint_as_float(w[i] << 16);
        acc[2 * i + 1] += __uint_as_float(w[i] & 0xffff0000u);
      }
    }
    uint16_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) from_f32(acc[i], &h[i]);
    *o = make_uint4(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16),
                    h[6] | ((uint32_t)h[7] << 16));
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (n0 + i < r) store_grad<T>(a, g, n0 + i, c, acc[i]);
}

template <typename T>
__global__ __launch_bounds__(256) void k_wgrad_reduce(WgradArgs a0, WgradArgs a1, int rpad,
                                                      const int32_t* __restrict__ chunk_first,
                                                      const int32_t* __restrict__ partial_first) {
  const int zsets = rpad >> 3;
  const bool second = (int)blockIdx.z >= zsets;
  const WgradArgs& a = second ? a1 : a0;
  const int n0 = 8 * (second ? blockIdx.z - zsets : blockIdx.z);
  if (a.pair_chunks) wgrad_reduce_body<T, true>(a, n0, chunk_first, partial_first);
  else wgrad_reduce_body<T, false>(a, n0, chunk_first, partial_first);
}

// Any number of argument sets of one padded rank (dA and dB of several projections) in one launch:
// blockIdx.z = octets * set + octet of rank indices, octets = rpad / 8.
template <typename T>
__global__ __launch_bounds__(256) void k_wgrad_reduce_multi(WgradReduceJobs jobs, int octets,
                                                            const int32_t* __restrict__ chunk_first,
                                                            const int32_t* __restrict__ partial_first) {
  const int set = blockIdx.z / octets;
  const WgradArgs& a = jobs.a[set];
  const int n0 = 8 * (blockIdx.z - set * octets);
  if (a.pair_chunks) wgrad_reduce_body<T, true>(a, n0, chunk_first, partial_first);
  else wgrad_reduce_body<T, false>(a, n0, chunk_first, partial_first);
}

// bT_g[n][m] = B_g[m][n], aT_g[k][n] = A_g[n][k]; zero for n >= rank[g].  A block turns 64 features x rpad rank indices
// over in LDS: both the reads and the writes run along the contiguous index of their matrix (element by element along
// one of them: 71 against 31 us for four adapters of rank 128, 4096 x 4096).
// (TS: the adapters' element type, T: that of the copies; they differ for fp32 adapters under bf16 activations)
template <typename TS, typename T>
__global__ __launch_bounds__(256) void k_transpose_weights(tk_lora_desc d, int rpad, int rank_lo, T* __restrict__ bT,
                                                           T* __restrict__ aT) {
  extern __shared__ float turn_s[];  // [64][rpad + 1]
  const int g = blockIdx.y;
  const int r = class_rank(d.rank[g], rank_lo, rpad);
  if (rank_lo > 0 && r <= 0) return;  // a group of a lower rank class: no launch of this class reads its copies
  const int blocks_b = (d.out_features + 63) >> 6;
  const bool is_b = (int)blockIdx.x < blocks_b;
  const int width = is_b ? d.out_features : d.in_features;
  const int f0 = ((int)blockIdx.x - (is_b ? 0 : blocks_b)) << 6, nf = min(64, width - f0);
  const int total = 64 * rpad, shift = __ffs(rpad) - 1, ls = rpad + 1;  // rpad is a power of two
  if (is_b) {
    const TS* B = (const TS*)d.lora_B[g] + (int64_t)f0 * d.ldb;
    for (int i = threadIdx.x; i < total; i += 256) {
      const int f = i >> shift, n = i & (rpad - 1);
      turn_s[f * ls + n] = f < nf && n < r ? to_f32(B[(int64_t)f * d.ldb + n]) : 0.f;
    }
  } else {
    const TS* A = (const TS*)d.lora_A[g] + f0;
    for (int i = threadIdx.x; i < total; i += 256) {
      const int n = i >> 6, f = i & 63;
      turn_s[f * ls + n] = f < nf && n < r ? to_f32(A[(int64_t)n * d.lda + f]) : 0.f;
    }
  }
  __syncthreads();
  if (is_b) {
    T* o = bT + (int64_t)g * rpad * width + f0;
    for (int i = threadIdx.x; i < total; i += 256) {
      const int n = i >> 6, f = i & 63;
      if (f < nf) from_f32(turn_s[f * ls + n], &o[(int64_t)n * width + f]);
    }
  } else {
    T* o = aT + ((int64_t)g * width + f0) * rpad;
    for (int i = threadIdx.x; i < nf * rpad; i += 256) from_f32(turn_s[(i >> shift) * ls + (i & (rpad - 1))], &o[i]);
  }
}

// bf16 copies of fp32 adapter weights (see WeightStage): the live rows of A_g as [rpad][in_features], the live
// columns of B_g as [out_features][rpad], eight elements per thread, and the two pointer tables.  Round to
// nearest even, as a cast of the tensors would.
struct ConvertJobs {  // one job per projection (blockIdx.z); a single call has one
  tk_lora_desc d[kMaxShared];
  char* stage[kMaxShared];
  WeightStage W[kMaxShared];
  int32_t rpad[kMaxShared];
};

__global__ __launch_bounds__(256) void k_convert_weights(ConvertJobs jobs, int want_a, int want_b) {
  const tk_lora_desc& d = jobs.d[blockIdx.z];
  const WeightStage& W = jobs.W[blockIdx.z];
  char* stage = jobs.stage[blockIdx.z];
  const int rpad = jobs.rpad[blockIdx.z];
  const int g = blockIdx.y;
  if (g >= d.num_groups) return;
  bf16_t* ac = (bf16_t*)(stage + W.off_a) + (int64_t)g * W.stride_a;
  bf16_t* bc = (bf16_t*)(stage + W.off_b) + (int64_t)g * W.stride_b;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (want_a) ((const void**)(stage + W.off_ptr_a))[g] = ac;
    if (want_b) ((const void**)(stage + W.off_ptr_b))[g] = bc;
  }
  const int r = min(d.rank[g], rpad);
  const float* A = (const float*)d.lora_A[g];
  const float* B = (const float*)d.lora_B[g];
  const int k8 = (d.in_features + 7) >> 3, n8 = rpad >> 3;
  const bool vec_a = (d.lda & 3) == 0 && (reinterpret_cast<uintptr_t>(A) & 15u) == 0;
  const bool vec_b = (d.ldb & 3) == 0 && (reinterpret_cast<uintptr_t>(B) & 15u) == 0;
  const int64_t units_a = want_a ? (int64_t)r * k8 : 0;                 // (n, k-octet)
  const int64_t units_b = want_b ? (int64_t)d.out_features * n8 : 0;    // (m, n-octet)
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < units_a + units_b; u += (int64_t)gridDim.x * 256) {
    float v[8];
    bf16_t* o;
    int keep;
    if (u < units_a) {
      const int n = (int)(u / k8), k0 = (int)(u % k8) * 8;
      keep = min(8, d.in_features - k0);
      const float* src = A + (int64_t)n * d.lda + k0;
      if (vec_a && keep == 8) {
        const float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = j < keep ? src[j] : 0.f;
      }
      o = ac + (int64_t)n * d.in_features + k0;
    } else {
      const int64_t q = u - units_a;
      const int m = (int)(q / n8), n0 = (int)(q % n8) * 8;
      keep = 8;  // the copy's rows are rpad long: columns past the rank are written as zeros
      const float* src = B + (int64_t)m * d.ldb + n0;
      if (vec_b && n0 + 8 <= r) {
        const float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = n0 + j < r ? src[j] : 0.f;
      }
      o = bc + (int64_t)m * rpad + n0;
    }
    if (keep == 8 && (reinterpret_cast<uintptr_t>(o) & 15u) == 0) {  // one 16-byte store
      uint16_t h[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) from_f32(v[j], &h[j]);
      *reinterpret_cast<uint4*>(o) = make_uint4(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16),
                                                h[4] | ((uint32_t)h[5] << 16), h[6] | ((uint32_t)h[7] << 16));
      continue;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < keep) from_f32(v[j], &o[j]);
  }
}

}  // namespace

int launch_convert_weights_multi(const tk_lora_desc* const* d, void* const* stage, int n, bool want_a, bool want_b,
                                 hipStream_t s) {
  if (n < 1 || n > kMaxShared) return TK_ERR_INVALID;
  ConvertJobs J{};
  int64_t per_group = 0;
  int groups = 0;
  for (int p = 0; p < n; ++p) {
    const int rpad = rank_pad(d[p]->max_rank);
    J.d[p] = *d[p];
    J.stage[p] = (char*)stage[p];
    J.W[p] = WeightStage(d[p]->num_groups, rpad, d[p]->in_features, d[p]->out_features);
    J.rpad[p] = rpad;
    per_group = std::max(per_group, (int64_t)rpad * (d[p]->in_features / 8 + 1) + (int64_t)d[p]->out_features * (rpad / 8));
    groups = std::max(groups, d[p]->num_groups);
  }
  const dim3 grid((unsigned)std::min<int64_t>(ceil_div(per_group, 512), 64), (unsigned)groups, (unsigned)n);
  hipLaunchKernelGGL(k_convert_weights, grid, dim3(256), 0, s, J, want_a ? 1 : 0, want_b ? 1 : 0);
  return check_launch();
}

int launch_convert_weights(const tk_lora_desc& d, void* stage, bool want_a, bool want_b, hipStream_t s) {
  const tk_lora_desc* dp = &d;
  return launch_convert_weights_multi(&dp, &stage, 1, want_a, want_b, s);
}

namespace {

template <typename T, int NB>
void launch_pass_any(const PassArgs& a0, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  constexpr int E = Piece<T>::E;
  // Up to three slices of at most 1536 columns: one block per tile walks them all where its steps cost less than the
  // launch that adds the slices and their way through memory.  Many tiles always: (one block / slices, us) fp32 8192 x 1536
  // rank 8 25 / 29, rank 128 68 / 83; bf16 32768 x 1000 rank 128 101 / 130.  Few tiles leave the chip idle meanwhile, so
  // there by the length of the steps, which grows with width and rank and is longer in fp32 (an eighth of the products per
  // instruction): fp32 512 x 1024 rank 8 16.1 / 16.8, 512 x 1536 rank 32 23.6 / 21.3 and at 3072 rows 26.1 / 27.8; 2048 x 1536
  // rank 64 37.6 / 28.9, rank 128 60.4 / 43.1, 4096 x 1024 rank 128 51.5 / 47.0; bf16 2048 x 1500 rank 32 22.7 / 24.2, rank
  // 64 equal, 1024 x 1500 rank 128 40.0 / 35.5.  (fp32 512 x 1536 rank 8: 18.5 / 17.0 on the GPU, but a launch less of an eager
  // pass that the host sets the pace of: 387 rows of 18 adapters 34 / 37.)
  PassArgs a = a0;
  if (a.kslices <= 3 && a.width_src <= 1536) {
    const int64_t tiles = L.live_tiles();
    const bool some = tiles >= 96;
    const bool one = tiles >= 192 || (sizeof(T) == 4 ? NB == 1 || (NB == 2 && (a.width_src <= 1280 || some)) : NB <= 4 || some);
    if (one) a.kslices = 1;
  }
  const int32_t* rows = seg.slot_table(a.map_rows);
  if (phases & 1) {
    // the slices of the split shrink's plan (its buffer holds kslices slices of every tile)
    const int slice_cols = (int)round_up(ceil_div(a.width_src, a.kslices), 8 * E);
    hipLaunchKernelGGL((k_shrink_any<T, NB>), dim3((unsigned)(L.max_tiles * a.kslices)), dim3(256), 0, s, a, slice_cols,
                       seg.tile_group, rows);
    if (a.kslices > 1)
      hipLaunchKernelGGL(k_shrink_any_finish<T>, dim3((unsigned)L.max_tiles, NB), dim3(256), 0, s, a, seg.tile_group,
                         rows);
  }
  if (a.dst && (phases & 2)) {
    const int64_t items = L.max_tiles * ceil_div(a.width_dst, 16 * E);
    hipLaunchKernelGGL((k_expand_any<T, NB>), dim3((unsigned)ceil_div(items, 4)), dim3(256), 0, s, a, seg.tile_group,
                       rows, seg.tile_walk(a.map_rows), (int)items);
  }
}

template <typename T>
void launch_pass_any(const PassArgs& a, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  if (a.rpad <= 16) launch_pass_any<T, 1>(a, seg, L, phases, s);
  else if (a.rpad <= 32) launch_pass_any<T, 2>(a, seg, L, phases, s);
  else if (a.rpad <= 64) launch_pass_any<T, 4>(a, seg, L, phases, s);
  else launch_pass_any<T, 8>(a, seg, L, phases, s);
}

template <typename T>
void launch_wgrad_any(const WgradArgs& a, const SegView& seg, const SegLayout& L, hipStream_t s) {
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t);
  // at most 32 rank indices per block: with 64 the accumulators leave one wave per SIMD (bf16: and spill)
  const int nb = a.rpad <= 16 ? 1 : 2;
  const dim3 grid((unsigned)(a.rpad / (16 * nb) * ceil_div(a.width, 64 * Piece<T>::E) * L.max_chunks));
  const auto kernel = nb == 1 ? k_wgrad_any<T, 1> : k_wgrad_any<T, 2>;
  hipLaunchKernelGGL(kernel, grid, dim3(256), dyn, s, a, seg.chunks, seg.slot_table(a.map_rows));
}

}  // namespace

int launch_pass_generic(const PassArgs& a, const SegView& seg, const SegLayout& L, int dtype, int phases,
                        hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  if (dtype == TK_DTYPE_F32) launch_pass_any<float>(a, seg, L, phases, s);
  else launch_pass_any<bf16_t>(a, seg, L, phases, s);
  return check_launch();
}

int launch_zero_rows(void* dst, int64_t ld, int width, int dtype, const int32_t* rank, int max_rank, int map_rows,
                     const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  const dim3 grid((unsigned)L.max_tiles, (unsigned)ceil_div(width, 256 * (dtype == TK_DTYPE_F32 ? 4 : 8)));
  const int32_t* rows = seg.slot_table(map_rows);
  if (dtype == TK_DTYPE_F32)
    hipLaunchKernelGGL(k_zero_rows<float>, grid, dim3(256), 0, s, (float*)dst, ld, width, rank, max_rank,
                       table_bounds(L), seg.tile_group, rows);
  else
    hipLaunchKernelGGL(k_zero_rows<bf16_t>, grid, dim3(256), 0, s, (bf16_t*)dst, ld, width, rank, max_rank,
                       table_bounds(L), seg.tile_group, rows);
  return check_launch();
}

int launch_wgrad_generic(const WgradArgs& a, const SegView& seg, const SegLayout& L, int dtype, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  if (dtype == TK_DTYPE_F32) launch_wgrad_any<float>(a, seg, L, s);
  else launch_wgrad_any<bf16_t>(a, seg, L, s);
  return check_launch();
}

int launch_wgrad_reduce(const WgradArgs* a0, const WgradArgs* a1, const SegView& seg, const SegLayout& L, int dtype,
                        hipStream_t s) {
  if (L.groups == 0 || (!a0 && !a1)) return TK_OK;
  WgradArgs none{};
  const WgradArgs& x0 = a0 ? *a0 : none;
  const WgradArgs& x1 = a1 ? *a1 : none;
  const int rpad = a0 ? a0->rpad : a1->rpad;
  const int width = std::max(a0 ? a0->width : 0, a1 ? a1->width : 0);
  const dim3 grid((unsigned)L.groups, (unsigned)ceil_div(width, 256), (unsigned)(a1 ? 2 * (rpad / 8) : rpad / 8));
  if (dtype == TK_DTYPE_F32 || x0.grad_f32 || x1.grad_f32)  // (both sets have the gradient type of their descriptor)
    hipLaunchKernelGGL(k_wgrad_reduce<float>, grid, dim3(256), 0, s, x0, x1, rpad, seg.chunk_first, seg.partial_first);
  else
    hipLaunchKernelGGL(k_wgrad_reduce<bf16_t>, grid, dim3(256), 0, s, x0, x1, rpad, seg.chunk_first,
                       seg.partial_first);
  return check_launch();
}

int launch_wgrad_reduce_multi(const WgradArgs* sets, int n, const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.groups == 0 || n == 0) return TK_OK;
  WgradReduceJobs J{};
  J.n = n;
  int width = 0;
  for (int i = 0; i < n; ++i) {
    J.a[i] = sets[i];
    width = std::max(width, sets[i].width);
  }
  const int octets = sets[0].rpad / 8;  // the sets share their padded rank
  const dim3 grid((unsigned)L.groups, (unsigned)ceil_div(width, 256), (unsigned)(octets * n));
  if (sets[0].grad_f32)  // fp32 adapters under bf16 activations (all sets of a call alike)
    hipLaunchKernelGGL(k_wgrad_reduce_multi<float>, grid, dim3(256), 0, s, J, octets, seg.chunk_first,
                       seg.partial_first);
  else
    hipLaunchKernelGGL(k_wgrad_reduce_multi<bf16_t>, grid, dim3(256), 0, s, J, octets, seg.chunk_first,
                       seg.partial_first);
  return check_launch();
}

int launch_transpose_weights(const tk_lora_desc& d, int rank_lo, void* bT, void* aT, hipStream_t s) {
  if (d.num_groups == 0) return TK_OK;
  const int rpad = rank_pad(d.max_rank);
  const dim3 grid((unsigned)(ceil_div(d.out_features, 64) + ceil_div(d.in_features, 64)), (unsigned)d.num_groups);
  const size_t lds = sizeof(float) * 64 * (size_t)(rpad + 1);
  if (d.dtype == TK_DTYPE_F32)
    hipLaunchKernelGGL((k_transpose_weights<float, float>), grid, dim3(256), lds, s, d, rpad, rank_lo, (float*)bT,
                       (float*)aT);
  else if (mixed_weights(d))
    hipLaunchKernelGGL((k_transpose_weights<float, bf16_t>), grid, dim3(256), lds, s, d, rpad, rank_lo,
                       (bf16_t*)bT, (bf16_t*)aT);
  else
    hipLaunchKernelGGL((k_transpose_weights<bf16_t, bf16_t>), grid, dim3(256), lds, s, d, rpad, rank_lo, (bf16_t*)bT,
                       (bf16_t*)aT);
  return check_launch();
}

}  // namespace tk
