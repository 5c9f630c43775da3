// Grouped base GEMM of packed experts with the LoRA term in its epilogue (gfx950, bf16 MFMA).
//
//   y[row(slot)][n] = sum_k x[row(slot)][k] * W_e[n][k]  (+ sum_r h[slot][r] * B_g[n][r])
//
// for every slot of the segment table, e = g / groups_per_weight the weight (expert) of the slot's group g.
// One launch serves all experts: the reference loops over the experts on the host and synchronises for each
// chunk boundary.  The LoRA term enters as extra contraction steps on the accumulators, so y is written once
// instead of written by the GEMM and then read, updated and written again by the expand kernel.
//
//   k_grouped_plan      the list of row blocks (up to 4 or 8 consecutive tiles of one expert, an expert's tiles cut into
//                       blocks of equal length)
//   k_grouped_gemm_dl   out_features a multiple of 256 and operands under 4 GB: block tile 256 x 256 x 64, eight
//                       waves, the operand tiles loaded from global memory straight into LDS (both weight layouts,
//                       with and without the LoRA term); described where it is defined
//   k_grouped_gemm      the rest: operands through registers into LDS; 8 waves on 256 x 256 tiles or 4 waves on
//                       128 x 128 (row stride 144 B in LDS: conflict-free 16-byte operand reads, a wave owns
//                       64 x 64 as 4 x 4 MFMA 16x16x32 tiles)
//
// A work item is one row block and one column block (k_grouped_gemm: a run of them) of the output: the row block's x stays
// in L2 across the column blocks, and the row blocks of one expert, which reach an XCD together, stream that expert's
// weights through the XCD's L2 side by side.  The weight fragment is the MFMA A operand and the x fragment the B operand, so
// a lane ends up with four consecutive output columns of one row.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "tk_mfma.h"

namespace tk {

namespace {

constexpr int kGBK = 64, kGLS = kGBK + 8;
#ifndef TK_GROUPED_ITEMS
#define TK_GROUPED_ITEMS 6144
#endif
#ifndef TK_GROUPED_BIG
#define TK_GROUPED_BIG 1
#endif
#ifndef TK_GROUPED_DL
#define TK_GROUPED_DL 1  // 8 waves, 256 x 256 tiles: operand tiles go from global memory straight into LDS
#endif
constexpr int kGroupedItems = TK_GROUPED_ITEMS;  // work items aimed at per launch
constexpr int kGroupedBlocks = 256;  // blocks of k_grouped_gemm_dl: one per CU

// One entry per row block, with everything the GEMM would otherwise look up through chains of dependent loads: rows and
// live rows of its tiles and the groups they belong to.  Every block makes the (short) scan over the experts, a block then
// fills its kPlanBlock entries.
constexpr int kPlanBlock = 32;

__global__ __launch_bounds__(256) void k_grouped_plan(GroupedArgs a, SegView V, int experts, int nt,
                                                      GroupedPlanEntry* __restrict__ plan,
                                                      int32_t* __restrict__ nblocks, int max_entries, int ptiles) {
  __shared__ int32_t sums[4];
  __shared__ GroupedPlanEntry mine[kPlanBlock];
  const int tid = threadIdx.x, base = blockIdx.x * kPlanBlock;
  const int per = (experts + 255) / 256;
  const int e0 = min(experts, tid * per), e1 = min(experts, e0 + per);
  int cnt = 0;
  // (tile numbers come from the caller's segment table: kept inside [0, max_tiles] and ascending before they index)
  auto first_tile = [&](int g) { return min(max(V.tile_first[g], 0), a.tb.max_tiles); };
  for (int e = e0; e < e1; ++e) cnt += (max(first_tile((e + 1) * nt) - first_tile(e * nt), 0) + ptiles - 1) / ptiles;
  int upto = cnt;  // inclusive scan over the block
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(upto, off, 64);
    if ((tid & 63) >= off) upto += v;
  }
  if ((tid & 63) == 63) sums[tid >> 6] = upto;
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < tid >> 6) upto += sums[w];
    total += sums[w];
  }
  total = min(total, max_entries);
  int at = upto - cnt;
  for (int e = e0; e < e1; ++e) {
    const int t0 = first_tile(e * nt), t1 = max(first_tile((e + 1) * nt), t0);
    // the expert's tiles in `count` row blocks of (almost) equal length: blocks of equal work stay in step, and
    // blocks in step find each other's weight and x tiles in the XCD's L2 (measured at config 4, 18 tiles per expert:
    // as 8 + 8 + 2 the short block runs ahead and L2 fetches 1.6 x the compulsory bytes, as 6 + 6 + 6 it fetches
    // 1.2 x)
    const int first = at, count = (t1 - t0 + ptiles - 1) / ptiles;
    const int per = count > 0 ? (t1 - t0 + count - 1) / count : ptiles;
    for (int t = t0; t < t1; t += per, ++at) {
      const int i = at - base;
      if (i < 0 || i >= kPlanBlock) continue;
      mine[i].tile0 = t;
      mine[i].ntiles = min(per, t1 - t);
      mine[i].expert = e;
      mine[i].first = first;
      mine[i].count = count;
    }
  }
  if (tid == 255 && blockIdx.x == 0) *nblocks = total;
  if (tid < 8 && blockIdx.x == 0) nblocks[8 + tid] = 0;  // k_grouped_gemm_dl: items drawn by each XCD
  __syncthreads();
  if (base >= total) return;
  // thread = (entry, tile of the entry): group, first position and live rows of the tile; the distinct groups of a block
  // that carry a LoRA term are numbered in the order of its tiles (the eight threads of an entry are neighbours in a wave)
  const int i = tid >> 3, t = tid & 7;
  const bool entry = base + i < total;
  GroupedPlanEntry& m = mine[i];
  const bool have = entry && t < m.ntiles;
  const int tile = have ? m.tile0 + t : 0;  // (tile0 + ntiles <= max_tiles)
  const int g = have ? checked_group(V.tile_group[tile], a.tb) : -1;
  const int row0 = have ? V.slot_pos[(int64_t)tile * kTileRows] : 0;
  const int end = g >= 0 ? V.offsets[g + 1] : 0;
  const int pos = min(max(row0, 0), a.tb.rows - 1);
  const bool lora = g >= 0 && a.rpad > 0 && a.rank[g] > 0;
  const int before = __shfl_up(lora ? g : -1, 1, 8);  // the tile in front of this one
  const bool opens = lora && (t == 0 || before != g);
  const unsigned mask = (unsigned)(__ballot(opens) >> (threadIdx.x & 56)) & 0xffu;
  const int number = __popc(mask & ((2u << t) - 1u)) - 1;
  if (entry) {
    m.pos[t] = pos;
    m.cnt[t] = row0 >= 0 ? min(max(min(end, a.tb.rows) - pos, 0), kTileRows) : 0;
    m.number[t] = lora ? number : -1;
    if (opens) {
      m.rank[number] = min(a.rank[g], a.rpad);
      m.matrix[number] = (const bf16_t*)a.lora_B[g];
    }
    if (t == 0) m.ngroups = __popc(mask);
  }
  // An entry's eight threads wrote it and now move it out together: a block barrier, which orders the LDS accesses of
  // different threads (a wave barrier does not), and words copied as bytes (the entry holds pointers, and a load of another
  // type may move ahead of their stores).
  __syncthreads();
  if (!entry) return;
  constexpr int kWords = sizeof(GroupedPlanEntry) / 4;
  const char* from = reinterpret_cast<const char*>(&m);
  char* to = reinterpret_cast<char*>(&plan[base + i]);
  for (int w = t; w < kWords; w += 8) {
    int32_t word;
    __builtin_memcpy(&word, from + 4 * w, 4);
    __builtin_memcpy(to + 4 * w, &word, 4);
  }
}

// NKS: MFMA steps of the LoRA term (0: none; 1: padded rank 16 or 32; 2: padded rank 64)
// BIG: 0: 4 waves (2 x 2), wave tile 64 x 64, block tile 128 x 128, two blocks per CU, loads two steps ahead;
//      1: 8 waves (2 x 4), wave tile 128 x 64, block tile 256 x 256, one block per CU: half the operand bytes per
//         FLOP out of L2 and three LDS reads per eight MFMAs instead of four; a wave whose rows are dead (the tail
//         of an expert) skips its MFMAs, so a half-empty block takes about half the time
// TR:  0: weight rows are output features (y = x W^T, the contraction runs along the weight's rows in memory);
//      1: weight rows are input features (y = x W: the backward of TR = 0 on the same memory).  The lower half of
//         the block then loads the weight tile as 8 x 8 blocks, transposes them in registers and writes them to LDS
//         with the 16-byte chunks of a row XOR-swizzled by the row's block number (conflict-free on both sides);
//         the upper half loads the x tile.
template <int NKS, int BIG, int TR>
__global__ __launch_bounds__(BIG ? 512 : 256) __attribute__((amdgpu_waves_per_eu(2))) void k_grouped_gemm(
    GroupedArgs a, const GroupedPlanEntry* __restrict__ plan, const int32_t* __restrict__ nblocks,
    const int32_t* __restrict__ tile_group, const int32_t* __restrict__ slot_rows, const int32_t* __restrict__ y_rows,
    int nsplit, int cpi) {
  constexpr int THREADS = BIG ? 512 : 256, WN = BIG ? 4 : 2, RB = BIG ? 8 : 4, CB = 4;
  constexpr int BM = 2 * 16 * RB, BN = WN * 16 * CB;  // 128 x 128 or 256 x 256
  constexpr int LROWS = THREADS / 8;                   // rows moved per pass of the block's loads
  constexpr int XP = BM / LROWS, WP = BN / LROWS;      // passes: 4 and 4
  constexpr int SETS = (BIG || TR) ? 1 : 2;            // register sets of loads in flight
  __shared__ __attribute__((aligned(16))) bf16_t As[2][BM * kGLS];  // x rows
  __shared__ __attribute__((aligned(16))) bf16_t Bs[2][BN * kGLS];  // weight rows
  // work item = (row block, run of cpi column blocks); the items of one expert are neighbours and reach one XCD
  // together
  const int blocks = *nblocks * nsplit;
  if ((int)blockIdx.x >= blocks) return;
  const int item = xcd_contiguous(blockIdx.x, blocks);
  // within an expert: column run major, row block minor, so that the blocks that read the same weight rows start
  // side by side (the expert's entries are contiguous: any of them names the range)
  const GroupedPlanEntry any = plan[item / nsplit];
  const int local = item - any.first * nsplit;
  const GroupedPlanEntry pe = plan[any.first + local % any.count];
  const int nb_first = (local / any.count) * cpi, nb_last = min(nb_first + cpi, a.N / BN);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int slot0 = pe.tile0 * kTileRows, live = pe.ntiles * kTileRows;
  const int live_w = min(max(live - 16 * RB * wm, 0), 16 * RB);  // live rows of this wave's strip (uniform)

  // global -> LDS (TR = 0): thread t moves 16 bytes of rows (t >> 3) + LROWS i at column chunk t & 7, of x and of
  // the weights alike.  (TR = 1): the upper half of the threads does that for x alone (XR rows per pass, 8 passes),
  // the lower half owns one 8 x 8 block of the weight tile each.
  constexpr int XR = TR ? THREADS / 16 : LROWS, XN = TR ? 8 : XP;
  const bool w_thread = TR && tid < THREADS / 2;           // uniform over a wave
  const int xt = TR ? (tid & (THREADS / 2 - 1)) : tid;
  const int lrow = xt >> 3, lchunk = (xt & 7) * 8;
  const bf16_t* xp[XN];
#pragma unroll
  for (int i = 0; i < XN; ++i) {
    const int r = lrow + XR * i;
    int row = r < live ? slot_rows[slot0 + r] : -1;  // padding and dead rows read row 0 and are never stored
    row = min(max(row, 0), a.src_rows - 1);
    xp[i] = a.x + (int64_t)row * a.ldx + lchunk;
  }
  const int cblk = tid / (BN / 8), jblk = tid % (BN / 8);  // TR: this thread's block of the weight tile
  // rows this lane stores: slots 16 RB wm + 16 rb + li
  int out_row[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = 16 * RB * wm + 16 * rb + li;
    out_row[rb] = r < live ? checked_row(y_rows[slot0 + r], a.tb) : -1;
  }
  const bf16_t* wbase = a.w + (int64_t)pe.expert * a.w_stride;
  const int nk = a.K / kGBK;
  const int ldsw = lrow * kGLS + lchunk;  // + LROWS i rows

  for (int nb = nb_first; nb < nb_last; ++nb) {
    const bf16_t* wp[TR ? 1 : WP];
    if constexpr (TR) {
      wp[0] = wbase + (int64_t)(8 * cblk) * a.ldw + nb * BN + 8 * jblk;
    } else {
#pragma unroll
      for (int i = 0; i < WP; ++i) wp[i] = wbase + (int64_t)(nb * BN + lrow + LROWS * i) * a.ldw + lchunk;
    }
    f32x4 acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // The loads of step ks + SETS are issued before step ks is computed and wait in registers across the barrier
    // (which orders LDS traffic only).
    uint4 gx[SETS][TR ? 8 : XP], gw[SETS][TR ? 1 : WP];  // TR: gx holds a thread's eight pieces of either tile
    auto fetch = [&](int ks, auto set) {
      const int k0 = ks * kGBK;
      if constexpr (TR) {
        if (w_thread) {
          const bf16_t* p = wp[0] + (int64_t)k0 * a.ldw;
#pragma unroll
          for (int i = 0; i < 8; ++i) gx[set][i] = ld16(p + (int64_t)i * a.ldw);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) gx[set][i] = ld16(xp[i] + k0);
        }
      } else {
#pragma unroll
        for (int i = 0; i < XP; ++i) gx[set][i] = ld16(xp[i] + k0);
#pragma unroll
        for (int i = 0; i < WP; ++i) gw[set][i] = ld16(wp[i] + k0);
      }
    };
    auto stash = [&](int buf, auto set) {
      if constexpr (TR) {
        if (w_thread) {
          // 8 x 8 transpose inside the thread: piece q becomes column q of the block, the eight contraction indices
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int d = q >> 1;
            const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
            uint32_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const uint32_t wsrc[4] = {gx[set][i].x, gx[set][i].y, gx[set][i].z, gx[set][i].w};
              e[i] = wsrc[d];
            }
            uint4 tr;
            tr.x = __builtin_amdgcn_perm(e[1], e[0], sel);
            tr.y = __builtin_amdgcn_perm(e[3], e[2], sel);
            tr.z = __builtin_amdgcn_perm(e[5], e[4], sel);
            tr.w = __builtin_amdgcn_perm(e[7], e[6], sel);
            st16(&Bs[buf][(8 * jblk + q) * kGLS + 8 * (cblk ^ (jblk & 7))], tr);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) st16(&As[buf][ldsw + XR * i * kGLS], gx[set][i]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < XP; ++i) st16(&As[buf][ldsw + LROWS * i * kGLS], gx[set][i]);
#pragma unroll
        for (int i = 0; i < WP; ++i) st16(&Bs[buf][ldsw + LROWS * i * kGLS], gw[set][i]);
      }
    };
    auto step = [&](int ks, auto parity) {  // parity = ks & 1 as a compile-time constant
      constexpr int cur = decltype(parity)::value;
      if (ks + SETS < nk) fetch(ks + SETS, std::integral_constant<int, SETS == 2 ? cur : 0>{});
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 fw[CB];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const int j = 16 * CB * wn + 16 * cb + li;
          const int chunk = TR ? ((4 * s + kb) ^ ((j >> 3) & 7)) : 4 * s + kb;
          fw[cb] = ld16(&Bs[cur][j * kGLS + 8 * chunk]);
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          if (16 * rb >= live_w) break;
          const uint4 fx = ld16(&As[cur][(16 * RB * wm + 16 * rb + li) * kGLS + 32 * s + 8 * kb]);
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma16(fw[cb], fx, acc[rb][cb]);
        }
      }
      if (ks + 1 < nk) stash(cur ^ 1, std::integral_constant<int, SETS == 2 ? (cur ^ 1) : 0>{});
      lds_barrier();
    };
    fetch(0, std::integral_constant<int, 0>{});
    if (SETS == 2 && nk > 1) fetch(1, std::integral_constant<int, SETS - 1>{});
    stash(0, std::integral_constant<int, 0>{});
    lds_barrier();
    for (int ks = 0; ks < nk; ks += 2) {
      step(ks, std::integral_constant<int, 0>{});
      if (ks + 1 < nk) step(ks + 1, std::integral_constant<int, 1>{});
    }

    if constexpr (NKS > 0) {
      // LoRA term: h[slot][0 .. rpad) against B_g[n][0 .. rank), per 32-row tile (a tile has one group)
#pragma unroll
      for (int tl = 0; tl < RB / 2; ++tl) {
        const int tile_in_block = (RB / 2) * wm + tl;
        if (tile_in_block >= pe.ntiles) break;
        const int g = checked_group(tile_group[pe.tile0 + tile_in_block], a.tb);
        const int r = g >= 0 ? min(a.rank[g], a.rpad) : 0;
        if (r <= 0) continue;
        const bf16_t* Bg = (const bf16_t*)a.lora_B[g];
#pragma unroll
        for (int s = 0; s < NKS; ++s) {
          const int n0 = 32 * s + 8 * kb;  // first rank index of this lane's operand piece
          if (32 * s >= r) break;          // uniform over the wave
          uint4 fh[2], fb[CB];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int slot = slot0 + 32 * tile_in_block + 16 * q + li;
            fh[q] = n0 < a.rpad ? ld16(a.hrow + (int64_t)slot * a.rpad + n0) : zero4();
          }
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) {
            const int n = nb * BN + 16 * CB * wn + 16 * cb + li;
            fb[cb] = n0 < r ? keep_first(ld16(Bg + (int64_t)n * a.ldb + n0), r - n0) : zero4();
          }
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) acc[2 * tl + q][cb] = mfma16(fb[cb], fh[q], acc[2 * tl + q][cb]);
        }
      }
    }

    // lane holds y[slot 16 RB wm + 16 rb + li][nb BN + 16 CB wn + 16 cb + 4 kb + v], v = 0..3: 8-byte stores
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (out_row[rb] < 0) continue;
      bf16_t* yp = a.y + (int64_t)out_row[rb] * a.ldy + nb * BN + 16 * CB * wn + 4 * kb;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const f32x4 v = acc[rb][cb];
        *reinterpret_cast<uint2*>(yp + 16 * cb) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same product with the operand tiles going from global memory straight into LDS (global_load_lds, 16 bytes per
// lane): no staging registers and no LDS stores, so the wave has room for all operand fragments of a 32-deep half
// step (12 x 16 bytes per lane) and reads them ahead of the MFMAs that use them.  Block tile 256 x 256 x 64, eight
// waves (2 x 4), wave tile 128 x 64, two stages of 32 KB for x and three for the weights: one block fills a CU's LDS, so
// there is one block per CU and it walks its share of the work items (persistent).
//
// Stage layout: x rows and weight rows alike, row r of the tile at byte 128 r, its 16-byte chunk c at position
// c ^ (r & 7).  A wave-wide load brings eight rows: lane L lands at byte 16 L of the wave's 1 KB window (the
// hardware's rule), i.e. row L >> 3, position L & 7, so it fetches chunk (L & 7) ^ (L >> 3) of that row: eight
// neighbouring lanes cover one whole 128-byte line of global memory.  An operand read (lane = row li, chunk
// 4 s + kb) goes to position (4 s + kb) ^ (li & 7): the eight lanes of one pass hit eight different 16-byte bank
// groups.  Row offsets are 32-bit (the launcher checks that x and one expert's weights span less than 4 GB).
//
// Per 64-deep step: 24 operand reads, 8 requests of coming tiles and 64 MFMAs per wave, one block barrier in the middle.
// What bounds it: an 8-wave block alternates between LDS and the matrix cores, which a step needs about equally long (160 KB
// of operands at 128 B a clock, 1536 clocks of MFMAs), and 35 % of a wave's time goes into waits at the barrier.  Requests
// and operand reads in one burst behind the barrier held the MFMAs behind them back; spread between them they do not.
// 65536 rows of 128 experts in 512 groups, us a launch, before (one block per item, bursts, LoRA term behind the products
// with a chain of four dependent loads per tile, 8-byte stores) and now:
//   2048 -> 1536 with the LoRA term 558 / 479, 768 -> 2048 with it 404 / 346; transposing 2048 -> 768 288 / 271, 1536 -> 2048
//   549 / 493
// Of these, the same tile requested over and over (every load a hit in L2) takes 75 us off, results not stored 40 to 90.
//
// The LoRA term is one more step (or more): 64 / R groups of a row block's tiles at a time (R = padded rank), h of the
// block's slots as the x tile, the groups' B (TR: A) as the weight tile, both loaded like the other tiles while the
// products before them run.  A tile multiplies with the piece of its own group only, picked out of the weight tile, so
// what another tenant's adapter holds (infinities, NaN) never meets its rows.
// ---------------------------------------------------------------------------
// 64 bits per lane from LDS, transposed among 16 lanes (ds_read_b64_tr_b16): with M[p][e] the four 16-bit elements
// e that lane p of a group of 16 points at, lane l receives M[4 e + (l >> 2)][l & 3], e = 0..3.
__device__ __forceinline__ uint2 lds_read_transposed(const char* p) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)p);
  return __builtin_bit_cast(uint2, v);
}

// `v`, which is not computed ahead of where it is used: what the compiler would derive from it once and keep in registers
// through the products is derived again where it is needed.
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// TR = 1: the weight rows are input features (y = x W, the backward of TR = 0 on the same memory).  The weight
// tile of a step is then 64 rows of 256 outputs, 512 bytes a row, and lies in LDS as it lies in memory (a wave-wide
// load brings two rows; the 16-byte chunk c of row r at position c ^ ((r & 3) << 1)).  The MFMA operand, eight
// consecutive contraction indices of one output, is a column of that tile: two transposing LDS reads fetch it, each
// from four rows (which the swizzle puts on different banks) of 16 outputs.
// REM: steps of the contraction mod 6 (the loop is unrolled six times: with the rest known the compiler follows which stage
// every load in flight goes to; with the rest in run-time branches it waits for all of them)
template <int TR, int REM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_grouped_gemm_dl(
    GroupedArgs a, const GroupedPlanEntry* __restrict__ plan, const int32_t* __restrict__ nblocks,
    int32_t* __restrict__ tickets, const int32_t* __restrict__ slot_rows, int ncb) {
  constexpr int WN = 4, RB = 8, CB = 4, BM = 256, BN = 256, WP = 4;  // WP: weight loads of a wave per step
  __shared__ __attribute__((aligned(1024))) bf16_t As0[BM * kGBK];
  __shared__ __attribute__((aligned(1024))) bf16_t As1[BM * kGBK];
  __shared__ __attribute__((aligned(1024))) bf16_t Bs0[BN * kGBK];
  __shared__ __attribute__((aligned(1024))) bf16_t Bs1[BN * kGBK];
  __shared__ __attribute__((aligned(1024))) bf16_t Bs2[BN * kGBK];
  const int entries = *nblocks, items = entries * ncb;
  // Each XCD has its own eighth of the items.  A block's first two are given, the others it draws from its XCD's counter:
  // items differ by the tiles they hold (dealt out evenly, a CU waited a sixth of the launch for the busiest one).
  const int xcd = blockIdx.x & 7, peers = (int)gridDim.x >> 3;
  auto item_of = [&](int k) __attribute__((always_inline)) {  // the XCD's k-th, -1 past its last
    const int per = items >> 3;
    return k < per ? xcd * per + k : k == per && xcd < (items & 7) ? 8 * per + xcd : -1;
  };
  int it = item_of(blockIdx.x >> 3), it_next = item_of(peers + (blockIdx.x >> 3)), nb;
  if (it < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  // (told to be uniform: the LDS windows of the wave's loads then live in scalar registers)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The two strips of waves take the 16-row blocks of the tile alternately: strip wm owns rows 16 (2 rb + wm) + li,
  // rb = 0..7, i.e. half of every 32-row tile.  A block with fewer than eight tiles (the last of an expert) then
  // leaves both strips the same, smaller number of live row blocks, and its time shrinks with its rows.
  const int wm = wave / WN, wn = wave % WN;

  // this wave's share of a stage: rows 32 wave + 8 i + (lane >> 3), i = 0..3, of the x tile (the wave's rows are one tile
  // of the table) and of the weight tile
  const int lrow = lane >> 3;
  const uint32_t lchunk = (uint32_t)(((lane & 7) ^ lrow) * 16);
  // (piece i of the weights lies at woff[i % WO] + a multiple of the row stride)
  constexpr int WO = TR ? 2 : 1;
  uint32_t woff[WO];
#pragma unroll
  for (int i = 0; i < WO; ++i) {
    if constexpr (TR) {
      const int kr = 8 * wave + 2 * i + (lane >> 5);  // row of the weight tile: two per load, 32 lanes each
      woff[i] = (uint32_t)kr * (uint32_t)(a.ldw * 2) + (uint32_t)(((lane & 31) ^ ((kr & 3) << 1)) * 16);
    } else {
      woff[i] = (uint32_t)(32 * wave + lrow) * (uint32_t)(a.ldw * 2) + lchunk;
    }
  }
  const uint32_t wpiece = (uint32_t)((TR ? 4 : 8) * a.ldw * 2);
  // operand reads: byte offsets inside a stage for s = 0, 1 (row block rb of the strip: + 4 KB rb, column block cb of
  // the wave: + 2 KB cb, as immediate offsets)
  uint32_t a_rd[2], b_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const uint32_t pos = (uint32_t)(((4 * s + kb) ^ (li & 7)) * 16);
    a_rd[s] = (uint32_t)(16 * wm + li) * 128u + pos;
    b_rd[s] = (uint32_t)(16 * CB * wn + li) * 128u + pos;
  }
  // TR: this lane's address in the weight tile for column block cb: row 8 kb + (li >> 2) (+ 32 s + 4 h as immediate
  // offsets), outputs 64 wn + 16 cb + 4 (li & 3) .. + 3
  uint32_t b_tr[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
    b_tr[cb] = (uint32_t)(8 * kb + (li >> 2)) * 512u +
               (uint32_t)((8 * wn + 2 * (cb ^ (li >> 2)) + ((li & 3) >> 1)) * 16 + (li & 1) * 8);
  const int nk = a.K / kGBK;
  const int window = (32 * wave) * kGBK;  // first element of this wave's rows in a stage
  // LoRA: R = 1 << rs rank indices per group in a step, 1 << gs groups a step
  const int rs = a.rshift, gs = 6 - a.rshift, R = 1 << rs;

  // a work item = (row block, column block); the items of one expert are neighbours and reach one XCD together, column
  // block major, so that the blocks that read the same weight rows run side by side (the expert's entries are
  // contiguous: any of them names the range)
  auto entry_of = [&](int item, int* nb) __attribute__((always_inline)) {
    const GroupedPlanEntry* any = plan + item / ncb;
    const int local = item - any->first * ncb, count = max(any->count, 1);
    *nb = local / count;
    return plan + min(max(any->first + local % count, 0), entries - 1);
  };
  // byte offsets of the wave's four x rows (rows past the end of a tile hold some row of x: their sums are never stored)
  auto x_rows = [&](const GroupedPlanEntry* pe, int (&row)[4]) __attribute__((always_inline)) {
    if (a.x_map) {
#pragma unroll
      for (int i = 0; i < 4; ++i) row[i] = wave < pe->ntiles ? slot_rows[(pe->tile0 + wave) * kTileRows + 8 * i + lrow] : 0;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) row[i] = (wave < pe->ntiles ? pe->pos[wave] : 0) + 8 * i + lrow;
    }
  };
  uint32_t xoff[4];
  const int64_t xbytes = ((int64_t)(a.src_rows - 1) * a.ldx + a.K) * 2;
  int64_t xbytes_now;  // (nothing for the tiles that the block does not have)
  auto x_offsets = [&](const GroupedPlanEntry* pe, const int (&row)[4]) __attribute__((always_inline)) {
    xbytes_now = wave < pe->ntiles ? xbytes : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      xoff[i] = (uint32_t)min(max(row[i], 0), a.src_rows - 1) * (uint32_t)(a.ldx * 2) + lchunk;
  };
  const bf16_t* wfrom;  // the first weight of the item's column block, and the bytes from there to the end of its expert
  int64_t wbytes;
  auto weights_of = [&](const GroupedPlanEntry* pe, int nb) __attribute__((always_inline)) {
    const int64_t at = TR ? nb * BN : (int64_t)nb * BN * a.ldw;
    const int64_t span = TR ? (int64_t)(a.K - 1) * a.ldw + a.N : (int64_t)(a.N - 1) * a.ldw + a.K;
    wfrom = a.w + (int64_t)pe->expert * a.w_stride + at;
    wbytes = (span - at) * 2;
  };
  const uint32_t wstep = TR ? (uint32_t)(kGBK * a.ldw * 2) : kGBK * 2;
  // (past the last step nothing is fetched: a buffer of no bytes.  The count of loads in flight stays the same and there is
  // no branch, across which the compiler would lose track of which stage a load goes to and wait for all of them)
  auto fetch_x1 = [&](int ks, bf16_t* As, int i) __attribute__((always_inline)) {
    buffer16_to_lds(buffer_of(a.x, ks < nk ? xbytes_now : 0), xoff[i], (uint32_t)ks * (kGBK * 2), As + window + 8 * i * kGBK);
  };
  auto fetch_w1 = [&](int ks, bf16_t* Bs, int i) __attribute__((always_inline)) {
    buffer16_to_lds(buffer_of(wfrom, ks < nk ? wbytes : 0), woff[i % WO], (uint32_t)ks * wstep + (uint32_t)(i / WO) * wpiece,
                    TR ? Bs + (8 * wave + 2 * i) * BN : Bs + window + 8 * i * kGBK);
  };
  auto fetch_x = [&](int ks, bf16_t* As) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch_x1(ks, As, i);
  };
  auto fetch_w = [&](int ks, bf16_t* Bs) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WP; ++i) fetch_w1(ks, Bs, i);
  };

  const GroupedPlanEntry* pe = entry_of(it, &nb);
  {
    int row[4];
    x_rows(pe, row);
    x_offsets(pe, row);
  }
  weights_of(pe, nb);
  fetch_x(0, As0);
  fetch_w(0, Bs0);
  fetch_w(1, Bs1);
  fetch_x(1, As1);
  fetch_w(2, Bs2);

  for (;;) {
    const bool more = it_next >= 0;
    int nb_next, drawn = 0;
    if (more && tid == 0) drawn = atomicAdd(tickets + xcd, 1);  // (used behind the products)
    const GroupedPlanEntry* pe_next = entry_of(more ? it_next : it, &nb_next);
    const int ntiles = min(pe->ntiles, 8), slot0 = pe->tile0 * kTileRows, ngroups = min(pe->ngroups, 8);

    // LoRA: this lane's group of step l (its matrix and live rank)
    const bf16_t* lora_p = nullptr;
    int lora_r = 0;
    auto lora_group = [&](int l) __attribute__((always_inline)) {
      const int ln = here(lane), d = (l << gs) + ((TR ? 8 * wave : 8 * ((ln & 7) ^ (ln >> 3))) >> rs);
      lora_p = pe->matrix[min(d, 7)];
      lora_r = d < ngroups ? min(pe->rank[min(d, 7)], R) : 0;
    };

    f32x4 acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // h of the block's slots, rows of rpad elements as they lie in memory
    auto lora_x = [&](bf16_t* As) __attribute__((always_inline)) {
      const int bytes = ntiles * kTileRows * a.rpad * 2;
      const Buffer hbuf = buffer_of(a.hrow + (int64_t)slot0 * a.rpad, bytes);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (8192 * i >= bytes) break;
        buffer16_to_lds(hbuf, (uint32_t)here(tid) * 16u, 8192u * i, As + (512 * i + 64 * wave) * 8);
      }
    };
    // The groups' weights in the layout of the base weight tile.  Pieces past a group's rank come from a block of zeros.
    // A piece that the rank ends in, or a matrix that is not 16-byte aligned, goes through registers.
    auto lora_w = [&](int l, bf16_t* Bs) __attribute__((always_inline)) {
      if (l > 0) lora_group(l);
      const int ln = here(lane);
      const int first = TR ? 8 * wave + (ln >> 5) : 32 * wave + (ln >> 3);         // row of the tile this lane's piece 0 is in
      const int chunk = TR ? (ln & 31) ^ ((ln >> 5) << 1) : (ln & 7) ^ (ln >> 3);  // (TR: of pieces 0 and 2)
      const int n0 = (TR ? first : 8 * chunk) & (R - 1);                            // rank index it starts at
      const bf16_t* p = lora_p + (TR ? (int64_t)n0 * a.ldb + nb * BN : (int64_t)(nb * BN + first) * a.ldb + n0);
      const bool odd = lora_r > 0 && ((reinterpret_cast<uintptr_t>(lora_p) & 15u) != 0 || (!TR && (lora_r & 7) != 0));
      const bool slow = __ballot(odd) != 0ull;
#pragma unroll
      for (int i = 0; i < WP; ++i) {
        const bool live = (TR ? n0 + 2 * i : n0) < lora_r;
        // TR: rows 8 wave + 2 i + (lane >> 5), whose chunks are swizzled by row & 3
        const bf16_t* src = TR ? p + (int64_t)(2 * i) * a.ldb + 8 * (chunk ^ ((i & 1) << 2)) : p + (int64_t)(8 * i) * a.ldb;
        bf16_t* to = TR ? Bs + (8 * wave + 2 * i) * BN : Bs + window + 8 * i * kGBK;
        if (!slow) {
          load16_to_lds(live ? src : reinterpret_cast<const bf16_t*>(kernel_zeros), 0u, to);
        } else {
          const int keep = !live ? 0 : TR ? 8 : min(lora_r - n0, 8);
#pragma unroll 1
          for (int e = 0; e < 8; ++e) to[8 * ln + e] = e < keep ? src[e] : (bf16_t)0;
        }
      }
    };
    // The weight tiles, most of which come from memory, are requested three stages ahead, the x tiles, most of which another
    // column block of the same rows has just brought into this XCD's L2, two.  A 64-deep step on NRB live row blocks per
    // strip (NRB even) is four quarters of 2 NRB MFMAs: half of the row blocks of one 32-deep half step.  The operands of a
    // quarter are read from LDS during the quarter before it, also those of the next step's first two, so that the matrix
    // cores have work right behind the barrier in the middle of a step: there the wave has read the last of its operands of
    // this step and waits for its loads of the next one (all but its youngest, the weights of the step after), behind
    // the barrier everybody has, so the step's own stages take the loads two and three steps ahead.
    auto stage_a = [&](auto i) __attribute__((always_inline)) -> bf16_t* {
      if constexpr (decltype(i)::value == 0) return As0;
      else return As1;
    };
    auto stage_b = [&](auto i) __attribute__((always_inline)) -> bf16_t* {
      if constexpr (decltype(i)::value == 0) return Bs0;
      else if constexpr (decltype(i)::value == 1) return Bs1;
      else return Bs2;
    };
    using std::integral_constant;
    auto k_loop = [&](auto nrb_c) __attribute__((always_inline)) {
      constexpr int NRB = decltype(nrb_c)::value, H = NRB / 2;
      uint4 fw[2][CB], fx[2][2][H];  // [half step], [half step][half of the row blocks]
      auto read_w1 = [&](const bf16_t* Bs, int s, int cb) __attribute__((always_inline)) {
        const char* Bb = reinterpret_cast<const char*>(Bs);
        if constexpr (TR) {
          const uint2 lo = lds_read_transposed(Bb + b_tr[cb] + 16384 * s);
          const uint2 hi = lds_read_transposed(Bb + b_tr[cb] + 16384 * s + 2048);
          fw[s][cb] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        } else {
          fw[s][cb] = *reinterpret_cast<const uint4*>(Bb + b_rd[s] + 2048 * cb);
        }
      };
      auto read_x1 = [&](const bf16_t* As, int s, int half, int i) __attribute__((always_inline)) {
        fx[s][half][i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(As) + a_rd[s] + 4096 * (H * half + i));
      };
      // one quarter's MFMAs; `between(i)` is issued behind those of its i-th row block: a burst of requests would hold the
      // MFMAs behind it back until the memory units have taken the last one
      auto quarter = [&](int s, int half, auto between) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < H; ++i) {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            acc[H * half + i][cb] = mfma16(fw[s][cb], fx[s][half][i], acc[H * half + i][cb]);
          __builtin_amdgcn_sched_barrier(0);
          between(i);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      // those of n things that fall to place i of H
      auto spread = [&](int i, int n, auto f) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < n; ++j)
          if (j * H / n == i) f(j);
      };
      auto first_half = [&](const bf16_t* As, const bf16_t* Bs) __attribute__((always_inline)) {
        quarter(0, 0, [&](int i) __attribute__((always_inline)) {
          spread(i, CB, [&](int j) __attribute__((always_inline)) { read_w1(Bs, 1, j); });
          read_x1(As, 1, 0, i);
        });
        quarter(0, 1, [&](int i) __attribute__((always_inline)) { read_x1(As, 1, 1, i); });
      };
      auto step = [&](int ks, auto phase) __attribute__((always_inline)) {  // phase = ks mod 6
        constexpr int P = decltype(phase)::value;
        bf16_t *As = stage_a(integral_constant<int, P % 2>{}), *An = stage_a(integral_constant<int, (P + 1) % 2>{});
        bf16_t *Bs = stage_b(integral_constant<int, P % 3>{}), *Bn = stage_b(integral_constant<int, (P + 1) % 3>{});
        first_half(As, Bs);
        loads_landed_barrier<WP>();
        quarter(1, 0, [&](int i) __attribute__((always_inline)) {
          spread(i, 4, [&](int j) __attribute__((always_inline)) { fetch_x1(ks + 2, As, j); });
          spread(i, CB, [&](int j) __attribute__((always_inline)) { read_w1(Bn, 0, j); });
          read_x1(An, 0, 0, i);
        });
        quarter(1, 1, [&](int i) __attribute__((always_inline)) {
          spread(i, WP, [&](int j) __attribute__((always_inline)) { fetch_w1(ks + 3, Bs, j); });
          read_x1(An, 0, 1, i);
        });
      };
      loads_landed_barrier<4 + 2 * WP>();
#pragma unroll
      for (int j = 0; j < CB; ++j) read_w1(Bs0, 0, j);
#pragma unroll
      for (int i = 0; i < H; ++i) {
        read_x1(As0, 0, 0, i);
        read_x1(As0, 0, 1, i);
      }
      int ks = 0;
      for (; ks + 6 < nk; ks += 6) {
        step(ks, integral_constant<int, 0>{});
        step(ks + 1, integral_constant<int, 1>{});
        step(ks + 2, integral_constant<int, 2>{});
        step(ks + 3, integral_constant<int, 3>{});
        step(ks + 4, integral_constant<int, 4>{});
        step(ks + 5, integral_constant<int, 5>{});
      }
      constexpr int LAST = (REM + 5) % 6;
      if constexpr (LAST > 0) step(ks, integral_constant<int, 0>{});
      if constexpr (LAST > 1) step(ks + 1, integral_constant<int, 1>{});
      if constexpr (LAST > 2) step(ks + 2, integral_constant<int, 2>{});
      if constexpr (LAST > 3) step(ks + 3, integral_constant<int, 3>{});
      if constexpr (LAST > 4) step(ks + 4, integral_constant<int, 4>{});
      // The last step: behind its barrier every stage is free.  The LoRA tiles come first, then the next item's first
      // two, which travel while this one ends; the number drawn goes to the other waves by way of Bs1
      int row_next[4];
      x_rows(pe_next, row_next);
      if (ngroups > 0) lora_group(0);
      first_half(stage_a(integral_constant<int, LAST % 2>{}), stage_b(integral_constant<int, LAST % 3>{}));
      loads_landed_barrier<0>();
      if (tid == 0) *reinterpret_cast<int*>(Bs1) = more ? 2 * peers + drawn : items;
      if (ngroups > 0) {
        lora_x(As1);
        lora_w(0, Bs2);
      }
      x_offsets(pe_next, row_next);
      weights_of(pe_next, nb_next);
      if (!more) xbytes_now = wbytes = 0;  // nothing follows: the same count of loads, which bring nothing
      fetch_x(0, As0);
      fetch_w(0, Bs0);
      __builtin_amdgcn_sched_barrier(0);
      quarter(1, 0, [](int) {});
      quarter(1, 1, [](int) {});
    };
    // live row blocks per strip = tiles of the block, rounded up to even
    if (ntiles > 6) k_loop(integral_constant<int, 8>{});
    else if (ntiles > 4) k_loop(integral_constant<int, 6>{});
    else if (ntiles > 2) k_loop(integral_constant<int, 4>{});
    else k_loop(integral_constant<int, 2>{});

    loads_landed_barrier<4 + WP>();
    const int k_after = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(Bs1));
    for (int l = 0; l << gs < ngroups; ++l) {
      if (l > 0) {
        loads_landed_barrier<4 + WP>();  // (the tiles have been read)
        lora_w(l, Bs2);
        loads_landed_barrier<0>();
      }
      const char* Bb = reinterpret_cast<const char*>(Bs2);
      const int ln = here(lane), li2 = ln & 15, kb2 = ln >> 4;
      // row block rb of a strip lies in tile rb of the block, which has one group
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        if (rb >= ntiles) break;
        const int d = pe->number[rb] - (l << gs);
        if (d < 0 || d >> gs) continue;
        for (int n = 0; n < R; n += 32) {
          // first rank index of this lane's operand pieces; past R: any piece, masked
          const uint32_t live = n + 8 * kb2 < R ? ~0u : 0u;
          const int n0 = (int)((uint32_t)(n + 8 * kb2) & live);
          auto masked = [live](uint4 v) { return make_uint4(v.x & live, v.y & live, v.z & live, v.w & live); };
          const uint4 fx = masked(*reinterpret_cast<const uint4*>(As1 + (32 * rb + 16 * wm + li2) * a.rpad + n0));
          uint4 fw[CB];
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) {
            if constexpr (TR) {
              const uint32_t at = (uint32_t)((d << rs) + n0 + (li2 >> 2)) * 512u +
                                  (uint32_t)((8 * wn + 2 * (cb ^ (li2 >> 2)) + ((li2 & 3) >> 1)) * 16 + (li2 & 1) * 8);
              const uint2 lo = lds_read_transposed(Bb + at), hi = lds_read_transposed(Bb + at + 2048);
              fw[cb] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            } else {
              const int c = ((d << rs) + n0) >> 3;
              fw[cb] = *reinterpret_cast<const uint4*>(Bb + (16 * CB * wn + 16 * cb + li2) * 128 + ((c ^ (li2 & 7)) * 16));
            }
          }
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma16(masked(fw[cb]), fx, acc[rb][cb]);
        }
      }
    }
    auto store = [&]() __attribute__((always_inline)) {
      // lane holds y[slot 16 (2 rb + wm) + li][nb BN + 16 CB wn + 16 cb + 4 kb + v], v = 0..3.  Column blocks 2 c and 2 c + 1
      // exchange between neighbouring kb, so that a lane has eight consecutive columns and a store covers 64 bytes of 16 rows.
      const int ln = here(lane), i = 16 * wm + (ln & 15), chunk = ((ln >> 4) & 1) * 2 + (ln >> 5);
      bf16_t* y0 = a.y + nb * BN + 16 * CB * wn + 8 * chunk;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        if (rb >= ntiles) break;
        int row;
        if (a.map_rows) row = checked_row(slot_rows[slot0 + kTileRows * rb + i], a.tb);
        else row = i < pe->cnt[rb] ? pe->pos[rb] + i : -1;
        uint4 out[CB / 2];
#pragma unroll
        for (int c = 0; c < CB / 2; ++c) {
          const f32x4 u = acc[rb][2 * c], v = acc[rb][2 * c + 1];
          const auto lo = __builtin_amdgcn_permlane16_swap(pack_bf16(u[0], u[1]), pack_bf16(v[0], v[1]), false, false);
          const auto hi = __builtin_amdgcn_permlane16_swap(pack_bf16(u[2], u[3]), pack_bf16(v[2], v[3]), false, false);
          out[c] = make_uint4(lo[0], hi[0], lo[1], hi[1]);
        }
        if (row < 0) continue;
        bf16_t* yp = y0 + (int64_t)row * a.ldy;
#pragma unroll
        for (int c = 0; c < CB / 2; ++c) st16(yp + 32 * c, out[c]);
      }
    };
    loads_landed_barrier<4 + WP>();
    // A block's last item: no tiles behind it, and its stores are the last thing it does.  (It fetched the first tiles of any
    // item before and waited for them and its stores: 160 KB a block.  us, forward with the LoRA term, then and now, and what
    // the kernel with one block per item took: 1024 rows of 128 experts 768 -> 2048 102.6 / 97.0 / 109.2, 65536 rows
    // 2048 -> 512 186.7 / 186.7 / 204.5; one item per block, 16 rows of 8 experts 2048 -> 1536 33.9 / 33.3 / 32.0.)
    if (!more) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no load may land in LDS that belongs to the next block
      store();
      return;
    }
    fetch_w(1, Bs1);
    fetch_x(1, As1);
    fetch_w(2, Bs2);
    store();
    it = it_next;
    it_next = item_of(k_after);
    pe = pe_next;
    nb = nb_next;
  }
}

}  // namespace

bool grouped_gemm_supported(const GroupedArgs& a) {
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (a.K < kGBK || a.K % kGBK != 0 || a.N < 128 || a.N % 128 != 0) return false;
  if (a.ldx % 8 != 0 || a.ldw % 8 != 0 || a.w_stride % 8 != 0 || a.ldy % 4 != 0) return false;
  if (!al16(a.x) || !al16(a.w) || (reinterpret_cast<uintptr_t>(a.y) & 7u) != 0) return false;
  if (a.rpad != 0 && (a.rpad > 64 || a.ldb % 8 != 0 || !al16(a.hrow))) return false;
  return true;
}

bool grouped_gemm_direct(const GroupedArgs& a) {
  // (TK_GROUPED_DIRECT=0 in the environment keeps the register-staged kernels in use: an A/B switch, read per call)
  const char* env_direct = getenv("TK_GROUPED_DIRECT");
  return TK_GROUPED_DL && !(env_direct && env_direct[0] == '0') && (int64_t)a.src_rows * a.ldx * 2 < (1ll << 32) &&
         (int64_t)(a.w_rows_are_inputs ? a.K : a.N) * a.ldw * 2 < (1ll << 32) && a.ldy % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(a.y) & 15u) == 0;  // (16-byte stores)
}

// upper bound of the row blocks, for either block size (workspace sizing)
int64_t grouped_plan_entries(const SegLayout& L, int64_t experts) { return ceil_div(L.max_tiles, 4) + experts; }

int launch_grouped_gemm(const GroupedArgs& a, int experts, int nt, GroupedPlanEntry* plan, int32_t* nblocks,
                        const SegView& seg, const SegLayout& L, hipStream_t s) {
  if (L.rows == 0) return TK_OK;
  // The 8-wave variants win wherever they apply.  Both weight layouts load their tiles straight into LDS
  // (k_grouped_gemm_dl: 32-bit row offsets, so x and one expert's weights must span less than 4 GB); what that kernel does
  // not take runs on the 8 waves of k_grouped_gemm, except with the LoRA term on small experts (its epilogue
  // has no registers to spare: measured at 512 rows per expert, 4 waves are then 5 % faster).
  const int nks = a.rpad == 0 ? 0 : (a.rpad <= 32 ? 1 : 2);
  const bool direct = grouped_gemm_direct(a);
  const bool big =
      TK_GROUPED_BIG && a.N % 256 == 0 && (nks == 0 || direct || L.rows >= (int64_t)1024 * experts);
  const int ptiles = big ? 8 : 4, bn = big ? 256 : 128;
  const int max_entries = (int)(ceil_div(L.max_tiles, ptiles) + experts);
  hipLaunchKernelGGL(k_grouped_plan, dim3((unsigned)ceil_div(max_entries, kPlanBlock)), dim3(256), 0, s, a, seg, experts, nt,
                     plan, nblocks, max_entries, ptiles);
  const int32_t* y_rows = seg.slot_table(a.map_rows);
  const int32_t* rows = a.x_map ? seg.slot_row : y_rows;
  const int ncb = a.N / bn;
  if (big && direct) {
    const dim3 blocks((unsigned)std::min<int64_t>(round_up((int64_t)max_entries * ncb, 8), kGroupedBlocks));
    auto launch = [&](auto rem) {
      constexpr int REM = decltype(rem)::value;
      if (a.w_rows_are_inputs)
        hipLaunchKernelGGL((k_grouped_gemm_dl<1, REM>), blocks, dim3(512), 0, s, a, plan, nblocks, nblocks + 8, rows, ncb);
      else
        hipLaunchKernelGGL((k_grouped_gemm_dl<0, REM>), blocks, dim3(512), 0, s, a, plan, nblocks, nblocks + 8, rows, ncb);
    };
    switch (a.K / kGBK % 6) {
      case 0: launch(std::integral_constant<int, 0>{}); break;
      case 1: launch(std::integral_constant<int, 1>{}); break;
      case 2: launch(std::integral_constant<int, 2>{}); break;
      case 3: launch(std::integral_constant<int, 3>{}); break;
      case 4: launch(std::integral_constant<int, 4>{}); break;
      default: launch(std::integral_constant<int, 5>{}); break;
    }
    return check_launch();
  }
  // several thousand work items, so that the last round of blocks on the 256 CUs is a small part of the run
  const int64_t row_blocks = ceil_div(L.max_tiles, ptiles);
  const int cpi = (int)std::min<int64_t>(ncb, std::max<int64_t>(1, ceil_div(ncb * row_blocks, kGroupedItems)));
  const int nsplit = (int)ceil_div(ncb, cpi);
  const dim3 grid((unsigned)((int64_t)max_entries * nsplit));
#define TK_LAUNCH_GROUPED(NKS, BIG)                                                                                  \
  hipLaunchKernelGGL((k_grouped_gemm<NKS, BIG, 0>), grid, dim3(BIG ? 512 : 256), 0, s, a, plan, nblocks, seg.tile_group, \
                     rows, y_rows, nsplit, cpi)
  if (a.w_rows_are_inputs) {  // never with the LoRA term (the caller checks)
    if (big)
      hipLaunchKernelGGL((k_grouped_gemm<0, 1, 1>), grid, dim3(512), 0, s, a, plan, nblocks, seg.tile_group, rows, y_rows, nsplit,
                         cpi);
    else
      hipLaunchKernelGGL((k_grouped_gemm<0, 0, 1>), grid, dim3(256), 0, s, a, plan, nblocks, seg.tile_group, rows, y_rows, nsplit,
                         cpi);
  } else if (big) {
    if (nks == 0) TK_LAUNCH_GROUPED(0, 1);
    else if (nks == 1) TK_LAUNCH_GROUPED(1, 1);
    else TK_LAUNCH_GROUPED(2, 1);
  } else {
    if (nks == 0) TK_LAUNCH_GROUPED(0, 0);
    else if (nks == 1) TK_LAUNCH_GROUPED(1, 0);
    else TK_LAUNCH_GROUPED(2, 0);
  }
#undef TK_LAUNCH_GROUPED
  return check_launch();
}

}  // namespace tk
