// bf16 launches of the segmented LoRA pass at padded rank 128 (kernel templates: lora_kernels.h).
//
// What bounds these kernels is the memory system, as at the lower ranks; the rank costs registers (accumulators and the
// weight block of the expand) and L2 reads of weights.  8192 rows x 4096 columns, four adapters, us, against the kernels
// for any shape (kernels_generic.hip): shrink 64 + 14 -> 29 + 8 (the slices hold half as many bytes as the source),
// expand 84 -> 49 (2.7 TB/s of y; 31 where it only writes), row contraction 94 -> 35 (chunks in pairs and one reader per
// tile), its reduction 36 -> 22.
#include <algorithm>

#include "lora_kernels.h"

namespace tk {

int launch_pass_rank128(const PassArgs& a, const SegView& seg, const SegLayout& L, int phases, hipStream_t s) {
  bf16_t* hrow = (bf16_t*)a.hT + (int64_t)a.rpad * a.ldh;  // second half of the h buffer
  const int32_t* rows = seg.slot_table(a.map_rows);
  if (phases & 1) {
    // weights shared in LDS where the plan asks for it; short groups and wide sources take the tile-by-tile kernel, whose
    // blocks of four waves do not wait for groups of eight tiles
    if (a.set_steps == 0) {
      const int rc = launch_pass_generic(a, seg, L, TK_DTYPE_BF16, 1, s);
      if (rc != TK_OK) return rc;
    } else if (shrink_dl_applies(a)) {
      hipLaunchKernelGGL(k_shrink_dl<8>, dim3((unsigned)(ceil_div(L.max_tiles, 8) * a.kslices)), dim3(512), 0, s, a,
                         seg.tile_group, rows, (int)L.max_tiles);
    } else {
      hipLaunchKernelGGL(k_shrink_oct<8>, dim3((unsigned)(ceil_div(L.max_tiles, 8) * a.kslices)), dim3(512), 0, s, a,
                         seg.tile_group, rows, (int)L.max_tiles);
    }
  }
  if (((phases & 4) || ((phases & 1) && a.set_steps > 0)) && a.kslices > 1)
    hipLaunchKernelGGL(k_shrink_finish<8>, shrink_finish_grid<8>(L), dim3(256), 0, s, a, hrow, seg.tile_group, rows);
  if (a.dst && (phases & 2)) launch_expand_multi<8>(a, hrow, seg, L, s);
  return check_launch();
}

int launch_wgrad_rank128(const WgradArgs& a0, const SegView& seg, const SegLayout& L, hipStream_t s) {
  WgradArgs a = a0;
  a.tr.y_blocks = 0;
  const int nx = a.width / 128;
  if (a.tr.aT) {
    const int64_t units = (int64_t)a.tr.groups * a.rpad * ((a.tr.out_features + a.tr.in_features) / 64);
    a.tr.y_blocks = (int)std::min<int64_t>(64, std::max<int64_t>(1, units / (2 * nx * 256)));
  }
  const size_t dyn = (size_t)L.chunk_tiles * kTileRows * sizeof(int32_t) * (a.pair_chunks ? 2 : 1);
  const dim3 grid((unsigned)nx, (unsigned)(L.max_chunks + a.tr.y_blocks));
  hipLaunchKernelGGL((k_wgrad_coop<8, TK_COOP_STAGES, 1>), grid, dim3(256), dyn, s, a, seg.chunks,
                     seg.slot_table(a.map_rows));
  return check_launch();
}

}  // namespace tk
