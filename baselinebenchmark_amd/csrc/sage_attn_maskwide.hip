// Fused attention kernel variants with an explicit mask whose keys are contiguous: four mask values per load (sage_attn_mask.hip
// holds those for other strides, and the rule).  Own translation unit so that the sets of instantiations compile in parallel.
#include "sage_attn_kernel.h"

namespace sage {

hipError_t launch_attn_masked_wide(const AttnArgs& a, int D, int pv, int grid, hipStream_t st) {
#define SAGE_ATTN_WS(DD, PVV) (a.mask_kind == 1 ? launch_one<DD, 4, 128, PVV, false, false, 4, 1>(a, grid, st) : launch_one<DD, 4, 128, PVV, false, false, 5, 1>(a, grid, st))
  if (a.tile_rows == kSmallTileRows) return D == 128 ? (pv ? SAGE_ATTN_WS(128, 1) : SAGE_ATTN_WS(128, 0)) : pv ? SAGE_ATTN_WS(64, 1) : SAGE_ATTN_WS(64, 0);
#undef SAGE_ATTN_WS
#define SAGE_ATTN_WK(DD, PVV, KS) (a.mask_kind == 1 ? launch_one<DD, 8, 128, PVV, false, false, 4, KS>(a, grid, st) : launch_one<DD, 8, 128, PVV, false, false, 5, KS>(a, grid, st))
#define SAGE_ATTN_W(DD, PVV) (a.k_interleave ? SAGE_ATTN_WK(DD, PVV, 3) : a.blkk == 16 ? SAGE_ATTN_WK(DD, PVV, 2) : SAGE_ATTN_WK(DD, PVV, 1))
  if (D == 128) return pv ? SAGE_ATTN_W(128, 1) : SAGE_ATTN_W(128, 0);
  return pv ? SAGE_ATTN_W(64, 1) : SAGE_ATTN_W(64, 0);
#undef SAGE_ATTN_W
#undef SAGE_ATTN_WK
}

}  // namespace sage
