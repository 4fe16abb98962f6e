// Fused attention kernel variants that follow a packed boolean mask (sage_common.h): only the key tiles that a q-tile sees
// are loaded and multiplied, and a partly visible tile costs two bit operations per score.  Own translation unit so that
// the sets of instantiations compile in parallel.
#include "sage_attn_kernel.h"

namespace sage {

hipError_t launch_attn_packed_mask(const AttnArgs& a, int D, int pv, int grid, hipStream_t st) {
  if (a.tile_rows == kSmallTileRows) {
    if (D == 128) return pv ? launch_one<128, 4, 128, 1, false, false, 3, 1>(a, grid, st) : launch_one<128, 4, 128, 0, false, false, 3, 1>(a, grid, st);
    return pv ? launch_one<64, 4, 128, 1, false, false, 3, 1>(a, grid, st) : launch_one<64, 4, 128, 0, false, false, 3, 1>(a, grid, st);
  }
#define SAGE_ATTN_B(DD, PVV) (a.k_interleave ? launch_one<DD, 8, 128, PVV, false, false, 3, 3>(a, grid, st) : a.blkk == 16 ? launch_one<DD, 8, 128, PVV, false, false, 3, 2>(a, grid, st) : launch_one<DD, 8, 128, PVV, false, false, 3, 1>(a, grid, st))
  if (D == 128) return pv ? SAGE_ATTN_B(128, 1) : SAGE_ATTN_B(128, 0);
  return pv ? SAGE_ATTN_B(64, 1) : SAGE_ATTN_B(64, 0);
#undef SAGE_ATTN_B
}

}  // namespace sage
