// Fused attention kernel variants with an explicit mask whose keys are contiguous: four mask values per load (sage_attn_mask.hip
// holds those for other strides, and the rule).  Own translation unit so that the sets of instantiations compile in parallel.
#include "sage_attn_kernel.h"

namespace sage {

namespace {
template <int D, int PV, int MASK>
hipError_t launch_mask(const AttnArgs& a, int grid, hipStream_t st) {
  if (a.k_interleave) return launch_one<D, 8, 128, PV, false, false, MASK, 3>(a, grid, st);
  if (a.blkk == 16) return launch_one<D, 8, 128, PV, false, false, MASK, 2>(a, grid, st);
  if (a.tile_rows == kSmallTileRows) return launch_one<D, 4, 128, PV, false, false, MASK, 1>(a, grid, st);
  if constexpr (PV == 0 && MASK == 4) return launch_one<D, 8, 128, PV, false, false, MASK, 1>(a, grid, st);
  else return hipErrorInvalidValue;   // (they take 128 rows at every size: small_tiles_pay)
}
template <int D, int PV>
hipError_t launch_kind(const AttnArgs& a, int grid, hipStream_t st) {
  return a.mask_kind == 1 ? launch_mask<D, PV, 4>(a, grid, st) : launch_mask<D, PV, 5>(a, grid, st);
}
}  // namespace

hipError_t launch_attn_masked_wide(const AttnArgs& a, int D, int pv, int grid, hipStream_t st) {
  if (D == 128) return pv ? launch_kind<128, 1>(a, grid, st) : launch_kind<128, 0>(a, grid, st);
  return pv ? launch_kind<64, 1>(a, grid, st) : launch_kind<64, 0>(a, grid, st);
}

}  // namespace sage
