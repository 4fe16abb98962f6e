// Fused attention kernel variants that follow a packed boolean mask (sage_common.h): only the key tiles that a q-tile sees
// are loaded and multiplied, and a partly visible tile costs two bit operations per score.  Own translation unit so that
// the sets of instantiations compile in parallel.
#include "sage_attn_kernel.h"

namespace sage {

namespace {
template <int D, int PV>
hipError_t launch_kind(const AttnArgs& a, int grid, hipStream_t st) {
  if (a.k_interleave) return launch_one<D, 8, 128, PV, false, false, 3, 3>(a, grid, st);
  if (a.blkk == 16) return launch_one<D, 8, 128, PV, false, false, 3, 2>(a, grid, st);
  if (a.tile_rows == kSmallTileRows) return launch_one<D, 4, 128, PV, false, false, 3, 1>(a, grid, st);
  if constexpr (PV == 0) return launch_one<D, 8, 128, PV, false, false, 3, 1>(a, grid, st);
  else return hipErrorInvalidValue;   // (they take 128 rows at every size: small_tiles_pay)
}
}  // namespace

hipError_t launch_attn_packed_mask(const AttnArgs& a, int D, int pv, int grid, hipStream_t st) {
  if (D == 128) return pv ? launch_kind<128, 1>(a, grid, st) : launch_kind<128, 0>(a, grid, st);
  return pv ? launch_kind<64, 1>(a, grid, st) : launch_kind<64, 0>(a, grid, st);
}

}  // namespace sage
