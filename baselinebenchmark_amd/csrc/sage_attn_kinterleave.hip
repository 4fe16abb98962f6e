// Fused attention kernel variants for four interleaved K scales per block (scale t of a block for its keys n with
// (n % 8) / 2 == t: the granularity upstream SageAttention calls per-thread for K).  Own translation unit so that the sets of
// instantiations compile in parallel.
#include "sage_attn_kernel.h"

namespace sage {

namespace {
template <int D, int PV, bool MS, bool QF, bool CAUSAL>
hipError_t launch_rows(const AttnArgs& a, int grid, hipStream_t st) {
  // FP8 P.V with LSE, and FP16 P.V of head_dim 64 where causal, take 128 rows at every size (small_tiles_pay)
  constexpr bool small_only = (PV == 1 && !MS) || (PV == 0 && D == 64 && CAUSAL);
  if (a.tile_rows == kSmallTileRows) return launch_one<D, 4, 128, PV, CAUSAL, MS, 0, 3, QF>(a, grid, st);
  if constexpr (small_only) return hipErrorInvalidValue;
  else return launch_one<D, 8, 128, PV, CAUSAL, MS, 0, 3, QF>(a, grid, st);
}
// Row sums on the matrix pipe for FP8 P.V without LSE, as for the plain K blocks; with a floating-point Q (a.q_raw)
// the q-tile is quantised in the prologue.
template <int D, int PV, bool MS>
hipError_t launch_kind(const AttnArgs& a, bool causal, int grid, hipStream_t st) {
  if (a.q_raw) return causal ? launch_rows<D, PV, MS, true, true>(a, grid, st) : launch_rows<D, PV, MS, true, false>(a, grid, st);
  return causal ? launch_rows<D, PV, MS, false, true>(a, grid, st) : launch_rows<D, PV, MS, false, false>(a, grid, st);
}
}  // namespace

hipError_t launch_attn_kinterleaved(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st) {
  if (!pv) return D == 128 ? launch_kind<128, 0, false>(a, causal, grid, st) : launch_kind<64, 0, false>(a, causal, grid, st);
  if (a.lse) return D == 128 ? launch_kind<128, 1, false>(a, causal, grid, st) : launch_kind<64, 1, false>(a, causal, grid, st);
  return D == 128 ? launch_kind<128, 1, true>(a, causal, grid, st) : launch_kind<64, 1, true>(a, causal, grid, st);
}

}  // namespace sage
