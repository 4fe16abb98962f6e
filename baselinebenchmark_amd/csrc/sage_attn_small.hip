// Fused attention kernel variants of four wavefronts (128 query rows to a workgroup), for short sequences and calls that do not fill the
// chip (the rule: small_tiles_pay in sage_api.hip; those with an explicit mask, K blocks of 16 keys or interleaved K scales stand beside their
// larger brothers).  Own translation unit so that the sets of instantiations compile in parallel.
//
// With eight wavefronts a workgroup takes a compute unit for itself, and the 9 us that a q-tile spends on its addresses, raw rows,
// quantisation and output run beside nothing; at 1000 keys that is half of its time.  Four wavefronts use half the registers and
// 32 to 64 KB of LDS, so two workgroups (three at head_dim 64: 168 registers, a few of them in scratch memory, see attn_small_per_cu) share a
// compute unit and run those parts, and each other's matrix and
// vector work, side by side without barriers between them.  A wavefront is raised over the others of its SIMD while it issues
// matrix instructions (1 to 3 %).  The last tile is cut down to the 32-key groups that a wavefront sees, and only it is masked.
// Whole calls, 256 rows -> 128: 96 packed prompts of 16..1024 rows, 32/8 heads, head_dim 128, causal, FP16 524 -> 446 us, FP8 462 -> 393; head_dim
// 64, FP16 354 -> 259; 2 x 24 heads of 4095 rows and 257 keys, head_dim 64, 41.7 -> 30.8; 8 heads of 1024, head_dim 64, 25.7 -> 22.2.
// Tried: two slots for K and V side by side and one barrier per tile in FP16 kernels too (+-0 to 2 % slower at head_dim 64; no room at 128);
// FP8 with one V slot, as FP16 has it: 8 heads of 4000 rows, head_dim 64, 64 -> 49 us with three slots of both.
#include "sage_attn_kernel.h"

namespace sage {

namespace {
template <int D, int PV, bool MS, bool QF, int KW, bool DOT>
hipError_t launch_causal_or_not(const AttnArgs& a, bool causal, int grid, hipStream_t st) {
  return causal ? launch_one<D, 4, 128, PV, true, MS, 0, 1, QF, KW, DOT>(a, grid, st) : launch_one<D, 4, 128, PV, false, MS, 0, 1, QF, KW, DOT>(a, grid, st);
}
template <int D, int PV, bool MS, bool QF, bool DOT>
hipError_t launch_scales(const AttnArgs& a, bool causal, int grid, hipStream_t st) {
  return a.blkk >= 64 ? launch_causal_or_not<D, PV, MS, QF, 2, DOT>(a, causal, grid, st) : launch_causal_or_not<D, PV, MS, QF, 1, DOT>(a, causal, grid, st);
}
template <int D, int PV>
hipError_t launch_kind(const AttnArgs& a, bool causal, int grid, hipStream_t st) {
  constexpr bool MS = PV == 1 || D == 64;
  if (a.q_raw) {
    if (a.q_dot_km) return launch_scales<D, PV, false, true, true>(a, causal, grid, st);
    return a.lse ? launch_scales<D, PV, false, true, false>(a, causal, grid, st) : launch_scales<D, PV, MS, true, false>(a, causal, grid, st);
  }
  return a.lse ? launch_scales<D, PV, false, false, false>(a, causal, grid, st) : launch_scales<D, PV, MS, false, false>(a, causal, grid, st);
}
}  // namespace

hipError_t launch_attn_small(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st) {
  if (D == 128) return pv ? launch_kind<128, 1>(a, causal, grid, st) : launch_kind<128, 0>(a, causal, grid, st);
  return pv ? launch_kind<64, 1>(a, causal, grid, st) : launch_kind<64, 0>(a, causal, grid, st);
}

}  // namespace sage
