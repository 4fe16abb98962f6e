// Launchers of the fused attention kernel (variants without an explicit mask) and of the packed-batch plan.
#include "sage_attn_kernel.h"
#include "sage_plan.h"

namespace sage {

// ---------------------------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------------------------
void finish_attn_args(AttnArgs& a, bool causal) {
  const bool packed = a.cu_q != nullptr;
  a.G = a.Hq / a.Hkv;
  const int heads = packed ? a.Hq : a.B * a.Hq, groups = packed ? a.Hkv : a.B * a.Hkv;
  a.div_G = make_fastdiv(a.G);
  a.div_Hkv = make_fastdiv(a.Hkv);
  a.div_heads = make_fastdiv(heads > 0 ? heads : 1);
  a.tier_shift = -1;
  a.div_range = a.div_last = make_fastdiv(1);
  // Per-XCD tile order (fixed-length batches whose heads and KV groups spread evenly over the eight XCDs): ranges of
  // R = 2^tier_shift consecutive q-tiles, R at most 32 and at most half of a head's q-tiles.  (The lines below were measured with q-tiles of
  // 256 rows and are the same numbers of q-tiles for those of 128.)  Causal problems with fewer than
  // 16 q-tiles per compute unit keep the plain heaviest-first order -- with so few rounds the balance of the last one
  // matters more than locality (1 x 32 heads of 4096 rows: 7 % slower with ranges) -- unless an XCD holds 16 heads or
  // more and 8 q-tiles per compute unit (4 x 32 heads of 4096 rows: 2 % faster with ranges, 8 x 32 of 2048 rows 5 %).
  if (!packed && (heads & 7) == 0 && (groups & 7) == 0 && (!causal || (int64_t)a.nqt * (heads >> 3) >= 512 || ((int64_t)a.nqt * (heads >> 3) >= 256 && (heads >> 3) >= 16))) {
    int shift = 5;
    while (shift > 0 && (2 << shift) > a.nqt) shift--;
    a.tier_shift = shift;
    const int R = 1 << shift, hpx = heads >> 3, last = a.nqt - (a.nqt >> shift << shift);
    a.div_range = make_fastdiv((uint32_t)R * hpx);
    a.div_last = make_fastdiv(last > 0 ? last : 1);
  }
}

hipError_t launch_attn(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st) {
  if (grid == 0) return hipSuccess;
  if (a.mask_bits) return launch_attn_packed_mask(a, D, pv, grid, st);
  if (a.mask) return launch_attn_masked(a, D, pv, grid, st);
  if (a.k_interleave) return launch_attn_kinterleaved(a, D, pv, causal, grid, st);
  if (a.blkk == 16) return launch_attn_k16(a, D, pv, causal, grid, st);
  if (a.tile_rows == kSmallTileRows) return launch_attn_small(a, D, pv, causal, grid, st);
  if (a.q_raw) return launch_attn_qfused(a, D, pv, causal, grid, st);
  // Row sums on the matrix pipe unless LSE is wanted (FP16 P.V: only head_dim 64 gains by it; head_dim 128 is
  // bound by its matrix phases and keeps the sums on the vector ALU).
  const bool msum = a.lse == nullptr;
  // (K scale blocks of 64 / 128 keys: the variants that know which 32-key groups share a scale)
#define SAGE_ATTN_W(DD, PVV, BNN, MS, KWW) (causal ? launch_one<DD, 8, BNN, PVV, true, MS, 0, 1, false, KWW>(a, grid, st) : launch_one<DD, 8, BNN, PVV, false, MS, 0, 1, false, KWW>(a, grid, st))
#define SAGE_ATTN(DD, PVV, BNN, MS) (a.blkk >= 128 ? SAGE_ATTN_W(DD, PVV, BNN, MS, 4) : a.blkk == 64 ? SAGE_ATTN_W(DD, PVV, BNN, MS, 2) : SAGE_ATTN_W(DD, PVV, BNN, MS, 1))
  if (D == 128) return pv ? (msum ? SAGE_ATTN(128, 1, 128, true) : SAGE_ATTN(128, 1, 128, false)) : SAGE_ATTN(128, 0, 128, false);
  if (pv || !msum) return pv ? (msum ? SAGE_ATTN(64, 1, 128, true) : SAGE_ATTN(64, 1, 128, false)) : SAGE_ATTN(64, 0, 128, false);
  // (FP16 P.V without LSE, not causal: the variant for 64-key scales also where they cover 128 keys, the same numbers.  The one for 128-key
  // scales comes out of the compiler with a phase of the loop in two copies, 3133 instructions against 2889: 16 heads of 6000 rows 161.4 us
  // instead of 166.1, 48 of 2222 74.1 / 75.8, 48 of 4096 182.5 / 185.1, 32 of 8192 460 / 468, 2 of 20000 236 / 246.  Causal, where neither
  // has that, the 128-key one is the smaller and faster.)
  if (!causal) return a.blkk >= 64 ? launch_one<64, 8, 128, 0, false, true, 0, 1, false, 2>(a, grid, st) : launch_one<64, 8, 128, 0, false, true, 0, 1, false, 1>(a, grid, st);
  return a.blkk >= 128 ? launch_one<64, 8, 128, 0, true, true, 0, 1, false, 4>(a, grid, st) : a.blkk == 64 ? launch_one<64, 8, 128, 0, true, true, 0, 1, false, 2>(a, grid, st) : launch_one<64, 8, 128, 0, true, true, 0, 1, false, 1>(a, grid, st);
#undef SAGE_ATTN_W
#undef SAGE_ATTN
}

__global__ void __launch_bounds__(kPlanThreads) varlen_plan_kernel(PlanArgs a) {
  __shared__ PlanLds<kPlanSeqsLds> lds;
  varlen_plan<kPlanThreads, kPlanSeqsLds>(a, lds);
}

hipError_t launch_varlen_plan(const int32_t* cu_q, const int32_t* cu_k, int nseq, int total_q, int blkq, int blkk, int bm,
                              int bn, int causal, int32_t* plan, hipStream_t st) {
  const PlanArgs a = {cu_q, cu_k, nseq, total_q, blkq, blkk, bm, bn, causal, plan};
  varlen_plan_kernel<<<1, kPlanThreads, 0, st>>>(a);
  return hipGetLastError();
}

}  // namespace sage
