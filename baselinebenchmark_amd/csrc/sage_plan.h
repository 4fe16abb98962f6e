// The plan of a packed variable-length batch, built on the device by one workgroup.
#pragma once
#include "sage_launch.h"

namespace sage {

// ---------------------------------------------------------------------------------------------
// Variable-length plan: block offsets per sequence and the cost-ordered tile list.
//
// Tiles are listed in cost TIERS of kTierCost cost units (eight causal q-tiles of 256 rows when the unit is 64 keys),
// most expensive tier first; inside a tier sequence by sequence, and inside a sequence the heavier q-tiles first.
// Consecutive entries of the list run at the same time (eight of them per XCD when an XCD holds one KV head), and q-tiles
// of one sequence walk the same K/V tiles from tile 0 on at about the same pace: one fetches a tile into the XCD's L2, the
// others hit it there.  Ordered by cost alone, neighbours in the list belong to different sequences and share nothing.
// (Attention kernel, 32/8 heads, causal, by cost alone / by tiers: 70 sequences of 500..8000 rows 10.67 / 10.06 ms, 80 of 16..1991 1.13 /
// 1.10.  The price is the last round of the chip: below 2048 keys all q-tiles are one tier, and a long prompt that the batch ends
// with starts last -- 127 of 64 rows and one of 2000 176 / 182 us, 500 of 100 and one of 1990 over 8 heads 165 / 189.)
//
// One workgroup, bound by the latency of its dependent steps.  The cost of a q-tile does not decrease with its index, so the
// tiles of a sequence in one tier are a contiguous range with ends in closed form, and no tile is ever visited to be counted:
// one wavefront owns a tier, a lane a sequence, and a wavefront scan gives every sequence its place in the tier's part of the
// list.  (A histogram over all tiles, with one pass of the whole workgroup and four barriers per sequence, took 82 us for
// 96 sequences of 16..1024 rows and 30 us for 16 of 512..32768; this takes 9 and 10.)
// ---------------------------------------------------------------------------------------------
constexpr int kCostMax = 2047, kTierCost = 32, kTiers = (kCostMax + 1) / kTierCost;
constexpr int kPlanThreads = 1024, kPlanSeqsLds = 4096;   // of the plan's own launch; the pre-pass launch that carries it has 256 lanes
static_assert(kTiers == 64, "one lane per tier in the scan over the tiers");
template <int SEQS>
struct PlanLds {
  int2 len[SEQS];   // (query rows, keys) of the first sequences; the rest is read again where needed
  int tier_total[kTiers], tier_start[kTiers], longest;
};

__device__ inline int wave_inclusive_scan(int x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(x, d, 64);
    if (lane >= d) x += up;
  }
  return x;
}

template <int THREADS, int SEQS>
__device__ __forceinline__ void varlen_plan(const PlanArgs& a, PlanLds<SEQS>& lds) {
  constexpr int kPlanThreads = THREADS, kPlanWaves = THREADS / 64, kPlanSeqsLds = SEQS;
  static_assert(kPlanWaves >= 3, "three wavefronts write the block offsets");
  const int32_t *cu_q = a.cu_q, *cu_k = a.cu_k;
  const int nseq = a.nseq, blkq = a.blkq, blkk = a.blkk, bm = a.bm, bn = a.bn, causal = a.causal;
  int32_t* plan = a.plan;
  const SagePlanLayout L = plan_layout(nseq, a.total_q);
  int32_t* tiles = plan + L.tiles;
  int2(&len_lds)[SEQS] = lds.len;
  int(&tier_total)[kTiers] = lds.tier_total;
  int(&tier_start)[kTiers] = lds.tier_start;
  int& longest = lds.longest;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if (tid == 0) longest = 0;
  __syncthreads();
  auto lengths_in_memory = [&](int i) { return make_int2(cu_q[i + 1] - cu_q[i], cu_k[i + 1] - cu_k[i]); };
  {
    int most = 0;
    for (int i = tid; i < nseq; i += kPlanThreads) {
      const int2 n = lengths_in_memory(i);
      if (i < kPlanSeqsLds) len_lds[i] = n;
      most = max(most, causal ? min(n.y, (n.x + bm - 1) / bm * bm) : n.y);
    }
    atomicMax(&longest, most);
  }
  __syncthreads();
  auto lengths = [&](int i) { return i < kPlanSeqsLds ? len_lds[i] : lengths_in_memory(i); };
  const int top_tier = min((longest + bn - 1) / bn, kCostMax) / kTierCost;   // the tiers above it are empty
  // First q-tile of a sequence whose tier is at least t: its cost, in units of bn keys, has to reach t * kTierCost.
  auto first_tile = [&](int2 n, int nqt, int t) {
    const int keys = bn * (t * kTierCost - 1) + 1;
    return t == 0 ? 0 : n.y < keys ? nqt : causal ? min(nqt, (keys + bm - 1) / bm - 1) : 0;
  };

  // block offsets: three running sums over the sequences, one wavefront each (the last ones: tiers start at the first)
  if (w >= kPlanWaves - 3) {
    const int which = kPlanWaves - 1 - w;
    int32_t* dst = plan + (which == 0 ? L.cu_qblk : which == 1 ? L.cu_kblk : L.cu_panel);
    const int unit = which == 0 ? blkq : which == 1 ? blkk : kPanelRows;
    int before = 0;
    for (int i0 = 0; i0 < nseq; i0 += 64) {
      const int i = i0 + lane;
      const int2 n = i < nseq ? lengths(i) : make_int2(0, 0);
      const int blocks = ((which == 0 ? n.x : n.y) + unit - 1) / unit;
      const int upto = before + wave_inclusive_scan(blocks);
      if (i < nseq) dst[i] = upto - blocks;
      before = __shfl(upto, 63, 64);
    }
    if (lane == 0) dst[nseq] = before;
  }
  // tiles per tier
  for (int t = w; t < kTiers; t += kPlanWaves) {
    int count = 0;
    if (t <= top_tier) {
      for (int i = lane; i < nseq; i += 64) {
        const int2 n = lengths(i);
        const int nqt = (n.x + bm - 1) / bm;
        count += (t == kTiers - 1 ? nqt : first_tile(n, nqt, t + 1)) - first_tile(n, nqt, t);
      }
      count = __shfl(wave_inclusive_scan(count), 63, 64);
    }
    if (lane == 0) tier_total[t] = count;
  }
  __syncthreads();
  if (w == 0) {   // where each tier starts in the list: lane l takes tier kTiers - 1 - l
    const int t = kTiers - 1 - lane, upto = wave_inclusive_scan(tier_total[t]);
    tier_start[t] = upto - tier_total[t];
    if (lane == 63) plan[L.ntiles] = upto;
  }
  __syncthreads();
  for (int t = w; t <= top_tier; t += kPlanWaves) {
    if (tier_total[t] == 0) continue;
    int before = tier_start[t];
    for (int i0 = 0; i0 < nseq; i0 += 64) {
      const int i = i0 + lane;
      int lo = 0, hi = 0;   // this sequence's q-tiles in the tier: lo .. hi - 1
      if (i < nseq) {
        const int2 n = lengths(i);
        const int nqt = (n.x + bm - 1) / bm;
        lo = first_tile(n, nqt, t);
        hi = t == kTiers - 1 ? nqt : first_tile(n, nqt, t + 1);
      }
      const int upto = before + wave_inclusive_scan(hi - lo);
      // A lane writes its own sequence's q-tiles; those of a few long sequences (non-causal, or past the last tier's start) the
      // whole wavefront, one after the other: 1 M rows, one sequence, took 137 us with one lane, 14 like this.  (Many long ones
      // keep as many lanes busy by themselves: 100 of 17000 rows and 300 keys 12.8 us, one after the other 23.)
      unsigned long long todo = __builtin_amdgcn_ballot_w64(hi - lo > 64);
      if (__popcll(todo) > 16) todo = 0;
      if (!(todo >> lane & 1))
        for (int qt = lo; qt < hi; qt++) tiles[upto - 1 - (qt - lo)] = (i << 16) | qt;
      for (; todo; todo &= todo - 1) {
        const int src = __builtin_ctzll(todo), first = __shfl(lo, src, 64), end = __shfl(hi, src, 64), last = __shfl(upto, src, 64) - 1;
        for (int qt = first + lane; qt < end; qt += 64) tiles[last - (qt - first)] = ((i0 + src) << 16) | qt;
      }
      before = __shfl(upto, 63, 64);
    }
  }
}

}  // namespace sage
