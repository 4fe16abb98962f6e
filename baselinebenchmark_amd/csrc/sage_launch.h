// Host-side launcher declarations shared between the kernel translation units and the C ABI.
#pragma once
#include "sage_common.h"

namespace sage {

struct QuantArgs {
  const u16* x;
  int8_t* out;
  float* scale;
  const u16* km;
  int B, H, L, D;
  int64_t x_sb, x_sh, x_sn, o_sb, o_sh, o_sn, km_sb, km_sh;
  int blk, blk_shift;   // rows per scale block and their log2
  int groups;   // scales per block: 1; 8 (scale g covers the rows r of the block with r % 8 == g); 4 ((r % 8) / 2 == g); fixed-length only
  float mult;
  const int32_t* cu_seqlens;
  const int32_t* cu_blocks;
  int64_t scale_sh;
  // optional row dot products (null dot_out: off): dotv is [B, H/dv_group, D] in the input dtype,
  // dot_out is [B, H, L] (or [H, dot_total] for packed rows) fp32
  const u16* dotv;
  float* dot_out;
  int64_t dv_sb, dv_sh;
  int dv_group;
  int dot_total;
  // K mean from its per-chunk sums (fused pre-pass): partial sums [B, H, nchunk, D], at most kFusedChunks chunks of a sequence; the
  // workgroup of a sequence's first rows also writes the mean to km_out [B, H, D].  km is ignored then.
  const double* km_partial;
  int km_nchunk;
  u16* km_out;
  int heads_first;   // set by the launcher: grid is (head, rows) instead of (rows, head)
  int cached;        // read through the caches (with_loads) instead of past them
};

// Geometry of the quantiser: a workgroup of 256 lanes takes quant_rows(D, blk) consecutive rows of one (batch, head), whole scale
// blocks of them, and a wavefront quant_passes(D, blk) times quant_wave_rows(D) neighbouring ones, never more than a scale block: the
// maximum of a block crosses wavefronts only where the block does, and no lane is idle at any block size.
// Bound by HBM (3 bytes per element) with the vector ALU close behind it: 14.6 vector instructions per element (SQ_INSTS_VALU), 17.6 when the
// differences were narrowed one by one, widened twice and packed by masks and shifts.  bf16, K mean subtracted, head_dim 128, one kernel: 4 x 32
// heads of 4096 rows, blocks of 64: 52.0 -> 40.8 us (201 MB, 4.9 TB/s); blocks of 16, 2 x 16 heads of 4096 rows, where a block a
// workgroup left half the lanes idle: 24.5 -> 13.1.
__host__ __device__ constexpr int quant_wave_rows(int D) { return 64 / (D / 16); }   // rows of a pass of a wavefront
__host__ __device__ constexpr int quant_passes(int D, int blk) { return D == 128 ? (blk == 128 ? 4 : 2) : (blk >= 64 ? 2 : 1); }
__host__ __device__ constexpr int quant_rows(int D, int blk) { return 4 * quant_passes(D, blk) * quant_wave_rows(D); }

struct ColStatArgs {
  const u16* x;
  void* partial;  // double or float [B*H*nchunk*D]
  int B, H, L, D;
  int64_t x_sb, x_sh, x_sn;
  int nchunk;
  const int32_t* cu_seqlens;
  int heads_first, cached;   // as in QuantArgs
};

struct PrepVArgs {
  const u16* v;
  uint8_t* panels;
  const float* vscale;  // [B*H*D] (fp8) or null
  int B, H, L, D;
  int64_t v_sb, v_sh, v_sn;
  const int32_t* cu_seqlens;
  const int32_t* cu_panels;
  int64_t panel_sh;
  // V scales from their per-chunk maxima (fused pre-pass), like QuantArgs::km_partial; vscale is ignored then.
  const float* vs_partial;
  int vs_nchunk;
  float* vscale_out;
  int heads_first, cached;   // as in QuantArgs
};

struct MaskPackArgs {
  const uint8_t* mask;
  int64_t m_sb, m_sh, m_sm, m_sn;
  MaskPlanes p;
  int Sq, Skv;
  uint8_t *bits, *seen;
};

struct PlanArgs {
  const int32_t *cu_q, *cu_k;
  int nseq, total_q, blkq, blkk, bm, bn, causal;
  int32_t* plan;
};

// Division of a 32-bit unsigned number by a launch constant as a multiply-high and two shifts (exact for every 32-bit
// dividend): the tile decode of the attention kernel divides the workgroup index by head counts that are no powers of
// two, and a true integer division is some twenty dependent instructions on this hardware, paid by every workgroup
// before its first memory request.
struct FastDiv {
  uint32_t mul, sh1, sh2;
};
inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f;
  uint32_t L = 0;
  while (L < 32 && (uint64_t(1) << L) < d) L++;               // ceil(log2 d); d >= 1
  f.mul = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << L) - d)) / d + 1);
  f.sh1 = L < 1 ? L : 1;
  f.sh2 = L < 1 ? 0 : L - 1;
  return f;
}
__device__ inline uint32_t fastdiv(uint32_t n, const FastDiv& f) {
  const uint32_t t = __umulhi(f.mul, n);
  return (t + ((n - t) >> f.sh1)) >> f.sh2;
}

// Few query rows over a long history (sage_attn_few.hip).  `part` holds nsplit partial results per (batch, KV head): O [rows, D],
// m [rows], l [rows], smoothing term [rows], rounded up to 16 bytes.
// The row limit is two 16-column score tiles: at head_dim 128 the output of a third would not fit the registers.  At the limit
// (4 x 32 heads, 16 rows, 4096 keys) a call takes 86.4 us here and 173.0 with the tiled kernel.
constexpr int kFewRows = 32;          // query rows per KV head, over all query heads of its group
constexpr int kFewWorkgroups = 512;   // two per compute unit, what the registers allow at once
// Chunks of a sequence up to which every workgroup combines the sums of K itself, FP16 P.V.  It walks them eight at a time, as the
// finalise kernel does, but all 512 workgroups do and read them from the L2.  Whole calls, 1 row, bf16, in the kernel / by a launch: 1 KV
// head of 64 chunks 25.2 / 25.6 us, 128 34.9 / 34.6, 512 79.2 / 74.5, 8192 1019 / 905; 8 heads of 64 48.2 / 49.3, 128 84.8 / 85.5, 1024
// 599 / 588; 32 of 64 148 / 149, 128 283 / 283.  (FP8 P.V walks both statistics side by side, two launches one after the other: 1 head
// of 8192 chunks 1364 / 1535, 8 of 256 253 / 263; always in the kernel.)
constexpr int kFewChunks = 128;
struct FewArgs {
  const u16 *q, *k, *v;
  // per-chunk statistics (ColStatArgs), combined in the kernel: sums of K or null (no smoothing), abs-maxima of V (FP8 P.V) or null.
  // nchunk 0, FP16 P.V: km_partial is the mean itself, [B, Hkv, D] in K's type
  const double* km_partial;
  const float* vs_partial;
  float* vscale;   // [B, Hkv, D], written by the main kernel for the merge
  int nchunk;
  u16* out;
  float *lse, *part;
  int64_t part_bytes;   // room for partial results
  int B, Hq, Hkv, Sq, Skv;
  int64_t q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, v_sb, v_sh, v_sn, o_sb, o_sh, o_sn;
  int blkq_shift, blkk_shift;
  float q_mult;
  int nsplit, tiles_per_split;   // filled in by launch_attn_few, like the next one
  FastDiv div_nsplit;
};
__host__ __device__ inline int64_t few_part_floats(int rows, int D) { return (int64_t)rows * D + (3 * rows + 3) / 4 * 4; }
// (at most one partial result per 128 keys: 32 rows of 524 bytes at head_dim 128, against the 32 KiB of an FP16 V panel; an FP8 panel
// has 16, and the launcher makes the ranges longer where they do not fit)
static_assert((kFewRows * 128 + 3 * kFewRows) * 4 <= 128 * 128 * 2 && (kFewRows * 64 + 3 * kFewRows) * 4 <= 128 * 64 * 2, "partials fit the panel region");
// Ranges of the keys, each of few_tiles_per_split() tiles; 0 where not even one range per pair fits.
inline int few_tiles_per_split(int B, int Hkv, int rows, int Skv, int D, int64_t part_bytes) {
  const int64_t ntiles = (Skv + 127) / 128, pairs = (int64_t)B * Hkv, want = (kFewWorkgroups + pairs - 1) / pairs;
  const int64_t room = part_bytes / (pairs * few_part_floats(rows, D) * 4);   // ranges per pair
  if (room < 1) return 0;
  const int64_t n = want < room ? want : room;
  return (int)((ntiles + n - 1) / n);
}
hipError_t launch_attn_few(FewArgs a, int dtype, int D, int pv, hipStream_t st);

struct AttnArgs {
  const int8_t* q;
  const int8_t* k;
  const uint8_t* vp;
  const float* qs;
  const float* ks;
  const float* vs;
  void* out;
  float* lse;
  int B, Hq, Hkv, Sq, Skv;
  int64_t q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, o_sb, o_sh, o_sn;
  int blkq, blkk;            // scale block sizes: powers of two (32, 64, 128)
  int blkq_shift, blkk_shift;  // their log2
  int qg_shift;              // log2 of the Q scales per block: 0, or 3 (eight interleaved scales: rows r, r + 8, ... share one)
  int k_interleave;          // 1: four interleaved K scales per block (scale t for the keys n with (n % 8) / 2 == t); host-side dispatch only
  int out_bf16;
  int nqt;  // q-tiles per sequence (fixed-length mode)
  // launch constants of the tile decode (filled in by finish_attn_args)
  int G;                    // q-heads per KV head
  int tier_shift;           // fixed-length mode, per-XCD tile order: log2 of the widest range of q-tiles; -1: plain order
  FastDiv div_G, div_Hkv, div_heads;   // heads = B*Hq (fixed-length) or Hq (packed)
  FastDiv div_range, div_last;         // full-attention tile order: q-tiles x heads-per-XCD of a range; width of the last range
  // packed mode (cu_q != nullptr)
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* cu_qblk;
  const int32_t* cu_kblk;
  const int32_t* cu_panel;
  const int32_t* ntiles;
  const int32_t* tiles;
  int64_t qs_sh, ks_sh, panel_sh;
  int total_q;
  // explicit mask (fixed-length mode only): [B, Hq, Sq, Skv] with element strides; kind 1 = bytes
  // (non-zero keeps the key), 2 = fp32 added to the base-2 logits
  const void* mask;
  int mask_kind;
  int64_t m_sb, m_sh, m_sm, m_sn;
  float mask_mult;          // additive masks are scaled by this before they are added
  const float* lse_offset;  // added to LSE2 per query row (same layout as lse) or null
  // fused Q quantisation: fp16/bf16 Q with the strides of q (q and qs are then unused)
  const void* q_raw;
  int q_is_bf16;
  float q_mult;
  const u16* q_dot_km;      // K mean [B, Hkv, D] (packed: [nseq, Hkv, D]) in the type of q, or null: its product with the scaled row joins the row's LSE2
  const uint8_t* mask_bits; // packed boolean mask (sage_common.h) or null: taken instead of `mask`
  const uint8_t* mask_seen;
  int mask_pb, mask_ph, mask_nqt, mask_ntk;
  int tile_rows;            // query rows per workgroup; host-side dispatch only
};

constexpr int kLargeTileRows = 256, kSmallTileRows = 128;   // query rows per workgroup: eight or four wavefronts of 32

hipError_t launch_quant_int8(const QuantArgs& a, int dtype, int max_rows, hipStream_t st);
int colstat_chunks(int L);
hipError_t launch_k_mean(const ColStatArgs& a, int dtype, void* km, hipStream_t st);
hipError_t launch_v_scale(const ColStatArgs& a, int dtype, float* vscale, hipStream_t st);
hipError_t launch_prep_v(const PrepVArgs& a, int dtype, int pv, int max_panels, hipStream_t st);
// Short fixed-length sequences: K mean + K quantiser + V scale + V panels in one launch (km_out / vscale_out take the statistics;
// qa.km is ignored and must be null).
hipError_t launch_prepass_small(const QuantArgs& qa, const PrepVArgs& va, int dtype, int pv, int smooth, void* km_out,
                                float* vscale_out, hipStream_t st);

// Packs a boolean mask [B, Hq, Sq, Skv] with element strides into the form of sage_common.h.
hipError_t launch_mask_pack(const MaskPackArgs& a, hipStream_t st);

// Several pre-passes in one launch: the jobs whose pointers are set, in the order of the members.  Jobs of one launch do not
// see each other's results.
constexpr int kFusedChunks = 8;   // chunks of a sequence whose statistics the quantiser and the panel job combine themselves
struct FusedPrepass {
  PlanArgs plan;          // if plan.plan
  ColStatArgs k_stat;     // if k_stat.partial: sums
  ColStatArgs v_stat;     // if v_stat.partial: abs-maxima
  QuantArgs k_quant;      // if k_quant.out
  QuantArgs q_quant;      // if q_quant.out
  PrepVArgs v_panels;     // if v_panels.panels
  MaskPackArgs mask;      // if mask.bits
};
// Whether one launch can run both quantisers (they share the rows per wavefront).
bool fused_quant_together(int D, int blk_a, int blk_b);
hipError_t launch_fused_prepass(const FusedPrepass& f, int dtype, int D, int pv, hipStream_t st);
// K mean / V scales from the per-chunk statistics a launch above has written (sequences of more than kFusedChunks chunks).
hipError_t launch_k_mean_finalize(const ColStatArgs& a, int dtype, void* km, hipStream_t st);
hipError_t launch_v_scale_finalize(const ColStatArgs& a, float* vscale, hipStream_t st);

// Fills in the launch constants of the tile decode from the dimensions already in `a` (B, Hq, Hkv, nqt, cu_q).
void finish_attn_args(AttnArgs& a, bool causal);
hipError_t launch_attn(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st);
hipError_t launch_attn_small(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st);
// Masks that the kernels of sage_attn_maskwide.hip take, rather than those of sage_attn_mask.hip (which gives the reasons).
inline bool mask_is_wide(int64_t m_sn, int kind, int Skv) { return m_sn == 1 && (kind == 1 || Skv >= 128); }
hipError_t launch_attn_masked(const AttnArgs& a, int D, int pv, int grid, hipStream_t st);
hipError_t launch_attn_masked_wide(const AttnArgs& a, int D, int pv, int grid, hipStream_t st);
hipError_t launch_attn_packed_mask(const AttnArgs& a, int D, int pv, int grid, hipStream_t st);
hipError_t launch_attn_qfused(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st);
hipError_t launch_attn_k16(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st);
hipError_t launch_attn_kinterleaved(const AttnArgs& a, int D, int pv, bool causal, int grid, hipStream_t st);
hipError_t launch_varlen_plan(const int32_t* cu_q, const int32_t* cu_k, int nseq, int total_q, int blkq, int blkk, int bm,
                              int bn, int causal, int32_t* plan, hipStream_t st);

}  // namespace sage
