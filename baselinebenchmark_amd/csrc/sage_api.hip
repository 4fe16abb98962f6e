// C ABI of libsage_mi355x.so (declared in include/sage_mi355x.h): argument validation with the
// reference's error classes, workspace carving, the one-call sageattn pipeline and the launch
// geometry of every kernel.  Nothing here allocates device memory or synchronises.
#include "sage_launch.h"
#include "../../include/sage_mi355x.h"

#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <cmath>
#include <cstdlib>

using namespace sage;

namespace {

thread_local char g_err[512] = "";
thread_local int g_tile_rows = 0;   // sage_last_tile_rows

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(SAGE_ELAUNCH, "%s: %s", what, hipGetErrorString(e));
}

inline size_t align_up(size_t x, size_t a = 256) { return (x + a - 1) / a * a; }

bool valid_blk_quant(int blk) { return blk == 16 || blk == 32 || blk == 64 || blk == 128; }
bool valid_blk_attn(int blk) { return blk == 16 || blk == 32 || blk == 64 || blk == 128; }
bool valid_blkk_attn(int blk) { return valid_blk_attn(blk); }
int ilog2(int x) { int r = 0; while ((1 << r) < x) r++; return r; }
// A Q block-size argument may carry SAGE_BLK_INTERLEAVE8: eight interleaved scales per block instead of one.
// ... or SAGE_BLK_INTERLEAVE4 (a K block size): four.  Both flags at once decode to 0 groups, which nothing accepts.
int blk_rows(int blk) { return blk > 0 ? (blk & ~(SAGE_BLK_INTERLEAVE8 | SAGE_BLK_INTERLEAVE4)) : blk; }
int blk_groups(int blk) {
  if (blk <= 0) return 1;
  const bool g8 = blk & SAGE_BLK_INTERLEAVE8, g4 = blk & SAGE_BLK_INTERLEAVE4;
  return g8 && g4 ? 0 : g8 ? 8 : g4 ? 4 : 1;
}

int check_common(int B, int H, int L, int D, int dtype) {
  if (B < 0 || H < 0 || L < 0) return fail(SAGE_EINVAL, "negative dimension (B=%d H=%d L=%d)", B, H, L);
  if (D != 64 && D != 128) return fail(SAGE_ENOTIMPL, "head_dim %d is not supported (64 or 128)", D);
  if (dtype != SAGE_DT_F16 && dtype != SAGE_DT_BF16) return fail(SAGE_ETYPE, "dtype flag %d is not fp16(0)/bf16(1)", dtype);
  return SAGE_OK;
}

int check_stride16(const char* name, int64_t sb, int64_t sh, int64_t sn, int esz, const void* p) {
  // 128-bit accesses: every row must start on a 16-byte boundary
  if ((sb * esz) % 16 || (sh * esz) % 16 || (sn * esz) % 16 || (reinterpret_cast<uintptr_t>(p) % 16))
    return fail(SAGE_EINVAL, "%s: base pointer and strides must be 16-byte aligned", name);
  return SAGE_OK;
}

}  // namespace

namespace sage {
int set_error(int code, const char* msg) { return fail(code, "%s", msg); }
}  // namespace sage

extern "C" {

const char* sage_backend_name(void) { return "mi355x_hip_int8_qk_fp8_fp16_pv"; }

const char* sage_last_error(void) { return g_err; }

int sage_last_tile_rows(void) { return g_tile_rows; }

}  // extern "C"

namespace {
constexpr int64_t kStatElements = (int64_t)56 << 20, kInputElements = (int64_t)20 << 20;
// What is read past the caches is faster by itself (sage_common.h) but found in none of them again.  Up to kStatElements elements, the
// tensors that a call takes statistics of are read through the caches: the quantiser, the panels or the few-rows kernel then find part of them in
// the last-level cache (256 MB).  Whole calls, bf16, past / through, us: 1 row, 32/8 heads, 8192 keys, K of 34 MB 30.9 / 29.7, 67 MB 48.6 / 47.8, 100 MB 82.2 /
// 79.4, 268 MB 149 / 153; 32 heads of 4096 rows (34 MB), FP16 P.V 142 / 140, FP8 (K and V) 113 / 112; 64 heads 272 / 274, FP8 212 / 215 (134 MB: not taken);
// 128 of them FP8 409 / 421; 220 of 1200 168.7 / 163.8.
// Up to kInputElements elements of K and V together the second reads go through the caches too, where the L2s still hold the first
// ones (past them, a line that others want is given up): with both, 31 heads of 2000 rows, head_dim 128, FP16 64.5 / 61.6, FP8 59.3 / 55.2, of 64 62.3 /
// 60.2; 7 of 4000, 64, 56.9 / 55.6.  So do those of the one-launch pre-pass, whose workgroups read each other's rows for their statistics: 52 of
// 600, FP8, 128, 39.4 / 36.7.  FP16 panels of head_dim 64 are then written through them as well: 15 of 4000 60.7 / 58.7, 31 of 2000 42.7 /
// 41.5; at 128 (28 of 1100 41.6 / 42.8), FP8 (15 of 2000 43.7 / 44.9) and INT8 K it is the slower.
bool statistics_stay(int64_t elements) { return elements <= kStatElements; }
bool inputs_stay(int64_t elements) { return elements <= kInputElements; }

struct RowDot {   // optional side output of the quantiser (see QuantArgs)
  const void* vec = nullptr;
  float* out = nullptr;
  int64_t sb = 0, sh = 0;
  int group = 1, total = 0;
};

// Checks a quantiser call and fills in its arguments; a.out stays null where there is nothing to do.
int quant_args(QuantArgs& a, const void* x, int8_t* out, float* scale, const void* km, int B, int H, int L, int D, int64_t x_sb,
               int64_t x_sh, int64_t x_sn, int64_t o_sb, int64_t o_sh, int64_t o_sn, int64_t km_sb, int64_t km_sh, int blk,
               float mult, int dtype, const int32_t* cu_seqlens, const int32_t* cu_blocks, int64_t scale_sh, const RowDot& dot) {
  memset(&a, 0, sizeof(a));
  if (int rc = check_common(B, H, L, D, dtype)) return rc;
  const int groups = blk_groups(blk);
  blk = blk_rows(blk);
  if (!valid_blk_quant(blk)) return fail(SAGE_ENOTIMPL, "quantisation block %d is not supported (16, 32, 64, 128)", blk);
  if (groups == 0) return fail(SAGE_EINVAL, "SAGE_BLK_INTERLEAVE8 and SAGE_BLK_INTERLEAVE4 exclude each other");
  if (groups > 1 && cu_seqlens) return fail(SAGE_ENOTIMPL, "interleaved scales are not supported for packed batches");
  if (groups == 4 && blk == 16) return fail(SAGE_ENOTIMPL, "four interleaved scales need blocks of 32, 64 or 128 rows");
  if (B == 0 || H == 0 || L == 0) return SAGE_OK;
  if (!x || !out || !scale) return fail(SAGE_EINVAL, "null tensor pointer");
  if (cu_seqlens && !cu_blocks) return fail(SAGE_EINVAL, "packed mode needs cu_blocks");
  if (int rc = check_stride16("x", x_sb, x_sh, x_sn, 2, x)) return rc;
  if (int rc = check_stride16("out", o_sb, o_sh, o_sn, 1, out)) return rc;
  if (km && int(check_stride16("km", km_sb, km_sh, 0, 2, km))) return SAGE_EINVAL;
  a.x = (const u16*)x; a.out = out; a.scale = scale; a.km = (const u16*)km;
  a.B = B; a.H = H; a.L = L; a.D = D;
  a.x_sb = x_sb; a.x_sh = x_sh; a.x_sn = x_sn; a.o_sb = o_sb; a.o_sh = o_sh; a.o_sn = o_sn;
  a.km_sb = km_sb; a.km_sh = km_sh; a.blk = blk; a.blk_shift = ilog2(blk); a.groups = groups; a.mult = mult;
  a.cu_seqlens = cu_seqlens; a.cu_blocks = cu_blocks; a.scale_sh = scale_sh;
  a.dotv = (const u16*)dot.vec; a.dot_out = dot.out; a.dv_sb = dot.sb; a.dv_sh = dot.sh; a.dv_group = dot.group;
  a.dot_total = dot.total;
  return SAGE_OK;
}
}  // namespace

extern "C" {

int sage_quant_int8(const void* x, int8_t* out, float* scale, const void* km, int B, int H, int L, int D, int64_t x_sb,
                    int64_t x_sh, int64_t x_sn, int64_t o_sb, int64_t o_sh, int64_t o_sn, int64_t km_sb, int64_t km_sh,
                    int blk, float mult, int dtype, const int32_t* cu_seqlens, const int32_t* cu_blocks,
                    int64_t scale_sh, sage_stream_t stream) {
  QuantArgs a;
  if (int rc = quant_args(a, x, out, scale, km, B, H, L, D, x_sb, x_sh, x_sn, o_sb, o_sh, o_sn, km_sb, km_sh, blk, mult, dtype,
                          cu_seqlens, cu_blocks, scale_sh, RowDot())) return rc;
  if (!a.out) return SAGE_OK;
  hipError_t e = launch_quant_int8(a, dtype, L, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sage_quant_int8");
  return SAGE_OK;
}

size_t sage_k_mean_workspace_bytes(int B, int H, int L, int D) {
  return align_up((size_t)B * H * colstat_chunks(L) * D * sizeof(double));
}

int sage_k_mean(const void* k, void* km, void* workspace, size_t workspace_bytes, int B, int H, int L, int D, int64_t k_sb,
                int64_t k_sh, int64_t k_sn, int dtype, const int32_t* cu_seqlens, sage_stream_t stream) {
  if (int rc = check_common(B, H, L, D, dtype)) return rc;
  if (B == 0 || H == 0) return SAGE_OK;
  if (!k || !km || !workspace) return fail(SAGE_EINVAL, "null tensor pointer");
  if (workspace_bytes < sage_k_mean_workspace_bytes(B, H, L, D)) return fail(SAGE_EWORKSPACE, "k_mean workspace too small");
  if (int rc = check_stride16("k", k_sb, k_sh, k_sn, 2, k)) return rc;
  ColStatArgs a;
  a.x = (const u16*)k; a.partial = workspace; a.B = B; a.H = H; a.L = L; a.D = D;
  a.x_sb = k_sb; a.x_sh = k_sh; a.x_sn = k_sn; a.nchunk = colstat_chunks(L); a.cu_seqlens = cu_seqlens;
  a.cached = !cu_seqlens && statistics_stay((int64_t)B * H * L * D);   // (its quantiser comes next)
  if (a.nchunk == 0) a.nchunk = 1;  // L == 0: the finalize kernel still writes zeros
  hipError_t e = launch_k_mean(a, dtype, km, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sage_k_mean");
  return SAGE_OK;
}

size_t sage_prep_v_workspace_bytes(int B, int H, int L, int D, int pv_mode) {
  if (pv_mode != SAGE_PV_FP8) return 0;
  int nc = colstat_chunks(L);
  return align_up((size_t)B * H * (nc ? nc : 1) * D * sizeof(float));
}

size_t sage_v_panel_bytes(int B, int H, int L, int D, int pv_mode) {
  size_t np = (L + SAGE_PANEL_ROWS - 1) / SAGE_PANEL_ROWS;
  return (size_t)B * H * np * SAGE_PANEL_ROWS * D * (pv_mode == SAGE_PV_FP8 ? 1 : 2);
}

int sage_prep_v(const void* v, void* panels, float* v_scale, void* workspace, size_t workspace_bytes, int B, int H, int L,
                int D, int64_t v_sb, int64_t v_sh, int64_t v_sn, int dtype, int pv_mode, const int32_t* cu_seqlens,
                const int32_t* cu_panels, int64_t panel_sh, sage_stream_t stream) {
  if (int rc = check_common(B, H, L, D, dtype)) return rc;
  if (pv_mode != SAGE_PV_FP16 && pv_mode != SAGE_PV_FP8) return fail(SAGE_EINVAL, "pv_mode %d unknown", pv_mode);
  if (B == 0 || H == 0 || L == 0) return SAGE_OK;
  if (!v || !panels) return fail(SAGE_EINVAL, "null tensor pointer");
  if (cu_seqlens && !cu_panels) return fail(SAGE_EINVAL, "packed mode needs cu_panels");
  if (int rc = check_stride16("v", v_sb, v_sh, v_sn, 2, v)) return rc;
  if (reinterpret_cast<uintptr_t>(panels) % 16) return fail(SAGE_EINVAL, "panels must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  if (pv_mode == SAGE_PV_FP8) {
    if (!v_scale || !workspace) return fail(SAGE_EINVAL, "fp8 mode needs v_scale and workspace");
    if (workspace_bytes < sage_prep_v_workspace_bytes(B, H, L, D, pv_mode)) return fail(SAGE_EWORKSPACE, "prep_v workspace too small");
    ColStatArgs c;
    c.x = (const u16*)v; c.partial = workspace; c.B = B; c.H = H; c.L = L; c.D = D;
    c.x_sb = v_sb; c.x_sh = v_sh; c.x_sn = v_sn; c.nchunk = colstat_chunks(L); c.cu_seqlens = cu_seqlens;
    c.cached = !cu_seqlens && statistics_stay((int64_t)B * H * L * D);
    hipError_t e = launch_v_scale(c, dtype, v_scale, st);
    if (e != hipSuccess) return hip_fail(e, "sage_prep_v(scale)");
  }
  PrepVArgs a;
  memset(&a, 0, sizeof(a));
  a.v = (const u16*)v; a.panels = (uint8_t*)panels; a.vscale = v_scale; a.B = B; a.H = H; a.L = L; a.D = D;
  a.v_sb = v_sb; a.v_sh = v_sh; a.v_sn = v_sn; a.cu_seqlens = cu_seqlens; a.cu_panels = cu_panels; a.panel_sh = panel_sh;
  hipError_t e = launch_prep_v(a, dtype, pv_mode, (L + SAGE_PANEL_ROWS - 1) / SAGE_PANEL_ROWS, st);
  if (e != hipSuccess) return hip_fail(e, "sage_prep_v");
  return SAGE_OK;
}

size_t sage_varlen_plan_ints(int nseq, int total_q) { return (size_t)plan_layout(nseq, total_q).total; }

void sage_varlen_plan_offsets(int nseq, int total_q, int64_t offs[5]) {
  SagePlanLayout L = plan_layout(nseq, total_q);
  offs[0] = L.cu_qblk; offs[1] = L.cu_kblk; offs[2] = L.cu_panel; offs[3] = L.ntiles; offs[4] = L.tiles;
}

int sage_varlen_plan(const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int nseq, int total_q, int blkq, int blkk,
                     int is_causal, int32_t* plan, size_t plan_ints, sage_stream_t stream) {
  if (nseq <= 0 || nseq > 32767) return fail(SAGE_EINVAL, "number of sequences %d out of range (1..32767)", nseq);
  if (!cu_seqlens_q || !cu_seqlens_k || !plan) return fail(SAGE_EINVAL, "null pointer");
  if (!valid_blk_quant(blkq) || !valid_blk_quant(blkk)) return fail(SAGE_ENOTIMPL, "block sizes %d/%d not supported", blkq, blkk);
  if (plan_ints < sage_varlen_plan_ints(nseq, total_q)) return fail(SAGE_EWORKSPACE, "plan buffer too small");
  hipError_t e = launch_varlen_plan(cu_seqlens_q, cu_seqlens_k, nseq, total_q, blkq, blkk, kLargeTileRows, 64, is_causal, plan,
                                    (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sage_varlen_plan");
  return SAGE_OK;
}

}  // extern "C"

namespace {
struct QRawArg {   // fp16/bf16 Q to be quantised by the attention kernel itself (q / q_scale are then ignored)
  const void* ptr = nullptr;
  int dtype = 0;
  float mult = 1.0f;
  const void* dot_km = nullptr;   // K mean [B, Hkv, D] in q's type: its product with each scaled row is added to the row's LSE
};

struct MaskArg {
  const void* ptr = nullptr;
  int kind = 0;
  int64_t sb = 0, sh = 0, sm = 0, sn = 0;
  const uint8_t* bits = nullptr;   // packed form of a boolean mask (with `planes`), taken instead of ptr
  const uint8_t* seen = nullptr;
  MaskPlanes planes = {};
  float mult = 1.0f;   // additive masks are multiplied by this (1 for base-2 units, log2(e) for natural units)
};

// Query rows per workgroup: 256 (eight wavefronts, two groups in step on one tile stream, sage_attn.hip) or 128 (four wavefronts,
// two or three workgroups to a compute unit, sage_attn_small.hip).  The results are the same bits; the line between them is cost.
// The small ones let a workgroup's prologue and epilogue run under another's tiles, leave fewer padded rows and fill the chip with half
// the rows, but fetch every K and V tile twice as often.  Which is the faster depends on how many rounds of the chip either makes: 7872 whole calls
// without a mask (2 head_dims, both P.V, full and causal, with and without LSE, the three kinds of K scales, 300 to 8000 rows, 150 to 1540 q-tiles of
// 256 rows; bf16) are 0.1 % longer than the better size by the rules below, 48 of them more than 2 % longer than with 256 rows (7.4 % always with 256); of 5808
// others of the same ranges 56 are, at most 6 %.
// Some of them, and what the rules do not compare, whole calls, 256 rows / 128 rows, us:
//   not filled (128 q-tiles of 256 rows and fewer): 8 heads of 2000 rows, head_dim 128, FP16 full 54.0 / 50.1, causal 54.0 / 50.1, FP8 47.1 / 43.1; of 4000
//     89.4 / 85.6, 89.3 / 84.5, 70.0 / 64.7; head_dim 64 FP16 of 4000 65.0 / 58.4; interleaved, FP8, causal 12 of 2000 38 / 37, but full, where the
//     small kernel keeps 36 bytes a lane in scratch memory, 33 of 700 27.0 / 27.8;
//   packed, 32/8 heads, the length between mean and maximum: head_dim 64, causal FP16, 200 prompts of 8..300 259 / 162, 96 of 16..512 208 / 146, 16 of
//     512..8000 1544 / 1434, 8 of 4000..16000 4345 / 4006, full FP8 5158 / 4910: always; head_dim 128, causal FP16 64 of 16..1024 424 / 370, 40 of
//     200..2000 680 / 635, 30 of 1000..4000 1822 / 1840, FP8 1366 / 1302, 16 of 512..8000 1666 / 1661, full FP16 40 of 200..2000 988 / 972, FP8 30 of
//     1000..4000 2124 / 2119;
//   masks: one bias per head, 2 x 16 heads of 1000 rows, head_dim 64 69 / 49, 128 82 / 60, 1 x 4 of 6000 325 / 211, 363 / 232; documents, head_dim 64, 2
//     x 16 of 1500 53 / 50, 4 x 32 123 / 110, FP8 128 1 x 32 of 2200 133 / 101; padding, head_dim 64, 1 x 32 of 2200 109 / 85; boolean ones over FP16 P.V
//     by rounds, as without a mask: head_dim 128, in one round, 2 x 16 of 1500 70 / 75 (one mask per head 101 / 106), in two, 67 of 1500 115 / 119, 42 of 3000 175 / 182, but 33
//     of 2078 139 / 125; head_dim 64, in one round, padding 22 of 2078 63 / 68, 12 of 4200 107 / 115, 33 of 1500 60 / 60, one mask per head 22 of 2078 105 / 110, but
//     documents 27 of 1500 48 / 46, 22 of 2078 59 / 58, and in two rounds padding 33 of 2078 105 / 82, one mask per head 175 / 145.
enum MaskClass { kNoMask, kKeepMask, kBiasMask, kOtherMask };   // boolean (in bits, or contiguous keys), additive with contiguous keys, other strides
struct TileRows { int B, Hq, Sq, Skv, D, pv, causal, blkk, kgroups; bool lse; MaskClass mask; bool packed; int total_q, total_k; };

// Calls that are not causal: all workgroups of a size cost the same.  A round of the chip of 256-row workgroups takes as long as their tiles
// and `hidden` tiles more than small ones (what of a prologue and an epilogue does not run beside another workgroup; less of it in the
// first round, where compute units with one small workgroup wait for those with two); one, two or three small ones together on a compute unit take
// `together` times their tiles.  Fitted to the calls above.  Examples, 256 / 128 rows, us: head_dim 128, FP16, 75 heads of 1500 rows 116 / 126, 37 of 1700 102 / 96, 47 of
// 2600 203 / 186, FP8 73 of 1700 112 / 118, 47 of 2600 158 / 143; head_dim 64, FP16, 18 of 4200 136 / 110, 32 of 3500 125 / 129, FP8 9 of 8000 160 / 125, 14 of 8000
// 168 / 180, 200 of 700 66 / 55.
struct RoundCost { float together[3], hidden; };
constexpr RoundCost kRoundCost128[2] = {{{0.68f, 1.25f, 0}, 1.6f}, {{0.80f, 1.22f, 0}, 1.8f}};   // FP16, FP8 P.V
constexpr RoundCost kRoundCost64[2] = {{{0.62f, 1.10f, 1.48f}, 0.9f}, {{0.65f, 1.08f, 1.46f}, 0.6f}};
constexpr RoundCost kRoundCost64Fp8Lse = {{0.50f, 1.04f, 1.33f}, 0.2f}, kRoundCost64Fp8Fine = {{0.78f, 1.15f, 1.46f}, 0.4f};   // (fine: see below)
bool fewer_rounds_pay(const RoundCost& cost, int per_cu, int64_t large, int64_t small, int Skv) {
  constexpr int kComputeUnits = 256;
  const int64_t rounds = (large + kComputeUnits - 1) / kComputeUnits, deepest = (small + kComputeUnits - 1) / kComputeUnits;
  const int rest = (int)(deepest % per_cu);
  const float tiles = Skv / 128.0f, small_tiles = (float)(deepest / per_cu) * cost.together[per_cu - 1] + (rest ? cost.together[rest - 1] : 0);
  return small_tiles * tiles <= rounds * tiles + (rounds == 1 ? 0.6f : (float)rounds) * cost.hidden;
}

bool small_tiles_pay(const TileRows& c) {
  const bool fine = c.kgroups != 1 || c.blkk == 16, fp8 = c.pv == SAGE_PV_FP8;   // fine: two or four K scales per 32 keys
  if (c.mask == kOtherMask || (c.mask != kNoMask && fine)) return false;   // (no such variants)
  if (c.packed && c.blkk == 16) return false;   // (their plan stays the one of sage_varlen_plan)
  if (c.packed && c.total_q >= kSmallTileRows << 16) return false;   // (a plan has 16 bits for the q-tile of a sequence)
  if (c.packed) {
    if (c.D == 64 || (fp8 && c.lse)) return true;
    const int64_t keys = ((int64_t)c.total_k / c.B + c.Skv) / 2;
    return keys <= (fp8 ? 1800 : 1500) * (c.causal ? 2 : 1);
  }
  const int64_t heads = (int64_t)c.B * c.Hq, large = heads * ((c.Sq + kLargeTileRows - 1) / kLargeTileRows);
  if (c.mask != kNoMask) {
    if (c.mask != kKeepMask || fp8 || large <= 128) return true;
    if (c.D == 64) return large > 256 || c.Skv <= 1792;
    return fewer_rounds_pay(kRoundCost128[0], 2, large, heads * ((c.Sq + kSmallTileRows - 1) / kSmallTileRows), c.Skv);
  }
  // FP8 P.V with LSE: the exact exponentials are the longer half, and nothing is lost by fetching a tile twice; full calls of head_dim 64 in
  // one round of the chip are the exception.
  if (fp8 && c.lse && (c.D == 128 || c.kgroups != 1 || c.causal)) return true;
  if (fp8 && c.D == 64 && !c.lse) {
    if (c.kgroups != 1 && !c.causal && large <= 128) return false;                  // (scratch memory, see above)
    if (c.blkk == 16 && c.causal && large > 128 && large <= 256) return false;      // 32 heads of 2000 rows 44.3 / 45.5, 27 of 1400 36.5 / 37.6
  }
  if (large <= 128) return true;
  if (!c.causal) {
    const RoundCost& cost = c.D == 128 ? kRoundCost128[fp8] : !fp8 ? kRoundCost64[0] : c.lse ? kRoundCost64Fp8Lse : fine ? kRoundCost64Fp8Fine : kRoundCost64[1];
    return fewer_rounds_pay(cost, c.D == 64 ? 3 : 2, large, heads * ((c.Sq + kSmallTileRows - 1) / kSmallTileRows), c.Skv);
  }
  // Causal ones differ by themselves.  Up to five quarters of a round the small ones spread the longest tiles over compute units that have
  // nothing else; in the second round, 256 rows pair a long tile with a short one and come out even; beyond, the tiles' cost decides, at half
  // the keys.  256 / 128 rows, us: head_dim 128, FP16, 12 heads of 5600 rows 127 / 122, 32 of 3500 114 / 124, 75 of 1500 86 / 88, 100 of 1500
  // 109 / 104, 85 of 2300 159 / 162, 73 of 3500 258 / 274, FP8 12 of 5600 101 / 98, 73 of 3500 205 / 227, with K blocks of 16 100 of 2300 167 / 158; head_dim 64, FP16, 20 of 5600
  // 104 / 107, 47 of 5600 237 / 218, FP8 32 of 3000 53 / 55, 64 of 3000 95 / 92.
  if (c.D == 128) return c.Skv <= (large <= 320 ? 8192 : large <= 512 ? 1400 : c.blkk == 16 ? 2700 : 2048);
  return large <= 320 || (!fp8 && fine) || c.Skv <= (large <= 512 ? (fp8 ? 2700 : 3000) : fp8 ? 8192 : 16384);
}
int tile_rows(const TileRows& c) {
#ifdef SAGE_TIMING   // (the timers that are read are those of the workgroups of 256 rows, of calls without a mask and interleaved scales)
  if (c.mask == kNoMask && c.kgroups == 1) return kLargeTileRows;
#endif
  return small_tiles_pay(c) ? kSmallTileRows : kLargeTileRows;
}
// ... of the entry points that take a plan of the caller's, whose q-tiles have 256 rows.
int public_tile_rows(int B, int Hq, int Sq, int Skv, int D, int pv_mode, int is_causal, int blkk, const float* lse, const int32_t* cu_seqlens_q) {
  if (cu_seqlens_q) return kLargeTileRows;
  return tile_rows({B, Hq, Sq, Skv, D, pv_mode, is_causal, blk_rows(blkk), blk_groups(blkk), lse != nullptr, kNoMask, false, 0, 0});
}

MaskClass mask_class(const MaskArg& m, int Skv) {
  if (!m.ptr) return kNoMask;
  if (!m.bits && !mask_is_wide(m.sn, m.kind, Skv)) return kOtherMask;
  return m.kind == SAGE_MASK_BOOL ? kKeepMask : kBiasMask;
}

int attn_impl(const int8_t* q, const int8_t* k, const void* v_panels, const float* q_scale, const float* k_scale,
              const float* v_scale, void* out, float* lse, int B, int Hq, int Hkv, int Sq, int Skv, int D, int64_t q_sb,
              int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn, int64_t o_sb, int64_t o_sh,
              int64_t o_sn, int blkq, int blkk, int is_causal, int pv_mode, int out_dtype, const int32_t* cu_seqlens_q,
              const int32_t* cu_seqlens_k, const int32_t* plan, int total_q, int64_t q_scale_sh, int64_t k_scale_sh,
              int64_t panel_sh, const MaskArg& mask, const float* lse_offset, const QRawArg& qraw, int tile_rows, sage_stream_t stream) {
  g_tile_rows = 0;
  if (int rc = check_common(B, Hq, Sq, D, out_dtype)) return rc;
  if (Hkv <= 0 || Hq % Hkv) return fail(SAGE_EINVAL, "query heads (%d) must be divisible by KV heads (%d)", Hq, Hkv);
  if (Skv < 0) return fail(SAGE_EINVAL, "negative kv length");
  if (pv_mode != SAGE_PV_FP16 && pv_mode != SAGE_PV_FP8) return fail(SAGE_EINVAL, "pv_mode %d unknown", pv_mode);
  const int qgroups = blk_groups(blkq), kgroups = blk_groups(blkk);
  blkq = blk_rows(blkq);
  blkk = blk_rows(blkk);
  if (!valid_blk_attn(blkq) || !valid_blkk_attn(blkk))
    return fail(SAGE_ENOTIMPL, "attention needs Q and K scale blocks of 16, 32, 64 or 128 rows (got %d/%d)", blkq, blkk);
  if ((qgroups != 1 && qgroups != 8) || (kgroups != 1 && kgroups != 4))
    return fail(SAGE_ENOTIMPL, "Q scale blocks take SAGE_BLK_INTERLEAVE8, K scale blocks SAGE_BLK_INTERLEAVE4");
  if ((qgroups > 1 || kgroups > 1) && cu_seqlens_q) return fail(SAGE_ENOTIMPL, "interleaved scales are not supported for packed batches");
  if (qgroups > 1 && qraw.ptr) return fail(SAGE_ENOTIMPL, "interleaved Q scales need the standalone Q quantiser (sage_quant_int8)");
  if (kgroups > 1 && blkk == 16) return fail(SAGE_ENOTIMPL, "interleaved K scales need blocks of 32, 64 or 128 keys");
  if (B == 0 || Hq == 0 || Sq == 0) return SAGE_OK;
  if (!out || (Skv > 0 && (!k || !v_panels || !k_scale))) return fail(SAGE_EINVAL, "null tensor pointer");
  if (!qraw.ptr && (!q || !q_scale)) return fail(SAGE_EINVAL, "null tensor pointer");
  if (qraw.ptr && mask.ptr) return fail(SAGE_ENOTIMPL, "fused Q quantisation: not with an explicit mask");
  if (pv_mode == SAGE_PV_FP8 && !v_scale) return fail(SAGE_EINVAL, "fp8 P.V needs v_scale");
  if (int rc = check_stride16("q", q_sb, q_sh, q_sn, qraw.ptr ? 2 : 1, qraw.ptr ? qraw.ptr : q)) return rc;
  if (int rc = check_stride16("k", k_sb, k_sh, k_sn, 1, k)) return rc;
  if (int rc = check_stride16("out", o_sb, o_sh, o_sn, 2, out)) return rc;   // rows are stored 16 bytes per lane
  // tile loads address a row of one (batch, head) slice with 32-bit byte offsets
  if ((int64_t)Skv * k_sn >= 0x7fffffff || (qraw.ptr && (int64_t)Sq * q_sn * 2 >= 0x7fffffff))
    return fail(SAGE_ENOTIMPL, "a (batch, head) slice of q or k spans 2 GiB or more");
  const bool packed = cu_seqlens_q != nullptr;
  if (mask.ptr) {
    if (mask.kind != SAGE_MASK_BOOL && mask.kind != SAGE_MASK_ADDITIVE) return fail(SAGE_EINVAL, "mask kind %d unknown", mask.kind);
    if (packed) return fail(SAGE_ENOTIMPL, "an explicit mask is not supported for packed batches");
    if (is_causal) return fail(SAGE_ENOTIMPL, "an explicit mask cannot be combined with is_causal");
    if (mask.kind == SAGE_MASK_ADDITIVE && reinterpret_cast<uintptr_t>(mask.ptr) % 4) return fail(SAGE_EINVAL, "additive mask must be 4-byte aligned");
  }
  if (packed && (!cu_seqlens_k || !plan)) return fail(SAGE_EINVAL, "packed mode needs cu_seqlens_k and plan");
  if (packed && B > 32767) return fail(SAGE_EINVAL, "too many sequences");
  const int BM = tile_rows;
  AttnArgs a;
  memset(&a, 0, sizeof(a));
  a.tile_rows = BM;
  a.q = q; a.k = k; a.vp = (const uint8_t*)v_panels; a.qs = q_scale; a.ks = k_scale; a.vs = v_scale;
  a.out = out; a.lse = lse;
  a.B = B; a.Hq = Hq; a.Hkv = Hkv; a.Sq = Sq; a.Skv = Skv;
  a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.o_sb = o_sb; a.o_sh = o_sh; a.o_sn = o_sn;
  a.blkq = blkq; a.blkk = blkk; a.blkq_shift = ilog2(blkq); a.blkk_shift = ilog2(blkk); a.qg_shift = qgroups == 8 ? 3 : 0; a.k_interleave = kgroups == 4;
  a.out_bf16 = out_dtype == SAGE_DT_BF16;
  a.nqt = (Sq + BM - 1) / BM;
  a.mask = mask.ptr; a.mask_kind = mask.kind; a.m_sb = mask.sb; a.m_sh = mask.sh; a.m_sm = mask.sm; a.m_sn = mask.sn;
  a.mask_bits = mask.bits; a.mask_seen = mask.seen;
  a.mask_pb = mask.planes.pb; a.mask_ph = mask.planes.ph; a.mask_nqt = mask.planes.nqt; a.mask_ntk = mask.planes.ntk;
  a.mask_mult = mask.mult; a.lse_offset = lse_offset;
  a.q_raw = qraw.ptr; a.q_is_bf16 = qraw.dtype == SAGE_DT_BF16; a.q_mult = qraw.mult; a.q_dot_km = (const u16*)qraw.dot_km;
  int64_t grid;
  if (packed) {
    SagePlanLayout L = plan_layout(B, total_q);
    a.cu_q = cu_seqlens_q; a.cu_k = cu_seqlens_k;
    a.cu_qblk = plan + L.cu_qblk; a.cu_kblk = plan + L.cu_kblk; a.cu_panel = plan + L.cu_panel;
    a.ntiles = plan + L.ntiles; a.tiles = plan + L.tiles;
    a.qs_sh = q_scale_sh; a.ks_sh = k_scale_sh; a.panel_sh = panel_sh; a.total_q = total_q;
    grid = ((int64_t)total_q / BM + B) * Hq;  // upper bound on tiles; surplus workgroups exit at once
  } else {
    grid = (int64_t)a.nqt * B * Hq;
  }
  if (grid > 0x7fffffff) return fail(SAGE_EINVAL, "too many tiles for one launch");
  finish_attn_args(a, is_causal != 0);
  hipError_t e = launch_attn(a, D, pv_mode, is_causal != 0, (int)grid, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sage_attn_fwd");
  g_tile_rows = BM;
  return SAGE_OK;
}
}  // namespace

extern "C" {

int sage_attn_fwd(const int8_t* q, const int8_t* k, const void* v_panels, const float* q_scale, const float* k_scale,
                  const float* v_scale, void* out, float* lse, int B, int Hq, int Hkv, int Sq, int Skv, int D, int64_t q_sb,
                  int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn, int64_t o_sb, int64_t o_sh,
                  int64_t o_sn, int blkq, int blkk, int is_causal, int pv_mode, int out_dtype, const int32_t* cu_seqlens_q,
                  const int32_t* cu_seqlens_k, const int32_t* plan, int total_q, int64_t q_scale_sh, int64_t k_scale_sh,
                  int64_t panel_sh, sage_stream_t stream) {
  const int rows = public_tile_rows(B, Hq, Sq, Skv, D, pv_mode, is_causal, blkk, lse, cu_seqlens_q);
  return attn_impl(q, k, v_panels, q_scale, k_scale, v_scale, out, lse, B, Hq, Hkv, Sq, Skv, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, o_sb, o_sh, o_sn, blkq, blkk, is_causal, pv_mode, out_dtype, cu_seqlens_q, cu_seqlens_k, plan, total_q, q_scale_sh, k_scale_sh, panel_sh, MaskArg(), nullptr, QRawArg(), rows, stream);
}

int sage_attn_fwd_qfused(const void* q, int q_dtype, double sm_scale, const int8_t* k, const void* v_panels,
                         const float* k_scale, const float* v_scale, void* out, float* lse, int B, int Hq, int Hkv, int Sq,
                         int Skv, int D, int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                         int64_t o_sb, int64_t o_sh, int64_t o_sn, int blkq, int blkk, int is_causal, int pv_mode,
                         int out_dtype, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, const int32_t* plan,
                         int total_q, int64_t k_scale_sh, int64_t panel_sh, sage_stream_t stream) {
  if (q_dtype != SAGE_DT_F16 && q_dtype != SAGE_DT_BF16) return fail(SAGE_ETYPE, "q dtype flag %d is not fp16(0)/bf16(1)", q_dtype);
  if (!q) return fail(SAGE_EINVAL, "null tensor pointer");
  QRawArg qr;
  qr.ptr = q; qr.dtype = q_dtype; qr.mult = (float)((sm_scale > 0 ? sm_scale : 1.0 / sqrt((double)D)) * 1.44269504);
  const int rows = public_tile_rows(B, Hq, Sq, Skv, D, pv_mode, is_causal, blkk, lse, cu_seqlens_q);
  return attn_impl(nullptr, k, v_panels, nullptr, k_scale, v_scale, out, lse, B, Hq, Hkv, Sq, Skv, D, q_sb, q_sh, q_sn, k_sb,
                   k_sh, k_sn, o_sb, o_sh, o_sn, blkq, blkk, is_causal, pv_mode, out_dtype, cu_seqlens_q, cu_seqlens_k, plan,
                   total_q, 0, k_scale_sh, panel_sh, MaskArg(), nullptr, qr, rows, stream);
}

int sage_attn_fwd_masked(const int8_t* q, const int8_t* k, const void* v_panels, const float* q_scale, const float* k_scale,
                         const float* v_scale, void* out, float* lse, int B, int Hq, int Hkv, int Sq, int Skv, int D,
                         int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn, int64_t o_sb,
                         int64_t o_sh, int64_t o_sn, int blkq, int blkk, int pv_mode, int out_dtype, const void* attn_mask,
                         int mask_kind, int64_t m_sb, int64_t m_sh, int64_t m_sm, int64_t m_sn, sage_stream_t stream) {
  if (!attn_mask) return fail(SAGE_EINVAL, "null mask");
  MaskArg m;
  m.ptr = attn_mask; m.kind = mask_kind; m.sb = m_sb; m.sh = m_sh; m.sm = m_sm; m.sn = m_sn;
  const int rows = tile_rows({B, Hq, Sq, Skv, D, pv_mode, 0, blk_rows(blkk), blk_groups(blkk), lse != nullptr, mask_class(m, Skv), false, 0, 0});
  return attn_impl(q, k, v_panels, q_scale, k_scale, v_scale, out, lse, B, Hq, Hkv, Sq, Skv, D, q_sb, q_sh, q_sn, k_sb, k_sh,
                   k_sn, o_sb, o_sh, o_sn, blkq, blkk, 0, pv_mode, out_dtype, nullptr, nullptr, nullptr, 0, 0, 0, 0, m, nullptr,
                   QRawArg(), rows, stream);
}

// ---- one-call pipeline --------------------------------------------------------------------
namespace {
// Up to this many keys per sequence the pre-passes run as one launch whose workgroups read their sequence's statistics themselves
// (sage_quant.hip: prepass_small_kernel) instead of two launches, statistics first ...
constexpr int kSmallPrepassRows = 1024;
// ... and up to this many element reads, where a K workgroup reads its sequence for the mean and a V panel for the scales, and a tensor without
// a statistic is read once.  More reads pay where two statistics would be two passes.  Whole calls in bf16, one launch / two, us:
//   mean alone (FP16 P.V): 20 M reads (72 heads of 452 rows, head_dim 128) 39.0 / 39.1; 21 M (96 of 590, 64) 39.9 / 40.1; 24 M (256 of 384, 64) 38.4 /
//   42.7; 23 M (24 of 648) 57.2 / 55.5; 27 M (32 of 852) 73.0 / 70.6; 29 M (96 of 704, 64) 49.6 / 48.1; 40 M (256 of 512, 64) 58.5 / 51.7;
//   scales alone (FP8, keys as they are): 25 M (32 of 795) 32.6 / 35.1; 27 M (96 of 647, 64) 38.8 / 40.5; 35 M (256 of 443, 64) 45.1 / 44.4;
//   both: 36 M (48 of 505) 29.9 / 33.9, (32 of 622) 33.0 / 33.3; 40 M (96 of 380) 34.0 / 36.6; 44 M (64 of 809, 64) 73.1 / 70.8; 47 M (96 of 671, 64)
//   32.3 / 31.4; 61 M (64 of 983, 64) 41.6 / 33.3;
//   neither: 10 M (48 of 832) 35.5 / 36.8: no reads twice, one launch either way, the smaller kernel is the faster.
constexpr int64_t small_prepass_reads(bool mean, bool scales) { return (int64_t)(mean && scales ? 42 : scales ? 32 : 24) << 20; }
// ... in this many heads: 12288 of a key, head_dim 64, 374 / 363; 16384 of 8 525 / 496; 8192 of 16 251 / 251, FP8 235 / 242.
constexpr int64_t kSmallPrepassHeads = 8192;
// A few query rows (sage_attn_few.hip) take at most three launches, some 2.5 us of host time more than the two of the tiled kernel behind
// the one-launch pre-pass, which is as fast as that as long as its workgroups (one per query head; measured with tiles of 256 rows, one
// to a compute unit) are one round of the chip, the keys of a head are few and so are the re-reads of the pre-pass.  Past one round the rows
// count: the few-rows kernel writes and reads FP32 results of every row.  Whole calls, K blocks of 64, bf16, tiled / few rows in us.
// FP16 P.V, up to 16 rows: 8 heads of 768 keys, head_dim 64, 19.9 / 20.2, of 900 23.3 / 19.9; head_dim 128, of 257 18.6 / 19.5, of 512 21.0 /
// 19.9; 64 of 256 (12 M reads) 18.7 / 19.5, 128 of 192 (15 M) 20.9 / 19.5; 320 of 64 26.8 / 19.1, head_dim 64 19.4 / 19.8, 640 of 64 27.5 /
// 18.9; 512 heads on 128 KV heads of 128, head_dim 64, 17.4 / 19.7, 1024 on 256 28.6 / 19.4.  20, 24 and 32 rows, head_dim 64: 256 heads of 256
// keys (16 M) 21.3 / 21.0, 21.1 / 22.2, 21.4 / 25.9; 1024 of 64 38.3 / 36.4, 38.0 / 39.3, 38.4 / 45.0.
// FP8 P.V, 1 and 16 rows: head_dim 128, 8 heads of 768 keys 23.2 / 25.1 and 23.2 / 27.0, of 900 27.7 / 25.4 and 27.5 / 26.7; 32 of 512 (24 M)
// 25.1 / 26.7 and 25.2 / 27.4; 16 of 768 (27 M) 28.8 / 26.7 and 28.8 / 27.9; 512 of 64 26.4 / 24.6 and 26.9 / 30.9; 1024 of 16 45.9 / 36.6 and
// 46.7 / 48.0; 2048 of 16 86.2 / 55.7 and 86.7 / 80.5.
bool tiled_beats_few_rows(int pv_mode, int D, int64_t rows, int Sq, int64_t query_heads, int Skv, int64_t group_reads) {
  const bool apart = rows == Sq, many = apart && rows > 20;   // apart: every query head has a KV head of its own
  const int64_t mega = 1 << 20;
  if (Skv > kSmallPrepassRows) return false;
  if (pv_mode == SAGE_PV_FP16) {
    if ((int64_t)Skv * D > 48 * 1024 || group_reads > (many ? 20 : 12) * mega) return false;
    return many || query_heads <= (D == 64 ? 512 : 256);
  }
  if ((int64_t)Skv * D > 896 * 128 || group_reads > 24 * mega) return false;
  return query_heads <= (apart && rows > 8 ? 1024 : D == 64 ? 512 : 256);
}
// Few keys in great number: the FP32 results of a KV head's rows are written and read again, the tiled kernel with one
// query head per KV head launches no more workgroups, and at head_dim 128 it wins where those bytes outweigh K and V.  16384 heads,
// bf16, tiled / few rows: 24 rows, 16 keys 729 / 725 us; 28 rows, 16 keys 733 / 782, 48 keys 814 / 803; 32 rows, 16 keys 743 / 846,
// 64 keys 846 / 878, 80 keys 925 / 897.  (At head_dim 64, 32 rows, 32 keys 513 / 461; two query heads per KV head: few rows always.)
bool few_rows_outweigh_keys(int64_t rows, int Sq, int Skv, int D) { return D == 128 && rows == Sq && Skv < 8 * (rows - 22); }
// FP8 P.V: up to 16 rows the rules above hold (4 x 32/8 heads, 1 row, 8192 keys, head_dim 128, tiled / few rows 146 / 77 us; 2 heads of
// 8192 keys 95 / 21).  With two score tiles the V quotients do not fit the registers of head_dim 128, and the pass that finds the first
// tile's maximum costs more: 32 rows, 8 x 8 heads of 2500 / 4200 / 8192 keys 77 / 83, 115 / 114, 196 / 172; 8 x 32 of 8192 546 / 564; at
// head_dim 64, 1500 / 1800 / 4200 keys 38.4 / 39.2, 41.7 / 37.2, 77.8 / 59.5.
bool few_rows_pay_fp8(int64_t rows, int64_t pairs, int Skv, int D) { return rows <= 16 || (D == 64 ? Skv >= 1792 : Skv >= 4096 && pairs <= 64); }
struct E2EWorkspace {
  size_t q_i8, k_i8, q_scale, k_scale, km, v_scale, panels, stat, plan, lse_off, total;
  size_t k_i8_bytes;
  int64_t qs_sh, ks_sh, panel_sh;
};
// What a call's workspace holds beyond K, V and their statistics: the INT8 copy of Q with its scales (calls that may quantise Q by
// the stand-alone pass: an explicit mask, the LSE correction of K smoothing, interleaved Q scales) and the per-row LSE
// correction term (LSE of smoothed keys).  LSE calls with K blocks of 32 keys and more form that term in the attention kernel and
// leave both untouched; the size they ask for stays, so that what the built-in scratch array takes and refuses does not
// move with the kernel a call happens to use.
bool needs_q_pass(int blkq, int has_mask, int want_lse, int smooth_k) {
  return has_mask || (want_lse && smooth_k) || blk_groups(blkq) != 1;
}
E2EWorkspace e2e_layout(int B, int Hq, int Hkv, int Sq, int Skv, int D, int blkq, int blkk, int pv, int total_q, int total_k,
                        int varlen, bool q_pass, bool lse_offset) {
  E2EWorkspace w;
  size_t off = 0;
  size_t nq = varlen ? (size_t)total_q * Hq * D : (size_t)B * Hq * Sq * D;
  size_t nk = varlen ? (size_t)total_k * Hkv * D : (size_t)B * Hkv * Skv * D;
  w.q_i8 = off; off += q_pass ? align_up(nq) : 0;
  w.k_i8 = off; w.k_i8_bytes = align_up(nk); off += w.k_i8_bytes;
  if (varlen) {
    w.qs_sh = total_q / blk_rows(blkq) + B; w.ks_sh = total_k / blk_rows(blkk) + B; w.panel_sh = total_k / SAGE_PANEL_ROWS + B;
    w.q_scale = off; off += q_pass ? align_up((size_t)Hq * w.qs_sh * 4) : 0;
    w.k_scale = off; off += align_up((size_t)Hkv * w.ks_sh * 4);
  } else {
    w.qs_sh = w.ks_sh = w.panel_sh = 0;
    w.q_scale = off; off += q_pass ? align_up((size_t)B * Hq * ((Sq + blk_rows(blkq) - 1) / blk_rows(blkq)) * blk_groups(blkq) * 4) : 0;
    w.k_scale = off; off += align_up((size_t)B * Hkv * ((Skv + blk_rows(blkk) - 1) / blk_rows(blkk)) * (blk_groups(blkk) ? blk_groups(blkk) : 1) * 4);
  }
  w.km = off; off += align_up((size_t)B * Hkv * D * 2);
  w.v_scale = off; off += align_up((size_t)B * Hkv * D * 4);
  size_t pbytes = varlen ? (size_t)Hkv * w.panel_sh * SAGE_PANEL_ROWS * D * (pv ? 1 : 2) : sage_v_panel_bytes(B, Hkv, Skv, D, pv);
  w.panels = off; off += align_up(pbytes);
  size_t stat = sage_k_mean_workspace_bytes(B, Hkv, Skv, D);
  size_t stat2 = sage_prep_v_workspace_bytes(B, Hkv, Skv, D, pv);
  w.stat = off; off += align_up(stat > stat2 ? stat : stat2);
  w.plan = off; off += varlen ? align_up(sage_varlen_plan_ints(B, total_q) * 4) : 0;
  w.lse_off = off; off += lse_offset ? align_up((varlen ? (size_t)Hq * total_q : (size_t)B * Hq * Sq) * 4) : 0;
  w.total = off;
  return w;
}
}  // namespace

size_t sage_sageattn_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Skv, int D, int blkq, int blkk, int pv_mode,
                                     int total_q, int total_k, int varlen) {
  if (blkq <= 0 || blkk <= 0) return 0;
  return e2e_layout(B, Hq, Hkv, Sq, Skv, D, blkq, blkk, pv_mode, total_q, total_k, varlen, true, true).total;
}

size_t sage_sageattn_workspace_bytes_for(int B, int Hq, int Hkv, int Sq, int Skv, int D, int blkq, int blkk, int pv_mode,
                                         int total_q, int total_k, int varlen, int smooth_k, int want_lse, int has_mask) {
  if (blkq <= 0 || blkk <= 0) return 0;
  return e2e_layout(B, Hq, Hkv, Sq, Skv, D, blkq, blkk, pv_mode, total_q, total_k, varlen,
                    needs_q_pass(blkq, has_mask, want_lse, smooth_k), want_lse && smooth_k).total;
}

// A boolean mask is packed into bits when the workspace has room for them behind what the call needs anyway, the grid
// and the kernel's tile list can hold its tiles, and the pass pays: the packing is one more launch, 3 to 6 us, and saves up to
// half the time of every key tile that a q-tile visits and all of those it does not see.  Three key tiles are enough (one head of
// 500 rows and 500 keys, head_dim 64, FP16 P.V, about four documents: 35.4 us packed, 36.9 read in place; 4 heads of 800: 35.6 / 63.0;
// two tiles, 2 x 16 heads of 500 rows, 200 keys: 30.3 / 27.2), or tiles for two rounds of the chip (4 x 32 heads of 1000 rows and
// 128 keys, 512 tile visits: 32.9 / 34.8; of 2000 rows and 77 keys, 1024: 55 / 71).  In place, keys that are not contiguous are no
// slower than others, packed they are: five key tiles there, or twice the visits (128 rows, 500 keys, four tiles, transposed, FP8 P.V:
// 40.6 / 36.2; 4 heads of 800: 45.9 / 48.1).
static int64_t mask_tile_visits(const MaskPlanes& p, int B, int Hq, int Sq) { return (int64_t)B * Hq * ((Sq + kMaskRows - 1) / kMaskRows) * p.ntk; }
static bool mask_can_be_packed(const MaskPlanes& p, int B, int Hq, int Sq, int Skv, int mask_kind) {
  return mask_kind == SAGE_MASK_BOOL && Sq > 0 && Skv > 0 && p.ntk <= kMaskMaxTiles && p.nqt <= 65535 && p.planes <= 65535 &&
         (p.ntk >= 3 || mask_tile_visits(p, B, Hq, Sq) >= 512);
}

size_t sage_sageattn_mask_bytes(int B, int Hq, int Sq, int Skv, int mask_kind, int64_t m_sb, int64_t m_sh, int64_t m_sm) {
  if (B <= 0 || Hq <= 0) return 0;
  const MaskPlanes p = mask_planes(B, Hq, Sq, Skv, m_sb, m_sh, m_sm);
  return mask_can_be_packed(p, B, Hq, Sq, Skv, mask_kind) ? (size_t)p.total_bytes : 0;
}

// Few query rows per KV head over a long history: sage_attn_few.hip.  Calls that the general
// path refuses (its pre-passes have the batch and the heads on grid axes of 65535), slices of 2 GiB and more (32-bit row offsets),
// rows that overlap and grids of 2^31 threads and more are left to that path.
struct FewCall {
  int varlen, is_causal, pv_mode, B, Hkv, Sq, Skv, D, blkq, blkk;
  int64_t rows, q_sn, k_sn, v_sn;   // rows: of all query heads of a KV head
  const void *q, *k, *v, *out, *mask;
  bool short_keys, want_lse;
  size_t k_i8_bytes;   // of the workspace: where the INT8 copy of K would be, the V statistics of FP8 P.V go
};
static bool few_rows_path(const FewCall& c) {
  const int64_t limit = 0x7fffffff, pairs = (int64_t)c.B * c.Hkv;
  if (c.varlen || c.short_keys || c.is_causal || c.mask || !c.q || !c.k || !c.v || !c.out) return false;
  if (blk_groups(c.blkq) != 1 || blk_groups(c.blkk) != 1 || c.rows > kFewRows) return false;
  if (c.B > 65535 || c.Hkv > 65535 || (pairs + kFewWorkgroups) * 256 > limit) return false;
  if (c.k_sn < c.D || c.v_sn < c.D || (int64_t)c.Sq * c.q_sn * 2 >= limit) return false;
  if (((int64_t)c.Skv + 128) * c.k_sn * 2 >= limit || ((int64_t)c.Skv + 128) * c.v_sn * 2 >= limit) return false;
  if (few_tiles_per_split(c.B, c.Hkv, (int)c.rows, c.Skv, c.D, (int64_t)sage_v_panel_bytes(c.B, c.Hkv, c.Skv, c.D, c.pv_mode)) <= 0) return false;
  if (few_rows_outweigh_keys(c.rows, c.Sq, c.Skv, c.D)) return false;
  if (c.pv_mode == SAGE_PV_FP16) return true;
  // (four bytes per channel and 512 rows against one per channel and row: one to three keys do not leave the room)
  if (sage_prep_v_workspace_bytes(c.B, c.Hkv, c.Skv, c.D, c.pv_mode) > c.k_i8_bytes) return false;
  return !c.want_lse && few_rows_pay_fp8(c.rows, pairs, c.Skv, c.D);
}

int sage_sageattn(const void* q, const void* k, const void* v, void* out, float* lse, void* workspace, size_t workspace_bytes,
                  int B, int Hq, int Hkv, int Sq, int Skv, int D, int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb,
                  int64_t k_sh, int64_t k_sn, int64_t v_sb, int64_t v_sh, int64_t v_sn, int64_t o_sb, int64_t o_sh,
                  int64_t o_sn, int dtype, int blkq, int blkk, double sm_scale, int is_causal, int smooth_k, int pv_mode,
                  const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int total_q, int total_k, sage_stream_t stream) {
  return sage_sageattn_masked(q, k, v, out, lse, workspace, workspace_bytes, B, Hq, Hkv, Sq, Skv, D, q_sb, q_sh, q_sn, k_sb,
                              k_sh, k_sn, v_sb, v_sh, v_sn, o_sb, o_sh, o_sn, dtype, blkq, blkk, sm_scale, is_causal, smooth_k,
                              pv_mode, cu_seqlens_q, cu_seqlens_k, total_q, total_k, nullptr, 0, 0, 0, 0, 0, stream);
}

int sage_sageattn_masked(const void* q, const void* k, const void* v, void* out, float* lse, void* workspace,
                         size_t workspace_bytes, int B, int Hq, int Hkv, int Sq, int Skv, int D, int64_t q_sb, int64_t q_sh,
                         int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                         int64_t o_sb, int64_t o_sh, int64_t o_sn, int dtype, int blkq, int blkk, double sm_scale,
                         int is_causal, int smooth_k, int pv_mode, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                         int total_q, int total_k, const void* attn_mask, int mask_kind, int64_t m_sb, int64_t m_sh,
                         int64_t m_sm, int64_t m_sn, sage_stream_t stream) {
  g_tile_rows = 0;
  if (int rc = check_common(B, Hq, Sq, D, dtype)) return rc;
  if (Hkv <= 0 || Hq % Hkv) return fail(SAGE_EINVAL, "query heads (%d) must be divisible by KV heads (%d)", Hq, Hkv);
  if (!valid_blk_attn(blk_rows(blkq)) || !valid_blkk_attn(blk_rows(blkk)))
    return fail(SAGE_ENOTIMPL, "Q and K scale blocks must be 16, 32, 64 or 128 rows (got %d/%d)", blk_rows(blkq), blk_rows(blkk));
  if ((blk_groups(blkq) != 1 && blk_groups(blkq) != 8) || (blk_groups(blkk) != 1 && blk_groups(blkk) != 4))
    return fail(SAGE_ENOTIMPL, "Q scale blocks take SAGE_BLK_INTERLEAVE8, K scale blocks SAGE_BLK_INTERLEAVE4");
  if (blk_groups(blkk) == 4 && blk_rows(blkk) == 16)
    return fail(SAGE_ENOTIMPL, "interleaved K scales need blocks of 32, 64 or 128 keys");
  if (pv_mode != SAGE_PV_FP16 && pv_mode != SAGE_PV_FP8) return fail(SAGE_EINVAL, "pv_mode %d unknown", pv_mode);
  const int varlen = cu_seqlens_q != nullptr;
  if (varlen && (blk_groups(blkq) > 1 || blk_groups(blkk) > 1)) return fail(SAGE_ENOTIMPL, "interleaved scales are not supported for packed batches");
  if (varlen && !cu_seqlens_k) return fail(SAGE_EINVAL, "packed mode needs cu_seqlens_k");
  if (B == 0 || Hq == 0 || Sq == 0) return SAGE_OK;
  if (!workspace) return fail(SAGE_EWORKSPACE, "null workspace");
  // (the workspace is laid out for what THIS call uses; sage_sageattn_workspace_bytes is the upper bound over all calls
  // of the shape, sage_sageattn_workspace_bytes_for the size for one kind of call)
  const bool q_pass = needs_q_pass(blkq, attn_mask != nullptr, lse != nullptr, smooth_k && !(!varlen && Skv == 0));
  E2EWorkspace w = e2e_layout(B, Hq, Hkv, Sq, Skv, D, blkq, blkk, pv_mode, total_q, total_k, varlen, q_pass,
                              lse != nullptr && smooth_k && !(!varlen && Skv == 0));
  if (workspace_bytes < w.total) return fail(SAGE_EWORKSPACE, "workspace too small: %zu < %zu", workspace_bytes, w.total);
  if (reinterpret_cast<uintptr_t>(workspace) % 256) return fail(SAGE_EINVAL, "workspace must be 256-byte aligned");
  // (before anything is launched; a packed batch of no rows at all has no tensors)
  if (((!varlen || total_q > 0) && (!q || !out)) || (!varlen && Skv > 0 && (!k || !v))) return fail(SAGE_EINVAL, "null tensor pointer");
  uint8_t* ws = (uint8_t*)workspace;
  int8_t* q_i8 = (int8_t*)(ws + w.q_i8);
  int8_t* k_i8 = (int8_t*)(ws + w.k_i8);
  float* q_scale = (float*)(ws + w.q_scale);
  float* k_scale = (float*)(ws + w.k_scale);
  void* km = ws + w.km;
  float* v_scale = (float*)(ws + w.v_scale);
  void* panels = ws + w.panels;
  void* stat = ws + w.stat;
  int32_t* plan = varlen ? (int32_t*)(ws + w.plan) : nullptr;
  const size_t stat_bytes = w.plan - w.stat;
  // The int8 copies of q and k are the library's own tensors: they get dense strides of their own ([B,H,L,D] with
  // whole rows contiguous, or packed [T,H,D]), whatever strides the caller's q and k have (views of a fused QKV
  // buffer, sliced heads, ...), so that they always fit the workspace regions sized for B*H*L*D bytes.
  const int64_t qi_sb = varlen ? 0 : (int64_t)Hq * Sq * D, qi_sh = varlen ? D : (int64_t)Sq * D, qi_sn = varlen ? (int64_t)Hq * D : D;
  const int64_t ki_sb = varlen ? 0 : (int64_t)Hkv * Skv * D, ki_sh = varlen ? D : (int64_t)Skv * D, ki_sn = varlen ? (int64_t)Hkv * D : D;
  const int32_t *cu_qblk = nullptr, *cu_kblk = nullptr, *cu_panel = nullptr;
  if (varlen) {
    if (B > 32767) return fail(SAGE_EINVAL, "number of sequences %d out of range (1..32767)", B);
    SagePlanLayout L = plan_layout(B, total_q);
    cu_qblk = plan + L.cu_qblk; cu_kblk = plan + L.cu_kblk; cu_panel = plan + L.cu_panel;
  }
  int rc = SAGE_OK;
  // No keys at all (fixed-length mode): nothing to smooth, quantise or lay out; the attention kernel writes zeros
  // and LSE = -inf without reading K, V or their scales.
  const bool no_keys = !varlen && Skv == 0;
  if (no_keys) smooth_k = 0;
  // Short sequences: all K and V pre-passes in one launch (every workgroup computes the statistic its tile needs over
  // the whole sequence itself); otherwise two launches, the statistics in two stages.
  const int64_t k_elements = (int64_t)B * Hkv * Skv * D;
  const int k_rows = quant_rows(D, blk_rows(blkk));
  const int k_groups = (Skv + k_rows - 1) / k_rows, v_groups = (Skv + kPanelRows - 1) / kPanelRows;
  const int64_t prepass_reads = k_elements * ((smooth_k ? k_groups : 1) + (pv_mode == SAGE_PV_FP8 ? v_groups : 1));
  const bool small_prepass = !varlen && !no_keys && Skv <= kSmallPrepassRows && prepass_reads <= small_prepass_reads(smooth_k, pv_mode == SAGE_PV_FP8) &&
                             (int64_t)B * Hkv <= kSmallPrepassHeads;
  const bool short_keys = no_keys || tiled_beats_few_rows(pv_mode, D, Hq / Hkv * (int64_t)Sq, Sq, (int64_t)B * Hq, Skv, k_elements * (k_groups + v_groups));
  const float q_mult = (float)((sm_scale > 0 ? sm_scale : 1.0 / sqrt((double)D)) * 1.44269504);
  const FewCall few = {varlen, is_causal, pv_mode, B, Hkv, Sq, Skv, D, blkq, blkk, Hq / Hkv * (int64_t)Sq, q_sn, k_sn, v_sn,
                       q, k, v, out, attn_mask, short_keys, lse != nullptr, w.k_i8_bytes};
  if (few_rows_path(few)) {
    if (int rc2 = check_stride16("q", q_sb, q_sh, q_sn, 2, q)) return rc2;
    if (int rc2 = check_stride16("k", k_sb, k_sh, k_sn, 2, k)) return rc2;
    if (int rc2 = check_stride16("v", v_sb, v_sh, v_sn, 2, v)) return rc2;
    if (int rc2 = check_stride16("out", o_sb, o_sh, o_sn, 2, out)) return rc2;
    // the statistics of K (smoothing) and V (FP8 P.V): per chunk; the kernel combines the chunks, but for very many of K.  V's lie where
    // the INT8 copy of K would (few_rows_path has made sure that they fit), the partial results where the panels would.
    FusedPrepass stats;
    memset(&stats, 0, sizeof(stats));
    ColStatArgs& ks = stats.k_stat;
    ks.x = (const u16*)k; ks.B = B; ks.H = Hkv; ks.L = Skv; ks.D = D; ks.x_sb = k_sb; ks.x_sh = k_sh; ks.x_sn = k_sn;
    ks.nchunk = colstat_chunks(Skv);
    // (FP8 P.V of head_dim 128, float16: its kernel is as long whether it finds the tensors or not.  1 row, through / past, us: 32 heads of 523 keys
    // 29.7 / 27.8, 24 of 900 28.5 / 27.2, 16 of 1600 28.9 / 27.6, but 64 of 1245 42.6 / 44.0, 128 of 900 46.1 / 47.5; bfloat16 32 of 523 27.4 / 28.5, 16 of 1600 27.8 / 28.8)
    const bool kept = pv_mode != SAGE_PV_FP8 || D != 128 || dtype != SAGE_DT_F16 || k_elements > (int64_t)5 << 20;
    ks.cached = kept && statistics_stay(k_elements * ((smooth_k != 0) + (pv_mode == SAGE_PV_FP8)));
    stats.v_stat = ks;
    stats.v_stat.x = (const u16*)v; stats.v_stat.x_sb = v_sb; stats.v_stat.x_sh = v_sh; stats.v_stat.x_sn = v_sn;
    if (smooth_k) ks.partial = stat;
    if (pv_mode == SAGE_PV_FP8) stats.v_stat.partial = k_i8;
    hipError_t e = launch_fused_prepass(stats, dtype, D, pv_mode == SAGE_PV_FP8, (hipStream_t)stream);
    const bool mean_first = ks.partial && pv_mode == SAGE_PV_FP16 && ks.nchunk > kFewChunks;
    if (e == hipSuccess && mean_first) e = launch_k_mean_finalize(ks, dtype, km, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(statistics)");
    FewArgs f;
    memset(&f, 0, sizeof(f));
    f.q = (const u16*)q; f.k = (const u16*)k; f.v = (const u16*)v;
    f.km_partial = mean_first ? (const double*)km : (const double*)ks.partial; f.nchunk = mean_first ? 0 : ks.nchunk;
    f.vs_partial = (const float*)stats.v_stat.partial; f.vscale = v_scale;
    f.out = (u16*)out; f.lse = lse; f.part = (float*)panels;   // (no panels here: their region holds the partial results)
    f.part_bytes = (int64_t)sage_v_panel_bytes(B, Hkv, Skv, D, pv_mode);
    f.B = B; f.Hq = Hq; f.Hkv = Hkv; f.Sq = Sq; f.Skv = Skv;
    f.q_sb = q_sb; f.q_sh = q_sh; f.q_sn = q_sn; f.k_sb = k_sb; f.k_sh = k_sh; f.k_sn = k_sn;
    f.v_sb = v_sb; f.v_sh = v_sh; f.v_sn = v_sn; f.o_sb = o_sb; f.o_sh = o_sh; f.o_sn = o_sn;
    f.blkq_shift = ilog2(blkq); f.blkk_shift = ilog2(blkk); f.q_mult = q_mult;
    e = launch_attn_few(f, dtype, D, pv_mode == SAGE_PV_FP8, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(few rows)");
    return SAGE_OK;
  }
  if (small_prepass) {
    if (int rc2 = check_stride16("k", k_sb, k_sh, k_sn, 2, k)) return rc2;
    if (int rc2 = check_stride16("v", v_sb, v_sh, v_sn, 2, v)) return rc2;
    const int kb = blk_rows(blkk);
    QuantArgs qa;
    memset(&qa, 0, sizeof(qa));
    qa.x = (const u16*)k; qa.out = k_i8; qa.scale = k_scale; qa.km = nullptr;
    qa.B = B; qa.H = Hkv; qa.L = Skv; qa.D = D;
    qa.x_sb = k_sb; qa.x_sh = k_sh; qa.x_sn = k_sn; qa.o_sb = ki_sb; qa.o_sh = ki_sh; qa.o_sn = ki_sn;
    qa.cached = true;   // (other workgroups read the rows for their statistics)
    qa.blk = kb; qa.blk_shift = ilog2(kb); qa.groups = blk_groups(blkk); qa.mult = 1.0f; qa.dv_group = 1;
    PrepVArgs va;
    memset(&va, 0, sizeof(va));
    va.v = (const u16*)v; va.panels = (uint8_t*)panels; va.vscale = v_scale; va.B = B; va.H = Hkv; va.L = Skv; va.D = D;
    va.v_sb = v_sb; va.v_sh = v_sh; va.v_sn = v_sn; va.cached = true;
    hipError_t e = launch_prepass_small(qa, va, dtype, pv_mode == SAGE_PV_FP8, smooth_k != 0, km, v_scale, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(pre-pass)");
  }
  // Q is quantised by the attention kernel itself (each q-tile exactly where it is consumed) unless a feature needs the
  // standalone pass: an explicit mask or interleaved scales.
  // (LSE of smoothed keys with K blocks of 16 keys or interleaved K scales: stand-alone pass)
  const bool want_dot = lse && smooth_k;
  const bool fuse_q = !attn_mask && blk_groups(blkq) == 1 && !(want_dot && (blk_rows(blkk) == 16 || blk_groups(blkk) != 1));
  // With K smoothing every logit of a query row loses q . k_mean; the softmax does not notice but the
  // log-sum-exp does, so when LSE is requested whoever quantises Q also forms that dot product (in the
  // base-2 units of the scaled Q) and the attention kernel adds it back.  In the attention kernel's prologue it costs one
  // multiply-add per element; the pass over Q that it saves took 14 of the 243 us of a call on 32 heads of 4096 rows.
  // (The workspace keeps room for that pass: its size is part of what callers have computed.)
  RowDot dot;
  float* lse_off = nullptr;
  if (want_dot && !fuse_q) {
    lse_off = (float*)(ws + w.lse_off);
    dot.vec = km; dot.out = lse_off; dot.sb = (int64_t)Hkv * D; dot.sh = D; dot.group = Hq / Hkv; dot.total = total_q;
  }
  QRawArg qr;
  if (fuse_q) { qr.ptr = q; qr.dtype = dtype; qr.mult = q_mult; qr.dot_km = want_dot ? km : nullptr; }
  MaskArg m;
  MaskPackArgs pack;
  memset(&pack, 0, sizeof(pack));
  size_t used = w.total;   // of the workspace
  if (attn_mask) {
    // sageattn's additive mask is in natural-log units on top of sm_scale * q.k (test_sage_attention_mate.py:171-176)
    m.ptr = attn_mask; m.kind = mask_kind; m.sb = m_sb; m.sh = m_sh; m.sm = m_sm; m.sn = m_sn; m.mult = 1.44269504f;
    const MaskPlanes p = mask_planes(B, Hq, Sq, Skv, m_sb, m_sh, m_sm);
    const bool pays = m_sn == 1 || p.ntk >= 5 || mask_tile_visits(p, B, Hq, Sq) >= 1024;
    if (!varlen && !is_causal && pays && mask_can_be_packed(p, B, Hq, Sq, Skv, mask_kind) && workspace_bytes - w.total >= (size_t)p.total_bytes) {
      uint8_t* bits = ws + w.total;
      used += align_up((size_t)p.total_bytes);
      m.planes = p; m.bits = bits; m.seen = bits + p.bits_bytes;
      pack.mask = (const uint8_t*)attn_mask; pack.m_sb = m_sb; pack.m_sh = m_sh; pack.m_sm = m_sm; pack.m_sn = m_sn;
      pack.p = p; pack.Sq = Sq; pack.Skv = Skv; pack.bits = bits; pack.seen = bits + p.bits_bytes;
    }
  }
  hipStream_t st = (hipStream_t)stream;
  QuantArgs kq, qq;
  memset(&kq, 0, sizeof(kq));
  memset(&qq, 0, sizeof(qq));
  if (!no_keys) {
    if (int rc2 = quant_args(kq, k, k_i8, k_scale, smooth_k ? km : nullptr, B, Hkv, Skv, D, k_sb, k_sh, k_sn, ki_sb, ki_sh, ki_sn,
                             (int64_t)Hkv * D, D, blkk, 1.0f, dtype, cu_seqlens_k, cu_kblk, w.ks_sh, RowDot())) return rc2;
  }
  if (!fuse_q) {
    if (int rc2 = quant_args(qq, q, q_i8, q_scale, nullptr, B, Hq, Sq, D, q_sb, q_sh, q_sn, qi_sb, qi_sh, qi_sn, 0, 0, blkq, q_mult, dtype,
                             cu_seqlens_q, cu_qblk, w.qs_sh, dot)) return rc2;
  }
  if (!no_keys && Skv > 0) {
    if (!k || !v) return fail(SAGE_EINVAL, "null tensor pointer");
    if (int rc2 = check_stride16("k", k_sb, k_sh, k_sn, 2, k)) return rc2;
    if (int rc2 = check_stride16("v", v_sb, v_sh, v_sn, 2, v)) return rc2;
  }
  const bool fp8 = pv_mode == SAGE_PV_FP8, keys = !no_keys && Skv > 0;
  ColStatArgs ks, vs;
  memset(&ks, 0, sizeof(ks));
  ks.x = (const u16*)k; ks.partial = stat; ks.B = B; ks.H = Hkv; ks.L = Skv; ks.D = D;
  ks.x_sb = k_sb; ks.x_sh = k_sh; ks.x_sn = k_sn; ks.nchunk = colstat_chunks(Skv); ks.cu_seqlens = cu_seqlens_k;
  const int64_t kv_elements = varlen ? (int64_t)total_k * Hkv * D : k_elements;   // of either
  ks.cached = statistics_stay(kv_elements * ((smooth_k != 0) + fp8));
  vs = ks;
  vs.x = (const u16*)v; vs.x_sb = v_sb; vs.x_sh = v_sh; vs.x_sn = v_sn;
  PrepVArgs pvn;
  memset(&pvn, 0, sizeof(pvn));
  pvn.v = (const u16*)v; pvn.panels = (uint8_t*)panels; pvn.vscale = v_scale; pvn.B = B; pvn.H = Hkv; pvn.L = Skv; pvn.D = D;
  pvn.v_sb = v_sb; pvn.v_sh = v_sh; pvn.v_sn = v_sn; pvn.cu_seqlens = cu_seqlens_k; pvn.cu_panels = cu_panel; pvn.panel_sh = w.panel_sh;
  kq.cached = pvn.cached = !varlen && inputs_stay(2 * kv_elements);
  PlanArgs pl;
  memset(&pl, 0, sizeof(pl));
  const int bm = tile_rows({B, Hq, Sq, Skv, D, pv_mode, is_causal, blk_rows(blkk), blk_groups(blkk), lse != nullptr, mask_class(m, Skv), varlen != 0, total_q, total_k});
  if (varlen) pl = {cu_seqlens_q, cu_seqlens_k, B, total_q, blkq, blkk, bm, 64, is_causal, plan};
  // The pre-passes in two launches: what depends on nothing but the call's tensors, then what needs the statistics or the plan.  The two
  // statistics then exist at the same time; where the workspace has no room for both (it is sized for one after the other) the
  // passes follow each other.
  FusedPrepass first, second;
  memset(&first, 0, sizeof(first));
  memset(&second, 0, sizeof(second));
  const size_t v_stat_bytes = fp8 && smooth_k ? sage_prep_v_workspace_bytes(B, Hkv, Skv, D, pv_mode) : 0;
  const bool k_long = smooth_k && ks.nchunk > kFusedChunks, v_long = fp8 && ks.nchunk > kFusedChunks;
  const bool fused = keys && !small_prepass && (int64_t)B <= 65535 && Hq <= 65535 && workspace_bytes - w.total >= v_stat_bytes + (used - w.total);
  if (fused) {
    first.plan = pl;
    if (smooth_k) first.k_stat = ks;
    if (fp8) { first.v_stat = vs; first.v_stat.partial = v_stat_bytes ? (void*)(ws + used) : stat; }
    first.mask = pack;
    (varlen || smooth_k ? second : first).k_quant = kq;
    (varlen || fp8 ? second : first).v_panels = pvn;
    if (smooth_k && !k_long) { second.k_quant.km_partial = (const double*)stat; second.k_quant.km_nchunk = ks.nchunk; second.k_quant.km_out = (u16*)km; }
    if (fp8 && !v_long) { second.v_panels.vs_partial = (const float*)first.v_stat.partial; second.v_panels.vs_nchunk = vs.nchunk; second.v_panels.vscale_out = v_scale; }
    if (!fuse_q && !qq.dot_out) {   // (with the row products it waits for the K mean in memory: a launch of its own)
      FusedPrepass& f = varlen ? second : first;
      if (!f.k_quant.out || fused_quant_together(D, f.k_quant.blk, qq.blk)) { f.q_quant = qq; qq.out = nullptr; }
    }
  }
  hipError_t e = hipSuccess;
  if (fused) {
    e = launch_fused_prepass(first, dtype, D, fp8, st);
    if (e == hipSuccess && k_long) e = launch_k_mean_finalize(ks, dtype, km, st);
    if (e == hipSuccess && v_long) e = launch_v_scale_finalize(first.v_stat, v_scale, st);
    if (e == hipSuccess) e = launch_fused_prepass(second, dtype, D, fp8, st);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(pre-pass)");
  } else {
    if (varlen) {
      e = launch_varlen_plan(cu_seqlens_q, cu_seqlens_k, B, total_q, blkq, blkk, bm, 64, is_causal, plan, st);
      if (e != hipSuccess) return hip_fail(e, "sage_sageattn(plan)");
    }
    if (!small_prepass && smooth_k) {
      rc = sage_k_mean(k, km, stat, stat_bytes, B, Hkv, Skv, D, k_sb, k_sh, k_sn, dtype, cu_seqlens_k, stream);
      if (rc) return rc;
    }
    if (!small_prepass && keys) e = launch_quant_int8(kq, dtype, Skv, st);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(K)");
    if (!small_prepass && keys) {
      rc = sage_prep_v(v, panels, v_scale, stat, stat_bytes, B, Hkv, Skv, D, v_sb, v_sh, v_sn, dtype, pv_mode, cu_seqlens_k,
                       cu_panel, w.panel_sh, stream);
      if (rc) return rc;
    }
    if (pack.bits) e = launch_mask_pack(pack, st);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(mask)");
  }
  if (qq.out) {
    e = launch_quant_int8(qq, dtype, Sq, st);
    if (e != hipSuccess) return hip_fail(e, "sage_sageattn(Q)");
  }
  // the attention kernel reads either the caller's floating-point q (its strides) or the int8 copy (dense strides)
  return attn_impl(q_i8, k_i8, panels, q_scale, k_scale, pv_mode == SAGE_PV_FP8 ? v_scale : nullptr, out, lse, B, Hq, Hkv, Sq,
                   Skv, D, fuse_q ? q_sb : qi_sb, fuse_q ? q_sh : qi_sh, fuse_q ? q_sn : qi_sn, ki_sb, ki_sh, ki_sn, o_sb, o_sh,
                   o_sn, blkq, blkk, is_causal, pv_mode, dtype, cu_seqlens_q, cu_seqlens_k, plan, total_q, w.qs_sh, w.ks_sh,
                   w.panel_sh, m, lse_off, qr, bm, stream);
}

}  // extern "C"
