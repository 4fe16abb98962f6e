// Shared declarations for the gfx950 SageAttention kernels: vector types, wave-level helpers,
// dtype conversion, the V panel byte order and the variable-length plan layout.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sage {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned short u16;

constexpr int kWave = 64;
constexpr int kPanelRows = 128;  // == SAGE_PANEL_ROWS

// ---------------------------------------------------------------------------------------------
// V panel byte order.  A panel holds 128 consecutive KV rows n (0..127) of one (batch, kv head)
// for all D channels d, arranged so that one wavefront-wide 16-byte load per lane yields an MFMA
// operand of V^T (rows = 32 channels, contraction = KV rows) with no shuffling:
//
//  FP8 (1 byte/elt, 128*D bytes): index = (((ks*(D/32) + dt)*2 + half)*64 + lane)*16 + j
//      ks = n/64, lane = 32*h + (d%32), dt = d/32,
//      n%64 = 32*half + 8*(j/4) + 4*h + (j%4)          (j = 0..15, h = 0..1, half = 0..1)
//    -> operand of v_mfma_f32_32x32x64_f8f6f4: lane (d%32, h) holds 32 bytes (half 0 then 1).
//  FP16 (2 bytes/elt, 256*D bytes): index(elements) = ((ks*(D/32) + dt)*64 + lane)*8 + j
//      ks = n/16, lane = 32*h + (d%32), n%16 = 8*(j/4) + 4*h + (j%4)      (j = 0..7)
//    -> operand of v_mfma_f32_32x32x16_f16.
//
// The row order inside a lane's bytes equals the order in which a lane of the S^T = K.Q^T
// accumulator (v_mfma_i32_32x32x32_i8: register r of lane (m, h) is KV row 8*(r/4)+4*h+(r%4))
// holds the probabilities of query row m, so P never leaves registers between the two MFMAs.
// ---------------------------------------------------------------------------------------------
__host__ __device__ inline int panel_index_fp8(int n, int d, int D) {
  int ks = n >> 6, nn = n & 63;
  int half = nn >> 5, r = nn & 31;
  int a = r >> 3, h = (r >> 2) & 1, b = r & 3;
  int lane = 32 * h + (d & 31), dt = d >> 5;
  return (((ks * (D / 32) + dt) * 2 + half) * 64 + lane) * 16 + 4 * a + b;
}
__host__ __device__ inline int panel_index_fp16(int n, int d, int D) {
  int ks = n >> 4, r = n & 15;
  int a = r >> 3, h = (r >> 2) & 1, b = r & 3;
  int lane = 32 * h + (d & 31), dt = d >> 5;
  return ((ks * (D / 32) + dt) * 64 + lane) * 8 + 4 * a + b;
}

// ---------------------------------------------------------------------------------------------
// Variable-length plan: int32 arrays packed in one device buffer, offsets in ints.
// ---------------------------------------------------------------------------------------------
struct SagePlanLayout {
  int64_t cu_qblk, cu_kblk, cu_panel, ntiles, tiles, total;
};
__host__ __device__ inline SagePlanLayout plan_layout(int nseq, int total_q) {
  SagePlanLayout L;
  L.cu_qblk = 0;
  L.cu_kblk = L.cu_qblk + nseq + 1;
  L.cu_panel = L.cu_kblk + nseq + 1;
  L.ntiles = L.cu_panel + nseq + 1;
  L.tiles = L.ntiles + 1;
  // an attention q-tile never has fewer than 128 rows, so at most total_q/128 + nseq tiles exist
  L.total = L.tiles + (int64_t)total_q / 128 + nseq + 1;
  return L;
}

// ---------------------------------------------------------------------------------------------
// Packed boolean mask: one bit per (query row, key), in the order in which the attention kernel's accumulators hold the
// scores, and one visibility bit per 32 query rows and key tile.
//   bits: [plane][q-tile of 256 rows][tile of 128 keys][row][h = 0, 1] -> 64 bits; bit 16 * nt + r is key
//         32 * nt + 8 * (r / 4) + 4 * h + r % 4 of the tile (0 past the last key and in rows past the last one)
//   seen: uint8 [plane][q-tile][tile], bit g: some row of the q-tile's 32-row group g sees some key of the tile
// A plane is one distinct [Sq, Skv] slice of the mask (broadcast batches and heads share one); a mask that is the same
// for every query row has one q-tile, whatever Sq is.
// ---------------------------------------------------------------------------------------------
constexpr int kMaskRows = 256, kMaskKeys = 128, kMaskTileBytes = kMaskRows * kMaskKeys / 8;
constexpr int kMaskMaxTiles = 2048;   // key tiles the attention kernel's tile list has room for
struct MaskPlanes {
  int planes, nqt, ntk;   // distinct slices, q-tiles and key tiles of each
  int pb, ph;             // plane of (batch b, head h) = b * pb + h * ph
  int64_t bits_bytes, total_bytes;
};
inline MaskPlanes mask_planes(int B, int Hq, int Sq, int Skv, int64_t m_sb, int64_t m_sh, int64_t m_sm) {
  MaskPlanes p;
  const int heads = m_sh ? Hq : 1;
  p.planes = (m_sb ? B : 1) * heads;
  p.pb = m_sb ? heads : 0;
  p.ph = m_sh ? 1 : 0;
  p.nqt = m_sm ? (Sq + kMaskRows - 1) / kMaskRows : 1;
  p.ntk = (Skv + kMaskKeys - 1) / kMaskKeys;
  const int64_t tiles = (int64_t)p.planes * p.nqt * p.ntk;
  p.bits_bytes = tiles * kMaskTileBytes;
  p.total_bytes = p.bits_bytes + (tiles + 255) / 256 * 256;
  return p;
}

// ---------------------------------------------------------------------------------------------
// dtype helpers (bf16 handled as raw bits: widening is a shift, narrowing is RNE).
// ---------------------------------------------------------------------------------------------
__device__ inline float bf16_to_f32(u16 v) { return __builtin_bit_cast(float, (uint32_t)v << 16); }
// narrowing: gfx950 has a hardware round-to-nearest-even conversion (v_cvt_pk_bf16_f32)
__device__ inline u16 f32_to_bf16(float f) { return __builtin_bit_cast(u16, (__bf16)f); }
__device__ inline float f16_to_f32(u16 v) { return (float)__builtin_bit_cast(_Float16, v); }
__device__ inline u16 f32_to_f16(float f) { return __builtin_bit_cast(u16, (_Float16)f); }

template <int DT>
__device__ inline float to_f32(u16 v) {
  if constexpr (DT == 1) return bf16_to_f32(v);
  else return f16_to_f32(v);
}
template <int DT>
__device__ inline u16 from_f32(float f) {
  if constexpr (DT == 1) return f32_to_bf16(f);
  else return f32_to_f16(f);
}
// Two values narrowed into one dword by one instruction (v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32, both round to nearest even).
template <int DT>
__device__ inline uint32_t pack2(float lo, float hi) {
  const v2f v = {lo, hi};
  if constexpr (DT == 1) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2bf));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2h));
}
// Both halves of a dword widened.
template <int DT>
__device__ inline void unpack2(uint32_t x, float& lo, float& hi) {
  if constexpr (DT == 1) { lo = __builtin_bit_cast(float, x << 16); hi = __builtin_bit_cast(float, x & 0xffff0000u); }
  else { lo = f16_to_f32((u16)x); hi = f16_to_f32((u16)(x >> 16)); }
}

// ---------------------------------------------------------------------------------------------
// Streaming accesses of the pre-pass kernels: every byte of an operand is touched once per pass and not again before
// hundreds of megabytes have gone by, so the accesses are marked non-temporal (no cache line is kept for them).  On
// this part a read-only pass over 0.5 GB measures 6.9-7.1 TB/s with such loads against 6.0-6.2 TB/s with plain ones.
// ---------------------------------------------------------------------------------------------
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
__device__ inline uint4 load_stream16(const void* p) {
  const v4u v = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p));
  return make_uint4(v[0], v[1], v[2], v[3]);
}
// ... unless a later pass of the same call finds them in the last-level cache (256 MB), or in an L2, which is for the caller to know:
// `load` is handed to the work as a function, so that the choice is one uniform branch around it.
template <class Work>
__device__ __forceinline__ void with_loads(bool cached, Work work) {
  if (cached) work([](const void* p) __attribute__((always_inline)) { return *reinterpret_cast<const uint4*>(p); });
  else work([](const void* p) __attribute__((always_inline)) { return load_stream16(p); });
}
__device__ inline void store_stream16(void* p, uint4 v) {
  const v4u t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, reinterpret_cast<v4u*>(p));
}
__device__ inline void store16(bool cached, void* p, uint4 v) {
  if (cached) *reinterpret_cast<uint4*>(p) = v;
  else store_stream16(p, v);
}

// Workgroup barrier that only orders LDS traffic: waits for this wavefront's outstanding LDS
// operations, then s_barrier (global-memory traffic issued ahead stays in flight).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---------------------------------------------------------------------------------------------
// Wavefront (64-lane) reductions with DPP inside rows of 16 lanes, then lane reads across rows.
// The result is uniform across the wavefront.
// ---------------------------------------------------------------------------------------------
template <int CTRL>
__device__ inline float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x),
                                                              CTRL, 0xf, 0xf, false));
}
// Maximum over the 16 lanes of a DPP row (lanes 16r .. 16r+15), in every lane of the row.
__device__ inline float row16_max(float x) {
  x = fmaxf(x, dpp_f<0xB1>(x));   // quad_perm [1,0,3,2]
  x = fmaxf(x, dpp_f<0x4E>(x));   // quad_perm [2,3,0,1]
  x = fmaxf(x, dpp_f<0x141>(x));  // row_half_mirror
  x = fmaxf(x, dpp_f<0x140>(x));  // row_mirror
  return x;
}
__device__ inline float wave_max(float x) {
  x = row16_max(x);
  float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 0));
  float b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 16));
  float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 32));
  float d = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// ---------------------------------------------------------------------------------------------
// Arithmetic shared by every place that produces INT8 operands (the standalone quantiser and the
// attention prologue that quantises its own Q tile): they must agree bit for bit.
// ---------------------------------------------------------------------------------------------
constexpr float kScaleFloor = 1.0e-12f;


// Correctly rounded x / s for a wavefront-uniform divisor whose reciprocal r = RN(1/s) is given.
// q0 = RN(x*r) is within 1 ulp of x/s; e = x - q0*s is exact in one FMA; RN(q0 + e*r) is then
// the correctly rounded quotient (Markstein's correction step), provided s's significand is not
// all ones and nothing under/overflows; the caller takes div_by_any otherwise.
__device__ inline float div_by_uniform(float x, float s, float r) {
  float q0 = x * r;
  float e = __builtin_fmaf(-q0, s, x);
  return __builtin_fmaf(e, r, q0);
}
// True where that holds for the divisor s.
__device__ inline bool reciprocal_is_exact(float s) {
  return (__builtin_bit_cast(uint32_t, s) & 0x7fffffu) != 0x7fffffu && s < 1.0e30f;
}
// The same quotient for any divisor, given r = RN(1/s) in binary64: x * r is off by less than 2^-51 of itself, and a quotient of
// two 24-bit significands that is no binary32 number keeps 2^-49 of itself away from every point where binary32 rounding changes.
// (Three instructions an element; inlined true divisions were a tenth of the attention kernels' code, nearly never run.)
__device__ inline float div_by_any(float x, double r) { return (float)((double)x * r); }

// FP8 probabilities as block-scaled linear-mantissa codes (explained at the softmax of sage_attn_kernel.h): the code of 2^t is
// 8 t + 56 + kCodeBias, t = s - m - e + kBlockTop; pack_probability_codes takes (256 code + 127.5) / 65535 of four scores.
constexpr float kCodeBias = -0.3f;       // centres the linear-mantissa code
constexpr float kBlockTop = 8.75f, kBlockMinExp = -110.0f;
constexpr float kCodeStep = 8.0f * 256.0f / 65535.0f, kCodeZero = 256.0f / 65535.0f * (56.0f + kCodeBias) + 127.5f / 65535.0f;
__device__ inline int pack_probability_codes(float a, float b, float c, float d) {
  const unsigned w01 = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pknorm_u16(a, b));
  const unsigned w23 = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pknorm_u16(c, d));
  return (int)__builtin_amdgcn_perm(w23, w01, 0x07050301u);
}

// INT8 codes of N quotients (a multiple of four): q = trunc(z + 0.5 sgn(z)), four to a dword.  |z| <= 127.5, so the low byte of the
// converted integer is the code, and three byte permutes gather four of them (masks and shifts took twice the instructions).
template <int N, class Quotient>
__device__ __forceinline__ void pack_codes(const float (&x)[N], uint32_t (&packed)[N / 4], Quotient quotient) {
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    int q[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      // For |x| so small that the residual of the correction step is subnormal the quotient is
      // below 1e-13 in magnitude (scale >= 1e-12): whatever its last bits, it rounds to 0.
      float z = quotient(x[i + e]);
      z = z + __builtin_copysignf(0.5f, z);   // +0.5 for z >= 0 (incl. -0: -0.5 + -0 = -0.5 -> 0), else -0.5
      q[e] = (int)z;   // truncation toward zero
    }
    const uint32_t lo = __builtin_amdgcn_perm((uint32_t)q[1], (uint32_t)q[0], 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm((uint32_t)q[3], (uint32_t)q[2], 0x0c0c0400u);
    packed[i / 4] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
  }
}


}  // namespace sage
