// Attention of a few query rows over a long history (token generation): no mask, not causal, at most kFewRows rows per KV head
// counting all query heads that share it.
//
// Bound by the bytes of K and V.  The tiled kernel gives a q-tile of 256 rows to every query head, so one row per head leaves
// 1/256 of its matrix work useful, puts B * Hq workgroups on 256 compute units and walks the whole history in each; in
// front of it K is written as an INT8 copy and V as panels, and both are read back by every query head.  Here
//   * the rows of the query heads of a KV head are the columns of one 16x16 tile (two above 16 rows), so K and V are read once
//     per KV head, from the caller's tensors: K is smoothed and quantised in registers with the quantiser's own arithmetic,
//     V is converted in registers, nothing is written back;
//   * the keys are cut into `nsplit` ranges of whole 128-key tiles, one workgroup each, so that a few (batch, KV head) pairs
//     fill the chip; a second small kernel merges the ranges' (O, m, l);
//   * a wavefront owns 32 keys of a tile, so nothing but the maximum of scale blocks of 64 and 128 keys crosses wavefronts.
// The order of the channels inside the Q.K^T contraction and of the keys inside the P.V one is free as long as both operands
// agree: K fragments take the channels as whole 64-byte pieces of a row arrive, V fragments the keys as the 16x16 score tile
// holds them, so neither the scores nor V go through LDS.
//   * the statistics (K mean, V scales) arrive per chunk of 512 rows and are combined by every workgroup: a launch less (not the K mean
//     of very long histories, kFewChunks);
//   * FP8 P.V: V is rounded to the e4m3 values of the panels in registers (a division per element: the vector ALU is what bounds it)
//     and multiplied in fp16, which holds them; the probabilities are the tiled kernel's block-scaled codes, read back the same way.
// Measured, whole calls in bf16, tiled kernel -> this one: 4 x 32/8 heads, 1 row, 8192 keys, head_dim 128: 170.7 -> 46.0 us (this
// kernel 30 us = 4.5 TB/s of K and V, half of it vector arithmetic of the quantisation; K sums 10, merge 5; requesting everything that the
// prologue needs before it waits for any of it took 1.0 of 47.8, keeping the differences as floats 0.8); 8 rows: 170.8
// -> 54; 8 x 32/8 heads, 4 rows, 16384 keys: 431.9 -> 150; 16 x 32 heads, 4096 keys: 600 -> 279; 1 x 8/2 heads, 8 rows, 32768 keys:
// 435 -> 34.  FP8 P.V: 146 -> 82 for the first, 311 -> 51 for the last.
#include "sage_launch.h"

#pragma clang fp contract(off)

namespace sage {
namespace {

constexpr float kNegInfFew = -__builtin_inff();
constexpr float kMInitFew = -1.0e30f;
constexpr float kTauFew = 8.0f;   // the running maximum moves when it grew by more than this: probabilities stay below 2^8

typedef unsigned int v2u __attribute__((ext_vector_type(2)));

__device__ inline float xor16_32_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
__device__ inline float xor16_32_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

template <class Quotient>
__device__ __forceinline__ v4i pack16(const float (&x)[16], Quotient quotient) {
  uint32_t packed[4];
  pack_codes(x, packed, quotient);
  return v4i{(int)packed[0], (int)packed[1], (int)packed[2], (int)packed[3]};
}

template <int DT, int D, int MT, int PV>
__global__ void __launch_bounds__(256, 2) attn_few_kernel(FewArgs a) {
  constexpr int LK = D / 32;   // 16-byte pieces of a K row per lane: piece i holds the channels 32 i + 8 (lane / 16) ..+7
  constexpr int KS = D / 64;   // contraction steps of Q.K^T
  constexpr int CV = D / 16;   // channels of V per lane
  constexpr int LDO = D + 4;   // floats per row of the merge buffer
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int bh = (int)fastdiv(blockIdx.x, a.div_nsplit), split = blockIdx.x - bh * a.nsplit, b = bh / a.Hkv, kvh = bh - b * a.Hkv;
  const int G = a.Hq / a.Hkv, rows = G * a.Sq, L = a.Skv;
  __shared__ float row_amax[16 * MT];
  __shared__ float block_amax[2][4];
  __shared__ float wave_m[4][16 * MT], wave_l[4][16 * MT];
  __shared__ __align__(16) float merged[16 * MT * LDO];

  // K and V through bounded buffers: rows past the end read as zeros
  const __amdgpu_buffer_rsrc_t krsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(a.k + (int64_t)b * a.k_sb + (int64_t)kvh * a.k_sh), 0,
                                                                         ((L - 1) * (int)a.k_sn + D) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(a.v + (int64_t)b * a.v_sb + (int64_t)kvh * a.v_sh), 0,
                                                                         ((L - 1) * (int)a.v_sn + D) * 2, 0x00020000);
  const int ntiles = (L + 127) >> 7;
  const int t0 = split * a.tiles_per_split, t1 = min(ntiles, t0 + a.tiles_per_split);
  v4u kraw[2][LK];
  auto load_k = [&](int tile) {
    const int off = ((tile * 128 + 32 * w + m) * (int)a.k_sn + 8 * g) * 2;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < LK; i++) kraw[t][i] = __builtin_amdgcn_raw_buffer_load_b128(krsrc, off + t * 16 * (int)a.k_sn * 2 + 64 * i, 0, 0);
  };
  // FP8 P.V: the probability codes of a row are taken relative to the maximum of its first 128 keys (what the tiled kernel's running
  // maximum is unless a later tile exceeds it by 2^20), so a range that starts later visits tile 0 first, for that maximum alone.
  const bool reference_first = PV == 1 && t0 > 0 && t0 < t1;
  const int first = reference_first ? 0 : t0;
  auto next_tile = [&](int tile) { return reference_first && tile == 0 ? t0 : tile + 1; };
  // FP16 P.V: the first statistics of K are requested, then Q and the first K tile, and only then does anything wait: one memory latency
  // instead of three.  (Loads complete in order: behind the K tile, the statistics would wait for it.  FP8 P.V, whose statistics of V come
  // along, has no registers left for it at head_dim 128 and gained nothing: 8 heads of 8192 keys 82.5 us, 82.9 like this.)
  constexpr bool EARLY = PV == 0;
  constexpr int AHEAD = EARLY ? 16 : 0;   // chunks
  const int64_t stat_at = (int64_t)bh * a.nchunk * D + tid % D;
  [[maybe_unused]] double sums[EARLY ? AHEAD : 1];
  [[maybe_unused]] v4u qraw[MT][LK];
  auto q_row = [&](int mt) {
    const int r = min(16 * mt + m, rows - 1), head = r / a.Sq, s = r - head * a.Sq;
    return a.q + (int64_t)b * a.q_sb + (int64_t)(kvh * G + head) * a.q_sh + (int64_t)s * a.q_sn + 8 * g;
  };
  if constexpr (EARLY) {
    if (a.km_partial && a.nchunk > 0 && tid < D) {
#pragma unroll
      for (int c = 0; c < AHEAD; c++) sums[c] = a.km_partial[stat_at + (int64_t)min(c, a.nchunk - 1) * D];
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const u16* qp = q_row(mt);
#pragma unroll
      for (int i = 0; i < LK; i++) qraw[mt][i] = *reinterpret_cast<const v4u*>(qp + 32 * i);
    }
    if (t0 < t1) load_k(first);
  }
  // ---- K mean and V scales from the per-chunk statistics, in chunk order (kmean_finalize_kernel, vscale_finalize_kernel) ----
  __shared__ __align__(16) u16 km_lds[D];
  [[maybe_unused]] __shared__ __align__(16) float2 vs_lds[PV ? D : 1];   // scale and its reciprocal
  [[maybe_unused]] bool v_exact = true;
  {
    const int64_t at = stat_at;
    // (head_dim 128: the lower half of the workgroup folds K, the upper one V; at 64 likewise with a quarter each)
    if (PV == 0 && a.km_partial && a.nchunk == 0) {
      if (tid < D) km_lds[tid] = reinterpret_cast<const u16*>(a.km_partial)[(int64_t)bh * D + tid];
    } else if (a.km_partial && tid < D) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < AHEAD; c++) s = c < a.nchunk ? s + sums[c] : s;
      for (int c0 = AHEAD; c0 < a.nchunk; c0 += 8) {
        double t[8];
#pragma unroll
        for (int c = 0; c < 8; c++) t[c] = a.km_partial[at + (int64_t)min(c0 + c, a.nchunk - 1) * D];
#pragma unroll
        for (int c = 0; c < 8; c++) s = c0 + c < a.nchunk ? s + t[c] : s;
      }
      km_lds[tid] = from_f32<DT>((float)(s / (double)L));
    }
    if constexpr (PV == 1) {
      if (tid >= D && tid < 2 * D) {
        float mx = 0.f;
        for (int c0 = 0; c0 < a.nchunk; c0 += 8) {
#pragma unroll
          for (int c = 0; c < 8; c++) mx = fmaxf(mx, a.vs_partial[at + (int64_t)min(c0 + c, a.nchunk - 1) * D]);
        }
        const float scale = fmaxf(mx / 448.0f, kScaleFloor);
        vs_lds[tid - D] = make_float2(scale, 1.0f / scale);
        if (split == 0) a.vscale[(int64_t)bh * D + tid - D] = scale;   // (applied to the merged, normalised output: infinities and
                                                                       // sums near fp32's end come out as in the tiled kernel)
      }
    }
    lds_barrier();
    if constexpr (PV == 1) v_exact = __builtin_amdgcn_ballot_w64(!reciprocal_is_exact(vs_lds[lane].x) || !reciprocal_is_exact(vs_lds[(lane + 64) % D].x)) == 0;
  }
  if constexpr (!EARLY)
    if (t0 < t1) load_k(first);

  float kmf[LK][8];
  if (a.km_partial) {
#pragma unroll
    for (int i = 0; i < LK; i++) {
      const v4u raw = *reinterpret_cast<const v4u*>(km_lds + 8 * g + 32 * i);
#pragma unroll
      for (int e = 0; e < 8; e++) kmf[i][e] = to_f32<DT>((u16)(raw[e >> 1] >> (16 * (e & 1))));
    }
  } else {
#pragma unroll
    for (int i = 0; i < LK; i++)
#pragma unroll
      for (int e = 0; e < 8; e++) kmf[i][e] = 0.f;
  }

  // ---- Q: row r of the tile is query row r % Sq of the group's head r / Sq; a scale per BLKQ rows of a head ----
  v4i qreg[MT][KS];
  float qscale[MT], dot[MT];
  {
    float x[MT][KS][16];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      float amax = 0.f, sum = 0.f;
#pragma unroll
      for (int i = 0; i < LK; i++) {
        v4u raw;
        if constexpr (EARLY) raw = qraw[mt][i];
        else raw = *reinterpret_cast<const v4u*>(q_row(mt) + 32 * i);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float v = to_f32<DT>((u16)(raw[e >> 1] >> (16 * (e & 1)))) * a.q_mult;
          x[mt][i >> 1][8 * (i & 1) + e] = v;
          amax = fmaxf(amax, fabsf(v));
          sum = __builtin_fmaf(v, kmf[i][e], sum);
        }
      }
      amax = xor16_32_max(amax);
      dot[mt] = xor16_32_sum(sum);   // what K smoothing takes from every logit of the row
      if (w == 0 && g == 0) row_amax[16 * mt + m] = amax;
    }
    lds_barrier();
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int r = min(16 * mt + m, rows - 1), head = r / a.Sq, s = r - head * a.Sq;
      const int s0 = s >> a.blkq_shift << a.blkq_shift, s1 = min(a.Sq, s0 + (1 << a.blkq_shift));
      float amax = 0.f;
      for (int i = s0; i < s1; i++) amax = fmaxf(amax, row_amax[head * a.Sq + i]);
      const float scale = fmaxf(amax / 127.0f, kScaleFloor), rcp = 1.0f / scale;
      qscale[mt] = scale;
      if (__builtin_amdgcn_ballot_w64(!reciprocal_is_exact(scale)) == 0) {
#pragma unroll
        for (int s = 0; s < KS; s++) qreg[mt][s] = pack16(x[mt][s], [&](float v) { return div_by_uniform(v, scale, rcp); });
      } else {
        const double wide = 1.0 / (double)scale;
#pragma unroll
        for (int s = 0; s < KS; s++) qreg[mt][s] = pack16(x[mt][s], [&](float v) { return div_by_any(v, wide); });
      }
    }
  }

  v4f o[MT][CV];
  // m_used: the maximum that the probabilities are relative to; FP8 P.V: their binary exponent over m_ref instead
  float m_used[MT], lsum[MT];
  [[maybe_unused]] float m_ref[MT], tile_scale[MT];   // tile_scale: of this tile's codes over m_used
  [[maybe_unused]] __shared__ float tile_max[PV ? 2 : 1][4][PV ? 16 * MT : 1];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    m_used[mt] = PV == 1 ? kBlockMinExp : kMInitFew;
    lsum[mt] = 0.f;
#pragma unroll
    for (int i = 0; i < CV; i++) o[mt][i] = v4f{0.f, 0.f, 0.f, 0.f};
  }

  int turn = 0;   // which of two sets in LDS: a wavefront writes the next tile's while a slower one still reads this tile's
  for (int tile = first; tile < t1; tile = next_tile(tile), turn ^= 1) {
    const int n0 = tile * 128 + 32 * w;
    const bool reference_only = reference_first && tile == 0;
    // V rows 16 t + 4 g + r of the 32 keys, CV channels each: the keys whose scores this lane will hold
    uint32_t vraw[2][4][CV / 2];
    if (!reference_only) {
      const int off = ((n0 + 4 * g) * (int)a.v_sn + CV * m) * 2;
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int at = off + (16 * t + r) * (int)a.v_sn * 2;
          if constexpr (D == 128) {
            const v4u x = __builtin_amdgcn_raw_buffer_load_b128(vrsrc, at, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) vraw[t][r][i] = x[i];
          } else {
            const v2u x = __builtin_amdgcn_raw_buffer_load_b64(vrsrc, at, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; i++) vraw[t][r][i] = x[i];
          }
        }
    }
    // ---- K: subtract the mean in the input type, block maxima, quantise ----
    // (one score tile and no V quotients: the differences stay as floats, a widening less each; at head_dim 128 this takes all 256 registers
    // and, with the sixteen sums ahead, 12 bytes a lane of scratch memory outside the loop; the others have no registers for it)
    constexpr bool WIDE = MT == 1 && PV == 0;
    float xk[2][WIDE ? D / 4 : 1];
    float amax[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const bool gone = n0 + 16 * t + m >= L;   // rows past the end are zeros
      float mx = 0.f;
#pragma unroll
      for (int i = 0; i < LK; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float lo, hi;
          unpack2<DT>(kraw[t][i][e], lo, hi);
          const uint32_t x = pack2<DT>(lo - kmf[i][2 * e], hi - kmf[i][2 * e + 1]);
          unpack2<DT>(x, lo, hi);
          if constexpr (WIDE) {
            xk[t][8 * i + 2 * e] = lo;
            xk[t][8 * i + 2 * e + 1] = hi;
          } else kraw[t][i][e] = gone ? 0u : x;
          mx = fmaxf(mx, fmaxf(fabsf(lo), fabsf(hi)));
        }
      if constexpr (WIDE) {
        if (tile * 128 + 128 > L && gone) {   // (in the one tile that has any)
#pragma unroll
          for (int e = 0; e < D / 4; e++) xk[t][e] = 0.f;
        }
      }
      if (gone) mx = 0.f;
      amax[t] = wave_max(mx);
    }
    if (a.blkk_shift >= 5) amax[0] = amax[1] = fmaxf(amax[0], amax[1]);
    if (a.blkk_shift >= 6) {
      if (lane == 0) block_amax[turn][w] = amax[0];
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (loads in flight stay in flight)
      const float* p = block_amax[turn];
      const float pair = fmaxf(p[w & ~1], p[w | 1]);
      amax[0] = amax[1] = a.blkk_shift == 6 ? pair : fmaxf(pair, fmaxf(p[(w & ~1) ^ 2], p[(w | 1) ^ 2]));
    }
    float kscale[2];
    v4i kreg[2][KS];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const float scale = fmaxf(amax[t] / 127.0f, kScaleFloor), rcp = 1.0f / scale;
      kscale[t] = scale;
      const bool fast = __builtin_amdgcn_ballot_w64(!reciprocal_is_exact(scale)) == 0;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        float x[16];
#pragma unroll
        for (int e = 0; e < 16; e++) {
          if constexpr (WIDE) x[e] = xk[t][16 * s + e];
          else x[e] = to_f32<DT>((u16)(kraw[t][2 * s + (e >> 3)][(e & 7) >> 1] >> (16 * (e & 1))));
        }
        if (fast) kreg[t][s] = pack16(x, [&](float v) { return div_by_uniform(v, scale, rcp); });
        else kreg[t][s] = pack16(x, [&, wide = 1.0 / (double)scale](float v) { return div_by_any(v, wide); });
      }
    }
    if (next_tile(tile) < t1) load_k(next_tile(tile));

    // ---- scores (lane: query row m, keys 16 t + 4 g + r), probabilities ----
    v8h p[MT];
    auto scores = [&](int mt, float (&sv)[8]) __attribute__((always_inline)) -> float {   // returns the row maximum over the wavefront's keys
      float mx = kNegInfFew;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        v4i acc = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KS; s++) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kreg[t][s], qreg[mt][s], acc, 0, 0, 0);
        const float sc = qscale[mt] * kscale[t];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float v = (float)acc[r] * sc;
          sv[4 * t + r] = n0 + 16 * t + 4 * g + r < L ? v : kNegInfFew;
          mx = fmaxf(mx, sv[4 * t + r]);
        }
      }
      return xor16_32_max(mx);
    };
    auto rescale = [&](int mt, float m_new) __attribute__((always_inline)) {
      const float alpha = __builtin_amdgcn_exp2f(m_used[mt] - m_new);
      lsum[mt] *= alpha;
#pragma unroll
      for (int i = 0; i < CV; i++) o[mt][i] *= alpha;
      m_used[mt] = m_new;
    };
    if constexpr (PV == 1) {
      // The codes of the tiled kernel (block-scaled by the exponent e of the row's maximum in the tile), read back as the values they
      // stand for, which fp16 holds.  Their common factor 2^(e - m_used) multiplies the tile's fp32 product, not the values: fp16 would
      // lose those of a tile 16 binades below another one, which large values of V can still bring into the result.
      float sv[MT][8];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const float mx = scores(mt, sv[mt]);
        if (g == 0) tile_max[turn][w][16 * mt + m] = mx;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const int r = 16 * mt + m;
        const float mall = fmaxf(fmaxf(tile_max[turn][0][r], tile_max[turn][1][r]), fmaxf(tile_max[turn][2][r], tile_max[turn][3][r]));
        if (tile == 0) m_ref[mt] = mall;
        const float e = fmaxf(__builtin_ceilf(mall - m_ref[mt]), kBlockMinExp);
        if (__builtin_amdgcn_ballot_w64(e > m_used[mt]) != 0) rescale(mt, fmaxf(m_used[mt], e));
        const float c = __builtin_fmaf(-kCodeStep, e, __builtin_fmaf(kCodeStep, kBlockTop - m_ref[mt], kCodeZero));
        tile_scale[mt] = __builtin_amdgcn_exp2f(e - m_used[mt]);
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = __builtin_fmaf(sv[mt][j + i], kCodeStep, c);
          const int code = pack_probability_codes(x[0], x[1], x[2], x[3]);
          const v2f lo = __builtin_amdgcn_cvt_pk_f32_fp8(code, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(code, true);
          const float v[4] = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
          for (int i = 0; i < 4; i++) {
            sum += v[i];
            p[mt][j + i] = (_Float16)v[i];
          }
        }
        lsum[mt] = __builtin_fmaf(sum, tile_scale[mt], lsum[mt]);
      }
      if (reference_only) {   // (nothing but m_ref was wanted)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) { m_used[mt] = kBlockMinExp; lsum[mt] = 0.f; }
        continue;
      }
    } else {
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        float sv[8];
        const float mx = scores(mt, sv);
        if (__builtin_amdgcn_ballot_w64(mx > m_used[mt] + kTauFew) != 0) rescale(mt, fmaxf(m_used[mt], mx));
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const float e = __builtin_amdgcn_exp2f(sv[j] - m_used[mt]);
          lsum[mt] += e;
          p[mt][j] = (_Float16)e;
        }
      }
    }
    // ---- O^T += V^T . P^T: matrix row c of product i is channel CV c + i ----
    auto accumulate = [&](auto narrow) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < CV; i++) {
        v8h vf;
        float2 vs = {1.f, 1.f};
        if constexpr (PV == 1) vs = vs_lds[CV * m + i];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const u16 b0 = (u16)(vraw[j >> 2][j & 3][i >> 1] >> (16 * (i & 1))), b1 = (u16)(vraw[(j + 1) >> 2][(j + 1) & 3][i >> 1] >> (16 * (i & 1)));
          if constexpr (PV == 1) {
            // the e4m3 code of the panels (prep_v_tile), widened again: fp16 holds every e4m3 value, so only V is rounded to 8 bits
            const float z0 = fminf(fmaxf(narrow(to_f32<DT>(b0), vs), -448.f), 448.f), z1 = fminf(fmaxf(narrow(to_f32<DT>(b1), vs), -448.f), 448.f);
            const int code = __builtin_amdgcn_cvt_pk_fp8_f32(z0, z1, 0, false);
            const v2f w2 = __builtin_amdgcn_cvt_pk_f32_fp8(code, false);
            const v2h h2 = __builtin_convertvector(w2, v2h);
            vf[j] = h2[0];
            vf[j + 1] = h2[1];
          } else {
            const v2h h2 = __builtin_bit_cast(v2h, DT == 0 ? (uint32_t)b0 | (uint32_t)b1 << 16 : pack2<0>(bf16_to_f32(b0), bf16_to_f32(b1)));
            vf[j] = h2[0];
            vf[j + 1] = h2[1];
          }
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          if constexpr (PV == 1) {
            const v4f part = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, p[mt], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) o[mt][i][r] = __builtin_fmaf(part[r], tile_scale[mt], o[mt][i][r]);
          } else o[mt][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, p[mt], o[mt][i], 0, 0, 0);
        }
        if constexpr (PV == 1) __builtin_amdgcn_sched_barrier(0);   // (one channel's quotients at a time: several do not fit the registers)
      }
    };
    if (PV == 0 || v_exact) accumulate([](float x, float2 vs) { return div_by_uniform(x, vs.x, vs.y); });
    else accumulate([](float x, float2 vs) { return div_by_any(x, 1.0 / (double)vs.x); });
  }

  // ---- the four wavefronts' parts into one, in their order ----
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    lsum[mt] = xor16_32_sum(lsum[mt]);
    if (g == 0) {
      wave_m[w][16 * mt + m] = m_used[mt];
      wave_l[w][16 * mt + m] = lsum[mt];
    }
  }
  __syncthreads();
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int r = 16 * mt + m;
    const float top = fmaxf(fmaxf(wave_m[0][r], wave_m[1][r]), fmaxf(wave_m[2][r], wave_m[3][r]));
    const float f = __builtin_amdgcn_exp2f(m_used[mt] - top);
#pragma unroll
    for (int i = 0; i < CV; i++) o[mt][i] *= f;
  }
  for (int part_of = 0; part_of < 4; part_of++) {
    if (w == part_of) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          float* dst = merged + (16 * mt + m) * LDO + CV * (4 * g + r);
#pragma unroll
          for (int i = 0; i < CV; i += 4) {
            float4 v = make_float4(o[mt][i][r], o[mt][i + 1][r], o[mt][i + 2][r], o[mt][i + 3][r]);
            if (part_of) {
              const float4 u = *reinterpret_cast<const float4*>(dst + i);
              v = make_float4(u.x + v.x, u.y + v.y, u.z + v.z, u.w + v.w);
            }
            *reinterpret_cast<float4*>(dst + i) = v;
          }
        }
    }
    __syncthreads();
  }
  float* part = a.part + ((int64_t)bh * a.nsplit + split) * few_part_floats(rows, D);
  for (int i = tid; i < rows * (D / 4); i += 256) {
    const int r = i / (D / 4), c = i - r * (D / 4);
    reinterpret_cast<float4*>(part)[i] = *reinterpret_cast<const float4*>(merged + r * LDO + 4 * c);
  }
  float* meta = part + rows * D;   // m, l and the smoothing term of every row
  if (tid < rows) {
    const float top = fmaxf(fmaxf(wave_m[0][tid], wave_m[1][tid]), fmaxf(wave_m[2][tid], wave_m[3][tid]));
    float l = 0.f;
    for (int i = 0; i < 4; i++) l += wave_l[i][tid] * __builtin_amdgcn_exp2f(wave_m[i][tid] - top);
    meta[tid] = top;
    meta[rows + tid] = l;
  }
  if (w == 0 && g == 0) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
      if (16 * mt + m < rows) meta[2 * rows + 16 * mt + m] = dot[mt];
  }
}

// One workgroup per (row, batch x KV head): out = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s.
// A few kilobytes per row out of the L2: bound by the latency of its rounds of loads.  D / 4 lanes take a partial result, as many
// groups of them as there are partial results (four wavefronts at most) every group's first eight at once, ahead of the maxima.  (With
// one lane per channel walking all of them, 256 ranges took 22 us: 2 heads of 32768 keys.)
template <int DT, int D>
__global__ void __launch_bounds__(256) attn_few_merge_kernel(FewArgs a) {
  constexpr int LN = D / 4, MAXG = 256 / LN, AHEAD = 8;
  const int bh = blockIdx.x, r = blockIdx.y, b = bh / a.Hkv, kvh = bh - b * a.Hkv, tid = threadIdx.x;
  const int lane4 = tid % LN, group = tid / LN, groups = blockDim.x / LN, nwaves = blockDim.x / 64;
  const int G = a.Hq / a.Hkv, rows = G * a.Sq, hq = kvh * G + r / a.Sq, s = r % a.Sq;
  const int64_t stride = few_part_floats(rows, D);
  const float* part = a.part + (int64_t)bh * a.nsplit * stride;
  const float* meta = part + rows * D + r;
  __shared__ float factor[kFewWorkgroups];
  __shared__ float wave_top[4], wave_sum[4];
  __shared__ float4 sums[MAXG][LN];
  float4 o[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; i++) o[i] = reinterpret_cast<const float4*>(part + min(group + i * groups, a.nsplit - 1) * stride + r * D)[lane4];
  float vs[4] = {1.f, 1.f, 1.f, 1.f};
  if (a.vs_partial) {
    const float4 t = reinterpret_cast<const float4*>(a.vscale + (int64_t)bh * D)[lane4];
    vs[0] = t.x; vs[1] = t.y; vs[2] = t.z; vs[3] = t.w;
  }
  float top = kMInitFew;
  for (int i = tid; i < a.nsplit; i += blockDim.x) top = fmaxf(top, meta[i * stride]);
  top = wave_max(top);
  if ((tid & 63) == 0) wave_top[tid >> 6] = top;
  __syncthreads();
  for (int i = 0; i < nwaves; i++) top = fmaxf(top, wave_top[i]);
  float l = 0.f;
  for (int i = tid; i < a.nsplit; i += blockDim.x) {
    const float f = __builtin_amdgcn_exp2f(meta[i * stride] - top);
    factor[i] = f;
    l = __builtin_fmaf(meta[i * stride + rows], f, l);
  }
#pragma unroll
  for (int i = 1; i < 64; i <<= 1) l += __shfl_xor(l, i);
  if ((tid & 63) == 0) wave_sum[tid >> 6] = l;
  __syncthreads();
  l = 0.f;
  for (int i = 0; i < nwaves; i++) l += wave_sum[i];
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  auto add = [&](const float4& v, float f) {
    acc.x = __builtin_fmaf(v.x, f, acc.x); acc.y = __builtin_fmaf(v.y, f, acc.y); acc.z = __builtin_fmaf(v.z, f, acc.z); acc.w = __builtin_fmaf(v.w, f, acc.w);
  };
#pragma unroll
  for (int i = 0; i < AHEAD; i++)
    if (group + i * groups < a.nsplit) add(o[i], factor[group + i * groups]);
#pragma unroll 8
  for (int i = group + AHEAD * groups; i < a.nsplit; i += groups) add(reinterpret_cast<const float4*>(part + i * stride + r * D)[lane4], factor[i]);
  sums[group][lane4] = acc;
  __syncthreads();
  if (group == 0) {
    for (int i = 1; i < groups; i++) add(sums[i][lane4], 1.0f);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    const uint2 out = make_uint2(pack2<DT>(acc.x * inv * vs[0], acc.y * inv * vs[1]), pack2<DT>(acc.z * inv * vs[2], acc.w * inv * vs[3]));
    *reinterpret_cast<uint2*>(a.out + (int64_t)b * a.o_sb + (int64_t)hq * a.o_sh + (int64_t)s * a.o_sn + 4 * lane4) = out;
    if (a.lse && lane4 == 0) a.lse[((int64_t)b * a.Hq + hq) * a.Sq + s] = l > 0.f ? top + __builtin_amdgcn_logf(l) + (a.km_partial ? meta[2 * rows] : 0.f) : kNegInfFew;
  }
}

// One range per (batch, KV head): nothing to merge, D / 4 lanes normalise a row, 1024 / D rows per workgroup.  (A workgroup of the merge
// kernel per row, with three barriers and eight loads of the one partial result: whole calls of 16384 heads, head_dim 64, 32 rows and 32 keys
// 535 -> 311 us, 1 row and 64 keys 164 -> 156; head_dim 128, 16 rows and 32 keys 467 -> 365.)
// At most kFewNormaliseGroups workgroups, which then walk the rows: 4 M pairs of 32 rows would be more threads than a grid axis holds.
constexpr int kFewNormaliseGroups = 1 << 16;
template <int DT, int D>
__global__ void __launch_bounds__(256) attn_few_normalise_kernel(FewArgs a) {
  constexpr int LN = D / 4, RPW = 256 / LN;
  const int G = a.Hq / a.Hkv, rows = G * a.Sq, total = a.B * a.Hkv * rows, lane4 = threadIdx.x % LN;
  for (int row = blockIdx.x * RPW + threadIdx.x / LN; row < total; row += gridDim.x * RPW) {
    const int bh = row / rows, r = row - bh * rows, b = bh / a.Hkv, kvh = bh - b * a.Hkv, head = r / a.Sq, hq = kvh * G + head, s = r - head * a.Sq;
    const float* part = a.part + (int64_t)bh * few_part_floats(rows, D);
    const float* meta = part + rows * D + r;
    const float4 o = reinterpret_cast<const float4*>(part + r * D)[lane4];
    const float m = meta[0], top = fmaxf(kMInitFew, m), f = __builtin_amdgcn_exp2f(m - top), l = meta[rows] * f;   // (f: 1, or NaN with m)
    float4 vs = make_float4(1.f, 1.f, 1.f, 1.f);
    if (a.vs_partial) vs = reinterpret_cast<const float4*>(a.vscale + (int64_t)bh * D)[lane4];
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    const uint2 out = make_uint2(pack2<DT>(o.x * f * inv * vs.x, o.y * f * inv * vs.y), pack2<DT>(o.z * f * inv * vs.z, o.w * f * inv * vs.w));
    *reinterpret_cast<uint2*>(a.out + (int64_t)b * a.o_sb + (int64_t)hq * a.o_sh + (int64_t)s * a.o_sn + 4 * lane4) = out;
    if (a.lse && lane4 == 0) a.lse[((int64_t)b * a.Hq + hq) * a.Sq + s] = l > 0.f ? top + __builtin_amdgcn_logf(l) + (a.km_partial ? meta[2 * rows] : 0.f) : kNegInfFew;
  }
}

}  // namespace

hipError_t launch_attn_few(FewArgs a, int dtype, int D, int pv, hipStream_t st) {
  const int rows = a.Hq / a.Hkv * a.Sq, ntiles = (a.Skv + 127) / 128, pairs = a.B * a.Hkv;
  // Two workgroups of four wavefronts per compute unit, no range shorter than one tile.
  a.tiles_per_split = few_tiles_per_split(a.B, a.Hkv, rows, a.Skv, D, a.part_bytes);
  if (a.tiles_per_split < 1) return hipErrorInvalidValue;
  a.nsplit = (ntiles + a.tiles_per_split - 1) / a.tiles_per_split;
  a.div_nsplit = make_fastdiv(a.nsplit);
  // The pairs go on x, the one grid axis that is not limited to 65535.  In the main kernel the ranges of a pair stay neighbours:
  // with the pairs next to each other instead, 4 x 32/8 heads of 8192 keys took 50.9 us instead of 49.2.
  if (a.nsplit > kFewWorkgroups) return hipErrorInvalidValue;   // (the merge holds a factor per range)
  const dim3 grid(pairs * a.nsplit), block(256);
#define SAGE_FEW_P(DT, DD, PVV) (rows > 16 ? attn_few_kernel<DT, DD, 2, PVV><<<grid, block, 0, st>>>(a) : attn_few_kernel<DT, DD, 1, PVV><<<grid, block, 0, st>>>(a))
#define SAGE_FEW(DT, DD) (pv ? SAGE_FEW_P(DT, DD, 1) : SAGE_FEW_P(DT, DD, 0))
  if (dtype == 0) { if (D == 64) SAGE_FEW(0, 64); else SAGE_FEW(0, 128); }
  else { if (D == 64) SAGE_FEW(1, 64); else SAGE_FEW(1, 128); }
#undef SAGE_FEW
#undef SAGE_FEW_P
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (a.nsplit == 1) {
    const int64_t groups = ((int64_t)pairs * rows * (D / 4) + 255) / 256;
    const dim3 ngrid((uint32_t)(groups < kFewNormaliseGroups ? groups : kFewNormaliseGroups));
    if (dtype == 0) { if (D == 64) attn_few_normalise_kernel<0, 64><<<ngrid, block, 0, st>>>(a); else attn_few_normalise_kernel<0, 128><<<ngrid, block, 0, st>>>(a); }
    else { if (D == 64) attn_few_normalise_kernel<1, 64><<<ngrid, block, 0, st>>>(a); else attn_few_normalise_kernel<1, 128><<<ngrid, block, 0, st>>>(a); }
    return hipGetLastError();
  }
  int threads = 64;   // of the merge: a group of D / 4 lanes per partial result
  while (threads < 256 && threads < a.nsplit * (D / 4)) threads *= 2;
  const dim3 mgrid(pairs, rows), mblock(threads);
  if (dtype == 0) { if (D == 64) attn_few_merge_kernel<0, 64><<<mgrid, mblock, 0, st>>>(a); else attn_few_merge_kernel<0, 128><<<mgrid, mblock, 0, st>>>(a); }
  else { if (D == 64) attn_few_merge_kernel<1, 64><<<mgrid, mblock, 0, st>>>(a); else attn_few_merge_kernel<1, 128><<<mgrid, mblock, 0, st>>>(a); }
  return hipGetLastError();
}

}  // namespace sage
