// Quantisers of the SageAttention forward path for gfx950 (MI355X):
//   * per-block INT8 quantiser for Q and K (optional K-mean subtraction in the input dtype),
//   * per-(batch, head, channel) column statistics over the sequence (K mean, V abs-max),
//   * V preparation into MFMA-ready panels (fp16, or fp8-e4m3fn with per-channel scales).
// All of them are streaming kernels bound by HBM bandwidth: 128-bit loads of 8 elements per
// lane, statistics reduced with DPP inside the wavefront and through LDS across wavefronts.
//
// Arithmetic contract of the INT8 quantiser (bit-exact target): IEEE binary32 throughout,
//   backends/_enflame/ops/sage_attention/quant_per_block.py:38-46  (+ :53-54 for k - km)
//   backends/_hygon/ops/sageattention/sageattention_triton.py:35   (1e-12 floor)
#include "sage_launch.h"

#pragma clang fp contract(off)

namespace sage {

// Geometry of the quantiser: a workgroup of 256 lanes takes quant_rows(D, blk) consecutive rows of one (batch, head), whole scale
// blocks of them, and a wavefront quant_passes(D, blk) times quant_wave_rows(D) neighbouring ones, never more than a scale block: the
// maximum of a block crosses wavefronts only where the block does, and no lane is idle at any block size.
// Bound by HBM (3 bytes per element) with the vector ALU close behind it: some 12 instructions per element, 19 when the differences
// were narrowed one by one, widened twice and packed by masks and shifts.  bf16, K mean subtracted, head_dim 128, one kernel: 4 x 32
// heads of 4096 rows, blocks of 64: 52.0 -> 40.8 us (201 MB, 4.9 TB/s); blocks of 16, 2 x 16 heads of 4096 rows, where a block a
// workgroup left half the lanes idle: 24.5 -> 13.1.
__host__ __device__ constexpr int quant_wave_rows(int D) { return 64 / (D / 16); }   // rows of a pass of a wavefront
__host__ __device__ constexpr int quant_passes(int D, int blk) { return D == 128 ? (blk == 128 ? 4 : 2) : (blk >= 64 ? 2 : 1); }
__host__ __device__ constexpr int quant_rows(int D, int blk) { return 4 * quant_passes(D, blk) * quant_wave_rows(D); }

// Quantises the rows chunk * quant_rows(D, blk) .. of (batch b, head h), which stay in registers, as floats, between the abs-max and
// the rounding.  A lane owns 16 consecutive channels of a row (two 128-bit loads, one 128-bit store); all its loads are issued
// before anything waits for one.
// (km_lds: the K mean of this (batch, head) in LDS, D values in the input dtype, instead of a.km in global memory:
// the fused pre-pass of short sequences computes it in the same workgroup.)
// UNIT: the multiplier is 1 (every K call; x * 1.0f is x, so leaving the product out changes no bit).
template <int DT, int D, int NP, bool UNIT>
__device__ __forceinline__ void quant_int8_rows(const QuantArgs& a, const int chunk, const int h, const int b, const u16* km_lds) {
  constexpr int TPR = D / 16;                  // lanes per row
  constexpr int RW = quant_wave_rows(D);       // rows per pass of a wavefront
  constexpr int WROWS = NP * RW;               // rows of a wavefront
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tr = lane / TPR, tc = lane % TPR;

  int L = a.L;
  int64_t xbase, obase, sidx, dbase;
  if (a.cu_seqlens) {
    int s0 = a.cu_seqlens[b];
    L = a.cu_seqlens[b + 1] - s0;
    dbase = (int64_t)h * a.dot_total + s0;
    xbase = (int64_t)s0 * a.x_sn + (int64_t)h * a.x_sh;
    obase = (int64_t)s0 * a.o_sn + (int64_t)h * a.o_sh;
    sidx = (int64_t)h * a.scale_sh + a.cu_blocks[b];
  } else {
    xbase = (int64_t)b * a.x_sb + (int64_t)h * a.x_sh;
    obase = (int64_t)b * a.o_sb + (int64_t)h * a.o_sh;
    sidx = (((int64_t)b * a.H + h) * ((L + a.blk - 1) >> a.blk_shift)) * a.groups;
    dbase = ((int64_t)b * a.H + h) * L;
  }
  const int n0 = chunk * 4 * WROWS;
  if (n0 >= L) return;
  const int wrow = n0 + w * WROWS, row = wrow + tr;   // first row of the wavefront, of this lane

  // (rows past the end read the last one again: no branch between the loads)
  uint4 raw[NP][2];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const u16* src = a.x + xbase + (int64_t)min(row + p * RW, L - 1) * a.x_sn + tc * 16;
    raw[p][0] = load_stream16(src);
    raw[p][1] = load_stream16(src + 8);
  }
  // k - km is rounded to the input dtype (quant_per_block.py:53-54: the subtraction happens in torch, in
  // the tensor's dtype); both passes then see the rounded difference.
  if (a.km != nullptr || km_lds != nullptr) {
    uint4 kmr[2];
    if (km_lds) {
      kmr[0] = *reinterpret_cast<const uint4*>(km_lds + tc * 16);
      kmr[1] = *reinterpret_cast<const uint4*>(km_lds + tc * 16 + 8);
    } else {
      const uint4* kp = reinterpret_cast<const uint4*>(a.km + (int64_t)b * a.km_sb + (int64_t)h * a.km_sh + tc * 16);
      kmr[0] = kp[0];
      kmr[1] = kp[1];
    }
    const uint32_t* km2 = reinterpret_cast<const uint32_t*>(kmr);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      float mlo, mhi;
      unpack2<DT>(km2[i], mlo, mhi);
#pragma unroll
      for (int p = 0; p < NP; p++) {
        uint32_t* x2 = reinterpret_cast<uint32_t*>(raw[p]);
        float lo, hi;
        unpack2<DT>(x2[i], lo, hi);
        x2[i] = pack2<DT>(lo - mlo, hi - mhi);
      }
    }
  }
  float x[NP][16];   // the fp32 values that are quantised
  float amax = 0.f;
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const uint32_t* x2 = reinterpret_cast<const uint32_t*>(raw[p]);
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      unpack2<DT>(x2[i], x[p][2 * i], x[p][2 * i + 1]);
      if constexpr (!UNIT) { x[p][2 * i] *= a.mult; x[p][2 * i + 1] *= a.mult; }
      mx = fmaxf(mx, fmaxf(fabsf(x[p][2 * i]), fabsf(x[p][2 * i + 1])));
    }
    amax = fmaxf(amax, row + p * RW < L ? mx : 0.f);
  }
  // Optional side output: the dot product of every (scaled) row with a per-(batch, kv-head) vector.
  // The one-call pipeline uses it with the K mean to return the LSE of the unsmoothed logits.
  if (a.dot_out != nullptr) {
    const uint4* dp = reinterpret_cast<const uint4*>(a.dotv + (int64_t)b * a.dv_sb + (int64_t)(h / a.dv_group) * a.dv_sh + tc * 16);
    const uint4 raw2[2] = {dp[0], dp[1]};
    const uint32_t* d2 = reinterpret_cast<const uint32_t*>(raw2);
#pragma unroll
    for (int p = 0; p < NP; p++) {
      float dsum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        float lo, hi;
        unpack2<DT>(d2[i], lo, hi);
        dsum = __builtin_fmaf(x[p][2 * i], lo, dsum);
        dsum = __builtin_fmaf(x[p][2 * i + 1], hi, dsum);
      }
#pragma unroll
      for (int o = 1; o < TPR; o <<= 1) dsum += __shfl_xor(dsum, o);   // the TPR lanes of a row are neighbours
      if (row + p * RW < L && tc == 0) a.dot_out[dbase + row + p * RW] = dsum;
    }
  }
  __shared__ float wmax[4];
  __shared__ int gmax[4][8];
  const int wpb = a.blk / WROWS;               // wavefronts per scale block (1, 2 or 4)
  const int blk_first = w & ~(wpb - 1);        // first wavefront of this one's block
  const int blkid = wrow >> a.blk_shift;
  const bool block_there = blkid << a.blk_shift < L;
  if (a.groups == 1) {
    amax = wave_max(amax);
    if (wpb > 1) {
      if (lane == 0) wmax[w] = amax;
      __syncthreads();
      for (int i = 0; i < wpb; i++) amax = fmaxf(amax, wmax[blk_first + i]);
    }
  } else {
    // Interleaved scales per block (eight: group = row % 8; four: group = (row % 8) / 2): every row this lane holds has
    // the same index modulo 8 (a wavefront's rows start at a multiple of 8 and its passes are RW rows apart), so the lane belongs
    // to one group.  Maximum over the lanes of a row, then over the rows of the group through LDS (the values are non-negative
    // floats: their bit patterns order like integers).
    static_assert(RW % 8 == 0 && WROWS % 8 == 0, "a lane's rows must share their index modulo 8");
    if (threadIdx.x < 32) gmax[threadIdx.x >> 3][threadIdx.x & 7] = 0;
    __syncthreads();
#pragma unroll
    for (int o = 1; o < TPR; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    const int gid = a.groups == 8 ? (tr & 7) : ((tr & 7) >> 1);
    if (tc == 0) atomicMax(&gmax[blk_first][gid], __builtin_bit_cast(int, amax));
    __syncthreads();
    amax = __builtin_bit_cast(float, gmax[blk_first][gid]);
  }
  const float scale = fmaxf(amax / 127.0f, kScaleFloor);
  if (w == blk_first && block_there) {
    if (a.groups == 1) { if (lane == 0) a.scale[sidx + blkid] = scale; }
    else if (lane < a.groups) a.scale[sidx + (int64_t)blkid * a.groups + lane] = fmaxf(__builtin_bit_cast(float, gmax[blk_first][lane]) / 127.0f, kScaleFloor);
  }

  const float rcp = 1.0f / scale;
  // One wavefront-uniform branch around the whole second pass, not one per element (the scale is uniform over the wavefront,
  // or, with interleaved scales, over a lane group: if any lane of the wavefront needs the general division, all take it --
  // where the correction step applies, the two quotients are the same numbers).
  auto quantise_rows = [&](auto quotient) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      uint32_t packed[4];
      pack_codes(x[p], packed, quotient);
      if (row + p * RW < L)
        store_stream16(a.out + obase + (int64_t)(row + p * RW) * a.o_sn + tc * 16, make_uint4(packed[0], packed[1], packed[2], packed[3]));
    }
  };
  if (__builtin_amdgcn_ballot_w64(!reciprocal_is_exact(scale)) == 0) quantise_rows([&](float v) { return div_by_uniform(v, scale, rcp); });
  else {
    const double wide = 1.0 / (double)scale;
    quantise_rows([&](float v) { return div_by_any(v, wide); });
  }
}

template <int DT, int D, int NP>
__global__ void __launch_bounds__(256) quant_int8_kernel(QuantArgs a) {
  if (a.mult == 1.0f) quant_int8_rows<DT, D, NP, true>(a, blockIdx.x, blockIdx.y, blockIdx.z, nullptr);
  else quant_int8_rows<DT, D, NP, false>(a, blockIdx.x, blockIdx.y, blockIdx.z, nullptr);
}

// ---------------------------------------------------------------------------------------------
// Column statistics over the sequence: MODE 0 = float64 sum (K mean), MODE 1 = fp32 abs-max (V).
// Stage 1: one workgroup per (chunk of kChunkRows rows, head, batch) writes D partials.
// Stage 2: one workgroup per (head, batch) combines the partials in chunk order.
// ---------------------------------------------------------------------------------------------
constexpr int kChunkRows = 512;


template <int DT, int D, int MODE>
__global__ void __launch_bounds__(256) colstat_partial_kernel(ColStatArgs a) {
  using acc_t = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int TPR = D / 8, RPP = 256 / TPR;
  const int chunk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, tr = tid / TPR, tc = tid % TPR;
  int L = a.L;
  int64_t xbase;
  if (a.cu_seqlens) {
    int s0 = a.cu_seqlens[b];
    L = a.cu_seqlens[b + 1] - s0;
    xbase = (int64_t)s0 * a.x_sn + (int64_t)h * a.x_sh;
  } else {
    xbase = (int64_t)b * a.x_sb + (int64_t)h * a.x_sh;
  }
  const int n0 = chunk * kChunkRows;
  if (n0 >= L) return;
  const int n1 = min(L, n0 + kChunkRows);
  acc_t acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++) acc[i] = 0;
  auto fold = [&](const uint4& raw) {
    const u16* e = reinterpret_cast<const u16*>(&raw);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      float x = to_f32<DT>(e[i]);
      if constexpr (MODE == 0) acc[i] += (double)x;
      else acc[i] = fmaxf(acc[i], fabsf(x));
    }
  };
  // Eight independent 16-byte loads per lane in flight (the pass is a pure read: what limits it is the bytes on their
  // way, not the arithmetic); the float64 sum of fp16/bf16 values is exact, so the order of the additions is free.
  constexpr int UNR = 8;
  const u16* base = a.x + xbase + tc * 8;
  int n = n0 + tr;
  for (; n + (UNR - 1) * RPP < n1; n += UNR * RPP) {
    uint4 raw[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) raw[u] = load_stream16(base + (int64_t)(n + u * RPP) * a.x_sn);
#pragma unroll
    for (int u = 0; u < UNR; u++) fold(raw[u]);
  }
  for (; n < n1; n += RPP) fold(load_stream16(base + (int64_t)n * a.x_sn));
  __shared__ acc_t red[RPP][D];
#pragma unroll
  for (int i = 0; i < 8; i++) red[tr][tc * 8 + i] = acc[i];
  __syncthreads();
  if (tid < D) {
    acc_t t = red[0][tid];
    for (int r = 1; r < RPP; r++) {
      if constexpr (MODE == 0) t += red[r][tid];
      else t = fmaxf(t, red[r][tid]);
    }
    reinterpret_cast<acc_t*>(a.partial)[(((int64_t)b * a.H + h) * a.nchunk + chunk) * D + tid] = t;
  }
}

// K mean: sum partials in chunk order (float64), /L, -> fp32 -> input dtype.
template <int DT>
__global__ void kmean_finalize_kernel(const double* partial, u16* km, int H, int L, int D, int nchunk,
                                      const int32_t* cu_seqlens) {
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  if (cu_seqlens) L = cu_seqlens[b + 1] - cu_seqlens[b];
  if (d >= D) return;
  int nc = (L + kChunkRows - 1) / kChunkRows;
  // eight partials in flight at a time (the loads are what this kernel waits for); still added in chunk order
  const double* p = partial + (((int64_t)b * H + h) * nchunk) * D + d;
  double s = 0;
  int c = 0;
  for (; c + 8 <= nc; c += 8) {
    double t[8];
#pragma unroll
    for (int i = 0; i < 8; i++) t[i] = p[(int64_t)(c + i) * D];
#pragma unroll
    for (int i = 0; i < 8; i++) s += t[i];
  }
  for (; c < nc; c++) s += p[(int64_t)c * D];
  float m = L > 0 ? (float)(s / (double)L) : 0.f;
  km[((int64_t)b * H + h) * D + d] = from_f32<DT>(m);
}

// V scale: max of partial abs-maxima, scale = max(amax/448, 1e-12).
__global__ void vscale_finalize_kernel(const float* partial, float* vscale, int H, int L, int D, int nchunk,
                                       const int32_t* cu_seqlens) {
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  if (cu_seqlens) L = cu_seqlens[b + 1] - cu_seqlens[b];
  if (d >= D) return;
  int nc = (L + kChunkRows - 1) / kChunkRows;
  const float* p = partial + (((int64_t)b * H + h) * nchunk) * D + d;
  float m = 0.f;
  int c = 0;
  for (; c + 8 <= nc; c += 8) {
    float t[8];
#pragma unroll
    for (int i = 0; i < 8; i++) t[i] = p[(int64_t)(c + i) * D];
#pragma unroll
    for (int i = 0; i < 8; i++) m = fmaxf(m, t[i]);
  }
  for (; c < nc; c++) m = fmaxf(m, p[(int64_t)c * D]);
  vscale[((int64_t)b * H + h) * D + d] = fmaxf(m / 448.0f, kScaleFloor);
}

// ---------------------------------------------------------------------------------------------
// V preparation: one workgroup per panel (128 rows x D of one (batch, head)).
// Elements are converted, scattered into LDS in panel byte order and streamed out linearly.
// ---------------------------------------------------------------------------------------------

// (vs_lds: the per-channel V scales of this (batch, head) in LDS instead of a.vscale in global memory.)
template <int DT, int D, int PV>
__device__ __forceinline__ void prep_v_tile(const PrepVArgs& a, const int pidx, const int h, const int b, const float* vs_lds) {
  // A lane converts 4 consecutive rows x 8 consecutive channels at a time, so that the 4 row values of
  // a channel pack into one dword (fp8) or two (fp16): exactly the (b = 0..3) group of the panel
  // order.  They are staged in LDS as T[channel][row quad] and read back in panel order.
  constexpr int TPR = D / 8, RPP = 256 / TPR;   // lanes per row, row quads handled per pass
  constexpr int NQ = kPanelRows / 4;            // 32 row quads per panel
  constexpr int QPT = NQ / RPP;                 // passes
  constexpr int ESZ = (PV == 1) ? 1 : 2;
  constexpr int QW = ESZ;                       // dwords per (channel, row quad)
  constexpr int TS = NQ * QW + 1;               // dword stride of a channel in LDS (padded)
  constexpr int PANEL_BYTES = kPanelRows * D * ESZ;
  constexpr int DTN = D / 32;
  __shared__ uint32_t T[D * TS];
  const int tid = threadIdx.x, tr = tid / TPR, tc = tid % TPR;
  int L = a.L;
  int64_t vbase, pbase;
  if (a.cu_seqlens) {
    int s0 = a.cu_seqlens[b];
    L = a.cu_seqlens[b + 1] - s0;
    vbase = (int64_t)s0 * a.v_sn + (int64_t)h * a.v_sh;
    pbase = ((int64_t)h * a.panel_sh + a.cu_panels[b] + pidx) * PANEL_BYTES;
  } else {
    vbase = (int64_t)b * a.v_sb + (int64_t)h * a.v_sh;
    pbase = (((int64_t)b * a.H + h) * ((L + kPanelRows - 1) / kPanelRows) + pidx) * PANEL_BYTES;
  }
  const int n0 = pidx * kPanelRows;
  if (n0 >= L) return;
  float sc[8], rc[8];
  bool fast = true;
  if constexpr (PV == 1) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      sc[i] = vs_lds ? vs_lds[tc * 8 + i] : a.vscale[((int64_t)b * a.H + h) * D + tc * 8 + i];
      rc[i] = 1.0f / sc[i];
      fast = fast && ((__builtin_bit_cast(uint32_t, sc[i]) & 0x7fffffu) != 0x7fffffu) && sc[i] < 1.0e30f;
    }
    fast = __builtin_amdgcn_ballot_w64(!fast) == 0;   // the correction-step division for the whole wavefront, or not at all
  }
#pragma unroll
  for (int qq = 0; qq < QPT; qq++) {
    const int quad = qq * RPP + tr;
    uint4 raw[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int r = n0 + 4 * quad + j;
      raw[j] = make_uint4(0, 0, 0, 0);
      if (r < L) raw[j] = load_stream16(a.v + vbase + (int64_t)r * a.v_sn + tc * 8);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; j++) x[j] = to_f32<DT>(reinterpret_cast<const u16*>(&raw[j])[i]);
      uint32_t* dst = &T[(tc * 8 + i) * TS + quad * QW];
      if constexpr (PV == 1) {
        float z[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          z[j] = fast ? div_by_uniform(x[j], sc[i], rc[i]) : x[j] / sc[i];
          z[j] = fminf(fmaxf(z[j], -448.f), 448.f);
        }
        int pk = __builtin_amdgcn_cvt_pk_fp8_f32(z[0], z[1], 0, false);
        pk = __builtin_amdgcn_cvt_pk_fp8_f32(z[2], z[3], pk, true);
        dst[0] = (uint32_t)pk;
      } else {
        dst[0] = (uint32_t)f32_to_f16(x[0]) | ((uint32_t)f32_to_f16(x[1]) << 16);
        dst[1] = (uint32_t)f32_to_f16(x[2]) | ((uint32_t)f32_to_f16(x[3]) << 16);
      }
    }
  }
  __syncthreads();
  uint4* out = reinterpret_cast<uint4*>(a.panels + pbase);
#pragma unroll
  for (int i = 0; i < PANEL_BYTES / 16 / 256; i++) {
    const int c = i * 256 + tid;           // 16-byte chunk of the panel
    const int lane = c & 63, hh = lane >> 5, d_lo = lane & 31;
    uint4 v;
    if constexpr (PV == 1) {
      // c = ((ks*DTN + dt)*2 + half)*64 + lane ; bytes 4a+b <-> row 64ks + 32half + 8a + 4h + b
      const int half = (c >> 6) & 1, dt = (c >> 7) % DTN, ks = (c >> 7) / DTN;
      const uint32_t* src = &T[(32 * dt + d_lo) * TS + 16 * ks + 8 * half + hh];
      v = make_uint4(src[0], src[2], src[4], src[6]);
    } else {
      // c = (ks16*DTN + dt)*64 + lane ; elements 4a+b <-> row 16ks16 + 8a + 4h + b
      const int dt = (c >> 6) % DTN, ks16 = (c >> 6) / DTN;
      const uint32_t* src = &T[(32 * dt + d_lo) * TS + (4 * ks16 + hh) * 2];
      v = make_uint4(src[0], src[1], src[4], src[5]);
    }
    store_stream16(out + c, v);
  }
}

template <int DT, int D, int PV>
__global__ void __launch_bounds__(256) prep_v_kernel(PrepVArgs a) {
  prep_v_tile<DT, D, PV>(a, blockIdx.x, blockIdx.y, blockIdx.z, nullptr);
}

// ---------------------------------------------------------------------------------------------
// Short sequences: every pre-pass of the one-call pipeline in ONE launch.  A workgroup is either a K tile or a V panel
// of one (batch, kv-head); it first computes the statistic its tile needs over the whole sequence itself (the K mean:
// float64 sums in the order of the two-stage kernels above -- per 512-row chunk, per-lane rows, the lanes of a channel
// in order, chunks in order -- so that the mean is the same bit pattern; the V scale: an abs-max, which has no order)
// and then runs the tile code of the kernels above.  The statistics are read again by every workgroup of the
// (batch, head): affordable while the sequence is short and the reads hit the L2; six dependent launches of a few
// microseconds each become one.
// ---------------------------------------------------------------------------------------------
template <int DT, int D, int PV, int NP>
__global__ void __launch_bounds__(256) prepass_small_kernel(QuantArgs qa, PrepVArgs va, int nk, int smooth, u16* km_out,
                                                            float* vscale_out) {
  constexpr int TPR = D / 8, RPP = 256 / TPR;
  const int h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, tr = tid / TPR, tc = tid % TPR;
  __shared__ double red[RPP][D];
  __shared__ __align__(16) u16 km_l[D];
  __shared__ float vs_l[D];
  if ((int)blockIdx.x < nk) {
    if (smooth) {
      const int L = qa.L;
      const int64_t xbase = (int64_t)b * qa.x_sb + (int64_t)h * qa.x_sh;
      double s = 0;
      for (int n0 = 0; n0 < L; n0 += kChunkRows) {
        const int n1 = min(L, n0 + kChunkRows);
        double acc[8];
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] = 0;
#pragma unroll 8
        for (int n = n0 + tr; n < n1; n += RPP) {   // (unrolled for loads in flight; the additions keep their order)
          uint4 raw = *reinterpret_cast<const uint4*>(qa.x + xbase + (int64_t)n * qa.x_sn + tc * 8);
          const u16* e = reinterpret_cast<const u16*>(&raw);
#pragma unroll
          for (int i = 0; i < 8; i++) acc[i] += (double)to_f32<DT>(e[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) red[tr][tc * 8 + i] = acc[i];
        __syncthreads();
        if (tid < D) {
          double t = red[0][tid];
          for (int r = 1; r < RPP; r++) t += red[r][tid];
          s += t;
        }
        __syncthreads();
      }
      if (tid < D) {
        const u16 m = from_f32<DT>(L > 0 ? (float)(s / (double)L) : 0.f);
        km_l[tid] = m;
        if (blockIdx.x == 0) km_out[((int64_t)b * qa.H + h) * D + tid] = m;
      }
      __syncthreads();
    }
    quant_int8_rows<DT, D, NP, true>(qa, blockIdx.x, h, b, smooth ? km_l : nullptr);   // (K: the multiplier is 1)
  } else {
    const int pidx = blockIdx.x - nk;
    if constexpr (PV == 1) {
      const int L = va.L;
      const int64_t vbase = (int64_t)b * va.v_sb + (int64_t)h * va.v_sh;
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; i++) acc[i] = 0.f;
#pragma unroll 8
      for (int n = tr; n < L; n += RPP) {
        uint4 raw = *reinterpret_cast<const uint4*>(va.v + vbase + (int64_t)n * va.v_sn + tc * 8);
        const u16* e = reinterpret_cast<const u16*>(&raw);
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] = fmaxf(acc[i], fabsf(to_f32<DT>(e[i])));
      }
      float* redf = reinterpret_cast<float*>(&red[0][0]);
#pragma unroll
      for (int i = 0; i < 8; i++) redf[tr * D + tc * 8 + i] = acc[i];
      __syncthreads();
      if (tid < D) {
        float t = redf[tid];
        for (int r = 1; r < RPP; r++) t = fmaxf(t, redf[r * D + tid]);
        const float sc = fmaxf(t / 448.0f, kScaleFloor);
        vs_l[tid] = sc;
        if (pidx == 0) vscale_out[((int64_t)b * va.H + h) * D + tid] = sc;
      }
      __syncthreads();
    }
    prep_v_tile<DT, D, PV>(va, pidx, h, b, PV == 1 ? vs_l : nullptr);
  }
}

// ---------------------------------------------------------------------------------------------
// Boolean mask -> bits and visibility (layout in sage_common.h).  One workgroup per (key tile, q-tile, plane): the
// mask's bytes are read once, 16 per lane and eight lanes per row where keys are contiguous, and leave as one bit each.
// ---------------------------------------------------------------------------------------------
__device__ inline unsigned nonzero_bytes(unsigned x) {   // bit i: byte i of x is not zero
  const unsigned t = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) >> 7) & 0x01010101u;
  return (t * 0x10204080u) >> 28;
}

__global__ void __launch_bounds__(256) mask_pack_kernel(const uint8_t* mask, int64_t m_sb, int64_t m_sh, int64_t m_sm, int64_t m_sn,
                                                        MaskPlanes p, int Sq, int Skv, uint8_t* bits, uint8_t* seen) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4), aligned(1)));
  __shared__ __align__(16) uint8_t packed[kMaskTileBytes];
  __shared__ unsigned wave_seen[4];
  const int tile = blockIdx.x, qt = blockIdx.y, tid = threadIdx.x;
  const int heads = p.ph ? (p.pb ? p.pb : p.planes) : 1;   // planes of one batch entry
  const int b = blockIdx.z / heads, hd = blockIdx.z - b * heads;
  const uint8_t* base = mask + (int64_t)b * m_sb + (int64_t)hd * m_sh;
  const int rows = m_sm ? min(kMaskRows, Sq - qt * kMaskRows) : kMaskRows;   // (rows that all read the same row are all valid)
  base += (int64_t)qt * kMaskRows * m_sm;
  // chunk c (16 keys from tile * kMaskKeys + 16 * c on) of row r: keys 0-3 and 8-11 belong to lane half 0, the others to half 1
  auto store = [&](int r, int c, const unsigned (&x)[4]) {
    packed[r * 16 + c] = (uint8_t)(nonzero_bytes(x[0]) | (nonzero_bytes(x[2]) << 4));
    packed[r * 16 + 8 + c] = (uint8_t)(nonzero_bytes(x[1]) | (nonzero_bytes(x[3]) << 4));
  };
  if (m_sn == 1 && Skv >= 16) {
    // One load per chunk; the chunk that ends a row is the row's last 16 keys, moved down.  (Key by key behind its bounds check
    // it was sixteen dependent loads for each of eight rows: 2 x 16 heads of 1500 rows, head_dim 64, FP16 P.V, a document mask,
    // the call 68.9 -> 62.5 us; transposed 100.4 -> 80.)
    const int c = tid & 7, k0 = tile * kMaskKeys + 16 * c, k = min(k0, Skv - 16), down = 8 * (k0 - k);
#pragma unroll
    for (int i = 0; i < kMaskRows / 32; i++) {
      const int r = tid / 8 + 32 * i;
      u32x4 v = {0, 0, 0, 0};
      if (r < rows && k0 < Skv) v = *reinterpret_cast<const u32x4*>(base + (int64_t)r * m_sm + k);
      uint64_t lo = v[0] | (uint64_t)v[1] << 32, hi = v[2] | (uint64_t)v[3] << 32;
      if (down >= 64) { lo = down < 128 ? hi >> (down - 64) : 0; hi = 0; }
      else if (down > 0) { lo = lo >> down | hi << (64 - down); hi >>= down; }
      const unsigned x[4] = {(unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32)};
      store(r, c, x);
    }
  } else {
    // Other strides: sixteen clamped byte loads in flight, neighbouring lanes on the axis whose elements are closer together
    // (along the rows only where most lanes have one).
    const bool rows_near = rows > kMaskRows / 2 && (m_sm < 0 ? -m_sm : m_sm) < (m_sn < 0 ? -m_sn : m_sn);
    for (int i = 0; i < kMaskRows / 32; i++) {
      const int r = rows_near ? tid : tid / 8 + 32 * i, c = rows_near ? i : tid & 7, k0 = tile * kMaskKeys + 16 * c;
      unsigned x[4] = {0, 0, 0, 0};
      if (r < rows && k0 < Skv) {
        const uint8_t* src = base + (int64_t)r * m_sm;
        uint8_t key[16];
#pragma unroll
        for (int e = 0; e < 16; e++) key[e] = src[(int64_t)min(k0 + e, Skv - 1) * m_sn];
#pragma unroll
        for (int e = 0; e < 16; e++) x[e >> 2] |= (unsigned)(k0 + e < Skv && key[e]) << (8 * (e & 3));
      }
      store(r, c, x);
    }
  }
  __syncthreads();
  const uint4 row = reinterpret_cast<const uint4*>(packed)[tid];
  const int64_t t = ((int64_t)blockIdx.z * p.nqt + qt) * p.ntk + tile;
  reinterpret_cast<uint4*>(bits + t * kMaskTileBytes)[tid] = row;
  const unsigned long long any = __builtin_amdgcn_ballot_w64((row.x | row.y | row.z | row.w) != 0);
  if ((tid & 63) == 0) wave_seen[tid >> 6] = ((unsigned)any != 0 ? 1 : 0) | ((any >> 32) != 0 ? 2 : 0);
  __syncthreads();
  if (tid == 0) seen[t] = (uint8_t)(wave_seen[0] | wave_seen[1] << 2 | wave_seen[2] << 4 | wave_seen[3] << 6);
}

// ---------------------------------------------------------------------------------------------
// Host-side launchers (called from the C ABI in sage_api.hip).
// ---------------------------------------------------------------------------------------------
hipError_t launch_quant_int8(const QuantArgs& a, int dtype, int max_rows, hipStream_t st) {
  const int rows = quant_rows(a.D, a.blk);
  dim3 grid((max_rows + rows - 1) / rows, a.H, a.B), block(256);
#define SAGE_QUANT(DT, DD, NP) quant_int8_kernel<DT, DD, NP><<<grid, block, 0, st>>>(a)
#define SAGE_QUANT_D(DT) \
  do { \
    if (a.D == 64) { if (quant_passes(64, a.blk) == 1) SAGE_QUANT(DT, 64, 1); else SAGE_QUANT(DT, 64, 2); } \
    else { if (quant_passes(128, a.blk) == 2) SAGE_QUANT(DT, 128, 2); else SAGE_QUANT(DT, 128, 4); } \
  } while (0)
  if (dtype == 0) SAGE_QUANT_D(0);
  else SAGE_QUANT_D(1);
#undef SAGE_QUANT_D
#undef SAGE_QUANT
  return hipGetLastError();
}

hipError_t launch_mask_pack(const uint8_t* mask, int64_t m_sb, int64_t m_sh, int64_t m_sm, int64_t m_sn, const MaskPlanes& p, int Sq,
                            int Skv, uint8_t* bits, uint8_t* seen, hipStream_t st) {
  mask_pack_kernel<<<dim3(p.ntk, p.nqt, p.planes), dim3(256), 0, st>>>(mask, m_sb, m_sh, m_sm, m_sn, p, Sq, Skv, bits, seen);
  return hipGetLastError();
}

int colstat_chunks(int L) { return (L + kChunkRows - 1) / kChunkRows; }

template <int MODE>
static hipError_t launch_colstat(const ColStatArgs& a, int dtype, hipStream_t st) {
  dim3 grid(a.nchunk, a.H, a.B), block(256);
  if (dtype == 0 && a.D == 64) colstat_partial_kernel<0, 64, MODE><<<grid, block, 0, st>>>(a);
  else if (dtype == 0 && a.D == 128) colstat_partial_kernel<0, 128, MODE><<<grid, block, 0, st>>>(a);
  else if (dtype == 1 && a.D == 64) colstat_partial_kernel<1, 64, MODE><<<grid, block, 0, st>>>(a);
  else colstat_partial_kernel<1, 128, MODE><<<grid, block, 0, st>>>(a);
  return hipGetLastError();
}

hipError_t launch_k_mean(const ColStatArgs& a, int dtype, void* km, hipStream_t st) {
  if (a.nchunk == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  hipError_t e = launch_colstat<0>(a, dtype, st);
  if (e != hipSuccess) return e;
  dim3 grid(a.H, a.B), block(a.D);
  if (dtype == 0) kmean_finalize_kernel<0><<<grid, block, 0, st>>>((const double*)a.partial, (u16*)km, a.H, a.L, a.D, a.nchunk, a.cu_seqlens);
  else kmean_finalize_kernel<1><<<grid, block, 0, st>>>((const double*)a.partial, (u16*)km, a.H, a.L, a.D, a.nchunk, a.cu_seqlens);
  return hipGetLastError();
}

hipError_t launch_v_scale(const ColStatArgs& a, int dtype, float* vscale, hipStream_t st) {
  if (a.nchunk == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  hipError_t e = launch_colstat<1>(a, dtype, st);
  if (e != hipSuccess) return e;
  dim3 grid(a.H, a.B), block(a.D);
  vscale_finalize_kernel<<<grid, block, 0, st>>>((const float*)a.partial, vscale, a.H, a.L, a.D, a.nchunk, a.cu_seqlens);
  return hipGetLastError();
}

hipError_t launch_prepass_small(const QuantArgs& qa, const PrepVArgs& va, int dtype, int pv, int smooth, void* km_out,
                                float* vscale_out, hipStream_t st) {
  const int rows = quant_rows(qa.D, qa.blk);
  const int nk = (qa.L + rows - 1) / rows, nv = (va.L + kPanelRows - 1) / kPanelRows;
  if (nk + nv == 0 || qa.B == 0 || qa.H == 0) return hipSuccess;
  dim3 grid(nk + nv, qa.H, qa.B), block(256);
#define SAGE_PREPASS(DT, DD, PVV, NP) prepass_small_kernel<DT, DD, PVV, NP><<<grid, block, 0, st>>>(qa, va, nk, smooth, (u16*)km_out, vscale_out)
#define SAGE_PREPASS_D(DT, PVV) \
  do { \
    if (qa.D == 64) { if (quant_passes(64, qa.blk) == 1) SAGE_PREPASS(DT, 64, PVV, 1); else SAGE_PREPASS(DT, 64, PVV, 2); } \
    else { if (quant_passes(128, qa.blk) == 2) SAGE_PREPASS(DT, 128, PVV, 2); else SAGE_PREPASS(DT, 128, PVV, 4); } \
  } while (0)
  if (dtype == 0) { if (pv) SAGE_PREPASS_D(0, 1); else SAGE_PREPASS_D(0, 0); }
  else { if (pv) SAGE_PREPASS_D(1, 1); else SAGE_PREPASS_D(1, 0); }
#undef SAGE_PREPASS_D
#undef SAGE_PREPASS
  return hipGetLastError();
}

hipError_t launch_prep_v(const PrepVArgs& a, int dtype, int pv, int max_panels, hipStream_t st) {
  if (max_panels == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  dim3 grid(max_panels, a.H, a.B), block(256);
#define SAGE_PREPV(DT, DD, PVV) prep_v_kernel<DT, DD, PVV><<<grid, block, 0, st>>>(a)
  if (dtype == 0) {
    if (a.D == 64) { if (pv) SAGE_PREPV(0, 64, 1); else SAGE_PREPV(0, 64, 0); }
    else { if (pv) SAGE_PREPV(0, 128, 1); else SAGE_PREPV(0, 128, 0); }
  } else {
    if (a.D == 64) { if (pv) SAGE_PREPV(1, 64, 1); else SAGE_PREPV(1, 64, 0); }
    else { if (pv) SAGE_PREPV(1, 128, 1); else SAGE_PREPV(1, 128, 0); }
  }
#undef SAGE_PREPV
  return hipGetLastError();
}

}  // namespace sage
