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
#include <cstring>
#include "sage_launch.h"
#include "sage_plan.h"

#pragma clang fp contract(off)

namespace sage {

constexpr int kChunkRows = 512;   // rows of a chunk of the column statistics

// Barrier that orders LDS traffic only: loads in flight stay in flight.
__device__ inline void lds_only_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Where a quantiser workgroup has the K mean from.  request() is called before the loads of the rows, read() after them (by every lane
// of the workgroup): 16 channels from tc * 16 on, in the input type; false: nothing to subtract.
template <int DT, int D>
struct MeanInMemory {   // QuantArgs::km
  const QuantArgs& a;
  const int h, b;
  __device__ void request(int) {}
  __device__ bool read(uint4 (&km)[2], int tc, int, bool) {
    if (a.km == nullptr) return false;
    const uint4* p = reinterpret_cast<const uint4*>(a.km + (int64_t)b * a.km_sb + (int64_t)h * a.km_sh + tc * 16);
    km[0] = p[0];
    km[1] = p[1];
    return true;
  }
};
template <int DT, int D>
struct MeanInLds {      // computed by the same workgroup; null: nothing to subtract
  const u16* km_lds;
  __device__ void request(int) {}
  __device__ bool read(uint4 (&km)[2], int tc, int, bool) {
    if (km_lds == nullptr) return false;
    km[0] = *reinterpret_cast<const uint4*>(km_lds + tc * 16);
    km[1] = *reinterpret_cast<const uint4*>(km_lds + tc * 16 + 8);
    return true;
  }
};
template <int DT, int D>
struct MeanFromPartials {   // QuantArgs::km_partial, combined in chunk order like kmean_finalize_kernel
  const QuantArgs& a;
  const int h, b;
  u16* km_lds;
  double t[kFusedChunks];
  __device__ int chunks(int L) const { return min((L + kChunkRows - 1) / kChunkRows, a.km_nchunk); }
  __device__ void request(int L) {
    const int nc = chunks(L);
    const double* p = a.km_partial + ((int64_t)b * a.H + h) * a.km_nchunk * D + threadIdx.x;
    if (threadIdx.x < D) {
#pragma unroll
      for (int c = 0; c < kFusedChunks; c++) t[c] = p[(int64_t)min(c, nc - 1) * D];
    }
  }
  __device__ bool read(uint4 (&km)[2], int tc, int L, bool first) {
    const int nc = chunks(L);
    if (threadIdx.x < D) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < kFusedChunks; c++) s = c < nc ? s + t[c] : s;
      const u16 m = from_f32<DT>((float)(s / (double)L));
      km_lds[threadIdx.x] = m;
      if (first) a.km_out[((int64_t)b * a.H + h) * D + threadIdx.x] = m;
    }
    lds_only_barrier();
    return MeanInLds<DT, D>{km_lds}.read(km, tc, L, first);
  }
};

// Quantises the rows chunk * quant_rows(D, blk) .. of (batch b, head h), which stay in registers, as floats, between the abs-max and
// the rounding.  A lane owns 16 consecutive channels of a row (two 128-bit loads, one 128-bit store); all its loads are issued
// before anything waits for one.
// UNIT: the multiplier is 1 (every K call; x * 1.0f is x, so leaving the product out changes no bit).
template <int DT, int D, int NP, bool UNIT, class Mean>
__device__ __forceinline__ void quant_int8_rows(const QuantArgs& a, const int chunk, const int h, const int b, Mean mean) {
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

  mean.request(L);
  // (rows past the end read the last one again: no branch between the loads)
  uint4 raw[NP][2];
  with_loads(a.cached, [&](auto load) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const u16* src = a.x + xbase + (int64_t)min(row + p * RW, L - 1) * a.x_sn + tc * 16;
      raw[p][0] = load(src);
      raw[p][1] = load(src + 8);
    }
  });
  // k - km is rounded to the input dtype (quant_per_block.py:53-54: the subtraction happens in torch, in
  // the tensor's dtype); both passes then see the rounded difference.
  uint4 kmr[2];
  if (mean.read(kmr, tc, L, chunk == 0)) {
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

template <int DT, int D, int NP, bool PARTIAL = false>
__global__ void __launch_bounds__(256) quant_int8_kernel(QuantArgs a) {
  const int chunk = a.heads_first ? blockIdx.y : blockIdx.x, h = a.heads_first ? blockIdx.x : blockIdx.y, b = blockIdx.z;
  if constexpr (PARTIAL) {
    __shared__ __align__(16) u16 km_lds[D];
    quant_int8_rows<DT, D, NP, true>(a, chunk, h, b, MeanFromPartials<DT, D>{a, h, b, km_lds});
    return;
  }
  const MeanInMemory<DT, D> mean = {a, h, b};
  if (a.mult == 1.0f) quant_int8_rows<DT, D, NP, true>(a, chunk, h, b, mean);
  else quant_int8_rows<DT, D, NP, false>(a, chunk, h, b, mean);
}

// ---------------------------------------------------------------------------------------------
// Column statistics over the sequence: MODE 0 = float64 sum (K mean), MODE 1 = fp32 abs-max (V).
// Stage 1: one workgroup per (chunk of kChunkRows rows, head, batch) writes D partials.
// Stage 2: one workgroup per (head, batch) combines the partials in chunk order.
// ---------------------------------------------------------------------------------------------
constexpr int colstat_lds_bytes(int D) { return 256 / (D / 8) * D * 8; }

template <int DT, int D, int MODE>
__device__ __forceinline__ void colstat_chunk(const ColStatArgs a, const int chunk, const int h, const int b, void* lds) {
  using acc_t = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int TPR = D / 8, RPP = 256 / TPR;
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
  with_loads(a.cached, [&](auto load) __attribute__((always_inline)) {
    for (; n + (UNR - 1) * RPP < n1; n += UNR * RPP) {
      uint4 raw[UNR];
#pragma unroll
      for (int u = 0; u < UNR; u++) raw[u] = load(base + (int64_t)(n + u * RPP) * a.x_sn);
#pragma unroll
      for (int u = 0; u < UNR; u++) fold(raw[u]);
    }
    for (; n < n1; n += RPP) fold(load(base + (int64_t)n * a.x_sn));
  });
  acc_t(*red)[D] = reinterpret_cast<acc_t(*)[D]>(lds);
#pragma unroll
  for (int i = 0; i < 8; i++) red[tr][tc * 8 + i] = acc[i];
  __syncthreads();
  if (tid < D) {
    acc_t t = red[0][tid];
#pragma unroll 1
    for (int r0 = 0; r0 < RPP; r0 += 8) {   // eight reads in flight; added in row order
      acc_t u[8];
#pragma unroll
      for (int i = 0; i < 8; i++) u[i] = red[r0 + i][tid];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (r0 + i == 0) continue;
        if constexpr (MODE == 0) t += u[i];
        else t = fmaxf(t, u[i]);
      }
    }
    reinterpret_cast<acc_t*>(a.partial)[(((int64_t)b * a.H + h) * a.nchunk + chunk) * D + tid] = t;
  }
}

template <int DT, int D, int MODE>
__global__ void __launch_bounds__(256) colstat_partial_kernel(ColStatArgs a) {
  __shared__ __align__(16) uint8_t lds[colstat_lds_bytes(D) / (MODE == 0 ? 1 : 2)];
  const bool hf = a.heads_first;
  colstat_chunk<DT, D, MODE>(a, hf ? blockIdx.y : blockIdx.x, hf ? blockIdx.x : blockIdx.y, blockIdx.z, lds);
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

// Where a panel workgroup has the V scales from: like the K mean of the quantiser, D values in LDS or in memory.
struct ScalesInMemory {
  const float* p;
  __device__ void request(int) {}
  __device__ const float* ready(int, bool) { return p; }
};
template <int D>
struct ScalesFromPartials {   // PrepVArgs::vs_partial, like vscale_finalize_kernel
  const PrepVArgs& a;
  const int h, b;
  float* vs_lds;
  float t[kFusedChunks];
  __device__ void request(int L) {
    const int nc = min((L + kChunkRows - 1) / kChunkRows, a.vs_nchunk);
    const float* p = a.vs_partial + ((int64_t)b * a.H + h) * a.vs_nchunk * D + threadIdx.x;
    if (threadIdx.x < D) {
#pragma unroll
      for (int c = 0; c < kFusedChunks; c++) t[c] = p[(int64_t)min(c, nc - 1) * D];
    }
  }
  __device__ const float* ready(int, bool first) {
    if (threadIdx.x < D) {
      float m = 0.f;
#pragma unroll
      for (int c = 0; c < kFusedChunks; c++) m = fmaxf(m, t[c]);   // (chunks past the last repeat it)
      const float s = fmaxf(m / 448.0f, kScaleFloor);
      vs_lds[threadIdx.x] = s;
      if (first) a.vscale_out[((int64_t)b * a.H + h) * D + threadIdx.x] = s;
    }
    lds_only_barrier();
    return vs_lds;
  }
};

// LDS of a panel job: T[channel][row quad], dword stride of a channel padded by one
__host__ __device__ constexpr int prep_v_lds_bytes(int D, int PV) { return D * (kPanelRows / 4 * (PV == 1 ? 1 : 2) + 1) * 4; }

template <int DT, int D, int PV, class Scales>
__device__ __forceinline__ void prep_v_tile(const PrepVArgs& a, const int pidx, const int h, const int b, Scales scales, uint32_t* T) {
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
  static_assert(D * TS * 4 == prep_v_lds_bytes(D, PV), "LDS size");
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
  if constexpr (PV == 1) scales.request(L);
  // (all rows are requested before anything waits; those past the end read the last one again and become zeros)
  uint4 raw[QPT][4];
  with_loads(a.cached, [&](auto load) __attribute__((always_inline)) {
#pragma unroll
    for (int qq = 0; qq < QPT; qq++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int r = n0 + 4 * (qq * RPP + tr) + j;
        raw[qq][j] = load(a.v + vbase + (int64_t)min(r, L - 1) * a.v_sn + tc * 8);
      }
  });
  auto row_there = [&](int qq, int j) { return n0 + 4 * (qq * RPP + tr) + j < L; };
  if constexpr (PV == 1) {
    const float* vs = scales.ready(L, pidx == 0);
    float sc[8];
    bool exact = true;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      sc[i] = vs[tc * 8 + i];
      exact = exact && reciprocal_is_exact(sc[i]);
    }
    auto convert = [&](auto quotient) __attribute__((always_inline)) {
#pragma unroll
      for (int qq = 0; qq < QPT; qq++) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          float z[4];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float x = to_f32<DT>(reinterpret_cast<const u16*>(&raw[qq][j])[i]);
            z[j] = fminf(fmaxf(quotient(row_there(qq, j) ? x : 0.f, i), -448.f), 448.f);
          }
          int pk = __builtin_amdgcn_cvt_pk_fp8_f32(z[0], z[1], 0, false);
          pk = __builtin_amdgcn_cvt_pk_fp8_f32(z[2], z[3], pk, true);
          T[(tc * 8 + i) * TS + qq * RPP + tr] = (uint32_t)pk;
        }
        __builtin_amdgcn_sched_barrier(0);   // (one pass after the other: both at once take twice the registers)
      }
    };
    // (the correction-step division for the whole wavefront, or the general one)
    if (__builtin_amdgcn_ballot_w64(!exact) == 0) {
      float rc[8];
#pragma unroll
      for (int i = 0; i < 8; i++) rc[i] = 1.0f / sc[i];
      convert([&](float x, int i) { return div_by_uniform(x, sc[i], rc[i]); });
    } else {
      convert([&](float x, int i) { return div_by_any(x, 1.0 / (double)sc[i]); });
    }
  } else {
#pragma unroll
    for (int qq = 0; qq < QPT; qq++)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          x[j] = to_f32<DT>(reinterpret_cast<const u16*>(&raw[qq][j])[i]);
          if (!row_there(qq, j)) x[j] = 0.f;
        }
        uint32_t* dst = &T[(tc * 8 + i) * TS + (qq * RPP + tr) * QW];
        dst[0] = pack2<0>(x[0], x[1]);
        dst[1] = pack2<0>(x[2], x[3]);
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
    store16(D == 64 && PV == 0 && a.cached, out + c, v);   // (see inputs_stay)
  }
}

template <int DT, int D, int PV, bool PARTIAL = false>
__global__ void __launch_bounds__(256) prep_v_kernel(PrepVArgs a) {
  __shared__ __align__(16) uint32_t T[prep_v_lds_bytes(D, PV) / 4];
  const int panel = a.heads_first ? blockIdx.y : blockIdx.x, h = a.heads_first ? blockIdx.x : blockIdx.y, b = blockIdx.z;
  if constexpr (PARTIAL) {
    __shared__ float vs_lds[D];
    prep_v_tile<DT, D, PV>(a, panel, h, b, ScalesFromPartials<D>{a, h, b, vs_lds}, T);
  } else prep_v_tile<DT, D, PV>(a, panel, h, b, ScalesInMemory{a.vscale + ((int64_t)b * a.H + h) * D}, T);
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
// Hands the rows n, n + RPP, ... below n1 of a lane's channels to `fold`, in that order, sixteen loads in flight: the statistic is
// latency from end to end, and with the unrolling left to the compiler it took between four and thirty of them, 35 to 45 us for
// the call on 8 heads of 1000 rows at head_dim 128.  (Rows past the end arrive as zeros, which no statistic notices.  Their loads are of
// one line, but their binary64 additions take as long as others: SUMS leaves them out, workgroup by workgroup.  3 x 32/8 heads of 648 rows, head_dim
// 128, FP16 P.V 57.3 -> 56.2 us, 2 x 24 of 4095 queries and 257 keys, 64, 42.3 -> 41.6.  Maxima are cheaper than the branches: FP8, no
// smoothing, 2 x 16 heads of 795 32.6 us without, 34.0 with them.)
template <int D, bool SUMS, class Fold>
__device__ __forceinline__ void stream_rows(const u16* base, int64_t stride, int n, int n0, int n1, Fold fold) {
  constexpr int RPP = 256 / (D / 8);
  auto batch = [&](auto unr) __attribute__((always_inline)) {
    constexpr int UNR = decltype(unr)::value;
    uint4 raw[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) raw[u] = *reinterpret_cast<const uint4*>(base + (int64_t)min(n + u * RPP, n1 - 1) * stride);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      if (SUMS && n0 + u * RPP >= n1) break;
      fold(n + u * RPP < n1 ? raw[u] : make_uint4(0, 0, 0, 0));
    }
    n0 += UNR * RPP;
    n += UNR * RPP;
  };
#pragma unroll 1
  while (n1 - n0 > 8 * RPP) batch(std::integral_constant<int, 16>());
  if (n1 - n0 > 4 * RPP) batch(std::integral_constant<int, 8>());
  else if (n0 < n1) batch(std::integral_constant<int, 4>());
}

template <int DT, int D, int PV, int NP>
__global__ void __launch_bounds__(256) prepass_small_kernel(QuantArgs qa, PrepVArgs va, int nk, int smooth, u16* km_out,
                                                            float* vscale_out) {
  constexpr int TPR = D / 8, RPP = 256 / TPR;
  const int h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, tr = tid / TPR, tc = tid % TPR;
  __shared__ __align__(16) uint8_t lds[prep_v_lds_bytes(D, PV) > colstat_lds_bytes(D) ? prep_v_lds_bytes(D, PV) : colstat_lds_bytes(D)];
  double(*red)[D] = reinterpret_cast<double(*)[D]>(lds);
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
        stream_rows<D, true>(qa.x + xbase + tc * 8, qa.x_sn, n0 + tr, n0, n1, [&](const uint4& raw) {   // (the additions in row order)
          const uint32_t* x2 = reinterpret_cast<const uint32_t*>(&raw);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float lo, hi;
            unpack2<DT>(x2[i], lo, hi);
            acc[2 * i] += (double)lo;
            acc[2 * i + 1] += (double)hi;
          }
        });
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
    quant_int8_rows<DT, D, NP, true>(qa, blockIdx.x, h, b, MeanInLds<DT, D>{smooth ? km_l : nullptr});   // (K: the multiplier is 1)
  } else {
    const int pidx = blockIdx.x - nk;
    if constexpr (PV == 1) {
      const int L = va.L;
      const int64_t vbase = (int64_t)b * va.v_sb + (int64_t)h * va.v_sh;
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; i++) acc[i] = 0.f;
      stream_rows<D, false>(va.v + vbase + tc * 8, va.v_sn, tr, 0, L, [&](const uint4& raw) {
        const uint32_t* x2 = reinterpret_cast<const uint32_t*>(&raw);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float lo, hi;
          unpack2<DT>(x2[i], lo, hi);
          acc[2 * i] = fmaxf(acc[2 * i], fabsf(lo));
          acc[2 * i + 1] = fmaxf(acc[2 * i + 1], fabsf(hi));
        }
      });
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
    prep_v_tile<DT, D, PV>(va, pidx, h, b, ScalesInMemory{vs_l}, reinterpret_cast<uint32_t*>(lds));
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

__device__ __forceinline__ void mask_pack_tile(const MaskPackArgs& a, const int tile, const int qt, const int plane, uint8_t* packed) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4), aligned(1)));
  __shared__ unsigned wave_seen[4];
  const uint8_t* mask = a.mask;
  const int64_t m_sb = a.m_sb, m_sh = a.m_sh, m_sm = a.m_sm, m_sn = a.m_sn;
  const MaskPlanes& p = a.p;
  const int Sq = a.Sq, Skv = a.Skv, tid = threadIdx.x;
  const int heads = p.ph ? (p.pb ? p.pb : p.planes) : 1;   // planes of one batch entry
  const int b = plane / heads, hd = plane - b * heads;
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
  const int64_t t = ((int64_t)plane * p.nqt + qt) * p.ntk + tile;
  reinterpret_cast<uint4*>(a.bits + t * kMaskTileBytes)[tid] = row;
  const unsigned long long any = __builtin_amdgcn_ballot_w64((row.x | row.y | row.z | row.w) != 0);
  if ((tid & 63) == 0) wave_seen[tid >> 6] = ((unsigned)any != 0 ? 1 : 0) | ((any >> 32) != 0 ? 2 : 0);
  __syncthreads();
  if (tid == 0) a.seen[t] = (uint8_t)(wave_seen[0] | wave_seen[1] << 2 | wave_seen[2] << 4 | wave_seen[3] << 6);
}

__global__ void __launch_bounds__(256) mask_pack_kernel(MaskPackArgs a) {
  __shared__ __align__(16) uint8_t packed[kMaskTileBytes];
  mask_pack_tile(a, blockIdx.x, blockIdx.y, blockIdx.z, packed);
}

// ---------------------------------------------------------------------------------------------
// Several pre-passes in one launch: a workgroup finds its job in the table of running workgroup counts and runs the code of that
// job's own kernel.  The launches of a call on a few thousand rows take 3 to 8 us each, most of it the start, the memory
// latency and the last workgroups of kernels too small to fill the chip, one after the other.
// ---------------------------------------------------------------------------------------------
enum FusedJob { kJobPlan, kJobKStat, kJobVStat, kJobKQuant, kJobQQuant, kJobVPanels, kJobMask, kJobs };
struct FusedTable {
  uint32_t end[kJobs];       // workgroups of the jobs up to this one
  uint32_t nx[kJobs], nh[kJobs];
  FastDiv div_x[kJobs], div_h[kJobs];   // workgroup of a job -> (x, head, batch)
  uint32_t heads_first;      // a bit per job: the heads are the inner index instead (nx and nh change places)
};
constexpr int kFusedPlanSeqs = 1024;
constexpr int fused_lds_bytes(int D, int PV) {
  const int a = prep_v_lds_bytes(D, PV) > colstat_lds_bytes(D) ? prep_v_lds_bytes(D, PV) : colstat_lds_bytes(D);
  return a > (int)sizeof(PlanLds<kFusedPlanSeqs>) ? a : (int)sizeof(PlanLds<kFusedPlanSeqs>);
}

// The jobs of the second launch alone (quantisers and panels, statistics combined on the way): fewer registers than with all of them.
template <int DT, int D, int PV, int NP>
__device__ __forceinline__ void fused_late_job(const FusedPrepass& f, const int job, const int x, const int h, const int b, uint32_t* lds, float* stat) {
  if (job == kJobKQuant) {
    if (f.k_quant.km_partial) quant_int8_rows<DT, D, NP, true>(f.k_quant, x, h, b, MeanFromPartials<DT, D>{f.k_quant, h, b, reinterpret_cast<u16*>(stat)});
    else quant_int8_rows<DT, D, NP, true>(f.k_quant, x, h, b, MeanInMemory<DT, D>{f.k_quant, h, b});
  } else if (job == kJobQQuant) {
    quant_int8_rows<DT, D, NP, false>(f.q_quant, x, h, b, MeanInLds<DT, D>{nullptr});
  } else {
    if (PV == 1 && f.v_panels.vs_partial) prep_v_tile<DT, D, PV>(f.v_panels, x, h, b, ScalesFromPartials<D>{f.v_panels, h, b, stat}, lds);
    else prep_v_tile<DT, D, PV>(f.v_panels, x, h, b, ScalesInMemory{f.v_panels.vscale + ((int64_t)b * f.v_panels.H + h) * D}, lds);
  }
}

template <int DT, int D, int PV, int NP, bool ALL>
__global__ void __launch_bounds__(256, ALL ? 3 : 4) fused_prepass_kernel(FusedPrepass f, FusedTable t) {
  __shared__ __align__(16) uint8_t lds[ALL ? fused_lds_bytes(D, PV) : prep_v_lds_bytes(D, PV)];
  __shared__ __align__(16) float stat[D];   // K mean or V scales of this workgroup's (batch, head)
  int job = 0;
  while (blockIdx.x >= t.end[job]) job++;
  const uint32_t i = blockIdx.x - (job ? t.end[job - 1] : 0), y = fastdiv(i, t.div_x[job]);
  const int b = fastdiv(y, t.div_h[job]), inner = i - y * t.nx[job], outer = y - b * t.nh[job];
  const bool hf = t.heads_first >> job & 1;
  const int x = hf ? outer : inner, h = hf ? inner : outer;
  if constexpr (ALL) {
    if (job == kJobPlan) { varlen_plan<256, kFusedPlanSeqs>(f.plan, *reinterpret_cast<PlanLds<kFusedPlanSeqs>*>(lds)); return; }
    if (job == kJobKStat) { colstat_chunk<DT, D, 0>(f.k_stat, x, h, b, lds); return; }
    if (PV == 1 && job == kJobVStat) { colstat_chunk<DT, D, 1>(f.v_stat, x, h, b, lds); return; }
    if (job == kJobMask) { mask_pack_tile(f.mask, x, h, b, lds); return; }
  }
  fused_late_job<DT, D, PV, NP>(f, job, x, h, b, reinterpret_cast<uint32_t*>(lds), stat);
}

// ---------------------------------------------------------------------------------------------
// Host-side launchers (called from the C ABI in sage_api.hip).
// ---------------------------------------------------------------------------------------------
// Where the heads of a row lie next to each other (packed and [B, L, H, D] tensors) the head can be the fastest grid index, so that whole
// rows are on their way at a time; with the rows of one head first, a workgroup and its neighbours read 128 or 256 bytes out of every
// few kilobytes.  (The y axis of a grid is limited to 65535.)
static bool heads_first(int64_t head_stride, int64_t row_stride, int64_t chunks) { return head_stride < row_stride && chunks <= 65535; }
// Statistics (512 rows per workgroup) and V panels (128), in packed batches: up to 4096 rows a sequence, heads first (most workgroups of a grid
// sized for the longest sequence find nothing to do), longer ones rows first.  Whole causal calls, heads first / rows first: 64 of 256..4096, 24
// heads of 128, FP8 2268 / 2379 us, of 64 1421 / 1472; 96 of 16..1024, 8 heads of 128 235 / 244; 16 of 512..32768, 24 heads of 64 17224 / 17117.
// Otherwise heads first where rows are a multiple of 4 KiB apart (a head's rows alone then crowd into a few memory channels), and
//   statistics at head_dim 128, and at 64 as long as a head is four chunks or all of them are 256.  Whole calls, 40 query rows: 4 x 32 heads of 8000
//   rows, 128, FP8 313 / 322, 24 of 1559 42.6 / 43.2; head_dim 64: 4 x 24 of 1559 48.0 / 48.9, 2 x 4 of 5696, FP8 69.1 / 70.1, 24 of 9000 110.2 /
//   109.3, 4 x 40 of 8000 231 / 224;
//   up to 1024 panels (which reader of them gains has not been isolated).  Whole calls, FP16: 2 x 8 heads of 4000 rows,
//   128 (512 panels) 81.8 / 85.6, 2 x 12, 64 (768) 65.2 / 68.5, 2 x 20, 128 (1280) 106.4 / 106.2, 4 x 40 of 1559, 64 (2080) 64.1 / 62.7; FP8: 4 of
//   9000, 128 (284) 109.5 / 110.5, 8 x 12 of 886 (672) 65.1 / 66.0, 12 of 9000 (852) 126.5 / 125.8, 4 x 12 of 2471, 64 (960) 45.2 / 46.1.
// Panels alone, 100 M elements: 16 heads of 128 (4 KiB) 71.6 / 77.7, 32 (8 KiB) 71.1 / 73.7, 24 (6 KiB) 73.2 / 67.7; 32 of 64 (4 KiB) 75.8 / 78.6,
// 40 (5 KiB) 78.9 / 68.0.
constexpr int64_t kFewStats = 256, kFewPanels = 1024;
static bool heads_first_streaming(int64_t head_stride, int64_t row_stride, int64_t chunks, bool packed, int max_rows, bool otherwise) {
  return heads_first(head_stride, row_stride, chunks) && (packed ? max_rows <= 4096 : otherwise || row_stride * 2 % 4096 == 0);
}
static bool heads_first(const ColStatArgs& a, int64_t chunks) {
  return heads_first_streaming(a.x_sh, a.x_sn, chunks, a.cu_seqlens, a.L, a.D == 128 || a.L <= 4 * kChunkRows || (int64_t)a.B * a.H * a.nchunk <= kFewStats);
}
static bool heads_first(const PrepVArgs& a, int64_t chunks) {
  const int64_t panels = (int64_t)a.B * a.H * ((a.L + kPanelRows - 1) / kPanelRows);
  return heads_first_streaming(a.v_sh, a.v_sn, chunks, a.cu_seqlens, a.L, panels <= kFewPanels);
}
// The quantiser.  Packed batches: heads first where the grid's row chunks are even in number: rows first, the same chunks of all heads and
// sequences then go to the same XCDs, and those with the last ones of a grid sized for the longest sequence run dry.  Whole causal calls, heads
// first / rows first: 96 of 16..1024, 24 heads of 64 441 / 467 us, of 128 624 / 660; 60 of 64..2000 554 / 584 and 835 / 879; 64 of 256..4096 1430 / 1485;
// an odd number: 23 of 52..2880 391 / 385 and 581 / 581.
// Otherwise in small tensors, in the largest, and where rows of heads of 128 are a multiple of 4 KiB apart.  Whole calls, 40
// query rows: 8 heads of 1500 rows, 64, 34.5 / 36.6, 12 of 1500 33.4 / 34.1, 32 of 1500, 128 (6 M elements) 40.8 / 41.0; 4 x 24 of 2471, 128 (30 M)
// 101.9 / 100.9, 4 x 32 of 8000, 64 (66 M) 195 / 189, 2 x 40 of 16000, 64 (82 M) 276 / 263, 24 of 32760, 128 (101 M) 472 / 468; 2 x 16 of 16000, 128
// (4 KiB, 66 M) 267.7 / 269.6, 2 x 32 of 16384 383 / 388; causal, as many query rows, 16 of 4096, 128, 98.2 / 101.8, 2 x 32 of 2048 100.5 / 101.3.  Alone, 160 M elements: 24 heads of 64 117 / 126, 12 of 128 91 / 96, 32 of 128 90 / 113;
// 8 of 128 (2 KiB) 90.5 / 88.6.
static bool heads_first(const QuantArgs& a, int64_t chunks) {
  if (!heads_first(a.x_sh, a.x_sn, chunks)) return false;
  const int64_t mega = 1 << 20, elements = (int64_t)a.B * a.H * a.L * a.D, row_bytes = a.x_sn * 2;
  if (a.cu_seqlens) return chunks % 2 == 0;
  return elements <= 8 * mega || (a.D == 128 && row_bytes % 4096 == 0) || (elements >= 128 * mega && row_bytes > 2048);
}

hipError_t launch_quant_int8(const QuantArgs& args, int dtype, int max_rows, hipStream_t st) {
  QuantArgs a = args;
  const int rows = quant_rows(a.D, a.blk);
  const uint32_t chunks = (max_rows + rows - 1) / rows;
  a.heads_first = heads_first(a, chunks);
  const dim3 grid = a.heads_first ? dim3(a.H, chunks, a.B) : dim3(chunks, a.H, a.B), block(256);
#define SAGE_QUANT(DT, DD, NP) (a.km_partial ? quant_int8_kernel<DT, DD, NP, true><<<grid, block, 0, st>>>(a) : quant_int8_kernel<DT, DD, NP><<<grid, block, 0, st>>>(a))
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

hipError_t launch_mask_pack(const MaskPackArgs& a, hipStream_t st) {
  mask_pack_kernel<<<dim3(a.p.ntk, a.p.nqt, a.p.planes), dim3(256), 0, st>>>(a);
  return hipGetLastError();
}

bool fused_quant_together(int D, int blk_a, int blk_b) {
  const int lo = blk_a < blk_b ? blk_a : blk_b, hi = blk_a < blk_b ? blk_b : blk_a;
  return quant_passes(D, hi) * quant_wave_rows(D) <= lo;   // the wider one's wavefronts still own whole blocks of the other
}

// (x, head, batch) extents of the jobs; zero where a job is not asked for
static void fused_extents(const FusedPrepass& f, int np_blk, int64_t (&e)[kJobs][3]) {
  memset(e, 0, sizeof(e));
  auto set = [&](int job, int64_t x, int64_t h, int64_t b) { e[job][0] = x; e[job][1] = h; e[job][2] = b; };
  if (f.plan.plan) set(kJobPlan, 1, 1, 1);
  if (f.k_stat.partial) set(kJobKStat, f.k_stat.nchunk, f.k_stat.H, f.k_stat.B);
  if (f.v_stat.partial) set(kJobVStat, f.v_stat.nchunk, f.v_stat.H, f.v_stat.B);
  auto quant = [&](int job, const QuantArgs& a) {
    const int rows = quant_rows(a.D, np_blk);
    if (a.out) set(job, (a.L + rows - 1) / rows, a.H, a.B);
  };
  quant(kJobKQuant, f.k_quant);
  quant(kJobQQuant, f.q_quant);
  if (f.v_panels.panels) set(kJobVPanels, (f.v_panels.L + kPanelRows - 1) / kPanelRows, f.v_panels.H, f.v_panels.B);
  if (f.mask.bits) set(kJobMask, f.mask.p.ntk, f.mask.p.nqt, f.mask.p.planes);
}
static int fused_block(const FusedPrepass& f) {   // the scale block that sets the rows of a quantiser workgroup
  const int k = f.k_quant.out ? f.k_quant.blk : 0, q = f.q_quant.out ? f.q_quant.blk : 0;
  return k > q ? k : q;
}

constexpr int64_t kFusedMaxWorkgroups = (int64_t)1 << 23;   // one grid axis holds 2^31 threads

template <int MODE>
static hipError_t launch_colstat(const ColStatArgs& a, int dtype, hipStream_t st);

// A job in a launch of its own.
static hipError_t launch_job(const FusedPrepass& f, int job, int dtype, int pv, hipStream_t st) {
  switch (job) {
    case kJobPlan: return launch_varlen_plan(f.plan.cu_q, f.plan.cu_k, f.plan.nseq, f.plan.total_q, f.plan.blkq, f.plan.blkk, f.plan.bm, f.plan.bn, f.plan.causal, f.plan.plan, st);
    case kJobKStat: return launch_colstat<0>(f.k_stat, dtype, st);
    case kJobVStat: return launch_colstat<1>(f.v_stat, dtype, st);
    case kJobKQuant: return launch_quant_int8(f.k_quant, dtype, f.k_quant.L, st);
    case kJobQQuant: return launch_quant_int8(f.q_quant, dtype, f.q_quant.L, st);
    case kJobVPanels: return launch_prep_v(f.v_panels, dtype, pv, (f.v_panels.L + kPanelRows - 1) / kPanelRows, st);
    default: return launch_mask_pack(f.mask, st);
  }
}

// Up to how many workgroups the jobs of a launch share it: past that each fills the chip by itself, and its own kernel, with fewer
// registers and less LDS than the shared one, is the faster.  With a plan the statistics share its launch whatever their size: its one
// workgroup starts first and works beside theirs, and a launch of its own costs more than they gain.  Packed, head_dim 128, 8 KV heads, a
// query row per sequence, shared / apart in us: 16 sequences of 512..32768 keys (15873 workgroups) FP8 841 / 852, FP16 943 / 950; 64 of
// 512..4096 FP8 380 / 385; 200 of 100..1500 442 / 452; whole causal calls, 32/8 heads, of 256 sequences 1497 / 1493 and FP8 1308 / 1316, of
// 4096 4551 / 4571 and FP8 4406 / 4364 (the plan has 256 lanes here and 1024 apart), of 32000 34.1 / 34.3 ms.
// Without one, whole calls in bf16, 40 query rows, us, before these launches / each job by itself / early, late or both jobs sharing: 8 heads of 4096 keys, FP8 P.V
// (512 early and 768 late workgroups) 71.9 / 65.4 / 63.2, 63.7, 61.6; 32 heads of 4096, FP8 (1024 early, 3072 late) 87.9 / 82.0 / 81.8,
// 83.0, 82.8; 4 x 32 of 4096, FP16 (5120 early) 181.8 / 174.3 / 177.1 early; packed, causal, 16 sequences of 100..600, 32/8 heads, FP16
// (1920 late) 90.2 / 84.5 / 81.0, 82.9, 79.3; 96 of 16..1024 (18432 late) 571 / 547 / 544, 565, 563.
constexpr int64_t kMergeEarly = 2048, kMergeLate = 8192;

hipError_t launch_fused_prepass(const FusedPrepass& f, int dtype, int D, int pv, hipStream_t st) {
  int64_t e[kJobs][3], n = 0;
  const int blk = fused_block(f);
  fused_extents(f, blk, e);
  FusedTable t;
  const bool inner_heads[kJobs] = {false, heads_first(f.k_stat, 0), heads_first(f.v_stat, 0), heads_first(f.k_quant, e[kJobKQuant][0]),
                                   heads_first(f.q_quant, e[kJobQQuant][0]), heads_first(f.v_panels, 0), false};
  t.heads_first = 0;
  for (int j = 0; j < kJobs; j++) {
    if (e[j][1] > 65535 || e[j][2] > 65535) return hipErrorInvalidConfiguration;   // (what the jobs' own grids take)
    n += e[j][0] * e[j][1] * e[j][2];
    t.end[j] = (uint32_t)(n < kFusedMaxWorkgroups ? n : kFusedMaxWorkgroups);
    const bool hf = inner_heads[j];
    t.heads_first |= (uint32_t)hf << j;
    t.nx[j] = e[j][hf] ? (uint32_t)e[j][hf] : 1;
    t.nh[j] = e[j][!hf] ? (uint32_t)e[j][!hf] : 1;
    t.div_x[j] = make_fastdiv(t.nx[j]);
    t.div_h[j] = make_fastdiv(t.nh[j]);
  }
  if (n == 0) return hipSuccess;
  int jobs = 0;
  for (auto& j : e) jobs += j[0] * j[1] * j[2] > 0;
  const bool all = e[kJobPlan][0] || e[kJobKStat][0] || e[kJobVStat][0] || e[kJobMask][0];
  if (jobs == 1 || n > kFusedMaxWorkgroups || (!f.plan.plan && n > (all ? kMergeEarly : kMergeLate))) {
    for (int j = 0; j < kJobs; j++)
      if (e[j][0] * e[j][1] * e[j][2] > 0)
        if (hipError_t err = launch_job(f, j, dtype, pv, st)) return err;
    return hipSuccess;
  }
  const dim3 grid((uint32_t)n), block(256);
  const int np = blk ? quant_passes(D, blk) : D == 128 ? 2 : 1;
#define SAGE_FUSED(DT, DD, PVV, NP) (all ? fused_prepass_kernel<DT, DD, PVV, NP, true><<<grid, block, 0, st>>>(f, t) : fused_prepass_kernel<DT, DD, PVV, NP, false><<<grid, block, 0, st>>>(f, t))
#define SAGE_FUSED_D(DT, PVV) \
  do { \
    if (D == 64) { if (np == 1) SAGE_FUSED(DT, 64, PVV, 1); else SAGE_FUSED(DT, 64, PVV, 2); } \
    else { if (np == 2) SAGE_FUSED(DT, 128, PVV, 2); else SAGE_FUSED(DT, 128, PVV, 4); } \
  } while (0)
  if (dtype == 0) { if (pv) SAGE_FUSED_D(0, 1); else SAGE_FUSED_D(0, 0); }
  else { if (pv) SAGE_FUSED_D(1, 1); else SAGE_FUSED_D(1, 0); }
#undef SAGE_FUSED_D
#undef SAGE_FUSED
  return hipGetLastError();
}

int colstat_chunks(int L) { return (L + kChunkRows - 1) / kChunkRows; }

template <int MODE>
static hipError_t launch_colstat(const ColStatArgs& args, int dtype, hipStream_t st) {
  ColStatArgs a = args;
  a.heads_first = heads_first(a, a.nchunk);
  const dim3 grid = a.heads_first ? dim3(a.H, a.nchunk, a.B) : dim3(a.nchunk, a.H, a.B), block(256);
  if (dtype == 0 && a.D == 64) colstat_partial_kernel<0, 64, MODE><<<grid, block, 0, st>>>(a);
  else if (dtype == 0 && a.D == 128) colstat_partial_kernel<0, 128, MODE><<<grid, block, 0, st>>>(a);
  else if (dtype == 1 && a.D == 64) colstat_partial_kernel<1, 64, MODE><<<grid, block, 0, st>>>(a);
  else colstat_partial_kernel<1, 128, MODE><<<grid, block, 0, st>>>(a);
  return hipGetLastError();
}

hipError_t launch_k_mean(const ColStatArgs& a, int dtype, void* km, hipStream_t st) {
  if (a.nchunk == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  hipError_t e = launch_colstat<0>(a, dtype, st);
  return e != hipSuccess ? e : launch_k_mean_finalize(a, dtype, km, st);
}
hipError_t launch_k_mean_finalize(const ColStatArgs& a, int dtype, void* km, hipStream_t st) {
  dim3 grid(a.H, a.B), block(a.D);
  if (dtype == 0) kmean_finalize_kernel<0><<<grid, block, 0, st>>>((const double*)a.partial, (u16*)km, a.H, a.L, a.D, a.nchunk, a.cu_seqlens);
  else kmean_finalize_kernel<1><<<grid, block, 0, st>>>((const double*)a.partial, (u16*)km, a.H, a.L, a.D, a.nchunk, a.cu_seqlens);
  return hipGetLastError();
}

hipError_t launch_v_scale(const ColStatArgs& a, int dtype, float* vscale, hipStream_t st) {
  if (a.nchunk == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  hipError_t e = launch_colstat<1>(a, dtype, st);
  return e != hipSuccess ? e : launch_v_scale_finalize(a, vscale, st);
}
hipError_t launch_v_scale_finalize(const ColStatArgs& a, float* vscale, hipStream_t st) {
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

hipError_t launch_prep_v(const PrepVArgs& args, int dtype, int pv, int max_panels, hipStream_t st) {
  PrepVArgs a = args;
  if (max_panels == 0 || a.B == 0 || a.H == 0) return hipSuccess;
  a.heads_first = heads_first(a, max_panels);
  const dim3 grid = a.heads_first ? dim3(a.H, max_panels, a.B) : dim3(max_panels, a.H, a.B), block(256);
#define SAGE_PREPV(DT, DD, PVV) (PVV && a.vs_partial ? prep_v_kernel<DT, DD, PVV, PVV == 1><<<grid, block, 0, st>>>(a) : prep_v_kernel<DT, DD, PVV><<<grid, block, 0, st>>>(a))
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
