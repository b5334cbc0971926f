// vx_codec.h -- the codec decoder (semantic + acoustic codes -> 24 kHz
// waveform) on MFMA: codecDecode, src/engine.ts:1402-1713, with the codec
// shaders of src/shaders.ts:817-1110, 1432-1868.
//
// Every projection and convolution is one f16 x f16 -> f32 GEMM on the
// matrix cores, the hand-written kernels of vx_gemm.h shared with the
// prefill: the f16 weights times the activations in hi/lo f16 form, so
// products keep f32 accuracy. A GEMM may leave its sum in up to 8 K-slice
// partials; the epilogue kernels below (template parameter NS) add them in
// slice order, so every result is bit-reproducible.
//   - the causal convs become GEMMs whose column t holds
//     x[t - (k_size-1) + kk][ci] at k = kk * c_in + ci, with the weights
//     reordered to match once after loading; their weight norm g/||w|| is
//     one scale per output row, applied in the epilogue.  For the output conv
//     (c_in = 1024) column t is the 7 consecutive packed rows t - 6 .. t, so
//     each row is packed once and the columns overlap (packing one copy per
//     tap took 18 us of a 250-frame decode and 57 MB); the input conv's 292
//     channels are no multiple of 16 bytes and are packed per tap;
//   - the stride-2 transposed conv (kernel 4) gives output step 2 tau + r
//     from input steps tau (tap r) and tau - 1 (tap r + 2): one GEMM of
//     2048 rows (both parities) over the packed rows x[tau - 1], x[tau],
//     scaled by the per-input-channel weight norm;
//   - the input conv's B is gathered straight from the codes (vqLookup,
//     fsqDequant and concatCodecInput fused into the packing).
// Tokens are processed in column chunks of at most CX_MAXT; a chunk's B
// holds nc = 2 * nt columns (nt = gm_cols(tokens), hi then lo),
// each column's K halves contiguous; the GEMM output C is [nc][M].
#pragma once
#include "vx_prefill.h"

namespace vx {

// codec dimensions (src/types.ts:98-122)
constexpr int CD = 1024, CHID = 4096, CNH = 8, CHDIM = 128;
constexpr int CSEM = 8192, CSEMD = 256, CIN = CSEMD + NAC;  // 292 input channels
constexpr int CPATCH = 240, CPATCH_ROWS = 256;  // output conv rows, padded to the GEMM tile
constexpr int CK_IN = 3, CK_OUT = 7, CK_UP = 4;
constexpr int CKIN = 896;            // CIN * CK_IN = 876, rounded up to 32
constexpr int CKOUT = CD * CK_OUT;   // 7168
constexpr int CKUP = 2 * CD;         // input steps tau and tau - 1
constexpr int CX_STAGES = 4, CX_LPS = 2;
constexpr int CX_FRAME_SAMPLES = 8 * CPATCH;  // 1920 samples = 80 ms at 24 kHz
constexpr int CX_MAXT = 1024;                 // tokens per GEMM chunk
constexpr int CX_NC = 2 * CX_MAXT;
constexpr size_t CX_CCAP = (size_t)CX_NC * 2 * CHID;  // GEMM output floats
constexpr float CX_NORM_EPS = 0.01f, CX_QK_EPS = 1e-6f;
static_assert(CKIN % 32 == 0 && CKIN >= CIN * CK_IN, "input conv k padding");

// output (token t, row m) of a chunk's GEMM: the sum of its NS K-slice
// blocks [nc / 2][ldc] (vx_gemm.h), in order
template <int NS>
__device__ __forceinline__ float cx_val(const float *C, int ldc, int nc, int t, int m) {
  float v[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) v[s] = C[((size_t)s * (nc >> 1) + t) * ldc + m];
  float y = v[0];
#pragma unroll
  for (int s = 1; s < NS; s++) y += v[s];
  return y;
}

// outputs m .. m + 7 (m % 8 == 0) of token t, the same in-order sums as
// cx_val, from two 16-byte loads per K-slice block
template <int NS>
__device__ __forceinline__ void cx_val8(const float *C, int ldc, int nc, int t, int m, float (&y)[8]) {
  f32x4 a[NS], b[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const float *p = C + ((size_t)s * (nc >> 1) + t) * ldc + m;
    a[s] = *(const f32x4 *)p;
    b[s] = *(const f32x4 *)(p + 4);
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    y[e] = a[0][e];
    y[4 + e] = b[0][e];
  }
#pragma unroll
  for (int s = 1; s < NS; s++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      y[e] += a[s][e];
      y[4 + e] += b[s][e];
    }
}

// 8 consecutive f32 / f16 values from 16-byte aligned addresses
__device__ __forceinline__ void cx_load8(const float *x, float (&y)[8]) {
  const f32x4 a = *(const f32x4 *)x, b = *(const f32x4 *)(x + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    y[e] = a[e];
    y[4 + e] = b[e];
  }
}
__device__ __forceinline__ void cx_load8h(const uint16_t *g, float (&y)[8]) {
  const h8 w = *(const h8 *)g;
#pragma unroll
  for (int e = 0; e < 8; e++) y[e] = (float)w[e];
}

// k group kb (8 halves) of columns t (hi) and nt + t (lo); kg = K / 8
__device__ __forceinline__ void cx_put(h8 *B, int nc, int kg, int kb, int t, const float (&y)[8]) {
  h8 hi, lo;
  split_n<8>(y, hi, lo);
  B[(size_t)t * kg + kb] = hi;
  B[(size_t)((nc >> 1) + t) * kg + kb] = lo;
}

// ------------------------------------------------------------- packing
// B from rows t0 + t of X [*][K], RMS-normalised with gains g
// (batchedRmsNorm, src/shaders.ts:1646-1692).  Grid: nt blocks of 256.
__global__ __launch_bounds__(256) void cx_pack_kernel(const float *X, int K, int t0, int n, int nc,
                                                      const uint16_t *g, float eps, h8 *B) {
  const int t = blockIdx.x, tid = threadIdx.x;
  const bool live = t < n;
  const float *x = X + (size_t)(t0 + t) * K;
  float r = 1.0f;
  if (live) {
    __shared__ float red[4];
    float s = 0.f;
    for (int k = tid; k < K; k += 256) s = fmaf(x[k], x[k], s);
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    r = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)K + eps);
  }
  for (int kb = tid; kb < K / 8; kb += 256) {
    float y[8];
    if (live) {
      float gv[8];
      cx_load8(x + kb * 8, y);
      cx_load8h(g + kb * 8, gv);
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = y[e] * r * gv[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = 0.f;
    }
    cx_put(B, nc, K / 8, kb, t, y);
  }
}

// input channel ci of frame tau: the normalised semantic codebook row of its
// semantic code (vqLookup, src/shaders.ts:817-845; rows past the 8192-entry
// table read as zero), then the 36 dequantised acoustic values
// (fsqDequant, src/shaders.ts:891-914: u32 code - 2, * 2 / (levels - 1) - 1)
__device__ __forceinline__ float cx_feature(const uint16_t *cbn, const uint32_t *sem,
                                            const uint32_t *ac, int levels, int tau, int ci) {
  if (ci < CSEMD) {
    const uint32_t c = sem[tau];
    return c < (uint32_t)CSEM ? h2f(cbn[(size_t)c * CSEMD + ci]) : 0.f;
  }
  const uint32_t c = ac[(size_t)tau * NAC + (ci - CSEMD)] - 2u;
  return (float)c * 2.0f / (float)(levels - 1) - 1.0f;
}

// im2col B of the input conv (k = 3) straight from the codes.
// Grid: nt blocks of 128.
__global__ __launch_bounds__(128) void cx_pack_in_kernel(const uint16_t *cbn, const uint32_t *sem,
                                                         const uint32_t *ac, int levels, int t0,
                                                         int n, int nc, h8 *B) {
  const int t = blockIdx.x, tau = t0 + t;
  for (int kb = threadIdx.x; kb < CKIN / 8; kb += blockDim.x) {
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int k = kb * 8 + e, kk = k / CIN, ci = k - kk * CIN;
      const int src = tau - (CK_IN - 1) + kk;
      y[e] = (t < n && k < CIN * CK_IN && src >= 0) ? cx_feature(cbn, sem, ac, levels, src, ci) : 0.f;
    }
    cx_put(B, nc, CKIN / 8, kb, t, y);
  }
}

// Packed rows of the convs over CD channels: row i of B (hi; lo blo halves
// further) is x[t0 - before + i], times scale[ci] if given; rows before the
// first step and rows past step t0 + n - 1 are zero.  Grid: before + nt
// blocks of 128.
__global__ __launch_bounds__(128) void cx_pack_rows_kernel(const float *X, const float *scale, int before, int t0,
                                                           int n, size_t blo, h8 *B) {
  const int i = blockIdx.x, kb = threadIdx.x, src = t0 - before + i;
  float y[8];
  if (src >= 0 && src < t0 + n) {
    cx_load8(X + (size_t)src * CD + kb * 8, y);
    if (scale) {
      float sc[8];
      cx_load8(scale + kb * 8, sc);
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = sc[e] * y[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  h8 hi, lo;
  split_n<8>(y, hi, lo);
  B[(size_t)i * (CD / 8) + kb] = hi;
  B[blo / 8 + (size_t)i * (CD / 8) + kb] = lo;
}
static_assert(CD == 128 * 8, "one 8-value group per thread");

// ----------------------------------------------------------- epilogues
// out[(t0 + t) * ldo + m] = rs[m] * y (conv weight norm g / ||w|| per
// output channel), m < mv.  Grid: (n, ceil(mv / 256)).
template <int NS>
__global__ void cx_scale_rows_epi_kernel(const float *C, int ldc, int nc, int t0, const float *rs,
                                         int mv, float *out, int ldo) {
  const int t = blockIdx.x, m = blockIdx.y * blockDim.x + threadIdx.x;
  if (m < mv) out[(size_t)(t0 + t) * ldo + m] = rs[m] * cx_val<NS>(C, ldc, nc, t, m);
}

// transposed conv output: step 2 (t0 + t) + r, channel co from row r * CD + co.
// Grid: (n, 2 * CD / 256).
template <int NS>
__global__ void cx_up_epi_kernel(const float *C, int nc, int t0, float *out) {
  const int t = blockIdx.x, m = blockIdx.y * blockDim.x + threadIdx.x;
  const int r = m / CD, co = m - r * CD;
  out[(size_t)(2 * (t0 + t) + r) * CD + co] = cx_val<NS>(C, 2 * CD, nc, t, m);
}

// layer scale + residual (batchedLayerScale, src/shaders.ts:1755-1781),
// X = y * scale + X, and, with PACK, the next GEMM's B from the RMS-normalised
// row (batchedRmsNorm, src/shaders.ts:1646-1692; zero for t >= n).  The sum
// of squares needs the whole row, which the block holds: a pack kernel of its
// own read X again (3.5-5.7 us and a launch per GEMM it fed).
// Grid: nt blocks (n without PACK) of 128, one 8-value group per thread.
template <bool PACK, int NS>
__global__ __launch_bounds__(128) void cx_resid_pack_kernel(const float *C, int nc, int t0, int n,
                                                            const uint16_t *scale, float *X, const uint16_t *g,
                                                            float eps, h8 *B) {
  const int t = blockIdx.x, kb = threadIdx.x;
  float y[8];
  if (t < n) {
    float *x = X + (size_t)(t0 + t) * CD + kb * 8;
    float xv[8], sc[8];
    cx_load8(x, xv);
    cx_load8h(scale + kb * 8, sc);
    cx_val8<NS>(C, CD, nc, t, kb * 8, y);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = y[e] * sc[e] + xv[e];
    *(f32x4 *)x = f32x4{y[0], y[1], y[2], y[3]};
    *(f32x4 *)(x + 4) = f32x4{y[4], y[5], y[6], y[7]};
  }
  if (!PACK) return;
  if (t < n) {
    __shared__ float red[2];
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) ss = fmaf(y[e], y[e], ss);
    ss = wave_sum(ss);
    if ((kb & 63) == 0) red[kb >> 6] = ss;
    __syncthreads();
    const float r = 1.0f / sqrtf((red[0] + red[1]) / (float)CD + eps);
    float gv[8];
    cx_load8h(g + kb * 8, gv);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = y[e] * r * gv[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  cx_put(B, nc, CD / 8, kb, t, y);
}

// The same residual at the end of a stage, and the next conv's packed rows
// (cx_pack_rows_kernel) from the row while the block holds it: row before + t
// of B is X[t], times conv_scale if given; the rows before the first step and
// past the last are zero.  For a stage of one chunk.  Grid: before + nt blocks
// of 128.
template <int NS>
__global__ __launch_bounds__(128) void cx_resid_rows_kernel(const float *C, int nc, int n, const uint16_t *scale,
                                                            float *X, const float *conv_scale, int before, size_t blo,
                                                            h8 *B) {
  const int t = (int)blockIdx.x - before, kb = threadIdx.x;
  float y[8];
  if (t >= 0 && t < n) {
    float *x = X + (size_t)t * CD + kb * 8;
    float xv[8], sc[8];
    cx_load8(x, xv);
    cx_load8h(scale + kb * 8, sc);
    cx_val8<NS>(C, CD, nc, t, kb * 8, y);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = y[e] * sc[e] + xv[e];
    *(f32x4 *)x = f32x4{y[0], y[1], y[2], y[3]};
    *(f32x4 *)(x + 4) = f32x4{y[4], y[5], y[6], y[7]};
    if (conv_scale) {
      cx_load8(conv_scale + kb * 8, sc);
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = sc[e] * y[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  h8 hi, lo;
  split_n<8>(y, hi, lo);
  B[(size_t)blockIdx.x * (CD / 8) + kb] = hi;
  B[blo / 8 + (size_t)blockIdx.x * (CD / 8) + kb] = lo;
}

// A conv's output rows, and the next stage's first B from each while the block
// holds it (cx_pack_kernel): UP, the transposed conv: step to = 2 t + r is rows
// r CD .. of column t; else the input conv, scaled per row.  n, nc: the
// output's steps and columns; nci: the conv chunk's columns.  For outputs of
// one chunk.  Grid: nc / 2 blocks of 128.
template <bool UP, int NS>
__global__ __launch_bounds__(128) void cx_conv_pack_kernel(const float *C, int nci, const float *rs, int n, int nc,
                                                           float *X, const uint16_t *g, float eps, h8 *B) {
  const int to = blockIdx.x, kb = threadIdx.x;
  float y[8];
  if (to < n) {
    __shared__ float red[2];
    const int t = UP ? to >> 1 : to, m = (UP ? (to & 1) * CD : 0) + kb * 8;
    cx_val8<NS>(C, UP ? 2 * CD : CD, nci, t, m, y);
    if (!UP) {
      float sc[8];
      cx_load8(rs + kb * 8, sc);
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = sc[e] * y[e];
    }
    float *x = X + (size_t)to * CD + kb * 8;
    *(f32x4 *)x = f32x4{y[0], y[1], y[2], y[3]};
    *(f32x4 *)(x + 4) = f32x4{y[4], y[5], y[6], y[7]};
    float ss = 0.f, gv[8];
#pragma unroll
    for (int e = 0; e < 8; e++) ss = fmaf(y[e], y[e], ss);
    ss = wave_sum(ss);
    if ((kb & 63) == 0) red[kb >> 6] = ss;
    __syncthreads();
    const float r = 1.0f / sqrtf((red[0] + red[1]) / (float)CD + eps);
    cx_load8h(g + kb * 8, gv);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = y[e] * r * gv[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  cx_put(B, nc, CD / 8, kb, to, y);
}

// SwiGLU of the stacked gate/up projection (batchedSwiGLU,
// src/shaders.ts:1697-1716), written as the packed B of the down projection
// (k = hidden unit).  Grid: (nt, CHID / 8 / 256) of 256; columns t >= n are 0.
template <int NS>
__global__ __launch_bounds__(256) void cx_swiglu_epi_kernel(const float *C, int nc, int n, h8 *B) {
  const int t = blockIdx.x, kb = blockIdx.y * 256 + threadIdx.x;
  float y[8];
  if (t < n) {
    float g[8], u[8];
    cx_val8<NS>(C, 2 * CHID, nc, t, kb * 8, g);
    cx_val8<NS>(C, 2 * CHID, nc, t, CHID + kb * 8, u);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = g[e] / (1.0f + expf(-g[e])) * u[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  cx_put(B, nc, CHID / 8, kb, t, y);
}

// ----------------------------------------------------------- attention
// From the stacked q, k, v projection to the O projection's B in one kernel:
// q and k RMS-normalised per head (qkNorm, src/shaders.ts:1787-1830: weight
// [CNH * CHDIM] read at h * CHDIM), then windowed causal attention with ALiBi
// biases (alibiAttnScore, codecSoftmax, codecAttnValue, src/shaders.ts:
// 1432-1585): keys ki in [max(0, qi - W + 1), qi], score q.k / sqrt(128) -
// 2^(-8(h+1)/8) (qi - ki), W <= 16.
// Block = (CXA_T query tokens, head), one wave per query.  The keys of the block's
// tokens, CXA_T + W - 1 rows at most, are summed over the K slices, normalised
// and held in LDS (recomputed by the next block: at most 2x of an L2-resident
// read, where q, k and v written and read again, one wave per query reading W
// rows each, took 47.7 + 18 us a 2000-token layer, this 2 x 11.1; with four
// waves a block, eight rows and four queries each in turn, it took 2 x 19).  A wave
// stages two rows and takes one query: lane 4 j + p scores key k0 + j over the 16-byte
// chunks 4 i + p of the row, the window's max and sum are 4 lane steps each, and
// lane l sums dims 2 l, 2 l + 1 of P.V.  LDS rows are 144 floats apart, so
// the 16 lanes of one read phase (4 keys x 4 chunks) touch distinct banks.
// Keys before the chunk (t < t0) come from the previous chunk's `halo_in`
// [CX_HALO][2][CD], normalised k and v; a chunk that has a successor leaves
// its last CX_HALO rows in halo_out.
// Grid: (nt / CXA_T, CNH) of 64 CXA_WAVES; B columns t >= n are zero.
constexpr int CX_MAXW = 16, CX_HALO = CX_MAXW - 1;
constexpr int CXA_T = 16, CXA_WAVES = CXA_T, CXA_ROWS = CXA_T + CX_HALO, CXA_LD = 144;
static_assert(CXA_ROWS <= 2 * CXA_WAVES, "two rows per wave");
template <int NS>
__global__ __launch_bounds__(64 * CXA_WAVES) void cx_attn_kernel(const float *C, int nc, int t0, int n, int W,
                                                      const uint16_t *qn, const uint16_t *kn, const float *halo_in,
                                                      float *halo_out, h8 *B) {
  __shared__ __attribute__((aligned(16))) float ks[CXA_ROWS * CXA_LD], vs[CXA_ROWS * CXA_LD], qs[CXA_T * CXA_LD];
  const int tb = blockIdx.x * CXA_T, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, d = 2 * lane;
  const int nt = nc >> 1;
  const int base = tb - (W - 1);  // token of K/V row 0, within the chunk (negative: the chunk before)
  // q.k / sqrt(128) rows: RMS-normalise the pair (y0, y1) of a row over the wave
  auto norm = [&](float2 y, const uint16_t *w) {
    const float r = 1.0f / sqrtf(wave_sum_dpp(y.x * y.x + y.y * y.y) / (float)CHDIM + CX_QK_EPS);
    return make_float2(y.x * r * h2f(w[h * CHDIM + d]), y.y * r * h2f(w[h * CHDIM + d + 1]));
  };
  auto row = [&](int t, int part) {
    const int m = part * CD + h * CHDIM + d;
    float2 v[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) v[s] = *(const float2 *)(C + ((size_t)s * nt + t) * (3 * CD) + m);
    float2 y = v[0];
#pragma unroll
    for (int s = 1; s < NS; s++) {
      y.x += v[s].x;
      y.y += v[s].y;
    }
    return y;
  };
  // rows i and i + CXA_WAVES of every wave, all loads ahead of the first use;
  // t past the chunk's tokens re-reads the last, t before it the halo
  float2 k[2], v[2], q[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int i = wave + CXA_WAVES * u, t = base + i;
    if (t >= 0) {
      const int tc = min(t, n - 1);
      k[u] = row(tc, 1);
      v[u] = row(tc, 2);
      q[u] = row(tc, 0);
    } else if (t0 + t >= 0 && i < W - 1) {
      const float *p = halo_in + (size_t)(t + CX_HALO) * 2 * CD + h * CHDIM + d;
      k[u] = *(const float2 *)p;
      v[u] = *(const float2 *)(p + CD);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int i = wave + CXA_WAVES * u, t = base + i;
    if (i >= CXA_T + W - 1 || t >= n || t0 + t < 0) continue;  // no such row, or never in a window
    if (t >= 0) k[u] = norm(k[u], kn);
    *(float2 *)(ks + i * CXA_LD + d) = k[u];
    *(float2 *)(vs + i * CXA_LD + d) = v[u];
    if (t < tb) continue;
    *(float2 *)(qs + (t - tb) * CXA_LD + d) = norm(q[u], qn);
    if (halo_out && t >= n - CX_HALO) {  // each row by the block that owns the token
      float *o = halo_out + (size_t)(t - (n - CX_HALO)) * 2 * CD + h * CHDIM + d;
      *(float2 *)o = k[u];
      *(float2 *)(o + CD) = v[u];
    }
  }
  __syncthreads();
  const float scale = 1.0f / sqrtf((float)CHDIM);
  const float slope = exp2f(-8.0f * (float)(h + 1) / (float)CNH);
  const int j = lane >> 2, p = lane & 3;
  {
    const int qi = wave, t = tb + qi;
    if (t >= nt) return;
    float2 o = make_float2(0.f, 0.f);
    if (t < n) {
      const int key = t - W + 1 + j;                    // this lane's key, LDS row qi + j
      const bool in = j < W && t0 + key >= 0;
      const float *kr = ks + (in ? qi + j : qi + W - 1) * CXA_LD + 4 * p, *qr = qs + qi * CXA_LD + 4 * p;
      f32x4 d4 = f32x4{0.f, 0.f, 0.f, 0.f};  // four sums of 8: in one of 32 the scores are a few ulps further off
#pragma unroll
      for (int i = 0; i < CHDIM / 16; i++) {
        const f32x4 a = *(const f32x4 *)(qr + 16 * i), b = *(const f32x4 *)(kr + 16 * i);
#pragma unroll
        for (int e = 0; e < 4; e++) d4[e] = fmaf(a[e], b[e], d4[e]);
      }
      float dot = (d4[0] + d4[1]) + (d4[2] + d4[3]);
      dot += __shfl_xor(dot, 1, 64);
      dot += __shfl_xor(dot, 2, 64);
      const float sc = in ? dot * scale - slope * (float)(t - key) : -INFINITY;
      float mx = sc;
#pragma unroll
      for (int x = 4; x < 64; x <<= 1) mx = fmaxf(mx, __shfl_xor(mx, x, 64));
      const float e = in ? expf(sc - mx) : 0.f;  // the query's own key is always in: mx is finite
      float sum = e;
#pragma unroll
      for (int x = 4; x < 64; x <<= 1) sum += __shfl_xor(sum, x, 64);
      const float pr = e / sum;
      for (int jj = 0; jj < W; jj++) {
        if (t0 + t - W + 1 + jj < 0) continue;
        const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pr), 4 * jj));
        const float2 v = *(const float2 *)(vs + (qi + jj) * CXA_LD + d);
        o.x = fmaf(pj, v.x, o.x);
        o.y = fmaf(pj, v.y, o.y);
      }
    }
    h2 hi, lo;
    split2(o.x, o.y, hi, lo);
    _Float16 *b = (_Float16 *)B + h * CHDIM + d;
    *(h2 *)(b + (size_t)t * CD) = hi;
    *(h2 *)(b + (size_t)(nt + t) * CD) = lo;
  }
}

// the concatenated input features [T][292] (debugCodecDecode's "concat")
__global__ void cx_concat_kernel(const uint16_t *cbn, const uint32_t *sem, const uint32_t *ac,
                                 int levels, int T, float *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < T * CIN) out[i] = cx_feature(cbn, sem, ac, levels, i / CIN, i % CIN);
}

// ------------------------------------------------ weight preparation
// normalizeCodebook (src/shaders.ts:851-885): f16(sum / max(usage, 1e-5))
__global__ void cx_vq_norm_kernel(const uint16_t *sum, const uint16_t *usage, uint16_t *out) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)CSEM * CSEMD;
       i += (size_t)gridDim.x * blockDim.x) {
    const float u = fmaxf(h2f(usage[i / CSEMD]), 1e-5f);
    const _Float16 r = (_Float16)(h2f(sum[i]) / u);
    out[i] = __builtin_bit_cast(uint16_t, r);
  }
}

// causal conv weight norm per output row (causalConv1d, src/shaders.ts:
// 941-957): rs = g / sqrt(sum over pairs of (a^2 + b^2) + 1e-12), rows >= mv
// zero.  One thread per row.
__global__ void cx_conv_rowscale_kernel(const uint16_t *w, const uint16_t *g, int mv, int K,
                                        int rows, float *rs) {
  const int co = blockIdx.x * blockDim.x + threadIdx.x;
  if (co >= rows) return;
  if (co >= mv) {
    rs[co] = 0.f;
    return;
  }
  const uint16_t *wr = w + (size_t)co * K;
  float ss = 0.f;
  for (int p = 0; p < K / 2; p++) {
    const float a = h2f(wr[2 * p]), b = h2f(wr[2 * p + 1]);
    ss += a * a + b * b;
  }
  rs[co] = (1.0f / sqrtf(ss + 1e-12f)) * h2f(g[co]);
}

// transposed conv weight norm per input channel (convTransposeNormScale,
// src/shaders.ts:1009-1058, same 256-lane strided sums and tree):
// scale[ci] = g[ci] / ||w[ci, :, :]||.  One block of 256 per channel.
__global__ __launch_bounds__(256) void cx_up_scale_kernel(const uint16_t *w, const uint16_t *g,
                                                          float *scale) {
  __shared__ float sd[256];
  const int ci = blockIdx.x, tid = threadIdx.x, n = CD * CK_UP;
  const uint16_t *wr = w + (size_t)ci * n;
  float ss = 0.f;
  for (int i = tid; i < n; i += 256) {
    const float v = h2f(wr[i]);
    ss += v * v;
  }
  sd[tid] = ss;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) sd[tid] += sd[tid + s];
    __syncthreads();
  }
  if (tid == 0) scale[ci] = h2f(g[ci]) * (1.0f / sqrtf(sd[0] + 1e-12f));
}

// A of the input conv: [CD][CKIN], A[co][kk * CIN + ci] = w[co][ci][kk]
__global__ void cx_reorder_in_kernel(const uint16_t *w, uint16_t *A) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)CD * CKIN;
       i += (size_t)gridDim.x * blockDim.x) {
    const int co = (int)(i / CKIN), k = (int)(i % CKIN);
    uint16_t v = 0;
    if (k < CIN * CK_IN) {
      const int kk = k / CIN, ci = k - kk * CIN;
      v = w[((size_t)co * CIN + ci) * CK_IN + kk];
    }
    A[i] = v;
  }
}

// A of the output conv: [CPATCH_ROWS][CKOUT], A[co][kk * CD + ci] =
// w[co][ci][kk], rows >= CPATCH zero
__global__ void cx_reorder_out_kernel(const uint16_t *w, uint16_t *A) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)CPATCH_ROWS * CKOUT;
       i += (size_t)gridDim.x * blockDim.x) {
    const int co = (int)(i / CKOUT), k = (int)(i % CKOUT);
    const int kk = k / CD, ci = k - kk * CD;
    A[i] = co < CPATCH ? w[((size_t)co * CD + ci) * CK_OUT + kk] : (uint16_t)0;
  }
}

// A of a transposed conv: [2 * CD][CKUP], A[r * CD + co][(1 - j) * CD + ci] =
// w[ci][co][r + 2 j] (w is [c_in][c_out][4]; j = 1 is the step before, whose
// packed row comes first)
__global__ void cx_reorder_up_kernel(const uint16_t *w, uint16_t *A) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)2 * CD * CKUP;
       i += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(i / CKUP), k = (int)(i % CKUP);
    const int r = row / CD, co = row - r * CD, j = 1 - k / CD, ci = k % CD;
    A[i] = w[((size_t)ci * CD + co) * CK_UP + r + 2 * j];
  }
}

}  // namespace vx
