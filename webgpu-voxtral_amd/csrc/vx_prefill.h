// vx_prefill.h -- batched prefill of the backbone.  The reference prefills
// one token per backboneStep (src/engine.ts:2457-2472); here a chunk of up
// to PF_MAXT prompt tokens goes through each layer at once, so every weight
// is read once per chunk and the projections are GEMMs
//   C[s][col][m] = sum_{k in slice s} W[m][k] * (B[col][k] + B[nt + col][k])
// (f16 x f16 -> f32 on the matrix cores: vx_gemm.h).  W is the layer's f16
// weight matrix (row-major, as loaded); B holds the chunk's activations in
// hi/lo form (column t = f16(y_t), column nt + t = f16(y_t - hi), each
// column's K halves contiguous), so the product keeps f32 accuracy.  The
// GEMM leaves ns partial sums over slices of K in ns consecutive [nt][ldc]
// blocks of C, and the consumer adds them in order.  Small per-token kernels do RoPE + K/V writes and the causal
// attention, and each of them, or a residual add + RMSNorm, or SwiGLU,
// writes the next GEMM's B directly.  The
// result (K/V cache rows, residual stream, final norm of the last token,
// position) equals that of the per-token steps up to f32 summation order.
#pragma once
#include "vx_kernels.h"
#include <type_traits>

namespace vx {

constexpr int PF_MAXT = 1024;          // tokens per chunk, at most
constexpr int PF_NC = 2 * PF_MAXT;     // B columns (hi, lo), at most
// A chunk of n tokens uses nt = gm_cols(n) hi columns (16, 32 or a multiple of
// 64: the widths the GEMM grids come in) and as many lo columns.

// value of output (token t, row m): the sum of the NS K-slice blocks, in order
template <int NS>
__device__ __forceinline__ float pf_c(const float *C, int ldc, int nt, int t, int m) {
  float v[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) v[s] = C[((size_t)s * nt + t) * ldc + m];
  float y = v[0];
#pragma unroll
  for (int s = 1; s < NS; s++) y += v[s];
  return y;
}
// four consecutive rows m .. m + 3 (m % 4 == 0)
template <int NS>
__device__ __forceinline__ f32x4 pf_c4(const float *C, int ldc, int nt, int t, int m) {
  f32x4 v[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) v[s] = *(const f32x4 *)(C + ((size_t)s * nt + t) * ldc + m);
  f32x4 y = v[0];
#pragma unroll
  for (int s = 1; s < NS; s++) y += v[s];
  return y;
}

// ------------------------------------------------------- per-token kernels
// hi/lo halves of y into B columns t and nt + t at k (8 consecutive k)
__device__ __forceinline__ void pf_put8(h8 *B, int K, int nt, int t, int kb, const float (&y)[8]) {
  h8 hi, lo;
  split_n<8>(y, hi, lo);
  B[(size_t)t * (K / 8) + kb] = hi;
  B[(size_t)(nt + t) * (K / 8) + kb] = lo;
}

// The rows of a prompt are DIM = 384 groups of 8 values: a block of 384 threads
// holds one row, so every load of it is in flight at once and its sum of
// squares costs one barrier.  (256 threads, half of them with a second group
// behind the first: 7 us at 256 tokens for the residual, 8 us for the packing
// of the embeddings in a kernel of its own.)
constexpr int PF_ROW = DIM / 8;
static_assert(PF_ROW == 6 * 64, "one 8-value group per thread");

// B columns t and nt + t from rmsNorm(v) * g (src/shaders.ts:137-183), v the
// row's 8 values of this thread
__device__ __forceinline__ void pf_norm_pack(const float (&v)[8], const uint16_t *g, float eps, int nt, int t, h8 *B) {
  __shared__ float red[6];
  const int kb = threadIdx.x;
  const h8 gv = *(const h8 *)(g + kb * 8);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) ss = fmaf(v[e], v[e], ss);
  ss = wave_sum_dpp(ss);
  if ((kb & 63) == 0) red[kb >> 6] = ss;
  __syncthreads();
  const float r =
      1.0f / sqrtf((((red[0] + red[1]) + (red[2] + red[3])) + (red[4] + red[5])) / (float)DIM + eps);
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; e++) y[e] = v[e] * r * (float)gv[e];
  pf_put8(B, DIM, nt, t, kb, y);
}
__device__ __forceinline__ void pf_zero_pack(int nt, int t, h8 *B) {
  const float y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  pf_put8(B, DIM, nt, t, threadIdx.x, y);
}

// X[t] = token embedding row, or voice row v = t + tok0 - vstart for the
// tokens inside [vstart, vstart + vcount) (src/engine.ts:2457-2472), and the
// first layer's B from it; columns of tokens t >= n are zero.
// Grid: nt blocks of PF_ROW.
__global__ __launch_bounds__(PF_ROW) void pf_embed_pack_kernel(const uint16_t *table, const int32_t *tokens,
                                                               const float *voice, int vstart, int vcount, int tok0,
                                                               int n, int nt, float *X, const uint16_t *g, float eps,
                                                               h8 *B) {
  const int t = blockIdx.x, i = 8 * threadIdx.x, gi = tok0 + t;
  if (t >= n) {
    pf_zero_pack(nt, t, B);
    return;
  }
  float v[8];
  if (voice && gi >= vstart && gi < vstart + vcount) {
    const float *p = voice + (size_t)(gi - vstart) * DIM + i;
    const f32x4 a = *(const f32x4 *)p, b = *(const f32x4 *)(p + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
    const h8 w = *(const h8 *)(table + (size_t)tokens[t] * DIM + i);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (float)w[e];
  }
  float *x = X + (size_t)t * DIM + i;
  *(f32x4 *)x = f32x4{v[0], v[1], v[2], v[3]};
  *(f32x4 *)(x + 4) = f32x4{v[4], v[5], v[6], v[7]};
  pf_norm_pack(v, g, eps, nt, t, B);
}

// Residual add of a DIM-row GEMM output, X[t] += y (addInPlace,
// src/shaders.ts:532-547), then, with PACK, the next GEMM's B from
// rmsNorm(X[t]) * g; columns of tokens t >= n are zero.
// Grid: nt blocks (n without PACK) of PF_ROW.
template <bool PACK, int NS>
__global__ __launch_bounds__(PF_ROW) void pf_resid_pack_kernel(const float *C, int n, int nt, float *X,
                                                               const uint16_t *g, float eps, h8 *B) {
  const int t = blockIdx.x, i = 8 * threadIdx.x;
  if (t >= n) {
    if (PACK) pf_zero_pack(nt, t, B);
    return;
  }
  float *x = X + (size_t)t * DIM + i;
  const f32x4 xa = *(const f32x4 *)x, xb = *(const f32x4 *)(x + 4);
  const f32x4 a = pf_c4<NS>(C, DIM, nt, t, i), b = pf_c4<NS>(C, DIM, nt, t, i + 4);
  float v[8];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    v[e] = xa[e] + a[e];
    v[4 + e] = xb[e] + b[e];
  }
  *(f32x4 *)x = f32x4{v[0], v[1], v[2], v[3]};
  *(f32x4 *)(x + 4) = f32x4{v[4], v[5], v[6], v[7]};
  if (PACK) pf_norm_pack(v, g, eps, nt, t, B);
}

// SwiGLU of the stacked [W1; W3] output (ldc = 2 HID; swiGLU,
// src/shaders.ts:483-501) written as the down GEMM's B (K = HID); columns of
// tokens t >= n are zero.  Grid: (nt, HID / 8 / 128) of 128, one 8-value
// group per thread.
template <int NS>
__global__ __launch_bounds__(128) void pf_swiglu_pack_kernel(const float *C, int n, int nt, h8 *B) {
  const int t = blockIdx.x, kb = blockIdx.y * 128 + threadIdx.x;
  float y[8];
  if (t < n) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const f32x4 gt = pf_c4<NS>(C, 2 * HID, nt, t, kb * 8 + 4 * h);
      const f32x4 up = pf_c4<NS>(C, 2 * HID, nt, t, HID + kb * 8 + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; e++) y[4 * h + e] = (gt[e] / (1.0f + expf(-gt[e]))) * up[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = 0.f;
  }
  pf_put8(B, HID, nt, t, kb, y);
}
static_assert(DIM % 8 == 0 && (HID / 8) % 128 == 0, "prefill packing groups");

// ------------------------------------------------ causal attention on MFMA
// Causal attention of the chunk (attnScore + softmax + attnValue per prompt
// token over keys 0..pos0+t, src/shaders.ts:306-447) with the products on the
// matrix cores, in the transposed form (the token is the MFMA column, so every
// lane holds one token's values).  Per 32-key tile, wave and 16 tokens:
//   S^T[32 keys][16 tokens] = K[32][128] . Q^T[128][16]        16x16x32 f16
//   O^T[128 dims][16 tokens] += V^T[128][32 keys] . P^T[32][16]  16x16x32 f16
// Every f32 operand is split into f16 hi + lo and a product is hi.hi + hi.lo +
// lo.hi, about 2^-20 relative (the dropped lo.lo term), where the prefill
// GEMMs, with exact f16 weights, are at the split's 2^-21.  An f16 cache is
// exact in f16: its lo halves are zero, so they are neither stored nor
// multiplied.
//
// The D layout of S^T (lane l: keys 16 kt + 4 (l / 16) .. + 3 of token l % 16)
// becomes the B operand of the second product, which wants 8 consecutive
// contraction slots per lane, by numbering the slots to suit: slot 8 g + 4 kt
// + q is key 16 kt + 4 g + q, so P needs no shuffle.
//
// pf_qkv_epi_kernel writes the keys and values of the whole context as the
// operands of both products, a lane's 16 bytes together, hi and lo split:
// per KV head and 32-key tile, K hi [2 kt][4 chunks of 32 dims][64 lanes][8],
// K lo, V^T hi [8 tiles of 16 dims][64 lanes][8 slots], V^T lo (f16 cache: K
// and V^T hi only), 32 or 16 KB in all; keys past the last are zero.  So the
// attention's tiles go from memory to LDS by direct loads and from there to
// the MFMAs as they are.  Splitting and transposing in each attention block
// instead (16 tokens each, every block its own copy) took 2.2 us per pair of
// tiles, 0.5 of it in two barriers: 19 us at 256 tokens (13 now), 98 us at 1024
// tokens on 500 of context, f16 cache (51 now).
typedef _Float16 hf4 __attribute__((ext_vector_type(4)));
constexpr int PFA_K = 32;      // keys per tile
constexpr int PFA_PART = 8192; // bytes of K or V^T of one tile, hi or lo

// hi/lo operand halves (split2) of 8 or 4 f32 values
__device__ __forceinline__ void split8(const f32x4 a, const f32x4 b, h8 &hi, h8 &lo) {
  const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  split_n<8>(x, hi, lo);
}
__device__ __forceinline__ void split4(const f32x4 a, hf4 &hi, hf4 &lo) {
  const float x[4] = {a[0], a[1], a[2], a[3]};
  split_n<4>(x, hi, lo);
}

template <typename KVT>
__host__ __device__ constexpr int pfa_tile_bytes() {
  return sizeof(KVT) == 2 ? 2 * PFA_PART : 4 * PFA_PART;
}
// 8 consecutive cached values, and a value as the cache holds it
__device__ __forceinline__ void kv_load8(const float *p, float (&y)[8]) {
  const f32x4 a = *(const f32x4 *)p, b = *(const f32x4 *)(p + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    y[e] = a[e];
    y[4 + e] = b[e];
  }
}
__device__ __forceinline__ void kv_load8(const uint16_t *p, float (&y)[8]) {
  const h8 a = *(const h8 *)p;
#pragma unroll
  for (int e = 0; e < 8; e++) y[e] = (float)a[e];
}
__device__ __forceinline__ float kv_load(const float *p) { return *p; }
__device__ __forceinline__ float kv_load(const uint16_t *p) { return h2f(*p); }
__device__ __forceinline__ float kv_store(float *p, float v) { return *p = v; }
__device__ __forceinline__ float kv_store(uint16_t *p, float v) {
  const uint16_t b = f2h(v);
  *p = b;
  return h2f(b);
}

// QKV outputs, two kinds of block in one launch of 512 threads:
//  - block b < tiles * NKV (tiles = ceil((pos0 + n) / 32)): KV head b % NKV of
//    the 32 positions of tile b / NKV.  New keys and values (positions pos0 ..
//    pos0 + n - 1) come from the GEMM's K slices, the keys with interleaved
//    rope (src/shaders.ts:224-256), and go to the cache; older ones come from
//    the cache; both are written as the attention's operands (above), as the
//    cache holds them.  Thread i is fragment i / 64's lane i % 64 of both K
//    and V^T.
//  - the blocks after them: q of token (b - tiles * NKV) / 4, rope, one row
//    pair per thread.
// 6 us at 256 tokens: the epilogue alone took 5.6 and a second kernel that
// packed the operands from the cache 5.
// KVT = float (f32 cache) or uint16_t (f16 cache).
template <int NS, typename KVT>
__global__ __launch_bounds__(512) void pf_qkv_epi_kernel(const float *C, int nt, float *Q, KVT *kc, KVT *vc,
                                                         int max_seq, int pos0, int n, const float *inv_freq,
                                                         unsigned char *kv) {
  constexpr bool EXACT = sizeof(KVT) == 2;
  const int kend = pos0 + n, tiles = (kend + PFA_K - 1) / PFA_K;
  if ((int)blockIdx.x >= tiles * NKV) {
    const int b = blockIdx.x - tiles * NKV, t = b >> 2, row = 2 * ((b & 3) * 512 + threadIdx.x);
    const float y0 = pf_c<NS>(C, QKV_ROWS, nt, t, row), y1 = pf_c<NS>(C, QKV_ROWS, nt, t, row + 1);
    const float ang = (float)(pos0 + t) * inv_freq[(row & (HD - 1)) >> 1];
    const float cs = cosf(ang), sn = sinf(ang);
    *(float2 *)(Q + (size_t)t * QD + row) = make_float2(y0 * cs - y1 * sn, y0 * sn + y1 * cs);
    return;
  }
  const int it = blockIdx.x / NKV, kvh = blockIdx.x % NKV, f = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  KVT *Kb = kc + (size_t)kvh * max_seq * HD, *Vb = vc + (size_t)kvh * max_seq * HD;
  h8 *o = (h8 *)(kv + ((size_t)it * NKV + kvh) * pfa_tile_bytes<KVT>());
  // K: position key, dims d .. d + 7; V^T: dim dv of 8 positions.  Every load is
  // issued before the first use, from a clamped row where there is none; only
  // a tile that holds older positions (uniform) reads the cache as well.
  const int key = it * PFA_K + 16 * (f >> 2) + r, d = 32 * (f & 3) + 8 * g, dv = 16 * f + r;
  auto vpos = [&](int e) { return it * PFA_K + 16 * (e >> 2) + 4 * g + (e & 3); };
  auto row = [&](int pos) { return max(min(pos, kend - 1) - pos0, 0); };
  float k[8], v[8], fr[4];
  const f32x4 ka = pf_c4<NS>(C, QKV_ROWS, nt, row(key), QD + kvh * HD + d);
  const f32x4 kb = pf_c4<NS>(C, QKV_ROWS, nt, row(key), QD + kvh * HD + d + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) fr[e] = inv_freq[(d >> 1) + e];
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = pf_c<NS>(C, QKV_ROWS, nt, row(vpos(e)), QD + KVD + kvh * HD + dv);
  float ko[8], vo[8];
  if (it * PFA_K < pos0) {
    kv_load8(Kb + (size_t)min(key, pos0 - 1) * HD + d, ko);
#pragma unroll
    for (int e = 0; e < 8; e++) vo[e] = kv_load(Vb + (size_t)min(vpos(e), pos0 - 1) * HD + dv);
  }
  const float y[8] = {ka[0], ka[1], ka[2], ka[3], kb[0], kb[1], kb[2], kb[3]};
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const float ang = (float)key * fr[e >> 1];
    const float cs = cosf(ang), sn = sinf(ang);
    k[e] = y[e] * cs - y[e + 1] * sn;
    k[e + 1] = y[e] * sn + y[e + 1] * cs;
  }
  if (key >= pos0 && key < kend) {
#pragma unroll
    for (int e = 0; e < 8; e++) k[e] = kv_store(Kb + (size_t)key * HD + d + e, k[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) k[e] = key < pos0 ? ko[e] : 0.f;
  }
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int pos = vpos(e);
    if (pos >= pos0 && pos < kend) v[e] = kv_store(Vb + (size_t)pos * HD + dv, v[e]);
    else v[e] = pos < pos0 ? vo[e] : 0.f;
  }
  h8 hi, lo;
  h8 *ov = o + (EXACT ? 1 : 2) * (PFA_PART / 16);
  split_n<8>(k, hi, lo);
  o[f * 64 + lane] = hi;
  if (!EXACT) o[PFA_PART / 16 + f * 64 + lane] = lo;
  split_n<8>(v, hi, lo);
  ov[f * 64 + lane] = hi;
  if (!EXACT) ov[PFA_PART / 16 + f * 64 + lane] = lo;
}

// maximum / sum of a value over the four lane groups that hold one token, by
// two lane swaps of the value with a copy of itself (an LDS permute, __shfl_xor,
// is about 100 clocks on each of the tile's four steps).  In asm, with the
// two wait states that a swap needs after a VALU write: for the builtins this
// compiler uses the first of the two results twice.  The results only feed
// VALU instructions.
__device__ __forceinline__ void pfa_swap16(float &a, float &b) {
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void pfa_swap32(float &a, float &b) {
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float pfa_max4(float a) {
  float b = a;
  pfa_swap16(a, b);
  a = b = fmaxf(a, b);
  pfa_swap32(a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float pfa_sum4(float a) {
  float b = a;
  pfa_swap16(a, b);
  a = b = a + b;
  pfa_swap32(a, b);
  return a + b;
}

// Block = (16 tokens, KV head): two key groups of 4 waves, wave w of a group
// query head 4 kv_head + w.  Group g walks tiles g, g + 2, ... in two LDS
// stages of its own, one tile loading while the last is used, with its own
// online softmax; the groups' (max, sum, O) are merged through LDS at the end,
// in group order.  Writes hi/lo rows of the O projection's B (rows t and
// nt + t), zero for t >= n.
// 32 tokens per wave (half the LDS reads per MFMA, half the blocks) and four
// groups (f16 cache) were slower at every size: 1024 tokens, f32 cache, 56
// against 44 us; 512 tokens 31 against 21; 1024 tokens on 500 of context, f16
// cache, 62 and 64 against 49-50; 276 more on those 42 and 41 against 38.
// Launch: grid NKV * nt / 16, 512 threads, pfa_lds dynamic LDS.  Block b takes
// KV head b % 8 (blocks with equal b % 8 share an XCD, so its L2 holds that
// head's tiles) and the later, longer token tiles first.
constexpr int PFA_T = 16;            // tokens per block
constexpr int PFA_KG = 2;            // key groups per block
constexpr int PFA_RED = 2 + HD / 4;  // merged values per lane: m, l, O^T
template <typename KVT>
__host__ __device__ constexpr int pfa_lds() {
  static_assert((PFA_KG - 1) * 4 * PFA_RED * 256 <= PFA_KG * 2 * 2 * PFA_PART, "merge area");
  return PFA_KG * 2 * pfa_tile_bytes<KVT>();
}
template <typename KVT>
__global__ __launch_bounds__(256 * PFA_KG) void pf_attn_mfma_kernel(const float *Q, const unsigned char *kv, int pos0,
                                                                    int n, int nt, h8 *B) {
  constexpr bool EXACT = std::is_same<KVT, uint16_t>::value;  // f16 cache: no lo halves
  constexpr int TILE = pfa_tile_bytes<KVT>(), NL = TILE / 4096;  // bytes; direct loads per wave
  extern __shared__ __attribute__((aligned(16))) unsigned char pfa_smem[];
  const int kvh = blockIdx.x % NKV, t0 = (gridDim.x / NKV - 1 - blockIdx.x / NKV) * PFA_T;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp_k = wave >> 2, hw = wave & 3;  // key group, head within the KV group
  const int h = kvh * (NH / NKV) + hw;
  const int col = lane & 15, grp = lane >> 4;  // MFMA column (token) and row group
  const int t = t0 + col;                      // this lane's token
  _Float16 *const out = (_Float16 *)B + (size_t)t * QD + h * HD + 4 * grp;  // its hi row; lo: nt rows on
  if (t0 >= n) {  // padding columns of the GEMM: zero hi and lo (group 0 writes)
    if (grp_k == 0) {
#pragma unroll
      for (int dt = 0; dt < HD / 16; dt++) {
        *(hf4 *)(out + dt * 16) = hf4{0, 0, 0, 0};
        *(hf4 *)(out + (size_t)nt * QD + dt * 16) = hf4{0, 0, 0, 0};
      }
    }
    return;
  }
  const int last = pos0 + min(t, n - 1);            // last key of this lane's token
  const int kend = pos0 + min(t0 + PFA_T, n);       // keys of the block: [0, kend)
  const int ntile = (kend + PFA_K - 1) / PFA_K;
  const int iters = (ntile + PFA_KG - 1) / PFA_KG;  // the same count in every group
  unsigned char *const ring = pfa_smem + grp_k * 2 * TILE;
  // tile it into stage s: wave w of the group brings the KBs w, w + 4, ...
  auto load_tile = [&](int it, int s) {
    const unsigned char *src = kv + ((size_t)it * NKV + kvh) * TILE + hw * 1024 + lane * 16;
    unsigned char *dst = ring + s * TILE + hw * 1024;
#pragma unroll
    for (int i = 0; i < NL; i++)
      __builtin_amdgcn_global_load_lds((const void *)(src + i * 4096),
                                       (__attribute__((address_space(3))) void *)(dst + i * 4096), 16, 0, 0);
  };
  if (grp_k < ntile) load_tile(grp_k, 0);

  // The softmax is of powers of two, exp2(s scale - ms) with ms = m scale, m the
  // largest s: v_exp_f32 is off by 8.3e-8 at most and 2.0e-8 rms over [-126, 0], as
  // expf is (4.7 M arguments), and flushes what is below 2^-126, of sums of at
  // least 1.  The scale is applied to the score, in the exponent's fma, not to
  // q: a query is split in its own units, since lo halves of a q smaller by
  // 0.13 reach the f16 subnormals, whose quantum is fixed (queries of 0.02
  // against keys of 140: error of the attention 1.5e-5, and 1.8e-6 this way).
  const float scale = 1.44269504f / sqrtf((float)HD);
  // Q^T operand of S^T (token t, dims 32c + 8grp..+8), hi and lo; padding
  // tokens zero
  h8 qh[HD / 32], ql[HD / 32];
  {
    const float *qp = Q + (size_t)min(t, n - 1) * QD + h * HD + 8 * grp;
#pragma unroll
    for (int c = 0; c < HD / 32; c++) {
      f32x4 a = *(const f32x4 *)(qp + 32 * c), b = *(const f32x4 *)(qp + 32 * c + 4);
      if (t >= n) a = b = f32x4{0.f, 0.f, 0.f, 0.f};
      split8(a, b, qh[c], ql[c]);
    }
  }
  float m = -INFINITY, ms = -INFINITY, l = 0.f;
  f32x4 o[HD / 16];
#pragma unroll
  for (int dt = 0; dt < HD / 16; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int i = 0; i < iters; i++) {
    const int it = grp_k + PFA_KG * i, kb = it * PFA_K;
    // this wave's share of tile it is in (every load is: the next tile's go
    // out below), and past the barrier every wave's is, and no wave reads the
    // other stage any more
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    if (it == ntile - 1 && kend % PFA_K) {
      // The last tile's keys past kend are later blocks', hidden from every
      // token of this one, but 0 times a value that is not finite is NaN: each
      // lane zeroes those of the 16 bytes of V^T it brought, fragments hw and
      // hw + 4, whose slot 4 kt + q is key 16 kt + 4 grp + q.  (A token that is
      // not finite still reaches the up to 15 before it in its own block.)  Here
      // it needs no barrier of its own; with one, after this one, it took 0.9 us
      // of 13.8 at 256 tokens, and masks on the fragments as the product reads
      // them cost registers past the 128 that let two blocks share a CU.
      u32x4 keep, *f = (u32x4 *)(ring + (i & 1) * TILE + (EXACT ? 1 : 2) * PFA_PART) + hw * 64 + lane;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int key = kb + 16 * (j >> 1) + 4 * grp + 2 * (j & 1);
        keep[j] = (key < kend ? 0xFFFFu : 0u) | (key + 1 < kend ? 0xFFFF0000u : 0u);
      }
#pragma unroll
      for (int k = 0; k < (EXACT ? 2 : 4); k++) f[k * 256] &= keep;  // hi, then lo
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    }
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (it + PFA_KG < ntile) load_tile(it + PFA_KG, (i + 1) & 1);
    if (it >= ntile) continue;  // uniform over the group
    const h8 *kh = (const h8 *)(ring + (i & 1) * TILE) + lane, *kl = kh + PFA_PART / 16;
    const h8 *vh = kh + (EXACT ? 1 : 2) * (PFA_PART / 16), *vl = vh + PFA_PART / 16;

    // S^T of keys kb + 16kt + (4grp..+3), token t; the lo products in an
    // accumulator of their own, so no chain of dependent MFMAs is longer than 8
    f32x4 s[2], sl[2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) s[kt] = sl[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < HD / 32; c++)
#pragma unroll
      for (int kt = 0; kt < 2; kt++) {
        const h8 a = kh[(4 * kt + c) * 64];
        s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qh[c], s[kt], 0, 0, 0);
        sl[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ql[c], sl[kt], 0, 0, 0);
        if (!EXACT) sl[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl[(4 * kt + c) * 64], qh[c], sl[kt], 0, 0, 0);
      }
    // online softmax over this tile's keys (8 per lane, 4 lanes per token);
    // only a tile that reaches past the block's first token has keys to hide
    float p[8], mx = -INFINITY;
    const bool edge = kb + PFA_K - 1 > pos0 + t0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      p[q] = s[q >> 2][q & 3] + sl[q >> 2][q & 3];
      if (edge && kb + 16 * (q >> 2) + 4 * grp + (q & 3) > last) p[q] = -INFINITY;
      mx = fmaxf(mx, p[q]);
    }
    mx = pfa_max4(mx);
    if (__builtin_amdgcn_ballot_w64(mx > m)) {  // some token's maximum grows
      // a token whose keys all lie before this tile's start keeps m = -inf
      // (only in groups other than 0: key 0 <= last is in tile 0)
      m = fmaxf(m, mx);
      const float msnew = m * scale;
      const float corr = msnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(ms - msnew);
      ms = msnew;
      l *= corr;
#pragma unroll
      for (int dt = 0; dt < HD / 16; dt++) o[dt] = o[dt] * corr;
    }
    const float base = ms == -INFINITY ? 0.f : ms;
    float ps = 0.f;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      p[q] = __builtin_amdgcn_exp2f(fmaf(p[q], scale, -base));  // hidden keys: 0
      ps += p[q];
    }
    l += pfa_sum4(ps);
    h8 ph, pl;
    split_n<8>(p, ph, pl);
    // O^T += V^T . P^T
#pragma unroll
    for (int dt = 0; dt < HD / 16; dt++) {
      const h8 a = vh[dt * 64];
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ph, o[dt], 0, 0, 0);
      if (!EXACT) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl[dt * 64], ph, o[dt], 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, pl, o[dt], 0, 0, 0);
    }
  }
  // merge the groups' (m, l, O^T) in group order: groups 1.. write theirs
  // to LDS (lane-minor), group 0 combines them
  float *red = (float *)pfa_smem;
  __syncthreads();  // every group is done with its stages
  if (grp_k > 0) {
    float *r = red + ((grp_k - 1) * 4 + hw) * PFA_RED * 64 + lane;
    r[0] = ms;
    r[64] = l;
#pragma unroll
    for (int dt = 0; dt < HD / 16; dt++)
#pragma unroll
      for (int q = 0; q < 4; q++) r[(2 + 4 * dt + q) * 64] = o[dt][q];
  }
  __syncthreads();
  if (grp_k > 0) return;
  float mm = ms;
#pragma unroll
  for (int g = 1; g < PFA_KG; g++) mm = fmaxf(mm, red[((g - 1) * 4 + hw) * PFA_RED * 64 + lane]);
  const float c0 = __builtin_amdgcn_exp2f(ms - mm);  // ms is finite in group 0
  l *= c0;
#pragma unroll
  for (int dt = 0; dt < HD / 16; dt++) o[dt] = o[dt] * c0;
#pragma unroll
  for (int g = 1; g < PFA_KG; g++) {
    const float *rg = red + ((g - 1) * 4 + hw) * PFA_RED * 64 + lane;
    const float cg = __builtin_amdgcn_exp2f(rg[0] - mm);  // ms = -inf: 0
    l += rg[64] * cg;
#pragma unroll
    for (int dt = 0; dt < HD / 16; dt++)
#pragma unroll
      for (int q = 0; q < 4; q++) o[dt][q] += rg[(2 + 4 * dt + q) * 64] * cg;
  }
  // out[t][dims] = O^T / l, as hi and lo f16 rows of B (zero past n)
  const float inv = 1.0f / l;
#pragma unroll
  for (int dt = 0; dt < HD / 16; dt++) {
    hf4 hi = hf4{0, 0, 0, 0}, lo = hf4{0, 0, 0, 0};
    if (t < n) split4(o[dt] * inv, hi, lo);
    *(hf4 *)(out + dt * 16) = hi;
    *(hf4 *)(out + (size_t)nt * QD + dt * 16) = lo;
  }
}

}  // namespace vx
