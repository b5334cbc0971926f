// vx_gemm.h -- the prefill's projections as hand-written gfx950 MFMA GEMMs:
//   C[s][col][m] = sum_{k in slice s} W[m][k] * (Bhi[col][k] + Blo[col][k])
// W: f16 weights, row-major M x K as loaded (the decode GEMVs read the same
// copy).  B: the hi half of activation column col is K halves from
// B + col ldb, its f16 residual (lo) from B + blo + col ldb (16-byte
// aligned), as the producer kernels write them.  ldb = K for packed
// columns; a causal convolution's columns overlap (ldb = channels, K = taps x
// channels), so its input is packed once and not once per tap.  Hi and lo both go through MFMA with f32
// accumulators, so the product keeps f32 accuracy.  The K range is split
// into S_out slices whose partial sums land in S_out consecutive [nt][M]
// blocks of C; the consumer adds them (fixed order, so results are
// deterministic).
//
// Tiles: 256 weight rows x CN columns (2 CN B rows: hi and lo) per block of
// eight waves.  Four compute: wave w owns 32 RT weight rows and 64 columns, as
// RT x 2 tiles of v_mfma_f32_32x32x16_f16, hi and lo in sums of their own for
// the 256 x 64 tile, added at the end (the lo products then don't round the hi
// sum a second time in each step: error of a 250-frame codec decode against 64
// bits 1.93e-6 in one sum, 1.64e-6 in two, at the same time), in one sum for the
// 256 x 128 tile, whose registers hold no second.  Four load: a k-tile is 64 halves, 128 bytes of each of the 256 + 2 CN
// rows, brought to LDS by direct loads (global_load_lds_dwordx4, 1 KB per
// instruction = 8 rows) into a ring of DA weight stages and DB stages of B.
//
// What bounds it is power, then the matrix cores and the operands' way to them.
// Parts left out in a copy, per k-tile of the 256 x 64 tile (192 blocks): whole
// 1580 clocks, 0.94-1.01 us at 1.6 GHz; without the LDS reads more clocks at a
// higher clock, the same time; without the direct loads 0.74 us; the loads alone
// 0.51 us (43 bytes a clock and CU); the MFMAs alone 0.65 us, 1205 clocks for
// 1024 of issue.  A wave that issues a direct load beside its MFMAs holds them
// up by 39 clocks, and one wave issues a load every 70 clocks; hence loaders of
// their own, and four of them: QKV at 1024 columns took 97 us with the loads
// issued by the computing waves, 102 with one loader wave, 87 with four.  The
// 256 x 128 tile moves 64 KB for twice the MFMAs of the 256 x 64 tile's 48 KB
// and reads 8 fragments for 16 MFMAs, not 6 for 8: 1.41-1.50 us a k-tile, 1.5
// times the narrow one's.
// Issued rates in prompts: 1024 columns gate/up (18432 x 3072) 1.06 PFLOP/s, QKV
// 1.01; 256 columns 0.88 and 0.65; one 8192^3 f16 product of the vendor library
// reaches 1.18 on this card.
//
// A block works through k-tiles g0 .. g1 - 1 of one column tile's sequence
// g = mt nk + kt.  Two ways to cut it:
//  - K slices: one tile per block, K split in KS slices (S_out = KS);
//  - shares: every block an equal share of its column tile's sequence; S_out =
//    the most blocks a tile is split over (1 .. 8); for shapes with more tiles
//    than CUs, which would otherwise run in uneven rounds.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <type_traits>

namespace vx {

typedef _Float16 gm_h8 __attribute__((ext_vector_type(8)));
typedef float gm_f32x4 __attribute__((ext_vector_type(4)));
typedef float gm_f32x16 __attribute__((ext_vector_type(16)));

constexpr int GM_BM = 256;   // weight rows per tile
constexpr int GM_BN = 64;    // columns of the narrow tile, and of a compute wave
constexpr int GM_BK = 64;    // halves per k-tile
constexpr int GM_ROWB = 128; // bytes per LDS row (one k-tile of one row)

// s_waitcnt immediate for vmcnt(vm) with the other counters left open
constexpr int gm_vmcnt(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (15 << 8); }
constexpr int GM_LGKM0 = 0xC07F;  // lgkmcnt(0)

// LDS position of 16-byte chunk c of stage row R: c ^ ((R >> 1) & 7), so the
// 32 rows one fragment read touches spread over the banks
__device__ __forceinline__ int gm_key(int row) { return (row >> 1) & 7; }

__device__ __forceinline__ void gm_direct(const uint16_t *src, unsigned char *lds_row_block) {
  __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)lds_row_block, 16,
                                   0, 0);
}

// One tile shape: RT 32-row tiles and one of WC 64-column groups per compute
// wave, rings of DA weight stages and DB stages of B.
template <int RT_, int WC_, int DA_, int DB_>
struct GmShape {
  static constexpr int RT = RT_, WC = WC_, DA = DA_, DB = DB_;
  static constexpr int SUMS = RT == 2 ? 2 : 1;        // accumulators per tile: hi and lo, or one for both
  static constexpr int CN = GM_BN * WC;               // columns per tile
  static constexpr int ASTAGE = GM_BM * GM_ROWB;      // 32 KB
  static constexpr int BSTAGE = 2 * CN * GM_ROWB;     // 16 KB per 64 columns
  static constexpr int NA = GM_BM / 32, NB = 2 * CN / 32;  // direct loads per loader wave and stage
  static constexpr int LDS = DA * ASTAGE + DB * BSTAGE;
  static_assert(32 * RT * 4 / WC == GM_BM && DA == 3 && (DB == 2 || DB == 3), "tile");
};
using GmNarrow = GmShape<2, 1, 3, 3>;  // 256 x 64, 144 KB
using GmWide = GmShape<4, 2, 3, 2>;    // 256 x 128, 160 KB: the weights, which come from HBM, two k-tiles ahead

template <int SUMS, int RT>
__device__ __forceinline__ void gm_mfma(gm_f32x16 (&acc)[SUMS][RT][2], const gm_h8 (&fr)[RT + 4]) {
#pragma unroll
  for (int hl = 0; hl < 2; hl++)
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        acc[hl % SUMS][i][j] =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[i], fr[RT + 2 * hl + j], acc[hl % SUMS][i][j], 0, 0, 0);
}

// acc[.][i][j][e] is weight row 32 i + 8 (e / 4) + 4 h + e % 4 of the wave's,
// column 32 j + r: the sums added and written as C[col][m] with float4 stores
template <int SUMS, int RT>
__device__ __forceinline__ void gm_store(const gm_f32x16 (&acc)[SUMS][RT][2], float *cp, int ldc, bool zero) {
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      gm_f32x16 v = acc[0][i][j];
      if (SUMS == 2) v += acc[SUMS - 1][i][j];
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++)
        *(gm_f32x4 *)(cp + (size_t)j * 32 * ldc + i * 32 + 8 * g4) =
            zero ? gm_f32x4{0.f, 0.f, 0.f, 0.f} : gm_f32x4{v[4 * g4], v[4 * g4 + 1], v[4 * g4 + 2], v[4 * g4 + 3]};
    }
}

// KS > 0: block = K slice of one tile (K / 64 k-tiles in KS near-equal runs),
// C block = slice.  KS = 0: shares.  Block lb works on column tile
// c = lb % n_tiles, share j = lb / n_tiles: g in [j L, (j + 1) L).  A tile is
// split into the segments of the blocks whose shares overlap it; the segment
// of block j goes to C block j - j0(mt), j0(mt) = mt nk / L (its first block),
// and the block holding a tile's last segment writes zeros to the C blocks
// after it, up to the ns blocks the consumer reads.
// Needs M % 256 == 0, nt % 64 == 0, K % 64 == 0, KS <= K / 64.  Columns past nt
// (the last 256 x 128 tile of an odd multiple of 64) are computed from the
// rows that follow in B, which the caller's buffer holds, and not stored.
template <typename S>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_kernel(
    const uint16_t *__restrict__ W, int M, int K, const uint16_t *__restrict__ B, int ldb, size_t blo, int nt,
    float *__restrict__ C, int ldc, int Lshare, int ns, int ks) {
  constexpr int RT = S::RT, WC = S::WC;
  extern __shared__ __attribute__((aligned(16))) unsigned char gm_smem[];
  unsigned char *const a_ring = gm_smem, *const b_ring = gm_smem + S::DA * S::ASTAGE;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tiles = (nt + S::CN - 1) / S::CN, m_tiles = M / GM_BM, nk = K / GM_BK, total = m_tiles * nk;
  // this block's place in the list of work: the blocks b with b % 8 == x take
  // the x-th eighth (the first G % 8 eighths hold one more).  Workgroups are
  // dealt to the 8 XCDs round-robin (from a starting XCD that varies between
  // launches), so blocks with equal b % 8 share an XCD: the column tiles
  // sharing a weight tile run together and one L2 serves the re-reads.
  // (Without the grouping O at 320 columns, 60 tiles in 4 slices, took 28.5 us
  // against 23.)
  const int x = blockIdx.x & 7, G = gridDim.x;
  const int lb = x * (G >> 3) + min(x, G & 7) + (blockIdx.x >> 3);
  int c, j, g0, g1;
  if (ks > 0) {  // K slice j of tile (g0 / nk, c)
    const int tiles = m_tiles * n_tiles, tile = lb % tiles, mt = tile / n_tiles;
    j = lb / tiles;
    c = tile - mt * n_tiles;
    g0 = mt * nk + j * nk / ks;
    g1 = mt * nk + (j + 1) * nk / ks;
  } else {
    c = lb % n_tiles;
    j = lb / n_tiles;
    g0 = min(j * Lshare, total);
    g1 = min(g0 + Lshare, total);
    if (g0 >= g1) return;
  }
  const int last = g1 - 1;
  // Every wave passes one barrier before the first k-tile and one in each.  At
  // k-tile g's, k-tile g + 1 is in LDS and no wave reads k-tile g again.
  if (wave >= 4) {
    // loader wave l: its load k fills rows 32 k + 8 l + lane / 8 of a stage, at
    // position lane % 8, which holds chunk (lane % 8) ^ key(row)
    const int l = wave - 4, lrow = 8 * l + (lane >> 3), chunk = (lane & 7) ^ gm_key(lrow);
    const uint32_t aoff = (uint32_t)lrow * K + chunk * 8, boff = (uint32_t)lrow * ldb + chunk * 8;
    int a_mt = g0 / nk, a_kt = g0 - a_mt * nk, b_kt = a_kt, sa = 0, sb = 0;
    auto load_a = [&]() {  // the next weight stage
      const uint16_t *src = W + (size_t)a_mt * GM_BM * K + a_kt * GM_BK;
#pragma unroll
      for (int k = 0; k < S::NA; k++)
        gm_direct(src + (size_t)k * 32 * K + aoff, a_ring + sa * S::ASTAGE + (4 * k + l) * 1024);
      sa = sa + 1 == S::DA ? 0 : sa + 1;
      if (++a_kt == nk) {
        a_kt = 0;
        ++a_mt;
      }
    };
    auto load_b = [&]() {  // rows 0 .. CN - 1 hi, then lo
      const uint16_t *src = B + (size_t)c * S::CN * ldb + b_kt * GM_BK;
#pragma unroll
      for (int k = 0; k < S::NB; k++)
        gm_direct(src + (size_t)(k % (S::NB / 2)) * 32 * ldb + (k / (S::NB / 2)) * blo + boff,
                  b_ring + sb * S::BSTAGE + (4 * k + l) * 1024);
      sb = sb + 1 == S::DB ? 0 : sb + 1;
      if (++b_kt == nk) b_kt = 0;
    };
    constexpr int YOUNG = S::NA + (S::DB > 2 ? S::NB : 0);  // loads of k-tile g + 2 that may be in flight
    load_a();
    load_b();
    if (g0 + 1 <= last) {
      load_a();
      load_b();
    }
    if (g0 + 2 <= last) {
      load_a();
      if (S::DB > 2) load_b();
    }
    if (g0 + 2 <= last) __builtin_amdgcn_s_waitcnt(gm_vmcnt(S::NA + S::NB + YOUNG));
    else if (g0 + 1 <= last) __builtin_amdgcn_s_waitcnt(gm_vmcnt(S::NA + S::NB));
    else __builtin_amdgcn_s_waitcnt(gm_vmcnt(0));
    __builtin_amdgcn_s_barrier();
    for (int g = g0; g < g1; g++) {
      if (g + 2 <= last) __builtin_amdgcn_s_waitcnt(gm_vmcnt(YOUNG));
      else __builtin_amdgcn_s_waitcnt(gm_vmcnt(0));
      __builtin_amdgcn_s_barrier();
      if (g + S::DB <= last) load_b();
      if (g + S::DA <= last) load_a();
    }
    return;
  }
  const int r = lane & 31, h = lane >> 5, wr = wave / WC, wc = wave % WC;
  const size_t slot_stride = (size_t)nt * ldc;
  const int col0 = c * S::CN + wc * 64;
  const bool live = col0 < nt;
  float *cw = C + (size_t)(col0 + r) * ldc + wr * 32 * RT + 4 * h;
  gm_f32x16 acc[S::SUMS][RT][2];
  auto zero_acc = [&]() {
#pragma unroll
    for (int s = 0; s < S::SUMS; s++)
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int jj = 0; jj < 2; jj++)
#pragma unroll
          for (int e = 0; e < 16; e++) acc[s][i][jj][e] = 0.f;
  };
  zero_acc();
  // zeros for the C blocks past each tile whose last segment is this block's
  if (ks == 0 && live)
    for (int mt = g0 / nk; mt <= last / nk; mt++) {
      if ((mt + 1) * nk - 1 > last) break;  // the tile goes on in the next block
      for (int sl = j - mt * nk / Lshare + 1; sl < ns; sl++)
        gm_store(acc, cw + sl * slot_stride + mt * GM_BM, ldc, true);
    }
  // fragment f of step q: weight rows 32 RT wr + 32 f + r, B rows hi / lo
  // 64 wc + 32 j + r; every row's key is (r >> 1) & 7
  const int key = (r >> 1) & 7;
  const int ra = (wr * 32 * RT + r) * GM_ROWB, rb = (wc * 64 + r) * GM_ROWB;
  auto frag = [&](const unsigned char *pa, const unsigned char *pb, int q, int f) {
    const int pos = ((2 * q + h) ^ key) << 4;
    return f < RT ? *(const gm_h8 *)(pa + ra + f * 32 * GM_ROWB + pos)
                  : *(const gm_h8 *)(pb + rb + ((f - RT) >> 1) * S::CN * GM_ROWB + ((f - RT) & 1) * 32 * GM_ROWB + pos);
  };
  __builtin_amdgcn_s_barrier();
  gm_h8 f0[RT + 4], f1[RT + 4];
#pragma unroll
  for (int f = 0; f < RT + 4; f++) f0[f] = frag(a_ring, b_ring, 0, f);
  int c_mt = g0 / nk, c_kt = g0 - c_mt * nk;  // k-tile of iteration g
  int sa = 0, sb = 0;                         // its stages
  // MFMAs of `fr` with the reads of step q into `to`
  auto step = [&](const gm_h8 (&fr)[RT + 4], gm_h8 (&to)[RT + 4], int q) {
    const unsigned char *pa = a_ring + sa * S::ASTAGE, *pb = b_ring + sb * S::BSTAGE;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < RT + 4; f++) to[f] = frag(pa, pb, q, f);
    gm_mfma(acc, fr);
#pragma unroll
    for (int k = 0; k < RT + 4; k++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * RT - (RT + 4), 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int g = g0; g < g1; g++) {
    step(f0, f1, 1);
    step(f1, f0, 2);
    step(f0, f1, 3);
    __builtin_amdgcn_s_waitcnt(GM_LGKM0);
    __builtin_amdgcn_s_barrier();
    sa = sa + 1 == S::DA ? 0 : sa + 1;
    sb = sb + 1 == S::DB ? 0 : sb + 1;
    step(f1, f0, 0);  // the next k-tile's first fragments (past the last: unused)
    if (c_kt == nk - 1 || g == last) {
      const int slot = ks > 0 ? j : j - c_mt * nk / Lshare;  // this segment's C block
      if (live) gm_store(acc, cw + slot * slot_stride + c_mt * GM_BM, ldc, false);
      zero_acc();
    }
    if (++c_kt == nk) {
      c_kt = 0;
      ++c_mt;
    }
  }
}

// Thin grid, for chunks of few columns: the product is then bound
// by the weight stream (two flops per weight byte and column), so what
// matters is bytes in flight on every CU and few bytes of everything else.
// Block (x, s, z): BM = 32 RT weight rows, K slice s of gridDim.y, columns
// z NT .. + NT (all of them, up to GT_MAXN).  A k-tile's BM + 2 NT rows are staged as above (ring of S stages,
// 48-72 KB, so two or three blocks share a CU and one's barriers run under
// the others' loads), but the four waves split the k-tile's 64 halves, 16
// each, instead of its rows: every staged byte is read from LDS once (rows
// split over waves would read the B rows four times), and each wave holds the
// block's whole BM x 2 NT product, RT x NT / 16 tiles of
// v_mfma_f32_32x32x16_f16 whose columns are the hi rows, then the lo rows.
// At the end the four waves' hi and lo sums are added through LDS in a fixed
// order and only the live columns col < n are written.  NTW: the weight loads
// carry the non-temporal hint, as each weight is read by one block only.
// Weights cycled from HBM, all of M x K = 18432 x 3072 (113 MB): 16 columns
// 21.6 us (23.8 without the hint), 32 columns 26.7 us, where the tiled grid
// took 54 us (at its 128 columns) and the decode GEMV 18.4 us for one;
// 3072 x 9216: 11.7 and 14.0 us against 25; 1024 x 1024: 2.6 and 2.8 us
// against 6.5.
constexpr int GT_MAXN = 64;
template <int RT, int NT>
struct GtShape {
  static constexpr int BM = 32 * RT;
  static constexpr int STAGE = (BM + 2 * NT) * GM_ROWB;
  static constexpr int LOADS = (BM + 2 * NT) / 32;  // direct loads per wave per k-tile
  static constexpr int CT = NT / 16;                // 32-column tiles of the 2 NT B rows
  static constexpr int S = NT == 16 ? (RT == 1 ? 6 : 4) : NT == 32 && RT == 1 ? 4 : 3;
  static constexpr int RW = 36;                     // floats per reduction row: 32 weight rows + pad
  static constexpr int RED = 4 * 2 * NT * RW * 4;   // reduction area in bytes
  static constexpr int LDS = S * STAGE > RED ? S * STAGE : RED;
};

// waits until at most min(younger, S - 2) k-tiles of L loads are in flight
template <int S, int L>
__device__ __forceinline__ void gt_wait(int younger) {
  if constexpr (S > 2) {
    if (younger >= S - 2)
      __builtin_amdgcn_s_waitcnt(gm_vmcnt(L * (S - 2)));
    else
      gt_wait<S - 1, L>(younger);
  } else {
    __builtin_amdgcn_s_waitcnt(gm_vmcnt(0));
  }
}

template <bool NTW>
__device__ __forceinline__ void gt_direct(const uint16_t *src, unsigned char *lds_row_block) {
  __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)lds_row_block, 16, 0,
                                   NTW ? 2 : 0);
}

template <int RT, int NT, bool NTW>
__global__ __launch_bounds__(256) void gemm_thin_kernel(const uint16_t *__restrict__ W, int K,
                                                        const uint16_t *__restrict__ B, int ldb, size_t blo,
                                                        int n, float *__restrict__ C, int ldc) {
  using G = GtShape<RT, NT>;
  constexpr int S = G::S;
  extern __shared__ __attribute__((aligned(16))) unsigned char gm_smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.x * G::BM, nk = K / GM_BK, col0 = blockIdx.z * NT;
  B += (size_t)col0 * ldb;
  const int k0 = (int)(blockIdx.y * nk / gridDim.y), cnt = (int)((blockIdx.y + 1) * nk / gridDim.y) - k0;
  // direct load i of this wave fills stage rows 8 (4 i + wave) .. + 8: weight
  // rows for i < RT, then the B rows (hi, lo)
  const uint16_t *src[G::LOADS];
#pragma unroll
  for (int i = 0; i < G::LOADS; i++) {
    const int row = 8 * (4 * i + wave) + (lane >> 3), chunk = (lane & 7) ^ gm_key(row);
    const int br = row - G::BM, hl = br >= NT ? 1 : 0;  // i >= RT
    src[i] = (i < RT ? W + (size_t)(m0 + row) * K : B + hl * blo + (size_t)(br - hl * NT) * ldb) + k0 * GM_BK + chunk * 8;
  }
  auto issue = [&](int stage) {
#pragma unroll
    for (int i = 0; i < G::LOADS; i++) {
      unsigned char *dst = gm_smem + stage * G::STAGE + (4 * i + wave) * 1024;
      if (i < RT) gt_direct<NTW>(src[i], dst);
      else gt_direct<false>(src[i], dst);
      src[i] += GM_BK;
    }
  };
  gm_f32x16 acc[RT][G::CT];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < G::CT; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
#pragma unroll
  for (int s = 0; s < S - 1; s++)
    if (s < cnt) issue(s);
  const int c = 2 * wave + h;  // this lane's 16-byte chunk of every row
  int stage = 0, fill = S - 1;
  for (int t = 0; t < cnt; t++) {
    gt_wait<S, G::LOADS>(cnt - 1 - t);
    // every wave's part of k-tile t is in, and every wave has read k-tile
    // t - 1, whose stage k-tile t + S - 1 takes
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + S - 1 < cnt) issue(fill);
    const unsigned char *st = gm_smem + stage * G::STAGE;
    gm_h8 a[RT], b[G::CT];
#pragma unroll
    for (int i = 0; i < RT; i++) {
      const int row = 32 * i + r;
      a[i] = *(const gm_h8 *)(st + row * GM_ROWB + ((c ^ gm_key(row)) << 4));
    }
#pragma unroll
    for (int j = 0; j < G::CT; j++) {
      const int row = G::BM + 32 * j + r;
      b[j] = *(const gm_h8 *)(st + row * GM_ROWB + ((c ^ gm_key(row)) << 4));
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int j = 0; j < G::CT; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_waitcnt(GM_LGKM0);  // this wave's reads are done before the next barrier
    stage = stage + 1 == S ? 0 : stage + 1;
    fill = fill + 1 == S ? 0 : fill + 1;
  }
  float *red = (float *)gm_smem;
  C += ((size_t)blockIdx.y * gridDim.z * NT + col0) * ldc;
#pragma unroll
  for (int i = 0; i < RT; i++) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < G::CT; j++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++)
        *(gm_f32x4 *)(red + (wave * 2 * NT + 32 * j + r) * G::RW + 8 * g4 + 4 * h) =
            gm_f32x4{acc[i][j][4 * g4], acc[i][j][4 * g4 + 1], acc[i][j][4 * g4 + 2], acc[i][j][4 * g4 + 3]};
    __syncthreads();
    for (int o = tid; o < NT * 8; o += 256) {
      const int col = o >> 3, m = 4 * (o & 7);
      if (col0 + col < n) {
        gm_f32x4 v = *(const gm_f32x4 *)(red + col * G::RW + m);
#pragma unroll
        for (int w = 1; w < 4; w++) v += *(const gm_f32x4 *)(red + (w * 2 * NT + col) * G::RW + m);
#pragma unroll
        for (int w = 0; w < 4; w++) v += *(const gm_f32x4 *)(red + (w * 2 * NT + NT + col) * G::RW + m);
        *(gm_f32x4 *)(C + (size_t)col * ldc + m0 + 32 * i + m) = v;
      }
    }
  }
}

// ---------------------------------------------------------------- host side
// columns (hi, and as many lo) of a chunk of n tokens
inline int gm_cols(int n) { return n <= 16 ? 16 : n <= 32 ? 32 : (n + GM_BN - 1) / GM_BN * GM_BN; }

struct GemmPlan {
  int thin = 0;       // thin grid: 32-row tiles per block (0: the tiled grid)
  bool wide = false;  // 256 x 128 tiles, else 256 x 64
  int ks = 1;         // K slices (0: shares)
  int grid = 0;       // tiled grid: blocks
  int share = 0;      // k-tiles per block
  int slices = 1;     // C blocks the consumer sums
};

// Calls f(std::integral_constant<int, NS>) for the slice counts a plan can
// produce (ns in 1 .. 8), so the consumer kernels sum a compile-time number
// of slices; false for any other count.
template <typename F>
inline bool gm_with_slices(int ns, F &&f) {
  switch (ns) {
    case 1: f(std::integral_constant<int, 1>{}); return true;
    case 2: f(std::integral_constant<int, 2>{}); return true;
    case 3: f(std::integral_constant<int, 3>{}); return true;
    case 4: f(std::integral_constant<int, 4>{}); return true;
    case 5: f(std::integral_constant<int, 5>{}); return true;
    case 6: f(std::integral_constant<int, 6>{}); return true;
    case 7: f(std::integral_constant<int, 7>{}); return true;
    case 8: f(std::integral_constant<int, 8>{}); return true;
    default: return false;
  }
}

// Consumer slice count of shares of L k-tiles: the most segments any tile is
// cut into (0: more than 8)
inline int gemm_share_slices(int m_tiles, int nk, int L) {
  int most = 1;
  for (int mt = 0; mt < m_tiles; mt++) {
    const int segs = (mt * nk + nk - 1) / L - mt * nk / L + 1;
    if (segs > most) most = segs;
  }
  return most <= 8 ? most : 0;
}

// Thin grid: 64-row blocks where M has enough of them for KS <= 8 slices to
// give every CU three blocks, else 32-row blocks.  KS then is the largest
// power of two that keeps the grid within 4.5 blocks per CU (1.5 rounds of
// three) and leaves a block at least 4 k-tiles (2 while the grid is smaller
// than the device): more slices hide more latency, but each costs its share
// of the pipeline's fill and of C.
inline GemmPlan gemm_thin_plan(int M, int K, int nt, int cus) {
  GemmPlan p;
  const int nk = K / GM_BK;
  p.thin = nt >= 64 || M / 64 * 8 >= 3 * cus ? 2 : 1;
  const int blocks = M / (32 * p.thin) * (nt > GT_MAXN ? nt / GT_MAXN : 1);
  while (p.ks < 8 && blocks * p.ks * 2 * 2 <= 9 * cus &&
         nk / (p.ks * 2) >= (blocks * p.ks < cus ? 2 : 4))
    p.ks *= 2;
  p.slices = p.ks;
  return p;
}

// The tiled grid's plan, by estimated time.  A block spends 0.8 us on a k-tile
// of 256 x 64 and 1.2 us on one of 256 x 128, or the device does 300 or 180 of
// them per us (power), whichever takes longer; a slice of C is written and
// read again at 5 TB/s.  Candidates, for both tiles: one tile per block with K
// in 1 .. 8 slices while that is at most one block per CU; with more tiles
// than CUs, equal shares, or shares of whole tiles (no tile is cut: one
// slice).  c_cap: floats that C holds.
// The figures are a fit to timed plans (GEMM plus a reader of C, a copy of 200 MB
// before each, as other kernels run between a prompt's products).  Of 831 plans
// of 83 shapes (K 896 .. 9216, M 1024 .. 18432, 64 .. 1024 columns) the one
// picked is 0.17% slower than the best of its shape on average, 4.4% at most.
inline GemmPlan gemm_tiled_plan(int M, int K, int nt, int cus, size_t c_cap) {
  GemmPlan best;
  double best_us = -1;
  const int m_tiles = M / GM_BM, nk = K / GM_BK;
  for (int wide = 0; wide < 2; wide++) {
    const int n_tiles = (nt + (wide ? 127 : 63)) / (wide ? 128 : 64), tiles = m_tiles * n_tiles;
    auto consider = [&](int ks, int grid, int share, int slices) {
      if (slices < 1 || slices > 8 || (size_t)slices * nt * M > c_cap) return;
      const int per_block = ks ? (nk + ks - 1) / ks : share;
      const double us = std::max(per_block * (wide ? 1.2 : 0.8), (double)tiles * nk / (wide ? 180 : 300)) +
                        slices * (8.0 * nt * M / 5e6);
      if (best_us < 0 || us < best_us) {
        best_us = us;
        best.wide = wide;
        best.ks = ks;
        best.grid = grid;
        best.share = share;
        best.slices = slices;
      }
    };
    if (tiles <= cus) {
      for (int ks = 1; ks <= 8 && tiles * ks <= cus && (ks == 1 || nk / ks >= 2); ks++)
        consider(ks, tiles * ks, 0, ks);
    } else if (n_tiles <= cus) {
      const int per_col = cus / n_tiles, even = (m_tiles * nk + per_col - 1) / per_col;
      const int whole = (m_tiles + per_col - 1) / per_col;  // tiles
      consider(0, per_col * n_tiles, even, gemm_share_slices(m_tiles, nk, even));
      consider(0, (m_tiles + whole - 1) / whole * n_tiles, whole * nk, 1);
    }
  }
  return best;
}

// cus: the device's compute units (8 XCDs).  Shapes must satisfy
// M % 256 == 0, K % 64 == 0, nt = gm_cols(n).  From 64 columns on the thin grid
// is the faster one for outputs of up to 2^17 elements, whose few 256-row
// tiles leave the device idle (GEMM and a reader of C, us, thin / tiled: 2048 x
// 2048 at 64 columns 11.2 / 13.0, 1024 x 4096 at 128 12.5 / 15.7, 256 x 7168 at
// 256 13.7 / 19.2), and about equal or slower past that (1024 x 1024 at 192
// 12.4 / 12.0, 3072 x 1024 at 64 12.5 / 12.4, at 192 17.4 / 15.1).
inline GemmPlan gemm_plan(int M, int K, int nt, int cus, size_t c_cap) {
  if (nt < GT_MAXN || (size_t)M * nt <= (size_t)1 << 17) return gemm_thin_plan(M, K, nt, cus);
  return gemm_tiled_plan(M, K, nt, cus, c_cap);
}

// f(kernel, LDS bytes) for every thin kernel a plan can name
template <typename F>
inline void gm_with_thin(int rt, int nt, bool ntw, F &&f) {
  auto pick = [&](auto RT, auto NT) {
    using G = GtShape<RT, NT>;
    if (ntw) f(gemm_thin_kernel<RT, NT, true>, G::LDS);
    else f(gemm_thin_kernel<RT, NT, false>, G::LDS);
  };
  std::integral_constant<int, 1> one;
  std::integral_constant<int, 2> two;
  if (nt == 16) rt == 1 ? pick(one, std::integral_constant<int, 16>{}) : pick(two, std::integral_constant<int, 16>{});
  else if (nt == 32) rt == 1 ? pick(one, std::integral_constant<int, 32>{}) : pick(two, std::integral_constant<int, 32>{});
  else if (nt == 64) pick(two, std::integral_constant<int, 64>{});
}

// the kernels' dynamic LDS: 144 and 160 KB for the tiled grid, 48 or 72 KB
// for the thin one
inline hipError_t gemm_setup() {
  hipError_t e = hipFuncSetAttribute((const void *)gemm_kernel<GmNarrow>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     GmNarrow::LDS);
  if (e == hipSuccess)
    e = hipFuncSetAttribute((const void *)gemm_kernel<GmWide>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            GmWide::LDS);
  for (int rt = 1; rt <= 2; rt++)
    for (int nt : {16, 32, 64})
      for (bool ntw : {false, true})
        gm_with_thin(rt, nt, ntw, [&](auto kernel, int lds) {
          if (e == hipSuccess)
            e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        });
  return e;
}

// Whether the thin grid streams a matrix's weights with the non-temporal hint:
// from 16 MiB on, the prompt's four matrices and the codec's gate/up (8192 x
// 1024).  A decode of few frames reads the codec's 298 MB of weights once; with
// gate/up, a third of them, streamed past the 256 MB last-level cache, more of
// the rest is found there by the next decode.  Decodes of 13 frames one after
// the other take 436 us, with a line above gate/up 450, without a line (all
// matrices hinted) 450, at 8 MiB 446; behind other work 450, 450, 453 and 454;
// decodes of 1, 4 and 32 frames and prompts of 9 to 32 tokens are within 3% on
// every line.
inline bool gemm_thin_hint(int M, int K) { return (size_t)M * K * 2 >= (size_t)16 << 20; }

// n: the live columns of the nt (the thin grid writes only those)
inline void gemm_launch(const GemmPlan &p, hipStream_t st, const uint16_t *W, int M, int K, const uint16_t *B,
                        int ldb, size_t blo, int nt, int n, float *C) {
  if (p.thin)
    gm_with_thin(p.thin, std::min(nt, GT_MAXN), gemm_thin_hint(M, K), [&](auto kernel, int lds) {
      hipLaunchKernelGGL(kernel, dim3(M / (32 * p.thin), p.ks, std::max(nt / GT_MAXN, 1)), dim3(256), lds, st, W, K,
                         B, ldb, blo, n, C, M);
    });
  else if (p.wide)
    hipLaunchKernelGGL(gemm_kernel<GmWide>, dim3(p.grid), dim3(512), GmWide::LDS, st, W, M, K, B, ldb, blo, nt, C, M,
                       p.share, p.slices, p.ks);
  else
    hipLaunchKernelGGL(gemm_kernel<GmNarrow>, dim3(p.grid), dim3(512), GmNarrow::LDS, st, W, M, K, B, ldb, blo, nt, C,
                       M, p.share, p.slices, p.ks);
}

}  // namespace vx
