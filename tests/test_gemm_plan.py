"""The GEMM plans (vx_gemm.h, gemm_plan) on the CPU: for every product shape of
the prefill and the codec and chunk lengths up to 1024, the blocks that the
kernels derive from a plan, by the same index arithmetic restated here, cover
each (row tile, column tile, k-tile) once, write C blocks below the count the
consumer sums, leave none of those unwritten, and fit C.  Which weights stream
with the non-temporal hint, and which plans the GPU tests of long prompts and
decodes run."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "vx_gemm.h"
#include <cstdio>
#include <vector>
using namespace vx;
static int check(int M, int K, int n, int cus, size_t cap) {
  const int nt = gm_cols(n), nk = K / GM_BK;
  const GemmPlan p = gemm_plan(M, K, nt, cus, cap);
  if (nt < n || p.slices < 1 || p.slices > 8 || (size_t)p.slices * nt * M > cap) return 1;
  if (p.thin) {  // block (x, s, z): 32 thin rows, k-tiles s nk / ks .., columns z NT ..
    const int NT = nt < GT_MAXN ? nt : GT_MAXN, BM = 32 * p.thin, GX = M / BM, GZ = nt / GT_MAXN > 1 ? nt / GT_MAXN : 1;
    for (bool hint : {false, true}) {
      bool have = false;
      gm_with_thin(p.thin, NT, hint, [&](auto, int lds) { have = lds > 0 && lds <= 160 * 1024; });
      if (!have) return 8;
    }
    std::vector<char> seen((size_t)(M / 32) * (nt / 16) * nk, 0);  // 32 rows x 16 columns x k-tile
    for (int bx = 0; bx < GX; bx++)
      for (int s = 0; s < p.ks; s++)
        for (int z = 0; z < GZ; z++) {
          const int k0 = s * nk / p.ks, k1 = (s + 1) * nk / p.ks;
          if (k0 >= k1) return 9;
          for (int m = bx * BM; m < bx * BM + BM; m += 32)
            for (int c = z * NT; c < z * NT + NT; c += 16)
              for (int k = k0; k < k1; k++) {
                if (m >= M || c >= nt) return 10;
                seen[((size_t)(m / 32) * (nt / 16) + c / 16) * nk + k]++;
              }
        }
    for (char v : seen)
      if (v != 1) return 11;
    return p.ks != p.slices;  // block (., s, .) writes C block s of ks
  }
  const int CN = p.wide ? GmWide::CN : GmNarrow::CN, n_tiles = (nt + CN - 1) / CN, m_tiles = M / GM_BM;
  if (nt % 64) return 2;
  std::vector<char> seen((size_t)m_tiles * n_tiles * nk, 0);
  std::vector<unsigned> wrote((size_t)m_tiles * n_tiles, 0);  // C blocks of a tile, as bits
  std::vector<char> place(p.grid, 0);
  for (int b = 0; b < p.grid; b++) {
    const int x = b & 7, G = p.grid, lb = x * (G >> 3) + std::min(x, G & 7) + (b >> 3);
    if (lb < 0 || lb >= G || place[lb]++) return 3;
    int c, j, g0, g1;
    if (p.ks > 0) {
      const int tiles = m_tiles * n_tiles, tile = lb % tiles, mt = tile / n_tiles;
      j = lb / tiles, c = tile - mt * n_tiles;
      g0 = mt * nk + j * nk / p.ks, g1 = mt * nk + (j + 1) * nk / p.ks;
      if (j >= p.ks || g0 >= g1) return 4;
    } else {
      c = lb % n_tiles, j = lb / n_tiles;
      g0 = std::min(j * p.share, m_tiles * nk), g1 = std::min(g0 + p.share, m_tiles * nk);
      if (g0 >= g1) continue;
    }
    for (int g = g0; g < g1; g++) {
      const int mt = g / nk, slot = p.ks > 0 ? j : j - mt * nk / p.share;
      if (seen[((size_t)mt * n_tiles + c) * nk + g % nk]++ || slot < 0 || slot >= p.slices) return 5;
      wrote[(size_t)mt * n_tiles + c] |= 1u << slot;
      if (p.ks == 0 && g % nk == nk - 1)  // the tile's last segment: zeros to the C blocks after it
        for (int sl = slot + 1; sl < p.slices; sl++) wrote[(size_t)mt * n_tiles + c] |= 1u << sl;
    }
  }
  for (char s : seen)
    if (s != 1) return 6;
  for (unsigned w : wrote)
    if (w != (1u << p.slices) - 1) return 7;
  return 0;
}
int main() {
  const int pf[][2] = {{6144, 3072}, {3072, 4096}, {18432, 3072}, {3072, 9216}};
  const int cx[][2] = {{1024, 896}, {3072, 1024}, {1024, 1024}, {8192, 1024}, {1024, 4096}, {2048, 2048}, {256, 7168}};
  int bad = 0;
  auto all = [&](int M, int K, size_t cap) {
    for (int cus : {256, 64})
      for (int n = 1; n <= 1024; n += n < 136 ? 1 : 29)
        if (int rc = check(M, K, n, cus, cap)) printf("M %d K %d n %d cus %d: %d\n", M, K, n, cus, rc), bad++;
    if (int rc = check(M, K, 1024, 256, cap)) printf("M %d K %d n 1024: %d\n", M, K, rc), bad++;
  };
  for (auto &s : pf) all(s[0], s[1], (size_t)2048 * 18432);
  for (auto &s : cx) all(s[0], s[1], (size_t)2048 * 8192);
  // streamed past the caches: the prompt's matrices and the codec's gate/up, no other of the codec's
  for (auto &s : pf) bad += !gemm_thin_hint(s[0], s[1]);
  for (auto &s : cx) bad += gemm_thin_hint(s[0], s[1]) != (s[0] == 8192);
  // the plans that GPU tests of 700 and 1030 tokens and of 150 frames run: whole-tile shares of
  // 256 x 128 tiles, at an odd multiple of 64 columns too, and the 256 x 128 tile in the codec
  for (int n : {700, 1024}) {
    const GemmPlan p = gemm_plan(18432, 3072, gm_cols(n), 256, (size_t)2048 * 18432);
    bad += !p.wide || p.ks != 0 || p.slices != 1;
  }
  bad += gm_cols(700) % 128 != 64 || !gemm_plan(8192, 1024, 1024, 256, (size_t)2048 * 8192).wide;
  return bad != 0;
}
"""


def test_plans_cover_every_shape(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    src, exe = tmp_path / "plan.hip", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I",
                    os.path.join(ROOT, "webgpu-voxtral_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
