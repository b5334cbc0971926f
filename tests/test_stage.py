"""The staging of a call's operands and results (vx_stage.h) on the CPU, with
the HIP calls it makes counted: a call that returns before finish(), as on an
error, has waited for the stream when its Stage is gone; one that finishes waits
once; results reach the caller's memory at finish() and not before."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <hip/hip_runtime.h>
static int syncs, launches, copies;
static hipError_t sync_rc, copy_rc, last_rc;
#define hipStreamSynchronize(s) ((void)(s), syncs++, sync_rc)
#define hipMemcpyAsync(dst, src, n, kind, s) ((void)(dst), (void)(src), (void)(s), copies++, copy_rc)
#define hipGetLastError() (last_rc)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) (launches++)
#include "vx_stage.h"
#include <cstdio>
#include <vector>
using namespace vx;
static int bad;
#define WANT(c) (void)((c) || (printf("line %d: %s\n", __LINE__, #c), bad++))
static std::vector<unsigned char> mem(2 * STAGE_BYTES);
alignas(16) static unsigned char dev[64];
static Stage stage() { syncs = launches = copies = 0; return Stage(nullptr, mem.data(), mem.data()); }
int main() {
  std::vector<unsigned char> big(STAGE_BYTES + 4);
  unsigned src = 7, dst = 0;
  { Stage s = stage(); }
  WANT(syncs == 0);                                      // nothing staged: nothing to wait for
  { Stage s = stage(); WANT(s.in(dev, &src, 4) == hipSuccess && launches == 1 && mem[0] == 7); }
  WANT(syncs == 1);                                      // returned before finish()
  { Stage s = stage(); WANT(s.out(&dst, dev, 4) == hipSuccess); }
  WANT(syncs == 1 && dst == 0);
  { Stage s = stage(); s.hold(); }
  WANT(syncs == 1);
  copy_rc = hipErrorInvalidValue;                        // a copy past the staging size that fails
  { Stage s = stage(); WANT(s.in(dev, &src, 4) == hipSuccess && s.in(dev, big.data(), big.size()) != hipSuccess); }
  WANT(syncs == 1 && copies == 1);
  copy_rc = hipSuccess;
  last_rc = hipErrorInvalidConfiguration;                // a launch of the call that failed
  { Stage s = stage(); WANT(s.in(dev, &src, 4) == hipSuccess && s.finish() != hipSuccess && syncs == 0); }
  WANT(syncs == 1);
  last_rc = hipSuccess;
  {
    Stage s = stage();
    WANT(s.in(dev, &src, 4) == hipSuccess && s.out(&dst, dev, 4) == hipSuccess && syncs == 0);
    mem[STAGE_BYTES] = 9;                                // what the copy kernel would have brought
    WANT(dst == 0 && s.finish() == hipSuccess && dst == 9);
  }
  WANT(syncs == 1);                                      // finish() waited, the destructor need not
  {
    Stage s = stage();                                   // operands past the fourth, odd ones and unaligned ones go by copy
    for (int i = 0; i < 5; i++) WANT(s.out(&dst, dev, 4) == hipSuccess);
    WANT(launches == 4 && copies == 1);
    WANT(s.in(dev, &src, 3) == hipSuccess && s.out(&dst, dev + 4, 4) == hipSuccess && copies == 3 && launches == 4);
  }
  WANT(syncs == 1);
  return bad != 0;
}
"""


def test_stage_waits(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    src, exe = tmp_path / "stage.hip", tmp_path / "stage"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "webgpu-voxtral_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
