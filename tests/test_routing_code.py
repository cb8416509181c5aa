"""What the compiler makes of a row's routing (csrc/routing_device.h): K winners out of registers, nothing read back."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "layered-prefill_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# A row's scores out of numbers that the kernel has, so that any vector load is one of the winners.
_KERNELS = """
#include <hip/hip_runtime.h>
#include "routing_device.h"
template <int E>
__global__ void route(float* w, int32_t* ids, int32_t* tei, float a, int T, int K, int renormalize) {
  constexpr int TPR = Pow2Geom<E>::kTpr;
  float v[Pow2Geom<E>::kVpt];
  for (int i = 0; i < Pow2Geom<E>::kVpt; ++i) v[i] = a * static_cast<float>(threadIdx.x * 7 + i * i);
  const int row = threadIdx.x / TPR;
  route_row<E>(v, threadIdx.x % TPR, row, row < T, w, ids, tei, T, K, renormalize);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_winners_are_not_read_back(tmp_path):
    sizes = (1, 2, 4, 8, 16, 32, 64, 128, 256)
    (tmp_path / "route.hip").write_text(_KERNELS + "".join(
        f"template __global__ void route<{E}>(float*, int32_t*, int32_t*, float, int, int, int);\n" for E in sizes))
    subprocess.check_call([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-ffp-contract=off",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, "route.hip", "-o", "route.s"],
                          cwd=tmp_path, timeout=300)
    code = (tmp_path / "route.s").read_text()
    assert code.count("global_store_dword") >= 3 * len(sizes)
    assert re.findall(r"^\s*((?:global|flat|buffer|scratch)_load\w*)", code, re.M) == []
