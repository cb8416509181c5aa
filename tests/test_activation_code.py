"""What the compiler makes of the activations' exp (csrc/common.h): values inside its range pay nothing for the ends."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "layered-prefill_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

_KERNEL = """
#include <hip/hip_runtime.h>
#include "common.h"
__global__ void act(float* v, float alpha, float limit) {
  const int i = 2 * threadIdx.x;
  v[i] = %s;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("activation,clamps", [("moe_silu(v[i])", 0), ("moe_swigluoai(v[i], v[i + 1], alpha, limit)", 3)])
def test_values_inside_the_range_pay_nothing_for_its_ends(tmp_path, activation, clamps):
    (tmp_path / "act.hip").write_text(_KERNEL % activation)
    subprocess.check_call([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-ffp-contract=off",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, "act.hip", "-o", "act.s"],
                          cwd=tmp_path, timeout=300)
    code = (tmp_path / "act.s").read_text()
    blocks = re.split(r"^\.LBB\w+:.*$|^\s*s_(?:c?branch\w*|endpgm).*$", code, flags=re.M)
    exps = [b for b in blocks if "v_rndne_f32" in b]
    assert len(exps) == 2   # (a wavefront inside the range, and one that is not)
    assert len(re.findall(r"^\s*v_cndmask", code, re.M)) <= clamps
