"""Barriers of the weight-gradient kernels: a wave waits for its own LDS
accesses right before each, also where the compiler does not unroll the loop
over the waves.  (A barrier at the head of a loop whose last LDS store is at
its end lost that wait to the compiler, which let a wave add to sums that the
wave before had not stored yet.)  Read in the assembly of this source."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "primal-dual-toolbox_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("flags", [[], ["-fno-unroll-loops"]])
def test_weight_gradient_barriers_wait_for_lds(tmp_path, flags):
    out = str(tmp_path / "cnn.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, *flags,
                    "--cuda-device-only", "-S", os.path.join(CSRC, "pdt_cnn.hip"), "-o", out],
                   check=True, capture_output=True)
    kernels = re.findall(r"^(_ZN\S*wgrad(?:32|_in)_kernel\S*):(.*?)s_endpgm", open(out).read(), re.M | re.S)
    assert len(kernels) == 3
    for name, body in kernels:
        lines = [t for t in (x.split(";")[0].strip() for x in body.splitlines()) if t]
        at = [i for i, t in enumerate(lines) if t == "s_barrier"]
        assert len(at) >= 2, name
        for i in at:
            assert lines[i - 1].startswith("s_waitcnt") and "lgkmcnt(0)" in lines[i - 1], (name, lines[i - 3:i + 1])
