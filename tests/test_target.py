"""The reductions order their partial sums by what gfx950's stores do, not by the
language's memory model alone: for another target they do not compile."""
import os
import shutil
import subprocess

import pytest

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qphix_amd", "csrc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("arch,builds", [("gfx950", True), ("gfx942", False)])
def test_reductions_compile_for_gfx950_only(arch, builds):
    r = subprocess.run([HIPCC, f"--offload-arch={arch}", "--cuda-device-only", "-std=c++17", "-fsyntax-only", "-x", "hip",
                        os.path.join(CSRC, "blas.hip")], capture_output=True, text=True, timeout=300)
    assert (r.returncode == 0) == builds, r.stderr
    assert builds or "finish_reduction relies on gfx950" in r.stderr
