"""Build-time parameters that the kernels cannot work with are refused by the compiler.

The narrow mixed pass 1 finishes its tiles in waves 0 to 3 and stores (alpha, beta) for pass 2 from
wave 4, so a work-group of four waves would leave pass 2 with old values."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("waves, accepted", [(4, False), (5, True), (8, True), (17, False)])
def test_waves_of_the_narrow_passes(waves, accepted):
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "--cuda-device-only",
                        "-DKIN_NW=%d" % waves, "-I", os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "ggbtddft_amd", "csrc", "ggbtd.hip")],
                       capture_output=True, text=True, timeout=300)
    assert (r.returncode == 0) == accepted, r.stderr[-2000:]
    assert accepted or "waves per narrow work-group" in r.stderr
