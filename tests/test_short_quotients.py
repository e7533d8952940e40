"""The kernels' short quotients (no exponent scaling: linear_small.hip's 127 / amax
and amax / 127, ovh_common.h's SiLU quotient) are the IEEE ones over the ranges they
are used in, whichever way the hardware's reciprocal rounds."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_short_quotients_are_correctly_rounded(tmp_path):
    exe = str(tmp_path / "short_quotients")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-mfma", "-ffp-contract=off",
                    os.path.join(HERE, "short_quotients.cpp"), "-o", exe], check=True, timeout=120)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120).stdout
    assert out.splitlines() == ["quantiser 0", "silu 0"]
