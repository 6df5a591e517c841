"""The arithmetic of a draw on the CPU: the logarithm, root and quotient that
csrc/sn_device.h forms itself, compiled for the host (tests/draw_arithmetic.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# what the kernels' header takes from the HIP headers on the device
HIP = """#pragma once
#define __device__
#define __host__
#define __forceinline__ inline
"""


def test_logarithm_root_and_quotient_of_a_draw(tmp_path):
    """ln u within the 0.59 ulp that the header states; the root and the
    quotient are the rounded ones."""
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    exe = tmp_path / "draw_arithmetic"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", f"-I{tmp_path}",
                           "-I" + os.path.join(ROOT, "starrynight_amd", "csrc"), "-o", str(exe),
                           os.path.join(ROOT, "tests", "draw_arithmetic.cpp")])
    ulps, roots, quotients, limits = subprocess.check_output([str(exe)], text=True).split()
    assert float(ulps) <= 0.59
    assert (roots, quotients, limits) == ("0", "0", "1")
