"""The kernels' outcode (rf_math.hpp) has the bits of the six plane distances'
signs, special values included (host build of the same header)."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_outcode_is_the_sign_of_every_plane_distance():
    src = os.path.join(ROOT, "tests", "native", "outcode_check.cpp")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "outcode_check")
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-ffp-contract=off", "-x", "c++",
                               "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", src, "-o", exe])
        out = subprocess.run([exe], capture_output=True, text=True)
    total, bad = (int(x) for x in out.stdout.split())
    assert total > 4000000
    assert bad == 0, out.stdout
