"""The host copies by several threads (rf_copy.cpp) against memcpy, row by row
(host build of the same source)."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_of_many_shapes_from_several_callers():
    src = os.path.join(ROOT, "tests", "native", "copy_check.cpp")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "copy_check")
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__",
                               "-I/opt/rocm/include", src, "-o", exe, "-lpthread"])
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    total, bad = (int(x) for x in out.stdout.split())
    assert total == 1440 and bad == 0, out.stdout
