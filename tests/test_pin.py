"""rf_render's pinned staging where pinned memory runs out (rf_pin.cpp; host build
of the same source over an allocator that fails)."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failed_growth_of_pinned_memory():
    src = os.path.join(ROOT, "tests", "native", "pin_check.cpp")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "pin_check")
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__",
                               "-I/opt/rocm/include", src, "-o", exe])
        out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    checks, bad = (int(x) for x in out.stdout.split()[-2:])
    assert checks == 10 and bad == 0, out.stdout
