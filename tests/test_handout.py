"""The serving loop's hand-over of read-back space from rf_serve_poll to its
worker (rf_handout.hpp; host build of the same header): no wake-up is lost."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_returned_readback_space_wakes_the_worker():
    src = os.path.join(ROOT, "tests", "native", "handout_check.cpp")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "handout_check")
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "retrofire_amd", "csrc"), src,
                               "-o", exe, "-lpthread"])
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    cases, bad = (int(x) for x in out.stdout.split())
    assert cases == 6 and bad == 0, out.stdout
