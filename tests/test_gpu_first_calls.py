"""What the first calls of a process allocate."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = r"""
import ctypes, re
import pixie_amd as px
img = px.Image(512, 512)
star = "M 20 20 L 400 30 L 60 300 Z"
img.fillPath(star, (9, 8, 7, 255))
px.synchronize()
hip = ctypes.CDLL(re.search(r"(/\S*libamdhip64\.so\S*)", open("/proc/self/maps").read()).group(1))
def free():
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value
before = free()
for _ in range(10):
    img.fillPath(star, (9, 8, 7, 255))
px.synchronize()
print("allocated", before - free())
"""


def test_small_fills_allocate_once():
    """A small fill's upload space is there for those that follow it."""
    out = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    assert out.stdout.split() == ["allocated", "0"], out.stdout
