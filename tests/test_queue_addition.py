"""A work queue's head is added to by one lane of the wave, whatever the
compiler makes of the wave's lanes: the emitted code is looked at with the pass
that merges the lanes' additions turned off.  (Additions of 64 lanes are 64
operations, between which another wave's may fall; two waves then take the
same item, or none does.)"""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pixie_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# a loop that ends in a branch on lane 0, as the addition's own
KERNEL = r"""
#include "pxh_queue.h"
__global__ void __launch_bounds__(64) probe(int* heads, int n, int* out) {
  for (;;) {
    const int i = pxh::queue_next<32>(heads, n);
    if (i >= n) break;
    if (threadIdx.x == 0) out[i] = i;
  }
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("merge", ["None", "Iterative", "DPP"])
def test_one_lane_adds(tmp_path, merge):
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(KERNEL)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O3", "-std=c++17", "-I", CSRC, "-S",
                    "--cuda-device-only", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "-mllvm",
                    "-amdgpu-atomic-optimizer-strategy=" + merge, str(src), "-o", str(asm)], check=True)
    body = asm.read_text().split("s_endpgm")[0].splitlines()
    adds = [k for k, line in enumerate(body) if "global_atomic_add" in line]
    assert len(adds) == 1
    masks = [(k, line) for k, line in enumerate(body) if re.search(r"s_(and_saveexec|or)_b64\s+(s\[|exec)", line)
             or "v_readfirstlane" in line]
    # lanes are masked off before the addition and back before its value is read
    before = [line for k, line in masks if k < adds[0] and "readfirstlane" not in line]
    assert before and "s_and_saveexec" in before[-1], "the whole wave adds"
    compare = [line for line in body[:adds[0]] if re.search(r"v_cmp_(eq|ne|gt)_u32", line)]
    assert compare, "no lane is chosen"
    after = [line for k, line in masks if k > adds[0]]
    first_read = next(k for k, line in enumerate(after) if "readfirstlane" in line)
    assert any("exec, exec" in line for line in after[:first_read]), "the value is read by the adding lane alone"
