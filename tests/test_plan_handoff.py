"""The hand-over inside k_plan_blocks (plan.hip): the workgroup that finishes last
reads what every wave of the others has stored.  A barrier does not wait for a wave's
stores to memory, and the release of the thread that counts waits for its own wave's
only, so each wave has to wait for its stores before the barrier.  Read from the
compiled kernel."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor-tools_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_stores_are_waited_for_before_the_count(tmp_path):
    out = tmp_path / "plan.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                           "-packed-fp32-ops", "-I../../include", "-S", "--offload-device-only", "plan.hip", "-o", str(out)],
                          cwd=CSRC, stderr=subprocess.DEVNULL)
    lines = out.read_text().splitlines()
    start = next(i for i, l in enumerate(lines) if re.match(r"_ZN3ttg13k_plan_blocks\w*:", l))
    release = next(i for i in range(start, len(lines)) if "buffer_wbl2" in lines[i])
    barrier = max(i for i in range(start, release) if "s_barrier" in lines[i])
    before = []   # the straight run of code that ends at the barrier
    for l in reversed(lines[start:barrier]):
        if re.search(r"global_store|flat_store|s_branch|s_endpgm", l):
            break
        before.append(l)
    assert any("s_waitcnt" in l and "vmcnt(0)" in l for l in before)
