"""The block-scale kernels' loads in the compiled gfx950 code (no GPU): a step ends on a count of loads that may still fly, so
its activation loads have to be issued before its code and scale loads."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

SOURCE = os.path.join(ROOT, "siliconed_amd", "csrc", "sq8_blocks.hip")


@pytest.fixture(scope="module")
def steps(tmp_path_factory):
    """(rows, waves) of the instance → its loads between barriers, A an activation load into LDS, W one into registers."""
    from siliconed_amd.build import FLAGS, HIPCC
    out = str(tmp_path_factory.mktemp("asm") / "blocks.s")
    r = subprocess.run([HIPCC, *FLAGS, "--cuda-device-only", "-S", SOURCE, "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    with open(out) as f:
        text = f.read()
    found = {}
    for name, body in re.findall(r"^(_Z\w*gemm_blocks_kernel\w*):(.*?)s_endpgm", text, re.S | re.M):
        lines = [line.strip() for line in body.split("\n")]
        loads = ["A" if line.startswith("buffer_load") and line.endswith("lds") else "W" if line.startswith("global_load") else
                 "|" if line.startswith("s_barrier") else "" for line in lines]
        found[tuple(int(v) for v in re.search(r"ILi(\d+)ELi(\d+)E", name).groups())] = "".join(loads).split("|")
    return found


@pytest.mark.parametrize("rows,waves", [(128, 4), (128, 8), (64, 8)])
def test_a_steps_activation_loads_come_before_its_code_loads(steps, rows, waves):
    loop = [s for s in steps[rows, waves][1:] if "A" in s and "W" in s]  # after the prologue, which drains all its loads
    assert len(loop) >= 4, steps[rows, waves]
    assert all(re.fullmatch("A{%d}W{3}" % (rows // 8 // waves), s) for s in loop), loop
