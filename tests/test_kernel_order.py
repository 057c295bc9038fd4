"""Waits that count loads rest on the order the compiler leaves them in: read from the assembly of
this source, compiled with the build's own flags (no GPU).
"""

import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "prism-inference_amd")


def _asm(source, tmp_path):
    sys.path.insert(0, PKG)
    import build

    out = str(tmp_path / "out.s")
    cmd = [build.HIPCC, *build.FLAGS, "-S", "--cuda-device-only", "-o", out, os.path.join(build.CSRC, source)]
    subprocess.run(cmd, check=True, capture_output=True)
    with open(out) as f:
        return f.read()


def test_pinned_prefill_loads_stay_in_the_counted_order(tmp_path):
    """k_prefill_ptq1_pinned: between barriers, a first half issues two direct-to-LDS loads and ends on
    vmcnt(9); a second one three and then the four plain loads of the weights, and ends on vmcnt(13)."""
    text = _asm("prefill.hip", tmp_path)
    kernels = re.findall(r"^(_ZN\S*k_prefill_ptq1_pinned\S*):", text, re.M)
    assert len(kernels) == 2
    for name in kernels:
        body = text[text.index("\n" + name + ":"):]
        body = body[:body.index(".Lfunc_end")]
        loads, halves = [], []
        for line in body.splitlines():
            line = line.split(";")[0].strip()
            if line.startswith("buffer_load"):
                loads.append("L" if line.endswith("lds") else "w")
            elif line.startswith("s_waitcnt") and (m := re.search(r"vmcnt\((\d+)\)", line)):
                counted = int(m.group(1))
            elif line.startswith("s_barrier"):
                halves.append(("".join(loads), counted))
                loads = []
        pipeline = [h for h in halves if h[1] in (9, 13)]
        assert pipeline == [("LL", 9), ("LLLwwww", 13)] * 2, (name, halves)
