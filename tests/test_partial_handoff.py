"""The order that the attention's hand-off of partials between workgroups rests on, in the code that the compiler makes of it: a
relaxed atomic and a wait order nothing by themselves, and a compiler that moved one over the other would give wrong outputs
now and then without an error."""
import os
import re
import subprocess

import pytest

from retrievalattention_amd import build


def test_partials_are_out_before_their_arrival_is_announced(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    out = str(tmp_path / "attend.s")
    subprocess.run([hipcc] + [f for f in build.HIP_FLAGS if f != "-fPIC"] +
                   ["--offload-device-only", "-S", os.path.join(build.CSRC, "attend.hip"), "-o", out],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(out) as f:
        lines = [ln.strip() for ln in f]
    arrivals = [i for i, ln in enumerate(lines) if ln.startswith("global_atomic_add")]
    assert len(arrivals) == 6   # 4, 8 and 16 heads in two element types
    memory = re.compile(r"(global|flat|buffer|scratch)_(load|store|atomic)")
    for i in arrivals:
        # back to the wait for every store: no access to memory between it and the increment
        back = next(j for j in range(i - 1, 0, -1) if memory.match(lines[j]) or re.match(r"s_waitcnt .*vmcnt\(0\)", lines[j]))
        assert lines[back].startswith("s_waitcnt"), lines[back]
        # on to the next access: behind the wait for the increment and the branch on its count
        on = next(j for j in range(i + 1, len(lines)) if memory.match(lines[j]))
        between = lines[i + 1:on]
        wait = next(j for j, ln in enumerate(between) if re.match(r"s_waitcnt .*vmcnt\(0\)", ln))
        assert any(ln.startswith("s_cbranch") for ln in between[wait:]), between
