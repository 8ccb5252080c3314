"""The merged layout's evaluators keep their sums, staged rows and operand ring in
registers: compiled for gfx950 with the build's flags, none of them spills or uses scratch
memory (spilled, one Q at 27^3 nodes takes 7.7 ms instead of 4.6).  No GPU needed."""
import os
import re
import subprocess

import pytest

from dgv0d3v_direct_collision_amd import build


def resources(source):
    """{mangled kernel name: {resource: value}} from the compiler's remarks."""
    cmd = [build.hipcc(), *build.HIPFLAGS, *build.FILE_FLAGS.get(source, []), "--cuda-device-only", "-x", "hip", "-c",
           os.path.join(build.CSRC, source), "-o", os.devnull, "-Rpass-analysis=kernel-resource-usage"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    out, cur = {}, None
    for name, key, value in re.findall(r"remark: [^\n]*?(?:Function Name: (\S+)|\s([A-Za-z][A-Za-z ]*)(?:\[[^\]]*\])?: (\d+))", r.stderr):
        if name:
            cur = out.setdefault(name, {})
        elif cur is not None:
            cur[key.strip()] = int(value)
    return out


@pytest.mark.parametrize("source,kernel,count", [("dgv_quad.hip", "k_quad_eval", 4), ("dgv_batch.hip", "k_quad_batchI", 2)])
def test_no_scratch(source, kernel, count):
    try:
        build.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    found = {k: v for k, v in resources(source).items() if kernel in k}
    assert len(found) == count, sorted(found)
    for name, use in found.items():
        assert use["ScratchSize"] == 0 and use["VGPRs Spill"] == 0, (name, use)
