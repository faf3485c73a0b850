"""Orderings that no run can show to be there, read from the AMD assembly of this package's own
kernels (compiled here; no GPU needed).

A workgroup that is the last of several to finish takes what the others have stored only after it
has counted them all, so every wave's stores must have arrived before its workgroup counts itself.
On gfx950 neither a workgroup-scope release nor the barrier waits for vector memory: the wait has
to stand in the code, between the stores and the barrier in front of the count."""
import os
import re
import subprocess

import pytest

from graph_sampling_amd import build


def _assembly(source, tmp_path):
    out = str(tmp_path / (source + ".s"))
    build._run([build.HIPCC] + build.HIP_FLAGS + ["--offload-device-only", "-S", "-x", "hip",
               os.path.join(build._CSRC, source), "-o", out])
    with open(out) as f:
        return f.read()


def _kernels(text, name):
    """Bodies of the kernels whose mangled name holds `name`, as lists of instructions."""
    found = []
    for m in re.finditer(r"^(_Z\w*%s\w*):.*?^\.Lfunc_end" % name, text, re.S | re.M):
        lines = (line.split(";")[0].strip() for line in m.group(0).split("\n")[1:])
        found.append([line for line in lines if line and not line.endswith(":") and line[0] != "."])
    return found


def _last(lines, pattern):
    return max((i for i, line in enumerate(lines) if re.search(pattern, line)), default=-1)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("source,kernel,publish,instances", [
    # candidates of a chunk, then the row's chunks counted
    ("gs_weighted.hip", "weighted_fill_kernel", r"^global_store.* sc1$", 4),
    # a tile's class counts, then the workgroups counted
    ("gs_listsample.hip", "keys_hist_kernel", r"^global_atomic_add .* off$", 1),
])
def test_stores_have_arrived_before_the_workgroup_counts_itself(source, kernel, publish, instances, tmp_path):
    bodies = _kernels(_assembly(source, tmp_path), kernel)
    assert len(bodies) == instances
    for lines in bodies:
        count = [i for i, line in enumerate(lines) if re.match(r"global_atomic_add .* sc0$", line)]
        assert len(count) == 1  # (an addition whose result is asked for)
        before = lines[:count[0]]
        stored, barrier = _last(before, publish), _last(before, r"^s_barrier")
        assert 0 <= stored < barrier
        assert any(re.match(r"s_waitcnt vmcnt\(0\)", line) for line in before[stored:barrier])
