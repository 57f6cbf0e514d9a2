"""The stepping kernel's Krylov gathers from memory keep a row's loads in flight:
eight columns, then the values of eight entries.  Read from the assembly of the
512-thread variants, whose schedule the compiler took back before the gathers
were written in stages: two loads, a wait, two loads, a wait."""
import re
import subprocess

import pytest

from femhip import build

PROBE = """
#define FEMHIP_TEAM_BLOCK 512
#include "step_kernel.h"
namespace femhip {
const void* probe() { return (const void*)k_step<%d, float, %d, kFenced, false>; }
}
"""


def runs(block):
    """Loads between the waits for loads of a basic block."""
    out = [0]
    for op, args in block:
        if op.startswith("global_load"):
            out[-1] += 1
        elif op == "s_waitcnt" and "vmcnt" in args and out[-1]:
            out.append(0)
    return [n for n in out if n]


@pytest.mark.parametrize("k,kr,values", [(1, 1, 5), (16, 0, 5), (4, 2, 4)])
def test_loads_in_flight(tmp_path, k, kr, values):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE % (k, kr))
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, f"-I{build.INCLUDE}", f"-I{build.CSRC}", "--cuda-device-only", "-S", str(src),
           "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    blocks, cur = [], []
    for line in out.read_text().splitlines():
        line = line.split(";")[0].rstrip()
        if line.startswith(".LBB"):
            blocks.append(cur)
            cur = []
        elif m := re.match(r"\s+([a-z]\w+)\s*(.*)", line):
            cur.append((m[1], m[2]))
    blocks.append(cur)
    gathers = [b for b in blocks if sum(op.startswith("global_load") for op, _ in b) >= 8 * values
               and any("f32" in op for op, _ in b) and not any("f64" in op for op, _ in b)]
    assert gathers
    for b in gathers:
        assert runs(b)[0] >= 8 and max(runs(b)) >= 8 * (values - 1), runs(b)
