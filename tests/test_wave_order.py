"""The control wave of a stepping workgroup stores the reduced sums lane by lane
into LDS and its lanes then read each other's: a wavefront fence has to stand
between the two.  Read from the compiler's own IR before any optimisation."""
import re
import subprocess

import pytest

from femhip import build

PROBE = """
#define FEMHIP_TEAM_BLOCK 512
#include "step_kernel.h"
namespace femhip {
const void* probe(int kr) { return pick_kr<%s, %s, 2, float>(kr); }
}
"""


@pytest.mark.parametrize("mode,rows", [("kPlain", "false"), ("kCoherent", "true"), ("kFenced", "true")])
def test_fence_before_scalars(tmp_path, mode, rows):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.ll"
    src.write_text(PROBE % (mode, rows))
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, f"-I{build.INCLUDE}", f"-I{build.CSRC}", "--cuda-device-only", "-Xclang",
           "-disable-llvm-passes", "-emit-llvm", "-S", str(src), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    bodies = {m[1]: m[2] for m in re.finditer(r"^define [^@\n]*@(\w+)\([^\n]*\n(.*?)^}", out.read_text(), re.M | re.S)}
    calls = {name: re.findall(r"call [^@\n]*@([\w.]+)\(|(fence syncscope\(\"wavefront[\w-]*\"\) \w+)", body)
             for name, body in bodies.items()}
    calls = {name: [a or b for a, b in c] for name, c in calls.items()}
    scalars = re.compile(r"ENKUlvE\d*_clEv$")  # a lambda without arguments

    def events(name):
        """The stores of sums, fences and uses of sums below a function, in order."""
        for c in calls.get(name, ()):
            if re.match(r"_ZN6femhip12_GLOBAL__N_1(14block_partials|7collect)I", c):
                yield "sums"
            elif c.startswith("fence"):
                yield c.split()[-1]
            elif scalars.search(c):
                yield "scalars"
            elif "run_scalars" in c:
                yield from events(c)

    reduces = [n for n in bodies if re.search(r"^_ZN6femhip12_GLOBAL__N_111(team|rows)_reduceI", n)]
    assert reduces
    used = 0
    for n in reduces:
        seq = list(events(n))
        for i, ev in enumerate(seq):
            if ev == "scalars":
                used += 1
                last = max(j for j in range(i) if seq[j] == "sums")
                assert seq[last + 1:i].count("release") >= 1 and seq[i - 1] == "acquire", (n, seq)
    assert used
