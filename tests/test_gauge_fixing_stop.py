"""The end of the gauge-fixing loop as the waves of one launch see it
(lceq_internal.hpp gfix_ended, compiled here for the host).  The launch that
tests the loop condition after `iter` iterations writes the flag from one block
while the waves of the others read it, in any order.  Every wave of a block has
to reach the test whatever it read, because the test sums over the block's
waves: one that had left would leave its share of the sum unwritten."""
import itertools
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lceqcd_amd",
                    "csrc")
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "lceq_internal.hpp"
int main(int argc, char** argv) {
  for (int i = 1; i + 1 < argc; i += 2)
    std::printf("%d\\n", lceq::gfix_ended(atof(argv[i]), atof(argv[i + 1])));
}
"""


def test_every_wave_reaches_the_test(tmp_path):
    src, exe = tmp_path / "ended.hip", tmp_path / "ended"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-O1",
                    "-std=c++17", "-w", "-I", CSRC, str(src), "-o", str(exe)], check=True)

    def ended(pairs):
        args = ["%.17g" % v for p in pairs for v in p]
        out = subprocess.run([str(exe)] + args, check=True, capture_output=True, text=True).stdout
        return [bool(int(v)) for v in out.split()]

    for iters in (1, 2, 7, 255, 2047, 1000000):
        # the testing launch: 0 before its own entry, `iters` after it
        seen = list(itertools.product((0.0, float(iters)), repeat=4))
        for block in seen:
            assert ended([(v, iters) for v in block]) == [False] * 4
        # launches behind it, which do (one more iteration) or do not test
        assert ended([(iters, iters + 1), (iters, iters + 200), (iters, 0)]) == [True] * 3
        # nothing has ended: every launch runs
        assert ended([(0, iters), (0, 0)]) == [False] * 2
