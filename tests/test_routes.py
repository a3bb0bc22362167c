"""Which launches a call takes, by the lattice's extents and state: the rules of
lceq_internal.hpp, compiled here for the host."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lceqcd_amd",
                    "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """rule(expression, shape): the value of a C++ expression of `Geom g`."""
    folder = tmp_path_factory.mktemp("rules")
    built = {}

    def run(expression, shape):
        if expression not in built:
            src, exe = folder / ("r%d.hip" % len(built)), folder / ("r%d" % len(built))
            src.write_text("""
#include <cstdio>
#include <cstdlib>
#include "lceq_internal.hpp"
using namespace lceq;
int main(int, char** v) {
  Geom g = geom_init(atoi(v[1]), atoi(v[2]), atoi(v[3]));
  std::printf("%%d\\n", (int)(%s));
}
""" % expression)
            subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only",
                            "-O1", "-std=c++17", "-w", "-I", CSRC, str(src), "-o", str(exe)],
                           check=True)
            built[expression] = exe
        out = subprocess.run([str(built[expression])] + [str(e) for e in shape], check=True,
                             capture_output=True, text=True).stdout
        return int(out)

    return run


@pytest.mark.parametrize("shape,tiles", [
    ((18, 48, 64), 0), ((18, 64, 64), 0), ((18, 34, 66), 0), ((2, 128, 64), 0),
    ((18, 32, 64), 256), ((2, 64, 64), 256), ((34, 34, 50), 351), ((4, 128, 64), 512),
    ((44, 44, 44), 363), ((64, 64, 32), 512), ((64, 64, 64), 0), ((96, 96, 96), 3456),
    ((100, 100, 100), 0), ((128, 128, 128), 0)])
def test_three_directions_in_one_launch(rule, shape, tiles):
    """Link sweeps of lattices whose tiles are mostly two columns wide take the
    launches per direction beyond 256 tiles."""
    assert rule("link3_tiles(g)", shape) == tiles


@pytest.mark.parametrize("state,carried", [("", 1), ("L.prof_class = KC_HIGGS;", 0),
                                           ("L.prof_class = KC_GFIX;", 0),
                                           ("L.rng_mode = LCEQ_RNG_FED;", 0)])
def test_renorm_within_a_higgs_launch(rule, state, carried):
    """Timed Higgs launches do not do renorm's work (nor do fed ones)."""
    made = "[] { lceq_lattice L{}; L.rng_mode = LCEQ_RNG_PHILOX; %s return L; }" % state
    assert rule("([&] { lceq_lattice L = %s(); return carries_renorm(&L); })()" % made,
                (4, 4, 4)) == carried
