"""correlator, scalarcorr and polyakov against the CPU restatement at the edges
of their kernels: slices split over 1 to 16 blocks, separations and slices that
do not fill a block's 16 and 128, slice means in LDS (6 lz doubles up to 47 KB: lz <= 1002)
and beyond, results in pinned memory (lz <= 1634) and beyond; each measurement
called alone and in another order leaves the others' results alone.

The restatement adds a slice's sites in one run, the kernels in pieces: the
bound is 1e-12 of the correlator at separation 0 (sums of at most 9216 values
of order one, 2^-53 each)."""
import numpy as np
import pytest

from helpers import rand_conf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 2), (6, 4, 10), (24, 22, 6), (64, 64, 4), (96, 96, 2),
                                   (34, 30, 18), (4, 2, 300), (2, 2, 1002), (2, 2, 1004),
                                   (2, 2, 1634), (2, 2, 1636)])
def test_measurements(oracle_lib, shape):
    import lceqcd_amd
    print("correlators", shape, flush=True)
    u, a = rand_conf(shape, 31, 0.6)
    uf, af = rand_conf(shape, 32, 0.4)
    G, O = lceqcd_amd.Lattice(*shape), oracle_lib.OracleLattice(*shape)
    for L in (G, O):
        L.put_links(u)
        L.put_higgs(a)
        L.put_links_fixed(uf)
        L.put_higgs_fixed(af)

    def close(got, ref):
        got, ref = np.asarray(got), np.asarray(ref)
        assert np.max(np.abs(got - ref)) <= 1e-12 * max(1.0, np.max(np.abs(ref)))

    ref = {"scalarcorr": O.scalarcorr(), "polyakov": O.polyakov(), "correlator": O.correlator()}
    for name in ("polyakov", "correlator", "scalarcorr", "correlator", "polyakov"):
        for got, exp in zip(getattr(G, name)(), ref[name]):
            close(got, exp)
    close(G.observables()["a0f"], O.observables()["a0f"])
    G.close()
