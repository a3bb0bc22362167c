"""Blocks of the reference schedule (lceq_sweep, f/main.f:37-41) against the
same routines called one by one: the same fields, averages, acceptances and
passes bit for bit, although a block leaves out ahiggs2's averages (ahiggs3
overwrites them) and carries renorm in the next sweep's first launch.  Extents
of 2, where a link's two ends are neighbours both ways, ragged ones, several
block sizes, a strip order, and fed uniforms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,threads,order,imode,meas", [
    ((2, 2, 2), 256, 0, 0, 1), ((2, 4, 6), 64, 0, 1, 1), ((6, 2, 4), 256, 0, 0, 0),
    ((10, 6, 8), 128, 2, 0, 1), ((22, 18, 14), 256, 0, 1, 1), ((32, 32, 32), 512, 4, 0, 1),
    ((40, 36, 48), 256, 0, 0, 1), ((128, 128, 4), 256, 0, 1, 1)])
@pytest.mark.parametrize("fed", [False, True])
def test_block_equals_its_routines(shape, threads, order, imode, meas, fed):
    import lceqcd_amd
    from lceqcd_amd import couplings_from_xy
    n = shape[0] * shape[1] * shape[2] // 2
    sweeps, per = 3, 58 * n  # 2 x 7 n, 2 x n, 6 x 7 n uniforms a sweep
    if fed and n > 20000:
        pytest.skip("the fed stream of a large lattice only repeats the others")
    print("reference schedule", shape, threads, order, imode, meas, fed, flush=True)
    out = []
    for block in (True, False):
        L = lceqcd_amd.Lattice(*shape)
        L.set_couplings(9.0, *couplings_from_xy(9.0, 0.1, 0.5))
        L.set_imode(imode)
        L.set_shape(threads, True)
        L.set_site_order(order)
        L.hotstart(3, 0.2)
        if fed:
            L.rng_feed(np.random.default_rng(8).random(sweeps * per))
        else:
            L.rng_philox(3, 7)
        rows = None
        if block:
            L.sweep(lceqcd_amd.SWEEP_REFERENCE, sweeps - 1, measflag=meas)
            if meas:
                rows = [[r[0], r[1], r[2], r[3], r[7], r[8]] for r in L.history(sweeps - 1)]
            L.sweep(lceqcd_amd.SWEEP_REFERENCE, 1, measflag=meas)
        else:
            rows = []
            for _ in range(sweeps):
                L.ahiggs2(meas)
                ah = L.ahiggs3(meas)
                al = L.agauge(meas)
                o = L.observables()
                rows.append([o["plaq0"], o["a0kin"], o["a02"], o["a04"], al, ah])
                L.renorm()
            rows = rows[:sweeps - 1]
        o = L.observables()
        out.append((L.rng_state(), L.get_links(), L.get_higgs(), rows,
                    [o[k] for k in ("plaq0", "a0kin", "a02", "a04")]))
        L.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])
    if meas:
        assert np.array_equal(out[0][3], out[1][3])
        assert out[0][4] == out[1][4]
