"""Production sweeps in slabs of z planes (lattices of more than 288 MiB of
fields) against the same sweeps in whole-lattice launches, which a lattice
runs while one of its kernel classes is being timed: the same links, Higgs
field and step size bit for bit, and the same averages up to the order of
their sums.  Two slabs and more, planes that are and are not a multiple of the
block size, other block sizes, site orders and numbers of overrelaxation
sweeps; and the library's site order on large planes against a caller's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lattice(shape, seed):
    import lceqcd_amd
    L = lceqcd_amd.Lattice(*shape)
    L.set_couplings(9.0, 0.175, -0.45, 0.025)
    L.hotstart(seed, 0.5)
    L.rng_philox(seed, 0)
    return L


def _same_sums(a, b):
    # sums of up to 2e7 terms, added in different orders: n 2^-53 at the most
    # of their absolute sum, which for these averages is of their own size
    np.testing.assert_allclose(a, b, rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("shape,threads,order,n_or,meas", [
    ((128, 128, 160), 256, 0, 4, 1),   # two slabs, planes of whole blocks
    ((128, 128, 160), 64, 16, 1, 0),
    ((144, 144, 128), 256, 0, 4, 1),   # 40.5 blocks a plane: measured passes whole
    ((144, 144, 128), 128, 4, 0, 1),   # 81 blocks of 128; the heatbath measures
    ((64, 64, 700), 512, 0, 2, 1),     # many small planes
    ((256, 256, 44), 256, 0, 1, 1),    # few large ones
    ((160, 192, 180), 256, 0, 4, 1),   # more than two slabs
    ((170, 150, 130), 256, 0, 1, 1)])  # no order in strips but two rows
def test_slabs_equal_whole_lattice_launches(shape, threads, order, n_or, meas):
    import lceqcd_amd
    print("slab sweeps", shape, threads, order, n_or, meas, flush=True)
    out = []
    for whole in (False, True):
        L = _lattice(shape, 5)
        L.set_shape(threads, True)
        L.set_site_order(order)
        if whole:
            L.profile_begin(lceqcd_amd.KC_GFIX, 1)
        d = L.sweep(0, 2, n_or=n_or, delta=0.4, measflag=meas)
        d = L.sweep(0, 1, n_or=n_or, delta=d, measflag=meas)
        out.append((d, L.rng_state(), L.history(3) if meas else None, L.get_higgs(),
                    L.get_links()))
        L.close()
    assert out[0][:2] == out[1][:2]
    assert np.array_equal(out[0][3], out[1][3])
    assert np.array_equal(out[0][4], out[1][4])
    if meas:
        _same_sums(out[0][2], out[1][2])


@pytest.mark.parametrize("shape,order", [((128, 128, 8), 2), ((150, 150, 6), 0), ((20, 1024, 4), 4),
                                         ((160, 160, 6), 4), ((1024, 18, 4), 2)])
def test_library_order_on_large_planes(shape, order):
    """Every update of the library's own order against another order's."""
    import lceqcd_amd
    print("site order of large planes", shape, order, flush=True)
    out = []
    for so in (0, order):
        L = _lattice(shape, 6)
        if so:
            L.set_site_order(so)
        L.agauge(1)
        L.link_or(1)
        L.ahiggs1(0.4, 1)
        L.set_couplings(9.0, 0.175, 2.0, 0.025)
        L.ahiggs2(1)
        L.ahiggs3(1)
        L.sweep(lceqcd_amd.SWEEP_REFERENCE, 1, measflag=1)
        out.append((L.history(1), L.get_links(), L.get_higgs()))
        L.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])
    _same_sums(out[0][0], out[1][0])


@pytest.mark.parametrize("shape", [(144, 144, 128), (174, 150, 130), (256, 256, 44)])
def test_slabs_in_the_librarys_order(shape):
    """Slabs and the library's site order together (strips of 16 and of 2 rows),
    against whole-lattice launches in index order and against a batch of one
    replica, whose launches are whole and in index order."""
    import lceqcd_amd
    print("slabs in the library's order", shape, flush=True)
    coup = (9.0, 0.175, -0.45, 0.025)
    out = []
    for whole in (False, True):
        L = _lattice(shape, 5)
        if whole:
            assert L.get_site_order() > 0
            L.set_site_order(0)
            L.profile_begin(lceqcd_amd.KC_GFIX, 1)
        L.sweep(0, 2, n_or=2, delta=0.4, measflag=1)
        out.append((L.get_links(), L.get_higgs(), L.history(2)))
        L.close()
    B = lceqcd_amd.Batch([shape])
    B.set_couplings([coup])
    B.hotstart([5], 0.5)
    B.rng_philox([5])
    B.sweep(2, n_or=2, delta=0.4, measflag=1)
    out.append((B.get_links(0), B.get_higgs(0), B.history(2)[:, 0]))
    B.close()
    for got in out[1:]:
        assert np.array_equal(got[0], out[0][0])
        assert np.array_equal(got[1], out[0][1])
        _same_sums(got[2], out[0][2])
