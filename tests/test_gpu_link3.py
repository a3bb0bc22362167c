"""Link sweeps with the three directions of a parity in one launch, over tiles
of 16 x 4 x 4 sites, against the launches per direction, which a lattice runs
while one of its kernel classes is being timed: links, Higgs field, step size
and measured rows bit for bit.  Extents of 2, tiles cut off in each direction,
and several whole ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 2), (2, 10, 6), (4, 2, 2), (6, 10, 10), (16, 8, 4),
                                   (18, 10, 6), (14, 6, 2), (22, 18, 50), (34, 12, 4),
                                   (48, 48, 48),
                                   (64, 64, 100)])
def test_three_directions_in_one_launch(shape):
    import lceqcd_amd
    print("links of three directions", shape, flush=True)
    out = []
    for timed in (False, True):
        L = lceqcd_amd.Lattice(*shape)
        L.set_couplings(9.0, 0.175, -0.45, 0.025)
        L.hotstart(5, 0.5)
        L.rng_philox(5, 0)
        if timed:
            L.profile_begin(lceqcd_amd.KC_GFIX, 1)
        d = L.sweep(0, 1, n_or=2, delta=0.4, measflag=0)
        first = L.get_links()
        L.put_links(first)
        d = L.sweep(0, 3, n_or=2, delta=d, measflag=1)
        L.sweep(1, 2, measflag=0)
        out.append((d, L.rng_state(), L.history(3), first, L.get_links(), L.get_higgs()))
        L.close()
    assert out[0][:2] == out[1][:2]
    for a, b in zip(out[0][2:], out[1][2:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(2, 2, 2), (6, 10, 10), (22, 18, 50), (34, 12, 4), (48, 48, 48),
                                   (64, 64, 100)])
def test_three_directions_equal_the_batch(shape):
    """The same chain as a batch of one replica, whose link launches are always
    per direction."""
    import lceqcd_amd
    print("links of three directions and the batch", shape, flush=True)
    coup = (9.0, 0.175, -0.45, 0.025)
    B = lceqcd_amd.Batch([shape])
    B.set_couplings([coup])
    B.hotstart([5], 0.5)
    B.rng_philox([5])
    B.sweep(3, n_or=2, delta=0.4, measflag=0)
    L = lceqcd_amd.Lattice(*shape)
    L.set_couplings(*coup)
    L.hotstart(5, 0.5)
    L.rng_philox(5, 0)
    L.sweep(0, 3, n_or=2, delta=0.4, measflag=0)
    assert np.array_equal(L.get_links(), B.get_links(0))
    assert np.array_equal(L.get_higgs(), B.get_higgs(0))
    B.close()
    L.close()
