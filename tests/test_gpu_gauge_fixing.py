"""landau_gauge's device-side loop (f/landau_gauge.f:54-59) against the
reference's own loop written on the host: or_gauge_fixing + u_f_renorm
while da1 > limit_or.  The device loop runs its iterations in batches and
tests the loop condition inside the next iteration's first launch; the two
must stop after the same number of iterations with the same da1 and the same
fixed fields, bit for bit (the same kernels run on the same values).  The
iteration cap stops the loop after exactly max_iter iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _thermalised(shape, seed):
    import lceqcd_amd
    L = lceqcd_amd.Lattice(*shape)
    L.set_couplings(9.0, 0.175, -0.45, 0.025)
    L.hotstart(seed, 0.5)
    L.rng_philox(seed, 0)
    L.sweep(lceqcd_amd.SWEEP_KP_OR_METRO, 20, n_or=4, delta=0.4, measflag=0)
    u, a = L.get_links(), L.get_higgs()
    L.close()
    return u, a


def _host_loop(shape, u, a, lam, alpha, limit, nmax):
    import lceqcd_amd
    H = lceqcd_amd.Lattice(*shape)
    H.set_gauge_fixing(lam, alpha, limit)
    H.put_links_fixed(u)
    H.put_higgs_fixed(a)
    da, n = 1e4, 0
    while da > limit and n < nmax:
        da = H.or_gauge_fixing()
        H.u_f_renorm()
        n += 1
    return H, da, n


@pytest.mark.parametrize("shape,alpha,limit", [((8, 8, 8), 1.0, 1e-8), ((6, 4, 8), 0.7, 1e-9),
                                               ((16, 16, 16), 1.0, 1e-7), ((4, 4, 4), 1.0, 1e-12),
                                               ((128, 128, 80), 1.0, 1e-4)])
def test_device_loop_equals_host_loop(shape, alpha, limit):
    """128 x 128 x 80 has 2560 blocks per launch: the loop condition is then
    tested by a one-block launch after every iteration instead of inside the
    next iteration's first launch."""
    import lceqcd_amd
    print("landau_gauge device vs host loop", shape, alpha, limit, flush=True)
    u, a = _thermalised(shape, 41)
    G = lceqcd_amd.Lattice(*shape)
    G.put_links(u)
    G.put_higgs(a)
    G.set_gauge_fixing(1.7, alpha, limit)
    da, it = G.landau_gauge()
    H, dah, nh = _host_loop(shape, u, a, 1.7, alpha, limit, 100000)
    print("iterations device %d host %d, da %.3e" % (it, nh, da), flush=True)
    assert it == nh and it > 8
    assert da == dah and da <= limit
    assert np.array_equal(G.get_links_fixed(), H.get_links_fixed())
    assert np.array_equal(G.get_higgs_fixed(), H.get_higgs_fixed())
    # the unfixed fields are untouched; a second call repeats the first
    assert np.array_equal(G.get_links(), u)
    assert G.landau_gauge() == (da, it)


@pytest.mark.parametrize("cap,shape", [(1, (8, 8, 8)), (8, (8, 8, 8)), (13, (8, 8, 8)),
                                       (40, (8, 8, 8)), (13, (128, 128, 80))])
def test_iteration_cap(cap, shape):
    import lceqcd_amd
    print("landau_gauge cap", cap, flush=True)
    u, a = _thermalised(shape, 43)
    G = lceqcd_amd.Lattice(*shape)
    G.put_links(u)
    G.put_higgs(a)
    G.set_gauge_fixing(1.7, 1.0, 1e-14, cap)
    with pytest.raises(lceqcd_amd.LceqError, match="max_iter"):
        G.landau_gauge()
    H, _, n = _host_loop(shape, u, a, 1.7, 1.0, 1e-14, cap)
    assert n == cap
    assert np.array_equal(G.get_links_fixed(), H.get_links_fixed())


@pytest.mark.parametrize("shape,alpha", [((2, 2, 2), 1.0), ((2, 4, 6), 0.8), ((18, 2, 4), 1.0),
                                         ((16, 8, 4), 1.0), ((14, 10, 6), 1.0), ((34, 18, 10), 0.7),
                                         ((16, 16, 16), 1.0), ((30, 6, 130), 1.0),
                                         ((66, 34, 26), 1.0)])
@pytest.mark.parametrize("cap", [1, 2, 9, 24])
def test_tiles_equal_the_half_steps(shape, alpha, cap):
    """An iteration in one launch over tiles of 16 x 8 x 4 sites against the two
    half steps as launches of their own: tiles cut off at every face, extents of
    2, one tile, more than 64 tiles (the loop condition by block sums), and an odd
    and an even number of iterations (the result in either link array)."""
    import lceqcd_amd
    print("landau_gauge tiles", shape, cap, flush=True)
    rng = np.random.default_rng(3)
    n = shape[0] * shape[1] * shape[2] // 2
    u = rng.normal(size=(3, 2, n, 4))
    u /= np.linalg.norm(u, axis=-1, keepdims=True)
    a = rng.normal(size=(2, n, 3))
    G = lceqcd_amd.Lattice(*shape)
    G.put_links(u)
    G.put_higgs(a)
    G.set_gauge_fixing(1.7, alpha, 1e-300, cap)
    H, da, done = _host_loop(shape, u, a, 1.7, alpha, 1e-300, cap)
    assert done == cap
    for _ in range(2):  # the second call starts from the other link array
        with pytest.raises(lceqcd_amd.LceqError, match="da = %g" % da):
            G.landau_gauge()
        assert np.array_equal(G.get_links_fixed(), H.get_links_fixed())
        assert np.array_equal(G.get_higgs_fixed(), H.get_higgs_fixed())
        assert np.array_equal(G.get_links(), u)
    G.or_gauge_fixing()
    H.or_gauge_fixing()
    assert np.array_equal(G.get_links_fixed(), H.get_links_fixed())


@pytest.mark.parametrize("shape", [(128, 128, 100), (140, 140, 140)])
def test_lattices_beyond_the_cache(shape):
    """Two link arrays that the Infinity Cache does not hold (half steps in place),
    and one that it does not (one launch, the links stored without write-through)."""
    test_tiles_equal_the_half_steps(shape, 1.0, 9)


@pytest.mark.parametrize("shape,limit", [((96, 96, 64), 1e-4), ((104, 104, 104), 1e-4)])
def test_device_loop_of_many_tiles(shape, limit):
    """1152 tiles, whose sum over block sums tests the loop condition inside the
    next iteration's launch, and 2366 within the Infinity Cache, with a launch of
    its own for the test; the loop ends inside a batch of iterations."""
    test_device_loop_equals_host_loop(shape, 1.0, limit)


@pytest.mark.parametrize("shape,launches", [((2, 16, 16), 2), ((4, 4, 4), 2), ((4, 128, 256), 2),
                                            ((6, 256, 128), 2), ((6, 4, 8), 1), ((4, 32, 64), 1),
                                            ((8, 256, 128), 1), ((16, 16, 16), 1)])
def test_mostly_empty_tiles_take_the_half_steps(shape, launches):
    """An iteration is two launches in place where one launch's tiles would hold
    few sites each, and one otherwise; the same fields as the host loop."""
    import lceqcd_amd
    print("landau_gauge launches", shape, flush=True)
    u, a = _thermalised(shape, 47)
    G = lceqcd_amd.Lattice(*shape)
    G.put_links(u)
    G.put_higgs(a)
    G.set_gauge_fixing(1.7, 1.0, 1e-300, 8)
    G.profile_begin(lceqcd_amd.KC_GFIX, 100)
    with pytest.raises(lceqcd_amd.LceqError, match="max_iter"):
        G.landau_gauge()
    assert G.profile_end()[1] == 8 * launches
    H, _, _ = _host_loop(shape, u, a, 1.7, 1.0, 1e-300, 8)
    assert np.array_equal(G.get_links_fixed(), H.get_links_fixed())
    assert np.array_equal(G.get_higgs_fixed(), H.get_higgs_fixed())


@pytest.mark.parametrize("shape,limit", [((140, 140, 140), 1e-3), ((132, 132, 132), 1e-3),
                                         ((18, 128, 128), 1e-4), ((66, 66, 66), 1e-4),
                                         ((4, 256, 128), 1e-4), ((50, 64, 64), 1e-4)])
def test_one_da_for_both_loops(shape, limit):
    """The device loop and the host loop add da in the same order on every lattice:
    beyond the Infinity Cache in one launch per iteration and in place, and
    within it on tiles that are cut off (above and below 512 of them) and mostly
    empty."""
    test_device_loop_equals_host_loop(shape, 1.0, limit)


@pytest.mark.parametrize("shape,launches", [((96, 96, 96), 1), ((104, 104, 104), 1),
                                            ((108, 108, 108), 2), ((34, 256, 128), 2),
                                            ((128, 128, 100), 2), ((140, 140, 140), 2),
                                            ((50, 256, 400), 2), ((160, 160, 112), 1),
                                            ((148, 148, 148), 1)])
def test_launches_where_the_cache_ends(shape, launches):
    """Rows of whole tiles and others on either side of the Infinity Cache, with
    one and with two launches an iteration."""
    test_mostly_empty_tiles_take_the_half_steps(shape, launches)
