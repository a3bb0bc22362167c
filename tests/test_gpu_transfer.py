"""Field transfers between host arrays and the device layout: a download of
the device's own hot start equals the CPU restatement's, and an upload comes
back bit for bit, from one row of a transfer slot to several slots for each of
several host threads, with an exact and with a larger leading dimension (whose
gap is left alone), on a lattice and on a replica of a batch."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DP = C.POINTER(C.c_double)
# a chunk is 24576 to 49152 link rows or 32768 to 65536 Higgs rows; one worker
# up to three chunks, then one per two chunks up to eight
SHAPES = [(2, 2, 2), (6, 4, 8), (32, 16, 16), (32, 32, 24), (34, 26, 46), (64, 48, 40),
          (64, 64, 128)]


def _get(lib, fn, h, n, classes, ncomp, ld, *rep):
    out = np.full((classes, ld, ncomp), -7.0)
    assert getattr(lib, fn)(h, *rep, out.ctypes.data_as(DP), ld) == 0
    assert (out[:, n:] == -7.0).all()
    return out[:, :n]


def _put(lib, fn, h, field, ld, *rep):
    classes, n, ncomp = field.shape
    a = np.full((classes, ld, ncomp), np.nan)
    a[:, :n] = field
    assert getattr(lib, fn)(h, *rep, a.ctypes.data_as(DP), ld) == 0


@pytest.mark.parametrize("shape", SHAPES)
def test_fields_cross_the_bus(oracle_lib, shape):
    import lceqcd_amd
    n = shape[0] * shape[1] * shape[2] // 2
    print("field transfer", shape, flush=True)
    L, O = lceqcd_amd.Lattice(*shape), oracle_lib.OracleLattice(*shape)
    B = lceqcd_amd.Batch([(4, 4, 4), shape])
    L.hotstart(11, 0.5)
    O.hotstart(11, 0.5)
    B.hotstart([3, 11], 0.5)
    u, a = O.get_links().reshape(6, n, 4), O.get_higgs().reshape(2, n, 3)
    lib = L._L
    for ld in (n, n + 5):
        for got in (_get(lib, "lceq_get_links", L.h, n, 6, 4, ld),
                    _get(lib, "lceq_batch_get_links", B.h, n, 6, 4, ld, 1)):
            np.testing.assert_allclose(got, u, rtol=0, atol=1e-13)
        for got in (_get(lib, "lceq_get_higgs", L.h, n, 2, 3, ld),
                    _get(lib, "lceq_batch_get_higgs", B.h, n, 2, 3, ld, 1)):
            np.testing.assert_allclose(got, a, rtol=0, atol=1e-13)
    rng = np.random.default_rng(5)
    for ld in (n, n + 3):
        u, a = rng.normal(size=(6, n, 4)), rng.normal(size=(2, n, 3))
        _put(lib, "lceq_put_links", L.h, u, ld)
        _put(lib, "lceq_put_higgs", L.h, a, ld)
        _put(lib, "lceq_batch_put_links", B.h, u, ld, 1)
        _put(lib, "lceq_batch_put_higgs", B.h, a, ld, 1)
        assert np.array_equal(_get(lib, "lceq_get_links", L.h, n, 6, 4, n), u)
        assert np.array_equal(_get(lib, "lceq_get_higgs", L.h, n, 2, 3, n), a)
        assert np.array_equal(_get(lib, "lceq_batch_get_links", B.h, n, 6, 4, n, 1), u)
        assert np.array_equal(_get(lib, "lceq_batch_get_higgs", B.h, n, 2, 3, n, 1), a)
    L.close()
    B.close()


def test_transfers_of_several_threads():
    """Each thread its own lattice: the transfers share the pinned slots' pool."""
    import threading
    import lceqcd_amd
    print("field transfers of 4 threads", flush=True)
    bad = []

    def work(k):
        shape = (24 + 4 * k, 28, 24)
        n = shape[0] * shape[1] * shape[2] // 2
        rng = np.random.default_rng(k)
        L = lceqcd_amd.Lattice(*shape)
        for _ in range(5):
            u, a = rng.normal(size=(3, 2, n, 4)), rng.normal(size=(2, n, 3))
            L.put_links(u)
            L.put_higgs(a)
            if not (np.array_equal(L.get_links(), u) and np.array_equal(L.get_higgs(), a)):
                bad.append(k)
        L.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_history_ring_of_a_batch():
    """Rows asked for across the end of the batch's 1024-row history ring."""
    import lceqcd_amd
    print("batch history ring", flush=True)
    B = lceqcd_amd.Batch([(2, 2, 2), (4, 2, 2)])
    B.set_couplings([lceqcd_amd.couplings_from_trace_convention(9.0, 0.3, -0.9, 0.1)] * 2)
    B.hotstart([1, 2], 0.5)
    rows = []
    for k in (1000, 100):
        B.sweep(k, n_or=1, measflag=1)
        rows.append(B.history(k))
    assert np.array_equal(B.history(600)[500:], rows[1])
    assert np.array_equal(B.history(600)[:500], rows[0][500:])
    assert np.array_equal(B.observables(), rows[1][-1])
    B.close()


def test_pinned_blocks_are_used_again():
    """A pinned block that was given back is the next one taken, also when no
    lattice exists, and never by two at a time; the pool keeps a bounded number
    (csrc/lceq_transfer.hip KEEP and LEFT: 16 and 1 of the first kind)."""
    import gc
    import lceqcd_amd
    from lceqcd_amd import _lib
    lib = C.CDLL(_lib.load()._name)  # prototypes of its own
    take, give = lib._ZN4lceq11pinned_takeEii, lib._ZN4lceq11pinned_giveEPNS_6PinnedE
    host = lib._ZN4lceq11pinned_hostEPNS_6PinnedE
    take.restype, take.argtypes = C.c_void_p, [C.c_int, C.c_int]
    give.restype, give.argtypes = None, [C.c_void_p]
    host.restype, host.argtypes = C.c_void_p, [C.c_void_p]
    print("pinned blocks", flush=True)
    gc.collect()  # lattices of other tests
    L = lceqcd_amd.Lattice(4, 4, 4)
    for kind in range(3):
        blocks = [take(0, kind) for _ in range(3)]
        assert all(blocks) and len({host(b) for b in blocks}) == 3
        give(blocks[1])
        assert take(0, kind) == blocks[1]
        for b in blocks:
            give(b)
        again = [take(0, kind) for _ in range(3)]
        assert set(again) == set(blocks)
        for b in again:
            give(b)
    many = [take(0, 0) for _ in range(20)]
    for b in many:
        give(b)
    L.close()
    b = take(0, 0)
    assert b and host(b)
    C.memset(host(b), 0, 65536)
    give(b)
    assert take(0, 0) == b
    give(b)


@pytest.mark.parametrize("shape", [(2, 2, 2), (16, 16, 16), (52, 52, 52), (54, 54, 54)])
def test_arrays_of_a_lattice_are_apart(shape):
    """Up to 64 MiB a lattice's arrays share one allocation: what is written to
    each by its own calls leaves the others as they are, also when the link
    arrays have changed places."""
    import lceqcd_amd
    print("arrays of", shape, flush=True)
    n = shape[0] * shape[1] * shape[2] // 2
    rng = np.random.default_rng(2)
    fields = {"links": rng.normal(size=(3, 2, n, 4)), "higgs": rng.normal(size=(2, n, 3)),
              "links_fixed": rng.normal(size=(3, 2, n, 4)), "higgs_fixed": rng.normal(size=(2, n, 3))}
    L = lceqcd_amd.Lattice(*shape)
    L.set_couplings(9.0, 0.175, -0.45, 0.025)
    L.hotstart(3, 0.5)
    L.rng_philox(3, 0)
    L.sweep(0, 3, n_or=1, delta=0.4, measflag=1)
    rows = L.history(2)
    assert np.isfinite(rows).all()
    L.set_gauge_fixing(1.7, 1.0, 1e-300, 9)
    with pytest.raises(lceqcd_amd.LceqError, match="max_iter"):
        L.landau_gauge()
    for name, field in fields.items():
        getattr(L, "put_" + name)(field)
    L.correlator()
    L.polyakov()
    for name, field in fields.items():
        assert np.array_equal(getattr(L, "get_" + name)(), field)
    L.close()
