"""The work that programs on this framework have it do, as measured cases.

A case is a dict of plain values; ``prepare`` builds what a program holds
before the call (a lattice with its fields, a replica batch, a model),
``run`` is one pass through the public entry points and returns everything
the pass produced or changed, ``work`` counts the bytes and operations the
pass cannot do without, and ``exact`` computes the same outputs with numpy in
64 bits from the definitions of the updates.

The kinds, and what each stands for:

routines    the update loop of a program that keeps the original's subroutine
            calls (ahiggs2, ahiggs3, agauge, renorm, then the averages), every
            call returning its host values
plain       the plain-method run: one production sweep at a time, its averages
            and the Polyakov loop read after every sweep
production  a block of production sweeps (1 heatbath + 4 overrelaxation
            + 1 Metropolis) between two measurements, its history rows, and
            the configuration to be saved
reference   the same block in the original's schedule (ahiggs2, ahiggs3,
            agauge, renorm), for either Higgs proposal width
landau      one saved configuration read back from its files, gauge-fixed to
            the Landau gauge, its correlators
correlators the three correlator measurements on a gauge-fixed configuration
scan        a phase-diagram scan: many lattices of uneven size and coupling
            swept together
learned     the same for the learned Higgs proposal, one network for all
train       training records taken from a configuration, then Adam steps
"""
import math
import os
import tempfile

import numpy as np

import lceqcd_amd
from lceqcd_amd import workloads

COUPLING = workloads.coupling(0.33, -0.9)        # broken phase, the production runs
REFERENCE_COUPLING = (9.0,) + lceqcd_amd.couplings_from_xy(9.0, 0.1, 0.5)
LEARNED_COUPLINGS = ((0.34, -0.9), (0.34, 0.2))  # broken phase and the transition
THERMALISE = 40  # sweeps from the hot start to the configuration that is gauge-fixed
MAX_HOST_CONF = 64 ** 3  # larger configurations start from a device hot start


# ------------------------------------------------------------------- cases

def listed():
    return [
        # smallest: a test-sized lattice, where launches and host calls are all there is
        {"name": "routines_8", "kind": "routines", "lx": 8, "ly": 8, "lz": 8, "loops": 1},
        # the plain-method run's lattice and cadence
        {"name": "plain_16", "kind": "plain", "lx": 16, "ly": 16, "lz": 16, "sweeps": 20},
        # the production lattice and its measurement spacing
        {"name": "production_64", "kind": "production", "lx": 64, "ly": 64, "lz": 64,
         "sweeps": 50},
        # a lattice whose fields no cache holds
        {"name": "production_160", "kind": "production", "lx": 160, "ly": 160, "lz": 160,
         "sweeps": 50},
        # the original's schedule at the production size
        {"name": "reference_64", "kind": "reference", "lx": 64, "ly": 64, "lz": 64, "sweeps": 50,
         "imode": 0},
        # and on a ragged lattice with the other proposal width
        {"name": "reference_22x18x50", "kind": "reference", "lx": 22, "ly": 18, "lz": 50,
         "sweeps": 20, "imode": 1},
        # the gauge-fixing run: tight limit, 32^3
        {"name": "landau_32", "kind": "landau", "lx": 32, "ly": 32, "lz": 32, "limit": 1e-12},
        # the measurement of the production run
        {"name": "landau_64", "kind": "landau", "lx": 64, "ly": 64, "lz": 64, "limit": 1e-10},
        # correlators of the long production lattice
        {"name": "correlators_32x32x128", "kind": "correlators", "lx": 32, "ly": 32, "lz": 128},
        # a quarter of the replica scan: six shapes, 24 couplings
        {"name": "scan_24", "kind": "scan", "replicas": 24, "first": 0, "sweeps": 16},
        # the learned proposal on eight lattices at two couplings
        {"name": "learned_8x48", "kind": "learned", "lx": 48, "ly": 48, "lz": 48, "replicas": 8,
         "sweeps": 8},
        # training from one 48^3 configuration
        {"name": "train_48", "kind": "train", "lx": 48, "ly": 48, "lz": 48, "stride": 2,
         "steps": 200, "batch": 4096},
    ]


def _even(rng, lo, hi):
    """An even extent, spread over the logarithm of the range."""
    return 2 * int(round(math.exp(rng.uniform(math.log(lo / 2), math.log(hi / 2)))))


def _extents(rng, lo, hi, volume):
    while True:
        e = {k: _even(rng, lo, hi) for k in ("lx", "ly", "lz")}
        if e["lx"] * e["ly"] * e["lz"] <= volume:
            return e


def draw(rng):
    kind = rng.choice(["routines", "plain", "production", "production", "reference", "reference",
                       "landau", "correlators", "scan", "learned", "train"])
    c = {"kind": kind}
    if kind == "routines":
        c.update(_extents(rng, 4, 96, 64 ** 3), loops=rng.randint(1, 4))
    elif kind == "plain":
        c.update(_extents(rng, 6, 64, 48 ** 3), sweeps=rng.randint(5, 30))
    elif kind == "production":
        c.update(_extents(rng, 6, 180, 160 ** 3), sweeps=rng.randint(4, 20))
    elif kind == "reference":
        c.update(_extents(rng, 6, 128, 96 ** 3), sweeps=rng.randint(4, 40),
                 imode=rng.randint(0, 1))
    elif kind == "landau":
        c.update(_extents(rng, 4, 48, 32 ** 3), limit=10.0 ** -rng.uniform(8, 12))
    elif kind == "correlators":
        c.update(_extents(rng, 4, 160, 64 ** 3))
    elif kind == "scan":
        n = rng.randint(2, 24)
        c.update(replicas=n, first=rng.randint(0, 96 - n), sweeps=rng.randint(3, 20))
    elif kind == "learned":
        c.update(_extents(rng, 6, 64, 48 ** 3), replicas=rng.randint(1, 8),
                 sweeps=rng.randint(2, 10))
    else:
        e = _extents(rng, 16, 64, 48 ** 3)
        sites = e["lx"] * e["ly"] * e["lz"]
        stride = rng.randint(1, 4)
        most = max(1, sites // stride // 32)  # batches of at most the records, a multiple of 32
        batch = 32 * min(most, int(round(math.exp(rng.uniform(math.log(8), math.log(256))))))
        c.update(e, stride=stride, steps=rng.randint(20, 200), batch=batch)
    return c


# ------------------------------------------------------------------ inputs

def _shape(case):
    return (case["lx"], case["ly"], case["lz"])


def _qmul(p, q, dp=False, dq=False):
    """Products of SU(2) elements held as (Re a, Im a, Re b, Im b) in the last axis."""
    p0, p1, p2, p3 = (p[..., i] for i in range(4))
    q0, q1, q2, q3 = (q[..., i] for i in range(4))
    if dp:
        p1, p2, p3 = -p1, -p2, -p3
    if dq:
        q1, q2, q3 = -q1, -q2, -q3
    return np.stack([p0 * q0 - p1 * q1 - p2 * q2 - p3 * q3, p0 * q1 + p1 * q0 + p2 * q3 - p3 * q2,
                     p0 * q2 - p1 * q3 + p2 * q0 + p3 * q1, p0 * q3 + p1 * q2 - p2 * q1 + p3 * q0],
                    axis=-1)


def _rotate(u, b, transposed=False):
    """R(u) b of the adjoint representation, u = c0 + i c.sigma."""
    c0, c = u[..., 0:1], np.stack([u[..., 3], u[..., 2], u[..., 1]], axis=-1)
    s = c0 * c0 - np.sum(c * c, axis=-1, keepdims=True)
    k = 2.0 * np.sum(c * b, axis=-1, keepdims=True)
    w = 2.0 * c0 if transposed else -2.0 * c0
    return s * b + k * c + w * np.cross(c, b)


class _Sites:
    """Checkerboard numbering: index s = x/2 + (lx/2) y + (lx ly/2) z within a parity."""

    def __init__(self, shape):
        lx, ly, lz = shape
        h1, h2 = lx // 2, lx * ly // 2
        self.shape, self.n, self.h2 = shape, h2 * lz, h2
        s = np.arange(self.n)
        z, y, xh = s // h2, (s % h2) // h1, s % h1
        self.full, self.up, self.dn = [], [], []  # flat site; neighbours' indices (other parity)
        for p in range(2):
            x = 2 * xh + ((p + y + z) & 1)
            at = [x, y, z]
            self.full.append(x + lx * (y + ly * z))
            moves = []
            for step in (1, -1):
                m = []
                for mu in range(3):
                    c = list(at)
                    c[mu] = (c[mu] + step) % shape[mu]
                    m.append(c[0] // 2 + h1 * c[1] + h2 * c[2])
                moves.append(m)
            self.up.append(moves[0])
            self.dn.append(moves[1])


def _configuration(shape, seed, higgs):
    """A configuration with the plaquettes and Higgs lengths of a thermal one,
    in a random gauge: smooth links and a Higgs field about one direction."""
    lx, ly, lz = shape
    rng = np.random.default_rng(seed)
    v = lx * ly * lz

    def unit(q):
        return q / np.linalg.norm(q, axis=-1, keepdims=True)

    g = unit(rng.normal(size=(lz, ly, lx, 4)))
    sites = _Sites(shape)
    u = np.empty((3, 2, v // 2, 4))
    for mu in range(3):
        h = rng.normal(size=(lz, ly, lx, 4)) * 0.13
        h[..., 0] = 1.0
        w = _qmul(_qmul(g, unit(h)), np.roll(g, -1, axis=2 - mu), dq=True).reshape(v, 4)
        for p in range(2):
            u[mu, p] = w[sites.full[p]]
    length, spread = higgs
    b = rng.normal(size=(lz, ly, lx, 3)) * spread
    b[..., 2] += length
    b = _rotate(g, b).reshape(v, 3)
    return u, np.stack([b[sites.full[p]] for p in range(2)])


BROKEN, SYMMETRIC = (4.0, 0.7), (0.0, 0.15)  # Higgs length and spread of the two phases


def _fill(lattice, shape, seed, higgs=BROKEN):
    if shape[0] * shape[1] * shape[2] <= MAX_HOST_CONF:
        u, a = _configuration(shape, seed, higgs)
        lattice.put_links(u)
        lattice.put_higgs(a)
    else:
        lattice.hotstart(seed, 0.5)


def _lattice(shape, seed, coupling, higgs=BROKEN):
    lattice = lceqcd_amd.Lattice(*shape)
    lattice.set_couplings(*coupling)
    _fill(lattice, shape, seed, higgs)
    lattice.rng_philox(seed, 0)
    return lattice


def _weights(seed):
    """A model state: Glorot-uniform weights, zero biases, identity normalisation."""
    rng = np.random.default_rng(seed + 77)
    parts = []
    for fan_in, fan_out, gain in ((10, 64, 1.0), (64, 64, 1.0), (64, 6, 0.1)):
        lim = gain * math.sqrt(6.0 / (fan_in + fan_out))
        parts += [rng.uniform(-lim, lim, fan_in * fan_out), np.zeros(fan_out)]
    return np.concatenate(parts + [np.zeros(10), np.ones(10)]).astype(np.float32)


def _scan(case):
    """Shapes, couplings and Philox keys of a run of the replica scan."""
    k, n = case["first"], case["replicas"]
    shapes, coup, seeds, _ = workloads.c4_replicas(k + n)
    return shapes[k:], coup[k:], seeds[k:]


def _learned(case):
    n = case["replicas"]
    pairs = [LEARNED_COUPLINGS[0 if r < (n + 1) // 2 else 1] for r in range(n)]
    return [_shape(case)] * n, [workloads.coupling(a, b) for a, b in pairs]


def _batch(shapes, coup, seed, seeds):
    batch = lceqcd_amd.Batch(shapes)
    batch.set_couplings(coup)
    for r, shape in enumerate(shapes):
        u, a = _configuration(shape, seed * 1000 + r, BROKEN)
        batch.put_links(r, u)
        batch.put_higgs(r, a)
    batch.rng_philox([s + seed for s in seeds])
    return batch


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("routines", "reference"):
        lattice = _lattice(_shape(case), seed, REFERENCE_COUPLING, SYMMETRIC)
        lattice.set_imode(case.get("imode", 0))
        return {"case": case, "lattice": lattice}
    if kind in ("plain", "production"):
        return {"case": case, "lattice": _lattice(_shape(case), seed, COUPLING), "delta": 0.4}
    if kind == "landau":
        folder = tempfile.TemporaryDirectory(prefix="conf_")
        names = [os.path.join(folder.name, f) for f in ("u_conf", "a_conf")]
        lattice = lceqcd_amd.Lattice(*_shape(case))
        lattice.set_couplings(*COUPLING)
        # a configuration of a chain: how long the fixing takes depends on its
        # long waves, which the made-up configuration does not have
        lattice.hotstart(seed, 0.5)
        lattice.rng_philox(seed, 0)
        lattice.sweep(lceqcd_amd.SWEEP_KP_OR_METRO, THERMALISE, n_or=4, delta=0.4, measflag=0)
        lattice.confsave(*names)
        lattice.set_gauge_fixing(1.7, 1.0, case["limit"], 10000000)
        return {"case": case, "lattice": lattice, "folder": folder, "files": names}
    if kind == "correlators":
        lattice = lceqcd_amd.Lattice(*_shape(case))
        u, a = _configuration(_shape(case), seed, BROKEN)
        lattice.put_higgs(a)
        lattice.put_links_fixed(u)
        lattice.put_higgs_fixed(a)
        return {"case": case, "lattice": lattice}
    if kind == "scan":
        shapes, coup, seeds = _scan(case)
        return {"case": case, "batch": _batch(shapes, coup, seed, seeds), "delta": 0.4}
    if kind == "learned":
        shapes, coup = _learned(case)
        mlp = lceqcd_amd.Mlp()
        mlp.set_state(_weights(seed))
        return {"case": case, "mlp": mlp,
                "batch": _batch(shapes, coup, seed, range(31000, 31000 + len(shapes)))}
    lattice = _lattice(_shape(case), seed, COUPLING)
    lattice.ahiggs1(0.4, 1)  # sets the step size the collection uses
    return {"case": case, "lattice": lattice, "mlp": lceqcd_amd.Mlp(), "weights": _weights(seed)}


# --------------------------------------------------------------------- runs

def _fields(lattice):
    return {"links": lattice.get_links(), "higgs": lattice.get_higgs()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("scan", "learned"):
        batch, n = state["batch"], case["sweeps"]
        if kind == "scan":
            batch.sweep(n, n_or=4, delta=state["delta"], measflag=1)
            state["delta"] = None  # from here on the batch's own steps
        else:
            batch.sweep_mlp(state["mlp"], n, n_or=4, measflag=1)
        return {"history": batch.history(n), "averages": batch.observables(),
                "links": [batch.get_links(r) for r in range(batch.nrep)],
                "higgs": [batch.get_higgs(r) for r in range(batch.nrep)]}
    lattice = state["lattice"]
    if kind == "routines":
        accepted = []
        for _ in range(case["loops"]):
            accepted += [lattice.ahiggs2(1), lattice.ahiggs3(1), lattice.agauge(1)]
            lattice.renorm()
        return {"accepted": np.array(accepted), "averages": lattice.observables(),
                **_fields(lattice)}
    if kind == "plain":
        rows, loops = [], []
        for _ in range(case["sweeps"]):
            state["delta"] = lattice.sweep(lceqcd_amd.SWEEP_KP_OR_METRO, 1, n_or=4,
                                           delta=state["delta"], measflag=1)
            rows.append(lattice.history(1)[0])
            loops.append(np.append(*reversed(lattice.polyakov())))
        return {"history": np.array(rows), "polyakov": np.array(loops), "delta": state["delta"],
                **_fields(lattice)}
    if kind == "production":
        n = case["sweeps"]
        state["delta"] = lattice.sweep(lceqcd_amd.SWEEP_KP_OR_METRO, n, n_or=4,
                                       delta=state["delta"], measflag=1)
        return {"history": lattice.history(n), "delta": state["delta"], **_fields(lattice)}
    if kind == "reference":
        n = case["sweeps"]
        lattice.sweep(lceqcd_amd.SWEEP_REFERENCE, n, measflag=1)
        return {"history": lattice.history(n), **_fields(lattice)}
    if kind == "landau":
        lattice.oldconf(*state["files"])
        da, iterations = lattice.landau_gauge()
        return {"da": da, "iterations": iterations, "correlators": list(lattice.correlator()),
                "scalar": list(lattice.scalarcorr()), "links": lattice.get_links_fixed(),
                "higgs": lattice.get_higgs_fixed()}
    if kind == "correlators":
        return {"correlators": list(lattice.correlator()), "scalar": list(lattice.scalarcorr()),
                "polyakov": list(lattice.polyakov()), "averages": lattice.observables()}
    mlp = state["mlp"]
    mlp.set_state(state["weights"])
    mlp.clear()
    mlp.collect(lattice, nsteps=8, stride=case["stride"])
    loss = mlp.train(case["steps"], batch=case["batch"], lr=2e-3, seed=1)
    # the losses are means of single-precision values
    return {"loss": loss.astype(np.float32), "state": mlp.get_state(),
            "higgs": lattice.get_higgs()}


# --------------------------------------------------------------------- work

# operations per link or site of one update, a multiply-add as two: the staple
# (8 products), norms, the new link, two hopping actions, and the functions
# at about 20 each; six rotations for the Higgs force
LINK_OR, LINK_KP, HIGGS, GAUGE_FIX = 340, 520, 260, 380
NETWORK = 2 * (10 * 64 + 64 * 64 + 64 * 6)
FIELD = 120  # bytes of links and Higgs field per site


def work(case):
    kind = case["kind"]
    if kind in ("scan", "learned"):
        shapes = _scan(case)[0] if kind == "scan" else _learned(case)[0]
        v = sum(x * y * z for x, y, z in shapes)
        extra = 2 * NETWORK + 200 if kind == "learned" else 0
        # fields in and out of the chain, and out to the host
        return {"bytes": 3 * FIELD * v,
                "flops": v * case["sweeps"] * (3 * (LINK_KP + 4 * LINK_OR) + HIGGS + extra)}
    v = case["lx"] * case["ly"] * case["lz"]
    if kind in ("routines", "reference"):
        n = case["loops"] if kind == "routines" else case["sweeps"]
        return {"bytes": 3 * FIELD * v, "flops": v * n * (3 * (LINK_KP + 12) + 2 * HIGGS + 80)}
    if kind in ("plain", "production"):
        f = 3 * (LINK_KP + 4 * LINK_OR) + HIGGS + (30 if kind == "plain" else 0)
        return {"bytes": 3 * FIELD * v, "flops": v * case["sweeps"] * f}
    if kind == "landau":
        # as many iterations as the overrelaxation needs are not known before
        # the call; ten per site of the longest extent is a lower bound
        n = 10 * max(_shape(case))
        return {"bytes": 4 * FIELD * v, "flops": v * n * GAUGE_FIX}
    if kind == "correlators":
        return {"bytes": (FIELD + 24) * v, "flops": 60 * v}
    records = 2 * -(-v // 2 // case["stride"])
    return {"bytes": FIELD * v + 24 * v + 2 * 52 * records,
            "flops": 8 * HIGGS * v + 3 * NETWORK * case["batch"] * case["steps"]}


# ------------------------------------------------------------ 64-bit results

MOST_SITE_UPDATES = 8_000_000  # of the numpy updates below, about 20 s


def _philox(idx, stream, pair, number, key):
    """Philox4x32-10 draws 2 pair and 2 pair + 1 of every index in one pass."""
    m32 = np.uint64(0xFFFFFFFF)
    c = [idx.astype(np.uint64), np.full(idx.shape, (stream << 8) | pair, np.uint64),
         np.full(idx.shape, number & 0xFFFFFFFF, np.uint64),
         np.full(idx.shape, number >> 32, np.uint64)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF

    def uniform(hi, lo):
        x = (hi << np.uint64(20)) | (lo >> np.uint64(12))
        return (2 * x + np.uint64(1)).astype(np.float64) * 2.0 ** -53

    return uniform(c[0], c[1]), uniform(c[2], c[3])


def _dot(x, y):
    return np.sum(x * y, axis=-1)


def _hotstart(shape, key, sigma):
    """Haar links and normal Higgs components from their Philox streams."""
    n = shape[0] * shape[1] * shape[2] // 2

    def normals(cls, stream):
        idx = cls * n + np.arange(n)
        u = _philox(idx, stream, 0, 0, key) + _philox(idx, stream, 1, 0, key)
        r0, r1 = np.sqrt(-2.0 * np.log(u[0])), np.sqrt(-2.0 * np.log(u[2]))
        t0, t1 = 2.0 * np.pi * u[1], 2.0 * np.pi * u[3]
        return np.stack([r0 * np.cos(t0), r0 * np.sin(t0), r1 * np.cos(t1), r1 * np.sin(t1)],
                        axis=-1)

    u = np.stack([normals(cls, 1) for cls in range(6)]).reshape(3, 2, n, 4)
    a = sigma * np.stack([normals(p, 2)[:, :3] for p in range(2)])
    return u / np.sqrt(_dot(u, u))[..., None], a


class _Chain:
    """The updates on one lattice in numpy."""

    def __init__(self, shape, u, a, coupling, key, imode=0):
        self.sites = _Sites(shape)
        self.u, self.a = u.copy(), a.copy()
        self.beta, self.beta_a, self.beta_2, self.beta_4 = coupling
        self.key, self.number, self.imode = key, 0, imode
        self.n, self.v = self.sites.n, 2 * self.sites.n
        self.obs = np.zeros(16)

    def draws(self, count):
        idx = np.arange(self.n)
        out = []
        for pair in range((count + 1) // 2):
            out += _philox(idx, 0, pair, self.number, self.key)
        self.number += 1
        return out[:count]

    def staple(self, eo, mu):
        u, oe = self.u, 1 - eo
        up, dn = self.sites.up, self.sites.dn
        xm = up[eo][mu]
        total = np.zeros((self.n, 4))
        for nu in range(3):
            if nu == mu:
                continue
            xp, xn = up[eo][nu], dn[eo][nu]
            total += _qmul(u[nu, oe][xm], _qmul(u[mu, oe][xp], u[nu, eo], True, True))
            far = dn[oe][nu][xm]
            total += _qmul(u[nu, eo][far], _qmul(u[mu, oe][xn], u[nu, oe][xn], True), True)
        return total

    def link_sweep(self, heatbath, unit_on_write):
        plaq = hits = accepts = 0.0
        for eo in range(2):
            for mu in range(3):
                v = self.staple(eo, mu)
                t = 1.0 / np.sqrt(_dot(v, v))
                vh = t[:, None] * v
                u = self.u[mu, eo]
                a, b = self.a[eo], self.a[1 - eo][self.sites.up[eo][mu]]
                old = -self.beta_a * _dot(a, _rotate(u, b))
                if heatbath:
                    r1, r2, r3, r4, r5, r6, accept = self.draws(7)
                    cc = np.cos(2.0 * np.pi * r3)
                    a0 = -(np.log(r1) + np.log(r2) * cc * cc) * t / self.beta
                    hit = r4 * r4 <= 1.0 - 0.5 * a0
                    hits += hit.sum()
                    a0 = np.where(hit, 1.0 - a0, _qmul(u, vh)[:, 0])
                    a1 = np.sqrt(np.maximum(1.0 - a0 * a0, 0.0))
                    c = 2.0 * (r5 - 0.5)
                    s = a1 * np.sqrt(np.maximum(1.0 - c * c, 0.0))
                    w = np.stack([a0, a1 * c, s * np.sin(2.0 * np.pi * r6),
                                  s * np.cos(2.0 * np.pi * r6)], axis=-1)
                    new = _qmul(w, vh, dq=True)
                else:
                    accept, = self.draws(1)
                    adj = vh * np.array([1.0, -1.0, -1.0, -1.0])
                    new = 2.0 * _dot(u, adj)[:, None] * adj - u
                change = old + self.beta_a * _dot(a, _rotate(new, b))
                ok = np.exp(change) >= accept
                accepts += ok.sum()
                if unit_on_write:
                    new = new / np.sqrt(_dot(new, new))[:, None]
                u = np.where(ok[:, None], new, u)
                self.u[mu, eo] = u
                plaq += _qmul(u, v)[:, 0].sum()
        v = self.v
        self.obs[12], self.obs[13], self.obs[0] = hits, accepts, plaq / (12.0 * v)
        self.obs[7] = (hits / (3.0 * v)) * (accepts / (12.0 * v)) if heatbath \
            else accepts / (3.0 * v)
        return self.obs[7]

    def force(self, eo):
        oe, f = 1 - eo, np.zeros((self.n, 3))
        for mu in range(3):
            xp, xd = self.sites.up[eo][mu], self.sites.dn[eo][mu]
            f += _rotate(self.u[mu, eo], self.a[oe][xp])
            f += _rotate(self.u[mu, oe][xd], self.a[oe][xd], True)
        return f

    def higgs(self, kind, eo, delta=0.0):
        """One parity of ahiggs1, 2 or 3: accepts, sums of rho, rho^2 and a.F."""
        f, a = self.force(eo), self.a[eo]
        ro = _dot(a, a)
        if kind == 1:
            *r, accept = self.draws(4)
            an = a + (np.stack(r, axis=-1) - 0.5) * delta
            rn = _dot(an, an)
            change = self.beta_a * (_dot(an, f) - _dot(a, f)) + self.beta_2 * (ro - rn)
        else:
            width, alph = self.beta_2, 0.0
            if self.imode:
                f2 = self.beta_a * _dot(f, f)
                alph = self.beta_4 * f2 / (2.0 * (self.beta_2 + self.beta_4 * f2) ** 2)
                width = self.beta_2 + alph
            mean = self.beta_a * f * np.reshape(0.5 / width, (-1, 1))
            if kind == 2:
                *w, accept = self.draws(7)
                an = mean + np.stack([np.sqrt(-np.log(w[2 * i]) / width)
                                      * np.cos(2.0 * np.pi * w[2 * i + 1]) for i in range(3)],
                                     axis=-1)
            else:
                accept, = self.draws(1)
                an = 2.0 * mean - a
            rn = _dot(an, an)
            change = -alph * (ro - rn)
        ok = np.exp(change + self.beta_4 * (ro * ro - rn * rn)) >= accept
        a = np.where(ok[:, None], an, a)
        ro = np.where(ok, rn, ro)
        self.a[eo] = a
        return np.array([ok.sum(), ro.sum(), (ro * ro).sum(), _dot(a, f).sum()])

    def higgs_sweep(self, kind, delta=0.0):
        s = self.higgs(kind, 0, delta) + self.higgs(kind, 1, delta)
        self.obs[8], self.obs[2], self.obs[3] = s[:3] / self.v
        self.obs[1] = s[3] / (6.0 * self.v)
        return self.obs[8]

    def metropolis(self):
        accept = self.higgs_sweep(1, self.obs[11])
        if abs(accept - 0.5) > 0.1:
            self.obs[11] *= 1.1131241 if accept > 0.5 else 0.8989669

    def renorm(self):
        self.u /= np.sqrt(_dot(self.u, self.u))[..., None]

    def production_sweep(self):
        self.link_sweep(True, True)
        for _ in range(4):
            self.link_sweep(False, True)
        self.metropolis()
        return self.obs.copy()

    def reference_sweep(self):
        accepted = [self.higgs_sweep(2), self.higgs_sweep(3), self.link_sweep(True, False)]
        row = self.obs.copy()
        self.renorm()
        return row, accepted


def _correlators(shape, uf, af, a):
    """The z-correlators and means of correlator, scalarcorr and polyakov."""
    lx, ly, lz = shape
    h2 = lx * ly // 2

    def slices(x):  # (2, n) -> mean per z
        return x.reshape(2, lz, h2).sum(axis=(0, 2)) / (lx * ly)

    def periodic(x):
        return np.array([np.mean(x * np.roll(x, -z)) for z in range(lz)])

    fa = [slices(af[:, :, i]) for i in range(3)]
    fu = [[slices(uf[mu, :, :, c]) for c in (1, 3, 2)] for mu in range(3)]
    rho = _dot(a, a)
    sc, po = slices(rho), slices(np.cos(4.0 * np.sqrt(rho)))
    per_mu = [sum(periodic(x) for x in fu[mu]) for mu in range(3)]
    corr = [sum(periodic(x) for x in fa), (per_mu[0] + per_mu[1]) / 2.0, per_mu[2]]
    return (corr, [float(sc.mean()), periodic(sc)], [float(po.mean() ** 2), periodic(po)],
            np.array([x.mean() for x in fa]))


def _landau(shape, u, a, limit, most):
    """Overrelaxed Landau gauge fixing; None if it takes over `most` iterations."""
    sites, u, a = _Sites(shape), u.copy(), a.copy()
    conj = np.array([1.0, -1.0, -1.0, -1.0])
    for it in range(1, most + 1):
        for eo in range(2):
            oe, dn = 1 - eo, sites.dn[eo]
            back = [u[mu, oe][dn[mu]] for mu in range(3)]
            s1, s2 = sum(u[mu, eo] for mu in range(3)), sum(back)
            w = s1 + conj * s2
            if eo:
                da = np.sum((s1 - s2)[:, 1] ** 2 + w[:, 2] ** 2 + w[:, 3] ** 2) / sites.n
            o = w / np.sqrt(_dot(w, w))[:, None]
            r = np.clip(o[:, 0], -1.0, 1.0)
            th = np.arccos(r)
            sn = np.sqrt((1.0 - r) * (1.0 + r))
            f = np.where(sn > 0.0, np.sin(1.7 * th) / np.where(sn > 0.0, sn, 1.0), 0.0)
            g = -f[:, None] * o
            g[:, 0] = np.where(th != 0.0, np.cos(1.7 * th), o[:, 0])
            g = np.where((th != 0.0)[:, None], g, o)
            a[eo] = _rotate(g, a[eo])
            for mu in range(3):
                u[mu, eo] = _qmul(g, u[mu, eo])
                u[mu, oe][dn[mu]] = _qmul(back[mu], g, dq=True)
        u /= np.sqrt(_dot(u, u))[..., None]
        if not da > limit:
            return u, a, float(da), it
    return None


def _features(f, a, coupling):
    """Rows of the network's inputs and the frame they are in."""
    fn = np.sqrt(_dot(f, f))
    e1 = f / fn[:, None]
    h = np.where(np.abs(e1[:, 2:]) >= 0.9, [[1.0, 0.0, 0.0]], [[0.0, 0.0, 1.0]])
    e2 = np.cross(h, e1)
    e2 /= np.sqrt(_dot(e2, e2))[:, None]
    frame = np.stack([e1, e2, np.cross(e1, e2)], axis=1)
    y = np.einsum("nij,nj->ni", frame, a)
    zero = np.zeros_like(fn)
    x = np.stack([y[:, 0], y[:, 1], y[:, 2], fn, zero, zero, fn] + [zero + c for c in coupling[1:]],
                 axis=-1)
    return x, frame


def _splitmix(x):
    m = (1 << 64) - 1
    x = (x + 0x9E3779B97F4A7C15) & m
    z = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return x, z ^ (z >> 31)


def _train(x, y, state, steps, batch, lr, seed):
    """Adam on the negative log-likelihood of the moves, in 64 bits."""
    w = state[:5254].astype(np.float64)
    mean, sd = x.mean(axis=0), x.std(axis=0)
    mean = mean.astype(np.float32).astype(np.float64)
    inv = np.where(sd > 1e-6, 1.0 / np.where(sd > 1e-6, sd, 1.0), 1.0)
    inv = inv.astype(np.float32).astype(np.float64)
    m1, m2, n, pos, loss = np.zeros_like(w), np.zeros_like(w), len(x), len(x), []
    cuts = np.cumsum([640, 64, 4096, 64, 384])
    for t in range(1, steps + 1):
        if pos + batch > n:
            while True:
                seed, z = _splitmix(seed)
                mult = (z % n) | 1
                if math.gcd(mult, n) == 1:
                    break
            seed, z = _splitmix(seed)
            offs, pos = z % n, 0
        idx = [(mult * (pos + b) + offs) % n for b in range(batch)]
        pos += batch
        xb, yb = (x[idx] - mean) * inv, y[idx]
        w1, b1, w2, b2, w3, b3 = np.split(w, cuts)
        w1, w2, w3 = w1.reshape(10, 64), w2.reshape(64, 64), w3.reshape(64, 6)
        z1 = xb @ w1 + b1
        g1 = 1.0 / (1.0 + np.exp(-z1))
        z2 = (z1 * g1) @ w2 + b2
        g2 = 1.0 / (1.0 + np.exp(-z2))
        o = (z2 * g2) @ w3 + b3
        s = np.clip(o[:, 3:], -7.0, 4.0)
        r = (yb - o[:, :3]) * np.exp(-s)
        loss.append(np.mean(np.sum(s + 0.5 * r * r, axis=1)))
        d = np.concatenate([-r * np.exp(-s), np.where(s == o[:, 3:], 1.0 - r * r, 0.0)],
                           axis=1) / batch
        d2 = (d @ w3.T) * g2 * (1.0 + z2 * (1.0 - g2))
        d1 = (d2 @ w2.T) * g1 * (1.0 + z1 * (1.0 - g1))
        g = np.concatenate([(xb.T @ d1).ravel(), d1.sum(axis=0), ((z1 * g1).T @ d2).ravel(),
                            d2.sum(axis=0), ((z2 * g2).T @ d).ravel(), d.sum(axis=0)])
        m1 = 0.9 * m1 + 0.1 * g
        m2 = 0.999 * m2 + 0.001 * g * g
        w = w - lr * (m1 / (1.0 - 0.9 ** t)) / (np.sqrt(m2 / (1.0 - 0.999 ** t)) + 1e-8)
    return np.array(loss), np.concatenate([w, mean, inv])


def exact(case, seed):
    kind = case["kind"]
    if kind == "learned":
        return None  # a bf16 network proposes; its accepted moves have no 64-bit value
    if kind == "scan":
        shapes, coup, keys = _scan(case)
        n = case["sweeps"]
        if sum(x * y * z for x, y, z in shapes) // 2 * 33 * n > MOST_SITE_UPDATES:
            return None
        rows, links, higgs = [], [], []
        for r, shape in enumerate(shapes):
            c = _Chain(shape, *_configuration(shape, seed * 1000 + r, BROKEN), coup[r],
                       keys[r] + seed)
            c.obs[11] = 0.4
            rows.append([c.production_sweep() for _ in range(n)])
            links.append(c.u)
            higgs.append(c.a)
        rows = np.array(rows).transpose(1, 0, 2)
        return {"history": rows, "averages": rows[-1], "links": links, "higgs": higgs}
    shape = _shape(case)
    n = shape[0] * shape[1] * shape[2] // 2
    passes = {"routines": 10 * case.get("loops", 0), "reference": 10 * case.get("sweeps", 0),
              "plain": 33 * case.get("sweeps", 0), "production": 33 * case.get("sweeps", 0),
              "landau": 33 * THERMALISE, "train": 18}.get(kind, 1)
    if n * passes > MOST_SITE_UPDATES or 2 * n > MAX_HOST_CONF:
        return None
    symmetric = kind in ("routines", "reference")
    u, a = _configuration(shape, seed, SYMMETRIC if symmetric else BROKEN)
    if kind == "correlators":
        corr, scalar, loop, a0f = _correlators(shape, u, a, a)
        return {"correlators": corr, "scalar": scalar, "polyakov": loop,
                "averages": {"plaq0": 0.0, "a0kin": 0.0, "a02": 0.0, "a04": 0.0, "a0f": a0f}}
    if kind == "landau":
        chain = _Chain(shape, *_hotstart(shape, seed, 0.5), COUPLING, seed)
        chain.obs[11] = 0.4
        for _ in range(THERMALISE):
            chain.production_sweep()
        a = chain.a
        done = _landau(shape, chain.u, a, case["limit"], MOST_SITE_UPDATES // 4 // n)
        if done is None:
            return None
        uf, af, da, it = done
        corr, scalar, _, _ = _correlators(shape, uf, af, a)
        return {"da": da, "iterations": it, "correlators": corr, "scalar": scalar, "links": uf,
                "higgs": af}
    chain = _Chain(shape, u, a, REFERENCE_COUPLING if symmetric else COUPLING, seed,
                   case.get("imode", 0))
    if kind == "routines":
        accepted = []
        for _ in range(case["loops"]):
            accepted += chain.reference_sweep()[1]
        o = chain.obs
        return {"accepted": np.array(accepted), "links": chain.u, "higgs": chain.a,
                "averages": {"plaq0": o[0], "a0kin": o[1], "a02": o[2], "a04": o[3],
                             "a0f": o[4:7]}}
    if kind == "reference":
        rows = [chain.reference_sweep()[0] for _ in range(case["sweeps"])]
        return {"history": np.array(rows), "links": chain.u, "higgs": chain.a}
    chain.obs[11] = 0.4
    if kind == "train":
        chain.metropolis()
        xs, ys = [], []
        for eo in range(2):
            pick = slice(None, None, case["stride"])
            f = chain.force(eo)[pick]
            x, frame = _features(f, chain.a[eo][pick], COUPLING)
            for _ in range(8):
                chain.higgs(1, eo, chain.obs[11])
            xs.append(x)
            ys.append(np.einsum("nij,nj->ni", frame, chain.a[eo][pick]))
        x, y = (np.concatenate(v).astype(np.float32).astype(np.float64) for v in (xs, ys))
        if case["steps"] * case["batch"] > 2_000_000:
            return None
        loss, state = _train(x, y, _weights(seed), case["steps"], case["batch"], 2e-3, 1)
        return {"loss": loss, "state": state, "higgs": chain.a}
    rows, loops = [], []
    for _ in range(case["sweeps"]):
        rows.append(chain.production_sweep())
        if kind == "plain":
            _, _, loop, _ = _correlators(shape, u, a, chain.a)
            loops.append(np.append(loop[1], loop[0]))
    out = {"history": np.array(rows), "delta": float(chain.obs[11]), "links": chain.u,
           "higgs": chain.a}
    if kind == "plain":
        out["polyakov"] = np.array(loops)
    return out
