"""The calls a program makes of this package, as cases to be timed: what each stands for,
its inputs from a seed, one pass through the public entry points, the work that a pass
cannot do without, and its values in 64 bits from numpy alone.

`path` names the entry point of a case:

    spectrum   bse.bse_spectrum: eps(omega) from stored energies and activities
    plan       bse.BSEPlan: one whole matrix, k grid to eps(omega), execute() and results()
    zheev      bse.zheev: the eigensolver alone, on a host matrix
    bands      bse.BSEBands: exciton energies along a path of q-points
    batch      bse.BSEBatch: a set of uneven models
    lowest     bse.BSEPlan.lowest: the lowest excitons by the iterative solver

The models are the package's seeded random Wannier models (hexagonal 2D with 37 hopping
vectors, simple cubic with 33), their gap set to 2 eV on a coarse k grid.
"""
import math

import numpy as np

from wantibexos_amd import bse, tbmodel

GAP_GRID = {"hex": (6, 6, 1), "cubic": (4, 4, 4)}
# hexagonal Gamma-K-K'-Gamma, as pairs of segment ends
HEX_PATH = [(0.0, 0.0, 0.0), (0.6667, -0.3333, 0.0), (0.6667, -0.3333, 0.0), (0.3333, 0.3333, 0.0),
            (0.3333, 0.3333, 0.0), (0.0, 0.0, 0.0)]
EXACT_N3 = 2200.0 ** 3          # sum of N^3 up to which numpy's eigensolver takes a few seconds


def _plan(name, lattice, nw, n1, n2, n3, nc, nv, precision="fp64", nref=0, temp=0.0, numbse=1001):
    return dict(name=name, path="plan", lattice=lattice, nw=nw, n1=n1, n2=n2, n3=n3, nc=nc, nv=nv,
                precision=precision, nref=nref, temp=temp, numbse=numbse)


def listed():
    return [
        # the spectrum program on the stored activities of a small run: one short call
        dict(name="spectrum_576", path="spectrum", n=576, numbse=1001, renorm=True),
        # a first look at a 2D material on a coarse grid: launches and latency count
        _plan("plan_hex_576", "hex", 8, 12, 12, 1, 2, 2),
        # 3D crystal, finite temperature, uneven grid and band window
        _plan("plan_cubic_temp_1260", "cubic", 8, 7, 6, 5, 2, 3, temp=3000.0),
        # ZHEEV in place of the library's: eigenvalues, odd size
        dict(name="zheev_1001", path="zheev", n=1001, vectors=False),
        # ZHEEV with all its vectors
        dict(name="zheev_vectors_1290", path="zheev", n=1290, vectors=True),
        # an ordinary 2D run, odd grid
        _plan("plan_hex_2116", "hex", 12, 23, 23, 1, 2, 2),
        # the benchmark's matrix, plain form
        _plan("plan_hex_5184", "hex", 22, 36, 36, 1, 2, 2),
        # the benchmark's matrix, precision form with its refined lowest excitons
        _plan("plan_hex_5184_mixed", "hex", 22, 36, 36, 1, 2, 2, precision="mixed", nref=256),
        # a converged 2D grid: the largest single solve
        _plan("plan_hex_14400", "hex", 24, 60, 60, 1, 2, 2),
        # exciton bands, four points a segment, the plans kept
        dict(name="bands_1024", path="bands", nw=8, n1=16, n2=16, nc=2, nv=2, npts=4, lanes=4, precision="fp64"),
        # a set of uneven models in one call (N = 576 ... 2304)
        dict(name="batch_8", path="batch", models=8, nmin=12, nmax=24, wmin=6, wmax=12, lanes=4, precision="fp64"),
        # the iterative solver on the converged grid: lowest 256 excitons and eps(omega)
        dict(name="lowest_14400", path="lowest", nw=24, n1=60, n2=60, nc=2, nv=2, nev=256, tol=1e-6, lanczos=250),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["plan"] * 8 + ["plan_mixed"] * 2 + ["zheev"] * 3 + ["bands"] * 2 + ["batch"] * 2 + ["lowest", "spectrum"])
    if path == "spectrum":
        return dict(path=path, n=_log(rng, 100, 15000), numbse=rng.choice([501, 1001, 6001]), renorm=rng.random() < 0.7)
    if path == "zheev":
        vectors = rng.random() < 0.4
        return dict(path=path, n=_log(rng, 60, 1600 if vectors else 2500), vectors=vectors)
    if path == "bands":
        return dict(path=path, nw=rng.randint(6, 14), n1=rng.randint(8, 20), n2=rng.randint(8, 20), nc=rng.randint(1, 2),
                    nv=rng.randint(1, 2), npts=rng.randint(2, 5), lanes=rng.choice([1, 2, 4, 4]),
                    precision=rng.choice(["fp64", "fp64", "mixed"]))
    if path == "batch":
        nmin = rng.randint(8, 14)
        return dict(path=path, models=rng.randint(3, 12), nmin=nmin, nmax=nmin + rng.randint(2, 10), wmin=6,
                    wmax=rng.randint(8, 16), lanes=rng.choice([1, 2, 4, 4]), precision=rng.choice(["fp64", "fp64", "mixed"]))
    if path == "lowest":
        n = rng.randint(30, 56)
        return dict(path=path, nw=rng.randint(8, 24), n1=n, n2=n + rng.randint(-3, 3), nc=2, nv=2,
                    nev=rng.choice([64, 128, 256]), tol=1e-6, lanczos=rng.choice([150, 250]))
    mixed = path == "plan_mixed"
    nc, nv = rng.randint(1, 3), rng.randint(1, 3)
    N = _log(rng, 150, 10000)
    if rng.random() < 0.65:
        lattice, nw = "hex", rng.randint(6, 26)
        n1 = max(4, int(round(math.sqrt(N / (nc * nv) * math.exp(rng.uniform(-0.3, 0.3))))))
        n2, n3 = max(3, N // (nc * nv * n1)), 1
    else:
        lattice, nw = "cubic", rng.randint(6, 16)
        n1 = max(3, int(round((N / (nc * nv)) ** (1 / 3) * math.exp(rng.uniform(-0.2, 0.2)))))
        n2 = max(2, n1 + rng.randint(-1, 1))
        n3 = max(2, N // (nc * nv * n1 * n2))
    n = n1 * n2 * n3 * nc * nv
    nref = min(rng.choice([0, 64, 256]), n // 4) if mixed else 0
    c = _plan("", lattice, nw, n1, n2, n3, nc, nv, "mixed" if mixed else "fp64", nref,
              rng.choice([0.0, 0.0, 0.0, 300.0, 3000.0]), rng.choice([501, 1001, 1001, 3001]))
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _model(lattice, seed, nw):
    make = tbmodel.cubic3d if lattice == "cubic" else tbmodel.hex2d
    return make(seed, nw, GAP_GRID[lattice])


def _params(lattice, ngrid, nc, nv, precision="fp64", temp=0.0, numbse=1001, f154=True):
    pot = dict(coultype="V3DL", ediel=(6.0, 6.0, 6.0)) if lattice == "cubic" else dict(coultype="V2DRK", r0=40.0)
    hot = dict(bset=True, temp=temp, ta="VE", st=0.3, phavg=0.05) if temp > 0.0 else {}
    return bse.BSEParams(ngrid=ngrid, nc=nc, nv=nv, cshift=0.05, ebse0=0.0, ebsef=6.0, numbse=numbse, ktol=0.001,
                         dtfull=True, cpol=True, renorm=True, f154=f154,
                         precision=bse.MIXED if precision == "mixed" else bse.FP64, **pot, **hot)


def _hermitian(n, seed):
    """A dense matrix of the kind the BSE gives: transition energies of 2 to 10 eV on the
    diagonal, a coupling that spreads every state over many others."""
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = (a + a.conj().T) * (1.0 / math.sqrt(n))
    a[np.diag_indices(n)] = rng.uniform(2.0, 10.0, n)
    return a


def _spectrum_inputs(case, seed):
    rng = np.random.default_rng(seed)
    e = np.round(np.sort(rng.uniform(1.6, 12.0, case["n"])), 4)
    t = (rng.standard_normal((3, case["n"])) + 1j * rng.standard_normal((3, case["n"]))) * np.exp(-rng.uniform(0, 6, case["n"]))
    act = [(t[a] * t[b].conj()).real for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))]
    return e, np.round(np.array(act), 4)


def _batch_spec(case, seed):
    """(k grid, Wannier functions) of each model: sizes from the case, models from the seed."""
    m, span = case["models"], case["nmax"] - case["nmin"]
    return [(case["nmin"] + (i * span) // max(1, m - 1), case["wmin"] + (i * 5) % (case["wmax"] - case["wmin"] + 1))
            for i in range(m)]


def _qpath(rlat, npts):
    """Rows (path coordinate, qx, qy, qz): npts points on each segment of HEX_PATH."""
    ends = np.array(HEX_PATH) @ _recvec(rlat)
    rows, at = [], 0.0
    for a, b in zip(ends[0::2], ends[1::2]):
        t = np.arange(npts)[:, None] / (npts - 1.0)
        length = float(np.linalg.norm(b - a))
        rows.append(np.hstack([at + length * t, a + (b - a) * t]))
        at += length
    return np.vstack(rows)


class _State:
    """What the program keeps; released with its device memory."""

    def __init__(self, case, seed):
        self.case, self.ctx, self.obj = case, bse.Context(0), None
        p = case["path"]
        if p == "spectrum":
            self.e, self.act = _spectrum_inputs(case, seed)
            self.rlat = _spectrum_lattice()
        elif p == "zheev":
            self.a = _hermitian(case["n"], seed)
        elif p == "batch":
            spec = _batch_spec(case, seed)
            self.obj = bse.BSEBatch(self.ctx, [_model("hex", 100 * seed + i, nw) for i, (_, nw) in enumerate(spec)],
                                    [_params("hex", (n, n, 1), 2, 2, case["precision"]) for n, _ in spec], lanes=case["lanes"])
        elif p == "bands":
            m = _model("hex", seed, case["nw"])
            self.q = _qpath(m.rlat, case["npts"])
            self.obj = bse.BSEBands(self.ctx, m, _params("hex", (case["n1"], case["n2"], 1), case["nc"], case["nv"],
                                                         case["precision"]), lanes=case["lanes"])
        elif p == "lowest":
            m = _model("hex", seed, case["nw"])
            self.obj = bse.BSEPlan(self.ctx, m, _params("hex", (case["n1"], case["n2"], 1), case["nc"], case["nv"], "mixed",
                                                        f154=False))
        else:
            m = _model(case["lattice"], seed, case["nw"])
            self.obj = bse.BSEPlan(self.ctx, m, _plan_params(case))
            if case["nref"]:
                self.obj.set_refine(case["nref"])

    def __del__(self):
        if getattr(self, "obj", None) is not None:
            self.obj.close()
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


def _plan_params(case):
    return _params(case["lattice"], (case["n1"], case["n2"], case["n3"]), case["nc"], case["nv"], case["precision"],
                   case["temp"], case["numbse"])


def _spectrum_lattice():
    return np.array([[3.2, 0.0, 0.0], [-1.6, 2.7713, 0.0], [0.0, 0.0, 20.0]])


SPECTRUM_GRID = (12, 12, 1)
SPECTRUM = dict(ebse0=0.0, ebsef=6.0, sme=0.05)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    case, p = state.case, state.case["path"]
    if p == "spectrum":
        return bse.bse_spectrum(state.ctx, state.e, state.act, state.rlat, SPECTRUM_GRID, SPECTRUM["ebse0"], SPECTRUM["ebsef"],
                                case["numbse"], SPECTRUM["sme"], case["renorm"])
    if p == "zheev":
        return bse.zheev(state.ctx, state.a, vectors=case["vectors"])
    if p == "bands":
        return state.obj.run(state.q)
    if p == "batch":
        state.obj.execute()
        return [state.obj.results(i) for i in range(case["models"])]
    if p == "lowest":
        r = state.obj.lowest(nev=case["nev"], tol=case["tol"], lanczos_steps=case["lanczos"])
        return dict(W=r["W"], eps=r["eps"])     # resid and info are the solver's account of its own convergence
    state.obj.execute()
    return state.obj.results()


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------

def _plan_work(N, nk, nvec, nw, numbse, vectors=0, values_only=False):
    """One matrix from its model: H(k) and its derivatives, the band eigensolves, the matrix
    (its 8 N^2 / 2 flops of Hermitian products per orbital), the reduction to tridiagonal
    form (16/3 N^3 real flops), the tracked dipole vectors, eps(omega)."""
    flops = 8.0 * 4 * nk * nvec * nw * nw + 30.0 * nk * nw ** 3 + 8.0 * N * N / 2 + 16.0 / 3.0 * N ** 3
    flops += 16.0 * N * N * vectors
    if not values_only:
        flops += 3 * 16.0 * N * N + 6 * 10.0 * N * numbse
    b = 16.0 * nvec * nw * nw + 8.0 * N
    if not values_only:
        b += 8.0 * 8 * N + 96.0 * numbse
    return b, flops


def work(case):
    p = case["path"]
    if p == "spectrum":
        n, m = case["n"], case["numbse"]
        return {"bytes": 56.0 * n + 96.0 * m, "flops": 60.0 * n * m}
    if p == "zheev":
        n = float(case["n"])
        return {"bytes": (32.0 if case["vectors"] else 8.0) * n * n + 8.0 * n,
                "flops": (16.0 / 3.0 + (8.0 + 16.0 / 3.0 if case["vectors"] else 0.0)) * n ** 3}
    if p == "batch":
        w = [_plan_work(4.0 * g * g, g * g, 37, nw, 1001) for g, nw in _batch_spec(case, 0)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    if p == "bands":
        nk = case["n1"] * case["n2"]
        b, f = _plan_work(float(nk * case["nc"] * case["nv"]), nk, 37, case["nw"], 0, values_only=True)
        nq = 3 * case["npts"]
        return {"bytes": b * nq, "flops": f * nq}
    if p == "lowest":
        # about ten products of the matrix with a block of nev vectors, and the chains
        nk = case["n1"] * case["n2"]
        N = float(nk * case["nc"] * case["nv"])
        return {"bytes": 4.0 * N * N, "flops": 8.0 * N * N * (10 * case["nev"] + 9 * case["lanczos"])}
    nk = case["n1"] * case["n2"] * case["n3"]
    N = float(nk * case["nc"] * case["nv"])
    b, f = _plan_work(N, nk, 37 if case["lattice"] == "hex" else 33, case["nw"], case["numbse"], case["nref"])
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# values in 64 bits (numpy): the reference program's definitions, with the numbers that it
# holds in single precision rounded so here too
# ---------------------------------------------------------------------------

def _f32(x):
    return np.asarray(x, dtype=np.float64).astype(np.float32).astype(np.float64)


_PI32 = float(np.float32(math.pi))
_COULOMB = float(np.float32(-np.float32(0.0904756) * np.float32(1000.0)))
_KB = float(_f32(8.617330350e-5))


def _recvec(L):
    c = [np.cross(L[1], L[2]), np.cross(L[2], L[0]), np.cross(L[0], L[1])]
    return np.array(c) * (2.0 * _PI32 / abs(np.dot(L[0], c[0])))


def _kgrid(L, ngrid, q=(0.0, 0.0, 0.0)):
    b = _recvec(L)
    i, j, l = (x.ravel()[:, None] for x in np.meshgrid(*(np.arange(float(n)) for n in ngrid), indexing="ij"))
    return ((np.asarray(q)[None, :] + b[0] / ngrid[0] * i) + b[1] / ngrid[1] * j) + b[2] / ngrid[2] * l


def _bands(m, k, nc, nv, tcor):
    """Band window of nv valence and nc conduction states at every k: energies, vectors (with
    a real first component), H(R) phases."""
    rc = m.rvec @ m.rlat
    x = (k[:, 0:1] * rc[:, 0] + k[:, 1:2] * rc[:, 1]) + k[:, 2:3] * rc[:, 2]
    ph = np.exp(1j * _f32(x))
    hr = (m.hop + 1j * m.ihop) / m.ndeg[:, None, None]
    E, U = np.linalg.eigh(np.einsum("kr,rmn->kmn", ph, hr) - float(_f32(m.efermi)) * np.eye(m.nw))
    U = U * (np.conj(U[:, 0:1, :]) / np.abs(U[:, 0:1, :]))
    no = (E <= 0.0).sum(axis=1)
    E = E + (np.arange(m.nw)[None, :] >= no[:, None]) * (m.scs + tcor)
    at = no[:, None] - nv + np.arange(nc + nv)[None, :]
    return np.take_along_axis(E, at, 1), np.take_along_axis(U, at[:, None, :], 2).transpose(0, 2, 1), ph, hr


def _potential(p, L, dk):
    """V2DRK in vacuum (lc = ez = 1, w = 0: 1/(q (1 + r0 q))) and V3DL."""
    q = np.sqrt((dk[..., 0] ** 2 + dk[..., 1] ** 2) + dk[..., 2] ** 2)
    s = np.where(q < p.ktol, 1.0, q)
    area = np.linalg.norm(np.cross(L[0], L[1]))
    if p.coultype == "V2DRK":
        v = _COULOMB / (p.nk * area) / (1.0 + p.r0 * s) / s
    else:
        v = (_COULOMB / p.ediel[1]) / (p.nk * abs(np.dot(np.cross(L[0], L[1]), L[2]))) / (s * s)
    return np.where(q < p.ktol, 0.0, v)


def _matrix(m, p, k, ev, vv, ec, vc, q=None):
    """The Hermitian BSE matrix, and f_v - f_c of its basis states (k outer, c, v inner)."""
    nk, n = p.nk, p.dim
    pick = lambda c, v: (np.broadcast_to(x, (nk, p.nc, p.nv) + x.shape[3:]).reshape((n,) + x.shape[3:]) for x in (c[:, :, None], v[:, None]))
    de_c, de_v = pick(ec, ev)
    c, v = pick(vc, vv)
    V = _potential(p, m.rlat, k[:, None, :] - k[None, :, :])
    b = p.nc * p.nv
    ker = np.repeat(np.repeat(V, b, 0), b, 1) * (np.conj(c) @ c.T) * (np.conj(v) @ v.T)
    if q is not None and np.linalg.norm(q) != 0.0:
        a = np.einsum("nm,nm->n", np.conj(c), v)
        ker = ker - float(_potential(p, m.rlat, np.asarray(q)[None, :])[0]) * np.outer(a, np.conj(a))
    f = np.ones(n)
    if p.bset:
        fd = lambda e: 1.0 / (np.exp(np.minimum(e / (_KB * p.temp), 700.0)) + 1.0)
        f = fd(de_v) - fd(de_c)
    H = np.triu(ker * f[:, None], 1)
    H = H + H.conj().T
    H[np.diag_indices(n)] = de_c - de_v + np.diag(ker).real * f
    return H, f, c, v, de_c - de_v


def _round4(x):
    return np.array([float("%.4f" % v) for v in np.ravel(x)]).reshape(np.shape(x))


def _eps(e, act6, L, ngrid, ebse0, ebsef, numbse, sme, renorm):
    om = ebse0 + (ebsef - ebse0) * np.arange(numbse) / (numbse - 1.0)
    s = 0.0
    for a, b in zip(e[1:], e[:-1]):
        s = s + a - b
    s = 10.0 * (s / len(e)) + sme
    cell = abs(np.dot(np.cross(L[0], L[1]), L[2]))
    pre = float(np.float32(180.90)) / (float(np.float32(np.prod(ngrid))) * cell)
    out = np.zeros((6, 2, numbse))
    d = om[:, None] - e[None, :]
    den = d * d + s * s
    out[:, 0] = ((-d / den) @ act6.T).T * pre
    out[:3, 0] += 1.0
    out[:, 1] = ((s / den) @ act6.T).T * pre
    edge = e[0] - float(np.float32(0.15))
    if renorm and edge > 0.0:
        # zero up to the edge (the first point always), the first value above it taken off
        b = max(1, int(np.searchsorted(om, edge, side="right")))
        if b >= numbse:
            out[:, 1] = 0.0
        else:
            rest = out[:, 1, b:] - out[:, 1, b:b + 1]
            out[:, 1, :b] = 0.0
            out[:, 1, b:] = np.where(rest < 0.0, 0.0, rest)
    return out


def _exact_plan(m, p):
    tcor = 0.0
    if p.bset:
        tcor = float(-p.st * p.phavg * (1.0 / np.tanh(p.phavg / (2.0 * _KB * p.temp)) - 1.0))
    k = _kgrid(m.rlat, p.ngrid)
    E, U, ph, hr = _bands(m, k, p.nc, p.nv, tcor)
    H, f, c, v, de = _matrix(m, p, k, E[:, :p.nv], U[:, :p.nv], E[:, p.nv:], U[:, p.nv:])
    rc = _f32(m.rvec @ m.rlat)
    factor = (1.0 / (de + 1j * float(_f32(p.cshift)))).real
    ks = np.repeat(np.arange(p.nk), p.nc * p.nv)
    h = np.zeros((5, p.dim), dtype=np.complex128)
    for a in range(3):
        dH = np.einsum("kr,rmn->kmn", ph * (1j * rc[None, :, a]), hr)
        left = np.einsum("kcm,kmn->kcn", np.conj(U[:, p.nv:]), dH)
        h[a] = factor * np.einsum("kcn,kvn->kcv", left, U[:, :p.nv]).reshape(-1)
    r2 = float(np.float32(1.0) / np.sqrt(np.float32(2.0)))
    h[3], h[4] = (h[0] + 1j * h[1]) * r2, (h[0] - 1j * h[1]) * r2
    W, X = np.linalg.eigh(H)
    t, tf = h @ X, (h * f) @ X
    act = np.array([(t[a] * tf[b].conj()).real for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2), (3, 3), (4, 4))])
    e, a6 = (_round4(W), _round4(act[:6])) if p.f154 else (W, act[:6])
    eps = _eps(e, a6, m.rlat, p.ngrid, p.ebse0, p.ebsef, p.numbse, p.cshift, p.renorm)
    return dict(W=W, act=act, eps=eps, egap=float((E[:, p.nv] - E[:, p.nv - 1]).min()))


def exact(case, seed):
    p = case["path"]
    if p == "spectrum":
        e, act = _spectrum_inputs(case, seed)
        if case["n"] * case["numbse"] > 2e7:
            return None
        return _eps(e, act, _spectrum_lattice(), SPECTRUM_GRID, SPECTRUM["ebse0"], SPECTRUM["ebsef"], case["numbse"],
                    SPECTRUM["sme"], case["renorm"])
    if p == "zheev":
        if case["n"] ** 3 > EXACT_N3:
            return None
        a = _hermitian(case["n"], seed)
        if not case["vectors"]:
            return np.linalg.eigvalsh(a, UPLO="U")
        W, X = np.linalg.eigh(a, UPLO="U")
        return W, X * (np.conj(X[-1]) / np.abs(X[-1]))[None, :]
    if p == "batch":
        spec = _batch_spec(case, seed)
        if sum((4.0 * n * n) ** 3 for n, _ in spec) > EXACT_N3:
            return None
        return [_exact_plan(_model("hex", 100 * seed + i, nw), _params("hex", (n, n, 1), 2, 2, case["precision"]))
                for i, (n, nw) in enumerate(spec)]
    if p == "bands":
        N = case["n1"] * case["n2"] * case["nc"] * case["nv"]
        if 3 * case["npts"] * float(N) ** 3 > 2 * EXACT_N3:
            return None
        m = _model("hex", seed, case["nw"])
        prm = _params("hex", (case["n1"], case["n2"], 1), case["nc"], case["nv"], case["precision"])
        qp = _qpath(m.rlat, case["npts"])
        k = _kgrid(m.rlat, prm.ngrid)
        E, U, _, _ = _bands(m, k, prm.nc, prm.nv, 0.0)
        out = np.zeros((prm.dim, len(qp)))
        for i, q in enumerate(qp):
            Eq, Uq, _, _ = _bands(m, _kgrid(m.rlat, prm.ngrid, q[1:]), prm.nc, prm.nv, 0.0)
            H = _matrix(m, prm, k, E[:, :prm.nv], U[:, :prm.nv], Eq[:, prm.nv:], Uq[:, prm.nv:], q[1:])[0]
            out[:, i] = np.linalg.eigvalsh(H)
        return out
    if p == "lowest":
        return None                              # N from 3000 to 14400: numpy takes minutes
    if float(case["n1"] * case["n2"] * case["n3"] * case["nc"] * case["nv"]) ** 3 > EXACT_N3:
        return None
    return _exact_plan(_model(case["lattice"], seed, case["nw"]), _plan_params(case))
