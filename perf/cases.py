"""The work this framework is used for, as measurable cases over its public entry points.

A case is one pass of a user's program:

- md: a slice of a running simulation of one system (atvh_md_run through `System.run`), from 500
  atoms, where a step is launches and latency, to the 2,048,000-atom fluid; LJ and charged (LJ +
  real-space Coulomb + PME), FP64 and mixed, NVE and Nose-Hoover, with the thermo record and the
  snapshot a program writes at the end of the slice;
- npt: the same under the MTK barostat (`System.npt`);
- frame: one single-point evaluation of a new frame (upload, list build, forces, energy and virial),
  what a re-analysis of stored frames or an outer optimiser does;
- ladder: an ensemble of independent systems advanced together (`Batch` with graph replay);
- serve: MD segments submitted to a `Server` and fetched when done.

Mixed runs hand their snapshots on in 32 bits, as trajectory files hold them; FP64 runs in 64.
Positions start a quarter of a lattice constant off the box faces, displaced thermally.

`exact` restates each pass in 64-bit torch: a cell-list MD with velocity Verlet + Nose-Hoover (or
MTK), shifted LJ, erfc Coulomb and smooth PME, none of it through this package.
"""
import itertools
import math

import numpy as np
import torch

import atomiverse_amd as av
from atomiverse_amd.workloads import LJWorkload

KB = 8.617333262e-5       # eV/K
MVV2E = 103.6427          # amu Å^2/fs^2 -> eV
QQR2E = 14.399645         # e^2/Å -> eV
TAU = math.sqrt(MVV2E)    # fs, the LJ time unit of eps = 1 eV, sigma = 1 Å, m = 1 amu
DT = 0.005 * TAU
SKIN = 0.3


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest system of the replica ladder: a step is launch latency
        dict(name="lj_500_nve_fp64", kind="md", n=500, charged=False, mixed=False, nvt=False, steps=200),
        # the 4000-atom NVE fluid of the reference's own benchmark, default precision
        dict(name="lj_4000_nve_fp64", kind="md", n=4000, charged=False, mixed=False, nvt=False, steps=200),
        # a mid-size fluid: enough bricks for part of the chip only
        dict(name="lj_32000_nvt_mixed", kind="md", n=32000, charged=False, mixed=True, nvt=True, steps=100),
        # a ragged large system (not a whole lattice: void at the top), plain precision
        dict(name="lj_499999_nvt_fp64", kind="md", n=499999, charged=False, mixed=False, nvt=True, steps=60),
        # the headline workload of the benchmark
        dict(name="lj_2048000_nvt_mixed", kind="md", n=2048000, charged=False, mixed=True, nvt=True, steps=100),
        # a charged serving-size melt on a mesh that is no power of two
        dict(name="melt_8000_nvt_mixed", kind="md", n=8000, charged=True, mixed=True, nvt=True, steps=100,
             spacing=1.0 / 1.2, order=4),
        # a mid-size melt in plain precision (80^3 mesh)
        dict(name="melt_110592_nvt_fp64", kind="md", n=110592, charged=True, mixed=False, nvt=True, steps=50,
             spacing=0.65, order=4),
        # the 512,000-ion melt with the 128^3 mesh
        dict(name="melt_512000_nvt_mixed", kind="md", n=512000, charged=True, mixed=True, nvt=True, steps=50,
             spacing=0.65, order=4),
        # single points of new two-species frames: upload, list, forces, energy, virial
        dict(name="frame_131072_two_types_fp64", kind="frame", n=131072, charged=False, mixed=False),
        # the MTK regression of the reference (216 atoms, the small-grid list)
        dict(name="npt_216_fp64", kind="npt", n=216, steps=80),
        # the 256-system replica ladder
        dict(name="ladder_256_mixed", kind="ladder", members=256, lo=500, hi=20000, steps=100),
        # a handful of served segments, LJ and charged
        dict(name="serve_6_fp64", kind="serve", segments=6, lo=1000, hi=20000, steps=400),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "melt", "melt", "frame", "npt", "ladder", "serve"])
    if kind == "md":
        n = _log_int(rng, 500, 1500000)
        return dict(kind="md", n=n, charged=False, mixed=rng.random() < 0.5, nvt=rng.random() < 0.6,
                    steps=rng.randrange(50, 101))
    if kind == "melt":
        side = 2 * _log_int(rng, 5, 36)
        return dict(kind="md", n=side ** 3, charged=True, mixed=rng.random() < 0.5, nvt=rng.random() < 0.6,
                    steps=rng.randrange(30, 51), spacing=rng.choice([0.65, 1.0 / 1.2]),
                    order=rng.choice([4, 4, 5, 6]))
    if kind == "frame":
        charged = rng.random() < 0.4
        n = (2 * _log_int(rng, 5, 32)) ** 3 if charged else _log_int(rng, 500, 600000)
        c = dict(kind="frame", n=n, charged=charged, mixed=rng.random() < 0.5)
        return dict(c, spacing=0.65, order=4) if charged else c
    if kind == "npt":
        return dict(kind="npt", n=rng.randrange(5, 12) ** 3, steps=rng.randrange(50, 91))
    if kind == "ladder":
        return dict(kind="ladder", members=rng.randrange(8, 129), lo=500, hi=rng.randrange(2000, 20001),
                    steps=rng.randrange(50, 101))
    return dict(kind="serve", segments=rng.randrange(2, 7), lo=1000, hi=rng.randrange(4000, 20001),
                steps=rng.randrange(100, 401))


# ---------------------------------------------------------------- inputs

def _velocities(rng, n, T_star):
    v = rng.standard_normal((3, n))
    v -= v.mean(axis=1, keepdims=True)
    t = MVV2E * float((v * v).sum()) / (3 * n - 3)
    return v * math.sqrt(T_star / t)


def _lj_system(n, seed, T_star=0.72, nvt=True, rho=0.8442):
    """FCC sites in lattice order, the first n of them, in the box of density rho."""
    rng = np.random.default_rng(seed)
    L = (n / rho) ** (1.0 / 3.0)
    nc = math.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-12)
    a = L / nc
    k = np.arange(n)
    cell, site = k // 4, k % 4
    basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])[site]
    c = np.stack([cell % nc, (cell // nc) % nc, cell // (nc * nc)])
    x = (c + basis.T + 0.25) * a + 0.05 * rng.standard_normal((3, n))
    v = _velocities(rng, n, T_star)
    return LJWorkload("lj", x[0], x[1], x[2], v[0], v[1], v[2], np.ones(n), np.array([L, L, L]), dt=DT,
                      T=T_star / KB, tau_T=0.5 * TAU, thermostat=int(nvt))


def _melt(n, seed, nvt=True, spacing=0.65, order=4, T_star=1.2, rho=0.9, cutoff=3.0):
    """Rock salt on a cubic grid, +-1 reduced charges, species of sigma 1.0 and 0.8."""
    rng = np.random.default_rng(seed)
    side = round(n ** (1.0 / 3.0))
    a = (1.0 / rho) ** (1.0 / 3.0)
    L = side * a
    g = np.arange(side)
    c = np.stack(np.meshgrid(g, g, g, indexing="ij")).reshape(3, -1)
    x = (c + 0.5) * a + 0.05 * rng.standard_normal((3, n))
    t = (c.sum(axis=0) & 1).astype(np.int32)
    q = np.where(t == 0, 1.0, -1.0) / math.sqrt(QQR2E)
    v = _velocities(rng, n, T_star)
    return LJWorkload("melt", x[0], x[1], x[2], v[0], v[1], v[2], np.ones(n), np.array([L, L, L]), cutoff=cutoff,
                      dt=DT, T=T_star / KB, tau_T=0.5 * TAU, thermostat=int(nvt), type_=t, charge=q, pair="ljcoul",
                      eps_tab=np.array([[1.0, 0.0], [0.0, 1.0]]), sigma_tab=np.array([[1.0, 0.0], [0.0, 0.8]]),
                      set_tab=np.array([[1, 0], [0, 1]], np.int32), alpha=(1.35 - 0.15 * math.log(1e-5)) / cutoff,
                      pme_spacing=spacing, pme_order=order)


def _two_types(n, seed):
    """A binary LJ mixture (Lorentz-Berthelot, sigma 1.0 / 0.9, eps 1.0 / 0.8)."""
    w = _lj_system(n, seed, nvt=False)
    w.type_ = (np.random.default_rng(seed + 1).random(n) < 0.4).astype(np.int32)
    w.eps_tab = np.array([[1.0, math.sqrt(0.8)], [math.sqrt(0.8), 0.8]])
    w.sigma_tab = np.array([[1.0, 0.95], [0.95, 0.9]])
    return w


def _npt_system(n, seed):
    """Simple cubic at rho 0.8 (the MTK regression's), thermal velocities at T* = 1."""
    rng = np.random.default_rng(seed)
    side = round(n ** (1.0 / 3.0))
    L = (n / 0.8) ** (1.0 / 3.0)
    g = (np.arange(side) + 0.5) * (L / side)
    x = np.stack(np.meshgrid(g, g, g, indexing="ij")).reshape(3, -1) + 0.03 * rng.standard_normal((3, n))
    v = _velocities(rng, n, 1.0)
    return LJWorkload("npt", x[0], x[1], x[2], v[0], v[1], v[2], np.ones(n), np.array([L, L, L]), dt=0.02,
                      T=1.0 / KB, tau_T=2.0, delay=10)


NPT = dict(tau_P=20.0, P_target=0.0, mt=3, mp=3)


def _members(case, seed):
    """What a ladder or a request set holds: sizes log-uniform (the case's own, whatever the seed), the
    ladder's temperatures geometric."""
    k = case["members"] if case["kind"] == "ladder" else case["segments"]
    rng = np.random.default_rng([k, case["hi"]])
    sizes = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), k)).astype(int)
    out = []
    for i, n in enumerate(sizes):
        if case["kind"] == "serve" and i % 3 == 2:
            side = 2 * max(5, round(n ** (1.0 / 3.0) / 2))
            out.append(_melt(side ** 3, seed * 1000 + i, spacing=1.0 / 1.2))
        else:
            t = 0.7 * (1.5 / 0.7) ** (i / max(k - 1, 1)) if case["kind"] == "ladder" else 0.72
            out.append(_lj_system(int(n), seed * 1000 + i, T_star=t))
    return out


def _workload(case, seed):
    if case["kind"] == "npt":
        return _npt_system(case["n"], seed)
    if case["charged"]:
        return _melt(case["n"], seed, case.get("nvt", False), case["spacing"], case["order"])
    return _two_types(case["n"], seed) if case["kind"] == "frame" else _lj_system(case["n"], seed, nvt=case["nvt"])


# ---------------------------------------------------------------- prepare and run

def _configured(ctx, w):
    s = av.System(ctx, w.n, w.box)
    s.nlist_configure(w.cutoff, w.skin, w.every, w.delay, True)
    if w.pair == "ljcoul":
        s.pair_ljcoul(w.eps_tab, w.sigma_tab, w.set_tab, w.alpha, w.cutoff)
        s.pme(w.alpha, w.pme_spacing, w.pme_order)
    elif w.eps_tab is not None:
        s.pair_lj(1.0, 1.0, w.cutoff, w.eps_tab, w.sigma_tab)
    else:
        s.pair_lj(w.eps, w.sigma, w.cutoff)
    return s


def _upload(s, w):
    s.upload(w.x, w.y, w.z, w.mass, w.vx, w.vy, w.vz, type_=w.type_, charge=w.charge)


def _started(ctx, w, precision, virial=False):
    """A system as a program holds it between slices: frame, list, integrator, current forces."""
    s = _configured(ctx, w)
    _upload(s, w)
    s.integrator(w.dt, w.thermostat, w.T, w.tau_T, 0)
    s.nlist_build()
    s.compute(precision, virial, virial)
    return s


def prepare(case, seed):
    ctx = av.Context(0)
    kind = case["kind"]
    mixed = kind == "ladder" or case.get("mixed", False)
    prec = av.PREC_MIXED if mixed else av.PREC_FP64
    st = dict(case=case, ctx=ctx, prec=prec, mixed=mixed)
    if kind == "ladder":
        st["systems"] = [_started(ctx, w, prec) for w in _members(case, seed)]
        st["batch"] = av.Batch(ctx, st["systems"])
        st["batch"].set_graph(True)
    elif kind == "serve":
        st["work"] = _members(case, seed)
        st["server"] = av.Server(ctx, 64 << 30, 100, prec)
    elif kind == "frame":
        st["w"] = _workload(case, seed)
        st["sys"] = _configured(ctx, st["w"])
    elif kind == "npt":
        w = _workload(case, seed)
        st["sys"] = s = _started(ctx, w, prec, virial=True)
        s.npt(w.dt, w.T, w.tau_T, NPT["P_target"], NPT["tau_P"], mtchain=NPT["mt"], mpchain=NPT["mp"])
    else:
        st["sys"] = _started(ctx, _workload(case, seed), prec)
    return st


EVERY = 10  # steps between energy records


def _kept(a, mixed):
    """An output as the program keeps it: mixed runs in 32 bits."""
    return torch.from_numpy(a).float() if mixed else a


def run(state):
    case, prec, mixed = state["case"], state["prec"], state["mixed"]
    kind = case["kind"]
    if kind == "md":
        s, k = state["sys"], case["steps"]
        s.run(k, prec, energy_every=EVERY)
        d = s.download()
        pe, ke = s.thermo(k)
        out = {key: _kept(d[key], mixed) for key in ("x", "y", "z", "vx", "vy", "vz")}
        if not mixed:
            out.update(fx=d["fx"], fy=d["fy"], fz=d["fz"])
        out["pe"], out["ke"] = _kept(pe, mixed), _kept(ke, mixed)
        return out
    if kind == "npt":
        s, k = state["sys"], case["steps"]
        s.run(k, prec)
        out = s.download()
        out["pe"], out["ke"] = s.thermo(k)
        out["H"], out["V"] = s.npt_thermo(k)
        out["box"] = s.current_box()
        return out
    if kind == "frame":
        s = state["sys"]
        _upload(s, state["w"])
        s.nlist_build()
        s.compute(prec, True, True)
        pe, vir, _ = s.energy()
        d = s.download()
        return {"fx": _kept(d["fx"], mixed), "fy": _kept(d["fy"], mixed), "fz": _kept(d["fz"], mixed),
                "pe": _kept(np.array([pe]), mixed), "virial": _kept(vir, mixed)}
    if kind == "ladder":
        state["batch"].run(case["steps"], prec)
        got = [s.download() for s in state["systems"]]
        return {key: _kept(np.concatenate([d[key] for d in got]), mixed) for key in ("x", "y", "z", "vx", "vy", "vz")}
    srv, out = state["server"], {}
    ids = [srv.submit(w, case["steps"] + 50 * (i % 3)) for i, w in enumerate(state["work"])]
    left = set(ids)
    while left:
        srv.advance()
        for sid in srv.poll():
            out[sid] = srv.fetch(sid)
            left.discard(sid)
    got = [out[i] for i in ids]
    return {key: np.concatenate([np.atleast_1d(d[key]) for d in got])
            for key in ("x", "y", "z", "vx", "vy", "vz", "pe", "ke")}


# ---------------------------------------------------------------- what a pass cannot do without

def _step_work(n, charged, spacing=0.65):
    """One MD step: the state (x, v, f) read and written once; 27 flops a pair inside the cutoff
    (each pair once), 12 more with Coulomb, and spread, two transforms and gather of PME."""
    pairs = n * (0.9 * 18.0 * math.pi if charged else 0.8442 * 10.42 * math.pi) / 1.5
    bytes_, flops = n * 18 * 8, pairs * (39 if charged else 27) + 40 * n
    if charged:
        mesh = n / 0.9 / spacing ** 3
        flops += n * 64 * 8 + 5 * mesh * math.log2(max(mesh, 2)) + 10 * mesh
        bytes_ += 16 * mesh
    return bytes_, flops


def work(case):
    kind = case["kind"]
    if kind == "ladder":
        lo, hi = case["lo"], case["hi"]
        n = case["members"] * (hi - lo) / math.log(hi / lo)
        b, f = _step_work(n, False)
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if kind == "serve":
        lo, hi = case["lo"], case["hi"]
        n = case["segments"] * (hi - lo) / math.log(hi / lo)
        b, f = _step_work(2 * n / 3, False)
        c, g = _step_work(n / 3, True, 1.0 / 1.2)
        return {"bytes": (b + c) * case["steps"], "flops": (f + g) * case["steps"]}
    if kind == "frame":
        b, f = _step_work(case["n"], case["charged"], case.get("spacing", 0.65))
        return {"bytes": case["n"] * 16 * 8, "flops": 1.5 * f}
    b, f = _step_work(case["n"], case.get("charged", False), case.get("spacing", 0.65))
    return {"bytes": b * case["steps"], "flops": f * case["steps"]}


# ---------------------------------------------------------------- the same in 64-bit torch

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _half_pairs(x, box, rcut):
    """Index pairs (i < j) closer than rcut under the periodic box; x is (n, 3)."""
    n = x.shape[0]
    nc = [max(1, int(L / rcut)) for L in box.tolist()]
    if min(nc) < 3:
        i, j = torch.triu_indices(n, n, 1, device=x.device)
        d = x[i] - x[j]
        d -= box * torch.round(d / box)
        keep = (d * d).sum(1) < rcut * rcut
        return i[keep], j[keep]
    ncell = torch.tensor(nc, device=x.device)
    c = torch.minimum((x / box * ncell).long(), ncell - 1)
    cid = (c[:, 0] * nc[1] + c[:, 1]) * nc[2] + c[:, 2]
    order = torch.argsort(cid)
    count = torch.bincount(cid, minlength=nc[0] * nc[1] * nc[2])
    start = torch.cumsum(count, 0) - count
    m = int(count.max())
    slot = torch.arange(n, device=x.device) - start[cid[order]]
    table = torch.full((count.numel(), m), -1, dtype=torch.long, device=x.device)
    table[cid[order], slot] = order
    grid = torch.stack(torch.meshgrid(*[torch.arange(k, device=x.device) for k in nc], indexing="ij"), -1).reshape(-1, 3)
    out = []
    half = [o for o in itertools.product((-1, 0, 1), repeat=3) if o >= (0, 0, 0)]
    for o in half:
        g = (grid + torch.tensor(o, device=x.device)) % ncell
        other = (g[:, 0] * nc[1] + g[:, 1]) * nc[2] + g[:, 2]
        for b in range(0, table.shape[0], 200000):
            a_ = table[b:b + 200000]
            b_ = table[other[b:b + 200000]]
            i = a_[:, :, None].expand(-1, m, m).reshape(-1)
            j = b_[:, None, :].expand(-1, m, m).reshape(-1)
            ok = (i >= 0) & (j >= 0)
            if o == (0, 0, 0):
                ok &= i < j
            i, j = i[ok], j[ok]
            d = x[i] - x[j]
            d -= box * torch.round(d / box)
            keep = (d * d).sum(1) < rcut * rcut
            out.append((i[keep], j[keep]))
    return torch.cat([p[0] for p in out]), torch.cat([p[1] for p in out])


def _bspline(u, n):
    """Cardinal B-spline M_n(u) on tensors."""
    if n == 2:
        return torch.clamp(1.0 - torch.abs(u - 1.0), min=0.0)
    return u / (n - 1) * _bspline(u, n - 1) + (n - u) / (n - 1) * _bspline(u - 1.0, n - 1)


def _mesh_size(n):
    n = max(n, 4)
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


class _Field:
    """Forces, energy and virial of one system at given positions."""

    def __init__(self, w, dev):
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.dev, self.rc = dev, w.cutoff
        self.x = torch.stack([t(w.x), t(w.y), t(w.z)], 1)
        self.v = torch.stack([t(w.vx), t(w.vy), t(w.vz)], 1)
        self.box = t(w.box)
        self.q = None if w.charge is None else t(w.charge)
        eps, sig = np.array([[w.eps]]), np.array([[w.sigma]])
        if w.eps_tab is not None:
            eps, sig = w.eps_tab.copy(), w.sigma_tab.copy()
            for a, b in itertools.product(range(2), repeat=2):
                if w.set_tab is not None and not w.set_tab[a, b]:
                    eps[a, b] = math.sqrt(eps[a, a] * eps[b, b])
                    sig[a, b] = 0.5 * (sig[a, a] + sig[b, b])
        self.type = torch.zeros(w.n, dtype=torch.long, device=dev)
        if w.type_ is not None:
            self.type = torch.as_tensor(w.type_, device=dev).long()
        self.eps, self.s6 = t(eps).reshape(-1), t(sig).reshape(-1) ** 6
        r6 = self.s6 / self.rc ** 6
        self.shift = 4.0 * self.eps * (r6 * r6 - r6)
        self.nt = eps.shape[0]
        self.pairs, self.skin = None, 0.6
        self.alpha, self.order = w.alpha, w.pme_order
        if self.order:
            self.K = [_mesh_size(max(math.ceil(L / w.pme_spacing), self.order + 1)) for L in w.box]
            self.H = self._influence()

    def _influence(self):
        mod, freq = [], []
        for K, L in zip(self.K, self.box.tolist()):
            k = torch.arange(self.order - 1, dtype=torch.float64, device=self.dev)
            m = torch.arange(K, dtype=torch.float64, device=self.dev)
            b = (_bspline(k + 1.0, self.order) * torch.exp(2j * math.pi * m[:, None] * k / K)).sum(1)
            b2 = torch.abs(b) ** 2
            inv = torch.where(b2 > 1e-12, 1.0 / b2, torch.zeros_like(b2))
            fix = 0.5 * (torch.roll(inv, 1) + torch.roll(inv, -1))
            mod.append(torch.where(inv == 0.0, fix, inv))
            freq.append(torch.where(m <= K // 2, m, m - K) / L)
        m2 = freq[0][:, None, None] ** 2 + freq[1][None, :, None] ** 2 + freq[2][None, None, :] ** 2
        self.m = [f.reshape([-1 if a == d else 1 for a in range(3)]) for d, f in enumerate(freq)]
        self.m2 = m2
        H = torch.exp(-math.pi ** 2 * m2 / self.alpha ** 2) / m2
        H = H * mod[0][:, None, None] * mod[1][None, :, None] * mod[2][None, None, :]
        H[0, 0, 0] = 0.0
        return H

    def _pme(self, x, ev):
        n, vol = self.order, float(self.box.prod())
        idx, th, dth = [], [], []
        for d in range(3):
            K = self.K[d]
            s = x[:, d] / self.box[d]
            u = (s - torch.floor(s)) * K
            u0 = torch.floor(u)
            j = torch.arange(n, device=self.dev)
            arg = (u - u0)[:, None] + (n - 1 - j)
            th.append(_bspline(arg, n))
            dth.append((_bspline(arg, n - 1) - _bspline(arg - 1.0, n - 1)) * (K / self.box[d]))
            idx.append((u0.long()[:, None] - (n - 1) + j) % K)
        flat = ((idx[0][:, :, None, None] * self.K[1] + idx[1][:, None, :, None]) * self.K[2] + idx[2][:, None, None, :])
        w = th[0][:, :, None, None] * th[1][:, None, :, None] * th[2][:, None, None, :]
        grid = torch.zeros(self.K[0] * self.K[1] * self.K[2], dtype=torch.float64, device=self.dev)
        grid.index_add_(0, flat.reshape(-1), (self.q[:, None, None, None] * w).reshape(-1))
        F = torch.fft.fftn(grid.reshape(self.K))
        phi = torch.fft.ifftn(F * self.H).real.reshape(-1) * grid.numel()
        v = phi[flat]
        pre = -QQR2E / (math.pi * vol) * self.q
        f = torch.stack([pre * (v * dth[0][:, :, None, None] * th[1][:, None, :, None] * th[2][:, None, None, :]).sum((1, 2, 3)),
                         pre * (v * th[0][:, :, None, None] * dth[1][:, None, :, None] * th[2][:, None, None, :]).sum((1, 2, 3)),
                         pre * (v * th[0][:, :, None, None] * th[1][:, None, :, None] * dth[2][:, None, None, :]).sum((1, 2, 3))], 1)
        if not ev:
            return f, 0.0, None
        ug = self.H * torch.abs(F) ** 2
        scale = QQR2E / (2.0 * math.pi * vol)
        vt = -2.0 * (1.0 / torch.where(self.m2 == 0, torch.ones_like(self.m2), self.m2) + math.pi ** 2 / self.alpha ** 2)
        vir = []
        for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)):
            vir.append(float((ug * (vt * self.m[a] * self.m[b] + (1.0 if a == b else 0.0))).sum()) * scale)
        e = float(ug.sum()) * scale - QQR2E * self.alpha / math.sqrt(math.pi) * float((self.q ** 2).sum())
        e -= QQR2E * math.pi / (2.0 * vol * self.alpha ** 2) * float(self.q.sum()) ** 2
        return f, e, np.array(vir)

    def __call__(self, ev=False):
        x, box = self.x, self.box
        stale = self.pairs is None
        if not stale:
            d = x - self.x0 * (box / self.box0)
            stale = float((d * d).sum(1).max()) > (0.45 * self.skin) ** 2
        if stale:
            self.pairs = _half_pairs(x - box * torch.floor(x / box), box, self.rc + self.skin)
            self.x0, self.box0 = x.clone(), box.clone()
        i, j = self.pairs
        d = x[i] - x[j]
        d -= box * torch.round(d / box)
        r2 = (d * d).sum(1)
        keep = r2 < self.rc * self.rc
        i, j, d, r2 = i[keep], j[keep], d[keep], r2[keep]
        ab = self.type[i] * self.nt + self.type[j] if self.nt > 1 else None
        eps, s6, shift = (self.eps, self.s6, self.shift) if ab is None else (self.eps[ab], self.s6[ab], self.shift[ab])
        r6 = s6 / r2 ** 3
        fp = 24.0 * eps * (2.0 * r6 * r6 - r6) / r2
        e = 4.0 * eps * (r6 * r6 - r6) - shift
        if self.q is not None:
            r = torch.sqrt(r2)
            qq = QQR2E * self.q[i] * self.q[j]
            ec = torch.special.erfc(self.alpha * r) / r
            fp = fp + qq * (ec + 2.0 / math.sqrt(math.pi) * self.alpha * torch.exp(-(self.alpha * r) ** 2)) / r2
            e = e + qq * ec
        df = fp[:, None] * d
        f = torch.zeros_like(x)
        f.index_add_(0, i, df)
        f.index_add_(0, j, df, alpha=-1.0)
        pe, vir = 0.0, None
        if ev:
            pe = float(e.sum())
            vir = np.array([float((d[:, a] * df[:, b]).sum()) for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))])
        if self.order:
            fk, ek, vk = self._pme(x, ev)
            f, pe = f + fk, pe + ek
            vir = vir + vk if ev else None
        return f, pe, vir


def _verlet(w, steps, every, dev, cold=False):
    """Velocity Verlet (+ Nose-Hoover) from the frame of w: final state, pe and ke records. cold: a
    served segment, whose frame carries no forces for its first half kick."""
    F = _Field(w, dev)
    f = torch.zeros_like(F.x) if cold else F()[0]
    ndof = 3 * w.n - 3
    kT = KB * w.T
    Q, xi = ndof * kT * w.tau_T ** 2, 0.0
    pe, ke = np.full(steps, np.nan), np.full(steps, np.nan)

    def thermostat():
        nonlocal xi
        e = 0.5 * MVV2E * float((F.v * F.v).sum())
        if not w.thermostat:
            return e
        xi += 0.5 * w.dt * (2.0 * e - ndof * kT) / Q
        s = math.exp(-0.5 * w.dt * xi)
        F.v *= s
        return e * s * s

    for k in range(steps):
        F.v += 0.5 * w.dt / MVV2E * f
        F.x += w.dt * F.v
        thermostat()
        ev = k == steps - 1 or (every > 0 and k % every == 0)
        f, e, _ = F(ev)
        if ev:
            pe[k] = e
        F.v += 0.5 * w.dt / MVV2E * f
        ke[k] = thermostat()
    x = F.x - F.box * torch.floor(F.x / F.box)
    return x, F.v, f, pe, ke


def _mtk(w, steps, dev):
    """The MTK barostat's step (Nose-Hoover chains on atoms and on the isotropic box), 64-bit."""
    F = _Field(w, dev)
    f, _, vir = F(True)
    n, dt = w.n, w.dt
    ndof, kT = 3 * n - 3, KB * w.T
    tp2 = NPT["tau_P"] ** 2
    Wb = (ndof + 3) * kT * tp2
    Qt = [ndof * kT * w.tau_T ** 2] + [kT * w.tau_T ** 2] * (NPT["mt"] - 1)
    Qb = [kT * tp2] * NPT["mp"]
    et, etd, eb, ebd = [0.0] * NPT["mt"], [0.0] * NPT["mt"], [0.0] * NPT["mp"], [0.0] * NPT["mp"]
    eps, ke, h = 0.0, 0.5 * ndof * kT, 0.5 * dt

    def link(ed, Q, k, drive):
        m = len(ed)
        ex = math.exp(-ed[k + 1] * h / 4) if k < m - 1 else 1.0
        ed[k] = (ed[k] * ex + (drive() / Q[0] if k == 0 else (Q[k - 1] * ed[k - 1] ** 2 - kT) / Q[k]) * h / 2) * ex

    def chain(ed, eta, Q, drive, scaled):
        for k in reversed(range(len(ed))):
            link(ed, Q, k, drive)
        s = math.exp(-ed[0] * h)
        scaled(s)
        for k in range(len(ed)):
            eta[k] += ed[k] * h
        for k in range(len(ed)):
            link(ed, Q, k, drive)

    def scale_atoms(s):
        nonlocal ke
        ke *= s * s
        F.v *= s

    def scale_box(s):
        nonlocal eps
        eps *= s

    atoms = lambda: 2.0 * ke - ndof * kT  # noqa: E731
    baro = lambda: Wb * eps * eps - kT  # noqa: E731

    def push():
        nonlocal eps
        e = 0.5 * MVV2E * float((F.v * F.v).sum())
        V = float(F.box.prod())
        P = (float(vir[:3].sum()) + 2.0 * e) / (3.0 * V)
        eps += (3.0 * V * (P - NPT["P_target"]) + 6.0 * e / (3.0 * n)) / Wb * h

    out = dict(pe=np.empty(steps), ke=np.empty(steps), H=np.empty(steps), V=np.empty(steps))
    for k in range(steps):
        chain(ebd, eb, Qb, baro, scale_box)
        chain(etd, et, Qt, atoms, scale_atoms)
        push()
        damp = math.exp(-(eps + 3.0 * eps / (3.0 * n)) * h)
        F.v *= damp
        F.v += h / MVV2E * f
        g = min(max(eps * dt, -0.005), 0.005)
        F.x = F.x * math.exp(g) + F.v * dt * (math.expm1(g) / g if abs(g) > 2e-6 else 1.0 + 0.5 * g + g * g / 6.0)
        F.box = F.box * math.exp(g)
        f, pe, vir = F(True)
        F.v += h / MVV2E * f
        F.v *= damp
        ke = 0.5 * MVV2E * float((F.v * F.v).sum())
        push()
        chain(etd, et, Qt, atoms, scale_atoms)
        chain(ebd, eb, Qb, baro, scale_box)
        V = float(F.box.prod())
        H = ke + pe + 0.5 * Wb * eps * eps + ndof * kT * et[0] + kT * (sum(et[1:]) + sum(eb)) + NPT["P_target"] * V
        H += 0.5 * sum(a * b * b for a, b in zip(Qt, etd)) + 0.5 * sum(a * b * b for a, b in zip(Qb, ebd))
        out["pe"][k], out["ke"][k], out["H"][k], out["V"][k] = pe, ke, H, V
    x = F.x - F.box * torch.floor(F.x / F.box)
    out.update(_columns("x", x), **_columns("v", F.v), **_columns("f", f), box=F.box.cpu().numpy())
    return out


def _columns(name, a):
    a = a.cpu().numpy()
    keys = ("x", "y", "z") if name == "x" else [name + c for c in "xyz"]
    return {k: np.ascontiguousarray(a[:, d]) for d, k in enumerate(keys)}


def exact(case, seed):
    dev, kind = _device(), case["kind"]
    if kind in ("ladder", "serve"):
        ws = _members(case, seed)
        extra = (lambda i: 50 * (i % 3)) if kind == "serve" else (lambda i: 0)
        if len(ws) * case["steps"] > 30000:  # too many small launches for a short check
            return None
        got = [_verlet(w, case["steps"] + extra(i), 0, dev, kind == "serve") for i, w in enumerate(ws)]
        out = {k: np.concatenate([_columns(k[0], g[0] if k[0] == "x" else g[1])[k] for g in got])
               for k in ("x", "vx", "vy", "vz")}
        out.update({k: np.concatenate([_columns("x", g[0])[k] for g in got]) for k in ("y", "z")})
        if kind == "serve":
            out["pe"] = np.array([g[3][-1] for g in got])
            out["ke"] = np.array([g[4][-1] for g in got])
        return out
    w = _workload(case, seed)
    if kind == "npt":
        return _mtk(w, case["steps"], dev)
    if kind == "frame":
        f, pe, vir = _Field(w, dev)(True)
        return dict(_columns("f", f), pe=np.array([pe]), virial=vir)
    x, v, f, pe, ke = _verlet(w, case["steps"], EVERY, dev)
    out = dict(_columns("x", x), **_columns("v", v), pe=pe, ke=ke)
    if not case["mixed"]:
        out.update(_columns("f", f))
    return out
