"""Performance cases of gapx: the calls its users make, over the sizes they make them at.

Every case goes through the public Python entry points of ``gapx``:

* ``calc``      one structure per call from host arrays (``Model.calc``), as an
                ASE or FGAP_CALC program evaluates;
* ``batch``     a new population per call (``Context.load``, ``run``,
                ``results``), as a structure search scores a generation;
* ``replay``    new positions of a loaded cell (``Context.update``, ``run``,
                ``results`` with graph replay), as a program's own integrator
                or optimiser drives the device;
* ``md``        a block of NVT steps on the device (``Context.md``);
* ``surrogate`` energies of a new population from the MLP in place of the GAP
                (``Context.run_surrogate``), the pre-screen of a search;
* ``variance``  predictive variance of a loaded cell's new positions
                (``Context.variance``).

Structures are jittered lattice sites in triclinic cells (closest pairs at
about 0.7 of the site spacing, as in relaxed or thermally displaced crystals),
10 to 20 A^3 per atom, the species as in the synthetic workloads of
``gapx.synth``.  Models have that module's symmetry-function tables (``c96``,
``q128``, ``t256``) or a table of many cutoffs and shifted radial lines like
the shipped carbon/boron example (``general``); their sparse sets are
descriptors of separately seeded structures of the same kind, computed here in
FP64 with torch, so that a model's numbers do not depend on the library.

FP64 results are returned in FP64.  A mixed run's energies, forces and stress
have FP32 accuracy (its descriptors and contraction are FP32), and its callers
keep them as FP32 arrays.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "calypso-gap_amd"))

import gapx  # noqa: E402
from gapx import synth  # noqa: E402

PI = 3.141592654          # the potential's own constant
GPA = 6.24219e-3          # eV/A^3 per GPa
LENGTH_SCALE = 3.0        # model length scales in column standard deviations of the pool
MASS = {1: 1.008, 5: 10.811, 6: 12.011, 8: 15.999, 22: 47.867}

# A table of the shipped example's form: one zeta, shifted radial lines, a
# cutoff of its own for most angular lines, weights of both signs.
_CUTS = (6.0, 2.0, 1.5, 5.0, 4.0, 3.5, 3.0)


def _general_sf():
    lines = [(1, a, 6.0) for a in (1.0, 0.5, 0.1, 0.05, 0.01, 0.005, 0.001)]
    lines += [(3, r, 6.0) for r in (3.0, 2.5, 2.0, 1.5, 1.0)]
    for t, eta in ((2, 0.01), (2, 0.1), (4, 0.01)):
        lines += [(t, eta, c) for c in _CUTS]
    t, a, c = zip(*lines)
    return np.array(t, np.int32), np.array(a), np.array(c), np.ones(len(lines))


# name: symmetry-function table, species, weights, sparse points, sigma of the
# coefficients, neighbour cutoff, largest structure of the sparse set's pool
TABLES = {
    "c96": dict(sf=lambda: synth.workload_sf("c64"), z=(6,), w=(6.0,), M=500, sigma=0.1, rc=6.0),
    "general": dict(sf=_general_sf, z=(5, 6), w=(-1.0, 4.0), M=129, sigma=0.05, rc=6.0),
    "q128": dict(sf=synth.population_sf, z=(1, 6, 8, 22), w=(1.0, 6.0, 8.0, 22.0), M=4000, sigma=0.05, rc=6.0),
    "t256": dict(sf=lambda: synth.workload_sf("ternary32k"), z=(1, 8, 22), w=(1.0, 8.0, 22.0), M=8000, sigma=0.05,
                 rc=6.5),
}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: a conventional carbon cell through the drop-in entry point; latency only
        dict(name="calc_8_fp64", kind="calc", table="c96", atoms=8, precision="fp64", grad=True),
        # the reference's own use: a 64-atom cell, its example's kind of table, one call per step of an ASE program
        dict(name="calc_64_general_fp64", kind="calc", table="general", atoms=64, precision="fp64", grad=True),
        # one ragged structure of several species through the drop-in entry point in mixed precision
        dict(name="calc_197_mixed", kind="calc", table="q128", atoms=197, precision="mixed", grad=True),
        # a generation of a structure search, energies, forces and stress (the benchmark's population)
        dict(name="batch_512_fp64", kind="batch", table="q128", structs=512, nmin=8, nmax=256, precision="fp64",
             grad=True),
        dict(name="batch_512_mixed", kind="batch", table="q128", structs=512, nmin=8, nmax=256, precision="mixed",
             grad=True),
        # a generation scored by energy alone
        dict(name="batch_999_energy_mixed", kind="batch", table="q128", structs=999, nmin=16, nmax=128,
             precision="mixed", grad=False),
        # a device-resident cell driven step by step, both precisions (the benchmark's 4096-atom cell)
        dict(name="replay_4096_fp64", kind="replay", table="q128", atoms=4096, precision="fp64", grad=True),
        dict(name="replay_4096_mixed", kind="replay", table="q128", atoms=4096, precision="mixed", grad=True),
        # the largest: the benchmark's 32768-atom cell with the long table
        dict(name="replay_32768_mixed", kind="replay", table="t256", atoms=32768, precision="mixed", grad=True),
        # molecular dynamics of one small cell: a serial chain of small launches
        dict(name="md_64_fp64", kind="md", table="c96", atoms=64, structs=1, steps=16, precision="fp64", grad=True),
        # the search's pre-screen: surrogate energies of a new population
        dict(name="surrogate_2000", kind="surrogate", table="q128", structs=2000, nmin=16, nmax=128,
             precision="mixed", grad=False),
        # active learning: variance of a cell's environments
        dict(name="variance_2048", kind="variance", table="q128", atoms=2048, precision="fp64", grad=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["calc", "calc", "batch", "batch", "replay", "replay", "md", "surrogate", "variance"])
    precision = rng.choice(["fp64", "fp64", "mixed", "mixed", "bf16"])
    if kind == "calc":
        return dict(kind=kind, table=rng.choice(["c96", "general", "q128"]), atoms=_log_int(rng, 2, 600),
                    precision=precision, grad=rng.random() < 0.85)
    if kind == "batch":
        nmax = _log_int(rng, 12, 256)
        return dict(kind=kind, table=rng.choice(["c96", "general", "q128", "q128"]), structs=_log_int(rng, 4, 512),
                    nmin=rng.randint(2, 8), nmax=nmax, precision=precision, grad=rng.random() < 0.75)
    if kind == "replay":
        table = rng.choice(["q128", "q128", "t256"])
        top = {"fp64": 8192 if table == "t256" else 32768}.get(precision, 32768)
        return dict(kind=kind, table=table, atoms=_log_int(rng, 300, top), precision=precision, grad=True)
    if kind == "md":
        atoms = _log_int(rng, 8, 400)
        return dict(kind=kind, table=rng.choice(["c96", "q128"]), atoms=atoms,
                    structs=_log_int(rng, 1, min(24, 3200 // atoms)), steps=16, precision="fp64", grad=True)
    if kind == "surrogate":
        return dict(kind=kind, table="q128", structs=_log_int(rng, 50, 2000), nmin=16, nmax=128, precision="mixed",
                    grad=rng.random() < 0.3)
    return dict(kind=kind, table="q128", atoms=_log_int(rng, 64, 4096), precision="fp64", grad=False)


# ---------------------------------------------------------------------------
# structures and models
# ---------------------------------------------------------------------------

def _structure(rng, n, vpa, species, jitter=0.15):
    """n jittered sites of an m1 x m2 x m3 lattice in a triclinic cell of n vpa A^3."""
    m1 = max(1, round(n ** (1 / 3)))
    m2 = max(1, round(math.sqrt(n / m1)))
    m = np.array([m1, m2, -(-n // (m1 * m2))])
    lat = synth.triclinic_cell(1.0, rng) * m[:, None]
    lat *= (n * vpa / abs(np.linalg.det(lat))) ** (1 / 3)
    sites = rng.permutation(int(m.prod()))[:n]
    frac = np.stack(np.unravel_index(sites, m), axis=1) + 0.5 + rng.uniform(-jitter, jitter, (n, 3))
    return dict(species=rng.choice(np.asarray(species, np.int32), size=n), lat=lat, pos=(frac / m) @ lat)


def _cell(rng, n, table):
    """A single structure: all of the table's species, ordinary density."""
    return _structure(rng, n, rng.uniform(12.0, 17.0), TABLES[table]["z"])


def _population(rng, count, nmin, nmax, table):
    """Uneven structures of one to all of the table's species, 10 to 20 A^3 per
    atom; the atom counts of a case are the same for every seed."""
    z = np.asarray(TABLES[table]["z"])
    out = []
    for n in np.random.default_rng([count, nmin, nmax]).integers(nmin, nmax + 1, size=count):
        k = int(rng.integers(1, len(z) + 1))
        out.append(_structure(rng, int(n), rng.uniform(10.0, 20.0), rng.choice(z, size=k, replace=False)))
    return out


_arrays, _models = {}, {}


def _model_arrays(table):
    """The table's model: sparse set, length scales and coefficients (one per process, fixed seed)."""
    if table not in _arrays:
        t = TABLES[table]
        rng = np.random.default_rng(77)
        header = dict(z=t["z"], w=t["w"], sf=t["sf"](), rc=t["rc"])
        pool, have = [], 0
        while have < 1.25 * t["M"]:
            n = int(rng.integers(24, 128))
            pool.append(_cell(rng, 96, table) if len(pool) % 2 else _population(rng, 1, n, n, table)[0])
            have += len(pool[-1]["species"])
        x = _Exact(header).descriptors(pool).cpu().numpy()
        theta = LENGTH_SCALE * x.std(axis=0)
        theta = np.where(theta > 1e-8, theta, 1.0)
        mm = x[rng.choice(len(x), size=t["M"], replace=False)]
        _arrays[table] = dict(header, theta=theta, mm=mm, coeff=rng.normal(0.0, t["sigma"], size=t["M"]))
    return _arrays[table]


def _qmm(a):
    """Q of the variance: the inverse of the sparse set's own covariance with a noise of 0.1."""
    m = torch.as_tensor(a["mm"] / a["theta"], device=_device())
    n = (m * m).sum(1)
    k = torch.exp(-0.5 * (n[:, None] + n[None, :] - 2.0 * (m @ m.T)).clamp_min(0.0))
    q = torch.linalg.inv(k + 0.01 * torch.eye(len(m), dtype=torch.float64, device=m.device))
    return (0.5 * (q + q.T)).cpu().numpy()


def _model(table, variance=False):
    """The device model, kept for the life of the program as its users keep it."""
    key = (table, variance)
    if key not in _models:
        a = _model_arrays(table)
        t, alpha, cut, zeta = a["sf"]
        _models[key] = gapx.Model.from_arrays(a["z"], a["w"], t, alpha, cut, a["theta"], a["mm"], a["coeff"], zeta)
        if variance:
            a["qmm"] = _qmm(a)
            _models[key].set_qmm(a["qmm"])
    return _models[key]


def _mlp_params():
    """Random surrogate weights in the flat layout W1, b1, W2, b2, w3, b3."""
    rng = np.random.default_rng(5)
    s = 1.0 / math.sqrt(128.0)
    parts = [rng.normal(0, s, 128 * 128), rng.normal(0, 0.1, 128), rng.normal(0, s, 128 * 128),
             rng.normal(0, 0.1, 128), rng.normal(0, s, 128), rng.normal(0, 0.1, 1)]
    return np.concatenate(parts).astype(np.float32)


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------

def _inputs(case, seed):
    """Structures (and momenta) of a case, from the seed alone."""
    rng = np.random.default_rng([seed, 3])
    kind, table = case["kind"], case["table"]
    if kind in ("batch", "surrogate"):
        return _population(rng, case["structs"], case["nmin"], case["nmax"], table), None
    s = [_cell(rng, case["atoms"], table) for _ in range(case.get("structs", 1))]
    if kind != "md":
        return s, None
    masses = np.concatenate([[MASS[int(z)] for z in x["species"]] for x in s])
    return s, (masses, rng.normal(size=(len(masses), 3)) * np.sqrt(masses * 300.0 * gapx.KB)[:, None])


def _flags(case):
    f = gapx.GRAD if case["grad"] else 0
    return f | {"fp64": 0, "mixed": gapx.MIXED, "bf16": gapx.MIXED | gapx.BF16}[case["precision"]]


def prepare(case, seed):
    structs, momenta = _inputs(case, seed)
    kind, rc = case["kind"], TABLES[case["table"]]["rc"]
    model = _model(case["table"], kind == "variance")
    st = dict(kind=kind, model=model, structs=structs, rc=rc, flags=_flags(case), momenta=momenta,
              steps=case.get("steps"), out=np.float64 if case["precision"] == "fp64" else np.float32)
    if kind == "calc":
        return st
    st["ctx"] = gapx.Context(model)
    if kind in ("replay", "md", "variance"):
        st["pos"] = np.concatenate([s["pos"] for s in structs])
        st["ctx"].load(structs, rc)
        st["ctx"].use_graph(True)
    if kind == "surrogate":
        st["mlp"] = gapx.MLP(seed=0)
        st["mlp"].set_params(_mlp_params())
    return st


def run(st):
    kind, flags, out = st["kind"], st["flags"], st["out"]
    if kind == "calc":
        s = st["structs"][0]
        e, f, stress, _ = st["model"].calc(s["species"], s["lat"], s["pos"], st["rc"], flags=flags, grad=False)
        if not flags & gapx.GRAD:
            return out(e)
        return out(e), f.astype(out, copy=False), stress.astype(out, copy=False)
    ctx = st["ctx"]
    if kind == "md":
        masses, p0 = st["momenta"]
        ctx.update(st["pos"])
        log = ctx.md(masses, st["steps"], momenta=p0, flags=flags)
        return log, ctx.positions(), ctx.momenta()
    if kind in ("batch", "surrogate"):
        ctx.load(st["structs"], st["rc"])
    else:
        ctx.update(st["pos"])
    if kind == "surrogate":
        ctx.run_surrogate(st["mlp"], flags)
    else:
        ctx.run(flags)
    if kind == "variance":
        return ctx.variance()
    r = ctx.results()
    if not flags & gapx.GRAD:
        return r["energy"].astype(out, copy=False), r["eatom"].astype(out, copy=False)
    return tuple(r[k].astype(out, copy=False) for k in ("energy", "eatom", "forces", "stress"))


def work(case):
    """Bytes: positions and species in, the model once, results out.  Flops: the
    contraction's two products (one without forces), and per neighbour pair and
    per triplet the geometry and the accumulation of every line, forward and,
    with forces, backward, at the neighbour and triplet counts of a uniform
    density."""
    a = TABLES[case["table"]]
    t, _, cut, _ = a["sf"]()
    n_rad, n_ang = int(np.isin(t, (1, 3)).sum()), int(np.isin(t, (2, 4)).sum())
    mean = 0.5 * (case.get("nmin", 0) + case.get("nmax", 0))
    n = case["structs"] * mean if case["kind"] in ("batch", "surrogate") else case["atoms"] * case.get("structs", 1)
    vpa = 14.4
    k = 4.0 / 3.0 * math.pi * a["rc"] ** 3 / vpa
    ka = 4.0 / 3.0 * math.pi * float(cut[np.isin(t, (2, 4))].max()) ** 3 / vpa
    trip = 15.0 / 32.0 * ka * (ka - 1.0) / 2.0
    D, grad = 2 * len(t), case["grad"]
    flops = n * (k * (30.0 + 12.0 * n_rad) + trip * (40.0 + 4.0 * n_ang))
    if grad:
        flops += n * (k * (30.0 + 16.0 * n_rad) + trip * (80.0 + 10.0 * n_ang))
    wide = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "surrogate":
        flops += n * 2.0 * (2 * 128 * 128 + 128) * (2 if grad else 1)
        model = 4.0 * (2 * 128 * 128)
    else:
        flops += n * (4.0 if grad else 2.0) * D * a["M"]
        model = wide * a["M"] * (D + 1.0)
    io = n * (24.0 + 4.0) + n * wide * (4.0 if grad else 1.0)
    if case["kind"] == "variance":
        flops += n * 2.0 * a["M"] * (a["M"] + D)
        model += 8.0 * a["M"] ** 2
    steps = case.get("steps", 1)
    return {"bytes": steps * (io + model), "flops": steps * flops}


# ---------------------------------------------------------------------------
# the same results in 64 bits with torch: dense image search, padded triplet
# arrays, automatic derivatives with respect to the pair vectors
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Exact:
    def __init__(self, a):
        self.a, self.dev = a, _device()
        t, alpha, cut, zeta = a["sf"]
        self.lines = list(zip(t.tolist(), alpha.tolist(), cut.tolist(), zeta.tolist()))
        self.rc = a["rc"]
        self.rc_ang = max(c for k, _, c, _ in self.lines if k in (2, 4))
        if "mm" in a:
            self.theta = self.tensor(a["theta"])
            self.m = self.tensor(a["mm"]) / self.theta
            self.mu = self.m.mean(0)
            self.m = self.m - self.mu
            self.c = self.tensor(a["coeff"])

    def tensor(self, x):
        return torch.as_tensor(np.asarray(x, np.float64), device=self.dev)

    def neighbours(self, lat, pos):
        """(i, j, r_j + images - r_i) of every pair within the cutoff, sorted by i."""
        L, p = self.tensor(lat), self.tensor(pos)
        n = len(p)
        inv = torch.linalg.inv(L)
        spacing = 1.0 / torch.linalg.norm(inv, dim=0)
        if float(spacing.min()) > 2.0 * self.rc + 0.1:
            shifts = None                     # one image at most: the nearest in each lattice direction
            per = max(1, 20_000_000 // n)
        else:
            reach = [int(math.floor(self.rc / float(s))) + 1 for s in spacing]
            g = [torch.arange(-k, k + 1, device=self.dev, dtype=torch.float64) for k in reach]
            shifts = torch.cartesian_prod(*g) @ L
            per = max(1, 10_000_000 // (n * len(shifts)))
        oi, oj, od = [], [], []
        for r0 in range(0, n, per):
            d = p[None, :, :] - p[r0:r0 + per, None, :]
            if shifts is None:
                d = d - torch.round(d @ inv) @ L
                keep = ((d * d).sum(-1) <= self.rc ** 2)
                keep[torch.arange(len(d), device=self.dev), torch.arange(r0, r0 + len(d), device=self.dev)] = False
                i, j = keep.nonzero(as_tuple=True)
                od.append(d[i, j])
            else:
                d = d[:, :, None, :] + shifts[None, None]
                r2 = (d * d).sum(-1)
                keep = (r2 <= self.rc ** 2) & (r2 > 1e-12)
                i, j, s = keep.nonzero(as_tuple=True)
                od.append(d[i, j, s])
            oi.append(i + r0)
            oj.append(j)
        return torch.cat(oi), torch.cat(oj), torch.cat(od)

    def lists(self, structs, w):
        """Pair lists of all structures back to back, and each structure's first atom."""
        I, J, V, W, base = [], [], [], [], 0
        for s in structs:
            i, j, d = self.neighbours(s["lat"], s["pos"])
            wj = self.tensor([w[int(z)] for z in s["species"]])
            I.append(i + base)
            J.append(j + base)
            V.append(d)
            W.append(wj[j])
            base += len(s["species"])
        return torch.cat(I), torch.cat(J), torch.cat(V), torch.cat(W), base

    @staticmethod
    def fc(r, rc):
        return torch.where(r <= rc, 0.5 * (torch.cos(PI * r / rc) + 1.0), torch.zeros_like(r))

    def rows(self, d, w, valid):
        """Features of padded neighbour rows: d [n, K, 3], w [n, K], valid [n, K]."""
        n, K = valid.shape
        r = torch.sqrt(torch.where(valid, (d * d).sum(-1), torch.ones_like(w)))
        on = valid.to(torch.float64)
        plain, weighted = [None] * len(self.lines), [None] * len(self.lines)
        for s, (k, alpha, cut, _) in enumerate(self.lines):
            if k in (1, 3):
                t = torch.exp(-alpha * r * r) if k == 1 else torch.exp(-4.0 * (r - alpha) ** 2)
                t = t * self.fc(r, cut) * on
                plain[s], weighted[s] = t.sum(1), (t * w).sum(1)
        ang = [(cut, alpha, k, z, s) for s, (k, alpha, cut, z) in enumerate(self.lines) if k in (2, 4)]
        # triplets of each row, packed to the left
        A, B = torch.triu_indices(K, K, 1, device=self.dev)
        with torch.no_grad():
            near = valid & (r <= self.rc_ang)
            ok = near[:, A] & near[:, B]
            e2 = torch.zeros(ok.shape, dtype=torch.float64, device=self.dev)
            for c in range(3):
                e2 += (d[:, B, c] - d[:, A, c]) ** 2
            ok &= e2 <= self.rc_ang ** 2
            count = ok.sum(1)
            T = max(1, int(count.max()))
            row, col = ok.nonzero(as_tuple=True)
            at = torch.arange(len(row), device=self.dev) - (torch.cumsum(count, 0) - count)[row]
            a = torch.zeros((n, T), dtype=torch.long, device=self.dev)
            b = torch.zeros((n, T), dtype=torch.long, device=self.dev)
            mask = torch.zeros((n, T), dtype=torch.bool, device=self.dev)
            a[row, at], b[row, at], mask[row, at] = A[col], B[col], True
        g = lambda x, k: torch.gather(x, 1, k)  # noqa: E731
        ra, rb, ww = g(r, a), g(r, b), g(w, a) * g(w, b)
        e2 = sum((g(d[..., c], b) - g(d[..., c], a)) ** 2 for c in range(3))
        e = torch.sqrt(torch.where(mask, e2, torch.ones_like(e2)))
        e2 = e * e
        cth = (ra * ra + rb * rb - e2) / (2.0 * ra * rb)
        S2 = ra * ra + rb * rb + e2
        on = mask.to(torch.float64)
        groups = {}
        for cut, alpha, k, z, s in ang:
            groups.setdefault(cut, {}).setdefault(alpha, []).append((k, z, s))
        for cut, etas in groups.items():
            F = self.fc(ra, cut) * self.fc(rb, cut) * self.fc(e, cut) * on
            keys = sorted({(k, z) for v in etas.values() for k, z, _ in v})
            P = torch.stack([2.0 ** (1.0 - z) * (1.0 + (1.0 if k == 2 else -1.0) * cth).clamp_min(0.0) ** z
                             for k, z in keys], dim=2)
            for alpha, ls in etas.items():
                E = torch.exp(-alpha * S2) * F
                x = torch.bmm(torch.stack([E, E * ww], dim=1), P)
                for k, z, s in ls:
                    plain[s], weighted[s] = x[:, 0, keys.index((k, z))], x[:, 1, keys.index((k, z))]
        return torch.stack(plain + weighted, dim=1)

    def chunks(self, I, total):
        """Consecutive atoms whose padded triplet arrays stay small."""
        count = torch.bincount(I, minlength=total)
        start = torch.cumsum(count, 0) - count
        cnt, budget = count.tolist(), 64_000_000 // len(self.lines)
        lo = 0
        while lo < total:
            hi, top = lo, 0
            while hi < total and (hi - lo + 1) * (0.5 * max(top, cnt[hi]) ** 2 + 64) <= 2 * budget:
                top = max(top, cnt[hi])
                hi += 1
            hi = max(hi, lo + 1)
            K = max(2, max(cnt[lo:hi]))
            k = torch.arange(K, device=self.dev)
            valid = k[None, :] < count[lo:hi, None]
            yield lo, hi, torch.where(valid, start[lo:hi, None] + k[None, :], torch.zeros_like(k)[None, :]), valid
            lo = hi

    def weights(self):
        return {int(z): float(w) for z, w in zip(self.a["z"], self.a["w"])}

    def descriptors(self, structs):
        I, _, V, W, total = self.lists(structs, self.weights())
        with torch.no_grad():
            return torch.cat([self.rows(V[k], W[k], v) for _, _, k, v in self.chunks(I, total)])

    def gpr(self, x):
        xt = x / self.theta - self.mu
        d2 = (xt * xt).sum(1)[:, None] + (self.m * self.m).sum(1)[None, :] - 2.0 * (xt @ self.m.T)
        wk = torch.exp(-0.5 * d2) * self.c
        e = wk.sum(1)
        return e, -(xt * e[:, None] - wk @ self.m) / self.theta

    def mlp(self, x, p):
        p = self.tensor(p)
        W1, b1, W2, b2, w3, b3 = torch.split(p, [128 * 128, 128, 128 * 128, 128, 128, 1])
        xt = (x / self.theta - self.mu).requires_grad_(True)
        with torch.enable_grad():
            h = torch.nn.functional.silu(xt @ W1.reshape(128, 128) + b1)
            h = torch.nn.functional.silu(h @ W2.reshape(128, 128) + b2)
            e = h @ w3 + b3
            (g,) = torch.autograd.grad(e.sum(), xt)
        return e.detach(), g / self.theta

    def evaluate(self, structs, grad, atomic):
        """Energies per structure and per atom, forces and stress; atomic(x) gives (e, de/dx) of each row."""
        I, J, V, W, total = self.lists(structs, self.weights())
        eatom, gd = [], torch.zeros_like(V)
        for _, _, k, valid in self.chunks(I, total):
            if not grad:
                with torch.no_grad():
                    eatom.append(atomic(self.rows(V[k], W[k], valid))[0])
                continue
            d = V[k].detach().requires_grad_(True)
            x = self.rows(d, W[k], valid)
            with torch.no_grad():
                e, g = atomic(x.detach())
            (dd,) = torch.autograd.grad(x, d, g)
            gd[k[valid]] = dd[valid]
            eatom.append(e)
        eatom = torch.cat(eatom)
        n = torch.tensor([len(s["species"]) for s in structs], device=self.dev)
        of = torch.repeat_interleave(torch.arange(len(structs), device=self.dev), n)
        zeros = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.dev)  # noqa: E731
        ene = zeros(len(structs)).index_add_(0, of, eatom)
        if not grad:
            return ene, eatom
        force = zeros(total, 3).index_add_(0, I, gd).index_add_(0, J, -gd)
        vir = zeros(len(structs), 3, 3).index_add_(0, of[I], gd[:, :, None] * V[:, None, :])
        vol = self.tensor([abs(np.linalg.det(s["lat"])) for s in structs])
        s6 = torch.stack([vir[:, a, b] for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))], dim=1)
        return ene, eatom, force, -s6 / vol[:, None] / GPA


def exact(case, seed):
    if case["kind"] == "md":
        return None                            # a trajectory: its steps are the evaluations of the other cases
    structs, _ = _inputs(case, seed)
    ex = _Exact(_model_arrays(case["table"]))
    if case["kind"] == "variance":
        q = ex.tensor(_qmm(ex.a))
        x = ex.descriptors(structs) / ex.theta - ex.mu
        d2 = (x * x).sum(1)[:, None] + (ex.m * ex.m).sum(1)[None, :] - 2.0 * (x @ ex.m.T)
        k = torch.exp(-0.5 * d2)
        s2 = 1.0 - ((k @ q) * k).sum(1)
        return s2.mean().reshape(1), s2
    if case["kind"] == "surrogate":
        p = _mlp_params()
        return ex.evaluate(structs, case["grad"], lambda x: ex.mlp(x, p))
    out = ex.evaluate(structs, case["grad"], ex.gpr)
    if case["kind"] != "calc":
        return out
    return (out[0][0], out[2], out[3][0]) if case["grad"] else out[0][0]
