"""The work that the speed of this library is judged by: SCF residuals and
DIIS / Newton solves on 1-, 2- and 3-gradient lattices through the Python
binding, with sizes from the repository's own benchmark workloads
(`bench.py` and its batch1d, charged, box and serve workloads) and tests.

A case names a family (the kind of system) and an entry (the call):

* entry `residual`: ScfSystem.residual, one evaluation from host fields;
* entry `solve`: ScfSystem.solve or solve_batch, DIIS for `its` iterations
  from seeded host fields (a real solve takes tens to thousands of the same
  iterations; the limit keeps rounding from growing into the results);
* entry `newton`: ScfSystem.solve with the reference's default method, to
  the tolerance;
* entry `queue`: solve_jobs, every job three chained solves, `its`
  iterations each, on resident slots with the batch-tuned end-point storage.

`exact` evaluates the same equations in plain torch (FP64): per-site arrays
without ghost layers, every batch member in one tensor.
"""
import math

import numpy as np
import torch

PIE = 3.14159265
CHIS = (0.0, 0.5, 0.8)
DMAX, HISTORY = 0.1, 10


def listed():
    return [
        # one residual of the planar adsorption system (configuration 1): what
        # a program that drives the library with its own solver calls
        dict(name="residual 1d", family="adsorption", entry="residual", count=1, layers=100, layers_hi=100, N=100,
             N_hi=100, its=0),
        # the reference's default solver on the same kind of system
        dict(name="newton 1d", family="adsorption", entry="newton", count=1, layers=120, layers_hi=120, N=200,
             N_hi=200, its=0),
        # a parameter sweep in one launch (configuration 4): first- and
        # second-order chains in turn, every length and lattice size
        dict(name="batch 1d", family="adsorption", entry="solve", count=512, layers=50, layers_hi=400, N=20,
             N_hi=2000, its=3),
        # the charged sweep: the potential solved with the fields
        dict(name="batch charged", family="charged", entry="solve", count=512, layers=30, layers_hi=200, N=20,
             N_hi=500, its=8),
        # a surfactant with a branched head group at a wall (the test suite's
        # branched molecule, longer tail)
        dict(name="branched 1d", family="branched", entry="solve", count=1, layers=60, layers_hi=60, N=16, N_hi=16,
             its=12),
        # the default benchmark: brush jobs in the persistent queue, one per CU
        dict(name="brush queue", family="brush", entry="queue", count=256, nr=64, nz=128, N=200, its=4),
        # one such job on an idle GPU
        dict(name="brush alone", family="brush", entry="queue", count=1, nr=64, nz=128, N=200, its=12),
        # a served 2-gradient request (32-128 x 32-256 layers, N 50-400) of odd size
        dict(name="brush ragged", family="brush", entry="solve", count=1, nr=43, nz=101, N=120, its=8),
        # the largest served 2-gradient request
        dict(name="brush large", family="brush", entry="solve", count=1, nr=128, nz=256, N=400, its=3),
        # the 3-gradient configuration, save_memory on, FP64
        dict(name="box 96", family="box", entry="solve", count=1, n=96, mixed=False, its=12),
        # the same with FP32 propagators (every iteration is above the switch level)
        dict(name="box 96 mixed", family="box", entry="solve", count=1, n=96, mixed=True, its=12),
        # a small box of odd size
        dict(name="box 53", family="box", entry="solve", count=1, n=53, mixed=False, its=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["residual", "newton", "batch", "charged", "branched", "queue", "brush", "brush", "box", "box"])
    if kind == "residual":
        layers, N = rng.randint(20, 400), _log_int(rng, 10, 2000)
        return dict(family="adsorption", entry="residual", count=1, layers=layers, layers_hi=layers, N=N, N_hi=N, its=0)
    if kind == "newton":
        layers, N = rng.randint(40, 160), _log_int(rng, 20, 300)
        return dict(family="adsorption", entry="newton", count=1, layers=layers, layers_hi=layers, N=N, N_hi=N, its=0)
    if kind == "batch":
        lo, n = rng.randint(50, 200), _log_int(rng, 20, 200)
        return dict(family="adsorption", entry="solve", count=_log_int(rng, 2, 512), layers=lo,
                    layers_hi=rng.randint(lo, 400), N=n, N_hi=_log_int(rng, n, 2000), its=rng.randint(2, 3))
    if kind == "charged":
        lo, n = rng.randint(30, 100), _log_int(rng, 20, 100)
        return dict(family="charged", entry="solve", count=_log_int(rng, 2, 512), layers=lo,
                    layers_hi=rng.randint(lo, 200), N=n, N_hi=_log_int(rng, n, 500), its=rng.randint(3, 8))
    if kind == "branched":
        layers, N = rng.randint(20, 200), rng.randint(4, 40)
        return dict(family="branched", entry="solve", count=1, layers=layers, layers_hi=layers, N=N, N_hi=N,
                    its=rng.randint(3, 12))
    if kind == "queue":
        return dict(family="brush", entry="queue", count=_log_int(rng, 1, 256), nr=4 * rng.randint(8, 16),
                    nz=rng.randint(32, 128), N=_log_int(rng, 50, 200), its=rng.randint(3, 4))
    if kind == "brush":
        return dict(family="brush", entry="solve", count=1, nr=rng.randint(32, 128), nz=rng.randint(32, 256),
                    N=_log_int(rng, 50, 400), its=3)
    return dict(family="box", entry="solve", count=1, n=rng.randint(24, 96), mixed=rng.random() < 0.3,
                its=rng.randint(3, 12))


# ---------------------------------------------------------------- the systems
def _spread(lo, hi, count, log, step):
    """`count` whole numbers over [lo, hi] in a fixed scrambled order."""
    u = (0.5 + step * np.arange(count)) % 1.0 if count > 1 else np.zeros(1)
    v = lo * (hi / lo) ** u if log else lo + (hi - lo) * u
    return [int(round(t)) for t in v]


def _members(case, seed):
    """Parameters of every system of the case: sizes from the case, the
    physical parameters from the seed."""
    rng = np.random.default_rng([17, seed])
    if case["family"] == "brush":
        chi = float(rng.uniform(0.2, 0.6))
        return [dict(nr=case["nr"], nz=case["nz"], N=case["N"], chi=chi) for _ in range(case["count"])]
    if case["family"] == "box":
        return [dict(n=case["n"], frac=float(rng.uniform(0.04, 0.06)))]
    n = case["count"]
    layers = _spread(case["layers"], case["layers_hi"], n, False, 0.5698402910)
    Ns = _spread(case["N"], case["N_hi"], n, True, 0.7548776662)
    out = []
    for i in range(n):
        d = dict(layers=layers[i], N=Ns[i], markov=2 if i % 2 else 1, chi_s=float(rng.uniform(-1.5, -0.2)))
        if case["family"] == "adsorption":
            d.update(chi=float(rng.uniform(0.3, 0.55)), phib=float(np.exp(rng.uniform(np.log(1e-4), np.log(1e-2)))))
        elif case["family"] == "charged":
            d.update(valence=float(rng.uniform(-0.2, -0.05)), salt=float(np.exp(rng.uniform(np.log(1e-2), np.log(1e-1)))),
                     theta=float(rng.uniform(0.2, 1.0)))
        else:
            d.update(chi=float(rng.uniform(0.8, 1.2)), theta=float(rng.uniform(1.0, 3.0)))
        out.append(d)
    return out


def _branched_input(d):
    return """
lat : flat : gradients : 1
lat : flat : n_layers : {L}
lat : flat : lattice_type : simple_cubic
lat : flat : lowerbound : surface
mon : S : freedom : frozen
mon : S : frozen_range : lowerbound
mon : C : freedom : free
mon : N : freedom : free
mon : W : freedom : free
mon : S : chi_C : {cs!r}
mon : C : chi_W : {c!r}
mon : N : chi_W : -0.3
mol : surf : composition : (C){n}(N)1[(N)1][(N)1](N)1
mol : surf : freedom : restricted
mol : surf : theta : {th!r}
mol : water : composition : (W)1
mol : water : freedom : solvent
newton : isaac : method : DIIS
""".format(L=d["layers"], cs=d["chi_s"], c=d["chi"], n=d["N"], th=d["theta"])


def _text(case, d, chi=None):
    from namics_amd import workloads as wl
    fam = case["family"]
    if fam == "adsorption":
        t = wl.homopolymer_adsorption(d["layers"], d["N"], d["chi"], d["chi_s"], d["phib"], markov=d["markov"])
        if case["entry"] == "newton":
            t = t.replace("method : DIIS", "method : pseudohessian").replace("tolerance : 1e-07", "tolerance : 1e-10")
        return t
    if fam == "charged":
        return wl.polyelectrolyte_adsorption(d["layers"], d["N"], d["valence"], d["chi_s"], d["salt"], d["theta"],
                                             markov=d["markov"])
    if fam == "branched":
        return _branched_input(d)
    if fam == "brush":
        return wl.brush_cylinder(d["chi"] if chi is None else chi, n_r=d["nr"], n_z=d["nz"], N=d["N"])
    return wl.diblock_box(d["n"], frac=d["frac"])


def _start(case, d, seed, index, fields, nvar):
    """Starting fields of one system (what the program holds on the host)."""
    from namics_amd import workloads as wl
    if case["family"] == "box":
        return wl.seeded_box_fields(fields, d["n"], seed)
    if case["entry"] == "newton":
        return np.zeros(nvar)
    amp = {"brush": 0.05, "branched": 0.3}.get(case["family"], 0.02)
    return np.random.default_rng([seed, index]).uniform(-amp, amp, nvar)


def prepare(case, seed):
    from namics_amd import DeviceBuffer, ScfSystem, autotune_batch
    members = _members(case, seed)
    if case["entry"] == "queue":
        slots = [[ScfSystem(_text(case, d, chi)) for chi in CHIS] for d in members]
        autotune_batch([row[0] for row in slots])
        K = slots[0][0].checkpoint_interval()
        for row in slots:
            for s in row:
                s.set_checkpoint(K)
                s.set_solver(iterationlimit=case["its"])
        x0 = np.stack([_start(case, d, seed, i, None, slots[0][0].nvar) for i, d in enumerate(members)])
        return dict(case=case, slots=slots, seeds=DeviceBuffer(x0), jobs=len(members))
    systems = [ScfSystem(_text(case, d)) for d in members]
    for s in systems:
        if case["entry"] == "solve":
            s.set_solver(iterationlimit=case["its"])
        if case.get("mixed"):
            s.set_precision(True, 1e-6)
    x0 = [_start(case, d, seed, i, s.field_names, s.nvar) for i, (d, s) in enumerate(zip(members, systems))]
    return dict(case=case, systems=systems, x0=x0)


def run(state):
    from namics_amd import solve_batch, solve_jobs
    case = state["case"]
    if case["entry"] == "queue":
        jobs, _ = solve_jobs(state["slots"], state["seeds"], state["jobs"])
        out = {"free_energy": np.array([[r["free_energy"] for r in job] for job in jobs]),
               "grand_potential": np.array([[r["grand_potential"] for r in job] for job in jobs]),
               "residual": np.array([[r["residual"] for r in job] for job in jobs])}
        if state["jobs"] == 1:
            out["x"] = state["slots"][0][-1].download()
        return out
    systems, x0 = state["systems"], state["x0"]
    if case["entry"] == "residual":
        g, r = systems[0].residual(x0[0])
        return {"g": g, "residual": r}
    if case["entry"] == "newton":
        return {"x": systems[0].solve(x0[0])[0]}
    if len(systems) == 1:
        x, _, r, _ = systems[0].solve(x0[0])
        return {"x": x, "residual": r}
    xs, infos = solve_batch(systems, x0)
    return {"x": np.concatenate(xs), "residual": np.array([i[1] for i in infos])}


def _chain_sites(case):
    """(sum of N x sites x operations per site and step, sites) over the
    systems: 5 operations for the 3-point step, 15 for its three-component
    second-order form, 8 for the factored 9-point step, 7 for the 6-point."""
    ops = sites = 0
    for d in _members(case, 1):
        if case["family"] == "brush":
            w, per, N = d["nr"] * d["nz"], 8, d["N"]
        elif case["family"] == "box":
            w, per, N = d["n"] ** 3, 7, 20
        else:
            w, per = d["layers"], 15 if d["markov"] == 2 else 5
            N = d["N"] + 4 if case["family"] == "branched" else d["N"]
        ops += w * per * N
        sites += w
    return ops, sites


def work(case):
    """Per pass: fields in and out once; the forward and the backward
    propagation with the composition (2 more operations) of every evaluation."""
    ops, sites = _chain_sites(case)
    blocks = {"adsorption": 2, "charged": 5, "branched": 3, "brush": 3, "box": 2}[case["family"]]
    evals = {"residual": 1, "newton": 30, "solve": case["its"] + 1, "queue": 3 * (case["its"] + 1)}[case["entry"]]
    return {"bytes": 2.0 * 8 * blocks * sites, "flops": evals * 2.4 * ops}


def tolerance(case):
    # FP64 throughout: rounding grown by the DIIS steps (a relative change of
    # 1e-15 in the starting fields, or another order of the sums, moves the
    # results by up to 1e-7); Newton: the distance to the fixed point at the
    # tolerance; mixed: FP32 propagators (1e-5 from the FP64 results)
    if case["entry"] == "residual":
        return {"rel": 1e-10, "max": 1e-9}
    if case["entry"] == "newton":
        return {"rel": 1e-6, "max": 1e-5}
    if case.get("mixed"):
        return {"rel": 5e-5, "max": 5e-3}
    return {"rel": 4e-7, "max": 4e-5}


# ------------------------------------------------- the equations in plain torch
class _Planar:
    """1-gradient planar lattice, a surface below (no polymer there) and a
    mirror above; batch members may have different numbers of layers."""
    lam = 1.0 / 6.0

    def __init__(self, layers, dev):
        L = torch.tensor(layers, device=dev)
        self.dims = (int(max(layers)),)
        i = torch.arange(self.dims[0], device=dev)
        self.valid = (i[None] < L[:, None]).double()
        self.last = (L - 1)[:, None]
        self.up = torch.minimum(i[None] + 1, self.last)
        self.weight = self.valid

    def above(self, X):
        return torch.gather(X, 1, self.up.expand(X.shape[0], -1))

    @staticmethod
    def below(X, ghost=0.0):
        return torch.cat([torch.full_like(X[:, :1], ghost), X[:, :-1]], 1)

    def average(self, X, ghost=0.0):
        return self.lam * (self.below(X, ghost) + self.above(X)) + (1 - 2 * self.lam) * X


class _Cylinder:
    """2-gradient cylindrical lattice, mirrors all round."""

    def __init__(self, nr, nz, count, dev):
        self.dims = (nr, nz)
        r = torch.arange(1, nr + 1, device=dev, dtype=torch.float64)
        area = PIE * (r ** 2 - (r - 1) ** 2)
        self.weight = area[None, :, None].expand(count, nr, nz)
        self.valid = torch.ones(count, nr, nz, device=dev, dtype=torch.float64)
        self.out = (2 * PIE * r / area / 6.0)[None, :, None]
        self.inw = (2 * PIE * (r - 1) / area / 6.0)[None, :, None]

    def average(self, X, ghost=0.0):
        lo = torch.cat([X[:, :, :1], X[:, :, :-1]], 2)
        hi = torch.cat([X[:, :, 1:], X[:, :, -1:]], 2)
        q = X * (4.0 / 6.0) + (lo + hi) / 6.0
        qm = torch.cat([q[:, :1], q[:, :-1]], 1)
        qp = torch.cat([q[:, 1:], q[:, -1:]], 1)
        return q * (4.0 / 6.0) + self.inw * qm + self.out * qp


class _Box:
    """3-gradient periodic box, 6 neighbours."""

    def __init__(self, n, dev):
        self.dims = (n, n, n)
        self.weight = self.valid = torch.ones(1, n, n, n, device=dev, dtype=torch.float64)

    def average(self, X, ghost=0.0):
        return sum(torch.roll(X, s, d) for d in (1, 2, 3) for s in (1, -1)) / 6.0


def _col(v, like):
    """A per-member value [B] (or a number) shaped for site arrays."""
    return v.reshape([-1] + [1] * (like.dim() - 1)) if isinstance(v, torch.Tensor) else v


class _Exact:
    """Residual, free energy and DIIS of one group of alike systems.

    segs: names; chi: {(a, b): [B] or number}; masks of frozen and pinned
    segments; mols: dicts with `chain` (segment index per contour position),
    or `homo` (segment, [B] lengths), or `tree` (segments, bonds); `frac`
    per segment; freedom and its value."""

    def __init__(self, lat, segs, chi, mols, frozen=None, ghost=None, pinned=None, valence=None, bond=0.0):
        self.lat, self.segs, self.mols, self.dev = lat, segs, mols, lat.valid.device
        self.frozen, self.ghost, self.pinned = frozen or {}, ghost or {}, pinned or {}
        self.valence, self.bond = valence, bond
        self.chi = {}
        for (a, b), v in chi.items():
            self.chi[a, b] = self.chi[b, a] = v
        self.ksam = lat.valid.clone()
        for m in self.frozen.values():
            self.ksam = self.ksam * (1 - m)
        # segments of the molecules with alike interactions share a field
        used = [s for m in mols for s in m["segs"]]
        same = lambda a, b: all(self._alike(self.chi.get((a, k), 0.0), self.chi.get((b, k), 0.0)) for k in segs)  # noqa: E731
        self.blocks, self.block = [], {}
        for s in used:
            if s in self.block:
                continue
            j = next((k for k, t in enumerate(self.blocks) if same(s, t)), None)
            if j is None:
                j = len(self.blocks)
                self.blocks.append(s)
            self.block[s] = j
        self.nblocks = len(self.blocks) + (1 if valence else 0)

    @staticmethod
    def _alike(a, b):
        if isinstance(a, torch.Tensor) or isinstance(b, torch.Tensor):
            return a is b
        return a == b

    # -- chains: density sums rho[seg] (before normalisation) and GN [B]
    def _total(self, X):
        return (X * self.lat.weight).flatten(1).sum(1)

    def _chain(self, seg, G1):
        avg, f = self.lat.average, [G1[seg[0]]]
        for s in seg[1:]:
            f.append(avg(f[-1]) * G1[s])
        rho, b = {}, None
        for s, Gf in zip(seg[::-1], f[::-1]):
            b = G1[s] if b is None else avg(b) * G1[s]
            rho[s] = rho.get(s, 0.0) + Gf * b
        return rho, self._total(f[-1]), {}

    def _homo(self, s, N, G1):
        """A homopolymer (lengths N [B]); also the composition on the upper
        ghost, which a charged system's dielectric constant reads there: the
        bounded forward value times the unbounded backward one."""
        g, lat, n = G1[s], self.lat, int(N.max())
        f = [g]
        for k in range(1, n):
            f.append(lat.average(f[-1]) * g)
        f = torch.stack(f)
        b, rho, edge = g, torch.zeros_like(g), torch.zeros_like(g[:, :1])
        at = torch.arange(g.shape[0], device=self.dev)
        last = lambda X: torch.gather(X, 1, lat.last)  # noqa: E731
        for k in range(n):
            row = f[(N - 1 - k).clamp(min=0), at]
            live = (N > k).double()[:, None]
            if k:
                edge = edge + live * last(row) * (5.0 / 6.0) * last(b) * last(g)
                b = lat.average(b) * g
            rho = rho + live * row * b
        return {s: rho}, self._total(f[N - 1, at]), {s: edge}

    def _homo2(self, s, N, G1):
        """The same for a second-order chain with k_stiff = 1: components
        (+z, lateral, -z), a turn weighing exp(-pi^2 / 8)."""
        g, lat, n = G1[s], self.lat, int(N.max())
        t = math.exp(-0.5 * (math.pi / 2) ** 2)
        p0, p1 = 1.0 / (1 + 4 * t), t / (1 + 4 * t)
        i = torch.arange(lat.dims[0], device=self.dev)[None]
        top = i == lat.last

        def above(X, partner):  # the mirror turns a direction into its opposite
            return torch.where(top, partner, lat.above(X))

        f = torch.empty((n, 3) + tuple(g.shape), device=self.dev, dtype=torch.float64)
        f[0] = g
        for k in range(1, n):
            a, m, c = f[k - 1]
            f[k, 0] = (p0 * lat.below(a) + 4 * p1 * lat.below(m)) * g
            f[k, 1] = (p1 * (a + c) + (2 * p1 + p0) * m) * g
            f[k, 2] = (4 * p1 * lat.above(m) + p0 * above(c, a)) * g
        at = torch.arange(g.shape[0], device=self.dev)
        last = lambda X: torch.gather(X, 1, lat.last)  # noqa: E731
        w = (1.0 / 6.0, 4.0 / 6.0, 1.0 / 6.0)
        a, m, c = g, g, g
        rho, edge = torch.zeros_like(g), torch.zeros_like(g[:, :1])
        for k in range(n):
            row = f[(N - 1 - k).clamp(min=0), :, at].unbind(1)
            live = (N > k).double()[:, None]
            if k:
                gl, ml, cl = last(g), last(m), last(c)
                eb = (4 * p1 * ml, (2 * p1 + p0) * ml + p1 * cl, 4 * p1 * ml + p0 * cl)
                edge = edge + live * gl * sum(wk * last(row[2 - j]) * eb[j] for j, wk in enumerate(w))
                up, dn = above(a, c), lat.below(c)
                a, m, c = ((p0 * up + 4 * p1 * m) * g, (p1 * (up + dn) + (2 * p1 + p0) * m) * g,
                           (4 * p1 * m + p0 * dn) * g)
            rho = rho + live * sum(wk * r * x for wk, r, x in zip(w, row, (a, m, c)))
        e = f[N - 1, :, at]
        return {s: rho}, self._total((e[:, 0] + 4 * e[:, 1] + e[:, 2]) / 6.0), {s: edge}

    def _tree(self, seg, bonds, G1):
        """Segments as nodes, `bonds` of node pairs: the density of a node is
        its weight times the averaged branch weights of its neighbours."""
        near = {i: [] for i in range(len(seg))}
        for a, b in bonds:
            near[a].append(b)
            near[b].append(a)
        memo = {}

        def branch(i, parent):  # weight of the branch of i seen from parent
            if (i, parent) not in memo:
                v = G1[seg[i]]
                for j in near[i]:
                    if j != parent:
                        v = v * self.lat.average(branch(j, i))
                memo[i, parent] = v
            return memo[i, parent]

        rho, gn = {}, None
        for i, s in enumerate(seg):
            v = branch(i, None)
            gn = self._total(v) if gn is None else gn
            rho[s] = rho.get(s, 0.0) + v * G1[s]
        return rho, gn, {}

    def residual(self, x):
        """x: [B, blocks, sites...] -> (g, free energy [B], grand potential [B])"""
        lat, nb = self.lat, len(self.blocks)
        psi = x[:, nb] if self.valence else None
        if psi is not None:
            kT, e, eps0 = 1.38065e-23 * 298.15, 1.60217e-19, 8.85418e-12
            psi_lo = torch.cat([psi[:, :1], psi[:, :-1]], 1)
            EE = 0.25 * eps0 * self.bond / kT * (kT / e) ** 2 * ((psi_lo - psi) ** 2 + (psi - lat.above(psi)) ** 2)
        G1 = {}
        for s, j in self.block.items():
            u = x[:, j]
            if psi is not None:
                u = u - 80.0 * EE + _col(self.valence.get(s, 0.0), u) * psi
            G1[s] = torch.exp(-u) * self.ksam * self.pinned.get(s, 1.0)
        norm, bulk, tot, rhos, edges = [], [], [], [], []
        for m in self.mols:
            if "homo" in m:
                rho, gn, edge = (self._homo2 if m.get("markov") == 2 else self._homo)(*m["homo"], G1)
            elif "tree" in m:
                rho, gn, edge = self._tree(*m["tree"], G1)
            else:
                rho, gn, edge = self._chain(m["chain"], G1)
            rhos.append(rho)
            edges.append(edge)
            tot.append(gn)
        B = A = 0.0
        charge = lambda s: self.valence.get(s, 0.0)  # noqa: E731
        for m, gn in zip(self.mols, tot):
            f, v, N = m["freedom"], m.get("value"), m["N"]
            nrm = v / gn if f == "n" else (v / N / gn if f == "theta" else (v / N if f == "free" else None))
            pb = 0.0 * gn if m.get("grafted") else (N * nrm if f in ("n", "theta") else (v + 0.0 * gn if f == "free" else None))
            if f in ("n", "theta", "free"):
                B = B + pb
                if self.valence:
                    A = A + pb * charge(m["segs"][0])
            norm.append(nrm)
            bulk.append(pb)
        for k, m in enumerate(self.mols):  # the neutralizer, then the solvent, fill the bulk
            if m["freedom"] == "neutralizer":
                bulk[k] = -A / charge(m["segs"][0])
                B = B + bulk[k]
        for k, m in enumerate(self.mols):
            if m["freedom"] == "solvent":
                bulk[k] = 1.0 - B
            if norm[k] is None or m["freedom"] == "free":
                norm[k] = bulk[k] / m["N"]
        phi = {s: mk.clone() for s, mk in self.frozen.items()}
        pt = sum(self.frozen.values()) if self.frozen else torch.zeros_like(x[:, 0])
        edge_tot, mphi, seg_bulk = 0.0, [], {}
        for k, m in enumerate(self.mols):
            mine = 0.0
            for s, r in rhos[k].items():
                p = torch.where(G1[s] != 0, r / torch.where(G1[s] != 0, G1[s], torch.ones_like(r)), 0.0 * r) * _col(norm[k], r)
                phi[s] = phi.get(s, 0.0) + p
                mine = mine + p
                if edges[k]:
                    edge_tot = edge_tot + edges[k][s] / torch.gather(G1[s], 1, lat.last) * norm[k][:, None]
                seg_bulk[s] = seg_bulk.get(s, 0.0) + m["frac"][s] * bulk[k]
            mphi.append(mine)
            pt = pt + mine
        side = {s: lat.average(p, self.ghost.get(s, 0.0)) for s, p in phi.items()}
        for s, gh in self.ghost.items():
            if s not in phi:
                side[s] = lat.average(torch.zeros_like(pt), gh)
        ok = pt > 0
        safe = torch.where(ok, pt, torch.ones_like(pt))
        gv = []
        for j, s in enumerate(self.blocks):
            g = x[:, j]
            for k in side:
                c = self.chi.get((s, k), 0.0)
                if isinstance(c, torch.Tensor) or c != 0:
                    g = g - _col(c, g) * (side[k] / safe - _col(seg_bulk.get(k, 0.0), g))
            gv.append(g)
        alpha = sum(gv) / len(gv)
        out = [torch.where(ok, g - alpha + 1 / safe - 1, 0.0 * g) * self.ksam for g in gv]
        if psi is not None:
            out.append(self._poisson(psi, phi, safe, edge_tot))
        F, GP = (None, None) if psi is not None or self.ghost else self._thermo(G1, phi, side, mphi, bulk, tot, norm, seg_bulk, alpha)
        return torch.stack(out, 1), F, GP

    def _poisson(self, psi, phi, pt, edge_tot):
        """psi minus one upwind sweep of the Poisson equation from the wall."""
        lat = self.lat
        kT, e, eps0 = 1.38065e-23 * 298.15, 1.60217e-19, 8.85418e-12
        C = 2 * e * e / (eps0 * kT * self.bond)
        q = sum(_col(self.valence.get(s, 0.0), p) * p for s, p in phi.items()) / pt
        all_phi = sum(phi.values())
        eps = 80.0 * all_phi / pt
        eps_lo = lat.below(eps, 80.0)
        ghost = 80.0 * torch.gather(all_phi, 1, lat.last) / edge_tot
        top = torch.arange(lat.dims[0], device=self.dev)[None] == lat.last
        eps_hi = torch.where(top, ghost, lat.above(eps))
        em, ep, up = eps_lo + eps, eps + eps_hi, lat.above(psi)
        X, prev = [], psi[:, 0]
        for i in range(lat.dims[0]):
            prev = (em[:, i] * prev + C * q[:, i] + ep[:, i] * up[:, i]) / (em[:, i] + ep[:, i])
            X.append(prev)
        return torch.where(lat.valid > 0, psi - torch.stack(X, 1), 0.0 * psi)

    def _thermo(self, G1, phi, side, mphi, bulk, tot, norm, seg_bulk, alpha):
        F = GP = 0.0
        chi = lambda a, b: self.chi.get((a, b), 0.0)  # noqa: E731
        for k, m in enumerate(self.mols):
            N, fr = m["N"], m["frac"]
            mu0 = torch.log(N * norm[k]) / N
            const = sum(-fr[a] * fr[b] * chi(a, b) / 2 for a in fr for b in fr)
            F = F + (_col(mu0, alpha) + const) * mphi[k]
            GP = GP + (mphi[k] - _col(bulk[k], alpha)) / N
        GP = GP + alpha
        for s in G1:
            lg = torch.log(torch.where(G1[s] > 0, G1[s], torch.ones_like(G1[s])))
            F = F + phi[s] * lg
        for a in G1:
            for b in phi:
                half = 1.0 if b in self.frozen else 0.5
                F = F + phi[a] * side[b] * (chi(a, b) * half)
                if b not in self.frozen:
                    GP = GP + (phi[a] * side[b] - _col(seg_bulk[a] * seg_bulk[b], alpha)) * (chi(a, b) / 2)
        return self._total(F * self.ksam), self._total(-GP * self.ksam)

    def diis(self, x, its):
        """`its` iterations; returns x, the last residual norm, F and GP there"""
        B = x.shape[0]
        g = self.residual(x)[0]
        x = x - DMAX * g
        xr, er, res, F, GP = [], [], None, None, None
        for _ in range(its):
            g, F, GP = self.residual(x)
            res = g.flatten(1).norm(dim=1)
            new = x - DMAX * g
            xr, er = (xr + [new])[-HISTORY:], (er + [(new - x).flatten(1)])[-HISTORY:]
            A = torch.stack([torch.stack([(a * b).sum(1) for b in er], 1) for a in er], 1) + 1e-9
            c = torch.linalg.solve(A, torch.ones(B, len(er), 1, device=self.dev, dtype=torch.float64))[..., 0]
            c = c / c.sum(1, keepdim=True)
            x = sum(_col(c[:, i], x) * v for i, v in enumerate(xr))
        return x, res, F, GP


def _solvent(N=1):
    return dict(segs=["W"], chain=["W"], freedom="solvent", N=N, frac={"W": 1.0})


def _group(case, members, dev, chi=None):
    """The _Exact of members of one order."""
    fam, d0 = case["family"], members[0]
    val = lambda k: torch.tensor([float(d[k]) for d in members], device=dev, dtype=torch.float64)  # noqa: E731
    if fam in ("adsorption", "charged", "branched"):
        lat = _Planar([d["layers"] for d in members], dev)
    if fam in ("adsorption", "charged"):
        N = torch.tensor([d["N"] for d in members], device=dev)
        pol = dict(segs=["A"], homo=("A", N), markov=d0["markov"], N=N.double(), frac={"A": 1.0})
    if fam == "adsorption":
        pol.update(freedom="free", value=val("phib"))
        return _Exact(lat, ["S", "A", "W"], {("S", "A"): val("chi_s"), ("A", "W"): val("chi")}, [pol, _solvent()],
                      ghost={"S": 1.0})
    if fam == "charged":
        pol.update(freedom="theta", value=val("theta"))
        mono = lambda s, **k: dict(segs=[s], chain=[s], N=1, frac={s: 1.0}, **k)  # noqa: E731
        return _Exact(lat, ["S", "A", "W", "Na", "Cl"], {("S", "A"): val("chi_s")},
                      [pol, mono("Na", freedom="neutralizer"), mono("Cl", freedom="free", value=val("salt")), _solvent()],
                      ghost={"S": 1.0}, valence={"A": val("valence"), "Na": 1.0, "Cl": -1.0}, bond=3e-10)
    if fam == "branched":
        n = d0["N"]
        seg = ["C"] * n + ["N"] * 4  # the tail, the head segment, its two side segments, the end
        bonds = [(i, i + 1) for i in range(n)] + [(n, n + 1), (n, n + 2), (n, n + 3)]
        surf = dict(segs=["N", "C"], tree=(seg, bonds), N=n + 4, frac={"C": n / (n + 4.0), "N": 4 / (n + 4.0)},
                    freedom="theta", value=d0["theta"])
        return _Exact(lat, ["S", "C", "N", "W"], {("S", "C"): d0["chi_s"], ("C", "W"): d0["chi"], ("N", "W"): -0.3},
                      [surf, _solvent()], ghost={"S": 1.0})
    if fam == "brush":
        nr, nz, N = d0["nr"], d0["nz"], d0["N"]
        lat = _Cylinder(nr, nz, len(members), dev)
        rod, graft = torch.zeros_like(lat.valid), torch.zeros_like(lat.valid)
        rod[:, 0], graft[:, 1] = 1.0, 1.0
        brush = dict(segs=["X", "A"], chain=["X"] + ["A"] * (N - 1), N=N, frac={"X": 1.0 / N, "A": (N - 1.0) / N},
                     freedom="n", value=0.05 * 2 * PIE * nz, grafted=True)
        return _Exact(lat, ["S", "X", "A", "W"], {("A", "W"): d0["chi"] if chi is None else chi},
                      [brush, _solvent()], frozen={"S": rod}, pinned={"X": graft})
    n = d0["n"]
    surf = dict(segs=["A", "B"], chain=["A"] * 10 + ["B"] * 10, N=20, frac={"A": 0.5, "B": 0.5}, freedom="theta",
                value=d0["frac"] * n ** 3)
    return _Exact(_Box(n, dev), ["A", "B", "W"], {("B", "W"): 1.6, ("A", "B"): 1.6}, [surf, _solvent()])


def _inside(dims):
    return (slice(None),) + tuple(slice(1, n + 1) for n in dims)


def _strip(x, blocks, dims):
    """Flat fields with ghost layers -> [blocks, sites...] without them."""
    return x.reshape([blocks] + [n + 2 for n in dims])[_inside(dims)]


def _dress(flat, x, blocks, dims):
    """`flat` with the interior values replaced by x: ghost values never change."""
    out = np.array(flat).reshape([blocks] + [n + 2 for n in dims])
    out[_inside(dims)] = x
    return out.ravel()


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    members = _members(case, seed)
    if case["entry"] == "queue":
        e = _group(case, members, dev, CHIS[0])
        dims = e.lat.dims
        size = len(e.blocks) * (dims[0] + 2) * (dims[1] + 2)
        x0 = [_start(case, d, seed, i, None, size) for i, d in enumerate(members)]
        # the grafted segment's field is shared while chi is 0
        x = torch.tensor(np.stack([_strip(v, len(e.blocks), dims) for v in x0]), device=dev)
        edge, names, out = x0[0].reshape([len(e.blocks)] + [n + 2 for n in dims]), e.blocks, []
        for chi in CHIS:
            e = _group(case, members, dev, chi)
            zero = torch.zeros_like(x[:, 0])
            x = torch.stack([x[:, names.index(s)] if s in names else zero for s in e.blocks], 1)
            edge = np.stack([edge[names.index(s)] if s in names else 0 * edge[0] for s in e.blocks])
            names = e.blocks
            x, res, F, GP = e.diis(x, case["its"])
            out.append((F, GP, res))
        got = [torch.stack([o[k] for o in out], 1).cpu().numpy() for k in range(3)]
        got = dict(zip(("free_energy", "grand_potential", "residual"), got))
        if len(members) == 1:
            got["x"] = _dress(edge, x[0].cpu().numpy(), len(names), dims)
        return got
    groups = {}
    for i, d in enumerate(members):
        groups.setdefault(d.get("markov", 1), []).append(i)
    xs, rs = [None] * len(members), [None] * len(members)
    for ids in groups.values():
        mine = [members[i] for i in ids]
        e = _group(case, mine, dev)
        sizes = [tuple([d["layers"]]) if "layers" in d else e.lat.dims for d in mine]
        flat = [_start(case, d, seed, i, e.blocks, e.nblocks * int(np.prod([n + 2 for n in sz])))
                for i, d, sz in zip(ids, mine, sizes)]
        x = np.zeros((len(ids), e.nblocks) + e.lat.dims)
        for k, (v, sz) in enumerate(zip(flat, sizes)):
            x[k][(slice(None),) + tuple(slice(0, n) for n in sz)] = _strip(v, e.nblocks, sz)
        x = torch.tensor(x, device=dev)
        if case["entry"] == "residual":
            g = e.residual(x)[0]
            return {"g": _dress(0 * flat[0], g[0].cpu().numpy(), e.nblocks, sizes[0]), "residual": float(g.norm())}
        if case["entry"] == "newton":
            F = lambda v: e.residual(v.reshape(x.shape))[0].reshape(-1)  # noqa: E731
            v = x.reshape(-1)
            for _ in range(60):
                g = F(v)
                if float(g.norm()) < 1e-12:
                    break
                J = torch.func.jacfwd(F)(v)
                step = torch.linalg.solve(J, g)
                t = min(1.0, 1.0 / max(1e-300, float(step.abs().max())))
                while t > 1e-6 and not float(F(v - t * step).norm()) < float(g.norm()):
                    t *= 0.5
                if t <= 1e-6:
                    break
                v = v - t * step
            return {"x": _dress(flat[0], v.reshape(x.shape)[0].cpu().numpy(), e.nblocks, sizes[0])}
        x, res, _, _ = e.diis(x, case["its"])
        x, res = x.cpu().numpy(), res.cpu().numpy()
        for k, (i, v, sz) in enumerate(zip(ids, flat, sizes)):
            xs[i] = _dress(v, x[k][(slice(None),) + tuple(slice(0, n) for n in sz)], e.nblocks, sz)
            rs[i] = res[k]
    if len(members) == 1:
        return {"x": xs[0], "residual": float(rs[0])}
    return {"x": np.concatenate(xs), "residual": np.array(rs)}
