"""The measured work: the calls that programs built on this framework make, over the ranges they make
them in, each through its public entry points (Population.run, Network.run and the reads after them).

A case is one call that advances a population (or a network) by a number of 0.125 ms output intervals
and takes its recorded trace and its final voltages.  The populations and solvers are those of the
command line and the benchmark: the reference's own morphologies with the population-global solvers
(RKC, Crank-Nicolson, backward Euler), the exact tree solve, and the per-cell engines on synthetic
Purkinje trees.  A state keeps its population, as a program does, and every pass continues it.

exact() restates the Purkinje and olive models and their solvers in plain 64-bit torch and numpy.
Golgi and granule cells and the network have no such restatement.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cerebellum-neuron-model-simulation-using-rkc_amd"))

import cbrkc  # noqa: E402

DATA = os.path.join(ROOT, "tests", "golden", "ref_data")
H = 0.125
SOLVER = {"rkc": cbrkc.RKC, "cn": cbrkc.CN, "be": cbrkc.BE}
ENGINE = {"global": cbrkc.ENGINE_GLOBAL_FP64, "tree": cbrkc.ENGINE_TREE_FP64,
          "cell": cbrkc.ENGINE_CELL_FP64, "mixed": cbrkc.ENGINE_CELL_MIXED}
# cell: type, file, compartments, recorded compartment, initial voltage range [mV].  On the reference's
# morphologies the stimulus is the reference's own protocol (a window that opens 50 ms or more into the
# run), on the synthetic trees the benchmark's soma currents from the start.
CELL = {
    "olive": (cbrkc.IO, "IO.txt", 3, 0, (-62.0, -58.0)),
    "golgi": (cbrkc.GO, "Go_131.txt", 131, 30, (-62.0, -58.0)),
    "granule": (cbrkc.GR, "Gr.txt", 578, 16, (-72.0, -68.0)),
    "purkinje": (cbrkc.PKJ, "Pkj.txt", 1600, 1599, (-69.0, -66.0)),
}
CURRENT = (0.2e-3, 1.0e-3)   # soma currents of the synthetic trees
# the dendritic drive of the per-cell engines' benchmark
DRIVE = dict(rate_hz=5.0, g_mS=1e-6, tau_ms=2.0, e_mV=0.0)


def _case(name, cell, solver, engine, nx, ny, steps, synthetic=False, coupled=False):
    return dict(name=name, cell=cell, solver=solver, engine=engine, nx=nx, ny=ny, steps=steps,
                synthetic=synthetic, coupled=coupled)


def listed():
    return [
        # the reference's small olive grid, 5 ms a call
        _case("olive 8x8 rkc", "olive", "rkc", "global", 8, 8, 40),
        # a larger olive grid on the second solver (BiCG on the unsymmetric coupling)
        _case("olive 32x32 cn", "olive", "cn", "global", 32, 32, 8),
        # Golgi grid, gap junctions in the cable matrix
        _case("golgi 16x16 rkc", "golgi", "rkc", "global", 16, 16, 40),
        # granule cells at the reference's 1e-9 tolerance: hundreds of step attempts an interval
        _case("granule 4x4 rkc", "granule", "rkc", "global", 4, 4, 1),
        # the same cells, many of them, on the exact tree solve
        _case("granule 16x16 cn tree", "granule", "cn", "tree", 16, 16, 8),
        # the plain workload: nine synthetic Purkinje trees, one controller, rtol 1e-4
        _case("purkinje 9 rkc", "purkinje", "rkc", "global", 9, 1, 8, synthetic=True),
        # the reference's Purkinje grid with its gap junctions
        _case("purkinje 8x8 coupled rkc", "purkinje", "rkc", "global", 8, 8, 8, coupled=True),
        # the reference's CG, 100 iterations a step
        _case("purkinje 64 cn", "purkinje", "cn", "global", 1, 64, 2),
        # the exact tree solve at the size of the headline workload
        _case("purkinje 1024 cn tree", "purkinje", "cn", "tree", 1, 1024, 8),
        # the per-cell engines on driven synthetic trees: FP64, and the headline mixed engine
        _case("purkinje 256 cell", "purkinje", "rkc", "cell", 256, 1, 16, synthetic=True),
        _case("purkinje 1024 mixed", "purkinje", "rkc", "mixed", 1024, 1, 80, synthetic=True),
        # granule, Golgi and Purkinje cells with their synapses (a quarter of the full network's cells)
        _case("network 512/128/128", "network", "rkc", "mixed", 512, 128, 16, synthetic=True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["olive", "golgi", "granule", "granule tree", "purkinje", "coupled", "krylov", "tree", "cell",
                       "mixed", "network"])
    if kind == "olive":
        solver = rng.choice(["rkc", "cn", "be"])
        return _case("", "olive", solver, "global", _log(rng, 2, 40), _log(rng, 2, 40),
                     rng.randint(20, 60) if solver == "rkc" else rng.randint(4, 12))
    if kind == "golgi":
        solver = rng.choice(["rkc", "rkc", "cn", "be"])
        return _case("", "golgi", solver, "global", _log(rng, 1, 24), _log(rng, 1, 24),
                     rng.randint(20, 60) if solver == "rkc" else rng.randint(1, 4))
    if kind == "granule":
        solver = rng.choice(["rkc", "rkc", "cn", "be"])
        return _case("", "granule", solver, "global", _log(rng, 1, 12), _log(rng, 1, 12), rng.randint(1, 2))
    if kind == "granule tree":
        return _case("", "granule", rng.choice(["cn", "be"]), "tree", _log(rng, 1, 24), _log(rng, 1, 24),
                     rng.randint(4, 12))
    if kind == "purkinje":
        return _case("", "purkinje", "rkc", "global", _log(rng, 1, 160), 1, rng.randint(4, 12), synthetic=True)
    if kind == "coupled":
        return _case("", "purkinje", "rkc", "global", _log(rng, 2, 12), _log(rng, 1, 12), rng.randint(4, 12),
                     coupled=True)
    if kind == "krylov":
        return _case("", "purkinje", rng.choice(["cn", "be"]), "global", 1, _log(rng, 1, 150), rng.randint(1, 3))
    if kind == "tree":
        return _case("", "purkinje", rng.choice(["cn", "be"]), "tree", 1, _log(rng, 1, 1024), rng.randint(2, 10))
    if kind == "cell":
        return _case("", "purkinje", "rkc", "cell", _log(rng, 1, 400), 1, _log(rng, 2, 32), synthetic=True)
    if kind == "mixed":
        return _case("", "purkinje", "rkc", "mixed", _log(rng, 1, 1000), 1, _log(rng, 2, 80), synthetic=True)
    nx = _log(rng, 32, 512)
    return _case("", "network", "rkc", "mixed", nx, max(8, nx // 4), rng.randint(4, 16), synthetic=True)


def _file(name, n, write):
    """A generated morphology, written once: the reconstructed trees stay the same when the inputs change."""
    d = os.path.join(tempfile.gettempdir(), "cbrkc_perf_%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, "%s%d.txt" % (name, n))
    if not os.path.exists(path):
        part = "%s.%d" % (path, os.getpid())
        write(part)
        os.replace(part, path)
    return path


def _pkj_trees(n):
    return _file("pkj", n, lambda p: cbrkc.synth_pkj_morph(p, seed=2024, ncell=n))


def _inputs(case, seed):
    """initial voltages and stimulus amplitudes of every cell"""
    rng = np.random.default_rng(seed)
    n = case["nx"] * case["ny"]
    return rng.uniform(*CELL[case["cell"]][4], n), rng.uniform(*CURRENT, n)


def _tolerances(case):
    """the plain workload's for the population-global engine on synthetic trees, the defaults' elsewhere"""
    if not case["synthetic"]:
        return {}
    return dict(atol=1e-6, rtol=1e-4 if case["engine"] == "global" else 1e-6, **cbrkc.STABLE)


def prepare(case, seed):
    if case["cell"] == "network":
        return _prepare_network(case, seed)
    ctype, fname, _, rec, _ = CELL[case["cell"]]
    v0, amp = _inputs(case, seed)
    n = len(v0)
    morph = _pkj_trees(n) if case["synthetic"] else os.path.join(DATA, fname)
    kw = _tolerances(case)
    if case["engine"] in ("cell", "mixed"):
        kw["poisson"] = dict(DRIVE, seed=seed)
    pop = cbrkc.Population(ctype, case["nx"], case["ny"], solver=SOLVER[case["solver"]], engine=ENGINE[case["engine"]],
                           morph=morph, gj=os.path.join(DATA, "Pkj_GJ.csv") if case["coupled"] else "", v0=v0,
                           stim=(rec, 0.0, 1e9, amp) if case["synthetic"] else None, **kw)
    if case["engine"] == "mixed":
        pop.autotune(0, threads=512)
    return {"case": case, "pop": pop, "t": 0.0}


def _prepare_network(case, seed):
    n = (case["nx"], case["ny"], case["ny"])
    rng = np.random.default_rng(seed)
    v = [rng.uniform(lo, hi, k) for (lo, hi), k in zip(((-72.0, -68.0), (-62.0, -58.0), (-69.0, -66.0)), n)]
    gr_file = _file("gr", n[0], lambda p: cbrkc.synth_gr_chains(p, os.path.join(DATA, "Gr.txt"), 2024, n[0]))
    go_file = _file("go", n[1], lambda p: cbrkc.synth_go_trees(p, os.path.join(DATA, "Go_131.txt"), 2025, n[1]))
    gr = cbrkc.Population(cbrkc.GR, n[0], 1, morph=gr_file, comp=4, v0=v[0], stim="none")
    go = cbrkc.Population(cbrkc.GO, n[1], 1, morph=go_file, v0=v[1], stim="none")
    pkj = cbrkc.Population(cbrkc.PKJ, n[2], 1, morph=_pkj_trees(n[2]), v0=v[2], atol=1e-6, rtol=1e-6, stim="none",
                           engine=cbrkc.ENGINE_CELL_MIXED, **cbrkc.STABLE)
    pkj.autotune(0, threads=512)
    net = cbrkc.Network(gr, go, pkj, cfg=cbrkc.net_config(seed=seed, total=0))
    return {"case": case, "net": net, "pops": (gr, go, pkj)}


def run(state):
    case = state["case"]
    if "net" in state:
        state["net"].run(case["steps"])
        out = {"v%d" % k: p.read() for k, p in enumerate(state["pops"])}
        out["ampa"] = state["net"].conductance(cbrkc.NET_PKJ, cbrkc.NET_AMPA)
        return out
    pop = state["pop"]
    trace = pop.run(case["steps"], state["t"], CELL[case["cell"]][3])
    state["t"] += case["steps"] * H
    return {"trace": trace, "v": pop.read()}


# Per cell type: doubles of state per compartment that a call reads and writes (gates, Ca, reversal, the
# integrator's vectors) and reads only (conductances, cable, areas); operations of one ion update and
# of one right-hand side per compartment (an exponential counted as 20); and, per interval on the
# RKC path, ion updates and right-hand sides as the solver's counters give them on these workloads.
WORK = {
    "olive": (18, 14, 500, 20, 3, 100),
    "golgi": (38, 22, 1500, 20, 4, 115),
    "granule": (42, 16, 2500, 20, 50, 5000),
    "purkinje": (25, 18, 900, 20, 19, 160),
}


def work(case):
    if case["cell"] == "network":
        parts = [("granule", 4 * case["nx"]), ("golgi", 131 * case["ny"]), ("purkinje", 1600 * case["ny"])]
    else:
        parts = [(case["cell"], CELL[case["cell"]][2] * case["nx"] * case["ny"])]
    total = {"bytes": 0.0, "flops": 0.0}
    for cell, nc in parts:
        rw, ro, ion, rhs, ions, evals = WORK[cell]
        if case["solver"] != "rkc":   # five steps an interval, a solve each
            ions, evals = 5, (5 * 30 if case["engine"] == "tree" else 5 * 100)
        word = 4 if case["engine"] == "mixed" and cell == "purkinje" else 8
        total["bytes"] += nc * word * (2 * rw + ro) + 8 * nc
        total["flops"] += float(nc) * case["steps"] * (ions * ion + evals * rhs)
    return total


def tolerance(case):
    """About four times what the results move when the initial voltages change in their last bit (32-bit
    rounding on the mixed engine) or a norm is summed in another order.  An adaptive step near a spike
    amplifies such a change, most of all where every cell fires its first spike together."""
    if case["cell"] == "network":
        return {"rel": 2e-3, "max": 0.1}
    if case["engine"] == "mixed":
        return {"rel": 0.03, "max": 0.9}
    if case["engine"] == "cell":
        return {"rel": 2e-3, "max": 0.1}
    if case["solver"] != "rkc":
        if case["engine"] == "global" and (case["cell"] == "granule" or case["solver"] == "be"):
            return {"rel": 1e-6, "max": 4e-5}   # the iteration stops at its cap, far from converged
        return {"rel": 4e-9, "max": 1e-7}
    if case["cell"] == "purkinje":
        return {"rel": 1e-3, "max": 2e-2} if case["synthetic"] else {"rel": 1e-8, "max": 1e-7}
    return {"rel": 1e-5, "max": 1e-4} if case["cell"] == "granule" else {"rel": 1e-4, "max": 2e-3}


# ---- the same results in plain 64-bit torch and numpy ----

def exact(case, seed):
    if case["cell"] not in ("purkinje", "olive") or case["solver"] == "be":
        return None
    n = case["nx"] * case["ny"]
    if case["engine"] in ("cell", "mixed") and n * case["steps"] > 4000:
        return None   # the cells' controllers in lock step: over 20 s
    v0, amp = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() and n * CELL[case["cell"]][2] > 4000 else "cpu"
    cls = _Purkinje if case["cell"] == "purkinje" else _Olive
    m = cls(case, v0, amp, dev, seed)
    rec = CELL[case["cell"]][3]
    if case["solver"] == "rkc":
        sol = _Rkc(m, n if case["engine"] in ("cell", "mixed") else 1, case)
    else:
        sol = _Cn(m, case)
    trace = []
    for k in range(case["steps"]):
        m.interval(k)
        trace.append(sol.advance().view(n, -1)[:, rec].cpu().numpy())
    return {"trace": np.array(trace), "v": sol.v_out.cpu().numpy()}


class _Cable:
    """sum over neighbours of g (y_j - y_i), the neighbours of every compartment padded to one width"""

    def __init__(self, nc, i, j, g, dev):
        order = np.lexsort((j, i))
        i, j, g = i[order], j[order], g[order]
        deg = np.bincount(i, minlength=nc)
        slot = np.arange(len(i)) - np.repeat(np.cumsum(deg) - deg, deg)
        nb = np.tile(np.arange(nc), (max(1, deg.max()), 1))
        w = np.zeros(nb.shape)
        nb[slot, i], w[slot, i] = j, g
        self.nb, self.w = torch.tensor(nb, device=dev), torch.tensor(w, device=dev)
        self.gsum = self.w.sum(0)

    def lap(self, y):
        return (self.w * (y[self.nb] - y)).sum(0)


def _rate(v, A, B, C, D):
    return A / (B + torch.exp((v + C) / D))


def _cn(x, inf, tau, dt):
    return (2 * dt * inf + (2 * tau - dt) * x) / (2 * tau + dt)


class _Purkinje:
    HMIN, STRICT = 2.0 ** -10, False
    # gates of two rates: (alpha, beta) arguments of _rate
    TWO = {
        "mNaF": ((35, 0, 5, -10), (7, 0, 65, 20)), "hNaF": ((0.225, 1, 80, 10), (7.5, 0, -3, -18)),
        "mNaP": ((200, 1, -18, -16), (25, 1, 58, 8)), "mCaP": ((8.5, 1, -8, -12.5), (35, 1, 74, 14.5)),
        "hCaP": ((0.0015, 1, 29, 8), (0.0055, 1, 23, -8)), "mCaT": ((2.6, 1, 21, -8), (0.18, 1, 40, 4)),
        "hCaT": ((0.0025, 1, 40, 8), (0.19, 1, 50, -10)), "mKA": ((1.4, 1, 27, -12), (0.49, 1, 30, 4)),
        "hKA": ((0.0175, 1, 50, 8), (1.3, 1, 13, -10)),
    }
    DENSITY = np.array([[7500.0, 1.0, 0.0, 0.5, 0.3, 600.0, 0.040, 15.0, 0.0, 0.0],
                        [0.0, 0.0, 4.5, 0.5, 0.0, 60.0, 0.01, 2.0, 80.0, 0.39],
                        [0.0, 0.0, 4.5, 0.5, 0.0, 0.0, 0.013, 0.0, 80.0, 0.39]])

    def __init__(self, case, v0, amp, dev, seed):
        n, C = len(v0), 1600
        self.n, self.comp, self.dev = n, C, dev
        rows = np.loadtxt(_pkj_trees(n) if case["synthetic"] else os.path.join(DATA, "Pkj.txt"))[:, :7]
        rows = np.tile(rows, (n if len(rows) == C else 1, 1))
        base = np.repeat(np.arange(n) * C, C)
        at = base + rows[:, 0].astype(int)
        put = lambda x: (lambda o: (o.__setitem__(at, x), o)[1])(np.zeros(n * C))  # noqa: E731
        d, typ = put(rows[:, 5]) * 1e-4, put(rows[:, 6]).astype(int)
        par = put(rows[:, 1]).astype(int)
        soma = typ == 0
        ln = np.where(soma, d, np.sqrt(put((rows[:, 2:5] ** 2).sum(1))) * 1e-4)
        r = d / 2
        area = np.where(soma, 4 * np.pi * r * r, 2 * np.pi * r * ln)
        sh = 0.2e-4
        shell = np.where(soma, sh - 2 * sh ** 2 / d + 4 * sh ** 3 / (3 * d * d), sh - sh ** 2 / d) * area
        full = np.where(typ == 3, area + ln * 1.33e-8 * 13.0e4, area)
        i = np.nonzero(par >= 0)[0]
        p = base[i] + par[i]
        g = 2.0 / (0.25 * ln[i] / (r[i] ** 2 * np.pi) + 0.25 * ln[p] / (r[p] ** 2 * np.pi))
        self.parent = np.where(par >= 0, par, -1).reshape(n, C)
        self.g_parent = np.zeros(n * C)
        self.g_parent[i] = g
        a, b, w = [i, p], [p, i], [g, g]
        if case["coupled"]:
            gj = np.loadtxt(os.path.join(DATA, "Pkj_GJ.csv"), delimiter=",", dtype=int)
            for y in range(case["ny"]):
                for x in range(case["nx"] - 1):
                    e, f = gj[:, 0] + (x + y * case["nx"]) * C, gj[:, 1] + (x + 1 + y * case["nx"]) * C
                    a, b, w = a + [e, f], b + [f, e], w + [np.full(len(e), 2.5e-6)] * 2
        self.cable = _Cable(n * C, np.concatenate(a), np.concatenate(b), np.concatenate(w), dev)
        t = lambda x: torch.tensor(x, device=dev, dtype=torch.float64)  # noqa: E731
        self.cm, self.shell = t(1.64 * full), t(shell)
        dens = self.DENSITY[np.where(soma, 0, np.where(typ == 1, 1, 2))] * area[:, None]
        self.leak = t(full / np.where(soma, 10.0, 30.0))
        self.c = [t(dens[:, k]) for k in range(10)]
        self.v = t(np.repeat(v0, C))
        self.ca, self.rev = torch.full_like(self.v, 4.0e-5), torch.full_like(self.v, 135.0)
        self.fixed = torch.arange(n * C, device=dev) % 1599 == 0
        self.iext, self.amp = torch.zeros_like(self.v), t(amp) if case["synthetic"] else None
        v = self.v
        self.g = {k: (lambda x, y: x / (x + y))(_rate(v, *ab[0]), _rate(v, *ab[1])) for k, ab in self.TWO.items()}
        inf, _ = self._others(v, self.ca)
        self.g.update(inf)
        self.syn = None
        if case["engine"] in ("cell", "mixed"):
            self.syn, self.seed = torch.zeros_like(v), seed

    def interval(self, k):
        if self.amp is not None:
            self.iext.view(self.n, -1)[:, 1599] = self.amp
        if self.syn is not None:
            u = _philox_uniform(np.arange(len(self.v)), k, self.seed)
            hit = torch.tensor(u < 1.0 - math.exp(-DRIVE["rate_hz"] * H * 1e-3), device=self.dev)
            self.syn = self.syn * math.exp(-H / DRIVE["tau_ms"]) + hit * DRIVE["g_mS"]

    @staticmethod
    def _others(v, caq):
        """steady states and time constants of the gates that are not of two rates"""
        kdr = lambda u: torch.where(u.abs() > 1e-6, -0.0235 * u / (torch.exp(-u / 12) - 1), 0.0235 * 12.0)  # noqa: E731
        inf, tau = {}, {}
        e = 1 + torch.exp((v + 82) / 7)
        inf["mKh1"], tau["mKh1"], inf["mKh2"], tau["mKh2"] = 0.8 / e, 7.6, 0.2 / e, 36.8
        a, b = kdr(v - 8), 5 * torch.exp(-(v + 127) / 30)
        inf["mKdr"], tau["mKdr"] = a / (a + b), 1 / (kdr(v + 12) + 5 * torch.exp(-(v + 147) / 30))
        inf["hKdr"] = 1 / (1 + torch.exp((v + 25) / 4))
        tau["hKdr"] = torch.where(v < -25, 1200.0, 10.0)
        inf["mKM"] = 1 / (1 + torch.exp(-(v + 35) / 10))
        tau["mKM"] = 200 / (3.3 * torch.exp((v + 35) / 20) + torch.exp(-(v + 35) / 20))
        for k, a, (A, B, C, D), z, s in (("KC", 7.5, (0.11, 0, -35, 14.9), 4.0, "z"), ("K2", 25.0, (0.075, 0, 25, 6), 0.2, "z")):
            b = _rate(v, A, B, C, D)
            inf["m" + k], tau["m" + k] = a / (a + b), 1 / (a + b)
            inf[s + k], tau[s + k] = 1 / (1 + z / caq), 10.0
        return inf, tau

    def ion(self, v_new, dt, extrapolate=False):
        """the state after an ion update over dt [per compartment]; CN: gates at the extrapolated voltage"""
        g, c = dict(self.g), self.c
        vo = v_new if extrapolate else self.v
        vm = 1.5 * v_new - 0.5 * self.vold if extrapolate else 0.5 * (v_new + vo)
        i_ca = 1e-3 * (vo - self.rev) * (c[2] * g["mCaP"] * g["hCaP"] + c[3] * g["mCaT"] * g["hCaT"])
        i_ca = torch.clamp(-i_ca, min=0) / (2 * 9.6485e4 * self.shell)
        f = lambda ca: dt * (i_ca - 10.0 * (ca - 4.0e-5))  # noqa: E731
        k1 = f(self.ca)
        k2 = f(self.ca + k1 / 2)
        k3 = f(self.ca + k2 / 2)
        ca = self.ca + (k1 + 2 * k2 + 2 * k3 + f(self.ca + k3)) / 6
        mid = 0.5 * (self.ca + ca)
        rev = torch.where(self.fixed, 12.5 * math.log(2.4 / 4.0e-5), 13.361624877 * torch.log(2.4 / mid))
        caq = torch.floor((mid * 1000 - 0.04) / 0.099986667) * 0.099986667 + 0.04
        for k, (al, be) in self.TWO.items():
            x, y = _rate(vm, *al), _rate(vm, *be)
            g[k] = _cn(g[k], x / (x + y), 1 / (x + y), dt)
        inf, tau = self._others(vm, caq)
        for k in inf:
            g[k] = _cn(g[k], inf[k], tau[k], dt)
        return dict(g=g, ca=ca, rev=rev, v=v_new)

    def take(self, new, mask=None):
        if mask is not None:
            new = dict(new, g={k: torch.where(mask, x, self.g[k]) for k, x in new["g"].items()},
                       **{k: torch.where(mask, new[k], getattr(self, k)) for k in ("ca", "rev", "v")})
        self.__dict__.update(new)

    def sums(self):
        """conductance and conductance-weighted reversal of the present gates"""
        g, c = self.g, self.c
        ca = c[2] * g["mCaP"] * g["hCaP"] + c[3] * g["mCaT"] * g["hCaT"]
        na = c[0] * g["mNaF"] ** 3 * g["hNaF"] + c[1] * g["mNaP"] ** 3
        kh = c[4] * (g["mKh1"] + g["mKh2"])
        k = (c[5] * g["mKdr"] ** 2 * g["hKdr"] + c[6] * g["mKM"] + c[7] * g["mKA"] ** 4 * g["hKA"]
             + c[8] * g["mKC"] * g["zKC"] ** 2 + c[9] * g["mK2"] * g["zK2"] ** 2)
        return (self.leak + na + ca + kh + k,
                self.leak * -80.0 + na * 45.0 + ca * self.rev + kh * -30.0 + k * -85.0)

    def current(self, v):
        gs, es = self.sums()
        b = gs * v - es - self.iext
        return b if self.syn is None else b + self.syn * v

    def gap(self, v):
        return torch.zeros_like(v)

    def floor(self):
        """1.2 x the largest eigenvalue of the cable operator of every cell, by Lanczos"""
        s = 1 / torch.sqrt(self.cm)
        shape = (self.n, self.comp)
        q = torch.randn(shape, dtype=torch.float64, device=self.dev)
        q /= q.norm(dim=1, keepdim=True)
        Q, al, be = [q], [], []
        for k in range(80):
            w = -(self.cable.lap((Q[-1].reshape(-1) * s)) * s).view(shape)
            al.append((w * Q[-1]).sum(1))
            B = torch.stack(Q, 1)
            for _ in range(2):
                w = w - torch.bmm(torch.bmm(w[:, None], B.transpose(1, 2).contiguous()), B)[:, 0]
            be.append(w.norm(dim=1))
            Q.append(w / be[-1][:, None])
        T = torch.diag_embed(torch.stack(al, 1)) + torch.diag_embed(torch.stack(be[:-1], 1), 1)
        T = T + torch.diag_embed(torch.stack(be[:-1], 1), -1)
        return 1.2 * torch.linalg.eigvalsh(T.cpu())[:, -1].numpy()


class _Olive:
    HMIN, STRICT = 2.0 ** -10, True

    def __init__(self, case, v0, amp, dev, seed):
        n = len(v0)
        self.n, self.comp, self.dev = n, 3, dev
        t = lambda x: torch.tensor(x, device=dev, dtype=torch.float64)  # noqa: E731
        one = np.loadtxt(os.path.join(DATA, "IO.txt"))
        self.cm = t(np.tile(one[:, 4], n))
        gi = 0.13
        i = np.array([0, 1, 1, 2])
        j = np.array([1, 0, 2, 1])
        w = np.array([gi / 0.8, gi / 0.2, gi / 0.869, gi / (1 - 0.869)])
        cell = np.repeat(np.arange(n) * 3, 4)
        self.cable = _Cable(3 * n, cell + np.tile(i, n), cell + np.tile(j, n), np.tile(w, n), dev)
        rep = lambda d, s, a: t(np.tile([d, s, a], n))  # noqa: E731
        self.c = dict(CaL=rep(0, 0.83, 0), Na=rep(0, 120.0, 240.0), Kdr=rep(0, 9.0, 0), K=rep(0, 5.0, 20.0),
                      CaH=rep(4.5, 0, 0), KCa=rep(35.0, 0, 0), H=rep(0.15, 0, 0))
        self.kind = torch.arange(3 * n, device=dev) % 3
        self.v = t(np.repeat(v0, 3))
        self.iext = torch.zeros_like(self.v)
        # partners left, up, right, down; the grid row is id / ny, as the reference has it
        nx, ny = case["nx"], case["ny"]
        nbr = np.full((n, 4), -1)
        for k in range(n if n > 1 else 0):
            x, y = k % nx, k // ny
            corner = (x in (0, nx - 1)) and (y in (0, ny - 1))
            has = [True] * 4
            if corner:
                has = [x != 0, y != 0, x == 0, y == 0]
            elif y == 0:
                has[1] = False
            elif y == ny - 1:
                has[3] = False
            elif x == 0:
                has[0] = False
            elif x == nx - 1:
                has[2] = False
            for s, q in enumerate((k - 1, k - nx, k + 1, k + nx)):
                if has[s] and 0 <= q < n:
                    nbr[k, s] = q
        self.has = t(nbr >= 0)
        self.nbr = torch.tensor(np.maximum(nbr, 0), device=dev)
        v, inf = self.v, self._inf(self.v)
        self.g = {k: inf[k][0] for k in ("k", "l", "m", "h", "n", "p", "x", "r", "q")}
        self.ca = -self.c["CaH"] * self.g["r"] ** 2 * (v - 120.0) * 3.0 / 0.075
        self.g["s"] = self._s(self.ca)[0]

    def interval(self, k):
        pass

    @staticmethod
    def _s(ca):
        a = torch.clamp(0.00002 * ca, max=0.01)
        return a / (a + 0.015), 1 / (a + 0.015)

    def _inf(self, v):
        e = torch.exp
        sig = lambda x: 1 / (1 + e(x))  # noqa: E731
        h = torch.where(self.kind == 1, sig((-v - 70) / -5.8), torch.where(self.kind == 2, sig((-v - 60) / -5.8), 1.0))
        th = torch.where(self.kind == 1, 3 * e((-v - 40) / 33), torch.where(self.kind == 2, 1.5 * e((-v - 40) / 33), 1.0))
        tn = 47 * e((v + 50) / 900) + 5
        ar, br = 1.7 / (1 + e(-(v - 5) / 13.9)), 0.02 * (v + 8.5) / (e((v + 8.5) / 5) - 1)
        ax, bx = 0.13 * (v + 25) / (1 - e(-(v + 25) / 10)), 1.69 * e(-0.0125 * (v + 35))
        return dict(k=(sig((-v - 61) / 4.2), 1.0), l=(sig((v + 85.5) / 8.5), 20 * e((v + 160) / 30) / (1 + e((v + 84) / 7.3)) + 35),
                    m=(sig((-v - 30) / 5.5), None), h=(h, th), n=(sig((-v - 3) / 10), tn), p=(sig((-v - 51) / -12), tn),
                    x=(ax / (ax + bx), 1 / (ax + bx)), r=(ar / (ar + br), 5 / (ar + br)),
                    q=(sig((v + 80) / 4), 1 / (e(-0.086 * v - 14.6) + e(0.07 * v - 1.87))))

    def ion(self, v_new, dt, extrapolate=False):
        g = dict(self.g)
        v_ca = v_new if extrapolate else self.v
        vm = 1.5 * v_new - 0.5 * self.vold if extrapolate else 0.5 * (v_new + self.v)
        i_ca = self.c["CaH"] * g["r"] ** 2 * (v_ca - 120.0)
        f = lambda ca: dt * (-3.0 * i_ca - 0.075 * ca)  # noqa: E731
        k1 = f(self.ca)
        k2 = f(self.ca + k1 / 2)
        k3 = f(self.ca + k2 / 2)
        ca = self.ca + (k1 + 2 * k2 + 2 * k3 + f(self.ca + k3)) / 6
        inf = self._inf(vm)
        inf["s"] = self._s((self.ca + ca) / 2)
        for k, (x, tau) in inf.items():
            g[k] = x if tau is None else _cn(g[k], x, tau, dt)
        return dict(g=g, ca=ca, v=v_new)

    def take(self, new, mask=None):
        self.__dict__.update(new)

    def sums(self):
        g, c = self.g, self.c
        cal, cah = c["CaL"] * g["k"] ** 3 * g["l"], c["CaH"] * g["r"] ** 2
        na, h = c["Na"] * g["m"] ** 3 * g["h"], c["H"] * g["q"]
        k = c["Kdr"] * g["n"] * g["p"] + c["K"] * g["x"] ** 4 + c["KCa"] * g["s"]
        return 0.016 + cal + cah + na + h + k, 0.016 * 10.0 + (cal + cah) * 120.0 + na * 55.0 + h * -43.0 + k * -75.0

    def current(self, v):
        gs, es = self.sums()
        return gs * v - es - self.iext

    def gap(self, v):
        """the gap currents into the dendrites"""
        out = torch.zeros_like(v)
        d = v.view(self.n, 3)[:, 0]
        diff = (d[:, None] - d[self.nbr]) * self.has
        out.view(self.n, 3)[:, 0] = (0.04 * (0.8 * torch.exp(-0.01 * diff * diff) + 0.2) * diff).sum(1)
        return out


def _philox_uniform(i, step, seed):
    """53-bit uniforms of Philox4x32-10 at counters (i, step, 0x5359, 0)"""
    M = np.uint64(0xFFFFFFFF)
    c = [i.astype(np.uint64), np.full(len(i), step, np.uint64), np.full(len(i), 0x5359, np.uint64), np.zeros(len(i), np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32 & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        s = np.uint64(32)
        c = [(p1 >> s) ^ c[1] ^ np.uint64(k0), p1 & M, (p0 >> s) ^ c[3] ^ np.uint64(k1), p0 & M]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return ((c[0] >> np.uint64(5)).astype(float) * 67108864.0 + (c[1] >> np.uint64(6)).astype(float)) / 9007199254740992.0


def _stages(m):
    """the Chebyshev stage coefficients: mu~_1 and (mu, nu, mu~, a) of stages 2 .. m"""
    w0 = 1 + 2 / (13 * m * m)
    t1 = w0 * w0 - 1
    t2 = math.sqrt(t1)
    arg = m * math.log(w0 + t2)
    w1 = math.sinh(arg) * t1 / (math.cosh(arg) * m * t2 - w0 * math.sinh(arg))
    T, dT, d2T = [1.0, w0], [0.0, 1.0], [0.0, 0.0]
    for j in range(2, m + 1):
        T.append(2 * w0 * T[-1] - T[-2])
        dT.append(2 * w0 * dT[-1] - dT[-2] + 2 * T[j - 1])
        d2T.append(2 * w0 * d2T[-1] - d2T[-2] + 4 * dT[j - 1])
    b = [0.0, 0.0] + [d2T[j] / dT[j] ** 2 for j in range(2, m + 1)]
    b[0] = b[1] = b[2] if m >= 2 else 0.0
    out = []
    for j in range(2, m + 1):
        mu = 2 * w0 * b[j] / b[j - 1]
        out.append((mu, -b[j] / b[j - 2], mu * w1 / w0, 1 - T[j - 1] * b[j - 1]))
    return w1 * b[1], out


class _Rkc:
    """The adaptive Runge-Kutta-Chebyshev path with one controller per group of compartments (one group:
    the whole population).  Groups advance in lock step, each on its own step size."""

    def __init__(self, m, groups, case):
        self.m, self.G = m, groups
        kw = _tolerances(case)
        self.at, self.rt = kw.get("atol", 1e-6), kw.get("rtol", 1e-6)
        self.integ = kw.get("ion_interval", 2.0 ** math.log10(self.at))
        self.refresh = kw.get("refresh_fn", False)
        self.floor = np.zeros(groups)
        if kw.get("rho_floor"):
            f = m.floor()
            self.floor = f if groups > 1 or len(f) == 1 else np.array([f.max()])
        G = groups
        self.y = m.v.clone()
        self.vy = m.v.clone()
        self.b = m.current(m.v)
        self.fn = self.F(self.y)
        self.ede = self.fn.clone()
        self.rho = np.zeros(G)
        self._power(np.ones(G, bool))
        h = np.maximum(np.where(self.rho * H > 1, 1 / self.rho, H), m.HMIN)
        d = (self.F(self.y + self.col(h) * self.fn) - self.fn) / (self.at + self.rt * self.y.abs())
        est = h * np.sqrt(self.sq(d) / (len(self.y) / G))
        self.h = np.where(0.1 * h < H * np.sqrt(est), np.maximum(0.1 * h / np.sqrt(est), m.HMIN), H)
        self.mmax = int(round(math.sqrt(self.rt / (10 * 2.22e-16))))
        self.t, self.end, self.sum_dt = np.zeros(G), H, np.zeros(G)
        self.new, self.jac = np.ones(G, bool), np.zeros(G, bool)
        self.acc, self.err0, self.h0 = np.zeros(G), np.zeros(G), np.zeros(G)

    def col(self, x):
        """one value per group, spread over its compartments"""
        if self.G == 1:
            return float(x[0])
        return torch.tensor(x, device=self.y.device).repeat_interleave(len(self.y) // self.G)

    def mask(self, x):
        return None if self.G == 1 else self.col(x)

    def pick(self, x, a, b):
        if self.G == 1:
            return a if x[0] else b
        return torch.where(self.col(x), a, b)

    def sq(self, x):
        return (x * x).view(self.G, -1).sum(1).cpu().numpy()

    def F(self, y):
        return (self.m.cable.lap(y) - self.b) / self.m.cm

    def _power(self, todo):
        """the nonlinear power method's spectral radius for the groups of todo"""
        yn, vn = np.sqrt(self.sq(self.y)), np.sqrt(self.sq(self.ede))
        dy = yn * math.sqrt(2.22e-16)
        v = self.y + self.col(dy / vn) * self.ede
        live, sigma = todo.copy(), np.zeros(self.G)
        for k in range(1000):
            f = self.F(v) - self.fn
            df = np.sqrt(self.sq(f))
            old, sigma = sigma, np.where(live, df / dy, sigma)
            self.rho = np.where(live, 1.2 * sigma, self.rho)
            done = live & (np.abs(sigma - old) <= np.maximum(sigma, 8.0) * 0.001) if k else np.zeros(self.G, bool)
            if done.any():
                self.ede = self.pick(done, v - self.y, self.ede)
            live = live & ~done
            if not live.any():
                break
            v = self.pick(live, self.y + self.col(dy / df) * f, v)
        self.rho = np.maximum(self.rho, self.floor)

    def _ion(self, groups):
        if not groups.any():
            return
        m, mask = self.m, self.mask(groups)
        new = m.ion(self.vy, self.col(np.where(groups, self.sum_dt, H)))
        m.take(new, mask)
        b = m.current(self.vy) + m.gap(self.vy)
        self.b = b if mask is None else torch.where(mask, b, self.b)
        if self.refresh:
            self.fn = self.pick(groups, self.F(self.y), self.fn)
        self.sum_dt = np.where(groups, 0.0, self.sum_dt)

    def advance(self):
        self._ion(self.sum_dt != 0)
        live = np.ones(self.G, bool)
        while live.any():
            if (live & self.new).any():
                self._power(live & self.new)
                self.jac |= live & self.new
            last = 1.1 * self.h >= np.abs(self.end - self.t)
            self.h = np.where(live & last, np.abs(self.end - self.t), self.h)
            ms = 1 + np.sqrt(1.54 * self.h * self.rho + 1).astype(int)
            over = live & (ms > self.mmax)
            self.h = np.where(over, (self.mmax ** 2 - 1) / (1.54 * self.rho), self.h)
            ms, last = np.minimum(ms, self.mmax), last & ~over
            h = np.maximum(self.h, self.m.HMIN)
            d1, d0 = self._step(h, ms, live)
            f = self.F(self.y + d1)
            wt = self.at + self.rt * torch.maximum((self.y + d1).abs(), self.y.abs())
            est = (-0.8 * d1 + 0.4 * self.col(h) * (self.fn + f)) / wt
            err = np.sqrt(self.sq(est) / (len(self.y) / self.G))
            bad = live & (err > 1)
            cut = np.where(bad, 0.8 * self.h / np.maximum(err, 1e-300) ** (1 / 3), self.h)
            again = bad & (cut >= self.m.HMIN)
            self.h = cut
            self.new = np.where(again, ~self.jac, self.new)
            ok = live & ~again
            if not ok.any():
                continue
            self.acc += ok
            self.t += np.where(ok, h, 0)
            self.jac &= ~ok
            self.new &= ~ok
            self.vy = self.pick(ok, self.y + d0, self.vy)
            self.y, self.fn = self.pick(ok, self.y + d1, self.y), self.pick(ok, f, self.fn)
            with np.errstate(divide="ignore", invalid="ignore"):
                e3 = err ** (1 / 3)
                fac = np.where(self.acc == 1, np.where(0.8 < 10 * e3, 0.8 / e3, 10.0),
                               np.fmin(10.0, 0.8 * self.h * self.err0 ** (1 / 3) / (self.h0 * err ** (2 / 3))))
            nh = np.maximum(self.m.HMIN, np.minimum(H, np.maximum(0.1, fac) * self.h))
            self.h = np.where(ok, nh, self.h)
            self.err0, self.h0 = np.where(ok, err, self.err0), np.where(ok, h, self.h0)
            self.sum_dt += np.where(ok, h, 0)
            due = self.sum_dt > self.integ if self.m.STRICT else self.sum_dt >= self.integ
            live = live & ~(ok & last)
            self._ion(ok & due & ~last)
        self.end += H
        self.v_out = self.y
        return self.v_out

    def _step(self, h, ms, live):
        """D_m and D_{m-2} of the stage recurrence on increments D_j = Y_j - Y_0"""
        tab = {int(m): _stages(int(m)) for m in set(ms[live])}
        top = max(tab)
        a = self.F(self.y)
        per = lambda f: self.col(np.array([f(tab[int(m)], int(m)) if g else 0.0 for m, g in zip(ms, live)]))  # noqa: E731
        hc = self.col(h)
        prev, cur = torch.zeros_like(self.y), hc * per(lambda s, m: s[0]) * self.fn
        out0 = prev
        lap = lambda x: self.m.cable.lap(x) / self.m.cm  # noqa: E731
        for j in range(top - 1):
            mu, nu, mut, aj = (per(lambda s, m, q=q: s[1][j][q] if j < m - 1 else 0.0) for q in range(4))
            nxt = mu * cur + nu * prev + hc * mut * (a + lap(cur) - aj * self.fn)
            on = live & (j < ms - 1)
            out0 = self.pick(live & (j == ms - 2), prev, out0)
            prev, cur = self.pick(on, cur, prev), self.pick(on, nxt, cur)
        return cur, out0


class _Cn:
    """Crank-Nicolson steps of 0.025 ms: the reference's CG, the exact tree solve, or (olive cells, where
    the reference's BiCG converges) an exact solve per cell"""

    def __init__(self, m, case):
        self.m, self.case = m, case
        m.vold = m.v.clone()
        gs, es = m.sums()
        self.g1, self.o1 = gs / 2, es / 2   # the injected current starts at zero

    def advance(self):
        m, dt = self.m, 0.025
        for _ in range(5):
            v = m.v
            new = m.ion(v, dt, extrapolate=True)
            m.take(new)
            m.vold = v
            gs, es = m.sums()
            g2, o2 = gs / 2, (es + m.iext) / 2 - m.gap(v)
            c = m.cm / dt
            rhs = 0.5 * m.cable.lap(v) + (c - self.g1) * v + self.o1 + o2
            self.g1, self.o1 = g2, o2
            diag = c + g2 + 0.5 * m.cable.gsum
            m.v = self._solve(diag, rhs)
        self.v_out = m.v
        return m.v

    def _apply(self, diag, x):
        return diag * x - 0.5 * (self.m.cable.w * x[self.m.cable.nb]).sum(0)

    def _solve(self, diag, b):
        m = self.m
        if m.comp == 3:
            A = torch.diag_embed(diag.view(-1, 3))
            w, nb = 0.5 * m.cable.w, m.cable.nb
            i = torch.arange(len(b), device=b.device).expand_as(nb)
            A.view(-1).index_add_(0, (i // 3 * 9 + i % 3 * 3 + nb % 3).reshape(-1), -w.reshape(-1))
            return torch.linalg.solve(A, b.view(-1, 3, 1)).view(-1)
        if self.case["engine"] == "tree":
            return self._tree(diag, b)
        x = torch.zeros_like(b)
        r, p = b, b
        rr = first = r @ r
        for _ in range(100):
            ap = self._apply(diag, p)
            alpha = rr / (p @ ap)
            x, r = x + alpha * p, r - alpha * ap
            rr, old = r @ r, rr
            if math.sqrt(rr) <= 1e-15 * math.sqrt(first):
                break
            p = r + rr / old * p
        return x

    def _tree(self, diag, b):
        m = self.m
        par, g = m.parent[0], 0.5 * m.g_parent.reshape(m.n, -1)[0]
        depth = np.zeros(len(par), int)
        for i in range(len(par)):
            k = i
            while par[k] >= 0:
                k, depth[i] = par[k], depth[i] + 1
        order = np.argsort(-depth, kind="stable")
        d, r = diag.view(m.n, -1).T.cpu().numpy().copy(), b.view(m.n, -1).T.cpu().numpy().copy()
        for i in order[:-1]:
            f = g[i] / d[i]
            d[par[i]] -= f * g[i]
            r[par[i]] += f * r[i]
        r[order[-1]] /= d[order[-1]]
        for i in order[-2::-1]:
            r[i] = (r[i] + g[i] * r[par[i]]) / d[i]
        return torch.tensor(np.ascontiguousarray(r.T).reshape(-1), device=b.device)
