"""The resident RKC kernel (csrc/rkc_resident.hpp) built for the host from the
same source (tests/host_emu/resident_emu.cpp, one host thread per lane), on
cable matrices with constant frozen currents, against the oracle: voltages,
derivative, power-method vector, controller and counters bit for bit.  Here are
the branches that no morphology reaches at will."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def emu(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    out = tmp_path_factory.mktemp("resident_emu")
    subprocess.run(["bash", os.path.join(ROOT, "tests", "host_emu", "build_resident.sh"), str(out)], check=True)
    return ctypes.CDLL(str(out / "libresident.so"))


def run(emu, o, n, cpb=1, nsteps=1, nhelp=0, present=1 << 20, floor=0.0, refresh=False, wait=1 << 60):
    """nsteps macro steps of the oracle population o, as n cells, on the host
    build, from o's present state, with this floor of the spectral radius and
    refresh of fn after ion updates; o itself stays"""
    orc.lib().or_pop_set_rho_floor(o.h, floor)
    orc.lib().or_pop_set_refresh_fn(o.h, 1 if refresh else 0)
    comp = o.nc // n
    row, col, val = o.csr()
    keep = [np.ascontiguousarray(x, dtype=np.float64) for x in (val, o.get(orc.CM), o.get(orc.B))]
    vec = np.stack([o.get(k) for k in (orc.Y, orc.YN, orc.FN, orc.EDE, orc.VNEW)])
    c, hw = np.zeros(16), np.zeros(8)
    c[:14], hw[:] = o.controller()[0], o.controller()[1]
    cnt = np.array([o.stats()[k] for k in ("steps", "rejects", "stages", "rho_iters", "ion_updates")], dtype=np.int64)
    launches, polls = ctypes.c_int(), ctypes.c_longlong()
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    status = emu.emu_rkc(n, comp, cpb, nhelp, present, p(row), p(col), p(keep[0]), p(keep[1]), p(keep[2]), p(vec), p(c),
                         p(hw), p(cnt), nsteps, ctypes.c_double(floor), 1 if refresh else 0, ctypes.c_longlong(wait),
                         ctypes.byref(launches), ctypes.byref(polls))
    return dict(status=status, vec=vec, ctl=c[:14], hw=hw, cnt=cnt, launches=launches.value, polls=polls.value)


def check(o, r, nsteps=1):
    for _ in range(nsteps):
        o.advance()
    assert r["status"] == 0
    for k, f in enumerate((orc.Y, orc.YN, orc.FN, orc.EDE, orc.VNEW)):
        assert np.array_equal(r["vec"][k], o.get(f)), k
    assert np.array_equal(r["ctl"], o.controller()[0])
    assert np.array_equal(r["hw"], o.controller()[1])
    s = o.stats()
    assert list(r["cnt"][:4]) == [s[k] for k in ("steps", "rejects", "stages", "rho_iters")]


def cables(n, comp, g, seed=0, pairs=(), spread=1.0):
    """n chains of comp rows, their conductances about g, joined at pairs of rows; currents and voltages spread so far"""
    rng = np.random.default_rng(seed)
    L = np.zeros((n * comp, n * comp))
    for i in range(n * comp - 1):
        if (i + 1) % comp:
            L[i, i + 1] = L[i + 1, i] = g * rng.uniform(0.5, 1.5)
    for i, j in pairs:
        L[i, j] = L[j, i] = 0.3 * g
    return orc.Pop.generic(L, rng.uniform(0.8, 1.2, n * comp), spread * rng.uniform(-3.0, 3.0, n * comp),
                           -65.0 + spread * rng.uniform(-5.0, 5.0, n * comp))


@pytest.mark.parametrize("n,comp,cpb,nhelp", [(1, 40, 1, 0), (1, 150, 1, 2), (3, 20, 2, 0)])
def test_macro_steps(emu, n, comp, cpb, nhelp):
    o = cables(n, comp, 5.0)
    check(o, run(emu, o, n, cpb, nsteps=3, nhelp=nhelp), 3)


def test_coupled_workgroups(emu):
    o = cables(2, 30, 5.0, pairs=[(3, 41), (29, 30), (3, 55)])
    check(o, run(emu, o, 2, nsteps=2), 2)


@pytest.mark.parametrize("n,comp,nhelp,pairs", [(2, 30, 0, ()), (2, 30, 0, [(3, 41), (29, 30)]), (3, 30, 0, [(29, 30), (59, 60)]),
                                                (1, 150, 2, ())])
def test_a_lost_workgroup_ends_the_launch(emu, n, comp, nhelp, pairs):
    # Only the first workgroup runs (or, of three, the first two): it gives up
    # once, not at every one of a step's 140 exchanges, and says so
    o = cables(n, comp, 0.5, pairs=pairs, spread=1e-3)
    wait = 20000   # looks at mailboxes, a lane's clock on the host
    r = run(emu, o, n, nhelp=nhelp, present=max(1, n - 1), floor=2e5, wait=wait, nsteps=2)
    assert r["status"] == 8
    # two limits, and 128 looks at each of the step's other exchanges; not a limit at each
    assert r["polls"] < 2 * wait + 1000 + 200 * 128 < 10 * wait
    # no waiting at all: the first look that finds nothing
    assert run(emu, o, n, nhelp=nhelp, present=max(1, n - 1), floor=2e5, wait=0,
               nsteps=2)["status"] == 8


@pytest.mark.parametrize("pairs,refresh", [((), False), ([(3, 41), (29, 30)], True)])
@pytest.mark.parametrize("floor,m", [(2e5, 137), (6e8, 4097)])
def test_many_stages(emu, floor, m, pairs, refresh):
    # a spectral radius far above the cable's, as the power method gives it when
    # synaptic input sets in: steps past the coefficient table and the coupled
    # values' slots, and of more stages than RES_START, which the host is asked for
    o = cables(2, 30, 0.5, pairs=pairs, spread=1e-3)
    before = o.stats()
    k = 1 if m > 4096 else 3
    r = run(emu, o, 2, nsteps=k, floor=floor, refresh=refresh)
    check(o, r, k)
    s = o.stats()
    assert s["stages"] - before["stages"] > m * (s["steps"] + s["rejects"] - before["steps"] - before["rejects"])
    assert m < 4096 or r["launches"] >= 3 - refresh


def test_power_method_when_the_perturbation_moves_nothing(emu):
    # A uniform state perturbed uniformly: F does not move, and the method turns
    # one element's perturbation round about y_n (rand_elements_change,
    # solve_rkc.cu:22-27), whatever the stage vector holds, as after a rejected
    # step.  Of two equal rows that is the dominant eigenvector itself, found in
    # three iterations.
    o = orc.Pop.generic(np.array([[0.0, 5.0], [5.0, 0.0]]), np.ones(2), np.array([1.0, -2.0]), np.array([-66.0, -64.0]))
    before = o.stats()["rho_iters"]
    o.set(orc.YN, np.full(2, -65.0))
    o.set(orc.FN, o.dydt(np.full(2, -65.0)))
    o.set(orc.EDE, np.full(2, 0.5))
    o.set(orc.Y, np.array([-80.0, -50.0]))
    r = run(emu, o, 1)
    check(o, r)
    assert r["cnt"][3] - before == 3
