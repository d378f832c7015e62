"""The two paths of the population-global engines against each other
(cb_pop_launch_path): the resident kernels (csrc/rkc_resident.hpp,
csrc/kry_resident.hpp) and the kernel launches per Chebyshev stage and Krylov
iteration that larger populations take, and any population in a process that
may not launch cooperatively.  Every voltage, current, gate, controller value,
counter, recording and spike is the same bits, with ion updates, stimulus,
gap junctions, Poisson drive and synapses; so the small populations here, and
with them the oracle's tests of either path, cover both."""
import os
import subprocess
import sys

import numpy as np
import pytest

import cbrkc
import test_gpu_net as TN

pytestmark = pytest.mark.gpu

KIND = {"pkj": (cbrkc.PKJ, "Pkj.txt", -67.0, 18), "io": (cbrkc.IO, "IO.txt", -60.0, 10),
        "go": (cbrkc.GO, "Go_131.txt", -60.0, 24), "gr": (cbrkc.GR, "Gr.txt", -70.0, 24)}
T0 = 600.0   # inside the reference's stimulus windows
FIELDS = (cbrkc.F_VNEW, cbrkc.F_V, cbrkc.F_CA, cbrkc.F_B, cbrkc.F_IEXT)


def population(ref_data, cell, nx, ny, **kw):
    kind, f, v, _ = KIND[cell.split()[0]]
    gj = os.path.join(ref_data, "Pkj_GJ.csv") if cell == "pkj gj" else ""
    v0 = v + 0.05 * (np.arange(nx * ny) % 31)
    return cbrkc.Population(kind, nx, ny, morph=os.path.join(ref_data, f), gj=gj, v0=v0, **kw)


def make(ref_data, cell, nx, ny, **kw):
    pops = [population(ref_data, cell, nx, ny, **kw) for _ in range(2)]
    pops[1].launch_path()
    assert "workgroups" in pops[0].mapping() and "workgroups" not in pops[1].mapping(), [p.mapping() for p in pops]
    return pops


def same(a, b, fields):
    for f in fields:
        try:
            x = a.read(f)
        except cbrkc.CbError:
            continue
        assert np.array_equal(x, b.read(f)), f
    assert a.stats() == b.stats()


@pytest.mark.parametrize("cell,nx,ny,kw", [
    ("io", 2, 2, {}), ("io", 13, 40, {}), ("go", 1, 1, {}), ("go", 5, 3, {}), ("gr", 1, 1, {}), ("gr", 3, 1, {}),
    ("pkj", 1, 1, {}), ("pkj", 3, 1, {}), ("pkj gj", 2, 2, {}),
    ("pkj", 2, 1, dict(atol=1e-6, rtol=1e-4, **cbrkc.STABLE)),
    ("pkj", 2, 1, dict(poisson=dict(rate_hz=2000.0, g_mS=1e-6, tau_ms=2.0, e_mV=0.0, seed=3)))])
def test_rkc(ref_data, cell, nx, ny, kw):
    print(f"{cell} {nx}x{ny} {kw}", flush=True)
    a, b = make(ref_data, cell, nx, ny, **kw)
    out = []
    for p in (a, b):
        p.set_raster(0, -60.0)
        out.append([p.run(3, T0, 0), p.run(2, T0 + 0.375, -1)])
        p.set_current(T0 + 0.625)
        p.advance()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
    for x, y in zip(a.spikes(), b.spikes()):
        assert np.array_equal(x, y)
    same(a, b, FIELDS + (cbrkc.F_Y, cbrkc.F_YN, cbrkc.F_FN) + tuple(cbrkc.F_GATE0 + k for k in range(KIND[cell.split()[0]][3])))
    for x, y in zip(a.controller(), b.controller()):
        assert np.array_equal(x, y)
    with pytest.raises(cbrkc.CbError):
        a.launch_path()   # too late


@pytest.mark.parametrize("solver", [cbrkc.CN, cbrkc.BE], ids=["cn", "be"])
@pytest.mark.parametrize("cell,nx,ny", [("pkj", 1, 1), ("pkj", 3, 1), ("pkj gj", 3, 2), ("gr", 2, 4), ("go", 2, 2),
                                        ("go", 7, 7), ("io", 1, 1), ("io", 9, 9), ("io", 40, 24)])
def test_krylov(ref_data, cell, nx, ny, solver):
    print(f"{cell} {nx}x{ny} solver {solver}", flush=True)
    a, b = make(ref_data, cell, nx, ny, solver=solver)
    assert np.array_equal(a.run(2, T0, 0), b.run(2, T0, 0))
    b.launch_path(False)   # this engine may change its path at any time
    a.launch_path()
    assert np.array_equal(a.run(1, T0 + 0.25, -1), b.run(1, T0 + 0.25, -1))
    same(a, b, FIELDS)


def test_network(ref_data, tmp_path):
    # populations with their synapses: mossy fibres at a rate that
    # makes granule cells fire, 3 ms
    n = (64, 16, 3)
    files = [str(tmp_path / f) for f in ("gr.txt", "go.txt", "pkj.txt")]
    cbrkc.synth_gr_chains(files[0], os.path.join(ref_data, "Gr.txt"), 7, n[0])
    cbrkc.synth_go_trees(files[1], os.path.join(ref_data, "Go_131.txt"), 8, n[1])
    cbrkc.synth_pkj_morph(files[2], seed=9, ncell=n[2])
    v0 = TN.v0_of(n)
    pops, nets = [], []
    for launches in (False, True):
        p = TN.gpu_pops(files, v0)
        for x in p:
            if launches:
                x.launch_path()
        pops.append(p)
        nets.append(cbrkc.Network(*p, cfg=cbrkc.net_config(seed=4, total=0, mf_rate_hz=200.0)))
    for k in range(24):
        print("interval", k, flush=True)
        for net in nets:
            net.run(1)
        for x, y, name in zip(*pops, ("gr", "go", "pkj")):
            assert x.stats() == y.stats(), name
            same(x, y, FIELDS + (cbrkc.F_Y, cbrkc.F_YN, cbrkc.F_FN))
    for pop in (cbrkc.NET_GR, cbrkc.NET_GO, cbrkc.NET_PKJ):
        g = [net.conductance(pop, cbrkc.NET_AMPA) for net in nets]
        assert np.array_equal(*g) and g[0].any()


CHILD = """
import sys
sys.path[:0] = sys.argv[1:3]
import numpy as np
import cbrkc
import test_gpu_paths as T
out = {}
for name, cell, nx, ny, kw in T.ELSEWHERE:
    p = T.population(sys.argv[3], cell, nx, ny, **kw)
    print(name, p.mapping(), flush=True)
    out[name] = np.concatenate([p.run(2, T.T0, -1).ravel(), p.read(cbrkc.F_B)])
np.savez(sys.argv[4], **out)
"""
ELSEWHERE = [("io", "io", 13, 40, {}), ("gr", "gr", 1, 1, {}), ("pkj cn", "pkj", 4, 1, dict(solver=cbrkc.CN))]


def test_a_second_process(ref_data, tmp_path):
    # This process has launched cooperatively and keeps the barrier resource to its
    # end; another one that is refused it takes the other path, with the same results
    here, out = {}, str(tmp_path / "out.npz")
    for name, cell, nx, ny, kw in ELSEWHERE:
        p = population(ref_data, cell, nx, ny, **kw)
        here[name] = np.concatenate([p.run(2, T0, -1).ravel(), p.read(cbrkc.F_B)])
    r = subprocess.run([sys.executable, "-c", CHILD, os.path.dirname(cbrkc.__file__), os.path.dirname(__file__), ref_data,
                        out], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    there = np.load(out)
    for name in here:
        assert np.array_equal(here[name], there[name]), name
