"""The resident CG / BiCG kernel (csrc/kry_resident.hpp) at the edges of its
shapes, against the oracle over one output interval (five solves): one
workgroup, several with rows of one cell on either side of their border (1600
and 578 rows in 512-row workgroups), gap junctions across workgroups, the
unsymmetric olive system in one and in several workgroups, a last workgroup
of one chunk; and a population of each shape's threads x rows.  The products
and sums are the oracle's in its order, so the difference is that of exp in
the ion updates (1e-9 mV, the bar of the other CN tests; the truncated BE
iterates move by up to 2e-4 mV under one ulp of the input,
test_oracle_be.py::test_truncated_cg_noise_floor), and the iteration counts
are equal.  (That the iterates are those of the launches per iteration bit for
bit is tested in test_gpu_paths.py.)"""
import os

import numpy as np
import pytest

import cbrkc
import orc
from test_oracle_be import L as LB
from test_oracle_cn import L as LC
from test_oracle_gr import gr_pop
from test_oracle_go import go_pop
from test_oracle_io import io_pop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [cbrkc.CN, cbrkc.BE], ids=["cn", "be"])
@pytest.mark.parametrize("cell,nx,ny,grid", [("pkj", 1, 1, 1), ("pkj", 3, 1, 10), ("pkj gj", 3, 2, 19),
                                              ("gr", 2, 4, 10), ("go", 2, 2, 1), ("go", 7, 7, 13),
                                              ("io", 1, 1, 1), ("io", 9, 9, 1), ("io", 40, 24, 6)])
def test_one_interval(ref_data, solver, cell, nx, ny, grid):
    print(f"{cell} {nx}x{ny}, solver {solver}", flush=True)
    n = nx * ny
    v0 = {"pkj": -66.0, "pkj gj": -66.0, "gr": -70.0, "go": -60.0, "io": -60.0}[cell] + 0.05 * (np.arange(n) % 31)
    if cell.startswith("pkj"):
        gj = os.path.join(ref_data, "Pkj_GJ.csv") if cell == "pkj gj" else ""
        morph = os.path.join(ref_data, "Pkj.txt")
        o = orc.Pop.pkj(morph, nx, ny, v0=v0, libc_rand=False, gj=gj or None)
        p = cbrkc.Population(cbrkc.PKJ, nx, ny, solver=solver, morph=morph, gj=gj, v0=v0)
    else:
        make, kind, f = {"gr": (gr_pop, cbrkc.GR, "Gr.txt"), "go": (go_pop, cbrkc.GO, "Go_131.txt"),
                         "io": (io_pop, cbrkc.IO, "IO.txt")}[cell]
        o = make(ref_data, nx, ny, v0=v0)
        p = cbrkc.Population(kind, nx, ny, solver=solver, morph=os.path.join(ref_data, f), v0=v0)
    assert f", {grid} workgroups" in p.mapping(), p.mapping()
    lib, name = (LC(), "cn") if solver == cbrkc.CN else (LB(), "be")
    assert getattr(lib, f"or_{name}_init")(o.h) == 0
    getattr(lib, f"or_{name}_advance")(o.h, 0.0)
    p.run(1, 0.0, 0)
    d = np.abs(p.read(cbrkc.F_V) - o.get(orc.V)).max()
    print("max |GPU - oracle|", d, p.stats(), flush=True)
    assert d <= (1e-9 if solver == cbrkc.CN or cell in ("io", "go") else 1e-3)
    assert p.stats()["stages"] == o.stats()["stages"]
    if cell != "io":
        # trees at these steps never reach 1e-15: 100 iterations each
        assert cell == "go" or p.stats()["stages"] == 500
