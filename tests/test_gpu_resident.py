"""The resident kernel of the population-global RKC engine (csrc/rkc_resident.hpp)
where its layout has edges, against the oracle: one and several workgroups,
256-row chunks of the norms that span workgroups (Golgi cells of 131 rows:
three per chunk; a last workgroup of a few rows), gap junctions in the cable
matrix exchanged per stage, the olive's gap currents between workgroups, and
the largest population the kernel takes; ion updates shared with helper
workgroups (granule cells: 578 rows as 256 + 256 + 66).

Without ion updates the first macro step uses only correctly rounded
arithmetic and libm's pow for the step sizes, so voltages, derivative,
controller and counters are equal bit for bit.  With them the first macro step
agrees to the rounding of exp (1e-9 mV, the bar of the other grid tests) and
takes the same steps."""
import os

import numpy as np
import pytest

import cbrkc
import orc
from test_oracle_go import go_pop
from test_oracle_gr import gr_pop
from test_oracle_io import io_pop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,coupled", [(1, 1, False), (2, 1, False), (9, 1, False), (2, 1, True), (3, 2, True)])
def test_purkinje_without_ion_updates_is_bit_exact(ref_data, nx, ny, coupled):
    print(f"Purkinje {nx}x{ny}, gap junctions {coupled}", flush=True)
    n = nx * ny
    morph = os.path.join(ref_data, "Pkj.txt")
    gj = os.path.join(ref_data, "Pkj_GJ.csv") if coupled else ""
    v0 = -68.0 + np.arange(n) * 0.21
    kw = dict(nx=nx, ny=ny, v0=v0, atol=1e-6, rtol=1e-6)
    o = orc.Pop.pkj(morph, libc_rand=False, gj=gj or None, **kw)
    orc.lib().or_pop_set_integ(o.h, 1e30)
    p = cbrkc.Population(cbrkc.PKJ, morph=morph, gj=gj, ion_interval=1e30, **kw)
    assert "workgroups" in p.mapping()
    o.set_current(0.0)
    o.advance()
    p.set_current(0.0)
    p.advance()
    for fo, fg in ((orc.VNEW, cbrkc.F_VNEW), (orc.YN, cbrkc.F_YN), (orc.FN, cbrkc.F_FN), (orc.Y, cbrkc.F_Y)):
        assert np.array_equal(o.get(fo), p.read(fg)), fo
    assert np.array_equal(o.controller()[0], p.controller()[0])
    so, sg = o.stats(), p.stats()
    assert all(so[k] == sg[k] for k in ("steps", "rejects", "stages", "rho_iters")), (so, sg)


@pytest.mark.parametrize("cell,nx,ny", [("io", 5, 5), ("io", 10, 9), ("io", 13, 40), ("go", 1, 1), ("go", 5, 3), ("gr", 1, 1),
                                        ("gr", 3, 1)])
def test_grids_first_macro_step(ref_data, cell, nx, ny):
    print(f"{cell} {nx}x{ny}", flush=True)
    n = nx * ny
    v0 = (-70.0 if cell == "gr" else -60.0) + 0.03 * np.arange(n) % 2.0
    if cell == "gr":
        o, kind, f = gr_pop(ref_data, nx, ny, v0=v0), cbrkc.GR, "Gr.txt"
    elif cell == "io":
        o, kind, f = io_pop(ref_data, nx, ny, v0=v0), cbrkc.IO, "IO.txt"
    else:
        o, kind, f = go_pop(ref_data, nx, ny, v0=v0), cbrkc.GO, "Go_131.txt"
    p = cbrkc.Population(kind, nx, ny, morph=os.path.join(ref_data, f), v0=v0)
    assert "workgroups" in p.mapping()
    o.set_current(0.0)
    o.advance()
    out = p.run(1, 0.0, 0)
    v = p.read(cbrkc.F_VNEW)
    assert np.abs(v - o.get(orc.VNEW)).max() <= 1e-9
    assert np.array_equal(out[0], v[::p.comp])
    so, sg = o.stats(), p.stats()
    assert all(so[k] == sg[k] for k in ("steps", "rejects", "stages", "rho_iters", "ion_updates")), (so, sg)


@pytest.mark.parametrize("n,resident", [(256, True), (257, False)])
def test_largest_population(ref_data, n, resident):
    # a cell per CU fits; one more would take two 1600-row cells to a workgroup
    print(f"Purkinje {n} uncoupled cells", flush=True)
    # equal cells before their first ion update (which depends on the cell's index) share the single cell's
    # error norm, the mean of equal terms, to the rounding of its sum
    v0 = np.full(n, -67.0)
    kw = dict(morph=os.path.join(ref_data, "Pkj.txt"), ion_interval=1e30)
    p = cbrkc.Population(cbrkc.PKJ, n, 1, v0=v0, **kw)
    assert ("workgroups" in p.mapping()) == resident
    one = cbrkc.Population(cbrkc.PKJ, 1, 1, v0=v0[:1], **kw)
    a, b = p.run(1, 0.0, 1599), one.run(1, 0.0, 1599)
    assert np.abs(a - b).max() <= 1e-9
