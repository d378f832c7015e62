"""Failure paths of the RKC engines through the C-ABI (GPU).

* A NaN in a cell's state: the reference's main stops on a NaN voltage
  (main.cu:200, 228, 257, 287, `isnan ( memv_test_xx [ 1 ] )`); here
  cb_pop_run / cb_pop_advance return CB_E_SOLVER with a message naming the
  state (and, for the per-cell engines, the cell) instead of stepping NaNs.
* The step-size floor: when a rejected step would go below hmin the reference
  sets idid = 4 and falls through to the accept branch (solve_rkc.cu:1003-1010),
  so the run goes on with the step it attempted.  With hmin raised to H_MAX
  (cb_pop_config.hmin_ms) every step is clamped to [hmin, hmax] = 0.125 ms:
  each macro step is exactly one accepted step per controller, whatever its
  error; rejections that fall below hmin are counted and then accepted, and
  the run ends without an error.
* A workgroup that waits for another one in vain: with a limit of no time at
  all (cb_pop_wait_limit) the first empty mailbox ends the launch, and the call
  fails at once; solves already queued fall through.
"""
import os
import time

import numpy as np
import pytest

import cbrkc

CB_E_SOLVER = -4


@pytest.fixture(scope="module")
def morph2(tmp_path_factory):
    d = tmp_path_factory.mktemp("fail")
    path = str(d / "pkj2.txt")
    cbrkc.synth_pkj_morph(path, seed=7, ncell=2)
    return path


@pytest.mark.gpu
@pytest.mark.parametrize("engine", [cbrkc.ENGINE_CELL_MIXED, cbrkc.ENGINE_CELL_FP64, cbrkc.ENGINE_GLOBAL_FP64],
                         ids=["mixed", "cell_fp64", "global_fp64"])
def test_nan_state_stops_the_run(morph2, engine):
    print(f"NaN initial voltage in cell 1, engine {engine}", flush=True)
    p = cbrkc.Population(cbrkc.PKJ, 2, 1, engine=engine, morph=morph2, v0=[-68.0, float("nan")],
                         stim=(1599, 0.0, 1e9, 0.0), **cbrkc.STABLE)
    with pytest.raises(cbrkc.CbError) as e:
        p.run(2, 0.0, 1599)
    msg = str(e.value)
    assert "non-finite" in msg, msg
    if engine != cbrkc.ENGINE_GLOBAL_FP64:
        assert "cell 1" in msg, msg


@pytest.mark.gpu
@pytest.mark.parametrize("engine", [cbrkc.ENGINE_CELL_MIXED, cbrkc.ENGINE_GLOBAL_FP64], ids=["mixed", "global_fp64"])
def test_steps_below_hmin_fall_through_as_accepted(morph2, engine):
    print(f"hmin = H_MAX, engine {engine}", flush=True)
    p = cbrkc.Population(cbrkc.PKJ, 2, 1, engine=engine, morph=morph2, v0=[-68.0, -67.0], hmin_ms=0.125,
                         stim=(1599, 0.0, 1e9, 0.5e-3), **cbrkc.STABLE)
    s0 = p.stats()
    out = p.run(6, 0.0, 1599)
    s1 = p.stats()
    assert np.all(np.isfinite(out))
    ncontrollers = 1 if engine == cbrkc.ENGINE_GLOBAL_FP64 else 2
    assert s1["steps"] - s0["steps"] == 6 * ncontrollers, (s0, s1)
    # some 0.125 ms steps miss the 1e-6 tolerance: rejected, then accepted at hmin
    assert s1["rejects"] - s0["rejects"] > 0, (s0, s1)


@pytest.mark.gpu
@pytest.mark.parametrize("solver", [cbrkc.CN, cbrkc.BE], ids=["cn", "be"])
def test_a_solve_that_waits_in_vain_fails_the_run(tmp_path, solver):
    print(f"4 Purkinje cells, solver {solver}, no time to wait", flush=True)
    morph = str(tmp_path / "pkj4.txt")
    cbrkc.synth_pkj_morph(morph, seed=7, ncell=4)
    p = cbrkc.Population(cbrkc.PKJ, 4, 1, solver=solver, morph=morph, v0=[-68.0, -67.0, -66.0, -67.5])
    assert "13 workgroups" in p.mapping()
    p.wait_limit(0.0)
    t0 = time.monotonic()
    with pytest.raises(cbrkc.CbError, match="in vain"):
        p.run(4, 0.0, 0)   # 20 solves, queued before the first is looked at
    p.wait_limit(60.0)   # what is left in the mailboxes is never read
    with pytest.raises(cbrkc.CbError, match="in vain"):
        p.run(1, 0.5, 0)
    with pytest.raises(cbrkc.CbError, match="in vain"):
        p.read()
    q = cbrkc.Population(cbrkc.PKJ, 4, 1, solver=solver, morph=morph, v0=[-68.0, -67.0, -66.0, -67.5])
    q.wait_limit(0.0)
    q.set_current(0.0)
    for _ in range(2):   # the step itself, and every one after it
        with pytest.raises(cbrkc.CbError, match="in vain"):
            q.advance()
    assert time.monotonic() - t0 < 10.0


@pytest.mark.gpu
@pytest.mark.parametrize("cell,nx,ny,f,v", [("IO", 13, 40, "IO.txt", -60.0), ("GO", 3, 2, "Go_131.txt", -60.0),
                                            ("PKJ", 3, 1, "Pkj.txt", -68.0), ("GR", 1, 1, "Gr.txt", -70.0)])
def test_a_step_that_waits_in_vain_fails_the_population(ref_data, cell, nx, ny, f, v):
    # several workgroups, gap currents, gap junctions, and a single cell's helpers
    print(f"{nx * ny} {cell} cells, no time to wait", flush=True)
    p = cbrkc.Population(getattr(cbrkc, cell), nx, ny, morph=os.path.join(ref_data, f), v0=np.full(nx * ny, v))
    p.wait_limit(0.0)
    t0 = time.monotonic()
    with pytest.raises(cbrkc.CbError, match="in vain"):
        p.run(4, 0.0, 0)
    p.wait_limit(60.0)
    for call in (lambda: p.run(1, 0.5, 0), p.advance, p.read):
        with pytest.raises(cbrkc.CbError, match="in vain"):
            call()
    assert time.monotonic() - t0 < 10.0
