"""Faces applied in the collide launch and the rim's single launch, against a
launch per axis (FSIL_FACES=0) bit for bit, over every code the plan takes on
each axis, halves of it inactive, both storage forms, whole-wave rows and
others, and rows of several per workgroup; and the FP64 form against the
oracle."""
import numpy as np
import pytest

from oracle.refcase import Case
from tests.golden.cases import ParityCase
from tests.helpers import derived, flow_kwargs, mismatch, run_device_block, run_oracle_block

pytestmark = pytest.mark.gpu

X = [(101, 103), (102, 104), (201, 204), (203, 302), (301, 301)]
Y = [(302, 302), (201, 203), (101, 204), (202, 302), (301, 301)]
Z = [(302, 302), (201, 201), (203, 203), (302, 201), (203, 302), (201, 203), (301, 301)]
# every pair of (y, z) with x running through its codes
COMBOS = [X[(i + 2 * j) % len(X)] + y + z for i, y in enumerate(Y) for j, z in enumerate(Z)]
DIMS = {0: (9, 8, 33), 1: (8, 7, 64)}


def _run(dims, bc, precision, model=1, steps=4):
    from fsilbm3d_amd.block import LBMBlock
    pc = ParityCase("faces", Case(dims=dims, bc=bc, collide=model, Re=8.0, uvwIn=(0.05, 0.0, 0.0),
                                  shearRateIn=(1e-3, -2e-3, 5e-4), UrefType=9, Uref=0.05, LrefType=1, Lref=1.0,
                                  TrefType=0), nsteps=steps, seed=17, ubase=(0.05, 0, 0), neq=0.01)
    d = derived(pc.case)
    blk = LBMBlock(dims, 1.0, (0.0, 0.0, 0.0), bc, model, d["nu"], pc.case.params, precision=precision)
    blk.set_flow(**flow_kwargs(pc.case))
    blk.upload(np.array(pc.initial_state(), dtype=np.float64))
    blk.update_volume_force(0.0)
    blk.set_boundary_conditions()
    blk.steps(steps, 0.0, 1.0)
    blk.set_boundary_conditions()  # a later start-up call reads the saved planes of the last step
    blk.steps(1, float(steps), 1.0)
    f = blk.download()
    blk.close()
    return f


@pytest.mark.parametrize("bc", COMBOS)
@pytest.mark.parametrize("rows", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_plan_matches_launch_per_axis(monkeypatch, precision, rows, bc):
    print(f"[gpu] face plan {bc} p{precision} rows {rows}", flush=True)
    new = _run(DIMS[rows], bc, precision)
    monkeypatch.setenv("FSIL_FACES", "0")
    old = _run(DIMS[rows], bc, precision)
    assert np.isfinite(old).all()
    n, m = mismatch(new, old)
    assert n == 0, f"{n} differ, max {m:.3e}"


@pytest.mark.parametrize("bc", COMBOS)
def test_plan_matches_oracle(bc):
    print(f"[gpu] face plan oracle {bc}", flush=True)
    pc = ParityCase("faces", Case(dims=(9, 8, 20), bc=bc, Re=8.0, uvwIn=(0.05, 0.0, 0.0),
                                  shearRateIn=(1e-3, -2e-3, 5e-4), UrefType=9, Uref=0.05, LrefType=1, Lref=1.0,
                                  TrefType=0), nsteps=5, seed=18, ubase=(0.05, 0, 0), neq=0.01)
    n, m = mismatch(run_oracle_block(pc)[0], run_device_block(pc)[0])
    assert n == 0, f"{n} differ, max {m:.3e}"


@pytest.mark.parametrize("dims", [(6, 6, 6), (6, 6, 300), (7, 6, 513), (5, 8, 20)])
@pytest.mark.parametrize("precision", [0, 1])
def test_plan_sizes(monkeypatch, precision, dims):
    """The smallest block the plan takes, one row per workgroup, rows too long
    for it and a block too thin for it."""
    bc = (101, 103, 201, 203, 302, 203)
    new = _run(dims, bc, precision, model=2)
    monkeypatch.setenv("FSIL_FACES", "0")
    old = _run(dims, bc, precision, model=2)
    n, m = mismatch(new, old)
    assert n == 0, f"{n} differ, max {m:.3e}"
