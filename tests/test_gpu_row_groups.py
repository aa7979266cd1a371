"""Workgroups of several whole z-rows: row lengths that fill no wave, row
counts that leave the last workgroup part idle, rows too long for one
workgroup, and bands crossing them; the FP64 form bit for bit against the
oracle, the FP32-deviation form bit for bit against its launches without the
row exchange."""
import numpy as np
import pytest

from oracle.refcase import Case
from tests.golden.cases import ParityCase, Plate
from tests.helpers import derived, flow_kwargs, mismatch, run_device, run_device_block, run_oracle, run_oracle_block

pytestmark = pytest.mark.gpu

# 33: 9 rows of 10; 133: 3 rows of 7; 77: 4 rows of 6; 300: one row; 600: cut rows
DIMS = [(6, 10, 33), (5, 7, 133), (5, 6, 77), (4, 5, 300), (4, 4, 600), (7, 4, 4)]


def _case(dims, model=1, bc=(101, 104, 203, 302, 301, 301), **kw):
    return Case(dims=dims, bc=bc, collide=model, Re=8.0, uvwIn=(0.05, 0.0, 0.0), UrefType=9, Uref=0.05, LrefType=1,
                Lref=1.0, TrefType=0, **kw)


@pytest.mark.parametrize("model", [1, 2, 3, 11, 15])
@pytest.mark.parametrize("dims", DIMS)
def test_fp64_rows_match_oracle(dims, model):
    print(f"[gpu] rows {dims} model {model}", flush=True)
    pc = ParityCase("rows", _case(dims, model), nsteps=3, seed=81, ubase=(0.05, 0, 0), neq=0.01)
    fo, to = run_oracle_block(pc)
    fd, td = run_device_block(pc)
    n, m = mismatch(fo, fd)
    nt, mt = mismatch(to, td)
    assert n == 0 and nt == 0, (n, m, nt, mt)


def test_fp64_band_in_a_part_idle_group():
    """A plate whose band reaches the last, part idle workgroup of rows (the
    whole-block launch and, on the second form, the split step's hull)."""
    pc = ParityCase("rows_band", _case((24, 22, 33), bc=(101, 103, 302, 302, 302, 302), ntolLBM=3, dtolLBM=1e-14),
                    nsteps=4, seed=82, ubase=(0.05, 0, 0), neq=0.01,
                    plates=[Plate(5, -2.0, 2.0, 2.0, 4, XYZo=(10.0, 18.0, 16.0), XYZAmpl=(0.0, 1.0, 0.0), Freq=0.01)])
    print("[gpu] rows band", flush=True)
    want = run_oracle(pc)
    n, m = mismatch(want, run_device(pc))
    assert n == 0, f"{n} differ, max {m:.3e}"


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("precision", [0, 1])
def test_band_steps_match_shifted_stores(monkeypatch, split, precision):
    """Coupled steps on rows of 33 cells, with the exchange and without it
    (FSIL_ZROW=0), unsplit and split: the same state bit for bit."""
    from fsilbm3d_amd.block import LBMBlock
    from fsilbm3d_amd.fsi import DeviceBodyBlock
    from fsilbm3d_amd.workloads import FlexiblePlate
    print(f"[gpu] rows coupled split {split} precision {precision}", flush=True)
    w = FlexiblePlate(dims=(40, 31, 33), L=8.0, Re=60.0, le=(12.0, 18.0, 16.0), body_model=1, ntolLBM=3)
    out = []
    monkeypatch.setenv("FSIL_SPLIT", split)
    for zrow in ("0", None):
        if zrow:
            monkeypatch.setenv("FSIL_ZROW", zrow)
        else:
            monkeypatch.delenv("FSIL_ZROW")
        blk = LBMBlock(w.dims, 1.0, (0.0, 0.0, 0.0), w.bc, 1, w.nu, precision=precision)
        blk.set_flow(**w.flow_kwargs())
        blk.fill(w.equilibrium())
        blk.update_volume_force(0.0)
        blk.set_boundary_conditions()
        fsi = DeviceBodyBlock(blk, [w.plate()], **w.solver_kwargs())
        for k in range(6):
            fsi.step(float(k + 1))
        out.append(blk.download())
        blk.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("model", [1, 2, 3])
@pytest.mark.parametrize("dims", DIMS)
def test_fp32_rows_match_shifted_stores(monkeypatch, dims, model):
    from fsilbm3d_amd.block import LBMBlock
    print(f"[gpu] rows fp32 {dims} model {model}", flush=True)
    pc = ParityCase("rows32", _case(dims, model), nsteps=4, seed=83, ubase=(0.05, 0, 0), neq=0.01)
    d = derived(pc.case)
    out = []
    for zrow in ("0", "1", None):
        if zrow is None:
            monkeypatch.delenv("FSIL_ZROW")
        else:
            monkeypatch.setenv("FSIL_ZROW", zrow)
        blk = LBMBlock(dims, 1.0, (0.0, 0.0, 0.0), pc.case.bc, model, d["nu"], pc.case.params, precision=1)
        blk.set_flow(**flow_kwargs(pc.case))
        blk.upload(np.array(pc.initial_state(), dtype=np.float64))
        blk.update_volume_force(0.0)
        blk.set_boundary_conditions()
        blk.steps(4, 0.0, 1.0)
        out.append(blk.download())
        blk.close()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
