"""The MRT collision (rows of M_COLLID and M_FORCE through scalar registers)
in every form of the fused kernel: with and without a volume force, with the
auxiliary planes, and with the immersed-boundary band; FP64 bit for bit
against the oracle, FP32-deviation storage within the 1e-5 velocity L2 its
other blocks are held to."""
import numpy as np
import pytest

from oracle.refcase import Case
from tests.golden.cases import ParityCase, Plate
from tests.helpers import mismatch, run_device, run_oracle

pytestmark = pytest.mark.gpu

FORCE = dict(volumeForceIn=(2e-5, -1e-5, 3e-6))
FORMS = {
    "plain": ((301,) * 6, {}, False),
    "force": ((301,) * 6, FORCE, False),
    "aux": ((102, 103, 203, 204, 201, 302), {}, False),
    "aux_force": ((101, 103, 203, 203, 302, 302), FORCE, False),
    "band": ((101, 103, 302, 302, 302, 302), {}, True),
    "band_force": ((101, 103, 302, 302, 302, 302), FORCE, True),
}


def _case(form, dims):
    bc, extra, band = FORMS[form]
    case = Case(dims=dims, bc=bc, collide=3, Re=8.0, uvwIn=(0.05, 0.0, 0.0), UrefType=9, Uref=0.05, LrefType=1,
                Lref=1.0, TrefType=0, ntolLBM=3, dtolLBM=1e-14, **extra)
    plates = [Plate(5, -2.0, 2.0, 2.0, 4, XYZo=(10.0, 7.0, 8.0), XYZAmpl=(0.0, 1.0, 0.0), Freq=0.01)] if band else []
    return ParityCase(f"mrt_{form}", case, nsteps=4, seed=71, ubase=(0.05, 0.0, 0.0), neq=0.01, plates=plates)


@pytest.mark.parametrize("form", list(FORMS))
def test_mrt_matches_oracle(form):
    print(f"[gpu] mrt {form}", flush=True)
    pc = _case(form, (21, 15, 17))
    n, m = mismatch(run_oracle(pc), run_device(pc))
    assert n == 0, f"{n} differ, max {m:.3e}"


@pytest.mark.parametrize("form", ["plain", "force", "aux_force"])
def test_mrt_fp32_tracks_fp64(form):
    from fsilbm3d_amd.block import LBMBlock
    from tests.helpers import derived, flow_kwargs
    print(f"[gpu] mrt fp32 {form}", flush=True)
    pc = _case(form, (21, 15, 17))
    d = derived(pc.case)
    u = []
    for prec in (0, 1):
        blk = LBMBlock(pc.case.dims, pc.case.dh, pc.case.origin, pc.case.bc, 3, d["nu"], pc.case.params, precision=prec)
        blk.set_flow(**flow_kwargs(pc.case))
        blk.upload(np.array(pc.initial_state(), dtype=np.float64))
        blk.update_volume_force(0.0)
        blk.set_boundary_conditions()
        blk.steps(10, 0.0, 1.0)
        u.append(blk.calculate_macro_quantities()[1])
        blk.close()
    assert np.sqrt(((u[1] - u[0]) ** 2).sum() / (u[0] ** 2).sum()) < 1e-5
