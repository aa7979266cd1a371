"""Split coupled steps against unsplit ones over what a block can be: the
collision models, a volume force, the faces with auxiliary planes (102, 203,
204), both storage forms, one and two bodies; the state, forces and beam state
bit for bit."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FACES = {
    "open": (101, 103, 302, 302, 302, 302),
    "aux": (102, 103, 203, 204, 201, 302),
    "periodic": (301, 301, 301, 301, 203, 203),
}


def _run(monkeypatch, split, precision, model, faces, bodies):
    from fsilbm3d_amd.block import LBMBlock
    from fsilbm3d_amd.fsi import DeviceBodyBlock
    from fsilbm3d_amd.workloads import FlexiblePlate
    monkeypatch.setenv("FSIL_SPLIT", split)
    w = FlexiblePlate(dims=(54, 36, 28), L=8.0, Re=60.0, le=(12.0, 18.0, 14.0), ntolLBM=3, numsubstep=2,
                      bc=FACES[faces])
    blk = LBMBlock(w.dims, 1.0, (0.0, 0.0, 0.0), w.bc, model, w.nu, (0.1875,) + (0.0,) * 9, precision=precision)
    blk.set_flow(**w.flow_kwargs(), volumeForceIn=(1e-5, -2e-6, 0.0) if faces == "periodic" else (0.0, 0.0, 0.0))
    blk.fill(w.equilibrium())
    blk.update_volume_force(0.0)
    blk.set_boundary_conditions()
    plates = [w.plate()]
    if bodies == 2:
        plates.append(dataclasses.replace(dataclasses.replace(w, le=(30.0, 18.0, 14.0), body_model=1).plate(),
                                          XYZPhi=(0.0, 90.0, 0.0)))
    fsi = DeviceBodyBlock(blk, plates, **w.solver_kwargs())
    forces = []
    for k in range(6):
        fsi.step(float(k + 1))
        forces.append(fsi.Eforce.copy())
    out = [blk.download(), np.array(forces)] + [a.copy() for i in range(bodies) for a in fsi.state(i)]
    blk.close()
    return out


@pytest.mark.parametrize("bodies", [1, 2])
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("model", [1, 2, 3])
@pytest.mark.parametrize("precision", [0, 1])
def test_split_matches_unsplit(monkeypatch, precision, model, faces, bodies):
    print(f"[gpu] split forms p{precision} m{model} {faces} {bodies}", flush=True)
    a = _run(monkeypatch, "0", precision, model, faces, bodies)
    b = _run(monkeypatch, "1", precision, model, faces, bodies)
    for x, y in zip(a, b):
        assert np.isfinite(x).all() and np.array_equal(x, y)
