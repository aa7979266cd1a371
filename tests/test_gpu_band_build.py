"""The band of a coupling call (cells claimed, entries placed and ranked) at
the edges of its workgroups: 64 entries per marker against the claim's 1024
and the placing's 256, cells with few and with hundreds of entries.  Forces,
loads, iteration counts and the fluid after two coupled steps against the
oracle's serial loops bit for bit; and a second run, whose band numbers come
in another order, the same bits again."""
import numpy as np
import pytest

from fsilbm3d_amd import _lib

pytestmark = pytest.mark.gpu

DIMS = (40, 28, 36)
BC = (301,) * 6
NTOL, DTOL, UREF = 5, 1e-14, 0.05


def _case(m, layout):
    rng = np.random.default_rng(1000 + m)
    w = np.array([1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12)
    f = w[:, None, None, None] * (1.0 + 0.05 * rng.standard_normal((19,) + DIMS))
    if layout == "plane":
        k = np.arange(m)
        x = np.stack([8.3 + 0.9 * (k % 24), 5.1 + 0.7 * (k // 24), 17.4 + 0.05 * (k % 7)], 1)
    else:
        x = np.array([19.2, 13.7, 17.9]) + 0.8 * rng.standard_normal((m, 3)).clip(-3, 3)
    vel = 0.02 * rng.standard_normal((m, 3))
    area = rng.uniform(0.2, 0.6, m) * (1.0 if layout == "plane" else 4.0 / m)
    return f, np.ascontiguousarray(x), vel, area


def _device(f, x, vel, area):
    from fsilbm3d_amd.block import LBMBlock
    m = len(area)
    blk = LBMBlock(DIMS, 1.0, (0.0, 0.0, 0.0), BC, 1, 0.05)
    blk.set_flow(uvwIn=(0.05, 0.0, 0.0))
    blk.upload(f)
    blk.update_volume_force(0.0)
    i32 = lambda *a: np.array(a, np.int32)  # noqa: E731
    _lib.check(blk.lib.fsil_ibm_define_bodies(blk.handle, 1, _lib.iptr(i32(m)), _lib.iptr(i32(2)), _lib.iptr(i32(1)),
                                              _lib.iptr(np.zeros(m, np.int32)), _lib.iptr(i32(0, 1))))
    _lib.check(blk.lib.fsil_ibm_set_params(blk.handle, NTOL, DTOL, UREF, 1.0))
    xc = np.array([[19.0, 13.0, 18.0]])
    out = []
    for _ in range(2):
        force, lod, it, dm = np.zeros((m, 3)), np.zeros(12), np.zeros(1, np.int32), np.zeros(1)
        _lib.check(blk.lib.fsil_ibm_interaction_force(blk.handle, 1.0, _lib.dptr(x), _lib.dptr(vel), _lib.dptr(area),
                                                      _lib.dptr(xc), _lib.dptr(force), _lib.dptr(lod), _lib.iptr(it),
                                                      _lib.dptr(dm)))
        blk.collision_streaming_bc()
        out += [force, lod, int(it[0])]
        x = np.ascontiguousarray(x + 0.37)
    out.append(blk.download())
    blk.close()
    return out


def _oracle(f, x, vel, area):
    from fsilbm3d_amd import params as P
    from oracle.oracle import OracleBlock, lod_flow
    m = len(area)
    ob = OracleBlock(DIMS, 1.0, (0.0, 0.0, 0.0), BC, 1, P.srt(0.05, 1.0)[1], uvwIn=(0.05, 0.0, 0.0))
    f = f.copy()
    out = []
    for step in range(2):
        r = ob.step(f, 0.0, [dict(Exyz=x, Evel=vel, Ea=area)], dict(ntol=NTOL, dtol=DTOL, Uref=UREF, denIn=1.0))
        out += [r["Eforce"][0], lod_flow(r["Eforce"][0], x, np.zeros(m, np.int32), [[0, 1]],
                                         np.array([[19.0, 13.0, 18.0]]), 2), r["iters"]]
        x = np.ascontiguousarray(x + 0.37)
    out.append(f)
    return out


@pytest.mark.parametrize("m,layout", [(1, "cluster"), (15, "plane"), (16, "cluster"), (17, "plane"), (33, "plane"),
                                      (512, "cluster"), (513, "plane"), (640, "cluster")])
def test_band_build_against_the_serial_loops(m, layout):
    print(f"[gpu] band build m={m} {layout}", flush=True)
    case = _case(m, layout)
    ref = _oracle(*case)
    for _ in range(2):
        dev = _device(*case)
        assert len(dev) == len(ref)
        for a, b in zip(dev, ref):
            assert np.array_equal(a, b)
