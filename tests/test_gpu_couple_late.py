"""A coupling call whose one launch gives up at a barrier (FSIL_COUPLE_LATE=k:
every workgroup leaves the k-th barrier as if it had waited too long, from the
first to one of the forcing rounds): the call reports it, leaves an empty band,
and the next call on the same block runs by the launches and gives what a fresh
block gives, bit for bit."""
import numpy as np
import pytest

from fsilbm3d_amd import _lib
from tests import test_gpu_rounds as rounds

pytestmark = pytest.mark.gpu


def _block(monkeypatch, precision, m, env):
    from fsilbm3d_amd.block import LBMBlock
    rng = np.random.default_rng(m)
    blk = LBMBlock(rounds.DIMS, 1.0, (0.0, 0.0, 0.0), (301,) * 6, 1, 0.05, precision=precision)
    blk.set_flow(uvwIn=(0.05, 0.0, 0.0))
    f = np.empty(blk.download().shape)
    f[...] = rounds.D3Q19_W if f.shape[-1] == 19 else rounds.D3Q19_W.reshape((19,) + (1,) * (f.ndim - 1))
    blk.upload(f * (1.0 + 0.05 * rng.standard_normal(f.shape)))
    blk.update_volume_force(0.0)
    i32 = lambda *a: np.array(a, np.int32)  # noqa: E731
    with monkeypatch.context() as p:
        p.setenv(*env)
        _lib.check(blk.lib.fsil_ibm_define_bodies(blk.handle, 1, _lib.iptr(i32(m)), _lib.iptr(i32(2)),
                                                  _lib.iptr(i32(1)), _lib.iptr(np.zeros(m, np.int32)),
                                                  _lib.iptr(i32(0, 1))))
    _lib.check(blk.lib.fsil_ibm_set_params(blk.handle, 10, 1e-14, 0.05, 1.0))
    return blk


def _call(blk, x, vel, area):
    m = len(area)
    force, lod, it, dm = np.zeros((m, 3)), np.zeros(12), np.zeros(1, np.int32), np.zeros(1)
    rc = blk.lib.fsil_ibm_interaction_force(blk.handle, 1.0, _lib.dptr(x), _lib.dptr(vel), _lib.dptr(area),
                                            _lib.dptr(np.array([[19.0, 13.0, 18.0]])), _lib.dptr(force),
                                            _lib.dptr(lod), _lib.iptr(it), _lib.dptr(dm))
    return rc, [force, lod, it, dm]


def _band_cells(blk):
    n = np.zeros(1, np.int32)
    _lib.check(blk.lib.fsil_ibm_band_info(blk.handle, _lib.iptr(n), None))
    return int(n[0])


@pytest.mark.parametrize("precision,m", [(0, 9), (1, 300)])
@pytest.mark.parametrize("barrier", [1, 2, 3, 4, 5, 7])
def test_a_late_call_fails_and_the_next_one_is_right(monkeypatch, barrier, precision, m):
    print(f"[gpu] late coupling call at barrier {barrier}, precision {precision}, {m} markers", flush=True)
    rng = np.random.default_rng(m)
    x = rounds._markers(m, "plane", rng)
    vel, area = 0.02 * rng.standard_normal((m, 3)), rng.uniform(0.2, 0.6, m)
    late = _block(monkeypatch, precision, m, ("FSIL_COUPLE_LATE", str(barrier)))
    rc, _ = _call(late, x, vel, area)
    assert rc != 0 and late.lib.fsil_last_error().decode() == "forcing rounds: a workgroup did not start in time"
    assert _band_cells(late) == 0
    plain = _block(monkeypatch, precision, m, ("FSIL_ROUNDS", "0"))
    for _ in range(2):
        ra, a = _call(late, x, vel, area)
        rb, b = _call(plain, x, vel, area)
        assert ra == rb == 0
        for blk in (late, plain):
            blk.collision_streaming_bc()
        assert _band_cells(late) == _band_cells(plain) > 0
        for p, q in zip(a + [late.download()], b + [plain.download()]):
            assert np.array_equal(p, q)
        x = x + 0.37
    late.close()
    plain.close()
