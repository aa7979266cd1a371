"""The forcing rounds of a coupling call in their two forms: all rounds in one
launch with a barrier between them (few markers) and two launches per round
(FSIL_ROUNDS=0, and above 512 markers).  Markers around the edges of the
workgroups and of the range, cells with few and with hundreds of entries,
loops that end early, at the cap, at once and not at all: every output of two
coupling calls and of the fluid steps after them is the same bit for bit."""
import os

import numpy as np
import pytest

from fsilbm3d_amd import _lib

pytestmark = pytest.mark.gpu

DIMS = (40, 28, 36)
D3Q19_W = np.array([1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12)


def _markers(m, layout, rng):
    """Marker positions: a plane one cell apart, or a cluster with many markers per cell."""
    if layout == "plane":
        k = np.arange(m)
        x = np.stack([8.3 + 0.9 * (k % 24), 5.1 + 0.7 * (k // 24), 17.4 + 0.05 * (k % 7)], 1)
    else:
        x = np.array([19.2, 13.7, 17.9]) + 0.8 * rng.standard_normal((m, 3)).clip(-3, 3)
    return np.ascontiguousarray(x)


def _run(form, m, layout, precision, ntol, dtol, bad=False):
    from fsilbm3d_amd.block import LBMBlock
    rng = np.random.default_rng(m)
    blk = LBMBlock(DIMS, 1.0, (0.0, 0.0, 0.0), (301,) * 6, 1, 0.05, precision=precision)
    blk.set_flow(uvwIn=(0.05, 0.0, 0.0))
    f = np.empty(blk.download().shape)
    f[...] = (D3Q19_W if f.shape[-1] == 19 else D3Q19_W.reshape((19,) + (1,) * (f.ndim - 1)))
    f *= 1.0 + 0.05 * rng.standard_normal(f.shape)
    blk.upload(f)
    blk.update_volume_force(0.0)
    old = os.environ.pop("FSIL_ROUNDS", None)
    if form:
        os.environ["FSIL_ROUNDS"] = form
    i32 = lambda *a: np.array(a, np.int32)  # noqa: E731
    try:  # read when the bodies are defined
        _lib.check(blk.lib.fsil_ibm_define_bodies(blk.handle, 1, _lib.iptr(i32(m)), _lib.iptr(i32(2)),
                                                  _lib.iptr(i32(1)), _lib.iptr(np.zeros(m, np.int32)),
                                                  _lib.iptr(i32(0, 1))))
    finally:
        os.environ.pop("FSIL_ROUNDS", None)
        if old is not None:
            os.environ["FSIL_ROUNDS"] = old
    _lib.check(blk.lib.fsil_ibm_set_params(blk.handle, ntol, dtol, 0.05, 1.0))
    x = _markers(m, layout, rng)
    vel = 0.02 * rng.standard_normal((m, 3))
    area = rng.uniform(0.2, 0.6, m) * (1.0 if layout == "plane" else 0.02)
    if bad:
        vel[m // 2, 1] = np.nan
    xc = np.array([[19.0, 13.0, 18.0]])
    out, err = [], None
    for step in range(2):
        force, lod, it, dm = np.zeros((m, 3)), np.zeros(12), np.zeros(1, np.int32), np.zeros(1)
        rc = blk.lib.fsil_ibm_interaction_force(blk.handle, 1.0, _lib.dptr(x), _lib.dptr(vel), _lib.dptr(area),
                                                _lib.dptr(xc), _lib.dptr(force), _lib.dptr(lod), _lib.iptr(it),
                                                _lib.dptr(dm))
        if rc:
            err = blk.lib.fsil_last_error().decode()
            break
        rounds = np.zeros(1, np.int32)
        _lib.check(blk.lib.fsil_ibm_rounds(blk.handle, _lib.iptr(rounds)))
        blk.collision_streaming_bc()
        out += [force, lod, it, dm, rounds, blk.download()]
        x = x + 0.37
    blk.close()
    return out, err


@pytest.mark.parametrize("m,layout,precision,ntol,dtol", [
    (1, "plane", 0, 10, 1e-14), (3, "plane", 1, 10, 1e-14), (4, "cluster", 0, 10, 1e-14), (5, "plane", 0, 1, 1e-14),
    (64, "cluster", 0, 3, 1e-14), (255, "plane", 0, 10, 1e-14), (256, "cluster", 1, 10, 1e-14),
    (257, "plane", 1, 10, 0.5), (300, "plane", 0, 10, 0.1), (300, "plane", 0, 0, 1e-14), (300, "plane", 0, 4, 1e30),
    (511, "cluster", 0, 10, 1e-14), (512, "plane", 0, 10, 1e-14), (513, "plane", 0, 10, 1e-14)])
def test_rounds_in_one_launch_match_two_launches_per_round(m, layout, precision, ntol, dtol):
    print(f"[gpu] forcing rounds m={m} {layout} precision={precision} ntol={ntol} dtol={dtol}", flush=True)
    a, ea = _run(None, m, layout, precision, ntol, dtol)
    b, eb = _run("0", m, layout, precision, ntol, dtol)
    assert ea is None and eb is None
    assert len(a) == len(b) == 12
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    assert np.isfinite(a[0]).all() and (ntol == 0 or dtol > 1e20 or np.abs(a[0]).max() > 0.0)


def test_not_a_number_is_reported_by_both_forms():
    print("[gpu] forcing rounds with a NaN marker velocity", flush=True)
    for form in (None, "0"):
        _, err = _run(form, 130, "plane", 0, 10, 1e-14, bad=True)
        assert err == "Nan found in PenaltyForce"
