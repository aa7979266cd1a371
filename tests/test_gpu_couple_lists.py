"""The one-launch coupling call where some workgroups have cells of more than
sixteen entries and others have none (pitched plates one cell apart, sparse
markers beside a cluster, in either order): every output of two coupling calls
and of the fluid steps after them is the same bit for bit as with a launch per
stage and round (FSIL_ROUNDS=0)."""
import numpy as np
import pytest

from tests import test_gpu_rounds as rounds

pytestmark = pytest.mark.gpu

LIST = 16  # entries of a cell that a lane keeps in registers


def _pitched(side, degrees):
    i, j = np.divmod(np.arange(side * side), side)
    a = np.radians(degrees)
    return np.stack([6.2 + np.cos(a) * i, 4.3 + np.sin(a) * i, 7.4 + j], 1)


def _mixed(sparse, dense, dense_first):
    k = np.arange(sparse)
    far = np.stack([0.3 + 4.0 * (k % 10), 0.6 + 4.0 * (k // 10 % 7), 0.4 + 4.0 * (k // 70)], 1)
    rng = np.random.default_rng(sparse + dense)
    near = np.array([21.2, 14.7, 33.9]) + 0.6 * rng.standard_normal((dense, 3)).clip(-2, 2)
    return np.concatenate([near, far] if dense_first else [far, near])


LAYOUTS = {
    "16x16 at 20 degrees": _pitched(16, 20.0),
    "16x16 at 30 degrees": _pitched(16, 30.0),
    "22x22 at 20 degrees": _pitched(22, 20.0),
    "256 sparse, 256 dense": _mixed(256, 256, False),
    "300 dense, 4 sparse": _mixed(4, 300, True),
    "4 sparse, 300 dense": _mixed(4, 300, False),
    "40 dense, 200 sparse": _mixed(200, 40, True),
}


def _crowded_groups(x):
    """Per workgroup of four markers: whether one of its cells has more than LIST entries (periodic block)."""
    dims = np.array(rounds.DIMS)
    idx = np.floor(x[:, None, :] + 0.0).astype(int) + np.arange(-1, 3)[None, :, None]  # [m, 4, axis]
    idx %= dims
    cell = ((idx[:, :, None, None, 0] * dims[1] + idx[:, None, :, None, 1]) * dims[2] +
            idx[:, None, None, :, 2]).reshape(len(x), 64)
    n = np.bincount(cell.ravel(), minlength=int(dims.prod()))
    long = (n[cell] > LIST).any(1)
    return [bool(long[k:k + 4].any()) for k in range(0, len(x), 4)]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_mixed_entry_lists_match_the_launches(monkeypatch, layout, precision):
    x = LAYOUTS[layout]
    for shift in (0.0, 0.37):  # (the markers of the two calls)
        kinds = _crowded_groups(x + shift)
        assert any(kinds) and not all(kinds)
    print(f"[gpu] mixed entry lists: {layout}, precision {precision}, {sum(kinds)} of {len(kinds)} crowded", flush=True)
    monkeypatch.setattr(rounds, "_markers", lambda m, name, rng: np.ascontiguousarray(x))
    a, ea = rounds._run(None, len(x), layout, precision, 10, 1e-14)
    b, eb = rounds._run("0", len(x), layout, precision, 10, 1e-14)
    assert ea is None and eb is None
    assert len(a) == len(b) == 12
    for p, q in zip(a, b):
        assert np.array_equal(p, q)
    assert np.isfinite(a[0]).all() and np.abs(a[0]).max() > 0.0
