"""The network's row kernel (64-row tiles, up to 256 workgroups sharing them)
at its edges: fewer rows than a tile, a tile and one more, a last tile of one
row, and more tiles than workgroups; against the float64 oracle.

FP32 sums of up to 16,385 terms in products of depth 64: the outputs stay
within 64 ulp-sized roundings (64 * 2^-24 = 4e-6, taken as 1e-5) of the
largest, the gradients within 1e-4 of the largest, the loss within 1e-5."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200, 16384, 16385])
def test_rows_match_oracle(n):
    print(f"[gpu] mlp rows {n}", flush=True)
    from fsilbm3d_amd.mlp import WarmStartNet
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 12)).astype(np.float32)
    Y = (0.5 * np.tanh(X[:, :3]) + 0.1 * X[:, 3:6]).astype(np.float32)
    net = WarmStartNet(3 + n)
    th = net.params.astype(np.float64)
    ref, _ = MO.forward(th, X.astype(np.float64))
    assert np.abs(net.forward(X, bf16=False) - ref).max() < 1e-5 * max(1.0, np.abs(ref).max())
    # BF16 operands, as tests of the inference kernel hold them
    assert np.abs(net.forward(X, bf16=True) - ref).max() < 2e-2 * max(1.0, np.abs(ref).max())
    loss, g = net.loss_grad(X, Y)
    l_ref, g_ref = MO.loss_grad(th, X.astype(np.float64), Y.astype(np.float64))
    assert abs(loss - l_ref) < 1e-5 * l_ref
    assert np.abs(g - g_ref).max() < 1e-4 * np.abs(g_ref).max()
    # a batch of the same rows in a shuffled order: the first Adam step moves
    # every parameter by lr * sign(g) wherever g is not ~0
    before = net.params.astype(np.float64)
    net.train(X, Y, epochs=1, batch=n, lr=1e-3, seed=4)
    th1, _, _ = MO.adam_step(before, g_ref, np.zeros_like(g_ref), np.zeros_like(g_ref), 1, 1e-3)
    big = np.abs(g_ref) > 1e-3 * np.abs(g_ref).max()
    assert np.abs(net.params.astype(np.float64) - th1)[big].max() < 1e-6
