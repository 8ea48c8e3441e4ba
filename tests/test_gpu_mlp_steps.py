"""The training step's fused launches: gradients at row counts around the tiles
of the layers' backward launches (32 and 64 wide), and one step of a training
epoch against mlp_gradients on the epoch's rows with Adam on the host.

Tolerances: gradients 2e-3 in L2 per layer against the BF16 reference (as in
test_gpu_mlp.py); a step's parameters to 1e-5 of its length (the moments'
FP32 rounding) and half a unit of the parameter."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel
from oracle import mlp_ref

from .test_gpu_mlp import _params, _rel

pytestmark = pytest.mark.gpu


def _set(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, 54)).astype(np.float32),
            rng.standard_normal((n, 4)).astype(np.float32))


@pytest.mark.parametrize("n", [1, 16, 33, 272, 4032, 4112])
def test_gradients_at_tile_edges(n):
    print(f"\n[case] mlp gradients, {n} rows", flush=True)
    X, T = _set(n, n)
    P = _params(3)
    loss_o, G_o = mlp_ref.loss_and_grad(P, X, T, bf16_ops=True)
    with Channel(18, 17, 18) as ch:
        ch.mlp_init(1)
        ch.mlp_set_params(P)
        G, loss = ch.mlp_gradients(X, T)
    assert abs(loss - loss_o) <= 1e-4 * loss_o
    for w, b, i, o in mlp_ref.layout()[0]:
        assert _rel(G[w:w + o * i], G_o[w:w + o * i]) < 2e-3
        assert _rel(G[b:b + o], G_o[b:b + o]) < 2e-3


def _order(n, seed):
    """The shuffle of a first epoch: Fisher-Yates with splitmix64."""
    m = (1 << 64) - 1
    p, x = list(range(n)), seed
    for i in range(n - 1, 0, -1):
        x = (x + 0x9E3779B97F4A7C15) & m
        z = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
        z ^= z >> 31
        j = z % (i + 1)
        p[i], p[j] = p[j], p[i]
    return p


@pytest.mark.parametrize("n,batch", [(16, 16), (31, 16), (300, 272)])
def test_one_training_step(n, batch):
    print(f"\n[case] one training step, {n} rows in batches of {batch}", flush=True)
    X, T = _set(n, 5)
    P, lr, f = _params(4), 1e-3, np.float32
    rows = _order(n, 7)[:batch]
    with Channel(18, 17, 18) as ch:
        ch.mlp_init(1)
        ch.mlp_set_params(P)
        g, _ = ch.mlp_gradients(X[rows], T[rows])
        ch.mlp_train(X, T, 1, batch=batch, lr=lr, seed=7)
        got = ch.mlp_params()
    m, v = f(1 - f(0.9)) * g, f(1 - f(0.999)) * g * g
    lr_t = f(lr) * np.sqrt(f(1) - f(0.999)) / (f(1) - f(0.9))
    ref = P - lr_t * m / (np.sqrt(v) + f(1e-8))
    assert np.all(np.abs(got - ref) <= 1e-5 * lr + np.spacing(np.abs(P)))
