"""The network's product and update kernels at the edges of their shapes:
one k-tile and several more than are in flight (K = 64 to 704), both tile
sizes (fewer and more than 256 blocks of 64 x 64), batches whose bias sums take
one, part of a second and three passes through LDS (64 to 320 rows), padded
inputs and hidden widths, and a network of one layer.

Gradients against the CPU oracle with the same bfloat16 roundings within
5e-3 relative L2 (accumulation order and the occasional activation that
rounds to the neighbouring bfloat16 value), the loss within 1e-4; the first
Adam step moves every weight by lr * g / (|g| + eps'), so where |g| is far
above its error the step equals the oracle's to 2e-5.
"""
import numpy as np
import pytest

from nexd_amd import mlp
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("widths,B", [([9, 64], 64), ([70, 130, 64], 192), ([64, 704, 128], 320), ([9, 320, 8256], 128),
                                      ([5, 65, 577, 192], 256)])
def test_gradients_and_step(widths, B):
    print(f"[gpu mlp shapes] widths={widths} B={B}", flush=True)
    rng = np.random.default_rng(11)
    params = [(w, (rng.standard_normal(w.shape[0]) * 0.1).astype(np.float32)) for w, _ in mlp.init_params(widths, 12)]
    x = rng.standard_normal((B + 37, widths[0])).astype(np.float32)
    t = rng.standard_normal((B + 37, widths[-1])).astype(np.float32)
    idx = rng.permutation(B + 37)[:B].astype(np.int32)
    with mlp.MLP(widths, max_batch=B + 64) as net:
        net.set_params(params)
        net.upload_dataset(x, t)
        loss = net.gradients(idx)
        g = net.grads()
        assert all(np.array_equal(a, b) for p, q in zip(net.params(), params) for a, b in zip(p, q))
        losses = net.train(idx, B, lr=1e-3)
        g2, p2 = net.grads(), net.params()
    lo, go = mo.loss_and_grads(params, x[idx], t[idx], bf16_ops=True)
    assert abs(loss - lo) <= 1e-4 * lo and losses[0] == np.float32(loss)
    po = mo.adam_step([(w.astype(np.float64), b.astype(np.float64)) for w, b in params], go, {}, lr=1e-3)
    for l in range(len(params)):
        for k in range(2):
            assert rel(g[l][k], go[l][k]) <= 5e-3
            assert np.array_equal(g[l][k], g2[l][k])
            clear = np.abs(go[l][k]) > 0.1 * np.sqrt(np.mean(go[l][k] ** 2))
            assert clear.mean() > 0.5
            assert np.max(np.abs(p2[l][k] - po[l][k])[clear]) <= 2e-5
