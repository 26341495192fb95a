"""The surrogate's row, weight-gradient and update kernels at the edges of
their tiling (32 rows per workgroup, 32 row slices of which trailing ones may
be empty, 16 embedding columns at any offset P): the parameter gradient and
the prediction against the CPU oracle (oracle/mlp_oracle.py) with BF16
emulation, and the BF16 weight copies the update kernel leaves against those
packed from the parameters it wrote."""
import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.surrogate import Surrogate, split_parameters
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


# one row, a workgroup's last row and one more, one slice step per slice and
# one more (1024 rows), several steps per slice with empty slices, P = 16
@pytest.mark.parametrize("n,p", [(1, 2), (32, 1), (33, 16), (1024, 2), (1025, 8), (2177, 5)])
def test_gradient_and_prediction_at_tile_edges(n, p):
    print(f"surrogate kernels n={n} p={p}", flush=True)
    sur = Surrogate(n, p, 2, seed=n)
    rng = np.random.default_rng(n + p)
    params = (sur.get_parameters() + 0.05 * rng.standard_normal(sur.parameter_count())).astype(np.float32)
    sur.set_parameters(params)
    f32 = lambda v: np.asarray(v, np.float32).astype(np.float64)
    xc, gc = f32(rng.standard_normal((n, p))), f32(rng.standard_normal((n, p)))
    sx, sg = f32(0.5 + rng.random(p)), f32(0.5 + rng.random(p))
    sur.set_normalisation(xc, gc, sx, sg)
    pad = lambda v: np.concatenate([v, np.ones(16 - p)])
    oracle_params = [w.astype(np.float64) for w in split_parameters(params, n)]
    x = datagen.normals(11, 1, n * p).reshape(n, p)
    g = 3.0 * datagen.normals(11, 2, n * p).reshape(n, p)
    loss, grad = sur.loss_gradient(x, g)
    loss_o, grads_o = mo.forward_backward(oracle_params, x, g, xc, gc, pad(sx), pad(sg), p, bf16=True)
    # BF16 activations round to either side where the accumulation order
    # differs: 2^-9 of single values, far less in the norm of a block
    assert abs(loss - loss_o) <= 1e-4 * loss_o
    for name, got, ref in zip(["W1", "b1", "W2", "b2", "W3", "b3", "E"], split_parameters(grad, n), grads_o):
        assert _rel(got, ref) <= 2.0 ** -9, (name, _rel(got, ref))
    ref = mo.predict(oracle_params, x, xc, gc, pad(sx), pad(sg), p, bf16=True)
    assert _rel(sur.predict(x) - gc, ref - gc) <= 2.0 ** -9
    sur.close()


@pytest.mark.parametrize("n,p", [(40, 3), (1100, 5)])
def test_update_leaves_weight_copies_of_its_parameters(n, p):
    sur = Surrogate(n, p, 3, seed=4)
    for k in range(3):
        x = datagen.normals(20 + k, 1, n * p).reshape(n, p)
        sur.add_snapshot(x, -2.0 * x + 0.1 * datagen.normals(20 + k, 2, n * p).reshape(n, p))
    before = sur.get_parameters()
    loss = sur.train(2, 1e-3)
    params = sur.get_parameters()
    assert np.isfinite(loss) and np.all(np.isfinite(params)) and np.any(params != before)
    x = datagen.normals(30, 1, n * p).reshape(n, p)
    trained = sur.predict(x)
    sur.set_parameters(params)  # packs the copies from the parameters
    np.testing.assert_array_equal(sur.predict(x), trained)
    sur.close()
