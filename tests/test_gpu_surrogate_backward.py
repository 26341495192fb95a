"""The transposed BF16 weight copies that the update kernel leaves, which only
the backward pass reads: after training, a loss gradient is bit for bit that of
copies packed from the same parameters."""
import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.surrogate import Surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p", [(1, 1), (40, 3), (1100, 16)])
def test_backward_copies_follow_the_update(n, p):
    print(f"backward copies n={n} p={p}", flush=True)
    sur = Surrogate(n, p, 3, seed=5)
    for k in range(3):
        x = datagen.normals(20 + k, 1, n * p).reshape(n, p)
        sur.add_snapshot(x, -2.0 * x + 0.1 * datagen.normals(20 + k, 2, n * p).reshape(n, p))
    x = datagen.normals(30, 1, n * p).reshape(n, p)
    g = datagen.normals(30, 2, n * p).reshape(n, p)
    untrained = sur.loss_gradient(x, g)[1]
    sur.train(2, 1e-2)
    loss, grad = sur.loss_gradient(x, g)
    assert np.any(grad != untrained)
    sur.set_parameters(sur.get_parameters())
    again, packed = sur.loss_gradient(x, g)
    assert again == loss
    np.testing.assert_array_equal(packed, grad)
    sur.close()
