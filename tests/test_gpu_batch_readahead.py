"""A batch's gradients read back one by one, with others ahead of them: any
number, in any order, asked for again, across passes at other locations, over
more bytes than one read-ahead takes (160 KB of the largest against 256) --
always the rows of the last pass, bit for bit those of single instances."""
import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.batch import MultiDimensionalScalingBatch
from massivemds_amd.engine import Flags, MultiDimensionalScaling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,dims", [
    ([2000, 30, 1500, 2000, 64, 1, 1200, 2000, 900, 1700, 5, 2000], [10, 2, 8, 10, 5, 1, 10, 9, 2, 10, 3, 10]),
    ([40] * 70, [2] * 70),  # more than one launch's entries
    ([300], [3])])
def test_gradients_in_any_order_and_number(ns, dims):
    print(f"read-ahead ns={ns[:4]}.. count={len(ns)}", flush=True)
    flags, count = Flags.OPENCL | Flags.LEFT_TRUNCATION | Flags.FLOAT, len(ns)
    b = MultiDimensionalScalingBatch(dims, ns, flags, 0)
    at = [[datagen.locations(n, p, 100 * s + k) for k, (n, p) in enumerate(zip(ns, dims))] for s in range(2)]
    want = [[], []]
    for k, (n, p) in enumerate(zip(ns, dims)):
        delta = datagen.euclid10(n, 30 + k % 5, 0.1, 0.05)
        b.setPairwiseData(k, delta)
        b.setParameters(k, [1.3])
        e = MultiDimensionalScaling(p, n, flags, 0)
        e.setPairwiseData(delta)
        e.setParameters([1.3])
        for s in range(2):
            e.updateLocations(-1, at[s][k])
            want[s].append(e.getLogLikelihoodGradient().reshape(n, p))
        e.close()
    rng = np.random.default_rng(count)
    orders = [range(count), reversed(range(count)), [count - 1], [0, count - 1], [count // 2] * 3]
    orders += [rng.integers(0, count, m) for m in (3, 5, count, 3 * count)]
    for turn, order in enumerate(orders):
        s = turn % 2
        for k in range(count):
            b.updateLocations(k, at[s][k])
        b.evaluate()
        for k in order:
            assert np.array_equal(b.gradient(int(k)), want[s][int(k)], equal_nan=True), (turn, k)
    b.close()
