"""FP64 batches with datasets on both sides of the split walk's limit (990 tiles
at N = 2,816, 1,035 one row block further), whose additions follow one order or
the other: one launch of any dimension, one per class, one per class and order.
Whatever the launch, each dataset's result is the single instance's, bit for
bit."""
import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.batch import MultiDimensionalScalingBatch
from massivemds_amd.engine import Flags, MultiDimensionalScaling

pytestmark = pytest.mark.gpu


def _observations(n, seed, asymmetric):
    delta = datagen.euclid10(n, seed, 0.1, 0.05)
    if asymmetric:
        delta = np.abs(delta + 0.05 * datagen.normals(seed, 9, n * n).reshape(n, n))
        np.fill_diagonal(delta, 0.0)
    return delta


@pytest.mark.parametrize("ns,dims,truncated,asymmetric", [
    ([2817, 2816, 65, 1], [2] * 4, True, ()),
    ([2817, 2816, 65, 1], [4] * 4, True, (1, 3)),
    ([2000, 2100, 64], [3] * 3, False, (0, 1)),  # 528 and 561 tiles: two planes without truncation, limit 512
    ([2817, 2816, 65, 1], [5] * 4, True, ()),
    ([2817, 700, 130], [6] * 3, True, (1,)),
    ([2817, 2816, 65, 1], [8] * 4, True, (2,)),
    ([2817, 700, 130], [10] * 3, True, ()),
    ([700, 130], [10, 5], False, ()),
    ([2817, 700, 2817, 130, 400, 2900, 64, 90], [1, 2, 5, 10, 8, 6, 3, 4], True, (0, 3))])
def test_either_order_gives_the_single_instance(ns, dims, truncated, asymmetric):
    print(f"orders ns={ns} dims={dims} T={truncated}", flush=True)
    flags = Flags.OPENCL | (Flags.LEFT_TRUNCATION if truncated else 0)
    b = MultiDimensionalScalingBatch(dims, ns, flags, 0)
    want = []
    for k, (n, p) in enumerate(zip(ns, dims)):
        delta, x, tau = _observations(n, 50 + k, k in asymmetric), datagen.locations(n, p, 90 + k), 1.0 + 0.1 * k
        b.setPairwiseData(k, delta)
        b.setParameters(k, [tau])
        b.updateLocations(k, x)
        e = MultiDimensionalScaling(p, n, flags, 0)
        e.setPairwiseData(delta)
        e.setParameters([tau])
        e.updateLocations(-1, x)
        want.append((e.getSumOfIncrements(), e.getLogLikelihoodGradient().reshape(n, p)))
        e.close()
    for config in ((4, 8, 1, 0), (4, 8, 1, 1), (8, 2, 4, 0), (8, 2, 4, 1), (1, 8, 2, 1)):
        b.set_config(*config)
        b.evaluate()
        sums = b.sums()
        for k, (s, g) in enumerate(want):
            assert sums[k] == s, (config, k)
            assert np.array_equal(b.gradient(k), g, equal_nan=True), (config, k)
    b.close()
