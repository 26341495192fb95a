"""Small instances walked by several wavefronts per tile: parity with the
oracle and the batched launch's bits at the edges of the rule that chooses
them (1024 tiles; FP64: 512 for untruncated asymmetric observations, 768 for
P > 12), of their workgroups (one tile per workgroup up to 256 tiles, up to
four beyond) and of the tiles (ragged and single blocks)."""
import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.batch import MultiDimensionalScalingBatch
from massivemds_amd.engine import Flags, MultiDimensionalScaling

pytestmark = pytest.mark.gpu


def _data(n, p, asymmetric, seed):
    delta = datagen.euclid10(n, seed=seed, noise_sd=0.2, missing=0.1)
    if asymmetric:
        delta = np.abs(delta + 0.05 * datagen.normals(seed, 9, n * n).reshape(n, n))
        np.fill_diagonal(delta, 0.0)
    return delta, datagen.locations(n, p, seed=seed + 1)


# n, p, fp32, truncated, asymmetric
CASES = [
    (2, 2, False, True, False), (64, 2, False, True, True), (65, 3, False, False, False),
    (1408, 2, False, True, False), (1409, 2, False, True, False),    # 253, 276 tiles: one, two per workgroup
    (2049, 5, False, True, False),                                   # 561: three (the last workgroup not full)
    (2816, 2, False, True, False), (2817, 2, False, True, False),    # 990, 1035: split, whole
    (1984, 3, False, False, True), (1985, 3, False, False, True),    # 496, 528: split, whole
    (2816, 2, False, False, True),                                   # whole, four wavefronts per workgroup
    (2432, 16, False, True, False), (2433, 16, False, True, False),  # 741, 780: split, whole
    (700, 8, False, True, True), (700, 10, False, False, False),
    (90, 2, True, True, False), (1409, 10, True, True, False), (2816, 2, True, False, True),
    (2817, 5, True, True, True), (700, 16, True, True, False),
]


@pytest.mark.parametrize("n,p,fp32,truncated,asymmetric", CASES)
def test_split_walk(oracle, n, p, fp32, truncated, asymmetric):
    print(f"split walk n={n} p={p} fp32={fp32} truncated={truncated} asymmetric={asymmetric}", flush=True)
    tau = 1.3
    delta, x = _data(n, p, asymmetric, 5 + n)
    flags = Flags.OPENCL | (Flags.LEFT_TRUNCATION if truncated else 0) | (Flags.FLOAT if fp32 else 0)
    with MultiDimensionalScaling(p, n, flags, 0) as e:
        e.setPairwiseData(delta)
        e.updateLocations(-1, x)
        e.setParameters([tau])
        s = e.getSumOfIncrements()  # the likelihood pass by itself
        g = e.getLogLikelihoodGradient().reshape(n, p)
        e.makeDirty()
        np.testing.assert_array_equal(e.getLogLikelihoodGradient().reshape(n, p), g)
        assert e.getSumOfIncrements() == s  # now from the fused pass
    s_ref = oracle.sum_of_increments(delta, x, tau, truncated)
    g_ref = oracle.gradient(delta, x, tau, truncated)
    tol_s, tol_g = (1e-6, 1e-5) if fp32 else (1e-12, 1e-12)
    assert abs(s - s_ref) <= tol_s * abs(s_ref)
    assert np.max(np.abs(g - g_ref)) <= tol_g * np.max(np.abs(g_ref))
    if p <= 10:  # the batched launch, one wavefront per tile, adds in the same groups
        b = MultiDimensionalScalingBatch([p, p], [n, 50], flags, 0)
        small = _data(50, p, False, 3)
        for k, (d, y) in enumerate([(delta, x), small]):
            b.setPairwiseData(k, d)
            b.updateLocations(k, y)
            b.setParameters(k, [tau])
        for strategy in (0, 1):
            b.set_config(4, 4, 1, strategy)
            b.evaluate()
            assert b.sums()[0] == s, strategy
            np.testing.assert_array_equal(b.gradient(0), g)
        b.close()
