"""What kernels and the host exchange through pinned memory without a stream
wait: location uploads (a kernel reads the staging buffer), gradient rows that
arrive after the sum, and single-location moves whose row the next launch
carries.  Sequences of store, move, read, restore and accept are checked
against the serial FP64 oracle at the locations the reference's rules keep
(src/NewMultiDimensionalScaling.hpp:134-255): FP64 within 1e-12 relative, FP32
within 2e-6 on the sum and 2e-6 of the largest entry on the gradient."""
import numpy as np
import pytest
import torch

from massivemds_amd import datagen
from massivemds_amd.batch import MultiDimensionalScalingBatch
from massivemds_amd.engine import Flags, MultiDimensionalScaling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p,fp32,truncated", [
    (2, 1, False, True), (64, 2, False, True), (65, 7, False, False), (300, 3, True, True), (513, 2, False, True)])
def test_sequences_of_moves_and_states(oracle, n, p, fp32, truncated):
    print(f"exchange n={n} p={p} fp32={fp32} T={truncated}", flush=True)
    tau, tol = 1.7, 2e-6 if fp32 else 1e-12
    delta = datagen.euclid10(n, 31, 0.1, 0.05)
    x = datagen.locations(n, p, 32)
    e = MultiDimensionalScaling(p, n, Flags.OPENCL | (Flags.LEFT_TRUNCATION if truncated else 0)
                                | (Flags.FLOAT if fp32 else 0), 0)
    e.setPairwiseData(delta)
    e.setParameters([tau])
    e.updateLocations(-1, x)

    def check_sum():
        ref = oracle.sum_of_increments(delta, x, tau, truncated)
        assert abs(e.getSumOfIncrements() - ref) <= tol * max(abs(ref), 1.0)

    def check_gradient():
        g = e.getLogLikelihoodGradient().reshape(n, p)
        ref = oracle.gradient(delta, x, tau, truncated)
        assert np.max(np.abs(g - ref)) <= tol * np.max(np.abs(ref))

    check_sum()
    e.storeState()
    stored = x.copy()
    rng = np.random.default_rng(n * 7 + p)
    for step in range(120):
        what = rng.integers(0, 8)
        if what < 4:  # one row, the last one moved among them
            i = int(rng.integers(0, n)) if what else n - 1
            x[i] += 0.3 * rng.standard_normal(p)
            e.updateLocations(i, x[i])
            if what != 1:
                check_sum()
        elif what == 4:
            x = datagen.locations(n, p, 100 + step)
            e.updateLocations(-1, x)
            # the sum now or the rows of this pass later, after other work
            if rng.random() < 0.7:
                check_sum()
        elif what == 5:
            check_gradient()
        elif what == 6:
            check_sum()
            e.storeState()
            stored = x.copy()
            # moved and given up at once: neither copy of the state may change
            if rng.random() < 0.5:
                e.updateLocations(0, x[0] + 1.0)
                e.getSumOfIncrements()
                e.restoreState()
                check_gradient()
        else:
            e.restoreState()
            x = stored.copy()
            check_sum()
            if rng.random() < 0.5:
                check_gradient()
    check_sum()
    check_gradient()
    e.close()


@pytest.mark.parametrize("n,p", [(63, 1), (1025, 16), (8256, 16)])
def test_uploads_give_the_device_resident_result(n, p):
    """Sizes below one workgroup of the upload, at a ragged last one and past
    its largest launch; the same locations handed over on the device."""
    print(f"upload n={n} p={p}", flush=True)
    e = MultiDimensionalScaling(p, n, Flags.OPENCL, 0)
    e.setPairwiseData(np.ones((n, n)))
    e.setParameters([1.3])
    out = torch.empty(1, dtype=torch.float64, device="cuda")
    for k in range(4):  # both staging buffers, and each again
        x = datagen.locations(n, p, 50 + k)
        e.updateLocations(-1, datagen.locations(n, p, 60 + k))
        e.updateLocations(-1, x)
        s = e.getSumOfIncrements()
        at = torch.as_tensor(x, device="cuda").contiguous()
        torch.cuda.synchronize()
        e.evaluate_device_noalloc(at.data_ptr(), out.data_ptr(), None)
        assert float(out) == s
    e.close()


@pytest.mark.parametrize("count,fp32", [(1, False), (2, True), (65, False)])
def test_batch_uploads_and_gradients_in_any_order(count, fp32):
    """One upload and at most two gradient read-backs per evaluation: more
    datasets than one launch of either takes, gradients asked for in any order,
    twice or not at all, locations replaced before and after an evaluation --
    the bits of single-instance calls."""
    print(f"batch exchange count={count} fp32={fp32}", flush=True)
    flags = Flags.OPENCL | Flags.LEFT_TRUNCATION | (Flags.FLOAT if fp32 else 0)
    ns = [1 + (37 * k) % 150 for k in range(count)]
    dims = [(1, 2, 5, 7)[k % 4] for k in range(count)]
    b = MultiDimensionalScalingBatch(dims, ns, flags, 0)
    engines = []
    for k, (n, p) in enumerate(zip(ns, dims)):
        delta = datagen.euclid10(n, 70 + k, 0.1, 0.05)
        b.setPairwiseData(k, delta)
        b.setParameters(k, [1.0 + 0.01 * k])
        e = MultiDimensionalScaling(p, n, flags, 0)
        e.setPairwiseData(delta)
        e.setParameters([1.0 + 0.01 * k])
        engines.append(e)
    rng = np.random.default_rng(count)
    at = [None] * count
    for turn in range(5):
        for k in range(count):
            if turn == 0 or rng.random() < 0.6:
                b.updateLocations(k, datagen.locations(ns[k], dims[k], 7))  # replaced before it is used
                at[k] = datagen.locations(ns[k], dims[k], 1000 * turn + k)
                b.updateLocations(k, at[k])
        b.evaluate()
        sums = b.sums()
        wanted = rng.integers(0, count, (0, 1, count, 2 * count, 2)[turn])
        for k, e in enumerate(engines):
            e.updateLocations(-1, at[k])
            assert e.getSumOfIncrements() == sums[k]
        for k in wanted:
            want = engines[k].getLogLikelihoodGradient().reshape(ns[k], dims[k])
            assert np.array_equal(b.gradient(int(k)), want, equal_nan=True), (turn, k)
    b.close()
    for e in engines:
        e.close()
