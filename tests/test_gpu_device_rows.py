"""Gradient rows that stay on the device: written by the reduce without the pass
through LDS that rows for the host take, the same additions.  Dimensions below,
at and past its eight wavefronts, column blocks in groups of four and left over;
equal, bit for bit, to what the host reads."""
import pytest
import torch

import numpy as np

from massivemds_amd import datagen
from massivemds_amd.engine import Flags, MultiDimensionalScaling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p,fp32", [
    (1, 1, False), (64, 2, False), (65, 7, True), (513, 8, False), (2049, 9, False), (2113, 16, True), (2600, 3, False)])
def test_device_rows_equal_host_rows(n, p, fp32):
    print(f"device rows n={n} p={p} fp32={fp32}", flush=True)
    e = MultiDimensionalScaling(p, n, Flags.OPENCL | Flags.LEFT_TRUNCATION | (Flags.FLOAT if fp32 else 0), 0)
    e.setPairwiseData(datagen.euclid10(n, 21, 0.1, 0.05))
    e.setParameters([1.4])
    x = datagen.locations(n, p, 22)
    e.updateLocations(-1, x)
    s, g = e.getSumOfIncrements(), e.getLogLikelihoodGradient()
    at = torch.as_tensor(x, device="cuda").contiguous()
    total = torch.empty(1, dtype=torch.float64, device="cuda")
    rows = torch.full((n * p + 1,), -7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    e.evaluate_device_noalloc(at.data_ptr(), total.data_ptr(), rows.data_ptr())
    assert float(total) == s
    assert np.array_equal(rows[:-1].cpu().numpy(), g, equal_nan=True)
    assert float(rows[-1]) == -7.0  # nothing past the last row
    e.evaluate_async(True)  # into the engine's own buffer, copied when read
    assert np.array_equal(e.getLogLikelihoodGradient(), g, equal_nan=True)
    e.close()
