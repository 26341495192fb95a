"""One batch used from several threads: calls take turns, so every result is
that of whole calls.  One thread replaces an entry's locations by one of two
sets while another evaluates and reads the sums, and others read gradients:
each value read is, bit for bit, that of one of the two sets."""
import threading

import numpy as np
import pytest

from massivemds_amd import datagen
from massivemds_amd.batch import MultiDimensionalScalingBatch
from massivemds_amd.engine import Flags

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [True, False])
def test_updates_passes_and_gradients_from_several_threads(fp32):
    ns, dims = [2000, 1500, 60, 700], [10, 7, 2, 5]
    print(f"batch threads fp32={fp32}", flush=True)
    b = MultiDimensionalScalingBatch(dims, ns, Flags.OPENCL | Flags.LEFT_TRUNCATION | (Flags.FLOAT if fp32 else 0), 0)
    sets = [[datagen.locations(n, p, 10 * s + k) for k, (n, p) in enumerate(zip(ns, dims))] for s in range(2)]
    for k, n in enumerate(ns):
        b.setPairwiseData(k, datagen.euclid10(n, 40 + k, 0.1, 0.05))
        b.setParameters(k, [1.0 + 0.2 * k])
    sums, gradients = [], []
    for s in range(2):
        for k in range(len(ns)):
            b.updateLocations(k, sets[s][k])
        b.evaluate()
        sums.append(b.sums())
        gradients.append([b.gradient(k) for k in range(len(ns))])

    wrong, stop = [], threading.Event()

    def one_of(what, k, value, of):
        if not any(np.array_equal(value, o) for o in of):
            wrong.append((what, k))

    def guarded(f):
        def body():
            try:
                f()
            except Exception as error:  # reported by the test, not by the thread
                wrong.append(error)
            finally:
                stop.set()
        return body

    def updates():
        for turn in range(300):
            if stop.is_set():
                break
            for k in range(len(ns)):
                b.updateLocations(k, sets[(turn >> (k % 3)) % 2][k])

    def passes():
        while not stop.is_set():
            b.evaluate()
            for k, v in enumerate(b.sums()):
                one_of("sum", k, v, [s[k] for s in sums])

    def reads(order):
        def body():
            while not stop.is_set():
                for k in order:
                    one_of("gradient", k, b.gradient(k), [g[k] for g in gradients])
        return body

    threads = [threading.Thread(target=guarded(f)) for f in (updates, passes, reads((0, 1, 2, 3)), reads((3, 0)))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    b.close()
    assert not wrong, wrong[:5]
