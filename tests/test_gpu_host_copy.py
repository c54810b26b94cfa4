"""Downloads on both sides of the size from which they run through pinned pieces
on several threads (8 MiB), with ragged last pieces, and from two threads at
once: the bytes that were uploaded."""
import threading

import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases

pytestmark = pytest.mark.gpu


# cv of 14 variables over the padded points: 4.7, 7.88, 8.06, 24.4 and 81.8 MiB
@pytest.mark.parametrize("size", [(40, 32, 24), (45, 39, 31), (47, 36, 33), (96, 48, 40), (131, 77, 66)])
def test_roundtrip(size):
    from combustioncodegpu_amd.lib import Solver
    case = cases.c1(*size, n_spec=9)
    g = Solver(case)
    shp = case.blocks[0].padded_shape
    print(f"[copy] {size} {14 * np.prod(shp) * 8 / 2**20:.2f} MiB", flush=True)
    rng = np.random.default_rng(1)
    cv, bv, yk = (rng.standard_normal((n,) + shp) for n in (14, 6, 9))
    g.upload_state(0, cv, bv, yk)
    for _ in range(2):
        for sel, ref in ((abi.CV, cv), (abi.BV, bv), (abi.YK, yk)):
            assert np.array_equal(g.download(0, sel), ref)
    got = [None, None]

    def fetch(n, sel):
        got[n] = g.download(0, sel)

    threads = [threading.Thread(target=fetch, args=a) for a in ((0, abi.CV), (1, abi.YK))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert np.array_equal(got[0], cv) and np.array_equal(got[1], yk)
    g.close()
