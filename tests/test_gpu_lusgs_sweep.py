"""The LU-SGS sweeps at the edges of their patches (4 x 4 columns), of their
staged chunks (8 steps) and of their hand-over (blocks thinner than a patch,
with and without patches after them), against the oracle's increment at the
FP64 step bar of 1e-12; and many patches of several blocks per launch, block by
block and as a replayed graph: identical bytes."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel
from tests.test_gpu_lusgs import lusgs, pair

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (4, 4, 4), (5, 5, 5), (8, 4, 9), (17, 6, 5), (9, 33, 4), (40, 3, 13), (3, 21, 18)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2, 9])
def test_increment(size, n_spec):
    print(f"[sweep] {size} ns={n_spec}", flush=True)
    o, g = pair(lusgs(cases.c1(*size, n_spec=n_spec, perturb=0.2, rk_stages=1)))
    for c in (o, g):
        c.rhs()
        c.time_step(False)
        c.lusgs()
    assert_close_sel(abi.DQ, g.download(0, abi.DQ), o.download(0, abi.DQ), 1e-12, f"{size} ns={n_spec}")
    assert g.check()[0] == 0


def test_many_patches_identical():
    from combustioncodegpu_amd.lib import Solver
    case = lusgs(cases.lattice([[37, 21], [50, 9], [18, 41]], n_spec=2, rk_stages=1))
    nb = len(case.blocks)
    runs = [Solver(case) for _ in range(3)]
    for g, (batched, graph) in zip(runs, ((True, False), (False, False), (True, True))):
        g.set_execution(batched=batched, graph=graph)
        g.upload_initial()
        g.init_conservative()
    for rep in range(3):
        print(f"[sweep] lattice step {rep}", flush=True)
        for g in runs:
            g.step(1)
        ref = [runs[0].download(b, abi.CV) for b in range(nb)]
        for g in runs[1:]:
            for b in range(nb):
                assert np.array_equal(g.download(b, abi.CV), ref[b])
    for g in runs:
        assert g.check()[0] == 0
