"""The marching 3-D RHS at the sizes where it can go wrong.

One workgroup owns 16 x 8 cells and marches through a chunk of k planes, so
the cases sit on both sides of those tile edges, down to the smallest block
(3 points per axis), with every limiter and scheme switch, quirk setting and
compiled species count class, against the oracle's dq.  FP64 at the step bar
of 1e-12; mixed precision at 1e-4 (about 50 roundings of 6e-8 per flux,
amplified up to about 30 times by the difference of two face fluxes).
"""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (16, 8, 4), (17, 9, 5), (15, 7, 3), (33, 8, 9), (16, 17, 10), (48, 3, 6)]


def both(case):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    out = []
    for c in (Solver(case), Oracle(case)):
        c.upload_initial()
        c.init_conservative()
        c.rhs()
        out.append(c)
    return out


def check(case, tol, what):
    print(f"[march] {what}", flush=True)
    g, o = both(case)
    for b in range(len(case.blocks)):
        assert_close_sel(abi.DQ, g.download(b, abi.DQ), o.download(b, abi.DQ), tol, f"{what} block {b}")
    return g


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2, 9])
def test_tile_edges(size, n_spec):
    check(cases.c1(*size, n_spec=n_spec, perturb=0.2), 1e-12, f"{size} ns={n_spec}")


@pytest.mark.parametrize("kw", [dict(limiter=0), dict(reconstruction=1), dict(viscous=0), dict(quirks=0),
                                dict(t_low=700.0), dict(n_spec=1), dict(n_spec=5, limiter=0, quirks=0)])
def test_schemes(kw):
    check(cases.c1(18, 10, 7, perturb=0.25, **kw), 1e-12, str(kw))


@pytest.mark.parametrize("size", [(17, 9, 5), (33, 8, 9)])
@pytest.mark.parametrize("n_spec", [0, 9])
def test_mixed_precision(size, n_spec):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    case = cases.c1(*size, n_spec=n_spec, perturb=0.2)
    print(f"[march] mixed {size} ns={n_spec}", flush=True)
    o = Oracle(case)
    case.params["precision"] = abi.MIXED
    g = Solver(case)
    for c in (g, o):
        c.upload_initial()
        c.init_conservative()
        c.rhs()
    assert_close_sel(abi.DQ, g.download(0, abi.DQ), o.download(0, abi.DQ), 1e-4, f"mixed {size}")


@pytest.mark.parametrize("mixed", [False, True])
def test_chunk_lengths_identical(mixed):
    """Every chunk length, and one block at a time or all, gives the same bytes."""
    from combustioncodegpu_amd.lib import Solver
    case = cases.lattice([[19, 12], [9, 14], [37, 70]], n_spec=3)
    if mixed:
        case.params["precision"] = abi.MIXED
    ref = None
    for v in range(6):
        for batched in (True, False):
            g = Solver(case)
            g.set_execution(batched=batched)
            g.set_rhs_variant(v)
            g.upload_initial()
            g.init_conservative()
            g.rhs()
            got = [g.download(b, abi.DQ) for b in range(len(case.blocks))]
            g.close()
            ref = ref or got
            for b, r in enumerate(ref):
                assert np.array_equal(got[b], r), f"variant {v} batched {batched} block {b}"
