"""The 2-D RHS and the 2-D step at the sizes where they can go wrong.

One workgroup owns 16 x 15 (variant 1: 32 x 7) cells, so the cases sit on both
sides of those tile edges, down to the smallest block.  The uploaded ghost
planes along k differ from the plane: the first RHS has to read them, while
the stages within a step work on the plane alone, and a step has to leave
every plane of the primitives and the properties as the oracle does.  FP64:
dq at the step bar of 1e-12, two steps at 1e-11 (six stages, each with the dq
error and a Newton tolerance of 1e-10 K in 300 K); mixed dq at 1e-4 as in 3-D.
"""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (16, 15), (17, 16), (15, 31), (33, 7), (32, 8), (70, 37)]


def case2d(mx, my, **kw):
    c = cases.c1(mx, my, 1, perturb=0.2, **kw)
    c.blocks[0].bc = c.blocks[0].bc[:4]  # no faces along k
    return c


def run(case, variant, steps):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    out = []
    g = Solver(case)
    g.set_rhs_variant(variant)
    fp64 = dict(case.params)
    fp64.pop("precision", None)
    case.params = fp64
    for c in (g, Oracle(case)):
        c.upload_initial()
        c.init_conservative()
        if steps:
            c.step(steps)
        else:
            c.rhs()
        out.append(c)
    return out


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec,variant", [(0, 0), (2, 0), (9, 0), (0, 1), (9, 1)])
def test_rhs(size, n_spec, variant):
    print(f"[plane] rhs {size} ns={n_spec} variant {variant}", flush=True)
    g, o = run(case2d(*size, n_spec=n_spec), variant, 0)
    assert_close_sel(abi.DQ, g.download(0, abi.DQ), o.download(0, abi.DQ), 1e-12, f"{size}")


@pytest.mark.parametrize("kw", [dict(limiter=0), dict(reconstruction=1), dict(viscous=0), dict(quirks=0),
                                dict(t_low=700.0), dict(n_spec=1), dict(n_spec=5, limiter=0, quirks=0)])
def test_schemes(kw):
    print(f"[plane] {kw}", flush=True)
    g, o = run(case2d(18, 17, **kw), 0, 0)
    assert_close_sel(abi.DQ, g.download(0, abi.DQ), o.download(0, abi.DQ), 1e-12, str(kw))


@pytest.mark.parametrize("n_spec", [0, 9])
def test_rhs_mixed(n_spec):
    case = case2d(33, 17, n_spec=n_spec)
    case.params["precision"] = abi.MIXED
    print(f"[plane] mixed ns={n_spec}", flush=True)
    g, o = run(case, 0, 0)
    assert_close_sel(abi.DQ, g.download(0, abi.DQ), o.download(0, abi.DQ), 1e-4, "mixed")


@pytest.mark.parametrize("rk", [1, 3])
@pytest.mark.parametrize("size,n_spec", [((17, 16), 0), ((33, 8), 2), ((16, 31), 9)])
def test_steps(size, n_spec, rk):
    print(f"[plane] steps {size} ns={n_spec} rk={rk}", flush=True)
    g, o = run(case2d(*size, n_spec=n_spec, rk_stages=rk), 0, 2)
    for sel in (abi.CV, abi.BV, abi.PROPS) + ((abi.YK,) if n_spec else ()):
        assert_close_sel(sel, g.download(0, sel), o.download(0, sel), 1e-11, f"{size} selector {sel}")


@pytest.mark.parametrize("mixed", [False, True])
def test_step_equals_its_parts(mixed):
    """A step against the same operations called one by one (which work on all
    planes), eager and as a graph, replayed: equal up to the FP rounding of
    differences that are zero, 1e-13 FP64 and 1e-6 mixed."""
    from combustioncodegpu_amd.lib import Solver
    case = case2d(33, 17, n_spec=2)
    if mixed:
        case.params["precision"] = abi.MIXED
    ref, eager, graph = Solver(case), Solver(case), Solver(case)
    graph.set_execution(batched=True, graph=True)
    for s in (ref, eager, graph):
        s.upload_initial()
        s.init_conservative()
    for rep in range(3):
        print(f"[plane] parts mixed={mixed} step {rep}", flush=True)
        ref.store_last_step()
        for stage in range(3):
            ref.rhs()
            if stage == 0:
                ref.time_step(True)
            ref.update(stage)
            ref.apply_bc()
            ref.exchange()
            ref.eliminate_k_gradient()
            ref.update_properties()
        for s in (eager, graph):
            s.step(1)
            for sel in (abi.BV, abi.PROPS):
                assert_close_sel(sel, s.download(0, sel), ref.download(0, sel), 1e-6 if mixed else 1e-13, f"step {rep}")
