"""2-D blocks joined by inner faces: the steps whose later stages work on the
plane alone, with the copies of the ring near the faces that the exchange reads,
against the oracle; and batched, block by block and as a replayed graph:
identical bytes.  Two steps at 1e-11, as for single 2-D blocks (six stages, each
with the dq error and a Newton tolerance of 1e-10 K in 300 K)."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel

pytestmark = pytest.mark.gpu


def make(name, n_spec, rk=3, mixed=False):
    if name == "two":
        case = cases.split_i(cases.c1(34, 17, 1, n_spec=n_spec, perturb=0.2, rk_stages=rk), 15)
    else:  # 3 x 2 blocks, four meeting in a point; thin ones too
        case = cases.lattice([[19, 4, 16], [8, 21], [1]], n_spec=n_spec, rk_stages=rk)
    for b in case.blocks:  # no faces along k
        b.bc = [f for f in b.bc if f[0][0] == f[1][0] or f[0][1] == f[1][1]]
    if mixed:
        case.params["precision"] = abi.MIXED
    return case


@pytest.mark.parametrize("rk", [1, 3])
@pytest.mark.parametrize("n_spec", [0, 2])
@pytest.mark.parametrize("name", ["two", "six"])
def test_steps_against_the_oracle(name, n_spec, rk):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    case = make(name, n_spec, rk)
    print(f"[plane blocks] {name} ns={n_spec} rk={rk}", flush=True)
    g, o = Solver(case), Oracle(case)
    for c in (g, o):
        c.upload_initial()
        c.init_conservative()
        c.step(2)
    for b in range(len(case.blocks)):
        for sel in (abi.CV, abi.BV, abi.PROPS) + ((abi.YK,) if n_spec else ()):
            assert_close_sel(sel, g.download(b, sel), o.download(b, sel), 1e-11, f"{name} block {b} selector {sel}")
    assert g.check() == (0, 0)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n_spec", [0, 2])
def test_execution_modes_identical(n_spec, mixed):
    from combustioncodegpu_amd.lib import Solver
    case = make("six", n_spec, mixed=mixed)
    runs = [Solver(case) for _ in range(3)]
    for g, (batched, graph) in zip(runs, ((True, False), (False, False), (True, True))):
        g.set_execution(batched=batched, graph=graph)
        g.upload_initial()
        g.init_conservative()
    for rep in range(3):
        print(f"[plane blocks] modes ns={n_spec} mixed={mixed} step {rep}", flush=True)
        for g in runs:
            g.step(1)
        for b in range(len(case.blocks)):
            for sel in (abi.CV, abi.BV, abi.PROPS):
                ref = runs[0].download(b, sel)
                for g in runs[1:]:
                    assert np.array_equal(g.download(b, sel), ref), f"block {b} selector {sel}"
