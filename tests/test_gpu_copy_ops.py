"""Ghost fills that only copy and average (outflow conditions, inner faces),
whose arrays are worked on side by side: random independent values in every
array, against the oracle's fill, exactly equal."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n_spec", [0, 1, 9])
@pytest.mark.parametrize("mesh", ["block", "lattice", "plane"])
def test_fill(mesh, n_spec, mixed):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    if mesh == "lattice":
        case = cases.lattice([[13, 18], [9, 16], [12, 7]], n_spec=n_spec)
    else:
        case = cases.c1(19, 11, 1 if mesh == "plane" else 6, n_spec=n_spec)
        if mesh == "plane":
            case.blocks[0].bc = case.blocks[0].bc[:4]
    o = Oracle(case)
    if mixed:
        case.params["precision"] = abi.MIXED
    g = Solver(case)
    print(f"[copy] {mesh} ns={n_spec} mixed={mixed}", flush=True)
    rng = np.random.default_rng(5)
    for b, blk in enumerate(case.blocks):
        cv, bv, yk = (rng.standard_normal((max(1, n),) + blk.padded_shape) for n in (5 + n_spec, 6, n_spec))
        for s in (g, o):
            s.upload_state(b, cv, bv, yk if n_spec else None)
    for s in (g, o):
        s.apply_bc()
        s.exchange()
    for b in range(len(case.blocks)):
        for sel in (abi.CV, abi.BV) + ((abi.YK,) if n_spec and not mixed else ()):
            assert np.array_equal(g.download(b, sel), o.download(b, sel)), f"block {b} selector {sel}"
