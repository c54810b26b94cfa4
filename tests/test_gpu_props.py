"""The FP64 properties where wavefronts are in one NASA-7 range, in both, and
partly below t_low (the general path), against the oracle: 1e-13 (about a
hundred roundings of 1.1e-16 and a handful of one-ulp roots and quotients,
none amplified)."""
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_spec", [1, 2, 3, 5, 9])
@pytest.mark.parametrize("t_low", [200.0, 700.0])
@pytest.mark.parametrize("t", ["field", "cold", "hot"])
def test_properties(n_spec, t_low, t):
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    case = cases.c1(21, 13, 9, n_spec=n_spec, t_low=t_low)
    bv = case.bv0[0]
    if t != "field":  # every temperature on one side of t_mid (1000 K)
        f = bv[5] / bv[5].max()
        new = 720.0 + 200.0 * f if t == "cold" else 1100.0 + 1200.0 * f
        bv[0] *= bv[5] / new
        bv[5] = new
    out = []
    for c in (Solver(case), Oracle(case)):
        c.upload_initial()
        c.init_conservative()
        out.append(c.download(0, abi.PROPS))
    print(f"[props] ns={n_spec} t_low={t_low} {t}", flush=True)
    assert_close_sel(abi.PROPS, out[0], out[1], 1e-13, f"ns={n_spec} t_low={t_low} {t}")
