"""The RHS beside a point that holds NaN, an infinity or a vacuum: what is finite
there stays finite, and the rest of the field does not notice."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.helpers import assert_close_sel

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")
SIZES = [(37, 19, 11), (37, 19, 1)]


def make(size, n_spec, limiter, mixed=False):
    """viscous=0: the point's values enter through the limiter and AUSM+ alone."""
    case = cases.c1(*size, n_spec=n_spec, perturb=0.2, limiter=limiter, viscous=0)
    if size[2] == 1:
        case.blocks[0].bc = case.blocks[0].bc[:4]  # no faces along k
    if mixed:
        case.params["precision"] = abi.MIXED
    return case


def dq_with(ctx, var, value, at):
    """dq of the case with the value in variable var of point at (None: as it is)."""
    ctx.upload_initial()
    ctx.init_conservative()
    bv = ctx.download(0, abi.BV)
    i, j, k = at
    if value is not None:
        bv[var, k + 2, j + 2, i + 2] = value
    ctx.upload_primitive(0, bv, ctx.case.yk0[0])
    if ctx.case.params.get("precision") == abi.MIXED:
        ctx.update_properties()  # makes the FP32 primitives
    ctx.rhs()
    return ctx.download(0, abi.DQ)


def steps_from(size, at):
    """Per cell: the distance to the point along an axis (99 off the axes)."""
    idx = np.meshgrid(*[np.arange(n) for n in size[::-1]], indexing="ij")
    d = [np.abs(a - c) for a, c in zip(idx, at[::-1])]
    return np.where((d[0] > 0).astype(int) + (d[1] > 0) + (d[2] > 0) <= 1, d[0] + d[1] + d[2], 99)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2])
def test_slope_beside_a_broken_point_is_zero(n_spec, size, limiter, mixed):
    """NaN: the cells whose faces touch the point have no dq.  Two steps away only
    the slope of the cell between sees the point: it is 0, as if the point held that
    cell's value.  Everywhere else dq is the same to the bit."""
    from combustioncodegpu_amd.lib import Solver
    at = (18, 9, size[2] // 2)
    g = Solver(make(size, n_spec, limiter, mixed))
    steps = steps_from(size, at)
    for var in (0, 1, 4):
        got = dq_with(g, var, NAN, at)
        print(f"[broken] {size} ns={n_spec} limiter {limiter} mixed={mixed} bv[{var}]=nan", flush=True)
        assert np.array_equal(np.isfinite(got).all(0), steps > 1)
        assert np.array_equal(np.isfinite(got).any(0), steps > 1)
        clean = dq_with(g, var, None, at)
        assert np.array_equal(got[:, steps > 2], clean[:, steps > 2])
        bv = g.download(0, abi.BV)
        for axis in range(3 if size[2] > 1 else 2):
            for side in (-1, 1):
                near, two = list(at), list(at)
                near[axis] += side
                two[axis] += 2 * side
                flat = dq_with(g, var, bv[var, near[2] + 2, near[1] + 2, near[0] + 2], at)
                cell = (slice(None), two[2], two[1], two[0])
                assert np.array_equal(got[cell], flat[cell]), f"bv[{var}] axis {axis} side {side}"


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2])
def test_infinite_density_or_pressure(n_spec, size, limiter, mixed):
    """Finite in the oracle's cells (an infinite difference is limited as any other)."""
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    at = (18, 9, size[2] // 2)
    for var in (0, 4):
        ref = dq_with(Oracle(make(size, n_spec, limiter)), var, INF, at)
        got = dq_with(Solver(make(size, n_spec, limiter, mixed)), var, INF, at)
        print(f"[broken] {size} ns={n_spec} limiter {limiter} mixed={mixed} bv[{var}]=inf", flush=True)
        assert np.array_equal(np.isfinite(got), np.isfinite(ref))


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2, 9])
def test_zero_pressure(n_spec, size, limiter, mixed):
    """A vacuum's sound speed is 0: finite everywhere, and in FP64 the oracle's dq
    at the step bar of 1e-12."""
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    at = (18, 9, size[2] // 2)
    got = dq_with(Solver(make(size, n_spec, limiter, mixed)), 4, 0.0, at)
    print(f"[broken] {size} ns={n_spec} limiter {limiter} mixed={mixed} p=0", flush=True)
    assert np.isfinite(got).all()
    if not mixed:
        ref = dq_with(Oracle(make(size, n_spec, limiter)), 4, 0.0, at)
        assert_close_sel(abi.DQ, got, ref, 1e-12, f"{size}")


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_spec", [0, 2])
def test_infinite_velocity(n_spec, size, limiter, mixed):
    """Not finite in the oracle's cells, those upwind of the point included."""
    from combustioncodegpu_amd.lib import Solver
    from oracle.pyoracle import Oracle
    at = (18, 9, size[2] // 2)
    for var, value in ((1, INF), (2, -INF)):
        ref = dq_with(Oracle(make(size, n_spec, limiter)), var, value, at)
        got = dq_with(Solver(make(size, n_spec, limiter, mixed)), var, value, at)
        print(f"[broken] {size} ns={n_spec} limiter {limiter} mixed={mixed} bv[{var}]={value}", flush=True)
        assert np.array_equal(np.isfinite(got), np.isfinite(ref))
