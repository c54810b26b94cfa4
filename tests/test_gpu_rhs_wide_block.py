"""The marching RHS of a block whose nine metric fields pass 4 GiB, from which the
offsets of a metric row take 64 bits (59.7M padded points in FP64, 119.3M mixed).
The block is long along k and periodic in it: the fields repeat every 24 planes,
x and y do not depend on k, and z = k / 1024 is exact, so that its planes have the
metrics and the stencils of those of a block of three periods, which takes the form
with 32-bit offsets: dq is the same to the bit."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases

pytestmark = pytest.mark.gpu

PERIOD, NX, NY = 24, 60, 60


def block(n_planes, base, mixed):
    h = 1.0 / 1024
    k, j, i = (np.arange(n) for n in (n_planes, NY, NX))
    shape = (n_planes, NY, NX)
    x = (i * h)[None, None, :] + 0.2 * h * np.sin(0.7 * j)[None, :, None]
    y = (j * h)[None, :, None] + 0.2 * h * np.cos(0.5 * i)[None, None, :]
    xyz = [np.ascontiguousarray(np.broadcast_to(a, shape)).ravel() for a in (x, y, (k * h)[:, None, None])]
    blk = cases.BlockSpec(NX, NY, n_planes, *xyz, bc=cases.outflow_all_faces(NX, NY, n_planes))
    params = dict(base.params)
    if mixed:
        params["precision"] = abi.MIXED
    plane = (np.arange(n_planes + 4) - 2) % PERIOD  # of every padded plane
    bv = np.ascontiguousarray(base.bv0[0][:, 2:2 + PERIOD][:, plane])
    return cases.Case("long", params, None, [blk], [], [], [bv], [None])


def dq_of(case):
    from combustioncodegpu_amd.lib import Solver
    g = Solver(case)
    g.upload_initial()
    case.bv0 = None
    g.update_properties()
    g.rhs()
    dq = g.download(0, abi.DQ)
    g.close()
    return dq


@pytest.mark.parametrize("mixed", [False, True])
def test_long_block(mixed):
    n = PERIOD * (1215 if mixed else 609)
    np_ = (NX + 4) * (NY + 4) * (n + 4)
    assert 9 * (4 if mixed else 8) * np_ >= 2 ** 32 and np_ < 2 ** 29
    print(f"[wide] mixed={mixed}: {n} planes, {np_ / 1e6:.1f}M padded points", flush=True)
    base = cases.c1(NX, NY, PERIOD, n_spec=0)
    ref = dq_of(block(3 * PERIOD, base, mixed))
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    got = dq_of(block(n, base, mixed))
    for a in range(0, n, PERIOD):
        r = 0 if a == 0 else (2 * PERIOD if a + PERIOD == n else PERIOD)  # the ends, or between
        assert np.array_equal(got[:, a:a + PERIOD], ref[:, r:r + PERIOD]), f"planes from {a}"
