"""The exchange in two launches (middles of the inner faces, then the strips
near their edges by components of linked points) against the one-op-at-a-time
loop: identical bytes, whatever the number of blocks that meet at a point and
the extents (faces too small for a middle, ragged lattices, 2-D)."""
import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases

pytestmark = pytest.mark.gpu


def make(name):
    if name == "air2d":
        return cases.split_i(cases.c1(34, 17, 1, n_spec=0), 15)
    sizes = {"ragged": [[13, 16], [9, 21], [12, 7, 18]], "thin": [[4, 3, 5], [6, 3], [5, 4]],
             "wide": [[30, 41], [26], [19, 33]]}[name]
    return cases.lattice(sizes, n_spec=3)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("name", ["ragged", "thin", "wide", "air2d"])
def test_split_exchange_identical(name, mixed):
    from combustioncodegpu_amd.lib import Solver
    case = make(name)
    if mixed:
        case.params["precision"] = abi.MIXED
    print(f"[exchange] {name} mixed={mixed} blocks={[(b.mx, b.my, b.mz) for b in case.blocks]}", flush=True)
    # independent random values in every array: the two sides of a shared layer
    # differ, and no point equals another by coincidence
    rng = np.random.default_rng(3)
    state = [[rng.standard_normal((n,) + b.padded_shape) for n in (case.n_var, 6, max(1, case.n_spec))]
             for b in case.blocks]
    got = []
    for batched in (False, True):
        g = Solver(case)
        g.set_execution(batched=batched)
        for b, (cv, bv, yk) in enumerate(state):
            g.upload_state(b, cv, bv, yk if case.n_spec else None)
        g.exchange()
        n_ops, n_lev = g.schedule_info()
        print(f"[exchange] batched={batched} ops {n_ops} launches {n_lev}", flush=True)
        sels = (abi.CV, abi.BV) + ((abi.YK,) if case.n_spec and not mixed else ())
        got.append([g.download(b, s) for b in range(len(case.blocks)) for s in sels])
        g.close()
    changed = 0
    for x, y in zip(*got):
        assert np.array_equal(x, y)
    for b, (cv, _, _) in enumerate(state):
        changed += int((got[0][b * (len(got[0]) // len(state))] != cv).sum())
    assert changed > 0
