"""The surrogate's training kernels over species counts and batch sizes: one
workgroup per 32 samples, the gradients of the workgroups summed in quarters of
32 loads and a remainder, the parameters written into the packed operands."""
import os

import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases
from tests.test_gpu_mlp import identity_norm
from tests.test_oracle_mlp import random_params, samples

pytestmark = pytest.mark.gpu


def solver(ns):
    from combustioncodegpu_amd.lib import Solver
    c = cases.c1(12, 10, 8, n_spec=ns)
    c.params["precision"] = abi.MIXED
    return Solver(c)


@pytest.mark.parametrize("ns", [1, 2, 9])
@pytest.mark.parametrize("n", [32, 96, 1056, 4128])
def test_gradient(ns, n):
    """Against the oracle's backpropagation with the same BF16 rounding points:
    the bars of the 256-sample test (5e-3 of the largest gradient, loss 1e-3)."""
    from oracle import pyoracle
    g = solver(ns)
    p = random_params(ns + 2, ns + 2, 31)
    g.mlp_set_params(p, identity_norm())
    x, t = samples(n, ns + 2, ns + 2, 32)
    print(f"[mlp] gradient ns={ns} n={n}", flush=True)
    grad, loss = g.mlp_gradient(x, t)
    le, ge = pyoracle.mlp_loss_grad(p, ns + 2, ns + 2, x, t, emulate=True)
    assert abs(loss - le) <= 1e-3 * le
    assert np.abs(grad - ge).max() / np.abs(ge).max() <= 5e-3


@pytest.mark.parametrize("ns,batch,epochs", [(1, 1056, 8), (2, 32, 1), (5, 4096, 8), (9, 1056, 8)])
def test_training_trajectory(ns, batch, epochs):
    """Some hundred Adam steps (1152 at batch 32) against every 17th parameter,
    the normalisation with the envelope, and the losses of the form with one
    wavefront per 32 samples and the operands packed anew for each step.  The
    same products and sums in the same order: equal up to 1e-6 of the largest."""
    ref = np.load(os.path.join(os.path.dirname(__file__), "trajectories", "mlp_training.npz"))
    g = solver(ns)
    rep = g.mlp_train(n_samples=40960, epochs=epochs, batch=batch, holdout=0.1)
    params, norm = g.mlp_get_params()
    print(f"[mlp] trajectory ns={ns} batch={batch}: {rep}", flush=True)
    for name, got in (("params", params[::17]), ("norm", norm), ("loss", [rep["loss_first"], rep["loss_last"]])):
        r = ref[f"{name}_{ns}_{batch}"]
        assert np.abs(np.asarray(got) - r).max() <= 1e-6 * np.abs(r).max(), name
