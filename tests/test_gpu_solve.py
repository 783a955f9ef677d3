"""The projector solve at the edges of its forms: one, two and three 16-column
tiles (n = 16, 17, 32, 33, 48), row counts off the tile, derivatives written by
the solve and by the launch of their own (more than 32 tiles in the plan), each
with an orthonormal state (one Newton-Schulz step), a slightly perturbed one
(several) and one that eliminates, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
import qutree_amd as Q
import test_gpu_engine as TE
from qutree_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("amp", [0.0, 0.001, 0.3])
@pytest.mark.parametrize("n1,n2", [(5, 16), (13, 16), (17, 17), (20, 32), (23, 33), (20, 48)])
def test_derivative_at_the_edges_of_the_solve(n1, n2, amp):
    print(f"case solve edges {n1} {n2} amp={amp}", flush=True)
    text, H = W.balanced_tree_text(8, n1 + 1, [n1, n2, 7]), W.coupled_ho(8, 5, c_sigma=0.1)
    om = O.OracleModel(text, H)
    psi = om.fill_random(5, delta_lowest=False)
    rng = np.random.default_rng(n2)
    for nd in om.nodes:
        if nd["parent"] < 0:
            continue
        size, k = int(np.prod(nd["dims"])), int(nd["dims"][-1])
        X = psi[nd["off"]:nd["off"] + size].reshape(-1, k, order="F")
        R = rng.normal(size=(k, k)) + 1j * rng.normal(size=(k, k))
        psi[nd["off"]:nd["off"] + size] = (X @ (np.eye(k) + amp * R / np.sqrt(k))).ravel(order="F")
    ref = om.derivative(psi)
    app = om.apply_all(psi)
    eng = Q.Engine(text, H)
    eng.set_psi(psi)
    eng.derivative()
    err = TE.derivative_err(eng, om, eng.get(0), ref, app)
    print(f"  derivative err {err:.3e}", flush=True)
    assert err < 1e-12  # the bound of the engine's other derivative tests
