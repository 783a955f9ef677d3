"""The CMF integrator's per-node kernels at the edges of their choices, one
short step against the oracle: node tensors of 1024 elements (where the
products take more threads) and just below, more than 16 SPFs (square roots by
eigendecomposition, node errors from memory), and a node beyond the difference
that a tick keeps in LDS (8192 elements), also with orthogonal() in memory."""
import numpy as np
import pytest

import oracle_lib as O
import qutree_amd as Q
from qutree_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,spf", [(2, [1, 1, 1]), (9, [8, 16, 4]), (9, [8, 15, 4]), (6, [5, 17, 10]),
                                     (6, [5, 24, 16])])
def test_cmf_step_matches_oracle(dim, spf):
    print(f"case cmf edges {dim} {spf}", flush=True)
    text, H = W.balanced_tree_text(8, dim, spf), W.coupled_ho(8, 5, c_sigma=0.1)
    om = O.OracleModel(text, H)
    psi = om.fill_random(11, delta_lowest=False)
    ref = om.cmf(psi, 0.0, 0.02, 0.02, 0.02)
    got = Q.CMF(Q.Engine(text, H)).integrate(psi, 0.0, 0.02, 0.02, 0.02)
    de = np.max(np.abs(got["energies"] - ref["energies"]) / np.abs(ref["energies"]))
    da = np.max(np.abs(got["autocorr"] - ref["autocorr"]))
    top = om.nnodes - 1
    dt = np.max(np.abs(om.node_tensor(got["psi"], top) - om.node_tensor(ref["psi"], top)))
    om.build(psi)
    cond = max(np.linalg.cond(om.rho(k)) for k in range(top))
    worst = 0.0  # SPFs, weighted by the state's density (rho^-1 amplifies what it cannot see)
    om.build(ref["psi"])
    for k in range(top):
        A, B = om.node_tensor(ref["psi"], k), om.node_tensor(got["psi"], k)
        n = A.shape[-1]
        D, rho = (A - B).reshape(-1, n, order="F"), om.rho(k)
        worst = max(worst, np.sqrt(abs(np.trace(D.conj().T @ D @ rho.T).real / np.trace(rho).real)))
    print(f"  steps {got['steps']}/{ref['steps']} derivs {got['derivs']}/{ref['derivs']} dE {de:.1e} da {da:.1e} "
          f"top {dt:.1e} nodes {worst:.1e}", flush=True)
    assert got["steps"] == ref["steps"] and got["derivs"] == ref["derivs"]
    # some 1e2 derivatives of eps each, on values of order one; the state moves
    # by eps times the condition of rho (7e3 for 24 SPFs in 25 grid points),
    # whose inverse multiplies the rounded derivative of the SPFs
    tol = max(1e-12, 4.0 * np.finfo(float).eps * cond)
    assert de < 1e-12 and da < tol
    assert dt < max(1e-11, tol) and worst < max(1e-11, tol)
