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


@pytest.mark.parametrize("delta", [1e-3, 1e-5, 1e-7])
@pytest.mark.parametrize("dim,spf", [(9, [8, 4]), (20, [18, 4]), (21, [19, 64])])  # SPFs over 16; a node beyond LDS
def test_orthogonal_of_nearly_dependent_columns(dim, spf, delta):
    """orthogonal() alone (phase 0: the integrator moves nothing) on nodes
    whose columns lie within delta of the span of others.  All overlaps of a
    column are taken before it is updated where the reference updates after
    each; both iterate until they vanish.  Every node has to end orthonormal
    to the iteration's own 1e-12, and a bottom node's columns where the
    oracle's are: a direction left over at delta carries rounding / delta.
    (delta^2 above rounding: below, the Gram matrix that the integrator's
    first derivative solves with is singular.)"""
    print(f"case orthogonal dependent {dim} {spf} delta={delta}", flush=True)
    text, H = W.balanced_tree_text(4, dim, spf), W.coupled_ho(4, 5, c_sigma=0.1)
    om = O.OracleModel(text, H)
    psi = om.fill_random(3, delta_lowest=False)
    for nd in om.nodes:
        if nd["parent"] < 0:
            continue
        k = int(nd["dims"][-1])
        X = om.node_tensor(psi, om.nodes.index(nd)).reshape(-1, k, order="F").copy()
        X[:, k - 1] = X[:, 0] + delta * X[:, k - 1]
        if k > 3:
            X[:, 2] = X[:, 1] + delta * X[:, 2]
        psi[nd["off"]:nd["off"] + X.size] = X.ravel(order="F")
    ref = om.orthogonal(psi)
    got = Q.CMF(Q.Engine(text, H)).integrate(psi, 0.0, 1e-2, 1e-2, 1e-2, phase=0.0)["psi"]
    worst = off = 0.0
    for a, nd in enumerate(om.nodes):
        k = int(nd["dims"][-1])
        A, B = (om.node_tensor(p, a).reshape(-1, k, order="F") for p in (ref, got))
        if nd["parent"] >= 0:
            off = max(off, np.max(np.abs(B.conj().T @ B - np.eye(k))))
        if nd["bottom"]:
            worst = max(worst, np.max(np.abs(A - B)))
    print(f"  orthonormal to {off:.1e}, bottom columns {worst:.1e}", flush=True)
    assert off < 4e-12
    # L <= 21 rounding errors in a column of norm delta, on both sides
    assert worst < max(1e-13, 32 * np.finfo(float).eps / delta)
