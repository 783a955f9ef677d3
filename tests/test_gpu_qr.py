"""The thin QR at the edges of its register kernels (64, 128, 256 and 576 rows;
8, 16, 24 and 64 columns), in place and out of place, against a Householder QR
in numpy with the same sign (R's diagonal is -sign(Re alpha) times a norm)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import qutree_amd as Q
import test_oracle_apply_fit as TA
from qutree_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 2), (9, 9), (63, 8), (64, 9), (64, 24), (64, 25), (64, 64), (65, 16), (128, 24), (129, 24),
          (128, 25), (65, 64), (256, 16), (256, 17), (256, 64), (257, 24), (257, 25), (576, 1), (576, 24), (577, 24)]


def _householder(A):
    """LAPACK's convention: beta = -sign(Re alpha) |x|, Q = H_1 ... H_n."""
    A = A.astype(np.complex128).copy()
    m, n = A.shape
    vs = []
    for j in range(n):
        x = A[j:, j]
        alpha, s = x[0], np.sum(np.abs(x[1:]) ** 2)
        v = np.zeros(m, dtype=complex)
        v[j] = 1.0
        if s == 0.0 and alpha.imag == 0.0:
            vs.append((v, 0.0))
            continue
        beta = -np.copysign(np.sqrt(abs(alpha) ** 2 + s), alpha.real)
        tau = (beta - alpha) / beta
        v[j + 1:] = x[1:] / (alpha - beta)
        A[:, j:] -= np.outer(np.conj(tau) * v, v.conj() @ A[:, j:])
        vs.append((v, tau))
    q = np.eye(m, n, dtype=complex)
    for v, tau in reversed(vs):
        q -= np.outer(tau * v, v.conj() @ q)
    return q


def _qr(X, inplace):
    L = Q.lib()
    L.qtg_qr_batch_z.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_int64, C.c_void_p]
    count, m, n = X.shape
    a = Q.DeviceBuffer.from_array(np.ascontiguousarray(X.transpose(0, 2, 1)).ravel())
    q = a if inplace else Q.DeviceBuffer(a.nbytes)
    Q.check(L.qtg_qr_batch_z(a.ptr, q.ptr, m, n, count, None))
    return q.download(np.complex128).reshape(count, n, m).transpose(0, 2, 1)


@pytest.mark.parametrize("m,n", SHAPES)
def test_qr_at_the_edges_of_the_register_kernels(m, n):
    print(f"case qr edges m={m} n={n}", flush=True)
    rng = np.random.default_rng(m * 100 + n)
    X = rng.normal(size=(3, m, n)) + 1j * rng.normal(size=(3, m, n))
    X[1, :, n // 2] = 0.0  # its reflector is the identity
    X[2] = X[2].real
    for inplace in (False, True):
        got = _qr(X, inplace)
        for i in range(3):
            # n reflectors on columns of norm 1: at most a few n eps an element
            assert np.max(np.abs(got[i].conj().T @ got[i] - np.eye(n))) < 1e-15 * (20 + 4 * n)
            if i == 1:
                # the zero column's direction is arbitrary; the others span A
                r = got[i].conj().T @ X[i]
                assert np.max(np.abs(got[i] @ r - X[i])) < 1e-14 * (20 + n)
                continue
            # a square matrix's columns depend on A with its condition number
            tol = 2e-15 * n * max(10.0, np.linalg.cond(X[i]))
            assert np.max(np.abs(got[i] - _householder(X[i]))) < tol


def test_a_column_of_nan_leaves_the_columns_before_it():
    print("case qr nan column", flush=True)
    rng = np.random.default_rng(5)
    X = rng.normal(size=(1, 70, 20)) + 1j * rng.normal(size=(1, 70, 20))
    X[0, 3, 11] = np.nan
    got = _qr(X, False)[0]
    # a column of Q depends on the columns of A up to it and on no later one
    assert np.max(np.abs(got[:, :11] - _householder(X[0, :, :11]))) < 2e-15 * 20 * 10
    assert np.isnan(got[:, 11]).any()


@pytest.mark.parametrize("spf", [[4, 16, 18], [8, 20, 28], [5, 24, 24]])
def test_fit_start_at_the_edges_of_the_device_orthonormalisation(spf):
    """The fit's random start (Gram-Schmidt in the oracle): square nodes, 256
    rows, 576 x 24, and nodes (400 x 28, a top node of 784) left to the host."""
    print(f"case fit start {spf}", flush=True)
    text, H = W.balanced_tree_text(8, spf[0] + 1, spf), TA.contraction_sop(8, spf[0] + 1, 4, 2)
    om = O.OracleModel(text, H)
    psi = om.fill_random(21, delta_lowest=False)
    ref = om.apply_fit(psi, 5, 1)
    got = Q.ApplyFit(Q.Engine(text, H)).run(psi, 5, 1)
    # both starts are the exact one up to eps times a random node's condition
    # number (square ones: some 1e2), and one iteration is a product and a QR
    assert abs(got["fidelities"][0] / ref["fidelities"][0] - 1.0) < 1e-11
    ov = om.overlap(ref["psi"], got["psi"])
    n2 = om.overlap(ref["psi"], ref["psi"]).real * om.overlap(got["psi"], got["psi"]).real
    assert abs(1.0 - abs(ov) ** 2 / n2) < 1e-11
    top = om.nnodes - 1
    assert np.max(np.abs(om.node_tensor(got["psi"], top) - om.node_tensor(ref["psi"], top))) < 1e-11
