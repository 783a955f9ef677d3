"""The reduced sweep (engine_reduce.cpp: sums of h-matrices and holes formed
as contractions) against the oracle and against the sweep that forms every
matrix, on trees and Hamiltonians that its choices depend on.  Small plans are
left alone by its rule, so the tests move the line to zero."""
import numpy as np
import pytest

import oracle_lib as O
import qutree_amd as Q
from qutree_amd import workloads as W

pytestmark = pytest.mark.gpu


def _rand(rng, d):
    A = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    return A + A.conj().T


def _three_body(f, d, seed):
    """One-, two- and three-mode products of explicit matrices with complex
    coefficients (not Hermitian as a whole), repeated factors among them."""
    rng = np.random.default_rng(seed)
    H = W.Hamiltonian()
    mats = [_rand(rng, d) for _ in range(4)]
    for i in range(f):
        H.add_term(0.3 + 0.1j * i, [(i, W.FACTOR_MATRIX, mats[i % 4])])
        H.add_term(0.05, [(i, W.FACTOR_X), ((i + 1) % f, W.FACTOR_X), ((i + 3) % f, W.FACTOR_MATRIX, mats[i % 4])])
        H.add_term(0.2j, [(i, W.FACTOR_X2), ((i + 2) % f, W.FACTOR_KIN)])
    H.add_term(0.7, [(j, W.FACTOR_MATRIX, mats[j % 4]) for j in range(f)])
    H.add_term(-0.4, [(0, W.FACTOR_MATRIX, mats[0])])  # the first term's factor again
    return H


def _models():
    return {
        "f4": (W.balanced_tree_text(4, 3, [2, 3]), W.coupled_ho(4, 11, c_sigma=0.1)),
        "cmf8": W.cmf8_model(),
        "quartic16": (W.balanced_tree_text(16, 6, [4, 6, 8, 8]), W.coupled_quartic(16, 5, c_sigma=0.01)),
        "wide8": (W.balanced_tree_text(8, 8, [8, 18, 33]), W.coupled_quartic(8, 5, c_sigma=0.05)),
        "three8": (W.balanced_tree_text(8, 5, [4, 7, 9]), _three_body(8, 5, 3)),
        "one_mode": (W.balanced_tree_text(8, 5, [4, 6, 6]), _one_mode(8)),
    }


def _one_mode(f):
    H = W.Hamiltonian()
    for i in range(f):
        H.add_term(1.0, [(i, W.FACTOR_KIN)])
        H.add_term(0.5 + 0.1 * i, [(i, W.FACTOR_X2)])
    return H


@pytest.fixture
def every_size(monkeypatch):
    monkeypatch.setenv("QTG_REDUCE_MIN_FLOPS", "0")


def _err(x, y):
    return np.linalg.norm(x - y) / np.linalg.norm(y)


@pytest.mark.parametrize("heev_side", [1, 0])
@pytest.mark.parametrize("name", sorted(_models()))
def test_reduced_sweep_matches_oracle(name, heev_side, every_size):
    text, H = _models()[name]
    print(f"case reduced sweep {name} heev_side={heev_side}", flush=True)
    om = O.OracleModel(text, H)
    psi = om.fill_random(5, delta_lowest=False)
    ref = om.derivative(psi)
    # rho^-1 amplifies rounding by the smallest density eigenvalue (wide8: a
    # random 33 x 33 top node): the sweep that forms every matrix shows by how
    # much on this state
    full = Q.Engine(text, H, compress=False)
    full.set_psi(psi)
    full.derivative()
    lim = max(1e-12, 4 * _err(full.get(0), ref))
    eng = Q.Engine(text, H, heev_side=heev_side)
    for _ in range(2):  # captured, then replayed
        eng.set_psi(psi)
        eng.derivative()
        got = eng.get(0)
        print(f"  derivative rel err {_err(got, ref):.2e} limit {lim:.2e}", flush=True)
        assert _err(got, ref) < lim
    e = om.energy(psi)
    assert abs(eng.energy() - e) < 1e-12 * abs(e)


@pytest.mark.parametrize("name", sorted(_models()))
def test_reduced_sweep_matrices_of_single_terms(name, every_size):
    """get_matrix after a reduced sweep forms the terms' matrices at the state
    of the last build, also when the state has been replaced since."""
    text, H = _models()[name]
    print(f"case reduced matrices {name}", flush=True)
    om = O.OracleModel(text, H)
    eng = Q.Engine(text, H)
    for seed in (1, 2):
        psi = om.fill_random(seed, delta_lowest=False)
        om.build(psi)
        eng.set_psi(psi)
        eng.derivative()
        if seed == 2:
            eng.set_psi(om.fill_random(3, delta_lowest=False))
        for l in range(0, H.nterms, max(1, H.nterms // 7)):
            for a in om.sparse_tree(l):
                if a == om.nnodes - 1:
                    continue
                h, g = om.hmat(l, a), om.hole(l, a)
                assert np.max(np.abs(eng.matrix(2, l, a) - h)) < 1e-11 * max(1, np.max(np.abs(h)))
                assert np.max(np.abs(eng.matrix(3, l, a) - g)) < 1e-11 * max(1, np.max(np.abs(g)))


@pytest.mark.parametrize("name", ["f4", "cmf8", "quartic16", "wide8"])
def test_reduced_gradient_and_split_precision(name, every_size):
    text, H = _models()[name]
    print(f"case reduced gradient, split {name}", flush=True)
    om = O.OracleModel(text, H)
    psi = om.fill_random(21, delta_lowest=False)
    ref, e_ref = om.gradient(psi)
    eng = Q.Engine(text, H)
    eng.set_psi(psi)
    got, e = eng.gradient()
    print(f"  gradient rel err {_err(got, ref):.2e}", flush=True)
    assert _err(got, ref) < 1e-11 and abs(e - e_ref) < 1e-12 * abs(e_ref)
    dref = om.derivative(psi)
    full = Q.Engine(text, H, precision=2, compress=False)
    red = Q.Engine(text, H, precision=2)
    errs = []
    for g in (full, red):
        g.set_psi(psi)
        g.derivative()
        errs.append(_err(g.get(0), dref))
        assert abs(g.energy() - e_ref) < 1e-9 * abs(e_ref)
    print(f"  split derivative err, every matrix {errs[0]:.2e} reduced {errs[1]:.2e}", flush=True)
    assert errs[1] < max(4 * errs[0], 1e-7)


@pytest.mark.parametrize("order", ["large_small", "small_large", "large_small_large"])
def test_second_hamiltonian_on_the_other_side_of_the_line(order, monkeypatch):
    """One engine, Hamiltonians whose plans are reduced (large: 0.78 GFLOP of
    single matrices) and are not (small: 0.18) one after the other: buffers
    that only one of the plans has are not used by the other, and every matrix
    is that of the plan at hand."""
    monkeypatch.setenv("QTG_REDUCE_MIN_FLOPS", "5e8")
    print(f"case second hamiltonian {order}", flush=True)
    text = W.balanced_tree_text(16, 6, [5, 14, 20, 20])
    models = {"large": W.coupled_quartic(16, 5, c_sigma=0.01), "small": _one_mode(16)}
    oracles = {k: O.OracleModel(text, H) for k, H in models.items()}
    eng = Q.Engine(text)
    for i, k in enumerate(order.split("_")):
        om, H = oracles[k], models[k]
        eng.set_hamiltonian(H)
        for seed in (i, i + 10):
            psi = om.fill_random(seed, delta_lowest=False)
            ref = om.derivative(psi)
            full = Q.Engine(text, H, compress=False)  # as in test_reduced_sweep_matches_oracle
            full.set_psi(psi)
            full.derivative()
            lim = max(1e-12, 4 * _err(full.get(0), ref))
            eng.set_psi(psi)
            eng.derivative()
            print(f"  {k} derivative rel err {_err(eng.get(0), ref):.2e} limit {lim:.2e}", flush=True)
            assert _err(eng.get(0), ref) < lim
            e = om.energy(psi)
            assert abs(eng.energy() - e) < 1e-12 * abs(e)
            a = om.sparse_tree(0)[0]
            h = om.hmat(0, a)
            assert np.max(np.abs(eng.matrix(2, 0, a) - h)) < 1e-11 * max(1, np.max(np.abs(h)))


def test_matrices_are_those_of_the_last_build_without_an_apply(every_size):
    """build() alone, then another state: no solve or tick waits for the side
    stream, so the build itself has to order its copy of the state (behind
    the eigensolvers of earlier builds there) before what its stream does
    next."""
    text, H = _models()["wide8"]
    print("case matrices after build, then set_psi", flush=True)
    om = O.OracleModel(text, H)
    eng = Q.Engine(text, H)
    states = [om.fill_random(s, delta_lowest=False) for s in range(4)]
    dev = [Q.DeviceBuffer.from_array(p) for p in states]
    term, node = 0, om.sparse_tree(0)[0]

    def check(i):
        om.build(states[i])
        for which, ref in ((2, om.hmat(term, node)), (3, om.hole(term, node))):
            assert np.max(np.abs(eng.matrix(which, term, node) - ref)) < 1e-11 * max(1, np.max(np.abs(ref)))

    for setter in (lambda i: eng.set_psi(states[i]),
                   lambda i: Q.check(Q.lib().qtg_engine_set_psi_device(eng.ptr, dev[i].ptr, None))):
        for rounds in (1, 3):
            for r in range(rounds):  # eigensolvers of the earlier builds still queued
                setter(r)
                eng.build()
            setter(3)
            check(rounds - 1)
    eng.set_psi(states[1])
    eng.build()
    Q.check(Q.lib().qtg_engine_canonicalize(eng.ptr, None, None))  # rewrites the state on the device
    check(1)


def _coherent(f):
    """Pair couplings of one sign: sums that many matrices enter alike."""
    H = W.Hamiltonian()
    for i in range(f):
        H.add_term(1.0, [(i, W.FACTOR_KIN)])
        H.add_term(0.5, [(i, W.FACTOR_X2)])
    for i in range(f):
        for j in range(i):
            H.add_term(0.02, [(i, W.FACTOR_X2), (j, W.FACTOR_X2)])
    return H


def _apply_rms(text, H, precision, seeds):
    """RMS over random states of the relative error of Apply at all nodes
    against the complex128 engine."""
    ref, eng = Q.Engine(text, H), Q.Engine(text, H, precision=precision)
    err = []
    for s in range(seeds):
        psi = ref.fill_random(100 + s, delta_lowest=False)
        for e in (ref, eng):
            e.set_psi(psi)
            e.derivative()
        err.append(_err(eng.get(1), ref.get(1)))
    return float(np.sqrt(np.mean(np.square(err))))


# quartic64: more than 50 GFLOP, where the split form's sums are FP32 products
PRECISION_MODELS = {
    "coherent16": (1, 24, W.balanced_tree_text(16, 8, [4, 6, 6, 6]), _coherent(16)),
    "coherent16_split": (2, 24, W.balanced_tree_text(16, 8, [4, 6, 6, 6]), _coherent(16)),
    "ho16": (1, 24, W.balanced_tree_text(16, 8, [4, 6, 8, 8]), W.coupled_ho(16, 3, one_mode_matrix=True)),
    "quartic64": (1, 4, W.balanced_tree_text(64, 8, [8, 14, 21, 27, 34, 41]), W.coupled_quartic(64, 64)),
    "quartic64_split": (2, 4, W.balanced_tree_text(64, 8, [8, 14, 21, 27, 34, 41]), W.coupled_quartic(64, 64)),
}


@pytest.mark.parametrize("name", sorted(PRECISION_MODELS))
def test_reduced_precision_forms_lose_none_to_the_sums(name, monkeypatch):
    """The FP32 products of a plan that forms every matrix are rounded matrix
    by matrix and summed in FP64; sums formed as contractions must not be
    further off.  0.5 %: the sampling of the RMS over the states."""
    print(f"case reduced precision {name}", flush=True)
    precision, seeds, text, H = PRECISION_MODELS[name]
    err = {}
    for form, line in (("every matrix", "1e30"), ("reduced", "0")):
        monkeypatch.setenv("QTG_REDUCE_MIN_FLOPS", line)
        err[form] = _apply_rms(text, H, precision, seeds)
        print(f"  {form} {err[form]:.3e}", flush=True)
    assert err["reduced"] < 1.005 * err["every matrix"]


@pytest.mark.parametrize("precision,tol", [(0, 1e-11), (1, 1e-4), (2, 1e-4)])
def test_matrices_of_all_terms_in_any_order(precision, tol, every_size):
    """Every term's matrices from the growing groups of get_matrix, asked for
    in random order and after several builds, against the engine that forms
    all of them (complex64 and split: 100 times the rounding of its sums, for the
    amplification along the tree)."""
    text, H = _models()["quartic16"]
    print(f"case matrices of all terms precision={precision}", flush=True)
    full = Q.Engine(text, H, compress=False)
    eng = Q.Engine(text, H, precision=precision)
    rng = np.random.default_rng(5)
    om = O.OracleModel(text, H)
    act = [(l, a) for l in range(H.nterms) for a in om.sparse_tree(l) if a != om.nnodes - 1]
    for seed in (1, 2):
        psi = full.fill_random(seed, delta_lowest=False)
        full.set_psi(psi)
        full.derivative()
        eng.set_psi(psi)
        eng.derivative()
        for i in rng.permutation(len(act)):
            l, a = act[i]
            for which in (2, 3):
                ref = full.matrix(which, l, a)
                assert np.max(np.abs(eng.matrix(which, l, a) - ref)) < tol * max(1, np.max(np.abs(ref)))


def test_refused_hamiltonian_leaves_the_plan_at_hand(every_size):
    """A Hamiltonian with a factor out of range, in its first or a later term,
    is an error; the engine goes on with the one it has, matrices of single
    terms included (formed from its terms on demand)."""
    text, H = _models()["quartic16"]
    print("case refused hamiltonian", flush=True)
    om = O.OracleModel(text, H)
    eng = Q.Engine(text, H)
    psi = om.fill_random(1, delta_lowest=False)
    om.build(psi)
    ref = om.derivative(psi)
    act = [(l, a) for l in range(H.nterms) for a in om.sparse_tree(l) if a != om.nnodes - 1]
    for first in (True, False):
        bad = W.Hamiltonian()
        if not first:
            bad.add_term(1.0, [(0, W.FACTOR_X2)])
        bad.add_term(1.0, [(99, W.FACTOR_X)])
        eng.set_psi(psi)
        eng.derivative()
        with pytest.raises(Q.QtgError, match="factor mode out of range"):
            eng.set_hamiltonian(bad)
        for l, a in act[::7]:
            h, g = om.hmat(l, a), om.hole(l, a)
            assert np.max(np.abs(eng.matrix(2, l, a) - h)) < 1e-11 * max(1, np.max(np.abs(h)))
            assert np.max(np.abs(eng.matrix(3, l, a) - g)) < 1e-11 * max(1, np.max(np.abs(g)))
        eng.derivative()
        assert _err(eng.get(0), ref) < 1e-11
