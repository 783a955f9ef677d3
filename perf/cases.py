"""Timed cases of the framework: what its users have it do, through the public
entry points of `qutree_amd` (the C ABI of include/qutree_amd.h and its
Python binding), over the range of sizes, data types and options in use.

Families
  node   one node contraction at a time, on device pointers: the drop-in
         replacements of the Fortran kernels (matvec / ctmatvec / rhomat)
  plan   grouped node contractions of many tensors of uneven shape in one
         call (qtg_plan_execute): mode products, then hole contractions with
         the results; with terms = 2 a second, adjoint term is accumulated
  sweep  one H|Psi> sweep (Derivative: build + LayerDerivative at all nodes)
         for a state on the device, the derivative read back
  grad   the energy gradient dE/dA* of a state
  cmf    constant-mean-field steps of a wave packet
  scf    one Krylov-sweep SCF iteration
  fit    H|Psi> fitted into the tree (alternating sweeps)
"""
from __future__ import annotations

import math

import numpy as np
import torch

import qutree_amd as Q
from qutree_amd import workloads as W

DEV = "cuda:0"


def listed():
    return [
        # smallest calls: one small node tensor, where a program that replaces
        # the reference's Fortran kernels pays a launch per call
        dict(name="node_small", family="node", before=8, n=8, after=8, dtype="c128"),
        # one large tensor, its middle mode contracted
        dict(name="node_large", family="node", before=256, n=64, after=256, dtype="c128"),
        # the grouped node contractions of the benchmark: 4096 order-3 tensors
        # with legs 8..64, complex128
        dict(name="plan_4096", family="plan", count=4096, legs="8,16,24,32,48,64", shapes=4096, dtype="c128", terms=1),
        # odd, ragged legs in single precision, two terms summed per tensor
        dict(name="plan_ragged_c64", family="plan", count=1000, legs="3-61", shapes=17, dtype="c64", terms=2),
        # the smallest tree of the tests and of smoke(): latency only
        dict(name="sweep_8", family="sweep", modes=8, dvr=8, spf="4,4,4", model="ho", precision=0),
        # the benchmark's headline: 64 modes, 2080 terms
        dict(name="sweep_64", family="sweep", modes=64, dvr=16, spf="8,10,11,13,14,16", model="ho_leaf", precision=0),
        # the largest tree: 128 modes, SPF up to 48, 8256 terms
        dict(name="sweep_128", family="sweep", modes=128, dvr=8, spf="8,14,21,27,34,41,48", model="quartic", precision=0),
        # the same in the reduced-precision form that keeps 1e-8 in the energy
        dict(name="sweep_128_split", family="sweep", modes=128, dvr=8, spf="8,14,21,27,34,41,48", model="quartic",
             precision=2),
        # gradient-based optimisation of the 32-mode anharmonic model
        dict(name="grad_32", family="grad", modes=32, dvr=8, spf="8,24,24,24,24", model="quartic"),
        # time propagation of a wave packet on the 64-mode tree
        dict(name="cmf_64", family="cmf", modes=64, dvr=16, spf="8,10,11,13,14,16", model="ho_leaf", steps=2),
        # ground state by SCF on the 16-mode quartic model
        dict(name="scf_16", family="scf", modes=16, dvr=6, spf="4,6,8,8", model="quartic", krylov=5),
        # an operator applied and fitted back into the 32-mode tree
        dict(name="fit_32", family="fit", modes=32, dvr=8, spf="8,24,24,24,24", model="neighbours", iterations=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _spfs(rng, layers, dvr, top):
    """SPF counts rising toward the root, none above what the two children
    (or the grid) can carry."""
    out = [rng.randint(max(2, dvr // 2), dvr - 1)]
    for k in range(1, layers):
        hi = min(top, out[-1] ** 2 - 1, out[-1] + max(2, top // layers) + 2)
        out.append(rng.randint(min(out[-1], hi), hi))
    return ",".join(str(x) for x in out)


def draw(rng):
    family = rng.choice(["node", "plan", "plan", "sweep", "sweep", "grad", "cmf", "scf", "fit"])
    if family == "node":
        return dict(family="node", before=_log_int(rng, 3, 300), n=rng.randint(3, 64), after=_log_int(rng, 3, 300),
                    dtype=rng.choice(["c128", "c128", "c64"]))
    if family == "plan":
        lo, hi = rng.choice([(3, 20), (3, 61), (8, 64), (17, 48)])
        return dict(family="plan", count=_log_int(rng, 16, 2000), legs="%d-%d" % (lo, hi), shapes=rng.randint(1, 10 ** 6),
                    dtype=rng.choice(["c128", "c128", "c64"]), terms=rng.choice([1, 2]))
    if family == "sweep":
        layers = rng.choice([3, 4, 5, 6])
        dvr = rng.randint(5, 16)
        return dict(family="sweep", modes=2 ** layers, dvr=dvr, spf=_spfs(rng, layers, dvr, rng.choice([8, 16, 16, 28])),
                    model=rng.choice(["ho", "ho_leaf", "quartic"]), precision=rng.choice([0, 0, 0, 2]))
    if family == "grad":
        layers = rng.choice([3, 4, 5])
        dvr = rng.randint(5, 10)
        return dict(family="grad", modes=2 ** layers, dvr=dvr, spf=_spfs(rng, layers, dvr, 24), model="quartic")
    if family == "cmf":
        layers = rng.choice([3, 4, 5])
        dvr = rng.randint(8, 14)
        return dict(family="cmf", modes=2 ** layers, dvr=dvr, spf=_spfs(rng, layers, min(dvr, 8), 14), model="ho_leaf",
                    steps=2)
    if family == "scf":
        layers = rng.choice([2, 3, 4])
        dvr = rng.randint(4, 8)
        return dict(family="scf", modes=2 ** layers, dvr=dvr, spf=_spfs(rng, layers, min(dvr, 6), 10), model="quartic",
                    krylov=rng.randint(3, 6))
    layers = rng.choice([3, 4, 5])
    dvr = rng.randint(5, 8)
    return dict(family="fit", modes=2 ** layers, dvr=dvr, spf=_spfs(rng, layers, dvr, 20), model="neighbours",
                iterations=2)


# ------------------------------------------------------------------ node, plan
def _shapes(case):
    """(legs, mode) of every tensor of a plan case."""
    g = np.random.default_rng(case["shapes"])
    if "-" in case["legs"]:
        lo, hi = (int(x) for x in case["legs"].split("-"))
        legs = g.integers(lo, hi + 1, size=(case["count"], 3))
    else:
        pool = np.array([int(x) for x in case["legs"].split(",")])
        legs = pool[g.integers(0, len(pool), size=(case["count"], 3))]
    modes = g.integers(0, 3, size=case["count"])
    before = np.array([int(np.prod(l[:m])) for l, m in zip(legs, modes)])
    n = np.array([int(l[m]) for l, m in zip(legs, modes)])
    after = np.array([int(np.prod(l[m + 1:])) for l, m in zip(legs, modes)])
    return before, n, after


def _offsets(sizes):
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)


def _randn(gen, count, dtype):
    real = torch.float64 if dtype == "c128" else torch.float32
    return torch.view_as_complex(torch.randn(count, 2, dtype=real, device=DEV, generator=gen))


def _node_data(case, seed):
    """Tensors N(0,1) + i N(0,1) and matrices of norm about one."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    if case["family"] == "node":
        before, n, after, terms = np.array([case["before"]]), np.array([case["n"]]), np.array([case["after"]]), 2
    else:
        before, n, after = _shapes(case)
        terms = case["terms"]
    B = _randn(gen, int(np.sum(before * n * after)), case["dtype"])
    Ms = []
    for _ in range(terms):
        M = _randn(gen, int(np.sum(n * n)), case["dtype"])
        scale = torch.from_numpy(np.repeat(1.0 / np.sqrt(2.0 * n), n * n)).to(DEV)
        Ms.append(M * scale.to(M.real.dtype))
    return before, n, after, B, Ms


# ------------------------------------------------------------------------ trees
def _tree_text(case):
    return W.balanced_tree_text(case["modes"], case["dvr"], [int(x) for x in case["spf"].split(",")])


def _hamiltonian(case):
    f = case["modes"]
    if case["model"] == "ho":
        return W.coupled_ho(f, f, c_sigma=0.02)
    if case["model"] == "ho_leaf":
        return W.coupled_ho(f, f, c_sigma=0.01, one_mode_matrix=True)
    if case["model"] == "quartic":
        return W.coupled_quartic(f, f)
    # nearest-neighbour products of small matrices near the identity's scale
    g = np.random.default_rng(f)
    H, d = W.Hamiltonian(), case["dvr"]
    for i in range(f):
        mats = []
        for _ in range(2):
            A = g.normal(size=(d, d)) + 1j * g.normal(size=(d, d))
            mats.append(0.15 * A / np.linalg.norm(A, 2))
        H.add_term(1.0, [(i, W.FACTOR_MATRIX, mats[0]), ((i + 1) % f, W.FACTOR_MATRIX, mats[1])])
    return H


def _grid(d):
    """HO-DVR grid (omega 1), FBR -> DVR transformation, kinetic matrix."""
    k = np.arange(d - 1)
    X = np.diag(np.sqrt((k + 1) / 2.0), 1)
    x, U = np.linalg.eigh(X + X.T)
    U = U * np.sign(U[0])
    T = np.diag((2 * np.arange(d) + 1) / 4.0)
    k = np.arange(max(d - 2, 0))
    off = np.diag(-np.sqrt((k + 1.0) * (k + 2.0)) / 4.0, 2) if d > 2 else np.zeros((d, d))
    return x, U, U.T @ (T + off + off.T) @ U


def _nodes(case):
    """Node list in address order (post-order, last child first): children as
    addresses, dims, the modes below, the offset in the state."""
    spf = [int(x) for x in case["spf"].split(",")]
    layers = int(math.log2(case["modes"]))
    nodes = []

    def visit(h, m0):
        n = 1 if h == layers else spf[h]
        if h == 0:
            nodes.append(dict(children=[], dims=[case["dvr"], n], modes=[m0]))
            return len(nodes) - 1
        half = 2 ** (h - 1)
        right = visit(h - 1, m0 + half)
        left = visit(h - 1, m0)
        nodes.append(dict(children=[left, right], dims=[spf[h - 1], spf[h - 1], n],
                          modes=list(range(m0, m0 + 2 * half))))
        return len(nodes) - 1

    visit(layers, 0)
    off = 0
    for v in nodes:
        v["off"] = off
        v["N"] = int(np.prod(v["dims"]))
        off += v["N"]
    return nodes, off


def _state(case, seed):
    """A correlated wave packet: low harmonic-oscillator functions, slightly
    rotated, at the leaves; node tensors that favour low configurations;
    top-node weights that fall off over the SPFs.  Orthonormal nodes."""
    g = np.random.default_rng(seed)
    nodes, total = _nodes(case)
    psi = np.zeros(total, np.complex128)
    _, U, _ = _grid(case["dvr"])

    def noise(*shape):
        return g.normal(size=shape) + 1j * g.normal(size=shape)

    for v in nodes:
        n = v["dims"][-1]
        rows = v["N"] // n
        if not v["children"]:
            A, _ = np.linalg.qr(np.eye(rows, dtype=np.complex128) + 0.1 * noise(rows, rows))
            A = U.T.astype(np.complex128) @ A[:, :n]
        else:
            d = v["dims"][0]
            order = np.argsort((np.arange(d)[:, None] + np.arange(d)[None, :]).ravel(order="F"), kind="stable")
            if n == 1:
                i = np.arange(d)
                T = 0.03 * noise(d, d) / d + np.diag(np.exp(-4.0 * i / d) * np.exp(2j * np.pi * g.random(d)))
                A = (T / np.linalg.norm(T)).ravel(order="F")[:, None]
            else:
                A = 0.3 * noise(rows, n) / math.sqrt(rows)
                A[order[:n], np.arange(n)] += 1.0
                A, _ = np.linalg.qr(A)
        psi[v["off"]:v["off"] + v["N"]] = A.ravel(order="F")
    return psi


_kept = {}  # the handles (engine, plans) of the case in work, as a program keeps them for all its states


def _handles(case):
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _kept:
        _kept.clear()
        h = {}
        if case["family"] == "plan":
            before, n, after = _shapes(case)
            oT, oM = _offsets(before * n * after)[:-1], _offsets(n * n)[:-1]
            for t in range(case["terms"]):
                mp = np.zeros(len(n), Q.MP_DESC)
                mp["offC"], mp["offM"], mp["offB"] = oT, oM, oT
                mp["before"], mp["nB"], mp["nC"], mp["after"] = before, n, n, after
                mp["op"], mp["add"] = (0, 0) if t == 0 else (2, 1)
                h["product%d" % t] = Q.Plan("mode_product", mp, complex64=case["dtype"] == "c64")
            hc = np.zeros(len(n), Q.HC_DESC)
            hc["offS"], hc["offA"], hc["offB"] = oM, oT, oT
            hc["before"], hc["nA"], hc["nB"], hc["after"] = before, n, n, after
            h["hole"] = Q.Plan("hole_contraction", hc, complex64=case["dtype"] == "c64")
        elif case["family"] != "node":
            h["engine"] = Q.Engine(_tree_text(case), _hamiltonian(case), precision=case.get("precision", 0))
            if case["family"] == "cmf":
                h["cmf"] = Q.CMF(h["engine"])
            if case["family"] == "scf":
                h["scf"] = Q.SCF(h["engine"], case["krylov"])
            if case["family"] == "fit":
                h["fit"] = Q.ApplyFit(h["engine"])
        _kept[key] = h
    return _kept[key]


def prepare(case, seed):
    Q.init()
    s = dict(case=case, **_handles(case))
    if case["family"] in ("node", "plan"):
        before, n, after, B, Ms = _node_data(case, seed)
        s.update(B=B, Ms=Ms, C=torch.zeros_like(B), D=torch.zeros_like(B), S=torch.zeros_like(Ms[0]))
        return s
    psi = _state(case, seed)
    s["psi"] = psi
    if case["family"] == "sweep":
        s["psi_dev"] = torch.from_numpy(psi).to(DEV)
    if case["family"] in ("sweep", "grad"):
        s["out"] = torch.zeros(psi.size, dtype=torch.complex128, pin_memory=True)
        s["out_np"] = torch.view_as_real(s["out"]).numpy().reshape(-1)
    return s


def run(state):
    case, L = state["case"], Q.lib()
    if case["family"] == "node":
        # a product, an adjoint product and the contraction of the two results
        b, n, a = case["before"], case["n"], case["after"]
        B, M, G, C, D, S = (t.data_ptr() for t in (state["B"], *state["Ms"], state["C"], state["D"], state["S"]))
        product, hole = ((L.qtg_mode_product_z, L.qtg_hole_contraction_z) if case["dtype"] == "c128" else
                         (L.qtg_mode_product_c, L.qtg_hole_contraction_c))
        Q.check(product(C, M, B, b, n, n, a, 0, 0, None))
        Q.check(product(D, G, B, b, n, n, a, 2, 0, None))
        Q.check(hole(S, C, D, b, n, n, a, 0, None))
        return [state["C"], state["D"], state["S"]]
    if case["family"] == "plan":
        B, C, S = (state[k].data_ptr() for k in "BCS")
        for t in range(case["terms"]):
            Q.check(L.qtg_plan_execute(state["product%d" % t].ptr, C, state["Ms"][t].data_ptr(), B, None))
        Q.check(L.qtg_plan_execute(state["hole"].ptr, S, B, C, None))
        return [state["C"], state["S"]]
    if case["family"] == "sweep":
        eng = state["engine"]
        Q.check(L.qtg_engine_set_psi_device(eng.ptr, state["psi_dev"].data_ptr(), None))
        eng.derivative(sync=False)
        Q.check(L.qtg_engine_get_dpsi(eng.ptr, state["out_np"], 0, None))
        return state["out"]
    if case["family"] == "grad":
        eng = state["engine"]
        eng.set_psi(state["psi"])
        e = eng.forward()
        Q.check(L.qtg_engine_backward(eng.ptr, state["out_np"].ctypes.data, None))
        return [state["out"], e]
    if case["family"] == "cmf":
        r = state["cmf"].integrate(state["psi"], 0.0, 1000.0, 0.02, 0.02, acc_cmf=1e-4, acc_bs=1e-5,
                                   max_steps=case["steps"], max_out=64)
        return [r["psi"], r["energies"], r["autocorr"]]
    if case["family"] == "scf":
        r = state["scf"].run(state["psi"], 1)
        return [r["psi"], r["energies"]]
    r = state["fit"].run(state["psi"], 3, case["iterations"])
    return [r["psi"], r["fidelities"]]


def work(case):
    """Bytes: inputs once, outputs once.  FLOPs: 8 per complex multiply-add;
    for the trees those of the operator algebra itself: at every node the
    operators of the modes below (and the summed operators across), each
    applied and contracted once upward and once downward."""
    es = 16.0 if case.get("dtype", "c128") == "c128" else 8.0
    if case["family"] == "node":
        n, N = case["n"], case["before"] * case["n"] * case["after"]
        return dict(bytes=es * (3 * N + 3 * n * n), flops=3 * 8.0 * N * n)
    if case["family"] == "plan":
        before, n, after = _shapes(case)
        N = before * n * after
        t = case["terms"]
        return dict(bytes=es * float(np.sum(2 * N + (t + 1) * n * n)), flops=8.0 * (t + 1) * float(np.sum(N * n)))
    nodes, total = _nodes(case)
    f = case["modes"]
    flops = 0.0
    for v in nodes:
        n, N, l = v["dims"][-1], v["N"], len(v["modes"])
        if not v["children"]:
            flops += 8.0 * N * (4 * v["dims"][0] + 6 * n)
            continue
        d = v["dims"][0]
        up = (l + l // 2 + 2) * (d + n)  # x of every mode below, and the pair sums
        down = (min(l, f - l) + 3) * (2 * d + n) if n > 1 else 0
        flops += 8.0 * N * (up + down + 4 * n)
    # whole derivatives a pass needs at least: CMF two builds and some ten
    # node derivatives a step, an SCF iteration two visits of each node with
    # a Krylov space, a fit two iterations
    times = {"sweep": 1.0, "grad": 1.3, "cmf": 12.0 * case.get("steps", 1), "scf": 2.0 * case.get("krylov", 1),
             "fit": 2.0 * case.get("iterations", 1) * 0.3}[case["family"]]
    return dict(bytes=2 * 16.0 * total, flops=times * flops)


def tolerance(case):
    """About four times what the path showed against exact(), or with its
    sums in another order (other K splits), over some thirty cases."""
    single = case.get("dtype") == "c64"
    if case["family"] == "node":  # reductions of up to 90000 products
        return dict(rel=1.2e-5) if single else dict(rel=5e-14)
    if case["family"] == "plan":
        return dict(rel=1.2e-6) if single else dict(rel=8e-15)
    if case["family"] == "sweep":
        # rho^-1 carries the rounding of the smallest densities into the result
        return dict(rel=1.2e-13, max=2e-11) if case["precision"] == 0 else dict(rel=6e-8, max=2e-6)
    if case["family"] == "grad":
        return dict(rel=2.4e-13, max=5e-12)
    if case["family"] == "cmf":
        return dict(rel=5e-14, max=1e-12)
    if case["family"] == "scf":  # the sweep's QRs complete nearly unoccupied directions
        return dict(rel=6e-11, max=6e-10)
    return dict(rel=1.6e-13, max=6e-12)


# ------------------------------------------------------------- 64-bit reference
def exact(case, seed):
    if case["family"] in ("node", "plan"):
        return _exact_nodes(case, seed)
    if case["family"] in ("sweep", "grad"):
        return _exact_tree(case, seed)
    # the integrator, the SCF sweep and the fit are step-controlled or
    # alternating iterations: no value apart from the iteration itself
    return None


def _exact_nodes(case, seed):
    before, n, after, B, Ms = _node_data(case, seed)
    B, Ms = B.to(torch.complex128), [M.to(torch.complex128) for M in Ms]
    oT, oM = _offsets(before * n * after), _offsets(n * n)
    C, S = torch.zeros_like(B), torch.zeros_like(Ms[0])
    D = torch.zeros_like(B)
    for i in range(len(n)):
        b, m, a = int(before[i]), int(n[i]), int(after[i])
        x = B[oT[i]:oT[i + 1]].view(a, m, b)  # first index fastest
        mats = [M[oM[i]:oM[i + 1]].view(m, m).t() for M in Ms]  # column-major
        y = torch.matmul(mats[0].contiguous(), x)
        z = torch.matmul(mats[1].conj().t().contiguous(), x) if len(mats) > 1 else None
        if case["family"] == "plan":
            if z is not None:
                y = y + z
            bra, ket = x, y
        else:
            D[oT[i]:oT[i + 1]] = z.reshape(-1)
            bra, ket = y, z
        C[oT[i]:oT[i + 1]] = y.reshape(-1)
        # S(j, l) = sum conj(bra(b, j, a)) ket(b, l, a)
        bf = bra.permute(1, 0, 2).reshape(m, -1).contiguous()
        kf = ket.permute(1, 0, 2).reshape(m, -1).contiguous()
        S[oM[i]:oM[i + 1]] = torch.matmul(bf.conj(), kf.t().contiguous()).t().reshape(-1)
    return [C, S] if case["family"] == "plan" else [C, D, S]


def _couplings(case):
    """One-mode matrices on the grid and the pair couplings c_ij of
    sum_i h_i + sum_{i<j} c_ij x_i x_j, from the Hamiltonian's terms."""
    H, f = _hamiltonian(case), case["modes"]
    x, _, kin = _grid(case["dvr"])
    one = np.zeros((f, case["dvr"], case["dvr"]))
    c = np.zeros((f, f))
    for l in range(H.nterms):
        fs = range(H.term_off[l], H.term_off[l + 1])
        if len(fs) == 2:
            i, j = (H.fmode[q] for q in fs)
            c[i, j] += H.coeff[l].real
            c[j, i] += H.coeff[l].real
            continue
        q = fs[0]
        kind = H.fkind[q]
        if kind == W.FACTOR_KIN:
            m = kin
        elif kind == W.FACTOR_X2:
            m = np.diag(x ** 2)
        else:
            a = H.pool[2 * H.fpool[q]:2 * H.fpool[q] + 4]
            m = a[0] * kin + np.diag(a[1] * x + a[2] * x ** 2 + a[3] * x ** 4)
        one[H.fmode[q]] += H.coeff[l].real * m
    return x, one, c


def _exact_tree(case, seed):
    """<Psi|H|Psi> by the tree, its derivative by automatic differentiation.
    With the overlaps of the lower nodes held at one, d<H>/dA_v* is Apply at
    v, and the derivative is -i rho^-1 (1 - P) Apply(v); with them followed,
    d(<H>/<1>)/dA_v* is the energy gradient."""
    nodes, total = _nodes(case)
    x, one, c = _couplings(case)
    psi = _state(case, seed)
    cplx = torch.complex128
    x = torch.from_numpy(x).to(DEV, cplx)
    one, c = torch.from_numpy(one).to(DEV, cplx), torch.from_numpy(c).to(DEV, cplx)
    follow = case["family"] == "grad"
    A = []
    for v in nodes:
        t = torch.from_numpy(psi[v["off"]:v["off"] + v["N"]].reshape(v["dims"], order="F").copy()).to(DEV)
        A.append(t.contiguous().requires_grad_(True))

    def sandwich(bra, ops0, ops1, ket):
        """sum conj(bra)(i,j,k) op0(i,i') op1(j,j') ket(i',j',l) for a batch of
        operators; None: one"""
        z = ket[None]
        if ops0 is not None:
            z = torch.matmul(ops0, ket.reshape(ket.shape[0], -1)).view(-1, *ket.shape)
        if ops1 is not None:
            z = torch.matmul(ops1[:, None], z)
        b = bra.conj().reshape(-1, bra.shape[-1]).t().contiguous()
        return torch.matmul(b, z.reshape(z.shape[0], -1, z.shape[-1]))

    val = []
    for v, t in zip(nodes, A):
        if not v["children"]:
            m = v["modes"][0]
            b = t.conj().t().contiguous()
            val.append((torch.matmul(b, torch.matmul(one[m], t)), torch.matmul(b, x[:, None] * t)[None],
                        torch.matmul(b, t) if follow else None))
            continue
        (h0, X0, S0), (h1, X1, S1) = (val[k] for k in v["children"])
        m0, m1 = (nodes[k]["modes"] for k in v["children"])
        e0 = S0[None] if follow else None
        e1 = S1[None] if follow else None
        Y1 = torch.einsum("ij,jab->iab", c[m0][:, m1], X1)
        h = (sandwich(t, h0[None], e1, t) + sandwich(t, e0, h1[None], t))[0] + sandwich(t, X0, Y1, t).sum(0)
        if t.shape[-1] == 1:
            val.append((h, None, sandwich(t, e0, e1, t)[0]))
            continue
        X = torch.cat([sandwich(t, X0, e1, t), sandwich(t, e0, X1, t)])
        val.append((h, X, sandwich(t, e0, e1, t)[0] if follow else None))
    h, _, s = val[-1]
    if follow:
        e = h[0, 0].real / s[0, 0].real
        e.backward()
        g = [0.5 * t.grad for t in A]
        return [_flat(g), float(e.detach())]
    h[0, 0].real.backward()
    with torch.no_grad():
        rho = [None] * len(nodes)
        for a in range(len(nodes) - 1, -1, -1):
            t = A[a]
            z = t if rho[a] is None else torch.matmul(t, rho[a].t())  # rho x_last A
            for k, ch in enumerate(nodes[a]["children"]):
                br = t.movedim(k, 0).reshape(t.shape[k], -1)
                kt = z.movedim(k, 0).reshape(t.shape[k], -1)
                rho[ch] = torch.matmul(br.conj(), kt.t().contiguous())
        out = []
        for a, t in enumerate(A):
            y = 0.5 * t.grad
            if rho[a] is None:
                out.append(-1j * y)
                continue
            n = t.shape[-1]
            m, y = t.reshape(-1, n), y.reshape(-1, n)
            p = torch.linalg.solve(torch.matmul(m.conj().t(), m), torch.matmul(m.conj().t(), y))
            y = y - torch.matmul(m, p)
            w, U = torch.linalg.eigh(0.5 * (rho[a] + rho[a].conj().t()))
            w = 1.0 / (w + 1e-10 * torch.exp(-w / 1e-10))
            R = torch.matmul(U * w, U.conj().t())
            out.append((-1j * torch.matmul(y, R.t())).reshape(t.shape))
        return _flat(out)


def _flat(tensors):
    return torch.cat([t.detach().permute(*range(t.dim() - 1, -1, -1)).reshape(-1) for t in tensors]).cpu()
