"""The Lanczos recurrence of the Krylov-sweep SCF at the edges of its forms
(node tensors of up to 1024, 2048 and 4096 elements in registers, larger ones
not), one sweep against the oracle."""
import pytest

import oracle_lib as O
import qutree_amd as Q
import test_gpu_scf as TS
from qutree_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", [(8, 16), (8, 17), (10, 20), (16, 16), (14, 21)])  # n1 n1 n2: 1024 ... 4116
def test_scf_sweep_matches_oracle(n1, n2):
    print(f"case scf edges {n1} {n2}", flush=True)
    modes = 8 if n1 < 14 else 4
    text = W.balanced_tree_text(modes, n1, [n1, n2, 2])
    H = W.coupled_quartic(modes, 5, c_sigma=0.05)
    psi = O.OracleModel(text, H).fill_random(7, delta_lowest=False)
    om, ref, floor = TS.oracle_pair(text, H, psi, 1, 4)
    TS.compare(om, ref, Q.SCF(Q.Engine(text, H), 4).run(psi, 1), floor)
