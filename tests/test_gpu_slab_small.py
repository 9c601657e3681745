"""Small layers on the slab: which batches gather their contraction per particle, and which take the
regions, against the oracle (FP64 1e-11 of the largest value)."""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("support,N,B,contract", [
    (8, 120, 2, "gather_kernel<double, 4, true>"),
    (8, 120, 3, "contract_nb_mfma_kernel<double, 4, 10, true, 3, double>"),
    (6, 120, 3, "gather_kernel<double, 4, true>"),
    (8, 1025, 1, "contract_nb_mfma_kernel<double, 4, 10, true, 3, double>"),
])
def test_small_slabs_match_oracle(support, N, B, contract):
    print(f"small slab support={support} N={N} B={B}", flush=True)
    rng = np.random.default_rng(113)
    L, grid = [30.0, 28.0, 40.0], (34, 32, 61)
    pos = np.stack([rng.uniform(0, 1, N) * L[0], rng.uniform(0, 1, N) * L[1], np.zeros(N)], 1)
    op = Op(L, 1e-6, 0.5, grid=grid, support=support)
    op.set_positions(pos)
    assert op.info().slab_planes == support + 1
    sc = np.full(N, -0.3 + 0.05j)
    op.set_self_coef(sc)
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, C.PREC_DOUBLE)
    C.profile_enable(False)
    names = C.profile_names()
    assert contract in names, names
    assert any(n.startswith("contract") and n != "contract" for n in names) == contract.startswith("contract"), names
    ref = O.Operator(L, 1e-6, 0.5, grid=list(grid), P=support)
    ref.set_positions(pos)
    for b in range(B):
        assert rel(y[b], ref.apply(p[b], sc)) < 1e-11, b
