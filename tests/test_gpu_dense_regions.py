"""The full grid's region kernels where a region holds more candidate particles than one
staged chunk: regions of four planes, the 16- and 32-column forms of the spread
(spread_mfma_kernel) and the contraction with a wave per candidate block
(contract_nb_mfma_kernel), and the rule that leaves the contraction to the per-particle
gather; against the oracle's operator on the same grid and support.  FP64 to 1e-11 of the
largest value as everywhere; the FP32 reciprocal part to 2e-6: with u = 6e-8, up to 1,100 particles
on every voxel of the smallest grid sum to sqrt(1,100) u = 33 u of their size, the transforms of at
most 110,592 points and the rounded products add a few u.
"""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,N,support,B,spread,contract", [
    # more than 64 candidates per region, partial last chunks, narrow batches
    ((24, 22, 20), 1301, 8, 2, "spread_mfma_kernel<double, 4, 4, 16, 3>", "contract_nb_mfma_kernel<double, 4, 4, true, 3, double>"),
    ((24, 22, 20), 1999, 8, 4, "spread_mfma_kernel<double, 4, 4, 16, 3>", "contract_nb_mfma_kernel<double, 4, 4, true, 3, double>"),
    # odd z length (4-byte grid loads), axes shorter than the stencil (folded weights)
    ((23, 21, 19), 1500, 6, 3, "spread_mfma_kernel<double, 4, 4, 16, 3>", "contract_nb_mfma_kernel<double, 4, 4, false, 3, double>"),
    ((7, 9, 20), 1100, 8, 5, "spread_mfma_kernel<double, 4, 4, 16, 3>", "contract_nb_mfma_kernel<double, 4, 4, true, 3, double>"),
    # enough blocks for 32 columns each
    ((48, 48, 48), 900, 8, 30, "spread_mfma_kernel<double, 4, 4, 32, 3>", "contract_nb_mfma_kernel<double, 4, 4, true, 3, double>"),
    # five stencil points: gathered per particle
    ((24, 22, 20), 1999, 4, 4, "spread_mfma_kernel<double, 4, 4, 16, 3>", "gather_kernel<double, 4, false>"),
    # no more than a wave of particles per SIMD: gathered per particle
    ((24, 22, 20), 701, 8, 2, "spread_mfma_kernel<double, 4, 4, 16, 3>", "gather_kernel<double, 4, false>"),
    # one right-hand side on few regions: gathered per particle
    ((24, 22, 20), 1999, 8, 1, "spread_mfma_kernel<double, 4, 4, 16, 3>", "gather_kernel<double, 1, false>"),
])
def test_dense_full_grid_matches_oracle(grid, N, support, B, spread, contract):
    print(f"dense full grid {grid} N={N} support={support} B={B}", flush=True)
    rng = np.random.default_rng(23)
    L = [20.0, 18.0, 21.0]
    pos = rng.uniform(-0.5, 1.5, (N, 3)) * L  # also outside the box
    op = Op(L, 1e-6, 0.5, grid=grid, support=support, layout=1)
    op.set_positions(pos)
    sc = np.full(N, -0.3 + 0.05j)
    op.set_self_coef(sc)
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, C.PREC_DOUBLE)
    C.profile_enable(False)
    names = C.profile_names()
    assert spread in names and contract in names, names
    ref = O.Operator(L, 1e-6, 0.5, grid=list(grid), P=support)
    ref.set_positions(pos)
    for b in sorted({0, B // 2, B - 1}):
        assert rel(y[b], ref.apply(p[b], sc)) < 1e-11, b
    r64 = op.apply(p, C.PREC_DOUBLE, C.PART_RECIP)
    r32 = op.apply(p, C.PREC_MIXED, C.PART_RECIP)
    assert rel(r32, r64) < 2e-6
