"""Full-grid batches of several times the last-level cache, whose transforms run chunk by chunk
of components, against batches below it that take the same kernels (to 1e-14 of the largest value:
lines are only grouped otherwise), with the fused z pass in both precisions; and the polydisperse
operator's fused z pass against the oracle (FP64 1e-11; FP32 against FP64 1e-6: transforms of at
most 70,000 points forth and back grow as sqrt(2 log2 70,000) = 6 times 6e-8, the rounded products on
either side about as much)."""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,grid,B,part,kernel", [
    (C.PREC_MIXED, (256, 256, 256), 3, 1, "zline_scale_kernel<float, 1, 3>"),  # 1.2 GB
    # 1.3 GB, partial last chunk; parts of 4, as the contraction of fewer is another kernel
    (C.PREC_DOUBLE, (128, 180, 128), 9, 4, "zline_scale_kernel<double, 1, 3>"),
])
def test_chunked_transforms_equal_small_batches(precision, grid, B, part, kernel):
    print(f"chunked transforms {grid} B={B}", flush=True)
    rng = np.random.default_rng(47)
    L = [40.0, 41.0, 42.0]
    N = 60
    pos = rng.uniform(0, 1, (N, 3)) * L
    op = Op(L, 1e-6, 0.5, grid=grid, support=8, layout=1)
    op.set_positions(pos)
    op.set_self_coef(np.full(N, 0.2 - 0.1j))
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, precision, C.PART_RECIP)
    C.profile_enable(False)
    assert kernel in C.profile_names(), C.profile_names()
    for b in sorted({0, (B - part) // 2, B - part}):
        assert rel(op.apply(p[b:b + part], precision, C.PART_RECIP), y[b:b + part]) < 1e-14


@pytest.mark.parametrize("grid,B", [((40, 36, 48), 3), ((36, 40, 38), 5), ((36, 40, 47), 1)])
def test_polydisperse_z_pass_matches_oracle(grid, B):
    print(f"poly z pass {grid} B={B}", flush=True)
    rng = np.random.default_rng(53)
    L = [24.0, 25.0, 26.0]
    N = 30
    pos = rng.uniform(0, 1, (N, 3)) * L
    rad = rng.uniform(1.0, 2.0, N)
    op = Op(L, 1e-4, 0.5, grid=grid, radii=rad)
    op.set_positions(pos)
    sc = np.full(N, -0.2 + 0.1j)
    op.set_self_coef(sc)
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, C.PREC_DOUBLE)
    C.profile_enable(False)
    fused = any(n.startswith("zline_scale_kernel<double") for n in C.profile_names())
    assert fused == (grid[2] != 47)  # a prime above 23 has no two register stages
    ref = O.PolyOperator(L, 1e-4, 0.5, rad, grid=list(grid))
    ref.set_positions(pos)
    for b in sorted({0, B - 1}):
        assert rel(y[b], ref.apply(p[b], sc)) < 1e-11
    r64 = op.apply(p, C.PREC_DOUBLE, C.PART_RECIP)
    assert rel(op.apply(p, C.PREC_MIXED, C.PART_RECIP), r64) < 1e-6


@pytest.mark.parametrize("nz,B,precision,fused", [
    (46, 3, C.PREC_DOUBLE, False), (69, 1, C.PREC_DOUBLE, False),  # 23 x 2, 23 x 3
    (46, 3, C.PREC_MIXED, True), (51, 2, C.PREC_DOUBLE, True), (92, 2, C.PREC_DOUBLE, True),
    (92, 8, C.PREC_DOUBLE, False),  # 4.0 and 16.2 MB
    (68, 4, C.PREC_MIXED, True), (68, 30, C.PREC_MIXED, False),  # 17 x 4: 3.0 and 22.4 MB
])
def test_polydisperse_z_pass_of_large_radices(nz, B, precision, fused):
    print(f"poly z pass nz={nz} B={B} precision={precision}", flush=True)
    rng = np.random.default_rng(59)
    L, grid = [24.0, 25.0, 26.0], (40, 36, nz)
    N = 20
    pos = rng.uniform(0, 1, (N, 3)) * L
    rad = rng.uniform(1.0, 2.0, N)
    op = Op(L, 1e-4, 0.5, grid=grid, radii=rad)
    op.set_positions(pos)
    sc = np.full(N, -0.2 + 0.1j)
    op.set_self_coef(sc)
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, precision)
    C.profile_enable(False)
    assert any(n.startswith("zline_scale_kernel") for n in C.profile_names()) == fused, C.profile_names()
    ref = O.PolyOperator(L, 1e-4, 0.5, rad, grid=list(grid))
    ref.set_positions(pos)
    # FP32: rounded products on either side of transforms of at most 97,920 points, below 1e-6 of
    # the largest value of the reciprocal part, which the whole field exceeds
    for b in sorted({0, B - 1}):
        assert rel(y[b], ref.apply(p[b], sc)) < (1e-11 if precision == C.PREC_DOUBLE else 1e-6)
