"""Transforms of lengths with a prime factor above 23 (line_dft_kernel): every tile count it is
compiled for, its first and last lengths, even lengths (the unpaired middle element), each axis
of the full grid, the transposed slab passes, few and many lines (8, 16, 32 lines per block),
against the oracle's operator on the same grid (FP64 1e-11 of the largest value) and FP32
against FP64 (1e-6: with u = 6e-8, transforms of at most 500,000 points forth and back grow as
sqrt(2 log2 500,000) u = 6 u, and the sums of at most 7^3 rounded products on either side, whose
few largest dominate, by about as much)."""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,tiles,B,layout", [
    ((29, 31, 30), (1,), 1, 1),         # 16 rows: the last length of one tile
    ((20, 32, 47), (2,), 3, 1),
    ((24, 61, 22), (2,), 2, 1),
    ((62, 18, 24), (2,), 2, 1),         # 32 rows: two full tiles
    ((20, 24, 67), (3,), 4, 1),
    ((18, 94, 20), (3,), 1, 1),
    ((127, 16, 18), (4,), 1, 1),
    ((16, 131, 18), (6,), 2, 1),
    ((18, 16, 193), (8,), 2, 1),
    ((251, 16, 18), (8,), 1, 1),        # the last length
    ((16, 18, 257), (), 1, 1),          # beyond: the radix stages
    ((16, 18, 134), (), 1, 1),          # past four tiles with a smaller stage
    ((59, 43, 40), (2,), 12, 0),        # slab: y written transposed, x on contiguous rows
])
def test_lengths_with_large_primes_match_oracle(grid, tiles, B, layout):
    print(f"line dft grid={grid} B={B} layout={layout}", flush=True)
    rng = np.random.default_rng(43)
    L = [20.0, 18.0, 21.0]
    N = 40
    pos = rng.uniform(0, 1, (N, 3)) * L
    if layout == 0:
        pos[:, 2] = rng.uniform(-0.2, 0.2, N)
    op = Op(L, 1e-6, 0.5, grid=grid, support=6, layout=layout)
    op.set_positions(pos)
    sc = np.full(N, 0.3 - 0.2j)
    op.set_self_coef(sc)
    p = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(p, C.PREC_DOUBLE)
    C.profile_enable(False)
    names = C.profile_names()
    for t in tiles:
        assert f"line_dft_kernel<double, false, {t}>" in names and f"line_dft_kernel<double, true, {t}>" in names, names
    assert bool(tiles) or not any(n.startswith("line_dft_kernel") for n in names)
    ref = O.Operator(L, 1e-6, 0.5, grid=list(grid), P=6)
    ref.set_positions(pos)
    for b in sorted({0, B - 1}):
        assert rel(y[b], ref.apply(p[b], sc)) < 1e-11, b
    r64 = op.apply(p, C.PREC_DOUBLE, C.PART_RECIP)
    assert rel(op.apply(p, C.PREC_MIXED, C.PART_RECIP), r64) < 1e-6
