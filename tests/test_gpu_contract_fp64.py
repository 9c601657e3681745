"""Contractions of an FP32 grid that are summed in FP64 (few regions beside the particles), against
the single-stage FP64 contraction of the same grid's values: to 1e-13 of the largest value, where
sums in FP32 differ by about 1e-7."""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,N,B,kernel", [
    ((47, 42, 62), 1193, 2, "contract_full_mfma_kernel<double, 4, 8, 2, 3, float>"),
    ((47, 42, 62), 1193, 5, "contract_full_mfma_kernel<double, 4, 8, 2, 3, float>"),
    ((47, 42, 61), 1193, 5, "contract_mfma_kernel<double, 4, 8, 2, false, 3, float>"),
    ((16, 16, 16), 40, 5, "contract_full_mfma_kernel<double, 4, 8, 2, 3, float>"),
    ((16, 16, 15), 40, 5, "contract_mfma_kernel<double, 4, 8, 2, false, 3, float>"),
])
def test_few_regions_sum_in_fp64(grid, N, B, kernel):
    print(f"FP64 contraction {grid} N={N} B={B}", flush=True)
    rng = np.random.default_rng(103)
    L = [20.0, 18.0, 21.0]
    op = Op(L, 1e-4, 0.5, grid=grid, support=6, layout=1)
    op.set_positions(rng.uniform(0, 1, (N, 3)) * L)
    op.set_self_coef(np.zeros(N))
    x = rng.standard_normal((B, N, 3)) + 1j * rng.standard_normal((B, N, 3))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(x, C.PREC_MIXED, C.PART_RECIP)
    C.profile_enable(False)
    assert kernel in C.profile_names(), C.profile_names()
    lib = C.load()
    V = 3 * int(np.prod(grid))
    g32, g64 = np.zeros(V, np.complex64), C.DeviceBuffer(16 * V)
    gb, xb, yb = C.DeviceBuffer(8 * V), C.DeviceBuffer(x[0].nbytes), C.DeviceBuffer(x[0].nbytes)
    want = np.zeros_like(x[0])
    for b in range(B):
        xb.upload(x[b])
        for stage in (C.STAGE_SPREAD, C.STAGE_SCALE):
            C.check(lib.mpm_op_stage(op.h, stage, xb.ptr, gb.ptr, None, C.PREC_MIXED, None))
        gb.download(g32)
        g64.upload(g32.astype(np.complex128))
        yb.upload(np.zeros_like(want))
        C.check(lib.mpm_op_stage(op.h, C.STAGE_CONTRACT, xb.ptr, g64.ptr, yb.ptr, C.PREC_DOUBLE, None))
        yb.download(want)
        assert rel(y[b], want) < 1e-13, b
