"""The direct field's source slices: particle counts around the target block (8, 16, 64) and
the staged source tile (128), against the oracle's pair sums (FP64 1e-12 of the largest value,
FP32 1e-5: sums of at most 300 terms), and batches wide enough for 16 and 64 targets per block
against the same systems one at a time (8 targets per block; FP64 rounding of another order,
1e-13 times the square root of the number of terms)."""
import ctypes

import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


def _direct(pos, radii, quads):
    op = Op.__new__(Op)
    op.h = ctypes.c_void_p()
    r = np.ascontiguousarray(radii, np.float64)
    C.check(C.load().mpm_op_create_direct(C.dptr(r), r.size, ctypes.byref(op.h)))
    op.N, op.Q, op._quads = 0, 0, quads
    if quads is not None:
        C.check(C.load().mpm_op_set_quads(op.h, (ctypes.c_int * len(quads))(*quads), len(quads)))
    op.set_positions(pos)
    return op


def _points(N, rng):
    pos = rng.uniform(0, 2.6 * N ** (1 / 3) + 3.0, (N, 3))
    if N > 2:
        pos[1] = pos[0] + [0.3, -0.2, 0.1]  # closer than the radius
    return pos


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 127, 128, 129, 300])
@pytest.mark.parametrize("with_quads", [False, True])
def test_direct_slices_match_oracle(N, with_quads):
    print(f"direct N={N} quads={with_quads}", flush=True)
    rng = np.random.default_rng(N)
    pos, rad = _points(N, rng), rng.uniform(0.8, 1.5, N)
    quads = list(range(0, N, 2)) if with_quads else None
    op = _direct(pos, rad, quads)
    sc = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    op.set_self_coef(sc)
    x = rng.standard_normal((3, op.n)) + 1j * rng.standard_normal((3, op.n))
    ref = O.DirectOperator(rad, quads)
    ref.set_positions(pos)
    want = np.stack([np.asarray(ref.apply(v, sc)).reshape(-1) for v in x])
    y64 = op.apply(x, C.PREC_DOUBLE, C.PART_REAL).reshape(3, -1)
    assert rel(y64, want) < 1e-12
    assert rel(op.apply(x, C.PREC_MIXED, C.PART_REAL).reshape(3, -1), want) < 1e-5


@pytest.mark.parametrize("N,targets", [(1100, 16), (4200, 64)])
def test_direct_wide_batches_equal_single_systems(N, targets):
    print(f"direct N={N} targets={targets}", flush=True)
    rng = np.random.default_rng(5)
    op = _direct(_points(N, rng), [1.0], list(range(0, N, 3)))
    op.set_self_coef(np.full(N, 0.4 - 0.2j))
    x = rng.standard_normal((32, op.n)) + 1j * rng.standard_normal((32, op.n))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(x, C.PREC_DOUBLE, C.PART_REAL)
    C.profile_enable(False)
    assert f"direct_kernel<double, 2, true, {targets}>" in C.profile_names(), C.profile_names()
    for b in (0, 15, 31):
        assert rel(op.apply(x[b], C.PREC_DOUBLE, C.PART_REAL), y[b]) < 1e-13 * np.sqrt(N)
