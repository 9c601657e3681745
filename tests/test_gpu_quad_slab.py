"""The quadrupole operator's applies on the slab of occupied z-planes and on the full grid's
regions, against the oracle's operator on the same grid (FP64 to 1e-11 of the largest value):
every plane count the coupling kernel is compiled for, even and odd z lengths (Nyquist
plane), separated layers, Bloch wave vectors, quadrupoles on a subset, narrow and wide batches;
dense and sparse regions, and the per-particle gather of small problems.  The FP32 reciprocal part to
1e-6 of the FP64 one: with u = 6e-8, transforms of at most 65,536 points forth and back grow as
sqrt(2 log2 65,536) u = 6 u, and the sums of rounded products on either side, whose few largest
dominate, by about as much.
The stage-by-stage pipeline, whose grids are full grids, equals the apply.
"""
import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu


def _oracle(L, grid, support, pos, quads, kb):
    ref = O.Operator(L, 1e-6, 0.5, grid=list(grid), P=support)
    if kb is not None:
        ref.set_bloch(*kb)
    ref.set_positions(pos)
    ref.set_quads(None if quads is True else quads)
    return ref


@pytest.mark.parametrize("grid,support,layers,quads,B,kb,kernel", [
    ((30, 28, 61), 2, 1, True, 1, None, "quad_zcouple_kernel<double, 4>"),
    ((30, 28, 60), 4, 1, True, 2, None, "quad_zcouple_kernel<double, 6>"),
    ((30, 27, 61), 6, 1, [0, 3, 7], 3, (0.07, -0.11), "quad_zcouple_kernel<double, 8>"),
    ((32, 30, 40), 8, 1, True, 5, (0.05, 0.02), "quad_zcouple_kernel<double, 9>"),
    ((32, 30, 41), 8, 1.5, True, 2, None, "quad_zcouple_kernel<double, 10>"),
    ((35, 30, 61), 9, 1, list(range(0, 90, 2)), 17, None, "quad_zcouple_kernel<double, 9>"),
    # two layers ten planes apart
    ((30, 28, 60), 2, 2, True, 3, (-0.03, 0.04), "quad_zcouple_kernel<double, 6>"),
])
def test_quadrupole_slab_matches_oracle(grid, support, layers, quads, B, kb, kernel):
    print(f"quad slab grid={grid} support={support} layers={layers} B={B}", flush=True)
    rng = np.random.default_rng(31)
    L = [23.0, 22.0, 40.0]
    N = 91
    h = L[2] / grid[2]
    z = 3 * h + rng.uniform(-0.4, 0.4, N) * h
    if layers == 1.5:  # every other particle one plane up
        z[::2] += h
    if layers == 2:
        z[::2] += 10 * h
    pos = np.stack([rng.uniform(-0.2, 1.2, N) * L[0], rng.uniform(0, 1, N) * L[1], z], 1)
    op = Op(L, 1e-6, 0.5, grid=grid, support=support, quads=quads)
    if kb is not None:
        op.set_bloch(*kb)
    op.set_positions(pos)
    sc = np.full(N, -0.3 + 0.05j)
    op.set_self_coef(sc)
    x = rng.standard_normal((B, op.n)) + 1j * rng.standard_normal((B, op.n))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(x, C.PREC_DOUBLE)
    C.profile_enable(False)
    assert kernel in C.profile_names(), C.profile_names()
    ref = _oracle(L, grid, support, pos, quads, kb)
    for b in sorted({0, B - 1}):
        assert rel(y[b], ref.apply(x[b], sc).reshape(-1)) < 1e-11, b
    r64 = op.apply(x, C.PREC_DOUBLE, C.PART_RECIP)
    assert rel(op.apply(x, C.PREC_MIXED, C.PART_RECIP), r64) < 1e-6
    # layout=1 keeps the full grid: the same operator
    full = Op(L, 1e-6, 0.5, grid=grid, support=support, quads=quads, layout=1)
    if kb is not None:
        full.set_bloch(*kb)
    full.set_positions(pos)
    assert rel(full.apply(x, C.PREC_DOUBLE, C.PART_RECIP), r64) < 1e-11


@pytest.mark.parametrize("grid,N,support,quads,B,contract", [
    ((24, 22, 20), 701, 8, True, 5, "contract_nb_mfma_kernel<double, 4, 4, true, 8, double>"),
    ((23, 21, 19), 700, 4, list(range(0, 700, 3)), 5, "contract_nb_mfma_kernel<double, 4, 4, false, 8, double>"),
    ((40, 36, 44), 190, 6, True, 17, "contract_full_mfma_kernel<double, 4, 8, 2, 8, double>"),
    ((40, 36, 45), 100, 6, True, 31, "contract_mfma_kernel<double, 4, 8, 2, false, 8, double>"),
    # up to 3072 particles x right-hand sides: gathered per particle
    ((24, 22, 20), 701, 8, True, 3, "quad_finish_kernel<64, true, double>"),
    ((23, 21, 19), 700, 4, list(range(0, 700, 3)), 2, "quad_finish_kernel<64, true, double>"),
    ((40, 36, 44), 60, 6, True, 4, "quad_finish_kernel<64, true, double>"),
    ((40, 36, 45), 60, 6, True, 1, "quad_finish_kernel<64, true, double>"),
    ((7, 9, 20), 50, 10, [1, 49], 2, "quad_finish_kernel<64, true, double>"),  # axes shorter than the stencil
    ((30, 28, 61), 3072, 4, True, 1, "quad_finish_kernel<64, true, double>"),
])
def test_quadrupole_full_grid_matches_oracle(grid, N, support, quads, B, contract):
    print(f"quad full grid={grid} N={N} support={support} B={B}", flush=True)
    rng = np.random.default_rng(37)
    L = [20.0, 18.0, 21.0]
    pos = rng.uniform(0, 1, (N, 3)) * L
    op = Op(L, 1e-6, 0.5, grid=grid, support=support, quads=quads)
    op.set_positions(pos)
    sc = np.full(N, 0.2 - 0.1j)
    op.set_self_coef(sc)
    x = rng.standard_normal((B, op.n)) + 1j * rng.standard_normal((B, op.n))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(x, C.PREC_DOUBLE)
    C.profile_enable(False)
    assert contract in C.profile_names(), C.profile_names()
    ref = _oracle(L, grid, support, pos, quads, None)
    for b in sorted({0, B - 1}):
        assert rel(y[b], ref.apply(x[b], sc).reshape(-1)) < 1e-11, b
    r64 = op.apply(x, C.PREC_DOUBLE, C.PART_RECIP)
    assert rel(op.apply(x, C.PREC_MIXED, C.PART_RECIP), r64) < 1e-6


def test_stages_of_a_slab_operator_work_on_the_full_grid():
    import ctypes
    print("quad stages after a slab apply", flush=True)
    rng = np.random.default_rng(41)
    L, grid, N = [23.0, 22.0, 40.0], (30, 28, 61), 80
    pos = np.stack([rng.uniform(0, 1, N) * L[0], rng.uniform(0, 1, N) * L[1], rng.uniform(-0.2, 0.2, N)], 1)
    op = Op(L, 1e-6, 0.5, grid=grid, support=8, quads=True)
    op.set_positions(pos)
    op.set_self_coef(np.full(N, 0.2 - 0.1j))
    assert op.info().slab_planes == 0
    x = rng.standard_normal((1, op.n)) + 1j * rng.standard_normal((1, op.n))
    y = op.apply(x)
    lib = C.load()
    size = ctypes.c_size_t()
    C.check(lib.mpm_op_grid_bytes(op.h, C.PREC_DOUBLE, ctypes.byref(size)))
    assert size.value == 8 * 30 * 28 * 61 * 16
    # the reference's stencils and coefficients by address, built when asked for
    ptr, nb = ctypes.c_void_p(), ctypes.c_size_t()
    for name, count in (("spread_coef", N * 729 * 8), ("spread_idxs", N * 729 * 4), ("scale_coef", 30 * 28 * 61 * 128)):
        C.check(lib.mpm_op_device_pointer(op.h, name.encode(), ctypes.byref(ptr), ctypes.byref(nb)))
        assert ptr.value and nb.value == count, name
    xb, gb, yb = C.DeviceBuffer(x.nbytes), C.DeviceBuffer(size.value), C.DeviceBuffer(x.nbytes)
    xb.upload(x)
    yb.upload(np.zeros_like(x))
    for stage in (C.STAGE_SPREAD, C.STAGE_SCALE, C.STAGE_CONTRACT, C.STAGE_REAL_SPACE):
        C.check(lib.mpm_op_stage(op.h, stage, xb.ptr, gb.ptr, yb.ptr, C.PREC_DOUBLE, None))
    out = np.zeros_like(x)
    yb.download(out)
    assert rel(out, y) < 1e-11
    assert rel(op.apply(x), y) < 1e-11  # as before the stages
