"""One quadrupole operator over several frames (a trajectory's use): every set_positions and
set_bloch against the oracle's operator at the same positions, FP64 to 1e-11 of the largest
value, where the occupied z-planes change their places and not their number.
"""
import ctypes

import numpy as np
import pytest

from cumpm_amd import _capi as C
from oracle import oracle as O
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu

L, GRID, N = [23.0, 22.0, 40.0], (30, 28, 60), 60


def layers(rng, z_planes):
    """Every other particle in the layer of each of two z grid planes."""
    z = np.empty(N)
    for k, p in enumerate(z_planes):
        z[k::2] = (p + rng.uniform(-0.3, 0.3, z[k::2].size)) * L[2] / GRID[2]
    return np.stack([rng.uniform(0, 1, N) * L[0], rng.uniform(0, 1, N) * L[1], z], 1)


def check(op, pos, x, sc, kb=None):
    ref = O.Operator(L, 1e-6, 0.5, grid=list(GRID), P=4)
    if kb is not None:
        ref.set_bloch(*kb)
    ref.set_positions(pos)
    ref.set_quads(None)
    y = op.apply(x)
    for b in range(len(x)):
        assert rel(y[b], ref.apply(x[b], sc).reshape(-1)) < 1e-11, b


@pytest.mark.parametrize("first,second", [
    ((5, 15), (5, 21)),   # two separated layers, another gap
    ((5, 10), (5, 15)),   # one run of ten planes, then two of five
    ((5, 15), (5, 10)),   # and back
    ((5, 15), (0, 10)),   # the same gap across the end of the box: another plane order
    ((5, 10), (57, 62)),  # one run across the end of the box
])
def test_frames_with_equally_many_planes(first, second):
    print(f"quad frames {first} {second}", flush=True)
    rng = np.random.default_rng(61)
    op = Op(L, 1e-6, 0.5, grid=GRID, support=4, quads=True)
    sc = np.full(N, -0.3 + 0.05j)
    x = rng.standard_normal((2, 8 * N)) + 1j * rng.standard_normal((2, 8 * N))
    C.profile_reset()
    C.profile_enable(True)
    for pos in (layers(rng, first), layers(rng, second)):
        op.set_positions(pos)
        op.set_self_coef(sc)
        check(op, pos, x, sc)
    C.profile_enable(False)
    assert "quad_zcouple_kernel<double, 10>" in C.profile_names(), C.profile_names()


def test_frames_with_bloch_vectors():
    print("quad frames with Bloch vectors", flush=True)
    rng = np.random.default_rng(67)
    op = Op(L, 1e-6, 0.5, grid=GRID, support=4, quads=True)
    sc = np.full(N, 0.2 - 0.1j)
    x = rng.standard_normal((1, 8 * N)) + 1j * rng.standard_normal((1, 8 * N))
    for planes, kb in (((5, 15), (0.0, 0.0)), ((5, 15), (0.07, -0.04)), ((5, 19), (0.07, -0.04)),
                       ((5, 10), (0.0, 0.03))):
        pos = layers(rng, planes)
        op.set_bloch(*kb)
        op.set_positions(pos)
        op.set_self_coef(sc)
        check(op, pos, x, sc, kb)


@pytest.mark.parametrize("n,B,layout", [(60, 5, 0), (60, 3, 1), (1, 1, 0), (1, 2, 1)])
def test_no_quadrupoles_equals_the_dipole_operator(n, B, layout):
    # vectors of 3N values: the gradient columns of the grid have nothing to read
    print(f"no quadrupoles n={n} B={B} layout={layout}", flush=True)
    rng = np.random.default_rng(71)
    pos = layers(rng, (5, 10))[:n]
    sc = np.full(n, -0.3 + 0.05j)
    x = rng.standard_normal((B, n, 3)) + 1j * rng.standard_normal((B, n, 3))
    y = []
    for quads in (None, []):
        op = Op(L, 1e-6, 0.5, grid=GRID, support=4, quads=quads, layout=layout)
        op.set_positions(pos)
        op.set_self_coef(sc)
        assert op.n == 3 * n
        y.append((op.apply(x), op.apply(x, C.PREC_MIXED)))
    assert rel(y[1][0], y[0][0]) < 1e-11
    # FP32 grids: 125 rounded products on either side of transforms of 50,400 points
    assert rel(y[1][1], y[0][0]) < 1e-6


def read(op, name, dtype):
    ptr, nb = ctypes.c_void_p(), ctypes.c_size_t()
    C.check(C.load().mpm_op_device_pointer(op.h, name.encode(), ctypes.byref(ptr), ctypes.byref(nb)))
    return ptr.value, fetch(ptr.value, nb.value // np.dtype(dtype).itemsize, dtype)


def fetch(address, count, dtype):
    out = np.zeros(count, dtype)
    C.check(C.load().mpm_buffer_download(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(address), out.nbytes))
    return out


ADDRESSES = (("spread_coef", np.float64), ("spread_coef_fp32", np.float32), ("spread_idxs", np.int32),
             ("scale_coef", np.float64))


def test_buffers_asked_for_stay_current():
    print("quad buffers by address over frames", flush=True)
    rng = np.random.default_rng(97)
    op = Op(L, 1e-6, 0.5, grid=GRID, support=4, quads=True)
    a, b = layers(rng, (5, 15)), layers(rng, (5, 19))

    def fresh(pos, kb):
        o = Op(L, 1e-6, 0.5, grid=GRID, support=4, quads=True)
        o.set_bloch(*kb)
        o.set_positions(pos)
        return o

    op.set_positions(a)
    got = {name: read(op, name, dt) for name, dt in ADDRESSES}
    for pos, kb in ((b, (0.0, 0.0)), (b, (0.07, -0.04)), (a, (0.07, -0.04))):
        op.set_bloch(*kb)
        op.set_positions(pos)
        want = fresh(pos, kb)
        for name, dt in ADDRESSES:  # the sizes stay, and so do the addresses
            address, old = got[name]
            np.testing.assert_array_equal(fetch(address, old.size, dt), read(want, name, dt)[1], err_msg=name)


def test_coefficients_asked_for_follow_the_tuned_grid():
    print("quad coefficients by address over a grown grid", flush=True)
    rng = np.random.default_rng(101)
    grid = (93, 87, 60)  # 3 x 31 and 3 x 29: 96 and 90 transform faster
    op = Op(L, 1e-6, 0.5, grid=grid, support=4, quads=True)
    pos = layers(rng, (5, 15))
    op.set_positions(pos)
    op.set_self_coef(np.zeros(N))
    assert read(op, "scale_coef", np.float64)[1].size == 16 * 93 * 87 * 60
    tuned = C.TuneInfo()
    C.check(C.load().mpm_op_autotune(op.h, 4, C.PREC_DOUBLE, C.TUNE_GRID | C.TUNE_FORCE, ctypes.byref(tuned)))
    print("tuned grid", list(tuned.grid), flush=True)
    want = Op(L, 1e-6, 0.5, grid=list(tuned.grid), support=4, quads=True)
    want.set_positions(pos)
    for name, dt in ADDRESSES:
        a, b = read(op, name, dt)[1], read(want, name, dt)[1]
        assert a.size == b.size, name
        np.testing.assert_array_equal(a, b, err_msg=name)


def test_small_cells_need_no_more_scratch_than_the_full_grid():
    # ten of 20 planes, rows of 33 padded to 48: two slab buffers would exceed the 64 MiB that
    # the full grid's 24 right-hand sides fit
    print("quad scratch", flush=True)
    rng = np.random.default_rng(109)
    grid, B = (33, 33, 20), 24
    z = np.where(np.arange(N) % 2 == 0, 4, 14) * L[2] / grid[2]
    pos = np.stack([rng.uniform(0, 1, N) * L[0], rng.uniform(0, 1, N) * L[1], z], 1)
    op = Op(L, 1e-6, 0.5, grid=grid, support=4, quads=True)
    op.set_positions(pos)
    op.set_self_coef(np.full(N, 0.2 - 0.1j))
    x = rng.standard_normal((B, op.n)) + 1j * rng.standard_normal((B, op.n))
    xb, yb = C.DeviceBuffer(x.nbytes), C.DeviceBuffer(x.nbytes)
    xb.upload(x)
    C.check(C.load().mpm_op_apply_noalloc(op.h, xb.ptr, yb.ptr, B, C.PREC_DOUBLE, C.PART_ALL, None))
    y = np.zeros_like(x)
    yb.download(y)
    assert rel(y, op.apply(x)) < 1e-12
