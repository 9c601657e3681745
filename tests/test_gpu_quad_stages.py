"""The single stages of a quadrupole operator whose applies run on the slab: on the caller's full
grid, the grids of an operator kept on the full grid (layout = 1), and with nothing of the
operator rebuilt, moved or allocated by them.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # ahead of the library: one HIP runtime for both

from cumpm_amd import _capi as C
from cumpm_amd.dev import MonodisperseEwaldElectricField
from gpu_helpers import Op, rel

pytestmark = pytest.mark.gpu

L, N = [23.0, 22.0, 40.0], 80


def make(grid, support, z_planes, quads, layout, kb=(0.0, 0.0)):
    rng = np.random.default_rng(73)
    z = np.empty(N)
    for k, p in enumerate(z_planes):
        z[k::len(z_planes)] = p * L[2] / grid[2]
    pos = np.stack([rng.uniform(-0.2, 1.2, N) * L[0], rng.uniform(0, 1, N) * L[1], z], 1)
    op = Op(L, 1e-6, 0.5, grid=grid, support=support, quads=quads, layout=layout)
    op.set_bloch(*kb)
    op.set_positions(pos)
    op.set_self_coef(np.full(N, 0.2 - 0.1j))
    return op


def address(op, name):
    ptr = ctypes.c_void_p()
    C.check(C.load().mpm_op_device_pointer(op.h, name.encode(), ctypes.byref(ptr), None))
    return ptr.value


def stages(op, x, precision):
    """Grid after the spread, grid after the transforms, contraction, and all four stages."""
    lib = C.load()
    size = ctypes.c_size_t()
    C.check(lib.mpm_op_grid_bytes(op.h, precision, ctypes.byref(size)))
    xb, gb, yb = C.DeviceBuffer(x.nbytes), C.DeviceBuffer(size.value), C.DeviceBuffer(x.nbytes)
    xb.upload(x)
    gb.upload(np.full(size.value, 0x7e, np.uint8))  # the spread writes every voxel
    yb.upload(np.zeros_like(x))
    out = []
    for stage in (C.STAGE_SPREAD, C.STAGE_SCALE, C.STAGE_CONTRACT, C.STAGE_REAL_SPACE):
        C.check(lib.mpm_op_stage(op.h, stage, xb.ptr, gb.ptr, yb.ptr, precision, None))
        if stage in (C.STAGE_SPREAD, C.STAGE_SCALE):
            a = np.zeros(size.value // (8 if precision == C.PREC_MIXED else 16),
                         np.complex64 if precision == C.PREC_MIXED else np.complex128)
            gb.download(a)
        else:
            a = np.zeros_like(x)
            yb.download(a)
        out.append(a)
    return out


@pytest.mark.parametrize("grid,support,z_planes,quads,kb", [
    ((30, 28, 61), 8, (0.2,), True, (0.0, 0.0)),
    ((30, 27, 60), 4, (5.3, 15.1), [0, 3, 7], (0.07, -0.11)),
    ((9, 11, 60), 4, (59.8,), True, (0.0, 0.0)),  # a stencil over the end of the box
    ((5, 6, 120), 6, (60.2,), [], (0.02, 0.0)),  # axes shorter than the stencil, no quadrupole
])
def test_stages_match_the_full_grid_operator(grid, support, z_planes, quads, kb):
    print(f"quad stages {grid} support={support}", flush=True)
    rng = np.random.default_rng(79)
    op = make(grid, support, z_planes, quads, 0, kb)
    full = make(grid, support, z_planes, quads, 1, kb)
    x = rng.standard_normal((1, op.n)) + 1j * rng.standard_normal((1, op.n))
    # FP32: one rounding of weight, product and sum for each particle on a voxel, and transforms of
    # at most 50,400 points, each below 1e-6 of the largest value
    for precision, tol in ((C.PREC_DOUBLE, 1e-12), (C.PREC_MIXED, 2e-6)):
        for a, b in zip(stages(op, x, precision), stages(full, x, precision)):
            assert rel(a, b) < tol


def test_stages_leave_the_operator_alone():
    print("quad stages beside applies", flush=True)
    rng = np.random.default_rng(83)
    op = make((30, 28, 61), 8, (0.2,), True, 0)
    x = rng.standard_normal((1, op.n)) + 1j * rng.standard_normal((1, op.n))
    C.profile_reset()
    C.profile_enable(True)
    y = op.apply(x)
    names = ("neighbor_list", "pair_coef", "particle_index", "fes_grid", "self_coef")
    before = [address(op, n) for n in names]
    assert all(before)
    assert not address(op, "fe_grid")  # the slab's grid is not the stages' grid
    assert rel(stages(op, x, C.PREC_DOUBLE)[3], y) < 1e-11
    C.profile_reset()
    # the same kernels on the same data: the same bits
    np.testing.assert_array_equal(op.apply(x), y)
    C.profile_enable(False)
    assert "quad_zcouple_kernel<double, 9>" in C.profile_names(), C.profile_names()
    assert [address(op, n) for n in names] == before


def test_first_stages_can_be_captured():
    print("captured quad stages", flush=True)
    lib = C.load()
    op = make((30, 28, 61), 8, (0.2,), True, 0)
    size = ctypes.c_size_t()
    C.check(lib.mpm_op_grid_bytes(op.h, C.PREC_DOUBLE, ctypes.byref(size)))
    dev = torch.device("cuda")
    gen = torch.Generator(device="cpu").manual_seed(5)
    x = torch.randn(op.n, 2, dtype=torch.float64, generator=gen).to(dev)
    g = torch.zeros(size.value // 8, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        for stage in (C.STAGE_SPREAD, C.STAGE_SCALE):
            C.check(lib.mpm_op_stage(op.h, stage, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(g.data_ptr()), None,
                                     C.PREC_DOUBLE, ctypes.c_void_p(side.cuda_stream)))
    full = make((30, 28, 61), 8, (0.2,), True, 1)
    for scale in (1.0, -2.0, 0.5):
        x.mul_(scale)
        graph.replay()
        torch.cuda.synchronize()
        want = stages(full, x.cpu().numpy().view(np.complex128).reshape(1, -1), C.PREC_DOUBLE)[1]
        assert rel(g.cpu().numpy().view(np.complex128), want) < 1e-12


def test_field_class_keeps_its_full_grid():
    print("field class grid", flush=True)
    rng = np.random.default_rng(89)
    ef = MonodisperseEwaldElectricField(*L, 1e-6, 0.5, True, solve_quadrupoles=True, precision="double",
                                        grid=(30, 28, 61), support=8)
    pos = np.stack([rng.uniform(0, 1, N) * L[0], rng.uniform(0, 1, N) * L[1], np.zeros(N)], 1)
    ef.update_particle_coordinates(pos[:, 0], pos[:, 1], pos[:, 2])
    ef.set_self_coef(0.2)
    ef.set_dipoles(rng.standard_normal((N, 3)) + 1j * rng.standard_normal((N, 3)))
    ef.calculate()
    a = np.zeros(8 * 30 * 28 * 61, np.complex128)
    assert ef.dev_fe_grid
    C.check(C.load().mpm_buffer_download(a.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(ef.dev_fe_grid), a.nbytes))
    ef.spread()
    ef.scale()
    b = np.zeros_like(a)
    C.check(C.load().mpm_buffer_download(b.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(ef.dev_fe_grid), b.nbytes))
    assert rel(a, b) < 1e-12
