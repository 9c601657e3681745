"""The neighbour search's two forms (a wave or a thread per particle) on either side of the rule
that chooses between them: the pairs of a periodic k-d tree, and pair values interpolated in the
operator's tables (1e-12 of the largest value)."""
import ctypes

import numpy as np
import pytest
from scipy.spatial import cKDTree

from cumpm_amd import _capi as C
from gpu_helpers import Op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,neighbors", [
    (28000, 8), (36000, 8),    # short lists: waves, threads
    (45000, 19), (60000, 19),  # the same at 14 candidates a run
    (70000, 30),               # long lists: waves
])
def test_pairs_match_kd_tree(N, neighbors):
    print(f"neighbour search N={N} neighbors={neighbors}", flush=True)
    rng = np.random.default_rng(107)
    rc = np.sqrt(-np.log(1e-6)) / 0.5
    L = float((N * 4.0 / 3.0 * np.pi * rc ** 3 / neighbors) ** (1 / 3))
    op = Op([L] * 3, 1e-6, 0.5, grid=(16, 16, 16), support=4, layout=1)
    pos = rng.uniform(0, L, (N, 3))
    op.set_positions(pos)
    assert abs(op.info().rc - rc) < 1e-12
    lib = C.load()
    M = ctypes.c_int64()
    C.check(lib.mpm_op_get_neighbors(op.h, None, None, None, None, 0, ctypes.byref(M)))
    start, j = np.zeros(N + 1, np.int64), np.zeros(M.value, np.int32)
    perp, para = np.zeros(M.value), np.zeros(M.value)
    C.check(lib.mpm_op_get_neighbors(op.h, start.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                                     j.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), C.dptr(perp), C.dptr(para),
                                     M.value, ctypes.byref(M)))
    i = np.repeat(np.arange(N), np.diff(start))
    pairs = cKDTree(pos, boxsize=L).query_pairs(rc, output_type="ndarray")
    want = np.sort(np.concatenate([pairs[:, 0] * N + pairs[:, 1], pairs[:, 1] * N + pairs[:, 0]]))
    np.testing.assert_array_equal(np.sort(i * N + j), want)
    d = pos[i] - pos[j]
    d = np.maximum(np.linalg.norm(d - L * np.round(d / L), axis=1), 1.0)
    size = ctypes.c_int64()
    C.check(lib.mpm_op_get_pair_table(op.h, 0, None, None, 0, ctypes.byref(size)))
    for which, got in ((0, perp), (1, para)):
        r, v = np.zeros(size.value), np.zeros(size.value)
        C.check(lib.mpm_op_get_pair_table(op.h, which, C.dptr(r), C.dptr(v), size.value, ctypes.byref(size)))
        assert np.abs(got - np.interp(d, r[1:], v[1:])).max() < 1e-12 * np.abs(v).max()
