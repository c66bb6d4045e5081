"""The multigrid's dense last level: the inverse of a 9-point operator of at
most 64 cells. The operators are Galerkin products with weights of any sign, so
nothing bounds the pivots of the natural order; operators that have none are
inverted here, and steps whose last level has small ones are taken."""
import ctypes

import numpy as np
import pytest

import oracle as orc
import sayram_cases as sc
import sayram_gpu as sg
from conftest import rel_l2

# bands d|w|e|s|n|sw|se|nw|ne
OFFSETS = [(0, 0), (-1, 0), (1, 0), (0, -1), (0, 1), (-1, -1), (1, -1), (-1, 1), (1, 1)]


def _operator(nx, ny, kind, seed):
    """Nine bands (K = j nx + i; zero outside the grid) and the dense matrix."""
    rng = np.random.default_rng(seed)
    n = nx * ny
    bands, A = np.zeros((9, n)), np.zeros((n, n))
    for K in range(n):
        i, j = K % nx, K // nx
        for b, (di, dj) in enumerate(OFFSETS):
            if 0 <= i + di < nx and 0 <= j + dj < ny:
                v = rng.uniform(0.5, 2.0) * rng.choice([-1.0, 1.0])
                if b == 0:
                    v = {"dominant": 20.0, "zero": 0.0, "tiny": 1e-13 * v,
                         "last": 20.0 if K < n - 2 else 0.0}[kind] if n > 1 else v
                bands[b, K] = A[K, K + dj * nx + di] = v
    return bands, A


# Kinds: pivots in the natural order; none; useless ones; none for the last two
# rows alone. (A strip with a zero diagonal is singular if its length is odd.)
@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_PC32])
@pytest.mark.parametrize("kind", ["dominant", "zero", "tiny", "last"])
@pytest.mark.parametrize("shape", [(8, 8), (64, 1), (1, 64), (2, 32), (32, 2), (5, 7), (9, 7), (2, 2),
                                   (16, 1), (1, 2), (1, 1), (4, 4)])
def test_inverse_needs_no_natural_pivots(gpu_lib, shape, kind, precision):
    """Elimination with row pivoting has a forward error of about n cond(A) eps
    (growth is small for such bands); the FP32 V-cycle's inverse is that one
    rounded once, 2^-24 of each entry."""
    nx, ny = shape
    n = nx * ny
    bands, A = _operator(nx, ny, kind, 1000 * nx + ny)
    out = np.empty((n, n))
    p = ctypes.POINTER(ctypes.c_double)
    rc = gpu_lib.lib().sg_debug_dense_inverse(nx, ny, precision, bands.ctypes.data_as(p),
                                              out.ctypes.data_as(p))
    assert rc == gpu_lib.SG_OK, gpu_lib.lib().sg_last_error()
    ref = np.linalg.inv(A)
    tol = 8.0 * n * np.linalg.cond(A) * np.finfo(np.float64).eps
    tol += 2.0 ** -24 if precision != sg.SG_FP64 else 0.0
    assert np.isfinite(out).all() and rel_l2(out, ref) <= tol, (rel_l2(out, ref), tol)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("nx,ny,seed,dt", [(20, 20, 1, 1.0), (57, 61, 2, 100.0), (64, 64, 2, 1.0),
                                           (41, 33, 1, 1e-3), (16, 12, 1, 100.0)])
def test_large_steps_with_small_natural_pivots(gpu_lib, precision, nx, ny, seed, dt):
    """Steps of up to 100 days: the smallest pivot of the last level in the
    natural order is 7e-5 of its diagonal at 20 x 20. Within 1e-10 of the
    oracle, a step's specification."""
    p = sc.seeded_case(nx, ny, seed=seed)
    p.dt = dt
    s = gpu_lib.Solver(p, gpu_lib.make_opts(precision=precision))
    op, f = orc.OracleProblem(p), p.f0
    for _ in range(2):
        f = orc.step(op, f)
        s.update(1)
        assert rel_l2(s.f(), f) <= 1e-10
    s.close()


def test_dense_inverse_refuses_other_sizes():
    out = np.empty(1)
    p = ctypes.POINTER(ctypes.c_double)
    for nx, ny, prec in [(13, 5, 0), (65, 1, 0), (0, 4, 0), (65536, 65536, 0), (4, 4, 3)]:
        rc = sg.lib().sg_debug_dense_inverse(nx, ny, prec, out.ctypes.data_as(p), out.ctypes.data_as(p))
        assert rc == sg.SG_ERR_ARG, (nx, ny)
