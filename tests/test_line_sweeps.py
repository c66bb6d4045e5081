"""The line sweeps with lines in registers at the edges of their run lengths:
line lengths around every length at which a kernel takes longer runs or fewer
lines per workgroup, few lines and many, odd and even."""
import numpy as np
import pytest
import scipy.sparse as sps
import scipy.sparse.linalg as spl

import oracle as orc
import sayram_cases as sc
import sayram_gpu as sg
from conftest import rel_l2

# lengths at and around the run limits, in each direction
LENGTHS = [63, 64, 65, 127, 128, 129, 255, 256, 257, 383, 384, 385, 511, 512, 513, 767, 768, 769, 1023,
           1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097]


def _step(p, f):
    """The oracle's assembly, solved by SuperLU (the oracle's own banded solve
    takes nx^2 per cell, too long for rows of thousands of cells)."""
    (d, w, e, s, n), R = orc.assemble(orc.OracleProblem(p), f)
    nx, N = p.nx, p.ncells
    if nx == 1:
        A = sps.diags([d, s[1:], n[:-1]], [0, -1, 1], format="csc")
    else:
        A = sps.diags([d, w[1:], e[:-1], s[nx:], n[:N - nx]], [0, -1, 1, -nx, nx], format="csc")
    return np.maximum(spl.spsolve(A, R).reshape(p.ny, nx).T, 0.0)


def _trajectory(probs, precision, tiles, steps):
    b = sg.Batch(sg.make_opts(precision=precision, line_tiles=tiles, coarse_tiles=tiles))
    slots = [b.add(p) for p in probs]
    f, its = [], []
    for _ in range(steps):
        b.step(1)
        f.append([b.f(s) for s in slots])
        its.append([b.stats(s)["last_iters"] for s in slots])
    b.close()
    return f, its


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("direction", ["rows", "columns"])
def test_run_lengths(gpu_lib, precision, direction):
    """Every step on the oracle (1e-10, the step's specification) and equal to
    the tiled sweeps' up to the solve tolerance; the sweeps are exact line
    solves either way, so the iterations agree up to one (MIXED counts inner
    ones)."""
    probs = []
    for k, n in enumerate(LENGTHS):
        for m in ((3, 18) if n < 600 else (5,)):
            nx, ny = (n, m) if direction == "rows" else (m, n)
            probs.append(sc.seeded_case(nx, ny, seed=500 + k, scale=10.0 ** (k % 3 - 1)))
    steps = 2
    f, its = _trajectory(probs, precision, (0, 0, 0, 0), steps)
    g, itg = _trajectory(probs, precision, (16, 161, 16, 769), steps)   # tile shapes
    for k, p in enumerate(probs):
        r = p.f0
        for n in range(steps):
            r = _step(p, r)
            assert rel_l2(f[n][k], r) <= 1e-10, (p.nx, p.ny, n)
            assert rel_l2(f[n][k], g[n][k]) <= 1e-11, (p.nx, p.ny, n)
            slack = 1 if precision != sg.SG_MIXED else 3
            assert abs(its[n][k] - itg[n][k]) <= slack, (p.nx, p.ny, n)


# widths around the columns, and heights around the rows, that a workgroup takes;
# lines of every run length; fused levels and dense ones
POISONED = ([(nx, 90) for nx in (15, 16, 17, 31, 32, 33, 63, 65, 129)]
            + [(90, ny) for ny in (15, 16, 17, 31, 33, 63, 65)]
            + [(300, 7), (600, 9), (1100, 5), (2100, 3), (7, 300), (9, 600), (5, 1100), (3, 2100), (2, 90),
               (90, 2), (8, 8), (5, 13), (70, 1), (1, 70), (130, 2), (256, 4), (90, 150), (70, 900)])


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("smoother,coarse,fuse", [(0, 0, 0), (0, 0, -1), (8, 8, -1), (13, 13, -1), (15, 0, 0)])
def test_steps_read_only_what_they_wrote(gpu_lib, precision, smoother, coarse, fuse):
    """A step in work arrays full of NaN equals the same step in memory that an
    earlier step used, bit for bit: an unsolved neighbour of a boundary line is
    not read, not even times a zero coupling, and what the vector loads read
    past the end of a line is not used. (With y-lines alone, 8, long rows do not
    converge: those steps are rejected after the same iterations either way.)"""
    probs = [sc.seeded_case(nx, ny, seed=600 + k) for k, (nx, ny) in enumerate(POISONED)]
    out = []
    for poison in (False, True):
        b = sg.Batch(sg.make_opts(precision=precision, smoother=smoother, coarse_smoother=coarse,
                                  fuse_cells=fuse))
        slots = [b.add(p) for p in probs]
        for _ in range(3):
            if poison:
                for s in slots:
                    b.debug_poison(s)
            rc = b.step_status(1)
            assert rc == sg.SG_OK or (smoother == 8 and rc == sg.SG_ERR_NOCONV)
        out.append([(b.f(s), b.stats(s)) for s in slots])
        b.close()
    for p, (f, st), (g, tg) in zip(probs, *out):
        assert np.isfinite(g).all() and np.array_equal(f, g), (p.nx, p.ny)
        assert all(st[k] == tg[k] for k in ("steps", "last_iters", "total_iters", "status")), (p.nx, p.ny)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_PC32])
def test_column_groups(gpu_lib, precision):
    """Widths around the columns per workgroup, on the oracle."""
    shapes = [(nx, 90) for nx in (15, 16, 17, 31, 32, 33, 63, 65, 129)] + [(90, 150), (70, 900)]
    probs = [sc.seeded_case(nx, ny, seed=600 + k) for k, (nx, ny) in enumerate(shapes)]
    out = []
    for smoother, coarse in ((0, 0), (8, 8)):
        b = sg.Batch(sg.make_opts(precision=precision, smoother=smoother, coarse_smoother=coarse))
        slots = [b.add(p) for p in probs]
        b.step(2)
        out.append([b.f(s) for s in slots])
        b.close()
    for k, p in enumerate(probs):
        r = _step(p, _step(p, p.f0))
        for o in out:
            assert np.isfinite(o[k]).all() and rel_l2(o[k], r) <= 1e-10, (p.nx, p.ny)
