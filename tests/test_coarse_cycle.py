"""The fused coarse cycle at the edges of what one workgroup takes: sides at
and around powers of two (a line occupies a power-of-two segment of a wave's
lanes) and around the largest side, around the size of the dense last level,
strips, single rows and columns."""
import pytest

import oracle as orc
import sayram_cases as sc
import sayram_gpu as sg
from conftest import rel_l2

SHAPES = [(64, 64), (64, 63), (63, 64), (65, 64), (64, 65), (33, 31), (32, 32), (31, 33), (17, 60),
          (60, 17), (5, 13), (13, 5), (4, 16), (7, 9), (16, 64), (64, 16), (8, 9), (3, 64), (64, 3), (2, 2), (2, 64), (1, 64), (64, 1),
          (1, 65), (70, 2), (128, 130)]


# Long thin levels: lines of two and four rows of 16 lanes, sides and cells at and
# past what is fused, columns whose lanes fit with four steps each only, last
# levels that are a line of more than 64 cells, levels fused below others.
LONG = [(66, 2), (2, 66), (65, 15), (15, 65), (70, 14), (113, 9), (9, 113), (128, 8), (8, 128), (129, 7),
        (204, 5), (5, 204), (255, 3), (3, 255), (256, 4), (4, 256), (256, 2), (2, 256), (130, 2),
        (2, 130), (257, 3), (3, 257), (256, 5), (512, 3), (3, 512), (150, 32), (32, 150), (520, 8), (9, 600)]


def _run(precision, smoother, coarse, fuse, steps, shapes=SHAPES):
    b = sg.Batch(sg.make_opts(precision=precision, smoother=smoother, coarse_smoother=coarse,
                              fuse_cells=fuse))
    probs = [sc.seeded_case(nx, ny, seed=300 + k, scale=10.0 ** (k % 3 - 1))
             for k, (nx, ny) in enumerate(shapes)]
    slots = [b.add(p) for p in probs]
    out, its = [], []
    for _ in range(steps):
        b.step(1)
        out.append([b.f(s) for s in slots])
        its.append([b.stats(s)["last_iters"] for s in slots])
    b.close()
    return probs, out, its


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("smoother,coarse", [(0, 0), (13, 13), (12, 12), (5, 4), (9, 8)])
def test_edges_of_the_fused_cycle(gpu_lib, precision, smoother, coarse):
    """Every step on the oracle (1e-10, the step's specification), equal to the
    per-level cycle up to the solve tolerance, and as strong: the two cycles
    are the same operator up to rounding, so they need the same iterations up
    to one."""
    # limits that fuse from level 0 of other shapes (above 1024 cells with FP32
    # V-cycles only; they have a kernel with larger LDS arrays)
    caps = [0, 1024, 256] if precision == sg.SG_FP64 else [0, 2048, 1024, 256]
    probs, per_level, its0 = _run(precision, smoother, coarse, -1, 3)
    for cap in caps:
        _, fused, its = _run(precision, smoother, coarse, cap, 3)
        for k, p in enumerate(probs):
            f = p.f0
            op = orc.OracleProblem(p)
            for n in range(3):
                f = orc.step(op, f)
                assert rel_l2(fused[n][k], f) <= 1e-10, (SHAPES[k], n)
                assert rel_l2(fused[n][k], per_level[n][k]) <= 1e-11, (SHAPES[k], n)
                slack = 1 if precision != sg.SG_MIXED else 3   # MIXED counts inner iterations
                assert abs(its[n][k] - its0[n][k]) <= slack, (SHAPES[k], n, its[n][k], its0[n][k])


def _launches(problem, precision, **opts):
    """Dispatches of the V-cycle's kernel families in one step of a solo batch."""
    b = sg.Batch(sg.make_opts(precision=precision, **opts))
    slot = b.add(problem)
    b.time_kernel("all")
    b.step(1)
    n = {k: b.kernel_time(k)[1] for k in ("line_l0", "line_coarse", "restrict", "prolong", "coarse_cycle")}
    f = b.f(slot)
    b.close()
    assert rel_l2(f, orc.step(orc.OracleProblem(problem), problem.f0)) <= 1e-10
    return n


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("shape", [(64, 1), (1, 64), (40, 1), (1, 3), (1, 1), (65, 1), (1, 900)])
def test_a_single_line_takes_line_solves(gpu_lib, shape, precision):
    """A grid of one row or column has one level, solved by a line solve per
    V-cycle whatever its length."""
    n = _launches(sc.seeded_case(*shape, seed=7), precision)
    assert n["line_coarse"] > 0
    assert n["coarse_cycle"] == n["line_l0"] == n["restrict"] == n["prolong"] == 0


# (schedules that smooth along both sides: x-lines alone take 100 iterations on a
# strip along y, and the solve then ends wherever the stall rule takes it)
@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("smoother,coarse", [(0, 0), (13, 13), (12, 12), (9, 8)])
def test_long_thin_levels(gpu_lib, precision, smoother, coarse):
    """As test_edges_of_the_fused_cycle, for levels with a side above 64."""
    probs, per_level, its0 = _run(precision, smoother, coarse, -1, 2, LONG)
    _, fused, its = _run(precision, smoother, coarse, 0, 2, LONG)
    for k, p in enumerate(probs):
        f, op = p.f0, orc.OracleProblem(p)
        for n in range(2):
            f = orc.step(op, f)
            assert rel_l2(fused[n][k], f) <= 1e-10, (LONG[k], n)
            assert rel_l2(fused[n][k], per_level[n][k]) <= 1e-11, (LONG[k], n)
            slack = 1 if precision != sg.SG_MIXED else 3
            assert abs(its[n][k] - its0[n][k]) <= slack, (LONG[k], n, its[n][k], its0[n][k])


@pytest.mark.gpu
@pytest.mark.parametrize("precision,shape,limit,fused", [
    (sg.SG_FP64, (64, 48), 0, True), (sg.SG_FP64, (64, 48), 1024, False),
    (sg.SG_FP64, (45, 22), 990, True), (sg.SG_FP64, (45, 22), 989, False),
    (sg.SG_FP64, (32, 32), 1023, False), (sg.SG_FP64, (32, 32), 1024, True),
    (sg.SG_FP64, (33, 32), 1024, False), (sg.SG_FP64, (33, 32), 0, True),
    (sg.SG_PC32, (64, 48), 0, True), (sg.SG_PC32, (64, 48), 4096, True),
    (sg.SG_PC32, (64, 48), 3071, False), (sg.SG_PC32, (64, 48), 2048, False),
    (sg.SG_MIXED, (64, 48), 1024, False), (sg.SG_MIXED, (64, 64), 4095, False),
    (sg.SG_MIXED, (64, 64), 4096, True), (sg.SG_PC32, (8, 9), 1, False)])
def test_fuse_cells_is_the_largest_fused_level(gpu_lib, precision, shape, limit, fused):
    """Every limit means itself: a grid is fused from level 0, with no launch for
    its own lines, exactly if it has at most that many cells (0: any that fits)."""
    n = _launches(sc.seeded_case(*shape, seed=7), precision, fuse_cells=limit)
    assert n["coarse_cycle"] > 0 and (n["line_l0"] == 0) == fused


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [sg.SG_FP64, sg.SG_MIXED, sg.SG_PC32])
@pytest.mark.parametrize("shape", [(66, 2), (2, 66), (130, 3), (130, 2), (2, 130), (256, 4), (4, 256),
                                   (70, 14), (64, 64), (33, 2)])
def test_one_launch_per_v_cycle(gpu_lib, shape, precision):
    """Grids that fit run their whole V-cycle in the fused cycle: no launch per
    level, whichever of the sides is the long one."""
    n = _launches(sc.seeded_case(*shape, seed=7), precision)
    assert n["coarse_cycle"] > 0
    assert n["line_l0"] == n["line_coarse"] == n["restrict"] == n["prolong"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("precision,size", [(sg.SG_FP64, 8), (sg.SG_PC32, 4)])
def test_bytes_of_the_restrictions(gpu_lib, precision, size):
    """The byte model of the restrictions, per V-cycle: from level 0 b and two
    weights per cell; below, after the x-line pre-sweep, six couplings, one x and
    one weight per even-row cell (its odd columns read two weights); and the
    coarse right-hand side."""
    b = sg.Batch(sg.make_opts(precision=precision, fuse_cells=-1))
    b.add(sc.seeded_case(256, 128, seed=3))
    b.time_kernel("all")
    b.step(1)
    n0, levels = 256 * 128, 5   # 256 x 128, .., 16 x 8 (dense: 8 x 4)
    per_cycle = size * (3 * n0 + n0 / 4)
    per_cycle += sum(size * (8 * n / 2 + n / 4) for n in (n0 / 4 ** l for l in range(1, levels)))
    _, launches, nbytes = b.kernel_time("restrict")
    # V-cycles that ran (those launched after convergence exit and move nothing)
    cycles = nbytes / per_cycle
    assert launches % levels == 0 and 1 <= round(cycles) <= launches // levels
    assert abs(cycles - round(cycles)) < 1e-9, cycles
    b.close()
