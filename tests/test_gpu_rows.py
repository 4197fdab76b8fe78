"""Implicit lines with eight lanes per line (rows.hpp) at the sizes where its
chunks of eight levels and groups of eight lines are partly filled: caller
arrays against the CPU oracle, runs against the one-lane kernels (an explicit
launch shape), which evaluate the same operations in the same order and must
agree bit for bit."""
import ctypes
import time

import numpy as np
import pytest

import canoe_amd as ca
import oracle_lib as orl
from helpers import cfl_dt, perturbed_state, relerr

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the parity bar of every FP64 path; equal operations give 0


def _increments(blk, seed):
    rng = np.random.default_rng(seed)
    du = rng.uniform(-1, 1, blk.shape())
    scale = [1e-4] * (1 + blk.nmass) + [1e-2, 1e-2, 1e-2, 10.0]
    return du * np.array(scale)[:, None, None, None]


@pytest.mark.parametrize("config", [2, 4])
@pytest.mark.parametrize("flag", [1, 9])
@pytest.mark.parametrize("dims", [(3, 3, 3), (7, 4, 3), (8, 8, 4), (9, 5, 5),
                                  (16, 4, 4), (17, 7, 3), (40, 33, 1)])
def test_caller_columns_equal_the_oracle(ctx, config, flag, dims):
    blk, th, cfg, w = perturbed_state(config, dims)
    du = _increments(blk, 3)
    print("columns config=%d flag=%d dims=%s" % (config, flag, dims), flush=True)
    got = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    ref, r = orl.implicit_solve(blk, th, du, w, 0.4, flag)
    assert r == 0
    sk, sj, si = blk.interior()
    assert relerr(got[:, sk, sj, si], ref[:, sk, sj, si]) <= TOL
    # ghost cells of du untouched
    got[:, sk, sj, si] = du[:, sk, sj, si]
    np.testing.assert_array_equal(got, du)


@pytest.mark.parametrize("flag", [2, 4, 10, 12])
@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 9, 8), (6, 17, 7)])
def test_caller_lines_between_walls_equal_the_oracle(ctx, flag, dims):
    blk, th, cfg, w = perturbed_state(2, dims)
    for s in range(2, 6):
        blk.bc[s] = ca.BC_REFLECT
    w = ca.apply_bc_host(blk, w)
    du = _increments(blk, 5)
    print("lines flag=%d dims=%s" % (flag, dims), flush=True)
    got = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    ref, r = orl.implicit_solve(blk, th, du, w, 0.4, flag)
    assert r == 0
    sk, sj, si = blk.interior()
    assert relerr(got[:, sk, sj, si], ref[:, sk, sj, si]) <= TOL


@pytest.mark.parametrize("config", [2, 4])
@pytest.mark.parametrize("flag", [1, 9])
@pytest.mark.parametrize("dims,bc1", [((3, 3, 3), (0, 0)), ((8, 9, 3), (0, 2)),
                                      ((9, 4, 5), (2, 0)), ((17, 13, 5), (2, 2)),
                                      ((33, 64, 3), (0, 0))])
def test_run_stage_equals_the_one_lane_kernels(ctx, config, flag, dims, bc1):
    """Three steps: u, w with every ghost, and (through the second and third
    step's fluxes) the hydrostatic pressures the sweep leaves."""
    blk, th, cfg, w = perturbed_state(config, dims, vel=1.0, dp=1e-3)
    blk.bc[0], blk.bc[1] = bc1
    w = ca.apply_bc_host(blk, w)
    cfg.implicit_flag = flag
    dt = cfl_dt(blk, th, cfg, w, 0.5)
    print("run config=%d flag=%d dims=%s bc=%s" % (config, flag, dims, bc1), flush=True)
    out = []
    for grid in (0, 1):
        run = ca.Run(ctx, blk, th, cfg)
        try:
            if grid:
                run.set_tune(implicit_grid=4096)
            run.set_prim(w)
            run.step(dt, 3)
            out.append((run.cons(), run.prim()))
        finally:
            run.close()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a[:, blk.interior()[0], blk.interior()[1]]))
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("flag", [2, 4, 10, 12, 15, 7])
@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 8, 9), (4, 9, 17), (3, 16, 10),
                                  (6, 25, 7), (9, 5, 11)])
def test_caller_periodic_lines_equal_the_oracle(ctx, flag, dims):
    """Periodic x2 / x3 lines whose last level falls on every place of a chunk
    of eight (lines of 9, 17 and 25 cells start with a chunk of seven)."""
    blk, th, cfg, w = perturbed_state(2, dims)
    du = _increments(blk, 7)
    print("periodic flag=%d dims=%s" % (flag, dims), flush=True)
    got = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    ref, r = orl.implicit_solve(blk, th, du, w, 0.4, flag)
    assert r == 0
    sk, sj, si = blk.interior()
    assert relerr(got[:, sk, sj, si], ref[:, sk, sj, si]) <= TOL


# (x2 lines are nx1 x nx3 of nx2 cells, x3 lines nx1 x nx2 of nx3) on both
# sides of the heights from which the eight-lane kernels take them, and of the
# numbers of lines that they never take.  Walled x3 lines of moist blocks this
# wide are refused (the shuffled species weights would lie past the end of w).
DRY = [(10, True, (64, 16, 128)), (10, True, (64, 17, 128)), (10, True, (64, 40, 129)),
       (2, True, (64, 27, 128)), (2, True, (64, 28, 128)),
       (12, True, (129, 64, 6)), (4, True, (129, 64, 6)),
       (10, False, (64, 6, 128)), (10, False, (64, 7, 128)),
       (10, False, (128, 16, 128)), (10, False, (128, 17, 128)),
       (10, False, (128, 5, 257)), (12, False, (257, 128, 6)),
       (2, False, (64, 27, 128)), (2, False, (64, 28, 128)),
       (2, False, (128, 5, 129)), (4, False, (129, 128, 6))]
MOIST = [(10, True, (64, 12, 128)), (10, True, (64, 13, 128)),
         (2, True, (64, 16, 128)), (2, True, (64, 17, 128)),
         (10, False, (64, 5, 128)), (10, False, (64, 6, 128)),
         (2, False, (64, 21, 128)), (2, False, (64, 22, 128)),
         (12, False, (257, 128, 6)), (4, False, (129, 128, 6))]


@pytest.mark.parametrize("config,flag,walls,dims",
                         [(2,) + c for c in DRY] + [(4,) + c for c in MOIST])
def test_caller_lines_on_both_sides_of_the_limits(ctx, config, flag, walls, dims):
    blk, th, cfg, w = perturbed_state(config, dims)
    if walls:
        for s in range(2, 6):
            blk.bc[s] = ca.BC_REFLECT
        w = ca.apply_bc_host(blk, w)
    du = _increments(blk, 9)
    print("limits config=%d flag=%d walls=%s dims=%s" % (config, flag, walls, dims), flush=True)
    got = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    ref, r = orl.implicit_solve(blk, th, du, w, 0.4, flag)
    assert r == 0
    sk, sj, si = blk.interior()
    assert relerr(got[:, sk, sj, si], ref[:, sk, sj, si]) <= TOL


@pytest.mark.parametrize("flag,dims", [(10, (128, 41, 130)), (2, (96, 41, 130)),
                                       (12, (128, 130, 41)), (4, (96, 130, 41))])
def test_many_tall_lines_equal_the_same_lines_in_halves(ctx, flag, dims):
    """Lines of 41 cells between walls: the whole block has too many of them for
    the eight-lane kernel at that height and goes to the one-lane kernel, its
    halves do not; both give the same bits."""
    blk, th, cfg, w = perturbed_state(2, dims)
    for s in range(2, 6):
        blk.bc[s] = ca.BC_REFLECT
    w = ca.apply_bc_host(blk, w)
    du = _increments(blk, 11)
    print("halves flag=%d dims=%s" % (flag, dims), flush=True)
    whole = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    axis = 2 if flag & 4 else 1  # arrays (n, k, j, i): cut across the lines
    n = dims[1] if flag & 4 else dims[2]
    hdims = list(dims)
    hdims[1 if flag & 4 else 2] = n // 2
    hb = perturbed_state(2, tuple(hdims))[0]
    for q in range(6):
        hb.bc[q] = blk.bc[q]
    hb.dx1, hb.dx2, hb.dx3 = blk.dx1, blk.dx2, blk.dx3
    for lo in (0, n // 2):
        cut = [slice(None)] * 4
        cut[axis] = slice(lo, lo + n // 2 + 6)  # with three ghosts either side
        cut = tuple(cut)
        half = ca.ImplicitSolver(ctx, hb, th, flag).solve_implicit_3d(
            np.ascontiguousarray(du[cut]), np.ascontiguousarray(w[cut]), 0.4)
        sk, sj, si = hb.interior()
        np.testing.assert_array_equal(half[:, sk, sj, si], whole[cut][:, sk, sj, si])


@pytest.mark.parametrize("config,flag,dims", [
    (2, 9, (12, 64, 128)), (2, 9, (13, 64, 128)), (2, 9, (5, 130, 130)), (2, 9, (52, 130, 130)),
    (2, 1, (19, 64, 128)), (2, 1, (20, 64, 128)), (2, 1, (5, 130, 130)),
    (4, 9, (13, 64, 128)), (4, 9, (14, 64, 128)), (4, 9, (5, 130, 130)),
    (4, 1, (18, 64, 128)), (4, 1, (19, 64, 128)), (4, 1, (5, 130, 130))])
@pytest.mark.parametrize("bc1", [(0, 0), (2, 2)])
def test_caller_columns_on_both_sides_of_the_limits(ctx, config, flag, dims, bc1):
    """x1 columns of caller arrays that one or eight lanes take."""
    blk, th, cfg, w = perturbed_state(config, dims)
    blk.bc[0], blk.bc[1] = bc1
    w = ca.apply_bc_host(blk, w)
    du = _increments(blk, 13)
    print("columns config=%d flag=%d dims=%s" % (config, flag, dims), flush=True)
    got = ca.ImplicitSolver(ctx, blk, th, flag).solve_implicit_3d(du, w, 0.4)
    ref, r = orl.implicit_solve(blk, th, du, w, 0.4, flag)
    assert r == 0
    sk, sj, si = blk.interior()
    assert relerr(got[:, sk, sj, si], ref[:, sk, sj, si]) <= TOL


def _solve_us(ctx, dims, flag, walls):
    """Best time of a solve on resident arrays, microseconds; walls: whether
    the x2 / x3 sides are walls, or the two x1 sides."""
    lib = ca.lib()
    blk, th, cfg, w = perturbed_state(2, dims)
    if isinstance(walls, tuple):
        blk.bc[0], blk.bc[1] = walls
    elif walls:
        for s in range(2, 6):
            blk.bc[s] = ca.BC_REFLECT
        w = ca.apply_bc_host(blk, w)
    du, ww = ctx.array(_increments(blk, 1)), ctx.array(w)
    best = np.inf
    try:
        for _ in range(25):
            t0 = time.perf_counter()
            r = lib.cg_implicit_solve(ctx.h, ctypes.byref(blk), ctypes.byref(th), du.ptr,
                                      ww.ptr, 0.01, flag)
            best = min(best, time.perf_counter() - t0)
            assert r == 0
    finally:
        du.free()
        ww.free()
    return 1e6 * best


# Short lines just below a number of lines that only the one-lane kernels
# take, and just above it: the fewer must not take longer.  With eight lanes
# for every such line they took 1.3 (walls), 2.1 and 1.4 (periodic) times as
# long.
@pytest.mark.parametrize("few,many,flag,walls,bar", [
    ((64, 5, 128), (64, 5, 136), 10, True, 1.15), ((64, 8, 128), (64, 8, 136), 2, True, 1.15),
    ((128, 5, 128), (128, 5, 136), 2, False, 1.3), ((128, 5, 250), (128, 5, 264), 10, False, 1.3)])
def test_fewer_short_lines_take_no_longer(ctx, few, many, flag, walls, bar):
    a, b = _solve_us(ctx, few, flag, walls), _solve_us(ctx, many, flag, walls)
    print("lines %s %.1f us, %s %.1f us" % (few, a, many, b), flush=True)
    assert a <= bar * b


@pytest.mark.parametrize("flag", [9, 1])
def test_short_columns_take_the_faster_kernel(ctx, flag):
    """Columns of five levels between walls against the same with one periodic
    side, which only the eight-lane kernel takes: one lane per column needs
    about 0.3 of its time there."""
    a = _solve_us(ctx, (5, 400, 400), flag, (0, 0))
    b = _solve_us(ctx, (5, 400, 400), flag, (0, ca.BC_PERIODIC))
    print("one lane %.1f us, eight lanes %.1f us" % (a, b), flush=True)
    assert a <= 0.6 * b


@pytest.mark.parametrize("config,flag,dims", [(2, 9, (3, 64, 128)), (2, 1, (8, 64, 128)),
                                              (4, 9, (8, 64, 128)), (2, 9, (40, 128, 127))])
def test_default_column_solve_is_not_the_slower_one(ctx, config, flag, dims):
    """A run's column solve by the default launch shape against the one-lane
    kernel (a grid of its own), at sizes where eight lanes would take 1.2 to
    1.9 times as long."""
    blk, th, cfg, w = perturbed_state(config, dims, vel=1.0, dp=1e-3)
    cfg.implicit_flag = flag
    best = {}
    run = ca.Run(ctx, blk, th, cfg)
    try:
        run.set_prim(w)
        for grid in (0, 4096):
            run.set_tune(implicit_grid=grid)
            best[grid] = np.inf
            for _ in range(10):
                run.set_timing(True)
                run.step(1e-3, 1, graph=False)
                ms, n = run.kernel_stats()["k_implicit_fused"]
                run.set_timing(False)
                best[grid] = min(best[grid], ms / n)
    finally:
        run.close()
    print("default %.4f ms, one lane %.4f ms" % (best[0], best[4096]), flush=True)
    assert best[0] <= 1.12 * best[4096]
