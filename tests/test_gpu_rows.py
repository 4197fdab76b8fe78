"""Implicit lines with eight lanes per line (rows.hpp) at the sizes where its
chunks of eight levels and groups of eight lines are partly filled: caller
arrays against the CPU oracle, runs against the one-lane kernels (an explicit
launch shape), which evaluate the same operations in the same order and must
agree bit for bit."""
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
# sides of the limits of the eight-lane kernels: short lines between walls
# 8,192, periodic lines 32,768 (5 x 5) and 16,384 (3 x 3).  Walled x3 lines of
# moist blocks this wide are refused (the shuffled species weights would lie
# past the end of w).
LIMITS = [(10, True, (64, 5, 128)), (10, True, (64, 5, 129)), (2, True, (64, 5, 129)),
          (10, False, (128, 5, 256)), (10, False, (128, 5, 257)), (12, False, (257, 128, 6)),
          (2, False, (128, 5, 128)), (2, False, (128, 5, 129)), (4, False, (129, 128, 6))]


@pytest.mark.parametrize("config,flag,walls,dims",
                         [(2,) + c for c in LIMITS] + [(4,) + c for c in LIMITS] +
                         [(2, 12, True, (129, 64, 6)), (2, 4, True, (129, 64, 6))])
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
    """Lines of 41 cells between walls, just above the 16,384 (5 x 5) and 12,288
    (3 x 3) that the eight-lane kernel takes at that height: the one-lane
    kernel's whole block equals its halves, which are below, bit for bit."""
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
