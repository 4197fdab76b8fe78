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
