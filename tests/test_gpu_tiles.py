"""FP64 faces and divergence of 3D dry blocks by column tiles (fused64.hpp):
steps at sizes around the tile's 32 x 8 columns and its segments of levels
equal the CPU oracle."""
import time

import numpy as np
import pytest

import canoe_amd as ca
import oracle_lib as orl
from helpers import cfl_dt, perturbed_state, relerr

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the parity bar of every FP64 path; equal operations give 0


@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 32, 8), (17, 33, 9), (4, 31, 7),
                                  (34, 64, 17)])
@pytest.mark.parametrize("combo", [(5, 2, ca.RS_HLLC), (5, 5, ca.RS_LMARS),
                                   (2, 2, ca.RS_HLLC), (2, 5, ca.RS_LMARS)])
def test_step_at_tile_edges(ctx, dims, combo):
    blk, th, cfg, w = perturbed_state(2, dims, vel=1.0, dp=1e-3)
    cfg.order_h, cfg.order_v, cfg.rsolver = combo
    u = orl.prim_to_cons(blk, th, w)
    dt = cfl_dt(blk, th, cfg, w, 0.5)
    print("tiles dims=%s combo=%s" % (dims, combo), flush=True)
    uo, wo = orl.step(blk, th, cfg, dt, 2, u, w)
    sk, sj, si = blk.interior()
    # 16 is the length by rule, one level for every size here; the others are
    # taken as they are
    for seg in (16, 1, 5, 15):
        run = ca.Run(ctx, blk, th, cfg)
        try:
            run.set_tune(march_seg=seg)
            run.set_prim(w)
            run.step(dt, 2)
            got = run.cons()
        finally:
            run.close()
        assert np.all(np.isfinite(got[:, sk, sj, si]))
        assert relerr(got[:, sk, sj, si], uo[:, sk, sj, si]) <= TOL


@pytest.mark.parametrize("sides", [(0, 2), (2, 0), (2, 2)])
@pytest.mark.parametrize("combo", [(5, 2, ca.RS_LMARS), (5, 5, ca.RS_HLLC),
                                   (2, 2, ca.RS_LMARS), (2, 5, ca.RS_HLLC)])
def test_march_into_outflow_ghosts(ctx, combo, sides):
    """Segments whose windows of cells reach the ghosts beyond an outflow side,
    whose temperature and pressure are the last cell's, at their lower and
    upper end and in one go."""
    blk, th, cfg, w = perturbed_state(2, (17, 33, 9), vel=1.0, dp=1e-3)
    blk.bc[0], blk.bc[1] = sides
    w = ca.apply_bc_host(blk, w)
    cfg.order_h, cfg.order_v, cfg.rsolver = combo
    u = orl.prim_to_cons(blk, th, w)
    dt = cfl_dt(blk, th, cfg, w, 0.5)
    print("outflow tiles sides=%s combo=%s" % (sides, combo), flush=True)
    uo, wo = orl.step(blk, th, cfg, dt, 2, u, w)
    sk, sj, si = blk.interior()
    for seg in (17, 15):
        run = ca.Run(ctx, blk, th, cfg)
        try:
            run.set_tune(march_seg=seg)
            run.set_prim(w)
            run.step(dt, 2)
            got = run.cons()
        finally:
            run.close()
        assert np.all(np.isfinite(got[:, sk, sj, si]))
        assert relerr(got[:, sk, sj, si], uo[:, sk, sj, si]) <= TOL


@pytest.mark.parametrize("config", [2, 4])
@pytest.mark.parametrize("variant", [3, 4])
@pytest.mark.parametrize("combo", [(5, 2, ca.RS_HLLC), (5, 5, ca.RS_LMARS),
                                   (2, 2, ca.RS_HLLC), (2, 5, ca.RS_LMARS)])
def test_fp32_tiles_do_not_depend_on_the_segment(ctx, config, variant, combo):
    """The FP32-flux form's tiles march segments of any length to the same bits
    (an outflow top, whose ghosts the last window reads): one level, five with
    a remainder, the whole column, and the length by rule."""
    blk, th, cfg, w = perturbed_state(config, (17, 33, 9), vel=1.0, dp=1e-3)
    blk.bc[1] = 2
    w = ca.apply_bc_host(blk, w)
    cfg.order_h, cfg.order_v, cfg.rsolver = combo
    cfg.precision = ca.PREC_FP32
    dt = cfl_dt(blk, th, cfg, w, 0.5)
    print("fp32 segments config=%d variant=%d combo=%s" % (config, variant, combo), flush=True)
    sk, sj, si = blk.interior()
    want = None
    for seg in (1, 5, 17, 16):
        run = ca.Run(ctx, blk, th, cfg)
        try:
            run.set_tune(face_variant=variant, march_seg=seg)
            run.set_prim(w)
            run.step(dt, 2)
            got = run.cons()
        finally:
            run.close()
        assert np.all(np.isfinite(got[:, sk, sj, si]))
        want = got if want is None else want
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("prec", [ca.PREC_FP64, ca.PREC_FP32])
def test_runs_without_3d_blocks_plan_once(ctx, prec):
    """1,024 2D blocks, whose tile table is empty: a call of no steps takes as
    long as for a launch shape without tiles (FP32-flux face variant 2), since
    the blocks are not sorted and searched again (about half of the call)."""
    blk, th, cfg, w = perturbed_state(1, (8, 8, 1))
    runs, best = [], [np.inf, np.inf]
    try:
        for p, variant in ((ca.PREC_FP32, 2), (prec, 3)):
            cfg.precision = p
            run = ca.Run(ctx, None, th, cfg, blocks=[blk] * 1024)
            runs.append(run)
            run.set_tune(face_variant=variant)
        for _ in range(200):
            for k, run in enumerate(runs):
                t0 = time.perf_counter()
                run.step(1e-3, 0, graph=False)
                best[k] = min(best[k], time.perf_counter() - t0)
    finally:
        for run in runs:
            run.close()
    print("calls of no steps: %.1f and %.1f us" % (1e6 * best[0], 1e6 * best[1]), flush=True)
    assert best[1] <= 1.15 * best[0] + 2e-6
