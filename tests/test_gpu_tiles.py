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
    for seg in (16, 1, 5):
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


@pytest.mark.parametrize("prec", [ca.PREC_FP64, ca.PREC_FP32])
def test_runs_without_3d_blocks_plan_once(ctx, prec):
    """512 2D blocks, whose tile table is empty, with the longest march_seg: the
    search for a segment length (4,096 lengths over 512 blocks, 0.4 ms of host
    time and more) runs once and not on every call."""
    blk, th, cfg, w = perturbed_state(1, (8, 8, 1))
    cfg.precision = prec
    run = ca.Run(ctx, None, th, cfg, blocks=[blk] * 512)
    best = {}
    try:
        for seg in (1, 4096):
            run.set_tune(march_seg=seg)
            took = []
            for _ in range(20):
                t0 = time.perf_counter()
                run.step(1e-3, 0, graph=False)
                took.append(time.perf_counter() - t0)
            best[seg] = min(took)
    finally:
        run.close()
    print("calls of no steps: %s" % best, flush=True)
    assert best[4096] <= 2 * best[1] + 5e-5
