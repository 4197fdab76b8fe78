"""The hydrostatic scan with several columns per workgroup at the heights
where its LDS share changes (255 and 1,023 cells with ghosts) and with columns
left over: x1 fluxes of caller arrays equal the CPU oracle."""
import numpy as np
import pytest

import canoe_amd as ca
import oracle_lib as orl
from helpers import perturbed_state, relerr

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the parity bar of every FP64 path; equal operations give 0


@pytest.mark.parametrize("config", [2, 4])
@pytest.mark.parametrize("dims", [(3, 3, 3), (249, 5, 3), (250, 4, 4), (1017, 3, 3),
                                  (1018, 3, 3), (16, 17, 1)])
@pytest.mark.parametrize("bc1", [(0, 0), (2, 2), (0, 2)])
def test_fluxes_at_scan_limits(ctx, config, dims, bc1):
    blk, th, cfg = ca.pgen_setup(config, *dims)
    blk.dx1 = 12000.0 / dims[0]
    w = ca.pgen_init(config, 3, blk, th, cfg)
    blk.bc[0], blk.bc[1] = bc1
    rng = np.random.default_rng(5)
    sk, sj, si = blk.interior()
    w[0][sk, sj, si] *= 1 + 1e-3 * rng.uniform(-1, 1, w[0][sk, sj, si].shape)
    w = ca.apply_bc_host(blk, w)
    print("scan config=%d dims=%s bc=%s" % (config, dims, bc1), flush=True)
    got = ca.Hydro(ctx, blk, th, cfg).calculate_fluxes(w)
    ref = orl.calculate_fluxes(blk, th, cfg, w)
    assert relerr(got[0], ref[0]) <= TOL


def test_scan_of_many_short_columns_of_a_run(ctx):
    """A run's explicit step takes one column per lane there: 75,076 columns of
    three levels equal their own smaller block (few columns: the scan in LDS)
    bit for bit."""
    blk, th, cfg = ca.pgen_setup(2, 3, 274, 274)
    cfg.implicit_flag = 0
    w = ca.pgen_init(2, 3, blk, th, cfg)
    one = ca.pgen_setup(2, 3, 5, 4)[0]
    one.dx1, one.dx2, one.dx3 = blk.dx1, blk.dx2, blk.dx3
    w[:] = w[:, 3:4, 3:4, :]
    ws = np.ascontiguousarray(w[:, :10, :11])
    out = []
    for b, x in ((blk, w), (one, ws)):
        run = ca.Run(ctx, b, th, cfg)
        try:
            run.set_prim(x)
            run.step(1e-3, 2)
            out.append(run.cons())
        finally:
            run.close()
    sk, sj, si = blk.interior()
    assert np.all(np.isfinite(out[0][:, sk, sj, si]))
    np.testing.assert_array_equal(out[0][:, 3:7, 3:8, si], out[1][:, 3:7, 3:8, si])
    np.testing.assert_array_equal(out[0][:, sk, sj, si],
                                  np.broadcast_to(out[0][:, 3:4, 3:4, si],
                                                  out[0][:, sk, sj, si].shape))


def _scan_ms(ctx, blks, th, cfg, w):
    run = ca.Run(ctx, None, th, cfg, blocks=blks)
    best = np.inf
    try:
        for b in range(len(blks)):
            run.set_prim(w, b)
        for _ in range(8):
            run.set_timing(True)
            run.step(1e-4, 1, graph=False)
            best = min(best, run.kernel_stats()["k_hydrostatic_scan"][0])
            run.set_timing(False)
    finally:
        run.close()
    return best


def test_scan_of_many_short_columns_takes_the_faster_kernel(ctx):
    """Half a million columns of four levels in one block against eight times
    an eighth of them (65,536, where both kernels take about 15 us): one
    launch takes 0.35 of the eight with one column per lane, 0.65 in LDS."""
    blk, th, cfg = ca.pgen_setup(2, 4, 512, 1024)
    part = ca.pgen_setup(2, 4, 512, 128)[0]
    cfg.implicit_flag = 0
    w = ca.pgen_init(2, 3, part, th, cfg)
    big = np.empty(blk.shape())
    big[:] = w[:, 3:4, 3:4, :]
    a = _scan_ms(ctx, [blk], th, cfg, big)
    b = _scan_ms(ctx, [part] * 8, th, cfg, w)
    print("one block %.4f ms, eight %.4f ms" % (a, b), flush=True)
    assert a <= 0.5 * b
