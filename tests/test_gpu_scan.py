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
