"""Downloads through a context's two pinned buffers: sizes around the staged
limit (4 MiB) and the buffers (16 MiB), from several threads at once."""
import threading

import numpy as np
import pytest

import canoe_amd as ca

pytestmark = pytest.mark.gpu


# 5 x 70 x 38 x 38 doubles 4.04e6 B (not staged), 46: 5.9e6 B, 134 x 134:
# 50.3e6 B (three buffers and a remainder)
@pytest.mark.parametrize("nh", [32, 40, 128])
def test_threads_share_a_context(nh):
    ctx = ca.Context(0)
    blk, th, cfg = ca.pgen_setup(2, 64, nh, nh)
    states = [ca.pgen_init(2, seed, blk, th, cfg) for seed in (1, 2)]
    runs = [ca.Run(ctx, blk, th, cfg) for _ in states]
    for run, w in zip(runs, states):
        run.set_prim(w)
    want = [run.prim().copy() for run in runs]
    assert not np.array_equal(want[0], want[1])
    bad = []

    def fetch(k):
        for _ in range(4):
            if not np.array_equal(runs[k].prim(), want[k]):
                bad.append(k)

    threads = [threading.Thread(target=fetch, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    sk, sj, si = blk.interior()
    for got, w in zip(want, states):
        np.testing.assert_array_equal(got[:, sk, sj, si], w[:, sk, sj, si])
    for run in runs:
        run.close()
