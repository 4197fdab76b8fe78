"""Downloads through a context's two pinned buffers: sizes around the staged
limit (4 MiB) and the buffers (16 MiB), from several threads at once; and
downloads into page-locked memory, which do not take that way."""
import ctypes
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


def _device_file_maps():
    """Bytes of this process's mappings of the GPU's render node, where
    page-locked allocations of the runtime appear."""
    n = 0
    with open("/proc/self/maps") as f:
        for line in f:
            p = line.split()
            if len(p) > 5 and p[5].startswith("/dev/dri/render"):
                lo, hi = (int(x, 16) for x in p[0].split("-"))
                n += hi - lo
    return n


# 24 bytes into an allocation: a destination inside page-locked memory
@pytest.mark.parametrize("offset", [0, 24])
def test_page_locked_arrays_are_written_directly(offset):
    """A download into page-locked memory, whole or inside an allocation, does
    not allocate the two staging buffers: the first download into pageable
    memory after it still does (32 MiB of new mappings)."""
    lib = ca.lib()
    ctx = ca.Context(0)
    blk, th, cfg = ca.pgen_setup(2, 64, 128, 128)
    w = ca.pgen_init(2, 1, blk, th, cfg)
    run = ca.Run(ctx, blk, th, cfg)
    run.set_prim(w)
    mem = ctypes.c_void_p()
    assert lib.hipHostMalloc(ctypes.byref(mem), ctypes.c_size_t(w.nbytes + offset), 0) == 0
    try:
        dst = ctypes.cast(mem.value + offset, ctypes.POINTER(ctypes.c_double))
        assert lib.cg_run_block_get_prim_host(run.h, 0, dst) == 0
        got = np.ctypeslib.as_array(dst, w.shape).copy()
        before = _device_file_maps()
        want = run.prim()
        assert _device_file_maps() - before >= 32 << 20
        np.testing.assert_array_equal(got, want)
    finally:
        run.close()
        ctx.close()
        assert lib.hipHostFree(mem) == 0


def test_buffers_come_when_they_pay():
    """States of 7.6e6 B: the first four downloads of a context are the
    runtime's own, the fifth (33.5e6 B and more in all) allocates one buffer,
    later ones none; a large state then needs the second."""
    ctx = ca.Context(0)
    run, big = None, None
    try:
        blk, th, cfg = ca.pgen_setup(2, 64, 46, 46)
        w = ca.pgen_init(2, 1, blk, th, cfg)
        run = ca.Run(ctx, blk, th, cfg)
        run.set_prim(w)
        blk2, th2, cfg2 = ca.pgen_setup(2, 64, 128, 128)
        w2 = ca.pgen_init(2, 2, blk2, th2, cfg2)
        big = ca.Run(ctx, blk2, th2, cfg2)
        big.set_prim(w2)
        run.prim()  # and the device scratch of a download
        grown = []
        for r, x, b in [(run, w, blk)] * 7 + [(big, w2, blk2)]:
            before = _device_file_maps()
            got = r.prim()
            grown.append((_device_file_maps() - before) >> 20)
            sk, sj, si = b.interior()
            np.testing.assert_array_equal(got[:, sk, sj, si], x[:, sk, sj, si])
        print("MiB of new mappings: %s" % grown, flush=True)
        assert grown[:3] == [0, 0, 0] and grown[3] == 16 and grown[4:7] == [0, 0, 0]
        assert grown[7] >= 16  # the second buffer (and the larger device scratch)
    finally:
        for r in (run, big):
            if r:
                r.close()
        ctx.close()
