"""GPU tests of the saturation-guess network and the guided adjustment.

The device forward and gradient are checked against the oracle's bf16
emulation (tolerances below: the device accumulates in fp32 inside MFMA in
an order the oracle does not reproduce, so a bf16 rounding of an activation
can land on the other side of a tie), the training pairs bit for bit, and
the guided adjustment against the plain one (same tolerance, same result)
and against its iteration counts.
"""
import numpy as np
import pytest

import canoe_amd as ca
from canoe_amd import mlp as cm
import oracle_lib as orl

pytestmark = pytest.mark.gpu


def moist_states(dims=(32, 8, 8), seed=3):
    """(th, rho, ie, q) of the interior cells of the moist box: ie is the
    sensible internal energy density rho c_v T, q (3, n) mass fractions."""
    blk, th, cfg = ca.pgen_setup(4, *dims)
    w = ca.pgen_init(4, seed, blk, th, cfg)
    sk, sj, si = blk.interior()
    ivx = 1 + blk.nmass
    rho = w[0][sk, sj, si].ravel().copy()
    q = np.stack([w[n][sk, sj, si].ravel() for n in (1, 2, 3)]).copy()
    p = w[ivx + 3][sk, sj, si].ravel()
    cvd = th.rd / (th.gammad - 1)
    rv = th.rd * (1 + th.inv_mu_ratio_m1[0])
    qd = 1 - q.sum(0)
    R = th.rd * qd + rv * q[0]
    cv = cvd * qd + sum(cvd * (1 + th.cv_ratio_m1[n]) * q[n] for n in range(3))
    ie = rho * cv * p / (rho * R)
    return th, rho, ie, q


def supersaturated(th, rho, ie, q, n, seed):
    """n states drawn from the given cells with their water scaled by
    1.1..2.2 (all vapour) and the temperature shifted by -2..2 K (part of
    them stays sub-saturated)."""
    rng = np.random.default_rng(seed)
    b = rng.integers(0, rho.size, n)
    cvd = th.rd / (th.gammad - 1)
    cvv = cvd * (1 + th.cv_ratio_m1[0])
    cvp = cvd * (1 + th.cv_ratio_m1[2])
    r, qb = rho[b], q[:, b].copy()
    qd = 1 - qb.sum(0)
    cv = cvd * qd + cvv * qb[0] + cvd * (1 + th.cv_ratio_m1[1]) * qb[1] + cvp * qb[2]
    T = ie[b] / (r * cv) + rng.uniform(-2, 2, n)
    qn = qb.copy()
    qn[0] = (qb[0] + qb[1]) * rng.uniform(1.1, 2.2, n)
    qn[1] = 0.0
    qdn = 1 - qn.sum(0)
    cvn = cvd * qdn + cvv * qn[0] + cvp * qn[2]
    return r.copy(), r * cvn * T, np.ascontiguousarray(qn)


def test_params_round_trip_and_forward_matches_oracle(ctx):
    th, rho, ie, q = moist_states()
    x, t, _ = orl.mlp_pairs(th, rho, ie, q, 3000, seed=2)
    net = cm.Mlp(ctx, seed=5)
    try:
        p = net.params()
        assert p.size == cm.NPARAM and np.all(np.isfinite(p))
        p = p + np.float32(0.01) * np.random.default_rng(1).standard_normal(
            p.size).astype(np.float32)
        net.set_params(p)
        np.testing.assert_array_equal(net.params(), p)
        y = net.forward(x)
        yo = orl.mlp_forward(p, x, emulate=1)
        err = np.linalg.norm(y - yo) / np.linalg.norm(yo)
        print("forward rel L2 vs oracle %.3e, max abs %.3e"
              % (err, np.max(np.abs(y - yo))))
        assert err < 1e-3
        assert np.max(np.abs(y - yo)) < 1e-2 * max(1.0, np.max(np.abs(yo)))
    finally:
        net.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 255, 257])
def test_partly_filled_tiles_match_oracle(ctx, n):
    """Sample counts around the tiles of 16, the blocks of 64 and the gradient
    chunks of 256, with the bars of the full-size tests."""
    th, rho, ie, q = moist_states()
    x, t, _ = orl.mlp_pairs(th, rho, ie, q, 300, seed=8)
    x, t = np.ascontiguousarray(x[:n]), np.ascontiguousarray(t[:n])
    net = cm.Mlp(ctx, seed=9)
    try:
        p = net.params()
        y = net.forward(x)
        yo = orl.mlp_forward(p, x, emulate=1)
        assert np.linalg.norm(y - yo) < 1e-3 * np.linalg.norm(yo)
        g, loss = net.loss_grad(x, t)
        go, lo = orl.mlp_loss_grad(p, x, t, emulate=1)
        assert abs(loss - lo) <= 1e-4 * lo
        assert np.linalg.norm(g - go) < 1e-2 * np.linalg.norm(go)
    finally:
        net.close()


def test_forward_is_the_same_on_both_sides_of_the_tile_rule(ctx):
    """One and four sample tiles per wavefront: the same products per sample."""
    rng = np.random.default_rng(4)
    x = rng.uniform(-1, 1, ((1 << 21) + 1, 4)).astype(np.float32)
    net = cm.Mlp(ctx, seed=3)
    try:
        y = net.forward(x)
        np.testing.assert_array_equal(y[:70001], net.forward(x[:70001]))
        np.testing.assert_array_equal(y[-5:], net.forward(x[-5:]))
    finally:
        net.close()


def _gelu64(z):
    """tanh-form GELU, its derivative and |2 u| in 64 bits, by the sigmoid:
    (1 + tanh u) / 2 = 1 / (1 + e^(-2u))."""
    z = np.asarray(z, np.float64)
    u = np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3)
    e = np.exp(-np.clip(2 * u, -700, 700))
    s = 1 / (1 + e)
    dudz = np.sqrt(2 / np.pi) * (1 + 3 * 0.044715 * z * z)
    return z * s, s + 2 * z * (e * s * s) * dudz, np.abs(2 * u)


def _bf16(v):
    """Round to nearest even to the upper 16 bits of a float32."""
    b = np.asarray(v, np.float32).view(np.uint32).astype(np.uint64)
    return ((b + 0x7fff + ((b >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


# parameter offsets of the four layers: weights (outputs, inputs) and biases
W_AT, B_AT = (0, 320, 4480, 8640), (256, 4416, 8576, 8832)


@pytest.mark.parametrize("part", ["range", "large", "nan"])
def test_gelu_elementwise(ctx, part):
    """The device GELU of single numbers, read through a network that adds
    three bf16 parts of z, applies it once to that sum and passes the rounded
    result on (a weight of 2^100 takes it where GELU is the identity or zero,
    one unit per sign).  Bound: the bf16 number has to be that of a value
    within 1e-6 + 6e-7 |2u| (relative) of the 64-bit one, twice what the
    roundings of u, the 1-ulp exponential and the reciprocal add up to."""
    rng = np.random.default_rng(11)
    if part == "range":
        z = rng.uniform(-9, 12, 200001).astype(np.float32)
        small = 10.0 ** rng.uniform(-20, 0, 2000) * rng.choice([-1, 1], 2000)
        z = np.concatenate([z, small.astype(np.float32)])
        up = 2.0 ** 100
    else:
        z = (10.0 ** rng.uniform(1.1, 18, 4001) * rng.choice([-1, 1], 4001)).astype(np.float32)
        up = 1.0
        if part == "nan":
            z[5::16] = np.nan
    x = np.zeros((z.size, 4), np.float32)
    rest = z.copy()
    for c in range(3):  # truncated parts: their sum has no bit below z's
        x[:, c] = (rest.view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)
        rest = (rest - x[:, c]).astype(np.float32)
    p = np.zeros(cm.NPARAM, np.float32)
    p[W_AT[0]:W_AT[0] + 3] = 1.0
    p[W_AT[1]] = up
    p[W_AT[1] + 64] = -up
    for o in (0, 1):
        p[W_AT[2] + o * 64 + o] = 1.0
        p[W_AT[3] + o * 64 + o] = 1.0 / up
    net = cm.Mlp(ctx, seed=1)
    try:
        net.set_params(p)
        y = net.forward(x)
    finally:
        net.close()
    bad = np.isnan(z)
    assert np.all(np.isnan(y[bad][:, :2])) and np.all(np.isfinite(y[~bad]))
    got, z = (y[:, 0] - y[:, 1])[~bad], z[~bad]
    g, _, au = _gelu64(z)
    tol = np.abs(g) * (1e-6 + 6e-7 * np.minimum(au, 100))
    if part != "range":
        g = np.where(z > 0, g, 0.0)
        tol = np.where(z > 0, 0.0, 1e-30)
    assert np.all(_bf16(g - tol) <= got) and np.all(got <= _bf16(g + tol))


@pytest.mark.parametrize("lo,hi", [(-12.0, 12.0), (1.0, 18.0)])
def test_gelu_derivative_elementwise(ctx, lo, hi):
    """The device derivative of single numbers: with zero weights before it
    and one sample, layer 3 has its biases as pre-activations, a unit output
    weight sends the same power of two back to all of them, and the bias
    gradients are that times the derivative in fp32.  Bound 1e-6 absolute (1.1
    is its largest value; 16 roundings), also at |z| up to 1e18, where the
    derivative is one or zero."""
    rng = np.random.default_rng(12)
    net = cm.Mlp(ctx, seed=1)
    x = np.zeros((1, 4), np.float32)
    worst = 0.0
    try:
        for n in range(200 if hi == 12.0 else 40):
            if hi == 12.0:
                z = rng.uniform(lo, hi, 64).astype(np.float32)
                z[0] = 0.0
            else:
                z = (10.0 ** rng.uniform(lo, hi, 64)).astype(np.float32)
                z[::4] *= -1
            p = np.zeros(cm.NPARAM, np.float32)
            p[B_AT[2]:B_AT[2] + 64] = z
            p[W_AT[3]:W_AT[3] + 64] = 1.0
            net.set_params(p)
            y = float(net.forward(x)[0, 0])
            back = 2.0 ** np.floor(np.log2(abs(y) + 1.0))
            t = np.array([[y - 1.5 * back, 0, 0]], np.float32)
            grad, _ = net.loss_grad(x, t)
            got = grad[B_AT[2]:B_AT[2] + 64].astype(np.float64) / back
            worst = max(worst, np.max(np.abs(got - _gelu64(z)[1])))
    finally:
        net.close()
    print("derivative, z of %g..%g: largest error %.2e" % (lo, hi, worst), flush=True)
    assert worst <= 1e-6


def test_gradient_matches_oracle(ctx):
    th, rho, ie, q = moist_states()
    x, t, _ = orl.mlp_pairs(th, rho, ie, q, 1000, seed=4)
    net = cm.Mlp(ctx, seed=6)
    try:
        p = net.params()
        g, loss = net.loss_grad(x, t)
        go, lo = orl.mlp_loss_grad(p, x, t, emulate=1)
        g0, l0 = orl.mlp_loss_grad(p, x, t, emulate=0)
        print("loss gpu %.6e oracle %.6e exact %.6e" % (loss, lo, l0))
        assert abs(loss - lo) <= 1e-4 * lo
        o = 0
        for din, dout in ((4, 64), (64, 64), (64, 64), (64, 3)):
            for n in (din * dout, dout):
                a, b = g[o:o + n], go[o:o + n]
                e = np.linalg.norm(a - b) / np.linalg.norm(b)
                print("  block %d..%d rel L2 %.3e" % (o, o + n, e))
                assert e < 1e-2
                o += n
    finally:
        net.close()


def test_pairs_bit_exact(ctx):
    th, rho, ie, q = moist_states()
    x, t, it = cm.make_pairs(ctx, th, rho, ie, q, 5000, seed=8)
    xo, to, ito = orl.mlp_pairs(th, rho, ie, q, 5000, seed=8)
    np.testing.assert_array_equal(x, xo)
    np.testing.assert_array_equal(t, to)
    np.testing.assert_array_equal(it, ito)


def test_train_and_guided_adjustment(ctx):
    th, rho, ie, q = moist_states(dims=(48, 16, 16), seed=9)
    dx, dt, it = cm.make_pairs(ctx, th, rho, ie, q, 1 << 18, seed=12,
                               device=True)
    net = cm.Mlp(ctx, seed=13)
    try:
        losses = net.train(dx, dt, steps=20000, batch=8192, lr=3e-3,
                           lr_final=1e-5, seed=14)
        l0, l1 = losses[:20].mean(), losses[-100:].mean()
        print("training loss %.4e -> %.4e" % (l0, l1))
        assert np.all(np.isfinite(losses))
        assert l1 < 0.02 * l0
        # held-out pairs: temperature guess error
        xh, th_, ith = orl.mlp_pairs(th, rho, ie, q, 20000, seed=99)
        yh = net.forward(xh)
        sat = th_[:, 2] > 0
        rms = np.sqrt(np.mean((yh[sat, 0] - th_[sat, 0]) ** 2)) * 10.0
        print("held-out T guess rms error %.4f K (%d saturated)"
              % (rms, sat.sum()))
        assert rms < 0.5
        # guided vs plain adjustment on fresh supersaturated states
        r, e, qq = supersaturated(th, rho, ie, q, 50000, seed=21)
        ie_p, y_p, it_p = cm.saturation_adjust(ctx, th, r, e, qq)
        ie_g, y_g, it_g = cm.saturation_adjust(ctx, th, r, e, qq, net)
        ie_o, y_o, it_o, rc = orl.saturation_adjust(th, r, e, qq)
        assert rc == 0
        np.testing.assert_array_equal(ie_p, ie_o)
        np.testing.assert_array_equal(y_p, y_o)
        np.testing.assert_array_equal(it_p, it_o)
        np.testing.assert_allclose(ie_g, ie_p, rtol=1e-11, atol=0)
        np.testing.assert_allclose(y_g, y_p, rtol=0, atol=1e-13)
        s = it_p > 0
        mp, mg = it_p[s].mean(), it_g[s].mean()
        print("Newton iterations: plain %.3f guided %.3f (%d cells)"
              % (mp, mg, s.sum()))
        assert s.sum() > 10000
        assert np.all(it_g[~s] == 0)
        assert mg < 0.85 * mp
    finally:
        net.close()
        for d in (dx, dt):
            d.free()


def test_run_guided_adjustment_matches_newton(ctx):
    """A moist run with the guided adjustment (satadj = MLP) reproduces the
    plain Newton run and the oracle to the Newton tolerance."""
    from helpers import cfl_dt, perturbed_state, relerr
    blk, th, cfg, w = perturbed_state(4, (24, 8, 8), vel=1.0, dp=1e-3,
                                      cloud=True)
    sk, sj, si = blk.interior()
    # supersaturate the lower levels so that the adjustment condenses
    w[1][sk, sj, si][..., :12] *= 1.6
    w = ca.apply_bc_host(blk, w)
    dt = cfl_dt(blk, th, cfg, w, 0.6)
    u0 = orl.prim_to_cons(blk, th, w)
    ths, rho, ie, q = moist_states(dims=(24, 8, 8), seed=3)
    dx, dt_, _ = cm.make_pairs(ctx, th, rho, ie, q, 1 << 16, seed=5,
                               device=True)
    net = cm.Mlp(ctx, seed=6)
    try:
        net.train(dx, dt_, steps=2000, batch=4096)
        res = {}
        for mode in (ca.SATADJ_NEWTON, ca.SATADJ_MLP):
            cfg.satadj = mode
            run = ca.Run(ctx, blk, th, cfg)
            try:
                if mode == ca.SATADJ_MLP:
                    run.set_mlp(net)
                run.set_prim(w)
                run.step(dt, 2)
                res[mode] = run.cons()
            finally:
                run.close()
        cfg.satadj = ca.SATADJ_NEWTON
        uo, _ = orl.step(blk, th, cfg, dt, 2, u0, w)
        a = res[ca.SATADJ_MLP][:, sk, sj, si]
        b = res[ca.SATADJ_NEWTON][:, sk, sj, si]
        np.testing.assert_array_equal(b, uo[:, sk, sj, si])
        e = relerr(a, b)
        print("guided vs Newton run relerr %.3e" % e)
        # The two Newton iterations end within round-off of the same root;
        # the next stages amplify those ulp-level differences (the
        # hydrostatic decomposition subtracts nearly equal pressures) to
        # ~1e-11 after two steps, as any reordering of FP64 arithmetic does.
        assert e < 1e-9
        # the adjustment did condense
        assert np.max(b[2]) > 0
    finally:
        net.close()
        dx.free()
        dt_.free()
