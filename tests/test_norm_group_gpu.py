"""Group normalisation of groups that fit a workgroup (at most 4 chunks of
4096 floats, one launch per direction) against the two-pass kernels, bit for
bit, and against float64.

Tolerances: the statistics are double, rounded once to fp32 (mean) and twice
(rstd, with the hardware rsqrt's ulp), so y = (x - mean) r is within
2^-24 (|x| + |mean|) r + 8 2^-24 |y|; dx has a few roundings per term of
r (dy - s / N - y t / N), and t = sum(dy y) adds products rounded to fp32, each
within 2^-24 |dy y|: t / N is within 2^-24 mean(|dy y|)."""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu
EPS = 1e-5
U = 2.0 ** -24


def silu(x):
    return x / (1 + np.exp(-x))


def silu_grad(x):
    s = 1 / (1 + np.exp(-x))
    return s * (1 + x * (1 - s))


# (batch, channels, hw, groups): group sizes of one element, around each chunk
# count's edge, no multiple of 4, the largest that fits (16384) and past it, and
# more groups than CUs
@pytest.mark.parametrize("b,c,hw,g", [
    (3, 4, 1, 4), (2, 4, 49, 4), (1, 2, 4095, 2), (2, 3, 4096, 3), (1, 2, 4097, 2), (2, 2, 8192, 2), (1, 3, 8196, 3),
    (2, 2, 12289, 2), (3, 4, 16384, 4), (1, 2, 16388, 2), (2, 1, 20481, 1), (1, 1, 1, 1), (5, 64, 196, 8),
    (5, 64, 8200, 64), (5, 64, 8201, 64), (9, 32, 16384, 32)])
@pytest.mark.parametrize("acc", [0, 1])
def test_norm_whole_group(hip, b, c, hw, g, acc):
    r = rng(b + c + hw + g + acc)
    n, m = b * c * hw, c // g * hw
    x = (r.standard_normal(n, dtype=np.float32) * 2 + np.float32(0.5)).astype(np.float32)
    da, dy0, dx0, cb = (r.standard_normal(k, dtype=np.float32) for k in (n, n, n, c))
    B, kind = hip.Buffer.from_array, hip.ACT["silu"]
    nb = hip.lib().mle_norm_ws_bytes(b, c, hw, g)
    ws, gx, gz, gda, gcb = hip.Buffer(nb), B(x), B(np.zeros(n, np.float32)), B(da), B(cb)
    new = lambda k=n: B(np.full(k, np.nan, np.float32))  # noqa: E731
    dims = (b, c, hw, g, EPS)

    def fwd(ready):
        y, a, st = new(), new(), new(2 * b * g)
        if ready:  # the two-pass route: the statistics come from the producing add
            hip.call("mle_add_norm_partials", None, gx.ptr, gz.ptr, n, new().ptr, b, c, hw, g, ws.ptr, nb)
        if acc and hw % 4 == 0:  # with the broadcast channel add
            hip.call("mle_norm_fwd_act_bias", None, gx.ptr, y.ptr, a.ptr, kind, gcb.ptr, st.ptr, *dims, ws.ptr, nb, ready)
        else:
            hip.call("mle_norm_fwd_act", None, gx.ptr, y.ptr, a.ptr, kind, st.ptr, *dims, ws.ptr, nb, ready)
        y2, st2 = new(), new(2 * b * g)
        hip.call("mle_norm_fwd_ex", None, gx.ptr, y2.ptr, st2.ptr, *dims, ws.ptr, nb, ready)
        np.testing.assert_array_equal(y.numpy(), y2.numpy())
        np.testing.assert_array_equal(st.numpy(), st2.numpy())
        return y, a, st

    y, a, st = fwd(0)
    for one, two in zip((y, a, st), fwd(1)):
        np.testing.assert_array_equal(one.numpy(), two.numpy())
    x64 = x.astype(np.float64).reshape(b * g, m)
    mean, var = x64.mean(1, keepdims=True), x64.var(1, keepdims=True)
    rs = 1 / np.sqrt(var + EPS)
    want = (x64 - mean) * rs
    got = y.numpy().astype(np.float64).reshape(b * g, m)
    assert np.all(np.abs(got - want) <= U * (np.abs(x64) + np.abs(mean)) * rs + 8 * U * np.abs(want))

    dy, dx, dx2 = B(dy0), B(dx0), B(dx0)
    hip.call("mle_norm_bwd_act", None, y.ptr, gda.ptr, kind, dy.ptr, acc, dx.ptr, st.ptr, *dims, 0, ws.ptr, nb, acc)
    dy2, dxa = B(dy0), new()
    hip.call("mle_norm_bwd_partials", None, y.ptr, dy2.ptr, gda.ptr, kind, acc, b, c, hw, g, 0, ws.ptr, nb)
    hip.call("mle_norm_bwd_apply_add", None, y.ptr, dy2.ptr, dx2.ptr, acc, None, dxa.ptr, 0, None, 0, st.ptr, *dims, 0,
             ws.ptr, nb)
    np.testing.assert_array_equal(dy.numpy(), dy2.numpy())
    np.testing.assert_array_equal(dx.numpy(), dx2.numpy())
    dx3 = B(dx0)
    hip.call("mle_norm_bwd", None, y.ptr, dy.ptr, dx3.ptr, st.ptr, *dims, 0, ws.ptr, nb, acc)
    np.testing.assert_array_equal(dx.numpy(), dx3.numpy())
    g64, y64 = dy.numpy().astype(np.float64).reshape(b * g, m), got
    sg, sgy = g64.mean(1, keepdims=True), (g64 * y64).mean(1, keepdims=True)
    rs = 1 / np.sqrt(st.numpy().astype(np.float64).reshape(b * g, 2)[:, 1:] / m + EPS)
    grad = rs * (g64 - sg - y64 * sgy)
    mag = rs * (np.abs(g64) + np.abs(sg) + np.abs(y64) * (np.abs(sgy) + np.abs(g64 * y64).mean(1, keepdims=True)))
    old = dx0.astype(np.float64).reshape(b * g, m) * acc
    assert np.all(np.abs(dx.numpy().reshape(b * g, m) - (old + grad)) <= 8 * U * (mag + np.abs(old)))
    # the activation's backward in the same pass
    want_dy = dy0.astype(np.float64) * acc + silu_grad(y.numpy().astype(np.float64)) * da
    assert np.all(np.abs(dy.numpy() - want_dy) <= 32 * U * (np.abs(want_dy) + np.abs(da) + np.abs(dy0) * acc))
    if not (acc and hw % 4 == 0):
        assert np.all(np.abs(a.numpy() - silu(y.numpy().astype(np.float64))) <= 16 * U * np.abs(a.numpy()) + 1e-30)


# groups of 3 and 4 chunks on both sides of the rule between one kernel and two
# passes: few groups, just enough, more than CUs; aligned and not (odd sizes)
@pytest.mark.parametrize("groups,m", [(16, 16384), (135, 16384), (136, 16384), (181, 12288), (182, 12288), (300, 12288),
                                      (320, 16384), (427, 12288), (16, 11529), (134, 11529), (100, 16165), (300, 11529)])
@pytest.mark.parametrize("act", ["relu", "gelu", "silu"])
def test_norm_group_rule(hip, groups, m, act):
    """Whichever route a call takes, its results are the two passes' bit for bit."""
    r = rng(groups + m)
    n = groups * m
    x, da = (r.standard_normal(n, dtype=np.float32) for _ in range(2))
    B, kind = hip.Buffer.from_array, hip.ACT[act]
    nb = hip.lib().mle_norm_ws_bytes(groups, 1, m, 1)
    ws, gx, gda, gz = hip.Buffer(nb), B(x), B(da), hip.Buffer.zeros(n)
    new = lambda k=n: hip.Buffer.zeros(k)  # noqa: E731
    dims = (groups, 1, m, 1, EPS)
    y, a, st, y2, a2, st2 = new(), new(), new(2 * groups), new(), new(), new(2 * groups)
    hip.call("mle_norm_fwd_act", None, gx.ptr, y.ptr, a.ptr, kind, st.ptr, *dims, ws.ptr, nb, 0)
    hip.call("mle_add_norm_partials", None, gx.ptr, gz.ptr, n, new().ptr, groups, 1, m, 1, ws.ptr, nb)
    hip.call("mle_norm_fwd_act", None, gx.ptr, y2.ptr, a2.ptr, kind, st2.ptr, *dims, ws.ptr, nb, 1)
    for one, two in ((y, y2), (a, a2), (st, st2)):
        np.testing.assert_array_equal(one.numpy(), two.numpy())
    dy, dx, dy2, dx2 = new(), new(), new(), new()
    hip.call("mle_norm_bwd_act", None, y.ptr, gda.ptr, kind, dy.ptr, 0, dx.ptr, st.ptr, *dims, 0, ws.ptr, nb, 0)
    hip.call("mle_norm_bwd_partials", None, y.ptr, dy2.ptr, gda.ptr, kind, 0, groups, 1, m, 1, 0, ws.ptr, nb)
    hip.call("mle_norm_bwd_apply_add", None, y.ptr, dy2.ptr, dx2.ptr, 0, None, new().ptr, 0, None, 0, st.ptr, *dims, 0,
             ws.ptr, nb)
    for one, two in ((dy, dy2), (dx, dx2)):
        np.testing.assert_array_equal(one.numpy(), two.numpy())


@pytest.mark.parametrize("groups,m", [(3, 4096), (2, 11529), (300, 16384), (2, 40000), (2, 40001)])
def test_norm_gradient_added_with_one_rounding(hip, groups, m):
    """dx += g rounds once: added to the negative of the rounded gradient it leaves
    what that rounding dropped, not 0."""
    r = rng(groups + m)
    n = groups * m
    B = hip.Buffer.from_array
    nb = hip.lib().mle_norm_ws_bytes(groups, 1, m, 1)
    ws, x, dy = hip.Buffer(nb), B(r.standard_normal(n, dtype=np.float32)), B(r.standard_normal(n, dtype=np.float32))
    y, st, g = hip.Buffer.zeros(n), hip.Buffer.zeros(2 * groups), hip.Buffer.zeros(n)
    dims = (groups, 1, m, 1, EPS)
    hip.call("mle_norm_fwd_ex", None, x.ptr, y.ptr, st.ptr, *dims, ws.ptr, nb, 0)
    hip.call("mle_norm_bwd", None, y.ptr, dy.ptr, g.ptr, st.ptr, *dims, 0, ws.ptr, nb, 0)
    rounded = g.numpy()
    dx, dx2 = B(-rounded), B(-rounded)
    hip.call("mle_norm_bwd", None, y.ptr, dy.ptr, dx.ptr, st.ptr, *dims, 0, ws.ptr, nb, 1)
    hip.call("mle_norm_bwd_partials", None, y.ptr, dy.ptr, None, -1, 0, groups, 1, m, 1, 0, ws.ptr, nb)
    hip.call("mle_norm_bwd_apply_add", None, y.ptr, dy.ptr, dx2.ptr, 1, None, hip.Buffer.zeros(n).ptr, 0, None, 0, st.ptr,
             *dims, 0, ws.ptr, nb)
    left = dx.numpy()
    np.testing.assert_array_equal(left, dx2.numpy())
    assert np.all(np.abs(left) <= 2.0 ** -24 * np.abs(rounded))
    assert np.count_nonzero(left) > 0.9 * n
