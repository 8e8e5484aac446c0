"""The attention passes on split bf16 products (seq > 256, unmasked seq > 128)
against float64.

Tolerance: a score is a 64-term product, |error| <= 8 * 2^-24 of its terms'
magnitudes; it enters exp() as an absolute error of the exponent, next to
the rounding of the exponent itself and the hardware exp2's few ulp.  With
standard normal operands (scores below 8, terms below 64 / 8 per unit of
scale) that is a relative error of P below 1e-5; the outputs sum P against
the magnitudes of the other operand."""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu
HD = 64


def reference(q, k, v, do, scale, causal, kref):
    """One head, [s, 64] each, in float64: values and the sums of magnitudes
    that bound their errors."""
    q, k, v, do = (x.astype(np.float64) for x in (q, k, v, do))
    s = scale * q @ k.T
    e = np.exp(s - s.max(0))
    if causal:
        e = np.tril(e)
    l = e.sum(0)
    p = e / np.where(l < 1e-45, 1, l)
    dp = do @ v.T
    dc = (p * dp).sum(0)
    ds = p * (dp - dc)
    dsa = p * (np.abs(do) @ np.abs(v).T + (p * (np.abs(do) @ np.abs(v).T)).sum(0))
    o, dv, dq = p @ v, p.T @ do, scale * ds @ k
    oa, dva, dqa = p @ np.abs(v), p.T @ np.abs(do), scale * dsa @ np.abs(k)
    if kref:  # (dS Q)^T row-major into the [s x 64] block
        dk, dka = ((scale * x @ y).T.reshape(-1, HD) for x, y in ((ds, q), (dsa, np.abs(q))))
    else:
        dk, dka = scale * ds.T @ q, scale * dsa.T @ np.abs(q)
    return (o, dq, dk, dv), (oa, dqa, dka, dva)


def run(hip, q, k, v, do, b, h, s, ld, scale, causal, kref):
    B = hip.Buffer.from_array
    ws = hip.Buffer(hip.lib().mle_attention_ws_bytes(b, h, s))
    g = [B(np.ascontiguousarray(x)) for x in (q, k, v, do)]
    out = [B(np.full((b, s, ld), np.nan, np.float32)) for _ in range(4)]
    hip.call("mle_attention_fwd", None, g[0].ptr, g[1].ptr, g[2].ptr, out[0].ptr, b, h, s, HD, ld, scale, causal, ws.ptr, ws.nbytes)
    hip.call("mle_attention_bwd", None, *(x.ptr for x in g), out[1].ptr, out[2].ptr, out[3].ptr, b, h, s, HD, ld, scale, causal,
             0, 0, 0, kref, ws.ptr, ws.nbytes)
    return [x.numpy((b, s, ld)) for x in out]


# whole and half column blocks (128), several heads and batch items, a wider ld;
# unmasked up to 256 positions: split past 128 positions, few slices and many
@pytest.mark.parametrize("b,h,s,extra,causal,kref", [
    (2, 3, 320, 0, 1, 1), (1, 2, 448, 64, 0, 1), (2, 1, 512, 0, 1, 0), (1, 9, 576, 0, 0, 0), (1, 1, 1088, 128, 1, 1),
    (1, 2, 192, 64, 0, 1), (1, 2, 256, 0, 0, 0), (2, 64, 192, 0, 0, 1), (3, 43, 192, 0, 0, 1), (3, 43, 192, 0, 0, 0),
    (3, 43, 256, 0, 0, 1), (3, 43, 256, 0, 0, 0), (1, 2, 128, 0, 0, 1), (1, 2, 256, 0, 1, 1)])
def test_split_attention(hip, b, h, s, extra, causal, kref):
    r = rng(b + h + s + causal)
    ld = h * HD + extra
    q, k, v, do = (r.standard_normal((b, s, ld), dtype=np.float32) for _ in range(4))
    got = run(hip, q, k, v, do, b, h, s, ld, 0.125, causal, kref)
    for i in range(b):
        for j in range(h):
            c = slice(j * HD, (j + 1) * HD)
            want, mag = reference(q[i, :, c], k[i, :, c], v[i, :, c], do[i, :, c], 0.125, causal, kref)
            for name, g, w, m in zip(("out", "dq", "dk", "dv"), got, want, mag):
                assert np.all(np.abs(g[i, :, c] - w) <= 1e-5 * m + 1e-30), name
    if extra:
        assert all(np.isnan(g[:, :, h * HD:]).all() for g in got)


@pytest.mark.parametrize("causal", [0, 1])
def test_split_attention_special_values(hip, causal):
    """Values the split cannot hold go to the fp32 products: infinities and
    NaN appear where they do in float32 sums, gradients near the bottom of
    the range and rows of tiny probabilities keep their relative error."""
    s, h = 384, 4
    r = rng(77 + causal)
    q, k, v, do = (r.standard_normal((1, s, h * HD), dtype=np.float32) for _ in range(4))
    v[0, 200, 5] = np.inf           # head 0: one key's value
    v[0, 300, 9] = np.nan
    do[0, :, 64:128] *= np.float32(2.0 ** -112)   # head 1: a gradient the split would truncate
    q[0, :, 128:192] *= 10          # head 2: scores up to 50, rows whose every probability is tiny
    k[0, 7, 192:256] = 2.0 ** -115  # head 3: one tiny row
    got = run(hip, q, k, v, do, 1, h, s, h * HD, 0.125, causal, 1)
    for j in range(h):
        c = slice(j * HD, (j + 1) * HD)
        with np.errstate(invalid="ignore", over="ignore"):
            want, mag = reference(q[0, :, c], k[0, :, c], v[0, :, c], do[0, :, c], 0.125, causal, 1)
        if j == 0:  # columns of V without them are untouched; theirs are not finite for every query that sees the key
            clean = [x for x in range(HD) if x not in (5, 9)]
            assert np.all(np.abs(got[0][0, :, clean] - want[0].T[clean]) <= 1e-5 * mag[0].T[clean])
            seen = lambda key: slice(key if causal else 0, None)  # noqa: E731
            assert not np.isfinite(got[0][0, seen(200), 5]).any() and np.isnan(got[0][0, seen(300), 9]).all()
            continue
        # 10 times the scores: 10 times the exponent's error
        tol = 1e-4 if j == 2 else 1e-5
        for name, g, w, m in zip(("out", "dq", "dk", "dv"), got, want, mag):
            assert np.all(np.abs(g[0, :, c] - w) <= tol * m + 2.0 ** -140), (j, name)


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("exp", [-112, -125, -136])
def test_split_attention_small_operands(hip, causal, exp):
    """V and dO near and below the end of the normal range: the outputs that are
    linear in them keep every bit that fp32 products give (steps of 2^-149)."""
    s, h = 320, 2
    r = rng(5 - exp + causal)
    q, k, v, do = (r.standard_normal((1, s, h * HD), dtype=np.float32) for _ in range(4))
    v[0, :, :HD] *= np.float32(2.0 ** exp)   # head 0: all of V
    do[0, :, HD:] *= np.float32(2.0 ** exp)  # head 1: all of dO
    out, _, _, dv = run(hip, q, k, v, do, 1, h, s, h * HD, 0.125, causal, 1)
    for j, i in ((0, 0), (1, 3)):
        c = slice(j * HD, (j + 1) * HD)
        want, mag = reference(q[0, :, c], k[0, :, c], v[0, :, c], do[0, :, c], 0.125, causal, 1)
        got = (out if i == 0 else dv)[0, :, c]
        assert np.all(np.abs(got - want[i]) <= 1e-5 * mag[i] + 2.0 ** -148)


# the causal passes hand out blocks of one kind after another on each XCD: grids
# of no multiple of 8, XCDs that share a slice, fewer blocks than XCDs
@pytest.mark.parametrize("b,h,s,kref", [(3, 23, 320, 1), (1, 13, 576, 1), (1, 3, 384, 1), (5, 7, 448, 0)])
def test_causal_block_order(hip, b, h, s, kref):
    r = rng(b * h + s)
    q, k, v, do = (r.standard_normal((b, s, h * HD), dtype=np.float32) for _ in range(4))
    got = run(hip, q, k, v, do, b, h, s, h * HD, 0.125, 1, kref)
    for i in range(b):
        for j in range(h):
            c = slice(j * HD, (j + 1) * HD)
            want, mag = reference(q[i, :, c], k[i, :, c], v[i, :, c], do[i, :, c], 0.125, 1, kref)
            for name, g, w, m in zip(("out", "dq", "dk", "dv"), got, want, mag):
                assert np.all(np.abs(g[i, :, c] - w) <= 1e-5 * m + 1e-30), (name, i, j)


@pytest.mark.parametrize("causal", [0, 1])
def test_mathematical_k_gradient_error(hip, causal):
    """dK = scale dS^T Q and dQ = scale dS K sum the same dS over the same number
    of positions, so their relative errors (2-norm) are of one size.  Scores of
    two different products in one column (statistics of one, probabilities of
    the other) would show here: dK's error was 2.4 times dQ's."""
    s, h = 512, 4
    r = rng(31 + causal)
    q, k, v, do = (r.standard_normal((1, s, h * HD), dtype=np.float32) for _ in range(4))
    _, dq, dk, _ = run(hip, q, k, v, do, 1, h, s, h * HD, 0.125, causal, 0)
    err, ref = np.zeros(2), np.zeros(2)
    for j in range(h):
        c = slice(j * HD, (j + 1) * HD)
        want, _ = reference(q[0, :, c], k[0, :, c], v[0, :, c], do[0, :, c], 0.125, causal, 0)
        for n, (g, w) in enumerate(((dq, want[1]), (dk, want[2]))):
            err[n] += np.square(g[0, :, c] - w).sum()
            ref[n] += np.square(w).sum()
    rel = np.sqrt(err / ref)
    assert rel[1] <= 1.5 * rel[0], rel
