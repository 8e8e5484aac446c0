"""The split-bf16 GEMM (csrc/split_core.hpp) at the edges of its tiles and
stages, and on values that its split cannot represent.

Bound: of the six partial products per multiply, the leading one is summed in
one fp32 accumulator and the rest in another, one rounding (at most 2^-23,
the matrix core truncates) per 32-deep stage and accumulator; splitting K adds
a rounding per part, and the dropped terms are below 2^-25 of each product.
So |C - exact| <= (2 ceil(K / 32) + 8) 2^-23 sum |a b|, element by element
(half that for the fp32 MFMA fallback's K / 4 roundings of 2^-24 each)."""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


def bound(K):
    return (2 * ((K + 31) // 32) + 8) * 2.0 ** -23


def run(hip, ta, tb, M, N, K, A, Bm, C0=None, bias=None, colsum=None):
    """C (and the column sums) of mle_gemm_ex with its workspace."""
    B = hip.Buffer.from_array
    gA, gB = B(A), B(Bm)
    gC = B(np.full((M, N), np.nan, np.float32) if C0 is None else C0)
    gb = B(bias) if bias is not None else None
    gs = B(colsum) if colsum is not None else None
    nb = hip.lib().mle_gemm_ws_bytes(M, N, K, 1)
    ws = hip.Buffer(nb) if nb else None
    hip.call("mle_gemm_ex", None, ta, tb, M, N, K, 1.0, gA.ptr, A.shape[1], 0, gB.ptr, Bm.shape[1], 0,
             0.0 if C0 is None else 1.0, gC.ptr, N, 0, 1, gs.ptr if gs else None, gb.ptr if gb else None,
             ws.ptr if ws else None, nb)
    return gC.numpy((M, N)), gs.numpy() if gs else None


# Outputs above 4096 x 64 (the small-product kernels end there), each tile
# shape, one row or column less and more than whole tiles, K around one stage,
# no multiple of 4, and long enough to split.
SHAPES = [(1000, 516, 330), (513, 515, 1), (640, 449, 31), (640, 449, 32), (768, 513, 33), (257, 1025, 35),
          (255, 2047, 64), (2049, 129, 95), (4095, 127, 131), (4100, 65, 1027), (8192, 520, 70), (700, 400, 4099)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_split_gemm_edges(hip, ta, tb, M, N, K):
    r = rng(M + 3 * N + 7 * K + ta + 2 * tb)
    a, b = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((K, N), dtype=np.float32)
    bias = r.standard_normal(N, dtype=np.float32)
    # row strides of no alignment: 3 columns that must not be read as part of the matrix
    wide = lambda t: np.concatenate([t, np.full((t.shape[0], 3), 1e30, np.float32)], 1)  # noqa: E731
    A, Bm = wide(a.T if ta else a), wide(b.T if tb else b)
    cs0 = r.standard_normal(N, dtype=np.float32) if (ta, tb) == (1, 0) else None
    C, cs = run(hip, ta, tb, M, N, K, np.ascontiguousarray(A), np.ascontiguousarray(Bm), bias=bias, colsum=cs0)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want, terms = a64 @ b64 + bias, np.abs(a64) @ np.abs(b64) + np.abs(bias)
    assert np.all(np.abs(C - want) <= bound(K) * terms)
    if cs is not None:  # a sequential fp32 sum per lane group, then four of them
        lim = (K / 4 + 8) * 2.0 ** -24 * (np.abs(b64).sum(0) + np.abs(cs0))
        assert np.all(np.abs(cs - (b64.sum(0) + cs0)) <= lim)
    # adding to C
    C0 = r.standard_normal((M, N), dtype=np.float32)
    C, _ = run(hip, ta, tb, M, N, K, np.ascontiguousarray(A), np.ascontiguousarray(Bm), C0=C0.copy())
    assert np.all(np.abs(C - (a64 @ b64 + C0)) <= bound(K) * (terms + np.abs(C0)))


@pytest.mark.parametrize("what", ["inf", "nan", "max", "tiny", "denormal", "overflow"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_split_gemm_special_values(hip, ta, tb, what):
    """Infinities, NaN, the largest values (which round to infinity in bf16)
    and the smallest (whole rows near and below the end of the normal range,
    single values among ordinary ones): as fp32 products give them."""
    M, N, K = 700, 600, 200
    r = rng(77 + ta + 2 * tb)
    a, b = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((K, N), dtype=np.float32)
    fmax = np.finfo(np.float32).max
    if what == "inf":
        a[3, 5], a[300, 7], b[9, 400] = np.inf, -np.inf, np.inf
    elif what == "nan":
        a[699, 199], b[0, 0] = np.nan, np.nan
    elif what == "max":  # finite results: the row's other values vanish against them
        a[17, :], a[17, 3] = 0.0, -fmax
        b[3, :] = np.clip(b[3], -0.9, 0.9)
    elif what == "tiny":
        a[400:, :] *= np.float32(2.0 ** -112)
        b[:, 100:200] *= np.float32(2.0 ** 40)
    elif what == "denormal":
        a[400:, :] *= np.float32(2.0 ** -130)
        a[:400, ::7] *= np.float32(2.0 ** -120)
        b *= np.float32(2.0 ** 40)
    else:
        a[50, :], b[:, 60] = np.float32(1e30), np.float32(1e30)
    A, Bm = np.ascontiguousarray(a.T if ta else a), np.ascontiguousarray(b.T if tb else b)
    C, _ = run(hip, ta, tb, M, N, K, A, Bm)
    with np.errstate(invalid="ignore", over="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want = (a64 @ b64)
        terms = np.abs(a64) @ np.abs(b64)
        w32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(C), np.isnan(w32))
    assert np.array_equal(C[np.isinf(w32)], w32[np.isinf(w32)])
    ok = np.isfinite(w32)
    assert np.all(np.isfinite(C[ok]))
    # results below the normal range round to fp32's smallest step
    lim = bound(K) * terms[ok] + 2.0 ** -140
    assert np.all(np.abs(C[ok] - want[ok]) <= lim)


def test_split_gemm_identity_exact(hip):
    """A value times one is the value: the three parts add up to it exactly."""
    M, N = 600, 640
    r = rng(5)
    a = (r.standard_normal((M, N)) * np.exp2(r.integers(-60, 60, (M, N)))).astype(np.float32)
    C, _ = run(hip, 0, 0, M, N, N, a, np.eye(N, dtype=np.float32))
    np.testing.assert_array_equal(C, a)


# Convolutions at the edges of the split kernels' tiles and of their tap
# table's period (32 channels): maps of odd size (one-element loads), strides,
# depths of one, whole and part periods, a 25-tap filter, one pixel, few and
# many tiles (K groups), against float64 sums of the same products.
CONVS = [(3, 33, 7, 7, 70, 3, 1, 1), (2, 65, 9, 11, 130, 3, 1, 2), (1, 97, 5, 5, 66, 3, 0, 1), (2, 64, 14, 14, 129, 3, 1, 1),
         (1, 20, 13, 10, 67, 5, 2, 1), (4, 31, 3, 3, 257, 1, 0, 1), (1, 130, 1, 1, 72, 3, 1, 1), (5, 160, 28, 28, 72, 1, 0, 2),
         (33, 66, 32, 32, 67, 3, 1, 1)]


@pytest.mark.parametrize("n,cin,h,w,cout,k,pad,stride", CONVS)
def test_split_conv_edges(hip, n, cin, h, w, cout, k, pad, stride):
    r = rng(n + cin + h + w + cout + k + stride)
    oh, ow = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
    x = r.standard_normal((n, cin, h, w), dtype=np.float32)
    wt = r.standard_normal((cout, cin, k, k), dtype=np.float32)
    b = r.standard_normal(cout, dtype=np.float32)
    dy = r.standard_normal((n, cout, oh, ow), dtype=np.float32)
    xp = np.zeros((n, cin, h + 2 * pad, w + 2 * pad))
    xp[:, :, pad:pad + h, pad:pad + w] = x
    span = lambda o, s: slice(s, s + (o - 1) * stride + 1, stride)  # noqa: E731
    y, ya = np.zeros((n, cout, oh, ow)), np.zeros((n, cout, oh, ow))
    dxp, dxa = np.zeros_like(xp), np.zeros_like(xp)
    dw, dwa = np.zeros(wt.shape), np.zeros(wt.shape)
    for i in range(k):
        for j in range(k):
            xs, wij = xp[:, :, span(oh, i), span(ow, j)], wt[:, :, i, j].astype(np.float64)
            d = dy.astype(np.float64)
            y += np.einsum("oc,ncyx->noyx", wij, xs, optimize=True)
            ya += np.einsum("oc,ncyx->noyx", np.abs(wij), np.abs(xs), optimize=True)
            dxp[:, :, span(oh, i), span(ow, j)] += np.einsum("oc,noyx->ncyx", wij, d, optimize=True)
            dxa[:, :, span(oh, i), span(ow, j)] += np.einsum("oc,noyx->ncyx", np.abs(wij), np.abs(d), optimize=True)
            dw[:, :, i, j] = np.einsum("noyx,ncyx->oc", d, xs, optimize=True)
            dwa[:, :, i, j] = np.einsum("noyx,ncyx->oc", np.abs(d), np.abs(xs), optimize=True)
    y += b[:, None, None]
    dx, dxa = dxp[:, :, pad:pad + h, pad:pad + w], dxa[:, :, pad:pad + h, pad:pad + w]
    B = hip.Buffer.from_array
    dims = (n, cin, h, w, cout, k, k, pad, stride)
    gx, gw, gb, gdy = B(x), B(wt), B(b), B(dy)
    gy, gdx, gdw = B(np.full(y.shape, np.nan, np.float32)), B(np.full(x.shape, np.nan, np.float32)), B(np.full(wt.shape, np.nan, np.float32))
    gdb = B(np.full(cout, np.nan, np.float32))
    # the fp32 MFMA kernels, where they run, round once per 4 products
    lim = lambda K: max(bound(K), (K / 4 + 8) * 2.0 ** -24)  # noqa: E731
    hip.call("mle_conv2d_fwd", None, gx.ptr, gw.ptr, gb.ptr, gy.ptr, *dims)
    assert np.all(np.abs(gy.numpy(y.shape) - y) <= lim(cin * k * k) * (ya + np.abs(b)[:, None, None]))
    hip.call("mle_conv2d_dgrad", None, gdy.ptr, gw.ptr, gdx.ptr, *dims, 0)
    assert np.all(np.abs(gdx.numpy(x.shape) - dx) <= lim(cout * k * k) * dxa)
    hip.call("mle_conv2d_dgrad", None, gdy.ptr, gw.ptr, gdx.ptr, *dims, 1)
    assert np.all(np.abs(gdx.numpy(x.shape) - 2 * dx) <= 2 * lim(cout * k * k) * dxa + 2.0 ** -22 * np.abs(dx))
    nb = hip.lib().mle_conv2d_wgrad_ws_bytes(*dims)
    ws = hip.Buffer(nb)
    hip.call("mle_conv2d_wgrad_bias", None, gx.ptr, gdy.ptr, gdw.ptr, gdb.ptr, 0, *dims, ws.ptr, nb)
    K = n * oh * ow
    assert np.all(np.abs(gdw.numpy(wt.shape) - dw) <= lim(K) * dwa)
    db, dba = dy.astype(np.float64).sum((0, 2, 3)), np.abs(dy).sum((0, 2, 3))
    assert np.all(np.abs(gdb.numpy() - db) <= (K / 4 + 8) * 2.0 ** -24 * dba)


def test_split_conv_special_values(hip):
    """An infinity, a NaN and the largest value in x and dy: the same
    positions as fp32 products give them, everything else finite and right."""
    n, cin, h, cout = 2, 96, 20, 80
    r = rng(9)
    x = r.standard_normal((n, cin, h, h), dtype=np.float32)
    wt = (r.random((cout, cin, 3, 3)) * 0.5 + 0.1).astype(np.float32)
    x[0, 3, 4, 5], x[1, 90, 19, 19], x[0, 50, 10, 10] = np.inf, np.nan, np.finfo(np.float32).max
    xp = np.zeros((n, cin, h + 2, h + 2))
    xp[:, :, 1:-1, 1:-1] = x
    y = np.zeros((n, cout, h, h))
    ya = np.zeros_like(y)
    with np.errstate(invalid="ignore", over="ignore"):
        for i in range(3):
            for j in range(3):
                xs, wij = xp[:, :, i:i + h, j:j + h], wt[:, :, i, j].astype(np.float64)
                y += np.einsum("oc,ncyx->noyx", wij, xs)
                ya += np.einsum("oc,ncyx->noyx", wij, np.abs(xs))
        y32 = y.astype(np.float32)
    B = hip.Buffer.from_array
    gx, gw, gy = B(x), B(wt), B(np.zeros(y.shape, np.float32))
    hip.call("mle_conv2d_fwd", None, gx.ptr, gw.ptr, None, gy.ptr, n, cin, h, h, cout, 3, 3, 1, 1)
    got = gy.numpy(y.shape)
    assert np.array_equal(np.isnan(got), np.isnan(y32))
    assert np.array_equal(got[np.isinf(y32)], y32[np.isinf(y32)])
    ok = np.isfinite(y32)
    assert np.all(np.abs(got[ok] - y[ok]) <= bound(cin * 9) * ya[ok])


@pytest.mark.parametrize("M,N", [(2300, 2000), (3, 5)])
def test_empty_depth(hip, M, N):
    """K = 0: C = beta C + bias, whatever the size of C (more than 4 Mi values
    go past the small-product kernels); a Linear of no rows has zero gradients."""
    r = rng(M)
    C0, bias = r.standard_normal((M, N), dtype=np.float32), r.standard_normal(N, dtype=np.float32)
    gC, gb = hip.Buffer.from_array(C0), hip.Buffer.from_array(bias)
    hip.call("mle_gemm_ex", None, 0, 0, M, N, 0, 1.0, None, 0, 0, None, N, 0, 0.5, gC.ptr, N, 0, 1, None, gb.ptr, None, 0)
    np.testing.assert_array_equal(gC.numpy((M, N)), np.float32(0.5) * C0 + bias)
    gX, gW = hip.Buffer.from_array(np.zeros(4, np.float32)), hip.Buffer.from_array(C0)
    dW, db = hip.Buffer.from_array(C0), hip.Buffer.from_array(bias)
    hip.call("mle_linear_bwd_ex", None, 0, M, N, 1, gX.ptr, gX.ptr, 0, gW.ptr, 0, gX.ptr, 0, dW.ptr, db.ptr, 0, 0, None, 0)
    assert not dW.numpy().any() and not db.numpy().any()


# Weight gradients whose workgroups walk more pixels than their table holds
# (3072 and 2304): filled again, with a partial last fill, one-element loads
# (odd maps), 1 x 1 and 3 x 3 filters, each tile, two K groups.
REFILLS = [(1, 2048, 58, 58, 2048, 1), (1, 128, 113, 113, 4096, 3), (3, 4096, 56, 56, 64, 1), (3, 4096, 57, 57, 64, 1),
           (4, 2100, 50, 50, 64, 3), (8, 4096, 57, 57, 64, 1)]


@pytest.mark.parametrize("n,cin,h,w,cout,k", REFILLS)
def test_split_wgrad_refills_its_table(hip, n, cin, h, w, cout, k):
    r = rng(cin + h)
    x = r.standard_normal((n, cin, h, w), dtype=np.float32)
    dy = r.standard_normal((n, cout, h, w), dtype=np.float32)
    pad = k // 2
    dims = (n, cin, h, w, cout, k, k, pad, 1)
    nb = hip.lib().mle_conv2d_wgrad_ws_bytes(*dims)
    K, splits = n * h * w, max(1, nb // (4 * (cout * cin * k * k + cout)))
    assert K / splits > (2304 if cout == 64 else 3072)
    B = hip.Buffer.from_array
    gx, gdy, gdw, gdb = B(x), B(dy), B(np.full((cout, cin, k, k), np.nan, np.float32)), B(np.full(cout, np.nan, np.float32))
    ws = hip.Buffer(nb) if nb else None
    hip.call("mle_conv2d_wgrad_bias", None, gx.ptr, gdy.ptr, gdw.ptr, gdb.ptr, 0, *dims, ws.ptr if ws else None, nb)
    got = gdw.numpy((cout, cin, k, k))
    # 20 rows of dW and 20 of its columns, in float64
    xp = np.zeros((n, cin, h + 2 * pad, w + 2 * pad), np.float32)
    xp[:, :, pad:pad + h, pad:pad + w] = x
    rows, cols = r.choice(cout, 20, replace=False), r.choice(cin, 20, replace=False)
    for i in range(k):
        for j in range(k):
            xs = xp[:, :, i:i + h, j:j + w].transpose(1, 0, 2, 3).reshape(cin, -1)
            d = dy.transpose(1, 0, 2, 3).reshape(cout, -1)
            for ci, co in ((np.arange(cin), rows), (cols, np.arange(cout))):
                a, b = d[co].astype(np.float64), xs[ci].astype(np.float64).T
                assert np.all(np.abs(got[np.ix_(co, ci)][:, :, i, j] - a @ b) <= bound(K) * (np.abs(a) @ np.abs(b)))
    db, dba = dy.astype(np.float64).sum((0, 2, 3)), np.abs(dy).sum((0, 2, 3))
    assert np.all(np.abs(gdb.numpy() - db) <= (K / 4 + 8) * 2.0 ** -24 * dba)


def test_column_sums_of_a_long_depth(hip):
    """The fused column sums (a bias gradient) round like sums of eight in a tree
    (three roundings) and one final rounding, at any depth: the stages add in
    double."""
    M, N, K = 256, 320, 65536
    r = rng(8)
    A, Bm = r.random((K, M), dtype=np.float32), r.random((K, N), dtype=np.float32)
    B = hip.Buffer.from_array
    gA, gB, gC, gs = B(A), B(Bm), hip.Buffer.zeros((M, N)), hip.Buffer.zeros(N)
    hip.call("mle_gemm_ex", None, 1, 0, M, N, K, 1.0, gA.ptr, M, 0, gB.ptr, N, 0, 0.0, gC.ptr, N, 0, 1, gs.ptr, None, None, 0)
    want = Bm.astype(np.float64).sum(0)
    assert np.all(np.abs(gs.numpy() - want) <= 4 * 2.0 ** -24 * want)


@pytest.mark.parametrize("K", [4096, 16384])
@pytest.mark.parametrize("kind", ["uniform", "near one", "magnitudes"])
def test_split_gemm_one_signed_error(hip, K, kind):
    """Operands of one sign, where truncation inside the matrix core would add up:
    the relative error (2-norm) stays below the fp32 MFMA kernel's, which a
    column sum of an untransposed A still reaches."""
    M, N = 300, 700
    r = rng(K)
    draw = {"uniform": lambda s: r.random(s), "near one": lambda s: 1 + 1e-3 * r.random(s),
            "magnitudes": lambda s: np.abs(r.standard_normal(s))}[kind]
    a, b = draw((M, K)).astype(np.float32), draw((K, N)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    B = hip.Buffer.from_array
    gA, gB, gC, gs = B(a), B(b), hip.Buffer.zeros((M, N)), hip.Buffer.zeros(N)
    err = []
    for colsum in (None, gs.ptr):  # without a workspace: one accumulation over all of K
        hip.call("mle_gemm_ex", None, 0, 0, M, N, K, 1.0, gA.ptr, K, 0, gB.ptr, N, 0, 0.0, gC.ptr, N, 0, 1, colsum, None, None, 0)
        err.append(np.linalg.norm(gC.numpy((M, N)) - want) / np.linalg.norm(want))
    assert err[0] <= err[1], err


def test_split_wgrad_long_sums_error(hip):
    """Few splits over many pixels: the stages are summed in runs of at most 24.  A
    running sum of n random stages is truncated by up to 2^-23 of itself, rms half
    of that, at sizes that grow with the square root: 2^-24 sqrt(n / 2) of the
    result.  One sum per split (over 100 stages) would be at 4.2e-7."""
    n, cin, h, cout = 22, 188, 56, 16
    r = rng(12)
    x, dy = (r.standard_normal((n, c, h, h), dtype=np.float32) for c in (cin, cout))
    dims = (n, cin, h, h, cout, 3, 3, 1, 1)
    nb = hip.lib().mle_conv2d_wgrad_ws_bytes(*dims)
    assert n * h * h / 32 / max(1, nb // (4 * (cout * cin * 9 + cout))) > 100
    B = hip.Buffer.from_array
    gx, gdy, gdw, ws = B(x), B(dy), hip.Buffer.zeros((cout, cin, 3, 3)), hip.Buffer(max(nb, 4))
    hip.call("mle_conv2d_wgrad", None, gx.ptr, gdy.ptr, gdw.ptr, *dims, ws.ptr, nb)
    got = gdw.numpy((cout, cin, 3, 3))
    xp = np.zeros((n, cin, h + 2, h + 2), np.float32)
    xp[:, :, 1:-1, 1:-1] = x
    d = dy.transpose(1, 0, 2, 3).reshape(cout, -1).astype(np.float64)
    err = ref = 0.0
    for i in range(3):
        for j in range(3):
            want = d @ xp[:, :, i:i + h, j:j + h].transpose(1, 0, 2, 3).reshape(cin, -1).astype(np.float64).T
            err += np.square(got[:, :, i, j] - want).sum()
            ref += np.square(want).sum()
    assert np.sqrt(err / ref) <= 2.0 ** -24 * np.sqrt(24 / 2)
