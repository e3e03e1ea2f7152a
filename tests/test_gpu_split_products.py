"""Products whose float32 operands are split into three bf16 parts for the matrix cores, at the edges
of their tiles, against the same contraction in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip as tf
    tf.set_backend("hip")
    return tf


def _kernel(tf):
    be = tf.backend()
    return be.lib.tfhip_last_kernel(be.ctx).decode()


def _bound(k, magnitude):
    """Every 16 k of a sum are rounded once in float32 (2^-24 of a partial sum, which the sum of the
    products' magnitudes bounds), the products that are left out are below 2^-22 of theirs, and a
    block, a cut along K and the bias add a few roundings more."""
    return (k / 16.0 + 16) * 2.0 ** -24 * magnitude


def _check(got, want, magnitude, k):
    bound = _bound(k, magnitude)
    worst = np.max(np.abs(got - want) - bound)
    assert worst <= 0, (worst, np.abs(got - want).max())


@pytest.mark.parametrize("batch,m,k,n,ta,tb", [
    (1, 2048, 1024, 1024, True, False), (1, 2051, 783, 1027, True, True),   # odd: element-wise loads
    (1, 2048, 260, 1000, False, True), (1, 1500, 1036, 1284, False, True),  # K and N past a tile
    (1, 4096, 20, 4100, True, True), (1, 2052, 16, 2044, True, False),     # one step and a little
    (1, 128, 4096, 4096, True, False),                                     # cut along K, summed in blocks
    (96, 300, 50, 300, False, False), (40, 301, 67, 203, False, True), (3, 1000, 700, 640, True, False),
])
def test_matmul(tf, batch, m, k, n, ta, tb):
    print("split matmul", batch, m, k, n, ta, tb, flush=True)
    rng = np.random.default_rng(m + 3 * k + 7 * n)
    a = rng.uniform(-1, 1, (batch, k, m) if ta else (batch, m, k)).astype(np.float32)
    b = (rng.standard_normal((batch, n, k) if tb else (batch, k, n)) * 10).astype(np.float32)
    with tf.tidy():
        got = tf.matmul(tf.tensor(a), tf.tensor(b), ta, tb).data_sync().astype(np.float64)
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    a64 = a.astype(np.float64).transpose(0, 2, 1) if ta else a.astype(np.float64)
    b64 = b.astype(np.float64).transpose(0, 2, 1) if tb else b.astype(np.float64)
    _check(got, a64 @ b64, np.abs(a64) @ np.abs(b64), k)


@pytest.mark.parametrize("m,k,n,ta,tb", [(2100, 1024, 1030, True, False), (4100, 300, 1100, False, True)])
def test_values_that_bf16_parts_do_not_hold(tf, m, k, n, ta, tb):
    """Infinities, NaN, values next to the largest and rows of tiny ones: as in float32."""
    rng = np.random.default_rng(k)
    a = rng.uniform(0.5, 1, (m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (k, n)).astype(np.float32)
    a[3, 5], a[300, 80], a[500, 7] = np.inf, np.nan, 3.4e38
    a[700] *= np.float32(1e-36)     # below 2^-110: part of the bf16 parts would vanish
    a[800] = 0
    b[11, 200] = -np.inf
    b[7] *= np.float32(0.01)        # (3.4e38 times it is finite)
    with tf.tidy():
        got = tf.matmul(tf.tensor(np.ascontiguousarray(a.T) if ta else a),
                        tf.tensor(np.ascontiguousarray(b.T) if tb else b), ta, tb).data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = a64 @ b64
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    assert not got[800, np.isfinite(want[800])].any()
    fin = np.isfinite(want)
    magnitude = np.abs(np.nan_to_num(a64, posinf=0)) @ np.abs(np.nan_to_num(b64, neginf=0))
    # (a tile that holds such a value is summed in float32, once per two k)
    assert np.all(np.abs(np.where(fin, got - np.where(fin, want, 0), 0)) <= (k / 2 + 16) * 2.0 ** -24 * magnitude)


def _conv64(x, w, stride, dil, pad, oh, ow):
    p = np.pad(x, ((0, 0), (pad[0], pad[0] + 64), (pad[1], pad[1] + 64), (0, 0)))
    y = 0
    for i in range(w.shape[0]):
        for j in range(w.shape[1]):
            r, c = i * dil, j * dil
            y = y + p[:, r:r + (oh - 1) * stride + 1:stride, c:c + (ow - 1) * stride + 1:stride] @ w[i, j]
    return y


@pytest.mark.parametrize("n,h,w,cin,cout,f,stride,dil", [
    (8, 33, 47, 64, 136, 3, 1, 1), (16, 29, 31, 20, 200, 5, 1, 1),   # Cin above and off the step of 16
    (48, 56, 40, 36, 96, 3, 2, 1), (16, 40, 41, 32, 128, 3, 1, 3), (320, 7, 9, 96, 128, 3, 1, 1),
    (64, 31, 30, 4, 132, 5, 1, 1),                                   # four taps in a step
])
def test_conv2d_and_its_gradients(tf, n, h, w, cin, cout, f, stride, dil):
    """The convolution, whose loader walks the taps by additions, and the gradients, which are split."""
    print("split conv", n, h, w, cin, cout, f, stride, dil, flush=True)
    rng = np.random.default_rng(n + h + cin + cout)
    x = rng.standard_normal((n, h, w, cin)).astype(np.float32)
    wt = rng.standard_normal((f, f, cin, cout)).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    oh, ow = -(-h // stride), -(-w // stride)
    eff = (f - 1) * dil + 1
    pad = (max((oh - 1) * stride + eff - h, 0) // 2, max((ow - 1) * stride + eff - w, 0) // 2)
    x64, w64 = x.astype(np.float64), wt.astype(np.float64)
    with tf.tidy():
        got = tf.fused.conv2d(tf.tensor(x), tf.tensor(wt), stride, "same", dilations=dil, bias=tf.tensor(bias),
                              activation="relu").data_sync()
        assert "im2col" in _kernel(tf), _kernel(tf)
    want = _conv64(x64, w64, stride, dil, pad, oh, ow) + bias
    magnitude = _conv64(np.abs(x64), np.abs(w64), stride, dil, pad, oh, ow) + np.abs(bias)
    _check(got, np.maximum(want, 0), magnitude, f * f * cin * 8)   # (in float32: rounded once per two k)
    if dil > 1:
        return
    dy = rng.standard_normal((n, oh, ow, cout)).astype(np.float32)
    d64 = dy.astype(np.float64)
    with tf.tidy():
        dw = tf.conv2d_der_filter(tf.tensor(x), tf.tensor(dy), wt.shape, stride, "same").data_sync()
        kernel_w = _kernel(tf)
        dx = tf.conv2d_der_input(x.shape, tf.tensor(dy), tf.tensor(wt), stride, "same").data_sync()
        kernel_x = _kernel(tf)
    assert kernel_w.startswith("gemm_split_"), kernel_w
    assert stride > 1 or kernel_x.startswith("gemm_split_"), kernel_x
    for i in range(f):
        for j in range(f):
            p = np.pad(x64, ((0, 0), (pad[0], pad[0] + 64), (pad[1], pad[1] + 64), (0, 0)))
            part = p[:, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride].reshape(-1, cin).T
            flat = d64.reshape(-1, cout)
            _check(dw[i, j], part @ flat, np.abs(part) @ np.abs(flat), n * oh * ow)
    want, magnitude = np.zeros((n, h + 2 * f, w + 2 * f, cin)), np.zeros((n, h + 2 * f, w + 2 * f, cin))
    for i in range(f):
        for j in range(f):
            at = (slice(None), slice(i, i + (oh - 1) * stride + 1, stride), slice(j, j + (ow - 1) * stride + 1, stride))
            want[at] += d64 @ w64[i, j].T
            magnitude[at] += np.abs(d64) @ np.abs(w64[i, j].T)
    inside = (slice(None), slice(pad[0], pad[0] + h), slice(pad[1], pad[1] + w))
    # (the float32 gather of a strided layer rounds once per two k)
    _check(dx, want[inside], magnitude[inside], f * f * cout * (1 if stride == 1 else 8))


@pytest.mark.parametrize("k", [1, 2, 3, 4])
@pytest.mark.parametrize("batch,m,n,ta,tb", [(1, 2048, 2048, True, False), (64, 512, 512, False, False),
                                             (96, 201, 201, False, True)])
def test_sums_of_few_products_are_rounded_once_each(tf, batch, m, n, ta, tb, k):
    """Where the parts left out would show: an outer product is the rounded product of its factors."""
    print("few products", batch, m, k, n, ta, tb, flush=True)
    rng = np.random.default_rng(m + k)
    a, b = rng.uniform(-1, 1, (batch, m, k)).astype(np.float32), rng.uniform(-1, 1, (batch, k, n)).astype(np.float32)
    with tf.tidy():
        got = tf.matmul(tf.tensor(a.transpose(0, 2, 1).copy() if ta else a),
                        tf.tensor(b.transpose(0, 2, 1).copy() if tb else b), ta, tb).data_sync()
    if k == 1:
        np.testing.assert_array_equal(got, a * b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - a64 @ b64) <= k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)))


def _float32_bound(k, magnitude):
    """A tile that holds a value the bf16 parts do not is summed in float32, once per two k; a product
    that is denormal is rounded to a multiple of 2^-149."""
    return (k / 2 + 16) * 2.0 ** -24 * magnitude + k * 2.0 ** -149


@pytest.mark.parametrize("batch,m,k,n,ta,tb", [
    (1, 2048, 1024, 1024, True, False), (1, 4096, 64, 4096, True, False),  # 64 x 128 and 128 x 128 tiles
    (1, 128, 4096, 4096, True, False), (1, 2051, 783, 1027, True, True),   # cut along K; element-wise loads
    (40, 301, 67, 203, False, True), (96, 300, 50, 300, False, False),
])
def test_small_operands_against_large_ones(tf, batch, m, k, n, ta, tb):
    """The last parts of a value below 2^-110 are none that bf16 holds, whatever it is multiplied with."""
    print("split small operands", batch, m, k, n, ta, tb, flush=True)
    rng = np.random.default_rng(m + k + n)
    a = rng.uniform(-1, 1, (batch, m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (batch, k, n)).astype(np.float32)
    scaled = lambda x, e: (x.astype(np.float64) * 2.0 ** e).astype(np.float32)
    for row, e in ((0, -112), (m // 2, -120), (m - 1, -140)):
        a[-1, row] = scaled(a[-1, row], e)
    a[0, 5, 0] = 2.0 ** -130                       # one such value among ordinary ones
    for col, e in ((0, 60), (n // 2, 100), (n - 1, 20)):
        b[-1, :, col] = scaled(b[-1, :, col], e)
    b[0, 0, 3] = 2.0 ** 120
    with tf.tidy():
        got = tf.matmul(tf.tensor(a.transpose(0, 2, 1).copy() if ta else a),
                        tf.tensor(b.transpose(0, 2, 1).copy() if tb else b), ta, tb).data_sync().astype(np.float64)
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    worst = np.max(np.abs(got - a64 @ b64) / _float32_bound(k, np.abs(a64) @ np.abs(b64)))
    assert worst <= 1, worst


@pytest.mark.parametrize("n,h,w,cin,cout", [(8, 33, 47, 64, 136), (320, 7, 9, 96, 128)])
def test_small_operands_against_large_ones_in_gathers(tf, n, h, w, cin, cout):
    print("split small operands, gradients", n, h, w, cin, cout, flush=True)
    rng = np.random.default_rng(n + cin)
    x, dy = (rng.standard_normal((n, h, w, c)).astype(np.float32) for c in (cin, cout))
    wt = rng.standard_normal((3, 3, cin, cout)).astype(np.float32)
    x[..., 1] *= np.float32(2.0 ** -122)
    dy[..., 2] *= np.float32(2.0 ** 60)
    with tf.tidy():
        dw = tf.conv2d_der_filter(tf.tensor(x), tf.tensor(dy), wt.shape, 1, "same").data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    p = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    flat = dy.reshape(-1, cout).astype(np.float64)
    for i in range(3):
        for j in range(3):
            part = p[:, i:i + h, j:j + w].reshape(-1, cin).T
            assert np.all(np.abs(dw[i, j] - part @ flat) <= _float32_bound(n * h * w, np.abs(part) @ np.abs(flat)))
    dy[..., 2] *= np.float32(2.0 ** -60)
    dy[0] *= np.float32(2.0 ** -122)
    wt[:, :, 3] *= np.float32(2.0 ** 60)
    with tf.tidy():
        dx = tf.conv2d_der_input(x.shape, tf.tensor(dy), tf.tensor(wt), 1, "same").data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    back = np.ascontiguousarray(wt[::-1, ::-1].transpose(0, 1, 3, 2)).astype(np.float64)
    d64 = dy.astype(np.float64)
    want, magnitude = _conv64(d64, back, 1, 1, (1, 1), h, w), _conv64(np.abs(d64), np.abs(back), 1, 1, (1, 1), h, w)
    assert np.all(np.abs(dx - want) <= _float32_bound(9 * cout, magnitude))


@pytest.mark.parametrize("batch,m,k,n,ta,tb", [
    (24, 1813, 33, 251, False, False), (96, 201, 67, 201, False, True), (1, 3001, 65, 3001, True, True),
    (6, 2051, 130, 259, True, False), (60, 301, 66, 302, False, True),
])
def test_rows_that_are_not_whole_vectors(tf, batch, m, k, n, ta, tb):
    """A vector read at a row's end holds the next row's first values, one stored there would pass the
    row: infinities and NaN in those places stay in their own rows and columns."""
    print("unaligned rows", batch, m, k, n, ta, tb, flush=True)
    rng = np.random.default_rng(m + k + n)
    a = rng.uniform(0.5, 1, (batch, m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (batch, k, n)).astype(np.float32)
    # (1e38: a sum of two such products is below the largest float32, 3.4e38)
    a[0, 17, 0], a[-1, 100, 0], a[0, 0, k - 1], a[-1, m - 1, k - 1] = np.inf, np.nan, 1e38, -np.inf
    b[0, 0, 9], b[-1, k - 1, 0], b[0, 1, 0], b[-1, 2, n - 1] = -np.inf, np.nan, np.inf, 1e38
    with tf.tidy():
        got = tf.matmul(tf.tensor(a.transpose(0, 2, 1).copy() if ta else a),
                        tf.tensor(b.transpose(0, 2, 1).copy() if tb else b), ta, tb).data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = a64 @ b64
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    magnitude = np.abs(np.nan_to_num(a64, posinf=0, neginf=0)) @ np.abs(np.nan_to_num(b64, posinf=0, neginf=0))
    error = np.abs(np.where(fin, got, 0).astype(np.float64) - np.where(fin, want, 0))
    assert np.all(error <= _float32_bound(k, magnitude))


@pytest.mark.parametrize("m,k,n,ta,tb,kernel", [
    (4096, 64, 4096, True, False, "128x128"), (3136, 3072, 64, False, True, "128x64"),
    (64, 20000, 256, True, False, "_splitk"), (2048, 1024, 1028, True, True, "64x128"),
])
def test_special_values_in_every_tile_shape(tf, m, k, n, ta, tb, kernel):
    """Infinities and NaN reach the float32 pass of each tile shape and of tiles cut along K."""
    print("special values", m, k, n, ta, tb, flush=True)
    rng = np.random.default_rng(m)
    a, b = rng.uniform(0.5, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32)
    a[1, k // 2], a[m // 2, 3], a[m - 1, k - 1] = np.inf, np.nan, -np.inf
    b[k - 1, n - 1], b[0, n // 2] = np.inf, np.nan
    with tf.tidy():
        got = tf.matmul(tf.tensor(a.T.copy() if ta else a), tf.tensor(b.T.copy() if tb else b), ta, tb).data_sync()
        name = _kernel(tf)
    assert name.startswith("gemm_split_") and kernel in name, name
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = a64 @ b64
    _same_specials(got, want)
    fin = np.isfinite(want)
    magnitude = np.abs(np.nan_to_num(a64, posinf=0, neginf=0)) @ np.abs(np.nan_to_num(b64, posinf=0, neginf=0))
    assert np.all(np.abs(np.where(fin, got, 0) - np.where(fin, want, 0)) <= _float32_bound(k, magnitude))


def _same_specials(got, want):
    for test in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(test(got), test(want)), test.__name__


@pytest.mark.parametrize("n,h,w,cin,cout", [(8, 33, 47, 64, 136), (320, 7, 9, 96, 128)])
def test_special_values_in_gathers(tf, n, h, w, cin, cout):
    print("special values, gradients", n, h, w, cin, cout, flush=True)
    rng = np.random.default_rng(n + cout)
    x, dy = (rng.standard_normal((n, h, w, c)).astype(np.float32) for c in (cin, cout))
    wt = rng.standard_normal((3, 3, cin, cout)).astype(np.float32)
    x[0, 3, 4, 1], x[-1, -1, -1, 2], dy[1, 0, 0, 5] = np.inf, np.nan, -np.inf
    with tf.tidy():
        dw = tf.conv2d_der_filter(tf.tensor(x), tf.tensor(dy), wt.shape, 1, "same").data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    clean = lambda v: np.abs(np.nan_to_num(v.astype(np.float64), posinf=0, neginf=0))
    pad = lambda v: np.pad(v, ((0, 0), (1, 1), (1, 1), (0, 0)))
    p, flat = pad(x.astype(np.float64)), dy.reshape(-1, cout).astype(np.float64)
    for i in range(3):
        for j in range(3):
            part = p[:, i:i + h, j:j + w].reshape(-1, cin).T
            with np.errstate(invalid="ignore"):
                want = part @ flat
            # (the padding of x is zeros, which the infinite dy in a corner makes NaN: in the kernel too)
            _same_specials(dw[i, j], want)
            fin = np.isfinite(want)
            bound = _float32_bound(n * h * w, clean(part) @ clean(flat))
            assert np.all(np.abs(np.where(fin, dw[i, j], 0) - np.where(fin, want, 0)) <= bound)
    dy[0, 2, 2, 7] = np.nan
    with tf.tidy():
        dx = tf.conv2d_der_input(x.shape, tf.tensor(dy), tf.tensor(wt), 1, "same").data_sync()
        assert _kernel(tf).startswith("gemm_split_"), _kernel(tf)
    back = np.ascontiguousarray(wt[::-1, ::-1].transpose(0, 1, 3, 2)).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = _conv64(dy.astype(np.float64), back, 1, 1, (1, 1), h, w)
    _same_specials(dx, want)
    fin = np.isfinite(want)
    bound = _float32_bound(9 * cout, _conv64(clean(dy), clean(back), 1, 1, (1, 1), h, w))
    assert np.all(np.abs(np.where(fin, dx, 0) - np.where(fin, want, 0)) <= bound)


@pytest.mark.parametrize("n,h,w,cin,cout,f,pad", [
    (32, 56, 57, 48, 128, 3, "same"),     # taps of whole steps; ragged columns; leftover tiles cut along K
    (64, 57, 55, 30 * 2, 64, 3, "valid"), # every column count up to the tile's, padding of the gradient
    (8, 28, 28, 64, 256, 5, "same"),      # every tile cut
])
def test_input_gradient_in_tall_tiles(tf, n, h, w, cin, cout, f, pad):
    print("tall tiles", n, h, w, cin, cout, f, pad, flush=True)
    rng = np.random.default_rng(cin + cout)
    oh, ow = (h, w) if pad == "same" else (h - f + 1, w - f + 1)
    dy = rng.standard_normal((n, oh, ow, cout)).astype(np.float32)
    k = rng.standard_normal((f, f, cin, cout)).astype(np.float32)
    with tf.tidy():
        got = tf.conv2d_der_input((n, h, w, cin), tf.tensor(dy), tf.tensor(k), 1, pad).data_sync().astype(np.float64)
        assert _kernel(tf).startswith("gemm_split_256x64_im2col"), _kernel(tf)
    edge = f - 1 - ((f - 1) // 2 if pad == "same" else 0)
    wide = np.zeros((n, h + f - 1, w + f - 1, cout))
    wide[:, edge:edge + oh, edge:edge + ow] = dy
    for img in (0, n // 2, n - 1):
        want, magnitude = np.zeros((h, w, cin)), np.zeros((h, w, cin))
        for i in range(f):
            for j in range(f):
                part, tap = wide[img, i:i + h, j:j + w], k[f - 1 - i, f - 1 - j].astype(np.float64).T
                want += part @ tap
                magnitude += np.abs(part) @ np.abs(tap)
        _check(got[img], want, magnitude, f * f * cout)


@pytest.mark.parametrize("m,k,n", [(100000, 64, 64), (70001, 128, 60)])
def test_tall_tiles_of_products(tf, m, k, n):
    print("tall products", m, k, n, flush=True)
    rng = np.random.default_rng(m)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    a[7, 3], a[m - 1, k - 1] = np.inf, 2.0 ** -130            # a tile of each kind is summed again
    with tf.tidy():
        got = tf.matmul(tf.tensor(a), tf.tensor(b), False, True).data_sync().astype(np.float64)
        assert _kernel(tf).startswith("gemm_split_256x64"), _kernel(tf)
    want, magnitude = a.astype(np.float64) @ b.T.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).T
    fine = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fine)
    _check(got[fine], want[fine], magnitude[fine], k)
