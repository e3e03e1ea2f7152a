"""Convolutions whose filter taps are whole k steps (channels a multiple of 16), at the edges of that
path: borders, strides, dilations, the most taps, quantised filters, and one step beyond each limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("n,h,w,cin,cout,fh,fw,stride,dil,pad,quant", [
    (1, 1, 1, 16, 8, 3, 3, 1, 1, "same", False), (2, 7, 9, 16, 64, 3, 3, 1, 1, "same", False),
    (1, 13, 11, 48, 132, 3, 3, 2, 1, "same", False), (3, 9, 8, 32, 36, 5, 5, 1, 1, "same", False),
    (1, 20, 21, 16, 40, 3, 2, 1, (2, 3), "valid", False), (2, 15, 17, 64, 20, 2, 4, (1, 2), 1, "same", False),
    (1, 12, 12, 16, 12, 3, 3, 1, 1, 2, False),              # padding on all sides, rows before the first image
    (1, 40, 9, 16, 64, 31, 1, 1, 1, "same", False),         # 31 taps
    (1, 40, 9, 16, 64, 8, 4, 1, 1, "same", False),          # 32: the general gather
    (2, 11, 10, 24, 64, 3, 3, 1, 1, "same", False),         # taps that are not whole steps: the same
    (2, 10, 10, 80, 64, 3, 3, 1, 1, "same", True), (40, 28, 30, 32, 96, 3, 3, 2, 1, "same", False),
    (1, 30, 33, 256, 128, 1, 1, 2, 1, "valid", False),
])
def test_taps(tf, n, h, w, cin, cout, fh, fw, stride, dil, pad, quant):
    print("taps", n, h, w, cin, cout, fh, fw, stride, dil, pad, quant, flush=True)
    from oracle import cpu_ref as ref
    rng = np.random.default_rng(h * 31 + cin + cout)
    x = rng.standard_normal((n, h, w, cin)).astype(np.float32)
    ci = ref.compute_conv2d_info(x.shape, (fh, fw, cin, cout), stride, dil, pad)
    if quant:
        q = rng.integers(0, 256, (fh, fw, cin, cout)).astype(np.uint8)
        k = (q.astype(np.float64) * 0.01 - 1.2).astype(np.float32)
    else:
        k = rng.standard_normal((fh, fw, cin, cout)).astype(np.float32)
    with tf.tidy():
        tk = tf.quantized_tensor(q, 0.01, -1.2) if quant else tf.tensor(k)
        got = tf.conv2d(tf.tensor(x), tk, stride, pad, "NHWC", dil).data_sync()
    sh, sw, dh, dw = (ci[v] for v in ("strideHeight", "strideWidth", "dilationHeight", "dilationWidth"))
    oh, ow, p = ci["outHeight"], ci["outWidth"], ci["padInfo"]
    wide = np.zeros((n, (oh - 1) * sh + (fh - 1) * dh + 1 + h, (ow - 1) * sw + (fw - 1) * dw + 1 + w, cin))
    wide[:, p["top"]:p["top"] + h, p["left"]:p["left"] + w] = x
    want, magnitude = np.zeros((n, oh, ow, cout)), np.zeros((n, oh, ow, cout))
    for i in range(fh):
        for j in range(fw):
            part = wide[:, i * dh:i * dh + (oh - 1) * sh + 1:sh, j * dw:j * dw + (ow - 1) * sw + 1:sw]
            want += part @ k[i, j].astype(np.float64)
            magnitude += np.abs(part) @ np.abs(k[i, j]).astype(np.float64)
    # a rounding per product and per addition
    assert np.all(np.abs(got - want) <= (fh * fw * cin + 2) * 2.0 ** -24 * magnitude)
