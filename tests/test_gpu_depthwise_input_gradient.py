"""The gradient of a depthwise convolution's input at stride 1, which the forward kernels give by walking the
filter's taps from the last to the first: patches, rows of large images, and every other filter and width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("n,h,w,c,fh,fw,pad", [
    (1, 3, 3, 4, 3, 3, "valid"), (2, 9, 7, 8, 3, 3, "same"), (1, 12, 11, 20, 3, 3, 2),
    (2, 16, 16, 128, 3, 3, "valid"), (1, 112, 112, 128, 3, 3, "same"),           # patches of several sizes
    (16, 56, 56, 128, 3, 3, "same"), (32, 29, 30, 64, 3, 3, "valid"),             # rows
    (2, 9, 8, 6, 3, 3, "same"), (1, 10, 9, 8, 2, 5, "same"), (1, 8, 8, 4, 1, 1, "valid"), (2, 11, 12, 7, 5, 4, "valid"),
])
def test_input_gradient(tf, n, h, w, c, fh, fw, pad):
    print("dx", n, h, w, c, fh, fw, pad, flush=True)
    from oracle import cpu_ref as ref
    rng = np.random.default_rng(n + h + w + c)
    ci = ref.compute_conv2d_info((n, h, w, c), (fh, fw, c, 1), 1, 1, pad, depthwise=True)
    p, oh, ow = ci["padInfo"], ci["outHeight"], ci["outWidth"]
    k = rng.standard_normal((fh, fw, c, 1)).astype(np.float32)
    dy = rng.standard_normal(ci["outShape"]).astype(np.float32)
    with tf.tidy():
        got = tf.depthwise_conv2d_der_input((n, h, w, c), tf.tensor(dy), tf.tensor(k), 1, pad).data_sync()
    want, magnitude = np.zeros((n, oh + fh + h, ow + fw + w, c)), np.zeros((n, oh + fh + h, ow + fw + w, c))
    for i in range(fh):
        for j in range(fw):
            part = dy.astype(np.float64) * k[i, j, :, 0]
            want[:, i:i + oh, j:j + ow] += part
            magnitude[:, i:i + oh, j:j + ow] += np.abs(part)
    inside = (slice(None), slice(p["top"], p["top"] + h), slice(p["left"], p["left"] + w))
    # fh x fw products, one half ulp of the magnitudes for each of them and its sum
    assert np.all(np.abs(got.reshape(n, h, w, c) - want[inside]) <= (fh * fw + 1) * 2.0 ** -24 * magnitude[inside])
