"""The gradient of a 3 x 3 depthwise filter at the edges of its kernel: segments of rows, channel blocks,
padding, strides that have a kernel of their own and one that has not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("n,h,w,c,stride,pad", [
    (1, 1, 1, 4, 1, "same"), (1, 3, 3, 8, 1, "valid"), (2, 5, 4, 260, 1, "same"),      # a second, nearly empty block
    (1, 16, 9, 4, 1, "same"), (1, 17, 9, 12, 1, "valid"), (1, 41, 5, 4, 1, "same"),    # several segments, the last shorter
    (1, 40, 41, 20, 2, "same"), (2, 9, 8, 4, 2, "valid"), (1, 12, 12, 512, 2, "same"),
    (70, 19, 61, 4, 1, "same"), (40, 31, 33, 128, 1, "same"),                          # more units than lanes take at once
    (2, 20, 21, 8, 3, "same"), (2, 20, 21, 8, (2, 1), "valid"),                        # strides of the general kernel
    (1, 9, 9, 8, 1, 2),                                                                # padding beyond the filter's middle
])
def test_filter_gradient(tf, n, h, w, c, stride, pad):
    print("dW", n, h, w, c, stride, pad, flush=True)
    from oracle import cpu_ref as ref
    rng = np.random.default_rng(n + h + w + c)
    ci = ref.compute_conv2d_info((n, h, w, c), (3, 3, c, 1), stride, 1, pad, depthwise=True)
    p = ci["padInfo"]
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    dy = rng.standard_normal(ci["outShape"]).astype(np.float32)
    with tf.tidy():
        got = tf.depthwise_conv2d_der_filter(tf.tensor(x), tf.tensor(dy), (3, 3, c, 1), stride, pad).data_sync()
    oh, ow, sh, sw = ci["outHeight"], ci["outWidth"], ci["strideHeight"], ci["strideWidth"]
    padded = np.zeros((n, oh * sh + h + 8, ow * sw + w + 8, c))
    padded[:, p["top"]:p["top"] + h, p["left"]:p["left"] + w] = x
    for i in range(3):
        for j in range(3):
            part = padded[:, i:i + (oh - 1) * sh + 1:sh, j:j + (ow - 1) * sw + 1:sw]
            want, magnitude = (part * dy).sum((0, 1, 2)), np.abs(part * dy).sum((0, 1, 2))
            # a lane adds at most 64 products in float32, the rest is added in float64
            assert np.all(np.abs(got[i, j, :, 0] - want) <= 66 * 2.0 ** -24 * magnitude)


@pytest.mark.parametrize("n,h,w,c,stride,chain", [
    (8, 14, 14, 512, 1, 8), (32, 28, 28, 128, 1, 8), (16, 14, 14, 256, 2, 8), (6, 17, 20, 64, 1, 8), (1, 14, 14, 512, 1, 8),
    (1, 10, 6, 16, 1, 1), (2, 8, 4, 16, 1, 1), (1, 28, 28, 32, 1, 7),
])
def test_chains_of_low_images_are_short(tf, n, h, w, c, stride, chain):
    """Where there are lanes for them, no lane adds more than 8 products in float32, and fewer of a tiny image:
    a column of 2^25 and ones keeps the ones that its first sum does not meet."""
    print("chains", n, h, w, c, stride, flush=True)
    oh, ow = -(-h // stride), -(-w // stride)
    dy = np.ones((n, oh, ow, c), np.float32)
    columns = n * ow
    assert columns % 2 == 0
    dy[:, 0] = np.where(np.arange(columns) % 2, -2.0 ** 25, 2.0 ** 25).reshape(n, ow, 1)
    with tf.tidy():
        got = tf.depthwise_conv2d_der_filter(tf.tensor(np.ones((n, h, w, c), np.float32)), tf.tensor(dy),
                                             (3, 3, c, 1), stride, "same").data_sync()
    lost = columns * (oh - 1) - got[1, 1, :, 0]
    assert np.all(lost >= 0) and np.all(lost <= columns * (chain - 1)), (lost.min(), lost.max(), columns)
