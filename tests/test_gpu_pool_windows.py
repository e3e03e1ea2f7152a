"""Max and average pooling and the gradient of max pooling with the windows that have kernels of
their own, at the edges of images and blocks, against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("n,h,w,c,f,stride,pad", [
    (2, 8, 8, 4, 2, 2, "same"), (2, 9, 7, 12, 2, 2, "same"), (1, 9, 11, 8, 2, 2, "valid"),   # rows no window covers
    (2, 8, 9, 4, 3, 2, "same"), (3, 7, 10, 20, 3, 2, "valid"), (1, 1, 1, 4, 3, 2, "same"),
    (1, 2, 1, 8, 2, 2, "same"), (1, 9, 11, 4, 3, 2, 1), (1, 8, 6, 4, 2, 2, 1),               # padding on both sides
    (1, 7, 7, 4, 3, 2, 2), (4, 33, 35, 36, 3, 2, "same"), (2, 8, 7, 8, 3, 1, "same"), (1, 9, 9, 4, 2, 3, "same"),
])
def test_windows(tf, n, h, w, c, f, stride, pad):
    from oracle import cpu_ref as ref
    print("pool windows", n, h, w, c, f, stride, pad, flush=True)
    rng = np.random.default_rng(h * 100 + w + f)
    x = rng.integers(0, 5, (n, h, w, c)).astype(np.float32)     # ties: the first maximum wins
    x[0, h // 2, w // 2, 0] = np.nan                             # never wins
    x[-1, :, :, 1] = -np.inf                                     # windows without a winner
    x[0, 0, 0, 2] = np.inf
    ci = ref.compute_pool2d_info(x.shape, f, stride, 1, pad)
    dy = rng.standard_normal(ci["outShape"]).astype(np.float32)
    with tf.tidy():
        tx = tf.tensor(x)
        mx = tf.max_pool(tx, f, stride, pad).data_sync()
        avg = tf.avg_pool(tx, f, stride, pad).data_sync()
        dx = tf.max_pool_backprop(tf.tensor(dy), tx, f, stride, pad).data_sync()
    np.testing.assert_array_equal(mx, ref.max_pool(x, ci))
    np.testing.assert_array_equal(avg, ref.avg_pool(x, ci))      # summed in double, rounded once
    # a pixel's gradients are added in float32: fewer than f * f roundings of partial sums of |dy|
    bound = f * f * 2.0 ** -24 * ref.max_pool_backprop(np.abs(dy), x, ci)
    assert np.all(np.abs(dx.astype(np.float64) - ref.max_pool_backprop(dy, x, ci)) <= bound)


@pytest.mark.parametrize("f", [2, 3])
def test_gradient_of_a_window_below_everything(tf, f):
    """Infinite and NaN gradients reach the winning pixels and no others."""
    rng = np.random.default_rng(f)
    x = rng.permutation(8 * 8 * 4).reshape(1, 8, 8, 4).astype(np.float32)
    dy = np.full((1, 4, 4, 4), np.inf, np.float32)
    dy[0, 1] = np.nan
    with tf.tidy():
        dx = tf.max_pool_backprop(tf.tensor(dy), tf.tensor(x), f, 2, "same").data_sync()
    from oracle import cpu_ref as ref
    np.testing.assert_array_equal(dx, ref.max_pool_backprop(dy, x, ref.compute_pool2d_info(x.shape, f, 2, 1, "same")))
