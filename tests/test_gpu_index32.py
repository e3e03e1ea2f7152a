"""Kernels that find their operands by 32-bit index arithmetic: repeated operands of any length, box
copies over merged and mirrored dimensions, per-channel normalisation, pooling gradients."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip as tf
    tf.set_backend("hip")
    return tf


@pytest.mark.parametrize("shape,small", [
    ((6, 10, 4), (4,)), ((300, 7, 20), (7, 20)), ((5, 8, 3), (3,)), ((4, 9, 7), (9, 7)), ((12, 5), ()),
    ((1024, 1021), (1021,)), ((3, 5, 7), (7,)), ((64, 1), (1,)),
])
def test_repeated_operand(tf, shape, small):
    rng = np.random.default_rng(sum(shape))
    x, y = (rng.uniform(0.5, 2, s).astype(np.float32) for s in (shape, small))
    with tf.tidy():
        tx, ty = tf.tensor(x), tf.tensor(np.asarray(y))
        for op, ref in ((tf.sub, np.subtract), (tf.div, np.divide), (tf.maximum, np.maximum)):
            np.testing.assert_array_equal(op(tx, ty).data_sync(), ref(x, y))
            np.testing.assert_array_equal(op(ty, tx).data_sync(), ref(y, x))


@pytest.mark.parametrize("shape", [(3, 17, 19, 3), (2, 1, 33, 5), (1, 4, 1, 1), (2, 300, 257, 4)])
@pytest.mark.parametrize("dtype", ["float32", "bool"])
def test_box_copies(tf, shape, dtype):
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape).astype(np.float32) if dtype == "float32" else rng.random(shape) < 0.5
    as_np = lambda t: t.data_sync().astype(x.dtype)
    with tf.tidy():
        t = tf.tensor(x)
        for axes in ([2], [0, 2], [1, 3], [0, 1, 2, 3]):
            np.testing.assert_array_equal(as_np(tf.reverse(t, axes)), np.flip(x, axes))
        np.testing.assert_array_equal(as_np(tf.tile(t, [2, 1, 3, 1])), np.tile(x, [2, 1, 3, 1]))
        begin = [s // 3 for s in shape]
        size = [s - b for s, b in zip(shape, begin)]
        np.testing.assert_array_equal(as_np(tf.slice(t, begin, size)), x[tuple(slice(b, None) for b in begin)])
        np.testing.assert_array_equal(as_np(tf.concat([t, t], 2)), np.concatenate([x, x], 2))
        if dtype == "float32":
            np.testing.assert_array_equal(as_np(tf.pad(t, [[0, 0], [1, 2], [0, 3], [0, 0]])),
                                          np.pad(x, [[0, 0], [1, 2], [0, 3], [0, 0]]))


@pytest.mark.parametrize("shape", [(2, 5, 7, 4), (3, 33, 20, 36), (2, 3, 5, 6)])
def test_batch_norm_per_channel(tf, shape):
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape).astype(np.float32)
    m, o, s = (rng.standard_normal(shape[-1]).astype(np.float32) for _ in range(3))
    v = rng.uniform(0.1, 2, shape[-1]).astype(np.float32)
    for off, sc in ((o, s), (None, s), (o, None), (None, None)):
        with tf.tidy():
            got = tf.batch_norm(tf.tensor(x), tf.tensor(m), tf.tensor(v), None if off is None else tf.tensor(off),
                                None if sc is None else tf.tensor(sc), 0.001).data_sync()
        x64 = x.astype(np.float64)
        want = (x64 - m) * (1.0 if sc is None else sc.astype(np.float64)) / np.sqrt(v.astype(np.float64) + 0.001)
        # six float32 roundings
        bound = 6 * 2.0 ** -24 * (np.abs(want) + np.abs(x64 - m) * 4 + 4)
        want = want + (0.0 if off is None else off)
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("n,h,w,c,f,stride", [(2, 9, 11, 4, 2, 2), (3, 14, 15, 20, 3, 2), (2, 8, 7, 8, 3, 1), (1, 13, 10, 4, 2, 3)])
def test_pool_gradients(tf, n, h, w, c, f, stride):
    from oracle import cpu_ref as ref
    rng = np.random.default_rng(h * w)
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    ci = ref.compute_pool2d_info(x.shape, f, stride, 1, "same")
    dy = rng.standard_normal(ci["outShape"]).astype(np.float32)
    with tf.tidy():
        got = tf.max_pool_backprop(tf.tensor(dy), tf.tensor(x), f, stride, "same").data_sync()
        avg = tf.avg_pool_backprop(tf.tensor(dy), tf.tensor(x), f, stride, "same").data_sync()
    # at most f * f gradients meet in a pixel
    np.testing.assert_allclose(got, ref.max_pool_backprop(dy, x, ci), rtol=0, atol=f * f * 2.0 ** -23 * 8)
    np.testing.assert_allclose(avg, ref.avg_pool_backprop(dy, x, ci), rtol=0, atol=f * f * 2.0 ** -23 * 8)


@pytest.mark.parametrize("n,h,w,c,stride", [(2, 9, 10, 4, 1), (8, 56, 57, 36, 1), (3, 30, 31, 128, 2), (40, 40, 41, 8, 1)])
def test_depthwise_filter_gradient(tf, n, h, w, c, stride):
    """One slice, and many whose partial sums a workgroup adds."""
    rng = np.random.default_rng(n + h + c)
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    oh, ow = -(-h // stride), -(-w // stride)
    dy = rng.standard_normal((n, oh, ow, c)).astype(np.float32)
    with tf.tidy():
        got = tf.depthwise_conv2d_der_filter(tf.tensor(x), tf.tensor(dy), (3, 3, c, 1), stride, "same").data_sync()
    ph, pw = max((oh - 1) * stride + 3 - h, 0) // 2, max((ow - 1) * stride + 3 - w, 0) // 2
    p = np.pad(x.astype(np.float64), ((0, 0), (ph, 3), (pw, 3), (0, 0)))
    for i in range(3):
        for j in range(3):
            part = p[:, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride]
            want, magnitude = (part * dy).sum((0, 1, 2)), np.abs(part * dy).sum((0, 1, 2))
            # a lane's float32 sum of at most 64 pixels or so, then float64
            assert np.all(np.abs(got[i, j, :, 0] - want) <= 66 * 2.0 ** -24 * magnitude)
