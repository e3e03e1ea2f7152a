"""The entry points that the extension module of the Python host calls itself: operands, refusals and
messages as through ctypes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("a,b", [((3, 4), (3, 4)), ((3, 4), (4,)), ((3, 1), (1, 4)), ((), (2, 3)), ((5, 1, 2), (7, 1)),
                                 ((0, 3), (3,)), ((1,) * 6, (2,)), ((2, 1), ())])
def test_binary_shapes(tf, a, b):
    rng = np.random.default_rng(len(a))
    x, y = rng.standard_normal(a).astype(np.float32), rng.standard_normal(b).astype(np.float32)
    with tf.tidy():
        got = tf.add(tf.tensor(x), tf.tensor(y))
        assert got.shape == np.broadcast_shapes(a, b)
        np.testing.assert_array_equal(got.data_sync(), x + y)


def test_refusals(tf):
    base = tf.memory()
    with tf.tidy():
        x = tf.tensor(np.ones((2, 3), np.float32))
        with pytest.raises(ValueError, match="could not be broadcast"):
            tf.add(x, tf.tensor(np.ones((2, 2), np.float32)))
        with pytest.raises(RuntimeError):
            tf.add(tf.tensor(np.ones((1,) * 9, np.float32)), x)
        with pytest.raises(ValueError, match="has not been implemented"):
            tf.fused.matmul(x, x, False, True, activation="other")
        with pytest.raises(RuntimeError, match="already registered"):
            tf.backend().register(x.data_id, (2, 3), "float32")
        with pytest.raises(KeyError):
            tf.backend().register(object(), (2, 3), "float64")
        with pytest.raises(TypeError):
            tf.backend()._binary_out(0, x)
        gone = tf.tensor(np.ones(3, np.float32))
        gone.dispose()
        with pytest.raises(KeyError):
            tf.relu(gone)
    after = tf.memory()
    assert after["numTensors"] == base["numTensors"] and after["numDeviceBuffers"] == base["numDeviceBuffers"]


def test_products_of_any_rank_and_epilogue(tf):
    """The product straight from its operands, and the epilogues that take separate passes."""
    rng = np.random.default_rng(1)
    a, b = rng.standard_normal((2, 3, 4, 5)).astype(np.float32), rng.standard_normal((2, 3, 5, 6)).astype(np.float32)
    want = a.astype(np.float64) @ b
    odd = rng.standard_normal((4, 1)).astype(np.float32)      # a bias that no epilogue folds
    with tf.tidy():
        got = tf.matmul(tf.tensor(a), tf.tensor(b))
        assert got.shape == want.shape
        np.testing.assert_allclose(got.data_sync(), want, atol=1e-5)
        got = tf.fused.matmul(tf.tensor(a), tf.tensor(b), bias=tf.tensor(odd), activation="relu").data_sync()
        np.testing.assert_allclose(got, np.maximum(want + odd, 0), atol=1e-5)
        ints = np.arange(6, dtype=np.int32).reshape(2, 3)
        r = tf.matmul(tf.tensor(ints), tf.tensor(ints), False, True)
        assert r.dtype == "int32"
        np.testing.assert_array_equal(r.data_sync(), ints @ ints.T)
        for value in (2.5, -0.0, float("inf"), float("nan"), 1e-45):
            np.testing.assert_array_equal(tf.tensor(value).data_sync(), np.float32(value))


@pytest.mark.parametrize("quant", [(0.25, -3.0), [0.25, -3.0], [1, -3]])
def test_quantised_weights_in_any_sequence(tf, quant):
    """What the dense kernels take as (scale, min) is what dequantize takes."""
    from tfhip.engine import Tensor
    rng = np.random.default_rng(5)
    a, q = rng.standard_normal((6, 16)).astype(np.float32), rng.integers(0, 256, (16, 8)).astype(np.uint8)
    want = a.astype(np.float64) @ (q * float(quant[0]) + quant[1])
    with tf.tidy():
        w = Tensor((16, 8), "float32", None, q, tf.backend(), quant)
        got = tf.matmul(tf.tensor(a), w).data_sync()
        x, f = tf.tensor(a.reshape(1, 2, 3, 16)), tf.reshape(w, (1, 1, 16, 8))
        conv = tf.fused.conv2d(x, f, 1, "valid").data_sync()
    # (float32 sums of 16 products: 17 roundings of terms of at most this size)
    bound = 17 * 2.0 ** -24 * (np.abs(a) @ np.abs(q * float(quant[0]) + quant[1]))
    assert np.all(np.abs(got - want) <= bound)
    assert np.all(np.abs(conv.reshape(6, 8) - want) <= bound)
