"""Copies of boxes whose innermost dimension lies side by side on both sides, or is a mirrored row of small
pixels: every output element is one input element, so the results are exact.  Widths around the shortest
run (8), what four does not divide, starts that 16 bytes do not divide, and the types of one byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


def values(shape, dtype, seed):
    rng = np.random.default_rng(seed)
    if dtype == "bool":
        return rng.integers(0, 2, shape).astype(bool)
    if dtype == "int32":
        return rng.integers(-2 ** 31, 2 ** 31 - 1, shape).astype(np.int32)
    x = rng.standard_normal(shape).astype(np.float32)
    x.flat[::7] = [np.nan, np.inf, -np.inf, -0.0][seed % 4]  # bits, not numbers
    return x


def same(got, want):
    want = np.ascontiguousarray(want)
    got = np.asarray(got).reshape(want.shape).astype(want.dtype)
    np.testing.assert_array_equal(got.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("dtype", ["float32", "int32", "bool"])
@pytest.mark.parametrize("w", [1, 4, 7, 8, 9, 11, 64, 257])
@pytest.mark.parametrize("c", [1, 2, 3, 4, 8, 13])
def test_boxes(tf, dtype, w, c):
    print("boxes", dtype, w, c, flush=True)
    x = values((3, 5, w, c), dtype, w + c)
    with tf.tidy():
        t = tf.tensor(x, dtype=dtype)
        for axes in ([2], [1], [3], [0, 2], [1, 2], [2, 3], [0, 1, 2, 3]):
            same(tf.reverse(t, axes).data_sync(), np.flip(x, axes))
        for begin in (0, 1):
            if w - begin > 1:
                size = [2, 4, w - 1 - begin, c]
                same(tf.slice(t, [1, 1, begin, 0], size).data_sync(),
                     x[1:3, 1:5, begin:begin + size[2]])
        if c > 1:
            same(tf.slice(t, [0, 0, 0, 1], [3, 5, w, c - 1]).data_sync(), x[..., 1:])
        same(tf.strided_slice(t, [0, 0, w - 1, 0], [3, 5, -w - 1, c], [1, 2, -1, 1]).data_sync(),
             x[:, ::2, ::-1])
        same(tf.concat([t, t], 3).data_sync(), np.concatenate([x, x], 3))
        same(tf.concat([t, t], 2).data_sync(), np.concatenate([x, x], 2))
        if dtype != "bool":
            same(tf.pad(t, [[0, 1], [1, 0], [1, 2], [0, 3]]).data_sync(),
                 np.pad(x, [[0, 1], [1, 0], [1, 2], [0, 3]]))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 1021, 300001])
def test_lines(tf, n):
    print("lines", n, flush=True)
    x = values((n + 3,), "float32", n)
    with tf.tidy():
        t = tf.tensor(x)
        same(tf.reverse(t, [0]).data_sync(), x[::-1])
        for b in range(4):
            same(tf.reverse(tf.slice(t, [b], [n]), [0]).data_sync(), x[b:b + n][::-1])
        same(tf.strided_slice(t, [n], [0], [-1]).data_sync(), x[n:0:-1])
