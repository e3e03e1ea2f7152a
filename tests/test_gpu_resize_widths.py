"""Resizes up and down by one and by four channels per lane: channels around four, images of one row or
column, last rows and columns, several images, integer pictures and rows that start off 16 bytes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("align", [False, True])
@pytest.mark.parametrize("c", [1, 3, 4, 5, 8, 12])
@pytest.mark.parametrize("n,h,w,oh,ow", [(1, 1, 1, 1, 1), (2, 1, 7, 5, 3), (3, 9, 1, 4, 1), (2, 13, 17, 31, 8),
                                         (1, 30, 40, 14, 15), (2, 6, 5, 18, 25)])
def test_resize(tf, n, h, w, oh, ow, c, align):
    print("resize", n, h, w, oh, ow, c, align, flush=True)
    from oracle import cpu_ref as ref
    rng = np.random.default_rng(h * 100 + w + c)
    x = rng.standard_normal((n, h, w, c)).astype(np.float32)
    pictures = rng.integers(0, 256, (n, h, w, c)).astype(np.int32)
    with tf.tidy():
        for host in (x, pictures):
            t = tf.tensor(host, dtype=str(host.dtype))
            got = tf.resize_bilinear(t, (oh, ow), align).data_sync().reshape(n, oh, ow, c)
            want = ref.resize_bilinear(host, oh, ow, align)
            # both interpolate in double, with up to 2^-50 of the pixels between them, and round once:
            # the same float32 or its neighbour
            np.testing.assert_array_less(np.abs(got - want.astype(np.float64)),
                                         2.0 ** -23 * np.abs(want) + 2.0 ** -48 * np.abs(host).max() + 1e-45)
            got = tf.resize_nearest_neighbor(t, (oh, ow), align).data_sync().reshape(n, oh, ow, c)
            np.testing.assert_array_equal(got, ref.resize_nearest_neighbor(host, oh, ow, align))
