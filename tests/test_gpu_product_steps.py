"""Matrix products at every number of k steps around the ends of the pipeline: one step to two blocks of 48
and on, whole and cut last steps, in the layouts that the tiled kernels read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("m,n", [(2048, 640), (1031, 517), (4096, 32), (1500, 1028)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_steps(tf, m, n, ta, tb):
    rng = np.random.default_rng(m + n)
    for k in (1, 4, 15, 16, 17, 32, 36, 48, 49, 63, 64, 80, 95, 96, 97, 112, 128, 144, 145, 192, 200, 260):
        print("steps", m, k, n, ta, tb, flush=True)
        a = rng.standard_normal((k, m) if ta else (m, k)).astype(np.float32)
        b = rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32)
        with tf.tidy():
            got = tf.matmul(tf.tensor(a), tf.tensor(b), ta, tb).data_sync().reshape(m, n)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        a64, b64 = a64.T if ta else a64, b64.T if tb else b64
        # k products, each rounded with its sum: at most one half ulp of the magnitudes for each of them
        # and for each block's sum
        bound = (min(k, 48) + k / 48 + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
        assert (np.abs(got - a64 @ b64) <= bound).all()
