"""scatterND and unsortedSegmentSum over slices of half a wavefront and more, where a
workgroup gathers the updates of its rows: list lengths around a pass, hot rows, ragged slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip as tf
    tf.set_backend("hip")
    return tf


@pytest.mark.parametrize("rows,slice_,n", [
    (1, 32, 1), (3, 33, 4095), (5000, 64, 4096), (70, 65, 4097), (20000, 128, 10240), (257, 129, 9000),
    (33, 300, 700), (1031, 31, 3000),   # the last: below the line
])
def test_segment_sum(tf, rows, slice_, n):
    rng = np.random.default_rng(rows + slice_ + n)
    # frequent rows (long chains), ids outside the range at both ends
    ids = np.minimum((np.exp(rng.random(n) * np.log(rows + 1)) - 1).astype(np.int32), rows - 1)
    ids[:: 17] = -3
    ids[5:: 19] = rows
    x = rng.standard_normal((n, slice_)).astype(np.float32)
    with tf.tidy():
        got = tf.unsorted_segment_sum(tf.tensor(x), tf.tensor(ids), rows).data_sync()
    want = np.zeros((rows, slice_))
    ok = (ids >= 0) & (ids < rows)
    np.add.at(want, ids[ok], x[ok].astype(np.float64))
    assert np.array_equal(got, want.astype(np.float32))   # summed in float64 in list order, rounded once


@pytest.mark.parametrize("dtype", ["float32", "int32"])
def test_scatter_nd_rounds_every_sum_in_order(tf, dtype):
    rng = np.random.default_rng(8)
    rows, slice_, n = 37, 130, 5000
    ids = rng.integers(0, rows, (n, 1)).astype(np.int32)
    x = rng.standard_normal((n, slice_)).astype(np.float32) if dtype == "float32" else \
        rng.integers(-2 ** 31, 2 ** 31, (n, slice_)).astype(np.int32)
    with tf.tidy():
        got = tf.scatter_nd(tf.tensor(ids), tf.tensor(x, dtype=dtype), [rows, slice_]).data_sync()
    want = np.zeros((rows, slice_), x.dtype)
    with np.errstate(over="ignore"):
        np.add.at(want, ids[:, 0], x)
    assert np.array_equal(got, want)

