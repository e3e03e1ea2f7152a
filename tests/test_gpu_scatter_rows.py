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
    want, magnitude = np.zeros((rows, slice_)), np.zeros((rows, slice_))
    ok = (ids >= 0) & (ids < rows)
    np.add.at(want, ids[ok], x[ok].astype(np.float64))
    np.add.at(magnitude, ids[ok], np.abs(x[ok]).astype(np.float64))
    # Summed in float64 and rounded once; in list order up to 64 entries of a row, beyond them in
    # parts, which moves the float64 sum by at most a rounding per entry.
    few = np.bincount(ids[ok], minlength=rows) <= 64
    assert np.array_equal(got[few], want[few].astype(np.float32))
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + n * 2.0 ** -52 * magnitude)


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



@pytest.mark.parametrize("rows,slice_,n", [
    (2, 40, 9001), (5, 128, 8193), (3, 200, 5000), (1, 257, 4097),     # rows whose chains are cut, in every width
    (20000, 128, 12000),                                               # as many workgroups as the machine holds
    (60000, 300, 6000), (150000, 64, 5000),                            # more of them: four wavefronts each
    (9, 64, 1024), (9, 64, 1025),                                      # the line between the two
])
def test_long_chains(tf, rows, slice_, n):
    """Rows with more entries than a set of wavefronts adds alone, next to rows with few."""
    print("long chains", rows, slice_, n, flush=True)
    rng = np.random.default_rng(rows + slice_ + n)
    ids = rng.integers(0, rows, n).astype(np.int32)
    ids[rng.random(n) < 0.6] = rows // 2
    ids[rng.random(n) < 0.2] = 0
    ids[::50] = -1
    x = rng.standard_normal((n, slice_)).astype(np.float32)
    with tf.tidy():
        got = tf.unsorted_segment_sum(tf.tensor(x), tf.tensor(ids), rows).data_sync()
        # exact sums in any order, and what must reach every element of a hot row and no other
        whole = rng.integers(-8, 9, (n, slice_)).astype(np.float32)
        got_whole = tf.unsorted_segment_sum(tf.tensor(whole), tf.tensor(ids), rows).data_sync()
        whole[np.flatnonzero(ids == 0)[-1], 3] = np.inf
        got_inf = tf.unsorted_segment_sum(tf.tensor(whole), tf.tensor(ids), rows).data_sync()
    ok = ids >= 0
    want, magnitude, want_whole = (np.zeros((rows, slice_)) for _ in range(3))
    np.add.at(want, ids[ok], x[ok].astype(np.float64))
    np.add.at(magnitude, ids[ok], np.abs(x[ok]).astype(np.float64))
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + n * 2.0 ** -52 * magnitude)
    finite = whole.copy()
    finite[np.flatnonzero(ids == 0)[-1], 3] = 0
    bad = np.argwhere(~np.isfinite(got_inf))
    assert bad.tolist() == [[0, 3]]
    got_inf[0, 3] = got_whole[0, 3] = 0
    np.add.at(want_whole, ids[ok], finite[ok].astype(np.float64))
    want_whole[0, 3] = 0
    np.testing.assert_array_equal(got_whole, want_whole)
    np.testing.assert_array_equal(got_inf, want_whole)
