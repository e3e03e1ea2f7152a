"""Reductions over axes that are not the innermost ones (tfhip_reduce_axis), at the edges of its
plans: one launch and two, four columns per lane and one, ragged columns, short axes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("shape,axes", [
    ((1000, 512), (0,)),            # one launch, four columns per lane
    ((2049, 12), (0,)),             # just beyond it: the axis is cut, 3 column lanes
    ((2048, 1), (0,)),              # one column
    ((9001, 3), (0,)),              # columns that no lane takes four of
    ((3, 1000, 37), (1,)),          # outer and inner extents, ragged columns
    ((5, 7), (0,)), ((1, 9), (0,)), # fewer elements than row lanes
    ((4, 33, 20, 128), (0, 1, 2)),  # the statistics of a batch norm
    ((2, 70001, 8), (1,)),          # a slice that ends before the others
    ((100003, 3, 2), (1,)),         # many short sums: one row lane, 512 columns of many outer indices
    ((70001, 5, 8), (1,)),          # the same, four columns per lane, some row lanes without elements
    ((1003, 33, 7), (1,)), ((5000, 9, 12), (1,)), ((300, 300, 20), (1,)),   # a few row lanes
])
def test_reduce_axis(tf, shape, axes):
    print("reduce axis", shape, axes, flush=True)
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape).astype(np.float32)
    n = int(np.prod([shape[a] for a in axes]))
    ints, flags = rng.integers(-1000, 1000, shape).astype(np.int32), x > 1.0
    with tf.tidy():
        t, ti, tb = tf.tensor(x), tf.tensor(ints), tf.tensor(flags)
        got = {k: getattr(tf, k)(t, list(axes)).data_sync() for k in ("sum", "mean", "max", "min")}
        np.testing.assert_array_equal(tf.sum(ti, list(axes)).data_sync(), ints.sum(axes))
        np.testing.assert_array_equal(tf.max(ti, list(axes)).data_sync(), ints.max(axes))
        np.testing.assert_array_equal(tf.any(tb, list(axes)).data_sync(), flags.any(axes))
        np.testing.assert_array_equal(tf.all(tb, list(axes), True).data_sync(), flags.all(axes, keepdims=True))
        if len(axes) == 1:
            np.testing.assert_array_equal(tf.arg_max(t, axes[0]).data_sync(), x.argmax(axes[0]))
            np.testing.assert_array_equal(tf.arg_min(t, axes[0]).data_sync(), x.argmin(axes[0]))
    np.testing.assert_array_equal(got["max"], x.max(axes))
    np.testing.assert_array_equal(got["min"], x.min(axes))
    # sums in double, rounded to float32 once; a mean rounds every quotient first
    x64 = x.astype(np.float64)
    assert np.all(np.abs(got["sum"] - x64.sum(axes)) <= 2.0 ** -24 * np.abs(x64.sum(axes)) + 1e-12 * n)
    q64 = (x / np.float32(n)).astype(np.float64)
    assert np.all(np.abs(got["mean"] - q64.sum(axes)) <= 2.0 ** -24 * np.abs(q64.sum(axes)) + 1e-12)


def test_reduce_axis_ties_and_nan(tf):
    """Of equal values the first index wins; NaN survives from element 0 only, as in a row."""
    x = np.zeros((3000, 8), np.float32)
    x[17, 2] = x[2500, 2] = 5
    x[0, 3] = np.nan
    x[9, 4] = np.nan
    x[11, 4] = 1
    with tf.tidy():
        t = tf.tensor(x)
        idx, top = tf.arg_max(t, 0).data_sync(), tf.max(t, 0).data_sync()
        want_idx, want_top = tf.arg_max(tf.transpose(t), 1).data_sync(), tf.max(tf.transpose(t), 1).data_sync()
    assert idx[2] == 17 and np.isnan(top[3]) and top[4] == 1
    np.testing.assert_array_equal(idx, want_idx)
    np.testing.assert_array_equal(top, want_top)


def test_more_outer_indices_than_a_launch_has_workgroups(tf):
    """8.4 million of them at one workgroup of 512 each would be more lanes than 32 bits count."""
    x = np.random.default_rng(4).standard_normal((8400000, 2, 2)).astype(np.float32)
    with tf.tidy():
        t = tf.tensor(x)
        got, top = tf.sum(t, 1).data_sync(), tf.arg_max(t, 1).data_sync()
    np.testing.assert_array_equal(got, x.astype(np.float64).sum(1).astype(np.float32))
    np.testing.assert_array_equal(top, x.argmax(1))
