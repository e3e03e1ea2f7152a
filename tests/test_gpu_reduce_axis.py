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


def _plan(tf, shape, parts):
    """The number of kernels such a reduction takes: the axis cut over workgroups needs a second one."""
    x = tf.tensor(np.ones(shape, np.float32))
    with tf.tidy():
        names = [k[0] if isinstance(k, tuple) else k["name"] for k in tf.time(lambda: tf.sum(x, 0))["kernelTimes"]]
    x.dispose()
    assert ("reduce_finish" in names) == (parts > 1), names


@pytest.mark.parametrize("rows,parts", [(900, 1), (20000, 2)])
def test_logical_outcomes_in_one_launch_and_two(tf, rows, parts):
    """Columns of every outcome, decided in the first, a middle and the last slice of the axis."""
    cols = 12
    _plan(tf, (rows, cols), parts)
    flags = np.ones((rows, cols), bool)
    flags[:, 1] = False                                       # all false
    for col, row in ((2, 0), (3, rows // 2), (4, rows - 1)):  # one false
        flags[row, col] = False
    flags[:, 5:8] = False
    for col, row in ((5, 0), (6, rows // 2), (7, rows - 1)):  # one true
        flags[row, col] = True
    flags[:, 8:] = np.random.default_rng(rows).random((rows, cols - 8)) < 0.5
    with tf.tidy():
        t = tf.tensor(flags)
        got_all, got_any = tf.all(t, 0).data_sync(), tf.any(t, 0).data_sync()
    np.testing.assert_array_equal(got_all, flags.all(0))
    np.testing.assert_array_equal(got_any, flags.any(0))
    assert flags.all(0).any() and not flags.any(0).all()


@pytest.mark.parametrize("rows,parts", [(900, 1), (20000, 2)])
def test_products_over_leading_axes(tf, rows, parts):
    rng = np.random.default_rng(rows)
    x = (1 + rng.uniform(-1, 1, (rows, 12)) / 64).astype(np.float32)
    x[rows // 3, 5] = 0
    x[:, 6] = -x[:, 6]
    ints = np.ones((rows, 8), np.int32)
    ints[0], ints[rows // 2, :4], ints[-1, 2:6] = 3, -7, 2
    _plan(tf, x.shape, parts)
    with tf.tidy():
        got, goti = tf.prod(tf.tensor(x), 0).data_sync(), tf.prod(tf.tensor(ints), 0).data_sync()
    want = x.astype(np.float64).prod(0)
    # products in double, one rounding each, and one to float32
    assert np.all(np.abs(got - want) <= (2.0 ** -24 + rows * 2.0 ** -52) * np.abs(want))
    np.testing.assert_array_equal(goti, ints.prod(0))


def test_ties_and_nan_across_slices(tf):
    """As in test_reduce_axis_ties_and_nan, with the axis cut: equal values in different slices, NaN in
    element 0 (which stays) and in others (which never win), infinities at the ends."""
    rows = 20000
    _plan(tf, (rows, 8), 2)
    x = np.zeros((rows, 8), np.float32)
    x[11000, 0] = x[19999, 0] = x[400, 0] = 5
    x[19999, 1] = 7
    x[0, 2] = np.nan
    x[9000:9100, 3] = np.nan
    x[15000, 3] = 2
    x[0, 4], x[rows - 1, 4] = -np.inf, np.inf
    x[:, 5] = -np.inf
    x[:, 6] = np.arange(rows, 0, -1)
    with tf.tidy():
        t, turned = tf.tensor(x), tf.tensor(np.ascontiguousarray(x.T))
        for name in ("arg_max", "arg_min", "max", "min"):
            got, want = getattr(tf, name)(t, 0).data_sync(), getattr(tf, name)(turned, 1).data_sync()
            np.testing.assert_array_equal(got, want, err_msg=name)
        idx, top = tf.arg_max(t, 0).data_sync(), tf.max(t, 0).data_sync()
    assert list(idx[:2]) == [400, 19999] and np.isnan(top[2]) and idx[2] == 0
    assert idx[3] == 15000 and top[3] == 2 and idx[4] == rows - 1 and idx[5] == 0 and idx[6] == 0


@pytest.mark.parametrize("shape,axis", [
    ((300001, 5), 0),      # 512 slices, combined by 32 rows of lanes in two trips; fewer columns than a workgroup takes
    ((70003, 36), 0),      # four columns per lane, a second workgroup of columns that is nearly empty
    ((4097, 44), 0),       # two slices
    ((3, 20011, 21), 1),   # outer extents among the columns
    ((1024, 4), 0),        # one launch: eight elements for every row lane
    ((1025, 4), 0),        # and one more
])
def test_sliced_columns_of_every_operation(tf, shape, axis):
    print("sliced columns", shape, axis, flush=True)
    rng = np.random.default_rng(sum(shape))
    x = rng.integers(-4, 5, shape).astype(np.float32)          # sums exact, extrema tied
    near = (1 + 1e-4 * rng.standard_normal(shape)).astype(np.float32)
    flags = rng.random(shape) < 2.0 / shape[axis]
    with tf.tidy():
        t, tn, tb = tf.tensor(x), tf.tensor(near), tf.tensor(flags)
        for op in ("sum", "max", "min"):
            np.testing.assert_array_equal(getattr(tf, op)(t, axis).data_sync(), getattr(np, op)(x, axis))
        for op, want in (("arg_max", np.argmax), ("arg_min", np.argmin)):
            np.testing.assert_array_equal(getattr(tf, op)(t, axis).data_sync(), want(x, axis))
        np.testing.assert_array_equal(tf.any(tb, axis).data_sync(), flags.any(axis))
        np.testing.assert_array_equal(tf.all(tf.logical_not(tb), axis).data_sync(), (~flags).all(axis))
        mean, prod = tf.mean(tn, axis).data_sync(), tf.prod(tn, axis).data_sync()
    # the quotients are rounded to float32 before they are added, the sum once more
    want = near.astype(np.float64).mean(axis)
    assert np.all(np.abs(mean - want) <= 2 * 2.0 ** -24 * np.abs(want) + 2.0 ** -24)
    want = near.astype(np.float64).prod(axis)
    assert np.all(np.abs(prod - want) <= 2 * 2.0 ** -24 * np.abs(want))
