"""Writes and reads that a kernel carries: sizes around what fits a launch, a pinned slot and the
staging block, with the stream idle and busy, and what is queued around them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.mark.parametrize("nbytes", [1, 3, 4, 63, 255, 256, 257, 511, 513, 65535, 65536, 65537, 65553, 602113,
                                    (1 << 20) - 1, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("busy", [False, True])
def test_round_trip(tf, nbytes, busy):
    print("round trip", nbytes, busy, flush=True)
    rng = np.random.default_rng(nbytes)
    flags = rng.integers(0, 2, nbytes).astype(bool)
    numbers = rng.standard_normal(max(1, nbytes // 4)).astype(np.float32)
    with tf.tidy():
        big = tf.tensor(np.ones((2048, 2048), np.float32))
        tf.backend().sync()
        if busy:
            big = tf.matmul(big, big)
        neighbour = tf.tensor(numbers + 1)
        a = tf.tensor(flags)
        b = tf.tensor(numbers)
        want = numbers.copy()
        numbers[:] = 0                               # the caller's array is its own again
        twice = tf.add(b, b)
        np.testing.assert_array_equal(a.data_sync().astype(bool), flags)
        np.testing.assert_array_equal(b.data_sync(), want)
        np.testing.assert_array_equal(twice.data_sync(), want + want)
        np.testing.assert_array_equal(neighbour.data_sync(), want + 1)   # (nothing past the end was touched)


@pytest.mark.parametrize("n", [1, 64, 65, 20000, 150528])
def test_rewrites_stay_in_order(tf, n):
    """New values into one tensor while kernels that read the old ones are queued, on both streams."""
    be = tf.backend()
    with tf.tidy():
        x = tf.tensor(np.zeros(n, np.float32))
        outs = []
        for i in range(12):
            be.select_stream(i % 2)
            be.write(x.data_id, np.full(n, i, np.float32))
            outs.append(tf.add(x, tf.tensor(np.full(n, 0.5, np.float32))))
            if i % 3 == 2:
                be.sync()                            # the stream is idle for the next write
        be.select_stream(0)
        for i, o in enumerate(outs):
            np.testing.assert_array_equal(o.data_sync(), np.full(n, i + 0.5, np.float32))


def test_a_copy_is_no_kernel_of_a_timed_region(tf):
    with tf.tidy():
        x = tf.tensor(np.ones(300000, np.float32))
        info = tf.time(lambda: tf.add(tf.mul(x, 2.0), tf.tensor(np.ones(300000, np.float32))).data_sync())
        assert len(info["kernelTimes"]) == 2


def _address_space():
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) << 10 for line in f if line.startswith("VmSize"))


def test_reads_of_many_sizes_share_their_memory(tf):
    """Page-locked memory for reads does not grow with the number of sizes that are read."""
    sizes = [(512 << 10) - 4 * i for i in range(0, 128 * 160, 160)] + [1, 3, 128, 129]
    with tf.tidy():
        made = [tf.add(tf.tensor(np.full(n // 4 or 1, n, np.float32)), tf.tensor(np.float32(0.5))) for n in sizes]
        made[0].data_sync()
        before = _address_space()
        for n, t in zip(sizes, made):
            got = t.data_sync()
            assert got.size == (n // 4 or 1) and np.all(got == np.float32(n + 0.5))
        # (a block per size would be 56 MB)
        assert _address_space() - before < 16 << 20


def test_reads_on_several_threads(tf):
    import threading
    wrong = []
    with tf.tidy():
        made = [tf.add(tf.tensor(np.arange(n, dtype=np.float32)), tf.tensor(np.float32(i)))
                for i, n in enumerate((1000, 70000, 250000, 200000))]
        tf.backend().sync()

        def read(i, t):
            for _ in range(200):
                got = t.data_sync()
                if not np.array_equal(got, np.arange(got.size, dtype=np.float32) + i):
                    wrong.append(i)
        threads = [threading.Thread(target=read, args=(i, t)) for i, t in enumerate(made)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong
