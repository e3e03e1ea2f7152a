"""Memory whose address was given out: work that others queued on it on the default stream comes before
the next upload into the same block, also where the context's own streams had nothing left to do."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D2H, D2D = 2, 3


@pytest.fixture(scope="module")
def tf():
    import tfhip
    tfhip.set_backend("hip")
    return tfhip


@pytest.fixture(scope="module")
def hip(tf):
    """The HIP runtime that the library itself is linked to."""
    tf.backend()
    with open("/proc/self/maps") as maps:
        paths = {line.split()[-1] for line in maps if "libamdhip64.so" in line}
    assert len(paths) == 1, paths
    lib = C.CDLL(paths.pop())
    lib.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    lib.hipFree.argtypes = [C.c_void_p]
    lib.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    lib.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    return lib


def _address(be, t):
    ptr, nbytes = C.c_void_p(), C.c_size_t()
    be._ck(be.lib.tfhip_device_ptr(be.ctx, be._h(t), C.byref(ptr), C.byref(nbytes)))
    return ptr.value, nbytes.value


@pytest.mark.parametrize("outside", ["reads", "writes"])
@pytest.mark.parametrize("n,pinned", [(1 << 20, False), (1 << 15, True), (1 << 20, True)])
@pytest.mark.parametrize("passed_on", [False, True])
def test_uploads_wait_for_work_queued_on_the_address(tf, hip, outside, n, pinned, passed_on):
    print("shared address", outside, n, pinned, passed_on, flush=True)
    be = tf.backend()
    new = (be.pinned_array("float32", (n,)) if pinned else np.empty(n, np.float32))
    new[:] = np.arange(n) + 7
    big, spare = C.c_void_p(), C.c_void_p()
    half = 1 << 29
    assert hip.hipMalloc(C.byref(big), 2 * half) == 0 and hip.hipMalloc(C.byref(spare), 4 * n) == 0
    try:
        with tf.tidy():
            result = tf.add(tf.tensor(np.arange(n, dtype=np.float32)), tf.tensor(np.full(n, 0.5, np.float32)))
            want = result.data_sync().copy()
            be.sync()                                      # the context has nothing left to do
            at, nbytes = _address(be, result)
            assert nbytes == 4 * n
            for _ in range(24):                            # some 10 ms of other work in front
                assert hip.hipMemcpyAsync(big.value + half, big, half, D2D, None) == 0
            to, source = (spare, at) if outside == "reads" else (at, big)
            assert hip.hipMemcpyAsync(to, source, nbytes, D2D, None) == 0
            result.dispose()
            if passed_on:                                  # (an owner that queues nothing of its own)
                tf.backend()._out((n,)).dispose()
            x = tf.tensor(new)
            got = x.data_sync()
            assert _address(be, x)[0] == at, "another block: the case is not the one meant"
            assert hip.hipDeviceSynchronize() == 0
            np.testing.assert_array_equal(got, new)
            if outside == "reads":
                kept = np.empty(n, np.float32)
                assert hip.hipMemcpy(kept.ctypes.data, spare, nbytes, D2H) == 0
                np.testing.assert_array_equal(kept, want)
            else:
                np.testing.assert_array_equal(x.data_sync(), new)
    finally:
        assert hip.hipDeviceSynchronize() == 0
        hip.hipFree(big)
        hip.hipFree(spare)
