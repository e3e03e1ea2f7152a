"""The extension module of the Python host: tensor records, reference counts and scopes behave as the
interpreted ones did, with backends written in Python, and hold nothing that was let go.  No GPU needed."""
import gc
import weakref

import numpy as np
import pytest

from test_host_logic import FakeBackend


@pytest.fixture
def fake():
    import tfhip
    from tfhip.engine import ENGINE
    be = FakeBackend()
    tfhip.register_backend("fake-native", lambda: be, 0)
    prev = ENGINE.backend_name
    tfhip.set_backend("fake-native")
    yield be
    tfhip.remove_backend("fake-native")
    if prev:
        ENGINE.set_backend(prev)


def counts():
    import tfhip
    m = tfhip.memory()
    return m["numTensors"], m["numDataBuffers"], m["numBytes"]


@pytest.mark.parametrize("kept", [0, 1, 3, 40])
def test_scopes_keep_what_is_returned(fake, kept):
    import tfhip as tf
    base = counts()

    def body():
        made = [tf.tensor(np.zeros(i + 1, np.float32)) for i in range(50)]
        inner = tf.tidy(lambda: {"a": made[:kept], "b": (tf.tensor(1.5),)})
        return [inner, made[:kept]]
    got = tf.tidy(body)
    assert counts() == (base[0] + kept + 1, base[1] + kept + 1, base[2] + 4 * (sum(range(1, kept + 1)) + 1))
    assert len(fake.live) == kept + 1
    tf.dispose(got[1] + list(got[0]["b"]))
    tf.dispose(got[1])                      # a second time is no error
    assert counts() == base and not fake.live


def test_errors_end_their_scopes(fake):
    import tfhip as tf
    from tfhip.engine import ENGINE
    base = counts()

    def body():
        tf.tensor(np.ones(3, np.float32))
        ENGINE.run_kernel(lambda be: tf.tensor(2.0) and be.nothing)
    with pytest.raises(AttributeError, match="nothing"):
        tf.tidy(body)
    with pytest.raises(ZeroDivisionError):
        with tf.tidy():
            tf.tensor(np.ones(3, np.float32))
            1 / 0
    assert counts() == base and ENGINE.scopes == [] and not fake.live
    with pytest.raises(IndexError):
        ENGINE.end_scope()
    fake.register = lambda *a: 1 / 0
    with pytest.raises(ZeroDivisionError):
        tf.tidy(lambda: tf.tensor(1.0))
    del fake.register
    assert ENGINE.scopes == []


def test_records(fake):
    from tfhip.engine import DataId, Tensor
    t = Tensor([2.0, np.int64(3)], None, None, None, fake)
    assert t.shape == (2, 3) and t.size == 6 and t.rank == 2 and t.dtype == "float32" and t.quant is None
    assert type(t.shape[0]) is int and isinstance(t.data_id, DataId) and not t.is_disposed
    other = Tensor((6,), "int32", t.data_id, backend=fake)
    assert other.data_id is t.data_id and other.id == t.id + 1 and len(fake.live) == 1
    t.note = "tensors take attributes"
    t.dispose()
    assert t.is_disposed and len(fake.live) == 1
    other.dispose()
    assert not fake.live
    big = Tensor((2 ** 40, 2 ** 30, 0), "bool", backend=fake)
    assert big.size == 0
    big.dispose()
    q = Tensor((4,), "float32", None, np.zeros(4, np.uint8), fake, (0.5, 1.0))
    q.dispose()
    with pytest.raises((TypeError, ValueError)):
        Tensor(("a",), "float32", backend=fake)
    with pytest.raises((AttributeError, RuntimeError)):
        Tensor.__new__(Tensor).dispose()


FIELDS = ["shape", "dtype", "size", "rank", "data_id", "quant", "is_disposed", "id"]


@pytest.mark.parametrize("field", FIELDS + ["all"])
def test_half_made_records_raise(fake, field):
    """A record without a field (made by __new__ alone, or the field deleted) is an AttributeError."""
    import tfhip as tf
    from tfhip import _capi, _native
    from tfhip.engine import ENGINE, Tensor
    _capi.lib()
    core = _native.BackendCore.__new__(_native.BackendCore)     # (no context: what reaches the library fails)
    base = counts()
    ENGINE.start_scope()
    t = tf.tensor(np.zeros((2, 3), np.float32)) if field != "all" else Tensor.__new__(Tensor)
    kept = {f: getattr(t, f, None) for f in FIELDS}
    if field == "all":
        ENGINE.scopes[-1].append(t)
    else:
        delattr(t, field)
    needed = lambda *fields: field == "all" or field in fields
    calls = [(lambda: ENGINE.dispose_tensor(t), needed("data_id")),
             (lambda: ENGINE.end_scope(), needed("is_disposed", "data_id")),
             (lambda: t.dispose(), needed("is_disposed", "data_id")),
             (lambda: core._alias(t, (6,)), needed("data_id", "dtype", "quant")),
             (lambda: core._unary_out(0, t, "float32", 0.0, 0.0), needed("shape")),
             (lambda: core._binary_out(0, t, t, "float32"), needed("shape")),
             (lambda: core._softmax_out(t, 2, 3), needed("shape")),
             (lambda: core._matmul_out(t, t, (1, 2, 2), 1, 2, 2, 3, 0, 1, None, 0, 0, None, 0), needed("quant"))]
    for call, missing in calls:
        if missing:
            with pytest.raises(AttributeError):
                call()
    if field == "all":
        while ENGINE.scopes:
            ENGINE.scopes.pop()
        return
    for f in FIELDS:
        setattr(t, f, kept[f])
    if not t.is_disposed:
        t.dispose()
    while ENGINE.scopes:
        ENGINE.end_scope()
    assert counts() == base and not fake.live


def test_an_engine_without_its_backend_field_raises(fake):
    import tfhip as tf
    from tfhip.engine import ENGINE, Tensor
    backend = ENGINE._backend
    del ENGINE._backend
    try:
        for call in (lambda: ENGINE.run_kernel(lambda be: be), lambda: ENGINE.tidy(lambda: tf.tensor(1.0)),
                     lambda: Tensor((1,), "float32", None, np.zeros(1, np.float32))):
            with pytest.raises(AttributeError):
                call()
    finally:
        ENGINE._backend = backend
    assert ENGINE.scopes == []


def test_arguments_by_name(fake):
    """The engine's and the backend's methods take their arguments by name, as Python functions do."""
    import tfhip as tf
    from tfhip import _capi, _native
    from tfhip.engine import ENGINE, DataId, Tensor
    _capi.lib()
    base = counts()
    ENGINE.start_scope()
    a, b = tf.tensor(1.0), tf.tensor(2.0)
    ENGINE.end_scope(result=a)
    assert b.is_disposed and not a.is_disposed
    assert ENGINE.run_kernel(forward=lambda be: be) is fake
    t = Tensor.__new__(Tensor)                                   # a record that the program registers itself
    t.shape, t.size, t.dtype, t.rank, t.data_id, t.is_disposed = (3,), 3, "int32", 1, DataId(), False
    ENGINE.register_tensor(t=t, backend=None, storage_dtype="int32")
    assert t.data_id in fake.live and counts() == (base[0] + 2, base[1] + 2, base[2] + 16)
    ENGINE.dispose_tensor(t=t)
    ENGINE.dispose_tensor(t=a)
    assert counts() == base and not fake.live
    core = _native.BackendCore.__new__(_native.BackendCore)
    core.dispose_data(data_id=DataId())
    with pytest.raises(KeyError):
        core.register(shape=[2, 3], dtype="float64", data_id=DataId())
    for call in (lambda: ENGINE.run_kernel(), lambda: ENGINE.run_kernel(lambda be: be, forward=None),
                 lambda: ENGINE.end_scope(a, a), lambda: ENGINE.dispose_tensor(tensor=a),
                 lambda: core.register(DataId(), (1,))):
        with pytest.raises(TypeError):
            call()
    assert ENGINE.scopes == []


@pytest.mark.parametrize("derived", [True, False])
def test_replaced_product_methods_are_called(fake, derived):
    """matMul goes through batch_mat_mul, fused_batch_mat_mul and reshape of a backend that replaces them, be it in
    a class of its own or in the instance."""
    import tfhip as tf
    from tfhip.backend_hip import MathBackendHIP
    from tfhip.engine import ENGINE
    calls = []

    def reshape(x, shape):
        calls.append(tuple(shape))
        return x

    def batch_mat_mul(a, b, transpose_a, transpose_b):
        calls.append((transpose_a, transpose_b))
        return a

    def fused_batch_mat_mul(a, b, transpose_a, transpose_b, bias, activation, weights):
        calls.append((transpose_a, transpose_b, bias, activation))
        return b
    methods = dict(reshape=reshape, batch_mat_mul=batch_mat_mul, fused_batch_mat_mul=fused_batch_mat_mul)
    if derived:
        as_methods = {k: (lambda f: lambda self, *a: f(*a))(f) for k, f in methods.items()}
        be = type("Derived", (MathBackendHIP,), dict(as_methods, __init__=lambda self: None))()
    else:
        be = MathBackendHIP.__new__(MathBackendHIP)
        for name, method in methods.items():
            setattr(be, name, method)
    assert type("Plain", (MathBackendHIP,), {})._own_product and MathBackendHIP._own_product
    a, b = tf.tensor(np.zeros((2, 3), np.float32)), tf.tensor(np.zeros((3, 4), np.float32))
    backend, ENGINE._backend = ENGINE._backend, be
    try:
        assert tf.matmul(a, b) is a
        assert calls == [(1, 2, 3), (1, 3, 4), (False, False), (2, 4)]
        del calls[:]
        assert tf.fused.matmul(a, b, activation="relu") is b
        assert calls == [(1, 2, 3), (1, 3, 4), (False, False, None, "relu"), (2, 4)]
    finally:
        ENGINE._backend = backend
    tf.dispose([a, b])


def test_copies_of_records(fake):
    import copy
    import tfhip as tf
    base = counts()
    t = tf.tensor(np.zeros((2, 3), np.float32))
    t.note = "kept"
    c = copy.copy(t)
    assert [getattr(c, f) for f in FIELDS] == [getattr(t, f) for f in FIELDS] and c.note == "kept" and c is not t
    assert type(c) is type(t) and counts() == (base[0] + 1, base[1] + 1, base[2] + 24)
    t.dispose()
    assert counts() == base and not c.is_disposed


def test_nothing_is_held(fake):
    import tfhip as tf
    value = np.zeros(7, np.float32)
    t = tf.tensor(value)
    r = tf.reshape(t, (7, 1))
    refs = [weakref.ref(t), weakref.ref(r), weakref.ref(t.data_id)]
    tf.dispose([t, r])
    del t, r
    gc.collect()
    assert [x() for x in refs] == [None] * 3

    def step():
        tf.tidy(lambda: [tf.reshape(tf.tensor(value), (1, 7)) for _ in range(4)][-1]).dispose()
    for _ in range(10):
        step()
    gc.collect()
    before = len(gc.get_objects())
    for _ in range(200):
        step()
    gc.collect()
    assert len(gc.get_objects()) <= before + 20


def test_geometry_is_remembered_by_value_only():
    from tfhip import shape_util as su
    a = su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), 2, 1, "same")
    want = dict(a, padInfo=dict(a["padInfo"]))
    a["padInfo"]["top"] = a["inHeight"] = 77
    assert su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), 2, 1, "same") == want
    for strides in (2.0, (2.0, 2), [2, 2]):        # equal numbers of other types are computed anew
        b = su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), strides, 1, "same")
        assert b == want and type(b["strideHeight"]) is type(strides if type(strides) is float else strides[0])
    c = su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), 2, 1, 0)
    assert type(su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), 2, 1, 0.0)["padInfo"]["top"]) is float
    assert type(c["padInfo"]["top"]) is int
    for _ in range(2):
        with pytest.raises(ValueError):
            su.compute_conv2d_info((1, 9, 9, 4), (3, 3, 4, 8), 2, 1, "other")


def test_the_entry_points_need_the_library():
    from tfhip import _native
    with pytest.raises(RuntimeError):
        _native.load("/nonexistent.so")
    with pytest.raises((TypeError, ValueError)):
        _native.set_backend_class(dict)
