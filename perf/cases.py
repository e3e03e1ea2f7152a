"""The work that programs on the `hip` backend do, as cases that can be timed and compared.

`listed()` names them, `draw()` gives further ones of the same ranges, `prepare()` makes what a
program holds before the call (tensors on the device, or the host image of a single-picture
classifier), `run()` is one pass through the public tf.* entry points.  Everything is float32 as
the backend computes it; weights are He-normal, activations what such layers produce.

Results stay on the device: the backend's own buffers are handed out as torch tensors that share
their memory (`tfhip_device_ptr`) and give them back to the backend when they are dropped.  Only
the single-picture classifier reads its probabilities to the host, as such a program does.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tfjs-core_amd", "python"))

import tfhip as tf  # noqa: E402
from tfhip import mobilenet  # noqa: E402

_TYPESTR = {"float32": "<f4", "int32": "<i4"}


def listed():
    return [
        # one small product, launched on its own: the call's latency
        dict(name="matmul_256x512x256", kind="matmul", batch=1, m=256, k=512, n=256, ta=False,
             tb=False),
        # scores of many short sequences against each other: sizes that no tile divides
        dict(name="matmul_batched_ragged", kind="matmul", batch=96, m=201, k=67, n=201, ta=False,
             tb=True),
        # a multi-layer perceptron: a large batch classified, and a training step (SGD) on an
        # ordinary batch
        dict(name="mlp_infer_b4096", kind="mlp", batch=4096, d0=784, d1=1024, d2=1024, d3=10,
             train=False),
        dict(name="mlp_train_b1000", kind="mlp", batch=1000, d0=784, d1=512, d2=256, d3=10,
             train=True),
        # MobileNetV1-1.0: one picture from host memory to its probabilities in host memory (a
        # page or camera application), a batch of 64 (the benchmark), 256 with uint8 weights
        dict(name="mobilenet_b1_host", kind="mobilenet", batch=1, size=224, uint8=False, host=True),
        dict(name="mobilenet_b64", kind="mobilenet", batch=64, size=224, uint8=False, host=False),
        dict(name="mobilenet_b256_uint8", kind="mobilenet", batch=256, size=224, uint8=True,
             host=False),
        # one dense convolution of an image network, forward
        dict(name="conv3x3_b32_112", kind="conv", batch=32, h=112, w=112, cin=64, cout=128, f=3,
             stride=1),
        # convolution + relu + max pool, forward and backward with every gradient
        dict(name="cnn_train_b32_56", kind="cnn_train", batch=32, h=56, w=56, cin=64, cout=128, f=3,
             stride=1, pool=2),
        # depthwise convolution + batch norm on batch statistics + relu, forward and backward
        dict(name="separable_train_b32_56", kind="separable_train", batch=32, h=56, w=56, c=128,
             stride=1),
        # camera frames: mirrored, resized, normalised per channel
        dict(name="preprocess_b16_480x640", kind="preprocess", batch=16, h=480, w=640, out=224),
        # bag of words: embeddings gathered and averaged, a softmax layer, and its training step
        dict(name="text_train_b256", kind="text_train", batch=256, length=40, vocab=20000, d=128,
             classes=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matmul", "matmul", "mlp", "mlp", "mobilenet", "conv", "cnn_train",
                       "separable_train", "preprocess", "text_train"))
    if kind == "matmul":
        while True:
            batch = rng.choice((1, 1, _log(rng, 2, 128)))
            # three of four products have sizes from the alignments that layers are given
            step = rng.choice((1, 4, 16, 64))
            m, k, n = (max(step, _log(rng, 16, 4096) // step * step) for _ in range(3))
            if batch * m * k * n < 2 ** 35 and batch * (m * k + k * n + m * n) < 2 ** 27:
                break
        return dict(kind=kind, batch=batch, m=m, k=k, n=n, ta=rng.random() < 0.3,
                    tb=rng.random() < 0.3)
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 8, 4096), d0=_log(rng, 64, 1024),
                    d1=rng.choice((128, 256, 300, 512, 1000, 1024)),
                    d2=rng.choice((64, 100, 256, 500, 512, 1024)), d3=rng.randint(2, 100),
                    train=rng.random() < 0.6)
    if kind == "mobilenet":
        batch = _log(rng, 1, 200)
        return dict(kind=kind, batch=batch, size=rng.choice((128, 160, 192, 224)),
                    uint8=rng.random() < 0.4, host=batch <= 4)
    if kind in ("conv", "cnn_train"):
        while True:
            case = dict(kind=kind, batch=_log(rng, 1, 64), h=_log(rng, 7, 128), w=_log(rng, 7, 128),
                        cin=rng.choice((3, 16, 24, 32, 48, 64, 96, 128, 256)),
                        cout=rng.choice((16, 24, 32, 64, 96, 128, 200, 256)),
                        f=rng.choice((1, 3, 3, 3, 5)), stride=rng.choice((1, 1, 2)))
            if kind == "cnn_train":
                case["pool"] = rng.choice((2, 3))
            macs = case["batch"] * case["h"] * case["w"] * case["cin"] * case["cout"] * case["f"] ** 2
            if macs * (3 if kind == "cnn_train" else 1) < 2 ** 34.5:
                return case
    if kind == "separable_train":
        while True:
            case = dict(kind=kind, batch=_log(rng, 1, 64), h=_log(rng, 7, 112), w=_log(rng, 7, 112),
                        c=rng.choice((16, 24, 32, 64, 96, 128, 200, 256, 512)),
                        stride=rng.choice((1, 2)))
            if case["batch"] * case["h"] * case["w"] * case["c"] <= 2 ** 23.7:
                return case
    if kind == "preprocess":
        return dict(kind=kind, batch=_log(rng, 1, 16), h=_log(rng, 120, 720), w=_log(rng, 160, 960),
                    out=rng.choice((128, 160, 192, 224, 299)))
    return dict(kind=kind, batch=_log(rng, 16, 300), length=_log(rng, 8, 40),
                vocab=_log(rng, 500, 20000), d=rng.choice((32, 50, 64, 100, 128)),
                classes=rng.randint(2, 30))


class _State(object):
    """What a program keeps between calls; its tensors go back to the backend with it."""

    def __init__(self, case):
        self.case = case

    def __del__(self):
        for v in self.__dict__.values():
            for t in (v.values() if isinstance(v, dict) else v if isinstance(v, list) else [v]):
                if isinstance(t, tf.Tensor):
                    t.dispose()


class _Shared(object):
    """The device buffer of a tensor, for torch; the tensor lives as long as this does."""

    def __init__(self, t):
        self._t = t
        be = tf.backend()
        ptr, nbytes = ctypes.c_void_p(), ctypes.c_size_t()
        be._ck(be.lib.tfhip_device_ptr(be.ctx, be._h(t), ctypes.byref(ptr), ctypes.byref(nbytes)))
        self.__cuda_array_interface__ = dict(shape=t.shape, typestr=_TYPESTR[t.dtype], strides=None,
                                             data=(ptr.value, False), version=2)

    def __del__(self):
        self._t.dispose()


def _out(*tensors):
    return [torch.as_tensor(_Shared(t), device="cuda") for t in tensors]


class _Inputs(object):
    """Random tensors made from the seed on the device, as tensors of the backend."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def host_uniform(self, shape, lo, hi):
        x = torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo
        return x.cpu().numpy()

    def host_normal(self, shape, sigma=1.0):
        return (torch.randn(shape, generator=self.gen, device="cuda") * sigma).cpu().numpy()

    def uniform(self, shape, lo, hi):
        return tf.tensor(self.host_uniform(shape, lo, hi))

    def normal(self, shape, sigma=1.0):
        return tf.tensor(self.host_normal(shape, sigma))

    def activations(self, shape):
        """What a relu layer hands on: half of the values are zero."""
        x = torch.randn(shape, generator=self.gen, device="cuda").clamp_min_(0)
        return tf.tensor(x.cpu().numpy())

    def integers(self, shape, n):
        x = torch.randint(0, n, shape, generator=self.gen, device="cuda", dtype=torch.int32)
        return tf.tensor(x.cpu().numpy())

    def word_ids(self, shape, n):
        """Word numbers as texts use them: frequency falls with the rank (log-uniform)."""
        u = torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float64)
        x = (torch.exp(u * math.log(n + 1)) - 1).to(torch.int32).clamp_(0, n - 1)
        return tf.tensor(x.cpu().numpy())


def _out_extent(case):
    """Output height and width of a 'same' convolution."""
    return -(-case["h"] // case["stride"]), -(-case["w"] // case["stride"])


def prepare(case, seed):
    if tf.get_backend() is None:
        tf.set_backend("hip")
    s, r, kind = _State(case), _Inputs(seed), case["kind"]
    if kind == "matmul":
        a, b = (case["m"], case["k"]), (case["k"], case["n"])
        a, b = a[::-1] if case["ta"] else a, b[::-1] if case["tb"] else b
        lead = (case["batch"],) if case["batch"] > 1 else ()
        s.a, s.b = r.uniform(lead + a, -1, 1), r.uniform(lead + b, -1, 1)
    elif kind == "mlp":
        d = [case["d%d" % i] for i in range(4)]
        s.x = r.uniform((case["batch"], d[0]), 0, 1)
        s.w = [r.normal((d[i], d[i + 1]), math.sqrt(2.0 / d[i])) for i in range(3)]
        s.b = [r.normal((d[i + 1],), 0.01) for i in range(3)]
        if case["train"]:
            s.labels = r.integers((case["batch"],), d[3])
            s.rate = tf.tensor(0.05)
    elif kind == "mobilenet":
        params = mobilenet.make_params(seed & 0x7fffffff)
        if case["uint8"]:
            params = mobilenet.quantize_params(params)
        s.w = mobilenet.upload(tf, params)
        shape = (case["batch"], case["size"], case["size"], 3)
        if case["host"]:
            s.image = r.host_uniform(shape, 0, 1)
        else:
            s.x = r.uniform(shape, 0, 1)
    elif kind in ("conv", "cnn_train"):
        f, cin, cout = case["f"], case["cin"], case["cout"]
        s.x = r.activations((case["batch"], case["h"], case["w"], cin))
        s.w = r.normal((f, f, cin, cout), math.sqrt(2.0 / (f * f * cin)))
        s.b = r.normal((cout,), 0.1)
        if kind == "cnn_train":
            oh, ow = _out_extent(case)
            s.dy = r.normal((case["batch"], -(-oh // 2), -(-ow // 2), cout))
    elif kind == "separable_train":
        c = case["c"]
        oh, ow = _out_extent(case)
        s.x = r.activations((case["batch"], case["h"], case["w"], c))
        s.w = r.normal((3, 3, c, 1), math.sqrt(2.0 / 9))
        s.gamma, s.beta = r.uniform((c,), 0.5, 1.5), r.normal((c,), 0.1)
        s.dy = r.normal((case["batch"], oh, ow, c))
    elif kind == "preprocess":
        x = r.host_uniform((case["batch"], case["h"], case["w"], 3), 0, 256)
        s.x = tf.tensor(x // 1)
        s.mean = tf.tensor(r.host_uniform((3,), 100, 130))
        s.std = tf.tensor(r.host_uniform((3,), 50, 70))
    else:
        s.ids = r.word_ids((case["batch"], case["length"]), case["vocab"])
        s.table = r.normal((case["vocab"], case["d"]), 0.5)
        s.w = r.normal((case["d"], case["classes"]), math.sqrt(1.0 / case["d"]))
        s.b = r.normal((case["classes"],), 0.01)
        s.labels = r.integers((case["batch"],), case["classes"])
        s.rate = tf.tensor(0.05)
    return s


def _logits_gradient(logits, labels, classes, batch):
    """Mean softmax cross-entropy: the gradient at the logits, and the probabilities."""
    probs = tf.softmax(logits)
    hot = tf.cast(tf.one_hot(labels, classes), "float32")
    return tf.div(tf.sub(probs, hot), float(batch)), probs


def _mlp(s):
    c = s.case
    h1 = tf.fused.matmul(s.x, s.w[0], bias=s.b[0], activation="relu")
    h2 = tf.fused.matmul(h1, s.w[1], bias=s.b[1], activation="relu")
    logits = tf.fused.matmul(h2, s.w[2], bias=s.b[2])
    if not c["train"]:
        return [logits, tf.softmax(logits), tf.arg_max(logits, 1)]
    g, _ = _logits_gradient(logits, s.labels, c["d3"], c["batch"])
    results = [logits]
    for i, h in ((2, h2), (1, h1), (0, s.x)):
        dw, db = tf.matmul(h, g, True, False), tf.sum(g, 0)
        if i:
            g = tf.mul(tf.matmul(g, s.w[i], False, True), tf.step(h))
        results += [dw, db, tf.sub(s.w[i], tf.mul(dw, s.rate)), tf.sub(s.b[i], tf.mul(db, s.rate))]
    return results


def _cnn_train(s):
    c = s.case
    y = tf.fused.conv2d(s.x, s.w, c["stride"], "same", bias=s.b, activation="relu")
    p = tf.max_pool(y, c["pool"], 2, "same")
    g = tf.max_pool_backprop(s.dy, y, c["pool"], 2, "same")
    g = tf.mul(g, tf.step(y))
    dx = tf.conv2d_der_input(s.x.shape, g, s.w, c["stride"], "same")
    dw = tf.conv2d_der_filter(s.x, g, s.w.shape, c["stride"], "same")
    return [y, p, dx, dw, tf.sum(g, [0, 1, 2])]


def _separable_train(s):
    c = s.case
    axes = [0, 1, 2]
    y = tf.depthwise_conv2d(s.x, s.w, c["stride"], "same")
    n = float(y.size // c["c"])
    mean = tf.mean(y, axes)
    centred = tf.sub(y, mean)
    variance = tf.mean(tf.square(centred), axes)
    z = tf.relu(tf.batch_norm(y, mean, variance, s.beta, s.gamma, 0.001))
    # backward
    g = tf.mul(s.dy, tf.step(z))
    inv = tf.rsqrt(tf.add(variance, 0.001))
    xhat = tf.mul(centred, inv)
    dbeta, dgamma = tf.sum(g, axes), tf.sum(tf.mul(g, xhat), axes)
    inner = tf.sub(tf.sub(g, tf.div(dbeta, n)), tf.mul(xhat, tf.div(dgamma, n)))
    g = tf.mul(inner, tf.mul(s.gamma, inv))
    dx = tf.depthwise_conv2d_der_input(s.x.shape, g, s.w, c["stride"], "same")
    dw = tf.depthwise_conv2d_der_filter(s.x, g, s.w.shape, c["stride"], "same")
    return [z, mean, variance, dx, dw, dgamma, dbeta]


def _preprocess(s):
    x = tf.resize_bilinear(tf.reverse(s.x, [2]), (s.case["out"], s.case["out"]))
    return [tf.div(tf.sub(x, s.mean), s.std)]


def _text_train(s):
    c = s.case
    words = tf.gather(s.table, s.ids)
    bag = tf.mean(words, 1)
    logits = tf.fused.matmul(bag, s.w, bias=s.b)
    g, _ = _logits_gradient(logits, s.labels, c["classes"], c["batch"])
    dw, db = tf.matmul(bag, g, True, False), tf.sum(g, 0)
    dbag = tf.div(tf.matmul(g, s.w, False, True), float(c["length"]))
    dwords = tf.tile(tf.reshape(dbag, (c["batch"], 1, c["d"])), [1, c["length"], 1])
    n = c["batch"] * c["length"]
    dtable = tf.unsorted_segment_sum(tf.reshape(dwords, (n, c["d"])), tf.reshape(s.ids, (n,)),
                                     c["vocab"])
    return [logits, dw, db, tf.sub(s.table, tf.mul(dtable, s.rate)),
            tf.sub(s.w, tf.mul(dw, s.rate)), tf.sub(s.b, tf.mul(db, s.rate))]


def run(s):
    c, kind = s.case, s.case["kind"]
    if kind == "matmul":
        return _out(tf.matmul(s.a, s.b, c["ta"], c["tb"]))
    if kind == "mobilenet":
        if not c["host"]:
            return _out(*mobilenet.forward(tf, s.w, s.x))
        x = tf.tensor(s.image)
        logits, probs = mobilenet.forward(tf, s.w, x)
        values = probs.data_sync()
        tf.dispose([x, probs])
        return _out(logits) + [values]
    if kind == "conv":
        return _out(tf.fused.conv2d(s.x, s.w, c["stride"], "same", bias=s.b, activation="relu6"))
    step = {"mlp": _mlp, "cnn_train": _cnn_train, "separable_train": _separable_train,
            "preprocess": _preprocess, "text_train": _text_train}[kind]
    return _out(*tf.tidy(lambda: step(s)))


def work(case):
    """Operands and results of a pass once, and the multiply-adds of its products (two
    operations each); elementwise arithmetic is not counted."""
    c, kind = case, case["kind"]
    if kind == "matmul":
        m, k, n, b = c["m"], c["k"], c["n"], c["batch"]
        return dict(bytes=4.0 * b * (m * k + k * n + m * n), flops=2.0 * b * m * k * n)
    if kind == "mlp":
        b, d = c["batch"], [c["d%d" % i] for i in range(4)]
        weights = sum(d[i] * d[i + 1] + d[i + 1] for i in range(3))
        macs = b * sum(d[i] * d[i + 1] for i in range(3))
        if not c["train"]:
            return dict(bytes=4.0 * (b * d[0] + weights + 2 * b * d[3] + b), flops=2.0 * macs)
        macs += macs + b * (d[1] * d[2] + d[2] * d[3])
        return dict(bytes=4.0 * (b * d[0] + 3 * weights + b * d[3] + b), flops=2.0 * macs)
    if kind == "mobilenet":
        rows = mobilenet.layer_table(c["batch"], c["size"])
        b, size = c["batch"], c["size"]
        weights = 4231976 if c["uint8"] else 4 * 4231976
        return dict(bytes=float(4 * b * (size * size * 3 + 2 * mobilenet.NUM_CLASSES) + weights),
                    flops=2.0 * sum(r["macs"] for r in rows))
    if kind in ("conv", "cnn_train"):
        oh, ow = _out_extent(c)
        x, y = c["batch"] * c["h"] * c["w"] * c["cin"], c["batch"] * oh * ow * c["cout"]
        w = c["f"] ** 2 * c["cin"] * c["cout"]
        macs = c["batch"] * oh * ow * w
        if kind == "conv":
            return dict(bytes=4.0 * (x + y + w + c["cout"]), flops=2.0 * macs)
        p = c["batch"] * -(-oh // 2) * -(-ow // 2) * c["cout"]
        return dict(bytes=4.0 * (2 * x + y + 2 * p + 2 * w + 2 * c["cout"]), flops=6.0 * macs)
    if kind == "separable_train":
        oh, ow = _out_extent(c)
        x, y = c["batch"] * c["h"] * c["w"] * c["c"], c["batch"] * oh * ow * c["c"]
        return dict(bytes=4.0 * (2 * x + 2 * y + 24 * c["c"]), flops=6.0 * 9 * y)
    if kind == "preprocess":
        x, y = c["batch"] * c["h"] * c["w"] * 3, c["batch"] * c["out"] ** 2 * 3
        return dict(bytes=4.0 * (min(x, 4 * y) + y), flops=8.0 * y)
    n, head = c["batch"] * c["length"], c["d"] * c["classes"]
    return dict(bytes=4.0 * (2 * c["vocab"] * c["d"] + 3 * head + n + c["batch"] * (1 + c["classes"])),
                flops=6.0 * c["batch"] * head + 2.0 * n * c["d"])


def tolerance(case):
    """About four times what the paths differ by from the same arithmetic in 64 bits: 1e-7 to 6e-7
    relative, 4e-6 of the root mean square at most (1.4e-6 and 5e-6 for the depthwise filter
    gradient), and no class number among 4096 differs.

    In the training steps a pre-activation within rounding of zero can land on either side of the
    relu, and two values of a pooling window within rounding of each other can change places: the
    whole gradient of that one element then appears or moves.  Seen: none in the perceptrons and
    the depthwise block, 7e-5 relative and 0.018 of the root mean square behind relu and max pool,
    where a gradient of the input collects hundreds of such elements; behind a depthwise filter it
    collects nine."""
    if case["kind"] == "mlp":
        if case["train"]:
            return {"rel": 3e-4, "max": 0.05}
        return {"rel": 3e-6, "max": 3e-5, "differ": 1e-3}
    if case["kind"] == "cnn_train":
        return {"rel": 3e-4, "max": 0.08}
    if case["kind"] == "separable_train":
        return {"rel": 3e-4, "max": 0.5}
    return {"rel": 3e-6, "max": 3e-5}
