"""The work a user of this framework has it do, as cases that can be timed.

A pass is one inference the way a program drives the library through its Python face
(webdnn_amd.hostops over the C ABI of include/webdnn_hip.h): the model's weights are on the device, the
input comes from the host or already lies there, the operators run either node by node or as a recorded
run that is replayed (what the runner does from the third run on), and the outputs are read back to the
host, which is how every run of the descriptor runner ends.  Layers use the fused operators the runner's
graph passes produce (bias, residual and Relu inside Conv and MatMul, attention in one node, the query,
key and value projections as a group), and temporaries are given back where the runner gives them back.

Networks, sizes and value distributions are those of webdnn_amd.modelgen and the benchmark (seeded random
initialisation, zero biases where the benchmark has zero biases), or generic ones of the same operators.
Everything is fp32 with int32 indices, the two types the framework has.
"""
import math

import numpy as np
import torch

from webdnn_amd import capi
from webdnn_amd import hostops as H


def listed():
    return [
        # one small Gemm with bias and a transposed weight, host to host: the benchmark's first model;
        # launch, transfer and host time are all there is
        dict(name="gemm_256x1024x512", kind="gemm", m=256, n=1024, k=512, trans_b=True, recorded=False),
        # one request through a wide fully connected net: every weight is read for a single row
        dict(name="mlp_one_row", kind="mlp", rows=1, width_in=2048, hidden=4096, layers=3, classes=1000, recorded=True),
        # the same operators at the size the Gemm kernels are quoted on (4096 x 4096 x 4096)
        dict(name="mlp_4096", kind="mlp", rows=4096, width_in=4096, hidden=4096, layers=3, classes=100, recorded=True),
        # the headline benchmark: ResNet-50, a batch of 32 resident on the device, replayed
        dict(name="resnet50_b32", kind="residual", batch=32, h=224, w=224, recorded=True, host_input=False),
        # a single picture from the host: what an interactive program asks for
        dict(name="resnet50_b1", kind="residual", batch=1, h=224, w=224, recorded=True, host_input=True),
        # pictures of an odd size, node by node: a program whose input shapes change from run to run
        dict(name="resnet50_b5_odd", kind="residual", batch=5, h=187, w=251, recorded=False, host_input=True),
        # throughput serving: the batch that fills the chip
        dict(name="resnet50_b128", kind="residual", batch=128, h=224, w=224, recorded=True, host_input=False),
        # the detector of the benchmark: one 800 x 1088 picture, 850 tokens, 6 + 6 transformer layers
        dict(name="detr_800x1088", kind="detector", h=800, w=1088, enc=6, dec=6, queries=100, recorded=True),
        # the benchmark's feed-forward block: [8, 512, 768] -> 3072 -> 768 with the residual added
        dict(name="ffn_8x512x768", kind="ffn", batch=8, seq=512, d=768, hidden=3072, recorded=False),
        # a text encoder over one sequence: embedding rows gathered by int32 ids, heads of 64
        dict(name="encoder_384", kind="encoder", tokens=384, d=768, heads=12, hidden=3072, layers=6, vocab=30000,
             recorded=True),
        # depthwise + pointwise convolutions, the usual net for small devices
        dict(name="separable_b8", kind="separable", batch=8, h=224, w=224, width=32, recorded=True),
        # what lies between the big products when an exporter writes everything out: concat, crop, broadcast
        # arithmetic, a decomposed layer normalisation, softmax, transposes and reductions
        dict(name="maps_b8", kind="maps", batch=8, ca=128, cb=64, h=97, w=129, recorded=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "mlp", "residual", "residual", "detector", "ffn", "encoder", "separable", "maps"])
    recorded = rng.random() < 0.6
    if kind == "gemm":
        return dict(kind=kind, m=_log_int(rng, 32, 2048), n=_log_int(rng, 32, 2048), k=_log_int(rng, 32, 4096),
                    trans_b=rng.random() < 0.5, recorded=recorded)
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), width_in=_log_int(rng, 256, 4096), hidden=_log_int(rng, 256, 4096),
                    layers=rng.randint(2, 3), classes=_log_int(rng, 10, 1000), recorded=recorded)
    if kind == "residual":
        h, w = _log_int(rng, 96, 320), _log_int(rng, 96, 320)
        most = 128 * 224 * 224 // (h * w)
        return dict(kind=kind, batch=_log_int(rng, 1, max(1, min(64, most))), h=h, w=w, recorded=recorded,
                    host_input=rng.random() < 0.5)
    if kind == "detector":
        return dict(kind=kind, h=rng.randint(300, 800), w=rng.randint(300, 1088), enc=rng.randint(2, 6), dec=rng.randint(2, 6),
                    queries=rng.choice([50, 100, 100, 300]), recorded=recorded)
    if kind == "ffn":
        d = 64 * rng.randint(4, 16)
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log_int(rng, 50, 512), d=d, hidden=4 * d, recorded=recorded)
    if kind == "encoder":
        heads, hd = rng.choice([(8, 32), (8, 64), (12, 64), (16, 64)])
        return dict(kind=kind, tokens=_log_int(rng, 16, 1024), d=heads * hd, heads=heads, hidden=4 * heads * hd,
                    layers=rng.randint(2, 6), vocab=rng.randint(5000, 30000), recorded=recorded)
    if kind == "separable":
        return dict(kind=kind, batch=_log_int(rng, 1, 16), h=_log_int(rng, 96, 320), w=_log_int(rng, 96, 320),
                    width=rng.choice([16, 24, 32]), recorded=recorded)
    return dict(kind="maps", batch=_log_int(rng, 1, 12), ca=rng.randint(24, 160), cb=rng.randint(24, 96),
                h=_log_int(rng, 24, 128), w=_log_int(rng, 24, 128), recorded=recorded)


# ---- state ------------------------------------------------------------------------------
class Model:
    """What a program keeps between runs: weights and input buffers on the device, the recorded run."""

    def __init__(self, seed):
        self.ctx = H.HipContext(0).initialize()
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.held = []       # device tensors this program owns
        self.inputs = []     # (device buffer, host array to upload before each run, or None)
        self.outputs = None  # of a recorded run
        self.graph = None

    # values: made on the device, kept by the library from then on
    def _keep(self, values):
        t = self.ctx.move_tensor(values.cpu().numpy())
        self.held.append(t)
        return t

    def normal(self, shape, std=1.0):
        return self._keep(torch.randn(shape, generator=self.gen, device="cuda") * std)

    def uniform(self, shape, lo, hi):
        return self._keep(torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo)

    def xavier(self, shape):
        bound = math.sqrt(6.0 / (shape[0] + shape[1]))
        return self.uniform(shape, -bound, bound)

    def full(self, shape, value):
        return self._keep(torch.full(shape, value, dtype=torch.float32, device="cuda"))

    def ids(self, n, below):
        return self._keep(torch.randint(0, below, (n,), generator=self.gen, device="cuda", dtype=torch.int32))

    def feed(self, tensor, host):
        """`tensor` is the run's input; host: it is uploaded before every run."""
        self.inputs.append((tensor, tensor.get_data() if host else None))

    def __del__(self):
        try:
            if self.graph is not None:
                self.ctx.graph_destroy(self.graph)
            for t in self.held + (self.outputs or []):
                t.dispose()
        except Exception:  # (the interpreter may be on its way out)
            pass


def _conv(m, cin, cout, k, group=1):
    w = m.normal((cout, cin // group, k, k), math.sqrt(2.0 / (cin // group * k * k)))
    return dict(w=w, b=m.full((cout,), 0.0), k=k, group=group, cout=cout)


def _linear(m, din, dout):
    return dict(w=m.xavier((din, dout)), b=m.full((dout,), 0.0))


def _norm(m, d):
    return dict(g=m.full((d,), 1.0), b=m.full((d,), 0.0))


def _dispose(*tensors):
    for t in tensors:
        t.dispose()


def _apply_conv(ctx, x, c, stride=1, relu=True, residual=None):
    pad = c["k"] // 2
    return H.conv(ctx, x, c["w"], c["b"], None, c["group"], None, [pad] * 4, [stride, stride],
                  epilogue="relu" if relu else None, residual=residual, constant_weights=True)


def _apply_linear(ctx, x, l, relu=False, residual=None):
    return H.matmul(ctx, x, l["w"], l["b"], residual, "relu" if relu else None)


def _build_trunk(m, width=64, blocks=(3, 4, 6, 3)):
    stages, cin = [], width
    stem = _conv(m, 3, width, 7)
    for s, count in enumerate(blocks):
        mid, cout = width << s, 4 * width << s
        for b in range(count):
            block = dict(c1=_conv(m, cin, mid, 1), c2=_conv(m, mid, mid, 3), c3=_conv(m, mid, cout, 1),
                         stride=2 if s > 0 and b == 0 else 1)
            if b == 0:
                block["shortcut"] = _conv(m, cin, cout, 1)
            stages.append(block)
            cin = cout
    return dict(stem=stem, blocks=stages, channels=cin)


def _run_trunk(ctx, trunk, x):
    """ResNet-50 v1 up to the last stage; shortcuts are side branches of a recorded run, as the runner has them."""
    y = _apply_conv(ctx, x, trunk["stem"], 2)
    x = H.maxpool(ctx, y, [3, 3], pads=[1, 1, 1, 1], strides=[2, 2])
    y.dispose()
    for blk in trunk["blocks"]:
        side = x
        if "shortcut" in blk:
            capi.call("wdh_branch_begin")
            side = _apply_conv(ctx, x, blk["shortcut"], blk["stride"], relu=False)
            capi.call("wdh_branch_end")
        a = _apply_conv(ctx, x, blk["c1"], blk["stride"])
        b = _apply_conv(ctx, a, blk["c2"])
        a.dispose()
        if side is not x:
            capi.call("wdh_branch_join")
        y = _apply_conv(ctx, b, blk["c3"], residual=side)
        b.dispose()
        if side is not x:
            side.dispose()
        x.dispose()
        x = y
    return x


def _build_attention(m, d):
    return dict(q=_linear(m, d, d), k=_linear(m, d, d), v=_linear(m, d, d), o=_linear(m, d, d))


def _run_attention(ctx, p, q_in, k_in, v_in, heads, residual):
    d = q_in.dims[1]
    q, k, v = H.linear_group(ctx, [(q_in, p["q"]["w"], p["q"]["b"]), (k_in, p["k"]["w"], p["k"]["b"]),
                                   (v_in, p["v"]["w"], p["v"]["b"])])
    a = H.attention(ctx, q, k, v, heads, 1.0 / math.sqrt(d // heads))
    _dispose(q, k, v)
    y = _apply_linear(ctx, a, p["o"], residual=residual)
    a.dispose()
    return y


def _run_ffn(ctx, p, x):
    h = _apply_linear(ctx, x, p["f1"], relu=True)
    y = _apply_linear(ctx, h, p["f2"], residual=x)
    h.dispose()
    return y


def _layernorm(ctx, x, p):
    y = H.layer_normalization(ctx, x, p["g"], p["b"])
    x.dispose()
    return y


# ---- the nets: build(model, case) keeps weights and inputs and returns forward(ctx) -> outputs ------------
def _gemm(m, c):
    a = m.uniform((c["m"], c["k"]), -1, 1)
    b = m.uniform((c["n"], c["k"]) if c["trans_b"] else (c["k"], c["n"]), -1, 1)
    bias = m.uniform((c["n"],), -1, 1)
    m.feed(a, True)
    return lambda ctx: [H.gemm(ctx, a, b, bias, 1.0, 1.0, 0, 1 if c["trans_b"] else 0)]


def _mlp(m, c):
    widths = [c["width_in"]] + [c["hidden"]] * (c["layers"] - 1) + [c["classes"]]
    weights = [(m.normal((o, i), math.sqrt(2.0 / i)), m.uniform((o,), -0.1, 0.1)) for i, o in zip(widths, widths[1:])]
    x0 = m.normal((c["rows"], c["width_in"]))
    m.feed(x0, False)

    def forward(ctx):
        x = x0
        for i, (w, b) in enumerate(weights):
            y = H.gemm(ctx, x, w, b, 1.0, 1.0, 0, 1, epilogue="relu" if i + 1 < len(weights) else None)
            if x is not x0:
                x.dispose()
            x = y
        return [x]

    return forward


def _residual(m, c):
    trunk = _build_trunk(m)
    w, b = m.normal((1000, trunk["channels"]), 0.01), m.full((1000,), 0.0)
    x0 = m.normal((c["batch"], 3, c["h"], c["w"]))
    m.feed(x0, c["host_input"])

    def forward(ctx):
        x = _run_trunk(ctx, trunk, x0)
        p = H.global_average_pool(ctx, x)
        x.dispose()
        f = H.flatten(ctx, p)
        y = H.gemm(ctx, f, w, b, 1.0, 1.0, 0, 1)
        _dispose(f, p)
        return [y]

    return forward


def _detector(m, c):
    d, heads, classes = 256, 8, 92
    trunk = _build_trunk(m)
    proj = _conv(m, trunk["channels"], d, 1)
    half = lambda v: (v + 1) // 2
    th, tw = c["h"], c["w"]
    for _ in range(5):
        th, tw = half(th), half(tw)
    tokens = th * tw
    pos = m.uniform((tokens, d), -1, 1)
    query = m.normal((c["queries"], d))
    target = m.full((c["queries"], d), 0.0)
    layer = lambda: dict(sa=_build_attention(m, d), f1=_linear(m, d, 2048), f2=_linear(m, 2048, d), n1=_norm(m, d), n2=_norm(m, d))
    enc = [layer() for _ in range(c["enc"])]
    dec = [dict(layer(), ca=_build_attention(m, d), n3=_norm(m, d)) for _ in range(c["dec"])]
    last = _norm(m, d)
    cls, box = _linear(m, d, classes), [_linear(m, d, d), _linear(m, d, d), _linear(m, d, 4)]
    x0 = m.normal((1, 3, c["h"], c["w"]))
    m.feed(x0, True)

    def norm_add(ctx, x, p, addend):
        y, y2 = H.layer_normalization_add(ctx, x, p["g"], p["b"], addend)
        x.dispose()
        return y, y2

    def forward(ctx):
        x = _run_trunk(ctx, trunk, x0)
        p = _apply_conv(ctx, x, proj, relu=False)
        x.dispose()
        flat = H.reshape(ctx, p, [d, tokens])
        src = H.transpose(ctx, flat, [1, 0])
        _dispose(flat, p)
        qk = H.binary(ctx, "Add", src, pos)
        for e in enc:
            y = _run_attention(ctx, e["sa"], qk, qk, src, heads, src)
            _dispose(qk, src)
            src = _layernorm(ctx, y, e["n1"])
            y = _run_ffn(ctx, e, src)
            src.dispose()
            src, qk = norm_add(ctx, y, e["n2"], pos)
        tgt, tq = target.alias(target.dims), H.binary(ctx, "Add", target, query)
        for l in dec:
            y = _run_attention(ctx, l["sa"], tq, tq, tgt, heads, tgt)
            _dispose(tq, tgt)
            tgt, tq = norm_add(ctx, y, l["n1"], query)
            y = _run_attention(ctx, l["ca"], tq, qk, src, heads, tgt)
            _dispose(tq, tgt)
            tgt = _layernorm(ctx, y, l["n2"])
            y = _run_ffn(ctx, l, tgt)
            tgt.dispose()
            tgt, tq = norm_add(ctx, y, l["n3"], query)
        _dispose(tq, qk, src)
        hs = _layernorm(ctx, tgt, last)
        logits = H.gemm(ctx, hs, cls["w"], cls["b"])
        b1 = _apply_linear(ctx, hs, box[0], relu=True)
        b2 = _apply_linear(ctx, b1, box[1], relu=True)
        b3 = _apply_linear(ctx, b2, box[2])
        boxes = H.unary(ctx, "Sigmoid", b3)
        _dispose(hs, b1, b2, b3)
        return [logits, boxes]

    return forward


def _ffn(m, c):
    f1 = dict(w=m.normal((c["d"], c["hidden"]), 0.02), b=m.full((c["hidden"],), 0.0))
    f2 = m.normal((c["hidden"], c["d"]), 0.02)
    x0 = m.normal((c["batch"], c["seq"], c["d"]))
    m.feed(x0, True)

    def forward(ctx):
        h = _apply_linear(ctx, x0, f1, relu=True)
        y = H.matmul(ctx, h, f2, None, x0)
        h.dispose()
        return [y]

    return forward


def _encoder(m, c):
    d = c["d"]
    table, pos = m.normal((c["vocab"], d), 1.0), m.normal((c["tokens"], d), 0.1)
    layers = [dict(sa=_build_attention(m, d), f1=_linear(m, d, c["hidden"]), f2=_linear(m, c["hidden"], d), n1=_norm(m, d),
                   n2=_norm(m, d)) for _ in range(c["layers"])]
    first = _norm(m, d)
    ids = m.ids(c["tokens"], c["vocab"])
    m.feed(ids, True)

    def forward(ctx):
        e = H.gather(ctx, table, ids)
        s = H.binary(ctx, "Add", e, pos)
        e.dispose()
        x = _layernorm(ctx, s, first)
        for l in layers:
            y = _run_attention(ctx, l["sa"], x, x, x, c["heads"], x)
            x.dispose()
            x = _layernorm(ctx, y, l["n1"])
            y = _run_ffn(ctx, l, x)
            x.dispose()
            x = _layernorm(ctx, y, l["n2"])
        return [x]

    return forward


_SEPARABLE = [(2, 1), (4, 2), (4, 1), (8, 2), (8, 1), (16, 2), (16, 1), (16, 1), (16, 1), (16, 1), (16, 1), (32, 2), (32, 1)]


def _separable(m, c):
    width = c["width"]
    stem, blocks, cin = _conv(m, 3, width, 3), [], width
    for times, stride in _SEPARABLE:
        blocks.append((_conv(m, cin, cin, 3, group=cin), stride, _conv(m, cin, times * width, 1)))
        cin = times * width
    w, b = m.normal((1000, cin), 0.01), m.full((1000,), 0.0)
    x0 = m.normal((c["batch"], 3, c["h"], c["w"]))
    m.feed(x0, False)

    def forward(ctx):
        x = _apply_conv(ctx, x0, stem, 2)
        for depthwise, stride, pointwise in blocks:
            y = _apply_conv(ctx, x, depthwise, stride)
            x.dispose()
            x = _apply_conv(ctx, y, pointwise)
            y.dispose()
        p = H.global_average_pool(ctx, x)
        x.dispose()
        f = H.flatten(ctx, p)
        y = H.gemm(ctx, f, w, b, 1.0, 1.0, 0, 1)
        _dispose(f, p)
        return [y]

    return forward


def _maps(m, c):
    n, ch = c["batch"], c["ca"] + c["cb"]
    a, b = m.normal((n, c["ca"], c["h"], c["w"])), m.normal((n, c["cb"], c["h"], c["w"]))
    bias, scale = m.normal((ch, 1, 1)), m.uniform((ch, 1, 1), 0.5, 1.5)
    gamma, beta, eps, two = m.uniform((ch,), 0.5, 1.5), m.normal((ch,), 0.1), m.full((1,), 1e-5), m.full((1,), 2.0)
    pick = m.ids(ch // 2, ch)
    m.feed(a, False)
    m.feed(b, False)

    def forward(ctx):
        x = H.concat(ctx, [a, b], 1)
        y = H.slice_(ctx, x, [1, 1], [c["h"] - 1, c["w"] - 2], [2, 3])
        s = H.binary(ctx, "Mul", y, scale)
        z = H.binary(ctx, "Add", s, bias)
        gate = H.unary(ctx, "Sigmoid", z)
        r = H.unary(ctx, "Relu", z)
        g = H.binary(ctx, "Mul", r, gate)
        _dispose(x, y, s, z, gate, r)
        pooled = H.maxpool(ctx, g, [3, 3], pads=[1, 1, 1, 1], strides=[2, 2])
        gap = H.global_average_pool(ctx, pooled)
        t = H.transpose(ctx, g, [0, 2, 3, 1])
        _dispose(pooled, g)
        # layer normalisation over the channels as exporters before opset 17 write it
        mean = H.reduce_mean(ctx, t, [-1])
        cen = H.binary(ctx, "Sub", t, mean)
        sq = H.binary(ctx, "Pow", cen, two)
        var = H.reduce_mean(ctx, sq, [-1])
        ve = H.binary(ctx, "Add", var, eps)
        dev = H.unary(ctx, "Sqrt", ve)
        q = H.binary(ctx, "Div", cen, dev)
        qg = H.binary(ctx, "Mul", q, gamma)
        norm = H.binary(ctx, "Add", qg, beta)
        _dispose(t, mean, cen, sq, var, ve, dev, q, qg)
        prob = H.softmax(ctx, norm)
        avg = H.reduce_mean(ctx, prob, [1, 2], 0)
        back = H.transpose(ctx, norm, [0, 3, 1, 2])
        some = H.gather(ctx, back, pick, 1)
        left, right = H.split(ctx, some, 2, 3, [some.dims[3] // 2, some.dims[3] - some.dims[3] // 2])
        rows, columns = H.reduce_mean(ctx, left, [2, 3], 0), H.reduce_mean(ctx, right, [2, 3], 0)
        _dispose(norm, prob, back, some, left, right)
        return [gap, avg, rows, columns]

    return forward


_KINDS = dict(gemm=_gemm, mlp=_mlp, residual=_residual, detector=_detector, ffn=_ffn, encoder=_encoder, separable=_separable,
              maps=_maps)


# ---- what is timed ----------------------------------------------------------------------
def prepare(case, seed):
    m = Model(seed)
    m.forward = _KINDS[case["kind"]](m, case)
    if case["recorded"]:
        # the first run uploads, builds tables and fills the pool; the second is recorded
        for t in m.forward(m.ctx):
            t.dispose()
        m.ctx.graph_begin()
        m.outputs = m.forward(m.ctx)
        m.graph = m.ctx.graph_end()
    return m


def run(m):
    for tensor, host in m.inputs:
        if host is not None:
            tensor.set_data(host)
    if m.graph is not None:
        m.ctx.graph_launch(m.graph)
        return [t.get_data() for t in m.outputs]
    outputs = m.forward(m.ctx)
    values = [t.get_data() for t in outputs]
    for t in outputs:
        t.dispose()
    return values


# ---- what a pass cannot do without --------------------------------------------------------
def _trunk_work(batch, h, w, width=64, blocks=(3, 4, 6, 3)):
    half = lambda v: (v + 1) // 2
    h, w = half(h), half(w)
    flops, weights = 2 * batch * h * w * width * 147, width * 148
    h, w, cin = half(h), half(w), width
    for s, count in enumerate(blocks):
        mid, cout = width << s, 4 * width << s
        for b in range(count):
            if s > 0 and b == 0:
                h, w = half(h), half(w)
            per_pixel = cin * mid + 9 * mid * mid + mid * cout + (cin * cout if b == 0 else 0)
            flops += 2 * batch * h * w * per_pixel
            weights += per_pixel
            cin = cout
    return flops, weights, h * w, cin


def work(case):
    """Direct sums of every product, and inputs, weights and outputs once each (4 bytes an element)."""
    c, k = case, case["kind"]
    if k == "gemm":
        return {"bytes": 4 * (c["m"] * c["k"] + c["k"] * c["n"] + c["n"] + c["m"] * c["n"]), "flops": 2 * c["m"] * c["n"] * c["k"]}
    if k == "mlp":
        widths = [c["width_in"]] + [c["hidden"]] * (c["layers"] - 1) + [c["classes"]]
        products = sum(i * o for i, o in zip(widths, widths[1:]))
        return {"bytes": 4 * (products + sum(widths[1:]) + c["rows"] * (widths[0] + widths[-1])), "flops": 2 * c["rows"] * products}
    if k == "residual":
        flops, weights, _, ch = _trunk_work(c["batch"], c["h"], c["w"])
        return {"bytes": 4 * (weights + 1000 * ch + c["batch"] * (3 * c["h"] * c["w"] + 1000)),
                "flops": flops + 2 * c["batch"] * 1000 * ch}
    if k == "detector":
        flops, weights, t, ch = _trunk_work(1, c["h"], c["w"])
        d, f, q = 256, 2048, c["queries"]
        attend = lambda a, b: 2 * (2 * a * d * d + 2 * b * d * d) + 4 * a * b * d
        flops += 2 * t * ch * d + c["enc"] * (attend(t, t) + 4 * t * d * f)
        flops += c["dec"] * (attend(q, q) + attend(q, t) + 4 * q * d * f) + 2 * q * (d * 92 + 2 * d * d + 4 * d)
        weights += ch * d + c["enc"] * (4 * d * d + 2 * d * f) + c["dec"] * (8 * d * d + 2 * d * f) + d * 92 + 2 * d * d + 4 * d
        return {"bytes": 4 * (weights + t * d + 2 * q * d + 3 * c["h"] * c["w"] + 96 * q), "flops": flops}
    if k == "ffn":
        rows = c["batch"] * c["seq"]
        return {"bytes": 4 * (2 * c["d"] * c["hidden"] + 2 * rows * c["d"]), "flops": 4 * rows * c["d"] * c["hidden"]}
    if k == "encoder":
        t, d, f = c["tokens"], c["d"], c["hidden"]
        return {"bytes": 4 * (c["layers"] * (4 * d * d + 2 * d * f) + 3 * t * d),
                "flops": c["layers"] * (8 * t * d * d + 4 * t * t * d + 4 * t * d * f)}
    if k == "separable":
        half = lambda v: (v + 1) // 2
        h, w, cin = half(c["h"]), half(c["w"]), c["width"]
        flops, weights = 2 * h * w * cin * 27, cin * 27
        for times, stride in _SEPARABLE:
            if stride == 2:
                h, w = half(h), half(w)
            per_pixel = 9 * cin + cin * times * c["width"]
            flops, weights, cin = flops + 2 * h * w * per_pixel, weights + per_pixel, times * c["width"]
        return {"bytes": 4 * (weights + 1000 * cin + c["batch"] * (3 * c["h"] * c["w"] + 1000)),
                "flops": c["batch"] * (flops + 2000 * cin)}
    # maps: both inputs once; about thirty operations an element of the crop
    ch = c["ca"] + c["cb"]
    return {"bytes": 4 * c["batch"] * ch * c["h"] * c["w"], "flops": 30 * c["batch"] * ch * c["h"] * c["w"]}


def tolerance(case):
    """fp32 sums: about four times what each net's outputs were measured to differ by from the same net in 64 bits
    (2-norms: 0.13e-6 to 0.35e-6 for single products of K 512 to 4096, 0.22e-6 to 0.48e-6 for the nets, 0.05e-6
    for the element-wise chain)."""
    return {"rel": {"gemm": 1.5e-6, "mlp": 2e-6, "residual": 1.5e-6, "detector": 2e-6, "ffn": 1.5e-6, "encoder": 2e-6,
                    "separable": 1.5e-6, "maps": 4e-7}[case["kind"]]}
