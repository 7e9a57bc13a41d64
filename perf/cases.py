"""Performance cases: the work a user of this backend has it do, through HIPBackend and ResNet18Infer.

Each case names a kind (one of the functions below) and its sizes. Inputs and outputs are device tensors
whose addresses go to the backend, as a program that owns its buffers passes them; outputs are buffers
that the program allocated beforehand. exact() restates each kind in float64.
"""
import math
import types

import numpy as np
import torch

import omnimatchdeeplearningtool_amd as om

H = om.HIPBackend
EPS = 1e-5

# The dearest listed case (a 4096^3 product) bounds what draw() gives.
MAX_FLOPS = 137e9
MAX_BYTES = 1.2e9


# ---------------------------------------------------------------- inputs
class Source:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def randn(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def integers(self, n, *shape):
        return torch.randint(0, n, shape, generator=self.g, device="cuda")


def out(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def p(t):
    return None if t is None else t.data_ptr()


def half_type(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def out_size(h, k, stride, pad):
    return (h + 2 * pad - k) // stride + 1


# ---------------------------------------------------------------- fp32 GEMM
# The HAL's matmul and its transposed forms (Linear weights stored [out, in], gradients), one product or a batch.
def gemm_inputs(c, s):
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    lead = (b,) if b > 1 else ()
    A = s.randn(*lead, *((k, m) if c["layout"] == "tn" else (m, k)))
    B = s.randn(*lead, *((n, k) if c["layout"] == "nt" else (k, n)))
    return {"A": A, "B": B, "C": out(*lead, m, n)}


def gemm_run(c, st):
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    A, B, C = p(st["A"]), p(st["B"]), p(st["C"])
    if b > 1:
        (H.batchedMatmulTransB if c["layout"] == "nt" else H.batchedMatmul)(A, B, C, b, m, k, n)
    else:
        {"nn": H.matmul, "nt": H.matmulTransB, "tn": H.matmulTransA}[c["layout"]](A, B, C, m, k, n)
    return st["C"]


def gemm_exact(c, st):
    A, B = st["A"].double(), st["B"].double()
    if c["layout"] == "tn":
        A = A.transpose(-1, -2).contiguous()
    if c["layout"] == "nt":
        B = B.transpose(-1, -2).contiguous()
    return A @ B


def gemm_work(c):
    b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
    return 4.0 * b * (m * k + k * n + m * n), 2.0 * b * m * n * k


# ---------------------------------------------------------------- MLP training step
# Forward, softmax cross-entropy and backward of three Linear layers (ReLU between), every gradient; no optimizer.
# The ReLU gates of the backward are given (saved1, saved2), so that no rounding of the forward decides which way an
# activation near zero falls.
def mlp_dims(c):
    return [c["d0"], c["d1"], c["d2"], c["classes"]]


def mlp_inputs(c, s):
    b, d = c["batch"], mlp_dims(c)
    labels = s.integers(d[3], b)
    st = {"x": s.uniform(b, d[0]), "T": torch.nn.functional.one_hot(labels, d[3]).float().contiguous()}
    for j in range(3):
        lim = math.sqrt(6 / d[j])
        st["W%d" % j] = s.uniform(d[j], d[j + 1], lo=-lim, hi=lim)
        st["b%d" % j] = s.randn(d[j + 1], std=0.05)
        st["gW%d" % j], st["gb%d" % j] = out(d[j], d[j + 1]), out(d[j + 1])
        st["g%d" % j] = out(b, d[j + 1])
    st["saved1"], st["saved2"] = s.randn(b, d[1]).relu_(), s.randn(b, d[2]).relu_()
    st["a1"], st["a2"], st["z"], st["gx"], st["loss"] = out(b, d[1]), out(b, d[2]), out(b, d[3]), out(b, d[0]), out(1)
    return st


def mlp_run(c, st):
    b, d = c["batch"], mlp_dims(c)
    H.linearBiasAct(p(st["x"]), p(st["W0"]), p(st["b0"]), p(st["a1"]), b, d[0], d[1], 1)
    H.linearBiasAct(p(st["a1"]), p(st["W1"]), p(st["b1"]), p(st["a2"]), b, d[1], d[2], 1)
    H.linearSoftmaxCrossEntropyStep(p(st["a2"]), p(st["W2"]), p(st["b2"]), p(st["T"]), p(st["saved2"]), p(st["z"]),
                                    p(st["loss"]), p(st["g2"]), p(st["gW2"]), p(st["gb2"]), p(st["g1"]), b, d[2], d[3])
    H.linearBackward(p(st["a1"]), p(st["g1"]), p(st["W1"]), p(st["saved1"]), p(st["gW1"]), p(st["gb1"]), p(st["g0"]), b,
                     d[1], d[2])
    H.linearBackward(p(st["x"]), p(st["g0"]), p(st["W0"]), None, p(st["gW0"]), p(st["gb0"]), p(st["gx"]), b, d[0], d[1])
    return {k: st[k] for k in ("z", "loss", "gx", "gW0", "gb0", "gW1", "gb1", "gW2", "gb2")}


def mlp_exact(c, st):
    D = {k: v.double() for k, v in st.items()}
    a1 = (D["x"] @ D["W0"] + D["b0"]).relu()
    a2 = (a1 @ D["W1"] + D["b1"]).relu()
    z = a2 @ D["W2"] + D["b2"]
    prob = z.softmax(1)
    loss = -(prob.clamp_min(1e-7).log() * D["T"]).sum().reshape(1) / c["batch"]
    g2 = (prob - D["T"]) / c["batch"]
    g1 = (g2 @ D["W2"].T.contiguous()) * (st["saved2"] > 0)
    g0 = (g1 @ D["W1"].T.contiguous()) * (st["saved1"] > 0)
    return {"z": z, "loss": loss, "gx": g0 @ D["W0"].T.contiguous(), "gW0": D["x"].T.contiguous() @ g0, "gb0": g0.sum(0),
            "gW1": a1.T.contiguous() @ g1, "gb1": g1.sum(0), "gW2": a2.T.contiguous() @ g2, "gb2": g2.sum(0)}


def mlp_work(c):
    b, d = c["batch"], mlp_dims(c)
    w = sum(i * o for i, o in zip(d[:-1], d[1:]))
    return 4.0 * (2 * w + 2 * b * d[0] + 2 * b * d[3] + 2 * sum(d[1:])), 6.0 * b * w


# ---------------------------------------------------------------- convolution layers, inference
# conv -> BatchNorm(running statistics) -> (+ shortcut) -> ReLU as one call per layer. A layer is
# (cin, h, w, cout, k, stride, residual).
def resnet18_layers(side):
    """The 20 convs of ResNet-18 on side x side images (7x7/2 stem, 3x3 blocks, 1x1/2 downsamples)."""
    h = out_size(out_size(side, 7, 2, 3), 3, 2, 1)
    L = [(3, side, side, 64, 7, 2, False)] + [(64, h, h, 64, 3, 1, i % 2 == 1) for i in range(4)]
    for cin, cout in ((64, 128), (128, 256), (256, 512)):
        o = out_size(h, 3, 2, 1)
        L += [(cin, h, h, cout, 3, 2, False), (cout, o, o, cout, 3, 1, True), (cin, h, h, cout, 1, 2, False),
              (cout, o, o, cout, 3, 1, False), (cout, o, o, cout, 3, 1, True)]
        h = o
    return L


def conv_layers(c):
    if c["kind"] == "resnet18_convs":
        return resnet18_layers(c["side"])
    return [(c["cin"], c["h"], c["w"], c["cout"], c["k"], c["stride"], c["residual"])]


def conv_params(s, cin, cout, k):
    lim = math.sqrt(6 / (cin * k * k))
    return {"w": s.uniform(cout, cin, k, k, lo=-lim, hi=lim), "gamma": s.uniform(cout, lo=0.5, hi=1.5),
            "beta": s.randn(cout, std=0.1), "mean": s.randn(cout, std=0.1), "var": s.uniform(cout, lo=0.5, hi=1.5)}


def conv_call(L, x, y, res, n, cin, h, w, cout, k, stride, act):
    bn = (p(L["gamma"]), p(L["beta"]), p(L["mean"]), p(L["var"]), EPS)
    geo = (n, cin, h, w, cout, k, k, stride, k // 2)
    if res is None:
        H.conv2dBiasBnAct(p(x), p(L["w"]), None, *bn, act, p(y), *geo)
    else:
        H.conv2dBiasBnAddAct(p(x), p(L["w"]), None, *bn, p(res), act, p(y), *geo)


def conv64(x, w, stride, pad):
    """conv2d in float64 as unfold + matmul, a few images at a time."""
    n, cin, h, wd = x.shape
    cout, _, k, _ = w.shape
    ho, wo = out_size(h, k, stride, pad), out_size(wd, k, stride, pad)
    W = w.double().reshape(cout, -1)
    step = max(1, int(6e7 // (cin * k * k * ho * wo)))
    y = torch.empty(n, cout, ho * wo, dtype=torch.float64, device=x.device)
    for i in range(0, n, step):
        y[i:i + step] = W @ torch.nn.functional.unfold(x[i:i + step].double(), k, padding=pad, stride=stride)
    return y.reshape(n, cout, ho, wo)


def bn64(y, L):
    v = [L[k].double().reshape(1, -1, 1, 1) for k in ("gamma", "beta", "mean", "var")]
    return v[0] * (y - v[2]) / (v[3] + EPS).sqrt() + v[1]


def convs_inputs(c, s):
    n, layers = c["batch"], []
    for cin, h, w, cout, k, stride, res in conv_layers(c):
        L = conv_params(s, cin, cout, k)
        ho, wo = out_size(h, k, stride, k // 2), out_size(w, k, stride, k // 2)
        L["x"], L["y"] = s.randn(n, cin, h, w), out(n, cout, ho, wo)
        L["res"] = s.randn(n, cout, ho, wo) if res else None
        L["geo"] = (n, cin, h, w, cout, k, stride)
        layers.append(L)
    return {"layers": layers}


def convs_run(c, st):
    for L in st["layers"]:
        conv_call(L, L["x"], L["y"], L["res"], *L["geo"], 1)
    return [L["y"] for L in st["layers"]]


def convs_exact(c, st):
    got = []
    for L in st["layers"]:
        y = bn64(conv64(L["x"], L["w"], L["geo"][6], L["geo"][5] // 2), L)
        got.append((y if L["res"] is None else y + L["res"].double()).relu())
    return got


def convs_work(c):
    n, b, f = c["batch"], 0.0, 0.0
    for cin, h, w, cout, k, stride, res in conv_layers(c):
        o = n * cout * out_size(h, k, stride, k // 2) * out_size(w, k, stride, k // 2)
        b += 4.0 * (n * cin * h * w + cout * cin * k * k + o * (2 if res else 1) + 4 * cout)
        f += 2.0 * o * cin * k * k
    return b, f


# A ResNet-50 bottleneck block, inference: 1x1 -> 3x3 (stride) -> 1x1 + shortcut (1x1 stride when the shape changes).
def bottleneck_layers(c):
    cin, wd, hw, s = c["cin"], c["width"], c["hw"], c["stride"]
    o = out_size(hw, 3, s, 1)
    L = {"c1": (cin, hw, wd, 1, 1), "c2": (wd, hw, wd, 3, s), "c3": (wd, o, 4 * wd, 1, 1)}
    if s != 1 or cin != 4 * wd:
        L["ds"] = (cin, hw, 4 * wd, 1, s)
    return L, o


def bottleneck_inputs(c, s):
    layers, o = bottleneck_layers(c)
    st = {"x": s.randn(c["batch"], c["cin"], c["hw"], c["hw"]).relu_()}
    for name, (cin, h, cout, k, stride) in layers.items():
        ho = out_size(h, k, stride, k // 2)
        st[name], st["y_" + name] = conv_params(s, cin, cout, k), out(c["batch"], cout, ho, ho)
    return st


def bottleneck_run(c, st):
    layers, _ = bottleneck_layers(c)

    def conv(name, x, res, act):
        cin, h, cout, k, stride = layers[name]
        conv_call(st[name], x, st["y_" + name], res, c["batch"], cin, h, h, cout, k, stride, act)
        return st["y_" + name]

    sc = conv("ds", st["x"], None, 0) if "ds" in layers else st["x"]
    y = conv("c3", conv("c2", conv("c1", st["x"], None, 1), None, 1), sc, 1)
    return [st["y_c1"], st["y_c2"], y]


def bottleneck_exact(c, st):
    layers, _ = bottleneck_layers(c)

    def conv(name, x):
        return bn64(conv64(x, st[name]["w"], layers[name][4], layers[name][3] // 2), st[name])

    sc = conv("ds", st["x"]) if "ds" in layers else st["x"].double()
    y1 = conv("c1", st["x"]).relu()
    y2 = conv("c2", y1).relu()
    return [y1, y2, (conv("c3", y2) + sc).relu()]


def bottleneck_work(c):
    n, f, w = c["batch"], 0.0, 0
    layers, o = bottleneck_layers(c)
    for cin, h, cout, k, stride in layers.values():
        f += 2.0 * n * cout * out_size(h, k, stride, k // 2) ** 2 * cin * k * k
        w += cout * cin * k * k + 4 * cout
    # the block's input once, and the three outputs that run() returns
    acts = n * (c["cin"] * c["hw"] ** 2 + c["width"] * c["hw"] ** 2 + c["width"] * o * o + 4 * c["width"] * o * o)
    return 4.0 * (acts + w), f


# ---------------------------------------------------------------- convolution layer, training
# Forward conv -> BatchNorm (batch statistics) -> ReLU, and its backward from the gradient of the ReLU's output and
# the ReLU output saved for it. The gate is given, so that no rounding of this pass decides which way it falls.
def conv_train_inputs(c, s):
    n, cin, h, w, cout, k, stride = (c[k] for k in ("batch", "cin", "h", "w", "cout", "k", "stride"))
    ho, wo = out_size(h, k, stride, k // 2), out_size(w, k, stride, k // 2)
    st = {**conv_params(s, cin, cout, k), "x": s.randn(n, cin, h, w), "gout": s.randn(n, cout, ho, wo),
          "saved": s.randn(n, cout, ho, wo).relu_()}
    for name in ("y", "z", "gy"):
        st[name] = out(n, cout, ho, wo)
    st["gx"], st["gw"] = out(n, cin, h, w), out(cout, cin, k, k)
    for name in ("sm", "si", "ggamma", "gbeta"):
        st[name] = out(cout)
    st["geo"] = (n, cin, h, w, cout, k, k, stride, k // 2)
    st["bn"] = (n, cout, ho, wo, EPS)
    return st


def conv_train_run(c, st):
    q = {k: p(v) for k, v in st.items() if isinstance(v, torch.Tensor)}
    H.conv2d(q["x"], q["w"], None, q["y"], *st["geo"])
    H.batchNorm2dTrainAct(q["y"], q["z"], q["gamma"], q["beta"], q["mean"], q["var"], q["sm"], q["si"], *st["bn"], 0.1,
                          None, 1)
    H.batchNorm2dBackwardRelu(q["gout"], q["saved"], q["y"], q["sm"], q["si"], q["gamma"], q["gy"], q["ggamma"],
                              q["gbeta"], *st["bn"])
    H.conv2dBackwardWeight(q["x"], q["gy"], q["gw"], None, *st["geo"])
    H.conv2dBackwardInput(q["gy"], q["w"], q["gx"], *st["geo"])
    return {k: st[k] for k in ("z", "mean", "var", "gx", "gw", "ggamma", "gbeta")}


def conv_train_exact(c, st):
    n, cin, h, w, cout, k, _, stride, pad = st["geo"]
    y = conv64(st["x"], st["w"], stride, pad)
    m, v = y.mean((0, 2, 3), keepdim=True), y.var((0, 2, 3), unbiased=False, keepdim=True)
    inv = 1 / (v + EPS).sqrt()
    xhat = (y - m) * inv
    gamma, beta = (st[k].double().reshape(1, -1, 1, 1) for k in ("gamma", "beta"))
    g = st["gout"].double() * (st["saved"] > 0)
    ggamma, gbeta = (g * xhat).sum((0, 2, 3)), g.sum((0, 2, 3))
    count = y.numel() // cout
    gy = gamma * inv * (g - (gbeta.reshape(1, -1, 1, 1) + xhat * ggamma.reshape(1, -1, 1, 1)) / count)
    gw = torch.zeros(cout, cin * k * k, dtype=torch.float64, device=y.device)
    gx = torch.empty(n, cin, h, w, dtype=torch.float64, device=y.device)
    Wt = st["w"].double().reshape(cout, -1).T.contiguous()
    gf = gy.reshape(n, cout, -1)
    for i in range(n):
        col = torch.nn.functional.unfold(st["x"][i:i + 1].double(), k, padding=pad, stride=stride)[0]
        gw += gf[i] @ col.T.contiguous()
        gx[i] = torch.nn.functional.fold((Wt @ gf[i])[None], (h, w), k, padding=pad, stride=stride)[0]
    run = {s: 0.9 * st[s].double() + 0.1 * t.reshape(-1) for s, t in (("mean", m), ("var", v))}
    return {"z": (gamma * xhat + beta).relu(), **run, "gx": gx, "gw": gw.reshape(cout, cin, k, k), "ggamma": ggamma,
            "gbeta": gbeta}


def conv_train_work(c):
    n, k = c["batch"], c["k"]
    o = n * c["cout"] * out_size(c["h"], k, c["stride"], k // 2) * out_size(c["w"], k, c["stride"], k // 2)
    x, w = n * c["cin"] * c["h"] * c["w"], c["cout"] * c["cin"] * k * k
    return 4.0 * (2 * x + 2 * w + 3 * o), 6.0 * o * c["cin"] * k * k


# ---------------------------------------------------------------- a whole network
# The device-resident ResNet-18 classifier on normalised images already on the device: logits.
def net_inputs(c, s):
    n, nc = c["batch"], 1000
    layers = resnet18_layers(224)
    L = [conv_params(s, cin, cout, k) for cin, _, _, cout, k, _, _ in layers]
    # the network's order is conv1, conv2, downsample, conv1, conv2 per stage, as the layer list has it
    flat = [t.reshape(-1) for q in L for t in (q["w"], q["gamma"], q["beta"], q["mean"], q["var"])]
    fc, fb = s.randn(512, nc, std=math.sqrt(2.0 / 512)), s.randn(nc, std=0.1)
    x, y = s.randn(n, 3, 224, 224), out(n, nc)
    net = om.ResNet18Infer(torch.cat(flat + [fc.reshape(-1), fb]).cpu().numpy(), nc, n)
    return {"net": net, "x": x, "y": y, "px": types.SimpleNamespace(ptr=p(x)), "py": types.SimpleNamespace(ptr=p(y)),
            "L": L, "fc": fc, "fb": fb}


def net_run(c, st):
    st["net"].forward(st["px"], st["py"], c["batch"])
    return st["y"]


def net_exact(c, st):
    layers, i = resnet18_layers(224), 0

    def conv(x):
        nonlocal i
        L, (_, _, _, _, k, stride, _) = st["L"][i], layers[i]
        i += 1
        return bn64(conv64(x, L["w"], stride, k // 2), L)

    x = torch.nn.functional.max_pool2d(conv(st["x"]).relu(), 3, 2, 1)
    for block in range(8):
        y = conv(conv(x).relu())
        x = (y + (conv(x) if block in (2, 4, 6) else x)).relu()
    return x.mean((2, 3)) @ st["fc"].double() + st["fb"].double()


def net_work(c):
    n = c["batch"]
    f = sum(2.0 * n * cout * out_size(h, k, s, k // 2) ** 2 * cin * k * k for cin, h, _, cout, k, s, _ in resnet18_layers(224))
    w = sum(cout * cin * k * k + 4 * cout for cin, _, _, cout, k, _, _ in resnet18_layers(224)) + 513 * 1000
    return 4.0 * (n * 3 * 224 * 224 + w + 1000 * n), f + 2.0 * n * 512 * 1000


# ---------------------------------------------------------------- half-precision transformer parts
# MultiHeadAttention forward (QKV Linear, attention, output Linear), fp16 / bf16 activations and weights.
def mha_inputs(c, s):
    dt, b, n, h, d = half_type(c), c["batch"], c["seq"], c["heads"], c["hd"]
    D = h * d
    return {"x": s.randn(b * n, D, dtype=dt), "wqkv": s.randn(D, 3 * D, std=0.02, dtype=dt), "bqkv": s.randn(3 * D, std=0.02),
            "wout": s.randn(D, D, std=0.02, dtype=dt), "bout": s.randn(D, std=0.02), "y": out(b * n, D)}


def mha_run(c, st):
    H.multiHeadAttentionHalf(p(st["x"]), p(st["wqkv"]), p(st["bqkv"]), p(st["wout"]), p(st["bout"]), p(st["y"]),
                             c["batch"], c["seq"], c["heads"], c["hd"], bf16=c["dtype"] == "bf16")
    return st["y"]


def attention64(qkv, b, n, h, d, scale):
    q, k, v = (t.contiguous() for t in qkv.reshape(b, n, 3, h, d).permute(2, 0, 3, 1, 4))
    prob = ((q * scale) @ k.transpose(-1, -2).contiguous()).softmax(-1)
    return (prob @ v).transpose(1, 2).reshape(b * n, h * d)


def mha_exact(c, st):
    qkv = st["x"].double() @ st["wqkv"].double() + st["bqkv"].double()
    ctx = attention64(qkv, c["batch"], c["seq"], c["heads"], c["hd"], c["hd"] ** -0.5)
    return ctx @ st["wout"].double() + st["bout"].double()


def mha_work(c):
    t, D = c["batch"] * c["seq"], c["heads"] * c["hd"]
    return 6.0 * t * D + 8.0 * D * D + 16.0 * D, 8.0 * t * D * D + 4.0 * t * c["seq"] * D


# The MLP of a transformer block: Linear + ReLU kept in half precision, then Linear to fp32.
def ffn_inputs(c, s):
    dt, t, d, h = half_type(c), c["tokens"], c["dim"], c["hidden"]
    nt = c["layout"] == "nt"
    return {"x": s.randn(t, d, dtype=dt), "w1": s.randn(*((h, d) if nt else (d, h)), std=0.02, dtype=dt),
            "b1": s.randn(h, std=0.02), "w2": s.randn(*((d, h) if nt else (h, d)), std=0.02, dtype=dt),
            "b2": s.randn(d, std=0.02), "a": out(t, h, dtype=dt), "y": out(t, d)}


def ffn_run(c, st):
    t, d, h, nt, bf = c["tokens"], c["dim"], c["hidden"], c["layout"] == "nt", c["dtype"] == "bf16"
    H.linearHalf(p(st["x"]), p(st["w1"]), p(st["b1"]), p(st["a"]), t, d, h, bf16=bf, transW=nt, act=1, outHalf=True)
    H.linearHalf(p(st["a"]), p(st["w2"]), p(st["b2"]), p(st["y"]), t, h, d, bf16=bf, transW=nt)
    return [st["a"], st["y"]]


def ffn_exact(c, st):
    w1, w2 = ((st[k].double().T if c["layout"] == "nt" else st[k].double()).contiguous() for k in ("w1", "w2"))
    a = (st["x"].double() @ w1 + st["b1"].double()).relu()
    return [a, a @ w2 + st["b2"].double()]


def ffn_work(c):
    t, d, h = c["tokens"], c["dim"], c["hidden"]
    return 2.0 * (t * d + 2 * d * h + t * h) + 4.0 * (t * d + d + h), 4.0 * t * d * h


# ---------------------------------------------------------------- fp32 attention
# The attention core of the fp32 transformer branch: heads split, softmax(scale Q K^T) V, heads merged.
def attn_inputs(c, s):
    t, D = c["batch"] * c["seq"], c["heads"] * c["hd"]
    return {"qkv": s.randn(t, 3 * D), "y": out(t, D)}


def attn_run(c, st):
    H.attention(p(st["qkv"]), p(st["y"]), c["batch"], c["seq"], c["heads"], c["hd"], c["hd"] ** -0.5)
    return st["y"]


def attn_exact(c, st):
    return attention64(st["qkv"].double(), c["batch"], c["seq"], c["heads"], c["hd"], c["hd"] ** -0.5)


def attn_work(c):
    t, D = c["batch"] * c["seq"], c["heads"] * c["hd"]
    return 16.0 * t * D, 4.0 * t * c["seq"] * D


KINDS = {
    "gemm": (gemm_inputs, gemm_run, gemm_exact, gemm_work),
    "mlp": (mlp_inputs, mlp_run, mlp_exact, mlp_work),
    "conv": (convs_inputs, convs_run, convs_exact, convs_work),
    "resnet18_convs": (convs_inputs, convs_run, convs_exact, convs_work),
    "bottleneck": (bottleneck_inputs, bottleneck_run, bottleneck_exact, bottleneck_work),
    "conv_train": (conv_train_inputs, conv_train_run, conv_train_exact, conv_train_work),
    "net": (net_inputs, net_run, net_exact, net_work),
    "mha": (mha_inputs, mha_run, mha_exact, mha_work),
    "ffn": (ffn_inputs, ffn_run, ffn_exact, ffn_work),
    "attention": (attn_inputs, attn_run, attn_exact, attn_work),
}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a small classifier's training step: five short launches, latency
        {"name": "mlp_step_b128", "kind": "mlp", "batch": 128, "d0": 784, "d1": 256, "d2": 128, "classes": 10},
        # a weight gradient of odd sizes: no row of either operand is a whole number of 16-byte words
        {"name": "gemm_tn_odd", "kind": "gemm", "layout": "tn", "batch": 1, "m": 1001, "n": 765, "k": 1537},
        # a Linear layer on few rows
        {"name": "gemm_nt_128x4096x4096", "kind": "gemm", "layout": "nt", "batch": 1, "m": 128, "n": 4096, "k": 4096},
        # a large product
        {"name": "gemm_nn_4096", "kind": "gemm", "layout": "nn", "batch": 1, "m": 4096, "n": 4096, "k": 4096},
        # the convolutions of ResNet-18 on a batch of 32 images
        {"name": "resnet18_convs_b32", "kind": "resnet18_convs", "batch": 32, "side": 224},
        # a convolution off the usual sizes: odd image, ragged channel counts, 5x5 stride 2
        {"name": "conv_odd_5x5", "kind": "conv", "batch": 5, "cin": 46, "h": 61, "w": 53, "cout": 75, "k": 5, "stride": 2,
         "residual": False},
        # a ResNet-50 block, mostly 1x1 convolutions
        {"name": "bottleneck_b64", "kind": "bottleneck", "batch": 64, "cin": 512, "width": 128, "hw": 28, "stride": 1},
        # one training layer, forward and backward
        {"name": "conv_train_b32", "kind": "conv_train", "batch": 32, "cin": 128, "h": 28, "w": 28, "cout": 128, "k": 3,
         "stride": 1},
        # one image through the classifier
        {"name": "resnet18_b1", "kind": "net", "batch": 1},
        # ViT-B/16 at batch 64, fp16: the attention layer
        {"name": "mha_fp16_b64", "kind": "mha", "dtype": "fp16", "batch": 64, "seq": 197, "heads": 12, "hd": 64},
        # ViT-B/16 at batch 64, bf16: the MLP
        {"name": "ffn_bf16_b64", "kind": "ffn", "dtype": "bf16", "layout": "nn", "tokens": 12608, "dim": 768, "hidden": 3072},
        # the fp32 branch's attention core
        {"name": "attention_fp32_b16", "kind": "attention", "batch": 16, "seq": 197, "heads": 12, "hd": 64},
    ]


def spread(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def sized(rng, lo, hi, step):
    """spread(), three times in four rounded to a multiple of `step`, otherwise as it falls."""
    v = spread(rng, lo, hi)
    return max(step, v // step * step) if rng.random() < 0.75 else v


def drawn(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "mlp", "conv", "conv", "resnet18_convs", "bottleneck", "conv_train",
                       "conv_train", "net", "mha", "ffn", "attention"])
    if kind == "gemm":
        batch = spread(rng, 2, 256) if rng.random() < 0.25 else 1
        top = 512 if batch > 1 else 8192
        return {"kind": kind, "layout": rng.choice(["nn", "nt"] if batch > 1 else ["nn", "nt", "tn"]), "batch": batch,
                **{a: sized(rng, 8, top, 8) for a in "mnk"}}
    if kind == "mlp":
        return {"kind": kind, "batch": spread(rng, 1, 1024), "d0": sized(rng, 16, 4096, 4), "d1": sized(rng, 16, 2048, 4),
                "d2": sized(rng, 16, 1024, 4), "classes": spread(rng, 2, 1000)}
    if kind in ("conv", "conv_train"):
        side = spread(rng, 7, 112)
        c = {"kind": kind, "batch": spread(rng, 1, 32), "cin": sized(rng, 4, 512, 8), "h": side,
             "w": side if rng.random() < 0.7 else spread(rng, 7, 112), "cout": sized(rng, 8, 512, 8),
             "k": rng.choice([1, 3, 3, 3, 5]), "stride": rng.choice([1, 1, 2])}
        return {**c, "residual": rng.random() < 0.4} if kind == "conv" else c
    if kind == "resnet18_convs":
        return {"kind": kind, "batch": spread(rng, 1, 32), "side": 32 * rng.randint(1, 7)}
    if kind == "bottleneck":
        i = rng.randint(0, 3)
        s = rng.choice([1, 2])
        width, hw = 64 << i, 56 >> i
        return {"kind": kind, "batch": spread(rng, 1, 64), "cin": 4 * width if s == 1 else 2 * width, "width": width,
                "hw": hw * s, "stride": s}
    if kind == "net":
        return {"kind": kind, "batch": spread(rng, 1, 32)}
    if kind == "mha":
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "batch": spread(rng, 1, 64), "seq": spread(rng, 16, 384),
                "heads": rng.choice([3, 6, 8, 12, 16]), "hd": 64}
    if kind == "ffn":
        dim = sized(rng, 64, 1024, 64)
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "layout": rng.choice(["nn", "nt"]),
                "tokens": spread(rng, 1, 12608), "dim": dim, "hidden": 4 * dim}
    return {"kind": kind, "batch": spread(rng, 1, 64), "seq": spread(rng, 16, 512), "heads": rng.choice([3, 6, 8, 12, 16]),
            "hd": rng.choice([32, 64, 64, 80])}


def draw(rng):
    while True:
        c = drawn(rng)
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


def prepare(case, seed):
    om.init(0)
    st = KINDS[case["kind"]][0](case, Source(seed))
    torch.cuda.synchronize()  # the inputs were made on torch's stream, the backend has its own
    return case, st


def run(state):
    case, st = state
    return KINDS[case["kind"]][1](case, st)


def exact(case, seed):
    return KINDS[case["kind"]][2](case, KINDS[case["kind"]][0](case, Source(seed)))


def work(case):
    b, f = KINDS[case["kind"]][3](case)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the difference seen between these outputs and float64."""
    kind = case["kind"]
    if kind in ("mha", "ffn"):
        # half-precision intermediates: a sum that rounds the other way moves one of them by a unit in the last place
        return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.02}
    return {"rel": 1e-5, "max": 2e-4}
