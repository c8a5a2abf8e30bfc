"""The work that programs have this library do, as measurable cases.

Every case goes through the public entry points (``neuralrs_amd._abi``, the
binding of ``include/nrs_hip.h``) on device tensors, on the default stream,
with output buffers and weights that the program keeps from call to call.
f32 is the library's only type.

A training step's forward and backward appear together: the forward runs on
this batch, the backward on the activations kept from the forward of the
batch before (they are part of the prepared state), so that every output
depends on the inputs alone and not on which side of zero a rounding error
put a ReLU.
"""
import math

import torch

from neuralrs_amd import _abi as nrs

LAYOUTS = {"NN": nrs.NN, "NT": nrs.NT, "TN": nrs.TN}
EPS = 1e-5  # LayerNorm


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest call: one classifier head on a small batch (the Linear
        # twin test's sizes), forward and backward. Launches and host time.
        {"name": "linear_16x24x10", "kind": "linear", "batch": 16, "in_f": 24, "out_f": 10},
        # A whole training step of the MNIST MLP 784-128-10 at batch 256.
        {"name": "mlp_256x784x128x10", "kind": "mlp", "batch": 256, "in_f": 784, "hidden": 128,
         "classes": 10},
        # A matrix product of no special size: odd rows, columns and depth.
        {"name": "gemm_nt_1000x1333x777", "kind": "gemm", "layout": "NT", "m": 1000, "n": 1333,
         "k": 777},
        # The headline product, and the largest case.
        {"name": "gemm_nn_4096", "kind": "gemm", "layout": "NN", "m": 4096, "n": 4096, "k": 4096},
        # A few rows against a large weight: inference of a wide layer.
        {"name": "gemm_nn_32x8192x8192", "kind": "gemm", "layout": "NN", "m": 32, "n": 8192,
         "k": 8192},
        # The convolution weight gradient as a product: a small output over a
        # reduction of batch times pixels.
        {"name": "splitk_64x576x100352", "kind": "splitk", "m": 64, "n": 576, "k": 100352},
        # The feed-forward half of a TransformerBlock (batch 32, sequence 128,
        # d 256, inner 1024) with its residual LayerNorm, both directions.
        {"name": "ffn_4096x256x1024", "kind": "ffn", "rows": 4096, "d": 256, "inner": 1024},
        # Its attention half: projections, the fused core, the output
        # projection, both directions.
        {"name": "mha_32x128x256h8", "kind": "mha", "batch": 32, "seq": 128, "heads": 8,
         "d_head": 32},
        # The attention core alone over a long, ragged sequence.
        {"name": "attention_4x1000h8", "kind": "attention", "batch": 4, "seq": 1000, "heads": 8,
         "d_head": 32},
        # Heads the fused core does not take: split heads, batched products
        # and softmax, as the operator layer composes them.
        {"name": "composed_8x256h8x64", "kind": "composed", "batch": 8, "seq": 256, "heads": 8,
         "d_head": 64},
        # The MNIST CNN's step at batch 128: conv 1->32, ReLU, 2x2 pool, conv
        # 32->64, both directions.
        {"name": "cnn_128x28x28", "kind": "cnn", "batch": 128, "size": 28, "c_mid": 32,
         "c_out": 64},
        # A single convolution layer of an image network, 16 -> 32 channels of
        # 64 x 64 pixels (the size of the CPU convolution benchmark).
        {"name": "conv_32x16x64_32k3", "kind": "conv", "batch": 32, "c_in": 16, "c_out": 32,
         "h": 64, "w": 64, "ksize": 3, "stride": 1, "pad": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size spread over the logarithm of its range: as it falls, or, as layer
    sizes mostly are, a multiple of 8."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.5 else max(lo, (v + 4) // 8 * 8)


def draw(rng):
    kind = rng.choice(["linear", "mlp", "gemm", "gemm", "skinny", "splitk", "ffn", "mha",
                       "attention", "composed", "cnn", "conv"])
    if kind == "linear":
        return {"kind": kind, "batch": _size(rng, 1, 4096), "in_f": _size(rng, 8, 2048),
                "out_f": _size(rng, 2, 2048)}
    if kind == "mlp":
        return {"kind": kind, "batch": _size(rng, 16, 2048), "in_f": _size(rng, 16, 1024),
                "hidden": _size(rng, 16, 256), "classes": rng.randint(2, 16)}
    if kind == "gemm":
        return {"kind": kind, "layout": rng.choice(list(LAYOUTS)), "m": _size(rng, 33, 4096),
                "n": _size(rng, 33, 4096), "k": _size(rng, 32, 4096)}
    if kind == "skinny":
        return {"kind": "gemm", "layout": rng.choice(list(LAYOUTS)), "m": _size(rng, 1, 32),
                "n": _size(rng, 1024, 8192), "k": _size(rng, 256, 8192)}
    if kind == "splitk":
        return {"kind": kind, "m": _size(rng, 16, 256), "n": _size(rng, 27, 1152),
                "k": _size(rng, 4096, 100352)}
    if kind == "ffn":
        d = _size(rng, 32, 512)
        return {"kind": kind, "rows": _size(rng, 64, 8192), "d": d, "inner": 4 * d}
    if kind == "mha":
        return {"kind": kind, "batch": _size(rng, 1, 64), "seq": rng.randint(16, 128),
                "heads": rng.choice([2, 4, 8]), "d_head": rng.choice([16, 32])}
    if kind == "attention":
        seq = _log(rng, 129, 2048)
        return {"kind": kind, "batch": _log(rng, 1, max(1, 8000 // seq)), "seq": seq,
                "heads": rng.choice([1, 2, 4, 8]), "d_head": rng.choice([16, 32])}
    if kind == "composed":
        seq = _log(rng, 32, 512)
        return {"kind": kind, "batch": _log(rng, 1, max(1, 4096 // seq)), "seq": seq,
                "heads": rng.choice([1, 2, 4, 8]), "d_head": rng.choice([20, 40, 48, 64, 80, 128])}
    if kind == "cnn":
        return {"kind": kind, "batch": _size(rng, 16, 256), "size": rng.choice([16, 20, 24, 28]),
                "c_mid": rng.choice([16, 32]), "c_out": rng.choice([32, 64])}
    size = rng.randint(7, 64)
    k = rng.choice([1, 3, 3, 3, 5])
    c_in = rng.choice([3, 8, 16, 24, 32, 64, 128])
    most = max(4, 40_000_000 // (size * size * c_in))
    return {"kind": kind, "batch": _log(rng, 4, max(4, min(128, most))), "c_in": c_in,
            "c_out": rng.choice([16, 20, 32, 64, 128]), "h": size, "w": size, "ksize": k,
            "stride": rng.choice([1, 1, 1, 2]), "pad": k // 2}


# ------------------------------------------------------------------ the inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda") * 2 - 1

    def he(self, fan_in, *shape):
        return self.normal(*shape, std=math.sqrt(2.0 / fan_in))

    def one_hot(self, batch, classes):
        t = torch.randint(classes, (batch,), generator=self.g, device="cuda")
        return torch.nn.functional.one_hot(t, classes).float()


def _norm64(s, gamma, beta):
    mean = s.mean(1, keepdim=True)
    inv = 1 / torch.sqrt(((s - mean) ** 2).mean(1, keepdim=True) + EPS)
    xn = (s - mean) * inv
    return xn * gamma + beta, xn, inv[:, 0]


def _pool64(y):
    """2 x 2 max pool over ReLU(y): values, and the first maximum's flat index."""
    b, c, h, w = y.shape
    t = y.clamp(min=0).reshape(b, c, h // 2, 2, w // 2, 2).permute(0, 1, 2, 4, 3, 5)
    t = t.reshape(b, c, h // 2, w // 2, 4)
    best = t.max(4).values
    first = (t == best[..., None]).int().argmax(4)
    oy = torch.arange(h // 2, device=y.device)[:, None] * 2 + first // 2
    ox = torch.arange(w // 2, device=y.device)[None, :] * 2 + first % 2
    plane = torch.arange(b * c, device=y.device).reshape(b, c, 1, 1) * (h * w)
    return best, (plane + oy * w + ox).int()


def _conv64(x, w, b, stride, pad):
    n, k = x.shape[0], w.shape[2]
    oh = (x.shape[2] + 2 * pad - k) // stride + 1
    ow = (x.shape[3] + 2 * pad - k) // stride + 1
    out = [torch.matmul(w.reshape(w.shape[0], -1),
                        torch.nn.functional.unfold(x[i:i + 8], k, padding=pad, stride=stride))
           for i in range(0, n, 8)]
    return torch.cat(out).reshape(n, w.shape[0], oh, ow) + b.reshape(1, -1, 1, 1)


def _conv64_backward(g, x, w, stride, pad):
    """dx, dw, db."""
    n, k = x.shape[0], w.shape[2]
    wm = w.reshape(w.shape[0], -1)
    wt = wm.t().contiguous()
    dx, dw = [], torch.zeros_like(wm)
    for i in range(0, n, 8):
        gi = g[i:i + 8].reshape(-1, w.shape[0], g.shape[2] * g.shape[3])
        cols = torch.nn.functional.unfold(x[i:i + 8], k, padding=pad, stride=stride)
        dw += torch.bmm(gi, cols.transpose(1, 2).contiguous()).sum(0)
        dx.append(torch.nn.functional.fold(torch.matmul(wt, gi), x.shape[2:], k, padding=pad,
                                           stride=stride))
    return torch.cat(dx), dw.reshape(w.shape), g.sum((0, 2, 3))


def _inputs(c, seed):
    """The case's input tensors: made from the seed alone."""
    r, kind = _Rand(seed), c["kind"]
    if kind == "linear":
        b, i, o = c["batch"], c["in_f"], c["out_f"]
        return dict(x=r.normal(b, i), w=r.he(i, i, o), b=r.normal(o, std=0.1),
                    g=r.normal(b, o, std=1.0 / b))
    if kind == "mlp":
        b, i, h, k = c["batch"], c["in_f"], c["hidden"], c["classes"]
        # pixels: a dark background and bright strokes
        x = r.uniform(b, i).clamp(min=0) * (r.uniform(b, i) > 0)
        return dict(x=x, w1=r.he(i, i, h), b1=r.normal(h, std=0.05), w2=r.he(h, h, k),
                    b2=r.normal(k, std=0.05), target=r.one_hot(b, k),
                    # kept from the batch before
                    h0=r.normal(b, h).clamp(min=0), gz0=r.normal(b, k, std=0.3 / b),
                    dh0=r.normal(b, h, std=0.2 / b).clamp(min=0))
    if kind in ("gemm", "splitk"):
        m, n, k = c["m"], c["n"], c["k"]
        layout = c.get("layout", "NT")
        if kind == "splitk":  # an output gradient against im2col'd activations
            return dict(a=r.normal(m, k, std=0.01), b=r.normal(n, k).clamp(min=0))
        return dict(a=r.uniform(*((k, m) if layout == "TN" else (m, k))),
                    b=r.uniform(*((n, k) if layout == "NT" else (k, n))))
    if kind == "ffn":
        n, d, f = c["rows"], c["d"], c["inner"]
        return dict(x=r.normal(n, d), w1=r.he(d, d, f), b1=r.normal(f, std=0.05),
                    w2=r.he(f, f, d), b2=r.normal(d, std=0.05), gamma=1 + r.normal(d, std=0.1),
                    beta=r.normal(d, std=0.1), g=r.normal(n, d, std=1.0 / n),
                    # kept from the batch before: its input, hidden activation,
                    # normalised sum and inverse deviations
                    x0=r.normal(n, d), h0=r.normal(n, f).clamp(min=0), xn0=r.normal(n, d),
                    inv0=0.5 + 0.2 * r.uniform(n))
    if kind == "mha":
        n, d = c["batch"] * c["seq"], c["heads"] * c["d_head"]
        s = 1 / math.sqrt(d)
        return dict(x=r.normal(n, d), wq=r.normal(d, d, std=s), wk=r.normal(d, d, std=s),
                    wv=r.normal(d, d, std=s), wo=r.normal(d, d, std=s),
                    g=r.normal(n, d, std=1.0 / n))
    if kind in ("attention", "composed"):
        n, d = c["batch"] * c["seq"], c["heads"] * c["d_head"]
        return dict(q=r.normal(n, d), k=r.normal(n, d), v=r.normal(n, d),
                    g=r.normal(n, d, std=1.0 / n))
    if kind == "cnn":
        b, s, m, o = c["batch"], c["size"], c["c_mid"], c["c_out"]
        i = dict(x=r.uniform(b, 1, s, s).clamp(min=0), w1=r.he(9, m, 1, 3, 3),
                 b1=r.normal(m, std=0.05), w2=r.he(9 * m, o, m, 3, 3), b2=r.normal(o, std=0.05),
                 g=r.normal(b, o, s // 2, s // 2, std=1.0 / b),
                 x0=r.uniform(b, 1, s, s).clamp(min=0))
        # kept from the batch before: its pooled activation and argmax
        p0, i["argmax0"] = _pool64(_conv64(i["x0"].double(), i["w1"].double(), i["b1"].double(),
                                           1, 1))
        i["pooled0"] = p0.float()
        return i
    assert kind == "conv", kind
    b, ci, co, k = c["batch"], c["c_in"], c["c_out"], c["ksize"]
    oh, ow = _conv_out(c)
    return dict(x=r.normal(b, ci, c["h"], c["w"]).clamp(min=0), w=r.he(ci * k * k, co, ci, k, k),
                b=r.normal(co, std=0.05), g=r.normal(b, co, oh, ow, std=1.0 / b))


def _conv_out(c):
    f = lambda v: (v + 2 * c["pad"] - c["ksize"]) // c["stride"] + 1
    return f(c["h"]), f(c["w"])


# --------------------------------------------------------------- prepare / run
def prepare(case, seed):
    nrs.init(0)
    c = dict(case)
    i = {k: v.contiguous() for k, v in _inputs(c, seed).items()}
    e = lambda *shape, dtype=torch.float32: torch.empty(*shape, dtype=dtype, device="cuda")
    like = lambda t: torch.empty_like(t)
    kind = c["kind"]
    if kind == "linear":
        o = dict(y=e(c["batch"], c["out_f"]), dx=like(i["x"]), dw=like(i["w"]), db=like(i["b"]))
    elif kind == "mlp":
        b, h, k = c["batch"], c["hidden"], c["classes"]
        o = dict(h=e(b, h), z=e(b, k), gz=e(b, k), dh=e(b, h), dx=like(i["x"]),
                 dw1=like(i["w1"]), db1=like(i["b1"]), dw2=like(i["w2"]), db2=like(i["b2"]))
    elif kind in ("gemm", "splitk"):
        o = dict(c=e(c["m"], c["n"]))
    elif kind == "ffn":
        n, d, f = c["rows"], c["d"], c["inner"]
        o = dict(h=e(n, f), y=e(n, d), out=e(n, d), xn=e(n, d), inv=e(n), ds=e(n, d),
                 dx=e(n, d), dh=e(n, f), dw1=like(i["w1"]), db1=like(i["b1"]), dw2=like(i["w2"]),
                 db2=like(i["b2"]), dgamma=e(d), dbeta=e(d))
    elif kind == "mha":
        n, d = c["batch"] * c["seq"], c["heads"] * c["d_head"]
        names = ["q", "k", "v", "a", "y", "da", "dq", "dk", "dv", "dx"]
        o = {k: e(n, d) for k in names}
        o.update({k: e(d, d) for k in ("dwq", "dwk", "dwv", "dwo")})
        o["stats"] = e(n * c["heads"] * 2)
    elif kind == "attention":
        o = {k: like(i["q"]) for k in ("out", "dq", "dk", "dv")}
        o["stats"] = e(c["batch"] * c["heads"] * c["seq"] * 2)
    elif kind == "composed":
        items, s, dh = c["batch"] * c["heads"], c["seq"], c["d_head"]
        o = {k: like(i["q"]) for k in ("out", "dq", "dk", "dv")}
        o.update({k: e(items, s, dh) for k in ("qh", "kh", "vh", "oh", "gh", "dqh", "dkh", "dvh")})
        o.update({k: e(items, s, s) for k in ("scores", "p", "dp", "dscores")})
    elif kind == "cnn":
        b, s, m = c["batch"], c["size"], c["c_mid"]
        o = dict(pooled=e(b, m, s // 2, s // 2), argmax=e(b, m, s // 2, s // 2, dtype=torch.int32),
                 y=like(i["g"]), dpooled=e(b, m, s // 2, s // 2), dw2=like(i["w2"]),
                 db2=like(i["b2"]), dw1=like(i["w1"]), db1=like(i["b1"]))
    else:
        o = dict(y=like(i["g"]), dx=like(i["x"]), dw=like(i["w"]), db=like(i["b"]))
    return {"case": c, "in": i, "out": o}


def run(state):
    c, i, o = state["case"], state["in"], state["out"]
    return _RUN[c["kind"]](c, i, o)


def _run_linear(c, i, o):
    b, n, k = c["batch"], c["out_f"], c["in_f"]
    nrs.gemm(nrs.NN, o["y"], i["x"], i["w"], b, n, k, 0.0, i["b"], nrs.EPI_BIAS_COL)
    nrs.call("nrs_linear_backward", o["dx"], o["dw"], o["db"], i["g"], i["x"], i["w"], b, k, n,
             0.0, 0.0, 0.0)
    return o


def _run_mlp(c, i, o):
    s = (c["batch"], c["in_f"], c["hidden"], c["classes"])
    nrs.call("nrs_mlp2_forward_seed", o["h"], o["z"], o["gz"], o["dh"], i["x"], i["w1"], i["b1"],
             i["w2"], i["b2"], i["target"], *s)
    nrs.call("nrs_mlp2_backward", o["dx"], o["dw1"], o["db1"], o["dw2"], o["db2"], i["dh0"],
             i["gz0"], i["x"], i["w1"], i["h0"], *s, 0.0, 0.0)
    return o


def _run_gemm(c, i, o):
    nrs.gemm(LAYOUTS[c["layout"]], o["c"], i["a"], i["b"], c["m"], c["n"], c["k"])
    return o


def _run_splitk(c, i, o):
    nrs.gemm_nt_splitk(o["c"], i["a"], i["b"], c["m"], c["n"], c["k"])
    return o


def _run_ffn(c, i, o):
    n, d, f = c["rows"], c["d"], c["inner"]
    nrs.gemm(nrs.NN, o["h"], i["x"], i["w1"], n, f, d, 0.0, i["b1"],
             nrs.EPI_BIAS_COL | nrs.EPI_RELU)
    nrs.gemm(nrs.NN, o["y"], o["h"], i["w2"], n, d, f, 0.0, i["b2"], nrs.EPI_BIAS_COL)
    nrs.call("nrs_add_layernorm_forward", o["out"], o["xn"], o["inv"], i["x"], o["y"],
             i["gamma"], i["beta"], n, d, EPS)
    # the sum's gradient goes to the residual (dx) and to the FFN's output (ds)
    nrs.call("nrs_add_layernorm_backward", o["dx"], o["ds"], o["dgamma"], o["dbeta"], i["g"],
             i["gamma"], i["xn0"], i["inv0"], n, d, 0.0, 0.0, 0.0)
    nrs.call("nrs_linear_backward_relu", o["dh"], o["dw2"], o["db2"], o["ds"], i["h0"], i["w2"],
             i["h0"], n, f, d, 0.0, 0.0, 0.0)
    nrs.call("nrs_linear_backward", o["dx"], o["dw1"], o["db1"], o["dh"], i["x0"], i["w1"], n, d,
             f, 1.0, 0.0, 0.0)
    return o


def _run_mha(c, i, o):
    b, s, h, dh = c["batch"], c["seq"], c["heads"], c["d_head"]
    n, d, scale = b * s, h * dh, 1 / math.sqrt(dh)
    nrs.gemm_group([(nrs.NN, o[t], i["x"], i["w" + t], n, d, d) for t in "qkv"])
    nrs.call("nrs_attention_forward", o["a"], o["stats"], o["q"], o["k"], o["v"], b, h, s, dh, d,
             scale)
    nrs.gemm(nrs.NN, o["y"], o["a"], i["wo"], n, d, d)
    nrs.gemm_group([(nrs.NT, o["da"], i["g"], i["wo"], n, d, d),
                    (nrs.TN, o["dwo"], o["a"], i["g"], d, d, n)])
    nrs.call("nrs_attention_backward", o["dq"], o["dk"], o["dv"], o["da"], o["a"], o["q"], o["k"],
             o["v"], o["stats"], b, h, s, dh, d, scale, 0.0)
    nrs.matmul_shared_lhs_backward(o["dx"], [o["dwq"], o["dwk"], o["dwv"]],
                                   [o["dq"], o["dk"], o["dv"]], i["x"],
                                   [i["wq"], i["wk"], i["wv"]], n, d, d)
    return {k: v for k, v in o.items() if k != "stats"}


def _run_attention(c, i, o):
    b, s, h, dh = c["batch"], c["seq"], c["heads"], c["d_head"]
    d, scale = h * dh, 1 / math.sqrt(dh)
    nrs.call("nrs_attention_forward", o["out"], o["stats"], i["q"], i["k"], i["v"], b, h, s, dh,
             d, scale)
    nrs.call("nrs_attention_backward", o["dq"], o["dk"], o["dv"], i["g"], o["out"], i["q"],
             i["k"], i["v"], o["stats"], b, h, s, dh, d, scale, 0.0)
    return {k: v for k, v in o.items() if k != "stats"}


def _run_composed(c, i, o):
    b, s, h, dh = c["batch"], c["seq"], c["heads"], c["d_head"]
    rows, items, scale = b * s, b * h, 1 / math.sqrt(dh)
    for t, th in (("q", "qh"), ("k", "kh"), ("v", "vh"), ("g", "gh")):
        nrs.call("nrs_split_heads", o[th], i[t], rows, h, dh, 0.0)
    nrs.bmm(nrs.NT, o["scores"], o["qh"], o["kh"], items, s, s, dh)
    nrs.call("nrs_softmax_forward_scaled", o["p"], o["scores"], items * s, s, scale)
    nrs.bmm(nrs.NN, o["oh"], o["p"], o["vh"], items, s, dh, s)
    nrs.call("nrs_merge_heads", o["out"], o["oh"], rows, h, dh, 0.0)
    nrs.bmm_backward(nrs.NN, o["dp"], o["dvh"], o["gh"], o["p"], o["vh"], items, s, s, dh)
    nrs.call("nrs_softmax_backward_scaled", o["dscores"], o["p"], o["dp"], items * s, s, scale,
             0.0)
    nrs.bmm_backward(nrs.NT, o["dqh"], o["dkh"], o["dscores"], o["qh"], o["kh"], items, s, dh, s)
    for t in ("dq", "dk", "dv"):
        nrs.call("nrs_merge_heads", o[t], o[t + "h"], rows, h, dh, 0.0)
    return {k: o[k] for k in ("p", "out", "dq", "dk", "dv")}


def _run_cnn(c, i, o):
    b, s, m, k = c["batch"], c["size"], c["c_mid"], c["c_out"]
    half = s // 2
    nrs.call("nrs_conv2d_relu_maxpool_forward", o["pooled"], o["argmax"], None, i["x"], i["w1"],
             i["b1"], b, 1, s, s, m, 3, 3, 1, 1, 2, 2)
    nrs.call("nrs_conv2d_forward", o["y"], o["pooled"], i["w2"], i["b2"], b, m, half, half, k, 3,
             3, 1, 1)
    nrs.call("nrs_conv2d_maxpool_relu_conv2d_backward", o["dpooled"], o["dw2"], o["db2"],
             o["dw1"], o["db1"], i["g"], i["pooled0"], i["w2"], i["argmax0"], i["x0"], i["w1"], b,
             1, s, s, m, 3, 3, 1, 1, 2, 2, k, 3, 3, 1, 1, 0.0)
    return o


def _run_conv(c, i, o):
    s = (c["batch"], c["c_in"], c["h"], c["w"], c["c_out"], c["ksize"], c["ksize"], c["stride"],
         c["pad"])
    nrs.call("nrs_conv2d_forward", o["y"], i["x"], i["w"], i["b"], *s)
    nrs.call("nrs_conv2d_backward_ex", o["dx"], o["dw"], o["db"], i["g"], i["x"], i["w"], *s, 0.0,
             0.0)
    return o


_RUN = {"linear": _run_linear, "mlp": _run_mlp, "gemm": _run_gemm, "splitk": _run_splitk,
        "ffn": _run_ffn, "mha": _run_mha, "attention": _run_attention,
        "composed": _run_composed, "cnn": _run_cnn, "conv": _run_conv}


# ------------------------------------------------------------------- the work
def work(case):
    """Bytes: every input read and every output written once. Operations: the
    products' multiplies and adds."""
    c, kind = case, case["kind"]
    if kind == "linear":
        b, i, n = c["batch"], c["in_f"], c["out_f"]
        return {"bytes": 4 * (2 * b * i + 2 * i * n + 2 * n + 2 * b * n), "flops": 6 * b * i * n}
    if kind == "mlp":
        b, i, h, k = c["batch"], c["in_f"], c["hidden"], c["classes"]
        return {"bytes": 4 * (2 * b * i + 2 * i * h + 2 * h * k + 4 * b * h + 4 * b * k),
                "flops": 6 * b * i * h + 6 * b * h * k}
    if kind in ("gemm", "splitk"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "ffn":
        n, d, f = c["rows"], c["d"], c["inner"]
        # x, g, x0, xn0 in; y, out, xn, ds, dx out; h, dh out, h0 in
        return {"bytes": 4 * (9 * n * d + 3 * n * f + 4 * d * f), "flops": 12 * n * d * f}
    if kind == "mha":
        n, d, s = c["batch"] * c["seq"], c["heads"] * c["d_head"], c["seq"]
        # x, g in; q, k, v, a, y, da, dq, dk, dv, dx out
        return {"bytes": 4 * (12 * n * d + 8 * d * d), "flops": 24 * n * d * d + 12 * n * s * d}
    if kind in ("attention", "composed"):
        n, d, s = c["batch"] * c["seq"], c["heads"] * c["d_head"], c["seq"]
        p = c["heads"] * n * s if kind == "composed" else 0
        return {"bytes": 4 * (8 * n * d + p), "flops": 12 * n * s * d}
    if kind == "cnn":
        b, s, m, o = c["batch"], c["size"], c["c_mid"], c["c_out"]
        px, half = b * s * s, b * (s // 2) ** 2
        return {"bytes": 4 * (2 * px + 5 * half * m + 2 * half * o + 18 * m * o),
                "flops": 2 * 2 * px * m * 9 + 3 * 2 * half * o * m * 9}
    oh, ow = _conv_out(c)
    x, y = c["batch"] * c["c_in"] * c["h"] * c["w"], c["batch"] * c["c_out"] * oh * ow
    w = c["c_in"] * c["c_out"] * c["ksize"] ** 2
    return {"bytes": 4 * (2 * x + 2 * y + 2 * w),
            "flops": 6 * y * c["c_in"] * c["ksize"] ** 2}


# ------------------------------------------------------------------ the oracle
def exact(case, seed):
    """What run() returns, in 64 bits, in plain torch."""
    c, kind = dict(case), case["kind"]
    i = {k: (v.double() if v.is_floating_point() else v) for k, v in _inputs(c, seed).items()}
    t = lambda m: m.t().contiguous()
    if kind == "linear":
        return dict(y=i["x"] @ i["w"] + i["b"], dx=i["g"] @ t(i["w"]), dw=t(i["x"]) @ i["g"],
                    db=i["g"].sum(0))
    if kind == "mlp":
        h = (i["x"] @ i["w1"] + i["b1"]).clamp(min=0)
        z = h @ i["w2"] + i["b2"]
        gz = (torch.softmax(z, 1) - i["target"]) / c["batch"]
        return dict(h=h, z=z, gz=gz, dh=(gz @ t(i["w2"])) * (h > 0), dx=i["dh0"] @ t(i["w1"]),
                    dw1=t(i["x"]) @ i["dh0"], db1=i["dh0"].sum(0), dw2=t(i["h0"]) @ i["gz0"],
                    db2=i["gz0"].sum(0))
    if kind in ("gemm", "splitk"):
        layout = c.get("layout", "NT")
        a = t(i["a"]) if layout == "TN" else i["a"]
        return dict(c=a @ (t(i["b"]) if layout == "NT" else i["b"]))
    if kind == "ffn":
        h = (i["x"] @ i["w1"] + i["b1"]).clamp(min=0)
        y = h @ i["w2"] + i["b2"]
        out, xn, inv = _norm64(i["x"] + y, i["gamma"], i["beta"])
        dxh = i["g"] * i["gamma"]
        ds = i["inv0"][:, None] * (dxh - dxh.mean(1, keepdim=True)
                                   - i["xn0"] * (dxh * i["xn0"]).mean(1, keepdim=True))
        dh = (ds @ t(i["w2"])) * (i["h0"] > 0)
        return dict(h=h, y=y, out=out, xn=xn, inv=inv, ds=ds, dx=ds + dh @ t(i["w1"]), dh=dh,
                    dw1=t(i["x0"]) @ dh, db1=dh.sum(0), dw2=t(i["h0"]) @ ds, db2=ds.sum(0),
                    dgamma=(i["g"] * i["xn0"]).sum(0), dbeta=i["g"].sum(0))
    if kind == "mha":
        q, k, v = (i["x"] @ i["w" + n] for n in "qkv")
        a, back = _attention64(c, q, k, v)
        da = i["g"] @ t(i["wo"])
        dq, dk, dv, _ = back(da)
        dx = dq @ t(i["wq"]) + dk @ t(i["wk"]) + dv @ t(i["wv"])
        xt = t(i["x"])
        return dict(q=q, k=k, v=v, a=a, y=a @ i["wo"], da=da, dq=dq, dk=dk, dv=dv, dx=dx,
                    dwq=xt @ dq, dwk=xt @ dk, dwv=xt @ dv, dwo=t(a) @ i["g"])
    if kind in ("attention", "composed"):
        out, back = _attention64(c, i["q"], i["k"], i["v"])
        dq, dk, dv, p = back(i["g"])
        r = dict(out=out, dq=dq, dk=dk, dv=dv)
        if kind == "composed":
            # split_heads puts the heads outermost: [heads][batch][seq]
            s = c["seq"]
            r["p"] = p.transpose(0, 1).reshape(c["batch"] * c["heads"], s, s)
        return r
    if kind == "cnn":
        pooled, argmax = _pool64(_conv64(i["x"], i["w1"], i["b1"], 1, 1))
        y = _conv64(pooled, i["w2"], i["b2"], 1, 1)
        dpooled, dw2, db2 = _conv64_backward(i["g"], i["pooled0"], i["w2"], 1, 1)
        m, s = c["c_mid"], c["size"]
        g1 = torch.zeros(c["batch"] * m * s * s, dtype=torch.float64, device="cuda")
        g1[i["argmax0"].long().reshape(-1)] = (dpooled * (i["pooled0"] > 0)).reshape(-1)
        _, dw1, db1 = _conv64_backward(g1.reshape(c["batch"], m, s, s), i["x0"], i["w1"], 1, 1)
        return dict(pooled=pooled, argmax=argmax, y=y, dpooled=dpooled, dw2=dw2, db2=db2,
                    dw1=dw1, db1=db1)
    dx, dw, db = _conv64_backward(i["g"], i["x"], i["w"], c["stride"], c["pad"])
    return dict(y=_conv64(i["x"], i["w"], i["b"], c["stride"], c["pad"]), dx=dx, dw=dw, db=db)


def _attention64(c, q, k, v):
    b, s, h, dh = c["batch"], c["seq"], c["heads"], c["d_head"]
    scale = 1 / math.sqrt(dh)
    split = lambda x: x.reshape(b, s, h, dh).permute(0, 2, 1, 3).contiguous()
    merge = lambda x: x.permute(0, 2, 1, 3).reshape(b * s, h * dh)
    tr = lambda x: x.transpose(2, 3).contiguous()
    qh, kh, vh = split(q), split(k), split(v)
    p = torch.softmax(qh @ tr(kh) * scale, 3)

    def back(g):
        gh = split(g)
        dp = gh @ tr(vh)
        ds = p * (dp - (p * dp).sum(3, keepdim=True)) * scale
        return merge(ds @ kh), merge(tr(ds) @ qh), merge(tr(p) @ gh), p

    return merge(p @ vh), back


def tolerance(case):
    """About four times what the library's f32 products and sums, in their
    own order, show against 64 bits: at most 1.1e-6 of the result's norm over
    the listed cases (the product of depth 4096; convolutions, and chains of
    products through a softmax or a LayerNorm, up to 8e-7)."""
    if case["kind"] == "cnn":  # two values of a pooling window an ulp apart
        return {"rel": 5e-6, "differ": 1e-4}
    return {"rel": 5e-6}
