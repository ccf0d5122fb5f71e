"""The work that the performance of this framework is measured on.

Each case is one pass through public entry points: the C-ABI calls a host makes
for one layer, forward and VJP, in the order the host core makes them (buffers
from oxi_hip_alloc, kept between passes), and for the smallest one a whole
training step through the Python surface. Sizes come from the benchmark's
configurations, the width sweep of the tests, or are generic; `draw` gives more
cases of the same ranges.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from oxitorch_amd import capi

F32, I64 = 4, 8
EPS = 1e-5
# activations: name of the forward/VJP pair, and the id the fused VJP takes
GELU_MODE = {"gelu_tanh": 0, "gelu_erf": 1}


def listed():
    return [
        # a whole training step of a tiny model from Python: embedding, layer
        # norm, gelu, rms norm, cross-entropy, backward, SGD with momentum;
        # launches, host work and copies are all there is
        {"name": "step_small", "kind": "step", "tokens": 64, "dim": 64, "vocab": 256},
        # one layer's norm on a few tokens (small batches, fine-tuning): latency
        {"name": "norm_small", "kind": "norm", "norm": "rms", "act": "none", "mode": "ref", "rows": 64, "cols": 768},
        # an odd model width of the width sweep, full derivative
        {"name": "norm_odd", "kind": "norm", "norm": "layer", "act": "none", "mode": "exact", "rows": 8192, "cols": 1003},
        # the benchmark's layer_norm + exact GELU block
        {"name": "norm_gelu_large", "kind": "norm", "norm": "layer", "act": "gelu_erf", "mode": "ref", "rows": 16384,
         "cols": 4096},
        # attention probabilities: batch 2, 12 heads, 1024 x 1024 scores
        {"name": "softmax_attention", "kind": "softmax", "log": False, "outer": 24576, "len": 1024, "inner": 1},
        # per-pixel class log-probabilities: the class dim is a middle one
        {"name": "softmax_channels", "kind": "softmax", "log": True, "outer": 16, "len": 150, "inner": 4096},
        # a language model's loss over the 50257-row vocabulary (odd rows)
        {"name": "xent_vocab_odd", "kind": "xent", "rows": 4096, "classes": 50257},
        # the benchmark's headline: the loss over 32000 classes with its gradient
        {"name": "xent_large", "kind": "xent", "rows": 8192, "classes": 32000},
        # a batch of tokens through the embedding table, both directions
        {"name": "embedding", "kind": "embed", "ids": 16384, "vocab": 50257, "dim": 768},
        # a bias gradient and the norm of a gradient (clipping)
        {"name": "grad_reduce", "kind": "reduce", "ops": "sum0,norm_flat", "rows": 16384, "cols": 768},
        # silu on the transposed view of a ragged sequence, positions added,
        # and back; 1023 = a sequence of 1024 less its last token
        {"name": "map_permuted", "kind": "map", "batch": 16, "tokens": 1023, "dim": 768},
        # one AdamW step over a 12-layer model's 148 parameter tensors
        {"name": "adamw_model", "kind": "adamw", "vocab": 50257, "positions": 1024, "dim": 768, "layers": 12},
    ]


def _log(rng, lo, hi):
    """A size in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A row width: half of them any number, half a multiple of 64 (or 4)."""
    w = _log(rng, lo, hi)
    if rng.random() < 0.5:
        m = 64 if w >= 128 else 4
        w = max(lo, min(hi, (w + m // 2) // m * m))
    return max(w, 1)


def draw(rng):
    kind = rng.choice(["norm", "norm", "norm", "softmax", "softmax", "xent", "xent", "embed", "reduce", "reduce", "map",
                       "adamw", "step"])
    if kind == "norm":
        cols = _width(rng, 16, 16384)
        return {"kind": kind, "norm": rng.choice(["rms", "layer"]),
                "act": rng.choice(["none", "none", "gelu_erf", "gelu_tanh", "silu"]),
                "mode": rng.choice(["ref", "exact"]), "rows": _log(rng, 1, min(32768, (1 << 26) // cols)), "cols": cols}
    if kind == "softmax":
        inner = 1 if rng.random() < 0.6 else _log(rng, 2, 16384)
        length = _width(rng, 2, min(65536, (1 << 25) // inner)) if inner == 1 else _log(rng, 2, min(4096, (1 << 25) // inner))
        return {"kind": kind, "log": rng.random() < 0.5, "outer": _log(rng, 1, max(1, min(65536, (1 << 25) // (inner * length)))),
                "len": length, "inner": inner}
    if kind == "xent":
        classes = _width(rng, 16, 131072)
        return {"kind": kind, "rows": _log(rng, 1, min(16384, (1 << 27) // classes)), "classes": classes}
    if kind == "embed":
        dim = _width(rng, 4, 1024)
        return {"kind": kind, "ids": _log(rng, 1, min(131072, (1 << 26) // dim)), "vocab": _log(rng, 64, 65536), "dim": dim}
    if kind == "reduce":
        cols = _width(rng, 1, 65536)
        ops = rng.sample(["sum0", "mean1", "max1", "argmax1", "norm_flat", "sum_flat"], 2)
        return {"kind": kind, "ops": ",".join(ops), "rows": _log(rng, 1, min(65536, (1 << 25) // cols)), "cols": cols}
    if kind == "map":
        dim = _width(rng, 8, 2048)
        tokens = _width(rng, 1, 2048)
        return {"kind": kind, "batch": _log(rng, 1, max(1, min(64, (1 << 25) // (dim * tokens)))), "tokens": tokens, "dim": dim}
    if kind == "adamw":
        return {"kind": kind, "vocab": _log(rng, 256, 50257), "positions": _log(rng, 64, 1024), "dim": 64 * rng.randint(1, 12),
                "layers": rng.randint(1, 12)}
    return {"kind": "step", "tokens": _log(rng, 8, 512), "dim": _width(rng, 16, 256), "vocab": _log(rng, 64, 2048)}


# ---- inputs -----------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, scale=1.0, shift=0.0):
    t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return t.mul_(scale).add_(shift)


def _zipf_p(vocab):
    """Token frequencies: 1/rank^1.1 over the vocabulary."""
    p = np.arange(1, vocab + 1, dtype=np.float64) ** -1.1
    return p / p.sum()


def _params(case):
    """Parameter sizes of a transformer with tied embeddings (the benchmark's list)."""
    h = case["dim"]
    block = [h, h, 3 * h * h, 3 * h, h * h, h, h, h, 4 * h * h, 4 * h, 4 * h * h, h]
    return [case["vocab"] * h, case["positions"] * h] + block * case["layers"] + [h, h]


def inputs(case, seed):
    """The case's input tensors on the GPU, from the seed alone."""
    k, g = case["kind"], _gen(seed)
    if k == "norm":
        r, c = case["rows"], case["cols"]
        return {"x": _randn(g, r, c, shift=0.1), "w": _randn(g, c, scale=0.1, shift=1.0), "b": _randn(g, c, scale=0.1),
                "g": _randn(g, r, c)}
    if k == "softmax":
        s = (case["outer"], case["len"], case["inner"])
        return {"x": _randn(g, *s, scale=2.0), "g": _randn(g, *s)}
    if k == "xent":
        n, c = case["rows"], case["classes"]
        return {"x": _randn(g, n, c, scale=2.0), "t": torch.randint(0, c, (n,), generator=g, device="cuda")}
    if k == "embed":
        n, v, d = case["ids"], case["vocab"], case["dim"]
        cdf = torch.from_numpy(np.cumsum(_zipf_p(v))).cuda()
        u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
        order = torch.randperm(v, generator=g, device="cuda")
        ids = order[torch.searchsorted(cdf, u).clamp_(max=v - 1)]
        return {"W": _randn(g, v, d, scale=0.05), "ids": ids, "g": _randn(g, n, d, scale=0.01)}
    if k == "reduce":
        return {"x": _randn(g, case["rows"], case["cols"], shift=0.5)}
    if k == "map":
        s = (case["batch"], case["tokens"], case["dim"])
        return {"x": _randn(g, *s), "pos": _randn(g, *s[1:], scale=0.1), "g": _randn(g, *s)}
    if k == "adamw":
        n = sum(_params(case))
        return {"p": _randn(g, n, scale=0.05), "g": _randn(g, n, scale=0.01), "m": _randn(g, n, scale=0.003),
                "v": _randn(g, n, scale=0.01).square_()}
    n, d, v = case["tokens"], case["dim"], case["vocab"]
    return {"W": _randn(g, v, d, scale=0.5), "lw": _randn(g, d, scale=0.1, shift=1.0), "lb": _randn(g, d, scale=0.1),
            "rw": _randn(g, d, scale=0.1, shift=1.0), "ids": torch.randint(0, v, (n,), generator=g, device="cuda"),
            "t": torch.randint(0, d, (n,), generator=g, device="cuda")}


class _Buffer:
    """An HBM buffer of the library, also seen as a torch tensor (no copy)."""

    def __init__(self, shape, dtype=torch.float32):
        shape = tuple(int(s) for s in shape)
        self.array = capi.DeviceArray(shape, np.int64 if dtype == torch.int64 else np.float32)
        self.ptr = self.array.ptr
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i8" if dtype == torch.int64 else "<f4",
                                         "data": (self.ptr, False), "version": 2}
        self.t = torch.as_tensor(self, device="cuda")


def _upload(tensor):
    b = _Buffer(tensor.shape, tensor.dtype)
    b.t.copy_(tensor)
    return b


def prepare(case, seed):
    torch.cuda.init()
    capi.init(torch.cuda.current_device())
    k = case["kind"]
    s = {"case": case}
    if k == "step":
        import oxitorch_amd as ox
        from oxitorch_amd import nn, optim

        h = {name: t.cpu().numpy() for name, t in inputs(case, seed).items()}
        s["params"] = [ox.from_numpy(h[n], True) for n in ("W", "lw", "lb", "rw")]
        s["opt"] = optim.Sgd(s["params"], lr=0.01, momentum=0.9)
        s["ids"], s["targets"] = h["ids"], h["t"]
        s["F"] = nn.functional
        return s
    for name, t in inputs(case, seed).items():
        s[name] = _upload(t)
    new = lambda *shape: _Buffer(shape)  # noqa: E731
    arr = capi._i64arr
    if k == "norm":
        r, c = case["rows"], case["cols"]
        s.update(y=new(r, c), dx=new(r, c), rstd=new(r), dw=new(c))
        if case["norm"] == "layer":
            s.update(mean=new(r), db=new(c))
        if case["act"] != "none":
            s.update(a=new(r, c))
            if not _fused(case):
                s.update(dy=new(r, c))
        s["sh"], s["st"] = arr((r, c)), arr((c, 1))
    elif k == "softmax":
        shape = (case["outer"], case["len"], case["inner"])
        s.update(y=new(*shape), dx=new(*shape))
    elif k == "xent":
        n, c = case["rows"], case["classes"]
        s.update(loss=new(1), lse=new(n), dx=new(n, c), one=_upload(torch.ones(1, device="cuda")))
    elif k == "embed":
        s.update(y=new(case["ids"], case["dim"]), dW=new(case["vocab"], case["dim"]))
    elif k == "reduce":
        r, c = case["rows"], case["cols"]
        s["calls"] = []
        for op in case["ops"].split(","):
            kind, where = (op[:-5], "flat") if op.endswith("_flat") else (op[:-1], int(op[-1]))
            shape, dim = ((r * c,), 0) if where == "flat" else ((r, c), where)
            out = new(1) if where == "flat" else new(c if dim == 0 else r)
            strides = (1,) if where == "flat" else (c, 1)
            s["calls"].append((op, capi.REDUCE.index(kind), arr(strides), arr(shape), len(shape), dim, out))
    elif k == "map":
        B, T, H = case["batch"], case["tokens"], case["dim"]
        s.update(y=new(B, H, T), r=new(B, T, H), dpos=new(T, H), dx=new(B, T, H))
        s["bht"], s["bth"] = arr((B, H, T)), arr((B, T, H))
        s["x_view"], s["y_st"] = arr((T * H, 1, H)), arr((H * T, T, 1))       # x.permute(0, 2, 1); y row-major
        s["y_view"], s["pos_st"] = arr((H * T, 1, T)), arr((0, H, 1))         # y.permute(0, 2, 1); pos over the batch
        s["r_st"] = arr((T * H, H, 1))
    elif k == "adamw":
        n = sum(_params(case))
        s.update(q=new(n))
        rows, off = [], 0
        for m in _params(case):
            o = off * F32
            rows.append((s["p"].ptr + o, s["g"].ptr + o, s["m"].ptr + o, s["v"].ptr + o, s["q"].ptr + o, m, 10))
            off += m
        s["slices"] = capi.slice_array(capi.AdamWSlice, rows)
        s["count"] = len(rows)
    torch.cuda.synchronize()
    return s


def _fused(case):
    """The fused norm + activation VJP takes rows of up to 8192 floats, a multiple of 4."""
    return case["act"] != "none" and case["cols"] % 4 == 0 and case["cols"] <= 8192


def _one_pass(case):
    """The one-pass cross-entropy takes up to 65536 classes, a multiple of 4."""
    return case["classes"] % 4 == 0 and case["classes"] <= 65536


def run(s):
    case = s["case"]
    return _RUN[case["kind"]](s, case)


def _run_norm(s, case):
    call, p = capi.call, lambda n: s[n].ptr
    r, c, act, mode = case["rows"], case["cols"], case["act"], capi.NORM_VJP[case["mode"]]
    layer = case["norm"] == "layer"
    names = ["y", "rstd", "dx", "dw"]
    if layer:
        names += ["mean", "db"]
        call("oxi_layer_norm_fwd", p("x"), p("w"), p("b"), p("y"), p("mean"), p("rstd"), r, c, EPS)
    else:
        call("oxi_rms_norm_fwd", p("x"), p("w"), p("y"), p("rstd"), r, c, EPS)
    up = "g"
    if act != "none":
        names.append("a")
        if act == "silu":
            call("oxi_silu_fwd", p("y"), s["st"], p("a"), s["st"], s["sh"], 2)
        else:
            call("oxi_gelu_fwd", p("y"), s["st"], p("a"), s["st"], s["sh"], 2, GELU_MODE[act])
        if _fused(case):
            if layer:
                call("oxi_layer_norm_act_bwd", p("x"), p("w"), p("b"), p("mean"), p("rstd"), p("g"), capi.ACT[act],
                     None, p("dx"), p("dw"), p("db"), r, c, mode)
            else:
                call("oxi_rms_norm_act_bwd", p("x"), p("w"), p("rstd"), p("g"), capi.ACT[act], None, p("dx"), p("dw"),
                     r, c, mode)
            return {n: s[n].t for n in names}
        if act == "silu":
            call("oxi_silu_bwd", p("y"), s["st"], p("g"), s["st"], p("dy"), s["st"], s["sh"], 2)
        else:
            call("oxi_gelu_bwd", p("y"), s["st"], p("g"), s["st"], p("dy"), s["st"], s["sh"], 2, GELU_MODE[act])
        names.append("dy")
        up = "dy"
    if layer:
        call("oxi_layer_norm_bwd", p("x"), p("w"), p("mean"), p("rstd"), p(up), p("dx"), p("dw"), p("db"), r, c, mode)
    else:
        call("oxi_rms_norm_bwd", p("x"), p("w"), p("rstd"), p(up), p("dx"), p("dw"), r, c, mode)
    return {n: s[n].t for n in names}


def _run_softmax(s, case):
    pre = "oxi_log_softmax" if case["log"] else "oxi_softmax"
    dims = (case["outer"], case["len"], case["inner"])
    capi.call(pre + "_fwd", s["x"].ptr, s["y"].ptr, *dims)
    capi.call(pre + "_bwd", s["y"].ptr, s["g"].ptr, s["dx"].ptr, *dims)
    return {"y": s["y"].t, "dx": s["dx"].t}


def _run_xent(s, case):
    n, c = case["rows"], case["classes"]
    if _one_pass(case):
        capi.call("oxi_cross_entropy_fwd_grad", s["x"].ptr, s["t"].ptr, s["loss"].ptr, s["lse"].ptr, s["dx"].ptr, n, c)
    else:
        capi.call("oxi_cross_entropy_fwd", s["x"].ptr, s["t"].ptr, s["loss"].ptr, s["lse"].ptr, n, c)
        capi.call("oxi_cross_entropy_bwd", s["x"].ptr, s["t"].ptr, s["lse"].ptr, s["one"].ptr, s["dx"].ptr, n, c)
    return {"loss": s["loss"].t, "lse": s["lse"].t, "dx": s["dx"].t}


def _run_embed(s, case):
    n, v, d = case["ids"], case["vocab"], case["dim"]
    plan = ctypes.c_void_p()
    capi.call("oxi_index_select_bwd_plan", s["ids"].ptr, n, v, ctypes.byref(plan))
    capi.call("oxi_embedding_fwd", s["W"].ptr, s["ids"].ptr, n, v, d, s["y"].ptr)
    capi.call("oxi_index_select_bwd_apply", plan, s["g"].ptr, 1, d, s["dW"].ptr)
    capi.call("oxi_index_select_bwd_plan_free", plan)
    return {"y": s["y"].t, "dW": s["dW"].t}


def _run_reduce(s, case):
    out = {}
    for op, kind, strides, shape, ndim, dim, buf in s["calls"]:
        capi.call("oxi_reduce", kind, s["x"].ptr, strides, shape, ndim, dim, buf.ptr)
        out[op] = buf.t
    return out


def _run_map(s, case):
    p = lambda n: s[n].ptr  # noqa: E731
    capi.call("oxi_silu_fwd", p("x"), s["x_view"], p("y"), s["y_st"], s["bht"], 3)
    capi.call("oxi_binary", 0, p("y"), s["y_view"], p("pos"), s["pos_st"], p("r"), s["r_st"], s["bth"], 3)
    capi.call("oxi_reduce", 0, p("g"), s["r_st"], s["bth"], 3, 0, p("dpos"))
    capi.call("oxi_silu_bwd", p("x"), s["x_view"], p("g"), s["x_view"], p("dx"), s["x_view"], s["bht"], 3)
    return {n: s[n].t for n in ("y", "r", "dpos", "dx")}


def _run_adamw(s, case):
    capi.call("oxi_adamw_step_multi", s["slices"], s["count"], *HYPER)
    return {n: s[n].t for n in ("q", "m", "v")}


HYPER = (6e-4, 0.9, 0.95, 1e-8, 0.1, 1)  # lr, betas, eps, decoupled decay


def _run_step(s, case):
    F, (W, lw, lb, rw) = s["F"], s["params"]
    s["opt"].zero_grad()
    h = F.gelu(F.layer_norm(F.embedding(s["ids"], W), lw, lb))
    loss = F.cross_entropy(F.rms_norm(h, rw), s["targets"])
    loss.backward()
    s["opt"].step()
    return {"loss": loss.item(), "W": W.numpy(), "lw": lw.numpy(), "lb": lb.numpy(), "rw": rw.numpy()}


_RUN = {"norm": _run_norm, "softmax": _run_softmax, "xent": _run_xent, "embed": _run_embed, "reduce": _run_reduce,
        "map": _run_map, "adamw": _run_adamw, "step": _run_step}


# ---- what a pass cannot do without -----------------------------------------------

def work(case):
    """Each call's inputs read once and its outputs written once."""
    k = case["kind"]
    if k == "norm":
        e = case["rows"] * case["cols"] * F32
        act = case["act"] != "none"
        # forward 2 crossings, activation 2, VJP 3 (node by node 6)
        n = 5 if not act else 7 if _fused(case) else 10
        return {"bytes": n * e + 8 * case["rows"] * F32 + 5 * case["cols"] * F32, "flops": 0}
    if k == "softmax":
        return {"bytes": 5 * case["outer"] * case["len"] * case["inner"] * F32, "flops": 0}
    if k == "xent":
        e = case["rows"] * case["classes"] * F32
        return {"bytes": (2 if _one_pass(case) else 3) * e + 24 * case["rows"], "flops": 0}
    if k == "embed":
        n, v, d = case["ids"], case["vocab"], case["dim"]
        rows = float(np.sum(-np.expm1(n * np.log1p(-np.minimum(_zipf_p(v), 1 - 1e-12)))))  # distinct rows expected
        return {"bytes": (rows + 2 * n + v) * d * F32 + 2 * n * I64, "flops": 0}
    if k == "reduce":
        r, c = case["rows"], case["cols"]
        return {"bytes": sum(r * c + (1 if op.endswith("flat") else c if op.endswith("0") else r)
                             for op in case["ops"].split(",")) * F32, "flops": 0}
    if k == "map":
        e = case["batch"] * case["tokens"] * case["dim"]
        return {"bytes": (8 * e + 2 * case["tokens"] * case["dim"]) * F32, "flops": 0}
    if k == "adamw":
        return {"bytes": 7 * sum(_params(case)) * F32, "flops": 0}
    n, d, v = case["tokens"], case["dim"], case["vocab"]
    # activations both ways, the table's gradient, and the update (read and
    # write weight and momentum) with the weights' way back to the host
    return {"bytes": (25 * n * d + 7 * v * d + 24 * d) * F32, "flops": 0}


def tolerance(case):
    """About four times what the kernels' sums differ by from their float64
    values (measured), per kind: 32-bit arithmetic throughout."""
    k = case["kind"]
    if k == "reduce":
        # sequential 32-bit sums: 1.9e-5 off over 12.6M values, 1.6e-6 over 16384
        return {"rel": 8e-5 if "flat" in case["ops"] else 1e-5}
    if k == "xent":
        # a row whose target holds nearly all the probability has a small loss
        return {"rel": 4e-6}
    return {"rel": 2e-6 if k == "norm" else 1e-6}


# ---- the same in 64 bits -----------------------------------------------------------

def _norm64(x, w, b, layer, eps=EPS):
    mu = x.mean(-1, keepdim=True) if layer else 0.0
    xc = x - mu
    inv = 1.0 / torch.sqrt((xc * xc).mean(-1, keepdim=True) + eps)
    xh = xc * inv
    return xh * w + (b if layer else 0.0), xh, inv, mu


def _norm_vjp64(xh, inv, w, dy, layer, mode):
    gw = dy * w
    if mode == "ref":  # the inverse deviation held constant
        dx = gw * inv
        return dx - dx.mean(-1, keepdim=True) if layer else dx
    dx = gw - xh * (gw * xh).mean(-1, keepdim=True)
    if layer:
        dx = dx - gw.mean(-1, keepdim=True)
    return dx * inv


def _act64(name, y):
    """The activation's value and derivative."""
    if name == "silu":
        sg = torch.sigmoid(y)
        return y * sg, sg * (1 + y * (1 - sg))
    if name == "gelu_erf":
        cdf = 0.5 * torch.special.erfc(-y / math.sqrt(2.0))
        return y * cdf, cdf + y * torch.exp(-0.5 * y * y) / math.sqrt(2 * math.pi)
    c = math.sqrt(2 / math.pi)
    th = torch.tanh(c * (y + 0.044715 * y ** 3))
    return 0.5 * y * (1 + th), 0.5 * (1 + th) + 0.5 * y * (1 - th * th) * c * (1 + 3 * 0.044715 * y * y)


def exact(case, seed):
    k = case["kind"]
    i = {n: t.double() if t.dtype == torch.float32 else t for n, t in inputs(case, seed).items()}
    if k == "norm":
        layer = case["norm"] == "layer"
        y, xh, inv, mu = _norm64(i["x"], i["w"], i["b"], layer)
        out = {"y": y, "rstd": inv[:, 0]}
        dy = i["g"]
        if case["act"] != "none":
            out["a"], d = _act64(case["act"], y)
            dy = dy * d
            if not _fused(case):
                out["dy"] = dy
        out["dx"] = _norm_vjp64(xh, inv, i["w"], dy, layer, case["mode"])
        out["dw"] = (dy * xh).sum(0)
        if layer:
            out["mean"], out["db"] = mu[:, 0], dy.sum(0)
        return out
    if k == "softmax":
        if case["log"]:
            y = torch.log_softmax(i["x"], 1)
            return {"y": y, "dx": i["g"] - y.exp() * i["g"].sum(1, keepdim=True)}
        y = torch.softmax(i["x"], 1)
        return {"y": y, "dx": y * (i["g"] - (i["g"] * y).sum(1, keepdim=True))}
    if k == "xent":
        lse = torch.logsumexp(i["x"], 1)
        picked = i["x"].gather(1, i["t"][:, None])[:, 0] - lse
        d = torch.exp(i["x"] - lse[:, None])
        d.scatter_add_(1, i["t"][:, None], torch.full_like(lse, -1.0)[:, None])
        return {"loss": -picked.mean().reshape(1), "lse": lse, "dx": d / case["rows"]}
    if k == "embed":
        dW = torch.zeros_like(i["W"]).index_add_(0, i["ids"], i["g"])
        return {"y": i["W"][i["ids"]], "dW": dW}
    if k == "reduce":
        x = i["x"]
        f = {"sum0": lambda: x.sum(0), "mean1": lambda: x.mean(1), "max1": lambda: x.max(1).values,
             "argmax1": lambda: x.argmax(1).double(), "norm_flat": lambda: x.square().sum().sqrt().reshape(1),
             "sum_flat": lambda: x.sum().reshape(1)}
        return {op: f[op]() for op in case["ops"].split(",")}
    if k == "map":
        x, g = i["x"], i["g"]
        a, d = _act64("silu", x)
        return {"y": a.permute(0, 2, 1).contiguous(), "r": a + i["pos"], "dpos": g.sum(0), "dx": d * g}
    if k == "adamw":
        # the hyperparameters as the call takes them: 32-bit, the bias
        # corrections of step 10 formed from them
        lr, b1, b2, eps, wd = (float(np.float32(h)) for h in HYPER[:5])
        m = b1 * i["m"] + (1 - b1) * i["g"]
        v = b2 * i["v"] + (1 - b2) * i["g"] ** 2
        step = lr * (m / (1 - b1 ** 10)) / (torch.sqrt(v / (1 - b2 ** 10)) + eps)
        return {"q": i["p"] - step - lr * wd * i["p"], "m": m, "v": v}
    e = i["W"][i["ids"]]
    h, xh, inv, _ = _norm64(e, i["lw"], i["lb"], True, 1e-5)
    a, da = _act64("gelu_tanh", h)
    z, ah, inv2, _ = _norm64(a, i["rw"], None, False, 1e-6)
    n = case["tokens"]
    lse = torch.logsumexp(z, 1)
    loss = (lse - z.gather(1, i["t"][:, None])[:, 0]).mean()
    dz = torch.exp(z - lse[:, None])
    dz.scatter_add_(1, i["t"][:, None], torch.full_like(lse, -1.0)[:, None])
    dz = dz / n
    dh = _norm_vjp64(ah, inv2, i["rw"], dz, False, "ref") * da
    de = _norm_vjp64(xh, inv, i["lw"], dh, True, "ref")
    dW = torch.zeros_like(i["W"]).index_add_(0, i["ids"], de)
    lr = float(np.float32(0.01))
    return {"loss": float(loss), "W": i["W"] - lr * dW, "lw": i["lw"] - lr * (dh * xh).sum(0),
            "lb": i["lb"] - lr * dh.sum(0), "rw": i["rw"] - lr * (dz * ah).sum(0)}
