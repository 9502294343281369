"""The work a program gives this package, as cases that can be timed and compared.

Every case goes through the package's public entry points (the modules of
``yggdrasil_amd.layers``, ``ops.geom_matmul`` and the routing functions) at sizes
of this repository's configurations, its tests, or generic ones.  ``listed`` holds
the cases by name, ``draw`` gives others of the same ranges, ``exact`` computes a
case's outputs in float64 with plain torch.

Kinds of case:
  layer        CliffordMoELayer: routing, the two expert products, combine (inference)
  block        CliffordMoEBlockFFN: x + moe(ffn_norm(x)) (inference)
  train        CliffordMoELayer forward, backward and a gradient-descent update of its weights
  linear       CliffordLinear on its own
  geom_matmul  the geometric matrix product of two multivector matrices (fp32)
  route        routing, dispatch and weighted combine of one payload
"""

from __future__ import annotations

import math

import torch

import yggdrasil_amd
from yggdrasil_amd import ops

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def _moe(kind, N, d, F, E, k, dtype, fmt="", router="logits", load="even", act="gelu", **more):
    return dict(kind=kind, N=N, d=d, F=F, E=E, k=k, dtype=dtype, fmt=fmt, router=router, load=load, act=act, **more)


def listed():
    return [
        # one decode step of a quantized model: 64 sequences, one token each, int8 expert weights
        dict(_moe("layer", 64, 128, 512, 32, 2, "bf16", fmt="int8_pauli"), name="decode_int8"),
        # one decode step of the bf16 12-layer model's layer at a small batch: the weights of the experts
        # that 16 tokens reach are read once each
        dict(_moe("layer", 16, 256, 1024, 64, 2, "bf16", router="energy"), name="decode_bf16"),
        # the smallest model's layer on a short batch, fp32, with the CliffordLinear head as its router
        dict(_moe("layer", 256, 64, 256, 8, 2, "f32", router="clifford_head"), name="small_f32"),
        # a prompt of odd length through widths that are no power of two
        dict(_moe("layer", 1500, 100, 300, 12, 3, "bf16", act="sigmoid"), name="ragged_bf16"),
        # prefill of a large prompt batch, expert load skewed by Zipf's law
        dict(_moe("layer", 8192, 128, 512, 32, 4, "bf16", load="zipf"), name="prefill_bf16"),
        # prompts of a model whose expert weights are held in int8 (larger than a decode batch)
        dict(_moe("layer", 2048, 128, 512, 32, 2, "bf16", fmt="int8"), name="prefill_int8"),
        # the FFN half of one block of the 12-layer model, mildly skewed experts
        dict(_moe("block", 4096, 256, 1024, 64, 2, "bf16", load="skewed"), name="block_bf16"),
        # a training step of the smallest model's layer
        dict(_moe("train", 256, 64, 256, 8, 2, "f32", router="energy"), name="train_small"),
        # a training step on a large batch, expert load skewed by Zipf's law
        dict(_moe("train", 8192, 128, 512, 32, 4, "f32", load="zipf"), name="train_large"),
        # the module CliffordLinear: an up projection of 4 x 1024 tokens
        dict(kind="linear", N=4096, d_in=128, d_out=512, dtype="f32", bias=True, name="linear_f32"),
        # the operator that the reference's layers are made of, at an up projection's sizes
        dict(kind="geom_matmul", M=512, K=128, N=8192, name="geom_matmul"),
        # routing, dispatch and combine alone (a caller with its own expert computation)
        dict(kind="route", N=16384, d=128, E=16, k=2, dtype="f32", name="route_combine"),
    ]


def _log_int(rng, lo, hi, odd=0.4):
    """A whole number of [lo, hi], spread over its logarithm; else rounded to a multiple of 8."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() >= odd:
        v = max(8, (v + 4) // 8 * 8)
    return min(max(v, lo), hi)


def _even(v):
    return v + v % 2


def draw(rng):
    kind = rng.choice(["decode_int8", "decode_bf16", "layer_f32", "prefill_bf16", "prefill_bf16", "prefill_int8",
                       "block", "train", "linear", "geom_matmul", "route"])
    act = rng.choice(["gelu", "gelu", "relu", "sigmoid"])
    E = rng.choice([4, 8, 12, 16, 32, 64])
    k = rng.choice([1, 2, 2, 3, 4])
    router = rng.choice(["logits", "energy"])
    load = rng.choice(["even", "skewed", "zipf"])
    if kind == "decode_int8":
        return _moe("layer", _log_int(rng, 1, 128), rng.choice([64, 96, 100, 128]), _log_int(rng, 128, 1024), E,
                    min(k, 3), "bf16", fmt="int8_pauli", router=router, act=act)
    if kind == "decode_bf16":
        return _moe("layer", _log_int(rng, 1, 128), rng.choice([64, 128, 200, 256]), _even(_log_int(rng, 128, 1024)),
                    E, min(k, 3), "bf16", router=router, act=act)
    if kind == "layer_f32":
        return _moe("layer", _log_int(rng, 16, 2048), _log_int(rng, 32, 128), _log_int(rng, 64, 512), E, k, "f32",
                    router=rng.choice(["logits", "energy", "clifford_head"]), act=act)
    if kind == "prefill_bf16":
        return _moe("layer", _log_int(rng, 256, 8192), _even(_log_int(rng, 64, 256)), _even(_log_int(rng, 128, 512)),
                    E, k, "bf16", router=router, load=load, act=act)
    if kind == "prefill_int8":
        return _moe("layer", _log_int(rng, 256, 4096), _log_int(rng, 64, 128), _log_int(rng, 128, 512), E, k, "bf16",
                    fmt="int8", router=router, load=load, act=act)
    if kind == "block":
        return _moe("block", _log_int(rng, 128, 4096), _even(_log_int(rng, 64, 256)), _even(_log_int(rng, 128, 512)),
                    E, k, rng.choice(["bf16", "bf16", "f32"]), router=router, load=load, act=act)
    if kind == "train":
        return _moe("train", _log_int(rng, 128, 4096), _log_int(rng, 32, 128), _log_int(rng, 64, 512),
                    min(E, 32), k, "f32", router=router, load=load, act=act)
    if kind == "linear":
        return dict(kind="linear", N=_log_int(rng, 16, 8192), d_in=_log_int(rng, 32, 256), d_out=_log_int(rng, 32, 512),
                    dtype=rng.choice(["f32", "f32", "bf16"]), bias=rng.random() < 0.7)
    if kind == "geom_matmul":
        return dict(kind="geom_matmul", M=_log_int(rng, 16, 512), K=_log_int(rng, 16, 512), N=_log_int(rng, 64, 8192))
    return dict(kind="route", N=_log_int(rng, 64, 32768), d=_log_int(rng, 32, 256), E=E, k=k,
                dtype=rng.choice(["f32", "bf16"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _inputs(c, seed):
    """A case's input tensors on the GPU, from the seed alone."""
    dev = "cuda"
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))

    def rn(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)

    if c["kind"] == "geom_matmul":
        return dict(a=rn(c["M"], c["K"], 8) / (8.0 * c["K"]) ** 0.5, b=rn(c["K"], c["N"], 8))
    dt = DTYPES[c["dtype"]]
    if c["kind"] == "linear":
        t = dict(x=rn(c["N"], c["d_in"], 8).to(dt), w=rn(c["d_out"], c["d_in"], 8) / (8.0 * c["d_in"]) ** 0.5)
        if dt == torch.bfloat16:
            t["w"] = t["w"].bfloat16().float()
        t["b"] = 0.1 * rn(c["d_out"], 8) if c["bias"] else None
        return t
    N, d, E, k = c["N"], c["d"], c["E"], c["k"]
    if c["kind"] == "route":
        return dict(x=rn(N, d, 8).to(dt), logits=rn(N, E))
    F = c["F"]
    x = rn(N, d, 8)
    if c["router"] == "energy":  # tokens whose energy lies in other grades from one to the next
        grade = torch.tensor([0, 1, 1, 1, 2, 2, 2, 3], device=dev)
        x = x * torch.exp(0.7 * rn(N, 1, 4))[..., grade]
    t = dict(x=x.to(dt))
    t["w_up"], t["w_down"] = rn(E, F, d, 8) / (8.0 * d) ** 0.5, rn(E, d, F, 8) / (8.0 * F) ** 0.5
    if dt == torch.bfloat16 and not c["fmt"].startswith("int8"):  # a bf16 model's weights
        t["w_up"], t["w_down"] = t["w_up"].bfloat16().float(), t["w_down"].bfloat16().float()
    t["b_up"], t["b_down"] = 0.1 * rn(E, F, 8), 0.1 * rn(E, d, 8)
    if c["router"] == "energy":
        t["router_weight"], t["router_bias"] = 2.0 * rn(E, 4), 0.1 * rn(E)
    elif c["router"] == "clifford_head":
        t["head_weight"] = rn(E, d, 8) / (8.0 * d) ** 0.5
    elif c["load"] == "zipf":  # k experts a token without replacement, the r-th most likely by r^-1.2
        ranking = torch.randperm(E, generator=g, device=dev)
        p = torch.arange(1, E + 1, device=dev, dtype=torch.float64) ** -1.2
        chosen = torch.multinomial((p / p.sum()).float().expand(N, E), k, replacement=False, generator=g)
        lg = 0.1 * rn(N, E)
        lg.scatter_add_(1, ranking[chosen], (k - torch.arange(k, device=dev, dtype=torch.float32)).expand(N, k))
        t["logits"] = lg
    else:
        t["logits"] = rn(N, E) + (0.5 * rn(E)[None, :] if c["load"] == "skewed" else 0.0)
    if c["kind"] == "block":
        t["gamma"], t["beta"] = 0.1 * rn(d, 8), 0.1 * rn(d, 8)
        t["gamma"][:, 0] += 1.0
    if c["kind"] == "train":
        t["grad"] = rn(N, d, 8)
    return t


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    if c["kind"] == "geom_matmul":
        return dict(c=c, a=t["a"], b=t["b"])
    if c["kind"] == "route":
        return dict(c=c, x=t["x"], logits=t["logits"])
    if c["kind"] == "linear":
        with torch.device("cuda"):
            lin = yggdrasil_amd.CliffordLinear(c["d_in"], c["d_out"], bias=c["bias"], dtype=DTYPES[c["dtype"]])
        with torch.no_grad():
            lin.weight.copy_(t["w"])
            if c["bias"]:
                lin.bias.copy_(t["b"])
        B = 4 if c["N"] % 4 == 0 else 1
        st = dict(c=c, m=lin, x=t["x"].reshape(B, c["N"] // B, c["d_in"], 8))
        with torch.no_grad():
            lin(st["x"][:, :1].contiguous())  # the weights laid out, as any program's second call finds them
        return st
    cfg = yggdrasil_amd.MoEHLMConfig(d_model=c["d"], d_ff=c["F"], n_experts=c["E"], top_k=c["k"], activation=c["act"],
                                     dtype=DTYPES[c["dtype"]], weight_format=c["fmt"] or None, router=c["router"])
    with torch.device("cuda"):
        m = (yggdrasil_amd.CliffordMoEBlockFFN if c["kind"] == "block" else yggdrasil_amd.CliffordMoELayer)(cfg)
    moe = m.moe if c["kind"] == "block" else m
    moe.load_reference_weights(w_up=t["w_up"], b_up=t["b_up"], w_down=t["w_down"], b_down=t["b_down"],
                               router_weight=t.get("router_weight"), router_bias=t.get("router_bias"),
                               head_weight=t.get("head_weight"))
    if c["kind"] == "block":
        with torch.no_grad():
            m.ffn_norm.gamma.copy_(t["gamma"])
            m.ffn_norm.beta.copy_(t["beta"])
    moe.prepare()
    B = 4 if c["N"] % 4 == 0 else 1
    x = t["x"].reshape(B, c["N"] // B, c["d"], 8)
    return dict(c=c, m=m, x=x, logits=t.get("logits"),
                grad=t["grad"].reshape(x.shape) if c["kind"] == "train" else None)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

LEARNING_RATE = 1e-6


def run(state):
    c = state["c"]
    if c["kind"] == "geom_matmul":
        return ops.geom_matmul(state["a"], state["b"])
    if c["kind"] == "route":
        r = ops.route(state["logits"], c["k"])
        rows = ops.dispatch(state["x"], r)
        out = ops.combine(rows, r)
        return dict(idx=r.topk_idx, w=r.topk_w, counts=r.counts, perm=r.perm, rows=rows, out=out)
    m, x = state["m"], state["x"]
    if c["kind"] == "linear":
        with torch.no_grad():
            return m(x)
    if c["kind"] == "block":
        with torch.no_grad():
            return m(x, logits=state["logits"])
    if c["kind"] == "layer":
        with torch.no_grad():
            return m.moe_forward(x, logits=state["logits"])
    # a training step: forward with the balance loss reported, gradients, gradient descent
    x = x.detach().requires_grad_(True)
    out, aux = m(x, logits=state["logits"])
    params = (m.w_up, m.b_up, m.w_down, m.b_down)
    grads = torch.autograd.grad(out, (x, *params), state["grad"])
    with torch.no_grad():
        for p, g in zip(params, grads[1:]):
            p.add_(g, alpha=-LEARNING_RATE)
    return dict(out=out.detach(), aux=aux, dx=grads[0], dw_up=grads[1], db_up=grads[2], dw_down=grads[3],
                db_down=grads[4])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    c = case
    mac = 2 * 32  # a geometric product as a product of complex 2x2 matrices: 32 real multiply-adds
    if c["kind"] == "geom_matmul":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=32 * (M * K + K * N + M * N), flops=mac * M * K * N)
    es = 4 if c["dtype"] == "f32" else 2
    if c["kind"] == "linear":
        n, i, o = c["N"], c["d_in"], c["d_out"]
        return dict(bytes=8 * es * (n * i + i * o + n * o), flops=mac * n * i * o)
    N, d, E, k = c["N"], c["d"], c["E"], c["k"]
    row = 8 * d * es
    if c["kind"] == "route":  # logits, payload in, grouped rows out and in, payload out, routing arrays
        return dict(bytes=4 * N * E + (2 + 2 * k) * N * row + 16 * N * k, flops=2 * 8 * d * N * k)
    P, F = N * k, c["F"]
    flops = 2 * mac * P * d * F
    touched = E * (1.0 - (1.0 - k / E) ** N)
    wbytes = (1 if c["fmt"].startswith("int8") else es) * 8 * 2 * d * F * touched
    io = 2 * N * row + (4 * N * E if c["router"] == "logits" else 0)
    if c["kind"] == "train":  # backward: two products and two weight gradients; weights read, gradients and weights out
        return dict(bytes=2 * io + 3 * wbytes, flops=3 * flops)
    return dict(bytes=io + wbytes, flops=flops)


def tolerance(case):
    c = case
    if c["kind"] == "route":  # copies, and at most a few 32-bit products and sums in a fixed order
        return dict(rel=1e-6 if c["dtype"] == "f32" else 4e-3)
    if c["kind"] == "geom_matmul" or c["dtype"] == "f32":  # 32-bit sums of up to a few thousand terms: 2e-7 to 7e-7 seen
        return dict(rel=4e-6, max=1e-3 if c["kind"] == "train" else 1e-4)
    # 16-bit inputs, hidden rows and outputs (whole-number weights in a fixed-point product: about half the error)
    return dict(rel=8e-3 if c.get("fmt") == "int8_pauli" else 1.5e-2, max=0.3)


# ---------------------------------------------------------------------------
# the same in float64, plain torch
# ---------------------------------------------------------------------------

_MASKS = (0, 1, 2, 4, 3, 5, 6, 7)  # generators of each blade: 1, e1, e2, e3, e12, e13, e23, e123


def _cayley():
    """left[r][q] = (p, sign): blade p times blade q is sign times blade r."""
    left = [[None] * 8 for _ in range(8)]
    for p, a in enumerate(_MASKS):
        for q, b in enumerate(_MASKS):
            swaps = sum(bin(a >> (s + 1)).count("1") for s in range(3) if b >> s & 1)
            left[_MASKS.index(a ^ b)][q] = (p, -1.0 if swaps % 2 else 1.0)
    return left


_LEFT = _cayley()


def _linear64(x, w, b=None):
    """y_j = sum_i w_ji x_i (+ b_j): x (n, d_in, 8), w (d_out, d_in, 8) float64."""
    n, (o, i) = x.shape[0], w.shape[:2]
    dense = torch.empty((i, 8, o, 8), device=x.device, dtype=torch.float64)
    for r in range(8):
        for q in range(8):
            p, s = _LEFT[r][q]
            dense[:, q, :, r] = s * w[:, :, p].T
    y = (x.reshape(n, i * 8) @ dense.reshape(i * 8, o * 8)).reshape(n, o, 8)
    return y if b is None else y + b


def _act64(v, act):
    def gelu(u):
        return 0.5 * u * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (u + 0.044715 * u ** 3)))

    f = {"gelu": gelu, "relu": lambda u: torch.clamp(u, min=0.0), "sigmoid": torch.sigmoid}[act]
    parts = [f(v[..., 0:1])]
    for lo in (1, 4):
        c = v[..., lo:lo + 3]
        mag = torch.sqrt((c * c).sum(-1, keepdim=True) + 1e-12)
        parts.append(c / mag * f(mag))
    parts.append(v[..., 7:8] if act == "relu" else torch.tanh(v[..., 7:8]))
    return torch.cat(parts, -1)


def _route64(logits, k):
    e = torch.exp(logits - logits.max(-1, keepdim=True).values)
    p = e / (e.sum(-1, keepdim=True) + 1e-12)
    w, idx = torch.sort(p, dim=-1, descending=True, stable=True)
    w, idx = w[:, :k], idx[:, :k]
    return idx, w / (w.sum(-1, keepdim=True) + 1e-12)


def _norm64(x, gamma, beta, eps=1e-6):
    rms = torch.sqrt((x * x).sum(-1).mean(-1) + 2.0 * eps)[:, None, None]
    xh = x / rms
    y = torch.empty_like(x)
    for r in range(8):
        y[..., r] = sum(s * gamma[:, p] * xh[..., q] for q in range(8) for p, s in [_LEFT[r][q]])
    return y + beta


def _entries(w):
    """The real entries of a multivector's complex 2x2 matrix: u00, v00, u01, v01, u10, v10, u11, v11."""
    s, v1, v2, v3, b12, b13, b23, t = w.unbind(-1)
    return torch.stack([s + v3, t + b12, v1 - b13, b23 - v2, v1 + b13, b23 + v2, s - v3, t - b12], -1)


def _from_entries(p):
    u00, v00, u01, v01, u10, v10, u11, v11 = p.unbind(-1)
    return 0.5 * torch.stack([u00 + u11, u10 + u01, v10 - v01, u00 - u11, v00 - v11, u10 - u01, v10 + v01,
                              v00 + v11], -1)


def _held64(w, fmt):
    """The weights that a format of whole numbers holds (one scale per output channel), else w."""
    w = w.double()
    if not fmt.startswith("int8"):
        return w
    v = _entries(w) if fmt == "int8_pauli" else w
    s = (v.abs().amax((-2, -1), keepdim=True).clamp(min=1e-12) / 127.0).float().double()
    v = torch.clamp(torch.round(v / s), -127, 127) * s
    return _from_entries(v) if fmt == "int8_pauli" else v


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    if c["kind"] == "geom_matmul":  # out[m, n] = sum_k a[m, k] b[k, n]
        return _linear64(t["b"].double().transpose(0, 1), t["a"].double()).transpose(0, 1).contiguous()
    if c["kind"] == "linear":
        y = _linear64(t["x"].double(), t["w"].double(), None if t["b"] is None else t["b"].double())
        B = 4 if c["N"] % 4 == 0 else 1
        return y.reshape(B, c["N"] // B, c["d_out"], 8)
    x = t["x"].double()
    k = c["k"]
    if c["kind"] == "route":
        idx, w = _route64(t["logits"].double(), k)
        return dict(idx=None, w=w, counts=None, perm=None, rows=None, out=x * w.sum(-1)[:, None, None])
    xin = x
    if c["kind"] == "block":
        x = _norm64(x, t["gamma"].double(), t["beta"].double())
    if c["router"] == "energy":
        en = torch.stack([(x[..., lo:hi] ** 2).sum((-2, -1)) for lo, hi in ((0, 1), (1, 4), (4, 7), (7, 8))], -1)
        logits = (en / (en.sum(-1, keepdim=True) + 1e-12)) @ t["router_weight"].double().T + t["router_bias"].double()
    elif c["router"] == "clifford_head":
        logits = _linear64(x, t["head_weight"].double())[..., 0]
    else:
        logits = t["logits"].double()
    idx, w = _route64(logits, k)
    train = c["kind"] == "train"
    w_up, w_down = _held64(t["w_up"], c["fmt"]), _held64(t["w_down"], c["fmt"])
    b_up, b_down = t["b_up"].double(), t["b_down"].double()
    out = torch.zeros_like(x)
    grads = dict(dx=torch.zeros_like(x), dw_up=torch.zeros_like(w_up), db_up=torch.zeros_like(b_up),
                 dw_down=torch.zeros_like(w_down), db_down=torch.zeros_like(b_down)) if train else {}
    for e in range(c["E"]):
        tok, slot = torch.nonzero(idx == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        xe, we = x[tok], w[tok, slot][:, None, None]
        if not train:
            h = _act64(_linear64(xe, w_up[e], b_up[e]), c["act"])
            out.index_add_(0, tok, we * _linear64(h, w_down[e], b_down[e]))
            continue
        with torch.enable_grad():
            leaves = [v.detach().requires_grad_(True) for v in (xe, w_up[e], b_up[e], w_down[e], b_down[e])]
            h = _act64(_linear64(leaves[0], leaves[1], leaves[2]), c["act"])
            y = we * _linear64(h, leaves[3], leaves[4])
            ge = torch.autograd.grad(y, leaves, t["grad"].double()[tok])
        out.index_add_(0, tok, y.detach())
        grads["dx"].index_add_(0, tok, ge[0])
        grads["dw_up"][e], grads["db_up"][e], grads["dw_down"][e], grads["db_down"][e] = ge[1:]
    if c["kind"] == "block":
        out = out + xin
    B = 4 if c["N"] % 4 == 0 else 1
    shape = (B, c["N"] // B, c["d"], 8)
    if train:
        counts = torch.bincount(idx.reshape(-1), minlength=c["E"]).double()
        grads["dx"] = grads["dx"].reshape(shape)
        return dict(out=out.reshape(shape), aux=((counts / counts.sum() - 1.0 / c["E"]) ** 2).sum(), **grads)
    return out.reshape(shape)
