"""Performance cases: the calls that programs built on this library spend their time in.

Each case is one pass through the public entry points (`aurora_amd.gpu`, `aurora_amd.model`):
single linear layers in the three forms a model uses (forward, input gradient, weight
gradient), causal attention forward and backward, one decode attention step, an optimizer
step, and two whole calls: a training step and a generation (prefill and decode).  Sizes are
those of the configurations that the benchmark and the tests use, plus odd and ragged ones of
the same ranges.  All device tensors are fp32; token ids are 32-bit.
"""
import math

import numpy as np
import torch

from aurora_amd.gpu import (CausalMhaBackwardKernel, CausalMhaForwardKernel, GemmKernel, GemmTransposeBKernel,
                            GpuContext, MhaKvCacheKernel, OuterProductAccumKernel)
from aurora_amd.model import DecoderTransformerGpu

_CTX = None


def _ctx():
    """The program's one context (one device, one stream)."""
    global _CTX
    if _CTX is None:
        _CTX = GpuContext.new(0)
    return _CTX


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # QKV projection of the tiny model (8 sequences x 64 tokens, d 128): a small call, where
        # latency counts
        {"name": "linear_tiny", "op": "linear", "m": 512, "n": 384, "k": 128},
        # one projection for 8 sequences decoded together: the weights are streamed once
        {"name": "linear_step", "op": "linear", "m": 8, "n": 4096, "k": 1024},
        # FFN up-projection at d 512 over 8 x 1024 tokens
        {"name": "linear_up", "op": "linear", "m": 8192, "n": 2048, "k": 512},
        # a layer of no round size: 3 windows of 259 tokens, rows of k and n floats that are not
        # multiples of 16 bytes
        {"name": "linear_odd", "op": "linear", "m": 777, "n": 1023, "k": 513},
        # input gradient of the FFN up-projection, d 1024 over 16 x 1024 tokens
        {"name": "linear_dx", "op": "linear_dx", "m": 16384, "n": 1024, "k": 4096},
        # weight gradient of the same layer: a long reduction over the tokens
        {"name": "linear_dw", "op": "linear_dw", "m": 4096, "n": 1024, "k": 16384},
        # attention of a d 512 model, 16 sequences of 1024
        {"name": "attn_fwd", "op": "attn", "b": 16, "t": 1024, "h": 8, "dh": 64, "fwd": True, "bwd": False},
        {"name": "attn_bwd", "op": "attn", "b": 16, "t": 1024, "h": 8, "dh": 64, "fwd": False, "bwd": True},
        # both directions at a ragged length and another head width
        {"name": "attn_ragged", "op": "attn", "b": 4, "t": 333, "h": 6, "dh": 48, "fwd": True, "bwd": True},
        # one decode step's attention, 32 sequences of different lengths up to 768
        {"name": "attn_decode", "op": "attn_decode", "b": 32, "h": 16, "dh": 64, "max_len": 768},
        # a training step (loss and gradients) of the d 1024, 12-layer model, 16 x 1024 tokens:
        # the largest call
        {"name": "train", "op": "train", "vocab": 8192, "d": 1024, "layers": 12, "heads": 16, "ff": 4096,
         "b": 16, "t": 1024},
        # serving the same model: 32 prompts of 512 tokens, then 32 steps whose logits the program
        # reads (it samples, or scores a given continuation) and whose tokens it feeds back
        {"name": "generate", "op": "generate", "vocab": 8192, "d": 1024, "layers": 12, "heads": 16, "ff": 4096,
         "b": 32, "t": 512, "steps": 32},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the same ranges: sizes over their logarithm, about half of them round."""
    op = rng.choice(["linear", "linear", "linear_dx", "linear_dw", "attn", "attn", "attn_decode", "train",
                     "generate"])

    def size(lo, hi, step):
        v = _log(rng, lo, hi)
        return max(step, v // step * step) if rng.random() < 0.6 else v

    if op == "linear":
        return {"op": op, "m": size(1, 16384, 64), "n": size(128, 8192, 128), "k": size(64, 4096, 64)}
    if op == "linear_dx":
        return {"op": op, "m": size(64, 16384, 64), "n": size(64, 4096, 64), "k": size(128, 8192, 128)}
    if op == "linear_dw":
        return {"op": op, "m": size(128, 4096, 64), "n": size(64, 4096, 64), "k": size(64, 16384, 64)}
    if op == "attn":
        both = rng.choice([(True, False), (False, True), (True, True)])
        return {"op": op, "b": _log(rng, 1, 16), "t": size(17, 1024, 64), "h": rng.randint(1, 16),
                "dh": rng.choice([16, 32, 40, 48, 64, 64, 64]), "fwd": both[0], "bwd": both[1]}
    if op == "attn_decode":
        return {"op": op, "b": _log(rng, 1, 64), "h": rng.randint(2, 16), "dh": rng.choice([16, 32, 48, 64, 64]),
                "max_len": _log(rng, 64, 2048)}
    heads, dh = rng.choice([2, 4, 6, 8, 16]), rng.choice([32, 48, 64])
    d = heads * dh
    model = {"vocab": rng.choice([256, 1000, 4096, 8192]), "d": d, "layers": rng.randint(1, 6), "heads": heads,
             "ff": 4 * d}
    if op == "train":
        return {"op": op, **model, "b": _log(rng, 1, 16), "t": size(16, 1024, 64)}
    return {"op": op, **model, "b": _log(rng, 1, 32), "t": _log(rng, 8, 512), "steps": rng.randint(4, 32)}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, std=1.0):
    x = torch.empty(shape, device="cuda", dtype=torch.float32)
    return x.normal_(0.0, std, generator=g)


def _linear_inputs(c, seed):
    """Activations N(0, 1) as a LayerNorm leaves them, weights N(0, 0.02); the gradient of a layer's
    output is small."""
    g = _gen(seed)
    m, n, k = c["m"], c["n"], c["k"]
    if c["op"] == "linear":  # y[m, n] = x[m, k] W[n, k]^T
        return _normal(g, (m, k)), _normal(g, (n, k), 0.02)
    if c["op"] == "linear_dx":  # dx[m, n] = dy[m, k] W[k, n]
        return _normal(g, (m, k), 1e-2), _normal(g, (k, n), 0.02)
    # dW[m, n] += dy[k, m]^T x[k, n]
    return _normal(g, (k, m), 1e-2), _normal(g, (k, n))


def _attn_inputs(c, seed):
    g = _gen(seed)
    shape = (c["b"] * c["t"], c["h"] * c["dh"])
    return [_normal(g, shape) for _ in range(4)]


def _decode_inputs(c, seed):
    g = _gen(seed)
    b, d, n = c["b"], c["h"] * c["dh"], c["max_len"]
    q, k, v = _normal(g, (b, d)), _normal(g, (b, n, d)), _normal(g, (b, n, d))
    lens = np.random.default_rng(seed).integers(max(1, 2 * n // 3), n + 1, b).astype(np.int32)
    return q, k, v, lens


class _DeviceFloats:
    """Device memory of a model, for torch: the model lives as long as a tensor of it does."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False), "strides": None,
                                         "version": 3}


class _Model:
    """A model and what the program keeps beside it; its memory is returned with it."""

    def __init__(self, c, seq_max, max_batch):
        self.m = DecoderTransformerGpu(_ctx(), c["vocab"], c["d"], c["layers"], c["heads"], c["ff"], seq_max,
                                       max_batch)
        self.cache = None

    def tensor(self, name, layer=-1, grad=False):
        return torch.as_tensor(_DeviceFloats(self, *self.m.tensor_ptr(name, layer, grad)), device="cuda")

    def __del__(self):
        if self.cache is not None:
            self.cache.destroy()
        self.m.destroy()


def _params(c, seq_max, seed):
    """Random initial parameters: N(0, 0.02), W_o and W_proj scaled by 1/sqrt(2 layers), LN 1 and 0."""
    g = _gen(seed)
    V, d, F, L = c["vocab"], c["d"], c["ff"], c["layers"]
    res = 0.02 / math.sqrt(2 * L)
    p = {("w_tok", -1): _normal(g, (V, d), 0.02), ("w_pos", -1): _normal(g, (seq_max, d), 0.02)}
    for name, layer in [("lnf", -1)] + [(n, l) for l in range(L) for n in ("ln1", "ln2")]:
        p[name + "_g", layer] = 1.0 + _normal(g, (d,), 0.02)
        p[name + "_b", layer] = _normal(g, (d,), 0.02)
    for l in range(L):
        p["w_qkv", l] = _normal(g, (3 * d, d), 0.02)
        p["w_o", l] = _normal(g, (d, d), res)
        p["w_fc", l] = _normal(g, (F, d), 0.02)
        p["w_proj", l] = _normal(g, (d, F), res)
    return p


def _seq_max(c):
    return c["t"] + c.get("steps", 0)


def _tokens(c, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, c["vocab"], (c["b"], c["t"] + max(1, c.get("steps", 0)))).astype(np.uint32)


def _load_model(c, seed):
    s = _Model(c, _seq_max(c), c["b"])
    for (name, layer), x in _params(c, _seq_max(c), seed).items():
        s.tensor(name, layer).copy_(x.reshape(-1))
    return s


def prepare(case, seed):
    c, ctx = case, _ctx()
    st = {"case": c}
    if c["op"].startswith("linear"):
        st["a"], st["b"] = _linear_inputs(c, seed)
        st["c"] = torch.zeros((c["m"], c["n"]), device="cuda")
    elif c["op"] == "attn":
        st["q"], st["k"], st["v"], st["do"] = _attn_inputs(c, seed)
        st["o"] = torch.empty_like(st["q"])
        st["lse"] = torch.empty((c["b"], c["h"], c["t"]), device="cuda")
        if c["bwd"]:
            st["grads"] = torch.zeros((3,) + tuple(st["q"].shape), device="cuda")
            st["ws"] = torch.empty(CausalMhaBackwardKernel.workspace_len(c["t"], c["h"], c["b"]), device="cuda")
            torch.cuda.synchronize()
            _attn_fwd(st)  # the backward's inputs include the forward's results
    elif c["op"] == "attn_decode":
        st["q"], st["k"], st["v"], lens = _decode_inputs(c, seed)
        st["lens"], st["t_max"] = torch.from_numpy(lens).cuda(), int(lens.max())
        st["o"] = torch.empty_like(st["q"])
        n = MhaKvCacheKernel.scratch_len(c["h"], c["max_len"], c["b"])
        st["ws"] = torch.empty(max(1, n), device="cuda")
    elif c["op"] == "train":
        st["model"] = _load_model(c, seed)
        seq = _tokens(c, seed)
        st["tok"], st["tgt"] = np.ascontiguousarray(seq[:, :-1]), np.ascontiguousarray(seq[:, 1:])
        st["grads"] = st["model"].tensor("grads", grad=True)
    else:
        st["model"] = s = _load_model(c, seed)
        s.cache = s.m.kv_cache(c["b"], _seq_max(c))
        st["seq"] = _tokens(c, seed)
    torch.cuda.synchronize()
    ctx.sync()
    return st


# ------------------------------------------------------------------ one pass


def _attn_fwd(st):
    c = st["case"]
    CausalMhaForwardKernel.new().dispatch_into(_ctx(), *(st[x].data_ptr() for x in ("q", "k", "v", "o", "lse")),
                                               c["t"], c["h"], c["dh"], b=c["b"])


def run(st):
    c, ctx = st["case"], _ctx()
    if c["op"].startswith("linear"):
        a, b, out = st["a"].data_ptr(), st["b"].data_ptr(), st["c"].data_ptr()
        if c["op"] == "linear":
            GemmTransposeBKernel.new().dispatch_into(ctx, a, b, out, c["m"], c["n"], c["k"])
        elif c["op"] == "linear_dx":
            GemmKernel.new().dispatch_into(ctx, a, b, out, c["m"], c["n"], c["k"])
        else:  # the gradient accumulates: a step begins with zero
            ctx.call("aur_memset0", out, 4 * c["m"] * c["n"])
            OuterProductAccumKernel.new().dispatch_into(ctx, b, a, out, c["m"], c["n"], c["k"])
        return st["c"]
    if c["op"] == "attn":
        if c["fwd"]:
            _attn_fwd(st)
        if not c["bwd"]:
            return {"o": st["o"], "lse": st["lse"]}
        g = st["grads"]
        ctx.call("aur_memset0", g.data_ptr(), 4 * g.numel())
        CausalMhaBackwardKernel.new().dispatch_into(
            ctx, *(st[x].data_ptr() for x in ("q", "k", "v", "o", "lse", "do")), g[0].data_ptr(), g[1].data_ptr(),
            g[2].data_ptr(), st["ws"].data_ptr(), c["t"], c["h"], c["dh"], b=c["b"])
        out = {"dq": g[0], "dk": g[1], "dv": g[2]}
        return {"o": st["o"], "lse": st["lse"], **out} if c["fwd"] else out
    if c["op"] == "attn_decode":
        MhaKvCacheKernel.new().dispatch_batched(
            ctx, *(st[x].data_ptr() for x in ("q", "k", "v", "o", "ws", "lens")), st["t_max"], c["b"], c["h"],
            c["dh"], c["max_len"])
        return st["o"]
    m = st["model"].m
    if c["op"] == "train":
        m.zero_grad()
        loss = m.train_step_batch(st["tok"], st["tgt"])
        return {"loss": loss, "grads": st["grads"]}
    seq, cache = st["seq"], st["model"].cache
    logits = [m.prefill_kv(cache, seq[:, :c["t"]])]
    for s in range(c["steps"]):
        logits.append(m.generate_step_kv(cache, seq[:, c["t"] + s])[0])
    return {"logits": np.stack(logits)}


# ------------------------------------------------------------------ work, tolerance


def _pairs(b, h, t):
    return b * h * t * (t + 1) / 2


def work(case):
    c = case
    if c["op"].startswith("linear"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4.0 * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    if c["op"] == "attn":
        x, pairs = c["b"] * c["t"] * c["h"] * c["dh"], _pairs(c["b"], c["h"], c["t"])
        rows = c["b"] * c["t"] * c["h"]
        nbytes = (4 * x + rows if c["fwd"] else 0) + (8 * x + rows if c["bwd"] else 0)
        flops = ((4 if c["fwd"] else 0) + (10 if c["bwd"] else 0)) * c["dh"] * pairs
        return {"bytes": 4.0 * nbytes, "flops": float(flops)}
    if c["op"] == "attn_decode":
        d, keys = c["h"] * c["dh"], c["b"] * c["max_len"] * 5.0 / 6.0
        return {"bytes": 4.0 * (2 * keys * d + 2 * c["b"] * d), "flops": 4.0 * keys * d}
    V, d, F, L, b, t = (c[x] for x in ("vocab", "d", "ff", "layers", "b", "t"))
    lin = L * (4 * d * d + 2 * d * F)
    if c["op"] == "train":
        params = lin + V * d + t * d + (4 * L + 2) * d
        return {"bytes": 4.0 * 2 * params,
                "flops": 6.0 * b * t * (lin + V * d) + L * 14.0 * (d // c["heads"]) * _pairs(b, c["heads"], t)}
    steps = c["steps"]
    nbytes, flops = lin + V * d, 2.0 * b * t * lin + L * 4.0 * (d // c["heads"]) * _pairs(b, c["heads"], t)
    for s in range(steps):
        nbytes += lin + V * d + 2 * L * b * (t + s + 1) * d + b * V
        flops += 2.0 * b * (lin + V * d) + L * 4.0 * b * (t + s + 1) * d
    return {"bytes": 4.0 * nbytes, "flops": flops}


def tolerance(case):
    """About four times (and a little more) what these paths show against 64 bits."""
    op = case["op"]
    if op.startswith("linear"):
        return {"rel": 1e-5}  # up to 1.6e-6 seen, at 16384 terms a sum
    if op in ("attn", "attn_decode"):
        return {"rel": 5e-6}  # up to 8e-7
    return {"rel": 2e-5 if op == "train" else 5e-6}  # 3e-6 in the gradients, 6e-7 in the logits


# ------------------------------------------------------------------ the same in 64 bits


def _f64_attention(q, k, v, causal_from=0):
    """softmax(q k^T / sqrt(dh)) v over the last two axes; query i sees keys 0 .. causal_from + i."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    i = torch.arange(q.shape[-2], device=q.device)[:, None] + causal_from
    s = s.masked_fill(torch.arange(k.shape[-2], device=q.device)[None, :] > i, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v), torch.logsumexp(s, -1)


def _heads(x, b, t, h):
    return x.double().reshape(b, t, h, -1).transpose(1, 2).contiguous()


def _rows(x):
    b, h, t, dh = x.shape
    return x.transpose(1, 2).reshape(b * t, h * dh)


def _f64_model(c, p, tok, last_only_from=None):
    """Pre-LN GPT with a tied head, learned positions and tanh-GELU on tokens [t] -> logits."""
    F = torch.nn.functional
    d, h, t = c["d"], c["heads"], tok.shape[0]
    x = p["w_tok", -1][tok] + p["w_pos", -1][:t]
    for l in range(c["layers"]):
        y = F.layer_norm(x, (d,), p["ln1_g", l], p["ln1_b", l], 1e-5)
        q, k, v = (F.linear(y, w).reshape(t, h, -1).transpose(0, 1).contiguous() for w in p["w_qkv", l].split(d))
        o, _ = _f64_attention(q, k, v)
        x = x + F.linear(o.transpose(0, 1).reshape(t, d), p["w_o", l])
        y = F.layer_norm(x, (d,), p["ln2_g", l], p["ln2_b", l], 1e-5)
        x = x + F.linear(F.gelu(F.linear(y, p["w_fc", l]), approximate="tanh"), p["w_proj", l])
    x = x if last_only_from is None else x[last_only_from:]
    return F.linear(F.layer_norm(x, (d,), p["lnf_g", -1], p["lnf_b", -1], 1e-5), p["w_tok", -1])


def _grad_order(c):
    """Tensor order of the model's flat gradient."""
    L = range(c["layers"])
    return ([("w_tok", -1)] + [(n, l) for l in L for n in ("w_qkv", "w_o", "w_fc", "w_proj")] + [("w_pos", -1)] +
            [(n, l) for l in L for n in ("ln1_g", "ln1_b", "ln2_g", "ln2_b")] + [("lnf_g", -1), ("lnf_b", -1)])


def exact(case, seed):
    c = case
    if c["op"].startswith("linear"):
        a, b = (x.double() for x in _linear_inputs(c, seed))
        if c["op"] == "linear":
            return torch.matmul(a, b.t())
        return torch.matmul(a, b) if c["op"] == "linear_dx" else torch.matmul(a.t(), b)
    if c["op"] == "attn":
        q, k, v, do = (_heads(x, c["b"], c["t"], c["h"]) for x in _attn_inputs(c, seed))
        for x in (q, k, v):
            x.requires_grad_(c["bwd"])
        o, lse = _f64_attention(q, k, v)
        out = {"o": _rows(o.detach()), "lse": lse.detach()} if c["fwd"] else {}
        if c["bwd"]:
            for name, g in zip(("dq", "dk", "dv"), torch.autograd.grad(o, (q, k, v), do)):
                out[name] = _rows(g)
        return out
    if c["op"] == "attn_decode":
        q, k, v, lens = _decode_inputs(c, seed)
        out, h = torch.empty(q.shape, dtype=torch.float64, device="cuda"), c["h"]
        for i, n in enumerate(lens.tolist()):
            o, _ = _f64_attention(_heads(q[i:i + 1], 1, 1, h), _heads(k[i, :n], 1, n, h), _heads(v[i, :n], 1, n, h),
                                  causal_from=n - 1)
            out[i] = _rows(o)[0]
        return out
    p = {name: x.double() for name, x in _params(c, _seq_max(c), seed).items()}
    seq = torch.from_numpy(_tokens(c, seed).astype(np.int64)).cuda()
    if c["op"] == "train":
        leaves = [p[name].requires_grad_() for name in _grad_order(c)]
        total, grads = 0.0, None
        for i in range(c["b"]):
            loss = torch.nn.functional.cross_entropy(_f64_model(c, p, seq[i, :-1]), seq[i, 1:])
            total += float(loss.detach())
            g = torch.autograd.grad(loss / c["b"], leaves)
            grads = list(g) if grads is None else [x.add_(y) for x, y in zip(grads, g)]
        return {"loss": total, "grads": torch.cat([x.reshape(-1) for x in grads])}
    with torch.no_grad():
        rows = [_f64_model(c, p, seq[i], c["t"] - 1) for i in range(c["b"])]
    return {"logits": torch.stack(rows, 1).cpu().numpy()}
