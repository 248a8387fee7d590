"""The work a user of this library has it do, as timed and compared cases.

Every case goes through a public entry point: the device-tensor attention
(`cpuforge_amd.device`), the layer's attention with its RoPE / q-k-norm
prologue (`cpuforge_amd.layer`), the reference-shaped host-slice functions
(`cpuforge_amd.attention_forward` / `attention_backward`), the layer ops
(`cpuforge_amd.autograd`), AdamW (`cpuforge_amd.optim`) and the SmolLM-135M
LoRA training step (`cpuforge_amd.train_bench`), eager and as graph replays.
Sizes are the benchmark configurations, the tests' shapes and generic ones.

`listed()` names the cases, `draw(rng)` gives another one of the same ranges,
`prepare` / `run` / `work` / `tolerance` / `exact` describe one case.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

import cpuforge_amd as cf
from cpuforge_amd import autograd as A
from cpuforge_amd import device as D
from cpuforge_amd.layer import LayerRope, layer_attention
from cpuforge_amd.optim import AdamW
from cpuforge_amd.rope import Llama3Scaling, RopeCache
from cpuforge_amd.train_bench import SMOLLM_135M, SmolLM, capture_step

DEV = "cuda"
IGNORE = -100
LORA_ALPHA_PER_RANK = 2.0  # alpha = 2 * rank, as `cpuforge bench-train` sets it
QK_EPS = 1e-6
NORM_EPS = 1e-5

# --------------------------------------------------------------------- cases


def listed():
    return [
        # One short sequence with a head_dim no matrix-core path takes (the
        # reference's own ragged test shape): launch latency.
        dict(name="attn_f32_tiny", kind="attn", dtype="f32", batch=1, seq=13, heads=6, kv=2, dim=4),
        # SmolLM-135M's attention at a training batch, in the reference's own
        # precision, forward and backward.
        dict(name="attn_f32_train", kind="attn", dtype="f32", batch=8, seq=2048, heads=9, kv=3, dim=64),
        # Llama-3-8B's attention layer, forward and backward: the benchmark's
        # headline workload.
        dict(name="attn_bf16_8k", kind="attn", dtype="bf16", batch=1, seq=8192, heads=32, kv=8, dim=128),
        # Llama-3.2-1B's layer attention (llama3 RoPE) as a training step runs
        # it: prologue, attention and both backwards.
        dict(name="layer_bf16_d64", kind="layer", dtype="bf16", batch=4, seq=4096, heads=32, kv=8, dim=64,
             theta=5e5, llama3=True, qk_norm=False),
        # Qwen3-0.6B's layer attention: per-head q/k RMSNorm with trained gains.
        dict(name="layer_bf16_qknorm", kind="layer", dtype="bf16", batch=4, seq=4096, heads=16, kv=8, dim=128,
             theta=1e6, llama3=False, qk_norm=True),
        # Evaluation: the layer's attention forward alone on ragged lengths.
        dict(name="prefill_bf16_ragged", kind="prefill", dtype="bf16", batch=2, seq=3001, heads=32, kv=8, dim=128,
             theta=5e5, llama3=False, qk_norm=False),
        # The drop-in a cpuforge host calls: host slices in and out, one
        # sequence at a time, f32.
        dict(name="host_f32", kind="host", dtype="f32", seq=512, heads=9, kv=3, dim=64),
        # SmolLM-135M's MLP half of a layer with LoRA adapters, forward and
        # backward, at the training batch (8 x 512 tokens).
        dict(name="mlp_lora", kind="mlp", tokens=4096, d=576, ffn=1536, rank=16, train="lora"),
        # The final norm's output through a trained LM head with its loss, a
        # tenth of the positions not scored (prompt tokens).
        dict(name="head_ce_full", kind="head", tokens=4096, d=576, vocab=49152, train="full"),
        # One optimizer step over SmolLM-135M's 420 adapter tensors.
        dict(name="adamw_lora", kind="adamw", layers=30, rank=16),
        # `cpuforge bench-train`'s own step: one sequence of 512 tokens, run
        # eagerly.
        dict(name="train_eager", kind="train", batch=1, seq=512, layers=30, rank=16, graph=False),
        # The same model at a training batch, the step replayed as a graph:
        # the benchmark's train figure.
        dict(name="train_graph", kind="train", batch=8, seq=512, layers=30, rank=16, graph=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_HEADS = ((9, 3), (32, 8), (16, 8), (6, 2), (8, 1), (4, 4))
_WIDTHS = ((576, 1536), (576, 1536), (1024, 3072), (2048, 8192), (500, 1333))


def _attn_shape(rng, dtype):
    heads, kv = rng.choice(_HEADS)
    dim = rng.choice((64, 64, 64, 128, 128, 128, 32, 80, 6))
    # Head dims other than 64 and 128 stand for small models; f32 lengths go
    # to 4096, bf16 to 8192.
    top = 1024 if dim not in (64, 128) else 4096 if dtype == "f32" else 8192
    seq = _log(rng, 8, top)
    most = max(1, int(2.0e12 if dtype == "bf16" else 1.5e11) // max(1, int(7 * heads * dim * seq * (seq + 1))))
    if dim not in (64, 128):
        most = 2
    return dict(batch=_log(rng, 1, min(8, most)), seq=seq, heads=heads, kv=kv, dim=dim)


def draw(rng):
    kind = rng.choice(("attn", "attn", "layer", "layer", "prefill", "host", "mlp", "mlp", "head", "adamw", "train"))
    if kind in ("attn", "layer", "prefill"):
        dtype = rng.choice(("f32", "bf16"))
        c = dict(kind=kind, dtype=dtype, **_attn_shape(rng, dtype))
        if kind != "attn":
            c.update(theta=rng.choice((1e4, 5e5, 1e6)), llama3=rng.random() < 0.3, qk_norm=rng.random() < 0.4)
        return c
    if kind == "host":
        heads, kv = rng.choice(((9, 3), (6, 2), (4, 4)))
        return dict(kind="host", dtype="f32", seq=_log(rng, 8, 1500), heads=heads, kv=kv, dim=rng.choice((64, 128, 6)))
    if kind == "mlp":
        d, ffn = rng.choice(_WIDTHS)
        return dict(kind="mlp", tokens=_log(rng, 16, 4096 if d == 2048 else 8192), d=d, ffn=ffn,
                    rank=rng.choice((4, 8, 16, 16, 32)), train=rng.choice(("lora", "lora", "full")))
    if kind == "head":
        d = rng.choice((576, 1024, 500))
        return dict(kind="head", tokens=_log(rng, 32, 4096), d=d, vocab=rng.choice((49152, 32000, 50001)),
                    train=rng.choice(("lora", "full")))
    if kind == "adamw":
        return dict(kind="adamw", layers=rng.randint(4, 30), rank=rng.choice((4, 8, 16)))
    return dict(kind="train", batch=rng.randint(1, 8), seq=_log(rng, 40, 512), layers=rng.randint(2, 12),
                rank=rng.choice((8, 16)), graph=rng.random() < 0.5)


# ------------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _rope(case):
    scaling = Llama3Scaling(32.0, 1.0, 4.0, 8192.0) if case["llama3"] else None
    return RopeCache(case["dim"], case["seq"], case["theta"], scaling)


def _attn_inputs(case, seed):
    """q, k, v, d_o of the attention, or q_pre, k_pre, v, d_o and the norm
    gains of the layer, unit variance as normalised projections give them."""
    g = _gen(seed)
    B, S, H, K, d = (case[k] for k in ("batch", "seq", "heads", "kv", "dim"))
    dt = _dtype(case)
    pre = torch.float32 if case["kind"] != "attn" else dt
    s = dict(q=_randn(g, B, S, H, d, dtype=pre), k=_randn(g, B, S, K, d, dtype=pre), v=_randn(g, B, S, K, d, dtype=dt),
             g=_randn(g, B, S, H, d, dtype=pre))
    if case.get("qk_norm"):
        s["qn"] = 1.0 + _randn(g, d, std=0.02)
        s["kn"] = 1.0 + _randn(g, d, std=0.02)
    return s


def _mlp_inputs(case, seed):
    g = _gen(seed)
    t, d, f, r = (case[k] for k in ("tokens", "d", "ffn", "rank"))
    lora = case["train"] == "lora"
    s = dict(x=_randn(g, t, d), norm=1.0 + _randn(g, d, std=0.02), dy=_randn(g, t, d, std=1e-2))
    for n, o, i in (("gate", f, d), ("up", f, d), ("down", d, f)):
        s[n] = dict(w=_randn(g, o, i, std=0.02), a=None, b=None)
        if lora:
            # An adapter some steps into training: B has left zero.
            s[n]["a"] = (torch.rand(r, i, generator=g, device=DEV) * 2 - 1) / i ** 0.5
            s[n]["b"] = _randn(g, o, r, std=0.01)
    return s


def _mlp_trained(case, s):
    """The tensors that train, x first."""
    if case["train"] == "lora":
        return [s["x"]] + [s[n][p] for n in ("gate", "up", "down") for p in ("a", "b")]
    return [s["x"], s["norm"]] + [s[n]["w"] for n in ("gate", "up", "down")]


def _head_inputs(case, seed):
    g = _gen(seed)
    t, d, vocab = case["tokens"], case["d"], case["vocab"]
    s = dict(hn=_randn(g, t, d), head=_randn(g, vocab, d, std=0.02),
             targets=torch.randint(0, vocab, (t,), generator=g, device=DEV))
    s["targets"][torch.rand(t, generator=g, device=DEV) < 0.1] = IGNORE
    s["targets"][0] = 1
    return s


def _train_model(case, seed):
    m = SmolLM(case["layers"], case["seq"], case["rank"], torch.float32, DEV, seed=int(seed) % (2 ** 31))
    g = _gen(seed + 1)
    for _, p in m.named_params():
        if p.requires_grad and p.dim() == 2 and p.shape[1] == case["rank"]:
            p.data.normal_(0.0, 0.01, generator=g)  # adapters some steps into training
    shape = (case["batch"], case["seq"])
    tokens = torch.randint(0, m.c["vocab"], shape, generator=g, device=DEV)
    targets = torch.randint(0, m.c["vocab"], shape, generator=g, device=DEV)
    return m, tokens, targets


class _Adapters:
    """Parameters under their names, as AdamW's model interface has them."""

    def __init__(self, named):
        self.named = named

    def named_params(self):
        return iter(self.named)


def _adamw_state(case, seed):
    """SmolLM-135M's adapter tensors with a gradient each and moments some
    steps into training, the buffers of each kind side by side in memory."""
    c, r = SMOLLM_135M, case["rank"]
    d, f, qd, kvd = c["d"], c["ffn"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    shapes = []
    for i in range(case["layers"]):
        for n, o, inn in (("self_attn.q_proj", qd, d), ("self_attn.k_proj", kvd, d), ("self_attn.v_proj", kvd, d),
                          ("self_attn.o_proj", d, qd), ("mlp.gate_proj", f, d), ("mlp.up_proj", f, d),
                          ("mlp.down_proj", d, f)):
            shapes.append((f"model.layers.{i}.{n}.lora_A", (r, inn)))
            shapes.append((f"model.layers.{i}.{n}.lora_B", (o, r)))
    total = sum(a * b for _, (a, b) in shapes)
    g = _gen(seed)
    flat = dict(p=_randn(g, total, std=0.02), m=_randn(g, total, std=1e-4),
                v=_randn(g, total, std=1e-3).square_())
    grads = _randn(g, total, std=1e-3)
    opt = AdamW(0.9, 0.999, 1e-8, 0.01)
    opt.step = 10
    named, off = [], 0
    for name, shape in shapes:
        n = shape[0] * shape[1]
        p, m, v, gr = (t[off:off + n].view(shape) for t in (flat["p"], flat["m"], flat["v"], grads))
        p.requires_grad_()
        p.grad = gr
        named.append((name, p))
        opt.state[name] = (m, v)
        off += n
    return dict(opt=opt, model=_Adapters(named), flat=flat)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "host":
        r = np.random.default_rng(int(seed))
        S, H, K, d = (case[k] for k in ("seq", "heads", "kv", "dim"))
        s = {n: r.standard_normal(S * h * d, dtype=np.float32) for n, h in (("q", H), ("k", K), ("v", K), ("g", H))}
        s.update(o=np.zeros(S * H * d, np.float32), lse=np.zeros(H * S, np.float32), dq=np.zeros(S * H * d, np.float32),
                 dk=np.zeros(S * K * d, np.float32), dv=np.zeros(S * K * d, np.float32), shape=cf.AttnShape(S, H, K, d))
        return dict(case=case, **s)
    if kind in ("attn", "layer", "prefill"):
        s = _attn_inputs(case, seed)
        if kind != "attn":
            if kind == "layer":
                for n in s:
                    if n != "g":
                        s[n].requires_grad_()
            s["rope"] = LayerRope(_rope(case), DEV, s.get("qn"), s.get("kn"), QK_EPS)
        return dict(case=case, **s)
    if kind == "mlp":
        s = _mlp_inputs(case, seed)
        for p in _mlp_trained(case, s):
            p.requires_grad_()
        return dict(case=case, scale=LORA_ALPHA_PER_RANK, **s)
    if kind == "head":
        s = _head_inputs(case, seed)
        s["hn"].requires_grad_()
        s["head"].requires_grad_(case["train"] == "full")
        return dict(case=case, **s)
    if kind == "adamw":
        return dict(case=case, **_adamw_state(case, seed))
    m, tokens, targets = _train_model(case, seed)
    s = dict(case=case, model=m, tokens=tokens, targets=targets, params=m.params())
    if case["graph"]:
        m.ce_on_device = True
        s["graph"], s["loss"] = capture_step(m, tokens, targets)
    return s


# ----------------------------------------------------------------- one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attn":
        o, lse = D.fwd(s["q"], s["k"], s["v"])
        return (o, lse, *D.bwd(s["g"], s["q"], s["k"], s["v"], o, lse))
    if kind == "layer":
        o = layer_attention(s["q"], s["k"], s["v"], s["rope"])
        inputs = [s[n] for n in ("q", "k", "v", "qn", "kn") if n in s]
        return (o.detach(), *torch.autograd.grad(o, inputs, s["g"]))
    if kind == "prefill":
        with torch.no_grad():
            return layer_attention(s["q"], s["k"], s["v"], s["rope"])
    if kind == "host":
        for n in ("dq", "dk", "dv"):
            s[n].fill(0.0)
        cf.attention_forward(s["q"], s["k"], s["v"], s["o"], s["lse"], s["shape"])
        cf.attention_backward(s["g"], s["q"], s["k"], s["v"], s["o"], s["lse"], s["dq"], s["dk"], s["dv"], s["shape"])
        return [s[n] for n in ("o", "lse", "dq", "dk", "dv")]
    if kind == "mlp":
        spec = lambda n: (s[n]["w"], s[n]["a"], s[n]["b"], s["scale"])  # noqa: E731
        h = A.rmsnorm(s["x"], s["norm"], NORM_EPS)
        g, u = A.shared_input_linears(h, [spec("gate"), spec("up")])
        y = s["x"] + A.linear(A.silu_mul(g, u), *spec("down"))
        return (y.detach(), *torch.autograd.grad(y, _mlp_trained(case, s), s["dy"]))
    if kind == "head":
        loss = A.lm_head_ce(s["hn"], s["head"], s["targets"])
        inputs = [s["hn"]] + ([s["head"]] if case["train"] == "full" else [])
        return (loss.detach(), *torch.autograd.grad(loss, inputs))
    if kind == "adamw":
        s["opt"].update(s["model"], 1e-4)
        return s["flat"]
    # The training step: loss and every adapter's gradient (in one tensor, as
    # gradient clipping takes them).
    if case["graph"]:
        s["graph"].replay()
        loss = s["loss"]
    else:
        for p in s["params"]:
            p.grad = None
        loss = s["model"].loss(s["tokens"], s["targets"])
        loss.backward()
    return loss.detach(), torch.cat([p.grad.view(-1) for p in s["params"]])


# ------------------------------------------------------- what a pass is worth


def _attn_work(case, fwd_only):
    B, S, H, K, d = (case.get("batch", 1), *(case[k] for k in ("seq", "heads", "kv", "dim")))
    pairs = B * H * S * (S + 1) / 2
    flops = (4 if fwd_only else 14) * pairs * d
    nq, nk, ns = B * S * H * d, B * S * K * d, B * S * H
    e = 2 if case["dtype"] == "bf16" else 4
    pre = e if case["kind"] in ("attn", "host") else 4  # q_pre, k_pre and d_o of the layer are f32
    byts = pre * (nq + nk) + e * nk + 4 * nq
    if not fwd_only:
        byts += pre * nq + 4 * (nq + nk) + (e if case["kind"] == "layer" else 4) * nk
    if case["kind"] in ("attn", "host"):
        byts += 4 * ns  # lse
    return byts, flops


def _mlp_work(t, d, f, r, full):
    w = 3 * d * f
    flops = 2.0 * t * w * (3 if full else 2)
    byts = 4.0 * (4 * t * d + w * (2 if full else 1))
    if not full:
        n = 3 * r * (d + f)
        flops += 6.0 * t * n
        byts += 8.0 * n
    return byts, flops


def work(case):
    kind = case["kind"]
    if kind in ("attn", "layer", "prefill", "host"):
        byts, flops = _attn_work(case, kind == "prefill")
    elif kind == "mlp":
        byts, flops = _mlp_work(case["tokens"], case["d"], case["ffn"], case["rank"], case["train"] == "full")
    elif kind == "head":
        t, d, v = case["tokens"], case["d"], case["vocab"]
        full = case["train"] == "full"
        byts, flops = 4.0 * (2 * t * d + v * d * (2 if full else 1)) + 8.0 * t, 2.0 * t * d * v * (3 if full else 2)
    elif kind == "adamw":
        c, r = SMOLLM_135M, case["rank"]
        qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        n = case["layers"] * r * (2 * (c["d"] + qd) + 2 * (c["d"] + kvd) + 3 * (c["d"] + c["ffn"]))
        byts, flops = 28.0 * n, 12.0 * n
    else:
        c, r, L, S = SMOLLM_135M, case["rank"], case["layers"], case["seq"]
        t, d, f, qd, kvd = case["batch"] * S, c["d"], c["ffn"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        w = 2 * d * qd + 2 * d * kvd + 3 * d * f
        lora = r * (2 * (d + qd) + 2 * (d + kvd) + 3 * (d + f))
        flops = L * (4.0 * t * w + 6.0 * t * lora + 7.0 * t * qd * (S + 1)) + 4.0 * t * d * c["vocab"]
        byts = 4.0 * (L * (w + 2 * lora) + c["vocab"] * d) + 16.0 * t
    return {"bytes": float(byts), "flops": float(flops)}


def tolerance(case):
    kind = case["kind"]
    if kind == "adamw":
        return "exact"  # a fixed order of f32 operations per element
    if case.get("dtype") == "bf16":
        return {"rel": 1.2e-2, "max": 0.5}  # q, k, P and dS in 16 bits
    if kind == "train":
        return {"rel": 1.2e-5, "max": 1e-2}  # f32 roundings through every layer and back
    return {"rel": 1e-5, "max": 1e-3}  # f32 sums


# ------------------------------------------------------------------- 64 bits


def _rope64(x, rope):
    cos = torch.from_numpy(rope.cos).to(DEV, torch.float64)[:x.shape[1], None]
    sin = torch.from_numpy(rope.sin).to(DEV, torch.float64)[:x.shape[1], None]
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attn64(q, k, v, g=None):
    """o, lse and, with g, dq, dk, dv; a sequence's KV group at a time."""
    B, S, H, d = q.shape
    K = k.shape[2]
    G = H // K
    mask = torch.ones(S, S, device=DEV, dtype=torch.bool).triu(1)
    o, lse = torch.empty_like(q), torch.empty(B, H, S, device=DEV, dtype=torch.float64)
    dq, dk, dv = (torch.zeros_like(t) for t in (q, k, v)) if g is not None else (None, None, None)
    for b in range(B):
        for h in range(H):
            kh, vh, qh = k[b, :, h // G], v[b, :, h // G], q[b, :, h]
            s = ((qh @ kh.t()) / math.sqrt(d)).masked_fill_(mask, -math.inf)
            l = torch.logsumexp(s, -1)
            p = torch.exp(s.sub_(l[:, None]))
            o[b, :, h], lse[b, h] = p @ vh, l
            if g is not None:
                gh = g[b, :, h]
                dv[b, :, h // G] += p.t() @ gh
                ds = p * (gh @ vh.t() - (gh * o[b, :, h]).sum(-1, keepdim=True)) / math.sqrt(d)
                dq[b, :, h] = ds @ kh
                dk[b, :, h // G] += ds.t() @ qh
    return o, lse, dq, dk, dv


class _Attn64Fn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v):
        ctx.save_for_backward(q, k, v)
        return _attn64(q, k, v)[0]

    @staticmethod
    def backward(ctx, g):
        return _attn64(*ctx.saved_tensors, g)[2:]


def _leaf(t, grad=True):
    return None if t is None else t.detach().double().requires_grad_(grad)


def _exact_attn(case, seed):
    s = _attn_inputs(case, seed)
    return _attn64(*(s[n].double() for n in ("q", "k", "v", "g")))


def _exact_layer(case, seed):
    s = {n: _leaf(t) for n, t in _attn_inputs(case, seed).items()}
    rope = _rope(case)
    q, k = s["q"], s["k"]
    if case["qk_norm"]:
        q, k = _norm64(q, s["qn"], QK_EPS), _norm64(k, s["kn"], QK_EPS)
    q, k = _rope64(q, rope), _rope64(k, rope)
    if case["kind"] == "prefill":
        with torch.no_grad():
            return _attn64(q, k, s["v"])[0]
    o = _Attn64Fn.apply(q, k, s["v"])
    return (o.detach(), *torch.autograd.grad(o, [s[n] for n in ("q", "k", "v", "qn", "kn") if n in s], s["g"]))


def _linear64(x, w, a, b, scale):
    y = x @ w.t()
    return y if a is None else y + (scale * (x @ a.t())) @ b.t()


def _exact_mlp(case, seed):
    s = _mlp_inputs(case, seed)
    s = {n: {p: _leaf(t) for p, t in v.items()} if isinstance(v, dict) else _leaf(v) for n, v in s.items()}
    lin = lambda n, x: _linear64(x, s[n]["w"], s[n]["a"], s[n]["b"], LORA_ALPHA_PER_RANK)  # noqa: E731
    h = _norm64(s["x"], s["norm"], NORM_EPS)
    y = s["x"] + lin("down", F.silu(lin("gate", h)) * lin("up", h))
    return (y.detach(), *torch.autograd.grad(y, _mlp_trained(case, s), s["dy"]))


def _exact_head(case, seed):
    s = _head_inputs(case, seed)
    full = case["train"] == "full"
    hn, head = _leaf(s["hn"]), _leaf(s["head"], full)
    loss = F.cross_entropy(hn @ head.t(), s["targets"], ignore_index=IGNORE)
    return (loss.detach(), *torch.autograd.grad(loss, [hn] + ([head] if full else [])))


def _exact_train(case, seed):
    m, tokens, targets = _train_model(case, seed)
    c, (B, S) = m.c, tokens.shape
    rope = m.rope.pr.rope
    leaves = []

    def lin(x, w):
        p = [_leaf(w.a), _leaf(w.b)]
        leaves.extend(p)
        return _linear64(x, w.w.double(), *p, w.scale)

    x = m.embed.double()[tokens]
    for layer in m.layers:
        n1 = _norm64(x, layer["attn_norm"].double(), c["eps"])
        q, k, v = (lin(n1, layer[n]).view(B, S, -1, c["head_dim"]) for n in ("wq", "wk", "wv"))
        o = _Attn64Fn.apply(_rope64(q, rope), _rope64(k, rope), v)
        x = x + lin(o.reshape(B, S, -1), layer["wo"])
        n2 = _norm64(x, layer["mlp_norm"].double(), c["eps"])
        gate, up = lin(n2, layer["gate"]), lin(n2, layer["up"])
        x = x + lin(F.silu(gate) * up, layer["down"])
    logits = _norm64(x, m.final_norm.double(), c["eps"]) @ m.embed.double().t()
    loss = F.cross_entropy(logits.view(-1, c["vocab"]), targets.view(-1))
    grads = torch.autograd.grad(loss, leaves)
    return loss.detach(), torch.cat([g.reshape(-1) for g in grads])


def exact(case, seed):
    kind = case["kind"]
    if kind == "adamw":
        return None  # compared bit for bit
    if kind == "attn":
        return _exact_attn(case, seed)
    if kind in ("layer", "prefill"):
        return _exact_layer(case, seed)
    if kind == "mlp":
        return _exact_mlp(case, seed)
    if kind == "head":
        return _exact_head(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    s = prepare(case, seed)
    H, K, d = case["heads"], case["kv"], case["dim"]
    q, k, v, g = (torch.from_numpy(s[n]).to(DEV, torch.float64).view(1, case["seq"], h, d)
                  for n, h in (("q", H), ("k", K), ("v", K), ("g", H)))
    return [t.reshape(-1) for t in _attn64(q, k, v, g)]
