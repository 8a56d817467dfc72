"""Performance cases of the framework: what is timed, on which inputs, and how close results must be.

A case is one pass through a public entry point: an attention call, a linear layer, the GPT's
MLP, a residual add with its LayerNorm, a row softmax, or one whole GPT training step.  Sizes
are those of the repository's benchmark workloads and tests, from its smallest ragged calls to
its long-sequence sweep; ``draw`` spreads more of them over the same ranges.
"""
import math

import torch

from cuda_transformer_amd import autograd_fns, gpt, ops

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def listed():
    return [
        # The smallest call: one short prompt's attention, forward only (launch latency).
        dict(name="attn_short_prompt", kind="attention", B=1, H=4, T=65, D=64, causal=True,
             dtype="float32", train=False),
        # One layer of the small GPT: attention on its packed qkv projection, a training step.
        dict(name="attn_gpt_layer", kind="attention_qkv", B=64, H=6, T=256, D=64, train=True),
        # Training at long context, FP32 causal: the benchmark's headline shape.
        dict(name="attn_causal_4k", kind="attention", B=4, H=32, T=4096, D=64, causal=True,
             dtype="float32", train=True),
        # Bidirectional (encoder) training at twice that length: the long end of the sweep.
        dict(name="attn_full_8k", kind="attention", B=4, H=32, T=8192, D=64, causal=False,
             dtype="float32", train=True),
        # Wide heads at a length that no tile divides.
        dict(name="attn_wide_head_odd", kind="attention", B=2, H=16, T=1999, D=128, causal=True,
             dtype="float32", train=True),
        # Mixed-precision training at the headline shape.
        dict(name="attn_bf16_4k", kind="attention", B=4, H=32, T=4096, D=64, causal=True,
             dtype="bfloat16", train=True),
        # A linear layer of a 768-wide model over 8192 tokens (its up projection), forward and
        # backward with weight and bias gradients.
        dict(name="linear_up", kind="linear", B=8, M=1024, K=768, N=3072, train=True),
        # A few short sequences through a layer whose sizes are not multiples of 4.
        dict(name="linear_odd", kind="linear", B=3, M=65, K=385, N=1155, train=True),
        # The small GPT's MLP over a training batch.
        dict(name="mlp_gpt", kind="mlp", B=64, M=256, K=384, N=1536),
        # Residual add + LayerNorm of a 768-wide model over 8192 tokens, both directions.
        dict(name="add_layernorm", kind="add_layernorm", B=8, M=1024, N=768),
        # Row softmax of materialised attention scores (48 heads of 1024 x 1024).
        dict(name="softmax_rows", kind="softmax", B=48, M=1024, N=1024),
        # One training step of the small character GPT: logits, loss and every layer's gradients.
        dict(name="gpt_step", kind="gpt", B=64, T=256, H=6, D=64, L=6, V=65),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "attention_qkv", "linear", "linear",
                       "mlp", "add_layernorm", "softmax", "gpt"])
    if kind == "attention":
        T, D = _log(rng, 65, 8192), rng.choice([32, 64, 64, 128])
        # B H T^2 D stays below the longest listed case's
        heads = max(1, min(128, int(128 * 8192**2 * 64 / (T * T * D))))
        BH = _log(rng, min(4, heads), heads)
        B = rng.choice([b for b in (1, 2, 4) if b <= BH])
        return dict(kind=kind, B=B, H=BH // B, T=T, D=D, causal=rng.random() < 0.6,
                    dtype=rng.choice(["float32", "float32", "bfloat16"]),
                    train=rng.random() < 0.75)
    if kind == "attention_qkv":
        T = _log(rng, 64, 2048)
        return dict(kind=kind, B=max(1, _log(rng, 1, 16384 * 2 // T)), H=rng.choice([4, 6, 8, 12]),
                    T=T, D=rng.choice([32, 64, 128]), train=rng.random() < 0.75)
    if kind in ("linear", "mlp"):
        rows, K = _log(rng, 130, 16384), _log(rng, 128, 2048)
        N = 4 * K if kind == "mlp" else _log(rng, 128, 4096)
        if rng.random() < 0.6:  # model widths are mostly multiples of 64
            K, N = max(64, K // 64 * 64), max(64, N // 64 * 64)
        B = rng.choice([1, 2, 4, 8])
        case = dict(kind=kind, B=B, M=max(1, rows // B), K=K, N=N)
        if kind == "linear":
            case["train"] = rng.random() < 0.75
        return case
    if kind == "add_layernorm":
        return dict(kind=kind, B=rng.choice([1, 2, 4, 8]), M=_log(rng, 33, 4096),
                    N=_log(rng, 128, 4096))
    if kind == "softmax":
        return dict(kind=kind, B=_log(rng, 1, 48), M=_log(rng, 17, 1024), N=_log(rng, 64, 4096))
    H = rng.choice([2, 4, 6])
    return dict(kind=kind, B=_log(rng, 4, 64), T=_log(rng, 65, 256), H=H, D=64,
                L=rng.choice([2, 4, 6]), V=rng.choice([65, 65, 256, 1000]))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    x = torch.randn(*shape, generator=g, device="cuda")
    return (x.mul_(std) if std != 1.0 else x).to(dtype)


# Gradients that reach a layer in training are small: means over a batch of tokens.
GRAD_STD = 1e-3


def _inputs(case, seed):
    """The tensors of a case by name: leaves first, then the gradient of its output."""
    g, k = _gen(seed), case["kind"]
    if k == "attention":
        shape, dt = (case["B"], case["H"], case["T"], case["D"]), DTYPES[case["dtype"]]
        return {n: _randn(g, *shape, dtype=dt) for n in ("q", "k", "v", "dy")}
    if k == "attention_qkv":
        C = case["H"] * case["D"]
        return {"qkv": _randn(g, case["B"], case["T"], 3 * C),
                "dy": _randn(g, case["B"], case["T"], C, std=GRAD_STD)}
    if k in ("linear", "mlp"):
        B, M, K, N = (case[n] for n in ("B", "M", "K", "N"))
        t = {"x": _randn(g, B, M, K), "w1": _randn(g, K, N, std=K**-0.5),
             "b1": _randn(g, N, std=0.02)}
        if k == "mlp":
            t["w2"], t["b2"] = _randn(g, N, K, std=N**-0.5), _randn(g, K, std=0.02)
        t["dy"] = _randn(g, B, M, K if k == "mlp" else N, std=GRAD_STD)
        return t
    if k == "add_layernorm":
        shape = (case["B"], case["M"], case["N"])
        return {"x": _randn(g, *shape), "f": _randn(g, *shape, std=0.3),
                "gamma": 1.0 + _randn(g, case["N"], std=0.1), "beta": _randn(g, case["N"], std=0.1),
                "dsum": _randn(g, *shape, std=GRAD_STD), "dy": _randn(g, *shape, std=GRAD_STD)}
    shape = (case["B"], case["M"], case["N"])
    return {"x": _randn(g, *shape, std=2.0), "dy": _randn(g, *shape, std=GRAD_STD)}


def _gpt_config(case):
    return gpt.GPTConfig(vocab_size=case["V"], d_model=case["H"] * case["D"], n_heads=case["H"],
                         n_layers=case["L"], block_size=case["T"])


def _gpt_inputs(case, seed):
    """Parameters by the reference GPT's names, token ids and targets."""
    g, C, V, T = _gen(seed), case["H"] * case["D"], case["V"], case["T"]
    p = {"embedding.embedding.weight": (V, C), "embedding.positional.weight": (T, C)}
    for i in range(case["L"]):
        b = "mha.%d." % i
        p.update({b + "ln1.alpha": (C,), b + "ln1.beta": (C,), b + "attn.qkv_weight": (C, 3 * C),
                  b + "attn.qkv_bias": (3 * C,), b + "attn.out_weight": (C, C),
                  b + "attn.out_bias": (C,), b + "ln2.alpha": (C,), b + "ln2.beta": (C,),
                  b + "mlp.fc1_weights": (C, 4 * C), b + "mlp.fc1_bias": (4 * C,),
                  b + "mlp.fc2_weights": (4 * C, C), b + "mlp.fc2_bias": (C,)})
    p.update({"ln.alpha": (C,), "ln.beta": (C,), "lm_head_weights": (C, V), "lm_head_bias": (V,)})
    p = {n: _randn(g, *s, std=0.02).add_(1.0 if n.endswith("alpha") else 0.0) for n, s in p.items()}
    ids = torch.randint(0, V, (case["B"], T + 1), generator=g, device="cuda")
    return p, ids[:, :-1].contiguous(), ids[:, 1:].contiguous()


def _gpt_returned(case, name):
    """Gradients that a step returns: every matrix, the vectors of the first and last block and
    of the head (62 tensors at most are compared)."""
    matrix = name.endswith(("weight", "weights"))
    return matrix or not name.startswith("mha.") or name.startswith(
        ("mha.0.", "mha.%d." % (case["L"] - 1)))


def prepare(case, seed):
    if case["kind"] == "gpt":
        p, ids, targets = _gpt_inputs(case, seed)
        model = gpt.GPT(_gpt_config(case)).cuda()
        with torch.no_grad():
            for n, q in model.named_parameters():
                q.copy_(p[n])
        return {"case": dict(case), "model": model, "ids": ids, "targets": targets}
    t = _inputs(case, seed)
    leaf = case.get("train", True)
    for n, x in t.items():
        x.requires_grad_(leaf and n not in ("dy", "dsum"))
    return {"case": dict(case), **t}


def run(state):
    case = state["case"]
    kind, train = case["kind"], case.get("train", True)
    if kind == "gpt":
        model = state["model"]
        for q in model.parameters():
            q.grad = None
        logits, loss = model(state["ids"], state["targets"])
        loss.backward()
        return {"logits": logits.detach(), "loss": loss.detach(),
                **{n: q.grad for n, q in model.named_parameters() if _gpt_returned(case, n)}}
    if kind == "attention":
        qkv = [state[n] for n in ("q", "k", "v")]
        if not train:
            return ops.flash_attention_fwd(*qkv, case["causal"])
        o, l = autograd_fns.CudaFlashAttention.apply(*qkv, case["causal"])
        return o.detach(), l.detach(), *torch.autograd.grad(o, qkv, state["dy"])
    if kind == "attention_qkv":
        if not train:
            return ops.flash_attention_qkv_fwd(state["qkv"], case["H"], True)
        o = autograd_fns.CudaFlashAttentionQKV.apply(state["qkv"], case["H"], True)
        return o.detach(), *torch.autograd.grad(o, [state["qkv"]], state["dy"])
    if kind == "linear":
        leaves = [state[n] for n in ("x", "w1", "b1")]
        if not train:
            return ops.cuda_fma(*leaves)
        y = autograd_fns.CudaLinearLayer.apply(*leaves)
        return y.detach(), *torch.autograd.grad(y, leaves, state["dy"])
    if kind == "mlp":
        leaves = [state[n] for n in ("x", "w1", "b1", "w2", "b2")]
        y = autograd_fns.CudaMLP.apply(*leaves)
        return y.detach(), *torch.autograd.grad(y, leaves, state["dy"])
    if kind == "add_layernorm":
        leaves = [state[n] for n in ("x", "f", "gamma", "beta")]
        s, y = autograd_fns.CudaAddLayerNorm.apply(*leaves)
        # x and f receive the same gradient
        return s.detach(), y.detach(), *torch.autograd.grad(
            [s, y], [leaves[0], *leaves[2:]], [state["dsum"], state["dy"]])
    y = autograd_fns.CudaSoftmaxLayer.apply(state["x"])
    return y.detach(), *torch.autograd.grad(y, [state["x"]], state["dy"])


def work(case):
    """Bytes of inputs read once and outputs written once, and the products' operations
    (attention by the usual count: 2 products forward, 5 backward, half of the scores causal)."""
    kind, train = case["kind"], case.get("train", True)
    if kind in ("attention", "attention_qkv"):
        B, H, T, D = (case[n] for n in ("B", "H", "T", "D"))
        size = 2 if case.get("dtype") == "bfloat16" else 4
        x, pairs = B * H * T * D * size, B * H * T * T * (0.5 if case.get("causal", True) else 1.0)
        return {"bytes": (8 if train else 4) * x + 4 * B * H * T,
                "flops": (7 if train else 2) * 2.0 * D * pairs}
    if kind in ("linear", "mlp"):
        M, K, N = case["B"] * case["M"], case["K"], case["N"]
        # x, y, dx, dy; an MLP has two layers' weights and gradients but no hidden tensor to read
        if kind == "mlp":
            return {"bytes": 4.0 * (4 * M * K + 4 * K * N + 2 * (K + N)), "flops": 12.0 * M * N * K}
        if train:
            return {"bytes": 4.0 * (2 * M * K + 2 * M * N + 2 * K * N + 2 * N), "flops": 6.0 * M * N * K}
        return {"bytes": 4.0 * (M * K + M * N + K * N + N), "flops": 2.0 * M * N * K}
    if kind == "add_layernorm":
        # x, f, their sum, y, both incoming gradients and the outgoing one; parameters
        M, N = case["B"] * case["M"], case["N"]
        return {"bytes": 4.0 * (7 * M * N + 4 * N), "flops": 20.0 * M * N}
    if kind == "softmax":
        n = case["B"] * case["M"] * case["N"]
        return {"bytes": 16.0 * n, "flops": 8.0 * n}
    rows, C, V, L = case["B"] * case["T"], case["H"] * case["D"], case["V"], case["L"]
    params = 12 * C * C * L + 2 * C * V + C * case["T"]
    return {"bytes": 8.0 * params + 4.0 * rows * V + 16.0 * rows,
            "flops": 6.0 * rows * (12 * C * C * L + C * V) + 7.0 * rows * case["T"] * C * L}


def tolerance(case):
    """About four times the error against ``exact`` measured for the path (largest over outputs:
    1.8e-6 for FP32 products over 8192 keys, 1.4e-7 for the row kernels, 2.5e-3 in bfloat16);
    a whole model adds the rounding that travels from layer to layer."""
    if case.get("dtype") == "bfloat16":
        return {"rel": 1e-2}
    if case["kind"] == "gpt":
        return {"rel": 2e-5}
    if case["kind"] in ("add_layernorm", "softmax"):
        return {"rel": 1e-6}
    return {"rel": 8e-6}


# ---- the same in 64 bits, plain torch ----

def _attention64(q, k, v, dy, causal):
    """One head: O, L and, with dy, dQ, dK, dV, all (T, D) or (T,) float64."""
    scale = q.shape[-1] ** -0.5
    s = (q @ k.mT).mul_(scale)
    if causal:
        i = torch.arange(s.shape[0], device=s.device)
        s.masked_fill_(i[None, :] > i[:, None], -math.inf)
    l = torch.logsumexp(s, -1)
    p = s.sub_(l[:, None]).exp_()
    o = p @ v
    if dy is None:
        return o, l
    dv = p.mT @ dy
    dp = dy @ v.mT
    ds = dp.sub_((dy * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
    return o, l, ds @ k, ds.mT @ q, dv


def _attention_heads64(q, k, v, dy, causal):
    """Over (B, H, T, D) inputs, a head at a time."""
    B, H = q.shape[:2]
    got = None
    for b in range(B):
        for h in range(H):
            r = _attention64(*(x[b, h].double() for x in (q, k, v)),
                             None if dy is None else dy[b, h].double(), causal)
            if got is None:
                got = [torch.empty(B, H, *x.shape, dtype=x.dtype, device=x.device) for x in r]
            for a, x in zip(got, r):
                a[b, h] = x
    return got


class _Heads64(torch.autograd.Function):
    """Packed causal attention (B, T, 3C) -> (B, T, C) in float64, a head at a time."""

    @staticmethod
    def _split(qkv, H):
        B, T, C3 = qkv.shape
        return [t.reshape(B, T, H, C3 // 3 // H).transpose(1, 2) for t in qkv.chunk(3, -1)]

    @staticmethod
    def _join(x):
        B, H, T, D = x.shape
        return x.transpose(1, 2).reshape(B, T, H * D)

    @staticmethod
    def forward(ctx, qkv, H):
        ctx.save_for_backward(qkv)
        ctx.H = H
        o, l = _attention_heads64(*_Heads64._split(qkv, H), None, True)
        ctx.mark_non_differentiable(l)
        return _Heads64._join(o), l

    @staticmethod
    def backward(ctx, dy, _):
        (qkv,) = ctx.saved_tensors
        B, T, C = dy.shape
        d = dy.reshape(B, T, ctx.H, C // ctx.H).transpose(1, 2)
        r = _attention_heads64(*_Heads64._split(qkv, ctx.H), d, True)
        return torch.cat([_Heads64._join(x) for x in r[2:]], -1), None


def _gelu64(x):
    return x * 0.5 * (1.0 + torch.erf(x * 0.5**0.5))


def _layernorm64(x, gamma, beta):
    m = x.mean(-1, keepdim=True)
    return (x - m) / ((x - m).square().mean(-1, keepdim=True) + 1e-5).sqrt() * gamma + beta


def _gpt64(case, seed):
    p, ids, targets = _gpt_inputs(case, seed)
    p = {n: x.double().requires_grad_() for n, x in p.items()}
    x = p["embedding.embedding.weight"][ids] + p["embedding.positional.weight"][: case["T"]]
    for i in range(case["L"]):
        w = lambda n, b="mha.%d." % i: p[b + n]  # noqa: E731
        z = _layernorm64(x, w("ln1.alpha"), w("ln1.beta"))
        a, _ = _Heads64.apply(z @ w("attn.qkv_weight") + w("attn.qkv_bias"), case["H"])
        x = x + a @ w("attn.out_weight") + w("attn.out_bias")
        z = _layernorm64(x, w("ln2.alpha"), w("ln2.beta"))
        z = _gelu64(z @ w("mlp.fc1_weights") + w("mlp.fc1_bias"))
        x = x + z @ w("mlp.fc2_weights") + w("mlp.fc2_bias")
    z = _layernorm64(x, p["ln.alpha"], p["ln.beta"])
    logits = z @ p["lm_head_weights"] + p["lm_head_bias"]
    loss = -torch.log_softmax(logits, -1).gather(-1, targets[..., None]).mean()
    loss.backward()
    return {"logits": logits.detach(), "loss": loss.detach(),
            **{n: q.grad for n, q in p.items() if _gpt_returned(case, n)}}


def exact(case, seed):
    kind, train = case["kind"], case.get("train", True)
    if kind == "gpt":
        return _gpt64(case, seed)
    t = _inputs(case, seed)
    if kind == "attention":
        return tuple(_attention_heads64(t["q"], t["k"], t["v"], t["dy"] if train else None,
                                        case["causal"]))
    t = {n: x.double() for n, x in t.items()}
    leaves = [x.requires_grad_() for n, x in t.items() if n not in ("dy", "dsum", "f")]
    if kind == "attention_qkv":
        y, l = _Heads64.apply(t["qkv"], case["H"])
        if not train:
            return y.detach(), l
    elif kind == "linear":
        y = t["x"] @ t["w1"] + t["b1"]
        if not train:
            return y.detach()
    elif kind == "mlp":
        y = _gelu64(t["x"] @ t["w1"] + t["b1"]) @ t["w2"] + t["b2"]
    elif kind == "add_layernorm":
        s = t["x"] + t["f"]
        y = _layernorm64(s, t["gamma"], t["beta"])
        return s.detach(), y.detach(), *torch.autograd.grad([s, y], leaves, [t["dsum"], t["dy"]])
    else:
        y = torch.softmax(t["x"], -1)
    return y.detach(), *torch.autograd.grad(y, leaves, t["dy"])
