"""Performance cases: the work that programs on this framework have it do, each a call or a short
sequence of calls through its public entry points (the torch-tensor binding of the C-ABI and the
native ``cuda_transformer`` module).

``listed()`` names the fixed cases, ``draw(rng)`` gives one more of the same ranges,
``prepare(case, seed)`` makes what a program holds before the call, ``run(state)`` makes one pass,
``work(case)`` is the least a pass must move and compute, ``exact(case, seed)`` is the same result
in 64-bit torch, and ``tolerance(case)`` bounds another correct implementation's difference.

Six kinds of case:
  attn   scaled-dot-product attention on [B, H, T, d], forward alone or forward + backward
  layer  the attention layer: QKV projection, attention, output projection, and their backward
  mlp    linear -> activation -> linear and its backward (weight and bias gradients included)
  norm   LayerNorm and its backward
  head   the language-model head: projection to the vocabulary, softmax, cross-entropy, backward
  gpt    the native NanoGPT, from token ids on the host to probabilities on the host
"""
import math

import numpy as np
import torch

import cudatransformer_amd as ct
from cudatransformer_amd import _capi

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_ACTS = {"relu": _capi.ACT_RELU, "gelu": _capi.ACT_GELU, "sigmoid": _capi.ACT_SIGMOID, "tanh": _capi.ACT_TANH}
_LN_EPS = 1e-5


def listed():
    return [
        # The smallest call: one short fp32 forward, all launch and host latency.
        dict(name="attn-infer-f32-small", kind="attn", dtype="f32", B=1, H=4, T=128, d=32, causal=True,
             train=False, keep_workspace=False),
        # The benchmark's headline: fp32 causal training attention.
        dict(name="attn-train-f32", kind="attn", dtype="f32", B=8, H=12, T=1024, d=64, causal=True, train=True,
             keep_workspace=False),
        # Long-context 16-bit training (the benchmark's bf16 shape), its workspace kept from step to
        # step as a training loop does: the largest case.
        dict(name="attn-train-bf16-long", kind="attn", dtype="bf16", B=1, H=32, T=8192, d=128, causal=True,
             train=True, keep_workspace=True),
        # A head dim between the native widths and a ragged length.
        dict(name="attn-train-bf16-d80", kind="attn", dtype="bf16", B=2, H=16, T=2000, d=80, causal=True,
             train=True, keep_workspace=False),
        # Wide heads, the largest head dim the attention takes, unmasked (an encoder).
        dict(name="attn-train-bf16-d256", kind="attn", dtype="bf16", B=2, H=8, T=1024, d=256, causal=False,
             train=True, keep_workspace=False),
        # The benchmark's attention layer in 16-bit storage.
        dict(name="layer-train-bf16", kind="layer", dtype="bf16", B=8, T=1024, E=1024, H=16, d=64, causal=False),
        # The same layer on sequences that are no multiple of any tile: whole documents as they come.
        dict(name="layer-train-bf16-ragged", kind="layer", dtype="bf16", B=4, T=1001, E=768, H=12, d=64,
             causal=True),
        # The MLP of the benchmark's small GPT (16 x 256 tokens, fp32).
        dict(name="mlp-train-f32", kind="mlp", dtype="f32", M=4096, K=384, N=1536, act="gelu"),
        # The MLP beside the benchmark's attention layer, 16-bit, four times as wide.
        dict(name="mlp-train-bf16", kind="mlp", dtype="bf16", M=8192, K=1024, N=4096, act="gelu"),
        # The normalisation in front of a wide 16-bit layer.
        dict(name="norm-train-bf16", kind="norm", dtype="bf16", N=8192, D=2048),
        # A language model's head over a real tokenizer's vocabulary (an odd one).
        dict(name="head-train-bf16", kind="head", dtype="bf16", N=2048, E=768, V=50257),
        # Scoring one prompt with the benchmark's small GPT on the native host.
        dict(name="gpt-score-f32", kind="gpt", dtype="f32", B=1, T=256, E=384, H=6, layers=6, V=65),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ---- attn -----------------------------------------------------------------------------------


def _draw_attn(rng):
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    d = rng.choice([32, 64, 64, 64, 128, 128, 128, 40, 48, 72, 80, 96, 96, 100, 112, 160, 192, 256])
    train = rng.random() < 0.7
    causal = rng.random() < 0.6
    # Head dims above 128 are used at moderate lengths; fp32 is a small model's type.
    most = 4e10 if d > 128 else (1e11 if dtype == "f32" else 8e11)
    while True:
        B, H, T = _log(rng, 1, 16), rng.choice([1, 2, 4, 6, 8, 12, 16, 20, 32]), _log(rng, 16, 8192)
        case = dict(kind="attn", dtype=dtype, B=B, H=H, T=T, d=d, causal=causal, train=train,
                    keep_workspace=bool(train and T >= 2048))
        if work(case)["flops"] <= most:
            return case


def _attn_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    std = 0.5 if c["T"] > 2048 else 1.0  # the benchmark's: unit normal, half of it for long context
    shape = (c["B"], c["H"], c["T"], c["d"])
    n = 4 if c["train"] else 3
    return [(std * torch.randn(shape, generator=g, device="cuda")).to(_DTYPES[c["dtype"]]) for _ in range(n)]


def _prepare_attn(c, seed):
    ws = None
    if c["keep_workspace"]:
        need = ct.bwd_workspace_bytes(_DTYPES[c["dtype"]], c["B"], c["H"], c["T"], c["d"], c["causal"], fastest=True)
        ws = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    return dict(x=_attn_inputs(c, seed), causal=c["causal"], train=c["train"], workspace=ws)


def _run_attn(s):
    q, k, v = s["x"][:3]
    o, lse = ct.flash_attn_fwd(q, k, v, causal=s["causal"])
    if not s["train"]:
        return o, lse
    dq, dk, dv = ct.flash_attn_bwd(q, k, v, o, s["x"][3], lse, causal=s["causal"], workspace=s["workspace"])
    return o, lse, dq, dk, dv


def _attention64(q, k, v, do, causal):
    """O, LSE and (with do) dQ, dK, dV of attention in the inputs' type, head by head."""
    B, H, T, d = q.shape
    outs = [torch.empty_like(q), q.new_empty((B, H, T))] + [torch.empty_like(q) for _ in range(3 if do is not None else 0)]
    mask = torch.ones((T, T), dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(B):
        for h in range(H):
            s = (q[b, h] @ k[b, h].t()) / math.sqrt(d)
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            lse = torch.logsumexp(s, -1, keepdim=True)
            p = torch.exp_(s - lse)
            o = p @ v[b, h]
            outs[0][b, h], outs[1][b, h] = o, lse[:, 0]
            if do is not None:
                g = do[b, h]
                ds = p * (g @ v[b, h].t() - (g * o).sum(-1, keepdim=True)) / math.sqrt(d)
                outs[2][b, h], outs[3][b, h], outs[4][b, h] = ds @ k[b, h], ds.t() @ q[b, h], p.t() @ g
    return outs


def _exact_attn(c, seed):
    x = [t.double() for t in _attn_inputs(c, seed)]
    return tuple(_attention64(*x[:3], x[3] if c["train"] else None, c["causal"]))


def _attn_flops(c):
    pairs = c["T"] * (c["T"] + 1) / 2 if c["causal"] else c["T"] ** 2
    return 4.0 * c["B"] * c["H"] * pairs * c["d"]


def _work_attn(c):
    el = c["B"] * c["H"] * c["T"] * c["d"] * _DTYPES[c["dtype"]].itemsize
    # q, k, v (and dO) read, O, LSE (and dQ, dK, dV) written; the backward is 2.5 forwards.
    return dict(bytes=el * (8 if c["train"] else 4) + 4 * c["B"] * c["H"] * c["T"],
                flops=_attn_flops(c) * (3.5 if c["train"] else 1.0))


# ---- layer ----------------------------------------------------------------------------------


def _draw_layer(rng):
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    most = 1.2e11 if dtype == "f32" else 4e11
    while True:
        H, d = rng.choice([4, 6, 8, 12, 16]), rng.choice([32, 48, 64, 64, 80, 128])
        E = rng.choice([H * d, H * d, 256, 384, 768, 1024])
        case = dict(kind="layer", dtype=dtype, B=_log(rng, 1, 16), T=_log(rng, 24, 2048), E=E, H=H, d=d,
                    causal=rng.random() < 0.5)
        if work(case)["flops"] <= most:
            return case


def _layer_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, E, I = _DTYPES[c["dtype"]], c["E"], c["H"] * c["d"]

    def normal(*shape, std=1.0):
        return (std * torch.randn(shape, generator=g, device="cuda")).to(dt)

    x, dy = normal(c["B"], c["T"], E), normal(c["B"], c["T"], E)  # a normalised input, an upstream gradient
    w = [normal(I, E, std=1.2 / math.sqrt(E)) for _ in range(3)] + [normal(E, I, std=1.0 / math.sqrt(I))]
    b = [normal(I, std=0.02) for _ in range(3)] + [normal(E, std=0.02)]
    return x, dy, w, b


def _prepare_layer(c, seed):
    x, dy, w, b = _layer_inputs(c, seed)
    # The Q, K and V bias gradients side by side in one buffer: the key bias moves every score of a
    # row alike, so its own gradient is 0 but for rounding and means something only beside the others.
    return dict(x=x, dy=dy, w=w, b=b, dw=[torch.empty_like(t) for t in w], H=c["H"], d=c["d"], causal=c["causal"],
                db_qkv=x.new_empty((3, c["H"] * c["d"])), db_out=torch.empty_like(b[3]))


def _run_layer(s):
    x, w, b, dw = s["x"], s["w"], s["b"], s["dw"]
    _capi.zero_multi([*dw, s["db_qkv"], s["db_out"]])  # the step's zero_grad: the backward accumulates
    q, k, v = ct.qkv_proj_fwd(x, *w[:3], *b[:3], s["H"], s["d"])
    o, lse = ct.flash_attn_fwd(q, k, v, causal=s["causal"])
    y = ct.out_proj_fwd(o, w[3], b[3])
    do = ct.out_proj_bwd(o, s["dy"], w[3], dw[3], s["db_out"])
    dq, dk, dv = ct.flash_attn_bwd(q, k, v, o, do, lse, causal=s["causal"])
    dx = ct.qkv_proj_bwd(x, dq, dk, dv, *w[:3], dw=tuple(dw[:3]), db=tuple(s["db_qkv"].unbind(0)))
    return (y, dx, *dw, s["db_qkv"], s["db_out"])


def _exact_layer(c, seed):
    x, dy, w, b = _layer_inputs(c, seed)
    B, T, H, d = c["B"], c["T"], c["H"], c["d"]
    x, dy = x.double().reshape(B * T, -1), dy.double().reshape(B * T, -1)
    w, b = [t.double() for t in w], [t.double() for t in b]

    def split(t):
        return t.reshape(B, T, H, d).transpose(1, 2).contiguous()

    def merge(t):
        return t.transpose(1, 2).reshape(B * T, H * d)

    q, k, v = (split(x @ w[i].t() + b[i]) for i in range(3))
    do = split(dy @ w[3])
    o, _, dq, dk, dv = _attention64(q, k, v, do, c["causal"])
    o, g = merge(o), [merge(t) for t in (dq, dk, dv)]
    y = o @ w[3].t() + b[3]
    dx = sum(g[i] @ w[i] for i in range(3))
    dw = [g[i].t() @ x for i in range(3)] + [dy.t() @ o]
    return (y.reshape(B, T, -1), dx.reshape(B, T, -1), *dw, torch.stack([t.sum(0) for t in g]), dy.sum(0))


def _work_layer(c):
    rows, E, I, it = c["B"] * c["T"], c["E"], c["H"] * c["d"], _DTYPES[c["dtype"]].itemsize
    # x, dy, y, dx; every weight and its gradient; every bias and its gradient.
    return dict(bytes=it * (4 * rows * E + 2 * 4 * E * I + 2 * (3 * I + E)),
                flops=3 * 2.0 * rows * E * I * 4 + 3.5 * _attn_flops(c))


# ---- mlp ------------------------------------------------------------------------------------


def _draw_mlp(rng):
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    most = 1e11 if dtype == "f32" else 4e11
    while True:
        K = rng.choice([64, 96, 200, 256, 384, 512, 768, 1000, 1024, 1600, 2048])
        N = rng.choice([4 * K, 4 * K, 2 * K, 8 * K // 3])
        case = dict(kind="mlp", dtype=dtype, M=_log(rng, 1, 16384), K=K, N=N,
                    act=rng.choice(["gelu", "gelu", "relu", "tanh", "sigmoid"]))
        if work(case)["flops"] <= most:
            return case


def _mlp_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, M, K, N = _DTYPES[c["dtype"]], c["M"], c["K"], c["N"]

    def normal(*shape, std=1.0):
        return (std * torch.randn(shape, generator=g, device="cuda")).to(dt)

    return (normal(M, K), normal(M, K), [normal(N, K, std=1 / math.sqrt(K)), normal(K, N, std=1 / math.sqrt(N))],
            [normal(N, std=0.1), normal(K, std=0.1)])


def _prepare_mlp(c, seed):
    x, dy, w, b = _mlp_inputs(c, seed)
    return dict(x=x, dy=dy, w=w, b=b, dw=[torch.empty_like(t) for t in w], db=[torch.empty_like(t) for t in b],
                act=_ACTS[c["act"]])


def _run_mlp(s):
    x, w, b, dw, db = s["x"], s["w"], s["b"], s["dw"], s["db"]
    _capi.zero_multi(dw + db)
    pre, h = _capi.linear_act_fwd(x, w[0], b[0], s["act"])
    y = _capi.linear_fwd(h, w[1], b[1])
    dpre = _capi.linear_act_bwd(h, w[1], s["dy"], pre, s["act"], dw=dw[1], db=db[1])
    dx = _capi.linear_bwd(x, w[0], dpre, dw=dw[0], db=db[0])
    return (y, dx, *dw, *db)


def _act64(kind, x):
    """act(x) and act'(x)."""
    if kind == "relu":
        return torch.relu(x), (x > 0).to(x.dtype)
    if kind == "sigmoid":
        y = torch.sigmoid(x)
        return y, y * (1 - y)
    if kind == "tanh":
        y = torch.tanh(x)
        return y, 1 - y * y
    a, b = math.sqrt(2 / math.pi), 0.044715
    t = torch.tanh(a * (x + b * x ** 3))
    return 0.5 * x * (1 + t), 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * a * (1 + 3 * b * x * x)


def _exact_mlp(c, seed):
    x, dy, w, b = _mlp_inputs(c, seed)
    x, dy, w, b = x.double(), dy.double(), [t.double() for t in w], [t.double() for t in b]
    h, slope = _act64(c["act"], x @ w[0].t() + b[0])
    y = h @ w[1].t() + b[1]
    dpre = (dy @ w[1]) * slope
    return (y, dpre @ w[0], dpre.t() @ x, dy.t() @ h, dpre.sum(0), dy.sum(0))


def _work_mlp(c):
    M, K, N, it = c["M"], c["K"], c["N"], _DTYPES[c["dtype"]].itemsize
    # x, dy, y, dx; both weights and biases and their gradients.  Three products per weight.
    return dict(bytes=it * (4 * M * K + 4 * N * K + 2 * (N + K)), flops=6 * 2.0 * M * K * N)


# ---- norm -----------------------------------------------------------------------------------


def _draw_norm(rng):
    while True:
        D = rng.choice([65, 96, 128, 256, 384, 512, 768, 1000, 1024, 1536, 2048, 3072, 4096, 5120, 8192])
        case = dict(kind="norm", dtype=rng.choice(["f32", "bf16", "bf16", "f16"]), N=_log(rng, 1, 65536), D=D)
        if case["N"] * D <= 1 << 26:
            return case


def _norm_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, N, D = _DTYPES[c["dtype"]], c["N"], c["D"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    # Activations with a mean and a spread of their own per row, a scale near 1, a small shift.
    x = normal(N, D) * (0.5 + normal(N, 1).abs()) + 0.5 * normal(N, 1)
    return x.to(dt), normal(N, D).to(dt), (1 + 0.1 * normal(D)).to(dt), (0.1 * normal(D)).to(dt)


def _prepare_norm(c, seed):
    x, dy, gamma, beta = _norm_inputs(c, seed)
    return dict(x=x, dy=dy, gamma=gamma, beta=beta, dg=torch.empty_like(gamma), db=torch.empty_like(beta))


def _run_norm(s):
    _capi.zero_multi([s["dg"], s["db"]])
    y, mean, rstd = _capi.layernorm_fwd(s["x"], s["gamma"], s["beta"], _LN_EPS)
    dx = _capi.layernorm_bwd(s["x"], s["gamma"], s["dy"], mean, rstd, dgamma=s["dg"], dbeta=s["db"])
    return y, mean, rstd, dx, s["dg"], s["db"]


def _exact_norm(c, seed):
    x, dy, gamma, beta = (t.double() for t in _norm_inputs(c, seed))
    mean = x.mean(-1, keepdim=True)
    rstd = torch.rsqrt(((x - mean) ** 2).mean(-1, keepdim=True) + _LN_EPS)
    xh = (x - mean) * rstd
    g = dy * gamma
    dx = rstd * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
    return xh * gamma + beta, mean[:, 0], rstd[:, 0], dx, (dy * xh).sum(0), dy.sum(0)


def _work_norm(c):
    n, it = c["N"] * c["D"], _DTYPES[c["dtype"]].itemsize
    # x, dy read, y, dx written; gamma, beta and their gradients; mean and rstd written.
    return dict(bytes=it * (4 * n + 4 * c["D"]) + 8 * c["N"], flops=20.0 * n)


# ---- head -----------------------------------------------------------------------------------


def _draw_head(rng):
    # No fp16: without a loss scale its gradients of a large vocabulary underflow.
    dtype = rng.choice(["f32", "bf16", "bf16"])
    while True:
        case = dict(kind="head", dtype=dtype, N=_log(rng, 8, 8192), E=rng.choice([256, 384, 512, 768, 1024]),
                    V=rng.choice([65, 65, 256, 1000, 5003, 32000, 32768, 50257]))
        if work(case)["flops"] <= (6e10 if dtype == "f32" else 3e11):
            return case


def _head_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[c["dtype"]]
    x = torch.randn((c["N"], c["E"]), generator=g, device="cuda").to(dt)  # a normalised last layer
    w = (torch.randn((c["V"], c["E"]), generator=g, device="cuda") / math.sqrt(c["E"])).to(dt)
    t = torch.randint(0, c["V"], (c["N"],), generator=g, device="cuda", dtype=torch.int32)
    return x, w, t


def _prepare_head(c, seed):
    x, w, t = _head_inputs(c, seed)
    return dict(x=x, w=w, t=t, dw=torch.empty_like(w))


def _run_head(s):
    _capi.zero_multi([s["dw"]])
    z = _capi.linear_fwd(s["x"], s["w"])
    p = _capi.softmax_fwd(z)
    loss = _capi.cross_entropy_fwd(p, s["t"])
    dz = _capi.softmax_cross_entropy_bwd(p, s["t"])
    dx = _capi.linear_bwd(s["x"], s["w"], dz, dw=s["dw"])
    return z, p, loss, dx, s["dw"]


def _exact_head(c, seed):
    x, w, t = _head_inputs(c, seed)
    x, w, rows, t = x.double(), w.double(), torch.arange(c["N"], device="cuda"), t.long()
    z = x @ w.t()
    p = torch.softmax(z, -1)
    loss = -torch.log(p[rows, t]) / c["N"]
    dz = p / c["N"]
    dz[rows, t] -= 1.0 / c["N"]
    return z, p, loss, dz @ w, dz.t() @ x


def _work_head(c):
    N, E, V, it = c["N"], c["E"], c["V"], _DTYPES[c["dtype"]].itemsize
    # x, w read, the logits, the probabilities, dx and dw written, targets and losses.
    return dict(bytes=it * (2 * N * E + 2 * V * E + 2 * N * V) + 8 * N, flops=3 * 2.0 * N * E * V)


# ---- gpt ------------------------------------------------------------------------------------


def _draw_gpt(rng):
    H = rng.choice([2, 4, 6, 8])
    return dict(kind="gpt", dtype=rng.choice(["f32", "f32", "bf16"]), B=rng.choice([1, 1, 1, 2, 4, 8]),
                T=_log(rng, 4, 256), E=64 * H, H=H, layers=rng.randint(1, 8), V=rng.choice([65, 65, 256, 1000]))


_GPT_MAX_LEN = 256


def _gpt_weights(c, seed):
    """Parameters by the native model's names, as numpy arrays: a model whose blocks have learnt
    something (weights well above their initial 0.02), so that the probabilities are not flat."""
    rng = np.random.default_rng(seed)
    E, F = c["E"], 4 * c["E"]

    def normal(*shape, std):
        return (std * rng.standard_normal(shape, dtype=np.float32)).astype(np.float32)

    p = {"tokenEmbedding": normal(c["V"], E, std=0.5), "positionEmbedding": normal(_GPT_MAX_LEN, E, std=0.2),
         "unEmbedding": normal(c["V"], E, std=1.0 / math.sqrt(E))}
    for i in range(c["layers"]):
        for n in ("query", "key", "value", "output"):
            p[f"layer_{i}.attention.{n}.weights"] = normal(E, E, std=1.0 / math.sqrt(E))
            p[f"layer_{i}.attention.{n}.biases"] = normal(E, std=0.02)
        for n in ("firstNorm", "secondNorm"):
            p[f"layer_{i}.{n}.weights"] = (1 + normal(E, std=0.1)).astype(np.float32)
            p[f"layer_{i}.{n}.biases"] = normal(E, std=0.1)
        p[f"layer_{i}.mlp.layer_0.weights"] = normal(F, E, std=1.0 / math.sqrt(E))
        p[f"layer_{i}.mlp.layer_0.biases"] = normal(F, std=0.02)
        p[f"layer_{i}.mlp.layer_2.weights"] = normal(E, F, std=1.0 / math.sqrt(E))
        p[f"layer_{i}.mlp.layer_2.biases"] = normal(E, std=0.02)
    ids = rng.integers(0, c["V"], (c["B"], c["T"]), dtype=np.int32)
    return p, ids


def _prepare_gpt(c, seed):
    from cudatransformer_amd import cuda_transformer as ctm

    name = {"f32": "Float", "bf16": "BFloat"}[c["dtype"]]
    p, ids = _gpt_weights(c, seed)
    model = getattr(ctm, name + "NanoGPT")(c["V"], _GPT_MAX_LEN, c["E"], c["H"], c["E"] // c["H"], 4 * c["E"],
                                           c["layers"], activation_type=ctm.ActivationType.GELU, causal=True)
    tensor = getattr(ctm, name + "Tensor")
    model.setParameters({n: tensor.fromNumpy(a) for n, a in p.items()})
    return dict(model=model, ids=ids)


def _run_gpt(s):
    return s["model"](s["ids"]).numpy()


def _exact_gpt(c, seed):
    p, ids = _gpt_weights(c, seed)
    p = {n: torch.from_numpy(a).cuda().to(_DTYPES[c["dtype"]]).double() for n, a in p.items()}
    B, T, E, H = c["B"], c["T"], c["E"], c["H"]

    def norm(x, n):
        return torch.nn.functional.layer_norm(x, (E,), p[n + ".weights"], p[n + ".biases"], _LN_EPS)

    def linear(x, n):
        return x @ p[n + ".weights"].t() + p[n + ".biases"]

    def heads(x):
        return x.reshape(B, T, H, E // H).transpose(1, 2).contiguous()

    x = (p["tokenEmbedding"][torch.from_numpy(ids).cuda().long()] + p["positionEmbedding"][:T]).reshape(B * T, E)
    for i in range(c["layers"]):
        a = norm(x, f"layer_{i}.firstNorm")
        q, k, v = (heads(linear(a, f"layer_{i}.attention.{n}")) for n in ("query", "key", "value"))
        o = _attention64(q, k, v, None, True)[0].transpose(1, 2).reshape(B * T, E)
        x = norm(linear(o, f"layer_{i}.attention.output"), f"layer_{i}.secondNorm")
        x = linear(_act64("gelu", linear(x, f"layer_{i}.mlp.layer_0"))[0], f"layer_{i}.mlp.layer_2")
    return torch.softmax(x @ p["unEmbedding"].t(), -1).reshape(B, T, c["V"]).cpu().numpy()


def _work_gpt(c):
    rows, E, it = c["B"] * c["T"], c["E"], _DTYPES[c["dtype"]].itemsize
    weights = c["layers"] * 12 * E * E + c["V"] * E
    pairs = c["T"] * (c["T"] + 1) / 2
    # Every weight and the used embedding rows read once, ids in, probabilities out.
    return dict(bytes=it * (weights + 2 * rows * E + rows * c["V"]) + 4 * rows,
                flops=2.0 * rows * weights + c["layers"] * 4.0 * c["B"] * pairs * E)


# ---- the interface --------------------------------------------------------------------------

_DRAW = {"attn": _draw_attn, "layer": _draw_layer, "mlp": _draw_mlp, "norm": _draw_norm, "head": _draw_head,
         "gpt": _draw_gpt}
_PREPARE = {"attn": _prepare_attn, "layer": _prepare_layer, "mlp": _prepare_mlp, "norm": _prepare_norm,
            "head": _prepare_head, "gpt": _prepare_gpt}
_RUN = {"attn": _run_attn, "layer": _run_layer, "mlp": _run_mlp, "norm": _run_norm, "head": _run_head,
        "gpt": _run_gpt}
_EXACT = {"attn": _exact_attn, "layer": _exact_layer, "mlp": _exact_mlp, "norm": _exact_norm, "head": _exact_head,
          "gpt": _exact_gpt}
_WORK = {"attn": _work_attn, "layer": _work_layer, "mlp": _work_mlp, "norm": _work_norm, "head": _work_head,
         "gpt": _work_gpt}


def draw(rng):
    return _DRAW[rng.choice(["attn", "attn", "attn", "layer", "layer", "mlp", "mlp", "norm", "head", "gpt"])](rng)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed) | dict(kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


# About four times the largest relative error against exact() seen over the listed and drawn cases
# of each kind and storage type.  The whole 16-bit model carries every layer's rounding on.
_REL = {
    "attn": dict(f32=3e-6, bf16=1.2e-2, f16=1.5e-3),
    "layer": dict(f32=5e-6, bf16=2e-2, f16=3e-3),
    "mlp": dict(f32=3e-6, bf16=1.2e-2, f16=1.6e-3),
    "norm": dict(f32=1e-6, bf16=7e-3, f16=1e-3),
    "head": dict(f32=6e-6, bf16=1.6e-2),
    "gpt": dict(f32=7e-6, bf16=3e-2),
}


def tolerance(case):
    return {"rel": _REL[case["kind"]][case["dtype"]]}
