"""Performance cases of prichs_amd: what a user's program has the framework do.

Each case is one call (or one training step) through the package's public
entry points, at the sizes of the repository's own configurations, tests and
benchmark, or generic ones.  Kinds:

* ``moe``    one MoE layer forward on an engine (``MoEEngine.forward``): decode
             steps, prompts, whole batches; bf16 or f32; with or without a
             concept bias; even or skewed routing.
* ``train``  one training step of the layer: a forward and its backward for
             each micro-batch, the first overwriting the f32 gradients and the
             others adding to them.
* ``block``  one transformer block forward (``BlockEngine.forward``): norms,
             projections, RoPE, causal GQA attention, residuals and the MoE.
* ``matmul`` one general f32 product (``ops.matmul_f32``): A B, A^T B or A B^T.

Weights are drawn N(0, 0.02), the activations N(0, 1) (row-normalised before
an MoE layer, as they are after its RMSNorm), and rounded to the layer's type.
"""
import math

import torch

from prichs_amd import _lib, block, moe, ops

EPS = 1e-5
SKEW = 1.0  # bias on experts 0 and 1 that sends them about 60% of the assignments


def _moe(name, T, d=1536, f=1280, E=8, k=2, dtype="bf16", skew=False, concept=False):
    return dict(name=name, kind="moe", T=T, d=d, f=f, E=E, k=k, dtype=dtype, skew=skew,
                concept=concept)


def _train(name, T, micro=1, d=1536, f=1280, E=8, k=2, dtype="bf16"):
    return dict(name=name, kind="train", T=T, micro=micro, d=d, f=f, E=E, k=k, dtype=dtype,
                skew=False, concept=False)


def _block(name, batch, S, d=1536, heads=12, kv=3, f=1280, E=8, k=2, pos=0):
    return dict(name=name, kind="block", batch=batch, S=S, pos=pos, heads=heads, kv=kv, d=d, f=f,
                E=E, k=k, dtype="bf16", skew=False, concept=False)


def _matmul(name, m, k, n, op):
    return dict(name=name, kind="matmul", m=m, k=k, n=n, op=op)


def listed():
    return [
        # One token of one sequence: the step of an interactive generation loop.
        _moe("decode_1", 1),
        # A decode step of 32 sequences.
        _moe("decode_32", 32),
        # A prompt of odd length, with the concept bias of the memory store.
        _moe("prompt_333", 333, concept=True),
        # The production layer over a batch of 4 x 2048 tokens.
        _moe("layer_8192", 8192),
        # Twice that batch, with experts 0 and 1 taking most of the tokens.
        _moe("layer_16384_skewed", 16384, skew=True),
        # The small f32 layer that results are checked against to 1e-4.
        _moe("layer_f32_512", 512, d=256, f=128, dtype="f32"),
        # A training step over a whole batch.
        _train("train_8192", 8192),
        # Gradient accumulation over two short micro-batches.
        _train("train_2x1000", 1000, micro=2),
        # A training step in the reference's own precision.
        _train("train_f32_2048", 2048, d=512, f=512, dtype="f32"),
        # A block forward over 4 x 2048 tokens.
        _block("block_4x2048", 4, 2048),
        # A block forward over one prompt of odd length.
        _block("block_1x777", 1, 777),
        # The general f32 product at the shape of one expert's projection.
        _matmul("matmul_f32_2048x1536x1280", 2048, 1536, 1280, "ab"),
    ]


def _loguniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "train", "train", "block", "block", "matmul"])
    if kind == "matmul":
        m, k, n = (_loguniform(rng, 16, 4096) for _ in range(3))
        return {**_matmul("", m, k, n, rng.choice(["ab", "atb", "abt"])), "name": "matmul"}
    E, k = rng.choice([(8, 2), (8, 2), (8, 2), (8, 1), (4, 2), (16, 2)])
    if kind == "block":
        d, heads, kv = rng.choice([(1536, 12, 3), (1536, 12, 3), (1024, 8, 2), (512, 4, 4)])
        S = _loguniform(rng, 1, 2048)
        batch = rng.randint(1, 4)
        return _block("block", batch, S, d=d, heads=heads, kv=kv,
                      f=rng.choice([1280, 1280, 64 * rng.randint(4, 20)]), E=E, k=k,
                      pos=rng.choice([0, 0, 37]))
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    if dtype == "bf16":
        d, f = rng.choice([(1536, 1280), (1536, 1280), (64 * rng.randint(4, 24),
                                                        64 * rng.randint(4, 20))])
    else:
        d, f = 16 * rng.randint(8, 32), 16 * rng.randint(8, 32)
    if kind == "moe":
        T = _loguniform(rng, 1, 16384 if dtype == "bf16" else 4096)
        return _moe("moe", T, d=d, f=f, E=E, k=k, dtype=dtype, skew=rng.random() < 0.25,
                    concept=rng.random() < 0.25)
    T = _loguniform(rng, 64, 4096 if dtype == "bf16" else 2048)
    return _train("train", T, micro=rng.choice([1, 2]), d=d, f=f, E=E, k=k, dtype=dtype)


# ------------------------------------------------------------------- inputs --
def _draws(case, seed):
    """The case's tensors on the GPU, from the seed alone: f32 values that are
    exact in the case's type."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    bf = case.get("dtype") == "bf16"

    def randn(*shape, std=1.0, mean=0.0, rounded=True):
        t = torch.randn(shape, generator=g, device="cuda") * std + mean
        return t.bfloat16().float() if bf and rounded else t

    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        a, b = {"ab": ((m, k), (k, n)), "atb": ((m, k), (m, n)), "abt": ((m, k), (n, k))}[
            case["op"]]
        return dict(a=randn(*a), b=randn(*b, std=0.02))
    d, f, E = case["d"], case["f"], case["E"]
    v = {}
    if case["kind"] == "block":
        hd, rows = d // case["heads"], case["batch"] * case["S"]
        v["x"] = [randn(rows, d)]
        v["input_norm"], v["post_norm"] = randn(d, std=0.02, mean=1.0), randn(d, std=0.02, mean=1.0)
        v["wq"], v["wo"] = randn(d, d, std=0.02), randn(d, d, std=0.02)
        v["wk"], v["wv"] = (randn(d, case["kv"] * hd, std=0.02) for _ in range(2))
    else:
        v["x"] = []
        for _ in range(case.get("micro", 1)):
            x = torch.randn((case["T"], d), generator=g, device="cuda")
            x = x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS)
            v["x"].append(x.bfloat16().float() if bf else x)
    v["w_router"] = randn(d, E, std=0.02)
    v["bias"] = randn(E, std=0.01, rounded=False)
    if case["skew"]:
        v["bias"] = torch.zeros_like(v["bias"])
        v["bias"][:2] = SKEW
    v["concept"] = randn(E, std=0.1, rounded=False) if case["concept"] else None
    # The shared expert first, then the routed ones.
    v["gate"] = randn(1 + E, d, f, std=0.02)
    v["up"] = randn(1 + E, d, f, std=0.02)
    v["down"] = randn(1 + E, f, d, std=0.02)
    if case["kind"] == "train":
        v["d_out"] = [randn(case["T"], d, std=0.1) for _ in range(case["micro"])]
    return v


def prepare(case, seed):
    v = _draws(case, seed)
    if case["kind"] == "matmul":
        op = {"ab": _lib.MATMUL_AB, "atb": _lib.MATMUL_ATB, "abt": _lib.MATMUL_ABT}[case["op"]]
        return dict(kind="matmul", op=op, a=v["a"], b=v["b"])
    d, f, E, k = case["d"], case["f"], case["E"], case["k"]
    host = {n: v[n].cpu().numpy() for n in ("w_router", "bias", "gate", "up", "down")}
    tdt = ops.torch_dtype(ops.dtype_code(case["dtype"]))
    state = dict(kind=case["kind"], x=[x.to(tdt) for x in v["x"]], concept=v["concept"])
    weights = (host["w_router"], host["bias"], list(host["gate"]), list(host["up"]),
               list(host["down"]))
    if case["kind"] == "block":
        eng = block.BlockEngine(d, case["heads"], case["kv"], f, E, k, 1,
                                max_tokens=case["batch"] * case["S"],
                                max_seq_len=case["S"] + case["pos"], rope_theta=500000.0, eps=EPS)
        dense = [v[n].cpu().numpy() for n in ("input_norm", "post_norm", "wq", "wk", "wv", "wo")]
        eng.upload(*dense, *weights)
        return dict(state, eng=eng, batch=case["batch"], S=case["S"], pos=case["pos"])
    eng = moe.MoEEngine(d, f, E, k, 1, case["dtype"], max_tokens=case["T"])
    if case["kind"] == "train":
        eng.enable_backward()
        state["d_out"] = [t.to(tdt) for t in v["d_out"]]
        state["grads"] = {n: torch.zeros(s, dtype=torch.float32, device="cuda")
                          for n, s in (("d_router", (d, E)), ("d_gate", (1 + E, d, f)),
                                       ("d_up", (1 + E, d, f)), ("d_down", (1 + E, f, d)))}
    eng.upload(*weights)
    return dict(state, eng=eng)


def run(state):
    if state["kind"] == "matmul":
        return ops.matmul_f32(state["op"], state["a"], state["b"])
    eng = state["eng"]
    if state["kind"] == "moe":
        return eng.forward(state["x"][0], concept_bias=state["concept"])
    if state["kind"] == "block":
        return eng.forward(state["x"][0], state["batch"], state["S"], state["pos"])
    got = []
    for i, (x, d_out) in enumerate(zip(state["x"], state["d_out"])):
        out = eng.forward(x)
        got += [out, eng.backward(x, d_out, state["grads"], beta=0 if i == 0 else 1)]
    return got + [state["grads"][n] for n in ("d_router", "d_gate", "d_up", "d_down")]


# --------------------------------------------------------------------- work --
def work(case):
    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        sizes = {"ab": m * k + k * n + m * n, "atb": m * k + m * n + k * n,
                 "abt": m * k + n * k + m * n}[case["op"]]
        return {"bytes": 4 * sizes, "flops": 2 * m * k * n}
    d, f, E, k = case["d"], case["f"], case["E"], case["k"]
    es = 2 if case["dtype"] == "bf16" else 4
    T = case["batch"] * case["S"] if case["kind"] == "block" else case["T"]
    # Experts that some token picks, when tokens pick evenly; the shared one.
    touched = 1 + E * (1 - (1 - k / E) ** T)
    expert = 3 * d * f
    flops = 6 * d * f * T * (1 + k) + 2 * T * d * E
    router = 4 * d * E
    if case["kind"] == "moe":
        return {"bytes": es * (2 * T * d + touched * expert) + router, "flops": flops}
    if case["kind"] == "block":
        kvd = case["kv"] * (d // case["heads"])
        dense = 2 * d * d + 2 * d * kvd
        # Pairs of a query and a key that is not after it, in every head.
        attn = 4 * d * case["batch"] * case["S"] * (case["S"] + 1) / 2
        return {"bytes": es * (2 * T * d + touched * expert + dense) + router,
                "flops": flops + 2 * T * dense + attn}
    n = case["micro"]
    # Forward, then the gradients of weights and of inputs: three products each.
    return {"bytes": n * (es * (4 * T * d + touched * expert) + router)
            + 4 * ((1 + E) * expert + d * E), "flops": 3 * n * flops}


def tolerance(case):
    """About four times what the outputs measure against ``exact``: f32 sums
    7e-7 (largest 1.5e-5), bf16 layers 2e-3 to 4e-3 (0.02; gradients 0.04).
    In a block the second norm's rounding reaches the router: 6e-3, and a
    token that a rounding sends to another expert is off by 0.66."""
    if case["kind"] == "matmul" or case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "block":
        return {"rel": 2e-2, "max": 0.9}
    return {"rel": 1e-2, "max": 0.1 if case["kind"] == "moe" else 0.2}


# -------------------------------------------------------------------- exact --
def _route(v, x):
    """(experts [T, k], gate weights [T, k]) in 64 bits."""
    raw = x @ v["w_router"].double()
    adj = raw + v["bias"].double()
    if v["concept"] is not None:
        adj = adj + v["concept"].double()
    sel = torch.argsort(adj, dim=1, descending=True, stable=True)[:, :v["k"]]
    return sel, torch.softmax(raw.gather(1, sel), 1)


def _experts(v, x, sel, g):
    """(slot, rows, weights, column of sel) of each expert's tokens; the shared
    expert has every token."""
    T = x.shape[0]
    yield 0, torch.arange(T, device=x.device), torch.ones(T, dtype=x.dtype, device=x.device), None
    for e in range(v["E"]):
        rows, col = (sel == e).nonzero(as_tuple=True)
        yield 1 + e, rows, g[rows, col], col


def _moe_exact(v, x):
    sel, g = _route(v, x)
    out = torch.zeros_like(x)
    for s, rows, w, _ in _experts(v, x, sel, g):
        xe = x[rows]
        gt = xe @ v["gate"][s].double()
        h = gt * torch.sigmoid(gt) * (xe @ v["up"][s].double())
        out[rows] += w[:, None] * (h @ v["down"][s].double())
    return out


def _train_exact(v, x, d_out, grads):
    """(out, d_x); the gradients are added to `grads`.  The routed input
    gradient carries the gate weight twice, as the layer's default has it."""
    sel, g = _route(v, x)
    out, d_x = torch.zeros_like(x), torch.zeros_like(x)
    dots = torch.zeros_like(g)
    for s, rows, w, col in _experts(v, x, sel, g):
        xe, wg, wu, wd = x[rows], *(v[n][s].double() for n in ("gate", "up", "down"))
        gt, up = xe @ wg, xe @ wu
        sig = torch.sigmoid(gt)
        h = gt * sig * up
        y = h @ wd
        out[rows] += w[:, None] * y
        if col is not None:
            dots[rows, col] = (y * d_out[rows]).sum(1)
        dy = w[:, None] * d_out[rows]
        dh = dy @ wd.T
        dg, du = dh * up * sig * (1 + gt * (1 - sig)), dh * gt * sig
        grads["d_down"][s] += h.T @ dy
        grads["d_gate"][s] += xe.T @ dg
        grads["d_up"][s] += xe.T @ du
        d_x[rows] += w[:, None] * (dg @ wg.T + du @ wu.T)
    dl = g * (dots - (g * dots).sum(1, keepdim=True))
    d_logits = torch.zeros(x.shape[0], v["E"], dtype=x.dtype, device=x.device).scatter(1, sel, dl)
    grads["d_router"] += x.T @ d_logits
    d_x += d_logits @ v["w_router"].double().T
    return out, d_x


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _block_exact(case, v):
    B, S, H, KV = case["batch"], case["S"], case["heads"], case["kv"]
    x = v["x"][0].double()
    hd = case["d"] // H
    n1 = _norm(x, v["input_norm"])
    q, k, val = ((n1 @ v[n].double()).view(B, S, -1, hd) for n in ("wq", "wk", "wv"))
    freq = 500000.0 ** (-torch.arange(0, hd, 2, device=x.device, dtype=torch.float64) / hd)
    angle = torch.arange(case["pos"], case["pos"] + S, device=x.device)[:, None] * freq
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(t):
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2)

    q, k = rope(q), rope(k)
    causal = torch.ones(S, S, dtype=torch.bool, device=x.device).tril()
    att = torch.empty_like(q)
    for b in range(B):
        for h in range(H):
            j = h // (H // KV)
            s = q[b, :, h].contiguous() @ k[b, :, j].T.contiguous() / math.sqrt(hd)
            att[b, :, h] = s.masked_fill(~causal, -math.inf).softmax(1) @ val[b, :, j].contiguous()
    x1 = x + att.view(B * S, -1) @ v["wo"].double()
    return x1 + _moe_exact(v, _norm(x1, v["post_norm"]))


def exact(case, seed):
    v = _draws(case, seed)
    if case["kind"] == "matmul":
        a, b = v["a"].double(), v["b"].double()
        return {"ab": lambda: a @ b, "atb": lambda: a.T @ b, "abt": lambda: a @ b.T}[case["op"]]()
    v["k"], v["E"] = case["k"], case["E"]
    if case["kind"] == "moe":
        return _moe_exact(v, v["x"][0].double())
    if case["kind"] == "block":
        return _block_exact(case, v)
    grads = {"d_router": torch.zeros_like(v["w_router"], dtype=torch.float64)}
    for n, like in (("d_gate", "gate"), ("d_up", "up"), ("d_down", "down")):
        grads[n] = torch.zeros_like(v[like], dtype=torch.float64)
    got = []
    for x, d_out in zip(v["x"], v["d_out"]):
        got += _train_exact(v, x.double(), d_out.double(), grads)
    return got + [grads[n] for n in ("d_router", "d_gate", "d_up", "d_down")]
