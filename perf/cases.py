"""The workloads this library's speed is judged on: quantization, single W4A16
linears, the linears of a decoder block, an MLP, and the whole Llama-style model,
each called through the package's public entry points.

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same
ranges; ``prepare`` builds what a program holds before the call, ``run`` is one
pass, ``work`` the bytes and operations it cannot do without, ``tolerance`` the
error another correct implementation may show and ``exact`` the 64-bit result.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn as nn
import torch.nn.functional as F

_PKG = Path(__file__).resolve().parent.parent / "itmo-final-project_amd"
_ROOTS = [str(p) for p in (Path.cwd() / "itmo-final-project_amd", _PKG) if p.is_dir()]
if _ROOTS and _ROOTS[0] not in sys.path:
    sys.path.insert(0, _ROOTS[0])

import int4_hip  # noqa: E402
from int4_hip.llama import MLP, LlamaConfig, LlamaForCausalLM  # noqa: E402

DEV = "cuda"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one token through the smallest linear of a block, called eagerly as a
        # layer: latency of a single call
        dict(name="linear_m1_512x2048", kind="linear", M=1, N=512, K=2048, G=128, dtype="bf16", bias=False),
        # decoding one token: the seven linears of 16 Llama-3.2-1B blocks, a
        # grouped launch per block, replayed from a graph as a serving loop does
        dict(name="block_m1", kind="block", M=1, hidden=2048, inter=8192, kv=512, G=128, dtype="bf16", layers=16,
             fused=True),
        # eight sequences decoded together, finer groups, fp16; the blocks as a
        # model calls them (q/k/v, o, gate/up, down)
        dict(name="block_m8_g32_fp16", kind="block", M=8, hidden=2048, inter=8192, kv=512, G=32, dtype="fp16",
             layers=8, fused=False),
        # a full small batch (or a short speculative draft) of 64 rows
        dict(name="block_m64_g64", kind="block", M=64, hidden=2048, inter=8192, kv=512, G=64, dtype="bf16", layers=8,
             fused=False),
        # the output head as int4, one token
        dict(name="lm_head_m1", kind="linear", M=1, N=128256, K=2048, G=128, dtype="bf16", bias=False),
        # a short prompt: MLP of a block on a ragged row count
        dict(name="mlp_m100", kind="mlp", M=100, hidden=2048, inter=8192, G=128, dtype="bf16"),
        # a long prompt: MLP of a block
        dict(name="mlp_m2048", kind="mlp", M=2048, hidden=2048, inter=8192, G=128, dtype="bf16"),
        # a wide layer of a larger model on a batch of long prompts, fp16
        dict(name="linear_m4096_14336x4096_fp16", kind="linear", M=4096, N=14336, K=4096, G=64, dtype="fp16",
             bias=False),
        # converting a model: the seven weights of a block quantized in a call
        dict(name="quantize_block", kind="quantize", hidden=2048, inter=8192, kv=512, G=128, dtype="bf16"),
        # the way back (fake-quant evaluation): one weight dequantized
        dict(name="dequantize_8192x2048", kind="dequantize", N=8192, K=2048, G=128, dtype="bf16"),
        # the 1B model on a ragged prompt, cut to four layers: bf16 rounding that
        # travels through all sixteen leaves too little to compare
        dict(name="model_prefill_500", kind="prefill", T=500, pos=0, max_len=640, hidden=2048, inter=8192, layers=4,
             heads=32, kv_heads=8, head_dim=64, vocab=128256, G=128, dtype="bf16", quantize_head=False),
        # the whole 1B model in fp16, one decode step from a graph at position 575
        dict(name="model_decode", kind="decode", T=1, pos=575, max_len=648, hidden=2048, inter=8192, layers=16,
             heads=32, kv_heads=8, head_dim=64, vocab=128256, G=128, dtype="fp16", quantize_head=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges; rows, tokens, layers or widths are
    halved until it costs no more than the largest of them."""
    c = _draw(rng)
    while work(c)["flops"] > 4.9e11 or work(c)["bytes"] > 1.1e9:
        k = next(k for k in ("M", "T", "layers", "vocab", "N") if c.get(k, 1) > 1)
        c[k] //= 2
    return c


def _draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "block", "block", "mlp", "quantize", "dequantize", "prefill",
                       "decode"])
    dt = rng.choice(["bf16", "bf16", "fp16"])
    G = rng.choice([32, 64, 128, 128, 256])
    if kind == "linear":
        M = _log(rng, 1, 4096)
        N = _log(rng, 64, 32768)
        if rng.random() < 0.7:  # most layers are multiples of 64 wide, some are odd
            N = max(64, N // 64 * 64)
        K = max(2, _log(rng, 512, 16384) // 256) * 256
        return dict(kind=kind, M=M, N=N, K=K, G=G, dtype=dt, bias=rng.random() < 0.25)
    hidden = rng.choice([1024, 1536, 2048, 2048, 2560, 3072, 4096])
    inter = hidden * rng.choice([6, 7, 8]) // 2
    kv = hidden // rng.choice([1, 4, 4, 8])
    if kind == "block":
        layers = max(1, min(8, int(5e8 / (2.0 * hidden * hidden + 2.0 * hidden * kv + 3.0 * hidden * inter))))
        return dict(kind=kind, M=_log(rng, 1, 64), hidden=hidden, inter=inter, kv=kv, G=G, dtype=dt, layers=layers,
                    fused=rng.random() < 0.4)
    if kind == "mlp":
        return dict(kind=kind, M=_log(rng, 65, 2500), hidden=hidden, inter=inter, G=G, dtype=dt)
    if kind == "quantize":
        groups = [g for g in (32, 64, 128, 128, 256, 512) if hidden % g == 0 and inter % g == 0]
        if hidden & (hidden - 1) == 0 and inter & (inter - 1) == 0:
            groups.append(-1)  # one group per row, a power of two too
        return dict(kind=kind, hidden=hidden, inter=inter, kv=kv, G=rng.choice(groups), dtype=dt)
    if kind == "dequantize":
        return dict(kind=kind, N=max(64, _log(rng, 512, 16384) // 8 * 8), K=max(2, _log(rng, 512, 16384) // 256) * 256,
                    G=G, dtype=rng.choice(["bf16", "fp16", "fp32"]))
    head_dim = rng.choice([64, 64, 128])
    heads = hidden // head_dim
    kv_heads = rng.choice([k for k in (heads, heads // 4, heads // 8) if k >= 1 and heads % k == 0])
    layers = rng.randint(1, 4 if dt == "bf16" else 8)
    vocab = rng.choice([1024, 32000, 128256])
    base = dict(hidden=hidden, inter=inter, layers=layers, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                vocab=vocab, G=G, dtype=dt, quantize_head=rng.random() < 0.3)
    if kind == "prefill":
        T = _log(rng, 2, 500)
        return dict(kind=kind, T=T, pos=0, max_len=T + rng.randint(0, 256), **base)
    pos = _log(rng, 1, 4096) - 1
    return dict(kind=kind, T=1, pos=pos, max_len=pos + 1 + rng.randint(0, 512), **base)


# ------------------------------------------------------------------ the inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, shape, dtype, sigma=1.0):
    """N(0, sigma) in fp32, rounded once to ``dtype``."""
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(sigma).to(dtype)


def _block_shapes(c):
    """(N, K) of q, k, v, o, gate, up, down."""
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    return [(h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i)]


def _linear_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    w = _randn(g, (c["N"], c["K"]), dt, 0.02)
    b = _randn(g, (c["N"],), dt, 0.1) if c["bias"] else None
    return w, b, _randn(g, (c["M"], c["K"]), dt)


def _block_inputs(c, seed):
    """Per layer the seven weights and the four activations (the block input, the
    attention output, the MLP input, the MLP's inner activation)."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    for _ in range(c["layers"]):
        ws = [_randn(g, s, dt, 0.02) for s in _block_shapes(c)]
        xs = [_randn(g, (c["M"], k), dt) for k in (c["hidden"], c["hidden"], c["hidden"], c["inter"])]
        yield ws, [xs[0], xs[0], xs[0], xs[1], xs[2], xs[2], xs[3]]


def _mlp_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    h, i = c["hidden"], c["inter"]
    ws = {n: _randn(g, s, dt, 0.02) for n, s in (("gate_proj", (i, h)), ("up_proj", (i, h)), ("down_proj", (h, i)))}
    return ws, _randn(g, (c["M"], h), dt)


def _model_inputs(c, seed):
    """Weights by module name, token ids and, for a decode step, the cache of the
    positions before it."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    h, i, d = c["hidden"], c["inter"], c["head_dim"]
    nq, nk = c["heads"] * d, c["kv_heads"] * d
    ws = {"model.embed_tokens": _randn(g, (c["vocab"], h), dt, 0.02)}
    for l in range(c["layers"]):
        for n, s in (("self_attn.q_proj", (nq, h)), ("self_attn.k_proj", (nk, h)), ("self_attn.v_proj", (nk, h)),
                     ("self_attn.o_proj", (h, nq)), ("mlp.gate_proj", (i, h)), ("mlp.up_proj", (i, h)),
                     ("mlp.down_proj", (h, i))):
            ws[f"model.layers.{l}.{n}"] = _randn(g, s, dt, 0.02)
    ids = torch.randint(0, c["vocab"], (c["T"],), generator=g, device=DEV)
    kc = vc = None
    if c["kind"] == "decode":
        kc = torch.zeros((c["layers"], c["kv_heads"], d, c["max_len"]), device=DEV)
        vc = torch.zeros((c["layers"], c["kv_heads"], c["max_len"], d), device=DEV)
        p = c["pos"]
        kc[..., :p] = torch.randn(kc[..., :p].shape, generator=g, device=DEV)
        vc[:, :, :p] = torch.randn(vc[:, :, :p].shape, generator=g, device=DEV)
    return ws, ids, kc, vc


def _capture(fn):
    """``fn`` captured once in a HIP graph on its warm-up stream (so that the
    library's per-stream workspace is in place), as GraphDecoder captures a step."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = fn()
    return graph, out


def _config(c):
    return LlamaConfig(vocab_size=c["vocab"], hidden_size=c["hidden"], intermediate_size=c["inter"],
                       num_hidden_layers=c["layers"], num_attention_heads=c["heads"],
                       num_key_value_heads=c["kv_heads"], head_dim=c["head_dim"])


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, b, x = _linear_inputs(case, seed)
        with torch.device("meta"):
            lin = nn.Linear(case["K"], case["N"], bias=b is not None)
        lin.weight = nn.Parameter(w, requires_grad=False)
        if b is not None:
            lin.bias = nn.Parameter(b, requires_grad=False)
        return dict(kind=kind, layer=int4_hip.Int4Linear.from_linear(lin, case["G"]), x=x)
    if kind == "block":
        blocks = [(int4_hip.quantize_int4_grouped(ws, case["G"]), xs) for ws, xs in _block_inputs(case, seed)]

        def step():
            outs = []
            for qs, xs in blocks:
                if case["fused"]:
                    flat = torch.empty(sum(case["M"] * q[0].shape[1] for q in qs), dtype=xs[0].dtype, device=DEV)
                    views, o = [], 0
                    for q in qs:
                        n = case["M"] * q[0].shape[1]
                        views.append(flat[o:o + n].view(case["M"], -1))
                        o += n
                    int4_hip.w4a16_matmul_grouped(xs, qs, out=views)
                    outs.append(flat)
                else:
                    outs += int4_hip.w4a16_matmul_grouped(xs[:3], qs[:3])
                    outs.append(int4_hip.w4a16_matmul(xs[3], *qs[3]))
                    outs += int4_hip.w4a16_matmul_grouped(xs[4:6], qs[4:6])
                    outs.append(int4_hip.w4a16_matmul(xs[6], *qs[6]))
            return outs

        graph, outs = _capture(step)
        return dict(kind=kind, graph=graph, outs=outs, blocks=blocks)
    if kind == "mlp":
        ws, x = _mlp_inputs(case, seed)
        with torch.device("meta"):
            mlp = MLP(LlamaConfig(hidden_size=case["hidden"], intermediate_size=case["inter"]))
        for n, w in ws.items():
            getattr(mlp, n).weight = nn.Parameter(w, requires_grad=False)
        return dict(kind=kind, mlp=int4_hip.quantize_model_linears(mlp, case["G"]), x=x)
    if kind == "quantize":
        g = _gen(seed)
        return dict(kind=kind, ws=[_randn(g, s, _DT[case["dtype"]], 0.02) for s in _block_shapes(case)], G=case["G"])
    if kind == "dequantize":
        w = _randn(_gen(seed), (case["N"], case["K"]), torch.bfloat16, 0.02)
        return dict(kind=kind, q=int4_hip.quantize_int4(w, case["G"]), dtype=_DT[case["dtype"]])
    ws, ids, kc, vc = _model_inputs(case, seed)
    dt = _DT[case["dtype"]]
    with torch.device("meta"):
        model = LlamaForCausalLM(_config(case))
    for name, m in model.named_modules():
        if hasattr(m, "eps"):
            m.weight = nn.Parameter(torch.ones(case["hidden"], dtype=dt, device=DEV), requires_grad=False)
        elif name in ws:
            m.weight = nn.Parameter(ws.pop(name), requires_grad=False)
    emb = model.model.embed_tokens.weight
    model.lm_head.weight = nn.Parameter(emb.detach().clone(), requires_grad=False) if case["quantize_head"] else emb
    model = model.eval()
    int4_hip.quantize_model_linears(model, case["G"], skip=() if case["quantize_head"] else ("lm_head",))
    model.allocate_cache(case["max_len"], dt, torch.device(DEV))
    if kind == "prefill":
        return dict(kind=kind, model=model, ids=ids)
    model.kc.copy_(kc)
    model.vc.copy_(vc)
    pos = torch.full((1,), case["pos"], dtype=torch.long, device=DEV)
    graph, logits = _capture(lambda: model.decode_step(ids, pos))
    return dict(kind=kind, model=model, ids=ids, pos=pos, graph=graph, logits=logits)


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "mlp":
        return state["mlp"](state["x"])
    if kind == "quantize":
        return int4_hip.quantize_int4_grouped(state["ws"], state["G"])
    if kind == "dequantize":
        return int4_hip.dequantize_int4(*state["q"], state["dtype"])
    if kind == "block":
        state["graph"].replay()
        return state["outs"]
    model = state["model"]
    if kind == "prefill":
        logits = model.prefill(state["ids"])
    else:
        state["graph"].replay()
        logits = state["logits"]
    return dict(logits=logits, kc=model.kc, vc=model.vc)


# ----------------------------------------------------------- work and tolerance
def _weight_bytes(N, K, G):
    return N * K // 2 + 4 * N * (K // (K if G == -1 else G))


def work(case):
    kind, G = case["kind"], case["G"]
    e = 4 if case["dtype"] == "fp32" else 2
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=_weight_bytes(N, K, G) + 2 * M * (N + K) + (2 * N if case["bias"] else 0),
                    flops=2 * M * N * K)
    if kind == "block":
        M, shapes = case["M"], _block_shapes(case)
        b = sum(_weight_bytes(n, k, G) + 2 * M * n for n, k in shapes) + 2 * M * (3 * case["hidden"] + case["inter"])
        return dict(bytes=b * case["layers"], flops=2 * M * sum(n * k for n, k in shapes) * case["layers"])
    if kind == "mlp":
        M, h, i = case["M"], case["hidden"], case["inter"]
        return dict(bytes=2 * _weight_bytes(i, h, G) + _weight_bytes(h, i, G) + 4 * M * h, flops=6 * M * h * i)
    if kind == "quantize":
        return dict(bytes=sum(2 * n * k + _weight_bytes(n, k, G) for n, k in _block_shapes(case)), flops=0)
    if kind == "dequantize":
        return dict(bytes=_weight_bytes(case["N"], case["K"], G) + e * case["N"] * case["K"], flops=0)
    T, h, i, L, V = case["T"], case["hidden"], case["inter"], case["layers"], case["vocab"]
    nq, nk = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    shapes = [(nq, h), (nk, h), (nk, h), (h, nq), (i, h), (i, h), (h, i)]
    head = _weight_bytes(V, h, G) if case["quantize_head"] else 2 * V * h
    ctx = case["pos"] * T + T * (T + 1) // 2  # attended positions, summed over the tokens
    cache = 8 * nk * (case["pos"] + T) * L    # keys and values, fp32, once
    return dict(bytes=L * sum(_weight_bytes(n, k, G) for n, k in shapes) + head + cache + 2 * T * (h + V),
                flops=2 * T * (L * sum(n * k for n, k in shapes) + V * h) + 4 * nq * ctx * L)


def tolerance(case):
    """About four times the distance to the 64-bit results (measured: linears 1.7e-3
    in bf16 and 2.1e-4 to 2.8e-4 in fp16, the MLP 4.8e-3, four layers of the model
    2e-2 at most); the largest single difference is that of a few roundings."""
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        return "exact"
    fp16 = case["dtype"] == "fp16"
    if kind in ("linear", "block"):
        return {"rel": 1.2e-3 if fp16 else 7e-3, "max": 8e-3 if fp16 else 4e-2}
    if kind == "mlp":
        return {"rel": 2.5e-3 if fp16 else 2e-2, "max": 2e-2 if fp16 else 0.15}
    return {"rel": 1.5e-2 if fp16 else 3e-2, "max": 0.1 if fp16 else 0.4}


# ----------------------------------------------------------- 64-bit references
def _rtn(w, G):
    """Codes, scales, zeros [N, K/G, G], [N, K/G], [N, K/G] of the group-wise
    asymmetric round-to-nearest quantization, fp32 steps as the format defines
    them (the scale stored as fp16)."""
    N, K = w.shape
    G = K if G == -1 else G
    wg = w.float().view(N, K // G, G)
    lo, hi = wg.amin(2).clamp(max=0.0), wg.amax(2).clamp(min=0.0)
    s = (hi - lo) / torch.full((), 15.0, device=w.device)
    s = torch.where(s == 0, torch.ones_like(s), s).half()
    z = torch.floor(-lo / s.float() + 0.5).clamp(0, 15)
    q = (torch.floor(wg / s.float()[..., None] + 0.5) + z[..., None]).clamp(0, 15)
    return q, s, z


def _what(w, G):
    """The dequantized weight [N, K], (q - z) s in 64 bits."""
    q, s, z = _rtn(w, G)
    return ((q - z[..., None]).double() * s.double()[..., None]).view(w.shape)


def _exact_model(case, seed):
    ws, ids, kc, vc = _model_inputs(case, seed)
    G, T, d = case["G"], case["T"], case["head_dim"]
    nh, nkv, p0 = case["heads"], case["kv_heads"], case["pos"]
    cfg = _config(case)
    # rotary frequencies with the Llama-3 scaling, angles in fp32 as a position
    # table holds them
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, d, 2, dtype=torch.float64) / d))
    factor, low, high, orig = cfg.rope_scaling
    wavelen = 2 * math.pi / inv
    smooth = (orig / wavelen - low) / (high - low)
    mid = (wavelen <= orig / low) & (wavelen >= orig / high)
    scaled = torch.where(wavelen > orig / low, inv / factor, inv)
    inv = torch.where(mid, (1 - smooth) * inv / factor + smooth * inv, scaled).float().to(DEV)
    ang = (torch.arange(p0, p0 + T, device=DEV, dtype=torch.float32)[:, None] * inv[None, :]).double()
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def rope(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    def norm(t):
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + cfg.rms_norm_eps)

    L = p0 + T
    ok = torch.zeros((case["layers"], nkv, d, case["max_len"]), dtype=torch.float64, device=DEV)
    ov = torch.zeros((case["layers"], nkv, case["max_len"], d), dtype=torch.float64, device=DEV)
    if kc is not None:
        ok.copy_(kc), ov.copy_(vc)
    causal = torch.arange(L, device=DEV)[None, :] > torch.arange(p0, L, device=DEV)[:, None]
    x = ws["model.embed_tokens"][ids].double()
    for l in range(case["layers"]):
        W = {n: _what(ws.pop(f"model.layers.{l}.{n}"), G) for n in (
            "self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj",
            "mlp.up_proj", "mlp.down_proj")}
        h = norm(x)
        q = rope((h @ W["self_attn.q_proj"].T).view(T, nh, d))
        ok[l, :, :, p0:L] = rope((h @ W["self_attn.k_proj"].T).view(T, nkv, d)).permute(1, 2, 0)
        ov[l, :, p0:L] = (h @ W["self_attn.v_proj"].T).view(T, nkv, d).transpose(0, 1)
        o = torch.empty((T, nh, d), dtype=torch.float64, device=DEV)
        for j in range(nh):
            s = (q[:, j] @ ok[l, j * nkv // nh, :, :L]) / math.sqrt(d)
            o[:, j] = torch.softmax(s.masked_fill(causal, float("-inf")), -1) @ ov[l, j * nkv // nh, :L]
        x = x + o.view(T, nh * d) @ W["self_attn.o_proj"].T
        h = norm(x)
        x = x + (F.silu(h @ W["mlp.gate_proj"].T) * (h @ W["mlp.up_proj"].T)) @ W["mlp.down_proj"].T
    emb = ws["model.embed_tokens"]
    head = _what(emb, G) if case["quantize_head"] else emb.double()
    return dict(logits=norm(x) @ head.T, kc=ok, vc=ov)


@torch.no_grad()
def exact(case, seed):
    kind, G = case["kind"], case["G"]
    if kind == "linear":
        w, b, x = _linear_inputs(case, seed)
        y = x.double() @ _what(w, G).T
        return y if b is None else y + b.double()
    if kind == "block":
        outs = []
        for ws, xs in _block_inputs(case, seed):
            ys = [x.double() @ _what(w, G).T for w, x in zip(ws, xs)]
            if case["fused"]:
                outs.append(torch.cat([y.reshape(-1) for y in ys]))
            else:
                outs += ys
        return outs
    if kind == "mlp":
        ws, x = _mlp_inputs(case, seed)
        x = x.double()
        return (F.silu(x @ _what(ws["gate_proj"], G).T) * (x @ _what(ws["up_proj"], G).T)) @ _what(ws["down_proj"], G).T
    if kind == "quantize":
        g, outs = _gen(seed), []
        for shape in _block_shapes(case):
            w = _randn(g, shape, _DT[case["dtype"]], 0.02)
            q, s, z = _rtn(w, G)
            words = torch.zeros((shape[0], shape[1] // 8), dtype=torch.int64, device=DEV)
            for i in range(8):
                words += q.view(shape[0], -1, 8)[..., i].long() << (4 * i)
            words = torch.where(words >= 2**31, words - 2**32, words).to(torch.int32)
            outs.append((words.T.contiguous(), s.double().T.contiguous(), z.double().T.contiguous()))
        return outs
    if kind == "dequantize":
        return _what(_randn(_gen(seed), (case["N"], case["K"]), torch.bfloat16, 0.02), G)
    return _exact_model(case, seed)
