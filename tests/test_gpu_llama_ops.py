"""GPU: the fused kernels between the linears of a decoder layer
(int4_hip/llama_ops.py) against 64-bit torch arithmetic on the CPU."""
import math

import pytest
import torch

import int4_hip
from _synth import randn
from int4_hip import llama_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
# one rounding to the output dtype (half an ulp: 2^-8 of the value for bf16's 8
# significant bits, 2^-11 for fp16's 11), plus fp32 arithmetic: sums of up to a
# few thousand positive terms of relative error 2^-24 each, far below it
ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
FP32 = 1e-5


def _rope(t, cos, sin):
    """t [T, heads, D] fp32, products rounded separately as the kernels do."""
    h = t.shape[-1] // 2
    a, b, c, s = t[..., :h], t[..., h:], cos[:, None, :], sin[:, None, :]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _tables(n, d):
    ang = torch.arange(n)[:, None] * (1.0 / 500000.0 ** (torch.arange(0, d, 2) / d))[None, :]
    return ang.cos().float(), ang.sin().float()


def _attention(q, kc, vc, pos0):
    """fp64 attention of q [T, nh, D] at positions pos0.. over kc [nkv, D, L], vc [nkv, L, D]."""
    T, nh, D = q.shape
    nkv, L = kc.shape[0], pos0 + T
    out = torch.empty((T, nh, D), dtype=torch.float64)
    mask = torch.arange(L)[None, :] > torch.arange(pos0, L)[:, None]
    for h in range(nh):
        s = q[:, h].double() @ kc[h * nkv // nh, :, :L].double() / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ vc[h * nkv // nh, :L].double()
    return out.reshape(T, nh * D)


def _check_out(got, want, dtype):
    got = got.double().cpu()
    scale = want.square().mean().sqrt()
    err = (got - want).abs() / torch.maximum(want.abs(), scale)
    assert err.max().item() <= ROUND[dtype] + 10 * FP32, err.max().item()


# positions at the edges of a 64-position chunk and of the cache; one, several
# and many query heads per key-value head (slices of four); caches past 4096
# positions (chunks of 128); cache lengths that are no multiple of four
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nh,nkv,d,max_len,pos", [
    (1, 1, 64, 1, 0), (8, 2, 64, 96, 0), (8, 2, 64, 96, 63), (8, 2, 64, 96, 64), (8, 8, 64, 97, 96),
    (32, 8, 64, 648, 575), (6, 2, 128, 200, 127), (20, 2, 128, 333, 332), (16, 2, 64, 4099, 4098),
    (4, 1, 128, 8193, 5000), (2, 1, 64, 130, 129)])
def test_attention_decode(dtype, nh, nkv, d, max_len, pos):
    print(f"[attn decode] {dtype} {nh}/{nkv}x{d} L={max_len} pos={pos}", flush=True)
    q, k, v = (randn((1, n * d), seed=i, dtype=dtype) for i, n in enumerate((nh, nkv, nkv)))
    kc, vc = randn((nkv, d, max_len), 5, dtype=torch.float32), randn((nkv, max_len, d), 6, dtype=torch.float32)
    # what lies at the position and past it takes no part, whatever it holds
    kc[..., pos:] = float("nan")
    vc[:, pos:] = float("inf")
    cos, sin = (t[pos:pos + 1] for t in _tables(max_len, d))
    p = torch.tensor([pos], device=DEV)
    args = [t.to(DEV) for t in (q, k, v, cos.contiguous(), sin.contiguous(), kc, vc)]
    assert llama_ops.attention_decode_ok(args[0], *args[5:], *args[3:5], p, nh, nkv, d)
    got = llama_ops.attention_decode(*args, p, nh, nkv, d)
    again = llama_ops.attention_decode(*args, p, nh, nkv, d)
    kc[:, :, pos] = _rope(k.float().view(1, nkv, d), cos, sin)[0]
    vc[:, pos] = v.float().view(nkv, d)
    assert torch.equal(args[5].cpu().nan_to_num(7.0), kc.nan_to_num(7.0)) and torch.equal(args[6].cpu(), vc)
    assert torch.equal(got, again)
    _check_out(got, _attention(_rope(q.float().view(1, nh, d), cos, sin), kc, vc, pos), dtype)


@pytest.mark.parametrize("nh,nkv,d", [(1, 1, 64), (6, 1, 128), (8, 2, 64)])
@pytest.mark.parametrize("pos", [-1, 70, 1 << 40])
def test_attention_decode_outside_the_cache(nh, nkv, d, pos):
    """A position the cache does not hold: the caches as they were, a NaN output."""
    q, k, v = (randn((1, n * d), seed=i).to(DEV) for i, n in enumerate((nh, nkv, nkv)))
    kc, vc = randn((nkv, d, 70), 5, dtype=torch.float32).to(DEV), randn((nkv, 70, d), 6, dtype=torch.float32).to(DEV)
    row = torch.ones((1, d // 2), device=DEV)
    before = kc.clone(), vc.clone()
    out = llama_ops.attention_decode(q, k, v, row, row, kc, vc, torch.tensor([pos], device=DEV), nh, nkv, d)
    assert out.shape == (1, nh * d) and out.isnan().all()
    assert torch.equal(kc, before[0]) and torch.equal(vc, before[1])


# tokens at the edges of a 16- / 32-query tile and of the 64-position blocks, a
# prompt continued at pos0, cache ends inside a block, odd and even heads per
# key-value head, cache rows that are no multiple of 16 bytes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,pos0,max_len,nh,nkv,d", [
    (1, 0, 1, 2, 1, 64), (15, 0, 15, 3, 1, 64), (16, 0, 64, 4, 2, 64), (33, 0, 40, 1, 1, 128), (64, 0, 64, 8, 8, 64),
    (65, 0, 129, 8, 2, 64), (500, 0, 640, 8, 2, 64), (130, 61, 191, 6, 2, 128), (1, 300, 303, 20, 2, 64),
    (270, 0, 271, 4, 4, 128)])
def test_attention_prefill(dtype, T, pos0, max_len, nh, nkv, d):
    print(f"[attn prefill] {dtype} T={T}+{pos0} L={max_len} {nh}/{nkv}x{d}", flush=True)
    q, k, v = (randn((T, n * d), seed=i, dtype=dtype) for i, n in enumerate((nh, nkv, nkv)))
    kc, vc = randn((nkv, d, max_len), 5, dtype=torch.float32), randn((nkv, max_len, d), 6, dtype=torch.float32)
    # what lies past the prompt takes no part, whatever it holds
    kc[..., pos0 + T:] = float("nan")
    vc[:, pos0 + T:] = float("inf")
    cos, sin = (t[pos0:pos0 + T].contiguous() for t in _tables(max_len, d))
    args = [t.to(DEV) for t in (q, k, v, cos, sin, kc, vc)]
    assert llama_ops.attention_prefill_ok(args[0], args[5], args[6], args[3], args[4], pos0, nh, nkv, d)
    got = llama_ops.attention_prefill(*args, pos0, nh, nkv, d)
    kc[:, :, pos0:pos0 + T] = _rope(k.float().view(T, nkv, d), cos, sin).permute(1, 2, 0)
    vc[:, pos0:pos0 + T] = v.float().view(T, nkv, d).transpose(0, 1)
    assert torch.equal(args[5].cpu().nan_to_num(7.0), kc.nan_to_num(7.0)) and torch.equal(args[6].cpu(), vc)
    assert torch.equal(got, llama_ops.attention_prefill(*args, pos0, nh, nkv, d))
    _check_out(got, _attention(_rope(q.float().view(T, nh, d), cos, sin), kc, vc, pos0), dtype)


def test_attention_prefill_infinities_and_nan():
    """As torch's softmax: rows that see only -inf scores, an infinite or a NaN score
    are NaN; -inf scores beside finite ones weigh nothing."""
    d, T = 64, 200
    cos, sin = torch.ones((T, d // 2)), torch.zeros((T, d // 2))
    # scores that overflow: an infinite key would be NaN after the rotation (inf * 0)
    q = torch.full((T, 4 * d), 64.0, dtype=torch.bfloat16)
    k = torch.zeros((T, 4, d), dtype=torch.bfloat16)
    k[:64, 0, 0] = -3e38
    k[100, 1, 0] = 3e38
    k[70, 2, 0] = float("nan")
    v = randn((T, 4, d), 1)
    kc, vc = torch.zeros((4, d, T), device=DEV), torch.zeros((4, T, d), device=DEV)
    got = llama_ops.attention_prefill(q.to(DEV), k.view(T, -1).to(DEV), v.view(T, -1).to(DEV), cos.to(DEV),
                                      sin.to(DEV), kc, vc, 0, 4, 4, d).cpu().view(T, 4, d)
    nan = got.isnan()
    assert nan[:64, 0].all() and not nan[64:, 0].any()
    torch.testing.assert_close(got[199, 0].float(), v[64:, 0].float().mean(0), rtol=1e-2, atol=1e-3)
    assert not nan[:100, 1].any() and nan[100:, 1].all()
    assert not nan[:70, 2].any() and nan[70:, 2].all()
    assert not nan[:, 3].any()


def test_attention_decode_infinities_and_nan():
    """-inf scores weigh nothing (a whole chunk of them included), an infinite or
    NaN score makes its head NaN, as torch's softmax does."""
    d, L, pos = 64, 256, 200
    cos, sin = torch.ones((1, d // 2)), torch.zeros((1, d // 2))
    q = torch.ones((1, 4 * d), dtype=torch.bfloat16)
    k = v = torch.zeros((1, 4 * d), dtype=torch.bfloat16)
    kc, vc = torch.zeros((4, d, L)), randn((4, L, d), 1, dtype=torch.float32)
    kc[0, 0, :64] = float("-inf")   # head 0: its first chunk weighs nothing
    kc[1, 0, 100] = float("inf")    # head 1: inf - inf
    kc[2, 0, 70] = float("nan")
    kc[3, 0, :pos] = float("-inf")  # head 3: only the new position weighs
    args = [t.to(DEV) for t in (q, k, v, cos, sin, kc, vc)]
    got = llama_ops.attention_decode(*args, torch.tensor([pos], device=DEV), 4, 4, d).view(4, d).cpu()
    vc[:, pos] = 0
    torch.testing.assert_close(got[0].float(), vc[0, 64:pos + 1].mean(0), rtol=1e-2, atol=1e-3)
    assert got[1].isnan().all() and got[2].isnan().all()
    assert torch.equal(got[3], torch.zeros(d, dtype=torch.bfloat16))


@pytest.mark.parametrize("pos", [0, 5, 64, 99])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_attention_decode_takes_an_infinite_new_value(bad, pos):
    """An infinity in the value being written weighs what its position weighs, as in torch's
    product, and nothing else of the block it shares with empty positions."""
    nh, nkv, d, L = 4, 2, 64, 100
    q, k, v = (randn((1, n * d), seed=i) for i, n in enumerate((nh, nkv, nkv)))
    v[0, 3] = bad
    kc, vc = randn((nkv, d, L), 5, dtype=torch.float32), randn((nkv, L, d), 6, dtype=torch.float32)
    cos, sin = (t[pos:pos + 1].contiguous() for t in _tables(L, d))
    args = [t.to(DEV) for t in (q, k, v, cos, sin, kc, vc)]
    got = llama_ops.attention_decode(*args, torch.tensor([pos], device=DEV), nh, nkv, d).cpu()
    kc[:, :, pos], vc[:, pos] = _rope(k.float().view(1, nkv, d), cos, sin)[0], v.float().view(nkv, d)
    want = _attention(_rope(q.float().view(1, nh, d), cos, sin), kc, vc, pos)
    assert torch.equal(got.isfinite(), want.isfinite()) and (~want.isfinite()).sum() == nh // nkv
    torch.testing.assert_close(got[~want.isfinite()].double(), want[~want.isfinite()], equal_nan=True)
    _check_out(got.nan_to_num(0, 0, 0), want.nan_to_num(0, 0, 0), torch.bfloat16)


@pytest.mark.parametrize("T", [1, 33, 64, 100])
@pytest.mark.parametrize("d", [64, 128])
def test_attention_prefill_takes_an_infinite_last_value(T, d):
    """The last token's row with an infinity in its own value; positions past the prompt in
    its block do not see it."""
    nh, nkv, L = 4, 2, 130
    q, k, v = (randn((T, n * d), seed=i) for i, n in enumerate((nh, nkv, nkv)))
    v[-1, 3] = float("inf")
    kc, vc = torch.zeros((nkv, d, L)), torch.zeros((nkv, L, d))
    cos, sin = (t[:T].contiguous() for t in _tables(L, d))
    args = [t.to(DEV) for t in (q, k, v, cos, sin, kc, vc)]
    got = llama_ops.attention_prefill(*args, 0, nh, nkv, d).cpu()[-1:]
    kc[:, :, :T] = _rope(k.float().view(T, nkv, d), cos, sin).permute(1, 2, 0)
    vc[:, :T] = v.float().view(T, nkv, d).transpose(0, 1)
    want = _attention(_rope(q.float().view(T, nh, d), cos, sin), kc, vc, 0)[-1:]
    assert torch.equal(got == math.inf, want == math.inf) and (want == math.inf).sum() == nh // nkv
    _check_out(got.nan_to_num(7, 7, 7), want.nan_to_num(7, 7, 7), torch.bfloat16)


# rows of one vector up to the widest (16384), widths that leave threads idle
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n", [(1, 8), (1, 2048), (3, 2056), (7, 4096), (2, 8200), (500, 512), (1, 16384)])
def test_rms_norm(dtype, rows, n):
    print(f"[rms norm] {dtype} {rows}x{n}", flush=True)
    x, d, w = randn((rows, n), 1, dtype=dtype), randn((rows, n), 2, 0.3, dtype=dtype), randn((n,), 3, dtype=dtype)

    def ref(t):
        t = t.double()
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-5) * w.double()

    xd, dd, wd = (t.to(DEV) for t in (x, d, w))
    assert llama_ops.rms_norm_ok(xd, wd) and llama_ops.rms_norm_ok(xd, wd, dd)
    _check_out(llama_ops.rms_norm(xd, wd, 1e-5), ref(x), dtype)
    s, y = llama_ops.rms_norm(xd, wd, 1e-5, dd)
    assert torch.equal(s.cpu(), x + d)
    _check_out(y, ref(x + d), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 8), (1, 8192), (100, 2056), (2, 3, 264)])
def test_silu_mul(dtype, shape):
    g, u = randn(shape, 1, 4.0, dtype=dtype), randn(shape, 2, dtype=dtype)
    gd, ud = g.to(DEV), u.to(DEV)
    assert llama_ops.silu_mul_ok(gd, ud)
    want = torch.nn.functional.silu(g.double()) * u.double()
    got = llama_ops.silu_mul(gd, ud).cpu().double()
    # relative to each value; fp16's smallest subnormal 2^-24 below that
    assert ((got - want).abs() <= (ROUND[dtype] + FP32) * want.abs() + 2.0 ** -25).all()


def test_fused_ops_leave_the_general_path_alone():
    """Autograd, other dtypes, strided and misaligned operands take the torch operations."""
    x = torch.randn(4, 64, device=DEV, dtype=torch.bfloat16)
    w = torch.ones(64, device=DEV, dtype=torch.bfloat16)
    assert llama_ops.rms_norm_ok(x, w) and llama_ops.silu_mul_ok(x, x)
    g = x.clone().requires_grad_()
    assert not llama_ops.rms_norm_ok(g, w) and not llama_ops.silu_mul_ok(g, x)
    with torch.no_grad():
        assert llama_ops.rms_norm_ok(g, w)
    for bad in (x.float(), x.t().contiguous().t(), x.cpu(), torch.empty(257, device=DEV, dtype=x.dtype)[1:].view(4, 64)):
        assert not llama_ops.rms_norm_ok(bad, w) and not llama_ops.silu_mul_ok(bad, bad)
    assert not llama_ops.rms_norm_ok(x, w.float()) and not llama_ops.rms_norm_ok(x, w, x[:2])
    with torch.autocast("cuda", dtype=torch.float16):
        assert not llama_ops.rms_norm_ok(x, w)
    assert not torch.func.vmap(lambda t: torch.zeros(()) + llama_ops.silu_mul_ok(t, t))(x).any()


def _rows(shapes, G, dtype, seed):
    """Quantized weights of the shapes, and their exact 64-bit values."""
    qs = [int4_hip.quantize_int4(randn(s, seed + i, 0.02, dtype=dtype).to(DEV), G) for i, s in enumerate(shapes)]
    return qs, [int4_hip.dequantize_int4(*q, torch.float32).double().cpu() for q in qs]


# one-row products behind a norm or a gated activation: the tile widths (128 / 64 /
# 32 columns, picked by K and the number of workgroups), K parts joined across
# workgroups, waves without steps (K = 256), the longest row of the norm.  Against
# the 64-bit result of the unrounded activations.  Bound per output, relative to
# the outputs' rms: one rounding of the output; one rounding of each activation,
# independent errors of at most ROUND / sqrt(3) rms, six deviations; 1e-3 for the
# fp32 accumulation of 128 x + x q terms (2^-24 of 143 sum |x| s).  The launch
# rounds as often as the separate ones, so its total error may not be larger
# (15 % for chance)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,Ns,G", [(256, (64, 8), 32), (2048, (2048, 512, 512), 128), (2048, (8192, 8192), 64),
                                    (4096, (1000,), 128), (8192, (72, 40), 512), (6144, (256,), 256)])
def test_norm_linears(dtype, K, Ns, G):
    print(f"[norm linears] {dtype} K={K} N={Ns} G={G}", flush=True)
    qs, ws = _rows([(n, K) for n in Ns], G, dtype, 40)
    x, d, w = randn((1, K), 1, dtype=dtype), randn((1, K), 2, 0.3, dtype=dtype), randn((K,), 3, dtype=dtype)
    xd, dd, wd = (t.to(DEV) for t in (x, d, w))
    for delta in (None, dd):
        got = llama_ops.norm_linears(xd, delta, wd, 1e-5, qs)
        assert got is not None
        total, ys = got
        if delta is None:
            h = llama_ops.rms_norm(xd, wd, 1e-5)
            assert total is xd
        else:
            s, h = llama_ops.rms_norm(xd, wd, 1e-5, dd)
            assert torch.equal(total, s)
        t = total.double().cpu()
        exact = t * torch.rsqrt(t.square().mean() + 1e-5) * w.double()
        for y, q, wx in zip(ys, qs, ws):
            want = exact @ wx.T
            _check_rows(y, int4_hip.w4a16_matmul(h, *q), want, dtype)
            again = llama_ops.norm_linears(xd, delta, wd, 1e-5, [q])[1][0]  # another tiling
            _check_rows(again, y, want, dtype)


def _check_rows(got, separate, want, dtype):
    got, separate = got.double().cpu(), separate.double().cpu()
    err = (got - want).abs() / torch.maximum(want.abs(), want.square().mean().sqrt())
    assert err.max().item() <= ROUND[dtype] * (1 + 6 / math.sqrt(3)) + 1e-3, err.max().item()
    if want.numel() >= 256:
        assert (got - want).norm() <= 1.15 * (separate - want).norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,N,G", [(256, 8, 32), (8192, 2048, 128), (2048, 520, 64), (8192, 64, 1024)])
def test_silu_linear(dtype, K, N, G):
    print(f"[silu linear] {dtype} K={K} N={N} G={G}", flush=True)
    (q,), (wx,) = _rows([(N, K)], G, dtype, 50)
    g, u = randn((1, K), 1, 2.0, dtype=dtype).to(DEV), randn((1, K), 2, dtype=dtype).to(DEV)
    got = llama_ops.silu_linear(g, u, q)
    assert got is not None
    gd, ud = g.double().cpu(), u.double().cpu()
    _check_rows(got, int4_hip.w4a16_matmul(llama_ops.silu_mul(g, u), *q),
                (torch.nn.functional.silu(gd) * ud) @ wx.T, dtype)
    assert torch.equal(got, llama_ops.silu_linear(g, u, q))


def test_prologue_launches_refuse_what_they_do_not_hold():
    """No launch for group sizes below 32, ragged N, several rows or a norm past 8192
    values: the callers then run the separate operations."""
    x, w = torch.ones((1, 512), device=DEV, dtype=torch.bfloat16), torch.ones(512, device=DEV, dtype=torch.bfloat16)
    for N, G in ((64, 16), (12, 64)):
        q = int4_hip.quantize_int4(randn((N, 512), 1).to(DEV), G)
        assert llama_ops.norm_linears(x, None, w, 1e-5, [q]) is None and llama_ops.silu_linear(x, x, q) is None
    q = int4_hip.quantize_int4(randn((64, 512), 1).to(DEV), 64)
    two = x.expand(2, 512).contiguous()
    assert llama_ops.norm_linears(two, None, w, 1e-5, [q]) is None and llama_ops.silu_linear(two, two, q) is None
    long = torch.ones((1, 16384), device=DEV, dtype=torch.bfloat16)
    q = int4_hip.quantize_int4(randn((64, 16384), 1).to(DEV), 64)
    assert llama_ops.norm_linears(long, None, long[0], 1e-5, [q]) is None


def test_decode_step_respects_hooks_and_replaced_modules():
    """A hook or a subclass anywhere in a layer keeps that layer on the module calls,
    with the same logits up to rounding."""
    from int4_hip.llama import LlamaConfig, LlamaForCausalLM
    cfg = LlamaConfig(vocab_size=512, hidden_size=512, intermediate_size=1024, num_hidden_layers=2,
                      num_attention_heads=8, num_key_value_heads=2, head_dim=64)
    with torch.device(DEV):
        m = LlamaForCausalLM(cfg)
    m.init_weights(3)
    m = int4_hip.quantize_model_linears(m.to(torch.bfloat16).eval(), 128)
    m.allocate_cache(16, torch.bfloat16, DEV)
    ids, pos = torch.tensor([7], device=DEV), torch.tensor([0], device=DEV)
    want = m.decode_step(ids, pos).float()
    seen = []
    layer = m.model.layers[1]
    for mod in (layer.post_attention_layernorm, layer.mlp, layer.self_attn.o_proj):
        handle = mod.register_forward_hook(lambda *a: seen.append(a[0]))
        got = m.decode_step(ids, pos).float()
        handle.remove()
        assert seen and seen.pop() is mod and not seen
        assert (got - want).abs().max() <= 3e-2 * want.abs().max()
    # a hook on an attention module sees the mask, as without the fused kernel
    handle = layer.self_attn.register_forward_pre_hook(lambda mod, args: seen.append(args[7]))
    got = m.decode_step(ids, pos).float()
    handle.remove()
    assert seen[0].tolist() == [0.0] + [float("-inf")] * 15
    assert (got - want).abs().max() <= 3e-2 * want.abs().max()


@pytest.mark.parametrize("scale", [1e-4, 1.0, 3e3, 6e4])
def test_norm_linears_fp16_range(scale):
    """Large and small rows whose x * weight leaves fp16's range before the norm's factor,
    with outliers of the size of the rest's sum: no overflow, no lost bits."""
    K = 2048
    (q,), (wx,) = _rows([(512, K)], 128, torch.float16, 60)
    x = (randn((1, K), 1, dtype=torch.float32) * scale / 8).clamp(-6e4, 6e4)
    x[0, 5] = scale
    x, w = x.half(), (randn((K,), 2, dtype=torch.float32) * 20).half()
    _, (y,) = llama_ops.norm_linears(x.to(DEV), None, w.to(DEV), 1e-5, [q])
    t = x.double()
    want = (t * torch.rsqrt(t.square().mean() + 1e-5) * w.double()) @ wx.T
    h = llama_ops.rms_norm(x.to(DEV), w.to(DEV), 1e-5)
    _check_rows(y, int4_hip.w4a16_matmul(h, *q), want, torch.float16)


def test_norm_linears_non_finite_rows():
    """A NaN or an infinity in the row makes every output NaN (inf * 0 in the norm); a zero
    row gives zeros."""
    K = 2048
    (q,), _ = _rows([(64, K)], 128, torch.float16, 61)
    w = torch.ones(K, device=DEV, dtype=torch.float16)
    for bad in (float("nan"), float("inf")):
        x = randn((1, K), 1, dtype=torch.float16).to(DEV)
        x[0, 300] = bad
        assert llama_ops.norm_linears(x, None, w, 1e-5, [q])[1][0].isnan().all()
    assert not llama_ops.norm_linears(torch.zeros_like(x), None, w, 1e-5, [q])[1][0].any()


# rows at the edges of a wave's 2 / 4 / 8 and of a full round of the grid; widths of
# one to eight chunks of 512, whole, ragged and short of a chunk
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,N", [(8, 1), (512, 9), (520, 40), (1024, 32769), (1536, 130), (2048, 1000),
                                 (2056, 16385), (2560, 17), (3072, 64), (3584, 33), (4096, 8193), (2048, 66001)])
def test_norm_head(dtype, K, N):
    print(f"[norm head] {dtype} K={K} N={N}", flush=True)
    x, d = randn((1, K), 1, 3.0, dtype=dtype).to(DEV), randn((1, K), 2, dtype=dtype).to(DEV)
    w, head = (1 + randn((K,), 3, 0.2, dtype=torch.float32)).to(dtype).to(DEV), randn((N, K), 4, 0.02, dtype=dtype).to(DEV)
    for delta in (None, d):
        got = llama_ops.norm_head(x, delta, w, 1e-5, head)
        h = llama_ops.rms_norm(x, w, 1e-5) if delta is None else llama_ops.rms_norm(x, w, 1e-5, delta)[1]
        want = h.double().cpu() @ head.double().cpu().T  # the rounded norm: its sum is all that may differ
        # K products of 2^-24 each (random walk), and a last bit of the norm here and there
        err = (got.double().cpu() - want).abs() / torch.maximum(want.abs(), want.square().mean().sqrt())
        assert err.max().item() <= 2 * ROUND[dtype] + 1e-4, err.max().item()
    for bad in (torch.nan, torch.inf):
        x[0, K - 1] = bad
        assert llama_ops.norm_head(x, None, w, 1e-5, head).isnan().all()


def test_norm_head_refuses_other_heads():
    x, w = torch.ones((1, 64), device=DEV, dtype=torch.bfloat16), torch.ones(64, device=DEV, dtype=torch.bfloat16)
    head = torch.ones((16, 64), device=DEV, dtype=torch.bfloat16)
    assert llama_ops.norm_head(x, None, w, 1e-5, head) is not None
    wide = torch.ones((16, 128), device=DEV, dtype=torch.bfloat16)
    for h in (head.half(), head.float(), head.t(), wide, wide[:, :64], wide.view(-1)[4:4 + 1024].view(16, 64)):
        assert llama_ops.norm_head(x, None, w, 1e-5, h) is None
    assert llama_ops.norm_head(x.expand(2, 64).contiguous(), None, w, 1e-5, head) is None


def _attention_pair(dtype):
    """An Attention module on the GPU and its copy on the CPU, trainable 16-bit projections."""
    import copy
    from int4_hip.llama import Attention, LlamaConfig
    cpu = Attention(LlamaConfig(hidden_size=128, num_attention_heads=4, num_key_value_heads=2, head_dim=64))
    with torch.no_grad():
        for i, w in enumerate(cpu.parameters()):
            w.copy_(randn(tuple(w.shape), 70 + i, 0.1, dtype=torch.float32))
    cpu = cpu.to(dtype)
    return copy.deepcopy(cpu).to(DEV), cpu


def _run_attention(att, dev, x, decode):
    cos, sin = (t[3:4] if decode else t[:x.shape[0]] for t in _tables(16, 64))
    kc, vc = torch.zeros((2, 64, 16)), torch.zeros((2, 16, 64))
    kc[..., :3], vc[:, :3] = randn((2, 64, 3), 80, dtype=torch.float32), randn((2, 3, 64), 81, dtype=torch.float32)
    args = [t.to(dev) for t in (x, cos.contiguous(), sin.contiguous(), kc, vc)]
    return att(*args, None, torch.tensor([3], device=dev), None) if decode else att(*args, 0, None, None)


# x plain, the projections trainable (a frozen embedding, adapters): every gradient
# flows.  Both sides round each projection, the attention output and their gradients
# to 16 bits (on the CPU one side is at most 1.5 half-ulps from 32-bit arithmetic)
@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_keeps_the_gradients_of_its_projections(dtype, decode):
    gpu, cpu = _attention_pair(dtype)
    x = randn((1 if decode else 9, 128), 82, dtype=dtype)
    outs = [_run_attention(a, dev, x, decode) for a, dev in ((gpu, DEV), (cpu, "cpu"))]
    for o in outs:
        o.float().square().sum().backward()
    assert (outs[0].cpu().float() - outs[1].float()).norm() <= 4 * ROUND[dtype] * outs[1].float().norm()
    for (name, a), b in zip(gpu.named_parameters(), cpu.parameters()):
        assert a.grad is not None, name
        assert (a.grad.cpu().float() - b.grad.float()).norm() <= 8 * ROUND[dtype] * b.grad.float().norm(), name


class _Out(torch.nn.Module):
    """A projection whose output is changed by ``f``."""

    def __init__(self, inner, f):
        super().__init__()
        self.inner, self.f = inner, f

    def forward(self, x):
        return self.f(self.inner(x))


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("form", ["fp32", "one_fp32", "heads", "subclass"])
def test_attention_takes_other_projection_outputs(form, decode):
    """Outputs the kernels do not read as they are (fp32, [T, heads, d], a subclass) go through
    the torch operations, as on the CPU."""
    f = {"fp32": torch.Tensor.float, "one_fp32": torch.Tensor.float, "heads": lambda t: t.view(t.shape[0], -1, 64),
         "subclass": lambda t: t.as_subclass(_Sub)}[form]
    x = randn((1 if decode else 9, 128), 83)
    outs = []
    for att, dev in zip(_attention_pair(torch.bfloat16), (DEV, "cpu")):
        for n in ("k_proj",) if form == "one_fp32" else ("q_proj", "k_proj", "v_proj"):
            setattr(att, n, _Out(getattr(att, n), f))
        with torch.no_grad():
            outs.append(_run_attention(att, dev, x, decode))
    assert outs[0].dtype == outs[1].dtype == x.dtype and isinstance(outs[0], _Sub) == (form == "subclass")
    got, want = (o.as_subclass(torch.Tensor).cpu().float() for o in outs)
    assert (got - want).norm() <= 4 * ROUND[x.dtype] * want.norm()
