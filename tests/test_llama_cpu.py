"""CPU checks of the Llama harness model (no GPU, no HIP library): the layer
math against Hugging Face's LlamaForCausalLM on the same weights, and the
static-cache decode step against the prefill logits."""
import pytest
import torch

import int4_hip
from int4_hip import llama, llama_ops
from int4_hip.llama import Attention, LlamaConfig, LlamaForCausalLM

TINY = LlamaConfig(vocab_size=97, hidden_size=64, intermediate_size=160, num_hidden_layers=2,
                   num_attention_heads=8, num_key_value_heads=2, head_dim=8, rope_theta=500000.0,
                   rope_scaling=(32.0, 1.0, 4.0, 64))


def _model(seed=0):
    m = LlamaForCausalLM(TINY)
    m.init_weights(seed)
    g = torch.Generator().manual_seed(seed + 100)
    with torch.no_grad():  # non-trivial norm weights
        for layer in m.model.layers:
            layer.input_layernorm.weight.uniform_(0.5, 1.5, generator=g)
            layer.post_attention_layernorm.weight.uniform_(0.5, 1.5, generator=g)
        m.model.norm.weight.uniform_(0.5, 1.5, generator=g)
    m.allocate_cache(40, torch.float32, "cpu")
    return m.eval()


def test_matches_hf_llama():
    transformers = pytest.importorskip("transformers")
    m = _model()
    hc = transformers.LlamaConfig(
        vocab_size=TINY.vocab_size, hidden_size=TINY.hidden_size, intermediate_size=TINY.intermediate_size,
        num_hidden_layers=TINY.num_hidden_layers, num_attention_heads=TINY.num_attention_heads,
        num_key_value_heads=TINY.num_key_value_heads, head_dim=TINY.head_dim, rms_norm_eps=TINY.rms_norm_eps,
        rope_theta=TINY.rope_theta, max_position_embeddings=128, tie_word_embeddings=True,
        rope_scaling={"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                      "original_max_position_embeddings": 64},
        attn_implementation="eager")
    hf = transformers.LlamaForCausalLM(hc).eval()
    missing, unexpected = hf.load_state_dict(
        {k: v for k, v in m.state_dict().items() if not k.startswith(("kc", "vc"))}, strict=False)
    assert not unexpected and all("rotary" in k for k in missing), (missing, unexpected)
    ids = torch.randint(0, TINY.vocab_size, (1, 33), generator=torch.Generator().manual_seed(3))
    with torch.no_grad():
        ref = hf(ids).logits[0]
        got = m.prefill(ids[0])
    torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-4)


def test_decode_steps_match_prefill():
    m = _model(1)
    ids = torch.randint(0, TINY.vocab_size, (30,), generator=torch.Generator().manual_seed(4))
    full = m.prefill(ids)
    m2 = _model(1)
    m2.prefill(ids[:10])
    for t in range(10, 30):
        step = m2.decode_step(ids[t:t + 1], torch.tensor([t]))
        torch.testing.assert_close(step[0], full[t], rtol=1e-4, atol=1e-4)


def test_decode_kernel_takes_only_caches_of_its_shapes(monkeypatch):
    """The host rule alone (what it asks about devices set aside): the kernel indexes both
    caches by the heads, the head size and the keys' length."""
    monkeypatch.setattr(llama_ops, "fusable", lambda *a: True)
    monkeypatch.setattr(llama_ops, "_attn_ws_bytes", lambda *a: 1)
    x, row, pos = torch.zeros(1, 8, dtype=torch.bfloat16), torch.zeros(1, 32), torch.zeros(1, dtype=torch.long)

    def ok(k, v):
        return llama_ops.attention_decode_ok(x, torch.zeros(k), torch.zeros(v), row, row, pos, 4, 2, 64)

    assert ok((2, 64, 20), (2, 20, 64)) and ok((3, 2, 64, 20), (3, 2, 20, 64))
    for k, v in (((2, 64, 20), (2, 19, 64)), ((2, 64, 20), (2, 21, 64)), ((2, 64, 20), (1, 20, 64)),
                 ((1, 64, 20), (1, 20, 64)), ((2, 32, 20), (2, 20, 32)), ((2, 64, 20), (2, 20, 32)),
                 ((3, 2, 64, 20), (2, 2, 20, 64)), ((64, 20), (20, 64)), ((2, 64, 20), (2 * 20 * 64,))):
        assert not ok(k, v), (k, v)


def _no_kernel(*a):
    raise AssertionError("the decode kernel was chosen")


def test_decode_step_leaves_other_tables_and_heads_to_torch(monkeypatch):
    """Tables longer than the cache would let a position past it through; an attention module
    with other heads does not fit the caches (torch says so)."""
    monkeypatch.setattr(llama_ops, "attention_decode_ok", lambda *a: True)
    monkeypatch.setattr(llama_ops, "attention_decode", _no_kernel)
    m, tok, pos = _model(), torch.tensor([3]), torch.tensor([0])
    with pytest.raises(AssertionError, match="chosen"):
        m.decode_step(tok, pos)
    m.cos, m.sin = (torch.cat((t, t)) for t in (m.cos, m.sin))
    m.decode_step(tok, pos)
    m = _model()
    m.model.layers[1].self_attn = Attention(LlamaConfig(**{**vars(TINY), "num_key_value_heads": 4}))
    with pytest.raises((RuntimeError, IndexError)):
        m.decode_step(tok, pos)


def test_decode_layer_leaves_other_modules_alone():
    """An MLP of another kind need not have this one's linears: not this function's layer."""
    layer = _model().model.layers[0]
    assert llama._decode_layer(layer, *[None] * 7) is None  # its linears are not int4
    for other in (torch.nn.Identity(), torch.nn.Sequential(layer.mlp)):
        layer.mlp = other
        assert llama._decode_layer(layer, *[None] * 7) is None


def test_norm_without_an_epsilon_is_left_to_torch(monkeypatch):
    """eps=None means torch's choice; the kernels take a number."""
    m = _model()
    for n in [m.model.norm] + [n for l in m.model.layers for n in (l.input_layernorm, l.post_attention_layernorm)]:
        n.eps = None
    want = m.prefill(torch.arange(5)), m.decode_step(torch.tensor([3]), torch.tensor([5]))
    monkeypatch.setattr(llama_ops, "rms_norm_ok", lambda *a: True)
    for f in ("rms_norm", "norm_linears", "norm_head"):
        monkeypatch.setattr(llama_ops, f, _no_kernel)
    assert torch.equal(m.prefill(torch.arange(5)), want[0])
    assert torch.equal(m.decode_step(torch.tensor([3]), torch.tensor([5])), want[1])


@pytest.mark.parametrize("cls", [llama.RMSNorm, llama.Attention, llama.MLP, int4_hip.Int4Linear, torch.nn.Linear])
def test_a_forward_replaced_on_the_class_counts(cls, monkeypatch):
    """A forward patched on the class (profilers, other kernels) is no longer the one the fused
    launches stand for."""
    m = _model()
    mod = {llama.RMSNorm: m.model.norm, llama.Attention: m.model.layers[0].self_attn,
           llama.MLP: m.model.layers[0].mlp, torch.nn.Linear: m.lm_head}.get(cls) or int4_hip.Int4Linear(64, 64, 32)
    assert llama._plain(mod, cls)
    own = cls.forward
    with monkeypatch.context() as patch:
        patch.setattr(cls, "forward", lambda self, *a: own(self, *a))
        assert not llama._plain(mod, cls)
    assert llama._plain(mod, cls)


def test_norm_and_activation_kernels_leave_launches_hip_refuses(monkeypatch):
    """A workgroup per row, or per 2048 values, of 256 threads: below 2^32 threads in all."""
    monkeypatch.setattr(llama_ops, "fusable", lambda *a: True)
    monkeypatch.setattr(llama_ops, "_dense", lambda *a: True)

    def meta(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="meta")

    assert llama_ops.rms_norm_ok(meta((1 << 24) - 1, 8), meta(8))
    assert not llama_ops.rms_norm_ok(meta(1 << 24, 8), meta(8))
    assert not llama_ops.rms_norm_ok(meta(1 << 12, 1 << 12, 8), meta(8), meta(1 << 12, 1 << 12, 8))
    for n, ok in (((1 << 24) - 1, True), (1 << 24, False)):
        assert llama_ops.silu_mul_ok(meta(n, 2048), meta(n, 2048)) == ok


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norm_and_mlp_can_be_traced_symbolically(dtype):
    """The host rules decide on what a symbolic tracer's stand-in cannot answer for: they
    leave it to torch's operations first."""
    m, x = _model().to(dtype), torch.randn(3, 64).to(dtype)
    for mod in (m.model.norm, m.model.layers[0].mlp):
        assert torch.equal(torch.fx.symbolic_trace(mod)(x), mod(x))
