"""Python side of the fused kernels that a decoder layer of ``llama.py`` runs
between its linears (csrc/w4_llama.hip).

``fusable`` says whether plain tensors on one GPU are at hand, outside autograd,
tracing and tensor subclasses: only then may a kernel be launched on raw
pointers.  Everything else takes the torch operations of ``llama.py``, which
define the results.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch import _C
from torch.autograd import forward_ad
from torch.compiler import is_compiling as _is_compiling

from . import _lib
from .gemm import _check_weight, _with_workspace

# dtypes of the activations the kernels take, with their codes
DTYPES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_FP16}
_PLAIN = (torch.Tensor, nn.Parameter)


def fusable(*tensors: torch.Tensor) -> bool:
    """Plain tensors on one GPU with nothing recording or transforming the call."""
    if (_is_compiling() or _C._get_tracing_state() is not None or _C._len_torch_dispatch_stack() or
            _C._len_torch_function_stack() or _C._functorch.peek_interpreter_stack() is not None or
            torch.is_autocast_enabled("cuda") or forward_ad._current_level >= 0):
        return False
    dev = tensors[0].device
    if dev.type != "cuda":
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if type(t) not in _PLAIN or t.device != dev or (grad and t.requires_grad):
            return False
    return True


def _on(device: torch.device, call) -> int:
    """``call(stream)`` on the current stream of ``device``, made current."""
    if _C._cuda_getDevice() == device.index:
        return call(_C._cuda_getCurrentRawStream(device.index))
    with torch.cuda.device(device):
        return call(_C._cuda_getCurrentRawStream(device.index))


def _dense(*tensors: torch.Tensor) -> bool:
    return all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in tensors)


_ATTN_WS: dict = {}


def _attn_ws_bytes(nh: int, nkv: int, d: int, max_len: int) -> int:
    """Workspace size of one decode step (0: unsupported shape); a pure function, memoised."""
    key = (nh, nkv, d, max_len)
    b = _ATTN_WS.get(key)
    if b is None:
        if len(_ATTN_WS) > 4096:
            _ATTN_WS.clear()
        b = _ATTN_WS[key] = _lib.load().w4_attention_decode_workspace_bytes(nh, nkv, d, max_len)
    return b


def _qkv_fit(x, qkv, nh: int, nkv: int, d: int) -> bool:
    """Projections of ``x`` [.., hidden] in its dtype and in the shapes the attention
    kernels read by pointer (``fusable`` answers for the rest)."""
    q, k, v = qkv
    lead = x.shape[:-1]
    return (q.dtype == k.dtype == v.dtype == x.dtype and q.shape == (*lead, nh * d)
            and k.shape == v.shape == (*lead, nkv * d))


def attention_decode_ok(x, kc, vc, cos, sin, pos, nh: int, nkv: int, d: int, qkv=()) -> bool:
    """Whether ``attention_decode`` takes a step with activations like ``x``
    ([1, hidden]), the caches ``kc`` [.., nkv, d, L], ``vc`` [.., nkv, L, d] and, where
    they are known, the projections ``qkv``."""
    if x.dtype not in DTYPES:  # (first: models of other types pay for no more)
        return False
    L = kc.shape[-1]
    return (kc.shape[-3:] == (nkv, d, L) and vc.shape == (*kc.shape[:-3], nkv, L, d)
            and x.shape[0] == 1
            and kc.dtype == vc.dtype == cos.dtype == sin.dtype == torch.float32 and pos.dtype == torch.int64
            and pos.numel() == 1 and cos.shape == sin.shape == (1, d // 2)
            and kc.is_contiguous() and vc.is_contiguous() and cos.is_contiguous() and sin.is_contiguous()
            and (not qkv or _qkv_fit(x, qkv, nh, nkv, d))
            and fusable(x, kc, vc, cos, sin, pos, *qkv) and _attn_ws_bytes(nh, nkv, d, L) > 0)


def attention_decode(q, k, v, cos, sin, kc, vc, pos, nh: int, nkv: int, d: int) -> torch.Tensor:
    """Attention output [1, nh * d] of one token: q [nh * d], k, v [nkv * d] values
    before the rotary embedding; the caches of one layer are updated in place."""
    dev = q.device
    max_len = kc.shape[-1]
    q, k, v = (t.contiguous() for t in (q, k, v))
    assert q.dtype == k.dtype == v.dtype and q.numel() == nh * d and k.numel() == v.numel() == nkv * d
    out = torch.empty((1, nh * d), dtype=q.dtype, device=dev)
    lib = _lib.load()
    rc = _on(dev, lambda st: _with_workspace(dev, st, _attn_ws_bytes(nh, nkv, d, max_len), lambda ws, nb:
             lib.w4_attention_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), DTYPES[q.dtype], nh, nkv, d,
                                     cos.data_ptr(), sin.data_ptr(), kc.data_ptr(), vc.data_ptr(), max_len,
                                     pos.data_ptr(), out.data_ptr(), ws, nb, st)))
    if rc:
        _lib.check(rc, "w4_attention_decode")
    return out


def attention_prefill_ok(x, kc, vc, cos, sin, pos0, nh: int, nkv: int, d: int, qkv=()) -> bool:
    """Whether ``attention_prefill`` takes the tokens of ``x`` [T, hidden] at positions
    pos0.. of the caches ``kc`` [nkv, d, L], ``vc`` [nkv, L, d], and their projections ``qkv``."""
    if x.dtype not in DTYPES:
        return False
    T, L = x.shape[0], kc.shape[-1]
    return (x.dim() == 2 and T >= 1 and d in (64, 128) and nh % nkv == 0 and type(pos0) is int
            and 0 <= pos0 <= L - T and L < 1 << 22 and T <= 65535 * 16 and nkv <= 65535
            and kc.dtype == vc.dtype == cos.dtype == sin.dtype == torch.float32
            and kc.shape == (nkv, d, L) and vc.shape == (nkv, L, d) and cos.shape == sin.shape == (T, d // 2)
            and kc.is_contiguous() and cos.is_contiguous() and sin.is_contiguous()
            and (not qkv or _qkv_fit(x, qkv, nh, nkv, d)) and fusable(x, kc, vc, cos, sin, *qkv) and _dense(vc))


def attention_prefill(q, k, v, cos, sin, kc, vc, pos0: int, nh: int, nkv: int, d: int) -> torch.Tensor:
    """Causal attention output [T, nh * d] of T tokens: q [T, nh * d], k, v [T, nkv * d]
    before the rotary embedding; the caches of one layer are updated in place."""
    T, dev = q.shape[0], q.device
    q, k, v = (t if _dense(t) else t.clone(memory_format=torch.contiguous_format) for t in (q, k, v))
    assert q.dtype == k.dtype == v.dtype and q.shape == (T, nh * d) and k.shape == v.shape == (T, nkv * d)
    out = torch.empty_like(q)
    lib = _lib.load()
    rc = _on(dev, lambda st: lib.w4_attention_prefill(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), DTYPES[q.dtype], T, nh, nkv, d, cos.data_ptr(), sin.data_ptr(),
        kc.data_ptr(), vc.data_ptr(), kc.shape[-1], pos0, out.data_ptr(), st))
    if rc:
        _lib.check(rc, "w4_attention_prefill")
    return out


MAX_NORM = 16384                # widest row of w4_rmsnorm
MAX_GRID = (2**32 - 1) // 256   # workgroups of 256 threads in a launch: a row, or 2048 values, each


def rms_norm_ok(x, weight, delta=None) -> bool:
    """Whether ``rms_norm`` takes ``x`` [..., n] (and a residual ``delta`` like it)."""
    if x.dtype not in DTYPES:
        return False
    n = x.shape[-1] if x.dim() else 0
    ts = (x, weight) if delta is None else (x, weight, delta)
    return (0 < n <= MAX_NORM and n % 8 == 0 and weight.shape == (n,)
            and x.numel() <= MAX_GRID * n
            and all(t.dtype == x.dtype for t in ts) and (delta is None or delta.shape == x.shape)
            and fusable(*ts) and _dense(*ts))


def rms_norm(x, weight, eps: float, delta=None):
    """RMSNorm of ``x``; with ``delta`` the pair (x + delta, its RMSNorm)."""
    n = x.shape[-1]
    y = torch.empty_like(x)
    s = None if delta is None else torch.empty_like(x)
    lib = _lib.load()
    rc = _on(x.device, lambda st: lib.w4_rmsnorm(
        x.data_ptr(), None if delta is None else delta.data_ptr(), weight.data_ptr(), DTYPES[x.dtype], x.numel() // n,
        n, eps, None if s is None else s.data_ptr(), y.data_ptr(), st))
    if rc:
        _lib.check(rc, "w4_rmsnorm")
    return y if delta is None else (s, y)


def silu_mul_ok(gate, up) -> bool:
    return (gate.dtype in DTYPES and up.dtype == gate.dtype and up.shape == gate.shape and gate.numel() % 8 == 0
            and gate.numel() <= MAX_GRID * 2048 and fusable(gate, up) and _dense(gate, up))


def silu_mul(gate, up) -> torch.Tensor:
    """silu(gate) * up in one pass, one rounding."""
    y = torch.empty_like(gate)
    lib = _lib.load()
    rc = _on(gate.device, lambda st: lib.w4_silu_mul(gate.data_ptr(), up.data_ptr(), DTYPES[gate.dtype], gate.numel(),
                                                     y.data_ptr(), st))
    if rc:
        _lib.check(rc, "w4_silu_mul")
    return y


def _row_problems(x, weights):
    """(problem array, outputs) of one-row products on ``x`` [1, K], or None where the
    weights are not plain dense buffers on x's GPU."""
    K, dev = x.shape[-1], x.device
    probs = (_lib.Problem * len(weights))()
    outs = []
    for i, (qw, s, z) in enumerate(weights):
        if not (fusable(x, qw, s, z) and qw.is_contiguous() and s.is_contiguous() and z.is_contiguous()):
            return None
        assert qw.shape[0] * 8 == K
        G, N = _check_weight(qw, s, z, K), qw.shape[1]
        y = torch.empty((1, N), dtype=x.dtype, device=dev)
        probs[i] = _lib.Problem(x.data_ptr(), qw.data_ptr(), s.data_ptr(), z.data_ptr(), y.data_ptr(), N, K, G, 0)
        outs.append(y)
    return probs, outs


def norm_linears(x, delta, weight, eps: float, weights):
    """(x + delta, [rmsnorm(x + delta) @ W_i^T ...]) of one row in one launch; None where
    no such launch exists (nothing has been launched then)."""
    if not (x.dim() == 2 and x.shape[0] == 1 and 1 <= len(weights) <= _lib.MAX_GROUPED
            and rms_norm_ok(x, weight, delta)):
        return None
    row = _row_problems(x, weights)
    if row is None:
        return None
    probs, outs = row
    total = x if delta is None else torch.empty_like(x)
    lib, dev = _lib.load(), x.device
    nbytes = lib.w4a16_grouped_workspace_bytes(probs, len(weights), 1)
    rc = _on(dev, lambda st: _with_workspace(dev, st, nbytes, lambda ws, nb: lib.w4a16_decode_norm(
        probs, len(weights), DTYPES[x.dtype], None if delta is None else delta.data_ptr(), weight.data_ptr(), eps,
        None if delta is None else total.data_ptr(), ws, nb, st)))
    if rc == _lib.ERR_UNSUPPORTED:
        return None
    if rc:
        _lib.check(rc, "w4a16_decode_norm")
    return total, outs


def silu_linear(gate, up, weight):
    """(silu(gate) * up) @ W^T of one row in one launch; None where no such launch exists."""
    if not (gate.dim() == 2 and gate.shape[0] == 1 and silu_mul_ok(gate, up)):
        return None
    row = _row_problems(gate, [weight])
    if row is None:
        return None
    probs, outs = row
    lib, dev = _lib.load(), gate.device
    nbytes = lib.w4a16_grouped_workspace_bytes(probs, 1, 1)
    rc = _on(dev, lambda st: _with_workspace(dev, st, nbytes, lambda ws, nb: lib.w4a16_decode_silu(
        probs, DTYPES[gate.dtype], up.data_ptr(), ws, nb, st)))
    if rc == _lib.ERR_UNSUPPORTED:
        return None
    if rc:
        _lib.check(rc, "w4a16_decode_silu")
    return outs[0]


def norm_head(x, delta, weight, eps: float, head):
    """rmsnorm(x + delta) @ head^T of one row for a 16-bit ``head`` [N, K] in one launch;
    None where no such launch exists."""
    if not (x.dim() == 2 and x.shape[0] == 1 and x.shape[1] <= 4096 and head.dim() == 2 and head.dtype == x.dtype
            and head.shape[1] == x.shape[1] and 0 < head.shape[0] < 1 << 30 and rms_norm_ok(x, weight, delta)
            and fusable(x, head) and _dense(head)):
        return None
    N, K = head.shape
    y = torch.empty((1, N), dtype=x.dtype, device=x.device)
    lib = _lib.load()
    rc = _on(x.device, lambda st: lib.w4_norm_head(
        x.data_ptr(), None if delta is None else delta.data_ptr(), weight.data_ptr(), eps, head.data_ptr(),
        DTYPES[x.dtype], N, K, y.data_ptr(), st))
    if rc:
        _lib.check(rc, "w4_norm_head")
    return y
