"""GPU: the native call path of the Python entry points (int4_hip._int4_torch)
against the general Python path: the same bits for what it takes, and None for
everything it leaves to that path."""
import threading

import pytest
import torch

import int4_hip
from _synth import randn
from int4_hip import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(call):
    """(native, general) results of ``call``."""
    _lib.load()
    ext = _lib.ext
    assert ext is not None
    native = call()
    _lib.ext = None
    try:
        general = call()
    finally:
        _lib.ext = ext
    return native, general


def _same(a, b):
    if isinstance(a, (list, tuple)):
        assert len(a) == len(b) and type(a) is type(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a.dtype == b.dtype and a.shape == b.shape and a.is_contiguous() == b.is_contiguous()
        assert a.requires_grad == b.requires_grad
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(2048,), (1, 2048), (2, 3, 2048), (100, 2048)])
def test_matmul_paths_agree(dtype, shape):
    q = int4_hip.quantize_int4(randn((520, 2048), 1, 0.02, dtype=dtype).to(DEV), 128)
    x = randn(shape, 2, dtype=dtype).to(DEV)
    for form in (x, torch.nn.Parameter(x), x.clone().requires_grad_()):
        assert _lib.ext.matmul(form, *q) is not None
        _same(*_both(lambda: int4_hip.w4a16_matmul(form, *q)))
    many = [q, int4_hip.quantize_int4(randn((64, 2048), 3, 0.02, dtype=dtype).to(DEV), 128)]
    assert _lib.ext.matmul_grouped([x, x], many, None) is not None
    _same(*_both(lambda: int4_hip.w4a16_matmul_grouped([x, x], many)))
    if x.dim() == 2:
        def into():
            outs = [torch.zeros((x.shape[0], w[0].shape[1]), dtype=dtype, device=DEV) for w in many]
            got = int4_hip.w4a16_matmul_grouped((x, x), tuple(many), out=outs)
            assert all(a.data_ptr() == b.data_ptr() for a, b in zip(got, outs))
            return got
        _same(*_both(into))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_quantize_paths_agree(dtype):
    w = randn((72, 1024), 1, 0.02, dtype=dtype).to(DEV)
    for v in (w, w.t().contiguous().t(), w[:, 512:], w[::2]):  # any strides
        for g in (32, 512, -1):
            assert _lib.ext.quantize(v, g) is not None and _lib.ext.quantize_grouped([v], g) is not None
            _same(*_both(lambda: int4_hip.quantize_int4(v, g)))
            _same(*_both(lambda: int4_hip.quantize_int4_grouped([v, w[:, -512:]], g)))
    q = int4_hip.quantize_int4(w, 64)
    for odt in (torch.bfloat16, torch.float16, torch.float32):
        assert _lib.ext.dequantize(*q, odt) is not None
        _same(*_both(lambda: int4_hip.dequantize_int4(*q, odt)))


def test_left_to_the_general_path():
    q, s, z = int4_hip.quantize_int4(randn((64, 512), 1, 0.02).to(DEV), 64)
    x = randn((4, 512), 2).to(DEV)
    ext = _lib.ext
    assert ext.matmul(x, q, s, z) is not None

    class Sub(torch.Tensor):
        pass

    odd = [(x.t().contiguous().t(), q, s, z), (x.cpu(), q, s, z), (x.float(), q, s, z), (x[:, :256], q, s, z),
           (x[:0], q, s, z), (x.as_subclass(Sub), q, s, z), (x, q.t().contiguous().t(), s, z), (x, q.cpu(), s, z),
           (x, q, s.float(), z), (x, q, s[:4], z), (x, q, s[:, :32], z[:, :32]), (x, q, s, None), (None, q, s, z)]
    for a in odd:
        assert ext.matmul(*a) is None and ext.matmul_grouped([a[0]], [a[1:]], None) is None
    assert ext.matmul_grouped([], [], None) is None and ext.matmul_grouped([x] * 9, [(q, s, z)] * 9, None) is None
    assert ext.matmul_grouped([x, x[:2]], [(q, s, z)] * 2, None) is None
    assert ext.matmul_grouped([x], [(q, s, z)], [torch.empty((4, 128), device=DEV, dtype=x.dtype)[:, :64]]) is None
    flat = torch.empty(4 * 512 + 1, device=DEV, dtype=x.dtype)[1:].view(4, 512)
    assert ext.matmul_grouped([flat], [(q, s, z)], None) is None  # misaligned: copied by the general path
    for w, g in ((x, 24), (x, 1024), (x, 0), (x, 4), (x.float(), 64), (x.cpu(), 64), (x[0], 64), (x, 64.0), (x[:0], 64)):
        assert ext.quantize(w, g) is None and ext.quantize_grouped([w], g) is None
    assert ext.dequantize(q, s, z, torch.int8) is None and ext.dequantize(q.cpu(), s, z, x.dtype) is None
    # errors stay the general path's
    with pytest.raises(AssertionError):
        int4_hip.w4a16_matmul(x.float(), q, s, z)
    with pytest.raises(AssertionError):
        int4_hip.quantize_int4(x, 24)
    # modes and transforms that have to see the operations
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert ext.matmul(x, q, s, z) is None
    with torch.overrides.TorchFunctionMode():
        assert ext.matmul(x, q, s, z) is None
    torch.func.vmap(lambda t: (_none(ext.matmul(t, q, s, z)), t)[1])(x)
    torch.func.jvp(lambda t: (_none(ext.matmul(t, q, s, z)), t)[1], (x,), (x,))


def _none(v):
    assert v is None


def test_threads_and_streams():
    """Calls from several threads, each on a stream of its own, with a product that needs
    that stream's workspace: the bits of a lone call."""
    q = int4_hip.quantize_int4(randn((2048, 8192), 1, 0.02).to(DEV), 128)
    x = randn((16, 8192), 2).to(DEV)
    want = int4_hip.w4a16_matmul(x, *q)
    torch.cuda.synchronize()
    bad = []

    def work():
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            outs = [int4_hip.w4a16_matmul(x, *q) for _ in range(50)]
        st.synchronize()
        if not all(torch.equal(o, want) for o in outs):
            bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("group", [1 << 31, 1 << 63, 1 << 70, -(1 << 70), -2])
def test_group_sizes_no_weight_has(group):
    """Refused as the general path refuses them, whatever their size."""
    w = randn((8, 64), 1).to(DEV)
    int4_hip.quantize_int4(w, 64)  # (loads the library)
    assert _lib.ext.quantize(w, group) is None and _lib.ext.quantize_grouped([w], group) is None
    for call in (lambda: int4_hip.quantize_int4(w, group), lambda: int4_hip.quantize_int4_grouped([w], group)):
        with pytest.raises(AssertionError):
            call()


def test_grouped_operands_outlive_the_callers_lists():
    """Another thread may take the operands out of the lists while the call waits for its
    workspace: it holds them itself."""
    from int4_hip import gemm
    q = int4_hip.quantize_int4(randn((2048, 8192), 1, 0.02).to(DEV), 128)
    x = randn((1, 8192), 2).to(DEV)
    assert int4_hip.gemm.grouped_workspace_bytes([x], [q]) > 0
    want = int4_hip.w4a16_matmul_grouped([x], [q])[0].clone()
    xs, ws, seen = [x.clone()], [tuple(t.clone() for t in q)], []

    def workspace(*args):
        sizes = [(t.shape, t.dtype) for t in (xs[0], *ws[0])]
        xs.clear(), ws.clear()
        seen.extend(torch.empty(s, dtype=d, device=DEV).fill_(1) for s, d in sizes)  # where they were, if freed
        return gemm._workspace_address(*args)

    lib = _lib.load()
    try:
        _lib._load_ext(lib, workspace)
        got = _lib.ext.matmul_grouped(xs, ws, None)[0]
    finally:
        _lib._load_ext(lib)
    assert len(seen) == 4 and torch.equal(got, want)
