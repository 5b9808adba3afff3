"""The automatic call through csrc/native.cpp: the same bits as the Python path's
call for every form it takes, and every other form left to the Python path.

The untuned call of the tuner (w4a16_matmul_untuned) always goes through the
Python checks and ctypes, so it is the other side of each comparison.
"""
from __future__ import annotations

import pytest
import torch

from _helpers import DEV, log

EMPTY = dict(device=DEV, dtype=torch.float16)


def _operands(M, K, N, G, frac=False, seed=0):
    from w4a16 import quantize_weight

    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.float16).to(DEV)
    qw, s, z = quantize_weight((torch.randn(K, N, generator=g) * 0.05).half().to(DEV), G)
    return x, qw, s, (z + 0.5 if frac else z)


def _native(*args):
    from w4a16 import _lib, hip_kernel

    return _lib.load_native(hip_kernel._ZKEY).gemm(*args)


def test_native_module_is_of_these_sources():
    """The module carries the hash of its source, the header and torch's version;
    operands it does not take (here: on the CPU, or not tensors) give None."""
    from w4a16 import _build, _lib, hip_kernel

    mod = _lib.load_native(hip_kernel._ZKEY)
    assert mod.build_id() == _build.native_hash()
    x = torch.zeros(2, 64, dtype=torch.float16)
    assert mod.gemm(x, x, x, x, None, 32, None, None, None) is None
    assert mod.gemm(None, x, x, x, None, 32, None, None, None) is None
    assert mod.gemm(x) is None


def test_without_the_native_module(monkeypatch):
    """A missing or foreign _native.so: one warning, and every call is left to the
    Python path; an unusable library stays an error."""
    from w4a16 import _lib, hip_kernel

    def missing(key):
        raise ImportError("cannot import _native.so")

    class OnDevice(torch.Tensor):
        is_cuda = True

    loader = hip_kernel._native_gemm
    x = torch.zeros(2, 64, dtype=torch.float16).as_subclass(OnDevice)
    monkeypatch.setattr(_lib, "load_native", missing)
    monkeypatch.setattr(hip_kernel, "_native_gemm", loader)   # undone afterwards
    with pytest.warns(RuntimeWarning, match="_native.so"):
        call = hip_kernel._load_native_gemm()
    assert call(x, x, x, x, None, 32, None, None, None) is None
    if getattr(loader, "__name__", "") == "_native_gemm":   # not taken the place of yet
        with pytest.warns(RuntimeWarning, match="_native.so"):
            assert loader(x, x, x, x, None, 32, None, None, None) is None

    def unusable():
        raise ImportError("no library")

    monkeypatch.setattr(_lib, "load", unusable)
    with pytest.raises(ImportError, match="no library"):
        hip_kernel._load_native_gemm()


@pytest.mark.gpu
def test_calls_without_the_native_module(monkeypatch):
    """The public entry points on the device with the native call out of the way."""
    from w4a16 import W4A16Linear, hip_kernel, w4a16_matmul

    x, qw, s, z = _operands(33, 512, 260, 64)
    lin = torch.nn.Linear(512, 260, device=DEV, dtype=torch.float16)
    layer = W4A16Linear.from_linear(lin, 64)
    want = w4a16_matmul(x, qw, s, z, 64), layer(x[None])
    monkeypatch.setattr(hip_kernel, "_native_gemm", lambda *args: None)
    log("without the native module")
    assert torch.equal(w4a16_matmul(x, qw, s, z, 64), want[0])
    assert torch.equal(layer(x[None]), want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,G,frac", [(1, 256, 256, 128, False), (7, 512, 260, 64, True),
                                          (33, 1024, 1003, 32, False), (300, 512, 1024, 128, True),
                                          (64, 4096, 512, 128, False)])
def test_native_equals_python_path(M, K, N, G, frac):
    from w4a16 import w4a16_matmul
    from w4a16.hip_kernel import w4a16_linear, w4a16_matmul_untuned

    x, qw, s, z = _operands(M, K, N, G, frac)
    log(f"native M={M} K={K} N={N} G={G} frac={frac}")
    args = (None, G, None, None, None)
    if frac:   # not checked yet: the Python path's turn
        assert _native(x, qw, s, z, *args) is None
    want = w4a16_matmul_untuned(x, qw, s, z, G, torch.empty(M, N, **EMPTY))
    y = _native(x, qw, s, z, *args)
    assert y is not None and torch.equal(y, want)
    assert y.shape == (M, N) and y.dtype == torch.float16 and not y.requires_grad
    bias = torch.randn(N, **EMPTY)
    assert torch.equal(w4a16_linear(x, qw, s, z, bias, G), want + bias)
    # row-strided views of x and out
    wide = torch.empty(M, K + 24, **EMPTY)
    xv = wide[:, 8:8 + K]
    xv.copy_(x)
    buf = torch.full((M, N + 16), float("nan"), **EMPTY)
    ov = buf[:, 8:8 + N]
    got = _native(xv, qw, s, z, None, G, ov, None, None)
    assert got is ov
    ref = w4a16_matmul_untuned(xv, qw, s, z, G, torch.empty_like(buf)[:, 8:8 + N])
    assert torch.equal(ov, ref)
    assert torch.isnan(buf[:, :8]).all() and torch.isnan(buf[:, 8 + N:]).all()
    # an in-place change of zeros is checked again
    z.add_(0.25)
    assert _native(x, qw, s, z, *args) is None
    changed = w4a16_matmul(x, qw, s, z, G)
    assert torch.equal(changed, w4a16_matmul_untuned(x, qw, s, z, G, torch.empty_like(changed)))
    # another stream, and a captured call replayed between eager ones
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        assert torch.equal(_native(x, qw, s, z, *args), changed)
    torch.cuda.current_stream().wait_stream(st)
    out = torch.empty(M, N, **EMPTY)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert _native(x, qw, s, z, None, G, out, None, None) is out
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, changed)
        w4a16_matmul(x, qw, s, z, G)


@pytest.mark.gpu
def test_native_leaves_other_forms_to_python():
    """Every call outside the plain ones gives None, and the public entry point
    then does what the Python path does: the same errors, results and modes."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from w4a16 import w4a16_matmul

    M, K, N, G = 4, 256, 256, 64
    x, qw, s, z = _operands(M, K, N, G)
    want = w4a16_matmul(x, qw, s, z, G)
    tail = (None, None, None)

    class Sub(torch.Tensor):
        pass

    refused = [
        (x.float(), qw, s, z, G), (x, qw.long(), s, z, G), (x, qw, s.float(), z, G),
        (x.cpu(), qw, s, z, G), (x, qw.cpu(), s, z, G), (x, qw, s, z, 0), (x, qw, s, z, -64),
        (x, qw, s, z, 8), (x, qw, s, z, 48), (x, qw, s, z, 128), (x[:, :128], qw, s, z, G),
        (x.t().contiguous().t(), qw, s, z, G), (x[0], qw, s, z, G), (x[None], qw, s, z, G),
        (x, qw.t().contiguous().t(), s, z, G), (x, qw, s[:2], z, G), (x, qw, s, z[:, :128], G),
    ]
    for i, (a, b, c, d, g) in enumerate(refused):
        assert _native(a, b, c, d, None, g, *tail) is None, i
        with pytest.raises(AssertionError):
            w4a16_matmul(a, b, c, d, g)
    for bad in (torch.empty(M, N, device=DEV), torch.empty(M, N + 8, **EMPTY),
                torch.empty(N, M, **EMPTY).t(), torch.empty(M, N, dtype=torch.float16)):
        assert _native(x, qw, s, z, None, G, bad, None, None) is None
        with pytest.raises(AssertionError):
            w4a16_matmul(x, qw, s, z, G, out=bad)
    assert _native(x[:0], qw, s, z, None, G, *tail) is None
    assert _native(x.as_subclass(Sub), qw, s, z, None, G, *tail) is None
    assert torch.equal(w4a16_matmul(x.as_subclass(Sub), qw, s, z, G), want)

    class F(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class D(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (F, D):
        with mode():
            assert _native(x, qw, s, z, None, G, *tail) is None
            got = w4a16_matmul(x, qw, s, z, G)
        assert torch.equal(got, want)
    with torch.inference_mode():
        assert torch.equal(w4a16_matmul(x, qw, s, z, G), want)
    with torch.device(DEV):
        assert torch.equal(w4a16_matmul(x, qw, s, z, G), want)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
def test_linear_forward_forms(bias):
    """W4A16Linear.forward: leading dimensions, strided rows, buffers and bias
    replaced after construction, and a subclass all agree with w4a16_linear."""
    from w4a16 import W4A16Linear
    from w4a16.hip_kernel import w4a16_linear

    torch.manual_seed(3)
    lin = torch.nn.Linear(256, 192, bias=bias, device=DEV, dtype=torch.float16)
    layer = W4A16Linear.from_linear(lin, 64)
    X = torch.randn(2, 3, 5, 256, **EMPTY)

    def want(m, rows):
        return w4a16_linear(rows.reshape(-1, 256).contiguous(), m.qweight, m.scales, m.zeros,
                            m.bias, 64)

    for x in (X, X[0], X[0, 0], X[0, 0, 0], X[0, 0][::2], X[:, 1], X.transpose(0, 1),
              torch.randn(256, 4, **EMPTY).t()):
        y = layer(x)
        assert y.shape == (*x.shape[:-1], 192)
        assert torch.equal(y.reshape(-1, 192), want(layer, x))
    assert layer(X[:0]).shape == (0, 3, 5, 192)
    layer.bias = torch.randn(192, **EMPTY)
    assert torch.equal(layer(X[0, 0]), want(layer, X[0, 0]))
    del layer.bias
    layer.bias = torch.nn.Parameter(torch.randn(192, **EMPTY), requires_grad=False)
    assert torch.equal(layer(X[0, 0]), want(layer, X[0, 0]))
    layer.in_features = 128
    with pytest.raises(AssertionError):
        layer(X[0, 0])
    layer.in_features = 256

    class Own(W4A16Linear):
        pass

    own = Own.from_linear(lin, 64)
    assert torch.equal(own(X[0, 0]), want(own, X[0, 0]))
