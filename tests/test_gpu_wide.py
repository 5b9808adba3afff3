"""GPU parity: the one-wave-per-SIMD prefill kernel that automatic calls take
(every tiling, k-split and form) vs the CPU oracle."""
from __future__ import annotations

import pytest
import torch

from _helpers import DEV, assert_gemm_close, log, np_
from oracle import w4a16_oracle as O

pytestmark = pytest.mark.gpu

# (M, K, N, G, tile_cfg, splits it): partial tiles in M and N, K of less than a
# panel, of an odd number of 32s, of panels short of a block of four, and longer
# than a slice; the 256-row tiles with and without a half-height last round
CASES = [
    (65, 32, 68, 32, 19, False), (129, 4096, 260, 64, 20, True), (257, 224, 1028, 32, 19, False),
    (300, 1056, 4100, 96, 19, False), (128, 4096, 4096, 128, 20, True),
    (300, 512, 14336, 128, 17, False), (600, 320, 4100, 64, 18, False),
    (256, 14336, 4096, 128, 18, True), (256, 4096, 4096, 128, 20, False), (1100, 256, 14340, 128, 16, False),
    (2300, 288, 7172, 32, 16, False), (1024, 256, 16384, 256, 16, False),
]
# small batches on the 32-row tiling: one row tile short, just over and full, k of
# whole and partial panel blocks, columns short of a block, odd group sizes
BATCH = [
    (17, 14336, 4096, 128, 21, True), (32, 4096, 14336, 64, 21, False), (9, 14400, 516, 96, 21, True),
    (16, 14336, 4, 128, 21, True), (31, 8224, 2052, 32, 21, True), (24, 8192, 8192, 128, 21, True),
    (25, 4128, 8196, 32, 21, False),
]
# N % 4 != 0 (M <= 64 keeps the skinny kernel)
ODD = [(65, 32, 7, 32), (93, 2080, 1003, 32), (200, 4096, 1001, 64), (129, 160, 1, 32),
       (300, 288, 4098, 96), (700, 640, 2047, 128)]


def _case(M, K, N, G, seed, frac):
    from w4a16 import quantize_weight

    g = torch.Generator().manual_seed(seed)
    X = torch.randn(M, K, generator=g).to(torch.float16)
    qw, s, z = quantize_weight(torch.randn(K, N, generator=g).to(torch.float16).to(DEV), G)
    if frac:
        z = (z + torch.rand(z.shape, generator=g).to(DEV)).to(torch.float16)
    b = (torch.randn(N, generator=g) * 2).to(torch.float16).to(DEV)
    return X.to(DEV), qw, s, z, b


def _check(X, qw, s, z, b, G, what):
    from w4a16 import w4a16_matmul
    from w4a16.hip_kernel import w4a16_linear

    ref = O.reference_w4a16(np_(X), np_(qw), np_(s), np_(z), G)
    out = w4a16_matmul(X, qw, s, z, G)
    assert_gemm_close(out, ref, what)
    assert torch.equal(w4a16_linear(X, qw, s, z, b, G), out + b), what
    return out


@pytest.mark.parametrize("frac", [False, True])
@pytest.mark.parametrize("M,K,N,G,cfg,split", CASES + BATCH)
def test_wide_tilings(M, K, N, G, cfg, split, frac):
    from w4a16 import _lib, w4a16_matmul

    p = _lib.auto_plan(M, N, K, G)
    log(f"wide M={M} K={K} N={N} G={G} cfg={p.tile_cfg} split={p.split_k} frac={frac}")
    assert (p.tile_cfg, p.split_k > 1) == (cfg, split)
    X, qw, s, z, b = _case(M, K, N, G, M + N + K, frac)
    out = _check(X, qw, s, z, b, G, f"cfg {cfg}")
    # rows apart by K + 8 and N + 4, the gap full of infinities: nothing past K is
    # read into a product (K % 64 == 32: a panel's second half), nothing past N
    # written
    xs = torch.full((M, K + 8), float("inf"), dtype=torch.float16, device=DEV)
    xs[:, :K] = X
    ys = torch.full((M, N + 4), 7.0, dtype=torch.float16, device=DEV)
    w4a16_matmul(xs[:, :K], qw, s, z, G, out=ys[:, :N])
    assert torch.equal(ys[:, :N], out) and bool((ys[:, N:] == 7.0).all())


@pytest.mark.parametrize("frac", [False, True])
@pytest.mark.parametrize("M,K,N,G", ODD)
def test_wide_any_width(M, K, N, G, frac):
    log(f"wide odd M={M} K={K} N={N} G={G} frac={frac}")
    _check(*_case(M, K, N, G, M + N + K, frac), G, f"N={N}")


@pytest.mark.parametrize("M", [1, 20, 64, 100, 300])
def test_unaligned_operands(M):
    """Scales, zeros, bias and out off the vector kernels' alignment (views one
    element into their storage): the skinny kernel up to M = 64, this one beyond.
    With scales and zeros off, the same bits wherever the weight, the output and
    the bias lie."""
    from w4a16 import w4a16_matmul
    from w4a16.hip_kernel import w4a16_linear

    K, N, G = 2080, 516, 32
    X, qw, s, z, b = _case(M, K, N, G, M, False)

    def off(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:]
        return flat.copy_(t.reshape(-1)).view(t.shape)

    ref = O.reference_w4a16(np_(X), np_(qw), np_(s), np_(z), G)
    log(f"unaligned M={M}")
    out = w4a16_matmul(X, qw, off(s), off(z), G)
    assert_gemm_close(out, ref, "unaligned scales and zeros")
    y = off(torch.zeros(M, N, dtype=torch.float16, device=DEV))
    w4a16_matmul(X, off(qw), off(s), off(z), G, out=y)
    assert torch.equal(y, out)
    assert torch.equal(w4a16_linear(X, qw, off(s), off(z), off(b), G), out + b)


def test_wide_nonfinite_scales():
    """An infinite scale and a NaN zero reach exactly the columns they belong to."""
    from w4a16 import w4a16_matmul

    M, K, N, G = 130, 512, 260, 128
    X, qw, s, z, _ = _case(M, K, N, G, 5, True)
    base = w4a16_matmul(X, qw, s, z, G)
    s, z = s.clone(), z.clone()
    s[1, 5], z[2, 77] = float("inf"), float("nan")
    out = w4a16_matmul(X, qw, s, z, G)
    bad = ~torch.isfinite(out)
    assert bool(bad[:, [5, 77]].all()) and int(bad.sum()) == 2 * M
    keep = [c for c in range(N) if c not in (5, 77)]
    assert torch.equal(out[:, keep], base[:, keep])
