"""GPU parity: quantise / pack / unpack / dequantise kernels vs the CPU oracle.

Bit-exact comparisons (int32 words, fp16 bit patterns including -0.0
zero-points) against ``oracle/w4a16_oracle.py`` on the same inputs; mirrors the
reference's test_quant.py (w4a16-kernel/tests/test_quant.py) on the device.
"""
from __future__ import annotations

import json
import os

import numpy as np
import pytest
import torch

from _helpers import DEV, log, np_
from oracle import w4a16_oracle as O

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "known_answers.json")


def _assert_quant_equal(W: torch.Tensor, G: int, what: str):
    from w4a16 import quantize_weight

    qw, s, z = quantize_weight(W.to(DEV), G)
    rq, rs, rz = O.quantize_weight(np_(W), G)
    assert qw.dtype == torch.int32 and s.dtype == torch.float16 and z.dtype == torch.float16
    assert np.array_equal(np_(qw), rq), f"{what}: qweight differs"
    assert np.array_equal(np_(s).view(np.uint16), rs.view(np.uint16)), f"{what}: scales differ"
    assert np.array_equal(np_(z).view(np.uint16), rz.view(np.uint16)), f"{what}: zeros differ"
    return qw, s, z


def test_quantize_known_answers():
    from w4a16 import pack_int4, quantize_weight, unpack_int4

    for c in json.load(open(GOLDEN)):
        log(c["name"])
        if c["kind"] == "pack":
            q = torch.tensor(c["codes"], dtype=torch.int32).reshape(c["K"], c["N"]).to(DEV)
            w = pack_int4(q)
            assert (np_(w).view(np.uint32).reshape(-1).tolist()) == c["words_u32"]
            assert torch.equal(unpack_int4(w), q)
        else:
            W = torch.tensor(c["W"], dtype=torch.float16).reshape(c["K"], c["N"]).to(DEV)
            qw, s, z = quantize_weight(W, c["G"])
            assert np_(unpack_int4(qw)).reshape(-1).tolist() == c["codes"]
            if "zeros_bits" in c:
                assert np_(z).view(np.uint16).reshape(-1).tolist() == c["zeros_bits"]
            if "scales_bits" in c:
                assert np_(s).view(np.uint16).reshape(-1).tolist() == c["scales_bits"]


@pytest.mark.parametrize("K,N,G", [
    (1024, 1024, 128),   # C1 shape
    (256, 64, 32),
    (128, 40, 64),
    (64, 33, 16),        # N % 4 != 0: one column per thread
    (8, 1, 4),           # G < 8: packed words straddle groups
    (24, 12, 12),        # G % 8 != 0
    (4096, 512, 128),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_quantize_bit_exact_random(K, N, G, dtype):
    log(f"quantize K={K} N={N} G={G} {dtype}")
    g = torch.Generator().manual_seed(K * 31 + N * 7 + G)
    W = (torch.randn(K, N, generator=g) * 0.05).to(dtype)
    _assert_quant_equal(W, G, f"K={K} N={N} G={G}")


def test_quantize_special_values():
    """Constant groups (scale 1), exact ties, zero minima (-0.0 zero-point), both
    zero signs, fp16 subnormals, huge ranges, and ties of W/scale at .5."""
    log("quantize special values")
    K, N, G = 64, 16, 32
    W = torch.zeros(K, N, dtype=torch.float16)
    W[:, 0] = 3.0
    W[:, 1] = -2.5
    W[:32, 2] = torch.tensor([0, 0.03125, 0.09375, 0.15625, 0.9375, 0.5, 0.25, 0.46875] * 4)
    W[:8, 3] = torch.tensor([0.0, -0.0, 1.0, 0.5, 0.25, 0.75, 0.125, 0.375])
    W[:8, 4] = torch.tensor([-0.0, 0.0, 1.0, 0.5, 0.25, 0.75, 0.125, 0.375])
    W[:, 5] = torch.tensor([6e-8, 1.2e-7, 3e-6, 6.1e-5] * 16, dtype=torch.float16)
    W[:, 6] = torch.linspace(-60000, 60000, K).to(torch.float16)
    W[:, 7] = -1e-3
    g = torch.Generator().manual_seed(5)
    W[:, 8:] = (torch.randn(K, 8, generator=g) * 1e-4).to(torch.float16)
    _assert_quant_equal(W, G, "special values")
    _assert_quant_equal(W, 8, "special values G=8")


@pytest.mark.parametrize("K,N,G", [
    (128, 68, 32),       # 4 columns per thread: block columns 0-63, tail 64-67
    (64, 33, 8),         # one column per thread: block 0-31, tail column 32
    (64, 70, 16),
    (48, 40, 12),        # G % 8 != 0 kernel
    (512, 1, 32),        # N = 1, G >= 32: torch's inner reduction
    (1024, 1, 64),
    (576, 1, 36),        # N = 1 through the G % 8 != 0 kernel
    (4096, 1, 4096),     # one group
    (256, 1, 16),        # N = 1, G < 32: first zero
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_quantize_mixed_zero_minima(K, N, G, dtype):
    """Groups whose minimum is a zero and that hold both +0.0 and -0.0 at random
    rows: the zero-point's sign bit follows which zero torch's CPU amin returns
    (block / tail columns, N = 1 lanes), bit-exact against the oracle."""
    log(f"quantize mixed zero minima K={K} N={N} G={G} {dtype}")
    rng = np.random.default_rng(K * 13 + N * 7 + G)
    ng = K // G
    W = (np.abs(rng.standard_normal((ng, G, N))) * 0.1 + 0.01).astype(np.float32)
    for _ in range(3):
        rows = rng.integers(0, G, (ng, N))
        gi, ni = np.nonzero(rng.random((ng, N)) < 0.85)
        W[gi, rows[gi, ni], ni] = np.where(rng.integers(0, 2, gi.size) == 1, -0.0, 0.0)
    Wt = torch.from_numpy(W.reshape(K, N)).to(dtype)
    _, _, z = _assert_quant_equal(Wt, G, f"mixed zeros K={K} N={N} G={G}")
    if ng * N >= 16:
        zb = np_(z).view(np.uint16)
        assert (zb == 0x8000).any() and (zb == 0x0000).any()   # both zero signs occur


@pytest.mark.parametrize("N", [260, 261])
@pytest.mark.parametrize("G", [8, 16, 24, 32, 40, 64, 72, 96, 128, 136, 256, 264, 520])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_quantize_ties_and_scales_every_group_split(G, dtype, N):
    """Every split of a group over waves and registers (one, two or four waves a
    group, one to eight packed rows a wave, long groups read twice), an odd
    number of groups and a partial column block (N % 4 == 0 and not), on columns
    whose quotients lie on or one ulp beside a rounding tie, whose scales are
    powers of two, or whose scales lie outside the range of the
    corrected-reciprocal quotient (fp32)."""
    log(f"quantize ties G={G} N={N} {dtype}")
    K = 5 * G
    rng = np.random.default_rng(G * 2 + N % 4)
    t = rng.integers(0, 16, (K, N)) + rng.choice([0.0, 0.5], (K, N))
    s = np.exp2(rng.integers(-6, 1, N)) * rng.choice([1.0, 1.0, 1.1, 1.37], N)
    W = ((np.minimum(t, 15.0) - rng.integers(0, 16, N)) * s).astype(np.float32)
    W[::G], W[1::G] = W.min(axis=0), W.min(axis=0) + 15 * s.astype(np.float32)
    if dtype == torch.float32:
        step = rng.integers(-1, 2, W.shape)
        beside = np.nextafter(W, np.where(step > 0, np.inf, -np.inf), dtype=np.float32)
        W = np.where(step == 0, W, beside)
        W[:, 64:68] *= np.float32(2.0 ** -110)
        W[:, 128:132] *= np.float32(2.0 ** 118)
        W[:, 200:204] += np.float32(1000.0)
    _assert_quant_equal(torch.from_numpy(W).to(dtype), G, f"ties G={G} N={N}")


@pytest.mark.parametrize("N", [8, 9])
@pytest.mark.parametrize("G,groups", [(16, 1023), (16, 1027), (24, 1027), (32, 1023), (32, 1027),
                                      (40, 511), (40, 515), (64, 511), (64, 515),
                                      (16, 255), (24, 257), (48, 513), (32, 4095), (32, 4097)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_quantize_many_groups(G, groups, dtype, N):
    """Just under and over the numbers of groups from which a short one is one or two
    waves' instead of four (four groups or two a workgroup, the last one partial),
    columns together and apart, with zero minima of both signs."""
    log(f"quantize many groups G={G} groups={groups} N={N} {dtype}")
    rng = np.random.default_rng(G * groups + N)
    W = (rng.integers(-8, 9, (G * groups, N)) * 0.25).astype(np.float32)
    W[:, ::3] = np.abs(W[:, ::3])
    W = np.where(W == 0, np.where(rng.random(W.shape) < 0.5, -0.0, 0.0), W)
    W[::7] += rng.standard_normal(W[::7].shape) * 0.01
    _assert_quant_equal(torch.from_numpy(W.astype(np.float32)).to(dtype), G,
                        f"many groups G={G} groups={groups} N={N}")


@pytest.mark.parametrize("G", [32, 64, 96, 128, 256, 512])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
def test_quantize_transposed_weight(G, dtype):
    """A W whose columns are contiguous (an nn.Linear weight's transpose) is read
    in place: partial 512-k chunks and column tiles, rows longer than K, ties,
    scales outside the corrected-reciprocal range, zero minima of either sign,
    and the layouts that are copied first (G = 96, rows off 16 bytes, N = 1)."""
    log(f"quantize transposed G={G} {dtype}")
    rng = np.random.default_rng(G)
    for K, N, pad, off in ((3 * G, 2, 0, 0), (5 * G, 67, 8, 0), (7 * G, 130, 0, 0), (2 * G, 64, 0, 1),
                           (2 * G, 33, 4, 0), (2 * G, 1, 8, 0)):
        W = rng.integers(-16, 17, (N, K + pad)).astype(np.float32) * 0.5
        W *= np.exp2(rng.integers(-4, 1, (N, 1)))
        W[::3] = np.abs(W[::3])
        W[::3] = np.where(W[::3] == 0, np.where(rng.random(W[::3].shape) < 0.5, -0.0, 0.0), W[::3])
        W[1::5] += rng.standard_normal(W[1::5].shape) * 0.01
        if dtype == torch.float32:
            W[2::7] *= np.float32(2.0 ** -110)
        flat = torch.zeros(N * (K + pad) + off, dtype=dtype, device=DEV)
        flat[off:] = torch.from_numpy(W).to(dtype).to(DEV).reshape(-1)
        view = flat[off:].view(N, K + pad)[:, :K].t()
        _assert_quant_equal(view.float() if dtype == torch.bfloat16 else view, G, f"transposed {K}x{N}")


def test_quantize_fp32_tiny_and_denormal_ranges():
    log("quantize fp32 tiny ranges")
    K, N, G = 64, 8, 32
    g = torch.Generator().manual_seed(9)
    W = torch.randn(K, N, generator=g) * 1e-30
    W[:, 3] = torch.randn(K, generator=g) * 1e-39    # fp32 subnormals
    W[:, 4] = torch.randn(K, generator=g) * 1e30
    _assert_quant_equal(W, G, "fp32 tiny/huge")


def test_quantize_non_finite_raises():
    from w4a16 import quantize_weight

    for bad in (float("inf"), float("-inf"), float("nan")):
        log(f"quantize non-finite {bad}")
        W = torch.zeros(64, 8, dtype=torch.float16, device=DEV)
        W[5, 3] = bad
        with pytest.raises(AssertionError):
            quantize_weight(W, 32)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("N", [8, 261])
@pytest.mark.parametrize("G", [8, 32, 64, 128, 256, 520])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_quantize_one_non_finite_weight(dtype, G, N, transposed):
    """One infinity or NaN anywhere raises: one, two and four waves a group, groups
    read twice, columns together and apart, and a transposed weight read in place
    (G = 32 .. 256) in a partial 512-k chunk and column tile.  The weight before it,
    and the one after, quantise."""
    from w4a16 import quantize_weight

    K = 5 * G
    log(f"quantize one non-finite G={G} N={N} {dtype} transposed={transposed}")
    g = torch.Generator().manual_seed(G + N)
    W = (torch.randn((N, K) if transposed else (K, N), generator=g) * 0.02).to(dtype).to(DEV)
    W = W.t() if transposed else W
    quantize_weight(W, G)
    spots = [(0, 0), (0, N - 1), (K - 1, 0), (K - 1, N - 1), (K - G, N // 2), (K - G // 2, N - 1),
             (2 * G - 1, 1), (G // 2 + 1, 4)]
    for i, (k, n) in enumerate(spots):
        bad = (float("inf"), float("-inf"), float("nan"))[(i + G + N) % 3]
        keep = W[k, n].clone()
        W[k, n] = bad
        with pytest.raises(AssertionError):
            quantize_weight(W, G)
        W[k, n] = keep
    _assert_quant_equal(W, G, f"finite again G={G} N={N}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_from_linear_non_finite_weight(dtype, bad):
    """from_linear raises what quantize_weight raises, and the next layer is made."""
    from w4a16 import W4A16Linear

    log(f"from_linear non-finite {bad} {dtype}")
    lin = torch.nn.Linear(640, 67, device=DEV, dtype=dtype)
    with torch.no_grad():
        keep = lin.weight[66, 639].clone()
        lin.weight[66, 639] = bad
        with pytest.raises(AssertionError, match="non-finite"):
            W4A16Linear.from_linear(lin, 128)
        lin.weight[66, 639] = keep
    layer = W4A16Linear.from_linear(lin, 128)
    ref = O.quantize_weight(np_(lin.weight.detach().float() if dtype == torch.bfloat16
                                else lin.weight).T.copy(), 128)
    assert np.array_equal(np_(layer.qweight), ref[0])


def test_quantize_cpu_input_returns_cpu():
    """CPU input: computed on the GPU, returned on the CPU, same bits."""
    from w4a16 import quantize_weight

    log("quantize cpu staging")
    W = (torch.randn(256, 64) * 0.1).to(torch.float16)
    qw, s, z = quantize_weight(W, 64)
    assert qw.device.type == "cpu" and s.device.type == "cpu"
    rq, rs, rz = O.quantize_weight(W.numpy(), 64)
    assert np.array_equal(qw.numpy(), rq) and np.array_equal(s.numpy().view(np.uint16), rs.view(np.uint16))


@pytest.mark.parametrize("cfg", ["C4", "C5a", "C5b"])
def test_quantize_full_size_layers(cfg):
    """Full-size weights of the large configs, quantised on the GPU; every group
    of three column slices compared bit-exact with the oracle (quantisation is
    independent per column), plus size-independent checks on all columns."""
    from w4a16 import quantize_weight, dequantize_weight
    from w4a16 import workloads as wl

    if cfg == "C4":
        case = wl.CONFIGS["C4"][0]
        Gs = [case.G]
    else:
        K, N = (8192, 28672) if cfg == "C5a" else (28672, 8192)
        case = [c for c in wl.CONFIGS["C5"] if c.K == K and c.N == N and c.M == 1][0]
        Gs = [32, 64, 128]
    W = wl.make_w(case)
    Wd = W.to(DEV)
    Kdim, N = W.shape
    for G in Gs:
        log(f"quantize full {cfg} K={Kdim} N={N} G={G}")
        qw, s, z = quantize_weight(Wd, G)
        # N and the slice width are multiples of 32, so each column is in a whole
        # 32-column block of both the slice and the full weight (zero-sign rule)
        for a, b in ((0, 256), (N // 2 - 128, N // 2 + 128), (N - 256, N)):
            rq, rs, rz = O.quantize_weight(W[:, a:b].numpy(), G)
            assert np.array_equal(np_(qw[:, a:b]), rq), (cfg, G, a)
            assert np.array_equal(np_(s[:, a:b]).view(np.uint16), rs.view(np.uint16)), (cfg, G, a)
            assert np.array_equal(np_(z[:, a:b]).view(np.uint16), rz.view(np.uint16)), (cfg, G, a)
        # all columns: zero-points are integers in [0, 15]; dequant error below one step
        zf = z.float()
        assert bool(((zf >= 0) & (zf <= 15) & (zf == zf.round())).all())
        dq = dequantize_weight(qw, s, z, G).float()
        step = s.float().repeat_interleave(G, dim=0)
        err = (dq - Wd.float()).abs()
        assert bool((err <= step * 1.01 + 1e-6).all())
        del qw, s, z, dq, step, err


# --------------------------------------------------------------------------- #
# pack / unpack / dequant                                                      #
# --------------------------------------------------------------------------- #
@pytest.mark.parametrize("K", [8, 64, 128, 4096])
@pytest.mark.parametrize("N", [1, 16, 4096])
def test_pack_unpack_roundtrip(K, N):
    """Reference test_quant.py:21-31 on the device, words compared with the oracle."""
    from w4a16 import pack_int4, unpack_int4

    log(f"pack/unpack K={K} N={N}")
    x = torch.randint(0, 16, (K, N), dtype=torch.int32, device=DEV)
    packed = pack_int4(x)
    assert packed.shape == (K // 8, N) and packed.dtype == torch.int32
    assert np.array_equal(np_(packed), O.pack_int4(np_(x)))
    restored = unpack_int4(packed, K)
    assert restored.shape == (K, N)
    assert torch.equal(restored, x)


def test_pack_extremes_and_position():
    from w4a16 import pack_int4, unpack_int4

    for val in (0, 15):
        x = torch.full((16, 8), val, dtype=torch.int32, device=DEV)
        assert torch.equal(unpack_int4(pack_int4(x)), x)
    x = torch.zeros((8, 1), dtype=torch.int32, device=DEV)
    x[3, 0] = 0xA
    assert int(pack_int4(x)[0, 0]) == (0xA << 12)


@pytest.mark.parametrize("bad", [16, -1, 1 << 20])
def test_pack_range_assertion(bad):
    from w4a16 import pack_int4

    x = torch.zeros((16, 4), dtype=torch.int32, device=DEV)
    x[9, 2] = bad
    with pytest.raises(AssertionError):
        pack_int4(x)


@pytest.mark.parametrize("K,N,G", [(128, 256, 64), (4096, 512, 128), (64, 33, 32), (24, 12, 12)])
def test_dequant_bit_exact(K, N, G):
    from w4a16 import dequantize_weight

    log(f"dequant K={K} N={N} G={G}")
    g = torch.Generator().manual_seed(K + N + G)
    q = torch.randint(0, 16, (K, N), generator=g, dtype=torch.int32)
    qw = torch.from_numpy(O.pack_int4(q.numpy()))
    s = (torch.rand(K // G, N, generator=g) * 0.1).to(torch.float16)
    z = torch.randint(0, 16, (K // G, N), generator=g).to(torch.float16)
    z[0, 0] = -0.0
    z[-1, -1] = 3.5      # non-integer zero-point: fp16 subtraction semantics
    out = dequantize_weight(qw.to(DEV), s.to(DEV), z.to(DEV), G)
    ref = O.dequantize_weight(qw.numpy(), s.numpy(), z.numpy(), G)
    assert np.array_equal(np_(out).view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("N,off", [(8, 0), (2056, 0), (4, 0), (1028, 0), (2048, 4), (2048, 2), (1027, 0),
                                   (124, 0), (128, 0), (132, 0), (64, 0), (120, 0), (64, 2)])
@pytest.mark.parametrize("G", [8, 40, 128])
def test_dequant_columns_per_lane(N, off, G):
    """8, 4 or 1 columns a lane by N and the alignment of scales and zeros (off =
    their offset in elements), partial column blocks, and zero-points and scales
    of every magnitude, infinities and NaN included, to the oracle's bits."""
    from w4a16 import dequantize_weight

    log(f"dequant columns N={N} off={off} G={G}")
    K = 3 * G
    rng = np.random.default_rng(N + off + G)
    qw = torch.from_numpy(rng.integers(-2**31, 2**31, (K // 8, N)).astype(np.int32))
    buf = torch.from_numpy(rng.integers(0, 2**16, 2 * 3 * N + 2 * off).astype(np.uint16).view(np.float16))
    s, z = buf[off:off + 3 * N].view(3, N), buf[2 * off + 3 * N:].view(3, N)
    dev = buf.to(DEV)
    out = dequantize_weight(qw.to(DEV), dev[off:off + 3 * N].view(3, N),
                            dev[2 * off + 3 * N:].view(3, N), G)
    with np.errstate(all="ignore"):
        ref = O.dequantize_weight(qw.numpy(), s.numpy(), z.numpy(), G)
    got, nan = np_(out), np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint16)[~nan], ref.view(np.uint16)[~nan])


def test_quant_dequant_roundtrip_error():
    """Reference test_quant.py:71-90 on the device: mean relative error < 0.15."""
    from w4a16 import dequantize_weight, quantize_weight

    for G in (64, 128):
        torch.manual_seed(1)
        W = torch.randn(4096, 1024, dtype=torch.float16, device=DEV)
        qw, s, z = quantize_weight(W, G)
        dq = dequantize_weight(qw, s, z, G)
        rel = ((dq.float() - W.float()).abs().mean() / W.float().abs().mean()).item()
        assert rel < 0.15
