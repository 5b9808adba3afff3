"""GPU: the kernels an automatic call really launches, by the profiler's names."""
from __future__ import annotations

import re

import pytest
import torch

from _helpers import DEV, assert_gemm_close, log, np_
from oracle import w4a16_oracle as O

pytestmark = pytest.mark.gpu

# tile_cfg -> (m-tiles a wave, waves along N, k-slices)
TILINGS = {16: (16, 4, 1), 17: (8, 4, 1), 18: (8, 2, 2), 19: (4, 2, 2), 20: (4, 1, 4), 21: (2, 1, 4)}


def launched(fn):
    """[(kernel, template arguments)] of the kernels fn() launches."""
    from torch.profiler import ProfilerActivity, profile

    fn()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    out = []
    if not any("w4a16" in e.name for e in prof.events()):
        pytest.skip("the profiler records no kernels here")
    for e in prof.events():
        m = re.search(r"w4a16\d+_GLOBAL__N_1(\d+)(\w+)", e.name)
        if m:
            name, rest = m.group(2)[:int(m.group(1))], m.group(2)[int(m.group(1)):]
            args = re.match(r"I((?:L[a-z]\w*?E)+)E", rest)
            out.append((name, tuple(int(v) for v in re.findall(r"L[a-z](\d+)E", args.group(1)))
                        if args else ()))
        # a name with no _Float16 in its signature comes demangled
        m = re.match(r"void w4a16::\(anonymous namespace\)::(\w+)<(.+?)>\(", e.name)
        if m:
            vals = (v.strip() for v in m.group(2).split(","))
            out.append((m.group(1), tuple(int({"true": 1, "false": 0}.get(v, v)) for v in vals
                                          if re.fullmatch(r"\d+|true|false", v))))
    return out


def operands(M, K, N, G, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    qw = torch.randint(-2**31, 2**31 - 1, (K // 8, N), generator=g, device=DEV, dtype=torch.int32)
    s = (torch.rand(K // G, N, generator=g, device=DEV) * 0.02 + 0.001).half()
    z = torch.randint(0, 16, (K // G, N), generator=g, device=DEV).half()
    return x, qw, s, z


def test_profiler_names_kernels():
    """What the other tests read: a forced SIMT plan shows as one simt kernel."""
    from w4a16.hip_kernel import plan_for, w4a16_matmul_planned

    x, qw, s, z = operands(4, 256, 64, 64)
    names = launched(lambda: w4a16_matmul_planned(x, qw, s, z, 64, plan_for(4, 64, 256, 64, "simt")))
    assert len(names) == 1 and "simt" in names[0][0], names


@pytest.mark.parametrize("M,K,N,G", [
    (1100, 256, 14340, 128), (300, 512, 14336, 128), (600, 320, 4100, 64), (256, 14336, 4096, 128),
    (300, 1056, 4100, 96), (129, 4096, 260, 64), (17, 14336, 4096, 128), (32, 4096, 14336, 64),
    (33, 8704, 24576, 32), (420, 14336, 8224, 32), (256, 128, 5120, 32),
])
def test_runs_what_auto_plan_says(M, K, N, G):
    from w4a16 import _lib, w4a16_matmul
    from w4a16.hip_kernel import plan_for, w4a16_matmul_planned

    p = _lib.auto_plan(M, N, K, G)
    log(f"dispatch M={M} K={K} N={N} G={G} kernel={p.kernel} cfg={p.tile_cfg} split={p.split_k}")
    x, qw, s, z = operands(M, K, N, G)
    names = launched(lambda: w4a16_matmul(x, qw, s, z, G))
    if p.tile_cfg in TILINGS:
        mt, wn, ks = TILINGS[p.tile_cfg]
        kernel, args = names[0]
        assert kernel == "wide_kernel" and (args[0], args[2], args[3]) == (mt, wn, ks), names
        assert bool(args[6]) == (N % 4 != 0)
        assert [k for k, _ in names[1:]] == (["splitk_reduce"] if p.split_k > 1 else
                                             ["wide_kernel"] * (len(names) - 1)), names
    else:
        plan = plan_for(M, N, K, G)
        assert names == launched(lambda: w4a16_matmul_planned(x, qw, s, z, G, plan)), names
        assert not [k for k, _ in names if k == "wide_kernel"]


@pytest.mark.parametrize("M,N,off,kernel", [
    (20, 516, 1, "skinny"), (64, 516, 1, "skinny"), (65, 516, 1, "wide_kernel"),
    (300, 516, 1, "wide_kernel"), (93, 1003, 0, "wide_kernel"), (129, 1, 0, "wide_kernel"),
    (7, 1003, 0, "skinny")])
def test_odd_widths_and_alignment(M, N, off, kernel):
    """Scales and zeros one element into their storage, or N % 4 != 0: never SIMT."""
    from w4a16 import w4a16_matmul

    K, G = 2080, 32
    x, qw, s, z = operands(M, K, N, G)
    ref = O.reference_w4a16(np_(x), np_(qw), np_(s), np_(z), G)
    if off:
        s, z = (torch.empty(t.numel() + off, dtype=t.dtype, device=DEV)[off:]
                .copy_(t.reshape(-1)).view(t.shape) for t in (s, z))
    log(f"dispatch odd M={M} N={N} off={off}")
    names = launched(lambda: w4a16_matmul(x, qw, s, z, G))
    assert kernel in names[0][0], names
    assert kernel != "wide_kernel" or names[0][1][6] == 1, names
    assert_gemm_close(w4a16_matmul(x, qw, s, z, G), ref, f"M={M} N={N} off={off}")


@pytest.mark.parametrize("M,K,N,G", [(24, 4096, 28672, 128), (32, 4096, 28672, 64), (100, 1024, 4096, 128)])
def test_scales_and_zeros_far_apart(M, K, N, G):
    """Scales and zeros 2 GiB and more apart: the streamed tiles' buffer resource does
    not reach both, so the call takes the wide kernel, with the same result."""
    from w4a16 import w4a16_matmul
    from w4a16.hip_kernel import plan_for

    p = plan_for(M, N, K, G)
    assert p.kernel == 2 and p.tile_cfg >= 11
    x, qw, s, z = operands(M, K, N, G)
    big = torch.empty((1 << 31) + 4 * s.numel(), dtype=torch.uint8, device=DEV)
    sf = big[:2 * s.numel()].view(torch.float16).view(s.shape).copy_(s)
    zf = big[big.numel() - 2 * z.numel():].view(torch.float16).view(z.shape).copy_(z)
    log(f"dispatch far M={M} K={K} N={N} G={G}")
    names = launched(lambda: w4a16_matmul(x, qw, sf, zf, G))
    assert names[0][0] == "wide_kernel", names
    near, far = w4a16_matmul(x, qw, s, z, G), w4a16_matmul(x, qw, sf, zf, G)
    cols = torch.arange(0, N, 97)
    ref = O.reference_w4a16(np_(x), np_(qw[:, cols]), np_(s[:, cols]), np_(z[:, cols]), G)
    assert_gemm_close(far[:, cols], ref, "far apart")
    assert_gemm_close(near[:, cols], ref, "near")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("G,groups,N,waves", [
    # octets that fill four waves (4, 7, 8)
    (32, 1023, 8, 4), (32, 1024, 8, 1), (56, 511, 8, 4), (56, 512, 8, 2), (64, 511, 8, 4), (64, 512, 8, 2),
    (32, 4095, 9, 4), (32, 4096, 9, 1), (56, 700, 2045, 4), (64, 600, 2045, 4),
    # and that leave one without (2, 3, 5, 6)
    (16, 256, 8, 4), (16, 257, 8, 1), (24, 256, 8, 4), (24, 257, 8, 1), (40, 256, 8, 4), (40, 257, 8, 2),
    (48, 102, 1024, 2), (16, 512, 9, 4), (24, 513, 9, 1), (40, 512, 9, 4), (40, 102, 2045, 2),
    (48, 513, 9, 2),
    # and the lengths with one split at every size
    (8, 2, 9, 1), (72, 2, 9, 4), (128, 2, 8, 4),
])
def test_quantise_waves_per_group(G, groups, N, waves, dtype):
    """Four waves share a short group only where they are all at work or the groups few."""
    from w4a16 import quantize_weight

    log(f"dispatch quantise G={G} groups={groups} N={N} {dtype}")
    W = torch.randn(G * groups, N, device=DEV).to(dtype)
    names = [n for n in launched(lambda: quantize_weight(W, G)) if n[0] == "quantize_tile_kernel"]
    assert len(names) == 1 and names[0][1][1:] == (waves, int(N % 4 == 0)), names


@pytest.mark.parametrize("N,G,columns", [(4, 96, 4), (8, 32, 4), (108, 128, 4), (120, 32, 4), (128, 32, 8),
                                         (132, 32, 4), (63, 32, 1), (64, 4, 1)])
def test_dequantise_columns_per_lane(N, G, columns):
    """Several columns a lane wherever rows allow them, eight from 128 columns."""
    from w4a16 import dequantize_weight

    log(f"dispatch dequantise N={N} G={G}")
    _, qw, s, z = operands(1, 384, N, G)
    names = launched(lambda: dequantize_weight(qw, s, z, G))
    assert names == [("dequant_vec_kernel", (columns,)) if columns > 1 else ("dequant_kernel", ())], names
