"""CPU: which kernel an automatic call takes, as the queries of the C ABI tell it (they
and the call share one function)."""
from __future__ import annotations

import random

import pytest

from w4a16 import _lib

WIDE = range(16, 22)   # tile_cfg numbers of the one-wave-per-SIMD kernel


def _same_launch(a, p):
    return all(getattr(a, f) == getattr(p, f) for f, _ in a._fields_)


@pytest.mark.parametrize("M,N,K,G,wide", [
    # large weights, few rows: the streamed tiles, two workgroups a CU
    (57, 16896, 26624, 32, False), (33, 17408, 15616, 64, False), (64, 28672, 28672, 128, False),
    (64, 18880, 18176, 32, False), (420, 8224, 14336, 32, False), (4096, 2104, 14336, 32, False),
    # at most three panels of k: the register-staged tiles
    (256, 2048, 32, 32, False), (256, 5120, 128, 32, False), (3305, 11008, 128, 32, False),
    (70, 4096, 192, 64, False), (1850, 8192, 32, 32, False),
    # the wide kernel beside them
    (64, 14336, 4096, 128, True), (64, 26560, 16384, 128, True), (33, 4096, 14336, 128, True),
    (128, 4096, 4096, 64, True), (256, 11008, 4096, 64, True), (512, 14336, 4096, 128, True),
    (1024, 4096, 4096, 32, True), (4096, 14336, 4096, 128, True), (300, 4096, 224, 32, True),
    (1024, 11008, 160, 32, True), (788, 8192, 128, 128, True),
    (32, 4096, 14336, 128, True), (93, 1003, 2080, 32, True),
])
def test_the_faster_kernel(M, N, K, G, wide):
    a, p = _lib.auto_plan(M, N, K, G), _lib.plan(M, N, K, G)
    assert (a.kernel == _lib.KERNEL_MFMA and a.tile_cfg in WIDE) == wide
    assert wide or _same_launch(a, p)


def test_queries_agree():
    """The wide kernel's partials and a plan's both fit the workspace asked for, its
    grid covers the result, and a call it does not take runs the plan as it is."""
    rng = random.Random(7)
    lib = _lib.load()
    seen = set()
    for _ in range(3000):
        M = int(2 ** rng.uniform(0, 12.5))
        G = rng.choice((32, 64, 96, 128, 256))
        K = G * max(1, int(2 ** rng.uniform(5, 15)) // G)
        N = max(1, int(2 ** rng.uniform(3, 15)) // rng.choice((1, 4, 64)) * rng.choice((1, 4, 64)))
        case = (M, N, K, G)
        a, p = _lib.auto_plan(*case), _lib.plan(*case)
        ws = lib.w4a16_gemm_workspace_bytes(*case)
        assert max(a.workspace_bytes, p.workspace_bytes) <= ws, case
        if a.kernel == _lib.KERNEL_MFMA and a.tile_cfg in WIDE:
            tiles = -(-N // a.tile_n) * -(-M // a.tile_m)
            assert a.grid_x == tiles * a.split_k, case
            assert a.workspace_bytes == (4 * a.split_k * M * N if a.split_k > 1 else 0), case
            assert a.tile_cfg != 21 or (9 <= M <= 32 and N % 4 == 0), case
            assert a.tile_cfg != 16 or N % 4 == 0, case
            seen.add(a.tile_cfg)
        else:
            assert _same_launch(a, p), case
    assert seen == set(WIDE)
