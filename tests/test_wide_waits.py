"""CPU: the counted waits of the one-wave-per-SIMD kernel (csrc/gemm_wide.h) in the
library as built.

A wait names how many of the newest loads may still be in flight, so what it waits
for depends on the loads issued behind it: here each kernel's machine code is
followed through its prologue and three trips of its loop, and every wait must cover
the activations that the step after it reads.
"""
from __future__ import annotations

import os
import re
import shutil
import struct
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects in a library's offload bundles."""
    with open(path, "rb") as f:
        data = f.read()
    for m in re.finditer(re.escape(MAGIC), data):
        at = m.start()
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        if count > 16:
            continue
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + n].decode()
            p += 24 + n
            if "gfx950" in triple and size:
                yield data[at + off:at + off + size]


def _kernels(tmp_path):
    """{template arguments: [(address, instruction), ...]} of every wide_kernel."""
    from w4a16 import _lib

    out = {}
    for i, obj in enumerate(_code_objects(_lib.LIB_PATH)):
        if b"wide_kernel" not in obj:
            continue
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True,
                              check=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(\S*wide_kernel\S*)>:\n(.*?)(?=^\S|\Z)", text,
                                     re.M | re.S):
            args = re.search(r"wide_kernelI((?:L[ib]\d+E)+)E", name)
            key = tuple(int(v) for v in re.findall(r"L[ib](\d+)E", args.group(1)))
            code = [(int(a, 16), ins.strip()) for ins, a in
                    re.findall(r"^\s+(\S.*?)\s*// ([0-9A-F]{12}):", body, re.M)]
            out[key] = code
    return out


def _loop(code):
    """(first, last) instruction of the loop over the panels: the backward branch
    that spans the most LDS-direct loads."""
    at = {a: i for i, (a, _) in enumerate(code)}
    best, span = 0, None
    for i, (a, ins) in enumerate(code):
        m = re.match(r"s_cbranch_\w+ (\d+)", ins)
        if not m or int(m.group(1)) < 32768:
            continue
        to = at[a + 4 + 4 * (int(m.group(1)) - 65536)]
        n = sum(" lds" in x for _, x in code[to:i])
        if n > best:
            best, span = n, (to, i)
    return span


def _loads_per_panel(key):
    mt, _, wn, _, sz1, _, any_ = key
    halves = 1 if sz1 else 2
    return 16 * mt // wn // 8, 2 + 2 * halves * (4 if any_ else 1)


def _deep(key):
    """Three panels of activations ahead: tiles of at most 64 rows in vector form."""
    return key[0] <= 4 and not key[6]


def _check(key, code):
    """Raises AssertionError where a counted wait covers too little."""
    acts, weights = _loads_per_panel(key)
    deep = _deep(key)
    first, last = _loop(code)
    prologue = [x for _, x in code[:first]]
    body = [x for _, x in code[first:last + 1]]
    barrier = prologue.index("s_barrier")
    entry = max(i for i in range(barrier) if "vmcnt" in prologue[i])
    # a step's four sub-steps each begin with this; its counted wait is in the last
    subs = [i for i, x in enumerate(body) if x == "s_nop 1"]
    assert len(subs) == 16, f"wide_kernel<{key}>: {len(subs)} sub-steps in a trip"
    counted = {i + 1 for i in subs[3::4]}
    assert all("vmcnt" in body[i] for i in counted), f"wide_kernel<{key}>: a wait is missing"
    issued, lds, wait = 0, [], 0
    for j, ins in enumerate(prologue + 3 * body):
        if re.match(r"(buffer|global|scratch|flat)_(load|store|atomic)", ins):
            issued += 1
            if " lds" in ins:
                lds.append(issued)
        m = re.search(r"vmcnt\((\d+)\)", ins)
        if not m:
            continue
        if j != entry and (j < len(prologue) or (j - len(prologue)) % len(body) not in counted):
            continue   # one of the compiler's, for a register it is about to read
        if j == entry:
            # the loads written ahead of the first wait are issued ahead of it
            # (two panels ahead no wait counts weights, and they may move)
            assert len(lds) == (3 if deep else 2) * acts
            assert not deep or issued - len(lds) == 4 * weights
        need = lds[(wait + 1) * acts - 1]      # the last of the panel the next step reads
        assert issued - need >= int(m.group(1)), (
            f"wide_kernel<{key}>: wait {wait} leaves {m.group(1)} in flight, but only "
            f"{issued - need} were issued behind panel {wait}'s activations")
        wait += 1
    assert wait == 13


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_counted_waits_cover_their_panels(tmp_path):
    kernels = _kernels(tmp_path)
    assert len(kernels) >= 30
    # no automatic call takes the 32-row tiles with operands off the vector alignment
    assert not [k for k in kernels if k[0] == 2 and k[6]]
    for key, code in kernels.items():
        _check(key, code)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_a_load_behind_its_wait_is_seen(tmp_path):
    """The check itself: a weight load of the prologue or of a step, moved past the
    wait that counts it in a copy of the listing, is reported."""
    for key, code in _kernels(tmp_path).items():
        first, last = _loop(code)
        weights = [i for i, (_, x) in enumerate(code) if "buffer_load" in x and " lds" not in x]
        wait = [i + 1 for i in range(first, last) if code[i][1] == "s_nop 1"][3]
        plants = []
        if _deep(key):   # (the others wait for activations behind activations)
            plants += [(max(i for i in weights if i < first), first),
                       (min(i for i in weights if i > first), wait + 1)]
        for load, to in plants:
            moved = code[:load] + code[load + 1:to] + [(-1, code[load][1])] + code[to:]
            with pytest.raises(AssertionError):
                _check(key, moved)
