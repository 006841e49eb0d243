"""The built library's transfers from global memory into LDS (buffer_load ... lds, written as inline asm, where
the compiler adds no wait states itself) keep the distances that gfx950 asks for: one wait state after
a scalar write of M0, five after a vector instruction wrote a scalar register that the transfer reads."""
import os
import re
import struct
import subprocess

import pytest

from qwen3_5_native import hip

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of a library (clang's offload bundles: count, then offset, size and target each)."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + n]:
                yield data[at + off:at + off + size]
            p += 24 + n
        at = data.find(MAGIC, at + len(MAGIC))


def scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    return {operand} if re.fullmatch(r"s\d+|m0|vcc|vcc_lo|vcc_hi", operand) else set()


def short_waits(lines):
    """(transfers, those too close to a write of M0 or of their scalar operands) of a listing."""
    before, count, bad = [], 0, []
    for line in lines:
        if re.match(r"[0-9a-f]+ <", line):
            before = []
            continue
        text = line.split("//")[0].strip()
        if not text:
            continue
        op, _, rest = text.partition(" ")
        args = [a.strip().split()[0] for a in rest.split(",") if a.strip()]
        if op.startswith("buffer_load") and text.endswith(" lds"):
            count += 1
            reads, states = set().union(*map(scalars, args)), 0
            for o, a, t in reversed(before[-8:]):
                writes = scalars(a[0]) if a else set()
                if (o.startswith("s_") and "m0" in writes and states < 1) or (o.startswith("v_") and writes & reads and states < 5):
                    bad.append((t, text))
                states += int(a[0], 0) + 1 if o == "s_nop" else 1
        before.append((op, args, text))
    return count, bad


def test_the_scan_sees_short_waits():
    near = ["s_mov_b32 m0, s4", "buffer_load_dwordx4 v1, s[8:11], s5 offen lds"]
    assert short_waits(near) == (1, [tuple(near)])
    vec = ["v_readfirstlane_b32 s9, v0", "s_mov_b32 m0, s4", "s_nop 2", "buffer_load_dwordx4 v1, s[8:11], s5 offen lds"]
    assert short_waits(vec) == (1, [(vec[0], vec[3])])
    assert short_waits([vec[0], vec[1], "s_nop 3", vec[3]]) == (1, [])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_transfers_into_lds_wait_long_enough(tmp_path):
    hip.load()
    total = 0
    for i, code in enumerate(code_objects(hip.default_library())):
        f = tmp_path / f"{i}.co"
        f.write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True).stdout
        count, bad = short_waits(text.splitlines())
        total += count
        assert not bad, (len(bad), bad[:4])
    assert total > 500  # the GEMM, attention and GDN kernels' transfers
