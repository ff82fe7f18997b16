"""The gfx950 code in the built library: no register spill ahead of the
instruction that restores the exec mask at a merge point. The compiler has
placed spills there (k_stage31, a per-lane flag live across the wall-closure
branch): only the lanes of the branch just left were stored, and the reload
behind the merge gave the others stale values, wrong fluxes next to a solid
block without any error. Wherever registers are short that can come back with
a change of the sources or of the compiler, so the code itself is read."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "uq_amd", "lib", "libuqlbm.so")
OBJDUMP = "/opt/rocm/lib/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def early_spills(lines):
    """(function, line) of every scratch store between a branch target and an
    exec restore, with no other change of the exec mask or branch between."""
    found, func, head = [], "", None  # head: stores since the branch target, None elsewhere
    for line in lines:
        m = re.match(r"^[0-9a-f]* ?<(\w+)>:", line)
        if m:
            if not re.fullmatch(r"L\d+", m.group(1)):
                func, head = m.group(1), None
            else:
                head = []
            continue
        op = line.strip()
        if head is None or not op:
            continue
        if op.startswith("scratch_store"):
            head.append((func, op.split("//")[0].strip()))
        elif re.match(r"s_or_b64 exec, exec|s_or_saveexec", op):
            found += head
            head = None
        elif re.match(r"s_c?branch|s_endpgm|s_setpc|s_\w*saveexec|s_\w+ exec\b", op):
            head = None
    return found


def code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if size and name.endswith(b"gfx950"):
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def test_scan_finds_a_planted_spill():
    bad = ["00 <k_x>:", "\ts_and_saveexec_b64 s[4:5], vcc", "\ts_cbranch_execz L1", "\tv_mov_b32 v1, v2", "",
           "10 <L1>:", "\tscratch_store_dword off, v164, off // 0: 0", "\ts_or_b64 exec, exec, s[4:5]"]
    assert early_spills(bad) == [("k_x", "scratch_store_dword off, v164, off")]
    good = bad[:6] + [bad[7], bad[6]]
    assert early_spills(good) == []
    # between s_or_saveexec and s_xor every lane is on
    assert early_spills(bad[:6] + ["\ts_or_saveexec_b64 s[6:7], s[8:9]", bad[6], "\ts_xor_b64 exec, exec, s[6:7]"]) == []


def test_built_library(tmp_path):
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIB):
        pytest.skip("no disassembler or no built library")
    with open(LIB, "rb") as fh:
        data = fh.read()
    kernels, found = 0, []
    for k, obj in enumerate(code_objects(data)):
        path = tmp_path / f"{k}.co"
        path.write_bytes(obj)
        r = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", "--symbolize-operands", str(path)], capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-500:]
        lines = r.stdout.split("\n")
        kernels += sum(1 for x in lines if re.match(r"^[0-9a-f]+ <_Z\w+>:", x))
        found += early_spills(lines)
    assert kernels > 40  # the flux, strip, fused, pointwise and boundary kernels were read
    assert not found, found
