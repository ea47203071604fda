"""A VALU write to a data VGPR in the instruction after a 16-byte buffer store
with a scalar offset corrupted the stored first dword on some runs.  The
library's own code objects are disassembled and searched for that pair."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from foundry_attn import _abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def code_objects(path):
    """The gfx950 images of the offload bundles inside a library (magic, entry
    count, then offset, size, triple length and triple of each entry)."""
    blob, magic = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        pos = at + len(magic)
        (count,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(magic, at + 1)


def vgprs(operand):
    m = re.fullmatch(r"v(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    lo, hi = (int(m[1]), int(m[1])) if m[1] else (int(m[2]), int(m[3]))
    return set(range(lo, hi + 1))


def hazards(asm):
    """(kernel, store, next instruction) of every such pair in a listing, and
    the number of stores looked at."""
    found, kernel, store, seen = [], "", None, 0
    for line in asm.splitlines():
        m = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if m:
            kernel, store = m[1], None
            continue
        ins = line.split("//")[0].split("#")[0].strip()
        if not re.match(r"[a-z]\w+(\s|$)", ins):
            continue
        ops = [o.strip() for o in ins.split(None, 1)[1].split(",")] if " " in ins else []
        if store and ins.startswith("v_"):
            written = vgprs(ops[0]) | (vgprs(ops[1]) if "swap" in ins else set())
            if written & vgprs(store[1]):
                found.append((kernel, store[0], ins))
        store = None
        if ins.startswith(("buffer_store_dwordx4", "buffer_store_dwordx3")):
            seen += 1
            if re.match(r"(s\d+|m0|vcc|ttmp)", ops[3]):
                store = (ins, ops[0])
    return found, seen


def test_scan_finds_the_pair():
    pair = ("0000000000000100 <k>:\n"
            "\tbuffer_store_dwordx4 v[4:7], v1, s[52:55], s9 offen nt // 0: 0\n\tv_fma_f32 v4, s0, v2, 0\n"
            "\tbuffer_store_dwordx4 v[4:7], v1, s[52:55], 0 offen\n\tv_mov_b32_e32 v4, 0\n"
            "\tbuffer_store_dwordx4 v[4:7], v1, s[52:55], s9 offen\n\ts_nop 1\n\tv_mov_b32_e32 v4, 0\n"
            "\tbuffer_store_dwordx4 v[4:7], v1, s[52:55], s9 offen\n\tv_mov_b32_e32 v8, 0\n")
    found, seen = hazards(pair)
    assert seen == 4 and [f[2] for f in found] == ["v_fma_f32 v4, s0, v2, 0"]


@pytest.mark.skipif(not shutil.which(OBJDUMP), reason="no llvm-objdump")
def test_no_store_is_followed_by_a_write_of_its_data(tmp_path):
    stores = 0
    for i, image in enumerate(code_objects(_abi.LIB_PATH)):
        path = tmp_path / f"{i}.o"
        path.write_bytes(image)
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True,
                             text=True).stdout
        found, seen = hazards(asm)
        assert not found, found
        stores += seen
    assert stores > 0


def test_one_helper_holds_every_16_byte_buffer_store():
    csrc = os.path.join(ROOT, "foundry-trainer_amd", "csrc")
    uses = [(name, line) for name in os.listdir(csrc) for line in open(os.path.join(csrc, name), encoding="utf-8")
            if re.search(r"raw_(ptr_)?buffer_store_b(96|128)", line)]
    assert [name for name, _ in uses] == ["fa_lds.hpp"], uses
