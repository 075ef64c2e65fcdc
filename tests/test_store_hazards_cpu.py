"""Disassembly check of the built library: a vector store of more than 8 bytes
still reads its data registers for two wait states after it has been issued, so
no vector instruction may write them before.  The compiler keeps that distance
for most forms of the store, but not for buffer stores whose offset lies in a
scalar register."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "public_amd", "libcruna_hip.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 2


def _code_objects(path):
    """The gfx950 code objects of a HIP library's bundles."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idl = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + idl].decode()
            p += 24 + idl
            if "gfx950" in triple and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def _registers(operand):
    out = set()
    for lo, hi, one in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", operand):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def _early_overwrites(lines):
    """(kernel, store, instruction that overwrites its data too early) in a disassembly."""
    kernel, waiting = "", []  # stores: [data registers, wait states passed, text]
    for line in lines:
        if line.endswith(">:"):
            kernel, waiting = line.split("<")[-1][:-2], []
            continue
        text = line.split("//")[0].strip()
        if not text:
            continue
        op, _, rest = text.partition(" ")
        if op.startswith("v_"):
            written = _registers(rest.split(",")[0])
            for data, _, store in waiting:
                if data & written:
                    yield kernel, store, text
        passed = int(rest.strip(), 0) + 1 if op == "s_nop" else 1
        waiting = [[d, w + passed, s] for d, w, s in waiting if w + passed < WAIT_STATES]
        m = re.match(r"(buffer|global|flat|scratch)_store_dwordx[34]$", op)
        if m:
            ops = rest.split(",")
            waiting.append([_registers(ops[0] if m.group(1) == "buffer" else ops[1]), 0, text])


def test_the_check_sees_an_early_overwrite():
    store = "\tbuffer_store_dwordx4 v[80:83], v128, s[48:51], s73 offen"
    mul = "\tv_mul_f64 v[80:81], v[24:25], v[60:61]"
    assert len(list(_early_overwrites(["0 <k>:", store, mul]))) == 1
    assert len(list(_early_overwrites(["0 <k>:", store, "\ts_nop 0", mul]))) == 1
    assert not list(_early_overwrites(["0 <k>:", store, "\ts_nop 1", mul]))
    assert not list(_early_overwrites(["0 <k>:", store, "\tv_mul_f64 v[84:85], v[80:81], v[60:61]"]))


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(OBJDUMP), reason="no built library or no llvm-objdump")
def test_store_data_is_left_alone(tmp_path):
    objects = list(_code_objects(LIB))
    assert objects
    kernels = 0
    for i, code in enumerate(objects):
        elf = tmp_path / f"{i}.co"
        elf.write_bytes(code)
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(elf)], capture_output=True, text=True, check=True)
        lines = out.stdout.splitlines()
        kernels += sum(line.endswith(">:") for line in lines)
        bad = list(_early_overwrites(lines))
        assert not bad, bad[:5]
    assert kernels > 300
