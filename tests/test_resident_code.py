"""The resident kernel's machine code, as built here: what only an instruction
can guarantee and no result shows.

A solve stores x in the plan's row order; the finalize reads it in row order,
so a wave reads rows that other waves of its workgroup stored.  On every path
between the two there is a workgroup barrier."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import chysx

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LIB = os.path.join(os.path.dirname(chysx.__file__), "libchysx_hip.so")


def _code_objects(path):
    raw = open(path, "rb").read()
    at = 0
    while (at := raw.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        (count,) = struct.unpack_from("<Q", raw, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", raw, p)
            if b"gfx950" in raw[p + 24:p + 24 + length] and size:
                yield raw[at + off:at + off + size]
            p += 24 + length
        at += 24


def _resident_kernels(folder):
    """{kernel: [(opcode, addresses that may come next)]} by address."""
    kernels = {}
    for k, obj in enumerate(_code_objects(LIB)):
        if b"resident_kernel" not in obj:
            continue
        file = folder / f"{k}.co"
        file.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(file)], capture_output=True, text=True, check=True).stdout
        body = None
        for line in text.splitlines():
            head = re.match(r"([0-9a-f]+) <(.*)>:$", line)
            if head:
                start = int(head[1], 16)
                body = kernels.setdefault(head[2], {}) if "resident_kernel" in head[2] else None
                continue
            m = re.match(r"\s+(\w+).*// ([0-9A-F]+): ((?:[0-9A-F]{8} ?)+)(?:<.*\+0x([0-9a-f]+)>|<.*>)?", line)
            if body is None or not m:
                continue
            at, op = int(m[2], 16), m[1]
            follows = [at + 4 * len(m[3].split())]
            if op.startswith("s_cbranch") or op == "s_branch":
                target = start + (int(m[4], 16) if m[4] else 0)
                follows = [target] if op == "s_branch" else follows + [target]
            elif op == "s_endpgm":
                follows = []
            assert op not in ("s_setpc_b64", "s_swappc_b64"), "a call: this walk does not follow it"
            body[at] = (op, follows)
    return kernels


def _reach(code, start, stop=()):
    """Opcodes that may run after `start`, up to the first of `stop`."""
    seen, todo, ops = set(), list(code[start][1]), set()
    while todo:
        at = todo.pop()
        if at in seen or at not in code:
            continue
        seen.add(at)
        op, follows = code[at]
        ops.add(op)
        if op not in stop:
            todo += follows
    return ops


@pytest.mark.skipif(not shutil.which(OBJDUMP), reason="no AMDGPU disassembler")
def test_a_barrier_stands_between_a_solution_and_its_readers(tmp_path):
    kernels = _resident_kernels(tmp_path)
    assert len(kernels) == 5  # sheet, half sheet, general (two solvers), rows
    for name, code in kernels.items():
        # the stores of triples that some barrier follows are x; the others
        # are the finalize's pos and vel
        stores = [at for at, (op, _) in code.items() if op == "global_store_dwordx3"]
        solution = [at for at in stores if "s_barrier" in _reach(code, at)]
        assert solution and len(stores) > len(solution), name
        for at in solution:
            ops = _reach(code, at, stop=("s_barrier",))
            assert "global_load_dwordx3" not in ops, (name, hex(at))
