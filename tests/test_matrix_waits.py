"""The built kernels wait for their matrix products: a product's result is there a fixed number of instructions behind it, and
nothing on the chip holds back a vector access that comes earlier.  The compiler puts the waits in, but not in front of inline
assembly, and along a branch that skips a few instructions not enough of them (it counts the way through those).  So the
instructions themselves are followed here, along every branch, from each product to the first access of what it writes."""
from __future__ import annotations

import re
import struct
import subprocess
from pathlib import Path

import pytest

from dynamo_exp_amd import _native

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
# gfx950: passes of the matrix pipe + 4 (fp32 products: + 2); what the compiler itself leaves where nothing branches
WAITS = {"v_mfma_f32_32x32x16_bf16": 12, "v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x16_bf16": 8,
         "v_mfma_f32_16x16x4_f32": 10}
REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def regs(text):
    return {(m[1], i) for m in REG.finditer(text)
            for i in (range(int(m[2]), int(m[3]) + 1) if m[2] else (int(m[4]),))}


def device_code(library):
    """The gfx950 code objects of a library's offload bundles."""
    b, at = library.read_bytes(), 0
    while (at := b.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        n, p = struct.unpack_from("<Q", b, at + 24)[0], at + 32
        for _ in range(n):
            start, size, width = struct.unpack_from("<QQQ", b, p)
            if size and b"gfx950" in b[p + 24:p + 24 + width]:
                yield b[at + start:at + start + size]
            p += 24 + width
        at += 24


def functions(listing):
    """{name: [(instruction, operands, branch target or None)]}"""
    out = {}
    for name, body in re.findall(r"^[0-9a-f]+ <(.+)>:\n((?:.+\n)*)", listing, re.M):
        if "v_mfma" not in body:
            continue
        code, at, jumps = [], {}, []
        for m in re.finditer(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$", body, re.M):
            at[int(m[3], 16)] = len(code)
            if m[1].startswith(("s_branch", "s_cbranch")):
                jumps.append((len(code), int(re.search(r"\+0x([0-9a-f]+)>", m[4])[1], 16) if "+0x" in m[4] else 0))
            code.append([m[1], m[2], None])
        first = min(at)
        for i, off in jumps:
            code[i][2] = at[first + off]
        out[name] = code
    return out


def early(code):
    """(product, access, instructions between) of every access that comes too early."""
    found = []
    for i, (op, args, _) in enumerate(code):
        if not op.startswith("v_mfma"):
            continue
        need, ways, seen = WAITS[op], [(i + 1, 0, frozenset(regs(args.split(",")[0])))], set()
        while ways:
            j, n, left = ways.pop()
            while n < need and left and (j, n, left) not in seen:
                seen.add((j, n, left))
                op2, args2, target = code[j]
                if op2.startswith("v_mfma"):  # (a product may go on with the sums that another one leaves)
                    dst, a, b = args2.split(", ")[:3]
                    if left & (regs(a) | regs(b)):
                        found.append((f"{op} {args}", f"{op2} {args2}", n))
                    left -= regs(dst)
                elif op2.startswith(("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")) and left & regs(args2):
                    found.append((f"{op} {args}", f"{op2} {args2}", n))
                    break
                n += int(args2, 0) + 1 if op2 == "s_nop" else 1
                if op2 == "s_endpgm":
                    break
                if target is not None and op2 != "s_branch":
                    ways.append((target, n, left))
                j = target if op2 == "s_branch" else j + 1
    return found


def kernels():
    out = {}
    for module in (_native.kernels(), _native.mixers()):
        for code in device_code(Path(module.__file__)):
            r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "-"], input=code, capture_output=True, check=True)
            out |= functions(r.stdout.decode())
    return out


@pytest.mark.skipif(not OBJDUMP.exists(), reason="no disassembler")
def test_products_are_waited_for():
    code = kernels()
    assert any("prompt_attention_kernel" in n for n in code) and any("gemm256_kernel" in n for n in code)
    assert {n: e for n, c in code.items() if (e := early(c))} == {}


def test_the_check_itself():
    """An access behind a branch that is taken, behind a product that goes on with the sums, and one that waits."""
    mfma, nop = ["v_mfma_f32_32x32x16_bf16", "v[0:15], v[16:19], v[20:23], v[0:15]", None], ["s_nop", "7", None]
    use, go = ["v_max3_f32", "v40, v3, v4, v5", None], ["s_cbranch_vccnz", "3", 4]
    end = ["s_endpgm", "", None]
    assert [e[2] for e in early([mfma, go, nop, nop, use, end])] == [1]
    assert [e[2] for e in early([mfma, mfma, nop, use, end])] == [8]
    assert early([mfma, nop, nop, use, end]) == []
    assert early([mfma, ["ds_read_b128", "v[24:27], v30", None], nop, nop, use, end]) == []
