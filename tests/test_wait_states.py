"""Wait states in the built device code that the hardware does not insert itself.

On gfx9 a vector memory instruction that reads a scalar register needs five wait
states behind a vector instruction that wrote it (v_readfirstlane_b32, a compare
into a register pair, ...).  The compiler keeps them for instructions that it
schedules and cannot see those inside inline assembly (the direct global -> LDS
loads of csrc/m2_common.h), so the library's own code is scanned: from every
vector memory instruction back over up to five wait states, along every path."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from mamba2_jax import _lib as L

NEEDED = 5
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(os.path.dirname(L.LIB_PATH)), "csrc")
INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.dirname(L.LIB_PATH))), "include")

SGPR = re.compile(r"\b(?:s\[(\d+):(\d+)\]|s(\d+)|(vcc(?:_lo|_hi)?))(?![\w\[])")
VMEM = ("global_", "buffer_", "flat_", "scratch_")
# vector instructions whose second operand is a scalar destination too
SDST2 = ("v_add_co", "v_sub_co", "v_subrev_co", "v_addc_co", "v_subb_co", "v_subbrev_co",
         "v_div_scale", "v_mad_u64_u32", "v_mad_i64_i32")


def code_objects(path):
    """The gfx950 code objects bundled into a HIP library."""
    d = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    p = d.find(magic)
    while p >= 0:
        n, o = struct.unpack_from("<Q", d, p + 24)[0], p + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", d, o)
            if b"gfx950" in d[o + 24:o + 24 + ln]:
                yield d[p + off:p + off + size]
            o += 24 + ln
        p = d.find(magic, p + 24)


def _regs(text):
    out = set()
    for a, b, one, vcc in SGPR.findall(text):
        if vcc:
            out |= {"vcc_lo", "vcc_hi"} if vcc == "vcc" else {vcc}
        else:
            out |= set(range(int(a), int(b) + 1)) if a else {int(one)}
    return out


def _written(op, operands):
    """Scalar registers a vector ALU instruction writes."""
    if not op.startswith("v_") or op.startswith("v_mfma"):
        return set()
    ops = operands.split(",")
    return _regs(ops[0]) | (_regs(ops[1]) if op.startswith(SDST2) and len(ops) > 1 else set())


def violations(disassembly):
    """[(kernel, memory instruction, writer, wait states)] of llvm-objdump -d's text."""
    bad, name, code = [], None, []

    def check():
        at = {a: i for i, (a, *_) in enumerate(code)}
        preds = {}
        for i, (addr, op, operands, target) in enumerate(code):
            if target is not None and target in at:
                preds.setdefault(at[target], []).append(i)
        for i, (addr, op, operands, _) in enumerate(code):
            reads = _regs(operands) if op.startswith(VMEM) else set()
            todo, seen = [(i, 0)], set()
            while todo and reads:
                j, ws = todo.pop()
                before = list(preds.get(j, ()))
                if j and code[j - 1][1] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                    before.append(j - 1)
                for k in before:
                    op2, operands2 = code[k][1:3]
                    if _written(op2, operands2) & reads:
                        bad.append((name, f"{op} {operands}", f"{op2} {operands2}", ws))
                        continue
                    w = ws + (int(operands2, 0) + 1 if op2 == "s_nop" else 1)
                    if w < NEEDED and (k, w) not in seen:
                        seen.add((k, w))
                        todo.append((k, w))

    start = 0
    for line in disassembly.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:$", line)
        if m:
            if code:
                check()
            start, name, code = int(m[1], 16), m[2], []
            continue
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):", line)
        if m:
            t = re.search(r"<.+?(?:\+0x([0-9a-f]+))?>$", line) if m[1].startswith(("s_cbranch", "s_branch")) else None
            code.append((int(m[3], 16), m[1], m[2], start + int(t[1] or "0", 16) if t else None))
    if code:
        check()
    return bad


def _scan(elf, tmp_path):
    f = tmp_path / "co.elf"
    f.write_bytes(elf)
    r = subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True, check=True)
    return violations(r.stdout)


needs_objdump = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not found")


def test_scanner_on_known_sequences():
    """Straight code, an s_nop's count, a branch into the load, a scalar ALU writer."""
    def text(*ins):
        return "0000000000000000 <k>:\n" + "\n".join(
            f"\t{s.split(' <')[0]} // {4 * i:012X}: 00000000{' <' + s.split(' <')[1] if ' <' in s else ''}"
            for i, s in enumerate(ins))
    load, w = "global_load_lds_dwordx4 v1, s[4:5]", "v_readfirstlane_b32 s5, v0"
    assert len(violations(text(w, "s_mov_b32 m0, s2", "s_nop 0", load))) == 1
    assert not violations(text(w, "s_mov_b32 m0, s2", "s_nop 3", load))
    assert len(violations(text(w, "s_mov_b32 m0, s2", "s_nop 2", load))) == 1
    assert not violations(text("s_add_u32 s4, s4, s6", load))
    assert not violations(text("v_mov_b32_e32 v2, s5", load))
    assert len(violations(text(load, "s_mov_b32 s9, 0", w, "s_cbranch_scc1 65532 <k>"))) == 1
    assert len(violations(text("v_cmp_gt_i32_e64 s[4:5], v1, v2", "s_nop 1", load))) == 1


@needs_objdump
@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_scalar_base_loads_by_themselves(tmp_path):
    """dma16s / dma4s whose base the compiler has to read out of a vector register
    (a uniform value that it cannot prove to be one) right before the load."""
    src = tmp_path / "k.hip"
    src.write_text('''#include "m2_common.h"
        __global__ void k(const char* const* p, int* o) {
            __shared__ __align__(16) char ring[4096];
            const char* b = p[threadIdx.x >> 6];
            const uint32_t l = lds_addr(ring);
            dma16s(b, 16 * (threadIdx.x & 63), l);
            dma4s(b + 1024 * (threadIdx.x >> 6), 4 * (threadIdx.x & 63), l + 1024);
            wait_vmem<0>();
            __syncthreads();
            o[threadIdx.x] = ring[threadIdx.x];
        }''')
    out = tmp_path / "k.co"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--genco",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I", INCLUDE, "-I", CSRC, str(src), "-o", str(out)],
                   check=True, capture_output=True)
    objs = list(code_objects(out))
    assert objs
    assert not [b for o in objs for b in _scan(o, tmp_path)]


@needs_objdump
def test_library_keeps_the_wait_states(tmp_path):
    objs = list(code_objects(L.LIB_PATH))
    assert len(objs) > 10
    bad = [b for o in objs for b in _scan(o, tmp_path)]
    assert not bad, f"{len(bad)} loads, the first: {bad[:4]}"
