#!/usr/bin/env python3
"""ISA audit of the built kernel library (the gfx950 code objects inside liblsa_kernels.so).

A read of a VGPR in the issue slot right after the instruction that writes it can return the OLD
value on MI355X for some writer / reader pairs unless a wait state separates them. hipcc's hazard
recognizer inserts those wait states; this audit checks the binary that ships instead of trusting
it. The rules and their evidence (scripts/probes/pk_hazard_gen.py: every writer / gap / reader
combination as raw inline asm, compared bitwise against the same sequence with 16 wait states, at
one wave per SIMD, eight waves per SIMD and four hazard waves beside four MFMA-issuing waves per
SIMD, 8.4-67 M lane tests per case; profiles/r6_isa_hazards.md):

* R1 ``trans``: a transcendental VALU op (v_exp / v_log / v_rcp / v_rsq / v_sqrt / v_sin / v_cos)
  whose result is read by the NEXT VALU instruction - packed, DPP or plain 32-bit: 22 % of lanes
  read the stale value. MEASURED HAZARD.
* R2 ``dpp``: any VALU write of a VGPR that the NEXT instruction reads through DPP: 44-49 % stale.
  MEASURED HAZARD.
* R3 ``valu32->pk``: a 32-bit VALU write of a VGPR that the next packed-FP32 instruction
  (v_pk_fma / mul / add_f32, v_pk_mov_b32) reads. NOT reproduced on hardware: 0 stale reads in
  every case, including the exact round-5 GEMV site (two v_fma_f32 updating both halves of a pair,
  then v_pk_fma_f32 accumulating into it) beside MFMA-issuing waves. Kept as a conservative rule:
  the product build (-fno-slp-vectorize, csrc/build.py) forms no packed FP32 from scalar code, so
  it costs nothing, and an SLP-vectorised build of the round-5 shared GEMV body computed wrong rows
  for a reason this rule's pattern does not explain (profiles/r5_gemv_nondeterminism.md, round-6
  section).

* R4 ``mfma``: an instruction that reads a result register of a v_mfma_f32_16x16x32_bf16 / 16x16x16 fewer
  than MFMA_SLOTS issue slots behind it (s_nop N counts N + 1), along any path. The compiler keeps 7 and
  more everywhere but at the exit of some loops, where it copied accumulators (v_mov) 2 or 3 slots behind
  the last product; on MI355X these copies read the values from before it, in every lane.

* R5 ``store``: a buffer_store of three or four dwords with a scalar offset whose data registers are written within
  STORE_SLOTS issue slots. The compiler keeps two slots behind every other wide store; here it takes the hardware to read
  the data in time, and on MI355X it does not while other waves of the CU keep the memory pipe busy: the store wrote the
  new value of the register (fp32 tiles in parts of K: rows 18 and 22 of every 32 held an address, in every launch of more
  than 256 workgroups of one build).

For R1 to R3 one slot is the whole window: with one wait state (s_nop 0) or one independent VALU instruction
between writer and reader, every case of every rule read the new value; distance-2 writers never
need a wait state. The shipped library has 0 findings under all three rules (the packed-FP32
instructions that remain come from explicit vector code, each behind a packed writer or at a
distance).

usage: python csrc/isa_audit.py [path/to/liblsa_kernels.so] [arch]   (exit 1 on any finding)"""
from __future__ import annotations

import os
import re
import subprocess
import sys
import tempfile

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
LLVM = os.path.join(ROCM, "lib", "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
TARGET = "hipv4-amdgcn-amd-amdhsa--{arch}"
PK = ("v_pk_fma_f32", "v_pk_mul_f32", "v_pk_add_f32", "v_pk_mov_b32")
TRANS = ("v_exp_", "v_log_", "v_rcp_", "v_rsq_", "v_sqrt_", "v_sin_", "v_cos_")
REG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")
RULES = ("trans", "dpp", "valu32->pk", "mfma", "store")
MFMA_SLOTS = 7
STORE_SLOTS = 2
AREG = re.compile(r"\ba(?:\[(\d+):(\d+)\]|(\d+)\b)")
STORES = ("ds_write", "ds_bpermute", "global_store", "buffer_store", "flat_store", "global_atomic")
LOADS = ("ds_read", "global_load", "buffer_load", "flat_load")


def _vregs(tok: str) -> set:
    out = set()
    for m in REG.finditer(tok):
        if m.group(3) is not None:
            out.add(int(m.group(3)))
        else:
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def disassemble(so_path: str, arch: str = "gfx950") -> list:
    """Disassembly text of every ``arch`` code object bundled in the library's .hip_fatbin."""
    texts = []
    with tempfile.TemporaryDirectory() as td:
        fat = os.path.join(td, "fat.bin")
        subprocess.run([os.path.join(LLVM, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", so_path,
                        os.path.join(td, "discard.so")], check=True, capture_output=True)
        data = open(fat, "rb").read()
        starts = [m.start() for m in re.finditer(re.escape(MAGIC), data)]
        for i, st in enumerate(starts):
            chunk = data[st:starts[i + 1] if i + 1 < len(starts) else len(data)]
            cp, co = os.path.join(td, f"b{i}.bin"), os.path.join(td, f"b{i}.co")
            with open(cp, "wb") as f:
                f.write(chunk)
            r = subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--type=o", f"--input={cp}",
                                f"--targets={TARGET.format(arch=arch)}", f"--output={co}", "--unbundle"],
                               capture_output=True)
            if r.returncode != 0 or not os.path.getsize(co):
                continue
            d = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", co], check=True, capture_output=True,
                               text=True)
            texts.append(d.stdout)
    return texts


def _is_dpp(op: str, text: str) -> bool:
    return "_dpp" in op or any(k in text for k in (" quad_perm:", " row_shl:", " row_shr:", " row_ror:",
                                                     " row_mirror", " row_half_mirror", " row_bcast",
                                                     " row_share:", " row_xmask:", " wave_"))


def audit_text(text: str, rules=RULES) -> tuple:
    """(findings, packed_fp32_count): findings = [(rule, kernel, writer, reader)] for every
    reader in the issue slot right after a writer of one of its source VGPRs."""
    findings, n_pk = [], 0
    kernel, prev = None, None
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(.+)>:$", line.strip())
        if m:
            kernel, prev = m.group(1), None
            continue
        s = line.split("//")[0].strip()
        if not s:
            continue
        op = s.split()[0]
        ops = [o.strip() for o in s[len(op):].split(",")] if len(s) > len(op) else []
        is_valu = op.startswith("v_") and not op.startswith(("v_mfma", "v_smfma"))
        if op.startswith(PK):
            n_pk += 1
        if is_valu and prev is not None:
            srcs = set().union(*[_vregs(o) for o in ops[1:]]) if len(ops) > 1 else set()
            if prev[2] & srcs:
                pop = prev[0]
                if "trans" in rules and pop.startswith(TRANS):
                    findings.append(("trans", kernel, prev[1], s))
                # DPP reads its first source through the permute network
                if "dpp" in rules and _is_dpp(op, s) and len(ops) > 1 and prev[2] & _vregs(ops[1]):
                    findings.append(("dpp", kernel, prev[1], s))
                if "valu32->pk" in rules and op.startswith(PK) and not pop.startswith(PK):
                    findings.append(("valu32->pk", kernel, prev[1], s))
        if is_valu and ops:
            prev = (op, s, _vregs(ops[0]))
        else:
            prev = None
    return findings, n_pk


def _regs(tok: str) -> set:
    """Vector and accumulator registers an operand names."""
    out = {("v", i) for i in _vregs(tok)}
    for m in AREG.finditer(tok):
        lo, hi = (m.group(3), m.group(3)) if m.group(3) is not None else (m.group(1), m.group(2))
        out |= {("a", i) for i in range(int(lo), int(hi) + 1)}
    return out


def _kernels(text: str):
    """(name, [(address, instruction, mnemonic, operands)]) of a disassembly."""
    name, ins = None, []
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(.+)>:$", line.strip())
        if m:
            if name is not None:
                yield name, ins
            name, ins = m.group(1), []
        elif "//" in line:
            s, note = (x.strip() for x in line.split("//", 1))
            if s:
                op = s.split()[0]
                ins.append((int(note.split(":")[0], 16), s, op, [o.strip() for o in s[len(op):].split(",")] if len(s) > len(op) else []))
    if name is not None:
        yield name, ins


def _target(addr: int, operand: str) -> int:
    """Where the branch at ``addr`` goes."""
    off = int(operand, 0)
    return addr + 4 + 4 * (off - 0x10000 if off >= 0x8000 else off)


def audit_mfma(text: str, slots: int = MFMA_SLOTS) -> list:
    """Findings of rule ``mfma``: every path from an MFMA, its branches taken and not."""
    findings = []
    for kernel, ins in _kernels(text):
        at = {a: i for i, (a, *_) in enumerate(ins)}
        for i, (_, writer, op, ops) in enumerate(ins):
            if not op.startswith("v_mfma"):
                continue
            seen, todo = {}, [(i + 1, 0, frozenset(_regs(ops[0])))]
            while todo:
                j, d, live = todo.pop()
                if j >= len(ins) or d >= slots or not live or seen.get(j, slots) <= d:
                    continue
                seen[j] = d
                addr, s, op2, o2 = ins[j]
                if op2 in ("s_endpgm", "s_setpc_b64"):
                    continue
                if op2 == "s_nop":
                    todo.append((j + 1, d + int(o2[0], 0) + 1, live))
                    continue
                if op2.startswith("v_mfma"):  # chains of accumulation are the hardware's
                    if (_regs(o2[1]) | _regs(o2[2])) & live:
                        findings.append(("mfma", kernel, writer, s))
                    else:
                        todo.append((j + 1, d + 1, live - _regs(o2[0])))
                    continue
                store, load = op2.startswith(STORES), op2.startswith(LOADS)
                if op2.startswith("v_") or store or load:
                    if set().union(*[_regs(o) for o in (o2 if store else o2[1:])]) & live:
                        findings.append(("mfma", kernel, writer, s))
                        continue
                    if not store and o2:
                        live = live - _regs(o2[0])
                if op2 == "s_branch" or op2.startswith("s_cbranch"):
                    todo.append((at.get(_target(addr, o2[0]), len(ins)), d + 1, live))
                    if op2 == "s_branch":
                        continue
                todo.append((j + 1, d + 1, live))
    return findings


def audit_stores(text: str, slots: int = STORE_SLOTS) -> list:
    """Findings of rule ``store``: every path from a store, its branches (a slot each) taken and not."""
    findings = []
    for kernel, ins in _kernels(text):
        at = {a: i for i, (a, *_) in enumerate(ins)}
        for i, (_, writer, op, ops) in enumerate(ins):
            if not op.startswith(("buffer_store_dwordx3", "buffer_store_dwordx4")) or not re.match(r"s\d+\b|m0\b", ops[3]):
                continue
            data, seen, todo = _regs(ops[0]), {}, [(i + 1, 0)]
            while todo:
                j, d = todo.pop()
                if j >= len(ins) or d >= slots or seen.get(j, slots) <= d:
                    continue
                seen[j] = d
                addr, s, op2, o2 = ins[j]
                if op2 in ("s_endpgm", "s_setpc_b64"):
                    continue
                if op2.startswith("v_") and o2 and _regs(o2[0]) & data:
                    findings.append(("store", kernel, writer, s))
                    continue
                if op2 == "s_branch" or op2.startswith("s_cbranch"):
                    todo.append((at.get(_target(addr, o2[0]), len(ins)), d + 1))
                    if op2 == "s_branch":
                        continue
                todo.append((j + 1, d + (int(o2[0], 0) + 1 if op2 == "s_nop" else 1)))
    return findings


def audit(so_path: str, arch: str = "gfx950") -> dict:
    findings, n_pk, n_obj = [], 0, 0
    for t in disassemble(so_path, arch):
        f, n = audit_text(t)
        findings += f + audit_mfma(t) + audit_stores(t)
        n_pk += n
        n_obj += 1
    by_rule = {r: sum(1 for f in findings if f[0] == r) for r in RULES}
    return {"code_objects": n_obj, "packed_fp32_instructions": n_pk, "findings": findings, "by_rule": by_rule}


def main() -> None:
    so = sys.argv[1] if len(sys.argv) > 1 else os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                                              "llm_sharding_amd", "_native", "liblsa_kernels.so")
    arch = sys.argv[2] if len(sys.argv) > 2 else "gfx950"
    res = audit(so, arch)
    for r, k, w, rd in res["findings"][:20]:
        print(f"{r:10s} {k[:80]}: [{w}] -> [{rd}]")
    print(f"code objects {res['code_objects']}, packed FP32 instructions {res['packed_fp32_instructions']}, "
          f"findings by rule {res['by_rule']}")
    sys.exit(1 if res["findings"] or not res["code_objects"] else 0)


if __name__ == "__main__":
    main()
