"""The wait states that gfx950 asks software for, checked over the machine code
of the built library.  The compiler's hazard pass inserts them for what it
emits itself, but takes an inline asm statement as no instruction at all: an
asm operand that is a matrix instruction's result, or a scalar register that a
vector instruction has just written, goes unguarded.

  matrix result -> any other vector, LDS or memory instruction that touches
  it: 8 wait states after v_mfma_*_16x16x32 (four passes, gfx950)
  scalar register written by a vector instruction -> memory instruction that
  reads it: 5
(LLVM's documented AMDGPU hazards for this part; an instruction is one wait
state, s_nop n is n + 1.)"""
import os
import re
import shutil
import subprocess

import pytest

import cuqwen_amd as cq

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MFMA_WAIT, SGPR_WAIT = 8, 5
_REG = re.compile(r"\b([vas])(?:(\d+)|\[(\d+):(\d+)\])|\b(vcc)\b")
_INS = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):")
_TARGET = re.compile(r"<[^>]*?\+0x([0-9a-f]+)>|<([^>]+)>")


def _regs(text):
    out = set()
    for kind, one, lo, hi, vcc in _REG.findall(text):
        if vcc:
            out.add("vcc")
        else:
            out.update(f"{kind}{i}" for i in range(int(one or lo), int(one or hi) + 1))
    return out


def _touched(op, args):
    """Vector registers whose value a non-matrix instruction needs or replaces."""
    if re.match(r"(global|buffer|flat|scratch|ds)_(load|read)", op) and "lds" not in op:
        args = args.split(",", 1)[1] if "," in args else ""   # a load's destination waits by itself
    return {r for r in _regs(args) if r[0] in "va" and r != "vcc"}


def _kernels(asm):
    name, body = None, []
    for line in asm.splitlines():
        m = re.match(r"^([0-9a-f]+) <(\S+)>:", line)
        if m:
            if body:
                yield name, body
            name, body = m.group(2), []
            continue
        m = _INS.match(line)
        if m:
            body.append((m.group(1), m.group(2), int(m.group(3), 16), line))
    if body:
        yield name, body


def _hazards(body):
    """(needed, found, instruction) for each violated rule of one kernel."""
    at = {ins[2]: i for i, ins in enumerate(body)}
    preds = [[] for _ in body]
    for i, (op, args, _, line) in enumerate(body):
        if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(body):
            preds[i + 1].append(i)
        if op.startswith("s_branch") or op.startswith("s_cbranch"):
            m = _TARGET.search(line)
            dst = body[0][2] + (int(m.group(1), 16) if m.group(1) else 0)
            preds[at[dst]].append(i)

    made = []   # per instruction: (wait, registers) that its result asks of the reader
    for op, args, _, _ in body:
        if op.startswith("v_mfma") or op.startswith("v_smfmac"):
            made.append(("mfma", _regs(args.split(",", 1)[0])))
        elif op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
            made.append(("sgpr", {r for r in _regs(args.split(",", 1)[0]) if r[0] == "s" or r == "vcc"}))
        else:
            made.append((None, set()))

    def back(i, kind, regs, need):
        stack, seen = [(p, 0) for p in preds[i]], {}
        while stack:
            p, waited = stack.pop()
            if waited >= need or seen.get(p, need) <= waited:
                continue
            seen[p] = waited
            if made[p][0] == kind and made[p][1] & regs:
                yield waited, body[p][3]
                continue
            op, args = body[p][0], body[p][1]
            step = int(args, 0) + 1 if op == "s_nop" else 1
            stack.extend((q, waited + step) for q in preds[p])

    for i, (op, args, _, line) in enumerate(body):
        if op.startswith(("v_mfma", "v_smfmac", "s_")):
            continue
        regs = _touched(op, args)
        for waited, src in back(i, "mfma", regs, MFMA_WAIT) if regs else ():
            yield MFMA_WAIT, waited, src, line
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            regs = {r for r in _regs(args) if r[0] == "s" or r == "vcc"}
            for waited, src in back(i, "sgpr", regs, SGPR_WAIT) if regs else ():
                yield SGPR_WAIT, waited, src, line


def _device_code(tmp_path):
    lib = shutil.copy(cq.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    files = [f for f in sorted(os.listdir(tmp_path)) if f.endswith("gfx950")]
    assert files
    return [subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", os.path.join(tmp_path, f)], check=True, capture_output=True,
                           text=True).stdout for f in files]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm toolchain")
def test_no_unguarded_hazards(tmp_path):
    bad, mfma = [], 0
    for asm in _device_code(tmp_path):
        for name, body in _kernels(asm):
            ops = {ins[0] for ins in body if ins[0].startswith(("v_mfma", "v_smfmac"))}
            mfma += len(ops)
            # the eight wait states are those of this shape
            assert all("_16x16x32_" in op for op in ops), (name, ops)
            bad += [f"{name}: {w} of {n} wait states\n  {src}\n  {line}" for n, w, src, line in _hazards(body)]
    assert mfma
    assert not bad, f"{len(bad)} unguarded\n" + "\n".join(bad[:20])


def test_asm_declares_m0():
    """An asm statement that writes m0 (the LDS address of a load that goes
    past the registers) says so, or a value the compiler keeps there is lost."""
    csrc, n = os.path.join(os.path.dirname(cq.LIB_PATH), "csrc"), 0
    for f in sorted(os.listdir(csrc)):
        with open(os.path.join(csrc, f)) as src:
            for stmt in re.findall(r"\basm\b[^;{]*;", src.read()):
                if re.search(r"\bs_\w+ m0\b", stmt):
                    n += 1
                    assert re.search(r':[^:]*"m0"[^:]*\)\s*;$', stmt), (f, stmt)
    assert n
