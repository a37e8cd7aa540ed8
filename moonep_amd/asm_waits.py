"""Loads in asm statements against the waits that make their results valid, in the compiler's assembly.

The 256 x 256 GEMM kernels issue some loads from asm statements, because for a load that the compiler knows it
also waits for every younger one.  To the compiler such a result is there at once: it may copy, spill
or read the register anywhere behind the statement.  The waits are counted by hand, and the statement
``; arrived %0 ..`` says from where on the result may be used.  ``check`` follows every path from such
a load through the assembly: until a wait that covers it no instruction may mention its registers, and
no path may reach the ``arrived`` of its registers before that wait.  Nothing may be spilled to memory
either (a spill is one of the copies meant above).
"""

from __future__ import annotations

import re
from collections import deque

_FUNCTION = re.compile(r"^(\S+):\s*; @\1")
_LABEL = re.compile(r"^(\.\w+):")
_REGS = re.compile(r"\bv(?:(\d+)|\[(\d+):(\d+)\])(?!\w)")
_ACC = re.compile(r"\ba(?:\d+|\[\d+:\d+\])(?!\w)")
_MOST = 63      # the largest count that s_waitcnt vmcnt can name


def _registers(text):
    regs = set()
    for one, lo, hi in _REGS.findall(text):
        regs.update((int(one),) if one else range(int(lo), int(hi) + 1))
    return regs


class _Instruction:
    def __init__(self, text, in_asm, line):
        self.text, self.line, self.in_asm = text, line, in_asm
        self.arrived = text.startswith("; arrived")
        self.op = "" if self.arrived else text.split()[0]
        self.regs = _registers(text)
        # vector memory loads count up vmcnt in order (stores do, too; without them the count is the
        # safe side)
        self.vmem = bool(re.match(r"(global|buffer|flat|scratch)_load", self.op))
        self.vm_wait = self.lgkm_wait = None
        if self.op == "s_waitcnt":
            vm, lgkm = re.search(r"vmcnt\((\d+)\)", text), re.search(r"lgkmcnt\((\d+)\)", text)
            self.vm_wait = int(vm.group(1)) if vm else None
            self.lgkm_wait = int(lgkm.group(1)) if lgkm else None


def functions(assembly):
    """name -> (instructions, label -> index) of every function with an asm statement's load or mark."""
    found, name = {}, None
    for number, raw in enumerate(assembly.splitlines(), 1):
        start = _FUNCTION.match(raw)
        if start:
            name, in_asm = start.group(1), False
            found[name] = ([], {})
            continue
        if name is None:
            continue
        if raw.startswith(".Lfunc_end"):
            name = None
            continue
        body, labels = found[name]
        label = _LABEL.match(raw)
        if label:
            labels[label.group(1)] = len(body)
            continue
        text = raw.strip()
        if text == ";;#ASMSTART":
            in_asm = True
        elif text == ";;#ASMEND":
            in_asm = False
        elif in_asm and text.startswith("; arrived"):
            body.append(_Instruction(text, True, number))
        else:
            text = text.split(";")[0].strip()
            if text and not text.startswith("."):
                body.append(_Instruction(text, in_asm, number))
    return found


def _successors(body, labels, i):
    ins = body[i]
    if ins.op == "s_endpgm":
        return ()
    target = labels.get(ins.text.split()[-1]) if ins.op.startswith(("s_branch", "s_cbranch")) else None
    if ins.op.startswith(("s_branch", "s_cbranch")) and target is None:
        raise ValueError(f"line {ins.line}: unknown branch target: {ins.text}")
    if ins.op.startswith(("s_setpc", "s_swappc", "s_call")):
        raise ValueError(f"line {ins.line}: a path that cannot be followed: {ins.text}")
    if ins.op == "s_branch":
        return (target,)
    return (i + 1,) if target is None else (i + 1, target)


def _follow(name, body, labels, start):
    load = body[start]
    dest = _registers(load.text.split(",")[0])
    lds = load.op.startswith("ds_")
    seen, queue = set(), deque((i, 0) for i in _successors(body, labels, start))
    faults = []
    while queue:
        at, younger = queue.popleft()
        if (at, younger) in seen or at >= len(body):
            continue
        seen.add((at, younger))
        ins = body[at]
        wait = ins.lgkm_wait if lds else ins.vm_wait
        if wait is not None and wait <= (0 if lds else younger):
            continue        # covered from here on
        if ins.regs & dest:
            faults.append(f"{name}: line {ins.line}: `{ins.text}` before the wait for the load of line {load.line}, `{load.text}`")
            break
        younger = min(younger + (ins.vmem and not lds), _MOST)
        queue.extend((n, younger) for n in _successors(body, labels, at))
    return faults


def _accumulators(name, body, labels):
    """Faults around matrix instructions in asm statements."""
    if not any(ins.in_asm and ins.op.startswith("v_mfma") for ins in body):
        return []
    faults = {}
    for i, ins in enumerate(body):
        if not ins.in_asm and _ACC.search(ins.text):
            faults[i] = "touches an accumulation register"
        if not ins.op.startswith("v_") or ins.op.startswith("v_mfma"):
            continue
        # a VALU write: two issue slots on every way from it, around loops too, before its register is an operand
        written = _registers(ins.text.split(",")[0])
        todo = [(at, 0) for at in _successors(body, labels, i)] if written else []
        while todo:
            at, slots = todo.pop()
            if slots >= 2 or at >= len(body):
                continue
            after = body[at]
            if after.op.startswith("v_mfma") and after.regs & written:
                faults[at] = "too early after the VALU write of an operand"
            slots += int(after.text.split()[1]) + 1 if after.op == "s_nop" else 0 if after.arrived else 1
            todo.extend((n, slots) for n in _successors(body, labels, at))
    return [f"{name}: line {body[i].line}: `{body[i].text}` {what}" for i, what in sorted(faults.items())]


def check(assembly, kernels=("gemm_",)):
    """(faults, loads followed) of the functions whose names hold one of ``kernels``."""
    faults, followed = [], 0
    for name, (body, labels) in functions(assembly).items():
        if not any(k in name for k in kernels):
            continue
        faults += _accumulators(name, body, labels)
        for i, ins in enumerate(body):
            if ins.in_asm and (ins.op.startswith("ds_read") or ins.vmem) and not ins.text.endswith(" lds"):
                followed += 1
                faults += _follow(name, body, labels, i)
    # the resources the compiler reports per kernel
    for block in re.split(r"^  - ", assembly[assembly.rfind("amdhsa.kernels:"):], flags=re.M)[1:]:
        name = re.search(r"^\s+\.name:\s+(\S+)$", block, re.M)
        if not name or not any(k in name.group(1) for k in kernels):
            continue
        for key in (".vgpr_spill_count", ".private_segment_fixed_size"):
            value = re.search(rf"^\s+\{key}:\s+(\d+)$", block, re.M)
            if value and int(value.group(1)):
                faults.append(f"{name.group(1)}: {key} {value.group(1)}")
    return faults, followed
