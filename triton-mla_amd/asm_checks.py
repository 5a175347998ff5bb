"""Scans of the compiler's gfx950 assembly for hazards of inline asm.

The compiler inserts the waits and wait states that its own instructions
need, but it does not look inside inline asm. Three things can therefore go
wrong without any message, depending on nothing but the register allocation
of one build:

  * ``inflight_touches``: the destination of an LDS or scalar load issued by
    inline asm is read, copied or overwritten before an ``s_waitcnt lgkmcnt``
    that covers it (LDS operations return in order, so ``lgkmcnt(n)`` covers
    all but the newest n; scalar loads return in any order and are covered by
    ``lgkmcnt(0)`` only);
  * ``operand_hazards``: a vector-ALU instruction (a copy out of an AGPR for
    instance) writes an operand of an MFMA or of a DPP move fewer than two wait
    states before it, where one of the two is inline asm;
  * ``mfma_result_touches``: the result of an MFMA is read or overwritten
    before the MFMA has finished, where one of the two is inline asm.

All three follow every branch of a kernel (a forward dataflow analysis over
its blocks, taking the worst of all paths that lead to a block, whatever the
branch conditions). An instruction counts as one wait state, ``s_nop n`` as
n + 1.
"""

from __future__ import annotations

import re
from typing import NamedTuple

OPERAND_WAIT_STATES = 2  # vector-ALU write of a register -> MFMA or DPP move that reads it
RESULT_WINDOW = 18       # wait states after which any MFMA used here has finished
_COUNTER = 15            # lgkmcnt counts to 15

_REG = re.compile(r"\b([vsa])(?:\[(\d+):(\d+)\]|(\d+))(?![\w\[])")


class Ins(NamedTuple):
    line: int
    op: str
    parts: tuple  # operands' registers, a frozenset each
    regs: frozenset  # of all operands
    asm: bool  # issued by inline asm
    text: str
    nop: int  # wait states it takes
    wait: int  # lgkmcnt it waits for (-1: none)
    target: str  # branch target, "" for none


class Block(NamedTuple):
    ins: list
    succ: list


_parsed: dict = {}


def _parse(text: str):
    got = _parsed.get(text)
    if got is None:
        op, _, args = text.partition(" ")
        parts = []
        for p in args.split(","):
            regs = set()
            for kind, lo, hi, one in _REG.findall(p):
                regs.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
            parts.append(frozenset(regs))
        nop = int(args.strip(), 0) + 1 if op == "s_nop" else 1
        wait = -1
        if op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", args)
            wait = int(m.group(1)) if m else 0 if args.strip() == "0" else -1
        target = args.split()[-1] if op.startswith(("s_cbranch", "s_branch")) else ""
        got = _parsed[text] = (op, tuple(parts), frozenset().union(*parts), nop, wait, target)
    return got


def kernels(asm_path: str):
    """(name, [Block]) of every function of an assembly file."""
    with open(asm_path) as f:
        name, body, in_asm = None, [], False
        for ln, raw in enumerate(f, 1):
            t = raw.strip()
            if t.startswith(";;#ASM"):
                in_asm = t.startswith(";;#ASMSTART")
                continue
            t = t.split(";")[0].strip()
            if not t:
                continue
            if t.endswith(":"):
                if re.match(r"[A-Za-z_]", t):
                    if name is not None:
                        yield name, _blocks(body)
                    name, body = t[:-1], []
                elif t.startswith(".Lfunc_end"):
                    if name is not None:
                        yield name, _blocks(body)
                    name, body = None, []
                elif t.startswith(".LBB"):
                    body.append(t[:-1])
                continue
            if t.startswith(".") or name is None:
                continue
            op, parts, regs, nop, wait, target = _parse(re.sub(r"\s+", " ", t))
            body.append(Ins(ln, op, parts, regs, in_asm, t, nop, wait, target))
        if name is not None:
            yield name, _blocks(body)


def _blocks(body: list) -> list:
    blocks, labels, cur = [], {}, []

    def close():
        nonlocal cur
        blocks.append(Block(cur, []))
        cur = []

    for item in body:
        if isinstance(item, str):
            if cur:
                close()
            labels[item] = len(blocks)
        else:
            cur.append(item)
            if item.target or item.op == "s_endpgm":
                close()
    close()
    for i, blk in enumerate(blocks):
        last = blk.ins[-1] if blk.ins else None
        if last is not None and last.target in labels:
            blk.succ.append(labels[last.target])
        if (last is None or last.op not in ("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            blk.succ.append(i + 1)
    return blocks


def _flow(blocks: list, step, merge) -> list:
    """Findings of ``step(state, ins, report)`` (which updates the state, a
    dict of registers, in place) over every path; ``merge`` picks the worse of
    two values a register has on two paths."""
    entry: list = [None] * len(blocks)
    entry[0] = {}
    work, found = [0], {}

    def report(ins, other):
        found.setdefault((ins.line, other.line), (other.text, ins.text))

    while work:
        i = work.pop()
        state = dict(entry[i])
        for ins in blocks[i].ins:
            step(state, ins, report)
        for j in blocks[i].succ:
            old = entry[j]
            if old is None:
                entry[j] = dict(state)
                work.append(j)
                continue
            changed = False
            for reg, val in state.items():
                new = merge(old[reg], val) if reg in old else val
                if old.get(reg) != new:
                    old[reg] = new
                    changed = True
            if changed and j not in work:
                work.append(j)
    return [found[k] for k in sorted(found)]


def _scan(asm_path: str, wanted, step, merge) -> list:
    found = []
    for _, blocks in kernels(asm_path):
        if any(wanted(ins) for blk in blocks for ins in blk.ins):
            found += _flow(blocks, step, merge)
    return found


def _asm_load(ins: Ins) -> bool:
    return ins.asm and ins.op.startswith(("ds_read", "s_load"))


def inflight_touches(asm_path: str) -> list:
    """(load, instruction) pairs: see the module's docstring."""

    # register -> (LDS operations issued since its load, the load); a scalar
    # load's count stays at -1, so that only lgkmcnt(0) covers it
    def step(state, ins, report):
        if ins.wait >= 0:
            for reg in [r for r, (since, _) in state.items() if ins.wait == 0 or since >= ins.wait]:
                del state[reg]
            return
        if state:
            for reg in ins.regs & state.keys():
                report(ins, state.pop(reg)[1])
            if ins.op.startswith("ds_"):
                for reg, (since, load) in state.items():
                    if 0 <= since < _COUNTER:
                        state[reg] = (since + 1, load)
        if _asm_load(ins):
            for reg in ins.parts[0]:
                state[reg] = (0 if ins.op.startswith("ds_") else -1, ins)

    return _scan(asm_path, _asm_load, step, min)


def _early_reader(ins: Ins) -> bool:
    return ins.op.startswith("v_mfma") or ins.op.endswith("_dpp")


def operand_hazards(asm_path: str) -> list:
    """(writer, MFMA or DPP move) pairs: see the module's docstring."""

    # register -> (wait states since a vector-ALU instruction wrote it, that instruction)
    def step(state, ins, report):
        if state and _early_reader(ins):
            # (the first operand is the result; a DPP move may keep old lanes of it)
            read = ins.parts[1:4] if ins.op.startswith("v_mfma") else ins.parts
            for reg in frozenset().union(*read) & state.keys():
                if ins.asm or state[reg][1].asm:
                    report(ins, state[reg][1])
        for reg, (since, writer) in list(state.items()):
            if since + ins.nop >= OPERAND_WAIT_STATES:
                del state[reg]
            else:
                state[reg] = (since + ins.nop, writer)
        if ins.op.startswith("v_") and not ins.op.startswith("v_mfma"):
            written = ins.parts[0] | ins.parts[1] if "swap" in ins.op else ins.parts[0]
            for reg in written:
                if reg[0] != "s":
                    state[reg] = (0, ins)

    return _scan(asm_path, lambda ins: ins.asm and ins.op.startswith("v_"), step, min)


def mfma_result_hazards(asm_path: str, window: int = RESULT_WINDOW) -> list:
    """(MFMA, instruction) pairs: see the module's docstring. Of the MFMAs
    that are not inline asm, those with an AGPR result are left to the
    compiler unless inline asm touches the result. An MFMA that accumulates
    into the exact result of the previous one is the hardware's back-to-back
    case."""

    # register -> (wait states left, the MFMA)
    def step(state, ins, report):
        mfma = ins.op.startswith("v_mfma")
        for reg in ins.regs & state.keys():
            by = state[reg][1]
            if not (by.asm or ins.asm or reg[0] == "v"):
                continue
            if mfma and by.parts[0] == ins.parts[0] == ins.parts[3] and reg not in ins.parts[1] | ins.parts[2]:
                continue
            report(ins, by)
        for reg, (left, by) in list(state.items()):
            if left <= ins.nop:
                del state[reg]
            else:
                state[reg] = (left - ins.nop, by)
        if mfma:
            for reg in ins.parts[0]:
                state[reg] = (window, ins)

    return _scan(asm_path, lambda ins: ins.op.startswith("v_mfma"), step, max)
