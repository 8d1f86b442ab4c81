"""Wait-state rules of gfx9 that the compiler cannot keep for inline assembly, checked on device assembly.

The kernels issue ``global_load_lds_dwordx4`` from inline asm (so that the compiler's wait-count pass does not
serialise ring reads behind it) and read DMA base addresses back to scalar registers there. The compiler's hazard
recognizer does not look inside, so three rules fall to the source:

* a vector-ALU write of an SGPR (``v_readfirstlane_b32`` of a DMA base address, the ``v_readlane_b32`` of a spilled
  one, a compare's lane mask, a carry-out) needs 5 wait states before a memory instruction reads that SGPR: a stale
  base reads a wild address;
* a scalar write of M0 needs 1 wait state before an LDS DMA reads M0;
* a vector-ALU write of a VGPR needs 1 wait state before a lane read of it.

The checks follow the control flow: each kernel's assembly is split into basic blocks (labels, branches,
``s_endpgm``), and from every reader they walk back over every path into it (fall-through, branch targets and loop
back-edges). ``build.py`` runs them on what it compiles and fails on a finding.
"""

from __future__ import annotations

import re
from typing import Dict, List, Set, Tuple

VALU_SGPR_WAITS = 5  # VALU writes an SGPR -> a VMEM instruction reads it
M0_WAITS = 1  # SALU writes M0 -> an LDS DMA reads it


def _sgprs(text: str) -> Set[str]:
    regs = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]", text):
        regs.update(f"s{r}" for r in range(int(m.group(1)), int(m.group(2)) + 1))
    regs.update(f"s{m.group(1)}" for m in re.finditer(r"\bs(\d+)\b", text))
    for m in re.finditer(r"\b(vcc|m0|exec)(_lo|_hi)?\b", text):
        regs.add(m.group(1))
    return regs


def _operands(line: str) -> List[str]:
    parts = line.split(None, 1)
    return [o.strip() for o in parts[1].split(",")] if len(parts) > 1 else []


# VOP3 forms whose second operand is a scalar destination (carry-out / lane mask)
_SDST2 = re.compile(r"^v_(add|sub|subrev)_co_(ci_)?u32_e64$|^v_(addc|subb|subbrev)_co_u32_e64$|"
                    r"^v_div_scale_f(32|64)|^v_mad_(u|i)64_(u|i)32")


def valu_sgpr_dests(line: str) -> Set[str]:
    """Scalar registers a vector-ALU instruction writes (empty for other instructions)."""
    op = line.split()[0]
    if not op.startswith("v_"):
        return set()
    ops = _operands(line)
    if not ops:
        return set()
    if op.startswith(("v_readfirstlane", "v_readlane")) or (op.startswith("v_cmp") and op.endswith("_e64")):
        return _sgprs(ops[0])
    if _SDST2.match(op) and len(ops) > 1:
        return _sgprs(ops[1])
    if op.startswith("v_cmp") or re.match(r"^v_(add|sub|subrev)_co_u32_e32$|^v_(addc|subb)_co_u32_e32$", op):
        return {"vcc"}  # e32 compares and carries write VCC
    return set()


# scalar-ALU and scalar-load opcodes whose first operand is their destination
_SALU_DST = re.compile(r"^s_(mov|movk|cmov|cmovk|cselect|add|addc|addk|sub|subb|mul|mulk|mul_hi|lshl|lshr|ashr|"
                       r"lshl[1-4]_add|and|or|xor|andn2|orn2|nand|nor|xnor|not|bfe|bfm|min|max|abs|absdiff|brev|"
                       r"ff0|ff1|flbit|bcnt0|bcnt1|sext|pack|getpc|load|buffer_load)(_|$)")


def sgpr_dests(line: str) -> Set[str]:
    """Scalar registers any instruction writes, as far as the checker needs to know: vector-ALU
    scalar destinations and the destinations of scalar-ALU ops and scalar loads."""
    op = line.split()[0]
    if op.startswith("v_"):
        return valu_sgpr_dests(line)
    ops = _operands(line)
    if ops and _SALU_DST.match(op):
        return _sgprs(ops[0])
    return set()


def _is_vmem(op: str) -> bool:
    return op.startswith(("global_", "buffer_", "flat_", "scratch_"))


def _waits_of(line: str) -> int:
    op = line.split()[0]
    if op == "s_nop":
        return int(_operands(line)[0], 0) + 1
    return 1


class Function:
    """One kernel's instructions as basic blocks: blocks[i] = list of instructions; preds[i]."""

    def __init__(self, name: str, lines: List[str]):
        self.name = name
        blocks: List[List[str]] = [[]]
        labels: Dict[str, int] = {}
        ends_flow: List[bool] = []
        targets: List[List[str]] = []
        cur_targets: List[str] = []
        for raw in lines:
            t = raw.split(";")[0].strip()
            if not t:
                continue
            if t.endswith(":") and not t.startswith("s_"):
                if blocks[-1] or cur_targets:
                    ends_flow.append(False)
                    targets.append(cur_targets)
                    blocks.append([])
                    cur_targets = []
                labels[t[:-1]] = len(blocks) - 1
                continue
            if t.startswith("."):
                continue
            blocks[-1].append(t)
            op = t.split()[0]
            if op.startswith("s_branch") or op.startswith("s_cbranch"):
                cur_targets = [_operands(t)[0]]
                ends_flow.append(op.startswith("s_branch"))
                targets.append(cur_targets)
                blocks.append([])
                cur_targets = []
            elif op in ("s_endpgm", "s_setpc_b64"):
                ends_flow.append(True)
                targets.append([])
                blocks.append([])
                cur_targets = []
        ends_flow.append(True)
        targets.append(cur_targets)
        self.blocks = blocks
        self.preds: List[List[int]] = [[] for _ in blocks]
        for i in range(len(blocks)):
            if not ends_flow[i] and i + 1 < len(blocks):
                self.preds[i + 1].append(i)
            for lab in targets[i]:
                if lab in labels:
                    self.preds[labels[lab]].append(i)

    def writers_within(self, block: int, index: int, regs: Set[str], budget: int, pick) -> List[str]:
        """Instructions on any path into (block, index) that ``pick(line) & regs`` and lie fewer
        than ``budget`` wait states before it, counting only the last write of each register on
        the path (a later write by any instruction, scalar ALU included, hides an earlier one)."""
        found: List[str] = []
        seen: Set[Tuple[int, int, frozenset]] = set()

        def walk(b: int, i: int, left: int, live: frozenset):
            if (b, left, live) in seen:
                return
            seen.add((b, left, live))
            ins = self.blocks[b]
            for j in range(i - 1, -1, -1):
                if pick(ins[j]) & live:
                    found.append(ins[j])
                    return
                live = live - sgpr_dests(ins[j])
                if not live:
                    return
                left -= _waits_of(ins[j])
                if left <= 0:
                    return
            for p in self.preds[b]:
                walk(p, len(self.blocks[p]), left, live)

        walk(block, index, budget, frozenset(regs))
        return found


def functions(asm: str) -> List[Function]:
    """The code symbols of ``asm`` (``.type <name>,@function``: kernels and device functions), each
    up to its .Lfunc_end."""
    code = set(re.findall(r"\.type\s+([\w.$]+),@function", asm))
    out, name, body = [], None, []
    for line in asm.splitlines():
        m = re.match(r"^([A-Za-z_][\w.$]*):(\s|;|$)", line)
        if m and m.group(1) in code:
            if name is not None:
                out.append(Function(name, body))
            name, body = m.group(1), []
            continue
        if name is not None:
            if line.startswith(".Lfunc_end"):
                out.append(Function(name, body))
                name, body = None, []
            else:
                body.append(line)
    if name is not None:
        out.append(Function(name, body))
    return out


def _m0_write(line: str) -> Set[str]:
    op = line.split()[0]
    ops = _operands(line)
    if op.startswith("s_") and not op.startswith(("s_nop", "s_waitcnt", "s_cbranch", "s_branch")) and ops:
        return {"m0"} if ops[0] == "m0" else set()
    return set()


def find_hazards(asm: str):
    """(VALU SGPR write -> VMEM read within 5 wait states, SALU M0 write -> LDS DMA) instances,
    over every control-flow path of every function in ``asm``."""
    sgpr_hazards, m0_hazards = [], []
    for fn in functions(asm):
        for b, ins in enumerate(fn.blocks):
            for i, line in enumerate(ins):
                op = line.split()[0]
                if not _is_vmem(op):
                    continue
                reads = _sgprs(" ".join(_operands(line))) - {"exec"}
                if "_lds_" in op:
                    reads.add("m0")
                if reads:
                    for w in fn.writers_within(b, i, reads, VALU_SGPR_WAITS, valu_sgpr_dests):
                        sgpr_hazards.append((fn.name, w, line))
                if "_lds_" in op:
                    for w in fn.writers_within(b, i, {"m0"}, M0_WAITS, _m0_write):
                        m0_hazards.append((fn.name, w, line))
    dedup = lambda hs: list(dict.fromkeys(hs))  # noqa: E731  (one entry per writer and reader)
    return dedup(sgpr_hazards), dedup(m0_hazards)


def open_dma_statements(asm: str) -> List[List[str]]:
    """Inline-asm statements whose first LDS DMA with a scalar base comes before the statement has waited out a
    vector-ALU write of that base: whatever register restore the compiler puts before such a statement is a hazard."""
    bad = []
    for body in re.findall(r";+#?\s*ASMSTART\n(.*?);+#?\s*ASMEND", asm, re.S):
        lines = [t for t in (raw.split(";")[0].strip() for raw in body.splitlines()) if t]
        waits = 0
        for line in lines:
            if "_lds_" in line.split()[0] and any("s" in r for r in _sgprs(" ".join(_operands(line)[1:]))):
                if waits < VALU_SGPR_WAITS:
                    bad.append(lines)
                break
            waits += _waits_of(line)
    return bad


def _vgprs(text: str) -> Set[int]:
    regs = set()
    for m in re.finditer(r"\bv\[(\d+):(\d+)\]", text):
        regs.update(range(int(m.group(1)), int(m.group(2)) + 1))
    regs.update(int(m.group(1)) for m in re.finditer(r"\bv(\d+)\b", text))
    return regs


def _valu_dests(line: str) -> Set[int]:
    op = line.split()[0]
    if not op.startswith("v_") or op.startswith(("v_cmp", "v_readfirstlane", "v_readlane")):
        return set()
    ops = _operands(line)
    both = op.startswith("v_swap") or ("permlane" in op and "swap" in op)
    return _vgprs(" ".join(ops[: 2 if both else 1]))


def find_lane_read_hazards(asm: str):
    found = []
    for fn in functions(asm):
        for b, ins in enumerate(fn.blocks):
            for i, line in enumerate(ins):
                if not line.startswith(("v_readfirstlane_b32", "v_readlane_b32")):
                    continue
                reads = _vgprs(_operands(line)[1])
                before, stack, seen = [], [(b, i)], set()
                while stack:  # the instruction before, on every path
                    blk, at = stack.pop()
                    if at > 0:
                        before.append(fn.blocks[blk][at - 1])
                        continue
                    for p in fn.preds[blk]:
                        if p not in seen:
                            seen.add(p)
                            stack.append((p, len(fn.blocks[p])))
                found += [(fn.name, w, line) for w in before if _valu_dests(w) & reads]
    return list(dict.fromkeys(found))
