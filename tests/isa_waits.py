"""Follows the outstanding memory requests of a kernel through its assembly (gfx950, as the compiler prints it): which
registers may still be waiting for their load, on any path, at every instruction.

Requests of one counter are answered in the order they were issued, so a load has arrived behind `s_waitcnt vmcnt(n)`
exactly when at least n requests were issued after it.  The state at an instruction is, for every register with a load that
may be outstanding, the least number of such later requests over the paths that lead there; vmcnt counts global, buffer
and scratch accesses (stores and loads into LDS among them), lgkmcnt those of LDS.  Scalar loads also count in lgkmcnt;
they can only make a wait longer, so they are left out.

Paths that cannot be taken are told apart as far as two things go: scalar registers that hold a small constant and are
compared with one (a position in a ring that is entered in the middle), and, up to the first barrier, scalar pairs of all ones or
zero that are branched on more than once.  States that differ in these are kept apart, all others are merged."""
import heapq
import re

_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_SREG = re.compile(r"^s(?:\[(\d+):(\d+)\]|(\d+))$")
_WAIT = re.compile(r"(vmcnt|lgkmcnt)\((\d+)\)")
_MANY = 64  # above every count an s_waitcnt can name


def registers(text):
    out = set()
    for kind, lo, hi, one in _REG.findall(text):
        first, last = (int(lo), int(hi)) if lo else (int(one), int(one))
        out.update((kind, n) for n in range(first, last + 1))
    return frozenset(out)


def scalars(operand):
    m = _SREG.match(operand)
    if not m:
        return range(0)
    return range(int(m[3]), int(m[3]) + 1) if m[3] else range(int(m[1]), int(m[2]) + 1)


class Instruction:
    def __init__(self, line, text, in_asm):
        self.line, self.text, self.in_asm = line, text, in_asm
        self.op, _, rest = text.partition(" ")
        op = self.op
        self.operands = [o.strip() for o in rest.split(",")]
        self.regs = registers(rest)
        self.queue, self.dest, self.waits, self.target, self.ends = None, frozenset(), (), None, False
        if op == "s_waitcnt":
            self.waits = tuple((k, int(n)) for k, n in _WAIT.findall(rest))
        elif op.startswith(("global_", "buffer_", "scratch_")) and not op.startswith(("buffer_wbl2", "buffer_inv")):
            self.queue = "vmcnt"
            to_lds = "_load_lds_" in op or re.search(r"\blds\b", rest)
            if ("_load_" in op and not to_lds) or ("atomic" in op and re.search(r"\bsc0\b", rest)):
                self.dest = registers(self.operands[0])
        elif op.startswith("ds_") and op != "ds_nop":
            self.queue = "lgkmcnt"
            if op.startswith(("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle", "ds_consume", "ds_append")) or "_rtn_" in op:
                self.dest = registers(self.operands[0])
        elif op.startswith(("s_branch", "s_cbranch")):
            self.target, self.ends = self.operands[0], op == "s_branch"
        elif op in ("s_endpgm", "s_setpc_b64"):
            self.ends = True


def kernels(assembly):
    """{kernel name: (instructions, {label: index of the instruction it stands before})}"""
    found, name, in_asm = {}, None, False
    names = set(re.findall(r"^\s*\.amdhsa_kernel\s+(\S+)", assembly, flags=re.M))
    for number, raw in enumerate(assembly.splitlines(), 1):
        if "ASMSTART" in raw or "ASMEND" in raw:
            in_asm = "ASMSTART" in raw
            continue
        text = raw.split(";")[0].split("//")[0].strip().replace("\t", " ")
        if not text:
            continue
        if text.endswith(":"):
            if text[:-1] in names:
                name = text[:-1]
                found[name] = ([], {})
            elif text.startswith(".Lfunc_end"):
                name = None
            elif name:
                found[name][1][text[:-1]] = len(found[name][0])
        elif name and not text.startswith("."):
            found[name][0].append(Instruction(number, text, in_asm))
    return found


def _followed(code):
    """The scalar registers whose value tells paths apart: compared with a constant inside an assembly block, or pairs a
    branch depends on; with those they are copied from."""
    keep = {i.operands[0] for i in code if i.in_asm and i.op in ("s_cmp_lt_u32", "s_cmp_eq_u32") and i.operands[1].isdigit()
            and i.operands[1] != "0"}
    tested = [i.operands[2] for i in code if i.op in ("s_and_b64", "s_andn2_b64") and i.operands[:2] == ["vcc", "exec"]]
    fixed = {i.operands[0] for i in code if i.op == "s_mov_b64" and i.operands[1] in ("0", "-1")}
    keep |= {r for r in tested if tested.count(r) > 1 or r in fixed}
    grown = True
    while grown:
        grown = False
        for i in code:
            if i.op in ("s_mov_b32", "s_mov_b64") and i.operands[0] in keep and _SREG.match(i.operands[1]) and i.operands[1] not in keep:
                keep.add(i.operands[1])
                grown = True
    return keep


def _step(ins, known, keep, flags):
    """What is known of the scalar registers behind an instruction; flags: what the last compare and vcc depend on."""
    o = ins.operands
    if ins.op == "s_barrier":  # (the pairs are let go here: fewer states to follow)
        return {**{r: v for r, v in known.items() if "[" not in r}, "late": 1}
    if ins.op in ("s_cmp_lt_u32", "s_cmp_eq_u32") and len(o) == 2 and o[1].isdigit():
        flags["scc"] = (ins.op, o[0], int(o[1]))
        return known
    if ins.op.startswith("s_cmp") or (ins.op.startswith("s_") and ins.op.split("_")[1] in (
            "add", "sub", "and", "andn2", "or", "orn2", "xor", "lshl", "lshr", "ashr", "bfe", "min", "max", "abs", "not", "addc", "subb", "bitcmp0",
            "bitcmp1", "lshl1", "lshl2", "lshl3", "lshl4")):
        flags["scc"] = None
    if o[0] == "exec" or "saveexec" in ins.op:
        flags["exec"] = True
    if o[0] == "vcc":
        flags["vcc"] = (ins.op, o[2]) if ins.op in ("s_and_b64", "s_andn2_b64") and o[1] == "exec" else None
        return known
    if ins.op.startswith("v_cmp") and "_e32" in ins.op:
        flags["vcc"] = None
    hit = scalars(o[0])
    if len(hit) and not ins.queue and ins.op not in ("s_cbranch", "s_branch") and not ins.op.startswith("s_cmp"):
        gone = set(hit)
        value = None
        if o[0] in keep and not ("late" in known and "[" in o[0]) and ins.op in ("s_mov_b32", "s_mov_b64"):
            value = known.get(o[1], int(o[1]) if re.match(r"^-?\d+$", o[1]) else None)
        if any(gone & set(scalars(r)) for r in known) or value is not None:
            known = {r: v for r, v in known.items() if not gone & set(scalars(r))}
            if value is not None:
                known[o[0]] = value
    return known


def _branch(ins, known, keep, flags):
    """[(taken, what is known then)] of the ways out of a conditional branch that are possible."""
    both = [(True, known), (False, known)]
    if ins.op in ("s_cbranch_execz", "s_cbranch_execnz") and not flags.get("exec"):
        return [(ins.op == "s_cbranch_execnz", known)]  # (a uniform branch the compiler could decide: some lane is active)
    if ins.op in ("s_cbranch_scc0", "s_cbranch_scc1") and flags.get("scc"):
        op, reg, n = flags["scc"]
        if reg in known:
            truth = known[reg] < n if op == "s_cmp_lt_u32" else known[reg] == n
            return [(truth == (ins.op == "s_cbranch_scc1"), known)]
    if ins.op in ("s_cbranch_vccz", "s_cbranch_vccnz") and flags.get("vcc"):
        op, reg = flags["vcc"]
        if reg in keep and "late" not in known:
            ways = []
            for value in (-1, 0):
                if known.get(reg, value) == value:
                    nonzero = (value == -1) == (op == "s_and_b64")
                    ways.append((nonzero == (ins.op == "s_cbranch_vccnz"), {**known, reg: value}))
            return ways
    return both


def early_uses(code, labels):
    """[(line, instruction, registers)] of the instructions that name a register whose load may not have arrived."""
    keep = _followed(code)
    starts = sorted({0, *labels.values(), *(i + 1 for i, ins in enumerate(code) if ins.target or ins.ends)})
    ends = dict(zip(starts, starts[1:] + [len(code)]))
    before = {(0, ()): {}}
    todo, queued, bad = [(0, ())], {(0, ())}, {}
    while todo:  # in the order of the code, so that most blocks see all that leads to them at once
        at, facts = heapq.heappop(todo)
        queued.discard((at, facts))
        # inside a block: register -> (counter, number of the request), and how many each counter has issued
        issued, known, flags, following = {"vmcnt": 0, "lgkmcnt": 0}, dict(facts), {}, []
        waiting = {r: (c, -1 - later) for r, (c, later) in before[at, facts].items()}
        for i in range(at, ends.get(at, at)):
            ins = code[i]
            for counter, n in ins.waits:
                waiting = {r: q for r, q in waiting.items() if q[0] != counter or issued[counter] - q[1] - 1 < n}
            if waiting and not ins.regs.isdisjoint(waiting):
                # (a load over an earlier one of the same counter arrives behind it)
                early = sorted(r for r in ins.regs & waiting.keys() if r not in ins.dest or waiting[r][0] != ins.queue)
                if early:
                    bad[ins.line] = (ins.line, ins.text, early)
            assert not ins.op.startswith("flat_"), f"line {ins.line}: {ins.text}: flat accesses are not answered in order"
            if ins.queue:
                for r in ins.dest:
                    waiting[r] = (ins.queue, issued[ins.queue])
                issued[ins.queue] += 1
            if ins.target and not ins.ends:
                ways = _branch(ins, known, keep, flags)
                following += [(labels[ins.target] if taken else i + 1, k) for taken, k in ways]
                break
            if ins.ends:
                if ins.target:
                    following.append((labels[ins.target], known))
                break
            known = _step(ins, known, keep, flags)
        else:
            following.append((ends.get(at, len(code)), known))
        state = {r: (c, min(issued[c] - number - 1, _MANY)) for r, (c, number) in waiting.items()}
        for to, k in following:
            if to >= len(code):
                continue
            key = (to, tuple(sorted(k.items())))
            old = before.get(key)
            merged = dict(state if old is None else old)
            for r, q in state.items():
                if r not in merged or q[1] < merged[r][1]:
                    merged[r] = q
            if merged != old:
                before[key] = merged
                if key not in queued:
                    queued.add(key)
                    heapq.heappush(todo, key)
    return sorted(bad.values())
