"""Looks over the gfx950 assembly of a source for wait states that the hardware
does not check and that the compiler cannot count inside an inline-assembly
string: the distance, in issued instructions, between a write and a use that
the CDNA3 / CDNA4 instruction set documents ask the program to keep.

  sgpr    a vector-memory instruction reads a scalar register that a vector
          instruction (v_readfirstlane, a compare, ...) wrote: 5
  m0      an LDS-direct load (``lds``, ``global_load_lds_*``) reads m0 that a
          scalar instruction wrote: 1
  dot     a vector instruction reads or overwrites the result of a v_dot*,
          other than the same opcode as accumulator or result: 3
  sdwa    a vector instruction reads what an SDWA instruction wrote to a part
          of a register: 1

An instruction is one wait state, ``s_nop N`` N + 1.  Distances are the least
over all paths (a fixed point over the basic blocks)."""
from __future__ import annotations

import re

NEED = {"sgpr": 5, "m0": 1, "dot": 3, "sdwa": 1}
_REG = re.compile(r"\b([sv])(\d+)\b|\b([sv])\[(\d+):(\d+)\]|\b(vcc|m0)\b")
_VMEM = ("buffer_", "global_", "flat_", "scratch_", "tbuffer_")


def _regs(text: str, kind: str) -> set:
    out = set()
    for one, n, many, lo, hi, named in _REG.findall(text):
        if one == kind:
            out.add(kind + n)
        elif many == kind:
            out.update(f"{kind}{i}" for i in range(int(lo), int(hi) + 1))
        elif named and kind == "s":
            out.add(named)
    return out


class Instruction:
    def __init__(self, line: int, text: str):
        self.line, self.text = line, text
        name, _, rest = text.partition(" ")
        self.name = name
        ops = [o.strip() for o in rest.split(",")]
        valu, self.vmem = name.startswith("v_"), name.startswith(_VMEM)
        self.valu = valu
        self.states = int(rest, 0) + 1 if name == "s_nop" else 1
        self.writes = {}  # register -> the rule its next use falls under
        self.kills = set()
        no_result = name.startswith(("v_nop", "s_nop", "s_waitcnt", "s_barrier"))
        dst = "" if no_result else ops[0]
        n_dst = 2 if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[ui]64", name) else 1
        if valu:
            for r in _regs(" ".join(ops[:n_dst]), "s"):
                self.writes[r] = "sgpr"
            if name.startswith("v_dot"):
                for r in _regs(dst, "v"):
                    self.writes[r] = "dot"
            elif "dst_sel:" in rest and "dst_sel:DWORD" not in rest:
                for r in _regs(dst, "v"):
                    self.writes[r] = "sdwa"
            else:
                self.kills = _regs(dst, "v")
        elif name.startswith("s_") and not no_result:
            self.kills = _regs(dst, "s")
            if "m0" in self.kills:
                self.kills = self.kills - {"m0"}
                self.writes["m0"] = "m0"
        # what is read, by rule
        self.uses = []  # (register, rule)
        if self.vmem:
            self.uses += [(r, "sgpr") for r in _regs(rest, "s")]
            if "_lds_" in name or re.search(r"\blds\b", rest):
                self.uses += [("m0", "m0"), ("m0", "sgpr")]
        if valu:
            src = _regs(rest, "v") if re.search(r"UNUSED_PRESERVE", rest) else _regs(",".join(ops[n_dst:]), "v")
            self.uses += [(r, k) for r in src for k in ("dot", "sdwa")]
            self.uses += [(r, "dot") for r in _regs(dst, "v")]
        self.factors = _regs(",".join(ops[1:3]), "v")  # of a v_dot*: not its accumulator or result


def parse(asm: str):
    """The functions of an assembly text: name -> list of basic blocks
    (label, instructions, successors by label, falls through)."""
    out, name, blocks = {}, None, []
    for line, raw in enumerate(asm.splitlines(), 1):
        text = raw.split(";")[0].split("//")[0].strip()
        if not text:
            continue
        label = re.match(r"([\w.$]+):$", text)
        if label:
            if not label[1].startswith(".L"):
                name, blocks = label[1], []
                out[name] = blocks
            elif label[1].startswith(".Lfunc_end"):
                name = None
            if name is not None:
                blocks.append([label[1], [], [], True])
        elif name is not None and not text.startswith("."):
            if not re.match(r"[a-z]\w+", text):
                continue
            ins = Instruction(line, re.sub(r"\s+", " ", text))
            b = blocks[-1]
            b[1].append(ins)
            if ins.name.startswith(("s_cbranch", "s_branch")):
                b[2].append(ins.text.split(" ")[1])
                b[3] = ins.name != "s_branch"
                blocks.append([f"{b[0]}+{line}", [], [], True])
            elif ins.name in ("s_endpgm", "s_setpc_b64"):
                b[3] = False
    return {k: v for k, v in out.items() if any(b[1] for b in v)}


def _step(state: dict, ins: Instruction, found):
    """state: register, rule -> (wait states since the write, opcode)."""
    for reg, rule in ins.uses:
        got = state.get((reg, rule))
        if got is None or got[0] >= NEED[rule]:
            continue
        if rule == "dot" and got[1] == ins.name and reg not in ins.factors:
            continue
        if found is not None:
            found.append((ins.line, rule, reg, got[0], ins.text))
    for key in [k for k in state]:
        d, op = state[key]
        if d + ins.states >= NEED[key[1]] or key[0] in ins.kills or (key[0] in ins.writes and key[1] != ins.writes[key[0]]):
            del state[key]
        else:
            state[key] = (d + ins.states, op)
    for reg, rule in ins.writes.items():
        state[(reg, rule)] = (0, ins.name)


def violations(asm: str) -> list:
    """(line, rule, register, wait states there are, instruction) of every use
    that comes too soon."""
    out = []
    for blocks in parse(asm).values():
        at = {b[0]: i for i, b in enumerate(blocks)}
        entry = [{} for _ in blocks]
        todo = list(range(len(blocks)))
        while todo:
            i = todo.pop()
            state = dict(entry[i])
            for ins in blocks[i][1]:
                _step(state, ins, None)
            succ = [at[t] for t in blocks[i][2] if t in at]
            if blocks[i][3] and i + 1 < len(blocks):
                succ.append(i + 1)
            for s in succ:
                grew = False
                for k, v in state.items():
                    if k not in entry[s] or v[0] < entry[s][k][0]:
                        entry[s][k] = v
                        grew = True
                if grew:
                    todo.append(s)
        for i, b in enumerate(blocks):
            state = dict(entry[i])
            for ins in b[1]:
                _step(state, ins, out)
    return sorted(set(out))
