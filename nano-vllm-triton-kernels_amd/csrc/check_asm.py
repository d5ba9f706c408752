"""Checks the assembly of kernels that use matrix or memory instructions in inline asm.

The compiler keeps its own instructions at the distances that the hardware asks for, but does not look into asm statements:
an operand that it copies, spills or reloads right beside one would be read too early, without a message. Of the named
kernels (substrings of the symbols) the build therefore checks, along every path:

  - a matrix instruction's result is touched by any other instruction, but for the accumulation of the next matrix
    instruction into the same registers, only `passes + 4` wait states later;
  - a vector instruction's result is read by a matrix instruction at least 2 wait states later;
  - a scalar register that a vector instruction wrote (a spilled one that comes back, for instance) is read by a memory
    instruction at least 5 wait states later, unless a scalar instruction has written it since;
  - m0 is written at least one wait state before a load into LDS;
  - the kernel uses no scratch memory (spilled vector registers).

One instruction is one wait state, s_nop n is n + 1.

usage: check_asm.py FILE.s KERNEL...
"""
import re
import sys

PASSES = {"v_mfma_f32_32x32x16_bf16": 8, "v_mfma_f32_16x16x32_bf16": 4}  # of 4 clocks
_REG = re.compile(r"\b([vas])(?:(\d+)|\[(\d+):(\d+)\])|\b(vcc|m0)\b")
_MEMORY = ("global_", "buffer_", "flat_", "scratch_", "ds_")
_NO_RESULT = ("v_cmpx", "v_nop")


def registers(operand):
    """The registers of an operand as a set of names (v0, a17, s4, vcc, m0)."""
    out = set()
    for kind, one, lo, hi, special in _REG.findall(operand):
        if special:
            out.add(special)
        elif one:
            out.add(kind + one)
        else:
            out.update(f"{kind}{i}" for i in range(int(lo), int(hi) + 1))
    return out


class Instruction:
    """name, the registers it writes and reads, its wait states and where control goes after it."""

    def __init__(self, text):
        self.text = text
        self.name, _, rest = text.partition(" ")
        operands = [o.strip() for o in rest.split(",")] if rest else []
        self.mfma = self.name.startswith("v_mfma")
        self.vector = self.name.startswith("v_") and not self.mfma
        self.memory = self.name.startswith(_MEMORY)
        self.states = int(operands[0], 0) + 1 if self.name == "s_nop" else 1
        regs = [registers(o) for o in operands]
        # results: the first operand, of a store or a load into LDS none, of a carry or a swap the second too
        results = 1
        if self.name.startswith(_NO_RESULT) or "store" in self.name or "_load_lds" in self.name or "ds_write" in self.name:
            results = 0
        elif self.name.startswith(("s_cmp", "s_cbranch", "s_branch", "s_waitcnt", "s_barrier", "s_nop", "s_endpgm",
                                   "s_setprio", "s_sleep")) or (self.name.startswith("buffer_load") and "lds" in text):
            results = 0
        elif "swap" in self.name or (len(regs) > 3 and re.search(r"_co_|v_div_scale|v_mad_[iu]64", self.name)):
            results = 2
        self.writes = set().union(*regs[:results]) if regs else set()
        self.reads = set().union(*regs[results:]) if regs else set()
        if "swap" in self.name or self.name.startswith(("v_writelane", "v_fmac", "v_cmpx")):
            self.reads |= self.writes  # read and written
        if self.name.startswith("v_cmp") and "_e32" in self.name:
            self.writes, self.reads = {"vcc"}, set().union(*regs) - {"vcc"}
        self.to_lds = self.memory and "lds" in text and not self.name.startswith("ds_")
        if self.mfma:
            self.d, self.a, self.b, self.c = regs[:4]
            self.passes = PASSES[self.name]
        target = re.match(r"s_c?branch\S*\s+(\S+)", text)
        self.target = target.group(1) if target else None
        self.ends = self.name in ("s_branch", "s_endpgm", "s_setpc_b64")


def parse(lines):
    code, labels = [], {}
    for line in lines:
        line = line.split(";")[0].split("//")[0].strip()
        label = re.match(r"([.\w$]+):$", line)
        if label:
            labels[label.group(1)] = len(code)
        elif line and not line.startswith("."):
            code.append(Instruction(re.sub(r"\s+", " ", line)))
    return code, labels


def needed(first, scalars, then):
    """Wait states that `then` has to keep from `first` (scalars: the scalar registers that still hold its results), and
    why (0: none)."""
    if first.mfma:
        if then.mfma:
            if then.c == first.d and then.d == first.d and not (first.d & (then.a | then.b)):
                return 0, ""
            if first.d & (then.a | then.b | then.c | then.d):
                return first.passes + 4, "matrix result used by another matrix instruction"
        elif first.d & (then.reads | then.writes):
            return first.passes + 4, "matrix result used"
    elif first.vector:
        if then.mfma and first.writes & (then.a | then.b | then.c):
            return 2, "vector result read by a matrix instruction"
        if then.memory and scalars & (then.reads | then.writes):
            return 5, "scalar register written by a vector instruction read by a memory instruction"
    elif "m0" in first.writes and then.to_lds:
        return 1, "m0 written right before a load into LDS"
    return 0, ""


def hazards(code, labels):
    found = []
    for i, first in enumerate(code):
        reach = first.passes + 4 if first.mfma else 5 if first.vector else 1 if "m0" in first.writes else 0
        if reach == 0:
            continue
        todo, seen = [], set()

        def follow(j, instruction, waited, scalars):
            if instruction.name.startswith("s_"):
                scalars = scalars - instruction.writes
            if instruction.target is not None and instruction.target in labels:
                todo.append((labels[instruction.target], waited, scalars))
            if not instruction.ends and j + 1 < len(code):
                todo.append((j + 1, waited, scalars))
        follow(i, first, 0, frozenset(r for r in first.writes if r[0] == "s" or r == "vcc") if first.vector else frozenset())
        while todo:
            state = j, waited, scalars = todo.pop()
            if waited >= reach or state in seen:
                continue
            seen.add(state)
            least, why = needed(first, scalars, code[j])
            if waited < least:
                found.append(f"{why} after {waited} of {least} wait states: {first.text} -> {code[j].text}")
            follow(j, code[j], waited + code[j].states, scalars)
    return found


def functions(text):
    """Name -> lines of every function of an assembly file, and name -> bytes of scratch of every kernel."""
    bodies, name = {}, None
    for line in text.splitlines():
        kind = re.match(r"\s*\.type\s+(\S+),@function", line)
        if kind:
            name = kind.group(1)
            bodies[name] = []
        elif name and re.match(r"\s*\.(Lfunc_end|section|size)", line):
            name = None
        elif name:
            bodies[name].append(line)
    scratch = {}
    for block in re.split(r"\n\s*- \.a", text)[1:]:
        symbol, size = re.search(r"\.name:\s+(\S+)", block), re.search(r"\.private_segment_fixed_size:\s+(\d+)", block)
        if symbol and size:
            scratch[symbol.group(1)] = int(size.group(1))
    return bodies, scratch


def check(text, kernels):
    """Messages of what is wrong with the kernels whose symbols hold one of these names."""
    bodies, scratch = functions(text)
    messages = []
    for wanted in kernels:
        names = [n for n in bodies if wanted in n and n in scratch]
        if not names:
            messages.append(f"no kernel {wanted}")
        for n in names:
            if scratch[n]:
                messages.append(f"{n}: {scratch[n]} bytes of scratch")
            messages += [f"{n}: {h}" for h in hazards(*parse(bodies[n]))]
    return messages


if __name__ == "__main__":
    with open(sys.argv[1]) as f:
        problems = check(f.read(), sys.argv[2:])
    for p in problems:
        print(p, file=sys.stderr)
    sys.exit(1 if problems else 0)
