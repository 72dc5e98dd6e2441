"""The gfx950 code of the built library, read for what the compiler cannot check: inline assembly is opaque
to its hazard recognizer and to its bookkeeping of loads in flight, so these look at every path of the
finished machine code instead."""
import os
import re
import shutil
import subprocess

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"

# Wait states between a VALU instruction that writes a scalar register and a memory instruction that reads it
SCALAR_WAIT = 5

# Wait states between a 32x32x16 MFMA (8 passes) and whatever else touches its result: passes + 4 on gfx950
MFMA_WAIT = 12

MEMORY = ("global_", "buffer_", "scratch_", "flat_")
LOADS = tuple(m + "load" for m in MEMORY)


class Ins:
    __slots__ = ("addr", "op", "args", "target")

    def __init__(self, addr, op, args, target=None):
        self.addr, self.op, self.args, self.target = addr, op, args, target

    def __repr__(self):
        return f"{self.addr:x}: {self.op} {', '.join(self.args)}"


def functions(lib, tmp):
    """{name: [Ins]} of every kernel in the library's code objects (extracted into the folder `tmp`)."""
    shutil.copy(lib, os.path.join(tmp, "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp, check=True, capture_output=True)
    out = {}
    for f in sorted(os.listdir(tmp)):
        if "gfx950" in f:
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp, check=True, capture_output=True, text=True).stdout
            out.update(parse(text))
    return out


def parse(text):
    out, body = {}, None
    for line in text.splitlines():
        m = re.match(r"[0-9a-f]+ <(\S+)>:$", line)
        if m:
            if not m.group(1).startswith("LVX_"):       # a label of a generated loop
                body = out[m.group(1)] = []
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+): ([0-9A-F]+)", line)
        if m is None or body is None:
            continue
        op, args, addr, word = m.groups()
        addr, target = int(addr, 16), None
        if op.startswith(("s_branch", "s_cbranch")):    # a signed distance in words from the next instruction
            target = addr + 4 + 4 * ((int(word, 16) & 0xffff ^ 0x8000) - 0x8000)
        body.append(Ins(addr, re.sub(r"_e(32|64)$", "", op), [a.strip() for a in args.split(",")], target))
    return {n: b for n, b in out.items() if b}


def regs(arg):
    """{(file, number)} of the vector registers an operand names."""
    arg = arg.split(" ")[0].strip("-|")
    m = re.match(r"([va])\[(\d+):(\d+)\]$", arg)
    if m:
        return {(m.group(1), r) for r in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([va])(\d+)$", arg)
    return {(m.group(1), int(m.group(2)))} if m else set()


def touched(ins):
    return set().union(*(regs(a) for a in ins.args)) if ins.args else set()


def after(body, index):
    """Index of an instruction by address, and the successors of instruction i."""
    def successors(i):
        ins = body[i]
        if ins.op == "s_endpgm":
            return []
        nxt = [] if ins.op == "s_branch" else [i + 1]
        if ins.target is not None and ins.target in index:
            nxt.append(index[ins.target])
        return [n for n in nxt if n < len(body)]
    return successors


def mfma_results_touched_early(body):
    """[(mfma, instruction, wait states)]: instructions that read or write an MFMA's result - another MFMA that
    adds to it aside - fewer than MFMA_WAIT wait states behind it on some path."""
    index = {ins.addr: i for i, ins in enumerate(body)}
    successors = after(body, index)
    found = []
    for i, ins in enumerate(body):
        if not ins.op.startswith("v_mfma"):
            continue
        result = regs(ins.args[0])
        best = {}
        todo = [(n, 0) for n in successors(i)]
        while todo:
            j, waited = todo.pop()
            if waited >= MFMA_WAIT or best.get(j, MFMA_WAIT) <= waited:
                continue
            best[j] = waited
            x = body[j]
            if x.op.startswith("v_mfma"):
                if (regs(x.args[1]) | regs(x.args[2])) & result:
                    found.append((ins, x, waited))
                if regs(x.args[0]) == result:       # its own wait is counted from there
                    continue
            elif touched(x) & result:
                found.append((ins, x, waited))
                continue
            step = int(x.args[0], 0) + 1 if x.op == "s_nop" else 1
            todo += [(n, waited + step) for n in successors(j)]
    return found


def to_lds(ins):
    """Is this a load straight to LDS?"""
    return ins.op.startswith(("global_load", "buffer_load", "scratch_load")) and ("_lds_" in ins.op or "lds" in ins.args[-1].split(" "))


def m0_used_early(body):
    """[(write, load)]: loads to LDS with no wait state between them and a scalar write of M0, on some path."""
    successors = after(body, {ins.addr: i for i, ins in enumerate(body)})
    return [(ins, body[j]) for i, ins in enumerate(body) if ins.op.startswith("s_") and ins.args[0] == "m0"
            for j in successors(i) if to_lds(body[j])]


def scalars(arg):
    """Numbers of the scalar registers an operand names ("vcc": that pair)."""
    arg = arg.split(" ")[0]
    m = re.match(r"s\[(\d+):(\d+)\]$", arg) or re.match(r"s(\d+)()$", arg)
    return set(range(int(m.group(1)), int(m.group(2) or m.group(1)) + 1)) if m else {arg} & {"vcc"}


def scalars_used_early(body):
    """[(write, instruction, wait states)]: memory instructions that read a scalar register fewer than SCALAR_WAIT wait
    states behind the VALU instruction that wrote it - a spilled scalar coming back from a lane, mostly -
    on some path."""
    successors = after(body, {ins.addr: i for i, ins in enumerate(body)})
    found = []
    for i, ins in enumerate(body):
        if not ins.op.startswith(("v_readlane", "v_readfirstlane", "v_cmp_")):
            continue
        written = scalars(ins.args[0])
        best = {}
        todo = [(n, 0, written) for n in successors(i)]
        while todo:
            j, waited, left = todo.pop()
            if waited >= SCALAR_WAIT or best.get(j, SCALAR_WAIT) <= waited:
                continue
            best[j] = waited
            x = body[j]
            if x.op.startswith(MEMORY):
                if set().union(*(scalars(a) for a in x.args)) & left:
                    found.append((ins, x, waited))
            elif x.op.startswith("s_"):
                left = left - scalars(x.args[0])        # a scalar write needs no wait
            step = int(x.args[0], 0) + 1 if x.op == "s_nop" else 1
            todo += [(n, waited + step, left) for n in successors(j)]
    return found


def waits_for(ins):
    """How many of the youngest memory operations an instruction leaves in flight; None when it waits for none."""
    m = re.search(r"vmcnt\((\d+)\)", " ".join(ins.args)) if ins.op == "s_waitcnt" else None
    return int(m.group(1)) if m else None


def loads_touched_early(body, stated=()):
    """[(load, instruction)]: instructions that touch the destination of a load to registers on a path that has
    not come by a wait for it yet: what a compiler would do with registers that inline assembly requested, if
    it copied or spilled them.  Operations complete in order, so a wait that leaves n in flight is one for this load
    when at least n were issued behind it.  `stated`: waits that are taken for one whatever the path."""
    index = {ins.addr: i for i, ins in enumerate(body)}
    successors = after(body, index)
    found = []
    for i, ins in enumerate(body):
        if not ins.op.startswith(LOADS) or to_lds(ins):
            continue
        result = regs(ins.args[0])
        fewest = {}                 # operations issued behind the load, on the path that has the fewest
        todo = [(n, 0) for n in successors(i)]
        while todo:
            j, younger = todo.pop()
            if fewest.get(j, younger + 1) <= younger:
                continue
            fewest[j] = younger
            x = body[j]
            left = waits_for(x)
            if left is not None and (left <= younger or x in stated):
                continue
            if touched(x) & result:
                found.append((ins, x))
                continue
            todo += [(n, younger + x.op.startswith(MEMORY)) for n in successors(j)]
    return found
