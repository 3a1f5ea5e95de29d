"""Checks the machine code of kernels whose MFMAs are placed by hand (opaque instructions that the compiler neither
schedules nor guards): build.py runs it on every build and refuses code that breaks one of the rules.

1. Accumulation registers 0 .. OWNED-1 hold the kernel's sums and resident operands by number: besides MFMAs, one write at
   the start and one read at the end, no instruction may touch them.
2. Two instructions lie between a vector instruction that writes an operand of an MFMA and that MFMA.
3. What an MFMA writes to vector registers is read, or overwritten by something else, no sooner than two further MFMAs or
   twenty instructions later.
Branches are ignored: instructions are taken in the order they stand in.
"""
import os
import re
import subprocess
import tempfile

OWNED = 192
_REG = re.compile(r"\b([va])(\d+)\b|\b([va])\[(\d+):(\d+)\]")
_STORES = ("ds_write", "global_store", "scratch_store", "buffer_store", "global_load_lds")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        if m.group(1):
            out.add((m.group(1), int(m.group(2))))
        else:
            out.update((m.group(3), x) for x in range(int(m.group(4)), int(m.group(5)) + 1))
    return out


def violations(lines, kernels):
    """Rule breaks in a disassembly (an iterable of lines) of the functions whose name holds `kernels`."""
    bad, on, name = [], False, ""
    for line in lines:
        m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if m:
            name, on = m.group(1), kernels in m.group(1)
            recent, tiles, writes, reads, at, mfmas = [], {}, set(), set(), 0, 0
            continue
        text = line.split("//")[0].strip()
        if not on or not text or not re.match(r"[a-z]+_", text):
            continue
        op = text.split()[0]
        args = text[len(op):].split(",")
        store, mfma = op.startswith(_STORES), op.startswith("v_mfma")
        dst = set() if store or op.startswith("s_") else _regs(args[0])
        src = _regs(",".join(args)) if store else _regs(",".join(args[1:]))
        own = {r for r in dst | src if r[0] == "a" and r[1] < OWNED}
        if own and not mfma:
            seen = writes if op == "v_accvgpr_write_b32" else reads if op == "v_accvgpr_read_b32" else None
            if seen is None or own & seen:
                bad.append((1, name, text))
            else:
                seen |= own
        if mfma:
            if any(w & src for o, w in recent[-2:] if o.startswith("v_") and not o.startswith("v_mfma")):
                bad.append((2, name, text))
        elif not op.startswith("s_"):
            if any(at - a < 20 and mfmas - k < 2 and tile & (dst | src) for tile, (a, k) in tiles.items()):
                bad.append((3, name, text))
        at += 1
        if mfma:
            mfmas += 1
            tiles = {t: v for t, v in tiles.items() if not t & dst}
            if any(r[0] == "v" for r in dst):
                tiles[frozenset(dst)] = (at, mfmas)
        if op == "s_nop":
            recent += [("s_nop", set())] * (int(args[0]) + 1)
        else:
            recent.append((op, dst))
        recent = recent[-3:]
    return bad


def check_object(obj, kernels, llvm="/opt/rocm/llvm/bin"):
    """Disassembles the gfx950 code of an object file built here; raises where a rule is broken."""
    with tempfile.TemporaryDirectory() as tmp:
        link = os.path.join(tmp, "x.o")
        os.symlink(os.path.abspath(obj), link)
        subprocess.run([os.path.join(llvm, "llvm-objdump"), "--offloading", link], check=True, capture_output=True)
        code = [f for f in os.listdir(tmp) if f.endswith("gfx950")]
        if len(code) != 1:
            raise RuntimeError("no gfx950 code in %s" % obj)
        res = subprocess.run([os.path.join(llvm, "llvm-objdump"), "-d", os.path.join(tmp, code[0])], check=True,
                             capture_output=True, text=True)
    lines = res.stdout.splitlines()
    found = sum(1 for l in lines if l.endswith(">:") and kernels in l)
    if not found:
        raise RuntimeError("%s: no kernel %s" % (obj, kernels))
    bad = violations(lines, kernels)
    if bad:
        raise RuntimeError("%s: hand-placed MFMAs are not safe as compiled (rule, kernel, instruction): %s" % (obj, bad[:4]))
    return found
