"""Checks the listings of kernels whose MFMAs are placed by hand (opaque instructions that the compiler neither schedules
nor guards): build.py runs it on every build and refuses code that breaks one of the rules.

1. Accumulation registers 0 .. owned-1 hold the kernel's sums and resident operands by number: no instruction but the
   hand-placed ones (between ASMSTART and ASMEND) may touch them.
2. Two instructions lie between a vector instruction that writes an operand of an MFMA and that MFMA.
3. What an MFMA writes to vector registers is read, or overwritten by something else, no sooner than two further MFMAs or
   twenty instructions later.
4. Only the hand-placed instructions name m0 (they write it, and it is a reserved register that an asm statement cannot declare
   as destroyed).
Branches are ignored: instructions are taken in the order they stand in.
"""
import re

_REG = re.compile(r"\b([va])(\d+)\b|\b([va])\[(\w+):(\w+)\]")
_STORES = ("ds_write", "global_store", "scratch_store", "buffer_store", "global_load_lds")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        if m.group(1):
            out.add((m.group(1), int(m.group(2))))
        else:
            out.update((m.group(3), x) for x in range(int(m.group(4), 0), int(m.group(5), 0) + 1))
    return out


def violations(lines, kernels, owned):
    """Rule breaks in a compiler listing (an iterable of lines) of the functions whose name matches `kernels`, and their number."""
    bad, found, on, hand, name = [], 0, False, False, ""
    for line in lines:
        m = re.match(r"^(_Z\w+|\w+_kernel\w*):", line)
        if m:
            name, on, hand = m.group(1), bool(re.search(kernels, m.group(1))), False
            found += on
            recent, tiles, at, mfmas = [], {}, 0, 0
            continue
        if not on:
            continue
        if "ASMSTART" in line or "ASMEND" in line:
            hand = "ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if not re.match(r"(v|s|ds|global|scratch|buffer|flat)_", text):
            continue
        op = text.split()[0]
        args = text[len(op):].split(",")
        store, mfma = op.startswith(_STORES), op.startswith("v_mfma")
        dst = set() if store or op.startswith("s_") else _regs(args[0])
        src = _regs(",".join(args)) if store else _regs(",".join(args[1:]))
        if not hand and any(r[0] == "a" and r[1] < owned for r in dst | src):
            bad.append((1, name, text))
        if not hand and re.search(r"\bm0\b", text):
            bad.append((4, name, text))
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
            tiles[frozenset(dst)] = (at, mfmas)
        if op == "s_nop":
            at += int(args[0], 0)
            recent += [("s_nop", set())] * (int(args[0], 0) + 1)
        else:
            recent.append((op, dst))
        recent = recent[-3:]
    return bad, found


def check(path, kernels, owned):
    """Raises where the listing at `path` breaks a rule, or holds no such kernel."""
    with open(path) as f:
        bad, found = violations(f, kernels, owned)
    if bad or not found:
        raise RuntimeError("%s: %d kernels %s; hand-placed MFMAs are not safe as compiled (rule, kernel, instruction): %s"
                           % (path, found, kernels, bad[:4]))
