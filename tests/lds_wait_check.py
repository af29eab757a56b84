"""Checks compiled gfx950 assembly for LDS loads whose results are used
before they have arrived.

The pipelined prefill GEMM issues some LDS reads as inline asm (the
compiler cannot tell its DMA ring slots apart and would otherwise wait for
every DMA in flight before each read).  The compiler does not know such an
asm result is still in flight, so it must not copy, read or overwrite the
destination registers before the s_waitcnt lgkmcnt that retires the load.
This follows every path through each function whose name matches a pattern
(reads may be in flight over a loop's back edge, where the compiler may place
the copies of a rotated loop) and reports any instruction that touches the
VGPRs of a pending ds_read.  LDS operations retire in issue order, so
lgkmcnt(n) leaves at most the newest n of them; scalar loads, which share the
counter and return in any order, are taken as returned already.

usage: python tests/lds_wait_check.py file.s [name-substring]
"""
import re
import sys


def _regs(tok):
    m = re.fullmatch(r"[va]\[(\d+):(\d+)\]", tok)
    if m:
        pre = tok[0]
        return frozenset((pre, i) for i in range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"([va])(\d+)", tok)
    if m:
        return frozenset({(m.group(1), int(m.group(2)))})
    return frozenset()


def _parse(lines):
    """([(line number, text, op, operands)], {label: index of the instruction after it})."""
    ins, labels = [], {}
    for ln, raw in lines:
        t = raw.split(";")[0].strip()
        m = re.match(r"([.\w$]+):\s*(.*)", t)
        if m:
            labels[m.group(1)] = len(ins)
            t = m.group(2)
        if not t or t.startswith("."):
            continue
        op, _, rest = t.partition(" ")
        ins.append((ln, t, op, [o.strip().split()[0] for o in rest.split(",") if o.strip()]))
    return ins, labels


def check_function(lines):
    """Returns the list of (line number, text) hazards in one function."""
    ins, labels = _parse(lines)
    bad = {}
    work, seen = [(0, ())], set()                       # (instruction, pending loads, oldest first)
    while work:
        i, pend = work.pop()
        while i < len(ins):
            ln, t, op, ops = ins[i]
            i += 1
            if op == "s_endpgm":
                break
            if op in ("s_setpc_b64", "s_swappc_b64", "s_call_b64"):
                bad[ln] = t + " (a jump that is not followed)"
                break
            if op == "s_branch" or op.startswith("s_cbranch"):
                target = labels.get(ops[-1])
                if target is None:
                    bad[ln] = t + " (unknown label)"
                    break
                # both ways are joints, so that every loop meets a state it has seen
                for nxt in (target,) if op == "s_branch" else (target, i):
                    if (nxt, pend) not in seen:
                        seen.add((nxt, pend))
                        work.append((nxt, pend))
                break
            if op == "s_waitcnt":
                m = re.search(r"lgkmcnt\((\d+)\)", t)
                if m:
                    n = int(m.group(1))
                    pend = pend[max(0, len(pend) - n):] if n else ()
                continue
            if op.startswith("s_"):
                continue
            touched = frozenset().union(*map(_regs, ops))
            if any(touched & p for p in pend):
                bad[ln] = t
            if op.startswith("ds_"):
                pend += (_regs(ops[0]) if op.startswith("ds_read") and ops else frozenset(),)
                pend = pend[-64:]                       # (the counter stalls the wave long before that)
    return sorted(bad.items())


def check_file(path, pattern=""):
    """{function name: hazards} for the functions whose name contains pattern."""
    funcs, cur = {}, None
    for i, line in enumerate(open(path).read().splitlines(), 1):
        m = re.match(r"^(_Z\w+):", line)
        if m:
            cur = m.group(1)
            funcs[cur] = []
            continue
        if line.startswith(".Lfunc_end"):
            cur = None
        if cur is not None:
            funcs[cur].append((i, line))
    return {f: check_function(ls) for f, ls in funcs.items() if pattern in f}


if __name__ == "__main__":
    res = check_file(sys.argv[1], sys.argv[2] if len(sys.argv) > 2 else "")
    n = 0
    for f, bad in res.items():
        for ln, t in bad:
            print(f"{f}:{ln}: {t}")
        n += len(bad)
        print(f"{f}: {'ok' if not bad else str(len(bad)) + ' hazards'}")
    sys.exit(1 if n else 0)
