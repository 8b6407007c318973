"""A look over a gfx950 assembly listing: inline assembly that writes EXEC stands only where all 64 lanes are on.

kq_raise and its like (csrc/rpeg_kernel_quad.h) and the dispatch of kp_lanes (csrc/rpeg_kernel_sched.h) set EXEC to a mask and then to
-1.  Behind a branch that some lanes did not take that would switch these on.  The compiler does not know that they write it: it keeps
them out of such a branch because all inline assembly is convergent, and the source has to keep them out of one of its own.

What is followed, from the entry of a function through every path: sets of registers ("covers") that together hold every lane, as
branches and loops take lanes out of EXEC and bring them back.  All lanes are on where EXEC alone is one.  A kernel's wavefronts
start whole (its blocks are multiples of 64 threads), a function's where they are at every call of it."""

import re

MOST = 48      # covers that are kept (fewer: less is known)


def _names(operand: str) -> set:
    """The 32-bit registers of an operand; of EXEC and VCC both halves have one name."""
    m = re.fullmatch(r"([sv])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    if m:
        return {f"{m.group(1)}{n}" for n in range(int(m.group(2) or m.group(4)), int(m.group(3) or m.group(4)) + 1)}
    return {x for x in ("exec", "vcc") if operand.startswith(x)}


def _half(operand: str, half: int) -> str:
    m = re.fullmatch(r"s\[(\d+):\d+\]", operand)
    return f"s{int(m.group(1)) + half}" if m else operand


def _least(covers):
    """Without those that hold another."""
    kept = []
    for c in sorted(covers, key=lambda c: (len(c), sorted(c))):
        if len(c) <= 5 and not any(x <= c for x in kept):
            kept.append(c)
    return frozenset(kept[:MOST])


def _after(op: str, a: list, covers, half: int):
    """The covers behind an instruction of operands `a`.  (A call gives EXEC back as it was; of the registers that it does not, the
    compiler reads none behind it that it has not written again.)"""
    if not a or op[0] not in "svdgb" or op.startswith(("s_cmp", "s_bitcmp", "s_waitcnt", "s_nop")):
        return covers
    to, saves, new = _half(a[0], half), op.endswith("saveexec_b64"), set()
    written = _names(a[0])
    if saves or op.startswith("v_cmpx"):
        written = written | {"exec"}
    if len(a) > 1 and re.match(r"v_\w*(_co_|div_scale|mad_[ui]64)", op):
        written = written | _names(a[1])
    if op == "v_writelane_b32":
        to = f"{a[0]}.{a[2]}"
        written = {to}

    def gone(x):
        return x in written or x.split(".")[0] in written

    def held(old, by, grows=False):      # what `old` held is held by the registers `by`
        for c in covers:
            rest = c - {old}
            if saves:                    # (EXEC as it was is in `to`)
                stale = to in rest
                rest = {to if x == "exec" else x for x in rest}
            else:
                stale = any(gone(x) for x in rest) and not grows
            if old in c and not stale:
                new.add(frozenset(rest) | frozenset(by))

    a = [_half(x, half) for x in a]
    if op == "s_mov_b64" and a[1] == "-1":
        new.add(frozenset({to}))
    elif op == "s_mov_b64" or (op == "s_mov_b32" and a[1][0] == "s"):
        held(a[1], {to})
    elif op == "v_writelane_b32":        # (what finds no register lies in the lanes of one)
        held(a[1], {to})
    elif op == "v_readlane_b32":
        held(f"{a[1]}.{a[2]}", {to})
    elif op == "s_or_b64":
        held(a[1], {to}, grows=to == a[2])
        held(a[2], {to}, grows=to == a[1])
    elif op in ("s_andn2_b64", "s_xor_b64"):     # (the result and the second operand hold all of the first)
        if a[2] != to:
            held(a[1], {to, a[2]})
        if op == "s_xor_b64" and a[1] != to:
            held(a[2], {to, a[1]})
    elif saves:
        held("exec", {to})
        if op == "s_or_saveexec_b64":
            held("exec", {"exec"})
            held(a[1], {"exec"})
        elif op == "s_andn2_saveexec_b64":
            held(a[1], {to, "exec"})
    return _least(new | {c for c in covers if not any(gone(x) for x in c)})


def _split(line: str):
    op, _, rest = line.replace("\t", " ").partition(" ")
    return op, [x.strip() for x in rest.split(",")] if rest.strip() else []


def _flow(lines: list, whole: bool, half: int):
    """The covers ahead of every line that is reached; None where a jump goes to an address."""
    at = {m.group(1): i for i, m in enumerate(re.match(r"(\.\w+):", line) for line in lines) if m}
    known, todo = {}, [(0, frozenset({frozenset({"exec"})} if whole else ()))]
    while todo:
        i, covers = todo.pop()
        while i < len(lines):
            if i in known:
                covers = _least({x | y for x in known[i] for y in covers})
                if covers == known[i]:
                    break
            known[i] = covers
            op, a = _split(lines[i])
            if op == "s_endpgm" or (op == "s_setpc_b64" and a == ["s[30:31]"]):
                break
            if op == "s_setpc_b64":
                return None
            if op == "s_branch":
                i = at[a[0]]
                continue
            if op.startswith("s_cbranch"):
                todo.append((at[a[0]], covers))
            elif op:
                covers = _after(op, a, covers, half)
            i += 1
    return known


def _called(lines: list, i: int):
    """The function that the call in line i goes to, whose address is put together ahead of it; None if that is not seen."""
    low = re.match(r"s\[(\d+):", _split(lines[i])[1][1])
    for line in reversed(lines[:i]):
        op, a = _split(line)
        if op.startswith("s_add_u32") and low and a[0] == "s" + low.group(1):
            m = re.match(r"([\w.$]+)@rel32@lo", a[2])
            return m.group(1) if m else None
        if re.match(r"\.\w+:", line):
            return None
    return None


def exec_set_under_a_mask(asm: str) -> list:
    """(function, instruction) for inline assembly that writes EXEC where it is not certain that all lanes are on ahead of it and
    behind it."""
    kernels = set(re.findall(r"\.amdhsa_kernel\s+(\S+)", asm))
    if not kernels:
        raise RuntimeError("no kernel in the assembly listing")
    body, name = {}, None
    for line in asm.splitlines():
        label = re.match(r"([A-Za-z_][\w.$]*):", line)
        if label:
            name = label.group(1)
            body[name] = []
        elif name:
            body[name].append(line.strip() if "#ASM" in line else line.split(";")[0].strip())
    flows = {}

    def flow(f):
        if f not in flows:
            whole = f in kernels or called_whole(f)
            both = [_flow(body[f], whole, half) for half in (0, 1)]
            flows[f] = set() if None in both else {i for i in both[0] if all(frozenset({"exec"}) in x.get(i, ()) for x in both)}
        return flows[f]

    def called_whole(f):
        flows[f] = set()      # (no function calls itself)
        calls = 0
        for g, lines in body.items():
            for i, line in enumerate(lines):
                if line.startswith("s_swappc") and (to := _called(lines, i)) in (f, None):
                    calls += to == f
                    if i not in flow(g):
                        return False
        return calls == asm.count(f + "@rel32@lo")      # (its address goes nowhere else)

    found = []
    for f, lines in body.items():
        blocks, start, writes = [], 0, False
        for i, line in enumerate(lines):
            if line.endswith("#ASMSTART"):
                start, writes = i, False
            elif line.endswith("#ASMEND"):
                blocks += [(start, i)] if writes else []
            elif re.match(r"(s_\S+|v_readlane_b32|v_readfirstlane_b32)\s+exec|s_\w+saveexec|v_cmpx", line):
                writes = True
        if blocks:
            found += [(f, lines[start + 1]) for start, end in blocks if not {start, end} <= flow(f)]
    return found
