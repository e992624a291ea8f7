"""Path analysis of gfx950 assembly (test helper): inline-asm vector loads whose destination registers the
compiler does not know to be in flight must not be touched before an s_waitcnt vmcnt(N) that has at least N
vector-memory instructions issued after the load, on every path: around the innermost loop's back-edge and out
of it (the asm is a function's instruction list; backward branches mark loops)."""
import re

_VMEM = re.compile(r"(global_load|global_store|scratch_|buffer_|global_atomic)")


def _regs(text):
    out = set()
    for m in re.finditer(r"v\[(\d+):(\d+)\]", text):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1))
    for m in re.finditer(r"(?<![\[:\w])v(\d+)(?![\d:\]])", text):
        out.add(int(m.group(1)))
    return out


def function_lines(asm: str, symbol: str):
    """(instruction, inside inline asm) pairs of one function's body."""
    start = asm.index(symbol + ":")
    end = asm.index(".Lfunc_end", start)
    out, in_asm = [], False
    for line in asm[start:end].split("\n"):
        t = line.strip()
        if t.startswith(";;#ASMSTART"):
            in_asm = True
        elif t.startswith(";;#ASMEND"):
            in_asm = False
        elif t and not t.startswith(";"):
            out.append((t, in_asm))
    return out


def unsafe_asm_loads(ins, opcode="global_load_dwordx4"):
    """[(load, reason)] for inline-asm loads of `opcode` touched before they are known complete; also returns
    how many such loads were checked."""
    labels = {t.split(":")[0]: i for i, (t, _) in enumerate(ins) if t.startswith(".LBB")}
    loops = []
    for i, (t, _) in enumerate(ins):
        m = re.match(r"s_(?:cbranch_\w+|branch)\s+(\.LBB\S+)", t)
        if m and labels.get(m.group(1), len(ins)) < i:
            loops.append((labels[m.group(1)], i))

    def scan(order, dst):
        after = 0
        for j in order:
            t, _ = ins[j]
            if t.startswith(".LBB"):
                continue
            if t.startswith("s_waitcnt") and "vmcnt" in t:
                m = re.search(r"vmcnt\((\d+)\)", t)
                if m and after >= int(m.group(1)):
                    return None
                continue
            if _VMEM.match(t):
                after += 1
            if t.startswith("s_"):
                continue
            parts = t.split(None, 1)
            if len(parts) > 1 and _regs(parts[1]) & dst:
                return f"touched at {j}: {t}"
        return None

    bad, n = [], 0
    for i, (t, in_asm) in enumerate(ins):
        if not (in_asm and t.startswith(opcode + " ")):
            continue
        n += 1
        dst = _regs(t.split(",")[0].split(None, 1)[1])
        inner = [lp for lp in loops if lp[0] <= i <= lp[1]]
        paths = [list(range(i + 1, len(ins)))]
        if inner:
            h, b = min(inner, key=lambda x: x[1] - x[0])
            paths.append(list(range(i + 1, b + 1)) + list(range(h, i + 1)))
        for pth in paths:
            r = scan(pth, dst)
            if r:
                bad.append((t, r))
    return bad, n


def _all_regs(text):
    """Vector and accumulation registers named in an instruction's operands."""
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]", text):
        out |= {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    for m in re.finditer(r"(?<![\[:\w])([va])(\d+)(?![\d:\]])", text):
        out.add((m.group(1), int(m.group(2))))
    return out


def _successors(ins):
    labels = {t.split(":")[0]: i for i, (t, _) in enumerate(ins) if re.match(r"\.L\w+:", t)}
    succ = []
    for i, (t, _) in enumerate(ins):
        nxt = [i + 1] if i + 1 < len(ins) else []
        m = re.match(r"s_(cbranch_\w+|branch)\s+(\.L\S+)", t)
        if m:
            succ.append([labels[m.group(2)]] + (nxt if m.group(1) != "branch" else []))
        else:
            assert not re.match(r"s_(setpc|swappc|call)", t), t
            succ.append([] if t.startswith("s_endpgm") else nxt)
    return succ


def early_mfma_reads(ins, states=18):
    """[(mfma, index, touching instruction)]: results of inline-asm MFMAs, whose latency the compiler does not know,
    named by another instruction than an MFMA fewer than `states` wait states after it on some path (an instruction
    counts one, s_nop N one more than N; a 16-pass MFMA's result needs 18 before the VALU or memory reads it)."""
    succ, state, work, bad = _successors(ins), {0: {}}, [0], {}
    while work:
        i = work.pop()
        t, in_asm = ins[i]
        name, _, args = t.partition(" ")
        mfma = name.startswith("v_mfma")
        if not (mfma or name.startswith("s_") or re.match(r"\.L\w+:", t)):
            for r in _all_regs(args) & state[i].keys():
                bad.setdefault((state[i][r][1], i), (ins[state[i][r][1]][0], state[i][r][1], t))
        step = int(args) + 1 if name == "s_nop" else 0 if re.match(r"\.L\w+:", t) else 1
        cur = {r: (n + step, j) for r, (n, j) in state[i].items() if n + step < states}
        if mfma and in_asm:
            cur.update({r: (0, i) for r in _all_regs(args.split(",")[0])})
        for j in succ[i]:
            old = state.setdefault(j, None)
            if old is None:
                state[j] = dict(cur)
                work.append(j)
                continue
            changed = False
            for r, v in cur.items():
                if r not in old or v[0] < old[r][0]:
                    old[r] = v
                    changed = True
            if changed:
                work.append(j)
    return sorted(bad.values(), key=lambda x: x[1])


def unsafe_in_flight(ins):
    """Inline-asm loads (global_load_dwordx4 counted by vmcnt, ds_read_b128 by lgkmcnt) whose destination an
    instruction names before a wait covers the load, over every path of the control flow graph: at each point the
    fewest instructions of the load's counter issued after it on any path to that point. A wait for N covers a load
    with at least N such instructions after it. Only LDS instructions count for lgkmcnt (scalar loads return out of
    order). Returns ([(load, index, touching instruction)], global loads, LDS reads)."""
    cap = 64
    ops, succ = [], _successors(ins)
    for t, in_asm in ins:
        name, _, args = t.partition(" ")
        if re.match(r"\.L\w+:", t):
            ops.append(("none",))
        elif name == "s_waitcnt":
            ops.append(("wait", {k: int(n) for k, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", args)}))
        elif name.startswith("s_"):
            ops.append(("none",))
        else:
            counter = "vmcnt" if _VMEM.match(t) else "lgkmcnt" if name.startswith("ds_") else None
            load = in_asm and name in ("global_load_dwordx4", "ds_read_b128")
            ops.append(("op", counter, _all_regs(args), _all_regs(args.split(",")[0]) if load else set()))
    bad, state, work = {}, {0: {}}, [0]
    while work:
        i = work.pop()
        cur = state[i]
        op = ops[i]
        if op[0] == "wait":
            cur = {r: (c, n, j) for r, (c, n, j) in cur.items() if not (c in op[1] and n >= op[1][c])}
        elif op[0] == "op":
            _, counter, regs, dst = op
            for r in regs & cur.keys():
                bad.setdefault((cur[r][2], i), (ins[cur[r][2]][0], cur[r][2], ins[i][0]))
            if counter:
                cur = {r: (c, min(n + 1, cap) if c == counter else n, j) for r, (c, n, j) in cur.items()}
                cur.update({r: (counter, 0, i) for r in dst})
        for j in succ[i]:
            old = state.get(j)
            if old is None:
                state[j] = dict(cur)
                work.append(j)
                continue
            changed = False
            for r, v in cur.items():
                if r not in old or v[1] < old[r][1]:
                    old[r] = v
                    changed = True
            if changed:
                work.append(j)
    n = [sum(1 for (t, a) in ins if a and t.startswith(o + " ")) for o in ("global_load_dwordx4", "ds_read_b128")]
    return sorted(bad.values(), key=lambda x: x[1]), n[0], n[1]
