#!/usr/bin/env python3
"""Static check of gfx950 device assembly for two hazards of hand-issued loads.

The recurrence kernels request their operand fragments (`global_load_dwordx4 ... sc1`) and the operands they stream
from memory (`... nt`) in inline assembly and wait for them later with an explicit `s_waitcnt vmcnt(n)`.  The compiler does not know that the destination registers are
still being written in between; if it copies, reads or reuses them there (a copy at a join of two definitions, a split
live range) the kernel multiplies garbage.  This script walks the control-flow graph of the assembly from every such
load and reports any instruction that names a destination register on a path before the first wait that covers it.
A wait for vector memory covers a load if it leaves no more operations outstanding than were issued after it.
Branches on flags that the path itself has set to a constant are followed only the way the flag points.

The second hazard: a vector-memory instruction must not read a scalar register within five wait states of a vector
instruction writing it (v_readlane / v_readfirstlane, which is how spilled scalars come back).  The compiler keeps that
distance for its own instructions and does not look into inline assembly.

usage: check_inflight.py file.s [...]      exit status 1 if a hazard is found
"""
import re
import sys

# hand-issued loads carry a cache policy the compiler never emits for its own loads of these kernels: sc1 (device
# scope: the exchanged fragments) or nt (the operands streamed from memory one or two phases ahead)
LOAD = re.compile(r'^\s+global_load_(?:dword|dwordx2|dwordx4|ushort) (?:v\[(\d+):(\d+)\]|v(\d+)), .*\b(?:sc1|nt)\s*$')
# everything that counts into vmcnt (operations complete in issue order)
VMEM = re.compile(r'^(?:global|buffer|flat|scratch)_(?:load|store|atomic)')
SADDR = re.compile(r'^\s+global_load_(?:dword|dwordx2|dwordx4|ushort) \S+ v\d+, s\[(\d+):(\d+)\].*\b(?:sc1|nt)\s*$')
LANE_TO_SCALAR = re.compile(r'^(?:v_readlane_b32|v_readfirstlane_b32) s(\d+)')
VMCNT = re.compile(r'vmcnt\((\d+)\)')
LABEL = re.compile(r'^([.\w$]+):')
REG = re.compile(r'\bv\[(\d+):(\d+)\]|\bv(\d+)\b')


HERE = 'every wave has lanes here'   # (every_wave_here() in the sources)
SPAIR = re.compile(r'^s\[(\d+):(\d+)\]$')
SREG = re.compile(r'^s(\d+)$')


def check(path):
    lines = open(path).read().split('\n')
    label_at = {}
    for i, l in enumerate(lines):
        m = LABEL.match(l)
        if m:
            label_at[m.group(1)] = i
    hazards = []

    # The compiler lowers structured control flow to flags: a block sets a pair of scalar registers to 0 or -1 and a
    # later block branches on `exec & flag`.  Paths are followed with the flags that are known constants (and what
    # they make of vcc), so that a path the flags rule out is not walked.
    def step(i, known, vcc):
        """-> list of (next line, known, vcc) after executing line i"""
        t = lines[i].split(';')[0].strip()
        if not t or t.startswith('.') or LABEL.match(lines[i]):
            return [(i + 1, known, vcc)]
        parts = t.replace(',', ' ').split()
        op, ops = parts[0], parts[1:]
        if op == 's_endpgm':
            return []
        if op == 's_branch':
            return [(label_at[ops[0]], known, vcc)] if ops[0] in label_at else []
        if op.startswith('s_cbranch'):
            tgt = label_at.get(ops[0])
            taken = None
            if op == 's_cbranch_execz' and tgt is not None and i < tgt < i + 60 and any(HERE in l for l in lines[i:tgt]):
                taken = False
            if op == 's_cbranch_vccnz' and vcc is not None:
                taken = (vcc == 'nz')
            if op == 's_cbranch_vccz' and vcc is not None:
                taken = (vcc == 'z')
            out = []
            if taken is not True:
                out.append((i + 1, known, vcc))
            if taken is not False and tgt is not None:
                out.append((tgt, known, vcc))
            return out
        # writes: the first operand (conservatively also for compares, whose first operand is only read)
        if ops:
            d = ops[0]
            if d == 'vcc' or d.startswith('vcc_'):
                vcc = None
                if op in ('s_andn2_b64', 's_and_b64') and len(ops) == 3 and ops[1] == 'exec':
                    m = SPAIR.match(ops[2])
                    if m and (int(m.group(1)), int(m.group(2))) in known:
                        val = known[(int(m.group(1)), int(m.group(2)))]
                        vcc = ('nz' if val == 0 else 'z') if op == 's_andn2_b64' else ('z' if val == 0 else 'nz')
            m = SPAIR.match(d)
            m1 = SREG.match(d)
            if m or m1:
                lo, hi = (int(m.group(1)), int(m.group(2))) if m else (int(m1.group(1)), int(m1.group(1)))
                known = {k: v for k, v in known.items() if k[1] < lo or k[0] > hi}
                if op == 's_mov_b64' and m and len(ops) == 2:
                    if ops[1] in ('0', '-1'):
                        known = dict(known)
                        known[(lo, hi)] = 0 if ops[1] == '0' else -1
                    else:
                        ms = SPAIR.match(ops[1])
                        if ms and (int(ms.group(1)), int(ms.group(2))) in known:
                            known = dict(known)
                            known[(lo, hi)] = known[(int(ms.group(1)), int(ms.group(2)))]
        return [(i + 1, known, vcc)]

    for i, l in enumerate(lines):
        m = LOAD.match(l)
        if not m:
            continue
        a, b = (int(m.group(1)), int(m.group(2))) if m.group(1) else (int(m.group(3)), int(m.group(3)))
        seen = set()
        # (line, known flags, vcc, operations issued after the load)
        stack = [st + (0,) for st in step(i, {}, None)]
        while stack:
            k, known, vcc, younger = stack.pop()
            key = (k, tuple(sorted(known.items())), vcc, younger)
            if key in seen or k >= len(lines):
                continue
            seen.add(key)
            t = lines[k].strip()
            if not t or t.startswith(';') or t.startswith('.') or LABEL.match(lines[k]):
                stack.extend(st + (younger,) for st in step(k, known, vcc))
                continue
            if t.startswith('s_waitcnt') and 'vmcnt' in t:
                if younger >= int(VMCNT.search(t).group(1)):
                    continue   # landed
                stack.extend(st + (younger,) for st in step(k, known, vcc))
                continue
            m2 = LOAD.match(lines[k])
            if m2 and int(m2.group(1) or m2.group(3)) == a and int(m2.group(2) or m2.group(3)) == b:
                continue   # requested again into the same registers (a reload loop)
            code = t.split(';')[0]
            hit = False
            for r in REG.finditer(code):
                lo = int(r.group(1) or r.group(3))
                hi = int(r.group(2) or r.group(3))
                if lo <= b and hi >= a:
                    hazards.append((i + 1, a, b, k + 1, code.strip()))
                    hit = True
                    break
            if hit:
                continue   # (one report per path)
            n = min(younger + (1 if VMEM.match(code) else 0), 63)
            stack.extend(st + (n,) for st in step(k, known, vcc))
    # ---- scalar base written by a vector instruction just before
    close = []
    for i, l in enumerate(lines):
        m = SADDR.match(l)
        if not m:
            continue
        states, k = 0, i - 1
        while states < 5 and k >= 0:
            t = lines[k].split(';')[0].strip()
            if t and not t.startswith('.') and not LABEL.match(lines[k]):
                if t.startswith('s_nop'):
                    states += int(t.split()[1], 0) + 1
                else:
                    w = LANE_TO_SCALAR.match(t)
                    if w and int(m.group(1)) <= int(w.group(1)) <= int(m.group(2)):
                        close.append((path, i + 1, l.strip(), k + 1, t))
                        break
                    states += 1
            k -= 1
    for h in close[:40]:
        print('%s: load at line %d (%s) reads a scalar that line %d writes too shortly before: %s' % h)
    for h in hazards[:40]:
        print('%s: load at line %d into v[%d:%d] is in flight when line %d runs: %s' % ((path,) + h))
    return len(hazards) + len(close)


if __name__ == '__main__':
    total = sum(check(p) for p in sys.argv[1:])
    print('check_inflight: %d hazard(s)' % total)
    sys.exit(1 if total else 0)
