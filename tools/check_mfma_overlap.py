#!/usr/bin/env python3
"""Static check of the gfx950 MFMA register hazards described in vllm_rs_amd/csrc/common.cuh.

For every v_mfma in the given .s files, along every path of the control flow (an instruction, a branch or a barrier counts as one wait state):
  (1) its destination must not overlap SrcA or SrcB;
  (2) within the next 12 wait states nothing but an MFMA accumulating into the SAME destination may
      read or write the destination registers (the inline-asm form is invisible to hipcc's hazard
      recogniser, so the code places VRA_MFMA_DRAIN() = `s_nop 7; s_nop 4` itself).
  (2b) its operands must not be written by a vector instruction within the two wait states before it (most of the
      inline-asm forms carry an `s_nop 1`; DT::mfma_ready does not and is for operands that come from LDS).
Exit status 1 if any violation is found (the Makefile fails the build).

Also a performance lint: (3) no kernel may fetch KERNEL ARGUMENTS with vector loads.  A struct field selected under a
per-lane index (`a.seg[i].out` with i varying across lanes) makes hipcc select the field's ADDRESS inside the kernel-argument block
(s[0:1]) and read it with global_load — followed by `s_waitcnt vmcnt(0)`, which also waits for every weight tile in flight: a full HBM
round trip per occurrence.  Wave-uniform indices (readfirstlane) give scalar selects and s_loads.
"""
import re
import sys

REG = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")
WAIT = 12


def regset(text):
    s = set()
    for m in REG.finditer(text):
        if m.group(1) is not None:
            s.update(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            s.add(int(m.group(3)))
    return s


def instrs(path):
    """yield (function, [instruction lines], {label: index of the instruction behind it}) with comments and directives stripped"""
    cur, body, labels = None, [], {}
    for line in open(path, errors="ignore"):
        m = re.match(r"^(_Z\w+):", line)
        if m:
            if cur and body:
                yield cur, body, labels
            cur, body, labels = m.group(1), [], {}
            continue
        if cur is None:
            continue
        if line.startswith(".Lfunc_end"):
            if body:
                yield cur, body, labels
            cur, body, labels = None, [], {}
            continue
        t = line.split(";")[0].strip()
        if t.endswith(":"):
            labels[t[:-1]] = len(body)
            continue
        if not t or t.startswith("."):
            continue
        body.append(t)
    if cur and body:
        yield cur, body, labels


def flow(body, labels):
    """successors and predecessors of every instruction"""
    succ, pred = [[] for _ in body], [[] for _ in body]
    for i, t in enumerate(body):
        to = []
        if t.startswith(("s_cbranch", "s_branch")):
            to.append(labels.get(t.split()[-1]))
        if not t.startswith(("s_branch", "s_endpgm", "s_setpc")):
            to.append(i + 1)
        for j in to:
            if j is not None and j < len(body):
                succ[i].append(j)
                pred[j].append(i)
    return succ, pred


MFMA = re.compile(r"v_mfma_\w+\s+(\S+),\s*(\S+),\s*(\S+),\s*(\S+)")


def states(t):
    m = re.match(r"s_nop\s+(\d+)", t)
    return int(m.group(1)) + 1 if m else 1


def walk(start, edges, limit, see, body):
    """calls see(instruction, wait states since the MFMA) along all paths from `start` until `limit` states have passed or it returns a true value;
    an instruction is looked at again only when it is reached with fewer states"""
    least, todo = {}, [(j, 0) for j in edges[start]]
    while todo:
        i, waited = todo.pop()
        if waited >= limit or least.get(i, limit) <= waited:
            continue
        least[i] = waited
        if see(body[i], waited):
            continue
        todo += [(j, waited + states(body[i])) for j in edges[i]]


def check(path):
    total = bad = 0
    for fn, body, labels in instrs(path):
        found = []
        mfmas = [(i, m) for i, m in ((i, MFMA.match(t)) for i, t in enumerate(body)) if m]
        if not mfmas:
            continue
        succ, pred = flow(body, labels)
        for i, m in mfmas:
            total += 1
            t = body[i]
            D, A, B, C = (regset(x) for x in m.groups())
            if D & A or D & B:
                found.append(f"[overlap] {fn}: {t}")
                continue
            ops = A | B | C

            def written(u, back):
                if u.startswith("v_") and not u.startswith(("v_mfma", "v_cmp", "v_readfirstlane", "v_readlane", "v_nop")):
                    dst = [regset(x) for x in u.split(None, 1)[1].split(",")[:2 if "swap" in u else 1]]
                    if set().union(*dst) & ops:
                        found.append(f"[operand written {back} states ahead] {fn}: {u}  ->  {t}")
                        return True

            def used(u, waited):
                mm = MFMA.match(u)
                if mm:
                    d2, a2, b2, c2 = (regset(x) for x in mm.groups())
                    if d2 == D and c2 == D and not (a2 & D) and not (b2 & D):
                        return True  # accumulate chain: the next MFMA takes over the tracking
                    if (d2 | a2 | b2 | c2) & D:
                        found.append(f"[early use by another mfma after {waited} states] {fn}: {t}  ->  {u}")
                        return True
                elif regset(u) & D:
                    found.append(f"[early use after {waited} states] {fn}: {t}  ->  {u}")
                    return True
            walk(i, pred, 2, written, body)
            walk(i, succ, WAIT, used, body)
        bad += len(found)
        for f in found:
            print(f, file=sys.stderr)
    return total, bad


KERNARG_VEC = re.compile(r"v_lshl_add_u64\s+v\[\d+:\d+\],\s*s\[0:1\]|global_load_\w+\s+\S+,\s*v\d+,\s*s\[0:1\]")


# tolerated: the peer-pointer table of the one-shot all-reduce is indexed by the thread on purpose (one load per launch); the
# prologue of kernel B and the epilogue wave of kernel A (int4) — both off the decode path since kernels E / W — pay one round trip
KERNARG_VEC_OK = ("oneshot_all_reduce_kernel", "gemm_skinny_kernel", "gemv_q4_kernel")
SDST = re.compile(r"^s_\w+\s+(s\[(\d+):(\d+)\]|s(\d+))(?=[,\s]|$)")


def check_kernarg_vector_loads(path):
    """s[0:1] holds the kernel-argument pointer from entry until something else is written to it"""
    bad = 0
    for fn, body, _ in instrs(path):
        n = 0
        for t in body:
            if KERNARG_VEC.search(t):
                n += 1
            m = SDST.match(t)
            if m and not t.startswith(("s_cmp", "s_cbranch", "s_waitcnt", "s_nop", "s_barrier", "s_bitcmp")):
                lo, hi = (int(m.group(2)), int(m.group(3))) if m.group(2) is not None else (int(m.group(4)), int(m.group(4)))
                if lo <= 1 and hi >= 0:
                    break  # s0 / s1 rewritten: no longer the kernel-argument pointer
        if n and any(k in fn for k in KERNARG_VEC_OK):
            print(f"[note: kernel arguments fetched with {n} vector loads, tolerated] {fn}", file=sys.stderr)
        elif n:
            bad += n
            print(f"[kernel arguments fetched with {n} vector loads] {fn}", file=sys.stderr)
    return bad


def main(paths):
    T = B = K = 0
    for p in paths:
        t, b = check(p)
        T += t
        B += b
        K += check_kernarg_vector_loads(p)
    print(f"check_mfma_overlap: {T} MFMA instructions, {B} violations" + (f", {K} vector loads of kernel arguments" if K else ""))
    return 1 if B or K else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
