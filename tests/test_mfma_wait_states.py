"""CPU-only check of the generated code of every product kernel: the waits around the matrix instructions.

The MFMAs are inline assembly, so the compiler inserts no wait states for them.  What it inserts for the builtin of the same
instruction is what has to be there otherwise: two wait states between a vector instruction that writes an operand and the MFMA
that reads it, eight between an MFMA and the first read of its result.  The second wait is the kernel's own (two s_nop 15
after the last MFMA of a tile), and every use of a result has to stand behind it."""
import os
import re
import subprocess

REG = re.compile(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b")
OPERAND_WAIT = 2


def _regs(text):
    return {(k, i) for k, a, b, k1, n in REG.findall(text) for i in (range(int(a), int(b) + 1) if k else [int(n)])
            for k in [k or k1]}


def _kernels(lines):
    """{mangled name: [[instruction, ...] per basic block, labels]} of the product kernels"""
    out, cur = {}, None
    for line in lines:
        code = line.split(";")[0].strip()
        if code.endswith(":") and not code.startswith("."):
            cur = None
            if re.search(r"ns_gemm_(deep_)?kernelI", code):
                cur = out.setdefault(code[:-1], [("", [])])
                assert cur == [("", [])], f"{code} seen twice"
        elif cur is not None and code:
            if code.startswith(".Lfunc_end"):
                cur = None
            elif code.startswith(".LBB") and code.endswith(":"):
                cur.append((code[:-1], []))
            elif not code.startswith("."):
                cur[-1][1].append(code)
                if code.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                    cur.append(("", []))
    return out


def _successors(blocks):
    index = {label: i for i, (label, _) in enumerate(blocks) if label}
    succ = []
    for i, (_, code) in enumerate(blocks):
        last, to = code[-1] if code else "", set()
        assert not any(c.startswith(("s_setpc", "s_swappc")) for c in code), "indirect jump"
        if last.startswith(("s_cbranch", "s_branch")):
            to.add(index[last.split()[-1]])
        if not last.startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            to.add(i + 1)
        succ.append(to)
    return succ


def _walk(code, pending, fresh, check):
    """pending: registers that hold an MFMA result not waited for yet; fresh: wait states since a vector instruction wrote
    a register (below OPERAND_WAIT only).  `check` gets a message for every violation."""
    pending, fresh = set(pending), dict(fresh)
    previous = ""
    for c in code:
        mention = _regs(c)
        passed = int(c.split()[1]) + 1 if c.startswith("s_nop") else 1
        if c.startswith("v_mfma"):
            d, a, b, s = (_regs(o) for o in c.split(" ", 1)[1].split(",")[:4])
            if check:
                if d != s or (a | b) & pending:
                    check(f"operands of {c}")
                if any(r in fresh for r in mention):
                    check(f"operand written by a vector instruction less than {OPERAND_WAIT} wait states before {c}")
            written = set()
            pending |= d
        else:
            if check and mention & pending:
                check(f"result of an MFMA used before the wait: {c}")
            written = set()
            if c.startswith("v_"):
                if c.startswith("v_cmpx") and check:
                    check(f"vector write of EXEC: {c}")
                operands = c.split(" ", 1)[1].split(",") if " " in c else []
                written = _regs(",".join(operands[:2] if "swap" in c.split()[0] else operands[:1]))
            if c == previous == "s_nop 15":
                pending = set()
        fresh = {r: n + passed for r, n in fresh.items() if n + passed < OPERAND_WAIT and r not in written}
        fresh.update({r: 0 for r in written})
        previous = c
    return pending, fresh


def test_waits_around_the_matrix_instructions(tmp_path):
    from archscale_amd.build import CSRC, HIPCC_FLAGS, find_hipcc
    out = tmp_path / "ns_gemm.s"
    subprocess.run([find_hipcc(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, "ns_gemm.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    kernels = _kernels(out.read_text().splitlines())
    faults = {}
    for name, blocks in kernels.items():
        succ = _successors(blocks)
        # what is pending or fresh at the entry of a block: the union (the shortest wait) over its predecessors
        entry = [(set(), {}) for _ in blocks]
        todo = set(range(len(blocks)))
        while todo:
            i = todo.pop()
            pending, fresh = _walk(blocks[i][1], *entry[i], None)
            for j in succ[i]:
                p, f = entry[j]
                merged = (p | pending, {r: min(f.get(r, 99), fresh.get(r, 99)) for r in f.keys() | fresh.keys()})
                if merged != entry[j]:
                    entry[j] = merged
                    todo.add(j)
        found = []
        for (_, code), at in zip(blocks, entry):
            _walk(code, *at, found.append)
        if found:
            faults[name] = found[:3]
        # four waves of (side / 2)^2 in fragments of 16 x 16, two k-steps in the one loop body
        m = re.search(r"ns_gemm_kernelILi(\d+)E", name)
        side = int(m.group(1)) if m else {2: 128, 3: 64}[int(re.search(r"deep_kernelILi(\d+)E", name).group(1))]
        assert sum(c.startswith("v_mfma") for _, code in blocks for c in code) == 2 * (side // 32) ** 2, name
    assert not faults, faults
    # K-split (6), tiles of 256 and of 128 with both pipelines (21 each), tiles of 64 (16: no hi+lo pair)
    assert len(kernels) == 6 + 3 * 21 + 16, len(kernels)
