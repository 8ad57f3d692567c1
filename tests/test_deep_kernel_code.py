"""CPU-only check of the generated code of the deeper-pipelined product kernels (64 tiles, lone 128 tiles)."""
import os
import re
import subprocess


def test_transpose_reads_of_the_deep_kernels_are_waited_for(tmp_path):
    """Inline-assembly LDS transpose reads are invisible to the compiler's waits: no instruction may mention their registers
    before a full LGKM wait, and none may be in flight at a label or branch (so straight-line order is enough)."""
    from archscale_amd.build import CSRC, HIPCC_FLAGS, find_hipcc
    out = tmp_path / "ns_gemm.s"
    subprocess.run([find_hipcc(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, "ns_gemm.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    # <CFG, MODE, SPLIT, FINAL, ADDEND, F16>; MODE 3 reads its operand K-major
    name = re.compile(r"ns_gemm_deep_kernelILi(\d+)ELi(\d+)ELb[01]ELb[01]ELb[01]ELi(\d+)EE")
    reg = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")

    def regs(s):
        return {i for a, b, c in reg.findall(s) for i in (range(int(a), int(b) + 1) if a else [int(c)])}

    seen, current, in_asm, pending = {}, None, False, set()
    for line in out.read_text().splitlines():
        if "#ASMSTART" in line or "#ASMEND" in line:
            in_asm = "#ASMSTART" in line
            continue
        code = line.split(";")[0].strip()
        if code.endswith(":") and "kernel" in code:
            m = name.search(code)
            current = (int(m.group(1)), int(m.group(3))) if m and m.group(2) == "3" else None
            if current:
                assert current not in seen
                seen[current] = 0
            continue
        if current is None or not code:
            continue
        if code.startswith(".Lfunc_end"):
            current = None
        elif code.endswith(":") or code.startswith(("s_cbranch", "s_branch", "s_endpgm")):
            assert not pending, f"transpose reads in flight at {code}"
        elif code.startswith("s_waitcnt") and "lgkmcnt(0)" in code:
            pending = set()
        elif not code.startswith("."):
            assert not (regs(code) & pending), f"touches a transpose-read result before the wait: {code}"
            if in_asm and code.startswith("ds_read_b64_tr_b16"):
                pending |= regs(code.split(",")[0])
                seen[current] += 1
    # both configurations, bfloat16 and half; two k-steps x (FR + FR) fragments x two reads in each k-tile
    assert set(seen) == {(2, 0), (2, 1), (3, 0), (3, 1)}, seen
    assert all(n >= 2 * (8 if cfg == 2 else 4) * 2 for (cfg, _), n in seen.items()), seen
