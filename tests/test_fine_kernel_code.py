"""CPU-only check of the generated code of the X X^T kernel with tiles of 32: the waits around transpose reads and MFMAs."""
import os
import re
import subprocess

from test_mfma_wait_states import _kernels, _successors, _walk


def test_waits_of_the_kernel_with_tiles_of_32(tmp_path):
    from archscale_amd.build import CSRC, HIPCC_FLAGS, find_hipcc
    out = tmp_path / "ns_gemm.s"
    subprocess.run([find_hipcc(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, "ns_gemm.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    # the walk of test_mfma_wait_states, over this kernel in the place of the others
    lines = [l.replace("ns_gemm_kernelI", "othersI").replace("ns_gemm_deep_kernelI", "othersI").replace("ns_gemm_fine_kernelI", "ns_gemm_kernelI")
             for l in out.read_text().splitlines()]
    kernels = _kernels(lines)
    assert len(kernels) == 2, sorted(kernels)   # bfloat16 and half
    for name, blocks in kernels.items():
        succ = _successors(blocks)
        entry, todo = [(set(), {}) for _ in blocks], set(range(len(blocks)))
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
        assert not found, (name, found[:3])
        assert sum(c.startswith("v_mfma") for _, code in blocks for c in code) == 2, name
        # transpose reads: nobody touches a result before a full LGKM wait, none is in flight where a block ends
        reads = 0
        for _, code in blocks:
            flight = set()
            for c in code:
                regs = {i for a, b, n in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", c) for i in (range(int(a), int(b) + 1) if a else [int(n)])}
                if c.startswith("s_waitcnt") and "lgkmcnt(0)" in c:
                    flight = set()
                elif c.startswith("ds_read_b64_tr_b16"):
                    dst, addr = c.split(",")[0], c.split(",")[1]
                    assert not ({int(n) for n in re.findall(r"v(\d+)", addr)} & flight), c
                    flight |= {i for a, b in re.findall(r"v\[(\d+):(\d+)\]", dst) for i in range(int(a), int(b) + 1)}
                    reads += 1
                else:
                    assert not (regs & flight), c
            assert not flight, name
        assert reads == 2 * 8, reads   # before the loop and in it: two k-steps, two operands, two reads each
