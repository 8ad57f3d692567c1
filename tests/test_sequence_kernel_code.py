"""CPU-only check of the generated code of the products whose parts one block walks in sequence: the waits around the MFMAs, the ones
where a part's sum is taken out of the accumulators included."""
import os
import subprocess

from test_mfma_wait_states import _kernels, _successors, _walk


def test_waits_between_the_parts_of_a_reduction(tmp_path):
    from archscale_amd.build import CSRC, HIPCC_FLAGS, find_hipcc
    # the kernels without the launch code, which would instantiate all the others as well
    source = open(os.path.join(CSRC, "ns_gemm.hip")).read()
    source = source[:source.index("// launch\n")] + "".join(
        f"template __global__ void ns_gemm_sequence_kernel<{cfg}, {mode}>(GroupedGemmParams);\n"
        for cfg in ("CFG_128", "CFG_128_DEEP") for mode in ("MODE_SYRK", "MODE_SYRK2")) + "}\n"
    (tmp_path / "sequence.hip").write_text(source)
    out = tmp_path / "sequence.s"
    subprocess.run([find_hipcc(), *HIPCC_FLAGS, "--cuda-device-only", "-S", "-I", CSRC, str(tmp_path / "sequence.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    lines = [l.replace("ns_gemm_kernelI", "othersI").replace("ns_gemm_deep_kernelI", "othersI").replace("ns_gemm_sequence_kernelI", "ns_gemm_kernelI")
             for l in out.read_text().splitlines()]
    kernels = _kernels(lines)
    assert len(kernels) == 4, sorted(kernels)   # both pipelines, with and without an addend
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
        assert sum(c.startswith("v_mfma") for _, code in blocks for c in code) == 32, name
        assert not any(c.startswith("scratch_") for _, code in blocks for c in code), f"{name} spills registers"
