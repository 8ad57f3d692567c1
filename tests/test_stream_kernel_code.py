"""CPU-only check of the generated code of the kernel whose tiles of X' = B X follow one another: the waits around the MFMAs, over the
tile boundary included, no spills, and the number of vector-memory operations that its counted wait at a tile's start assumes."""
import os
import subprocess

from test_mfma_wait_states import _kernels, _successors, _walk


def test_waits_over_the_tile_boundary(tmp_path):
    from archscale_amd.build import CSRC, HIPCC_FLAGS, find_hipcc
    # the kernels without the launch code, which would instantiate all the others as well; <FINAL, ADDEND, F16>
    wanted = [(0, 0, 0), (0, 0, 1), (0, 0, 2), (0, 1, 0), (0, 1, 1), (0, 1, 2), (1, 0, 0), (1, 0, 1)]
    source = open(os.path.join(CSRC, "ns_gemm.hip")).read()
    source = source[:source.index("// launch\n")] + "".join(
        f"template __global__ void ns_gemm_stream_kernel<{f}, {a}, {h}>(GroupedGemmParams);\n" for f, a, h in wanted) + "}\n"
    (tmp_path / "stream.hip").write_text(source)
    out = tmp_path / "stream.s"
    subprocess.run([find_hipcc(), *HIPCC_FLAGS, "--cuda-device-only", "-S", "-I", CSRC, str(tmp_path / "stream.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    lines = [l.replace("ns_gemm_kernelI", "othersI").replace("ns_gemm_deep_kernelI", "othersI").replace("ns_gemm_stream_kernelI", "ns_gemm_kernelI")
             for l in out.read_text().splitlines()]
    kernels = _kernels(lines)
    assert len(kernels) == len(wanted), sorted(kernels)
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
        found, code = [], [c for _, b in blocks for c in b]
        for (_, b), at in zip(blocks, entry):
            _walk(b, *at, found.append)
        assert not found, (name, found[:3])
        assert not any(c.startswith("scratch_") for c in code), f"{name} spills registers"
        assert sum(c.startswith("v_mfma") for c in code) == 2 * 64, name
        # the first wait of a tile leaves the stores of the tile before it and eight copies outstanding: no more stores than that
        # between the copies that it waits for and itself, and nothing else there that stays in flight
        assert sum(c.startswith("buffer_store") for c in code) == 32, name
        assert any("vmcnt(40)" in c for c in code), name
        assert not any(c.startswith(("global_", "flat_")) for c in code), name
