"""CPU-only: the launches of the weight update for sets of parameters of any size.  HIP takes fewer than 2^32 threads in a dimension; the
update has to be cut so that every chunk is covered once.  The launch calls are recorded in place of the runtime's."""
import subprocess

import pytest

PROGRAM = r"""
#include <cstdio>
#include "elementwise.hip"
static dim3 G, B;
extern "C" {
extern const char __hip_fatbin[64] = {0};
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { G = g; B = b; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t*, hipStream_t*) { *g = G; *b = B; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  if (f == (const void*)archscale::post_apply_kernel) printf("%u %u %u %u %d ", grid.x, grid.y, grid.z, block.x, *(int*)args[8]);
  return hipSuccess;
}
}
int main() {
  int n;
  while (scanf("%d", &n) == 1) {
    const hipError_t e = archscale::launch_post_plain(nullptr, nullptr, 1, n, 0.1f, 0.f, 0, nullptr, nullptr);
    printf("%d\n", (int)e);
  }
}
"""


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """chunks -> [(blocks, first chunk)]"""
    from archscale_amd.build import CSRC, find_hipcc
    d = tmp_path_factory.mktemp("apply")
    (d / "apply.hip").write_text(PROGRAM)
    subprocess.run([find_hipcc(), "--offload-host-only", "-fuse-cuid=none", "-O1", "-std=c++17", "-I", CSRC, "-c", str(d / "apply.hip"),
                    "-o", str(d / "apply.o")], check=True)
    subprocess.run([find_hipcc(), str(d / "apply.o"), "-o", str(d / "apply")], check=True)

    def ask(chunks):
        out = [int(v) for v in subprocess.run([str(d / "apply")], input=f"{chunks}\n", capture_output=True, text=True, check=True).stdout.split()]
        assert out[-1] == 0 and len(out) % 5 == 1
        rows = [tuple(out[i:i + 5]) for i in range(0, len(out) - 1, 5)]
        assert all(r[1:4] == (1, 1, 256) for r in rows)
        return [(r[0], r[4]) for r in rows]

    return ask


# one chunk; the largest single launch and the next; 2^24 - 1 chunks (2^37 elements), which a block per chunk would take at most; the largest int
@pytest.mark.parametrize("chunks", [1, 5, 4194303, 4194304, 4194305, (1 << 24) - 1, 1 << 24, 0x7fffffff])
def test_every_chunk_once_and_no_launch_too_large(launches, chunks):
    at = 0
    for blocks, first in launches(chunks):
        assert first == at and blocks % 4 == 0 and 0 < blocks * 256 < 1 << 32
        at += blocks // 4
    assert at == chunks
    assert chunks > 4194303 or len(launches(chunks)) == 1
