"""CPU-only: which launches of X' = B X the kernel takes whose tiles follow one another in a block.  What it cannot do (bounds checks,
unaligned stores, rows further apart than its 32-bit store offsets reach) has to be left to the other kernel."""
import subprocess

import pytest

PROGRAM = r"""
#include <cstdio>
#include "ns_gemm.h"
using namespace archscale;
int main() {
  int rows, final_, ld, stride, base, off, batch, mv, k, mode, split, tile, quarter, addend;
  while (scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d %d", &rows, &final_, &ld, &stride, &base, &off, &batch, &mv, &k, &mode, &split, &tile,
               &quarter, &addend) == 14) {
    GroupedGemmParams gp = {};
    gp.n_groups = 2;
    gp.quarter = quarter;
    for (int i = 0; i < 2; ++i) {
      GemmParams& g = gp.g[i];
      g.K = k; g.tilesM = 1; g.tilesN = 8; g.batch = batch; g.ldp = g.ldq = k;
      g.m_valid = 256; g.n_valid = 2048;
      g.Ct = (__bf16*)(uintptr_t)4096; g.ldct = 256; g.strideCt = 256 * 2048;
      gp.tile_start[i + 1] = gp.tile_start[i] + 8 * 160;
    }
    GemmParams& g = gp.g[1];   // the last problem alone decides
    g.m_valid = mv;
    if (addend) g.E = (const __bf16*)(uintptr_t)4096;
    __bf16* to = (__bf16*)(uintptr_t)(4096 + 2 * off);
    if (rows) { g.C = to; g.Ct = nullptr; g.ldc = ld; g.strideC = stride; }
    else { g.Ct = to; g.ldct = ld; g.strideCt = stride; }
    if (base) g.C = g.Ct = to;
    printf("%d\n", (int)stream_takes(tile, mode, split != 0, final_ != 0, gp, 256));
  }
}
"""


@pytest.fixture(scope="module")
def takes(tmp_path_factory):
    from archscale_amd.build import CSRC, find_hipcc
    d = tmp_path_factory.mktemp("takes")
    (d / "takes.hip").write_text(PROGRAM)
    subprocess.run([find_hipcc(), "--offload-host-only", "-std=c++17", "-I", CSRC, str(d / "takes.hip"), "-o", str(d / "takes")], check=True)

    def ask(**change):
        c = dict(rows=0, final=1, ld=2048, stride=2048 * 256, both=0, off=0, batch=160, mv=256, k=256, mode=2, split=0, tile=256, quarter=0, addend=0)
        assert not change.keys() - c.keys()
        text = " ".join(str(v) for v in {**c, **change}.values()) + "\n"
        return subprocess.run([str(d / "takes")], input=text, capture_output=True, text=True, check=True).stdout.strip() == "1"

    return ask


@pytest.mark.parametrize("rows", [0, 1])
def test_final_results_that_it_takes(takes, rows):
    assert takes(rows=rows)
    assert takes(rows=rows, ld=2056) and takes(rows=rows, off=8) and takes(rows=rows, stride=2048 * 256 + 8)
    assert not takes(rows=rows, ld=2052) and not takes(rows=rows, off=4) and not takes(rows=rows, stride=2048 * 256 + 4)
    assert not takes(rows=rows, mv=250) and not takes(rows=rows, addend=1) and not takes(rows=rows, both=1)
    assert takes(rows=rows, stride=4, batch=1)
    assert not takes(rows=rows, k=192) and not takes(rows=rows, k=2112)
    assert not takes(rows=rows, mode=1) and not takes(rows=rows, split=1) and not takes(rows=rows, tile=128) and not takes(rows=rows, quarter=1)


@pytest.mark.parametrize("rows", [0, 1])
def test_rows_within_reach_of_the_store_offsets(takes, rows):
    """The last of a tile's 256 rows lies 255 * ld elements and its last store 248 elements further on: 2^31 bytes at most, which is what
    the kernel's signed 32-bit offsets hold.  Results inside wider matrices (any out_ld is valid) go to the other kernel."""
    most = (1 << 22) - 8
    assert 2 * (255 * most + 248) < 1 << 31
    assert takes(rows=rows, ld=most)
    for ld in (1 << 22, 7_500_000, 8_421_504, 15_000_000, 2_000_000_000):
        assert not takes(rows=rows, ld=ld), ld


def test_iterates_between_launches(takes):
    assert takes(final=0) and takes(final=0, addend=1) and takes(final=0, mv=250)
    assert not takes(final=0, rows=1) and not takes(final=0, both=1)
