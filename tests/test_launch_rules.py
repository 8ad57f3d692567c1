"""CPU-only: how the tiles of a launch are cut for devices of any number of compute units."""
import os
import subprocess

import pytest

PROGRAM = r"""
#include <cstdio>
#include "launch_rules.h"
int main() {
  int units, tile, pair, total, blocks, k;
  double all, longest;
  while (scanf("%d %d %d %d %lf %lf %d %d", &units, &tile, &pair, &total, &all, &longest, &blocks, &k) == 8) {
    const archscale::LaunchSplit s = archscale::launch_split(units, tile, pair != 0, total, all, longest);
    printf("%d %d %d %d\n", s.whole, s.quarters, s.sixteenths, (int)archscale::deep_pipeline(units, 128, blocks, k));
  }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    from archscale_amd.build import CSRC
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "rules.cpp"), "-o", str(d / "rules")], check=True)

    def ask(rows):
        text = "".join("%d %d %d %d %.17g %.17g %d %d\n" % r for r in rows)
        out = subprocess.run([str(d / "rules")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return ask


def test_lines_on_256_units(rules):
    # (tile, pair, total, all k-values, longest) -> (whole, quarters, sixteenths)
    want = {
        (256, 0, 256, 256e3, 1e3): (256, 0, 0),
        (256, 0, 272, 272e3, 1e3): (256, 0, 16),
        (256, 0, 273, 273e3, 1e3): (256, 17, 0),
        (256, 1, 272, 272e3, 1e3): (256, 16, 0),
        (256, 0, 384, 384e3, 1e3): (256, 128, 0),
        (256, 0, 385, 385e3, 1e3): (385, 0, 0),
        (256, 0, 128, 128e3, 1e3): (0, 128, 0),
        (256, 0, 136, 136e3, 1e3): (0, 128, 8),
        (256, 1, 136, 136e3, 1e3): (0, 136, 0),
        (256, 0, 145, 145e3, 1e3): (0, 145, 0),
        (256, 0, 160, 160e3, 1e3): (160, 0, 0),
        (256, 0, 208, 208 * 590.0, 1e3): (0, 208, 0),
        # (one round of quadrants, two to a unit, whatever the reductions)
        (128, 0, 128, 1.0, 1088.0): (0, 128, 0),
        (128, 0, 129, 1.0, 1088.0): (129, 0, 0),
        (128, 0, 128, 1.0, 256.0): (0, 128, 0),
        (128, 0, 129, 1.0, 256.0): (129, 0, 0),
        (128, 1, 10, 1.0, 1024.0): (10, 0, 0),
    }
    got = rules([(256, *k, 1, 64) for k in want])
    for k, g in zip(want, got):
        assert g[:3] == want[k], (k, g)


@pytest.mark.parametrize("units", [32, 38, 64, 128, 256, 304])
def test_every_tile_once_and_rounds_of_the_device(rules, units):
    rows = [(units, tile, pair, total, total * load * 1e3, 1e3, blocks, k)
            for tile in (256, 128, 64) for pair in (0, 1) for total in range(1, 3 * units + 2, max(1, units // 16))
            for load in (0.5, 1.0) for blocks in (units - 1, units, units + 1) for k in (960, 1024)]
    for (_, tile, pair, total, _, _, blocks, k), (whole, quarters, sixteenths, deep) in zip(rows, rules(rows)):
        assert min(whole, quarters, sixteenths) >= 0 and whole + quarters + sixteenths == total
        assert whole == total or whole % units == 0
        assert not sixteenths or (tile == 256 and not pair and 16 * sixteenths <= units)
        assert tile != 64 or whole == total
        # a block of the deep form holds most of a unit's LDS: never more of them than the device has units
        assert deep == (blocks <= units and k >= 1024)


def test_division_by_reciprocals(tmp_path):
    """What the start of a tile computes instead of dividing: exact over the whole range, the ends of it included."""
    from archscale_amd.build import CSRC
    (tmp_path / "divide.cpp").write_text(r"""
#include <cstdio>
#include <initializer_list>
#include "launch_rules.h"
int main() {
  const int top = 0x7fffffff;
  long wrong = 0;
  auto check = [&](int x, int d) {
    if (x < 0 || d < 1) return;
    int rest = -1;
    const int q = archscale::divide(x, d, archscale::reciprocal(d), rest);
    wrong += q != x / d || rest != x % d;
    if (d <= 4) wrong += archscale::divide_1_to_4(x, d) != x / d;
  };
  for (int d = 1; d <= 300; ++d)
    for (int x = 0; x <= 3000; ++x) check(x, d);
  for (long d = 1; d <= top; d = d * 5 / 3 + 1)
    for (long near : {0L, d, 7 * d, (top / d) * d, (long)top})
      for (long e = -2; e <= 2; ++e)
        if (near + e <= top) check((int)(near + e), (int)d);
  printf("%ld\n", wrong);
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "divide.cpp"), "-o", str(tmp_path / "divide")],
                   check=True)
    out = subprocess.run([str(tmp_path / "divide")], capture_output=True, text=True, check=True).stdout
    assert out.strip() == "0", out


def test_parts_of_a_single_product(tmp_path):
    """Parts of the K-split on 256 units: (tiles, k-tiles) -> parts; every part walks at least 20 k-tiles, one block to a unit."""
    from archscale_amd.build import CSRC
    (tmp_path / "parts.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int u, t, k; while (scanf("%d %d %d", &u, &t, &k) == 3) printf("%d\n", archscale::product_parts(u, t, k)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "parts.cpp"), "-o", str(tmp_path / "parts")], check=True)
    want = {(3, 59): 1, (3, 60): 3, (2, 99): 1, (1, 100): 5, (3, 64): 3, (10, 128): 6, (10, 256): 8, (36, 64): 3, (36, 256): 7, (78, 128): 3, (85, 256): 3,
            (86, 256): 1, (136, 88): 1, (1, 4096): 8}
    text = "".join(f"256 {t} {k}\n" for t, k in want)
    out = subprocess.run([str(tmp_path / "parts")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())


def test_blocks_that_sum_squares_follow_the_data(tmp_path):
    """(16-byte runs, strips of the short side) -> blocks: eight runs per thread at a time up to 512 blocks, never fewer than strips."""
    from archscale_amd.build import CSRC
    (tmp_path / "sums.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { long r; int s; while (scanf("%ld %d", &r, &s) == 2) printf("%d\n", archscale::sum_blocks(r, s)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "sums.cpp"), "-o", str(tmp_path / "sums")], check=True)
    want = {(6144 * 16, 8): 48, (4096 * 128, 64): 256, (2816 * 128, 64): 176, (1, 8): 8, (2048 * 512, 8): 512, (2048 * 512 + 1, 8): 512,
            (1 << 28, 600): 600, (2048 * 9, 8): 9, (2048 * 9 + 1, 8): 10}
    out = subprocess.run([str(tmp_path / "sums")], input="".join(f"{r} {s}\n" for r, s in want), capture_output=True, text=True, check=True)
    assert [int(v) for v in out.stdout.split()] == list(want.values())


def test_products_that_tiles_of_64_serve_are_cut_later(tmp_path):
    """(tile that the extents call for, tiles of 128, k-tiles) -> parts."""
    from archscale_amd.build import CSRC
    (tmp_path / "cut.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int c, t, k; while (scanf("%d %d %d", &c, &t, &k) == 3) printf("%d\n", archscale::matrix_parts(c, t, k)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "cut.cpp"), "-o", str(tmp_path / "cut")], check=True)
    want = {(256, 10, 60): 3, (256, 10, 127): 6, (128, 6, 70): 1, (128, 15, 60): 1, (128, 28, 127): 1, (128, 28, 128): 6, (128, 45, 70): 1,
            (128, 1, 100): 5, (128, 1, 99): 1, (256, 36, 64): 3, (256, 3, 59): 1}
    out = subprocess.run([str(tmp_path / "cut")], input="".join(f"{c} {t} {k}\n" for c, t, k in want), capture_output=True, text=True, check=True)
    assert [int(v) for v in out.stdout.split()] == list(want.values())


def test_lines_of_the_tiles_of_32(tmp_path):
    """(units, tile, tiles, longest reduction) -> tiles of 32 or not: sixteen tiles of 128 on 256 units and as many per unit elsewhere."""
    from archscale_amd.build import CSRC
    (tmp_path / "fine.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int u, t, n, k; while (scanf("%d %d %d %d", &u, &t, &n, &k) == 4) printf("%d\n", (int)archscale::fine_tiles(u, t, n, k)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "fine.cpp"), "-o", str(tmp_path / "fine")], check=True)
    want = {(256, 128, 1, 1024): 1, (256, 128, 16, 1024): 1, (256, 128, 17, 1024): 0, (256, 128, 16, 960): 0, (256, 256, 1, 4096): 0,
            (128, 128, 8, 2048): 1, (128, 128, 9, 2048): 0, (38, 128, 2, 2048): 1, (38, 128, 3, 2048): 0, (304, 128, 19, 2048): 1, (304, 128, 20, 2048): 0}
    text = "".join("%d %d %d %d\n" % w for w in want)
    out = subprocess.run([str(tmp_path / "fine")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())


def test_lines_of_the_stream_of_tiles(tmp_path):
    """(units, tiles, longest reduction) -> one block for all tiles of a unit or not."""
    from archscale_amd.build import CSRC
    (tmp_path / "stream.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int u, t, k; while (scanf("%d %d %d", &u, &t, &k) == 3) printf("%d\n", (int)archscale::stream_of_tiles(u, t, k)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "stream.cpp"), "-o", str(tmp_path / "stream")], check=True)
    want = {(256, 384, 2048): 1, (256, 383, 2048): 0, (256, 384, 2112): 0, (256, 4096, 256): 1, (304, 456, 512): 1, (304, 455, 512): 0, (38, 400, 512): 0}
    text = "".join("%d %d %d\n" % w for w in want)
    out = subprocess.run([str(tmp_path / "stream")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())


def test_lines_of_halved_tiles(tmp_path):
    """(tile, pair, tiles of 256, tiles of 128 of the same matrices, all k-values, longest; the k-values of those of 128 beyond two to a unit where
    they are not all of the longest) on 256 units -> in tiles of 128 or not."""
    from archscale_amd.build import CSRC
    (tmp_path / "halved.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() {
  int t, p, n, s; double a, l, m;
  while (scanf("%d %d %d %d %lf %lf %lf", &t, &p, &n, &s, &a, &l, &m) == 7)
    printf("%d\n", (int)archscale::halved_tiles(256, t, p != 0, n, s, m < 0 ? (s - 512) * l : m, l, archscale::launch_split(256, t, p != 0, n, a, l)));
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "halved.cpp"), "-o", str(tmp_path / "halved")], check=True)
    want = {
        # quartered as a whole: little more than one smaller tile to a unit and less than a third of a round; and beyond half of it
        (256, 0, 80, 288, 80 * 4096.0, 4096.0): 1,
        (256, 0, 80, 289, 80 * 4096.0, 4096.0): 0,
        (256, 0, 85, 255, 85 * 4096.0, 4096.0): 1,
        (256, 0, 86, 258, 86 * 4096.0, 4096.0): 0,
        (256, 0, 128, 460, 128 * 4096.0, 4096.0): 0,
        (256, 0, 129, 464, 129 * 4096.0, 4096.0): 1,
        (256, 0, 140, 504, 140 * 4096.0, 4096.0): 1,     # quarters and sixteenths, two smaller tiles to a unit hold it
        (256, 0, 144, 544, 144 * 4096.0, 4096.0): 0,     # they do not
        (256, 0, 208, 744, 208 * 590.0, 1000.0): 1,
        # the second round of smaller tiles: up to half of it; not where it is nearly empty and the reductions are long
        (256, 0, 216, 768, 216 * 768.0, 768.0): 1,
        (256, 0, 216, 769, 216 * 768.0, 768.0): 0,
        (256, 0, 216, 768, 216 * 1024.0, 1024.0): 1,
        (256, 0, 216, 769, 216 * 1024.0, 1024.0): 0,
        (256, 0, 170, 597, 170 * 832.0, 832.0): 0,
        (256, 0, 170, 598, 170 * 832.0, 832.0): 1,
        (256, 0, 170, 570, 170 * 768.0, 768.0): 1,
        (256, 0, 160, 576, 160 * 1024.0, 1024.0): 0,
        # short reductions whatever it holds, up to a full round of tiles of 256
        (256, 0, 256, 968, 256 * 256.0, 256.0): 1,
        (256, 0, 257, 972, 257 * 256.0, 256.0): 0,
        (256, 0, 256, 968, 256 * 320.0, 320.0): 0,
        # matrices of one tile a side (three smaller tiles for one)
        (256, 0, 181, 543, 181 * 1024.0, 1024.0): 1,
        (256, 0, 182, 546, 182 * 1024.0, 1024.0): 0,
        (256, 0, 202, 606, 202 * 512.0, 512.0): 1,
        (256, 0, 203, 609, 203 * 512.0, 512.0): 0,
        (256, 0, 256, 768, 256 * 256.0, 256.0): 1,
        (256, 0, 256, 768, 256 * 768.0, 768.0): 0,
        # a second round whose tiles are not all of the longest reduction: 128 of 512 and 192 of 256 k-values; up to half a round of 512, 160 more for every tile
        (256, 0, 256, 832, 256 * 448.0, 512.0, 128 * 512.0 + 192 * 256.0): 1,
        (256, 0, 256, 832, 256 * 448.0, 512.0, 256 * (512.0 + 160) - 320 * 160): 1,
        (256, 0, 256, 832, 256 * 448.0, 512.0, 256 * (512.0 + 160) - 320 * 160 + 64): 0,
        (256, 0, 224, 798, 210 * 1024.0 + 14 * 256.0, 1024.0, 244 * 1024.0 + 42 * 256.0): 0,   # (half a round by k-values alone)
        (256, 0, 256, 832, 256 * 512.0, 512.0): 0,
        (256, 0, 208, 744, 208 * 1088.0, 1088.0): 0,     # longer reductions stay
        (256, 1, 208, 744, 208 * 1024.0, 1024.0): 0,     # hi+lo pairs stay
        (128, 0, 208, 744, 208 * 1024.0, 1024.0): 0,
    }
    text = "".join("%d %d %d %d %.17g %.17g %.17g\n" % (w if len(w) == 7 else (*w, -1.0)) for w in want)
    out = subprocess.run([str(tmp_path / "halved")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())


def test_lines_of_one_round_of_quadrants(tmp_path):
    """(units, tile, pair, tiles) -> quartered because two quadrants to a unit hold them all."""
    from archscale_amd.build import CSRC
    (tmp_path / "round.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int u, t, p, n; while (scanf("%d %d %d %d", &u, &t, &p, &n) == 4) printf("%d\n", (int)archscale::one_round_of_quadrants(u, t, p != 0, n)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "round.cpp"), "-o", str(tmp_path / "round")], check=True)
    want = {(256, 128, 0, 128): 1, (256, 128, 0, 129): 0, (256, 128, 1, 100): 0, (256, 256, 0, 100): 0, (38, 128, 0, 19): 1, (38, 128, 0, 20): 0}
    text = "".join("%d %d %d %d\n" % w for w in want)
    out = subprocess.run([str(tmp_path / "round")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())


def test_which_plain_updates_go_in_runs_of_eight(tmp_path):
    """(AdamW, weights, gradient, momentum, variance in fp32, whole runs at aligned places) -> in runs, or element by element."""
    from archscale_amd.build import CSRC
    (tmp_path / "runs.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() {
  int a, w, g, m, v, o;
  while (scanf("%d %d %d %d %d %d", &a, &w, &g, &m, &v, &o) == 6) printf("%d\n", (int)archscale::update_in_runs(a, w, g, m, v, o));
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "runs.cpp"), "-o", str(tmp_path / "runs")], check=True)
    by_element = {(1, 1, 1, 1, 1, 0), (1, 0, 0, 1, 1, 0), (0, 1, 1, 1, 0, 0), (0, 1, 0, 1, 0, 0), (0, 0, 1, 1, 0, 0), (0, 1, 1, 0, 0, 0)}
    every = [tuple(i >> k & 1 for k in range(6)) for i in range(64) if i & 1 or not i & 16]
    text = "".join("%d %d %d %d %d %d\n" % w for w in every)
    out = subprocess.run([str(tmp_path / "runs")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert {w for w, o in zip(every, out) if o == "0"} == by_element and len(out) == 48


def test_which_sums_of_squares_go_in_runs_of_eight(tmp_path):
    """(rows, columns, leading dimension), chunks of 8192 -> in runs; never a matrix of fewer than eight elements, which has no run."""
    from archscale_amd.build import CSRC
    (tmp_path / "sums.cpp").write_text(r"""
#include <cstdio>
#include "launch_rules.h"
int main() { int r, c, l; while (scanf("%d %d %d", &r, &c, &l) == 3) printf("%d\n", (int)archscale::sums_in_runs(r, c, l, 8192)); }
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "sums.cpp"), "-o", str(tmp_path / "sums")], check=True)
    want = {(1, 8, 8): 1, (2, 4, 4): 1, (67, 33, 33): 0, (64, 128, 128): 1, (8193, 1, 1): 1, (8191, 1, 1): 0, (95, 121, 121): 1, (64, 64, 72): 0,
            (95, 121, 128): 0, (65536, 65537, 65537): 1, **{(1, n, n): 0 for n in range(1, 8)}}
    text = "".join("%d %d %d\n" % w for w in want)
    out = subprocess.run([str(tmp_path / "sums")], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())
