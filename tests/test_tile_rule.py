"""The tile rules of the products, compiled for the host (no GPU): which calls share one order of sums.

A product's bits depend on the order its tile sums K in: one MFMA sequence over K (128-, 224- and 256-row tiles), the K
steps split over two or four wave groups, or the short-M kernels' own."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "siliconed_amd", "csrc")
PROBE = r"""
#include "sq8_gemm.hip"
#include <stdio.h>
int main() {
    char route[8];
    int m, n, glu, cus, steps, residual;
    while (scanf("%7s %d %d %d %d %d %d", route, &m, &n, &glu, &cus, &steps, &residual) == 7) {
        if (route[0] == 'q') {
            const int tile = sq8::choose_blocks_tile(m, n, glu != 0, cus, steps);
            if (tile > sq8::BLOCKS16_ROWS) printf("short %d\n", tile - sq8::BLOCKS16_ROWS);
            else printf("one %s\n", tile == sq8::BL_128x128 ? "128x128" : tile == sq8::BL_64x256 ? "64x256" : "128x256");
            continue;
        }
        const int tile = route[0] == 'w' ? sq8::choose_i8_tile(m, n, glu != 0, cus, steps, residual != 0)
                                         : sq8::choose_wd_tile(m, n, glu != 0, cus, steps, route[0] == 'f');
        if (tile >= sq8::GROUP_TILE0) {
            const sq8::GroupShape &g = sq8::group_shapes[tile - sq8::GROUP_TILE0];
            printf("%s %s\n", g.groups == 2 ? "two" : g.groups == 4 ? "four" : "eight", g.name);
        } else if (route[0] == 'w' || tile == sq8::WD_128 || tile == sq8::WD_224 || tile == sq8::WD_256) {
            printf("one %s\n", route[0] == 'w' || tile == sq8::WD_128 ? "128" : tile == sq8::WD_224 ? "224" : "256");
        } else if (tile == sq8::WD_64 || tile == sq8::WD_64N) {
            printf("one %s\n", tile == sq8::WD_64 ? "64" : "64n");
        } else {
            printf("short %s\n", tile == sq8::WD_GEMV ? "gemv" : "skinny");
        }
    }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """[(route, m, n, glu, cus, steps, residual), …] → each product's (order of sums, tile) by the rule."""
    from siliconed_amd.build import HIPCC
    d = tmp_path_factory.mktemp("tile_rule")
    src, exe = str(d / "probe.hip"), str(d / "probe")
    with open(src, "w") as f:
        f.write(PROBE)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-O1", "-ffunction-sections", "-I", CSRC,
                        "-Wl,--gc-sections", src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(cases):
        text = "".join(" ".join(str(v if isinstance(v, str) else int(v)) for v in c) + "\n" for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return [tuple(line.split()) for line in out.stdout.splitlines()]

    return run


@pytest.mark.parametrize("route", ["bf16", "fp32"])
@pytest.mark.parametrize("n", [1025, 2048, 3072, 3840, 4608, 5120, 9217, 12288, 20480])
def test_tall_products_sum_in_one_sequence(rule, n, route):
    """From 4096 rows on and past 1024 columns a product's rows have the same bits however they are chunked."""
    cases = [(route, m, n, glu, 256, steps, 0) for m in [*range(4096, 12289, 61), 4352, 4608, 5376, 6144, 8192, 20000, 100000]
             for glu in (False, True) if n % 2 == 0 or not glu for steps in (1, 16, 48, 60, 192)]
    assert {order for order, _ in rule(cases)} == {"one"}


def test_short_products_split_k(rule):
    """The rule still splits K where tiles are few."""
    assert [order for order, _ in rule([("bf16", 77, 3072, 0, 256, 48, 0), ("fp32", 1531, 3072, 0, 256, 48, 0),
                                        ("bf16", 1, 3072, 0, 256, 48, 0), ("bf16", 4096, 128, 0, 256, 48, 0),
                                        ("w8a8", 77, 3072, 0, 256, 24, 0)])] == ["four", "two", "short", "four", "eight"]


@pytest.mark.parametrize("case,tile", [
    # Up to 16 rows of one group of GLU columns, the activation not in the short-M kernel's LDS; one row of three groups.
    (("bf16", 10, 3072, 1, 256, 60, 0), "gemv"), (("bf16", 5, 3200, 1, 256, 18, 0), "gemv"), (("bf16", 11, 256, 1, 256, 26, 0), "gemv"),
    (("bf16", 1, 10944, 0, 256, 122, 0), "g32x64k4"), (("bf16", 1, 9216, 0, 256, 48, 0), "gemv"), (("bf16", 16, 3072, 0, 256, 96, 0), "g32x32k4"),
    # The same of one group of plain columns, to ten rows (fp32 route: four).
    (("bf16", 6, 4043, 0, 256, 59, 0), "gemv"), (("bf16", 5, 64, 0, 256, 53, 0), "gemv"), (("fp32", 4, 2295, 0, 256, 129, 0), "gemv"),
    (("bf16", 16, 2880, 0, 256, 60, 0), "g32x32k4"), (("fp32", 13, 2295, 0, 256, 145, 0), "g32x32k4"),
    # One row of three groups on short K; the skinny kernel's slabs past half the CUs.
    (("bf16", 1, 8447, 0, 256, 13, 0), "gemv"), (("bf16", 6, 8352, 0, 256, 11, 0), "skinny"), (("bf16", 10, 9216, 0, 256, 108, 0), "g32x64k4"),
    # 64 rows without groups: few K steps, odd counts of them; output rows of odd values; a second round of small tiles.
    (("bf16", 2840, 1152, 0, 256, 7, 0), "64n"), (("bf16", 139, 17856, 0, 256, 6, 0), "64n"), (("bf16", 652, 5120, 1, 256, 59, 0), "64"),
    (("bf16", 1119, 2944, 0, 256, 9, 0), "64n"), (("bf16", 1032, 6559, 0, 256, 8, 0), "g128x128k2"),
    (("bf16", 21, 16576, 0, 256, 46, 0), "g64x96k4"), (("bf16", 441, 12800, 1, 256, 24, 0), "128"),
    (("fp32", 855, 8064, 0, 256, 12, 0), "128"), (("fp32", 188, 4640, 0, 256, 4, 0), "g64x64k4"),
    # Tall products, of few K steps and of many.
    (("bf16", 7887, 7104, 0, 256, 12, 0), "128"), (("fp32", 5813, 12288, 0, 256, 16, 0), "224"),
    (("fp32", 6054, 1408, 0, 256, 8, 0), "224"), (("bf16", 4096, 12288, 0, 256, 48, 0), "256"), (("bf16", 4608, 9216, 0, 256, 48, 0), "224"),
    # W8A8: a round of more than one and fewer than two workgroups a CU; rounds of K-group tiles past the first.
    (("w8a8", 3912, 3072, 0, 256, 24, 0), "128"), (("w8a8", 1975, 6144, 0, 256, 24, 0), "128"),
    (("w8a8", 3277, 1024, 1, 256, 8, 0), "g128x128k2"), (("w8a8", 239, 16000, 0, 256, 8, 0), "g128x128k2"),
    (("w8a8", 498, 18752, 0, 256, 7, 0), "128"), (("w8a8", 512, 3072, 0, 256, 24, 0), "g64x96k4"), (("w8a8", 1531, 3072, 0, 256, 24, 0), "g96x192k2"),
    # Q8_0: half-height tiles where they fit a round; few K steps; a full chip.
    (("q8", 575, 7040, 1, 256, 16, 0), "64x256"), (("q8", 1065, 7488, 1, 256, 24, 0), "64x256"), (("q8", 486, 5696, 1, 256, 186, 0), "64x256"),
    (("q8", 300, 10944, 0, 256, 54, 0), "64x256"), (("q8", 664, 8384, 0, 256, 14, 0), "128x256"),
    (("q8", 3913, 8960, 0, 256, 18, 0), "128x128"),
    (("q8", 4096, 12288, 0, 256, 48, 0), "128x256"), (("q8", 77, 12288, 0, 256, 48, 0), "80"), (("q8", 1, 3072, 0, 256, 48, 0), "16"),
], ids=str)
def test_measured_choices(rule, case, tile):
    """Shapes on which another tile measured 10 % slower or more."""
    assert rule([case])[0][1] == tile
