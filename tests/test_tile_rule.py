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
    int m, n, glu, cus, steps, f32;
    while (scanf("%d %d %d %d %d %d", &m, &n, &glu, &cus, &steps, &f32) == 6) {
        const int tile = sq8::choose_wd_tile(m, n, glu != 0, cus, steps, f32 != 0);
        const int groups = tile >= sq8::GROUP_TILE0 ? sq8::group_shapes[tile - sq8::GROUP_TILE0].groups : 0;
        const bool one = tile == sq8::WD_128 || tile == sq8::WD_224 || tile == sq8::WD_256;
        printf("%s\n", one ? "one" : groups == 2 ? "two" : groups == 4 ? "four" : "short");
    }
}
"""


@pytest.fixture(scope="module")
def families(tmp_path_factory):
    """[(m, n, glu, cus, steps, f32), …] → each product's order of sums by the rule."""
    from siliconed_amd.build import HIPCC
    d = tmp_path_factory.mktemp("tile_rule")
    src, exe = str(d / "probe.hip"), str(d / "probe")
    with open(src, "w") as f:
        f.write(PROBE)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-O1", "-ffunction-sections", "-I", CSRC,
                        "-Wl,--gc-sections", src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(cases):
        text = "".join(" ".join(str(int(v)) for v in c) + "\n" for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return out.stdout.split()

    return run


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "fp32"])
@pytest.mark.parametrize("n", [1025, 2048, 3072, 3840, 4608, 5120, 9217, 12288, 20480])
def test_tall_products_sum_in_one_sequence(families, n, f32):
    """From 4096 rows on and past 1024 columns a product's rows have the same bits however they are chunked."""
    cases = [(m, n, glu, 256, steps, f32) for m in [*range(4096, 12289, 61), 4352, 4608, 5376, 6144, 8192, 20000, 100000]
             for glu in (False, True) if n % 2 == 0 or not glu for steps in (1, 16, 48, 60, 192)]
    assert set(families(cases)) == {"one"}


def test_short_products_split_k(families):
    """The rule still splits K where tiles are few."""
    assert families([(77, 3072, 0, 256, 48, 0), (1531, 3072, 0, 256, 48, 1), (1, 3072, 0, 256, 48, 0), (4096, 128, 0, 256, 48, 0)]) == [
        "four", "two", "short", "four"]
