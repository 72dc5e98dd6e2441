"""The tile of the projections and their gradients by shape: the rule of lvx_gemm_tiles.hpp, compiled by itself, against
what each tile took on an MI355X (256 CUs)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lv-xattn_amd", "csrc")
PROGRAM = """
#include <cstdio>
#include "lvx_gemm_tiles.hpp"
int main() {
    long m, n; int nprob, lower;
    while (std::scanf("%ld %ld %d %d", &m, &n, &nprob, &lower) == 4) std::printf("%d\\n", (int)lvx::gemm_tile(m, n, nprob, 256, lower));
}
"""

# (rows, columns, products): us with tiles of 256 x 256, 256 x 128 (None: not measured) and 224 x 256, in turn on one
# card, medians of seven; K and V of a hidden size of 4096, then dX of the same layer
MEASURED = {
    (3000, 1024, 2): (77.2, 50.1, 69.4), (5000, 1024, 2): (83.7, 99.9, 77.7), (6404, 1024, 2): (91.6, 106.2, 88.0),
    (7000, 1024, 2): (95.4, 108.4, 93.6), (9000, 1024, 2): (172.0, 156.0, 156.8), (11000, 1024, 2): (180.4, 165.7, 164.9),
    (12808, 1024, 2): (184.3, 213.9, 173.6), (14000, 1024, 2): (190.2, 218.5, 185.5), (20000, 1024, 2): (281.2, None, 264.8),
    (28000, 1024, 2): (382.2, None, 362.2), (50000, 1024, 2): (683.6, None, 659.6), (57000, 1024, 2): (743.6, None, 761.7),
    (66000, 1024, 2): (883.3, None, 898.8), (71500, 1024, 2): (938.1, None, 954.2), (74000, 1024, 2): (993.8, None, 1009.3),
    (76848, 1024, 2): (1057.8, None, 1073.3),       # with the norm
    (84000, 1024, 2): (1134.4, None, 1121.2), (92000, 1024, 2): (1236.7, None, 1216.2), (108000, 1024, 2): (1419.0, None, 1455.1),
    (130000, 1024, 2): (1692.6, None, 1736.8), (143000, 1024, 2): (1879.1, None, 1894.7), (150000, 1024, 2): (1979.7, None, 1983.2),
    (1601, 4096, 1): (45.3, 32.5, 41.6), (2300, 4096, 1): (45.3, 55.7, 42.3), (3500, 4096, 1): (53.1, 64.0, 51.9),
    (5000, 4096, 1): (96.9, 95.1, 89.4), (6404, 4096, 1): (102.8, 124.4, 96.4), (9000, 4096, 1): (154.0, 158.5, 141.9),
    (12808, 4096, 1): (206.7, 222.4, 191.8), (25000, 4096, 1): (372.4, None, 349.2), (28000, 4096, 1): (382.4, None, 389.4),
    (33000, 4096, 1): (476.5, None, 474.2), (38000, 4096, 1): (529.4, None, 527.8), (42000, 4096, 1): (592.5, None, 582.2),
    (46000, 4096, 1): (648.7, None, 636.5), (60000, 4096, 1): (825.7, None, 840.3), (76848, 4096, 1): (1077.6, None, 1130.7),
}


@pytest.fixture(scope="module")
def chosen(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", f"-I{CSRC}", str(d / "rule.cpp"), "-o", str(d / "rule")], check=True)

    def ask(shapes, lower):
        text = "".join(f"{m} {n} {p} {int(lower)}\n" for m, n, p in shapes)
        out = subprocess.run([str(d / "rule")], input=text, check=True, capture_output=True, text=True).stdout
        return [int(x) for x in out.split()]
    return ask


def test_no_tile_was_measured_faster(chosen):
    """Within 1 %, which is what the medians of one tile differ by."""
    for shape, tile in zip(MEASURED, chosen(MEASURED, True)):
        us = MEASURED[shape]
        assert us[tile] is not None and us[tile] <= 1.01 * min(t for t in us if t), (shape, tile)


def test_lower_tile_only_where_it_is_built(chosen):
    for shape, tile in zip(MEASURED, chosen(MEASURED, False)):
        us = MEASURED[shape]
        assert tile != 2 and (us[1] is None or us[tile] <= 1.01 * min(us[:2])), (shape, tile)
