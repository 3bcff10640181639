"""The rule that picks an f32 product's output tile (nelisp-gpu_amd/csrc/
nlg_mm_tile.h), compiled on the CPU, against the times measured with every form:
no product is slower than on 16 x 16 tiles, where padded rows and columns cost
least, and none is far from its fastest form.  Rows and columns of 1 to 48 among
them: the count of tiles alone takes such products to forms that compute mostly
padding."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# us at k = 2,048 with 16 x 16, 32 x 32, 64 x 32 and 64 x 64 tiles on 256 CUs
MEASURED = {
    ("matmul", 1, 6912): (44, 57, 96, 156), ("matmul", 1, 8192): (45, 58, 96, 156),
    ("matmul", 1, 32000): (142, 138, 183, 171), ("matmul", 16, 9000): (61, 75, 107, 158),
    ("matmul", 16, 32000): (142, 138, 186, 172), ("matmul", 17, 6144): (60, 58, 96, 157),
    ("matmul", 32, 8192): (76, 58, 97, 158), ("matmul", 32, 32000): (269, 139, 191, 177),
    ("matmul", 48, 16384): (206, 138, 114, 158), ("matmul", 64, 2048): (42, 57, 94, 158),
    ("matmul", 300, 300): (43, 58, 96, 158), ("matmul", 512, 512): (75, 58, 96, 157),
    ("matmul", 768, 768): (154, 110, 108, 158), ("matmul", 1024, 1024): (265, 139, 117, 159),
    ("matmul", 1536, 1536): (582, 291, 239, 272), ("matmul", 2048, 2048): (1029, 506, 384, 352),
    ("matmul", 6912, 1): (44, 69, 111, 178), ("matmul", 8192, 1): (43, 67, 111, 179),
    ("matmul", 6144, 17): (61, 68, 111, 179), ("matmul", 16384, 17): (141, 83, 112, 180),
    ("matmul", 8192, 24): (76, 58, 97, 158),
    ("linear", 1, 8192): (46, 58, 96, 165), ("linear", 1, 32000): (141, 140, 184, 179),
    ("linear", 16, 9000): (62, 76, 108, 165), ("linear", 96, 2048): (61, 58, 97, 171),
    ("linear", 16384, 17): (143, 79, 98, 170), ("linear", 2048, 2048): (1020, 510, 387, 358),
    ("matmul-tiled", 1, 8192): (45, 69, 101, 157), ("matmul-tiled", 16, 9000): (62, 71, 103, 159),
    ("matmul-tiled", 17, 6144): (62, 69, 101, 159), ("matmul-tiled", 32, 8192): (78, 69, 101, 159),
    ("matmul-tiled", 48, 16384): (205, 119, 112, 159), ("matmul-tiled", 96, 2048): (61, 69, 101, 158),
    ("matmul-tiled", 768, 768): (155, 89, 104, 159), ("matmul-tiled", 2048, 2048): (1030, 415, 373, 350),
}

PROGRAM = r'''
#include <stdio.h>
#include "nlg_mm_tile.h"
int main(void) {
  unsigned m, n, tiled, vec;
  while (scanf("%u %u %u %u", &m, &n, &tiled, &vec) == 4) printf("%d\n", mm_tile(m, n, 256, tiled, vec));
  return 0;
}
'''


@pytest.fixture(scope="module")
def choose():
    with tempfile.TemporaryDirectory() as t:
        src, exe = os.path.join(t, "m.cpp"), os.path.join(t, "m")
        with open(src, "w") as f:
            f.write(PROGRAM)
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "nelisp-gpu_amd", "csrc"), src,
                        "-o", exe], check=True)

        def run(asked):
            text = "".join(f"{m} {n} {int(name == 'matmul-tiled')} {int(name == 'linear' or n % 4 == 0)}\n"
                           for name, m, n in asked)
            out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
            return [int(x) for x in out.split()]
        yield run


def test_no_product_is_slower_than_on_the_smallest_tiles(choose):
    # 3%: what the runs of one form differ by at these times
    for (case, us), form in zip(MEASURED.items(), choose(MEASURED)):
        assert us[form] <= 1.03 * us[0] and us[form] <= 1.07 * min(us), (case, us, form)


def test_thin_products_stay_on_the_smallest_tiles(choose):
    """Up to 16 rows or columns a 16 x 16 tile holds as many useful outputs as any."""
    thin = [("matmul", m, n) for m in (1, 4, 16) for n in (64, 2560, 6912, 8192, 9000, 16384)]
    assert set(choose(thin)) <= {0, 1}
    assert set(choose([c for c in thin if c[2] <= 9000])) == {0}
    assert set(choose([("matmul", n, m) for _, m, n in thin if n <= 9000])) == {0}
