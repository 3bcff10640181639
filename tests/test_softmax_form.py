"""The form that a softmax row takes (nelisp-gpu_amd/csrc/nlg_softmax_form.h),
compiled on the CPU: the rows of every call that 256 threads a row would take fit
the grid that is chosen, and up to 1,024 columns the choice is the faster of a wave
and 256 threads by the times measured with both."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# (rows, columns): us with a wave a row, with 256 threads
MEASURED = {(1, 257): (2.91, 2.58), (512, 257): (3.22, 2.95), (16384, 257): (14.3, 18.1), (20, 511): (3.19, 2.74),
            (4096, 511): (6.16, 7.11), (128, 512): (2.96, 2.79), (1024, 512): (3.23, 3.76), (20, 777): (3.40, 2.91),
            (512, 600): (3.26, 3.48), (512, 1000): (3.51, 3.81), (1, 1000): (3.44, 2.79), (128, 1021): (3.76, 3.07),
            (1024, 1021): (4.36, 4.12), (4096, 1021): (8.54, 8.78), (20, 1024): (3.16, 2.85), (512, 1024): (3.48, 3.19),
            (2048, 1024): (4.54, 4.81), (65536, 1024): (84.3, 105.7)}

PROGRAM = r'''
#include <stdio.h>
#include "nlg_softmax_form.h"
int main(void) {
  unsigned rows, n;
  while (scanf("%u %u", &rows, &n) == 2) printf("%u\n", softmax_threads(rows, n, n % 4 == 0, 256));
  return 0;
}
'''


@pytest.fixture(scope="module")
def choose():
    with tempfile.TemporaryDirectory() as t:
        src, exe = os.path.join(t, "s.cpp"), os.path.join(t, "s")
        with open(src, "w") as f:
            f.write(PROGRAM)
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "nelisp-gpu_amd", "csrc"), src,
                        "-o", exe], check=True)

        def run(asked):
            out = subprocess.run([exe], input="".join(f"{r} {n}\n" for r, n in asked), capture_output=True, text=True,
                                 check=True).stdout
            return [int(x) for x in out.split()]
        yield run


def test_every_grid_can_be_launched(choose):
    asked = [(rows, n) for rows in (1, 2 ** 22 - 1, 2 ** 22, 2 ** 22 + 1, 2 ** 24 - 1)
             for n in (1, 256, 257, 1024, 1025, 8192, 8193, 16384, 32768, 32769)]
    for (rows, n), threads in zip(asked, choose(asked)):
        blocks = (rows + 3) // 4 if threads == 64 else rows
        assert blocks * max(threads, 256) < 2 ** 32, (rows, n, threads)
        held = {64: 1024, 256: 8192, 1024: 32768, 0: 2 ** 32}[threads]
        assert n <= held, (rows, n, threads)


def test_the_faster_form_is_chosen(choose):
    for (case, (wave, group)), threads in zip(MEASURED.items(), choose(MEASURED)):
        assert threads == (64 if wave < group else 256), case
