"""The grid of the fp16 decode attention's chunk pass (nelisp-gpu_amd/csrc/
nlg_attn_grid.h), compiled on the CPU: the workgroups of the grid that the host
chooses read every (row, head group, first chunk) once, on both sides of the
2^32 threads that a grid's x dimension holds, for every kernel form that the
launcher pairs with it."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "nlg_attn_grid.h"
static int fail(const char *what, uint32_t rows, uint32_t kvh, uint32_t grp, int G, uint32_t gx) {
  printf("%s: rows %u kvheads %u grp %u G %d gx %u\n", what, rows, kvh, grp, G, gx);
  return 1;
}
// one form: every workgroup (all: the whole grid; else a sample) reads a unit of
// its own, and the grid is one that can be launched
template <int G>
int form(uint32_t rows, uint32_t kvh, uint32_t grp, uint32_t gx, bool loop, bool rot, bool all, bool last = false) {
  if (!last && !loop && !rot && form<G>(rows, kvh, grp, gx, loop, rot, all, true)) return 1;  // chunks last too
  const AttnGrid g = attn_grid(rows, kvh, grp, G, gx, last);
  if ((uint64_t)g.x * ATTN_WAVES * 64 >= (1ull << 32)) return fail("too many threads", rows, kvh, grp, G, gx);
  if (g.nunits && !attn_reads_units(G, loop, rot)) return fail("units not read", rows, kvh, grp, G, gx);
  if (g.clast && (!last || g.nunits || g.z > 65535)) return fail("chunks last", rows, kvh, grp, G, gx);
  uint32_t before = 0;
  const uint32_t nunits = attn_reads_units(G, loop, rot) ? g.nunits : 0u;
  const uint64_t want = (uint64_t)rows * kvh * (grp / G) * gx, total = (uint64_t)g.x * g.y * g.z;
  if (total < want) return fail("too few workgroups", rows, kvh, grp, G, gx);
  std::vector<char> seen(all ? want : 0);
  uint64_t n = 0;
  const uint64_t step = all ? 1 : total / 100003 + 1;
  for (uint64_t i = 0; i < total; i += step) {
    uint32_t c = ~0u, h0 = ~0u, qr = ~0u;
    if (!attn_unit<G>(i % g.x, i / g.x % g.y, i / g.x / g.y, nunits, g.clast, gx, kvh, grp, c, h0, qr)) continue;
    if (g.clast && c < before) return fail("chunks not last", rows, kvh, grp, G, gx);
    before = c;
    if (c >= gx || qr >= rows || h0 % G || h0 / G >= kvh * (grp / G) || h0 / grp != (h0 + G - 1) / grp)
      return fail("out of range", rows, kvh, grp, G, gx);
    const uint64_t at = ((uint64_t)qr * kvh * (grp / G) + h0 / G) * gx + c;
    if (all && seen[at]++) return fail("read twice", rows, kvh, grp, G, gx);
    n++;
  }
  if (all ? n != want : n * 2 < (total + step - 1) / step) return fail("units missing", rows, kvh, grp, G, gx);
  return 0;
}
int main(void) {
  // rows x kvheads x first chunks: small ones whole; around and past the limit of
  // 2^23 one-head workgroups (32 heads, 256 sequences, 1,024 chunks) a sample
  const struct { uint32_t rows, kvh, gx; bool all; } sizes[] = {
      {1, 1, 1, true}, {3, 5, 7, true}, {17, 3, 13, true}, {16, 8, 64, true}, {33, 1, 9, true},
      {255, 32, 1024, false}, {256, 32, 1023, false}, {256, 32, 1024, false}, {512, 32, 1024, false}, {65535, 8, 200, false},
      {128, 32, 1024, false}, {129, 32, 1024, false},
      {2, 3, 65535, false}, {2, 3, 65536, false}};
  for (const auto &s : sizes)
    for (int rot = 0; rot < 2; rot++) {
      for (uint32_t grp = 1; grp <= 8; grp *= 2)
        if (form<1>(s.rows, s.kvh, grp, s.gx, false, rot, s.all)) return 1;
      for (int loop = 0; loop < 2 - rot; loop++)
        if (form<2>(s.rows, s.kvh, 2, s.gx, loop, rot, s.all) || form<4>(s.rows, s.kvh, 4, s.gx, loop, rot, s.all)) return 1;
      if (rot ? form<8>(s.rows, s.kvh, 8, s.gx, false, true, s.all) : form<4>(s.rows, s.kvh, 8, s.gx, false, false, s.all))
        return 1;
    }
  printf("ok\n");
  return 0;
}
'''


def test_every_unit_of_the_chosen_grid_is_read():
    with tempfile.TemporaryDirectory() as t:
        src, exe = os.path.join(t, "g.cpp"), os.path.join(t, "g")
        with open(src, "w") as f:
            f.write(PROGRAM)
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "nelisp-gpu_amd", "csrc"), src,
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
