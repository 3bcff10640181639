// nlg_mm_tile.h -- which output tile an f32 product by name takes (plain C++:
// checked against measured times on the CPU).
#pragma once

#include <stdint.h>

enum { MM_16X16 = 0, MM_32X32 = 1, MM_64X32 = 2, MM_64X64 = 3 };

// The form with the least estimated time.  Larger tiles read less per product,
// but a workgroup's chain over k is longer, rows and columns past the product are
// computed all the same, and the tiles come in rounds: with w the tiles per CU,
// rounded up, a form takes about max(one, base + per * w).  Measured at k = 2,048
// (256 CUs; the times scale with k alike), us by w = 1 / 2 / 3 / 4 / 8:
//   16 x 16  31 / 43 / 60 / 76 / 141
//   32 x 32  58 / 76 / - / 138 / 261      (matmul-tiled's sums: 69 / 73 / - / 118 / 217)
//   64 x 32  96 / 108-115 / - / 183-197 / 384
//   64 x 64  157 / 171-181 / 270 / 351 / -
// and from unaligned rows 67 / 112 / 179 at w = 1.  So one row of 8,192 outputs stays
// on 16 x 16 (45 us; 64 x 32, which the count of tiles alone chose, 97), as do 16 rows
// of 9,000 (61; 107); 32 rows of 8,192 take 32 x 32 (58; 16 x 16 76), 1,024^3
// 64 x 32 (56 of 133), 2,048^3 64 x 64 (349 of 1,024).
inline int mm_tile(uint32_t M, uint32_t N, uint32_t cu, bool tiled, bool vec) {
  struct Form {
    uint32_t ta, tb, one, odd, base, per;  // tenths of a microsecond; odd: one, from unaligned rows
  };
  static const Form forms[4] = {
      {16, 16, 430, 430, 100, 165}, {32, 32, 580, 680, 140, 310}, {64, 32, 960, 1120, 150, 460}, {64, 64, 1580, 1800, 0, 880}};
  int best = MM_16X16;
  uint64_t least = ~0ull;
  for (int i = 0; i < 4; i++) {
    Form f = forms[i];
    if (tiled && i == MM_32X32) f.one = f.odd = 700, f.per = 260;
    const uint64_t tiles = (((uint64_t)M + f.ta - 1) / f.ta) * (((uint64_t)N + f.tb - 1) / f.tb);
    const uint64_t one = vec ? f.one : f.odd, all = f.base + f.per * ((tiles + cu - 1) / cu);
    const uint64_t t = one > all ? one : all;
    if (t <= least) {  // of two equals the larger
      least = t;
      best = i;
    }
  }
  return best;
}
