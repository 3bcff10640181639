// nlg_softmax_form.h -- how many threads take a row of a softmax (plain C++:
// checked on the CPU).
#pragma once

#include <stdint.h>

// 64 (a wave, four rows a workgroup), 256 or 1,024 with the row in registers; 0:
// 256 that read it three times.  whole: rows of whole, aligned float4s.
//  * A wave has no barrier to wait at, and four times the rows of a workgroup of
//    256 in flight: 131,072 x 64 126 -> 33 us, 4,096 x 1,024 7.5 -> 6.2.  But past 256
//    columns its lanes issue four times the loads, and few rows wait for one: us, wave
//    / 256 threads, 20 rows of 1,021 3.6 / 3.0, 512 rows 4.1 / 3.5, 1,024 rows 4.4 /
//    4.1, 2,048 rows 5.6 / 5.5 (elements); 20 rows of 1,024 3.2 / 2.9, 512 rows 3.5 /
//    3.2, 1,024 rows 3.8 / 3.9 (float4s of rows on 64-byte lines; off them the wave
//    is ahead from some rows on: 1 row of 1,000 3.4 / 2.8, 20 rows 3.2 / 3.1, 512 rows
//    3.5 / 3.8).
//  * 1,024 threads hold up to 32,768 columns (20,000 x 12,000: 865 us read three
//    times -> 315), where the grid's x dimension, fewer than 2^32 threads, holds the rows.
inline uint32_t softmax_threads(uint32_t rows, uint32_t n, bool whole, uint32_t cu) {
  if (n <= 256) return 64;
  if (n <= 1024) return rows <= (whole ? n % 16 ? 8 : 2 * cu : 4 * cu) ? 256 : 64;
  if (n <= 8192) return 256;
  return n <= 32768 && rows < (1u << 22) ? 1024 : 0;
}
