// Where a kernel reads its largest operand non-temporally, so that its lines leave the caches first.  Plain C++ without device
// code, so that the rules can be checked on the host.
#pragma once
#include <stdint.h>

namespace mx {

// Quantiser: the input, from 48 Mi elements on (96 MB of 16-bit input, 192 MB of 32-bit).  By then a pass no longer finds its
// input, the codes of the pass before and its own in the 256 MB Infinity Cache, and the input's lines push out codes that the
// product behind still needs.  us, plain | non-temporal, 8192 columns -> E4M3 (product: 1024 columns):
//   bf16, just written by an element-wise kernel (its time included): 103 MB 61 | 57, 134 MB 78 | 73, 201 MB 121 | 110;
//     with a product behind 120 | 113, 148 | 137, 200 | 189; from memory, with a product behind 83 | 83, 97 | 97, 133 | 128, without one
//     28.5 | 26.4, 36.6 | 33.4, 53 | 49.  The very same input every time, written by nobody: 23.8 | 26.4, 30.2 | 33.5, 52 | 49.
//     84 MB is the same either way (just written 47.7 | 47.8, with a product behind 100 | 100.5).
//   fp32: 101 MB, just written 52 | 56, with a product behind 91 | 95; 168 MB 90 | 92, 153 | 150; 201 MB 112 | 110, 177 | 175,
//     from memory with a product behind 107 | 100; 235 MB 133 | 128, 201 | 195, 118 | 111.
// The codes are stored as ever: non-temporal stores win 3 % of the quantiser in front of them and cost the product that reads
// them next more (134 MB from memory 97 | 107 us for the two).
constexpr int64_t kQuantizeOnceElements = (int64_t)48 << 20;
inline bool quantize_loads_once(int64_t elements) { return elements >= kQuantizeOnceElements; }

// Weights: from 96 MB a launch on.  Two such matrices do not fit into the 256 MB Infinity Cache with what lies between, so that a
// loop over a model's layers finds none of their lines again, and the plain policy costs 7 - 10 % (28672 x 8192 FP8, 8 rows,
// 45 -> 40 us; FP4, 32 rows, 25.9 -> 23.7).  Smaller ones gain as much where they come from memory (14336 x 4096 FP8, 8 rows,
// 16.1 -> 14.7) and lose more where two or three of them take turns (11.5 -> 14.3).  (Two alone that take turns with
// nothing between still gain from the cache at 117 MB, 14336 x 8192 FP8 at 32 rows 21.8 against 24.6, three no longer, 27.7 against
// 24.9; at 235 MB two do not, 48.7 against 45.2.)  Of a view or of overlapping rows the bytes that are read count, once each.
// ... rows of whole 128-byte lines only.  A line that two rows share is asked for by two waves, the second time after it has gone
// (25600 x 11392 MXFP4, rows of 44.5 lines: 33 rows 51.0 -> 52.6 us, 8 rows 38.9 -> 39.3).
// The decode kernel keeps to this where it runs slab by slab of 32 rows, and where W starts inside a line, too: 28672 x 8192 at 33,
// 64 and 128 rows 48.2 | 46.0, 49.6 | 46.6, 96 | 92 us (the same matrix again and again 45 | 42, 46 | 43, 92 | 87), 16 bytes into
// a line at 8 and 32 rows 24.6 | 23.3, 26.0 | 23.9.
constexpr int64_t kLoadOnceBytes = (int64_t)96 << 20;
inline bool weights_load_once(int64_t rows, int64_t row_bytes, int64_t pitch) {
  return rows * (row_bytes < pitch ? row_bytes : pitch) >= kLoadOnceBytes && pitch % 128 == 0;
}

// The streaming kernels' load instructions take 128 bytes of a row: W has to start at a line as well (`at`: its address, and the
// pitch of its experts), or a line is asked for twice by the same wave, a stage apart (16 bytes into a line, 28672 x 8192 FP8
// at 8, 32, 64 rows 57 | 68, 63 | 73, 73 | 80 us; FP4 35 | 37.5, 41 | 43, 48 | 50).  And one row tile: with several, neighbouring
// workgroups share W through L2, which keeps nothing of it then (28672 x 8192 FP8, 65 and 128 rows 76 | 102, 88 | 98; FP4 65 | 77,
// 78 | 92; 14336 x 8192 FP8, 65 and 256 rows 41 | 52, 74 | 88; 7168 x 28672 FP4, 33 rows 38.5 | 50.5).
inline bool stream_loads_once(int64_t rows, int64_t row_bytes, int64_t pitch, uint64_t at, int row_tiles) {
  return row_tiles == 1 && at % 128 == 0 && weights_load_once(rows, row_bytes, pitch);
}

}  // namespace mx
