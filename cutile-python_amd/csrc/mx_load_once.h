// Where a kernel reads its largest operand non-temporally, so that its lines leave the caches first.  Plain C++ without device
// code, so that the rules can be checked on the host.
#pragma once
#include <stdint.h>

namespace mx {

// Quantiser: the input, from 48 Mi elements on (96 MB of 16-bit input, 192 MB of 32-bit).  By then a pass no longer finds its
// input, the codes of the pass before and its own in the 256 MB Infinity Cache, and the input's lines push out codes that the
// product behind still needs.  us, plain | non-temporal, 8192 columns -> E4M3 (product: 1024 columns):
//   bf16, just written by an element-wise kernel (its time included): 84 MB 47.7 | 47.8, 103 MB 61 | 57, 134 MB 78 | 73, 201 MB 121 | 110; with a
//     product behind 120 | 113, 148 | 137, 200 | 189; from memory, with a product behind 83 | 83, 97 | 97, 133 | 128, without one
//     28.5 | 26.4, 36.6 | 33.4, 53 | 49.  The very same input every time, written by nobody: 23.8 | 26.4, 30.2 | 33.5, 52 | 49.
//   fp32: 101 MB, just written 52 | 56, with a product behind 91 | 95; 168 MB 90 | 92, 153 | 150; 201 MB 112 | 110, 177 | 175, from
//     memory with a product behind 107 | 100; 235 MB 133 | 128, 201 | 195, 118 | 111.
// The codes are stored as ever: non-temporal stores win 3 % of the quantiser in front of them and cost the product that reads
// them next more (134 MB from memory 97 | 107 us for the two).
constexpr int64_t kQuantizeOnceElements = (int64_t)48 << 20;
inline bool quantize_loads_once(int64_t elements) { return elements >= kQuantizeOnceElements; }

}  // namespace mx
