// Which kernels route the copies of a mixture-of-experts layer, and where streaming ends.  Plain C++ without device code, so that the rules can be checked on the host.
#pragma once
#include <stdint.h>

namespace mx {

// One workgroup sorts the ids (moe_align_one_kernel) as long as its ballots, one for each bit of an expert's number and 1024 ids, take less than
// the second launch and the round trips of several workgroups.  us, several | one, launches included, replayed from a graph: 8192
// ids, 8 experts 14.0 | 9.5, 256 experts 25.2 | 20.2; 12288 ids, 8 experts 14.2 | 11.7, 64 experts 18.1 | 16.0, 256 experts 24.1 | 23.8; 14336 ids, 8
// experts 14.7 | 13.1, 64 experts 19.0 | 17.5, 256 experts 24.2 | 25.7; 16384 ids, 8 experts 14.7 | 14.0, 16 experts 16.0 | 15.4, 32
// experts 17.9 | 19.6, 64 experts 19.0 | 19.2, 128 experts 20.4 | 22.6, 256 experts 23.9 | 27.1.
constexpr int kAlignOneIds = 16384, kAlignOneExperts = 256;   // most that the kernel takes
inline bool moe_align_in_one_workgroup(int64_t ids, int64_t experts) {
  return ids > 0 && experts > 0 && experts <= kAlignOneExperts && ids <= (experts <= 16 ? kAlignOneIds : experts <= 64 ? 14336 : 12288);
}

// Whether the copies of a layer (`ids`, top-k of `experts`) leave streaming, where row tiles are the alternative.  Streaming reads an expert's weights
// once for 32 rows, so it is behind as soon as one expert has more, and mostly ahead before: beyond 24 rows on average that depends on how far random
// routing spreads, sqrt(rows * (1 - k / E)), not at all with k = E, and with more than eight experts one of them has got more.  The line is 1.5 of
// these below 32.  us per layer, mean of eight routings, streamed | row tiles, 24.5, 26, 28 and 30 rows on average: 4 of 4 experts of 4096 x 4096 FP8 - ,
// 46 | 64, 47 | 64, 47 | 64, of 2048 x 14336 FP4 - , 55 | 68, 55 | 70, 55 | 69, FP8 - , 92 | 90, 94 | 90, 94 | 90; 2 of 4 of 4096 x 4096 FP8 48 | 62, 46 | 62,
// 50 | 62, 62 | 63, FP4 39 | 40, 36 | 40, 41 | 41, 52 | 41, of 2048 x 14336 FP8 94 | 86, 93 | 87, 96 | 86, 109 | 87; 4 of 8 of 2048 x 4096 FP8 47 | 56, 52 |
// 57, 57 | 57, 62 | 57; 2 of 8 of 2048 x 4096 FP8 50 | 55, 54 | 55, 60 | 55, 62 | 55, of 4096 x 14336 FP8 268 | 262, 284 | 262, 296 | 264, 314 | 265; 1 of 2 of
// 2048 x 14336 FP8 48 | 51, 51 | 52, 54 | 51, 59 | 52; 2 of 16 of 4096 x 4096 FP8 173 | 182, 186 | 183, 192 | 183, FP4 112 | 99, 120 | 99, 125 | 100.
inline bool moe_leaves_streaming(int64_t ids, int64_t experts, int64_t k) {
  const int64_t room = 32 * experts - ids;
  return ids > 24 * experts && (experts > 8 || room < 0 || 4 * room * room < 9 * ids * (experts - k));
}

}  // namespace mx
