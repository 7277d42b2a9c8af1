// Which kernels route the copies of a mixture-of-experts layer.  Plain C++ without device code, so that the rule can be checked on the host.
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

}  // namespace mx
