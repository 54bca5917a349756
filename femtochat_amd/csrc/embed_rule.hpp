// Which way the embedding gradient takes into a fresh table: one kernel in which
// every workgroup looks at every token (embed_grad.hip), or a cleared table and
// one atomic per value.  Plain C++ (no HIP), so a host-only harness can check it.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace fc {

constexpr int kEgSlots = 128;  // table columns per workgroup at most
constexpr int kEgCols = 256;   // values of a column per workgroup, four per lane

// At least 256 groups (one per CU and value block), at most kEgSlots columns each.
inline int embed_groups(int vocab) {
  return vocab < 256 ? vocab : vocab <= 256 * kEgSlots ? 256 : (vocab + kEgSlots - 1) / kEgSlots;
}

// Estimates, in us, of the two ways (bf16 dy).  One kernel: 512 workgroups run at
// a time (62 KB of LDS each); a round of them takes 8 us and 1.2 us per 1000
// tokens, unless writing the table (6.5 TB/s) takes longer.  Atomics: two
// launches, the fill, and 77 values per ns where ids differ, with a cost per token
// for the frequent ones.  The lines cross where a large table of short columns
// makes many workgroups that each read all tokens, or where few tokens meet many.
// Measured, one kernel / atomics, ids as frequent as words:
//   8192 tokens:  V 32768 D 512 33 / 87, D 32 23 / 34, V 131072 D 512 73 / 113,
//                 D 128 37 / 49, D 32 33 / 33, V 262144 D 32 51 / 34,
//                 V 524288 D 32 86 / 37, D 64 87 / 50, D 128 94 / 73
//   65536 tokens: V 32768 D 32 129 / 232, V 524288 D 32 398 / 197, D 128 511 / 312
//   64 tokens:    V 32768 D 512 18 / 15, D 32 10 / 6.6, V 100000 D 32 16 / 7.4,
//                 V 1000 D 1280 17 / 9, V 524288 D 32 47 / 14
// While the workgroups all run at once the one kernel is taken at any number of
// tokens: the same bits on every call and one launch less on the host stand
// against at most 5 us.  Ids of equal frequency profit from atomics longer (8192
// tokens at V 32768, D 32 take 14 us, 10 with atomics).
inline bool embed_one_kernel_pays(int64_t N, int vocab, int D) {
  const double table = 4.0 * vocab * D;
  const double blocks = (double)embed_groups(vocab) * ((D + kEgCols - 1) / kEgCols);
  const double rounds = std::ceil(blocks / 512);
  const double one = std::max(8.0 * rounds, 8.0 + table / 6.5e6) + 1.2e-3 * (double)N * rounds;
  const double atomics = 8.0 + table / 6.0e6 + (double)N * (D + 128) / 77e3;
  return one <= atomics;
}

}  // namespace fc
