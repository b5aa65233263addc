// Where a workgroup of a skinny product (gemv.hip, gemv2.hip) begins its K.
//
// Workgroup i begins kSkinnyTurn i steps of 64 into its K and goes round.  Begun at column 0, all of them read the same few columns of W at
// a time, and where a row is a multiple of 4 KB long these lie in a part of the memory's channels.  us in order -> turned (cold weights, N x K of
// 1 / 32 / 64 rows): 28672 x 4096 47.2 / 45.6 / 52.3 -> 41.2 / 42.6 / 50.0, 32768 x 4096 55.3 / 54.4 / 58.1 -> 53.0 / 48.6 / 52.8, 16384 x 8192
// 62.8 / 59.3 / 62.1 -> 44.6 / 47.3 / 49.5, 16384 x 2048 15.6 / 16.1 / 17.6 -> 13.4 / 14.4 / 16.3.  By two or four steps some are slower than in order
// (28672 x 4096 53.7, 16384 x 8192 68.1); other row lengths (1024, 1280, 3072) and fewer workgroups than CUs (11008 x 4096, 1 row
// 24.2 -> 25.0) gain nothing, and a K that is cut over workgroups does not either.
#pragma once
#include "launchers.h"

namespace shai {

constexpr int kSkinnyTurn = 3;

// (Kernels of their own: what the turn takes at a launch's start and each step is 0.25 us of the 7 of 32 x 5632 x 1024.)
inline bool skinny_turned(const GemmArgs& a, int kgroups) {
  return kgroups == 1 && a.ldw * (a.w_scale ? 1 : 2) % 4096 == 0 && a.N >= 256 * 64;
}

}  // namespace shai
