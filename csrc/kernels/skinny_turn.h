// Where a workgroup of a skinny product (gemv.hip, gemv2.hip) begins its K.
//
// Workgroup i begins kSkinnyTurn i steps of 64 into its K and goes round.  Begun at column 0, all of them read the same few columns of W at
// a time, and where a row is a multiple of 4 KB long these lie in a part of the memory's channels.  us in order -> turned (cold weights, N x K of
// 1 / 32 / 64 rows):
//   gemv.hip (64 columns a workgroup) 16384 x 2048 16.0 / 15.8 / 17.3 -> 12.9 / 13.9 / 16.5, 16384 x 8192 63.6 / 60.4 / 65.5 -> 44.1 / 47.5 / 55.7,
//     28672 x 4096 44.4 / 46.6 / 53.9 -> 41.7 / 43.4 / 52.1, 32768 x 4096 55.4 / 53.4 / 57.5 -> 50.8 / 48.1 / 53.7, 128256 x 4096 190 / 194 / 229 ->
//     174 / 178 / 216; fp8 16384 x 4096 23.5 / 25.2 / 28.2 -> 23.4 / 24.6 / 27.4, 28672 x 8192 58.6 / 72.5 / 87.2 -> 54.5 / 69.0 / 83.9;
//   gemv2.hip (128 columns) 24576 x 4096 43.9 / 44.6 / 47.7 -> 38.4 / 40.4 / 43.2, 32768 x 4096 66.1 / 64.8 / 72.6 -> 45.7 / 46.8 / 49.5, 128256 x 4096
//     217 / 230 / 245 -> 165 / 178 / 195, and with fewer workgroups than CUs no gain and no loss: 16384 x 2048 21.2 / 21.9 / 24.3 -> 21.1 / 22.1 / 24.0,
//     20480 x 4096 43.3 / 45.0 / 48.6 -> 43.0 / 44.7 / 47.6.
// By two or four steps some are slower than in order (28672 x 4096 53.7, 16384 x 8192 68.1); other row lengths (1024, 1280, 3072) and fewer
// workgroups than CUs in gemv.hip (11008 x 4096, 1 row 24.2 -> 25.0) gain nothing, and a K that is cut over workgroups does not either.
#pragma once
#include "launchers.h"

namespace shai {

constexpr int kSkinnyTurn = 3;

// (Kernels of their own: what the turn takes at a launch's start and each step is 0.25 us of the 7 of 32 x 5632 x 1024.)
inline bool skinny_turned(const GemmArgs& a, int kgroups) {
  return kgroups == 1 && a.ldw * (a.w_scale ? 1 : 2) % 4096 == 0 && a.N >= 256 * 64;
}

}  // namespace shai
