// Host choice between the two attention kernels (attention.hip).
#pragma once

#include <stdint.h>

namespace w8a8 {

constexpr int kAttnWaveQ = 32;     // queries per wavefront
constexpr int kAttnWaves = 4;      // wavefronts per workgroup (one per SIMD; two workgroups per CU)

// Whether the split kernel is the faster one, from both kernels' measured times
// in tenths of a microsecond: a round of split workgroups (one per CU) costs
// 4.9 us and 2.6 us for each step of its longest wave, the other kernel 14 us
// and 2.6 us a block while its grid fits the GPU. Both sides (us, plain and
// split): 16 heads x 353 x 1000 27.9 / 12.5, 8 x 64 x 32768 540 / 188, 28 x 350
// x 256 15.6 / 14.0, 28 x 700 x 256 19.5 / 20.1, 20 x 1000 x 512 26.1 / 22.2,
// 28 x 1100 x 512 28.7 / 31.0, 24 x 700 x 3000 68.7 / 65.3, 12 x 2000 x 2000
// 52.0 / 50.4, 16 x 2000 x 2000 55.0 / 65.5. A single block has nothing to
// split (28 x 700 x 128 9.0 / 20.2). The line lies at three rounds: there the
// split wins where the blocks fill its steps (4 x 6000 x 512 23.9 / 22.1, 1024
// 33.2 / 30.3, 2048 51.2 / 46.1) and loses where they do not (6 x 2752 x 357
// 18.4 / 21.6, 4 x 6000 x 768 28.5 / 30.2). The FP32 sums over key blocks take another
// order in each kernel, so a head's last bits depend on the call it is part of.
inline bool split_wins(int64_t nq, int64_t bh, int64_t nblk, int64_t cus) {
  if (nblk < 2) return false;
  const int64_t rounds = ((nq + kAttnWaveQ - 1) / kAttnWaveQ * bh + cus - 1) / cus;
  return rounds * (49 + 26 * ((nblk + kAttnWaves - 1) / kAttnWaves)) < 140 + 26 * nblk;
}

}  // namespace w8a8
