// Where a head_dim 64 softmax takes its per-key constants from (same values, same bits); no HIP
// dependency, so that a host program can evaluate it.
#pragma once
#include <stdint.h>

namespace sage {

// True: from LDS, false: as DPP broadcasts, for a launch of `blocks` blocks on `cus` compute units
// (<= 0: 256).
// As DPP broadcasts they cost a 4-cycle multiply per score instead of a 2-cycle one; as 16-byte LDS
// reads that a half-wave shares they cost the read's latency, which only other waves of the SIMD
// hide. So LDS once a launch keeps several blocks on every CU. Main loop on 256 CUs, DPP -> LDS: at
// 1 block per CU 62.7 -> 69.3 us, at 2 92.4 -> 93.1, at 2.5 128.0 -> 123.8, at 4 155.7 -> 153.0
// (N = 4096), 30 planes of 17550 2601 -> 2523, 3 of 65536 3582 -> 3515 (bf16 3313 -> 3263), 6 of
// 32768 1777 -> 1731. (On a card that throttled under its power cap LDS lost 1.3 % at 3 planes of
// 65536, 1.5 % at 6 of 32768 and 2.0 % at 3 of 32768 bf16, where others gained 1.9, 2.7 and 2.3.)
// A causal launch of fewer than ~3 blocks per CU ends in its longest tiles, each alone on its
// SIMDs: at 1.9 34.9 -> 38.3, at 3 67.7 -> 72.8, at 3.5 79.1 -> 75.3, at 3.75 84.9 -> 79.5. The key
// split's blocks: at 1 39.3 -> 42.1, at 1.25 53.6 -> 52.6 and 17.7 -> 17.6, at 2.5 72.0 -> 69.5.
// head_dim 128 (three blocks per CU, twice the matrix work a score) gained nothing.
inline bool consts_from_lds(int64_t blocks, int64_t cus, bool causal, bool split) {
  return blocks > (cus > 0 ? cus : 256) * (split ? 1 : causal ? 3 : 2);
}

}  // namespace sage
