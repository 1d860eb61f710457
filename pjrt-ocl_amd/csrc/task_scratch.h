// Scratch that the loader lays out per task (vmrt.cpp), and the matmul K split that
// does the work.  Host code; the scheduler mirrors both (scheduler.py
// `mma_effective_split`, `split_scratch_bytes`).
#pragma once
#include <algorithm>

#include "vm_abi.h"

namespace vm {

// The splits of a TOP_MMA task over K that do the work (vm_abi.h MmaRec::S): the
// task's, where the K loop that they shorten (0.022 us per f32 k of a 64-wide tile,
// 0.007 in 16 bits, three times that 128-wide) is worth publishing the partials and
// combining them, about 8 us (measured: 1.5 us to publish, 2 for the arrival, 4.4 to
// read the partials).  Else one: the first split's tile sums all of K.
inline uint32_t mma_effective_split(uint32_t S, uint32_t K, uint32_t T, uint32_t adt) {
  const bool h16 = adt == DT_BF16 || adt == DT_F16;
  const double per_k = (h16 ? 0.007 : 0.022) * (T == 128 ? 3 : 1);
  return S > 1 && K * (1.0 - 1.0 / S) * per_k < 8.0 ? 1 : S;
}

// Scratch bytes a task needs (0: none): a split decode attention keeps one
// partial (running max, sum, hd channels) per split and head, and one arrival
// counter per head; a split column reduction 64 partials per split and block of
// outputs, and one counter per block; a matmul whose K split does the work one f32
// partial tile per split and output tile, and one arrival counter per output tile.
inline uint64_t task_scratch_bytes(const Task& t, uint32_t mma_t) {
  if ((t.tile_op & 0xFF) == TOP_MMA) {
    const uint32_t code = (t.p[3] >> 24) & 0xF;
    const uint64_t T = code == 1 ? 64 : code == 2 ? 128 : code == 3 ? 256 : mma_t;
    const uint64_t S = mma_effective_split(1u << (t.p[3] >> 28), t.p[2], uint32_t(T), (t.tile_op >> 16) & 0xFF);
    if (S <= 1) return 0;
    const uint64_t tiles = ((t.p[0] + T - 1) / T) * ((t.p[1] + T - 1) / T) * std::max<uint64_t>(1, t.p[3] & 0xFFFFFF);
    // a 256-wide tile runs as four 128-wide ones, each with a counter of its own
    return (tiles * S * T * T + tiles * (T == 256 ? 4 : 1)) * 4;
  }
  if ((t.tile_op & 0xFF) == TOP_RED_STRIDED && t.p[4] > 1) {
    const uint64_t blocks = (uint64_t(t.p[0]) + 63) / 64;
    return (blocks * t.p[4] * 64 + blocks) * 4;
  }
  if ((t.tile_op & 0xFF) == TOP_ARGMAX_SEG && t.p[3] > 1) return (2ull * t.p[0] * t.p[3] + t.p[0]) * 4;
  if ((t.tile_op & 0xFF) == TOP_DECODE_ATTN && (t.p[4] >> 16) > 1) {
    const uint64_t H = t.p[4] & 0xFFFF, S = t.p[4] >> 16, hd = t.p[5] & 0xFFFF;
    return (H * S * (hd + 2) + H) * 4;
  }
  return 0;
}

}  // namespace vm
