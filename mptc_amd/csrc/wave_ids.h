// The ids that k_intra_wave (wave_kernels.h) gives the words of a window, as
// far as its waves share them inside a step: plain C++, so that the CPU can
// check them too.
#pragma once

#include <stdint.h>

namespace mptc {

constexpr unsigned kNoId = 0xFFFFu;
constexpr int kAboveIds = 60;   // of 64 ids, those of wave 1 (the others: wave 2)
constexpr int kWaveEval = 12;   // waves that evaluate
constexpr int kQuadIds = 384;   // up to so many ids, four lanes evaluate a word

// One more than the highest id in use, by the parity of the step and the wave
// (0: wave 1, 1: wave 2) that gave it out.  A step's readers take the count
// that the step before left, which nobody changes meanwhile: the waves that
// evaluate choose their ids by it, so they have to agree on it.  The words that
// the next block's window needs have their ids by then (column p + S enters in
// step p - 1).
struct IdCount {
  int n[2][2];
  __host__ __device__ __forceinline__ void publish(int step, int who, int count) { n[step & 1][who] = count; }
  __host__ __device__ __forceinline__ int before(int step) const {
    const int* c = n[(step & 1) ^ 1];
    return c[0] > c[1] ? c[0] : c[1];
  }
};

// The ids (below n_ids) that a lane of evaluating wave ev takes: first, then
// every stride-th.
struct EvalSplit {
  bool quad;  // four lanes an id
  int first, stride;
};
__host__ __device__ __forceinline__ EvalSplit eval_split(int n_ids, int ev, int lane) {
  EvalSplit s;
  s.quad = n_ids <= kQuadIds;
  s.first = s.quad ? ev * 16 + (lane >> 2) : ev * 64 + lane;
  s.stride = kWaveEval * (s.quad ? 16 : 64);
  return s;
}

}  // namespace mptc
