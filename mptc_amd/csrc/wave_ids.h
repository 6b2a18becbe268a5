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

// How many ids a window of search area S has: every position of it, and of the
// columns ahead of it, distinct, in pairs of 64-id chunks; at S = 32 as many as
// LDS holds.  At least 384, of which wave 2 has 24: the words of the row above
// alone are up to 2 S + 4 at a time, and one that the other rows repeat keeps
// its id (with 128 ids at S = 4, 8 of them wave 2's, 1080p frames gave up).
constexpr int kWaveLook = 2;  // columns of the row above that may enter early
constexpr int kWaveIds = 1152, kWaveMinIds = 384;
constexpr __host__ __device__ int wave_id_count(int S) {
  const int ids = ((2 * S * (2 * S + 4 + kWaveLook) + 8) * 64 / kAboveIds + 127) / 128 * 128;
  return ids < kWaveMinIds ? kWaveMinIds : ids < kWaveIds ? ids : kWaveIds;
}

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

// Waves 1 and 2 look words up in one map while each may give an id of its own
// that no column holds to another word.  Each reads and writes the ids' words
// and the last columns they were seen at through a T: last, word, set_word,
// set_table, raise, and order, which keeps the wave's accesses on either side
// of it in that order.
//
// Whether id i (kNoId: none) is word w's.  Another wave's id has to be in use
// (seen at column `oldest` or later: then its word does not change in this
// step), and the column is read before the word: an id that its owner puts to
// use meanwhile has its new word by the time the new column shows.  The other
// way round, the old word with the new column passes for an id in use.
template <typename T>
__host__ __device__ __forceinline__ bool id_holds(const T& t, unsigned i, uint32_t w, bool own, int oldest) {
  const unsigned at = i != kNoId ? i : 0u;
  const int last = t.last(at);
  t.order();
  const uint32_t word = t.word(at);
  return i != kNoId && word == w && (own || last >= oldest);
}

// The owner's part, after set_word: the table of id `given`, then the column of
// `id` (another id of the same word where the wave found one).
template <typename T, typename Table>
__host__ __device__ __forceinline__ void id_publish(const T& t, unsigned given, const Table& table, unsigned id,
                                                    int column) {
  t.set_table(given, table);
  t.order();
  t.raise(id, column);
}

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
