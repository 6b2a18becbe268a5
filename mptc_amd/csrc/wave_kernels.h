// The exact intra search in dependency order: k_intra_wave takes every block's
// intra decision once, from the final words of its causal window, instead of
// re-evaluating candidates until the words of the frame stop changing
// (k_intra_dense and the fixpoint passes of batch_kernels.h).
//
// Measured, whole frames (1080p intra, MI355X): S = 8, threshold 8: passes
// 23.3 ms, this 4.7; S = 32, threshold 32: 770 ms, 11.8.  A step takes 1.1-1.5
// us (wave 1's lookups and the wait for the row above bound it).
//
// What bounds the passes: at thresholds above about 4 most blocks reuse a
// word, a changed word is re-tried on all 4S^2 blocks that see it, and the
// words change 8-28 times before they settle.  In dependency order a word is
// tried once, and a window holds few distinct words (1080p, threshold 8: 90 of
// 248 positions at S = 8, 460 of 4032 at S = 32; threshold 32: 43 and 50),
// because most blocks repeat one.  So a block evaluates the distinct words of
// its window, not its positions.
//
// Layout.  A workgroup owns one block row of one frame and walks it from left
// to right; a window reaches S - 1 columns to the right in the rows above, so
// the row above is ahead by S + 2 columns and a frame has about bw / (S + 2)
// rows in flight.  The time is the dependency chain, bw + (S + 2) bh steps, so
// the step is split over waves that work side by side, one step = one barrier
// (a wave alone issues an instruction about every nine cycles, so each role's
// instruction count is what a step costs):
//   wave 0    the decision of block p from the evaluated words
//   waves 1,2 words entering the window, from the second row above on and from
//             the row above (which they wait for): each word gets its id (LDS
//             hash; equal words share an id)
//   wave 3    the window's step to block p + 1
//   others    evaluate every live word against block p + 1, four lanes a word
//
// The window in LDS.  gid[row][column ring] holds the ids, rowset[chunk][row]
// the set of ids that a window row holds (a bit per id), lastcol[id][row] the
// last column at which it does (a column leaving the window clears the bit if
// it is that one).  The selection rule (codec/dxt_image.cpp:697-708) then needs
// no scan of the positions: with a delta <= 0 in the window, the last row (in
// scan order) after the first such row that holds a negative one gives the
// selection, else that first row; without one, the nearest row that holds a
// word of the smallest delta.  A lane per row tests its set against the ids'
// comparison masks; one row is then searched for the first such position.
// An id belongs to its word until the last column it was seen at has left the
// window (lastany).  The word -> id map keeps one id in each of a word's two
// buckets; a word that others have driven out of both gets a second id, which
// costs an evaluation and changes nothing else.
//
// Rows hand words on through fin[g] (bit 63: final; bits 32-62: the block whose
// starting word it is, for the word's table; low half: the word), read and
// written with agent-scope atomics, data and flag in one 64-bit word, so no
// fence is needed.  Rows are taken from a ticket counter in raster order: a
// row waits only for rows of smaller tickets, whose workgroups run already.
// Every wait is bounded (kWaveSpin); a row that gives up, or a window with more
// distinct words than ids, sets wave_fail, every other row then leaves, and the
// host runs the fixpoint passes.  It does so too where k_wave_sample finds that
// few blocks would reuse a word.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_kernels.h"
#include "wave_ids.h"

namespace mptc {

constexpr int kWaveMaxS = 32;           // a lane per window row and per window column
constexpr int kWaveSpin = 1 << 22;      // polls (about a microsecond each) before a wait gives up
constexpr int kWaveRoles = 4;           // the waves above
constexpr int kWaveWaves = kWaveRoles + kWaveEval;
constexpr int kProdBytes = 16 * 96;     // a block's products: per pixel, index value and channel, (p a, p b)
constexpr int kRawCols = 16;            // columns of the rows above staged for wave 1
constexpr int kPxBlocks = 16;           // blocks staged at once for the evaluation

// Sizes that follow from S; offsets of the LDS arrays in bytes.
struct WaveDims {
  int ring, look, ids, bucket_log;  // ring is a power of two
  int o_tab, o_rows, o_prod, o_wr, o_raw, o_px, o_last, o_e, o_head, o_gid, o_lcol, bytes;
};

constexpr __host__ __device__ int wave_take(int& o, int bytes) {
  const int at = o;
  o += (bytes + 15) / 16 * 16;
  return at;
}

constexpr __host__ __device__ WaveDims wave_dims(int S) {
  WaveDims d{};
  d.ring = 16;
  while (d.ring < 2 * S + 8) d.ring *= 2;
  // columns of the row above that may enter early: a column's ring slot is
  // written only after the column a ring before it left the window
  d.look = kWaveLook;
  d.ids = wave_id_count(S);
  d.bucket_log = S <= 8 ? 10 : 12;
  int o = 0;
  d.o_tab = wave_take(o, 16 * d.ids);
  d.o_rows = wave_take(o, 8 * d.ids);
  d.o_prod = wave_take(o, 2 * kProdBytes);
  d.o_wr = wave_take(o, 8 * d.ids);
  d.o_raw = wave_take(o, 8 * 2 * S * kRawCols);
  d.o_px = wave_take(o, 4 * 2 * 5 * 64);
  d.o_last = wave_take(o, 4 * d.ids);
  d.o_e = wave_take(o, 2 * 2 * d.ids);
  d.o_head = wave_take(o, 2 << d.bucket_log);
  d.o_gid = wave_take(o, 2 * 2 * S * d.ring);
  d.o_lcol = wave_take(o, 2 * S * d.ids);
  d.bytes = o;
  return d;
}
static_assert(wave_dims(kWaveMaxS).bytes <= 159 * 1024, "the window fits the LDS of a compute unit");  // 150 KB

// Barrier over the workgroup's LDS: outstanding global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders one wave's LDS accesses across lanes (they execute in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The id tables in LDS, as wave_ids.h accesses them.
struct WaveIds {
  int* lastany;
  uint64_t* wr;
  float4* tab;
  __device__ __forceinline__ int last(unsigned i) const { return lastany[i]; }
  __device__ __forceinline__ uint32_t word(unsigned i) const { return (uint32_t)wr[i]; }
  __device__ __forceinline__ void set_word(unsigned i, uint64_t v) const { wr[i] = v; }
  __device__ __forceinline__ void set_table(unsigned i, const float4& t) const { tab[i] = t; }
  __device__ __forceinline__ void raise(unsigned i, int column) const { atomicMax(&lastany[i], column); }
  __device__ __forceinline__ void order() const { lds_order(); }
};

template <int kCtrl, int kRows>
__device__ __forceinline__ int dpp_min(int v) {
  return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, kCtrl, kRows, 0xf, false));
}
__device__ __forceinline__ int wave_min(int v) {
  v = dpp_min<0x111, 0xf>(v);
  v = dpp_min<0x112, 0xf>(v);
  v = dpp_min<0x114, 0xf>(v);
  v = dpp_min<0x118, 0xf>(v);
  v = dpp_min<0x142, 0xa>(v);
  v = dpp_min<0x143, 0xc>(v);
  return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ uint64_t fin_load(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool fin_is(uint64_t v) { return (int64_t)v < 0; }
__device__ __forceinline__ uint32_t fin_root(uint64_t v) { return (uint32_t)(v >> 32) & 0x7FFFFFFFu; }

template <int kCtrl>
__device__ __forceinline__ uint32_t quad_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, false);
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]

// One channel of the block that a quad of lanes tries words on (lanes 0-2 of
// the quad: r, g, b; lane 3 repeats b and adds nothing).
struct ChannelEval {
  uint32_t pc[4];      // the channel of pixels 4j..4j+3, one byte each
  uint32_t sq;         // sum of squares
  uint32_t prod_off;   // 8 x the channel, in each byte
  uint32_t mask565;    // the channel's bits that Pack565 keeps (lane 3: none)
  uint32_t shift565;   // its place there: (v & mask) << shift >> 3
  uint32_t snap_off;   // its snap table
  uint32_t own;        // the block's own word and error
  int orig;
};

// eval_candidate with the three channels on three lanes: the same operations
// per channel in the same order, the products p a and p b of the least-squares
// sums (one rounding each, as there) read from the block's table `prod`.
// Every lane of the quad returns the delta as stored in E.
__device__ __forceinline__ int eval_candidate_quad(const ChannelEval& ce, uint32_t c, const float4& t,
                                                   const uint8_t* __restrict__ snap, const char* __restrict__ prod) {
  uint32_t sel[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) sel[j] = spread_indices(c, j);
  float ax = 0.0f, bx = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t s24 = ((sel[j] << 4) + (sel[j] << 3)) + ce.prod_off;  // byte n: 24 index + 8 channel <= 88
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const float2 w = *reinterpret_cast<const float2*>(prod + ((s24 >> (8 * n)) & 0xFFu) + 96 * (4 * j + n));
      if (j == 0 && n == 0) {
        ax = w.x;
        bx = w.y;
      } else {
        ax += w.x;
        bx += w.y;
      }
    }
  }
  const float asq = t.x, bsq = t.y, ab = t.z, f = t.w;
  const float s1 = f * (ax * bsq - bx * ab), s2 = f * (bx * asq - ax * ab);
  uint32_t v1, v2;
  if (fabsf(f) <= kSmallF) {
    v1 = snap[ce.snap_off + quant255_small(s1)];
    v2 = snap[ce.snap_off + quant255_small(s2)];
  } else {
    v1 = snap[ce.snap_off + quant255(s1)];
    v2 = snap[ce.snap_off + quant255(s2)];
  }
  uint32_t k1 = ((v1 & ce.mask565) << ce.shift565) >> 3, k2 = ((v2 & ce.mask565) << ce.shift565) >> 3;
  k1 |= quad_dpp<kQuadXor1>(k1);
  k2 |= quad_dpp<kQuadXor1>(k2);
  k1 |= quad_dpp<kQuadXor2>(k1);
  k2 |= quad_dpp<kQuadXor2>(k2);
  const uint32_t pal = v1 | (v2 << 8) | (div3(2 * v1 + v2) << 16) | (div3(v1 + 2 * v2) << 24);
  uint32_t dot = 0, qq = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t q = byte_gather(pal, sel[j]);
    dot = __builtin_amdgcn_udot4(ce.pc[j], q, dot, false);
    qq = __builtin_amdgcn_udot4(q, q, qq, false);
  }
  uint32_t sse = ce.mask565 ? ce.sq - 2u * dot + qq : 0u;
  sse += quad_dpp<kQuadXor1>(sse);
  sse += quad_dpp<kQuadXor2>(sse);
  const int e = (int)sat16((int)(sse / 48u) - ce.orig);
  return c == ce.own ? 0 : k1 > k2 ? e : (int)kNoCand;
}

// A word's two buckets in the word -> id map.
__device__ __forceinline__ uint32_t wave_hash(uint32_t w, int log) { return (w * 0x9E3779B1u) >> (32 - log); }
__device__ __forceinline__ uint32_t wave_hash2(uint32_t w, int log) { return ((w ^ w >> 15) * 0x85EBCA6Bu) >> (32 - log); }

// Global loads through pointers kept in memory (a generic pointer's load would
// also count as an LDS access).
template <typename T>
__device__ __forceinline__ T gload(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}

// Whether the blocks of a batch reuse words widely enough for k_intra_wave: n
// blocks spread over it take their first decision (from the starting words, as
// k_intra_dense), a workgroup each; smp counts those that search and those whose
// word changes, in 16 slots (one word for all workgroups: 28 us at 1,024 blocks).  Where few change the fixpoint passes
// settle after a handful of rounds, while the wave's time is its chain of steps
// whatever the frame holds (1080p, S = 8, threshold 8: noise, 0 % changed, passes
// 0.41 ms, wave 5.6; 24 grey levels, 11 %, 1.9 and 5.7; gradients with noise,
// 96 %, 21.5 and 4.7).  A thread takes up to four positions (S = 32: 16 of them,
// one after the other, 37 us; four, 28; S = 8, one, 9.7 us).
__global__ void __launch_bounds__(1024) k_wave_sample(const FrameDev* __restrict__ fr, const uint8_t* __restrict__ sid,
                                                     int total, int n, int S, int thr,
                                                     const uint64_t* __restrict__ own, const uint8_t* __restrict__ need,
                                                     const uint32_t* __restrict__ cw, const float4* __restrict__ ctab,
                                                     const int* __restrict__ orig, DevStats* __restrict__ st) {
  __shared__ uint8_t s_snap[512];
  __shared__ float2 s_ab[4];
  __shared__ int16_t s_e[4 * kWaveMaxS * kWaveMaxS];
  const int i = (int)blockIdx.x;
  // block i of n: somewhere in the i-th part of the batch, so that no stride meets the frames' widths
  const uint64_t at = ((uint64_t)i << 16) + (((uint32_t)i * 0x9E3779B1u) >> 16);
  const int g = n == total ? i : (int)(at * (uint64_t)total / ((uint64_t)n << 16));
  if (need[g] == 0) return;  // the whole workgroup
  load_lds_tables(s_snap, s_ab);  // ends with a barrier
  const FrameDev& d = fr[sid[g]];
  const int k = g - d.base, bw = d.bw, bx = k % bw, by = k / bw, W2 = 2 * S, slots = W2 * W2;
  BlockPx px;
  load_block(d.rgb, d.width, bx, by, px);
  BlockEval be;
  make_block_eval(px, own[g], orig[g], be);
  for (int p = threadIdx.x; p < slots; p += blockDim.x) {
    const int r = p / W2, t = p - r * W2, j = by - r, x = bx + S - 1 - t;
    int e = kNoCand;
    if (j >= 0 && x >= 0 && x < bw && !(r == 0 && t < S)) {
      const int q = d.base + j * bw + x;
      const float4 t4 = ctab[q];
      const CandResult res = eval_candidate<false>(be, cw[q], CandTab{t4.x, t4.y, t4.z, t4.w}, s_snap, s_ab);
      if (res.valid) e = sat16(res.err);
    }
    s_e[p] = (int16_t)e;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  // the selection rule (codec/dxt_image.cpp:697-708): the last row after that of the first delta <= 0 which holds a
  // negative one gives the selection, else that delta; without one, the smallest delta's first position
  const int lane = (int)threadIdx.x;
  constexpr int kNone = 0x7fffffff;
  static_assert(4 * kWaveMaxS * kWaveMaxS <= 1 << 12, "a position fits 12 bits");
  int le0 = kNone, least = kNone;
  for (int p = lane; p < slots; p += 64) {
    const int e = s_e[p];
    if (e <= 0) le0 = min(le0, p);
    if (e != kNoCand) least = min(least, ((e + 32768) << 12) | p);
  }
  int sel = wave_min(le0);
  if (sel != kNone) {
    const int r1 = sel / W2;
    int last = kNone;  // the row, negated
    for (int p = lane; p < slots; p += 64)
      if (s_e[p] < 0 && p / W2 > r1) last = min(last, -(p / W2));
    last = wave_min(last);
    if (last != kNone) {
      int pos = kNone;
      for (int p = lane; p < slots; p += 64)
        if (s_e[p] < 0 && p / W2 == -last) pos = min(pos, p);
      sel = wave_min(pos);
    }
  } else {
    const int m = wave_min(least);
    sel = m != kNone && (m >> 12) - 32768 <= thr ? m & 4095 : kNone;
  }
  if (lane != 0) return;
  bool changed = false;
  if (sel != kNone) {
    const int r = sel / W2, x = bx + S - 1 - (sel - r * W2);
    changed = cw[d.base + (by - r) * bw + x] != cw[g];
  }
  atomicAdd(&st->smp[i % kSmpSlots * kSlot32], changed ? 0x10001u : 1u);
}

// Least share of blocks that change, of those of the sample that search (the
// batch's rule, in percent) and of the whole sample: k_intra_wave takes all
// rows of a batch, also those of frames in which few blocks search.
struct WaveRule {
  int sampled, pct, pct_all;
};

// rows: (row << 6 | frame) in ticket order, every row after the row above it;
// null: one frame, rows in order.  fin: per block, its starting word (of the
// block itself), final where the block does not search; ctab: the starting
// words' tables; rec: per block, own word, own error, whether it searches
// (all from k_intra_prep).  kS: the search area, or 0 (S_ is it).
//
// A role's loads are used several steps after they were issued, never moved
// between registers meanwhile (that would wait for them), and wave 0 loads
// nothing from global memory: waiting for a load would wait for its stores.
template <int kS>
__global__ void __launch_bounds__(64 * kWaveWaves) k_intra_wave(
    const FrameDev* __restrict__ fr, const int* __restrict__ rows, int S_, int thr, const uint4* __restrict__ rec,
    const float4* __restrict__ ctab, uint64_t* fin, uint64_t* __restrict__ dec, DevStats* __restrict__ st,
    unsigned int* __restrict__ conv, WaveRule rule) {
  {  // not worth it (k_wave_sample): the passes take the batch
    uint32_t smp = 0;
#pragma unroll
    for (int i = 0; i < kSmpSlots; ++i) smp += st->smp[i * kSlot32];
    const int changed = (int)(smp >> 16), need = (int)(smp & 0xFFFFu);
    if (changed * 100 < rule.pct * need || changed * 100 < rule.pct_all * rule.sampled) {
      if (blockIdx.x == 0 && threadIdx.x == 0 && conv) {
        *reinterpret_cast<volatile unsigned int*>(conv) = 1u;
        __threadfence_system();
      }
      return;
    }
  }
  extern __shared__ __align__(16) unsigned char s_mem[];
  __shared__ uint8_t s_snap[512];
  __shared__ float2 s_ab[4];
  __shared__ int s_ticket;
  __shared__ IdCount s_count;
  __shared__ int s_read[2];        // by step parity: the step whose row sets wave 0 has read
  __shared__ int s_fail[2];        // by step parity: set in a step, read in the next
  __shared__ uint32_t s_blk[4][16];  // block b & 3: its 12 channel words, own word, own error, need
  const int S = kS ? kS : S_;
  const WaveDims D = wave_dims(S);
  float4* tab = reinterpret_cast<float4*>(s_mem + D.o_tab);
  unsigned long long* rowset = reinterpret_cast<unsigned long long*>(s_mem + D.o_rows);  // [chunk][window row]
  char* prod = reinterpret_cast<char*>(s_mem + D.o_prod);                                // by block parity
  uint64_t* wr = reinterpret_cast<uint64_t*>(s_mem + D.o_wr);  // the id's word, its block << 32
  uint64_t* raw = reinterpret_cast<uint64_t*>(s_mem + D.o_raw);
  uint32_t* px = reinterpret_cast<uint32_t*>(s_mem + D.o_px);
  int* lastany = reinterpret_cast<int*>(s_mem + D.o_last);
  int16_t* E = reinterpret_cast<int16_t*>(s_mem + D.o_e);  // [step parity][id]: delta of the id's word
  uint16_t* head = reinterpret_cast<uint16_t*>(s_mem + D.o_head);
  uint16_t* gid = reinterpret_cast<uint16_t*>(s_mem + D.o_gid);
  uint8_t* lastcol = reinterpret_cast<uint8_t*>(s_mem + D.o_lcol);
  const WaveIds ids{lastany, wr, tab};

  const int lane = (int)(threadIdx.x & 63);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int W2 = 2 * S, rmask = D.ring - 1;

  if (threadIdx.x == 0) {
    s_ticket = (int)atomicAdd(&st->wave_ticket, 1u);
    s_count = IdCount{};
    s_fail[0] = s_fail[1] = 0;
    s_read[0] = s_read[1] = -4;
  }
  for (int i = threadIdx.x; i < D.ids; i += blockDim.x) {
    rowset[i] = 0ull;
    lastany[i] = -(1 << 30);
    E[i] = E[D.ids + i] = kNoCand;
  }
  for (int i = threadIdx.x; i < 1 << D.bucket_log; i += blockDim.x) head[i] = (uint16_t)kNoId;
  for (int i = threadIdx.x; i < W2 * D.ring; i += blockDim.x) gid[i] = (uint16_t)kNoId;
  // an entry not fetched yet names no block (wave 1 reads one ahead)
  for (int i = threadIdx.x; i < W2 * kRawCols; i += blockDim.x) raw[i] = 0ull;
  load_lds_tables(s_snap, s_ab);  // ends with a barrier

  const int tk = __builtin_amdgcn_readfirstlane(s_ticket);
  const int rw = rows ? __builtin_amdgcn_readfirstlane(rows[tk]) : tk << 6;
  const FrameDev& d = fr[rw & 63];
  const int y = rw >> 6, bw = d.bw, base = d.base, row0 = base + y * bw;
  const bool lane_row = lane < W2 && y - lane >= 0;  // lane = window row: block row y - lane

  auto fail_at = [&](int p) { s_fail[p & 1] = 1; };
  // End of step p: every wave passes the barrier; true to leave (the step
  // before failed somewhere; `f` was read in this step).
  auto step_end = [&](int f) -> bool {
    lds_barrier();
    return f != 0;
  };
  auto give_up = [&](int& spin) -> bool {
    if (++spin > kWaveSpin) return true;
    return (spin & 15) == 0 && __hip_atomic_load(&st->wave_fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
  };
  // Waits until the second row above has passed the first window (the row
  // above then starts, and this row's turn is S + 2 steps away): one word, rarely
  auto turn = [&]() -> bool {
    if (y < 2) return true;
    for (int spin = 0; !fin_is(fin_load(fin + row0 - 2 * bw + min(S, bw) - 1));) {
      if (give_up(spin)) return false;
      __builtin_amdgcn_s_sleep(16);
    }
    return true;
  };
  auto enter = [&](unsigned id, int c) {  // the lane's row holds id at column c
    lastcol[id * W2 + lane] = (uint8_t)c;
    atomicOr(&rowset[(id & ~63u) + lane], 1ull << (id & 63u));
  };
  auto leave = [&](unsigned id) { atomicAnd(&rowset[(id & ~63u) + lane], ~(1ull << (id & 63u))); };

  // Waves 1 and 2 insert, in step p, column p + S + 1 of the rows above and the
  // starting word of column p + 1; before step -1, the columns up to S - 1: the
  // window of block 0.
  // Two barriers come before the steps: the staged pixels', and the window's.
  if (wv == 0) {
    // ---- the decisions -------------------------------------------------------
    lds_barrier();
    lds_barrier();
    for (int p = -1; p < bw; ++p) {
      const int f = s_fail[(p & 1) ^ 1];
      if (p >= 0) {
        const int16_t* Ep = E + (p & 1) * D.ids;
        const uint32_t need = s_blk[p & 3][14];
        const unsigned start_id = gid[p & rmask];
        const unsigned id_out = p >= S ? gid[(p - S) & rmask] : kNoId;  // leaves row 0
        const int nu = __builtin_amdgcn_readfirstlane(s_count.before(p));
        unsigned sel_id = start_id;
        bool bad = false;
        if (__builtin_amdgcn_readfirstlane((int)need) != 0) {
          uint64_t accl = 0, accn = 0;
          int mn = 0x7fffffff;
          for (int i0 = 0; i0 < nu; i0 += 128) {
            const int e0 = Ep[i0 + lane], e1 = Ep[i0 + 64 + lane];
            const uint64_t r0 = rowset[i0 + lane], r1 = rowset[i0 + 64 + lane];
            accl |= (r0 & __ballot(e0 <= 0)) | (r1 & __ballot(e1 <= 0));
            accn |= (r0 & __ballot(e0 < 0)) | (r1 & __ballot(e1 < 0));
            mn = min(mn, min(e0, e1));  // used where none is <= 0
          }
          const unsigned long long rows_l = __ballot(accl != 0);
          int R = -1, lo = -32768, hi = 0;  // the selected row and the range of its deltas
          if (rows_l != 0) {
            const int r1 = __builtin_ctzll(rows_l);
            const unsigned long long rows_n = __ballot(accn != 0) & ~((2ull << r1) - 1ull);  // rows after r1
            R = r1;
            if (rows_n) {
              R = 63 - __builtin_clzll(rows_n);
              hi = -1;
            }
          } else {
            // the smallest delta that some row holds (ids ahead of the window,
            // and starting words not taken, have a delta but no row)
            int m = wave_min(mn);
            while (m <= thr) {
              uint64_t at = 0;
              int more = 0x7fffffff;
              for (int i0 = 0; i0 < nu; i0 += 128) {
                const int e0 = Ep[i0 + lane], e1 = Ep[i0 + 64 + lane];
                at |= (rowset[i0 + lane] & __ballot(e0 == m)) | (rowset[i0 + 64 + lane] & __ballot(e1 == m));
                more = min(more, min(e0 > m ? e0 : 0x7fffffff, e1 > m ? e1 : 0x7fffffff));
              }
              const unsigned long long rows_m = __ballot(at != 0);
              if (rows_m != 0) {
                R = __builtin_ctzll(rows_m);
                lo = hi = m;
                break;
              }
              m = wave_min(more);
            }
          }
          lds_order();
          __hip_atomic_store(&s_read[p & 1], p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          uint32_t mot = 0;
          if (R >= 0) {
            const int col = p + S - 1 - lane;
            const bool there = lane < W2 && (unsigned)col < (unsigned)bw && (R > 0 || lane >= S);
            const unsigned id = there ? gid[R * D.ring + (col & rmask)] : kNoId;
            const int e = id != kNoId ? (int)Ep[id] : (int)kNoCand;
            const unsigned long long at = __ballot(id != kNoId && e >= lo && e <= hi);
            const int t = at ? __builtin_ctzll(at) : 0;
            bad = at == 0ull;
            if (at) sel_id = (unsigned)__builtin_amdgcn_readlane((int)id, t);
            mot = (uint32_t)(W2 - 1 - t) | (uint32_t)(W2 - 1 - R) << 8 | 1u << 16;  // pack_dec's upper half
          }
          if (sel_id != kNoId) {
            const uint64_t v = wr[sel_id];
            if (lane == 0) {
              __hip_atomic_store(fin + row0 + p, v | 1ull << 63, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              dec[row0 + p] = R >= 0 ? (uint64_t)mot << 32 | (uint32_t)v : 0ull;
            }
          }
        } else {
          __hip_atomic_store(&s_read[p & 1], p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        // the block enters row 0, column p - S leaves it
        if (bad || sel_id == kNoId || (p >= S && id_out == kNoId)) {
          fail_at(p);
        } else if (lane == 0) {
          gid[p & rmask] = (uint16_t)sel_id;
          enter(sel_id, p);
          atomicMax(&lastany[sel_id], p);
          if (id_out != kNoId && id_out != sel_id && lastcol[id_out * W2] == (uint8_t)(p - S)) leave(id_out);
        }
      }
      if (step_end(f)) break;
    }
  } else if (wv == 1) {
    // ---- the rows from the second above on (a lane each) at column S + r, and -
    // the starting word of column r (lane 0).  v: the lane's entry for the next
    // r, from raw (wave 3 fetches it); t0: its word's table.  The ids of its
    // own: those with (id & 63) < kAboveIds.
    const bool act = lane >= 2 && lane_row;
    const uint64_t* lane_fin = fin + base + (size_t)(lane_row ? y - lane : y) * bw + (lane ? S : 0);  // at r = 0
    uint64_t v = 0;
    float4 t0 = make_float4(0.f, 0.f, 0.f, 0.f);
    bool t_ok = false, dead = false;
    int n_ids = 0;  // one more than the highest id given out
    // more: the entry for r + 1 has been fetched too
    auto insert = [&](int r, bool more) -> bool {
      const int p = r - 1;
      const bool has = lane == 0 ? r >= 0 && r < bw : act && S + r < bw;
      for (int spin = 0; __ballot(has && lane != 0 && !fin_is(v)) != 0ull;) {  // fetched before it was final
        if (give_up(spin)) return false;
        if (has && lane != 0 && !fin_is(v)) v = fin_load(lane_fin + r);
      }
      // a starting word lives through its block's step unless the block takes it
      const int col = lane == 0 ? r : S + r, seen = lane == 0 ? r - S : col;
      const uint32_t w = (uint32_t)v;
      uint32_t h = wave_hash(w, D.bucket_log);
      const uint32_t h2 = wave_hash2(w, D.bucket_log);
      unsigned id = head[h], id2 = head[h2];
      auto is = [&](unsigned i) { return id_holds(ids, i, w, (i & 63u) < kAboveIds, p - S); };
      const bool hit1 = has && is(id), hit2 = has && is(id2), hit = hit1 || hit2;
      if (hit2 && !hit1) id = id2;
      if (hit) atomicMax(&lastany[id], seen);
      const bool fresh = has && !hit;
      const unsigned long long fm = __ballot(fresh);
      if (fm) {
        lds_order();
        const bool first_live = fresh && id != kNoId && lastany[id] >= p - S;  // another word's, still in use
        const int n = (int)__popcll(fm), rank = (int)__popcll(fm & ((1ull << lane) - 1));
        int got = 0;
        for (int chunk = 0; got < n; chunk += 64) {  // the lowest ids that no column holds
          if (chunk >= D.ids) return false;
          unsigned long long fb = __ballot(lane < kAboveIds && lastany[chunk + lane] < p - S);
          while (fb && got < n) {
            const int b = __builtin_ctzll(fb);
            fb &= fb - 1;
            if (fresh && rank == got) id = (unsigned)(chunk + b);
            n_ids = max(n_ids, chunk + b + 1);
            ++got;
          }
        }
        const unsigned mine = id;
        if (fresh) {
          if (first_live) h = h2;
          ids.set_word(id, v & 0x7FFFFFFFFFFFFFFFull);
          head[h] = (uint16_t)id;
        }
        lds_order();
        if (n > 1 && fresh) {  // equal words among them share the id that the bucket kept
          const unsigned kept = head[h];
          if (kept != id && (kept & 63u) < kAboveIds && (uint32_t)wr[kept] == w) id = kept;
        }
        if (fresh) {
          // an id given up for an equal word's keeps this word (a bucket may still name it), so its table too
          if (!t_ok) t0 = ctab[fin_root(v)];
          id_publish(ids, mine, t0, id, seen);
        }
      }
      if (has) gid[lane * D.ring + (col & rmask)] = (uint16_t)id;
      if (lane == 0) s_count.publish(p, 0, n_ids);
      v = raw[(lane < W2 ? lane : 0) * kRawCols + ((r + 1) & (kRawCols - 1))];
      t_ok = more && (lane == 0 ? r + 1 >= 0 : act && fin_is(v)) && col + 1 < bw;
      if (t_ok) t0 = ctab[fin_root(v)];
      lds_order();
      return true;
    };
    lds_barrier();
    if (!turn()) {
      dead = true;
      fail_at(-2);
    }
    for (int c = 0; c < S + 8 && !dead; c += 8) {
      uint64_t g[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int r = c + k - S;
        g[k] = lane == 0 ? (r >= 0 && r < bw ? fin_load(lane_fin + r) : 0) : act && S + r < bw ? fin_load(lane_fin + r) : 0;
      }
      if (lane < W2)
#pragma unroll
        for (int k = 0; k < 8; ++k) raw[lane * kRawCols + ((c + k - S) & (kRawCols - 1))] = g[k];
      lds_order();
      v = raw[(lane < W2 ? lane : 0) * kRawCols + ((c - S) & (kRawCols - 1))];
      t_ok = false;
      for (int k = 0; k < 8 && c + k < S; ++k)
        if (!dead && !insert(c + k - S, k < 7)) {
          dead = true;
          fail_at(-2);
        }
    }
    v = raw[(lane < W2 ? lane : 0) * kRawCols];
    t_ok = false;
    lds_barrier();
    for (int p = -1; p < bw; ++p) {
      const int f = s_fail[(p & 1) ^ 1];
      if (!dead && !insert(p + 1, true)) {
        dead = true;
        fail_at(p);
      }
      if (step_end(f)) break;
    }
  } else if (wv == 2) {
    // ---- the row above, column cB, polled 64 columns at a time ---------------
    // pv: that row from column pb, nB of them final; pn: the poll in flight,
    // taken three steps after it was issued or when it is needed.  Its own ids:
    // those with (id & 63) >= kAboveIds.
    int cB = y < 1 ? bw : 0, pb = 0, nB = 0, pn_at = -1, pn_step = 0, n_ids = 0;
    uint64_t pv = 0, pn = 0;
    bool dead = false;
    auto insert = [&](int p) -> bool {
      const int req = min(p + S + 1, bw - 1), ahead = min(p + S + 1 + D.look, bw - 1);
      int spin = 0;
      for (;;) {
        if (pn_at >= 0 && (p - pn_step >= 3 || (cB <= req && cB - pb >= nB))) {
          pv = pn;
          pb = pn_at;
          pn_at = -1;
          const unsigned long long ok = __ballot(pb + lane < bw && fin_is(pv));
          nB = ok == ~0ull ? 64 : __builtin_ctzll(~ok);
        }
        const bool gb = cB <= ahead && cB - pb < nB;
        if (gb) {
          const uint32_t w = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pv, cB - pb);
          const uint32_t rt = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(pv >> 32), cB - pb) & 0x7FFFFFFFu;
          uint32_t h = wave_hash(w, D.bucket_log);
          const uint32_t h2 = wave_hash2(w, D.bucket_log);
          // the lanes read the same, but not all at once: wave 1 may write in between, so one lane's reads count
          unsigned id = (unsigned)__builtin_amdgcn_readfirstlane((int)head[h]);
          const unsigned id2 = (unsigned)__builtin_amdgcn_readfirstlane((int)head[h2]);
          auto is = [&](unsigned i) {
            return __builtin_amdgcn_readfirstlane((int)id_holds(ids, i, w, (i & 63u) >= kAboveIds, p - S)) != 0;
          };
          const bool hit1 = is(id), hit2 = is(id2);
          if (hit2 && !hit1) id = id2;
          if (!hit1 && !hit2) {
            if (id != kNoId && lastany[id] >= p - S) h = h2;  // the first bucket's word is still in use
            int nid = -1;
            constexpr int kOwn = 64 - kAboveIds, kAt = 64 / kOwn * 64;  // its ids of 64 / kOwn chunks at a time
            for (int c = 0; c < D.ids && nid < 0; c += kAt) {
              const int i = c + lane / kOwn * 64 + kAboveIds + lane % kOwn;
              const unsigned long long fb = __ballot(i < D.ids && lastany[min(i, D.ids - 1)] < p - S);
              if (fb) {
                const int l = __builtin_ctzll(fb);
                nid = c + l / kOwn * 64 + kAboveIds + l % kOwn;
              }
            }
            if (nid < 0) return false;
            id = (unsigned)nid;
            n_ids = max(n_ids, nid + 1);
            if (lane == 0) {
              ids.set_word(id, (uint64_t)rt << 32 | w);
              head[h] = (uint16_t)id;
              id_publish(ids, id, ctab[rt], id, cB);
            }
          } else if (lane == 0) {
            ids.raise(id, cB);
          }
          if (lane == 0) gid[D.ring + (cB & rmask)] = (uint16_t)id;
          lds_order();
          ++cB;
        }
        if (cB < bw && pn_at < 0 && pb + nB < bw && pb + nB - cB < 16) {
          pn_at = cB;
          pn_step = p;
          pn = cB + lane < bw ? fin_load(fin + row0 - bw + cB + lane) : 0;
        }
        if (cB > req) {
          if (lane == 0) s_count.publish(p, 1, n_ids);
          return true;
        }
        if (!gb) {
          if (give_up(spin)) return false;
        }
      }
    };
    lds_barrier();
    if (!turn() || !insert(-2)) {
      dead = true;
      fail_at(-2);
    }
    lds_barrier();
    for (int p = -1; p < bw; ++p) {
      const int f = s_fail[(p & 1) ^ 1];
      if (!dead && !insert(p)) {
        dead = true;
        fail_at(p);
      }
      if (step_end(f)) break;
    }
  } else if (wv == 3) {
    // ---- the window's rows above: column p + S enters, column p - S leaves, --
    // once wave 0 has read the row sets of block p's window.  It also fetches
    // wave 1's entries, four columns at a time, four steps before they go to raw
    const bool row = lane_row && lane >= 1, act = lane >= 2 && lane_row;
    const uint64_t* lane_fin = fin + base + (size_t)(lane_row ? y - lane : y) * bw + (lane ? S : 0);  // at r = 0
    uint64_t g[4] = {0, 0, 0, 0};
    lds_barrier();
    lds_barrier();
    for (int p = -1; p < bw; ++p) {
      const int f = s_fail[(p & 1) ^ 1];
      bool bad = false;
      if ((p & 3) == 1) {
        const int r = p + 3;  // entries r .. r + 3: read from step r - 2 on (the first eight are there)
        if (p > 1 && lane < W2)
#pragma unroll
          for (int k = 0; k < 4; ++k) raw[lane * kRawCols + ((r + k) & (kRawCols - 1))] = g[k];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int n = r + 4 + k;
          if (lane == 0 ? n < bw : act && S + n < bw) g[k] = fin_load(lane_fin + n);
        }
      }
      if (p < 0) {
        for (int c = 0; c < S && c < bw; ++c)
          if (row) {
            const unsigned id = gid[lane * D.ring + (c & rmask)];
            if (id == kNoId) bad = true;
            else enter(id, c);
          }
      } else {
        const bool in = row && p + S < bw, out = row && p >= S;
        const unsigned id_in = in ? gid[lane * D.ring + ((p + S) & rmask)] : kNoId;
        const unsigned id_out = out ? gid[lane * D.ring + ((p - S) & rmask)] : kNoId;
        const bool last = id_out != kNoId && lastcol[id_out * W2 + lane] == (uint8_t)(p - S) && id_out != id_in;
        bad = (in && id_in == kNoId) || (out && id_out == kNoId);
        for (int spin = 0; __hip_atomic_load(&s_read[p & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != p;)
          if (++spin > kWaveSpin) {  // wave 0 stores it on every path of its step
            bad = true;
            break;
          }
        lds_order();
        if (id_in != kNoId) enter(id_in, p + S);
        if (last) leave(id_out);
      }
      if (__ballot(bad) != 0ull) fail_at(p);
      if (step_end(f)) break;
    }
  } else {
    // ---- the words' deltas of block p + 1 ------------------------------------
    // Blocks are staged 16 at a time, waves 0-3 of these a pixel row each, wave
    // 4 the records; in step p waves 0-2 make the products of block p + 2 and
    // wave 3 its channel words.
    const int ev = wv - kWaveRoles;
    uint32_t in_flight = 0;
    auto stage_load = [&](int grp) {
      if (ev < 4) {
        const int i = grp * kPxBlocks * 3 + lane;
        if (lane < 3 * kPxBlocks && i < 3 * bw)
          in_flight = gload(reinterpret_cast<const uint32_t*>(d.rgb + (size_t)(4 * y + ev) * d.width * 3) + i);
      } else if (ev == 4) {
        if (grp * kPxBlocks + (lane >> 2) < bw)
          in_flight = reinterpret_cast<const uint32_t*>(rec + row0 + grp * kPxBlocks)[lane];
      }
    };
    auto stage_store = [&](int grp) {
      if (ev < 5) px[((grp & 1) * 5 + ev) * 64 + lane] = in_flight;
    };
    // entry (pixel, index value, channel) of the products, a lane of waves 0-2
    const int pe = ev * 64 + lane, p_px = pe / 12, p_idx = pe % 12 / 3, p_ch = pe % 3;
    // wave 3: lanes 0-11 one channel (lane % 3) of a pixel row (lane / 3): bytes ch, ch + 3, ch + 6, ch + 9 of
    // its 12; the other lanes the record
    const int b_row = min(lane / 3, 4), b_ch = lane % 3, b_step = lane < 12 ? 3 : 4;
    const uint32_t px_sel01 = b_ch == 0 ? 0x00060300u : b_ch == 1 ? 0x00070401u : 0x00000502u;
    const uint32_t px_sel2 = b_ch == 0 ? 0x05020100u : b_ch == 1 ? 0x06020100u : 0x07040100u;
    const float2 p_w = s_ab[min(p_idx, 3)];
    auto block_setup = [&](int b) {
      const int at = (b / kPxBlocks & 1) * 5 * 64;
      if (ev < 3) {
        const uint8_t* bytes = reinterpret_cast<const uint8_t*>(px + at + (p_px >> 2) * 64);
        const float v = (float)bytes[(b & (kPxBlocks - 1)) * 12 + 3 * (p_px & 3) + p_ch];
        *reinterpret_cast<float2*>(prod + (b & 1) * kProdBytes + 96 * p_px + 24 * p_idx + 8 * p_ch) =
            make_float2(v * p_w.x, v * p_w.y);
      } else if (ev == 3) {
        const uint32_t* q = px + at + b_row * 64 + (b & (kPxBlocks - 1)) * b_step;
        const uint32_t x0 = q[0], x1 = q[1], x2 = q[2];
        if (lane < 12) s_blk[b & 3][lane] = __builtin_amdgcn_perm(x2, __builtin_amdgcn_perm(x1, x0, px_sel01), px_sel2);
        if (lane == 12) {
          s_blk[b & 3][12] = x0;
          s_blk[b & 3][13] = x1;
          s_blk[b & 3][14] = x2;
        }
      }
    };
    ChannelEval ce{};
    const int q = lane & 3, qc = min(q, 2);
    ce.mask565 = q == 0 ? 0xF8u : q == 1 ? 0xFCu : q == 2 ? 0xF8u : 0u;
    ce.shift565 = q == 0 ? 11u : q == 1 ? 6u : 0u;
    ce.snap_off = q == 1 ? 256u : 0u;
    ce.prod_off = 0x08080808u * (uint32_t)qc;
    unsigned long long n_cand = 0;
    stage_load(0);
    stage_store(0);
    stage_load(1);
    lds_barrier();
    block_setup(0);
    if (bw > 1) block_setup(1);
    lds_barrier();
    for (int p = -1; p < bw; ++p) {
      const int f = s_fail[(p & 1) ^ 1];
      const int b = p + 1;
      if (((b + 2) & (kPxBlocks - 1)) == 0) {  // group of block p + 3: used from the next step on
        stage_store((b + 2) / kPxBlocks);
        stage_load((b + 2) / kPxBlocks + 1);
      }
      if (b >= 1 && b + 1 < bw) block_setup(b + 1);
      if (b < bw && __builtin_amdgcn_readfirstlane((int)s_blk[b & 3][14]) != 0) {
        int16_t* En = E + (b & 1) * D.ids;
        const uint32_t* blk = s_blk[b & 3];
        const int nu = __builtin_amdgcn_readfirstlane(s_count.before(p));
        const EvalSplit sp = eval_split(nu, ev, lane);
        if (sp.quad) {
          ce.sq = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            ce.pc[j] = blk[3 * j + qc];
            ce.sq = __builtin_amdgcn_udot4(ce.pc[j], ce.pc[j], ce.sq, false);
          }
          ce.own = blk[12];
          ce.orig = (int)blk[13];
          for (int i = sp.first; i < nu; i += sp.stride) {
            int e = kNoCand;
            if (lastany[i] >= p - S)
              e = eval_candidate_quad(ce, (uint32_t)wr[i], tab[i], s_snap, prod + (b & 1) * kProdBytes);
            if (q == 0) En[i] = (int16_t)e;
          }
        } else {
          BlockEval be;
          be.sq = 0;
#pragma unroll
          for (int k = 0; k < 12; ++k) {
            be.pc[k] = blk[k];
            be.sq = __builtin_amdgcn_udot4(be.pc[k], be.pc[k], be.sq, false);
          }
          be.own = blk[12];
          be.orig = (int)blk[13];
          for (int i = sp.first; i < nu; i += sp.stride) {
            int16_t e = kNoCand;
            if (lastany[i] >= p - S) {
              const float4 t4 = tab[i];
              const CandResult res =
                  eval_candidate<false, true>(be, (uint32_t)wr[i], CandTab{t4.x, t4.y, t4.z, t4.w}, s_snap, s_ab);
              if (res.valid) e = sat16(res.err);
            }
            En[i] = e;
          }
        }
        if (ev == kWaveEval - 1)
          n_cand += (unsigned)(min(y, W2 - 1) * (min(bw, b + S) - max(0, b - S)) + b - max(0, b - S));
      }
      if (step_end(f)) break;
    }
    if (ev == kWaveEval - 1 && lane == 0 && n_cand)
      atomicAdd(&st->wave_cands[(blockIdx.x % kStatSlots) * kSlot64], n_cand);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (s_fail[0] | s_fail[1]) {
      atomicExch(&st->wave_fail, 1u);
      __threadfence();
    }
    // the last row to finish reports to the host
    if (atomicAdd(&st->wave_done, 1u) + 1 == gridDim.x) {
      const unsigned failed = atomicAdd(&st->wave_fail, 0u);
      st->wave_ok = failed ? 0u : 1u;
      if (conv) {
        *reinterpret_cast<volatile unsigned int*>(conv) = failed;
        __threadfence_system();
      }
    }
  }
}

}  // namespace mptc
