// Pruned exhaustive search: the same decisions as k_inter / k_intra_dense
// (bit-exact), with most candidate evaluations replaced by a cheap lower
// bound on their error.
//
// Why it is exact.  For a threshold thr >= 0 a block's decision depends only
// on the candidates whose error delta passes (valid, delta <= thr): before the
// first passing candidate (scan order) the others can only raise the running
// minimum, which that candidate then undercuts; after it they can never update
// it (codec/dxt_image.cpp:697-708).  So a candidate proved non-passing may be
// recorded as not passing without changing the decision.
//
// The bound.  A valid candidate's palette is two endpoints and the points a
// third and two thirds between them, rounded down: q_i = a_i e1 + (1 - a_i) e2 -
// r_i, a_i = 0, 1/3, 2/3, 1 by the index value, r_i = 0 at the endpoints and 0,
// 1/3 or 2/3 between.  Over all real endpoints the squared error against the
// line without r is at least its least-squares residual,
//   L_c = sum |p|^2 - (sum b^2 |A|^2 - 2 sum ab A.B + sum a^2 |B|^2) / det,
// A = sum a p, B = sum b p, b = 1 - a (a shift of all pixels leaves L_c as it
// is).  The endpoints absorb any shift common to all pixels, so r counts only
// up to one: eta = the norm of what is left at the best shift (at most 2.31).
// So the error of a candidate that passes satisfies
//   sqrt(L_c) - eta <= sqrt(SSE) < sqrt(48 (thr + err_own + 1))
// (Error() = floor(SSE / 48), codec/dxt_image.cpp:258-276), and one with
// L_c >= (sqrt(48 (thr + err_own + 1)) + eta)^2 + 16 is pruned; 16 covers the
// fp32 rounding of L_c (< 2).  A and B are integer dot products (v_dot4) of
// the pixels less 128 with the weights: 12 a candidate, where the scatter
// around the index values' means, the bound used before, took 36; 13 % of the
// candidates survive at threshold 0 and 37 % at 2 where 23 % and 47 % did
// (1080p, S = 8, threshold 0: inter search 239 -> 165 us, intra 219 -> 145).
//   The own word's delta is 0 by definition: its block is a candidate of this
// form too, unless its endpoints are in the order that means a three-colour
// palette; such a block prunes nothing.
//
//   k_pruned_search wave tiles as the search kernels; per position the bound;
//                   the wave's survivors are compacted in LDS and evaluated
//                   exactly, 64 per round.  Inter: the
//                   chunk summaries of the selection rule (as k_inter, then
//                   inter_decision in k_intra_prep); intra: E for the
//                   fixpoint passes
//   k_fold_intra    per block, the reference's selection over the passing
//                   deltas of E: the intra decision with the changed-word list
//                   (as k_intra_combine).  With 1, 2 or 4 chunks a workgroup
//                   holds every chunk of its tiles and the intra search takes
//                   these decisions itself, after a workgroup barrier.
//
// The words' bound tables (BoundTab, batch_kernels.h) are built by
// k_block_prep (the previous frame's words) and k_intra_prep (the current
// words, which also clears the passing sets).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_kernels.h"

namespace mptc {

// Pixel side of the bound for one block.
struct BoundBlk {
  uint32_t pc[12];  // pc[3j + ch]: channel ch of pixels 4j..4j+3, less 128, signed bytes
  float p3[3];      // 3 x the channel sums
  float q;          // sum of squares
  float rl;         // sqrt(48 (thr + err_own + 1)); 1e9: prune nothing
};

__device__ __forceinline__ float bound_limit(int thr, int err_own, bool line) {
  return line ? sqrtf((float)(48 * (thr + err_own + 1))) : 1e9f;
}

// Whether a physical block's palette is on the line between its endpoints.
__device__ __forceinline__ bool line_palette(uint64_t phys) {
  return (uint32_t)(phys & 0xFFFF) > (uint32_t)((phys >> 16) & 0xFFFF);
}

// pc, p3 and q from the packed channel bytes c[12].
__device__ __forceinline__ void make_bound_blk(const uint32_t* c, BoundBlk& b) {
  int q = 0, s[3] = {0, 0, 0};
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    const uint32_t v = c[k] ^ 0x80808080u;
    b.pc[k] = v;
    q = __builtin_amdgcn_sdot4((int)v, (int)v, q, false);
    s[k % 3] = __builtin_amdgcn_sdot4((int)v, 0x03030303, s[k % 3], false);
  }
#pragma unroll
  for (int ch = 0; ch < 3; ++ch) b.p3[ch] = (float)s[ch];
  b.q = (float)q;
}

// True when the candidate word of `t` provably does not pass.
__device__ __forceinline__ bool bound_prunes(const BoundBlk& b, const BoundTab& t) {
  float ex = 0.0f;
#pragma unroll
  for (int ch = 0; ch < 3; ++ch) {
    int a = __builtin_amdgcn_sdot4((int)b.pc[ch], (int)t.w.x, 0, false);
    a = __builtin_amdgcn_sdot4((int)b.pc[3 + ch], (int)t.w.y, a, false);
    a = __builtin_amdgcn_sdot4((int)b.pc[6 + ch], (int)t.w.z, a, false);
    a = __builtin_amdgcn_sdot4((int)b.pc[9 + ch], (int)t.w.w, a, false);
    const float A = (float)a, B = b.p3[ch] - A;
    ex = __builtin_fmaf(A, __builtin_fmaf(t.k.y, B, t.k.x * A), ex);
    ex = __builtin_fmaf(B, t.k.z * B, ex);
  }
  const float r = b.rl + t.k.w;
  return b.q - ex >= __builtin_fmaf(r, r, 16.0f);
}

// Window position (row r, column t; position r * 2S + t) of block (bx, by) ->
// the candidate block (j, i); false outside the frame or (intra) outside the
// causal window.
template <bool kIntra>
__device__ __forceinline__ bool window_block(int r, int t, int S, int bx, int by, int bw, int bh, int& j, int& i) {
  if (kIntra) {
    j = by - r;
    i = bx + S - 1 - t;
    return j >= 0 && i >= 0 && i < bw && !(r == 0 && t < S);
  }
  j = by - S + r;
  i = bx - S + t;
  return j >= 0 && j < bh && i >= 0 && i < bw;
}

constexpr int kPruneBatch = 16;  // window positions per bound / evaluate round of a wave
constexpr int kPackedBlk = 15;   // LDS words per block: pc[12], sum of squares, own word, own error
constexpr int kFoldWords = 8;    // LDS words of an inter lane's fold: ChunkFold's 7 fields and its row

// An inter lane's ChunkFold lives in LDS between the (rare) batches that
// have passing deltas, so that it holds no registers through the rest.  Its
// fields fit 16 bits: positions < 15,876, rows < 126, and min_val is a passing
// delta (<= thr) or the initial "none" (stored as kNoCand).
__device__ __forceinline__ void cf_load(int16_t (*s)[64], int lane, ChunkFold& cf, int& row) {
  cf.first_le0 = s[0][lane];
  cf.le0_row = s[1][lane];
  cf.after_sel = s[2][lane];
  cf.last_neg = s[3][lane];
  cf.min_val = s[4][lane] == kNoCand ? 0x7fffffff : (int)s[4][lane];
  cf.min_pos = s[5][lane];
  cf.row_neg = s[6][lane];
  row = s[7][lane];
}
__device__ __forceinline__ void cf_store(int16_t (*s)[64], int lane, const ChunkFold& cf, int row) {
  s[0][lane] = (int16_t)cf.first_le0;
  s[1][lane] = (int16_t)cf.le0_row;
  s[2][lane] = (int16_t)cf.after_sel;
  s[3][lane] = (int16_t)cf.last_neg;
  s[4][lane] = (int16_t)min(cf.min_val, (int)kNoCand);
  s[5][lane] = (int16_t)cf.min_pos;
  s[6][lane] = (int16_t)cf.row_neg;
  s[7][lane] = (int16_t)row;
}

// Pruned search over the window of every searching block (inter: blocks of
// inter frames against the previous frame's words; intra: blocks with need[]
// set against the current words), in the wave-tile mapping of the dense
// kernels.  Per batch of kPruneBatch positions each lane bounds its block's
// candidates; the survivors of the whole wave are compacted in LDS and
// evaluated exactly 64 at a time, a lane taking any block's survivor (the
// pixel side of the wave's 64 blocks is kept in LDS).  Passing survivors leave
// their delta and a bit of their block's batch.  The bounds are what the time
// goes to, so their loop holds little else: 52 vector instructions a position
// where it had 97 (the window row's part of the address and of the edge test is
// kept for the row, positions that do not pass are not recorded, the bounded
// positions are counted from the window's shape), and two positions' tables are
// requested together (one at a time behind its edge test: 17.5 ms).  A
// 3840x2160 inter frame of S = 32 at threshold 0: 14.7 -> 13.7 ms.
// Intra: the values go to E.  Inter: each lane folds its
// chunk's passing values in scan order into the chunk summary summ[chunk][g]
// of the dense inter kernel (for thr >= 0 the selection depends only on the
// passing deltas, and a row without one leaves a summary as it is).
template <bool kIntra>
__global__ void __launch_bounds__(256) k_pruned_search(const FrameDev* __restrict__ fr, const uint8_t* __restrict__ tsid,
                                                       int n_wtiles, int tw, int n_chunks, int S, int thr,
                                                       const uint64_t* __restrict__ own,
                                                       const uint8_t* __restrict__ need,
                                                       const uint32_t* __restrict__ words,
                                                       const float4* __restrict__ tabs,
                                                       const BoundTab* __restrict__ btab, int* __restrict__ orig,
                                                       uint2* __restrict__ E4, size_t nbs, uint32_t* __restrict__ pm,
                                                       uint4* __restrict__ summ, DevStats* __restrict__ st,
                                                       uint64_t* __restrict__ dec, uint32_t* __restrict__ cw_new,
                                                       int* __restrict__ chg_list, int fold) {
  __shared__ uint8_t s_snap[512];
  __shared__ float2 s_ab[4];
  __shared__ uint32_t s_blk[4][kPackedBlk][64];      // [wave][field][lane]
  __shared__ int16_t s_e[4][kPruneBatch][64];        // the batch's passing deltas, [wave][position][lane]
  __shared__ uint16_t s_list[4][kPruneBatch * 64 + 64];  // survivors: lane | position << 6; + per-lane dummies
  __shared__ uint32_t s_pass[4][64];                     // the lane's passing positions of the batch
  __shared__ int16_t s_cf[4][kFoldWords][64];            // inter: each lane's ChunkFold state and row
  __shared__ unsigned long long s_acc;
  __shared__ unsigned int s_base;
  load_lds_tables(s_snap, s_ab);
  int f = 0, bx = 0, by = 0, chunk = 0;
  const bool in = tile_block(fr, tsid, n_wtiles, tw, n_chunks, f, bx, by, chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const FrameDev& d = fr[f];
  const int g = in ? d.base + by * d.bw + bx : 0;
  const bool act = in && (kIntra ? need[g] != 0 : !d.is_intra);
  // origin of the wave tile (a wave with survivors is a tile inside the batch);
  // tw is a power of two
  const int tw_log = __builtin_ctz((unsigned)tw);
  const int bx0 = bx - (lane & (tw - 1)), by0 = by - (lane >> tw_log);
  bool line = false;
  if (act) {
    BlockPx px;
    load_block(d.rgb, d.width, bx, by, px);
    const int e_own = kIntra ? orig[g] : own_error(px, own[g]);
    if (!kIntra && orig && chunk == 0) orig[g] = e_own;  // inter: k_intra_prep then skips the block's own error
    uint32_t sq = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) {
        const uint32_t v = px.ch(4 * j, ch) | (px.ch(4 * j + 1, ch) << 8) | (px.ch(4 * j + 2, ch) << 16) |
                           (px.ch(4 * j + 3, ch) << 24);
        s_blk[wave][3 * j + ch][lane] = v;
        sq = __builtin_amdgcn_udot4(v, v, sq, false);
      }
    s_blk[wave][12][lane] = sq;
    line = line_palette(own[g]);
    s_blk[wave][13][lane] = (uint32_t)(own[g] >> 32);
    s_blk[wave][14][lane] = (uint32_t)e_own;
  }
  unsigned long long n_exact = 0;
  const int W2 = 2 * S, rows = W2 / n_chunks, p0 = chunk * rows * W2, p1 = p0 + rows * W2;
  // (rb, tb): window row and column of the batch's first position, stepped
  // without divisions
  int rb = chunk * rows, tb = 0;
  // A wave none of whose blocks searches has nothing to do.  Otherwise every
  // lane computes every bound (a vector instruction costs the same for any
  // number of active lanes) and the lanes without a candidate ignore theirs:
  // no divergent branches in the loop.
  const bool wave_act = __ballot(act) != 0ull;
  // the frame's fields in registers (the loops' stores could otherwise alias them)
  const int fbw = d.bw, fbh = d.bh, fbase = d.base;
  // window row of the running position: whether the block has it, and its first block in the frame (clamped into it)
  const char* const ftab = reinterpret_cast<const char*>(btab + fbase);
  bool row_in = false;
  int row_at = 0;
  auto set_row = [&](int r) {
    const int j = kIntra ? by - r : by - S + r;
    row_in = act && j >= 0 && j < fbh;
    row_at = min(max(j, 0), fbh - 1) * fbw;
  };
  set_row(rb);
  // inter: the selection rule over the chunk's positions in scan order
  if (!kIntra) {
    ChunkFold cf;
    cf.begin_row();
    cf_store(s_cf[wave], lane, cf, rb);
  }
  for (int pb = p0; wave_act && pb < p1; pb += kPruneBatch) {
    const int nb = min(kPruneBatch, p1 - pb);  // a multiple of 4
    uint32_t cnt = 0;                          // wave-uniform
    int r = rb, t = tb;
    s_pass[wave][lane] = 0u;
    // the block's bound constants, rebuilt from LDS for each batch so that they
    // hold no registers through the evaluations (zero for lanes that do not
    // search: their bounds are computed and ignored)
    BoundBlk b{};
    if (act) {
      uint32_t c[12];
#pragma unroll
      for (int w = 0; w < 12; ++w) c[w] = s_blk[wave][w][lane];
      make_bound_blk(c, b);
      b.rl = bound_limit(thr, (int)s_blk[wave][14][lane], line);
    }
    // two positions a step (rows and batches are of even length): both tables are requested before the first is used
    for (int k = 0; k < nb; k += 2) {
      bool there[2];
      BoundTab tb4[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int i = kIntra ? bx + S - 1 - t - u : bx - S + t + u;
        const int ic = min(max(i, 0), fbw - 1);  // clamped into the frame: the load is always in bounds
        there[u] = row_in & (i == ic) & !(kIntra && r == 0 && t + u < S);
        // 32-bit offset into the frame's tables (batches of at most 2^27 blocks)
        tb4[u] = *reinterpret_cast<const BoundTab*>(ftab + (uint32_t)(row_at + ic) * (uint32_t)sizeof(BoundTab));
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool surv = there[u] & !bound_prunes(b, tb4[u]);
        const unsigned long long bal = __builtin_amdgcn_ballot_w64(surv);
        // survivors take the next list slots; the others write their lane's dummy slot
        const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, cnt));
        const uint32_t slot = surv ? before : (uint32_t)(kPruneBatch * 64 + lane);
        s_list[wave][slot] = (uint16_t)(lane | ((k + u) << 6));
        cnt += (uint32_t)__popcll(bal);
      }
      t += 2;
      if (t == W2) {
        t = 0;
        set_row(++r);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (uint32_t e0 = 0; e0 < cnt; e0 += 64) {
      if (e0 + lane < cnt) {
        const uint32_t e = s_list[wave][e0 + lane];
        const int lb = (int)(e & 63u), k = (int)(e >> 6);
        int re = rb, te = tb + k;  // k < kPruneBatch: a few steps at most
        while (te >= W2) {
          te -= W2;
          ++re;
        }
        int j = 0, i = 0;
        window_block<kIntra>(re, te, S, bx0 + (lb & (tw - 1)), by0 + (lb >> tw_log), fbw, fbh, j, i);
        const int q = fbase + j * fbw + i;
        BlockEval be;  // the pixel side from LDS; eval_candidate converts the bytes itself
#pragma unroll
        for (int w = 0; w < 12; ++w) be.pc[w] = s_blk[wave][w][lb];
        be.sq = s_blk[wave][12][lb];
        be.own = s_blk[wave][13][lb];
        be.orig = (int)s_blk[wave][14][lb];
        const float4 t4 = tabs[q];
        const CandResult res =
            eval_candidate<false, true>(be, words[q], CandTab{t4.x, t4.y, t4.z, t4.w}, s_snap, s_ab);
        if (res.valid && res.err <= thr) {
          s_e[wave][k][lb] = sat16(res.err);
          atomicOr(&s_pass[wave][lb], 1u << k);
        }
        ++n_exact;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint32_t bits = act ? s_pass[wave][lane] : 0u;  // bit k: position pb + k passes
    if (kIntra && bits) {  // E and the passing set, for the fixpoint passes
      for (int k = 0; k < nb; k += 4) {
        if ((bits >> k) & 15u) {  // E is kept only where a delta passes (the passing set says where)
          const uint32_t lo = (uint32_t)(uint16_t)s_e[wave][k][lane] | ((uint32_t)(uint16_t)s_e[wave][k + 1][lane] << 16);
          const uint32_t hi =
              (uint32_t)(uint16_t)s_e[wave][k + 2][lane] | ((uint32_t)(uint16_t)s_e[wave][k + 3][lane] << 16);
          E4[(size_t)((pb + k) >> 2) * nbs + g] = make_uint2(lo, hi);
        }
      }
      // rare; the batch's 16 bits may straddle two words, which other chunks' waves share
      const int sh = pb & 31;
      uint32_t* wp = pm + (size_t)g * pass_words(S) + (pb >> 5);
      atomicOr(wp, bits << sh);
      if (sh > 16 && (bits >> (32 - sh)) != 0u) atomicOr(wp + 1, bits >> (32 - sh));
    } else if (!kIntra && bits) {
      // inter: fold the batch's passing deltas in scan order.  The selection
      // depends only on them (thr >= 0), and a row without one leaves the
      // summary as it is, so the other positions are skipped.
      ChunkFold cf;
      int cf_row;
      cf_load(s_cf[wave], lane, cf, cf_row);
      int rr = rb, t0 = tb;  // row rr holds positions t0 .. W2 - 1, counted from the batch's first
      while (bits) {
        const int k = __builtin_ctz(bits);
        bits &= bits - 1u;
        while (t0 + k >= W2) {
          t0 -= W2;
          ++rr;
        }
        if (rr != cf_row) {
          cf.end_row(cf_row);
          cf.begin_row();
          cf_row = rr;
        }
        cf.step(s_e[wave][k][lane], pb + k, rr);
      }
      cf_store(s_cf[wave], lane, cf, cf_row);
    }
    // the next batch overwrites s_e and s_list
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    rb = r;
    tb = t;
  }
  if (act && !kIntra) {
    ChunkFold cf;
    int cf_row;
    cf_load(s_cf[wave], lane, cf, cf_row);
    cf.end_row(cf_row);
    summ[(size_t)chunk * nbs + g] = cf.pack();
  }
  if (kIntra && fold) {
    // Intra decisions (as k_fold_intra), when every tile's chunks are waves of
    // this workgroup (n_chunks divides 4): once all of them have written
    // their passing sets and E, the chunk-0 wave of each tile folds its
    // blocks.  The workgroup's waves share the CU's L1, so the barrier
    // orders those writes before the reads.
    __syncthreads();
    bool changed = false;
    if (chunk == 0 && act) {
      const Fold fd = fold_passing_set(pm, E4, nbs, g, S);
      const uint64_t dc = intra_decision(words, fbase, fbw, bx, by, S, thr, fd);
      dec[g] = dc;
      const uint32_t w = dec_acc(dc) ? dec_word(dc) : (uint32_t)(own[g] >> 32);
      if (w != words[g]) {
        cw_new[g] = w;
        changed = true;
      }
    }
    wg_append(changed, g, chg_list, &st->n_changed[0], &s_base);
  }
  // positions bounded: the chunk's window rows and columns inside the frame
  unsigned long long n_bound = 0;
  if (act) {
    const int r0 = chunk * rows, lo = kIntra ? r0 : max(r0, S - by), hi = min(r0 + rows, kIntra ? by + 1 : fbh - by + S);
    const int left = bx - max(0, bx - S), cols = left + min(fbw, bx + S) - bx;
    if (hi > lo) n_bound = (unsigned long long)(hi - lo) * cols - (kIntra && lo == 0 ? cols - left : 0);
  }
  wg_count(&s_acc, n_bound, kIntra ? st->intra_cands : st->inter_cands);
  wg_count(&s_acc, n_exact, kIntra ? st->exact_intra : st->exact_inter);
}

// Intra decisions from the passing sets and E (as k_intra_combine): dec, the
// new current word and the first changed-word list.
__global__ void __launch_bounds__(256) k_fold_intra(const FrameDev* __restrict__ fr, const uint8_t* __restrict__ sid,
                                                    int total, int S, int thr, const uint64_t* __restrict__ own,
                                                    const uint8_t* __restrict__ need,
                                                    const uint32_t* __restrict__ words,
                                                    const uint2* __restrict__ E4, size_t nbs,
                                                    const uint32_t* __restrict__ pm,
                                                    uint64_t* __restrict__ dec, uint32_t* __restrict__ cw_new,
                                                    int* __restrict__ chg_list, DevStats* __restrict__ st) {
  __shared__ unsigned int s_base;
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  bool changed = false;
  if (g < total && need[g]) {
    const FrameDev& d = fr[sid[g]];
    const int k = g - d.base, bx = k % d.bw, by = k / d.bw;
    const Fold fd = fold_passing_set(pm, E4, nbs, g, S);
    const uint64_t dc = intra_decision(words, d.base, d.bw, bx, by, S, thr, fd);
    dec[g] = dc;
    const uint32_t w = dec_acc(dc) ? dec_word(dc) : (uint32_t)(own[g] >> 32);
    if (w != words[g]) {
      cw_new[g] = w;
      changed = true;
    }
  }
  wg_append(changed, g, chg_list, &st->n_changed[0], &s_base);
}

}  // namespace mptc
