"""What the waves of k_intra_wave share about the ids of a window's words
(mptc_amd/csrc/wave_ids.h), compiled for the CPU: in any order of the accesses
inside a step, every wave sees the same and nothing is left out."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MOST_IDS = 1152

SOURCE = """
#include <functional>
#include <vector>
#include "wave_ids.h"
using namespace mptc;
// one id: the last column it was seen at, its word and its table
struct Id {
  int last;
  uint32_t word;
  int table;
};
// the owner's writes in its order, for the reader to meet at any point
struct Owner {
  Id& id;
  std::vector<std::function<void()>>& ops;
  void set_word(unsigned, uint64_t v) const { ops.push_back([this, v] { id.word = (uint32_t)v; }); }
  void set_table(unsigned, int t) const { ops.push_back([this, t] { id.table = t; }); }
  void raise(unsigned, int c) const { ops.push_back([this, c] { if (c > id.last) id.last = c; }); }
  void order() const {}
};
// a reader before whose k-th read at[k] of the writes are done
struct Reader {
  Id& id;
  std::vector<std::function<void()>>& ops;
  const int* at;
  mutable int k, done;
  void upto(int n) const { while (done < n) ops[done++](); }
  int last(unsigned) const { upto(at[k++]); return id.last; }
  uint32_t word(unsigned) const { upto(at[k++]); return id.word; }
  void order() const {}
};
// the test the other way round: the word first
static bool holds_word_first(const Reader& t, unsigned i, uint32_t w, bool own, int oldest) {
  return t.word(i) == w && (own || t.last(i) >= oldest);
}
static int g_log[8], g_n;
struct Logged {
  int last(unsigned) const { g_log[g_n++] = 1; return 0; }
  uint32_t word(unsigned) const { g_log[g_n++] = 2; return 0; }
  void set_table(unsigned, int) const { g_log[g_n++] = 3; }
  void raise(unsigned, int) const { g_log[g_n++] = 4; }
  void order() const { g_log[g_n++] = 0; }
};
extern "C" {
// Another wave's id, seen at column `last` with word `old`; its owner gives it
// to word `fresh` at column `now` if no column holds it.  A reader looks for
// `want` with at[0] and at[1] of the owner's writes done before its two reads.
// 1: an id in use and right, or none; 0: an id that holds another word (or no table).
int lookup(int last, unsigned old, unsigned fresh, int now, unsigned want, int oldest, const int* at, int word_first) {
  Id id{last, old, (int)old};
  std::vector<std::function<void()>> ops;
  const Owner o{id, ops};
  if (last < oldest) {
    o.set_word(3, fresh);
    id_publish(o, 3, (int)fresh, 3, now);
  }
  const int n = (int)ops.size();
  const int seq[2] = {at[0] < n ? at[0] : n, at[1] < n ? at[1] : n};
  const Reader r{id, ops, seq, 0, 0};
  const bool hit = word_first ? holds_word_first(r, 3, want, false, oldest) : id_holds(r, 3, want, false, oldest);
  r.upto(n);
  return !hit || (id.word == want && id.table == (int)want);
}
// the accesses of a look-up and of a publication: 0 order, 1 column, 2 word, 3 table, 4 column raised
int accesses(int publish, int* out) {
  g_n = 0;
  if (publish)
    id_publish(Logged{}, 1, 0, 1, 0);
  else
    (void)id_holds(Logged{}, 1, 0, false, 0);
  for (int i = 0; i < g_n; ++i) out[i] = g_log[i];
  return g_n;
}
static IdCount count;
int waves() { return kWaveEval; }
int quad_ids() { return kQuadIds; }
int id_count(int S) { return wave_id_count(S); }
int look() { return kWaveLook; }
int above_ids() { return kAboveIds; }
void start() { count = IdCount{}; }
void publish(int step, int who, int n) { count.publish(step, who, n); }
int before(int step) { return count.before(step); }
// adds to hits[id] the lanes that evaluate it in wave ev, which sees n_ids
void take(int n_ids, int ev, int* hits) {
  for (int lane = 0; lane < 64; ++lane) {
    const EvalSplit s = eval_split(n_ids, ev, lane);
    for (int i = s.first; i < n_ids; i += s.stride) ++hits[i];
  }
}
}
"""


@pytest.fixture(scope="module")
def ids(tmp_path_factory):
    d = tmp_path_factory.mktemp("wave_ids")
    src, out = d / "ids.cpp", d / "ids.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-D__forceinline__=inline",
                    "-I", os.path.join(ROOT, "mptc_amd", "csrc"), str(src), "-o", str(out)], check=True, timeout=120)
    return C.CDLL(str(out))


def _hits(ids, counts):
    """Lanes per id where wave ev sees counts[ev] ids."""
    h = np.zeros(MOST_IDS, np.int32)
    for ev, n in enumerate(counts):
        ids.take(n, ev, h.ctypes.data_as(C.POINTER(C.c_int)))
    return h


def test_every_id_is_evaluated_once(ids):
    for n in range(MOST_IDS + 1):
        h = _hits(ids, [n] * ids.waves())
        lanes = 4 if n <= ids.quad_ids() else 1
        assert (h[:n] == lanes).all() and not h[n:].any(), n


def test_a_step_has_one_count(ids):
    """Two waves give out ids (one more than the highest: raised in a step, at
    any moment of it), twelve read the count at any moment of the same step."""
    rng = np.random.default_rng(3)
    for _ in range(300):
        ids.start()
        done = [0, 0]
        for step in range(-2, 40):
            # events of the step in a random order: readers 0..11, writers 12 and 13
            now = [min(MOST_IDS, d + int(rng.integers(0, 60))) if rng.random() < 0.7 else d for d in done]
            seen = []
            for who in rng.permutation(14):
                if who >= 12:
                    ids.publish(step, int(who) - 12, now[who - 12])
                elif step > -2:
                    seen.append(ids.before(step))
            if seen:
                assert set(seen) == {max(done)}  # what the step before left: the same for all
                assert _hits(ids, seen)[:max(done)].all()
            done = now


def test_differing_counts_would_leave_ids_out(ids):
    """The waves have to agree: where some see the count before it passes the
    four-lanes limit and some after, ids below both counts are not evaluated."""
    q = ids.quad_ids()
    h = _hits(ids, [q - 4] * 8 + [q + 61] * 4)
    assert (h[:q - 4] == 0).sum() > 100


def _lookups(ids, word_first):
    """Wrong outcomes over every order of the reader's two accesses and the
    owner's writes, for ids in use, just out of use and never used."""
    wrong = runs = 0
    for last in (-(1 << 30), 4, 5, 6, 30):
        for fresh in (7, 8):
            for want in (7, 8):
                for a in range(4):
                    for b in range(a, 4):
                        at = (C.c_int * 2)(a, b)
                        wrong += not ids.lookup(last, 7, fresh, 30, want, 6, at, word_first)
                        runs += 1
    assert runs == 5 * 4 * 10
    return wrong


def test_an_id_found_in_use_holds_the_word(ids):
    assert _lookups(ids, 0) == 0


def test_the_word_before_the_column_is_caught(ids):
    assert _lookups(ids, 1) > 0


def test_accesses_are_ordered(ids):
    out = (C.c_int * 8)()
    assert out[:ids.accesses(0, out)] == [1, 0, 2]
    assert out[:ids.accesses(1, out)] == [3, 0, 4]


def test_every_wait_counts_its_polls():
    """The loops of k_intra_wave that wait for another wave or row give up after
    a number of polls."""
    import re
    lines = open(os.path.join(ROOT, "mptc_amd", "csrc", "wave_kernels.h")).read().split("\n")
    waits = [i for i, t in enumerate(lines) if re.match(r"\s*(while|for) \(.*(atomic_load|fin_is|fin_load)", t)]
    assert len(waits) == 3
    for i in waits:
        assert re.search(r"give_up\(|> kWaveSpin", "\n".join(lines[i:i + 4])), lines[i]


@pytest.mark.parametrize("S", range(1, 33))
def test_the_row_above_has_ids_enough(ids, S):
    """Wave 2's share of the ids covers a window's columns of the row above, all
    distinct, with room for words that other rows keep in use."""
    n = ids.id_count(S)
    assert n % 128 == 0 and n <= MOST_IDS
    own = n // 64 * (64 - ids.above_ids())
    assert own >= 2 * S + 2 + ids.look() and own >= 24
