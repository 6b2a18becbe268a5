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
#include "wave_ids.h"
using namespace mptc;
extern "C" {
static IdCount count;
int waves() { return kWaveEval; }
int quad_ids() { return kQuadIds; }
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
