"""The inter search by distinct words (thresholds above 4, search areas 8 to 16)
against the CPU oracle and, in its counts, the candidate-by-candidate search."""
from __future__ import annotations

import numpy as np
import pytest

from mptc_amd.workloads import SynthCfg
from tests.helpers import compare_results

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def enc():
    from mptc_amd import lib
    e = lib.Encoder(200, 160, search_area=16, err_threshold=8)
    yield e
    e.close()


def _noise(w, h, n):
    return np.random.default_rng(w * h).integers(0, 256, (n, h, w, 3)).astype(np.uint8)


# window rows that the waves share unevenly; tiles over the frame's edges; tiles with more words than there are ids
@pytest.mark.parametrize("w,h,S,thr,tile_w,noise", [
    (4, 4, 8, 5, 8, False), (36, 20, 8, 8, 8, False), (100, 60, 7, 9, 16, False), (100, 60, 10, 9, 16, False), (160, 96, 8, 5, 8, False),
    (160, 96, 8, 8, 64, False), (100, 60, 8, 128, 32, False), (132, 68, 9, 8, 8, False), (132, 68, 15, 16, 16, False),
    (200, 160, 16, 8, 8, False), (200, 160, 16, 30000, 64, False), (4, 160, 16, 8, 8, False), (200, 4, 8, 32, 64, False),
    (160, 96, 8, 8, 8, True), (200, 120, 16, 60, 8, True)])
def test_word_search_matches_oracle(enc, orc, w, h, S, thr, tile_w, noise):
    print(f"{w}x{h} S={S} thr={thr} tile_w={tile_w} noise={noise}", flush=True)
    frames = _noise(w, h, 2) if noise else orc.synth_frames(SynthCfg(w, h, w + S, 5, 1, 3, 8, 0), 2)
    enc.set_tuning(tile_w=tile_w)
    enc.set_params(S, thr)
    got = enc.encode_sequence(frames, 8)
    st = enc.stats()
    enc.set_tuning()
    want = orc.encode_sequence(frames, S, thr, 8)
    for f, (a, b) in enumerate(zip(got, want)):
        compare_results(a, b, f"frame {f}")
        assert np.array_equal(a["kind"], b["kind"])
    bw, bh = w // 4, h // 4
    window = sum((min(bw, x + S) - max(0, x - S)) * (min(bh, y + S) - max(0, y - S)) for x in range(bw) for y in range(bh))
    assert st["inter_candidates"] == window
