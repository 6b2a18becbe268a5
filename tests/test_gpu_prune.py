"""Pruned searches beyond S = 8 (thresholds to 4) and the listed intra search of
inter frames (thresholds above) against the CPU oracle."""
from __future__ import annotations

import numpy as np
import pytest

from mptc_amd.workloads import SynthCfg
from tests.helpers import compare_results

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def enc():
    from mptc_amd import lib
    e = lib.Encoder(320, 320, search_area=63, err_threshold=0)
    yield e
    e.close()


# windows whose positions fill no whole vector, chunk or batch; sizes under the window; one set word to several
@pytest.mark.parametrize("w,h,S,thr", [(100, 60, 9, 0), (100, 60, 9, 3), (132, 68, 11, 4), (160, 96, 16, 0), (160, 96, 16, 4),
                                       (140, 80, 17, 2), (200, 120, 32, 0), (200, 120, 32, 4), (96, 64, 63, 1),
                                       (4, 100, 12, 2), (200, 4, 12, 2), (160, 96, 8, 8), (160, 96, 3, 9), (100, 60, 5, 300),
                                       (160, 96, 16, 8), (200, 120, 32, 16), (160, 96, 33, 8), (36, 36, 8, 30000)])
def test_searches_match_oracle(enc, orc, w, h, S, thr):
    print(f"{w}x{h} S={S} thr={thr}", flush=True)
    frames = orc.synth_frames(SynthCfg(w, h, w + S, 5, 1, 3, 8, 0), 3)
    enc.set_params(S, thr)
    got = enc.encode_sequence(frames, 8)
    st = enc.stats()
    want = orc.encode_sequence(frames, S, thr, 8)
    for f, (a, b) in enumerate(zip(got, want)):
        compare_results(a, b, f"frame {f}")
        assert np.array_equal(a["kind"], b["kind"])
    assert (st["exact_inter_candidates"] > 0) == (thr <= 4)
    assert st["exact_inter_candidates"] <= st["inter_candidates"]


@pytest.mark.parametrize("prune", [0, 1])
def test_flat_and_saturated_blocks(enc, orc, prune):
    """Blocks of one colour (equal endpoints: nothing is pruned for them), of two
    extreme colours, and reference words of one index value."""
    rng = np.random.default_rng(8)
    a = np.repeat(np.repeat(rng.choice([0, 7, 255], (30, 40, 3)), 4, 0), 4, 1).astype(np.uint8)
    b = np.where(rng.random((120, 160, 3)) < 0.3, 255 - a, a).astype(np.uint8)
    frames = np.stack([a, b, np.roll(a, 4, 1)])
    enc.set_tuning(prune=prune)
    for S, thr in ((8, 0), (8, 9), (12, 2)):
        enc.set_params(S, thr)
        for f, (x, y) in enumerate(zip(enc.encode_sequence(frames, 8), orc.encode_sequence(frames, S, thr, 8))):
            compare_results(x, y, f"S={S} thr={thr} frame {f}")
    enc.set_tuning()


@pytest.mark.parametrize("w,h,S", [(4, 4, 1), (12, 8, 1), (100, 60, 2), (36, 132, 5), (132, 36, 8), (96, 64, 12), (40, 200, 32)])
def test_bounded_positions_are_the_window_inside_the_frame(enc, orc, w, h, S):
    """The candidate counts of the pruned searches are those of the plain ones."""
    frames = orc.synth_frames(SynthCfg(w, h, w + S, 5, 1, 3, 8, 0), 2)
    bw, bh = w // 4, h // 4
    window = sum((min(bw, x + S) - max(0, x - S)) * (min(bh, y + S) - max(0, y - S)) for x in range(bw) for y in range(bh))
    counts = []
    for prune in (0, 1):
        enc.set_tuning(prune=prune)
        enc.set_params(S, 0)
        enc.encode_sequence(frames, 8)
        st = enc.stats()
        counts.append((st["inter_candidates"], st["intra_candidates"]))
    enc.set_tuning()
    assert counts[0] == counts[1]
    assert counts[1][0] in (window, 2 * window)  # of the last frame, or of both where the counts run on


def _batch(lib, hip, orc, e, frames, flags, S, thr):
    """One call with frames[1:], intra or inter by flag, each inter frame after frames[0]; checked against the oracle."""
    h, w = frames.shape[1:3]
    nb = (w // 4) * (h // 4)
    ref = orc.reencode(frames[0], orc.fit_frame(frames[0]), S, thr, True)["phys"]
    jobs = [dict(d_rgb=hip.Buffer.from_array(np.ascontiguousarray(f)), width=w, height=h, is_intra=flag,
                 d_ref=hip.Buffer.from_array(ref), d_phys=hip.Buffer(8 * nb), d_motion=hip.Buffer(2 * nb),
                 d_unique=hip.Buffer(4 * nb), d_n_unique=hip.Buffer(4), d_eps=hip.Buffer(6 * nb), d_kind=hip.Buffer(nb))
            for f, flag in zip(frames[1:], flags)]
    e.encode_batch_device(jobs)
    for i, (j, f, flag) in enumerate(zip(jobs, frames[1:], flags)):
        want = orc.reencode(f, orc.fit_frame(f), S, thr, flag, None if flag else ref)
        assert np.array_equal(j["d_phys"].download(np.uint64, nb), want["phys"]), (flags, i)
        assert np.array_equal(j["d_motion"].download(np.uint8, 2 * nb), want["motion"]), (flags, i)
    return e.stats()


# whether the intra search of a batch of these frames is pruned: small windows, thresholds up to the limit, few intra blocks
@pytest.mark.parametrize("S,thr,flags,pruned", [
    (8, 4, "IIIII", True), (8, 3, "IPPPP", True), (16, 2, "IIPPP", True), (16, 3, "IPPPP", True), (16, 3, "IIPPP", False),
    (16, 4, "IIIII", False), (16, 4, "PPPPP", True), (24, 1, "IIIPP", True), (24, 2, "IIIPP", False), (24, 4, "IPPPP", True)])
@pytest.mark.parametrize("graph", [0, 1])
def test_intra_search_pruned_by_its_share(orc, S, thr, flags, pruned, graph):
    """The inter search is pruned wherever there is one, the intra search by its
    limit; with graphs, calls of one shape and other flags follow each other."""
    from mptc_amd import hip, lib
    w, h = 100, 60
    frames = orc.synth_frames(SynthCfg(w, h, S + thr, 5, 1, 3, 8, 0), 6)
    e = lib.Encoder(w, h, search_area=S, err_threshold=thr, max_batch_frames=5, max_batch_blocks=5 * (w // 4) * (h // 4))
    e.set_tuning(use_graph=graph)
    for _ in range(2):
        st = _batch(lib, hip, orc, e, frames, [c == "I" for c in flags], S, thr)
        assert (st["exact_inter_candidates"] > 0) == ("P" in flags)
        assert (st["exact_intra_candidates"] > 0) == pruned
        if graph:
            _batch(lib, hip, orc, e, frames, [c == "I" for c in "IIIPI"], S, thr)
            _batch(lib, hip, orc, e, frames, [c == "I" for c in "PIPPP"], S, thr)
    e.close()


def test_autotune_tries_pruning_whatever_ran_before(orc):
    """A context last used for intra frames that are not pruned finds the pruned
    inter search, which is about twice as fast here."""
    from mptc_amd import hip, lib
    S, thr, w, h = 16, 3, 640, 360
    nb = (w // 4) * (h // 4)
    frames = orc.synth_frames(SynthCfg(w, h, 3, 5, 1, 3, 8, 0), 2)
    e = lib.Encoder(w, h, search_area=S, err_threshold=thr)
    ref = hip.Buffer(8 * nb)
    out = [hip.Buffer(2 * nb), hip.Buffer(4 * nb), hip.Buffer(4), hip.Buffer(6 * nb), hip.Buffer(nb)]
    e.encode_frame_device(hip.Buffer.from_array(frames[0]), w, h, True, None, ref, *out)
    assert e.stats()["exact_intra_candidates"] == 0
    e.set_tuning(prune=0)
    job = dict(d_rgb=hip.Buffer.from_array(frames[1]), width=w, height=h, is_intra=False, d_ref=ref, d_phys=hip.Buffer(8 * nb),
               d_motion=out[0], d_unique=out[1], d_n_unique=out[2], d_eps=out[3], d_kind=out[4])
    best, _ = e.autotune([job], 1)
    assert best["prune"] == 1
    e.close()


def test_context_without_room_for_the_pruned_tables(orc):
    """A context that takes most of the free memory, with no room for the pruned
    searches' tables, encodes as before, with every candidate evaluated."""
    import ctypes as C

    from mptc_amd import hip, lib
    S, w, h = 63, 64, 64
    free, total = C.c_size_t(), C.c_size_t()
    hip.check(hip.rt().hipMemGetInfo(C.byref(free), C.byref(total)))
    # a block of the context: E, 8 chunk summaries, words, tables and maps; the pruned tables are 6 % more
    per_block = 8 * S * S + 8 * 16 + 116
    blocks = int(0.955 * free.value) // per_block
    assert blocks * (64 + 1984) > free.value - blocks * per_block + (1 << 28)
    e = lib.Encoder(w, h, search_area=S, err_threshold=0, max_batch_frames=1, max_batch_blocks=blocks)
    frames = orc.synth_frames(SynthCfg(w, h, 3, 5, 1, 3, 8, 0), 2)
    for _ in range(2):
        for x, y in zip(e.encode_sequence(frames, 8), orc.encode_sequence(frames, S, 0, 8)):
            compare_results(x, y, "no room")
        assert e.stats()["exact_inter_candidates"] == 0
    e.close()
