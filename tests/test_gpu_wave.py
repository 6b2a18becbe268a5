"""Intra search in dependency order (k_intra_wave) against the CPU oracle, at
the sizes where its window, its rings and its id tables have their edges."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests.helpers import compare_results

pytestmark = pytest.mark.gpu


def log(msg: str):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def enc():
    from mptc_amd import lib
    e = lib.Encoder(512, 512, search_area=32, err_threshold=0, max_batch_frames=3, max_batch_blocks=3 * 128 * 128)
    yield e
    e.close()


def _frame(kind: str, w: int, h: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    if kind == "noise":  # words that few blocks can reuse
        return rng.integers(0, 256, (h, w, 3)).astype(np.uint8)
    yy, xx = np.mgrid[0:h, 0:w]
    img = np.stack([30 + xx // 3, 60 + yy // 2, 200 - (xx + yy) // 5], -1)
    if kind == "flat":  # wide steps: equal words, blocks that keep their own
        return np.clip(img // 32 * 32, 0, 255).astype(np.uint8)
    return np.clip(img + rng.integers(-8, 9, (h, w, 3)), 0, 255).astype(np.uint8)


def _intra(enc, orc, rgb, S, thr):
    enc.set_params(S, thr)
    fit = enc.fit(rgb)
    got = enc.reencode(rgb, fit, True)
    want = orc.reencode(rgb, fit, S, thr, True)
    compare_results(got, want, f"{rgb.shape[1]}x{rgb.shape[0]} S={S} thr={thr}")
    assert np.array_equal(got["kind"], want["kind"])


# one block; one row; one column; narrower and wider than the window; rows of 15, 16, 17 and 63-65 blocks (staging
# groups, polled vectors, need chunks); S at its ends, odd, and past the ring and id sizes' steps
@pytest.mark.parametrize("kind,w,h,S,thr", [
    ("soft", 4, 4, 1, 8), ("soft", 260, 4, 8, 8), ("soft", 4, 200, 8, 8), ("soft", 28, 60, 8, 5), ("soft", 60, 40, 8, 8),
    ("soft", 64, 48, 1, 8), ("soft", 68, 48, 2, 30), ("flat", 68, 52, 3, 8), ("soft", 252, 64, 4, 8), ("soft", 256, 64, 5, 16),
    ("soft", 260, 64, 7, 8), ("soft", 300, 120, 8, 30000), ("flat", 300, 120, 8, 8), ("noise", 200, 100, 8, 300),
    ("soft", 200, 100, 9, 8), ("soft", 220, 96, 15, 8), ("soft", 220, 96, 16, 6), ("noise", 160, 160, 16, 900),
    ("soft", 260, 132, 17, 8), ("soft", 300, 140, 31, 12), ("soft", 300, 140, 32, 8), ("flat", 264, 132, 32, 32)])
def test_intra_wave_matches_oracle(enc, orc, kind, w, h, S, thr):
    log(f"{kind} {w}x{h} S={S} thr={thr}")
    enc.profile_enable(True)
    _intra(enc, orc, _frame(kind, w, h, w + h + S), S, thr)
    launches, _ = enc.profile_read("intra_wave")
    enc.profile_enable(False)
    assert launches == 1


def test_more_distinct_words_than_ids(enc, orc):
    """A noise frame holds more distinct words than the S = 32 window has ids:
    the fixpoint passes take over, with the same result."""
    rgb = _frame("noise", 300, 280, 5)
    enc.profile_enable(True)
    _intra(enc, orc, rgb, 32, 8)
    waves, passes = enc.profile_read("intra_wave")[0], enc.profile_read("intra_reeval")[0]
    enc.profile_enable(False)
    assert waves == 1 and passes > 0


def test_batch_of_intra_and_inter_frames(enc, orc):
    """One call with intra and inter frames of uneven sizes: every frame as by itself."""
    from mptc_amd import hip
    S, thr = 8, 8
    enc.set_params(S, thr)
    jobs, want = [], []
    for i, (w, h, intra) in enumerate([(200, 100, True), (64, 120, False), (324, 36, True)]):
        a, b = _frame("soft", w, h, 10 + i), _frame("soft", w, h, 20 + i)
        nb = (w // 4) * (h // 4)
        ref = orc.reencode(a, orc.fit_frame(a), S, thr, True)["phys"]
        want.append(orc.reencode(b, orc.fit_frame(b), S, thr, intra, None if intra else ref))
        jobs.append(dict(d_rgb=hip.Buffer.from_array(b), width=w, height=h, is_intra=intra, d_ref=hip.Buffer.from_array(ref),
                         d_phys=hip.Buffer(8 * nb), d_motion=hip.Buffer(2 * nb), d_unique=hip.Buffer(4 * nb),
                         d_n_unique=hip.Buffer(4), d_eps=hip.Buffer(6 * nb), d_kind=hip.Buffer(nb)))
    enc.encode_batch_device(jobs)
    for i, (j, wnt) in enumerate(zip(jobs, want)):
        nb = (j["width"] // 4) * (j["height"] // 4)
        n = int(j["d_n_unique"].download(np.uint32, 1)[0])
        got = dict(phys=j["d_phys"].download(np.uint64, nb), motion=j["d_motion"].download(np.uint8, 2 * nb),
                   unique=j["d_unique"].download(np.uint32, n), eps=j["d_eps"].download(np.uint8, 6 * nb))
        compare_results(got, wnt, f"frame {i}")


@pytest.mark.parametrize("w,h,S,thr,seed", [(1920, 1080, 8, 8, 3), (1280, 720, 16, 8, 4), (960, 540, 32, 16, 5)])
def test_intra_wave_matches_tile_passes(w, h, S, thr, seed):
    """Ordinary frame sizes, where ids are given out and taken back thousands of
    times a row: the same bytes as the tile-resolved fixpoint passes, and the
    same from one encode to the next."""
    from mptc_amd import lib
    from mptc_amd.workloads import SynthCfg
    rgb = lib.synth_frames(SynthCfg(w, h, seed, 32, 1, 4, 8, 10), 0, 1)[0]
    e = lib.Encoder(w, h, S, thr)
    fit = e.fit(rgb)
    runs = [e.reencode(rgb, fit, True) for _ in range(4)]
    e.set_tuning(itile_w=8)
    want = e.reencode(rgb, fit, True)
    e.close()
    for i, r in enumerate(runs):
        compare_results(r, want, f"{w}x{h} S={S} thr={thr} run {i}")
        assert np.array_equal(r["kind"], want["kind"])


@pytest.mark.parametrize("S,thr", [(9, 300), (10, 8), (12, 300), (16, 8), (16, 300)])
def test_rows_that_pass_the_four_lane_limit(enc, orc, S, thr):
    """Rows that begin with few distinct words and end with more than four lanes
    each are kept for: the split of the ids changes in the middle of them."""
    w, h = 320, 128
    rgb = _frame("flat", w, h, 3)
    noise = _frame("noise", w, h, 4)
    for i, x0 in enumerate(range(0, w, 32)):  # block rows pass the limit at different columns
        y0 = (40 + 24 * i) % h
        rgb[y0:, x0 + 16:x0 + 32] = noise[y0:, x0 + 16:x0 + 32]
    rgb[:, w // 2:] = noise[:, w // 2:]
    log(f"S={S} thr={thr}")
    _intra(enc, orc, rgb, S, thr)


@pytest.mark.parametrize("S,thr", [(2, 8), (3, 8), (4, 8), (4, 32), (5, 6), (6, 8)])
def test_small_windows_have_ids_enough(enc, orc, S, thr):
    """Rows of many reused words at small search areas are decided without the
    fixpoint passes."""
    log(f"S={S} thr={thr}")
    rgb = _frame("soft", 480, 256, 40 + S)
    _intra(enc, orc, rgb, S, thr)
    assert enc.stats()["intra_iterations"] == 1


def _route(enc, run):
    """The call's result and whether the fixpoint passes followed the wave."""
    enc.profile_enable(True)
    got = run()
    passes = enc.profile_read("intra_reeval")[0]
    enc.profile_enable(False)
    return got, passes > 0


# content and size by which a batch is left to the passes: hardly any reuse, and words that change for few blocks
@pytest.mark.parametrize("kind,w,h,S,thr,passes", [
    ("noise", 320, 200, 8, 8, True), ("noise", 64, 64, 16, 8, True), ("noise", 320, 200, 4, 32, True),
    ("noise", 200, 200, 32, 8, True), ("flat", 400, 300, 16, 5, True), ("soft", 400, 300, 8, 8, False),
    ("soft", 64, 64, 8, 32, False), ("soft", 300, 200, 32, 16, False), ("soft", 400, 300, 5, 32, False)])
def test_route_by_reuse(enc, orc, kind, w, h, S, thr, passes):
    log(f"{kind} {w}x{h} S={S} thr={thr}")
    _, by_passes = _route(enc, lambda: _intra(enc, orc, _frame(kind, w, h, w + S), S, thr))
    assert by_passes == passes


def _window(bw, bh, S):
    """Intra window positions of a frame whose blocks all search."""
    return sum(min(y, 2 * S - 1) * (min(bw, x + S) - max(0, x - S)) + x - max(0, x - S) for y in range(bh) for x in range(bw))


# edges of the window, its rings, staging groups and polled vectors, with words that most blocks reuse
@pytest.mark.parametrize("w,h,S", [(68, 400, 1), (200, 200, 1), (260, 160, 3), (16, 240, 8), (60, 40, 8), (252, 64, 8), (256, 64, 8),
                                   (260, 64, 7), (200, 100, 9), (220, 96, 15), (220, 96, 16), (260, 132, 17), (300, 140, 31),
                                   (300, 140, 32)])
def test_edges_with_wide_reuse(enc, orc, w, h, S):
    log(f"{w}x{h} S={S}")
    _, by_passes = _route(enc, lambda: _intra(enc, orc, _frame("soft", w, h, w + h), S, 64))
    assert not by_passes
    assert enc.stats()["intra_candidates"] == _window(w // 4, h // 4, S)


def test_ids_run_out_in_a_frame_of_wide_reuse(enc, orc):
    """Reuse over half a frame and noise in the other: the wave begins, a window
    holds more distinct words than ids, and the passes take the frame."""
    w, h, S = 400, 300, 32
    rgb = _frame("soft", w, h, 6)
    rgb[:, w // 2:] = _frame("noise", w, h, 7)[:, w // 2:]
    _, by_passes = _route(enc, lambda: _intra(enc, orc, rgb, S, 8))
    assert by_passes
    assert enc.stats()["intra_candidates"] == _window(w // 4, h // 4, S)


def test_small_intra_frame_among_inter_frames(enc, orc):
    """An intra frame of few blocks does not send the batch's inter frames
    through the wave."""
    from mptc_amd import hip
    S, thr = 8, 8
    enc.set_params(S, thr)
    jobs, want = [], []
    for i, (w, h, intra) in enumerate([(32, 32, True), (400, 300, False), (400, 300, False)]):
        a = _frame("soft", w, h, 10 + i)
        b = np.clip(a.astype(int) + _frame("noise", w, h, 20 + i) % 5 - 2, 0, 255).astype(np.uint8)
        nb = (w // 4) * (h // 4)
        ref = orc.reencode(a, orc.fit_frame(a), S, thr, True)["phys"]
        want.append(orc.reencode(b, orc.fit_frame(b), S, thr, intra, None if intra else ref))
        jobs.append(dict(d_rgb=hip.Buffer.from_array(b), width=w, height=h, is_intra=intra, d_ref=hip.Buffer.from_array(ref),
                         d_phys=hip.Buffer(8 * nb), d_motion=hip.Buffer(2 * nb), d_unique=hip.Buffer(4 * nb),
                         d_n_unique=hip.Buffer(4), d_eps=hip.Buffer(6 * nb), d_kind=hip.Buffer(nb)))
    _, by_passes = _route(enc, lambda: enc.encode_batch_device(jobs))
    assert by_passes
    for i, (j, wnt) in enumerate(zip(jobs, want)):
        nb = (j["width"] // 4) * (j["height"] // 4)
        assert np.array_equal(j["d_phys"].download(np.uint64, nb), wnt["phys"]), f"frame {i}"
        assert np.array_equal(j["d_motion"].download(np.uint8, 2 * nb), wnt["motion"]), f"frame {i}"


@pytest.mark.parametrize("kind,S,thr", [("soft", 8, 8), ("soft", 3, 32), ("noise", 8, 8), ("flat", 5, 6)])
def test_allocation_free_call_takes_the_same_routes(orc, kind, S, thr):
    from mptc_amd import hip, lib
    w, h = 300, 200
    nb = (w // 4) * (h // 4)
    rgb = _frame(kind, w, h, 30 + S)
    d_rgb = hip.Buffer.from_array(rgb)
    o = [hip.Buffer(8 * nb), hip.Buffer(2 * nb), hip.Buffer(4 * nb), hip.Buffer(4), hip.Buffer(6 * nb), hip.Buffer(nb)]
    stream = hip.Stream()
    want = orc.reencode(rgb, orc.fit_frame(rgb), S, thr, True)
    for _ in range(2):
        lib.encode_frame_noalloc(0, d_rgb, w, h, S, thr, True, None, *o, stream=stream.handle)
        assert np.array_equal(o[0].download(np.uint64, nb), want["phys"])
        assert np.array_equal(o[1].download(np.uint8, 2 * nb), want["motion"])
    stream.destroy()


def test_replayed_graphs_take_the_route_of_each_frame(orc):
    """Graphs captured on one frame are replayed on others of its shape: frames
    for the wave, for the passes, and one that the wave gives up on, in turn."""
    from mptc_amd import hip, lib
    S, thr, w, h = 32, 8, 320, 240
    nb = (w // 4) * (h // 4)
    mixed = _frame("soft", w, h, 6)
    mixed[:, w // 2:] = _frame("noise", w, h, 7)[:, w // 2:]
    frames = [_frame("soft", w, h, 5), _frame("noise", w, h, 8), mixed, _frame("soft", w, h, 9)]
    want = [orc.reencode(f, orc.fit_frame(f), S, thr, True) for f in frames]
    e = lib.Encoder(w, h, S, thr)
    e.set_tuning(use_graph=1)
    d = [hip.Buffer.from_array(f) for f in frames]
    o = [hip.Buffer(8 * nb), hip.Buffer(2 * nb), hip.Buffer(4 * nb), hip.Buffer(4), hip.Buffer(6 * nb), hip.Buffer(nb)]
    its = []
    for k in (0, 1, 2, 3, 1, 0, 2, 0):
        e.encode_frame_device(d[k], w, h, True, None, *o)
        e.synchronize()
        assert np.array_equal(o[0].download(np.uint64, nb), want[k]["phys"]), k
        assert np.array_equal(o[1].download(np.uint8, 2 * nb), want[k]["motion"]), k
        its.append((k, e.stats()["intra_iterations"]))
    assert all((n == 1) == (k in (0, 3)) for k, n in its), its
    e.close()
