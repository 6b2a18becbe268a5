"""The pruned search's bound (bound_table / bound_prunes in mptc_amd/csrc),
restated in numpy with the kernel's fp32 operations, against the oracle's exact
candidate evaluation: no candidate it prunes passes, and its rounding stays
far below the margin of 16."""
from __future__ import annotations

import numpy as np
import pytest

from mptc_amd.workloads import SynthCfg

F = np.float32
WEIGHT = np.array([3, 0, 2, 1])


def _fma(a, b, c):
    return F(np.float64(a) * np.float64(b) + np.float64(c))  # one rounding, up to a double's


def line_bound(px48, word):
    """(L_c in fp32, L_c in float64, slack) of a word; slack 1e9: never pruned."""
    px = px48.reshape(16, 3).astype(np.int64) - 128
    idx = (int(word) >> (2 * np.arange(16))) & 3
    wa = WEIGHT[idx]
    aa, sa, n23 = int((wa * wa).sum()), int(wa.sum()), int((idx >= 2).sum())
    bb, ab = 144 - 6 * sa + aa, 3 * sa - aa
    assert bb == int(((3 - wa) ** 2).sum()) and ab == int((wa * (3 - wa)).sum())
    det = aa * bb - ab * ab
    q = int((px * px).sum())
    if det == 0:
        return F(q), float(q), 1e9
    s = min(F(1 / 3), F(n23) * F(1 / 24))
    r = max(s, F(2 / 3) - s)
    eta = np.sqrt(F(3) * (F(16 - n23) * s * s + F(n23) * r * r)) + F(0.001)
    inv = F(1) / F(det)
    k = [F(bb) * inv, F(-2 * ab) * inv, F(aa) * inv]
    ex, exact = F(0), 0.0
    for ch in range(3):
        A, p3 = int((wa * px[:, ch]).sum()), 3 * int(px[:, ch].sum())
        B = p3 - A
        ex = _fma(F(A), _fma(k[1], F(B), k[0] * F(A)), ex)
        ex = _fma(F(B), k[2] * F(B), ex)
        exact += (bb * A * A - 2 * ab * A * B + aa * B * B) / det
    return F(q) - ex, q - exact, float(eta)


def prunes(px48, word, err_own, thr):
    L, _, eta = line_bound(px48, word)
    r = np.sqrt(F(48 * (thr + err_own + 1))) + F(eta)
    return L >= _fma(r, r, F(16))


def _blocks(orc):
    f = orc.synth_frames(SynthCfg(160, 96, 9, 6, 1, 4, 8, 0), 1)[0]
    px = f.reshape(24, 4, 40, 4, 3).transpose(0, 2, 1, 3, 4).reshape(-1, 48)
    rng = np.random.default_rng(4)
    yield from px[rng.choice(len(px), 30, replace=False)]
    yield np.full(48, 77, np.uint8)
    yield np.where(rng.random(48) < 0.5, 0, 255).astype(np.uint8)
    yield np.repeat(np.where(np.arange(16) % 3 == 0, 250, 3), 3).astype(np.uint8)
    yield rng.integers(0, 256, 48).astype(np.uint8)


@pytest.mark.parametrize("thr", [0, 2, 4, 16])
def test_no_pruned_candidate_passes(orc, thr):
    rng = np.random.default_rng(thr)
    words = None
    pruned = passing = 0
    for px in _blocks(orc):
        own = int(orc.fit_block(px))
        near = [own >> 32 ^ (int(b) << (2 * int(i))) for b, i in zip(rng.integers(1, 4, 40), rng.integers(0, 16, 40))]
        words = near + [int(w) for w in rng.integers(0, 1 << 32, 60, dtype=np.uint64)] + [own >> 32, 0, 0xAAAAAAAA, 0xAAAAAAAB]
        e1, e2 = own & 0xFFFF, own >> 16 & 0xFFFF
        eo = orc.error(orc.p2l(own), px)
        for w in words:
            L32, L64, _ = line_bound(px, w)
            assert abs(float(L32) - L64) < 2.0
            ok, e, _, _ = orc.eval_candidate(own, px, w)
            p = e1 > e2 and bool(prunes(px, w, eo, thr))
            pruned += p
            passing += ok and e <= thr
            assert not (p and ok and e <= thr), f"pruned a passing word {w:#010x}: delta {e}"
    assert pruned > 200 and passing > 30


def test_planted_mistakes_are_caught(orc):
    """Weights of the wrong endpoint, a dropped slack and a limit without the own
    error each prune a candidate that passes."""
    caught = {"order": 0, "own": 0}
    for px in _blocks(orc):
        own = int(orc.fit_block(px))
        if own & 0xFFFF <= own >> 16 & 0xFFFF:
            continue
        eo = orc.error(orc.p2l(own), px)
        w = own >> 32
        L, _, eta = line_bound(px, w ^ 0xAAAAAAAA)  # index values 0 <-> 2, 1 <-> 3: another order along the line
        r = np.sqrt(48.0 * (eo + 1)) + eta
        caught["order"] += bool(L >= r * r + 16)
        caught["own"] += bool(line_bound(px, w)[0] >= (np.sqrt(48.0) + eta) ** 2 + 16)
    assert all(caught.values()), caught
