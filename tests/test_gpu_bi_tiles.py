"""Breakpoint searches of large BiWFA sub-problems advanced in tiles
(bi_tile_kernel) against the oracle: status, score, every CIGAR operation and
the diagonal-step count.

Beside mapped reads: identical pairs and pairs that meet within the first
block, very different lengths and unrelated sequences (sides that touch the
matrix's borders, which ends the tiles' part early), repeats (breakpoints with
many equal candidates), and symbol counts around the threshold."""
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen
from test_gpu_tiles import BASES, mutate, rand

pytestmark = pytest.mark.gpu


def mapped(rng):
    P, T = [], []
    for i in range(14):
        t = rand(rng, int(rng.integers(2100, 6000)))
        P.append(mutate(rng, t, float(rng.uniform(0.002, 0.2)), 1 + 3 * (i % 3)))
        T.append(t.tobytes())
    return P, T


def edges(rng):
    t = rand(rng, 5000)
    P = [t.tobytes(), mutate(rng, t, 0.0008, 1), t[2100:4400].tobytes(), (b"ACAC" * 700), b"A" * 2300,
         rand(rng, 2200).tobytes(), rand(rng, 600).tobytes(), rand(rng, 7).tobytes(),
         (t[:2000].tobytes() + t[3000:].tobytes())]
    T = [t.tobytes(), t.tobytes(), t.tobytes(), (b"ACAC" * 650 + b"CA" * 90), b"A" * 1900,
         rand(rng, 2100).tobytes(), t[:3600].tobytes(), t[:4100].tobytes(), t.tobytes()]
    return P, T


def threshold(rng):
    P, T = [], []
    for n in list(range(508, 517)) + [768, 1500]:
        t = rand(rng, n)
        P.append(mutate(rng, t, 0.06, 1)[:n])
        T.append(t.tobytes())
    return P, T


@pytest.mark.parametrize("make", [mapped, edges, threshold], ids=lambda f: f.__name__)
@pytest.mark.parametrize("pen", [(0, 4, 6, 2), (0, 2, 3, 1)], ids=str)
def test_tiled_searches_equal_oracle(pen, make):
    ps = datagen.PairSet.from_lists(*make(np.random.default_rng(91)))
    ref = O.oracle_align(O.Conf("affine", pen, "ultralow"), O.Pairs(ps.patterns(), ps.texts()))
    for score_only in (False, True):
        print("%s %s score_only=%s: %d pairs" % (make.__name__, pen, score_only, ps.n), flush=True)
        al = wfa_amd.Aligner(metric="affine", penalties=pen, memory="ultralow", score_only=score_only)
        db = al.upload(ps)
        assert db.run() == 0
        got, st = db.download(cigars=not score_only), db.stats()
        bad = [i for i in range(ps.n) if got.status[i] != ref.status[i] or
               (not score_only and (got.score[i] != ref.score[i] or got.ops(i) != ref.ops(i)))]
        assert not bad, (bad, got.status[bad[0]], got.score[bad[0]], ref.score[bad[0]])
        if score_only:
            ref1 = O.oracle_align(O.Conf("affine", pen, "ultralow", score_only=True), O.Pairs(ps.patterns(), ps.texts()))
            assert np.array_equal(got.score, ref1.score)
            assert st.diagonal_steps == int(ref1.dsteps.sum())
        else:
            assert st.diagonal_steps == int(ref.dsteps.sum())
