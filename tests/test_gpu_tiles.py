"""Pairs above 1,024 bases in tiles of diagonals (wfa_tile.hip) against the
oracle: status, score, every CIGAR operation and the diagonal-step count
(which pins each step's [lo, hi], hence the trimming that only the first and
last tile of a pair do).

Beside mapped reads: unrelated sequences and sequences of very different
lengths (wavefronts that reach every border of the matrix, trimmed at both
ends over hundreds of steps), repeats and homopolymers (long match runs),
identical pairs, an empty side, and lengths around the tile width."""
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen

pytestmark = pytest.mark.gpu

SHAPES = [("affine", (0, 4, 6, 2)), ("affine", (0, 2, 3, 1)), ("affine2p", (0, 4, 6, 2, 24, 1)),
          ("affine2p", (0, 8, 12, 4, 48, 2))]
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mutate(rng, t, e, mean):
    out = []
    i = 0
    while i < len(t):
        u = rng.random()
        if u < e / 3:
            out.append(BASES[rng.integers(0, 4)])
        elif u < 2 * e / 3:
            out.extend(BASES[rng.integers(0, 4, rng.geometric(1 / mean))])
            out.append(t[i])
        elif u < e:
            i += int(rng.geometric(1 / mean)) - 1
        else:
            out.append(t[i])
        i += 1
    return np.array(out, dtype=np.uint8).tobytes()


def rand(rng, n):
    return BASES[rng.integers(0, 4, n)]


def mapped(seed):
    rng = np.random.default_rng(seed)
    P, T = [], []
    for i in range(24):
        t = rand(rng, int(rng.integers(1025, 3000)))
        P.append(mutate(rng, t, float(rng.uniform(0, 0.18)), 1 + 2 * (i % 2)))
        T.append(t.tobytes())
    return datagen.PairSet.from_lists(P, T)


def borders(seed):
    rng = np.random.default_rng(seed)
    P = [rand(rng, n).tobytes() for n in (1025, 1100, 300, 1300, 40, 1500, 1)]
    T = [rand(rng, n).tobytes() for n in (1025, 1300, 1100, 280, 1400, 35, 1200)]
    sk = datagen.skewed(seed, 4, tlen=(300, 600), insert=(900, 1200))
    return datagen.PairSet.from_lists(P + sk.patterns(), T + sk.texts())


def odd(seed):
    rng = np.random.default_rng(seed)
    t = rand(rng, 2048).tobytes()
    P = [t, b"", t[:1100], b"A" * 1200, b"AC" * 700, b"A" * 1500, t[:1024] + b"G" + t[1024:], t[500:1800]]
    T = [t, t[:1030], b"", b"A" * 1100, b"AC" * 690 + b"A", b"T" * 1030, t, t]
    for n in range(1025, 1025 + 12):
        u = rand(rng, n)
        P.append(mutate(rng, u, 0.02, 1))
        T.append(u.tobytes())
    return datagen.PairSet.from_lists(P, T)


@pytest.mark.parametrize("make", [mapped, borders, odd], ids=lambda f: f.__name__)
@pytest.mark.parametrize("metric,pen", SHAPES, ids=["%s%s" % (m, p) for m, p in SHAPES])
def test_tiles_equal_oracle(metric, pen, make):
    ps = make(77)
    ref = O.oracle_align(O.Conf(metric, pen, "high"), O.Pairs(ps.patterns(), ps.texts()))
    for score_only in (False, True):
        say("%s %s %s score_only=%s: %d pairs" % (make.__name__, metric, pen, score_only, ps.n))
        al = wfa_amd.Aligner(metric=metric, penalties=pen, score_only=score_only)
        db = al.upload(ps)
        assert db.run() == 0
        got, st = db.download(cigars=not score_only), db.stats()
        bad = [i for i in range(ps.n) if got.status[i] != ref.status[i] or got.score[i] != ref.score[i] or
               (not score_only and got.ops(i) != ref.ops(i))]
        assert not bad, (bad, got.status[bad[0]], got.score[bad[0]], ref.score[bad[0]])
        assert st.diagonal_steps == int(ref.dsteps.sum())
        assert st.forward_launches <= 2, "most pairs must stay in their tiles"
