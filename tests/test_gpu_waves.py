"""Pairs of at most 1,024 bases on the wave family (wfa_wave.hip) against the
oracle: status, score, every CIGAR operation and the diagonal-step count.

The sets reach every phase of the kernels (1, 2, 4 and 8 diagonals per lane,
and past them: unrelated sequences of up to 1,024 bases outgrow a wave), the
matrix borders at every score (tiny and very uneven pairs, empty sides, where
ranges are trimmed and null wavefronts count), repeats, 8-bit symbols (with
and without distinct low halves), and the ends-free form with flanks that
start in each phase."""
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen

pytestmark = pytest.mark.gpu

SHAPES = [("affine", (0, 4, 6, 2)), ("affine", (0, 6, 9, 3)), ("edit", (0, 1, 1)), ("indel", (0, 1, 1)),
          ("linear", (0, 4, 2)), ("linear", (0, 2, 1)), ("affine2p", (0, 4, 6, 2, 24, 1)),
          ("affine2p", (0, 8, 12, 4, 48, 2))]
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mutate(rng, t, e):
    out = []
    for c in t:
        u = rng.random()
        if u < e / 3:
            out.append(BASES[rng.integers(0, 4)])
        elif u < 2 * e / 3:
            out.extend((BASES[rng.integers(0, 4)], c))
        elif u >= e:
            out.append(c)
    return np.array(out, dtype=np.uint8).tobytes()


def rand(rng, n):
    return BASES[rng.integers(0, 4, n)].tobytes()


def mapped(rng):
    P, T = [], []
    for i in range(400):
        t = np.frombuffer(rand(rng, int(rng.integers(1, 330 if i % 4 else 1024))), dtype=np.uint8)
        P.append(mutate(rng, t, float(rng.uniform(0, 0.3))))
        T.append(t.tobytes())
    return P, T


def borders(rng):
    P = [rand(rng, int(n)) for n in rng.integers(0, 30, 300)]
    T = [rand(rng, int(n)) for n in rng.integers(0, 30, 300)]
    for n, m in ((100, 100), (250, 260), (320, 20), (5, 300), (0, 200), (600, 640), (1024, 1024), (1024, 30)):
        P.append(rand(rng, n))
        T.append(rand(rng, m))
    P += [b"A" * 90, b"AC" * 60, b"A" * 33, b"ACG" * 100, b"T" * 200, b"A" * 64]
    T += [b"A" * 70, b"AC" * 55 + b"A", b"C" * 33, b"ACG" * 100, b"T" * 190 + b"G" * 9, b"A" * 64]
    return P, T


def wider(rng):
    P, T = mapped(rng)
    P = [bytes(b"N"[0] if rng.random() < 0.03 else c for c in p) for p in P[:120]]
    return P, T[:120]


def clashing(rng):  # 'A' and 'Q' share their low four bits
    P, T = mapped(rng)
    return [p.replace(b"ACG", b"QCG") for p in P[:60]], T[:60]


def check(metric, pen, ps, **kw):
    conf = O.Conf(metric, pen, "high", **kw)
    ref = O.oracle_align(conf, O.Pairs(ps.patterns(), ps.texts()))
    for score_only in (False, True):
        say("%s %s %s score_only=%s: %d pairs" % (metric, pen, kw, score_only, ps.n))
        al = wfa_amd.Aligner(metric=metric, penalties=pen, score_only=score_only, **kw)
        db = al.upload(ps)
        assert db.run() == 0
        got, st = db.download(cigars=not score_only), db.stats()
        want = ref if not (kw and score_only) else O.oracle_align(
            O.Conf(metric, pen, "high", True, **kw), O.Pairs(ps.patterns(), ps.texts()))
        bad = [i for i in range(ps.n) if got.status[i] != want.status[i] or got.score[i] != want.score[i] or
               (not score_only and got.ops(i) != want.ops(i))]
        assert not bad, (bad[:10], ps.pattern(bad[0]), ps.text(bad[0]), got.score[bad[0]], want.score[bad[0]])
        assert st.diagonal_steps == int(ref.dsteps.sum())


@pytest.mark.parametrize("make", [mapped, borders, wider, clashing], ids=lambda f: f.__name__)
@pytest.mark.parametrize("metric,pen", SHAPES, ids=["%s%s" % (m, p) for m, p in SHAPES])
def test_waves_equal_oracle(metric, pen, make):
    P, T = make(np.random.default_rng(5))
    check(metric, pen, datagen.PairSet.from_lists(P, T))


@pytest.mark.parametrize("free", [(0, 0, 30, 30), (12, 7, 0, 25), (40, 40, 40, 40), (0, 0, 90, 90), (100, 0, 90, 0)],
                         ids=str)
def test_ends_free_waves_equal_oracle(free):
    rng = np.random.default_rng(11)
    P, T = [], []
    for i in range(150):
        t = np.frombuffer(rand(rng, int(rng.integers(110, 400))), dtype=np.uint8)
        core = t[int(rng.integers(0, 20)):len(t) - int(rng.integers(0, 20))]
        p = mutate(rng, core, float(rng.uniform(0, 0.2))) if i % 10 else rand(rng, 120)
        P.append(p if len(p) >= 100 else rand(rng, 105))
        T.append(t.tobytes())
    for metric, pen in (("affine", (0, 4, 6, 2)), ("affine2p", (0, 4, 6, 2, 24, 1))):
        check(metric, pen, datagen.PairSet.from_lists(P, T), ends_free=free)
