"""The wave family (wfa_wave.hip) in a record arena that holds a fraction of
the pairs' records: the pairs run in rounds, and a pair that a wave does not
finish leaves no records behind."""
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen

pytestmark = pytest.mark.gpu

BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mutate(rng, t, e):
    u = rng.random(len(t))
    out = t.copy()
    sub = u < e / 3
    out[sub] = BASES[rng.integers(0, 4, int(sub.sum()))]
    reps = np.ones(len(t), dtype=np.int64)
    reps[(u >= e / 3) & (u < 2 * e / 3)] = 2
    reps[(u >= 2 * e / 3) & (u < e)] = 0
    return np.repeat(out, reps).tobytes()


@pytest.mark.parametrize("metric,pen,length,kw", [
    ("affine2p", (0, 4, 6, 2, 24, 1), 1000, {}),  # nearly all outgrow 4 diagonals per lane, half of them 8
    ("affine", (0, 4, 6, 2), 1000, {}),           # 8 diagonals per lane from the start
    ("affine", (0, 4, 6, 2), 1000, dict(heuristic=(4, 10, 50, 1))),
    ("affine2p", (0, 4, 6, 2, 24, 1), 300, {}),
    ("edit", (0, 1, 1), 1000, {})], ids=["2p-1000", "affine-1000", "adaptive-1000", "2p-300", "edit-1000"])
def test_rounds_in_a_small_arena(monkeypatch, metric, pen, length, kw):
    monkeypatch.setenv("WFA_RECORD_ARENA_MB", "64")
    rng = np.random.default_rng(31)
    P, T = [], []
    for i in range(100):
        t = BASES[rng.integers(0, 4, length - int(rng.integers(0, length // 10)))]
        P.append(mutate(rng, t, 0.06))
        T.append(t.tobytes())
    times = 60
    ref = O.oracle_align(O.Conf(metric, pen, "high", **kw), O.Pairs(P, T))
    ps = datagen.PairSet.from_lists(P * times, T * times)
    al = wfa_amd.Aligner(metric=metric, penalties=pen, **kw)
    db = al.upload(ps)
    for run in range(2):
        assert db.run() == 0
        got, st = db.download(), db.stats()
        say("%s: %d launches, %.1f ms" % (metric, st.forward_launches, st.forward_ms))
        assert st.diagonal_steps == times * int(ref.dsteps.sum())
        for i in range(ps.n):
            assert (got.status[i], got.score[i]) == (ref.status[i % 100], ref.score[i % 100]), i
            assert got.ops(i) == ref.ops(i % 100), i
