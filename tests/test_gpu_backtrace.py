"""The backtrace's operation stack and CIGAR writer against the oracle at the
edges of their words: slots of every size and alignment around 8 operations a
stack word and 16 bytes a store, from empty pairs to unrelated ones (a slot
full of operations), beside their neighbours' slots."""
import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen
from test_gpu_tiles import mutate, rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric,pen,free", [("affine", (0, 4, 6, 2), None), ("affine", (0, 3, 1, 4), None),
                                             ("affine2p", (0, 4, 6, 2, 24, 1), None), ("edit", (0, 1, 1), None),
                                             ("indel", (0, 1, 1), None), ("linear", (0, 4, 2), None),
                                             ("affine", (0, 4, 6, 2), (0, 0, 3, 5)), ("affine", (0, 4, 6, 2), (4, 2, 0, 3))],
                         ids=str)
def test_small_slots(metric, pen, free):
    rng = np.random.default_rng(5)
    P, T = [], []
    for i in range(1200):
        t = rand(rng, int(rng.integers(6 if free else 0, 40)))
        P.append(mutate(rng, t, float(rng.uniform(0, 0.6)), 3) if i % 3 else
                 rand(rng, int(rng.integers(6 if free else 0, 40))).tobytes())
        T.append(t.tobytes())
    if free:
        P = [p + b"ACGTAC"[:max(0, 6 - len(p))] for p in P]
    ps = datagen.PairSet.from_lists(P, T)
    print("%s %s %s: %d pairs" % (metric, pen, free, ps.n), flush=True)
    ref = O.oracle_align(O.Conf(metric, pen, "high", ends_free=free), O.Pairs(P, T))
    al = wfa_amd.Aligner(metric=metric, penalties=pen, ends_free=free)
    got = al.align_batch(ps)
    bad = [i for i in range(ps.n) if got.status[i] != ref.status[i] or got.score[i] != ref.score[i] or
           got.ops(i) != ref.ops(i)]
    assert not bad, (bad[:10], P[bad[0]], T[bad[0]], got.ops(bad[0]), ref.ops(bad[0]))
