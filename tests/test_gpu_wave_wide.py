"""Pairs that outgrow 4 diagonals per lane within a group large enough for the
second launch of the wave family (8 per lane, straight behind the first),
against the oracle: beside pairs that stay, pairs that outgrow 8 too (tiles or
the ring families), and several pairs more than the second launch has
workgroups on none or all of them."""
import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen
from test_gpu_tiles import mutate, rand

pytestmark = pytest.mark.gpu


def pairs(seed, n, share):
    rng = np.random.default_rng(seed)
    P, T = [], []
    for i in range(n):
        if rng.random() < share:  # unrelated or far apart in length: hundreds of diagonals
            t = rand(rng, int(rng.integers(120, 320)))
            p = rand(rng, int(rng.integers(100, 320))).tobytes()
        else:
            t = rand(rng, int(rng.integers(40, 120)))
            p = mutate(rng, t, float(rng.uniform(0, 0.1)), 1)
        P.append(p)
        T.append(t.tobytes())
    return P, T


@pytest.mark.parametrize("share", [0.0, 0.03, 1.0])
@pytest.mark.parametrize("metric,pen,free", [("affine2p", (0, 4, 6, 2, 24, 1), None),
                                             ("affine", (0, 4, 6, 2), (0, 0, 20, 20)), ("edit", (0, 1, 1), (0, 7, 0, 9))],
                         ids=str)
def test_second_launch_equals_oracle(metric, pen, free, share):
    P, T = pairs(29, 2300, share)
    P = [p if len(p) >= 30 else p + b"ACGTTGCAAC" * 3 for p in P]
    ps = datagen.PairSet.from_lists(P, T)
    ref = O.oracle_align(O.Conf(metric, pen, "high", ends_free=free), O.Pairs(P, T))
    for score_only in (False, True):
        print("%s %s share %g score_only=%s: %d pairs" % (metric, free, share, score_only, ps.n), flush=True)
        al = wfa_amd.Aligner(metric=metric, penalties=pen, ends_free=free, score_only=score_only)
        db = al.upload(ps)
        for _ in range(2):
            assert db.run() == 0
            got, st = db.download(cigars=not score_only), db.stats()
            bad = [i for i in range(ps.n) if got.status[i] != ref.status[i] or
                   (not score_only and (got.score[i] != ref.score[i] or got.ops(i) != ref.ops(i)))]
            assert not bad, (bad[:10], got.status[bad[0]], got.score[bad[0]], ref.score[bad[0]])
            assert st.diagonal_steps == int(ref.dsteps.sum())
