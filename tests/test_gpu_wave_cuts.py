"""The wf-adaptive wave kernel (cut_pair) against the oracle: status, score,
every CIGAR operation and the diagonal-step count, which pins each step's
limits.  Cut-offs that change almost every step or none, that empty gap
wavefronts (whose cells the next records probe), pairs that leave 64 diagonals
(two per lane) and 128 (the lean kernel), end diagonals off to a side, and
pairs that reach the borders."""
import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen
from test_gpu_tiles import mutate, rand

pytestmark = pytest.mark.gpu


def reads(rng):
    P, T = [], []
    for i in range(400):
        t = rand(rng, int(rng.integers(1, 400)))
        P.append(mutate(rng, t, float(rng.uniform(0, 0.25)), 1 + 2 * (i % 3)))
        T.append(t.tobytes())
    return P, T


def off_side(rng):
    P, T = [], []
    for i in range(120):
        t = rand(rng, int(rng.integers(60, 500)))
        p = mutate(rng, t, 0.05, 1)
        cut = int(rng.integers(0, 75))
        if i % 2:
            P.append(p[cut:])
            T.append(t.tobytes())
        else:
            P.append(p)
            T.append(t.tobytes()[:max(1, len(t) - cut)])
    return P, T


def wide(rng):
    P = [rand(rng, int(rng.integers(40, 1000))).tobytes() for _ in range(60)]
    T = [rand(rng, max(1, len(p) + int(rng.integers(-40, 40)))).tobytes() for p in P]
    for _ in range(20):
        t = rand(rng, int(rng.integers(600, 1025)))
        P.append(mutate(rng, t, 0.3, 4))
        T.append(t.tobytes())
    return P, T


@pytest.mark.parametrize("make", [reads, off_side, wide], ids=lambda f: f.__name__)
@pytest.mark.parametrize("heur", [(4, 10, 50, 1), (4, 1, 3, 1), (4, 5, 12, 7), (4, 10, 1 << 30, 1)], ids=str)
def test_cut_waves_equal_oracle(heur, make):
    P, T = make(np.random.default_rng(17))
    P = [p[:1024] for p in P]
    ps = datagen.PairSet.from_lists(P, T)
    for pen in ((0, 4, 6, 2), (0, 2, 3, 1)):
        ref = O.oracle_align(O.Conf("affine", pen, "high", heuristic=heur), O.Pairs(P, T))
        for score_only in (False, True):
            print("%s %s %s score_only=%s: %d pairs" % (make.__name__, heur, pen, score_only, ps.n), flush=True)
            al = wfa_amd.Aligner(metric="affine", penalties=pen, heuristic=heur, score_only=score_only)
            db = al.upload(ps)
            db.run()
            got, st = db.download(cigars=not score_only), db.stats()
            if score_only:
                ref1 = O.oracle_align(O.Conf("affine", pen, "high", heuristic=heur, score_only=True), O.Pairs(P, T))
                assert np.array_equal(got.status, ref1.status) and np.array_equal(got.score, ref1.score)
                assert st.diagonal_steps == int(ref1.dsteps.sum())
                continue
            # (a trace through a wavefront that the cut-off emptied is refused)
            ok = [i for i in range(ps.n) if got.status[i] != wfa_amd.WF_STATUS_UNSUPPORTED]
            assert len(ok) >= 0.9 * ps.n
            bad = [i for i in ok if got.status[i] != ref.status[i] or got.score[i] != ref.score[i] or
                   got.ops(i) != ref.ops(i)]
            assert not bad, (bad[:10], got.status[bad[0]], got.score[bad[0]], ref.score[bad[0]])
            assert st.diagonal_steps == int(ref.dsteps.sum())
