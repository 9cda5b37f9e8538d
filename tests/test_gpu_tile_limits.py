"""Pairs whose sequences just fill the tiles' LDS (64 KB for both: 131,007
bases, in BiWFA 130,975) and the next longer ones, which run on the HBM-ring
kernel and from the start on one workgroup or team, against the oracle."""
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


def pair(rng, n):
    t = BASES[rng.integers(0, 4, n)]
    p = t.copy()
    at = rng.integers(0, n, 24)
    p[at] = BASES[rng.integers(0, 4, 24)]
    p = np.delete(p, rng.integers(0, n, 3))
    return p.tobytes(), t.tobytes()


@pytest.mark.parametrize("memory,metric,pen,longest", [
    ("high", "affine", (0, 4, 6, 2), 131007), ("high", "affine2p", (0, 4, 6, 2, 24, 1), 131007),
    ("ultralow", "affine", (0, 4, 6, 2), 130975)])
def test_longest_pairs_of_the_tiles(memory, metric, pen, longest):
    rng = np.random.default_rng(21)
    for n in (longest, longest + 1):
        p, t = pair(rng, n)
        ps = datagen.PairSet.from_lists([p, t], [t, p])  # the longest pattern, the longest text
        for score_only in (True, False):
            say("%s %s %d score_only=%s" % (memory, metric, n, score_only))
            al = wfa_amd.Aligner(metric=metric, penalties=pen, memory=memory, score_only=score_only)
            db = al.upload(ps)
            assert db.run() == 0
            got = db.download(cigars=not score_only)
            ref = O.oracle_align(O.Conf(metric, pen, memory, score_only), O.Pairs(ps.patterns(), ps.texts()))
            for i in range(ps.n):
                assert (got.status[i], got.score[i]) == (ref.status[i], ref.score[i])
                assert score_only or got.ops(i) == ref.ops(i)
            db.free()
            al.close()
