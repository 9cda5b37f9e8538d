"""Run counts made by the backtrace (and, for batches with pairs in tiles, by
the counting pass) against the runs of the CIGARs themselves: leading and
trailing free gaps, gaps next to each other, empty and failed pairs."""
import itertools

import numpy as np
import pytest

import wfa_amd
from wfa_amd import datagen
from test_gpu_tiles import mutate, rand

pytestmark = pytest.mark.gpu

CODES = {ord("M"): 7, ord("X"): 8, ord("I"): 1, ord("D"): 2}


@pytest.mark.parametrize("long_pairs", [0, 3], ids=["counted", "with_tiles"])
@pytest.mark.parametrize("metric,pen,kw", [("affine", (0, 4, 6, 2), {}), ("affine", (0, 4, 6, 2), {"ends_free": (6, 3, 0, 5)}),
                                           ("affine", (0, 4, 6, 2), {"heuristic": (4, 5, 10, 1)}),
                                           ("affine", (0, 4, 6, 2), {"max_steps": 60}),
                                           ("affine2p", (0, 4, 6, 2, 24, 1), {}), ("edit", (0, 1, 1), {}),
                                           ("indel", (0, 1, 1), {})], ids=str)
def test_runs_are_those_of_the_operations(metric, pen, kw, long_pairs):
    rng = np.random.default_rng(41)
    P, T = [], []
    for i in range(300):
        t = rand(rng, int(rng.integers(10, 200)))
        P.append(mutate(rng, t, float(rng.uniform(0, 0.3)), 2) + b"ACGTAC")
        T.append(t.tobytes())
    if not kw.get("ends_free"):
        P += [b"", b"A", b"ACGT"]
        T += [b"ACGT", b"", b"ACGT"]
    for _ in range(long_pairs):
        t = rand(rng, 1300)
        P.append(mutate(rng, t, 0.05, 1))
        T.append(t.tobytes())
    al = wfa_amd.Aligner(metric=metric, penalties=pen, **kw)
    db = al.upload(datagen.PairSet.from_lists(P, T))
    for _ in range(2):
        db.run()
        ref, got = db.download(), db.download_runs()
        for i in range(len(P)):
            want = [(len(list(g)) << 4) | CODES[c] for c, g in itertools.groupby(ref.ops(i))]
            assert got.pair_runs(i).tolist() == want, (i, got.status[i])
