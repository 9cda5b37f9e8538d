"""One resident batch run again after its aligner's attributes changed: each
run against the oracle under the attributes of that run (status, score, every
CIGAR operation).  The batch keeps its launch plan from run to run; what the
plan chose kernels by must not outlive the choice."""
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen

pytestmark = pytest.mark.gpu

PEN = (0, 4, 6, 2)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def pairs(seed):
    a, b = datagen.generate(1, seed, 400), datagen.generate(0, seed + 1, 20)
    s = datagen.semiglobal(1, seed + 2, 100)
    return datagen.PairSet.from_lists(a.patterns() + b.patterns() + s.patterns(),
                                      a.texts() + b.texts() + s.texts())


def check(al, db, ps, label, metric="affine", pen=PEN, **kw):
    say(label)
    db.run()
    got = db.download()
    ref = O.oracle_align(O.Conf(metric, pen, "high", **kw), O.Pairs(ps.patterns(), ps.texts()))
    stale = np.asarray(ref.stale[:ps.n], dtype=bool)
    assert [i for i in range(ps.n) if got.status[i] == wfa_amd.WF_STATUS_UNSUPPORTED] == list(np.flatnonzero(stale)), label
    bad = [i for i in range(ps.n) if not stale[i] and
           (got.status[i] != ref.status[i] or got.score[i] != ref.score[i] or got.ops(i) != ref.ops(i))]
    assert not bad, "%s: %d pairs differ (first %d: status %d/%d score %d/%d)" % (
        label, len(bad), bad[0], got.status[bad[0]], ref.status[bad[0]], got.score[bad[0]], ref.score[bad[0]])


def test_heuristics_changed_between_runs():
    """Strategies that share a kernel instance elsewhere: wf-adaptive (which
    short pairs run on the wave family), a band beside it, a band alone,
    wfmash, wf-adaptive again, none."""
    ps = pairs(611)
    al = wfa_amd.Aligner(metric="affine", penalties=PEN)
    L = wfa_amd.lib()
    db = al.upload(ps)
    L.wavefront_aligner_set_heuristic_wfadaptive(al.wf, 10, 50, 1)
    check(al, db, ps, "wf-adaptive", heuristic=(4, 10, 50, 1))
    L.wavefront_aligner_set_heuristic_banded_static(al.wf, -6, 6)
    check(al, db, ps, "wf-adaptive and band", heuristic=(5, 10, 50, 1, -6, 6))
    L.wavefront_aligner_set_heuristic_none(al.wf)
    L.wavefront_aligner_set_heuristic_banded_static(al.wf, -8, 8)
    check(al, db, ps, "band", heuristic=(1, 10, 50, 1, -8, 8))
    L.wavefront_aligner_set_heuristic_none(al.wf)
    L.wavefront_aligner_set_heuristic_wfmash(al.wf, 10, 30, 1)
    check(al, db, ps, "wfmash", heuristic=(0x40, 10, 30, 1))
    L.wavefront_aligner_set_heuristic_none(al.wf)
    L.wavefront_aligner_set_heuristic_wfadaptive(al.wf, 10, 30, 2)
    check(al, db, ps, "wf-adaptive, other limits", heuristic=(4, 10, 30, 2))
    L.wavefront_aligner_set_heuristic_none(al.wf)
    check(al, db, ps, "none")


@pytest.mark.parametrize("metric,pen", [("affine", PEN), ("affine2p", (0, 4, 6, 2, 24, 1)), ("linear", (0, 4, 2))],
                         ids=["affine", "affine2p", "linear"])
def test_free_ends_changed_between_runs(metric, pen):
    """Free ends whose score-0 wavefront fits a wave at 1, 4 and 8 diagonals
    per lane and not at all (a pair starts on 4 at most), grown and shrunk."""
    rng = np.random.default_rng(612)
    base = np.frombuffer(b"ACGT", dtype=np.uint8)
    P, T = [], []
    for i in range(48):
        t = base[rng.integers(0, 4, int(rng.integers(640, 900)))]
        at = int(rng.integers(0, len(t) - 300)) if i % 3 else 250
        p = t[at:at + int(rng.integers(200, 300))].copy()
        p[rng.integers(0, len(p), 8)] = base[rng.integers(0, 4, 8)]
        P.append(base[rng.integers(0, 4, 180 if i % 2 else 1)].tobytes() + p.tobytes())
        T.append(t.tobytes())
    ps = datagen.PairSet.from_lists(P, T)
    al = wfa_amd.Aligner(metric=metric, penalties=pen)
    L = wfa_amd.lib()
    db = al.upload(ps)
    for free in ((0, 0, 30, 30), (0, 0, 300, 100), (0, 0, 600, 200), (100, 0, 140, 20), (150, 0, 150, 0), (0, 10, 30, 0)):
        L.wavefront_aligner_set_alignment_free_ends(al.wf, *free)
        check(al, db, ps, "%s %s" % (metric, free), metric, pen, ends_free=free)
    L.wavefront_aligner_set_alignment_end_to_end(al.wf)
    check(al, db, ps, "%s end to end" % metric, metric, pen)
