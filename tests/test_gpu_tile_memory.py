"""Device memory of the tile family (wfa_tile.hip, wfa_tile_run.cpp)."""
import ctypes
import sys

import numpy as np
import pytest

import oracle as O
import wfa_amd
from wfa_amd import datagen

pytestmark = pytest.mark.gpu

PEN = (0, 4, 6, 2, 24, 1)
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def free_device_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def mutate(rng, t, e):
    u = rng.random(len(t))
    out = t.copy()
    sub = u < e / 3
    out[sub] = BASES[rng.integers(0, 4, int(sub.sum()))]
    reps = np.ones(len(t), dtype=np.int64)
    reps[(u >= e / 3) & (u < 2 * e / 3)] = 2
    reps[(u >= 2 * e / 3) & (u < e)] = 0
    return np.repeat(out, reps).tobytes()


def pair(rng, n, e):
    t = BASES[rng.integers(0, 4, n)]
    return mutate(rng, t, e), t.tobytes()


def assert_same(got, ref, ids):
    bad = [i for x, i in enumerate(ids) if got.status[i] != ref.status[x] or got.score[i] != ref.score[x] or
           got.ops(i) != ref.ops(x)]
    assert not bad, (bad[:10], got.status[bad[0]], got.score[bad[0]])


def test_one_long_pair_among_many_reads(monkeypatch):
    """100,000 reads and one pair of 30 kbp: beside what the reads take, the
    pair takes its 62 rows of 61,000 diagonals (15 MB), a table of 5,000
    blocks and its sequences and CIGAR, not a table for every read (2 GB)."""
    monkeypatch.setenv("WFA_RECORD_ARENA_MB", "256")
    rng = np.random.default_rng(5)
    reads = datagen.generate(1, 91, 100000)
    P, T = reads.patterns(), reads.texts()
    long_p, long_t = pair(rng, 30000, 0.003)
    used = []
    for extra in (0, 1):
        ps = datagen.PairSet.from_lists(P + [long_p] * extra, T + [long_t] * extra)
        al = wfa_amd.Aligner(metric="affine2p", penalties=PEN)
        db = al.upload(ps)
        before = free_device_bytes()
        assert db.run() == 0
        used.append(before - free_device_bytes())
        say("%d pairs: %.0f MB" % (ps.n, used[-1] / 1e6))
        if extra:
            got = db.download()
            ids = list(range(0, reads.n, 997)) + [reads.n]
            ref = O.oracle_align(O.Conf("affine2p", PEN, "high"),
                                 O.Pairs([ps.pattern(i) for i in ids], [ps.text(i) for i in ids]))
            assert_same(got, ref, ids)
        db.free()
        al.close()
    assert used[1] - used[0] < 128e6


def check(metric, pen, ps, **kw):
    al = wfa_amd.Aligner(metric=metric, penalties=pen, **kw)
    db = al.upload(ps)
    ref = O.oracle_align(O.Conf(metric, pen, kw.get("memory", "high")), O.Pairs(ps.patterns(), ps.texts()))
    assert db.run() == 0
    assert_same(db.download(), ref, range(ps.n))
    return al, db, ref


@pytest.mark.parametrize("metric,pen", [("affine2p", PEN), ("affine", (0, 4, 6, 2))], ids=["affine2p", "affine"])
def test_little_memory_for_rows(monkeypatch, metric, pen):
    """1 MB of rows (affine2p takes 0.8 MB for a pair of 1,100 bp, affine 0.15
    MB): a pass for every pair or few of them, one of 9 kbp and one of 17 kbp
    that do not fit at all, and pairs that change over to single steps."""
    monkeypatch.setenv("WFA_ROWS_MB", "1")
    rng = np.random.default_rng(6)
    pairs = [pair(rng, n, 0.04) for n in (1100, 1290, 9000, 1150, 1030, 17000, 1200, 1250)]
    sk = datagen.skewed(8, 2, tlen=(300, 600), insert=(900, 1100))
    ps = datagen.PairSet.from_lists([p for p, _ in pairs] + sk.patterns(), [t for _, t in pairs] + sk.texts())
    al, db, ref = check(metric, pen, ps)
    assert db.stats().diagonal_steps == int(ref.dsteps.sum())
    say("%s: %d launches" % (metric, db.stats().forward_launches))
    assert db.stats().forward_launches >= 4
    assert db.run() == 0  # the statuses of the first run are there now
    assert_same(db.download(), ref, range(ps.n))


def test_little_memory_for_biwfa_rows(monkeypatch):
    """1 MB of rows: sub-problems of up to 1,700 symbols a side in tiles, a
    few at a time, larger ones without."""
    monkeypatch.setenv("WFA_ROWS_MB", "1")
    rng = np.random.default_rng(7)
    pairs = [pair(rng, n, 0.06) for n in (1100, 6000, 700, 2500, 1300, 900)]
    check("affine", (0, 4, 6, 2), datagen.PairSet.from_lists([p for p, _ in pairs], [t for _, t in pairs]),
          memory="ultralow")


def test_reap_gives_the_rows_back():
    """wavefront_aligner_reap frees what the tiles hold; the aligner goes on."""
    rng = np.random.default_rng(9)
    pairs = [pair(rng, 5000, 0.02) for _ in range(40)]
    ps = datagen.PairSet.from_lists([p for p, _ in pairs], [t for _, t in pairs])
    L = wfa_amd.lib()
    for memory in ("high", "ultralow"):
        metric, pen = ("affine2p", PEN) if memory == "high" else ("affine", (0, 4, 6, 2))
        al = wfa_amd.Aligner(metric=metric, penalties=pen, memory=memory)
        al.upload(ps).free()
        held = free_device_bytes()
        results = []
        for _ in range(2):
            db = al.upload(ps)
            assert db.run() == 0
            results.append(db.download())
            db.free()
            taken = held - free_device_bytes()
            L.wavefront_aligner_reap(al.wf)
            left = held - free_device_bytes()
            say("%s: %.0f MB held by a run, %.0f MB after" % (memory, taken / 1e6, left / 1e6))
            assert taken > 64e6 and left < 32e6
        want, got = results
        assert np.array_equal(got.score, want.score)
        assert all(got.ops(i) == want.ops(i) for i in range(ps.n))


def test_a_lane_keeps_to_its_memory():
    """128 requests of 12 kbp, scores only, in a lane of 256 MB: 6 MB of rows
    each, nearly all of them admitted at once under an error prior of 0.2%.
    The lane may take its 64 MB arena, 128 MB of rows, what the rows outgrew
    (kept while the server runs: about their size again), and its sequences."""
    rng = np.random.default_rng(10)
    pairs = [pair(rng, 12000, 0.002) for _ in range(128)]
    ref = O.oracle_align(O.Conf("affine2p", PEN, "high", True), O.Pairs([p for p, _ in pairs], [t for _, t in pairs]))
    before = free_device_bytes()
    srv = wfa_amd.Server(metric="affine2p", penalties=PEN, medium_lanes=1, lane_memory_bytes=256 << 20,
                         error_prior=0.002)
    wfa_amd.lib().wfa_server_destroy(srv.h)
    srv.attr.alignment_scope = 0
    srv.h = wfa_amd.lib().wfa_server_create(ctypes.byref(srv.attr), ctypes.byref(srv.config))
    ids = [srv.submit(p, t) for p, t in pairs]
    got, t0 = {}, srv.clock()
    while len(got) < len(ids):
        for r in srv.collect(max_results=256, timeout_ms=200):
            got[r.id] = r
        assert srv.clock() - t0 < 60, "requests did not finish"
    taken = before - free_device_bytes()
    srv.close()
    say("%.0f MB taken" % (taken / 1e6))
    for x, i in enumerate(ids):
        assert (got[i].status, got[i].score) == (ref.status[x], ref.score[x]), x
    assert taken < (64 + 2 * 128 + 64) * 1.05e6
