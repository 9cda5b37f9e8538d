"""Workloads of the aligner as user programs meet them, for timing and for
comparing outputs.

Every case aligns synthetic pairs through the package's public entry points:
`Aligner.align` (one pair per call), `Aligner.align_batch` (host buffers in,
host results out) or a resident batch (`Aligner.upload` once, then
`DeviceBatch.run` and a download of the results).  The pairs are drawn from
the seed alone: a uniform ACGT text and a pattern that is the text with
substitutions, insertions and deletions in equal parts, as a read and its
place in a reference differ.  Outputs are whole: status, score, and for
alignments the whole CIGAR (operation bytes or run-length form).
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(os.getcwd(), "wfa2-lib_amd")
sys.path.insert(0, PACKAGE if os.path.isdir(PACKAGE) else os.path.join(ROOT, "wfa2-lib_amd"))

import wfa_amd  # noqa: E402
from wfa_amd.datagen import PairSet  # noqa: E402

PENALTIES = {"affine": (0, 4, 6, 2), "affine2p": (0, 4, 6, 2, 24, 1), "linear": (0, 4, 2), "edit": (0, 1, 1),
             "indel": (0, 1, 1)}
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def case(name, entry, pairs, min_len, max_len, min_err, max_err, metric="affine", memory="high", score_only=False,
         adaptive=False, free=0, indel=1.0, n_rate=0.0):
    """entry: "align", "call" or "resident"; lengths of the texts and error
    events per base are uniform in their ranges (lengths in their logarithm
    over more than a factor of ten); indel: mean length of an insertion or
    deletion; free: the text carries up to that many bases more on each side,
    free to be left out; n_rate: share of N among the pattern's bases."""
    d = dict(entry=entry, pairs=pairs, min_len=min_len, max_len=max_len, min_err=min_err, max_err=max_err,
             metric=metric, memory=memory, score_only=score_only, adaptive=adaptive, free=free, indel=indel,
             n_rate=n_rate)
    return dict(name=name, **d) if name else d


def listed():
    return [
        # A caller of the C API aligns one read per wavefront_align call: latency.
        case("one-read", "align", 1, 150, 150, 0.05, 0.05),
        # One call on host buffers with a thousand 1 kbp pairs at 5% errors, each CIGAR read as bytes.
        case("call-1kbp", "call", 1000, 1000, 1000, 0.05, 0.05),
        # Read mapping: many short reads, scores and run-length CIGARs.
        case("reads", "resident", 150000, 100, 300, 0.0, 0.10),
        # Filtering or clustering reads by score alone.
        case("reads-score", "resident", 150000, 100, 300, 0.0, 0.10, score_only=True),
        # The library's default attributes: the wf-adaptive heuristic.
        case("reads-adaptive", "resident", 100000, 100, 300, 0.0, 0.10, adaptive=True),
        # A read placed inside a longer window of the reference: free text ends.
        case("reads-endsfree", "resident", 100000, 100, 300, 0.0, 0.10, free=30),
        # Edit distance of reads (barcodes, deduplication).
        case("reads-edit", "resident", 150000, 100, 300, 0.0, 0.10, metric="edit"),
        # Reads under dual-cost gaps, as long-read mappers score them.
        case("reads-2p", "resident", 50000, 100, 300, 0.0, 0.10, metric="affine2p"),
        # Reads with unknown bases, as sequencers write them: one byte per base.
        case("reads-n", "resident", 50001, 100, 301, 0.0, 0.10, n_rate=0.005),
        # Assembled fragments of 0.5-1 kbp.
        case("reads-1kbp", "resident", 20000, 500, 1000, 0.02, 0.08),
        # Long reads under dual-cost gaps.
        case("long-reads", "resident", 256, 1000, 20000, 0.01, 0.15, metric="affine2p", indel=3.0),
        # Very long reads in the linear-memory mode (BiWFA).
        case("very-long", "resident", 64, 20000, 60000, 0.05, 0.15, memory="ultralow", indel=2.0),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["align", "call", "resident", "resident", "resident", "resident", "resident", "long",
                       "ultralow"])
    if kind == "align":
        n = spread(60, 1000)
        e = rng.uniform(0.0, 0.10)
        return case(None, "align", 1, n, n, e, e, metric=rng.choice(["affine", "affine", "edit", "affine2p"]))
    if kind == "call":
        n = spread(100, 1000)
        return case(None, "call", spread(200, 2000), max(60, n // 2), n, 0.0, rng.uniform(0.02, 0.10),
                    metric=rng.choice(["affine", "affine", "linear"]))
    if kind == "long":
        hi = spread(3000, 20000)
        return case(None, "resident", spread(32, 256), max(1000, hi // rng.choice([2, 5, 20])), hi, 0.01,
                    rng.uniform(0.05, 0.15), metric=rng.choice(["affine2p", "affine2p", "affine"]), indel=3.0)
    if kind == "ultralow":
        hi = spread(12000, 60000)
        return case(None, "resident", spread(8, 64), hi // rng.choice([1, 2, 3]), hi, 0.05,
                    rng.uniform(0.06, 0.15), memory="ultralow", indel=2.0)
    hi = spread(100, 1000)
    lo = max(60, hi // rng.choice([1, 2, 3]))
    most = min(150000, 30000000 // hi)
    metric, option = rng.choice([("affine", None), ("affine", None), ("affine", "score"), ("affine", "adaptive"),
                                 ("affine", "free"), ("affine", "n"), ("edit", None), ("edit", "score"),
                                 ("indel", None), ("linear", None), ("affine2p", None), ("affine2p", "score")])
    return case(None, "resident", spread(2000, most), lo, hi, 0.0, rng.uniform(0.02, 0.10), metric=metric,
                score_only=option == "score", adaptive=option == "adaptive",
                free=rng.randrange(10, 31) if option == "free" else 0, n_rate=0.005 if option == "n" else 0.0)


def make_pairs(c, seed):
    """The pairs of a case, whole batch at once."""
    rng = np.random.default_rng(seed)
    n = c["pairs"]
    if c["max_len"] > 10 * c["min_len"]:
        length = np.exp(rng.uniform(math.log(c["min_len"]), math.log(c["max_len"]), n)).astype(np.int64)
    else:
        length = rng.integers(c["min_len"], c["max_len"] + 1, n)
    rate = rng.uniform(c["min_err"], c["max_err"], n)
    before = rng.integers(0, c["free"] + 1, n)
    after = rng.integers(0, c["free"] + 1, n)
    tlen = length + before + after
    t_off = np.cumsum(tlen) - tlen
    text = rng.integers(0, 4, int(tlen.sum()), dtype=np.uint8)
    # the stretch of each text that the pattern copies
    first = np.cumsum(length) - length
    if c["free"]:
        core = np.zeros(len(text) + 1, dtype=np.int8)
        np.add.at(core, t_off + before, 1)
        np.add.at(core, t_off + before + length, -1)
        pattern = text[np.cumsum(core[:-1], dtype=np.int8) > 0]
    else:
        pattern = text.copy()
    # events: substitutions, deletions and insertions at uniform places
    count = np.ceil(rate * length - 1e-9).astype(np.int64)
    pair = np.repeat(np.arange(n), count)
    place = first[pair] + (rng.random(len(pair)) * length[pair]).astype(np.int64)
    kind = rng.integers(0, 3, len(pair))
    size = rng.geometric(1.0 / c["indel"], len(pair))
    sub = place[kind == 0]
    pattern[sub] = (pattern[sub] + rng.integers(1, 4, len(sub), dtype=np.uint8)) & 3
    dele = kind == 1
    gone = np.zeros(len(pattern) + 1, dtype=np.int32)
    np.add.at(gone, place[dele], 1)
    np.add.at(gone, np.minimum(place[dele] + size[dele], (first + length)[pair[dele]]), -1)
    keep = np.cumsum(gone[:-1]) == 0
    kept = np.concatenate([[0], np.cumsum(keep)])
    ins = kind == 2
    at = np.repeat(kept[place[ins]], size[ins])
    plen = kept[first + length] - kept[first] + np.bincount(pair[ins], weights=size[ins], minlength=n).astype(np.int64)
    pattern = np.insert(pattern[keep], at, rng.integers(0, 4, len(at), dtype=np.uint8))
    letters = BASES[pattern]
    if c["n_rate"]:
        letters[rng.integers(0, len(letters), int(c["n_rate"] * len(letters)) + 1)] = ord("N")
    p_off = np.cumsum(plen) - plen
    return PairSet(letters.tobytes() + BASES[text].tobytes(), p_off, plen, t_off + len(letters), tlen)


def aligner(c):
    return wfa_amd.Aligner(
        metric=c["metric"], penalties=PENALTIES[c["metric"]], memory=c["memory"], score_only=c["score_only"],
        heuristic=(4, 10, 50, 1) if c["adaptive"] else None,
        ends_free=(0, 0, c["free"], c["free"]) if c["free"] else None)


def prepare(c, seed):
    """The pairs and the aligner a program holds, with a buffer for the CIGARs
    of every pair (zeros where none is written); a resident batch is uploaded,
    and its buffer for run-length CIGARs is pinned."""
    ps = make_pairs(c, seed)
    state = {"case": c, "aligner": aligner(c)}
    events = math.ceil(c["max_err"] * c["max_len"])
    if c["entry"] == "resident":
        state["batch"] = state["aligner"].upload(ps)
        if not c["score_only"]:
            runs = c["pairs"] * (5 * events // 2 + 16)
            state["cigars"] = torch.zeros(runs, dtype=torch.int32, pin_memory=True).numpy()
        return state
    if c["entry"] == "align":
        state["pair"] = (ps.pattern(0), ps.text(0))
    else:
        state["pairs"] = ps
    state["cigars"] = np.zeros(c["pairs"] * int(c["max_len"] + 3 * c["indel"] * events + 64), dtype=np.uint8)
    return state


def run(state):
    c, al, out = state["case"], state["aligner"], state.get("cigars")
    if c["entry"] == "align":
        status, score, ops = al.align(*state["pair"])
        out[:len(ops)] = np.frombuffer(ops, dtype=np.uint8)
        return {"status": status, "score": score, "ops": out, "length": len(ops)}
    if c["entry"] == "call":
        r = al.align_batch(state["pairs"])
        ops = np.frombuffer(b"".join([r.ops(i) for i in range(r.n)]), dtype=np.uint8)
        out[:len(ops)] = ops
        return {"status": r.status, "score": r.score, "ops": out, "length": r.cigar_length}
    batch = state["batch"]
    batch.run()
    if c["score_only"]:
        r = batch.download(cigars=False)
        return {"status": r.status, "score": r.score}
    r = batch.download_runs(out.view(np.uint32))
    return {"status": r.status, "score": r.score, "runs": out, "first": r.cigar_offset, "length": r.cigar_length}


def exact(c, seed):
    """Statuses, scores and CIGARs are whole numbers: there is nothing to
    compute in 64 bits that is closer."""
    return None


def work(c):
    """Bytes: the sequences (2 bits per base, 8 with other letters) read once,
    status, score and CIGAR (4 bytes a run, a byte an operation) written once.
    Operations: the cells of the wavefronts, which the scores bound: a pair of
    score s under gap-affine costs has about s / 2 wavefronts, s / 2 wide on
    average (edit and indel: s wavefronts, s wide), 20 integer operations a
    cell (30 with dual-cost gaps, 8 with one component)."""
    n = c["pairs"]
    length = 0.5 * (c["min_len"] + c["max_len"])
    square = (c["min_len"] ** 2 + c["min_len"] * c["max_len"] + c["max_len"] ** 2) / 3.0
    if c["max_len"] > 10 * c["min_len"]:
        span = math.log(c["max_len"] / c["min_len"])
        length = (c["max_len"] - c["min_len"]) / span
        square = (c["max_len"] ** 2 - c["min_len"] ** 2) / (2.0 * span)
    rate = 0.5 * (c["min_err"] + c["max_err"])
    rate2 = (c["min_err"] ** 2 + c["min_err"] * c["max_err"] + c["max_err"] ** 2) / 3.0
    cost = {"affine": 6.0 + c["indel"], "affine2p": 6.0 + c["indel"], "linear": 2.5 * c["indel"]}.get(c["metric"], c["indel"])
    ops = {"affine": 20, "affine2p": 30}.get(c["metric"], 8)
    score2 = square * rate2 * cost * cost
    cells = {"affine": 0.25, "linear": 0.25, "affine2p": 0.5}.get(c["metric"], 1.0) * score2 + 1
    sequence = 2 * length * (1.0 if c["n_rate"] else 0.25)
    events = length * rate
    cigar = 0 if c["score_only"] else (8 * events + 4 if c["entry"] == "resident" else 2 * length)
    return {"bytes": n * (sequence + 8 + cigar), "flops": n * cells * ops}
