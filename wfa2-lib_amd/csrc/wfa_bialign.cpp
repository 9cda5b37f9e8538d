// BiWFA (memory mode ultralow) on the device, for whole batches.
//
// wavefront_bialign_alignment (wavefront_bialign.c:1145-1222) recurses depth
// first; every sub-problem depends only on its own bounds and components, so
// here the recursion runs breadth first: all sub-problems of one level, from
// every pair of the batch, go to one breakpoint-kernel launch; their halves
// form the next level.  Base cases (score_remaining <= 250, or the whole pair
// when max(n,m) <= 100, or an end reached at score <= 500) are collected and
// aligned in one pass of the unidirectional kernels, with their begin/end
// components; trivial halves (an empty side) are runs of D or I.  A final
// gather kernel concatenates the pieces of every pair in sequence order.
#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "wfa_internal.h"
#include "wfa_shapes.h"

namespace wfa_host {
namespace {

// wavefront_bialign.c:52-54
constexpr int kFallbackMinScore = 250;
constexpr int kFallbackMinLength = 100;
constexpr int kRecoveryMinScore = 500;

struct Node {
  wfa::BiProblem prob;
  int score_remaining;
  int level;
};

struct Leaf {
  int pb, tb;      // start of the piece in the pair's sequences
  char op;         // run operation (D or I) when base < 0
  int len;         // run length
  int base;        // index of the base-case job, or -1
};

struct BaseScore {
  int pb, tb, score;
};

struct PairState {
  int status = WF_STATUS_ALG_COMPLETED;
  int fail_pb = INT_MAX, fail_tb = INT_MAX;  // leftmost failing sub-problem (depth-first order)
  bool fail_base = false;  // ... and whether it is a base alignment, with its score
  int fail_score = INT32_MIN;
  int score = INT32_MIN;   // cigar->score
  std::vector<Leaf> leaves;
  std::vector<BaseScore> bases;  // completed base alignments
};

// The reference's recursion stops at the first failing sub-problem in
// depth-first order, which is the leftmost one.
void fail_pair(PairState& ps, int status, int pb, int tb, bool base = false, int score = INT32_MIN) {
  if (pb < ps.fail_pb || (pb == ps.fail_pb && tb < ps.fail_tb)) {
    ps.fail_pb = pb;
    ps.fail_tb = tb;
    ps.status = status;
    ps.fail_base = base;
    ps.fail_score = score;
  }
}

// cigar->score of a failed pair: every base alignment sets it
// (wavefront_bialign.c:181-182), so it is the failing base's own score, or
// that of the last base alignment run before the failing search, if any.
int failed_score(const PairState& ps) {
  if (ps.fail_base) return ps.fail_score;
  int best = INT32_MIN, bpb = INT_MIN, btb = INT_MIN;
  for (const BaseScore& b : ps.bases) {
    const bool before = b.pb < ps.fail_pb || (b.pb == ps.fail_pb && b.tb < ps.fail_tb);
    if (before && (b.pb > bpb || (b.pb == bpb && b.tb > btb))) {
      bpb = b.pb;
      btb = b.tb;
      best = b.score;
    }
  }
  return best;
}

bool ensure_reverse(Engine* e, wfa_device_batch_t* b) {
  if (b->have_reverse) return true;
  const int n = b->n;
  if (!b->rev_words.ensure(std::max<int64_t>(b->words_used, 1) * 8)) return false;
  std::vector<int64_t> pos(2 * (size_t)n);
  std::vector<int> len(2 * (size_t)n);
  for (int i = 0; i < n; ++i) {
    pos[i] = b->pat_pos[i];
    pos[n + i] = b->txt_pos[i];
    len[i] = b->plen[i];
    len[n + i] = b->tlen[i];
  }
  DevBuf& d_pos = e->bi.pos;
  DevBuf& d_len = e->bi.len;
  if (!d_pos.ensure(pos.size() * 8) || !d_len.ensure(len.size() * 4)) return false;
  hipStream_t st = e->stream;
  bool ok = hip_ok(hipMemcpyAsync(d_pos.p, pos.data(), pos.size() * 8, hipMemcpyHostToDevice, st), "reverse") &&
            hip_ok(hipMemcpyAsync(d_len.p, len.data(), len.size() * 4, hipMemcpyHostToDevice, st), "reverse") &&
            hip_ok(wfa::launch_reverse_pack(b->words.as<uint64_t>(), d_pos.as<int64_t>(), d_pos.as<int64_t>(),
                                            d_len.as<int>(), 2 * n, b->bits, b->rev_words.as<uint64_t>(), st),
                   "reverse pack") &&
            hip_ok(hipStreamSynchronize(st), "reverse pack");
  b->have_reverse = ok;
  return ok;
}

int bp_block(int size) { return size <= 512 ? 64 : (size <= 8192 ? 256 : 1024); }

// Bound of every wait of a paired search: 4 s of the 100 MHz device clock.
// WFA_PAIR_WAIT_TICKS sets another (tests force the one-workgroup fallback
// with a bound of a few ticks).
unsigned long long pair_wait_ticks() {
  const char* v = getenv("WFA_PAIR_WAIT_TICKS");
  return v ? strtoull(v, nullptr, 10) : 400000000ull;
}

// WFA_PAIR_SEARCH=0 turns paired-workgroup breakpoint searches off.
bool pair_searches_enabled() {
  const char* v = getenv("WFA_PAIR_SEARCH");
  return !v || v[0] != '0';
}

// LDS for the four sequences of a breakpoint problem (2-bit sequences of a
// 100 kbp pair take 100 KB of gfx950's 160 KB per CU).
constexpr size_t kBreakpointSeqLdsBytes = 120 * 1024;

// Sub-problems of at least this many symbols (both sequences) are advanced in
// tiles first.  Below, one workgroup steps through the whole search in less
// than the launches of its blocks take.  64 pairs of 20-60 kbp: from 4,096
// symbols 69.2 ms, from 2,048 67.0 ms, from 1,024 66.8 ms, from 512 66.4 ms
// (few sub-problems of a long pair are that small); one workgroup or team per
// search throughout, 482 ms.
constexpr int kBiTileMinSize = 1024;
// Rows of the sub-problems of one launch, and their number (the grid has two
// rows of workgroups for each).
constexpr size_t kBiTileStateBytes = size_t(8) << 30;
constexpr size_t kBiTileMaxProblems = 16384;

// Tables of the tiles' ranges for the begin components M, I1 and D1.
bool bi_table(Engine* e, int steps) {
  Engine::BiTiles& t = e->bi_tiles;
  if (t.steps >= steps) return true;
  steps = std::max({steps, 4096, 2 * t.steps});
  std::vector<int> hull((size_t)3 * steps * 2);
  std::vector<long long> dsteps((size_t)3 * (steps + 1), 0);
  t.lo.assign(steps, 0);
  t.hi.assign(steps, 0);
  const wfa::TileGeometry g = wfa::tile_geometry(1);
  for (int begin = 0; begin < 3; ++begin) {
    std::vector<wfa::StepRanges> rows((size_t)steps + 1);
    rows[0].c[begin].lo = rows[0].c[begin].hi = 0;
    int lo = 0, hi = 0;
    long long* ds = dsteps.data() + (size_t)begin * (steps + 1);
    for (int i = 0; i < steps; ++i) {
      auto row = [&](int back, int c) { return i + 1 - back >= 0 ? rows[i + 1 - back].c[c] : wfa::StepRange{}; };
      rows[i + 1] = wfa::next_ranges(3, g.dx, g.do1, g.de1, 0, 0, row);
      const wfa::StepRange m = rows[i + 1].c[wfa::kM];
      ds[i + 1] = ds[i] + wfa::step_diagonals(m, 3, g.dx, g.do1, g.de1, 0, 0, row);
      if (m.valid()) {
        lo = std::min(lo, m.lo);
        hi = std::max(hi, m.hi);
      }
      hull[2 * ((size_t)begin * steps + i)] = lo;
      hull[2 * ((size_t)begin * steps + i) + 1] = hi;
      t.lo[i] = std::min(t.lo[i], lo);
      t.hi[i] = std::max(t.hi[i], hi);
    }
  }
  t.steps = 0;
  hipStream_t st = e->stream;
  if (!t.d_hull.ensure(hull.size() * sizeof(int)) || !t.d_dsteps.ensure(dsteps.size() * sizeof(long long)) ||
      !hip_ok(hipMemcpyAsync(t.d_hull.p, hull.data(), hull.size() * sizeof(int), hipMemcpyHostToDevice, st), "bi table") ||
      !hip_ok(hipMemcpyAsync(t.d_dsteps.p, dsteps.data(), dsteps.size() * sizeof(long long), hipMemcpyHostToDevice, st),
              "bi table") ||
      !hip_ok(hipStreamSynchronize(st), "bi table"))
    return false;
  t.steps = steps;
  return true;
}

// Advances the sub-problems probs[0..n) (already in d_probs) in tiles until
// the block in which phase 1 ends, and sets a's resume fields; without memory
// for their rows (which grow up to max_bytes) the search runs from the start.
bool bi_fast_forward(Engine* e, const std::vector<wfa::BiProblem>& probs, size_t max_bytes, wfa::BiArgs& a) {
  Engine::BiTiles& t = e->bi_tiles;
  const int n = (int)probs.size(), T = wfa::bi_tile_steps(), U = wfa::bi_tile_useful();
  hipStream_t st = e->stream;
  // a side that never meets the other ends at its own end: no more steps
  // than that alignment can cost
  const wfa::TileGeometry g = wfa::tile_geometry(1);
  int max_steps = 0, lw = 0;
  int64_t ints = 0;
  std::vector<int64_t> off(n);
  for (int i = 0; i < n; ++i) {
    const int pl = probs[i].pe - probs[i].pb, tl = probs[i].te - probs[i].tb;
    const int64_t mn = std::min(pl, tl), mx = std::max(pl, tl);
    max_steps = (int)std::max<int64_t>(max_steps, mn * g.dx + 2 * g.do1 + (mx - mn) * g.de1);
    lw = std::max(lw, (int)mx / 32 + 4);
    off[i] = ints;
    ints += (int64_t)2 * wfa::kBiTileRows * wfa::tile_pitch(pl, tl);
  }
  const int max_blocks = max_steps / T + 2;  // (a search not done by then starts over: wfa_breakpoint_kernel)
  if (!bi_table(e, (max_blocks + 1) * T)) return false;
  if (!t.h_n.ensure(4096) || !t.d_state.ensure((size_t)ints * 4, std::max(max_bytes, (size_t)ints * 4)) || !t.d_off.ensure((size_t)n * 8) ||
      !t.d_marks.ensure((size_t)n * 5 * 4) || !t.d_act.ensure((size_t)2 * n * 4 + 64))
    return true;
  for (auto& ev : t.ev)
    if (!ev && !hip_ok(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate")) return false;
  volatile int* h_n = t.h_n.as<int>();
  int* n_act = t.d_act.as<int>();
  int* act[2] = {n_act + 16, n_act + 16 + n};
  wfa::BiTileArgs f{};
  f.n = n;
  f.probs = a.probs;
  f.words = a.words;
  f.rev_words = a.rev_words;
  f.fwd_ppos = a.fwd_ppos;
  f.fwd_tpos = a.fwd_tpos;
  f.rev_ppos = a.rev_ppos;
  f.rev_tpos = a.rev_tpos;
  f.plen_total = a.plen_total;
  f.tlen_total = a.tlen_total;
  f.state = t.d_state.as<int>();
  f.st_off = t.d_off.as<int64_t>();
  f.done = t.d_marks.as<int>();
  f.far = f.done + n;
  f.hull = t.d_hull.as<int2>();
  f.steps = t.steps;
  f.lmax_words = lw;
  if (!hip_ok(hipMemcpyAsync(t.d_off.p, off.data(), (size_t)n * 8, hipMemcpyHostToDevice, st), "bi tiles") ||
      !hip_ok(wfa::launch_tile_fill(f.state, ints, st), "bi tile fill") ||
      !hip_ok(wfa::launch_bi_tile_init(f, act[0], n_act, st), "bi tile init") ||
      !hip_ok(hipStreamSynchronize(st), "bi tiles"))  // (off is read by then)
    return false;
  int known = n, which = 0, chunk = 0;
  for (int blk = 0; blk < max_blocks && known > 0;) {
    const int to = std::min(max_blocks, blk + (chunk < 4 ? 4 : 16));
    for (; blk < to; ++blk) {
      f.act = act[which];
      f.n_act = n_act + which;
      f.blk = blk;
      const int lo = blk ? t.lo[(size_t)blk * T - 1] : 0, hi = blk ? t.hi[(size_t)blk * T - 1] : 0;
      if (!hip_ok(wfa::launch_bi_tile_block(f, known, (hi - lo + 2 * T + 8) / U + 1, st), "bi tile launch")) return false;
    }
    const int slot = chunk & 1;
    if (!hip_ok(wfa::launch_tile_compact(act[which], n_act + which, f.done, nullptr, blk, act[which ^ 1],
                                         n_act + (which ^ 1), nullptr, const_cast<int*>(h_n) + slot, st), "bi tile compact") ||
        !hip_ok(hipEventRecord(t.ev[slot], st), "bi tile event"))
      return false;
    which ^= 1;
    if (chunk > 0) {
      if (!hip_ok(hipEventSynchronize(t.ev[slot ^ 1]), "bi tiles")) return false;
      known = h_n[slot ^ 1];
    }
    ++chunk;
  }
  a.resume = f.done;
  a.resume_state = f.state;
  a.resume_off = f.st_off;
  a.resume_far = f.far;
  a.resume_dsteps = t.d_dsteps.as<long long>();
  a.resume_table = t.steps + 1;
  a.resume_block = T;
  return true;
}

// Runs the breakpoint search of `nodes` (grouped by size) and returns the outcomes.
bool run_breakpoints(wavefront_aligner_t* wf, Engine* e, wfa_device_batch_t* b, const std::vector<Node>& nodes,
                     std::vector<wfa::BiOutcome>& out, RunTotals* tot) {
  const wfa::Penalties pen = make_penalties(wf->penalties);
  const int ncomp = pen.ncomp;
  out.assign(nodes.size(), wfa::BiOutcome{});
  if (nodes.empty()) return true;
  // groups by workgroup size
  std::vector<int> groups[3];
  for (int i = 0; i < (int)nodes.size(); ++i) {
    const wfa::BiProblem& p = nodes[i].prob;
    const int size = (p.pe - p.pb) + (p.te - p.tb);
    const int bl = bp_block(size);
    groups[bl == 64 ? 0 : (bl == 256 ? 1 : 2)].push_back(i);
  }
  hipStream_t st = e->stream;
  const wfa::HeurArgs heur = heuristic_of(wf);
  const bool tiles_ok = wfa::tile_shape(pen) == 1 && b->bits == 2 && heur.cut() == 0 &&
                        (wf->system.max_alignment_steps <= 0 || wf->system.max_alignment_steps == INT_MAX);
  // large sub-problems in tiles: as many at once as their rows' memory allows
  std::vector<std::vector<int>> runs(groups, groups + 3);
  std::vector<int> run_block = {64, 256, 1024};
  size_t rows_bytes = kBiTileStateBytes;
  if (tiles_ok) {
    auto rows_of = [&](int i) {
      const wfa::BiProblem& p = nodes[i].prob;
      return (size_t)2 * wfa::kBiTileRows * wfa::tile_pitch(p.pe - p.pb, p.te - p.tb) * 4;
    };
    size_t want = 0;
    for (size_t i = 0; i < nodes.size(); ++i) want += rows_of((int)i);
    rows_bytes = rows_limit(e, want, kBiTileStateBytes, e->bi_tiles.d_state.cap);
    for (int gi = 0; gi < 3; ++gi) {
      int64_t bytes = INT64_MAX;
      std::vector<int> rest;
      for (int i : groups[gi]) {
        const wfa::BiProblem& p = nodes[i].prob;
        const int pl = p.pe - p.pb, tl = p.te - p.tb;
        const int64_t need = (int64_t)rows_of(i);
        if (pl + tl < kBiTileMinSize || 2 * (size_t)(std::max(pl, tl) / 32 + 4) * 8 > wfa::kTileSeqLdsBytes ||
            (e->rows_cap && (size_t)need > e->rows_cap)) {
          rest.push_back(i);
          continue;
        }
        if (bytes > (int64_t)rows_bytes - need || runs.back().size() >= kBiTileMaxProblems) {
          runs.emplace_back();
          run_block.push_back(run_block[gi]);
          bytes = 0;
        }
        runs.back().push_back(i);
        bytes += need;
      }
      runs[gi].swap(rest);
    }
  }
  for (size_t ri = 0; ri < runs.size(); ++ri) {
    const bool tile = ri >= 3;
    const std::vector<int>& ids = runs[ri];
    if (ids.empty()) continue;
    const int block = run_block[ri];
    // One launch over the sub-problems `sel` (indices into nodes); paired:
    // two workgroups per sub-problem.  Outcomes go to out[].
    auto launch = [&](const std::vector<int>& sel, bool paired) -> bool {
      std::vector<wfa::BiProblem> probs(sel.size());
      int wmax = 0;
      for (size_t j = 0; j < sel.size(); ++j) {
        probs[j] = nodes[sel[j]].prob;
        wmax = std::max(wmax, (probs[j].pe - probs[j].pb) + (probs[j].te - probs[j].tb));
      }
      const int wcap = wmax + 8;
      // The four sequences of the launch's longest problem in LDS when they fit.
      const int spw = 64 / b->bits;
      int lw = 0;
      for (const wfa::BiProblem& p : probs) lw = std::max(lw, std::max(p.pe - p.pb, p.te - p.tb) / spw + 3);
      if (wfa::breakpoint_lds_bytes(lw) > kBreakpointSeqLdsBytes) lw = 0;
      int grid = 0;
      wfa::Penalties lpen = pen;
      if (paired) {
        lpen.nslots = pen.nslots + 1;  // room for the speculative reverse step
        grid = 2 * (int)probs.size();
      } else {
        int per_cu = wfa::breakpoint_max_blocks_per_cu(ncomp, b->bits, block, heur.cut() != 0,
                                                       wfa::breakpoint_lds_bytes(lw));
        if (per_cu <= 0 && lw > 0) {
          lw = 0;
          per_cu = wfa::breakpoint_max_blocks_per_cu(ncomp, b->bits, block, heur.cut() != 0);
        }
        if (per_cu <= 0) per_cu = 1;
        grid = (int)std::min<int64_t>((int64_t)probs.size(), (int64_t)per_cu * e->num_cus);
      }
      const long long stride = 2LL * lpen.nslots * ncomp * wcap;
      const size_t ring_units = paired ? probs.size() : (size_t)grid;  // teams or workgroups
      DevBuf& d_probs = e->bi.probs;
      DevBuf& d_out = e->bi.out;
      const size_t hand_ints = wfa::breakpoint_pair_handover_ints(ncomp);
      if (!d_probs.ensure(probs.size() * sizeof(wfa::BiProblem)) ||
          !d_out.ensure(probs.size() * sizeof(wfa::BiOutcome)) ||
          !e->ring.ensure((size_t)stride * ring_units * sizeof(int)) ||
          (paired && (!e->bi.mail.ensure(probs.size() * 4 * sizeof(unsigned long long)) ||
                      !e->bi.hand.ensure(probs.size() * hand_ints * sizeof(int))))) {
        fprintf(stderr, "[WFA] cannot allocate BiWFA breakpoint buffers\n");
        return false;
      }
      wfa::Counters* c = counters_of(e);
      wfa::BiArgs a{};
      a.n = (int)probs.size();
      a.probs = d_probs.as<wfa::BiProblem>();
      a.words = b->words.as<uint64_t>();
      a.rev_words = b->rev_words.as<uint64_t>();
      a.fwd_ppos = b->d_patw.as<int64_t>();
      a.fwd_tpos = b->d_txtw.as<int64_t>();
      a.rev_ppos = b->d_patw.as<int64_t>();
      a.rev_tpos = b->d_txtw.as<int64_t>();
      a.plen_total = b->d_plen.as<int>();
      a.tlen_total = b->d_tlen.as<int>();
      a.out = d_out.as<wfa::BiOutcome>();
      a.ring = e->ring.as<int>();
      a.ring_stride = stride;
      a.wcap = wcap;
      a.queue = c->queue;
      a.dsteps_total = &c->dsteps;
      a.max_steps = wf->system.max_alignment_steps > 0 ? wf->system.max_alignment_steps : INT_MAX;
      a.lmax_words = lw;
      a.heur = heur;  // the breakpoint aligners inherit the heuristic (wavefront_bialigner.c:53)
      a.pen = lpen;
      a.mail = paired ? e->bi.mail.as<unsigned long long>() : nullptr;
      a.handover = paired ? e->bi.hand.as<int>() : nullptr;
      a.pair_wait_ticks = pair_wait_ticks();
      for (auto& ev : e->bi.ev)
        if (!ev && !hip_ok(hipEventCreate(&ev), "hipEventCreate")) return false;
      hipEvent_t e0 = e->bi.ev[0], e1 = e->bi.ev[1];
      std::vector<wfa::BiOutcome> res(probs.size());
      wfa::Counters host_c{};
      bool ok = hip_ok(hipMemcpyAsync(d_probs.p, probs.data(), probs.size() * sizeof(wfa::BiProblem),
                                      hipMemcpyHostToDevice, st), "bi upload") &&
                hip_ok(wfa::launch_reset_counters(c, 2, st), "reset") &&
                (!paired || hip_ok(hipMemsetAsync(a.mail, 0, probs.size() * 4 * sizeof(unsigned long long), st),
                                   "mailboxes"));
      (void)hipEventRecord(e0, st);
      if (ok && tile && !bi_fast_forward(e, probs, rows_bytes, a)) return false;
      ok = ok && hip_ok(paired ? wfa::launch_breakpoint_pair(a, ncomp, b->bits, block, st)
                               : wfa::launch_breakpoint(a, ncomp, b->bits, block, grid, st),
                        "breakpoint launch");
      (void)hipEventRecord(e1, st);
      ok = ok && hip_ok(hipMemcpyAsync(res.data(), d_out.p, res.size() * sizeof(wfa::BiOutcome),
                                       hipMemcpyDeviceToHost, st), "bi download") &&
           hip_ok(hipMemcpyAsync(&host_c, e->counters.p, wfa::kCounterTotals, hipMemcpyDeviceToHost, st), "counters") &&
           hip_ok(hipStreamSynchronize(st), "breakpoint");
      float ms = 0;
      (void)hipEventElapsedTime(&ms, e0, e1);
      if (!ok) return false;
      tot->forward_ms += ms;
      tot->launches += 1;
      tot->dsteps += host_c.dsteps;
      for (size_t j = 0; j < sel.size(); ++j) out[sel[j]] = res[j];
      return true;
    };
    // Paired workgroups when every team fits on the device at once beside
    // nothing else of this launch (large sub-problems, fewer than half the
    // workgroups the CUs hold); not with a heuristic cut-off, or where the
    // extra ring slot would pass the 64 slots of the slot metadata.
    bool paired = false;
    if (!tile && block == 1024 && heur.cut() == 0 && pen.nslots + 1 <= 64 && pair_searches_enabled()) {
      const int spw = 64 / b->bits;
      int lw = 0;
      for (int i : ids) {
        const wfa::BiProblem& p = nodes[i].prob;
        lw = std::max(lw, std::max(p.pe - p.pb, p.te - p.tb) / spw + 3);
      }
      if (wfa::breakpoint_lds_bytes(lw) > kBreakpointSeqLdsBytes) lw = 0;
      const int per_cu = wfa::breakpoint_pair_max_blocks_per_cu(ncomp, b->bits, block, wfa::breakpoint_lds_bytes(lw));
      paired = per_cu > 0 && 2 * (int64_t)ids.size() <= (int64_t)per_cu * e->num_cus;
    }
    if (!launch(ids, paired)) return false;
    if (paired) {
      // a team whose partner did not answer in time: search again on one workgroup
      std::vector<int> again;
      for (int i : ids)
        if (out[i].status == wfa::kBiPairAbort) again.push_back(i);
      if (!again.empty()) {
        fprintf(stderr, "[WFA] %zu paired breakpoint searches timed out; searching them again on one workgroup\n",
                again.size());
        if (!launch(again, false)) return false;
      }
    }
  }
  return true;
}

}  // namespace

int bialign_run(wavefront_aligner_t* wf, Engine* e, wfa_device_batch_t* b, RunTotals* tot) {
  const int n = b->n;
  const int records = b->records;
  if (!ensure_reverse(e, b)) return WF_STATUS_OOM;
  std::vector<PairState> ps(n);
  std::vector<Node> nodes, next;
  std::vector<wfa::BiOutcome> outc;
  std::vector<Node> base_nodes;
  for (int i = 0; i < n; ++i) {
    Node nd;
    nd.prob = wfa::BiProblem{i, 0, b->plen[i], 0, b->tlen[i], wfa::kM, wfa::kM, 0};
    nd.level = 0;
    // wavefront_bialign, wavefront_bialign.c:1276-1284
    nd.score_remaining = std::max(b->plen[i], b->tlen[i]) <= kFallbackMinLength ? 0 : INT_MAX;
    nodes.push_back(nd);
  }
  if (!records) {
    // wavefront_bialign_compute_score (:1226-1262): the top-level breakpoint only.
    if (!run_breakpoints(wf, e, b, nodes, outc, tot)) return WF_STATUS_OOM;
    for (int i = 0; i < n; ++i) {
      const wfa::BiOutcome& o = outc[i];
      if (o.status == wfa::kBiOk || o.status == wfa::kBiEndReached) {
        const int s = (o.status == wfa::kBiOk) ? o.score : (o.fwd_end_score >= 0 ? o.fwd_end_score : o.rev_end_score);
        ps[i].score = classic_score(wf->penalties, b->plen[i], b->tlen[i], s);
      } else {
        ps[i].status = (o.status == wfa::kDevMaxSteps) ? WF_STATUS_MAX_STEPS_REACHED : WF_STATUS_UNATTAINABLE;
      }
    }
  } else {
    while (!nodes.empty()) {
      next.clear();
      std::vector<Node> bp_nodes;
      for (const Node& nd : nodes) {
        PairState& st = ps[nd.prob.pair];
        // After a failure the reference's depth-first recursion has still
        // run everything to its left (whose base alignments set the score).
        if (st.status != WF_STATUS_ALG_COMPLETED &&
            !(nd.prob.pb < st.fail_pb || (nd.prob.pb == st.fail_pb && nd.prob.tb < st.fail_tb)))
          continue;
        const wfa::BiProblem& p = nd.prob;
        const int pl = p.pe - p.pb, tl = p.te - p.tb;
        if (tl == 0) {
          st.leaves.push_back(Leaf{p.pb, p.tb, 'D', pl, -1});
        } else if (pl == 0) {
          st.leaves.push_back(Leaf{p.pb, p.tb, 'I', tl, -1});
        } else if (nd.score_remaining <= kFallbackMinScore) {
          base_nodes.push_back(nd);
        } else {
          bp_nodes.push_back(nd);
        }
      }
      if (!run_breakpoints(wf, e, b, bp_nodes, outc, tot)) return WF_STATUS_OOM;
      for (size_t j = 0; j < bp_nodes.size(); ++j) {
        const Node& nd = bp_nodes[j];
        const wfa::BiProblem& p = nd.prob;
        const wfa::BiOutcome& o = outc[j];
        PairState& st = ps[p.pair];
        if (o.status == wfa::kBiOk) {
          const int bp_h = o.offset_forward;
          const int bp_v = o.offset_forward - o.k_forward;
          Node left, right;
          left.prob = wfa::BiProblem{p.pair, p.pb, p.pb + bp_v, p.tb, p.tb + bp_h, p.comp_begin, o.component, 0};
          left.score_remaining = o.score_forward;
          left.level = nd.level + 1;
          right.prob = wfa::BiProblem{p.pair, p.pb + bp_v, p.pe, p.tb + bp_h, p.te, o.component, p.comp_end, 0};
          right.score_remaining = o.score_reverse;
          right.level = nd.level + 1;
          next.push_back(left);
          next.push_back(right);
          if (nd.level == 0) st.score = classic_score(wf->penalties, p.pe - p.pb, p.te - p.tb, o.score);
        } else if (o.status == wfa::kBiEndReached) {
          // wavefront_bialign_find_breakpoint_exception (:1084-1111)
          const int reached = o.fwd_end_score >= 0 ? o.fwd_end_score : o.rev_end_score;
          if (reached <= kRecoveryMinScore) base_nodes.push_back(nd);
          else fail_pair(st, WF_STATUS_UNATTAINABLE, p.pb, p.tb);
        } else if (o.status == wfa::kDevMaxSteps) {
          fail_pair(st, WF_STATUS_MAX_STEPS_REACHED, p.pb, p.tb);
        } else if (o.status == wfa::kDevUnreachable) {
          // a side the cut-off left unreachable (wavefront_bialign.c:1084-1111, 1286-1294)
          fail_pair(st, WF_STATUS_UNATTAINABLE, p.pb, p.tb);
        } else {
          if (o.status != wfa::kDevMaxSteps)
            fprintf(stderr, "[WFA] BiWFA breakpoint search failed (status %d) for pair %d\n", o.status, p.pair);
          fail_pair(st, WF_STATUS_UNATTAINABLE, p.pb, p.tb);
        }
      }
      nodes.swap(next);
    }
    // Base cases: one pass of the unidirectional kernels over all of them.
    const int nb = (int)base_nodes.size();
    std::vector<int> bpl(nb), btl(nb), bstatus, bscore(nb), bbegin(nb);
    std::vector<int64_t> bpp(nb), btp(nb), boff(nb);
    std::vector<signed char> bcb(nb), bce(nb);
    int64_t bops = 0;
    for (int j = 0; j < nb; ++j) {
      const wfa::BiProblem& p = base_nodes[j].prob;
      bpl[j] = p.pe - p.pb;
      btl[j] = p.te - p.tb;
      bpp[j] = b->pat_pos[p.pair] + p.pb;
      btp[j] = b->txt_pos[p.pair] + p.tb;
      bcb[j] = (signed char)p.comp_begin;
      bce[j] = (signed char)p.comp_end;
      boff[j] = bops;
      bops += (int64_t)bpl[j] + btl[j];
    }
    Engine::BiBuffers& bb = e->bi;
    DevBuf &d_pl = bb.pl, &d_tl = bb.tl, &d_pp = bb.pp, &d_tp = bb.tp, &d_cb = bb.cb, &d_ce = bb.ce,
           &d_st = bb.st, &d_sc = bb.sc, &d_last = bb.last, &d_ds = bb.ds, &d_off = bb.off, &d_beg = bb.beg,
           &d_ops = bb.ops;
    hipStream_t st = e->stream;
    if (nb > 0) {
      const size_t m = (size_t)nb;
      bool ok = d_pl.ensure(m * 4) && d_tl.ensure(m * 4) && d_pp.ensure(m * 8) && d_tp.ensure(m * 8) &&
                d_cb.ensure(m) && d_ce.ensure(m) && d_st.ensure(m * 4) && d_sc.ensure(m * 4) && d_last.ensure(m * 4) &&
                d_ds.ensure(m * 8) && d_off.ensure(m * 8) && d_beg.ensure(m * 4) &&
                d_ops.ensure(std::max<int64_t>(bops, 1));
      if (!ok) return WF_STATUS_OOM;
      ok = hip_ok(hipMemcpyAsync(d_pl.p, bpl.data(), m * 4, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_tl.p, btl.data(), m * 4, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_pp.p, bpp.data(), m * 8, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_tp.p, btp.data(), m * 8, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_cb.p, bcb.data(), m, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_ce.p, bce.data(), m, hipMemcpyHostToDevice, st), "base upload") &&
           hip_ok(hipMemcpyAsync(d_off.p, boff.data(), m * 8, hipMemcpyHostToDevice, st), "base upload");
      if (!ok) return WF_STATUS_OOM;
      JobSet js;
      js.n = nb;
      js.bits = b->bits;
      js.h_plen = bpl.data();
      js.h_tlen = btl.data();
      js.words = b->words.as<uint64_t>();
      js.plen = d_pl.as<int>();
      js.tlen = d_tl.as<int>();
      js.ppos = d_pp.as<int64_t>();
      js.tpos = d_tp.as<int64_t>();
      js.cbeg = d_cb.as<signed char>();
      js.cend = d_ce.as<signed char>();
      js.status = d_st.as<int>();
      js.score = d_sc.as<int>();
      js.last = d_last.as<uint32_t>();
      js.dsteps = d_ds.as<long long>();
      js.ops = d_ops.as<char>();
      js.ops_off = d_off.as<int64_t>();
      js.ops_begin = d_beg.as<int>();
      std::vector<int> ids(nb);
      for (int j = 0; j < nb; ++j) ids[j] = j;
      std::sort(ids.begin(), ids.end(), [&](int x, int y) { return bpl[x] + btl[x] > bpl[y] + btl[y]; });
      std::vector<PlanGroup> plan = make_plan(js, ids, make_penalties(wf->penalties));
      RunTotals bt;
      const int rc = run_jobs(wf, e, js, plan, 1, &bt, bstatus);
      give_back_groups(e, plan);
      if (rc != WF_STATUS_OK) return rc;
      tot->forward_ms += bt.forward_ms;
      tot->backtrace_ms += bt.backtrace_ms;
      tot->launches += bt.launches;
      tot->dsteps += bt.dsteps;
      bstatus.resize(m);
      ok = hip_ok(hipMemcpyAsync(bstatus.data(), d_st.p, m * 4, hipMemcpyDeviceToHost, st), "base download") &&
           hip_ok(hipMemcpyAsync(bscore.data(), d_sc.p, m * 4, hipMemcpyDeviceToHost, st), "base download") &&
           hip_ok(hipMemcpyAsync(bbegin.data(), d_beg.p, m * 4, hipMemcpyDeviceToHost, st), "base download") &&
           hip_ok(hipStreamSynchronize(st), "base download");
      if (!ok) return WF_STATUS_OOM;
      for (int j = 0; j < nb; ++j) {
        const Node& nd = base_nodes[j];
        const wfa::BiProblem& p = nd.prob;
        PairState& s = ps[p.pair];
        if (bstatus[j] != WF_STATUS_ALG_COMPLETED) {
          // wavefront_bialign_base (:159-190): anything but completed is
          // unattainable; the base's own score stays (the step limit's)
          fail_pair(s, WF_STATUS_UNATTAINABLE, p.pb, p.tb, true,
                    bstatus[j] == WF_STATUS_MAX_STEPS_REACHED ? -wf->system.max_alignment_steps : INT32_MIN);
          continue;
        }
        s.leaves.push_back(Leaf{p.pb, p.tb, 0, bpl[j] + btl[j] - bbegin[j], j});
        s.bases.push_back(BaseScore{p.pb, p.tb, classic_score(wf->penalties, bpl[j], btl[j], bscore[j])});
        // the base call sets cigar->score; at level 0 nothing overrides it
        if (nd.level == 0) s.score = classic_score(wf->penalties, bpl[j], btl[j], bscore[j]);
      }
    }
    // Assemble every pair right-aligned in its slot of the batch's operations:
    // all its pieces, or for a failed pair the ones the reference's recursion
    // appended before the failure (the cigar it leaves, wavefront_bialign.c:
    // 159-190, 1145-1222).
    std::vector<wfa::OpsPiece> pieces;
    std::vector<int> begin(n, 0);
    for (int i = 0; i < n; ++i) {
      PairState& s = ps[i];
      const int cap = b->plen[i] + b->tlen[i];
      if (s.status != WF_STATUS_ALG_COMPLETED) {
        std::vector<Leaf> kept;
        for (const Leaf& l : s.leaves)
          if (l.pb < s.fail_pb || (l.pb == s.fail_pb && l.tb < s.fail_tb)) kept.push_back(l);
        s.leaves.swap(kept);
      }
      std::sort(s.leaves.begin(), s.leaves.end(),
                [](const Leaf& x, const Leaf& y) { return x.pb != y.pb ? x.pb < y.pb : x.tb < y.tb; });
      int64_t total = 0;
      for (const Leaf& l : s.leaves) total += l.len;
      if (total > cap) {
        fprintf(stderr, "[WFA] internal error: BiWFA CIGAR longer than its slot for pair %d\n", i);
        s.status = WF_STATUS_UNATTAINABLE;
        begin[i] = cap;
        continue;
      }
      begin[i] = (int)(cap - total);
      int64_t dst = b->ops_off[i] + begin[i];
      for (const Leaf& l : s.leaves) {
        if (l.len == 0) continue;
        wfa::OpsPiece pc{};
        pc.dst = dst;
        pc.len = l.len;
        if (l.base >= 0) {
          pc.src = boff[l.base] + bbegin[l.base];
          pc.op = 0;
        } else {
          pc.src = -1;
          pc.op = l.op;
        }
        pieces.push_back(pc);
        dst += l.len;
      }
    }
    if (!pieces.empty()) {
      DevBuf& d_pieces = e->bi.pieces;
      if (!d_pieces.ensure(pieces.size() * sizeof(wfa::OpsPiece))) return WF_STATUS_OOM;
      bool ok = hip_ok(hipMemcpyAsync(d_pieces.p, pieces.data(), pieces.size() * sizeof(wfa::OpsPiece),
                                      hipMemcpyHostToDevice, st), "pieces") &&
                hip_ok(wfa::launch_gather_ops(d_pieces.as<wfa::OpsPiece>(), (int)pieces.size(),
                                              d_ops.p ? d_ops.as<char>() : nullptr, b->d_ops.as<char>(), st), "gather") &&
                hip_ok(hipStreamSynchronize(st), "gather");
      if (!ok) return WF_STATUS_OOM;
    }
    if (!hip_ok(hipMemcpyAsync(b->d_ops_begin.p, begin.data(), (size_t)n * 4, hipMemcpyHostToDevice, e->stream),
                "results") ||
        !hip_ok(hipStreamSynchronize(e->stream), "results"))
      return WF_STATUS_OOM;
  }
  // Per-pair results into the batch (status on the device, scores on the host).
  std::vector<int> status(n);
  b->bi_score.assign(n, INT32_MIN);
  for (int i = 0; i < n; ++i) {
    status[i] = ps[i].status;
    b->bi_score[i] = (records && status[i] != WF_STATUS_ALG_COMPLETED) ? failed_score(ps[i]) : ps[i].score;
    if (status[i] != WF_STATUS_ALG_COMPLETED) tot->fail++;
  }
  if (n > 0 && (!hip_ok(hipMemcpyAsync(b->d_status.p, status.data(), (size_t)n * 4, hipMemcpyHostToDevice, e->stream),
                        "results") ||
                 !hip_ok(hipStreamSynchronize(e->stream), "results")))
    return WF_STATUS_OOM;
  return WF_STATUS_OK;
}

}  // namespace wfa_host
