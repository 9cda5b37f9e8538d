// Host side of the tile kernels (wfa_tile.hip): the table of wavefront
// ranges, and the loop that advances a set of long pairs block by block.
#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>

#include "wfa_internal.h"
#include "wfa_shapes.h"

namespace wfa_host {
namespace {

// Buffers of the jobs that run at once (wfa::TileJob), at most.
constexpr size_t kTileStateBytes = size_t(24) << 30;
constexpr int kTileMaxJobs = 32768;  // grid y
// Records a long pair is planned with: 1-20 kbp pairs of 1-15% error write
// 0.25 L^2 bytes on average and up to 0.7 L^2.
constexpr double kTileRecordShareOfL2 = 0.5;
// Blocks between two looks at the number of jobs left: 1, 2, 4 at a time up to
// some 32, then 16.
constexpr int kTileChunk = 16;

bool put(DevBuf& d, const void* from, size_t bytes, hipStream_t st) {
  return d.ensure(bytes) && hip_ok(hipMemcpyAsync(d.p, from, bytes, hipMemcpyHostToDevice, st), "range table") &&
         hip_ok(hipStreamSynchronize(st), "range table");
}

}  // namespace

// The table of at least `steps` steps for a tile shape: per step the range of
// M (lo > hi: none), the hull of the ranges so far, and the diagonal-steps up
// to it.
bool tile_table(Engine* e, int shape, int steps) {
  Engine::TileState& t = e->tile;
  if (t.shape == shape && (int)t.lo.size() >= steps) return true;
  steps = std::max(steps, 4096);
  if (t.shape == shape) steps = std::max(steps, 2 * (int)t.lo.size());
  t.shape = 0;
  const wfa::TileGeometry g = wfa::tile_geometry(shape);
  std::vector<wfa::StepRanges> rows((size_t)steps + 1);
  rows[0].c[wfa::kM].lo = rows[0].c[wfa::kM].hi = 0;
  std::vector<int> m_range(2 * (size_t)steps);
  std::vector<long long> dsteps((size_t)steps + 1, 0);
  t.lo.assign(steps, 0);
  t.hi.assign(steps, 0);
  int lo = 0, hi = 0;
  for (int i = 0; i < steps; ++i) {
    rows[i + 1] = wfa::next_ranges(g.do2 ? 5 : 3, g.dx, g.do1, g.de1, g.do2, g.de2, [&](int back, int c) {
      return i + 1 - back >= 0 ? rows[i + 1 - back].c[c] : wfa::StepRange{};
    });
    const wfa::StepRange m = rows[i + 1].c[wfa::kM];
    dsteps[i + 1] = dsteps[i] + (m.valid() ? m.hi - m.lo + 1 : 0);
    if (m.valid()) {
      lo = std::min(lo, m.lo);
      hi = std::max(hi, m.hi);
    }
    t.lo[i] = lo;
    t.hi[i] = hi;
    m_range[2 * (size_t)i] = m.lo;
    m_range[2 * (size_t)i + 1] = m.hi;
  }
  hipStream_t st = e->stream;
  if (!put(t.d_range, m_range.data(), m_range.size() * sizeof(int), st) ||
      !put(t.d_dsteps, dsteps.data(), dsteps.size() * sizeof(long long), st))
    return false;
  t.shape = shape;
  return true;
}

size_t rows_limit(const Engine* e, size_t want, size_t most, size_t held) {
  if (e->rows_cap) most = std::min(most, e->rows_cap);
  if (std::min(want, most) <= held) return most;
  // (two such buffers, and room for other aligners)
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return most;
  return std::min(most, std::max(held, (held + free_b) / 4));
}

// Whether a job of these lengths can run in tiles: its sequences in LDS.
bool tile_fits(int plen, int tlen) {
  const int lw = std::max(plen, tlen) / 32 + 3;
  return 2 * (size_t)lw * sizeof(uint64_t) <= wfa::kTileSeqLdsBytes;
}

// The jobs whose ends moved past their end tiles, one step per launch from
// the start of the block that found it, all of them side by side.  `unit`:
// record units taken so far.  Jobs left when the records run out stay
// unfinished (they are re-run with the records free again), and so do jobs
// whose rows do not fit (they go to the HBM-ring family).  Jobs are slots of
// the pass.
int run_steps(Engine* e, const JobSet& js, int shape, const wfa::TileGeometry& g, const wfa::TileArgs& a,
              const std::vector<wfa::TileSlot>& slots, int n_pass, const std::vector<wfa::TileBlockInfo>& info, int records,
              uint64_t rec_units, uint64_t* unit) {
  Engine::TileState& t = e->tile;
  hipStream_t st = e->stream;
  const int T = g.steps;
  std::vector<int> marks(2 * (size_t)n_pass);
  if (!hip_ok(hipMemcpyAsync(marks.data(), a.done, marks.size() * 4, hipMemcpyDeviceToHost, st), "tile marks") ||
      !hip_ok(hipStreamSynchronize(st), "tile marks"))
    return WF_STATUS_OOM;
  const int* done = marks.data();
  const int* irr = done + n_pass;
  std::vector<int> jobs;
  for (int x = 0; x < n_pass; ++x)
    if (irr[x] != INT_MAX && irr[x] < done[x]) jobs.push_back(x);
  const bool ok = jobs.empty() || (t.d_ends.ensure((size_t)n_pass * 4 * wfa::kTileStepEnds * 4) &&
                                   t.d_flags.ensure((size_t)n_pass * wfa::kTileStepFlags * 4) &&
                                   t.d_dsum.ensure((size_t)n_pass * 8) && t.d_step0.ensure((size_t)n_pass * 4) &&
                                   t.d_step_off.ensure((size_t)n_pass * 8));
  if (!ok) return WF_STATUS_OK;
  auto rows_of = [&](int x) {
    return (size_t)wfa::tile_pitch(js.h_plen[slots[x].id], js.h_tlen[slots[x].id]) * g.step_rows * 4;
  };
  size_t want = 0;
  for (int x : jobs) want += rows_of(x);
  size_t limit = rows_limit(e, want, kTileStateBytes, t.d_step_state.cap);
  // as many at once as their rows' memory allows
  for (size_t first = 0; first < jobs.size();) {
    std::vector<int64_t> off(n_pass, 0);
    int64_t ints = 0;
    int n = 0, max_pitch = 0, max_width = 0;
    while (first + n < jobs.size()) {
      const int x = jobs[first + n], i = slots[x].id;
      const size_t need = rows_of(x);
      if (n > 0 && (size_t)ints * 4 + need > limit) break;
      off[x] = ints;
      ints += need / 4;
      max_pitch = std::max(max_pitch, wfa::tile_pitch(js.h_plen[i], js.h_tlen[i]));
      max_width = std::max(max_width, js.h_plen[i] + js.h_tlen[i] + 4);
      ++n;
    }
    const int* sel = jobs.data() + first;
    if (!t.d_step_state.ensure((size_t)ints * 4, std::max(limit, (size_t)ints * 4)) ||
        !t.d_step_act.ensure((size_t)2 * n * 4 + 64)) {
      limit = (size_t)ints * 2;  // fewer at once, or without this one
      if (n == 1) ++first;
      continue;
    }
    int* n_act = t.d_step_act.as<int>();
    int* act[2] = {n_act + 16, n_act + 16 + n};
    wfa::StepArgs s{};
    s.act = act[0];
    s.n_act = n_act;
    s.jobs = a.jobs;
    s.words = js.words;
    s.state = t.d_step_state.as<int>();
    s.st_off = t.d_step_off.as<int64_t>();
    s.done = a.done;
    s.ends = t.d_ends.as<int>();
    s.flags = t.d_flags.as<int>();
    s.dsum = t.d_dsum.as<long long>();
    s.step0 = t.d_step0.as<int>();
    s.rec = a.rec;
    s.rec_tab = a.rec_tab;
    s.tab_stride = a.tab_stride;
    s.blocks = t.d_up.as<wfa::TileBlockInfo>();
    volatile int* h_n = t.h_n.as<int>() + 8;
    if (!hip_ok(hipMemcpyAsync(t.d_step_off.p, off.data(), (size_t)n_pass * 8, hipMemcpyHostToDevice, st), "steps") ||
        !hip_ok(hipMemcpyAsync(act[0], sel, (size_t)n * 4, hipMemcpyHostToDevice, st), "steps") ||
        !hip_ok(hipMemcpyAsync(n_act, &n, 4, hipMemcpyHostToDevice, st), "steps") ||
        !hip_ok(wfa::launch_tile_step_init(shape, s, a, n, max_pitch, st), "step init"))
      return WF_STATUS_OOM;
    // blocks of T steps, every job at the same place of its block
    int known = n, which = 0;
    for (int b = 0; known > 0; ++b) {
      uint32_t units = 0;
      bool any = false;
      for (int x = 0; x < n; ++x) {
        const size_t blk = (size_t)irr[sel[x]] / T + b;
        if (blk >= info.size()) continue;
        any = true;
        units = std::max(units, (uint32_t)((size_t)T * info[blk].pitch / 16));
      }
      if (!any) break;
      if (records && *unit + (uint64_t)known * units > rec_units) break;
      s.act = act[which];
      s.n_act = n_act + which;
      s.rec_unit0 = (uint32_t)*unit;
      s.rec_job_units = units;
      if (records) *unit += (uint64_t)known * units;
      for (int x = 0; x < T; ++x)
        if (!hip_ok(wfa::launch_tile_step(shape, records != 0, s, b * T + x, known, max_width, st), "step launch"))
          return WF_STATUS_OOM;
      const int slot = b & 1;
      if (!hip_ok(wfa::launch_tile_compact(act[which], n_act + which, a.done, nullptr, INT_MAX, act[which ^ 1],
                                           n_act + (which ^ 1), nullptr, const_cast<int*>(h_n) + slot, st),
                  "tile compact") ||
          !hip_ok(hipEventRecord(t.ev[slot], st), "tile event"))
        return WF_STATUS_OOM;
      which ^= 1;
      if (b > 0) {
        if (!hip_ok(hipEventSynchronize(t.ev[slot ^ 1]), "steps")) return WF_STATUS_OOM;
        known = h_n[slot ^ 1];
      }
    }
    if (!hip_ok(hipStreamSynchronize(st), "steps")) return WF_STATUS_OOM;
    first += n;
  }
  return WF_STATUS_OK;
}

// Aligns the jobs of a tile group; statuses, scores and CIGARs stay on the
// device, and jobs to be re-run are counted in the run counters.  The last
// pass is only queued, with the group's events around its kernels (a single
// pair of 1,100 bp at 0.5% errors spent more time on waits than on kernels).
int run_tile_group(Engine* e, const JobSet& js, PlanGroup& grp, const wfa::Penalties& pen, int records,
                   RunTotals* tot, std::vector<int>* ring) {
  Engine::TileState& t = e->tile;
  const int shape = wfa::tile_shape(pen);
  const wfa::TileGeometry g = wfa::tile_geometry(shape);
  hipStream_t st = e->stream;
  wfa::Counters* c = counters_of(e);
  const int T = g.steps;
  // no alignment costs more than deleting and inserting everything, or than
  // mismatches along the shorter sequence
  int max_steps = 0;
  for (int i : grp.ids) {
    const int64_t mn = std::min(js.h_plen[i], js.h_tlen[i]), mx = std::max(js.h_plen[i], js.h_tlen[i]);
    max_steps = (int)std::max<int64_t>(max_steps, mn * g.dx + g.do1 + (mx - mn) * g.de1);
  }
  const int max_blocks = max_steps / T + 2;
  if (!tile_table(e, shape, (max_blocks + 1) * T)) return WF_STATUS_OOM;
  for (auto& ev : t.ev)
    if (!ev && !hip_ok(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate")) return WF_STATUS_OOM;
  for (auto& ev : grp.ev)
    if (!ev && !hip_ok(hipEventCreate(&ev), "hipEventCreate")) return WF_STATUS_OOM;
  if (!t.h_n.ensure(4096)) return WF_STATUS_OOM;
  volatile int* h_n = t.h_n.as<int>();
  // per block the tiles a job has at most, and its records' first diagonal
  // and bytes per step (no range goes beyond the longest sequences)
  int pmax = 0, tmax = 0;
  for (int i : grp.ids) { pmax = std::max(pmax, js.h_plen[i]); tmax = std::max(tmax, js.h_tlen[i]); }
  std::vector<wfa::TileBlockInfo> info(max_blocks);
  std::vector<int> tiles(max_blocks);
  for (int b = 0; b < max_blocks; ++b) {
    const int lo = std::max(t.lo[(size_t)(b + 1) * T - 1], -pmax - 1), hi = std::min(t.hi[(size_t)(b + 1) * T - 1], tmax + 1);
    const int kb = -((-lo + 15) / 16 * 16);
    info[b] = wfa::TileBlockInfo{kb, (hi - kb + 16) / 16 * 16};
    const int lo0 = b ? std::max(t.lo[(size_t)b * T - 1], -pmax - 1) : 0, hi0 = b ? std::min(t.hi[(size_t)b * T - 1], tmax + 1) : 0;
    tiles[b] = (hi0 - lo0 + 1 + 2 * T + 8) / g.useful + 1;
  }
  const int n_all = (int)grp.ids.size();
  const uint64_t rec_units = records ? std::min<uint64_t>(e->rec.cap / 16, 0xFFFFFFF0ull) : 0;

  // device bytes of a job: its rows, its blocks' records, and what the kernels keep of it
  auto rows_of = [&](int i) { return (size_t)wfa::tile_pitch(js.h_plen[i], js.h_tlen[i]) * g.state_rows * 4; };
  const size_t tab_bytes = (records ? (size_t)max_blocks * 4 : 0) + (size_t)4 * T * 8 + sizeof(wfa::TileJob) +
                           sizeof(wfa::TileSlot) + 4 * sizeof(wfa::TileRange) + 7 * 4;
  size_t want = 0;
  for (int i : grp.ids) want += rows_of(i);
  size_t limit = rows_limit(e, want, kTileStateBytes, t.d_state.cap);
  bool some = false, timed = false;  // a pass has run; the group's events are its own

  for (int first = 0; first < n_all;) {
    // the jobs of one pass: their buffers and planned records fit
    size_t bytes = 0;
    int64_t ints = 0;
    double rec_plan = 0;
    int n = 0, lw = 0, taken = 0;
    std::vector<wfa::TileSlot> slots;
    for (; first + taken < n_all && n < kTileMaxJobs; ++taken) {
      const int i = grp.ids[first + taken];
      const size_t need = rows_of(i) + tab_bytes;
      const double L = std::max(js.h_plen[i], js.h_tlen[i]);
      if (e->rows_cap && need > e->rows_cap) {
        ring->push_back(i);
        continue;
      }
      if (n > 0 && (bytes + need > limit || grp.max_grid == n ||
                    (records && rec_plan + L * L * kTileRecordShareOfL2 > (double)rec_units * 16)))
        break;
      slots.push_back(wfa::TileSlot{ints, i, 0});
      bytes += need;
      ints += (int64_t)(rows_of(i) / 4);
      rec_plan += L * L * kTileRecordShareOfL2;
      lw = std::max(lw, (int)L / 32 + 3);
      ++n;
    }
    if (n == 0) break;
    const size_t nn = (size_t)n, up_info = (size_t)max_blocks * sizeof(wfa::TileBlockInfo);
    const size_t up = up_info + nn * sizeof(wfa::TileSlot);
    if (!t.d_state.ensure((size_t)ints * 4, std::max(limit, (size_t)ints * 4)) || !t.d_up.ensure(up) ||
        !t.h_up.ensure(up) || !t.d_jobs.ensure(nn * sizeof(wfa::TileJob)) || !t.d_marks.ensure(nn * 5 * 4) ||
        !t.d_job_range.ensure(nn * 4 * sizeof(wfa::TileRange)) || !t.d_dev.ensure(nn * 4 * T * 8) ||
        !t.d_act.ensure(2 * nn * 4 + 64) || (records && !t.d_tab.ensure(nn * max_blocks * 4))) {
      // fewer at once, or without this one
      limit = bytes / 2;
      if (n == 1) {
        ring->push_back(slots[0].id);
        first += taken;
      } else {
        ring->resize(ring->size() - (size_t)(taken - n));
      }
      continue;
    }
    // block infos and slots go up in one copy (once the one before is through)
    (void)hipEventSynchronize(t.ev[2]);
    memcpy(t.h_up.p, info.data(), up_info);
    memcpy(t.h_up.as<char>() + up_info, slots.data(), nn * sizeof(wfa::TileSlot));
    if (!hip_ok(hipMemcpyAsync(t.d_up.p, t.h_up.p, up, hipMemcpyHostToDevice, st), "tiles") ||
        !hip_ok(hipEventRecord(t.ev[2], st), "tile event"))
      return WF_STATUS_OOM;
    int* marks = t.d_marks.as<int>();
    int* n_act = t.d_act.as<int>();  // counts of the two lists, and of the jobs lost
    int* act[2] = {n_act + 16, n_act + 16 + n};
    int* lost = n_act + 2;
    wfa::TileArgs a{};
    a.act = act[0];
    a.n_act = n_act;
    a.jobs = t.d_jobs.as<wfa::TileJob>();
    a.words = js.words;
    a.state = t.d_state.as<int>();
    a.done = marks;
    a.irr = marks + nn;
    a.range = t.d_job_range.as<wfa::TileRange>();
    a.m_range = t.d_range.as<int2>();
    a.exact_lo = marks + 2 * nn;
    a.exact_hi = marks + 3 * nn;
    a.stepped = marks + 4 * nn;
    for (int x = 0; x < 4; ++x) a.dev[x / 2][x % 2] = t.d_dev.as<long long>() + nn * T * x;
    a.dsteps_upto = t.d_dsteps.as<long long>();
    a.rec = e->rec.as<uint4>();
    a.rec_tab = t.d_tab.as<uint32_t>();
    a.tab_stride = max_blocks;
    a.lmax_words = lw;
    (void)hipEventRecord(grp.ev[0], st);
    if (!hip_ok(wfa::launch_tile_fill(a.state, ints, st), "tile fill") ||
        !hip_ok(wfa::launch_tile_init(shape, a, n, reinterpret_cast<wfa::TileSlot*>(t.d_up.as<char>() + up_info),
                                      wfa::TileSeqs{js.plen, js.tlen, js.ppos, js.tpos}, act[0], n_act, lost, st),
                "tile init"))
      return WF_STATUS_OOM;
    int known = n, jobs_lost = 0, which = 0, chunk = 0;
    uint64_t unit = 0;
    bool full = false;
    for (int b = 0; b < max_blocks && known > 0 && !full;) {
      const int to = std::min(max_blocks, b + (b < 3 ? 1 + b : b < 2 * kTileChunk ? 4 : kTileChunk));
      for (; b < to; ++b) {
        a.act = act[which];
        a.n_act = n_act + which;
        a.blk = b;
        a.tiles = tiles[b];
        a.rec_kb = info[b].kb;
        a.rec_pitch = info[b].pitch;
        a.rec_job_units = (uint32_t)((size_t)T * info[b].pitch / 16);
        a.rec_unit0 = (uint32_t)unit;
        if (records) {
          if (unit + (uint64_t)known * a.rec_job_units > rec_units) { full = true; break; }
          unit += (uint64_t)known * a.rec_job_units;
        }
        if (!hip_ok(wfa::launch_tile_block(shape, records != 0, a, known, st), "tile launch")) return WF_STATUS_OOM;
      }
      if (full) break;
      // drop the finished jobs; the host looks at the count one chunk later,
      // so that the device always has launches queued
      const int slot = chunk & 1;
      if (!hip_ok(wfa::launch_tile_compact(act[which], n_act + which, a.done, a.irr, b * T, act[which ^ 1],
                                           n_act + (which ^ 1), lost, const_cast<int*>(h_n) + slot, st), "tile compact") ||
          !hip_ok(hipEventRecord(t.ev[slot], st), "tile event"))
        return WF_STATUS_OOM;
      which ^= 1;
      if (chunk > 0) {
        if (!hip_ok(hipEventSynchronize(t.ev[slot ^ 1]), "tiles")) return WF_STATUS_OOM;
        known = h_n[slot ^ 1];
        jobs_lost = h_n[(slot ^ 1) + wfa::kTileHostLost];
      }
      ++chunk;
    }
    // (known == 0: the last list that was seen was empty, so every job was done or lost by then)
    if (!full && (known > 0 || jobs_lost > 0)) {
      const int rc = run_steps(e, js, shape, g, a, slots, n, info, records, rec_units, &unit);
      if (rc != WF_STATUS_OK) return rc;
    }
    wfa::TileFinishArgs f{};
    f.n = n;
    f.jobs = a.jobs;
    f.done = a.done;
    f.irr = a.irr;
    f.exact_lo = a.exact_lo;
    f.exact_hi = a.exact_hi;
    for (int x = 0; x < 4; ++x) f.dev[x / 2][x % 2] = a.dev[x / 2][x % 2];
    f.stepped = a.stepped;
    f.step_ends = t.d_ends.as<int>();
    f.flags = t.d_flags.as<int>();
    f.dsum = t.d_dsum.as<long long>();
    f.steps = T;
    f.dsteps_upto = t.d_dsteps.as<long long>();
    f.g = pen.g;
    f.out_status = js.status;
    f.out_score = js.score;
    f.out_dsteps = js.dsteps;
    f.out_last_block = js.last;
    f.out_end_k = js.end_k;
    f.out_end_off = js.end_off;
    f.dsteps_total = &c->dsteps;
    f.retry_count = &c->retry;
    if (!hip_ok(wfa::launch_tile_finish(shape, f, st), "tile finish")) return WF_STATUS_OOM;
    (void)hipEventRecord(grp.ev[1], st);
    if (records) {
      wfa::TileTraceArgs ta{};
      ta.jobs = a.jobs;
      ta.status = js.status;
      ta.score = js.score;
      ta.rec = a.rec;
      ta.rec_tab = a.rec_tab;
      ta.tab_stride = a.tab_stride;
      ta.blocks = t.d_up.as<wfa::TileBlockInfo>();
      ta.words = js.words;
      ta.ops = js.ops;
      ta.ops_off = js.ops_off;
      ta.ops_begin = js.ops_begin;
      ta.fail_count = &c->fail;
      ta.g = pen.g;
      ta.lmax_words = lw;
      if (!hip_ok(wfa::launch_tile_backtrace(shape, ta, n, st), "tile backtrace")) return WF_STATUS_OOM;
    }
    (void)hipEventRecord(grp.ev[2], st);
    if (some) ++tot->launches;  // a further pass (the caller counts one)
    some = timed = true;
    first += taken;
    if (first < n_all) {
      // the buffers and events are used again
      if (!hip_ok(hipStreamSynchronize(st), "tiles")) return WF_STATUS_OOM;
      float fms = 0, bms = 0;
      (void)hipEventElapsedTime(&fms, grp.ev[0], grp.ev[1]);
      (void)hipEventElapsedTime(&bms, grp.ev[1], grp.ev[2]);
      tot->forward_ms += fms;
      tot->backtrace_ms += bms;
      timed = false;
    }
  }
  if (!timed)
    for (auto& ev : grp.ev) (void)hipEventRecord(ev, st);  // (no time, for the caller to read)
  return WF_STATUS_OK;
}

}  // namespace wfa_host
