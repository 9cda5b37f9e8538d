// Long pairs in tiles of diagonals, a block of score steps per launch.
//
// The wavefronts of a long pair are thousands of diagonals wide and thousands
// of steps deep.  One workgroup per pair with a ring in HBM spends its time
// waiting: each step reads nine neighbours per diagonal from the ring, then a
// barrier, and the longest pair of a batch keeps one CU busy while the others
// have nothing left.  Here a wave takes 64 * N neighbouring diagonals through
// T steps in registers (wfa_rows.h), without a barrier: the T diagonals at
// each end of its stretch are halo, computed by the neighbouring tile as well
// and thrown away.  A launch runs one block of T steps of every pair still
// running, so all tiles of all pairs spread over the whole device, and the
// launch boundary is the only synchronization between tiles.
//
// What makes the tiles independent of each other is where the reference trims
// (wavefront_compute.c:579-613): only invalid cells at the two ends of a
// wavefront's range are dropped, and a cell is invalid only when nothing
// reaches it or when it has left the matrix.  The ranges are therefore the
// same for every pair (the host tabulates them once per penalties) until an
// end cell leaves the matrix, and everything that follows from such a cell
// concerns the tile at that end alone: gap cells beyond the last valid one
// read as NULL from then on.  The first and the last tile of a pair watch for
// it (`exact` below); the tiles between never trim.  The tiles are laid out
// anew at each block over the range of the pair, all of one width, so an end
// sits at least half a tile away from the border of its tile.  Where scores
// exceed the sequences' lengths (very different sequences) the ends jump:
// whole stretches of cells leave the matrix together.  A pair whose end moved
// past its tile's border goes on from the start of that block one step per
// launch (tile_step_kernel), with the ranges of every step reduced over all
// tiles; that is a few hundred steps at the end of such a pair.
#include <algorithm>
#include <climits>

#include "wfa_rows.h"
#include "wfa_tile.h"

namespace wfa {
namespace {

constexpr int kTileWaves = 4;  // waves per workgroup: they share the sequences in LDS

// N, T: at most 25 steps per block for gap-affine-2p, so that the rows of the
// second gap's opening (25 steps back) all come from earlier blocks.  More
// steps mean fewer launches and wider halos: 256 gap-affine pairs of 1-20 kbp
// take 10.5 ms with 16, 9.8 with 24, 9.5 with 32 (score only 8.0, 7.3, 6.9).
template <class S>
struct TileGeom;
template <>
struct TileGeom<Shape2p> {
  static constexpr int N = 4, T = 24, UNROLL = 8, MS = 50;  // every row goes to the ring of MS rows
};
template <>
struct TileGeom<ShapeAffine> {
  static constexpr int N = 4, T = 32, UNROLL = 4, MS = 8;   // the last RM rows of a block, by its parity
};
template <class S>
constexpr int tile_halo() { return (TileGeom<S>::T + 3) / 4 * 4; }
template <class S>
constexpr int tile_useful() { return 64 * TileGeom<S>::N - 2 * tile_halo<S>(); }

// Ring slot of M row i: gap-affine-2p keeps every row; otherwise the last RM
// rows of block `blk` sit in the half of the block's parity.
template <class S>
__device__ __forceinline__ int m_slot(int i, int blk) {
  constexpr int MS = TileGeom<S>::MS;
  if constexpr (S::NC == 5) {
    const int r = i % MS;
    return r < 0 ? r + MS : r;
  } else {
    return (blk & 1) * S::RM + (i & (S::RM - 1));
  }
}

__device__ __forceinline__ int4 load4(const int* p) { return *reinterpret_cast<const int4*>(p); }

template <int N>
__device__ __forceinline__ void load_row(int* r, const int* p) {
#pragma unroll
  for (int c = 0; c < N; c += 4) {
    const int4 v = load4(p + c);
    r[c] = v.x; r[c + 1] = v.y; r[c + 2] = v.z; r[c + 3] = v.w;
  }
}
template <int N>
__device__ __forceinline__ void store_row(int* p, const int* r) {
#pragma unroll
  for (int c = 0; c < N; c += 4) *reinterpret_cast<int4*>(p + c) = make_int4(r[c], r[c + 1], r[c + 2], r[c + 3]);
}

// One block of T steps [ib, ib + T) of the active pairs: blockIdx.y the pair,
// blockIdx.x a group of kTileWaves tiles.
template <class S, bool REC>
__global__ void __launch_bounds__(64 * kTileWaves) wfa_tile_kernel(TileArgs a) {
  using G = TileGeom<S>;
  constexpr int N = G::N, T = G::T, H = tile_halo<S>(), U = tile_useful<S>();
  static_assert(T % G::UNROLL == 0 && H % N == 0 && U % N == 0 && T >= 2 * S::DE1, "tile geometry");
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.y >= *a.n_act) return;
  const int job = a.act[blockIdx.y];
  const int ib = a.blk * T;
  // finished or handed back in an earlier block (a mark of this block does
  // not count: its records before the mark are still needed)
  if (a.done[job] < ib || a.irr[job] < ib) return;
  if (REC && blockIdx.x == 0 && threadIdx.x == 0)
    a.rec_tab[(long long)job * a.tab_stride + a.blk] = a.rec_unit0 + blockIdx.y * a.rec_job_units;
  // the pair's diagonals [left, right) of this block, in tiles
  const TileRange r1 = a.range[4 * job + ((a.blk + 3) & 3)], r2 = a.range[4 * job + ((a.blk + 2) & 3)];
  const int left = (min(r1.min_lo, r2.min_lo) - T) & ~3;
  const int right = (max(r1.max_hi, r2.max_hi) + T + 4) & ~3;
  const int tiles = (right - left + U - 1) / U;
  const int quads = (right - left) / 4;  // tiles of equal width, in units of four diagonals
  if ((int)blockIdx.x * kTileWaves >= tiles) return;
  const TileJob jb = a.jobs[job];
  const int plen = jb.plen, tlen = jb.tlen;
  const long long ppos = jb.ppos, tpos = jb.tpos;
  uint64_t* seqP = reinterpret_cast<uint64_t*>(smem);
  uint64_t* seqT = seqP + a.lmax_words;
  {
    const uint64_t* gP = a.words + (ppos >> 5);
    const uint64_t* gT = a.words + (tpos >> 5);
    const int nwp = ((int)(ppos & 31) + plen) / 32 + 2, nwt = ((int)(tpos & 31) + tlen) / 32 + 2;
    for (int i = threadIdx.x; i < nwp; i += 64 * kTileWaves) seqP[i] = gP[i];
    for (int i = threadIdx.x; i < nwt; i += 64 * kTileWaves) seqT[i] = gT[i];
    __syncthreads();
  }
  const int lane = threadIdx.x & 63;
  const int tile = (int)blockIdx.x * kTileWaves + uniform(threadIdx.x >> 6);
  if (tile >= tiles) return;
  const int first = left + 4 * (quads * tile / tiles);  // the tile's own diagonals [first, past)
  const int past = left + 4 * (quads * (tile + 1) / tiles);
  const WaveSeqs<2> q{reinterpret_cast<const uint32_t*>(seqP), reinterpret_cast<const uint32_t*>(seqT),
                   2u * (unsigned)(ppos & 31), 2u * (unsigned)(tpos & 31), plen, tlen};
  const int kt = first - H, k0 = kt + N * lane;
  const bool own = k0 >= first && k0 < past;
  const int kend = tlen - plen;
  const bool has_end = kend >= first && kend < past;
  const bool low = tile == 0, high = past == right;
  const int pitch = jb.pitch;
  int* st = a.state + jb.st_off + (k0 + tile_kpad(plen));
  auto mrow = [&](int slot) { return st + (long long)slot * pitch; };
  auto grow = [&](int par, int row) { return st + (long long)(G::MS + par * S::kGapRows + row) * pitch; };
  // Rows were written over the diagonals of their block: beyond them the
  // memory holds rows of earlier, wider blocks.
  const bool in1 = k0 >= r1.left && k0 < r1.right, in2 = k0 >= r2.left && k0 < r2.right;
  auto load = [&](int* r, const int* p, bool in) {
    load_row<N>(r, p);
#pragma unroll
    for (int c = 0; c < N; ++c) r[c] = in ? r[c] : kNullTagged;
  };

  WaveRows<S, N> w;
#pragma unroll
  for (int r = 0; r < S::RM; ++r) load(w.m[r], mrow(m_slot<S>(ib - S::RM + r, a.blk - 1)), in1);
  const int pin = (a.blk & 1) ^ 1;
#pragma unroll
  for (int r = 0; r < S::DE1; ++r) {
    load(w.i1[r], grow(pin, r), in1);
    load(w.d1[r], grow(pin, S::DE1 + r), in1);
  }
  if constexpr (S::NC == 5) {
#pragma unroll
    for (int r = 0; r < S::DE2; ++r) {
      load(w.i2[r], grow(pin, 2 * S::DE1 + r), in1);
      load(w.d2[r], grow(pin, 2 * S::DE1 + S::DE2 + r), in1);
    }
  }
  static_assert(T % S::RM == 0 && T % S::DE1 == 0 && T % S::DE2 == 0, "blocks start at phase 0");
  static_assert(S::NC != 5 || (S::DO2 > T && S::DO2 <= 2 * T && S::DE2 == 1), "second gap's rows");
  uint8_t* rec = nullptr;
  bool rec_own = false;
  if constexpr (REC) {
    rec_own = own && k0 >= a.rec_kb && k0 < a.rec_kb + a.rec_pitch;
    rec = reinterpret_cast<uint8_t*>(a.rec + a.rec_unit0 + (long long)blockIdx.y * a.rec_job_units) + (k0 - a.rec_kb);
  }

  int o2[N], o2n[N];
  int so2 = 0, sw = 0;  // ring slots of the second gap's opening row and of the row written
  if constexpr (S::NC == 5) {
    so2 = m_slot<S>(ib - S::DO2, 0);
    sw = m_slot<S>(ib, 0);
    load(o2n, mrow(so2), ib - S::DO2 >= ib - T ? in1 : in2);
  }
  // Ends.  Until a cell of the end tile has left the matrix the ranges are
  // the tabulated ones; from then on (exact) they are taken from the cells:
  // a diagonal is in the computed range [lo, hi] iff some source reaches it.
  bool exact = (low && a.exact_lo[job]) || (high && a.exact_hi[job]);
  long long dev_lo = 0, dev_hi = 0;  // exact minus tabulated limits, summed over the steps
  long long* const devs[2] = {a.dev[a.blk & 1][0] + (long long)job * T, a.dev[a.blk & 1][1] + (long long)job * T};
  int min_lo = INT_MAX, max_hi = INT_MIN;
  if (exact) {
    if (low && a.exact_lo[job]) dev_lo = a.dev[(a.blk & 1) ^ 1][0][(long long)job * T + T - 1];
    if (high && a.exact_hi[job]) dev_hi = a.dev[(a.blk & 1) ^ 1][1][(long long)job * T + T - 1];
  }
  bool ended = false, lost = false;
  auto one = [&](auto phc, int t) {
    constexpr int PH = decltype(phc)::value;
    const int i = ib + t;
    if constexpr (S::NC == 5) {
#pragma unroll
      for (int c = 0; c < N; ++c) o2[c] = o2n[c];
      so2 = so2 + 1 == G::MS ? 0 : so2 + 1;
      if (t + 1 < T) load(o2n, mrow(so2), i + 1 - S::DO2 >= ib - T ? in1 : in2);  // one step ahead: a row of an earlier block
    }
    StepCells<N> cell;
    for (uint32_t& r : cell.rec) r = 0;
    wave_step<S, N, PH, 2>(w, o2, k0, q, cell);
    if constexpr (REC) {
      if (rec_own) {
#pragma unroll
        for (int c = 0; c < N; c += 4) *reinterpret_cast<uint32_t*>(rec + c) = cell.rec[c / 4];
      }
      rec += a.rec_pitch;
    }
    if (low || high) {
      uint32_t okm = 0, obm = 0;
#pragma unroll
      for (int c = 0; c < N; ++c) {
        okm |= cell.ok[c] ? 1u << c : 0u;
        obm |= cell.oob[c] ? 1u << c : 0u;
      }
      const int2 tab = a.m_range[i];
      if (!exact && __ballot(obm != 0)) {
        // (the steps before this one kept the tabulated limits)
        exact = true;
        if (lane == 0)
          for (int x = 0; x < t; ++x) {
            if (low) devs[0][x] = 0;
            if (high) devs[1][x] = 0;
          }
      }
      if (exact) {
        const int lo = first_diagonal<N>(okm | obm, kt), hi = last_diagonal<N>(okm | obm, kt);
        if (low) {
          if (lo != INT_MAX && tab.x <= tab.y) dev_lo += lo - tab.x;
          min_lo = min(min_lo, lo);
          if (lane == 0) devs[0][t] = dev_lo;
          const int f = first_diagonal<N>(okm, kt);
          lost |= (f != INT_MAX ? f >= past : lo != INT_MAX) || lo > 0;  // (lo > 0: see step_width)
        }
        if (high) {
          if (hi != INT_MIN && tab.x <= tab.y) dev_hi += hi - tab.y;
          max_hi = max(max_hi, hi);
          if (lane == 0) devs[1][t] = dev_hi;
          const int f = last_diagonal<N>(okm, kt);
          lost |= (f != INT_MIN ? f < first : hi != INT_MIN) || hi < 0;
        }
        // gap cells beyond the first and last valid ones read as NULL
        auto trim = [&](int* g) {
          uint32_t vm = 0, some = 0;
#pragma unroll
          for (int c = 0; c < N; ++c) {
            vm |= in_bounds(g[c] >> S::SH, k0 + c, plen, tlen) ? 1u << c : 0u;
            some |= g[c] >= 0 ? 1u << c : 0u;
          }
          if (!__ballot(some != 0)) return;
          const int f = first_diagonal<N>(vm, kt), l = last_diagonal<N>(vm, kt);
          if (low) {
            lost |= f >= past;  // (none: INT_MAX)
#pragma unroll
            for (int c = 0; c < N; ++c) g[c] = k0 + c < f ? kNullTagged : g[c];
          }
          if (high) {
            lost |= l < first;
#pragma unroll
            for (int c = 0; c < N; ++c) g[c] = k0 + c > l ? kNullTagged : g[c];
          }
        };
        trim(w.i1[PH % S::DE1]);
        trim(w.d1[PH % S::DE1]);
        if constexpr (S::NC == 5) {
          trim(w.i2[PH % S::DE2]);
          trim(w.d2[PH % S::DE2]);
        }
        if (lost) {
          if (lane == 0) atomicMin(a.irr + job, i);
          ended = true;
        }
      } else {
        if (tab.x <= tab.y) {
          min_lo = min(min_lo, tab.x);
          max_hi = max(max_hi, tab.y);
        }
      }
    }
    if constexpr (S::NC == 5) {
      if (own) store_row<N>(mrow(sw), w.m[PH % S::RM]);
      sw = sw + 1 == G::MS ? 0 : sw + 1;
    }
    if (has_end) {
      bool fin = false;
#pragma unroll
      for (int c = 0; c < N; ++c) fin |= cell.ok[c] & (k0 + c == kend) & (cell.h[c] >= tlen);
      if (__ballot(fin)) {
        if (lane == 0) atomicMin(a.done + job, i);
        // an end tile goes on: the counts of its steps belong to the block
        ended = ended || !(low || high);
      }
    }
  };
  for (int t = 0; t < T && !ended; t += G::UNROLL) {
    one(std::integral_constant<int, 0>{}, t);
    one(std::integral_constant<int, 1>{}, t + 1);
    one(std::integral_constant<int, 2>{}, t + 2);
    one(std::integral_constant<int, 3>{}, t + 3);
    if constexpr (G::UNROLL == 8) {
      one(std::integral_constant<int, 4>{}, t + 4);
      one(std::integral_constant<int, 5>{}, t + 5);
      one(std::integral_constant<int, 6>{}, t + 6);
      one(std::integral_constant<int, 7>{}, t + 7);
    }
  }
  if (lane == 0) {
    TileRange* mine = a.range + 4 * job + (a.blk & 3);
    if (low) {
      mine->left = left;
      mine->min_lo = min(min_lo, r1.max_hi);  // (a block without a wavefront keeps a place)
      if (exact && !a.exact_lo[job]) a.exact_lo[job] = a.blk + 1;
    }
    if (high) {
      mine->right = right;
      mine->max_hi = max(max_hi, r1.min_lo);
      if (exact && !a.exact_hi[job]) a.exact_hi[job] = a.blk + 1;
    }
  }
  if (ended || !own) return;
  const int pout = a.blk & 1;
  if constexpr (S::NC != 5) {
#pragma unroll
    for (int r = 0; r < S::RM; ++r) store_row<N>(mrow(m_slot<S>(ib + T - S::RM + r, a.blk)), w.m[r]);
  }
#pragma unroll
  for (int r = 0; r < S::DE1; ++r) {
    store_row<N>(grow(pout, r), w.i1[r]);
    store_row<N>(grow(pout, S::DE1 + r), w.d1[r]);
  }
  if constexpr (S::NC == 5) {
#pragma unroll
    for (int r = 0; r < S::DE2; ++r) {
      store_row<N>(grow(pout, 2 * S::DE1 + r), w.i2[r]);
      store_row<N>(grow(pout, 2 * S::DE1 + S::DE2 + r), w.d2[r]);
    }
  }
}

// Every state cell NULL.
__global__ void __launch_bounds__(256) tile_fill_kernel(int4* p, long long n4) {
  const int4 v = make_int4(kNullTagged, kNullTagged, kNullTagged, kNullTagged);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n4; i += (long long)gridDim.x * 256) p[i] = v;
}

// Score 0 of every job (M holds offset 0 at k = 0, extended;
// wavefront_aligner.c:252-380), its marks, and the first active list.
template <class S>
__global__ void __launch_bounds__(64) tile_init_kernel(TileArgs a, int n, const TileSlot* slots, TileSeqs seqs, int* act,
                                                       int* n_act, int* lost) {
  const int job = blockIdx.x * 64 + threadIdx.x;
  if (job == 0) {
    *n_act = n;
    *lost = 0;
  }
  if (job >= n) return;
  act[job] = job;
  const TileSlot sl = slots[job];
  const int plen = seqs.plen[sl.id], tlen = seqs.tlen[sl.id];
  const long long ppos = seqs.pat_pos[sl.id], tpos = seqs.txt_pos[sl.id];
  const int pitch = tile_pitch(plen, tlen);
  a.jobs[job] = TileJob{ppos, tpos, sl.st_off, plen, tlen, pitch, sl.id};
  const int h = lcp_extend<2>(a.words + (ppos >> 5), (int)(ppos & 31), a.words + (tpos >> 5), (int)(tpos & 31), plen,
                              tlen, 0, 0);
  a.state[sl.st_off + (long long)m_slot<S>(-1, -1) * pitch + tile_kpad(plen)] = h << S::SH;
  a.done[job] = (plen == tlen && h >= tlen) ? -1 : INT_MAX;
  a.irr[job] = INT_MAX;
  a.exact_lo[job] = a.exact_hi[job] = a.stepped[job] = 0;
  // before block 0: score 0 at diagonal 0, every other cell of the state NULL
  for (int x = 0; x < 4; ++x) a.range[4 * job + x] = TileRange{INT_MIN / 2, INT_MAX / 2, 0, 0};
}

// ------------------------------------------------- one step per launch
// Rows of the step kernels: M in a ring of 32 (8 without a second gap), every
// gap component in a ring of 4, so that a launch never writes a row it reads.
template <class S>
struct StepRows {
  static constexpr int MS = S::NC == 5 ? 32 : 8, G = S::NC == 5 ? 4 : 2, ROWS = MS + 4 * G;
  static __device__ __forceinline__ int m(int i) { return i & (MS - 1); }
  static __device__ __forceinline__ int gap(int comp, int i) { return MS + 4 * (comp - 1) + (i & 3); }
};
// Per job and step (ring of 4): the first and last valid cell of each gap
// component (I1, D1, I2, D2) and of M, and of the cells some source reaches.
constexpr int kStepEnds = kTileStepEnds, kEndsM = 8, kEndsReach = 10;
// Per job and step (ring of 32): bit c, whether component c has a valid cell.
constexpr int kStepFlags = kTileStepFlags;
__device__ __forceinline__ int* step_ends(const StepArgs& a, int job, int i) {
  return a.ends + ((long long)job * 4 + (i & 3)) * kStepEnds;
}

// Diagonals of step i (its ends e): from the first to the last cell a source
// reaches, widened by the limits (1, -1) that a null source contributes
// (wavefront_compute.c:40-86), shifted as its gap moves it.
template <class S>
__device__ __forceinline__ int step_width(const int* e, const int* flags, int i) {
  int lo = e[kEndsReach], hi = e[kEndsReach + 1];
  if (lo > hi) return 0;
  auto null = [&](int c, int from) { return !((flags[from & (kStepFlags - 1)] >> c) & 1); };
  if (null(kM, i - S::DX)) { lo = min(lo, 1); hi = max(hi, -1); }
  if (null(kM, i - S::DO1)) { lo = min(lo, 0); hi = max(hi, 0); }
  if (null(kI1, i - S::DE1)) { lo = min(lo, 2); hi = max(hi, 0); }
  if (null(kD1, i - S::DE1)) { lo = min(lo, 0); hi = max(hi, -2); }
  if constexpr (S::NC == 5) {
    if (null(kM, i - S::DO2)) { lo = min(lo, 0); hi = max(hi, 0); }
    if (null(kI2, i - S::DE2)) { lo = min(lo, 2); hi = max(hi, 0); }
    if (null(kD2, i - S::DE2)) { lo = min(lo, 0); hi = max(hi, -2); }
  }
  return hi - lo + 1;
}

// The first step's rows have no flags yet.
__global__ void __launch_bounds__(64) tile_step_flags_kernel(const int* act, int n, int* flags) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  if (j < n * kStepFlags) flags[(long long)act[j / kStepFlags] * kStepFlags + j % kStepFlags] = 0;
}

// Copies the rows the first step reads out of the tiles' state (NULL outside
// the diagonals they were written over) and sets the job's counts.
template <class S>
__global__ void __launch_bounds__(256) tile_step_init_kernel(StepArgs a, TileArgs tl) {
  using R = StepRows<S>;
  constexpr int T = TileGeom<S>::T, MT = TileGeom<S>::MS;
  const int job = a.act[blockIdx.y];
  const int ib = tl.irr[job] / T * T, blk = ib / T;
  const TileJob jb = tl.jobs[job];
  const int pitch = jb.pitch, kpad = tile_kpad(jb.plen);
  const TileRange r1 = tl.range[4 * job + ((blk + 3) & 3)], r2 = tl.range[4 * job + ((blk + 2) & 3)];
  const int* from = tl.state + jb.st_off;
  int* to = a.state + a.st_off[job];
  const int x = blockIdx.x * 256 + threadIdx.x;
  int* flags = a.flags + (long long)job * kStepFlags;
  auto copy = [&](int comp, int i, int row_to, int row_from) {
    const int v = from[(long long)row_from * pitch + x];
    to[(long long)row_to * pitch + x] = v;
    if (v >= 0 && !((flags[i & (kStepFlags - 1)] >> comp) & 1)) atomicOr(flags + (i & (kStepFlags - 1)), 1 << comp);
  };
  if (x < pitch) {
    const int k = x - kpad;
    const bool in1 = k >= r1.left && k < r1.right, in2 = k >= r2.left && k < r2.right;
    for (int r = 0; r < R::ROWS; ++r) to[(long long)r * pitch + x] = kNullTagged;
    constexpr int back = S::NC == 5 ? S::DO2 : S::RM;
    for (int i = ib - back; i < ib; ++i)
      if (i >= ib - T ? in1 : in2) copy(kM, i, R::m(i), m_slot<S>(i, blk - 1));
    const int pin = (blk & 1) ^ 1;
    if (in1) {
      for (int r = 0; r < S::DE1; ++r) {
        const int i = ib - S::DE1 + r;
        copy(kI1, i, R::gap(kI1, i), MT + pin * S::kGapRows + r);
        copy(kD1, i, R::gap(kD1, i), MT + pin * S::kGapRows + S::DE1 + r);
      }
      if constexpr (S::NC == 5) {
        for (int r = 0; r < S::DE2; ++r) {
          const int i = ib - S::DE2 + r;
          copy(kI2, i, R::gap(kI2, i), MT + pin * S::kGapRows + 2 * S::DE1 + r);
          copy(kD2, i, R::gap(kD2, i), MT + pin * S::kGapRows + 2 * S::DE1 + S::DE2 + r);
        }
      }
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < 4) {
    // the rows before ib are trimmed already: no limits on them
    int* e = a.ends + ((long long)job * 4 + threadIdx.x) * kStepEnds;
    const bool next = (int)threadIdx.x == (ib & 3);
    for (int c = 0; c < kStepEnds / 2; ++c) {
      e[2 * c] = next ? INT_MAX : INT_MIN;
      e[2 * c + 1] = next ? INT_MIN : INT_MAX;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int x0 = tl.exact_lo[job], x1 = tl.exact_hi[job];
    long long sum = tl.dsteps_upto[ib];
    if (x0 && x0 - 1 < blk) sum -= tl.dev[(blk & 1) ^ 1][0][(long long)job * T + T - 1];
    if (x1 && x1 - 1 < blk) sum += tl.dev[(blk & 1) ^ 1][1][(long long)job * T + T - 1];
    a.dsum[job] = sum;
    a.step0[job] = ib;
    tl.done[job] = INT_MAX;
  }
}

// Clears the marks of the jobs that change over (after their rows are copied).
__global__ void __launch_bounds__(64) tile_step_mark_kernel(const int* act, int n, int* irr, int* stepped) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  if (j >= n) return;
  irr[act[j]] = INT_MAX;
  stepped[act[j]] = 1;
}

constexpr int kStepWaves = 8;
// One step of every active job over all its diagonals; each wave owns 62 * 4
// of them (a lane at each end is halo).
template <class S, bool REC>
__global__ void __launch_bounds__(64 * kStepWaves) tile_step_kernel(StepArgs a, int t) {
  using R = StepRows<S>;
  constexpr int N = 4, T = TileGeom<S>::T;
  __shared__ int sh[kStepWaves][kStepEnds];
  if ((int)blockIdx.y >= *a.n_act) return;
  const int job = a.act[blockIdx.y];
  const int i = a.step0[job] + t;
  if (a.done[job] < i) return;
  const int lane = threadIdx.x & 63, wid = uniform(threadIdx.x >> 6);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (t > 0) {
      const int* p = step_ends(a, job, i - 1);
      int* fl = a.flags + (long long)job * kStepFlags;
      a.dsum[job] += step_width<S>(p, fl, i - 1);
      int f = p[kEndsM] <= p[kEndsM + 1] ? 1 << kM : 0;
      for (int c = kI1; c <= kD2; ++c) f |= p[2 * (c - 1)] <= p[2 * (c - 1) + 1] ? 1 << c : 0;
      fl[(i - 1) & (kStepFlags - 1)] = f;
    }
    int* nx = step_ends(a, job, i + 1);
    for (int c = 0; c < kStepEnds / 2; ++c) {
      nx[2 * c] = INT_MAX;
      nx[2 * c + 1] = INT_MIN;
    }
    if (REC && i % T == 0) a.rec_tab[(long long)job * a.tab_stride + i / T] = a.rec_unit0 + blockIdx.y * a.rec_job_units;
  }
  const TileJob jb = a.jobs[job];
  const int plen = jb.plen, tlen = jb.tlen;
  const int base = (-plen - 2) & ~3;
  const int first = base + ((int)blockIdx.x * kStepWaves + wid) * (62 * N);
  if (base + (int)blockIdx.x * kStepWaves * (62 * N) > tlen + 1) return;
  const int k0 = first + N * (lane - 1);
  const bool own = lane >= 1 && lane < 63;
  const int pitch = jb.pitch;
  const bool some = first <= tlen + 1;  // a wave past the last diagonal has nothing to do
  int rng[kStepEnds];
#pragma unroll
  for (int c = 0; c < kStepEnds / 2; ++c) { rng[2 * c] = INT_MAX; rng[2 * c + 1] = INT_MIN; }
  if (some) {
    int* st = a.state + a.st_off[job] + (k0 + tile_kpad(plen));
    const int* e1 = step_ends(a, job, i - S::DE1);
    const int* e2 = step_ends(a, job, i - S::DE2);
    auto load_gap = [&](int* r, int comp, int from, const int* e) {
      load_row<N>(r, st + (long long)R::gap(comp, from) * pitch);
      const int lo = e[2 * (comp - 1)], hi = e[2 * (comp - 1) + 1];
#pragma unroll
      for (int c = 0; c < N; ++c) r[c] = (k0 + c < lo || k0 + c > hi) ? kNullTagged : r[c];
    };
    int mx[N], mo[N], mo2[N], i1[N], d1[N], i2[N], d2[N], m[N];
    load_row<N>(mx, st + (long long)R::m(i - S::DX) * pitch);
    load_row<N>(mo, st + (long long)R::m(i - S::DO1) * pitch);
    load_gap(i1, kI1, i - S::DE1, e1);
    load_gap(d1, kD1, i - S::DE1, e1);
    if constexpr (S::NC == 5) {
      load_row<N>(mo2, st + (long long)R::m(i - S::DO2) * pitch);
      load_gap(i2, kI2, i - S::DE2, e2);
      load_gap(d2, kD2, i - S::DE2, e2);
    }
    const long long ppos = jb.ppos, tpos = jb.tpos;
    const WaveSeqs<2> q{reinterpret_cast<const uint32_t*>(a.words + (ppos >> 5)),
                     reinterpret_cast<const uint32_t*>(a.words + (tpos >> 5)), 2u * (unsigned)(ppos & 31),
                     2u * (unsigned)(tpos & 31), plen, tlen};
    StepCells<N> cell;
    for (uint32_t& r : cell.rec) r = 0;
    wave_cells<S, N, 2>(mx, mo, i1, d1, mo2, i2, d2, m, k0, q, cell);
    if (own) {
      store_row<N>(st + (long long)R::m(i) * pitch, m);
      store_row<N>(st + (long long)R::gap(kI1, i) * pitch, i1);
      store_row<N>(st + (long long)R::gap(kD1, i) * pitch, d1);
      if constexpr (S::NC == 5) {
        store_row<N>(st + (long long)R::gap(kI2, i) * pitch, i2);
        store_row<N>(st + (long long)R::gap(kD2, i) * pitch, d2);
      }
      if constexpr (REC) {
        const TileBlockInfo bi = a.blocks[i / T];
        if (k0 >= bi.kb && k0 < bi.kb + bi.pitch)
          *reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(a.rec + a.rec_unit0 + (long long)blockIdx.y * a.rec_job_units) +
                                       (long long)(i % T) * bi.pitch + (k0 - bi.kb)) = cell.rec[0];
      }
    }
    // the ends of this step over the wave's own cells
    const int kt = first - N, kend = tlen - plen;
    auto ends_of = [&](auto valid, int at) {
      uint32_t vm = 0;
#pragma unroll
      for (int c = 0; c < N; ++c) vm |= (own && valid(c)) ? 1u << c : 0u;
      rng[at] = first_diagonal<N>(vm, kt);
      rng[at + 1] = last_diagonal<N>(vm, kt);
    };
    ends_of([&](int c) { return in_bounds(i1[c] >> S::SH, k0 + c, plen, tlen); }, 0);
    ends_of([&](int c) { return in_bounds(d1[c] >> S::SH, k0 + c, plen, tlen); }, 2);
    if constexpr (S::NC == 5) {
      ends_of([&](int c) { return in_bounds(i2[c] >> S::SH, k0 + c, plen, tlen); }, 4);
      ends_of([&](int c) { return in_bounds(d2[c] >> S::SH, k0 + c, plen, tlen); }, 6);
    }
    ends_of([&](int c) { return cell.ok[c]; }, kEndsM);
    ends_of([&](int c) { return cell.ok[c] | cell.oob[c]; }, kEndsReach);
    bool fin = false;
#pragma unroll
    for (int c = 0; c < N; ++c) fin |= own & cell.ok[c] & (k0 + c == kend) & (cell.h[c] >= tlen);
    if (fin) a.done[job] = i;
  }
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < kStepEnds; ++c) sh[wid][c] = rng[c];
  }
  __syncthreads();
  if (threadIdx.x < kStepEnds) {
    int v = sh[0][threadIdx.x];
    const bool lo = (threadIdx.x & 1) == 0;
    for (int x = 1; x < kStepWaves; ++x) v = lo ? min(v, sh[x][threadIdx.x]) : max(v, sh[x][threadIdx.x]);
    int* e = step_ends(a, job, i) + threadIdx.x;
    if (lo && v != INT_MAX) atomicMin(e, v);
    if (!lo && v != INT_MIN) atomicMax(e, v);
  }
}

// Drops the jobs marked before step ib from the active list (one workgroup;
// the order stays) and tells the host how many are left, and how many were
// lost so far (their end left its tile).
__global__ void __launch_bounds__(1024) tile_compact_kernel(const int* act, const int* n_act, const int* done,
                                                            const int* irr, int ib, int* act2, int* n_act2,
                                                            int* lost, int* host_n) {
  __shared__ int wave_n[16];
  __shared__ int total, gone;
  const int n = *n_act, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (threadIdx.x == 0) total = gone = 0;
  __syncthreads();
  for (int b = 0; b < n; b += 1024) {
    const int j = b + (int)threadIdx.x;
    int job = 0;
    bool keep = false;
    if (j < n) {
      job = act[j];
      keep = done[job] >= ib && (!irr || irr[job] >= ib);
      if (irr && irr[job] < ib && irr[job] < done[job]) atomicAdd(&gone, 1);
    }
    const unsigned long long bal = __ballot(keep);
    if (lane == 0) wave_n[wid] = (int)__popcll(bal);
    __syncthreads();
    int at = total;
    for (int x = 0; x < wid; ++x) at += wave_n[x];
    if (keep) act2[at + (int)__popcll(bal & ((1ull << lane) - 1))] = job;
    __syncthreads();
    if (threadIdx.x == 0)
      for (int x = 0; x < 16; ++x) total += wave_n[x];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *n_act2 = total;
    host_n[0] = total;
    if (irr) host_n[kTileHostLost] = *lost += gone;
  }
}

// Results of the jobs: completed at their end step; handed back where an end
// cell was lost before it, or where the records ran out.
template <class S>
__global__ void __launch_bounds__(256) tile_finish_kernel(TileFinishArgs a) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  unsigned long long ds = 0;
  unsigned retry = 0;
  if (j < a.n) {
    const int job = j, id = a.jobs[j].id;
    const int d = a.done[job], r = a.irr[job];
    const bool good = d != INT_MAX && r >= d;
    const int status = good ? (int)kDevCompleted : r != INT_MAX ? (int)kDevRingOverflow : (int)kDevArenaFull;
    if (good) {
      // the tabulated widths, corrected where an end was trimmed (the last
      // block run is the one of step d)
      long long sum = a.dsteps_upto[d + 1];
      if (a.stepped[job]) {
        sum = a.dsum[job] + step_width<S>(a.step_ends + ((long long)job * 4 + (d & 3)) * kStepEnds,
                                          a.flags + (long long)job * kStepFlags, d);
      } else if (d >= 0) {
        const int par = d / a.steps & 1;
        if (a.exact_lo[job]) sum -= a.dev[par][0][(long long)job * a.steps + d % a.steps];
        if (a.exact_hi[job]) sum += a.dev[par][1][(long long)job * a.steps + d % a.steps];
      }
      ds = (unsigned long long)sum;
    } else {
      retry = 1;
    }
    a.out_status[id] = status;
    a.out_score[id] = good ? (d + 1) * a.g : 0;
    a.out_dsteps[id] = (long long)ds;
    a.out_last_block[id] = kNoBlock;
    if (a.out_end_k) {
      a.out_end_k[id] = a.jobs[j].tlen - a.jobs[j].plen;
      a.out_end_off[id] = a.jobs[j].tlen;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    ds += __shfl_xor(ds, o, 64);
    retry += __shfl_xor(retry, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (ds) atomicAdd(a.dsteps_total, ds);
    if (retry) atomicAdd(a.retry_count, retry);
  }
}

// ------------------------------------------------------------- backtrace
// One wave per pair.  The walk needs one record byte per step of the path,
// and the place of every byte is known (block, row, diagonal): the wave loads
// a window of 64 rows x 16 diagonals at once, 16 bytes per lane, and walks
// inside it from LDS, so HBM latency is paid once per 64 score steps instead
// of once per step.  The replay extends with all 64 lanes (1,024 symbols at a
// time) from sequences in LDS.  Same two passes over the CIGAR slot as
// wfa_backtrace_kernel.
template <class S>
__global__ void __launch_bounds__(64) tile_backtrace_kernel(TileTraceArgs a) {
  constexpr int T = TileGeom<S>::T;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ __align__(16) uint32_t win[64 * 4];
  __shared__ int win_k[64];
  const int lane = threadIdx.x;
  const int job = (int)blockIdx.x;
  const TileJob jb = a.jobs[job];
  const int plen = jb.plen, tlen = jb.tlen, cap = plen + tlen;
  if (a.status[jb.id] != kDevCompleted) {
    if (lane == 0) a.ops_begin[jb.id] = cap;
    return;
  }
  unsigned char* out = reinterpret_cast<unsigned char*>(a.ops + a.ops_off[jb.id]);
  int i = a.score[jb.id] / a.g - 1;  // row of the end cell
  int k = tlen - plen, comp = kM, n = 0, nx = 0;
  bool mark = true, bad = false;
  int win_i = INT_MIN;             // row of lane 0's window line
  unsigned held = 0;               // this lane's operation of the current 64
  auto put = [&](unsigned op) {
    if (lane == (n & 63)) held = op;
    ++n;
    if ((n & 63) == 0) out[cap - n + 63 - lane] = (unsigned char)held;
  };
  while (i >= 0 && !bad) {
    if (n >= cap) { bad = true; break; }
    int l = win_i - i;
    bool in = win_i >= 0 && l < 64;
    if (in) {
      const int d = k - win_k[l];
      in = d >= 0 && d < 16;
    }
    if (!in) {
      wave_sync();
      const int r = i - lane;
      uint32_t v0 = 0, v1 = 0, v2 = 0, v3 = 0;
      int kk = INT_MAX / 2;
      if (r >= 0) {
        const int b = r / T;
        const int kb = a.blocks[b].kb, pitch = a.blocks[b].pitch;
        int off = ((k - 7) & ~3) - kb;
        off = max(0, min(off, pitch - 16));
        kk = kb + off;
        const uint8_t* p = reinterpret_cast<const uint8_t*>(a.rec + a.rec_tab[(long long)job * a.tab_stride + b]) +
                           (long long)(r - b * T) * pitch + off;
        const uint32_t* p32 = reinterpret_cast<const uint32_t*>(p);
        v0 = p32[0]; v1 = p32[1]; v2 = p32[2]; v3 = p32[3];
      }
      win[lane * 4] = v0; win[lane * 4 + 1] = v1; win[lane * 4 + 2] = v2; win[lane * 4 + 3] = v3;
      win_k[lane] = kk;
      wave_sync();
      win_i = i;
      l = 0;
      const int d = k - win_k[0];
      if (d < 0 || d >= 16) { bad = true; break; }
    }
    const unsigned byte = uniform((int)reinterpret_cast<const uint8_t*>(win)[l * 16 + (k - win_k[l])]);
    if (comp == kM) {
      const int src = S::NC == 5 ? (int)(byte >> 1) & 7 : (int)(byte >> 1) & 3;
      if (src == S::kTagX) {
        put('X' | (mark ? 0x80u : 0u));
        ++nx;
        i -= S::DX;
        mark = true;
        continue;
      }
      if (S::NC == 5 && src == S::kTagD2) comp = kD2;
      else if (src == S::kTagD1) comp = kD1;
      else if (S::NC == 5 && src == S::kTagI2) comp = kI2;
      else comp = kI1;
    }
    const bool ins = comp == kI1 || comp == kI2, one = comp == kI1 || comp == kD1;
    const int bit = (S::NC == 5 ? 4 : 6) + (one ? 0 : 2) + (ins ? 0 : 1);
    put((ins ? 'I' : 'D') | (mark ? 0x80u : 0u));
    k += ins ? -1 : 1;
    if ((byte >> bit) & 1u) {
      i -= one ? S::DE1 : S::DE2;
      mark = false;
    } else {
      i -= one ? S::DO1 : S::DO2;
      comp = kM;
      mark = true;
    }
  }
  if ((n & 63) != 0 && lane < (n & 63)) out[cap - (n & ~63) - 1 - lane] = (unsigned char)held;
  if (!bad && (i != -1 || comp != kM || k != 0)) bad = true;
  // 2M + 2X + I + D = plen + tlen gives the matches and the CIGAR's start
  const int pos = cap - n;
  const int rest = cap - 2 * nx - (n - nx);
  if (rest < 0 || (rest & 1)) bad = true;
  const int start = bad ? cap : pos - rest / 2;
  if (!bad) {
    const long long ppos = jb.ppos, tpos = jb.tpos;
    const uint32_t* P = reinterpret_cast<const uint32_t*>(a.words + (ppos >> 5));
    const uint32_t* Q = reinterpret_cast<const uint32_t*>(a.words + (tpos >> 5));
    const unsigned pbit = 2u * (unsigned)(ppos & 31), tbit = 2u * (unsigned)(tpos & 31);
    uint32_t* sP = reinterpret_cast<uint32_t*>(smem);
    uint32_t* sT = sP + 2 * a.lmax_words;
    const int nwp = (((int)(ppos & 31) + plen) / 32 + 2) * 2, nwt = (((int)(tpos & 31) + tlen) / 32 + 2) * 2;
    for (int x = lane; x < nwp; x += 64) sP[x] = P[x];
    for (int x = lane; x < nwt; x += 64) sT[x] = Q[x];
    __threadfence_block();  // the walk's operations, before other lanes read them
    wave_sync();
    int v = 0, h = 0, w = start;
    auto extend = [&]() {
      for (;;) {
        const int rem = min(plen - v, tlen - h);
        const int at = min(16 * lane, rem);
        const WaveSeqs<2> q{sP, sT, pbit, tbit, plen, tlen};
        const int m1 = q.run(h + at, v + at, rem - at);
        const unsigned long long stop = __ballot(m1 < 16);
        const int f = stop ? (int)__builtin_ctzll(stop) : 0;
        const int m = stop ? 16 * f + lane_of(m1, f) : 1024;
        if (w + m > cap) { bad = true; return; }
        for (int x2 = lane; x2 < m; x2 += 64) out[w + x2] = 'M';
        w += m;
        v += m;
        h += m;
        if (stop) return;
      }
    };
    extend();
    for (int b = pos; b < cap && !bad; b += 64) {
      const int mine = b + lane < cap ? (int)out[b + lane] : 0;
      const int cnt = min(64, cap - b);
      for (int x = 0; x < cnt && !bad; ++x) {
        const int op = lane_of(mine, x);
        if (w > b + x) { bad = true; break; }
        if (lane == 0) out[w] = (unsigned char)(op & 0x7F);
        ++w;
        const int c = op & 0x7F;
        if (c != 'D') ++h;
        if (c != 'I') ++v;
        if (op & 0x80) extend();
      }
    }
    if (!bad && (v != plen || h != tlen || w != cap)) bad = true;
  }
  if (lane == 0) {
    if (bad) {
      a.status[jb.id] = kDevBadTrace;
      atomicAdd(a.fail_count, 1u);
    }
    a.ops_begin[jb.id] = bad ? cap : start;
  }
}

// ------------------------------------------------------------------ BiWFA
// A side's sub-sequences (see setup_sides of the breakpoint kernels).
struct BiSide {
  long long ppos, tpos;
  const uint64_t* words;
  int plen, tlen, begin, end;
};
__device__ __forceinline__ BiSide bi_side(const BiTileArgs& a, int prob, int side) {
  const BiProblem pr = a.probs[prob];
  BiSide s;
  s.plen = pr.pe - pr.pb;
  s.tlen = pr.te - pr.tb;
  if (side == 0) {
    s.words = a.words;
    s.ppos = a.fwd_ppos[pr.pair] + pr.pb;
    s.tpos = a.fwd_tpos[pr.pair] + pr.tb;
    s.begin = pr.comp_begin;
    s.end = pr.comp_end;
  } else {
    s.words = a.rev_words;
    s.ppos = a.rev_ppos[pr.pair] + (a.plen_total[pr.pair] - pr.pe);
    s.tpos = a.rev_tpos[pr.pair] + (a.tlen_total[pr.pair] - pr.te);
    s.begin = pr.comp_end;
    s.end = pr.comp_begin;
  }
  return s;
}

// Steps per block, and the halo: 64 pairs of 20-60 kbp take 63.4 ms with 16,
// 60.3 with 24, 60.2 with 32 (and more for the breakpoint kernel to do again).
struct BiGeom {
  static constexpr int N = 4, T = 24, H = 24, U = 64 * N - 2 * H;
};

// One block of T steps of both sides of every active sub-problem, score only:
// blockIdx.y / 2 the sub-problem, blockIdx.y % 2 the side.  Nothing is trimmed
// here: an end cell that leaves the matrix ends the block's validity like a
// side that reaches its end or the sides' meeting, and the breakpoint kernel
// takes over from the rows at the block's start, which sit in the other half.
//
// Bound by the vector units and, while few tiles are alive, by the latency of
// a step: a launch costs 5.5 us for its loads and 0.85 us (one wave per SIMD) to 1.5 us
// (four) per step.  One workgroup or team per search instead pays a barrier
// and a trip to its ring in HBM per step, and the longest search decides: 64
// pairs of 20-60 kbp took 482 ms that way, 60 ms in tiles (40 ms here, 14 ms
// in the breakpoint kernel's last block and overlap scans).  Plain offsets
// instead of tagged ones, and the furthest antidiagonal taken only where it
// can be: 66.6 -> 63.8 ms, 24 steps a launch instead of 16: 60.3 ms.
__global__ void __launch_bounds__(64 * kTileWaves) bi_tile_kernel(BiTileArgs a) {
  using S = ScoreOnly<ShapeAffine>;
  constexpr int N = BiGeom::N, T = BiGeom::T, H = BiGeom::H, U = BiGeom::U;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int far_lds[kTileWaves];
  if ((int)blockIdx.y >= 2 * *a.n_act) return;
  const int prob = a.act[blockIdx.y >> 1], side = blockIdx.y & 1;
  if (a.done[prob] < a.blk) return;
  const int* far_in = a.far + ((a.blk & 1) ^ 1) * 2 * a.n + 2 * prob;
  int* far_out = a.far + (a.blk & 1) * 2 * a.n + 2 * prob;
  const BiSide sd = bi_side(a, prob, side);
  const int plen = sd.plen, tlen = sd.tlen;
  if (far_in[0] + far_in[1] >= plen + tlen - 1) {  // the sides met in the block before
    if (threadIdx.x == 0 && blockIdx.x == 0) atomicMin(a.done + prob, a.blk - 1);
    return;
  }
  const int ib = a.blk * T;
  const int2 hull = ib > 0 ? a.hull[sd.begin * a.steps + ib - 1] : make_int2(0, 0);
  const int left = (hull.x - T) & ~3, right = (hull.y + T + 4) & ~3;
  const int tiles = (right - left + U - 1) / U;
  if ((int)blockIdx.x * kTileWaves >= tiles) return;
  uint64_t* seqP = reinterpret_cast<uint64_t*>(smem);
  uint64_t* seqT = seqP + a.lmax_words;
  {
    const uint64_t* gP = sd.words + (sd.ppos >> 5);
    const uint64_t* gT = sd.words + (sd.tpos >> 5);
    const int nwp = ((int)(sd.ppos & 31) + plen) / 32 + 2, nwt = ((int)(sd.tpos & 31) + tlen) / 32 + 2;
    for (int i = threadIdx.x; i < nwp; i += 64 * kTileWaves) seqP[i] = gP[i];
    for (int i = threadIdx.x; i < nwt; i += 64 * kTileWaves) seqT[i] = gT[i];
    __syncthreads();
  }
  const int lane = threadIdx.x & 63, wid = uniform(threadIdx.x >> 6);
  const int tile = (int)blockIdx.x * kTileWaves + wid;
  int far = 0;
  if (tile < tiles) {
    const int quads = (right - left) / 4;
    const int first = left + 4 * (quads * tile / tiles), past = left + 4 * (quads * (tile + 1) / tiles);
    const WaveSeqs<2> q{reinterpret_cast<const uint32_t*>(seqP), reinterpret_cast<const uint32_t*>(seqT),
                        2u * (unsigned)(sd.ppos & 31), 2u * (unsigned)(sd.tpos & 31), plen, tlen};
    const int kt = first - H, k0 = kt + N * lane;
    const bool own = k0 >= first && k0 < past;
    const int kend = tlen - plen;
    const bool has_end = kend >= first && kend < past;
    const bool ends = tile == 0 || tile == tiles - 1;
    const int pitch = tile_pitch(plen, tlen);
    int* st = a.state + a.st_off[prob] + (long long)side * kBiTileRows * pitch + (k0 + tile_kpad(plen));
    const int pin = (a.blk & 1) ^ 1, pout = a.blk & 1;
    WaveRows<S, N> w;
#pragma unroll
    for (int r = 0; r < 4; ++r) load_row<N>(w.m[r], st + (long long)bi_row(pin, kM, 3 - r) * pitch);
    load_row<N>(w.i1[0], st + (long long)bi_row(pin, kI1, 0) * pitch);
    load_row<N>(w.d1[0], st + (long long)bi_row(pin, kD1, 0) * pitch);
    const int end_not_m = sd.end == kM ? 0 : INT_MIN, end_not_i1 = sd.end == kI1 ? 0 : INT_MIN,
              end_not_d1 = sd.end == kD1 ? 0 : INT_MIN;
    bool stop = false;
    auto one = [&](auto phc, int t) {
      constexpr int PH = decltype(phc)::value;
      StepCells<N> cell;
      for (uint32_t& r : cell.rec) r = 0;
      wave_step<S, N, PH, 2>(w, nullptr, k0, q, cell);
      // The furthest antidiagonal: along a diagonal M gains at least one cell
      // every DX steps, so the block's last DX steps have it, or a step with a
      // cell on a border (what a border cuts off lies behind such a cell).
      int rem = cell.rem[0];
#pragma unroll
      for (int c = 1; c < N; ++c) rem = min(rem, cell.rem[c]);
      if (t >= T - S::DX || __ballot(rem <= 0)) {
#pragma unroll
        for (int c = 0; c < N; ++c) far = (cell.ok[c] & own) ? max(far, 2 * cell.h[c] - (k0 + c)) : far;
      }
      if (ends) {
        bool out = false;
#pragma unroll
        for (int c = 0; c < N; ++c) out |= cell.oob[c] & own;
        stop |= __ballot(out) != 0;
      }
      if (has_end) {
        bool fin = false;
#pragma unroll
        for (int c = 0; c < N; ++c) {
          // (masks, not a choice between the rows: that would put the rows in scratch memory)
          const int g = max(max(w.m[PH % S::RM][c] | end_not_m, w.i1[0][c] | end_not_i1), w.d1[0][c] | end_not_d1);
          fin |= (k0 + c == kend) & ((g >> S::SH) >= tlen);
        }
        stop |= __ballot(fin) != 0;
      }
      if (t >= T - kBiTileAges && own) {
        store_row<N>(st + (long long)bi_row(pout, kM, T - 1 - t) * pitch, w.m[PH % S::RM]);
        store_row<N>(st + (long long)bi_row(pout, kI1, T - 1 - t) * pitch, w.i1[0]);
        store_row<N>(st + (long long)bi_row(pout, kD1, T - 1 - t) * pitch, w.d1[0]);
      }
    };
    static_assert(T % 4 == 0 && S::RM == 4 && S::DE1 == 1, "rows of a block");
    for (int t = 0; t < T; t += 4) {
      one(std::integral_constant<int, 0>{}, t);
      one(std::integral_constant<int, 1>{}, t + 1);
      one(std::integral_constant<int, 2>{}, t + 2);
      one(std::integral_constant<int, 3>{}, t + 3);
    }
    if (stop && lane == 0) atomicMin(a.done + prob, a.blk);
    for (int o = 32; o > 0; o >>= 1) far = max(far, __shfl_xor(far, o, 64));
  }
  if (lane == 0) far_lds[wid] = far;
  __syncthreads();
  if (threadIdx.x == 0) {
    int f = far_in[side];
    for (int x = 0; x < kTileWaves; ++x) f = max(f, far_lds[x]);
    atomicMax(far_out + side, f);
  }
}

// Score 0 of both sides, and the first active list.
__global__ void __launch_bounds__(64) bi_tile_init_kernel(BiTileArgs a, int* act, int* n_act) {
  const int x = blockIdx.x * 64 + threadIdx.x;
  if (x == 0) *n_act = a.n;
  if (x >= 2 * a.n) return;
  const int prob = x >> 1, side = x & 1;
  if (side == 0) {
    act[prob] = prob;
    a.done[prob] = INT_MAX;
  }
  const BiSide sd = bi_side(a, prob, side);
  const int pitch = tile_pitch(sd.plen, sd.tlen);
  int h = 0;
  if (sd.begin == kM)
    h = lcp_extend<2>(sd.words + (sd.ppos >> 5), (int)(sd.ppos & 31), sd.words + (sd.tpos >> 5), (int)(sd.tpos & 31),
                      sd.plen, sd.tlen, 0, 0);
  a.state[a.st_off[prob] + ((long long)side * kBiTileRows + bi_row(1, sd.begin, 0)) * pitch + tile_kpad(sd.plen)] =
      h;
  // (an end reached at score 0: found again by the breakpoint kernel)
  const bool end0 = sd.begin == kM && sd.end == kM && sd.plen == sd.tlen && h >= sd.tlen;
  a.far[2 * prob + side] = a.far[2 * a.n + 2 * prob + side] = end0 ? sd.plen + sd.tlen : 2 * h;
}

template <class S>
bool shape_matches(const Penalties& p) {
  if (p.g <= 0 || p.ncomp != S::NC) return false;
  const bool one = p.x == S::DX * p.g && p.o1 + p.e1 == S::DO1 * p.g && p.e1 == S::DE1 * p.g;
  return one && (S::NC != 5 || (p.o2 + p.e2 == S::DO2 * p.g && p.e2 == S::DE2 * p.g));
}

template <class S>
TileGeometry geometry() {
  using G = TileGeom<S>;
  TileGeometry t;
  t.steps = G::T;
  t.useful = tile_useful<S>();
  t.state_rows = G::MS + 2 * S::kGapRows;
  t.step_rows = StepRows<S>::ROWS;
  t.dx = S::DX; t.do1 = S::DO1; t.de1 = S::DE1;
  t.do2 = S::NC == 5 ? S::DO2 : 0; t.de2 = S::NC == 5 ? S::DE2 : 0;
  return t;
}

}  // namespace

int tile_shape(const Penalties& pen) {
  if (shape_matches<Shape2p>(pen)) return 2;
  if (shape_matches<ShapeAffine>(pen)) return 1;
  return 0;
}

TileGeometry tile_geometry(int shape) { return shape == 2 ? geometry<Shape2p>() : geometry<ShapeAffine>(); }

int bi_tile_steps() { return BiGeom::T; }
int bi_tile_useful() { return BiGeom::U; }

hipError_t launch_bi_tile_init(const BiTileArgs& a, int* act, int* n_act, hipStream_t st) {
  hipLaunchKernelGGL(bi_tile_init_kernel, dim3((2 * a.n + 63) / 64), dim3(64), 0, st, a, act, n_act);
  return hipGetLastError();
}

hipError_t launch_bi_tile_block(const BiTileArgs& a, int problems, int tiles, hipStream_t st) {
  const size_t lds = (size_t)2 * a.lmax_words * sizeof(uint64_t);
  const dim3 grid((tiles + kTileWaves - 1) / kTileWaves, 2 * problems);
  hipLaunchKernelGGL(bi_tile_kernel, grid, dim3(64 * kTileWaves), lds, st, a);
  return hipGetLastError();
}

hipError_t launch_tile_fill(int* state, long long ints, hipStream_t st) {
  const long long n4 = ints / 4;
  if (n4 <= 0) return hipSuccess;
  const int grid = (int)std::min<long long>((n4 + 255) / 256, 4096);
  hipLaunchKernelGGL(tile_fill_kernel, dim3(grid), dim3(256), 0, st, reinterpret_cast<int4*>(state), n4);
  return hipGetLastError();
}

hipError_t launch_tile_init(int shape, const TileArgs& a, int n, const TileSlot* slots, const TileSeqs& seqs, int* act,
                            int* n_act, int* lost, hipStream_t st) {
  const dim3 grid((n + 63) / 64), block(64);
  if (shape == 2) hipLaunchKernelGGL(tile_init_kernel<Shape2p>, grid, block, 0, st, a, n, slots, seqs, act, n_act, lost);
  else hipLaunchKernelGGL(tile_init_kernel<ShapeAffine>, grid, block, 0, st, a, n, slots, seqs, act, n_act, lost);
  return hipGetLastError();
}

hipError_t launch_tile_block(int shape, bool records, const TileArgs& a, int jobs, hipStream_t st) {
  const dim3 grid((a.tiles + kTileWaves - 1) / kTileWaves, jobs), block(64 * kTileWaves);
  const size_t lds = (size_t)2 * a.lmax_words * sizeof(uint64_t);
  if (shape == 2) {
    if (records) hipLaunchKernelGGL((wfa_tile_kernel<Shape2p, true>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((wfa_tile_kernel<Shape2p, false>), grid, block, lds, st, a);
  } else {
    if (records) hipLaunchKernelGGL((wfa_tile_kernel<ShapeAffine, true>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((wfa_tile_kernel<ShapeAffine, false>), grid, block, lds, st, a);
  }
  return hipGetLastError();
}

hipError_t launch_tile_step_init(int shape, const StepArgs& a, const TileArgs& t, int n, int max_pitch, hipStream_t st) {
  const dim3 grid((max_pitch + 255) / 256, n);
  hipLaunchKernelGGL(tile_step_flags_kernel, dim3((n * kStepFlags + 63) / 64), dim3(64), 0, st, a.act, n, a.flags);
  if (shape == 2) hipLaunchKernelGGL(tile_step_init_kernel<Shape2p>, grid, dim3(256), 0, st, a, t);
  else hipLaunchKernelGGL(tile_step_init_kernel<ShapeAffine>, grid, dim3(256), 0, st, a, t);
  hipLaunchKernelGGL(tile_step_mark_kernel, dim3((n + 63) / 64), dim3(64), 0, st, a.act, n, t.irr, t.stepped);
  return hipGetLastError();
}

hipError_t launch_tile_step(int shape, bool records, const StepArgs& a, int t, int jobs, int max_width, hipStream_t st) {
  const dim3 grid((max_width + 8 + kStepWaves * 248 - 1) / (kStepWaves * 248), jobs), block(64 * kStepWaves);
  if (shape == 2) {
    if (records) hipLaunchKernelGGL((tile_step_kernel<Shape2p, true>), grid, block, 0, st, a, t);
    else hipLaunchKernelGGL((tile_step_kernel<Shape2p, false>), grid, block, 0, st, a, t);
  } else {
    if (records) hipLaunchKernelGGL((tile_step_kernel<ShapeAffine, true>), grid, block, 0, st, a, t);
    else hipLaunchKernelGGL((tile_step_kernel<ShapeAffine, false>), grid, block, 0, st, a, t);
  }
  return hipGetLastError();
}

hipError_t launch_tile_compact(const int* act, const int* n_act, const int* done, const int* irr, int ib, int* act2,
                               int* n_act2, int* lost, int* host_n, hipStream_t st) {
  hipLaunchKernelGGL(tile_compact_kernel, dim3(1), dim3(1024), 0, st, act, n_act, done, irr, ib, act2, n_act2, lost, host_n);
  return hipGetLastError();
}

hipError_t launch_tile_finish(int shape, const TileFinishArgs& a, hipStream_t st) {
  if (shape == 2) hipLaunchKernelGGL(tile_finish_kernel<Shape2p>, dim3((a.n + 255) / 256), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(tile_finish_kernel<ShapeAffine>, dim3((a.n + 255) / 256), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_tile_backtrace(int shape, const TileTraceArgs& a, int n, hipStream_t st) {
  const size_t lds = (size_t)2 * a.lmax_words * sizeof(uint64_t);
  if (shape == 2) hipLaunchKernelGGL((tile_backtrace_kernel<Shape2p>), dim3(n), dim3(64), lds, st, a);
  else hipLaunchKernelGGL((tile_backtrace_kernel<ShapeAffine>), dim3(n), dim3(64), lds, st, a);
  return hipGetLastError();
}

}  // namespace wfa
