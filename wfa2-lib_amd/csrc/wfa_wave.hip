// Short pairs: one wave per pair, its wavefronts in registers.
//
// A pair's diagonals are spread over the 64 lanes of one wave, N neighbours
// per lane (wfa_rows.h), with the score-0 diagonals in the middle.  Rows of
// the last steps sit in registers (moved along at each step), a gap source is a
// neighbouring register or a DPP shift,
// and LDS holds nothing but the two packed sequences: the step has no ring,
// no clamped index, no per-source range and no LDS round trip but the
// extension's.  N starts at the least that holds the score-0 diagonals and
// doubles as the wavefront outgrows the wave (1 up to 64 diagonals, then 2, 4,
// 8); the step at which it does is the same for every pair.
//
// Ranges need no bookkeeping either: until a cell leaves the matrix nothing
// is trimmed (wavefront_compute.c:579-613) and the widths are tabulated; after
// that the limits are read off the cells, as in the end tiles of wfa_tile.hip.
//
// Records: a word per lane holds four cells (of one step, or of 4 / N
// consecutive ones), so a wave writes 256 contiguous bytes per four cells of
// its lanes, and the place of every record byte follows from the step and the
// diagonal: the backtrace reads no headers.
#include <climits>

#include "wfa_rows.h"
#include "wfa_wave.h"

namespace wfa {
namespace {

// One copy of a shape's table in device memory, one for the host.
template <class S>
__device__ const WaveTable wave_table = make_wave_table<S>();
template <class S>
constexpr WaveTable host_wave_table = make_wave_table<S>();

// Everything of one pair that outlives a step.
struct WavePair {
  int plen, tlen, kend;
  int i;            // steps done: the last row is i - 1
  int status;       // 1: running
  int dev;          // exact minus tabulated widths
  int slot;         // ring row about to be written (a second gap)
  bool exact;
  uint32_t hist_m, hist_gap;  // exact: components with a valid cell in the last steps (WaveTable)
  int end_k, end_off;
  uint32_t base[kWavePhases];  // record units of each phase
};

// With a second gap the M rows of the last 25 steps are needed: they sit in
// LDS, 16 bits a cell (offset << 4; at most 1,024 symbols), a row holding the
// diagonals of the widest phase in order, so that a phase reads and writes
// its lanes' cells in one access each and a change of phase moves nothing.
constexpr int kRingRows = 26;
constexpr int kRingNull = -32768;
template <int NMAX>
struct WaveRing {
  int16_t* rows;
  static constexpr int kPitch = 64 * NMAX;
  static constexpr int kBytes = kRingRows * kPitch * 2;
  __device__ __forceinline__ void clear() const {
    const uint32_t v = 0x80008000u;
    for (int x = threadIdx.x & 63; x < kBytes / 16; x += 64) reinterpret_cast<uint4*>(rows)[x] = make_uint4(v, v, v, v);
  }
  // the lane's N cells of the row `back` steps ago (at: this lane's first
  // cell in a row; slot: the row about to be written)
  template <int N>
  __device__ __forceinline__ void read(int* r, int at, int slot, int back) const {
    int x = slot - back;
    if (x < 0) x += kRingRows;
    const int16_t* p = rows + x * kPitch + at;
    if constexpr (N == 1) {
      r[0] = p[0];
    } else {
#pragma unroll
      for (int c = 0; c < N; c += 2) {
        const int v = *reinterpret_cast<const int*>(p + c);
        r[c] = (int)(int16_t)v;
        r[c + 1] = v >> 16;
      }
    }
  }
  template <int N>
  __device__ __forceinline__ void write(const int* m, int at, int slot) const {
    int16_t* p = rows + slot * kPitch + at;
    if constexpr (N == 1) {
      p[0] = (int16_t)max(m[0], kRingNull);
    } else {
#pragma unroll
      for (int c = 0; c < N; c += 2)
        *reinterpret_cast<uint32_t*>(p + c) =
            ((uint32_t)max(m[c], kRingNull) & 0xFFFFu) | ((uint32_t)max(m[c + 1], kRingNull) << 16);
    }
  }
};

struct WaveChunk {  // record chunk of this wave (16-byte units)
  uint32_t cur, end, begin;
  // The records written since `from` (a copy of this) go back: those of a pair
  // that does not finish here.  Where the pair took a new chunk, all of that.
  __device__ __forceinline__ void give_back(const WaveChunk& from) { cur = begin == from.begin ? from.cur : begin; }
};

// Room for `units` of records in the wave's chunk, or a new chunk (twice as
// large where the last phase alone may fill one: what is left of a chunk when
// the next phase does not fit is lost).
template <int NMAX>
__device__ __forceinline__ bool reserve_records(WaveChunk& ch, uint32_t units) {
  if (ch.cur + units <= ch.end) return true;
  KernArgs A = args_now();
  constexpr uint32_t chunk = NMAX == 8 ? 2 * kChunkUnits : kChunkUnits;
  const uint32_t want = units > chunk ? units : chunk;
  unsigned long long b = 0;
  if ((threadIdx.x & 63) == 0) b = atomicAdd(A->rec_top, (unsigned long long)want);
  const unsigned blo = (unsigned)lane_of((int)(unsigned)(b & 0xFFFFFFFFull), 0);
  const unsigned bhi = (unsigned)lane_of((int)(unsigned)(b >> 32), 0);
  if (bhi != 0 || (unsigned long long)blo + want > A->rec_units) return false;
  ch.cur = ch.begin = blo;
  ch.end = blo + want;
  return true;
}

// The steps of one phase (N diagonals per lane): from row p.i up to the last
// step whose wavefront fits, or the end of the pair.
template <class S, int N, int NMAX, int BITS, bool REC, bool EF>
__device__ __forceinline__ void wave_phase(WavePair& p, WaveChunk& ch, WaveRows<S, N>& w, const WaveSeqs<BITS>& q,
                                           const WaveRing<NMAX>& ring) {
  KernArgs A = args_now();
  static_assert(S::DE1 <= 2 && S::DE2 == 1 && S::DO2 < kRingRows, "gap rows");
  constexpr int PH = N == 1 ? 0 : N == 2 ? 1 : N == 4 ? 2 : 3;
  constexpr int G = N < 4 ? 4 / N : 1;  // steps per record word
  const int lane = threadIdx.x & 63;
  const int kt = (EF ? A->wave.center : 0) - 32 * N, k0 = kt + N * lane;
  const int first = PH ? A->wave.last[PH ? PH - 1 : 0] : 0, last = A->wave.last[PH];
  const int pef = EF ? A->pef : 0, tef = EF ? A->tef : 0;
  uint32_t* rec = nullptr;
  if constexpr (REC) {
    const uint32_t units = (uint32_t)((last - first + G - 1) / G * (N > 4 ? N / 4 : 1)) * 16u;
    if (!reserve_records<NMAX>(ch, units)) {
      p.status = kDevArenaFull;
      return;
    }
    p.base[PH] = ch.cur;
    rec = reinterpret_cast<uint32_t*>(A->rec_arena + ch.cur) + lane;
  }
  uint32_t endm = 0;  // the lane's cell on the end diagonal
#pragma unroll
  for (int c = 0; c < N; ++c) endm |= (k0 + c == p.kend) ? 1u << c : 0u;
  StepCells<N> cell;
#pragma unroll
  for (uint32_t& r : cell.rec) r = 0;
  int i = p.i;
  while (i < last) {
    // w.m[r]: row i - 1 - r, and so the gap rows (of the last DE1 steps)
    int m[N];
    constexpr int og = S::DE1 - 1;
    if constexpr (S::NC == 5) {
      int mx[N], mo[N], mo2[N];
      const int at = k0 - (kt - 32 * (NMAX - N));
      ring.template read<N>(mx, at, p.slot, S::DX);
      ring.template read<N>(mo, at, p.slot, S::DO1);
      ring.template read<N>(mo2, at, p.slot, S::DO2);
      wave_cells<S, N, BITS>(mx, mo, w.i1[og], w.d1[og], mo2, w.i2[0], w.d2[0], m, k0, q, cell);
      ring.template write<N>(m, at, p.slot);
      p.slot = p.slot + 1 == kRingRows ? 0 : p.slot + 1;
    } else {
      wave_cells<S, N, BITS>(w.m[S::kMismatch ? S::DX - 1 : 0], w.m[S::DO1 - 1], w.i1[og], w.d1[og], nullptr, nullptr,
                             nullptr, m, k0, q, cell);
#pragma unroll
      for (int r = S::RM - 1; r > 0; --r)
#pragma unroll
        for (int c = 0; c < N; ++c) w.m[r][c] = w.m[r - 1][c];
#pragma unroll
      for (int c = 0; c < N; ++c) w.m[0][c] = m[c];
    }
    if constexpr (S::NC > 1 && S::DE1 == 2) {
#pragma unroll
      for (int c = 0; c < N; ++c) {
        const int ni = w.i1[1][c], nd = w.d1[1][c];
        w.i1[1][c] = w.i1[0][c];
        w.d1[1][c] = w.d1[0][c];
        w.i1[0][c] = ni;
        w.d1[0][c] = nd;
      }
    }
    ++i;
    if constexpr (REC) {
      if (G == 1 || ((i - first) & (G - 1)) == 0) {
#pragma unroll
        for (int c = 0; c < (N + 3) / 4; ++c) rec[64 * c] = cell.rec[c];
        rec += 64 * ((N + 3) / 4);
      }
    }
    bool out = false, fin = false;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      out |= cell.oob[c];
      if constexpr (EF) fin |= cell.ok[c] & endsfree_done(cell.h[c], k0 + c, p.plen, p.tlen, pef, tef);
      else fin |= cell.ok[c] & (cell.h[c] >= p.tlen) & (((endm >> c) & 1u) != 0);
    }
    const unsigned long long bfin = __ballot(fin);
    if (__ballot(out) || p.exact) {
      // limits and trimming from the cells
      KernArgs B = args_now();
      if (!p.exact) {
        p.exact = true;
        p.hist_m = wave_table<typename S::Slots>.hist_m[i - 1];
        p.hist_gap = wave_table<typename S::Slots>.hist_gap[i - 1];
      }
      uint32_t okm = 0, reach = 0;
#pragma unroll
      for (int c = 0; c < N; ++c) {
        okm |= cell.ok[c] ? 1u << c : 0u;
        reach |= (cell.ok[c] | cell.oob[c]) ? 1u << c : 0u;
      }
      int lo = first_diagonal<N>(reach, kt), hi = last_diagonal<N>(reach, kt);
      const bool some = lo <= hi;
      if (B->pen.metric > kEdit) {
        // a null source still contributes the limits (1, -1), shifted as its
        // gap moves it (wavefront_compute.c:40-86)
        auto null_m = [&](int back) { return !((p.hist_m >> (back - 1)) & 1u); };
        auto null_gap = [&](int c, int back) { return !((p.hist_gap >> (4 * (back - 1) + c - kI1)) & 1u); };
        if (null_m(S::DX > 0 ? S::DX : 1)) { lo = min(lo, 1); hi = max(hi, -1); }
        if (null_m(S::DO1)) { lo = min(lo, 0); hi = max(hi, 0); }
        if constexpr (S::NC > 1) {
          if (null_gap(kI1, S::DE1)) { lo = min(lo, 2); hi = max(hi, 0); }
          if (null_gap(kD1, S::DE1)) { lo = min(lo, 0); hi = max(hi, -2); }
        }
        if constexpr (S::NC == 5) {
          if (null_m(S::DO2)) { lo = min(lo, 0); hi = max(hi, 0); }
          if (null_gap(kI2, S::DE2)) { lo = min(lo, 2); hi = max(hi, 0); }
          if (null_gap(kD2, S::DE2)) { lo = min(lo, 0); hi = max(hi, -2); }
        }
      }
      const int tlo = wave_table<typename S::Slots>.lo[i - 1], thi = wave_table<typename S::Slots>.hi[i - 1];
      p.dev += (some ? hi - lo + 1 : 0) - (tlo <= thi ? thi - tlo + 1 + (EF ? B->pbf + B->tbf : 0) : 0);
      p.hist_m = (p.hist_m << 1) | (__ballot(okm != 0) ? 1u : 0u);
      p.hist_gap <<= 4;
      if constexpr (S::NC > 1) {
        auto trim = [&](int* g, int comp) {
          uint32_t vm = 0;
#pragma unroll
          for (int c = 0; c < N; ++c) vm |= in_bounds(g[c] >> S::SH, k0 + c, p.plen, p.tlen) ? 1u << c : 0u;
          const int f = first_diagonal<N>(vm, kt), l = last_diagonal<N>(vm, kt);
#pragma unroll
          for (int c = 0; c < N; ++c) g[c] = (k0 + c < f || k0 + c > l) ? kNullTagged : g[c];
          p.hist_gap |= f <= l ? 1u << (comp - kI1) : 0u;
        };
        trim(w.i1[0], kI1);
        trim(w.d1[0], kD1);
        if constexpr (S::NC == 5) {
          trim(w.i2[0], kI2);
          trim(w.d2[0], kD2);
        }
      }
    }
    if (bfin) {
      if constexpr (EF) {
        uint32_t fm = 0;
        int off = 0;
#pragma unroll
        for (int c = N - 1; c >= 0; --c) {
          const bool f = cell.ok[c] & endsfree_done(cell.h[c], k0 + c, p.plen, p.tlen, pef, tef);
          fm |= f ? 1u << c : 0u;
          off = f ? cell.h[c] : off;
        }
        p.end_k = first_diagonal<N>(fm, kt);
        p.end_off = lane_of(off, (int)__builtin_ctzll(bfin));
      }
      p.status = kDevCompleted;
      break;
    }
  }
  if constexpr (REC && G > 1) {
    // the started record word, its steps moved down to their places
    const int rest = (i - first) & (G - 1);
    if (rest) rec[0] = cell.rec[0] >> (8 * N * (G - rest));
  }
  p.i = i;
  if constexpr (REC) ch.cur = p.base[PH] + (uint32_t)((i - first + G - 1) / G * (N > 4 ? N / 4 : 1)) * 16u;
}

// Rows of N diagonals per lane spread over 2N per lane: the lane's first N
// come from lane 2l - 32, its last N from lane 2l - 31.
template <class S, int N>
__device__ __forceinline__ void widen(const WaveRows<S, N>& w, WaveRows<S, 2 * N>& x) {
  const int lane = threadIdx.x & 63;
  const bool in = lane >= 16 && lane < 48;
  const int from = 4 * (2 * lane - 32);
  auto spread = [&](const int* a, int* b) {
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const int u = __builtin_amdgcn_ds_bpermute(from, a[c]), v = __builtin_amdgcn_ds_bpermute(from + 4, a[c]);
      b[c] = in ? u : kNullTagged;
      b[N + c] = in ? v : kNullTagged;
    }
  };
  if constexpr (S::NC < 5) {
#pragma unroll
    for (int r = 0; r < S::RM; ++r) spread(w.m[r], x.m[r]);
  } else {
    spread(w.i2[0], x.i2[0]);
    spread(w.d2[0], x.d2[0]);
  }
  if constexpr (S::NC > 1) {
#pragma unroll
    for (int r = 0; r < S::DE1; ++r) {
      spread(w.i1[r], x.i1[r]);
      spread(w.d1[r], x.d1[r]);
    }
  }
}

// Row -1 (score 0): offset 0 at diagonal 0, or, ends-free, the free
// beginnings (wavefront_aligner.c:252-307), each extended; every other row
// NULL.  Returns whether the alignment ends there.
template <class S, int N, int NMAX, int BITS, bool EF>
__device__ __forceinline__ bool wave_start(WavePair& p, WaveRows<S, N>& w, const WaveSeqs<BITS>& q,
                                           const WaveRing<NMAX>& ring) {
  KernArgs A = args_now();
  const int lane = threadIdx.x & 63;
  const int kt = (EF ? A->wave.center : 0) - 32 * N, k0 = kt + N * lane;
#pragma unroll
  for (int r = 0; r < S::RM; ++r)
#pragma unroll
    for (int c = 0; c < N; ++c) w.m[r][c] = kNullTagged;
  if constexpr (S::NC > 1) {
#pragma unroll
    for (int r = 0; r < S::DE1; ++r)
#pragma unroll
      for (int c = 0; c < N; ++c) w.i1[r][c] = w.d1[r][c] = kNullTagged;
  }
  if constexpr (S::NC == 5) {
#pragma unroll
    for (int c = 0; c < N; ++c) w.i2[0][c] = w.d2[0][c] = kNullTagged;
    ring.clear();
    wave_sync();
  }
  int m0[N];
  const int lo = EF ? -A->pbf : 0, hi = EF ? A->tbf : 0;
  uint32_t done = 0;
  int off = 0;
#pragma unroll
  for (int c = N - 1; c >= 0; --c) {
    const int k = k0 + c;
    int h = k > 0 ? k : 0;
    bool more = k >= lo && k <= hi;
    const bool on = more;
    while (more) {
      const int r = min(p.tlen - h, p.plen - (h - k));
      const int n = r > 0 ? q.run(h, h - k, r) : 0;
      h += n;
      more = (n == WaveSeqs<BITS>::kSpan) & (r > n);
    }
    m0[c] = on ? h << S::SH : kNullTagged;
    const bool fin = on && (EF ? endsfree_done(h, k, p.plen, p.tlen, A->pef, A->tef) : (k == p.kend && h >= p.tlen));
    done |= fin ? 1u << c : 0u;
    off = fin ? h : off;
  }
  if constexpr (S::NC == 5) {
    ring.template write<N>(m0, k0 - (kt - 32 * (NMAX - N)), 0);
    p.slot = 1;
  } else {
#pragma unroll
    for (int c = 0; c < N; ++c) w.m[0][c] = m0[c];
  }
  const unsigned long long b = __ballot(done != 0);
  if (b) {
    p.end_k = first_diagonal<N>(done, kt);
    p.end_off = lane_of(off, (int)__builtin_ctzll(b));
  }
  return b != 0;
}

// The 2-bit sequences of pair id into LDS.
__device__ __forceinline__ void stage_sequences(WaveSeqs<2>& q, KernArgs A, int id, uint32_t* seqP, uint32_t* seqT) {
  const int lane = threadIdx.x & 63;
  const long long ppos = A->pat_pos[id], tpos = A->txt_pos[id];
  q.pbit = 2u * (unsigned)(ppos & 31);
  q.tbit = 2u * (unsigned)(tpos & 31);
  const uint64_t* gP = A->words + (ppos >> 5);
  const uint64_t* gT = A->words + (tpos >> 5);
  const int nwp = ((int)(ppos & 31) + q.plen) / 32 + 2, nwt = ((int)(tpos & 31) + q.tlen) / 32 + 2;
  uint64_t* dP = reinterpret_cast<uint64_t*>(seqP);
  uint64_t* dT = reinterpret_cast<uint64_t*>(seqT);
  for (int x = lane; x < nwp; x += 64) dP[x] = gP[x];
  for (int x = lane; x < nwt; x += 64) dT[x] = gT[x];
}

// NMAX: most diagonals per lane (4: pairs up to 254 diagonals, 8: 510).
// SRC: bits per symbol of the packed sequences in memory.  8-bit symbols that
// differ in their low four bits are kept as 4-bit ones in LDS.
template <class S, int NMAX, int SRC, bool REC, bool EF>
__global__ void __launch_bounds__(64, S::NC == 5 ? (NMAX == 8 ? 2 : 3) : (NMAX == 8 ? 3 : 5)) wfa_wave_kernel(ForwardArgs a) {
  constexpr int BITS = SRC == 2 ? 2 : 4;
  extern __shared__ __align__(16) unsigned char smem[];
  uint32_t* seqP = reinterpret_cast<uint32_t*>(smem);
  uint32_t* seqT = seqP + a.wave.lds_words;
  __shared__ __align__(16) int16_t ring_lds[S::NC == 5 ? WaveRing<NMAX>::kBytes / 2 : 8];
  const WaveRing<NMAX> ring{ring_lds};
  const int lane = threadIdx.x;
  WaveChunk ch{0, 0, 0};
  unsigned long long wg_dsteps = 0;
  bool q_first = true;
  for (;;) {
    KernArgs A = args_now();
    int qv = 0;
    if (!q_first && lane == 0) qv = (int)atomicAdd(work_queue(A->queue, A->queues), 1u);
    const int qi = work_item(A->queues, q_first, lane_of(qv, 0));
    q_first = false;
    if (qi >= (A->n_over ? uniform((int)*A->n_over) : A->n_pairs)) break;
    const int id = A->order ? A->order[qi] : qi;
    WavePair p;
    p.plen = A->plen[id];
    p.tlen = A->tlen[id];
    p.kend = p.tlen - p.plen;
    p.i = 0;
    p.status = 1;
    p.dev = 0;
    p.exact = false;
    p.slot = 0;
    p.hist_m = p.hist_gap = 0;
    p.end_k = p.kend;
    p.end_off = p.tlen;
    for (int x = 0; x < kWavePhases; ++x) p.base[x] = 0;
    WaveSeqs<BITS> q{seqP, seqT, 0u, 0u, p.plen, p.tlen};
    wave_sync();  // the previous pair is done reading the sequences
    if constexpr (SRC == 2) {
      stage_sequences(q, A, id, seqP, seqT);
    } else {
      const long long ppos = A->pat_pos[id], tpos = A->txt_pos[id];
      q.pbit = 4u * (unsigned)(ppos & 7);
      q.tbit = 4u * (unsigned)(tpos & 7);
      // eight bytes to eight nibbles
      auto squeeze = [](uint64_t v) {
        v &= 0x0F0F0F0F0F0F0F0Full;
        v = (v | (v >> 4)) & 0x00FF00FF00FF00FFull;
        v = (v | (v >> 8)) & 0x0000FFFF0000FFFFull;
        return (uint32_t)(v | (v >> 16));
      };
      const uint64_t* gP = A->words + (ppos >> 3);
      const uint64_t* gT = A->words + (tpos >> 3);
      const int nwp = ((int)(ppos & 7) + p.plen) / 8 + 2, nwt = ((int)(tpos & 7) + p.tlen) / 8 + 2;
      for (int x = lane; x < nwp; x += 64) seqP[x] = squeeze(gP[x]);
      for (int x = lane; x < nwt; x += 64) seqT[x] = squeeze(gT[x]);
    }
    wave_sync();
    uint32_t header = kNoBlock;
    const WaveChunk before = ch;
    if constexpr (REC) {
      // the pair's header: the units of its phases' records
      if (reserve_records<NMAX>(ch, 1)) header = ch.cur++;
      else p.status = kDevArenaFull;
    }
    // phases: rows of 1, 2, 4 (and 8) diagonals per lane in turn
    WaveRows<S, 1> w1;
    WaveRows<S, 2> w2;
    WaveRows<S, 4> w4;
    const int phase0 = EF ? A->wave.phase0 : 0;
    bool ended = false;
    if (p.status == 1) {
      if (phase0 == 0) ended = wave_start<S, 1, NMAX, BITS, EF>(p, w1, q, ring);
      else if (phase0 == 1) ended = wave_start<S, 2, NMAX, BITS, EF>(p, w2, q, ring);
      else ended = wave_start<S, 4, NMAX, BITS, EF>(p, w4, q, ring);
      if (ended) p.status = kDevCompleted;
    }
    if (p.status == 1 && phase0 == 0) {
      wave_phase<S, 1, NMAX, BITS, REC, EF>(p, ch, w1, q, ring);
      if (p.status == 1) widen<S, 1>(w1, w2);
    }
    if (p.status == 1 && phase0 <= 1) {
      wave_phase<S, 2, NMAX, BITS, REC, EF>(p, ch, w2, q, ring);
      if (p.status == 1) widen<S, 2>(w2, w4);
    }
    if (p.status == 1) wave_phase<S, 4, NMAX, BITS, REC, EF>(p, ch, w4, q, ring);
    if constexpr (NMAX >= 8) {
      if (p.status == 1) {
        WaveRows<S, 8> w8;
        widen<S, 4>(w4, w8);
        wave_phase<S, 8, NMAX, BITS, REC, EF>(p, ch, w8, q, ring);
      }
    }
    if (p.status == 1) p.status = kDevRingOverflow;  // wider than the wave holds
    KernArgs B = args_now();
    const bool good = p.status == kDevCompleted;
    if (REC && !good) ch.give_back(before);
    const int ds = good ? wave_table<typename S::Slots>.dsteps[p.i] + p.dev + (EF ? wave_table<typename S::Slots>.nonnull[p.i] * (B->pbf + B->tbf) : 0) : 0;
    if (lane == 0) {
      B->out_status[id] = p.status;
      B->out_score[id] = p.i * B->pen.g;
      B->out_last_block[id] = header;
      B->out_dsteps[id] = (long long)ds;
      if (REC && good) B->rec_arena[header] = make_uint4(p.base[0], p.base[1], p.base[2], p.base[3]);
      if (B->out_end_k) {
        B->out_end_k[id] = p.end_k;
        B->out_end_off[id] = p.end_off;
      }
      if (!good) {
        if (p.status == kDevRingOverflow && B->over_ids) B->over_ids[atomicAdd(B->over_n, 1u)] = id;
        else atomicAdd(B->retry_count, 1u);
      }
    }
    wg_dsteps += (unsigned long long)ds;
  }
  if (lane == 0 && wg_dsteps) atomicAdd(args_now()->dsteps_total, wg_dsteps);
}

// A set of the wave's 64 * N diagonals, counted from the first: bit l of w[c]
// is diagonal N * l + c.
template <int N>
struct Diagonals {
  uint64_t w[N];
  static __device__ __forceinline__ Diagonals none() {
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) r.w[c] = 0;
    return r;
  }
  // (not empty)
  static __device__ __forceinline__ Diagonals range(int first, int last) {
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const int f = (first - c + N - 1) / N, l = last < c ? -1 : (last - c) / N;
      r.w[c] = N == 1 || f <= l ? (~0ull >> (63 - (l - f))) << f : 0ull;
    }
    return r;
  }
  __device__ __forceinline__ bool any() const {
    uint64_t r = 0;
#pragma unroll
    for (int c = 0; c < N; ++c) r |= w[c];
    return r != 0;
  }
  // (of a set that is not empty)
  __device__ __forceinline__ int first() const {
    if constexpr (N == 1) return (int)__builtin_ctzll(w[0]);
    int r = INT_MAX;
#pragma unroll
    for (int c = 0; c < N; ++c) r = min(r, w[c] ? N * (int)__builtin_ctzll(w[c]) + c : INT_MAX);
    return r;
  }
  __device__ __forceinline__ int last() const {
    if constexpr (N == 1) return 63 - (int)__builtin_clzll(w[0]);
    int r = -1;
#pragma unroll
    for (int c = 0; c < N; ++c) r = max(r, w[c] ? N * (63 - (int)__builtin_clzll(w[c])) + c : -1);
    return r;
  }
  __device__ __forceinline__ Diagonals hull() const { return any() ? range(first(), last()) : none(); }
  __device__ __forceinline__ Diagonals up() const {  // each diagonal's set bit on the next
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) r.w[c] = c ? w[c > 0 ? c - 1 : 0] : w[N - 1] << 1;
    return r;
  }
  __device__ __forceinline__ Diagonals down() const {
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) r.w[c] = c + 1 < N ? w[c + 1 < N ? c + 1 : 0] : w[0] >> 1;
    return r;
  }
  __device__ __forceinline__ Diagonals operator|(const Diagonals& o) const {
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) r.w[c] = w[c] | o.w[c];
    return r;
  }
  __device__ __forceinline__ Diagonals operator&(const Diagonals& o) const {
    Diagonals r;
#pragma unroll
    for (int c = 0; c < N; ++c) r.w[c] = w[c] & o.w[c];
    return r;
  }
  __device__ __forceinline__ bool edges() const { return ((w[0] & 1ull) | (w[N - 1] >> 63)) != 0; }
  __device__ __forceinline__ bool mine(int c) const { return (w[c] >> (threadIdx.x & 63)) & 1u; }
};

// The choices of a lane's cells: their best tagged values, and the record bytes.
template <class S, int N>
__device__ __forceinline__ uint32_t cell_choices(const int* mx, const int* mo, const int* i1, const int* d1, int* best) {
  constexpr int ONE = 1 << S::SH;
  int a[N], b[N];
#pragma unroll
  for (int c = 0; c < N; ++c) {
    a[c] = max(mo[c], i1[c]);
    b[c] = max(mo[c], d1[c]);
  }
  const int al = from_lower_lane(a[N - 1]), bu = from_upper_lane(b[0]);
  uint32_t bytes = 0;
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const int ins = (c ? a[c > 0 ? c - 1 : 0] : al) + ONE;
    const int del = (c + 1 < N ? b[c + 1 < N ? c + 1 : 0] : bu) + 2 * S::kTagD1;
    best[c] = max(max(ins, del), mx[c] + ONE + 2 * S::kTagX);
    bytes |= (((uint32_t)best[c] & 63u) | (((uint32_t)ins & 1u) << 6) | (((uint32_t)del & 1u) << 7)) << (8 * c);
  }
  return bytes;
}

// One pair with the wf-adaptive cut-off on N diagonals per lane, the middle
// between its score-0 and its end diagonal in the middle of the wave.
// Returns the status; kDevRingOverflow when the pair leaves the wave's
// diagonals or its steps.
template <class S, int N, bool REC>
__device__ __forceinline__ int cut_pair(const WaveSeqs<2>& q, WaveChunk& ch, uint32_t* base, int& steps, int& dsteps) {
  static_assert(S::NC == 3 && S::DE1 == 1 && S::RM == 4 && N <= 2, "gap-affine");
  using D = Diagonals<N>;
  constexpr int G = 4 / N;  // steps per record word
  KernArgs A = args_now();
  const int lane = threadIdx.x & 63;
  const int plen = q.plen, tlen = q.tlen, kend = tlen - plen;
  const int kt = wave_cut_center(kend) - 32 * N, k0 = kt + N * lane;
  const int z = -kt, ke = kend - kt;  // diagonal 0 and the end diagonal within the wave
  steps = dsteps = 0;
  if (z < 1 || z > 64 * N - 2) return kDevRingOverflow;
  // rows (newest first) and what the cut-off left of them
  WaveRows<S, N> w;
  D rm[S::RM], ri = D::none(), rd = D::none();
  int h0 = 0, n0 = 0;
  do {
    const int r = min(plen, tlen) - h0;
    n0 = r > 0 ? uniform(q.run(h0, h0, r)) : 0;
    h0 += n0;
  } while (n0 == WaveSeqs<2>::kSpan);
  if (kend == 0 && h0 >= tlen) return kDevCompleted;
#pragma unroll
  for (int r = 0; r < S::RM; ++r) {
    rm[r] = r ? D::none() : D::range(z, z);
#pragma unroll
    for (int c = 0; c < N; ++c) w.m[r][c] = r == 0 && k0 + c == 0 ? h0 << S::SH : kNullTagged;
  }
  uint32_t endm = 0;
#pragma unroll
  for (int c = 0; c < N; ++c) {
    w.i1[0][c] = w.d1[0][c] = kNullTagged;
    endm |= k0 + c == kend ? 1u << c : 0u;
  }
  int wait = A->heur.steps - 1;
  if (wait <= 0 && A->heur.min_len <= 1) wait = A->heur.steps;  // (a single diagonal is never cut)
  StepCells<N> cell;
  cell.rec[0] = 0;
  uint32_t* rec = nullptr;
  int seg = -1, first = 0, last = 0, i = 0;
  bool probe = false;  // the last step's I1 or D1 was emptied: its cells are in pi, pd
  int pi[N], pd[N];
  int status = kDevRingOverflow;
  for (;;) {
    if (i == last) {  // the next segment of records
      if (++seg == kWaveCutSegments) {
        steps = i;
        return kDevRingOverflow;
      }
      KernArgs B = args_now();
      first = last;
      last = B->wave.last[seg];
      if constexpr (REC) {
        const uint32_t units = (uint32_t)((last - first) / G) * 16u;
        if (!reserve_records<2>(ch, units)) return kDevArenaFull;
#pragma unroll
        for (int x = 0; x < kWaveCutSegments; ++x) base[x] = x == seg ? ch.cur : base[x];
        rec = reinterpret_cast<uint32_t*>(B->rec_arena + ch.cur) + lane;
        ch.cur += units;  // (what is not used goes back at the end)
      }
    }
    // wavefront_compute_limits_input (wavefront_compute.c:40-86)
    const D mo = rm[S::DO1 - 1];
    const D reach = rm[S::DX - 1] | mo.up() | mo.down() | ri.up() | rd.down();
    D in = D::none();
    if (reach.any()) {
      int lo = reach.first(), hi = reach.last();
      if (lo > z || hi < z) {
        // a null source still contributes the limits (1, -1), shifted as its gap moves it
        if (!rm[S::DX - 1].any()) { lo = min(lo, z + 1); hi = max(hi, z - 1); }
        if (!mo.any()) { lo = min(lo, z); hi = max(hi, z); }
        if (!ri.any()) { lo = min(lo, z + 2); hi = max(hi, z); }
        if (!rd.any()) { lo = min(lo, z); hi = max(hi, z - 2); }
      }
      in = D::range(lo, hi);
      dsteps += hi - lo + 1;
    }
    int chosen[N], probed[N], m[N];
    uint32_t bytes = 0;
    if (REC && probe) {
      (void)cell_choices<S, N>(w.m[S::DX - 1], w.m[S::DO1 - 1], w.i1[0], w.d1[0], chosen);
      bytes = cell_choices<S, N>(w.m[S::DX - 1], w.m[S::DO1 - 1], pi, pd, probed);
    }
    wave_cells<S, N, 2>(w.m[S::DX - 1], w.m[S::DO1 - 1], w.i1[0], w.d1[0], nullptr, nullptr, nullptr, m, k0, q, cell);
    if (REC && probe) {
      probe = false;
#pragma unroll
      for (int c = 0; c < N; ++c)  // (source 3: a trace through the cell would take operations back)
        if ((probed[c] >= 0) & ((probed[c] >> S::SH) > max(chosen[c], m[c]) >> S::SH)) bytes |= 6u << (8 * c);
      cell.rec[0] = (cell.rec[0] & ((1u << (32 - 8 * N)) - 1u)) | (bytes << (32 - 8 * N));
    }
    D bm, bi, bd;
    bool out = false, fin = false;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const bool mine = in.mine(c);
      m[c] = mine ? m[c] : kNullTagged;
      w.i1[0][c] = mine ? w.i1[0][c] : kNullTagged;
      w.d1[0][c] = mine ? w.d1[0][c] : kNullTagged;
      bm.w[c] = __ballot(m[c] >= 0);
      bi.w[c] = __ballot(w.i1[0][c] >= 0);
      bd.w[c] = __ballot(w.d1[0][c] >= 0);
      out |= cell.oob[c] & mine;
      fin |= (((endm >> c) & 1u) != 0) & (m[c] >= (tlen << S::SH));
    }
#pragma unroll
    for (int r = S::RM - 1; r > 0; --r) {
      rm[r] = rm[r - 1];
#pragma unroll
      for (int c = 0; c < N; ++c) w.m[r][c] = w.m[r - 1][c];
    }
#pragma unroll
    for (int c = 0; c < N; ++c) w.m[0][c] = m[c];
    ++i;
    if constexpr (REC) {
      if (((i - first) & (G - 1)) == 0) {
        *rec = cell.rec[0];
        rec += 64;
      }
    }
    if (__ballot(out)) {
      // gap cells outside the matrix: not in the trimmed ranges, and NULL
      // beyond them (wavefront_compute.c:498-613)
#pragma unroll
      for (int c = 0; c < N; ++c) {
        bi.w[c] = __ballot(in_bounds(w.i1[0][c] >> S::SH, k0 + c, plen, tlen));
        bd.w[c] = __ballot(in_bounds(w.d1[0][c] >> S::SH, k0 + c, plen, tlen));
      }
      const D hi = bi.hull(), hd = bd.hull();
#pragma unroll
      for (int c = 0; c < N; ++c) {
        w.i1[0][c] = hi.mine(c) ? w.i1[0][c] : kNullTagged;
        w.d1[0][c] = hd.mine(c) ? w.d1[0][c] : kNullTagged;
      }
    }
    if (__ballot(fin)) {
      status = kDevCompleted;
      break;
    }
    if ((bm | bi | bd).edges()) break;  // (the outermost diagonals have no neighbour)
    rm[0] = bm;
    ri = bi;
    rd = bd;
    if (bm.any() && --wait <= 0) {
      KernArgs B = args_now();
      const int lo = bm.first(), hi = bm.last();
      if (hi - lo + 1 >= B->heur.min_len) {
        wait = B->heur.steps;
        int d[N], dmin = kNullDistance;
#pragma unroll
        for (int c = 0; c < N; ++c) {
          const int h = m[c] >> S::SH;
          d[c] = m[c] >= 0 ? max(plen - (h - (k0 + c)), tlen - h) : kNullDistance;
          dmin = min(dmin, d[c]);
        }
        dmin = min(wave_min(dmin), max(plen, tlen));
        D keep;
#pragma unroll
        for (int c = 0; c < N; ++c) keep.w[c] = __ballot(d[c] - dmin <= B->heur.thr);
        keep = keep & D::range(lo, hi);
        const int top = min(ke, hi);
        const int clo = lo >= top ? lo : keep.any() ? min(keep.first(), top) : top;
        const int bottom = max(ke, clo);
        const int chi = hi <= bottom ? hi : keep.any() ? max(keep.last(), bottom) : bottom;
        if (clo != lo || chi != hi) {
          const D cut = D::range(clo, chi);  // (never empty)
          rm[0] = cut;
          ri = bi.hull() & cut;
          rd = bd.hull() & cut;
          const bool no_i = !ri.any(), no_d = !rd.any();
          if ((bi.any() && no_i) || (bd.any() && no_d)) {
            probe = true;
#pragma unroll
            for (int c = 0; c < N; ++c) {
              pi[c] = w.i1[0][c];
              pd[c] = w.d1[0][c];
              w.i1[0][c] = no_i ? kNullTagged : w.i1[0][c];
              w.d1[0][c] = no_d ? kNullTagged : w.d1[0][c];
            }
          }
        }
      }
    }
  }
  if constexpr (REC) {
    // the started word, its steps moved down to their places; the unused rest
    // of the segment goes back
    const int done = i - first, rest = done & (G - 1);
    if (rest) *rec = cell.rec[0] >> (8 * N * (G - rest));
    ch.cur -= (uint32_t)((last - first) / G - (done + G - 1) / G) * 16u;
  }
  steps = i;
  return status;
}

// wf-adaptive (wavefront_heuristic.c:190-290): the cut-off keeps a wavefront
// some tens of diagonals wide, so a lane holds one diagonal throughout; a pair
// that leaves the wave's 64 diagonals starts again with two per lane (and,
// leaving those too, goes to the lean kernel).  A step computes [lo, hi] from
// the ranges the cut-off left of its sources; cells outside are NULL, cells
// the cut-off dropped are still read (their wavefronts hold them).  Ranges are
// lane masks: a source one diagonal off is a shift, the limits are the ends of
// the union, and the computed range masks lanes as it is.  A gap range that
// the cut-off empties is not read by the next step, but the reference's
// backtrace probes its cells: that step's records are the choices with them.
//
// Records lie in up to three segments of steps (WaveArgs::last), reserved as
// the pair reaches them: short pairs take only the first.
//
// Bound by the instructions of a step, about 85 on the vector and 100 on the
// scalar side (100,000 reads of 100-300 bp, cut-off (10, 50, 1): 1.00 ms; the
// lean kernel, with a ring in LDS and clamped reads, 1.48 ms; the same loop
// with ranges as pairs of limits, 1.03 ms beside 0.34 ms and two more launches
// for the 0.3% of the pairs that leave 64 diagonals).
template <class S, bool REC>
__global__ void __launch_bounds__(64, 7) wfa_wave_cut_kernel(ForwardArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint32_t* seqP = reinterpret_cast<uint32_t*>(smem);
  uint32_t* seqT = seqP + a.wave.lds_words;
  const int lane = threadIdx.x;
  WaveChunk ch{0, 0, 0};
  unsigned long long wg_dsteps = 0;
  bool q_first = true;
  for (;;) {
    KernArgs A = args_now();
    int qv = 0;
    if (!q_first && lane == 0) qv = (int)atomicAdd(work_queue(A->queue, A->queues), 1u);
    const int qi = work_item(A->queues, q_first, lane_of(qv, 0));
    q_first = false;
    if (qi >= A->n_pairs) break;
    const int id = uniform(A->order ? A->order[qi] : qi);
    WaveSeqs<2> q{seqP, seqT, 0u, 0u, uniform(A->plen[id]), uniform(A->tlen[id])};
    wave_sync();  // the previous pair is done reading the sequences
    stage_sequences(q, A, id, seqP, seqT);
    wave_sync();
    int status = kDevArenaFull, steps = 0, dsteps = 0, wide = 0;
    uint32_t header = kNoBlock, base[kWaveCutSegments] = {0, 0, 0};
    const WaveChunk before = ch;
    if (!REC || reserve_records<2>(ch, 1)) {
      if constexpr (REC) header = ch.cur++;
      const WaveChunk narrow = ch;
      status = cut_pair<S, 1, REC>(q, ch, base, steps, dsteps);
      if (status == kDevRingOverflow) {
        wide = 1;
        if constexpr (REC) ch.give_back(narrow);
        status = cut_pair<S, 2, REC>(q, ch, base, steps, dsteps);
      }
    }
    KernArgs B = args_now();
    const bool good = status == kDevCompleted;
    if (REC && !good) ch.give_back(before);
    if (lane == 0) {
      B->out_status[id] = status;
      B->out_score[id] = steps * B->pen.g;
      B->out_last_block[id] = header;
      B->out_dsteps[id] = good ? (long long)dsteps : 0;
      if (REC && good) B->rec_arena[header] = make_uint4(base[0], base[1], base[2], (uint32_t)wide);
      if (B->out_end_k) {
        B->out_end_k[id] = q.tlen - q.plen;
        B->out_end_off[id] = q.tlen;
      }
      if (!good) atomicAdd(B->retry_count, 1u);
    }
    wg_dsteps += good ? (unsigned long long)dsteps : 0ull;
  }
  if (lane == 0 && wg_dsteps) atomicAdd(args_now()->dsteps_total, wg_dsteps);
}

template <class S>
bool wave_matches(const Penalties& p) {
  if (p.g <= 0 || p.ncomp != S::NC) return false;
  if (S::NC == 1) {
    if (!S::kMismatch) return p.metric == kIndel;
    return p.metric != kIndel && p.x == S::DX * p.g && p.o1 == S::DO1 * p.g;
  }
  return p.x == S::DX * p.g && p.o1 + p.e1 == S::DO1 * p.g && p.e1 == S::DE1 * p.g &&
         (S::NC != 5 || (p.o2 + p.e2 == S::DO2 * p.g && p.e2 == S::DE2 * p.g));
}

template <class S, int SRC, bool EF>
const void* wave_fn(int nmax, bool rec) {
  if (nmax <= 4)
    return rec ? reinterpret_cast<const void*>(&wfa_wave_kernel<S, 4, SRC, true, EF>)
               : reinterpret_cast<const void*>(&wfa_wave_kernel<ScoreOnly<S>, 4, SRC, false, EF>);
  return rec ? reinterpret_cast<const void*>(&wfa_wave_kernel<S, 8, SRC, true, EF>)
             : reinterpret_cast<const void*>(&wfa_wave_kernel<ScoreOnly<S>, 8, SRC, false, EF>);
}
template <class S>
const void* wave_fn_of(int nmax, bool rec, int bits, bool ef) {
  if (bits == 2) return ef ? wave_fn<S, 2, true>(nmax, rec) : wave_fn<S, 2, false>(nmax, rec);
  return ef ? wave_fn<S, 8, true>(nmax, rec) : wave_fn<S, 8, false>(nmax, rec);
}
const void* select_wave(int shape, int nmax, bool rec, int bits, bool ef) {
  switch (shape) {
    case 1: return wave_fn_of<ShapeAffine>(nmax, rec, bits, ef);
    case 2: return wave_fn_of<Shape2p>(nmax, rec, bits, ef);
    case 3: return wave_fn_of<ShapeEdit>(nmax, rec, bits, ef);
    case 4: return wave_fn_of<ShapeIndel>(nmax, rec, bits, ef);
    case 5: return wave_fn_of<ShapeLinear>(nmax, rec, bits, ef);
  }
  return nullptr;
}

const void* select_wave_cut(bool rec) {
  return rec ? reinterpret_cast<const void*>(&wfa_wave_cut_kernel<ShapeAffine, true>)
             : reinterpret_cast<const void*>(&wfa_wave_cut_kernel<ScoreOnly<ShapeAffine>, false>);
}

}  // namespace

int wave_shape(const Penalties& pen) {
  if (wave_matches<ShapeAffine>(pen)) return 1;
  if (wave_matches<Shape2p>(pen)) return 2;
  if (wave_matches<ShapeEdit>(pen)) return 3;
  if (wave_matches<ShapeIndel>(pen)) return 4;
  if (wave_matches<ShapeLinear>(pen)) return 5;
  return 0;
}

bool wave_phases(int shape, int pbf, int tbf, int nmax, WaveArgs* w) {
  const WaveTable* t = shape == 1 ? &host_wave_table<ShapeAffine> : shape == 2 ? &host_wave_table<Shape2p>
                     : shape == 3 ? &host_wave_table<ShapeEdit>
                     : shape == 4 ? &host_wave_table<ShapeIndel> : shape == 5 ? &host_wave_table<ShapeLinear> : nullptr;
  if (!t) return false;
  *w = WaveArgs{};
  w->center = (tbf - pbf) / 2;
  w->phase0 = -1;
  for (int ph = 0; ph < kWavePhases; ++ph) {
    const int n = 1 << ph, kt = w->center - 32 * n;
    // wavefronts keep clear of the wave's first and last diagonal
    auto fits = [&](int lo, int hi) { return lo - pbf > kt && hi + tbf < kt + 64 * n - 1; };
    int steps = 0;
    if (n <= nmax && fits(0, 0)) {
      while (steps < kWaveSteps && fits(t->hull_lo[steps], t->hull_hi[steps])) ++steps;
      if (w->phase0 < 0) w->phase0 = ph;
    }
    const int per_word = n < 4 ? 4 / n : 1;
    w->last[ph] = steps / per_word * per_word;
    if (ph && w->last[ph] < w->last[ph - 1]) w->last[ph] = w->last[ph - 1];
  }
  return w->phase0 >= 0 && w->phase0 <= 2;
}

size_t wave_lds_bytes(int lds_words) { return (size_t)2 * lds_words * sizeof(uint32_t); }

bool wave_cuts(int shape, const HeurArgs& h) {
  return shape == 1 && h.wfadaptive == 1 && !h.xdrop && !h.zdrop && !h.banded;
}

void wave_cut_phases(WaveArgs* w) {
  *w = WaveArgs{};
  w->cut = 1;
  w->last[0] = 48;
  w->last[1] = 176;
  w->last[2] = w->last[3] = kWaveSteps;
  static_assert(kWaveCutSegments == 3 && kWaveSteps % 4 == 0, "segments");
}

uint32_t wave_record_units(const WaveArgs& w, int nmax) {
  if (w.cut) return 1 + (uint32_t)(w.last[kWaveCutSegments - 1] / 2) * 16u;  // two diagonals per lane
  uint32_t units = 1;
  for (int ph = 0, first = 0; ph < kWavePhases && (1 << ph) <= nmax; first = w.last[ph++]) {
    const int n = 1 << ph, g = n < 4 ? 4 / n : 1;
    units += (uint32_t)((w.last[ph] - first + g - 1) / g * (n > 4 ? n / 4 : 1)) * 16u;
  }
  return units;
}

int wave_max_blocks_per_cu(int shape, int nmax, bool rec, int bits, bool ef, bool cut, size_t lds) {
  const void* f = cut ? select_wave_cut(rec) : select_wave(shape, nmax, rec, bits, ef);
  int n = 0;
  if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, 64, lds) != hipSuccess) return 0;
  return n;
}

hipError_t launch_forward_wave(const ForwardArgs& a, int shape, int nmax, int bits, const LaunchShape& ls,
                               hipStream_t stream) {
  // a cut-off that the kernel does not do, or one where none is asked for
  if ((a.wave.cut != 0) != (a.heur.cut() != 0) || (a.wave.cut && !wave_cuts(shape, a.heur))) return hipErrorInvalidValue;
  // a score-0 wavefront that needs more than the 4 diagonals per lane a pair starts with at most
  if (!a.wave.cut && (a.wave.phase0 < 0 || a.wave.phase0 > 2)) return hipErrorInvalidValue;
  const void* f = a.wave.cut ? select_wave_cut(a.records != 0)
                             : select_wave(shape, nmax, a.records != 0, bits, a.endsfree != 0);
  if (!f || ls.block != 64) return hipErrorInvalidValue;
  void* args[] = {const_cast<ForwardArgs*>(&a)};
  return hipLaunchKernel(f, dim3(ls.grid), dim3(64), args, ls.lds_bytes, stream);
}

}  // namespace wfa
