// Slot structures of the penalties that the wave and tile kernels are built
// for, and the ranges of their wavefronts.
#pragma once
#include "wfa_device.h"

namespace wfa {

// Distances between wavefronts in steps (score / g), known at compile time.
template <int NC_, int DX_, int DO1_, int DE1_, int DO2_, int DE2_>
struct SlotShape {
  using Slots = SlotShape;
  static constexpr int NC = NC_, DX = DX_, DO1 = DO1_, DE1 = DE1_, DO2 = DO2_, DE2 = DE2_;
  static constexpr int RM = DX > DO1 ? DX : DO1;  // M rows kept in registers (the second gap's come from memory)
  static constexpr int SH = NC == 5 ? 4 : 3;      // bits below the offset
  static constexpr bool kMismatch = DX > 0;       // (indel distance has no mismatches)
  static constexpr bool kTags = true;             // ... which hold a cell's source
  static constexpr int kTagX = NC == 5 ? 4 : 2, kTagD2 = 3, kTagD1 = NC == 5 ? 2 : 1, kTagI2 = 1;
  static constexpr int kGapRows = 2 * DE1 + (NC == 5 ? 2 * DE2 : 0);
};
// The shape without records: values are plain offsets, which saves the tags'
// masking (150,000 reads of 100-300 bp, score only: 0.574 -> 0.533 ms).
template <class S>
struct ScoreOnly : S {
  static constexpr bool kTags = false;
  static constexpr int SH = 0, kTagX = 0, kTagD2 = 0, kTagD1 = 0, kTagI2 = 0;
};
using Shape2p = SlotShape<5, 4, 8, 2, 25, 1>;  // gap-affine-2p (x 4, o1 6, e1 2, o2 24, e2 1) and its multiples
using ShapeAffine = SlotShape<3, 2, 4, 1, 0, 1>;  // gap-affine (x 4, o 6, e 2) and its multiples
// One component: a gap symbol costs DO1 steps (DE1, DE2 are not used).
using ShapeEdit = SlotShape<1, 1, 1, 1, 0, 1>;
using ShapeIndel = SlotShape<1, 0, 1, 1, 0, 1>;
using ShapeLinear = SlotShape<1, 2, 1, 1, 0, 1>;  // gap-linear (x 4, indel 2) and its multiples


struct StepRange {
  int lo = 1, hi = -1;
  constexpr bool valid() const { return lo <= hi; }
  // takes in s shifted by d
  constexpr void add(const StepRange& s, int d) {
    if (!s.valid()) return;
    if (!valid()) {
      lo = s.lo + d;
      hi = s.hi + d;
    } else {
      lo = s.lo + d < lo ? s.lo + d : lo;
      hi = s.hi + d > hi ? s.hi + d : hi;
    }
  }
};

// The ranges of the five components at one step, from those of the earlier
// ones (row(back, c): component c `back` steps ago), each as wide as its
// sources make it (wavefront_compute_limits_input, wavefront_compute.c:
// 40-86): the same for all pairs until an end cell leaves the matrix.
struct StepRanges {
  StepRange c[5];
};
template <class Row>
constexpr StepRanges next_ranges(int ncomp, int dx, int do1, int de1, int do2, int de2, Row row) {
  StepRanges r;
  const StepRange mo = row(do1, kM);
  if (dx > 0) r.c[kM].add(row(dx, kM), 0);
  r.c[kM].add(mo, 1);
  r.c[kM].add(mo, -1);
  if (ncomp > 1) {
    r.c[kI1].add(mo, 1);
    r.c[kI1].add(row(de1, kI1), 1);
    r.c[kD1].add(mo, -1);
    r.c[kD1].add(row(de1, kD1), -1);
  }
  if (ncomp == 5) {
    const StepRange mo2 = row(do2, kM);
    r.c[kI2].add(mo2, 1);
    r.c[kI2].add(row(de2, kI2), 1);
    r.c[kD2].add(mo2, -1);
    r.c[kD2].add(row(de2, kD2), -1);
  }
  for (int g = kI1; g <= kD2; ++g) r.c[kM].add(r.c[g], 0);
  return r;
}

// Diagonals of a step whose sources are row(...) and whose cells reach [m.lo,
// m.hi]: a null source still contributes the limits (1, -1), shifted as its
// gap moves it.
template <class Row>
constexpr int step_diagonals(const StepRange& m, int ncomp, int dx, int do1, int de1, int do2, int de2, Row row) {
  if (!m.valid()) return 0;
  int lo = m.lo, hi = m.hi;
  auto null = [&](int back, int c, int l, int h) {
    if (row(back, c).valid()) return;
    lo = l < lo ? l : lo;
    hi = h > hi ? h : hi;
  };
  if (dx > 0) null(dx, kM, 1, -1);
  null(do1, kM, 0, 0);
  if (ncomp > 1) {
    null(de1, kI1, 2, 0);
    null(de1, kD1, 0, -2);
  }
  if (ncomp == 5) {
    null(do2, kM, 0, 0);
    null(de2, kI2, 2, 0);
    null(de2, kD2, 0, -2);
  }
  return hi - lo + 1;
}

// The first steps' ranges of a shape, tabulated by the compiler.  Row i is
// step i; row -1, score 0, holds M = [0, 0].
constexpr int kWaveSteps = 560;  // a wave of 8 diagonals per lane is outgrown before
struct WaveTable {
  int lo[kWaveSteps], hi[kWaveSteps];            // range of M (lo > hi: none)
  int hull_lo[kWaveSteps], hull_hi[kWaveSteps];  // of the rows so far
  int dsteps[kWaveSteps + 1];                    // diagonal-steps of the first i steps
  int nonnull[kWaveSteps + 1];                   // wavefronts among them
  // Components with a wavefront before step i: bit r - 1: M of row i - r; and
  // in four bits from 4 (r - 1) on, I1, D1, I2 and D2 of row i - r.
  uint32_t hist_m[kWaveSteps], hist_gap[kWaveSteps];
};
template <class S>
constexpr WaveTable make_wave_table() {
  WaveTable t{};
  StepRanges rows[kWaveSteps + 1];
  rows[0].c[kM].lo = rows[0].c[kM].hi = 0;
  uint32_t hm = 1, hg = 0;
  int hlo = 0, hhi = 0;
  for (int i = 0; i < kWaveSteps; ++i) {
    rows[i + 1] = next_ranges(S::NC, S::DX, S::DO1, S::DE1, S::DO2, S::DE2, [&](int back, int c) {
      return i + 1 - back >= 0 ? rows[i + 1 - back].c[c] : StepRange{};
    });
    const StepRange m = rows[i + 1].c[kM];
    t.hist_m[i] = hm;
    t.hist_gap[i] = hg;
    hm = (hm << 1) | (m.valid() ? 1u : 0u);
    hg <<= 4;
    for (int c = kI1; c <= kD2; ++c) hg |= rows[i + 1].c[c].valid() ? 1u << (c - kI1) : 0u;
    t.lo[i] = m.lo;
    t.hi[i] = m.hi;
    if (m.valid()) {
      hlo = m.lo < hlo ? m.lo : hlo;
      hhi = m.hi > hhi ? m.hi : hhi;
    }
    t.hull_lo[i] = hlo;
    t.hull_hi[i] = hhi;
    t.dsteps[i + 1] = t.dsteps[i] + (m.valid() ? m.hi - m.lo + 1 : 0);
    t.nonnull[i + 1] = t.nonnull[i] + (m.valid() ? 1 : 0);
  }
  return t;
}

}  // namespace wfa
