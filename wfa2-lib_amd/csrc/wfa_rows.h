// One score step of the wavefront recurrence on a stretch of diagonals held
// in the registers of one wave.  Included by .hip files only.
//
// Lane l of the wave owns N neighbouring diagonals k0 .. k0+N-1 with
// k0 = kt + N*l, for the whole run: a diagonal never moves between lanes, so a
// gap source k-1 or k+1 is the lane's own neighbouring register, or, at the
// edge of its N diagonals, one DPP wave shift that the adding instruction
// takes for free.  No step re-reads a ring through clamped indices; cells
// outside a wavefront's range hold NULL by themselves, because everything
// they are computed from does.
//
// Values are kept as (offset << SH) | source << 1 | flag.  One maximum over
// the candidates then takes the largest offset with the reference's
// tie-breaks (M > D2 > D1 > I2 > I1, extension before opening,
// wavefront_backtrace.c:64-219): the source codes rise in that order below
// the offset, and bit 0 of a gap value says "extended".  The record of a cell
// is cut out of the low bits with v_alignbit: one instruction per field,
// already packed for the lane's N cells.
#pragma once
#include "wfa_common.h"

namespace wfa {

// Distances between wavefronts in steps (score / g), known at compile time.
template <int NC_, int DX_, int DO1_, int DE1_, int DO2_, int DE2_>
struct SlotShape {
  static constexpr int NC = NC_, DX = DX_, DO1 = DO1_, DE1 = DE1_, DO2 = DO2_, DE2 = DE2_;
  static constexpr int RM = DX > DO1 ? DX : DO1;  // M rows kept in registers (the second gap's come from memory)
  static constexpr int SH = NC == 5 ? 4 : 3;      // bits below the offset
  static constexpr int kTagX = NC == 5 ? 4 : 2, kTagD2 = 3, kTagD1 = NC == 5 ? 2 : 1, kTagI2 = 1;
  static constexpr int kGapRows = 2 * DE1 + (NC == 5 ? 2 * DE2 : 0);
};
using Shape2p = SlotShape<5, 4, 8, 2, 25, 1>;  // gap-affine-2p (x 4, o1 6, e1 2, o2 24, e2 1) and its multiples
using ShapeAffine = SlotShape<3, 2, 4, 1, 0, 1>;  // gap-affine (x 4, o 6, e 2) and its multiples

constexpr int kNullTagged = -(1 << 30);

template <class S, int N>
struct WaveRows {
  int m[S::RM][N];  // row i in m[i % RM]
  int i1[S::DE1][N], d1[S::DE1][N];
  int i2[S::DE2][N], d2[S::DE2][N];  // NC == 5
};

// The value of the lane below / above; NULL from beyond the wave.
__device__ __forceinline__ int from_lower_lane(int v) {
  return __builtin_amdgcn_update_dpp(kNullTagged, v, 0x138, 0xf, 0xf, false);  // wave_shr:1
}
__device__ __forceinline__ int from_upper_lane(int v) {
  return __builtin_amdgcn_update_dpp(kNullTagged, v, 0x130, 0xf, 0xf, false);  // wave_shl:1
}

// 16 symbols of a 2-bit packed sequence whose first symbol sits at bit `bit`
// of W (v_alignbit takes the shift modulo 32 by itself).
template <typename P32>
__device__ __forceinline__ uint32_t window16(P32 W, unsigned bit) {
  const unsigned w = bit >> 5;
  return __builtin_amdgcn_alignbit(W[w + 1], W[w], bit);
}

// Matching symbols at the start of a 16-symbol window whose xor is x (0..16):
// v_ffbl gives -1 for x == 0, which the shift turns into a large value.
__device__ __forceinline__ int match_run16(uint32_t x, int cap) {
  uint32_t f;
  asm("v_ffbl_b32 %0, %1" : "=v"(f) : "v"(x));
  return min(min((int)(f >> 1), 16), cap);
}

// The sequences of the pair in LDS: symbol 0 of the pattern / text at bit
// pbit / tbit of P / T.
struct WaveSeqs {
  const uint32_t* P;
  const uint32_t* T;
  unsigned pbit, tbit;
  int plen, tlen;
};

// What a step tells about its cells.
template <int N>
struct StepCells {
  int h[N];        // extended M offset (meaningless where !ok)
  bool ok[N];      // valid M cell
  bool oob[N];     // a path reaches the cell, but outside the matrix
  uint32_t rec[(N + 3) / 4];  // record bytes
};

// The cells of one step from their source rows (tagged values of the lane's N
// diagonals): mx, mo (rows i - DX and i - DO1 of M), i1, d1 (rows i - DE1) and,
// with a second gap, mo2 (row i - DO2), i2, d2 (rows i - DE2).  The new gap
// rows replace i1, d1, i2, d2; the new M row goes to m (which may be mo).
// wavefront_compute_affine.c:44-86, wavefront_compute_affine2p.c:45-106,
// wavefront_extend_kernels.c:68-123.
template <class S, int N>
__device__ __forceinline__ void wave_cells(const int* mx, const int* mo, int* i1, int* d1, const int* mo2, int* i2,
                                           int* d2, int* m, int k0, const WaveSeqs& q, StepCells<N>& out) {
  constexpr int SH = S::SH, ONE = 1 << SH;
  int a1[N], b1[N], a2[N], b2[N];
#pragma unroll
  for (int c = 0; c < N; ++c) {
    a1[c] = max(mo[c], i1[c]);
    b1[c] = max(mo[c], d1[c]);
    if constexpr (S::NC == 5) {
      a2[c] = max(mo2[c], i2[c]);
      b2[c] = max(mo2[c], d2[c]);
    }
  }
  const int a1l = from_lower_lane(a1[N - 1]), b1u = from_upper_lane(b1[0]);
  int a2l = 0, b2u = 0;
  if constexpr (S::NC == 5) {
    a2l = from_lower_lane(a2[N - 1]);
    b2u = from_upper_lane(b2[0]);
  }
  uint32_t full = 0;  // cells whose run fills the window
  int rem[N];
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const int ins1 = (c ? a1[c > 0 ? c - 1 : 0] : a1l) + ONE;
    const int del1 = (c + 1 < N ? b1[c + 1 < N ? c + 1 : 0] : b1u) + 2 * S::kTagD1;
    const int x = mx[c] + ONE + 2 * S::kTagX;
    int best = max(max(ins1, del1), x);
    int ins2 = 0, del2 = 0;
    if constexpr (S::NC == 5) {
      ins2 = (c ? a2[c > 0 ? c - 1 : 0] : a2l) + ONE + 2 * S::kTagI2;
      del2 = (c + 1 < N ? b2[c + 1 < N ? c + 1 : 0] : b2u) + 2 * S::kTagD2;
      best = max(max(best, ins2), del2);
    }
    i1[c] = (ins1 & ~(ONE - 1)) | 1;
    d1[c] = (del1 & ~(ONE - 1)) | 1;
    if constexpr (S::NC == 5) {
      i2[c] = (ins2 & ~(ONE - 1)) | 1;
      d2[c] = (del2 & ~(ONE - 1)) | 1;
    }
    // record byte: NC == 5: source and flag of the best (4 bits), then the
    // flags of I1, D1, I2, D2; NC == 3: 6 bits of the best (source in bits
    // 1..2), then the flags of I1 and D1
    uint32_t& acc = out.rec[c / 4];
    if constexpr (S::NC == 5) {
      acc = __builtin_amdgcn_alignbit((uint32_t)best, c % 4 ? acc : 0u, 4);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins2, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del2, acc, 1);
    } else {
      acc = __builtin_amdgcn_alignbit((uint32_t)best, c % 4 ? acc : 0u, 6);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del1, acc, 1);
    }
    // null-after-max, then one 16-symbol window of the extension
    const int off = best >> SH, k = k0 + c, v = off - k;
    const bool ok = ((unsigned)off <= (unsigned)q.tlen) & ((unsigned)v <= (unsigned)q.plen);
    const int o = ok ? off : 0, vv = ok ? v : 0;
    const int r = min(q.tlen - o, q.plen - vv);
    const uint32_t d = window16(q.T, q.tbit + 2u * (unsigned)o) ^ window16(q.P, q.pbit + 2u * (unsigned)vv);
    const int n = match_run16(d, r);
    out.ok[c] = ok;
    out.oob[c] = !ok & (best >= 0);
    out.h[c] = o + n;
    rem[c] = r - n;
    full |= (ok & (n == 16) & (r > 16)) ? 1u << c : 0u;
  }
  // long runs (rare away from the main diagonal): more windows, cell by cell
  if (__ballot(full != 0)) {
#pragma unroll
    for (int c = 0; c < N; ++c) {
      bool more = (full >> c) & 1u;
      if (__ballot(more)) {
        int h = out.h[c], r = rem[c];
        while (more) {
          const uint32_t d = window16(q.T, q.tbit + 2u * (unsigned)h) ^
                             window16(q.P, q.pbit + 2u * (unsigned)(h - (k0 + c)));
          const int n = match_run16(d, r);
          h += n;
          r -= n;
          more = (n == 16) & (r > 0);
        }
        out.h[c] = h;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < N; ++c) m[c] = out.ok[c] ? out.h[c] << SH : kNullTagged;
}

// Step i (compile-time phase PH = i mod the unroll) over rows in registers;
// o2: row i - DO2, tagged (NC == 5).  The oldest rows are replaced by the new.
template <class S, int N, int PH>
__device__ __forceinline__ void wave_step(WaveRows<S, N>& w, const int* o2, int k0, const WaveSeqs& q,
                                          StepCells<N>& out) {
  constexpr int rx = (PH + 8 * S::RM - S::DX) % S::RM, ro = (PH + 8 * S::RM - S::DO1) % S::RM, rn = PH % S::RM;
  constexpr int g1 = PH % S::DE1, g2 = PH % S::DE2;
  wave_cells<S, N>(w.m[rx], w.m[ro], w.i1[g1], w.d1[g1], o2, w.i2[g2], w.d2[g2], w.m[rn], k0, q, out);
}

}  // namespace wfa
