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
// Values are kept as (offset << SH) | source << 1 | flag (ScoreOnly shapes:
// as offsets).  One maximum over
// the candidates then takes the largest offset with the reference's
// tie-breaks (M > D2 > D1 > I2 > I1, extension before opening,
// wavefront_backtrace.c:64-219): the source codes rise in that order below
// the offset, and bit 0 of a gap value says "extended".  The record of a cell
// is cut out of the low bits with v_alignbit: one instruction per field,
// already packed for the lane's N cells.
#pragma once
#include "wfa_common.h"
#include "wfa_shapes.h"

namespace wfa {

constexpr int kNullTagged = -(1 << 30);

template <class S, int N>
struct WaveRows {
  int m[S::RM][N];  // row i in m[i % RM]
  int i1[S::DE1][N], d1[S::DE1][N];  // NC > 1
  int i2[S::DE2][N], d2[S::DE2][N];  // NC == 5
};

// The value of the lane below / above; NULL from beyond the wave.
__device__ __forceinline__ int from_lower_lane(int v) {
  return __builtin_amdgcn_update_dpp(kNullTagged, v, 0x138, 0xf, 0xf, false);  // wave_shr:1
}
__device__ __forceinline__ int from_upper_lane(int v) {
  return __builtin_amdgcn_update_dpp(kNullTagged, v, 0x130, 0xf, 0xf, false);  // wave_shl:1
}

// First / last diagonal whose bit is set: lane l holds the bits of its N
// diagonals kt + N * l + c.
template <int N>
__device__ __forceinline__ int first_diagonal(uint32_t bits, int kt) {
  const unsigned long long bal = __ballot(bits != 0);
  if (!bal) return INT_MAX;
  const int l = (int)__builtin_ctzll(bal);
  if constexpr (N == 1) return kt + l;
  return kt + N * l + (int)__builtin_ctz((unsigned)lane_of((int)bits, l));
}
template <int N>
__device__ __forceinline__ int last_diagonal(uint32_t bits, int kt) {
  const unsigned long long bal = __ballot(bits != 0);
  if (!bal) return INT_MIN;
  const int l = 63 - (int)__builtin_clzll(bal);
  if constexpr (N == 1) return kt + l;
  return kt + N * l + 31 - (int)__builtin_clz((unsigned)lane_of((int)bits, l));
}

// The 32 bits of a packed sequence from bit `bit` of W (v_alignbit takes the
// shift modulo 32 by itself).
template <typename P32>
__device__ __forceinline__ uint32_t window32(P32 W, unsigned bit) {
  const unsigned w = bit >> 5;
  return __builtin_amdgcn_alignbit(W[w + 1], W[w], bit);
}

// Matching symbols at the start of a window whose xor is x (0..32 / BITS), at
// most cap: v_ffbl gives -1 for x == 0, which the shift turns into a large
// value.
template <int BITS>
__device__ __forceinline__ int match_run(uint32_t x, int cap) {
  uint32_t f;
  asm("v_ffbl_b32 %0, %1" : "=v"(f) : "v"(x));
  return min(min((int)(f / BITS), 32 / BITS), cap);
}

// The sequences of the pair, BITS bits per symbol: symbol 0 of the pattern /
// text at bit pbit / tbit of P / T.
template <int BITS>
struct WaveSeqs {
  const uint32_t* P;
  const uint32_t* T;
  unsigned pbit, tbit;
  int plen, tlen;
  static constexpr int kSpan = 32 / BITS;  // symbols per window
  // matching symbols (at most cap) of the window at text offset h of diagonal h - v
  __device__ __forceinline__ int run(int h, int v, int cap) const {
    return match_run<BITS>(window32(T, tbit + (unsigned)(BITS * h)) ^ window32(P, pbit + (unsigned)(BITS * v)), cap);
  }
};

// What a step tells about its cells.
template <int N>
struct StepCells {
  int h[N];        // extended M offset (meaningless where !ok)
  bool ok[N];      // valid M cell
  int rem[N];      // symbols left to the nearer border after the extension
  bool oob[N];     // a path reaches the cell, but outside the matrix
  // Record bytes, shifted in from the top: after four cells (of one step, or
  // with N < 4 of consecutive steps) a word holds them in order.
  uint32_t rec[(N + 3) / 4];
};

// The cells of one step from their source rows (tagged values of the lane's N
// diagonals): mx, mo (rows i - DX and i - DO1 of M), i1, d1 (rows i - DE1) and,
// with a second gap, mo2 (row i - DO2), i2, d2 (rows i - DE2).  The new gap
// rows replace i1, d1, i2, d2; the new M row goes to m (which may be mo).
// wavefront_compute_affine.c:44-86, wavefront_compute_affine2p.c:45-106,
// wavefront_extend_kernels.c:68-123.
template <class S, int N, int BITS>
__device__ __forceinline__ void wave_cells(const int* mx, const int* mo, int* i1, int* d1, const int* mo2, int* i2,
                                           int* d2, int* m, int k0, const WaveSeqs<BITS>& q, StepCells<N>& out) {
  constexpr int SH = S::SH, ONE = 1 << SH, SPAN = WaveSeqs<BITS>::kSpan;
  int a1[N], b1[N], a2[N], b2[N];
#pragma unroll
  for (int c = 0; c < N; ++c) {
    a1[c] = S::NC == 1 ? mo[c] : max(mo[c], i1[c]);
    b1[c] = S::NC == 1 ? mo[c] : max(mo[c], d1[c]);
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
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const int ins1 = (c ? a1[c > 0 ? c - 1 : 0] : a1l) + ONE;
    const int del1 = (c + 1 < N ? b1[c + 1 < N ? c + 1 : 0] : b1u) + 2 * S::kTagD1;
    int best = max(ins1, del1);
    if constexpr (S::kMismatch) best = max(best, mx[c] + ONE + 2 * S::kTagX);
    int ins2 = 0, del2 = 0;
    if constexpr (S::NC == 5) {
      ins2 = (c ? a2[c > 0 ? c - 1 : 0] : a2l) + ONE + 2 * S::kTagI2;
      del2 = (c + 1 < N ? b2[c + 1 < N ? c + 1 : 0] : b2u) + 2 * S::kTagD2;
      best = max(max(best, ins2), del2);
    }
    if constexpr (S::NC > 1) {
      i1[c] = S::kTags ? (ins1 & ~(ONE - 1)) | 1 : ins1;
      d1[c] = S::kTags ? (del1 & ~(ONE - 1)) | 1 : del1;
    }
    if constexpr (S::NC == 5) {
      i2[c] = S::kTags ? (ins2 & ~(ONE - 1)) | 1 : ins2;
      d2[c] = S::kTags ? (del2 & ~(ONE - 1)) | 1 : del2;
    }
    // record byte: NC == 5: source and flag of the best (4 bits), then the
    // flags of I1, D1, I2, D2; NC == 3: 6 bits of the best (source in bits
    // 1..2), then the flags of I1 and D1; NC == 1: 8 bits of the best
    uint32_t& acc = out.rec[c / 4];
    if constexpr (S::NC == 5) {
      acc = __builtin_amdgcn_alignbit((uint32_t)best, acc, 4);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins2, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del2, acc, 1);
    } else if constexpr (S::NC == 3) {
      acc = __builtin_amdgcn_alignbit((uint32_t)best, acc, 6);
      acc = __builtin_amdgcn_alignbit((uint32_t)ins1, acc, 1);
      acc = __builtin_amdgcn_alignbit((uint32_t)del1, acc, 1);
    } else {
      acc = __builtin_amdgcn_alignbit((uint32_t)best, acc, 8);
    }
    // null-after-max, then one 16-symbol window of the extension
    const int off = best >> SH, k = k0 + c, v = off - k;
    const bool ok = ((unsigned)off <= (unsigned)q.tlen) & ((unsigned)v <= (unsigned)q.plen);
    const int o = ok ? off : 0, vv = ok ? v : 0;
    const int r = min(q.tlen - o, q.plen - vv);
    const int n = q.run(o, vv, r);
    out.ok[c] = ok;
    out.oob[c] = !ok & (best >= 0);
    out.h[c] = o + n;
    out.rem[c] = r - n;
    full |= (ok & (n == SPAN) & (r > SPAN)) ? 1u << c : 0u;
  }
  // long runs (rare away from the main diagonal): more windows, cell by cell
  if (__ballot(full != 0)) {
#pragma unroll
    for (int c = 0; c < N; ++c) {
      bool more = (full >> c) & 1u;
      if (__ballot(more)) {
        int h = out.h[c], r = out.rem[c];
        while (more) {
          const int n = q.run(h, h - (k0 + c), r);
          h += n;
          r -= n;
          more = (n == SPAN) & (r > 0);
        }
        out.h[c] = h;
        out.rem[c] = r;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < N; ++c) m[c] = out.ok[c] ? out.h[c] << SH : kNullTagged;
}

// Step i (compile-time phase PH = i mod the unroll) over rows in registers;
// o2: row i - DO2, tagged (NC == 5).  The oldest rows are replaced by the new.
template <class S, int N, int PH, int BITS>
__device__ __forceinline__ void wave_step(WaveRows<S, N>& w, const int* o2, int k0, const WaveSeqs<BITS>& q,
                                          StepCells<N>& out) {
  constexpr int rx = (PH + 8 * S::RM - (S::kMismatch ? S::DX : 0)) % S::RM, ro = (PH + 8 * S::RM - S::DO1) % S::RM, rn = PH % S::RM;
  constexpr int g1 = PH % S::DE1, g2 = PH % S::DE2;
  wave_cells<S, N, BITS>(w.m[rx], w.m[ro], w.i1[g1], w.d1[g1], o2, w.i2[g2], w.d2[g2], w.m[rn], k0, q, out);
}

}  // namespace wfa
