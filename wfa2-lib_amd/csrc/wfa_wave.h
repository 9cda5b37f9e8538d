// Interface of the short-pair wave kernels (wfa_wave.hip).
#pragma once
#include "wfa_device.h"

namespace wfa {

// 0: no instance.  1 gap-affine, 2 gap-affine-2p, 3 edit, 4 indel, 5 gap-linear.
int wave_shape(const Penalties& pen);
// The phases of a form of alignment: the steps at which a lane's diagonals
// double (last), for at most nmax per lane.  False when the score-0 wavefront
// does not fit.
bool wave_phases(int shape, int pbf, int tbf, int nmax, WaveArgs* w);
// Whether the wave family runs the penalties with the cut-offs of `heur`, and
// the place of its records (segments of steps).
bool wave_cuts(int shape, const HeurArgs& heur);
void wave_cut_phases(WaveArgs* w);
// Most record units (16 bytes) that a wave reserves for one pair.
uint32_t wave_record_units(const WaveArgs& w, int nmax);
size_t wave_lds_bytes(int lds_words);
int wave_max_blocks_per_cu(int shape, int nmax, bool rec, int bits, bool ef, bool cut, size_t lds);
// nmax: most diagonals per lane (4 or 8; 1 with a cut-off).
hipError_t launch_forward_wave(const ForwardArgs& a, int shape, int nmax, int bits, const LaunchShape& ls,
                               hipStream_t stream);

}  // namespace wfa
