// Interface of the tile kernels (wfa_tile.hip): long pairs advanced a block
// of score steps per launch, in tiles of diagonals.  Steps are counted in
// slots: step i is score (i + 1) * g, and score 0 is step -1.
#pragma once
#include "wfa_device.h"

namespace wfa {

// State diagonals below the pattern's and above the text's length: a tile
// reads its halo there, and the last tile reaches past the last diagonal.
constexpr int kTilePadLow = 128, kTilePadHigh = 768;
// Index of diagonal 0 in a job's state rows (a multiple of 4).
__host__ __device__ inline int tile_kpad(int plen) { return (plen + kTilePadLow + 3) / 4 * 4; }
__host__ __device__ inline int tile_pitch(int plen, int tlen) { return tile_kpad(plen) + (tlen + kTilePadHigh + 3) / 4 * 4; }

// LDS for the two sequences of a job (2-bit sequences up to 130 kbp).
constexpr size_t kTileSeqLdsBytes = 64 * 1024;

struct TileBlockInfo {  // records of one block: first diagonal and bytes per step
  int kb, pitch;
};

// The diagonals of a job in one block: rows written over [left, right), and
// the lowest and highest diagonal a wavefront of the block reached.
struct TileRange {
  int left, right, min_lo, max_hi;
};

// A job of a pass.  Everything the tiles keep of a job is found by its slot in
// the pass, not by its id in the batch: the buffers are as large as the pass,
// however many other pairs the batch has.
struct TileJob {
  int64_t ppos, tpos;          // its sequences (symbols)
  int64_t st_off;              // first int of its state
  int plen, tlen;
  int pitch;                   // ints per state row
  int id;
};
struct TileSeqs {              // of the batch, by id
  const int* plen;
  const int* tlen;
  const int64_t* pat_pos;
  const int64_t* txt_pos;
};
struct TileSlot {              // what the host says of a job
  int64_t st_off;
  int id, pad;
};

struct TileArgs {
  const int* act;              // slots of the active jobs
  const int* n_act;
  TileJob* jobs;
  const uint64_t* words;
  int* state;                  // rows of every job
  int* done;                   // step at which the job reached its end (INT_MAX: not yet)
  int* irr;                    // first step whose end left its tile (INT_MAX: none)
  TileRange* range;            // per job, of the last four blocks
  const int2* m_range;         // per step, the untrimmed range of M (lo > hi: none)
  int* exact_lo;               // 1 + the block in which the job's low / high end was first
  int* exact_hi;               // trimmed, or 0
  long long* dev[2][2];        // by block parity and end: the limits minus the tabulated ones, summed
                               // up to each step of the block (steps-per-block entries per job)
  const long long* dsteps_upto;  // untrimmed diagonal-steps up to and including step i at [i + 1]
  int* stepped;                // whether the job changed over to one step per launch
  uint4* rec;                  // record arena
  uint32_t* rec_tab;           // per job and block: first unit of its records
  int tab_stride;
  uint32_t rec_unit0;          // this block's records: job y at rec_unit0 + y * rec_job_units
  uint32_t rec_job_units;
  int rec_kb;                  // first diagonal of the records
  int rec_pitch;               // bytes per step
  int blk;
  int tiles;                   // at most
  int lmax_words;              // LDS words per sequence
};

constexpr int kTileStepEnds = 12, kTileStepFlags = 32;

// Jobs whose ends jump, one step per launch (tile_step_kernel).
struct StepArgs {
  const int* act;
  const int* n_act;
  const TileJob* jobs;
  const uint64_t* words;
  int* state;
  const int64_t* st_off;       // first int of a job's rows here
  int* done;
  int* ends;                   // per job, ring of 4 steps: kTileStepEnds ends of the components
  int* flags;                  // per job, ring of kTileStepFlags steps: which components have a valid cell
  long long* dsum;             // diagonal-steps before the latest step
  int* step0;                  // the job's first step
  uint4* rec;
  uint32_t* rec_tab;
  int tab_stride;
  uint32_t rec_unit0;          // this block's records: job y at rec_unit0 + y * rec_job_units
  uint32_t rec_job_units;
  const TileBlockInfo* blocks;
};

struct TileFinishArgs {
  int n;
  const TileJob* jobs;
  const int* done;
  const int* irr;
  const long long* dsteps_upto;
  const int* exact_lo;
  const int* exact_hi;
  const long long* dev[2][2];
  const int* stepped;
  const int* step_ends;        // StepArgs::ends
  const int* flags;
  const long long* dsum;
  int steps;                   // per block
  int g;
  int* out_status;
  int* out_score;
  long long* out_dsteps;
  uint32_t* out_last_block;
  int* out_end_k;
  int* out_end_off;
  unsigned long long* dsteps_total;
  unsigned int* retry_count;
};

struct TileTraceArgs {
  const TileJob* jobs;
  int* status;
  const int* score;
  const uint4* rec;
  const uint32_t* rec_tab;
  int tab_stride;
  const TileBlockInfo* blocks;
  const uint64_t* words;
  char* ops;
  const int64_t* ops_off;
  int* ops_begin;
  unsigned int* fail_count;
  int g;
  int lmax_words;
};

// BiWFA: both sides of every large sub-problem advanced in tiles up to the
// block in which phase 1 ends (the sides meet, or a side reaches its end or a
// border); the breakpoint kernel goes on from the start of that block.
struct BiTileArgs {
  int n;                       // sub-problems
  const int* act;              // active ones
  const int* n_act;
  const BiProblem* probs;
  const uint64_t* words;
  const uint64_t* rev_words;
  const int64_t* fwd_ppos;
  const int64_t* fwd_tpos;
  const int64_t* rev_ppos;
  const int64_t* rev_tpos;
  const int* plen_total;
  const int* tlen_total;
  int* state;                  // per side: kBiTileRows rows
  const int64_t* st_off;       // first int of a sub-problem's forward rows; its reverse rows follow
  int* done;                   // block in which phase 1 ends (INT_MAX: not yet)
  int* far;                    // [2][2 n]: by block parity, furthest antidiagonal of each side
  const int2* hull;            // [3][steps]: hull of the ranges up to each step, by the begin component
  int steps;                   // steps in the tables
  int blk;
  int lmax_words;
};
// Rows of a side: M, I1 and D1 of the last kBiTileAges steps of a block, by
// block parity and age (0: the latest).  The step kernels of a search need
// four; its overlap scans look one step further back.
constexpr int kBiTileAges = 5, kBiTileRows = 2 * 3 * kBiTileAges;
__host__ __device__ inline int bi_row(int par, int comp, int age) { return (3 * par + comp) * kBiTileAges + age; }

struct TileGeometry {
  int steps;                   // per block
  int useful;                  // diagonals per tile
  int state_rows;
  int step_rows;               // of the step kernels
  int dx, do1, de1, do2, de2;  // distances in steps (do2 = 0: no second gap)
};

// 0: no instance for these penalties.
int tile_shape(const Penalties& pen);
TileGeometry tile_geometry(int shape);
int bi_tile_steps();           // steps per block
int bi_tile_useful();          // diagonals per tile
hipError_t launch_bi_tile_init(const BiTileArgs& a, int* act, int* n_act, hipStream_t st);
hipError_t launch_bi_tile_block(const BiTileArgs& a, int problems, int tiles, hipStream_t st);
hipError_t launch_tile_fill(int* state, long long ints, hipStream_t st);
// The jobs of a pass from their slots, their score-0 rows and marks, the first
// active list (act, n_act) and the count of lost jobs.
hipError_t launch_tile_init(int shape, const TileArgs& a, int n, const TileSlot* slots, const TileSeqs& seqs, int* act,
                            int* n_act, int* lost, hipStream_t st);
hipError_t launch_tile_block(int shape, bool records, const TileArgs& a, int jobs, hipStream_t st);
hipError_t launch_tile_step_init(int shape, const StepArgs& a, const TileArgs& t, int n, int max_pitch, hipStream_t st);
hipError_t launch_tile_step(int shape, bool records, const StepArgs& a, int t, int jobs, int max_width, hipStream_t st);
// host_n[0]: the jobs left, host_n[kTileHostLost]: the jobs lost so far (with irr).
constexpr int kTileHostLost = 4;
hipError_t launch_tile_compact(const int* act, const int* n_act, const int* done, const int* irr, int ib, int* act2,
                               int* n_act2, int* lost, int* host_n, hipStream_t st);
hipError_t launch_tile_finish(int shape, const TileFinishArgs& a, hipStream_t st);
hipError_t launch_tile_backtrace(int shape, const TileTraceArgs& a, int n, hipStream_t st);

}  // namespace wfa
