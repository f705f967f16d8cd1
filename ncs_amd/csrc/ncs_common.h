// ncs_common.h -- shared device/host definitions of libncs_hip.so (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/ncs_hip.h"

namespace ncs {

constexpr int kTile = 16;          // tile edge (the reference's r_size = 16)
constexpr int kTilePix = 256;      // pixels per tile
constexpr int kWave = 64;          // gfx950 wavefront
constexpr int kWavesPerBlock = 4;  // 256-thread workgroups, one tile per wave
constexpr int kMaxWavesPerGroup = 4;  // persistent solver: waves per workgroup 1..4

// Work queue of the persistent solver: kQueues counters, one per XCD
// (workgroups are dispatched round-robin over the 8 XCDs), each on its own
// 128-byte line (see TileSchedule).
constexpr int kQueues = 8;
constexpr int kQueueStride = 32;   // unsigned ints between counters
constexpr size_t kQueueBytes = kQueues * kQueueStride * sizeof(unsigned int);
constexpr float kFitMin = 1.0e-6f; // negative-value guard (ncs.cl:45, ncs.c:169)

// Per-lane tables, kTableF4 16-byte entries per lane: the real-DFT basis
// entries in FP32 (two), the mask's even-even and odd-odd weights, the
// learned linear start's two coefficient sets, the basis entries again as
// FP16 hi/lo pairs for the FP16 matrix-core basis changes (four; see
// ncs_solver.hip, LdsTables), and the linear start's two slopes in
// ln(alpha) (kTableSlope, kTableSlope + 1).  The solver keeps entries
// kSolveTableFirst .. kSolveTableFirst + kSolveTableF4 - 1 in LDS; the
// slopes, read once per tile, stay in the global table.
constexpr int kTableF4 = 12;
constexpr int kSolveTableFirst = 2;
constexpr int kSolveTableF4 = 8;
constexpr int kTableSlope = 10;
constexpr int kTableLaneFloats = 4 * kTableF4;
constexpr int kTableFloats = kWave * kTableLaneFloats;

// Division of n < 2^31 by d >= 1 with one multiplication (Granlund and
// Montgomery 1994): with l = ceil(log2 d) and m = floor(2^(31 + l) / d) + 1,
// n / d = (n m) >> (31 + l).  d = 1 has no such m in 32 bits and takes 0.
inline unsigned int div_magic(unsigned int d) {
  if (d <= 1) return 0;
  int l = 0;
  while ((1ull << l) < d) l++;
  // l <= 31, and the quotient is below 2^32
  const unsigned long long p = 1ull << (31 + l);
  return (unsigned int)(p / d + 1);
}
#if defined(__HIPCC__)
__host__ __device__
#endif
inline unsigned int div_by(unsigned int n, unsigned int d, unsigned int magic) {
  if (magic == 0) return n;
  const unsigned int hi = (unsigned int)(((unsigned long long)n * magic) >> 32);
  return hi >> (31 - __builtin_clz(d - 1));  // l - 1
}

// One frame of a batch, as the kernel sees it.  A batch's tiles are claimed
// in frame-table order (`first`, increasing along the table); per-tile arrays
// (warm starts, tile outputs, iterations, status, cost) are indexed in the
// caller's frame order (`slot`).  The two differ when the host schedules the
// frames in another order than the caller passed them.
struct FrameDev {
  const float *data;
  const float *gamma;
  float *out;
  int H, W;
  int ds, gs, os;      // row strides (elements)
  float alpha;
  int geom;            // NCS_GEOM_*
  int ty;              // tiles along the fast axis
  int win;             // window side r of the reference geometry (even, 4..16);
                       // a window fills the top-left r x r of the 16 x 16 tile
  unsigned int ty_magic;  // div_magic(ty)
  long long first;     // schedule position of the frame's first tile
  long long slot;      // per-tile array index of the frame's first tile
};

// How a launch's tiles are shared out.  The first dyn0 tiles are static: the
// first `extra` waves own per_wave + 1 contiguous tiles each, the others
// per_wave.  The tiles from dyn0 on form kQueues ranges, one per XCD, that
// waves take from one by one with an atomic, their home range first, then
// the next one.
struct TileSchedule {
  unsigned int per_wave, extra;
  unsigned int dyn0;
};

// Arguments of the conv net's kernel over frames.
struct NetWarmArgs {
  const FrameDev *frames;      // device table, or nullptr: the inline one
  int n_frames;
  long long total;
  float *u0;                   // [tiles][256]
  const void *packs;
  const float *params;
};

// Solver parameters in the kernel's units.
struct SolveArgs {
  const FrameDev *frames;      // device table, or nullptr: the inline one
  int n_frames;
  long long total_tiles;
  TileSchedule sched;          // filled in by launch_solve
  unsigned int *queue;         // kQueues work-queue counters (kQueueBytes)
  unsigned int *queue_next;    // the next solve's, cleared by this one (or nullptr)
  const float *tables;         // [64][16] per-lane OTF/DFT tables
  const float *u0;             // [tiles][256] warm start or nullptr
  int *iterations;             // [tiles] or nullptr
  int *status;                 // [tiles] or nullptr
  float *cost;                 // [tiles] or nullptr
  int max_it;
  float eps;
  float eps2;                  // eps^2
  int ls;
  int max_ls;
  float ftol, gtol, xtol, min_step, max_step, stepm;
  int fallback;
  int precond;                 // spectral initial inverse Hessian (else s.y / y.y)
  int lin_start;               // learned linear start (coefficients in the tables)
  float lin_c;                 // its DC bias
  float lin_c1;                // the bias's slope in ln(alpha)
  float lin_aref;              // alpha the coefficients were fitted at
  int lin_slope;               // nonzero: the coefficients follow alpha
  float k_norm;                // bound on the NC Hessian's norm (row sums of the mask tables)
};

// A frame table of up to kInlineFrames frames travels in the kernel's
// arguments (read by scalar loads from the kernel-argument segment): no copy
// to the device before the launch and no table shared between launches.
// Larger ones are in device memory (`frames`).
constexpr int kInlineFrames = 32;

template <class Args>
struct WithFrames {
  Args args;
  FrameDev inl[kInlineFrames];
};
static_assert(sizeof(WithFrames<SolveArgs>) <= 4096, "kernel argument too large");

// Fills the inline table from n frames in host memory.
template <class Args>
inline void set_inline(WithFrames<Args> &w, const FrameDev *frames, int n) {
  for (int i = 0; i < n; i++) w.inl[i] = frames[i];
}

#if defined(__HIPCC__)
// The frame table seen through the constant address space (scalar loads into
// SGPRs; no kernel writes it).
typedef __attribute__((address_space(4))) const FrameDev FrameConst;

// The table of a kernel whose only argument is a WithFrames<Args>: `frames`,
// or the inline one when that is null.
template <class Args>
__device__ __forceinline__ const FrameConst *frame_table(const FrameDev *frames) {
  typedef __attribute__((address_space(4))) const char ConstByte;
  const FrameConst *inl =
      (const FrameConst *)((ConstByte *)__builtin_amdgcn_kernarg_segment_ptr() +
                           offsetof(WithFrames<Args>, inl));
  return frames != nullptr ? (const FrameConst *)frames : inl;
}
#endif

}  // namespace ncs
