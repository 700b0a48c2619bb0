// Host side of the scatter log (GradTargets): its pool, which gradients it
// takes, and its reduction.
#pragma once

#include <hip/hip_runtime.h>

#include "volpath.hpp"

namespace rcv {

// A pool of kLogPool chunks of kLogChunk 16-byte records (3.2 GB).
constexpr unsigned kLogPool = 786432;

struct LogBuf {
  float4 *rec = nullptr;
  unsigned *ctl = nullptr;   // chunks drawn
  unsigned *meta = nullptr;  // kLogPool chunk bins and record counts
};

// The scatter log of one launch; target.g null: none, the scatter-adds stay
// atomics.
struct LogLaunch {
  LogBuf buf;
  LogTarget target{};
  int tiles = 0;
};

// Voxels per reduction tile on the current device.
int log_tile();

// Whether the density gradient `g` of medium m of scene s can be logged (its
// grid fits the reduction tiles and a footprint spans at most two of them);
// fills target's grid and returns its tiles, or 0.
int log_target(const Scene *s, const MediumInfo &m, float *g, LogTarget &target);

// Points G at the pool for gradient `param` with chunk bins from bin0 on.
void log_into(const LogBuf &buf, int param, unsigned bin0, GradTargets &G);

// Sets up the log of a launch on `stream` for the density gradient of the
// first heterogeneous medium that has one, with the stream's pool. Without
// memory for it, or with fewer than `min_samples` (per reduction tile) of the
// launch's `samples`, the scatter-adds stay atomics.
void open_log(const Scene *s, const GradTargets &G, hipStream_t stream, LogLaunch &log, GradTargets &GL,
              int64_t samples = 0, int64_t min_samples = 0);

// Adds the records of a launch to its gradient.
void reduce_log(const LogLaunch &log, const GradTargets &GL, hipStream_t stream);

// A batch's log: emptied before its adjoint launches, its records added to
// the gradients of n targets (in device memory, `first` the first of them)
// of `tiles` tiles in all.
void zero_log(const LogBuf &buf, hipStream_t stream);
void reduce_log_batch(const LogBuf &buf, const LogTarget &first, const LogTarget *targets, int n, int tiles,
                      hipStream_t stream);

// A pool for a batch's lifetime on the current device: the one kept there,
// or a new one. False without memory. Given back once nothing uses it, it is
// kept for the next batch, or freed if one is kept already.
bool take_log_pool(LogBuf &buf);
void give_log_pool(const LogBuf &buf, int dev);

}  // namespace rcv
