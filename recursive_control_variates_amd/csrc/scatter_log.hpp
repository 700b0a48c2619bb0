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
  unsigned *ctl = nullptr;   // chunks drawn, bins' sums of magnitudes
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

// Reduction tiles per bin of a large grid's log, as a power of two, at most
// (every tile of a bin reads the bin's records), and the samples per tile and
// in all from which a launch on such a grid is logged: below them the
// reduction's cost per tile, and the chunks its wavefronts leave nearly empty,
// weigh more than the atomics, which a launch that does not fill the device
// hides behind its longest path. Adjoint call with atomics / logged, one
// view, optical depth ~3: 80^3 (32 tiles) with 128 Ki samples 1.01 / 1.09 ms,
// 256 Ki 1.03 / 1.08, 512 Ki 1.64 / 1.35; 100^3 (62) with 512 Ki 1.63 / 1.57,
// 1 Mi 3.04 / 2.26; 128^3 (128) with 512 Ki 1.70 / 1.90, 1 Mi 3.09 / 2.76,
// 2 Mi 5.45 / 3.99; 150^3 (206) with 2 Mi 5.39 / 5.09. Optical depth ~15:
// 80^3 with 512 Ki 12.3 / 3.7 ms, 128^3 with 1 Mi 24.9 / 10.8.
constexpr int kLogWide = 4;
constexpr int64_t kWideLogSamples = 8192;
constexpr int64_t kWideLogLaunch = int64_t(1) << 19;

// Whether the density gradient `g` of medium m of scene s can be logged with
// bins of up to 2^wide reduction tiles (its grid fits the bins and a footprint
// spans at most two of them, and every medium over the grid places it alike: a
// record holds its world point, from which the reduction forms the footprint
// with the target's one box); fills target's grid and returns its tiles, or 0.
int log_target(const Scene *s, const MediumInfo &m, float *g, int wide, LogTarget &target);

// Points G at the pool for gradient `param` with chunk bins of 2^shift voxels
// from bin0 on.
void log_into(const LogBuf &buf, int param, unsigned bin0, int shift, GradTargets &G);

// Sets up the log of a launch on `stream` for the density gradient of the
// first heterogeneous medium that has one, with the stream's pool. Without
// memory for it, under capture, or with fewer of the launch's `samples` than the bins ask for
// (kWideLogSamples; `min_samples` per tile for bins of one tile), the
// scatter-adds stay atomics.
void open_log(const Scene *s, const GradTargets &G, hipStream_t stream, LogLaunch &log, GradTargets &GL,
              int64_t samples, int64_t min_samples = 0);

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
