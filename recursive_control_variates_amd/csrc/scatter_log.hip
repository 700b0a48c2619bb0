// Scatter log of the volume adjoints: pools and reduction (GradTargets,
// scatter_density).

#include "scatter_log.hpp"

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <utility>

#include "common.hpp"

namespace rcv {
namespace {

// Reduction. A block takes one tile of a gradient and the chunks c = x (mod
// gridDim.x) of the launch, and adds up the records of those whose bin
// reaches into the tile: the tile's own, the seams below and above it. (A
// record is read once, or twice when it lies across a seam; every block
// reads the bins of its share of the chunks, 4 bytes each beside their 4 KB
// of records.) The block looks at kReduceBlock chunks at a time, lists those
// it takes in LDS and reads them kStepChunks per step: thread i slot i %
// kLogChunk of kReduceUnroll of them, all loads in flight together (unused
// slots are read, every index stays inside the pool, and skipped). The
// records of one chunk come from one wavefront of the adjoint, whose lanes
// trace neighbouring pixels; the 8-lane groups of a wavefront take their
// chunks in rotated order so that one instruction adds records of several
// chunks.
constexpr int kReduceBlock = 1024;
constexpr int kReduceUnroll = 8;
constexpr unsigned kChunkGroups = unsigned(kReduceBlock) / kLogChunk;
constexpr unsigned kStepChunks = kChunkGroups * kReduceUnroll;
constexpr int kLogSplits = 64;  // blocks per tile
static_assert(kReduceBlock % int(kLogChunk) == 0, "a reduction block covers whole chunks");

// Calls fn(record) for each record of the block's share that reaches `tile`.
// picked: kReduceBlock words of LDS, n_picked one.
template <class Fn>
__device__ inline void log_block_records(const float4 *__restrict__ rec, const unsigned *__restrict__ meta,
                                         unsigned drawn, unsigned bin0, int tile, unsigned *picked,
                                         unsigned *n_picked, Fn &&fn) {
  const unsigned slot = threadIdx.x % kLogChunk;
  const unsigned sub = threadIdx.x / kLogChunk;
  const unsigned grp = (threadIdx.x >> 3) % kReduceUnroll;
  constexpr unsigned kFillMask = (1u << kLogFillBits) - 1u;
  for (unsigned c0 = blockIdx.x; c0 < drawn; c0 += gridDim.x * unsigned(kReduceBlock)) {
    if (threadIdx.x == 0) *n_picked = 0;
    __syncthreads();
    const unsigned c = c0 + threadIdx.x * gridDim.x;
    const unsigned m = c < drawn ? meta[c] : 0u;
    const int b = int(m >> kLogFillBits) - int(bin0);
    const bool mine = (m & kFillMask) != 0 && (b == tile || b == kLogMaxTiles + tile ||
                                               (tile > 0 && b == kLogMaxTiles + tile - 1));
    if (mine) picked[atomicAdd(n_picked, 1u)] = c;
    __syncthreads();
    const unsigned nb = *n_picked;
    for (unsigned p0 = 0; p0 < nb; p0 += kStepChunks) {
      unsigned id[kReduceUnroll], n[kReduceUnroll];
      float4 e[kReduceUnroll];
#pragma unroll
      for (int u = 0; u < kReduceUnroll; ++u) {
        const unsigned j = p0 + sub + kChunkGroups * ((grp + unsigned(u)) % kReduceUnroll);
        id[u] = j < nb ? picked[j] : picked[0];
        n[u] = j < nb ? meta[id[u]] & kFillMask : 0u;
      }
#pragma unroll
      for (int u = 0; u < kReduceUnroll; ++u) e[u] = rec[size_t(id[u]) * kLogChunk + slot];
#pragma unroll
      for (int u = 0; u < kReduceUnroll; ++u)
        if (slot < n[u]) fn(e[u]);
    }
    __syncthreads();
  }
}

// Calls add(voxel - lo, value x weight) for the corners of a record that
// fall in [lo, hi): the products of scatter_grid over the footprint of the
// record's point.
template <class Add>
__device__ inline void record_corners(const float4 &e, const LogTarget &T, int lo, int hi, Add &&add) {
  GridFoot f;
  grid_footprint(T, T, v3(e.x, e.y, e.z), f);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int idx = f.idx(q);
    if (idx >= lo && idx < hi) add(idx - lo, e.w * f.w(q));
  }
}

// Adds the scatter log of a launch to its gradients, tile by tile (block y:
// a tile of one of n targets; `one` for n = 1). The tile is summed in LDS in
// 64-bit fixed point: integer LDS atomics run ~5x faster than float ones
// here. A first pass over the share's values finds its record count N and
// largest magnitude M; terms are scaled by 2^s with M N 2^s <= 2^62, so no
// partial sum overflows and each term is kept to ~2^-44 of M (float atomics
// keep 2^-24 of the running sum). A share holding a non-finite value is
// summed with float atomics as it stands.
__global__ __launch_bounds__(kReduceBlock) void log_reduce_kernel(const float4 *__restrict__ rec,
                                                                  const unsigned *__restrict__ ctl,
                                                                  const unsigned *__restrict__ meta, unsigned nchunks,
                                                                  LogTarget one, const LogTarget *__restrict__ many,
                                                                  int n, int tile_voxels) {
  extern __shared__ long long acc[];  // tile words (floats in the first half for a non-finite share)
  __shared__ float wave_max[kReduceBlock / 64];
  __shared__ unsigned wave_count[kReduceBlock / 64];
  __shared__ unsigned picked[kReduceBlock];
  __shared__ unsigned n_picked;
  LogTarget T = one;
  if (n > 1) {
    int k = 0;
    while (k + 1 < n && many[k + 1].tile0 <= int(blockIdx.y)) ++k;
    T = many[k];
  }
  const int tile = int(blockIdx.y) - T.tile0;
  const int lo = tile * tile_voxels;
  const int hi = min(lo + tile_voxels, T.nx * T.ny * T.nz);
  const unsigned drawn = min(*ctl, nchunks);
  float m = 0.0f;
  unsigned total = 0;
  log_block_records(rec, meta, drawn, T.bin0, tile, picked, &n_picked, [&](const float4 &e) {
    const float a = fabsf(e.w);
    m = (a <= m) ? m : (a == a ? a : INFINITY);  // NaN and inf both give inf
    ++total;
  });
  for (int off = 32; off > 0; off >>= 1) {
    m = fmaxf(m, __shfl_xor(m, off, 64));
    total += __shfl_xor(total, off, 64);
  }
  if ((threadIdx.x & 63u) == 0) {
    wave_max[threadIdx.x >> 6] = m;
    wave_count[threadIdx.x >> 6] = total;
  }
  __syncthreads();
  m = 0.0f;
  total = 0;
  for (int w = 0; w < kReduceBlock / 64; ++w) {
    m = fmaxf(m, wave_max[w]);
    total += wave_count[w];
  }
  if (total == 0 || m == 0.0f) return;
  if (isfinite(m)) {
    int em = 0, en = 0;
    (void)frexpf(m, &em);               // m < 2^em
    (void)frexpf(float(total), &en);    // total <= 2^en
    const int sc = 62 - em - en;
    for (int v = threadIdx.x; v < tile_voxels; v += blockDim.x) acc[v] = 0;
    __syncthreads();
    log_block_records(rec, meta, drawn, T.bin0, tile, picked, &n_picked, [&](const float4 &e) {
      record_corners(e, T, lo, hi, [&](int a, float t) {
        atomicAdd(reinterpret_cast<unsigned long long *>(&acc[a]), (unsigned long long)__float2ll_rn(ldexpf(t, sc)));
      });
    });
    __syncthreads();
    for (int v = threadIdx.x; v < hi - lo; v += blockDim.x)
      if (acc[v] != 0) atomicAdd(&T.g[lo + v], ldexpf(__ll2float_rn(acc[v]), -sc));
  } else {
    float *facc = reinterpret_cast<float *>(acc);
    for (int v = threadIdx.x; v < tile_voxels; v += blockDim.x) facc[v] = 0.0f;
    __syncthreads();
    log_block_records(rec, meta, drawn, T.bin0, tile, picked, &n_picked, [&](const float4 &e) {
      record_corners(e, T, lo, hi, [&](int a, float t) { atomicAdd(&facc[a], t); });
    });
    __syncthreads();
    for (int v = threadIdx.x; v < hi - lo; v += blockDim.x)
      if (facc[v] != 0.0f) atomicAdd(&T.g[lo + v], facc[v]);
  }
}

__global__ void zero_ctl_kernel(unsigned *p) { *p = 0u; }

int allocate(LogBuf &out) {
  LogBuf nb;
  hipError_t e = hipMalloc(&nb.rec, size_t(kLogPool) * kLogChunk * sizeof(float4));
  if (e == hipSuccess) e = hipMalloc(&nb.ctl, sizeof(unsigned));
  if (e == hipSuccess) e = hipMalloc(&nb.meta, size_t(kLogPool) * sizeof(unsigned));
  if (e != hipSuccess) {
    (void)hipFree(nb.rec);
    (void)hipFree(nb.ctl);
    (void)hipFree(nb.meta);
    (void)hipGetLastError();
    return hip_fail(e, "scatter log: allocation");
  }
  out = nb;
  return RCV_OK;
}

// The pool of single launches: one per (device, stream), kept for the
// process (launches on one stream run in order; other streams get their own).
// None is allocated while the stream is being captured, which an allocation
// would break off: a launch captured before any other has no log.
int stream_pool(hipStream_t stream, LogBuf &out) {
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, LogBuf> bufs;
  int dev = 0;
  RCV_TRY_HIP(hipGetDevice(&dev), "hipGetDevice");
  std::lock_guard<std::mutex> lock(mu);
  const auto key = std::make_pair(dev, stream);
  auto it = bufs.find(key);
  if (it == bufs.end()) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
      (void)hipGetLastError();
      return 1;
    }
    if (capture != hipStreamCaptureStatusNone) return 1;
    LogBuf nb;
    if (int rc = allocate(nb)) return rc;
    it = bufs.emplace(key, nb).first;
  }
  out = it->second;
  return RCV_OK;
}

// The pool kept per device for batches.
std::mutex kept_mu;
std::map<int, LogBuf> kept;

// Chunks of the pool a launch may draw: kLogPool, or fewer when the
// environment sets RCV_SCATTER_LOG_CHUNKS (a test of the adjoint past the
// pool's end, where the scatter-adds fall back to atomics).
unsigned log_pool_chunks() {
  const char *e = std::getenv("RCV_SCATTER_LOG_CHUNKS");
  if (!e || !*e) return kLogPool;
  char *end = nullptr;
  const unsigned long v = std::strtoul(e, &end, 10);
  if (end == e || *end != '\0' || v == 0) return kLogPool;
  return unsigned(std::min<unsigned long>(v, kLogPool));
}

}  // namespace

// 16384 voxels (a 64-bit word each, 128 KB of LDS), or the largest power of
// two the device's LDS per block holds.
int log_tile() {
  static std::mutex mu;
  static std::map<int, int> tiles;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lock(mu);
  auto it = tiles.find(dev);
  if (it != tiles.end()) return it->second;
  int max_lds = 0;
  (void)hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  constexpr size_t kStatic = 4608;  // the kernel's static LDS, rounded up
  int tile = 16384;
  while (tile > 1024 && size_t(tile) * sizeof(long long) + kStatic > size_t(max_lds)) tile >>= 1;
  if (tile * sizeof(long long) > 65536 &&
      hipFuncSetAttribute(reinterpret_cast<const void *>(log_reduce_kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, int(tile * sizeof(long long))) != hipSuccess) {
    (void)hipGetLastError();
    tile = 65536 / int(sizeof(long long)) / 2;
  }
  tiles[dev] = tile;
  return tile;
}

int log_target(const Scene *s, const MediumInfo &m, float *g, LogTarget &target) {
  const int tile = log_tile();
  const Param &P = s->params[m.sigma_param];
  const int64_t n = int64_t(P.nx) * P.ny * P.nz;
  if (n > int64_t(tile) * kLogMaxTiles || int64_t(P.nx) * P.ny + P.nx + 1 > tile) return 0;
  target.g = g;
  target.nx = P.nx;
  target.ny = P.ny;
  target.nz = P.nz;
  for (int k = 0; k < 3; ++k) {
    target.lo[k] = m.lo[k];
    target.hi[k] = m.hi[k];
  }
  target.bin0 = 0;
  target.tile0 = 0;
  return int((n + tile - 1) / tile);
}

void log_into(const LogBuf &buf, int param, unsigned bin0, GradTargets &G) {
  G.log_rec = buf.rec;
  G.log_ctl = buf.ctl;
  G.log_meta = buf.meta;
  G.log_chunks = log_pool_chunks();
  G.log_bin0 = bin0;
  G.log_shift = __builtin_ctz(unsigned(log_tile()));
  G.log_param = param;
}

void open_log(const Scene *s, const GradTargets &G, hipStream_t stream, LogLaunch &log, GradTargets &GL,
              int64_t samples, int64_t min_samples) {
  for (const MediumInfo &M : s->media) {
    if (M.homogeneous || M.sigma_param < 0 || !G.g[M.sigma_param]) continue;
    log.tiles = log_target(s, M, G.g[M.sigma_param], log.target);
    if (log.tiles > 0 && samples >= min_samples * log.tiles && stream_pool(stream, log.buf) == RCV_OK) {
      log_into(log.buf, M.sigma_param, 0, GL);
      hipLaunchKernelGGL(zero_ctl_kernel, dim3(1), dim3(1), 0, stream, log.buf.ctl);
    } else {
      log.target.g = nullptr;
    }
    return;
  }
}

void reduce_log(const LogLaunch &log, const GradTargets &GL, hipStream_t stream) {
  if (!log.target.g) return;
  const int tile = log_tile();
  hipLaunchKernelGGL(log_reduce_kernel, dim3(kLogSplits, log.tiles), dim3(kReduceBlock),
                     size_t(tile) * sizeof(long long), stream, log.buf.rec, log.buf.ctl, log.buf.meta, GL.log_chunks,
                     log.target, static_cast<const LogTarget *>(nullptr), 1, tile);
}

void zero_log(const LogBuf &buf, hipStream_t stream) {
  hipLaunchKernelGGL(zero_ctl_kernel, dim3(1), dim3(1), 0, stream, buf.ctl);
}

void reduce_log_batch(const LogBuf &buf, const LogTarget &first, const LogTarget *targets, int n, int tiles,
                      hipStream_t stream) {
  const int tile = log_tile();
  // about 4096 blocks
  const int splits = std::min(kLogSplits, std::max(4, 4096 / tiles));
  hipLaunchKernelGGL(log_reduce_kernel, dim3(splits, tiles), dim3(kReduceBlock), size_t(tile) * sizeof(long long),
                     stream, buf.rec, buf.ctl, buf.meta, log_pool_chunks(), first, targets, n, tile);
}

bool take_log_pool(LogBuf &buf) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  {
    std::lock_guard<std::mutex> lock(kept_mu);
    auto it = kept.find(dev);
    if (it != kept.end()) {
      buf = it->second;
      kept.erase(it);
      return true;
    }
  }
  return allocate(buf) == RCV_OK;
}

void give_log_pool(const LogBuf &buf, int dev) {
  {
    std::lock_guard<std::mutex> lock(kept_mu);
    if (kept.emplace(dev, buf).second) return;
  }
  (void)hipFree(buf.rec);
  (void)hipFree(buf.ctl);
  (void)hipFree(buf.meta);
}

}  // namespace rcv
