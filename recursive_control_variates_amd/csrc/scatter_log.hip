// Scatter log of the volume adjoints: pools and reduction (GradTargets,
// scatter_density).

#include "boxpath.hpp"
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
// kLogChunk of kReduceUnroll of them, all loads in flight together. The
// records of one chunk come from one wavefront of the adjoint, whose lanes
// trace neighbouring pixels; the 8-lane groups of a wavefront take their
// chunks in rotated order so that one instruction adds records of several
// chunks.
//
// A grid of more than kLogMaxTiles tiles has bins of several tiles, and each
// of them reads its bin's records: 8 times at 128^3, whose step with an albedo
// grid (192^2 per view, 8 samples) takes 8.8 ms (adjoint 2.7, reduction 2.3,
// sums 0.09), with atomics 11.7 (adjoint 7.2). Those bins' sums
// come from one pass over all records (log_bound_kernel) instead of one per
// tile: 2.95 -> 2.16 ms of reduction.
//
// Chunks that are mostly empty (SPARSE: a short launch leaves every
// wavefront a few records in each of up to 31 chunks) are read 64 slots of
// kReduceUnroll chunks per wavefront instead, as long as one of them has more.
// With bins of several tiles a block counts its records first and takes this
// walk when fewer than half the slots are used: the 128^3 adjoint call of
// 512 Ki thin samples 2.63 -> 1.90 ms; full chunks are read better as above
// (that step by rows 9.1 ms).
constexpr int kReduceBlock = 1024;
constexpr int kReduceUnroll = 8;
constexpr unsigned kChunkGroups = unsigned(kReduceBlock) / kLogChunk;
constexpr unsigned kStepChunks = kChunkGroups * kReduceUnroll;
constexpr unsigned kSparseChunks = unsigned(kReduceBlock) / 64u * unsigned(kReduceUnroll);
// Blocks per tile: an odd number, so that the chunks c = x (mod it) of a block
// lie at every place of the draws of kLogDraw chunks. In a short launch the
// first of a wavefront's draw hold records and the last are empty: with 64
// blocks an eighth of them got all first chunks (two tiles, 262144 samples:
// 203 us, with 63 blocks 88).
constexpr int kLogSplits = 63;  // at most
constexpr int kLogMinSplits = 17;
constexpr int odd_splits(int n) { return n | 1; }
static_assert(kLogSplits % 2 == 1 && kLogMinSplits % 2 == 1 && kLogDraw % 2 == 0, "odd against the draw size");
static_assert(kReduceBlock % int(kLogChunk) == 0 && kLogChunk % 64 == 0,
              "a reduction block covers whole chunks, a wavefront whole rows of one");

// The bins whose records can reach the tile [lo, hi) of T: the one it lies in,
// and the seams at either end of that which footprints on the tile can cross.
struct TileBins {
  int bin;
  bool before, after;
  __device__ TileBins(const LogTarget &T, int lo, int hi) : bin(lo >> T.shift) {
    const int span = T.nx * T.ny + T.nx + 1;
    before = bin > 0 && lo - (bin << T.shift) < span;
    after = hi + span > ((bin + 1) << T.shift);
  }
  __device__ bool holds(int b) const {
    return b == bin || (after && b == kLogMaxTiles + bin) || (before && b == kLogMaxTiles + bin - 1);
  }
};

// Calls fn(record) for each record of the block's share that reaches `tile`.
// picked: kReduceBlock words of LDS, n_picked one.
template <bool SPARSE, class Fn>
__device__ inline void log_block_records(const float4 *__restrict__ rec, const unsigned *__restrict__ meta,
                                         unsigned drawn, const LogTarget &T, const TileBins &bins,
                                         unsigned *picked, unsigned *n_picked, Fn &&fn) {
  const unsigned slot = threadIdx.x % kLogChunk;
  const unsigned sub = threadIdx.x / kLogChunk;
  const unsigned lane = threadIdx.x & 63u;
  const unsigned wave_sub = (threadIdx.x >> 6) * unsigned(kReduceUnroll);
  const unsigned grp = (threadIdx.x >> 3) % kReduceUnroll;
  constexpr unsigned kFillMask = (1u << kLogFillBits) - 1u;
  for (unsigned c0 = blockIdx.x; c0 < drawn; c0 += gridDim.x * unsigned(kReduceBlock)) {
    if (threadIdx.x == 0) *n_picked = 0;
    __syncthreads();
    const unsigned c = c0 + threadIdx.x * gridDim.x;
    const unsigned m = c < drawn ? meta[c] : 0u;
    const bool mine = (m & kFillMask) != 0 && bins.holds(int(m >> kLogFillBits) - int(T.bin0));
    if (mine) picked[atomicAdd(n_picked, 1u)] = c;
    __syncthreads();
    const unsigned nb = *n_picked;
    if constexpr (SPARSE) {
      for (unsigned p0 = 0; p0 < nb; p0 += kSparseChunks) {
        unsigned id[kReduceUnroll], n[kReduceUnroll], most = 0;
#pragma unroll
        for (int u = 0; u < kReduceUnroll; ++u) {
          const unsigned j = p0 + wave_sub + (grp + unsigned(u)) % kReduceUnroll;
          id[u] = j < nb ? picked[j] : picked[0];
          n[u] = j < nb ? meta[id[u]] & kFillMask : 0u;
          most = max(most, n[u]);
        }
        for (unsigned row = 0; row < most; row += 64u) {
          float4 e[kReduceUnroll];
#pragma unroll
          for (int u = 0; u < kReduceUnroll; ++u)
            if (row + lane < n[u]) e[u] = rec[size_t(id[u]) * kLogChunk + row + lane];
#pragma unroll
          for (int u = 0; u < kReduceUnroll; ++u)
            if (row + lane < n[u]) fn(e[u]);
        }
      }
    } else {
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
        for (int u = 0; u < kReduceUnroll; ++u)
          if (slot < n[u]) e[u] = rec[size_t(id[u]) * kLogChunk + slot];
#pragma unroll
        for (int u = 0; u < kReduceUnroll; ++u)
          if (slot < n[u]) fn(e[u]);
      }
    }
    __syncthreads();
  }
}

// grid_footprint of the records' points, the extents' reciprocals formed once
// (UniformDiv rounds as the division does, so the footprints are the same).
struct RecordGrid {
  UniformDiv ex, ey, ez;
  __device__ explicit RecordGrid(const LogTarget &T)
      : ex(T.hi[0] - T.lo[0]), ey(T.hi[1] - T.lo[1]), ez(T.hi[2] - T.lo[2]) {}
};

// Calls add(voxel - lo, value x weight) for the corners of a record that
// fall in [lo, hi): the products of scatter_grid over the footprint of the
// record's point. A footprint without one is passed over before its weights.
template <class Add>
__device__ inline void record_corners(const float4 &e, const LogTarget &T, const RecordGrid &D, int lo, int hi,
                                      Add &&add) {
  GridFoot f;
  grid_footprint_at(T, D.ex(e.x - T.lo[0]), D.ey(e.y - T.lo[1]), D.ez(e.z - T.lo[2]), f);
  if (f.base >= hi || f.base + f.dx + f.dy + f.dz < lo) return;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int idx = f.idx(q);
    if (idx >= lo && idx < hi) add(idx - lo, e.w * f.w(q));
  }
}

// Sum of the magnitudes of each bin's records, for a log whose bins hold
// several tiles: one pass over the records instead of one per tile.
constexpr int kBoundBlock = int(kLogChunk);
constexpr int kBoundUnroll = 4;
constexpr int kBoundBlocks = 2048;
__global__ __launch_bounds__(kBoundBlock) void log_bound_kernel(const float4 *__restrict__ rec,
                                                                const unsigned *__restrict__ ctl,
                                                                const unsigned *__restrict__ meta, unsigned nchunks,
                                                                float *bound) {
  __shared__ float sum[kLogBins];
  if (threadIdx.x < unsigned(kLogBins)) sum[threadIdx.x] = 0.0f;
  __syncthreads();
  const unsigned drawn = min(*ctl, nchunks);
  constexpr unsigned kFillMask = (1u << kLogFillBits) - 1u;
  for (unsigned c0 = blockIdx.x; c0 < drawn; c0 += gridDim.x * kBoundUnroll) {
    unsigned m[kBoundUnroll];
    float w[kBoundUnroll];
#pragma unroll
    for (int u = 0; u < kBoundUnroll; ++u) {
      const unsigned c = c0 + unsigned(u) * gridDim.x;
      m[u] = c < drawn ? meta[c] : 0u;
      w[u] = threadIdx.x < (m[u] & kFillMask) ? rec[size_t(c) * kLogChunk + threadIdx.x].w : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kBoundUnroll; ++u) {
      float t = fabsf(w[u]);
      for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
      if ((threadIdx.x & 63u) == 0 && t != 0.0f) atomicAdd(&sum[(m[u] >> kLogFillBits) % unsigned(kLogBins)], t);
    }
  }
  __syncthreads();
  if (threadIdx.x < unsigned(kLogBins) && sum[threadIdx.x] != 0.0f) atomicAdd(bound + threadIdx.x, sum[threadIdx.x]);
}

// Adds the scatter log of a launch to its gradients, tile by tile (block y:
// a tile of one of n targets; `one` for n = 1). The tile is summed in LDS in
// 64-bit fixed point: integer LDS atomics run ~5x faster than float ones
// here. A first pass over the share finds the sum M of its records'
// magnitudes; terms are scaled by 2^s with M 2^s <= 2^62 (float rounding adds
// less than 2^-9 to that), so no partial sum overflows and each term is kept to
// 2^-62 of M: as exactly as its float value for voxels down to 2^-38 of M,
// where float atomics keep 2^-24 of the running sum. (The largest magnitude
// times the count in place of M, up to 2^23 times as much, cost as many bits.)
// A share holding a non-finite value is summed with float atomics as it
// stands. WIDE: a log whose bins hold several tiles; M is then its bins' sum
// (`bound`), over all shares.
template <bool WIDE>
__global__ __launch_bounds__(kReduceBlock) void log_reduce_kernel(const float4 *__restrict__ rec,
                                                                  const unsigned *__restrict__ ctl,
                                                                  const unsigned *__restrict__ meta, unsigned nchunks,
                                                                  LogTarget one, const LogTarget *__restrict__ many,
                                                                  int n, int tile_voxels,
                                                                  const float *__restrict__ bound) {
  extern __shared__ long long acc[];  // tile words (floats in the first half for a non-finite share)
  __shared__ float wave_sum[kReduceBlock / 64];
  __shared__ unsigned wave_count[kReduceBlock / 64];
  __shared__ unsigned wave_chunks[kReduceBlock / 64];
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
  const TileBins bins(T, lo, hi);
  const RecordGrid div(T);
  float m = 0.0f;
  unsigned total = 0, chunks = 0;
  if constexpr (WIDE) {
    // the bins' sums are known; how full the chunks are
    for (unsigned c = blockIdx.x + threadIdx.x * gridDim.x; c < drawn; c += gridDim.x * unsigned(kReduceBlock)) {
      const unsigned w = meta[c];
      const unsigned fill = w & ((1u << kLogFillBits) - 1u);
      if (fill != 0 && bins.holds(int(w >> kLogFillBits) - int(T.bin0))) {
        total += fill;
        ++chunks;
      }
    }
  } else {
    log_block_records<false>(rec, meta, drawn, T, bins, picked, &n_picked, [&](const float4 &e) { m += fabsf(e.w); });
  }
  for (int off = 32; off > 0; off >>= 1) {
    m += __shfl_xor(m, off, 64);
    if constexpr (WIDE) {
      total += __shfl_xor(total, off, 64);
      chunks += __shfl_xor(chunks, off, 64);
    }
  }
  if ((threadIdx.x & 63u) == 0) {
    wave_sum[threadIdx.x >> 6] = m;
    wave_count[threadIdx.x >> 6] = total;
    wave_chunks[threadIdx.x >> 6] = chunks;
  }
  __syncthreads();
  if constexpr (WIDE) {
    total = chunks = 0;
    for (int w = 0; w < kReduceBlock / 64; ++w) {
      total += wave_count[w];
      chunks += wave_chunks[w];
    }
    if (total == 0) return;
    m = bound[bins.bin] + (bins.after ? bound[kLogMaxTiles + bins.bin] : 0.0f) +
        (bins.before ? bound[kLogMaxTiles + bins.bin - 1] : 0.0f);
  } else {
    m = 0.0f;
    for (int w = 0; w < kReduceBlock / 64; ++w) m += wave_sum[w];
  }
  if (m == 0.0f) return;
  if (isfinite(m)) {
    int em = 0;
    (void)frexpf(m, &em);  // m < 2^em
    const int sc = 62 - em;
    for (int v = threadIdx.x; v < tile_voxels; v += blockDim.x) acc[v] = 0;
    __syncthreads();
    // (scaled before the weights: the same products times 2^sc)
    auto add = [&](const float4 &e) {
      record_corners(make_float4(e.x, e.y, e.z, ldexpf(e.w, sc)), T, div, lo, hi, [&](int a, float t) {
        atomicAdd(reinterpret_cast<unsigned long long *>(&acc[a]), (unsigned long long)__float2ll_rn(t));
      });
    };
    if (WIDE && total < chunks * (kLogChunk / 2))
      log_block_records<WIDE>(rec, meta, drawn, T, bins, picked, &n_picked, add);
    else
      log_block_records<false>(rec, meta, drawn, T, bins, picked, &n_picked, add);
    __syncthreads();
    for (int v = threadIdx.x; v < hi - lo; v += blockDim.x)
      if (acc[v] != 0) atomicAdd(&T.g[lo + v], ldexpf(__ll2float_rn(acc[v]), -sc));
  } else {
    float *facc = reinterpret_cast<float *>(acc);
    for (int v = threadIdx.x; v < tile_voxels; v += blockDim.x) facc[v] = 0.0f;
    __syncthreads();
    log_block_records<false>(rec, meta, drawn, T, bins, picked, &n_picked, [&](const float4 &e) {
      record_corners(e, T, div, lo, hi, [&](int a, float t) { atomicAdd(&facc[a], t); });
    });
    __syncthreads();
    for (int v = threadIdx.x; v < hi - lo; v += blockDim.x)
      if (facc[v] != 0.0f) atomicAdd(&T.g[lo + v], facc[v]);
  }
}

__global__ void zero_ctl_kernel(unsigned *p) { p[threadIdx.x] = 0u; }

// Chunks drawn, then the bins' sums (log_bound_kernel).
constexpr int kCtlWords = 1 + kLogBins;

int allocate(LogBuf &out) {
  const RelaxedCapture relaxed;
  LogBuf nb;
  hipError_t e = hipMalloc(&nb.rec, size_t(kLogPool) * kLogChunk * sizeof(float4));
  if (e == hipSuccess) e = hipMalloc(&nb.ctl, kCtlWords * sizeof(unsigned));
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
// A captured launch has none: its graph is replayed on any stream, beside
// launches that log into the pool of the capture's.
int stream_pool(hipStream_t stream, LogBuf &out) {
  if (capturing(stream)) return 1;
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, LogBuf> bufs;
  int dev = 0;
  RCV_TRY_HIP(hipGetDevice(&dev), "hipGetDevice");
  std::lock_guard<std::mutex> lock(mu);
  const auto key = std::make_pair(dev, stream);
  auto it = bufs.find(key);
  if (it == bufs.end()) {
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
      (hipFuncSetAttribute(reinterpret_cast<const void *>(log_reduce_kernel<false>),
                           hipFuncAttributeMaxDynamicSharedMemorySize, int(tile * sizeof(long long))) != hipSuccess ||
       hipFuncSetAttribute(reinterpret_cast<const void *>(log_reduce_kernel<true>),
                           hipFuncAttributeMaxDynamicSharedMemorySize, int(tile * sizeof(long long))) != hipSuccess)) {
    (void)hipGetLastError();
    tile = 65536 / int(sizeof(long long)) / 2;
  }
  tiles[dev] = tile;
  return tile;
}

int log_target(const Scene *s, const MediumInfo &m, float *g, int wide, LogTarget &target) {
  for (const MediumInfo &o : s->media)
    if (!o.homogeneous && o.sigma_param == m.sigma_param &&
        !(std::equal(o.lo, o.lo + 3, m.lo) && std::equal(o.hi, o.hi + 3, m.hi)))
      return 0;
  const int tile = log_tile();
  const Param &P = s->params[m.sigma_param];
  const int64_t n = int64_t(P.nx) * P.ny * P.nz, span = int64_t(P.nx) * P.ny + P.nx + 1;
  int extra = 0;
  while (extra <= wide && (n > (int64_t(tile) << extra) * kLogMaxTiles || span > (int64_t(tile) << extra))) ++extra;
  if (extra > wide) return 0;
  target.shift = __builtin_ctz(unsigned(tile)) + extra;
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

void log_into(const LogBuf &buf, int param, unsigned bin0, int shift, GradTargets &G) {
  G.log_rec = buf.rec;
  G.log_ctl = buf.ctl;
  G.log_meta = buf.meta;
  G.log_chunks = log_pool_chunks();
  G.log_bin0 = bin0;
  G.log_shift = shift;
  G.log_param = param;
}

void open_log(const Scene *s, const GradTargets &G, hipStream_t stream, LogLaunch &log, GradTargets &GL,
              int64_t samples, int64_t min_samples) {
  for (const MediumInfo &M : s->media) {
    if (M.homogeneous || M.sigma_param < 0 || !G.g[M.sigma_param]) continue;
    log.tiles = log_target(s, M, G.g[M.sigma_param], kLogWide, log.target);
    const bool wide = log.tiles > 0 && (1 << log.target.shift) > log_tile();
    const int64_t enough = wide ? std::max(kWideLogSamples * log.tiles, kWideLogLaunch) : min_samples * log.tiles;
    if (log.tiles > 0 && samples >= enough && stream_pool(stream, log.buf) == RCV_OK) {
      log_into(log.buf, M.sigma_param, 0, log.target.shift, GL);
      hipLaunchKernelGGL(zero_ctl_kernel, dim3(1), dim3(kCtlWords), 0, stream, log.buf.ctl);
    } else {
      log.target.g = nullptr;
    }
    return;
  }
}

void reduce_log(const LogLaunch &log, const GradTargets &GL, hipStream_t stream) {
  if (!log.target.g) return;
  const int tile = log_tile();
  // about 2048 blocks
  const dim3 grid(std::min(kLogSplits, std::max(kLogMinSplits, odd_splits(2048 / log.tiles))), log.tiles);
  const LogBuf &L = log.buf;
  const size_t lds = size_t(tile) * sizeof(long long);
  const LogTarget *const none = nullptr;
  if ((1 << log.target.shift) > tile) {
    float *const bound = reinterpret_cast<float *>(L.ctl + 1);
    hipLaunchKernelGGL(log_bound_kernel, dim3(kBoundBlocks), dim3(kBoundBlock), 0, stream, L.rec, L.ctl, L.meta,
                       GL.log_chunks, bound);
    hipLaunchKernelGGL(log_reduce_kernel<true>, grid, dim3(kReduceBlock), lds, stream, L.rec, L.ctl, L.meta,
                       GL.log_chunks, log.target, none, 1, tile, bound);
  } else {
    hipLaunchKernelGGL(log_reduce_kernel<false>, grid, dim3(kReduceBlock), lds, stream, L.rec, L.ctl, L.meta,
                       GL.log_chunks, log.target, none, 1, tile, static_cast<const float *>(nullptr));
  }
}

void zero_log(const LogBuf &buf, hipStream_t stream) {
  hipLaunchKernelGGL(zero_ctl_kernel, dim3(1), dim3(kCtlWords), 0, stream, buf.ctl);
}

void reduce_log_batch(const LogBuf &buf, const LogTarget &first, const LogTarget *targets, int n, int tiles,
                      hipStream_t stream) {
  const int tile = log_tile();
  // about 4096 blocks
  const int splits = std::min(kLogSplits, std::max(5, odd_splits(4096 / tiles)));
  hipLaunchKernelGGL(log_reduce_kernel<false>, dim3(splits, tiles), dim3(kReduceBlock), size_t(tile) * sizeof(long long),
                     stream, buf.rec, buf.ctl, buf.meta, log_pool_chunks(), first, targets, n, tile,
                     static_cast<const float *>(nullptr));
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
