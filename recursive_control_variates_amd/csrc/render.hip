// Render entry points of librcv: plain, two-state and adjoint launches of the
// surface (path.hpp) and volume (volpath.hpp) integrators.
//
// Launch shape: the spp camera samples of a pixel are split over 2^chunk_log2
// threads (chunk c traces samples [c spp >> chunk_log2, (c + 1) spp >>
// chunk_log2) in sequence); the threads of a pixel sit in the same wavefront
// and their sums are combined with cross-lane shuffles, so the film needs no
// atomics and the pixel average (box filter develop, plugins/
// twostatepath.py:168-177) is written once, coalesced. The random stream of a
// camera sample depends only on (seed, pixel * spp + sample), so the launch
// shape changes results only through the float summation order of a pixel.
// The BVH traversal stack of each thread lives in LDS (as deep as the
// scene's BVH, strided by the block size), followed by per-lane slots (the
// adjoint's NEE weights): kLdsWordsPerThread words per thread in all.

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>

#include "common.hpp"
#include "path.hpp"
#include "render_internal.hpp"
#include "scatter_log.hpp"
#include "volpath.hpp"
#include "volsimple.hpp"

namespace rcv {
namespace {

constexpr int kMaxBlock = 256;      // launch bound of the render kernels
constexpr int kDefaultBlock = 256;  // threads per block when the descriptor says 0
constexpr int kAdjUnitSamples = 16;  // camera samples per work unit of the persistent per-sample adjoints

template <int NS, int INTEG, int F>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(kWavesPerEuRender<NS, INTEG>))) void render_kernel(
    SceneView S, IntegArgs I, int sensor, uint32_t seed,
                                                        int spp, int spt, int chunk_log2, float *img_old,
                                                        float *img_new) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  const int64_t n_pix = int64_t(film_w) * sen.film_h;
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t pixel = tid >> chunk_log2;
  const int chunk = int(tid & ((1 << chunk_log2) - 1));
  V3 acc[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) acc[k] = v3(0.f);
  LocalCounters cnt{S.counters};
  if (pixel < n_pix) {
    const int px = int(pixel % film_w), py = int(pixel / film_w);
    const int s_end = sample_end(chunk, spp, chunk_log2);
    if (INTEG == RCV_INTEGRATOR_VOLPATH)
      volpath_render_samples<NS, F>(S, I, sen, seed, px, py, pixel, spp, sample_end(chunk - 1, spp, chunk_log2),
                                    s_end, acc, stack, cnt);
    else for (int s = sample_end(chunk - 1, spp, chunk_log2); s < s_end; ++s) {
      Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
      const Ray ray = camera_ray(sen, px, py, rng);
      V3 L[NS];
      if (INTEG == RCV_INTEGRATOR_VOLPATH_SIMPLE)
        L[0] = simple_sample<false, F>(S, I, 0, rng, ray, simple_camera_start(), stack, cnt, nullptr, nullptr,
                                       nullptr);
      else
        path_sample<NS, false>(S, I, rng, ray, L, stack, cnt, nullptr, nullptr);
#pragma unroll
      for (int k = 0; k < NS; ++k) acc[k] += L[k];
    }
  }
  for (int off = 1; off < (1 << chunk_log2); off <<= 1) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      acc[k].x += __shfl_xor(acc[k].x, off, 64);
      acc[k].y += __shfl_xor(acc[k].y, off, 64);
      acc[k].z += __shfl_xor(acc[k].z, off, 64);
    }
  }
  if (pixel < n_pix && chunk == 0) {
    const float inv = float(spp);
    float *o0 = (NS == 2 ? img_old : img_new) + 3 * pixel;
    o0[0] = acc[0].x / inv;
    o0[1] = acc[0].y / inv;
    o0[2] = acc[0].z / inv;
    if (NS == 2) {
      float *o1 = img_new + 3 * pixel;
      o1[0] = acc[NS - 1].x / inv;
      o1[1] = acc[NS - 1].y / inv;
      o1[2] = acc[NS - 1].z / inv;
    }
  }
}

// The adjoint of camera sample s of a pixel for the per-sample integrators:
// the surface path tracer's (path_adjoint_sample), or volpathsimple's primal
// pass, then its adjoint with the same random numbers and its gradient-only
// stream (DRT contributes even where L = 0).
template <int INTEG, int F>
__device__ inline void adjoint_one_sample(const SceneView &S, const IntegArgs &I, const SensorInfo &sen,
                                          uint32_t seed, int px, int py, int64_t pixel, int spp, int s, V3 dL,
                                          const GradTargets &G, const LdsStack &stack, LocalCounters &cnt) {
  Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
  const Ray ray = camera_ray(sen, px, py, rng);
  if constexpr (INTEG == RCV_INTEGRATOR_VOLPATH_SIMPLE) {
    const Pcg32 rng0 = rng;
    V3 L[1];
    L[0] = simple_sample<false, F>(S, I, 0, rng, ray, simple_camera_start(), stack, cnt, nullptr, nullptr, nullptr);
    AdjState adj{dL, L[0]};
    rng = rng0;
    Pcg32 alt = lane_rng(simple_alt_seed(seed), uint32_t(pixel * spp + s));
    (void)simple_sample<true, F>(S, I, 0, rng, ray, simple_camera_start(), stack, cnt, &adj, &alt, &G);
  } else {
    path_adjoint_sample(S, I, rng, ray, dL, G, stack, cnt);
  }
}

// Path-replay adjoint (NEW state): primal pass for L, then a replay with the
// same random numbers that scatters d(log weight)/d(theta) times the radiance
// still to come into the parameter gradients. dimage/dL = 1/spp (box filter).
template <int INTEG, int F>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(kWavesPerEu<INTEG>))) void adjoint_kernel(
    SceneView S, IntegArgs I, int sensor, uint32_t seed,
                                                         int spp, int spt, int chunk_log2,
                                                         const float *__restrict__ grad_img, GradTargets G) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  const int64_t n_pix = int64_t(film_w) * sen.film_h;
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t pixel = tid >> chunk_log2;
  const int chunk = int(tid & ((1 << chunk_log2) - 1));
  LocalCounters cnt{S.counters};
  HomSum hom{0.0f, v3(0.f)};
  if (pixel < n_pix) {
    const int px = int(pixel % film_w), py = int(pixel / film_w);
    const float inv = float(spp);
    const V3 dL = v3(grad_img[3 * pixel] / inv, grad_img[3 * pixel + 1] / inv, grad_img[3 * pixel + 2] / inv);
    if (any_nonzero(dL) && INTEG == RCV_INTEGRATOR_VOLPATH) {
      volpath_adjoint_samples<F>(S, I, sen, seed, px, py, pixel, spp, sample_end(chunk - 1, spp, chunk_log2),
                                 sample_end(chunk, spp, chunk_log2), dL, &G, stack, cnt, &hom);
    } else if (any_nonzero(dL)) {
      const int s_end = sample_end(chunk, spp, chunk_log2);
      for (int s = sample_end(chunk - 1, spp, chunk_log2); s < s_end; ++s)
        adjoint_one_sample<INTEG, F>(S, I, sen, seed, px, py, pixel, spp, s, dL, G, stack, cnt);
    }
  }
  if constexpr (INTEG == RCV_INTEGRATOR_VOLPATH && (F & kFeatHomog) != 0) flush_homogeneous(S, G, hom);
}

// Forward mode (NEW state): per pixel, d(image)/d(theta) . tangent, from the
// primal pass of each sample and its replay with the same random numbers,
// which gathers the tangents (in T) where the adjoint scatters (the
// transpose of adjoint_kernel on the same samples). Launch shape and pixel
// reduction as render_kernel.
template <int INTEG, int F>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(kWavesPerEu<INTEG>))) void forward_kernel(
    SceneView S, IntegArgs I, int sensor, uint32_t seed, int spp, int spt, int chunk_log2, GradTargets T,
    float *__restrict__ dimg) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  const int64_t n_pix = int64_t(film_w) * sen.film_h;
  const int64_t tid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t pixel = tid >> chunk_log2;
  const int chunk = int(tid & ((1 << chunk_log2) - 1));
  LocalCounters cnt{S.counters};
  V3 acc = v3(0.f);
  if (pixel < n_pix) {
    const int px = int(pixel % film_w), py = int(pixel / film_w);
    const int s0 = sample_end(chunk - 1, spp, chunk_log2), s1 = sample_end(chunk, spp, chunk_log2);
    if constexpr (INTEG == RCV_INTEGRATOR_VOLPATH) {
      volpath_forward_samples<F>(S, I, sen, seed, px, py, pixel, spp, s0, s1, &T, stack, cnt, acc);
    } else {
      for (int s = s0; s < s1; ++s) {
        Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
        const Ray ray = camera_ray(sen, px, py, rng);
        const Pcg32 rng0 = rng;
        V3 L[1];
        path_sample<1, false>(S, I, rng, ray, L, stack, cnt, nullptr, nullptr);
        if (!any_nonzero(L[0])) continue;
        AdjState adj{v3(0.f), L[0], v3(0.f)};
        rng = rng0;
        V3 L2[1];
        path_sample<1, true, true>(S, I, rng, ray, L2, stack, cnt, &adj, &T);
        acc += adj.dI;
      }
    }
  }
  for (int off = 1; off < (1 << chunk_log2); off <<= 1) {
    acc.x += __shfl_xor(acc.x, off, 64);
    acc.y += __shfl_xor(acc.y, off, 64);
    acc.z += __shfl_xor(acc.z, off, 64);
  }
  if (pixel < n_pix && chunk == 0) {
    const float inv = float(spp);
    float *o = dimg + 3 * pixel;
    o[0] = acc.x / inv;
    o[1] = acc.y / inv;
    o[2] = acc.z / inv;
  }
}

// Path-replay adjoint of the volume path tracer as a persistent launch: one
// grid of resident waves whose lanes pull work units (a pixel's chunk of
// kVolUnitSamples camera samples) from a device counter, a wavefront's
// requests combined into one atomic, and keep tracing until the units run
// out, so no wave waits at the end of the launch for a few long pixels. The
// result per sample is that of adjoint_kernel; only the order of the gradient
// scatter-adds differs.
template <int F, int W, bool ONCE = false>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(W))) void
adjoint_persistent_kernel(SceneView S, IntegArgs I, int sensor, uint32_t seed, int spp, int chunk_log2,
                          const float *__restrict__ grad_img, GradTargets G, unsigned *queue, unsigned total_units) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  LocalCounters cnt{S.counters};
  VolPath<1, true, F, false, ONCE> t;
  t.L[0] = v3(0.f);
  t.init_hom();
  log_begin(G, stack);
  bool live = false, want_replay = false;
  int s = 0, s_end = 0, px = 0, py = 0;
  int64_t pixel = 0;
  V3 dL = v3(0.f);
  const float inv = float(spp);
  while (true) {
    if (!live) {
      if (!want_replay && s >= s_end) {
        // the lanes that need a unit in this trip share one atomic
        const uint64_t m = __ballot(1);
        const int leader = __ffsll((unsigned long long)m) - 1;
        unsigned base = 0;
        if (int(__lane_id()) == leader) base = atomicAdd(queue, unsigned(__popcll(m)));
        base = __shfl(base, leader, 64);
        const unsigned u = base + unsigned(__popcll(m & __lanemask_lt()));
        if (u >= total_units) break;
        pixel = int64_t(u >> chunk_log2);
        const int chunk = int(u & ((1u << chunk_log2) - 1u));
        px = int(pixel % film_w);
        py = int(pixel / film_w);
        s = sample_end(chunk - 1, spp, chunk_log2);
        s_end = sample_end(chunk, spp, chunk_log2);
        dL = v3(grad_img[3 * pixel] / inv, grad_img[3 * pixel + 1] / inv, grad_img[3 * pixel + 2] / inv);
        if (!any_nonzero(dL)) {
          s = s_end;
          continue;
        }
      }
      Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
      const Ray r = camera_ray(sen, px, py, rng);
      t.begin_adjoint(rng, r, cnt, want_replay, dL, t.L[0]);
    }
    live = t.bounce(S, I, stack, cnt, &G);
    if (!live) {
      want_replay = !t.end_adjoint(S, cnt, &G);
      if (!want_replay) ++s;
    }
  }
  if constexpr ((F & kFeatHomog) != 0) flush_homogeneous(S, G, t.hom);
  // the whole wavefront is past its loop
  log_close(G, stack);
  log_end(G, stack);
}

// The per-sample integrators' adjoint (volpathsimple, surface path tracer) as
// a persistent launch (see adjoint_persistent_kernel): lanes pull work units
// (a pixel's chunk of camera samples) from a device counter and run
// adjoint_one_sample for each, so long pixels do not hold their wavefronts at
// the end of the launch. The result per sample is that of adjoint_kernel;
// only the order of the gradient scatter-adds differs. volpathsimple's density
// scatter-adds go through the log where it is set: each is a 16-byte record
// in place of 8 atomics, and a sample has ~50 of them (64^3, 128^2, 16
// samples, majorant supergrid: 6.1 ms and 0.5 ms of reduction against 7.5 ms
// with atomics). What is
// left is issue in the nested tracking loops, whose lanes diverge.
template <int INTEG, int F>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(kWavesPerEu<INTEG>))) void
adjoint_sample_persistent_kernel(
    SceneView S, IntegArgs I, int sensor, uint32_t seed, int spp, int chunk_log2, const float *__restrict__ grad_img,
    GradTargets G, unsigned *queue, unsigned total_units) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  LocalCounters cnt{S.counters};
  constexpr bool kLogs = INTEG == RCV_INTEGRATOR_VOLPATH_SIMPLE;
  if constexpr (kLogs) log_begin(G, stack);
  int s = 0, s_end = 0, px = 0, py = 0;
  int64_t pixel = 0;
  V3 dL = v3(0.f);
  const float inv = float(spp);
  while (true) {
    if (s >= s_end) {
      // the lanes that need a unit in this trip share one atomic
      const uint64_t m = __ballot(1);
      const int leader = __ffsll((unsigned long long)m) - 1;
      unsigned base = 0;
      if (int(__lane_id()) == leader) base = atomicAdd(queue, unsigned(__popcll(m)));
      base = __shfl(base, leader, 64);
      const unsigned u = base + unsigned(__popcll(m & __lanemask_lt()));
      if (u >= total_units) break;
      pixel = int64_t(u >> chunk_log2);
      const int chunk = int(u & ((1u << chunk_log2) - 1u));
      px = int(pixel % film_w);
      py = int(pixel / film_w);
      s = sample_end(chunk - 1, spp, chunk_log2);
      s_end = sample_end(chunk, spp, chunk_log2);
      dL = v3(grad_img[3 * pixel] / inv, grad_img[3 * pixel + 1] / inv, grad_img[3 * pixel + 2] / inv);
      if (!any_nonzero(dL)) {
        s = s_end;
        continue;
      }
    }
    adjoint_one_sample<INTEG, F>(S, I, sen, seed, px, py, pixel, spp, s, dL, G, stack, cnt);
    ++s;
  }
  // the whole wavefront is past its loop
  if constexpr (kLogs) {
    log_close(G, stack);
    log_end(G, stack);
  }
}

// The volume path tracer's render as a persistent launch (see
// adjoint_persistent_kernel): a lane traces the samples of a work unit (a
// pixel's chunk) in order and stores their sum in the unit's slot of
// `partial`; reduce_units_kernel then forms each pixel's mean from its units
// in order, so the image does not depend on which lane took which unit.
template <int NS, int F>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(kWavesPerEuRender<NS, RCV_INTEGRATOR_VOLPATH>))) void
render_persistent_kernel(SceneView S, IntegArgs I, int sensor, uint32_t seed, int spp, int chunk_log2,
                         float *__restrict__ partial, unsigned *queue, unsigned total_units) {
  extern __shared__ int lds_stack[];  // kLdsWordsPerThread words per thread
  const LdsStack stack = lds_of(S, lds_stack);
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  LocalCounters cnt{S.counters};
  VolPath<NS, false, F> t;
  bool live = false;
  int s = 0, s_end = 0, px = 0, py = 0;
  unsigned u = 0;
  int64_t pixel = 0;
  V3 acc[NS];
  while (true) {
    if (!live) {
      if (s >= s_end) {
        const uint64_t m = __ballot(1);
        const int leader = __ffsll((unsigned long long)m) - 1;
        unsigned base = 0;
        if (int(__lane_id()) == leader) base = atomicAdd(queue, unsigned(__popcll(m)));
        base = __shfl(base, leader, 64);
        u = base + unsigned(__popcll(m & __lanemask_lt()));
        if (u >= total_units) break;
        pixel = int64_t(u >> chunk_log2);
        const int chunk = int(u & ((1u << chunk_log2) - 1u));
        px = int(pixel % film_w);
        py = int(pixel / film_w);
        s = sample_end(chunk - 1, spp, chunk_log2);
        s_end = sample_end(chunk, spp, chunk_log2);
#pragma unroll
        for (int k = 0; k < NS; ++k) acc[k] = v3(0.f);
      }
      Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
      const Ray r = camera_ray(sen, px, py, rng);
      t.begin(rng, r, cnt, false);
    }
    live = t.bounce(S, I, stack, cnt, nullptr);
    if (!live) {
#pragma unroll
      for (int k = 0; k < NS; ++k) acc[k] += t.L[k];
      if (++s >= s_end) {
        float *o = partial + int64_t(u) * (3 * NS);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
          o[3 * k] = acc[k].x;
          o[3 * k + 1] = acc[k].y;
          o[3 * k + 2] = acc[k].z;
        }
      }
    }
  }
}

// Pixel mean from the unit sums, units in order (a pixel of two units adds
// them as the cross-lane reduction of render_kernel does).
template <int NS>
__global__ void reduce_units_kernel(const float *__restrict__ partial, int64_t n_pix, int chunk_log2, int spp,
                                    float *__restrict__ img_old, float *__restrict__ img_new) {
  const int64_t pixel = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (pixel >= n_pix) return;
  const int units = 1 << chunk_log2;
  const float inv = float(spp);
  for (int k = 0; k < NS; ++k) {
    float x = 0.f, y = 0.f, z = 0.f;
    for (int c = 0; c < units; ++c) {
      const float *src = partial + ((pixel << chunk_log2) + c) * (3 * NS) + 3 * k;
      if (c == 0) {
        x = src[0];
        y = src[1];
        z = src[2];
      } else {
        x += src[0];
        y += src[1];
        z += src[2];
      }
    }
    float *o = (NS == 2 ? (k == 0 ? img_old : img_new) : img_new) + 3 * pixel;
    o[0] = x / inv;
    o[1] = y / inv;
    o[2] = z / inv;
  }
}

__global__ void zero_u32_kernel(unsigned *p) { p[threadIdx.x] = 0u; }

__global__ void zero_counters_kernel(unsigned long long *c) {
  if (threadIdx.x < kNumCounters) c[threadIdx.x] = 0ull;
}


}  // namespace

static size_t stack_bytes(int block) { return size_t(kLdsWordsPerThread) * block * sizeof(int); }

unsigned resident_grid(const void *kern, int block, size_t lds) {
  static std::mutex mu;
  static std::map<std::tuple<int, const void *, int>, unsigned> cache;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lock(mu);
  const auto key = std::make_tuple(dev, kern, block);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int cus = 0, per_cu = 0;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds);
  const unsigned g = unsigned(std::max(1, per_cu) * std::max(1, cus));
  cache[key] = g;
  return g;
}

// Work-unit split of the one-box renders: up to 64 units per pixel of at
// least kVolUnitSamples samples, within the unit-sum buffer (floats per
// unit: `words`).
static int box_chunk_log2(const Scene *s, int64_t n_pix, int spp, int static_cl2, int words) {
  int cl2 = 0;
  while (cl2 < 6 && ((n_pix << (cl2 + 1)) * words) <= s->partial_cap &&
         ((spp >> (cl2 + 1)) >= kVolUnitSamples || (cl2 < static_cl2 && (2 << cl2) <= spp)))
    ++cl2;
  return cl2;
}

// Work-unit split of a persistent volume launch: the chunk count of the
// static launch (enough units to fill the device), raised while a unit keeps
// at least min_samples samples.
static int unit_chunk_log2(int spp, int static_cl2, int min_samples) {
  int ucl2 = 0;
  while ((1 << ucl2) < 64 && (spp >> (ucl2 + 1)) >= min_samples) ++ucl2;
  return std::max(ucl2, static_cl2);
}

int plan_launch(const rcv_integrator_desc *d, int64_t n_pix, int spp, int &spt, int &chunk_log2, int max_spt,
                int64_t min_threads) {
  if (d && d->block_size != 0 && (d->block_size < 64 || d->block_size > kMaxBlock || d->block_size % 64 != 0))
    return fail(RCV_E_INVALID, "block_size %d must be 0 or a multiple of 64 in [64, %d]", d->block_size, kMaxBlock);
  int chunks;
  int cap = 1;
  while (cap < 64 && 2 * cap <= spp) cap <<= 1;  // largest power of two <= min(spp, 64)
  if (d && d->samples_per_thread > 0) {
    if (spp % d->samples_per_thread != 0)
      return fail(RCV_E_INVALID, "samples_per_thread %d must divide spp %d", d->samples_per_thread, spp);
    chunks = spp / d->samples_per_thread;
    if (chunks > 64 || (chunks & (chunks - 1)) != 0)
      return fail(RCV_E_INVALID, "spp / samples_per_thread = %d must be a power of two <= 64", chunks);
  } else {
    chunks = 1;
    while (chunks < cap && (n_pix * chunks < min_threads || (max_spt > 0 && spp > max_spt * chunks)))
      chunks <<= 1;
  }
  spt = (spp + chunks - 1) / chunks;  // samples of the busiest thread
  chunk_log2 = 0;
  while ((1 << chunk_log2) < chunks) ++chunk_log2;
  return RCV_OK;
}

static int check_states(const Scene *s, int ns, const char *fn) {
  auto need = [&](int param, const char *what) -> int {
    if (param < 0) return RCV_OK;
    const Param &p = s->params[param];
    if (!p.data[RCV_STATE_NEW]) return fail(RCV_E_STATE, "%s: %s parameter %d has no NEW state bound", fn, what, param);
    if (ns == 2 && !p.data[RCV_STATE_OLD])
      return fail(RCV_E_STATE, "%s: %s parameter %d has no OLD state bound", fn, what, param);
    return RCV_OK;
  };
  for (auto &b : s->bsdfs)
    if (int rc = need(b.texture_param, "texture")) return rc;
  for (auto &m : s->media) {
    if (int rc = need(m.sigma_param, "sigma_t")) return rc;
    if (int rc = need(m.albedo_param, "albedo")) return rc;
  }
  return RCV_OK;
}

static GradTargets no_targets() {
  GradTargets g;
  g.clear();
  return g;
}

struct RenderLaunch {
  dim3 grid;
  int block;
  hipStream_t stream;
  const SceneView *view;
  IntegArgs I;
  int sensor;
  uint32_t seed;
  int spp, spt, cl2;
  float *img_old, *img_new;
};

template <int NS, int INTEG, int F>
static void launch_render_kernel(const RenderLaunch &L) {
  hipLaunchKernelGGL((render_kernel<NS, INTEG, F>), L.grid, dim3(L.block), stack_bytes(L.block), L.stream, *L.view,
                     L.I, L.sensor,
                     L.seed, L.spp, L.spt, L.cl2, L.img_old, L.img_new);
}

// get_single_medium and the class docstring of plugins/volpathsimple.py
// (:9-30): one shape with an interior medium and a null BSDF, the
// environment as the only emitter.
static int check_simple(const Scene *s, const char *fn) {
  if (s->shapes.size() != 1)
    return fail(RCV_E_SCENE, "%s: volpathsimple: Not supported: more than 1 shape in the scene (found %d).", fn,
                int(s->shapes.size()));
  if (s->media.size() != 1 || s->shapes[0].interior != 0)
    return fail(RCV_E_SCENE, "%s: volpathsimple: Expected a single shape with an interior medium.", fn);
  if (s->features() & kFeatSurfaces)
    return fail(RCV_E_SCENE, "%s: volpathsimple: the medium boundary must use a null BSDF", fn);
  if (s->features() & kFeatHomog)
    return fail(RCV_E_SCENE, "%s: volpathsimple: heterogeneous media only", fn);
  if (s->emitters.size() != 1 || s->emitters[0].type != RCV_EMITTER_CONSTANT)
    return fail(RCV_E_SCENE, "%s: volpathsimple: the only emitter must be an infinite light", fn);
  return RCV_OK;
}

// with_features over the masks without surfaces (volpathsimple scenes).
template <typename Fn>
static void with_volume_features(int f, Fn &&fn) {
  switch (f & (kFeatAlbedoGrid | kFeatSupergrid)) {
    case 0: fn(std::integral_constant<int, 0>{}); break;
    case kFeatAlbedoGrid: fn(std::integral_constant<int, kFeatAlbedoGrid>{}); break;
    case kFeatSupergrid: fn(std::integral_constant<int, kFeatSupergrid>{}); break;
    default: fn(std::integral_constant<int, kFeatAlbedoGrid | kFeatSupergrid>{}); break;
  }
}

int launch_render(const Scene *s, const rcv_integrator_desc *d, int sensor, uint32_t seed, int spp,
                  float *img_old, float *img_new, int ns, hipStream_t stream, const char *fn) {
  RCV_REQUIRE(s && s->committed, "%s: scene not committed", fn);
  RCV_REQUIRE(d, "%s: null integrator", fn);
  RCV_REQUIRE(d->type == RCV_INTEGRATOR_PATH || d->type == RCV_INTEGRATOR_VOLPATH ||
                  d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE,
              "%s: bad integrator type", fn);
  if (d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE) {
    RCV_REQUIRE(ns == 1, "%s: volpathsimple renders one state", fn);
    if (int rc = check_simple(s, fn)) return rc;
  }
  RCV_REQUIRE(sensor >= 0 && sensor < int(s->sensors.size()), "%s: bad sensor %d", fn, sensor);
  RCV_REQUIRE(spp > 0, "%s: spp must be positive", fn);
  RCV_REQUIRE(img_new && (ns == 1 || img_old), "%s: null image", fn);
  if (int rc = check_states(s, ns, fn)) return rc;
  const SensorInfo &sen = s->sensors[sensor];
  const int64_t n_pix = int64_t(sen.film_w) * sen.film_h;
  RCV_REQUIRE(n_pix * spp < (int64_t(1) << 32), "%s: pixels * spp must stay below 2^32", fn);
  int spt, cl2;
  if (int rc = plan_launch(d, n_pix, spp, spt, cl2)) return rc;
  const IntegArgs I{d->max_depth, d->rr_depth, d->hide_emitters, d->flags};
  const int64_t threads = n_pix << cl2;
  const int block = d->block_size ? d->block_size : kDefaultBlock;
  const unsigned grid = ceil_div(threads, block);
  if (s->view.counters) hipLaunchKernelGGL(zero_counters_kernel, dim3(1), dim3(64), 0, stream, s->view.counters);
  const RenderLaunch L{dim3(grid), block, stream, &s->view, I, sensor, seed, spp, spt, cl2, img_old, img_new};
  // under capture, launches that would be static without the tracker stay so:
  // several graphs of a scene share its scratch
  const bool captured = capturing(stream);
  const bool few_units = (1 << cl2) <= kRenderMaxUnitsPerPixel;
  const bool box = takes_box(s, d) && (!captured || few_units);
  const bool persistent = d->type == RCV_INTEGRATOR_VOLPATH && !d->samples_per_thread && few_units;
  LaunchScratch tmp;
  if (box || persistent)
    if (int rc = s->scratch(stream, captured, tmp)) return rc;
  if (box) {
    const int ucl2 = box_chunk_log2(s, n_pix, spp, cl2, 3 * ns);
    const GradTargets none = no_targets();
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
    launch_box(s, ns, kBoxRender,
               BoxLaunch{stream, block, I, sensor, seed, spp, ucl2, unsigned(n_pix << ucl2), nullptr, &none,
                         tmp.partial, tmp.queue});
    if (ns == 2)
      hipLaunchKernelGGL(reduce_units_kernel<2>, dim3(ceil_div(n_pix, 256)), dim3(256), 0, stream, tmp.partial, n_pix,
                         ucl2, spp, img_old, img_new);
    else
      hipLaunchKernelGGL(reduce_units_kernel<1>, dim3(ceil_div(n_pix, 256)), dim3(256), 0, stream, tmp.partial, n_pix,
                         ucl2, spp, img_old, img_new);
  } else if (d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE) {
    with_volume_features(s->features(), [&](auto f) {
      launch_render_kernel<1, RCV_INTEGRATOR_VOLPATH_SIMPLE, decltype(f)::value>(L);
    });
  } else if (persistent) {
    // persistent, with at most kRenderMaxUnitsPerPixel units per pixel (the
    // unit-sum buffer); smaller images that need more units per pixel to
    // fill the device take the static launch below
    int ucl2 = cl2;
    while ((2 << ucl2) <= kRenderMaxUnitsPerPixel && (spp >> (ucl2 + 1)) >= kVolUnitSamples) ++ucl2;
    const unsigned units = unsigned(n_pix << ucl2);
    RCV_REQUIRE(int64_t(units) * 3 * ns <= s->partial_cap, "%s: unit buffer too small", fn);
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
    auto go = [&](auto kern) {
      const unsigned pgrid = std::min(resident_grid(reinterpret_cast<const void *>(kern), block, stack_bytes(block)), grid);
      hipLaunchKernelGGL(kern, dim3(pgrid), dim3(block), stack_bytes(block), stream, s->view, I, sensor, seed, spp,
                         ucl2, tmp.partial, tmp.queue, units);
    };
    if (ns == 2) {
      with_render_features(s->features(), [&](auto f) { go(render_persistent_kernel<2, decltype(f)::value>); });
      hipLaunchKernelGGL(reduce_units_kernel<2>, dim3(ceil_div(n_pix, 256)), dim3(256), 0, stream, tmp.partial, n_pix,
                         ucl2, spp, img_old, img_new);
    } else {
      with_render_features(s->features(), [&](auto f) { go(render_persistent_kernel<1, decltype(f)::value>); });
      hipLaunchKernelGGL(reduce_units_kernel<1>, dim3(ceil_div(n_pix, 256)), dim3(256), 0, stream, tmp.partial, n_pix,
                         ucl2, spp, img_old, img_new);
    }
  } else if (d->type == RCV_INTEGRATOR_VOLPATH) {
    if (ns == 2)
      with_render_features(s->features(), [&](auto f) { launch_render_kernel<2, RCV_INTEGRATOR_VOLPATH, decltype(f)::value>(L); });
    else
      with_render_features(s->features(), [&](auto f) { launch_render_kernel<1, RCV_INTEGRATOR_VOLPATH, decltype(f)::value>(L); });
  } else {
    if (ns == 2)
      launch_render_kernel<2, RCV_INTEGRATOR_PATH, 0>(L);
    else
      launch_render_kernel<1, RCV_INTEGRATOR_PATH, 0>(L);
  }
  return check_launch(fn);
}

int launch_adjoint(const Scene *s, const rcv_integrator_desc *d, int sensor, uint32_t seed, int spp,
                   const float *grad_img, int n_params, const int32_t *param_ids, float *const *grad_ptrs,
                   hipStream_t stream) {
  const char *fn = "rcv_render_backward";
  RCV_REQUIRE(s && s->committed, "%s: scene not committed", fn);
  RCV_REQUIRE(d, "%s: null integrator", fn);
  RCV_REQUIRE(sensor >= 0 && sensor < int(s->sensors.size()), "%s: bad sensor %d", fn, sensor);
  RCV_REQUIRE(spp > 0 && grad_img, "%s: bad spp or null grad_img", fn);
  RCV_REQUIRE(n_params >= 0 && (n_params == 0 || (param_ids && grad_ptrs)), "%s: bad gradient targets", fn);
  RCV_REQUIRE(d->type == RCV_INTEGRATOR_PATH || d->type == RCV_INTEGRATOR_VOLPATH ||
                  d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE,
              "%s: bad integrator type", fn);
  if (d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE)
    if (int rc = check_simple(s, fn)) return rc;
  if (int rc = check_states(s, 1, fn)) return rc;
  GradTargets G;
  G.clear();
  for (int i = 0; i < n_params; ++i) {
    RCV_REQUIRE(param_ids[i] >= 0 && param_ids[i] < int(s->params.size()), "%s: bad param id %d", fn, param_ids[i]);
    RCV_REQUIRE(grad_ptrs[i], "%s: null gradient buffer for param %d", fn, param_ids[i]);
    G.g[param_ids[i]] = grad_ptrs[i];
  }
  const SensorInfo &sen = s->sensors[sensor];
  const int64_t n_pix = int64_t(sen.film_w) * sen.film_h;
  RCV_REQUIRE(n_pix * spp < (int64_t(1) << 32), "%s: pixels * spp must stay below 2^32", fn);
  int spt, cl2;
  if (int rc = plan_launch(d, n_pix, spp, spt, cl2)) return rc;
  const IntegArgs I{d->max_depth, d->rr_depth, d->hide_emitters, d->flags};
  const int block = d->block_size ? d->block_size : kDefaultBlock;
  const unsigned grid = ceil_div(n_pix << cl2, block);
  if (s->view.counters) hipLaunchKernelGGL(zero_counters_kernel, dim3(1), dim3(64), 0, stream, s->view.counters);
  LaunchScratch tmp;
  if (!d->samples_per_thread)
    if (int rc = s->scratch(stream, capturing(stream), tmp)) return rc;
  // the per-sample integrators' persistent adjoint, as the volume path
  // tracer's below
  auto launch_sample_persistent = [&](auto kern, const GradTargets &targets) {
    const int ucl2 = unit_chunk_log2(spp, cl2, kAdjUnitSamples);
    const unsigned units = unsigned(n_pix << ucl2);
    const unsigned pgrid =
        std::min(resident_grid(reinterpret_cast<const void *>(kern), block, stack_bytes(block)), ceil_div(int64_t(units), block));
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
    hipLaunchKernelGGL(kern, dim3(pgrid), dim3(block), stack_bytes(block), stream, s->view, I, sensor, seed, spp, ucl2,
                       grad_img, targets, tmp.queue, units);
  };
  if (d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE && !d->samples_per_thread) {
    GradTargets GL = G;
    LogLaunch log;
    open_log(s, G, stream, log, GL, n_pix * spp, kSimpleLogSamples);
    if (takes_simple_box(s, d)) {
      const int ucl2 = unit_chunk_log2(spp, cl2, kVolUnitSamples);
      hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
      launch_simple_box(s, BoxLaunch{stream, block, I, sensor, seed, spp, ucl2, unsigned(n_pix << ucl2), grad_img, &GL,
                                     nullptr, tmp.queue});
    } else {
      with_volume_features(s->features(), [&](auto f) {
        launch_sample_persistent(adjoint_sample_persistent_kernel<RCV_INTEGRATOR_VOLPATH_SIMPLE, decltype(f)::value>,
                                 GL);
      });
    }
    reduce_log(log, GL, stream);
  } else if (d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE)
    with_volume_features(s->features(), [&](auto f) {
      hipLaunchKernelGGL((adjoint_kernel<RCV_INTEGRATOR_VOLPATH_SIMPLE, decltype(f)::value>), dim3(grid),
                         dim3(block), stack_bytes(block), stream, s->view, I, sensor, seed, spp, spt, cl2, grad_img,
                         G);
    });
  else if (d->type == RCV_INTEGRATOR_VOLPATH && !d->samples_per_thread) {
    const bool box = takes_box(s, d);
    const bool taped = !box && (s->features() & kFeatSupergrid) && !(s->features() & kFeatAlbedoGrid);
    // (taped kernels keep kAdjUnitSamples: their per-lane tape in scratch
    // gains nothing from coherence; the 64^3 k = 8 adjoint took 59.4 ms
    // with 2-sample units against 51.2 ms)
    const int ucl2 = unit_chunk_log2(spp, cl2, taped ? kAdjUnitSamples : kVolUnitSamples);
    const unsigned units = unsigned(n_pix << ucl2);
    GradTargets GL = G;
    // only constants of the homogeneous medium to differentiate
    const int hom = s->view.hom_medium;
    bool hom_once = hom >= 0;
    for (int i = 0; i < n_params; ++i)
      if (hom < 0 || (param_ids[i] != s->media[hom].sigma_param && param_ids[i] != s->media[hom].albedo_param))
        hom_once = false;
    LogLaunch log;
    if (!taped) open_log(s, G, stream, log, GL, n_pix * spp);
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
    if (box)
      launch_box(s, 1, kBoxAdjoint,
                 BoxLaunch{stream, block, I, sensor, seed, spp, ucl2, units, grad_img, &GL, nullptr, tmp.queue});
    else
      with_render_features(s->features(), [&](auto f) {
        // the waves that fit, pulling units of >= kVolUnitSamples samples
        // (fewer where the image is too small to fill the device otherwise)
        constexpr int F = decltype(f)::value;
        auto go = [&](auto kern) {
          const unsigned pgrid = std::min(resident_grid(reinterpret_cast<const void *>(kern), block, stack_bytes(block)),
                                          ceil_div(int64_t(units), block));
          hipLaunchKernelGGL(kern, dim3(pgrid), dim3(block), stack_bytes(block), stream, s->view, I, sensor, seed, spp,
                             ucl2, grad_img, GL, tmp.queue, units);
        };
        if constexpr ((F & kFeatHomog) != 0) {
          if (hom_once) return go(adjoint_persistent_kernel<F, kWavesPerEuLoggedAdjoint, true>);
        }
        // three waves per SIMD with the log or without scatter-adds, four
        // with atomics (kWavesPerEuLoggedAdjoint)
        if constexpr (kTapeAdjoint<F>)
          go(adjoint_persistent_kernel<F, kWavesPerEu<RCV_INTEGRATOR_VOLPATH>>);
        else if (log.target.g)
          go(adjoint_persistent_kernel<F, kWavesPerEuLoggedAdjoint>);
        else
          go(adjoint_persistent_kernel<F, kWavesPerEu<RCV_INTEGRATOR_VOLPATH>>);
      });
    reduce_log(log, GL, stream);
  }
  else if (d->type == RCV_INTEGRATOR_VOLPATH)
    with_render_features(s->features(), [&](auto f) {
      hipLaunchKernelGGL((adjoint_kernel<RCV_INTEGRATOR_VOLPATH, decltype(f)::value>), dim3(grid), dim3(block),
                         stack_bytes(block), stream, s->view, I, sensor, seed, spp, spt, cl2, grad_img, G);
    });
  else if (!d->samples_per_thread)
    launch_sample_persistent(adjoint_sample_persistent_kernel<RCV_INTEGRATOR_PATH, 0>, G);
  else
    hipLaunchKernelGGL((adjoint_kernel<RCV_INTEGRATOR_PATH, 0>), dim3(grid), dim3(block), stack_bytes(block), stream,
                       s->view, I, sensor, seed, spp, spt, cl2, grad_img, G);
  return check_launch(fn);
}

int launch_forward(const Scene *s, const rcv_integrator_desc *d, int sensor, uint32_t seed, int spp,
                   int n_params, const int32_t *param_ids, const float *const *tangents, float *dimg,
                   hipStream_t stream) {
  const char *fn = "rcv_render_forward";
  RCV_REQUIRE(s && s->committed, "%s: scene not committed", fn);
  RCV_REQUIRE(d, "%s: null integrator", fn);
  RCV_REQUIRE(sensor >= 0 && sensor < int(s->sensors.size()), "%s: bad sensor %d", fn, sensor);
  RCV_REQUIRE(spp > 0 && dimg, "%s: bad spp or null output image", fn);
  RCV_REQUIRE(n_params >= 0 && (n_params == 0 || (param_ids && tangents)), "%s: bad tangent arguments", fn);
  // volpathsimple's adjoint is written with backward-mode calls only
  // (dr.backward_from, plugins/volpathsimple.py:183,502,593,620): no forward mode
  RCV_REQUIRE(d->type == RCV_INTEGRATOR_PATH || d->type == RCV_INTEGRATOR_VOLPATH,
              "%s: forward mode exists for the path-replay integrators (prb, prbvolpath) only", fn);
  if (int rc = check_states(s, 1, fn)) return rc;
  GradTargets T;
  T.clear();
  for (int i = 0; i < n_params; ++i) {
    RCV_REQUIRE(param_ids[i] >= 0 && param_ids[i] < int(s->params.size()), "%s: bad param id %d", fn, param_ids[i]);
    RCV_REQUIRE(tangents[i], "%s: null tangent for param %d", fn, param_ids[i]);
    T.g[param_ids[i]] = const_cast<float *>(tangents[i]);
  }
  const SensorInfo &sen = s->sensors[sensor];
  const int64_t n_pix = int64_t(sen.film_w) * sen.film_h;
  RCV_REQUIRE(n_pix * spp < (int64_t(1) << 32), "%s: pixels * spp must stay below 2^32", fn);
  int spt, cl2;
  if (int rc = plan_launch(d, n_pix, spp, spt, cl2)) return rc;
  const IntegArgs I{d->max_depth, d->rr_depth, d->hide_emitters, d->flags};
  const int block = d->block_size ? d->block_size : kDefaultBlock;
  const unsigned grid = ceil_div(n_pix << cl2, block);
  if (s->view.counters) hipLaunchKernelGGL(zero_counters_kernel, dim3(1), dim3(64), 0, stream, s->view.counters);
  // (captured: the static launch, which needs no scratch)
  if (takes_box(s, d) && !capturing(stream)) {
    LaunchScratch tmp;
    if (int rc = s->scratch(stream, false, tmp)) return rc;
    const int ucl2 = box_chunk_log2(s, n_pix, spp, cl2, 3);
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, tmp.queue);
    launch_box(s, 1, kBoxForward,
               BoxLaunch{stream, block, I, sensor, seed, spp, ucl2, unsigned(n_pix << ucl2), nullptr, &T, tmp.partial,
                         tmp.queue});
    hipLaunchKernelGGL(reduce_units_kernel<1>, dim3(ceil_div(n_pix, 256)), dim3(256), 0, stream, tmp.partial, n_pix,
                       ucl2, spp, nullptr, dimg);
  } else if (d->type == RCV_INTEGRATOR_VOLPATH)
    with_render_features(s->features(), [&](auto f) {
      hipLaunchKernelGGL((forward_kernel<RCV_INTEGRATOR_VOLPATH, decltype(f)::value>), dim3(grid), dim3(block),
                         stack_bytes(block), stream, s->view, I, sensor, seed, spp, spt, cl2, T, dimg);
    });
  else
    hipLaunchKernelGGL((forward_kernel<RCV_INTEGRATOR_PATH, 0>), dim3(grid), dim3(block), stack_bytes(block), stream,
                       s->view, I, sensor, seed, spp, spt, cl2, T, dimg);
  return check_launch(fn);
}

namespace {
// A wavefront per cell.
__global__ __launch_bounds__(256) void supergrid_kernel(const float *__restrict__ grid, int nx, int ny, int nz, int sx,
                                                        int sy, int sz, float *__restrict__ out) {
  const int c = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (c >= sx * sy * sz) return;
  const float m = supergrid_cell_max(grid, nx, ny, nz, sx, sy, sz, c);
  if ((threadIdx.x & 63u) == 0) out[c] = m;
}
}  // namespace

int Scene::build_supergrid(int medium, int state, hipStream_t stream) {
  const MediumInfo &m = media[medium];
  const Param &p = params[m.sigma_param];
  const int cells = m.sg_res[0] * m.sg_res[1] * m.sg_res[2];
  float *out = supergrids + m.supergrid_offset + state * cells;
  hipLaunchKernelGGL(supergrid_kernel, dim3(ceil_div(cells, 4)), dim3(256), 0, stream, p.data[state], p.nx, p.ny,
                     p.nz, m.sg_res[0], m.sg_res[1], m.sg_res[2], out);
  return check_launch("majorant supergrid");
}

}  // namespace rcv

using namespace rcv;

extern "C" int rcv_render(const rcv_scene *scene, const rcv_integrator_desc *integrator, int32_t sensor,
                          uint32_t seed, int32_t spp, float *img, void *stream) {
  return launch_render(static_cast<const Scene *>(scene), integrator, sensor, seed, spp, nullptr, img, 1,
                       as_stream(stream), "rcv_render");
}

extern "C" int rcv_render_twostates(const rcv_scene *scene, const rcv_integrator_desc *integrator,
                                    int32_t sensor, uint32_t seed, int32_t spp, float *img_old, float *img_new,
                                    void *stream) {
  return launch_render(static_cast<const Scene *>(scene), integrator, sensor, seed, spp, img_old, img_new, 2,
                       as_stream(stream), "rcv_render_twostates");
}

extern "C" int rcv_render_forward(const rcv_scene *scene, const rcv_integrator_desc *integrator, int32_t sensor,
                                  uint32_t seed, int32_t spp, int32_t n_params, const int32_t *param_ids,
                                  const float *const *tangents, float *dimg, void *stream) {
  return launch_forward(static_cast<const Scene *>(scene), integrator, sensor, seed, spp, n_params, param_ids,
                        tangents, dimg, as_stream(stream));
}

extern "C" int rcv_render_backward(const rcv_scene *scene, const rcv_integrator_desc *integrator, int32_t sensor,
                                   uint32_t seed, int32_t spp, const float *grad_img, int32_t n_params,
                                   const int32_t *param_ids, float *const *grad_ptrs, void *stream) {
  return launch_adjoint(static_cast<const Scene *>(scene), integrator, sensor, seed, spp, grad_img, n_params,
                        param_ids, grad_ptrs, as_stream(stream));
}
