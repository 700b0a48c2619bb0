// Launch helpers shared by the render entry points.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/rcv.h"
#include "scene_internal.hpp"

namespace rcv {

// Calls fn(std::integral_constant<int, F>{}) for the run-time feature mask
// f, so a launch site can pick the kernel compiled for exactly the scene's
// features (kFeat* bits).
template <typename Fn>
inline void with_features(int f, Fn &&fn) {
  switch (f & kFeatAll) {
    case 0: fn(std::integral_constant<int, 0>{}); break;
    case 1: fn(std::integral_constant<int, 1>{}); break;
    case 2: fn(std::integral_constant<int, 2>{}); break;
    case 3: fn(std::integral_constant<int, 3>{}); break;
    case 4: fn(std::integral_constant<int, 4>{}); break;
    case 5: fn(std::integral_constant<int, 5>{}); break;
    case 6: fn(std::integral_constant<int, 6>{}); break;
    default: fn(std::integral_constant<int, 7>{}); break;
  }
}

// with_features for the single-scene volume kernels, which also take scenes
// with a homogeneous medium: those run one of two kernels, with surface code
// (and heterogeneous media without albedo grids or supergrids), or with every
// feature.
template <typename Fn>
inline void with_render_features(int f, Fn &&fn) {
  if (f & kFeatHomog) {
    if (f & (kFeatAlbedoGrid | kFeatSupergrid))
      fn(std::integral_constant<int, kFeatAll | kFeatHomog>{});
    else
      fn(std::integral_constant<int, kFeatSurfaces | kFeatHomog>{});
    return;
  }
  with_features(f, fn);
}

// Waves per SIMD of the render kernels: the trackers are bound by memory
// latency, so occupancy pays while spills stay small. Measured: the volume
// path tracer (<= 128 VGPRs, few spills) is fastest at four; volpathsimple and
// the surface path tracer, whose state is larger, at three (<= 168 VGPRs).
template <int INTEG>
constexpr int kWavesPerEu = INTEG == RCV_INTEGRATOR_VOLPATH ? 4 : 3;

// The volume path tracer's two-state render and its adjoint carry more
// state (two throughputs and images; the replay's gradient terms): at four
// waves they spilled 60 / 72 B per lane, and at three (up to 168 VGPRs, no
// spills) they run 12-14 % / 17-18 % faster over the optimisation (two
// waves: no faster than three). That holds for the adjoint whose density
// gradient goes through the scatter log; adjoints that add with device-scope
// atomics (static, in batches, of grids past the log) are faster at four,
// whose extra wave covers the atomics' waits (64 volume jobs in a batch on
// these kernels: 348 ms per iteration against 376 ms with the adjoint at
// three). The single-state render stays at four. (All of the general kernels;
// the one-box tracker's wave count is kBoxWaves.)
template <int NS, int INTEG>
constexpr int kWavesPerEuRender = INTEG == RCV_INTEGRATOR_VOLPATH && NS == 2 ? 3 : kWavesPerEu<INTEG>;
constexpr int kWavesPerEuLoggedAdjoint = 3;

// Camera samples per reduction tile from which volpathsimple's adjoint logs
// its density scatter-adds. A launch too small to fill the device waits for
// its longest path, which hides the atomics, and the reduction costs ~5 us a
// tile. On the tracker (simplebox.hpp), a call with atomics / logged: 64^3 (16
// tiles) with 16 Ki samples 1.05 / 1.11 ms, 64 Ki 1.03 / 1.05, 128 Ki 1.45 /
// 1.21; 48^3 (7 tiles) with 16 Ki 1.07 / 1.06, 32 Ki 1.02 / 1.02; 32^3 (2
// tiles) with 1 Ki 0.97 / 0.92, 16 Ki 1.05 / 1.05. The general kernel: 64^3
// with 64 Ki 1.18 / 1.23, 96 Ki 2.08 / 2.08, 128 Ki 1.65 / 1.55, 256 Ki 2.67 /
// 2.16; 48^3 with 64 Ki 1.18 / 1.15.
constexpr int64_t kSimpleLogSamples = 8192;

// Splits the spp camera samples of a pixel over 2^chunk_log2 threads (at
// most spt samples each): a user-given samples_per_thread must divide spp
// into a power of two <= 64 chunks; otherwise chunks double, up to the
// largest power of two <= min(spp, 64), while the launch has fewer than
// min_threads threads or (max_spt > 0) a thread would trace more than
// max_spt samples.
int plan_launch(const rcv_integrator_desc *d, int64_t n_pix, int spp, int &spt, int &chunk_log2,
                int max_spt = 0, int64_t min_threads = int64_t(1) << 19);

// One past the last sample of chunk c (chunk -1 ends at 0): chunk c traces
// samples [sample_end(c - 1), sample_end(c)), an even split when the chunk
// count divides spp.
__host__ __device__ inline int sample_end(int c, int spp, int chunk_log2) {
  return int((int64_t(c + 1) * spp) >> chunk_log2);
}

// Camera samples per work unit of the volume path tracer's persistent
// launches (the adjoint; the renders, within kRenderMaxUnitsPerPixel). With
// small units the lanes of a wavefront trace samples of the same few pixels,
// whose paths start alike and share L1 lines of the grid, and the last units
// of a launch are short. The general kernels' 64^3 adjoint at the mid / final
// state of the optimisation: 46.1 / 67.5 ms with 16-sample units, 39.7 / 51.4
// with 8, 37.0 / 47.8 with 4, 36.2 / 46.4 with 2. On the one-box tracker, units
// of 16, 8, 4, 2 and 1: the 64^3 step (4 x 256^2, 32 samples) 16.3, 13.4, 12.2,
// 11.4 and 11.1 ms; the 128^3 step with an albedo grid 7.7 ms from 2 on, 7.1
// with 1; 64^3 with a supergrid and volpathsimple's adjoint 5.4 ms from 2 on,
// 4.7 with 1.
constexpr int kVolUnitSamples = 2;

// Render, adjoint and forward mode of the one-box volume tracker.
constexpr int kBoxRender = 0;
constexpr int kBoxAdjoint = 1;
constexpr int kBoxForward = 2;

// Waves per SIMD of the one-box volume tracker (boxpath.hpp): four, up to 128
// VGPRs, within which all variants but the two-state renders with an albedo
// grid fit. It is bound by instruction issue: at three, four and five waves the
// 64^3 step takes 11.3, 11.5 and 11.5 ms, the 128^3 render 3.76, 3.77 and 3.80.
// The two-state render spills 44 bytes per lane at four with an albedo grid, 72
// with a supergrid besides: the 128^3 step with an albedo grid 7.1 ms at three
// (no spills), 7.7 at four, 8.6 at five.
template <int NS, int MODE>
constexpr int kBoxWaves = 4;

// Blocks of `kern` the current device holds at once (compute units x
// resident blocks per unit) with `lds` bytes of dynamic LDS per block,
// cached per (device, kernel, block size).
unsigned resident_grid(const void *kern, int block, size_t lds);

struct GradTargets;

// One launch of the one-box volume tracker (box.hip): work units, where the
// unit sums go (render, forward) and the gradients or tangents.
struct BoxLaunch {
  hipStream_t stream;
  int block;
  IntegArgs I;
  int sensor;
  uint32_t seed;
  int spp, chunk_log2;
  unsigned units;
  const float *grad_img;
  const GradTargets *G;
  float *partial;
  unsigned *queue;
};
BoxScene bound_box(const Scene *s);  // the tracker's scene with the bound states

// Whether the one-box volume tracker takes a launch of integrator d on scene
// s (an explicit samples_per_thread asks for the static launch).
inline bool takes_box(const Scene *s, const rcv_integrator_desc *d) {
  return d->type == RCV_INTEGRATOR_VOLPATH && !d->samples_per_thread && d->max_depth != 0 && s->box_path();
}

// Whether the tracker takes volpathsimple's adjoint (simplebox.hpp): the
// default estimator.
inline bool takes_simple_box(const Scene *s, const rcv_integrator_desc *d) {
  return d->type == RCV_INTEGRATOR_VOLPATH_SIMPLE && !d->samples_per_thread && s->box_path() &&
         !(d->flags & (RCV_SIMPLE_NO_NEE | RCV_SIMPLE_NO_DRT | RCV_SIMPLE_NO_DRT_SUBSAMPLING));
}

// Waves per SIMD of volpathsimple's adjoint on the tracker: four, which its
// LDS allows (64^3 with a supergrid: the step 5.34 ms, at three 5.36, at five
// 5.75). With an albedo grid it spills 48 to 80 bytes per lane at four.
constexpr int kSimpleBoxWaves = 4;

// Calls fn with the compile-time feature mask of a one-box scene.
template <typename Fn>
inline void with_box_features(int f, Fn &&fn) {
  switch (f & (kFeatAlbedoGrid | kFeatSupergrid)) {
    case 0: fn(std::integral_constant<int, 0>{}); break;
    case kFeatAlbedoGrid: fn(std::integral_constant<int, kFeatAlbedoGrid>{}); break;
    case kFeatSupergrid: fn(std::integral_constant<int, kFeatSupergrid>{}); break;
    default: fn(std::integral_constant<int, kFeatAlbedoGrid | kFeatSupergrid>{}); break;
  }
}

void launch_box(const Scene *s, int ns, int mode, const BoxLaunch &L);
void launch_simple_box(const Scene *s, const BoxLaunch &L);

int launch_render(const Scene *s, const rcv_integrator_desc *d, int sensor, uint32_t seed, int spp,
                  float *img_old, float *img_new, int ns, hipStream_t stream, const char *fn);

int launch_adjoint(const Scene *s, const rcv_integrator_desc *d, int sensor, uint32_t seed, int spp,
                   const float *grad_img, int n_params, const int32_t *param_ids, float *const *grad_ptrs,
                   hipStream_t stream);

}  // namespace rcv
