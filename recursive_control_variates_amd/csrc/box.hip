// Launches of the one-box volume tracker (boxpath.hpp): render, adjoint and
// forward mode of the volume path tracer for scenes it covers
// (Scene::box_scene). Persistent grids of the resident waves whose lanes
// pull work units (a pixel's chunk of camera samples) from a device counter,
// as the general volume kernels do.

#include <algorithm>

#include "boxpath.hpp"
#include "common.hpp"
#include "render_internal.hpp"

namespace rcv {
namespace {

constexpr int kBoxMaxBlock = 256;

// Render (partial: per unit the NS radiance sums), adjoint (into G, through
// the scatter log where it is set) and forward mode (partial: per unit the
// derivative's sum, the tangents in G).
template <int NS, int MODE, int F>
__global__ __launch_bounds__(kBoxMaxBlock) __attribute__((amdgpu_waves_per_eu(kBoxWaves<NS, MODE>))) void box_kernel(
    SceneView S, BoxScene B, IntegArgs I, int sensor, uint32_t seed, int spp, int chunk_log2,
    const float *__restrict__ grad_img, GradTargets G, float *__restrict__ partial, unsigned *queue,
    unsigned total_units) {
  extern __shared__ int lds_words[];  // kBoxWords<MODE> words per thread
  int *const lds = lds_words + threadIdx.x;
  const LdsStack log{lds, int(blockDim.x), nullptr, 0};
  if constexpr (MODE == kBoxAdjoint) log_begin(G, log);
  UnitPool units(queue, total_units, gridDim.x * (blockDim.x >> 6));
  box_run<NS, MODE, F>(S, B, I, S.sensors[sensor], seed, spp, chunk_log2, grad_img, G, units, lds, log,
                       [&](unsigned u, const V3(&acc)[NS]) { store_unit<NS>(partial, u, acc); });
  // the whole wavefront is past its loop
  if constexpr (MODE == kBoxAdjoint) {
    log_close(G, log);
    log_end(G, log);
  }
}

}  // namespace

BoxScene bound_box(const Scene *s) {
  BoxScene B = s->box_scene;
  B.med = s->media[0];
  B.sigma = s->view.params[B.med.sigma_param];
  if (B.med.albedo_param >= 0) B.albedo = s->view.params[B.med.albedo_param];
  B.unit_extent = 1;
  for (int k = 0; k < 3; ++k)
    if (B.med.hi[k] - B.med.lo[k] != 1.0f) B.unit_extent = 0;
  return B;
}

void launch_box(const Scene *s, int ns, int mode, const BoxLaunch &L) {
  BoxScene B = bound_box(s);
  with_box_features(s->features(), [&](auto f) {
    constexpr int F = decltype(f)::value;
    auto go = [&](auto kern, size_t words) {
      const size_t lds = words * size_t(L.block) * sizeof(int);
      const unsigned grid = std::min(resident_grid(reinterpret_cast<const void *>(kern), L.block, lds),
                                     ceil_div(int64_t(L.units), L.block));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(L.block), lds, L.stream, s->view, B, L.I, L.sensor, L.seed, L.spp,
                         L.chunk_log2, L.grad_img, *L.G, L.partial, L.queue, L.units);
    };
    if (mode == kBoxAdjoint)
      go(box_kernel<1, kBoxAdjoint, F>, kBoxWords<kBoxAdjoint>);
    else if (mode == kBoxForward)
      go(box_kernel<1, kBoxForward, F>, kBoxWords<kBoxForward>);
    else if (ns == 2)
      go(box_kernel<2, kBoxRender, F>, kBoxWords<kBoxRender>);
    else
      go(box_kernel<1, kBoxRender, F>, kBoxWords<kBoxRender>);
  });
}

}  // namespace rcv
