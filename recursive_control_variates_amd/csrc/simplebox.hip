// Launch of volpathsimple's adjoint on the one-box tracker (simplebox.hpp): a
// persistent grid of the resident waves whose lanes pull work units (a
// pixel's chunk of camera samples) from a device counter.

#include <algorithm>

#include "common.hpp"
#include "render_internal.hpp"
#include "simplebox.hpp"

namespace rcv {
namespace {

constexpr int kSimpleBoxMaxBlock = 256;

template <int F>
__global__ __launch_bounds__(kSimpleBoxMaxBlock) __attribute__((amdgpu_waves_per_eu(kSimpleBoxWaves))) void
simple_box_kernel(SceneView S, BoxScene B, IntegArgs I, int sensor, uint32_t seed, int spp, int chunk_log2,
                  const float *__restrict__ grad_img, GradTargets G, unsigned *queue, unsigned total_units) {
  extern __shared__ int lds_words[];  // kLdsWordsPerThread words per thread
  int *const lds = lds_words + threadIdx.x;
  const LdsStack log{lds, int(blockDim.x), nullptr, 0};
  log_begin(G, log);
  UnitPool units(queue, total_units, gridDim.x * (blockDim.x >> 6));
  simple_box_run<F>(S, B, I, S.sensors[sensor], seed, spp, chunk_log2, grad_img, G, units, lds, log);
  // the whole wavefront is past its loop
  log_close(G, log);
  log_end(G, log);
}

}  // namespace

void launch_simple_box(const Scene *s, const BoxLaunch &L) {
  const BoxScene B = bound_box(s);
  with_box_features(s->features(), [&](auto f) {
    auto kern = simple_box_kernel<decltype(f)::value>;
    const size_t lds = size_t(kLdsWordsPerThread) * size_t(L.block) * sizeof(int);
    const unsigned grid =
        std::min(resident_grid(reinterpret_cast<const void *>(kern), L.block, lds), ceil_div(int64_t(L.units), L.block));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(L.block), lds, L.stream, s->view, B, L.I, L.sensor, L.seed, L.spp,
                       L.chunk_log2, L.grad_img, *L.G, L.queue, L.units);
  });
}

}  // namespace rcv
