// The one-box volume tracker (boxpath.hpp) over the jobs of a batch: one
// persistent launch per feature mask whose wavefronts start on the job that
// lies at their share of the class's work units, draw that job's units from
// its own counter, and move on to the other jobs in order when it runs out. A
// wavefront works on one job at a time, so the job's scene is wave-uniform
// and is read through the scalar cache.

#include <algorithm>

#include "batch_internal.hpp"
#include "boxpath.hpp"

namespace rcv {
namespace {

constexpr int kBatchBoxBlock = 256;  // at most

template <int NS, int MODE, int F>
__global__ __launch_bounds__(kBatchBoxBlock) __attribute__((amdgpu_waves_per_eu(kBoxWaves<NS, MODE>))) void
batch_box_kernel(const BatchJobDev *jobs, BoxClass c, int64_t total, GradTargets pool) {
  extern __shared__ int lds_words[];  // kBoxWords<MODE> words per thread
  int *const lds = lds_words + threadIdx.x;
  const LdsStack log{lds, int(blockDim.x), nullptr, 0};
  if constexpr (MODE == kBoxAdjoint) log_begin(pool, log);
  const int64_t waves = int64_t(gridDim.x) * (blockDim.x >> 6);
  const int64_t wave = int64_t(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int first = __builtin_amdgcn_readfirstlane(find_job(c.ends, c.n, wave * total / waves));
  for (int k = 0; k < c.n; ++k) {
    const int q = first + k < c.n ? first + k : first + k - c.n;
    const int id = __builtin_amdgcn_readfirstlane(c.ids[q]);
    // job records do not change while the kernel runs: constant address space
    const BatchJobDev &J =
        *(const BatchJobDev *)(reinterpret_cast<const __attribute__((address_space(4))) BatchJobDev *>(
            reinterpret_cast<uintptr_t>(jobs + id)));
    if (!J.active) continue;
    constexpr bool kRender = MODE == kBoxRender;
    const int cl2 = kRender ? J.box_cl2 : J.box_cl2_g;
    const unsigned n_units = unsigned(J.n_pix) << cl2;
    unsigned *const queue = J.box_queue + (kRender ? 0 : 1);
    const unsigned drawn = __hip_atomic_load(queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (unsigned(__builtin_amdgcn_readfirstlane(int(drawn))) >= n_units) continue;
    UnitPool units(queue, n_units, unsigned(max(int64_t(1), waves * int64_t(n_units) / total)));
    const uint32_t seed = kRender ? iter_seed(J) : iter_seed_grad(J);
    box_run<NS, MODE, F>(J.view, J.box, J.integ, J.view.sensors[J.sensor], seed, kRender ? J.spp : J.spp_g, cl2,
                         J.grad_img, J.gt, units, lds, log, [&](unsigned u, const V3(&acc)[NS]) {
                           if (J.box_partial) {
                             store_unit<NS>(J.box_partial, u, acc);
                             return;
                           }
                           // one unit per pixel: its means
                           const float n = float(J.spp);
#pragma unroll
                           for (int q = 0; q < NS; ++q) {
                             float *o = (q == NS - 1 ? J.F : J.H) + int64_t(u) * 3;
                             o[0] = acc[q].x / n;
                             o[1] = acc[q].y / n;
                             o[2] = acc[q].z / n;
                           }
                         });
    if constexpr (MODE == kBoxAdjoint) log_close(J.gt, log);
  }
  if constexpr (MODE == kBoxAdjoint) log_end(pool, log);
}

}  // namespace

void launch_box_batch(int features, int ns, BatchJobDev *jobs, const BoxClass &c, int64_t total, int block,
                      const GradTargets &pool, hipStream_t stream) {
  with_box_features(features, [&](auto f) {
    constexpr int F = decltype(f)::value;
    auto go = [&](auto kern, size_t words) {
      const int threads = std::min(block, kBatchBoxBlock);
      const size_t lds = words * size_t(threads) * sizeof(int);
      const unsigned grid =
          std::min(resident_grid(reinterpret_cast<const void *>(kern), threads, lds), ceil_div(total, threads));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, stream, jobs, c, total, pool);
    };
    if (ns == 0)
      go(batch_box_kernel<1, kBoxAdjoint, F>, kBoxWords<kBoxAdjoint>);
    else if (ns == 2)
      go(batch_box_kernel<2, kBoxRender, F>, kBoxWords<kBoxRender>);
    else
      go(batch_box_kernel<1, kBoxRender, F>, kBoxWords<kBoxRender>);
  });
}

}  // namespace rcv
