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

// Units a wavefront draws from the device counter at once, for its lanes to
// take one by one (fewer towards the end of a launch). Every draw is an
// atomic on one address that all XCDs share, ~20 ns each: one draw per
// request of its lanes took as long as the tracking itself (128^3 render,
// 64 samples per pixel: 5.8 ms against 4.3 ms; 256 units at once: 4.4 ms).
constexpr unsigned kBoxGrab = 64;

// The work units of a wavefront: drawn from the launch's counter in grabs.
struct UnitPool {
  unsigned *queue;
  unsigned total, next, end;

  __device__ UnitPool(unsigned *q, unsigned n) : queue(q), total(n), next(0), end(0) {}

  // A unit for each lane that needs one (>= total: none left). All lanes of
  // the wavefront call it together, so next and end stay wave-uniform.
  __device__ unsigned take(bool need) {
    const uint64_t m = __ballot(need);
    if (m == 0) return 0;
    const unsigned want = unsigned(__popcll(m)), rank = unsigned(__popcll(m & __lanemask_lt()));
    const unsigned have = end - next;
    unsigned u = next + rank;
    if (have >= want || end >= total) {
      next = min(next + want, end);  // (past the end: u >= total)
    } else {
      const unsigned left = total - end;
      const unsigned grab = max(want - have, min(kBoxGrab, left / (gridDim.x * (blockDim.x >> 6) * 4u)));
      unsigned base = 0;
      if (__lane_id() == 0) base = atomicAdd(queue, grab);
      base = unsigned(__builtin_amdgcn_readfirstlane(int(base)));
      if (rank >= have) u = base + (rank - have);
      next = base + (want - have);
      end = base + grab;
    }
    return u;
  }
};

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
  const SensorInfo &sen = S.sensors[sensor];
  const int film_w = sen.film_w;
  const int max_depth = I.max_depth < 0 ? 0x7fffffff : I.max_depth;
  const UniformDiv by_maj((F & kFeatSupergrid) ? 1.0f : box_majorant<NS>(B, S.majorants));
  if constexpr (MODE == kBoxAdjoint) log_begin(G, log);
  BoxPath<NS, MODE, F> t;
  t.mode = kPathEnd;
  bool open = false;  // a sample of this lane's unit is under way
  int s = 0, s_end = 0, px = 0, py = 0;
  unsigned u = 0;
  V3 acc[NS];
  UnitPool units(queue, total_units);
  const float inv_spp = float(spp);
  while (true) {
    bool done;
    if (box_events_due(t.tracking(), t.mode == kIdle, done)) {
      const bool was_tracking = t.tracking();
      if (t.mode == kShadowExit) t.shadow_exit(B, lds);
      if (t.mode == kNeeDone) t.nee_done(B, lds);
      if (t.mode == kScatter) t.scatter(B, lds, G);
      if (t.mode == kPathExit) t.path_exit(B, I, lds);
      bool replay = false, need = false;
      if (t.mode == kPathEnd) {
        if (open) {
          if constexpr (MODE == kBoxRender) {
#pragma unroll
            for (int k = 0; k < NS; ++k) acc[k] += t.L[k];
            ++s;
          } else {
            if (MODE == kBoxForward && t.replay) acc[0] += t.dI;
            replay = !t.replay && any_nonzero(t.L[0]);
            if (!replay) ++s;
          }
          if (MODE != kBoxAdjoint && s >= s_end) {
            float *o = partial + int64_t(u) * (3 * NS);
#pragma unroll
            for (int k = 0; k < NS; ++k) {
              o[3 * k] = acc[k].x;
              o[3 * k + 1] = acc[k].y;
              o[3 * k + 2] = acc[k].z;
            }
          }
        }
        need = !replay && s >= s_end;
      }
      const unsigned taken = units.take(need);
      if (t.mode == kPathEnd) {
        open = true;
        if (need) {
          u = taken;
          if (u >= total_units) {
            t.mode = kIdle;
          } else {
            const unsigned pixel = u >> chunk_log2;
            const int chunk = int(u & ((1u << chunk_log2) - 1u));
            px = int(pixel % unsigned(film_w));
            py = int(pixel / unsigned(film_w));
            s = sample_end(chunk - 1, spp, chunk_log2);
            s_end = sample_end(chunk, spp, chunk_log2);
#pragma unroll
            for (int k = 0; k < NS; ++k) acc[k] = v3(0.f);
            if constexpr (MODE == kBoxAdjoint) {
              const float *gi = grad_img + 3 * int64_t(pixel);
              t.dL = v3(gi[0] / inv_spp, gi[1] / inv_spp, gi[2] / inv_spp);
              if (!any_nonzero(t.dL)) {
                s = s_end;
                open = false;
              }
            }
          }
        }
        if (t.mode != kIdle && open) {
          const int64_t pixel = int64_t(u >> chunk_log2);
          Pcg32 rng = lane_rng(seed, uint32_t(pixel * spp + s));
          const Ray r = camera_ray(sen, px, py, rng);
          t.begin(rng, r, replay, t.L[0]);
        }
      }
      if (t.mode == kOutside) t.outside(B, I, lds);
      if (!was_tracking && t.tracking()) t.begin_segment(B, lds);
    } else if (done) {
      break;
    }
    if (t.tracking()) t.step(S, B, I, max_depth, by_maj, G, log);
  }
  // the whole wavefront is past its loop
  if constexpr (MODE == kBoxAdjoint) log_end(G, log);
}

template <typename Fn>
void with_box_features(int f, Fn &&fn) {
  switch (f & (kFeatAlbedoGrid | kFeatSupergrid)) {
    case 0: fn(std::integral_constant<int, 0>{}); break;
    case kFeatAlbedoGrid: fn(std::integral_constant<int, kFeatAlbedoGrid>{}); break;
    case kFeatSupergrid: fn(std::integral_constant<int, kFeatSupergrid>{}); break;
    default: fn(std::integral_constant<int, kFeatAlbedoGrid | kFeatSupergrid>{}); break;
  }
}

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

}  // namespace

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
