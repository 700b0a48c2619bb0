// Host-side scene object behind the opaque rcv_scene handle.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "scene_types.hpp"

namespace rcv {

// Persistent volume renders split a pixel into at most this many work units;
// their unit-sum buffer is sized for it at scene commit. Four units (8 of 32
// samples each) against two: the 64^3 two-state render at the mid / final
// state of the optimisation 15.9 / 21.5 -> 12.6 / 15.8 ms, 3.1 -> 3.7 ms at
// the uniform initial state (eight: 12.3 / 14.8, 4.4 ms).
constexpr int kRenderMaxUnitsPerPixel = 4;
// Small images of the one-box tracker's scenes may be split further, into up
// to 64 units per pixel, as long as the buffer stays within this many units
// (6 MB; one per lane the device holds).
constexpr int64_t kRenderMinUnits = int64_t(1) << 18;

struct Param {
  int kind = 0;
  int nx = 0, ny = 0, nz = 0, ch = 0;
  const float *data[2] = {nullptr, nullptr};
};

// What a persistent launch needs beside its arguments: the counter its lanes
// draw work units from and, for renders and forward mode, the units' sums
// (Scene::partial_cap floats). One per stream that a scene is used on, so that
// launches on different streams may overlap, and one for the launches of
// captured graphs, which run on whatever stream replays them.
struct LaunchScratch {
  unsigned *queue = nullptr;
  float *partial = nullptr;
};
// Streams with a scratch of their own, at most: another one takes over the
// scratch that was used longest ago, once the device is idle.
constexpr int kMaxScratchStreams = 32;

struct Scene {
  // collected before commit
  std::vector<Param> params;
  std::vector<BsdfInfo> bsdfs;
  std::vector<MediumInfo> media;
  std::vector<EmitterInfo> emitters;
  std::vector<ShapeInfo> shapes;
  std::vector<SensorInfo> sensors;
  std::vector<float> tri_v;     // 9 floats per triangle
  std::vector<float> tri_uv;    // 6 floats per triangle
  std::vector<int32_t> tri_shape;
  std::vector<float> sph;       // center xyz, radius
  std::vector<int32_t> sph_shape;
  std::vector<float> box_xf;    // per box: 3x4 object-to-world map, row-major
  std::vector<int32_t> box_shape;

  // after commit
  bool committed = false;
  void *dev_block = nullptr;
  uint32_t *majorant_keys = nullptr;  // [param][state], order-preserving float keys
  float *supergrids = nullptr;      // sg_block: [medium][state][cell]
  void *sg_block = nullptr;
  int64_t sg_capacity = 0;          // floats
  MediumInfo *media_dev = nullptr;  // device copy of `media`
  int batch_refs = 0;               // batches holding this scene (no relayout then)
  unsigned long long *counters = nullptr;
  int64_t partial_cap = 0;          // floats of a LaunchScratch's unit sums
  struct OwnedScratch {
    LaunchScratch mem;
    hipStream_t stream;  // of eager launches
    bool captured;       // of captured launches
    uint64_t used;       // 0: not used yet
  };
  mutable std::vector<OwnedScratch> scratches;
  mutable uint64_t scratch_uses = 0;
  int n_nodes = 0;
  float bs_center[3] = {0, 0, 0};
  float bs_radius = 0;
  SceneView view{};
  bool one_box = false;             // box_scene describes the scene (set at commit)
  BoxScene box_scene{};

  Scene() = default;
  Scene(const Scene &) = delete;
  Scene &operator=(const Scene &) = delete;
  ~Scene();

  int upload(hipStream_t stream);
  // The scratch of eager launches on `stream`, or of captured ones.
  int scratch(hipStream_t stream, bool captured, LaunchScratch &out) const;
  int add_scratch(hipStream_t stream, bool captured) const;
  int reduce_param(int param, int state, hipStream_t stream);
  int build_supergrid(int medium, int state, hipStream_t stream);
  int64_t plan_supergrids();
  int alloc_supergrids();
  int relayout_supergrids(hipStream_t stream);
  int features() const;  // kFeat* mask of the committed scene
  bool box_path() const;  // whether the one-box volume tracker covers the scene
};

// Decodes an order-preserving key written by the majorant reduction.
__host__ __device__ inline float key_to_float(uint32_t k) {
  const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __builtin_bit_cast(float, u);
}

}  // namespace rcv

// The opaque C handle is the scene object itself.
struct rcv_scene : public rcv::Scene {};
