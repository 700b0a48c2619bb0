// Device-side job table of a batch, shared by the batch's kernels.
#pragma once

#include "common.hpp"
#include "render_internal.hpp"
#include "scatter_log.hpp"
#include "volpath.hpp"

namespace rcv {

struct BatchJobDev {
  SceneView view;       // params[param].data[] rotated on the device
  IntegArgs integ;
  int32_t itype;        // RCV_INTEGRATOR_*
  int32_t method;       // 0 baseline (plain), 1 cv_ps (two-state + combine)
  int32_t loss;         // RCV_LOSS_*
  int32_t sensor;
  int32_t spp, spt, cl2;
  int32_t spp_g, spt_g, cl2_g;
  int32_t film_w, n_pix;
  uint32_t seed;
  int32_t param;
  int64_t n_param;
  int64_t n_img;
  int64_t unit_begin, unit_begin_g;  // in this job's render / adjoint class space
  int64_t elem_begin, pelem_begin;   // padded image / parameter element offsets
  float *ring[3];
  int32_t ring_old, ring_new, ring_next;
  uint32_t *maj_keys;   // scene majorant keys of `param`: [OLD], [NEW]
  uint32_t next_key;    // max key of the ring's next buffer (written by adam)
  int32_t iter;
  int32_t active;       // 0: the job sits out this iteration (no state changes)
  float *H, *F, *img, *grad_img;
  const float *img_ref;
  float *cv[8];
  int32_t warmup;
  float cv_b1, cv_b2;
  double cv_log_b1, cv_log_b2;
  int32_t pre_update;
  float *grad, *m, *v;
  GradTargets gt;       // gt.g[param] = grad, others null
  float lr, b1, b2, eps, clamp_lo, clamp_hi;
  double log_b1, log_b2;
  float *sg_out;        // supergrids [OLD][NEW] of the optimised grid's medium, or null
  int32_t sg_res[3];
  // One-box volume jobs (box_batch.hip): the tracker's scene, units per pixel
  // of the render and the adjoint, the job's unit counters and where the
  // render's unit sums go (null: one unit per pixel, written to F and H).
  BoxScene box;
  int32_t box_cl2, box_cl2_g;
  unsigned *box_queue;    // [0] render, [1] adjoint
  float *box_partial;
};

// Launch class of one-box volume jobs of one feature mask: job indices and
// their cumulative unit counts (render or adjoint).
struct BoxClass {
  const int32_t *ids;
  const int64_t *ends;
  int n;
};

// Launches the tracker over a class's jobs (ns 1 or 2: render; 0: adjoint,
// with the batch's scatter log pool).
void launch_box_batch(int features, int ns, BatchJobDev *jobs, const BoxClass &c, int64_t total, int block,
                      const GradTargets &pool, hipStream_t stream);

__device__ inline int find_job(const int64_t *__restrict__ ends, int n, int64_t u) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (ends[mid] <= u)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

__device__ inline uint32_t iter_seed(const BatchJobDev &J) { return J.seed + uint32_t(J.iter); }

__device__ inline uint32_t iter_seed_grad(const BatchJobDev &J) {
  uint32_t a = iter_seed(J), b = 1u;
  tea(a, b);
  return a;
}

}  // namespace rcv
