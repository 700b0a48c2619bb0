// The adjoint of volpathsimple (volsimple.hpp: plugins/volpathsimple.py) on
// the one-box tracker's machinery (boxpath.hpp): for its default estimator
// (NEE, DRT with subsampling) in scenes of one heterogeneous medium.
//
// A camera sample is a primal pass, the adjoint pass, one DRT segment and the
// recursive path from it, each a sequence of tracking loops whose lengths
// differ between the lanes. As nested loops a wavefront runs each as long as
// its longest lane does, and the calls' state goes through scratch memory
// (1.7 KB per lane). Here every lane is a state machine whose two kinds of
// tracking step -- free flight to a real collision, ratio tracking of a shadow
// ray or of the DRT segment -- are one instruction sequence, and everything
// between them an event, run when enough lanes wait for one
// (box_events_due). A shadow ray's weight is known before its replay from the
// primal pass (LDS slots), so the replay scatters as it tracks. Random
// numbers, decisions and scatter-adds are those of simple_sample, in the same
// order per sample.
//
// 64^3 grid, 128^2, 16 samples, majorant supergrid: 3.45 ms against 6.1 ms of
// the nested loops (both logged, and 0.5 ms of reduction); a 64^2 call of 4
// samples on 32^3, which waits for its longest path, 1.06 against 1.12 ms.
// Bound by instruction issue with 13 % of the lanes active: a tracking step
// walks the supergrid's cells one by one. With events run at half, one, two and three times as many waiting
// as tracking lanes the step takes 7.03, 6.64, 6.51 and 6.73 ms.
#pragma once

#include "boxpath.hpp"
#include "volsimple.hpp"

namespace rcv {

enum SimpleBoxMode : int {
  kSimFlight = 0,  // (tracking modes first)
  kSimRatio,
  kSimSegEnd,    // flight over: a real collision at o, or the boundary
  kSimRatioEnd,  // transmittance in T
  kSimEnd,       // pass over
  kSimIdle,
};
enum SimpleBoxPhase : int { kSimPrimal = 0, kSimAdjoint, kSimDrt, kSimRecursive };

// LDS words per lane.
constexpr int kSimPoint = 0;      // the path's point while a shadow ray is tracked (3)
constexpr int kSimSegment = 3;    // origin of the current flight (3), its boundary distance and face
constexpr int kSimReservoir = 8;  // kept segment: origin, direction (6), boundary distance, depth;
constexpr int kSimWeights = 16;   // its weights: sum and kept (6)
constexpr int kSimDrtPoint = 8;   // once it is sampled: the DRT point (3)
constexpr int kSimDrtWeight = 19; // after the segment's weight in kSimWeights (3): pdf, then weight; sigma_t
constexpr int kSimRng = 22;       // random state at a shadow ray's start and end when it is tracked again (4)
constexpr int kSimSlot0 = 26;     // NEE weights; the last word is the scatter log's
constexpr int kSimSlots = kLdsWordsPerThread - 1 - kSimSlot0;

template <int F>
struct SimpleBox {
  Pcg32 rng, alt;  // (rng continues alt from the DRT segment on)
  V3 o, d, inv, exit;
  float left;      // distance to the end of the segment
  float run_t;     // distance flown before the last tentative collision
  float T;         // transmittance; at a real collision: sigma_t
  float cs;        // replay: the shadow ray's weight
  V3 thr, L, dL;   // L: radiance gathered; in the adjoint pass: still to be gathered
  int mode, phase, depth, nee_k;
  bool inside, scattered, kept, retrack, entered, first;

  __device__ static int &word(int *lds, int j) { return lds[j * int(blockDim.x)]; }
  __device__ static float wordf(int *lds, int j) { return __int_as_float(word(lds, j)); }
  __device__ static void putf(int *lds, int j, float v) { word(lds, j) = __float_as_int(v); }
  __device__ static V3 words3(int *lds, int j) { return v3(wordf(lds, j), wordf(lds, j + 1), wordf(lds, j + 2)); }
  __device__ static void put3(int *lds, int j, V3 v) {
    putf(lds, j, v.x);
    putf(lds, j + 1, v.y);
    putf(lds, j + 2, v.z);
  }
  __device__ static uint64_t words64(int *lds, int j) {
    return (uint64_t(unsigned(word(lds, j + 1))) << 32) | uint64_t(unsigned(word(lds, j)));
  }
  __device__ static void put64(int *lds, int j, uint64_t v) {
    word(lds, j) = int(unsigned(v));
    word(lds, j + 1) = int(unsigned(v >> 32));
  }

  __device__ bool tracking() const { return mode <= kSimRatio; }

  // Closest crossing of the box along (o, d), kInf and face -1 for none.
  __device__ float boundary(const BoxScene &B, V3 from, V3 dir, int &face) const {
    Ray r;
    r.o = from;
    r.d = dir;
    r.maxt = kInf;
    return box_trace(B, r, v3(1.0f / dir.x, 1.0f / dir.y, 1.0f / dir.z), face);
  }

  // (o, d) is set: what the tracking steps along it need.
  __device__ void begin_segment(const MediumInfo &M) {
    inv = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    exit = v3(inv.x >= 0.0f ? M.hi[0] : M.lo[0], inv.y >= 0.0f ? M.hi[1] : M.lo[1], inv.z >= 0.0f ? M.hi[2] : M.lo[2]);
    inside = o.x > M.lo[0] && o.x < M.hi[0] && o.y > M.lo[1] && o.y < M.hi[1] && o.z > M.lo[2] && o.z < M.hi[2];
  }

  // spawn_ray at the stored boundary of the flight from `from` along d.
  __device__ V3 crossed(const BoxScene &B, V3 from, float t, int face) const {
    Ray r;
    r.o = from;
    r.d = d;
    r.maxt = kInf;
    return offset_point(ray_at(r, t), v3(B.box.n[3 * face], B.box.n[3 * face + 1], B.box.n[3 * face + 2]), d);
  }

  // The environment at the end of an escaped path (:253-281) whose ray starts
  // at `from`.
  __device__ void gather_env(const BoxScene &B, const IntegArgs &I, V3 from) {
    if (depth <= 0 && I.hide_emitters) return;
    int face;
    (void)boundary(B, from, d, face);
    if (face >= 0) return;
    const float mis = depth > 0 ? mis_weight(kInv4Pi, kInv4Pi) : mis_weight(1.0f, 0.0f);
    L += thr * v3(B.env[0], B.env[1], B.env[2]) * mis;
  }

  // The primal or the adjoint pass of a camera sample (:86-108).
  __device__ void begin(const BoxScene &B, const IntegArgs &I, int *lds, const Pcg32 &r, const Ray &camera,
                        int phase_) {
    rng = r;
    phase = phase_;
    thr = v3(1.f);
    depth = 0;
    nee_k = 0;
    retrack = kept = first = false;
    o = camera.o;
    d = camera.d;
    if (phase == kSimPrimal) L = v3(0.f);
    else put3(lds, kSimWeights, v3(0.f));
    (void)rng.next_1d();
    mode = kSimEnd;
    int face;
    const float t = boundary(B, o, d, face);
    entered = face >= 0;
    if (!entered) {
      gather_env(B, I, o);  // (no adjoint pass follows)
      return;
    }
    o = crossed(B, o, t, face);
    (void)next_boundary(B, lds);
    if (word(lds, kSimSegment + 4) < 0) return;
    (void)rng.next_1d();  // seed of the gradient-only stream (:108)
    begin_flight(I, lds);
  }

  __device__ int next_boundary(const BoxScene &B, int *lds) {
    int face;
    putf(lds, kSimSegment + 3, boundary(B, o, d, face));
    word(lds, kSimSegment + 4) = face;
    return face;
  }

  // Russian roulette (:127-132), then a flight from o along d.
  __device__ void begin_flight(const IntegArgs &I, int *lds) {
    const float q = fminf(hmax(thr), 0.99f);
    const bool perform_rr = depth > I.rr_depth;
    const float urr = rng.next_1d();
    if (!any_nonzero(thr) || (perform_rr && !(urr < q))) {
      mode = kSimEnd;
      return;
    }
    if (perform_rr) thr = thr * (1.0f / q);
    put3(lds, kSimSegment, o);
    left = wordf(lds, kSimSegment + 3);
    run_t = 0.0f;
    mode = kSimFlight;
  }

  // One tentative collision of the flight or of ratio tracking.
  __device__ void step(const SceneView &S, const BoxScene &B, const UniformDiv &by_maj, const GradTargets &G,
                       const LdsStack &log) {
    const MediumInfo &M = B.med;
    const bool ratio = mode == kSimRatio;
    const float u = rng.next_1d();
    float mint = 0.0f;
    float maxt = fminf(fminf((exit.x - o.x) * inv.x, (exit.y - o.y) * inv.y), (exit.z - o.z) * inv.z);
    bool ok = inside && maxt > 0.0f;
    if (!ok) {
      float t0;
      ok = box_slab(o, inv, M.lo, M.hi, t0, maxt);
      ok = ok && (t0 < kInf || maxt < kInf);
      mint = ok ? fmaxf(0.0f, t0) : 0.0f;
    }
    maxt = ok ? fminf(left, maxt) : kInf;
    const float tau = tau_of(u);
    Ray r;
    r.o = o;
    r.d = d;
    r.maxt = left;
    float maj, t;
    if constexpr ((F & kFeatSupergrid) != 0) {
      maj = 0.0f;
      t = kInf;
      if (ok) t = supergrid_free_flight<1>(S, M, r, mint, maxt, tau, maj);
    } else {
      maj = by_maj.y;
      t = mint + by_maj(tau);
    }
    ok = ok && maj > 0.0f && maj < kInf;
    if (!(ok && t <= maxt)) {
      scattered = false;
      mode = ratio ? kSimRatioEnd : kSimSegEnd;
      return;
    }
    auto over_maj = [&](float x) {
      if constexpr ((F & kFeatSupergrid) != 0)
        return x / maj;
      else
        return by_maj(x);
    };
    const V3 p = ray_at(r, t);
    GridFoot foot;
    int x0;
    box_footprint(B, p, foot, x0);
    const float st = M.scale * box_eval1(B.sigma.data[RCV_STATE_NEW], foot, x0, B.sigma.nx);
    const float sn = sigma_null(maj, st);
    o = p;
    left -= t;
    if (ratio) {
      const float tr = over_maj(sn);
      float *const g = G.g[M.sigma_param];
      if (phase == kSimAdjoint && tr > 0.0f && cs != 0.0f && g)
        scatter_density(&G, log, M.sigma_param, g, foot, p, -cs * M.scale / sn);
      T *= tr;
      if (T == 0.0f) mode = kSimRatioEnd;
    } else {
      const float un = rng.next_1d();
      if (!(un >= over_maj(st))) {
        scattered = true;
        T = st;
        run_t = t + run_t;
        mode = kSimSegEnd;
      } else {
        run_t += t;
      }
    }
  }

  __device__ V3 albedo_at(const BoxScene &B, V3 p, GridFoot &fa) const {
    if constexpr ((F & kFeatAlbedoGrid) != 0) {
      grid_footprint(B.albedo, B.med, p, fa);
      return grid_eval3(B.albedo.data[RCV_STATE_NEW], fa);
    }
    return v3(B.med.albedo[0], B.med.albedo[1], B.med.albedo[2]);
  }

  // The end of a flight (:137-236).
  __device__ void seg_end(const BoxScene &B, const IntegArgs &I, int max_depth, int *lds, const GradTargets &G,
                          const LdsStack &log) {
    const MediumInfo &M = B.med;
    const float si_t = wordf(lds, kSimSegment + 3);
    Ray seg;
    seg.o = words3(lds, kSimSegment);
    seg.d = d;
    seg.maxt = kInf;
    GridFoot fa;
    const V3 alb = scattered ? albedo_at(B, o, fa) : v3(1.f);
    if (phase == kSimAdjoint) {
      // reservoir over the segments, weight = throughput (:743-766)
      const V3 wsum = words3(lds, kSimWeights) + thr;
      put3(lds, kSimWeights, wsum);
      const float ur = alt.next_1d();
      const V3 ratio = v3(thr.x / wsum.x, thr.y / wsum.y, thr.z / wsum.z);
      if (ur <= (ratio.x + ratio.y + ratio.z) * (1.0f / 3.0f)) {
        kept = true;
        put3(lds, kSimWeights + 3, thr);
        put3(lds, kSimReservoir, seg.o);
        put3(lds, kSimReservoir + 3, d);
        putf(lds, kSimReservoir + 6, si_t);
        word(lds, kSimReservoir + 7) = depth;
      }
      float *const gd = G.g[M.sigma_param];
      // collision term (:150-180)
      if (scattered && !(I.flags & kSimpleNoDrtMis) && T > 0.0f) {
        const float s2 = T * T;
        const float mis = s2 / (1.0f + s2);
        const V3 li = v3(L.x / fmaxf(1e-8f, alb.x), L.y / fmaxf(1e-8f, alb.y), L.z / fmaxf(1e-8f, alb.z));
        const V3 dl = dL * li;
        if (gd) {
          GridFoot f;
          grid_footprint(B.sigma, M, o, f);
          scatter_density(&G, log, M.sigma_param, gd, f, o, mis * dot(dl, alb) * M.scale / T);
        }
        if constexpr ((F & kFeatAlbedoGrid) != 0) {
          float *const ga = G.g[M.albedo_param];
          if (ga) scatter_grid3(ga, fa, dl * mis);
        }
      }
      // transmittance: 4 uniform points of the segment (:559-583)
      const float interval = scattered ? run_t : si_t;
      const float lr = dot(dL, L);
      for (int j = 0; j < 4; ++j) {
        const float tj = alt.next_1d() * interval;
        if (gd && lr != 0.0f && interval < kInf) {
          GridFoot f;
          const V3 pj = ray_at(seg, tj);
          grid_footprint(B.sigma, M, pj, f);
          scatter_density(&G, log, M.sigma_param, gd, f, pj, -lr * M.scale * interval * 0.25f);
        }
      }
    }
    thr = thr * alb;
    if (!scattered) {
      const int face = word(lds, kSimSegment + 4);
      if (phase != kSimAdjoint) gather_env(B, I, face >= 0 ? crossed(B, seg.o, si_t, face) : seg.o);
      mode = kSimEnd;
      return;
    }
    depth += 1;
    if (depth < max_depth)
      begin_nee(B, lds);
    else
      mode = kSimEnd;
  }

  // NEE at o (:370-413): the emitter sample and the shadow ray to the boundary.
  __device__ void begin_nee(const BoxScene &B, int *lds) {
    put3(lds, kSimPoint, o);
    cs = 0.0f;
    if (phase == kSimAdjoint) {
      if (nee_k < kSimSlots)
        cs = wordf(lds, kSimSlot0 + nee_k);
      else
        put64(lds, kSimRng, rng.state);
    }
    begin_shadow(B);
  }

  __device__ void begin_shadow(const BoxScene &B) {
    const float u1 = rng.next_1d();
    const float u2 = rng.next_1d();
    d = square_to_uniform_sphere(u1, u2);
    int face;
    left = boundary(B, o, d, face);
    T = face >= 0 ? 1.0f : 0.0f;
    mode = face >= 0 ? kSimRatio : kSimRatioEnd;
  }

  // Transmittance known: the NEE's contribution and the next flight, or the
  // DRT point.
  __device__ void ratio_end(const BoxScene &B, const IntegArgs &I, int max_depth, int *lds) {
    if (phase == kSimDrt) {
      drt_point(B, lds);
      return;
    }
    o = words3(lds, kSimPoint);
    if (retrack) {
      retrack = false;
      rng.state = words64(lds, kSimRng + 2);
    } else {
      const V3 em = v3(B.env[0], B.env[1], B.env[2]) * (4.0f * kPi * 1.0f) * T;
      const V3 c = thr * em * (kInv4Pi * mis_weight(kInv4Pi, kInv4Pi));
      const int k = nee_k++;
      if (phase == kSimAdjoint) {
        L -= c;
        const float w = dot(dL, c);
        if (k >= kSimSlots && w != 0.0f) {
          // past the slots: track the shadow ray again, now with its weight
          put64(lds, kSimRng + 2, rng.state);
          rng.state = words64(lds, kSimRng);
          cs = w;
          retrack = true;
          begin_shadow(B);
          return;
        }
      } else {
        L += c;
        if (phase == kSimPrimal && k < kSimSlots) putf(lds, kSimSlot0 + k, dot(dL, c));
      }
    }
    // phase sampling, isotropic (:203-210)
    (void)rng.next_1d();
    const float a = rng.next_1d();
    const float b = rng.next_1d();
    d = square_to_uniform_sphere(a, b);
    const int face = next_boundary(B, lds);
    mode = kSimEnd;
    if (first) {
      // the recursive path starts here (:586-633)
      first = false;
      (void)rng.next_1d();
      if (depth < max_depth) begin_flight(I, lds);
    } else if (face >= 0) {  // (accidental escape: absorbed)
      begin_flight(I, lds);
    }
  }

  // DRT along the reservoir's segment (simple_drt).
  __device__ void begin_drt(const SceneView &S, const BoxScene &B, int *lds) {
    const MediumInfo &M = B.med;
    const V3 wsum = words3(lds, kSimWeights), cur = words3(lds, kSimWeights + 3);
    const float dm = (cur.x + cur.y + cur.z) * (1.0f / 3.0f);
    const float wm = (wsum.x + wsum.y + wsum.z) * (1.0f / 3.0f);
    const V3 sw = dm != 0.0f ? cur * (wm / dm) : v3(0.f);
    Ray ray;
    ray.o = words3(lds, kSimReservoir);
    ray.d = words3(lds, kSimReservoir + 3);
    ray.maxt = wordf(lds, kSimReservoir + 6);
    float t0, t1;
    const bool hit = ray_aabb(ray, M.lo, M.hi, t0, t1);
    const float mint = fmaxf(0.0f, t0);
    const float maxt = fminf(ray.maxt, t1);
    const float maj = majorant_of(S, M.sigma_param, RCV_STATE_NEW) * M.scale;
    rng = alt;
    const float u = rng.next_1d();
    const float len = maxt - mint;
    mode = kSimEnd;
    phase = kSimRecursive;
    kept = false;
    if (!hit || !(len > 0.0f) || !(len < kInf) || !(maj > 0.0f) || !(maj < kInf)) return;
    const float norm = -expm1f(-maj * len);
    const float s = -log1pf(-u * norm) / maj;
    put3(lds, kSimWeights, sw * dL);
    putf(lds, kSimDrtWeight, maj * expf(-maj * s) / norm);
    put3(lds, kSimDrtPoint, ray_at(ray, mint + s));
    depth = word(lds, kSimReservoir + 7);
    o = ray_at(ray, mint);
    d = ray.d;
    left = s;
    T = 1.0f;
    cs = 0.0f;
    kept = true;
    phase = kSimDrt;
    mode = kSimRatio;
  }

  // T(s) known: the weight of the DRT point, and its incident radiance by NEE
  // and a recursive path.
  __device__ void drt_point(const BoxScene &B, int *lds) {
    const float pdf = wordf(lds, kSimDrtWeight);
    const float weight = pdf > 0.0f ? T / pdf : 0.0f;
    phase = kSimRecursive;
    mode = kSimEnd;
    if (weight == 0.0f) {  // adds nothing
      kept = false;
      return;
    }
    putf(lds, kSimDrtWeight, weight);
    o = words3(lds, kSimDrtPoint);
    L = v3(0.f);
    thr = v3(1.f);
    depth += 1;
    nee_k = 0;
    first = true;
    begin_nee(B, lds);
  }

  // The DRT term, L its incident radiance.
  __device__ void drt_scatter(const BoxScene &B, const IntegArgs &I, int *lds, const GradTargets &G,
                              const LdsStack &log) {
    const MediumInfo &M = B.med;
    const V3 p = words3(lds, kSimDrtPoint);
    GridFoot f, fa;
    grid_footprint(B.sigma, M, p, f);
    const float st = M.scale * grid_eval1(B.sigma.data[RCV_STATE_NEW], f);
    const V3 alb = albedo_at(B, p, fa);
    const float mis = (I.flags & kSimpleNoDrtMis) ? 1.0f : 1.0f / (1.0f + st * st);
    const V3 a = words3(lds, kSimWeights) * L * (mis * wordf(lds, kSimDrtWeight));
    float *const gd = G.g[M.sigma_param];
    if (gd) scatter_density(&G, log, M.sigma_param, gd, f, p, dot(a, alb) * M.scale);
    if constexpr ((F & kFeatAlbedoGrid) != 0) {
      float *const ga = G.g[M.albedo_param];
      if (ga) scatter_grid3(ga, fa, a * st);
    }
  }
};

// Runs the units a wavefront draws from `units` until none is left for any of
// its lanes (all 64 lanes call it): the adjoint of their camera samples into
// G, through the scatter log where it is set.
template <int F>
__device__ inline void simple_box_run(const SceneView &S, const BoxScene &B, const IntegArgs &I,
                                      const SensorInfo &sen, uint32_t seed, int spp, int chunk_log2,
                                      const float *grad_img, const GradTargets &G, UnitPool &units, int *lds,
                                      const LdsStack &log) {
  const int film_w = sen.film_w;
  const int max_depth = I.max_depth < 0 ? 0x7fffffff : I.max_depth;
  const uint32_t alt_seed = simple_alt_seed(seed);
  const UniformDiv by_maj((F & kFeatSupergrid) ? 1.0f : box_majorant<1>(B, S.majorants));
  SimpleBox<F> t;
  t.mode = kSimEnd;
  bool open = false;  // a sample of this lane's unit is under way
  int s = 0, s_end = 0, px = 0, py = 0;
  unsigned u = 0;
  const float inv_spp = float(spp);
  while (true) {
    bool done;
    if (box_events_due(t.tracking(), t.mode == kSimIdle, done)) {
      const bool was_tracking = t.tracking();
      if (t.mode == kSimRatioEnd) t.ratio_end(B, I, max_depth, lds);
      if (t.mode == kSimSegEnd) t.seg_end(B, I, max_depth, lds, G, log);
      bool need = false, adjoint = false;
      if (t.mode == kSimEnd) {
        if (open) {
          if (t.phase == kSimPrimal && t.entered) {
            adjoint = true;
          } else if (t.phase == kSimAdjoint && t.kept) {
            t.begin_drt(S, B, lds);
          } else if (t.phase == kSimRecursive && t.kept) {
            t.drt_scatter(B, I, lds, G, log);
          }
          if (t.mode == kSimEnd && !adjoint) ++s;
        }
        need = t.mode == kSimEnd && !adjoint && s >= s_end;
      }
      const unsigned taken = units.take(need);
      if (t.mode == kSimEnd) {
        open = true;
        if (need) {
          u = taken;
          if (u >= units.total) {
            t.mode = kSimIdle;
          } else {
            const unsigned pixel = u >> chunk_log2;
            const int chunk = int(u & ((1u << chunk_log2) - 1u));
            px = int(pixel % unsigned(film_w));
            py = int(pixel / unsigned(film_w));
            s = sample_end(chunk - 1, spp, chunk_log2);
            s_end = sample_end(chunk, spp, chunk_log2);
            const float *gi = grad_img + 3 * int64_t(pixel);
            t.dL = v3(gi[0] / inv_spp, gi[1] / inv_spp, gi[2] / inv_spp);
            if (!any_nonzero(t.dL)) {
              s = s_end;
              open = false;
            }
          }
        }
        if (t.mode != kSimIdle && open) {
          const int64_t pixel = int64_t(u >> chunk_log2);
          const uint32_t lane = uint32_t(pixel * spp + s);
          Pcg32 rng = lane_rng(seed, lane);
          const Ray r = camera_ray(sen, px, py, rng);
          if (adjoint) t.alt = lane_rng(alt_seed, lane);
          t.begin(B, I, lds, rng, r, adjoint ? kSimAdjoint : kSimPrimal);
        }
      }
      if (!was_tracking && t.tracking()) t.begin_segment(B.med);
    } else if (done) {
      break;
    }
    if (t.tracking()) t.step(S, B, by_maj, G, log);
  }
}

}  // namespace rcv
