// The volumetric path tracer (VolPath, volpath.hpp) for the scenes its
// optimisations run in: one heterogeneous medium inside one null-boundary
// box under a constant environment (BoxScene). Same random numbers, same
// decisions and the same floating-point expressions per camera sample; what
// differs is how the lanes of a wavefront are scheduled and where the scene
// lives.
//
// What bounds the tracker is instruction issue with most lanes masked off
// (12 % of the lanes of a VALU instruction active in the general adjoint, 21
// % in the general two-state render, 64^3 workload): paths alternate between
// many cheap tracking steps (free flight, one grid lookup, a decision) and
// rare long events (a real scattering with its emitter sample, a boundary
// crossing, the next camera sample), and a wavefront that runs a path one
// bounce at a time executes every event with the few lanes that are at one.
// Here a lane is a state machine (BoxMode). One tracking step serves a path
// and a shadow ray alike, so in each trip every lane that can track takes a
// step, and lanes at an event wait until twice as many wait as track (or none
// can track); then all events run together: 28 % (two-state) and 31 %
// (adjoint) of the lanes active, ~310 and ~280 lane operations per tracking step
// with its share of the events. The scene's uniform
// data are kernel arguments (scalar registers) instead of tables in memory,
// a direction's reciprocals are kept between its steps, and the two x
// neighbours of a lookup are one 8-byte load.
#pragma once

#include "render_internal.hpp"
#include "volpath.hpp"

namespace rcv {

// What a lane does next: track (path or shadow ray), or the event it waits
// for.
enum BoxMode : int {
  kOnPath = 0,
  kOnShadow = 1,
  kShadowExit = 2,  // the shadow ray has reached the box boundary
  kNeeDone = 3,     // its transmittance is known
  kScatter = 4,     // real collision
  kPathExit = 5,    // the path has reached the box boundary
  kPathEnd = 6,     // the path is over
  kOutside = 7,     // a path outside the box
  kIdle = 8,        // no work left
};

// LDS words per lane (one per lane and word, strided by the block size): the
// path's point and direction while a shadow ray is tracked (0-5), the next
// boundary point (6-8) and face (9), and for the adjoint the random state at
// a shadow ray's start (10-11) and at its end (12-13) when it is tracked
// again, then the NEE weights (kBoxSlot0 ..). The last word of kLdsWords is
// the scatter log's.
constexpr int kBoxRenderWords = 10;
constexpr int kBoxSlot0 = 14;
constexpr int kBoxSlots = kLdsWordsPerThread - 1 - kBoxSlot0;

template <int MODE>
constexpr int kBoxWords = MODE == kBoxAdjoint ? kLdsWordsPerThread : kBoxRenderWords;

// Division by a wave-uniform value y, correctly rounded, from its correctly
// rounded reciprocal: two residual corrections of x r (Markstein, "Computation
// of elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34, 1990: with r = RN(1 / y) and a quotient within one ulp, adding the
// exactly computed residual times r rounds correctly). The first correction
// brings the quotient within one ulp, the second rounds it. Five
// instructions in place of a division's eleven; y outside [2^-100, 2^100],
// where a residual could underflow, divides.
struct UniformDiv {
  float y, r;
  bool fast;
  __device__ explicit UniformDiv(float v) : y(v), r(1.0f / v), fast(v >= 0x1p-100f && v <= 0x1p+100f) {}
  __device__ float operator()(float x) const {
    if (!fast) return x / y;
    float q = x * r;
    q = __builtin_fmaf(__builtin_fmaf(-q, y, x), r, q);
    return __builtin_fmaf(__builtin_fmaf(-q, y, x), r, q);
  }
};

// Pcg32 kept at the state of the last number drawn instead of the next one,
// so that a number that is skipped costs nothing when one is drawn after it:
// two steps of the generator are a^2 state + (a + 1) inc, with inc2 = (a +
// 1) inc kept. Its 64-bit multiply is the largest part of a draw.
struct LazyPcg {
  static constexpr uint64_t kMul = 6364136223846793005ULL;
  uint64_t state, inc, inc2;

  // The numbers of `r`, its next one skipped.
  __device__ void begin_skip(const Pcg32 &r) {
    state = r.state;
    inc = r.inc;
    inc2 = inc * (kMul + 1u);
  }
  __device__ float current() const {
    const uint32_t xs = uint32_t(((state >> 18u) ^ state) >> 27u);
    const uint32_t rot = uint32_t(state >> 59u);
    const uint32_t out = (xs >> rot) | (xs << ((~rot + 1u) & 31u));
    return __builtin_bit_cast(float, (out >> 9) | 0x3f800000u) - 1.0f;
  }
  __device__ float next() {
    state = state * kMul + inc;
    return current();
  }
  __device__ float skip_next() {
    skip2();
    return current();
  }
  __device__ void skip() { state = state * kMul + inc; }
  __device__ void skip2() { state = state * (kMul * kMul) + inc2; }
};

// hit_box / hit_boxprim of the scene's only primitive: the closest crossing
// of the box in (0, maxt), kInf and face -1 for none (trace() and its BVH
// root test).
__device__ inline float box_trace(const BoxScene &B, const Ray &r, V3 inv, int &face) {
  float tn, t;
  face = -1;
  if (!hit_box(B.root, r.o, inv, r.maxt, tn)) return kInf;
  int f = 0;
  if (!hit_boxprim(B.box, r, r.maxt, t, f)) return kInf;
  face = f;
  return t;
}

// ray_aabb with the direction's reciprocals at hand.
__device__ inline bool box_slab(V3 o, V3 inv3, const float lo[3], const float hi[3], float &t0, float &t1) {
  t0 = -kInf;
  t1 = kInf;
  const float oo[3] = {o.x, o.y, o.z};
  const float id[3] = {inv3.x, inv3.y, inv3.z};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float inv = id[k];
    float ta = (lo[k] - oo[k]) * inv;
    float tb = (hi[k] - oo[k]) * inv;
    if (ta > tb) {
      const float tmp = ta;
      ta = tb;
      tb = tmp;
    }
    t0 = ta > t0 ? ta : t0;
    t1 = tb < t1 ? tb : t1;
  }
  return t0 <= t1;
}

// grid_footprint (rows and their length below 2^24, Scene::box_path); x0: the
// footprint's first column.
__device__ inline void box_footprint(const BoxScene &B, V3 p, GridFoot &g, int &x0) {
  const ParamBind &P = B.sigma;
  const MediumInfo &M = B.med;
  float lx = p.x - M.lo[0], ly = p.y - M.lo[1], lz = p.z - M.lo[2];
  if (!B.unit_extent) {
    lx = lx / (M.hi[0] - M.lo[0]);
    ly = ly / (M.hi[1] - M.lo[1]);
    lz = lz / (M.hi[2] - M.lo[2]);
  }
  const float x = voxel_coord(lx, P.nx), y = voxel_coord(ly, P.ny), z = voxel_coord(lz, P.nz);
  const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
  g.tx = x - fx;
  g.ty = y - fy;
  g.tz = z - fz;
  const int ix = int(fx), iy = int(fy), iz = int(fz);
  x0 = min(max(ix, 0), P.nx - 1);
  const int y0 = min(max(iy, 0), P.ny - 1);
  const int z0 = min(max(iz, 0), P.nz - 1);
  g.base = int(__umul24(__umul24(unsigned(z0), unsigned(P.ny)) + unsigned(y0), unsigned(P.nx))) + x0;
  // the second corner of an axis is the next voxel, or the same one where
  // both are clamped to an end
  g.dx = unsigned(ix) < unsigned(P.nx - 1) ? 1 : 0;
  g.dy = unsigned(iy) < unsigned(P.ny - 1) ? P.nx : 0;
  g.dz = unsigned(iz) < unsigned(P.nz - 1) ? P.nx * P.ny : 0;
}

struct __attribute__((packed, aligned(4))) FloatPair {
  float a, b;
};

// grid_eval1 with the x neighbours of a row read by one 8-byte load (rows of
// at least two voxels): the pair starts at column min(x0, nx - 2), and the
// two corners are picked out of it (both its second value, or both its
// first, where the footprint is clamped). Byte offsets stay below 2^32
// (BoxScene's grids hold fewer than 2^29 voxels).
__device__ inline float box_eval1(const float *data, const GridFoot &g, int x0, int nx) {
  const int xb = min(x0, nx - 2);
  const bool hi0 = x0 > xb, hi1 = x0 + g.dx > xb;
  const unsigned b0 = unsigned(g.base - (x0 - xb)) * 4u;
  const unsigned oy = unsigned(g.dy) * 4u, oz = unsigned(g.dz) * 4u;
  const char *const q = reinterpret_cast<const char *>(data);
  const FloatPair p00 = *reinterpret_cast<const FloatPair *>(q + b0);
  const FloatPair p10 = *reinterpret_cast<const FloatPair *>(q + (b0 + oy));
  const FloatPair p01 = *reinterpret_cast<const FloatPair *>(q + (b0 + oz));
  const FloatPair p11 = *reinterpret_cast<const FloatPair *>(q + (b0 + oz + oy));
  const float c000 = hi0 ? p00.b : p00.a, c100 = hi1 ? p00.b : p00.a;
  const float c010 = hi0 ? p10.b : p10.a, c110 = hi1 ? p10.b : p10.a;
  const float c001 = hi0 ? p01.b : p01.a, c101 = hi1 ? p01.b : p01.a;
  const float c011 = hi0 ? p11.b : p11.a, c111 = hi1 ? p11.b : p11.a;
  const float x00 = c000 + (c100 - c000) * g.tx, x10 = c010 + (c110 - c010) * g.tx;
  const float x01 = c001 + (c101 - c001) * g.tx, x11 = c011 + (c111 - c011) * g.tx;
  const float y0v = x00 + (x10 - x00) * g.ty, y1v = x01 + (x11 - x01) * g.ty;
  return y0v + (y1v - y0v) * g.tz;
}


// sigma_n = majorant - sigma_t of a rounded sigma_t: exactly 0 where sigma_t
// is the majorant, as a shadow ray that ends there requires (a fused
// majorant - scale x density would leave the product's rounding error).
__device__ inline float sigma_null(float maj, float st) {
#pragma clang fp contract(off)
  return maj - st;
}

// The majorant of one global majorant's free flights: the NEW state's, or
// the larger of both states', times the scale. Wave-uniform.
template <int NS>
__device__ inline float box_majorant(const BoxScene &B, const float *majorants) {
  const uint32_t *k = reinterpret_cast<const uint32_t *>(majorants) + 2 * B.med.sigma_param;
  float m = key_to_float(__builtin_amdgcn_readfirstlane(k[RCV_STATE_NEW]));
  if (NS == 2) m = fmaxf(m, key_to_float(__builtin_amdgcn_readfirstlane(k[RCV_STATE_OLD])));
  return m * B.med.scale;
}

// One lane of the tracker: the state of one camera sample (MODE kBoxRender:
// NS states; kBoxAdjoint, kBoxForward: primal pass, then the replay pass
// with the same random numbers, which scatters into G or gathers the
// tangents in G).
template <int NS, int MODE, int F>
struct BoxPath {
  static_assert(NS == 1 || MODE == kBoxRender, "the adjoint and forward mode trace one state");
  static constexpr bool kAdj = MODE == kBoxAdjoint;
  static constexpr bool kFwd = MODE == kBoxForward;
  static constexpr bool kReplays = kAdj || kFwd;
  LazyPcg rng;
  V3 o, d, inv;   // current segment (path or shadow ray); inv = 1 / d
  V3 exit;        // the medium's far plane per axis along d
  float si_t;     // distance to the next boundary crossing
  float dist, total;  // shadow ray: distance of the emitter sample, distance tracked
  float T[NS];    // shadow ray: transmittances; at a real collision: sigma_t
  V3 thr[NS], L[NS];
  int mode, depth;
  bool inside;    // the segment began strictly inside the medium's bounds
  // adjoint and forward mode
  V3 dL, Lrem, dI;
  float cs, tsum;
  int nee_k;
  bool replay, retrack;

  __device__ static int &word(int *lds, int j) { return lds[j * int(blockDim.x)]; }
  __device__ static V3 words3(int *lds, int j) {
    return v3(__int_as_float(word(lds, j)), __int_as_float(word(lds, j + 1)), __int_as_float(word(lds, j + 2)));
  }
  __device__ static void put3(int *lds, int j, V3 v) {
    word(lds, j) = __float_as_int(v.x);
    word(lds, j + 1) = __float_as_int(v.y);
    word(lds, j + 2) = __float_as_int(v.z);
  }

  __device__ void reciprocals() { inv = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z); }
  __device__ float remaining() const { return dist * (1.0f - kShadowEps) - total; }

  // The next boundary crossing of the current segment within maxt; its point
  // and face go to LDS for the event that uses them.
  __device__ int find_boundary(const BoxScene &B, int *lds, float maxt) {
    Ray r;
    r.o = o;
    r.d = d;
    r.maxt = maxt;
    int face;
    si_t = box_trace(B, r, inv, face);
    put3(lds, 6, ray_at(r, si_t));
    word(lds, 9) = face;
    return face;
  }

  // A segment inside the medium is set (o, d): what its tracking steps need.
  __device__ void begin_segment(const BoxScene &B, int *lds) {
    reciprocals();
    const MediumInfo &M = B.med;
    exit = v3(inv.x >= 0.0f ? M.hi[0] : M.lo[0], inv.y >= 0.0f ? M.hi[1] : M.lo[1], inv.z >= 0.0f ? M.hi[2] : M.lo[2]);
    inside = o.x > M.lo[0] && o.x < M.hi[0] && o.y > M.lo[1] && o.y < M.hi[1] && o.z > M.lo[2] && o.z < M.hi[2];
    find_boundary(B, lds, mode == kOnShadow ? remaining() : kInf);
  }

  // Crosses the null boundary at the stored crossing (spawn_ray); true when
  // the segment goes on inside the medium.
  __device__ bool cross_boundary(const BoxScene &B, int *lds, int face) {
    const V3 n = v3(B.box.n[3 * face], B.box.n[3 * face + 1], B.box.n[3 * face + 2]);
    o = offset_point(words3(lds, 6), n, d);
    return !(dot(n, d) > 0.0f);
  }

  // A camera sample: its random numbers from the one after the colour
  // channel of free-flight sampling on (:171-173).
  __device__ void begin(const Pcg32 &r, const Ray &camera, bool is_replay, V3 Lp) {
    rng.begin_skip(r);
    o = camera.o;
    d = camera.d;
    reciprocals();
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      L[k] = v3(0.f);
      thr[k] = v3(1.f);
    }
    depth = 0;
    mode = kOutside;
    if constexpr (kReplays) {
      replay = is_replay;
      retrack = false;
      Lrem = Lp;
      nee_k = 0;
      if constexpr (kFwd) dI = v3(0.f);
    }
  }

  __device__ bool any_throughput() const {
    bool nonzero = false;
#pragma unroll
    for (int k = 0; k < NS; ++k) nonzero = nonzero || any_nonzero(thr[k]);
    return nonzero;
  }

  // Russian roulette of a bounce at depth > rr_depth (:182-188); false when
  // the path ends. (At lower depths its random number is skipped.)
  __device__ bool roulette() {
    const float urr = rng.next();
    const V3 tm = NS == 2 ? vmax(thr[NS - 1], thr[0]) : thr[0];
    const float q = fminf(hmax(tm), 0.99f);
    if (!(urr < q)) return false;
    const float rq = 1.0f / q;
#pragma unroll
    for (int k = 0; k < NS; ++k) thr[k] = thr[k] * rq;
    return true;
  }

  // The environment reached by a path (:284-308).
  __device__ void gather_env(const BoxScene &B, const IntegArgs &I) {
    if (depth == 0 && I.hide_emitters) return;
    const V3 emitted = v3(B.env[0], B.env[1], B.env[2]);
    const float mis = mis_weight(kInv4Pi, kInv4Pi);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const V3 c = depth == 0 ? thr[k] * emitted : thr[k] * mis * emitted;
      L[k] += c;
      if (kReplays && replay) Lrem -= c;
    }
  }

  // A path outside the box: one bounce that ends at the environment, or
  // crosses the boundary.
  __device__ void outside(const BoxScene &B, const IntegArgs &I, int *lds) {
    if (!any_throughput()) {
      mode = kPathEnd;
      return;
    }
    if (depth > I.rr_depth) {
      if (!roulette()) {
        mode = kPathEnd;
        return;
      }
    } else {
      rng.skip();
    }
    const int face = find_boundary(B, lds, kInf);
    if (face < 0) {
      gather_env(B, I);
      mode = kPathEnd;
      return;
    }
    cross_path(B, lds, face);
  }

  // (three BSDF random numbers, :347-380)
  __device__ void cross_path(const BoxScene &B, int *lds, int face) {
    rng.skip();
    rng.skip2();
    mode = cross_boundary(B, lds, face) ? kOnPath : kOutside;
  }

  // One tracking step of the path or of the shadow ray.
  __device__ void step(const SceneView &S, const BoxScene &B, const IntegArgs &I, int max_depth,
                       const UniformDiv &by_maj, const GradTargets &G, const LdsStack &log) {
    const bool shadow = mode == kOnShadow;
    float maxt_ray = kInf, u;
    if (shadow) {
      maxt_ray = remaining();
      if (!(maxt_ray > 0.0f)) {
        mode = kNeeDone;
        return;
      }
      u = rng.next();
    } else {
      if (!any_throughput()) {
        mode = kPathEnd;
        return;
      }
      if (depth > I.rr_depth) {
        if (!roulette()) {
          mode = kPathEnd;
          return;
        }
        u = rng.next();
      } else {
        u = rng.skip_next();
      }
    }
    const MediumInfo &M = B.med;
    // ---- free flight (sample_medium). From a point strictly inside the
    // medium's bounds the interval is [0, the nearest far plane]; a point on
    // the segment stays past its near planes, so only the far ones are
    // looked at again.
    float mint = 0.0f;
    float maxt = fminf(fminf((exit.x - o.x) * inv.x, (exit.y - o.y) * inv.y), (exit.z - o.z) * inv.z);
    bool ok = inside && maxt > 0.0f;
    if (!ok) {
      float t0;
      ok = box_slab(o, inv, M.lo, M.hi, t0, maxt);
      ok = ok && (t0 < kInf || maxt < kInf);
      mint = ok ? fmaxf(0.0f, t0) : 0.0f;
    }
    maxt = ok ? fminf(maxt_ray, maxt) : kInf;
    const float tau = tau_of(u);
    float maj, t;
    if constexpr ((F & kFeatSupergrid) != 0) {
      maj = 0.0f;
      t = kInf;
      Ray r;
      r.o = o;
      r.d = d;
      r.maxt = maxt_ray;
      if (ok) t = supergrid_free_flight<NS>(S, M, r, mint, maxt, tau, maj);
    } else {
      maj = by_maj.y;
      t = mint + by_maj(tau);
    }
    ok = ok && maj > 0.0f && maj < kInf;
    const bool hit = ok && t <= maxt && !(si_t < t);
    if (!hit) {
      mode = shadow ? kShadowExit : kPathExit;
      return;
    }
    // ---- collision: sigma_t and sigma_n of the states
    Ray r;
    r.o = o;
    r.d = d;
    const V3 p = ray_at(r, t);
    GridFoot foot;
    int x0;
    float st[NS], sn[NS];
    box_footprint(B, p, foot, x0);
#pragma unroll
    for (int k = 0; k < NS; ++k)
      st[k] = M.scale * box_eval1(B.sigma.data[state_index<NS>(k)], foot, x0, B.sigma.nx);
#pragma unroll
    for (int k = 0; k < NS; ++k) sn[k] = sigma_null(maj, st[k]);
    auto over_maj = [&](float x) {
      if constexpr ((F & kFeatSupergrid) != 0)
        return x / maj;
      else
        return by_maj(x);
    };
    o = p;
    si_t = si_t - t;
    float coef = 0.0f;     // replay: d log(weight)/d(density) times its radiance
    bool add = false;
    if (shadow) {
      bool any_t = false;
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        T[k] *= over_maj(sn[k]);
        any_t = any_t || T[k] != 0.0f;
      }
      if (any_t)
        total += t;
      else
        mode = kNeeDone;
      if constexpr (kReplays) {
        if (replay && sn[0] != 0.0f) {
          add = !kAdj || cs != 0.0f;
          coef = kAdj ? -cs * M.scale / sn[0] : -M.scale / sn[0];
        }
      }
    } else {
      float pr;
      if (NS == 2)
        pr = (over_maj(st[NS - 1]) + over_maj(st[0])) * 0.5f;
      else
        pr = over_maj(st[0]);
      const float un = rng.next();
      const bool null = un >= pr;
      bool alive = true;
      if (null) {
        if (NS == 2) {
          const float den = sn[NS - 1] + sn[0];
          const float w1 = 2.0f * sn[NS - 1] / den, w0 = 2.0f * sn[0] / den;
          thr[NS - 1] *= w1;
          thr[0] *= w0;
        }
      } else {
        depth += 1;
        alive = depth < max_depth;
        mode = alive ? kScatter : kPathEnd;
#pragma unroll
        for (int k = 0; k < NS; ++k) T[k] = st[k];
      }
      if constexpr (kReplays) {
        if (replay && alive && !(null && sn[0] == 0.0f)) {
          add = true;
          if constexpr (kAdj) {
            const float lr = dot(dL, Lrem);
            coef = (null ? -lr * M.scale : lr * M.scale) / (null ? sn[0] : st[0]);
            add = lr != 0.0f;
          } else {
            coef = (null ? -M.scale : M.scale) / (null ? sn[0] : st[0]);
          }
        }
      }
    }
    if constexpr (kAdj) {
      float *const g = G.g[M.sigma_param];
      if (add && g) scatter_density(&G, log, M.sigma_param, g, foot, p, coef);
    } else if constexpr (kFwd) {
      const float *const tg = G.g[M.sigma_param];
      if (add && tg) {
        const float tv = coef * box_eval1(tg, foot, x0, B.sigma.nx);
        if (shadow)
          tsum += tv;
        else
          dI += Lrem * tv;
      }
    }
  }

  // Emitter sample of a NEE at the path's point o (in the medium) and the
  // shadow ray towards it (shadow_begin, sample_emitter_direction of a
  // constant environment).
  __device__ void begin_shadow(const BoxScene &B) {
    const float u1 = rng.next();
    const float u2 = rng.next();
    const V3 c = v3(B.bs_center[0], B.bs_center[1], B.bs_center[2]);
    const float radius = fmaxf(B.bs_radius, norm(o - c));
    dist = 2.0f * radius;
    total = 0.0f;
    d = square_to_uniform_sphere(u1, u2);
#pragma unroll
    for (int k = 0; k < NS; ++k) T[k] = 1.0f;
    mode = kOnShadow;
  }

  // Real collision at o with sigma_t in T (:253-281): albedo weights, phase
  // sample, NEE.
  __device__ void scatter(const BoxScene &B, int *lds, const GradTargets &G) {
    const MediumInfo &M = B.med;
    GridFoot fa;
    V3 alb_new = v3(0.f);
    V3 ss[NS];
    if constexpr ((F & kFeatAlbedoGrid) != 0) grid_footprint(B.albedo, M, o, fa);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      V3 alb;
      if constexpr ((F & kFeatAlbedoGrid) != 0)
        alb = grid_eval3(B.albedo.data[state_index<NS>(k)], fa);
      else
        alb = v3(M.albedo[0], M.albedo[1], M.albedo[2]);
      if (k == NS - 1) alb_new = alb;
      ss[k] = alb * T[k];
    }
    if (NS == 2) {
      const float den = T[NS - 1] + T[0];
      const V3 w1 = 2.0f * ss[NS - 1] / den, w0 = 2.0f * ss[0] / den;
      thr[NS - 1] *= w1;
      thr[0] *= w0;
    } else {
      thr[0] *= ss[0] / T[0];
    }
    if constexpr (kReplays && (F & kFeatAlbedoGrid) != 0) {
      float *const ga = G.g[M.albedo_param];
      if (replay && ga) {
        if constexpr (kAdj) {
          const V3 dl = dL * Lrem;
          scatter_grid3(ga, fa, v3(alb_new.x != 0.f ? dl.x / alb_new.x : 0.f, alb_new.y != 0.f ? dl.y / alb_new.y : 0.f,
                                   alb_new.z != 0.f ? dl.z / alb_new.z : 0.f));
        } else {
          const V3 ta = grid_eval3(ga, fa);
          dI += Lrem * v3(alb_new.x != 0.f ? ta.x / alb_new.x : 0.f, alb_new.y != 0.f ? ta.y / alb_new.y : 0.f,
                          alb_new.z != 0.f ? ta.z / alb_new.z : 0.f);
        }
      }
    }
    const float a = rng.skip_next();
    const float b = rng.next();
    put3(lds, 0, o);
    put3(lds, 3, square_to_uniform_sphere(a, b));
    if constexpr (kAdj) {
      cs = 0.0f;
      if (replay) {
        if (nee_k < kBoxSlots) {
          cs = __int_as_float(word(lds, kBoxSlot0 + nee_k));
        } else {
          word(lds, 10) = int(unsigned(rng.state));
          word(lds, 11) = int(unsigned(rng.state >> 32));
        }
      }
    } else if constexpr (kFwd) {
      tsum = 0.0f;
    }
    begin_shadow(B);
  }

  // The shadow ray at the box boundary: a null surface, crossed.
  __device__ void shadow_exit(const BoxScene &B, int *lds) {
    int face = word(lds, 9);
    mode = kNeeDone;
    while (face >= 0) {
      const bool in = cross_boundary(B, lds, face);
      total += si_t;
      const float rem = remaining();
      if (!(rem > 0.0f)) return;
      if (in) {
        mode = kOnShadow;
        return;
      }
      face = find_boundary(B, lds, rem);
    }
  }

  // The NEE's contribution (nee_account), then back to the path.
  __device__ void nee_done(const BoxScene &B, int *lds) {
    mode = kOnPath;
    o = words3(lds, 0);
    if constexpr (kAdj) {
      if (retrack) {
        retrack = false;
        rng.state = (uint64_t(unsigned(word(lds, 13))) << 32) | uint64_t(unsigned(word(lds, 12)));
        d = words3(lds, 3);
        return;
      }
    }
    const V3 ev = v3(B.env[0], B.env[1], B.env[2]) * (4.0f * kPi * 1.0f);
    const float mis_em = mis_weight(kInv4Pi, kInv4Pi);
    const V3 nw = v3(kInv4Pi);
    V3 c0 = v3(0.f);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const V3 em = ev * T[k];
      const V3 c = thr[k] * nw * mis_em * em;
      L[k] += c;
      if (k == 0) c0 = c;
    }
    if constexpr (kFwd) {
      if (replay && any_nonzero(c0)) dI += c0 * tsum;
    }
    if constexpr (kReplays) {
      if (replay) Lrem -= c0;
    }
    if constexpr (kAdj) {
      const int k = nee_k++;
      const float w = dot(dL, c0);
      if (!replay) {
        if (k < kBoxSlots) word(lds, kBoxSlot0 + k) = __float_as_int(w);
      } else if (k >= kBoxSlots && w != 0.0f && any_nonzero(c0)) {
        // past the slots: track the shadow ray again, now with its weight
        word(lds, 12) = int(unsigned(rng.state));
        word(lds, 13) = int(unsigned(rng.state >> 32));
        rng.state = (uint64_t(unsigned(word(lds, 11))) << 32) | uint64_t(unsigned(word(lds, 10)));
        cs = w;
        retrack = true;
        begin_shadow(B);
        return;
      }
    }
    d = words3(lds, 3);
  }

  // The path at the box boundary: crossed, and on to the environment. (No
  // boundary ahead -- the path's point lies outside by rounding: the
  // environment at once.)
  __device__ void path_exit(const BoxScene &B, const IntegArgs &I, int *lds) {
    const int face = word(lds, 9);
    if (face < 0) {
      gather_env(B, I);
      mode = kPathEnd;
      return;
    }
    cross_path(B, lds, face);
    if (mode == kOutside) outside(B, I, lds);
  }

  __device__ bool tracking() const { return mode <= kOnShadow; }
};

// Whether the wavefront runs its events now: twice as many of its lanes wait
// at one as can track. An event section costs about three tracking steps
// whichever lanes are at an event, so it pays to let lanes gather; the 64^3
// step with a ratio of 1/2, 1, 2, 3 and 6: 25.6, 18.4, 18.2, 18.2 and 18.4
// ms, a 64^2 launch of 4 samples per pixel, which waits for its longest path,
// 1.27, 1.19, 1.23, 1.28 and 1.35 ms.
__device__ inline bool box_events_due(bool tracking, bool idle, bool &done) {
  const int run = __popcll(__ballot(tracking));
  const int wait = __popcll(__ballot(!tracking && !idle));
  done = run + wait == 0;
  return wait > 0 && wait >= 2 * run;
}

// Units a wavefront draws from the device counter at once, for its lanes to
// take one by one (fewer towards the end of a launch). Every draw is an
// atomic on one address that all XCDs share, ~20 ns each: one draw per
// request of its lanes took as long as the tracking itself (128^3 render,
// 64 samples per pixel: 5.8 ms against 4.3 ms; 256 units at once: 4.4 ms).
constexpr unsigned kBoxGrab = 64;

// The work units of a wavefront: drawn from the launch's counter in grabs.
struct UnitPool {
  unsigned *queue;
  unsigned total, waves, next, end;

  // n units that about `w` wavefronts share
  __device__ UnitPool(unsigned *q, unsigned n, unsigned w) : queue(q), total(n), waves(w), next(0), end(0) {}

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
      const unsigned grab = max(want - have, min(kBoxGrab, left / (waves * 4u)));
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

// The NS sums of work unit u to the unit-sum buffer.
template <int NS>
__device__ inline void store_unit(float *partial, unsigned u, const V3 (&acc)[NS]) {
  float *o = partial + int64_t(u) * (3 * NS);
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    o[3 * k] = acc[k].x;
    o[3 * k + 1] = acc[k].y;
    o[3 * k + 2] = acc[k].z;
  }
}

// Runs the units a wavefront draws from `units` until none is left for any of
// its lanes (all 64 lanes call it). Render: store(unit, sums) takes a unit's
// NS radiance sums; adjoint: into G, through the scatter log where it is set;
// forward mode: store takes a unit's derivative sum, the tangents in G.
template <int NS, int MODE, int F, class Store>
__device__ inline void box_run(const SceneView &S, const BoxScene &B, const IntegArgs &I, const SensorInfo &sen,
                               uint32_t seed, int spp, int chunk_log2, const float *grad_img, const GradTargets &G,
                               UnitPool &units, int *lds, const LdsStack &log, Store &&store) {
  const int film_w = sen.film_w;
  const int max_depth = I.max_depth < 0 ? 0x7fffffff : I.max_depth;
  const UniformDiv by_maj((F & kFeatSupergrid) ? 1.0f : box_majorant<NS>(B, S.majorants));
  BoxPath<NS, MODE, F> t;
  t.mode = kPathEnd;
  bool open = false;  // a sample of this lane's unit is under way
  int s = 0, s_end = 0, px = 0, py = 0;
  unsigned u = 0;
  V3 acc[NS];
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
            store(u, acc);
          }
        }
        need = !replay && s >= s_end;
      }
      const unsigned taken = units.take(need);
      if (t.mode == kPathEnd) {
        open = true;
        if (need) {
          u = taken;
          if (u >= units.total) {
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
}

}  // namespace rcv
