// ncx_toi.hip -- batched linear time of impact and batched shape ray casts on the GPU.
//
// query::time_of_impact (src/query/time_of_impact/time_of_impact.rs:66-158) for Ball, Cuboid,
// Capsule and ConvexHull under translational motion: the Ball-Ball closed form
// (time_of_impact_ball_ball.rs:7-61) and, for every other pair, GJK's ray cast on the Minkowski
// difference (gjk::directional_distance, src/query/algorithms/gjk.rs:214-365) as
// time_of_impact_support_map_support_map does (time_of_impact_support_map_support_map.rs:10-116).
// RayCast::toi_and_normal_with_ray of the same four shapes (ray_ball.rs, ray_cuboid.rs,
// ray_aabb.rs, ray_support_map.rs) over a batch of (shape, ray) pairs.
//
// What bounds both: GJK's ray cast is a serial chain of iterations (a support point, a simplex
// reduction, square roots and divisions; about 570 vector instructions, 1.8 us), 6 to 15 of them on
// average by shape types, and in a few casts hundreds, up to the cap of 10000.  So the step has few
// branches (rc_step); the casts of one launch have alike shapes next to each other (pairs in
// partition order, rays in lists by shape kind), because a support function of another shape is
// another path; and everything runs in one launch, because its longest cast decides how long it
// takes.  262,144 mixed pairs 2.6 -> 1.14 ms, a million rays 2.6 -> 1.6 ms (their longest casts take
// 1,000 iterations; batches with a cast that runs to the cap 21.7 -> 19.7 ms).  All arithmetic
// restates the reference in f32 with its operation order.
#include "ncx_gjk.h"

#define TOI_BS 128

struct TOIOut {
  int has;
  float toi;
  f3 w1, w2, n1, n2;
  int status;  // 0 OutOfIterations, 1 Converged, 2 Failed, 3 Penetrating (time_of_impact.rs:7-25)
};

__device__ __forceinline__ void toi_none(TOIOut& o) {
  o.has = 0;
  o.toi = 0.f;
  o.status = 0;
  o.w1 = o.w2 = o.n1 = o.n2 = f3{0.f, 0.f, 0.f};
}

// time_of_impact_ball_ball (time_of_impact_ball_ball.rs:7-61), then the frame change of
// query::time_of_impact (time_of_impact.rs:75-98)
__device__ __forceinline__ void toi_ball_ball(TOIOut& o, const iso& m1, f3 v1, float r1, const iso& m2, f3 v2, float r2,
                                              float max_toi, float target) {
  const f3 vel = v1 - v2;
  const float rsum = r1 + r2;
  const float radius = rsum + target;
  const f3 center = m1.t + (-m2.t);
  const f3 ro = f3{0.f, 0.f, 0.f}, rd = -vel;
  bool inside;
  float t;
  if (!ray_toi_with_ball(center, radius, ro, rd, true, inside, t)) return;
  if (t > max_toi) return;
  const f3 dpt = (ro + rd * t) - center;
  f3 n1, n2, w1, w2;
  if (radius == 0.f) {
    n1 = f3{1.f, 0.f, 0.f}; n2 = n1; w1 = f3{0.f, 0.f, 0.f}; w2 = w1;
  } else {
    n1 = dpt / radius;
    n2 = -n1;
    w1 = n1 * r1;
    w2 = n2 * r2;
  }
  o.has = 1;
  o.toi = t;
  o.status = (inside && norm_sq(center) < rsum * rsum) ? 3 : 1;
  o.w1 = qrot_inv(m1.q, w1);
  o.w2 = qrot_inv(m2.q, w2);
  o.n1 = qrot_inv(m1.q, n1);
  o.n2 = qrot_inv(m2.q, n2);
}

// time_of_impact_support_map_support_map (time_of_impact_support_map_support_map.rs:10-116) after
// its ray cast hit.  DIL: a target distance is set (c is dilated by it).
template <int G, bool DIL>
__device__ __forceinline__ void toi_finish(TOIOut& o, const RCtx& c, const RCState& r, float max_toi, float target,
                                           const Pool& P, int gl) {
  const float t = r.ltoi / r.ray_length;
  const f3 normal = r.ldir;
  f3 w1 = f3{0.f, 0.f, 0.f}, w2 = w1;
  if (t != 0.f) gjk_result(r.s, r.s.dim == 3, w1, w2);  // gjk.rs:228-237
  if (t > max_toi) return;
  o.has = 1;
  o.toi = t;
  o.w2 = inv_xform_pt(c.m2, w2);
  o.n1 = inv_xform_vec(c.m1, normal);
  o.n2 = inv_xform_vec(c.m2, -normal);
  o.w1 = inv_xform_pt(c.m1, w1);
  if (!DIL) {
    o.status = t == 0.f ? 3 : 1;
    return;
  }
  o.status = 1;
  if (t == 0.f) {
    // closest_points_support_map_support_map_with_params(.., target_distance, Some(normal))
    // (src/query/closest_points/closest_points_support_map_support_map.rs:40-67)
    Ctx2 c2;
    c2.m1 = c.m1; c2.m2 = c.m2; c2.g1 = c.g1; c2.g2 = c.g2;
    f3 d;
    float nl;
    if (!try_normalize(normal, NCX_FLT_EPS, &d, &nl)) d = f3{1.f, 0.f, 0.f};
    Simplex s2;
    const GJKOut g = gjk<G>(c2, d, target, s2, P, gl, 10000);
    if (g.status == GJK_S_CLOSEST) {
      const f3 nn = normalize(g.p2 - g.p1);
      o.n1 = inv_xform_vec(c.m1, nn);
      o.n2 = inv_xform_vec(c.m2, -nn);
      return;
    } else if (g.status == GJK_S_INTERSECTION) {
      o.status = 3;
    }
  }
  o.w1 = o.w1 - o.n1 * target;
}

struct TOIArgs {
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  const float* vel;
  const uint32_t* ia;
  const uint32_t* ib;
  size_t n;
  uint32_t nshapes;
  float max_toi, target;
  uint8_t* has;
  float* toi;
  float* w1;
  float* w2;
  float* n1;
  float* n2;
  uint8_t* status;
  uint32_t* err;
  const uint32_t* list;                // optional: the pairs' order
  uint32_t* work;                      // pair counter (zero at launch)
};

__device__ __forceinline__ void store3(float* p, size_t k, f3 v) {
  p[3 * k] = v.x;
  p[3 * k + 1] = v.y;
  p[3 * k + 2] = v.z;
}

// Times of impact, one group of G lanes per pair, 64 / G pairs of a wavefront at a time.  (Groups
// that take a new pair as soon as theirs has ended are slower, 1.4 against 1.14 ms: their casts'
// simplices then differ in dimension, and every dimension's reduction is another path.)
template <int G, bool DIL>
__global__ __launch_bounds__(TOI_BS, 2) void k_toi(TOIArgs a) {
  __shared__ float snaps[TOI_BS / G][RC_SNAP];
  const int lane = threadIdx.x & 63, gl = lane & (G - 1);
  float* const snap = snaps[threadIdx.x / G];
  for (;;) {
    uint32_t q = 0;
    if (lane == 0) q = atomicAdd(a.work, 64u / G);
    q = (uint32_t)__builtin_amdgcn_readfirstlane((int)q) + (uint32_t)lane / G;
    if (__ballot(q < a.n) == 0) break;
    if (q >= a.n) continue;
    const size_t k = a.list ? a.list[q] : q;
    const uint32_t i = a.ia[k], j = a.ib[k];
    TOIOut o;
    toi_none(o);
    if (i >= a.nshapes || j >= a.nshapes) {
      if (gl == 0) atomicOr(a.err, 1u);
    } else {
      RCtx c;
      c.m1 = load_pose(a.poses, i);
      c.m2 = load_pose(a.poses, j);
      c.g1 = load_shape(a.shapes, i);
      c.g2 = load_shape(a.shapes, j);
      c.dil = a.target;
      c.dilated = DIL;
      c.local = false;
      const f3 v1 = f3{a.vel[3 * i], a.vel[3 * i + 1], a.vel[3 * i + 2]};
      const f3 v2 = f3{a.vel[3 * j], a.vel[3 * j + 1], a.vel[3 * j + 2]};
      if (c.g1.type == NCX_BALL && c.g2.type == NCX_BALL) {
        toi_ball_ball(o, c.m1, v1, c.g1.a, c.m2, v2, c.g2.a, a.max_toi, a.target);
      } else {
        RCState r;
        float t;
        f3 n;
        if (minkowski_ray_cast<G>(c, f3{0.f, 0.f, 0.f}, v2 - v1, NCX_FLT_MAX, r, a.P, gl, snap, t, n))
          toi_finish<G, DIL>(o, c, r, a.max_toi, a.target, a.P, gl);
      }
    }
    if (gl == 0) {
      a.has[k] = (uint8_t)o.has;
      a.toi[k] = o.toi;
      store3(a.w1, k, o.w1);
      store3(a.w2, k, o.w2);
      store3(a.n1, k, o.n1);
      store3(a.n2, k, o.n2);
      a.status[k] = (uint8_t)o.status;
    }
  }
}

struct SRArgs {
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  const uint32_t* idx;
  const float *ox, *oy, *oz, *dx, *dy, *dz;
  size_t n;
  uint32_t nshapes;
  float max_toi;
  int solid;
  float* toi;
  float* nrm;
  uint32_t* feat;
  uint32_t* err;
  uint32_t* list;   // rays on hulls from the front, on capsules from the back (n entries)
  uint32_t* count;  // their numbers (hulls, capsules), SR_STRIDE words apart
  uint32_t* work;   // and work counters
};
#define SR_STRIDE 64

// Rays against balls and cuboids (closed forms), one lane per ray; the rays on support-map shapes
// are listed by kind, with one atomic per kind and block (one per wavefront took 0.2 ms for a
// million rays: atomics on one address come one after another).
#define SR_BLOCK 1024
__global__ __launch_bounds__(SR_BLOCK) void k_shape_rays(SRArgs a) {
  __shared__ uint32_t cnt[2], base[2];
  if (threadIdx.x < 2) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const size_t k = (size_t)blockIdx.x * SR_BLOCK + threadIdx.x;
  int cls = 0;  // 0: done by this lane; 1: ConvexHull; 2: Capsule
  if (k < a.n) {
    const uint32_t i = a.idx[k];
    float t = -1.f;
    f3 nn = f3{0.f, 0.f, 0.f};
    uint32_t f = 0xFFFFFFFFu;
    if (i >= a.nshapes) {
      atomicOr(a.err, 1u);
    } else {
      const ShapeD g = load_shape(a.shapes, i);
      if (g.type == NCX_CONVEX_HULL) cls = 1;
      else if (g.type == NCX_CAPSULE) cls = 2;
      else {
        float tt;
        f3 n;
        uint32_t ff;
        if (shape_ray_cast_closed(g, load_pose(a.poses, i), f3{a.ox[k], a.oy[k], a.oz[k]},
                                  f3{a.dx[k], a.dy[k], a.dz[k]}, a.max_toi, a.solid != 0, tt, n, ff)) {
          t = tt;
          nn = n;
          f = ff;
        }
      }
    }
    if (cls == 0) {
      a.toi[k] = t;
      store3(a.nrm, k, nn);
      a.feat[k] = f;
    }
  }
  uint32_t e = 0;  // this ray's place among the block's of its kind
  for (int kind = 1; kind <= 2; ++kind) {
    const uint64_t m = __ballot(cls == kind);
    if (!m) continue;
    uint32_t t = 0;
    const int first = __builtin_ctzll(m);
    if (lane == first) t = atomicAdd(&cnt[kind - 1], (uint32_t)__popcll(m));
    t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
    if (cls == kind) e = t + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  }
  __syncthreads();
  if (threadIdx.x < 2 && cnt[threadIdx.x])
    base[threadIdx.x] = atomicAdd(a.count + threadIdx.x * SR_STRIDE, cnt[threadIdx.x]);
  __syncthreads();
  if (cls == 1) a.list[base[0] + e] = (uint32_t)k;
  if (cls == 2) a.list[a.n - 1 - (base[1] + e)] = (uint32_t)k;
}

// The next rays of a wavefront's groups that want one: each such group gets its own index, with
// one atomic for all of them.  `wm` has the group's first lane's bit.
__device__ __forceinline__ uint32_t take_next(uint32_t* work, uint64_t wm, int lane, int gbase) {
  uint32_t t = 0;
  const int first = __builtin_ctzll(wm);
  if (lane == first) t = atomicAdd(work, (uint32_t)__popcll(wm));
  t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
  return t + (uint32_t)__popcll(wm & ((1ull << gbase) - 1ull));
}

// The listed rays on shapes of type KIND, one group of G lanes per ray: the ray cast in the shape's
// frame (ray_support_map.rs:15-62, 117-163).
template <int G, int KIND, bool SOLID>
__device__ __forceinline__ void map_rays(const SRArgs& a, float (*snaps)[RC_SNAP]) {
  constexpr int kind = KIND == NCX_CONVEX_HULL ? 0 : 1;
  constexpr int REFILL = 64 / G >= 16 ? 64 / G / 8 : 1;
  const int lane = threadIdx.x & 63, gl = lane & (G - 1), gbase = lane & ~(G - 1);
  float* const snap = snaps[threadIdx.x / G];
  const uint32_t n = a.count[kind * SR_STRIDE];
  uint32_t* const work = a.work + kind * SR_STRIDE;
  bool live = false, done = false, behind = false;
  uint32_t k = 0;
  ShapeD g;
  f3 lo, ld;
  float limit = 0.f, shift = 0.f;
  RCState r;
  int st = RC_RUNNING;
  for (;;) {
    const uint64_t wm = __ballot(!live && !done && gl == 0), lm = __ballot(live);
    if ((wm | lm) == 0) break;
    if (wm && (lm == 0 || __popcll(wm) >= REFILL)) {
      const uint32_t q = take_next(work, wm, lane, gbase);
      if (!live && !done) {
        if (q >= n) {
          done = true;
        } else {
          live = true;
          behind = false;
          k = a.list[kind == 0 ? q : a.n - 1 - q];
          const uint32_t i = a.idx[k];  // a shape of the set: it was listed
          g = load_shape(a.shapes, i);
          const iso m = load_pose(a.poses, i);
          lo = inv_xform_pt(m, f3{a.ox[k], a.oy[k], a.oz[k]});
          ld = inv_xform_vec(m, f3{a.dx[k], a.dy[k], a.dz[k]});
          limit = a.max_toi;
          st = rc_begin<G, KIND>(ray_ctx(g), r, lo, ld, a.P, gl);
        }
      }
    }
    if (live) {
      const RCtx c = ray_ctx(g);
      if (st == RC_RUNNING) st = rc_step<G, KIND>(c, limit, r, a.P, gl, snap);
      if (st != RC_RUNNING) {
        float t = r.ltoi / r.ray_length;
        bool again = false;
        if (!SOLID && st == RC_HIT) {
          if (behind) {
            t = shift - t;
            if (!(t <= a.max_toi)) st = RC_MISS;
          } else if (t == 0.f) {
            f3 back;
            shift = ray_from_behind<G>(c, lo, ld, a.P, gl, back);
            limit = shift + 0.001f;
            st = rc_begin<G, KIND>(c, r, back, -ld, a.P, gl);
            behind = true;
            again = true;
          }
        }
        if (!again) {
          if (gl == 0) {
            const bool hit = st == RC_HIT;
            const f3 nn = xform_vec(load_pose(a.poses, a.idx[k]), r.ldir);
            a.toi[k] = hit ? t : -1.f;
            store3(a.nrm, k, sel3(hit, nn, f3{0.f, 0.f, 0.f}));
            a.feat[k] = hit ? NCX_FEAT_UNKNOWN : 0xFFFFFFFFu;
          }
          live = false;
        }
      }
    }
  }
}

// Both kinds in one launch, the first hblocks blocks on the hulls' rays: the last casts of one kind
// take as long as a few hundred iterations one after another, and the other's work fills the chip
// meanwhile.
template <bool SOLID>
__global__ __launch_bounds__(TOI_BS, 2) void k_map_rays(SRArgs a, uint32_t hblocks) {
  __shared__ float snaps[TOI_BS][RC_SNAP];
  if (blockIdx.x < hblocks) map_rays<2, NCX_CONVEX_HULL, SOLID>(a, snaps);
  else map_rays<1, NCX_CAPSULE, SOLID>(a, snaps);
}

static int query_err_check(ncx_ctx* ctx, const uint32_t* err_dev, const char* what) {
  uint32_t err = 0;
  NCX_HIP_CHECK(hipMemcpyAsync(&err, err_dev, 4, hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  if (err) {
    ncx_set_error(std::string(what) + ": a shape index is not a shape of the set");
    return NCX_E_INVALID;
  }
  return NCX_OK;
}

static unsigned cast_blocks(ncx_ctx* ctx, size_t n, int G) {
  return (unsigned)std::max<size_t>(1, std::min<size_t>((n * G + TOI_BS - 1) / TOI_BS, (size_t)ctx->num_cus * 4));
}

template <bool DIL> static void launch_toi(ncx_ctx* ctx, int G, const TOIArgs& a, size_t n) {
  const dim3 nb(cast_blocks(ctx, n, G)), bs(TOI_BS);
  switch (G) {
    case 1: hipLaunchKernelGGL((k_toi<1, DIL>), nb, bs, 0, ctx->stream, a); break;
    case 2: hipLaunchKernelGGL((k_toi<2, DIL>), nb, bs, 0, ctx->stream, a); break;
    default: hipLaunchKernelGGL((k_toi<4, DIL>), nb, bs, 0, ctx->stream, a); break;
  }
}

// Lanes per pair, for sets with hulls of up to 96 vertices and larger ones.
#define TOI_G 2
#define TOI_LARGE_G 4
// Queries of one launch: bounds the scratch memory (8 bytes a pair, 4 a ray).
static const size_t CAST_CHUNK = (size_t)1 << 26;

extern "C" int ncx_time_of_impact_batch(ncx_shapes* s, const ncx_pose* poses_dev, const float* vel_dev,
                                        const uint32_t* ia_dev, const uint32_t* ib_dev, size_t npairs, float max_toi,
                                        float target_distance, uint8_t* has_dev, float* toi_dev,
                                        float* witness1_dev, float* witness2_dev, float* normal1_dev,
                                        float* normal2_dev, uint8_t* status_dev) {
  NCX_REQUIRE(s && poses_dev && vel_dev && ia_dev && ib_dev && has_dev && toi_dev && witness1_dev && witness2_dev &&
                  normal1_dev && normal2_dev && status_dev,
              "ncx_time_of_impact_batch: null argument");
  NCX_REQUIRE(target_distance >= 0.f, "ncx_time_of_impact_batch: negative target distance");
  if (npairs == 0) return NCX_OK;
  ncx_ctx* ctx = s->ctx;
  int rc;
  if (npairs > CAST_CHUNK) {
    for (size_t o = 0; o < npairs; o += CAST_CHUNK)
      if ((rc = ncx_time_of_impact_batch(s, poses_dev, vel_dev, ia_dev + o, ib_dev + o, std::min(CAST_CHUNK, npairs - o),
                                         max_toi, target_distance, has_dev + o, toi_dev + o, witness1_dev + 3 * o,
                                         witness2_dev + 3 * o, normal1_dev + 3 * o, normal2_dev + 3 * o, status_dev + o)))
        return rc;
    return NCX_OK;
  }
  // the order is worth its memory, but not a refusal
  const bool partition = npairs >= NCX_PARTITION_MIN_PAIRS && contact_tiers_reserve_list(s->tiers, npairs) == NCX_OK;
  if (partition) rc = pairs_partition(s, s->tiers, ctx, poses_dev, ia_dev, ib_dev, npairs, nullptr);
  else rc = fill_u32(ctx, s->tiers.ovf.as<uint32_t>(), NCX_OVF_HEADER, 0u);
  if (rc) return rc;
  uint32_t* hdr = s->tiers.ovf.as<uint32_t>();
  TOIArgs a = {};
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>()};
  a.poses = poses_dev;
  a.vel = vel_dev;
  a.ia = ia_dev;
  a.ib = ib_dev;
  a.n = npairs;
  a.nshapes = (uint32_t)s->n;
  a.max_toi = max_toi;
  a.target = target_distance;
  a.has = has_dev;
  a.toi = toi_dev;
  a.w1 = witness1_dev;
  a.w2 = witness2_dev;
  a.n1 = normal1_dev;
  a.n2 = normal2_dev;
  a.status = status_dev;
  a.err = hdr + NCX_OVF_BAD;
  if (partition) a.list = s->tiers.blist.as<uint32_t>();
  a.work = ncx_work_set(hdr, NCX_WORK_BKT);
  // one launch for all buckets: the last casts take as long as a few hundred iterations one after
  // another, and with a launch per bucket nothing else runs meanwhile
  const int G = s->buckets == 1u ? 1 : (s->buckets & 8u ? TOI_LARGE_G : TOI_G);
  if (target_distance != 0.f) launch_toi<true>(ctx, G, a, npairs);
  else launch_toi<false>(ctx, G, a, npairs);
  NCX_HIP_CHECK(hipGetLastError());
  return query_err_check(ctx, a.err, "ncx_time_of_impact_batch");
}

extern "C" int ncx_shapes_cast_rays(ncx_shapes* s, const ncx_pose* poses_dev, const uint32_t* shape_dev,
                                    const float* const ray_soa_dev[6], size_t n, float max_toi, int solid,
                                    float* toi_dev, float* normal_dev, uint32_t* feature_dev) {
  NCX_REQUIRE(s && poses_dev && shape_dev && ray_soa_dev && toi_dev && normal_dev && feature_dev,
              "ncx_shapes_cast_rays: null argument");
  for (int d = 0; d < 6; ++d) NCX_REQUIRE(ray_soa_dev[d], "ncx_shapes_cast_rays: null ray array");
  if (n == 0) return NCX_OK;
  ncx_ctx* ctx = s->ctx;
  int rc;
  // an error flag, the two lists' lengths and work counters on lines of their own, the lists; fewer
  // rays at a time where there is no memory for all
  size_t chunk = std::min(n, CAST_CHUNK);
  while ((rc = s->qerr.reserve(4 * (5 * SR_STRIDE + chunk)))) {
    if (chunk <= 4096) return rc;
    chunk = std::max<size_t>(chunk / 2, 4096);
  }
  if (n > chunk) {
    for (size_t o = 0; o < n; o += chunk) {
      const float* soa[6];
      for (int d = 0; d < 6; ++d) soa[d] = ray_soa_dev[d] + o;
      if ((rc = ncx_shapes_cast_rays(s, poses_dev, shape_dev + o, soa, std::min(chunk, n - o), max_toi, solid,
                                     toi_dev + o, normal_dev + 3 * o, feature_dev + o)))
        return rc;
    }
    return NCX_OK;
  }
  if ((rc = fill_u32(ctx, s->qerr.as<uint32_t>(), 5 * SR_STRIDE, 0u))) return rc;
  SRArgs a;
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>()};
  a.poses = poses_dev;
  a.idx = shape_dev;
  a.ox = ray_soa_dev[0]; a.oy = ray_soa_dev[1]; a.oz = ray_soa_dev[2];
  a.dx = ray_soa_dev[3]; a.dy = ray_soa_dev[4]; a.dz = ray_soa_dev[5];
  a.n = n;
  a.nshapes = (uint32_t)s->n;
  a.max_toi = max_toi;
  a.solid = solid;
  a.toi = toi_dev;
  a.nrm = normal_dev;
  a.feat = feature_dev;
  a.err = s->qerr.as<uint32_t>();
  a.count = a.err + SR_STRIDE;
  a.work = a.err + 3 * SR_STRIDE;
  a.list = a.err + 5 * SR_STRIDE;
  hipLaunchKernelGGL(k_shape_rays, dim3(ceil_div(n, SR_BLOCK)), dim3(SR_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  const bool hulls = s->types >> NCX_CONVEX_HULL & 1u, capsules = s->types >> NCX_CAPSULE & 1u;
  const unsigned hb = hulls ? cast_blocks(ctx, n, 2) / 2 + 1 : 0, cb = capsules ? cast_blocks(ctx, n, 1) / 2 + 1 : 0;
  if (hb + cb) {
    if (solid) hipLaunchKernelGGL(k_map_rays<true>, dim3(hb + cb), dim3(TOI_BS), 0, ctx->stream, a, hb);
    else hipLaunchKernelGGL(k_map_rays<false>, dim3(hb + cb), dim3(TOI_BS), 0, ctx->stream, a, hb);
    NCX_HIP_CHECK(hipGetLastError());
  }
  return query_err_check(ctx, a.err, "ncx_shapes_cast_rays");
}
