// ncx_composite.hip -- a TriMesh (composite shape) against a batch of convex shapes on the GPU.
//
// Contact: contact_composite_shape_shape (src/query/contact/contact_composite_shape_shape.rs:9-45).
// For each query shape, the mesh triangles whose box intersects the shape's box in the mesh frame,
// loosened by the prediction, are its candidates (BoundingVolumeInterferencesCollector over the
// mesh's tree); query::contact(mesh pose, triangle, shape pose, shape, prediction) runs on every
// candidate pair in the batched, tiered contact kernels (the triangles join the shape set as
// Triangle parts); the deepest contact of each query is kept.
// Distance: distance_composite_shape_shape (src/query/distance/distance_composite_shape_shape.rs:
// 9-35): a search of the mesh's tree ordered by the distance from the origin to the Minkowski sum
// of a node's box and the shape's box (CompositeShapeAgainstAnyDistanceVisitor, :56-101), skipping
// boxes no nearer than the best distance so far; query::distance (GJK) on each triangle reached.
//
// The tree is the mesh's LBVH (its node boxes grown slightly for the ray cast, which only keeps
// more nodes); at the leaves the triangle's own box (its vertices' min and max) decides, as the
// reference's BVT leaves do.  The reference keeps the first of equally deep contacts in its tree's
// visiting order; here the least triangle id wins such an exact tie.
#include "ncx_contact.h"

#define MC_BLOCK 128
#define MC_STACK (LBVH_MAX_DEPTH + 2)

void ncx_mesh::release_composite() {
  if (comp) {
    comp->shapes.release(); comp->qerr.release();
    contact_tiers_release(comp->tiers);
    delete comp;
    comp = nullptr;
  }
  DevBuf* bufs[] = {&cposes, &ccnt, &coffs, &cscan, &ctot, &ca, &cb, &chas, &cw1, &cw2, &cn, &cdepth, &citers};
  for (DevBuf* b : bufs) b->release();
}

// Triangle k of the mesh as the shape record n + k of the combined set.
__global__ void k_mc_tri_records(ncx_shape* __restrict__ out, size_t ntri) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ntri) return;
  ncx_shape s = {};
  s.type = SHAPE_TRIANGLE;
  s.hull_offset = (uint32_t)k;
  s.pad[0] = __float_as_uint(1.f);  // bounding radius for the pair order (a heuristic only)
  out[k] = s;
}

__global__ void k_mc_fill_pose(ncx_pose* __restrict__ out, size_t n, ncx_pose p) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) out[k] = p;
}

struct MCArgs {
  const LNode* nodes;
  const float4* tris;
  uint32_t ntri;
  ncx_pose mesh_pose;
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  const uint32_t* qshape;
  uint32_t nq, nshapes;
  float prediction;
  uint32_t* count;
  const uint32_t* offs;
  uint32_t* ca;
  uint32_t* cb;
  uint32_t* err;
};

__device__ __forceinline__ void tri_box(const float4* tris, uint32_t k, f3& mn, f3& mx) {
  const float4 a = tris[3 * (size_t)k], b = tris[3 * (size_t)k + 1], c = tris[3 * (size_t)k + 2];
  mn = f3{fminf(fminf(a.x, b.x), c.x), fminf(fminf(a.y, b.y), c.y), fminf(fminf(a.z, b.z), c.z)};
  mx = f3{fmaxf(fmaxf(a.x, b.x), c.x), fmaxf(fmaxf(a.y, b.y), c.y), fmaxf(fmaxf(a.z, b.z), c.z)};
}

__device__ __forceinline__ bool box_hit(f3 amn, f3 amx, f3 bmn, f3 bmx) {  // AABB::intersects (aabb.rs:156-158)
  return amn.x <= bmx.x && amn.y <= bmx.y && amn.z <= bmx.z && amx.x >= bmn.x && amx.y >= bmn.y && amx.z >= bmn.z;
}

// Candidate triangles of each query (one lane per query): count pass, then write pass.
template <bool WRITE>
__global__ __launch_bounds__(MC_BLOCK) void k_mc_candidates(MCArgs a) {
  const uint32_t q = blockIdx.x * MC_BLOCK + threadIdx.x;
  if (q >= a.nq) return;
  const uint32_t s = a.qshape[q];
  if (s >= a.nshapes) {
    atomicOr(a.err, 1u);
    if (!WRITE) a.count[q] = 0;
    return;
  }
  iso m1;
  m1.t = f3{a.mesh_pose.tx, a.mesh_pose.ty, a.mesh_pose.tz};
  m1.q = quat{a.mesh_pose.qi, a.mesh_pose.qj, a.mesh_pose.qk, a.mesh_pose.qw};
  const iso ls = iso_inv_mul(m1, load_pose(a.poses, s));  // ls_m2 = m1.inverse() * m2
  f3 bmn, bmx;
  shape_aabb_g<1>(load_shape(a.shapes, s), ls, a.P, 0, bmn, bmx);
  // AABB::loosened (aabb.rs:190-199)
  bmn = bmn + f3{-a.prediction, -a.prediction, -a.prediction};
  bmx = bmx + f3{a.prediction, a.prediction, a.prediction};
  uint32_t cnt = 0, slot = WRITE ? a.offs[q] : 0u;
  auto leaf = [&](uint32_t k) {
    f3 tmn, tmx;
    tri_box(a.tris, k, tmn, tmx);
    if (!box_hit(tmn, tmx, bmn, bmx)) return;
    if (WRITE) {
      a.ca[slot] = a.nshapes + k;  // the triangle's record in the combined set
      a.cb[slot] = s;
      ++slot;
    }
    ++cnt;
  };
  if (a.ntri == 1) {
    leaf(0);
  } else {
    uint32_t stk[MC_STACK];
    int sp = 0;
    uint32_t node = 0;
    for (;;) {
      const LNode nd = a.nodes[node];
      bool hl = box_hit(f3{nd.lminx, nd.lminy, nd.lminz}, f3{nd.lmaxx, nd.lmaxy, nd.lmaxz}, bmn, bmx);
      bool hr = box_hit(f3{nd.rminx, nd.rminy, nd.rminz}, f3{nd.rmaxx, nd.rmaxy, nd.rmaxz}, bmn, bmx);
      if (hl && (nd.child_l & NCX_LEAF_BIT)) { leaf(nd.child_l & ~NCX_LEAF_BIT); hl = false; }
      if (hr && (nd.child_r & NCX_LEAF_BIT)) { leaf(nd.child_r & ~NCX_LEAF_BIT); hr = false; }
      if (hl && hr) {
        if (sp == MC_STACK) { atomicOr(a.err, 2u); break; }
        stk[sp++] = nd.child_r;
        node = nd.child_l;
      } else if (hl) {
        node = nd.child_l;
      } else if (hr) {
        node = nd.child_r;
      } else if (sp > 0) {
        node = stk[--sp];
      } else {
        break;
      }
    }
  }
  if (!WRITE) a.count[q] = cnt;
}

// The deepest contact of each query over its candidates (contact_composite_shape_shape.rs:33-42:
// replace when deeper), ties to the least triangle id.
__global__ void k_mc_best(const uint32_t* __restrict__ offs, uint32_t nq, const uint32_t* __restrict__ ca,
                          uint32_t nshapes, const float4* __restrict__ tris, const uint8_t* __restrict__ chas,
                          const float* __restrict__ cw1, const float* __restrict__ cw2, const float* __restrict__ cn,
                          const float* __restrict__ cdepth, uint8_t* __restrict__ has, float* __restrict__ w1,
                          float* __restrict__ w2, float* __restrict__ nrm, float* __restrict__ depth,
                          uint32_t* __restrict__ face) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  uint32_t best = 0xFFFFFFFFu, best_face = 0xFFFFFFFFu;
  float best_d = 0.f;
  for (uint32_t j = offs[q]; j < offs[q + 1]; ++j) {
    if (chas[j] != 1) continue;
    const float d = cdepth[j];
    const uint32_t f = __float_as_uint(tris[3 * (size_t)(ca[j] - nshapes)].w);
    if (best == 0xFFFFFFFFu || d > best_d || (d == best_d && f < best_face)) {
      best = j;
      best_d = d;
      best_face = f;
    }
  }
  const bool h = best != 0xFFFFFFFFu;
  has[q] = h ? 1 : 0;
  for (int d = 0; d < 3; ++d) {
    w1[3 * (size_t)q + d] = h ? cw1[3 * (size_t)best + d] : 0.f;
    w2[3 * (size_t)q + d] = h ? cw2[3 * (size_t)best + d] : 0.f;
    nrm[3 * (size_t)q + d] = h ? cn[3 * (size_t)best + d] : 0.f;
  }
  depth[q] = h ? best_d : 0.f;
  if (face) face[q] = best_face;
}

// AABB::distance_to_point of the origin, solid (src/query/point/point_aabb.rs:138-150), for the
// Minkowski sum of box (mn, mx) and the shape's box: mins + shift + (-margin), maxs + shift + margin
// (distance_composite_shape_shape.rs:74-79).
__device__ __forceinline__ float msum_dist(f3 mn, f3 mx, f3 shift, f3 margin) {
  const f3 lo = (mn + shift) + (-margin), hi = (mx + shift) + margin;
  const f3 z = f3{0.f, 0.f, 0.f};
  const f3 mins_pt = lo - z, pt_maxs = z - hi;
  const f3 sh = f3{fmaxf(fmaxf(mins_pt.x, pt_maxs.x), 0.f), fmaxf(fmaxf(mins_pt.y, pt_maxs.y), 0.f),
                   fmaxf(fmaxf(mins_pt.z, pt_maxs.z), 0.f)};
  return norm(sh);
}

struct MDArgs {
  const LNode* nodes;
  const float4* tris;
  uint32_t ntri;
  ncx_pose mesh_pose;
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  const uint32_t* qshape;
  uint32_t nq, nshapes;
  float* dist;
  uint32_t* err;
  uint32_t* work;  // query counter (zero at launch)
};

#define MD_G 32
#define MD_BLOCK 128
#define MD_STACK 400
#define MD_RAW 128
#define MD_KEEP 64
#define MD_BLOCKS_PER_CU 4u  // resident: two wavefronts per SIMD

template <int G> __device__ __forceinline__ float group_min(float v) {
  v = fminf(v, __uint_as_float(lane_across<1>(__float_as_uint(v))));
  v = fminf(v, __uint_as_float(lane_across<2>(__float_as_uint(v))));
  if constexpr (G >= 8) v = fminf(v, __uint_as_float(lane_across<4>(__float_as_uint(v))));
  if constexpr (G >= 16) v = fminf(v, __uint_as_float(lane_across<8>(__float_as_uint(v))));
  if constexpr (G >= 32) v = fminf(v, __uint_as_float(lane_across<16>(__float_as_uint(v))));
  return v;
}
template <int G> __device__ __forceinline__ uint32_t group_min(uint32_t v) {
  v = min(v, lane_across<1>(v));
  v = min(v, lane_across<2>(v));
  if constexpr (G >= 8) v = min(v, lane_across<4>(v));
  if constexpr (G >= 16) v = min(v, lane_across<8>(v));
  if constexpr (G >= 32) v = min(v, lane_across<16>(v));
  return v;
}

// The answer so far of one query.  The reference takes the triangles by increasing cost m (msum_dist
// of their box), those of equal cost by id here, and stops at the first whose cost is not below the
// least distance d so far.  GJK in f32 can report a distance below the cost, zero above all, for a
// triangle that is large next to the shape; the reference then stops at that triangle if it comes
// to it.  So its answer is the d of the triangle with the least (max(d, m), m, id): a triangle whose
// cost is above that maximum comes after the one that has it, and no order of visiting changes
// which one that is.
struct MDBest {
  float cut, m, d;  // the maximum, the cost, the distance
  uint32_t id;
  __device__ __forceinline__ void start() {
    cut = d = NCX_FLT_MAX;
    m = -1.f;  // a cost of NCX_FLT_MAX is not below the first distance either
    id = 0u;
  }
  // whether a triangle or a box of cost c can still matter; a zero cost with a zero distance ends it
  __device__ __forceinline__ bool reaches(float c) const { return c < cut || (c == cut && c <= m && cut > 0.f); }
  __device__ __forceinline__ bool reaches(float c, uint32_t i) const {
    return c < cut || (c == cut && cut > 0.f && (c < m || (c == m && i < id)));
  }
};

// Distance of each query, one group of G lanes per query: a search of the tree that skips boxes and
// triangles whose cost says that the reference's search does not come to them.  Nothing but the cost
// may skip a triangle: bounds on the true distance are closer (with them and with GJK stopped at
// them 65,536 mixed shapes over a terrain of 131,072 triangles took 4.7 ms), but GJK's result can
// lie below the true distance, and which triangles such a bound skipped depended on the order in
// which lanes came to them.
// What bounds it: the latency of node and triangle fetches and of GJK's steps, which a query needs
// a few hundred of, one after another.  So the lanes of a group work on different things: each
// takes a node of the group's stack (in LDS, nearer children on top), or a triangle to test, or a
// triangle to run GJK on by itself.  The three kinds of step are kept apart, in lists of LDS, and
// run when most groups of the wavefront have enough of them, because a step that one lane takes
// costs the wavefront as much as one that all do.
// The shapes over a terrain above: 50 ms with one search per 2 lanes, 7.1 ms so (8 and 16 lanes a
// query 17 and 8.2 ms; lists twice as long 7.7 ms, three wavefronts on a SIMD 9.4 with 16 lanes).
template <int G>
__global__ __launch_bounds__(MD_BLOCK) void k_md(MDArgs a) {
  constexpr int GROUPS = 64 / G, REFILL = std::max(1, GROUPS / 4);
  static_assert(G >= 4 && G <= 32 && MD_RAW >= 4 * G && MD_KEEP >= 2 * G && MD_STACK >= LBVH_MAX_DEPTH + 2 * G, "list sizes");
  __shared__ uint2 stacks[MD_BLOCK / G][MD_STACK];
  __shared__ uint32_t raws[MD_BLOCK / G][MD_RAW];
  __shared__ uint2 keeps[MD_BLOCK / G][MD_KEEP];
  const int lane = threadIdx.x & 63, gl = lane & (G - 1), gbase = lane & ~(G - 1);
  const uint32_t gmask = ~0u >> (32 - G), below = (1u << gl) - 1u;
  uint2* const stk = stacks[threadIdx.x / G];
  uint32_t* const raw = raws[threadIdx.x / G];
  uint2* const keep = keeps[threadIdx.x / G];
  iso m1;
  m1.t = f3{a.mesh_pose.tx, a.mesh_pose.ty, a.mesh_pose.tz};
  m1.q = quat{a.mesh_pose.qi, a.mesh_pose.qj, a.mesh_pose.qk, a.mesh_pose.qw};
  bool live = false, done = false;
  uint32_t q = 0;
  int sp = 0, nr = 0, nk = 0;  // stack, raw triangles, tested triangles
  MDBest best;
  best.start();
  Ctx2 c;
  c.m1 = m1;
  c.g1.type = SHAPE_TRIANGLE;
  c.g1.off = 0;
  c.g1.cnt = 0;
  c.g1.a = c.g1.b = c.g1.c = 0.f;
  f3 shift, margin;
  auto mask_of = [&](bool v) { return (uint32_t)(__ballot(v) >> gbase) & gmask; };
  for (;;) {
    const uint64_t wm = __ballot(!live && !done && gl == 0), lm = __ballot(live);
    if ((wm | lm) == 0) break;
    if (wm && (lm == 0 || __popcll(wm) >= REFILL)) {
      uint32_t t = 0;
      const int first = __builtin_ctzll(wm);
      if (lane == first) t = atomicAdd(a.work, (uint32_t)__popcll(wm));
      t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
      if (!live && !done) {
        q = t + (uint32_t)__popcll(wm & ((1ull << gbase) - 1ull));
        const uint32_t s = q < a.nq ? a.qshape[q] : 0u;
        if (q >= a.nq) {
          done = true;
        } else if (s >= a.nshapes) {
          if (gl == 0) {
            atomicOr(a.err, 1u);
            a.dist[q] = 0.f;
          }
        } else {
          live = true;
          c.m2 = load_pose(a.poses, s);
          c.g2 = load_shape(a.shapes, s);
          const iso ls = iso_inv_mul(m1, c.m2);
          f3 bmn, bmx;
          shape_aabb_g<G>(c.g2, ls, a.P, gl, bmn, bmx);
          shift = -((bmn + bmx) * 0.5f);  // -ls_aabb2.center() (aabb.rs:95-97)
          margin = (bmx - bmn) * 0.5f;     // ls_aabb2.half_extents() (aabb.rs:101-104)
          best.start();
          nk = 0;
          sp = a.ntri > 1 ? 1 : 0;
          nr = a.ntri > 1 ? 0 : 1;
          if (gl == 0) {
            stk[0] = uint2{0u, __float_as_uint(0.f)};
            raw[0] = 0u;
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // nodes, while at least half of the live groups have some and room for their triangles
    for (;;) {
      const bool act = live && sp > 0 && nr + 2 * G <= MD_RAW;
      const uint64_t am = __ballot(act);
      if (am == 0) break;
      if (act) {
        // a full step at a time while the stack has room, else as deep as the tree may be
        const int room = MD_STACK - (int)LBVH_MAX_DEPTH - sp;
        const int p = min(min(G, sp), max(1, room));
        bool have = gl < p;
        uint2 e = uint2{0u, 0u};
        if (have) e = stk[sp - 1 - gl];
        sp -= p;
        have = have && best.reaches(__uint_as_float(e.y));
        bool inner0 = false, inner1 = false, leaf0 = false, leaf1 = false;
        uint32_t c0 = 0, c1 = 0;
        float k0 = 0.f, k1 = 0.f;
        if (have) {
          const LNode nd = a.nodes[e.x];
          const float cl = msum_dist(f3{nd.lminx, nd.lminy, nd.lminz}, f3{nd.lmaxx, nd.lmaxy, nd.lmaxz}, shift, margin);
          const float cr = msum_dist(f3{nd.rminx, nd.rminy, nd.rminz}, f3{nd.rmaxx, nd.rmaxy, nd.rmaxz}, shift, margin);
          const bool lfirst = cl <= cr;
          c0 = lfirst ? nd.child_l : nd.child_r;
          c1 = lfirst ? nd.child_r : nd.child_l;
          k0 = lfirst ? cl : cr;
          k1 = lfirst ? cr : cl;
          const bool h0 = best.reaches(k0), h1 = best.reaches(k1);
          leaf0 = h0 && (c0 & NCX_LEAF_BIT);
          leaf1 = h1 && (c1 & NCX_LEAF_BIT);
          inner0 = h0 && !leaf0;
          inner1 = h1 && !leaf1;
        }
        const uint32_t l0 = mask_of(leaf0), l1 = mask_of(leaf1), i0 = mask_of(inner0), i1 = mask_of(inner1);
        if (leaf0) raw[nr + __popc(l0 & below)] = c0 & ~NCX_LEAF_BIT;
        if (leaf1) raw[nr + __popc(l0) + __popc(l1 & below)] = c1 & ~NCX_LEAF_BIT;
        nr += __popc(l0) + __popc(l1);
        if (sp + __popc(i0) + __popc(i1) > MD_STACK) {
          if (gl == 0) atomicOr(a.err, 2u);
        } else {
          // farther children below, the first lane's (the nearest node's) on top
          if (inner1) stk[sp + __popc(i1) - 1 - __popc(i1 & below)] = uint2{c1, __float_as_uint(k1)};
          sp += __popc(i1);
          if (inner0) stk[sp + __popc(i0) - 1 - __popc(i0 & below)] = uint2{c0, __float_as_uint(k0)};
          sp += __popc(i0);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (2 * __popcll(am) < __popcll(__ballot(live))) break;
    }
    // costs of the triangles reached
    if (live && nr > 0 && nk + G <= MD_KEEP) {
      const int p = min(G, nr);
      bool ok = gl < p;
      uint32_t k = 0;
      if (ok) k = raw[nr - 1 - gl];
      nr -= p;
      float m = 0.f;
      if (ok) {
        f3 mn, mx;
        tri_box(a.tris, k, mn, mx);
        m = msum_dist(mn, mx, shift, margin);
        ok = best.reaches(m);
      }
      const uint32_t km = mask_of(ok);
      if (ok) keep[nk + __popc(km & below)] = uint2{k, __float_as_uint(m)};
      nk += __popc(km);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // GJK, once most live groups have a lane's worth each or nothing else to do
    const bool ready = live && nk > 0 && (nk >= G || (sp == 0 && nr == 0));
    const bool more = live && (sp > 0 || nr > 0) && !ready;
    const uint64_t rm = __ballot(ready);
    if (rm && 2 * __popcll(rm) >= __popcll(__ballot(more))) {
      if (ready) {
        const int p = min(G, nk);
        const bool mine = gl < p;
        uint2 e = uint2{0u, 0u};
        if (mine) e = keep[nk - 1 - gl];
        nk -= p;
        const float m = __uint_as_float(e.y);
        float d = NCX_FLT_MAX;
        uint32_t id = 0xFFFFFFFFu;
        if (mine) id = __float_as_uint(a.tris[3 * (size_t)e.x].w);
        if (mine && best.reaches(m, id)) {
          // query::distance(m1, triangle, m2, g2): distance_support_map_support_map (GJK from
          // m1.t - m2.t, distance_support_map_support_map.rs:25-53)
          c.g1.off = e.x;
          f3 dir;
          float nl;
          if (!try_normalize(c.m1.t - c.m2.t, NCX_FLT_EPS, &dir, &nl)) dir = f3{1.f, 0.f, 0.f};
          Simplex sx;
          const GJKOut r = gjk<1>(c, dir, NCX_FLT_MAX, sx, a.P, 0, 10000);
          d = r.status == GJK_S_CLOSEST ? norm(r.p1 - r.p2) : 0.f;
        }
        // the least (max(d, m), m, id) of the lanes; a distance that is no number counts as none
        const bool has = d < NCX_FLT_MAX;
        const float cut = has ? fmaxf(d, m) : NCX_FLT_MAX, gcut = group_min<G>(cut);
        const float gm = group_min<G>(has && cut == gcut ? m : NCX_FLT_MAX);
        const bool cand = has && cut == gcut && m == gm;
        const uint32_t gid = group_min<G>(cand ? id : 0xFFFFFFFFu);
        const float gd = group_min<G>(cand && id == gid ? d : NCX_FLT_MAX);
        if (gcut < best.cut || (gcut == best.cut && (gm < best.m || (gm == best.m && gid < best.id)))) {
          best.cut = gcut;
          best.m = gm;
          best.id = gid;
          best.d = gd;
        }
      }
    }
    if (live && sp == 0 && nr == 0 && nk == 0) {
      if (gl == 0) a.dist[q] = best.d;
      live = false;
    }
  }
}

static int mc_check(ncx_mesh* m, ncx_shapes* s, const char* what) {
  NCX_REQUIRE(m && s, std::string(what) + ": null argument");
  NCX_REQUIRE(m->ctx->device == s->ctx->device, std::string(what) + ": mesh and shapes on different devices");
  NCX_REQUIRE(s->n + m->ntri < 0x7FFFFFFFull, std::string(what) + ": too many shapes and triangles");
  return NCX_OK;
}

static int mc_err(ncx_mesh* m, const char* what) {
  uint32_t err = 0;
  ncx_ctx* ctx = m->ctx;
  NCX_HIP_CHECK(hipMemcpyAsync(&err, m->ctot.as<uint32_t>() + 1, 4, hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  if (err & 1u) {
    ncx_set_error(std::string(what) + ": a shape index is not a shape of the set");
    return NCX_E_INVALID;
  }
  if (err & 2u) {
    ncx_set_error(std::string(what) + ": traversal stack overflow");
    return NCX_E_CAPACITY;
  }
  return NCX_OK;
}

extern "C" int ncx_mesh_contact_batch(ncx_mesh* m, const ncx_pose* mesh_pose, ncx_shapes* s,
                                      const ncx_pose* poses_dev, const uint32_t* shape_dev, size_t n,
                                      float prediction, uint8_t* has_dev, float* world1_dev, float* world2_dev,
                                      float* normal_dev, float* depth_dev, uint32_t* face_dev) {
  int rc;
  if ((rc = mc_check(m, s, "ncx_mesh_contact_batch"))) return rc;
  NCX_REQUIRE(mesh_pose && poses_dev && shape_dev && has_dev && world1_dev && world2_dev && normal_dev && depth_dev,
              "ncx_mesh_contact_batch: null argument");
  NCX_REQUIRE(prediction >= 0.f, "ncx_mesh_contact_batch: negative prediction");
  NCX_REQUIRE(n < 0xFFFFFFFFull, "ncx_mesh_contact_batch: too many queries");
  if (n == 0) return NCX_OK;
  ncx_ctx* ctx = m->ctx;
  const size_t ns = s->n, nt = m->ntri, nc = ns + nt;
  // the combined shape set: the shapes, then the triangles as Triangle parts
  if (!m->comp) {
    m->comp = new ncx_shapes;
    m->comp->ctx = ctx;
  }
  ncx_shapes* C = m->comp;
  if ((rc = C->shapes.reserve(nc * sizeof(ncx_shape)))) return rc;
  if (ns) NCX_HIP_CHECK(hipMemcpyAsync(C->shapes.p, s->shapes.p, ns * sizeof(ncx_shape), hipMemcpyDeviceToDevice,
                                       ctx->stream));
  hipLaunchKernelGGL(k_mc_tri_records, dim3(ceil_div(nt, 256)), dim3(256), 0, ctx->stream,
                     C->shapes.as<ncx_shape>() + ns, nt);
  C->n = nc;
  C->buckets = s->buckets;  // a triangle changes no pair's bucket
  C->npts = s->npts;
  C->hx = s->hx; C->hy = s->hy; C->hz = s->hz;  // borrowed (never released through C)
  C->tri = m->tris.as<float4>();
  if ((rc = m->cposes.reserve(nc * sizeof(ncx_pose)))) return rc;
  if (ns) NCX_HIP_CHECK(hipMemcpyAsync(m->cposes.p, poses_dev, ns * sizeof(ncx_pose), hipMemcpyDeviceToDevice,
                                       ctx->stream));
  hipLaunchKernelGGL(k_mc_fill_pose, dim3(ceil_div(nt, 256)), dim3(256), 0, ctx->stream,
                     m->cposes.as<ncx_pose>() + ns, nt, *mesh_pose);
  NCX_HIP_CHECK(hipGetLastError());
  // candidates
  if ((rc = m->ccnt.reserve(n * 4)) || (rc = m->coffs.reserve((n + 1) * 4)) || (rc = m->ctot.reserve(16))) return rc;
  if ((rc = fill_u32(ctx, m->ctot.as<uint32_t>(), 2, 0u))) return rc;
  MCArgs a = {};
  a.nodes = m->bvh.nodes.as<LNode>();
  a.tris = m->tris.as<float4>();
  a.ntri = (uint32_t)nt;
  a.mesh_pose = *mesh_pose;
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), m->tris.as<float4>()};
  a.poses = poses_dev;
  a.qshape = shape_dev;
  a.nq = (uint32_t)n;
  a.nshapes = (uint32_t)ns;
  a.prediction = prediction;
  a.count = m->ccnt.as<uint32_t>();
  a.err = m->ctot.as<uint32_t>() + 1;
  const unsigned nb = ceil_div(n, MC_BLOCK);
  hipLaunchKernelGGL((k_mc_candidates<false>), dim3(nb), dim3(MC_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  if ((rc = scan_exclusive_u32(ctx, a.count, m->coffs.as<uint32_t>(), n, m->cscan, m->ctot.as<uint32_t>()))) return rc;
  NCX_HIP_CHECK(hipMemcpyAsync(m->coffs.as<uint32_t>() + n, m->ctot.p, 4, hipMemcpyDeviceToDevice, ctx->stream));
  if ((rc = mc_err(m, "ncx_mesh_contact_batch"))) return rc;
  uint32_t total = 0;
  NCX_HIP_CHECK(hipMemcpyAsync(&total, m->ctot.p, 4, hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  const size_t cap = std::max<size_t>(total, 1);
  if ((rc = m->ca.reserve(cap * 4)) || (rc = m->cb.reserve(cap * 4)) || (rc = m->chas.reserve(cap)) ||
      (rc = m->cw1.reserve(cap * 12)) || (rc = m->cw2.reserve(cap * 12)) || (rc = m->cn.reserve(cap * 12)) ||
      (rc = m->cdepth.reserve(cap * 4)) || (rc = m->citers.reserve(cap * 4)))
    return rc;
  a.offs = m->coffs.as<uint32_t>();
  a.ca = m->ca.as<uint32_t>();
  a.cb = m->cb.as<uint32_t>();
  hipLaunchKernelGGL((k_mc_candidates<true>), dim3(nb), dim3(MC_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  if (total) {
    // query::contact(mesh pose, triangle, shape pose, shape, prediction) on every candidate
    if ((rc = contact_tiers_reserve(C->tiers, ctx, total, total))) return rc;
    if ((rc = contacts_launch_device_count(C, C->tiers, ctx, m->cposes.as<ncx_pose>(), m->ca.as<uint32_t>(),
                                           m->cb.as<uint32_t>(), m->ctot.as<uint32_t>(), total, prediction, nullptr,
                                           10000, m->chas.as<uint8_t>(), m->cw1.as<float>(), m->cw2.as<float>(),
                                           m->cn.as<float>(), m->cdepth.as<float>(), m->citers.as<int32_t>(), true)))
      return rc;
    NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    size_t large = 0;
    if ((rc = contacts_resolve_overflow(C->tiers, ctx, &large))) return rc;
  }
  hipLaunchKernelGGL(k_mc_best, dim3(ceil_div(n, 256)), dim3(256), 0, ctx->stream, m->coffs.as<uint32_t>(),
                     (uint32_t)n, m->ca.as<uint32_t>(), (uint32_t)ns, m->tris.as<float4>(), m->chas.as<uint8_t>(),
                     m->cw1.as<float>(), m->cw2.as<float>(), m->cn.as<float>(), m->cdepth.as<float>(), has_dev,
                     world1_dev, world2_dev, normal_dev, depth_dev, face_dev);
  NCX_HIP_CHECK(hipGetLastError());
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  return NCX_OK;
}

extern "C" int ncx_mesh_distance_batch(ncx_mesh* m, const ncx_pose* mesh_pose, ncx_shapes* s,
                                       const ncx_pose* poses_dev, const uint32_t* shape_dev, size_t n,
                                       float* dist_dev) {
  int rc;
  if ((rc = mc_check(m, s, "ncx_mesh_distance_batch"))) return rc;
  NCX_REQUIRE(mesh_pose && poses_dev && shape_dev && dist_dev, "ncx_mesh_distance_batch: null argument");
  NCX_REQUIRE(n < 0xFFFFFFFFull, "ncx_mesh_distance_batch: too many queries");
  if (n == 0) return NCX_OK;
  // the query counter counts past n by what the waiting wavefronts ask for, in 32 bits
  const size_t chunk = (size_t)1 << 30;
  if (n > chunk) {
    for (size_t o = 0; o < n; o += chunk)
      if ((rc = ncx_mesh_distance_batch(m, mesh_pose, s, poses_dev, shape_dev + o, std::min(chunk, n - o), dist_dev + o)))
        return rc;
    return NCX_OK;
  }
  ncx_ctx* ctx = m->ctx;
  if ((rc = m->ctot.reserve(16)) || (rc = fill_u32(ctx, m->ctot.as<uint32_t>(), 3, 0u))) return rc;
  MDArgs a = {};
  a.nodes = m->bvh.nodes.as<LNode>();
  a.tris = m->tris.as<float4>();
  a.ntri = (uint32_t)m->ntri;
  a.mesh_pose = *mesh_pose;
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), m->tris.as<float4>()};
  a.poses = poses_dev;
  a.qshape = shape_dev;
  a.nq = (uint32_t)n;
  a.nshapes = (uint32_t)s->n;
  a.dist = dist_dev;
  a.err = m->ctot.as<uint32_t>() + 1;
  a.work = m->ctot.as<uint32_t>() + 2;
  const unsigned blocks =
      std::max(1u, std::min<unsigned>(ceil_div(n * MD_G, MD_BLOCK), (unsigned)ctx->num_cus * MD_BLOCKS_PER_CU));
  hipLaunchKernelGGL(k_md<MD_G>, dim3(blocks), dim3(MD_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  return mc_err(m, "ncx_mesh_distance_batch");
}
