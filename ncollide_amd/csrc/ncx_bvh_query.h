// ncx_bvh_query.h -- batched LBVH queries with one query per lane: boxes, points and rays against
// the broad phase's stored boxes (BroadPhase::interferences_with_bounding_volume / _with_point /
// _with_ray, src/pipeline/broad_phase/dbvt_broad_phase.rs:387-432), and the world-level ray
// queries that also cast the ray on each proxy's shape (glue::interferences_with_ray and
// first_interference_with_ray, src/pipeline/glue/query.rs:13-66, 200-224).
//
// Each lane walks the tree depth-first with its own stack (the tree is at most LBVH_MAX_DEPTH
// levels deep, so the stack never holds more entries than that).  The collectors run twice: a
// count pass, then, after a scan, a write pass to each query's slots.  The first-hit search
// visits the nearer child first and skips boxes entered after the best hit so far, with a result
// that does not depend on the visiting order (k_bq_first_ray).
#pragma once
#include "ncx_gjk.h"

#define BQ_BOX 0
#define BQ_POINT 1
#define BQ_RAY 2
#define BQ_BLOCK 128
#define BQ_NONE 0xFFFFFFFFu

struct BQArgs {
  const LNode* nodes;
  const uint32_t* order;  // sorted leaf position -> primitive index
  const uint32_t* alive;  // primitive index -> handle (null: the identity)
  const uint32_t* in_tree;  // per handle: nonzero while the proxy is in the tree (null: all are)
  const float* leaf_soa;  // primitive boxes, 6 SoA arrays of stride nleaves (read when nleaves == 1)
  uint32_t nleaves;
  const float* q[6];      // queries: box (mins, maxs), point (x, y, z), ray (origin, dir)
  uint32_t nq;
  float max_toi;
  // shapes, for the world-level ray queries
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  int cast_shapes;
  // outputs
  uint32_t* count;        // count pass: hits per query
  const uint32_t* offs;   // write pass: first slot of each query
  uint32_t* handles;
  float* toi;
  float* nrm;
  uint32_t* err;          // set when a traversal stack would overflow (a tree deeper than the bound)
  const uint32_t* perm;   // first-hit rays: the k-th ray taken is perm[k] (null: ray k)
  uint32_t* work;         // first-hit rays: ray counter (zero at launch)
};

#define BQ_STACK (LBVH_MAX_DEPTH + 2)

// AABB::toi_with_ray with solid = true at the identity (src/query/ray/ray_aabb.rs:13-50).
__device__ __forceinline__ bool bq_ray_box(f3 o, f3 d, float max_toi, float mnx, float mny, float mnz, float mxx,
                                           float mxy, float mxz, float& toi) {
  float tmin = 0.f, tmax = max_toi;
  const float mn[3] = {mnx, mny, mnz}, mx[3] = {mxx, mxy, mxz};
  const float oo[3] = {o.x, o.y, o.z}, dd[3] = {d.x, d.y, d.z};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (dd[i] == 0.f) {
      if (oo[i] < mn[i] || oo[i] > mx[i]) return false;
    } else {
      const float denom = 1.f / dd[i];
      float tn = (mn[i] - oo[i]) * denom;
      float tf = (mx[i] - oo[i]) * denom;
      if (tn > tf) { float x = tn; tn = tf; tf = x; }
      tmin = fmaxf(tmin, tn);
      tmax = fminf(tmax, tf);
      if (tmin > tmax) return false;
    }
  }
  toi = tmin;
  return true;
}

// The interference test of query kind K against one box; for rays `cost` is the box's entry toi.
template <int K>
__device__ __forceinline__ bool bq_test(const float qv[6], float max_toi, float mnx, float mny, float mnz, float mxx,
                                        float mxy, float mxz, float& cost) {
  cost = 0.f;
  if (K == BQ_BOX)  // AABB::intersects (src/bounding_volume/aabb.rs:156-158)
    return mnx <= qv[3] && mny <= qv[4] && mnz <= qv[5] && mxx >= qv[0] && mxy >= qv[1] && mxz >= qv[2];
  if (K == BQ_POINT)  // AABB::contains_local_point (aabb.rs:138-146)
    return !(qv[0] < mnx || qv[0] > mxx || qv[1] < mny || qv[1] > mxy || qv[2] < mnz || qv[2] > mxz);
  return bq_ray_box(f3{qv[0], qv[1], qv[2]}, f3{qv[3], qv[4], qv[5]}, max_toi, mnx, mny, mnz, mxx, mxy, mxz, cost);
}

__device__ __forceinline__ uint32_t bq_handle(const BQArgs& a, uint32_t leaf_pos) {
  const uint32_t prim = a.order[leaf_pos];
  return a.alive ? a.alive[prim] : prim;
}

// Collects every leaf whose box passes the test (and, with cast_shapes, whose shape the ray hits,
// solid = true).  WRITE = false counts; WRITE = true writes handles (and toi/normal) from offs[q].
template <int K, bool WRITE>
__global__ __launch_bounds__(BQ_BLOCK) void k_bq_collect(BQArgs a) {
  const uint32_t qi = blockIdx.x * BQ_BLOCK + threadIdx.x;
  if (qi >= a.nq) return;
  __shared__ float snaps[K == BQ_RAY ? BQ_BLOCK : 1][RC_SNAP];
  float* const snap = snaps[K == BQ_RAY ? threadIdx.x : 0];
  const int nq = K == BQ_POINT ? 3 : 6;
  float qv[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int d = 0; d < nq; ++d) qv[d] = a.q[d][qi];
  uint32_t cnt = 0;
  uint32_t slot = WRITE ? a.offs[qi] : 0u;
  auto emit = [&](uint32_t leaf_pos) {
    const uint32_t h = bq_handle(a, leaf_pos);
    if (a.in_tree && !a.in_tree[h]) return;  // removed since the last update
    float t = 0.f;
    f3 n = f3{0.f, 0.f, 0.f};
    if (K == BQ_RAY && a.cast_shapes) {
      uint32_t feat;
      if (!shape_ray_cast<1>(load_shape(a.shapes, h), load_pose(a.poses, h), f3{qv[0], qv[1], qv[2]},
                             f3{qv[3], qv[4], qv[5]}, a.max_toi, true, a.P, 0, snap, t, n, feat))
        return;
    }
    if (WRITE) {
      a.handles[slot] = h;
      if (a.toi) a.toi[slot] = t;
      if (a.nrm) {
        a.nrm[3 * (size_t)slot] = n.x;
        a.nrm[3 * (size_t)slot + 1] = n.y;
        a.nrm[3 * (size_t)slot + 2] = n.z;
      }
      ++slot;
    }
    ++cnt;
  };
  if (a.nleaves == 1) {
    const float* b = a.leaf_soa;
    float c;
    if (bq_test<K>(qv, a.max_toi, b[0], b[1], b[2], b[3], b[4], b[5], c)) emit(0);
  } else if (a.nleaves > 1) {
    uint32_t stk[BQ_STACK];
    int sp = 0;
    uint32_t node = 0;
    for (;;) {
      const LNode nd = a.nodes[node];
      float cl, cr;
      bool hl = bq_test<K>(qv, a.max_toi, nd.lminx, nd.lminy, nd.lminz, nd.lmaxx, nd.lmaxy, nd.lmaxz, cl);
      bool hr = bq_test<K>(qv, a.max_toi, nd.rminx, nd.rminy, nd.rminz, nd.rmaxx, nd.rmaxy, nd.rmaxz, cr);
      if (hl && (nd.child_l & NCX_LEAF_BIT)) { emit(nd.child_l & ~NCX_LEAF_BIT); hl = false; }
      if (hr && (nd.child_r & NCX_LEAF_BIT)) { emit(nd.child_r & ~NCX_LEAF_BIT); hr = false; }
      if (hl && hr) {
        if (sp == BQ_STACK) { atomicOr(a.err, 1u); break; }
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
  if (!WRITE) a.count[qi] = cnt;
}

// First hit of each ray among the proxies' shapes (solid = true, toi <= max_toi): the least
// (toi, handle) over the leaves whose box the ray enters no later than the best hit so far, taken by
// the boxes' entry tois as the reference's best-first search does.  A cast can report a toi below
// its own box's entry -- GJK's on a capsule or hull by up to its absolute tolerance of 1e-3, a ball's
// closed form where the ray starts hundreds of radii away -- and such a hit counts only if no other
// is as early as its box's entry.  So the hit kept is the one with the least (max(toi, entry), toi,
// handle), and a box is skipped when its entry is past that maximum: a rule without an order, while
// the leaves come in an order that depends on the wavefront's other rays.
// What bounds it: the ray casts on capsules and hulls (GJK, 7 to 20 iterations), and divergence --
// the rays of a wavefront reach them at different times, and a cast that one lane does alone takes
// as long as one that all do.  So one lane walks the tree for one ray; balls and cuboids (closed
// forms) are cast as they are reached; capsules and hulls are kept, up to BQ_KEEP of them, while the
// lane goes on; and when BQ_WAITING lanes have kept all they can, or have nothing left to walk, each
// casts its nearest kept one.  A lane whose ray has ended takes the next at the wavefront's next
// refill.  524,288 rays over 262,144 mixed shapes: 6.45 ms with one ray a lane and casts in place,
// 1.7 ms now (3.5 ms where one ray's cast runs to thousands of iterations).  Casting at 16, 32, 48,
// 56, 60 and 64 waiting lanes (whole call): 3.2, 2.6, 2.38, 2.3, 2.29, 2.32 ms with two wavefronts on
// a SIMD; three of them 2.03; four, which spill, 2.34.  Every kept one is cast, without a test of its bounding ball or segment first: GJK's ray
// cast reports rays that pass a shape by several hundredths of its size as hits.
#define BQ_KEEP 2
#define BQ_LDS_STACK 14
#define BQ_WAITING 56  // lanes that wait before the kept shapes are cast
#define BQ_REFILL 8    // idle lanes before the next rays are taken
#define BQ_CU_BLOCKS 6
static __global__ __launch_bounds__(BQ_BLOCK, 3) void k_bq_first_ray(BQArgs a) {
  __shared__ float snaps[BQ_BLOCK][RC_SNAP];
  __shared__ uint2 lstk[BQ_LDS_STACK][BQ_BLOCK];
  float* const snap = snaps[threadIdx.x];
  uint2 deep[BQ_STACK + 1 - BQ_LDS_STACK];  // entries past the LDS ones; one more for a leaf put back
  const int lane = threadIdx.x & 63;
  bool live = false, done = false, walk = false;
  uint32_t qi = 0, node = 0, best_h = BQ_NONE, kh0 = 0, kh1 = 0;
  int sp = 0, nk = 0;
  float cut = 0.f, best_t = 0.f, kt0 = 0.f, kt1 = 0.f;
  f3 o = f3{0.f, 0.f, 0.f}, dir = o, best_n = o;
  auto hit = [&](uint32_t h, float entry, float t, f3 n) {
    const float c = t < entry ? entry : t;
    if (c < cut || (c == cut && (t < best_t || (t == best_t && h < best_h)))) {
      cut = c;
      best_t = t;
      best_h = h;
      best_n = n;
    }
  };
  auto leaf = [&](uint32_t leaf_pos, float entry) {
    const uint32_t h = bq_handle(a, leaf_pos);
    const ShapeD g = load_shape(a.shapes, h);
    const iso m = load_pose(a.poses, h);
    if (g.type == NCX_CAPSULE || g.type == NCX_CONVEX_HULL) {
      // the nearest of the kept ones first
      const bool front = nk == 0 || entry < kt0;
      kh1 = front ? kh0 : h;
      kt1 = front ? kt0 : entry;
      kh0 = front ? h : kh0;
      kt0 = front ? entry : kt0;
      ++nk;
    } else {
      float t;
      f3 n;
      uint32_t feat;
      if (shape_ray_cast_closed(g, m, o, dir, a.max_toi, true, t, n, feat)) hit(h, entry, t, n);
    }
  };
  auto push = [&](uint32_t child, float entry) {
    if (sp == BQ_STACK + 1) {
      atomicOr(a.err, 1u);
      return;
    }
    const uint2 e = uint2{child, __float_as_uint(entry)};
    if (sp < BQ_LDS_STACK) lstk[sp][threadIdx.x] = e;
    else deep[sp - BQ_LDS_STACK] = e;
    ++sp;
  };
  for (;;) {
    const uint64_t wm = __ballot(!live && !done), lm = __ballot(live);
    if ((wm | lm) == 0) break;
    if (wm && (lm == 0 || __popcll(wm) >= BQ_REFILL)) {
      uint32_t t = 0;
      const int first = __builtin_ctzll(wm);
      if (lane == first) t = atomicAdd(a.work, (uint32_t)__popcll(wm));
      t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
      if (!live && !done) {
        const uint32_t gi = t + (uint32_t)__popcll(wm & ((1ull << lane) - 1ull));
        if (gi >= a.nq) {
          done = true;
        } else {
          live = true;
          qi = a.perm ? a.perm[gi] : gi;
          o = f3{a.q[0][qi], a.q[1][qi], a.q[2][qi]};
          dir = f3{a.q[3][qi], a.q[4][qi], a.q[5][qi]};
          cut = best_t = a.max_toi;
          best_h = BQ_NONE;
          best_n = f3{0.f, 0.f, 0.f};
          sp = nk = 0;
          node = 0;
          walk = a.nleaves > 1;
          if (a.nleaves == 1) {
            const float* b = a.leaf_soa;
            float c;
            if (bq_ray_box(o, dir, a.max_toi, b[0], b[1], b[2], b[3], b[4], b[5], c)) leaf(0, c);
          }
        }
      }
    }
    for (;;) {
      const bool act = live && walk && nk < BQ_KEEP;
      const uint64_t am = __ballot(act);
      if (am == 0 || __popcll(__ballot(live && !act)) >= BQ_WAITING) break;
      if (act) {
        uint32_t next = BQ_NONE;
        float next_t = 0.f;
        if (node != BQ_NONE) {
          const LNode nd = a.nodes[node];
          float cl, cr;
          const bool hl = bq_ray_box(o, dir, a.max_toi, nd.lminx, nd.lminy, nd.lminz, nd.lmaxx, nd.lmaxy, nd.lmaxz, cl);
          const bool hr = bq_ray_box(o, dir, a.max_toi, nd.rminx, nd.rminy, nd.rminz, nd.rmaxx, nd.rmaxy, nd.rmaxz, cr);
          const bool lfirst = hl && (!hr || cl <= cr);
          const bool h0 = (lfirst ? hl : hr) && (lfirst ? cl : cr) <= cut;
          const bool h1 = (lfirst ? hr : hl) && (lfirst ? cr : cl) <= cut;
          const uint32_t c0 = lfirst ? nd.child_l : nd.child_r, c1 = lfirst ? nd.child_r : nd.child_l;
          const float t1 = lfirst ? cr : cl;
          if (h0) {
            next = c0;
            next_t = lfirst ? cl : cr;
            if (h1) push(c1, t1);
          } else if (h1) {
            next = c1;
            next_t = t1;
          }
        }
        // the next node; leaves are taken on the way
        for (;;) {
          if (next == BQ_NONE) {
            if (sp == 0) break;
            --sp;
            uint2 e;
            if (sp < BQ_LDS_STACK) e = lstk[sp][threadIdx.x];
            else e = deep[sp - BQ_LDS_STACK];
            next_t = __uint_as_float(e.y);
            if (!(next_t <= cut)) continue;
            next = e.x;
          }
          if (!(next & NCX_LEAF_BIT)) break;
          if (nk == BQ_KEEP) {  // no room: back onto the stack
            push(next, next_t);
            next = BQ_NONE;
            break;
          }
          leaf(next & ~NCX_LEAF_BIT, next_t);
          next = BQ_NONE;
        }
        node = next;
        walk = node != BQ_NONE || sp > 0;
      }
    }
    if (live && nk > 0 && (nk == BQ_KEEP || !walk)) {
      const uint32_t h = kh0;
      const float entry = kt0;
      kh0 = kh1;
      kt0 = kt1;
      --nk;
      if (entry <= cut) {
        float t;
        f3 n;
        uint32_t feat;
        if (shape_ray_cast<1>(load_shape(a.shapes, h), load_pose(a.poses, h), o, dir, a.max_toi, true, a.P, 0, snap, t,
                              n, feat))
          hit(h, entry, t, n);
      }
    }
    if (live && nk == 0 && !walk) {
      a.handles[qi] = best_h;
      a.toi[qi] = best_h == BQ_NONE ? -1.f : best_t;
      a.nrm[3 * (size_t)qi] = best_n.x;
      a.nrm[3 * (size_t)qi + 1] = best_n.y;
      a.nrm[3 * (size_t)qi + 2] = best_n.z;
      live = false;
    }
  }
}

// Count pass, scan, write pass.  *total = hits over all queries; NCX_E_CAPACITY when above cap
// (nothing written).  offs (nq + 1 entries) receives each query's first slot and the total.
inline int bq_collect_run(ncx_ctx* ctx, BQArgs a, int kind, uint32_t* offs, size_t cap, size_t* total, DevBuf& cnt,
                          DevBuf& scan_tmp, DevBuf& tot) {
  if (a.nq == 0) {
    *total = 0;
    return NCX_OK;
  }
  int rc;
  if ((rc = cnt.reserve((size_t)a.nq * 4)) || (rc = tot.reserve(16))) return rc;
  if ((rc = fill_u32(ctx, tot.as<uint32_t>() + 1, 1, 0u))) return rc;
  a.count = cnt.as<uint32_t>();
  a.err = tot.as<uint32_t>() + 1;
  const unsigned nb = ceil_div(a.nq, BQ_BLOCK);
  if (kind == BQ_BOX) hipLaunchKernelGGL((k_bq_collect<BQ_BOX, false>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  else if (kind == BQ_POINT) hipLaunchKernelGGL((k_bq_collect<BQ_POINT, false>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  else hipLaunchKernelGGL((k_bq_collect<BQ_RAY, false>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  if ((rc = scan_exclusive_u32(ctx, a.count, offs, a.nq, scan_tmp, tot.as<uint32_t>()))) return rc;
  uint32_t t[2] = {0, 0};
  NCX_HIP_CHECK(hipMemcpyAsync(t, tot.p, 8, hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipMemcpyAsync(offs + a.nq, tot.p, 4, hipMemcpyDeviceToDevice, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  NCX_REQUIRE(t[1] == 0, "interference query: traversal stack overflow");
  *total = t[0];
  if (t[0] > cap) {
    ncx_set_error("interference query: " + std::to_string(t[0]) + " hits exceed the output capacity");
    return NCX_E_CAPACITY;
  }
  a.offs = offs;
  if (kind == BQ_BOX) hipLaunchKernelGGL((k_bq_collect<BQ_BOX, true>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  else if (kind == BQ_POINT) hipLaunchKernelGGL((k_bq_collect<BQ_POINT, true>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  else hipLaunchKernelGGL((k_bq_collect<BQ_RAY, true>), dim3(nb), dim3(BQ_BLOCK), 0, ctx->stream, a);
  NCX_HIP_CHECK(hipGetLastError());
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  return NCX_OK;
}
