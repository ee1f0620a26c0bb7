// ncx_narrow.hip -- batched convex contact / distance (GJK + EPA) on the GPU.
//
// Contacts take two kernels.  k_contact_gjk runs GJK and the closed forms, one group of G lanes per
// pair, finishes every pair that needs no EPA and writes an EPA record (the pair and its simplex)
// for the others; k_epa (ncx_epa.h) runs the records on LDS arenas, in tiers of growing capacity.
// Distances need GJK alone (k_distance).  Every lane of a group runs the same control flow on the
// same values, and the lanes split the vertex scans of ConvexHull support functions with an argmax
// reduction that reproduces point_cloud_support_point_id's first-maximum rule
// (src/utils/point_cloud_support_point.rs:6-24).
//
// All arithmetic restates the reference in f32 with its operation order:
//   GJK      src/query/algorithms/gjk.rs:76-177
//   simplex  src/query/algorithms/voronoi_simplex3.rs:49-280
//   EPA      src/query/algorithms/epa3.rs:219-454
//   dispatch src/query/contact/contact_shape_shape.rs:10-48,
//            src/query/distance/distance.rs:9-33
#include <algorithm>
#include "ncx_epa.h"

struct KArgs {
  const ncx_shape* shapes;
  Pool P;
  const ncx_pose* poses;
  const uint32_t* ia;
  const uint32_t* ib;
  const uint32_t* list;  // optional indirection (re-runs)
  size_t npairs;
  float prediction;
  const float* init_dir;
  int max_iter;
  int cap_seg;  // contact-manifold mode: a capsule is its core segment, and each capsule of a pair
                // adds its radius to the pair's prediction
  uint8_t* has;
  float* w1;
  float* w2;
  float* nrm;
  float* depth;
  int32_t* iters;
  float* fdir;  // optional: the support-map result direction per pair (PairOut::fdir; the init_dir
                // when that path returned nothing), for a per-pair direction cache
  float* dist;
  uint8_t* arena;       // device-memory tier: EPA arenas of vcap vertices and fcap faces
  uint32_t vcap, fcap;
  EpaRec* rec;               // EPA records: GJK writes them, the EPA kernels read them
  uint32_t* rec_count;       // their number
  float* sup;                // per EPA group: its polytope's support points, 6 floats a vertex
  uint32_t* ovf_count;  // EPA runs that outgrew the arena
  uint32_t* ovf_list;   // their records (first ovf_cap of them)
  uint32_t ovf_cap;
  int ovf_pairs;        // the list holds the runs' pairs instead
  int distance_mode;
  uint32_t nshapes;
  uint32_t* bad_index;  // set to 1 when a pair names a shape >= nshapes
  const uint32_t* n_dev;  // optional device-side count of pairs or listed records (capped by npairs)
  uint32_t* work;         // work counter (zero at launch): pairs and records are taken from it
  const uint32_t* range_b;  // optional device begin and end into list: a run of buckets
  const uint32_t* range_e;
  uint32_t part_lo, part_hi;  // the part of that list the launch takes (contacts)
  const uint8_t* sus_load;  // saved EPA runs of the list's ENTRY_SAVED entries, slot = list position
  size_t sus_load_bytes;
  uint8_t* sus_save;        // slots for runs this launch suspends (LDS tiers only; null: none)
  size_t sus_save_bytes;
  uint32_t sus_save_cap;
};

// EPA arenas (ncx_epa.h): the first tier's two (40 and 20 iterations, of which 6 or 11 blocks of 8
// runs fit a CU), then the tiers for the runs that outgrow them.
typedef EpaArena<44, 86, 104, 32, 0, 10> ArenaT1;
typedef EpaArena<24, 46, 54, 24, 0, 10> ArenaT1S;
typedef EpaArena<64, 126, 150, 48, 0, 10> ArenaT2;
typedef EpaArena<256, 510, 600, 96, 0, 10> ArenaT3;
typedef EpaArena<2000, 4000, 4400, 256, 256, 16> ArenaT4;
#define T1_BLOCKS 6u
#define T1S_BLOCKS 11u
#define T2_G 16
#define T2_BS 64
#define T2_BLOCKS_PER_CU 8u
#define T3_BLOCKS_PER_CU 8u
static_assert(ArenaT1::BYTES * 8 * T1_BLOCKS <= 163840 && ArenaT1S::BYTES * 8 * T1S_BLOCKS <= 163840, "blocks per CU");
static_assert(ArenaT2::BYTES * (T2_BS / T2_G) * T2_BLOCKS_PER_CU <= 163840 && ArenaT4::BYTES <= 163840 &&
                  ArenaT3::BYTES * T3_BLOCKS_PER_CU <= 163840, "blocks per CU");
// Support points of the polytopes in flight, the most of any tier (per CU).
constexpr size_t EPA_SUP_FLOATS_PER_CU = 6 * (size_t)std::max({T1_BLOCKS * 8 * ArenaT1::VC, T1S_BLOCKS * 8 * ArenaT1S::VC,
                                                              T2_BLOCKS_PER_CU * (T2_BS / T2_G) * ArenaT2::VC,
                                                              T3_BLOCKS_PER_CU * ArenaT3::VC, ArenaT4::VC});

constexpr uint32_t ilog2_floor(uint32_t x) { return x <= 1 ? 0u : 1u + ilog2_floor(x >> 1); }

// The pair's shapes and poses, with the contact-manifold mode's capsules as their core segments
// (capsule_shape_manifold_generator.rs:34-37, capsule_capsule_manifold_generator.rs:36-40), and
// the pair's prediction.
__device__ __forceinline__ Ctx2 contact_ctx(const KArgs& a, uint32_t i1, uint32_t i2, float& pred) {
  Ctx2 c;
  c.g1 = load_shape(a.shapes, i1);
  c.g2 = load_shape(a.shapes, i2);
  c.m1 = load_pose(a.poses, i1);
  c.m2 = load_pose(a.poses, i2);
  pred = a.prediction;
  if (a.cap_seg) {
    if (c.g1.type == NCX_CAPSULE) { pred = pred + c.g1.b; c.g1.type = SHAPE_SEGMENT; }
    if (c.g2.type == NCX_CAPSULE) { pred = pred + c.g2.b; c.g2.type = SHAPE_SEGMENT; }
  }
  return c;
}

__device__ __forceinline__ void write_contact(const KArgs& a, size_t k, const PairOut& o, f3 idir) {
  a.has[k] = (uint8_t)o.has;
  const bool h = o.has == 1;
  const f3 z = f3{0.f, 0.f, 0.f}, w1 = sel3(h, o.w1, z), w2 = sel3(h, o.w2, z), n = sel3(h, o.n, z);
  a.w1[3 * k] = w1.x; a.w1[3 * k + 1] = w1.y; a.w1[3 * k + 2] = w1.z;
  a.w2[3 * k] = w2.x; a.w2[3 * k + 1] = w2.y; a.w2[3 * k + 2] = w2.z;
  a.nrm[3 * k] = n.x; a.nrm[3 * k + 1] = n.y; a.nrm[3 * k + 2] = n.z;
  a.depth[k] = h ? o.depth : 0.f;
  if (a.fdir) {
    // ConvexPolyhedronConvexPolyhedronManifoldGenerator keeps its last_gjk_dir when the
    // result carries no direction (manifold_generator.rs:115-146)
    const bool z = o.fdir.x == 0.f && o.fdir.y == 0.f && o.fdir.z == 0.f;
    const f3 fd = z ? idir : o.fdir;
    a.fdir[3 * k] = fd.x; a.fdir[3 * k + 1] = fd.y; a.fdir[3 * k + 2] = fd.z;
  }
}

__device__ __forceinline__ f3 load_init_dir(const KArgs& a, size_t k) {
  if (!a.init_dir) return f3{0.f, 0.f, 0.f};
  return f3{a.init_dir[3 * k], a.init_dir[3 * k + 1], a.init_dir[3 * k + 2]};
}

#define GJK_BS 256

// The pairs of a wavefront's next pass: 64 / G of them, with one atomic.
template <int G>
__device__ __forceinline__ size_t next_pairs(uint32_t* work, int lane) {
  uint32_t t = 0;
  if (lane == 0) t = atomicAdd(work, 64u / G);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)t) + (uint32_t)lane / G;
}

// GJK and closed forms of contact pairs; the pairs that need EPA leave a record.
template <int G>
__global__ __launch_bounds__(GJK_BS, 2) void k_contact_gjk(KArgs a) {
  const int lane = threadIdx.x & 63, gl = lane & (G - 1);
  size_t npairs = a.npairs;
  if (a.n_dev) npairs = min(npairs, (size_t)*a.n_dev);
  size_t lbase = 0, rbase = 0;
  if (a.range_b) {
    lbase = max(*a.range_b, a.part_lo);
    const size_t end = min(*a.range_e, a.part_hi);
    npairs = end > lbase ? end - lbase : 0;
    rbase = lbase - a.part_lo;
  }
  for (;;) {
    const size_t q = next_pairs<G>(a.work, lane);
    if (__ballot(q < npairs) == 0) break;
    bool epa_pair = false;
    uint32_t k = 0, kind = 0;
    Simplex s;
    if (q < npairs) {
      k = a.list ? a.list[lbase + q] : (uint32_t)q;
      const uint32_t i1 = a.ia[k], i2 = a.ib[k];
      if (i1 >= a.nshapes || i2 >= a.nshapes) {
        if (gl == 0) atomicOr(a.bad_index, 1u);
      } else {
        float pred;
        const Ctx2 c = contact_ctx(a, i1, i2, pred);
        // An all-zero init_dir means None for this pair (the reference's default direction).
        const f3 idir = load_init_dir(a, k);
        bool has_init = idir.x != 0.f || idir.y != 0.f || idir.z != 0.f;
        PairOut o;
        int extra_iters = 0;
        for (;;) {
          o = contact_pair<G>(c, pred, has_init, idir, a.P, gl, has_init ? a.max_iter : 10000, s, kind);
          if (o.has != 3) break;
          // a warm start that hit its iteration cap: plain GJK (init_dir = None) judges the pair
          extra_iters = o.gjk_iters;
          has_init = false;
        }
        epa_pair = o.has == 5;
        if (gl == 0) {
          if (a.iters) a.iters[k] = o.gjk_iters + extra_iters;
          if (!epa_pair) write_contact(a, k, o, idir);
        }
      }
    }
    const uint64_t em = __ballot(epa_pair && gl == 0);
    if (em) {
      uint32_t t = 0;
      const int first = __builtin_ctzll(em);
      if (lane == first) t = atomicAdd(a.rec_count, (uint32_t)__popcll(em));
      t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
      if (epa_pair && gl == 0) {
        float4* r = (float4*)(a.rec + rbase + t + (uint32_t)__popcll(em & ((1ull << lane) - 1ull)));
        r[0] = float4{__uint_as_float(k), __uint_as_float((uint32_t)s.dim | (kind << 2)), 0.f, 0.f};
        r[1] = float4{s.v0.o1.x, s.v0.o1.y, s.v0.o1.z, s.v0.o2.x};
        r[2] = float4{s.v0.o2.y, s.v0.o2.z, s.v1.o1.x, s.v1.o1.y};
        r[3] = float4{s.v1.o1.z, s.v1.o2.x, s.v1.o2.y, s.v1.o2.z};
        r[4] = float4{s.v2.o1.x, s.v2.o1.y, s.v2.o1.z, s.v2.o2.x};
        r[5] = float4{s.v2.o2.y, s.v2.o2.z, s.v3.o1.x, s.v3.o1.y};
        r[6] = float4{s.v3.o1.z, s.v3.o2.x, s.v3.o2.y, s.v3.o2.z};
      }
    }
  }
}

// The two support maps of a record's pair.
__device__ __forceinline__ Ctx2 epa_ctx(const KArgs& a, uint32_t k, uint32_t kind) {
  float pred;
  const Ctx2 c = contact_ctx(a, a.ia[k], a.ib[k], pred);
  if (kind == EPA_KIND_SM) return c;
  if (kind == EPA_KIND_BALL_FIRST) return ball_projection_ctx(c.m1.t, c.m2, c.g2);
  return ball_projection_ctx(c.m2.t, c.m1, c.g1);
}

// Completes pair k from its EPA run's points and normal (ok) or failure, as the path that started
// it does (contact_sm, contact_ball_convex), and writes it.
__device__ __forceinline__ void epa_write(const KArgs& a, uint32_t k, uint32_t kind, bool ok, f3 p1, f3 p2, f3 n) {
  PairOut o;
  pair_none(o);
  if (kind == EPA_KIND_SM) {
    if (ok) contact_sm_finish(o, p1, p2, n);
    else o.fdir = f3{1.f, 0.f, 0.f};  // NoIntersection(x_axis)
  } else {
    float pred;
    const Ctx2 c = contact_ctx(a, a.ia[k], a.ib[k], pred);
    const bool first = kind == EPA_KIND_BALL_FIRST;
    const f3 c1 = first ? c.m1.t : c.m2.t;
    ball_convex_finish(o, c1, first ? c.g1.a : c.g2.a, ok ? p1 + c1 : c1, true, true, f3{0.f, 0.f, 0.f}, pred);
    contact_flip(o, !first);
  }
  write_contact(a, k, o, load_init_dir(a, k));
}

// EPA records on LDS arenas (ncx_epa.h says what bounds them), BS threads per block in groups of G
// lanes, one record per group at a time.  Every pass of the loop runs one iteration of each group's record; groups without one take
// the next records together, with one atomic per wavefront, once REFILL of them wait or none runs.
// SAVES: a run about to outgrow the arena is saved for the next tier.  LISTED: the records come
// from the overflow list of the tier before (entries may be saved runs), otherwise those that the GJK
// launch of the same bucket wrote, from the place of its first pair in the part on.
template <int G, int BS, class L, int REFILL, bool SAVES, bool LISTED>
__global__ __launch_bounds__(BS, 1) void k_epa(KArgs a) {
  static_assert(ilog2_floor(L::HC) <= (uint32_t)G, "the heap steps need a lane per heap level");
  __shared__ __align__(16) uint8_t lds[(BS / G) * L::BYTES];
  const int lane = threadIdx.x & 63, gl = lane & (G - 1), gbase = lane & ~(G - 1);
  const uint64_t gmask = G == 64 ? ~0ull : ((1ull << (G & 63)) - 1ull);
  L A;
  A.p = lds + (threadIdx.x / G) * L::BYTES;
  float* const sup = a.sup + ((size_t)blockIdx.x * (BS / G) + threadIdx.x / G) * (6 * (size_t)L::VC);
  uint32_t n = LISTED ? min(*a.n_dev, a.ovf_cap) : *a.rec_count;
  const uint32_t rbase = !LISTED && a.range_b ? max(*a.range_b, a.part_lo) - a.part_lo : 0u;
  bool live = false, done = false;
  Ctx2 c;
  EpaState<L> s;
  uint32_t rec = 0, k = 0, kind = 0;
  int st = EPA_RUNNING;
  for (;;) {
    const uint64_t wm = __ballot(!live && !done && gl == 0), lm = __ballot(live);
    if ((wm | lm) == 0) break;
    if (wm && (lm == 0 || __popcll(wm) >= REFILL)) {
      uint32_t t = 0;
      const int first = __builtin_ctzll(wm);
      if (lane == first) t = atomicAdd(a.work, (uint32_t)__popcll(wm));
      t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
      if (!live && !done) {
        const uint32_t q = t + (uint32_t)__popcll(wm & ((1ull << gbase) - 1ull));
        if (q >= n) {
          done = true;
        } else {
          live = true;
          const uint32_t entry = LISTED ? a.list[q] : rbase + q;
          rec = entry & ~ENTRY_SAVED;
          const EpaRec* r = a.rec + rec;
          k = r->k;
          kind = r->dim_kind >> 2;
          c = epa_ctx(a, k, kind);
          if (LISTED && (entry & ENTRY_SAVED)) {
            epa_read_saved<G>(a.sus_load + (size_t)q * a.sus_load_bytes, A, sup, s, gl);
            st = EPA_RUNNING;
          } else {
            st = epa_begin<G>(A, r, sup, s, gl, gbase, gmask);
          }
        }
      }
    }
    if (live) {
      if (st == EPA_RUNNING) st = epa_step<G, L, SAVES>(A, c, a.P, sup, s, gl, gbase, gmask);
      if (st != EPA_RUNNING) {
        live = false;
        if (st == EPA_TOO_LARGE || st == EPA_SUSPEND) {
          uint32_t slot = 0;
          if (gl == 0) slot = atomicAdd(a.ovf_count, 1u);
          slot = (uint32_t)__shfl((int)slot, gbase, 64);
          bool saved = false;
          if constexpr (SAVES) {
            saved = st == EPA_SUSPEND && slot < a.sus_save_cap;
            if (saved) {
              __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
              epa_write_saved<G>(a.sus_save + (size_t)slot * a.sus_save_bytes, A, sup, s, gl);
            }
          }
          if (gl == 0 && slot < a.ovf_cap) a.ovf_list[slot] = a.ovf_pairs ? k : rec | (saved ? ENTRY_SAVED : 0u);
        } else if (gl == 0) {
          f3 p1 = f3{0.f, 0.f, 0.f}, p2 = p1, nn = f3{0.f, 1.f, 0.f};
          if (st == EPA_FACE) {
            // Face::closest_points with the barycentric coordinates new_with_proj stored (zero
            // unless the projection was inside the face)
            const typename L::W w = s.end;
            const float* q0 = sup + 6 * fld<L::BITS>(w, 0);
            const float* q1 = sup + 6 * fld<L::BITS>(w, 1);
            const float* q2 = sup + 6 * fld<L::BITS>(w, 2);
            const f3 a1 = f3{q0[0], q0[1], q0[2]}, a2 = f3{q0[3], q0[4], q0[5]};
            const f3 b1 = f3{q1[0], q1[1], q1[2]}, b2 = f3{q1[3], q1[4], q1[5]};
            const f3 c1 = f3{q2[0], q2[1], q2[2]}, c2 = f3{q2[3], q2[4], q2[5]};
            const f3 va = a1 - a2, vb = b1 - b2, vc = c1 - c2;
            Loc loc;
            proj_triangle(va, vb, vc, loc);
            float b0 = 0.f, b1c = 0.f, b2c = 0.f;
            if (loc.kind == LOC_FACE) { b0 = loc.bc0; b1c = loc.bc1; b2c = loc.bc2; }
            p1 = a1 * b0 + b1 * b1c + c1 * b2c;
            p2 = a2 * b0 + b2 * b1c + c2 * b2c;
            nn = tri_normal(va, vb, vc);
          }
          epa_write(a, k, kind, st != EPA_NOTHING, p1, p2, nn);
        }
      }
    }
  }
}

// EPA records on device-memory arenas (a.vcap, a.fcap), a wavefront per listed record.
__global__ __launch_bounds__(64, 1) void k_epa_global(KArgs a) {
  const int gl = threadIdx.x & 63;
  const size_t q = blockIdx.x;
  if (q >= a.npairs) return;
  const Arena A = arena_at(a.arena, q, a.vcap, a.fcap, a.fcap, 2 * a.fcap);
  const uint32_t entry = a.list[q], rec = entry & ~ENTRY_SAVED;
  const EpaRec* r = a.rec + rec;
  const uint32_t k = r->k, kind = r->dim_kind >> 2;
  const Ctx2 c = epa_ctx(a, k, kind);
  Simplex s;
  sx_init(s);
  s.dim = (int)(r->dim_kind & 3u);
  auto vertex = [&](int i) {
    CSO v;
    v.o1 = f3{r->v[i][0], r->v[i][1], r->v[i][2]};
    v.o2 = f3{r->v[i][3], r->v[i][4], r->v[i][5]};
    return v;
  };
  s.v0 = vertex(0);
  s.v1 = vertex(1);
  s.v2 = vertex(2);
  s.v3 = vertex(3);
  const uint8_t* load = (entry & ENTRY_SAVED) && a.sus_load ? a.sus_load + q * a.sus_load_bytes : nullptr;
  f3 p1, p2, n;
  int it;
  const int e = epa<64>(c, s, a.P, gl, A, p1, p2, n, it, load);
  if (gl != 0) return;
  if (e == EPA_OVERFLOW) {
    const uint32_t slot = atomicAdd(a.ovf_count, 1u);
    if (slot < a.ovf_cap) a.ovf_list[slot] = rec;
  } else {
    epa_write(a, k, kind, e == EPA_OK, p1, p2, n);
  }
}

// Distances (query::distance, distance.rs:9-33), BS threads per block in groups of G lanes, one
// pair per group at a time from the work counter.
template <int G, int BS>
__global__ __launch_bounds__(BS, 3) void k_distance(KArgs a) {
  const int gl = threadIdx.x & (G - 1);
  size_t npairs = a.npairs;
  size_t lbase = 0;
  if (a.range_b) {
    lbase = *a.range_b;
    npairs = *a.range_e - lbase;
  }
  for (;;) {
    uint32_t t = 0;
    if (gl == 0) t = atomicAdd(a.work, 1u);
    const size_t q = (uint32_t)__shfl((int)t, 0, G);
    if (q >= npairs) break;
    const size_t k = a.list ? a.list[lbase + q] : (uint32_t)q;
    const uint32_t i1 = a.ia[k], i2 = a.ib[k];
    if (i1 >= a.nshapes || i2 >= a.nshapes) {
      if (gl == 0) atomicOr(a.bad_index, 1u);
      continue;
    }
    Ctx2 c;
    c.g1 = load_shape(a.shapes, i1);
    c.g2 = load_shape(a.shapes, i2);
    c.m1 = load_pose(a.poses, i1);
    c.m2 = load_pose(a.poses, i2);
    float d = 0.f;
    int it = 0;
    if (c.g1.type == NCX_BALL && c.g2.type == NCX_BALL) {
      // distance_ball_ball (distance_ball_ball.rs:7-24)
      f3 delta = c.m2.t - c.m1.t;
      float d2 = norm_sq(delta);
      float sr = c.g1.a + c.g2.a;
      d = d2 <= sr * sr ? 0.f : __builtin_sqrtf(d2) - sr;
    } else {
      // distance_support_map_support_map_with_params (distance_support_map_support_map.rs:25-53)
      // init_dir (an all-zero entry means None) with GJK capped at max_iter; on the cap,
      // plain GJK from the default direction judges the pair.
      f3 d0 = c.m1.t - c.m2.t;
      const f3 idir = load_init_dir(a, k);
      bool warm = idir.x != 0.f || idir.y != 0.f || idir.z != 0.f;
      if (warm) d0 = idir;
      for (int pass = 0; pass < 2; ++pass) {
        f3 dir;
        float nl;
        if (!try_normalize(d0, NCX_FLT_EPS, &dir, &nl)) dir = f3{1.f, 0.f, 0.f};
        Simplex s;
        GJKOut r = gjk<G, false, 8>(c, dir, NCX_FLT_MAX, s, a.P, gl, warm ? a.max_iter : 10000);
        it += r.iters;
        if (warm && r.status == GJK_S_CAP && a.max_iter < 10000) {
          warm = false;
          d0 = c.m1.t - c.m2.t;
          continue;
        }
        d = r.status == GJK_S_CLOSEST ? norm(r.p1 - r.p2) : 0.f;
        break;
      }
    }
    if (gl == 0) {
      a.dist[k] = d;
      if (a.iters) a.iters[k] = it;
    }
  }
}

// The same with one pair a lane, the lanes of a group of DW_G scanning each other's hulls in turn.
// What bounds k_distance on hulls: two thirds of its VALU slots are taken, three quarters of them by
// the simplex's projection and reduction, which every lane of a group repeats for the one pair; and
// the scans' loads, which the second-level cache serves.  Here a lane projects its own pair's simplex
// and only the scans are shared, so that both are done once a pair; the loads still come 8 lanes at a
// time from one hull.  262,144 hull pairs of up to 256 vertices, whole batch: 2.37 ms in groups,
// 1.76 ms so (groups of 4 and 16: 2.1 and 1.78 ms; a wavefront's lanes that wait for new pairs at 4
// or 16 idle ones, the same).  It needs 64 pairs a wavefront to pay, so the autotuner chooses it or a
// group's kernel for each vertex-count bucket by timing both on a sample, for batches that fill the
// chip (bucket_variant).
#define DW_G 8
#define DW_REFILL 16  // idle lanes before the wavefront takes more pairs
template <int BS>
__global__ __launch_bounds__(BS, 2) void k_distance_wave(KArgs a) {
  const int lane = __lane_id();
  size_t npairs = a.npairs;
  size_t lbase = 0;
  if (a.range_b) {
    lbase = *a.range_b;
    npairs = *a.range_e - lbase;
  }
  bool live = false, done = false, warm = false;
  size_t k = 0;
  int it = 0;
  Ctx2 c = {};
  Simplex s;
  GJKRun g;
  GJKOut r;
  g.dir = f3{0.f, 0.f, 0.f};
  auto begin = [&](f3 d0) {
    f3 dir;
    float nl;
    if (!try_normalize(d0, NCX_FLT_EPS, &dir, &nl)) dir = f3{1.f, 0.f, 0.f};
    gjk_begin(g, s, r, dir);
  };
  auto write = [&](float d) {
    a.dist[k] = d;
    if (a.iters) a.iters[k] = it;
  };
  for (;;) {
    const uint64_t idle = __ballot(!live && !done), lm = __ballot(live);
    if ((idle | lm) == 0) break;
    if (idle && (lm == 0 || __popcll(idle) >= DW_REFILL)) {
      uint32_t t = 0;
      const int first = __builtin_ctzll(idle);
      if (lane == first) t = atomicAdd(a.work, (uint32_t)__popcll(idle));
      t = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
      if (!live && !done) {
        const size_t q = (size_t)t + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
        if (q >= npairs) {
          done = true;
        } else {
          k = a.list ? a.list[lbase + q] : (uint32_t)q;
          const uint32_t i1 = a.ia[k], i2 = a.ib[k];
          if (i1 >= a.nshapes || i2 >= a.nshapes) {
            atomicOr(a.bad_index, 1u);
          } else {
            c.g1 = load_shape(a.shapes, i1);
            c.g2 = load_shape(a.shapes, i2);
            c.m1 = load_pose(a.poses, i1);
            c.m2 = load_pose(a.poses, i2);
            it = 0;
            f3 d0 = c.m1.t - c.m2.t;
            if (c.g1.type == NCX_BALL && c.g2.type == NCX_BALL) {
              const float d2 = norm_sq(c.m2.t - c.m1.t), sr = c.g1.a + c.g2.a;
              write(d2 <= sr * sr ? 0.f : __builtin_sqrtf(d2) - sr);
            } else {
              const f3 idir = load_init_dir(a, k);
              warm = idir.x != 0.f || idir.y != 0.f || idir.z != 0.f;
              if (warm) d0 = idir;
              begin(d0);
              live = true;
            }
          }
        }
      }
    }
    if (__ballot(live) == 0) continue;
    const CSO cso = cso_wave<DW_G>(c, g.dir, a.P, live);
    if (live && gjk_step<false>(g, s, cso, NCX_FLT_MAX, warm ? a.max_iter : 10000, r)) {
      it += r.iters;
      if (warm && r.status == GJK_S_CAP && a.max_iter < 10000) {
        warm = false;
        begin(c.m1.t - c.m2.t);
      } else {
        write(r.status == GJK_S_CLOSEST ? norm(r.p1 - r.p2) : 0.f);
        live = false;
      }
    }
  }
}

// ------------------------------------------------------------------ host side
// Vertex-count bucket of the larger hull vertex count m of a pair (0: no hull).
__host__ __device__ __forceinline__ uint32_t count_bucket(uint32_t m) {
  return m == 0 ? 0u : (m <= 32 ? 1u : (m <= 96 ? 2u : 3u));
}
__global__ void k_shape_radius(ncx_shape* __restrict__ shapes, size_t n, Pool P);

extern "C" int ncx_shapes_create(ncx_ctx* ctx, const ncx_shape* shapes, size_t n, const float* hx, const float* hy,
                                 const float* hz, size_t npts, ncx_shapes** out) {
  NCX_REQUIRE(ctx && out && (shapes || n == 0), "ncx_shapes_create: null argument");
  for (size_t i = 0; i < n; ++i) {
    const ncx_shape& s = shapes[i];
    NCX_REQUIRE(s.type <= NCX_CONVEX_HULL, "ncx_shapes_create: unknown shape type");
    if (s.type == NCX_CONVEX_HULL)
      NCX_REQUIRE(s.hull_count > 0 && (size_t)s.hull_offset + s.hull_count <= npts,
                  "ncx_shapes_create: hull range outside the point pool");
  }
  ncx_shapes* S = new ncx_shapes;
  S->buckets = n ? 0u : 1u;  // a set without shapes: the launch that finds every pair's index bad
  for (size_t i = 0; i < n; ++i) S->types |= 1u << shapes[i].type;
  for (size_t i = 0; i < n; ++i)
    S->buckets |= 1u << (shapes[i].type == NCX_CONVEX_HULL ? count_bucket(shapes[i].hull_count) : 0u);
  S->ctx = ctx;
  S->n = n;
  S->npts = npts;
  int rc;
  if ((rc = S->shapes.reserve(n * sizeof(ncx_shape) + 64)) || (rc = S->hx.reserve(npts * 4 + 4)) ||
      (rc = S->hy.reserve(npts * 4 + 4)) || (rc = S->hz.reserve(npts * 4 + 4)) || (rc = contact_tiers_reserve(S->tiers, ctx, 4096, 4096))) {
    delete S;
    return rc;
  }
  if (n) NCX_HIP_CHECK(hipMemcpyAsync(S->shapes.p, shapes, n * sizeof(ncx_shape), hipMemcpyHostToDevice, ctx->stream));
  if (npts) {
    NCX_HIP_CHECK(hipMemcpyAsync(S->hx.p, hx, npts * 4, hipMemcpyHostToDevice, ctx->stream));
    NCX_HIP_CHECK(hipMemcpyAsync(S->hy.p, hy, npts * 4, hipMemcpyHostToDevice, ctx->stream));
    NCX_HIP_CHECK(hipMemcpyAsync(S->hz.p, hz, npts * 4, hipMemcpyHostToDevice, ctx->stream));
  }
  if (n) {
    hipLaunchKernelGGL(k_shape_radius, dim3(ceil_div(n, 256)), dim3(256), 0, ctx->stream, S->shapes.as<ncx_shape>(), n,
                       Pool{S->hx.as<float>(), S->hy.as<float>(), S->hz.as<float>(), S->tri});
    NCX_HIP_CHECK(hipGetLastError());
  }
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  *out = S;
  return NCX_OK;
}

extern "C" int ncx_shapes_destroy(ncx_shapes* s) {
  if (!s) return NCX_OK;
  s->shapes.release(); s->hx.release(); s->hy.release(); s->hz.release(); contact_tiers_release(s->tiers);
  s->qerr.release();
  s->hf_shape.release(); s->hf_fn.release(); s->hf_floop.release(); s->hf_loop.release();
  s->hf_edir.release(); s->hf_ev.release(); s->hf_vadj.release(); s->hf_adj.release();
  delete s;
  return NCX_OK;
}

// The autotuner's state for one query (0 contact, 1 distance): per vertex-count bucket the
// chosen variant (T1_VARIANT_G; -1 untuned) and each variant's sample time.
extern "C" int ncx_shapes_tuning(ncx_shapes* s, int query, int32_t* choice, float* sample_ms) {
  NCX_REQUIRE(s && choice && (query == 0 || query == 1), "ncx_shapes_tuning: bad argument");
  for (int b = 0; b < NCX_NBUCKETS; ++b) {
    choice[b] = s->tune[query][b];
    if (sample_ms)
      for (int v = 0; v < NCX_T1_VARIANTS; ++v) sample_ms[NCX_T1_VARIANTS * b + v] = s->tune_ms[query][b][v];
  }
  return NCX_OK;
}

extern "C" int ncx_shapes_count(ncx_shapes* s, size_t* n) {
  NCX_REQUIRE(s && n, "ncx_shapes_count: null argument");
  *n = s->n;
  return NCX_OK;
}

// ------------------------------------------------------------------ vertex-count buckets
// Sort key of a pair: its vertex-count bucket (by the larger hull vertex count of its shapes: 0 no
// hull, 1 up to 32, 2 up to 96, 3 more; pairs of one bucket have similar support-scan costs and
// get one kernel variant) times 128, plus 8 x its pair of shape types, plus an overlap bin:
// floor(8 x centre distance / (sum of the shapes' bounding radii)), at most 7.  Pairs of one
// type pair take the same dispatch branch, and pairs of one bin are about as likely to need EPA
// (on a 1M-shape scene: bins 0-2 ~100% penetrating, 4: 80%, 6: 31%, 8 and up: none), so the groups
// of a wavefront stay on one code path.  On that scene's 10.2 M pairs contacts took 144 ms in
// their own order, 133 ms sorted by type pair, 121 ms by type pair and bin.  The radius of shape i
// is kept in its record's pad[0] (ncx_shapes_create).
__device__ __forceinline__ uint32_t pair_key(const ncx_shape* __restrict__ shapes, uint32_t nshapes,
                                             const ncx_pose* __restrict__ poses, uint32_t i1, uint32_t i2,
                                             uint32_t bad_key) {
  if (i1 >= nshapes || i2 >= nshapes) return bad_key;  // the pair kernel reports the bad index
  const ncx_shape s1 = shapes[i1], s2 = shapes[i2];
  uint32_t c1 = s1.type == NCX_CONVEX_HULL ? s1.hull_count : 0;
  uint32_t c2 = s2.type == NCX_CONVEX_HULL ? s2.hull_count : 0;
  uint32_t m = c1 > c2 ? c1 : c2;
  const uint32_t b = count_bucket(m);
  uint32_t t1 = s1.type < 3u ? s1.type : 3u, t2 = s2.type < 3u ? s2.type : 3u;
  const float dx = poses[i1].tx - poses[i2].tx, dy = poses[i1].ty - poses[i2].ty, dz = poses[i1].tz - poses[i2].tz;
  const float rs = __uint_as_float(s1.pad[0]) + __uint_as_float(s2.pad[0]);
  const float bin = (float)NCX_OVERLAP_BINS * __builtin_sqrtf(dx * dx + dy * dy + dz * dz) / rs;
  const uint32_t o = bin < (float)(NCX_OVERLAP_BINS - 1) ? (uint32_t)bin : NCX_OVERLAP_BINS - 1;  // NaN and large: last bin
  return 16u * NCX_OVERLAP_BINS * b + NCX_OVERLAP_BINS * (4u * (t1 < t2 ? t1 : t2) + (t1 < t2 ? t2 : t1)) + o;
}

// Bounding radius of each shape about its local origin, into pad[0] of its device record, for the
// sort key.
__global__ __launch_bounds__(256) void k_shape_radius(ncx_shape* __restrict__ shapes, size_t n, Pool P) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const ncx_shape s = shapes[i];
  float r = 0.f;
  if (s.type == NCX_BALL) r = fabsf(s.p0);
  else if (s.type == NCX_CUBOID) r = __builtin_sqrtf(s.p0 * s.p0 + s.p1 * s.p1 + s.p2 * s.p2);
  else if (s.type == NCX_CAPSULE) r = fabsf(s.p0) + fabsf(s.p1);
  else {
    for (uint32_t k = 0; k < s.hull_count; ++k) {
      const uint32_t j = s.hull_offset + k;
      r = fmaxf(r, P.x[j] * P.x[j] + P.y[j] * P.y[j] + P.z[j] * P.z[j]);
    }
    r = __builtin_sqrtf(r);
  }
  shapes[i].pad[0] = __float_as_uint(r);
}

#define BKT_BLOCK 256
#define BKT_ITEMS 8

// Pass 1: each pair's key, and per-key counts (LDS histogram per block, one atomic per key per
// block).
__global__ __launch_bounds__(BKT_BLOCK) void k_bucket_count(const uint32_t* __restrict__ ia,
                                                            const uint32_t* __restrict__ ib,
                                                            const ncx_shape* __restrict__ shapes, uint32_t nshapes,
                                                            const ncx_pose* __restrict__ poses, size_t npairs,
                                                            const uint32_t* __restrict__ n_dev,
                                                            uint32_t* __restrict__ hdr, uint32_t* __restrict__ keys,
                                                            uint32_t bad_key) {
  __shared__ uint32_t h[NCX_NKEYS];
  for (uint32_t k = threadIdx.x; k < NCX_NKEYS; k += BKT_BLOCK) h[k] = 0;
  __syncthreads();
  size_t n = npairs;
  if (n_dev) n = min(n, (size_t)*n_dev);
  const size_t base = (size_t)blockIdx.x * BKT_BLOCK * BKT_ITEMS;
  for (int r = 0; r < BKT_ITEMS; ++r) {
    size_t q = base + (size_t)r * BKT_BLOCK + threadIdx.x;
    if (q < n) {
      const uint32_t key = pair_key(shapes, nshapes, poses, ia[q], ib[q], bad_key);
      keys[q] = key;
      atomicAdd(&h[key], 1u);
    }
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < NCX_NKEYS; k += BKT_BLOCK)
    if (h[k]) atomicAdd(&hdr[NCX_KEY_CNT + k], h[k]);
}

// Key offsets (the scatter cursors) and each bucket's range [begin, end) in the partitioned list:
// one thread per key, an inclusive scan in LDS (one thread over all keys took 20 us).
__global__ __launch_bounds__(NCX_NKEYS) void k_bucket_offsets(uint32_t* __restrict__ hdr) {
  constexpr uint32_t per_bucket = NCX_NKEYS / NCX_NBUCKETS;
  __shared__ uint32_t sum[NCX_NKEYS];
  const uint32_t key = threadIdx.x, c = hdr[NCX_KEY_CNT + key];
  uint32_t x = c;
  sum[key] = x;
  for (uint32_t o = 1; o < NCX_NKEYS; o *= 2) {
    __syncthreads();
    const uint32_t y = key >= o ? sum[key - o] : 0u;
    __syncthreads();
    x += y;
    sum[key] = x;
  }
  hdr[NCX_KEY_FILL + key] = x - c;
  if (key % per_bucket == 0) hdr[NCX_BKT_RANGE + 2 * (key / per_bucket)] = x - c;
  if (key % per_bucket == per_bucket - 1) hdr[NCX_BKT_RANGE + 2 * (key / per_bucket) + 1] = x;
}

// Pass 2: scatter pair indices to their key's range (one atomic per key per block for the
// block's base, LDS atomics within the block).
__global__ __launch_bounds__(BKT_BLOCK) void k_bucket_scatter(const uint32_t* __restrict__ keys, size_t npairs,
                                                              const uint32_t* __restrict__ n_dev,
                                                              uint32_t* __restrict__ hdr, uint32_t* __restrict__ list) {
  __shared__ uint32_t h[NCX_NKEYS], bb[NCX_NKEYS];
  for (uint32_t k = threadIdx.x; k < NCX_NKEYS; k += BKT_BLOCK) h[k] = 0;
  __syncthreads();
  size_t n = npairs;
  if (n_dev) n = min(n, (size_t)*n_dev);
  const size_t base = (size_t)blockIdx.x * BKT_BLOCK * BKT_ITEMS;
  uint32_t mine[BKT_ITEMS];
#pragma unroll
  for (int r = 0; r < BKT_ITEMS; ++r) {
    size_t q = base + (size_t)r * BKT_BLOCK + threadIdx.x;
    mine[r] = q < n ? keys[q] : 0xFFFFFFFFu;
    if (mine[r] != 0xFFFFFFFFu) atomicAdd(&h[mine[r]], 1u);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < NCX_NKEYS; k += BKT_BLOCK) {
    bb[k] = h[k] ? atomicAdd(&hdr[NCX_KEY_FILL + k], h[k]) : 0u;
    h[k] = 0;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < BKT_ITEMS; ++r) {
    if (mine[r] == 0xFFFFFFFFu) continue;
    size_t q = base + (size_t)r * BKT_BLOCK + threadIdx.x;
    list[bb[mine[r]] + atomicAdd(&h[mine[r]], 1u)] = (uint32_t)q;
  }
}

// Arena tiers, all but the last in LDS and in the graph:
//   T1: 8 records per block (8, 16 or 32 lanes each, the autotuner's choice), arenas of 44 or 24
//       vertices (3.3 and 1.9 KB; 6 or 11 blocks fit a CU);
//   T2: 16 lanes, 4 records per 64-thread block, 64 vertices (5.0 KB);
//   T3: 64 lanes, one record per block, 256 vertices (20 KB);
//   T4: 64 lanes, one record per block, 2000 vertices (132 KB, one block per CU);
//   then device-memory arenas 8x larger than T4's, 64 lanes per record, host-driven.

// Saved-run slots handed from each LDS tier to the next (the first SUS_CAP[t] suspended runs of
// a launch are saved; later ones start again in the next tier) and their sizes.  The first tier's
// are at most one for 32 pairs.  About one run in ten takes more than 20 iterations (12 on average)
// on a scene of mixed shapes, so runs started again would cost the second tier three times the
// iterations that continued ones do.
static const uint32_t SUS_CAP[4] = {1u << 19, 4096, 1024, 256};
static const size_t SUS_BYTES[4] = {epa_save_bytes(ArenaT1::VC, ArenaT1::HC), epa_save_bytes(ArenaT2::VC, ArenaT2::HC),
                                    epa_save_bytes(ArenaT3::VC, ArenaT3::HC), epa_save_bytes(ArenaT4::VC, ArenaT4::HC)};
static_assert(ArenaT1::FC + 2 <= ArenaT1::HC && ArenaT1S::HC <= ArenaT1::HC, "a saved run's faces");
static_assert(ArenaT2::FC + 2 <= ArenaT2::HC && ArenaT3::FC + 2 <= ArenaT3::HC && ArenaT4::FC + 2 <= ArenaT4::HC,
              "a saved run's faces");

// Records of a launch: for one of more pairs it goes over them in parts.  A part of 2^26 pairs has
// 7.5 GB of records; fewer where that much memory cannot be had, down to REC_LEAST (15 MB).  A part
// costs about 0.3 ms also where a scene has no pairs for it (three parts of 2^24 pairs: a step of a
// 1,048,576-shape scene with room for 42 M pairs 42.0 -> 42.7 ms).
static const size_t REC_MOST = (size_t)1 << 26, REC_LEAST = (size_t)1 << 17;

// Overflow lists of at least cap entries each (at most 2^24: a call with more overflowing pairs
// fails with NCX_E_CAPACITY), the saved-run slots, and EPA records for nrec pairs (0: none, for
// distances).
int contact_tiers_reserve(ContactTiers& t, ncx_ctx* ctx, size_t cap, size_t nrec) {
  nrec = std::min(nrec, REC_MOST);
  if (nrec > t.nrec && nrec > t.rec_asked) {
    // one allocation: support points, records, the first tier's saved runs; a quarter more than there
    // were, so that batches that grow a little from call to call seldom come here
    const size_t sup = (size_t)ctx->num_cus * EPA_SUP_FLOATS_PER_CU * 4, asked = nrec;
    nrec = std::min(std::max(nrec, t.nrec + t.nrec / 4), REC_MOST);
    t.epa.release();
    t.nrec = t.rec_asked = 0;
    for (;;) {
      const size_t slots = std::min<size_t>(SUS_CAP[0], nrec / 32);
      const int rc = t.epa.reserve(sup + nrec * sizeof(EpaRec) + slots * SUS_BYTES[0]);
      if (!rc) {
        t.sus0_cap = (uint32_t)slots;
        break;
      }
      if (nrec <= REC_LEAST) return rc;
      nrec = std::max(nrec / 2, REC_LEAST);
    }
    t.nrec = nrec;
    t.rec_asked = asked;
    t.sup = t.epa.as<float>();
    t.rec = (EpaRec*)(t.epa.as<uint8_t>() + sup);
    t.sus0 = (uint8_t*)(t.rec + nrec);
  }
  for (int i = 0; i < 3; ++i) {
    if (t.sus[i].p) continue;
    int rc = t.sus[i].reserve((size_t)SUS_CAP[i + 1] * SUS_BYTES[i + 1]);
    if (rc) return rc;
  }
  cap = std::min<size_t>(std::max<size_t>(cap, 4096), (size_t)1 << 24);
  if (cap <= t.cap) return NCX_OK;
  // the present lists stay where larger ones cannot be had: later calls, the queries without
  // overflows among them, use the header
  DevBuf lists;
  int rc = lists.reserve(4 * (NCX_OVF_HEADER + 4 * cap));
  if (rc) return rc;
  t.ovf.release();
  t.ovf = lists;
  t.cap = (uint32_t)cap;
  return NCX_OK;
}

void contact_tiers_release(ContactTiers& t) {
  t.ovf.release();
  t.blist.release();
  t.bkey.release();
  t.epa.release();
  t.nrec = t.rec_asked = 0;
  t.bcap = 0;
  t.cap = 0;
  t.sus0_cap = 0;
  for (int i = 0; i < 3; ++i) t.sus[i].release();
  delete t.last;
  t.last = nullptr;
}

__global__ void k_iota_u32(uint32_t* __restrict__ p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

// Re-runs the n records listed at list_src (device; null: the first n) with device-memory arenas 8x
// larger per round (starting from 8 x the last tier's vcap/fcap) until none overflows; host-driven
// (synchronises the stream).  Chunks keep each round's arenas <= 2 GiB.  The first round continues the runs
// the last LDS tier saved (sus_src, slot = list position); device-memory rounds do not suspend.
static int rerun_overflows(ContactTiers& T, ncx_ctx* ctx, KArgs a, uint32_t n, const uint32_t* list_src,
                           uint32_t vcap, uint32_t fcap, const uint8_t* sus_src, size_t sus_bytes) {
  if (n == 0) return NCX_OK;
  uint32_t* ovf = T.ovf.as<uint32_t>();
  DevBuf lst;
  int rc;
  if ((rc = lst.reserve((size_t)n * 4))) return rc;
  if (list_src) {
    NCX_HIP_CHECK(hipMemcpyAsync(lst.p, list_src, (size_t)n * 4, hipMemcpyDeviceToDevice, ctx->stream));
  } else {
    hipLaunchKernelGGL(k_iota_u32, dim3(ceil_div(n, 256)), dim3(256), 0, ctx->stream, lst.as<uint32_t>(), n);
    NCX_HIP_CHECK(hipGetLastError());
  }
  while (n > 0) {
    vcap *= 8;
    fcap *= 8;
    if (fcap > 65535) fcap = 65535;
    if (vcap > 32767) vcap = 32767;
    const size_t per = arena_bytes(vcap, fcap);
    const size_t chunk = std::max<size_t>(1, ((size_t)2 << 30) / per);
    DevBuf big;
    if ((rc = big.reserve(std::min<size_t>(n, chunk) * per))) return rc;
    if ((rc = fill_u32(ctx, ovf + NCX_OVF_T2_COUNT, 1, 0u))) return rc;
    for (size_t off = 0; off < n; off += chunk) {
      size_t m = std::min<size_t>(chunk, n - off);
      KArgs b = a;
      b.list = lst.as<uint32_t>() + off;
      b.n_dev = nullptr;
      b.arena = big.as<uint8_t>();
      b.vcap = vcap;
      b.fcap = fcap;
      b.ovf_count = ovf + NCX_OVF_T2_COUNT;
      b.ovf_list = T.t2_list();
      b.ovf_cap = T.cap;
      b.sus_load = sus_src ? sus_src + off * sus_bytes : nullptr;
      b.sus_load_bytes = sus_bytes;
      b.npairs = m;
      hipLaunchKernelGGL(k_epa_global, dim3((unsigned)m), dim3(64), 0, ctx->stream, b);
      NCX_HIP_CHECK(hipGetLastError());
    }
    sus_src = nullptr;  // later rounds list this tier's own overflows, with nothing saved
    uint32_t left = 0;
    NCX_HIP_CHECK(hipMemcpyAsync(&left, ovf + NCX_OVF_T2_COUNT, 4, hipMemcpyDeviceToHost, ctx->stream));
    NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    big.release();
    if (left) NCX_REQUIRE(fcap < 65535, "contact batch: EPA polytope exceeds 65535 faces");
    n = left;
    if (n) {
      NCX_REQUIRE(n <= T.cap, "contact batch: too many EPA arena overflows");
      NCX_HIP_CHECK(hipMemcpyAsync(lst.p, T.t2_list(), (size_t)n * 4, hipMemcpyDeviceToDevice,
                                   ctx->stream));
    }
  }
  return NCX_OK;
}

// First-tier kernel variants, the autotuner's choices.  Contact: EPA with G = 8, 16, 32 lanes per
// record on the 44-vertex arena (variants 0-2), and G = 8, 16 on the 24-vertex arena (variants
// 3-4); every variant holds 8 records per block.  The small arena's hold more records per CU and
// send more of them to the second tier, which the tuner times with them.  Distance queries have no
// arena: 128-thread variants with 8, 16, 32 or 4 lanes per pair, and one pair a lane (variant 4).
static const int T1_NVARIANTS[2] = {NCX_T1_VARIANTS, NCX_T1_VARIANTS};
static const int T1_VARIANT_G[2][NCX_T1_VARIANTS] = {{8, 16, 32, 8, 16}, {8, 16, 32, 4, 1}};
static const int T1_VARIANT_BS[2][NCX_T1_VARIANTS] = {{64, 128, 256, 64, 128}, {128, 128, 128, 128, 128}};
// contact: the resident blocks (LDS); distance: twice the resident blocks (VGPRs: 8 waves), or they
static const unsigned T1_BLOCKS_PER_CU[2][NCX_T1_VARIANTS] = {{T1_BLOCKS, T1_BLOCKS, T1_BLOCKS, T1S_BLOCKS, T1S_BLOCKS},
                                                               {8, 8, 8, 8, 4}};
// Lanes per pair of the GJK kernel by vertex-count bucket: without hulls the supports are closed
// forms and a group's lanes would only repeat each other.
static const int GJK_BUCKET_G[NCX_NBUCKETS] = {1, 4, 4, 8};
#define GJK_BLOCKS_PER_CU 4u
#define GJK_SMALL_G 8  // batches too small to partition

extern "C" int ncx_shapes_set_tuning(ncx_shapes* s, int query, const int32_t* choice) {
  NCX_REQUIRE(s && choice && (query == 0 || query == 1), "ncx_shapes_set_tuning: bad argument");
  for (int b = 0; b < NCX_NBUCKETS; ++b)
    NCX_REQUIRE(choice[b] >= -1 && choice[b] < T1_NVARIANTS[query], "ncx_shapes_set_tuning: no such variant");
  for (int b = 0; b < NCX_NBUCKETS; ++b) s->tune[query][b] = (int8_t)choice[b];
  return NCX_OK;
}

// The variant of a batch's pairs of one bucket.  The tuner's samples are large; one pair a lane needs
// enough pairs to fill the chip (distances, 8 lanes a pair or the best other variant against one
// pair a lane: 300 pairs of 256-vertex hulls 65 and 186 us, 16,384 185 and 287; 16,384 of 64-vertex
// hulls 110 and 148, of mixed shapes 129 and 154; 32,768 of mixed shapes 167 and 174, 65,536 204 and
// 184 us), so that smaller batches take the fastest of the others on the samples, and those too
// small to partition 8 lanes a pair.
#define DW_VARIANT 4
#define DW_MIN_PAIRS 32768u
static int bucket_variant(const ncx_shapes* S, int mode, int b, size_t npairs) {
  const int v = S->tune[mode][b] >= 0 ? S->tune[mode][b] : 1;
  if (mode == 0 || v != DW_VARIANT || npairs >= DW_MIN_PAIRS) return v;
  int best = 0;
  if (npairs >= NCX_PARTITION_MIN_PAIRS)
    for (int u = 1; u < DW_VARIANT; ++u)
      if (S->tune_ms[mode][b][u] > 0.f && S->tune_ms[mode][b][u] < S->tune_ms[mode][b][best]) best = u;
  return best;
}

static unsigned capped_blocks(ncx_ctx* ctx, unsigned per_cu, size_t n, size_t per_block) {
  return (unsigned)std::max<size_t>(1, std::min<size_t>((size_t)ctx->num_cus * per_cu, (n + per_block - 1) / per_block));
}

static int launch_distance(int variant, ncx_ctx* ctx, const KArgs& a, size_t n) {
  const unsigned blocks = capped_blocks(ctx, T1_BLOCKS_PER_CU[1][variant], n,
                                        (size_t)T1_VARIANT_BS[1][variant] / T1_VARIANT_G[1][variant]);
  switch (variant) {
    case 0: hipLaunchKernelGGL((k_distance<8, 128>), dim3(blocks), dim3(128), 0, ctx->stream, a); break;
    case 2: hipLaunchKernelGGL((k_distance<32, 128>), dim3(blocks), dim3(128), 0, ctx->stream, a); break;
    case 3: hipLaunchKernelGGL((k_distance<4, 128>), dim3(blocks), dim3(128), 0, ctx->stream, a); break;
    case 4: hipLaunchKernelGGL((k_distance_wave<128>), dim3(blocks), dim3(128), 0, ctx->stream, a); break;
    default: hipLaunchKernelGGL((k_distance<16, 128>), dim3(blocks), dim3(128), 0, ctx->stream, a); break;
  }
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}

// GJK over at most n pairs with G lanes each, then the first-tier EPA variant over its records
// (work counters `work` and `epa_work`).
static int launch_contact_t1(int variant, int G, ncx_ctx* ctx, const KArgs& a, size_t n, uint32_t* work,
                             uint32_t* epa_work) {
  KArgs g = a;
  g.work = work;
  const unsigned gb = capped_blocks(ctx, GJK_BLOCKS_PER_CU, n, GJK_BS / G);
  switch (G) {
    case 1: hipLaunchKernelGGL(k_contact_gjk<1>, dim3(gb), dim3(GJK_BS), 0, ctx->stream, g); break;
    case 4: hipLaunchKernelGGL(k_contact_gjk<4>, dim3(gb), dim3(GJK_BS), 0, ctx->stream, g); break;
    default: hipLaunchKernelGGL(k_contact_gjk<8>, dim3(gb), dim3(GJK_BS), 0, ctx->stream, g); break;
  }
  NCX_HIP_CHECK(hipGetLastError());
  KArgs e = a;
  e.work = epa_work;
  const unsigned eb = capped_blocks(ctx, T1_BLOCKS_PER_CU[0][variant], n, 8);
  const dim3 bs(T1_VARIANT_BS[0][variant]);
  switch (variant) {
    case 0: hipLaunchKernelGGL((k_epa<8, 64, ArenaT1, 2, true, false>), dim3(eb), bs, 0, ctx->stream, e); break;
    case 2: hipLaunchKernelGGL((k_epa<32, 256, ArenaT1, 1, true, false>), dim3(eb), bs, 0, ctx->stream, e); break;
    case 3: hipLaunchKernelGGL((k_epa<8, 64, ArenaT1S, 2, true, false>), dim3(eb), bs, 0, ctx->stream, e); break;
    case 4: hipLaunchKernelGGL((k_epa<16, 128, ArenaT1S, 2, true, false>), dim3(eb), bs, 0, ctx->stream, e); break;
    default: hipLaunchKernelGGL((k_epa<16, 128, ArenaT1, 2, true, false>), dim3(eb), bs, 0, ctx->stream, e); break;
  }
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}

// Saved-run buffers of LDS tier `tier` (0 = T1): it continues the runs T(tier) saved and saves
// its own suspended runs for the next tier.
static uint8_t* sus_slots(const ContactTiers& T, int tier) { return tier == 0 ? T.sus0 : T.sus[tier - 1].as<uint8_t>(); }

static void set_sus(ContactTiers& T, KArgs& b, int tier) {
  b.sus_load = tier > 0 ? sus_slots(T, tier - 1) : nullptr;
  b.sus_load_bytes = tier > 0 ? SUS_BYTES[tier - 1] : 0;
  b.sus_save = sus_slots(T, tier);
  b.sus_save_bytes = SUS_BYTES[tier];
  b.sus_save_cap = tier == 0 ? T.sus0_cap : SUS_CAP[tier];
}

// Tier t (1 = T2, ...) over the device-counted overflow list of the tier before it.
static KArgs tier_args(ContactTiers& T, const KArgs& a, int t) {
  uint32_t* ovf = T.ovf.as<uint32_t>();
  uint32_t* const counts[4] = {ovf + NCX_OVF_T1_COUNT, ovf + NCX_OVF_T2_COUNT, ovf + NCX_OVF_T3_COUNT,
                               ovf + NCX_OVF_T4_COUNT};
  uint32_t* const lists[4] = {T.t1_list(), T.t2_list(), T.t3_list(), T.t4_list()};
  const uint32_t works[4] = {0, NCX_WORK_T2, NCX_WORK_T3, NCX_WORK_T4};
  KArgs b = a;
  b.range_b = nullptr;
  b.range_e = nullptr;
  b.list = lists[t - 1];
  b.n_dev = counts[t - 1];
  b.ovf_count = counts[t];
  b.ovf_list = lists[t];
  b.work = ncx_work_set(ovf, works[t]);
  set_sus(T, b, t);
  if (t == 3 && T.parts) {  // the next part takes the records: contacts_resolve_overflow makes them again
    b.ovf_pairs = 1;
    b.sus_save_cap = 0;
  }
  return b;
}

// T2 to T4 after the first tier of about n pairs.  The grids are persistent, so any size is right:
// about one pair in twenty is taken to reach T2, one in 400 T3 and one in 4,000 T4, because the
// blocks of an empty launch cost time too (16 us for 1,280 blocks of 30 KB).
static int launch_upper_tiers(ncx_ctx* ctx, ContactTiers& T, const KArgs& a, size_t n) {
  hipLaunchKernelGGL((k_epa<T2_G, T2_BS, ArenaT2, 2, true, true>),
                     dim3(capped_blocks(ctx, T2_BLOCKS_PER_CU, n, 20 * (T2_BS / T2_G))), dim3(T2_BS), 0, ctx->stream,
                     tier_args(T, a, 1));
  NCX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL((k_epa<64, 64, ArenaT3, 1, true, true>), dim3(capped_blocks(ctx, T3_BLOCKS_PER_CU, n, 400)), dim3(64),
                     0, ctx->stream, tier_args(T, a, 2));
  NCX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL((k_epa<64, 64, ArenaT4, 1, true, true>), dim3(capped_blocks(ctx, 1u, n, 4000)), dim3(64), 0,
                     ctx->stream, tier_args(T, a, 3));
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}

int contact_tiers_reserve_list(ContactTiers& t, size_t npairs) {
  if (npairs <= t.bcap) return NCX_OK;
  t.blist.release();
  t.bkey.release();
  t.bcap = 0;
  int rc = t.blist.reserve(npairs * 4 + 64);
  if (!rc) rc = t.bkey.reserve(npairs * 4 + 64);
  if (rc) return rc;
  t.bcap = npairs;
  return NCX_OK;
}

// Autotuner: for each bucket with enough pairs and no choice yet, time every first-tier variant
// on a sample of the bucket's pairs (HIP events; the least of three rounds after a warm-up
// round, the variants interleaved within each round) and keep the fastest.  The
// sample's results are real results (the full launch recomputes them identically).  Host-driven;
// the choice is kept in the shape set for every later call and scene step.
// Clears the tiers' counts and work counters (not the buckets').
static int clear_tier_counters(ncx_ctx* ctx, uint32_t* hdr) {
  int rc = fill_u32(ctx, hdr, NCX_OVF_TIER_WORDS, 0u);
  if (rc) return rc;
  static_assert(NCX_WORK_TUNE == 0 && NCX_WORK_T2 == 1 && NCX_WORK_T3 == 2 && NCX_WORK_T4 == 3 && NCX_WORK_TUNE_EPA == 4,
                "work sets");
  return fill_u32(ctx, ncx_work_set(hdr, 0), 5 * NCX_WORK_SET, 0u);
}

// Between the parts of a launch: the counts and work counters start again; the pairs that outgrew T1
// are summed, a list that overflowed is noted, and what outgrew T4 stays listed.
__global__ __launch_bounds__(256) void k_next_part(uint32_t* __restrict__ hdr, uint32_t cap) {
  for (uint32_t i = threadIdx.x; i < NCX_WORK_SETS; i += 256) hdr[NCX_WORK_BASE + i * NCX_WORK_SET] = 0u;
  if (threadIdx.x == 0) {
    const uint32_t t1 = hdr[NCX_OVF_T1_COUNT], t2 = hdr[NCX_OVF_T2_COUNT], t3 = hdr[NCX_OVF_T3_COUNT];
    hdr[NCX_OVF_EARLIER] += t1;
    if (t1 > cap || t2 > cap || t3 > cap) hdr[NCX_OVF_FULL] = 1u;
    hdr[NCX_OVF_T1_COUNT] = hdr[NCX_OVF_T2_COUNT] = hdr[NCX_OVF_T3_COUNT] = 0u;
    for (int b = 0; b < NCX_NBUCKETS; ++b) hdr[NCX_REC_COUNT + b] = 0u;
  }
}

#define TUNE_MIN_PAIRS 4096u
#define TUNE_SAMPLE 131072u
#define TUNE_ROUNDS 4
// Every stride-th entry of a bucket's run of the partitioned list, so the sample holds each of
// the bucket's type pairs in proportion.
__global__ void k_tune_sample(const uint32_t* __restrict__ list, uint32_t begin, uint32_t stride, uint32_t n,
                              uint32_t* __restrict__ out) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = list[begin + (size_t)i * stride];
}

static int autotune(ncx_shapes* S, ContactTiers& T, ncx_ctx* ctx, const KArgs& base, int mode) {
  uint32_t* hdr = T.ovf.as<uint32_t>();
  uint32_t rng[2 * NCX_NBUCKETS];
  NCX_HIP_CHECK(hipMemcpyAsync(rng, hdr + NCX_BKT_RANGE, sizeof(rng), hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  DevBuf dr, smp;
  int rc;
  if ((rc = dr.reserve(16)) || (rc = smp.reserve((size_t)TUNE_SAMPLE * 4))) return rc;
  hipEvent_t e0, e1;
  NCX_HIP_CHECK(hipEventCreate(&e0));
  NCX_HIP_CHECK(hipEventCreate(&e1));
  for (int b = 0; b < NCX_NBUCKETS; ++b) {
    const uint32_t cnt = rng[2 * b + 1] - rng[2 * b];
    if (S->tune[mode][b] >= 0 || cnt < (size_t)TUNE_MIN_PAIRS) continue;
    const uint32_t ns = std::min(cnt, TUNE_SAMPLE);
    hipLaunchKernelGGL(k_tune_sample, dim3(ceil_div(ns, 256)), dim3(256), 0, ctx->stream, base.list, rng[2 * b],
                       cnt / ns, ns, smp.as<uint32_t>());
    NCX_HIP_CHECK(hipGetLastError());
    const uint32_t sr[2] = {0, ns};
    NCX_HIP_CHECK(hipMemcpyAsync(dr.p, sr, 8, hipMemcpyHostToDevice, ctx->stream));
    // Rounds over the variants, so clock ramps and noise fall on every variant alike; the first
    // round warms up, each variant keeps its least time of the others.
    const int nv = T1_NVARIANTS[mode];
    float ms_v[NCX_T1_VARIANTS] = {};
    for (int rep = 0; rep < TUNE_ROUNDS && !rc; ++rep) {
      for (int v = 0; v < nv; ++v) {
        KArgs a = base;
        a.list = smp.as<uint32_t>();
        a.range_b = dr.as<uint32_t>();
        a.range_e = dr.as<uint32_t>() + 1;
        a.work = ncx_work_set(hdr, NCX_WORK_TUNE);
        a.rec_count = hdr + NCX_REC_COUNT_TUNE;
        if ((rc = clear_tier_counters(ctx, hdr))) break;
        NCX_HIP_CHECK(hipEventRecord(e0, ctx->stream));
        if (mode == 1) rc = launch_distance(v, ctx, a, ns);
        else rc = launch_contact_t1(v, GJK_BUCKET_G[b], ctx, a, ns, a.work, ncx_work_set(hdr, NCX_WORK_TUNE_EPA));
        if (rc) break;
        // the variant's first-tier overflows cost runs in the later tiers: time them too
        if (mode == 0 && (rc = launch_upper_tiers(ctx, T, a, ns))) break;
        NCX_HIP_CHECK(hipEventRecord(e1, ctx->stream));
        NCX_HIP_CHECK(hipEventSynchronize(e1));
        float ms = 0.f;
        NCX_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
        if (rep == 1 || (rep > 1 && ms < ms_v[v])) ms_v[v] = ms;
      }
    }
    int best = 1;
    for (int v = 0; v < nv && !rc; ++v) {
      S->tune_ms[mode][b][v] = ms_v[v];
      if (ms_v[v] < ms_v[best]) best = v;
    }
    if (rc) break;
    S->tune[mode][b] = (int8_t)best;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  dr.release();
  smp.release();
  if (rc) return rc;
  // the samples left entries in the overflow lists and moved the work counter: start clean
  return clear_tier_counters(ctx, hdr);
}

// Partitions the pair indices by sort key (vertex-count bucket, then type pair and overlap bin)
// into T.blist, each bucket's range in the header (which is clear).
static int partition_launch(ncx_shapes* S, ContactTiers& T, ncx_ctx* ctx, const ncx_pose* poses, const uint32_t* ia,
                            const uint32_t* ib, size_t npairs, const uint32_t* n_dev) {
  int rc;
  if ((rc = contact_tiers_reserve_list(T, npairs))) return rc;
  uint32_t* ovf = T.ovf.as<uint32_t>();
  // a pair with a bad index goes to a bucket that is launched
  const uint32_t bad_key = (NCX_NKEYS / NCX_NBUCKETS) * (uint32_t)__builtin_ctz(S->buckets | 1u << NCX_NBUCKETS);
  const unsigned bblocks = std::max(1u, ceil_div(npairs, (size_t)BKT_BLOCK * BKT_ITEMS));
  hipLaunchKernelGGL(k_bucket_count, dim3(bblocks), dim3(BKT_BLOCK), 0, ctx->stream, ia, ib, S->shapes.as<ncx_shape>(),
                     (uint32_t)S->n, poses, npairs, n_dev, ovf, T.bkey.as<uint32_t>(),
                     bad_key < NCX_NKEYS ? bad_key : 0u);
  NCX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_bucket_offsets, dim3(1), dim3(NCX_NKEYS), 0, ctx->stream, ovf);
  NCX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_bucket_scatter, dim3(bblocks), dim3(BKT_BLOCK), 0, ctx->stream, T.bkey.as<uint32_t>(), npairs,
                     n_dev, ovf, T.blist.as<uint32_t>());
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}

int pairs_partition(ncx_shapes* S, ContactTiers& T, ncx_ctx* ctx, const ncx_pose* poses, const uint32_t* ia,
                    const uint32_t* ib, size_t npairs, const uint32_t* n_dev) {
  int rc = fill_u32(ctx, T.ovf.as<uint32_t>(), NCX_OVF_HEADER, 0u);
  return rc ? rc : partition_launch(S, T, ctx, poses, ia, ib, npairs, n_dev);
}

// The launch: partition the pairs into vertex-count buckets (device-side counts, so it is
// graph-safe), run each bucket with its variant (T1, LDS arenas), then T2, T3 and T4
// rerun the device-counted overflow list of the tier before with larger LDS arenas, the last
// listing what outgrows it for contacts_resolve_overflow.  Every launch takes pairs from a work counter, so uneven pair
// costs balance across the chip.  npairs caps the pair count; n_dev (optional) holds the actual
// count on the device.  may_tune: run the autotuner first if a bucket has no choice yet (host
// synchronisation; never inside graph capture).
static int launch_tiers(ncx_shapes* S, ContactTiers& T, ncx_ctx* ctx, KArgs a, size_t npairs,
                        const uint32_t* n_dev, bool may_tune) {
  uint32_t* ovf = T.ovf.as<uint32_t>();
  NCX_REQUIRE(ovf, "contact launch: overflow lists not allocated");
  NCX_REQUIRE(npairs < ((size_t)1 << 31), "contact launch: more than 2^31 pairs");
  int rc;
  if ((rc = fill_u32(ctx, ovf, NCX_OVF_HEADER, 0u))) return rc;
  const int mode = a.distance_mode ? 1 : 0;
  a.nshapes = (uint32_t)S->n;
  a.bad_index = ovf + NCX_OVF_BAD;
  a.arena = nullptr;
  a.vcap = ArenaT4::VC;
  a.fcap = ArenaT4::FC;
  a.rec = T.rec;
  a.part_lo = 0u;
  a.part_hi = 0xFFFFFFFFu;
  a.sup = T.sup;
  a.ovf_count = ovf + NCX_OVF_T1_COUNT;
  a.ovf_list = T.t1_list();
  a.ovf_cap = T.cap;
  set_sus(T, a, 0);
  a.range_b = nullptr;
  a.range_e = nullptr;
  // a device-counted call's likely number of pairs, for grid sizes
  const size_t likely = n_dev ? std::min(npairs, 16 * S->n) : npairs;
  bool untuned = false;
  for (int b = 0; b < NCX_NBUCKETS; ++b) untuned = untuned || S->tune[mode][b] < 0;
  const bool tune_now = may_tune && untuned && npairs >= TUNE_MIN_PAIRS;
  // Partition (sort by key) unless the batch is small: below 16,384 pairs the three partition
  // kernels and the launches per bucket cost more (about 60 us) than the order saves.
  const bool partition = tune_now || npairs >= NCX_PARTITION_MIN_PAIRS;
  NCX_REQUIRE(mode == 1 || T.nrec >= (partition ? 1 : npairs), "contact launch: EPA records not allocated");
  T.parts = false;
  if (partition) {
    if ((rc = partition_launch(S, T, ctx, a.poses, a.ia, a.ib, npairs, n_dev))) return rc;
    KArgs t = a;
    t.list = T.blist.as<uint32_t>();
    t.n_dev = nullptr;
    t.npairs = npairs;
    if (tune_now && (rc = autotune(S, T, ctx, t, mode))) return rc;
  }
  if (!partition) {
    // one launch over all pairs, in their own order
    const int big = 31 - __builtin_clz(S->buckets | 1u);  // the variant of the set's largest hulls
    const int v = bucket_variant(S, mode, big, npairs);
    KArgs ab = a;
    ab.list = nullptr;
    ab.n_dev = n_dev;
    ab.npairs = npairs;
    ab.work = ncx_work_set(ovf, NCX_WORK_BKT);
    ab.rec_count = ovf + NCX_REC_COUNT;
    if (mode == 1) rc = launch_distance(v, ctx, ab, npairs);
    else rc = launch_contact_t1(v, GJK_SMALL_G, ctx, ab, likely, ab.work, ncx_work_set(ovf, NCX_WORK_EPA));
    if (rc) return rc;
  } else {
    // distance: one launch per run of consecutive buckets sharing a variant, over the partitioned
    // list; contact: one GJK and one EPA launch per bucket, its records from its own range on, for
    // each part of the list that the records suffice for
    const size_t part = mode == 0 ? T.nrec : npairs;
    T.parts = npairs > part;
    for (size_t lo = 0; lo < npairs; lo += part) {
      if (lo) {
        // the part before
        if ((rc = launch_upper_tiers(ctx, T, a, std::min(likely, part)))) return rc;
        hipLaunchKernelGGL(k_next_part, dim3(1), dim3(256), 0, ctx->stream, ovf, T.cap);
        NCX_HIP_CHECK(hipGetLastError());
      }
      a.part_lo = (uint32_t)lo;
      a.part_hi = (uint32_t)std::min(npairs, lo + part);
      for (int b0 = 0; b0 < NCX_NBUCKETS;) {
        if (mode == 0 && !(S->buckets >> b0 & 1u)) {  // no shape of the set makes such a pair
          ++b0;
          continue;
        }
        const int v = bucket_variant(S, mode, b0, npairs);
        int b1 = b0;
        while (mode == 1 && b1 + 1 < NCX_NBUCKETS && bucket_variant(S, mode, b1 + 1, npairs) == v) ++b1;
        KArgs ab = a;
        ab.list = T.blist.as<uint32_t>();
        ab.n_dev = nullptr;
        ab.npairs = npairs;
        ab.range_b = ovf + NCX_BKT_RANGE + 2 * b0;
        ab.range_e = ovf + NCX_BKT_RANGE + 2 * b1 + 1;
        ab.work = ncx_work_set(ovf, NCX_WORK_BKT + b0);
        ab.rec_count = ovf + NCX_REC_COUNT + b0;
        if (mode == 1) rc = launch_distance(v, ctx, ab, npairs);
        else rc = launch_contact_t1(v, GJK_BUCKET_G[b0], ctx, ab, likely, ab.work, ncx_work_set(ovf, NCX_WORK_EPA + b0));
        if (rc) return rc;
        b0 = b1 + 1;
      }
    }
  }
  if (mode == 0 && (rc = launch_upper_tiers(ctx, T, a, likely))) return rc;
  if (!T.last) T.last = new KArgs;
  *T.last = tier_args(T, a, 3);
  return NCX_OK;
}

// Graph-safe tiered contact launch over a device-counted pair list (the scene step); the caller
// runs contacts_resolve_overflow with the same tiers after the work completes.
int contacts_launch_device_count(ncx_shapes* S, ContactTiers& T, ncx_ctx* ctx, const ncx_pose* poses,
                                 const uint32_t* ia, const uint32_t* ib, const uint32_t* n_dev, size_t cap,
                                 float prediction, const float* init_dir, int max_iter, uint8_t* has, float* w1,
                                 float* w2, float* nrm, float* depth, int32_t* iters, bool may_tune, float* fdir,
                                 bool cap_seg) {
  KArgs a = {};
  a.fdir = fdir;
  a.cap_seg = cap_seg ? 1 : 0;
  a.shapes = S->shapes.as<ncx_shape>();
  a.P = Pool{S->hx.as<float>(), S->hy.as<float>(), S->hz.as<float>(), S->tri};
  a.poses = poses;
  a.ia = ia;
  a.ib = ib;
  a.prediction = prediction;
  a.init_dir = init_dir;
  a.max_iter = max_iter;
  a.has = has; a.w1 = w1; a.w2 = w2; a.nrm = nrm; a.depth = depth; a.iters = iters;
  a.distance_mode = 0;
  return launch_tiers(S, T, ctx, a, cap, n_dev, may_tune);
}

// After a launch in parts, whose records are gone: GJK again for the n pairs listed past T4, then their
// EPA from the start on device-memory arenas.
static int rerun_pairs(ContactTiers& T, ncx_ctx* ctx, uint32_t n) {
  uint32_t* hdr = T.ovf.as<uint32_t>();
  for (uint32_t o = 0; o < n; o += (uint32_t)T.nrec) {
    KArgs g = *T.last;
    g.list = T.t4_list() + o;
    g.npairs = std::min<size_t>(n - o, T.nrec);
    g.n_dev = nullptr;
    g.ovf_pairs = 0;
    g.rec_count = hdr + NCX_REC_COUNT;
    g.work = ncx_work_set(hdr, NCX_WORK_BKT);
    int rc;
    if ((rc = fill_u32(ctx, g.rec_count, 1, 0u)) || (rc = fill_u32(ctx, g.work, 1, 0u))) return rc;
    hipLaunchKernelGGL(k_contact_gjk<GJK_SMALL_G>, dim3(capped_blocks(ctx, GJK_BLOCKS_PER_CU, g.npairs, GJK_BS / GJK_SMALL_G)),
                       dim3(GJK_BS), 0, ctx->stream, g);
    NCX_HIP_CHECK(hipGetLastError());
    uint32_t recs = 0;
    NCX_HIP_CHECK(hipMemcpyAsync(&recs, g.rec_count, 4, hipMemcpyDeviceToHost, ctx->stream));
    NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    if ((rc = rerun_overflows(T, ctx, g, recs, nullptr, ArenaT4::VC, ArenaT4::FC, nullptr, 0))) return rc;
  }
  return NCX_OK;
}

// After the last launch_tiers on T has completed on ctx's stream: fails on a bad pair index or on
// more overflows than the lists hold, re-runs what T4 could not hold with device-memory arenas,
// and reports how many pairs needed more than the T1 arena.
int contacts_resolve_overflow(ContactTiers& T, ncx_ctx* ctx, size_t* n_large) {
  NCX_REQUIRE(T.last, "contact resolve: no tiered launch to resolve");
  uint32_t hdr[NCX_OVF_COUNTS];
  NCX_HIP_CHECK(hipMemcpyAsync(hdr, T.ovf.p, sizeof(hdr), hipMemcpyDeviceToHost, ctx->stream));
  NCX_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  NCX_REQUIRE(hdr[NCX_OVF_BAD] == 0, "contact batch: a pair index is not a shape of the set");
  if (hdr[NCX_OVF_FULL] || hdr[NCX_OVF_T1_COUNT] > T.cap || hdr[NCX_OVF_T2_COUNT] > T.cap ||
      hdr[NCX_OVF_T3_COUNT] > T.cap || hdr[NCX_OVF_T4_COUNT] > T.cap) {
    ncx_set_error("contact batch: more EPA arena overflows in one call than the overflow list holds");
    return NCX_E_CAPACITY;
  }
  if (n_large) *n_large = hdr[NCX_OVF_EARLIER] + hdr[NCX_OVF_T1_COUNT];
  if (T.parts) return rerun_pairs(T, ctx, hdr[NCX_OVF_T4_COUNT]);
  return rerun_overflows(T, ctx, *T.last, hdr[NCX_OVF_T4_COUNT], T.t4_list(), ArenaT4::VC, ArenaT4::FC, sus_slots(T, 3),
                         SUS_BYTES[3]);
}

static int run_pairs(ncx_shapes* S, KArgs a, size_t npairs) {
  if (npairs == 0) return NCX_OK;
  int rc;
  if ((rc = contact_tiers_reserve(S->tiers, S->ctx, npairs, a.distance_mode ? 0 : npairs))) return rc;
  if ((rc = launch_tiers(S, S->tiers, S->ctx, a, npairs, nullptr, true))) return rc;
  return contacts_resolve_overflow(S->tiers, S->ctx, nullptr);
}

extern "C" int ncx_contact_batch(ncx_shapes* s, const ncx_pose* poses, const uint32_t* ia, const uint32_t* ib,
                                 size_t npairs, float prediction, const float* init_dir, uint8_t* has, float* w1,
                                 float* w2, float* nrm, float* depth, int32_t* iters) {
  NCX_REQUIRE(s && poses && ia && ib && has && w1 && w2 && nrm && depth, "ncx_contact_batch: null argument");
  KArgs a = {};
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri};
  a.poses = poses;
  a.ia = ia;
  a.ib = ib;
  a.prediction = prediction;
  a.init_dir = init_dir;
  a.max_iter = 10000;
  a.has = has;
  a.w1 = w1;
  a.w2 = w2;
  a.nrm = nrm;
  a.depth = depth;
  a.iters = iters;
  a.distance_mode = 0;
  return run_pairs(s, a, npairs);
}

// Warm-started variant used by the learned initial direction: GJK from init_dir is capped at
// max_iter iterations, after which plain GJK (init_dir = None) recomputes the pair.
extern "C" int ncx_contact_batch_capped(ncx_shapes* s, const ncx_pose* poses, const uint32_t* ia, const uint32_t* ib,
                                        size_t npairs, float prediction, const float* init_dir, int32_t max_iter,
                                        uint8_t* has, float* w1, float* w2, float* nrm, float* depth,
                                        int32_t* iters) {
  NCX_REQUIRE(s && poses && ia && ib && has && w1 && w2 && nrm && depth, "ncx_contact_batch_capped: null argument");
  NCX_REQUIRE(max_iter >= 1 && max_iter <= 10000, "ncx_contact_batch_capped: max_iter out of range");
  KArgs a = {};
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri};
  a.poses = poses;
  a.ia = ia;
  a.ib = ib;
  a.prediction = prediction;
  a.init_dir = init_dir;
  a.max_iter = init_dir ? max_iter : 10000;
  a.has = has;
  a.w1 = w1;
  a.w2 = w2;
  a.nrm = nrm;
  a.depth = depth;
  a.iters = iters;
  a.distance_mode = 0;
  return run_pairs(s, a, npairs);
}

extern "C" int ncx_distance_batch(ncx_shapes* s, const ncx_pose* poses, const uint32_t* ia, const uint32_t* ib,
                                  size_t npairs, float* dist, int32_t* iters) {
  NCX_REQUIRE(s && poses && ia && ib && dist, "ncx_distance_batch: null argument");
  KArgs a = {};
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri};
  a.poses = poses;
  a.ia = ia;
  a.ib = ib;
  a.max_iter = 10000;
  a.dist = dist;
  a.iters = iters;
  a.distance_mode = 1;
  return run_pairs(s, a, npairs);
}

// distance_support_map_support_map_with_params with init_dir: GJK from init_dir capped at
// max_iter iterations, after which plain GJK (init_dir = None) recomputes the pair.
extern "C" int ncx_distance_batch_capped(ncx_shapes* s, const ncx_pose* poses, const uint32_t* ia,
                                         const uint32_t* ib, size_t npairs, const float* init_dir, int32_t max_iter,
                                         float* dist, int32_t* iters) {
  NCX_REQUIRE(s && poses && ia && ib && dist, "ncx_distance_batch_capped: null argument");
  NCX_REQUIRE(max_iter >= 1 && max_iter <= 10000, "ncx_distance_batch_capped: max_iter out of range");
  KArgs a = {};
  a.shapes = s->shapes.as<ncx_shape>();
  a.P = Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri};
  a.poses = poses;
  a.ia = ia;
  a.ib = ib;
  a.init_dir = init_dir;
  a.max_iter = init_dir ? max_iter : 10000;
  a.dist = dist;
  a.iters = iters;
  a.distance_mode = 1;
  return run_pairs(s, a, npairs);
}

// ------------------------------------------------------------------ shape AABBs
// One thread per shape, except hulls: a wavefront takes its hull lanes four at a time, 16 lanes
// per hull, each lane transforming four of the hull's points per pass with independent loads
// (coalesced across the lanes: the point pool is SoA), and reduces min/max over its 16 lanes.
// A thread looping over its own hull paid one memory round trip per point; one hull per
// wavefront at a time paid one per hull.  The min/max of a set does not depend on the visiting
// order (a point read twice, to keep the loads unconditional, changes nothing).
__device__ __forceinline__ float grp16_min(float x) {
#pragma unroll
  for (int s = 8; s >= 1; s >>= 1) x = fminf(x, __shfl_xor(x, s, 64));
  return x;
}
__device__ __forceinline__ float grp16_max(float x) {
#pragma unroll
  for (int s = 8; s >= 1; s >>= 1) x = fmaxf(x, __shfl_xor(x, s, 64));
  return x;
}

// STAGE: the boxes go through the broad phase's stored-box rule instead of to b0..b5 (the scene
// step's staging, fused): `st` holds the stored boxes (six SoA arrays of n), each is replaced by
// the new box loosened by `stage_margin` unless it contains the new box
// (dbvt_broad_phase.rs:325-347), or by the new box itself on the first step; the stored box is
// mirrored as two float4 in `sb`.
template <bool STAGE>
__global__ __launch_bounds__(256) void k_shape_aabbs(const ncx_shape* __restrict__ shapes, Pool P,
                                                      const ncx_pose* __restrict__ poses, size_t n, float margin,
                                                      float* b0, float* b1, float* b2, float* b3, float* b4,
                                                      float* b5, float* __restrict__ st = nullptr,
                                                      float4* __restrict__ sb = nullptr, float stage_margin = 0.f,
                                                      int first = 0) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < n;  // no early exit: every lane takes part in the hull loop
  const int lane = __lane_id();
  ShapeD g = {};
  iso m = {};
  f3 mn = f3{0.f, 0.f, 0.f}, mx = f3{0.f, 0.f, 0.f};
  bool hull = false;
  if (live) {
    g = load_shape(shapes, (uint32_t)i);
    m = load_pose(poses, (uint32_t)i);
    switch (g.type) {
      case NCX_BALL:  // ball_aabb (aabb_ball.rs:8-13)
        mn = m.t + f3{-g.a, -g.a, -g.a};
        mx = m.t + f3{g.a, g.a, g.a};
        break;
      case NCX_CUBOID: {  // center +- |R| h (aabb_cuboid.rs:7-14, isometry_ops.rs:43-45)
        float qi = m.q.i, qj = m.q.j, qk = m.q.k, qw = m.q.w;
        float ww = qw * qw, ii = qi * qi, jj = qj * qj, kk = qk * qk;
        float ij = qi * qj * 2.f, wk = qw * qk * 2.f, wj = qw * qj * 2.f;
        float ik = qi * qk * 2.f, jk = qj * qk * 2.f, wi = qw * qi * 2.f;
        float M[3][3] = {{ww + ii - jj - kk, ij - wk, wj + ik},
                         {wk + ij, ww - ii + jj - kk, jk - wi},
                         {ik - wj, wi + jk, ww - ii - jj + kk}};
        f3 ws;
        ws.x = (fabsf(M[0][0]) * g.a + fabsf(M[0][1]) * g.b) + fabsf(M[0][2]) * g.c;
        ws.y = (fabsf(M[1][0]) * g.a + fabsf(M[1][1]) * g.b) + fabsf(M[1][2]) * g.c;
        ws.z = (fabsf(M[2][0]) * g.a + fabsf(M[2][1]) * g.b) + fabsf(M[2][2]) * g.c;
        mn = m.t - ws;
        mx = m.t + ws;
        break;
      }
      case NCX_CAPSULE: {  // support_map_aabb (aabb_utils.rs:9-31)
        for (int d = 0; d < 3; ++d) {
          f3 e = f3{0.f, 0.f, 0.f};
          set_comp(e, d, 1.f);
          set_comp(mx, d, comp(support<1>(g, m, e, P, 0), d));
          set_comp(e, d, -1.f);
          set_comp(mn, d, comp(support<1>(g, m, e, P, 0), d));
        }
        break;
      }
      default:
        hull = true;
        break;
    }
  }
  // point_cloud_aabb (aabb_utils.rs:59-79): the componentwise min and max of the transformed points
  uint64_t hm = __ballot(hull);
  const int grp = lane >> 4, gl = lane & 15;
  while (hm) {
    // group grp takes the grp-th lowest remaining hull lane (none when fewer remain)
    uint64_t t = hm;
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q < grp) t &= t - 1;
    const int h = t ? __ffsll((unsigned long long)t) - 1 : lane;
    // shuffles outside any condition: a lane inactive at a shuffle does not supply its value
    const uint32_t off = (uint32_t)__shfl((int)g.off, h, 64);
    const uint32_t cnt_h = (uint32_t)__shfl((int)g.cnt, h, 64);
    const uint32_t cnt = t ? cnt_h : 0u;
    iso mh;
    mh.t = f3{__shfl(m.t.x, h, 64), __shfl(m.t.y, h, 64), __shfl(m.t.z, h, 64)};
    mh.q.i = __shfl(m.q.i, h, 64);
    mh.q.j = __shfl(m.q.j, h, 64);
    mh.q.k = __shfl(m.q.k, h, 64);
    mh.q.w = __shfl(m.q.w, h, 64);
    float lx = __builtin_inff(), ly = __builtin_inff(), lz = __builtin_inff();
    float ux = -__builtin_inff(), uy = -__builtin_inff(), uz = -__builtin_inff();
    for (uint32_t v0 = (uint32_t)gl; v0 < cnt; v0 += 64) {
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t v = v0 + 16u * u < cnt ? v0 + 16u * u : v0;
        const f3 p = xform_pt(mh, f3{P.x[off + v], P.y[off + v], P.z[off + v]});
        lx = fminf(lx, p.x); ly = fminf(ly, p.y); lz = fminf(lz, p.z);
        ux = fmaxf(ux, p.x); uy = fmaxf(uy, p.y); uz = fmaxf(uz, p.z);
      }
    }
    lx = grp16_min(lx); ly = grp16_min(ly); lz = grp16_min(lz);
    ux = grp16_max(ux); uy = grp16_max(uy); uz = grp16_max(uz);
    // a hull lane among the four taken fetches its box from the first lane of its group
    const bool mine = ((hm >> lane) & 1ull) != 0;
    const int rank = mine ? __popcll(hm & ((1ull << lane) - 1ull)) : 4;
    const int src = rank < 4 ? rank * 16 : lane;
    const float rlx = __shfl(lx, src, 64), rly = __shfl(ly, src, 64), rlz = __shfl(lz, src, 64);
    const float rux = __shfl(ux, src, 64), ruy = __shfl(uy, src, 64), ruz = __shfl(uz, src, 64);
    if (rank < 4) {
      mn = f3{rlx, rly, rlz};
      mx = f3{rux, ruy, ruz};
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) hm &= hm - 1;
  }
  if (!live) return;
  if (margin != 0.f) {  // AABB::loosened (aabb.rs:190-199)
    mn = mn + f3{-margin, -margin, -margin};
    mx = mx + f3{margin, margin, margin};
  }
  if constexpr (STAGE) {
    float b[6] = {mn.x, mn.y, mn.z, mx.x, mx.y, mx.z};
    if (!first) {
      // AABB::contains (aabb.rs:161-163)
      const bool contained = st[0 * n + i] <= b[0] && st[1 * n + i] <= b[1] && st[2 * n + i] <= b[2] &&
                             st[3 * n + i] >= b[3] && st[4 * n + i] >= b[4] && st[5 * n + i] >= b[5];
      if (contained) return;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        b[d] = b[d] + (-stage_margin);
        b[3 + d] = b[3 + d] + stage_margin;
      }
    }
#pragma unroll
    for (int d = 0; d < 6; ++d) st[d * n + i] = b[d];
    sb[2 * i] = make_float4(b[0], b[1], b[2], b[3]);
    sb[2 * i + 1] = make_float4(b[4], b[5], 0.f, 0.f);
  } else {
    b0[i] = mn.x; b1[i] = mn.y; b2[i] = mn.z;
    b3[i] = mx.x; b4[i] = mx.y; b5[i] = mx.z;
  }
}

// The scene step's shape boxes (loosened by `margin`) through the stored-box rule, into the
// stored boxes `st` and their float4 mirror `sb` (see k_shape_aabbs<true>).
int shapes_aabbs_stage_on(ncx_shapes* s, ncx_ctx* ctx, const ncx_pose* poses, float margin, float* st, float4* sb,
                          float stage_margin, bool first) {
  if (s->n == 0) return NCX_OK;
  hipLaunchKernelGGL(k_shape_aabbs<true>, dim3(ceil_div(s->n, 256)), dim3(256), 0, ctx->stream,
                     s->shapes.as<ncx_shape>(), Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri}, poses,
                     s->n, margin, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, st, sb, stage_margin,
                     first ? 1 : 0);
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}

extern "C" int ncx_shapes_aabbs_dev(ncx_shapes* s, const ncx_pose* poses, float margin, float* const out[6]) {
  NCX_REQUIRE(s && poses && out, "ncx_shapes_aabbs_dev: null argument");
  NCX_REQUIRE(margin >= 0.f, "ncx_shapes_aabbs_dev: the loosening margin must be positive");
  for (int d = 0; d < 6; ++d) NCX_REQUIRE(out[d], "ncx_shapes_aabbs_dev: null output");
  if (s->n == 0) return NCX_OK;
  hipLaunchKernelGGL(k_shape_aabbs<false>, dim3(ceil_div(s->n, 256)), dim3(256), 0, s->ctx->stream,
                     s->shapes.as<ncx_shape>(), Pool{s->hx.as<float>(), s->hy.as<float>(), s->hz.as<float>(), s->tri}, poses,
                     s->n, margin, out[0], out[1], out[2], out[3], out[4], out[5]);
  NCX_HIP_CHECK(hipGetLastError());
  return NCX_OK;
}
