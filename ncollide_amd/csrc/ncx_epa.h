// ncx_epa.h -- EPA of intersecting pairs on LDS arenas: the second kernel of a batched contact.
//
// The GJK kernel (k_contact_gjk) finishes every pair that does not need EPA and writes an EPA
// record -- the pair and its simplex -- for each pair that does; these kernels run the records.
//
// What bounds it: one EPA iteration is a serial chain of about twenty LDS round trips (heap, face
// and vertex reads), and pairs differ in their number of iterations (polytope pairs 2 to 4 on
// average, pairs with a capsule 10, up to hundreds).  Hence:
//   * a wavefront runs one iteration of each of its 64 / G pairs at a time, and a group whose pair
//     has ended takes the next record at the wavefront's next refill, so no group waits for the
//     longest pair of its wavefront;
//   * arenas are small, because the pairs in flight per CU are what LDS holds: polytope vertices
//     keep only their CSO point there (16 B; the two support points, needed at the end for one
//     face, go to a scratch array in device memory), the slots of deleted faces are used again,
//     ids are packed, and the silhouette search stack of the smaller arenas is two registers;
//   * a face keeps its normal, so neither its support direction nor a visibility test repeats the
//     square root and the divisions.
// Measured on one step of a 1,048,576-shape scene (10.2 M pairs, 3.4 M of them through EPA, 12
// iterations each on average): 99 ms in one kernel that ran GJK and EPA of a pair together (66 ms
// first tier, 27 ms second), 37 ms in two (GJK 9.5 ms; EPA 18.7, 3.1, 2.2 and 3.2 ms in its tiers).
// Results do not depend on any of this: every value is computed by the reference's operations in
// its order (src/query/algorithms/epa3.rs:219-454).
#pragma once
#include <type_traits>
#include "ncx_contact.h"

// ------------------------------------------------------------------ EPA records
// What GJK hands on: the pair, how its result is completed, and the simplex's support points (the
// CSO points are their differences).  A segment comes with its third point added (epa3.rs:299-305),
// so dim is 0, 2 or 3.
struct alignas(16) EpaRec {
  uint32_t k, dim_kind, pad0, pad1;
  float v[4][6];
};
static_assert(sizeof(EpaRec) == 112, "seven 16-byte words");

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------------------------ arenas
// VC vertices, FC faces, HC heap entries, SC silhouette edges, STC search-stack entries.
// BITS: width of vertex and face ids.  10-bit arenas keep a face as its normal and packed vertex
// ids in one 16-byte word, and its neighbours in a 4-byte word; 16-bit ones (the longest runs) keep
// no normals.  The vertex word's bits from 3 * BITS on are the deleted flag.
// A closed triangulated surface of V vertices has 2 V - 4 faces, and an iteration adds one vertex:
// the slots of the faces it deletes are used for the ones it makes, so FC is about 2 VC, where
// keeping every face ever made took 4 VC.  A heap entry names a face by its slot and its third
// vertex (the point of the iteration that made it, so no two faces of one slot share it); an entry
// whose face is gone is skipped when popped, as the reference skips deleted faces.
template <uint32_t VC_, uint32_t FC_, uint32_t HC_, uint32_t SC_, uint32_t STC_, int BITS_>
struct EpaArena {
  static constexpr uint32_t VC = VC_, FC = FC_, HC = HC_, SC = SC_, STC = STC_;
  static constexpr int BITS = BITS_;
  static constexpr bool FN = BITS == 10;
  typedef typename std::conditional<BITS == 10, uint32_t, uint64_t>::type W;   // three ids and a flag
  typedef typename std::conditional<BITS == 10, uint16_t, uint32_t>::type S;   // a silhouette edge
  static constexpr size_t r16(size_t n) { return (n + 15) & ~(size_t)15; }
  static constexpr size_t OFF_F = (size_t)VC * 16;                          // normals and vertex ids
  static constexpr size_t OFF_H = OFF_F + r16((size_t)FC * (FN ? 16 : sizeof(W)));
  static constexpr size_t OFF_A = OFF_H + r16(((size_t)HC + 1) * 8);          // neighbours
  static constexpr size_t OFF_S = OFF_A + r16((size_t)FC * sizeof(W));
  static constexpr size_t OFF_D = OFF_S + r16((size_t)SC * sizeof(S));        // faces this iteration deletes
  static constexpr size_t OFF_T = OFF_D + r16((size_t)SC * 2);
  static constexpr size_t BYTES = OFF_T + (BITS == 10 ? 0 : r16((size_t)STC * 4));
  static_assert(VC < (1u << BITS) && FC < (1u << BITS), "ids");
  typedef uint16_t __attribute__((may_alias)) u16a;
  typedef uint32_t __attribute__((may_alias)) u32a;
  typedef uint64_t __attribute__((may_alias)) u64a;
  typedef typename std::conditional<BITS == 10, u32a, u64a>::type WA;
  typedef typename std::conditional<BITS == 10, u16a, u32a>::type SA;
  typedef float4 __attribute__((may_alias)) f4a;
  typedef uint4 __attribute__((may_alias)) u4a;
  typedef HeapE __attribute__((may_alias)) hea;

  uint8_t* p;
  __device__ __forceinline__ f3 vert(uint32_t i) const {
    const float4 v = ((const f4a*)p)[i];
    return f3{v.x, v.y, v.z};
  }
  __device__ __forceinline__ void set_vert(uint32_t i, f3 v) const { ((f4a*)p)[i] = float4{v.x, v.y, v.z, 0.f}; }
  __device__ __forceinline__ W pts(uint32_t f) const {
    if constexpr (FN) return ((const u32a*)(p + OFF_F))[4 * f + 3];
    else return ((const WA*)(p + OFF_F))[f];
  }
  __device__ __forceinline__ W adj(uint32_t f) const { return ((const WA*)(p + OFF_A))[f]; }
  // The face's vertex ids, with its normal where one is kept.
  __device__ __forceinline__ W face(uint32_t f, f3& n) const {
    if constexpr (FN) {
      const float4 v = ((const f4a*)(p + OFF_F))[f];
      n = f3{v.x, v.y, v.z};
      return __float_as_uint(v.w);
    } else {
      return ((const WA*)(p + OFF_F))[f];
    }
  }
  __device__ __forceinline__ static W pack(uint32_t a, uint32_t b, uint32_t c) {
    return (W)a | ((W)b << BITS) | ((W)c << (2 * BITS));
  }
  __device__ __forceinline__ void set_face(uint32_t f, W w, W a, f3 n) const {
    if constexpr (FN) ((f4a*)(p + OFF_F))[f] = float4{n.x, n.y, n.z, __uint_as_float((uint32_t)w)};
    else ((WA*)(p + OFF_F))[f] = w;
    ((WA*)(p + OFF_A))[f] = a;
  }
  __device__ __forceinline__ void set_deleted(uint32_t f, W w) const {
    const W d = w | ((W)1 << (3 * BITS));
    if constexpr (FN) ((u32a*)(p + OFF_F))[4 * f + 3] = d;
    else ((WA*)(p + OFF_F))[f] = d;
  }
  // Neighbour j of face f becomes id, where it was `old`: an atomic add of the difference, because
  // two lanes may change two neighbours of one face at once.
  __device__ __forceinline__ void change_adj(uint32_t f, uint32_t j, uint32_t old, uint32_t id) const {
    const W d = ((W)id - (W)old) << (BITS * j);
    if constexpr (BITS == 10) {
      (void)__hip_atomic_fetch_add((uint32_t*)(p + OFF_A) + f, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
      (void)__hip_atomic_fetch_add((unsigned long long*)(p + OFF_A) + f, (unsigned long long)d, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  // heap entry 1 is 16-byte aligned, so the two children of any entry are one 16-byte word
  __device__ __forceinline__ hea* heap() const { return (hea*)(p + OFF_H + 8); }
  __device__ __forceinline__ SA* sil() const { return (SA*)(p + OFF_S); }
  __device__ __forceinline__ u16a* del() const { return (u16a*)(p + OFF_D); }
  __device__ __forceinline__ u32a* stack() const { return (u32a*)(p + OFF_T); }
};
template <int BITS, typename W> __device__ __forceinline__ uint32_t fld(W w, uint32_t i) {
  return (uint32_t)(w >> (BITS * i)) & ((1u << BITS) - 1u);
}
template <int BITS, typename W> __device__ __forceinline__ bool is_deleted(W w) { return (w >> (3 * BITS)) != 0; }
// Face::next_ccw_pt_id
template <int BITS, typename W> __device__ __forceinline__ uint32_t next_ccw_w(W w, uint32_t id) {
  return fld<BITS>(w, 0) == id ? 1u : (fld<BITS>(w, 1) == id ? 2u : 0u);
}
// A heap entry's name of the face with vertex ids w in slot f.
template <int BITS, typename W> __device__ __forceinline__ uint32_t heap_id(uint32_t f, W w) {
  return f | (fld<BITS>(w, 2) << 16);
}

// The silhouette search's stack: entries of 16 bits in two 64-bit registers (10-bit arenas), or in
// the arena.
template <class L> struct SilStack {
  uint64_t lo = 0, hi = 0;
  uint32_t n = 0;
  static constexpr uint32_t CAP = L::BITS == 10 ? 8u : L::STC;
  __device__ __forceinline__ void push(const L& A, uint32_t e) {
    if constexpr (L::BITS == 10) {
      hi = (hi << 16) | (lo >> 48);
      lo = (lo << 16) | e;
    } else {
      A.stack()[n] = e;
    }
    ++n;
  }
  __device__ __forceinline__ uint32_t pop(const L& A) {
    --n;
    if constexpr (L::BITS == 10) {
      const uint32_t e = (uint32_t)lo & 0xFFFFu;
      lo = (lo >> 16) | (hi << 48);
      hi >>= 16;
      return e;
    } else {
      return A.stack()[n];
    }
  }
};

// ------------------------------------------------------------------ the heap
// Rust's BinaryHeap (max-heap on neg_dist).  A pop's sift_down_to_bottom reads one level's two
// children at a time; lane j keeps the element that level j moves up.  The sift_up that follows
// climbs the same path: the highest level whose element the last entry does not exceed is where it
// stays, the levels above it have moved up, and those below it are where they were.  Needs a lane
// per heap level.
template <int G, class L>
__device__ __forceinline__ HeapE epa_heap_pop(const L& A, uint32_t& len, int gl, int gbase, uint64_t gmask) {
  auto* h = A.heap();
  len -= 1;
  HeapE item = h[len];
  if (len > 0) {
    const HeapE top = h[0];
    const HeapE e = item;
    item = top;
    uint32_t child = 1, lvl = 0, mypos = 0;
    HeapE mine = e;
    while (len >= 2 && child <= len - 2) {
      const uint4 pr = *(const typename L::u4a*)(h + child);
      const bool r = __uint_as_float(pr.x) <= __uint_as_float(pr.z);
      const HeapE pk = r ? HeapE{__uint_as_float(pr.z), pr.w} : HeapE{__uint_as_float(pr.x), pr.y};
      child += r ? 1u : 0u;
      if ((uint32_t)gl == lvl) { mine = pk; mypos = child; }
      ++lvl;
      child = 2 * child + 1;
    }
    if (child == len - 1) {
      const HeapE pk = h[child];
      if ((uint32_t)gl == lvl) { mine = pk; mypos = child; }
      ++lvl;
    }
    const bool stop = (uint32_t)gl < lvl && e.neg_dist <= mine.neg_dist;
    const uint64_t sm = (__ballot(stop) >> gbase) & gmask;
    const uint32_t up = sm ? 64u - (uint32_t)__builtin_clzll(sm) : 0u;  // levels that stay moved up
    wave_sync();
    if ((uint32_t)gl < up) h[(mypos - 1) >> 1] = mine;
    if (up == 0) h[0] = e;
    else if ((uint32_t)gl == up - 1) h[mypos] = e;
    wave_sync();
  }
  return item;
}

// sift_up with the group's lanes: lane j reads the j-th ancestor of the new entry (0 = the parent),
// the first ancestor that the entry does not exceed is where the climb stops, and the ancestors
// below it move down one level.
template <int G, class L>
__device__ __forceinline__ void epa_heap_push(const L& A, uint32_t& len, HeapE e, int gl, int gbase, uint64_t gmask) {
  auto* h = A.heap();
  const uint32_t k = len + 1;
  const uint32_t depth = 31u - (uint32_t)__builtin_clz(k);
  const bool have = (uint32_t)gl < depth;
  HeapE a = HeapE{0.f, 0u};
  if (have) a = h[(k >> (gl + 1)) - 1u];
  const uint64_t sm = (__ballot(have && e.neg_dist <= a.neg_dist) >> gbase) & gmask;
  const uint32_t s = sm ? (uint32_t)__builtin_ctzll(sm) : depth;
  wave_sync();
  if ((uint32_t)gl < s) h[(k >> gl) - 1u] = a;
  if (gl == 0) h[(k >> s) - 1u] = e;
  wave_sync();
  ++len;
}

// Face::new's inside test (proj_is_inside: the origin projects into the triangle) and its normal.
__device__ __forceinline__ bool face_inside(f3 a, f3 b, f3 c, f3& n) {
  Loc loc;
  proj_triangle(a, b, c, loc);
  n = tri_normal(a, b, c);
  return loc.kind == LOC_FACE;
}

// Face::can_be_seen_by (epa3.rs:143-156) of the face with vertex ids w and normal n (recomputed
// where the arena keeps none).
template <class L>
__device__ __forceinline__ bool epa_seen(const L& A, typename L::W w, f3 n, f3 pt, uint32_t opp) {
  const uint32_t o1 = opp == 2 ? 0u : opp + 1, o2 = opp == 0 ? 2u : opp - 1;
  const f3 p0 = A.vert(fld<L::BITS>(w, opp)), p1 = A.vert(fld<L::BITS>(w, o1)), p2 = A.vert(fld<L::BITS>(w, o2));
  if constexpr (!L::FN) {
    const f3 v0 = sel3(opp == 0, p0, sel3(opp == 1, p2, p1));
    const f3 v1 = sel3(opp == 0, p1, sel3(opp == 1, p0, p2));
    const f3 v2 = sel3(opp == 0, p2, sel3(opp == 1, p1, p0));
    n = tri_normal(v0, v1, v2);
  }
  return dot(pt - p0, n) >= -(NCX_FLT_EPS * 10.f) || affinely_dependent(p1, p2, pt);
}

// ------------------------------------------------------------------ one run
#define EPA_RUNNING 0
#define EPA_FACE 1       // ended on face `end`
#define EPA_NOTHING 2    // None
#define EPA_ZERO 3       // a one-point simplex: both points zero, normal +y
#define EPA_TOO_LARGE 4  // outgrew the arena
#define EPA_SUSPEND 5    // about to outgrow it, at an iteration boundary

template <class L> struct EpaState {
  uint32_t nv, nf, hl;
  int niter, iters;
  float max_dist;
  typename L::W best;  // vertex ids of the best face so far
  typename L::W end;   // EPA_FACE: of the face the run ends on
};

// The polytope of a record's simplex (epa3.rs:229-335).
template <int G, class L>
__device__ __forceinline__ int epa_begin(const L& A, const EpaRec* __restrict__ r, float* __restrict__ sup, EpaState<L>& s,
                                         int gl, int gbase, uint64_t gmask) {
  const float gjk_tol = NCX_FLT_EPS * 10.f;
  s.niter = 0;
  s.iters = 0;
  s.max_dist = NCX_FLT_MAX;
  const uint32_t dim = r->dim_kind & 3u;
  if (dim == 0) return EPA_ZERO;
  const float4* rv = (const float4*)r->v;
  const float4 q0 = rv[0], q1 = rv[1], q2 = rv[2], q3 = rv[3], q4 = rv[4], q5 = rv[5];
  f3 a1 = f3{q0.x, q0.y, q0.z}, a2 = f3{q0.w, q1.x, q1.y};
  f3 b1 = f3{q1.z, q1.w, q2.x}, b2 = f3{q2.y, q2.z, q2.w};
  f3 c1 = f3{q3.x, q3.y, q3.z}, c2 = f3{q3.w, q4.x, q4.y};
  f3 d1 = f3{q4.z, q4.w, q5.x}, d2 = f3{q5.y, q5.z, q5.w};
  const f3 a = a1 - a2, d = d1 - d2;
  f3 b = b1 - b2, c = c1 - c2;
  if (dim == 3 && dot(cross(b - a, c - a), d - a) > 0.f) {
    f3 t = b; b = c; c = t;
    t = b1; b1 = c1; c1 = t;
    t = b2; b2 = c2; c2 = t;
  }
  if (gl == 0) {
    float2* o = (float2*)sup;
    o[0] = float2{a1.x, a1.y}; o[1] = float2{a1.z, a2.x}; o[2] = float2{a2.y, a2.z};
    o[3] = float2{b1.x, b1.y}; o[4] = float2{b1.z, b2.x}; o[5] = float2{b2.y, b2.z};
    o[6] = float2{c1.x, c1.y}; o[7] = float2{c1.z, c2.x}; o[8] = float2{c2.y, c2.z};
    o[9] = float2{d1.x, d1.y}; o[10] = float2{d1.z, d2.x}; o[11] = float2{d2.y, d2.z};
  }
  A.set_vert(0, a);
  A.set_vert(1, b);
  A.set_vert(2, c);
  if (dim == 3) {
    A.set_vert(3, d);
    // faces (0,1,2) (1,3,2) (0,2,3) (0,3,1), one per lane; face f's distance is taken at vertex f
    const uint32_t f = (uint32_t)gl & 3u;
    const f3 va = sel3(f == 1, b, a), vb = sel3(f == 0, b, sel3(f == 2, c, d)),
             vc = sel3(f == 2, d, sel3(f == 3, b, c));
    f3 n;
    const bool inside = face_inside(va, vb, vc, n);
    const float dist = dot(n, sel3(f == 0, a, sel3(f == 1, b, sel3(f == 2, c, d))));
    if (gl < 4) {
      const uint32_t p0 = f == 1 ? 1u : 0u, p1 = f == 0 ? 1u : (f == 2 ? 2u : 3u), p2 = f == 2 ? 3u : (f == 3 ? 1u : 2u);
      // neighbours (3,1,2) (3,2,0) (0,1,3) (2,1,0)
      const uint32_t n0 = f < 2 ? 3u : (f == 2 ? 0u : 2u), n1 = f == 1 ? 2u : 1u, n2 = f == 0 ? 2u : (f == 2 ? 3u : 0u);
      A.set_face(f, L::pack(p0, p1, p2), L::pack(n0, n1, n2), n);
    }
    const bool four = gl < 4;
    const uint64_t im = (__ballot(four && inside) >> gbase) & gmask;
    if ((__ballot(four && inside && -dist > gjk_tol) >> gbase) & gmask) return EPA_NOTHING;
    wave_sync();
    s.nv = 4;
    s.nf = 4;
    s.hl = 0;
    for (uint32_t m = (uint32_t)im; m; m &= m - 1) {
      const uint32_t i = (uint32_t)__builtin_ctz(m);
      const float di = __shfl(dist, gbase + (int)i, 64);
      epa_heap_push<G>(A, s.hl, HeapE{-di, heap_id<L::BITS>(i, A.pts(i))}, gl, gbase, gmask);
    }
  } else {
    f3 n1, n2;
    face_inside(a, b, c, n1);
    face_inside(a, c, b, n2);
    A.set_face(0, L::pack(0, 1, 2), L::pack(1, 1, 1), n1);
    A.set_face(1, L::pack(0, 2, 1), L::pack(0, 0, 0), n2);
    A.heap()[0] = HeapE{0.f, heap_id<L::BITS>(0u, L::pack(0, 1, 2))};
    A.heap()[1] = HeapE{0.f, heap_id<L::BITS>(1u, L::pack(0, 2, 1))};
    wave_sync();
    s.nv = 3;
    s.nf = 2;
    s.hl = 2;
  }
  if (s.hl == 0) return EPA_NOTHING;
  s.best = A.pts(A.heap()[0].id & 0xFFFFu);
  return EPA_RUNNING;
}

// One iteration (epa3.rs:337-428).
template <int G, class L, bool SAVES>
__device__ __forceinline__ int epa_step(const L& A, const Ctx2& c, const Pool& P, float* __restrict__ sup, EpaState<L>& s,
                                        int gl, int gbase, uint64_t gmask) {
  constexpr int B = L::BITS;
  typedef typename L::W W;
  const float eps_tol = NCX_FLT_EPS * 100.f;
  const float gjk_tol = NCX_FLT_EPS * 10.f;
  // an iteration adds one vertex, two faces and the few heap entries of its new faces
  if (SAVES && (s.nv >= L::VC || s.nf + 2 > L::FC || s.hl + 6 > L::HC)) return EPA_SUSPEND;
  HeapE fid;
  uint32_t slot;
  W fw;
  f3 n;
  do {
    if (s.hl == 0) {
      s.end = s.best;
      return EPA_FACE;
    }
    fid = epa_heap_pop<G>(A, s.hl, gl, gbase, gmask);
    slot = fid.id & 0xFFFFu;
    fw = A.face(slot, n);
  } while (is_deleted<B>(fw) || fld<B>(fw, 2) != fid.id >> 16);
  if (s.nv >= L::VC) return EPA_TOO_LARGE;
  const W fa = A.adj(slot);
  if constexpr (!L::FN) n = tri_normal(A.vert(fld<B>(fw, 0)), A.vert(fld<B>(fw, 1)), A.vert(fld<B>(fw, 2)));
  const CSO cso = cso_from<G>(c, n, P, gl);
  s.iters += 1;
  const uint32_t sp_id = s.nv;
  const f3 pt = cso.pt();
  A.set_vert(sp_id, pt);
  if (gl == 0) {
    float2* o = (float2*)(sup + 6 * sp_id);
    o[0] = float2{cso.o1.x, cso.o1.y}; o[1] = float2{cso.o1.z, cso.o2.x}; o[2] = float2{cso.o2.y, cso.o2.z};
  }
  s.nv += 1;
  const float cand = dot(pt, n);
  if (cand < s.max_dist) { s.best = fw; s.max_dist = cand; }
  const float curr_dist = -fid.neg_dist;
  if (s.max_dist - curr_dist < eps_tol) {
    s.end = s.best;
    return EPA_FACE;
  }
  A.set_deleted(slot, fw);
  A.del()[0] = (uint16_t)slot;
  uint32_t nd = 1;
  wave_sync();
  // compute_silhouette for the three neighbours, depth first.  An entry's visibility is computed
  // when it is pushed, the entries pushed together on different lanes: it depends only on the
  // face's vertices, the new point and the edge.
  uint32_t ns = 0;
  SilStack<L> st;
  {
    f3 m0, m1, m2;
    const uint32_t f0 = fld<B>(fa, 0), f1 = fld<B>(fa, 1), f2 = fld<B>(fa, 2);
    const W w0 = A.face(f0, m0), w1 = A.face(f1, m1), w2 = A.face(f2, m2);
    const uint32_t o0 = next_ccw_w<B>(w0, fld<B>(fw, 0)), o1 = next_ccw_w<B>(w1, fld<B>(fw, 1)),
                   o2 = next_ccw_w<B>(w2, fld<B>(fw, 2));
    const int k = gl % 3;
    const bool v = epa_seen(A, k == 0 ? w0 : (k == 1 ? w1 : w2), sel3(k == 0, m0, sel3(k == 1, m1, m2)), pt,
                            k == 0 ? o0 : (k == 1 ? o1 : o2));
    const uint32_t vb = (uint32_t)(__ballot(v) >> gbase);
    st.push(A, f2 | (o2 << B) | (((vb >> 2) & 1u) << (B + 2)));
    st.push(A, f1 | (o1 << B) | (((vb >> 1) & 1u) << (B + 2)));
    st.push(A, f0 | (o0 << B) | ((vb & 1u) << (B + 2)));
  }
  while (st.n > 0) {
    const uint32_t e = st.pop(A);
    const uint32_t f = e & ((1u << B) - 1u), opp = (e >> B) & 3u;
    const W w = A.pts(f);
    const W wa = A.adj(f);
    if (is_deleted<B>(w)) continue;
    if (!(e >> (B + 2))) {
      if (ns >= L::SC) return EPA_TOO_LARGE;
      A.sil()[ns++] = (typename L::S)e;
    } else {
      if (nd >= L::SC) return EPA_TOO_LARGE;
      A.set_deleted(f, w);
      A.del()[nd++] = (uint16_t)f;
      wave_sync();
      if (st.n + 2 > SilStack<L>::CAP) return EPA_TOO_LARGE;
      const uint32_t i1 = opp == 0 ? 2u : opp - 1;
      const uint32_t g1 = fld<B>(wa, i1), g2 = fld<B>(wa, opp);
      f3 m1, m2;
      const W w1 = A.face(g1, m1), w2 = A.face(g2, m2);
      const uint32_t o1 = next_ccw_w<B>(w1, fld<B>(w, i1)), o2 = next_ccw_w<B>(w2, fld<B>(w, opp));
      const bool odd = (gl & 1) != 0;
      const bool v = epa_seen(A, odd ? w1 : w2, sel3(odd, m1, m2), pt, odd ? o1 : o2);
      const uint32_t vb = (uint32_t)(__ballot(v) >> gbase);
      st.push(A, g2 | (o2 << B) | ((vb & 1u) << (B + 2)));
      st.push(A, g1 | (o1 << B) | (((vb >> 1) & 1u) << (B + 2)));
    }
  }
  if (ns == 0) return EPA_NOTHING;
  wave_sync();
  // The new faces, silhouette edge q by lane q mod G.  Which edges get a face (their silhouette
  // face is still live), and so every new face's slot -- those of the deleted faces first -- is known
  // before any face is made; past one round the live edges are marked beforehand, because a new
  // face may take the slot of a deleted one.  A new face ends the run when its distance is below
  // the popped one's (the popped face is the answer) or negative (None), the first such edge
  // deciding; otherwise the faces that the origin projects into are pushed in edge order.
  constexpr uint32_t LIVE = 1u << (B + 3);
  if (ns > (uint32_t)G) {
    for (uint32_t q = (uint32_t)gl; q < ns; q += G) {
      const uint32_t e = A.sil()[q];
      if (!is_deleted<B>(A.pts(e & ((1u << B) - 1u)))) A.sil()[q] = (typename L::S)(e | LIVE);
    }
    wave_sync();
  }
  auto slot_of = [&](uint32_t i) { return i < nd ? (uint32_t)A.del()[i] : s.nf + i - nd; };
  uint32_t made = 0;
  const uint64_t below = (1ull << (gl & 63)) - 1ull;
  for (uint32_t base = 0; base < ns; base += G) {
    const uint32_t q = base + (uint32_t)gl;
    bool valid = false;
    uint32_t ef = 0, eo = 0;
    W w = 0;
    if (q < ns) {
      const uint32_t e = A.sil()[q];
      ef = e & ((1u << B) - 1u);
      eo = (e >> B) & 3u;
      w = A.pts(ef);
      valid = ns > (uint32_t)G ? (e & LIVE) != 0 : !is_deleted<B>(w);
    }
    const uint64_t vm = (__ballot(valid) >> gbase) & gmask;
    const uint32_t nnew = (uint32_t)__popcll(vm);
    if (made + nnew > nd && s.nf + made + nnew - nd > L::FC) return EPA_TOO_LARGE;
    const uint32_t mine = made + (uint32_t)__popcll(vm & below);
    const uint32_t new_id = slot_of(mine);
    bool inside = false;
    float dist = 0.f;
    if (valid) {
      const uint32_t j1 = eo == 0 ? 2u : eo - 1, j2 = eo == 2 ? 0u : eo + 1;
      const uint32_t pt1 = fld<B>(w, j1), pt2 = fld<B>(w, j2);
      const f3 v1 = A.vert(pt1), v2 = A.vert(pt2);
      const uint32_t old = fld<B>(A.adj(ef), j2);
      const uint32_t next = slot_of(mine + 1), prev = mine == 0 ? 0u : slot_of(mine - 1);
      f3 nn;
      inside = face_inside(v1, v2, pt, nn);
      dist = dot(nn, v1);
      A.change_adj(ef, j2, old, new_id);
      A.set_face(new_id, L::pack(pt1, pt2, sp_id), L::pack(ef, next & ((1u << B) - 1u), prev), nn);
    }
    const bool nearer = inside && dist < curr_dist;
    const bool wrong = inside && !nearer && -dist > gjk_tol;
    const uint64_t nm = (__ballot(nearer) >> gbase) & gmask, wm = (__ballot(wrong) >> gbase) & gmask;
    if (nm | wm) {
      const uint64_t f = (nm | wm) & (0ull - (nm | wm));
      if (nm & f) {
        s.end = fw;
        return EPA_FACE;
      }
      return EPA_NOTHING;
    }
    wave_sync();
    uint64_t im = (__ballot(inside) >> gbase) & gmask;
    if (s.hl + (uint32_t)__popcll(im) > L::HC) return EPA_TOO_LARGE;
    while (im) {
      const int i = gbase + (int)__builtin_ctzll(im);
      const float di = __shfl(dist, i, 64);
      const uint32_t id = (uint32_t)__shfl((int)new_id, i, 64) | (sp_id << 16);
      epa_heap_push<G>(A, s.hl, HeapE{-di, id}, gl, gbase, gmask);
      im &= im - 1;
    }
    made += nnew;
  }
  if (made == 0) return EPA_NOTHING;
  {
    // the ring of new faces closes
    const uint32_t f = slot_of(0), l = slot_of(made - 1);
    if (gl == 0) {
      A.change_adj(f, 2, 0u, l);
      A.change_adj(l, 1, slot_of(made) & ((1u << B) - 1u), f);
    }
  }
  if (made > nd) s.nf += made - nd;
  wave_sync();
  s.niter += 1;
  if (s.niter > 10000) return EPA_NOTHING;
  return EPA_RUNNING;
}

// Saved runs, in the layout of epa_load (ncx_contact.h), which the device-memory tier reads.  A
// heap entry whose face is gone names an extra deleted face; the best face, whose slot may hold
// another by now, is a second extra one.
template <int G, class L>
__device__ __forceinline__ void epa_write_saved(uint8_t* slot, const L& A, const float* sup, const EpaState<L>& s,
                                                int gl) {
  constexpr int B = L::BITS;
  typedef typename L::W W;
  uint32_t* d = (uint32_t*)slot;
  if (gl == 0) {
    d[0] = s.nv; d[1] = s.nf + 2; d[2] = s.hl; d[3] = (uint32_t)s.niter; d[4] = (uint32_t)s.iters;
    d[5] = 0; d[6] = s.nf + 1; d[7] = __float_as_uint(s.max_dist);
  }
  d += SAVE_HEADER_WORDS;
  copy_words<G>(d, (const uint32_t*)sup, s.nv * (uint32_t)(sizeof(VertA) / 4), gl);
  d += s.nv * (sizeof(VertA) / 4);
  for (uint32_t f = (uint32_t)gl; f < s.nf + 2; f += G) {
    const bool extra = f >= s.nf;
    const W w = extra ? s.best : A.pts(f), a = extra ? (W)0 : A.adj(f);
    d[4 * f] = fld<B>(w, 0) | (fld<B>(w, 1) << 16);
    d[4 * f + 1] = fld<B>(w, 2) | (fld<B>(a, 0) << 16);
    d[4 * f + 2] = fld<B>(a, 1) | (fld<B>(a, 2) << 16);
    d[4 * f + 3] = extra || is_deleted<B>(w) ? 1u : 0u;
  }
  d += 4 * ((size_t)s.nf + 2);
  for (uint32_t i = (uint32_t)gl; i < s.hl; i += G) {
    const HeapE e = A.heap()[i];
    const uint32_t f = e.id & 0xFFFFu;
    const W w = A.pts(f);
    d[2 * i] = __float_as_uint(e.neg_dist);
    d[2 * i + 1] = is_deleted<B>(w) || fld<B>(w, 2) != e.id >> 16 ? s.nf : f;
  }
}

template <int G, class L>
__device__ __forceinline__ void epa_read_saved(const uint8_t* slot, const L& A, float* sup, EpaState<L>& s, int gl) {
  constexpr int B = L::BITS;
  typedef typename L::W W;
  const uint32_t* d = (const uint32_t*)slot;
  s.nv = d[0]; s.nf = d[1]; s.hl = d[2]; s.niter = (int)d[3]; s.iters = (int)d[4];
  const uint32_t best = d[6];
  s.max_dist = __uint_as_float(d[7]);
  d += SAVE_HEADER_WORDS;
  copy_words<G>((uint32_t*)sup, d, 6 * s.nv, gl);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // lane 0 reads them at the run's end
  for (uint32_t i = (uint32_t)gl; i < s.nv; i += G) {
    const float* v = (const float*)d + 6 * (size_t)i;
    A.set_vert(i, f3{v[0], v[1], v[2]} - f3{v[3], v[4], v[5]});
  }
  wave_sync();
  d += 6 * (size_t)s.nv;
  for (uint32_t f = (uint32_t)gl; f < s.nf; f += G) {
    const uint32_t x = d[4 * f], y = d[4 * f + 1], z = d[4 * f + 2];
    const uint32_t p0 = x & 0xFFFFu, p1 = x >> 16, p2 = y & 0xFFFFu;
    f3 n = f3{0.f, 0.f, 0.f};
    if constexpr (L::FN) n = tri_normal(A.vert(p0), A.vert(p1), A.vert(p2));
    const W w = L::pack(p0, p1, p2) | ((d[4 * f + 3] & 0xFFFFu) ? (W)1 << (3 * B) : (W)0);
    A.set_face(f, w, L::pack(y >> 16, z & 0xFFFFu, z >> 16), n);
  }
  wave_sync();
  s.best = A.pts(best);
  d += 4 * (size_t)s.nf;
  for (uint32_t i = (uint32_t)gl; i < s.hl; i += G) {
    const uint32_t f = d[2 * i + 1];
    A.heap()[i] = HeapE{__uint_as_float(d[2 * i]), heap_id<B>(f, A.pts(f))};
  }
  wave_sync();
}
