// ncx_gjk.h -- device support maps, CSO points, the Voronoi simplex and GJK, shared by the
// contact/distance, time-of-impact, shape ray-cast and composite-shape kernels.
//
// One group of G lanes (a power of two inside a 64-wide wavefront) evaluates one query; every
// lane runs the same control flow on the same values and the lanes split ConvexHull vertex scans.
// Arithmetic restates the reference in f32 with its operation order:
//   supports  src/shape/{ball,cuboid,capsule,convex}.rs, src/utils/point_cloud_support_point.rs
//   simplex   src/query/algorithms/voronoi_simplex3.rs:49-280
//   GJK       src/query/algorithms/gjk.rs:76-177
#pragma once
#include "ncx_internal.h"

#define SHAPE_ORIGIN 4u
#define GJK_S_INTERSECTION 0
#define GJK_S_CLOSEST 1
#define GJK_S_NOINTER 3
#define GJK_S_NAN 4
#define GJK_S_CAP 5  // iteration cap reached (NoIntersection(+x) in the reference)

struct ShapeD {
  uint32_t type, off, cnt;
  float a, b, c;
};

__device__ __forceinline__ ShapeD load_shape(const ncx_shape* __restrict__ s, uint32_t i) {
  const uint4* p = (const uint4*)(s + i);
  uint4 u = p[0];
  uint4 v = p[1];
  ShapeD g;
  g.type = u.x;
  g.off = u.y;
  g.cnt = u.z;
  g.a = __uint_as_float(u.w);
  g.b = __uint_as_float(v.x);
  g.c = __uint_as_float(v.y);
  return g;
}

struct Pool {
  const float* __restrict__ x;
  const float* __restrict__ y;
  const float* __restrict__ z;
  // TriMesh triangles (three float4 per triangle: a with the face id in a.w, b, c), the parts of
  // a composite shape; SHAPE_TRIANGLE records index them by `off`
  const float4* __restrict__ tri;
};

// A part of a composite shape: triangle `off` of Pool::tri (TriMesh::triangle_at,
// src/shape/trimesh.rs:471-475), in the mesh's frame.
#define SHAPE_TRIANGLE 5u
// The core segment of a capsule (Capsule::segment, src/shape/capsule.rs:54-61): a = (0, -a, 0),
// b = (0, a, 0) with `a` the capsule's half height.  The contact-manifold generators replace a
// capsule by it (capsule_shape_manifold_generator.rs:34-46).
#define SHAPE_SEGMENT 6u

__device__ __forceinline__ void tri_vertices(const Pool& P, uint32_t k, f3& a, f3& b, f3& c) {
  const float4* t = P.tri + 3 * (size_t)k;
  const float4 A = t[0], B = t[1], C = t[2];
  a = f3{A.x, A.y, A.z};
  b = f3{B.x, B.y, B.z};
  c = f3{C.x, C.y, C.z};
}

// The value of another lane for a reduction step over 2 O lanes whose O-lane halves hold equal
// values already: lane ^ O for O = 1, 2; within 8 or 16 lanes the mirrored lane serves as well.
// These are DPP moves (a few cycles); __shfl_xor goes through the LDS crossbar, whose latency the
// support scans would pay up to four times per call.
template <int O> __device__ __forceinline__ uint32_t lane_across(uint32_t v) {
  if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);        // quad_perm 1,0,3,2
  else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
  else if constexpr (O == 4) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true);  // row_half_mirror
  else if constexpr (O == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, true);  // row_mirror
  else return (uint32_t)__shfl_xor((int)v, O, 64);
}

#define HULL_NONE 0xFFFFFFFFu
// The lane reduction of a hull scan: the larger value and, on ties, the lower index.
template <int G, int O = 1> __device__ __forceinline__ void hull_best(float& best, uint32_t& bi) {
  if constexpr (O < G) {
    const float ob = __uint_as_float(lane_across<O>(__float_as_uint(best)));
    const uint32_t oi = lane_across<O>(bi);
    if (oi != HULL_NONE && (bi == HULL_NONE || ob > best || (ob == best && oi < bi))) {
      best = ob;
      bi = oi;
    }
    hull_best<G, 2 * O>(best, bi);
  }
}

// point_cloud_support_point_id (src/utils/point_cloud_support_point.rs:6-24), split over G lanes.
// The reference keeps index 0 when dot(p_0, dir) is NaN and otherwise returns the first index of
// the maximum over the non-NaN dots (NaN never compares greater).  Each lane scans vertices
// gl, gl + G, ... in increasing order keeping its first maximum over non-NaN dots; the lane
// reduction keeps the larger value and, on ties, the lower index (vertex 0 with a NaN dot enters
// it as infinity).  U vertices' loads are issued together so their latencies overlap:
// the hulls in flight are far more than the first-level cache holds.  262,144 hull pairs of up to 256
// vertices, U = 4 and 8: contacts 2.71 and 2.48 ms, distances 2.12 and 1.76 ms; 12 and 16 no better.
// In the other kernels, whose scans are shorter or whose registers decide how many wavefronts run,
// 4: 65,536 shapes over a terrain take 27.2 ms with 4 and 30.3 ms with 8.
template <int G, int U = 4>
__device__ __forceinline__ uint32_t hull_support_id(const Pool& P, uint32_t off, uint32_t cnt, f3 dir, int gl) {
  float best = 0.f;
  uint32_t bi = HULL_NONE;
  bool nan0 = false;
  for (uint32_t v0 = gl; v0 < cnt; v0 += U * G) {
    float px[U], py[U], pz[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint32_t v = v0 + u * G;
      uint32_t vv = off + (v < cnt ? v : v0);  // always a vertex of this hull
      px[u] = P.x[vv];
      py[u] = P.y[vv];
      pz[u] = P.z[vv];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint32_t v = v0 + u * G;
      float d = dot(f3{px[u], py[u], pz[u]}, dir);
      if (v < cnt) {
        if (v == 0) nan0 = d != d;
        if (d > best || (bi == HULL_NONE && d == d)) {
          best = d;
          bi = v;
        }
      }
    }
  }
  if (nan0) {
    best = __builtin_inff();
    bi = 0;
  }
  hull_best<G>(best, bi);
  return bi == HULL_NONE ? 0u : bi;
}

// SupportMap::support_point (src/shape/support_map.rs:26-29) and the overrides of
// Ball (ball.rs:31-38), Cuboid (cuboid.rs:135-146), Capsule (capsule.rs:72-84),
// ConvexHull (convex.rs:418-423), ConstantOrigin (special_support_maps.rs:9-13).
// HULLS false: for shapes other than hulls.
template <int G, bool HULLS = true, int U = 4>
__device__ __forceinline__ f3 support(const ShapeD& g, const iso& m, f3 dir, const Pool& P, int gl) {
  switch (g.type) {
    case NCX_BALL: {
      f3 u = normalize(dir);
      return m.t + u * g.a;
    }
    case NCX_CUBOID: {
      f3 ld = inv_xform_vec(m, dir);
      f3 p = f3{copysignf(g.a, ld.x), copysignf(g.b, ld.y), copysignf(g.c, ld.z)};
      return xform_pt(m, p);
    }
    case NCX_CAPSULE: {
      f3 ld = inv_xform_vec(m, dir);
      f3 u = normalize(ld);
      f3 res = f3{0.f, copysignf(g.a, u.y), 0.f};
      return xform_pt(m, res + u * g.b);
    }
    case NCX_CONVEX_HULL: {
      if constexpr (!HULLS) return f3{0.f, 0.f, 0.f};
      f3 ld = inv_xform_vec(m, dir);
      uint32_t id = hull_support_id<G, U>(P, g.off, g.cnt, ld, gl);
      f3 p = f3{P.x[g.off + id], P.y[g.off + id], P.z[g.off + id]};
      return xform_pt(m, p);
    }
    case SHAPE_TRIANGLE: {  // Triangle::local_support_point (src/shape/triangle.rs:290-307)
      f3 ld = inv_xform_vec(m, dir);
      f3 a, b, c;
      tri_vertices(P, g.off, a, b, c);
      const float d1 = dot(a, ld), d2 = dot(b, ld), d3 = dot(c, ld);
      const f3 p = d1 > d2 ? (d1 > d3 ? a : c) : (d2 > d3 ? b : c);
      return xform_pt(m, p);
    }
    case SHAPE_SEGMENT: {  // Segment::local_support_point (src/shape/segment.rs:182-191)
      f3 ld = inv_xform_vec(m, dir);
      const f3 a = f3{0.f, -g.a, 0.f}, b = f3{0.f, g.a, 0.f};
      return xform_pt(m, dot(a, ld) > dot(b, ld) ? a : b);
    }
    default:
      return f3{0.f, 0.f, 0.f};
  }
}

// A point of the Minkowski difference with the two support points it came from.
struct CSO {
  f3 o1, o2;
  __device__ __forceinline__ f3 pt() const { return o1 - o2; }
};
// The same with the point kept apart: the ray cast moves it and leaves the support points.
struct CSOR {
  f3 p, o1, o2;
  __device__ __forceinline__ f3 pt() const { return p; }
};

struct Ctx2 {
  iso m1, m2;
  ShapeD g1, g2;
};

template <int G, int U = 4>
__device__ __forceinline__ CSO cso_from(const Ctx2& c, f3 dir, const Pool& P, int gl) {
  CSO r;
  r.o1 = support<G, true, U>(c.g1, c.m1, dir, P, gl);
  r.o2 = support<G, true, U>(c.g2, c.m2, -dir, P, gl);
  return r;
}

// support() of a shape per lane, called by the whole wavefront (`on`: the lanes that want one).  The
// hulls' scans are shared: group by group of GS lanes, the lanes of a group scan the hull of one of
// them after the other.
template <int GS>
__device__ __forceinline__ f3 support_wave(const ShapeD& g, const iso& m, f3 dir, const Pool& P, bool on) {
  const int lane = __lane_id(), gl = lane & (GS - 1);
  const bool hull = on && g.type == NCX_CONVEX_HULL;
  f3 r = f3{0.f, 0.f, 0.f};
  const uint64_t need = __ballot(hull);
  if (need) {
    const f3 ld = inv_xform_vec(m, dir);
    const uint32_t off = g.off, cnt = hull ? g.cnt : 0u;
    uint32_t id = 0;
#pragma unroll 1
    for (int j = 0; j < GS; ++j) {
      if (!(need & ((~0ull / ((1ull << GS) - 1ull)) << j))) continue;
      const int src = 4 * ((lane & ~(GS - 1)) + j);
      auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v); };
      const f3 d = f3{__uint_as_float(of(__float_as_uint(ld.x))), __uint_as_float(of(__float_as_uint(ld.y))),
                      __uint_as_float(of(__float_as_uint(ld.z)))};
      const uint32_t best = hull_support_id<GS, 8>(P, of(off), of(cnt), d, gl);
      id = gl == j ? best : id;
    }
    if (hull) r = xform_pt(m, f3{P.x[off + id], P.y[off + id], P.z[off + id]});
  }
  if (on && !hull) r = support<1, false>(g, m, dir, P, 0);
  return r;
}
template <int GS>
__device__ __forceinline__ CSO cso_wave(const Ctx2& c, f3 dir, const Pool& P, bool on) {
  CSO r;
  r.o1 = support_wave<GS>(c.g1, c.m1, dir, P, on);
  r.o2 = support_wave<GS>(c.g2, c.m2, -dir, P, on);
  return r;
}

// ------------------------------------------------------------------ Voronoi projections of the origin
#define LOC_VERTEX 0
#define LOC_EDGE 1
#define LOC_FACE 2
#define LOC_SOLID 3
struct Loc {
  int kind, id;
  float bc0, bc1, bc2;
};

// xform_pt(iso_identity(), v), bit for bit, without its products by zero: they add +0 to finite
// components (which turns -0 into +0) and make all three NaN when one is infinite or NaN.
__device__ __forceinline__ f3 ident_pt(f3 v) {
  const float z = ((0.f * v.x + 0.f * v.y) + 0.f * v.z) + 0.f;
  return f3{v.x + z, v.y + z, v.z + z};
}

// point_segment.rs:52-91 (identity isometry, point = origin)
__device__ __forceinline__ f3 proj_segment(f3 a, f3 b, Loc& loc) {
  iso m = iso_identity();
  f3 ls = inv_xform_pt(m, f3{0.f, 0.f, 0.f});
  f3 ab = b - a, ap = ls - a;
  float ab_ap = dot(ab, ap), sqnab = norm_sq(ab);
  if (ab_ap <= 0.f) { loc.kind = LOC_VERTEX; loc.id = 0; return ident_pt(a); }
  if (ab_ap >= sqnab) { loc.kind = LOC_VERTEX; loc.id = 1; return ident_pt(b); }
  float u = ab_ap / sqnab;
  loc.kind = LOC_EDGE; loc.id = 0; loc.bc0 = 1.f - u; loc.bc1 = u;
  return ident_pt(a + ab * u);
}

// point_triangle.rs:61-309, dim3, solid = true
__device__ __forceinline__ f3 proj_triangle(f3 a, f3 b, f3 c, Loc& loc) {
  iso m = iso_identity();
  f3 o = f3{0.f, 0.f, 0.f};
  f3 p = inv_xform_pt(m, o);
  f3 ab = b - a, ac = c - a, ap = p - a;
  float ab_ap = dot(ab, ap), ac_ap = dot(ac, ap);
  if (ab_ap <= 0.f && ac_ap <= 0.f) { loc.kind = LOC_VERTEX; loc.id = 0; return ident_pt(a); }
  f3 bp = p - b;
  float ab_bp = dot(ab, bp), ac_bp = dot(ac, bp);
  if (ab_bp >= 0.f && ac_bp <= ab_bp) { loc.kind = LOC_VERTEX; loc.id = 1; return ident_pt(b); }
  f3 cp = p - c;
  float ab_cp = dot(ab, cp), ac_cp = dot(ac, cp);
  if (ac_cp >= 0.f && ab_cp <= ac_cp) { loc.kind = LOC_VERTEX; loc.id = 2; return ident_pt(c); }
  f3 bc = c - b;
  f3 n = cross(ab, ac);
  float vc = dot(n, cross(ab, ap));
  if (vc < 0.f && ab_ap >= 0.f && ab_bp <= 0.f) {
    float v = ab_ap / norm_sq(ab);
    loc.kind = LOC_EDGE; loc.id = 0; loc.bc0 = 1.f - v; loc.bc1 = v;
    return ident_pt(a + ab * v);
  }
  float vb = -dot(n, cross(ac, cp));
  if (vb < 0.f && ac_ap >= 0.f && ac_cp <= 0.f) {
    float w = ac_ap / norm_sq(ac);
    loc.kind = LOC_EDGE; loc.id = 2; loc.bc0 = 1.f - w; loc.bc1 = w;
    return ident_pt(a + ac * w);
  }
  float va = dot(n, cross(bc, bp));
  if (va < 0.f && ac_bp - ab_bp >= 0.f && ab_cp - ac_cp >= 0.f) {
    float w = dot(bc, bp) / norm_sq(bc);
    loc.kind = LOC_EDGE; loc.id = 1; loc.bc0 = 1.f - w; loc.bc1 = w;
    return ident_pt(b + bc * w);
  }
  int clockwise = dot(n, ap) >= 0.f ? 0 : 1;
  if (va + vb + vc != 0.f) {
    float denom = 1.f / (va + vb + vc);
    float v = vb * denom, w = vc * denom;
    loc.kind = LOC_FACE; loc.id = clockwise; loc.bc0 = 1.f - v - w; loc.bc1 = v; loc.bc2 = w;
    return ident_pt(a + ab * v + ac * w);
  }
  loc.kind = LOC_SOLID; loc.id = 0;
  return o;
}

// check_edge of point_tetrahedron.rs:106-152
__device__ __forceinline__ bool tet_edge(int i, f3 a, f3 nabc, f3 nabd, f3 ap, f3 ab, float ap_ab,
                                         float bp_ab, float& dabc, float& dabd, Loc& loc, f3& out) {
  float ab_ab = ap_ab - bp_ab;
  f3 ap_x_ab = cross(ap, ab);
  dabc = dot(ap_x_ab, nabc);
  dabd = dot(ap_x_ab, nabd);
  if (ab_ab != 0.f && dabc >= 0.f && dabd >= 0.f && ap_ab >= 0.f && ap_ab <= ab_ab) {
    float u = ap_ab / ab_ab;
    loc.kind = LOC_EDGE; loc.id = i; loc.bc0 = 1.f - u; loc.bc1 = u;
    out = ident_pt(a + ab * u);
    return true;
  }
  return false;
}

// check_face of point_tetrahedron.rs:251-306
__device__ __forceinline__ bool tet_face(int i, f3 a, f3 b, f3 c, f3 ap, f3 bp, f3 cp, f3 ab, f3 ac,
                                         f3 ad, float d1, float d2, float d3, Loc& loc, f3& out) {
  if (d1 < 0.f && d2 < 0.f && d3 < 0.f) {
    f3 n = cross(ab, ac);
    if (dot(n, ad) * dot(n, ap) < 0.f) {
      f3 nn;
      float nl;
      if (!try_normalize(n, NCX_FLT_EPS, &nn, &nl)) return false;
      float vc = dot(nn, cross(ap, bp));
      float va = dot(nn, cross(bp, cp));
      float vb = dot(nn, cross(cp, ap));
      float denom = va + vb + vc;
      float inv_denom = 1.f / denom;
      float b0 = va * inv_denom, b1 = vb * inv_denom, b2 = vc * inv_denom;
      loc.kind = LOC_FACE; loc.id = i; loc.bc0 = b0; loc.bc1 = b1; loc.bc2 = b2;
      out = ident_pt(a * b0 + b * b1 + c * b2);
      return true;
    }
  }
  return false;
}

// point_tetrahedron.rs:35-353, solid = true
__device__ __forceinline__ f3 proj_tetrahedron(f3 A, f3 B, f3 C, f3 D, Loc& loc) {
  iso m = iso_identity();
  f3 p = inv_xform_pt(m, f3{0.f, 0.f, 0.f});
  f3 ab = B - A, ac = C - A, ad = D - A, ap = p - A;
  float ap_ab = dot(ap, ab), ap_ac = dot(ap, ac), ap_ad = dot(ap, ad);
  if (ap_ab <= 0.f && ap_ac <= 0.f && ap_ad <= 0.f) { loc.kind = LOC_VERTEX; loc.id = 0; return ident_pt(A); }
  f3 bc = C - B, bd = D - B, bp = p - B;
  float bp_bc = dot(bp, bc), bp_bd = dot(bp, bd), bp_ab = dot(bp, ab);
  if (bp_bc <= 0.f && bp_bd <= 0.f && bp_ab >= 0.f) { loc.kind = LOC_VERTEX; loc.id = 1; return ident_pt(B); }
  f3 cd = D - C, cp = p - C;
  float cp_ac = dot(cp, ac), cp_bc = dot(cp, bc), cp_cd = dot(cp, cd);
  if (cp_cd <= 0.f && cp_bc >= 0.f && cp_ac >= 0.f) { loc.kind = LOC_VERTEX; loc.id = 2; return ident_pt(C); }
  f3 dp = p - D;
  float dp_cd = dot(dp, cd), dp_bd = dot(dp, bd), dp_ad = dot(dp, ad);
  if (dp_ad >= 0.f && dp_bd >= 0.f && dp_cd >= 0.f) { loc.kind = LOC_VERTEX; loc.id = 3; return ident_pt(D); }
  f3 out;
  float dabc, dabd, dacd, dacb, dadb, dadc, dbca, dbcd, dbdc, dbda, dcda, dcdb;
  f3 nabc = cross(ab, ac), nabd = cross(ab, ad);
  if (tet_edge(0, A, nabc, nabd, ap, ab, ap_ab, bp_ab, dabc, dabd, loc, out)) return out;
  f3 nacd = cross(ac, ad);
  if (tet_edge(1, A, nacd, -nabc, ap, ac, ap_ac, cp_ac, dacd, dacb, loc, out)) return out;
  if (tet_edge(2, A, -nabd, -nacd, ap, ad, ap_ad, dp_ad, dadb, dadc, loc, out)) return out;
  f3 nbcd = cross(bc, bd);
  if (tet_edge(3, B, nabc, nbcd, bp, bc, bp_bc, cp_bc, dbca, dbcd, loc, out)) return out;
  if (tet_edge(4, B, -nbcd, nabd, bp, bd, bp_bd, dp_bd, dbdc, dbda, loc, out)) return out;
  if (tet_edge(5, C, nacd, nbcd, cp, cd, cp_cd, dp_cd, dcda, dcdb, loc, out)) return out;
  if (tet_face(0, A, B, C, ap, bp, cp, ab, ac, ad, dabc, dbca, dacb, loc, out)) return out;
  if (tet_face(1, A, B, D, ap, bp, dp, ab, ad, ac, dadb, dabd, dbda, loc, out)) return out;
  if (tet_face(2, A, C, D, ap, cp, dp, ac, ad, ab, dacd, dcda, dadc, loc, out)) return out;
  if (tet_face(3, B, C, D, bp, cp, dp, bc, bd, -ab, dbcd, dcdb, dbdc, loc, out)) return out;
  loc.kind = LOC_SOLID; loc.id = 0;
  return xform_pt(m, p);
}

// ------------------------------------------------------------------ VoronoiSimplex (voronoi_simplex3.rs:12-352)
// The four vertices are separate members and the "previous vertex" permutation is
// packed 2 bits per slot, so no runtime index reaches an array: everything stays in
// registers.
template <class V> struct SimplexT {
  V v0, v1, v2, v3;
  uint32_t pv;  // prev_vertices, slot i in bits [2i, 2i+2)
  float proj0, proj1, proj2, pproj0, pproj1, pproj2;
  int dim, pdim;
};
typedef SimplexT<CSO> Simplex;
typedef SimplexT<CSOR> SimplexR;

// Value selects (never a select between addresses), so the simplex stays in registers.
__device__ __forceinline__ f3 sel3(bool c, f3 a, f3 b) { return f3{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z}; }
__device__ __forceinline__ CSO csel(bool c, const CSO& a, const CSO& b) {
  return CSO{sel3(c, a.o1, b.o1), sel3(c, a.o2, b.o2)};
}
__device__ __forceinline__ CSOR csel(bool c, const CSOR& a, const CSOR& b) {
  return CSOR{sel3(c, a.p, b.p), sel3(c, a.o1, b.o1), sel3(c, a.o2, b.o2)};
}
template <class V> __device__ __forceinline__ V sx_get(const SimplexT<V>& s, int i) {
  return csel(i == 0, s.v0, csel(i == 1, s.v1, csel(i == 2, s.v2, s.v3)));
}
template <class V> __device__ __forceinline__ void sx_set(SimplexT<V>& s, int i, const V& c) {
  s.v0 = csel(i == 0, c, s.v0);
  s.v1 = csel(i == 1, c, s.v1);
  s.v2 = csel(i == 2, c, s.v2);
  s.v3 = csel(i == 3, c, s.v3);
}
template <class V> __device__ __forceinline__ void sx_swap(SimplexT<V>& s, int i, int j) {
  V a = sx_get(s, i), b = sx_get(s, j);
  sx_set(s, i, b);
  sx_set(s, j, a);
  uint32_t pi = (s.pv >> (2 * i)) & 3u, pj = (s.pv >> (2 * j)) & 3u;
  s.pv &= ~((3u << (2 * i)) | (3u << (2 * j)));
  s.pv |= (pj << (2 * i)) | (pi << (2 * j));
}

#define PV_IDENTITY 0xE4u  // slots (0, 1, 2, 3)

template <class V> __device__ __forceinline__ void sx_init(SimplexT<V>& s) {
  s.pv = PV_IDENTITY;
  s.proj0 = s.proj1 = s.proj2 = 0.f;
  s.pproj0 = s.pproj1 = s.pproj2 = 0.f;
  s.dim = 0;
  s.pdim = 0;
}

template <class V> __device__ __forceinline__ void sx_reset(SimplexT<V>& s, const V& p) {
  s.dim = 0;
  s.pdim = 0;
  s.v0 = p;
}

template <class V> __device__ __forceinline__ bool sx_add(SimplexT<V>& s, const V& pt) {
  const float tol = NCX_FLT_EPS * 10.f;
  s.pdim = s.dim;
  s.pproj0 = s.proj0; s.pproj1 = s.proj1; s.pproj2 = s.proj2;
  s.pv = PV_IDENTITY;
  if (s.dim == 0) {
    if (norm_sq(s.v0.pt() - pt.pt()) < tol) return false;
  } else if (s.dim == 1) {
    f3 ab = s.v1.pt() - s.v0.pt(), ac = pt.pt() - s.v0.pt();
    if (norm_sq(cross(ab, ac)) < tol) return false;
  } else {
    f3 ab = s.v1.pt() - s.v0.pt(), ac = s.v2.pt() - s.v0.pt(), ap = pt.pt() - s.v0.pt();
    f3 n = normalize(cross(ab, ac));
    if (fabsf(dot(n, ap)) < tol) return false;
  }
  s.dim += 1;
  sx_set(s, s.dim, pt);
  return true;
}

template <class V> __device__ __forceinline__ f3 sx_project_reduce(SimplexT<V>& s) {
  if (s.dim == 0) {
    s.proj0 = 1.f;
    return s.v0.pt();
  } else if (s.dim == 1) {
    Loc loc;
    f3 pr = proj_segment(s.v0.pt(), s.v1.pt(), loc);
    if (loc.kind == LOC_VERTEX && loc.id == 0) { s.proj0 = 1.f; s.dim = 0; }
    else if (loc.kind == LOC_VERTEX) { sx_swap(s, 0, 1); s.proj0 = 1.f; s.dim = 0; }
    else { s.proj0 = loc.bc0; s.proj1 = loc.bc1; }
    return pr;
  } else if (s.dim == 2) {
    Loc loc;
    f3 pr = proj_triangle(s.v0.pt(), s.v1.pt(), s.v2.pt(), loc);
    if (loc.kind == LOC_VERTEX) { sx_swap(s, 0, loc.id); s.proj0 = 1.f; s.dim = 0; }
    else if (loc.kind == LOC_EDGE) {
      if (loc.id == 0) { s.proj0 = loc.bc0; s.proj1 = loc.bc1; }
      else if (loc.id == 1) { sx_swap(s, 0, 2); s.proj0 = loc.bc1; s.proj1 = loc.bc0; }
      else { sx_swap(s, 1, 2); s.proj0 = loc.bc0; s.proj1 = loc.bc1; }
      s.dim = 1;
    } else if (loc.kind == LOC_FACE) {
      s.proj0 = loc.bc0; s.proj1 = loc.bc1; s.proj2 = loc.bc2;
    }
    return pr;
  } else {
    Loc loc;
    f3 pr = proj_tetrahedron(s.v0.pt(), s.v1.pt(), s.v2.pt(), s.v3.pt(), loc);
    if (loc.kind == LOC_VERTEX) { sx_swap(s, 0, loc.id); s.proj0 = 1.f; s.dim = 0; }
    else if (loc.kind == LOC_EDGE) {
      switch (loc.id) {
        case 1: sx_swap(s, 1, 2); break;
        case 2: sx_swap(s, 1, 3); break;
        case 3: sx_swap(s, 0, 2); break;
        case 4: sx_swap(s, 0, 3); break;
        case 5: sx_swap(s, 0, 2); sx_swap(s, 1, 3); break;
        default: break;
      }
      if (loc.id == 3 || loc.id == 4) { s.proj0 = loc.bc1; s.proj1 = loc.bc0; }
      else { s.proj0 = loc.bc0; s.proj1 = loc.bc1; }
      s.dim = 1;
    } else if (loc.kind == LOC_FACE) {
      const int fid = loc.id;
      s.v2 = csel(fid == 1, s.v3, s.v2);
      s.v1 = csel(fid == 2, s.v3, s.v1);
      s.v0 = csel(fid >= 3, s.v3, s.v0);
      switch (fid) {
        case 0: s.proj0 = loc.bc0; s.proj1 = loc.bc1; s.proj2 = loc.bc2; break;
        case 1: s.proj0 = loc.bc0; s.proj1 = loc.bc1; s.proj2 = loc.bc2; break;
        case 2: s.proj0 = loc.bc0; s.proj1 = loc.bc2; s.proj2 = loc.bc1; break;
        default: s.proj0 = loc.bc2; s.proj1 = loc.bc0; s.proj2 = loc.bc1; break;
      }
      s.dim = 2;
    }
    return pr;
  }
}

// gjk.rs:367-388
template <class V> __device__ __forceinline__ void gjk_result(const SimplexT<V>& s, bool prev, f3& p1, f3& p2) {
  f3 r1 = f3{0.f, 0.f, 0.f}, r2 = f3{0.f, 0.f, 0.f};
  const int n = prev ? s.pdim : s.dim;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i <= n) {
      float c = prev ? (i == 0 ? s.pproj0 : (i == 1 ? s.pproj1 : s.pproj2))
                     : (i == 0 ? s.proj0 : (i == 1 ? s.proj1 : s.proj2));
      const V pt = sx_get(s, prev ? (int)((s.pv >> (2 * i)) & 3u) : i);
      r1 = r1 + pt.o1 * c;
      r2 = r2 + pt.o2 * c;
    }
  }
  p1 = r1;
  p2 = r2;
}

struct GJKOut {
  int status;
  f3 p1, p2, dir;
  int iters;
};

// gjk::closest_points (gjk.rs:76-177), exact_dist = true, from the simplex of the support point
// along dir.  The first point, the loop's points and (FOR_EPA) an intersecting segment's third
// point (epa3.rs:294-305) are taken by one support call in the loop, so a kernel holds the support
// functions of every shape once; with a call each, the contact kernel's GJK spilled 103 registers
// more.
struct GJKRun {
  f3 dir, old_dir;
  float max_bound;
  int niter;  // -1: the first point; -2: a segment's third point
};
__device__ __forceinline__ void gjk_begin(GJKRun& g, Simplex& s, GJKOut& r, f3 dir) {
  r.iters = 0;
  sx_init(s);
  g.dir = dir;
  g.old_dir = f3{0.f, 0.f, 0.f};
  g.max_bound = NCX_FLT_MAX;
  g.niter = -1;
}
// What follows the support point along g.dir; true when the run has ended, with its result in r.
template <bool FOR_EPA>
__device__ __forceinline__ bool gjk_step(GJKRun& g, Simplex& s, const CSO& cso, float max_dist, int max_iter,
                                         GJKOut& r) {
  const float eps_tol = NCX_FLT_EPS * 10.f;
  const float eps_rel = __builtin_sqrtf(eps_tol);
  f3 proj;
  if (FOR_EPA && g.niter == -2) {
    s.v2 = cso;
    s.dim = 2;
    r.status = GJK_S_INTERSECTION;
    return true;
  }
  bool meets = false;
  if (g.niter < 0) {
    sx_reset(s, cso);
    proj = sx_project_reduce(s);
    f3 pd;
    float nl;
    if (try_normalize(proj, 0.f, &pd, &nl)) g.old_dir = -pd;
    else meets = true;
  } else {
    r.iters += 1;
    const float min_bound = -dot(g.dir, cso.pt());
    if (!(min_bound == min_bound)) { r.status = GJK_S_NAN; return true; }
    if (min_bound > max_dist) { r.dir = g.dir; r.status = GJK_S_NOINTER; return true; }
    if (g.max_bound - min_bound <= eps_rel * g.max_bound || !sx_add(s, cso)) {
      gjk_result(s, false, r.p1, r.p2);
      r.dir = g.dir;
      r.status = GJK_S_CLOSEST;
      return true;
    }
    g.old_dir = g.dir;
    proj = sx_project_reduce(s);
    if (s.dim == 3) {
      if (min_bound >= eps_tol) {
        gjk_result(s, true, r.p1, r.p2);
        r.dir = g.old_dir;
        r.status = GJK_S_CLOSEST;
        return true;
      }
      r.status = GJK_S_INTERSECTION;
      return true;
    }
  }
  g.niter += 1;
  if (g.niter > 0 && g.niter == max_iter) { r.dir = f3{1.f, 0.f, 0.f}; r.status = GJK_S_CAP; return true; }
  const float old_max_bound = g.max_bound;
  f3 nd;
  float dist;
  if (!meets && try_normalize(-proj, eps_tol, &nd, &dist)) {
    g.dir = nd;
    g.max_bound = dist;
  } else {
    if (FOR_EPA && s.dim == 1) {
      const f3 dpt = s.v1.pt() - s.v0.pt();
      // nalgebra orthonormal_subspace_basis for one vector; epa3.rs:299-305 keeps a x dpt.
      f3 a = fabsf(dpt.x) > fabsf(dpt.y) ? f3{dpt.z, 0.f, -dpt.x} : f3{0.f, -dpt.z, dpt.y};
      a = normalize(a);
      g.dir = cross(a, dpt);
      g.niter = -2;
      return false;
    }
    r.status = GJK_S_INTERSECTION;
    return true;
  }
  if (g.max_bound >= old_max_bound) {
    gjk_result(s, true, r.p1, r.p2);
    r.dir = g.old_dir;
    r.status = GJK_S_CLOSEST;
    return true;
  }
  return false;
}
template <int G, bool FOR_EPA = false, int U = 4>
__device__ __forceinline__ GJKOut gjk(const Ctx2& c, f3 dir, float max_dist, Simplex& s, const Pool& P, int gl,
                                      int max_iter) {
  GJKOut r;
  GJKRun g;
  gjk_begin(g, s, r, dir);
  while (!gjk_step<FOR_EPA>(g, s, cso_from<G, U>(c, g.dir, P, gl), max_dist, max_iter, r)) {
  }
  return r;
}

// ------------------------------------------------------------------ time of impact and ray casts on support maps
// approx::relative_eq!(x, 0) with the default epsilon and max_relative: |x| <= f32::EPSILON.
__device__ __forceinline__ bool relative_eq_zero(float x) { return fabsf(x) <= NCX_FLT_EPS; }

// SupportMap::support_point_toward (src/shape/support_map.rs:31-34): `u` is unit and used as given.
// Ball overrides it (ball.rs:36-39); Capsule's local_support_point_toward does not normalise
// (capsule.rs:79-83); Cuboid and ConvexHull fall back to support_point.
template <int G>
__device__ __forceinline__ f3 support_toward(const ShapeD& g, const iso& m, f3 u, const Pool& P, int gl) {
  if (g.type == NCX_BALL) return m.t + u * g.a;
  if (g.type == NCX_CAPSULE) {
    f3 ld = inv_xform_vec(m, u);
    f3 res = f3{0.f, copysignf(g.a, ld.y), 0.f};
    return xform_pt(m, res + ld * g.b);
  }
  return support<G>(g, m, u, P, gl);
}

// Two support maps, the first dilated by `dil` when `dilated` (DilatedShape,
// src/query/algorithms/special_support_maps.rs:32-59: support_point normalises the direction and
// adds the ball's support point to the shape's).
struct RCtx {
  iso m1, m2;
  ShapeD g1, g2;
  float dil;
  bool dilated;
  bool local;  // the first map at the identity against ConstantOrigin (m1, m2 and g2 unused)
};

// inv_xform_vec(iso_identity(), v), bit for bit: v itself unless a component is zero (whose sign the
// products by zero may change), infinite or NaN.
__device__ __forceinline__ f3 ident_inv_vec(f3 v) {
  const float p = (v.x * v.y) * v.z;
  if (p != 0.f && p - p == 0.f) return v;
  return inv_xform_vec(iso_identity(), v);
}

// support() of a shape at the identity.
template <int G, int KIND>
__device__ __forceinline__ f3 support_local(const ShapeD& g, f3 dir, const Pool& P, int gl) {
  const f3 ld = ident_inv_vec(dir);
  if (KIND == NCX_CAPSULE || (KIND < 0 && g.type == NCX_CAPSULE)) {
    const f3 u = normalize(ld);
    return ident_pt(f3{0.f, copysignf(g.a, u.y), 0.f} + u * g.b);
  }
  if (KIND == NCX_CONVEX_HULL || (KIND < 0 && g.type == NCX_CONVEX_HULL)) {
    const uint32_t id = g.off + hull_support_id<G>(P, g.off, g.cnt, ld, gl);
    return ident_pt(f3{P.x[id], P.y[id], P.z[id]});
  }
  return support<G>(g, iso_identity(), dir, P, gl);
}

// KIND: the first map's shape type where the caller knows it (any: RC_ANY), which leaves the other
// types' code out.
#define RC_ANY -1
template <int G, int KIND = RC_ANY>
__device__ __forceinline__ CSOR cso_from_r(const RCtx& c, f3 dir, const Pool& P, int gl) {
  CSOR r;
  if (KIND != RC_ANY || c.local) {  // ConstantOrigin (special_support_maps.rs:9-13) is the second map
    r.o1 = support_local<G, KIND>(c.g1, dir, P, gl);
    r.o2 = f3{0.f, 0.f, 0.f};
    r.p = r.o1 - r.o2;
    return r;
  }
  if (c.dilated) {
    f3 u = normalize(dir);
    r.o1 = support_toward<G>(c.g1, c.m1, u, P, gl) + u * c.dil;
  } else {
    r.o1 = support<G>(c.g1, c.m1, dir, P, gl);
  }
  r.o2 = support<G>(c.g2, c.m2, -dir, P, gl);
  r.p = r.o1 - r.o2;
  return r;
}

__device__ __forceinline__ bool same_bits(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }

// gjk::minkowski_ray_cast (src/query/algorithms/gjk.rs:245-365) on m1*g1 - m2*g2, ray (o, d), as a
// state that rc_step advances by one iteration.  The improved_fixed_point_support feature is off
// (the crate's default).
#define RC_RUNNING 0
#define RC_HIT 1
#define RC_MISS 2
struct RCState {
  f3 co, cd, ldir, proj;
  float ray_length, ltoi, max_bound;
  bool last_chance;
  int niter;
  int still;  // iterations since ltoi last changed
  SimplexR s;
};

// The loop is a deterministic function of the simplex's points and dimension, the ray origin and
// toi, the projection, max_bound and last_chance, and it ends in None after 10000 iterations.  So a
// cast whose values repeat, bit for bit, those of an earlier iteration is in a cycle that nothing
// but that cap ends: it returns None at once.  (A shift too small to change the origin with a
// support point the simplex rejects repeats at once.  About one time of impact in 10,000 of
// ball-capsule and capsule-capsule pairs does, and one such cast made a batch of 262,144 last 20 ms.)
// The toi never falls, so it is constant in a cycle: once it has been for RC_STILL iterations, the
// values of every 2^k-th such iteration are kept in RC_SNAP floats of LDS and those of the ones
// after it compared with them (Brent's cycle search).
#define RC_SNAP 21  // odd: the lanes' areas start in different banks
#define RC_STILL 8
__device__ __forceinline__ bool rc_repeats(const RCState& r, float* snap) {
  if (r.still < RC_STILL) return false;
  const bool keep = (r.still & (r.still - 1)) == 0;
  if (!keep) {  // the projection alone tells most iterations apart
    const uint32_t d = (__float_as_uint(snap[0]) ^ __float_as_uint(r.proj.x)) |
                       (__float_as_uint(snap[1]) ^ __float_as_uint(r.proj.y)) |
                       (__float_as_uint(snap[2]) ^ __float_as_uint(r.proj.z));
    if (d != 0) return false;
  }
  const int dim = r.s.dim;
  const f3 z = f3{0.f, 0.f, 0.f};
  const f3 v[6] = {r.proj, r.co, r.s.v0.p, sel3(dim >= 1, r.s.v1.p, z), sel3(dim >= 2, r.s.v2.p, z),
                   sel3(dim >= 3, r.s.v3.p, z)};
  const float w[3] = {r.max_bound, (float)dim, r.last_chance ? 1.f : 0.f};
  uint32_t diff = keep ? 1u : 0u;
#pragma unroll
  for (int i = 0; i < 21; ++i) {
    const f3 q = v[i < 18 ? i / 3 : 0];
    const float x = i < 18 ? (i % 3 == 0 ? q.x : (i % 3 == 1 ? q.y : q.z)) : w[i < 18 ? 0 : i - 18];
    diff |= __float_as_uint(snap[i]) ^ __float_as_uint(x);
    if (keep) snap[i] = x;
  }
  return diff == 0;
}

// The start of a cast, with its first support point.  Returns RC_MISS for a ray without a direction.
template <int G, int KIND = RC_ANY>
__device__ __forceinline__ int rc_begin(const RCtx& c, RCState& r, f3 ro, f3 rd, const Pool& P, int gl) {
  r.ray_length = norm(rd);
  if (relative_eq_zero(r.ray_length)) return RC_MISS;
  r.co = ro;
  r.cd = rd / r.ray_length;
  r.ldir = -r.cd;
  r.ltoi = 0.f;
  r.max_bound = NCX_FLT_MAX;
  r.last_chance = false;
  r.niter = 0;
  r.still = 0;
  sx_init(r.s);
  CSOR sp = cso_from_r<G, KIND>(c, r.ldir, P, gl);
  sp.p = sp.p + (-r.co);
  sx_reset(r.s, sp);
  r.proj = sx_project_reduce(r.s);
  return RC_RUNNING;
}

// One iteration.  RC_HIT: the toi is ltoi / ray_length and the normal ldir.  Casts that run for
// hundreds of iterations do so alone in their wavefront, so the step has few branches: updates that
// an iteration does not make are selects, or additions of -0, which change no value.
template <int G, int KIND = RC_ANY>
__device__ __forceinline__ int rc_step(const RCtx& c, float max_toi, RCState& r, const Pool& P, int gl, float* snap) {
  const float eps_tol = NCX_FLT_EPS * 10.f;
  const float eps_rel = __builtin_sqrtf(eps_tol);
  // try_normalize(-proj, eps_tol)
  const float dist = norm(-r.proj);
  const f3 dir = -r.proj / dist;
  const bool single = dist >= r.max_bound;  // CSOPoint::single_point (cso_point.rs:42-44)
  const bool lc = r.last_chance || single;
  if (dist <= eps_tol || (lc && r.ltoi > 0.f)) return RC_HIT;
  CSOR sp = cso_from_r<G, KIND>(c, dir, P, gl);
  const f3 pc = r.proj + r.co;
  sp.p = sel3(single, pc, sp.p);
  sp.o1 = sel3(single, pc, sp.o1);
  sp.o2 = sel3(single, f3{0.f, 0.f, 0.f}, sp.o2);
  // query::ray_toi_with_plane(support point, dir, curr_ray) (src/query/ray/ray_plane.rs:8-37)
  const float denom = dot(dir, r.cd);
  const float t = dot(dir, sp.p - r.co) / denom;
  const bool has_t = !relative_eq_zero(denom) && t >= 0.f;
  const bool moves = has_t && denom < 0.f && t > 0.f;
  const float ltoi = r.ltoi + t;
  const f3 shift = r.cd * t;
  r.still = moves && !same_bits(ltoi, r.ltoi) ? 0 : r.still + 1;
  r.ldir = sel3(moves, dir, r.ldir);
  r.ltoi = moves ? ltoi : r.ltoi;
  r.co = sel3(moves, r.co + shift, r.co);
  r.max_bound = moves ? NCX_FLT_MAX : dist;
  r.last_chance = lc && !moves;
  {  // VoronoiSimplex::modify_pnts over vertices 0..=dim (voronoi_simplex3.rs:347-351)
    const f3 z = f3{-0.f, -0.f, -0.f}, ns = -shift;
    r.s.v0.p = r.s.v0.p + sel3(moves, ns, z);
    r.s.v1.p = r.s.v1.p + sel3(moves && r.s.dim >= 1, ns, z);
    r.s.v2.p = r.s.v2.p + sel3(moves && r.s.dim >= 2, ns, z);
    r.s.v3.p = r.s.v3.p + sel3(moves && r.s.dim >= 3, ns, z);
  }
  const float min_bound = -dot(dir, sp.p - r.co);
  if ((moves && r.ltoi / r.ray_length > max_toi) || (!has_t && denom > eps_tol) || r.last_chance ||
      r.max_bound - min_bound <= eps_rel * r.max_bound)
    return RC_MISS;
  sp.p = sp.p + (-r.co);
  sx_add(r.s, sp);
  r.proj = sx_project_reduce(r.s);
  if (r.s.dim == 3) return min_bound >= eps_tol ? RC_MISS : RC_HIT;
  r.niter += 1;
  return r.niter == 10000 || rc_repeats(r, snap) ? RC_MISS : RC_RUNNING;
}

// The whole cast.  Returns false for None.  snap: RC_SNAP floats of LDS of this group's own.
template <int G>
__device__ __forceinline__ bool minkowski_ray_cast(const RCtx& c, f3 ro, f3 rd, float max_toi, RCState& r,
                                                   const Pool& P, int gl, float* snap, float& toi_out, f3& normal_out) {
  int st = rc_begin<G>(c, r, ro, rd, P, gl);
  while (st == RC_RUNNING) st = rc_step<G>(c, max_toi, r, P, gl, snap);
  toi_out = r.ltoi / r.ray_length;
  normal_out = r.ldir;
  return st == RC_HIT;
}

// ray_intersection_with_support_map_with_params (src/query/ray/ray_support_map.rs:15-62), shape
// at the identity (the callers pass a local-frame ray): the shape against ConstantOrigin.
__device__ __forceinline__ RCtx ray_ctx(const ShapeD& g) {
  RCtx c;
  c.m1 = iso_identity();
  c.m2 = iso_identity();
  c.g1 = g;
  c.g2.type = SHAPE_ORIGIN;
  c.dil = 0.f;
  c.dilated = false;
  c.local = true;
  return c;
}

// A ray that starts inside a shape that is not solid is cast back from a point past its far side:
// the second ray, and how far along the first its origin lies.
template <int G>
__device__ __forceinline__ float ray_from_behind(const RCtx& c, f3 ro, f3 rd, const Pool& P, int gl, f3& back) {
  const f3 ndir = normalize(rd);
  const f3 supp = support<G>(c.g1, c.m1, ndir, P, gl);
  const float shift = dot(supp - ro, ndir) + 0.001f;
  back = ro + ndir * shift;
  return shift;
}

template <int G>
__device__ __forceinline__ bool ray_support_map(const ShapeD& g, f3 ro, f3 rd, float max_toi, bool solid,
                                                const Pool& P, int gl, float* snap, float& toi, f3& normal) {
  const RCtx c = ray_ctx(g);
  RCState r;
  f3 o = ro, d = rd;
  float limit = max_toi, shift = 0.f;
  bool behind = false;
  for (;;) {  // one copy of the cast's code
    float t;
    f3 n;
    if (!minkowski_ray_cast<G>(c, o, d, limit, r, P, gl, snap, t, n)) return false;
    if (behind) t = shift - t;
    if (behind && !(t <= max_toi)) return false;
    if (behind || solid || t != 0.f) {
      toi = t;
      normal = n;
      return true;
    }
    behind = true;
    shift = ray_from_behind<G>(c, ro, rd, P, gl, o);
    d = -rd;
    limit = shift + 0.001f;
  }
}

// ray_toi_with_ball (src/query/ray/ray_ball.rs:83-124).
__device__ __forceinline__ bool ray_toi_with_ball(f3 center, float radius, f3 ro, f3 rd, bool solid, bool& inside,
                                                  float& toi) {
  const f3 dc = ro - center;
  const float a = norm_sq(rd);
  const float b = dot(dc, rd);
  const float c = norm_sq(dc) - radius * radius;
  inside = false;
  if (a == 0.f) {
    if (c > 0.f) return false;
    inside = true;
    toi = 0.f;
    return true;
  }
  if (c > 0.f && b > 0.f) return false;
  const float delta = b * b - a * c;
  if (delta < 0.f) return false;
  const float t = (-b - __builtin_sqrtf(delta)) / a;
  if (t <= 0.f) {
    inside = true;
    toi = solid ? 0.f : (-b + __builtin_sqrtf(delta)) / a;
    return true;
  }
  toi = t;
  return true;
}

#define NCX_FEAT_UNKNOWN 0xFFFFFFFEu

// AABB ray cast with normals: clip_line (src/query/ray/ray_aabb.rs:178-268) and ray_aabb
// (:270-290), local frame; side is +(i+1) / -(i+1) as in the reference.
__device__ __forceinline__ bool ray_box_normal(f3 h, f3 ro, f3 rd, float max_toi, bool solid, float& toi, f3& normal,
                                               int& side) {
  float tmax = NCX_FLT_MAX;
  float tmin = -tmax;
  int near_side = 0, far_side = 0;
  bool near_diag = false, far_diag = false;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float di = comp(rd, i), oi = comp(ro, i), hi = comp(h, i);
    if (di == 0.f) {
      if (oi < -hi || oi > hi) return false;
    } else {
      const float denom = 1.f / di;
      float tn = (-hi - oi) * denom;
      float tf = (hi - oi) * denom;
      const bool flip = tn > tf;
      if (flip) { float x = tn; tn = tf; tf = x; }
      if (tn > tmin) { tmin = tn; near_side = flip ? -(i + 1) : i + 1; near_diag = false; }
      else if (tn == tmin) near_diag = true;
      if (tf < tmax) { tmax = tf; far_side = !flip ? -(i + 1) : i + 1; far_diag = false; }
      else if (tf == tmax) far_diag = true;
      if (tmax < 0.f || tmin > tmax) return false;
    }
  }
  f3 nn = f3{0.f, 0.f, 0.f}, nf = nn;
  if (near_diag) nn = -normalize(rd);
  else if (near_side < 0) set_comp(nn, -near_side - 1, 1.f);
  else set_comp(nn, near_side - 1, -1.f);
  if (far_diag) nf = -normalize(rd);
  else if (far_side < 0) set_comp(nf, -far_side - 1, -1.f);
  else set_comp(nf, far_side - 1, 1.f);
  if (tmin < 0.f) {
    if (solid) { toi = 0.f; normal = f3{0.f, 0.f, 0.f}; side = far_side; return true; }
    if (tmax <= max_toi) { toi = tmax; normal = nf; side = far_side; return true; }
    return false;
  }
  if (tmin <= max_toi) { toi = tmin; normal = nn; side = near_side; return true; }
  return false;
}

// RayCast::toi_and_normal_with_ray of Ball (src/query/ray/ray_ball.rs:32-43, 127-142), Cuboid
// (ray_cuboid.rs:17-26 -> ray_aabb.rs:45-61), Capsule and ConvexHull (ray_support_map.rs:117-163:
// local-frame ray, normal rotated back).  feature: face id, 0 for a ball, NCX_FEAT_UNKNOWN for
// support-map shapes.
// The closed forms (Ball, Cuboid) of shape_ray_cast below; no cross-lane work, so one lane can
// cast a ray alone.  A shape of another type gives no hit.
__device__ __forceinline__ bool shape_ray_cast_closed(const ShapeD& g, const iso& m, f3 ro, f3 rd, float max_toi,
                                                      bool solid, float& toi, f3& normal, uint32_t& feature) {
  if (g.type == NCX_BALL) {
    bool inside;
    float t;
    if (!ray_toi_with_ball(m.t, g.a, ro, rd, solid, inside, t)) return false;
    const f3 n = normalize((ro + rd * t) - m.t);
    if (!(t <= max_toi)) return false;
    toi = t;
    normal = inside ? -n : n;
    feature = 0;
    return true;
  }
  if (g.type == NCX_CUBOID) {
    const f3 lo = inv_xform_pt(m, ro), ld = inv_xform_vec(m, rd);
    float t;
    f3 n;
    int side;
    if (!ray_box_normal(f3{g.a, g.b, g.c}, lo, ld, max_toi, solid, t, n, side)) return false;
    toi = t;
    normal = xform_vec(m, n);
    feature = side < 0 ? (uint32_t)(-side - 1 + 3) : (uint32_t)(side - 1);
    return true;
  }
  return false;
}

template <int G>
__device__ __forceinline__ bool shape_ray_cast(const ShapeD& g, const iso& m, f3 ro, f3 rd, float max_toi, bool solid,
                                               const Pool& P, int gl, float* snap, float& toi, f3& normal,
                                               uint32_t& feature) {
  if (g.type == NCX_BALL || g.type == NCX_CUBOID)
    return shape_ray_cast_closed(g, m, ro, rd, max_toi, solid, toi, normal, feature);
  if (g.type == NCX_CAPSULE || g.type == NCX_CONVEX_HULL) {
    const f3 lo = inv_xform_pt(m, ro), ld = inv_xform_vec(m, rd);
    float t;
    f3 n;
    if (!ray_support_map<G>(g, lo, ld, max_toi, solid, P, gl, snap, t, n)) return false;
    toi = t;
    normal = xform_vec(m, n);
    feature = NCX_FEAT_UNKNOWN;
    return true;
  }
  return false;
}

// ------------------------------------------------------------------ triangles and isometries for composite shapes
// approx::relative_eq!(x, y) with the default epsilon and max_relative (f32::EPSILON).
__device__ __forceinline__ bool relative_eq_f(float x, float y) {
  if (x == y) return true;
  if (__builtin_isinf(x) || __builtin_isinf(y)) return false;
  const float d = fabsf(x - y);
  if (d <= NCX_FLT_EPS) return true;
  const float ax = fabsf(x), ay = fabsf(y);
  return d <= (ay > ax ? ay : ax) * NCX_FLT_EPS;
}

// Triangle::project_point_with_location with solid = true (src/query/point/point_triangle.rs:61-240)
// for the triangle (a, b, c) placed by m: the projection in the world frame; *inside is the
// PointProjection's is_inside (relative_eq!(projection, pt) in 3D, :6-19; true on the solid
// branch).
__device__ __forceinline__ f3 proj_triangle_at(const iso& m, f3 a, f3 b, f3 c, f3 pt, Loc& loc, bool& inside) {
  const f3 p = inv_xform_pt(m, pt);
  const f3 ab = b - a, ac = c - a, ap = p - a;
  const float ab_ap = dot(ab, ap), ac_ap = dot(ac, ap);
  f3 res;
  if (ab_ap <= 0.f && ac_ap <= 0.f) { loc.kind = LOC_VERTEX; loc.id = 0; res = xform_pt(m, a); }
  else {
    const f3 bp = p - b;
    const float ab_bp = dot(ab, bp), ac_bp = dot(ac, bp);
    if (ab_bp >= 0.f && ac_bp <= ab_bp) { loc.kind = LOC_VERTEX; loc.id = 1; res = xform_pt(m, b); }
    else {
      const f3 cp = p - c;
      const float ab_cp = dot(ab, cp), ac_cp = dot(ac, cp);
      if (ac_cp >= 0.f && ab_cp <= ac_cp) { loc.kind = LOC_VERTEX; loc.id = 2; res = xform_pt(m, c); }
      else {
        const f3 bc = c - b;
        const f3 n = cross(ab, ac);
        const float vc = dot(n, cross(ab, ap));
        const float vb = -dot(n, cross(ac, cp));
        const float va = dot(n, cross(bc, bp));
        if (vc < 0.f && ab_ap >= 0.f && ab_bp <= 0.f) {
          const float v = ab_ap / norm_sq(ab);
          loc.kind = LOC_EDGE; loc.id = 0; loc.bc0 = 1.f - v; loc.bc1 = v;
          res = xform_pt(m, a + ab * v);
        } else if (vb < 0.f && ac_ap >= 0.f && ac_cp <= 0.f) {
          const float w = ac_ap / norm_sq(ac);
          loc.kind = LOC_EDGE; loc.id = 2; loc.bc0 = 1.f - w; loc.bc1 = w;
          res = xform_pt(m, a + ac * w);
        } else if (va < 0.f && ac_bp - ab_bp >= 0.f && ab_cp - ac_cp >= 0.f) {
          const float w = dot(bc, bp) / norm_sq(bc);
          loc.kind = LOC_EDGE; loc.id = 1; loc.bc0 = 1.f - w; loc.bc1 = w;
          res = xform_pt(m, b + bc * w);
        } else if (va + vb + vc != 0.f) {
          const float denom = 1.f / (va + vb + vc);
          const float v = vb * denom, w = vc * denom;
          loc.kind = LOC_FACE; loc.id = dot(n, ap) >= 0.f ? 0 : 1;
          loc.bc0 = 1.f - v - w; loc.bc1 = v; loc.bc2 = w;
          res = xform_pt(m, a + ab * v + ac * w);
        } else {
          loc.kind = LOC_SOLID; loc.id = 0;
          inside = true;
          return pt;
        }
      }
    }
  }
  inside = relative_eq_f(res.x, pt.x) && relative_eq_f(res.y, pt.y) && relative_eq_f(res.z, pt.z);
  return res;
}

// Segment::project_point_with_location (src/query/point/point_segment.rs:49-91) for the segment
// (a, b) placed by m, and project_point_with_feature's feature (:13-41): vertex 0 or 1 (kind
// LOC_VERTEX) or the edge (LOC_EDGE).  *inside = relative_eq!(projection, pt).
__device__ __forceinline__ f3 proj_segment_at(const iso& m, f3 a, f3 b, f3 pt, int& kind, int& id, bool& inside) {
  const f3 ls = inv_xform_pt(m, pt);
  const f3 ab = b - a, ap = ls - a;
  const float ab_ap = dot(ab, ap), sqnab = norm_sq(ab);
  f3 proj;
  if (ab_ap <= 0.f) { kind = LOC_VERTEX; id = 0; proj = xform_pt(m, a); }
  else if (ab_ap >= sqnab) { kind = LOC_VERTEX; id = 1; proj = xform_pt(m, b); }
  else {
    const float u = ab_ap / sqnab;
    kind = LOC_EDGE; id = 0;
    proj = xform_pt(m, a + ab * u);
  }
  inside = relative_eq_f(proj.x, pt.x) && relative_eq_f(proj.y, pt.y) && relative_eq_f(proj.z, pt.z);
  return proj;
}

// Segment::feature_normal (src/shape/segment.rs:238-273), local frame, for the segment (a, b):
// vertex 0 -> its direction, vertex 1 -> minus it, the edge -> the unit vector along the
// direction's smallest component with the direction's part removed; +y when degenerate.
__device__ __forceinline__ f3 segment_feature_normal(f3 a, f3 b, int kind, int id) {
  f3 d;
  float nl;
  if (!try_normalize(b - a, NCX_FLT_EPS, &d, &nl)) return f3{0.f, 1.f, 0.f};
  if (kind == LOC_VERTEX) return id == 0 ? d : -d;
  // Vector::iamin: the first index of the smallest |component|
  int im = 0;
  float best = fabsf(d.x);
  if (fabsf(d.y) < best) { best = fabsf(d.y); im = 1; }
  if (fabsf(d.z) < best) im = 2;
  f3 n = f3{0.f, 0.f, 0.f};
  set_comp(n, im, 1.f);
  n = n - d * comp(d, im);
  return normalize(n);
}

// Quaternion product (nalgebra's Quaternion * Quaternion), coordinates (i, j, k, w).
__device__ __forceinline__ quat quat_mul(quat a, quat b) {
  quat r;
  r.w = ((a.w * b.w - a.i * b.i) - a.j * b.j) - a.k * b.k;
  r.i = ((a.w * b.i + a.i * b.w) + a.j * b.k) - a.k * b.j;
  r.j = ((a.w * b.j - a.i * b.k) + a.j * b.w) + a.k * b.i;
  r.k = ((a.w * b.k + a.i * b.j) - a.j * b.i) + a.k * b.w;
  return r;
}

// m1.inverse() * m2 (nalgebra Isometry::inverse then Isometry * Isometry): rotation q1^-1 q2,
// translation q1^-1 (-t1) + q1^-1 t2.
__device__ __forceinline__ iso iso_inv_mul(const iso& m1, const iso& m2) {
  const quat qi = quat{-m1.q.i, -m1.q.j, -m1.q.k, m1.q.w};
  iso r;
  const f3 t_inv = qrot(qi, -m1.t);
  r.t = t_inv + qrot(qi, m2.t);
  r.q = quat_mul(qi, m2.q);
  return r;
}

// |R| h of a cuboid rotated by q (isometry_ops.rs:43-45 through UnitQuaternion::to_rotation_matrix).
__device__ __forceinline__ f3 cuboid_world_half(quat q, float hx, float hy, float hz) {
  const float qi = q.i, qj = q.j, qk = q.k, qw = q.w;
  const float ww = qw * qw, ii = qi * qi, jj = qj * qj, kk = qk * qk;
  const float ij = qi * qj * 2.f, wk = qw * qk * 2.f, wj = qw * qj * 2.f;
  const float ik = qi * qk * 2.f, jk = qj * qk * 2.f, wi = qw * qi * 2.f;
  const float M[3][3] = {{ww + ii - jj - kk, ij - wk, wj + ik},
                         {wk + ij, ww - ii + jj - kk, jk - wi},
                         {ik - wj, wi + jk, ww - ii - jj + kk}};
  f3 ws;
  ws.x = (fabsf(M[0][0]) * hx + fabsf(M[0][1]) * hy) + fabsf(M[0][2]) * hz;
  ws.y = (fabsf(M[1][0]) * hx + fabsf(M[1][1]) * hy) + fabsf(M[1][2]) * hz;
  ws.z = (fabsf(M[2][0]) * hx + fabsf(M[2][1]) * hy) + fabsf(M[2][2]) * hz;
  return ws;
}

// Shape::aabb at m (aabb_ball.rs:8-13, aabb_cuboid.rs:7-14, aabb_support_map.rs:35-45,
// aabb_convex.rs:7-11 -> aabb_utils.rs:59-79), every lane of a group of G the same result (the
// hull's points split over the lanes; a min/max does not depend on the order).
template <int G>
__device__ __forceinline__ void shape_aabb_g(const ShapeD& g, const iso& m, const Pool& P, int gl, f3& mn, f3& mx) {
  if (g.type == NCX_BALL) {
    mn = m.t + f3{-g.a, -g.a, -g.a};
    mx = m.t + f3{g.a, g.a, g.a};
  } else if (g.type == NCX_CUBOID) {
    const f3 ws = cuboid_world_half(m.q, g.a, g.b, g.c);
    mn = m.t - ws;
    mx = m.t + ws;
  } else if (g.type == NCX_CAPSULE) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      f3 e = f3{0.f, 0.f, 0.f};
      set_comp(e, d, 1.f);
      set_comp(mx, d, comp(support<1>(g, m, e, P, 0), d));
      set_comp(e, d, -1.f);
      set_comp(mn, d, comp(support<1>(g, m, e, P, 0), d));
    }
  } else {
    f3 lo = f3{__builtin_inff(), __builtin_inff(), __builtin_inff()};
    f3 hi = -lo;
    for (uint32_t v = gl; v < g.cnt; v += G) {
      const f3 p = xform_pt(m, f3{P.x[g.off + v], P.y[g.off + v], P.z[g.off + v]});
      lo = f3{fminf(lo.x, p.x), fminf(lo.y, p.y), fminf(lo.z, p.z)};
      hi = f3{fmaxf(hi.x, p.x), fmaxf(hi.y, p.y), fmaxf(hi.z, p.z)};
    }
#pragma unroll
    for (int o = G / 2; o >= 1; o >>= 1) {
      lo.x = fminf(lo.x, __shfl_xor(lo.x, o, 64)); lo.y = fminf(lo.y, __shfl_xor(lo.y, o, 64));
      lo.z = fminf(lo.z, __shfl_xor(lo.z, o, 64));
      hi.x = fmaxf(hi.x, __shfl_xor(hi.x, o, 64)); hi.y = fmaxf(hi.y, __shfl_xor(hi.y, o, 64));
      hi.z = fmaxf(hi.z, __shfl_xor(hi.z, o, 64));
    }
    mn = lo;
    mx = hi;
  }
}
