// HIP kernels for gfx950: closest-hit traversal of one geometry-type BVH per launch.
//
// FP64 path (the drop-in): bit-identical to blazeRT's traverse() (blazert/bvh/accel.h:79-120). The reference
// pops a node, slab-tests it against [tmin, current hit] and pushes far then near. Here an internal record holds
// both child boxes: the near child is tested at the parent (the reference tests it at the very next pop, with the
// same hit distance), and the far child goes on the stack with the h-independent half of its slab test already
// applied and its entry distance as the key, so the pop-time check `!(h < key)` reproduces the reference's
// decision exactly, NaN propagation of std::max/std::min included (blazert/bvh/intersect.h:32-51).
//
// FP32 path (split precision): the same DFS with slab tests on outward-rounded FP32 child boxes and a per-ray
// absolute error bound, so it visits a superset of the FP64 path's nodes; primitive tests stay FP64.
//
// All arithmetic is compiled with -ffp-contract=off so that products and sums round exactly as the reference's.
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include <hipcub/hipcub.hpp>

#include "../../include/blazert_amd/device/exact.h"
#include "engine.h"
#include "f32_round.h"
#include "wave.h"

namespace brt {

namespace {

constexpr uint32_t PREC_FP64 = 0;
constexpr uint32_t FLAG_INOUT = 1u;
constexpr uint32_t FLAG_ANY_HIT = 2u;
// Internal: an FP64 launch that traces only the rays a split-precision launch of the same geometry type deferred
// (see deferred_to_exact), and none at all when that launch deferred nothing.
constexpr uint32_t FLAG_DEFERRED_ONLY = 1u << 31;
constexpr uint32_t FLAG_SPLIT = 1u << 30;  // k_trace_tri and the launch behind it: split precision
// Exact paths: primitives of a leaf tested per traversal step, per primitive type (triangles, spheres, planes,
// cylinders). They are tested in leaf order, each against the hit distance the previous one left, so the count
// changes speed only.
#ifndef BRT_EXACT_GROUP_TRI
#define BRT_EXACT_GROUP_TRI 2  // 1.31M-triangle incoherent set: 2-3% faster than 1, bit-identical hits
#endif
#ifndef BRT_EXACT_GROUP_SPH
#define BRT_EXACT_GROUP_SPH 1  // mixed scene: 2 and 4 per step 4% and 15% slower (the FP64 sphere test is long)
#endif
#ifndef BRT_EXACT_GROUP_PLA
#define BRT_EXACT_GROUP_PLA 1  // mixed scene: 2 per step 13% slower
#endif
#ifndef BRT_EXACT_GROUP_CYL
#define BRT_EXACT_GROUP_CYL 1  // mixed scene: 2 per step 18% slower
#endif
template <uint32_t KIND>
constexpr int exact_group() {
  return KIND == TRIANGLES ? BRT_EXACT_GROUP_TRI
         : KIND == SPHERES ? BRT_EXACT_GROUP_SPH
         : KIND == PLANES  ? BRT_EXACT_GROUP_PLA
                           : BRT_EXACT_GROUP_CYL;
}

// Deepest stack a traversal can build: the binary FP64 DFS pushes at most one entry per level (trees are limited
// to depth 63 at upload); the 4-wide FP32 DFS at most three per Node4 record, and a record spans at least one
// binary level on every path, so at most 3 * 63 = 189.
template <bool SPLIT>
constexpr int stack_cap() { return SPLIT ? 192 : 64; }

// The reference's ray setup and exact slab test (Real, RayT, setup_ray, slab_exact, product_sign, dsqrt) are shared
// with user-collection traversal: include/blazert_amd/device/exact.h.
using namespace exact;
using Ray = RayT<double>;

// Rays the split-precision path hands to the exact FP64 path: those whose reference slab test can produce a NaN
// term or culls boxes its line crosses, i.e. every ray without RAY_NAN_FREE (a zero, non-finite or reciprocal-
// overflowing direction component, a non-finite origin, a NaN tmin). For a raw component -0.0 the reference takes
// the near plane from `direction < 0` (false) but multiplies by 1/-0.0 = -inf, so it culls every box the ray's line
// lies in; an origin on a box plane of a zero component gives 0 * inf = NaN. The FP32 path's |1/d| > 1e30 axes
// never cull, so on such rays it would reach primitives the reference cannot. Every other ray has NaN-free slab
// terms in the reference, and the FP32 path's conservative boxes visit a superset of its nodes.
template <class R>
__device__ __forceinline__ bool deferred_to_exact(const RayT<R> &r) {
  return !(r.sign & RAY_NAN_FREE);
}

// A pointer into device memory viewed in the global address space. Pointers loaded from memory (the batch kernel's
// job table) are generic, and accesses through generic pointers are flat accesses; through this view they are global.
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gmem(T *p) {
  return (__attribute__((address_space(1))) T *)p;
}

// Rays are read once and hits written once per launch: streamed with non-temporal hints, so that they do not evict
// the tree's lines from the caches (a launch of 4M rays streams ~335 MB, more than the last-level cache).
template <class T>
__device__ __forceinline__ T ld_stream(const T *p, uint64_t i) {
  return __builtin_nontemporal_load(gmem(p) + i);
}
template <class T, class V>
__device__ __forceinline__ void st_stream(T *p, uint64_t i, V v) {
  __builtin_nontemporal_store((T)v, gmem(p) + i);
}

template <class R>
__device__ __forceinline__ void make_ray(const RaysViewT<R> &V, uint64_t i, RayT<R> &r) {
  const R org[3] = {ld_stream(V.ox, i), ld_stream(V.oy, i), ld_stream(V.oz, i)};
  const R raw[3] = {ld_stream(V.dx, i), ld_stream(V.dy, i), ld_stream(V.dz, i)};
  setup_ray(org, raw, V.tmin ? ld_stream(V.tmin, i) : V.tmin0, V.tmax ? ld_stream(V.tmax, i) : V.tmax0, r);
}

// Conservative FP32 slab test: per axis lower/upper bounds of the FP64 entry/exit distances.
struct Ray32 {
  float inv[3];
  float offn[3];  // rounded-down (-o*inv - E)
  float offf[3];  // rounded-up   (-o*inv + E)
  float tmin;     // rounded down
  float om;       // max |o_i| rounded up; +inf when above FILTER_MAX_EXTENT (no FP32 triangle pre-test)
  uint32_t sign;
};

// E_i = 5 * 2^-24 * |inv_i| * (S + |o_i|) bounds |fma(b32, inv32, off32) - (b - o) inv| for every |b| <= S,
// including the FP64 reference's own rounding and its 1 + 4 eps far-plane factor. For a Scene<float>, whose reference rounds
// its two operations (2 units u = 2^-24), and the far-plane factor's 8 u, in FP32, the factor is 16 and the denormal range
// (its results' and the fma's) adds 1e-40.
template <bool F32 = false>
__device__ __forceinline__ void make_ray32(const Ray &r, double S, Ray32 &q) {
  q.sign = r.sign;
  q.tmin = f32_down(r.tmin);
  const double om = fmax(fabs(r.o[0]), fmax(fabs(r.o[1]), fabs(r.o[2])));
  q.om = om <= FILTER_MAX_EXTENT ? f32_up(om) : __builtin_inff();
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const double inv = r.inv[i];
    const double ainv = fabs(inv);
    if (!(ainv <= 1e30)) {  // zero / tiny direction component: this axis never culls
      q.inv[i] = 0.0f;
      q.offn[i] = -__builtin_inff();
      q.offf[i] = __builtin_inff();
      continue;
    }
    const double off = -(r.o[i] * inv);
    const double E = (F32 ? 16.0 : 5.0) * 5.9604644775390625e-08 * ainv * (S + fabs(r.o[i])) + (F32 ? 1e-40 : 0.0);
    q.inv[i] = (float)inv;
    q.offn[i] = f32_down(off - E);
    q.offf[i] = f32_up(off + E);
  }
}

__device__ __forceinline__ bool slab32(const float *b, const Ray32 &q, float &key) {
  float A = q.tmin;
  float M = __builtin_inff();
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const bool s = (q.sign >> i) & 1u;
    const float nearp = s ? b[3 + i] : b[i];
    const float farp = s ? b[i] : b[3 + i];
    A = fmaxf(A, __builtin_fmaf(nearp, q.inv[i], q.offn[i]));
    M = fminf(M, __builtin_fmaf(farp, q.inv[i], q.offf[i]));
  }
  key = A;
  return A <= M;
}

// Conservative FP32 pre-test of one triangle for the split path: returns false only when the FP64 test isect_tri
// (blazert/primitives/trimesh.h:153-181) rejects the triangle for the ray at the current hit distance h <= h32.
//
// With u = 2^-24, Pm = vmax + om >= |v0_i| + |o_i|, sa = sum |e1_i|, sb = sum |e2_i|, the values computed here from
// v0, e1, e2, n and o rounded to nearest and the unit direction d rounded to nearest differ from the exact ones (and
// from the FP64 test's, whose own rounding is ~2^-29 smaller) by at most
//   u, v:  13.1 u Pm sb and 13.1 u Pm sa     (c = v0 - o: 2.01 u Pm per component; r = d x c: 5.1 u sqrt2 Pm)
//   det:    5.1 u sa sb                      (n rounded once from the FP64 test's own n)
//   t:      6.1 u sa sb Pm
//   w = |det| - u - v: the sum of those plus 2 u (|det| + |u| + |v|) <= 0.2 Ed + 0.18 (Eu + Ev)
// The bounds used (Ed = ed, Et = 1.2 ed Pm, and for u, v and w alike E = kw Pm + cw, with kw = 1.2 * 16 u (sa + sb) and
// cw = 1.3 ed + tol) keep a margin for the rounding of the bounds themselves; ed and Et hold an absolute 1e-29, E the
// reference's tolerance, for results in the FP32 denormal range. The reference accepts u, v, w >= -4 DBL_EPSILON (tol),
// t >= |det| tmin and |det| h > t with the signs
// taken from det; where the sign of det is not certain (|det| <= Ed) the triangle passes. Scenes and ray origins
// above FILTER_MAX_EXTENT are not pre-tested, so no value here overflows; every rejection is a comparison that is
// false for NaN operands.
__device__ __forceinline__ bool tri_filter(const TriFilt &T, const float D[3], const float O[3], float om,
                                           float tmin32, float h32) {
  const float u = 5.9604644775390625e-08f;
  // fused multiply-adds round once where a product and a sum round twice, so the bounds below hold for them too
  auto dot3 = [](float a0, float a1, float a2, float b0, float b1, float b2) {
    return __builtin_fmaf(a0, b0, __builtin_fmaf(a1, b1, a2 * b2));
  };
  const float det = dot3(T.n[0], T.n[1], T.n[2], D[0], D[1], D[2]);
  const float ad = fabsf(det);
  const float c0 = T.v0[0] - O[0], c1 = T.v0[1] - O[1], c2 = T.v0[2] - O[2];
  const float rx = __builtin_fmaf(D[1], c2, -(D[2] * c1));
  const float ry = __builtin_fmaf(D[2], c0, -(D[0] * c2));
  const float rz = __builtin_fmaf(D[0], c1, -(D[1] * c0));
  const float Pm = T.vmax + om;
  const float *a = T.e1, *b = T.e2;
  const float us = product_sign(dot3(rx, ry, rz, b[0], b[1], b[2]), det);
  const float vs = product_sign(dot3(rx, ry, rz, a[0], a[1], a[2]), det);
  const float E = __builtin_fmaf(T.kw, Pm, T.cw);
  const float ts = product_sign(dot3(T.n[0], T.n[1], T.n[2], c0, c1, c2), det);
  const float Et = __builtin_fmaf(1.2f * T.ed, Pm, 1e-29f);
  // t >= |det| tmin: a lower bound of the right side (tmin32 <= tmin; none for negative tmin)
  const float L = (ad - T.ed) * (tmin32 >= 0.0f ? tmin32 * (1.0f - 4.0f * u) : -__builtin_inff());
  // |det| h > t: an upper bound of the left side (h32 >= h)
  const float H = (ad + T.ed) * (h32 * (1.0f + 4.0f * u));
  // without branches: lanes of a wave rarely agree on one, and the tests of a group overlap
  const bool out = (fminf(fminf(us, vs), (ad - us) - vs) < -E) | (ts + Et < L) | (ts - Et >= H);
  return !(ad > T.ed) | !out;  // where the sign of det is not certain the triangle passes
}

// Conservative FP32 pre-test of one sphere for the split path: returns false only when the FP64 test isect_sph
// (blazert/primitives/sphere.h:364-406) reports no hit for the ray at the current hit distance h <= h32.
//
// The FP64 test computes, from v = o - c and the unit direction d, A = d.d, B = 2 v.d, C = v.v - r r and
// D = B B - 4 A C, and accepts a root t = (-B -+ sqrt(D)) / 2A with tmin < t < h when D >= 0. With exact arithmetic
// on its inputs D = 4 (A r^2 - |v x d|^2); its roundings move D by at most 1e-13 (P^2 + r^2), where
// P >= |c_i| + |o_i| (P = (max |c32_i| + om) (1 + 4u), u = 2^-24). So
//   (a) D < 0 whenever |v x d| > r + 1.61e-7 (P + r), and
//   (b) every root lies within r + 1.61e-7 (P + r) of -v.d.
// Here v, v x d (one FMA per component) and v.d are computed in FP32 from the rounded center, origin and direction:
// each component of v is within 2.01 u P of the exact one, v x d within 12 u P (as a vector) and v.d within 10 u P.
// The record's radius is |r| rounded up. The test rejects when |v x d| in FP32 exceeds the radius plus both error
// terms (compared as squares, each rounding covered by a factor), or when the interval of (b), widened by the error
// of -v.d and the rounding of its ends, lies below tmin32 <= tmin or at or above h32 >= h (s.h carries the FP64 unit
// direction's norm, within 4 DBL_EPSILON of 1: covered by the 1 + 4u factor). A radius term below 1e-18, whose
// square would fall in the FP32 denormal range, skips test (a). Scenes and origins above FILTER_MAX_EXTENT are not
// pre-tested, and every rejection is a comparison that is false for NaN operands.
__device__ __forceinline__ bool sph_filter(const SphFilt &S, const float D[3], const float O[3], float om,
                                           float tmin32, float h32) {
  const float u = 5.9604644775390625e-08f;
  const float cm = fmaxf(fabsf(S.c[0]), fmaxf(fabsf(S.c[1]), fabsf(S.c[2])));
  const float P = (cm + om) * (1.0f + 4.0f * u);
  const float v0 = O[0] - S.c[0], v1 = O[1] - S.c[1], v2 = O[2] - S.c[2];
  const float wx = __builtin_fmaf(v1, D[2], -(v2 * D[1]));
  const float wy = __builtin_fmaf(v2, D[0], -(v0 * D[2]));
  const float wz = __builtin_fmaf(v0, D[1], -(v1 * D[0]));
  const float dist2 = __builtin_fmaf(wx, wx, __builtin_fmaf(wy, wy, wz * wz));
  const float e64 = __builtin_fmaf(1.61e-7f, P + S.r, 1e-30f);  // the FP64 test's own rounding, as a distance
  const float R = (S.r + __builtin_fmaf(12.0f * u, P, e64)) * (1.0f + 4.0f * u);
  if (R >= 1e-18f && dist2 * (1.0f - 8.0f * u) > (R * R) * (1.0f + 4.0f * u)) return false;
  const float tc = -__builtin_fmaf(v0, D[0], __builtin_fmaf(v1, D[1], v2 * D[2]));
  float rho = S.r + __builtin_fmaf(10.0f * u, P, e64);
  rho = __builtin_fmaf(4.0f * u, fabsf(tc) + rho, rho);
  if (tc + rho < tmin32) return false;
  if (tc - rho >= h32 * (1.0f + 4.0f * u)) return false;
  return true;
}

// Conservative FP32 pre-test of one cylinder: returns false only when the FP64 test cyl_eval
// (blazert/primitives/cylinder.h:181-495) reports no hit, whatever the hit distance (its last hit counts, at any t >= 0).
//
// A hit's point lies in the bounding sphere (sph_filter with the window [0, inf)), and the ray's line, projected along the
// axis, reaches the ellipse of semi-axes a, b: in the local frame (org, dir) = R^T (o - c, d) the shell's quadratic needs
// T^2 <= a^2 k^2 + b^2 j^2 for T = j y0 - k x0, a cap's point is on or in the ellipse and so is an origin inside, up to
// roundings of 2e-15 (P^2 + max(a,b)^2) in T^2. T = (o - c) . (d x axis) for the record's axis, and the right side is at most
// max(a,b)^2 (|d x axis|^2 + 1e-5) for a rotation within 1e-6 of orthonormal (others have infinite radii and pass). In FP32 T
// is within 27 u P, u = 2^-24; the test rejects when it is outside by 32 u P, whose square covers the FP64 roundings too. A
// semi-axis below 1e-15, with which the right side could fall in the FP32 denormal range, is recorded as infinite.
__device__ __forceinline__ bool cyl_filter(const CylFilt &C, const float D[3], const float O[3], float om) {
  const float u = 5.9604644775390625e-08f;
  const SphFilt sphere{{C.c[0], C.c[1], C.c[2]}, C.r};
  const float cm = fmaxf(fabsf(C.c[0]), fmaxf(fabsf(C.c[1]), fabsf(C.c[2])));
  const float P = (cm + om) * (1.0f + 4.0f * u);
  const float v0 = O[0] - C.c[0], v1 = O[1] - C.c[1], v2 = O[2] - C.c[2];
  const float nx = __builtin_fmaf(D[1], C.axis[2], -(D[2] * C.axis[1]));
  const float ny = __builtin_fmaf(D[2], C.axis[0], -(D[0] * C.axis[2]));
  const float nz = __builtin_fmaf(D[0], C.axis[1], -(D[1] * C.axis[0]));
  const float n2 = __builtin_fmaf(nx, nx, __builtin_fmaf(ny, ny, nz * nz));
  const float T = fabsf(__builtin_fmaf(v0, nx, __builtin_fmaf(v1, ny, v2 * nz))) - 32.0f * u * P;
  if (T > 0.0f && T * T > (C.shell * C.shell) * (n2 * (1.0f + 16.0f * u) + 2e-5f)) return false;
  return sph_filter(sphere, D, O, om, 0.0f, __builtin_inff());
}

// ------------------------------------------------------------------------------------------------ intersectors
// Closest-hit state of one traversal (prepare_traversal: hit = tmax, uv = 0, prim invalid).
template <class R>
struct HitT {
  R h;
  R u, v;
  uint32_t leaf_idx;  // leaf-order index of the current hit; the user primitive id for records that carry it
};

// FP64 triangle records carry their user primitive id (TriRec::prim).
template <class Rec>
__device__ constexpr bool id_in_record() {
  return std::is_same<Rec, TriRec>::value;
}
using Hit = HitT<double>;

// Every intersector runs in the scene type of its record (Rec::real): the same operation sequence for double and
// float, with the reference's constants of that type.

// blazert/primitives/trimesh.h:153-181. accepted(u, v, w, t, |det|, |det| h) is called on a hit, before s is updated.
template <class Rec, class F>
__device__ __forceinline__ bool isect_tri(const Rec &T, const RayT<typename Rec::real> &r,
                                          HitT<typename Rec::real> &s, uint32_t idx, F accepted) {
  using R = typename Rec::real;
  const R tol = R(4) * Real<R>::eps;
  const R c0 = T.v0[0] - r.o[0], c1 = T.v0[1] - r.o[1], c2 = T.v0[2] - r.o[2];
  const R rx = r.d[1] * c2 - r.d[2] * c1;
  const R ry = r.d[2] * c0 - r.d[0] * c2;
  const R rz = r.d[0] * c1 - r.d[1] * c0;
  const R *e1 = T.e1, *e2 = T.e2;
  R nx, ny, nz;  // cross(e1, e2)
  if constexpr (Rec::has_normal) {
    nx = T.n[0];
    ny = T.n[1];
    nz = T.n[2];
  } else {
    R n[3];
    tri_normal(e1, e2, n);
    nx = n[0];
    ny = n[1];
    nz = n[2];
  }
  const R det = nx * r.d[0] + ny * r.d[1] + nz * r.d[2];
  const R abs_det = fabs(det);
  const R u = product_sign(rx * e2[0] + ry * e2[1] + rz * e2[2], det);
  const R v = product_sign(rx * e1[0] + ry * e1[1] + rz * e1[2], det);
  const R w = abs_det - u - v;
  if (u >= -tol && v >= -tol && w >= -tol) {
    const R t = product_sign(nx * c0 + ny * c1 + nz * c2, det);
    if (t >= abs_det * r.tmin && abs_det * s.h > t) {
      accepted(u, v, w, t, abs_det, abs_det * s.h);
      const R inv_det = R(1) / abs_det;
      s.h = t * inv_det;
      s.u = u * inv_det;
      s.v = v * inv_det;
      if constexpr (id_in_record<Rec>()) s.leaf_idx = (uint32_t)T.prim;
      else s.leaf_idx = idx;
      return true;
    }
  }
  return false;
}

template <class Rec>
__device__ __forceinline__ bool isect_tri(const Rec &T, const RayT<typename Rec::real> &r,
                                          HitT<typename Rec::real> &s, uint32_t idx) {
  using R = typename Rec::real;
  return isect_tri(T, r, s, idx, [](R, R, R, R, R, R) {});
}

template <class R>
__device__ __forceinline__ R norm_scaled(R t, const R *d) {
  const R x = t * d[0], y = t * d[1], z = t * d[2];
  return dsqrt(x * x + y * y + z * z);
}

// blazert/primitives/sphere.h:364-406
template <class Rec>
__device__ __forceinline__ bool isect_sph(const Rec &S, const RayT<typename Rec::real> &r,
                                          HitT<typename Rec::real> &s, uint32_t idx) {
  using R = typename Rec::real;
  const R v0 = r.o[0] - S.c[0], v1 = r.o[1] - S.c[1], v2 = r.o[2] - S.c[2];
  const R A = r.d[0] * r.d[0] + r.d[1] * r.d[1] + r.d[2] * r.d[2];
  const R B = R(2) * (v0 * r.d[0] + v1 * r.d[1] + v2 * r.d[2]);
  const R C = (v0 * v0 + v1 * v1 + v2 * v2) - S.r * S.r;
  const R D = B * B - R(4) * A * C;
  if (D < R(0)) return false;
  const R Q = dsqrt(D);
  const R rcpA = R(1) / A;
  const R t0 = R(0.5) * rcpA * (-B - Q);
  const R t1 = R(0.5) * rcpA * (-B + Q);
  if ((t0 > r.tmin) && (t0 < s.h)) {
    s.h = norm_scaled(t0, r.d);
    s.leaf_idx = idx;
    return true;
  }
  if ((t1 > r.tmin) && (t1 < s.h)) {
    s.h = norm_scaled(t1, r.d);
    s.leaf_idx = idx;
    return true;
  }
  return false;
}

// trans(R) * v and R * v for row-major R
template <class R>
__device__ __forceinline__ void matTvec(const R *M, const R *v, R *o) {
  o[0] = M[0] * v[0] + M[3] * v[1] + M[6] * v[2];
  o[1] = M[1] * v[0] + M[4] * v[1] + M[7] * v[2];
  o[2] = M[2] * v[0] + M[5] * v[1] + M[8] * v[2];
}
template <class R>
__device__ __forceinline__ void matvec(const R *M, const R *v, R *o) {
  o[0] = M[0] * v[0] + M[1] * v[1] + M[2] * v[2];
  o[1] = M[3] * v[0] + M[4] * v[1] + M[5] * v[2];
  o[2] = M[6] * v[0] + M[7] * v[1] + M[8] * v[2];
}

// Plane: local frame, t = -o_z / d_z, interior / edge / corner branches (blazert/primitives/plane.h:180-270).
// Returns the branch (0 = miss, 1 interior, 2..5 edges, 6..9 corners) for the given [tnear, tfar].
template <class Rec>
__device__ __forceinline__ int plane_branch(const Rec &P, const RayT<typename Rec::real> &r,
                                            typename Rec::real tnear, typename Rec::real tfar,
                                            typename Rec::real *org, typename Rec::real *dir,
                                            typename Rec::real &t1, bool check_t) {
  using R = typename Rec::real;
  const R oc[3] = {r.o[0] - P.c[0], r.o[1] - P.c[1], r.o[2] - P.c[2]};
  matTvec(P.R, oc, org);
  matTvec(P.R, r.d, dir);
  t1 = -org[2] / dir[2];
  const R X = org[0] + t1 * dir[0];
  const R Y = org[1] + t1 * dir[1];
  const R x_min = -P.dx / 2, x_max = P.dx / 2, y_min = -P.dy / 2, y_max = P.dy / 2;
  const bool tok = !check_t || ((t1 > tnear) && (t1 < tfar));
  if (!tok) return 0;
  if ((X > x_min) && (X < x_max) && (Y > y_min) && (Y < y_max)) return 1;
  if ((X == x_min) && (X < x_max) && (Y > y_min) && (Y < y_max)) return 2;
  if ((X > x_min) && (X == x_max) && (Y > y_min) && (Y < y_max)) return 3;
  if ((X > x_min) && (X < x_max) && (Y == y_min) && (Y < y_max)) return 4;
  if ((X > x_min) && (X < x_max) && (Y > y_min) && (Y == y_max)) return 5;
  if ((X == x_min) && (X < x_max) && (Y == y_min) && (Y < y_max)) return 6;
  if ((X == x_min) && (X < x_max) && (Y > y_min) && (Y == y_max)) return 7;
  if ((X > x_min) && (X == x_max) && (Y == y_min) && (Y < y_max)) return 8;
  if ((X > x_min) && (X == x_max) && (Y > y_min) && (Y == y_max)) return 9;
  return 0;
}

template <class Rec>
__device__ __forceinline__ bool isect_pla(const Rec &P, const RayT<typename Rec::real> &r,
                                          HitT<typename Rec::real> &s, uint32_t idx) {
  using R = typename Rec::real;
  R org[3], dir[3], t1;
  const int br = plane_branch(P, r, r.tmin, s.h, org, dir, t1, true);
  if (!br) return false;
  s.h = norm_scaled(t1, dir);
  s.leaf_idx = idx;
  return true;
}

// Plane normal of the accepted branch (before the final normalize of post_traversal).
template <class Rec>
__device__ void plane_normal(const Rec &P, const RayT<typename Rec::real> &r, typename Rec::real *nrm) {
  using R = typename Rec::real;
  R org[3], dir[3], t1;
  const int br = plane_branch(P, r, R(0), R(0), org, dir, t1, false);
  const R sgn = org[2] / fabs(org[2]);
  if (br == 1) {
    const R ez[3] = {R(0), R(0), R(1)};
    R rz[3];
    matvec(P.R, ez, rz);
    nrm[0] = sgn * rz[0];
    nrm[1] = sgn * rz[1];
    nrm[2] = sgn * rz[2];
    return;
  }
  const R lx[10] = {0, 0, -1, 1, 0, 0, -1, -1, 1, 1};
  const R ly[10] = {0, 0, 0, 0, -1, 1, -1, 1, -1, 1};
  const R l[3] = {lx[br], ly[br], sgn};
  matvec(P.R, l, nrm);
}

// Cylinder (blazert/primitives/cylinder.h:181-495). No hit-distance checks: the last accepted cylinder wins.
// Returns true on a hit with the parametric t and the (pre-normalisation) normal.
template <class R>
struct CylOut {
  R t;
  R n[3];
};

template <class R>
__device__ __forceinline__ void cyl_ng(const R *M, const R *nn, R *out) {
  R rn[3];
  matvec(M, nn, rn);
  const R len = dsqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
  const R is = R(1) / len;
  out[0] = rn[0] * is;
  out[1] = rn[1] * is;
  out[2] = rn[2] * is;
}

template <class Rec>
__device__ bool cyl_eval(const Rec &Cy, const RayT<typename Rec::real> &r, typename Rec::real *dir,
                         CylOut<typename Rec::real> &out, bool want_normal) {
  using R = typename Rec::real;
  const R oc[3] = {r.o[0] - Cy.c[0], r.o[1] - Cy.c[1], r.o[2] - Cy.c[2]};
  R org[3];
  matTvec(Cy.R, oc, org);
  matTvec(Cy.R, r.d, dir);
  const R x0 = org[0], y0 = org[1], z0 = org[2];
  const R j = dir[0], k = dir[1], l = dir[2];
  const R a = Cy.a, b = Cy.b, h = Cy.h;
  const R zt = h / R(2), zb = -h / R(2);

  // shell quadratic shared by every region
  auto shell = [&](bool ordered, bool &hit) {
    hit = false;
    const R A = a * a * k * k + b * b * j * j;
    const R B = a * a * k * y0 + b * b * j * x0;
    const R C = a * a * k * k + b * b * j * j - j * j * y0 * y0 + 2 * j * k * x0 * y0 - k * k * x0 * x0;
    if (C < 0) return true;  // reference returns false immediately
    // R(-1) / A is -(R(1) / A) exactly (round to nearest is symmetric under negation): one division for both roots
    const R inv_a = R(1) / A;
    const R s0 = inv_a * (-B + a * b * dsqrt(C));
    const R s1 = -inv_a * (B + a * b * dsqrt(C));
    const R i0z = org[2] + dir[2] * s0;
    const R i1z = org[2] + dir[2] * s1;
    if ((s1 > 0) && (!ordered || s1 < s0) && (i1z <= zt) && (i1z >= zb)) {
      out.t = s1;
      if (want_normal) {
        const R nn[3] = {2 * (org[0] + dir[0] * s1) / (a * a), 2 * (org[1] + dir[1] * s1) / (b * b), 0};
        cyl_ng(Cy.R, nn, out.n);
      }
      hit = true;
      return true;
    }
    if ((s0 > 0) && (!ordered || s0 < s1) && (i0z <= zt) && (i0z >= zb)) {
      out.t = s0;
      if (want_normal) {
        const R nn[3] = {2 * (org[0] + dir[0] * s0) / (a * a), 2 * (org[1] + dir[1] * s0) / (b * b), 0};
        cyl_ng(Cy.R, nn, out.n);
      }
      hit = true;
      return true;
    }
    return false;  // fall through
  };
  auto cap = [&](R zc, R sgn) {
    out.t = (zc - z0) / l;
    if (want_normal) {
      const R nz[3] = {R(0), R(0), sgn};
      cyl_ng(Cy.R, nz, out.n);
    }
  };

  if (z0 > zt || z0 < zb) {  // areas 1 and 2
    const bool top = z0 > zt;
    if (l == 0) return false;
    const R t0 = top ? (zt - z0) / l : (zb - z0) / l;
    if (t0 < 0) return false;
    const R ix = org[0] + t0 * dir[0], iy = org[1] + t0 * dir[1];
    if (b * b * ix * ix + a * a * iy * iy <= a * a * b * b) {
      cap(top ? zt : zb, top ? R(1) : R(-1));
      return true;
    }
    bool hit;
    if (shell(true, hit)) return hit;
  } else if ((z0 > zb) && (z0 < zt) && (x0 * x0 * b * b + y0 * y0 * a * a > a * a * b * b)) {  // area 3
    bool hit;
    if (shell(true, hit)) return hit;
  }
  if ((z0 >= zb) && (z0 <= zt) && (x0 * x0 * b * b + y0 * y0 * a * a <= a * a * b * b)) {  // area 4
    if (l == 0) {
      if ((z0 == zb) || (z0 == zt)) return false;
      bool hit;
      if (shell(false, hit)) return hit;
    } else if ((j == R(0)) && (k == R(0))) {
      if (b * b * x0 * x0 + a * a * y0 * y0 == a * a * b * b) return false;
      if (l < 0) {
        cap(zb, R(-1));
        return true;
      }
      if (l > 0) {
        cap(zt, R(1));
        return true;
      }
    } else {
      const R A = a * a * k * k + b * b * j * j;
      const R B = a * a * k * y0 + b * b * j * x0;
      const R C = a * a * k * k + b * b * j * j - j * j * y0 * y0 + 2 * j * k * x0 * y0 - k * k * x0 * x0;
      if (C < 0) return false;
      const R inv_a = R(1) / A;
      const R s0 = inv_a * (-B + a * b * dsqrt(C));
      const R s1 = -inv_a * (B + a * b * dsqrt(C));
      const R i0z = org[2] + dir[2] * s0;
      const R i1z = org[2] + dir[2] * s1;
      if ((s1 > 0) && (i1z <= zt) && (i1z >= zb)) {
        out.t = s1;
        if (want_normal) {
          const R nn[3] = {2 * (org[0] + dir[0] * s1) / (a * a), 2 * (org[1] + dir[1] * s1) / (b * b), 0};
          cyl_ng(Cy.R, nn, out.n);
        }
        return true;
      }
      if ((s0 > 0) && (i0z <= zt) && (i0z >= zb)) {
        out.t = s0;
        if (want_normal) {  // reference stores the un-rotated normal here (cylinder.h:462-463)
          out.n[0] = 2 * (org[0] + dir[0] * s0) / (a * a);
          out.n[1] = 2 * (org[1] + dir[1] * s0) / (b * b);
          out.n[2] = 0;
        }
        return true;
      }
      if (l < 0) {
        cap(zb, R(-1));
        return true;
      }
      if (l > 0) {
        cap(zt, R(1));
        return true;
      }
    }
  }
  return false;
}

template <class Rec>
__device__ __forceinline__ bool isect_cyl(const Rec &Cy, const RayT<typename Rec::real> &r,
                                          HitT<typename Rec::real> &s, uint32_t idx) {
  using R = typename Rec::real;
  R dir[3];
  CylOut<R> o;
  if (!cyl_eval(Cy, r, dir, o, false)) return false;
  s.h = norm_scaled(o.t, dir);
  s.leaf_idx = idx;
  return true;
}

template <class Rec>
__device__ __forceinline__ bool isect(const Rec &rec, const RayT<typename Rec::real> &r, HitT<typename Rec::real> &s,
                                      uint32_t idx) {
  if constexpr (Rec::kind == TRIANGLES) return isect_tri(rec, r, s, idx);
  else if constexpr (Rec::kind == SPHERES) return isect_sph(rec, r, s, idx);
  else if constexpr (Rec::kind == PLANES) return isect_pla(rec, r, s, idx);
  else return isect_cyl(rec, r, s, idx);
}

template <class R>
__device__ __forceinline__ void normalize3(R *v) {
  const R len = dsqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  const R il = (len != R(0)) ? R(1) / len : R(0);
  v[0] *= il;
  v[1] *= il;
  v[2] *= il;
}

// post_traversal normals (trimesh.h:133-143, sphere.h:336-343, plane.h:153-159, cylinder.h:154-160)
template <class Rec>
__device__ void post_normal(const BvhView &bvh, const RayT<typename Rec::real> &r, const HitT<typename Rec::real> &s,
                            uint32_t pid, typename Rec::real *n) {
  using R = typename Rec::real;
  const Rec *recs = reinterpret_cast<const Rec *>(bvh.prims);
  if constexpr (Rec::kind == TRIANGLES) {
    const uint32_t *f = bvh.faces + 3ull * pid;
    const R *vn;
    if constexpr (sizeof(R) == 8) vn = bvh.vnormals;
    else vn = bvh.vnormals32;
    const R *n0 = vn + 3ull * f[0];
    const R *n1 = vn + 3ull * f[1];
    const R *n2 = vn + 3ull * f[2];
    const R w = (R(1) - s.u) - s.v;
#pragma unroll
    for (int k = 0; k < 3; k++) n[k] = (w * n0[k] + s.u * n1[k]) + s.v * n2[k];
  } else if constexpr (Rec::kind == SPHERES) {
    const Rec S = recs[s.leaf_idx];
#pragma unroll
    for (int k = 0; k < 3; k++) n[k] = (r.o[k] + s.h * r.d[k]) - S.c[k];
  } else if constexpr (Rec::kind == PLANES) {
    plane_normal(recs[s.leaf_idx], r, n);
  } else {
    R dir[3];
    CylOut<R> o;
    cyl_eval(recs[s.leaf_idx], r, dir, o, true);
    n[0] = o.n[0];
    n[1] = o.n[1];
    n[2] = o.n[2];
  }
  normalize3(n);
}

// ------------------------------------------------------------------------------------------------ traversal
// Per-lane traversal state. The DFS of the reference is advanced one unit at a time (one internal node, or one
// whole leaf), so a persistent wave can retire finished rays and pull new ones between steps.
struct Trav {
  uint32_t cur, cnt;  // current node reference and leaf count
  uint32_t pos;       // next primitive of the current leaf (with the triangle pre-test: first of the current group)
  uint32_t cand;      // split-precision triangles: group members that passed the FP32 pre-test, still to test
  bool active;        // traversal still running
  float h32;          // split precision: hit distance rounded up to FP32
};

// Traversal stack: the top `ring` entries of each lane live in LDS (slot-major, lane-minor, so a wave's accesses
// spread over all banks); older entries spill to private memory only when a ray goes deeper than the ring, and come
// back when the ring drains. Invariant: entries [lo, sp) are in LDS, [0, lo) in the private spill area.
// The ring depth is a launch parameter (a power of two, 4..16): deeper rings spill less but take more LDS per block.
// Defaults: 8 for FP64 keys; 16 for the FP32 path over triangles, whose 4-wide steps push up to three entries at a
// time (1.31M-triangle incoherent set); 8 for the FP32 path over the other types, where the fourth wave per SIMD
// that a shallower ring leaves room for pays more than the spills it causes (mixed scene, 8M rays: spheres 3.87 ->
// 3.35 ms, cylinders 4.97 -> 4.32, planes 1.66 -> 1.47 with 8 instead of 16).
template <class Rec, bool SPLIT>
constexpr uint32_t ring_default() { return (SPLIT && Rec::kind == TRIANGLES) ? 16u : 8u; }
// Default refill threshold (idle lanes of a wave before it takes new rays). Exact path: 32 for triangles (1.31M-
// triangle incoherent set: 16 is 3% slower, 40 5% slower), 16 for the other types, whose longer primitive tests
// favour earlier refills (mixed scene: spheres 3% and cylinders 5% faster than at 32). 4-wide split path: 16 for
// every type (icosphere: 32 is 7% slower).
template <class Rec, bool SPLIT>
constexpr uint32_t refill_default() { return (SPLIT || Rec::kind != TRIANGLES) ? 16u : 32u; }
// Default block size of a single-scene launch: 256, except 128 for FP64 spheres on the exact path (mixed scene, 8M
// rays: 4.30-4.33 ms against 4.44-4.51 with 256; the other types and the split path do not change between 64 and
// 256).
template <class Rec, bool SPLIT>
constexpr uint32_t block_default() { return (!SPLIT && std::is_same<Rec, SphRec>::value) ? 128u : 256u; }

// Stack keys: FP32 entry distances on the split path, otherwise the scene type's.
template <bool SPLIT, class R>
using StackKey = typename std::conditional<SPLIT, float, R>::type;

template <bool SPLIT, class R = double>
struct SpillArea {  // private (scratch) memory for entries pushed deeper than the ring
  using Key = StackKey<SPLIT, R>;
  Key key[stack_cap<SPLIT>()];
  uint32_t ref[stack_cap<SPLIT>()], cnt[stack_cap<SPLIT>()];
};

// The counters and pointers are kept apart from the spill arrays so that they stay in registers.
template <bool SPLIT, class R = double>
struct RingStack {
  using Key = StackKey<SPLIT, R>;
  BRT_LDS Key *lkey;  // this lane's slot 0 in LDS; slot j is at [64 * j]
  BRT_LDS uint32_t *lref, *lcnt;
  SpillArea<SPLIT, R> *spill;
  int sp, lo;
  int ring;  // LDS slots per lane (power of two)

  __device__ __forceinline__ void reset() {
    sp = 0;
    lo = 0;
  }
  __device__ __forceinline__ void push(uint32_t r, uint32_t c, Key k) {
    if (sp - lo == ring) {
      const int j = (lo & (ring - 1)) * 64;
      spill->key[lo] = lkey[j];
      spill->ref[lo] = lref[j];
      spill->cnt[lo] = lcnt[j];
      lo++;
    }
    const int j = (sp & (ring - 1)) * 64;
    lkey[j] = k;
    lref[j] = r;
    lcnt[j] = c;
    sp++;
  }
  // requires sp > 0
  __device__ __forceinline__ void pop(uint32_t &r, uint32_t &c, Key &k) {
    sp--;
    if (sp < lo) {
      lo = sp;
      r = spill->ref[sp];
      c = spill->cnt[sp];
      k = spill->key[sp];
    } else {
      const int j = (sp & (ring - 1)) * 64;
      r = lref[j];
      c = lcnt[j];
      k = lkey[j];
    }
  }
};

// LDS bytes of the ring stacks of one block
template <bool SPLIT, class R = double>
constexpr size_t ring_lds_bytes(uint32_t block, uint32_t ring) {
  return (size_t)(block / 64) * ring * 64 * (sizeof(StackKey<SPLIT, R>) + 8);
}

template <bool SPLIT, class R>
__device__ __forceinline__ void ring_bind(RingStack<SPLIT, R> &st, unsigned char *smem, SpillArea<SPLIT, R> *spill,
                                          uint32_t ring) {
  using Key = StackKey<SPLIT, R>;
  const uint32_t waves = blockDim.x / 64, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  BRT_LDS unsigned char *lds = (BRT_LDS unsigned char *)smem;
  const size_t slots = (size_t)waves * ring * 64;
  BRT_LDS Key *keys = (BRT_LDS Key *)lds;
  BRT_LDS uint32_t *refs = (BRT_LDS uint32_t *)(lds + slots * sizeof(Key));
  BRT_LDS uint32_t *cnts = (BRT_LDS uint32_t *)(lds + slots * (sizeof(Key) + 4));
  st.lkey = keys + (size_t)wave * ring * 64 + lane;
  st.lref = refs + (size_t)wave * ring * 64 + lane;
  st.lcnt = cnts + (size_t)wave * ring * 64 + lane;
  st.ring = (int)ring;
  st.spill = spill;
  st.reset();
}

// Ascending sort of four (key, ref, cnt) triples: compare-exchange network (0,1)(2,3)(0,2)(1,3)(1,2), every index
// a compile-time constant so the arrays stay in registers.
template <int I, int J>
__device__ __forceinline__ void cmpx(float (&k)[4], uint32_t (&r)[4], uint32_t (&c)[4]) {
  const bool sw = k[J] < k[I];
  const float ki = k[I], kj = k[J];
  const uint32_t ri = r[I], rj = r[J], ci = c[I], cj = c[J];
  k[I] = sw ? kj : ki;
  k[J] = sw ? ki : kj;
  r[I] = sw ? rj : ri;
  r[J] = sw ? ri : rj;
  c[I] = sw ? cj : ci;
  c[J] = sw ? ci : cj;
}
__device__ __forceinline__ void sort4(float (&k)[4], uint32_t (&r)[4], uint32_t (&c)[4]) {
  cmpx<0, 1>(k, r, c);
  cmpx<2, 3>(k, r, c);
  cmpx<0, 2>(k, r, c);
  cmpx<1, 3>(k, r, c);
  cmpx<1, 2>(k, r, c);
}

// Root test (the reference pushes node 0 and slab-tests it on the first pop with the ray's tmax).
template <bool SPLIT, class R>
__device__ __forceinline__ void trav_begin(const BvhView &bvh, const RayT<R> &r, const Ray32 &q, const HitT<R> &s,
                                           Trav &t) {
  t.cur = SPLIT ? bvh.root_ref4 : bvh.root_ref;
  t.cnt = bvh.root_cnt;
  t.pos = 0;
  t.cand = 0;
  if constexpr (SPLIT) {
    float k32;
    const float rb[6] = {bvh.root_min32[0], bvh.root_min32[1], bvh.root_min32[2],
                         bvh.root_max32[0], bvh.root_max32[1], bvh.root_max32[2]};
    t.h32 = f32_up(s.h);
    t.active = slab32(rb, q, k32) && !(t.h32 < k32);
  } else {
    // the descriptor holds the root box in FP64; a Scene<float> box converts back exactly
    R key;
    const R rb[6] = {R(bvh.root_min[0]), R(bvh.root_min[1]), R(bvh.root_min[2]),
                     R(bvh.root_max[0]), R(bvh.root_max[1]), R(bvh.root_max[2])};
    t.h32 = 0.0f;
    t.active = slab_exact(rb, r, key) && !(s.h < key);
  }
}

// One unit of the DFS: an internal node (test both children, push far, descend near) or a leaf's next primitives
// (exact_group per type, in order, blazert/bvh/intersect.h:66-78), followed by pops until a node passes or the stack
// is empty. On the split path with triangle or sphere pre-test records, a leaf step is either a pre-test of the
// next FILTER_GROUP triangles or SPH_FILTER_GROUP spheres in FP32 (tri_filter, sph_filter) or the FP64 test of the
// next one that passed it, in leaf order.
template <class Rec, bool SPLIT>
__device__ __forceinline__ void trav_step(const BvhView &bvh, const RayT<typename Rec::real> &r, const Ray32 &q,
                                          bool any_hit, HitT<typename Rec::real> &s, Trav &t,
                                          RingStack<SPLIT, typename Rec::real> &st) {
  using R = typename Rec::real;
  using Node = typename std::conditional<SPLIT, Node4,
                                         typename std::conditional<sizeof(R) == 8, Node64, Node32>::type>::type;
  // One fetch per lane, issued together: the internal record for lanes at an inner node, the primitive record (or
  // the group of pre-test records) for lanes at a leaf. Written as separate branches, each would wait for its own
  // loads, and a wave holding several kinds of lanes would pay several memory round trips per step. The chunks the
  // records have in common are loaded from a per-lane address in one set of instructions; the rest of the longer
  // ones follow in short branches (from the same lines, already on their way), and the compute branches below run
  // without waiting in between.
  // split precision, triangles, spheres and cylinders: FP32 pre-test records, FG of them per step
  constexpr bool FILTER = SPLIT && (Rec::kind == TRIANGLES || Rec::kind == SPHERES || Rec::kind == CYLINDERS);
  using Filt = typename std::conditional<Rec::kind == TRIANGLES, TriFilt,
                                         typename std::conditional<Rec::kind == CYLINDERS, CylFilt, SphFilt>::type>::type;
  constexpr uint32_t FG = Rec::kind == TRIANGLES ? FILTER_GROUP : SPH_FILTER_GROUP;
  constexpr int NODE_Q = SPLIT ? 8 : (sizeof(R) == 8 ? 7 : 4);  // 16-byte chunks of the record used (Node64: 112 B)
  constexpr int REC_Q = (int)(sizeof(Rec) / 16);
  constexpr int FILT_Q = FILTER ? (int)(FG * sizeof(Filt) / 16) : 0;
  // exact paths: primitives tested per leaf step
  constexpr int PG = SPLIT ? 1 : exact_group<Rec::kind>();
  constexpr int QMAX0 = NODE_Q < PG * REC_Q ? PG * REC_Q : NODE_Q;
  constexpr int QMAX = QMAX0 < FILT_Q ? FILT_Q : QMAX0;
  static_assert(sizeof(Rec) % 16 == 0 && sizeof(Node) >= 16 * NODE_Q, "record chunking");
  const bool at_leaf = (t.cur & LEAF_BIT) != 0;
  const Filt *frecs = nullptr;
  if constexpr (FILTER) {
    if constexpr (Rec::kind == TRIANGLES) frecs = bvh.tri_filter;
    else if constexpr (Rec::kind == CYLINDERS) frecs = bvh.cyl_filter;
    else frecs = bvh.sph_filter;
  }
  const bool filt = FILTER && frecs != nullptr;  // the same for every lane of a launch
  const bool filter_step = filt && at_leaf && t.cand == 0u && t.pos < t.cnt;
  const bool fetch_rec = at_leaf && t.pos < t.cnt && !filter_step;
  const uint32_t p = (t.cur & ~LEAF_BIT) + t.pos + (filt ? (uint32_t)__builtin_ctz(t.cand | 0x80000000u) : 0u);
  const Node *nodes;
  if constexpr (SPLIT) nodes = reinterpret_cast<const Node *>(bvh.nodes4);
  else if constexpr (sizeof(R) == 8) nodes = reinterpret_cast<const Node *>(bvh.nodes64);
  else nodes = reinterpret_cast<const Node *>(bvh.nodes32);
  // The loads go through a pointer in the global address space: the batch kernel's tree pointers come from its job
  // table in memory, and as generic pointers every access through them would be a flat access.
  using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
  using GlobalChunk = const __attribute__((address_space(1))) u32x4;
  GlobalChunk *src = !at_leaf ? (GlobalChunk *)(nodes + t.cur)
                     : filter_step ? (GlobalChunk *)(frecs + ((t.cur & ~LEAF_BIT) + t.pos))
                                   : (GlobalChunk *)(reinterpret_cast<const Rec *>(bvh.prims) + p);
  u32x4 chunk[QMAX];
  if constexpr (FILTER) {
    // three record kinds: each chunk is loaded by the lanes whose record has it
    const int nq = !at_leaf ? NODE_Q : (filter_step ? FILT_Q : (fetch_rec ? REC_Q : 0));
#pragma unroll
    for (int k = 0; k < QMAX; k++)
      if (k < nq) chunk[k] = src[k];
  } else {
    constexpr int COMMON = NODE_Q < REC_Q ? NODE_Q : REC_Q;
    if (!at_leaf || fetch_rec) {
#pragma unroll
      for (int k = 0; k < COMMON; k++) chunk[k] = src[k];
    }
    if (!at_leaf) {
#pragma unroll
      for (int k = COMMON; k < NODE_Q; k++) chunk[k] = src[k];
    } else if (fetch_rec) {
#pragma unroll
      for (int k = COMMON; k < REC_Q; k++) chunk[k] = src[k];
#pragma unroll
      for (int g = 1; g < PG; g++)
        if (t.pos + g < t.cnt) {
#pragma unroll
          for (int k = g * REC_Q; k < (g + 1) * REC_Q; k++) chunk[k] = src[k];
        }
    }
  }
  // an empty asm taking every chunk as an operand: the loads cannot be sunk into the compute branches below, so all
  // of them are issued first and waited for once
#pragma unroll
  for (int k = 0; k < QMAX; k++) asm volatile("" : "+v"(chunk[k]));
  if (!at_leaf) {
    bool near_ok, far_ok;
    uint32_t nref, ncnt, fref, fcnt;
    StackKey<SPLIT, R> fkey;
    Node nd;
    __builtin_memcpy(&nd, chunk, 16 * NODE_Q);
    if constexpr (SPLIT) {
      // up to four children per record, visited nearest entry first (the FP32 path needs no particular order:
      // it only has to test every primitive the FP64 path tests)
      float k[4];
      uint32_t rf[4], cn[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        float A = q.tmin, M = t.h32;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const bool sg = (q.sign >> a) & 1u;
          const float lo = nd.lo[a][c], hi = nd.hi[a][c];
          A = fmaxf(A, __builtin_fmaf(sg ? hi : lo, q.inv[a], q.offn[a]));
          M = fminf(M, __builtin_fmaf(sg ? lo : hi, q.inv[a], q.offf[a]));
        }
        k[c] = (nd.cnt[c] != EMPTY_SLOT && A <= M) ? A : __builtin_inff();
        rf[c] = nd.ref[c];
        cn[c] = nd.cnt[c];
      }
      sort4(k, rf, cn);
      const float INF = __builtin_inff();
      if (k[3] < INF) st.push(rf[3], cn[3], k[3]);
      if (k[2] < INF) st.push(rf[2], cn[2], k[2]);
      if (k[1] < INF) st.push(rf[1], cn[1], k[1]);
      if (k[0] < INF) {
        t.cur = rf[0];
        t.cnt = cn[0];
        t.pos = 0;
        return;
      }
      near_ok = far_ok = false;
      nref = ncnt = fref = fcnt = 0;
      fkey = 0.0f;
    } else {
      const uint32_t axis = nd.cnt[1] >> AXIS_SHIFT;
      const uint32_t nc = (r.sign >> axis) & 1u;
      R k0 = R(0), k1 = R(0);
      const bool p0 = slab_exact(nd.b, r, k0);
      const bool p1 = slab_exact(nd.b + 6, r, k1);
      near_ok = (nc ? p1 : p0) && !(s.h < (nc ? k1 : k0));
      far_ok = nc ? p0 : p1;
      fkey = nc ? k0 : k1;
      const uint32_t r0 = nd.ref[0], r1 = nd.ref[1], c0 = nd.cnt[0] & CNT_MASK, c1 = nd.cnt[1] & CNT_MASK;
      nref = nc ? r1 : r0;
      ncnt = nc ? c1 : c0;
      fref = nc ? r0 : r1;
      fcnt = nc ? c0 : c1;
    }
    if (far_ok) st.push(fref, fcnt, fkey);
    if (near_ok) {
      t.cur = nref;
      t.cnt = ncnt;
      t.pos = 0;
      return;
    }
  } else if (filter_step) {
    if constexpr (FILTER) {
      // pre-test the group; members past the leaf's end are padding or the next leaf's primitives
      Filt g[FG];
      __builtin_memcpy(g, chunk, sizeof g);
      const float D[3] = {(float)r.d[0], (float)r.d[1], (float)r.d[2]};
      const float O[3] = {(float)r.o[0], (float)r.o[1], (float)r.o[2]};
      const uint32_t left = t.cnt - t.pos;
      uint32_t mask = 0;
#pragma unroll
      for (uint32_t j = 0; j < FG; j++) {
        bool pass;
        if constexpr (Rec::kind == TRIANGLES) pass = tri_filter(g[j], D, O, q.om, q.tmin, t.h32);
        else if constexpr (Rec::kind == SPHERES) pass = sph_filter(g[j], D, O, q.om, q.tmin, t.h32);
        else pass = cyl_filter(g[j], D, O, q.om);
        if (j < left && pass) mask |= 1u << j;
      }
      t.cand = mask;
      if (mask) return;
      t.pos += FG;
      if (t.pos < t.cnt) return;
    }
  } else {
    // a few primitives per step: a leaf's tests (blazert/bvh/intersect.h:66-78, in order, each against the hit
    // distance the previous one left) are spread over consecutive steps, so lanes at leaves and lanes at inner
    // nodes run branches of similar length instead of inner-node lanes idling through a whole leaf
    if (fetch_rec) {
      Rec rec;
      __builtin_memcpy(&rec, chunk, sizeof(Rec));
      if (isect(rec, r, s, p)) {
        if (SPLIT) t.h32 = f32_up(s.h);
        if (any_hit) {
          t.active = false;
          return;
        }
      }
#pragma unroll
      for (int g = 1; g < PG; g++) {  // the leaf's next primitives, each against the hit distance just left
        if (t.pos + 1 >= t.cnt) break;
        __builtin_memcpy(&rec, chunk + g * REC_Q, sizeof(Rec));
        t.pos++;
        if (isect(rec, r, s, p + g) && any_hit) {
          t.active = false;
          return;
        }
      }
      if (filt) {
        t.cand &= t.cand - 1u;
        if (t.cand) return;
        t.pos += FG;
        if (t.pos < t.cnt) return;
      } else if (++t.pos < t.cnt) {
        return;
      }
    }
  }
  // pop the next far child whose entry distance does not exceed the current hit distance
  while (st.sp > 0) {
    uint32_t ref, cnt;
    StackKey<SPLIT, R> key;
    st.pop(ref, cnt, key);
    bool ok;
    if constexpr (SPLIT) ok = !(t.h32 < key);
    else ok = !(s.h < key);
    if (ok) {
      t.cur = ref;
      t.cnt = cnt;
      t.pos = 0;
      return;
    }
  }
  t.active = false;
}

// Merge into the hit record (blazert/scene.h:169-209): triangles replace unconditionally, later types only if
// strictly closer; the first type of the scene also writes the default RayHit for misses.
template <class Rec>
__device__ __forceinline__ void finish_ray(const BvhView &bvh, const HitsViewT<typename Rec::real> &hits, uint64_t i,
                                           const RayT<typename Rec::real> &r, const HitT<typename Rec::real> &s,
                                           uint32_t flags, uint32_t first, uint32_t is_tri) {
  using R = typename Rec::real;
  const bool hit = s.h < r.tmax;
  bool write = false;
  if (hit) {
    if (is_tri) write = true;
    else write = s.h < ((first && !(flags & FLAG_INOUT)) ? Real<R>::max : gmem(hits.t)[i]);
  }
  if (write) {
    const uint32_t pid = id_in_record<Rec>() ? s.leaf_idx : gmem(bvh.prim_ids)[s.leaf_idx];
    if (hits.merged) st_stream(hits.merged, i, 1u);
    st_stream(hits.t, i, s.h);
    if (hits.u) st_stream(hits.u, i, s.u);
    if (hits.v) st_stream(hits.v, i, s.v);
    st_stream(hits.prim_id, i, pid);
    if (hits.geom_id) st_stream(hits.geom_id, i, bvh.geom_id);
    if (hits.nx) {
      R nrm[3];
      post_normal<Rec>(bvh, r, s, pid, nrm);
      st_stream(hits.nx, i, nrm[0]);
      st_stream(hits.ny, i, nrm[1]);
      st_stream(hits.nz, i, nrm[2]);
    }
  } else if (first && !(flags & FLAG_INOUT)) {
    st_stream(hits.t, i, Real<R>::max);
    if (hits.u) st_stream(hits.u, i, R(0));
    if (hits.v) st_stream(hits.v, i, R(0));
    st_stream(hits.prim_id, i, INVALID_ID);
    if (hits.geom_id) st_stream(hits.geom_id, i, INVALID_ID);
    if (hits.nx) {
      st_stream(hits.nx, i, R(0));
      st_stream(hits.ny, i, R(0));
      st_stream(hits.nz, i, R(0));
    }
  }
}

template <bool SPLIT, class R>
__device__ __forceinline__ void start_ray(const BvhView &bvh, const RaysViewT<R> &rays, uint64_t i, double S,
                                          RayT<R> &r, Ray32 &q, HitT<R> &s) {
  make_ray(rays, i, r);
  if (bvh.irregular_boxes) r.sign &= ~RAY_NAN_FREE;
  if constexpr (SPLIT) make_ray32(r, S, q);
  s.h = r.tmax;  // prepare_traversal
  s.u = R(0);
  s.v = R(0);
  s.leaf_idx = INVALID_ID;
}

// Rays whose reference traversal the FP32 bounds enclose: no slab term can be NaN or leave the FP32 range, tmin >= 0
// and a direction of at least unit length (its slab distances are then the hit distances, or shorter: the reference skips no
// more by them, except through tmin, see certified).
// Split precision takes shorter ones too: it need not tell the boxes that the reference reaches from those a rounding away.
constexpr double SHORT_LEN2 = 1.0 - 0x1p-20;
__device__ __forceinline__ bool fast_ray(const Ray &r, double len2, double S, bool split) {
  bool ok = (r.sign & RAY_NAN_FREE) && r.tmin >= 0.0 && (split || len2 >= SHORT_LEN2) && len2 <= 1e20;
#pragma unroll
  for (int k = 0; k < 3; k++) ok = ok && fabs(r.inv[k]) * (S + fabs(r.o[k])) <= 1e36 && fabs(r.inv[k]) <= 1e30;
  return ok && fabs(r.o[0]) <= FILTER_MAX_EXTENT && fabs(r.o[1]) <= FILTER_MAX_EXTENT &&
         fabs(r.o[2]) <= FILTER_MAX_EXTENT;
}

// Rays of k_trace_wide: the FP32 bounds enclose the reference's traversal, whatever the length of the direction, within
// limits that keep 1/d a normal FP32 number: as 0 it would make the infinite planes of a node's unused slots NaN, and the
// slots passable.
template <class R>
__device__ __forceinline__ bool wide_ray(const RayT<R> &r, double S) {
  bool ok = (r.sign & RAY_NAN_FREE) && r.tmin >= R(0);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double inv = fabs((double)r.inv[k]), o = fabs((double)r.o[k]);
    ok = ok && inv * (S + o) <= 1e36 && inv <= 1e30 && inv >= 1e-30 && o <= FILTER_MAX_EXTENT;
  }
  return ok;
}

// A ray's columns as they stand in memory.
template <class R>
struct RawRayT {
  R org[3], dir[3], tmin, tmax;
};
using RawRay = RawRayT<double>;
template <class R>
__device__ __forceinline__ RawRayT<R> load_ray(const RaysViewT<R> &V, uint64_t i) {
  return RawRayT<R>{{ld_stream(V.ox, i), ld_stream(V.oy, i), ld_stream(V.oz, i)},
                    {ld_stream(V.dx, i), ld_stream(V.dy, i), ld_stream(V.dz, i)},
                    V.tmin ? ld_stream(V.tmin, i) : V.tmin0,
                    V.tmax ? ld_stream(V.tmax, i) : V.tmax0};
}
__device__ __forceinline__ double squared_length(const RawRay &w) {
  return w.dir[0] * w.dir[0] + w.dir[1] * w.dir[1] + w.dir[2] * w.dir[2];
}

// The type's predicate from the ray's columns.
template <class Rec>
__device__ __forceinline__ bool fast_ray(const RaysViewT<typename Rec::real> &V, uint64_t i, double S, bool split) {
  using R = typename Rec::real;
  const RawRayT<R> w = load_ray(V, i);
  RayT<R> r;
  setup_ray(w.org, w.dir, w.tmin, w.tmax, r);
  if constexpr (Rec::kind == TRIANGLES && sizeof(R) == 8) return fast_ray(r, squared_length(w), S, split);
  else return wide_ray(r, S);
}

// Whether a launch has passed rays over, on any of its lines, one read by each of a wave's first lanes. Called by whole waves.
__device__ __forceinline__ bool any_passed(const unsigned long long *group) {
  const uint32_t lane = __lane_id();
  unsigned long long x = 0;
  if (lane < (uint32_t)CLAIM_COUNTERS) {
    x = __atomic_load_n(group + lane * COUNTER_STRIDE + COUNTER_DEFERRED, __ATOMIC_RELAXED);
  }
  return __ballot(x != 0ull) != 0ull;
}

// One ray per thread (grid-stride). left: only the rays whose bits a launch of `fixed` rays per wave set there.
template <class Rec, bool SPLIT>
__global__ void __launch_bounds__(256) k_trace(BvhView bvh, RaysViewT<typename Rec::real> rays,
                                               HitsViewT<typename Rec::real> hits, uint64_t n, uint32_t flags,
                                               uint32_t first, uint32_t is_tri, double S, const uint32_t *order,
                                               uint32_t ring, unsigned long long *deferred,
                                               const unsigned long long *left = nullptr, uint32_t fixed = 1) {
  using R = typename Rec::real;
  extern __shared__ unsigned char smem[];
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const bool any_hit = (flags & FLAG_ANY_HIT) != 0;
  const bool deferred_only = !SPLIT && (flags & FLAG_DEFERRED_ONLY);
  if (deferred_only && !any_passed(deferred - COUNTER_DEFERRED)) return;
  SpillArea<SPLIT, R> spill;
  RingStack<SPLIT, R> st;
  ring_bind<SPLIT, R>(st, smem, &spill, ring);
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    if (left && !((left[k / fixed] >> (k % fixed)) & 1ull)) continue;
    const uint64_t i = order ? (uint64_t)order[k] : k;
    RayT<R> r;
    Ray32 q;
    HitT<R> s;
    start_ray<SPLIT>(bvh, rays, i, S, r, q, s);
    if (SPLIT && deferred_to_exact(r)) {
      __atomic_store_n(deferred, 1ull, __ATOMIC_RELAXED);
      continue;
    }
    if (deferred_only && !deferred_to_exact(r)) continue;
    Trav t;
    trav_begin<SPLIT>(bvh, r, q, s, t);
    st.reset();
    while (t.active) trav_step<Rec, SPLIT>(bvh, r, q, any_hit, s, t, st);
    finish_ray<Rec>(bvh, hits, i, r, s, flags, first, is_tri);
  }
}

// Occupancy target of the persistent kernels (waves per SIMD the register allocation must allow).
#ifndef BRT_WAVES_PER_EU
#define BRT_WAVES_PER_EU 4
#endif

// The ray and hit column pointers (17 of them) are used only where a lane starts or finishes a ray. Held in
// scalar registers for the whole kernel they overflowed the scalar register file, and the compiler reloaded them
// from spill lanes as whole 16-register tuples at every start and finish. The persistent triangle kernels instead
// keep one copy per block in LDS and re-read it (volatile, so it is not hoisted back into registers) where it is
// used: incoherent triangle launches 1-2% and coherent ones 3-5% faster. The cylinder launch was 2% slower that way
// and the sphere and plane launches no faster, so they keep the kernel arguments.
template <class T>
__device__ __forceinline__ void lds_store(uint64_t *dst, const T &x) {
  static_assert(sizeof(T) % 8 == 0, "8-byte words");
  __builtin_memcpy(dst, &x, sizeof(T));
}
template <class T>
__device__ __forceinline__ T lds_fresh(const uint64_t *src) {
  using lds_u64 = const volatile __attribute__((address_space(3))) uint64_t;
  lds_u64 *v = (lds_u64 *)src;
  uint64_t w[sizeof(T) / 8];
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 8); k++) {
    const uint64_t x = v[k];  // the same in every lane: moved to scalar registers for the address arithmetic
    w[k] = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  }
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// Sets the launch's flag of rays passed over, when a wave that has passed some ends, and on the block's own line: stores to one
// line are served one after the other. 2,073,600 rays of an axis-parallel camera, all passed over, take k_trace_tri 0.14 ms
// (0.27 with one line, 1.5 with a store per ray).
__device__ __forceinline__ void note_passed(bool noted, unsigned long long *group, uint32_t lane) {
  if (noted && lane == 0) {
    __atomic_store_n(group + (blockIdx.x % CLAIM_COUNTERS) * COUNTER_STRIDE + COUNTER_DEFERRED, 1ull, __ATOMIC_RELAXED);
  }
}

// Lists a ray in the block's part.
__device__ __forceinline__ void list_ray(uint64_t ray, unsigned long long *group) {
  const uint32_t part = blockIdx.x % CLAIM_COUNTERS;
  const unsigned long long k = atomicAdd(group + part * COUNTER_STRIDE + COUNTER_LISTED, 1ull);
  if (k < (unsigned long long)LIST_PART) group[COUNTER_CLEARED + part * LIST_PART + k] = ray;
}

// What the exact launch behind k_trace_tri or k_trace_wide has to trace: positions [0, scan) (of the rays passed over, or
// of all rays when more were listed than a part of the list holds) and then `listed` entries of the list. ends: a block's place
// for the parts' running ends, valid behind the block's next barrier.
struct Leftover {
  uint64_t scan, listed;
  bool all;
};
__device__ __forceinline__ Leftover leftover(const unsigned long long *group, uint64_t n, uint32_t *ends) {
  const uint32_t lane = __lane_id();
  unsigned long long x = 0;
  if (lane < (uint32_t)CLAIM_COUNTERS) {
    x = __atomic_load_n(group + lane * COUNTER_STRIDE + COUNTER_LISTED, __ATOMIC_RELAXED);
  }
  const bool all = __ballot(x > (unsigned long long)LIST_PART) != 0ull;
  uint32_t listed = 0;
#pragma unroll
  for (int k = 0; k < CLAIM_COUNTERS; k++) {
    listed += (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, k);
    if (threadIdx.x == 0) ends[k] = listed;
  }
  const bool passed = any_passed(group);
  return Leftover{all || passed ? n : 0ull, all ? 0ull : listed, all};
}
__device__ __forceinline__ uint64_t list_entry(const unsigned long long *group, const uint32_t *ends, uint32_t i) {
  uint32_t k = 0, begin = 0;
  while (i >= ends[k]) begin = ends[k++];
  return group[COUNTER_CLEARED + k * LIST_PART + (i - begin)];
}

// AFTER_FAST: the launch behind k_trace_tri or k_trace_wide (see leftover).
template <class Rec, bool SPLIT, bool AFTER_FAST = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BRT_WAVES_PER_EU)))
k_trace_persistent(BvhView bvh, RaysViewT<typename Rec::real> rays, HitsViewT<typename Rec::real> hits, uint64_t n,
                   uint32_t flags, uint32_t first, uint32_t is_tri, double S, unsigned long long *counter,
                   uint32_t refill, const uint32_t *order, uint32_t ring, unsigned long long *deferred,
                   uint32_t chunk) {
  using R = typename Rec::real;
  extern __shared__ unsigned char smem[];
  const bool any_hit = (flags & FLAG_ANY_HIT) != 0;
  const bool deferred_only = !SPLIT && !AFTER_FAST && (flags & FLAG_DEFERRED_ONLY);
  if (deferred_only && !any_passed(deferred - COUNTER_DEFERRED)) return;
  Leftover left{};
  __shared__ uint32_t list_ends[AFTER_FAST ? CLAIM_COUNTERS : 1];
  if constexpr (AFTER_FAST) {
    left = leftover(deferred - COUNTER_DEFERRED, n, list_ends);
    n = left.scan + left.listed;
    if (n == 0) return;
    __syncthreads();
  }
  constexpr bool LDS_VIEWS = Rec::kind == TRIANGLES;
  constexpr int RW = (int)(sizeof(RaysViewT<R>) / 8), HW = (int)(sizeof(HitsViewT<R>) / 8);
  __shared__ uint64_t views[RW + HW];
  if constexpr (LDS_VIEWS) {
    if (threadIdx.x == 0) {
      lds_store(views, rays);
      lds_store(views + RW, hits);
    }
    __syncthreads();
  }
  auto rays_view = [&]() -> RaysViewT<R> {
    if constexpr (LDS_VIEWS) return lds_fresh<RaysViewT<R>>(views);
    else return rays;
  };
  auto hits_view = [&]() -> HitsViewT<R> {
    if constexpr (LDS_VIEWS) return lds_fresh<HitsViewT<R>>(views + RW);
    else return hits;
  };
  const uint32_t lane = __lane_id();
  SpillArea<SPLIT, R> spill;
  RingStack<SPLIT, R> st;
  ring_bind<SPLIT, R>(st, smem, &spill, ring);
  RayT<R> r;
  Ray32 q;
  HitT<R> s;
  Trav t;
  t.active = false;
  bool has_ray = false;
  bool exhausted = false;  // wave-uniform
  uint64_t idx = 0;
  WavePool pool;
  for (;;) {
    if (!exhausted) {
      const unsigned long long idle = __ballot(!has_ray);
      const uint32_t nidle = (uint32_t)__popcll(idle);
      if (nidle >= refill || nidle == 64u) {
        bool got;
        uint64_t cand = 0;
        pool_refill(pool, counter, n, chunk, idle, nidle, lane, got, cand, exhausted);
        if (got) {
          bool trace = true;
          if (AFTER_FAST && cand >= left.scan) {
            idx = list_entry(deferred - COUNTER_DEFERRED, list_ends, (uint32_t)(cand - left.scan));
            start_ray<SPLIT>(bvh, rays_view(), idx, S, r, q, s);
          } else {
            idx = order ? (uint64_t)order[cand] : cand;
            start_ray<SPLIT>(bvh, rays_view(), idx, S, r, q, s);
            if constexpr (AFTER_FAST) trace = left.all || !fast_ray<Rec>(rays_view(), idx, S, (flags & FLAG_SPLIT) != 0u);
          }
          if (SPLIT && deferred_to_exact(r)) {
            __atomic_store_n(deferred, 1ull, __ATOMIC_RELAXED);
          } else if (trace && (!deferred_only || deferred_to_exact(r))) {
            has_ray = true;
            trav_begin<SPLIT>(bvh, r, q, s, t);
            st.reset();
          }
        }
      }
    }
    // lanes may drop the rays they were handed (deferred or skipped), so an idle wave leaves only once the pool is
    // exhausted
    if (!__ballot(has_ray) && exhausted) break;
    if (has_ray) {
      if (t.active) trav_step<Rec, SPLIT>(bvh, r, q, any_hit, s, t, st);
      if (!t.active) {
        finish_ray<Rec>(bvh, hits_view(), idx, r, s, flags, first, is_tri);
        has_ray = false;
      }
    }
  }
}

// Many scenes in one launch: the claimed index runs over the concatenated rays of all jobs (one job = one scene's
// BVH of this geometry type + its own rays and hits). A lane finds its job by binary search over the prefix offsets
// and reads that job's BVH view from the table (a few cached loads per step), so waves freely mix scenes and the
// uneven batch drains with no per-scene tail.
constexpr uint32_t BATCH_LDS_JOBS = 32;

__device__ __forceinline__ uint32_t find_job(const BatchJob *jobs, uint32_t njobs, uint64_t g) {
  uint32_t lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (jobs[mid].offset <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

template <class Rec, bool SPLIT, bool AFTER_FAST = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BRT_WAVES_PER_EU)))
k_trace_batch(const BatchJob *__restrict__ jobs, uint32_t njobs, uint64_t total, uint32_t flags,
              unsigned long long *counter, uint32_t refill, uint32_t ring, unsigned long long *deferred,
              uint32_t chunk) {
  extern __shared__ unsigned char smem[];
  const bool any_hit = (flags & FLAG_ANY_HIT) != 0;
  const bool deferred_only = !SPLIT && !AFTER_FAST && (flags & FLAG_DEFERRED_ONLY);
  if (deferred_only && !any_passed(deferred - COUNTER_DEFERRED)) return;
  Leftover left{};
  __shared__ uint32_t list_ends[AFTER_FAST ? CLAIM_COUNTERS : 1];
  if constexpr (AFTER_FAST) {
    left = leftover(deferred - COUNTER_DEFERRED, total, list_ends);
    total = left.scan + left.listed;
    if (total == 0) return;
    __syncthreads();
  }
  // Finishing a ray needs its job's hit columns and flags: for batches of up to BATCH_LDS_JOBS jobs every block
  // keeps them in LDS, so that a finish does not wait on a load from the job table.
  constexpr int JW = (int)(sizeof(HitsView) / 8) + 1;  // hit column pointers, then first | is_tri << 32
  __shared__ uint64_t job_fin[BATCH_LDS_JOBS * JW];
  const bool fin_lds = njobs <= BATCH_LDS_JOBS;
  if (fin_lds) {
    for (uint32_t k = threadIdx.x; k < njobs; k += blockDim.x) {
      lds_store(job_fin + k * JW, jobs[k].hits);
      job_fin[k * JW + JW - 1] = (uint64_t)jobs[k].first | ((uint64_t)jobs[k].is_tri << 32);
    }
    __syncthreads();
  }
  const uint32_t lane = __lane_id();
  SpillArea<SPLIT> spill;
  RingStack<SPLIT> st;
  ring_bind<SPLIT>(st, smem, &spill, ring);
  Ray r;
  Ray32 q;
  Hit s;
  Trav t;
  t.active = false;
  bool has_ray = false;
  bool exhausted = false;  // wave-uniform
  uint64_t idx = 0;
  uint32_t j = 0;
  BvhView bv{};  // this lane's job's tree, kept across steps (the step reads only its node and record pointers)
  WavePool pool;
  for (;;) {
    if (!exhausted) {
      const unsigned long long idle = __ballot(!has_ray);
      const uint32_t nidle = (uint32_t)__popcll(idle);
      if (nidle >= refill || nidle == 64u) {
        bool got;
        uint64_t g = 0;
        pool_refill(pool, counter, total, chunk, idle, nidle, lane, got, g, exhausted);
        // A claim is a run of consecutive indices and usually lies in one job: find the jobs of its first and last
        // index once per wave (wave-uniform, so scalar loads), and search per lane only when they differ.
        bool from_list = false;
        if constexpr (AFTER_FAST) {
          from_list = got && g >= left.scan;
          if (from_list) g = list_entry(deferred - COUNTER_DEFERRED, list_ends, (uint32_t)(g - left.scan));
        }
        const unsigned long long gm = __ballot(got);
        if (gm) {
          const int lo = __ffsll((long long)gm) - 1, hi = 63 - __clzll((long long)gm);
          const uint64_t g_lo = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(g >> 32), lo) << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)g, lo);
          const uint64_t g_hi = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(g >> 32), hi) << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)g, hi);
          const uint32_t j_lo = find_job(jobs, njobs, g_lo);
          // (indices from the list are in no order)
          const bool one_job = !AFTER_FAST && (j_lo + 1u >= njobs || jobs[j_lo + 1u].offset > g_hi);
          if (got) {
            j = one_job ? j_lo : find_job(jobs, njobs, g);
            const BatchJob &J = jobs[j];
            const uint64_t local = g - J.offset;
            idx = J.order ? (uint64_t)J.order[local] : local;
            bv = J.bvh;
            start_ray<SPLIT>(bv, J.rays, idx, J.extent, r, q, s);
            bool trace = true;
            if constexpr (AFTER_FAST) trace = from_list || left.all || !fast_ray<Rec>(J.rays, idx, J.extent, (flags & FLAG_SPLIT) != 0u);
            if (SPLIT && deferred_to_exact(r)) {
              __atomic_store_n(deferred, 1ull, __ATOMIC_RELAXED);
            } else if (trace && (!deferred_only || deferred_to_exact(r))) {
              has_ray = true;
              trav_begin<SPLIT>(bv, r, q, s, t);
              st.reset();
            }
          }
        }
      }
    }
    if (!__ballot(has_ray) && exhausted) break;
    if (has_ray) {
      if (t.active) trav_step<Rec, SPLIT>(bv, r, q, any_hit, s, t, st);
      if (!t.active) {
        HitsView hv;
        uint32_t jfirst, jtri;
        if (fin_lds) {
          __builtin_memcpy(&hv, job_fin + j * JW, sizeof(HitsView));
          const uint64_t w = job_fin[j * JW + JW - 1];
          jfirst = (uint32_t)w;
          jtri = (uint32_t)(w >> 32);
        } else {
          const BatchJob &J = jobs[j];
          hv = J.hits;
          jfirst = J.first;
          jtri = J.is_tri;
        }
        finish_ray<Rec>(bv, hv, idx, r, s, flags, jfirst, jtri);
        has_ray = false;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------ triangles, fast
// Closest hits of a triangle tree, bit-identical to the exact FP64 kernels (k_trace_persistent<TriRec, false>), at
// the cost of FP32 boxes and pre-tests.
//
// The reference's depth-first order is kept (NodeQ::ord), with the reference's own hit distance at every point of it.
// A box is skipped only when the FP32 bounds prove that the reference's slab test or its pop test skips it (Ray32
// below), a triangle only when tri_filter proves that the FP64 test rejects it, and every other triangle gets the FP64
// test itself, in leaf order. So the primitives tested are the reference's, in its order, plus some of boxes that its
// FP64 slab test rejects by a rounding. Those change nothing unless one is accepted. Every accepted hit is therefore
// checked (certified): one that lies inside its triangle by more than the rounding of the test, and clear of the earlier
// hit distance and of tmin by more than the error of its own distance, lies inside every box above it by more than the
// rounding of the slab test (whose far planes are widened by 4 eps), so the reference tests it too, with the same hit
// distance, and accepts it. A ray with a hit that fails the check ends there (what it would find next is of no use), writes
// nothing and is listed for the exact kernel that follows on the stream: 1,048,576 rays aimed at vertices and edges are traced
// at 0.6 of the exact kernel's own speed. Testing the accepted hit's leaf box in FP64 instead spills registers in this loop and
// costs 8-12% on rays that need no check. Rays outside the assumptions of the argument (fast_ray) go there as well.
//
// What bounds it (4,194,304 incoherent rays, 1.31M triangles): the data path of the vector L1 (87% busy: every step reads a
// 128-byte record per lane in eight loads) and the vector ALU (73%, a quarter of the lanes active), with 5.7 TB/s of
// lines beyond L2. Near and far rows are therefore chosen by address instead of by selects, references carry no second
// word, the pre-test has no branches and finished rays are written together.
//
// Once a wave's pool is exhausted, its idle lanes take over stack entries of the busy ones: always the bottom entry,
// the last subtree in the lane's part of the order, with the lane's hit distance as it stands. That distance is at
// least the one the reference would have there, so the helper tests a superset of the reference's primitives; an
// accepted hit is certified as before, and one nearer than the hit of the parts before it would have been accepted in
// the reference's order too. A part also skips what lies behind a hit of a part before it (never of one after it). The
// parts' hits are merged by distance when the last of them ends, and a ray whose parts have two hits within their error
// bounds of each other, and what its direction falls short of unit length, is listed. Sharing takes the incoherent set from
// 3.57 to 3.16 ms and 50,000 rays on 328k triangles from 450 to 268 us; the camera set, whose rays mostly end at their first
// hit, loses 4%.
struct RayQ {
  float inv[3];
  float offn[3], offf[3];  // entry / exit plane offsets, rounded apart (make_ray32)
  float D[3], O[3];        // unit direction and origin, for the pre-test
  float om, tmin;
  float slack;             // >= 1 - |raw direction| where that is positive, else <= it
  // bits 0-4: shift of the octant's order mask, bit 5: its word, bits 6-8: direction signs, bit 9: mask complemented, bit 10:
  // a direction too short for its hits' distances to be merged (split precision)
  uint32_t code;
};

template <bool F32 = false>
__device__ __forceinline__ void make_rayq(const Ray &r, double len2, double S, RayQ &q) {
  Ray32 a;
  make_ray32<F32>(r, S, a);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    q.inv[k] = a.inv[k];
    q.offn[k] = a.offn[k];
    q.offf[k] = a.offf[k];
    q.D[k] = (float)r.d[k];
    q.O[k] = (float)r.o[k];
  }
  q.om = a.om;
  q.tmin = fmaxf(a.tmin, 0.0f);
  const bool brief = len2 < SHORT_LEN2;
  q.slack = brief ? 0.0f : len2 < 1.0 ? f32_up(1.0 - len2) : f32_down(1.0 - __builtin_sqrt(len2));
  const uint32_t s = r.sign & 7u, c = (s & 4u) ? (~s & 3u) : s;
  q.code = ((c & 1u) << 4) | ((c >> 1) << 5) | (s << 6) | ((s >> 2) << 9) | (brief ? 1024u : 0u);
}

// Whether an accepted hit is one that the reference's traversal must reach as well (see above). `thr` is |det| times
// the hit distance before it, `slack` what the ray's direction falls short of unit length. The FP64 test's errors are
// those of tri_filter's table with u = 2^-53; 32 u covers them and the rounding of the record's edges and of the
// normalised direction. The distance h = t / |det| is then known to err / |det|, err = 4 (Et + Ed h), twice over; `rel` is
// that relative to h. The boxes' exits are distances along the direction as given, so a hit has to lie behind tmin by that
// direction's length where it is longer than one.
struct Certificate {
  bool sure;
  float rel;
};
__device__ __forceinline__ Certificate certified(const TriRec &T, const double o[3], double tmin, double slack, double u,
                                                 double v, double w, double t, double ad, double thr) {
  const double sa = fabs(T.e1[0]) + fabs(T.e1[1]) + fabs(T.e1[2]);
  const double sb = fabs(T.e2[0]) + fabs(T.e2[1]) + fabs(T.e2[2]);
  const double Pm = fmax(fabs(T.v0[0]), fmax(fabs(T.v0[1]), fabs(T.v0[2]))) +
                    fmax(fabs(o[0]), fmax(fabs(o[1]), fabs(o[2])));
  const double k = 32.0 * 0x1p-53;
  const double Ed = k * sa * sb + 1e-290, Eu = k * Pm * sb + 1e-290, Ev = k * Pm * sa + 1e-290, Et = Ed * Pm + 1e-290;
  const double err = 4.0 * (Et + Ed * (t * (1.0 / ad)));
  Certificate c;
  c.sure = u > Eu && v > Ev && w > Eu + Ev + Ed && ad >= 0x1p12 * Ed && t >= 0x1p12 * Et &&
           t - err >= ad * tmin * (1.0 + 0x1p-46) * (1.0 - fmin(slack, 0.0)) &&
           t + err < thr * (1.0 - (0x1p-46 + fmax(slack, 0.0)));
  c.rel = (float)(err * (1.0 / t)) * (1.0f + 0x1p-20f);
  return c;
}

__device__ __forceinline__ float max3_nn(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float min3_nn(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

struct TriTrees {
  const NodeQ *nodes;
  const TriFilt *filt;
  const TriRec *recs;
};

// A lane's traversal: cur is a node, or LEAF_BIT | the next primitive of a leaf with `cnt` of them left; cand marks
// the members of the current pre-test group that still need the FP64 test.
struct TriTrav {
  uint32_t cur, cnt, cand;
  float h32;
  float rel;  // largest relative error bound of the accepted hits
  bool active, listed;
};

// One unit of the traversal: an internal node, the pre-test of a leaf's next FILTER_GROUP triangles, or the FP64 test of
// one that passed. As in trav_step, every lane fetches its record by the same instructions and waits once.
__device__ __forceinline__ void tri_step(const TriTrees &T, const Ray &r, const RayQ &q, Hit &s, TriTrav &t,
                                         WideStack &st) {
  using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
  using Bytes = const __attribute__((address_space(1))) unsigned char;
  using GlobalChunk = const __attribute__((address_space(1))) u32x4;
  const bool at_leaf = (t.cur & LEAF_BIT) != 0;
  const bool test = t.cand != 0u;
  const uint32_t first = t.cur & ~LEAF_BIT;
  const uint32_t p = first + (uint32_t)__builtin_ctz(t.cand | 0x80000000u);
  // without pre-test records every triangle of the leaf gets the FP64 test (the fetch then reads node 0)
  Bytes *base = !at_leaf          ? (Bytes *)(T.nodes + t.cur)
                : test            ? (Bytes *)(T.recs + p)
                : T.filt != nullptr ? (Bytes *)(T.filt + first)
                                  : (Bytes *)T.nodes;
  // node lanes read the near row of each axis into chunk a and the far row into chunk 4 + a; the others read 16-byte
  // chunks in order
  const uint32_t code = at_leaf ? 0u : q.code;
  const uint32_t near0 = code & 64u, near1 = (code >> 1) & 64u, near2 = (code >> 2) & 64u;
  u32x4 c0, c1, c2, c3, c4, c5, c6, c7;
  c0 = *(GlobalChunk *)(base + near0);
  c1 = *(GlobalChunk *)(base + near1 + 16);
  c2 = *(GlobalChunk *)(base + near2 + 32);
  c3 = *(GlobalChunk *)(base + 48);
  c4 = *(GlobalChunk *)(base + (64u - near0));
  if (!test) {  // a triangle record ends with chunk 4
    c5 = *(GlobalChunk *)(base + (64u - near1) + 16);
    c6 = *(GlobalChunk *)(base + (64u - near2) + 32);
    c7 = *(GlobalChunk *)(base + 112);
  }
  asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3), "+v"(c4), "+v"(c5), "+v"(c6), "+v"(c7));
  if (!at_leaf) {
    uint32_t m = 0;
    uint32_t key[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float n0 = __builtin_fmaf(__uint_as_float(c0[c]), q.inv[0], q.offn[0]);
      const float n1 = __builtin_fmaf(__uint_as_float(c1[c]), q.inv[1], q.offn[1]);
      const float n2 = __builtin_fmaf(__uint_as_float(c2[c]), q.inv[2], q.offn[2]);
      const float f0 = __builtin_fmaf(__uint_as_float(c4[c]), q.inv[0], q.offf[0]);
      const float f1 = __builtin_fmaf(__uint_as_float(c5[c]), q.inv[1], q.offf[1]);
      const float f2 = __builtin_fmaf(__uint_as_float(c6[c]), q.inv[2], q.offf[2]);
      const float A = max_nn(max3_nn(n0, n1, n2), q.tmin);
      const float M = min_nn(min3_nn(f0, f1, f2), t.h32);
      key[c] = __float_as_uint(A);
      m |= A <= M ? 1u << c : 0u;
    }
    if (m) {
      // the visiting order: slot c goes below the entries of the slots before it, i.e. at sp + the number of entered
      // slots after it; the first one is visited next
      const uint32_t word = (code & 32u) ? c7[1] : c7[0];
      const uint32_t later = (word >> (code & 31u)) ^ (uint32_t)(((int)(code << 22)) >> 31);
      const int n = __popc(m);
      st.room(n - 1);
      uint32_t ncur = 0, ncnt = 0;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        if ((m >> c) & 1u) {
          const int rank = __popc(m & (later >> (4 * c)) & (15u & ~(1u << c)));
          const uint32_t k = __builtin_amdgcn_perm(key[c], c7[2], 0x07060500u | (uint32_t)c);
          if (rank == n - 1) {
            ncur = c3[c];
            ncnt = k & 255u;
          } else {
            st.put(st.sp + rank, c3[c], k);
          }
        }
      }
      st.sp += n - 1;
      t.cur = ncur;
      t.cnt = ncnt;
      return;
    }
  } else if (!test) {
    TriFilt g[2];
    u32x4 raw[8] = {c0, c1, c2, c3, c4, c5, c6, c7};
    __builtin_memcpy(g, raw, sizeof g);
    bool p0 = true, p1 = true;
    if (T.filt != nullptr) {
      p0 = tri_filter(g[0], q.D, q.O, q.om, q.tmin, t.h32);
      p1 = tri_filter(g[1], q.D, q.O, q.om, q.tmin, t.h32);
    }
    t.cand = (p0 ? 1u : 0u) | (p1 && t.cnt > 1u ? 2u : 0u);
    if (t.cand) return;
    if (t.cnt > 2u) {
      t.cnt -= 2u;
      t.cur += 2u;
      return;
    }
  } else {
    TriRec rec;
    u32x4 raw[5] = {c0, c1, c2, c3, c4};
    __builtin_memcpy(&rec, raw, sizeof rec);
    Certificate c{true, 0.0f};
    if (isect_tri(rec, r, s, p, [&](double u, double v, double w, double tt, double ad, double thr) {
          c = certified(rec, r.o, r.tmin, (double)q.slack, u, v, w, tt, ad, thr);
        })) {
      t.h32 = f32_up(s.h);
      t.rel = fmaxf(t.rel, c.rel);
      if (!c.sure) {  // the exact kernel's
        t.listed = true;
        t.active = false;
        return;
      }
    }
    t.cand &= t.cand - 1u;
    if (t.cand) return;
    if (t.cnt > 2u) {
      t.cnt -= 2u;
      t.cur += 2u;
      return;
    }
  }
  while (st.sp > st.bot) {
    const WideEntry e = st.pop();
    if (!(t.h32 < __uint_as_float(e.key & ~255u))) {
      t.cur = e.ref;
      t.cnt = e.key & 255u;
      return;
    }
  }
  t.active = false;
}

// Starts a ray: its root test, with the FP32 bounds.
struct TriRoot {
  float lo[3], hi[3];
  uint32_t ref, cnt;
};
__device__ __forceinline__ TriRoot tri_root(const BvhView &bvh) {
  return TriRoot{{bvh.root_min32[0], bvh.root_min32[1], bvh.root_min32[2]},
                 {bvh.root_max32[0], bvh.root_max32[1], bvh.root_max32[2]}, bvh.root_ref4, bvh.root_cnt};
}
template <class R>
__device__ __forceinline__ void tri_begin(const TriRoot &root, const RayT<R> &r, const RayQ &q, const HitT<R> &s,
                                          TriTrav &t) {
  t.cur = root.ref;
  t.cnt = root.cnt;
  t.cand = 0;
  t.listed = false;
  t.rel = 0.0f;
  t.h32 = f32_up(s.h);
  float A = q.tmin, M = t.h32;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const bool sg = (r.sign >> a) & 1u;
    const float lo = root.lo[a], hi = root.hi[a];
    A = fmaxf(A, __builtin_fmaf(sg ? hi : lo, q.inv[a], q.offn[a]));
    M = fminf(M, __builtin_fmaf(sg ? lo : hi, q.inv[a], q.offf[a]));
  }
  t.active = A <= M;
}

// Rays whose parts several lanes trace.
struct TriShare {
  double h[SHARE_SLOTS], u[SHARE_SLOTS], v[SHARE_SLOTS];
  uint32_t prim[SHARE_SLOTS];
  uint32_t parts[SHARE_SLOTS];  // parts still running; bit 31: the ray is to be listed
  float rel[SHARE_SLOTS];
  // smallest accepted hit distance so far, as the bits of its FP32 upper bound above the position of the part that
  // accepted it in the traversal order: the parts after that one skip what lies behind it
  unsigned long long bound[SHARE_SLOTS];
};

__device__ __forceinline__ unsigned long long bound_of(float h32, uint32_t pos) {
  return ((unsigned long long)__float_as_uint(h32) << 32) | pos;  // h32 >= 0: its bits order as it does
}

// Persistent waves as in k_trace_persistent. BATCH: the rays of many jobs, as in k_trace_batch. LONE: one ray by one wave,
// without counters; where it would be listed or deferred, `merged` says so (RAY_LEFT) and nothing else is written.
// FIXED: the waves of a single-scene launch take `fixed` rays each and mark the rays left in a word of their own (a kernel of
// its own: in the claiming one that code costs 7%).
template <bool BATCH, bool LONE = false, bool FIXED = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BRT_WAVES_PER_EU)))
k_trace_tri(BvhView bvh, RaysView rays, HitsView hits, const BatchJob *__restrict__ jobs, uint32_t njobs, uint64_t n,
            uint32_t flags, uint32_t first, double S, unsigned long long *group, uint32_t refill,
            const uint32_t *order, uint32_t ring, uint32_t chunk, uint32_t fixed) {
  extern __shared__ unsigned char smem[];
  __shared__ TriShare shares[4];
  constexpr int RW = (int)(sizeof(RaysView) / 8), HW = (int)(sizeof(HitsView) / 8);
  __shared__ uint64_t views[RW + HW];  // ray and hit columns, read back where they are used (see k_trace_persistent)
  if constexpr (!BATCH) {
    if (threadIdx.x == 0) {
      lds_store(views, rays);
      lds_store(views + RW, hits);
    }
    __syncthreads();
  }
  // as in k_trace_batch, with the geometry id in place of is_tri
  constexpr int JW = HW + 1;
  __shared__ uint64_t job_fin[BATCH ? BATCH_LDS_JOBS * JW : 1];
  const bool fin_lds = njobs <= BATCH_LDS_JOBS;
  if constexpr (BATCH) {
    if (fin_lds) {
      for (uint32_t k = threadIdx.x; k < njobs; k += blockDim.x) {
        lds_store(job_fin + k * JW, jobs[k].hits);
        job_fin[k * JW + JW - 1] = (uint64_t)jobs[k].first | ((uint64_t)jobs[k].bvh.geom_id << 32);
      }
      __syncthreads();
    }
  }
  const uint32_t lane = __lane_id(), wave = threadIdx.x / 64;
  BRT_LDS volatile TriShare *sh = (BRT_LDS volatile TriShare *)&shares[wave];
  uint64_t spill[WIDE_SPILL];
  WideStack st;
  st.ring = (BRT_LDS uint32_t *)smem + (size_t)wave * ring * 128 + lane;
  st.spill = spill;
  st.mask = (int)ring - 1;
  st.reset();
  TriTrees T{bvh.nodesq, bvh.tri_filter, reinterpret_cast<const TriRec *>(bvh.prims)};
  Ray r;
  RayQ q;
  Hit s;
  TriTrav t;
  t.active = false;
  t.cand = 0;
  bool has_ray = false, shared = false;
  bool done = false;       // a traced ray, still to be written
  bool exhausted = false;  // wave-uniform
  uint32_t pos = 0, pos_end = 0;  // shared rays: this part's positions in the traversal order
  uint32_t slot = 0, slots = 0;  // the share slot of this lane's ray; slots given out (wave-uniform)
  uint64_t idx = 0;        // ray index, within its job
  uint32_t j = 0;
  uint32_t number = 0;  // FIXED: the ray's in the wave's range
  unsigned long long mask = 0;  // wave-uniform
  // Finished rays are written together, when the wave refills: a ray ends in almost every iteration, and writing it
  // there would run this code for a lane or two each time.
  auto write_rays = [&]() {
    if constexpr (FIXED) mask_add(mask, done && t.listed, number);
    if (done) {
      done = false;
      if (t.listed) {
        if constexpr (LONE) st_stream(lds_fresh<HitsView>(views + RW).merged, idx, RAY_LEFT);
        else if constexpr (!FIXED) list_ray(BATCH ? jobs[j].offset + idx : idx, group);
      } else {
        r.tmax = s.leaf_idx == INVALID_ID ? -__builtin_inf() : __builtin_inf();  // hit or not, for finish_ray
        if constexpr (BATCH) {
          HitsView hv;
          BvhView fb{};
          uint32_t jfirst;
          if (fin_lds) {
            __builtin_memcpy(&hv, job_fin + j * JW, sizeof(HitsView));
            const uint64_t w = job_fin[j * JW + JW - 1];
            jfirst = (uint32_t)w;
            fb.geom_id = (uint32_t)(w >> 32);
          } else {
            hv = jobs[j].hits;
            jfirst = jobs[j].first;
            fb.geom_id = jobs[j].bvh.geom_id;
          }
          if (hv.nx) {
            fb.faces = jobs[j].bvh.faces;
            fb.vnormals = jobs[j].bvh.vnormals;
          }
          finish_ray<TriRec>(fb, hv, idx, r, s, flags, jfirst, 1u);
        } else {
          finish_ray<TriRec>(bvh, lds_fresh<HitsView>(views + RW), idx, r, s, flags, first, 1u);
        }
      }
    }
  };
  WavePool pool;
  const uint64_t global_wave = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave, range = global_wave * fixed;
  if (fixed)  // a small launch: no claims, and the other lanes help from the start
    pool.take_fixed(range, fixed, n);
  uint32_t turn = 0;
  bool noted = false;  // see note_passed
  for (;;) {
    if (!exhausted) {
      const unsigned long long idle = __ballot(!has_ray);
      const uint32_t nidle = (uint32_t)__popcll(idle);
      if (nidle >= refill || nidle == 64u) {
        write_rays();
        bool got;
        uint64_t cand = 0;
        pool_refill(pool, group + COUNTER_POOL, n, chunk, idle, nidle, lane, got, cand, exhausted);
        bool defer = false;
        double ext = S;
        TriRoot root{};
        RawRay raw{};
        if constexpr (BATCH) {
          const unsigned long long gm = __ballot(got);
          if (gm) {
            // The jobs of the claim's first and last index, once per wave. Nearly always they are one job, whose record
            // is then read by scalar loads; otherwise every lane searches for its own.
            const int lo = __ffsll((long long)gm) - 1, hi = 63 - __clzll((long long)gm);
            const uint64_t g_lo = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(cand >> 32), lo) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)cand, lo);
            const uint64_t g_hi = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(cand >> 32), hi) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)cand, hi);
            const uint32_t j_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)find_job(jobs, njobs, g_lo));
            const bool one_job = j_lo + 1u >= njobs || jobs[j_lo + 1u].offset > g_hi;
            const auto take = [&](const BatchJob &J) {
              idx = cand - J.offset;  // batches trace in input order
              ext = J.extent;
              T = TriTrees{J.bvh.nodesq, J.bvh.tri_filter, reinterpret_cast<const TriRec *>(J.bvh.prims)};
              root = tri_root(J.bvh);
              raw = load_ray(J.rays, idx);
            };
            if (one_job) {
              const BatchJob &J = jobs[j_lo];
              if (got) {
                j = j_lo;
                take(J);
              }
            } else if (got) {
              j = find_job(jobs, njobs, cand);
              take(jobs[j]);
            }
          }
        } else if (LONE || got) {
          if constexpr (FIXED) number = (uint32_t)(cand - range);
          idx = order ? (uint64_t)order[cand] : cand;
          root = tri_root(bvh);
          raw = load_ray(lds_fresh<RaysView>(views), idx);
        }
        if (LONE || got) {
          setup_ray(raw.org, raw.dir, raw.tmin, raw.tmax, r);
          const double len2 = squared_length(raw);
          if (fast_ray(r, len2, ext, (flags & FLAG_SPLIT) != 0u)) {
            has_ray = got;
            make_rayq(r, len2, ext, q);
            s.h = r.tmax;
            s.u = s.v = 0.0;
            s.leaf_idx = INVALID_ID;
            tri_begin(root, r, q, s, t);
            st.reset();
          } else if (r.o[2] != r.o[2] || r.inv[2] != r.inv[2]) {
            // NaN far-plane terms on the last axis: the reference rejects every box, the root first (a mirror ray
            // that has left the scene)
            has_ray = got;
            s.leaf_idx = INVALID_ID;
            t.active = t.listed = false;
          } else if constexpr (LONE) {
            st_stream(lds_fresh<HitsView>(views + RW).merged, idx, RAY_LEFT);
          } else {
            defer = true;
          }
        }
        if constexpr (FIXED) mask_add(mask, defer, number);
        else if constexpr (!LONE) {
          if (!noted && __ballot(defer)) {
            noted = true;
            note_passed(true, group, lane);
          }
        }
      }
    }
    const unsigned long long busy = __ballot(has_ray);
    if (exhausted) {
      if (!busy) {
        write_rays();
        if (FIXED && lane == 0) group[COUNTER_CLEARED + global_wave] = mask;
        break;
      }
      const unsigned long long can = __ballot(has_ray && st.sp > st.bot && !(q.code & 1024u));
      const uint32_t nidle = 64u - (uint32_t)__popcll(busy);
      // in every other iteration: sharing costs about as many instructions as a traversal step (every one: 3-5% slower);
      // a lone ray has the instruction slots to itself and shares in every one (41.4 -> 38.4 us a call; not at all: 46.0 us)
      if (nidle >= SHARE_MIN_IDLE && can && (LONE || (++turn & 1u) == 0u)) {
        write_rays();  // the helpers' state is overwritten
        const unsigned long long below = (1ull << lane) - 1ull;
        const uint32_t ncan = (uint32_t)__popcll(can), k = nidle < ncan ? nidle : ncan;
        const uint32_t rank = (uint32_t)__popcll((has_ray ? can : ~busy) & below);
        const bool donor = ((can >> lane) & 1ull) && rank < k, helper = !has_ray && rank < k;
        const uint32_t pos_end0 = shared ? pos_end : 0xffffffffu;
        // the r-th helper takes from the r-th donor, whose lane number lane r receives
        const unsigned long long fresh = __ballot(donor && !shared);
        uint64_t e = 0;
        if (donor) {
          e = st.take_bottom();
          if (!shared) {
            shared = true;
            slot = slots + (uint32_t)__popcll(fresh & below);
            sh->parts[slot] = 1u;
            sh->prim[slot] = INVALID_ID;
            sh->h[slot] = __builtin_inf();
            sh->rel[slot] = 0.0f;
            sh->bound[slot] = bound_of(t.h32, 0u);
            pos = 0u;
            pos_end = 0xffffffffu;
          }
          pos_end -= (pos_end - pos) >> 3;  // the helper's part is the last eighth of the positions
        }
        slots += (uint32_t)__popcll(fresh);
        wave_fence();
        if (donor) atomicAdd(&shares[wave].parts[slot], 1u);
        // (at most 32 donors: lane 63 takes what the others push)
        const uint32_t by_rank = (uint32_t)__builtin_amdgcn_ds_permute((donor ? (int)rank : 63) << 2, (int)lane);
        const uint32_t from = lane_get(by_rank, (int)rank);  // with all lanes: a permute reads active lanes only
        const int src = helper ? (int)from : (int)lane;
        lane_take(e, src, helper);
        if constexpr (!LONE) {  // all lanes hold a lone ray, in slot 0
          lane_take(r.o, src, helper);
          lane_take(r.d, src, helper);
          lane_take(r.tmin, src, helper);
          lane_take(q, src, helper);
          lane_take(idx, src, helper);
          lane_take(slot, src, helper);
          if constexpr (FIXED) lane_take(number, src, helper);
        }
        lane_take(s.h, src, helper);
        lane_take(t.h32, src, helper);
        {
          const uint32_t from_end = lane_get(pos_end, src), old_end = lane_get(pos_end0, src);
          pos = helper ? from_end : pos;
          pos_end = helper ? old_end : pos_end;
        }
        if constexpr (BATCH) {
          lane_take(T, src, helper);
          lane_take(j, src, helper);
        }
        if (helper) {
          has_ray = true;
          shared = true;
          s.leaf_idx = INVALID_ID;
          t.cur = (uint32_t)e;
          t.cnt = (uint32_t)(e >> 32) & 255u;
          t.cand = 0;
          t.listed = false;
          t.rel = 0.0f;
          t.active = !(t.h32 < __uint_as_float((uint32_t)(e >> 32) & ~255u));
          st.reset();
        }
        wave_fence();
      }
    }
    if (has_ray && t.active) {
      if (shared) {
        const unsigned long long b = sh->bound[slot];
        const float h32 = __uint_as_float((uint32_t)(b >> 32));
        if ((uint32_t)b < pos && h32 < t.h32) {  // an earlier part's hit: this part's own, if it lies behind, is void
          t.h32 = h32;
          s.h = (double)h32;
          s.leaf_idx = INVALID_ID;
        }
      }
      const uint32_t before = s.leaf_idx;
      tri_step(T, r, q, s, t, st);
      if (shared && s.leaf_idx != before && s.h >= 0.0) atomicMin(&shares[wave].bound[slot], bound_of(t.h32, pos));
    }
    bool fin = has_ray && !t.active;
    if (exhausted) {
      // the parts of a shared ray are merged one lane at a time; the last one writes the ray
      unsigned long long m = __ballot(fin && shared);
      while (m) {
        const uint32_t l = (uint32_t)__ffsll((long long)m) - 1u;
        m &= m - 1ull;
        if (lane == l) {
          uint32_t parts = sh->parts[slot];
          if (t.listed) parts |= 0x80000000u;
          if (s.leaf_idx != INVALID_ID) {
            const double h = sh->h[slot];
            const float rel = fmaxf(t.rel, sh->rel[slot]);
            sh->rel[slot] = rel;
            // (the nearer one may lie in a box whose entry, along a direction shorter than one, is behind the other)
            const double close = 2.0 * ((double)rel + (double)fmaxf(q.slack, 0.0f)) + 0x1p-46;
            if (fabs(s.h - h) <= close * s.h) parts |= 0x80000000u;
            if (s.h < h) {
              sh->h[slot] = s.h;
              sh->u[slot] = s.u;
              sh->v[slot] = s.v;
              sh->prim[slot] = s.leaf_idx;
            }
          }
          parts--;
          sh->parts[slot] = parts;
          has_ray = false;
          shared = false;
          if ((parts & 0x7fffffffu) == 0u) {
            s.h = sh->h[slot];
            s.u = sh->u[slot];
            s.v = sh->v[slot];
            s.leaf_idx = sh->prim[slot];
            t.listed = (parts >> 31) != 0u;
          } else {
            fin = false;
          }
        }
        wave_fence();
      }
    }
    done = done || fin;
    if (fin) has_ray = false;
  }
}

// ------------------------------------------------------------------------------------------------ leaf checks, fast
// Closest hits of spheres and cylinders, and of a Scene<float>'s triangles, bit-identical to the exact kernel
// (k_trace_persistent<Rec, false>), with the FP32 boxes and the visiting order of k_trace_tri. No certificate is needed: when
// a primitive reports a hit and its leaf has
// not been checked yet, the reference's own slab and pop tests of the leaf's box, in the scene type and at the hit distance as
// it stands, decide whether the reference tests the leaf at all. That leaf's test decides for the boxes above it too. They hold its box
// and every operation of the slab test is monotone, so they pass the slab test with it, with an entry distance no larger. As
// to their pop tests: of the boxes above it, those popped before the last accepted hit are boxes above that hit's leaf as
// well (a depth-first stack holds only siblings of the path), which was checked; those popped since saw the hit distance
// that the leaf's test sees. An FP32 pop test (at most the reference's entry distance against at least its hit distance)
// skips only what the reference skips. So does a box left out of the stack, since hit distances only shrink: a ray on which
// a sphere's grows by a rounding is listed for the exact kernel; a cylinder's last hit counts, so its distance may grow, and
// only the slab test leaves its boxes out.
//
// What bounds it (8,388,608 incoherent rays): the vector ALU, 74% busy with a quarter of the lanes active, since a wave runs
// the node, pre-test and FP64 branches in almost every iteration for a few lanes each. Lanes with an FP64 test, or with a
// pre-test, therefore wait until WIDE_MIN_LANES of the wave have one (or no other lane has anything else to do): 50,000
// spheres 4.19 -> 3.24 ms (8 lanes: 3.36, 24: 3.62), against 4.44 ms for the exact kernel; 10,000 cylinders 4.90 -> 4.59 ms
// (3.30 with the pre-test against the axis), against 5.45 ms. (k_trace_tri, bound by the data path of the L1, gains nothing
// from it.) A wave with no rays left to take
// doesn't wait: there the longest ray counts. In FP32 the primitives are tested without a pre-test.
// Primitives without a pre-test tested per step. Triangles in FP32, 1,000,003 incoherent rays on 327,680: 1 per step 0.88,
// 2: 0.71, 3: 0.68, 4: 0.65 ms.
template <class Rec>
constexpr uint32_t wide_tests() { return Rec::kind == CYLINDERS ? 1u : 4u; }

// FP32 pre-tests belong to the FP64 types: a Scene<float>'s own tests cost no more.
template <class Rec>
constexpr bool wide_filter() { return sizeof(typename Rec::real) == 8; }

struct WideTrav {
  uint32_t cur, cnt, cand;
  uint32_t leaf;  // first primitive of the leaf
  float h32;
  bool active, listed, seen;  // seen: the reference tests this leaf
};

// One unit of the traversal: an internal node, the pre-test of a leaf's next SPH_FILTER_GROUP primitives or the FP64 test of
// one, or in FP32 the tests of its next wide_tests.
template <class Rec, class Inv>
__device__ __forceinline__ void wide_step(const BvhView &bvh, const RayT<typename Rec::real> &r, const RayQ &q,
                                          HitT<typename Rec::real> &s, WideTrav &t, WideStack &st, Inv &&load_inv,
                                          bool wait) {
  using R = typename Rec::real;
  using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
  using Bytes = const __attribute__((address_space(1))) unsigned char;
  using GlobalChunk = const __attribute__((address_space(1))) u32x4;
  constexpr bool FILTER = wide_filter<Rec>();
  constexpr bool GROWS = Rec::kind == CYLINDERS;
  using Filt = typename std::conditional<GROWS, CylFilt, SphFilt>::type;
  constexpr uint32_t FG = FILTER ? SPH_FILTER_GROUP : wide_tests<Rec>();  // primitives per pre-test, or per test without
  constexpr int REC_Q = (int)(sizeof(Rec) / 16), FILT_Q = FILTER ? (int)(FG * sizeof(Filt) / 16) : 0;
  constexpr int MORE = FILTER || FG * REC_Q <= 8 ? 0 : FG * REC_Q - 8;  // chunks a leaf step reads beyond a node's eight
  const Filt *filt = nullptr;
  if constexpr (FILTER && GROWS) filt = bvh.cyl_filter;
  else if constexpr (FILTER) filt = bvh.sph_filter;
  const bool at_leaf = (t.cur & LEAF_BIT) != 0;
  const bool test = FILTER ? t.cand != 0u : at_leaf;
  if (wait) {
    const bool group = at_leaf && !test;
    const int tests = __popcll(__ballot(test)), groups = FILTER ? __popcll(__ballot(group)) : 0;
    const int nodes = __popcll(__ballot(true)) - tests - groups;
    if (test && tests < WIDE_MIN_LANES && nodes + groups != 0) return;
    if (group && groups < WIDE_MIN_LANES && nodes != 0) return;
  }
  const uint32_t first = t.cur & ~LEAF_BIT;
  const uint32_t p = first + (FILTER ? (uint32_t)__builtin_ctz(t.cand | 0x80000000u) : 0u);
  // without pre-test records every primitive gets the FP64 test (the fetch then reads node 0)
  Bytes *base = !at_leaf          ? (Bytes *)(bvh.nodesq + t.cur)
                : test            ? (Bytes *)(reinterpret_cast<const Rec *>(bvh.prims) + p)
                : filt != nullptr ? (Bytes *)(filt + first)
                                  : (Bytes *)bvh.nodesq;
  const uint32_t code = at_leaf ? 0u : q.code;
  const uint32_t near0 = code & 64u, near1 = (code >> 1) & 64u, near2 = (code >> 2) & 64u;
  // chunk k of the records a leaf step reads: only those of the leaf's own primitives are sure to be there
  const auto has = [&](int k) {
    if constexpr (FILTER) return test ? k < REC_Q : k < FILT_Q;
    else return k / REC_Q < (int)FG && (uint32_t)(k / REC_Q) < t.cnt;
  };
  u32x4 c0, c1, c2, c3, c4, c5, c6, c7;
  c0 = *(GlobalChunk *)(base + near0);
  if constexpr (FILTER) {
    c1 = *(GlobalChunk *)(base + near1 + 16);
    if (!at_leaf || has(3)) {
      c2 = *(GlobalChunk *)(base + near2 + 32);
      c3 = *(GlobalChunk *)(base + 48);
    }
    if (!at_leaf || has(7)) {
      c4 = *(GlobalChunk *)(base + (64u - near0));
      c5 = *(GlobalChunk *)(base + (64u - near1) + 16);
      c6 = *(GlobalChunk *)(base + (64u - near2) + 32);
      c7 = *(GlobalChunk *)(base + 112);
    }
  } else {
    if (!at_leaf || has(1)) c1 = *(GlobalChunk *)(base + near1 + 16);
    if (!at_leaf || has(2)) c2 = *(GlobalChunk *)(base + near2 + 32);
    if (!at_leaf || has(3)) c3 = *(GlobalChunk *)(base + 48);
    if (!at_leaf || has(4)) c4 = *(GlobalChunk *)(base + (64u - near0));
    if (!at_leaf || has(5)) c5 = *(GlobalChunk *)(base + (64u - near1) + 16);
    if (!at_leaf || has(6)) c6 = *(GlobalChunk *)(base + (64u - near2) + 32);
    if (!at_leaf || has(7)) c7 = *(GlobalChunk *)(base + 112);
  }
  u32x4 more[MORE + 1];
#pragma unroll
  for (int k = 0; k < MORE; k++)
    if (at_leaf && has(8 + k)) more[k] = *(GlobalChunk *)(base + 128 + 16 * k);
#pragma unroll
  for (int k = 0; k < MORE; k++) asm volatile("" : "+v"(more[k]));
  asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3), "+v"(c4), "+v"(c5), "+v"(c6), "+v"(c7));
  if (!at_leaf) {
    uint32_t m = 0;
    uint32_t key[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float n0 = __builtin_fmaf(__uint_as_float(c0[c]), q.inv[0], q.offn[0]);
      const float n1 = __builtin_fmaf(__uint_as_float(c1[c]), q.inv[1], q.offn[1]);
      const float n2 = __builtin_fmaf(__uint_as_float(c2[c]), q.inv[2], q.offn[2]);
      const float f0 = __builtin_fmaf(__uint_as_float(c4[c]), q.inv[0], q.offf[0]);
      const float f1 = __builtin_fmaf(__uint_as_float(c5[c]), q.inv[1], q.offf[1]);
      const float f2 = __builtin_fmaf(__uint_as_float(c6[c]), q.inv[2], q.offf[2]);
      const float A = max_nn(max3_nn(n0, n1, n2), q.tmin);
      float M = min3_nn(f0, f1, f2);
      if constexpr (!GROWS) M = min_nn(M, t.h32);  // a cylinder's hit distance may have grown when the entry is popped
      key[c] = __float_as_uint(A);
      m |= A <= M ? 1u << c : 0u;
    }
    if (m) {
      const uint32_t word = (code & 32u) ? c7[1] : c7[0];
      const uint32_t later = (word >> (code & 31u)) ^ (uint32_t)(((int)(code << 22)) >> 31);
      const int n = __popc(m);
      st.room(n - 1);
      uint32_t ncur = 0, ncnt = 0;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        if ((m >> c) & 1u) {
          const int rank = __popc(m & (later >> (4 * c)) & (15u & ~(1u << c)));
          const uint32_t k = __builtin_amdgcn_perm(key[c], c7[2], 0x07060500u | (uint32_t)c);
          if (rank == n - 1) {
            ncur = c3[c];
            ncnt = k;
          } else {
            st.put(st.sp + rank, c3[c], k);
          }
        }
      }
      st.sp += n - 1;
      if (!GROWS || !(t.h32 < __uint_as_float(ncnt & ~255u))) {
        t.cur = ncur;
        t.cnt = ncnt & 255u;
        t.leaf = ncur & ~LEAF_BIT;
        t.seen = false;
        return;
      }
    }
  } else if (FILTER && !test) {
    Filt g[FG];
    u32x4 raw[8] = {c0, c1, c2, c3, c4, c5, c6, c7};
    __builtin_memcpy(g, raw, sizeof g);
    uint32_t mask = 0;
#pragma unroll
    for (uint32_t j = 0; j < FG; j++) {
      bool pass = true;
      if (filt != nullptr) {
        if constexpr (GROWS) pass = cyl_filter(g[j], q.D, q.O, q.om);
        else pass = sph_filter(g[j], q.D, q.O, q.om, q.tmin, t.h32);
      }
      if (j < t.cnt && pass) mask |= 1u << j;
    }
    t.cand = mask;
    if (mask) return;
    if (t.cnt > FG) {
      t.cnt -= FG;
      t.cur += FG;
      return;
    }
  } else {
    u32x4 raw[8 + MORE] = {c0, c1, c2, c3, c4, c5, c6, c7};
#pragma unroll
    for (int k = 0; k < MORE; k++) raw[8 + k] = more[k];
#pragma unroll
    for (uint32_t g = 0; g < (FILTER ? 1u : FG); g++) {
      if (g >= t.cnt) break;
      Rec rec;
      __builtin_memcpy(&rec, raw + g * REC_Q, sizeof rec);
      const HitT<R> old = s;
      if (isect(rec, r, s, p + g)) {
        if (!t.seen) {
          RayT<R> x = r;
          load_inv(x);
          const R *b = (const R *)bvh.leaf_boxes + 6ull * t.leaf;
          const R box[6] = {gmem(b)[0], gmem(b)[1], gmem(b)[2], gmem(b)[3], gmem(b)[4], gmem(b)[5]};
          R key;
          t.seen = slab_exact(box, x, key) && !(old.h < key);
        }
        if (t.seen) {
          t.h32 = f32_up(s.h);
          if constexpr (!GROWS) t.listed = t.listed || !(s.h <= old.h);
        } else {  // not a leaf of the reference's: none of its primitives counts
          s = old;
          t.cnt = 0;
          t.cand = 0;
        }
      }
    }
    if constexpr (FILTER) {
      t.cand &= t.cand - 1u;
      if (t.cand) return;
    }
    if (t.cnt > FG) {
      t.cnt -= FG;
      t.cur += FG;
      return;
    }
  }
  while (st.sp > 0) {
    const WideEntry e = st.pop();
    if (!(t.h32 < __uint_as_float(e.key & ~255u))) {
      t.cur = e.ref;
      t.cnt = e.key & 255u;
      t.leaf = e.ref & ~LEAF_BIT;
      t.seen = false;
      return;
    }
  }
  t.active = false;
}

template <class Rec, bool FIXED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BRT_WAVES_PER_EU)))
k_trace_wide(BvhView bvh, RaysViewT<typename Rec::real> rays, HitsViewT<typename Rec::real> hits, uint64_t n,
             uint32_t flags, uint32_t first, uint32_t is_tri, double S, unsigned long long *group, uint32_t refill,
             const uint32_t *order, uint32_t ring, uint32_t chunk,
             uint32_t fixed) {
  using R = typename Rec::real;
  using RaysV = RaysViewT<R>;
  using HitsV = HitsViewT<R>;
  extern __shared__ unsigned char smem[];
  constexpr int RW = (int)(sizeof(RaysV) / 8), HW = (int)(sizeof(HitsV) / 8);
  __shared__ uint64_t views[RW + HW];  // ray and hit columns, read back where they are used (see k_trace_persistent)
  if (threadIdx.x == 0) {
    lds_store(views, rays);
    lds_store(views + RW, hits);
  }
  __syncthreads();
  const uint32_t lane = __lane_id(), wave = threadIdx.x / 64;
  uint64_t spill[WIDE_SPILL];
  WideStack st;
  st.ring = (BRT_LDS uint32_t *)smem + (size_t)wave * ring * 128 + lane;
  st.spill = spill;
  st.mask = (int)ring - 1;
  st.reset();
  RayT<R> r;
  RayQ q;
  HitT<R> s;
  WideTrav t;
  t.active = false;
  t.cand = 0;
  bool has_ray = false, done = false, exhausted = false;
  uint64_t idx = 0;
  uint32_t number = 0;  // see k_trace_tri
  unsigned long long mask = 0;
  const auto write_rays = [&]() {  // finished rays are written together (see k_trace_tri)
    if constexpr (FIXED) mask_add(mask, done && t.listed, number);
    if (done) {
      done = false;
      if (t.listed) {
        if constexpr (!FIXED) list_ray(idx, group);
      } else {
        finish_ray<Rec>(bvh, lds_fresh<HitsV>(views + RW), idx, r, s, flags, first, is_tri);
      }
    }
  };
  const auto load_inv = [&](RayT<R> &x) {
    const RaysV V = lds_fresh<RaysV>(views);
    x.inv[0] = R(1) / V.dx[idx];
    x.inv[1] = R(1) / V.dy[idx];
    x.inv[2] = R(1) / V.dz[idx];
  };
  WavePool pool;
  const uint64_t global_wave = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave, range = global_wave * fixed;
  if constexpr (FIXED) pool.take_fixed(range, fixed, n);
  bool noted = false;  // see note_passed
  for (;;) {
    if (!exhausted) {
      const unsigned long long idle = __ballot(!has_ray);
      const uint32_t nidle = (uint32_t)__popcll(idle);
      if (nidle >= refill || nidle == 64u) {
        write_rays();
        bool got;
        uint64_t cand = 0;
        pool_refill(pool, group + COUNTER_POOL, n, chunk, idle, nidle, lane, got, cand, exhausted);
        bool defer = false;
        if (got) {
          if constexpr (FIXED) number = (uint32_t)(cand - range);
          idx = order ? (uint64_t)order[cand] : cand;
          const RawRayT<R> raw = load_ray(lds_fresh<RaysV>(views), idx);
          setup_ray(raw.org, raw.dir, raw.tmin, raw.tmax, r);
          if (wide_ray(r, S)) {
            has_ray = true;
            if constexpr (sizeof(R) == 8) {
              make_rayq(r, 1.0, S, q);
            } else {
              const Ray x{{r.o[0], r.o[1], r.o[2]}, {r.d[0], r.d[1], r.d[2]}, {r.inv[0], r.inv[1], r.inv[2]}, r.sign,
                          r.tmin, r.tmax};
              make_rayq<true>(x, 1.0, S, q);
            }
            s.h = r.tmax;
            s.u = s.v = R(0);
            s.leaf_idx = INVALID_ID;
            TriTrav b;
            tri_begin(tri_root(bvh), r, q, s, b);
            t = WideTrav{b.cur, b.cnt, 0u, b.cur & ~LEAF_BIT, b.h32, b.active, false, false};
            st.reset();
          } else {
            defer = true;
          }
        }
        if constexpr (FIXED) mask_add(mask, defer, number);
        else noted = noted || __ballot(defer) != 0ull;
      }
    }
    if (exhausted && !__ballot(has_ray)) {
      write_rays();
      if (FIXED && lane == 0) group[COUNTER_CLEARED + global_wave] = mask;
      if constexpr (!FIXED) note_passed(noted, group, lane);
      break;
    }
    if (has_ray) {
      if (t.active) wide_step<Rec>(bvh, r, q, s, t, st, load_inv, !exhausted);
      if (!t.active) {
        done = true;
        has_ray = false;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------ any hit, fast
// Any hit of triangles in split precision: the first hit in the visiting order of trav_step<TriRec, true> (nearest box first,
// ties as its sorting network leaves them), bit for bit. The hit distance never shrinks before the ray ends, so an entry
// that was pushed is always visited: the stack needs no keys, and the parts of a ray are independent. A wave with nothing
// left to start therefore shares its rays' bottom stack entries (the last parts of the order, as k_trace_tri does), and the
// hit of the first part in the order that has one is the ray's; parts behind a hit are dropped.
//
// What bounds it (500,009 shadow rays, 100k triangles): the longest rays; k_trace_persistent<TriRec, true> kept the CUs busy
// for 59% of the launch. Shared work, stack entries of two words and planes chosen by address take 20,000 rays from 136 to
// 88 us a call, 500,009 from 318 to 302, 2,000,000 on 400k triangles from 1.10 to 0.98 ms; of that, waves that refill at 32 idle
// lanes instead of 16 give 3%.
struct AnyShare {
  double h[SHARE_SLOTS], u[SHARE_SLOTS], v[SHARE_SLOTS];
  uint32_t prim[SHARE_SLOTS];
  uint32_t parts[SHARE_SLOTS];  // parts still running
  uint32_t first[SHARE_SLOTS];  // position of the first part with a hit
};

struct AnyRay {
  Ray32 b;
  float D[3], O[3];
};

struct AnyTrav {
  uint32_t cur, cnt, cand;
  float h32;
  bool active;
};

// One unit of the traversal (see tri_step): a Node4, the pre-test of two triangles, or the FP64 test of one.
__device__ __forceinline__ void any_step(const BvhView &bvh, const Ray &r, const AnyRay &q, Hit &s, AnyTrav &t, WideStack &st) {
  using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
  using Bytes = const __attribute__((address_space(1))) unsigned char;
  using GlobalChunk = const __attribute__((address_space(1))) u32x4;
  const bool at_leaf = (t.cur & LEAF_BIT) != 0;
  const bool test = t.cand != 0u;
  const uint32_t first = t.cur & ~LEAF_BIT;
  const uint32_t p = leaf_record(first, t.cand);
  // without pre-test records every triangle of the leaf gets the FP64 test (the fetch then reads triangle `first`)
  Bytes *base = !at_leaf                            ? (Bytes *)(bvh.nodes4 + t.cur)
                : test || bvh.tri_filter == nullptr ? (Bytes *)(reinterpret_cast<const TriRec *>(bvh.prims) + p)
                                                    : (Bytes *)(bvh.tri_filter + first);
  const bool record = test || (at_leaf && bvh.tri_filter == nullptr);
  // node lanes read the near row of each axis into chunk a and the far row into chunk 3 + a (see tri_step)
  const uint32_t sign = at_leaf ? 0u : q.b.sign;
  const uint32_t n0 = (sign & 1u) * 48u, n1 = ((sign >> 1) & 1u) * 48u, n2 = ((sign >> 2) & 1u) * 48u;
  u32x4 c0, c1, c2, c3, c4, c5, c6, c7;
  c0 = *(GlobalChunk *)(base + n0);
  c1 = *(GlobalChunk *)(base + n1 + 16);
  c2 = *(GlobalChunk *)(base + n2 + 32);
  c3 = *(GlobalChunk *)(base + (48u - n0));
  c4 = *(GlobalChunk *)(base + (64u - n1));
  if (!record) {  // a triangle record ends with chunk 4
    c5 = *(GlobalChunk *)(base + (80u - n2));
    c6 = *(GlobalChunk *)(base + 96);
    c7 = *(GlobalChunk *)(base + 112);
  }
  asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3), "+v"(c4), "+v"(c5), "+v"(c6), "+v"(c7));
  if (!at_leaf) {
    float k[4];
    uint32_t rf[4], cn[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float a0 = __builtin_fmaf(__uint_as_float(c0[c]), q.b.inv[0], q.b.offn[0]);
      const float a1 = __builtin_fmaf(__uint_as_float(c1[c]), q.b.inv[1], q.b.offn[1]);
      const float a2 = __builtin_fmaf(__uint_as_float(c2[c]), q.b.inv[2], q.b.offn[2]);
      const float f0 = __builtin_fmaf(__uint_as_float(c3[c]), q.b.inv[0], q.b.offf[0]);
      const float f1 = __builtin_fmaf(__uint_as_float(c4[c]), q.b.inv[1], q.b.offf[1]);
      const float f2 = __builtin_fmaf(__uint_as_float(c5[c]), q.b.inv[2], q.b.offf[2]);
      const float A = max_nn(max3_nn(a0, a1, a2), q.b.tmin);
      const float M = min_nn(min3_nn(f0, f1, f2), t.h32);
      k[c] = (c7[c] != EMPTY_SLOT && A <= M) ? A : __builtin_inff();
      rf[c] = c6[c];
      cn[c] = c7[c];
    }
    sort4(k, rf, cn);
    const float INF = __builtin_inff();
    const int n = (k[0] < INF ? 1 : 0) + (k[1] < INF ? 1 : 0) + (k[2] < INF ? 1 : 0) + (k[3] < INF ? 1 : 0);
    if (n) {
      st.room(n - 1);
      if (n > 1) st.put(st.sp + n - 2, rf[1], cn[1]);
      if (n > 2) st.put(st.sp + n - 3, rf[2], cn[2]);
      if (n > 3) st.put(st.sp, rf[3], cn[3]);
      st.sp += n - 1;
      t.cur = rf[0];
      t.cnt = cn[0];
      return;
    }
  } else if (!test) {
    bool p0 = true, p1 = true;
    if (bvh.tri_filter != nullptr) {
      TriFilt g[2];
      u32x4 raw[8] = {c0, c1, c2, c3, c4, c5, c6, c7};
      __builtin_memcpy(g, raw, sizeof g);
      p0 = tri_filter(g[0], q.D, q.O, q.b.om, q.b.tmin, t.h32);
      p1 = tri_filter(g[1], q.D, q.O, q.b.om, q.b.tmin, t.h32);
    }
    t.cand = (p0 ? 1u : 0u) | (p1 && t.cnt > 1u ? 2u : 0u);
    if (t.cand) return;
    if (t.cnt > 2u) {
      t.cnt -= 2u;
      t.cur += 2u;
      return;
    }
  } else {
    TriRec rec;
    u32x4 raw[5] = {c0, c1, c2, c3, c4};
    __builtin_memcpy(&rec, raw, sizeof rec);
    if (isect_tri(rec, r, s, p)) {
      t.active = false;
      return;
    }
    t.cand &= t.cand - 1u;
    if (t.cand) return;
    if (t.cnt > 2u) {
      t.cnt -= 2u;
      t.cur += 2u;
      return;
    }
  }
  if (st.sp > st.bot) {
    const WideEntry e = st.pop();
    t.cur = e.ref;
    t.cnt = e.key;
    return;
  }
  t.active = false;
}

template <bool FIXED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BRT_WAVES_PER_EU)))
k_trace_any(BvhView bvh, RaysView rays, HitsView hits, uint64_t n, uint32_t flags, uint32_t first, double S,
            unsigned long long *group, uint32_t refill, const uint32_t *order, uint32_t ring, uint32_t chunk,
            uint32_t fixed) {
  extern __shared__ unsigned char smem[];
  __shared__ AnyShare shares[4];
  constexpr int RW = (int)(sizeof(RaysView) / 8), HW = (int)(sizeof(HitsView) / 8);
  __shared__ uint64_t views[RW + HW];  // ray and hit columns, read back where they are used (see k_trace_persistent)
  if (threadIdx.x == 0) {
    lds_store(views, rays);
    lds_store(views + RW, hits);
  }
  __syncthreads();
  const uint32_t lane = __lane_id(), wave = threadIdx.x / 64;
  BRT_LDS volatile AnyShare *sh = (BRT_LDS volatile AnyShare *)&shares[wave];
  uint64_t spill[WIDE_SPILL];
  WideStack st;
  st.ring = (BRT_LDS uint32_t *)smem + (size_t)wave * ring * 128 + lane;
  st.spill = spill;
  st.mask = (int)ring - 1;
  st.reset();
  Ray r;
  AnyRay q;
  Hit s;
  AnyTrav t;
  t.active = false;
  t.cand = 0;
  bool has_ray = false, shared = false;
  bool done = false;              // a traced ray, still to be written
  bool exhausted = false;         // wave-uniform
  uint32_t pos = 0, pos_end = 0;  // shared rays: this part's positions in the visiting order
  uint32_t slot = 0, slots = 0;   // the share slot of this lane's ray; slots given out (wave-uniform)
  uint64_t idx = 0;
  unsigned long long mask = 0;  // see k_trace_tri
  const auto write_rays = [&]() {  // finished rays are written together (see k_trace_tri)
    if (done) {
      done = false;
      finish_ray<TriRec>(bvh, lds_fresh<HitsView>(views + RW), idx, r, s, flags, first, 1u);
    }
  };
  WavePool pool;
  const uint64_t global_wave = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave, range = global_wave * fixed;
  if constexpr (FIXED) pool.take_fixed(range, fixed, n);
  uint32_t turn = 0;
  bool noted = false;  // see note_passed
  for (;;) {
    if (!exhausted) {
      const unsigned long long idle = __ballot(!has_ray);
      const uint32_t nidle = (uint32_t)__popcll(idle);
      if (nidle >= refill || nidle == 64u) {
        write_rays();
        bool got;
        uint64_t cand = 0;
        pool_refill(pool, group + COUNTER_POOL, n, chunk, idle, nidle, lane, got, cand, exhausted);
        bool defer = false;
        if (got) {
          idx = order ? (uint64_t)order[cand] : cand;
          const RaysView V = lds_fresh<RaysView>(views);
          start_ray<true>(bvh, V, idx, S, r, q.b, s);
          if (deferred_to_exact(r)) {
            defer = true;
          } else {
            has_ray = true;
            Trav b;
            trav_begin<true>(bvh, r, q.b, s, b);
            t = AnyTrav{b.cur, b.cnt, 0u, b.h32, b.active};
#pragma unroll
            for (int k = 0; k < 3; k++) {
              q.D[k] = (float)r.d[k];
              q.O[k] = (float)r.o[k];
            }
            st.reset();
          }
        }
        if constexpr (FIXED) mask_add(mask, defer, (uint32_t)(cand - range));
        else noted = noted || __ballot(defer) != 0ull;
      }
    }
    const unsigned long long busy = __ballot(has_ray);
    if (exhausted) {
      if (!busy) {
        write_rays();
        if (FIXED && lane == 0) group[COUNTER_CLEARED + global_wave] = mask;
        if constexpr (!FIXED) note_passed(noted, group, lane);
        break;
      }
      // a part hands on the last eighth of its positions, so it needs eight for the order to stay strict
      const unsigned long long can = __ballot(has_ray && st.sp > st.bot && (!shared || pos_end - pos >= 8u));
      const uint32_t nidle = 64u - (uint32_t)__popcll(busy);
      if (nidle >= SHARE_MIN_IDLE && can && (++turn & 1u) == 0u) {
        write_rays();  // the helpers' state is overwritten
        const unsigned long long below = (1ull << lane) - 1ull;
        const uint32_t ncan = (uint32_t)__popcll(can), k = nidle < ncan ? nidle : ncan;
        const bool able = ((can >> lane) & 1ull) != 0ull;
        const uint32_t rank = (uint32_t)__popcll((has_ray ? can : ~busy) & below);
        const bool donor = able && rank < k, helper = !has_ray && rank < k;
        const uint32_t pos_end0 = shared ? pos_end : 0xffffffffu;
        // the r-th helper takes from the r-th donor, whose lane number lane r receives
        const unsigned long long fresh = __ballot(donor && !shared);
        uint64_t e = 0;
        if (donor) {
          e = st.take_bottom();
          if (!shared) {
            shared = true;
            slot = slots + (uint32_t)__popcll(fresh & below);
            sh->parts[slot] = 1u;
            sh->prim[slot] = INVALID_ID;
            sh->h[slot] = r.tmax;
            sh->first[slot] = 0xffffffffu;
            pos = 0u;
            pos_end = 0xffffffffu;
          }
          pos_end -= (pos_end - pos) >> 3;
        }
        slots += (uint32_t)__popcll(fresh);
        wave_fence();
        if (donor) atomicAdd(&shares[wave].parts[slot], 1u);
        // (at most 32 donors: lane 63 takes what the others push)
        const uint32_t by_rank = (uint32_t)__builtin_amdgcn_ds_permute((donor ? (int)rank : 63) << 2, (int)lane);
        const uint32_t from = lane_get(by_rank, (int)rank);  // with all lanes: a permute reads active lanes only
        const int src = helper ? (int)from : (int)lane;
        lane_take(e, src, helper);
        lane_take(r.o, src, helper);
        lane_take(r.d, src, helper);
        lane_take(r.tmin, src, helper);
        lane_take(r.tmax, src, helper);
        lane_take(q, src, helper);
        lane_take(s.h, src, helper);
        lane_take(t.h32, src, helper);
        lane_take(idx, src, helper);
        lane_take(slot, src, helper);
        {
          const uint32_t from_end = lane_get(pos_end, src), old_end = lane_get(pos_end0, src);
          pos = helper ? from_end : pos;
          pos_end = helper ? old_end : pos_end;
        }
        if (helper) {
          has_ray = true;
          shared = true;
          s.leaf_idx = INVALID_ID;
          t.cur = (uint32_t)e;
          t.cnt = (uint32_t)(e >> 32);
          t.cand = 0;
          t.active = true;
          st.reset();
        }
        wave_fence();
      }
    }
    if (has_ray && t.active) {
      if (shared && sh->first[slot] < pos) {  // behind a hit
        t.active = false;
      } else {
        any_step(bvh, r, q, s, t, st);
        if (shared && s.leaf_idx != INVALID_ID) atomicMin(&shares[wave].first[slot], pos);
      }
    }
    bool fin = has_ray && !t.active;
    if (exhausted) {
      // the parts of a shared ray are merged one lane at a time; the last one writes the ray
      unsigned long long m = __ballot(fin && shared);
      while (m) {
        const uint32_t l = (uint32_t)__ffsll((long long)m) - 1u;
        m &= m - 1ull;
        if (lane == l) {
          const uint32_t parts = sh->parts[slot] - 1u;
          sh->parts[slot] = parts;
          if (s.leaf_idx != INVALID_ID && sh->first[slot] == pos) {
            sh->h[slot] = s.h;
            sh->u[slot] = s.u;
            sh->v[slot] = s.v;
            sh->prim[slot] = s.leaf_idx;
          }
          has_ray = false;
          shared = false;
          if (parts == 0u) {
            s.h = sh->h[slot];
            s.u = sh->u[slot];
            s.v = sh->v[slot];
            s.leaf_idx = sh->prim[slot];
          } else {
            fin = false;
          }
        }
        wave_fence();
      }
    }
    done = done || fin;
    if (fin) has_ray = false;
  }
}

// Split-precision pre-test records of the triangles in leaf order (TriFilt), from their FP64 records; the FILTER_PAD
// records after the last one are zero.
__global__ void k_tri_filter_records(const TriRec *__restrict__ recs, uint32_t n, TriFilt *out, uint32_t total) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    TriFilt f{};
    if (i < n) {
      const TriRec &T = recs[i];
      double nn[3];
      tri_normal(T.e1, T.e2, nn);  // the FP64 test's n, operation for operation
      double vm = 0.0, sa = 0.0, sb = 0.0;
      for (int k = 0; k < 3; k++) {
        f.v0[k] = (float)T.v0[k];
        f.e1[k] = (float)T.e1[k];
        f.e2[k] = (float)T.e2[k];
        f.n[k] = (float)nn[k];
        vm = fmax(vm, fabs(T.v0[k]));
        sa += fabs(T.e1[k]);
        sb += fabs(T.e2[k]);
      }
      // upper bounds (the FP64 sums and products of non-negative terms are within a few ulps of exact)
      const double up = 1.0 + 0x1p-48, u = 0x1p-24;
      f.vmax = f32_up(vm * up);
      f.ed = f32_up((10.0 * u * sa * sb + 1e-29) * up);
      f.kw = f32_up(1.2 * 16.0 * u * (sa + sb) * up);
      f.cw = f32_up((1.3 * (double)f.ed + 9e-16) * up);  // 9e-16: 4 DBL_EPSILON rounded up
    }
    out[i] = f;
  }
}

// Split-precision pre-test records of the spheres in leaf order (SphFilt): the center rounded to nearest and |r|
// rounded up; the SPH_FILTER_PAD records after the last one are zero.
__global__ void k_sph_filter_records(const SphRec *__restrict__ recs, uint32_t n, SphFilt *out, uint32_t total) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    SphFilt f{};
    if (i < n) {
      const SphRec &S = recs[i];
      for (int k = 0; k < 3; k++) f.c[k] = (float)S.c[k];
      f.r = f32_up(fabs(S.r));
    }
    out[i] = f;
  }
}

// Pre-test records of the cylinders (cyl_filter). The cylinder test (cylinder.h:181-495) accepts any hit at t >= 0, with no
// distance check, at a point of the local frame org + t dir = R^T (o + t d - c) with |z| <= h/2 and, up to the rounding of
// the test, on or inside the elliptic shell of semi-axes a, b; for an orthonormal R that point lies within
// sqrt(max(a,b)^2 + (h/2)^2) of c. Both radii are enlarged by 2^-10 of themselves, the sphere's also by 2^-20 of the
// coordinate magnitude, far above any rounding of the FP64 test, and are infinite (never reject) when R R^T differs from
// the identity by more than 1e-6 or an input is not finite; so is a semi-axis whose square leaves the FP32 range.
__global__ void k_cyl_filter_records(const CylRec *__restrict__ recs, uint32_t n, CylFilt *out, uint32_t total) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    CylFilt f{};
    if (i < n) {
      const CylRec &C = recs[i];
      double dev = 0.0;
      for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) {
          const double d = C.R[3 * a] * C.R[3 * b] + C.R[3 * a + 1] * C.R[3 * b + 1] + C.R[3 * a + 2] * C.R[3 * b + 2];
          dev = fmax(dev, fabs(d - (a == b ? 1.0 : 0.0)));
        }
      const double ab = fmax(fabs(C.a), fabs(C.b)), hh = 0.5 * fabs(C.h);
      const double rb = sqrt(ab * ab + hh * hh);
      const double cm = fmax(fabs(C.c[0]), fmax(fabs(C.c[1]), fabs(C.c[2])));
      double rad = rb * (1.0 + 0x1p-10) + 0x1p-20 * (cm + rb);
      double shell = ab * (1.0 + 0x1p-10);
      if (!(dev <= 1e-6) || !(rad < 1e300)) rad = shell = __builtin_inf();
      if (shell < 1e-15) shell = __builtin_inf();
      for (int k = 0; k < 3; k++) {  // first column of R x second
        const int x = (k + 1) % 3, y = (k + 2) % 3;
        f.axis[k] = (float)(C.R[3 * x] * C.R[3 * y + 1] - C.R[3 * y] * C.R[3 * x + 1]);
      }
      for (int k = 0; k < 3; k++) f.c[k] = (float)C.c[k];
      f.r = f32_up(rad);
      f.shell = f32_up(shell);
    }
    out[i] = f;
  }
}

__global__ void k_nodeq_records(const Node4 *__restrict__ in, const uint32_t *__restrict__ ord, uint32_t n,
                                NodeQ *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Node4 a = in[i];
  NodeQ b;
  for (int c = 0; c < 4; c++) {
    for (int k = 0; k < 3; k++) {
      b.lo[k][c] = a.lo[k][c];
      b.hi[k][c] = a.hi[k][c];
    }
    b.ref[c] = a.ref[c];
    b.cnt[c] = a.cnt[c] == EMPTY_SLOT ? 0 : (uint8_t)a.cnt[c];
  }
  b.ord[0] = ord[2ull * i];
  b.ord[1] = ord[2ull * i + 1];
  b.pad = 0;
  out[i] = b;
}

// The boxes of the leaves, each at its first primitive's place (six values). A root leaf's box is the tree's.
template <class Node, class R>
__global__ void k_leaf_boxes(const Node *__restrict__ nodes, uint32_t n, BvhView bvh, R *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0 && n == 0)
    for (int k = 0; k < 3; k++) {
      out[k] = (R)bvh.root_min[k];
      out[3 + k] = (R)bvh.root_max[k];
    }
  if (i >= n) return;
  for (int c = 0; c < 2; c++)
    if (nodes[i].ref[c] & LEAF_BIT)
      for (int k = 0; k < 6; k++) out[6ull * (nodes[i].ref[c] & ~LEAF_BIT) + k] = nodes[i].b[6 * c + k];
}

// Clears a launch's counter group (a fill kernel, not hipMemsetAsync, so that graph captures replay correctly).
__global__ void k_zero_counters(unsigned long long *c) {
  for (uint32_t k = threadIdx.x; k < (uint32_t)COUNTER_CLEARED; k += blockDim.x) c[k] = 0ull;
}

// 3 x 9-bit Morton interleave
__device__ __forceinline__ uint32_t spread9(uint32_t x) {
  x &= 0x1ffu;
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

// Sort key of ray i: direction octant (3 bits, the children visit order depends only on it) above a 27-bit Morton
// code of the origin quantised in the scene box (mode 1), or the Morton code alone (mode 2).
__global__ void k_sort_keys(RaysView rays, uint64_t n, double lx, double ly, double lz, double sx, double sy,
                            double sz, uint32_t mode, uint32_t *keys, uint32_t *vals) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double q[3] = {(rays.ox[i] - lx) * sx, (rays.oy[i] - ly) * sy, (rays.oz[i] - lz) * sz};
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double c = q[k] != q[k] ? 0.0 : fmin(fmax(q[k], 0.0), 511.0);
      m |= spread9((uint32_t)c) << k;
    }
    uint32_t oct = (rays.dx[i] < 0.0 ? 1u : 0u) | (rays.dy[i] < 0.0 ? 2u : 0u) | (rays.dz[i] < 0.0 ? 4u : 0u);
    keys[i] = mode == 1u ? ((oct << 27) | m) : m;
    vals[i] = (uint32_t)i;
  }
}

template <class R>
__global__ void k_init_hits(HitsViewT<R> hits, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    hits.t[i] = Real<R>::max;
    if (hits.u) hits.u[i] = R(0);
    if (hits.v) hits.v[i] = R(0);
    hits.prim_id[i] = INVALID_ID;
    if (hits.geom_id) hits.geom_id[i] = INVALID_ID;
    if (hits.nx) {
      hits.nx[i] = R(0);
      hits.ny[i] = R(0);
      hits.nz[i] = R(0);
    }
  }
}

// (n, 3) rows to three columns of n. Memory bound: the rows are read once (the second and third loads of a wave hit the
// lines of the first) and each column written in whole lines.
constexpr uint32_t ROWS_PER_THREAD = 4;
template <class T>
__global__ void __launch_bounds__(256) k_rows_to_columns(const T *__restrict__ rows, uint64_t n, T *__restrict__ x,
                                                         T *__restrict__ y, T *__restrict__ z) {
  const uint64_t i0 = (uint64_t)blockIdx.x * (256u * ROWS_PER_THREAD) + threadIdx.x;
  T r[ROWS_PER_THREAD][3];
#pragma unroll
  for (uint32_t k = 0; k < ROWS_PER_THREAD; k++) {
    const uint64_t i = i0 + k * 256u;
    if (i < n)
      for (int a = 0; a < 3; a++) r[k][a] = rows[3 * i + a];
  }
#pragma unroll
  for (uint32_t k = 0; k < ROWS_PER_THREAD; k++) {
    const uint64_t i = i0 + k * 256u;
    if (i < n) {
      x[i] = r[k][0];
      y[i] = r[k][1];
      z[i] = r[k][2];
    }
  }
}

// Blocks of a persistent launch: as many as fit on the device at once, but no more than the rays need.
template <class K>
hipError_t persistent_blocks(K kernel, uint32_t block, size_t lds, uint64_t n, uint64_t &blocks) {
  int dev = 0, cus = 0, per_cu = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)kernel, (int)block, lds);
  if (e != hipSuccess) return e;
  blocks = (uint64_t)cus * (uint64_t)(per_cu > 0 ? per_cu : 1);
  const uint64_t need = (n + block - 1) / block;
  if (blocks > need) blocks = need;
  return hipSuccess;
}

// The FP64 launch over the rays a split-precision launch deferred (default launch shape of the exact path).
template <class Rec>
hipError_t launch_deferred(const BvhView &bvh, const RaysViewT<typename Rec::real> &rays,
                           const HitsViewT<typename Rec::real> &hits, uint64_t n, const TraceLaunch &cfg,
                           const SplitParams &sp, uint32_t is_tri, hipStream_t stream) {
  using R = typename Rec::real;
  const uint32_t ring64 = ring_default<Rec, false>();
  const size_t lds64 = ring_lds_bytes<false, R>(256, ring64);
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_persistent<Rec, false>, 256, lds64, n, blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_trace_persistent<Rec, false>), dim3((uint32_t)blocks), dim3(256), lds64, stream, bvh, rays,
                     hits, n, cfg.flags | FLAG_DEFERRED_ONLY, cfg.first ? 1u : 0u, is_tri, sp.scene_extent,
                     cfg.counter + COUNTER_DEFERRED_POOL, refill_default<Rec, false>(), cfg.order, ring64,
                     cfg.counter + COUNTER_DEFERRED, POOL_CHUNK);
  return hipGetLastError();
}

// The exact launch over the rays that a launch of `fixed` rays per wave left.
template <class Rec>
hipError_t launch_left(const BvhView &bvh, const RaysViewT<typename Rec::real> &rays,
                       const HitsViewT<typename Rec::real> &hits, uint64_t n, const TraceLaunch &cfg, const SplitParams &sp,
                       uint32_t is_tri, uint32_t fixed, hipStream_t stream) {
  const uint32_t ring = ring_default<Rec, false>();
  hipLaunchKernelGGL((k_trace<Rec, false>), dim3((uint32_t)((n + 255) / 256)), dim3(256),
                     (ring_lds_bytes<false, typename Rec::real>(256, ring)), stream, bvh, rays, hits, n, cfg.flags,
                     cfg.first ? 1u : 0u, is_tri, sp.scene_extent, cfg.order, ring, cfg.counter + COUNTER_DEFERRED,
                     cfg.counter + COUNTER_CLEARED, fixed);
  return hipGetLastError();
}

// Enqueues one traversal of a geometry type: the counter group is cleared, then the trace kernel runs. A split-
// precision launch is followed by the FP64 launch over the rays it deferred (deferred_to_exact), which returns at
// once when there are none; both run in stream order before the next geometry type, so intersect1's merge order
// holds for the deferred rays too.
template <class Rec, bool SPLIT>
hipError_t launch_kernel(const BvhView &bvh, const RaysViewT<typename Rec::real> &rays,
                         const HitsViewT<typename Rec::real> &hits, uint64_t n, const TraceLaunch &cfg,
                         const SplitParams &sp, uint32_t is_tri, hipStream_t stream) {
  using R = typename Rec::real;
  const uint32_t block = cfg.block ? cfg.block : block_default<Rec, SPLIT>();
  const uint32_t first = cfg.first ? 1u : 0u;
  const uint32_t ring = cfg.ring ? cfg.ring : ring_default<Rec, SPLIT>();
  const size_t lds = ring_lds_bytes<SPLIT, R>(block, ring);
  unsigned long long *grp = cfg.counter;
  if (!grp) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  if (cfg.schedule == SCHEDULE_PERSISTENT) {
    uint64_t blocks = 0;
    hipError_t e = persistent_blocks(k_trace_persistent<Rec, SPLIT>, block, lds, n, blocks);
    if (e != hipSuccess) return e;
    const uint32_t refill = cfg.refill ? cfg.refill : refill_default<Rec, SPLIT>();
    hipLaunchKernelGGL((k_trace_persistent<Rec, SPLIT>), dim3((uint32_t)blocks), dim3(block), lds, stream, bvh, rays,
                       hits, n, cfg.flags, first, is_tri, sp.scene_extent, grp + COUNTER_POOL, refill, cfg.order,
                       ring, grp + COUNTER_DEFERRED, cfg.pool ? cfg.pool : POOL_CHUNK);
  } else {
    uint64_t blocks = (n + block - 1) / block;
    if (blocks > (1ull << 30)) blocks = 1ull << 30;
    hipLaunchKernelGGL((k_trace<Rec, SPLIT>), dim3((uint32_t)blocks), dim3(block), lds, stream, bvh, rays, hits, n,
                       cfg.flags, first, is_tri, sp.scene_extent, cfg.order, ring, grp + COUNTER_DEFERRED,
                       (const unsigned long long *)nullptr, 1u);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !SPLIT) return e;
  return launch_deferred<Rec>(bvh, rays, hits, n, cfg, sp, is_tri, stream);
}

// The fast triangle traversal (k_trace_tri) takes closest-hit launches on the persistent schedule, in either precision:
// 1.31M-triangle mesh, 4,194,304 incoherent rays 3.03 ms, against 5.6-5.8 ms for the exact FP64 kernel and 3.8 ms for
// nearest-first split precision; a 1920x1080 camera with normals 2.24 against 3.57 ms. Any-hit launches return the first
// hit of their own visiting order; the one-ray-per-thread schedule keeps its kernel.
bool fast_triangles(const TraceLaunch &cfg) {
  return cfg.schedule == SCHEDULE_PERSISTENT && !(cfg.flags & FLAG_ANY_HIT);
}
// Spheres' and cylinders' (k_trace_wide), in FP64 (split precision has a visiting order of its own): 8,388,608 incoherent
// rays, 50,000 spheres 3.3 against 4.44 ms, 10,000 cylinders 3.30 against 5.45 ms; a 512x512 camera over 1,024 spheres 0.091
// against 0.137 ms a call. 100 planes 1.75 against 1.61 ms: they keep the exact kernel. In a Scene<float>, incoherent rays:
// 1,000,003 on 327,680 triangles 0.63 against 0.83 ms, on 50,000 spheres 0.45 against 0.48, 2,000 on 81,920 triangles 0.089
// against 0.192; 1920x1080 camera rays on 1.31M triangles 2.05 against 2.62 ms.
bool fast_wide(const BvhView &bvh, const TraceLaunch &cfg) {
  return bvh.nodesq && bvh.leaf_boxes && cfg.precision == PREC_FP64 && fast_triangles(cfg);
}
// Any hit of triangles in split precision on the persistent schedule takes k_trace_any (figures there). In FP64 the hit that
// counts is the first one accepted in the reference's order, and k_trace_any takes parts of a ray in any order: the exact
// kernel. (The first certified hit of k_trace_tri would be that hit too; no such launch has been built.)
bool fast_any(const TraceLaunch &cfg) {
  return cfg.schedule == SCHEDULE_PERSISTENT && cfg.precision != PREC_FP64 && (cfg.flags & FLAG_ANY_HIT);
}
constexpr uint32_t TRI_RING = 16, TRI_REFILL = 16, ANY_REFILL = 32;
constexpr size_t tri_lds_bytes(uint32_t block, uint32_t ring) { return (size_t)block * ring * sizeof(uint64_t); }

hipError_t launch_tri(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n,
                      const TraceLaunch &cfg, const SplitParams &sp, hipStream_t stream) {
  const uint32_t block = cfg.block ? cfg.block : 256;
  const uint32_t ring = cfg.ring ? cfg.ring : TRI_RING;
  const uint32_t first = cfg.first ? 1u : 0u;
  const uint32_t flags = cfg.flags | (cfg.precision != PREC_FP64 ? FLAG_SPLIT : 0u);
  const size_t lds = tri_lds_bytes(block, ring);
  unsigned long long *grp = cfg.counter;
  if (!grp) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_tri<false>, block, lds, n * 64, blocks);
  if (e != hipSuccess) return e;
  const uint32_t wpb = block / 64;
  uint32_t fixed = fixed_per_wave(n, blocks * wpb);
  if (blocks * wpb > (uint64_t)LIST_CAPACITY) fixed = 0;  // (a word per wave)
  if (!fixed) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  const uint64_t need = fixed ? (n + fixed * wpb - 1) / (fixed * wpb) : (n + block - 1) / block;
  if (blocks > need) blocks = need;
  hipLaunchKernelGGL((fixed ? k_trace_tri<false, false, true> : k_trace_tri<false>), dim3((uint32_t)blocks), dim3(block),
                     lds, stream, bvh, rays, hits,
                     (const BatchJob *)nullptr, 0u, n, flags, first, sp.scene_extent, grp,
                     cfg.refill ? cfg.refill : TRI_REFILL, cfg.order, ring, cfg.pool ? cfg.pool : POOL_CHUNK, fixed);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (fixed) return launch_left<TriRec>(bvh, rays, hits, n, cfg, sp, 1u, fixed, stream);
  // the rays it left to the exact kernel (default launch shape of the exact path)
  const uint32_t ring64 = ring_default<TriRec, false>();
  const size_t lds64 = ring_lds_bytes<false, double>(256, ring64);
  e = persistent_blocks(k_trace_persistent<TriRec, false, true>, 256, lds64, n, blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_trace_persistent<TriRec, false, true>), dim3((uint32_t)blocks), dim3(256), lds64, stream, bvh,
                     rays, hits, n, flags, first, 1u, sp.scene_extent, grp + COUNTER_DEFERRED_POOL,
                     refill_default<TriRec, false>(), cfg.order, ring64, grp + COUNTER_DEFERRED, POOL_CHUNK);
  return hipGetLastError();
}

template <class Rec>
hipError_t launch_wide(const BvhView &bvh, const RaysViewT<typename Rec::real> &rays,
                       const HitsViewT<typename Rec::real> &hits, uint64_t n, const TraceLaunch &cfg, const SplitParams &sp,
                       uint32_t is_tri, hipStream_t stream) {
  using R = typename Rec::real;
  const uint32_t block = cfg.block ? cfg.block : 256;
  const uint32_t ring = cfg.ring ? cfg.ring : TRI_RING;
  const uint32_t first = cfg.first ? 1u : 0u;
  const size_t lds = tri_lds_bytes(block, ring);
  unsigned long long *grp = cfg.counter;
  if (!grp) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_wide<Rec, false>, block, lds, n * 64, blocks);
  if (e != hipSuccess) return e;
  const uint32_t wpb = block / 64;
  uint32_t fixed = fixed_per_wave(n, blocks * wpb);
  if (blocks * wpb > (uint64_t)LIST_CAPACITY) fixed = 0;  // (a word per wave)
  if (!fixed) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  const uint64_t need = fixed ? (n + fixed * wpb - 1) / (fixed * wpb) : (n + block - 1) / block;
  if (blocks > need) blocks = need;
  hipLaunchKernelGGL((fixed ? k_trace_wide<Rec, true> : k_trace_wide<Rec, false>), dim3((uint32_t)blocks), dim3(block),
                     lds, stream, bvh, rays, hits, n, cfg.flags,
                     first, is_tri, sp.scene_extent, grp, cfg.refill ? cfg.refill : TRI_REFILL, cfg.order, ring,
                     cfg.pool ? cfg.pool : POOL_CHUNK, fixed);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (fixed) return launch_left<Rec>(bvh, rays, hits, n, cfg, sp, is_tri, fixed, stream);
  const uint32_t ring64 = ring_default<Rec, false>();
  const size_t lds64 = ring_lds_bytes<false, R>(256, ring64);
  e = persistent_blocks(k_trace_persistent<Rec, false, true>, 256, lds64, n, blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_trace_persistent<Rec, false, true>), dim3((uint32_t)blocks), dim3(256), lds64, stream, bvh, rays,
                     hits, n, cfg.flags, first, is_tri, sp.scene_extent, grp + COUNTER_DEFERRED_POOL,
                     refill_default<Rec, false>(), cfg.order, ring64, grp + COUNTER_DEFERRED, POOL_CHUNK);
  return hipGetLastError();
}

// Any hit of triangles in split precision (k_trace_any).
hipError_t launch_any(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n, const TraceLaunch &cfg,
                      const SplitParams &sp, hipStream_t stream) {
  const uint32_t block = cfg.block ? cfg.block : 256;
  const uint32_t ring = cfg.ring ? cfg.ring : TRI_RING;
  const size_t lds = tri_lds_bytes(block, ring);
  unsigned long long *grp = cfg.counter;
  if (!grp) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_any<false>, block, lds, n * 64, blocks);
  if (e != hipSuccess) return e;
  const uint32_t wpb = block / 64;
  uint32_t fixed = fixed_per_wave(n, blocks * wpb);
  if (blocks * wpb > (uint64_t)LIST_CAPACITY) fixed = 0;  // (a word per wave)
  if (!fixed) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  const uint64_t need = fixed ? (n + fixed * wpb - 1) / (fixed * wpb) : (n + block - 1) / block;
  if (blocks > need) blocks = need;
  hipLaunchKernelGGL((fixed ? k_trace_any<true> : k_trace_any<false>), dim3((uint32_t)blocks), dim3(block), lds, stream, bvh,
                     rays, hits, n, cfg.flags,
                     cfg.first ? 1u : 0u, sp.scene_extent, grp, cfg.refill ? cfg.refill : ANY_REFILL, cfg.order, ring,
                     cfg.pool ? cfg.pool : POOL_CHUNK, fixed);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (fixed) return launch_left<TriRec>(bvh, rays, hits, n, cfg, sp, 1u, fixed, stream);
  return launch_deferred<TriRec>(bvh, rays, hits, n, cfg, sp, 1u, stream);
}

hipError_t launch_tri_batch(const BatchJob *jobs, uint32_t njobs, uint64_t total, const TraceLaunch &cfg,
                            hipStream_t stream) {
  const uint32_t block = cfg.block ? cfg.block : 256;
  const uint32_t ring = cfg.ring ? cfg.ring : TRI_RING;
  const size_t lds = tri_lds_bytes(block, ring);
  const uint32_t flags = cfg.flags | (cfg.precision != PREC_FP64 ? FLAG_SPLIT : 0u);
  unsigned long long *grp = cfg.counter;
  if (!grp || njobs == 0) return hipErrorInvalidValue;
  if (total == 0) return hipSuccess;
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_tri<true>, block, lds, total * 64, blocks);
  if (e != hipSuccess) return e;
  const uint32_t wpb = block / 64, fixed = fixed_per_wave(total, blocks * wpb);
  const uint64_t need = fixed ? (total + fixed * wpb - 1) / (fixed * wpb) : (total + block - 1) / block;
  if (blocks > need) blocks = need;
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  hipLaunchKernelGGL(k_trace_tri<true>, dim3((uint32_t)blocks), dim3(block), lds, stream, BvhView{}, RaysView{},
                     HitsView{}, jobs, njobs, total, flags, 0u, 0.0, grp, cfg.refill ? cfg.refill : TRI_REFILL,
                     (const uint32_t *)nullptr, ring, cfg.pool ? cfg.pool : POOL_CHUNK, fixed);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  const uint32_t ring64 = ring_default<TriRec, false>();
  const size_t lds64 = ring_lds_bytes<false>(256, ring64);
  e = persistent_blocks(k_trace_batch<TriRec, false, true>, 256, lds64, total, blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_trace_batch<TriRec, false, true>), dim3((uint32_t)blocks), dim3(256), lds64, stream, jobs,
                     njobs, total, flags, grp + COUNTER_DEFERRED_POOL, refill_default<TriRec, false>(), ring64,
                     grp + COUNTER_DEFERRED, POOL_CHUNK);
  return hipGetLastError();
}

template <class Rec, bool SPLIT>
hipError_t launch_batch_kernel(const BatchJob *jobs, uint32_t njobs, uint64_t total, const TraceLaunch &cfg,
                               hipStream_t stream) {
  const uint32_t block = cfg.block ? cfg.block : 256;
  const uint32_t ring = cfg.ring ? cfg.ring : ring_default<Rec, SPLIT>();
  const size_t lds = ring_lds_bytes<SPLIT>(block, ring);
  unsigned long long *grp = cfg.counter;
  if (!grp || njobs == 0) return hipErrorInvalidValue;
  if (total == 0) return hipSuccess;
  uint64_t blocks = 0;
  hipError_t e = persistent_blocks(k_trace_batch<Rec, SPLIT>, block, lds, total, blocks);
  if (e != hipSuccess) return e;
  const uint32_t refill = cfg.refill ? cfg.refill : refill_default<Rec, SPLIT>();
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, grp);
  hipLaunchKernelGGL((k_trace_batch<Rec, SPLIT>), dim3((uint32_t)blocks), dim3(block), lds, stream, jobs, njobs, total,
                     cfg.flags, grp + COUNTER_POOL, refill, ring, grp + COUNTER_DEFERRED, cfg.pool ? cfg.pool : POOL_CHUNK);
  e = hipGetLastError();
  if (e != hipSuccess || !SPLIT) return e;
  const uint32_t ring64 = ring_default<Rec, false>();
  const size_t lds64 = ring_lds_bytes<false>(256, ring64);
  e = persistent_blocks(k_trace_batch<Rec, false>, 256, lds64, total, blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_trace_batch<Rec, false>), dim3((uint32_t)blocks), dim3(256), lds64, stream, jobs, njobs, total,
                     cfg.flags | FLAG_DEFERRED_ONLY, grp + COUNTER_DEFERRED_POOL, refill_default<Rec, false>(),
                     ring64, grp + COUNTER_DEFERRED, POOL_CHUNK);
  return hipGetLastError();
}

template <class Rec>
hipError_t launch_typed(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n,
                        const TraceLaunch &cfg, const SplitParams &sp, uint32_t is_tri, hipStream_t stream) {
  if (cfg.precision == PREC_FP64) return launch_kernel<Rec, false>(bvh, rays, hits, n, cfg, sp, is_tri, stream);
  return launch_kernel<Rec, true>(bvh, rays, hits, n, cfg, sp, is_tri, stream);
}

template <class Rec>
hipError_t launch_other(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n, const TraceLaunch &cfg,
                        const SplitParams &sp, hipStream_t stream) {
  const uint32_t ow = cfg.overwrite ? 1u : 0u;
  if (fast_wide(bvh, cfg)) return launch_wide<Rec>(bvh, rays, hits, n, cfg, sp, ow, stream);
  return launch_typed<Rec>(bvh, rays, hits, n, cfg, sp, ow, stream);
}

}  // namespace

hipError_t launch_trace(GeomType type, const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n,
                        const TraceLaunch &cfg, const SplitParams &split, hipStream_t stream) {
  switch (type) {
  case TRIANGLES:
    if (bvh.nodesq && fast_triangles(cfg)) return launch_tri(bvh, rays, hits, n, cfg, split, stream);
    if (fast_any(cfg)) return launch_any(bvh, rays, hits, n, cfg, split, stream);
    return launch_typed<TriRec>(bvh, rays, hits, n, cfg, split, 1u, stream);
  case SPHERES: return launch_other<SphRec>(bvh, rays, hits, n, cfg, split, stream);
  case PLANES: return launch_typed<PlaRec>(bvh, rays, hits, n, cfg, split, cfg.overwrite ? 1u : 0u, stream);
  default: return launch_other<CylRec>(bvh, rays, hits, n, cfg, split, stream);
  }
}

// The closest hit of one ray among the triangles, by a wave whose lanes share the ray's tree: the chain of dependent
// reads bounds it, which one lane alone follows through every node. `hits.merged` is required.
hipError_t launch_tri_lone(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint32_t flags,
                           const SplitParams &sp, hipStream_t stream) {
  hipLaunchKernelGGL((k_trace_tri<false, true>), dim3(1), dim3(64), tri_lds_bytes(64, TRI_RING), stream, bvh, rays, hits,
                     (const BatchJob *)nullptr, 0u, (uint64_t)1, flags, 0u, sp.scene_extent,
                     (unsigned long long *)nullptr, TRI_REFILL, (const uint32_t *)nullptr, TRI_RING, POOL_CHUNK, 1u);
  return hipGetLastError();
}

hipError_t launch_rows_to_columns(const void *rows, uint32_t elem_bytes, uint64_t n, void *columns, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint64_t blocks = (n + 256u * ROWS_PER_THREAD - 1) / (256u * ROWS_PER_THREAD);
  if (blocks > 0x7fffffffu) return hipErrorInvalidValue;
  const auto run = [&](auto zero) {
    using T = decltype(zero);
    T *c = static_cast<T *>(columns);
    hipLaunchKernelGGL(k_rows_to_columns<T>, dim3((uint32_t)blocks), dim3(256), 0, stream, static_cast<const T *>(rows), n,
                       c, c + n, c + 2 * n);
  };
  if (elem_bytes == 8) run(uint64_t{});
  else run(uint32_t{});
  return hipGetLastError();
}

hipError_t launch_sph_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream) {
  const uint32_t total = n + SPH_FILTER_PAD;
  uint32_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_sph_filter_records, dim3(blocks), dim3(256), 0, stream, static_cast<const SphRec *>(recs), n,
                     static_cast<SphFilt *>(out), total);
  return hipGetLastError();
}

hipError_t launch_cyl_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream) {
  const uint32_t total = n + SPH_FILTER_PAD;
  uint32_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_cyl_filter_records, dim3(blocks), dim3(256), 0, stream, static_cast<const CylRec *>(recs), n,
                     static_cast<CylFilt *>(out), total);
  return hipGetLastError();
}

hipError_t launch_zero_counters(unsigned long long *group, hipStream_t stream) {
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, group);
  return hipGetLastError();
}

hipError_t launch_leaf_boxes(const BvhView &bvh, bool f32, void *out, hipStream_t stream) {
  const uint32_t num_nodes = bvh.n_nodes;
  const dim3 grid(num_nodes / 256 + 1), block(256);
  if (f32)
    hipLaunchKernelGGL((k_leaf_boxes<Node32, float>), grid, block, 0, stream, bvh.nodes32, num_nodes, bvh,
                       static_cast<float *>(out));
  else
    hipLaunchKernelGGL((k_leaf_boxes<Node64, double>), grid, block, 0, stream, bvh.nodes64, num_nodes, bvh,
                       static_cast<double *>(out));
  return hipGetLastError();
}

hipError_t launch_nodeq_records(const Node4 *nodes4, const uint32_t *ord, uint32_t n, NodeQ *out, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_nodeq_records, dim3((n + 255) / 256), dim3(256), 0, stream, nodes4, ord, n, out);
  return hipGetLastError();
}

hipError_t launch_tri_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream) {
  const uint32_t total = n + FILTER_PAD;
  uint32_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_tri_filter_records, dim3(blocks), dim3(256), 0, stream, static_cast<const TriRec *>(recs), n,
                     static_cast<TriFilt *>(out), total);
  return hipGetLastError();
}

hipError_t sort_workspace_reserve(SortWorkspace &ws, uint64_t n) {
  if (n > 0x7fffffffull) return hipErrorInvalidValue;
  if (ws.capacity >= n && ws.base) return hipSuccess;
  size_t temp = 0;
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, temp, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                                    (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)n, 0, 30);
  if (e != hipSuccess) return e;
  if (ws.base) {
    e = hipFree(ws.base);
    ws.base = nullptr;
    ws.capacity = 0;
    if (e != hipSuccess) return e;
  }
  const size_t arr = ((size_t)n * 4 + 255) & ~(size_t)255;
  void *p = nullptr;
  e = hipMalloc(&p, 4 * arr + temp);
  if (e != hipSuccess) return e;
  unsigned char *b = static_cast<unsigned char *>(p);
  ws.base = p;
  ws.keys_in = reinterpret_cast<uint32_t *>(b);
  ws.keys_out = reinterpret_cast<uint32_t *>(b + arr);
  ws.vals_in = reinterpret_cast<uint32_t *>(b + 2 * arr);
  ws.vals_out = reinterpret_cast<uint32_t *>(b + 3 * arr);
  ws.temp = b + 4 * arr;
  ws.temp_bytes = temp;
  ws.capacity = n;
  return hipSuccess;
}

hipError_t sort_workspace_in(SortWorkspace &ws, void *base, size_t bytes, uint64_t n) {
  if (n > 0x7fffffffull) return hipErrorInvalidValue;
  size_t temp = 0;
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, temp, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                                    (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)n, 0, 30);
  if (e != hipSuccess) return e;
  const size_t arr = ((size_t)n * 4 + 255) & ~(size_t)255;
  if (4 * arr + temp > bytes) return hipErrorInvalidValue;
  unsigned char *b = static_cast<unsigned char *>(base);
  ws.base = nullptr;  // not owned
  ws.keys_in = reinterpret_cast<uint32_t *>(b);
  ws.keys_out = reinterpret_cast<uint32_t *>(b + arr);
  ws.vals_in = reinterpret_cast<uint32_t *>(b + 2 * arr);
  ws.vals_out = reinterpret_cast<uint32_t *>(b + 3 * arr);
  ws.temp = b + 4 * arr;
  ws.temp_bytes = temp;
  ws.capacity = n;
  return hipSuccess;
}

hipError_t sort_rays(const RaysView &rays, uint64_t n, const double lo[3], const double hi[3], uint32_t mode,
                     SortWorkspace &ws, hipStream_t stream, const uint32_t **order) {
  *order = nullptr;
  if (n == 0) return hipSuccess;
  if (ws.capacity < n) return hipErrorInvalidValue;
  double sc[3];
  for (int k = 0; k < 3; k++) {
    const double ext = hi[k] - lo[k];
    sc[k] = (ext > 0.0 && ext == ext) ? 512.0 / ext : 0.0;
  }
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_sort_keys, dim3((uint32_t)blocks), dim3(256), 0, stream, rays, n, lo[0], lo[1], lo[2], sc[0],
                     sc[1], sc[2], mode, ws.keys_in, ws.vals_in);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  size_t temp = ws.temp_bytes;
  e = hipcub::DeviceRadixSort::SortPairs(ws.temp, temp, ws.keys_in, ws.keys_out, ws.vals_in, ws.vals_out, (int)n, 0,
                                         30, stream);
  if (e != hipSuccess) return e;
  *order = ws.vals_out;
  return hipSuccess;
}

hipError_t launch_trace_batch(GeomType type, const BatchJob *jobs, uint32_t njobs, uint64_t total,
                              const TraceLaunch &cfg, hipStream_t stream) {
  const bool split = cfg.precision != PREC_FP64;
  switch (type) {
  case TRIANGLES:
    if (cfg.fast && fast_triangles(cfg)) return launch_tri_batch(jobs, njobs, total, cfg, stream);
    return split ? launch_batch_kernel<TriRec, true>(jobs, njobs, total, cfg, stream)
                 : launch_batch_kernel<TriRec, false>(jobs, njobs, total, cfg, stream);
  case SPHERES:
    return split ? launch_batch_kernel<SphRec, true>(jobs, njobs, total, cfg, stream)
                 : launch_batch_kernel<SphRec, false>(jobs, njobs, total, cfg, stream);
  case PLANES:
    return split ? launch_batch_kernel<PlaRec, true>(jobs, njobs, total, cfg, stream)
                 : launch_batch_kernel<PlaRec, false>(jobs, njobs, total, cfg, stream);
  default:
    return split ? launch_batch_kernel<CylRec, true>(jobs, njobs, total, cfg, stream)
                 : launch_batch_kernel<CylRec, false>(jobs, njobs, total, cfg, stream);
  }
}

template <class R>
hipError_t init_hits(const HitsViewT<R> &hits, uint64_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > (1ull << 30)) blocks = 1ull << 30;
  hipLaunchKernelGGL(k_init_hits<R>, dim3((uint32_t)blocks), dim3(256), 0, stream, hits, n);
  return hipGetLastError();
}
hipError_t launch_init_hits(const HitsView &hits, uint64_t n, hipStream_t stream) { return init_hits(hits, n, stream); }
hipError_t launch_init_hits_f32(const HitsViewF &hits, uint64_t n, hipStream_t stream) {
  return init_hits(hits, n, stream);
}

// Scratch memory of brt_intersect_noalloc, for callers that cannot allocate (graph capture, serving loops): each
// GPU that loads this library holds one copy until the process ends. Host code never passes the array's name to a
// kernel (on the host it is only a stand-in for the symbol); it uses the device address from noalloc_scratch.
__device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

hipError_t noalloc_scratch(unsigned char **ptr) {
  constexpr int MAX_DEVICES = 64;
  static std::mutex mu;
  static unsigned char *addr[MAX_DEVICES] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(mu);
  if (!addr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[dev] = static_cast<unsigned char *>(p);
  }
  *ptr = addr[dev];
  return hipSuccess;
}

// Scene<float>: the exact path in FP32 (no split precision: the scene type is already FP32).
hipError_t launch_trace_f32(GeomType type, const BvhView &bvh, const RaysViewF &rays, const HitsViewF &hits,
                            uint64_t n, const TraceLaunch &cfg, double extent, hipStream_t stream) {
  const SplitParams sp{extent};
  const uint32_t ow = cfg.overwrite ? 1u : 0u;
  const auto run = [&](auto rec, uint32_t is_tri) {
    using Rec = decltype(rec);
    if (fast_wide(bvh, cfg)) return launch_wide<Rec>(bvh, rays, hits, n, cfg, sp, is_tri, stream);
    return launch_kernel<Rec, false>(bvh, rays, hits, n, cfg, sp, is_tri, stream);
  };
  switch (type) {
  case TRIANGLES: return run(TriRecF{}, 1u);
  case SPHERES: return run(SphRecF{}, ow);
  case PLANES: return launch_kernel<PlaRecF, false>(bvh, rays, hits, n, cfg, sp, ow, stream);
  default: return run(CylRecF{}, ow);
  }
}

}  // namespace brt
