// HIP kernels for distance queries: blazeRT's distance_to_surface per (point, primitive) pair, and the closest
// surface of a whole scene per point.
//
// Per-primitive distances follow the reference's operation order in FP64 (contraction off):
//   spheres    blazert/primitives/sphere.h:179-182   |norm(center - p) - radius|
//   planes     blazert/primitives/plane.h:272-284    |local.z| when local.x, local.y lie within the plane's
//              world-space center +- half extent (the reference mixes the two frames), else DBL_MAX
//   cylinders  blazert/primitives/cylinder.h:507-759 (Newton iteration on the ellipse, region logic)
//   triangles  norm(p - closest_point_on_triangle(v0, v1, v2, p)), blazert/primitives/trimesh_distance.h:36-221.
//              The reference's triangle overload (trimesh.h:183-191) cannot be instantiated (it returns the point
//              as a scalar and rebuilds the vertices from the wrong edges); this is its evident intent.
//
// Closest surface: the smallest distance over every primitive of the scene, ties going to the earlier geometry
// type (triangles, spheres, planes, cylinders) and then to the lower primitive id -- the brute-force minimum.
// Triangles and spheres are searched through their BVHs: a child box is skipped when its distance from the point,
// less a margin of 1e-10 (|p| + scene extent), exceeds the best distance found, which no primitive inside it can
// then reach or tie. Planes and cylinders are scanned in full: the reference's plane distance can be smaller than
// the distance to the plane's box, and its cylinder box can miss part of a rotated cylinder.
#include <hip/hip_runtime.h>

#include <float.h>
#include <stdint.h>

#include "../../include/blazert_amd/user_geometry.h"  // RingStack: LDS stack ring with a private spill area
#include "engine.h"
#include "f32_round.h"
#include "wave.h"

namespace brt {

namespace {

__device__ __forceinline__ double dot3(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
// trans(R) * v for row-major R
__device__ __forceinline__ void mat_t_vec(const double *R, const double *v, double *r) {
  const double x = R[0] * v[0] + R[3] * v[1] + R[6] * v[2];
  const double y = R[1] * v[0] + R[4] * v[1] + R[7] * v[2];
  const double z = R[2] * v[0] + R[5] * v[1] + R[8] * v[2];
  r[0] = x;
  r[1] = y;
  r[2] = z;
}
__device__ __forceinline__ double min2(double a, double b) { return (b < a) ? b : a; }  // std::min(a, b)

// ------------------------------------------------------------------------------------------------ primitives
__device__ double sphere_distance(const SphRec &S, const double *p) {
  const double v[3] = {S.c[0] - p[0], S.c[1] - p[1], S.c[2] - p[2]};
  return fabs(__builtin_sqrt(dot3(v, v)) - S.r);
}

__device__ double plane_distance(const PlaRec &P, const double *p) {
  const double v[3] = {p[0] - P.c[0], p[1] - P.c[1], p[2] - P.c[2]};
  double l[3];
  mat_t_vec(P.R, v, l);
  const double dx = P.dx / 2, dy = P.dy / 2;
  const double cx = P.c[0], cy = P.c[1];
  if ((l[0] >= cx - dx) && (l[0] <= cx + dx) && (l[1] >= cy - dy) && (l[1] <= cy + dy)) return fabs(l[2]);
  return DBL_MAX;
}

enum : int { UPPER_X = 0, LOWER_X = 1, UPPER_Y = 2, LOWER_Y = 3 };

// cylinder.h:517-545
__device__ double distance_derivative(int kind, double a, double b, double xq, double yq, double val) {
  if (kind == UPPER_X || kind == LOWER_X) {
    const double s = (val * val > a * a) ? __builtin_sqrt(val * val - a * a) : __builtin_sqrt(a * a - val * val);
    if (kind == UPPER_X) return -2 * (xq - val) - 2 * b * val * (b / a * s - yq) / (a * s);
    return -2 * (xq - val) - 2 * b * val * (b / a * s + yq) / (a * s);
  }
  const double s = (val * val > b * b) ? __builtin_sqrt(val * val - b * b) : __builtin_sqrt(b * b - val * val);
  if (kind == UPPER_Y) return -2 * (yq - val) - 2 * a * val * (a / b * s + xq) / (b * s);
  return -2 * (yq - val) - 2 * a * val * (a / b * s - xq) / (b * s);
}

// cylinder.h:548-583
__device__ double single_newton_iteration(int kind, double a, double b, double xq, double yq, double val) {
  if (kind == UPPER_X || kind == LOWER_X) {
    const double s = (val * val > a * a) ? __builtin_sqrt(val * val - a * a) : __builtin_sqrt(a * a - val * val);
    if (kind == UPPER_X)
      return ((a * a * a * xq - a * val * val * xq) * s + b * val * val * val * yq) /
             ((a * a * a - a * b * b - a * val * val + b * b * val * val / a) * s + a * a * b * yq);
    return ((-a * a * a * xq + a * val * val * xq) * s + b * val * val * val * yq) /
           ((-a * a * a + a * b * b + a * val * val - b * b * val * val / a) * s + a * a * b * yq);
  }
  const double s = (val * val > b * b) ? __builtin_sqrt(val * val - b * b) : __builtin_sqrt(b * b - val * val);
  if (kind == UPPER_Y)
    return ((b * b * b * yq - b * val * val * yq) * s + a * val * val * val * xq) /
           ((b * b * b - b * a * a - b * val * val + a * a * val * val / b) * s + b * b * a * xq);
  return ((-b * b * b * yq + b * val * val * yq) * s + a * val * val * val * xq) /
         ((-b * b * b + b * a * a + b * val * val - a * a * val * val / b) * s + b * b * a * xq);
}

// cylinder.h:586-607: at most 100 steps, so every thread leaves the loop
__device__ double newton_iteration(int kind, double a, double b, double xq, double yq, double x0) {
  double val0 = x0;
  double cnt = 0;
  const double epsilon = 1e-7;
  while ((fabs(distance_derivative(kind, a, b, xq, yq, val0)) >= epsilon) && (cnt < 100)) {
    const double val = single_newton_iteration(kind, a, b, xq, yq, val0);
    val0 = val;
    cnt++;
    if (fabs(val0) == a) val0 += DBL_EPSILON;
  }
  return val0;
}

// cylinder.h:615-665
__device__ double min_distance_to_ellipse(double a, double b, double xq, double yq) {
  const double percentage = 0.95;
  if (((xq >= 0) && (yq >= (b / a) * xq)) || ((xq <= 0) && (yq >= (-b / a) * xq))) {
    const double x0 = xq > 0 ? percentage * a : -percentage * a;
    const double x_min = newton_iteration(UPPER_X, a, b, xq, yq, x0);
    const double s = __builtin_sqrt(a * a - x_min * x_min);
    const double y_min = b / a * s;
    return __builtin_sqrt((xq - x_min) * (xq - x_min) + (yq - y_min) * (yq - y_min));
  } else if (((xq >= 0) && (yq <= (-b / a) * xq)) || ((xq <= 0) && (yq <= (b / a) * xq))) {
    const double x0 = xq > 0 ? percentage * a : -percentage * a;
    const double x_min = newton_iteration(LOWER_X, a, b, xq, yq, x0);
    const double s = __builtin_sqrt(a * a - x_min * x_min);
    const double y_min = -b / a * s;
    return __builtin_sqrt((xq - x_min) * (xq - x_min) + (yq - y_min) * (yq - y_min));
  } else if ((xq >= 0) && (yq <= (b / a) * xq) && (yq >= (-b / a) * xq)) {
    const double y0 = yq > 0 ? percentage * b : -percentage * b;
    const double y_min = newton_iteration(UPPER_Y, a, b, xq, yq, y0);
    const double s = __builtin_sqrt(b * b - y_min * y_min);
    const double x_min = a / b * s;
    return __builtin_sqrt((yq - y_min) * (yq - y_min) + (xq - x_min) * (xq - x_min));
  } else {
    const double y0 = yq > 0 ? percentage * b : -percentage * b;
    const double y_min = newton_iteration(LOWER_Y, a, b, xq, yq, y0);
    const double s = __builtin_sqrt(b * b - y_min * y_min);
    const double x_min = -a / b * s;
    return __builtin_sqrt((yq - y_min) * (yq - y_min) + (xq - x_min) * (xq - x_min));
  }
}

// cylinder.h:677-759
__device__ double cylinder_distance(const CylRec &Cy, const double *p) {
  const double v[3] = {p[0] - Cy.c[0], p[1] - Cy.c[1], p[2] - Cy.c[2]};
  double l[3];
  mat_t_vec(Cy.R, v, l);
  const double a = Cy.a, b = Cy.b, h = Cy.h;
  const double dist_top = fabs(l[2] - h / 2);
  const double dist_bottom = fabs(l[2] + h / 2);
  const double xq = l[0], yq = l[1], zq = l[2];
  if (xq == 0 && yq == 0) {  // isZero(point_xy); std::min({...}) keeps the first smallest
    if ((zq > h / 2) || (zq < -h / 2)) return (dist_bottom < dist_top) ? dist_bottom : dist_top;
    double m = a;
    if (b < m) m = b;
    if (dist_top < m) m = dist_top;
    if (dist_bottom < m) m = dist_bottom;
    return m;
  }
  const double ellipse = (xq * xq) / (a * a) + (yq * yq) / (b * b) - 1;
  if (fabs(ellipse) < DBL_EPSILON) {
    if ((zq > h / 2) || (zq < -h / 2)) return min2(dist_top, dist_bottom);
    return 0.0;
  }
  if (ellipse < 0) {
    if (zq >= h / 2) return dist_top;
    if (zq <= -h / 2) return dist_bottom;
    double m = min_distance_to_ellipse(a, b, xq, yq);
    if (dist_bottom < m) m = dist_bottom;
    if (dist_top < m) m = dist_top;
    return m;
  }
  if (ellipse > 0) {
    if ((zq < h / 2) && (zq > -h / 2)) return min_distance_to_ellipse(a, b, xq, yq);
    const double ds = min_distance_to_ellipse(a, b, xq, yq);
    const double d1 = __builtin_sqrt(ds * ds + dist_top * dist_top);
    const double d2 = __builtin_sqrt(ds * ds + dist_bottom * dist_bottom);
    return (d2 < d1) ? d2 : d1;
  }
  return -1;
}

// trimesh_distance.h:176-221 with the region helpers r0-r6 (:36-171) in the same order
__device__ double triangle_distance(const double *v0, const double *v1, const double *v2, const double *p) {
  double E0[3], E1[3], D[3];
  for (int k = 0; k < 3; k++) {
    E0[k] = v1[k] - v0[k];
    E1[k] = v2[k] - v0[k];
    D[k] = v0[k] - p[k];
  }
  const double a = dot3(E0, E0), b = dot3(E0, E1), c = dot3(E1, E1), d = dot3(E0, D), e = dot3(E1, D);
  const double det = a * c - b * b;
  double s = b * e - c * d;
  double t = b * d - a * e;
  if (s + t <= det) {
    if (s < 0) {
      if (t < 0) {  // r4
        if (d < 0) {
          t = 0;
          s = (-d >= a) ? 1 : -d / a;
        } else {
          s = 0;
          if (e >= 0) t = 0;
          else t = (-e >= c) ? 1 : -e / c;
        }
      } else {  // r3
        s = 0;
        if (e >= 0) t = 0;
        else t = (-e >= c) ? 1 : -e / c;
      }
    } else if (t < 0) {  // r5
      t = 0;
      if (d >= 0) s = 0;
      else s = (-d >= a) ? 1 : -d / a;
    } else {  // r0
      const double inv_det = 1. / det;
      s *= inv_det;
      t *= inv_det;
    }
  } else {
    if (s < 0) {  // r2
      const double tmp0 = b + d, tmp1 = c + e;
      if (tmp1 > tmp0) {
        const double numer = tmp1 - tmp0, denom = a - 2. * b + c;
        s = (numer >= denom) ? 1 : numer / denom;
        t = 1. - s;
      } else {
        s = 0;
        if (tmp1 <= 0) t = 1;
        else if (e >= 0) t = 0;
        else t = -e / c;
      }
    } else if (t < 0) {  // r6
      const double tmp0 = b + e, tmp1 = a + d;
      if (tmp1 > tmp0) {
        const double numer = tmp1 - tmp0, denom = a - 2. * b + c;
        t = (numer >= denom) ? 1 : numer / denom;
        s = 1. - t;
      } else {
        t = 0;
        if (tmp1 <= 0) s = 1;
        else if (d >= 0) s = 0;
        else s = -d / a;
      }
    } else {  // r1
      const double numer = c + e - b - d;
      if (numer <= 0) {
        s = 0;
      } else {
        const double denom = a - 2. * b + c;
        s = (numer >= denom) ? 1 : numer / denom;
      }
      t = 1. - s;
    }
  }
  double w[3];
  for (int k = 0; k < 3; k++) w[k] = p[k] - (v0[k] + s * E0[k] + t * E1[k]);
  return __builtin_sqrt(dot3(w, w));
}

__device__ __forceinline__ double tri_distance_by_id(const BvhView &bvh, uint32_t id, const double *p) {
  const double *V = bvh.vertices;
  const uint32_t *F = bvh.faces + 3ull * id;
  return triangle_distance(V + 3ull * F[0], V + 3ull * F[1], V + 3ull * F[2], p);
}

// ------------------------------------------------------------------------------------------------ pairs
template <int TYPE>
__global__ void k_distance_pairs(BvhView bvh, const uint32_t *__restrict__ inv, const double *__restrict__ px,
                                 const double *__restrict__ py, const double *__restrict__ pz,
                                 const uint32_t *__restrict__ ids, uint64_t n, double *__restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double p[3] = {px[i], py[i], pz[i]};
  const uint32_t id = ids[i];
  double d = __builtin_nan("");
  if (id < bvh.n_prims) {
    if (TYPE == TRIANGLES) {
      d = tri_distance_by_id(bvh, id, p);
    } else if (TYPE == SPHERES) {
      d = sphere_distance(reinterpret_cast<const SphRec *>(bvh.prims)[inv[id]], p);
    } else if (TYPE == PLANES) {
      d = plane_distance(reinterpret_cast<const PlaRec *>(bvh.prims)[inv[id]], p);
    } else {
      d = cylinder_distance(reinterpret_cast<const CylRec *>(bvh.prims)[inv[id]], p);
    }
  }
  out[i] = d;
}

__global__ void k_leaf_vertices(const uint32_t *__restrict__ order, const uint32_t *__restrict__ F,
                                const double *__restrict__ V, uint32_t n, double *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t *f = F + 3ull * order[i];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int k = 0; k < 3; k++) out[9ull * i + 3 * c + k] = V[3ull * f[c] + k];
}

__global__ void k_inverse_order(const uint32_t *__restrict__ order, uint32_t n, uint32_t *__restrict__ inv) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) inv[order[i]] = i;
}

// ------------------------------------------------------------------------------------------------ closest
struct Best {
  double d;
  uint32_t id;
};

// within one geometry type the smaller distance wins, then the lower id (NaN never wins)
__device__ __forceinline__ void consider(Best &b, double d, uint32_t id) {
  if (d < b.d || (d == b.d && id < b.id)) {
    b.d = d;
    b.id = id;
  }
}

__device__ __forceinline__ double box_gap(const double *lo, const double *hi, const double *p) {
  double s = 0.0;
  for (int k = 0; k < 3; k++) {
    double g = 0.0;
    if (lo[k] - p[k] > g) g = lo[k] - p[k];
    if (p[k] - hi[k] > g) g = p[k] - hi[k];
    s += g * g;
  }
  return __builtin_sqrt(s);
}

// Traversal stack of the closest-surface query: the newest CLOSEST_RING entries of each point in LDS, deeper ones
// in a private spill area (trees are at most 63 levels deep on the device, so 64 entries always suffice).
constexpr int CLOSEST_RING = 8;
constexpr uint32_t CLOSEST_BLOCK = 128;
using ClosestStack = blazert_amd::RingStack<double, CLOSEST_RING>;

// Depth-first search of one BVH, nearer child first. `bound` is the best distance of earlier geometry types.
template <int TYPE, class Stack>
__device__ void closest_in_bvh(const BvhView &bvh, const double *leaf_vertices, const double *p, double margin,
                               double bound, Best &best, Stack &st) {
  st.sp = st.lo = 0;
  auto limit = [&]() { return best.d < bound ? best.d : bound; };
  if (box_gap(bvh.root_min, bvh.root_max, p) - margin > limit()) return;
  uint32_t ref = bvh.root_ref, cnt = bvh.root_cnt;
  while (true) {
    if (ref & LEAF_BIT) {
      const uint32_t first = ref & ~LEAF_BIT;
      for (uint32_t k = 0; k < cnt; k++) {
        // triangles read their vertices from the leaf-order copy: one gather instead of id -> face -> vertices
        const uint32_t id = bvh.prim_ids[first + k];
        const double *lv = leaf_vertices + 9ull * (first + k);
        const double d = (TYPE == TRIANGLES) ? triangle_distance(lv, lv + 3, lv + 6, p)
                                             : sphere_distance(reinterpret_cast<const SphRec *>(bvh.prims)[first + k], p);
        consider(best, d, id);
      }
    } else {
      const Node64 &nd = bvh.nodes64[ref];
      const double g0 = box_gap(nd.b, nd.b + 3, p), g1 = box_gap(nd.b + 6, nd.b + 9, p);
      const uint32_t r0 = nd.ref[0], r1 = nd.ref[1], c0 = nd.cnt[0], c1 = nd.cnt[1] & CNT_MASK;
      const double lim = limit();
      const bool ok0 = !(g0 - margin > lim), ok1 = !(g1 - margin > lim);
      if (ok0 && ok1) {
        const bool first0 = !(g1 < g0);
        st.push(first0 ? r1 : r0, first0 ? c1 : c0, first0 ? g1 : g0);
        ref = first0 ? r0 : r1;
        cnt = first0 ? c0 : c1;
        continue;
      }
      if (ok0 || ok1) {
        ref = ok0 ? r0 : r1;
        cnt = ok0 ? c0 : c1;
        continue;
      }
    }
    // pop the next entry still within reach
    bool found = false;
    while (!st.empty()) {
      double key;
      st.pop(ref, cnt, key);
      if (!(key - margin > limit())) {
        found = true;
        break;
      }
    }
    if (!found) return;
  }
}

__device__ __forceinline__ double rec_distance(const SphRec &r, const double *p) { return sphere_distance(r, p); }
__device__ __forceinline__ double rec_distance(const PlaRec &r, const double *p) { return plane_distance(r, p); }
__device__ __forceinline__ double rec_distance(const CylRec &r, const double *p) { return cylinder_distance(r, p); }

__device__ void closest_scan_triangles(const BvhView &bvh, const double *leaf_vertices, const double *p, Best &best) {
  for (uint32_t k = 0; k < bvh.n_prims; k++) {
    const double *lv = leaf_vertices + 9ull * k;
    consider(best, triangle_distance(lv, lv + 3, lv + 6, p), bvh.prim_ids[k]);
  }
}

template <class Rec>
__device__ void closest_scan(const BvhView &bvh, const double *p, Best &best) {
  const Rec *recs = reinterpret_cast<const Rec *>(bvh.prims);
  for (uint32_t k = 0; k < bvh.n_prims; k++) consider(best, rec_distance(recs[k], p), bvh.prim_ids[k]);
}

// ------------------------------------------------------------------------------------------------ closest, triangles
// The triangles of a scene with 4-wide FP32 nodes (NodeQ), one point per lane, nearest child first. A box or a triangle is
// skipped only when an FP32 lower bound of its distance, less the error of that bound, exceeds the best distance; every
// other triangle gets the FP64 distance, and the smallest (distance, id) does not depend on the visiting order.
//
// With u = 2^-24, Sm = max |p_i| + the largest |coordinate| of the boxes, and FP32 boxes rounded outward, the box gap
// computed here exceeds the exact one by at most 9 u Sm (three differences of inputs rounded once, and their norm). For a
// triangle and any vector w, |p - q| >= min_i (p - v_i).w / |w| over its vertices; w is taken from the centroid to p, which is
// nearly exact for a triangle that is small against its distance, and as the plane's normal. Those dot products are within
// 26 u Sm |w| of exact (each p - v_i within 4 u Sm per component, each dot within 3 u of its factors' norms).
// The normal serves for one vertex only where its own FP64 rounding, 2^-50 of the edges' product sa sb, turns it by less than
// u from the edges: for |n| > ed = 10 u sa sb, which leaves out triangles that are lines but for a rounding.
// slack = 32 u Sm covers both, and the FP64 distance's own 1e-10 Sm. The gaps are compared as squares: from
// WIDE_MIN_EXTENT on, slack alone keeps the squared limit above 3e-36, where the FP32 range still has all digits.
constexpr double WIDE_MIN_EXTENT = 1e-12;
constexpr uint32_t WIDE_RING = 16;
constexpr uint32_t WIDE_BLOCK = 256;

// The FP64 search with its stack in private memory.
__device__ __attribute__((noinline)) void closest_exact(const BvhView &bvh, const double *leaf_vertices, const double *p,
                                                        double margin, Best &best) {
  struct Stack {
    double key[64];
    uint32_t ref[64], cnt[64];
    int sp = 0, lo = 0;
    __device__ bool empty() const { return sp == 0; }
    __device__ void push(uint32_t r, uint32_t c, double k) {
      key[sp] = k;
      ref[sp] = r;
      cnt[sp++] = c;
    }
    __device__ void pop(uint32_t &r, uint32_t &c, double &k) {
      k = key[--sp];
      r = ref[sp];
      c = cnt[sp];
    }
  } st;
  closest_in_bvh<TRIANGLES>(bvh, leaf_vertices, p, margin, __builtin_inf(), best, st);
}

// Whether the triangle may hold a point nearer than lim (the best distance plus slack, rounded up).
__device__ __forceinline__ bool tri_in_reach(const TriFilt &T, const float P[3], float lim) {
  const float u = 5.9604644775390625e-08f;
  auto dot = [](float a0, float a1, float a2, float b0, float b1, float b2) {
    return __builtin_fmaf(a0, b0, __builtin_fmaf(a1, b1, a2 * b2));
  };
  const float c0 = P[0] - T.v0[0], c1 = P[1] - T.v0[1], c2 = P[2] - T.v0[2];  // p - v0; v1 = v0 - e1, v2 = v0 + e2
  const float k = 1.0f / 3.0f;
  const float w0 = __builtin_fmaf(k, T.e1[0] - T.e2[0], c0), w1 = __builtin_fmaf(k, T.e1[1] - T.e2[1], c1),
              w2 = __builtin_fmaf(k, T.e1[2] - T.e2[2], c2);
  const float cw = dot(c0, c1, c2, w0, w1, w2);
  const float m = fminf(cw, fminf(cw + dot(T.e1[0], T.e1[1], T.e1[2], w0, w1, w2),
                                  cw - dot(T.e2[0], T.e2[1], T.e2[2], w0, w1, w2)));
  const float ww = dot(w0, w1, w2, w0, w1, w2);
  const float cn = dot(c0, c1, c2, T.n[0], T.n[1], T.n[2]);
  const float nn = dot(T.n[0], T.n[1], T.n[2], T.n[0], T.n[1], T.n[2]);
  const float l2 = (lim * lim) * (1.0f + 16.0f * u);
  // products below 1e-30 may have lost digits to the denormal range: no rejection (nor on infinities and NaN)
  return !((m > 0.0f) & (m * m > l2 * ww) & (l2 * ww > 1e-30f)) &
         !((cn * cn > l2 * nn) & (l2 * nn > 1e-30f) & (nn > T.ed * T.ed));
}

__device__ __forceinline__ void order_pair(uint32_t &ka, uint32_t &ra, uint32_t &kb, uint32_t &rb) {
  const bool sw = kb < ka;
  const uint32_t k = ka, r = ra;
  ka = sw ? kb : ka;
  ra = sw ? rb : ra;
  kb = sw ? k : kb;
  rb = sw ? r : rb;
}

// Points whose parts several lanes search.
struct ClosestShare {
  double d[SHARE_SLOTS];
  unsigned long long bound[SHARE_SLOTS];  // bits of the smallest distance any part has found (distances are >= 0)
  uint32_t id[SHARE_SLOTS];
  uint32_t parts[SHARE_SLOTS];  // parts still running
};

// What bounds it: 1,048,576 points in [-2,2]^3 around 1.31M triangles take 3.41 ms (6.5 with binary FP64 nodes and FP64
// distances only, one point per thread), about 90 steps a point with a far from even spread; lines beyond L2 at 3.7 TB/s.
// 1,000 points on 82k triangles 351 -> 130 us, 50,000 on 328k 735 -> 463 us. Searches of a few steps each gain least, since a
// wave's lanes are then seldom at one kind of step: 1,000,000 points within 0.001 of 82k triangles 1.68 ms (1.60 one per
// thread), of a flat grid of 524,288 triangles 0.59 (0.31). Waiting lanes take these from 1.75 and 0.62, and the first from 3.70.
//
// Persistent waves as in the ray traversal (or `fixed` points per wave): lanes whose point is done start the wave's next
// ones, and once there are none, idle lanes take over stack entries of the busy ones, whose best distances they share.
__global__ void __launch_bounds__(WIDE_BLOCK)
k_closest_triangles(ClosestViews V, const double *__restrict__ px, const double *__restrict__ py,
                    const double *__restrict__ pz, uint64_t n, unsigned long long *group, uint32_t fixed,
                    double *__restrict__ dist, uint32_t *__restrict__ prim, uint32_t *__restrict__ geom) {
  using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
  using Bytes = const __attribute__((address_space(1))) unsigned char;
  typedef u32x4 __attribute__((aligned(8))) Chunk;  // the vertices are 72-byte records
  using GlobalChunk = const __attribute__((address_space(1))) Chunk;
  __shared__ uint64_t ring[WIDE_RING * WIDE_BLOCK];
  __shared__ ClosestShare shares[WIDE_BLOCK / 64];
  const BvhView &bvh = V.view[TRIANGLES];
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  BRT_LDS volatile ClosestShare *sh = (BRT_LDS volatile ClosestShare *)&shares[wave];
  uint64_t spill[WIDE_SPILL];
  WideStack st;
  st.ring = (BRT_LDS uint32_t *)ring + (size_t)wave * WIDE_RING * 128 + lane;
  st.spill = spill;
  st.mask = (int)WIDE_RING - 1;
  st.reset();
  WavePool pool;
  if (fixed) pool.take_fixed(((uint64_t)blockIdx.x * (WIDE_BLOCK / 64) + wave) * fixed, fixed, n);
  bool exhausted = false;  // wave-uniform
  uint64_t i = 0;
  double p[3] = {0.0, 0.0, 0.0};
  float P[3] = {0.0f, 0.0f, 0.0f}, slack = 0.0f;
  float lim = 0.0f;  // best distance + slack, rounded up
  Best best{__builtin_inf(), INVALID_ID};
  uint32_t cur = 0, cnt = 0, cand = 0;
  bool busy = false, shared = false;
  uint32_t slot = 0, slots = 0, turn = 0;
  for (;;) {
    const unsigned long long working = __ballot(busy);
    const uint32_t nidle = 64u - (uint32_t)__popcll(working);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (!exhausted) {
      if (nidle >= 16u) {
        bool got;
        pool_refill(pool, group + COUNTER_POOL, n, POOL_CHUNK, ~working, nidle, lane, got, i, exhausted);
        if (got) {
          p[0] = px[i];
          p[1] = py[i];
          p[2] = pz[i];
          const double pm = fmax(fabs(p[0]), fmax(fabs(p[1]), fabs(p[2])));
          best = Best{__builtin_inf(), INVALID_ID};
          if (pm <= FILTER_MAX_EXTENT && p[0] == p[0] && p[1] == p[1] && p[2] == p[2]) {
#pragma unroll
            for (int k = 0; k < 3; k++) P[k] = (float)p[k];
            slack = f32_up(32.0 * 0x1p-24 * (pm + V.extent[TRIANGLES]));
            lim = __builtin_inff();
            cur = bvh.root_ref4;
            cnt = bvh.root_cnt;
            cand = 0;
            busy = true;
            st.reset();
          } else {
            // a point outside the FP32 bounds' range, or not a number: the FP64 search
            closest_exact(bvh, V.leaf_vertices, p, 1e-10 * (pm + V.extent[TRIANGLES]), best);
            const bool found = best.d < __builtin_inf();
            dist[i] = found ? best.d : __builtin_inf();
            prim[i] = found ? best.id : INVALID_ID;
            geom[i] = found ? bvh.geom_id : INVALID_ID;
          }
        }
      }
    } else {
      if (!working) break;
      const unsigned long long can = __ballot(busy && st.sp > st.bot);
            if (nidle >= SHARE_MIN_IDLE && can && (++turn & 1u) == 0u) {
        const uint32_t ncan = (uint32_t)__popcll(can), k = nidle < ncan ? nidle : ncan;
        const uint32_t rank = (uint32_t)__popcll((busy ? can : ~working) & below);
        const bool donor = ((can >> lane) & 1ull) && rank < k, helper = !busy && rank < k;
        const unsigned long long fresh = __ballot(donor && !shared);
        uint64_t e = 0;
        if (donor) {
          const WideEntry t = st.pop();  // the nearest entry: the bottom one would mostly be out of reach in the end
          e = ((uint64_t)t.key << 32) | t.ref;
          if (!shared) {
            shared = true;
            slot = slots + (uint32_t)__popcll(fresh & below);
            sh->d[slot] = __builtin_inf();
            sh->bound[slot] = (unsigned long long)__double_as_longlong(best.d);
            sh->id[slot] = INVALID_ID;
            sh->parts[slot] = 1u;
          }
        }
        slots += (uint32_t)__popcll(fresh);
        wave_fence();
        if (donor) atomicAdd(&shares[wave].parts[slot], 1u);
        // the r-th helper takes from the r-th donor, whose lane number lane r receives (at most 32 donors: lane 63 takes
        // what the others push); both permutes with all lanes, since they serve active lanes only
        const uint32_t by_rank = (uint32_t)__builtin_amdgcn_ds_permute((donor ? (int)rank : 63) << 2, (int)lane);
        const uint32_t from = lane_get(by_rank, (int)rank);
        const int src = helper ? (int)from : (int)lane;
        lane_take(e, src, helper);
        lane_take(p, src, helper);
        lane_take(P, src, helper);
        lane_take(slack, src, helper);
        lane_take(lim, src, helper);
        lane_take(slot, src, helper);
        lane_take(i, src, helper);
        if (helper) {
          busy = shared = true;
          best = Best{__builtin_inf(), INVALID_ID};
          cur = (uint32_t)e;
          cnt = (uint32_t)(e >> 32) & 255u;
          cand = 0;
          st.reset();
        }
        wave_fence();
      }
    }
    bool fin = false;
    bool go = busy;
    if (!exhausted) {  // lanes with a pre-test or an FP64 distance wait until WIDE_MIN_LANES have one, or nothing else is left
      const bool leaf = busy && (cur & LEAF_BIT) != 0, test = leaf && cand != 0u, group = leaf && cand == 0u;
      const int tests = __popcll(__ballot(test)), groups = __popcll(__ballot(group));
      const int nodes = __popcll(__ballot(busy)) - tests - groups;
      if (test && tests < WIDE_MIN_LANES && nodes + groups != 0) go = false;
      if (group && groups < WIDE_MIN_LANES && nodes != 0) go = false;
    }
    if (go) {
      if (shared) {
        const double d = __longlong_as_double((long long)sh->bound[slot]);
        lim = fminf(lim, f32_up((double)f32_up(d) + (double)slack));
      }
      // one unit per iteration, as in the ray traversal: a node, a pre-test of two triangles or an FP64 distance
      const bool at_leaf = (cur & LEAF_BIT) != 0, test = cand != 0u;
      const uint32_t first = cur & ~LEAF_BIT;
      const uint32_t q = first + (uint32_t)__builtin_ctz(cand | 0x80000000u);
      Bytes *base = !at_leaf ? (Bytes *)(bvh.nodesq + cur)
                    : test   ? (Bytes *)(V.leaf_vertices + 9ull * q)
                             : (Bytes *)(bvh.tri_filter + first);
      u32x4 c[8];
#pragma unroll
      for (int k = 0; k < 4; k++) c[k] = *(GlobalChunk *)(base + 16 * k);
      if (!test) {
#pragma unroll
        for (int k = 4; k < 8; k++) c[k] = *(GlobalChunk *)(base + 16 * k);
      } else {
        const __attribute__((address_space(1))) uint32_t *w = (const __attribute__((address_space(1))) uint32_t *)(base + 64);
        c[4][0] = w[0];
        c[4][1] = w[1];
      }
#pragma unroll
      for (int k = 0; k < 8; k++) asm volatile("" : "+v"(c[k]));
      bool pop = true;
      if (!at_leaf) {
        const float l2 = (lim * lim) * (1.0f + 0x1p-20f);
        uint32_t key[4], ref[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          float g2 = 0.0f;
#pragma unroll
          for (int a = 0; a < 3; a++) {
            const float g = fmaxf(fmaxf(__uint_as_float(c[a][s]) - P[a], P[a] - __uint_as_float(c[4 + a][s])), 0.0f);
            g2 = __builtin_fmaf(g, g, g2);
          }
          // (an unused slot's inverted box is infinitely far)
          const bool in = g2 <= l2 && g2 < __builtin_inff();
          key[s] = in ? __builtin_amdgcn_perm(__float_as_uint(g2), c[7][2], 0x07060500u | (uint32_t)s) : 0xFFFFFFFFu;
          ref[s] = c[3][s];
        }
        order_pair(key[0], ref[0], key[1], ref[1]);
        order_pair(key[2], ref[2], key[3], ref[3]);
        order_pair(key[0], ref[0], key[2], ref[2]);
        order_pair(key[1], ref[1], key[3], ref[3]);
        order_pair(key[1], ref[1], key[2], ref[2]);
        if (key[0] != 0xFFFFFFFFu) {
          st.room(3);
#pragma unroll
          for (int s = 3; s > 0; s--)
            if (key[s] != 0xFFFFFFFFu) st.put(st.sp++, ref[s], key[s]);
          cur = ref[0];
          cnt = key[0] & 255u;
          pop = false;
        }
      } else if (!test) {
        TriFilt g[2];
        __builtin_memcpy(g, c, sizeof g);
        cand = (tri_in_reach(g[0], P, lim) ? 1u : 0u) | (tri_in_reach(g[1], P, lim) && cnt > 1u ? 2u : 0u);
        pop = cand == 0u;
      } else {
        double v[9];
        __builtin_memcpy(v, c, sizeof v);
        const double d = triangle_distance(v, v + 3, v + 6, p);
        if (d <= best.d) {
          consider(best, d, bvh.prim_ids[q]);
          lim = fminf(lim, f32_up((double)f32_up(best.d) + (double)slack));
          if (shared) atomicMin(&shares[wave].bound[slot], (unsigned long long)__double_as_longlong(best.d));
        }
        cand &= cand - 1u;
        pop = cand == 0u;
      }
      if (pop) {
        if (at_leaf && cnt > 2u) {
          cnt -= 2u;
          cur += 2u;
        } else {
          const float l2 = (lim * lim) * (1.0f + 0x1p-20f);
          fin = true;
          while (st.sp > st.bot) {
            const WideEntry e = st.pop();
            if (!(__uint_as_float(e.key & ~255u) > l2)) {
              cur = e.ref;
              cnt = e.key & 255u;
              fin = false;
              break;
            }
          }
        }
      }
    }
    if (exhausted) {
      // the parts of a shared point are merged one lane at a time; the last one writes it
      unsigned long long m = __ballot(fin && shared);
      while (m) {
        const uint32_t l = (uint32_t)__ffsll((long long)m) - 1u;
        m &= m - 1ull;
        if (lane == l) {
          consider(best, sh->d[slot], sh->id[slot]);
          sh->d[slot] = best.d;
          sh->id[slot] = best.id;
          const uint32_t parts = sh->parts[slot] - 1u;
          sh->parts[slot] = parts;
          busy = shared = false;
          fin = parts == 0u;
        }
        wave_fence();
      }
    }
    if (fin) {
      busy = false;
      const bool found = best.d < __builtin_inf();
      dist[i] = found ? best.d : __builtin_inf();
      prim[i] = found ? best.id : INVALID_ID;
      geom[i] = found ? bvh.geom_id : INVALID_ID;
    }
  }
}

// `from`: the geometry types before it are done, their result is in the output arrays.
__global__ void k_closest_surface(ClosestViews V, int from, const double *__restrict__ px, const double *__restrict__ py,
                                  const double *__restrict__ pz, uint64_t n, double *__restrict__ dist,
                                  uint32_t *__restrict__ prim, uint32_t *__restrict__ geom) {
  __shared__ double lkey[CLOSEST_RING * CLOSEST_BLOCK];
  __shared__ uint32_t lref[CLOSEST_RING * CLOSEST_BLOCK], lcnt[CLOSEST_RING * CLOSEST_BLOCK];
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  blazert_amd::StackArea<double> spill;
  ClosestStack st{(blazert_amd::LdsPtr<double>)(lkey + threadIdx.x), (blazert_amd::LdsPtr<uint32_t>)(lref + threadIdx.x),
                  (blazert_amd::LdsPtr<uint32_t>)(lcnt + threadIdx.x), CLOSEST_BLOCK, &spill};
  const double p[3] = {px[i], py[i], pz[i]};
  const double pm = fmax(fabs(p[0]), fmax(fabs(p[1]), fabs(p[2])));
  double gd = __builtin_inf();
  uint32_t gp = INVALID_ID, gg = INVALID_ID;
  if (from) {
    gd = dist[i];
    gp = prim[i];
    gg = geom[i];
  }
  for (int t = from; t < NUM_TYPES; t++) {
    const BvhView &bvh = V.view[t];
    if (!V.present[t] || bvh.n_prims == 0) continue;
    Best b{__builtin_inf(), INVALID_ID};
    const double margin = 1e-10 * (pm + V.extent[t]);
    // box pruning needs boxes that contain their primitives: a tree with an inverted or NaN node box (a sphere with a
    // negative radius) is scanned in full instead
    if (t == TRIANGLES && !bvh.irregular_boxes) closest_in_bvh<TRIANGLES>(bvh, V.leaf_vertices, p, margin, gd, b, st);
    else if (t == TRIANGLES) closest_scan_triangles(bvh, V.leaf_vertices, p, b);
    else if (t == SPHERES && !bvh.irregular_boxes) closest_in_bvh<SPHERES>(bvh, nullptr, p, margin, gd, b, st);
    else if (t == SPHERES) closest_scan<SphRec>(bvh, p, b);
    else if (t == PLANES) closest_scan<PlaRec>(bvh, p, b);
    else closest_scan<CylRec>(bvh, p, b);
    if (b.d < gd) {  // a later type replaces only when strictly closer
      gd = b.d;
      gp = b.id;
      gg = bvh.geom_id;
    }
  }
  dist[i] = gd;
  prim[i] = gp;
  geom[i] = gg;
}

}  // namespace

hipError_t launch_inverse_order(const uint32_t *order, uint32_t n, uint32_t *inv, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  k_inverse_order<<<(n + 255) / 256, 256, 0, stream>>>(order, n, inv);
  return hipGetLastError();
}

hipError_t launch_leaf_vertices(const uint32_t *order, const uint32_t *faces, const double *vertices, uint32_t n,
                                double *out, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  k_leaf_vertices<<<(n + 255) / 256, 256, 0, stream>>>(order, faces, vertices, n, out);
  return hipGetLastError();
}

hipError_t launch_distance_pairs(GeomType type, const BvhView &bvh, const uint32_t *inv, const double *px,
                                 const double *py, const double *pz, const uint32_t *ids, uint64_t n, double *out,
                                 hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint32_t blocks = (uint32_t)((n + 255) / 256);
  switch (type) {
  case TRIANGLES: k_distance_pairs<TRIANGLES><<<blocks, 256, 0, stream>>>(bvh, inv, px, py, pz, ids, n, out); break;
  case SPHERES: k_distance_pairs<SPHERES><<<blocks, 256, 0, stream>>>(bvh, inv, px, py, pz, ids, n, out); break;
  case PLANES: k_distance_pairs<PLANES><<<blocks, 256, 0, stream>>>(bvh, inv, px, py, pz, ids, n, out); break;
  default: k_distance_pairs<CYLINDERS><<<blocks, 256, 0, stream>>>(bvh, inv, px, py, pz, ids, n, out); break;
  }
  return hipGetLastError();
}

hipError_t launch_closest_surface(const ClosestViews &views, const double *px, const double *py, const double *pz,
                                  uint64_t n, double *dist, uint32_t *prim, uint32_t *geom,
                                  const std::function<unsigned long long *()> &claims, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  int from = 0;
  const BvhView &tri = views.view[TRIANGLES];
  if (views.present[TRIANGLES] && tri.nodesq && tri.tri_filter && views.extent[TRIANGLES] >= WIDE_MIN_EXTENT) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_closest_triangles, WIDE_BLOCK, 0);
    if (e != hipSuccess) return e;
    constexpr uint32_t waves = WIDE_BLOCK / 64;
    uint64_t blocks = (uint64_t)(cus > 0 ? cus : 1) * (uint64_t)(per_cu > 0 ? per_cu : 1);
    const uint64_t per_wave = (n + blocks * waves - 1) / (blocks * waves);
    uint32_t fixed = fixed_per_wave(n, blocks * waves);
    unsigned long long *group = fixed ? nullptr : claims();
    // Without counters every wave takes one range, as large as it has to be. 4,000,000 points on 1.31M triangles take
    // 12.1 ms that way and 11.6 with claims, 1,048,576 points 3.73 and 3.69 ms.
    if (!fixed && !group) {
      if (per_wave > 0xffffffffull) return hipErrorInvalidValue;
      fixed = (uint32_t)per_wave;
    }
    if (group) e = launch_zero_counters(group, stream);
    if (e != hipSuccess) return e;
    const uint64_t range = fixed ? (uint64_t)fixed * waves : WIDE_BLOCK, need = (n + range - 1) / range;
    if (blocks > need) blocks = need;
    k_closest_triangles<<<(uint32_t)blocks, WIDE_BLOCK, 0, stream>>>(views, px, py, pz, n, group, fixed, dist, prim, geom);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    from = TRIANGLES + 1;
    bool more = false;
    for (int t = from; t < NUM_TYPES; t++) more = more || views.present[t];
    if (!more) return hipSuccess;
  }
  k_closest_surface<<<(uint32_t)((n + CLOSEST_BLOCK - 1) / CLOSEST_BLOCK), CLOSEST_BLOCK, 0, stream>>>(
      views, from, px, py, pz, n, dist, prim, geom);
  return hipGetLastError();
}

}  // namespace brt
