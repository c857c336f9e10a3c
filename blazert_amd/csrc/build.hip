// Device build of one geometry type's BVH (commit() on the GPU).
//
// Produces the host builder's tree (scene.cpp, itself blazert/bvh/builder.h:46-226 with binbuffer.h:15-167 and
// bbox.h:27-39), the same primitive order and the same flattened Node64 / Node4 / primitive-record arrays, bit for
// bit, whenever no primitive box coordinate is NaN or a negative zero. Under that condition every min / max the
// builder takes has one result whatever the evaluation order, so node bounds and bins are reduced with atomics.
// The order-dependent steps are reproduced exactly:
//   * the SAH sweeps of find_best_split_binned (binbuffer.h:115-166) become prefix / suffix scans over the bins,
//     one lane per bin, with the same products and sums; the first minimum wins as in the sequential loop;
//   * the partition is libstdc++'s std::partition on random-access iterators (bidirectional algorithm). It swaps
//     the i-th element of the left part [begin, begin + T) that fails the predicate with the i-th element of the
//     right part that passes it, counted from the right end, and leaves every other element in place (T = number
//     of passing elements). Ranks from prefix counts therefore give its exact result.
// Nodes with more than SMALL primitives are processed level by level, several blocks per node; the nodes of more than TINY
// primitives in a subtree of at most SMALL are then split by one wave out of LDS, and each subtree of at most TINY by 16
// lanes, one primitive per lane, all its nodes of a level at once. Nodes are numbered in pre-order in closed form: a node
// whose primitives begin at b and whose path from the root has l left turns is number 2 L(b) + l, L(b) being the number of
// leaves that begin before b (the left subtrees hanging off its path hold 2 L(b) nodes less one for every right turn, and
// its ancestors are as many as the turns). Its number among the internal nodes is L(b) + l.
#include <hip/hip_runtime.h>

#include <float.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "../../include/blazert_amd/device/exact.h"
#include "engine.h"
#include "f32_round.h"

namespace brt {

namespace {

typedef unsigned long long u64;

constexpr uint32_t SMALL = 256;          // subtrees of at most this many primitives are split by one wave
constexpr uint32_t TINY = 16;            // subtrees of at most this many primitives are built by 16 lanes
constexpr uint32_t CHUNK = 2048;         // primitives per block in the level passes
constexpr uint32_t BLOCK = 256;          // threads per block in the level passes
constexpr uint32_t STACK = 64;           // depth-first stack of the subtree waves (max_depth <= 62)

// Order-preserving unsigned key of a double (NaN excluded): min / max of keys = min / max of values.
__device__ __forceinline__ u64 okey(double x) {
  const u64 b = (u64)__double_as_longlong(x);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double okey_value(u64 k) {
  return __longlong_as_double((long long)((k >> 63) ? (k & 0x7fffffffffffffffull) : ~k));
}
__device__ __forceinline__ double dmin(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double dmax(double a, double b) { return a < b ? b : a; }

// unsigned(std::round(x)) as the reference's x86-64 build evaluates it, clamped to the last bin
// (blazert/bvh/binbuffer.h:86-88)
__device__ __forceinline__ uint32_t bin_of(double x, uint32_t last) {
  const double r = round(x);
  uint32_t u = 0;
  if (r == r && r < 9.2e18 && r > -9.2e18) u = (uint32_t)(uint64_t)(int64_t)r;
  return u < last ? u : last;
}

// blazert/bvh/bbox.h:27-39
__device__ __forceinline__ double surface(const double *lo, const double *hi) {
  const double b0 = fabs(hi[0] - lo[0]), b1 = fabs(hi[1] - lo[1]), b2 = fabs(hi[2] - lo[2]);
  return 2.0 * (b0 * b1 + b1 * b2 + b2 * b0);
}

// Bins of one node: bin t = axis * nb + b holds a count and the min / max keys of the boxes binned there
// (3 keys each, at 3t + k).
struct Bins {
  uint32_t *cnt;
  u64 *klo, *khi;
};

// SAH sweep of one node over its bins (find_best_split_binned, binbuffer.h:115-166): all 64 lanes of a wave call
// it with the same arguments (nb <= 64); returns the split axis and writes the three cut positions.
__device__ uint32_t sah_sweep(const uint32_t *cnt, const u64 *klo, const u64 *khi, uint32_t nb, const double *lo,
                              const double *hi, double *cut) {
  const int lane = threadIdx.x & 63;
  double min_cost[3];
  for (int j = 0; j < 3; j++) {
    const bool in = lane < (int)nb;
    const uint32_t t = j * nb + lane;
    const uint64_t c = in ? cnt[t] : 0;
    double bl[3], bh[3];
    for (int k = 0; k < 3; k++) {
      bl[k] = in ? okey_value(klo[3 * t + k]) : DBL_MAX;
      bh[k] = in ? okey_value(khi[3 * t + k]) : -DBL_MAX;
    }
    // right side: bins lane .. nb-1 (the right-to-left sweep)
    double sl[3] = {bl[0], bl[1], bl[2]}, sh[3] = {bh[0], bh[1], bh[2]};
    uint64_t sc = c;
    for (int off = 1; off < 64; off <<= 1) {
      const bool ok = lane + off < 64;
      const uint64_t oc = __shfl_down(sc, off);
      if (ok) sc += oc;
      for (int k = 0; k < 3; k++) {
        const double ol = __shfl_down(sl[k], off), oh = __shfl_down(sh[k], off);
        if (ok) {
          sl[k] = dmin(sl[k], ol);
          sh[k] = dmax(sh[k], oh);
        }
      }
    }
    const double rcost = (double)sc * surface(sl, sh);
    // left side: bins 0 .. lane (the left-to-right sweep)
    double pl[3] = {bl[0], bl[1], bl[2]}, ph[3] = {bh[0], bh[1], bh[2]};
    uint64_t pc = c;
    for (int off = 1; off < 64; off <<= 1) {
      const bool ok = lane >= off;
      const uint64_t oc = __shfl_up(pc, off);
      if (ok) pc += oc;
      for (int k = 0; k < 3; k++) {
        const double ol = __shfl_up(pl[k], off), oh = __shfl_up(ph[k], off);
        if (ok) {
          pl[k] = dmin(pl[k], ol);
          ph[k] = dmax(ph[k], oh);
        }
      }
    }
    const double rnext = __shfl_down(rcost, 1);
    const double cost = (double)pc * surface(pl, ph) + rnext;
    // the sequential loop keeps the first cost below its running minimum (which starts at DBL_MAX): the first
    // lane holding the smallest cost below DBL_MAX, NaN never taken
    const bool valid = lane + 1 < (int)nb && cost < DBL_MAX;
    double m = valid ? cost : __builtin_inf();
    for (int off = 32; off > 0; off >>= 1) m = dmin(m, __shfl_xor(m, off));
    uint32_t min_bin = 1;
    min_cost[j] = DBL_MAX;
    if (m < DBL_MAX) {
      const u64 mask = __ballot(valid && cost == m);
      min_bin = (uint32_t)__ffsll((long long)mask);  // lowest such lane + 1
      min_cost[j] = m;
    }
    cut[j] = (double)min_bin * ((hi[j] - lo[j]) / (double)nb) + lo[j];
  }
  uint32_t axis = 0;
  if (min_cost[0] > min_cost[1]) axis = 1;
  if (min_cost[axis] > min_cost[2]) axis = 2;
  return axis;
}

// Exclusive rank of `flag` among the block's threads (thread order) and the block's total; every thread of the
// block must call it.
__device__ __forceinline__ uint32_t block_rank(bool flag, uint32_t *wave_tot, uint32_t &total) {
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const u64 m = __ballot(flag);
  const uint32_t in_wave = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  if (lane == 0) wave_tot[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = 0, tot = 0;
  for (uint32_t w = 0; w < nw; w++) {
    const uint32_t c = wave_tot[w];
    before += (w < wave) ? c : 0u;
    tot += c;
  }
  __syncthreads();
  total = tot;
  return before + in_wave;
}

// ------------------------------------------------------------------------------------------------ inputs
// What the triangles' inputs mean for the device build.
struct MeshFlags {
  uint32_t refused;   // some box coordinate is not finite or is -0.0: the order-free reductions would not be exact
  uint32_t max_fan;   // most corners at one vertex of a long fan; 2^32 - 1 when some face normal is NaN
  uint32_t num_long;  // vertices of more than FAN_SHORT corners
};
constexpr uint32_t FAN_SHORT = 64;    // corners one thread sums
constexpr uint32_t FAN_LONG = 4096;   // corners one block sums; beyond, the host computes the normals

// Triangle boxes and centers exactly as the host collection precompute (blazert/primitives/trimesh.h:78-130), each face's
// share of its vertices' normals, normalize(cross(v1 - v0, v2 - v0)) / 3, and the number of corners at every vertex.
__global__ void k_tri_boxes(const double *__restrict__ V, const uint32_t *__restrict__ F, uint32_t n,
                            double *__restrict__ lo, double *__restrict__ hi, double *__restrict__ ctr,
                            double *__restrict__ fn3, uint32_t *__restrict__ fan, MeshFlags *__restrict__ flags) {
  const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n) return;
  const uint32_t i0 = F[3ull * f], i1 = F[3ull * f + 1], i2 = F[3ull * f + 2];
  const double *v0 = V + 3ull * i0, *v1 = V + 3ull * i1, *v2 = V + 3ull * i2;
  const double third = 1.0 / 3.0;
  bool odd = false;
  double a[3], b[3];
  for (int k = 0; k < 3; k++) {
    double l = v0[k], h = v0[k];
    l = (l < v1[k]) ? l : v1[k];
    h = (v1[k] < h) ? h : v1[k];
    l = (l < v2[k]) ? l : v2[k];
    h = (v2[k] < h) ? h : v2[k];
    lo[3ull * f + k] = l;
    hi[3ull * f + k] = h;
    ctr[3ull * f + k] = ((v0[k] + v1[k]) + v2[k]) * third;
    const u64 neg0 = 0x8000000000000000ull;
    odd = odd || !(fabs(l) <= DBL_MAX) || !(fabs(h) <= DBL_MAX) || (u64)__double_as_longlong(l) == neg0 ||
          (u64)__double_as_longlong(h) == neg0;
    a[k] = v1[k] - v0[k];
    b[k] = v2[k] - v0[k];
  }
  if (odd) flags->refused = 1u;
  const double c[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
  const double len = __builtin_sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
  const double il = (len != 0.0) ? 1.0 / len : 0.0;
  bool nan = false;
  for (int k = 0; k < 3; k++) {
    const double x = (c[k] * il) * third;
    fn3[3ull * f + k] = x;
    nan = nan || x != x;
  }
  if (nan) flags->max_fan = 0xFFFFFFFFu;  // a NaN's sign and payload are the host's to choose
  atomicAdd(&fan[i0], 1u);
  atomicAdd(&fan[i1], 1u);
  atomicAdd(&fan[i2], 1u);
}

__global__ void k_zero_words(uint32_t *p, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// Corner c = 3 face + k goes to one of its vertex's places [start[v], start[v] + fan[v]), in no particular order;
// `left` starts as the fans and counts down.
__global__ void k_corners(const uint32_t *__restrict__ F, uint32_t corners, const uint32_t *__restrict__ start,
                          uint32_t *__restrict__ left, uint32_t *__restrict__ at) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= corners) return;
  const uint32_t v = F[c];
  at[start[v] + atomicSub(&left[v], 1u) - 1u] = c;
}

// Vertex normals as the host sums them (trimesh.h:91-93): every corner's share in ascending corner order. A short fan is
// summed by one thread, which looks for the next larger corner each time (six of them as a rule); long ones are listed.
__global__ void k_vertex_normals(const uint32_t *__restrict__ start, const uint32_t *__restrict__ ends, uint32_t nv,
                                 const uint32_t *__restrict__ at, const double *__restrict__ fn3,
                                 double *__restrict__ out, uint32_t *__restrict__ longs, MeshFlags *__restrict__ flags) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const uint32_t b = start[v], m = ends[v] - b;
  if (m > FAN_SHORT) {
    longs[atomicAdd(&flags->num_long, 1u)] = v;
    atomicMax(&flags->max_fan, m);  // (after k_tri_boxes: a NaN's mark stays)
    return;
  }
  double s[3] = {0.0, 0.0, 0.0};
  uint32_t from = 0;
  for (uint32_t k = 0; k < m; k++) {
    uint32_t c = 0xFFFFFFFFu;
    for (uint32_t j = 0; j < m; j++) {
      const uint32_t x = at[b + j];
      c = (x >= from && x < c) ? x : c;
    }
    const double *f = fn3 + 3ull * (c / 3u);
    for (int a = 0; a < 3; a++) s[a] = s[a] + f[a];
    from = c + 1u;
  }
  for (int a = 0; a < 3; a++) out[3ull * v + a] = s[a];
}

// Long fans, one block each: every corner's rank by counting, then the sum in order.
__global__ void k_vertex_normals_long(const uint32_t *__restrict__ start, const uint32_t *__restrict__ ends,
                                      const uint32_t *__restrict__ at, const double *__restrict__ fn3,
                                      const uint32_t *__restrict__ longs, const MeshFlags *__restrict__ flags,
                                      double *__restrict__ out) {
  __shared__ uint32_t sorted[FAN_LONG];
  for (uint32_t l = blockIdx.x; l < flags->num_long; l += gridDim.x) {
    const uint32_t v = longs[l], b = start[v], m = ends[v] - b;
    if (m > FAN_LONG) continue;
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) {
      const uint32_t x = at[b + i];
      uint32_t rank = 0;
      for (uint32_t j = 0; j < m; j++) rank += at[b + j] < x ? 1u : 0u;
      sorted[rank] = x;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      double s = 0.0;
      for (uint32_t i = 0; i < m; i++) s = s + fn3[3ull * (sorted[i] / 3u) + threadIdx.x];
      out[3ull * v + threadIdx.x] = s;
    }
    __syncthreads();
  }
}

__global__ void k_iota(uint32_t *idx, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) idx[i] = i;
}

// ------------------------------------------------------------------------------------------------ large nodes
// One node of the current level (nodes with more than SMALL primitives).
struct LNode {
  uint32_t begin, n, depth, leaf;
  uint32_t axis, mid, bad, split;
  uint32_t blk0, nblk, misplaced, pad;
  uint32_t cnt3[4];
  u64 klo[3], khi[3];
  double lo[3], hi[3], cut[3];
};

struct Level {
  LNode *nodes;
  const uint32_t *blk_node, *blk_start;  // block -> level node, first position of the block
  uint32_t *blk_l, *blk_r, *off_l, *off_r;
  Bins bins;
};

__device__ __forceinline__ uint32_t block_stop(const LNode &nd, uint32_t start) {
  const uint32_t end = nd.begin + nd.n;
  return (end - start < CHUNK) ? end : start + CHUNK;
}

__global__ void k_lv_init(Level L, uint32_t nb) {
  LNode &nd = L.nodes[blockIdx.x];
  const uint32_t tid = threadIdx.x;
  if (tid < 3) {
    nd.klo[tid] = okey(DBL_MAX);
    nd.khi[tid] = okey(-DBL_MAX);
    nd.cnt3[tid] = 0;
  }
  const size_t base = (size_t)blockIdx.x * 3 * nb;
  for (uint32_t t = tid; t < 3 * nb; t += blockDim.x) {
    L.bins.cnt[base + t] = 0;
    for (int k = 0; k < 3; k++) {
      L.bins.klo[3 * (base + t) + k] = okey(DBL_MAX);
      L.bins.khi[3 * (base + t) + k] = okey(-DBL_MAX);
    }
  }
}

// Node bounds (the reference's compute_bounding_box over the node's primitive boxes, bbox.h:27-39).
__global__ void k_lv_bounds(Level L, const uint32_t *__restrict__ idx, const double *__restrict__ lo,
                            const double *__restrict__ hi) {
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  LNode &nd = L.nodes[node];
  const uint32_t stop = block_stop(nd, start);
  double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (uint32_t pos = start + threadIdx.x; pos < stop; pos += blockDim.x) {
    const uint32_t p = idx[pos];
    for (int k = 0; k < 3; k++) {
      mn[k] = dmin(mn[k], lo[3ull * p + k]);
      mx[k] = dmax(mx[k], hi[3ull * p + k]);
    }
  }
  for (int off = 32; off > 0; off >>= 1)
    for (int k = 0; k < 3; k++) {
      mn[k] = dmin(mn[k], __shfl_xor(mn[k], off));
      mx[k] = dmax(mx[k], __shfl_xor(mx[k], off));
    }
  // one atomic per block and side: they serialise on a large node's six words (16 levels of 1.31M: 558 ->
  // 255 us)
  __shared__ double part[BLOCK / 64][6];
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 3; k++) {
      part[threadIdx.x / 64][k] = mn[k];
      part[threadIdx.x / 64][3 + k] = mx[k];
    }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = part[0][threadIdx.x];
    for (int w = 1; w < BLOCK / 64; w++) v = dmin(v, part[w][threadIdx.x]);
    atomicMin(&nd.klo[threadIdx.x], okey(v));
  } else if (threadIdx.x < 6) {
    double v = part[0][threadIdx.x];
    for (int w = 1; w < BLOCK / 64; w++) v = dmax(v, part[w][threadIdx.x]);
    atomicMax(&nd.khi[threadIdx.x - 3], okey(v));
  }
}

__global__ void k_lv_prep(Level L, uint32_t m, uint32_t min_leaf, uint32_t max_depth) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  LNode &nd = L.nodes[i];
  for (int k = 0; k < 3; k++) {
    nd.lo[k] = okey_value(nd.klo[k]);
    nd.hi[k] = okey_value(nd.khi[k]);
  }
  nd.leaf = (nd.n <= min_leaf || nd.depth >= max_depth) ? 1u : 0u;
}

// Binning (sort_collection_into_bins, binbuffer.h:67-91): per-block bins in LDS, merged into the node's bins.
__global__ void k_lv_bin(Level L, uint32_t nb, const uint32_t *__restrict__ idx, const double *__restrict__ lo,
                         const double *__restrict__ hi, const double *__restrict__ ctr) {
  __shared__ uint32_t scnt[3 * 64];
  __shared__ u64 sklo[3 * 64 * 3], skhi[3 * 64 * 3];
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  const LNode &nd = L.nodes[node];
  if (nd.leaf) return;
  const uint32_t stop = block_stop(nd, start);
  for (uint32_t t = threadIdx.x; t < 3 * nb; t += blockDim.x) {
    scnt[t] = 0;
    for (int k = 0; k < 3; k++) {
      sklo[3 * t + k] = okey(DBL_MAX);
      skhi[3 * t + k] = okey(-DBL_MAX);
    }
  }
  __syncthreads();
  double inv[3];
  for (int k = 0; k < 3; k++) {
    const double size = nd.hi[k] - nd.lo[k];
    inv[k] = (size > 0.0) ? 1.0 / size : 0.0;
  }
  const double scale = (double)(nb - 1);
  for (uint32_t pos = start + threadIdx.x; pos < stop; pos += blockDim.x) {
    const uint32_t p = idx[pos];
    u64 kl[3], kh[3];
    for (int k = 0; k < 3; k++) {
      kl[k] = okey(lo[3ull * p + k]);
      kh[k] = okey(hi[3ull * p + k]);
    }
    for (uint32_t j = 0; j < 3; j++) {
      const uint32_t t = j * nb + bin_of(((ctr[3ull * p + j] - nd.lo[j]) * inv[j]) * scale, nb - 1);
      atomicAdd(&scnt[t], 1u);
      for (int k = 0; k < 3; k++) {
        atomicMin(&sklo[3 * t + k], kl[k]);
        atomicMax(&skhi[3 * t + k], kh[k]);
      }
    }
  }
  __syncthreads();
  const size_t base = (size_t)node * 3 * nb;
  for (uint32_t t = threadIdx.x; t < 3 * nb; t += blockDim.x) {
    if (!scnt[t]) continue;
    atomicAdd(&L.bins.cnt[base + t], scnt[t]);
    for (int k = 0; k < 3; k++) {
      atomicMin(&L.bins.klo[3 * (base + t) + k], sklo[3 * t + k]);
      atomicMax(&L.bins.khi[3 * (base + t) + k], skhi[3 * t + k]);
    }
  }
}

// One wave per node.
__global__ void k_lv_sweep(Level L, uint32_t nb) {
  LNode &nd = L.nodes[blockIdx.x];
  if (nd.leaf) return;
  const size_t base = (size_t)blockIdx.x * 3 * nb;
  double cut[3];
  const uint32_t axis = sah_sweep(L.bins.cnt + base, L.bins.klo + 3 * base, L.bins.khi + 3 * base, nb, nd.lo, nd.hi,
                                  cut);
  if (threadIdx.x == 0) {
    nd.axis = axis;
    for (int k = 0; k < 3; k++) nd.cut[k] = cut[k];
  }
}

// Elements left of each axis's cut (the partition predicate center[axis] < cut[axis], builder.h:213-215).
__global__ void k_lv_count(Level L, const uint32_t *__restrict__ idx, const double *__restrict__ ctr) {
  __shared__ uint32_t sc[3];
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  LNode &nd = L.nodes[node];
  if (nd.leaf) return;
  const uint32_t stop = block_stop(nd, start);
  if (threadIdx.x < 3) sc[threadIdx.x] = 0;
  __syncthreads();
  uint32_t c[3] = {0, 0, 0};
  for (uint32_t pos = start + threadIdx.x; pos < stop; pos += blockDim.x) {
    const uint32_t p = idx[pos];
    for (int j = 0; j < 3; j++) c[j] += (ctr[3ull * p + j] < nd.cut[j]) ? 1u : 0u;
  }
  for (int j = 0; j < 3; j++)
    if (c[j]) atomicAdd(&sc[j], c[j]);
  __syncthreads();
  if (threadIdx.x < 3 && sc[threadIdx.x]) atomicAdd(&nd.cnt3[threadIdx.x], sc[threadIdx.x]);
}

// The builder's three partition attempts (blazert/bvh/builder.h:210-223): a partition that leaves one side
// empty changes nothing, falls back to the middle and moves on to the next axis.
__global__ void k_lv_decide(Level L, uint32_t m) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  LNode &nd = L.nodes[i];
  if (nd.leaf) return;
  uint32_t axis = nd.axis, mid = nd.begin, bad = 0, split = 0;
  for (int a = 0; a < 3; a++) {
    const uint32_t T = nd.cnt3[axis];
    if (T == 0 || T == nd.n) {
      bad++;
      mid = nd.begin + (nd.n >> 1);
      axis = (axis + 1) % 3;
    } else {
      mid = nd.begin + T;
      split = 1;
      break;
    }
  }
  nd.axis = axis;
  nd.mid = mid;
  nd.bad = bad;
  nd.split = split;
}

__device__ __forceinline__ bool left_of_cut(const LNode &nd, const uint32_t *idx, const double *ctr, uint32_t pos) {
  return ctr[3ull * idx[pos] + nd.axis] < nd.cut[nd.axis];
}

// Per block: elements on the wrong side (left part failing, right part passing).
__global__ void k_lv_rank1(Level L, const uint32_t *__restrict__ idx, const double *__restrict__ ctr) {
  __shared__ uint32_t s[2];
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  const LNode &nd = L.nodes[node];
  if (nd.leaf || !nd.split) return;
  const uint32_t stop = block_stop(nd, start);
  if (threadIdx.x < 2) s[threadIdx.x] = 0;
  __syncthreads();
  uint32_t cl = 0, cr = 0;
  for (uint32_t pos = start + threadIdx.x; pos < stop; pos += blockDim.x) {
    const bool pass = left_of_cut(nd, idx, ctr, pos);
    cl += (pos < nd.mid && !pass) ? 1u : 0u;
    cr += (pos >= nd.mid && pass) ? 1u : 0u;
  }
  if (cl) atomicAdd(&s[0], cl);
  if (cr) atomicAdd(&s[1], cr);
  __syncthreads();
  if (threadIdx.x == 0) {
    L.blk_l[blockIdx.x] = s[0];
    L.blk_r[blockIdx.x] = s[1];
  }
}

// Per node: block offsets of the misplaced counts, a wave's scan (one thread walking a large node's blocks: 276 us for
// 16 levels of 1.31M, 75 us this way).
__global__ void __launch_bounds__(64) k_lv_rank2(Level L) {
  LNode &nd = L.nodes[blockIdx.x];
  if (nd.leaf || !nd.split) return;
  const uint32_t lane = threadIdx.x;
  uint32_t sl = 0, sr = 0;
  for (uint32_t base = 0; base < nd.nblk; base += 64u) {
    const uint32_t b = nd.blk0 + base + lane;
    const bool in = base + lane < nd.nblk;
    const uint32_t l = in ? L.blk_l[b] : 0u, r = in ? L.blk_r[b] : 0u;
    uint32_t pl = l, pr = r;  // inclusive sums
    for (uint32_t off = 1; off < 64u; off <<= 1) {
      const uint32_t ul = __shfl_up(pl, off), ur = __shfl_up(pr, off);
      if (lane >= off) {
        pl += ul;
        pr += ur;
      }
    }
    if (in) {
      L.off_l[b] = sl + pl - l;
      L.off_r[b] = sr + pr - r;
    }
    sl += __shfl(pl, 63);
    sr += __shfl(pr, 63);
  }
  if (lane == 0) nd.misplaced = sr;
}

// Positions of the right part's passing elements, indexed by their rank from the right end.
__global__ void k_lv_rank3(Level L, const uint32_t *__restrict__ idx, const double *__restrict__ ctr,
                           uint32_t *__restrict__ pos_r) {
  __shared__ uint32_t wt[BLOCK / 64];
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  const LNode &nd = L.nodes[node];
  if (nd.leaf || !nd.split) return;
  const uint32_t stop = block_stop(nd, start);
  uint32_t run = L.off_r[blockIdx.x];
  for (uint32_t base = start; base < stop; base += blockDim.x) {
    const uint32_t pos = base + threadIdx.x;
    const bool f = pos < stop && pos >= nd.mid && left_of_cut(nd, idx, ctr, pos);
    uint32_t tot;
    const uint32_t r = block_rank(f, wt, tot);
    if (f) pos_r[nd.begin + (nd.misplaced - 1u - (run + r))] = pos;
    run += tot;
  }
}

// The swaps: the r-th failing element of the left part trades places with the r-th passing element of the right
// part counted from the right end. Only left-part positions are read here, each by the one thread that swaps it.
__global__ void k_lv_swap(Level L, uint32_t *__restrict__ idx, const double *__restrict__ ctr,
                          const uint32_t *__restrict__ pos_r) {
  __shared__ uint32_t wt[BLOCK / 64];
  const uint32_t node = L.blk_node[blockIdx.x], start = L.blk_start[blockIdx.x];
  const LNode &nd = L.nodes[node];
  if (nd.leaf || !nd.split) return;
  const uint32_t stop = block_stop(nd, start);
  uint32_t run = L.off_l[blockIdx.x];
  for (uint32_t base = start; base < stop; base += blockDim.x) {
    const uint32_t pos = base + threadIdx.x;
    const bool f = pos < stop && pos < nd.mid && !left_of_cut(nd, idx, ctr, pos);
    uint32_t tot;
    const uint32_t r = block_rank(f, wt, tot);
    if (f) {
      const uint32_t partner = pos_r[nd.begin + run + r];
      const uint32_t a = idx[pos];
      idx[pos] = idx[partner];
      idx[partner] = a;
    }
    run += tot;
  }
}

// ------------------------------------------------------------------------------------------------ small subtrees
struct SmallRoot {
  uint32_t begin, n, depth, left;  // left: left turns on the path from the tree's root
};

struct BuildStatsDev {
  uint32_t max_depth, bad, max_prims, min_prims;
};
__device__ __forceinline__ void add_stats(BuildStatsDev &a, const BuildStatsDev &b) {
  a.max_depth = a.max_depth > b.max_depth ? a.max_depth : b.max_depth;
  a.bad += b.bad;
  a.max_prims = a.max_prims > b.max_prims ? a.max_prims : b.max_prims;
  a.min_prims = a.min_prims < b.min_prims ? a.min_prims : b.min_prims;
}

// A node before it has its number: internal nodes are kept at the position that parts their children, which no two share,
// leaves at their first position.
struct RawNode {
  double lo[3], hi[3];
  uint32_t begin;
  uint32_t info;  // internal: split axis; leaf: primitives
  uint32_t left;  // left turns on the path from the root
  uint32_t pad;
};
static_assert(sizeof(RawNode) == 64, "RawNode size");
struct RawTree {
  RawNode *inner, *leaf;
  uint32_t *is_inner, *is_leaf;  // 0 / 1 per position
};

// One wave splits the nodes of more than TINY primitives of a small subtree depth first (build_recursive,
// blazert/bvh/builder.h:85-115), its primitives' boxes and centers staged in LDS and permuted through an LDS index array.
// The subtrees of at most TINY primitives that remain are listed at tiny[R.begin ...], their number in num_tiny.
__global__ void __launch_bounds__(64) k_small(const SmallRoot *__restrict__ roots, uint32_t *__restrict__ idx,
                                              const double *__restrict__ lo, const double *__restrict__ hi,
                                              const double *__restrict__ ctr, uint32_t nb, uint32_t min_leaf,
                                              uint32_t max_depth, RawTree raw, SmallRoot *__restrict__ tiny,
                                              uint32_t *__restrict__ num_tiny, BuildStatsDev *__restrict__ stats) {
  __shared__ uint32_t e_idx[SMALL];
  __shared__ double e_lo[3][SMALL], e_hi[3][SMALL], e_ctr[3][SMALL];
  __shared__ uint16_t perm[SMALL];
  __shared__ uint16_t pos_r[SMALL / 2];
  __shared__ uint32_t bcnt[3 * 64];
  __shared__ u64 bklo[3 * 64 * 3], bkhi[3 * 64 * 3];
  __shared__ uint32_t stk[STACK][4];

  const SmallRoot R = roots[blockIdx.x];
  const uint32_t lane = threadIdx.x;
  BuildStatsDev st{0, 0, 0, 0xFFFFFFFFu};
  if (R.n <= TINY) {
    if (lane == 0) {
      tiny[R.begin] = R;
      num_tiny[blockIdx.x] = 1;
      stats[blockIdx.x] = st;
    }
    return;
  }
  for (uint32_t k = lane; k < R.n; k += 64) {
    const uint32_t p = idx[R.begin + k];
    e_idx[k] = p;
    for (int c = 0; c < 3; c++) {
      e_lo[c][k] = lo[3ull * p + c];
      e_hi[c][k] = hi[3ull * p + c];
      e_ctr[c][k] = ctr[3ull * p + c];
    }
    perm[k] = (uint16_t)k;
  }
  if (lane == 0) {
    stk[0][0] = 0;
    stk[0][1] = R.n;
    stk[0][2] = R.depth;
    stk[0][3] = R.left;
  }
  __syncthreads();
  uint32_t sp = 1, tinies = 0;
  while (sp > 0) {
    sp--;
    const uint32_t b = stk[sp][0], e = stk[sp][1], d = stk[sp][2], left = stk[sp][3];
    __syncthreads();
    const uint32_t n = e - b;
    // bounds
    double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (uint32_t k = b + lane; k < e; k += 64) {
      const uint32_t q = perm[k];
      for (int c = 0; c < 3; c++) {
        mn[c] = dmin(mn[c], e_lo[c][q]);
        mx[c] = dmax(mx[c], e_hi[c][q]);
      }
    }
    for (int off = 32; off > 0; off >>= 1)
      for (int c = 0; c < 3; c++) {
        mn[c] = dmin(mn[c], __shfl_xor(mn[c], off));
        mx[c] = dmax(mx[c], __shfl_xor(mx[c], off));
      }
    st.max_depth = d > st.max_depth ? d : st.max_depth;
    RawNode node{{mn[0], mn[1], mn[2]}, {mx[0], mx[1], mx[2]}, R.begin + b, n, left, 0};
    if (n <= min_leaf || d >= max_depth) {
      st.max_prims = n > st.max_prims ? n : st.max_prims;
      st.min_prims = n < st.min_prims ? n : st.min_prims;
      if (lane == 0) {
        raw.leaf[R.begin + b] = node;
        raw.is_leaf[R.begin + b] = 1u;
      }
      continue;
    }
    // binning
    for (uint32_t t = lane; t < 3 * nb; t += 64) {
      bcnt[t] = 0;
      for (int k = 0; k < 3; k++) {
        bklo[3 * t + k] = okey(DBL_MAX);
        bkhi[3 * t + k] = okey(-DBL_MAX);
      }
    }
    __syncthreads();
    double inv[3];
    for (int k = 0; k < 3; k++) {
      const double size = mx[k] - mn[k];
      inv[k] = (size > 0.0) ? 1.0 / size : 0.0;
    }
    const double scale = (double)(nb - 1);
    for (uint32_t k = b + lane; k < e; k += 64) {
      const uint32_t q = perm[k];
      for (uint32_t j = 0; j < 3; j++) {
        const uint32_t t = j * nb + bin_of(((e_ctr[j][q] - mn[j]) * inv[j]) * scale, nb - 1);
        atomicAdd(&bcnt[t], 1u);
        for (int c = 0; c < 3; c++) {
          atomicMin(&bklo[3 * t + c], okey(e_lo[c][q]));
          atomicMax(&bkhi[3 * t + c], okey(e_hi[c][q]));
        }
      }
    }
    __syncthreads();
    double cut[3];
    uint32_t axis = sah_sweep(bcnt, bklo, bkhi, nb, mn, mx, cut);
    // partition attempts
    uint32_t mid = b;
    bool split = false;
    for (int a = 0; a < 3; a++) {
      uint32_t T = 0;
      for (uint32_t base = b; base < e; base += 64) {
        const uint32_t k = base + lane;
        T += (uint32_t)__popcll(__ballot(k < e && e_ctr[axis][perm[k]] < cut[axis]));
      }
      if (T == 0 || T == n) {
        st.bad++;
        mid = b + (n >> 1);
        axis = (axis + 1) % 3;
      } else {
        mid = b + T;
        split = true;
        break;
      }
    }
    if (split) {
      const double c = cut[axis];
      uint32_t run = 0;
      for (uint32_t base = mid; base < e; base += 64) {
        const uint32_t k = base + lane;
        const bool f = k < e && e_ctr[axis][perm[k]] < c;
        const u64 msk = __ballot(f);
        if (f) pos_r[run + (uint32_t)__popcll(msk & ((1ull << lane) - 1ull))] = (uint16_t)k;
        run += (uint32_t)__popcll(msk);
      }
      __syncthreads();
      const uint32_t misplaced = run;
      run = 0;
      for (uint32_t base = b; base < mid; base += 64) {
        const uint32_t k = base + lane;
        const bool f = k < mid && !(e_ctr[axis][perm[k]] < c);
        const u64 msk = __ballot(f);
        if (f) {
          const uint32_t r = run + (uint32_t)__popcll(msk & ((1ull << lane) - 1ull));
          const uint32_t partner = pos_r[misplaced - 1u - r];
          const uint16_t x = perm[k];
          perm[k] = perm[partner];
          perm[partner] = x;
        }
        run += (uint32_t)__popcll(msk);
      }
      __syncthreads();
    }
    node.info = axis;
    if (lane == 0) {
      raw.inner[R.begin + mid] = node;
      raw.is_inner[R.begin + mid] = 1u;
    }
    for (int c = 1; c >= 0; c--) {
      const uint32_t cb = c ? mid : b, ce = c ? e : mid, cl = c ? left : left + 1u;
      if (ce - cb <= TINY) {
        if (lane == 0) tiny[R.begin + tinies] = SmallRoot{R.begin + cb, ce - cb, d + 1, cl};
        tinies++;
      } else {
        if (lane == 0) {
          stk[sp][0] = cb;
          stk[sp][1] = ce;
          stk[sp][2] = d + 1;
          stk[sp][3] = cl;
        }
        sp++;
      }
    }
    __syncthreads();
  }
  for (uint32_t k = lane; k < R.n; k += 64) idx[R.begin + k] = e_idx[perm[k]];
  if (lane == 0) {
    num_tiny[blockIdx.x] = tinies;
    stats[blockIdx.x] = st;
  }
}

// The lists of the small subtrees' waves, one after the other.
__global__ void k_tiny_list(const SmallRoot *__restrict__ roots, const uint32_t *__restrict__ num_tiny,
                            const uint32_t *__restrict__ at, const SmallRoot *__restrict__ tiny,
                            SmallRoot *__restrict__ list) {
  const uint32_t r = blockIdx.x;
  for (uint32_t k = threadIdx.x; k < num_tiny[r]; k += blockDim.x) list[at[r] + k] = tiny[roots[r].begin + k];
}

// Rotates a value by one lane within the row of 16.
__device__ __forceinline__ uint32_t row_next(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xf, 0xf, false);
}
__device__ __forceinline__ double row_next(double x) {
  const u64 b = (u64)__double_as_longlong(x);
  return __longlong_as_double((long long)(((u64)row_next((uint32_t)(b >> 32)) << 32) | row_next((uint32_t)b)));
}

// Subtrees of at most TINY primitives, four per wave: a row of 16 lanes holds one primitive per lane and splits all nodes of
// a level at once, each lane seeing the others of its node as their values rotate through the row. A bin boundary that
// can be chosen is one after an occupied bin (the boundaries behind empty bins cost the same and come later), so every lane
// evaluates the one after its own bin, on each axis. The primitives stay in their lanes; `pos` is the order.
__global__ void __launch_bounds__(256) k_tiny(const SmallRoot *__restrict__ list, const uint32_t *__restrict__ total,
                                              uint32_t *__restrict__ idx, const double *__restrict__ lo,
                                              const double *__restrict__ hi, const double *__restrict__ ctr, uint32_t nb,
                                              uint32_t min_leaf, uint32_t max_depth, RawTree raw,
                                              BuildStatsDev *__restrict__ stats) {
  using exact::max_nn;
  using exact::min_nn;
  const uint32_t lane = threadIdx.x & 63u, in_row = lane & 15u;
  const uint32_t waves = gridDim.x * (blockDim.x >> 6), wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint32_t count = *total;
  const double scale = (double)(nb - 1);
  constexpr uint32_t GONE = 0xFFu;
  BuildStatsDev st{0, 0, 0, 0xFFFFFFFFu};
  for (uint32_t first = 4u * wave; first < count; first += 4u * waves) {  // wave-uniform
    const uint32_t g = first + (lane >> 4);
    const SmallRoot R = g < count ? list[g] : SmallRoot{0, 0, 0, 0};
    const bool mine = in_row < R.n;
    const uint32_t prim = mine ? idx[R.begin + in_row] : 0u;
    double l[3], h[3], c[3];
    for (int k = 0; k < 3; k++) {
      l[k] = mine ? lo[3ull * prim + k] : 0.0;
      h[k] = mine ? hi[3ull * prim + k] : 0.0;
      c[k] = mine ? ctr[3ull * prim + k] : 0.0;
    }
    uint32_t node = mine ? 0u : GONE;  // first position of this lane's node in the subtree
    uint32_t size = R.n, depth = R.depth, left = R.left, pos = in_row;
    while (__ballot(node != GONE)) {
      // bounds of the node
      double mn[3], mx[3];
      {
        double ol[3], oh[3];
        uint32_t on = node;
        for (int k = 0; k < 3; k++) {
          ol[k] = mn[k] = l[k];
          oh[k] = mx[k] = h[k];
        }
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          on = row_next(on);
          const bool same = on == node;
#pragma unroll
          for (int k = 0; k < 3; k++) {
            ol[k] = row_next(ol[k]);
            oh[k] = row_next(oh[k]);
            mn[k] = min_nn(mn[k], same ? ol[k] : mn[k]);
            mx[k] = max_nn(mx[k], same ? oh[k] : mx[k]);
          }
        }
      }
      if (node != GONE) st.max_depth = depth > st.max_depth ? depth : st.max_depth;
      if (node != GONE && (size <= min_leaf || depth >= max_depth)) {
        if (pos == node) {
          const uint32_t at = R.begin + node;
          raw.leaf[at] = RawNode{{mn[0], mn[1], mn[2]}, {mx[0], mx[1], mx[2]}, at, size, left, 0};
          raw.is_leaf[at] = 1u;
          st.max_prims = size > st.max_prims ? size : st.max_prims;
          st.min_prims = size < st.min_prims ? size : st.min_prims;
        }
        node = GONE;
      }
      if (!__ballot(node != GONE)) break;
      // bins of the three axes, packed
      uint32_t bins = 0;
      double step[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double len = mx[k] - mn[k];
        const double inv = (len > 0.0) ? 1.0 / len : 0.0;
        bins |= bin_of(((c[k] - mn[k]) * inv) * scale, nb - 1) << (8 * k);
        step[k] = len / (double)nb;
      }
      // the cost of the boundary after this lane's bin, and the node's least one with its first bin
      double cost[3];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        double ll[3], lh[3], rl[3], rh[3];
        uint32_t nl = 1, nr = 0;
        double ol[3], oh[3];
        uint32_t on = node, ob = (bins >> (8 * j)) & 255u;
        const uint32_t mine_b = ob;
        for (int k = 0; k < 3; k++) {
          ll[k] = ol[k] = l[k];
          lh[k] = oh[k] = h[k];
          rl[k] = DBL_MAX;
          rh[k] = -DBL_MAX;
        }
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          on = row_next(on);
          ob = row_next(ob);
          const bool same = on == node, is_l = same && ob <= mine_b, is_r = same && ob > mine_b;
          nl += is_l ? 1u : 0u;
          nr += is_r ? 1u : 0u;
#pragma unroll
          for (int k = 0; k < 3; k++) {
            ol[k] = row_next(ol[k]);
            oh[k] = row_next(oh[k]);
            ll[k] = min_nn(ll[k], is_l ? ol[k] : DBL_MAX);
            lh[k] = max_nn(lh[k], is_l ? oh[k] : -DBL_MAX);
            rl[k] = min_nn(rl[k], is_r ? ol[k] : DBL_MAX);
            rh[k] = max_nn(rh[k], is_r ? oh[k] : -DBL_MAX);
          }
        }
        const double x = (double)nl * surface(ll, lh) + (double)nr * surface(rl, rh);
        cost[j] = (nr > 0u && x < DBL_MAX) ? x : __builtin_inf();  // an empty right side costs NaN in the sweep
      }
      double cut[3], least[3];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        double m = cost[j], oc = cost[j];
        uint32_t mb = (bins >> (8 * j)) & 255u, ob = mb, on = node;
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          on = row_next(on);
          ob = row_next(ob);
          oc = row_next(oc);
          const bool take = on == node && (oc < m || (oc == m && ob < mb));
          m = take ? oc : m;
          mb = take ? ob : mb;
        }
        const bool any = m < DBL_MAX;
        least[j] = any ? m : DBL_MAX;
        cut[j] = (double)(any ? mb + 1u : 1u) * step[j] + mn[j];
      }
      uint32_t axis = 0;
      if (least[0] > least[1]) axis = 1;
      if ((axis ? least[1] : least[0]) > least[2]) axis = 2;
      // elements left of each axis's cut, counted over the node (packed), and the partition attempts
      const uint32_t pass3 = (c[0] < cut[0] ? 1u : 0u) | (c[1] < cut[1] ? 0x100u : 0u) | (c[2] < cut[2] ? 0x10000u : 0u);
      uint32_t T3 = pass3;
      {
        uint32_t on = node, op = pass3;
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          on = row_next(on);
          op = row_next(op);
          T3 += on == node ? op : 0u;
        }
      }
      uint32_t mid = 0, bad = 0;  // mid: within the node
      bool split = false;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        if (!split) {
          const uint32_t T = (T3 >> (8 * axis)) & 255u;
          if (T == 0 || T == size) {
            bad++;
            mid = size >> 1;
            axis = axis == 2 ? 0u : axis + 1u;
          } else {
            mid = T;
            split = true;
          }
        }
      }
      // the r-th failing element of the left part trades places with the r-th passing one of the right part from the end
      const bool pass = ((pass3 >> (8 * axis)) & 1u) != 0u;
      const uint32_t at = pos - node;
      const bool out_l = split && at < mid && !pass, out_r = split && at >= mid && pass;
      // tag: 0 in place, else side (1 left, 2 right); rank among the misplaced of the side
      const uint32_t side = node == GONE ? 0u : out_l ? 1u : out_r ? 2u : 0u;
      uint32_t rank = 0;
      {
        uint32_t o = (node << 16) | (side << 8) | pos;
        const uint32_t self = o;
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          o = row_next(o);
          const bool same = (o & 0xFFFFFF00u) == (self & 0xFFFFFF00u);
          const uint32_t op = o & 255u;
          rank += same && (side == 1u ? op < pos : op > pos) ? 1u : 0u;
        }
      }
      uint32_t to = pos;
      {
        uint32_t o = (node << 24) | (side << 16) | (rank << 8) | pos;
        const uint32_t want = (node << 24) | ((3u - side) << 16) | (rank << 8);
#pragma unroll 1
        for (int r = 1; r < 16; r++) {
          o = row_next(o);
          if (side && (o & 0xFFFFFF00u) == want) to = o & 255u;
        }
      }
      if (node != GONE) {
        if (pos == node) {
          raw.inner[R.begin + node + mid] =
              RawNode{{mn[0], mn[1], mn[2]}, {mx[0], mx[1], mx[2]}, R.begin + node, axis, left, 0};
          raw.is_inner[R.begin + node + mid] = 1u;
          st.bad += bad;
        }
        pos = to;
        const bool right = pos - node >= mid;
        node = right ? node + mid : node;
        size = right ? size - mid : mid;
        left += right ? 0u : 1u;
        depth++;
      }
    }
    if (mine) idx[R.begin + pos] = prim;
  }
  for (int off = 32; off > 0; off >>= 1) {
    BuildStatsDev o;
    o.max_depth = __shfl_xor(st.max_depth, off);
    o.bad = __shfl_xor(st.bad, off);
    o.max_prims = __shfl_xor(st.max_prims, off);
    o.min_prims = __shfl_xor(st.min_prims, off);
    add_stats(st, o);
  }
  if (lane == 0) stats[wave] = st;
}

// One block: the waves' statistics added up into stats[0].
__global__ void k_sum_stats(BuildStatsDev *stats, uint32_t n) {
  __shared__ BuildStatsDev part[256];
  BuildStatsDev st{0, 0, 0, 0xFFFFFFFFu};
  for (uint32_t i = threadIdx.x; i < n; i += 256) add_stats(st, stats[i]);
  part[threadIdx.x] = st;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 256; i++) add_stats(st, part[i]);
    stats[0] = st;
  }
}

// ------------------------------------------------------------------------------------------------ assembly
struct RawPut {
  RawNode node;
  uint32_t at, leaf;
};

__global__ void k_put_raw(const RawPut *__restrict__ puts, uint32_t m, RawTree raw) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const RawPut p = puts[i];
  if (p.leaf) {
    raw.leaf[p.at] = p.node;
    raw.is_leaf[p.at] = 1u;
  } else {
    raw.inner[p.at] = p.node;
    raw.is_inner[p.at] = 1u;
  }
}

// Writes every node at its number. before[p]: leaves that begin before position p; ni: number among the internal nodes.
__global__ void k_emit(RawTree raw, uint32_t n, const uint32_t *__restrict__ before, brt_tree_node *__restrict__ tree,
                       uint32_t *__restrict__ ni) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  if (raw.is_leaf[p]) {
    const RawNode r = raw.leaf[p];
    brt_tree_node t;
    for (int k = 0; k < 3; k++) {
      t.min[k] = r.lo[k];
      t.max[k] = r.hi[k];
    }
    t.leaf = 1;
    t.axis = t.children[0] = t.children[1] = INVALID_ID;
    t.prim_begin = p;
    t.prim_count = r.info;
    const uint32_t i = 2u * before[p] + r.left;
    tree[i] = t;
    ni[i] = 0;
  }
  if (raw.is_inner[p]) {
    const RawNode r = raw.inner[p];
    brt_tree_node t;
    for (int k = 0; k < 3; k++) {
      t.min[k] = r.lo[k];
      t.max[k] = r.hi[k];
    }
    const uint32_t b = before[r.begin], i = 2u * b + r.left;
    t.leaf = 0;
    t.axis = r.info;
    t.children[0] = i + 1u;
    t.children[1] = 2u * before[p] + r.left;
    t.prim_begin = t.prim_count = 0;
    tree[i] = t;
    ni[i] = b + r.left;
  }
}

// ------------------------------------------------------------------------------------------------ flatten
// Every internal node becomes one Node64 (numbered in pre-order among internal nodes). The root and every internal
// slot of a record (collapse4) become one Node4 each, numbered as the host's depth-first allocation does: a Node4's
// internal slots get consecutive indices when it is processed, and Node4s are processed in pre-order, so slot r of
// node P gets 1 + (internal slots of all Node4s before P) + r.

// is_root[i] = 1 when internal node i roots a Node4. A node's status depends on the records above it, so each
// thread walks from the root down to its node: in pre-order the left subtree of v is [v + 1, right child), and on
// the way the current record's slots tell whether the next node starts a record or lies inside the current one.
__global__ void k_roots4(const brt_tree_node *__restrict__ T, uint32_t M, uint32_t *__restrict__ is_root) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  uint32_t root = 0;
  if (i > 0 && !T[i].leaf) {
    uint32_t slot[4];
    int m = collapse4(T, 0, slot);
    uint32_t v = 0;
    // every step descends one level towards i, which lies below v, so v never is a leaf here and the loop ends
    // within the tree's depth (at most 63); the bound and the leaf test only guard the reads
    for (int level = 0; level < 64 && !T[v].leaf; level++) {
      const uint32_t right = T[v].children[1];
      v = (i >= right) ? right : T[v].children[0];
      bool is_slot = false;
      for (int c = 0; c < m; c++) is_slot = is_slot || slot[c] == v;
      if (v == i) {
        root = is_slot ? 1u : 0u;
        break;
      }
      if (is_slot) m = collapse4(T, v, slot);
    }
  } else if (i == 0) {
    root = T[0].leaf ? 0u : 1u;
  }
  is_root[i] = root;
}

__global__ void k_flags(const brt_tree_node *__restrict__ T, const uint32_t *__restrict__ is_root, uint32_t M,
                        uint32_t *__restrict__ islots) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  uint32_t s = 0;
  if (is_root[i]) {
    uint32_t slot[4];
    const int m = collapse4(T, i, slot);
    for (int c = 0; c < m; c++) s += T[slot[c]].leaf ? 0u : 1u;
  }
  islots[i] = s;
}

__global__ void k_assign4(const brt_tree_node *__restrict__ T, const uint32_t *__restrict__ is_root, uint32_t M,
                          const uint32_t *__restrict__ S, uint32_t *__restrict__ k4) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M || !is_root[i]) return;
  if (i == 0) k4[0] = 0;
  uint32_t slot[4];
  const int m = collapse4(T, i, slot);
  uint32_t r = 0;
  for (int c = 0; c < m; c++)
    if (!T[slot[c]].leaf) k4[slot[c]] = 1u + S[i] + r++;
}

__global__ void k_node64(const brt_tree_node *__restrict__ T, uint32_t M, const uint32_t *__restrict__ ni,
                         Node64 *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M || T[i].leaf) return;
  Node64 a;
  for (int c = 0; c < 2; c++) {
    const uint32_t chi = T[i].children[c];
    const brt_tree_node &ch = T[chi];
    for (int k = 0; k < 3; k++) {
      a.b[6 * c + k] = ch.min[k];
      a.b[6 * c + 3 + k] = ch.max[k];
    }
    a.ref[c] = ch.leaf ? (LEAF_BIT | ch.prim_begin) : ni[chi];
    a.cnt[c] = ch.leaf ? ch.prim_count : 0u;
  }
  a.cnt[1] |= T[i].axis << AXIS_SHIFT;
  for (int k = 0; k < 4; k++) a.pad[k] = 0;
  out[ni[i]] = a;
}

__global__ void k_node4(const brt_tree_node *__restrict__ T, const uint32_t *__restrict__ is_root, uint32_t M,
                        const uint32_t *__restrict__ k4, Node4 *__restrict__ out, uint32_t *__restrict__ ord4) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M || !is_root[i]) return;
  uint32_t slot[4], axis[16] = {};
  const int m = collapse4(T, i, slot, axis);
  uint32_t ord[2];
  visit_order4(axis, m, ord);
  ord4[2ull * k4[i]] = ord[0];
  ord4[2ull * k4[i] + 1] = ord[1];
  Node4 nd;
  for (int c = 0; c < 4; c++) {
    for (int k = 0; k < 3; k++) {
      nd.lo[k][c] = __builtin_inff();
      nd.hi[k][c] = -__builtin_inff();
    }
    nd.ref[c] = 0;
    nd.cnt[c] = EMPTY_SLOT;
  }
  for (int c = 0; c < m; c++) {
    const brt_tree_node &sn = T[slot[c]];
    for (int k = 0; k < 3; k++) {
      nd.lo[k][c] = f32_down(sn.min[k]);
      nd.hi[k][c] = f32_up(sn.max[k]);
    }
    nd.ref[c] = sn.leaf ? (LEAF_BIT | sn.prim_begin) : k4[slot[c]];
    nd.cnt[c] = sn.leaf ? sn.prim_count : 0u;
  }
  out[k4[i]] = nd;
}

// Primitive records in leaf order (the host flatten's record loops).
__global__ void k_tri_recs(const uint32_t *__restrict__ order, const double *__restrict__ V,
                           const uint32_t *__restrict__ F, uint32_t n, TriRec *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = order[i];
  const double *v0 = V + 3ull * F[3ull * p], *v1 = V + 3ull * F[3ull * p + 1], *v2 = V + 3ull * F[3ull * p + 2];
  TriRec r;
  for (int k = 0; k < 3; k++) {
    r.v0[k] = v0[k];
    r.e1[k] = v0[k] - v1[k];
    r.e2[k] = v2[k] - v0[k];
  }
  r.prim = p;
  out[i] = r;
}

__global__ void k_sph_recs(const uint32_t *__restrict__ order, const double *__restrict__ c,
                           const double *__restrict__ rad, uint32_t n, SphRec *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = order[i];
  SphRec r;
  for (int k = 0; k < 3; k++) r.c[k] = c[3ull * p + k];
  r.r = rad[p];
  out[i] = r;
}

__global__ void k_pla_recs(const uint32_t *__restrict__ order, const double *__restrict__ c,
                           const double *__restrict__ dx, const double *__restrict__ dy,
                           const double *__restrict__ R, uint32_t n, PlaRec *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = order[i];
  PlaRec r;
  for (int k = 0; k < 3; k++) r.c[k] = c[3ull * p + k];
  r.dx = dx[p];
  r.dy = dy[p];
  for (int k = 0; k < 9; k++) r.R[k] = R[9ull * p + k];
  r.pad[0] = r.pad[1] = 0.0;
  out[i] = r;
}

__global__ void k_cyl_recs(const uint32_t *__restrict__ order, const double *__restrict__ c,
                           const double *__restrict__ a, const double *__restrict__ b, const double *__restrict__ h,
                           const double *__restrict__ R, uint32_t n, CylRec *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = order[i];
  CylRec r;
  for (int k = 0; k < 3; k++) r.c[k] = c[3ull * p + k];
  r.a = a[p];
  r.b = b[p];
  r.h = h[p];
  for (int k = 0; k < 9; k++) r.R[k] = R[9ull * p + k];
  r.pad = 0.0;
  out[i] = r;
}

// ------------------------------------------------------------------------------------------------ host driver
inline uint32_t blocks_for(uint64_t n, uint32_t t) { return (uint32_t)((n + t - 1) / t); }

// Device allocations of one build; temporaries go back to the pool in the destructor (after the build's stream has
// drained, also on an error path), results are handed over.
struct Arena {
  hipStream_t stream;
  int device = -1;
  std::vector<void *> ptrs;
  hipError_t err = hipSuccess;
  explicit Arena(hipStream_t s) : stream(s) { err = hipGetDevice(&device); }
  template <class T>
  T *get(size_t count) {
    if (err != hipSuccess) return nullptr;
    void *p = nullptr;
    err = pool_get(device, std::max<size_t>(count, 1) * sizeof(T), &p);
    if (err != hipSuccess) return nullptr;
    ptrs.push_back(p);
    return static_cast<T *>(p);
  }
  void release(void *p) {
    for (auto &q : ptrs)
      if (q == p) q = nullptr;
  }
  ~Arena() {
    const bool idle = hipStreamSynchronize(stream) == hipSuccess;
    for (void *p : ptrs)
      if (p) pool_put(device, p, idle);
  }
};

template <class T>
hipError_t to_device(Arena &A, const T *host, size_t count, const T **dst, hipStream_t st) {
  *dst = nullptr;
  if (!count) return hipSuccess;
  T *d = A.get<T>(count);
  if (!d) return A.err;
  *dst = d;
  return hipMemcpyAsync(d, host, count * sizeof(T), hipMemcpyHostToDevice, st);
}

struct HostTop {
  uint32_t begin, n, depth, left;
};

}  // namespace

// Each failing step records its source line in out.failed_line.
#define BRT_CHECK(x)                 \
  do {                               \
    const hipError_t e_ = (x);       \
    if (e_ != hipSuccess) {          \
      out.failed_line = __LINE__;    \
      return e_;                     \
    }                                \
  } while (0)
#define BRT_LAUNCH(...)           \
  do {                            \
    __VA_ARGS__;                  \
    BRT_CHECK(hipGetLastError()); \
  } while (0)

bool device_build_supported(uint32_t nbins, uint32_t max_depth) { return nbins >= 2 && nbins <= 64 && max_depth <= 62; }

hipError_t device_build(const DeviceBuildIn &in, DeviceBuildOut &out, hipStream_t st) {
  out = DeviceBuildOut{};
  const uint32_t n = in.n, nb = in.nbins;
  if (n == 0 || !device_build_supported(nb, in.max_depth)) return hipErrorInvalidValue;
  BRT_CHECK(hipGetLastError());  // an error left by earlier work is reported as such, not as this build's
  Arena A(st);
  // primitive boxes and centers
  double *lo = A.get<double>(3ull * n), *hi = A.get<double>(3ull * n), *ctr = A.get<double>(3ull * n);
  uint32_t *idx = A.get<uint32_t>(n), *pos_r = A.get<uint32_t>(n);
  BRT_CHECK(A.err);
  MeshFlags *d_flags = nullptr, hflags{};
  double *vnormals = nullptr;
  if (in.type == TRIANGLES) {
    const uint32_t nv = in.num_vertices, corners = 3u * n;
    double *fn3 = A.get<double>(3ull * n);
    // fans and their running ends (the scan's extra element), corner places, the list of long fans
    uint32_t *fan = A.get<uint32_t>(nv + 1ull), *start = A.get<uint32_t>(nv + 1ull), *at = A.get<uint32_t>(corners);
    uint32_t *longs = A.get<uint32_t>(corners / FAN_SHORT + 1);
    d_flags = A.get<MeshFlags>(1);
    vnormals = A.get<double>(3ull * nv);
    size_t tb = 0;
    BRT_CHECK(A.err);
    BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, fan, start, (int)(nv + 1), st));
    unsigned char *tmp_scan = A.get<unsigned char>(tb);
    BRT_CHECK(A.err);
    BRT_LAUNCH(k_zero_words<<<blocks_for(nv + 1ull, 256), 256, 0, st>>>(fan, nv + 1ull));
    BRT_LAUNCH(k_zero_words<<<1, 64, 0, st>>>(reinterpret_cast<uint32_t *>(d_flags), sizeof(MeshFlags) / 4));
    BRT_LAUNCH(k_tri_boxes<<<blocks_for(n, 256), 256, 0, st>>>(in.vertices, in.faces, n, lo, hi, ctr, fn3, fan, d_flags));
    BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp_scan, tb, fan, start, (int)(nv + 1), st));
    BRT_LAUNCH(k_corners<<<blocks_for(corners, 256), 256, 0, st>>>(in.faces, corners, start, fan, at));
    if (nv)
      BRT_LAUNCH(k_vertex_normals<<<blocks_for(nv, 256), 256, 0, st>>>(start, start + 1, nv, at, fn3, vnormals, longs,
                                                                      d_flags));
    BRT_LAUNCH(k_vertex_normals_long<<<256, 256, 0, st>>>(start, start + 1, at, fn3, longs, d_flags, vnormals));
    BRT_CHECK(hipMemcpyAsync(&hflags, d_flags, sizeof hflags, hipMemcpyDeviceToHost, st));
  } else {
    BRT_CHECK(hipMemcpyAsync(lo, in.box_lo, 3ull * n * 8, hipMemcpyHostToDevice, st));
    BRT_CHECK(hipMemcpyAsync(hi, in.box_hi, 3ull * n * 8, hipMemcpyHostToDevice, st));
    BRT_CHECK(hipMemcpyAsync(ctr, in.box_ctr, 3ull * n * 8, hipMemcpyHostToDevice, st));
  }
  BRT_LAUNCH(k_iota<<<blocks_for(n, 256), 256, 0, st>>>(idx, n));

  // ---- large nodes, level by level
  const uint32_t cap_nodes = n / SMALL + 2;                 // large nodes of one level are disjoint, > SMALL each
  const uint32_t cap_blocks = n / CHUNK + cap_nodes + 1;
  LNode *d_nodes = A.get<LNode>(cap_nodes);
  uint32_t *d_map = A.get<uint32_t>(2ull * cap_blocks);
  uint32_t *d_cnt4 = A.get<uint32_t>(4ull * cap_blocks);
  uint32_t *bcnt = A.get<uint32_t>((size_t)cap_nodes * 3 * nb);
  u64 *bklo = A.get<u64>((size_t)cap_nodes * 9 * nb), *bkhi = A.get<u64>((size_t)cap_nodes * 9 * nb);
  BRT_CHECK(A.err);
  Level L{d_nodes, d_map, d_map + cap_blocks, d_cnt4, d_cnt4 + cap_blocks, d_cnt4 + 2 * cap_blocks,
          d_cnt4 + 3 * cap_blocks, Bins{bcnt, bklo, bkhi}};

  BuildStatsDev hs{0, 0, 0, 0xFFFFFFFFu};
  std::vector<SmallRoot> small;
  std::vector<RawPut> puts;  // the large nodes
  auto add_child = [&](uint32_t begin, uint32_t cnt, uint32_t depth, uint32_t left, std::vector<HostTop> &next) {
    if (cnt > SMALL) next.push_back(HostTop{begin, cnt, depth, left});
    else small.push_back(SmallRoot{begin, cnt, depth, left});
  };
  std::vector<HostTop> level;
  add_child(0, n, 0, 0, level);
  std::vector<LNode> hn;
  std::vector<uint32_t> hmap;
  while (!level.empty()) {
    const uint32_t m = (uint32_t)level.size();
    hn.assign(m, LNode{});
    hmap.clear();
    uint32_t nblocks = 0;
    for (uint32_t i = 0; i < m; i++) {
      const HostTop &t = level[i];
      LNode &x = hn[i];
      x.begin = t.begin;
      x.n = t.n;
      x.depth = t.depth;
      x.blk0 = nblocks;
      x.nblk = blocks_for(t.n, CHUNK);
      nblocks += x.nblk;
    }
    hmap.resize(2ull * cap_blocks);
    for (uint32_t i = 0; i < m; i++)
      for (uint32_t b = 0; b < hn[i].nblk; b++) {
        hmap[hn[i].blk0 + b] = i;
        hmap[cap_blocks + hn[i].blk0 + b] = hn[i].begin + b * CHUNK;
      }
    BRT_CHECK(hipMemcpyAsync(d_nodes, hn.data(), m * sizeof(LNode), hipMemcpyHostToDevice, st));
    BRT_CHECK(hipMemcpyAsync(d_map, hmap.data(), 2ull * cap_blocks * 4, hipMemcpyHostToDevice, st));
    BRT_LAUNCH(k_lv_init<<<m, 256, 0, st>>>(L, nb));
    BRT_LAUNCH(k_lv_bounds<<<nblocks, BLOCK, 0, st>>>(L, idx, lo, hi));
    BRT_LAUNCH(k_lv_prep<<<blocks_for(m, 64), 64, 0, st>>>(L, m, in.min_leaf, in.max_depth));
    BRT_LAUNCH(k_lv_bin<<<nblocks, BLOCK, 0, st>>>(L, nb, idx, lo, hi, ctr));
    BRT_LAUNCH(k_lv_sweep<<<m, 64, 0, st>>>(L, nb));
    BRT_LAUNCH(k_lv_count<<<nblocks, BLOCK, 0, st>>>(L, idx, ctr));
    BRT_LAUNCH(k_lv_decide<<<blocks_for(m, 64), 64, 0, st>>>(L, m));
    BRT_LAUNCH(k_lv_rank1<<<nblocks, BLOCK, 0, st>>>(L, idx, ctr));
    BRT_LAUNCH(k_lv_rank2<<<m, 64, 0, st>>>(L));
    BRT_LAUNCH(k_lv_rank3<<<nblocks, BLOCK, 0, st>>>(L, idx, ctr, pos_r));
    BRT_LAUNCH(k_lv_swap<<<nblocks, BLOCK, 0, st>>>(L, idx, ctr, pos_r));
    BRT_CHECK(hipMemcpyAsync(hn.data(), d_nodes, m * sizeof(LNode), hipMemcpyDeviceToHost, st));
    BRT_CHECK(hipStreamSynchronize(st));
    if (hflags.refused) {
      out.refused = true;
      return hipSuccess;
    }
    std::vector<HostTop> next;
    for (uint32_t i = 0; i < m; i++) {
      const LNode &x = hn[i];
      const uint32_t left = level[i].left;
      hs.max_depth = std::max(hs.max_depth, x.depth);
      RawPut put{{{x.lo[0], x.lo[1], x.lo[2]}, {x.hi[0], x.hi[1], x.hi[2]}, x.begin, x.leaf ? x.n : x.axis, left, 0},
                 x.leaf ? x.begin : x.mid, x.leaf};
      puts.push_back(put);
      if (x.leaf) {
        hs.max_prims = std::max(hs.max_prims, x.n);
        hs.min_prims = std::min(hs.min_prims, x.n);
        continue;
      }
      hs.bad += x.bad;
      add_child(x.begin, x.mid - x.begin, x.depth + 1, left + 1, next);
      add_child(x.mid, x.begin + x.n - x.mid, x.depth + 1, left, next);
    }
    level.swap(next);
  }

  // ---- small and tiny subtrees
  const uint32_t ns = (uint32_t)small.size();
  const uint32_t tiny_blocks = std::min(blocks_for(n, 64), 4096u), tiny_waves = tiny_blocks * 4u;
  RawTree raw{A.get<RawNode>(n), A.get<RawNode>(n), A.get<uint32_t>(n), A.get<uint32_t>(n + 1ull)};
  uint32_t *before = A.get<uint32_t>(n + 1ull);
  SmallRoot *tiny = A.get<SmallRoot>(n), *list = A.get<SmallRoot>(n), *d_small = A.get<SmallRoot>(ns);
  uint32_t *num_tiny = A.get<uint32_t>(ns + 1ull), *tiny_at = A.get<uint32_t>(ns + 1ull);
  BuildStatsDev *d_stats = A.get<BuildStatsDev>((size_t)ns + tiny_waves);
  RawPut *d_puts = A.get<RawPut>(puts.size());
  size_t tb_tiny = 0, tb_before = 0;
  BRT_CHECK(A.err);
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb_tiny, num_tiny, tiny_at, (int)(ns + 1), st));
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb_before, raw.is_leaf, before, (int)(n + 1), st));
  unsigned char *scan_tmp = A.get<unsigned char>(std::max(tb_tiny, tb_before));
  BRT_CHECK(A.err);
  BRT_LAUNCH(k_zero_words<<<blocks_for(n, 256), 256, 0, st>>>(raw.is_inner, n));
  BRT_LAUNCH(k_zero_words<<<blocks_for(n + 1ull, 256), 256, 0, st>>>(raw.is_leaf, n + 1ull));
  BRT_LAUNCH(k_zero_words<<<1, 64, 0, st>>>(num_tiny + ns, 1));
  if (!puts.empty()) {
    BRT_CHECK(hipMemcpyAsync(d_puts, puts.data(), puts.size() * sizeof(RawPut), hipMemcpyHostToDevice, st));
    BRT_LAUNCH(k_put_raw<<<blocks_for(puts.size(), 64), 64, 0, st>>>(d_puts, (uint32_t)puts.size(), raw));
  }
  if (ns) {
    BRT_CHECK(hipMemcpyAsync(d_small, small.data(), ns * sizeof(SmallRoot), hipMemcpyHostToDevice, st));
    BRT_LAUNCH(k_small<<<ns, 64, 0, st>>>(d_small, idx, lo, hi, ctr, nb, in.min_leaf, in.max_depth, raw, tiny, num_tiny,
                                          d_stats));
  }
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(scan_tmp, tb_tiny, num_tiny, tiny_at, (int)(ns + 1), st));
  if (ns) BRT_LAUNCH(k_tiny_list<<<ns, 64, 0, st>>>(d_small, num_tiny, tiny_at, tiny, list));
  BRT_LAUNCH(k_tiny<<<tiny_blocks, 256, 0, st>>>(list, tiny_at + ns, idx, lo, hi, ctr, nb, in.min_leaf, in.max_depth, raw,
                                                 d_stats + ns));
  BRT_LAUNCH(k_sum_stats<<<1, 256, 0, st>>>(d_stats, ns + tiny_waves));
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(scan_tmp, tb_before, raw.is_leaf, before, (int)(n + 1), st));
  BuildStatsDev ds{};
  uint32_t leaves = 0;
  BRT_CHECK(hipMemcpyAsync(&leaves, before + n, 4, hipMemcpyDeviceToHost, st));
  BRT_CHECK(hipMemcpyAsync(&ds, d_stats, sizeof ds, hipMemcpyDeviceToHost, st));
  BRT_CHECK(hipStreamSynchronize(st));
  if (hflags.refused) {
    out.refused = true;
    return hipSuccess;
  }
  out.host_normals = hflags.max_fan > FAN_LONG;

  // ---- numbering
  const uint32_t M = 2u * leaves - 1u;
  brt_tree_node *tree = A.get<brt_tree_node>(M);
  uint32_t *ni = A.get<uint32_t>(M);
  BRT_CHECK(A.err);
  BRT_LAUNCH(k_emit<<<blocks_for(n, 256), 256, 0, st>>>(raw, n, before, tree, ni));

  // ---- flatten
  uint32_t *islots = A.get<uint32_t>(M), *S = A.get<uint32_t>(M), *k4 = A.get<uint32_t>(M),
           *is_root = A.get<uint32_t>(M);
  BRT_CHECK(A.err);
  BRT_LAUNCH(k_roots4<<<blocks_for(M, 256), 256, 0, st>>>(tree, M, is_root));
  BRT_LAUNCH(k_flags<<<blocks_for(M, 256), 256, 0, st>>>(tree, is_root, M, islots));
  size_t tb2 = 0;
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb2, islots, S, (int)M, st));
  unsigned char *tstore = A.get<unsigned char>(tb2);
  BRT_CHECK(A.err);
  BRT_CHECK(hipcub::DeviceScan::ExclusiveSum(tstore, tb2, islots, S, (int)M, st));
  uint32_t last[2] = {0, 0};
  BRT_CHECK(hipMemcpyAsync(&last[0], S + M - 1, 4, hipMemcpyDeviceToHost, st));
  BRT_CHECK(hipMemcpyAsync(&last[1], islots + M - 1, 4, hipMemcpyDeviceToHost, st));
  BRT_CHECK(hipMemcpyAsync(&out.root, tree, sizeof(brt_tree_node), hipMemcpyDeviceToHost, st));
  BRT_CHECK(hipStreamSynchronize(st));
  const uint32_t n64 = leaves - 1u;
  const uint32_t n4 = out.root.leaf ? 0u : 1u + last[0] + last[1];
  Node64 *nodes64 = A.get<Node64>(n64);
  Node4 *nodes4 = A.get<Node4>(n4);
  uint32_t *ord4 = A.get<uint32_t>(2ull * n4);
  size_t rec_size = 0;
  switch (in.type) {
  case TRIANGLES: rec_size = sizeof(TriRec); break;
  case SPHERES: rec_size = sizeof(SphRec); break;
  case PLANES: rec_size = sizeof(PlaRec); break;
  default: rec_size = sizeof(CylRec); break;
  }
  unsigned char *recs = A.get<unsigned char>((size_t)n * rec_size);
  BRT_CHECK(A.err);
  BRT_LAUNCH(k_assign4<<<blocks_for(M, 256), 256, 0, st>>>(tree, is_root, M, S, k4));
  BRT_LAUNCH(k_node64<<<blocks_for(M, 256), 256, 0, st>>>(tree, M, ni, nodes64));
  BRT_LAUNCH(k_node4<<<blocks_for(M, 256), 256, 0, st>>>(tree, is_root, M, k4, nodes4, ord4));
  const uint32_t g = blocks_for(n, 256);
  switch (in.type) {
  case TRIANGLES:
    BRT_LAUNCH(k_tri_recs<<<g, 256, 0, st>>>(idx, in.vertices, in.faces, n, reinterpret_cast<TriRec *>(recs)));
    break;
  case SPHERES: {
    const double *c = nullptr, *r = nullptr;
    BRT_CHECK(to_device(A, in.centers, 3ull * n, &c, st));
    BRT_CHECK(to_device(A, in.radii, n, &r, st));
    BRT_LAUNCH(k_sph_recs<<<g, 256, 0, st>>>(idx, c, r, n, reinterpret_cast<SphRec *>(recs)));
    break;
  }
  case PLANES: {
    const double *c = nullptr, *dx = nullptr, *dy = nullptr, *R = nullptr;
    BRT_CHECK(to_device(A, in.centers, 3ull * n, &c, st));
    BRT_CHECK(to_device(A, in.dxs, n, &dx, st));
    BRT_CHECK(to_device(A, in.dys, n, &dy, st));
    BRT_CHECK(to_device(A, in.rot, 9ull * n, &R, st));
    BRT_LAUNCH(k_pla_recs<<<g, 256, 0, st>>>(idx, c, dx, dy, R, n, reinterpret_cast<PlaRec *>(recs)));
    break;
  }
  default: {
    const double *c = nullptr, *a = nullptr, *b = nullptr, *h = nullptr, *R = nullptr;
    BRT_CHECK(to_device(A, in.centers, 3ull * n, &c, st));
    BRT_CHECK(to_device(A, in.sa, n, &a, st));
    BRT_CHECK(to_device(A, in.sb, n, &b, st));
    BRT_CHECK(to_device(A, in.heights, n, &h, st));
    BRT_CHECK(to_device(A, in.rot, 9ull * n, &R, st));
    BRT_LAUNCH(k_cyl_recs<<<g, 256, 0, st>>>(idx, c, a, b, h, R, n, reinterpret_cast<CylRec *>(recs)));
    break;
  }
  }
  BRT_CHECK(hipStreamSynchronize(st));

  out.tree = tree;
  out.num_nodes = M;
  out.order = idx;
  out.n64 = nodes64;
  out.num_n64 = n64;
  out.n4 = nodes4;
  out.num_n4 = n4;
  out.ord4 = ord4;
  out.vnormals = vnormals;
  out.recs = recs;
  out.rec_size = rec_size;
  out.max_depth = std::max(hs.max_depth, ds.max_depth);
  out.leaves = leaves;
  out.branches = leaves - 1u;
  out.bad_splits = hs.bad + ds.bad;
  out.max_prims = std::max(hs.max_prims, ds.max_prims);
  out.min_prims = std::min(hs.min_prims, ds.min_prims);
  for (void *p : {(void *)tree, (void *)idx, (void *)nodes64, (void *)nodes4, (void *)ord4, (void *)recs, (void *)vnormals})
    A.release(p);
  return hipSuccess;
}

}  // namespace brt
