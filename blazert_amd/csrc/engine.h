// Host-side interface between the C ABI (scene.cpp) and the HIP kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <functional>

#include "../../include/blazert_amd.h"
#include "layout.h"

namespace brt {

// Slots of the Node4 record rooted at binary internal node b (pre-order tree T): start from b's two children and,
// while fewer than four slots are filled, replace the internal slot of largest surface area (the first of equal
// ones) by its two children in place, so the slots stay in the binary tree's left-to-right order. The internal slots
// are the roots of further records. Shared by the host flatten and the device build, which give identical records.
// A record advances a root-to-leaf path by at least one binary level and pushes at most three stack entries.
// With `axis` the split axis of every slot pair's lowest common ancestor is reported too: axis[4 * i + j], i < j.
__host__ __device__ inline int collapse4(const brt_tree_node *T, uint32_t b, uint32_t slot[4],
                                         uint32_t *axis = nullptr) {
#pragma clang fp contract(off)
  slot[0] = T[b].children[0];
  slot[1] = T[b].children[1];
  if (axis) axis[1] = T[b].axis;
  int m = 2;
  while (m < 4) {
    int best = -1;
    double area = 0.0;
    for (int c = 0; c < m; c++) {
      const brt_tree_node &x = T[slot[c]];
      if (x.leaf) continue;
      const double dx = x.max[0] - x.min[0], dy = x.max[1] - x.min[1], dz = x.max[2] - x.min[2];
      const double a = dx * dy + dy * dz + dz * dx;
      if (best < 0 || a > area) {
        best = c;
        area = a;
      }
    }
    if (best < 0) break;
    const uint32_t e = slot[best];
    for (int c = m; c > best + 1; c--) slot[c] = slot[c - 1];
    slot[best] = T[e].children[0];
    slot[best + 1] = T[e].children[1];
    if (axis) {
      uint32_t old[16];
      for (int i = 0; i < 16; i++) old[i] = axis[i];
      const auto from = [&](int c) { return c > best ? c - 1 : c; };  // slot c's place before the split
      for (int i = 0; i <= m; i++)
        for (int j = i + 1; j <= m; j++)
          axis[4 * i + j] = (i == best && j == best + 1) ? T[e].axis : old[4 * from(i) + from(j)];
    }
    m++;
  }
  return m;
}

// The visiting order of a record's m slots (NodeQ::ord) from the split axes collapse4 reports: of two slots the left
// one comes first when the direction is not negative along the axis that parts them (blazert/bvh/accel.h:95-104).
__host__ __device__ inline void visit_order4(const uint32_t axis[16], int m, uint32_t ord[2]) {
  ord[0] = ord[1] = 0;
  for (uint32_t oct = 0; oct < 4; oct++) {
    uint32_t later = 0;
    for (int i = 0; i < m; i++)
      for (int j = i + 1; j < m; j++) {
        const bool right_first = (oct >> axis[4 * i + j]) & 1u;
        later |= right_first ? 1u << (4 * j + i) : 1u << (4 * i + j);
      }
    ord[oct >> 1] |= later << (16 * (oct & 1u));
  }
}

// Device counters of one traversal launch, in a group cleared by the launch itself: the persistent schedule's ray
// pool; a flag a split-precision launch sets when it defers rays to the exact path; the ray pool of the FP64 launch
// that traces them. Launches on one stream run in order, so one group per stream serves all of them.
// The ray pools take claims from CLAIM_COUNTERS counters, each on its own 128-byte line (COUNTER_STRIDE slots apart):
// slot k * COUNTER_STRIDE + COUNTER_POOL for the launch, + COUNTER_DEFERRED_POOL for its deferred-ray launch.
constexpr int COUNTER_POOL = 0;
constexpr int COUNTER_DEFERRED = 1;
constexpr int COUNTER_DEFERRED_POOL = 2;
constexpr int CLAIM_COUNTERS = 8;
constexpr int COUNTER_STRIDE = 16;
constexpr int COUNTER_CLEARED = CLAIM_COUNTERS * COUNTER_STRIDE;  // slots a launch clears (1 KiB)
// What a fast traversal leaves to the exact launch behind it: COUNTER_DEFERRED says that rays were passed over, and others are
// listed behind the counters, COUNTER_LISTED counting them. Both have a slot on each of the CLAIM_COUNTERS lines, and each line
// its own part of the list, for the blocks that start claiming there: one line for all of them is busy for longer than such
// rays take. When a part overflows, the launch behind traces every ray. A launch with a fixed range of at most 64 rays per wave
// writes one word per wave there instead, a bit for each ray left, and needs no cleared counters.
constexpr int COUNTER_LISTED = 3;
constexpr int LIST_CAPACITY = 32640;
constexpr int LIST_PART = LIST_CAPACITY / CLAIM_COUNTERS;
constexpr int COUNTER_GROUP = COUNTER_CLEARED + LIST_CAPACITY;  // slots per group (256 KiB)

constexpr uint32_t SCHEDULE_PERSISTENT = 0;  // persistent waves with per-lane ray refill (default)
constexpr uint32_t SCHEDULE_PER_THREAD = 1;  // one ray per thread, grid-stride

struct TraceLaunch {
  uint32_t precision;  // BRT_PRECISION_*
  uint32_t flags;      // BRT_FLAG_*
  uint32_t block;      // threads per block
  bool first;          // first geometry type of the scene: initialises every hit record
  uint32_t schedule;   // SCHEDULE_*
  uint32_t refill;     // persistent: refill a wave once this many lanes are idle (1..64)
  unsigned long long *counter;  // COUNTER_GROUP device counters for this launch (cleared on the stream)
  const uint32_t *order;        // optional ray permutation (sorted launches); kernels trace rays[order[k]]
  uint32_t ring = 0;            // LDS stack slots per lane: 4, 8 or 16 (0 = default of the precision)
  uint32_t pool = 0;            // persistent: ray indices per claim, 32, 64 or 128 (0 = 64)
  bool fast = false;            // batches: every job's triangle tree has reference-order nodes (BvhView::nodesq)
  bool overwrite = false;       // every hit replaces the record (traverse semantics), not only closer ones
};

// One (scene, geometry type, ray batch) of a multi-scene launch; jobs are sorted by offset.
struct BatchJob {
  BvhView bvh;
  RaysView rays;
  HitsView hits;
  uint64_t n;       // rays of this job
  uint64_t offset;  // prefix sum of n over the preceding jobs
  uint32_t first;   // this geometry type is the first one of the job's scene
  uint32_t is_tri;
  double extent;    // split precision: scene extent
  const uint32_t *order;
};

// Enqueues one persistent launch over all jobs of one geometry type (total = sum of n).
hipError_t launch_trace_batch(GeomType type, const BatchJob *jobs, uint32_t njobs, uint64_t total,
                              const TraceLaunch &cfg, hipStream_t stream);

// Device buffers of one ray sort (keys, values, radix-sort temporary storage).
struct SortWorkspace {
  void *base = nullptr;
  uint32_t *keys_in = nullptr, *keys_out = nullptr, *vals_in = nullptr, *vals_out = nullptr;
  void *temp = nullptr;
  size_t temp_bytes = 0;
  uint64_t capacity = 0;
};

// Grows ws to hold n rays (frees the previous buffers; not capturable in a graph).
hipError_t sort_workspace_reserve(SortWorkspace &ws, uint64_t n);
// Lays out a workspace for n rays in caller memory [base, base + bytes) without allocating; hipErrorInvalidValue
// when it does not fit.
hipError_t sort_workspace_in(SortWorkspace &ws, void *base, size_t bytes, uint64_t n);

// Device scratch of the allocation-free intersect (brt_intersect_noalloc): a file-scope __device__ array, one copy
// per GPU, holding a launch counter group at its start and then the workspace of a ray sort of up to
// NOALLOC_MAX_SORTED_RAYS rays.
constexpr uint64_t NOALLOC_MAX_SORTED_RAYS = 1ull << 20;
constexpr size_t NOALLOC_SCRATCH_BYTES = (24ull << 20) + COUNTER_GROUP * 8;
// This device's address of the scratch array (looked up once per device with hipGetSymbolAddress).
hipError_t noalloc_scratch(unsigned char **ptr);
// Computes the sort keys (mode 1: direction octant + origin Morton code, mode 2: Morton only) and radix-sorts the
// ray indices on `stream`; *order points into ws afterwards.
hipError_t sort_rays(const RaysView &rays, uint64_t n, const double lo[3], const double hi[3], uint32_t mode,
                     SortWorkspace &ws, hipStream_t stream, const uint32_t **order);

// Per-scene constants for the split-precision path: the largest finite |coordinate| of any node box.
struct SplitParams {
  double scene_extent;
};

// Writes the FP32 pre-test records (TriFilt, n + FILTER_PAD of them) of n leaf-order TriRecs.
hipError_t launch_tri_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream);
// Writes the FP32 pre-test records (SphFilt, n + SPH_FILTER_PAD of them) of n leaf-order SphRecs.
hipError_t launch_sph_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream);
// Writes the FP32 pre-test records (CylFilt, n + SPH_FILTER_PAD of them) of n leaf-order CylRecs.
hipError_t launch_cyl_filter_records(const void *recs, uint32_t n, void *out, hipStream_t stream);

// Writes the leaves' boxes, each at its first primitive's place in leaf order (six numbers of the scene's type).
hipError_t launch_leaf_boxes(const BvhView &bvh, bool f32, void *out, hipStream_t stream);
// Assembles the reference-order nodes (NodeQ) from n Node4 records and their visiting orders (two words per record,
// visit_order4).
hipError_t launch_nodeq_records(const Node4 *nodes4, const uint32_t *ord, uint32_t n, NodeQ *out, hipStream_t stream);

// Clears the counters of a group on the stream.
hipError_t launch_zero_counters(unsigned long long *group, hipStream_t stream);

// Enqueues the traversal of one geometry type over n rays on `stream` (asynchronous).
hipError_t launch_trace(GeomType type, const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint64_t n,
                        const TraceLaunch &cfg, const SplitParams &split, hipStream_t stream);
// n rows of three elements (4 or 8 bytes each) to three columns of n, one after another.
hipError_t launch_rows_to_columns(const void *rows, uint32_t elem_bytes, uint64_t n, void *columns, hipStream_t stream);
// The closest hit of one ray (index 0) among the triangles of an FP64 scene whose view has nodesq. hits.merged is required
// and set to RAY_LEFT where the ray needs launch_trace, and nothing else is then written.
hipError_t launch_tri_lone(const BvhView &bvh, const RaysView &rays, const HitsView &hits, uint32_t flags,
                           const SplitParams &split, hipStream_t stream);

// Mirror tracing: the next bounce's rays from this bounce's hits (positions o + t normalize(d), mirror directions;
// NaN for misses). pos / dir are x, y, z arrays of n doubles.
hipError_t launch_mirror_step(const RaysView &rays, const HitsView &hits, const double *vertices,
                              const uint32_t *faces, uint64_t n, double *const pos[3], double *const dir[3],
                              hipStream_t stream);

// Upstream gradients in, parameter gradients out, of the mirror-tracing adjoint (any pointer may be NULL).
struct MirrorGrads {
  const double *gt;              // dL/dt, bounces * n
  const double *gpx, *gpy, *gpz;  // dL/d(hit position), bounces * n each
  double *gv;                    // dL/dvertex, 3 per vertex, accumulated
  double *gox, *goy, *goz;       // dL/d(ray origin), n each, written
  double *gdx, *gdy, *gdz;       // dL/d(raw ray direction), n each, written
};

// Adjoint of `bounces` (1..8) mirror bounces recomputed from the stored face ids prims[b * n + i]; a ray's chain
// ends at its first id >= num_faces (a miss).
hipError_t launch_mirror_adjoint(const RaysView &rays, const uint32_t *prims, uint32_t bounces,
                                 const double *vertices, const uint32_t *faces, uint32_t num_faces, uint64_t n,
                                 const MirrorGrads &g, hipStream_t stream);

// Writes the default RayHit (t = DBL_MAX, ids invalid, u = v = 0, normal 0) for n rays.
hipError_t launch_init_hits(const HitsView &hits, uint64_t n, hipStream_t stream);

// Scene<float>: traversal of one geometry type in FP32 (bvh.nodes32 and FP32 records), and the FP32 default RayHit.
hipError_t launch_trace_f32(GeomType type, const BvhView &bvh, const RaysViewF &rays, const HitsViewF &hits,
                            uint64_t n, const TraceLaunch &cfg, double extent, hipStream_t stream);
hipError_t launch_init_hits_f32(const HitsViewF &hits, uint64_t n, hipStream_t stream);

// Distance queries (distance.hip). inv maps primitive ids to leaf positions (spheres, planes, cylinders; built by
// launch_inverse_order from the view's prim_ids); ids >= n_prims give NaN.
hipError_t launch_inverse_order(const uint32_t *order, uint32_t n, uint32_t *inv, hipStream_t stream);
hipError_t launch_distance_pairs(GeomType type, const BvhView &bvh, const uint32_t *inv, const double *px,
                                 const double *py, const double *pz, const uint32_t *ids, uint64_t n, double *out,
                                 hipStream_t stream);
// All geometry types of a scene for the closest-surface query; extent = largest |coordinate| of a type's boxes.
struct ClosestViews {
  BvhView view[NUM_TYPES];
  double extent[NUM_TYPES];
  uint32_t present[NUM_TYPES];
  const double *leaf_vertices;  // triangles in leaf order: v0, v1, v2 (9 doubles each)
};
// Gathers the triangles' vertices in leaf order (9 doubles per triangle) for the closest-surface query.
hipError_t launch_leaf_vertices(const uint32_t *order, const uint32_t *faces, const double *vertices, uint32_t n,
                                double *out, hipStream_t stream);
// claims: called when a search of triangles is too large for one range per wave (fixed_per_wave); gives COUNTER_CLEARED
// words that no other launch uses before this one has ended, or NULL where there are none to be had.
hipError_t launch_closest_surface(const ClosestViews &views, const double *px, const double *py, const double *pz,
                                  uint64_t n, double *dist, uint32_t *prim, uint32_t *geom,
                                  const std::function<unsigned long long *()> &claims, hipStream_t stream);

// Device memory of scenes and builds (scene.cpp). hipMalloc and hipFree of a scene's arrays and a build's workspace cost
// more than building it (1.31M triangles: 50 and 46 calls, 10.5 of 20 ms), so freed blocks are kept for the next one: up
// to POOL_BYTES per device, and only while a scene lives on that device; the last one gives everything back. A block freed
// with idle = false may still be in use by kernels in flight: whoever takes it waits for the device first. Thread safe.
constexpr size_t POOL_BYTES = 2ull << 30;
hipError_t pool_get(int device, size_t bytes, void **p);
void pool_put(int device, void *p, bool idle);
// Host memory that kernels read and write in place, LONE_SLOT_BYTES of it: kept and given back like the device memory, up
// to LONE_SLOTS of them. The caller has waited for the kernels that use it (`idle`), or it isn't kept.
constexpr size_t LONE_SLOT_BYTES = 256, LONE_SLOTS = 64;
hipError_t pool_get_slot(int device, void **p);
void pool_put_slot(int device, void *p, bool idle);
void pool_retain(int device);
void pool_release(int device);

// Device build of one geometry type's BVH (build.hip): the host builder's tree, primitive order and flattened
// records, bit for bit, provided no primitive box coordinate is NaN or -0.0 (the caller checks) and
// device_build_supported() holds for the options.
struct DeviceBuildIn {
  GeomType type;
  uint32_t n;  // primitives (> 0)
  uint32_t min_leaf, max_depth, nbins;
  const double *vertices;  // triangles: device vertices and faces (boxes and normals are computed on the device)
  const uint32_t *faces;
  uint32_t num_vertices;
  const double *box_lo, *box_hi, *box_ctr;  // other types: host boxes and centers, 3 per primitive
  const double *centers, *radii, *dxs, *dys, *rot, *sa, *sb, *heights;  // other types: host record inputs
};
// Results are pool allocations owned by the caller afterwards.
struct DeviceBuildOut {
  brt_tree_node *tree;  // reference-form nodes in pre-order
  uint32_t num_nodes;
  uint32_t *order;      // leaf order -> primitive id
  Node64 *n64;
  uint32_t num_n64;
  Node4 *n4;
  uint32_t num_n4;
  uint32_t *ord4;       // visiting order of every Node4's slots, two words each (visit_order4)
  void *recs;           // primitive records in leaf order
  double *vnormals;     // triangles: vertex normals
  bool host_normals;    // triangles: some vertex has too many corners, vnormals are left to the host
  bool refused;         // triangles: some box coordinate is not finite or is -0.0; nothing else is set
  size_t rec_size;
  brt_tree_node root;   // host copy of node 0
  uint32_t max_depth, leaves, branches, bad_splits, max_prims, min_prims;
  uint32_t failed_line;  // on error: source line (build.hip) of the failing call
};
bool device_build_supported(uint32_t nbins, uint32_t max_depth);
// Builds on `stream` and waits for it.
hipError_t device_build(const DeviceBuildIn &in, DeviceBuildOut &out, hipStream_t stream);

}  // namespace brt
