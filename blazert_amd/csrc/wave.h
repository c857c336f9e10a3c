// What the persistent kernels' waves share: the traversal stack of the 4-wide FP32 trees (NodeQ), a ring of entries per lane
// in LDS with the older ones in private memory; the pool a wave takes its rays or points from; and what lanes need to take
// over each other's work.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "engine.h"

// LDS pointers of the ring stack carry the LDS address space explicitly: as generic pointers the compiler had to
// resolve their address space at run time in places (flat accesses), which costs time on the coherent sets.
#define BRT_LDS __attribute__((address_space(3)))

namespace brt {

// One entry: a node or leaf reference, and its entry distance with the low 8 bits (rounded towards 0; keys are not
// negative) replaced by the leaf's primitive count.
struct WideEntry {
  uint32_t ref, key;
};
constexpr uint32_t WIDE_SPILL = 192;  // three entries per level, at most 63 levels (stack_cap)

// The lane's stack: entries [bot, sp), of which [lo, sp) lie in the LDS ring and the older ones in private memory.
// Entries below bot have been given away.
struct WideStack {
  BRT_LDS uint32_t *ring;  // the lane's slot 0; slot i: reference at [128 i], key at [128 i + 64]
  uint64_t *spill;
  int sp, lo, bot;
  int mask;  // ring slots - 1

  __device__ __forceinline__ void reset() { sp = lo = bot = 0; }
  __device__ __forceinline__ void room(int n) {  // n more entries fit the ring
    while (sp + n - lo > mask + 1) {
      spill[lo] = slot(lo);
      lo++;
    }
  }
  __device__ __forceinline__ void put(int i, uint32_t ref, uint32_t key) {
    BRT_LDS uint32_t *e = ring + (i & mask) * 128;
    e[0] = ref;
    e[64] = key;
  }
  __device__ __forceinline__ uint64_t slot(int i) const {
    BRT_LDS uint32_t *e = ring + (i & mask) * 128;
    return ((uint64_t)e[64] << 32) | e[0];
  }
  __device__ __forceinline__ WideEntry pop() {  // requires sp > bot
    sp--;
    uint64_t e;
    if (sp < lo) {
      lo = sp;
      e = spill[sp];
    } else {
      e = slot(sp);
    }
    return WideEntry{(uint32_t)e, (uint32_t)(e >> 32)};
  }
  __device__ __forceinline__ uint64_t take_bottom() {  // requires sp > bot
    uint64_t e;
    if (bot < lo) e = spill[bot];
    else e = slot(bot);
    bot++;
    lo = lo < bot ? bot : lo;
    return e;
  }
};

// A value of another lane, for the lanes that take over its work.
__device__ __forceinline__ uint32_t lane_get(uint32_t x, int src) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)x);
}
template <class V>
__device__ __forceinline__ void lane_take(V &x, int src, bool take) {
  static_assert(sizeof(V) % 4 == 0, "words");
  uint32_t w[sizeof(V) / 4];
  __builtin_memcpy(w, &x, sizeof(V));
#pragma unroll
  for (size_t k = 0; k < sizeof(V) / 4; k++) {
    const uint32_t y = lane_get(w[k], src);
    w[k] = take ? y : w[k];
  }
  __builtin_memcpy(&x, w, sizeof(V));
}
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Persistent waves: every lane owns one ray at a time; when at least `refill` lanes of a wave are idle, they start
// the next indices of the wave's pool. Skewed per-ray work (many rays miss the root box, a few visit hundreds of
// nodes) then no longer idles the wave until its slowest ray ends. The pool is a chunk of `chunk` consecutive indices
// (POOL_CHUNK unless the launch asks for 32 or 128) claimed with one atomic add. Claims on one address serialise
// across the GPU (about 14 ns each), which bounded short launches and image-order rays, so they are spread over
// CLAIM_COUNTERS counters on separate 128-byte lines: counter k hands out chunks k, k + CLAIM_COUNTERS,
// k + 2 CLAIM_COUNTERS, ... A wave starts at the counter of its block (block index mod CLAIM_COUNTERS: blocks are
// dealt to the eight XCDs in turn, so each XCD's waves start at a counter of their own) and moves on to the next
// counter once one has passed n. When all have, the pool is exhausted; every lane leaves the loop once its pool is
// exhausted and its own ray is done, so the grid always drains.
constexpr uint32_t POOL_CHUNK = 64;

// Wave-uniform pool of claimed, not yet started ray indices [next, end).
struct WavePool {
  uint64_t next = 0, end = 0;
  bool last = false;  // every counter has passed n
  // A wave of a small launch (fixed_per_wave) takes `count` indices from `first` on and claims none.
  __device__ __forceinline__ void take_fixed(uint64_t first, uint32_t count, uint64_t n) {
    next = first < n ? first : n;
    end = next + count < n ? next + count : n;
    last = true;
  }
};

// Rays per wave of a launch that the device's `waves` resident waves take in one go (up to a full wave each; 262,144 on
// 256 CUs): the waves then have idle lanes from the start, which share their rays' work, and none waits for a claim.
// 0 for larger launches, whose waves claim. Incoherent rays, 82k-triangle mesh: 2,000 rays 123 -> 74 us against claims
// of 64; 328k-triangle mesh: 50,000 rays 265 -> 202 us, 200,000 rays 375 -> 324 us; a 200x150 camera 394 -> 250 us.
inline uint32_t fixed_per_wave(uint64_t n, uint64_t waves) {
  const uint64_t per = (n + waves - 1) / waves;
  return per <= 64 ? (uint32_t)per : 0u;
}

// Adds the numbers of the lanes with `set` to a wave-uniform mask; called by the whole wave.
__device__ __forceinline__ void mask_add(unsigned long long &mask, bool set, uint32_t number) {
  unsigned long long m = __ballot(set);
  while (m) {
    const int l = __ffsll((long long)m) - 1;
    mask |= 1ull << (uint32_t)__builtin_amdgcn_readlane((int)number, l);
    m &= m - 1ull;
  }
}

// Called by every lane of a wave with the same pool state when the wave refills. An idle lane handed an index gets
// it in `idx` and `got`; `exhausted` is set once nothing is left to hand out. `counter` is the first of the
// launch's CLAIM_COUNTERS counters (COUNTER_STRIDE slots apart).
__device__ __forceinline__ void pool_refill(WavePool &P, unsigned long long *counter, uint64_t n, uint32_t chunk,
                                            unsigned long long idle, uint32_t nidle, uint32_t lane, bool &got,
                                            uint64_t &idx, bool &exhausted) {
  got = false;
  if (P.next == P.end && !P.last) {
    unsigned long long base = n;
    const uint32_t leader = (uint32_t)__ffsll((long long)idle) - 1u;
    if (lane == leader) {
      const uint32_t home = blockIdx.x % (uint32_t)CLAIM_COUNTERS;
      for (uint32_t a = 0; a < (uint32_t)CLAIM_COUNTERS; a++) {
        const uint32_t k = (home + a) % (uint32_t)CLAIM_COUNTERS;
        const unsigned long long c = atomicAdd(counter + k * COUNTER_STRIDE, 1ull);
        const unsigned long long start = (c * CLAIM_COUNTERS + k) * chunk;
        if (start < n) {
          base = start;
          break;
        }
      }
    }
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)base, (int)leader);
    const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(base >> 32), (int)leader);
    base = ((unsigned long long)hi << 32) | lo;
    if (base >= n) {
      P.last = true;
      P.next = P.end = n;
    } else {
      P.next = base;
      P.end = base + chunk < n ? base + chunk : n;
    }
  }
  const uint64_t avail = P.end - P.next;
  const uint32_t take = avail < nidle ? (uint32_t)avail : nidle;
  const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
  if (((idle >> lane) & 1ull) && rank < take) {
    idx = P.next + rank;
    got = true;
  }
  P.next += take;
  if (P.last && P.next == P.end) exhausted = true;
}
// Lanes of k_trace_wide and k_closest_triangles with an FP64 test, or with a pre-test, wait for as many of the wave (see there).
constexpr int WIDE_MIN_LANES = 16;

// Work sharing in a wave with nothing left to start: from SHARE_MIN_IDLE idle lanes on, these take over stack entries of
// the busy ones. At most SHARE_SLOTS queries of a wave are then ever shared.
constexpr uint32_t SHARE_MIN_IDLE = 32;
constexpr uint32_t SHARE_SLOTS = 32;
static_assert(64u - SHARE_MIN_IDLE <= SHARE_SLOTS, "a slot for every query left");

}  // namespace brt
