// Device-side closest-hit traversal shared by the triangle-accel and instance-accel trace kernels.
//
// One node fetch decides both children (64-byte node with both child boxes); leaf children are handed to
// a leaf callback in batches across the wave; the near inner child is descended and the far one pushed on
// a per-lane stack whose first entries live in LDS and the rest in a per-lane global spill area. A plain
// trace runs trace_stream; with a proposal or fetch counts, or for trees of kSmallTreePrims primitives
// and more, a lane walks one ray at a time with walk_batched.
#pragma once

#include <climits>

#include "bvh.hpp"

namespace gprt {

constexpr int kTraceBlock = 128;
constexpr int kLdsStack = 20;
// 14 workgroups (28 waves) per CU: 16, the most the LDS stacks allow, measured no faster.
constexpr int kBlocksPerCU = 14;
// A binary radix tree over distinct 64-bit keys is at most 64 levels deep, so a walk needs at most 64
// entries.
constexpr int kMaxStack = 64;
// Words of work counters before the spill area.
constexpr uint32_t kTraceHeaderWords = 256;

// First of the next 64 rays of a wave of the one-ray-per-lane kernels: the wave's own, or, where there are
// more rays than lanes, from a counter (zeroed). (Then even the first 64: each wave's own first and the
// counter after them took the primary rays of a dynamic frame from 1,690 to 1,830 us, its bounce rays from
// 2,290 to 2,130.)
__device__ __forceinline__ uint32_t next_rays(uint32_t *__restrict__ work, bool more) {
  uint32_t base = blockIdx.x * kTraceBlock + (threadIdx.x & ~63u);
  if (more && (threadIdx.x & 63) == 0) base = atomicAdd(work, 64u);
  return __builtin_amdgcn_readfirstlane(base);
}

// Closest hit so far. Hits are ordered by (t, inst, prim) with unsigned comparisons, so the
// result does not depend on the order in which subtrees or instances are visited.
struct HitState {
  float t, u, v;
  int prim;      // -1: none yet
  uint32_t inst; // instance index (0 for a triangle accel); 0xFFFFFFFF: none yet
  int leaf;      // instance accels: index of the top-level leaf (sub-root) holding the hit
};

__device__ __forceinline__ void hit_init(HitState &h, float tmax) {
  h.t = tmax;
  h.u = h.v = 0.f;
  h.prim = -1;
  h.inst = 0xFFFFFFFFu;
  h.leaf = -1;
}

__device__ __forceinline__ bool hit_closer(float t, uint32_t inst, int prim, const HitState &h) {
  return t < h.t || (t == h.t && (inst < h.inst || (inst == h.inst && (unsigned)prim < (unsigned)h.prim)));
}

struct LaneStack {
  uint32_t (*lds)[kTraceBlock];
  int tid;
  uint32_t *spill;  // per-lane global entries [kLdsStack, maxStack)
};

// Reads stack entry `sp` (the first kLdsStack in LDS, the rest in the lane's spill area). The spill
// read is a relaxed wave-scope atomic load, an ordinary global load in the code, so that the
// compiler does not fold the two reads into one flat load behind an address select: that costs
// about seven more vector instructions per pop and waits for every outstanding memory operation.
__device__ __forceinline__ uint32_t stack_read(const LaneStack &st, int sp) {
  if (sp < kLdsStack) return st.lds[sp][st.tid];
  return __hip_atomic_load(&st.spill[sp - kLdsStack], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Tests one triangle record ({v0, primID} {v1} {v2}) of instance `inst`; `tag` is recorded with a hit.
__device__ __forceinline__ void intersect_record(const RayPre &r, const TriRecord &tr, uint32_t inst, int tag,
                                                 HitState &h) {
  float t, u, v;
  if (tri_hit(r, tr.v0, tr.v1, tr.v2, t, u, v)) {
    const int prim = (int)__float_as_uint(tr.v0.w);
    if (hit_closer(t, inst, prim, h)) {
      h.t = t;
      h.prim = prim;
      h.u = u;
      h.v = v;
      h.inst = inst;
      h.leaf = tag;
    } else if (t == h.t && inst == h.inst && prim == h.prim && h.leaf < 0) {
      h.leaf = tag;  // the same hit, first found by a walk that did not know its top-level leaf
    }
  }
}

// Tests one box-primitive record ({lo, primID} {hi} {0}); box hits report u = v = 0.
__device__ __forceinline__ void intersect_box_record(const RayPre &r, const TriRecord &tr, uint32_t inst, int tag,
                                                     HitState &h) {
  float t;
  if (boxprim_hit(r, tr.v0, tr.v1, t)) {
    const int prim = (int)__float_as_uint(tr.v0.w);
    if (hit_closer(t, inst, prim, h)) {
      h.t = t;
      h.prim = prim;
      h.u = 0.f;
      h.v = 0.f;
      h.inst = inst;
      h.leaf = tag;
    } else if (t == h.t && inst == h.inst && prim == h.prim && h.leaf < 0) {
      h.leaf = tag;
    }
  }
}

// kBoxes: the leaves are box primitives rather than triangles.
// kSmall: the tree has fewer than 2^26 primitives, so node and record byte offsets fit in 32 bits
// (an address is then one shift from the array's base instead of 64-bit arithmetic).
constexpr uint32_t kSmallTreePrims = 1u << 26;

template <class T>
__device__ __forceinline__ const T &at32(const T *base, uint32_t i) {
  return *(const T *)((const char *)base + i * (uint32_t)sizeof(T));
}

template <bool kBoxes = false, bool kSmall = false>
__device__ __forceinline__ void intersect_leaf(const RayPre &r, const TriRecord *__restrict__ tris, int leaf,
                                               uint32_t nprims, uint32_t inst, int tag, HitState &h) {
  if ((uint32_t)leaf >= nprims) return;
  const TriRecord &rec = kSmall ? at32(tris, (uint32_t)leaf) : tris[(uint32_t)leaf];
  if (kBoxes)
    intersect_box_record(r, rec, inst, tag, h);
  else
    intersect_record(r, rec, inst, tag, h);
}

constexpr int kNoSkip = INT_MIN;

// Depth-first walk of the subtree rooted at `start` (an inner node index, or ~leaf position) of a
// tree with `nprims` leaves, using stack slots [sp0, MaxStack). leaf(position, spTop) is called for
// every leaf whose box the ray meets; spTop is the first free stack slot. A child equal to `skip` (a
// subtree already searched completely; kNoSkip for none) is not entered.
//
// Leaf tests are postponed and batched across the wave: a lane
// queues the leaf children it meets (up to kLeafQueue, in registers) and keeps walking; the wave
// runs its leaf tests when at least half of its active lanes have leaves queued, or when a lane can
// go no further (no node left, or no room for another node's two leaves). The triangle test is
// long, and run per node it executes whenever any one lane of the wave needs it; batched, it
// executes for many lanes at once. Queued leaves are tested later, so box culling sees a
// bound that is less tight in between (a few more node fetches); the closest-hit rule makes the
// result independent of the order of the tests. Returns the number of inner nodes fetched.
constexpr int kLeafQueue = 4;

template <int MaxStack, class LeafFn>
__device__ __forceinline__ uint32_t walk_batched(const RayPre &r, const BVHNode *__restrict__ nodes, uint32_t nprims,
                                                 int start, const HitState &h, const LaneStack &st, int sp0, int skip,
                                                 LeafFn &&leaf) {
  constexpr int kDone = INT_MIN;
  if (nprims == 0) return 0;  // an empty tree has no nodes
  // Queued leaves as child codes (~position, negative; q0 is the next tested): decoded when tested.
  int q0 = -1, q1 = -1, q2 = -1, q3 = -1, nq = 0;
  auto enqueue = [&](int code) __attribute__((always_inline)) {
    q3 = q2;
    q2 = q1;
    q1 = q0;
    q0 = code;
    ++nq;
  };
  int node = start;
  if (start < 0) {
    enqueue(start);
    node = kDone;
  }
  int sp = sp0;
  uint32_t visits = 0;
  // Every iteration either fetches a node (each inner node at most once per walk) or tests all
  // queued leaves, so the bound only guards against a malformed tree.
  const uint32_t limit = 4u * nprims + 8u;
  for (uint32_t it = 0; it < limit; ++it) {
    if (node != kDone && nq <= kLeafQueue - 2) {
      if ((uint32_t)node >= nprims - 1) {
        node = kDone;  // only a malformed tree
      } else {
        const BVHNode nd = nodes[(uint32_t)node];  // node >= 0 here: no sign extension
        ++visits;
        float tn0, tn1;
        bool h0 = box_hit(r, nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y, h.t, tn0);
        bool h1 = box_hit(r, nd.b.z, nd.b.w, nd.c.x, nd.c.y, nd.c.z, nd.c.w, h.t, tn1);
        const int c0 = nd.d.x, c1 = nd.d.y;
        h0 = h0 && c0 != skip;
        h1 = h1 && c1 != skip;
        if (h0 && c0 < 0) {
          enqueue(c0);
          h0 = false;
        }
        if (h1 && c1 < 0) {
          enqueue(c1);
          h1 = false;
        }
        if (h0 && h1) {
          const bool firstNear = tn0 <= tn1;
          const int farC = firstNear ? c1 : c0;
          if (sp < kLdsStack)
            st.lds[sp][st.tid] = (uint32_t)farC;
          else if (sp < MaxStack)
            st.spill[sp - kLdsStack] = (uint32_t)farC;
          ++sp;
          node = firstNear ? c0 : c1;
        } else if (h0) {
          node = c0;
        } else if (h1) {
          node = c1;
        } else if (sp == sp0 || sp > MaxStack) {
          node = kDone;
        } else {
          --sp;
          node = (int)stack_read(st, sp);
        }
      }
    }
    const bool stuck = nq > 0 && (node == kDone || nq > kLeafQueue - 2);
    const uint64_t active = __ballot(1);
    const uint64_t waiting = __ballot(nq > 0);
    if (__ballot(stuck) || 2 * __popcll(waiting) >= __popcll(active)) {
      // One call site for the triangle test: lanes drain their queues together.
      while (nq > 0) {
        const int code = q0;
        q0 = q1;
        q1 = q2;
        q2 = q3;
        --nq;
        leaf(~code, sp);
      }
    }
    if (node == kDone && nq == 0) break;
  }
  return visits;
}

// Primitive-accel walk: leaves are triangles (or, with kBoxes, box primitives) of instance `inst`;
// `tag` is recorded with a hit.
template <int MaxStack, bool kBoxes = false>
__device__ __forceinline__ uint32_t traverse(const RayPre &r, const BVHNode *__restrict__ nodes,
                                             const TriRecord *__restrict__ tris, uint32_t nprims, int start,
                                             HitState &h, const LaneStack &st, int sp0, uint32_t inst, int tag,
                                             int skip = kNoSkip) {
  auto leafTest = [&](int leaf, int) __attribute__((always_inline)) {
    intersect_leaf<kBoxes>(r, tris, leaf, nprims, inst, tag, h);
  };
  return walk_batched<MaxStack, decltype(leafTest) &>(r, nodes, nprims, start, h, st, sp0, skip, leafTest);
}

// The plain trace: no proposal and no fetch counts. A wave keeps its 64 lanes busy. A lane whose ray has
// ended gets the next one (with 64 fixed rays per wave, which walk until the longest one ends, 17 of 64
// lanes are active on average), and once there is none left, a part of another lane's ray: the far subtree
// at the bottom of its stack. The lanes fetch their nodes together.
//
// Node fetch: four lanes load one lane's node, 16 B each, into LDS (global_load_lds), for each of the
// four lanes of the quad in turn; then every lane reads its node from LDS. Where each lane loads its
// own node, every 16-byte load is one access of the vector cache, whose address and data paths were
// busy 94 % of the time; the 64 contiguous bytes of a quad are one access for four lanes. Lane j loads
// part j ^ k of the node of lane k of its quad, so that neighbouring lanes' reads of one part fall into
// different banks. A lane without a node loads the root's.
//
// Rays: the waves of one XCD (workgroups are dealt to the eight XCDs in turn) take chunks of rays from
// one contiguous share of them, so that its L2 holds what neighbouring rays meet (L2 misses 292 -> 222
// million), then from the others' shares. A wave's first chunk is its own, the next ones are taken from a
// counter per share, each on a line of its own: updates of one line by all CUs pass one at a time, about
// 10 ns each (one counter for all cost 80 us for the first chunks alone). Chunks hold 64 rays or
// 32 (128 and 256 measured no better), or, where that is less, an equal part of the rays for every wave, but
// two at least (1 to 4 measured alike, 16 slower below 100,000 rays). A wave hands rays out when kRefill lanes
// are free: 4 to 16 measured alike, 32 2 % slower.
//
// Split rays: a trace of few rays, and the end of one of many, otherwise waits for single lanes that walk
// the longest rays (the longest meets 1,093 nodes, the average one 131). Hits are the minimum over (t,
// inst, prim), so the parts of a ray may be walked in any order and by any lane; what order adds is the
// bound, so the lanes of one ray share it. Every kSplitEvery steps with kSplitIdle idle lanes: 24 and 2
// measured best of 8 to 64 and 1 to 16 (8 and 4: 8 % slower at 65,536 rays through 16,384 triangles).
//
// Times before and after, us, half primary and half bounce rays:
//   through          512 rays     8,192       65,536      262,144     1,048,352    8,388,608
//     16,384 tris   160 -> 40   185 -> 51   198 -> 69   226 -> 124    409 -> 271   2174 -> 1503
//    262,144        270 -> 51   404 -> 70   443 -> 145  481 -> 326    941 -> 639   4844 -> 3364
//  4,194,304        429 -> 62   584 -> 101  703 -> 226  811 -> 500   1610 -> 1041  7971 -> 5571
// What bounds the largest now is what the vector cache misses: 56 % of its accesses, 28 % of those L2 too, for
// 27.5 GB of which the bounce half takes 26 (6.2 KB a ray); the smallest the longest chain of nodes. Only very
// many coherent rays were faster with one ray per lane, as their waves stay together by themselves: 8 million
// primary rays through 4 instances of 60,000 triangles 2,270 -> 2,580, 16 of 20,000 2,650 -> 2,990, through
// 60,000 triangles 1,720 -> 1,860, 240,000 2,550 -> 2,800 (their bounce rays 6,450 -> 3,880; 20,000 triangles
// 1,555 -> 1,330, a million 3,930 -> 3,880). The host cannot tell them from others. Handing rays out only to a
// whole free wave gave 0 to 9 % of it back and doubled the bounce rays' time; a node that all lanes share,
// loaded without LDS, cost all traces 2 to 10 %.
// The node test stays box_hit, as in every other walk: a test of 18 instead of 26 instructions (planes by one
// FMA each, widened for its rounding) gained 1 % and found hits that box_hit does not enter, for rays in the
// plane of a box's face.
constexpr int kRefill = 12;
constexpr int kSplitIdle = 24;
constexpr uint32_t kSplitEvery = 2;
constexpr uint32_t kShares = 8;
constexpr uint32_t kShareWords = 32;  // a counter's 128-byte line
constexpr uint32_t kChunk = 64, kMinChunk = 2;
static_assert(kShares * kShareWords <= kTraceHeaderWords, "the counters lie before the spill area");
// 4 KB of nodes, 13 stack entries and the bounds per wave: 10 workgroups (20 waves) fit a CU. 11 entries
// and 11 workgroups measured the same.
constexpr int kStreamStack = 13;
constexpr int kStreamBlocksPerCU = 10;
static_assert((kMaxStack - kStreamStack) * kStreamBlocksPerCU <= (kMaxStack - kLdsStack) * kBlocksPerCU,
              "the spill area is sized for the other kernels");

struct StreamLds {
  float4 node[kTraceBlock / 64][4 * 64];  // also scratch between two fetches
  uint32_t stack[kStreamStack][kTraceBlock];
  float best[kTraceBlock];  // split rays: closest hit distance so far, at the ray's owner
};

typedef __attribute__((address_space(3))) void LdsVoid;
typedef __attribute__((address_space(1))) void GlobalVoid;

__device__ __forceinline__ bool lane_of(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

__device__ __forceinline__ uint32_t lane_rank(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The value of lane `src`; all lanes take part.
template <class T>
__device__ __forceinline__ T from_lane(const T &v, int src) {
  static_assert(sizeof(T) % 4 == 0, "moved word by word");
  int w[sizeof(T) / 4];
  __builtin_memcpy(w, &v, sizeof(T));
  for (int &x : w) x = __builtin_amdgcn_ds_bpermute(src * 4, x);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// Keeps the LDS accesses of a wave's lanes, which the LDS executes in order, in program order.
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int K>
__device__ __forceinline__ void fetch_quad_lane(const BVHNode *__restrict__ nodes, uint32_t at, uint32_t part,
                                                char *stage) {
  const uint32_t theirs = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)at, K * 0x55, 0xF, 0xF, true);
  __builtin_amdgcn_global_load_lds((GlobalVoid *)((const char *)nodes + (theirs | (part ^ (K * 16u)))),
                                   (LdsVoid *)(stage + K * 1024), 16, 0, 0);
}

// `at`: byte offset of the lane's node. All 64 lanes take part.
__device__ __forceinline__ void fetch_nodes(const BVHNode *__restrict__ nodes, uint32_t at, char *stage) {
  const uint32_t part = (threadIdx.x & 3u) * 16u;
  fetch_quad_lane<0>(nodes, at, part, stage);
  fetch_quad_lane<1>(nodes, at, part, stage);
  fetch_quad_lane<2>(nodes, at, part, stage);
  fetch_quad_lane<3>(nodes, at, part, stage);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Chunks of the rays, and of each share.
struct Shares {
  uint32_t chunk, chunks, seg;
};
__device__ __forceinline__ Shares shares_of(uint32_t count, uint32_t chunk) {
  Shares s;
  s.chunk = chunk;
  s.chunks = (count - 1) / chunk + 1;
  s.seg = (s.chunks - 1) / kShares + 1;
  return s;
}
// Chunk c of share x, counted over all rays (beyond the last one if the share has no more).
__device__ __forceinline__ uint32_t share_chunk(const Shares &s, uint32_t x, uint32_t c) {
  return c < s.seg ? x * s.seg + c : 0xFFFFFFFFu;
}
// Chunks of share x that its own waves take first, one each.
__device__ __forceinline__ uint32_t share_static(uint32_t x) {
  return (gridDim.x + kShares - 1 - x) / kShares * (kTraceBlock / 64);
}

// The wave's next chunk: `left` rays from `next` on; false when all shares are used up. `share` counts
// the shares that the wave found used up; their order differs between XCDs.
__device__ __forceinline__ bool stream_chunk(uint32_t *__restrict__ work, uint32_t count, const Shares &s,
                                             uint32_t &share, uint32_t &next, uint32_t &left) {
  for (; share < kShares; ++share) {
    const uint32_t x = (blockIdx.x ^ __builtin_bitreverse32(share << 29)) % kShares;
    const uint32_t first = share_static(x);
    uint32_t c = share_chunk(s, x, first);
    if (c < s.chunks) {
      uint32_t base = 0;
      if ((threadIdx.x & 63) == 0) base = atomicAdd(work + kShareWords * x, 1u);
      c = share_chunk(s, x, first + __builtin_amdgcn_readfirstlane(base));
      if (c < s.chunks) {
        next = c * s.chunk;
        left = min(s.chunk, count - next);
        return true;
      }
    }
  }
  return false;
}

// Split rays: `own` is the lane that holds the ray's hit, itself for a lane without a part of another's.
// Takes the hits of the lanes that have ended their parts to the owners (the closest one by the rule of
// hit_closer: first the distance, then instance and primitive) and tells at stage + kSplitActive, a word
// per lane, whether a lane that still walks belongs to the owner. All 64 lanes take part.
constexpr int kSplitActive = 1792;

__device__ __forceinline__ void settle_parts(char *stage, int lane, int own, bool busy, HitState &h) {
  uint32_t *sT = (uint32_t *)stage;
  unsigned long long *sKey = (unsigned long long *)(stage + 256);
  float *sHitT = (float *)(stage + 768), *sU = (float *)(stage + 1024), *sV = (float *)(stage + 1280);
  int *sLeaf = (int *)(stage + 1536);
  uint32_t *sActive = (uint32_t *)(stage + kSplitActive);
  const bool hit = h.prim >= 0, owner = own == lane;
  const uint32_t t = hit ? ford(h.t + 0.0f) : ~0u;  // + 0: distances -0 and +0 are equal
  const unsigned long long key = hit ? ((unsigned long long)h.inst << 32 | (uint32_t)h.prim) : ~0ull;
  lds_order();
  sT[lane] = owner ? t : ~0u;
  sKey[lane] = owner ? key : ~0ull;
  sActive[lane] = 0;
  lds_order();
  const bool found = !busy && !owner && hit;
  if (found) atomicMin(&sT[own], t);
  if (busy) sActive[own] = 1;
  lds_order();
  const bool closest = found && sT[own] == t;
  if (owner && sT[lane] != t) sKey[lane] = ~0ull;
  lds_order();
  if (closest) atomicMin(&sKey[own], key);
  lds_order();
  if (closest && sKey[own] == key) {
    sHitT[own] = h.t;
    sU[own] = h.u;
    sV[own] = h.v;
    sLeaf[own] = h.leaf;
  }
  lds_order();
  if (owner && (sT[lane] != t || sKey[lane] != key)) {
    h.t = sHitT[lane];
    h.u = sU[lane];
    h.v = sV[lane];
    h.leaf = sLeaf[lane];
    h.prim = (int)(uint32_t)sKey[lane];
    h.inst = (uint32_t)(sKey[lane] >> 32);
  }
}

// Traces rays [0, count), `chunk` at a time: begin(i) sets up ray i in the caller's `ray` and `h`,
// leaf(position) tests a leaf, end(i) stores ray i's hit. `work`: kShares counters, zeroed (read only if
// there are more chunks than waves), kShareWords apart. `spill`: this lane's kMaxStack - kStreamStack
// words. The tree has fewer than kSmallTreePrims primitives.
template <class Begin, class Leaf, class End>
__device__ __forceinline__ void trace_stream(const BVHNode *__restrict__ nodes, uint32_t nprims, uint32_t count,
                                             uint32_t chunk, uint32_t *__restrict__ work, RayPre &ray, HitState &h,
                                             StreamLds &lds, uint32_t *__restrict__ spill, Begin &&begin,
                                             Leaf &&leaf, End &&end) {
  constexpr uint32_t kDone = 0x80000000u, kNoRay = 0xFFFFFFFFu;
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t waveInBlock = __builtin_amdgcn_readfirstlane(tid >> 6);
  char *stage = (char *)lds.node[waveInBlock];
  float *best = lds.best + waveInBlock * 64;
  const uint32_t quad = tid & 3u;
  const char *mine = stage + quad * 1024u + (tid & 60u) * 16u;
  // Queued leaves as child codes, as in walk_batched.
  int q0 = -1, q1 = -1, q2 = -1, q3 = -1, nq = 0;
  auto enqueue = [&](int code) __attribute__((always_inline)) {
    q3 = q2;
    q2 = q1;
    q1 = q0;
    q0 = code;
    ++nq;
  };
  const uint32_t inner = nprims > 1 ? nprims - 1 : 0u;  // a node at or above it: none (or a malformed tree)
  // In every iteration a lane with a ray fetches a node (each at most once) or tests its queued leaves.
  const uint32_t limit = 4u * nprims + 8u;
  uint32_t ri = kNoRay, began = 0, node = kDone;
  int own = lane;
  int sp = 0, bot = 0;  // the stack's entries are [bot, sp)
  // Wave-uniform: the chunk's remaining rays, and which lanes have a node to visit and queued leaves.
  const Shares shares = shares_of(count, chunk);
  uint32_t share = 0, next = 0, left = 0;
  const uint32_t c = share_chunk(shares, blockIdx.x % kShares, blockIdx.x / kShares * (kTraceBlock / 64) + waveInBlock);
  if (c < shares.chunks) {
    next = c * chunk;
    left = min(chunk, count - next);
  }
  bool more = true;
  uint64_t walk = 0, wait = 0;
  for (uint32_t it = 0;; ++it) {
    const uint64_t idle = ~(walk | wait);
    if (__builtin_expect(more && __popcll(idle) >= kRefill, 0)) {
      const bool free = lane_of(idle);
      if (free && ri != kNoRay) {
        end(ri);
        ri = kNoRay;
      }
      if (left == 0) more = stream_chunk(work, count, shares, share, next, left);
      if (!more) {
        best[lane] = h.t;
        continue;
      }
      const uint32_t rank = lane_rank(idle);
      if (free && rank < left) {
        ri = next + rank;
        begin(ri);
        began = it;
        sp = bot = 0;
        if (inner > 0)
          node = 0;
        else if (nprims == 1)
          enqueue(~0);
      }
      const uint32_t took = min((uint32_t)__popcll(idle), left);
      next += took;
      left -= took;
      walk = __ballot(node < inner);
      wait = __ballot(nq > 0);
    }
    if (!more && __builtin_expect(idle == ~0ull || (__popcll(idle) >= kSplitIdle && it % kSplitEvery == 0), 0)) {
      const bool busy = !lane_of(idle);
      settle_parts(stage, lane, own, busy, h);
      if (!busy) {
        if (own == lane && ri != kNoRay && ((const uint32_t *)(stage + kSplitActive))[lane] == 0) {
          end(ri);
          ri = kNoRay;
        } else if (own != lane) {
          ri = kNoRay;
          own = lane;
        }
      }
      if (idle == ~0ull) break;
      // The k-th lane that gives takes the bottom of its stack to the k-th free lane.
      const bool free = !busy && ri == kNoRay, gives = busy && sp > bot && bot < kStreamStack;
      const uint64_t frees = __ballot(free), givers = __ballot(gives);
      if (frees && givers) {
        const uint32_t toRank = lane_rank(frees), fromRank = lane_rank(givers);
        uint32_t *from = (uint32_t *)stage, *entry = from + 64;
        lds_order();
        if (gives && fromRank < (uint32_t)__popcll(frees)) {
          from[fromRank] = lane;
          entry[fromRank] = lds.stack[bot][tid];
          ++bot;
        }
        lds_order();
        const bool takes = free && toRank < (uint32_t)__popcll(givers);
        const int src = takes ? (int)from[toRank] : lane;
        const RayPre theirs = from_lane(ray, src);
        const uint32_t theirRi = from_lane(ri, src);
        const int theirOwn = from_lane(own, src);
        if (takes) {
          ray = theirs;
          ri = theirRi;
          own = theirOwn;
          hit_init(h, best[own]);
          node = entry[toRank];
          began = it;
          sp = bot = 0;
        }
        walk = __ballot(node < inner);
        lds_order();
      }
    }
    if ((it & 4095u) == 4095u) {
      if (it - began > limit) {  // only a malformed tree
        node = kDone;
        nq = 0;
      }
      walk = __ballot(node < inner);
      wait = __ballot(nq > 0);
    }
    if (walk) fetch_nodes(nodes, lane_of(walk) ? node * (uint32_t)sizeof(BVHNode) : 0u, stage);
    if (lane_of(walk)) {
      const float4 a = *(const float4 *)(mine + (0u ^ quad) * 16u), b = *(const float4 *)(mine + (1u ^ quad) * 16u);
      const float4 d = *(const float4 *)(mine + (2u ^ quad) * 16u);
      const int2 child = *(const int2 *)(mine + (3u ^ quad) * 16u);
      // The stack's top, should both children fail: read ahead, so that no step waits for it.
      uint32_t top = lds.stack[min((uint32_t)sp - 1u, kStreamStack - 1u)][tid];
      float tn0, tn1, bound = h.t;
      if (!more) bound = fminf(bound, best[own]);
      // Lane masks rather than flags: they stay in scalar registers.
      const uint64_t h0 = __ballot(box_hit(ray, a.x, a.y, a.z, a.w, b.x, b.y, bound, tn0));
      const uint64_t h1 = __ballot(box_hit(ray, b.z, b.w, d.x, d.y, d.z, d.w, bound, tn1));
      const uint64_t n0 = __ballot(child.x >= 0), n1 = __ballot(child.y >= 0), near0 = __ballot(tn0 <= tn1);
      const uint64_t i0 = h0 & n0, i1 = h1 & n1, l0 = h0 & ~n0, l1 = h1 & ~n1;
      if (lane_of(l0 | l1)) {
        enqueue(lane_of(l0) ? child.x : child.y);
        if (lane_of(l0 & l1)) enqueue(child.y);
      }
      const uint64_t first0 = i0 & (~i1 | near0), push = i0 & i1;
      const uint64_t pop = walk & ~(i0 | i1) & __ballot(sp != bot);
      const uint64_t below = __ballot(sp < kStreamStack), above = __ballot(sp > kStreamStack);
      if (lane_of(push & below)) lds.stack[sp][tid] = (uint32_t)(lane_of(first0) ? child.y : child.x);
      if (__builtin_expect(push & ~below, 0)) {
        if (lane_of(push & ~below) && sp < kMaxStack)
          spill[sp - kStreamStack] = (uint32_t)(lane_of(first0) ? child.y : child.x);
      }
      if (__builtin_expect(pop & above, 0)) {
        if (lane_of(pop & above))  // an ordinary load: see stack_read
          top = sp <= kMaxStack ? __hip_atomic_load(&spill[sp - 1 - kStreamStack], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WAVEFRONT)
                                : kDone;
      }
      node = (uint32_t)(lane_of(first0) ? child.x : child.y);
      node = lane_of(i0 | i1) ? node : lane_of(pop) ? top : kDone;
      sp += (lane_of(push) ? 1 : 0) - (lane_of(pop) ? 1 : 0);
    }
    walk = __ballot(node < inner);
    wait = __ballot(nq > 0);
    // A lane that walks no further, or has no room for another node's two leaves (so that no queue is ever
    // full at the top of the loop), needs its leaves tested.
    if ((wait & (~walk | __ballot(nq > kLeafQueue - 2))) || 2 * __popcll(wait) >= __popcll(walk | wait)) {
      while (nq > 0) {
        const int code = q0;
        q0 = q1;
        q1 = q2;
        q2 = q3;
        --nq;
        leaf(~code);
      }
      if (!more && lane_of(wait))
        __hip_atomic_fetch_min(&best[own], h.t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      wait = 0;
    }
  }
}

}  // namespace gprt
