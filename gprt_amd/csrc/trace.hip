// Closest-hit traversal of the triangle LBVH for gfx950.
//
// The reference has no software traversal: closest hit comes from the Vulkan driver via
// TraceRay / vkCmdTraceRaysKHR (gprt/gprt_builtins.slang:105-124, gprt/gprt.cpp:9404); its
// conventions are kept: a ray {origin, tmin, direction, tmax} (RayDesc), an open interval
// tmin < t (gprt/gprt_fallbacks.slang:108,139) and a closest hit reporting PrimitiveIndex, t and
// barycentrics (samples/s2-hitPrograms/s2-0-triangles/deviceCode.slang:16-19).
//
// Kernel shape: workgroups of 128 lanes. A plain trace is streamed (trace_stream); in the general form a
// lane takes one ray, and beyond a full launch each wave takes 64 more from a global counter (load balance
// across rays of very different cost). One node fetch decides both children (64-byte node with both child
// boxes); leaf children are queued and tested in batches across the wave (the triangle test then runs for
// many lanes at once); the near inner child is descended and the far one pushed on a per-lane stack whose
// first entries live in LDS and the rest in a per-lane global spill area. A binary radix tree over distinct
// 64-bit keys is at most 64 levels deep, so 64 entries always suffice.
//
// With a proposal, each ray first traverses the subtree of its proposed treelet (a real hit found
// there becomes the starting (t, primID)), then the ordinary traversal from the root runs with
// that tighter bound; the lexicographic (t, primID) rule makes the result identical.
#include <algorithm>
#include <climits>

#include "bvh.hpp"
#include "device_common.hpp"
#include "internal.hpp"
#include "traverse.hpp"

namespace gprt {

namespace {

// The general form: with a proposal, per-ray fetch counts, or trees of kSmallTreePrims primitives and more.
// kBoxes: the leaves are box primitives.
template <bool kBoxes>
__global__ void __launch_bounds__(kTraceBlock)
    k_trace(const BVHNode *__restrict__ nodes, const TriRecord *__restrict__ tris, uint32_t nprims,
            const GPRTRay *__restrict__ rays, GPRTHit *__restrict__ hits, uint32_t count,
            uint32_t *__restrict__ work, uint32_t *__restrict__ spill, const int32_t *__restrict__ proposal,
            const int32_t *__restrict__ classRoot, uint32_t numClasses, uint32_t *__restrict__ visitsOut) {
  __shared__ uint32_t s_stack[kLdsStack][kTraceBlock];
  const int tid = threadIdx.x;
  const uint32_t gtid = blockIdx.x * kTraceBlock + tid;
  const LaneStack st{s_stack, tid, spill + (size_t)gtid * (kMaxStack - kLdsStack)};
  const int l = tid & 63;

  const bool more = count > gridDim.x * kTraceBlock;
  do {
    const uint32_t base = next_rays(work, more);
    if (base >= count) break;
    const uint32_t ri = base + (uint32_t)l;
    if (ri < count) {
      const GPRTRay ray = load_ray_stream(rays + ri);
      const RayPre r = ray_setup(ray.ox, ray.oy, ray.oz, ray.tmin, ray.dx, ray.dy, ray.dz);
      HitState h;
      hit_init(h, ray.tmax);
      uint32_t visits = 0;
      int skip = kNoSkip;
      if (proposal) {
        const int32_t c = proposal[ri];
        if (c >= 0 && (uint32_t)c < numClasses) {
          const int32_t root = classRoot[c];
          // A treelet rooted at the tree's root (cut depth 0) would only repeat the full pass.
          if (root != 0) {
            visits += traverse<kMaxStack, kBoxes>(r, nodes, tris, nprims, root, h, st, 0, 0u, -1);
            skip = root;  // searched completely: the full pass does not enter it again
          }
        }
      }
      visits +=
          traverse<kMaxStack, kBoxes>(r, nodes, tris, nprims, nprims == 1 ? ~0 : 0, h, st, 0, 0u, -1, skip);
      if (visitsOut) visitsOut[ri] = visits;
      GPRTHit o;
      o.t = h.prim >= 0 ? h.t : ray.tmax;
      o.primID = h.prim;
      o.u = h.u;
      o.v = h.v;
      store_hit_stream(hits + ri, o);
    }
  } while (more);
}

// The plain trace.
template <bool kBoxes>
__global__ void __launch_bounds__(kTraceBlock)
    k_trace_stream(const BVHNode *__restrict__ nodes, const TriRecord *__restrict__ tris, uint32_t nprims,
                   const GPRTRay *__restrict__ rays, GPRTHit *__restrict__ hits, uint32_t count,
                   uint32_t chunk, uint32_t *__restrict__ work, uint32_t *__restrict__ spill) {
  __shared__ StreamLds lds;
  const uint32_t gtid = blockIdx.x * kTraceBlock + threadIdx.x;
  RayPre r = {};
  HitState h;
  hit_init(h, 0.0f);
  trace_stream(
      nodes, nprims, count, chunk, work, r, h, lds, spill + (size_t)gtid * (kMaxStack - kStreamStack),
      [&](uint32_t ri) __attribute__((always_inline)) {
        const GPRTRay ray = load_ray_stream(rays + ri);
        r = ray_setup(ray.ox, ray.oy, ray.oz, ray.tmin, ray.dx, ray.dy, ray.dz);
        hit_init(h, ray.tmax);
      },
      [&](int pos) __attribute__((always_inline)) { intersect_leaf<kBoxes, true>(r, tris, pos, nprims, 0u, -1, h); },
      [&](uint32_t ri) __attribute__((always_inline)) {
        store_hit_stream(hits + ri, GPRTHit{h.t, h.prim, h.u, h.v});  // t is still tmax if nothing was hit
      });
}

}  // namespace

uint32_t *ensure_trace_scratch(Context *ctx, hipStream_t s, int spillWordsPerLane) {
  const unsigned blocks = (unsigned)ctx->cuCount * kBlocksPerCU;
  const size_t need = (size_t)blocks * kTraceBlock * (size_t)spillWordsPerLane * 4 + kTraceHeaderWords * 4;
  if (need > ctx->traceBytes) {
    if (ctx->traceScratch) {
      hipStreamSynchronize(s);
      hipFree(ctx->traceScratch);
      ctx->traceScratch = nullptr;
      ctx->traceBytes = 0;
    }
    if (!hip_ok(hipMalloc(&ctx->traceScratch, need), "hipMalloc(trace scratch)")) return nullptr;
    ctx->traceBytes = need;
  }
  return (uint32_t *)ctx->traceScratch;
}

// How `count` rays are traced through a tree of n leaves. Plain: trace_stream by a full launch, in one chunk
// of equal size for every wave where that holds at most kChunk rays (and then without counters), else in
// chunks of half of kChunk for large trees, whose rays differ most (us for 0.52 / 1.05 / 8.4 million rays
// in chunks of 64 and 32: 4.2 million triangles 798 / 1141 / 5661 and 690 / 1068 / 5583, 262,144 461 / 649 /
// 3360 and 403 / 625 / 3341; 16,384 196 / 268 / 1455 and 196 / 285 / 1495). General: one ray per lane, in as
// many workgroups as that needs (a full launch of waves that each ask a counter cost 80 us), persistent
// beyond a full launch.
TraceGrid trace_grid(const Context *ctx, uint32_t n, uint32_t count, bool plain, unsigned blocksPerCU) {
  const unsigned perCU = blocksPerCU ? blocksPerCU : UINT_MAX;
  if (plain) {
    const unsigned blocks = (unsigned)ctx->cuCount * std::min<unsigned>(perCU, kStreamBlocksPerCU);
    const uint32_t waves = blocks * (kTraceBlock / 64);
    const uint32_t even = std::max(kMinChunk, (count - 1) / waves + 1);
    const uint32_t chunk = even <= kChunk ? even : n < 1u << 16 ? kChunk : kChunk / 2;
    // Of each share's waves and chunks (trace_stream's numbers).
    const uint32_t least = blocks / kShares * (kTraceBlock / 64), seg = (count - 1) / chunk / kShares + 1;
    return TraceGrid{blocks, seg <= least ? 0u : kShares * kShareWords, chunk};
  }
  const unsigned blocks = (unsigned)ctx->cuCount * std::min<unsigned>(perCU, kBlocksPerCU);
  const unsigned needed = (count - 1) / kTraceBlock + 1;
  return TraceGrid{std::min(blocks, needed), needed > blocks ? 1u : 0u, 0u};
}

bool trace_closest_ex(Context *ctx, hipStream_t s, Accel *a, const void *rays, void *hits, uint32_t count,
                      const int32_t *proposal, const int32_t *classRoot, uint32_t numClasses, uint32_t *visits,
                      unsigned blocksPerCU) {
  if (count == 0) return true;
  uint32_t *work = ensure_trace_scratch(ctx, s, kMaxStack - kLdsStack);
  if (!work) return false;
  const bool plain = !proposal && !visits && a->n < kSmallTreePrims;
  const TraceGrid g = trace_grid(ctx, a->n, count, plain, blocksPerCU);
  if (g.counters) fill_u32(ctx, s, work, 0u, g.counters);
  if (plain) {
    auto go = [&](auto kernel) {
      launch(ctx, s, "trace_closest", kernel, dim3(g.blocks), dim3(kTraceBlock), 0, (const BVHNode *)a->nodes,
             (const TriRecord *)a->tris, a->n, (const GPRTRay *)rays, (GPRTHit *)hits, count, g.chunk,
             work, work + kTraceHeaderWords);
    };
    a->kind == AccelKind::AABBs ? go(k_trace_stream<true>) : go(k_trace_stream<false>);
    return true;
  }
  const char *name = proposal ? "trace_closest_proposal" : "trace_closest";
  auto go = [&](auto kernel) {
    launch(ctx, s, name, kernel, dim3(g.blocks), dim3(kTraceBlock), 0, (const BVHNode *)a->nodes,
           (const TriRecord *)a->tris, a->n, (const GPRTRay *)rays, (GPRTHit *)hits, count, work,
           work + kTraceHeaderWords, proposal, classRoot, numClasses, visits);
  };
  if (a->kind == AccelKind::AABBs)
    go(k_trace<true>);
  else
    go(k_trace<false>);
  return true;
}

bool trace_closest(Context *ctx, hipStream_t s, Accel *a, const void *rays, void *hits, uint32_t count) {
  return trace_closest_ex(ctx, s, a, rays, hits, count, nullptr, nullptr, 0, nullptr);
}

}  // namespace gprt
