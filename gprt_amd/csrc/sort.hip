// Stable LSD radix sort (keys 32/64-bit, optional 32/64-bit payload) for gfx950.
//
// Semantics follow GPRT's buffer sort (gprt/gprt.cpp:8821-9073, gprt/gprt_sort.slang): ascending,
// stable, in place, payload follows its key. The reference runs 16 passes of 4-bit digits, each
// as five dispatches (count, count-reduce, scan, scan-add, scatter; gprt/gprt_sort.slang:109-637).
// This implementation is a one-sweep design instead:
//  * k_hist reads the keys once and builds the digit histograms of every pass (LDS atomics);
//  * k_hist_scan turns them into global digit offsets and marks passes whose digit is constant
//    over all keys as inactive (they would be identity permutations);
//  * one k_onesweep launch per pass: a tile ticket, wave64 multisplit ranking (BITS ballots per
//    key give each lane the mask of peers with the same digit), per-digit decoupled look-back
//    across tiles (four predecessors per step), a stable local reorder in LDS and a global write
//    in digit runs;
//  * ping-pong buffers are picked on the device from the active-pass mask, and k_final_copy
//    moves the result back when an odd number of passes ran — no host round trip, so the whole
//    sort can be captured in a hipGraph.
// Up to 16,384 keys, where those launches would be all the time there is, k_rank places every key by
// comparing it with all others and k_copy_pairs puts the result back: two launches.
#include <algorithm>

#include "device_common.hpp"
#include "internal.hpp"

namespace gprt {

namespace {

constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagInc = 2u << 30;
constexpr uint32_t kValueMask = (1u << 30) - 1u;

// State layout (uint32 words):
//   [0, P*R)            digit counts, then exclusive digit starts, per pass
//   [P*R]               active-pass mask
//   [P*R + 1, +P)       tile tickets per pass
//   [P*R + 32, ...)     look-back status [P][tiles][R]
struct SortState {
  uint32_t *hist;
  uint32_t *activeMask;
  uint32_t *tickets;
  uint32_t *status;
};

__host__ __device__ inline SortState state_view(void *base, int passes, int radix) {
  uint32_t *p = (uint32_t *)base;
  SortState s;
  s.hist = p;
  s.activeMask = p + (size_t)passes * radix;
  s.tickets = s.activeMask + 1;
  s.status = p + (size_t)passes * radix + 32;
  return s;
}

template <typename KT>
__device__ __forceinline__ uint32_t digit_of(KT k, int shift, uint32_t mask) {
  return (uint32_t)(k >> shift) & mask;
}

// ------------------------------------------------------------------------------------------------
// Histogram of all passes.
// ------------------------------------------------------------------------------------------------
// 512 threads, up to four workgroups a CU: all of its wave slots (with 256, half of them: 16 million
// 32-bit pairs sorted in 407 us, now 397, 4 million in 160, now 152), and half the additions at the end.
constexpr int kHistThreads = 512;

// Its workgroups: 8,192 keys each, of which fewer mean fewer additions at the end (4 million 32-bit pairs
// sorted in 132 us, with 4,096 each 139), but 4,096 while every one can have a CU to itself, as its additions
// to one counter pass one at a time (a million equal 32-bit keys 48 and 36 us); at most four a CU.
inline size_t hist_blocks(size_t n, size_t cus) {
  const size_t blocks = std::max((n + 8191) / 8192, std::min((n + 4095) / 4096, cus));
  return std::max<size_t>(1, std::min(blocks, 4 * cus));
}

template <typename KT, int BITS>
__global__ void __launch_bounds__(kHistThreads)
    k_hist(const KT *__restrict__ keys, size_t n, int loBit, int hiBit, int passes, uint32_t *__restrict__ hist) {
  constexpr int R = 1 << BITS;
  extern __shared__ uint32_t s_h[];  // [passes][R]
  for (int i = threadIdx.x; i < passes * R; i += blockDim.x) s_h[i] = 0;
  __syncthreads();
  // kHistBatch keys per thread at a time, each load coalesced over the grid: the batch's loads are
  // all in flight before the first key's counts (a load per thread at a time leaves HBM idle).
  constexpr int kHistBatch = 8;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += stride * kHistBatch) {
    KT k[kHistBatch];
#pragma unroll
    for (int u = 0; u < kHistBatch; ++u) {
      const size_t i = i0 + (size_t)u * stride;
      k[u] = i < n ? keys[i] : (KT)0;
    }
#pragma unroll
    for (int u = 0; u < kHistBatch; ++u) {
      if (i0 + (size_t)u * stride >= n) break;  // the rest of the batch is past the end too
      for (int p = 0; p < passes; ++p) {
        const int shift = loBit + p * BITS;
        const int bits = (hiBit - shift) < BITS ? (hiBit - shift) : BITS;
        const uint32_t d = digit_of(k[u], shift, (1u << bits) - 1u);
        atomicAdd(&s_h[p * R + d], 1u);
      }
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < passes * R; j += blockDim.x) {
    const uint32_t c = s_h[j];
    if (c) atomicAdd(&hist[j], c);
  }
}

// Exclusive scan of every pass's histogram; a pass is active unless one digit holds every key.
template <int BITS>
__global__ void __launch_bounds__(256) k_hist_scan(uint32_t *__restrict__ hist, uint32_t *__restrict__ activeMask,
                                                   int passes, uint32_t n) {
  constexpr int R = 1 << BITS;
  constexpr int PER = (R + 255) / 256;
  __shared__ uint32_t s_w[4];
  __shared__ uint32_t s_any;
  const int tid = threadIdx.x;
  uint32_t mask = 0;
  for (int p = 0; p < passes; ++p) {
    uint32_t c[PER];
    uint32_t sum = 0;
    bool full = false;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = tid * PER + j;
      c[j] = d < R ? hist[p * R + d] : 0u;
      full |= (c[j] == n);
      sum += c[j];
    }
    if (tid == 0) s_any = 0;
    __syncthreads();
    if (full) s_any = 1;
    const uint32_t incl = wave_incl_sum(sum);
    if ((tid & 63) == 63) s_w[tid >> 6] = incl;
    __syncthreads();
    uint32_t off = incl - sum;
    for (int w = 0; w < (tid >> 6); ++w) off += s_w[w];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = tid * PER + j;
      if (d < R) hist[p * R + d] = off;
      off += c[j];
    }
    __syncthreads();
    if (!s_any) mask |= 1u << p;
    __syncthreads();
  }
  if (tid == 0) *activeMask = mask;
}

// ------------------------------------------------------------------------------------------------
// One pass: ticketed tiles, wave multisplit ranking, per-digit look-back, LDS reorder, scatter.
// ------------------------------------------------------------------------------------------------
template <int VB>
struct ValType;
template <>
struct ValType<0> {
  using T = uint32_t;
};
template <>
struct ValType<32> {
  using T = uint32_t;
};
template <>
struct ValType<64> {
  using T = uint64_t;
};

// Writes element `at` of fewer than 2^30: 32-bit offsets of 32-bit elements need one register less.
template <typename T>
__device__ __forceinline__ void put_at(T *base, uint32_t at, T v) {
  if constexpr (sizeof(T) == 4)
    *(T *)((char *)base + at * 4u) = v;
  else
    base[at] = v;
}

// A lane's ITEMS elements of a wave's consecutive ones, of which the first `here` exist (all if `whole`).
template <int ITEMS, typename T>
__device__ __forceinline__ void load_items(const T *__restrict__ p, bool whole, uint32_t here, T none, T (&out)[ITEMS]) {
  const uint32_t l = threadIdx.x & 63u;
  if (whole) {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) out[j] = p[j * 64u + l];
  } else {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) out[j] = j * 64u + l < here ? p[j * 64u + l] : none;
  }
}

// A pass alternates between memory (its loads, the look-back, its writes) and ranking, which keeps the
// vector units busy for a third of the time (14,000 of 45,000 cycles a tile of 16,384); two workgroups of
// 1,024 threads a CU overlap the two. That takes 64 registers per thread and 80 KB of LDS: 16-bit wave
// counts and positions, digits computed again rather than kept, payloads loaded once the keys are in LDS,
// few writes at a time, and a compiler that is kept from mixing the ranking of several keys and from
// holding both halves of a pair of positions. Wider keys or payloads fill the LDS with one workgroup. A copy
// of the input and the sort, us: 67 million 32-bit pairs 1597 -> 1472, keys 1195 -> 970, 16 million pairs
// 443 -> 378; 16 million 64-bit pairs 1477 -> 1267 (fewer registers).
template <typename KT, int VB, int THREADS>
constexpr bool kTwoPerCU = THREADS == 1024 && sizeof(KT) == 4 && VB <= 32;

template <typename KT, int VB, int BITS, int THREADS, int ITEMS>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(kTwoPerCU<KT, VB, THREADS> ? 8 : 1)))
    k_onesweep(KT *__restrict__ keys0, KT *__restrict__ keys1, void *__restrict__ vals0, void *__restrict__ vals1,
               uint32_t n, int pass, int shift, int hiBit, void *__restrict__ stateBase, int passes,
               uint32_t numTiles) {
  using VT = typename ValType<VB>::T;
  constexpr int R = 1 << BITS;
  constexpr int NB = VB && kTwoPerCU<KT, VB, THREADS> ? 2 : 8;  // keys per thread written at a time: more need more registers
  constexpr int W = THREADS / 64;
  constexpr int TILE = THREADS * ITEMS;
  constexpr int DPT = (R + THREADS - 1) / THREADS;  // digits per thread
  constexpr size_t KBYTES = sizeof(KT) * TILE;
  constexpr size_t VBYTES = VB ? sizeof(VT) * TILE : 0;
  constexpr size_t BUFBYTES = KBYTES > VBYTES ? KBYTES : VBYTES;

  __shared__ __attribute__((aligned(16))) unsigned char s_buf[BUFBYTES];
  __shared__ uint16_t s_whist[W][R];
  __shared__ uint32_t s_tdigit[R];
  __shared__ uint32_t s_gbase[R];
  __shared__ uint32_t s_wtot[W];
  __shared__ uint32_t s_tile;

  SortState st = state_view(stateBase, passes, R);
  const uint32_t active = *st.activeMask;
  if (!((active >> pass) & 1u)) return;
  const int before = __builtin_popcount(active & ((1u << pass) - 1u));
  const KT *__restrict__ src = (before & 1) ? keys1 : keys0;
  KT *__restrict__ dst = (before & 1) ? keys0 : keys1;
  const VT *__restrict__ vsrc = (const VT *)((before & 1) ? vals1 : vals0);
  VT *__restrict__ vdst = (VT *)((before & 1) ? vals0 : vals1);

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int bits = (hiBit - shift) < BITS ? (hiBit - shift) : BITS;
  const uint32_t dmask = (1u << bits) - 1u;

  if (tid == 0) s_tile = ticket(&st.tickets[pass]);
  for (int i = tid; i < W * R / 2; i += THREADS) ((uint32_t *)&s_whist[0][0])[i] = 0u;
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
  const size_t tileBase = (size_t)tile * TILE;
  const size_t waveBase = tileBase + (size_t)w * (ITEMS * 64);
  const uint32_t valid = (n - tileBase) < (size_t)TILE ? (uint32_t)(n - tileBase) : (uint32_t)TILE;

  KT k[ITEMS];
  uint32_t pos[ITEMS / 2];  // two 16-bit positions each
  const KT *__restrict__ wsrc = src + waveBase;
  const VT *__restrict__ wvsrc = vsrc + (VB ? waveBase : 0);
  const uint32_t here = valid > (uint32_t)w * (ITEMS * 64) ? valid - (uint32_t)w * (ITEMS * 64) : 0u;
  load_items<ITEMS>(wsrc, valid == TILE, here, ~(KT)0, k);

  // The payloads: in small workgroups loaded with the keys, which hides their latency best, in large
  // ones once the keys are in LDS, when their registers are free.
  constexpr bool kEarlyVals = VB != 0 && THREADS == 256;
  VT ve[VB ? ITEMS : 1];
  if constexpr (kEarlyVals) load_items<ITEMS>(wvsrc, valid == TILE, here, (VT)0, ve);

  // Wave multisplit: peers with the same digit, rank among them, wave-private running counts.
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t dj = digit_of(k[j], shift, dmask);
    const uint64_t m = match_digit<BITS>(dj, ~0ull);
    const uint32_t r = mask_rank(m);
    const uint32_t c = (uint32_t)__popcll(m);
    const uint32_t pre = s_whist[w][dj];
    if (r == 0) s_whist[w][dj] = (uint16_t)(pre + c);
    pos[j / 2] = j & 1 ? pos[j / 2] | (pre + r) << 16 : pre + r;
    if constexpr (kTwoPerCU<KT, VB, THREADS>) {
      asm volatile("" : "+v"(pos[j / 2]));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();

  // Tile digit counts; wave offsets become exclusive; publish aggregates as early as possible.
  uint32_t cnt[DPT];
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    const int dd = tid * DPT + q;
    cnt[q] = 0;
    if (dd < R) {
      uint32_t sum = 0;
#pragma unroll
      for (int ww = 0; ww < W; ++ww) {
        const uint32_t c = s_whist[ww][dd];
        s_whist[ww][dd] = (uint16_t)sum;
        sum += c;
      }
      cnt[q] = sum;
      uint32_t *slot = &st.status[((size_t)pass * numTiles + tile) * R + dd];
      st_agent(slot, (tile == 0 ? kFlagInc : kFlagAgg) | sum);
    }
  }

  // Local exclusive scan of the tile's digit counts (thread-contiguous digits).
  {
    uint32_t tsum = 0;
#pragma unroll
    for (int q = 0; q < DPT; ++q) tsum += cnt[q];
    const uint32_t incl = wave_incl_sum(tsum);
    if (l == 63) s_wtot[w] = incl;
    __syncthreads();
    uint32_t off = incl - tsum;
    for (int ww = 0; ww < w; ++ww) off += s_wtot[ww];
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
      const int dd = tid * DPT + q;
      if (dd < R) s_tdigit[dd] = off;
      off += cnt[q];
    }
  }

  // Per-digit look-back over preceding tiles.
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    const int dd = tid * DPT + q;
    if (dd >= R) continue;
    uint32_t excl = 0;
    if (tile > 0) {
      // Four predecessors per step (four loads in flight): aggregates are summed up to the first
      // inclusive value; at a tile that has not published yet the walk waits and resumes there.
      int64_t t = (int64_t)tile - 1;
      while (t >= 0) {
        const int nb = (int)(t + 1 < 4 ? t + 1 : 4);
        uint32_t sv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < nb) sv[i] = ld_agent(&st.status[((size_t)pass * numTiles + (t - i)) * R + dd]);
        int used = 0;
        bool done = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (done || i >= nb || used < i) continue;
          const uint32_t flag = sv[i] & ~kValueMask;
          if (flag == 0u) continue;  // not published: stop consuming here
          excl += sv[i] & kValueMask;
          used = i + 1;
          done = flag == kFlagInc;
        }
        if (done) break;
        t -= used;
        if (used < nb) __builtin_amdgcn_s_sleep(1);
      }
      st_agent(&st.status[((size_t)pass * numTiles + tile) * R + dd], kFlagInc | (excl + cnt[q]));
    }
    s_gbase[dd] = st.hist[pass * R + dd] + excl;
  }
  __syncthreads();
  // s_gbase[d] - s_tdigit[d] maps a local sorted position to its global position.
#pragma unroll
  for (int q = 0; q < DPT; ++q) {
    const int dd = tid * DPT + q;
    if (dd < R) s_gbase[dd] -= s_tdigit[dd];
  }

  // Stable local reorder of the keys in LDS.
  KT *s_keys = (KT *)s_buf;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if constexpr (kTwoPerCU<KT, VB, THREADS>) asm volatile("" : "+v"(k[j]));  // the digit is taken from the key again, not kept from the ranking
    const uint32_t dj = digit_of(k[j], shift, dmask);
    const uint32_t pj = s_tdigit[dj] + s_whist[w][dj] + (j & 1 ? pos[j / 2] >> 16 : pos[j / 2] & 0xFFFFu);
    pos[j / 2] = j & 1 ? (pos[j / 2] & 0xFFFFu) | pj << 16 : (pos[j / 2] & 0xFFFF0000u) | pj;
    s_keys[pj] = k[j];
    if constexpr (kTwoPerCU<KT, VB, THREADS>) {
      asm volatile("" : "+v"(pos[j / 2]));
    }
  }
  __syncthreads();

  if constexpr (VB != 0 && !kEarlyVals) load_items<ITEMS>(wvsrc, valid == TILE, here, (VT)0, ve);
  // The sorted keys back from LDS (every position of the tile holds a key, the padding included)
  // and their global positions.
  uint32_t dig[VB ? ITEMS / 4 : 1];  // the write positions' digits, a byte each
#pragma unroll
  for (int j0 = 0; j0 < ITEMS; j0 += NB) {
    KT sk[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) sk[j] = s_keys[(j0 + j) * THREADS + tid];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const uint32_t dj = digit_of(sk[j], shift, dmask);
      if constexpr (VB != 0) {
        const int q = j0 + j;
        dig[q / 4] = q & 3 ? dig[q / 4] | dj << 8 * (q & 3) : dj;
      }
      const uint32_t at = s_gbase[dj] + (uint32_t)((j0 + j) * THREADS + tid);
      if ((uint32_t)((j0 + j) * THREADS + tid) < valid && at < n) put_at(dst, at, sk[j]);
    }
    if constexpr (kTwoPerCU<KT, VB, THREADS>) __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr (VB != 0) {
    __syncthreads();
    VT *s_vals = (VT *)s_buf;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) s_vals[j & 1 ? pos[j / 2] >> 16 : pos[j / 2] & 0xFFFFu] = ve[j];
    __syncthreads();
#pragma unroll
    for (int j0 = 0; j0 < ITEMS; j0 += NB) {
      VT sv[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) sv[j] = s_vals[(j0 + j) * THREADS + tid];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int q = j0 + j;
        const uint32_t at = s_gbase[(dig[q / 4] >> 8 * (q & 3)) & 255u] + (uint32_t)(q * THREADS + tid);
        if ((uint32_t)((j0 + j) * THREADS + tid) < valid && at < n) put_at(vdst, at, sv[j]);
      }
      if constexpr (kTwoPerCU<KT, VB, THREADS>) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Moves the result back into the caller's buffers when an odd number of passes ran.
template <typename KT, int VB>
__global__ void __launch_bounds__(256) k_final_copy(KT *__restrict__ keys0, const KT *__restrict__ keys1,
                                                     void *__restrict__ vals0, const void *__restrict__ vals1,
                                                     size_t n, const uint32_t *__restrict__ activeMask) {
  using VT = typename ValType<VB>::T;
  if (!(__builtin_popcount(*activeMask) & 1)) return;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    keys0[i] = keys1[i];
    if (VB) ((VT *)vals0)[i] = ((const VT *)vals1)[i];
  }
}

// ------------------------------------------------------------------------------------------------
// Small sorts: every key's rank by comparing it with every key.
// ------------------------------------------------------------------------------------------------
// One workgroup per 64 keys (key_rank): the rank is the key's place in `outKeys`.
template <typename KT, int VB>
__global__ void __launch_bounds__(1024)
    k_rank(const KT *__restrict__ keys, const void *__restrict__ vals, KT *__restrict__ outKeys,
           void *__restrict__ outVals, uint32_t n) {
  using VT = typename ValType<VB>::T;
  __shared__ uint32_t s_count[16][64];
  const uint32_t l = threadIdx.x & 63u, i0 = blockIdx.x * 64u, i = min(i0 + l, n - 1);
  const KT k = keys[i];
  VT v = 0;
  if (VB && threadIdx.x < 64) v = ((const VT *)vals)[i];
  const uint32_t rank = key_rank(keys, n, i0, k, s_count);
  if (threadIdx.x < 64 && i0 + l < n) {
    outKeys[rank] = k;
    if (VB) ((VT *)outVals)[rank] = v;
  }
}

template <typename KT, int VB>
__global__ void __launch_bounds__(256) k_copy_pairs(const KT *__restrict__ keys, const void *__restrict__ vals,
                                                    KT *__restrict__ outKeys, void *__restrict__ outVals, uint32_t n) {
  using VT = typename ValType<VB>::T;
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  outKeys[i] = keys[i];
  if (VB) ((VT *)outVals)[i] = ((const VT *)vals)[i];
}

// ------------------------------------------------------------------------------------------------
// Host dispatch
// ------------------------------------------------------------------------------------------------
// Up to here ranks beat the radix passes, whose 8 to 12 dependent launches take 6 to 10 us each however
// few keys there are (a copy of the keys and the sort, us, 64-bit pairs / 32-bit keys, ranks against
// passes): 3,000 keys 13 against 89 / 13 against 41, 16,000 keys 40 against 124 / 38 against 49; 24,000
// keys 95 against 129 / 93 against 49, as the compares grow with the square.
constexpr size_t kRankSortMax = 16384;

template <typename KT, int VB>
void run_rank(Context *ctx, hipStream_t s, void *keys, void *vals, void *keysAlt, void *valsAlt, size_t n) {
  launch(ctx, s, "sort_rank", k_rank<KT, VB>, dim3((unsigned)((n + 63) / 64)), dim3(1024), 0, (const KT *)keys,
         (const void *)vals, (KT *)keysAlt, valsAlt, (uint32_t)n);
  launch(ctx, s, "sort_rank_copy", k_copy_pairs<KT, VB>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
         (const KT *)keysAlt, (const void *)valsAlt, (KT *)keys, vals, (uint32_t)n);
}

inline int passes_for(int loBit, int hiBit, int bits) { return (hiBit - loBit + bits - 1) / bits; }

// Keys per tile of one sort. Automatically 2,048 (256 threads x 8) up to 2^18 keys, where a pass is as long
// as one tile takes; 4,096 (256 x 16) for 64-bit keys or payloads and 8,192 (512 x 16) for narrow ones; and
// 16,384 (1,024 x 16) from 1.6 million wide or 2.6 million narrow keys on, where longer digit runs and fewer
// look-back steps count more. Us, with the smaller against the larger tile: 60,000 64-bit pairs 105 against
// 147, 260,000 134 against 173, 400,000 151 against 145; 60,000 32-bit pairs 66 against 79, 400,000 89 against
// 87; 1 million 64-bit pairs 194 against 242, 2 million 277 against 264, 64-bit keys 176 against 189 and 218
// against 217; 2 million 32-bit pairs 124 against 129, 3 million 156 against 143. Asked for: 2,048, 4,096,
// and with narrow keys 8,192 and 16,384 are taken as they are, with wide ones as 4,096.
constexpr size_t kAutoSmallTileKeys = (size_t)1 << 18;
constexpr size_t large_tile_keys(int keyBits, int valBits) {
  return keyBits == 64 || valBits == 64 ? (size_t)3 << 19 : (size_t)5 << 19;
}

int tile_keys_effective(const SortConfig &cfg, size_t n, int keyBits, int valBits) {
  const bool wide = keyBits == 64 || valBits == 64;
  if (cfg.tileKeys == 0) {
    if (n <= kAutoSmallTileKeys) return 2048;
    return n >= large_tile_keys(keyBits, valBits) ? 16384 : wide ? 4096 : 8192;
  }
  return wide ? std::min(cfg.tileKeys, 4096) : cfg.tileKeys;
}

template <typename KT, int VB, int BITS, int THREADS, int ITEMS>
void run_typed(Context *ctx, hipStream_t s, void *keys, void *vals, void *keysAlt, void *valsAlt, size_t n, int loBit,
               int hiBit, void *scratch) {
  constexpr int R = 1 << BITS;
  constexpr int TILE = THREADS * ITEMS;
  const int passes = passes_for(loBit, hiBit, BITS);
  const uint32_t tiles = (uint32_t)((n + TILE - 1) / TILE);
  SortState st = state_view(scratch, passes, R);
  const size_t words = (size_t)passes * R + 32 + (size_t)passes * tiles * R;
  fill_u32(ctx, s, scratch, 0u, words);
  const size_t hb = hist_blocks(n, (size_t)ctx->cuCount);
  launch(ctx, s, "sort_hist", k_hist<KT, BITS>, dim3((unsigned)hb), dim3(kHistThreads), (size_t)passes * R * 4,
         (const KT *)keys, n, loBit, hiBit, passes, st.hist);
  launch(ctx, s, "sort_hist_scan", k_hist_scan<BITS>, dim3(1), dim3(256), 0, st.hist, st.activeMask, passes,
         (uint32_t)n);
  for (int p = 0; p < passes; ++p) {
    launch(ctx, s, "sort_onesweep", k_onesweep<KT, VB, BITS, THREADS, ITEMS>, dim3(tiles), dim3(THREADS), 0,
           (KT *)keys, (KT *)keysAlt, vals, valsAlt, (uint32_t)n, p, loBit + p * BITS, hiBit, scratch, passes,
           tiles);
  }
  size_t cb = (n + 255) / 256;
  if (cb > 8192) cb = 8192;
  launch(ctx, s, "sort_final_copy", k_final_copy<KT, VB>, dim3((unsigned)cb), dim3(256), 0, (KT *)keys,
         (const KT *)keysAlt, vals, (const void *)valsAlt, n, (const uint32_t *)st.activeMask);
}

template <typename KT, int VB, int BITS>
bool run_bits(Context *ctx, hipStream_t s, void *keys, void *vals, void *keysAlt, void *valsAlt, size_t n, int loBit,
              int hiBit, void *scratch, const SortConfig &cfg) {
  switch (tile_keys_effective(cfg, n, (int)sizeof(KT) * 8, VB)) {
    case 2048: run_typed<KT, VB, BITS, 256, 8>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch); return true;
    case 4096: run_typed<KT, VB, BITS, 256, 16>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch); return true;
    case 8192:
      if constexpr (sizeof(KT) == 4 && VB <= 32) {
        run_typed<KT, VB, BITS, 512, 16>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch);
        return true;
      }
      break;
    case 16384: run_typed<KT, VB, BITS, 1024, 16>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch); return true;
  }
  fail("sort: tileKeys %d is not one of 0, 2048, 4096, 8192, 16384", cfg.tileKeys);
  return false;
}

template <typename KT, int VB>
bool run_kv(Context *ctx, hipStream_t s, void *keys, void *vals, void *keysAlt, void *valsAlt, size_t n, int loBit,
            int hiBit, void *scratch, const SortConfig &cfg) {
  if (n <= kRankSortMax && loBit == 0 && hiBit == (int)sizeof(KT) * 8) {
    run_rank<KT, VB>(ctx, s, keys, vals, keysAlt, valsAlt, n);
    return true;
  }
  switch (cfg.digitBits) {
    case 4: return run_bits<KT, VB, 4>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
    case 6: return run_bits<KT, VB, 6>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
    case 8: return run_bits<KT, VB, 8>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
    default: fail("sort: digitBits %d is not one of 4, 6, 8", cfg.digitBits); return false;
  }
}

}  // namespace

size_t sort_scratch_bytes(size_t n, int keyBits, int valBits, int loBit, int hiBit, const SortConfig &cfg) {
  const int R = 1 << cfg.digitBits;
  const int passes = passes_for(loBit, hiBit, cfg.digitBits);
  // Not less than for fewer keys, whose tiles may be smaller: scratch for n keys does for all up to n.
  size_t tiles = 0;
  for (size_t m : {n, std::min(n, kAutoSmallTileKeys), std::min(n, large_tile_keys(keyBits, valBits) - 1)}) {
    const size_t tile = (size_t)tile_keys_effective(cfg, m, keyBits, valBits);
    tiles = std::max(tiles, (m + tile - 1) / tile);
  }
  return ((size_t)passes * R + 32 + (size_t)passes * tiles * R) * 4;
}

bool sort_run(Context *ctx, hipStream_t s, void *keys, void *vals, void *keysAlt, void *valsAlt, size_t n, int keyBits,
              int valBits, int loBit, int hiBit, void *scratch, const SortConfig &cfg) {
  if (n <= 1) return true;
  if (loBit < 0 || hiBit > keyBits || loBit >= hiBit) {
    fail("sort: bit range [%d, %d) invalid for %d-bit keys", loBit, hiBit, keyBits);
    return false;
  }
  if (keyBits == 32) {
    if (valBits == 0) return run_kv<uint32_t, 0>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
    if (valBits == 32) return run_kv<uint32_t, 32>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
    return run_kv<uint32_t, 64>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
  }
  if (valBits == 0) return run_kv<uint64_t, 0>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
  if (valBits == 32) return run_kv<uint64_t, 32>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
  return run_kv<uint64_t, 64>(ctx, s, keys, vals, keysAlt, valsAlt, n, loBit, hiBit, scratch, cfg);
}

}  // namespace gprt
