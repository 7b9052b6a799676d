// Single-pass exclusive scan / partition / select over 32-bit items for gfx950.
//
// Behaviour follows GPRT's scan family (gprt/gprt_scan.slang:84-392; host side
// gprt/gprt.cpp:8739-8818, commented-out path): an atomic ticket assigns tiles in launch order so
// a tile only ever waits on tiles that are already resident (gprt/gprt_scan.slang:112-115), and
// each tile publishes an aggregate, looks back over its predecessors, then publishes its inclusive
// prefix. Partition writes selected items at their exclusive rank and unselected items at
// (n-1) - (i - rank) (gprt/gprt_scan.slang:89-92); select writes only the selected items.
//
// MI355X design:
//  * A tile is 16 wave64s; each wave owns 64 lanes x K uint4 = 256K consecutive items, loaded with
//    16-byte coalesced nontemporal loads and scanned with DPP wave prefix sums. What bounds a large
//    scan is HBM: 10^8 items in 165 us (4.85 TB/s, a plain copy's rate), 175 us with the host's wait.
//  * Large sums use large tiles (44 items per lane, one workgroup per CU): a tile waits in its
//    look-back for predecessors that are still loading, and that wait grows with the number of tiles
//    in flight. Small inputs use small tiles, so that every CU has one (scan_k).
//  * Partition / select put the tile's items in their order of writing in LDS, so that the selected
//    and the unselected run are each written as whole lines: 10^7 items in 27 us where four scattered
//    4-byte writes per lane took 53 us (10^8: 396 -> 207 us with the host's wait).
//  * The look-back is done by a whole wave: lane l inspects predecessor tile (p-1-l), so 64
//    predecessors are examined per round trip instead of one.
//  * One launch per call: the status words carry the call's epoch, so the context's state is never
//    cleared, and the kernel hands the total to the host itself. 1,000 items took 33 us as fill, scan,
//    4-byte copy and a polled stream; 11 us now.
//  * Values wrap modulo 2^32 with no 2^30 limit (the reference packs value<<2|flag into 32 bits,
//    gprt/gprt_scan.slang:223-228).
//  * State layout (uint64 words): [0] total (low 32 bits), [1] tile ticket, [2 + t] tile t status.
#include <algorithm>
#include <mutex>
#include <vector>

#include "device_common.hpp"
#include "internal.hpp"

namespace gprt {

namespace {

// A status word: the value in the low 32 bits, {epoch:30 | flag:2} above it (flag 1: the tile's own
// aggregate, 2: its inclusive prefix). A word counts only under the call's epoch, so a state that
// outlives the call needs no clearing between calls; a cleared state serves epoch 0.
constexpr uint32_t kAgg = 1u, kInc = 2u;
__device__ __forceinline__ uint64_t status_word(uint32_t epoch, uint32_t flag, uint32_t value) {
  return ((uint64_t)(epoch << 2 | flag) << 32) | value;
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// MODE 0: exclusive sum; 1: partition; 2: select. `hostWord` (may be null) gets {seq | total} in
// host memory; a single tile writes it after everything else, ordered behind its own output, so the
// host may take it as the call's completion.
template <int WAVES, int K, int MODE>
__global__ void __launch_bounds__(WAVES * 64)
    k_scan(const uint32_t *__restrict__ in, uint32_t *__restrict__ out, uint32_t n, int selectPositive,
           uint64_t *__restrict__ state, uint32_t numTiles, uint32_t epoch, uint64_t *__restrict__ hostWord,
           uint32_t seq) {
  constexpr uint32_t THREADS = WAVES * 64;
  constexpr uint32_t WAVE_ITEMS = 64 * K * 4;
  constexpr uint32_t TILE = WAVES * WAVE_ITEMS;
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_wsum[WAVES];
  __shared__ uint32_t s_prefix;
  __shared__ uint32_t s_items[MODE == 0 ? 1 : TILE];

  const uint32_t tid = threadIdx.x;
  const uint32_t w = tid >> 6;
  const uint32_t l = tid & 63;

  uint32_t tile = 0;
  if (numTiles > 1) {  // uniform over the grid
    if (tid == 0) {
      s_tile = ticket((uint32_t *)&state[1]);
      if (s_tile == numTiles - 1) st_agent((uint32_t *)&state[1], 0u);  // no ticket follows: the next call's start
    }
    __syncthreads();
    tile = s_tile;
  }
  const size_t waveBase = (size_t)tile * TILE + (size_t)w * WAVE_ITEMS;

  // Only the items stay in registers; what an item counts (itself for the sum, its selection flag
  // for partition / select) is recomputed from it, and its prefix from its 4-item group's exclusive
  // offset, when the results are written.
  uint32_t v[K][4];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const size_t idx = waveBase + ((size_t)k * 64 + l) * 4;
    if (idx + 3 < n) {
      const u32x4_t q = __builtin_nontemporal_load((const u32x4_t *)(in + idx));
      v[k][0] = q.x;
      v[k][1] = q.y;
      v[k][2] = q.z;
      v[k][3] = q.w;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) v[k][c] = (idx + c < n) ? in[idx + c] : 0u;
    }
  }
  auto counted = [&](int k, int c) -> uint32_t {
    if (MODE == 0) return v[k][c];
    const size_t idx = waveBase + ((size_t)k * 64 + l) * 4 + c;
    const bool sel = selectPositive ? ((int32_t)v[k][c] >= 0) : ((int32_t)v[k][c] < 0);
    return (idx < n && sel) ? 1u : 0u;
  };

  // Exclusive prefix of each lane's 4-item group within the wave's chunk (order: k, lane, item).
  uint32_t gex[K];
  uint32_t carry = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t s = counted(k, 0) + counted(k, 1) + counted(k, 2) + counted(k, 3);
    const uint32_t incl = wave_incl_sum(s);
    gex[k] = incl - s + carry;
    carry += wave_read(incl, 63);
  }
  if (l == 0) s_wsum[w] = carry;
  __syncthreads();

  uint32_t woff = 0, agg = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const uint32_t x = s_wsum[i];
    if ((uint32_t)i < w) woff += x;
    agg += x;
  }
  if (numTiles > 1 && tid == 0) st_agent(&state[2 + tile], status_word(epoch, tile == 0 ? kInc : kAgg, agg));

  // Partition / select: the tile's items in their order of writing, selected ones first, so that
  // both runs leave the tile as coalesced writes. Independent of the look-back, which the other
  // waves' LDS writes therefore overlap.
  if (MODE != 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const uint32_t local = w * WAVE_ITEMS + ((uint32_t)k * 64 + l) * 4;
      uint32_t r = woff + gex[k];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (counted(k, c)) {
          s_items[r] = v[k][c];
          ++r;
        } else if (MODE == 1) {
          s_items[agg + (local + c - r)] = v[k][c];  // past the tile's valid items: after them all
        }
      }
    }
  }

  if (w == 0) {
    uint32_t excl = 0;
    if (tile > 0) {
      int64_t base = (int64_t)tile - 1;
      uint32_t acc = 0;
      while (true) {
        const int64_t t = base - (int64_t)l;
        const uint64_t word = (t >= 0) ? ld_agent(&state[2 + t]) : status_word(epoch, kInc, 0u);
        const uint32_t tag = (uint32_t)(word >> 32);
        const uint32_t flag = (tag >> 2) == epoch ? tag & 3u : 0u;
        const uint64_t incMask = wave_ballot(flag == kInc);
        const uint64_t readyMask = wave_ballot(flag != 0u);
        if (incMask) {
          const int first = __builtin_ctzll(incMask);
          const uint64_t need = (first == 63) ? ~0ull : ((1ull << (first + 1)) - 1ull);
          if ((readyMask & need) == need) {
            acc += wave_sum((int)l <= first ? (uint32_t)word : 0u);
            break;
          }
        } else if (readyMask == ~0ull) {
          acc += wave_sum((uint32_t)word);
          base -= 64;
          continue;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      excl = acc;
      if (l == 0) st_agent(&state[2 + tile], status_word(epoch, kInc, excl + agg));
    }
    if (l == 0) {
      s_prefix = excl;
      if (tile == numTiles - 1) {
        st_agent(&state[0], (uint64_t)(uint32_t)(excl + agg));
        if (hostWord && numTiles > 1)
          __hip_atomic_store(hostWord, ((uint64_t)seq << 32) | (uint32_t)(excl + agg), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  __syncthreads();

  if (MODE == 0) {
    const uint32_t prefix = s_prefix + woff;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const size_t idx = waveBase + ((size_t)k * 64 + l) * 4;
      uint32_t r[4];
      r[0] = prefix + gex[k];
#pragma unroll
      for (int c = 1; c < 4; ++c) r[c] = r[c - 1] + v[k][c - 1];
      if (idx + 3 < n) {
        __builtin_nontemporal_store(u32x4_t{r[0], r[1], r[2], r[3]}, (u32x4_t *)(out + idx));
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (idx + c < n) out[idx + c] = r[c];
      }
    }
  } else {
    const uint32_t prefix = s_prefix, tileBase = tile * TILE;
    const uint32_t valid = min(TILE, n - tileBase);
    // Unselected item u of the tile goes to (n - 1) - (unselected before it).
    const uint32_t tail = (n - 1) - (tileBase - prefix);
#pragma unroll
    for (int j = 0; j < 4 * K; ++j) {
      const uint32_t p = (uint32_t)j * THREADS + tid;
      if (p < agg)
        out[prefix + p] = s_items[p];
      else if (MODE == 1 && p < valid)
        out[tail - (p - agg)] = s_items[p];
    }
  }
  if (hostWord && numTiles == 1) {
    __threadfence_system();
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(hostWord, ((uint64_t)seq << 32) | agg, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Items per lane (4 K) and so per tile (16 waves x 64 lanes x 4 K), by the number of items. Host times
// of the call, us, for K = 1 / 4 / 11 (sum) and K = 1 / 4 (partition):
//   up to one K = 1 tile     1,000: 11.4 / 11.9 / 13.8      11.8 / 14.2
//   up to one K = 4 tile    10,000: 14.1 / 12.4 / 13.1      14.4 / 14.0   (one tile: no look-back)
//   up to 2^19             300,000: 15.3 / 15.6 / 17.2      15.5 / 17.4   (K = 4 leaves most CUs idle)
//   up to 6 x 2^20       4,000,000: 32.6 / 21.4 / 22.8      33.5 / 23.0   (512 tiles are resident)
//   above               16,000,000: 72.3 / 46.5 / 41.0      75.7 / 49.1   (fewer look-backs in flight)
// Partition / select stay at K = 4, whose 64 KB of reordered items let two tiles share a CU.
constexpr int kScanWaves = 16;
constexpr uint32_t scan_tile(int k) { return (uint32_t)kScanWaves * 64u * 4u * (uint32_t)k; }
constexpr int kScanKSmall = 1, kScanKMid = 4, kScanKLarge = 11;
int scan_k(size_t n, int mode) {
  if (n <= scan_tile(kScanKSmall)) return kScanKSmall;
  if (n > scan_tile(kScanKMid) && n <= (size_t)1 << 19) return kScanKSmall;
  return (mode != 0 || n <= (size_t)6 << 20) ? kScanKMid : kScanKLarge;
}

// The look-back state of gprtBufferExclusiveSumNoAlloc: one device-resident array per GPU that
// the library runs on, held until the process ends, so that the call allocates nothing. It holds
// the state of one exclusive sum of up to kNoAllocMaxItems items: [0] total, [1] tile ticket,
// [2 + t] the status of tile t. Host code never passes `scratch` itself to a kernel (in host code
// the name stands for a host-side shadow); it uses the device address hipGetSymbolAddress returns
// for the current device, kept per device in g_noAllocState.
constexpr size_t kNoAllocMaxItems = 1ull << 31;
constexpr size_t kNoAllocWords = (1ull << 17) + 2;  // 1 MiB + 16 B
static_assert(kNoAllocWords >= (kNoAllocMaxItems + scan_tile(kScanKLarge) - 1) / scan_tile(kScanKLarge) + 2,
              "the static state holds every tile status of the largest allowed input");

std::mutex g_noAllocMutex;
std::vector<void *> g_noAllocState;  // device address of `scratch` per device ordinal

}  // namespace

static __device__ __align__(256) uint64_t scratch[kNoAllocWords];

bool scan_noalloc_init(int device) {
  std::lock_guard<std::mutex> lock(g_noAllocMutex);
  if (device < 0) return false;
  if ((size_t)device < g_noAllocState.size() && g_noAllocState[device]) return true;
  void *p = nullptr;
  if (!hip_ok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scan state)") || !p) return false;
  if (g_noAllocState.size() <= (size_t)device) g_noAllocState.resize((size_t)device + 1, nullptr);
  g_noAllocState[device] = p;
  return true;
}

void *scan_noalloc_state(int device) {
  std::lock_guard<std::mutex> lock(g_noAllocMutex);
  return (device >= 0 && (size_t)device < g_noAllocState.size()) ? g_noAllocState[device] : nullptr;
}

size_t scan_noalloc_max_items() { return kNoAllocMaxItems; }

size_t scan_scratch_bytes(size_t n) {
  const size_t tile = scan_tile(std::min(scan_k(n, 0), scan_k(n, 1)));
  return ((n + tile - 1) / tile + 2) * sizeof(uint64_t);
}

namespace {

template <int MODE>
void scan_launch(Context *ctx, hipStream_t s, const uint32_t *in, uint32_t *out, size_t n, bool selectPositive,
                 void *state, uint32_t tiles, uint32_t epoch, uint64_t *hostWord, uint32_t seq) {
  auto go = [&](auto kernel) {
    launch(ctx, s, "scan_lookback", kernel, dim3(tiles), dim3(kScanWaves * 64), 0, in, out, (uint32_t)n,
           selectPositive ? 1 : 0, (uint64_t *)state, tiles, epoch, hostWord, seq);
  };
  switch (scan_k(n, MODE)) {
    case kScanKSmall: go(k_scan<kScanWaves, kScanKSmall, MODE>); break;
    case kScanKMid: go(k_scan<kScanWaves, kScanKMid, MODE>); break;
    default:
      if constexpr (MODE == 0) go(k_scan<kScanWaves, kScanKLarge, MODE>);
  }
}

void scan_mode(Context *ctx, hipStream_t s, const uint32_t *in, uint32_t *out, size_t n, int mode, bool selectPositive,
               void *state, uint32_t tiles, uint32_t epoch, uint64_t *hostWord, uint32_t seq) {
  if (mode == 0)
    scan_launch<0>(ctx, s, in, out, n, selectPositive, state, tiles, epoch, hostWord, seq);
  else if (mode == 1)
    scan_launch<1>(ctx, s, in, out, n, selectPositive, state, tiles, epoch, hostWord, seq);
  else
    scan_launch<2>(ctx, s, in, out, n, selectPositive, state, tiles, epoch, hostWord, seq);
}

uint32_t scan_tiles(size_t n, int mode) {
  const size_t tile = scan_tile(scan_k(n, mode));
  return (uint32_t)((n + tile - 1) / tile);
}

}  // namespace

bool scan_signals(size_t n, int mode) { return scan_tiles(n, mode) == 1; }

void scan_run(Context *ctx, hipStream_t s, const uint32_t *in, uint32_t *out, size_t n, int mode, bool selectPositive,
              void *state, uint64_t *hostWord, uint32_t seq) {
  const uint32_t tiles = scan_tiles(n, mode);
  if (tiles > 1) fill_u32(ctx, s, state, 0u, ((size_t)tiles + 2) * 2);
  scan_mode(ctx, s, in, out, n, mode, selectPositive, state, tiles, 0u, hostWord, seq);
}

// The context's own look-back state is cleared once, when it is allocated (or its epochs run out):
// every call takes the next epoch, and the kernel leaves its ticket counter at 0.
bool scan_run_kept(Context *ctx, hipStream_t s, const uint32_t *in, uint32_t *out, size_t n, int mode,
                   bool selectPositive, uint64_t *hostWord, uint32_t seq) {
  const uint32_t tiles = scan_tiles(n, mode);
  ScanState &st = ctx->scan;
  if (tiles > st.tiles) {
    if (st.words) {
      hipStreamSynchronize(s);
      hipFree(st.words);
      st = ScanState{};
    }
    if (!hip_ok(hipMalloc((void **)&st.words, ((size_t)tiles + 2) * 8), "hipMalloc(scan state)")) return false;
    st.tiles = tiles;
    st.epoch = kScanEpochs;  // to be cleared
  }
  if (st.epoch >= kScanEpochs) {
    fill_u32(ctx, s, st.words, 0u, ((size_t)st.tiles + 2) * 2);
    st.epoch = 0;
  }
  ++st.epoch;
  scan_mode(ctx, s, in, out, n, mode, selectPositive, st.words, tiles, st.epoch, hostWord, seq);
  return true;
}

}  // namespace gprt
