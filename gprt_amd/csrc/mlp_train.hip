// Training of the proposal MLP on MFMA: one minibatch step in three launches.
//
//   k_train_rows    forward and the backward of the activations, 16 rays per workgroup: encode, the
//                   three hidden layers, all 4096 logits of the rays in the workgroup's accumulators
//                   (8 waves x 32 blocks of 16 x 16), softmax and its gradient dZ there, dA3 = dZ W4
//                   from LDS, dA2 and dA1. Neither logits nor activations are read back from memory;
//                   what the weight gradients need (X, H1..H3, dA1..dA3, dZ, all bf16) is written
//                   once, in fragments that k_train_weights loads as they are.
//   k_train_weights dW = dA^T H of the four layers, split over the rays, and the bias gradients'
//                   partial sums from the same fragments.
//   k_train_update  adds the splits in order and applies Adam (or stores the gradients), and writes
//                   the bf16 weights in the three layouts their readers want.
//
// A batch of 8,192 rays takes 74 + 28 + 8 us (HIP events); it took 580 us as 28 launches (GEMMs over a
// 128 MB logit matrix that the softmax read back, column sums, bias copies).
//
// Every sum keeps a fixed order: K ascends in steps of 32 within a split, splits and column chunks are
// added in order, and the softmax denominator is the sum of 256 partial sums of 16 classes (classes
// 1024 j + 4 t + q for t = 0..255, j outer), reduced by halves within each 64 of them. Results
// therefore do not depend on scheduling.
//
// Fragment layouts (bf16, 512 elements = 64 lanes x 8 per fragment, lane = (g, n), g = lane >> 4):
//   forward weights, layer l   [block of 16 outputs][K step of 32][lane][8]: W[out n][32 ks + 8 g + e]
//     the output layer's block b of wave w holds classes class_of(w, b, n), see below
//   backward weights           [block of 16 inputs][step of 32 outputs][lane][8]: W[32 s + 8 g + e][in n]
//   activations and gradients  [block of 16 columns][16 rays]: element (column c, ray r) at
//     (((r >> 3) * 16 + c) * 8 + (r & 7)), so that two neighbouring blocks are a 32-ray fragment
#include <algorithm>
#include <cmath>

#include "bvh.hpp"
#include "device_common.hpp"
#include "internal.hpp"
#include "mlp_device.hpp"

namespace gprt {

namespace {

constexpr int kRowWaves = 8;                       // waves of k_train_rows
constexpr int kRowRays = 16;                       // its rays
constexpr int kRowBlocks = kMlpOut / 16 / kRowWaves;  // 32 blocks of 16 classes per wave
constexpr int kDzPitch = kMlpOut * 2 + 16;         // bytes of a dZ row in LDS: 16 rows fall into distinct banks
constexpr int kActPitch = kMlpHid * 2 + 16;        // bytes of an activation row in LDS
constexpr size_t kRowLds = (size_t)kRowRays * kDzPitch + 2 * kRowRays * kActPitch;

// Wave w's block b = 16 gi + 4 j + q holds, in column n, class 1024 j + 4 t + q of the partial sum
// t = 64 (w >> 1) + 16 (w & 1) + 32 gi + n: a lane adds a partial sum's classes in their order, and the
// two groups gi are the first halves to be added.
__host__ __device__ constexpr uint32_t class_of(uint32_t w, uint32_t b, uint32_t n) {
  return 1024u * ((b >> 2) & 3u) + 4u * (64u * (w >> 1) + 16u * (w & 1u) + 32u * (b >> 4) + n) + (b & 3u);
}
struct ClassPlace {
  uint32_t w, b, n;
};
__host__ __device__ constexpr ClassPlace place_of(uint32_t c) {
  const uint32_t t = (c & 1023u) >> 2;
  return {2u * (t >> 6) + ((t >> 4) & 1u), 16u * ((t >> 5) & 1u) + 4u * (c >> 10) + (c & 3u), t & 15u};
}

// Offsets (elements) of the fragments of weight (o, i) of a layer.
__host__ __device__ inline size_t fwd_fragment(int layer, uint32_t o, uint32_t i) {
  uint32_t block = o >> 4, n = o & 15u;
  if (layer == 3) {
    const ClassPlace p = place_of(o);
    block = p.w * kRowBlocks + p.b;
    n = p.n;
  }
  return mlp_bf16_offset(layer) + ((size_t)(block * 4 + (i >> 5)) * 64 + ((i >> 3) & 3u) * 16 + n) * 8 + (i & 7u);
}
__host__ __device__ inline size_t bwd_fragment(int layer, uint32_t o, uint32_t i) {
  const uint32_t steps = layer == 3 ? kMlpOut / 32 : kMlpHid / 32;
  return mlp_bf16_offset(layer) + ((size_t)((i >> 4) * steps + (o >> 5)) * 64 + ((o >> 3) & 3u) * 16 + (i & 15u)) * 8 +
         (o & 7u);
}

struct TrainArgs {
  const GPRTRay *rays;
  const int32_t *labels;
  uint32_t n, blocks;  // rays, and blocks of 16 rays written (an even number)
  float scale;
  const uint16_t *wf, *wb;  // forward and backward fragments
  const float *bias;        // b1 b2 b3 b4
  uint16_t *act;            // X H1 H2 H3 dA1 dA2 dA3: 8 column blocks each
  uint16_t *dz;             // 256 column blocks (in class_of's order)
  int dzSteps;              // K steps of 32 classes per split of dA3 = dZ W4
  float *loss;        // per ray
  uint32_t *correct;  // top-1 count
};

// Column block cb, ray block rb of an array of column blocks.
__host__ __device__ __forceinline__ size_t block_at(uint32_t blocks, uint32_t cb, uint32_t rb) {
  return ((size_t)cb * blocks + rb) * 256;
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)lo) | (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)hi) << 16;
}

// Rotation by `o` within each row of 16 lanes: after the steps 8, 4 and 2 have made the values periodic,
// it pairs the same lanes as an exchange over lane bit o.
template <int kCtrl>
__device__ __forceinline__ float row_rotate(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float v) {
  v += row_rotate<0x128>(v);  // row_ror:8
  v += row_rotate<0x124>(v);
  v += row_rotate<0x122>(v);
  v += row_rotate<0x121>(v);
  return v;
}

// What bounds it (8,192 rays, 74 us): its phases follow one another. 512 accumulator registers per SIMD hold 16
// rays' logits, so a CU runs one workgroup of two waves per SIMD, and nothing overlaps its encoding, hidden
// layers and barriers, the logits' products (17 us less without them), the exponentials (11), dZ's writes (4)
// and dA3's products (15). The 2.2 MB of weights that each of the 512 workgroups reads are 15 TB/s from L2.
__global__ void __launch_bounds__(kRowWaves * 64) k_train_rows(TrainArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned char *const sDz = smem;
  unsigned char *const sAct0 = smem + kRowRays * kDzPitch, *const sAct1 = sAct0 + kRowRays * kActPitch;
  // Before dZ is written its space holds the reductions' partial results.
  float *const sMax = (float *)smem;                                  // [wave][row]
  uint32_t *const sArg = (uint32_t *)(smem + 512);                    // [row]
  float *const sSum = (float *)(smem + 1024);                         // [wave][row][16]
  __shared__ uint32_t s_correct;
  const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
  const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)tid >> 6);
  if (tid == 0) s_correct = 0;
  const uint32_t rb = blockIdx.x, ray0 = rb * kRowRays;

  // The hidden layers' weight fragments of this wave's columns, under way during the encoding.
  Frag hid[3][4];
#pragma unroll
  for (int layer = 0; layer < 3; ++layer)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      hid[layer][ks].u = *(const uint4 *)(a.wf + mlp_bf16_offset(layer) + ((size_t)w * 4 + ks) * 512 + l * 8);
  // Encoding, a pair of words per thread: ray tid / 32; words 0..2 the raw values, word 3 + p the sine and
  // cosine of band p & 7 of value p >> 3, the rest 0.
  {
    const uint32_t r = (uint32_t)tid >> 5, s = (uint32_t)tid & 31u;
    uint32_t *row = (uint32_t *)(sAct0 + r * kActPitch);
    const bool live = ray0 + r < a.n;
    GPRTRay ray{};
    if (live) ray = load_ray_stream(a.rays + ray0 + r);
    const float v[6] = {ray.ox, ray.oy, ray.oz, ray.dx, ray.dy, ray.dz};
    auto band = [&](uint32_t p) -> uint32_t {
      const uint32_t c = p >> 3;
      const float x = c == 0 ? v[0] : c == 1 ? v[1] : c == 2 ? v[2] : c == 3 ? v[3] : c == 4 ? v[4] : v[5];
      float sn, cs;
      sincospif(x * (float)(1u << (p & 7u)), &sn, &cs);  // 2^k * v is exact
      return pack2(sn, cs);
    };
    row[3 + s] = live ? band(s) : 0u;
    if (s < 16u)
      row[3 + 32 + s] = live ? band(32 + s) : 0u;
    else if (s < 19u)
      row[s - 16u] = live ? pack2(s == 16u ? v[0] : s == 17u ? v[2] : v[4], s == 16u ? v[1] : s == 17u ? v[3] : v[5]) : 0u;
    else
      row[51 + s - 19u] = 0u;
  }
  __syncthreads();
  // The features as fragments of column block w.
  const size_t stored = (size_t)(((g >> 1) * 16 + n) * 8 + (g & 1) * 4);
  {
    uint16_t h[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) h[q] = *(const uint16_t *)(sAct0 + (4 * g + q) * kActPitch + (16 * w + n) * 2);
    *(uint2 *)(a.act + block_at(a.blocks, w, rb) + stored) =
        make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
  }

  // A 16 x 16 block of act @ W^T: A fragments of the 16 rays, one block of weight fragments.
  auto load_rows = [&](const unsigned char *act, Frag (&f)[4]) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) f[ks].u = *(const uint4 *)(act + n * kActPitch + ks * 64 + g * 16);
  };
  // The output layer's first weight blocks, under way during the hidden layers.
  constexpr int kAhead = 4;
  const uint16_t *w4 = a.wf + mlp_bf16_offset(3) + (size_t)w * kRowBlocks * 4 * 512 + l * 8;
  Frag out4[kAhead][4];
#pragma unroll
  for (int b = 0; b < kAhead; ++b)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) out4[b][ks].u = *(const uint4 *)(w4 + (b * 4 + ks) * 512);
  // Hidden layers: wave w computes outputs 16 w .. 16 w + 15; lane (g, n) holds rows 4 g + q of column n.
  uint32_t live[3];  // bit q: the activation of row 4 g + q is positive
  unsigned char *cur = sAct0, *nxt = sAct1;
#pragma unroll
  for (int layer = 0; layer < 3; ++layer) {
    Frag x[4];
    load_rows(cur, x);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc = mfma16(x[ks], hid[layer][ks], acc);
    const float bc = a.bias[layer * kMlpHid + 16 * w + n];
    float h[4];
    live[layer] = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      h[q] = fmaxf(acc[q] + bc, 0.f);
      if (ray0 + 4 * g + q >= a.n) h[q] = 0.f;  // rays past the end add nothing to any gradient
      live[layer] |= (bf2f(f2bf(h[q])) > 0.f ? 1u : 0u) << q;
    }
    const uint2 packed = make_uint2(pack_bf16(h[0], h[1]), pack_bf16(h[2], h[3]));
    *(uint16_t *)(nxt + (4 * g + 0) * kActPitch + (16 * w + n) * 2) = (uint16_t)packed.x;
    *(uint16_t *)(nxt + (4 * g + 1) * kActPitch + (16 * w + n) * 2) = (uint16_t)(packed.x >> 16);
    *(uint16_t *)(nxt + (4 * g + 2) * kActPitch + (16 * w + n) * 2) = (uint16_t)packed.y;
    *(uint16_t *)(nxt + (4 * g + 3) * kActPitch + (16 * w + n) * 2) = (uint16_t)(packed.y >> 16);
    *(uint2 *)(a.act + block_at(a.blocks, 8 * (layer + 1) + w, rb) + stored) = packed;
    __syncthreads();
    unsigned char *t = cur;
    cur = nxt;
    nxt = t;
  }

  // All logits of the 16 rays: block b of this wave in acc[b]; kAhead blocks of weights are in flight.
  f32x4_t acc[kRowBlocks];
  {
    Frag x[4];
    load_rows(cur, x);
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b) {
      acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        acc[b] = mfma16(x[ks], out4[b % kAhead][ks], acc[b]);
        if (b + kAhead < kRowBlocks) out4[b % kAhead][ks].u = *(const uint4 *)(w4 + ((b + kAhead) * 4 + ks) * 512);
      }
    }
    const float *b4 = a.bias + 3 * kMlpHid;
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b) {
      const float bc = b4[class_of(w, b, n)];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[b][q] += bc;
    }
  }

  // Row maxima.
  float mx[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) mx[q] = -INFINITY;
#pragma unroll
  for (int b = 0; b < kRowBlocks; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) mx[q] = fmaxf(mx[q], acc[b][q]);
  float own[4];  // the lane's own
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    own[q] = mx[q];
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) mx[q] = fmaxf(mx[q], __shfl_xor(mx[q], o, 64));
    if (n == 0) sMax[w * kRowRays + 4 * g + q] = mx[q];
  }
  if (tid < kRowRays) sArg[tid] = kMlpOut;
  // The label of each row, and which block of this wave holds it in this lane's column.
  int32_t y[4];
  int yb[4];
  uint32_t labelBlocks = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t ri = ray0 + 4 * g + q;
    y[q] = ri < a.n ? a.labels[ri] : -1;
    const ClassPlace p = place_of((uint32_t)y[q] & (kMlpOut - 1u));
    yb[q] = (y[q] >= 0 && y[q] < kMlpOut && p.w == w && p.n == (uint32_t)n) ? (int)p.b : -1;
    if (yb[q] >= 0) labelBlocks |= 1u << yb[q];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) labelBlocks |= __shfl_xor(labelBlocks, o, 64);
  labelBlocks = __builtin_amdgcn_readfirstlane(labelBlocks);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    mx[q] = sMax[4 * g + q];
#pragma unroll
    for (int i = 1; i < kRowWaves; ++i) mx[q] = fmaxf(mx[q], sMax[i * kRowRays + 4 * g + q]);
    // The lowest class at the maximum, which few lanes hold.
    if (__ballot(own[q] == mx[q])) {
      uint32_t c = kMlpOut;
#pragma unroll
      for (int b = kRowBlocks - 1; b >= 0; --b) c = acc[b][q] == mx[q] ? min(c, class_of(w, b, n)) : c;
      if (c < kMlpOut) atomicMin(&sArg[4 * g + q], c);
    }
  }

  // Exponentials in place; the lane's two partial sums per row are added, then the rest of each 64.
  float zy[4] = {0.f, 0.f, 0.f, 0.f};
  {
    float part[2][4];
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
#pragma unroll
      for (int q = 0; q < 4; ++q) part[gi][q] = 0.f;
#pragma unroll
      for (int b = 16 * gi; b < 16 * gi + 16; ++b) {
        if (labelBlocks >> b & 1u) {
#pragma unroll
          for (int q = 0; q < 4; ++q) zy[q] = yb[q] == b ? acc[b][q] : zy[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[b][q] = expf(acc[b][q] - mx[q]);
          part[gi][q] += acc[b][q];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) sSum[(w * kRowRays + 4 * g + q) * 16 + n] = part[0][q] + part[1][q];
  }
  __syncthreads();
  float sum[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float s[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const float *p = sSum + ((2 * o) * kRowRays + 4 * g + q) * 16 + n;
      s[o] = row_sum(p[0] + p[kRowRays * 16]);
    }
    sum[q] = s[0] + s[1] + s[2] + s[3];
  }
  uint32_t arg[4];  // every maximum NaN: class 0
#pragma unroll
  for (int q = 0; q < 4; ++q) arg[q] = sArg[4 * g + q] & (kMlpOut - 1u);
  __syncthreads();  // the sums are read; dZ takes their space

  // dZ = (softmax - onehot) * scale, 0 for rows without a label: to LDS by row (for dA3), and as
  // fragments to memory (for dW4).
  {
    float inv[4], scale[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      inv[q] = y[q] >= 0 ? 1.0f / sum[q] : 0.f;
      scale[q] = y[q] >= 0 ? a.scale : 0.f;
    }
#pragma unroll
    for (int gj = 0; gj < 8; ++gj) {
      uint2 z[4];  // block 4 gj + r: rows {0, 1}, {2, 3}
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int b = 4 * gj + r;
        float d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = acc[b][q] * inv[q];
        if (labelBlocks >> b & 1u) {
#pragma unroll
          for (int q = 0; q < 4; ++q) d[q] = yb[q] == b ? d[q] - 1.f : d[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] *= scale[q];
        z[r] = make_uint2(pack_bf16(d[0], d[1]), pack_bf16(d[2], d[3]));
        *(uint2 *)(a.dz + block_at(a.blocks, w * kRowBlocks + b, rb) + stored) = z[r];
      }
      // By row: the four blocks' classes follow one another. 0x05040100 joins low halves, 0x07060302 high ones.
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t sel = q & 1 ? 0x07060302u : 0x05040100u;
        const uint32_t lo = __builtin_amdgcn_perm(q < 2 ? z[1].x : z[1].y, q < 2 ? z[0].x : z[0].y, sel);
        const uint32_t hi = __builtin_amdgcn_perm(q < 2 ? z[3].x : z[3].y, q < 2 ? z[2].x : z[2].y, sel);
        *(uint2 *)(sDz + (4 * g + q) * kDzPitch + class_of(w, 4 * gj, n) * 2) = make_uint2(lo, hi);
      }
    }
  }
  // Loss and top-1 count: each row's label is in one lane of one wave. (Adding the losses to one word from
  // here made 8,192 atomics queue on it: 53 us.)
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (yb[q] >= 0) {
      a.loss[ray0 + 4 * g + q] = (logf(sum[q]) + mx[q] - zy[q]) * a.scale;
      if (arg[q] == (uint32_t)y[q]) atomicAdd(&s_correct, 1u);
    } else if (w == 0 && n == 0 && (y[q] < 0 || y[q] >= kMlpOut)) {
      a.loss[ray0 + 4 * g + q] = 0.f;
    }
  __syncthreads();
  if (tid == 0 && s_correct) atomicAdd(a.correct, s_correct);

  Frag back[2][4];  // layers 2 and 1, for dA2 and dA1
#pragma unroll
  for (int layer = 1; layer < 3; ++layer)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      back[layer - 1][ks].u = *(const uint4 *)(a.wb + mlp_bf16_offset(layer) + ((size_t)w * 4 + ks) * 512 + l * 8);
  // dA3 = (dZ W4) * (H3 > 0): wave w's 16 columns, K = 4096 in ascending steps of 32, in splits of
  // dzSteps that are summed in order.
  f32x4_t total = {0.f, 0.f, 0.f, 0.f};
  {
    const uint16_t *wb = a.wb + mlp_bf16_offset(3) + (size_t)w * (kMlpOut / 32) * 512 + l * 8;
    const unsigned char *dz = sDz + n * kDzPitch + g * 16;
    constexpr int kBatch = 16;
    Frag f[2][kBatch];
    f32x4_t part = {0.f, 0.f, 0.f, 0.f};
    int left = a.dzSteps;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) f[0][u].u = *(const uint4 *)(wb + u * 512);
#pragma unroll
    for (int s0 = 0; s0 < kMlpOut / 32; s0 += kBatch) {
      const int cb = (s0 / kBatch) & 1;
      if (s0 + kBatch < kMlpOut / 32) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u) f[cb ^ 1][u].u = *(const uint4 *)(wb + (s0 + kBatch + u) * 512);
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        Frag z;
        z.u = *(const uint4 *)(dz + (s0 + u) * 64);
        part = mfma16(z, f[cb][u], part);
        if ((u & 1) == 1) {  // splits are whole multiples of 64 classes
          left -= 2;
          if (left == 0) {
            total += part;
            part = f32x4_t{0.f, 0.f, 0.f, 0.f};
            left = a.dzSteps;
          }
        }
      }
    }
    total += part;
  }
  // dA3, dA2 and dA1 in turn: masked, as fragments to memory and by row to LDS for the next product.
#pragma unroll
  for (int layer = 2; layer >= 0; --layer) {
    float d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q] = (live[layer] >> q & 1u) ? total[q] : 0.f;
    const uint2 packed = make_uint2(pack_bf16(d[0], d[1]), pack_bf16(d[2], d[3]));
    *(uint2 *)(a.act + block_at(a.blocks, 8 * (4 + layer) + w, rb) + stored) = packed;
    if (layer == 0) break;
    *(uint16_t *)(nxt + (4 * g + 0) * kActPitch + (16 * w + n) * 2) = (uint16_t)packed.x;
    *(uint16_t *)(nxt + (4 * g + 1) * kActPitch + (16 * w + n) * 2) = (uint16_t)(packed.x >> 16);
    *(uint16_t *)(nxt + (4 * g + 2) * kActPitch + (16 * w + n) * 2) = (uint16_t)packed.y;
    *(uint16_t *)(nxt + (4 * g + 3) * kActPitch + (16 * w + n) * 2) = (uint16_t)(packed.y >> 16);
    __syncthreads();
    Frag x[4];
    load_rows(nxt, x);
    total = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) total = mfma16(x[ks], back[layer - 1][ks], total);
    unsigned char *t = cur;
    cur = nxt;
    nxt = t;
  }
}

// ------------------------------------------------------------------------------------------------
// Weight gradients
// ------------------------------------------------------------------------------------------------
constexpr int kSumRows = 256;  // rays per partial sum of a bias gradient

struct WeightArgs {
  const uint16_t *act, *dz;
  uint32_t n, blocks;
  uint32_t per4, split4, per3, split3;  // rays per split, splits
  float *ws4, *ws3;                     // partial products [split][4096][128], [layer][split][128][128]
  float *sum4, *sum3;                   // bias partial sums [chunk][4096], [layer][chunk][128]
  uint32_t chunks;
  const float *loss;                    // per ray (a multiple of 32 of them)
  TrainStats *stats;
};

constexpr int kSteps = 4;  // 32-ray steps per chunk of input activations staged in LDS (32 KB, two of them)
constexpr uint32_t kChunkRays = 32 * kSteps;
typedef uint4 ChunkLds[2][kSteps][8][64];

// One wave: MB blocks of 16 gradient columns (fragments at A, A + aStride...) against all 128 input
// columns B, over rays [beg, end); and the columns' sums over the 256-ray chunks that start there. The
// workgroup's four waves share the input fragments through LDS: every wave multiplies with all of them,
// and from L2 each step's eight loads would be waited for. A wave's own fragments are prefetched
// kAhead steps ahead, as dZ comes from beyond L2.
// out(mb, row): where row `row` of block mb goes; sumOut(mb, chunk, value) for the lanes that hold a sum.
template <int MB, class Out, class Sum>
__device__ __forceinline__ void weight_block(const uint16_t *__restrict__ A, size_t aStride,
                                             const uint16_t *__restrict__ B, uint32_t blocks, uint32_t n, uint32_t beg,
                                             uint32_t end, ChunkLds &lds, Out out, Sum sumOut) {
  const int tid = threadIdx.x, l = tid & 63, g = l >> 4;
  const uint32_t rays = (n + 31u) / 32u * 32u;
  const uint32_t sumBeg = (beg + kSumRows - 1) / kSumRows * kSumRows;
  const uint32_t sumEnd = min((end + kSumRows - 1) / kSumRows * kSumRows, rays);
  const uint32_t last = max(end, sumEnd > sumBeg ? sumEnd : 0u);  // end <= rays
  f32x4_t acc[MB][8];
  float col[MB][8];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[m][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      col[m][j] = 0.f;
    }
  constexpr int kAhead = 2 * kSteps;
  Frag a[kAhead][MB];
  auto load_a = [&](uint32_t r, Frag (&f)[MB]) {
#pragma unroll
    for (int m = 0; m < MB; ++m) f[m].u = *(const uint4 *)(A + m * aStride + (size_t)(r >> 4) * 256 + l * 8);
  };
  // Wave w copies fragments w, w + 4, ... of a chunk's 32.
  uint4 next[8];
  auto load_b = [&](uint32_t r0) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t f = (uint32_t)(tid >> 6) + 4u * u, r = r0 + 32u * (f >> 3);
      next[u] = r < end ? *(const uint4 *)(B + (size_t)(f & 7u) * blocks * 256 + (size_t)(r >> 4) * 256 + l * 8)
                        : make_uint4(0, 0, 0, 0);
    }
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t f = (uint32_t)(tid >> 6) + 4u * u;
      lds[buf][f >> 3][f & 7u][l] = next[u];
    }
  };
  load_b(beg);
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (beg + 32u * u < last) load_a(beg + 32u * u, a[u]);
  store_b(0);
  __syncthreads();
  for (uint32_t r0 = beg; r0 < last; r0 += 2 * kChunkRays) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t rc = r0 + half * kChunkRays;
      if (rc >= last) break;  // uniform over the workgroup
      if (rc + kChunkRays < last) load_b(rc + kChunkRays);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const uint32_t r = rc + 32u * s;
        if (r >= last) break;
        Frag x[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) x[m] = a[half * kSteps + s][m];
        if (r + 32u * kAhead < last) load_a(r + 32u * kAhead, a[half * kSteps + s]);
        if (r < end) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            Frag b;
            b.u = lds[half][s][j][l];
#pragma unroll
            for (int m = 0; m < MB; ++m) acc[m][j] = mfma16(x[m], b, acc[m][j]);
          }
        }
        // Rays 8 g + e of every 32 are summed apart, then in order over g and e.
        if (r >= sumBeg && r < sumEnd) {
#pragma unroll
          for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int e = 0; e < 8; ++e) col[m][e] += bf2f(x[m].h[e]);
          if ((r + 32u) % kSumRows == 0u || r + 32u >= sumEnd) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
              float t = 0.f;
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                float c = q ? __shfl(t, (l - 16) & 63, 64) : 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) c += col[m][e];
                if (g == q) t = c;
              }
              if (g == 3) sumOut(m, r / kSumRows, t);
#pragma unroll
              for (int e = 0; e < 8; ++e) col[m][e] = 0.f;
            }
          }
        }
      }
      if (rc + kChunkRays < last) store_b(half ^ 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float *row = out(m, 4 * g + q) + (l & 15);
#pragma unroll
      for (int j = 0; j < 8; ++j) row[16 * j] = acc[m][j][q];
    }
}

// Adds the batch's losses to the epoch's, in 64 bits and in a fixed order (a thread's own, then by halves
// over the threads). In one running fp32 sum a ray adds 1 / batch of a loss to a sum of one loss per batch:
// half a million rays in batches of 1,024 were off by 2.5e-4, 131,072 in batches of 8,192 by 5e-6.
__device__ __forceinline__ void sum_losses(const WeightArgs &a, double *lds) {
  double sum = 0.0;
  for (uint32_t u = threadIdx.x; u < a.blocks * 4u; u += 256u) {
    const float4 x = ((const float4 *)a.loss)[u];
    sum += ((double)x.x + (double)x.y) + ((double)x.z + (double)x.w);
  }
  lds[threadIdx.x] = sum;
  for (uint32_t o = 128; o >= 1; o >>= 1) {
    __syncthreads();
    if (threadIdx.x < o) lds[threadIdx.x] += lds[threadIdx.x + o];
  }
  if (threadIdx.x == 0) a.stats->loss += lds[0];
}

// Workgroup 0 adds the rays' losses to the epoch's; then 64 split4 workgroups: four class
// blocks of the output layer, a wave each, over one split; then 3 split3 of the hidden layers, two of
// their eight column blocks per wave. The output layer reads dZ once (67 MB for 8,192 rays, 14 us at a
// copy's rate, of 28); H3 comes from L2 (loaded by each wave itself instead of through LDS: 84 us).
__global__ void __launch_bounds__(256) k_train_weights(WeightArgs a) {
  __shared__ ChunkLds s_in;
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t l = threadIdx.x & 63u;
  if (blockIdx.x == 0) {
    sum_losses(a, (double *)s_in);
    return;
  }
  const uint32_t bid = blockIdx.x - 1u;
  const size_t cols = (size_t)8 * a.blocks * 256;  // an array of 128 columns
  if (bid < 64u * a.split4) {
    const uint32_t z = bid / 64u, cb = (bid % 64u) * 4u + w;
    const uint32_t beg = z * a.per4, end = min(beg + a.per4, (a.n + 31u) / 32u * 32u);
    auto out = [&](int, uint32_t m) {
      return a.ws4 + ((size_t)z * kMlpOut + class_of(cb / kRowBlocks, cb % kRowBlocks, m)) * kMlpHid;
    };
    auto sum = [&](int, uint32_t chunk, float t) {
      a.sum4[(size_t)chunk * kMlpOut + class_of(cb / kRowBlocks, cb % kRowBlocks, l & 15u)] = t;
    };
    weight_block<1>(a.dz + block_at(a.blocks, cb, 0), 0, a.act + 3 * cols, a.blocks, a.n, beg, end, s_in, out, sum);
  } else {
    const uint32_t k = bid - 64u * a.split4, layer = k / a.split3, z = k % a.split3;
    const uint32_t beg = z * a.per3, end = min(beg + a.per3, (a.n + 31u) / 32u * 32u);
    auto out = [&](int mb, uint32_t m) {
      return a.ws3 + (((size_t)layer * a.split3 + z) * kMlpHid + (2 * w + mb) * 16 + m) * kMlpHid;
    };
    auto sum = [&](int mb, uint32_t chunk, float t) {
      a.sum3[((size_t)layer * a.chunks + chunk) * kMlpHid + (2 * w + mb) * 16 + (l & 15u)] = t;
    };
    weight_block<2>(a.act + (4 + layer) * cols + block_at(a.blocks, 2 * w, 0), (size_t)a.blocks * 256,
                    a.act + layer * cols, a.blocks, a.n, beg, end, s_in, out, sum);
  }
}

// ------------------------------------------------------------------------------------------------
// Reduction and update
// ------------------------------------------------------------------------------------------------
// Where flat parameter i belongs.
struct ParamPlace {
  int layer;
  bool bias;
  uint32_t out, in;
};
__host__ __device__ inline ParamPlace param_place(uint32_t i) {
  constexpr uint32_t kLayer = (uint32_t)(kMlpW + kMlpHid);
  const uint32_t layer = i < 3 * kLayer ? i / kLayer : 3u;
  const uint32_t at = i - layer * kLayer, weights = layer < 3 ? (uint32_t)kMlpW : (uint32_t)kMlpW4;
  if (at >= weights) return {(int)layer, true, at - weights, 0u};
  return {(int)layer, false, at / kMlpHid, at % kMlpHid};
}

__device__ __forceinline__ void store_param(const ParamPlace &p, float v, const MlpWeights &o) {
  if (p.bias) {
    o.bias[p.layer * kMlpHid + p.out] = v;
    return;
  }
  const uint16_t h = f2bf(v);
  o.rows[mlp_bf16_offset(p.layer) + (size_t)p.out * kMlpHid + p.in] = h;
  o.fwd[fwd_fragment(p.layer, p.out, p.in)] = h;
  o.bwd[bwd_fragment(p.layer, p.out, p.in)] = h;
}

struct AdamArgs {
  float *w, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};

// kAdam: Adam (bias-corrected) on the fp32 parameters, else the gradients go to `grads`.
template <bool kAdam>
__global__ void __launch_bounds__(256) k_train_update(WeightArgs a, AdamArgs d, MlpWeights o, float *__restrict__ grads) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= kMlpParams) return;
  const ParamPlace p = param_place(i);
  const float *src;
  size_t stride;
  uint32_t count;
  if (p.bias) {
    src = p.layer == 3 ? a.sum4 + p.out : a.sum3 + (size_t)p.layer * a.chunks * kMlpHid + p.out;
    stride = p.layer == 3 ? kMlpOut : kMlpHid;
    count = a.chunks;
  } else {
    const size_t at = (size_t)p.out * kMlpHid + p.in;
    src = p.layer == 3 ? a.ws4 + at : a.ws3 + (size_t)p.layer * a.split3 * kMlpW + at;
    stride = p.layer == 3 ? kMlpW4 : kMlpW;
    count = p.layer == 3 ? a.split4 : a.split3;
  }
  float gi = 0.f;
  uint32_t z = 0;
  for (; z + 4 <= count; z += 4) {  // four loads in flight, added in order
    const float x0 = src[z * stride], x1 = src[(z + 1) * stride], x2 = src[(z + 2) * stride], x3 = src[(z + 3) * stride];
    gi += x0;
    gi += x1;
    gi += x2;
    gi += x3;
  }
  for (; z < count; ++z) gi += src[z * stride];
  if (!kAdam) {
    grads[i] = gi;
    return;
  }
  const float mi = d.b1 * d.m[i] + (1.f - d.b1) * gi;
  const float vi = d.b2 * d.v[i] + (1.f - d.b2) * gi * gi;
  d.m[i] = mi;
  d.v[i] = vi;
  const float mh = mi / d.c1, vh = vi / d.c2;
  const float wi = d.w[i] - d.lr * mh / (sqrtf(vh) + d.eps);
  d.w[i] = wi;
  store_param(p, wi, o);
}

__global__ void __launch_bounds__(256) k_store_params(const float *__restrict__ w, MlpWeights o) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < kMlpParams) store_param(param_place(i), w[i], o);
}

uint32_t even_blocks(uint32_t n) { return (n + 31u) / 32u * 2u; }

// Splits of a product's K range: few output tiles (64 x 64) over a long K are split so that about 512
// workgroups run, each over at least 256 of K in whole steps of 64.
void split_k(uint32_t tiles, uint32_t k, uint32_t &per, uint32_t &split) {
  split = 1;
  if (tiles < 256 && k >= 512) split = std::min(std::max(512 / tiles, 1u), k / 256);
  per = ((k + split - 1) / split + 63) / 64 * 64;
  split = std::max(1u, (k + per - 1) / per);
}

WeightArgs weight_args(const Proposal *p, uint32_t n) {
  WeightArgs a{};
  a.act = p->act;
  a.dz = p->dZ;
  a.n = n;
  a.blocks = even_blocks(n);
  split_k(kMlpOut / 64 * (kMlpHid / 64), n, a.per4, a.split4);
  split_k(4, n, a.per3, a.split3);
  a.chunks = (n + kSumRows - 1) / kSumRows;
  a.ws4 = p->trainWs;
  a.ws3 = a.ws4 + (size_t)a.split4 * kMlpW4;
  a.sum4 = a.ws3 + (size_t)3 * a.split3 * kMlpW;
  a.sum3 = a.sum4 + (size_t)a.chunks * kMlpOut;
  a.loss = p->rowLoss;
  a.stats = p->stats;
  return a;
}

}  // namespace

TrainBytes mlp_train_bytes(uint32_t maxBatch) {
  const size_t rays = (size_t)even_blocks(maxBatch) * 16, chunks = (maxBatch + kSumRows - 1) / kSumRows;
  // splits: at most 4 of the output layer, K / 256 up to 128 of the hidden ones
  const size_t split3 = std::min<size_t>(128, std::max<size_t>(1, maxBatch / 256));
  return {rays * 7 * kMlpHid * 2, rays * kMlpOut * 2, rays * 4,
          (4 * kMlpW4 + 3 * split3 * kMlpW + chunks * (kMlpOut + 3 * kMlpHid)) * 4};
}

void mlp_store_params(Context *ctx, hipStream_t s, Proposal *p) {
  launch(ctx, s, "mlp_store_params", k_store_params, dim3((unsigned)((kMlpParams + 255) / 256)), dim3(256), 0,
         (const float *)p->w, p->weights);
}

// Forward and backward of one batch: what the weight gradients are reduced from, loss and top-1 count.
// The loss and its gradient are scaled by 1 / labelled.
static void train_batch(Context *ctx, hipStream_t s, Proposal *p, const void *rays, const int32_t *labels, uint32_t n,
                        uint32_t labelled, const WeightArgs &wa) {
  TrainArgs a{};
  a.rays = (const GPRTRay *)rays;
  a.labels = labels;
  a.n = n;
  a.blocks = wa.blocks;
  a.scale = labelled ? 1.0f / (float)labelled : 0.f;
  a.wf = p->weights.fwd;
  a.wb = p->weights.bwd;
  a.bias = p->weights.bias;
  a.act = p->act;
  a.dz = p->dZ;
  uint32_t per, split;
  split_k(2 * ((n + 63) / 64), kMlpOut, per, split);
  a.dzSteps = (int)per / 32;
  a.loss = p->rowLoss;
  a.correct = &p->stats->correct;
  launch(ctx, s, "mlp_train_rows", k_train_rows, dim3(a.blocks), dim3(kRowWaves * 64), kRowLds, a);
  launch(ctx, s, "mlp_train_weights", k_train_weights, dim3(1 + 64 * wa.split4 + 3 * wa.split3), dim3(256), 0, wa);
}

void mlp_gradients(Context *ctx, hipStream_t s, Proposal *p, const void *rays, const int32_t *labels, uint32_t n,
                   uint32_t labelled) {
  const WeightArgs wa = weight_args(p, n);
  train_batch(ctx, s, p, rays, labels, n, labelled, wa);
  launch(ctx, s, "mlp_train_update", k_train_update<false>, dim3((unsigned)((kMlpParams + 255) / 256)), dim3(256), 0,
         wa, AdamArgs{}, p->weights, p->g);
}

void mlp_train_step(Context *ctx, hipStream_t s, Proposal *p, const void *rays, const int32_t *labels, uint32_t n,
                    float lr) {
  const WeightArgs wa = weight_args(p, n);
  train_batch(ctx, s, p, rays, labels, n, n, wa);
  p->step += 1;
  AdamArgs d{p->w, p->m, p->v, lr, 0.9f, 0.999f, 1e-8f, 0.f, 0.f};
  d.c1 = 1.f - std::pow(d.b1, (float)p->step);
  d.c2 = 1.f - std::pow(d.b2, (float)p->step);
  launch(ctx, s, "mlp_train_update", k_train_update<true>, dim3((unsigned)((kMlpParams + 255) / 256)), dim3(256), 0, wa,
         d, p->weights, p->g);
}

}  // namespace gprt
