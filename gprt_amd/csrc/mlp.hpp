// Treelet proposal network: sizes, parameter layout and host-side state.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>

namespace gprt {

struct Context;
struct Accel;

constexpr int kMlpBands = 8;
constexpr int kMlpIn = 6 + 6 * 2 * kMlpBands;  // 102
constexpr int kMlpInPad = 128;
constexpr int kMlpHid = 128;
constexpr int kMlpOut = 4096;
constexpr int kMlpCutDepth = 12;

// Flat fp32 parameter layout: W1t b1 W2t b2 W3t b3 W4t b4 (Wt[out][in], inputs padded to 128).
constexpr size_t kMlpW = (size_t)kMlpHid * kMlpInPad;  // 16384 per hidden layer
constexpr size_t kMlpW4 = (size_t)kMlpOut * kMlpHid;   // 524288
constexpr size_t kMlpParams = 3 * (kMlpW + kMlpHid) + kMlpW4 + kMlpOut;
constexpr size_t kMlpWeights = 3 * kMlpW + kMlpW4;    // bf16 copies
constexpr size_t kMlpBiases = 3 * kMlpHid + kMlpOut;  // contiguous bias vector used by inference

inline size_t mlp_weight_offset(int layer) { return (size_t)layer * (kMlpW + kMlpHid); }
inline size_t mlp_bias_offset(int layer) { return layer < 3 ? mlp_weight_offset(layer) + kMlpW : 3 * (kMlpW + kMlpHid) + kMlpW4; }
inline size_t mlp_weight_size(int layer) { return layer < 3 ? kMlpW : kMlpW4; }
constexpr size_t mlp_bf16_offset(int layer) { return (size_t)layer * kMlpW; }

// The bf16 weights in the layouts of their readers, and the biases b1 b2 b3 b4 in fp32.
struct MlpWeights {
  uint16_t *rows;  // W1t W2t W3t W4t, Wt[out][in]
  uint16_t *fwd;   // MFMA fragments of W^T (mlp_train.hip)
  uint16_t *bwd;   // MFMA fragments of W (W1's unused)
  float *bias;
};

// What an epoch has added up: the batches' mean losses, and the rays whose class was right.
struct TrainStats {
  double loss;
  uint32_t correct, unused;
};

struct Proposal {
  void *block = nullptr;
  size_t blockBytes = 0;
  uint32_t maxBatch = 0;
  float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // fp32 params, grads, Adam moments
  MlpWeights weights{};
  TrainStats *stats = nullptr;
  uint16_t *X = nullptr, *H = nullptr;  // features and hidden activations of gprtProposalLogits
  float *Z = nullptr;                   // its logits
  // A training batch: activations and their gradients, dZ (bf16 fragments), and the products' partial
  // sums (mlp_train_bytes).
  uint16_t *act = nullptr, *dZ = nullptr;
  float *trainWs = nullptr;
  float *rowLoss = nullptr;
  uint32_t step = 0;
  // Treelets of the accel the proposal serves.
  void *treeBlock = nullptr;
  uint32_t treeCap = 0, treePrims = 0, numClasses = 0;
  int32_t *classRoot = nullptr, *innerClass = nullptr, *leafClass = nullptr, *primClass = nullptr;
  uint32_t *numClassesDev = nullptr;
  Accel *accel = nullptr;
  bool instanceBound = false;  // bound to an instance accel: classes of its top-level leaves
  // Per-ray scratch for proposal-first traces.
  void *rayScratch = nullptr;
  size_t rayScratchBytes = 0;
  // Confidence gate of proposal-first traces: rays whose top logit is below it are traced without
  // their proposal (-INFINITY: every ray uses its proposal).
  float gate = -INFINITY;
  // Overlap of proposal-first traces: the rays go in `overlapChunks` chunks, each inferred on the
  // context's second stream while the previous chunk is traversed on its main stream with
  // `overlapBlocks` traversal workgroups per CU (room for the inference on the same CUs).
  // overlapChunks < 2: inference, then one traversal.
  uint32_t overlapChunks = 0;
  uint32_t overlapBlocks = 0;
};

size_t mlp_param_count();
bool mlp_alloc(Context *ctx, Proposal *p, uint32_t maxBatch);
void mlp_release(Proposal *p);
bool mlp_set_params(Context *ctx, hipStream_t s, Proposal *p, const float *host);
// Writes the bf16 weights and the biases from the fp32 parameters.
void mlp_store_params(Context *ctx, hipStream_t s, Proposal *p);
void mlp_forward_batch(Context *ctx, hipStream_t s, Proposal *p, const void *rays, uint32_t n);
// One minibatch of n <= maxBatch rays: forward, backward and Adam; loss (mean over the batch) and top-1
// count are added to stats.
void mlp_train_step(Context *ctx, hipStream_t s, Proposal *p, const void *rays, const int32_t *labels, uint32_t n,
                    float lr);
// The gradient of the mean cross-entropy over `labelled` rays, into p->g.
void mlp_gradients(Context *ctx, hipStream_t s, Proposal *p, const void *rays, const int32_t *labels, uint32_t n,
                   uint32_t labelled);
struct TrainBytes {
  size_t act, dz, loss, ws;
};
TrainBytes mlp_train_bytes(uint32_t maxBatch);
void mlp_labels(Context *ctx, hipStream_t s, Proposal *p, const void *hits, uint32_t n, int32_t *labels);
// Classes of top-level leaves (instance accels): labels[i] = leafClass[leaves[i]], or -1.
void mlp_labels_of_leaves(Context *ctx, hipStream_t s, Proposal *p, const int32_t *leaves, uint32_t n,
                          int32_t *labels);
// Top-1 class per ray (and its top logit when `logit` is set); a ray whose top logit is below
// `gate` gets class -1 (-INFINITY: every ray keeps its class).
void mlp_infer(Context *ctx, hipStream_t s, Proposal *p, const void *rays, uint32_t n, int32_t *cls, float *logit,
               float gate);
bool mlp_treelets(Context *ctx, hipStream_t s, Proposal *p, Accel *a, int depth);

}  // namespace gprt
