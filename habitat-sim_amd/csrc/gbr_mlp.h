// Chunk-visibility MLP: shapes, launch arguments and launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gbr {

constexpr int kMlpIn = 32;
constexpr int kMlpHidden = 256;  // GBR_VIS_HIDDEN

// One minibatch's forward and backward pass: batch rows (a multiple of 32)
// taken from X [total][32], Y [total] by hash(seed, step, i) mod total, or rows
// 0 .. batch - 1 of X and Y when total is 0.
struct TrainArgs {
  int batch;
  const uint16_t* X;
  const uint8_t* Y;
  uint64_t total, seed, step;
  float pos_weight;
  // weights
  const uint16_t *W1, *W2, *W2t, *w3;
  const float *b1, *b2, *b3;
  // scratch: X, H1, H2, dH2, dH1 in fragment order ([columns][batch] values;
  // frag_at() in gbr_mlp.hip), dH2 by rows, and per row the loss and its
  // gradient by the logit
  uint16_t *Xt, *H1t, *H2t, *dH2t, *dH1t, *dH2;
  float *dl, *loss;
  // gradients of the mean weighted loss, and the loss summed over the batch
  float *gW1, *gb1, *gW2, *gb2, *gw3, *gb3, *loss_sum;
};

// One Adam step on n master weights; the bf16 copies of W1, W2 (also
// transposed) and w3, which start at at_w1, at_w2 and at_w3 of w.
struct AdamArgs {
  float* w;
  const float* g;
  float *m, *v;
  size_t n;
  float lr, b1, b2, eps, bc1, bc2;
  size_t at_w1, at_w2, at_w3;
  uint16_t *W1, *W2, *W2t, *w3;
};

hipError_t mlp_train(const TrainArgs& t, hipStream_t s);
hipError_t mlp_to_bf16(const float* in, size_t n, uint16_t* out, uint16_t* out_t, int rows,
                       int cols, hipStream_t s);
// logits of rows [0, min(rows, *rows_dev)) of X for rendering, in one fused
// pass with no intermediates in memory; at most max_blocks workgroups (0: one
// per 128 rows), each looping over 32-row tiles.  H1 and H2 are the training
// forward's bit for bit; the logit sums in another order.
hipError_t mlp_score(const uint16_t* X, const uint16_t* W1, const float* b1, const uint16_t* W2,
                     const float* b2, const uint16_t* w3, const float* b3, int rows,
                     const uint32_t* rows_dev, float* logits, int max_blocks, hipStream_t s);
hipError_t mlp_adam(const AdamArgs& a, hipStream_t s);

}  // namespace gbr
