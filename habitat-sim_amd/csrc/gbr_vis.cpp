// Learned visibility proposal: parameter handling, training loop and the
// forward/backward launch sequences of the chunk-visibility MLP.
#include "gbr_vis.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <vector>

namespace gbr {

namespace {

// float -> bf16 bits, round to nearest even (as the device's conversion)
uint16_t host_f2bf(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

}  // namespace

gbr_status VisModel::refresh_bf16(hipStream_t s) {
  TRY(W1b.reserve((size_t)kMlpHidden * kMlpIn));
  TRY(W2b.reserve((size_t)kMlpHidden * kMlpHidden));
  TRY(W2tb.reserve((size_t)kMlpHidden * kMlpHidden));
  TRY(w3b.reserve(kMlpHidden));
  HIP_TRY(mlp_to_bf16(w.ptr + kVisW1, (size_t)kMlpHidden * kMlpIn, W1b.ptr, nullptr, kMlpHidden,
                      kMlpIn, s));
  HIP_TRY(mlp_to_bf16(w.ptr + kVisW2, (size_t)kMlpHidden * kMlpHidden, W2b.ptr, W2tb.ptr,
                      kMlpHidden, kMlpHidden, s));
  HIP_TRY(mlp_to_bf16(w.ptr + kVisW3, kMlpHidden, w3b.ptr, nullptr, 1, kMlpHidden, s));
  return GBR_OK;
}

gbr_status VisModel::set_weights(const float* host, hipStream_t s) {
  TRY(w.reserve(kVisParams));
  TRY(g.reserve(kVisParams));
  TRY(m.reserve(kVisParams));
  TRY(v.reserve(kVisParams));
  HIP_TRY(hipMemcpyAsync(w.ptr, host, kVisParams * sizeof(float), hipMemcpyHostToDevice, s));
  HIP_TRY(hipMemsetAsync(m.ptr, 0, kVisParams * sizeof(float), s));
  HIP_TRY(hipMemsetAsync(v.ptr, 0, kVisParams * sizeof(float), s));
  adam_t = 0;
  TRY(refresh_bf16(s));
  HIP_TRY(hipStreamSynchronize(s));
  ready = true;
  return GBR_OK;
}

gbr_status VisModel::get_weights(float* host, hipStream_t s) {
  if (!ready) return fail(GBR_ERR_STATE, "visibility model: no weights (gbr_vis_init first)");
  HIP_TRY(hipMemcpyAsync(host, w.ptr, kVisParams * sizeof(float), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  return GBR_OK;
}

// He-uniform weights (fan-in), zero biases, the output bias at the prior
// log-odds of a chunk being visible (about one in four)
gbr_status VisModel::init(uint64_t seed, hipStream_t s) {
  std::vector<float> h(kVisParams, 0.0f);
  std::mt19937_64 rng(seed);
  auto fill = [&](size_t off, size_t n, int fan_in) {
    const float lim = std::sqrt(6.0f / (float)fan_in);
    std::uniform_real_distribution<float> u(-lim, lim);
    for (size_t i = 0; i < n; ++i) h[off + i] = u(rng);
  };
  fill(kVisW1, (size_t)kMlpHidden * kMlpIn, kMlpIn);
  fill(kVisW2, (size_t)kMlpHidden * kMlpHidden, kMlpHidden);
  fill(kVisW3, kMlpHidden, kMlpHidden);
  for (size_t i = 0; i < kMlpHidden; ++i) h[kVisW3 + i] *= 0.1f;
  h[kVisB3] = -1.0f;
  return set_weights(h.data(), s);
}

gbr_status VisModel::reserve_dataset(uint64_t rows_cap) {
  if (rows_cap <= cap && Xd.ptr) return GBR_OK;
  TRY(Xd.reserve((size_t)rows_cap * kMlpIn, true));
  TRY(Yd.reserve(rows_cap, true));
  cap = rows_cap;
  if (!positives.ptr) {
    TRY(positives.reserve(1));
    HIP_TRY(hipMemset(positives.ptr, 0, sizeof(uint32_t)));
  }
  return GBR_OK;
}

gbr_status VisModel::reserve_infer(size_t n) {
  n = std::max<size_t>((n + 31) & ~size_t(31), 32);
  TRY(Xi.reserve(n * kMlpIn));
  TRY(logits_i.reserve(n));
  TRY(prop.reserve(n));
  return GBR_OK;
}

gbr_status VisModel::reserve_batch(int batch) {
  if (batch <= bcap) return GBR_OK;
  const size_t b = (size_t)batch;
  TRY(Xb.reserve(b * kMlpIn));
  TRY(Xbt.reserve(b * kMlpIn));
  for (DevBuf<uint16_t>* x : {&H1t, &H2t, &dH2t, &dH1t, &dH2}) TRY(x->reserve(b * kMlpHidden));
  TRY(Yb.reserve(b));
  TRY(logits.reserve(b));
  TRY(dl.reserve(b));
  TRY(lossr.reserve(b));
  bcap = batch;
  return GBR_OK;
}

gbr_status VisModel::score(const uint16_t* X, int nrows, const uint32_t* rows_dev, float* out,
                           int max_blocks, hipStream_t s) {
  HIP_TRY(mlp_score(X, W1b.ptr, w.ptr + kVisB1, W2b.ptr, w.ptr + kVisB2, w3b.ptr, w.ptr + kVisB3,
                    nrows, rows_dev, out, max_blocks, s));
  return GBR_OK;
}

// gradients of the mean weighted loss over a batch of rows of X, Y (hashed by
// seed and step out of `total` rows, or the first `b` with total 0); the
// batch's loss lands in *loss_sum
gbr_status VisModel::backward(const uint16_t* X, const uint8_t* Y, uint64_t total, uint64_t seed,
                              uint64_t step, int b, float pos_weight, float* loss_sum, hipStream_t s) {
  TrainArgs t{};
  t.batch = b;
  t.X = X;
  t.Y = Y;
  t.total = total;
  t.seed = seed;
  t.step = step;
  t.pos_weight = pos_weight;
  t.W1 = W1b.ptr;
  t.W2 = W2b.ptr;
  t.W2t = W2tb.ptr;
  t.w3 = w3b.ptr;
  t.b1 = w.ptr + kVisB1;
  t.b2 = w.ptr + kVisB2;
  t.b3 = w.ptr + kVisB3;
  t.Xt = Xbt.ptr;
  t.H1t = H1t.ptr;
  t.H2t = H2t.ptr;
  t.dH2t = dH2t.ptr;
  t.dH1t = dH1t.ptr;
  t.dH2 = dH2.ptr;
  t.dl = dl.ptr;
  t.loss = lossr.ptr;
  t.gW1 = g.ptr + kVisW1;
  t.gb1 = g.ptr + kVisB1;
  t.gW2 = g.ptr + kVisW2;
  t.gb2 = g.ptr + kVisB2;
  t.gw3 = g.ptr + kVisW3;
  t.gb3 = g.ptr + kVisB3;
  t.loss_sum = loss_sum;
  HIP_TRY(mlp_train(t, s));
  return GBR_OK;
}

gbr_status VisModel::adam_step(const gbr_vis_fit_params& fp, hipStream_t s) {
  ++adam_t;
  AdamArgs a{};
  a.w = w.ptr;
  a.g = g.ptr;
  a.m = m.ptr;
  a.v = v.ptr;
  a.n = kVisParams;
  a.lr = fp.learning_rate;
  a.b1 = fp.beta1;
  a.b2 = fp.beta2;
  a.eps = fp.eps;
  a.bc1 = 1.0f - std::pow(fp.beta1, (float)adam_t);
  a.bc2 = 1.0f - std::pow(fp.beta2, (float)adam_t);
  a.at_w1 = kVisW1;
  a.at_w2 = kVisW2;
  a.at_w3 = kVisW3;
  a.W1 = W1b.ptr;
  a.W2 = W2b.ptr;
  a.W2t = W2tb.ptr;
  a.w3 = w3b.ptr;
  HIP_TRY(mlp_adam(a, s));
  return GBR_OK;
}

gbr_status VisModel::fit(const gbr_vis_fit_params& fp, gbr_vis_fit_report* rep, hipStream_t s) {
  if (!ready) return fail(GBR_ERR_STATE, "vis_fit: no weights (gbr_vis_init first)");
  if (rows == 0) return fail(GBR_ERR_STATE, "vis_fit: no training rows (gbr_vis_collect first)");
  if (fp.steps < 1 || fp.batch < 32 || fp.batch > 65536 || fp.batch % 32)
    return fail(GBR_ERR_ARGUMENT, "vis_fit: steps >= 1 and batch a multiple of 32 in [32, 65536]");
  TRY(reserve_batch(fp.batch));
  std::vector<float> sums((size_t)fp.steps, 0.0f);
  TRY(losses.reserve((size_t)fp.steps));
  for (int k = 0; k < fp.steps; ++k) {
    TRY(backward(Xd.ptr, Yd.ptr, rows, fp.seed, (uint64_t)k, fp.batch, fp.pos_weight, losses.ptr + k, s));
    TRY(adam_step(fp, s));
  }
  HIP_TRY(hipMemcpyAsync(sums.data(), losses.ptr, sums.size() * sizeof(float),
                         hipMemcpyDeviceToHost, s));
  uint32_t pos = 0;
  HIP_TRY(hipMemcpyAsync(&pos, positives.ptr, sizeof pos, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  if (rep) {
    rep->loss_first = sums[0] / (float)fp.batch;
    const int tail = std::max(1, fp.steps / 10);
    double t = 0.0;
    for (int k = fp.steps - tail; k < fp.steps; ++k) t += sums[(size_t)k];
    rep->loss_last = (float)(t / tail / fp.batch);
    rep->rows = rows;
    rep->positives = pos;
  }
  return GBR_OK;
}

gbr_status VisModel::loss_grad(const float* X, const uint8_t* labels, int n, float pos_weight,
                               float* loss, float* grad, hipStream_t s) {
  if (!ready) return fail(GBR_ERR_STATE, "vis_loss_grad: no weights (gbr_vis_init first)");
  if (n < 32 || n > 65536 || n % 32)
    return fail(GBR_ERR_ARGUMENT, "vis_loss_grad: rows must be a multiple of 32 in [32, 65536]");
  TRY(reserve_batch(n));
  TRY(losses.reserve(1));
  std::vector<uint16_t> xb((size_t)n * kMlpIn);
  for (size_t i = 0; i < xb.size(); ++i) xb[i] = host_f2bf(X[i]);
  HIP_TRY(hipMemcpyAsync(Xb.ptr, xb.data(), xb.size() * 2, hipMemcpyHostToDevice, s));
  HIP_TRY(hipMemcpyAsync(Yb.ptr, labels, (size_t)n, hipMemcpyHostToDevice, s));
  TRY(backward(Xb.ptr, Yb.ptr, 0, 0, 0, n, pos_weight, losses.ptr, s));
  float l = 0.0f;
  HIP_TRY(hipMemcpyAsync(&l, losses.ptr, sizeof l, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipMemcpyAsync(grad, g.ptr, kVisParams * sizeof(float), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  *loss = l / (float)n;
  return GBR_OK;
}

gbr_status VisModel::predict(const float* X, int n, float* out, hipStream_t s) {
  if (!ready) return fail(GBR_ERR_STATE, "vis_predict: no weights (gbr_vis_init first)");
  if (n < 1 || n > 65536) return fail(GBR_ERR_ARGUMENT, "vis_predict: rows must be in [1, 65536]");
  const int np = (n + 31) & ~31;
  TRY(reserve_batch(np));
  std::vector<uint16_t> xb((size_t)np * kMlpIn, 0);
  for (size_t i = 0; i < (size_t)n * kMlpIn; ++i) xb[i] = host_f2bf(X[i]);
  HIP_TRY(hipMemcpyAsync(Xb.ptr, xb.data(), xb.size() * 2, hipMemcpyHostToDevice, s));
  // the renderer's fused scorer, on few workgroups so that each loops over
  // several row tiles as it does on a frame's candidate rows
  TRY(score(Xb.ptr, n, nullptr, logits.ptr, 16, s));
  HIP_TRY(hipMemcpyAsync(out, logits.ptr, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  return GBR_OK;
}

}  // namespace gbr
