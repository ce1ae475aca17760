// opt_update.h — the arithmetic of the optimizers, one element at a time: the kernels of elementwise.hip
// and the fused update of a small net's step (tiny_net.hip). Built with -ffp-contract=off, like the
// reference's scalar code.
#pragma once
#include "common.h"

namespace tdh {
namespace {

// tiny_dnn/optimizers/optimizer.h; g = merged * grad_scale is layer::update_weight's
// diff (tiny_dnn/layers/layer.h:668-673). Scalars that the reference derives once per
// call from its float members (1 - b1_t, ...) arrive precomputed in float.
struct OptScalars {
  float alpha, lambda, mu, b1, b2, eps, omb1, omb2, omb1t, omb2t, grad_scale;
  double adamax_lr;  // alpha / (1.0 - b1_t), evaluated in double as the reference does
};

template <int KIND>
__device__ __forceinline__ void opt_one(float g, float &w, float &s0, float &s1,
                                        const OptScalars &p) {
  g *= p.grad_scale;
  if (KIND == TDH_OPT_SGD) {  // :185-188
    w = w - p.alpha * (g + p.lambda * w);
  } else if (KIND == TDH_OPT_MOMENTUM) {  // :205-213
    const float V = p.mu * s0 - p.alpha * (g + w * p.lambda);
    w += V;
    s0 = V;
  } else if (KIND == TDH_OPT_NESTEROV) {  // :231-239
    const float V = p.mu * s0 - p.alpha * (g + w * p.lambda);
    w += (-p.mu) * s0 + (1 + p.mu) * V;
    s0 = V;
  } else if (KIND == TDH_OPT_ADAM) {  // :112-127, eps inside the square root
    s0 = p.b1 * s0 + p.omb1 * g;
    s1 = p.b2 * s1 + p.omb2 * g * g;
    w -= p.alpha * (s0 / p.omb1t) / sqrtf((s1 / p.omb2t) + p.eps);
  } else if (KIND == TDH_OPT_ADAGRAD) {  // :60-66
    s0 += g * g;
    w -= p.alpha * g / (sqrtf(s0) + p.eps);
  } else if (KIND == TDH_OPT_RMSPROP) {  // :81-88
    s0 = p.mu * s0 + (1 - p.mu) * g * g;
    w -= p.alpha * g / sqrtf(s0 + p.eps);
  } else if (KIND == TDH_OPT_ADAMAX) {  // :153-165
    s0 = p.b1 * s0 + p.omb1 * g;
    s1 = fmaxf(p.b2 * s1, fabsf(g));
    w  = static_cast<float>(static_cast<double>(w) -
                           p.adamax_lr * static_cast<double>(s0 / (s1 + p.eps)));
  }
}

// state vectors of an optimizer, and how many of its powers advance with every update() call
__host__ __device__ constexpr int opt_states(const int kind) {
  return kind == TDH_OPT_SGD ? 0 : kind == TDH_OPT_ADAM || kind == TDH_OPT_ADAMAX ? 2 : 1;
}
__host__ __device__ constexpr int opt_powers(const int kind) { return kind == TDH_OPT_ADAM ? 2 : kind == TDH_OPT_ADAMAX ? 1 : 0; }
// (what depends on the powers is left to the kernel)
inline OptScalars opt_scalars(const tdh_opt &o, const float grad_scale) {
  OptScalars p;
  p.alpha = o.alpha; p.lambda = o.lambda; p.mu = o.mu; p.b1 = o.b1; p.b2 = o.b2;
  p.eps = o.eps;
  p.omb1 = 1.0f - o.b1; p.omb2 = 1.0f - o.b2;
  p.omb1t = p.omb2t = 0.0f;
  p.grad_scale = grad_scale;
  p.adamax_lr  = 0.0;
  return p;
}
// the powers after n update() calls
inline void opt_advance(tdh_opt *o, const int n) {
  for (int j = 0; j < n; ++j) {
    if (opt_powers(o->kind) >= 1) o->b1_t *= o->b1;
    if (opt_powers(o->kind) == 2) o->b2_t *= o->b2;
  }
}

}  // namespace
}  // namespace tdh
