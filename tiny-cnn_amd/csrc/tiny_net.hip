// tiny_net.hip — the whole train step of a small net in two to five launches, the optimizer's included.
//
// A net whose activations of one sample fit in LDS (LeNet-5: 15 k floats) spends its step in
// launches, not in arithmetic: 24 kernels of 3-10 us on tensors of a few kilobytes. Here one
// workgroup takes one sample through the chain that has to run in order: forward through every
// layer with all layer outputs kept in LDS, the loss gradient, and the input gradients backward
// through every layer, reading the filters through the caches (tiny_net_step_kernel). Where the batch
// leaves compute units for it, the ends of that chain run a channel a workgroup, in a launch in front
// and one behind (tiny_net_front_kernel, tiny_net_back_kernel). Layer outputs, input gradients
// and max-pool records are also written to the net's tensors in memory, so a caller sees what
// the layer-by-layer path leaves. Nothing in that chain waits for a weight gradient, so those
// are a launch behind it, (piece of a layer's parameters) x (group of samples), that reads
// the layer's input and output gradient back from memory (tiny_net_param_kernel). A batch of one
// group is updated there; what several leave as one slice each ([group][tensor]) the
// optimizer's kernel adds up on its way (the split sums it also takes from the
// layer-by-layer step); a step that stops at the gradients adds the slices to the gradient tensors in the groups'
// order, as edge::merge_grads does with samples (tiny_dnn/node.h:89-103), with a kernel of its own.
//
// The arithmetic of each layer follows the reference's scalar kernels: convolution sums the
// taps of one input channel, then adds channel sums in channel order, then the bias
// (conv2d_op_internal.h:13-74); pooling scans windows row by row (maxpool_op_internal.h:16-40,
// average_pooling_layer.h:25-106). Sums that one thread would walk alone for too long (a bias
// gradient, a first layer's weight gradient, a fully-connected output) are split over a group
// of neighbouring lanes and added with butterfly shuffles, a fixed tree.
// Built with -ffp-contract=off like the other scalar kernels.
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <vector>

#include "opt_update.h"
#include "tiny_net.h"

namespace tdh {

namespace {

constexpr int TN_THREADS = 1024;

__device__ __forceinline__ float tn_act_fwd(int act, float p0, float x) {
  switch (act) {
    case TDH_ACT_TANH: return tanhf(x);
    case TDH_ACT_RELU: return x > 0.0f ? x : 0.0f;
    case TDH_ACT_SIGMOID: return 1.0f / (1.0f + expf(-x));
    case TDH_ACT_LEAKY_RELU: return x > 0.0f ? x : p0 * x;
    default: return x;
  }
}
// the factor of the activation's backward pass, from its OUTPUT (tanh_layer.h:30-38,
// relu_layer.h:31-39, sigmoid_layer.h:30-38, leaky_relu_layer.h:80-88)
__device__ __forceinline__ float tn_act_bwd(int act, float p0, float y, float dy) {
  switch (act) {
    case TDH_ACT_TANH: return dy * (1.0f - y * y);
    case TDH_ACT_RELU: return dy * (y > 0.0f ? 1.0f : 0.0f);
    case TDH_ACT_SIGMOID: return dy * y * (1.0f - y);
    case TDH_ACT_LEAKY_RELU: return dy * (y > 0.0f ? 1.0f : p0);
    default: return dy;
  }
}

// sum over the `group` (a power of two <= 64) neighbouring lanes that hold the pieces of one value
__device__ __forceinline__ float group_sum(float v, int group) {
  for (int off = group >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
// sum over a wave, in lane 63, without LDS: rows of sixteen lanes, then the rows in order
__device__ __forceinline__ float wave_sum_63(float v) {
  auto step = [](float x, auto ctrl, auto rows) {
    return x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), ctrl(), rows(), 0xf, false));
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0xf> all;
  v = step(v, integral_constant<int, 0x111>(), all);   // row_shr:1
  v = step(v, integral_constant<int, 0x112>(), all);
  v = step(v, integral_constant<int, 0x114>(), all);
  v = step(v, integral_constant<int, 0x118>(), all);
  v = step(v, integral_constant<int, 0x142>(), integral_constant<int, 0xa>());   // row_bcast:15
  return step(v, integral_constant<int, 0x143>(), integral_constant<int, 0xc>());   // row_bcast:31
}
// sum over each sixteen lanes, in all of them
__device__ __forceinline__ float row_sum(float v) {
  auto step = [](float x, auto ctrl) {
    return x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), ctrl(), 0xf, 0xf, false));
  };
  using std::integral_constant;
  v = step(v, integral_constant<int, 0x128>());   // row_ror:8
  v = step(v, integral_constant<int, 0x124>());
  v = step(v, integral_constant<int, 0x122>());
  return step(v, integral_constant<int, 0x121>());
}
// lanes per value, so that `values` of them make at least two rounds of the workgroup busy
// and no lane's share of `length` terms is empty
__device__ __forceinline__ int group_for(int values, int length) {
  int g = 64;
  while (g > 1 && (values * g > 2 * TN_THREADS || g > length)) g >>= 1;
  return g;
}

// A barrier for data that went through LDS only: the waves wait for their own LDS traffic and
// meet, while their stores to memory stay in flight (__syncthreads would also wait for those,
// a microsecond per layer here). Wherever one thread reads memory another thread of the
// workgroup wrote, __syncthreads stays.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// memory -> LDS with eight reads in flight per thread
template <int NT>
__device__ __forceinline__ void fill_lds(float *dst, const float *__restrict__ src, const int n) {
  for (int base = 0; base < n; base += 8 * NT) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = base + j * NT + static_cast<int>(threadIdx.x);
      v[j] = src[i < n ? i : 0];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = base + j * NT + static_cast<int>(threadIdx.x);
      if (i < n) dst[i] = v[j];
    }
  }
}

// Every function below copies the sizes it needs out of the plan (uniform values: scalar
// registers) before its loops, and is inlined into the kernel so that `in`, `out`, `dy`, `dx`
// stay LDS addresses.
#define TN_INLINE __device__ __forceinline__

// Where a layer's outputs go, and those of a pointwise activation behind it that runs in the same phase (later layers
// read that one's outputs only)
struct FwdOut {
  float *out, *gout;      // LDS: what the next layer reads; memory: this layer's
  int act;                // the activation's, or TDH_ACT_NONE
  float p0, *gact;
  __device__ __forceinline__ void operator()(const int i, float v) const {
    gout[i] = v;
    if (act != TDH_ACT_NONE) {
      v = tn_act_fwd(act, p0, v);
      gact[i] = v;
    }
    out[i] = v;
  }
};
// The same on the way back: a gradient with respect to a layer's input (gdx: its place in memory, or NULL), and through
// the activation in front of that layer
struct BwdOut {
  float *dx, *gdx;
  int act;
  float p0, *gact;
  const float *y;         // the activation's outputs
  __device__ __forceinline__ void operator()(const int i, float v) const {
    if (gdx) gdx[i] = v;
    if (act != TDH_ACT_NONE) {
      v = tn_act_bwd(act, p0, y[i], v);
      if (gact) gact[i] = v;
    }
    dx[i] = v;
  }
};
TN_INLINE FwdOut fwd_out(const TinyPlan *__restrict__ plan, float *lds, const int li, const int s, const bool with_act) {
  const TinyLayer *L = &plan->l[li], *A = with_act ? L + 1 : L;   // (a pointwise activation has its input's size)
  const size_t at = static_cast<size_t>(s) * L->out_size;
  return {lds + A->lds_out, L->out + at, with_act ? A->act : TDH_ACT_NONE, A->p0, A->out + at};
}
TN_INLINE BwdOut bwd_out(const TinyPlan *__restrict__ plan, const float *lds, float *dx, const int li, const int s,
                         const bool with_act) {
  const TinyLayer *L = &plan->l[li], *A = with_act ? L - 1 : L;
  const size_t at = static_cast<size_t>(s) * L->in_size;
  return {dx, L->dx ? L->dx + at : nullptr, with_act ? A->act : TDH_ACT_NONE, A->p0, A->dx ? A->dx + at : nullptr, lds + A->lds_out};
}
__host__ __device__ inline bool is_pointwise(const TinyLayer &L) { return L.kind == TDH_L_ACT && L.act != TDH_ACT_SOFTMAX; }
__host__ __device__ inline bool is_pool(const TinyLayer &L) { return L.kind == TDH_L_MAXPOOL || L.kind == TDH_L_AVEPOOL; }

// ------------------------------------------------------------------ forward
TN_INLINE void conv_fwd(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, K = Lp->K, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S;
  const int sh = Lp->sh, sw = Lp->sw, ph = Lp->ph, pw = Lp->pw, has_bias = Lp->has_bias;
  const FastDiv d_plane = Lp->d_oplane, d_ow = Lp->d_ow;
  const float *__restrict__ w = Lp->w;
  const float *__restrict__ b = Lp->b;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  const int plane = OH * OW, total = K * plane, taps = R * S;
  for (int o = threadIdx.x; o < total; o += TN_THREADS) {
    uint32_t co, r, oy, ox;
    d_plane.divmod(o, co, r);
    d_ow.divmod(r, oy, ox);
    const int y0 = static_cast<int>(oy) * sh - ph, x0 = static_cast<int>(ox) * sw - pw;
    const int wy0 = max(0, -y0), wy1 = min(R, H - y0), wx0 = max(0, -x0), wx1 = min(S, W - x0);
    float acc = 0.0f;
    for (int ci = 0; ci < C; ++ci) {
      if (tbl && !tbl[ci * K + co]) continue;
      const float *wp = w + static_cast<size_t>(co * C + ci) * taps;
      const float *ip = in + ci * H * W + y0 * W + x0;
      float sum = 0.0f;
      for (int wy = wy0; wy < wy1; ++wy)
        for (int wx = wx0; wx < wx1; ++wx) sum += wp[wy * S + wx] * ip[wy * W + wx];
      acc += sum;
    }
    if (has_bias) acc += b[co];
    out[o]  = acc;
    gout[o] = acc;
  }
}

// fully_connected_op_internal.h:15-36: out[i] = sum_c W[c*out + i] * in[c] + b[i]; the sum over
// c is split over a group of lanes
TN_INLINE void fc_fwd(const TinyLayer *__restrict__ Lp, const float *in, const FwdOut out) {
  const int n_out = Lp->out_size, n_in = Lp->in_size, has_bias = Lp->has_bias;
  const float *__restrict__ w = Lp->w;
  const float *__restrict__ b = Lp->b;
  const int g = group_for(n_out, n_in), total = n_out * g, gs = __ffs(g) - 1;
  for (int base = 0; base < total; base += TN_THREADS) {
    const int it = base + threadIdx.x, i = it >> gs, part = it & (g - 1);
    float sum = 0.0f;
    if (it < total)
      for (int c = part; c < n_in; c += g) sum += w[static_cast<size_t>(c) * n_out + i] * in[c];
    sum = group_sum(sum, g);
    if (it < total && part == 0) {
      if (has_bias) sum += b[i];
      out(i, sum);
    }
  }
}

// max_pooling_layer.h:195-222 + maxpool_op_internal.h:16-40: windows clipped at the edges,
// strict '>' from lowest(), the record is the flat CHW input index (0 when nothing wins)
TN_INLINE void maxpool_fwd(const TinyLayer *__restrict__ Lp, const float *in, const FwdOut out,
                           int32_t *__restrict__ gargmax) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S, sh = Lp->sh, sw = Lp->sw;
  const FastDiv d_plane = Lp->d_oplane, d_ow = Lp->d_ow;
  const int total = C * OH * OW;
  for (int o = threadIdx.x; o < total; o += TN_THREADS) {
    uint32_t c, r, oy, ox;
    d_plane.divmod(o, c, r);
    d_ow.divmod(r, oy, ox);
    const int x0 = ox * sw, y0 = oy * sh;
    const int dxmax = min(S, W - x0), dymax = min(R, H - y0);
    float best = -FLT_MAX;
    int idx    = 0;
    for (int wy = 0; wy < dymax; ++wy)
      for (int wx = 0; wx < dxmax; ++wx) {
        const int j   = (H * c + y0 + wy) * W + x0 + wx;
        const float v = in[j];
        if (v > best) {
          best = v;
          idx  = j;
        }
      }
    out(o, best);
    gargmax[o] = idx;
  }
}

// average_pooling_layer.h:25-55: value = sum(window) * (W[c] * scale) + b[c]
TN_INLINE void avepool_fwd(const TinyLayer *__restrict__ Lp, const float *in, const FwdOut out) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S, sh = Lp->sh, sw = Lp->sw;
  const FastDiv d_plane = Lp->d_oplane, d_ow = Lp->d_ow;
  const float scale = Lp->scale;
  const float *__restrict__ w = Lp->w;
  const float *__restrict__ b = Lp->b;
  const int total = C * OH * OW;
  for (int o = threadIdx.x; o < total; o += TN_THREADS) {
    uint32_t c, r, oy, ox;
    d_plane.divmod(o, c, r);
    d_ow.divmod(r, oy, ox);
    const int x0 = ox * sw, y0 = oy * sh;
    float value  = 0.0f;
    if (x0 + S <= W && y0 + R <= H)
      for (int wy = 0; wy < R; ++wy)
        for (int wx = 0; wx < S; ++wx) value += in[(c * H + y0 + wy) * W + x0 + wx];
    const float weight = w[c] * scale;
    value *= weight;
    value += b[c];
    out(o, value);
  }
}

TN_INLINE void act_fwd(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout) {
  const int n = Lp->out_size, act = Lp->act;
  const float p0 = Lp->p0;
  for (int o = threadIdx.x; o < n; o += TN_THREADS) {
    const float v = tn_act_fwd(act, p0, in[o]);
    out[o]  = v;
    gout[o] = v;
  }
}

// softmax_layer.h:24-34 on one row, by the first wave
TN_INLINE void softmax_fwd(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x, len = Lp->out_size;
  float m = -FLT_MAX;
  for (int j = lane; j < len; j += 64) m = fmaxf(m, in[j]);
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  float s = 0.0f;
  for (int j = lane; j < len; j += 64) {
    const float e = expf(in[j] - m);
    out[j]        = e;
    s += e;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  for (int j = lane; j < len; j += 64) {
    const float v = out[j] / s;
    out[j]  = v;
    gout[j] = v;
  }
}

// ------------------------------------------------------------------ backward
// conv2d_op_internal.h:91-127 as a gather: dX[ci][iy][ix] = sum over connected co and taps of
// W[co][ci][wy][wx] * dY[co][oy][ox] with iy = oy*sh + wy - ph, ix = ox*sw + wx - pw
TN_INLINE void conv_bwd_dx(const TinyLayer *__restrict__ Lp, const float *dy, float *dx, float *__restrict__ gdx) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, K = Lp->K, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S;
  const int sh = Lp->sh, sw = Lp->sw, ph = Lp->ph, pw = Lp->pw;
  const FastDiv d_plane = Lp->d_iplane, d_w = Lp->d_w;
  const float *__restrict__ w = Lp->w;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  const int total = C * H * W, taps = R * S, oplane = OH * OW;
  const bool unit = sh == 1 && sw == 1;
  for (int e = threadIdx.x; e < total; e += TN_THREADS) {
    uint32_t ci, r, iy, ix;
    d_plane.divmod(e, ci, r);
    d_w.divmod(r, iy, ix);
    float acc = 0.0f;
    if (unit) {
      // oy = iy + ph - wy in [0, OH): wy from max(0, iy+ph-OH+1) to min(R-1, iy+ph)
      const int ty = iy + ph, tx = ix + pw;
      const int wy0 = max(0, ty - OH + 1), wy1 = min(R - 1, ty), wx0 = max(0, tx - OW + 1), wx1 = min(S - 1, tx);
      for (int co = 0; co < K; ++co) {
        if (tbl && !tbl[ci * K + co]) continue;
        const float *wp = w + static_cast<size_t>(co * C + ci) * taps;
        const float *dp = dy + co * oplane + ty * OW + tx;
        for (int wy = wy0; wy <= wy1; ++wy)
          for (int wx = wx0; wx <= wx1; ++wx) acc += wp[wy * S + wx] * dp[-wy * OW - wx];
      }
    } else {
      for (int co = 0; co < K; ++co) {
        if (tbl && !tbl[ci * K + co]) continue;
        const float *wp = w + static_cast<size_t>(co * C + ci) * taps;
        const float *dp = dy + co * oplane;
        for (int wy = 0; wy < R; ++wy) {
          const int ty = static_cast<int>(iy) + ph - wy;
          if (ty < 0) break;
          const int oy = ty / sh;
          if (oy * sh != ty || oy >= OH) continue;
          for (int wx = 0; wx < S; ++wx) {
            const int tx = static_cast<int>(ix) + pw - wx;
            if (tx < 0) break;
            const int ox = tx / sw;
            if (ox * sw == tx && ox < OW) acc += wp[wy * S + wx] * dp[oy * OW + ox];
          }
        }
      }
    }
    dx[e] = acc;
    if (gdx) gdx[e] = acc;
  }
}

// fully_connected_op_internal.h:38-71
TN_INLINE void fc_bwd_dx(const TinyLayer *__restrict__ Lp, const float *dy, const BwdOut dx) {
  const int n_out = Lp->out_size, n_in = Lp->in_size;
  const float *__restrict__ w = Lp->w;
  for (int c = threadIdx.x; c < n_in; c += TN_THREADS) {
    const float *wr = w + static_cast<size_t>(c) * n_out;
    float acc = 0.0f;
    int i = 0;
    for (; i + 8 <= n_out; i += 8) {   // eight reads in flight
      float wv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = wr[i + j];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += dy[i + j] * wv[j];
    }
    for (; i < n_out; ++i) acc += dy[i] * wr[i];
    dx(c, acc);
  }
}
// maxpool_op_internal.h:42-57: an input takes the gradient of the LAST window that contains it
// when that window's record names it
TN_INLINE void maxpool_bwd(const TinyLayer *__restrict__ Lp, const float *dy, const int32_t *gargmax, const BwdOut dx) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S, sh = Lp->sh, sw = Lp->sw;
  const FastDiv d_plane = Lp->d_iplane, d_w = Lp->d_w;
  const int total = C * H * W;
  for (int e = threadIdx.x; e < total; e += TN_THREADS) {
    uint32_t c, r, yy, xx;
    d_plane.divmod(e, c, r);
    d_w.divmod(r, yy, xx);
    const int ox = min(OW - 1, static_cast<int>(xx) / sw), oy = min(OH - 1, static_cast<int>(yy) / sh);
    const bool covered = (static_cast<int>(xx) < ox * sw + S) && (static_cast<int>(yy) < oy * sh + R);
    const int outi = covered ? (OH * c + oy) * OW + ox : 0;
    dx(e, (gargmax[outi] == e) ? dy[outi] : 0.0f);
  }
}

// average_pooling_layer.h:58-106
TN_INLINE void avepool_bwd_dx(const TinyLayer *__restrict__ Lp, const float *dy, const BwdOut dx) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S, sh = Lp->sh, sw = Lp->sw;
  const FastDiv d_plane = Lp->d_iplane, d_w = Lp->d_w;
  const float scale = Lp->scale;
  const float *__restrict__ w = Lp->w;
  const int total = C * H * W;
  const bool two = R == 2 && S == 2 && sh == 2 && sw == 2;
  for (int e = threadIdx.x; e < total; e += TN_THREADS) {
    uint32_t c, r, iy, ix;
    d_plane.divmod(e, c, r);
    d_w.divmod(r, iy, ix);
    int ox, oy;
    if (two) {
      ox = static_cast<int>(ix) < 2 ? 0 : static_cast<int>(ix) >> 1;
      oy = static_cast<int>(iy) < 2 ? 0 : static_cast<int>(iy) >> 1;
    } else {
      ox = static_cast<int>(ix) < S ? 0 : (static_cast<int>(ix) - S + sw) / sw;
      oy = static_cast<int>(iy) < R ? 0 : (static_cast<int>(iy) - R + sh) / sh;
    }
    const float weight = w[c] * scale;
    dx(e, weight * dy[(c * OH + oy) * OW + ox]);
  }
}
TN_INLINE void act_bwd(const TinyLayer *__restrict__ Lp, const float *y, const float *dy, float *dx,
                       float *__restrict__ gdx) {
  const int n = Lp->out_size, act = Lp->act;
  const float p0 = Lp->p0;
  for (int e = threadIdx.x; e < n; e += TN_THREADS) {
    const float v = tn_act_bwd(act, p0, y[e], dy[e]);
    dx[e] = v;
    if (gdx) gdx[e] = v;
  }
}


// ---- the convolutions' fast forms -------------------------------------------------------
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
constexpr int TN_WAVES = TN_THREADS / 64;

// dX of a stride-1 convolution reads dY from a copy with a frame of zeros,
// [K][H + R - 1][W + S - 1] with dY[co][0][0] at row R-1-ph, column S-1-pw, so that every tap of
// every input pixel reads inside the copy and the loops hold no bounds test: the tap (wy, wx) of
// input pixel (iy, ix) is the copy's element (iy + R-1 - wy, ix + S-1 - wx).
TN_INLINE void stage_framed_dy(const TinyLayer *__restrict__ Lp, const float *dy, float *framed) {
  const int K = Lp->K, H = Lp->H, W = Lp->W, OH = Lp->OH, OW = Lp->OW, R = Lp->R, S = Lp->S;
  const int PW = W + S - 1, PP = (H + R - 1) * PW, oy0 = R - 1 - Lp->ph, ox0 = S - 1 - Lp->pw;
  const FastDiv d_pplane = Lp->d_pplane, d_pw = Lp->d_pw;
  for (int e = threadIdx.x; e < K * PP; e += TN_THREADS) {
    uint32_t co, r, py, px;
    d_pplane.divmod(e, co, r);
    d_pw.divmod(r, py, px);
    const int oy = static_cast<int>(py) - oy0, ox = static_cast<int>(px) - ox0;
    const bool in = static_cast<unsigned>(oy) < static_cast<unsigned>(OH) && static_cast<unsigned>(ox) < static_cast<unsigned>(OW);
    const float v = dy[in ? (co * OH + oy) * OW + ox : 0];
    framed[e] = in ? v : 0.0f;
  }
}
__host__ __device__ inline int conv_framed_floats(const TinyLayer &L) {
  return L.K * (L.H + L.R - 1) * (L.W + L.S - 1);
}

// A wave's 64 lanes are 64 pixels of one block of NB channels, so every filter value a wave needs
// is the same for all its lanes: it comes through the scalar cache straight from the weight
// tensor, W[co][ci][tap], and enters the multiply-add as a scalar operand; LDS carries one
// 4-byte read per tap, the pixel. (Filters staged in LDS and read 16 bytes per lane and tap make
// LDS the bound: it serves the four SIMDs together.) Windows of 3x3 and 5x5 are unrolled; other
// sizes take the general loops further up. Waves without an item of their own take a part
// of the summed-over channels of somebody else's; the parts meet in `scratch`.
// how many parts (1, 2 or 4) when there are `items` items and `channels` channels to sum over
// (loads through a pointer to the constant address space with a wave-uniform address are scalar
// loads; the filters are not written while these kernels run)
typedef const float __attribute__((address_space(4))) *ScalarFloats;
TN_INLINE int scalar_parts(const int items, const int channels, const int waves) {
  int parts = 1;
  while (parts < 4 && 2 * parts * items <= waves && 2 * parts <= channels) parts <<= 1;
  return parts;
}
// channels of a block: three when that divides the count and four does not
__host__ __device__ inline int scalar_block(const int channels) {
  return channels == 1 ? 1 : ((channels % 3 == 0 && (channels & 3) != 0) ? 3 : 4);
}

template <int R, int S, bool PAD, int NB, bool TBL>
TN_INLINE void conv_fwd_scalar(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout,
                               float *scratch) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, K = Lp->K, OH = Lp->OH, OW = Lp->OW;
  const int sh = Lp->sh, sw = Lp->sw, ph = Lp->ph, pw = Lp->pw, has_bias = Lp->has_bias;
  const FastDiv d_ow = Lp->d_ow;
  const float *__restrict__ w = Lp->w;
  const float *__restrict__ b = Lp->b;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  constexpr int taps = R * S;
  const int plane = OH * OW, chunks = (plane + 63) >> 6, blocks = (K + NB - 1) / NB, items = blocks * chunks;
  const int parts = scalar_parts(items, C, TN_WAVES), Ch = (C + parts - 1) / parts, total = items * parts;
  const int lane = threadIdx.x & 63;
  for (int it0 = 0; it0 < total; it0 += TN_WAVES) {
    const int item = it0 + wave_index();
    const bool active = item < total;
    const int it = active ? item : 0;
    const int cp = it / items, rem = it - cp * items, blk = rem / chunks, chunk = rem - blk * chunks, co0 = blk * NB;
    const int p = (chunk << 6) + lane;
    const bool live = p < plane;
    uint32_t oy, ox;
    d_ow.divmod(live ? p : 0, oy, ox);
    const int y0 = static_cast<int>(oy) * sh - ph, x0 = static_cast<int>(ox) * sw - pw;
    int cob[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) cob[q] = min(co0 + q, K - 1);
    float acc[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) acc[q] = 0.0f;
    const int c_lo = cp * Ch, c_hi = active ? min(C, c_lo + Ch) : c_lo;
    for (int ci = c_lo; ci < c_hi; ++ci) {
      const float *ip = in + ci * H * W + y0 * W + x0;
      ScalarFloats wq[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) wq[q] = (ScalarFloats)(w + static_cast<size_t>(cob[q] * C + ci) * taps);
      float sum[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) sum[q] = 0.0f;
#pragma unroll
      for (int wy = 0; wy < R; ++wy) {
#pragma unroll
        for (int wx = 0; wx < S; ++wx) {
          float v;
          if (PAD) {
            const bool ok = static_cast<unsigned>(y0 + wy) < static_cast<unsigned>(H) &&
                            static_cast<unsigned>(x0 + wx) < static_cast<unsigned>(W);
            v = ip[ok ? wy * W + wx : -(y0 * W + x0)];
            v = ok ? v : 0.0f;
          } else {
            v = ip[wy * W + wx];
          }
#pragma unroll
          for (int q = 0; q < NB; ++q) sum[q] = __builtin_fmaf(wq[q][wy * S + wx], v, sum[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < NB; ++q)
        if (!TBL || tbl[ci * K + cob[q]]) acc[q] += sum[q];
    }
    if (parts > 1) {
      if (active && cp > 0) {
#pragma unroll
        for (int q = 0; q < NB; ++q) scratch[(((cp - 1) * items + rem) * NB + q) * 64 + lane] = acc[q];
      }
      lds_barrier();
      if (active && cp == 0)
        for (int o = 1; o < parts; ++o) {
#pragma unroll
          for (int q = 0; q < NB; ++q) acc[q] += scratch[(((o - 1) * items + rem) * NB + q) * 64 + lane];
        }
      lds_barrier();
    }
    if (active && cp == 0 && live) {
#pragma unroll
      for (int q = 0; q < NB; ++q)
        if (co0 + q < K) {
          const float v = has_bias ? acc[q] + b[co0 + q] : acc[q];
          out[(co0 + q) * plane + p]  = v;
          gout[(co0 + q) * plane + p] = v;
        }
    }
  }
}
template <int R, int S, bool PAD>
TN_INLINE void conv_fwd_scalar_any(const TinyLayer *__restrict__ Lp, const float *in, float *out,
                                   float *__restrict__ gout, float *scratch) {
  // (a connection table makes every channel sum conditional: a version of its own, so that the
  // loops of a net without one stay free of branches)
  const bool tbl = Lp->tbl != nullptr;
  if (scalar_block(Lp->K) == 3) {
    if (tbl) conv_fwd_scalar<R, S, PAD, 3, true>(Lp, in, out, gout, scratch);
    else conv_fwd_scalar<R, S, PAD, 3, false>(Lp, in, out, gout, scratch);
  } else {
    if (tbl) conv_fwd_scalar<R, S, PAD, 4, true>(Lp, in, out, gout, scratch);
    else conv_fwd_scalar<R, S, PAD, 4, false>(Lp, in, out, gout, scratch);
  }
}

// dX from the zero-framed dY (stage_framed_dy); the waves take items * parts in turn
// (item = part * items + block * chunks + chunk)
template <int R, int S, int NB, bool TBL>
TN_INLINE void conv_bwd_dx_scalar(const TinyLayer *__restrict__ Lp, const float *framed, float *dx,
                                  float *__restrict__ gdx, float *scratch) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, K = Lp->K;
  const FastDiv d_w = Lp->d_w;
  const float *__restrict__ w = Lp->w;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  constexpr int taps = R * S;
  const int plane = H * W, chunks = (plane + 63) >> 6, blocks = (C + NB - 1) / NB, items = blocks * chunks;
  const int parts = scalar_parts(items, K, TN_WAVES), PW = W + S - 1, PP = (H + R - 1) * PW, Kh = (K + parts - 1) / parts;
  const int total = items * parts, lane = threadIdx.x & 63;
  for (int it0 = 0; it0 < total; it0 += TN_WAVES) {
    const int item = it0 + wave_index();
    const bool active = item < total;
    const int it = active ? item : 0;
    const int kp = it / items, rem = it - kp * items, blk = rem / chunks, chunk = rem - blk * chunks, ci0 = blk * NB;
    const int p = (chunk << 6) + lane;
    const bool live = p < plane;
    uint32_t iy, ix;
    d_w.divmod(live ? p : 0, iy, ix);
    const float *dp0 = framed + (static_cast<int>(iy) + R - 1) * PW + static_cast<int>(ix);
    int cib[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) cib[q] = min(ci0 + q, C - 1);
    float acc[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) acc[q] = 0.0f;
    const int c_lo = kp * Kh, c_hi = active ? min(K, c_lo + Kh) : c_lo;
    for (int co = c_lo; co < c_hi; ++co) {
      const float *dp = dp0 + co * PP;
      ScalarFloats wq[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) wq[q] = (ScalarFloats)(w + static_cast<size_t>(co * C + cib[q]) * taps);
      float sum[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) sum[q] = 0.0f;
#pragma unroll
      for (int wy = 0; wy < R; ++wy) {
        const float *row = dp - wy * PW;
#pragma unroll
        for (int wx = 0; wx < S; ++wx) {
          const float v = row[S - 1 - wx];
#pragma unroll
          for (int q = 0; q < NB; ++q) sum[q] = __builtin_fmaf(wq[q][wy * S + wx], v, sum[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < NB; ++q)
        if (!TBL || tbl[cib[q] * K + co]) acc[q] += sum[q];
    }
    if (parts > 1) {
      if (active && kp > 0) {
#pragma unroll
        for (int q = 0; q < NB; ++q) scratch[(((kp - 1) * items + rem) * NB + q) * 64 + lane] = acc[q];
      }
      lds_barrier();
      if (active && kp == 0)
        for (int o = 1; o < parts; ++o) {
#pragma unroll
          for (int q = 0; q < NB; ++q) acc[q] += scratch[(((o - 1) * items + rem) * NB + q) * 64 + lane];
        }
      lds_barrier();
    }
    if (active && kp == 0 && live) {
#pragma unroll
      for (int q = 0; q < NB; ++q)
        if (ci0 + q < C) {
          dx[(ci0 + q) * plane + p] = acc[q];
          if (gdx) gdx[(ci0 + q) * plane + p] = acc[q];
        }
    }
  }
}
template <int R, int S>
TN_INLINE void conv_bwd_dx_scalar_any(const TinyLayer *__restrict__ Lp, const float *framed, float *dx,
                                      float *__restrict__ gdx, float *scratch) {
  const int nb = scalar_block(Lp->C);
  if (Lp->tbl) {
    if (nb == 1) conv_bwd_dx_scalar<R, S, 1, true>(Lp, framed, dx, gdx, scratch);
    else if (nb == 3) conv_bwd_dx_scalar<R, S, 3, true>(Lp, framed, dx, gdx, scratch);
    else conv_bwd_dx_scalar<R, S, 4, true>(Lp, framed, dx, gdx, scratch);
  } else {
    if (nb == 1) conv_bwd_dx_scalar<R, S, 1, false>(Lp, framed, dx, gdx, scratch);
    else if (nb == 3) conv_bwd_dx_scalar<R, S, 3, false>(Lp, framed, dx, gdx, scratch);
    else conv_bwd_dx_scalar<R, S, 4, false>(Lp, framed, dx, gdx, scratch);
  }
}

// ---------------------------------------------------------------- convolutions on the matrix cores
// out[m][p] = bias[m] + sum_k A[m][k] * in[koff[k] + poff(p)]: the forward pass of a stride-1
// convolution without padding (every tap of every output pixel lies inside the input) as a
// product of the filters with the patches of the input. v_mfma_f32_16x16x4_f32: lane
// (r = lane % 16, q = lane / 16) supplies A[row r][one k] and B[the same k][column r] and holds
// D[row 4 q + i][column r], i = 0..3; which four k an instruction adds up is free, and here step
// st of `steps` takes k = q * steps + st, so that a lane's operands of four steps in a row are
// 16 consecutive bytes of a filter row and of the offset table. A wave takes 16 channels x
// T tiles of 16 pixels at once (what bounds a tile is the chain of LDS reads in front of its
// first product, not the products: T tiles share that chain). `a` holds A as [M][pitch] with
// zeros from n_k on, `koff` the input offset of every k < 4 * steps, `bias` the bias or NULL,
// all in LDS (stage_mfma_operands); steps is a multiple of four.
typedef float tn_f4 __attribute__((ext_vector_type(4)));
constexpr int MFMA_AHEAD = 4;   // filter values a thread holds for the layer whose filters wait in registers
__host__ __device__ inline int mfma_steps(const int n_k) { return ((n_k + 15) >> 4) << 2; }
// (a row pitch of 4 * odd floats: sixteen rows read 16 bytes each from different banks, two rows a bank group)
__host__ __device__ inline int mfma_pitch(const int n_k) { return (4 * mfma_steps(n_k)) | 4; }
template <int T, typename Out>
TN_INLINE void conv_mfma(const float *src, const float *a, const int *koff, const int M, const int n_k,
                         const int plane, const FastDiv d_row, const int src_pitch, const float *bias, const Out out) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int steps = mfma_steps(n_k), pitch = mfma_pitch(n_k), groups = steps >> 2;
  const int m_tiles = (M + 15) >> 4, p_tiles = (plane + 15) >> 4, p_items = (p_tiles + T - 1) / T;
  const int total = m_tiles * p_items;
  const int k_left = n_k - q * steps;   // this lane's steps from k_left on are padding
  for (int it0 = 0; it0 < total; it0 += TN_WAVES) {
    const int item = it0 + wave_index();
    if (item >= total) break;     // (no barrier inside)
    const int mt = item / p_items, pi = item - mt * p_items;
    const int arow = min(mt * 16 + r, M - 1);
    const float *sp[T];
#pragma unroll
    for (int j = 0; j < T; ++j) {
      uint32_t py, px;
      d_row.divmod(min((pi * T + j) * 16 + r, plane - 1), py, px);
      sp[j] = src + static_cast<int>(py) * src_pitch + static_cast<int>(px);
    }
    const float4 *a4 = reinterpret_cast<const float4 *>(a + arow * pitch + q * steps);
    const int4 *k4 = reinterpret_cast<const int4 *>(koff + q * steps);
    tn_f4 acc[T];
#pragma unroll
    for (int j = 0; j < T; ++j) acc[j] = tn_f4{0.0f, 0.0f, 0.0f, 0.0f};
    float4 av = a4[0];
    int4 ko   = k4[0];
    for (int g = 0; g < groups; ++g) {
      float b[T][4];
#pragma unroll
      for (int j = 0; j < T; ++j) {
        b[j][0] = sp[j][ko.x]; b[j][1] = sp[j][ko.y]; b[j][2] = sp[j][ko.z]; b[j][3] = sp[j][ko.w];
      }
      const float4 ac = av;
      const int gn = min(g + 1, groups - 1);
      av = a4[gn];
      ko = k4[gn];
      // (a zero filter value times an infinity would be a NaN)
      const int st = 4 * g;
      const bool on0 = st < k_left, on1 = st + 1 < k_left, on2 = st + 2 < k_left, on3 = st + 3 < k_left;
#pragma unroll
      for (int j = 0; j < T; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.x, on0 ? b[j][0] : 0.0f, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.y, on1 ? b[j][1] : 0.0f, acc[j], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < T; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.z, on2 ? b[j][2] : 0.0f, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.w, on3 ? b[j][3] : 0.0f, acc[j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + 4 * q + i;
      if (m >= M) continue;
      const float bv = bias ? bias[m] : 0.0f;
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const int p = (pi * T + j) * 16 + r;
        if (p < plane) out(m * plane + p, bias ? acc[j][i] + bv : acc[j][i]);
      }
    }
  }
}
// The same with a tile a wave where there are fewer tiles than waves: `splits` waves take a tile, a range of k each, and
// leave their sums in `scratch` ([split][tile][i][lane]), from where all threads take the outputs: the chain of a tile's
// products is shorter, and what follows them (an activation) has all the workgroup's lanes. LeNet-5's second convolution
// with the tanh behind it, 7 tiles: 3.9 us, in two phases of whole tiles 4.6.
TN_INLINE void conv_mfma_split(const TinyLayer *__restrict__ L, const float *src, const float *a, const int *koff,
                               const float *bias, const FwdOut out, float *scratch) {
  const int M = L->K, n_k = L->C * L->R * L->S, plane = L->OH * L->OW, src_pitch = L->W;
  const FastDiv d_plane = L->d_oplane, d_row = L->d_ow;
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int steps = mfma_steps(n_k), pitch = mfma_pitch(n_k), groups = steps >> 2;
  const int p_tiles = (plane + 15) >> 4, tiles = ((M + 15) >> 4) * p_tiles;
  int log_splits = 0;
  while ((2 << log_splits) * tiles <= TN_WAVES && (2 << log_splits) <= groups) ++log_splits;
  const int splits = 1 << log_splits, item = wave_index();
  if (item < tiles << log_splits) {
    int part = 0, mt = 0, pt = item;   // (at most sixteen items: no divisions)
    while (pt >= tiles) { pt -= tiles; ++part; }
    while (pt >= p_tiles) { pt -= p_tiles; ++mt; }
    const int share = (groups + splits - 1) >> log_splits, g0 = part * share, g1 = min(groups, g0 + share);
    const int k_left = n_k - q * steps;   // this lane's steps from k_left on are padding
    uint32_t py, px;
    d_row.divmod(min(pt * 16 + r, plane - 1), py, px);
    const float *sp  = src + static_cast<int>(py) * src_pitch + static_cast<int>(px);
    const float4 *a4 = reinterpret_cast<const float4 *>(a + min(mt * 16 + r, M - 1) * pitch + q * steps);
    const int4 *k4   = reinterpret_cast<const int4 *>(koff + q * steps);
    tn_f4 acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;   // (two chains)
    for (int g = g0; g < g1; ++g) {
      const int4 ko   = k4[g];
      const float4 ac = a4[g];
      const float bc[4] = {sp[ko.x], sp[ko.y], sp[ko.z], sp[ko.w]};
      const int st = 4 * g;   // (a zero filter value times an infinity would be a NaN)
      acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.x, st < k_left ? bc[0] : 0.0f, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.y, st + 1 < k_left ? bc[1] : 0.0f, acc1, 0, 0, 0);
      acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.z, st + 2 < k_left ? bc[2] : 0.0f, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(ac.w, st + 3 < k_left ? bc[3] : 0.0f, acc1, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) scratch[(item * 4 + i) * 64 + lane] = acc0[i] + acc1[i];
  }
  lds_barrier();
  for (int e = threadIdx.x; e < M * plane; e += TN_THREADS) {
    uint32_t m, p;
    d_plane.divmod(e, m, p);
    const int tile = (m >> 4) * p_tiles + (p >> 4);
    const float *sum = scratch + (tile * 4 + (m & 3)) * 64 + ((m >> 2) & 3) * 16 + (p & 15);
    float v = sum[0];
    for (int o = 1; o < splits; ++o) v += sum[o * tiles * 256];
    out(e, bias ? v + bias[m] : v);
  }
}
// the forward pass of a layer with operands in LDS
TN_INLINE void conv_fwd_mfma(const TinyLayer *__restrict__ L, const float *lds, float *scratch, const FwdOut out) {
  const float *in = lds + L->lds_in, *fa = lds + L->mf_fwd_w, *fb = L->has_bias ? lds + L->mf_fwd_b : nullptr;
  const int *fk = reinterpret_cast<const int *>(lds + L->mf_fwd_ko);
  const int K = L->K, n_k = L->C * L->R * L->S, plane = L->OH * L->OW;
  // (several pixel tiles a wave when there are more tiles than waves)
  if (((K + 15) >> 4) * ((plane + 15) >> 4) > TN_WAVES) conv_mfma<4>(in, fa, fk, K, n_k, plane, L->d_ow, L->W, fb, out);
  else conv_mfma_split(L, in, fa, fk, fb, out, scratch);
}
// The operand and the offset table of the input gradient described at TinyLayer::mf_dx_w, from
// the filter values the thread still holds (mfma_filters_load: value j is element
// e0 + j * TN_THREADS + thread of the weight tensor), the rows' ends zeroed.
TN_INLINE void mfma_dx_operand_store(const TinyLayer *__restrict__ L, const float (&v)[MFMA_AHEAD], float *lds) {
  const int C = L->C, K = L->K, R = L->R, S = L->S, taps = R * S, nw = K * C * taps;
  const int n_k = K * R, pitch = mfma_pitch(n_k), k4 = 4 * mfma_steps(n_k), rows = C * S;
  const int PW = L->W + S - 1, PP = (L->H + R - 1) * PW;
  const uint8_t *__restrict__ tbl = L->tbl;
  float *a = lds + L->mf_dx_w;
  int *ko  = reinterpret_cast<int *>(lds + L->mf_dx_ko);
#pragma unroll
  for (int j = 0; j < MFMA_AHEAD; ++j) {
    const int e = j * TN_THREADS + threadIdx.x;
    if (e >= nw) continue;
    uint32_t pair, t, co, ci, wy, wx;
    L->d_taps.divmod(e, pair, t);
    L->d_c.divmod(pair, co, ci);
    L->d_s.divmod(t, wy, wx);
    a[(ci * S + wx) * pitch + co * R + wy] = (tbl && !tbl[ci * K + co]) ? 0.0f : v[j];
  }
  const int pad = pitch - n_k;
  for (int row = threadIdx.x >> 5; row < rows; row += TN_THREADS / 32)   // (pad <= 20)
    if (static_cast<int>(threadIdx.x & 31) < pad) a[row * pitch + n_k + (threadIdx.x & 31)] = 0.0f;
  for (int k = threadIdx.x; k < k4; k += TN_THREADS) {
    const int co = k / R, wy = k - co * R;
    ko[k] = k < n_k ? co * PP + (R - 1 - wy) * PW : 0;
  }
}
// dX from D (TinyLayer::mf_dx_d): the filter columns' shifted sums, in column order
TN_INLINE void mfma_dx_gather(const TinyLayer *__restrict__ L, const float *d, float *dx, float *__restrict__ gdx) {
  const int C = L->C, H = L->H, W = L->W, S = L->S, PW = W + S - 1, cols = H * PW;
  const FastDiv d_iplane = L->d_iplane, d_w = L->d_w;
  for (int e = threadIdx.x; e < C * H * W; e += TN_THREADS) {
    uint32_t ci, r, iy, ix;
    d_iplane.divmod(e, ci, r);
    d_w.divmod(r, iy, ix);
    const float *row = d + (ci * S) * cols + iy * PW + ix + S - 1;
    float sum = 0.0f;
    for (int wx = 0; wx < S; ++wx) sum += row[wx * cols - wx];
    dx[e] = sum;
    if (gdx) gdx[e] = sum;
  }
}
// The operands above for a layer that has them, straight from the weight tensor. Every filter
// value is read once, in the tensor's own order ([co][(ci, tap)], which is A's); pairs of
// channels that a connection table leaves unconnected get a zero, and so do the ends of the
// rows. In two halves, so that the reads can be in flight while other layers run: the first
// asks for up to MFMA_AHEAD values a thread, the second puts them in LDS.
TN_INLINE void mfma_filters_load(const TinyLayer *__restrict__ L, const int e0, float (&v)[MFMA_AHEAD], float &bias) {
  const int nw = L->K * L->C * L->R * L->S;
#pragma unroll
  for (int j = 0; j < MFMA_AHEAD; ++j) v[j] = L->w[min(e0 + j * TN_THREADS + static_cast<int>(threadIdx.x), nw - 1)];
  // (the bias goes with the first piece: a value a thread, there are fewer channels than threads)
  bias = (e0 == 0 && L->has_bias) ? L->b[min(static_cast<int>(threadIdx.x), L->K - 1)] : 0.0f;
}
TN_INLINE void mfma_filters_store(const TinyLayer *__restrict__ L, const int e0, const float (&v)[MFMA_AHEAD],
                                  const float bias, float *lds) {
  const int K = L->K, n_k = L->C * L->R * L->S, nw = K * n_k, pitch = mfma_pitch(n_k);
  const uint8_t *__restrict__ tbl = L->tbl;
  float *fa = lds + L->mf_fwd_w;
#pragma unroll
  for (int j = 0; j < MFMA_AHEAD; ++j) {
    const int e = e0 + j * TN_THREADS + threadIdx.x;
    if (e >= nw) continue;
    uint32_t co, k;
    L->d_nk.divmod(e, co, k);
    bool on = true;
    if (tbl) on = tbl[L->d_taps.div(k) * K + co];
    fa[co * pitch + k] = on ? v[j] : 0.0f;
  }
  if (e0 == 0 && L->has_bias && static_cast<int>(threadIdx.x) < K) lds[L->mf_fwd_b + threadIdx.x] = bias;
}
// everything else: the rows' zero ends and the offset table
TN_INLINE void mfma_tables(const TinyLayer *__restrict__ L, float *lds) {
  const int K = L->K, H = L->H, W = L->W, taps = L->R * L->S;
  const int n_k = L->C * taps, pitch = mfma_pitch(n_k), k4 = 4 * mfma_steps(n_k), pad = pitch - n_k;
  float *fa = lds + L->mf_fwd_w;
  int *ko   = reinterpret_cast<int *>(lds + L->mf_fwd_ko);
  // (pad <= 20)
  for (int row = threadIdx.x >> 5; row < K; row += TN_THREADS / 32)
    if (static_cast<int>(threadIdx.x & 31) < pad) fa[row * pitch + n_k + (threadIdx.x & 31)] = 0.0f;
  for (int k = threadIdx.x; k < k4; k += TN_THREADS) {
    uint32_t ci, t, wy, wx;
    L->d_taps.divmod(min(k, n_k - 1), ci, t);
    L->d_s.divmod(t, wy, wx);
    ko[k] = k < n_k ? static_cast<int>(ci) * H * W + static_cast<int>(wy) * W + static_cast<int>(wx) : 0;
  }
}
// every layer but the one whose filters travel in registers (`ahead`, or -1): when the kernel starts
TN_INLINE void stage_mfma_operands(const TinyPlan *__restrict__ plan, float *lds, const int m, const int ahead) {
  const int n = plan->n_mfma;
  for (int q = 0; q < n; ++q) {   // (the plan lists them: walking every layer is a scalar load and a wait each)
    const int li = plan->mfma_layers[q];
    if (li == ahead || li < m) continue;
    const TinyLayer *__restrict__ L = &plan->l[li];
    mfma_tables(L, lds);
    const int nw = L->K * L->C * L->R * L->S;
    for (int e0 = 0; e0 < nw; e0 += MFMA_AHEAD * TN_THREADS) {
      float v[MFMA_AHEAD], bias;
      mfma_filters_load(L, e0, v, bias);
      mfma_filters_store(L, e0, v, bias, lds);
    }
  }
}

// A convolution whose window is the whole input (one output pixel per channel, no padding) is a
// matrix-vector product: out[co] = sum_k W[co][k] in[k], dX[k] = sum_co W[co][k] dY[co]. Lanes
// run along k, so the filter rows are read in whole cache lines, and a lane asks for all the
// filter values of a round before it uses the first: what bounds these few kilobytes is the
// latency of a read, not its size.
__host__ __device__ inline bool conv_is_matvec(const TinyLayer &L) {
  return L.OH == 1 && L.OW == 1 && L.ph == 0 && L.pw == 0 && L.R == L.H && L.S == L.W;
}
// shapes the dX from a framed dY takes (whether it runs is the plan's dx_framed, set where LDS is laid out)
inline bool conv_dx_shape_is_framed(const TinyLayer &L) {
  return !conv_is_matvec(L) && L.sh == 1 && L.sw == 1 &&
         ((L.R == 5 && L.S == 5) || (L.R == 3 && L.S == 3));
}
// the same with 16-byte reads: no connection table, n_k a multiple of four, `in` 16-byte aligned.
// A group of lanes per output channel, as many as keep the whole workgroup busy in one round;
// the lanes of a group read neighbouring 16-byte pieces of the filter row, eight in flight each.
TN_INLINE void conv_fwd_matvec4(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout) {
  const int K = Lp->K, has_bias = Lp->has_bias;
  const float *__restrict__ b = Lp->b;
  const int n_k4 = (Lp->C * Lp->R * Lp->S) >> 2;
  const float4 *__restrict__ w4 = reinterpret_cast<const float4 *>(Lp->w);
  const float4 *in4 = reinterpret_cast<const float4 *>(in);
  int g = 64;
  while (g > 1 && (K * g > TN_THREADS || 4 * g > n_k4)) g >>= 1;
  const int gs = __ffs(g) - 1, total = K * g;
  for (int base = 0; base < total; base += TN_THREADS) {
    const int it = base + threadIdx.x, part = it & (g - 1);
    const bool on = it < total;
    const int co = on ? it >> gs : 0;
    const float4 *wr = w4 + static_cast<size_t>(co) * n_k4;
    float sum = 0.0f;
    for (int k0 = 0; k0 < n_k4; k0 += 8 * g) {
      float4 a[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + g * j + part;
        a[j] = wr[k < n_k4 ? k : 0];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + g * j + part;
        if (k < n_k4) {
          const float4 xv = in4[k];
          sum += (a[j].x * xv.x + a[j].y * xv.y) + (a[j].z * xv.z + a[j].w * xv.w);
        }
      }
    }
    sum = group_sum(sum, g);
    if (on && part == 0) {
      const float v = has_bias ? sum + b[co] : sum;
      out[co]  = v;
      gout[co] = v;
    }
  }
}
// dX[k] with 16-byte reads along k (same conditions): a thread takes four neighbouring k for one
// of `parts` ranges of output channels; the parts' sums meet in `scratch` and add up in order
TN_INLINE void conv_bwd_dx_matvec4(const TinyLayer *__restrict__ Lp, const float *dy, float *dx,
                                   float *__restrict__ gdx, float *scratch) {
  const int K = Lp->K, n_k = Lp->C * Lp->R * Lp->S, n_k4 = n_k >> 2;
  const float4 *__restrict__ w4 = reinterpret_cast<const float4 *>(Lp->w);
  int parts = 1;
  while (parts < 8 && 2 * parts * n_k4 <= TN_THREADS && 2 * parts * n_k <= TINY_SCRATCH_FLOATS) parts <<= 1;
  const int Kh = (K + parts - 1) / parts;
  for (int k0 = 0; k0 < n_k4; k0 += TN_THREADS / parts) {
    const int span = min(n_k4 - k0, TN_THREADS / parts);   // pieces of this trip
    const int part = threadIdx.x / span, kk = threadIdx.x - part * span;
    const bool on = part < parts;
    const int k = k0 + kk, c_lo = part * Kh, c_hi = on ? min(K, c_lo + Kh) : c_lo;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    int co = c_lo;
    for (; co + 4 <= c_hi; co += 4) {   // four rows in flight
      float4 wv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = w4[static_cast<size_t>(co + j) * n_k4 + k];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d = dy[co + j];
        acc.x += wv[j].x * d; acc.y += wv[j].y * d; acc.z += wv[j].z * d; acc.w += wv[j].w * d;
      }
    }
    for (; co < c_hi; ++co) {
      const float4 wv = w4[static_cast<size_t>(co) * n_k4 + k];
      const float d   = dy[co];
      acc.x += wv.x * d; acc.y += wv.y * d; acc.z += wv.z * d; acc.w += wv.w * d;
    }
    if (parts > 1) {
      if (on) reinterpret_cast<float4 *>(scratch)[part * span + kk] = acc;
      lds_barrier();
      if (part == 0)
        for (int q = 1; q < parts; ++q) {
          const float4 o = reinterpret_cast<const float4 *>(scratch)[q * span + kk];
          acc.x += o.x; acc.y += o.y; acc.z += o.z; acc.w += o.w;
        }
      lds_barrier();
    }
    if (part == 0) {
      const float r[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dx[4 * k + j] = r[j];
        if (gdx) gdx[4 * k + j] = r[j];
      }
    }
  }
}
TN_INLINE void conv_fwd_matvec(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout) {
  const int C = Lp->C, K = Lp->K, taps = Lp->R * Lp->S, has_bias = Lp->has_bias;
  const FastDiv d_taps = Lp->d_taps;
  const float *__restrict__ w = Lp->w;
  const float *__restrict__ b = Lp->b;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  const int n_k = C * taps, lane = threadIdx.x & 63;
  constexpr int ROWS = 4;   // filter rows per wave and round, eight values of each per lane
  for (int co0 = wave_index(); co0 < K; co0 += ROWS * TN_WAVES) {
    float s[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) s[r] = 0.0f;
    for (int k0 = 0; k0 < n_k; k0 += 512) {
      float a[ROWS][8];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int co = co0 + r * TN_WAVES;
        const float *wr = w + static_cast<size_t>(co < K ? co : co0) * n_k;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = k0 + 64 * j + lane;
          a[r][j] = wr[k < n_k ? k : 0];
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + 64 * j + lane;
        const bool ok = k < n_k;
        const float xv = in[ok ? k : 0];
        const int ci = d_taps.div(ok ? k : 0);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          const int co = co0 + r * TN_WAVES;
          const float v = a[r][j] * xv;
          if (ok && co < K && (!tbl || tbl[ci * K + co])) s[r] += v;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int co = co0 + r * TN_WAVES;
      const float sum = group_sum(s[r], 64);
      if (lane == 0 && co < K) {
        const float v = has_bias ? sum + b[co] : sum;
        out[co]  = v;
        gout[co] = v;
      }
    }
  }
}
// dX[k]: the threads split into `parts` ranges of output channels when k leaves most of them
// idle; the parts' sums meet in `scratch` (parts * stride floats of LDS) and add up in order
TN_INLINE void conv_bwd_dx_matvec(const TinyLayer *__restrict__ Lp, const float *dy, float *dx, float *__restrict__ gdx,
                                  float *scratch) {
  const int C = Lp->C, K = Lp->K, taps = Lp->R * Lp->S;
  const FastDiv d_taps = Lp->d_taps;
  const float *__restrict__ w = Lp->w;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  const int n_k = C * taps;
  const int parts = n_k <= 256 ? 4 : (n_k <= 512 ? 2 : 1), stride = TN_THREADS / parts;
  const int part = threadIdx.x / stride, kk = threadIdx.x - part * stride;
  const int Kh = (K + parts - 1) / parts, c_lo = part * Kh, c_hi = min(K, c_lo + Kh);
  for (int k0 = 0; k0 < n_k; k0 += stride) {
    const int k = k0 + kk;
    const bool ok = k < n_k;
    const int kc = ok ? k : 0, ci = d_taps.div(kc);
    float acc = 0.0f;
    int co = c_lo;
    for (; co + 8 <= c_hi; co += 8) {   // eight rows in flight
      float wv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = w[static_cast<size_t>(co + j) * n_k + kc];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (!tbl || tbl[ci * K + co + j]) acc += wv[j] * dy[co + j];
    }
    for (; co < c_hi; ++co)
      if (!tbl || tbl[ci * K + co]) acc += w[static_cast<size_t>(co) * n_k + kc] * dy[co];
    if (parts > 1) {
      scratch[part * stride + kk] = acc;
      lds_barrier();
      if (part == 0) {
        for (int q = 1; q < parts; ++q) acc += scratch[q * stride + kk];
      }
      lds_barrier();
    }
    if (part == 0 && ok) {
      dx[k] = acc;
      if (gdx) gdx[k] = acc;
    }
  }
}

// The same product with its filters held in registers: read once, while the layers in front run, and used on the way
// forward and on the way back. A thread holds the filter values of four neighbouring k for HELD_ROWS output channels or
// fewer: `span` threads (a power of two) lie along k, and each of the TN_THREADS / span ranges of channels is theirs.
// Forward a wave adds up its channels' sums with the lanes of two channels swapped into one register (sixteen sums in 40
// instructions), and the waves' sums meet in scratch; back a thread sums its channels alone and the ranges meet.
// LeNet-5's 120 x 400 (190 KB, which a compute unit takes 1.3 us to read), 16 samples, us: forward 1.7 with the tanh
// behind it, back 1.5; asked for when they were needed, 4.6 (and 0.6 the tanh) and 3.2.
constexpr int HELD_ROWS = 16;
struct Held {
  int shift, rows;   // 1 << shift threads along k; channels a thread holds
};
// (host; a division costs the sixteen waves of the kernel half a microsecond)
inline Held held_shape(const TinyLayer &L) {
  const int n_k4 = (L.C * L.R * L.S) >> 2;
  int shift = 6;
  while ((1 << shift) < n_k4) ++shift;
  const int parts = TN_THREADS >> shift;
  return {shift, parts ? ceil_div(L.K, parts) : L.K};
}
TN_INLINE void held_load(const TinyLayer *__restrict__ L, const Held h, float4 (&w)[HELD_ROWS], float &bias) {
  const int K = L->K, n_k4 = (L->C * L->R * L->S) >> 2;
  const int c0 = (wave_index() >> (h.shift - 6)) * h.rows, span = 1 << h.shift;
  const int k = min(static_cast<int>(threadIdx.x) & (span - 1), n_k4 - 1);
  const float4 *__restrict__ w4 = reinterpret_cast<const float4 *>(L->w);
#pragma unroll
  for (int r = 0; r < HELD_ROWS; ++r) w[r] = w4[static_cast<size_t>(min(c0 + min(r, h.rows - 1), K - 1)) * n_k4 + k];
  bias = L->has_bias ? L->b[min(static_cast<int>(threadIdx.x), K - 1)] : 0.0f;
}
TN_INLINE void held_fwd(const TinyLayer *__restrict__ L, const Held h, const FastDiv d_rows, const float4 (&w)[HELD_ROWS], const float bias,
                        const float *in, const FwdOut out, float *scratch) {
  const int K = L->K, n_k4 = (L->C * L->R * L->S) >> 2, lane = threadIdx.x & 63;
  const int k = static_cast<int>(threadIdx.x) & ((1 << h.shift) - 1);
  float p[HELD_ROWS];
#pragma unroll
  for (int r = 0; r < HELD_ROWS; ++r) p[r] = 0.0f;
  if (k < n_k4) {
    const float4 xv = reinterpret_cast<const float4 *>(in)[k];
#pragma unroll
    for (int r = 0; r < HELD_ROWS; ++r) p[r] = (w[r].x * xv.x + w[r].y * xv.y) + (w[r].z * xv.z + w[r].w * xv.w);
  }
  // register j of each sixteen lanes, the g-th of the wave: the sum of row j + HELD_ROWS / 4 * g
#pragma unroll
  for (int r = 0; r < HELD_ROWS / 2; ++r) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[r]), __float_as_uint(p[r + HELD_ROWS / 2]), false, false);
    p[r] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  const int j = lane & 15;
  float mine = 0.0f;
#pragma unroll
  for (int r = 0; r < HELD_ROWS / 4; ++r) {
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(p[r]), __float_as_uint(p[r + HELD_ROWS / 4]), false, false);
    p[r] = row_sum(__uint_as_float(sw[0]) + __uint_as_float(sw[1]));
    if (j == r) mine = p[r];
  }
  if (j < HELD_ROWS / 4) scratch[wave_index() * HELD_ROWS + HELD_ROWS / 4 * (lane >> 4) + j] = mine;
  const bool has_bias = L->has_bias;
  lds_barrier();
  for (int co = threadIdx.x; co < K; co += TN_THREADS) {
    uint32_t part, r;
    d_rows.divmod(co, part, r);
    const int waves = 1 << (h.shift - 6);
    const float *q  = scratch + part * waves * HELD_ROWS + r;
    float sum = q[0];
    for (int v = 1; v < waves; ++v) sum += q[v * HELD_ROWS];
    out(co, has_bias ? sum + (co < TN_THREADS ? bias : L->b[co]) : sum);
  }
}
TN_INLINE void held_bwd(const TinyLayer *__restrict__ L, const Held h, const float4 (&w)[HELD_ROWS], const float *dy,
                        const BwdOut dx, float *scratch) {
  const int K = L->K, n_k = L->C * L->R * L->S, parts = TN_THREADS >> h.shift;
  const int c0 = (wave_index() >> (h.shift - 6)) * h.rows;
  const int rows = min(h.rows, K - c0);   // (negative in a range past the last channel)
  const float dr = dy[min(c0 + static_cast<int>(threadIdx.x & (HELD_ROWS - 1)), K - 1)];   // lane r: row r's
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int r = 0; r < HELD_ROWS; ++r) {
    const float d = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(dr), r));
    if (r < rows) {   // (the whole wave)
      acc.x += w[r].x * d; acc.y += w[r].y * d; acc.z += w[r].z * d; acc.w += w[r].w * d;
    }
  }
  reinterpret_cast<float4 *>(scratch)[threadIdx.x] = acc;
  lds_barrier();
  for (int k = threadIdx.x; k < n_k; k += TN_THREADS) {
    float sum = 0.0f;
    for (int q0 = 0; q0 < parts; q0 += 4) {   // (four reads in flight)
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = scratch[(min(q0 + j, parts - 1) << (h.shift + 2)) + k];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (q0 + j < parts) sum += v[j];
    }
    dx(k, sum);
  }
}
static_assert(4 * TN_THREADS <= TINY_SCRATCH_FLOATS, "four sums a thread");

// The loss gradient with respect to the net's output (loss_function.h:28-36, 120-150); with a
// closing softmax and cross_entropy_multiclass the gradient with respect to the softmax's
// INPUT in closed form, y * sum(t) - t, and the softmax layer's own backward pass is skipped.
// Returns the first layer to go back through.
TN_INLINE int loss_gradient(const TinyPlan *__restrict__ plan, const float *lds, const int s, const int loss, const int softmax_xent,
                            const float *__restrict__ t, float *ga) {
  const int n = plan->n;
  const TinyLayer *__restrict__ last = &plan->l[n - 1];
  const int n_out = last->out_size;
  const float *y  = lds + last->lds_out;
  const float *tr = t + static_cast<size_t>(s) * n_out;
  if (softmax_xent) {
    float st = 0.0f;  // (every thread adds up the same few targets, in order)
    for (int j = 0; j < n_out; ++j) st += tr[j];
    float *gdz = last->dx + static_cast<size_t>(s) * n_out;
    for (int j = threadIdx.x; j < n_out; j += TN_THREADS) {
      const float v = fmaf(y[j], st, -tr[j]);
      ga[j]  = v;
      gdz[j] = v;
    }
    return n - 2;
  }
  const float mse_factor = plan->mse_factor;
  float *gdl = plan->dloss + static_cast<size_t>(s) * n_out;
  for (int j = threadIdx.x; j < n_out; j += TN_THREADS) {
    float v;
    if (loss == TDH_LOSS_MSE) v = mse_factor * (y[j] - tr[j]);
    else if (loss == TDH_LOSS_CE_MULTICLASS) v = -tr[j] / y[j];
    else v = (y[j] - tr[j]) / (y[j] * (1.0f - y[j]));
    ga[j]  = v;
    gdl[j] = v;
  }
  return n - 1;
}

// From the convolution in front of TinyPlan::held to the end of the net and back to that convolution's output: the
// activation behind a layer runs in the layer's own phase, forward and back (a phase is half a microsecond of barrier and
// layer sizes before its first value), with the filters of `held` in registers throughout. Only the kinds that
// tiny_layout lets through are in these loops, so that the other layers' registers are free for the filters. Returns
// with the gradient with respect to that convolution's output in `ga`.
// LeNet-5, 16 samples: the kernel 21.8 us without this, 17.3 with it (with 512 threads and twice the filters each, 19).
TN_INLINE void held_chain(const TinyPlan *__restrict__ plan, float *lds, const int s, const int loss,
                          const int softmax_xent, const float *__restrict__ t, const int last_bwd, const float (&ahead_w)[MFMA_AHEAD],
                          const float4 (&w)[HELD_ROWS], const float bias, float *&ga, float *&gb) {
  const int n = plan->n, held = plan->held, from = plan->held_from;
  const TinyLayer *__restrict__ H = &plan->l[held];
  float *wl = lds + plan->lds_w;
  const Held shape{plan->held_shift, plan->held_rows};
  {
    const bool act = is_pointwise(plan->l[from + 1]);
    conv_fwd_mfma(&plan->l[from], lds, wl, fwd_out(plan, lds, from, s, act));
    lds_barrier();
    for (int li = from + 1 + act; li < held;) {
      const TinyLayer *__restrict__ L = &plan->l[li];
      const float *in = lds + L->lds_in;
      const bool with = is_pool(*L) && is_pointwise(L[1]);
      const FwdOut out = fwd_out(plan, lds, li, s, with);
      if (L->kind == TDH_L_MAXPOOL) maxpool_fwd(L, in, out, L->argmax + static_cast<size_t>(s) * L->out_size);
      else if (L->kind == TDH_L_AVEPOOL) avepool_fwd(L, in, out);
      else act_fwd(L, in, out.out, out.gout);
      lds_barrier();
      li += 1 + with;
    }
  }
  {
    const bool act = held + 1 < n && is_pointwise(H[1]);
    held_fwd(H, shape, plan->d_held_rows, w, bias, lds + H->lds_in, fwd_out(plan, lds, held, s, act), wl);
    lds_barrier();
    for (int li = held + 1 + act; li < n;) {
      const TinyLayer *__restrict__ L = &plan->l[li];
      const float *in = lds + L->lds_in;
      const bool with = L->kind == TDH_L_FC && li + 1 < n && is_pointwise(L[1]);
      const FwdOut out = fwd_out(plan, lds, li, s, with);
      if (L->kind == TDH_L_FC) fc_fwd(L, in, out);
      else if (L->act == TDH_ACT_SOFTMAX) softmax_fwd(L, in, out.out, out.gout);
      else act_fwd(L, in, out.out, out.gout);
      lds_barrier();
      li += 1 + with;
    }
  }
  int li = loss_gradient(plan, lds, s, loss, softmax_xent, t, ga);
  __syncthreads();   // (also: the max-pool records written to memory above are read back below)
  auto next = [&](const int done) {
    lds_barrier();
    float *sw = ga;
    ga = gb;
    gb = sw;
    li -= done;
  };
  while (li > held) {
    const TinyLayer *__restrict__ L = &plan->l[li];
    const bool with = L->kind == TDH_L_FC && is_pointwise(L[-1]);   // (`held` is a convolution, so L[-1] lies behind it)
    const BwdOut dx = bwd_out(plan, lds, gb, li, s, with);
    if (L->kind == TDH_L_FC) fc_bwd_dx(L, ga, dx);
    else act_bwd(L, lds + L->lds_out, ga, gb, dx.gdx);
    next(1 + with);
  }
  // (the scratch area takes the filters of `from` for its input gradient while the layer behind it runs: there the
  // gradient of `held`, which also meets in that area, stops short of it)
  const int ahead = plan->mf_ahead;
  const bool operand = ahead == from && ahead >= last_bwd && plan->l[from].mf_dx_w >= 0;
  {
    const bool with = held - 1 > from + operand && is_pointwise(H[-1]);
    held_bwd(H, shape, w, ga, bwd_out(plan, lds, gb, held, s, with), wl);
    next(1 + with);
  }
  while (li > from) {
    const TinyLayer *__restrict__ L = &plan->l[li];
    const bool with = is_pool(*L) && is_pointwise(L[-1]);
    if (operand && li - with == from + 1) mfma_dx_operand_store(&plan->l[from], ahead_w, lds);
    const BwdOut dx = bwd_out(plan, lds, gb, li, s, with);
    if (L->kind == TDH_L_MAXPOOL) maxpool_bwd(L, ga, L->argmax + static_cast<size_t>(s) * L->out_size, dx);
    else if (L->kind == TDH_L_AVEPOOL) avepool_bwd_dx(L, ga, dx);
    else act_bwd(L, lds + L->lds_out, ga, gb, dx.gdx);
    next(1 + with);
  }
}

// One workgroup per sample, from layer m on (0, or the plan's split). LDS: its input, every layer's output, two gradient
// buffers, the staging area. HELD: the plan holds a layer's filters in registers (held_chain; a kernel of its own, so that
// the others do without its registers. us, one kernel / two: 12x12, 3 -> 16 -> 32 channels, 3x3, two fully-connected layers, 64 samples
// 45.8 / 44.5; 28x28, 1 -> 8 -> 16, stride 2, 64 samples 159.2 / 155.6).
template <bool HELD>
__global__ void __launch_bounds__(TN_THREADS)
tiny_net_step_kernel(const TinyPlan *__restrict__ plan, const int m, const int loss, const int softmax_xent,
                     const float *__restrict__ x, const float *__restrict__ t) {
  extern __shared__ float lds[];
  const int s = blockIdx.x, n = plan->n, in_size = plan->l[m].in_size;
  float *wl = lds + plan->lds_w;   // where partial sums of split layers meet (TINY_SCRATCH_FLOATS)
  // (one layer's filters for the matrix cores are asked for here, in front of the sample's input,
  // and put in LDS while the layer in front of that layer runs: no layer waits for them)
  const int ahead = plan->mf_ahead;
  float ahead_w[MFMA_AHEAD] = {}, ahead_b = 0.0f;
  if (ahead > 0) mfma_filters_load(&plan->l[ahead], 0, ahead_w, ahead_b);
  const float *src = (m ? plan->l[m - 1].out : x) + static_cast<size_t>(s) * in_size;
  float *dst       = lds + plan->l[m].lds_in;
  const int held = HELD ? plan->held : 0, generic = HELD ? plan->held_from : n;
  float4 held_w[HELD_ROWS];
  float held_b, touch = 0.0f;
  if (HELD && generic == m) {
    // (memory answers in order: what the first phases wait for is asked for in front of the held filters, what the last
    // ones read behind them: those lines then lie in the cache)
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = src[min(j * TN_THREADS + static_cast<int>(threadIdx.x), in_size - 1)];
    held_load(&plan->l[held], Held{plan->held_shift, plan->held_rows}, held_w, held_b);
    touch = t[static_cast<size_t>(s) * plan->l[n - 1].out_size + min(static_cast<int>(threadIdx.x), plan->l[n - 1].out_size - 1)];
    const TinyLayer *__restrict__ F = &plan->l[min(held + 1 + (held + 1 < n && is_pointwise(plan->l[held + 1])), n - 1)];
    if (F->kind == TDH_L_FC) touch += F->w[min(32 * static_cast<int>(threadIdx.x), F->nw - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j * TN_THREADS + static_cast<int>(threadIdx.x) < in_size) dst[j * TN_THREADS + threadIdx.x] = v[j];
    if (in_size > 4 * TN_THREADS) fill_lds<TN_THREADS>(dst + 4 * TN_THREADS, src + 4 * TN_THREADS, in_size - 4 * TN_THREADS);
    stage_mfma_operands(plan, lds, m, ahead);
    if (m && ahead == m) {   // (there is no layer in front of it here)
      mfma_filters_store(&plan->l[m], 0, ahead_w, ahead_b, lds);
      mfma_tables(&plan->l[m], lds);
    }
    lds_barrier();
  } else {
    fill_lds<TN_THREADS>(dst, src, in_size);
    stage_mfma_operands(plan, lds, m, ahead);
    if (m && ahead == m) {
      mfma_filters_store(&plan->l[m], 0, ahead_w, ahead_b, lds);
      mfma_tables(&plan->l[m], lds);
    }
    lds_barrier();
    for (int li = m; li < generic; ++li) {
      const TinyLayer *__restrict__ L = &plan->l[li];
      if (li + 1 == ahead) {
        mfma_filters_store(&plan->l[ahead], 0, ahead_w, ahead_b, lds);
        mfma_tables(&plan->l[ahead], lds);
      }
      const int kind = L->kind, out_size = L->out_size;
      const float *in = lds + L->lds_in;
      float *out      = lds + L->lds_out;
      float *gout     = L->out + static_cast<size_t>(s) * out_size;
      const FwdOut plain = fwd_out(plan, lds, li, s, false);
      switch (kind) {
        case TDH_L_CONV:
          if (conv_is_matvec(*L)) {
            if (!L->tbl && ((L->C * L->R * L->S) & 3) == 0 && (L->lds_in & 3) == 0) conv_fwd_matvec4(L, in, out, gout);
            else conv_fwd_matvec(L, in, out, gout);
          }
          else if (L->mf_fwd_w >= 0) conv_fwd_mfma(L, lds, wl, plain);
          else if (L->R == 5 && L->S == 5 && L->ph == 0 && L->pw == 0) conv_fwd_scalar_any<5, 5, false>(L, in, out, gout, wl);
          else if (L->R == 5 && L->S == 5) conv_fwd_scalar_any<5, 5, true>(L, in, out, gout, wl);
          else if (L->R == 3 && L->S == 3 && L->ph == 0 && L->pw == 0) conv_fwd_scalar_any<3, 3, false>(L, in, out, gout, wl);
          else if (L->R == 3 && L->S == 3) conv_fwd_scalar_any<3, 3, true>(L, in, out, gout, wl);
          else conv_fwd(L, in, out, gout);
          break;
        case TDH_L_FC: fc_fwd(L, in, plain); break;
        case TDH_L_MAXPOOL: maxpool_fwd(L, in, plain, L->argmax + static_cast<size_t>(s) * out_size); break;
        case TDH_L_AVEPOOL: avepool_fwd(L, in, plain); break;
        default:
          if (L->act == TDH_ACT_SOFTMAX) softmax_fwd(L, in, out, gout);
          else act_fwd(L, in, out, gout);
          break;
      }
      lds_barrier();
    }
    if (HELD) held_load(&plan->l[held], Held{plan->held_shift, plan->held_rows}, held_w, held_b);
  }
  if (HELD) asm volatile("" ::"v"(touch));
  float *ga = lds + plan->lds_g0, *gb = lds + plan->lds_g1;
  // input gradients only: the parameter-gradient kernel reads what this leaves in memory
  const int last_bwd = m ? m + 1 : (plan->first_dx_as_job || plan->skip_first_dx) ? 1 : 0;
  int first_bwd;
  if constexpr (HELD) {
    held_chain(plan, lds, s, loss, softmax_xent, t, last_bwd, ahead_w, held_w, held_b, ga, gb);
    first_bwd = generic;
  } else {
    first_bwd = loss_gradient(plan, lds, s, loss, softmax_xent, t, ga);
    __syncthreads();   // (also: the max-pool records written to memory above are read back below)
  }
  for (int li = first_bwd; li >= last_bwd; --li) {
    const TinyLayer *__restrict__ L = &plan->l[li];
    const int kind = L->kind, in_sz = L->in_size;
    // (the layer in front of this one in memory order is the next to run: its operand goes into
    // the scratch area now, which this phase does not use when that is so; see tiny_layout)
    if (li - 1 == ahead && ahead >= last_bwd && plan->l[ahead].mf_dx_w >= 0) mfma_dx_operand_store(&plan->l[ahead], ahead_w, lds);
    float *gdx = L->dx ? L->dx + static_cast<size_t>(s) * in_sz : nullptr;
    const BwdOut plain = bwd_out(plan, lds, gb, li, s, false);
    switch (kind) {
      case TDH_L_CONV:
        if (conv_is_matvec(*L)) {
          if (!L->tbl && ((L->C * L->R * L->S) & 3) == 0) conv_bwd_dx_matvec4(L, ga, gb, gdx, wl);
          else conv_bwd_dx_matvec(L, ga, gb, gdx, wl);
        }
        else if (!L->dx_framed) conv_bwd_dx(L, ga, gb, gdx);
        else {
          float *framed = lds + plan->lds_pad;
          stage_framed_dy(L, ga, framed);
          lds_barrier();
          if (L->mf_dx_w >= 0) {
            // (the operand was written into the scratch area while the layer behind ran; D has every
            // position of H framed rows as a column, so a column's offset is its index)
            float *dd = lds + L->mf_dx_d;
            const int PW = L->W + L->S - 1, cols = L->H * PW;
            conv_mfma<2>(framed, lds + L->mf_dx_w, reinterpret_cast<const int *>(lds + L->mf_dx_ko), L->C * L->S,
                         L->K * L->R, cols, L->d_pw, PW, nullptr, [dd](const int i, const float v) { dd[i] = v; });
            lds_barrier();
            mfma_dx_gather(L, dd, gb, gdx);
          }
          else if (L->R == 5) conv_bwd_dx_scalar_any<5, 5>(L, framed, gb, gdx, wl);
          else conv_bwd_dx_scalar_any<3, 3>(L, framed, gb, gdx, wl);
        }
        break;
      case TDH_L_FC: fc_bwd_dx(L, ga, plain); break;
      case TDH_L_MAXPOOL: maxpool_bwd(L, ga, L->argmax + static_cast<size_t>(s) * L->out_size, plain); break;
      case TDH_L_AVEPOOL: avepool_bwd_dx(L, ga, plain); break;
      default: act_bwd(L, lds + L->lds_out, ga, gb, gdx); break;
    }
    lds_barrier();
    float *sw = ga;
    ga = gb;
    gb = sw;
  }
  // (the launch that updates the first layer's filters also reads them, for the input gradient)
  if (s == 0 && plan->first_dx_as_job)
    for (int i = threadIdx.x; i < plan->l[0].nw; i += TN_THREADS) plan->first_w[i] = plan->l[0].w[i];
}

// ------------------------------------------------------------- the two ends of the chain, spread out
// One workgroup per sample leaves most of the chip idle at the batches of such nets, and the first
// convolution's block and the way back to it are half of its time. Where a net begins with
//   convolution (3x3 or 5x5), pointwise activations and pools, convolution (3x3 or 5x5, stride 1)
// (TinyPlan::split is the index of the second one), everything in front of the second convolution
// keeps to one channel: a workgroup takes one channel of a sample through it, forward in a launch in
// front of the step kernel, and in a launch behind it from the second convolution's dX back to the
// gradient of the first one's output. Bound: latency, a launch and some three trips to memory each.
// LeNet-5, batch 16, us in a trace: front 5.0, step kernel 17.9, back 10.0, and the whole step 40.6 where in one launch it is 52.1 (which batches: tiny_most_split).
constexpr int TF_THREADS = 1024;   // front, at most
constexpr int TB_THREADS = 1024;   // back
static_assert(TB_THREADS / 64 == 16, "sixteen shares of a pool's sums; a wave left over from five rows of three and from three of five");

// the sums of channel co, a lane a pixel, filters as scalar operands (as conv_fwd_scalar adds them up)
template <int R, int S, bool PAD>
TN_INLINE void conv_front(const TinyLayer *__restrict__ Lp, const float *in, float *out, float *__restrict__ gout,
                          const int co) {
  const int C = Lp->C, H = Lp->H, W = Lp->W, K = Lp->K, OH = Lp->OH, OW = Lp->OW;
  const int sh = Lp->sh, sw = Lp->sw, ph = Lp->ph, pw = Lp->pw;
  const FastDiv d_ow = Lp->d_ow;
  const float *__restrict__ w = Lp->w;
  const uint8_t *__restrict__ tbl = Lp->tbl;
  constexpr int taps = R * S;
  const int plane = OH * OW;
  const float bias = Lp->has_bias ? ((ScalarFloats)Lp->b)[co] : 0.0f;
  for (int p = threadIdx.x; p < plane; p += blockDim.x) {
    uint32_t oy, ox;
    d_ow.divmod(p, oy, ox);
    const int y0 = static_cast<int>(oy) * sh - ph, x0 = static_cast<int>(ox) * sw - pw;
    float acc = 0.0f;
    for (int ci = 0; ci < C; ++ci) {
      if (tbl && !tbl[ci * K + co]) continue;
      const float *ip = in + ci * H * W + y0 * W + x0;
      const ScalarFloats wq = (ScalarFloats)(w + static_cast<size_t>(co * C + ci) * taps);
      float sum = 0.0f;
#pragma unroll
      for (int wy = 0; wy < R; ++wy)
#pragma unroll
        for (int wx = 0; wx < S; ++wx) {
          float v;
          if (PAD) {
            const bool ok = static_cast<unsigned>(y0 + wy) < static_cast<unsigned>(H) &&
                            static_cast<unsigned>(x0 + wx) < static_cast<unsigned>(W);
            v = ip[ok ? wy * W + wx : -(y0 * W + x0)];
            v = ok ? v : 0.0f;
          } else {
            v = ip[wy * W + wx];
          }
          sum = __builtin_fmaf(wq[wy * S + wx], v, sum);
        }
      acc += sum;
    }
    const float v = Lp->has_bias ? acc + bias : acc;
    out[p]  = v;
    gout[p] = v;
  }
}

__global__ void __launch_bounds__(TF_THREADS)
tiny_net_front_kernel(const TinyPlan *__restrict__ plan, const int m, const int in_size, const float *__restrict__ x) {
  extern __shared__ float lds[];
  const int s = blockIdx.x, co = blockIdx.y, nt = blockDim.x;
  for (int base = threadIdx.x; base < in_size; base += 4 * nt) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = x[static_cast<size_t>(s) * in_size + min(base + j * nt, in_size - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (base + j * nt < in_size) lds[base + j * nt] = v[j];
  }
  const TinyLayer *__restrict__ L = &plan->l[0];
  int plane  = L->OH * L->OW;
  float *cur = lds + in_size, *g0 = L->out + static_cast<size_t>(s) * L->out_size + co * plane;
  lds_barrier();
  const bool pad = L->ph != 0 || L->pw != 0;
  if (L->R == 5) pad ? conv_front<5, 5, true>(L, lds, cur, g0, co) : conv_front<5, 5, false>(L, lds, cur, g0, co);
  else pad ? conv_front<3, 3, true>(L, lds, cur, g0, co) : conv_front<3, 3, false>(L, lds, cur, g0, co);
  for (int li = 1; li < m; ++li) {
    L = &plan->l[li];
    lds_barrier();
    if (L->kind == TDH_L_ACT) {
      const int act = L->act;
      const float p0 = L->p0;
      float *gout = L->out + static_cast<size_t>(s) * L->out_size + co * plane;
      for (int i = threadIdx.x; i < plane; i += nt) {
        const float v = tn_act_fwd(act, p0, cur[i]);
        cur[i]  = v;
        gout[i] = v;
      }
      continue;
    }
    const int H = L->H, W = L->W, OH = L->OH, OW = L->OW, R = L->R, S = L->S, sh = L->sh, sw = L->sw, oplane = OH * OW;
    const bool most = L->kind == TDH_L_MAXPOOL;
    const FastDiv d_ow = L->d_ow;
    const size_t at = static_cast<size_t>(s) * L->out_size + co * oplane;
    const float weight = most ? 0.0f : L->w[co] * L->scale, bias = most ? 0.0f : L->b[co];
    float *nxt = cur + plane;
    for (int o = threadIdx.x; o < oplane; o += nt) {
      uint32_t oy, ox;
      d_ow.divmod(o, oy, ox);
      const int x0 = ox * sw, y0 = oy * sh;
      const float *win = cur + y0 * W + x0;
      float v;
      if (most) {   // maxpool_fwd
        const int dxmax = min(S, W - x0), dymax = min(R, H - y0);
        int idx = 0;
        v = -FLT_MAX;
        for (int wy = 0; wy < dymax; ++wy)
          for (int wx = 0; wx < dxmax; ++wx)
            if (win[wy * W + wx] > v) {
              v   = win[wy * W + wx];
              idx = (H * co + y0 + wy) * W + x0 + wx;
            }
        L->argmax[at + o] = idx;
      } else {      // avepool_fwd
        v = 0.0f;
        if (x0 + S <= W && y0 + R <= H)
          for (int wy = 0; wy < R; ++wy)
            for (int wx = 0; wx < S; ++wx) v += win[wy * W + wx];
        v *= weight;
        v += bias;
      }
      nxt[o]         = v;
      L->out[at + o] = v;
    }
    cur   = nxt;
    plane = oplane;
  }
}

// LDS words of 16 bytes: what a lane reads of a row starts on one (a stride of four floats from lane to lane would
// put a wave's 4-byte reads on a quarter of the banks)
__host__ __device__ inline int quad_pitch(const int columns) { return (columns + 3) & ~3; }
template <int N>
TN_INLINE void read_row(float (&v)[N], const float *row) {
  const float4 *r = reinterpret_cast<const float4 *>(row);
#pragma unroll
  for (int k = 0; k < (N + 3) / 4; ++k) {
    const float4 w = r[k];
    v[4 * k] = w.x;
    if (4 * k + 1 < N) v[4 * k + 1 < N ? 4 * k + 1 : 0] = w.y;
    if (4 * k + 2 < N) v[4 * k + 2 < N ? 4 * k + 2 : 0] = w.z;
    if (4 * k + 3 < N) v[4 * k + 3 < N ? 4 * k + 3 : 0] = w.w;
  }
}
// dX of the second convolution for channel ci, [H][W], from the zero-framed dY. A lane takes four
// neighbouring pixels of a row, whose taps share eight values of a framed row; the waves are chunks of
// 64 such units x `parts` ranges of output channels, whose sums meet in `scratch` ([part][chunk][4][64]).
// connected: bit b stands for the output channel c_lo + b of this wave's range
struct BackSplit {
  int units_w, chunks, parts, per_part;
};
__host__ __device__ inline BackSplit back_split(const int H, const int W, const int K) {
  BackSplit b;
  b.units_w  = (W + 3) >> 2;
  b.chunks   = (H * b.units_w + 63) >> 6;
  b.parts    = min(max(TB_THREADS / 64 / b.chunks, 1), K);
  b.per_part = (K + b.parts - 1) / b.parts;
  return b;
}
template <int R, int S>
TN_INLINE void conv_back_dx(const TinyLayer *__restrict__ Lp, const BackSplit b, const float *framed, float *dx,
                            float *__restrict__ gdx, float *scratch, const int ci, const int kp, const int c_lo,
                            const int c_hi, const uint64_t connected) {
  const int C = Lp->C, H = Lp->H, W = Lp->W;
  const float *__restrict__ w = Lp->w;
  constexpr int taps = R * S;
  const int PW = quad_pitch(W + S - 1), PP = (H + R - 1) * PW, lane = threadIdx.x & 63, units = H * b.units_w;
  const int step = b.parts > 1 ? b.chunks : TB_THREADS / 64;
  if (kp < b.parts)
    for (int chunk = wave_index() - kp * step; chunk < b.chunks; chunk += step) {   // (one trip where parts > 1)
      const int unit = min((chunk << 6) + lane, units - 1);
      const int iy = unit / b.units_w, ix = (unit - iy * b.units_w) << 2;
      const float *dp = framed + c_lo * PP + iy * PW + ix;
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int co = c_lo; co < c_hi; ++co, dp += PP) {
        if (!(connected >> (co - c_lo) & 1)) continue;
        const ScalarFloats wq = (ScalarFloats)(w + static_cast<size_t>(co * C + ci) * taps);
        float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int wy = 0; wy < R; ++wy) {
          float v[S + 3];
          read_row(v, dp + (R - 1 - wy) * PW);
#pragma unroll
          for (int wx = 0; wx < S; ++wx)
#pragma unroll
            for (int k = 0; k < 4; ++k) sum[k] = __builtin_fmaf(wq[wy * S + wx], v[k + S - 1 - wx], sum[k]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] += sum[k];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) scratch[((kp * b.chunks + chunk) * 4 + k) * 64 + lane] = acc[k];
    }
  lds_barrier();
  const FastDiv d_w = Lp->d_w;
  for (int p = threadIdx.x; p < H * W; p += TB_THREADS) {
    uint32_t iy, ix;
    d_w.divmod(p, iy, ix);
    const int unit = static_cast<int>(iy) * b.units_w + (static_cast<int>(ix) >> 2);
    const float *part = scratch + ((unit >> 6) * 4 + (ix & 3)) * 64 + (unit & 63);
    float v = part[0];
    for (int o = 1; o < b.parts; ++o) v += part[o * b.chunks * 256];
    dx[p]  = v;
    gdx[p] = v;
  }
}

// Four neighbouring output pixels of a unit-stride convolution and one filter row, from the four gradients d: acc[wx] += d * X.
// xr: X's row under that filter row, at the first pixel's column with the padding in front (rows of xp floats, a multiple of
// four); iy, ix0: that row and column of the image. Products that do not exist (past the row's end, or outside the
// input) are left out, not multiplied by zero: an infinity stays out of sums that it is no part of.
template <int S, bool PAD>
TN_INLINE void dw_quad(float (&acc)[S], const float *xr, const int xp, const float (&d)[4], const int iy, const int ix0,
                       const int H, const int W, const int left) {
  const bool row = !PAD || static_cast<unsigned>(iy) < static_cast<unsigned>(H);
  float v[S + 3];
  read_row(v, xr + (row ? 0 : -iy * xp));
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k < left) {
#pragma unroll
      for (int wx = 0; wx < S; ++wx) {
        const float sum = __builtin_fmaf(d[k], v[k + wx], acc[wx]);
        const bool in   = !PAD || (row && static_cast<unsigned>(ix0 + k + wx) < static_cast<unsigned>(W));
        acc[wx] = in ? sum : acc[wx];
      }
    }
}
// floats of a staged row of X for it
__host__ __device__ inline int dw_x_pitch(const TinyLayer *__restrict__ L) {
  return quad_pitch(max(L->W + L->pw, quad_pitch(L->OW) + L->S - 1));
}

// This sample's part of a first convolution's dW and db, output channel co: a lane adds up the taps of four pixels of a
// filter row at a time (16 / R waves a row), waves and lanes meet in `red` ((S + 1) floats a wave)
template <int R, int S, bool PAD>
TN_INLINE void conv_back_param(const TinyLayer *__restrict__ L, const float *x, const float *dy, const int s, const int co,
                               float *red) {
  constexpr int WAVES = TB_THREADS / 64, PER_ROW = WAVES / R, taps = R * S;
  const int C = L->C, H = L->H, W = L->W, OH = L->OH, OW = L->OW, quads = (OW + 3) >> 2, units = OH * quads;
  const int xp = dw_x_pitch(L), ph = L->ph, pw0 = L->pw;
  const FastDiv d_quads = L->d_quads;
  const int wave = wave_index(), wy = wave / PER_ROW, sub = wave - wy * PER_ROW, lane = threadIdx.x & 63;
  float *pw = L->pw_part + static_cast<size_t>(s) * L->nw + static_cast<size_t>(co) * C * taps;
  for (int ci = 0; ci < C; ++ci) {
    float acc[S], db = 0.0f;
#pragma unroll
    for (int wx = 0; wx < S; ++wx) acc[wx] = 0.0f;
    if (wy < R)
      for (int i = sub * 64 + lane; i < units; i += 64 * PER_ROW) {
        uint32_t oy, q;
        d_quads.divmod(i, oy, q);
        const int left  = OW - 4 * static_cast<int>(q), iy = static_cast<int>(oy) - ph + wy;
        const float *dr = dy + oy * OW + 4 * q;
        float d[4];
        if ((OW & 3) == 0) {
          read_row(d, dr);
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) d[k] = dr[k < left ? k : 0];
        }
        dw_quad<S, PAD>(acc, x + (ci * H + iy) * xp + 4 * q, xp, d, iy, 4 * static_cast<int>(q) - pw0, H, W, left);
#pragma unroll
        for (int k = 0; k < 4; ++k) db += k < left ? d[k] : 0.0f;
      }
#pragma unroll
    for (int wx = 0; wx < S; ++wx) acc[wx] = wave_sum_63(acc[wx]);
    db = wave_sum_63(db);
    if (lane == 63) {
#pragma unroll
      for (int wx = 0; wx < S; ++wx) red[wave * (S + 1) + wx] = acc[wx];
      red[wave * (S + 1) + S] = db;
    }
    lds_barrier();
    // thread: filter row tid / (S + 1), column tid % (S + 1); of the last column, the bias gradient, row 0 alone
    const int row = threadIdx.x / (S + 1), col = threadIdx.x - row * (S + 1);
    if (row < R) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < PER_ROW; ++k) v += red[(row * PER_ROW + k) * (S + 1) + col];
      const bool on = !L->tbl || L->tbl[ci * L->K + co];
      if (col < S) pw[ci * taps + row * S + col] = on ? v : 0.0f;
      else if (row == 0 && ci == 0 && L->nb) L->pb_part[static_cast<size_t>(s) * L->nb + co] = v;
    }
    lds_barrier();
  }
}

// (everything from memory is asked for first: the gradient, the filters' cache lines, the table, the
// outputs of the layers on the way, and the sample)
__global__ void __launch_bounds__(TB_THREADS)
tiny_net_back_kernel(const TinyPlan *__restrict__ plan, const int m, const float *__restrict__ x) {
  extern __shared__ float lds[];
  constexpr int AHEAD = 4;   // gradients a thread holds, and layers whose outputs it does
  const int s = blockIdx.x, ci = blockIdx.y, n = plan->n, tid = threadIdx.x;
  const TinyLayer *__restrict__ L = &plan->l[m];
  const int K = L->K, H = L->H, W = L->W, R = L->R, S = L->S, out_size = L->out_size, taps = R * S;
  const float *gdy = (m == n - 1 ? plan->dloss : plan->l[m + 1].dx) + static_cast<size_t>(s) * out_size;
  float dy[AHEAD];
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) dy[j] = gdy[min(tid + TB_THREADS * j, out_size - 1)];
  int plane = H * W;
  const BackSplit b = back_split(H, W, K);
  const int kp = b.parts > 1 ? wave_index() / b.chunks : 0;
  const int c_lo = min(K, kp * b.per_part), c_hi = kp < b.parts ? min(K, c_lo + b.per_part) : c_lo;
  // y[j]: this channel of the output of layer m - 1 - j
  float y[AHEAD], xv[AHEAD];
  int p_li = plane;
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) {
    y[j] = 0.0f;
    const TinyLayer *__restrict__ A = &plan->l[max(m - 1 - j, 0)];
    if (m - 1 - j < 0) continue;
    y[j] = A->out[static_cast<size_t>(s) * A->out_size + ci * p_li + min(tid, p_li - 1)];
    if (A->kind != TDH_L_ACT) p_li = A->H * A->W;
  }
  const int in_size = plan->in_size;
  x += static_cast<size_t>(s) * in_size;
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) xv[j] = x[min(tid + TB_THREADS * j, in_size - 1)];
  uint64_t connected = ~0ull;
  if (L->tbl) connected = __ballot((tid & 63) < c_hi - c_lo && L->tbl[ci * K + min(c_lo + (tid & 63), K - 1)] != 0);
  int touch = 0;
  for (int co = c_lo; co < c_hi; ++co) {
    typedef const int __attribute__((address_space(4))) *ScalarInts;
    const ScalarInts line = (ScalarInts)(L->w + static_cast<size_t>(co * L->C + ci) * taps);
    touch |= line[0] | line[taps - 1];
  }
  float *framed = lds, *scratch = lds + plan->back_scratch, *cur = lds + plan->back_planes, *sample = lds + plan->back_sample;
  float *pool_sums = sample + plan->back_sample_floats;
  float *gdx = L->dx + static_cast<size_t>(s) * L->in_size + ci * plane;
  // dY into its frame of zeros
  const int PW = quad_pitch(W + S - 1), PP = (H + R - 1) * PW, corner = (R - 1 - L->ph) * PW + S - 1 - L->pw;
  const FastDiv d_oplane = L->d_oplane, d_ow = L->d_ow;
  for (int i = tid; i < K * PP; i += TB_THREADS) framed[i] = 0.0f;
  asm volatile("" ::"s"(touch));
  lds_barrier();
  auto place = [&](int e, float v) {
    uint32_t co, r, oy, ox;
    d_oplane.divmod(e, co, r);
    d_ow.divmod(r, oy, ox);
    framed[co * PP + corner + oy * PW + ox] = v;
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j)
    if (tid + TB_THREADS * j < out_size) place(tid + TB_THREADS * j, dy[j]);
  for (int e = tid + TB_THREADS * AHEAD; e < out_size; e += TB_THREADS) place(e, gdy[e]);
  const TinyLayer *__restrict__ F = &plan->l[0];
  const FastDiv d_w0 = F->d_w;
  const int xp = dw_x_pitch(F), pw0 = F->pw;
  auto put = [&](int e, float v) {
    uint32_t row, col;
    d_w0.divmod(e, row, col);
    sample[row * xp + col + pw0] = v;
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j)
    if (tid + TB_THREADS * j < in_size) put(tid + TB_THREADS * j, xv[j]);
  for (int e = tid + TB_THREADS * AHEAD; e < in_size; e += TB_THREADS) put(e, x[e]);
  lds_barrier();
  if (R == 5) conv_back_dx<5, 5>(L, b, framed, cur, gdx, scratch, ci, kp, c_lo, c_hi, connected);
  else conv_back_dx<3, 3>(L, b, framed, cur, gdx, scratch, ci, kp, c_lo, c_hi, connected);
  for (int li = m - 1; li >= 1; --li) {
    L = &plan->l[li];
    lds_barrier();
    if (L->kind == TDH_L_ACT) {
      const int act = L->act, j = m - 1 - li;
      const float p0 = L->p0;
      const size_t at = static_cast<size_t>(s) * L->out_size + ci * plane;
      const float *out = L->out + at;
      float *g = L->dx + at;
      const float first = j == 0 ? y[0] : j == 1 ? y[1] : j == 2 ? y[2] : y[3];
      for (int i = tid; i < plane; i += TB_THREADS) {
        const float v = tn_act_bwd(act, p0, i == tid && j < AHEAD ? first : out[i], cur[i]);
        cur[i] = v;
        g[i]   = v;
      }
      continue;
    }
    const int H = L->H, W = L->W, OH = L->OH, OW = L->OW, R = L->R, S = L->S, sh = L->sh, sw = L->sw, iplane = H * W;
    const bool most = L->kind == TDH_L_MAXPOOL, two = R == 2 && S == 2 && sh == 2 && sw == 2;
    const FastDiv d_w = L->d_w;
    const int32_t *argmax = most ? L->argmax + static_cast<size_t>(s) * L->out_size + ci * plane : nullptr;
    const float weight = most ? 0.0f : L->w[ci] * L->scale;
    float *nxt = cur + quad_pitch(plane), *g = L->dx + static_cast<size_t>(s) * L->in_size + ci * iplane;
    const int j_in = m - li;
    const float *in = plan->l[li - 1].out + static_cast<size_t>(s) * L->in_size + ci * iplane;
    const float first = j_in == 1 ? y[1] : j_in == 2 ? y[2] : y[3];
    float pw = 0.0f, pb = 0.0f;   // an average pool's own gradients
    for (int o = tid; o < plane && !most; o += TB_THREADS) pb += cur[o];
    for (int e = tid; e < iplane; e += TB_THREADS) {
      uint32_t yy, xx;
      d_w.divmod(e, yy, xx);
      const int iy = yy, ix = xx;
      float v;
      if (most) {   // maxpool_bwd
        const int ox = min(OW - 1, two ? ix >> 1 : ix / sw), oy = min(OH - 1, two ? iy >> 1 : iy / sh);
        const bool covered = ix < ox * sw + S && iy < oy * sh + R;
        const int outi = covered ? oy * OW + ox : 0;
        v = covered && argmax[outi] == ci * iplane + e ? cur[outi] : 0.0f;
      } else {      // avepool_bwd_dx
        const int ox = two ? ix >> 1 : ix < S ? 0 : (ix - S + sw) / sw, oy = two ? iy >> 1 : iy < R ? 0 : (iy - R + sh) / sh;
        const float d = cur[oy * OW + ox];
        v = weight * d;
        pw = __builtin_fmaf(e == tid && j_in < AHEAD ? first : in[e], d, pw);
      }
      nxt[e] = v;
      g[e]   = v;
    }
    if (!most) {   // (a wave's share; they are added up behind the last layer)
      pw = wave_sum_63(pw);
      pb = wave_sum_63(pb);
      if ((tid & 63) == 63) {
        pool_sums[32 * li + (tid >> 6)]      = pw;
        pool_sums[32 * li + 16 + (tid >> 6)] = pb;
      }
    }
    cur   = nxt;
    plane = iplane;
  }
  lds_barrier();
  if (tid >= TB_THREADS - 64)   // (the last wave has no filter row below)
    for (int li = 1; li < m; ++li) {
      L = &plan->l[li];
      if (L->kind != TDH_L_AVEPOOL) continue;
      const float sum = group_sum(pool_sums[32 * li + (tid & 31)], 16);
      if ((tid & 63) == 0) L->pw_part[static_cast<size_t>(s) * L->nw + ci] = sum * L->scale;
      if ((tid & 63) == 16) L->pb_part[static_cast<size_t>(s) * L->nb + ci] = sum;
    }
  L = &plan->l[0];
  const bool pad = L->ph != 0 || L->pw != 0;
  if (L->R == 5) pad ? conv_back_param<5, 5, true>(L, sample, cur, s, ci, scratch) : conv_back_param<5, 5, false>(L, sample, cur, s, ci, scratch);
  else pad ? conv_back_param<3, 3, true>(L, sample, cur, s, ci, scratch) : conv_back_param<3, 3, false>(L, sample, cur, s, ci, scratch);
}

// ------------------------------------------------------------- the parameter gradients
// One launch over the whole batch: a workgroup owns some of a layer's parameters and adds up their
// gradients over all samples of its group (tiny_groups), from the layer inputs and output
// gradients that the launches in front left in memory. A batch of one group updates its parameters right
// there; the groups of a larger one leave a slice each ([group][tensor]) for the optimizer's kernel, or for
// tiny_net_merge_kernel. Behind those workgroups come the ones of the first layer's input gradient, which
// nothing waits for either. Bound: latency (kernel arguments, the layer's sizes, one trip for the operands, the sums).
// us, a slice per sample and the optimizer's launch / here: LeNet-5, batch 16 8.7 + 4.9 / 8.0 (and 2 in the back kernel), 64
// 23.6 + 6.2 / 13.8 + 4.6, 128 40.2 + 9.6 / 21.8 + 5.4, 256 70.9 + 15.8 / 38.7 + 7.7.
constexpr int TP_THREADS = 512, TP_WAVES = TP_THREADS / 64;
constexpr int TR_THREADS = 256;   // where the convolutions go sample by sample: more and smaller workgroups share the chip more evenly
enum { TP_CONV, TP_CONV_WAVES, TP_ROWS, TP_OUTER, TP_OUTER4, TP_COLUMNS, TP_POOL, TP_SLICES_W, TP_SLICES_B };   // what a range of workgroups does
constexpr int TP_RANGES = 2 * TINY_MAX_LAYERS;
struct TinyRanges {
  int first[TP_RANGES];     // first workgroup; past the last range larger than any
  int job[TP_RANGES];       // layer * 16 + TP_*
  int per_group[TP_RANGES]; // workgroups per group of samples
  int size[TP_RANGES];      // samples of a group
};
// What becomes of a finished gradient: KIND < 0: a slice; else that optimizer's update (elementwise.hip,
// opt_multi_kernel). A kernel for each: with a choice at every update in one kernel, its code was 200 KB, and
// a workgroup waited for instructions.
struct TinyUpdate {
  OptScalars p;
  float b1_t, b2_t;
  const float *powers_in;
  float *powers_out;
  int n_tensors;
};
struct TinyTarget {
  float *g, *w, *s0, *s1, *slice;
  OptScalars p;
};
struct TinyOld {
  float g, w, s0, s1;
};
template <int KIND>
TN_INLINE TinyTarget tn_target(const TinyUpdate &u, const TinyLayer *__restrict__ L, const bool bias, const int group) {
  TinyTarget t;
  if (KIND < 0) {
    t.slice = bias ? L->gb + static_cast<size_t>(group) * L->nb : L->gw + static_cast<size_t>(group) * L->nw;
    return t;
  }
  const TinyTensor &e = bias ? L->tb : L->tw;
  t.g = e.g; t.w = e.w; t.s0 = e.s0; t.s1 = e.s1;
  t.p = u.p;
  if (opt_powers(KIND) == 0) return t;
  // the reference multiplies b1_t by b1 after every update() call (optimizer.h:125-126)
  float p1 = u.powers_in ? u.powers_in[0] : u.b1_t, p2 = u.powers_in ? u.powers_in[1] : u.b2_t;
  for (int i = 0; i < e.index; ++i) {
    p1 *= u.p.b1;
    p2 *= u.p.b2;
  }
  t.p.omb1t     = 1.0f - p1;
  t.p.omb2t     = 1.0f - p2;
  t.p.adamax_lr = static_cast<double>(u.p.alpha) / (1.0 - static_cast<double>(p1));
  return t;
}
// what the update of element e needs, asked for before the gradient is computed
template <int KIND>
TN_INLINE TinyOld tn_old(const TinyTarget &t, const int e, const bool on) {
  TinyOld o = {0.0f, 0.0f, 0.0f, 0.0f};
  if (KIND < 0 || !on) return o;
  o.g = t.g[e];
  o.w = t.w[e];
  if (opt_states(KIND) >= 1) o.s0 = t.s0[e];
  if (opt_states(KIND) >= 2) o.s1 = t.s1[e];
  return o;
}
template <int KIND>
TN_INLINE void tn_finish(const TinyTarget &t, TinyOld o, const int e, const float value) {
  if constexpr (KIND < 0) {
    t.slice[e] = value;
  } else {
    opt_one<KIND>(value + o.g, o.w, o.s0, o.s1, t.p);   // (o.g: what passes without an update left there)
    t.w[e] = o.w;
    if (opt_states(KIND) >= 1) t.s0[e] = o.s0;
    if (opt_states(KIND) >= 2) t.s1[e] = o.s1;
    t.g[e] = 0.0f;
  }
}

// x_plane values of the layer's input (one of its planes, or some that follow each other) and one plane of its output
// gradient, of ns samples, into LDS, all of a trip's reads before its first store
template <int NT>
TN_INLINE void stage_planes(const TinyLayer *__restrict__ L, float *xl, const float *__restrict__ x, const int x_stride,
                            const int x_plane, const FastDiv d_x, float *dl, const float *__restrict__ d, const int d_stride,
                            const int ns) {
  const int d_plane = L->OH * L->OW, nx = ns * x_plane, total = nx + ns * d_plane;
  const FastDiv d_d = L->d_oplane;
  const bool vec = ((x_plane | x_stride | d_plane | d_stride) & 3) == 0 &&
                   ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(d)) & 15u) == 0;
  auto from = [&](int e) {
    const bool of_x  = e < nx;
    const uint32_t i = of_x ? e : e - nx;
    const uint32_t s = of_x ? d_x.div(i) : d_d.div(i);
    return of_x ? x + static_cast<size_t>(s) * (x_stride - x_plane) + i : d + static_cast<size_t>(s) * (d_stride - d_plane) + i;
  };
  if (vec) {
    constexpr int AHEAD = 4;
    for (int base = 4 * threadIdx.x; base < total; base += 4 * AHEAD * NT) {
      float4 v[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) v[j] = *reinterpret_cast<const float4 *>(from(min(base + 4 * j * NT, total - 4)));
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        const int e = base + 4 * j * NT;
        if (e < total) *reinterpret_cast<float4 *>(e < nx ? xl + e : dl + e - nx) = v[j];
      }
    }
  } else {
    constexpr int AHEAD = 12;
    for (int base = threadIdx.x; base < total; base += AHEAD * NT) {
      float v[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) v[j] = *from(min(base + j * NT, total - 1));
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        const int e = base + j * NT;
        if (e < total) *(e < nx ? xl + e : dl + e - nx) = v[j];
      }
    }
  }
}
// sum over the workgroup, in every thread of its first wave; `red`: NT / 64 floats of LDS that nobody else uses
template <int NT>
TN_INLINE float workgroup_sum(float v, float *red) {
  v = wave_sum_63(v);
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
  lds_barrier();
  v = red[0];
#pragma unroll
  for (int k = 1; k < NT / 64; ++k) v += red[k];
  return v;
}

// What the functions below need of a layer, asked for at once (left to their first uses, its scalar loads are four trips
// to memory, one behind the other)
TN_INLINE void at_hand(const TinyLayer *__restrict__ L) {
  const FastDiv a = L->d_iplane, b = L->d_oplane, d = L->d_ow, e = L->d_vquads;
  asm volatile("" ::"s"(L->C), "s"(L->H), "s"(L->W), "s"(L->K), "s"(L->OH), "s"(L->OW), "s"(L->ph), "s"(L->pw), "s"(L->nb), "s"(L->nw),
               "s"(L->dw_chunk), "s"(L->tbl), "s"(L->gw), "s"(L->gb), "s"(L->tw.g), "s"(L->tw.w), "s"(L->tw.s0), "s"(L->tw.s1),
               "s"(L->tw.index));
  asm volatile("" ::"s"(L->tb.g), "s"(L->tb.w), "s"(L->tb.s0), "s"(L->tb.s1), "s"(L->tb.index), "s"(a.mul), "s"(a.shift), "s"(b.mul),
               "s"(b.shift), "s"(d.mul), "s"(d.shift), "s"(d.d), "s"(e.mul), "s"(e.shift), "s"(e.d));
}
// dW of a channel pair (and, with the first input channel, the output channel's bias gradient), over the samples
// [s_beg, s_end), some of them in LDS at a time. A thread adds up the taps of four output pixels below each other at
// a time (neighbouring lanes read neighbouring columns, whatever the row's length); the waves' sums meet in LDS.
// WAVES: a wave a pair, up to TP_WAVES input channels of one output channel side by side (`ci` is their block). A
// workgroup's time is mostly its latency, so that many pairs of small planes are many rounds of the chip. 12x12, 3 -> 16 -> 32
// channels, 3x3 (512 pairs of 6x6 planes behind a pool), the launch, us, a workgroup a pair / a wave: 64 samples 25.6 / 11.3, 256 88 / 29; LeNet-5's
// 96 pairs of 14x14, 5x5, 33 samples 11 / 16, 256 47 / 37 (pair_split chooses).
template <int KIND, int R, int S, bool PAD, bool WAVES>
TN_INLINE void conv_param_pair(const TinyLayer *__restrict__ L, const float *__restrict__ gin, const int in_sz,
                               const float *__restrict__ gdy, const int out_sz, const int s_beg, const int s_end,
                               const int co, const int ci_or_block, const int group, const TinyUpdate &u, float *lds) {
  constexpr int taps = R * S, TEAM = WAVES ? 64 : TP_THREADS;
  at_hand(L);
  const int channels = WAVES ? min(L->C, TP_WAVES) : 1, tid = threadIdx.x & (TEAM - 1);
  // (the last block of channels begins early enough to be whole, and leaves what the one in front of it has)
  const int ci_first = WAVES ? min(ci_or_block * TP_WAVES, L->C - channels) : ci_or_block;
  const int place = WAVES ? min(wave_index(), channels - 1) : 0, ci = ci_first + place;
  const bool here = !WAVES || (wave_index() < channels && ci >= ci_or_block * TP_WAVES);
  const bool connected = !L->tbl || L->tbl[ci * L->K + co];
  const int tap = tid, e = (co * L->C + ci) * taps + tap;
  const bool mine = here && tap < taps, mine_b = here && tap == taps && ci == 0 && L->nb;
  const TinyTarget tw = tn_target<KIND>(u, L, false, group), tb = tn_target<KIND>(u, L, true, group);
  const TinyOld old_w = tn_old<KIND>(tw, e, mine), old_b = tn_old<KIND>(tb, co, mine_b);
  const int H = L->H, W = L->W, OH = L->OH, OW = L->OW, plane = OH * OW, iplane = H * W;
  const int chunk = WAVES ? L->dw_chunk_waves : L->dw_chunk, x_plane = channels * iplane;
  const int ph = L->ph, pw = L->pw, quads = (OH + 3) >> 2;
  const FastDiv d_ow = L->d_ow, d_quads = L->d_vquads, d_x = WAVES ? L->d_iplanes : L->d_iplane;
  float acc[R][S], db = 0.0f;
#pragma unroll
  for (int wy = 0; wy < R; ++wy)
#pragma unroll
    for (int wx = 0; wx < S; ++wx) acc[wy][wx] = 0.0f;
  float *xl = lds, *dl = lds + quad_pitch(chunk * x_plane);
  for (int s0 = s_beg; s0 < s_end; s0 += chunk) {
    const int ns = min(chunk, s_end - s0);
    if (s0 > s_beg) lds_barrier();
    stage_planes<TP_THREADS>(L, xl, gin + static_cast<size_t>(s0) * in_sz + ci_first * iplane, in_sz, x_plane, d_x, dl,
                 gdy + static_cast<size_t>(s0) * out_sz + co * plane, out_sz, ns);
    lds_barrier();
    const int units = here ? ns * quads * OW : 0;
    for (int i = tid; i < units; i += TEAM) {
      uint32_t line, ox, s, q;
      d_ow.divmod(i, line, ox);
      d_quads.divmod(line, s, q);
      const int oy = 4 * static_cast<int>(q), left = OH - oy, iy0 = oy - ph, ix0 = static_cast<int>(ox) - pw;
      const float *dr = dl + s * plane + oy * OW + ox, *xr = xl + s * x_plane + place * iplane + iy0 * W + ix0;
      float d[4], v[R + 3][S];
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = dr[k < left ? k * OW : 0];
      // (rows behind the last one that a live pixel needs: some row that exists)
#pragma unroll
      for (int r = 0; r < R + 3; ++r) {
        const bool row = PAD ? static_cast<unsigned>(iy0 + r) < static_cast<unsigned>(H) : r < left + R - 1;
#pragma unroll
        for (int wx = 0; wx < S; ++wx) {
          const bool in = row && (!PAD || static_cast<unsigned>(ix0 + wx) < static_cast<unsigned>(W));
          v[r][wx] = xr[in ? r * W + wx : -(iy0 * W + ix0)];
        }
      }
      // Products that do not exist (past the last row, or outside the input) are left out, not multiplied by zero: an
      // infinity stays out of sums that it is no part of.
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < left) {
#pragma unroll
          for (int wy = 0; wy < R; ++wy)
#pragma unroll
            for (int wx = 0; wx < S; ++wx) {
              const float sum = __builtin_fmaf(d[k], v[k + wy][wx], acc[wy][wx]);
              const bool in   = !PAD || (static_cast<unsigned>(iy0 + k + wy) < static_cast<unsigned>(H) &&
                                       static_cast<unsigned>(ix0 + wx) < static_cast<unsigned>(W));
              acc[wy][wx] = in ? sum : acc[wy][wx];
            }
          db += d[k];
        }
    }
  }
#pragma unroll
  for (int wy = 0; wy < R; ++wy)
#pragma unroll
    for (int wx = 0; wx < S; ++wx) acc[wy][wx] = wave_sum_63(acc[wy][wx]);
  db = wave_sum_63(db);
  if constexpr (WAVES) {
    // (lane 63 has the sums, lane t finishes tap t)
    float sum = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(db), 63));
#pragma unroll
    for (int t = 0; t < taps; ++t) {
      const float v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(acc[t / S][t % S]), 63));
      sum = tap == t ? v : sum;
    }
    if (mine) tn_finish<KIND>(tw, old_w, e, connected ? sum : 0.0f);
    if (mine_b) tn_finish<KIND>(tb, old_b, co, sum);
    return;
  }
  lds_barrier();
  if ((threadIdx.x & 63) == 63) {
    float *red = lds + wave_index() * (taps + 1);
#pragma unroll
    for (int wy = 0; wy < R; ++wy)
#pragma unroll
      for (int wx = 0; wx < S; ++wx) red[wy * S + wx] = acc[wy][wx];
    red[taps] = db;
  }
  lds_barrier();
  if (tap > taps) return;
  float sum = lds[tap];
#pragma unroll
  for (int k = 1; k < TP_WAVES; ++k) sum += lds[k * (taps + 1) + tap];
  if (mine) tn_finish<KIND>(tw, old_w, e, connected ? sum : 0.0f);
  if (mine_b) tn_finish<KIND>(tb, old_b, co, sum);
}
// dW of one sample for any window and stride: a group of lanes per weight, which take output rows in turn; a lane walks the
// pixels of its rows whose window element lies inside the input, and the group adds up with butterfly shuffles. Workgroup
// `block` has as many (weight, lane) units as threads. (A workgroup per channel pair over several samples, as above, is few and long
// for wide windows, and short of work for small planes. 28x28, 1 -> 8, 7x7, pool, 8 -> 16, 4x4, the launch, us, so / here: 16 samples
// 26.9 / 6.4, 256 53 / 33; 32x32, 1 -> 8, 4x4, pool, 16 samples 84 / 6.7; 8x8, 1 -> 24, 4x4, 24 -> 8, 2x2, 8 -> 16, 3x3, 218 samples 65 / 15.)
// A few samples may be one group, added up one after the other and updated here (tiny_groups): 12x12, 3 -> 4, 2x2, the step, us, two samples
// 20.1 where a slice each takes 23, four 24.2 and 23.8; 32x32, 1 -> 8, 4x4, two 67.4 and 65.6.
__host__ __device__ inline int conv_rows_lanes(const TinyLayer &L, const int batch) {
  int g = 32;
  const int pixels = batch <= 8 ? 8 : 32;   // or more per lane; few samples leave units to spare
  while (g > 1 && (pixels * g > L.OH * L.OW || g > L.OH)) g >>= 1;
  return g;
}
// Behind the weights' units, in waves of their own, come the biases', conv_rows_bias_lanes a channel.
__host__ __device__ inline int conv_rows_bias_lanes(const TinyLayer &L) {
  int g = 64;
  while (g > 1 && (L.nb * g > TR_THREADS || g > L.OH * L.OW)) g >>= 1;
  return g;
}
__host__ __device__ inline int conv_rows_weight_units(const TinyLayer &L, const int batch) { return (L.nw * conv_rows_lanes(L, batch) + 63) & ~63; }
template <int KIND>
TN_INLINE void conv_param_rows(const TinyLayer *__restrict__ L, const float *__restrict__ gin, const int in_sz,
                               const float *__restrict__ gdy, const int out_sz, const int s_beg, const int s_end, const int block,
                               const int group, const int batch, const TinyUpdate &u, float *lds) {
  const int H = L->H, W = L->W, K = L->K, OH = L->OH, OW = L->OW, sh = L->sh, sw = L->sw, plane = OH * OW, nw = L->nw, nb = L->nb;
  const FastDiv d_taps = L->d_taps, d_s = L->d_s, d_c = L->d_c;
  const uint8_t *__restrict__ tbl = L->tbl;
  const int g = conv_rows_lanes(*L, batch), gs = __ffs(g) - 1, end = nw << gs, biases = conv_rows_weight_units(*L, batch);
  const int base = block * TR_THREADS, it = base + static_cast<int>(threadIdx.x);
  const bool of_bias = base + 64 * wave_index() >= biases;
  const int lanes = of_bias ? conv_rows_bias_lanes(*L) : g, part = it & (lanes - 1);
  const int idx = of_bias ? (it - biases) >> (__ffs(lanes) - 1) : min(it, end - 1) >> gs;
  const bool mine = of_bias ? idx < nb : it < end;
  const TinyTarget target = tn_target<KIND>(u, L, of_bias, group);
  const TinyOld old = tn_old<KIND>(target, idx, mine && part == 0);
  // (of dY, the planes of the output channels that these units are of)
  const bool has_bias = base + TR_THREADS > biases && nb;
  const int co_lo = has_bias ? 0 : static_cast<int>(L->d_nk.div(base >> gs));
  const int co_hi = has_bias ? K - 1 : static_cast<int>(L->d_nk.div((min(base + TR_THREADS, end) - 1) >> gs));
  float *in = lds, *dy = lds + quad_pitch(in_sz);
  uint32_t pair, tap, co, ci, wy, wx;
  d_taps.divmod(of_bias ? 0 : idx, pair, tap);
  d_c.divmod(pair, co, ci);
  d_s.divmod(tap, wy, wx);
  // iy = oy*sh + wy - ph in [0, H), ix = ox*sw + wx - pw in [0, W)
  const int yoff = static_cast<int>(wy) - L->ph, xoff = static_cast<int>(wx) - L->pw;
  int oy_lo = max(0, -yoff), oy_hi = min(OH, H - yoff), ox_lo = max(0, -xoff), ox_hi = min(OW, W - xoff);
  if (sh != 1 || sw != 1) {
    oy_lo = yoff >= 0 ? 0 : (-yoff + sh - 1) / sh, oy_hi = H - 1 - yoff < 0 ? 0 : min(OH, (H - 1 - yoff) / sh + 1);
    ox_lo = xoff >= 0 ? 0 : (-xoff + sw - 1) / sw, ox_hi = W - 1 - xoff < 0 ? 0 : min(OW, (W - 1 - xoff) / sw + 1);
  }
  const bool connected = mine && (of_bias || !tbl || tbl[ci * K + co]);
  float sum = 0.0f;
  for (int s = s_beg; s < s_end; ++s) {
    if (s > s_beg) lds_barrier();
    if (base < end) fill_lds<TR_THREADS>(in, gin + static_cast<size_t>(s) * in_sz, in_sz);
    fill_lds<TR_THREADS>(dy, gdy + static_cast<size_t>(s) * out_sz + co_lo * plane, (co_hi - co_lo + 1) * plane);
    lds_barrier();
    if (!connected) continue;
    if (of_bias) {
      for (int p = part; p < plane; p += lanes) sum += dy[idx * plane + p];
      continue;
    }
    const float *ip = in + (static_cast<int>(ci) * H + yoff) * W + xoff, *dp = dy + (static_cast<int>(co) - co_lo) * plane;
    const auto rows = [&](auto step) {
      for (int oy = oy_lo + part; oy < oy_hi; oy += g) {
        const float *ir = ip + oy * sh * W, *dr = dp + oy * OW;
        int ox = ox_lo;
        for (; ox + 4 <= ox_hi; ox += 4)
          sum += ir[ox * step] * dr[ox] + ir[(ox + 1) * step] * dr[ox + 1] + ir[(ox + 2) * step] * dr[ox + 2] + ir[(ox + 3) * step] * dr[ox + 3];
        for (; ox < ox_hi; ++ox) sum += ir[ox * step] * dr[ox];
      }
    };
    if (g > 4 && (OW & 7) == 0 && ox_lo < ox_hi) {
      // The lanes of a group read rows that lie a multiple of eight words apart: each begins a pixel further, or they
      // meet on a few banks (32x32, 1 -> 8, 4x4, one sample, the launch 17.7 us without, 6 so).
      const int n = ox_hi - ox_lo, first = ox_lo + (part < n ? part : part % n);
      for (int oy = oy_lo + part; oy < oy_hi; oy += g) {
        const float *ir = ip + oy * sh * W, *dr = dp + oy * OW;
        int ox = first;
        for (int i = 0; i < n; ++i) {
          sum += ir[ox * sw] * dr[ox];
          ox = ox + 1 == ox_hi ? ox_lo : ox + 1;
        }
      }
    } else if (sw == 1) {
      rows(std::integral_constant<int, 1>());   // (words that follow each other: two a read)
    } else {
      rows(sw);
    }
  }
  sum = group_sum(sum, lanes);
  if (mine && part == 0) tn_finish<KIND>(target, old, idx, sum);
}
// A fully-connected layer, or a convolution that is one: a weight is the sum over the samples of one input times one
// output gradient. V weights a thread, neighbours along the faster index (V = 4: its rows are whole, aligned words).
template <int KIND, int V, int AHEAD, int NT>
TN_INLINE void outer_param(const TinyLayer *__restrict__ L, const float *__restrict__ gin, const int in_sz,
                           const float *__restrict__ gdy, const int out_sz, const int s_beg, const int s_end,
                           const int block, const int group, const TinyUpdate &u) {
  const bool conv = L->kind == TDH_L_CONV;   // [co][k], or [input][output]
  const float *fast = conv ? gin : gdy, *slow = conv ? gdy : gin;
  const int fast_stride = conv ? in_sz : out_sz, slow_stride = conv ? out_sz : in_sz, nw = L->nw;
  const int e = (block * NT + static_cast<int>(threadIdx.x)) * V;
  if (e >= nw) return;
  uint32_t r, c;
  if (conv) L->d_nk.divmod(e, r, c);
  else L->d_out.divmod(e, r, c);
  const TinyTarget t = tn_target<KIND>(u, L, false, group);
  TinyOld old[V];
#pragma unroll
  for (int k = 0; k < V; ++k) old[k] = tn_old<KIND>(t, e + k, true);
  float sum[V];
#pragma unroll
  for (int k = 0; k < V; ++k) sum[k] = 0.0f;
  for (int s0 = s_beg; s0 < s_end; s0 += AHEAD) {
    float f[AHEAD][V], d[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const size_t s = min(s0 + j, s_end - 1);
      const float *fp = fast + s * fast_stride + c;
      if (V == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(fp);
        f[j][0] = v.x; f[j][1 % V] = v.y; f[j][2 % V] = v.z; f[j][3 % V] = v.w;
      } else {
        f[j][0] = fp[0];
      }
      d[j] = slow[s * slow_stride + r];
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (s0 + j < s_end) {
#pragma unroll
        for (int k = 0; k < V; ++k) sum[k] = __builtin_fmaf(f[j][k], d[j], sum[k]);
      }
  }
  const uint8_t *tbl = L->tbl;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (conv && tbl && !tbl[L->d_taps.div(c + k) * L->K + r]) sum[k] = 0.0f;
    tn_finish<KIND>(t, old[k], e + k, sum[k]);
  }
}
// element e of n: the sum over the samples of src[sample][stride]
template <int KIND, int NT>
TN_INLINE void column_param(const float *__restrict__ src, const size_t stride, const int n, const int s_beg, const int s_end,
                            const int block, const TinyTarget &t) {
  const int e = block * NT + threadIdx.x;
  if (e >= n) return;
  const TinyOld old = tn_old<KIND>(t, e, true);
  constexpr int AHEAD = 16;
  float sum = 0.0f;
  for (int s0 = s_beg; s0 < s_end; s0 += AHEAD) {
    float v[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) v[j] = src[min(s0 + j, s_end - 1) * stride + e];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) sum += s0 + j < s_end ? v[j] : 0.0f;
  }
  tn_finish<KIND>(t, old, e, sum);
}
// an average pool's channel (average_pooling_layer.h:58-106): dW = scale * sum of (window sum * dY), db = sum of dY
template <int KIND, int NT>
TN_INLINE void pool_param(const TinyLayer *__restrict__ L, const float *__restrict__ gin, const int in_sz,
                          const float *__restrict__ gdy, const int out_sz, const int s_beg, const int s_end, const int c,
                          const int group, const TinyUpdate &u, float *lds) {
  const int H = L->H, W = L->W, OW = L->OW, plane = L->OH * OW, iplane = H * W, R = L->R, S = L->S, chunk = L->dw_chunk;
  const FastDiv d_oplane = L->d_oplane, d_ow = L->d_ow;
  float *xl = lds, *dl = lds + quad_pitch(chunk * iplane);
  float dw = 0.0f, db = 0.0f;
  for (int s0 = s_beg; s0 < s_end; s0 += chunk) {
    const int ns = min(chunk, s_end - s0);
    lds_barrier();
    stage_planes<NT>(L, xl, gin + static_cast<size_t>(s0) * in_sz + c * iplane, in_sz, iplane, L->d_iplane, dl,
                 gdy + static_cast<size_t>(s0) * out_sz + c * plane, out_sz, ns);
    lds_barrier();
    for (int i = threadIdx.x; i < ns * plane; i += NT) {
      uint32_t s, r, oy, ox;
      d_oplane.divmod(i, s, r);
      d_ow.divmod(r, oy, ox);
      const int x0 = ox * L->sw, y0 = oy * L->sh;
      const float d = dl[i], *win = xl + s * iplane + y0 * W + x0;
      db += d;
      if (x0 + S <= W && y0 + R <= H)
        for (int wy = 0; wy < R; ++wy)
          for (int wx = 0; wx < S; ++wx) dw = __builtin_fmaf(win[wy * W + wx], d, dw);
    }
  }
  lds_barrier();
  dw = workgroup_sum<NT>(dw, lds);
  db = workgroup_sum<NT>(db, lds + NT / 64);
  if (threadIdx.x == 0) {
    const TinyTarget tw = tn_target<KIND>(u, L, false, group), tb = tn_target<KIND>(u, L, true, group);
    tn_finish<KIND>(tw, tn_old<KIND>(tw, c, true), c, dw * L->scale);
    tn_finish<KIND>(tb, tn_old<KIND>(tb, c, true), c, db);
  }
}

// The first layer's dX of one sample and input channel, a band of `rows` rows: dY's rows under it go into their frame
// of zeros, a lane takes four pixels (conv_back_dx), the waves share the output channels.
struct DxBand {
  int rows, bands, floats;   // floats of LDS
};
__host__ __device__ inline DxBand dx_band(const TinyLayer &L) {
  const int units_w = (L.W + 3) >> 2;
  DxBand b;
  b.rows   = units_w >= 64 ? 1 : min(64 / units_w, L.H);
  b.bands  = (L.H + b.rows - 1) / b.rows;
  b.floats = L.K * (b.rows + L.R - 1) * quad_pitch(L.W + L.S - 1) + 4 + TP_THREADS * 4;
  return b;
}
template <int R, int S, int NT>
TN_INLINE void conv_dx_band(const TinyLayer *__restrict__ L, const float *__restrict__ w, const float *__restrict__ gdy,
                            float *__restrict__ gdx, const int ci, const int band, float *lds) {
  const int C = L->C, H = L->H, W = L->W, K = L->K, OH = L->OH, OW = L->OW, PW = quad_pitch(W + S - 1), units_w = (W + 3) >> 2;
  const int full = units_w >= 64 ? 1 : min(64 / units_w, H), y0 = band * full, rows = min(full, H - y0);
  const int fr = rows + R - 1, PP = fr * PW, cells = K * PP, oy0 = y0 - (R - 1 - L->ph), ox0 = -(S - 1 - L->pw);
  const FastDiv d_pw = L->d_pw4;
  const uint8_t *__restrict__ tbl = L->tbl;
  constexpr int AHEAD = 8;
  for (int base = threadIdx.x; base < cells; base += AHEAD * NT) {
    float v[AHEAD];
    bool in[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      uint32_t line, px;
      d_pw.divmod(min(base + j * NT, cells - 1), line, px);
      const int co = static_cast<int>(line) / fr, oy = oy0 + static_cast<int>(line) - co * fr, ox = ox0 + static_cast<int>(px);
      in[j] = static_cast<unsigned>(oy) < static_cast<unsigned>(OH) && static_cast<unsigned>(ox) < static_cast<unsigned>(OW);
      v[j]  = gdy[in[j] ? (co * OH + oy) * OW + ox : 0];
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (base + j * NT < cells) lds[base + j * NT] = in[j] ? v[j] : 0.0f;
  }
  lds_barrier();
  constexpr int taps = R * S;
  const int lane = threadIdx.x & 63, wave = wave_index(), units = rows * units_w;
  float *scratch = lds + cells + 4;            // (a row's last read may pass its end)
  for (int u0 = 0; u0 < units; u0 += 64) {     // (one trip unless a row has more units than a wave lanes)
    const int unit = min(u0 + lane, units - 1), iy = unit / units_w, ix = (unit - iy * units_w) << 2;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int co = wave; co < K; co += NT / 64) {
      if (tbl && !tbl[ci * K + co]) continue;
      const ScalarFloats wq = (ScalarFloats)(w + static_cast<size_t>(co * C + ci) * taps);
      const float *dp = lds + co * PP + iy * PW + ix;
      float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int wy = 0; wy < R; ++wy) {
        float v[S + 3];
        read_row(v, dp + (R - 1 - wy) * PW);
#pragma unroll
        for (int wx = 0; wx < S; ++wx)
#pragma unroll
          for (int k = 0; k < 4; ++k) sum[k] = __builtin_fmaf(wq[wy * S + wx], v[k + S - 1 - wx], sum[k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] += sum[k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) scratch[(wave * 64 + lane) * 4 + k] = acc[k];
    lds_barrier();
    // thread: pixel tid%4 of unit u0 + tid/4, of the first 64
    const int mine = u0 + (threadIdx.x >> 2), my = mine / units_w, mx = ((mine - my * units_w) << 2) + (threadIdx.x & 3);
    if (threadIdx.x < 256 && mine < units && mx < W) {
      float v = scratch[threadIdx.x];
#pragma unroll
      for (int k = 1; k < NT / 64; ++k) v += scratch[256 * k + threadIdx.x];
      gdx[(y0 + my) * W + mx] = v;
    }
    lds_barrier();
  }
}

// ROADS: what there is code for. TP_HAS_PAIRS: 3x3 or 5x5 windows of stride 1, and the first layer's dX; TP_HAS_WAVES: a wave a pair;
// TP_HAS_ROWS: sample by sample, any window; TP_HAS_DX: the first layer's dX beside it. (All of it in one kernel, LeNet-5's step at 16
// samples takes 41.1 us instead of 40.7: more scalars than there are registers for.)
constexpr int TP_HAS_PAIRS = 1, TP_HAS_WAVES = 2, TP_HAS_ROWS = 4, TP_HAS_DX = 8;
__host__ __device__ constexpr int param_threads(const int roads) { return roads & TP_HAS_ROWS ? TR_THREADS : TP_THREADS; }
template <int KIND, int ROADS>
__global__ void __launch_bounds__(param_threads(ROADS), ROADS & TP_HAS_PAIRS ? 4 : 7)
tiny_net_param_kernel(const TinyPlan *__restrict__ plan, const float *__restrict__ x, const TinyRanges ranges,
                      const TinyUpdate u, const int batch, const int param_blocks) {
  extern __shared__ float lds[];
  constexpr int NT = param_threads(ROADS);
  constexpr int AHEAD = ROADS & TP_HAS_PAIRS ? 16 : 4;   // samples that an outer product has in flight
  if (KIND >= 0 && opt_powers(KIND) > 0 && u.powers_in && blockIdx.x == 0 && threadIdx.x == 0) {   // (as opt_multi_kernel)
    float q1 = u.powers_in[0], q2 = u.powers_in[1];
    for (int i = 0; i < u.n_tensors; ++i) {
      q1 *= u.p.b1;
      if (opt_powers(KIND) == 2) q2 *= u.p.b2;
    }
    u.powers_out[0] = q1;
    u.powers_out[1] = q2;
  }
  const int n = plan->n;
  int id = blockIdx.x;
  if ((ROADS & (TP_HAS_PAIRS | TP_HAS_DX)) && id >= param_blocks) {   // workgroups (band, input channel, sample), samples fastest
    id -= param_blocks;
    const TinyLayer *__restrict__ L = &plan->l[0];
    const int rest = id / batch, s = id - rest * batch, ci = rest % L->C, band = rest / L->C;
    const float *gdy = plan->l[1].dx + static_cast<size_t>(s) * L->out_size;
    float *gdx = L->dx + static_cast<size_t>(s) * L->in_size + ci * L->H * L->W;
    if (L->R == 5) conv_dx_band<5, 5, NT>(L, plan->first_w, gdy, gdx, ci, band, lds);
    else conv_dx_band<3, 3, NT>(L, plan->first_w, gdy, gdx, ci, band, lds);
    return;
  }
  int first = 0, job = ranges.job[0], per_group = ranges.per_group[0], size = ranges.size[0];
#pragma unroll
  for (int k = 1; k < TP_RANGES; ++k) {   // (indices known to the compiler: the argument stays in scalar registers)
    const bool on = ranges.first[k] <= id;
    first     = on ? ranges.first[k] : first;
    job       = on ? ranges.job[k] : job;
    per_group = on ? ranges.per_group[k] : per_group;
    size      = on ? ranges.size[k] : size;
  }
  const int li = job >> 4, what = job & 15, part = id - first;
  // (a sample after the other in dispatch order, where a group is one: the workgroups of a sample then meet on few of the chip's second-level caches)
  const int groups = (batch + size - 1) / size, group = ROADS & TP_HAS_ROWS ? part % groups : part / per_group;
  const int block = ROADS & TP_HAS_ROWS ? part / groups : part - group * per_group;
  const TinyLayer *__restrict__ L = &plan->l[li];
  const int in_sz = L->in_size, out_sz = L->out_size;
  const float *gin = li == 0 ? x : plan->l[li - 1].out;
  const float *gdy = li == n - 1 ? plan->dloss : plan->l[li + 1].dx;
  const int s_beg = group * size, s_end = min(batch, s_beg + size);
  switch (what) {
    case TP_CONV:
    case TP_CONV_WAVES:
      if constexpr (ROADS & TP_HAS_PAIRS) {
        const bool waves = (ROADS & TP_HAS_WAVES) && what == TP_CONV_WAVES, pad = L->ph != 0 || L->pw != 0;
        uint32_t co, ci;
        (waves ? L->d_cblocks : L->d_c).divmod(block, co, ci);
        const auto run = [&](auto window, auto padded) {
          constexpr int R = decltype(window)::value;
          constexpr bool PAD = decltype(padded)::value, MAY_WAVES = (ROADS & TP_HAS_WAVES) != 0;
          if (waves) conv_param_pair<KIND, R, R, PAD, MAY_WAVES>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, co, ci, group, u, lds);
          else conv_param_pair<KIND, R, R, PAD, false>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, co, ci, group, u, lds);
        };
        const std::integral_constant<int, 5> five;
        const std::integral_constant<int, 3> three;
        if (L->R == 5) pad ? run(five, std::true_type()) : run(five, std::false_type());
        else pad ? run(three, std::true_type()) : run(three, std::false_type());
      }
      break;
    case TP_ROWS:
      if constexpr (ROADS & TP_HAS_ROWS) conv_param_rows<KIND>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, block, group, batch, u, lds);
      break;
    case TP_OUTER: outer_param<KIND, 1, AHEAD, NT>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, block, group, u); break;
    case TP_OUTER4: outer_param<KIND, 4, AHEAD, NT>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, block, group, u); break;
    case TP_COLUMNS: column_param<KIND, NT>(gdy, out_sz, L->nb, s_beg, s_end, block, tn_target<KIND>(u, L, true, group)); break;
    case TP_POOL: pool_param<KIND, NT>(L, gin, in_sz, gdy, out_sz, s_beg, s_end, block, group, u, lds); break;
    case TP_SLICES_W: column_param<KIND, NT>(L->pw_part, L->nw, L->nw, s_beg, s_end, block, tn_target<KIND>(u, L, false, group)); break;
    default: column_param<KIND, NT>(L->pb_part, L->nb, L->nb, s_beg, s_end, block, tn_target<KIND>(u, L, true, group)); break;
  }
}

// g[i] += slice[0][i] + slice[1][i] + ... in the order of the groups (edge::merge_grads, node.h:89-103)
__global__ void __launch_bounds__(256)
tiny_net_merge_kernel(const TinyMerge m) {
  int j = 0;
  while (j + 1 < m.n && m.first_block[j + 1] <= static_cast<int>(blockIdx.x)) ++j;
  const int i = (static_cast<int>(blockIdx.x) - m.first_block[j]) * 256 + threadIdx.x;
  if (i >= m.len[j]) return;
  const float *p = m.slices[j] + i;
  float sum = p[0];
  for (int s = 1; s < m.count[j]; ++s) sum += p[static_cast<size_t>(s) * m.len[j]];
  m.g[j][i] += sum;
}

}  // namespace

// of an optimizer kind, or -1 for slices, which may be of every road
template <int KIND>
static decltype(&tiny_net_param_kernel<-1, 0>) param_kernel_of(const int roads) {
  if (roads & TP_HAS_ROWS) return roads & TP_HAS_DX ? tiny_net_param_kernel<KIND, TP_HAS_ROWS | TP_HAS_DX> : tiny_net_param_kernel<KIND, TP_HAS_ROWS>;
  if constexpr (KIND < 0)
    if (roads & TP_HAS_WAVES) return tiny_net_param_kernel<KIND, TP_HAS_PAIRS | TP_HAS_WAVES>;
  return tiny_net_param_kernel<KIND, TP_HAS_PAIRS>;
}
static decltype(&tiny_net_param_kernel<-1, 0>) param_kernel(const int kind, const int roads) {
  switch (kind) {
    case -1: return param_kernel_of<-1>(roads);
    case TDH_OPT_SGD: return param_kernel_of<TDH_OPT_SGD>(roads);
    case TDH_OPT_MOMENTUM: return param_kernel_of<TDH_OPT_MOMENTUM>(roads);
    case TDH_OPT_NESTEROV: return param_kernel_of<TDH_OPT_NESTEROV>(roads);
    case TDH_OPT_ADAM: return param_kernel_of<TDH_OPT_ADAM>(roads);
    case TDH_OPT_ADAGRAD: return param_kernel_of<TDH_OPT_ADAGRAD>(roads);
    case TDH_OPT_RMSPROP: return param_kernel_of<TDH_OPT_RMSPROP>(roads);
    case TDH_OPT_ADAMAX: return param_kernel_of<TDH_OPT_ADAMAX>(roads);
    default: return nullptr;
  }
}

int tiny_prepare() {
  static bool attr_set = false;
  if (!attr_set) {
    const auto of = [](auto k) { return reinterpret_cast<const void *>(k); };
    std::vector<const void *> kernels = {of(&tiny_net_step_kernel<false>), of(&tiny_net_step_kernel<true>), of(&tiny_net_front_kernel),
                                         of(&tiny_net_back_kernel)};
    for (int kind = -1; kind <= TDH_OPT_NESTEROV; ++kind)
      for (int roads : {TP_HAS_PAIRS, TP_HAS_ROWS, TP_HAS_ROWS | TP_HAS_DX}) kernels.push_back(of(param_kernel(kind, roads)));
    kernels.push_back(of(param_kernel(-1, TP_HAS_WAVES)));
    for (const void *k : kernels)
      TDH_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(TINY_LDS_MAX_BYTES)));
    attr_set = true;
  }
  return TDH_OK;
}

// Whether the net begins with what the front and back kernels take, and their LDS
static void plan_split(TinyPlan &P) {
  P.split = 0;
  const TinyLayer &F = P.l[0];
  if (F.kind != TDH_L_CONV || !((F.R == 5 && F.S == 5) || (F.R == 3 && F.S == 3)) || conv_is_matvec(F) ||
      F.sh != 1 || F.sw != 1 || !(P.first_dx_as_job || P.skip_first_dx))
    return;
  int m = 1;
  size_t front = F.OH * F.OW, back = 0;
  for (; m < P.n; ++m) {
    const TinyLayer &L = P.l[m];
    if (L.kind == TDH_L_ACT && L.act != TDH_ACT_SOFTMAX) continue;
    if (L.kind != TDH_L_MAXPOOL && L.kind != TDH_L_AVEPOOL) break;
    front += L.OH * L.OW;
    back += quad_pitch(L.H * L.W);
  }
  if (m == P.n || !P.l[m].dx_framed || P.l[m].K > 64) return;   // (64: conv_back_dx)
  const TinyLayer &L = P.l[m];
  P.back_scratch = L.K * (L.H + L.R - 1) * quad_pitch(L.W + L.S - 1) + 4;   // (a row's last read may pass its end)
  const BackSplit b = back_split(L.H, L.W, L.K);
  P.back_planes  = P.back_scratch + b.parts * b.chunks * 256;
  P.back_sample  = P.back_planes + static_cast<int>(back) + quad_pitch(L.H * L.W);
  P.back_sample_floats = F.C * F.H * dw_x_pitch(&F);
  P.back_floats  = P.back_sample + P.back_sample_floats + 32 * m;
  P.front_floats = static_cast<int>(front);
  if (std::max(static_cast<size_t>(P.back_floats), P.in_size + front) * sizeof(float) > TINY_LDS_MAX_BYTES) return;
  P.split = m;
}

// A window without an unrolled form in conv_param_pair
static bool conv_any_window(const TinyLayer &L) {
  return L.kind == TDH_L_CONV && !conv_is_matvec(L) &&
         !(L.sh == 1 && L.sw == 1 && ((L.R == 5 && L.S == 5) || (L.R == 3 && L.S == 3)));
}
// Convolutions whose weight gradients are added up sample by sample (conv_param_rows): all of a net that has any such window
static bool conv_by_rows(const TinyPlan &plan, const TinyLayer &L) {
  return plan.by_rows && L.kind == TDH_L_CONV && !conv_is_matvec(L);
}
int tiny_layout(TinyPlan &P) {
  size_t framed = 0, lds = 26 * TP_WAVES;   // (conv_param_pair's sums)
  for (int i = 0; i < P.n; ++i) {
    TinyLayer &L = P.l[i];
    L.dx_framed = L.kind == TDH_L_CONV && conv_dx_shape_is_framed(L) && L.dx != nullptr;
    if (L.dx_framed) {
      L.d_pplane = FastDiv(static_cast<uint32_t>((L.H + L.R - 1) * (L.W + L.S - 1)));
      L.d_pw     = FastDiv(static_cast<uint32_t>(L.W + L.S - 1));
      L.d_pw4    = FastDiv(static_cast<uint32_t>(quad_pitch(L.W + L.S - 1)));
    }
  }
  P.first_dx_as_job = P.l[0].dx_framed && P.n > 1 && !P.skip_first_dx;
  P.by_rows = std::any_of(P.l, P.l + P.n, conv_any_window);
  int room = P.by_rows ? 4096 : 12288;
  for (int i = 0; i < P.n; ++i)
    if (conv_by_rows(P, P.l[i])) room = std::min(std::max(room, quad_pitch(P.l[i].in_size) + P.l[i].out_size), 12288);
  for (int i = 0; i < P.n; ++i) {
    TinyLayer &L = P.l[i];
    L.dw_chunk = 512;   // (what needs no LDS)
    if (i == 0 && P.first_dx_as_job) lds = std::max(lds, static_cast<size_t>(dx_band(L).floats));
    else if (L.dx_framed) framed = std::max(framed, static_cast<size_t>(conv_framed_floats(L)));
    if (!L.nw || L.kind == TDH_L_FC || conv_is_matvec(L)) continue;
    if (conv_by_rows(P, L)) {
      lds = std::max(lds, static_cast<size_t>(quad_pitch(L.in_size)) + L.out_size);
      continue;
    }
    // planes of the input and the output gradient: as many samples at a time as fit 48 KB, or beside single samples' sums
    // no more than those take, or 16 KB (a workgroup a sample and lot of weights: three or four of them a compute unit)
    const int planes = L.H * L.W + L.OH * L.OW;
    L.dw_chunk = std::min(std::max(room / planes, 1), 32);
    lds = std::max(lds, static_cast<size_t>(L.dw_chunk) * planes + 4);
    if (L.kind != TDH_L_CONV || L.C == 1) continue;
    const int channels = std::min(L.C, TP_WAVES), more = channels * L.H * L.W + L.OH * L.OW;
    L.dw_chunk_waves = more > 12288 ? 0 : std::min(12288 / more, 32);
    L.d_iplanes = FastDiv(static_cast<uint32_t>(channels * L.H * L.W));
    L.d_cblocks = FastDiv(static_cast<uint32_t>(ceil_div(L.C, TP_WAVES)));
    lds = std::max(lds, static_cast<size_t>(L.dw_chunk_waves) * more + 4);
  }
  plan_split(P);
  P.lds_pad = P.lds_floats;
  P.lds_floats += static_cast<int>(framed);
  // operands of the products that run on the matrix cores, while LDS has room for them
  P.n_mfma = 0;
  P.mf_ahead = -1;
  for (int i = 0; i < P.n; ++i) {
    TinyLayer &L = P.l[i];
    L.mf_fwd_w = L.mf_fwd_ko = L.mf_fwd_b = -1;
    // (few output channels leave most of a 16-row tile empty, and a short sum is over before
    // the operands of its first product have arrived: those stay with the scalar loops)
    if (L.kind != TDH_L_CONV || conv_is_matvec(L) || L.sh != 1 || L.sw != 1 || L.K < 8 ||
        L.C * L.R * L.S < 48)
      continue;
    const size_t room = TINY_LDS_MAX_BYTES / sizeof(float);
    const int taps = L.R * L.S;
    // (both areas start on 16 bytes: rows and offset tables are read four values at a time)
    if (L.ph == 0 && L.pw == 0) {
      const int n_k = L.C * taps;
      const size_t need = static_cast<size_t>(mfma_pitch(n_k)) * L.K + 4 * mfma_steps(n_k) + L.K;
      const int at = (P.lds_floats + 3) & ~3;
      if (at + need <= room) {
        L.mf_fwd_w = at; L.mf_fwd_ko = at + mfma_pitch(n_k) * L.K; L.mf_fwd_b = L.mf_fwd_ko + 4 * mfma_steps(n_k);
        P.lds_floats = at + static_cast<int>(need);
        P.mfma_layers[P.n_mfma++] = i;
        if (P.mf_ahead < 0 && i > 0 && L.K * n_k <= MFMA_AHEAD * TN_THREADS) P.mf_ahead = i;
      }
    }
  }
  for (int i = 0; i < P.n; ++i) P.l[i].mf_dx_w = P.l[i].mf_dx_ko = P.l[i].mf_dx_d = -1;
  if (P.mf_ahead > 0 && P.mf_ahead + 1 < P.n) {
    // the input gradient of that layer on the matrix cores: its operand goes into the scratch
    // area while the layer behind it runs its backward phase, which therefore must be one that
    // leaves that area alone (a pointwise activation or a pool), and D needs room of its own
    TinyLayer &L = P.l[P.mf_ahead];
    const TinyLayer &behind = P.l[P.mf_ahead + 1];
    // (not a closing softmax either: under cross_entropy_multiclass its backward phase is skipped)
    const bool quiet = (behind.kind == TDH_L_ACT && behind.act != TDH_ACT_SOFTMAX) || behind.kind == TDH_L_MAXPOOL ||
                       behind.kind == TDH_L_AVEPOOL;
    const int n_k = L.K * L.R, rows = L.C * L.S, cols = L.H * (L.W + L.S - 1);
    const size_t operand = static_cast<size_t>(mfma_pitch(n_k)) * rows + 4 * mfma_steps(n_k);
    const int at = (P.lds_floats + 3) & ~3;
    if (L.dx_framed && quiet && operand <= TINY_SCRATCH_FLOATS &&
        at + static_cast<size_t>(rows) * cols <= TINY_LDS_MAX_BYTES / sizeof(float)) {
      L.mf_dx_w  = P.lds_w;
      L.mf_dx_ko = P.lds_w + mfma_pitch(n_k) * rows;
      L.mf_dx_d  = at;
      P.lds_floats = at + rows * cols;
    }
  }
  // A matrix-vector layer whose filters a workgroup holds in registers while everything behind them runs: its rows are a
  // multiple of 16 bytes, in front of it lie pools and activations behind a product on the matrix cores, and behind
  // it fully-connected layers and activations (the loops that run meanwhile know no other kinds)
  P.held = P.held_from = 0;
  for (int h = 1; h < P.n; ++h) {
    const TinyLayer &L = P.l[h];
    if (L.kind != TDH_L_CONV || !conv_is_matvec(L) || L.tbl || ((L.C * L.R * L.S) & 3) || (L.lds_in & 3) ||
        (reinterpret_cast<uintptr_t>(L.w) & 15) || (1 << held_shape(L).shift) > TN_THREADS || held_shape(L).rows > HELD_ROWS)
      continue;
    int from = h - 1, end = h + 1;
    while (from > 0 && (is_pointwise(P.l[from]) || is_pool(P.l[from]))) --from;
    while (end < P.n && (P.l[end].kind == TDH_L_FC || P.l[end].kind == TDH_L_ACT)) ++end;
    if (P.l[from].mf_fwd_w < 0 || end < P.n || from < P.split) continue;
    P.held = h; P.held_from = from;
    P.held_shift  = held_shape(L).shift;
    P.held_rows   = held_shape(L).rows;
    P.d_held_rows = FastDiv(static_cast<uint32_t>(P.held_rows));
  }
  P.lds_job_floats = static_cast<int>(lds);
  return TDH_OK;
}

// The ends of the chain a channel a workgroup while there is a compute unit for each. LeNet-5's step, us, with them / one
// workgroup per sample throughout: 16 samples 40.7 / 52.1, 32 43.1 / 54.0, 42 50.7 / 55.8, 44 57.4 / 56.4, 64 60.6 / 61.4, 104 77.1 /
// 70.7: with several workgroups a compute unit, each of which frames all of dY for its one channel, they lose.
int tiny_most_split(const TinyPlan &plan) { return plan.split ? 256 / std::max(plan.l[0].K, plan.l[plan.split].C) : 0; }
static bool tiny_splits(const TinyPlan &plan, int batch) { return batch <= tiny_most_split(plan); }
// How the parameter gradients of a batch are split. Estimated us of a layer of channel pairs, fitted to LeNet-5's and to layers of 12 to 512
// pairs of 6x6 to 28x28 planes, 1 to 512 samples: whole rounds of 512 workgroups (two a compute unit, by their registers), each of which takes
// its latency, another trip to memory for every further lot of samples in LDS, and its products; and a share of the time of the launch's other
// workgroups. The step, us, with groups of 16 samples and a workgroup a pair / as chosen: LeNet-5, 33 samples 48.7 / 47.2, 256 100.9 / 91.3;
// 28x28, 1 -> 8 -> 16 channels, 3x3, pools, 128 samples 77.6 / 71.8; 12x12, 3 -> 16 -> 32, 3x3, pools, 33 samples 70.7 / 61.1, 256 145 / 84; 28x28,
// 1 -> 12, 5x5, pool, 64 samples 60.0 / 57.5.
struct PairSplit {
  int size, waves;   // samples of a group; a wave a pair instead of a workgroup
  double us;
};
static PairSplit pair_split(const TinyLayer &L, const int batch, const int size, const int waves) {
  const int chunk = waves ? L.dw_chunk_waves : L.dw_chunk, units = size * ((L.OH + 3) / 4) * L.OW;
  const int workgroups = ceil_div(batch, size) * L.K * (waves ? ceil_div(L.C, TP_WAVES) : L.C);
  const double each = 8.0 + 3.0 * (ceil_div(size, chunk) - 1) + 0.032 * L.R * L.S * ceil_div(units, waves ? 64 : TP_THREADS);
  return {size, waves, ceil_div(workgroups, 512) * each + workgroups / 170.0};
}
// of groups of up to 32 samples, or of all of them
static PairSplit best_pair_split(const TinyLayer &L, const int batch, const bool whole) {
  PairSplit best = {0, 0, 0.0};
  for (int waves = 0; waves <= (L.dw_chunk_waves > 0 && !whole); ++waves)
    for (int size = whole ? batch : 4; size <= std::min(whole ? batch : 32, batch); size *= 2) {
      const PairSplit p = pair_split(L, batch, size, waves);
      if (!best.size || p.us < best.us) best = p;
    }
  if (!best.size) best = pair_split(L, batch, batch, 0);   // (fewer than four samples)
  return best;
}
TinyGroups tiny_groups(const TinyPlan &plan, const int batch) {
  TinyGroups g = {};
  const int m = tiny_splits(plan, batch) ? plan.split : 0;
  // One group is updated by the launch that adds it up, and the optimizer's launch, 5 us, left out: where no layer takes
  // longer for it than that. (Outer products and column sums have sixteen samples at a time in flight, a trip to memory each; a step of
  // 784-30-10 fully connected, us, in several groups / one: 33 samples 28.8 / 25.4, 64 29.1 / 26.6; of 64-64-10, 33 22.2 / 20.5, 64 22.3 / 21.7.)
  bool pairs = false, pools = false, rows = false;
  double one = 0.0, several = 0.0;
  g.one = batch <= 64;
  for (int i = 0; i < plan.n; ++i) {
    const TinyLayer &L = plan.l[i];
    if (!L.nw || i < m) continue;
    if (conv_by_rows(plan, L)) {
      rows  = true;
      // (a sample after the other: a trip to memory and some 0.1 us a lane's pixel, where the optimizer's launch takes 4.3)
      g.one = g.one && (batch - 1) * (1.2 + 0.1 * ceil_div(L.OH, conv_rows_lanes(L, batch)) * L.OW) <= 4.3;
    } else if (L.kind == TDH_L_CONV && !conv_is_matvec(L)) {
      pairs   = true;
      if (!g.one) continue;
      one     = std::max(one, best_pair_split(L, batch, true).us);
      several = std::max(several, best_pair_split(L, batch, false).us);
    } else if (L.kind == TDH_L_AVEPOOL) {
      pools = true;
      g.one = g.one && batch <= L.dw_chunk;
    }
  }
  g.one = g.one && one <= several + 5.0 && (batch <= 32 || !(pairs || pools || m));
  for (int i = 0; i < plan.n; ++i) {
    const TinyLayer &L = plan.l[i];
    // (beside single samples' sums the kernel has registers for four samples in flight: one trip each, unless that makes many slices)
    g.size[i] = g.one ? batch : std::min(batch, rows && static_cast<long>(L.nw) * ceil_div(batch, 4) <= 1L << 18 ? 4 : 16);
    if (!L.nw || i < m) continue;
    if (conv_by_rows(plan, L)) {
      g.size[i] = g.one ? batch : 1;
    } else if (L.kind == TDH_L_CONV && !conv_is_matvec(L)) {
      const PairSplit p = best_pair_split(L, batch, g.one);
      g.size[i]  = p.size;
      g.waves[i] = p.waves;
    } else if (L.kind == TDH_L_AVEPOOL) {
      g.size[i] = std::min({g.size[i], L.dw_chunk, rows ? std::max(4, batch * L.C / 256) : batch});
    }
  }
  return g;
}

int launch_tiny_step(const TinyPlan &plan, const TinyPlan *dev_plan, int loss, int softmax_xent, int batch,
                     const float *x, const float *t) {
  const TinyLayer &F = plan.l[0], &M = plan.l[plan.split];
  const int m = tiny_splits(plan, batch) ? plan.split : 0;
  const double front_flop = m ? 2.0 * F.out_size * F.C * F.R * F.S * batch : 0.0;
  const double back_flop  = m ? 2.0 * M.out_size * M.C * M.R * M.S * batch : 0.0;
  if (m) {
    ProfScope prof("tiny_net_front", front_flop, WORK_FLOP);
    // (a pixel a thread, in whole waves)
    const int plane = F.OH * F.OW, rounds = ceil_div(plane, TF_THREADS), threads = 64 * ceil_div(plane, 64 * rounds);
    TDH_LAUNCH(tiny_net_front_kernel, dim3(batch, F.K), dim3(threads), (plan.in_size + plan.front_floats) * sizeof(float),
               ctx().stream, dev_plan, m, plan.in_size, x);
    TDH_LAUNCH_CHECK();
  }
  {
    ProfScope prof("tiny_net_step", plan.flop_per_sample * batch * (2.0 / 3.0) - front_flop - back_flop, WORK_FLOP);
    auto kernel = plan.held ? tiny_net_step_kernel<true> : tiny_net_step_kernel<false>;
    TDH_LAUNCH(kernel, dim3(batch), dim3(TN_THREADS), plan.lds_floats * sizeof(float), ctx().stream,
               dev_plan, m, loss, softmax_xent, x, t);
    TDH_LAUNCH_CHECK();
  }
  if (m) {
    ProfScope prof("tiny_net_back", back_flop, WORK_FLOP);
    TDH_LAUNCH(tiny_net_back_kernel, dim3(batch, M.C), dim3(TB_THREADS), plan.back_floats * sizeof(float), ctx().stream,
               dev_plan, m, x);
    TDH_LAUNCH_CHECK();
  }
  return TDH_OK;
}

int launch_tiny_params(const TinyPlan &plan, const TinyPlan *dev_plan, const TinyGroups &groups, int batch, const float *x,
                       tdh_opt *update, int n_tensors, const float *powers_in, float *powers_out) {
  TinyRanges r;
  int n = 0, blocks = 0;
  int roads = (plan.first_dx_as_job ? TP_HAS_DX : 0) | (plan.by_rows ? TP_HAS_ROWS : 0);
  const int threads = param_threads(roads);
  auto add = [&](int layer, int what, int count) {
    r.first[n]     = blocks;
    r.job[n]       = layer * 16 + what;
    r.per_group[n] = count;
    r.size[n++]    = groups.size[layer];
    blocks += count * ceil_div(batch, groups.size[layer]);
  };
  const int m = tiny_splits(plan, batch) ? plan.split : 0;
  for (int pass = 0; pass < 2; ++pass)   // (the convolutions first: they take longest)
    for (int i = 0; i < plan.n; ++i) {
      const TinyLayer &L = plan.l[i];
      const bool pair = L.kind == TDH_L_CONV && !conv_is_matvec(L);
      if (!L.nw || pair != (pass == 0)) continue;
      if (i < m) {   // left by the back kernel, sample by sample
        add(i, TP_SLICES_W, ceil_div(L.nw, threads));
        if (L.nb) add(i, TP_SLICES_B, ceil_div(L.nb, threads));
      } else if (conv_by_rows(plan, L)) {
        add(i, TP_ROWS, ceil_div(conv_rows_weight_units(L, batch) + L.nb * conv_rows_bias_lanes(L), threads));
      } else if (pair) {
        const bool waves = groups.waves[i];
        roads |= waves ? TP_HAS_WAVES : 0;
        add(i, waves ? TP_CONV_WAVES : TP_CONV, L.K * (waves ? ceil_div(L.C, TP_WAVES) : L.C));
      } else if (L.kind == TDH_L_AVEPOOL) {
        add(i, TP_POOL, L.C);
      } else {
        const bool conv = L.kind == TDH_L_CONV;
        const int fast = conv ? L.in_size : L.out_size;
        const bool vec = fast % 4 == 0 && (i > 0 || !conv || (reinterpret_cast<uintptr_t>(x) & 15u) == 0);
        add(i, vec ? TP_OUTER4 : TP_OUTER, ceil_div(L.nw, (vec ? 4 : 1) * threads));
        if (L.nb) add(i, TP_COLUMNS, ceil_div(L.nb, threads));
      }
    }
  for (int k = n; k < TP_RANGES; ++k) {
    r.first[k] = 0x7fffffff;
    r.job[k] = r.per_group[k] = r.size[k] = 0;
  }
  const int dx_blocks = plan.first_dx_as_job ? dx_band(plan.l[0]).bands * plan.l[0].C * batch : 0;
  TinyUpdate u;
  if (update) {
    u.p = opt_scalars(*update, 1.0f);
    u.n_tensors = n_tensors;
    u.b1_t = update->b1_t; u.b2_t = update->b2_t;
    u.powers_in = powers_in; u.powers_out = powers_out;
  }
  if (blocks + dx_blocks > 0) {
    ProfScope prof(roads & TP_HAS_ROWS ? "tiny_net_param_grads_any" : roads & TP_HAS_WAVES ? "tiny_net_param_grads_waves" : "tiny_net_param_grads", plan.flop_per_sample * batch * (1.0 / 3.0), WORK_FLOP);
    const auto kernel = param_kernel(update ? update->kind : -1, roads);
    if (!kernel) return set_error(TDH_ERR_INVALID, "optimizer kind %d is not supported", update->kind);
    TDH_LAUNCH(kernel, dim3(blocks + dx_blocks), dim3(threads), plan.lds_job_floats * sizeof(float),
               ctx().stream, dev_plan, x, r, u, batch, blocks);
    TDH_LAUNCH_CHECK();
  }
  if (update) opt_advance(update, n_tensors);
  return TDH_OK;
}

int launch_tiny_merge(const TinyMerge &m) {
  if (m.n == 0) return TDH_OK;
  double bytes = 0.0;
  for (int j = 0; j < m.n; ++j) bytes += 4.0 * m.len[j] * (m.count[j] + 2);
  ProfScope prof("tiny_net_merge_grads", bytes, WORK_BYTE);
  TDH_LAUNCH(tiny_net_merge_kernel, dim3(m.first_block[m.n]), dim3(256), 0, ctx().stream, m);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace tdh
