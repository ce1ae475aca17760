// norm.hip — batch normalization and dropout: the two layers of the reference whose backward
// pass needs more than the layer's own output gradient (batch statistics, a mask).
//
// Both are bound by HBM on large tensors and by the number of launches on small ones: every
// kernel here reads or writes each element once, and the small sums between two passes are taken
// by every workgroup of the next pass for itself (a wave adds a channel's partial sums in a
// fixed order, so all of them get the same bits) instead of by a launch in between. Tensors are
// [batch][channels][spatial] floats; a channel's elements are `batch` runs of `spatial`
// consecutive floats.
//
// Statistics follow tiny_dnn/util/math_functions.h:25-96: mean = sum / (batch*spatial), variance
// = sum (x - mean)^2 / max(1, batch*spatial - 1), two passes. The sums are taken in a fixed
// order that depends on the shape only: workgroup (channel, group) adds the runs of images
// g, g+G, ... (a block-wide tree behind the threads' own sums), a wave of every workgroup of the
// next pass adds the group sums.
//
// 64 channels of 56x56, batch 32 (25.7 MB a tensor), us: forward 32.6 in five launches of one
// 4-byte access per thread and step, now 18.8 in three; backward 28.5 in three, now 21.7 in two.
#include <algorithm>
#include <cfloat>

#include "common.h"

namespace tdh {

namespace {

constexpr int NT = 256;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ float block_sum(float v, float *smem4) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) smem4[threadIdx.x >> 6] = v;
  __syncthreads();
  const float r = (smem4[0] + smem4[1]) + (smem4[2] + smem4[3]);
  __syncthreads();
  return r;
}

template <int V>
__device__ __forceinline__ void load_run(const float *p, float (&v)[V]) {
  if (V == 4) {
    const float4 q = *reinterpret_cast<const float4 *>(p);
    v[0] = q.x; v[V > 1 ? 1 : 0] = q.y; v[V > 2 ? 2 : 0] = q.z; v[V - 1] = q.w;
  } else {
    v[0] = p[0];
  }
}
template <int V>
__device__ __forceinline__ void store_run(float *p, const float (&v)[V]) {
  if (V == 4)
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[V > 1 ? 1 : 0], v[V > 2 ? 2 : 0], v[V - 1]);
  else
    p[0] = v[0];
}

// A workgroup's piece of its channel: elements [beg, end) of the channel's batch*spatial values
// in steps of V adjacent ones (V = 4 where spatial is a multiple of 4 and the tensors are
// 16-byte aligned: a step then never leaves its run). A channel may have just under 2^31 of them, so
// positions are unsigned: the step behind the last one passes 2^31.
struct BnGeom {
  int channels, spatial, batch, total;  // total: batch * spatial
  int chunk, groups;                    // pieces of the elementwise passes
  int sum_groups;                       // workgroups, and partial sums, per channel of the sums
  FastDiv div_spatial;
};
template <typename F>
__device__ __forceinline__ void for_piece(const BnGeom &g, const int v, const F &visit) {
  const int ch       = blockIdx.x;
  const uint32_t beg = blockIdx.y * static_cast<uint32_t>(g.chunk);
  const uint32_t end = min(static_cast<uint32_t>(g.total), beg + g.chunk);
  for (uint32_t e = beg + v * threadIdx.x; e < end; e += v * NT) {
    uint32_t img, i;
    g.div_spatial.divmod(e, img, i);
    visit((static_cast<size_t>(img) * g.channels + ch) * g.spatial + i);
  }
}

// the sum of a channel's partial sums, the same bits in every wave of every workgroup
__device__ __forceinline__ float group_sum(const float *__restrict__ partial, const int row, const int groups) {
  float s = 0.0f;
  for (int g = threadIdx.x & 63; g < groups; g += 64) s += partial[row * groups + g];
  return wave_sum(s);
}

// MODE 0: sum a; MODE 1: sum (a - mean)^2, the mean from the partial sums of MODE 0 (and left
// in mean_out); MODE 2: sum a and sum a*b (two partials). Workgroup (channel, group) adds the runs
// of images group, group + groups, ...: a thread every 256th value of a run, one after the other.
// The loads of four of its values travel together (a load per addition left the kernel waiting for
// one cache line after the other).
template <int MODE>
__global__ void __launch_bounds__(NT)
bn_partial_kernel(const float *__restrict__ a, const float *__restrict__ b, const float *__restrict__ sums,
                  const float denom, const BnGeom g, float *__restrict__ mean_out, float *__restrict__ partial) {
  __shared__ float smem4[4];
  const int ch = blockIdx.x;
  float c = 0.0f;
  if (MODE == 1) {
    c = group_sum(sums, ch, g.sum_groups) / denom;
    if (blockIdx.y == 0 && threadIdx.x == 0) mean_out[ch] = c;
  }
  float s0 = 0.0f, s1 = 0.0f;
  const auto add = [&](const float va, const float vb) {
    if (MODE == 0) s0 += va;
    if (MODE == 1) s0 += (va - c) * (va - c);
    if (MODE == 2) { s0 += va; s1 += va * vb; }
  };
  for (int o = blockIdx.y; o < g.batch; o += g.sum_groups) {
    const size_t base = (static_cast<size_t>(o) * g.channels + ch) * g.spatial;
    const uint32_t spatial = g.spatial;
    uint32_t i             = threadIdx.x;
    for (; i + 3 * NT < spatial; i += 4 * NT) {
      float va[4], vb[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        va[k] = a[base + i + k * NT];
        vb[k] = MODE == 2 ? b[base + i + k * NT] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) add(va[k], vb[k]);
    }
    for (; i < spatial; i += NT) add(a[base + i], MODE == 2 ? b[base + i] : 0.0f);
  }
  s0 = block_sum(s0, smem4);
  if (MODE == 2) s1 = block_sum(s1, smem4);
  if (threadIdx.x == 0) {
    partial[ch * g.sum_groups + blockIdx.y] = s0;
    if (MODE == 2) partial[(g.channels + ch) * g.sum_groups + blockIdx.y] = s1;
  }
}

// batch_normalization_layer.h:150-163: y = (x - mean[ch]) / stddev[ch]. squares: the partial sums
// of (x - mean)^2 that give this batch's variance (left in `variance`), or null: `variance` is given.
template <int V>
__global__ void __launch_bounds__(NT)
bn_apply_kernel(const float *__restrict__ x, const float *__restrict__ mean, const float *__restrict__ squares,
                const float denom, const float eps, const BnGeom g, float *__restrict__ variance,
                float *__restrict__ stddev, float *__restrict__ y) {
  const int ch   = blockIdx.x;
  const float m  = mean[ch];
  const float va = squares ? group_sum(squares, ch, g.sum_groups) / denom : variance[ch];
  const float sd = sqrtf(va + eps);
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    if (squares) variance[ch] = va;
    stddev[ch] = sd;
  }
  for_piece(g, V, [&](const size_t at) {
    float v[V];
    load_run<V>(x + at, v);
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = (v[k] - m) / sd;
    store_run<V>(y + at, v);
  });
}

// The rectifier behind a batch normalization (relu_layer.h:25-39, leaky_relu_layer.h:74-88), as the layer's own
// kernels compute it.
template <bool LEAKY>
__device__ __forceinline__ float rectify(const float x, const float slope) {
  return x > 0.0f ? x : LEAKY ? slope * x : 0.0f;
}
template <bool LEAKY>
__device__ __forceinline__ float rectify_grad(const float y, const float dy, const float slope) {
  return dy * (y > 0.0f ? 1.0f : LEAKY ? slope : 0.0f);
}

// A 2x2 / stride-2 max-pool behind them: the planes of its input in blocks of 2x2, the last row and column of
// an odd plane in blocks that are no window.
struct BnPoolGeom {
  int H, W, OH, OW, bw, blocks;   // blocks of a row, of a plane
  int total, piece;               // blocks of a channel, of a workgroup's piece
  FastDiv div_blocks, div_bw, div_w;
};

// bn_apply_kernel with the rectifier and the max-pool behind it: every output is written, with the bits of the
// three kernels (max-pool: row by row, strict '>', start value lowest(), an all-NaN window reports index 0).
// Bound, small nets: launches of 4 us each. 24 channels of 30x30 and 48 of 15x15, batch 37: the three layers
// 13.9 and 13.3 us in a launch each, here 5.9 and 5.4.
template <bool LEAKY>
__global__ void __launch_bounds__(NT)
bn_apply_act_pool_kernel(const float *__restrict__ x, const float *__restrict__ mean, const float *__restrict__ squares,
                         const float denom, const float eps, const BnGeom g, const BnPoolGeom p, const float slope,
                         float *__restrict__ variance, float *__restrict__ stddev, float *__restrict__ y,
                         float *__restrict__ act, float *__restrict__ pooled, int32_t *__restrict__ argmax) {
  const int ch   = blockIdx.x;
  const float m  = mean[ch];
  const float va = squares ? group_sum(squares, ch, g.sum_groups) / denom : variance[ch];
  const float sd = sqrtf(va + eps);
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    if (squares) variance[ch] = va;
    stddev[ch] = sd;
  }
  const uint32_t end = min(static_cast<uint32_t>(p.total), (blockIdx.y + 1u) * p.piece);
  for (uint32_t e = blockIdx.y * p.piece + threadIdx.x; e < end; e += NT) {
    uint32_t img, b, by, bx;
    p.div_blocks.divmod(e, img, b);
    p.div_bw.divmod(b, by, bx);
    const int x0 = 2 * bx, y0 = 2 * by;
    const bool right = x0 + 1 < p.W, low = y0 + 1 < p.H;
    const size_t plane = static_cast<size_t>(img) * g.channels + ch;
    const size_t at    = plane * g.spatial + y0 * p.W + x0;
    const int off[4]   = {0, 1, p.W, p.W + 1};
    const bool on[4]   = {true, right, low, right && low};
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = x[at + (on[k] ? off[k] : 0)];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float n = (v[k] - m) / sd;
      v[k]          = rectify<LEAKY>(n, slope);
      if (on[k]) {
        y[at + off[k]]   = n;
        act[at + off[k]] = v[k];
      }
    }
    if (!(right && low)) continue;
    float best = -FLT_MAX;
    int sel    = -1;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (v[k] > best) {
        best = v[k];
        sel  = k;
      }
    const size_t o = (plane * p.OH + by) * p.OW + bx;
    pooled[o] = best;
    argmax[o] = sel < 0 ? 0 : (p.H * ch + y0) * p.W + x0 + off[sel];
  }
}

// bn_partial_kernel<2> on a gradient that comes through the max-pool and the rectifier behind the layer: each
// element's own gradient is routed from dpool (max_pooling_layer.h:218: the last window that holds it), written
// (d_act: of the rectifier's output, where somebody reads it; d_norm: of this layer's) and summed where the
// kernel of one layer would read it, so the sums are the same bits.
template <bool LEAKY>
__global__ void __launch_bounds__(NT)
bn_pool_grad_partial_kernel(const float *__restrict__ dpool, const int32_t *__restrict__ argmax, const float *__restrict__ act,
                            const float *__restrict__ y, const BnGeom g, const BnPoolGeom p, const float slope,
                            float *__restrict__ d_act, float *__restrict__ d_norm, float *__restrict__ partial) {
  __shared__ float smem4[4];
  const int ch = blockIdx.x;
  float s0 = 0.0f, s1 = 0.0f;
  for (int o = blockIdx.y; o < g.batch; o += g.sum_groups) {
    const size_t base   = (static_cast<size_t>(o) * g.channels + ch) * g.spatial;
    const size_t sample = static_cast<size_t>(o) * g.channels * p.OH * p.OW;
    const uint32_t spatial = g.spatial;
    for (uint32_t i0 = threadIdx.x; i0 < spatial; i0 += 4 * NT) {
      float d[4], a[4], b[4];
      int rec[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t i = min(i0 + k * NT, spatial - 1);
        uint32_t yy, xx;
        p.div_w.divmod(i, yy, xx);
        const int ox = min(p.OW - 1, static_cast<int>(xx) >> 1), oy = min(p.OH - 1, static_cast<int>(yy) >> 1);
        const bool covered = static_cast<int>(xx) < 2 * ox + 2 && static_cast<int>(yy) < 2 * oy + 2;
        const size_t w     = sample + (covered ? (p.OH * ch + oy) * p.OW + ox : 0);
        rec[k] = argmax[w];
        d[k]   = dpool[w];
        a[k]   = act[base + i];
        b[k]   = y[base + i];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t i = i0 + k * NT;
        if (i >= spatial) break;
        const float da = rec[k] == static_cast<int>(g.spatial * ch + i) ? d[k] : 0.0f;
        const float dn = rectify_grad<LEAKY>(a[k], da, slope);
        if (d_act) d_act[base + i] = da;
        d_norm[base + i] = dn;
        s0 += dn;
        s1 += dn * b[k];
      }
    }
  }
  s0 = block_sum(s0, smem4);
  s1 = block_sum(s1, smem4);
  if (threadIdx.x == 0) {
    partial[ch * g.sum_groups + blockIdx.y] = s0;
    partial[(g.channels + ch) * g.sum_groups + blockIdx.y] = s1;
  }
}

// batch_normalization_layer.h:112-125:
//   dx = (dy - mean(dy)[ch] - mean(dy*y)[ch] * y) / stddev[ch]
template <int V>
__global__ void __launch_bounds__(NT)
bn_bwd_apply_kernel(const float *__restrict__ y, const float *__restrict__ dy, const float *__restrict__ sums,
                    const float denom, const float *__restrict__ stddev, const BnGeom g, float *__restrict__ dx) {
  const int ch   = blockIdx.x;
  const float m0 = group_sum(sums, ch, g.sum_groups) / denom;
  const float m1 = group_sum(sums, g.channels + ch, g.sum_groups) / denom;
  const float sd = stddev[ch];
  for_piece(g, V, [&](const size_t at) {
    float v[V], w[V];
    load_run<V>(dy + at, v);
    load_run<V>(y + at, w);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const float u = v[k] - m0 - m1 * w[k];
      v[k]          = u / sd;
    }
    store_run<V>(dx + at, v);
  });
}

// batch_normalization_layer.h:171-177 (post_update), of every layer of a net in one launch
__global__ void __launch_bounds__(NT) bn_moving_kernel(const BnMovingJobs jobs) {
  const BnMoving &j = jobs.job[blockIdx.y];
  const int c       = blockIdx.x * NT + threadIdx.x;
  if (c >= j.channels) return;
  j.mean[c] = j.momentum * j.mean[c] + (1 - j.momentum) * j.mean_cur[c];
  j.var[c]  = j.momentum * j.var[c] + (1 - j.momentum) * j.var_cur[c];
}

// dropout_layer.h:104-113: y = mask * scale * x in the train phase, y = x otherwise
__global__ void __launch_bounds__(NT)
dropout_fwd_kernel(const uint8_t *__restrict__ mask, const float scale, const float *__restrict__ x,
                   const size_t total, float *__restrict__ y) {
  const size_t i = static_cast<size_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= total) return;
  y[i] = mask ? (static_cast<float>(mask[i]) * scale) * x[i] : x[i];
}

// dropout_layer.h:74-82: dx = mask * dy (the scale is NOT applied on the way back)
__global__ void __launch_bounds__(NT)
dropout_bwd_kernel(const uint8_t *__restrict__ mask, const float *__restrict__ dy,
                   const size_t total, float *__restrict__ dx) {
  const size_t i = static_cast<size_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= total) return;
  dx[i] = static_cast<float>(mask[i]) * dy[i];
}

// The same, and through the pointwise activation in front of the dropout layer (tanh_layer.h:30-38, relu_layer.h:31-39,
// sigmoid_layer.h:30-38, on its output y). Bound: a launch; of 37 x 64 values 1.9 and 2.2 us apart, 2.2 together, and the step of that
// net, mean of three processes each, 169.3 -> 167.5.
__global__ void __launch_bounds__(NT)
dropout_act_bwd_kernel(const uint8_t *__restrict__ mask, const float *__restrict__ dy, const size_t total,
                       float *__restrict__ dx, const int act, const float *__restrict__ y, float *__restrict__ act_dx) {
  const size_t i = static_cast<size_t>(blockIdx.x) * NT + threadIdx.x;
  if (i >= total) return;
  const float g = static_cast<float>(mask[i]) * dy[i], v = y[i];
  dx[i]     = g;
  act_dx[i] = act == TDH_ACT_TANH ? g * (1.0f - v * v) : act == TDH_ACT_RELU ? g * (v > 0.0f ? 1.0f : 0.0f) : g * v * (1.0f - v);
}

int bn_groups(int batch) { return batch < 64 ? batch : 64; }

// The elementwise passes: about 2048 workgroups where the tensor is large enough, and at least
// four values a thread. The sums: a workgroup per image and channel, up to 64 per channel.
BnGeom bn_geom(int channels, int spatial, int batch) {
  BnGeom g;
  g.channels = channels; g.spatial = spatial; g.batch = batch; g.total = batch * spatial;
  const auto up = [](long a, long b) { return (a + b - 1) / b; };
  g.chunk       = static_cast<int>(up(up(g.total, std::min(256, std::max(1, 2048 / channels))), 4 * NT) * 4 * NT);
  g.groups      = static_cast<int>(up(g.total, g.chunk));
  g.sum_groups  = bn_groups(batch);
  g.div_spatial = FastDiv(spatial);
  return g;
}

bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

size_t batchnorm_workspace_bytes(int channels, int batch) {
  // partial sums of two quantities
  return ws_align(sizeof(float) * 2 * static_cast<size_t>(channels) * bn_groups(batch));
}

#define BN_LAUNCH(kernel, groups, ...)                                                                    \
  do {                                                                                            \
    const dim3 grid(g.channels, groups);                                                          \
    TDH_LAUNCH((kernel), grid, dim3(NT), 0, ctx().stream, __VA_ARGS__);                           \
    TDH_LAUNCH_CHECK();                                                                           \
  } while (0)

// the mean, and the partial sums of the squares around it
static int moments(const BnGeom &g, const float *x, float *mean, float **squares) {
  void *ws = nullptr;
  TDH_TRY(ws_take(sizeof(float) * 2 * static_cast<size_t>(g.channels) * g.sum_groups, &ws));
  float *sums = static_cast<float *>(ws);
  *squares    = sums + static_cast<size_t>(g.channels) * g.sum_groups;
  ProfScope prof("batchnorm_moments", 8.0 * g.channels * static_cast<double>(g.total), WORK_BYTE);
  BN_LAUNCH((bn_partial_kernel<0>), g.sum_groups, x, nullptr, nullptr, 1.0f, g, nullptr, sums);
  BN_LAUNCH((bn_partial_kernel<1>), g.sum_groups, x, nullptr, sums, static_cast<float>(g.total), g, mean, *squares);
  return TDH_OK;
}

template <int V>
static int batchnorm_fwd_run(const BnGeom &g, float eps, int train, const float *x, float *mean, float *variance,
                             float *stddev, float *y) {
  const double bytes = 8.0 * g.channels * static_cast<double>(g.total);
  const float n      = static_cast<float>(g.total);
  float *squares     = nullptr;
  if (train) TDH_TRY(moments(g, x, mean, &squares));
  ProfScope prof("batchnorm_fwd", bytes, WORK_BYTE);
  BN_LAUNCH(bn_apply_kernel<V>, g.groups, x, mean, squares, std::max(1.0f, n - 1.0f), eps, g, variance, stddev, y);
  return TDH_OK;
}

int batchnorm_fwd(int channels, int spatial, int batch, float eps, int train, const float *x,
                  float *mean, float *variance, float *stddev, float *y) {
  const BnGeom g = bn_geom(channels, spatial, batch);
  return spatial % 4 == 0 && aligned16(x) && aligned16(y)
           ? batchnorm_fwd_run<4>(g, eps, train, x, mean, variance, stddev, y)
           : batchnorm_fwd_run<1>(g, eps, train, x, mean, variance, stddev, y);
}

template <int V>
static int batchnorm_bwd_run(const BnGeom &g, const float *y, const float *dy, const float *stddev, float *dx) {
  const double bytes = 4.0 * g.channels * static_cast<double>(g.total);
  void *ws = nullptr;
  TDH_TRY(ws_take(sizeof(float) * 2 * static_cast<size_t>(g.channels) * g.sum_groups, &ws));
  float *sums = static_cast<float *>(ws);
  {
    ProfScope prof("batchnorm_bwd_moments", 2 * bytes, WORK_BYTE);
    BN_LAUNCH((bn_partial_kernel<2>), g.sum_groups, dy, y, nullptr, 1.0f, g, nullptr, sums);
  }
  ProfScope prof("batchnorm_bwd", 3 * bytes, WORK_BYTE);
  BN_LAUNCH(bn_bwd_apply_kernel<V>, g.groups, y, dy, sums, static_cast<float>(g.total), stddev, g, dx);
  return TDH_OK;
}

int batchnorm_bwd(int channels, int spatial, int batch, const float *y, const float *dy,
                  const float *stddev, float *dx) {
  const BnGeom g = bn_geom(channels, spatial, batch);
  return spatial % 4 == 0 && aligned16(y) && aligned16(dy) && aligned16(dx)
           ? batchnorm_bwd_run<4>(g, y, dy, stddev, dx) : batchnorm_bwd_run<1>(g, y, dy, stddev, dx);
}

static BnPoolGeom bn_pool_geom(const BnGeom &g, const tdh_pool_desc *d) {
  BnPoolGeom p;
  p.H = d->in_h; p.W = d->in_w; p.OH = d->in_h / 2; p.OW = d->in_w / 2;
  p.bw     = ceil_div(p.W, 2);
  p.blocks = p.bw * ceil_div(p.H, 2);
  p.total  = g.batch * p.blocks;
  // (pieces as in bn_geom, a block to a thread at least)
  const int pieces = std::min(256, std::max(1, 2048 / g.channels));
  p.piece      = ceil_div(ceil_div(p.total, pieces), NT) * NT;
  p.div_blocks = FastDiv(p.blocks); p.div_bw = FastDiv(p.bw); p.div_w = FastDiv(p.W);
  return p;
}

// A batch normalization, a rectifier and a 2x2 / stride-2 max-pool on its planes, whole windows only.
bool batchnorm_takes_pool(int channels, int spatial, int act_kind, const tdh_pool_desc *d) {
  return (act_kind == TDH_ACT_RELU || act_kind == TDH_ACT_LEAKY_RELU) && d->pool_w == 2 && d->pool_h == 2 &&
         d->stride_w == 2 && d->stride_h == 2 && !d->ceil_mode && !d->pad_same && d->in_c == channels &&
         d->in_w * d->in_h == spatial && d->in_w >= 2 && d->in_h >= 2;
}
int batchnorm_act_pool_fwd(int channels, int spatial, int batch, float eps, int train, const float *x, float *mean,
                           float *variance, float *stddev, float *y, int act_kind, float slope, float *act,
                           const tdh_pool_desc *d, float *pooled, int32_t *argmax) {
  const BnGeom g     = bn_geom(channels, spatial, batch);
  const BnPoolGeom p = bn_pool_geom(g, d);
  float *squares     = nullptr;
  if (train) TDH_TRY(moments(g, x, mean, &squares));
  ProfScope prof("batchnorm_fwd_act_pool", 4.0 * channels * (3.0 * g.total + 2.0 * batch * p.OH * p.OW), WORK_BYTE);
  const float n    = static_cast<float>(g.total);
  const int groups = ceil_div(p.total, p.piece);
  if (act_kind == TDH_ACT_RELU)
    BN_LAUNCH(bn_apply_act_pool_kernel<false>, groups, x, mean, squares, std::max(1.0f, n - 1.0f), eps, g, p, slope, variance,
              stddev, y, act, pooled, argmax);
  else
    BN_LAUNCH(bn_apply_act_pool_kernel<true>, groups, x, mean, squares, std::max(1.0f, n - 1.0f), eps, g, p, slope, variance,
              stddev, y, act, pooled, argmax);
  return TDH_OK;
}
int batchnorm_act_pool_bwd(int channels, int spatial, int batch, const float *y, const float *stddev, int act_kind,
                           float slope, const float *act, const tdh_pool_desc *d, const float *dpool, const int32_t *argmax,
                           float *d_act, float *d_norm, float *dx) {
  const BnGeom g     = bn_geom(channels, spatial, batch);
  const BnPoolGeom p = bn_pool_geom(g, d);
  const double bytes = 4.0 * channels * static_cast<double>(g.total);
  void *ws = nullptr;
  TDH_TRY(ws_take(sizeof(float) * 2 * static_cast<size_t>(channels) * g.sum_groups, &ws));
  float *sums = static_cast<float *>(ws);
  {
    ProfScope prof("batchnorm_bwd_pool_moments", (d_act ? 4 : 3) * bytes + 8.0 * channels * batch * p.OH * p.OW, WORK_BYTE);
    if (act_kind == TDH_ACT_RELU)
      BN_LAUNCH(bn_pool_grad_partial_kernel<false>, g.sum_groups, dpool, argmax, act, y, g, p, slope, d_act, d_norm, sums);
    else
      BN_LAUNCH(bn_pool_grad_partial_kernel<true>, g.sum_groups, dpool, argmax, act, y, g, p, slope, d_act, d_norm, sums);
  }
  ProfScope prof("batchnorm_bwd", 3 * bytes, WORK_BYTE);
  if (spatial % 4 == 0 && aligned16(y) && aligned16(d_norm) && aligned16(dx))
    BN_LAUNCH(bn_bwd_apply_kernel<4>, g.groups, y, d_norm, sums, static_cast<float>(g.total), stddev, g, dx);
  else
    BN_LAUNCH(bn_bwd_apply_kernel<1>, g.groups, y, d_norm, sums, static_cast<float>(g.total), stddev, g, dx);
  return TDH_OK;
}

int batchnorm_update_moving(const BnMoving *jobs, int n) {
  for (int at = 0; at < n; at += BN_MOVING_MAX) {
    BnMovingJobs j;
    const int here = std::min(BN_MOVING_MAX, n - at);
    int most       = 0;
    for (int k = 0; k < here; ++k) {
      j.job[k] = jobs[at + k];
      most     = std::max(most, j.job[k].channels);
    }
    if (most <= 0) continue;
    TDH_LAUNCH(bn_moving_kernel, dim3(ceil_div(most, NT), here), dim3(NT), 0, ctx().stream, j);
    TDH_LAUNCH_CHECK();
  }
  return TDH_OK;
}

int dropout_fwd(size_t total, int train, float scale, const uint8_t *mask, const float *x, float *y) {
  ProfScope prof("dropout_fwd", (train ? 9.0 : 8.0) * total, WORK_BYTE);
  TDH_LAUNCH(dropout_fwd_kernel, dim3(static_cast<unsigned>(ceil_div_sz(total, NT))),
                     dim3(NT), 0, ctx().stream, train ? mask : nullptr, scale, x, total, y);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

int dropout_act_bwd(size_t total, const uint8_t *mask, const float *dy, float *dx, int act, const float *y, float *act_dx) {
  ProfScope prof("dropout_act_bwd", 17.0 * total, WORK_BYTE);
  TDH_LAUNCH(dropout_act_bwd_kernel, dim3(static_cast<unsigned>(ceil_div_sz(total, NT))), dim3(NT), 0, ctx().stream, mask, dy,
             total, dx, act, y, act_dx);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

int dropout_bwd(size_t total, const uint8_t *mask, const float *dy, float *dx) {
  ProfScope prof("dropout_bwd", 9.0 * total, WORK_BYTE);
  TDH_LAUNCH(dropout_bwd_kernel, dim3(static_cast<unsigned>(ceil_div_sz(total, NT))),
                     dim3(NT), 0, ctx().stream, mask, dy, total, dx);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace tdh
