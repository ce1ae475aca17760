// fc_fwd_direct.hip — forward pass of a fully-connected layer for a few samples (inference), with the
// pointwise activation or the softmax behind it in the same launch.
//
//   y[n][o] = b[o] + sum_k x[n][k] W[k][o]
//
// A workgroup owns 16 outputs of 16 samples, as conv_fwd_direct.hip does, and its waves share the inputs in
// blocks of 16, straight from memory: a lane takes four consecutive inputs of its sample (16 bytes)
// and its output's column of the same four rows of W (64 bytes a row of the tile). Four blocks'
// loads are under way before the first product. The waves' sums meet in LDS, one thread finishes
// one output; with at most 16 outputs a workgroup has whole rows and takes the softmax as well.
// us in a net's inference, kernels before / here, one sample: 1024 -> 64 7.1 / 4.0, 64 -> 10 4.9 / 3.2; 32 samples,
// 512 -> 512 20.0 / 3.6. (tdh_fc_fwd does not come here, see Context::keep_f32.)
// Bound: latency, and for large layers the read of W.
//
// Reference: fully_connected_op_internal.h:13-37 (forward), softmax_layer.h:36-55.
#include <algorithm>
#include <cfloat>

#include "common.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int FCD_DEPTH = 4;   // blocks of 16 whose loads are under way together

struct FcDirectArgs {
  const float *x, *w, *bias;
  float *y;
  float *act_out;   // act(y), or null
  int act_kind;     // pointwise, or softmax (out <= 16)
  int in, out, batch, blocks;
};

// XVEC: rows of x start at multiples of 16 bytes
template <int WAVES, bool XVEC>
__global__ void __launch_bounds__(64 * WAVES) fc_fwd_direct_kernel(const FcDirectArgs a) {
  __shared__ float red[WAVES * 256 > 512 ? WAVES * 256 : 512];   // [WAVES][64][4]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int o0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  const float *xr = a.x + static_cast<size_t>(min(n0 + n, a.batch - 1)) * a.in;
  const float *wc = a.w + min(o0 + n, a.out - 1);
  const float bias = a.bias ? a.bias[min(o0 + (tid & 15), a.out - 1)] : 0.0f;
  floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int b0 = wave; b0 < a.blocks; b0 += WAVES * FCD_DEPTH) {
    float wv[FCD_DEPTH][4];
    floatx4 xv[FCD_DEPTH];
#pragma unroll
    for (int i = 0; i < FCD_DEPTH; ++i) {
      const int k = 16 * (b0 + WAVES * i) + 4 * g;
      if (b0 + WAVES * i < a.blocks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = wc[static_cast<size_t>(min(k + j, a.in - 1)) * a.out];
          wv[i][j]      = k + j < a.in ? v : 0.0f;
        }
        if (XVEC) {
          xv[i] = k < a.in ? *reinterpret_cast<const floatx4 *>(xr + k) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) xv[i][j] = k + j < a.in ? xr[k + j] : 0.0f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < FCD_DEPTH; ++i)
      if (b0 + WAVES * i < a.blocks)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i][j], xv[i][j], acc, 0, 0, 0);
  }
  // reg r of lane l: output 4 * (l / 16) + r, sample l % 16
  *reinterpret_cast<floatx4 *>(red + (wave * 64 + lane) * 4) = acc;
  __syncthreads();
  const int m = tid & 15, s = tid >> 4;   // (neighbours store neighbouring outputs of a sample)
  float v = 0.0f;
  if (tid < 256) {
#pragma unroll
    for (int k = 0; k < WAVES; ++k) v += red[(k * 64 + (m >> 2) * 16 + s) * 4 + (m & 3)];
  }
  if (tid >= 256) return;
  const int o = o0 + m;
  const bool store = o < a.out && n0 + s < a.batch;
  const size_t at  = static_cast<size_t>(n0 + s) * a.out + o;
  v += bias;
  if (store) a.y[at] = v;
  if (!a.act_out) return;
  if (a.act_kind == TDH_ACT_SOFTMAX) {
    float most = o < a.out ? v : -FLT_MAX;   // the 16 lanes of a sample
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) most = fmaxf(most, __shfl_xor(most, off, 64));
    const float e = o < a.out ? expf(v - most) : 0.0f;
    float sum     = e;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    v = e / sum;
  } else {
    v = act_apply(a.act_kind, v);
  }
  if (store) a.act_out[at] = v;
}

}  // namespace

// The line of conv_fwd_direct.hip: two rounds of workgroups' worth of products at most, and a longer
// reduction is better cut over workgroups (8192 -> 256, one sample, us before / here: 7.6 / 19.8;
// 4096 -> 4096 21 / 23). Not where a result must not depend on the kernel: the order of the sums
// is its own.
bool fc_fwd_direct_applicable(int in, int out, int batch) {
  const long tiles = static_cast<long>(ceil_div(out, 16)) * ceil_div(batch, 16);
  return !ctx().keep_f32 && in <= 2048 && tiles <= 2048 && tiles * in <= 600000;
}
bool fc_fwd_direct_applies_softmax(int in, int out, int batch) {
  return out <= 16 && fc_fwd_direct_applicable(in, out, batch);
}

int fc_fwd_direct_run(int in, int out, int batch, const float *x, const float *w, const float *bias, float *y,
                      float *act_out, int act_kind) {
  FcDirectArgs a{x, w, bias, y, act_out, act_kind, in, out, batch, ceil_div(in, 16)};
  const dim3 grid(ceil_div(out, 16), ceil_div(batch, 16));
  const bool xvec = in % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
  ProfScope prof("fc_fwd_direct", batch, out, in);
  // a wave for every four blocks, at most 16
  auto launch = [&](auto waves) {
    constexpr int NW = decltype(waves)::value;
    if (xvec)
      TDH_LAUNCH((fc_fwd_direct_kernel<NW, true>), grid, dim3(64 * NW), 0, ctx().stream, a);
    else
      TDH_LAUNCH((fc_fwd_direct_kernel<NW, false>), grid, dim3(64 * NW), 0, ctx().stream, a);
  };
  if (a.blocks > 32) launch(std::integral_constant<int, 16>());
  else if (a.blocks > 16) launch(std::integral_constant<int, 8>());
  else launch(std::integral_constant<int, 4>());
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace tdh
