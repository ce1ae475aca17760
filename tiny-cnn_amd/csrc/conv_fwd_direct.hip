// conv_fwd_direct.hip — forward convolution where the whole layer is a few small tiles (inference of one
// image, or of a few): any window, stride, dilation and padding, with the activation, the 2x2 /
// stride-2 max-pool and the activation behind it in the same launch.
//
// As a product M = output channels, N = output pixels, K = input channels x window, and nothing of
// it fills the chip: what counts is the longest chain of dependent steps and the number of
// launches. A workgroup owns 16 channels x 16 pixels (four pooling windows when the pool is in the
// launch) and its waves share K in blocks of 16, read straight from memory: the filters are rows of
// W (16 bytes a lane), the input pixel of an index k is a table entry (offset and filter position,
// built once in LDS) away from the lane's pixel. Four blocks' loads are under way before the first
// product (v_mfma_f32_16x16x4_f32, the four products of a lane's 16 bytes). The waves' sums meet in
// LDS, one thread finishes one output.
// us, kernels before / here, one image: 5x5, 3 -> 32 channels of 32x32 8.1 / 4.0, 32 -> 32 of 16x16
// 8.2 / 6.0, 3x3, 128 -> 128 of 16x16 10.4 / 7.0, 64 -> 64 of 32x32 10.2 / 4.8.
// Bound: latency (one trip to memory for the first loads, the table, the sums).
//
// Reference: conv2d_op_internal.h:13-74 (forward), maxpool_op_internal.h:17-47 (window scan:
// row by row, strict '>', start value lowest()).
#include <algorithm>
#include <cfloat>

#include "common.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int FD_K_MAX = 2048;   // the table's 16 KB, two blocks' loads of sixteen waves
constexpr int FD_DEPTH = 4;      // blocks of 16 whose loads are under way together

struct FwdDirectArgs {
  const float *x, *w, *bias;
  float *out;              // or null
  float *act_out;          // act(out), or null
  float *pool_out;         // 2x2 max of (act_out ? act(out) : out), or null
  int32_t *pool_argmax;    // flat CHW index inside the sample of the pool's input
  float *pool_act_out;     // act2(pool_out), or null
  int act_kind, pool_act_kind;
  int C, Kc, H, W, OH, OW;
  int R, S, sh, sw, dh, dw, ph, pw;
  int K, blocks;           // blocks of 16 indices
  int pixels;              // batch * OH * OW
  FastDiv div_rs, div_s;
  FastDiv div_image, div_row;  // of a pixel, or of a pooling window
};

// WVEC: rows of W start at multiples of 16 bytes
template <int WAVES, bool WVEC>
__global__ void __launch_bounds__(64 * WAVES) conv_fwd_direct_kernel(const FwdDirectArgs a) {
  extern __shared__ __align__(16) int smem[];
  int2 *tab  = reinterpret_cast<int2 *>(smem);                            // [16 * blocks]: offset, fy | fx << 8
  float *red = reinterpret_cast<float *>(smem + 2 * 16 * a.blocks);       // [WAVES][64][4]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * 16;

  // the first filters and the bias are asked for before anything else
  const float *wrow = a.w + static_cast<size_t>(min(m0 + n, a.Kc - 1)) * a.K;
  floatx4 wv[FD_DEPTH];
  auto load_filters = [&](int b0) {
#pragma unroll
    for (int i = 0; i < FD_DEPTH; ++i) {
      const int k = 16 * (b0 + WAVES * i) + 4 * g;
      if (b0 + WAVES * i < a.blocks) {
        if (WVEC) {
          wv[i] = k < a.K ? *reinterpret_cast<const floatx4 *>(wrow + k) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) wv[i][j] = k + j < a.K ? wrow[k + j] : 0.0f;
        }
      }
    }
  };
  load_filters(wave);
  const float bias = a.bias ? a.bias[min(m0 + (tid >> 4 & 15), a.Kc - 1)] : 0.0f;

  // this lane's output pixel; with a pool the four pixels of a window are neighbouring lanes
  int p = blockIdx.x * 16 + n;
  const bool on = p < a.pixels;
  p = min(p, a.pixels - 1);
  uint32_t img, rest, oy, ox;
  if (a.pool_out) {
    a.div_image.divmod(p >> 2, img, rest);
    a.div_row.divmod(rest, oy, ox);
    oy = 2 * oy + ((p >> 1) & 1);
    ox = 2 * ox + (p & 1);
  } else {
    a.div_image.divmod(p, img, rest);
    a.div_row.divmod(rest, oy, ox);
  }
  const int iy = static_cast<int>(oy) * a.sh - a.ph, ix = static_cast<int>(ox) * a.sw - a.pw;
  const float *xp = a.x + static_cast<size_t>(img) * a.C * a.H * a.W;
  const int at    = iy * a.W + ix;
  uint32_t rows = 0, cols = 0;   // the window's rows and columns that lie in the image
  for (int f = 0; f < a.R; ++f) rows |= (static_cast<unsigned>(iy + f * a.dh) < static_cast<unsigned>(a.H) ? 1u : 0u) << f;
  for (int f = 0; f < a.S; ++f) cols |= (static_cast<unsigned>(ix + f * a.dw) < static_cast<unsigned>(a.W) ? 1u : 0u) << f;

  for (int k = tid; k < 16 * a.blocks; k += 64 * WAVES) {
    uint32_t c, t, fy, fx;
    a.div_rs.divmod(k, c, t);
    a.div_s.divmod(t, fy, fx);
    // (past the end: row 31 of the window, which no window has)
    tab[k] = k < a.K ? make_int2((c * a.H + fy * a.dh) * a.W + fx * a.dw, fy | fx << 8) : make_int2(0, 31);
  }
  __syncthreads();

  floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int b0 = wave; b0 < a.blocks; b0 += WAVES * FD_DEPTH) {
    float xv[FD_DEPTH][4];
#pragma unroll
    for (int i = 0; i < FD_DEPTH; ++i) {
      const int k = 16 * (b0 + WAVES * i) + 4 * g;
      if (b0 + WAVES * i < a.blocks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int2 e  = tab[k + j];
          const bool in = (rows >> (e.y & 31) & cols >> (e.y >> 8)) & 1u;
          const float v = xp[in ? at + e.x : 0];
          xv[i][j]      = in ? v : 0.0f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < FD_DEPTH; ++i)
      if (b0 + WAVES * i < a.blocks)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i][j], xv[i][j], acc, 0, 0, 0);
    load_filters(b0 + WAVES * FD_DEPTH);
  }
  // reg r of lane l: channel 4 * (l / 16) + r, pixel l % 16
  *reinterpret_cast<floatx4 *>(red + (wave * 64 + lane) * 4) = acc;
  __syncthreads();
  if (tid >= 256) return;
  const int m = tid >> 4, co = m0 + m;
  float v = 0.0f;
#pragma unroll
  for (int s = 0; s < WAVES; ++s) v += red[(s * 64 + (m >> 2) * 16 + n) * 4 + (m & 3)];
  const bool store = on && co < a.Kc;
  const int ohw    = a.OH * a.OW, pix = oy * a.OW + ox;
  const size_t o   = (static_cast<size_t>(img) * a.Kc + co) * ohw + pix;
  v += bias;
  if (a.out && store) a.out[o] = v;
  if (a.act_out) {
    v = act_apply(a.act_kind, v);
    if (store) a.act_out[o] = v;
  }
  if (a.pool_out) {
    const float w4[4] = {v, __shfl_xor(v, 1), __shfl_xor(v, 2), __shfl_xor(v, 3)};
    float best = -FLT_MAX;
    int sel    = -1;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (w4[k] > best) {
        best = w4[k];
        sel  = k;
      }
    if (store && !(n & 3)) {
      const size_t q = (static_cast<size_t>(img) * a.Kc + co) * (ohw >> 2) + (oy >> 1) * (a.OW >> 1) + (ox >> 1);
      a.pool_out[q]    = best;
      a.pool_argmax[q] = sel < 0 ? 0 : co * ohw + pix + (sel >> 1) * a.OW + (sel & 1);
      if (a.pool_act_out) a.pool_act_out[q] = act_apply(a.pool_act_kind, best);
    }
  }
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

// Up to two rounds of workgroups' worth of products (a tile of 16 x 16 and a block of 16 indices is
// four instructions; 16x16 images, 32 -> 32 channels, 5x5, us before / here: 512 tiles 16 / 9, 1024
// tiles 16 / 16) and eight workgroups a compute unit, whose prologue is what the shortest
// reductions consist of (32x32 images, 3 -> 32 channels, 5x5: 2048 tiles 8.4 / 6.5). A longer reduction
// is better cut over workgroups (9x9, 128 -> 128, 5x5, one image: 11 / 16). Not where a
// result must not depend on the kernel: the order of the sums is its own.
bool conv_fwd_direct_applicable(int batch, int C, int Kc, int H, int W, int OH, int OW, int R, int S) {
  const long pixels = static_cast<long>(batch) * OH * OW, k = static_cast<long>(C) * R * S;
  const long tiles  = ceil_div(Kc, 16) * ((pixels + 15) / 16);
  return !ctx().keep_f32 && pixels <= 32768 && tiles <= 2048 && tiles * k <= 600000 && k <= FD_K_MAX && R <= 31 && S <= 31 &&
         static_cast<long>(C) * H * W < (1L << 30);
}

int conv_fwd_direct_run(int batch, int C, int Kc, const float *x, const float *w, const float *bias, float *out, int H, int W,
                        int OH, int OW, int R, int S, int sh, int sw, int dh, int dw, int ph, int pw, float *act_out,
                        int act_kind, const PoolFuse *pool) {
  if (pool && ((OH | OW) & 1))
    return set_error(TDH_ERR_INVALID, "conv_fwd_direct_run: a fused 2x2 pool needs even output sizes");
  FwdDirectArgs a{};
  a.x = x; a.w = w; a.bias = bias; a.out = out; a.act_out = act_out; a.act_kind = act_kind;
  if (pool) {
    a.pool_out = pool->out; a.pool_argmax = pool->argmax;
    a.pool_act_out = pool->act_out; a.pool_act_kind = pool->act_kind;
  }
  a.C = C; a.Kc = Kc; a.H = H; a.W = W; a.OH = OH; a.OW = OW;
  a.R = R; a.S = S; a.sh = sh; a.sw = sw; a.dh = dh; a.dw = dw; a.ph = ph; a.pw = pw;
  a.K      = C * R * S;
  a.blocks = ceil_div(a.K, 16);
  a.pixels = batch * OH * OW;
  a.div_rs = FastDiv(R * S);
  a.div_s  = FastDiv(S);
  a.div_image = FastDiv(pool ? OH / 2 * (OW / 2) : OH * OW);
  a.div_row   = FastDiv(pool ? OW / 2 : OW);
  const dim3 grid(ceil_div(a.pixels, 16), ceil_div(Kc, 16));
  const bool wvec = a.K % 4 == 0 && aligned16(w);
  ProfScope prof(pool ? "conv_fwd_direct_pool" : "conv_fwd_direct", Kc, a.pixels, a.K);
  // a wave for every four blocks, at most 16
  auto launch = [&](auto waves) {
    constexpr int NW  = decltype(waves)::value;
    const size_t lds  = sizeof(int2) * 16 * a.blocks + sizeof(float) * NW * 256;
    if (wvec)
      TDH_LAUNCH((conv_fwd_direct_kernel<NW, true>), grid, dim3(64 * NW), lds, ctx().stream, a);
    else
      TDH_LAUNCH((conv_fwd_direct_kernel<NW, false>), grid, dim3(64 * NW), lds, ctx().stream, a);
  };
  if (a.blocks > 32) launch(std::integral_constant<int, 16>());
  else if (a.blocks > 16) launch(std::integral_constant<int, 8>());
  else launch(std::integral_constant<int, 4>());
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace tdh
