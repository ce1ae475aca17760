// conv_bwd_direct.hip — dX, dW and db of a convolution that is a few small tiles, as one launch: any window,
// stride and padding.
//
// What conv_fwd_direct.hip says about the forward pass holds here: nothing of such a layer fills the
// chip, so launches and the longest dependent chain count. Workgroups of 16 x 16 results, the
// waves share the reduction in blocks of 16 indices, operands straight from memory, four blocks'
// loads under way before the first v_mfma_f32_16x16x4_f32, the waves' sums added in LDS.
//   dX: 16 input channels x 16 input pixels, reduction over (output channel, tap); where a tap's
//       output pixel lies is a table entry away from the lane's pixel (strides: a tap counts for
//       the pixels whose remainder it matches, and floor(fy / stride) rows back).
//   dW: 16 output channels x 16 of the C*R*S columns, reduction over the output pixels of the
//       batch; the bias gradient is one more column, of ones.
// us for dX + dW + db, launches before (3 to 7) / here: 3x3, 12 -> 17 channels of 31x12, one image 19.6 /
// 5.5; 5x5, 32 -> 32 of 16x16, one image 24.6 / 8.3; 3x3, 64 -> 64 of 32x32, one image 37.4 / 13.1; 5x5,
// stride 2, 25 -> 7 of 14x12, 19 images 23.9 / 9.8.
// Bound: latency.
//
// Reference: conv2d_grad_op.h:52-106 by way of conv2d_op_internal.h:79-158.
#include <algorithm>

#include "common.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BD_K_MAX = 2048;   // dX: the table's 32 KB
constexpr int BD_DEPTH = 4;      // blocks of 16 whose loads are under way together

struct BwdDirectArgs {
  const float *x, *w, *dy;
  float *dx, *dw, *db;     // any of them null
  ActGrad ag;              // of dx
  int accumulate;          // dw, db
  int C, Kc, H, W, OH, OW;
  int R, S, sh, sw, ph, pw;
  int dx_pixels, dx_tiles, dx_blocks;    // input pixels of the batch, tiles along them, workgroups
  int dx_k, dx_kblocks;                  // reduction of dX
  int pixels, dw_cols, dw_tiles, dw_kblocks;
  FastDiv div_rs, div_s, div_dxtiles, div_hw, div_w, div_dwtiles, div_ohw, div_ow, div_sh, div_sw;
};

template <int WAVES>
__device__ __forceinline__ float add_waves(float *red, const floatx4 &acc, const int wave, const int lane, const int m,
                                           const int n) {
  // reg r of lane l: row 4 * (l / 16) + r, column l % 16
  *reinterpret_cast<floatx4 *>(red + (wave * 64 + lane) * 4) = acc;
  __syncthreads();
  float v = 0.0f;
  if (threadIdx.x < 256) {
#pragma unroll
    for (int s = 0; s < WAVES; ++s) v += red[(s * 64 + (m >> 2) * 16 + n) * 4 + (m & 3)];
  }
  return v;
}

template <int WAVES>
__device__ __forceinline__ void direct_dx(const BwdDirectArgs &a, int4 *tab, float *red, const int block) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  uint32_t mt, pt;
  a.div_dxtiles.divmod(block, mt, pt);
  const int m0 = mt * 16;
  const int p0 = pt * 16 + n;
  const bool on = p0 < a.dx_pixels;
  uint32_t img, rest, iy, ix;
  a.div_hw.divmod(min(p0, a.dx_pixels - 1), img, rest);
  a.div_w.divmod(rest, iy, ix);
  // the taps that reach this pixel, and the output pixel of tap (0, 0)
  uint32_t rows = 0, cols = 0, by, ry, bx, rx;
  a.div_sh.divmod(iy + a.ph, by, ry);
  a.div_sw.divmod(ix + a.pw, bx, rx);
  for (int f = 0; f < a.R; ++f) {
    uint32_t q, r;
    a.div_sh.divmod(f, q, r);
    const int oy = static_cast<int>(by) - static_cast<int>(q);
    rows |= (r == ry && static_cast<unsigned>(oy) < static_cast<unsigned>(a.OH) ? 1u : 0u) << f;
  }
  for (int f = 0; f < a.S; ++f) {
    uint32_t q, r;
    a.div_sw.divmod(f, q, r);
    const int ox = static_cast<int>(bx) - static_cast<int>(q);
    cols |= (r == rx && static_cast<unsigned>(ox) < static_cast<unsigned>(a.OW) ? 1u : 0u) << f;
  }
  const float *dyp = a.dy + static_cast<size_t>(img) * a.Kc * a.OH * a.OW;
  const int at     = static_cast<int>(by) * a.OW + static_cast<int>(bx);

  const int rs = a.R * a.S;
  for (int k = tid; k < 16 * a.dx_kblocks; k += 64 * WAVES) {
    uint32_t co, t, fy, fx;
    a.div_rs.divmod(k, co, t);
    a.div_s.divmod(t, fy, fx);
    // (past the end: row 31 of the window, which no window has)
    tab[k] = k < a.dx_k ? make_int4((static_cast<int>(co) * a.OH - static_cast<int>(a.div_sh.div(fy))) * a.OW -
                                        static_cast<int>(a.div_sw.div(fx)),
                                    fy | fx << 8, co * a.C * rs + t, 0)
                        : make_int4(0, 31, 0, 0);
  }
  __syncthreads();

  const float *wr = a.w + static_cast<size_t>(min(m0 + n, a.C - 1)) * rs;
  floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int b0 = wave; b0 < a.dx_kblocks; b0 += WAVES * BD_DEPTH) {
    float wv[BD_DEPTH][4], yv[BD_DEPTH][4];
#pragma unroll
    for (int i = 0; i < BD_DEPTH; ++i)
      if (b0 + WAVES * i < a.dx_kblocks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int4 e  = tab[16 * (b0 + WAVES * i) + 4 * g + j];
          const bool in = (rows >> (e.y & 31) & cols >> (e.y >> 8)) & 1u;
          const float v = dyp[in ? at + e.x : 0];
          wv[i][j]      = e.y == 31 ? 0.0f : wr[e.z];   // (past the end: 0 times an infinite weight is NaN)
          yv[i][j]      = in ? v : 0.0f;
        }
      }
#pragma unroll
    for (int i = 0; i < BD_DEPTH; ++i)
      if (b0 + WAVES * i < a.dx_kblocks)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i][j], yv[i][j], acc, 0, 0, 0);
  }
  const int c  = m0 + (tid >> 4 & 15);
  const bool store = tid < 256 && on && c < a.C;
  const size_t o   = ((static_cast<size_t>(img) * a.C + c) * a.H + iy) * a.W + ix;
  float factor     = 1.0f;
  if (store && a.ag.kind != TDH_ACT_NONE) factor = act_grad_factor(a.ag.kind, a.ag.y[o]);
  const float v = add_waves<WAVES>(red, acc, wave, lane, tid >> 4, n);
  if (store) a.dx[o] = v * factor;
}

// QUAD: four output pixels in a row lie in one row of the image, 16-byte aligned
template <int WAVES, bool QUAD>
__device__ __forceinline__ void direct_dw(const BwdDirectArgs &a, float *red, const int block) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  uint32_t mt, nt;
  a.div_dwtiles.divmod(block, mt, nt);
  const int m0 = mt * 16, col = nt * 16 + n;
  const int rs = a.R * a.S, crs = a.C * rs, ohw = a.OH * a.OW, hw = a.H * a.W;
  uint32_t ci, t, fy, fx;
  a.div_rs.divmod(min(col, crs - 1), ci, t);
  a.div_s.divmod(t, fy, fx);
  const int y0 = static_cast<int>(fy) - a.ph, x0 = static_cast<int>(fx) - a.pw;
  const float *xc  = a.x + static_cast<size_t>(ci) * hw;
  const float *dyc = a.dy + static_cast<size_t>(min(m0 + n, a.Kc - 1)) * ohw;
  const bool inner = col < crs;
  const float rim  = col == crs ? 1.0f : 0.0f;   // the bias gradient's column
  const int m = tid >> 4 & 15, co = m0 + m;
  float *dst  = nullptr;
  if (tid < 256 && co < a.Kc) {
    if (inner && a.dw) dst = a.dw + static_cast<size_t>(co) * crs + col;
    if (col == crs && a.db) dst = a.db + co;
  }
  const float before = dst && a.accumulate ? *dst : 0.0f;

  floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int b0 = wave; b0 < a.dw_kblocks; b0 += WAVES * BD_DEPTH) {
    floatx4 av[BD_DEPTH];
    float bv[BD_DEPTH][4];
#pragma unroll
    for (int i = 0; i < BD_DEPTH; ++i)
      if (b0 + WAVES * i < a.dw_kblocks) {
        const int p = 16 * (b0 + WAVES * i) + 4 * g;
        uint32_t img = 0, rest = 0, oy = 0, ox = 0;
        if (QUAD) {
          a.div_ohw.divmod(min(p, a.pixels - 4), img, rest);
          a.div_ow.divmod(rest, oy, ox);
          const floatx4 v = *reinterpret_cast<const floatx4 *>(dyc + static_cast<size_t>(img) * a.Kc * ohw + rest);
          av[i] = p < a.pixels ? v : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (!QUAD) {
            a.div_ohw.divmod(min(p + j, a.pixels - 1), img, rest);
            a.div_ow.divmod(rest, oy, ox);
            const float v = dyc[static_cast<size_t>(img) * a.Kc * ohw + rest];
            av[i][j]      = p + j < a.pixels ? v : 0.0f;
          }
          const int iy  = static_cast<int>(oy) * a.sh + y0, ix = static_cast<int>(ox + (QUAD ? j : 0)) * a.sw + x0;
          const bool in = inner && p + j < a.pixels && static_cast<unsigned>(iy) < static_cast<unsigned>(a.H) &&
                          static_cast<unsigned>(ix) < static_cast<unsigned>(a.W);
          const float v = xc[in ? static_cast<size_t>(img) * a.C * hw + iy * a.W + ix : 0];
          bv[i][j]      = in ? v : rim;
        }
      }
#pragma unroll
    for (int i = 0; i < BD_DEPTH; ++i)
      if (b0 + WAVES * i < a.dw_kblocks)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i][j], bv[i][j], acc, 0, 0, 0);
  }
  const float v = add_waves<WAVES>(red, acc, wave, lane, tid >> 4, n);
  if (dst) *dst = a.accumulate ? before + v : v;
}

template <int WAVES, bool QUAD>
__global__ void __launch_bounds__(64 * WAVES) conv_bwd_direct_kernel(const BwdDirectArgs a) {
  extern __shared__ __align__(16) int smem[];
  float *red = reinterpret_cast<float *>(smem);                    // [WAVES][64][4]
  int4 *tab  = reinterpret_cast<int4 *>(smem + WAVES * 256);       // [16 * dx_kblocks]
  const int id = blockIdx.x;
  if (id < a.dx_blocks)
    direct_dx<WAVES>(a, tab, red, id);
  else
    direct_dw<WAVES, QUAD>(a, red, id - a.dx_blocks);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

// The lines of conv_fwd_direct.hip, and 2048 output pixels at most: dW gathers its columns pixel by
// pixel, 16 waves to a compute unit, and from there on that takes as long as the launches it saves
// (us before / here: 16x16 images, 32 -> 32, 5x5, 8 images 19.5 / 18.0; 32x32, 3 -> 32, 4 images 22.5 /
// 27.9). dX has no use for that many waves: with them 512 tiles of it at most (42x11, stride 2, 60 -> 13,
// 14 images, 1620 tiles: 27.7 / 28.0). Not where a result must not depend on the kernel: the order of the sums is its own.
bool conv_bwd_direct_applicable(int batch, int C, int Kc, int H, int W, int OH, int OW, int R, int S) {
  const long in_pixels = static_cast<long>(batch) * H * W, pixels = static_cast<long>(batch) * OH * OW;
  const long k = static_cast<long>(Kc) * R * S, cols = static_cast<long>(C) * R * S + 1;
  const long dx_tiles = ceil_div(C, 16) * ((in_pixels + 15) / 16), dw_tiles = ceil_div(Kc, 16) * ((cols + 15) / 16);
  return !ctx().keep_f32 && R <= 31 && S <= 31 && in_pixels <= 32768 &&
         k <= BD_K_MAX && dx_tiles <= (pixels > 512 ? 512 : 2048) && dx_tiles * k <= 600000 && pixels <= 2048 && dw_tiles <= 2048 &&
         dw_tiles * pixels <= 600000 && static_cast<long>(batch) * C * H * W < (1L << 30) && pixels * Kc < (1L << 30);
}

int conv_bwd_direct_run(int batch, int C, int Kc, const float *x, const float *w, const float *dy, float *dx, float *dw,
                        float *db, int H, int W, int OH, int OW, int R, int S, int sh, int sw, int ph, int pw,
                        int accumulate, ActGrad dx_act) {
  BwdDirectArgs a{};
  a.x = x; a.w = w; a.dy = dy; a.dx = dx; a.dw = dw; a.db = db; a.ag = dx_act; a.accumulate = accumulate;
  a.C = C; a.Kc = Kc; a.H = H; a.W = W; a.OH = OH; a.OW = OW;
  a.R = R; a.S = S; a.sh = sh; a.sw = sw; a.ph = ph; a.pw = pw;
  a.dx_pixels  = batch * H * W;
  a.dx_tiles   = ceil_div(a.dx_pixels, 16);
  a.dx_blocks  = dx ? a.dx_tiles * ceil_div(C, 16) : 0;
  a.dx_k       = Kc * R * S;
  a.dx_kblocks = dx ? ceil_div(a.dx_k, 16) : 0;
  a.pixels     = batch * OH * OW;
  a.dw_cols    = C * R * S + (db ? 1 : 0);
  a.dw_tiles   = ceil_div(a.dw_cols, 16);
  a.dw_kblocks = ceil_div(a.pixels, 16);
  a.div_rs = FastDiv(R * S); a.div_s = FastDiv(S);
  a.div_dxtiles = FastDiv(a.dx_tiles); a.div_hw = FastDiv(H * W); a.div_w = FastDiv(W);
  a.div_dwtiles = FastDiv(a.dw_tiles); a.div_ohw = FastDiv(OH * OW); a.div_ow = FastDiv(OW);
  a.div_sh = FastDiv(sh); a.div_sw = FastDiv(sw);
  const int blocks = a.dx_blocks + (dw || db ? a.dw_tiles * ceil_div(Kc, 16) : 0);
  if (blocks == 0) return TDH_OK;
  const bool quad = OW % 4 == 0 && aligned16(dy);
  const int longest = std::max(a.dx_kblocks, dw || db ? a.dw_kblocks : 0);
  ProfScope prof("conv_bwd_direct", 2.0 * ((dx ? static_cast<double>(a.dx_pixels) * C * Kc * R * S / (sh * sw) : 0.0) +
                                           (dw || db ? static_cast<double>(a.pixels) * Kc * a.dw_cols : 0.0)), WORK_FLOP);
  // a wave for every four blocks of the longer reduction, at most 16
  auto launch = [&](auto waves) {
    constexpr int NW = decltype(waves)::value;
    const size_t lds = sizeof(float) * NW * 256 + sizeof(int4) * 16 * a.dx_kblocks;
    if (quad)
      TDH_LAUNCH((conv_bwd_direct_kernel<NW, true>), dim3(blocks), dim3(64 * NW), lds, ctx().stream, a);
    else
      TDH_LAUNCH((conv_bwd_direct_kernel<NW, false>), dim3(blocks), dim3(64 * NW), lds, ctx().stream, a);
  };
  if (longest > 32) launch(std::integral_constant<int, 16>());
  else if (longest > 16) launch(std::integral_constant<int, 8>());
  else launch(std::integral_constant<int, 4>());
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace tdh
