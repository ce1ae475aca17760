// conv_any.hip — forward convolution and dX of any window, stride and size on the bf16 matrix cores
// with three-part operands (split_bf16.h), where no kernel built for one shape applies.
//
// Both directions are one correlation: output pixel (oy, ox) of a grid meets input row
// oy * sy + by + j * dy for the window rows j, and likewise in x; dX of a strided convolution is such a
// grid per phase (the input pixels of one remainder, with the taps that reach them), all phases in one
// launch. Columns of the product are the grid's pixels counted through rows and images, so odd
// widths leave no lane idle; a tile's input rows lie next to each other in a space where the images are
// stacked with the rows that their window reaches, and those rows are staged in LDS once per
// chunk of channels, split once, as [part][8-channel group][pixel][8 channels]. The reduction is
// taken in units of (8 channels, one tap), four of them a step of v_mfma_f32_16x16x32_bf16 (the
// quarters of a wave stand for one each), so channel counts are padded to 8 and no further. Where a
// unit's operands lie is a table in LDS, which is all that the kernel knows of the window. Columns of a
// strided input are staged by remainder, so that neighbouring lanes read neighbouring words.
// The filters come packed in parts (any_pack_kernel, a launch of 4 us): read where they lie, eight scattered
// words a unit and lane, they took longer than everything else (24 us instead of 14 for the layer below).
// Few tiles: the waves of a workgroup share the units (WK), so that a tile can be 16 to 64 pixels.
//
// us, the generic GEMM with its split sums / this kernel and its packing, forward and dX: 45x37, 21 -> 45, 5x5,
// stride 2, 19 images 21 / 18 and 37 / 19; 31x91, 3 -> 20, 7x7, stride 2, 105 images 37 / 25 and 143 / 41; 68x57,
// 9 -> 85, 5x5, 12 images dX 257 / 71; 59x56, 46 -> 3, 5x5, 69 images forward 348 / 100; 62x13, 15 -> 104, 7x7,
// 100 images dX 1249 / 187.
// Bound, few tiles: latency (stamps for the first of these, forward, 12 us in the kernel: 1.3 until the tables
// stand, 3.6 until the patch is staged, 3 to 5 for the products, 1.5 for the stores); code that runs once costs
// as much as its loads, so the loops are not unrolled further. Many tiles: LDS reads beside bf16 MFMA issue, one
// to one at 32 channels a wave.
//
// Reference: conv2d_op_internal.h:13-74 (forward), :79-158 (backward).
#include <algorithm>

#include "conv_any.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uintx4_any uintx4;

constexpr int ANY_MAX_PHASES = 4;
constexpr uint32_t ANY_NOWHERE = 0x80000000u;   // past the end of every tile's images

// A grid of output pixels and the taps that reach it.
struct AnyPhase {
  int tile0;                 // its first tile
  int count;                 // pixels of all images
  int nx, pix;               // columns, pixels of an image
  int by, bx;                // input position of output (0, 0), tap (0, 0)
  int tx, taps;
  int t0, tj, ti;            // filter position of tap (j, i): t0 + j * tj + i * ti
  int oy0, ox0;              // output position of pixel (0, 0)
  int hv;                    // input rows of one image in the stacked space
  int pw, cw;                // staged columns of a row; words a remainder's columns take
  FastDiv div_pix, div_nx, div_hv, div_pw, div_tx, div_taps;
};

struct AnyArgs {
  const float *in, *w, *bias;
  const void *wp;            // packed filters [group][tap][part][m_pad][8 channels]
  float *out, *act_out;
  int act_kind;
  ActGrad ag;
  int M, KC;
  int IH, IW, OH, OW;        // planes in memory
  int wm, wk;                // floats from one output / reduction channel of the filters to the next
  int sy, sx, dy, dx;        // steps of the input per output pixel, and per tap
  int oy_step, ox_step;      // steps of the output per pixel
  int groups;                // 8-channel groups of a chunk
  int plane;                 // words of one group's staged patch
  int m_pad;
  int bias_at;               // floats of LDS in front of the tile's bias
  int phases;
  FastDiv div_sx;
  AnyPhase p[ANY_MAX_PHASES];
};

__global__ void __launch_bounds__(256) any_pack_kernel(const AnyPack p) { any_pack_block(p, blockIdx.x); }

// One output once more in fp32, for sums that the three parts leave infinite or NaN.
__device__ __forceinline__ float any_redo(const AnyArgs &a, const AnyPhase &ph, const int m, const int img,
                                                    const int oy, const int ox) {
  float sum = 0.0f;
  for (int kc = 0; kc < a.KC; ++kc) {
    const float *w  = a.w + static_cast<size_t>(m) * a.wm + static_cast<size_t>(kc) * a.wk;
    const float *in = a.in + (static_cast<size_t>(img) * a.KC + kc) * a.IH * a.IW;
    for (int t = 0; t < ph.taps; ++t) {
      uint32_t j, i;
      ph.div_tx.divmod(t, j, i);
      const int y = oy * a.sy + ph.by + static_cast<int>(j) * a.dy, x = ox * a.sx + ph.bx + static_cast<int>(i) * a.dx;
      const bool inside = static_cast<unsigned>(y) < static_cast<unsigned>(a.IH) &&
                          static_cast<unsigned>(x) < static_cast<unsigned>(a.IW);
      const float v = inside ? in[y * a.IW + x] : 0.0f;
      sum = __builtin_fmaf(w[ph.t0 + static_cast<int>(j) * ph.tj + static_cast<int>(i) * ph.ti], v, sum);
    }
    if (sum != sum) break;
  }
  return sum;
}

// MB x NB: blocks of 16 channels x 16 pixels of a wave; WK waves share the units, 4 / WK the pixels. SUMS: workgroups behind the
// tiles add up dW's slices. (An instance of its own: the look at whether there are any, a scalar load in front of everything else, takes 0.4 us
// of 10 to 30. dX of 12x82, 10 <- 60, 3x3, 14 images 13.1 us without it, 13.5 with.)
template <int MB, int NB, int WK, bool SUMS>
__global__ void __launch_bounds__(256, 2) conv_any_kernel(const AnyArgs a, const AnySums sums) {
  constexpr int WN    = 4 / WK;
  constexpr int PIX   = WN * NB * 16;
  constexpr int ITEMS = 2;           // patch words a thread has under way
  constexpr int DEPTH = WK == 4 && MB * NB <= 6 ? 2 : 1;   // (few steps, and filters fresh from another XCD)
  extern __shared__ __align__(16) uintx4 any_lds[];
  if (SUMS && static_cast<int>(blockIdx.x) >= sums.first_x) {
    const int block = (static_cast<int>(blockIdx.x) - sums.first_x) * gridDim.y + blockIdx.y;
    if (block < sums.blocks)
      any_sums_block(sums, block, reinterpret_cast<float(*)[ANY_SUMS]>(any_lds));
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % WK, nw = wave / WK;
  const int col = lane & 15, quarter = lane >> 4;

  int pi = 0;
  while (pi + 1 < a.phases && static_cast<int>(blockIdx.x) >= a.p[pi + 1].tile0) ++pi;
  const AnyPhase &ph = a.p[pi];
  const int n0   = (static_cast<int>(blockIdx.x) - ph.tile0) * PIX;
  const int last = min(n0 + PIX, ph.count) - 1;
  const int m0   = blockIdx.y * (16 * MB);

  auto place = [&](int n, int &img, int &oy, int &ox) {
    uint32_t i, q, y, x;
    ph.div_pix.divmod(n, i, q);
    ph.div_nx.divmod(q, y, x);
    img = i; oy = y; ox = x;
  };
  int img0, oy_first, ox_first, img1, oy_last, ox_last;
  place(n0, img0, oy_first, ox_first);
  place(last, img1, oy_last, ox_last);
  const int v0    = img0 * ph.hv + oy_first * a.sy;
  const int reach = ph.taps ? (ph.taps / ph.tx - 1) * a.dy + 1 : 0;
  const int rows  = img1 * ph.hv + oy_last * a.sy + reach - v0;
  const int npix  = ph.taps ? rows * ph.pw : 0;
  const int row   = ph.cw * a.sx;    // words from one staged row to the next

  int ppix[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    int img, oy, ox;
    place(min(n0 + (nw * NB + b) * 16 + col, last), img, oy, ox);
    ppix[b] = (img * ph.hv + oy * a.sy - v0) * row + ox;
  }

  uintx4 *patch = any_lds;                                                      // [part][group][plane]
  const int part_stride = a.groups * a.plane;
  int2 *units = reinterpret_cast<int2 *>(any_lds + X3_PARTS * part_stride);     // patch word, word of the packed filters
  const int rs = a.wm < a.wk ? a.wm : a.wk;   // taps of a whole window
  for (int u = tid; u < a.groups * ph.taps; u += 256) {
    uint32_t g, t, j, i, r, c;
    ph.div_taps.divmod(u, g, t);
    ph.div_tx.divmod(t, j, i);
    a.div_sx.divmod(i * a.dx, c, r);
    const int at = ph.t0 + static_cast<int>(j) * ph.tj + static_cast<int>(i) * ph.ti;
    units[u] = make_int2(static_cast<int>(g * a.plane + j * a.dy * row + r * ph.cw + c),
                         static_cast<int>(g * rs + at) * X3_PARTS * a.m_pad);
  }

  float *bias = reinterpret_cast<float *>(any_lds) + a.bias_at;
  if (tid < 16 * MB) bias[tid] = a.bias && m0 + tid < a.M ? a.bias[m0 + tid] : 0.0f;

  floatx4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[i][b] = floatx4{};

  const float *in0 = a.in + static_cast<size_t>(img0) * a.KC * a.IH * a.IW;
  const int ihw    = a.IH * a.IW;
  const uint32_t image = static_cast<uint32_t>(a.KC) * ihw;
  // (a tile's images end before ANY_NOWHERE bytes)
  const auto desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(in0), 0, 4u * (img1 - img0 + 1) * image, 0x00027000);
  auto load = [&](const uint32_t off, const int at) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(desc, off, at, 0));
  };
  float sign = 1.0f;

  // filters on their way and where the patch's operands lie, for the wave's next DEPTH steps
  const uintx4 *wp = static_cast<const uintx4 *>(a.wp) + m0 + col;
  uintx4 ready[DEPTH][MB][X3_PARTS];
  int word[DEPTH];
  auto ask = [&](const int d, const int s, const int n_units, const uintx4 *wchunk) {
    const int u   = 4 * s + quarter;
    const bool on = u < n_units;
    int2 e = units[on ? u : 0];
    if (!on) e = make_int2(0, 0);
    word[d] = e.x;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p) {
        const uintx4 x = wchunk[static_cast<uint32_t>(e.y + p * a.m_pad + 16 * i)];
#pragma unroll
        for (int c = 0; c < 4; ++c) ready[d][i][p][c] = on ? x[c] : 0u;
      }
  };

  for (int c0 = 0; c0 < a.KC; c0 += 8 * a.groups) {
    const int left   = a.KC - c0;
    const int groups = min(a.groups, (left + 7) >> 3);
    const int n_units = groups * ph.taps, steps = (n_units + 3) >> 2;
    const uintx4 *wchunk = wp + static_cast<size_t>(c0 >> 3) * rs * X3_PARTS * a.m_pad;
    __syncthreads();   // the table is complete; everyone is done with the chunk before
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) ask(d, kw + WK * d, n_units, wchunk);
    // Item = (256 pixels, group), a pixel to a thread, ITEMS of them under way together: addresses, then all
    // loads, then their use. Words that do not exist have an offset past the end of the descriptor and
    // come back as zeros.
    const int items = ((npix + 255) >> 8) * groups;
    int slot = 0, group = 0;   // of the next item
#pragma unroll 1
    for (int t = 0; t < items; t += ITEMS) {
      uint32_t off[ITEMS];
      int at[ITEMS], first[ITEMS];
#pragma unroll
      for (int q = 0; q < ITEMS; ++q) {
        const int pe  = tid + 256 * slot;
        const bool on = t + q < items && pe < npix;
        uint32_t r, c, im, y, cd, cr;
        ph.div_pw.divmod(on ? pe : 0, r, c);
        ph.div_hv.divmod(v0 + r, im, y);
        a.div_sx.divmod(c, cd, cr);
        const int iy = static_cast<int>(y) + ph.by, ix = static_cast<int>(c) + ph.bx;
        const bool inside = on && static_cast<unsigned>(iy) < static_cast<unsigned>(a.IH) &&
                            static_cast<unsigned>(ix) < static_cast<unsigned>(a.IW);
        off[q]   = inside ? 4u * ((im - img0) * image + iy * a.IW + ix) : ANY_NOWHERE;
        at[q]    = on ? static_cast<int>(group * a.plane + r * row + cr * ph.cw + cd) : -1;
        first[q] = 8 * group;
        const bool wrap = group + 1 == groups;
        slot += wrap ? 1 : 0;
        group = wrap ? 0 : group + 1;
      }
      float v[ITEMS][8];
#pragma unroll
      for (int q = 0; q < ITEMS; ++q)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool there = first[q] + k < left;   // (the same for all lanes)
          v[q][k] = load(there ? off[q] : ANY_NOWHERE, there ? 4 * (c0 + first[q] + k) * ihw : 0);
        }
#pragma unroll
      for (int q = 0; q < ITEMS; ++q) {
        uintx4 part[X3_PARTS];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint32_t p3[X3_PARTS];
          split_pair(v[q][2 * c] * X3_SCALE, v[q][2 * c + 1] * X3_SCALE, p3);
#pragma unroll
          for (int p = 0; p < X3_PARTS; ++p) part[p][c] = p3[p];
        }
        if (at[q] >= 0)
#pragma unroll
          for (int p = 0; p < X3_PARTS; ++p) patch[p * part_stride + at[q]] = part[p];
      }
    }
    __syncthreads();

    // Wave kw takes the steps s = kw, kw + WK, .. of the chunk; the filters of a step are asked for DEPTH of
    // the wave's steps ahead, the first ones before the patch is staged.
    for (int s = kw; s < steps; s += WK * DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        if (s + WK * d < steps) {
          bf16x8 x[NB][X3_PARTS], f[MB][X3_PARTS];
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int p = 0; p < X3_PARTS; ++p)
              x[b][p] = __builtin_bit_cast(bf16x8, patch[p * part_stride + word[d] + ppix[b]]);
          const uint32_t flip = sign < 0.0f ? 0x80008000u : 0u;
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int p = 0; p < X3_PARTS; ++p) f[i][p] = __builtin_bit_cast(bf16x8, ready[d][i][p] ^ flip);
          ask(d, s + WK * (d + DEPTH), n_units, wchunk);
          constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
          floatx4 sum[MB][NB];
#pragma unroll
          for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
              for (int b = 0; b < NB; ++b)
                sum[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][pa[q]], x[b][pb[q]], q ? sum[i][b] : floatx4{}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][b][r] = __builtin_fmaf(sum[i][b][r], sign * X3_UNSCALE, acc[i][b][r]);
          sign = -sign;
        }
      }
    }
  }

  // ---- epilogue: the sums go through LDS (lane l of a block holds channels 4 * (l / 16) + r, pixel l % 16), so
  // that a thread finishes one pixel for every 256 / PIX-th channel in a loop of little code
  __syncthreads();
  float *red = reinterpret_cast<float *>(any_lds);   // [share of the units][channel][PIX]
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(kw * 16 * MB + 16 * i + 4 * quarter + r) * PIX + (nw * NB + b) * 16 + col] = acc[i][b][r];
  __syncthreads();
  const int n = n0 + tid % PIX;
  if (n > last) return;
  int img, oy, ox;
  place(n, img, oy, ox);
  const size_t ohw = static_cast<size_t>(a.OH) * a.OW;
  const int rows_left = min(16 * MB, a.M - m0), m_first = tid / PIX;
  constexpr int STEP  = 256 / PIX;
  const size_t first  = (static_cast<size_t>(img) * a.M + m0) * ohw + static_cast<size_t>(ph.oy0 + oy * a.oy_step) * a.OW +
                       ph.ox0 + ox * a.ox_step;
  // First everything that reads memory, then stores alone: a load's wait counts the stores in front of it.
  auto finite = [](const float y) { return __builtin_fabsf(y) <= 3.402823466e+38f; };
  float *mine = red + tid % PIX;   // this thread's sums: mine[m * PIX]
  float probe  = 0.0f;             // 0 * infinity and 0 * NaN are NaN
#pragma unroll 4
  for (int m = m_first; m < rows_left; m += STEP) {
    float y = mine[m * PIX];
#pragma unroll
    for (int s = 1; s < WK; ++s) y += mine[(s * 16 * MB + m) * PIX];
    probe = __builtin_fmaf(y, 0.0f, probe);
    mine[m * PIX] = y + bias[m];
  }
  if (a.ag.kind != TDH_ACT_NONE)
#pragma unroll 1
    for (int m = m_first; m < rows_left; m += 8 * STEP) {
      float g[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) g[k] = a.ag.y[first + min(m + k * STEP, rows_left - 1) * ohw];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (m + k * STEP < rows_left) mine[(m + k * STEP) * PIX] *= act_grad_factor(a.ag.kind, g[k]);
    }
  if (__builtin_expect(!(probe == 0.0f), 0)) {
#pragma unroll 1
    for (int m = m_first; m < rows_left; m += STEP) {   // those sums again
      if (finite(mine[m * PIX])) continue;
      float y = any_redo(a, ph, m0 + m, img, oy, ox);
      y += bias[m];
      if (a.ag.kind != TDH_ACT_NONE) y *= act_grad_factor(a.ag.kind, a.ag.y[first + m * ohw]);
      mine[m * PIX] = y;
    }
  }
  if (a.out)
#pragma unroll 4
    for (int m = m_first; m < rows_left; m += STEP) a.out[first + m * ohw] = mine[m * PIX];
  if (a.act_out)
#pragma unroll 1
    for (int m = m_first; m < rows_left; m += STEP) a.act_out[first + m * ohw] = act_apply(a.act_kind, mine[m * PIX]);
}

}  // namespace

namespace {

constexpr size_t ANY_LDS_MAX = 156 * 1024;   // (and the bias)

struct AnyPlan {
  bool ok;
  int mb, nb, wk;
  size_t lds_bytes, pack_bytes;
  dim3 grid;
  AnyArgs args;
  double cost;
};

// the staged rows of a tile of `pix` pixels, at most
long most_rows(const AnyArgs &a, const AnyPhase &p, int batch, int pix) {
  const int ny = p.pix / p.nx, reach = (p.taps / p.tx - 1) * a.dy + 1;
  const long rows  = std::min<long>((pix + p.nx - 2) / p.nx + 1, static_cast<long>(batch) * ny);
  const long turns = std::min<long>(batch - 1, (rows - 2 + ny) / ny);   // images begun behind the first
  return (rows - 1) * a.sy + std::max<long>(0, turns) * std::max(0, reach - a.sy) + reach;
}

// blocks of 16 channels to a workgroup: up to four, and as many to each
int any_mb(int M) {
  const int blocks = ceil_div(M, 16);
  return ceil_div(blocks, ceil_div(blocks, 4));
}
size_t any_pack_bytes(int M, int KC, int rs) {
  const int mb = any_mb(M);
  return static_cast<size_t>(ceil_div(KC, 8)) * rs * X3_PARTS * (ceil_div(M, 16 * mb) * 16 * mb) * 16;
}

AnyPlan plan_tile(const AnyArgs &base, int batch, int mb, int nb, int wk) {
  AnyPlan p{};
  p.mb = mb; p.nb = nb; p.wk = wk;
  p.args     = base;
  AnyArgs &a = p.args;
  const int pix = 4 / wk * nb * 16;
  long tiles = 0, plane = 0, most_taps = 1, items = 0;
  for (int i = 0; i < a.phases; ++i) {
    AnyPhase &ph = a.p[i];
    ph.tile0 = static_cast<int>(tiles);
    tiles += ceil_div(ph.count, pix);
    if (!ph.taps) continue;
    const long rows = most_rows(a, ph, batch, pix);
    plane     = std::max(plane, rows * ph.cw * a.sx);
    items     = std::max(items, rows * ph.pw);
    most_taps = std::max<long>(most_taps, ph.taps);
    const long images = (static_cast<long>(pix) + ph.pix - 2) / ph.pix + 1;
    if (images * a.KC * a.IH * a.IW >= (1L << 29)) return p;
  }
  const int all = ceil_div(a.KC, 8), m_tiles = ceil_div(a.M, 16 * mb);
  const long blocks = tiles * m_tiles;
  if (tiles > GRID_X_MAX || m_tiles > 65535) return p;
  auto bytes = [&](int groups) {
    return 16 * static_cast<size_t>(groups) * plane * X3_PARTS + 8 * static_cast<size_t>(groups) * most_taps;
  };
  const size_t sums = std::max<size_t>(static_cast<size_t>(wk) * 16 * mb * pix, REDUCE_GROUPS * ANY_SUMS) * sizeof(float);   // (and any_sums_block's)
  if (plane <= 0 || bytes(1) > ANY_LDS_MAX || sums > ANY_LDS_MAX) return p;
  // two workgroups a compute unit where there are that many
  const size_t room = blocks > 256 ? 78 * 1024 : ANY_LDS_MAX;
  int groups = 1;
  while (groups < all && bytes(groups + 1) <= std::max(room, bytes(1))) ++groups;
  groups      = ceil_div(all, ceil_div(all, groups));
  a.groups    = groups;
  a.plane     = static_cast<int>(plane);
  const size_t body = (std::max(bytes(groups), sums) + 15) / 16 * 16;
  a.bias_at   = static_cast<int>(body / 4);
  p.lds_bytes = body + 64 * mb;
  p.grid      = dim3(static_cast<unsigned>(tiles), m_tiles);
  a.m_pad     = m_tiles * 16 * mb;
  p.pack_bytes = any_pack_bytes(a.M, a.KC, std::min(a.wm, a.wk));
  if (p.pack_bytes >= (1u << 31)) return p;
  // Estimated us, from stamps inside the kernel and 240 shapes at every tile (10 to 1400 us; over 400 others the chosen tile
  // is 3 % off the best one, the estimate 16 %): what a workgroup waits for by itself, what the workgroups
  // of a compute unit share, and how many of them run at once.
  const double chunks = ceil_div(all, groups);
  const double steps  = chunks * ceil_div(groups * static_cast<int>(most_taps), 4 * wk);
  const double mfma   = steps * mb * nb * 6 * 16 / 2200;
  const double lds    = steps * nb * 3 * 8 * 4 / 2200;
  const double issue  = steps * (1 + 0.48 * mb) * 0.126;
  const double words  = static_cast<double>((items + 255) / 256) * all;
  const double alone  = 2.6 + 16.0 * mb * pix / 256 * 0.107 + chunks * 0.32 + words * 0.47 + std::max(mfma, steps * 0.47);
  const double shared = std::max(mfma, lds) + words * 0.32 + issue;
  const int by_lds    = static_cast<int>(160 * 1024 / p.lds_bytes);
  const int by_regs   = mb == 1 || mb * nb <= 4 ? 4 : 2;
  const int resident  = std::max(1, std::min(by_lds, by_regs));
  // (whole rounds: 520 workgroups of which a compute unit holds two take twice the time of 512. 35x42, 125 -> 82, 3x3, stride
  // 2, 11 images: 22 us estimated without, 44 in fact)
  auto round = [&](double at_once) { return std::max(alone + (at_once - 1) * shared * 0.36, at_once * shared); };
  const double whole = std::floor(static_cast<double>(blocks) / (256 * resident));
  const double left  = std::ceil(static_cast<double>(blocks) / 256 - whole * resident);
  p.cost = 0.9 + whole * round(resident) + (left > 0 ? round(left) : 0.0);
  p.ok = true;
  return p;
}

AnyPlan best_tile(const AnyArgs &base, int batch) {
  const int mb = any_mb(base.M);
  AnyPlan best{};
  static const int tiles[7][2] = {{1, 4}, {2, 4}, {4, 4}, {1, 1}, {2, 2}, {2, 1}, {4, 1}};
  for (int t = 0; t < 7; ++t) {
    const AnyPlan p = plan_tile(base, batch, mb, tiles[t][0], tiles[t][1]);
    if (p.ok && (!best.ok || p.cost < best.cost)) best = p;
  }
  return best;
}

AnyArgs forward_args(const ConvShape &c) {
  AnyArgs a{};
  a.M = c.Kc; a.KC = c.C; a.IH = c.H; a.IW = c.W; a.OH = c.OH; a.OW = c.OW;
  a.wm = c.C * c.R * c.S; a.wk = c.R * c.S;
  a.sy = c.sh; a.sx = c.sw; a.dy = c.dh; a.dx = c.dw;
  a.oy_step = a.ox_step = 1;
  a.div_sx = FastDiv(c.sw);
  a.phases = 1;
  AnyPhase &p = a.p[0];
  p.count = c.batch * c.OH * c.OW; p.nx = c.OW; p.pix = c.OH * c.OW;
  p.by = -c.ph; p.bx = -c.pw;
  p.tx = c.S; p.taps = c.R * c.S;
  p.t0 = 0; p.tj = c.S; p.ti = 1;
  p.hv = (c.OH - 1) * c.sh + (c.R - 1) * c.dh + 1;
  p.pw = (c.OW - 1) * c.sw + (c.S - 1) * c.dw + 1;
  p.cw = ceil_div(p.pw, c.sw);
  return a;
}

// dX: one grid per remainder of the input position by the stride
bool backward_args(const ConvShape &c, AnyArgs &a) {
  if (c.sh * c.sw > ANY_MAX_PHASES) return false;
  a = AnyArgs{};
  a.M = c.C; a.KC = c.Kc; a.IH = c.OH; a.IW = c.OW; a.OH = c.H; a.OW = c.W;
  a.wm = c.R * c.S; a.wk = c.C * c.R * c.S;
  a.sy = a.sx = a.dy = a.dx = 1;
  a.oy_step = c.sh; a.ox_step = c.sw;
  a.div_sx = FastDiv(1);
  for (int py = 0; py < c.sh; ++py)
    for (int px = 0; px < c.sw; ++px) {
      // input rows iy = iy0 + sh * r; iy + ph = sh * (a0 + r) + py meets the taps ky = sh * j + py, at output row a0 + r - j
      const int iy0 = ((py - c.ph) % c.sh + c.sh) % c.sh, ix0 = ((px - c.pw) % c.sw + c.sw) % c.sw;
      const int ny = iy0 < c.H ? (c.H - 1 - iy0) / c.sh + 1 : 0, nx = ix0 < c.W ? (c.W - 1 - ix0) / c.sw + 1 : 0;
      if (ny == 0 || nx == 0) continue;
      const int ty = py < c.R ? (c.R - 1 - py) / c.sh + 1 : 0, tx = px < c.S ? (c.S - 1 - px) / c.sw + 1 : 0;
      AnyPhase &p = a.p[a.phases++];
      p.count = c.batch * ny * nx; p.nx = nx; p.pix = ny * nx;
      p.taps = ty * tx;
      p.tx   = std::max(1, tx);
      p.by   = (iy0 + c.ph - py) / c.sh - (ty - 1);
      p.bx   = (ix0 + c.pw - px) / c.sw - (tx - 1);
      // (window rows in rising order of the output row: tap j is the filter row sh * (ty - 1 - j) + py)
      p.t0 = (c.sh * (ty - 1) + py) * c.S + c.sw * (tx - 1) + px;
      p.tj = -c.sh * c.S; p.ti = -c.sw;
      p.oy0 = iy0; p.ox0 = ix0;
      p.hv = std::max(1, ny - 1 + ty);
      p.pw = std::max(1, nx - 1 + tx);
      p.cw = p.pw;
    }
  return a.phases > 0;
}

// (functions of the shape alone; the last of each is kept, because a call asks for it more than once)
const AnyPlan &forward_plan(const ConvShape &c) {
  static thread_local ConvShape shape{};
  static thread_local AnyPlan plan{};
  if (!(shape == c)) {
    shape = c;
    plan  = best_tile(forward_args(c), c.batch);
  }
  return plan;
}
const AnyPlan &backward_plan(const ConvShape &c) {
  static thread_local ConvShape shape{};
  static thread_local AnyPlan plan{};
  if (!(shape == c)) {
    AnyArgs a;
    shape = c;
    plan  = c.dh == 1 && c.dw == 1 && backward_args(c, a) ? best_tile(a, c.batch) : AnyPlan{};
  }
  return plan;
}

void finish_args(AnyArgs &a) {
  for (int i = 0; i < a.phases; ++i) {
    AnyPhase &p = a.p[i];
    p.div_pix = FastDiv(p.pix); p.div_nx = FastDiv(p.nx); p.div_hv = FastDiv(p.hv); p.div_pw = FastDiv(p.pw);
    p.div_tx = FastDiv(p.tx); p.div_taps = FastDiv(std::max(1, p.taps));
  }
}

template <int MB, int NB, int WK, bool SUMS>
int launch_any_sums(const AnyPlan &p, const AnySums &sums) {
  auto kernel = conv_any_kernel<MB, NB, WK, SUMS>;
  if (p.lds_bytes > 64 * 1024) {
    static size_t raised = 0;
    if (p.lds_bytes > raised) {
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(p.lds_bytes)));
      raised = p.lds_bytes;
    }
  }
  const unsigned extra = ceil_div(sums.blocks, static_cast<int>(p.grid.y));
  TDH_LAUNCH(kernel, dim3(p.grid.x + extra, p.grid.y), dim3(256), p.lds_bytes, ctx().stream, p.args, sums);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}
template <int MB, int NB, int WK>
int launch_any_inst(const AnyPlan &p, const AnySums &sums) {
  return sums.blocks ? launch_any_sums<MB, NB, WK, true>(p, sums) : launch_any_sums<MB, NB, WK, false>(p, sums);
}
template <int MB>
int launch_any_mb(const AnyPlan &p, const AnySums &sums) {
  switch (10 * p.nb + p.wk) {
    case 14: return launch_any_inst<MB, 1, 4>(p, sums);
    case 24: return launch_any_inst<MB, 2, 4>(p, sums);
    case 44: return launch_any_inst<MB, 4, 4>(p, sums);
    case 11: return launch_any_inst<MB, 1, 1>(p, sums);
    case 22: return launch_any_inst<MB, 2, 2>(p, sums);
    case 21: return launch_any_inst<MB, 2, 1>(p, sums);
    default: return launch_any_inst<MB, 4, 1>(p, sums);
  }
}
int launch_any(const AnyPlan &p, const AnySums &sums) {
  switch (p.mb) {
    case 1: return launch_any_mb<1>(p, sums);
    case 2: return launch_any_mb<2>(p, sums);
    case 3: return launch_any_mb<3>(p, sums);
    default: return launch_any_mb<4>(p, sums);
  }
}

// the packing of a plan's filters, into scratch
int any_pack_of(const AnyPlan &p, const float *w, AnyPack *pack) {
  const AnyArgs &a = p.args;
  void *wp = nullptr;
  TDH_TRY(ws_take(p.pack_bytes, &wp));
  const int rs = std::min(a.wm, a.wk);
  pack->w = w; pack->wp = static_cast<uintx4 *>(wp);
  pack->M = a.M; pack->KC = a.KC; pack->m_pad = a.m_pad; pack->wm = a.wm; pack->wk = a.wk;
  pack->total  = ceil_div(a.KC, 8) * rs * a.m_pad;
  pack->blocks = ceil_div(pack->total, 256);
  pack->div_m = FastDiv(a.m_pad); pack->div_rs = FastDiv(rs);
  return TDH_OK;
}

int run_any(AnyPlan &p, const char *tag, int m, int n, int k, const AnyPack *packed, const AnySums *with) {
  AnyArgs &a = p.args;
  AnyPack pack;
  if (packed) {
    pack = *packed;
  } else {
    TDH_TRY(any_pack_of(p, a.w, &pack));
    ProfScope prof("conv_any_pack", 4.0 * a.M * a.KC * std::min(a.wm, a.wk) + static_cast<double>(p.pack_bytes), WORK_BYTE);
    TDH_LAUNCH(any_pack_kernel, dim3(pack.blocks), dim3(256), 0, ctx().stream, pack);
    TDH_LAUNCH_CHECK();
  }
  a.wp = pack.wp;
  AnySums sums{};
  if (with) sums = *with;
  sums.first_x = static_cast<int>(p.grid.x);
  ProfScope prof(tag, m, n, k);
  return launch_any(p, sums);
}

}  // namespace

// us of the packing launch, and of the generic kernel on `products` (rows of 32) of a dX with their split sums
constexpr double ANY_PACK_US = 5.0;
double generic_us(double products) { return 11.0 + products / 16e6; }

bool conv_any_fwd_applicable(const ConvShape &c) {
  if (ctx().keep_f32) return false;
  // Of 1600 shapes (5 to 1150 us) this takes 1215; 51 of those are over 3 % faster by the generic kernel, 34 of the others here, and
  // in all it is 97987 us there, 54671 here, 54325 with the faster one of each. 94x10, 92 -> 11, 1x1, 54 images 14 us there, 28 here.
  const AnyPlan &p = forward_plan(c);
  return p.ok && p.cost + ANY_PACK_US < gathered_gemm_us(c.Kc, c.batch * c.OH * c.OW, c.C * c.R * c.S);
}
bool conv_any_dx_applicable(const ConvShape &c, AnyOver over, double other_us) {
  if (ctx().keep_f32) return false;
  const AnyPlan &p = backward_plan(c);
  if (!p.ok) return false;
  const double pixels = static_cast<double>(c.batch) * c.H * c.W, k = static_cast<double>(c.Kc) * c.R * c.S / (c.sh * c.sw);
  switch (over) {
    // A reduction of a few steps is all staging, of which the estimate knows too little. Of the shapes that it alone would
    // take, how many are over 3 % slower here / there, and all of them in us, there / here: strided, k under 12 257 / 9
    // (2251 / 2545), 24 to 48 40 / 149 (3436 / 2812), 48 to 96 4 / 192 (5249 / 3345); stride 1, k of 24 to 48 34 / 21 (686 /
    // 731), 48 to 96 12 / 42 (973 / 845), 96 to 192 8 / 55 (1436 / 1055).
    case ANY_OVER_GENERIC:
      return k >= (c.sh * c.sw > 1 ? 48 : 96) && p.cost + ANY_PACK_US < generic_us(pixels * ceil_div(c.C, 32) * 32 * k);
    // The vector-ALU kernel is built for windows of 3 and 5. Of 1600 shapes with others, how many are over 3 % slower here / there,
    // and all of them in us, there / here: k from 1000 on and more than 4 images 66 / 397 (43746 / 26527; of the 444 that its
    // estimate leaves 47, and 26141 in all), up to 4 images 7 / 293 (16911 / 5403: a workgroup's chain of channels there), the
    // rest, which stay, 200 / 566 (15470 / 12622).
    case ANY_OVER_FIRST: {
      // (20 % rms over those 476)
      const double vector_us = 19 + 0.55 * c.Kc + pixels * c.Kc * 1e-6 * (0.39 * c.R * c.S - 7.3);
      return !(c.R == c.S && (c.R == 3 || c.R == 5)) && c.R * c.S > 9 &&
             (c.batch <= 4 || (k >= 1000 && p.cost + ANY_PACK_US < vector_us));
    }
    default: return p.cost + ANY_PACK_US < other_us;
  }
}
// (the packed filters: the same whatever the tile)
size_t conv_any_fwd_workspace_bytes(const ConvShape &c) { return ws_align(any_pack_bytes(c.Kc, c.C, c.R * c.S)); }
size_t conv_any_dx_workspace_bytes(const ConvShape &c) { return ws_align(any_pack_bytes(c.C, c.Kc, c.R * c.S)); }

int conv_any_fwd_run(const ConvShape &c, const float *x, const float *w, const float *bias, float *out, float *act_out,
                     int act_kind) {
  AnyPlan p = forward_plan(c);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_any_fwd_run: no plan for this shape");
  finish_args(p.args);
  p.args.in = x; p.args.w = w; p.args.bias = bias; p.args.out = out; p.args.act_out = act_out; p.args.act_kind = act_kind;
  return run_any(p, "conv_fwd_any_x3", c.Kc, c.batch * c.OH * c.OW, c.C * c.R * c.S, nullptr, nullptr);
}
int conv_any_dx_pack(const ConvShape &c, const float *w, AnyPack *pack) {
  const AnyPlan &p = backward_plan(c);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_any_dx_pack: no plan for this shape");
  return any_pack_of(p, w, pack);
}
bool conv_any_dx_has_room(const ConvShape &c, int blocks) {
  const AnyPlan &p = backward_plan(c);
  return p.ok && static_cast<long>(p.grid.x) + blocks <= GRID_X_MAX;
}
int conv_any_dx_run(const ConvShape &c, const float *dy, const float *w, float *dx, ActGrad ag, const AnyPack *packed,
                    const AnySums *with) {
  AnyPlan p = backward_plan(c);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_any_dx_run: no plan for this shape");
  finish_args(p.args);
  p.args.in = dy; p.args.w = w; p.args.out = dx; p.args.ag = ag;
  return run_any(p, "conv_dx_any_x3", c.C, c.batch * c.H * c.W, std::max(1, c.Kc * c.R * c.S / (c.sh * c.sw)), packed, with);
}

}  // namespace tdh
