// conv_dw_any.hip — dW and db of a convolution of any window, stride and size in fp32, where no kernel built
// for one shape applies.
//
// dW[co][ci, tap] = sum over the pixels of dY[co][p] * X[ci][input of p under tap], db one more column, of
// ones. A workgroup owns up to 64 output channels x 64 to 256 columns for one slice of the batch's pixels,
// counted through rows and images, in chunks of 64 to 256. Per chunk it stages dY, the input rows under the
// chunk for the channels that its columns belong to (stacked as conv_any.hip stacks them, columns of a
// strided input by remainder), and where each pixel's first input word lies; a column is a constant number of
// words away from that. So an input word is fetched once per chunk and not once per tap, and the loop is LDS
// reads and v_mfma_f32_16x16x4_f32: per 16 pixels a lane reads four of its channel's gradients and the four
// positions at once, and one word a column and pixel. The next 16 pixels' operands are read while these are
// multiplied. Partial sums per slice, added by the split reduction.
// Bound, few tiles: latency (a chunk's loads, the reduction behind); many: staging, and the LDS words of a column
// beside fp32 MFMA issue (46 -> 3 channels: 13 of 16 rows are padding, 51 TFLOP/s with them).
//
// Reference: conv2d_op_internal.h:79-158.
#include <algorithm>

#include "conv_any.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr uint32_t DWA_NOWHERE = 0x80000000u;   // past the end of every chunk's images

struct DwAnyArgs {
  const float *x, *dy;
  float *partial;            // [slice][M][N]
  int M, C, N, crs;          // N: crs, and one for db
  int IH, IW, ohw;
  int sy, sx, by, bx;        // input position of output (oy, ox), tap (0, 0): oy * sy + by, ox * sx + bx
  int reach;                 // input rows of a window
  int hv, pw, cw;            // rows of an image in the stacked space, staged columns, words of a remainder
  int plane;                 // words of one channel's staged rows
  int pixels, per;           // of the batch, of a slice
  int x_at, dy_at;           // words of LDS in front of the staged tensors
  FastDiv div_slices, div_n_tiles;   // of a workgroup's number where others follow: slices, then tiles of columns, then tiles of channels
  FastDiv div_pix, div_nx, div_hv, div_pw, div_sx, div_rs, div_s;
};

// MB blocks of 16 channels; NB blocks of 16 columns to each of the four waves; CH pixels a chunk. PACK: workgroups behind the
// slices' pack filters (an instance of its own, as in conv_any_kernel).
template <int MB, int NB, int CH, bool PACK>
__global__ void __launch_bounds__(256, 2) conv_dw_any_kernel(const DwAnyArgs a, const AnyPack pack) {
  if (PACK && static_cast<int>(blockIdx.x) >= pack.first) {
    any_pack_block(pack, static_cast<int>(blockIdx.x) - pack.first);
    return;
  }
  uint32_t slice = blockIdx.x, n_tile = blockIdx.y, m_tile = blockIdx.z;
  if (PACK) {
    uint32_t tile;
    a.div_slices.divmod(blockIdx.x, tile, slice);
    a.div_n_tiles.divmod(tile, m_tile, n_tile);
  }
  constexpr int DYP = CH + 4;        // (sixteen channels' 16-byte reads cover all banks)
  constexpr int ROWS = 256 / CH;     // channels of dY staged side by side
  extern __shared__ __align__(16) int dwa_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, quarter = lane >> 4;
  const int n0 = static_cast<int>(n_tile) * (64 * NB), m0 = static_cast<int>(m_tile) * (16 * MB);
  const int first = static_cast<int>(slice) * a.per, end = min(first + a.per, a.pixels);
  int *pos   = dwa_lds;                                       // [CH]
  float *dys = reinterpret_cast<float *>(dwa_lds) + a.dy_at;  // [16 * MB][DYP]
  float *xs  = reinterpret_cast<float *>(dwa_lds) + a.x_at;   // [channel][plane]
  const int row = a.cw * a.sx;

  uint32_t q0, q1, rest;
  a.div_rs.divmod(n0, q0, rest);
  a.div_rs.divmod(min(n0 + 64 * NB, a.crs) - 1, q1, rest);
  const int c_lo = min(static_cast<int>(q0), a.C - 1), channels = max(0, static_cast<int>(q1) - c_lo + 1);
  int at[NB];          // this lane's columns: words behind a pixel's position
  bool ones[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int n = n0 + (wave * NB + b) * 16 + col;
    uint32_t c, t, ky, kx, d, r;
    a.div_rs.divmod(n < a.crs ? n : n0, c, t);
    a.div_s.divmod(t, ky, kx);
    a.div_sx.divmod(kx, d, r);
    ones[b] = n >= a.crs;
    at[b]   = ones[b] ? 0 : (static_cast<int>(c) - c_lo) * a.plane + static_cast<int>(ky * row + r * a.cw + d);
  }
  auto place = [&](int n, int &img, int &oy, int &ox) {
    uint32_t i, q, y, x;
    a.div_pix.divmod(n, i, q);
    a.div_nx.divmod(q, y, x);
    img = i; oy = y; ox = x;
  };

  floatx4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[i][b] = floatx4{};

  const uint32_t ihw = a.IH * a.IW;
  for (int p0 = first; p0 < end; p0 += CH) {
    const int last = min(p0 + CH, end) - 1;
    int img0, oy, ox, img1;
    place(p0, img0, oy, ox);
    const int v0 = img0 * a.hv + oy * a.sy;
    place(last, img1, oy, ox);
    const int npix = (img1 * a.hv + oy * a.sy + a.reach - v0) * a.pw;
    const auto x_desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x + static_cast<size_t>(img0) * a.C * ihw), 0,
                                                          4u * (img1 - img0 + 1) * a.C * ihw, 0x00027000);
    const auto dy_desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.dy + static_cast<size_t>(img0) * a.M * a.ohw), 0,
                                                           4u * (img1 - img0 + 1) * a.M * a.ohw, 0x00027000);
    if (p0 > first) __syncthreads();   // everyone is done with the chunk before
    // dY: a pixel to a thread, ROWS channels side by side; and the pixel's place in the staged rows
    {
      const int p = p0 + tid % CH;
      int img;
      place(min(p, last), img, oy, ox);
      if (tid < CH) pos[tid] = (img * a.hv + oy * a.sy - v0) * row + ox;
      uint32_t i, q;
      a.div_pix.divmod(min(p, last), i, q);
      const uint32_t off = p <= last ? 4u * ((img - img0) * a.M * a.ohw + q) : DWA_NOWHERE;
#pragma unroll 1
      for (int r0 = 0; r0 < 16 * MB; r0 += 8 * ROWS) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int m = m0 + r0 + k * ROWS + tid / CH;
          v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dy_desc, m < a.M ? off + 4u * m * a.ohw : DWA_NOWHERE, 0, 0));
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (r0 + k * ROWS + tid / CH < 16 * MB) dys[(r0 + k * ROWS + tid / CH) * DYP + tid % CH] = v[k];
      }
    }
    // X: two positions of the stacked rows to a thread, eight channels' loads of both under way together
#pragma unroll 1
    for (int pe = tid; pe < npix; pe += 512) {
      uint32_t off[2];
      float *to[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool on = pe + 256 * q < npix;
        uint32_t r, c, im, y, cd, cr;
        a.div_pw.divmod(on ? pe + 256 * q : pe, r, c);
        a.div_hv.divmod(v0 + r, im, y);
        a.div_sx.divmod(c, cd, cr);
        const int iy = static_cast<int>(y) + a.by, ix = static_cast<int>(c) + a.bx;
        const bool inside = static_cast<unsigned>(iy) < static_cast<unsigned>(a.IH) &&
                            static_cast<unsigned>(ix) < static_cast<unsigned>(a.IW);
        off[q] = inside ? 4u * (((im - img0) * a.C + c_lo) * ihw + iy * a.IW + ix) : DWA_NOWHERE;
        to[q]  = xs + (r * row + cr * a.cw + cd);   // (a thread without a second position stages its first one twice)
      }
#pragma unroll 1
      for (int k0 = 0; k0 < channels; k0 += 8) {
        float v[2][8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool there = k0 + k < channels;   // (the same for all lanes)
#pragma unroll
          for (int q = 0; q < 2; ++q)
            v[q][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x_desc, there ? off[q] : DWA_NOWHERE,
                                                                                     there ? 4 * (k0 + k) * ihw : 0, 0));
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (k0 + k < channels) {
            to[0][(k0 + k) * a.plane] = v[0][k];
            to[1][(k0 + k) * a.plane] = v[1][k];
          }
      }
    }
    __syncthreads();

    const int count = last + 1 - p0, steps = (count + 15) >> 4;
    floatx4 g[2][MB];
    float v[2][NB][4];
    auto read = [&](const int to, const int s) {
      const int4 p = *reinterpret_cast<const int4 *>(pos + 16 * s + 4 * quarter);
      const int w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int i = 0; i < MB; ++i) g[to][i] = *reinterpret_cast<const floatx4 *>(dys + (16 * i + col) * DYP + 16 * s + 4 * quarter);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[to][b][j] = xs[w[j] + at[b]];
    };
    auto multiply = [&](const int from, const int s) {
      const int left = count - 16 * s - 4 * quarter;   // (past the end stands the last pixel again, which counts once)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const float x = ones[b] ? 1.0f : j < left ? v[from][b][j] : 0.0f;
#pragma unroll
          for (int i = 0; i < MB; ++i) acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[from][i][j], x, acc[i][b], 0, 0, 0);
        }
    };
    read(0, 0);
#pragma unroll 1
    for (int s = 0; s < steps; s += 2) {
      read(1, min(s + 1, steps - 1));
      multiply(0, s);
      if (s + 1 < steps) {
        read(0, min(s + 2, steps - 1));
        multiply(1, s + 1);
      }
    }
  }

  float *to = a.partial + static_cast<size_t>(slice) * a.M * a.N;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int n = n0 + (wave * NB + b) * 16 + col;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * i + 4 * quarter + r;
        if (m < a.M && n < a.N) to[static_cast<size_t>(m) * a.N + n] = acc[i][b][r];
      }
    }
}

struct DwAnyPlan {
  bool ok;
  int mb, nb, ch, slices;
  size_t lds_bytes;
  int n_tiles, m_tiles;
  DwAnyArgs args;
  double cost;
};

long most_rows(const ConvShape &c, int pix) {
  const long rows  = std::min<long>((pix + c.OW - 2) / c.OW + 1, static_cast<long>(c.batch) * c.OH);
  const long turns = std::min<long>(c.batch - 1, (rows - 2 + c.OH) / c.OH);
  return (rows - 1) * c.sh + std::max<long>(0, turns) * std::max(0, c.R - c.sh) + c.R;
}

DwAnyPlan plan_tile(const ConvShape &c, bool with_db, int nb, int ch, int rounds) {
  DwAnyPlan p{};
  DwAnyArgs &a = p.args;
  const int blocks = ceil_div(c.Kc, 16);
  p.mb = ceil_div(blocks, ceil_div(blocks, 4));
  p.nb = nb; p.ch = ch;
  a.M = c.Kc; a.C = c.C; a.crs = c.C * c.R * c.S; a.N = a.crs + (with_db ? 1 : 0);
  a.IH = c.H; a.IW = c.W; a.ohw = c.OH * c.OW;
  a.sy = c.sh; a.sx = c.sw; a.by = -c.ph; a.bx = -c.pw;
  a.reach = c.R;
  a.hv = (c.OH - 1) * c.sh + c.R;
  a.pw = (c.OW - 1) * c.sw + c.S;
  a.cw = ceil_div(a.pw, c.sw);
  const long rows = most_rows(c, ch), plane = rows * a.cw * a.sx;
  const int cols = 64 * nb, rs = c.R * c.S;
  const int channels = std::min(c.C, (cols + rs - 2) / rs + 1);
  const size_t words = ch + static_cast<size_t>(16) * p.mb * (ch + 4) + static_cast<size_t>(channels) * plane;
  a.plane = static_cast<int>(plane);
  a.dy_at = ch;
  a.x_at  = ch + 16 * p.mb * (ch + 4);
  p.lds_bytes = 4 * words;
  if (p.lds_bytes > 156 * 1024) return p;
  const long images = static_cast<long>(ch + a.ohw - 2) / a.ohw + 1;
  if (images * c.C * c.H * c.W >= (1L << 29) || images * c.Kc * a.ohw >= (1L << 29)) return p;
  const int m_tiles = ceil_div(c.Kc, 16 * p.mb), n_tiles = ceil_div(a.N, cols);
  a.pixels = c.batch * a.ohw;
  const int resident = p.lds_bytes <= 80 * 1024 ? 2 : 1;
  const int wanted   = std::max(1, 256 * resident * rounds / (m_tiles * n_tiles));
  a.per    = ceil_div(ceil_div(a.pixels, wanted), 16) * 16;
  if (a.per > ch) a.per = ceil_div(a.per, ch) * ch;
  a.per    = std::max(a.per, 64);
  p.slices = ceil_div(a.pixels, a.per);
  if (n_tiles > 65535 || m_tiles > 65535) return p;
  p.n_tiles = n_tiles; p.m_tiles = m_tiles;
  // Estimated us with the reduction, fitted to 92 shapes at every tile (8 to 460 us; over 400 others the chosen tile is 2 % off
  // the best one): what a workgroup waits for by itself, what the workgroups of a
  // compute unit share, and how many of them run at once.
  const double chunks = ceil_div(a.per, ch), steps = chunks * ceil_div(std::min(a.per, ch), 16);
  const double mfma   = steps * 4 * p.mb * nb * 32 / 2200;
  const double lds    = steps * 4 * (8 * (p.mb + 1) + 4 * nb * 9.9) / 2200;
  const double slots  = static_cast<double>((rows * a.pw + 255) / 256), dy_trips = 16.0 * p.mb * ch / 2048;
  const double stage  = chunks * (0.74 + 0.485 * slots * ceil_div(channels, 8) + 0.375 * std::ceil(dy_trips));
  const double shared = std::max(mfma, lds) + 0.025 * steps * (1 + 0.5 * nb) +
                        chunks * (0.048 * slots * channels / 8 + 0.071 * dy_trips);
  const double alone  = 2.0 + stage + std::max(mfma, steps * 0.044);
  const double at     = std::max<double>(1, std::min<double>(4, 160 * 1024 / p.lds_bytes));
  // (whole rounds: 600 workgroups of which a compute unit holds two take the time of 768)
  const double full   = static_cast<double>(p.slices) * n_tiles * m_tiles / 256;
  auto round = [&](double once) { return std::max(alone + (once - 1) * 0.82 * shared, once * shared); };
  const double whole = std::floor(full / at), left = std::ceil(full - whole * at);
  p.cost = 1.0 + whole * round(at) + (left > 0 ? round(left) : 0.0) + 4.6 + 0.665 * 4e-6 * p.slices * a.M * a.N;
  p.ok = true;
  return p;
}

// (a function of the shape alone; the last one is kept, because a call asks for it more than once)
const DwAnyPlan &make_plan(const ConvShape &c, bool with_db) {
  static thread_local ConvShape shape{};
  static thread_local bool db = false;
  static thread_local DwAnyPlan best{};
  if (shape == c && db == with_db) return best;
  shape = c; db = with_db;
  best  = DwAnyPlan{};
  static const int nbs[3] = {1, 2, 4};
  for (int nb : nbs)
    for (int ch = 64; ch <= 256; ch *= 2)
      for (int rounds = 1; rounds <= 2; ++rounds) {
        const DwAnyPlan p = plan_tile(c, with_db, nb, ch, rounds);
        if (p.ok && (!best.ok || p.cost < best.cost)) best = p;
      }
  return best;
}

template <int MB, int NB, int CH, bool PACK>
int launch_pack(const DwAnyPlan &p, const AnyPack &pack) {
  auto kernel = conv_dw_any_kernel<MB, NB, CH, PACK>;
  if (p.lds_bytes > 64 * 1024) {
    static size_t raised = 0;
    if (p.lds_bytes > raised) {
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(p.lds_bytes)));
      raised = p.lds_bytes;
    }
  }
  const dim3 grid = PACK ? dim3(pack.first + pack.blocks) : dim3(p.slices, p.n_tiles, p.m_tiles);
  TDH_LAUNCH(kernel, grid, dim3(256), p.lds_bytes, ctx().stream, p.args, pack);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}
template <int MB, int NB, int CH>
int launch_inst(const DwAnyPlan &p, const AnyPack &pack) {
  return pack.blocks ? launch_pack<MB, NB, CH, true>(p, pack) : launch_pack<MB, NB, CH, false>(p, pack);
}
template <int MB, int NB>
int launch_nb(const DwAnyPlan &p, const AnyPack &pack) {
  switch (p.ch) {
    case 64: return launch_inst<MB, NB, 64>(p, pack);
    case 128: return launch_inst<MB, NB, 128>(p, pack);
    default: return launch_inst<MB, NB, 256>(p, pack);
  }
}
template <int MB>
int launch_mb(const DwAnyPlan &p, const AnyPack &pack) {
  switch (p.nb) {
    case 1: return launch_nb<MB, 1>(p, pack);
    case 2: return launch_nb<MB, 2>(p, pack);
    default: return launch_nb<MB, 4>(p, pack);
  }
}

}  // namespace

// Against the generic GEMM with its split reduction, of which one workgroup gathers every input word of its columns by itself.
// Both us: 59x56, 46 -> 3, 5x5, 69 images 286 / 141; 48x85, 55 -> 12, 7x7, 26 images 362 / 155; 45x37, 21 -> 45, 5x5, stride 2,
// 19 images 19.4 / 17.4; 71x46, 1 -> 152, 1x1, 81 images 63 / 113 (two columns: the tile is empty), stays there, and so does
// 52x71, 24 -> 114, 3x3, stride 2, 47 images 56 / 68. Of 1600 shapes (7 to 440 us) this takes 620; 57 of those are over 3 % slower
// here, 184 of the others there, and in all it is 32378 us there, 28560 here, 28209 with the faster one of each.
// In fp32 like the GEMM, but in another order of its sums: a step that keeps to fp32 (Context::keep_f32) has the order it
// always had.
bool conv_dw_any_applicable(const ConvShape &c, bool with_db) {
  if (ctx().keep_f32 || c.dh != 1 || c.dw != 1) return false;
  const DwAnyPlan &p = make_plan(c, with_db);
  // (the estimate as it turns out at the tile it chooses: 10 % rms)
  return p.ok && 1.03 * p.cost - 2.0 < 0.87 * gathered_gemm_us(c.Kc, c.C * c.R * c.S + (with_db ? 1 : 0), c.batch * c.OH * c.OW);
}
size_t conv_dw_any_workspace_bytes(const ConvShape &c, bool with_db) {
  if (!conv_dw_any_applicable(c, with_db)) return 0;
  const DwAnyPlan &p = make_plan(c, with_db);
  return ws_align(sizeof(float) * static_cast<size_t>(p.slices) * p.args.M * p.args.N);
}
// what no plan exceeds
size_t conv_dw_any_most_bytes(const ConvShape &c, bool with_db) {
  const long columns = static_cast<long>(c.C) * c.R * c.S + (with_db ? 1 : 0);
  const long tiles   = ((columns + 255) / 256) * ceil_div(c.Kc, 64);
  const long slices  = std::min<long>((static_cast<long>(c.batch) * c.OH * c.OW + 63) / 64, std::max(1L, 1024 / tiles));
  return ws_align(sizeof(float) * static_cast<size_t>(slices) * c.Kc * columns);
}
int conv_dw_any_run(const ConvShape &c, const float *x, const float *dy, bool with_db, const float **partial, int *slices,
                    const AnyPack *pack) {
  DwAnyPlan p = make_plan(c, with_db);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_dw_any_run: no plan for this shape");
  DwAnyArgs &a = p.args;
  void *ws = nullptr;
  TDH_TRY(ws_take(sizeof(float) * static_cast<size_t>(p.slices) * a.M * a.N, &ws));
  a.x = x; a.dy = dy; a.partial = static_cast<float *>(ws);
  a.div_pix = FastDiv(a.ohw); a.div_nx = FastDiv(c.OW); a.div_hv = FastDiv(a.hv); a.div_pw = FastDiv(a.pw);
  a.div_sx = FastDiv(c.sw); a.div_rs = FastDiv(c.R * c.S); a.div_s = FastDiv(c.S);
  *partial = a.partial;
  *slices  = p.slices;
  AnyPack side{};
  if (pack) side = *pack;
  // (Behind all of the products' workgroups: those are planned as whole rounds of the chip, and a few in between
  // push as many of the last ones into a round of their own. us, dX, dW and db, packing apart / in between / behind: 13x50, 38 -> 155,
  // 7x7, stride 2, 54 images 137 / 186 / 134; 93x67, 10 -> 133, 7x7, 44 images 1106 / 1326 / 1100; 31x93, 33 -> 2, 7x7, 82 images
  // 264 / 325 / 261; 45x37, 21 -> 45, 5x5, stride 2, 19 images 34.8 / 27.7 / 27.9.)
  side.first    = p.slices * p.n_tiles * p.m_tiles;
  a.div_slices  = FastDiv(p.slices);
  a.div_n_tiles = FastDiv(p.n_tiles);
  ProfScope prof(with_db ? "conv_dw_db_any" : "conv_dw_any", a.M, a.N, a.pixels);
  switch (p.mb) {
    case 1: return launch_mb<1>(p, side);
    case 2: return launch_mb<2>(p, side);
    case 3: return launch_mb<3>(p, side);
    default: return launch_mb<4>(p, side);
  }
}

}  // namespace tdh
