// conv_fwd_small.hip — forward convolution with few input channels (Cin*KH*KW <= 96: the first
// layer of an image net), any stride and dilation, optionally with the layers behind it:
// a pointwise activation, a 2x2/stride-2 max-pool and the activation behind that pool.
//
//   y[img][co][oy][ox] = b[co] + sum_{ci,ky,kx} W[co][ci][ky][kx] * x[img][ci][oy*sh+ky*dh-ph][ox*sw+kx*dw-pw]
//
// As a product: M = Cout, N = output pixels, K = Cin*KH*KW (75 for 3 channels and 5x5). K is so
// short that a lane keeps its whole column of the filter matrix in registers. A workgroup owns
// a band of output rows of one image and 32 output channels; it stages the input patch under
// the band in LDS (zero-filled where the window leaves the image) and the filter slice, and a
// wave then computes tiles of 2 rows x 32 columns x 32 channels, one accumulator block per row:
// per k-step and row one LDS read at patch[pixel] + offset(k) and one v_mfma_f32_32x32x2_f32
// (A lane = (co, k), B lane = (pixel, k); indices past the last tap are zeros on both sides). A lane so
// holds both rows of its column, and two neighbours share a 2x2 pooling window: they exchange the values of
// two channels and pool one each. The max-pool (with its argmax record and the activation behind it) costs
// those lane swaps in the epilogue and needs no kernel or pass over y of its own. Stores of y are whole
// rows of 32 floats per channel.
//
// Reference: conv2d_op_internal.h:13-74 (forward), maxpool_op_internal.h:17-47 (window scan:
// row by row, strict '>', start value lowest()).
#include <algorithm>
#include <cfloat>

#include "conv_pack.h"
#include "gemm_mfma.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int intx4 __attribute__((ext_vector_type(4)));

struct FwdSmallArgs {
  const float *x, *w, *bias;
  float *out;
  float *act_out;          // act(out), or null
  float *pool_out;         // 2x2 max of (act_out ? act(out) : out), or null
  int32_t *pool_argmax;    // flat CHW index inside the sample of the pool's input
  float *pool_act_out;     // act2(pool_out), or null
  int act_kind, pool_act_kind;
  int C, Kc, H, W, OH, OW;
  int R, S, sh, sw, dh, dw, ph, pw;
  int band, bands, col_tiles;
  int rows_in, pitch, plane;
  int crs, x_floats;
  FastDiv div_pitch, div_rows_in, div_col_tiles;
  int co_step;               // output channels of a workgroup
  int batch, workgroups;     // of the convolution
  int packers, pack_threads; // workgroups in front of them
  int first;                 // of a launch's workgroups
};

// Workgroups in front of the convolution's own pack filters that later layers read: in a net whose
// weights may have been written since the last call that is a launch less, and beside four workgroups of the convolution on a CU
// it costs little: first convolution of the CIFAR-10-shape net at batch 128 15.0 us, with 590 KB of
// filters 15.8 (a launch of its own 5.0). No more than 192: a thread of them writes several pieces rather than 500 workgroups.
constexpr int FWD_SMALL_PACKERS = 192;
struct NoPacks {};
template <class Packs>
__device__ __forceinline__ bool fwd_small_packs(const FwdSmallArgs &a, const Packs &packs, const int id) {
  if constexpr (std::is_same_v<Packs, PackJobs>) {
    if (id >= a.packers) return false;
    // (whole pieces of a job's 256 threads: of three waves two work)
    const int threads = blockDim.x < 256 ? 128 : 256;
    if (static_cast<int>(threadIdx.x) >= threads) return true;
    const int step = a.packers * threads;
    for (int t = id * threads + threadIdx.x; t < a.pack_threads; t += step) pack_any(packs, t);
    return true;
  }
  return false;
}

// the value of lane l ^ 1 (a swap inside lane pairs, done by the DPP path of a move)
__device__ __forceinline__ float lane_xor1(const float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}

// act_apply on the values of an accumulator block; the choice is made once, not per value
template <int N>
__device__ __forceinline__ void act_apply_each(const int kind, float (&v)[N]) {
  switch (kind) {
    case TDH_ACT_RELU:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = act_apply(TDH_ACT_RELU, v[i]);
      break;
    case TDH_ACT_TANH:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = act_apply(TDH_ACT_TANH, v[i]);
      break;
    case TDH_ACT_SIGMOID:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = act_apply(TDH_ACT_SIGMOID, v[i]);
      break;
    default: break;
  }
}

// Stages the input patch under the band (zero-filled where the window leaves the image), the
// filter slice, the bias and the patch offset of every k into LDS: all loads of a thread are
// issued before its first store.
template <int NS>
__device__ __forceinline__ void fwd_small_stage(const FwdSmallArgs &a, float *xs, float *ws, float *bs, int *offs,
                                                const int img, const int co0, const int oy0, const int tid,
                                                const int nthr) {
  {
    const int iy0     = oy0 * a.sh - a.ph;
    const int x_total = a.C * a.rows_in * a.pitch;
    constexpr int DEPTH = 8;
    // the filter slice as 16-byte words, issued in front of the patch and stored behind it: one
    // trip to memory covers both (a thread's eight words hold 32 rows of up to 128 taps)
    const int w_total = 32 * a.crs;
    const int w_valid = min(32, a.Kc - co0) * a.crs;
    const float *wsrc = a.w + static_cast<size_t>(co0) * a.crs;
    const bool wvec   = (reinterpret_cast<uintptr_t>(wsrc) & 15u) == 0 && (w_valid & 3) == 0 &&
                      w_total <= 4 * DEPTH * nthr;
    floatx4 wq[DEPTH];
    if (wvec) {
#pragma unroll
      for (int k = 0; k < DEPTH; ++k)  // (every load is issued: a word past the slice repeats its last one)
        wq[k] = *reinterpret_cast<const floatx4 *>(wsrc + min(4 * (tid + k * nthr), w_valid - 4));
    }
    for (int e0 = tid; e0 < x_total; e0 += DEPTH * nthr) {
      float xv[DEPTH];
      int xo[DEPTH];
#pragma unroll
      for (int k = 0; k < DEPTH; ++k) {
        const int e = e0 + k * nthr;
        xv[k] = 0.0f;
        xo[k] = -1;
        if (e < x_total) {
          const int rr = a.div_pitch.div(e), cx = e - rr * a.pitch;
          const int ci = a.div_rows_in.div(rr), r = rr - ci * a.rows_in;
          const int iy = iy0 + r, ix = cx - a.pw;
          xo[k] = ci * a.plane + r * a.pitch + cx;
          if (iy >= 0 && iy < a.H && ix >= 0 && ix < a.W)
            xv[k] = a.x[(static_cast<size_t>(img * a.C + ci) * a.H + iy) * a.W + ix];
        }
      }
#pragma unroll
      for (int k = 0; k < DEPTH; ++k)
        if (xo[k] >= 0) xs[xo[k]] = xv[k];
    }
    if (wvec) {
#pragma unroll
      for (int k = 0; k < DEPTH; ++k) {
        const int e = 4 * (tid + k * nthr);
        const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
        if (e < w_total) *reinterpret_cast<floatx4 *>(ws + e) = e < w_valid ? wq[k] : zero4;
      }
    }
    for (int e0 = wvec ? w_total : tid; e0 < w_total; e0 += DEPTH * nthr) {
      float wv[DEPTH];
#pragma unroll
      for (int k = 0; k < DEPTH; ++k) {
        const int e = e0 + k * nthr;
        wv[k] = e < w_valid ? wsrc[e] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < DEPTH; ++k) {
        const int e = e0 + k * nthr;
        if (e < w_total) ws[e] = wv[k];
      }
    }
    if (tid < 32) {
      const int m = co0 + tid;
      bs[tid]     = (a.bias && m < a.Kc) ? a.bias[m] : 0.0f;
    }
    if (tid < 2 * NS) {
      int o = -1;
      if (tid < a.crs) {
        const int rs = a.R * a.S;
        const int ci = tid / rs, tap = tid - ci * rs;
        const int ky = tap / a.S, kx = tap - ky * a.S;
        o = ci * a.plane + ky * a.dh * a.pitch + kx * a.dw;
      }
      offs[(tid & 1) * NS + (tid >> 1)] = max(o, 0);
    }
  }
}

// Stores of a tile that has every channel and every pixel of its 32 x 2 x 32, or less: a value's address is
// a scalar offset of the tile plus one offset of the lane that is computed once, and what does not exist
// has a lane offset behind the buffer (guards, 64-bit addresses and saved exec masks were most of 25 vector
// instructions per MFMA).
constexpr uint32_t FWD_SMALL_NOWHERE = 0xfffffff0u;   // past the end of any 32 planes
template <bool STREAM, class T>
__device__ __forceinline__ void fwd_small_store(const T v, const __amdgpu_buffer_rsrc_t to, const uint32_t lane, const uint32_t tile) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), to, lane, tile, STREAM ? 2 : 0);
}

// PLAIN: the channels are a multiple of 32 and each activation is relu or none.
// Registers are what keeps workgroups from a CU: with patch offsets and biases read again per tile instead of held, and
// patch values a group of four steps ahead instead of eight, 176 -> 112 of them for 5x5 on three channels and two -> four
// workgroups. The kernel's us for 3 -> 32 channels, 5x5, 32x32 with a pool and relu behind, batch 1000, y past the caches: 101 -> 79; of three to four workgroups
// and the stores above, 3 -> 64 channels, 3x3, 128x128, batch 64 68 -> 59, 1 -> 32, 5x5, 28x28, batch 256 17.5 -> 13.1, 1 -> 6,
// 5x5, 70x50, batch 64 26 -> 18.
template <int NS, class Packs, bool PLAIN>
__global__ void __launch_bounds__(256, PLAIN ? 4 : 3) conv_fwd_small_kernel(const FwdSmallArgs a, const Packs packs) {
  extern __shared__ __align__(16) float lds[];
  const int id = a.first + blockIdx.x;
  if (fwd_small_packs(a, packs, id)) return;
  float *xs = lds;
  float *ws = lds + a.x_floats;  // [32][crs], rows past Cout are zero
  float *bs = ws + 32 * a.crs;   // [32] bias, zero past Cout or without bias
  int *offs = reinterpret_cast<int *>(bs + 32);  // [2][NS] patch offset of k = 2s, 2s + 1 (0 past K)
  const int tid = threadIdx.x, lane = tid & 63;
  // (an image's bands share rows: they go to one XCD)
  const int wg = xcd_compact_id(id - a.packers, a.workgroups);
  const int bandi = wg % a.bands, img = (wg / a.bands) % a.batch, co0 = (wg / (a.bands * a.batch)) * (PLAIN ? 32 : a.co_step);
  const int oy0 = bandi * a.band;
  const int nthr = blockDim.x;  // one wave per tile of the band, two to four waves
  fwd_small_stage<NS>(a, xs, ws, bs, offs, img, co0, oy0, tid, nthr);
  __syncthreads();

  // the lane's column of the filter matrix (k = 2*s + half)
  const int nl = lane & 31, half = lane >> 5;
  float areg[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int k = 2 * s + half;
    areg[s]     = k < a.crs ? ws[nl * a.crs + k] : 0.0f;
  }

  const uint32_t ohw = a.OH * a.OW, OW = a.OW, POW = a.OW >> 1, pohw = (a.OH >> 1) * POW;
  const uint32_t tiles = (a.band >> 1) * a.col_tiles;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = __builtin_amdgcn_readfirstlane(nthr >> 6);
  // the lane's own part of every address: its channel group and its column
  // (of two neighbours, which share a window, the odd one pools the next channel)
  const bool even = !(nl & 1);
  const uint32_t lane_out = half * 4 * ohw + nl, lane_window = even ? lane_out : lane_out - 1 + ohw;
  const uint32_t lane_pool = half * 4 * pohw + (nl >> 1) + (even ? 0 : pohw);
  const float floor_v = a.pool_act_kind == TDH_ACT_RELU ? 0.0f : -INFINITY;  // relu as a max
  const int channels  = PLAIN ? 32 : min(a.co_step, a.Kc - co0);
  auto planes = [&](auto *p, const uint32_t plane) {   // the planes of the workgroup's channels
    return __builtin_amdgcn_make_buffer_rsrc(p ? p + (static_cast<size_t>(img) * a.Kc + co0) * plane : nullptr, 0,
                                             p ? 4u * channels * plane : 0u, 0x00027000);
  };
  const auto out = planes(a.out, ohw), act_out = planes(a.act_out, ohw), pool_out = planes(a.pool_out, pohw),
             pool_argmax = planes(a.pool_argmax, pohw), pool_act_out = planes(a.pool_act_out, pohw);
#pragma unroll 1
  for (uint32_t tile = wave; tile < tiles; tile += nwaves) {
    const uint32_t rp = a.div_col_tiles.div(tile), ct = tile - rp * a.col_tiles;
    const uint32_t r = 2 * rp, c0 = 32 * ct;
    if (oy0 + r >= static_cast<uint32_t>(a.OH)) break;   // (so that a tile's offset is always inside its planes)
    const float *xb0 = xs + r * a.sh * a.pitch + (c0 + nl) * a.sw;
    const float *xb1 = xb0 + a.sh * a.pitch;
    floatx16 acc0, acc1;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc0[i] = acc1[i] = 0.0f;
    // The patch values of four k-steps are read while the products of the four before them
    // run, and their offsets a group earlier: read and product one after the other would wait for LDS in every step.
    constexpr int G = 4;
    static_assert(NS % G == 0 && NS >= 2 * G, "k-steps come in groups");
    int from = half * NS;
    asm volatile("" : "+v"(from));   // (not held over the tiles)
    intx4 o[2];
    float b0[2][G], b1[2][G];
    auto read_offsets = [&](int g) { o[g & 1] = *reinterpret_cast<const intx4 *>(offs + from + g * G); };
    auto read_patch = [&](int g) {
#pragma unroll
      for (int j = 0; j < G; ++j) {
        b0[g & 1][j] = xb0[o[g & 1][j]];
        b1[g & 1][j] = xb1[o[g & 1][j]];
      }
    };
    read_offsets(0);
    read_offsets(1);
    read_patch(0);
#pragma unroll
    for (int g = 0; g < NS / G; ++g) {
      const int cur = g & 1;
      if (g + 1 < NS / G) read_patch(g + 1);
      if (g + 2 < NS / G) read_offsets(g + 2);
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const int k = 2 * (g * G + j);
        if (g >= NS / G - 2) {   // (the steps come in eights)
          // No product of an index past the last tap: it would read the word of the first one, and zero times an infinity there is
          // NaN. The steps left out are time as well: 1 -> 32, 5x5, 28x28, batch 256 13.8 us / 13.2.
          if (k >= a.crs) break;
          if (k + 1 == a.crs && half) b0[cur][j] = b1[cur][j] = 0.0f;
        }
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(areg[g * G + j], b0[cur][j], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(areg[g * G + j], b1[cur][j], acc1, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // (the reads stay in front of the group they were written for)
    }
    // reg i of lane l holds channel 8*(i/4) + 4*(l/32) + i%4 at column l%32
    const uint32_t oy = oy0 + r;
    const uint32_t first = oy * OW + c0;  // of the tile inside a channel plane
    float v0[16], v1[16];
    int at_bias = half * 4;
    asm volatile("" : "+v"(at_bias));
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float bias = bs[at_bias + (i >> 2) * 8 + (i & 3)];
      v0[i] = acc0[i] + bias;
      v1[i] = acc1[i] + bias;
    }
    const bool in = c0 + nl < OW && oy < static_cast<uint32_t>(a.OH);
    const uint32_t lane0 = in ? 4 * lane_out : FWD_SMALL_NOWHERE;
    const uint32_t lane1 = in && oy + 1 < static_cast<uint32_t>(a.OH) ? 4 * (lane_out + OW) : FWD_SMALL_NOWHERE;
    // the lane holds channel c of register i (scalar: the first of the two halves'); of a channel that does not exist, nothing is in reach
    auto here  = [&](int c, uint32_t lane) { return PLAIN || c + 4 * half < channels ? lane : FWD_SMALL_NOWHERE; };
    auto plane = [&](int c, uint32_t size) { return PLAIN || c < channels ? c * size : 0u; };
    auto write = [&](auto stream, const auto to) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int c = (i >> 2) * 8 + (i & 3);
        fwd_small_store<decltype(stream)::value>(v0[i], to, here(c, lane0), 4 * (plane(c, ohw) + first));
        fwd_small_store<decltype(stream)::value>(v1[i], to, here(c, lane1), 4 * (plane(c, ohw) + first));
      }
    };
    if (a.out) {
      // (what is pooled here no kernel reads next: 86 us / 77 for 131 MB of it)
      if (a.pool_out)
        write(std::true_type(), out);
      else
        write(std::false_type(), out);
    }
    if (a.act_out) {
      if (PLAIN) {
        if (a.act_kind == TDH_ACT_RELU) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            v0[i] = act_apply(TDH_ACT_RELU, v0[i]);
            v1[i] = act_apply(TDH_ACT_RELU, v1[i]);
          }
        }
      } else {
        act_apply_each(a.act_kind, v0);
        act_apply_each(a.act_kind, v1);
      }
      write(std::false_type(), act_out);
    }
    if (a.pool_out) {
      // the window of two neighbours in scan order, strict '>', start value lowest();
      // where: the winner's distance from the window's first element (0, 1, OW, OW + 1), -1 when
      // no value beat the start value
      const uint32_t pfirst = (oy >> 1) * POW + (c0 >> 1);
      const uint32_t lane_p = in ? 4 * lane_pool : FWD_SMALL_NOWHERE;
      float best[8];
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float l0 = lane_xor1(v0[i + 1]), r0 = lane_xor1(v0[i]), l1 = lane_xor1(v1[i + 1]), r1 = lane_xor1(v1[i]);
        const float w4[4] = {even ? v0[i] : l0, even ? r0 : v0[i + 1], even ? v1[i] : l1, even ? r1 : v1[i + 1]};
        const int at[4]   = {0, 1, static_cast<int>(OW), static_cast<int>(OW) + 1};
        float &b  = best[i >> 1];
        b         = -FLT_MAX;
        int where = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (w4[j] > b) {
            b     = w4[j];
            where = at[j];
          }
        const int c = (i >> 2) * 8 + (i & 3);
        const uint32_t to = here(c + (even ? 0 : 1), lane_p), tile_p = 4 * (plane(c, pohw) + pfirst);
        const uint32_t cfirst = (co0 + c) * ohw + first;  // scalar: flat CHW index of the tile's first element
        fwd_small_store<false>(b, pool_out, to, tile_p);
        fwd_small_store<false>(where < 0 ? 0 : static_cast<int>(cfirst + lane_window) + where, pool_argmax, to, tile_p);
        if (PLAIN && a.pool_act_out) fwd_small_store<false>(b > floor_v ? b : floor_v, pool_act_out, to, tile_p);
      }
      if (!PLAIN && a.pool_act_out) {
        act_apply_each(a.pool_act_kind, best);
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const int c = (i >> 2) * 8 + (i & 3);
          fwd_small_store<false>(best[i >> 1], pool_act_out, here(c + (even ? 0 : 1), lane_p), 4 * (plane(c, pohw) + pfirst));
        }
      }
    }
  }
}

struct FwdSmallPlan {
  FwdSmallArgs a;
  int ns;  // k-steps, rounded up to the next instantiated count
  size_t lds_bytes;
  bool ok;
};

FwdSmallPlan make_fwd_small_plan(int batch, int C, int Kc, int H, int W, int OH, int OW, int R, int S,
                                 int sh, int sw, int dh, int dw, int ph, int pw) {
  FwdSmallPlan p;
  p.ok = false;
  FwdSmallArgs &a = p.a;
  a.x = a.w = a.bias = nullptr;
  a.out = a.act_out = a.pool_out = a.pool_act_out = nullptr;
  a.pool_argmax = nullptr;
  a.act_kind = a.pool_act_kind = TDH_ACT_NONE;
  a.C = C; a.Kc = Kc; a.H = H; a.W = W; a.OH = OH; a.OW = OW;
  a.R = R; a.S = S; a.sh = sh; a.sw = sw; a.dh = dh; a.dw = dw; a.ph = ph; a.pw = pw;
  a.crs = C * R * S;
  // A workgroup's planes are one buffer, with FWD_SMALL_NOWHERE behind it: of planes of 2^25 pixels and more it takes
  // fewer than 32 (1 input channel of 2050x16500, 3x3, us by the general kernel / here: to 3 channels 1015 / 636,
  // to 33 3619 / 2155).
  auto buffer = [&](int channels) { return 4LL * std::min(channels, Kc) * OH * OW; };
  a.co_step = 32;
  while (a.co_step > 1 && buffer(a.co_step) > FWD_SMALL_NOWHERE) a.co_step /= 2;
  if (buffer(a.co_step) > FWD_SMALL_NOWHERE) return p;
  if (a.crs > 96 || batch < 1 || batch > 65535 || OH < 1 || OW < 1) return p;
  p.ns = ((a.crs + 1) / 2 + 7) / 8 * 8;
  a.col_tiles = ceil_div(OW, 32);
  a.pitch     = (a.col_tiles * 32 - 1) * sw + (S - 1) * dw + 1;
  a.pitch |= 1;
  const int co_tiles = ceil_div(Kc, a.co_step);
  if (co_tiles > 65535) return p;
  const int cus  = ctx().compute_units > 0 ? ctx().compute_units : 256;
  const int OH2  = (OH + 1) & ~1;
  auto lds_floats = [&](int band) {
    const int rows_in = (band - 1) * sh + (R - 1) * dh + 1;
    const size_t x_fl = (static_cast<size_t>(C) * (rows_in * a.pitch + 1) + 3) & ~static_cast<size_t>(3);
    return x_fl + 32u * a.crs + 32u + 96u;
  };
  // an even band: the largest that fits and still gives two workgroups per compute unit; never
  // fewer than four tiles (one per wave) for that
  int best = 0;
  for (int band = OH2; band >= 2; band -= 2) {
    if (lds_floats(band) * sizeof(float) > 64 * 1024) continue;
    best = band;
    if (static_cast<long long>(batch) * ceil_div(OH, band) * co_tiles >= 4LL * cus ||
        (band / 2) * a.col_tiles <= 4)
      break;
  }
  if (best == 0) return p;
  // (the same number of bands, the rows spread evenly over them)
  best      = std::min(best, (ceil_div(OH2, ceil_div(OH2, best)) + 1) & ~1);
  a.band    = best;
  a.bands   = ceil_div(OH, best);
  a.rows_in = (best - 1) * sh + (R - 1) * dh + 1;
  a.plane   = a.rows_in * a.pitch + 1;
  a.x_floats = static_cast<int>((static_cast<size_t>(C) * a.plane + 3) & ~static_cast<size_t>(3));
  a.div_pitch     = FastDiv(a.pitch);
  a.div_rows_in   = FastDiv(a.rows_in);
  a.div_col_tiles = FastDiv(a.col_tiles);
  p.lds_bytes = lds_floats(best) * sizeof(float);
  const long workgroups = static_cast<long>(a.bands) * batch * co_tiles;
  if (workgroups > (1L << 30)) return p;
  a.batch      = batch;
  a.workgroups = static_cast<int>(workgroups);
  p.ok        = true;
  return p;
}

template <int NS, class Packs>
int launch_fwd_small(const FwdSmallPlan &p, const Packs &packs, int pack_blocks) {
  const int tiles = (p.a.band / 2) * p.a.col_tiles;
  FwdSmallArgs a = p.a;
  auto plain = [](int kind) { return kind == TDH_ACT_RELU || kind == TDH_ACT_NONE; };
  const dim3 block(64 * std::min(4, std::max(2, tiles)));
  a.packers = std::min(block.x < 256 ? 2 * pack_blocks : pack_blocks, FWD_SMALL_PACKERS);
  // (one launch but for more than 2^32 work-items. A grid of two directions instead cost the kernel a round trip for the grid's
  // size and scalar registers: 3 -> 24, 3x3, 30x30, batch 37 6.6 us / 6.9)
  const int total = a.packers + a.workgroups;
  for (a.first = 0; a.first < total; a.first += GRID_X_MAX) {
    const dim3 grid(std::min(total - a.first, GRID_X_MAX));
    if (a.Kc % 32 == 0 && a.co_step == 32 && (!a.act_out || plain(a.act_kind)) && (!a.pool_act_out || plain(a.pool_act_kind)))
      TDH_LAUNCH((conv_fwd_small_kernel<NS, Packs, true>), grid, block, p.lds_bytes, ctx().stream, a, packs);
    else
      TDH_LAUNCH((conv_fwd_small_kernel<NS, Packs, false>), grid, block, p.lds_bytes, ctx().stream, a, packs);
  }
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}
template <class Packs>
int launch_fwd_small_ns(const FwdSmallPlan &p, const Packs &packs, int pack_blocks) {
  switch (p.ns) {
    case 8: return launch_fwd_small<8>(p, packs, pack_blocks);
    case 16: return launch_fwd_small<16>(p, packs, pack_blocks);
    case 24: return launch_fwd_small<24>(p, packs, pack_blocks);
    case 32: return launch_fwd_small<32>(p, packs, pack_blocks);
    case 40: return launch_fwd_small<40>(p, packs, pack_blocks);
    default: return launch_fwd_small<48>(p, packs, pack_blocks);
  }
}

}  // namespace

bool conv_fwd_small_applicable(int batch, int C, int Kc, int H, int W, int OH, int OW, int R, int S,
                               int sh, int sw, int dh, int dw, int ph, int pw) {
  return make_fwd_small_plan(batch, C, Kc, H, W, OH, OW, R, S, sh, sw, dh, dw, ph, pw).ok;
}

int conv_fwd_small_run(int batch, int C, int Kc, const float *x, const float *w, const float *bias,
                       float *out, int H, int W, int OH, int OW, int R, int S, int sh, int sw, int dh,
                       int dw, int ph, int pw, float *act_out, int act_kind, const PoolFuse *pool) {
  FwdSmallPlan p = make_fwd_small_plan(batch, C, Kc, H, W, OH, OW, R, S, sh, sw, dh, dw, ph, pw);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_fwd_small_run: shape not supported");
  if (pool && ((OH | OW) & 1))
    return set_error(TDH_ERR_INVALID, "conv_fwd_small_run: a fused 2x2 pool needs even output sizes");
  if (!out && !pool && !act_out) return set_error(TDH_ERR_INVALID, "conv_fwd_small_run: no output");
  p.a.x = x; p.a.w = w; p.a.bias = bias; p.a.out = out;
  p.a.act_out  = act_out;
  p.a.act_kind = act_kind;
  if (pool) {
    p.a.pool_out      = pool->out;
    p.a.pool_argmax   = pool->argmax;
    p.a.pool_act_out  = pool->act_out;
    p.a.pool_act_kind = pool->act_kind;
  }
  ProfScope prof(pool ? "conv_fwd_small_pool" : "conv_fwd_small", Kc, batch * OH * OW, p.a.crs);
  std::vector<PackJob> jobs = take_left_packs();
  if (jobs.empty()) return launch_fwd_small_ns(p, NoPacks(), 0);
  PackJobs packs;
  int blocks   = 0;
  double bytes = 0.0;
  const int here = std::min<int>(CONV_PACK_JOBS, static_cast<int>(jobs.size()));
  plan_packs(jobs.data(), here, &packs, &blocks, &bytes);
  p.a.pack_threads = 256 * blocks;
  conv_pack_leave(jobs.data() + here, static_cast<int>(jobs.size()) - here);
  return launch_fwd_small_ns(p, packs, blocks);
}

}  // namespace tdh
