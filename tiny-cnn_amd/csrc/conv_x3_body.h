// conv_x3_body.h — the stride-1 convolution (forward and dX) of conv_s1_inst.hip on the bf16
// matrix cores with three-part operands (split_bf16.h): the same tiles and epilogue, another
// inner loop. Bound: bf16 MFMA issue; 6 instructions of 32768 FLOP stand for one fp32 product.
//
// Per chunk of 16 reduction channels a workgroup loads the input patch with its halo as 16-byte
// words of four pixels, eight channels of a word to a thread, splits them once and leaves them in
// LDS as [part][8-channel half][pixel][8 channels]: the operand of one lane of a
// 32x32x16 product is then one aligned 16-byte read at a pixel, every filter tap is a constant
// number of pixels away, and a split is shared by all taps and all output channels. The filters
// come split from memory ([chunk][tap][part][half][m][8 channels], x3_pack_kernel): a wave reads its
// own operands of the next tap from there while it multiplies the current one (the four waves of
// a workgroup read the same lines, so all but the first find them in L1), which leaves the LDS
// to the patch: 41 KB for 64 channels x 4 rows of 64 pixels, two workgroups a compute unit.
// What a workgroup does; the kernels around it are in conv_x3_inst.hip and conv_bwd_pair.hip.
#pragma once
#include "conv_s1_epilogue.h"
#include "split_bf16.h"
#include <type_traits>

namespace tdh {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr unsigned X3_NOWHERE = 0x80000000u;  // past the end of every tile's images

// The wave's infinite and NaN sums once more in fp32 (split_bf16.h): lane l brings channel l%32 of a
// filter block and pixel l%32 of a pixel block, for the reduction channel kc + l/32.
template <int R, int S, int TC, int TM, int TN>
__device__ __forceinline__ void x3_redo_exceptional(const ConvS1Args &a, floatx16 (&acc)[TM][TN], const int wn,
                                                    const int lane, const int img0, const int y0, const int x0,
                                                    const int m0, const int kc_lo, const int kc_hi) {
  constexpr int LOG_TC = TC == 64 ? 6 : TC == 32 ? 5 : TC == 16 ? 4 : 3;
  // (hidden from the compiler, which otherwise keeps this function's comparisons and addresses for the stores behind)
  int rows = a.MC - (m0 + 4 * (lane >> 5)), pix = wn * TN * 32 + (lane & 31);
  asm volatile("" : "+v"(rows), "+v"(pix));
  auto place = [&](int j, int &img, int &oy, int &ox) {
    const int q = pix + 32 * j;
    img = img0 + (q >> (a.log_tr + LOG_TC));
    oy  = y0 + ((q >> LOG_TC) & (a.TR - 1));
    ox  = x0 + (q & (TC - 1));
    return img < a.batch && oy < a.OH && ox < a.OW;
  };
  x3_redo(reinterpret_cast<floatx16(&)[TM * TN]>(acc), [&](int b, int r) {
    int img, oy, ox;
    return place(b % TN, img, oy, ox) && 32 * (b / TN) + 8 * (r >> 2) + (r & 3) < rows;
  }, [&](floatx16 (&sum)[TM * TN]) {
#pragma unroll 1
    for (int kc0 = kc_lo; kc0 < kc_hi; kc0 += 2) {
      const int kc = kc0 + (lane >> 5);
#pragma unroll 1
      for (int fy0 = 0; fy0 < R; ++fy0) {
        float wv[TM][S], xv[TN][S];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m   = m0 + 32 * i + (lane & 31);
          const bool on = kc < kc_hi && m < a.MC && (!a.tbl || a.tbl[a.flip ? m * a.KC + kc : kc * a.MC + m]);
          const float *w = a.w + static_cast<size_t>(on ? (a.flip ? kc * a.MC + m : m * a.KC + kc) : 0) * (R * S);
#pragma unroll
          for (int t = 0; t < S; ++t) wv[i][t] = on ? w[a.flip ? R * S - 1 - fy0 * S - t : fy0 * S + t] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          int img, oy, ox;
          const bool pixel = place(j, img, oy, ox) && kc < kc_hi;
          const float *in  = a.in + (static_cast<size_t>(pixel ? img : 0) * a.KC + (pixel ? kc : 0)) * a.IH * a.IW;
#pragma unroll
          for (int t = 0; t < S; ++t) {
            const int iy = oy - a.ph + fy0, ix = ox - a.pw + t;
            const bool inside = pixel && static_cast<unsigned>(iy) < static_cast<unsigned>(a.IH) &&
                                static_cast<unsigned>(ix) < static_cast<unsigned>(a.IW);
            xv[j][t] = inside ? in[iy * a.IW + ix] : 0.0f;
          }
        }
#pragma unroll
        for (int t = 0; t < S; ++t)
#pragma unroll
          for (int b = 0; b < TM * TN; ++b)
            sum[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[b / TN][t], xv[b % TN][t], sum[b], 0, 0, 0);
      }
      if (x3_all_nan(sum)) return;
    }
  });
}

// the workgroup at (bx, by, bz) of the grid. BY_TAPS: the four waves share the
// workgroup's 32 channels x 128 pixels (TM = TN = 1) by filter taps instead of by pixels. POOL: with the max-pool behind
// rows of 32 (shorter rows always can)
template <int R, int S, int TC, int TM, int TN, bool VEC, bool BY_TAPS, bool POOL = false>
__device__ __forceinline__ void conv_x3_workgroup(const ConvS1Args &a, const int bx, const int by, const int bz) {
  static_assert(!BY_TAPS || (TM == 1 && TN == 1), "a tile of 32 channels x 128 pixels");
  constexpr int RS     = R * S;
  constexpr int NI     = BY_TAPS ? 1 : x3_items(TM, TN);
  constexpr int NJ     = BY_TAPS ? 4 : TN;          // pixel blocks of a wave
  constexpr int NQ     = (3 + TC + S - 1 + 3) / 4;  // words per staged row
  constexpr int PITCH  = 4 * NQ;
  constexpr int BM     = 32 * TM;
  constexpr int LOG_TC = TC == 64 ? 6 : TC == 32 ? 5 : TC == 16 ? 4 : 3;

  extern __shared__ __align__(16) uintx4 patch[];   // [part][half][pixel]
  const int TRH    = a.TR + R - 1;
  const int planeq = a.TI * TRH * NQ;  // words of one channel of the staged patch
  const int npix   = 4 * planeq;

  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  int bt        = bx;
  const int tx  = bt % a.tiles_x;
  bt /= a.tiles_x;
  const int ty    = bt % a.tiles_y;
  const int tb    = bt / a.tiles_y;
  const int img0  = tb << a.log_ti;
  const int y0    = ty << a.log_tr;
  const int x0    = tx * TC;
  const int m0    = by * BM;
  const int ihw   = a.IH * a.IW;
  const int kc_lo = bz * a.kc_split;
  const int kc_hi = min(a.KC, kc_lo + a.kc_split);

  // ---- staging plan: item tid + 256*i -> channel half, word of the patch. Loads go through a
  // buffer descriptor that starts at the tile's first image and ends at the last one: words that
  // do not exist get an offset past its end and come back as zeros.
  const float *in0   = a.in + static_cast<size_t>(img0) * a.KC * ihw;
  const int n_img    = min(a.TI, a.batch - img0);
  const unsigned in_bytes = 4u * n_img * a.KC * ihw;
  unsigned goff[NI];
  int ihalf[NI], ipix[NI];
  unsigned gkeep = 0;  // scalar loads: 4 bits per item, float k lies inside the row
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int e = tid + 256 * i;
    goff[i]     = X3_NOWHERE;
    ipix[i]     = -1;
    ihalf[i]    = 0;
    if (e < 2 * planeq) {
      const int half = e >= planeq, pe = e - half * planeq;
      uint32_t ti, rem;
      a.div_rows.divmod(pe, ti, rem);
      const int r = rem / NQ, q = rem - r * NQ;
      const int iy = y0 - a.ph + r, ix = x0 - a.pwa + 4 * q;
      unsigned keep = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (static_cast<unsigned>(ix + k) < static_cast<unsigned>(a.IW)) keep |= 1u << k;
      ihalf[i] = half;
      ipix[i]  = half * npix + 4 * pe;
      if (static_cast<int>(ti) < n_img && static_cast<unsigned>(iy) < static_cast<unsigned>(a.IH) &&
          (VEC ? keep == 15u : keep != 0u)) {
        goff[i] = 4u * ((ti * a.KC + 8 * half) * ihw + iy * a.IW + ix);
        gkeep |= keep << (4 * i);
      }
    }
  }

  // ---- operand positions: pixel of lane l of block j, and this lane's filter operands
  int bpix[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int q  = ((BY_TAPS ? 0 : wn * TN) + j) * 32 + (lane & 31);
    const int ti = q >> (a.log_tr + LOG_TC);
    const int r  = (q >> LOG_TC) & (a.TR - 1);
    const int c  = q & (TC - 1);
    bpix[j]      = (ti * TRH + r) * PITCH + c + (a.pwa - a.pw) + (lane >> 5) * npix;
  }
  const char *wall     = static_cast<const char *>(a.wp);
  const uint32_t wlane = 16u * ((lane >> 5) * a.mc_pad + m0 + (lane & 31));
  const int wpart      = 2 * 16 * a.mc_pad;  // bytes from one part to the next

  floatx16 acc[TM][NJ];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  floatx4 rin[NI][8];
  // the eight channels of every item of the chunk starting at kc0
  auto fetch = [&](int kc0) {
    const auto desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(in0), 0, in_bytes, 0x00027000);
    const int left  = kc_hi - kc0;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int at       = 4 * (kc0 + c) * ihw;
        const unsigned off = left >= 16 || 8 * ihalf[i] + c < left ? goff[i] : X3_NOWHERE;
        if (VEC) {
          rin[i][c] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(desc, off, at, 0));
        } else {
          const unsigned keep = gkeep >> (4 * i);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            rin[i][c][k] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(desc, keep >> k & 1u ? off + 4 * k : X3_NOWHERE, at, 0));
        }
      }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (ipix[i] < 0) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uintx4 part[X3_PARTS];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint32_t p3[X3_PARTS];
          split_pair(X3_SCALE * rin[i][2 * c][k], X3_SCALE * rin[i][2 * c + 1][k], p3);
#pragma unroll
          for (int p = 0; p < X3_PARTS; ++p) part[p][c] = p3[p];
        }
#pragma unroll
        for (int p = 0; p < X3_PARTS; ++p) patch[p * 2 * npix + ipix[i] + k] = part[p];
      }
    }
  };

  if constexpr (BY_TAPS) {
    // Wave w multiplies the taps u = w, w + 4, .. (counted over the chunks, so the odd one moves
    // round the waves) with all four pixel blocks: the filters are read once per workgroup, not once
    // per wave, and each reading serves 24 products. The patch operands of two blocks are read
    // while the other two are multiplied.
    bf16x8 wf[1][X3_PARTS], wnext[1][X3_PARTS], xf[2][2][X3_PARTS];
    auto read_filters = [&](int u) {
      const char *w = wall + static_cast<size_t>(u) * X3_PARTS * wpart;
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p) wnext[0][p] = *reinterpret_cast<const bf16x8 *>(w + static_cast<size_t>(p) * wpart + wlane);
    };
    const int wave = __builtin_amdgcn_readfirstlane(wn);
    auto read_pair = [&](int pair, int off) {
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          xf[pair][j][p] = __builtin_bit_cast(bf16x8, patch[p * 2 * npix + bpix[2 * pair + j] + off]);
    };
    auto tap_at = [](int t) { return t / S * PITCH + t % S; };
    const int u_end = (kc_hi + 15) / 16 * RS;
    int u = kc_lo / 16 * RS;
    u += (wave - u) & 3;
    fetch(kc_lo);
    if (u < u_end) read_filters(u);
    for (int kc0 = kc_lo; kc0 < kc_hi; kc0 += 16) {
      if (kc0 > kc_lo) __syncthreads();  // everyone is done reading the previous chunk
      stage();
      __syncthreads();
      const int u0 = kc0 / 16 * RS;
      bool more    = kc0 + 16 < kc_hi;
      if (u < u0 + RS) read_pair(0, tap_at(u - u0));
#pragma unroll 1
      for (; u < u0 + RS; u += 4) {
#pragma unroll
        for (int p = 0; p < X3_PARTS; ++p) wf[0][p] = wnext[0][p];
        if (u + 4 < u_end) read_filters(u + 4);
        read_pair(1, tap_at(u - u0));
        if (more) fetch(kc0 + 16);   // (once per chunk, behind the first tap's loads)
        more = false;
        const float sign = x3_sign(u);
        mfma_x3<1, 2>(reinterpret_cast<floatx16(&)[1][2]>(acc[0][0]), wf, reinterpret_cast<const bf16x8(&)[2][X3_PARTS]>(xf[0]), sign);
        if (u + 4 < u0 + RS) read_pair(0, tap_at(u + 4 - u0));
        mfma_x3<1, 2>(reinterpret_cast<floatx16(&)[1][2]>(acc[0][2]), wf, reinterpret_cast<const bf16x8(&)[2][X3_PARTS]>(xf[1]), sign);
      }
    }
    // the waves' sums of a pixel block are added in wave order by the wave that stores the block
    __syncthreads();
    floatx4 *red = reinterpret_cast<floatx4 *>(patch);   // [wave][block][r/4][lane]
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[((wn * 4 + j) * 4 + r) * 64 + lane] =
            floatx4{acc[0][j][4 * r], acc[0][j][4 * r + 1], acc[0][j][4 * r + 2], acc[0][j][4 * r + 3]};
    __syncthreads();
    floatx16 sum[1][1];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      floatx4 v = red[(wn * 4 + r) * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += red[((w * 4 + wn) * 4 + r) * 64 + lane];
#pragma unroll
      for (int k = 0; k < 4; ++k) sum[0][0][4 * r + k] = v[k];
    }
    x3_redo_exceptional<R, S, TC, 1, 1>(a, sum, wn, lane, img0, y0, x0, m0, kc_lo, kc_hi);
    s1_epilogue<TC, 1, 1>(a, sum, wn, lane, img0, y0, x0, m0, bz);
    return;
  } else {
  // operands of tap u, counted over the chunks
  bf16x8 wf[2][TM][X3_PARTS], xf[TN][X3_PARTS];
  auto read_filters = [&](int u, int to) {
    const char *w = wall + static_cast<size_t>(u) * X3_PARTS * wpart;
#pragma unroll
    for (int p = 0; p < X3_PARTS; ++p)
#pragma unroll
      for (int i = 0; i < TM; ++i)
        wf[to][i][p] = *reinterpret_cast<const bf16x8 *>(w + static_cast<size_t>(p) * wpart + (wlane + 512u * i));
  };
  auto read_patch = [&](int t) {
#pragma unroll
    for (int p = 0; p < X3_PARTS; ++p)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        xf[j][p] = __builtin_bit_cast(bf16x8, patch[p * 2 * npix + bpix[j] + (t / S) * PITCH + t % S]);
  };

  // Loads are waited for in the order of their issue, so the filters of the tap after next would
  // wait for the patch of the next chunk, which comes from much further away, wherever that is
  // issued in between: it is issued once per chunk, behind the filters of tap 1, and has the
  // products of two taps to arrive. us for 64 -> 64 channels of 128x128 / 128 -> 128 of 64x64 /
  // 32 -> 64 of 64x64, batch 64: fp32 kernel 600 / 589 / 92, here 431 / 381 / 63 (179 / 203 / 153
  // TFLOP/s); the patch loads spread over the taps cost 6 % more, a second set of patch operands or
  // the reads pinned in front of the products 7-11 %. Without the loads, the LDS traffic and the
  // additions behind the products of all but the first chunk it is 327 / 290 / 50: what the matrix
  // cores and the power limit leave.
  fetch(kc_lo);
  read_filters(kc_lo / 16 * RS, 0);
  for (int kc0 = kc_lo; kc0 < kc_hi; kc0 += 16) {
    const bool more = kc0 + 16 < kc_hi;
    if (kc0 > kc_lo) __syncthreads();  // everyone is done reading the previous chunk
    stage();
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RS; ++t) {
      const int cur = t & 1;
      if (t + 1 < RS || more) read_filters(kc0 / 16 * RS + t + 1, cur ^ 1);
      read_patch(t);
      if (t == 0 && more) fetch(kc0 + 16);
      mfma_x3<TM, TN>(acc, wf[cur], xf, x3_sign(kc0 / 16 * RS + t));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (RS & 1) {  // the next chunk's first tap is read from buffer 0
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int p = 0; p < X3_PARTS; ++p) wf[0][i][p] = wf[1][i][p];
    }
  }
  x3_redo_exceptional<R, S, TC, TM, TN>(a, acc, wn, lane, img0, y0, x0, m0, kc_lo, kc_hi);
  s1_epilogue<TC, TM, TN, POOL>(a, acc, wn, lane, img0, y0, x0, m0, bz);
  }
}

}  // namespace
}  // namespace tdh
