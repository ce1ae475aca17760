// conv_s1_epilogue.h — what the stride-1 convolution kernels do with their accumulators: bias,
// activation gradient, the activation and the 2x2 max-pool behind the layer, or a split's partial
// sums. A workgroup of four wave64 owns 32*TM channels x 128*TN pixels of TI images x TR rows x
// TC columns; wave wn holds the pixel blocks wn*TN .. wn*TN+TN-1.
#pragma once
#include "conv_s1.h"

namespace tdh {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// the value of lane l ^ 1 (a swap inside lane pairs, done by the DPP path of a move)
__device__ __forceinline__ float s1_lane_xor1(const float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
// the value of lane l ^ X, X = 8 or 16 (a swizzle inside groups of 32 lanes: and 0x1F, or 0, xor X)
template <int X>
__device__ __forceinline__ float s1_lane_xor(const float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (X << 10) | 0x1F));
}

// The forward pass with a 2x2 max-pool behind it where a wave holds two rows of a block's columns (s1_block_pixel, s1_block_below): a lane
// holds both rows of its column, two neighbours share a window, exchange the values of two channels and pool one each,
// with strict '>' from lowest() in scan order (maxpool_op_internal.h:17-47). The pool's own kernel is bound by the read of
// the activation, which no kernel reads next once the pool is made here: y and it go past the caches. us of
// convolution and pool, apart / here: 64 -> 64 channels, 3x3, 128x128, batch 64 748 / 697, 128 -> 128, 64x64 655 / 620 (stores that
// stay in the caches 703 and 628).
template <int TC, int TM, int TN>
__device__ __forceinline__ void s1_epilogue_pool_rows(const ConvS1Args &a, const floatx16 (&acc)[TM][TN], const int wn,
                                                      const int lane, const int img0, const int y0, const int x0, const int m0) {
  constexpr int LOG_TC = TC == 64 ? 6 : 5;
  const int ohw = a.OH * a.OW, pw2 = a.OW >> 1, pohw = (a.OH >> 1) * pw2;
  const bool right = lane & 1;
#pragma unroll
  for (int pair = 0; pair < TN / 2; ++pair) {
    constexpr int BELOW = s1_block_below(TC, TN);
    const int j   = BELOW == 1 ? 2 * pair : pair;
    const int q   = s1_block_pixel<TC, TN>(wn * TN + j) + (lane & 31);
    const int img = img0 + (q >> (a.log_tr + LOG_TC));
    const int oy = y0 + ((q >> LOG_TC) & (a.TR - 1)), ox = x0 + (q & (TC - 1));
    if (img >= a.batch || oy >= a.OH || ox >= a.OW) continue;   // (even sizes: both rows, and both lanes of a window)
    const size_t pbase  = static_cast<size_t>(img) * a.MC * ohw + oy * a.OW + ox;
    const size_t pobase = static_cast<size_t>(img) * a.MC * pohw + (oy >> 1) * pw2 + (ox >> 1);
    const int pix = oy * a.OW + (ox & ~1);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int mb = m0 + 32 * i + 4 * (lane >> 5);
      float v0[16], v1[16];
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        v0[rr] = acc[i][j][rr];
        v1[rr] = acc[i][j + BELOW][rr];
      }
      if (a.bias) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const float b = a.bias[min(mb + 8 * (rr >> 2) + (rr & 3), a.MC - 1)];
          v0[rr] += b;
          v1[rr] += b;
        }
      }
      auto write = [&](float *to) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const int m = mb + 8 * (rr >> 2) + (rr & 3);
          if (m < a.MC) {
            float *p = to + pbase + static_cast<size_t>(m) * ohw;
            __builtin_nontemporal_store(v0[rr], p);
            __builtin_nontemporal_store(v1[rr], p + a.OW);
          }
        }
      };
      if (a.out) write(a.out);
      if (a.act_out) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          v0[rr] = act_apply(a.act_kind, v0[rr]);
          v1[rr] = act_apply(a.act_kind, v1[rr]);
        }
        write(a.act_out);
      }
#pragma unroll
      for (int rr = 0; rr < 16; rr += 2) {
        const float l0 = s1_lane_xor1(v0[rr + 1]), r0 = s1_lane_xor1(v0[rr]);
        const float l1 = s1_lane_xor1(v1[rr + 1]), r1 = s1_lane_xor1(v1[rr]);
        const float w4[4] = {right ? l0 : v0[rr], right ? v0[rr + 1] : r0, right ? l1 : v1[rr], right ? v1[rr + 1] : r1};
        float best = -3.402823466e+38f;
        int sel    = -1;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (w4[k] > best) {
            best = w4[k];
            sel  = k;
          }
        const int m = mb + 8 * (rr >> 2) + (rr & 3) + (right ? 1 : 0);
        if (m < a.MC) {
          const size_t at = pobase + static_cast<size_t>(m) * pohw;
          a.pool_out[at]    = best;
          a.pool_argmax[at] = sel < 0 ? 0 : m * ohw + pix + (sel >> 1) * a.OW + (sel & 1);
          if (a.pool_act_out) a.pool_act_out[at] = best > 0.0f ? best : 0.0f;
        }
      }
    }
  }
}

// ROWS: the wave's blocks lie as s1_block_pixel<TC, TN> has them and the pool behind rows of 32 and 64 can be made here, else
// the blocks lie one after the other
template <int TC, int TM, int TN, bool ROWS = true>
__device__ __forceinline__ void s1_epilogue(const ConvS1Args &a, const floatx16 (&acc)[TM][TN], const int wn,
                                            const int lane, const int img0, const int y0, const int x0,
                                            const int m0, const int bz) {
  constexpr int LOG_TC = TC == 64 ? 6 : TC == 32 ? 5 : TC == 16 ? 4 : 3;
  // reg r of lane l holds channel 8*(r/4) + 4*(l/32) + r%4, pixel l%32
  const int ohw = a.OH * a.OW;
  if constexpr (ROWS && TC >= 32 && TN % 2 == 0) {
    if (a.pool_out) {   // (forward, unsplit)
      s1_epilogue_pool_rows<TC, TM, TN>(a, acc, wn, lane, img0, y0, x0, m0);
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int q   = s1_block_pixel<TC, ROWS ? TN : 1>(wn * TN + j) + (lane & 31);
    const int ti  = q >> (a.log_tr + LOG_TC);
    const int r   = (q >> LOG_TC) & (a.TR - 1);
    const int c   = q & (TC - 1);
    const int img = img0 + ti, oy = y0 + r, ox = x0 + c;
    if (img >= a.batch || oy >= a.OH || ox >= a.OW) continue;
    const size_t pbase = static_cast<size_t>(img) * a.MC * ohw + oy * a.OW + ox;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      // the 16 values of this lane: channels mb + 8*(rr/4) + rr%4, all at pixel pbase
      const int mb = m0 + 32 * i + 4 * (lane >> 5);
      float *dst = a.part ? a.part + bz * a.part_stride : a.out;
      float v[16];
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) v[rr] = acc[i][j][rr];
      if (!a.part) {
        if (a.bias) {
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) {
            const int m = mb + 8 * (rr >> 2) + (rr & 3);
            v[rr] += a.bias[min(m, a.MC - 1)];
          }
        }
        if (a.ag.kind != TDH_ACT_NONE) {
          // all loads of y first: one at a time they would each cost a trip to memory
          float yv[16];
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) {
            const int m = mb + 8 * (rr >> 2) + (rr & 3);
            yv[rr] = a.ag.y[pbase + static_cast<size_t>(min(m, a.MC - 1)) * ohw];
          }
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) v[rr] *= act_grad_factor(a.ag.kind, yv[rr]);
        }
      }
      if (dst) {  // (null: the pool behind leaves this kernel too and nobody reads the convolution's own output)
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const int m = mb + 8 * (rr >> 2) + (rr & 3);
          if (m < a.MC) dst[pbase + static_cast<size_t>(m) * ohw] = v[rr];
        }
      }
      if (!a.part && a.act_out) {
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const int m = mb + 8 * (rr >> 2) + (rr & 3);
          v[rr]       = act_apply(a.act_kind, v[rr]);
          if (m < a.MC) a.act_out[pbase + static_cast<size_t>(m) * ohw] = v[rr];
        }
      }
      if constexpr (TC <= 16) {
        if (!a.part && a.pool_out) {
          // A 32-pixel block is whole rows of TC pixels, the first one even: a window belongs to four lanes, l, l^1, l^TC and
          // l^(TC+1) in scan order. They turn their 4 x 4 values of four channels and each pools the channel of its place, with
          // strict '>' from lowest() (maxpool_op_internal.h:17-47): a quarter of the code, which runs once, cold, and of the
          // stores of a lane that pools every channel and leaves three idle (16x16, 32 -> 32, 5x5: fp32,
          // batch 128, without y 22.2 / 20.8; three parts, batch 1000, with y 80 / 75).
          const bool right = lane & 1, below = lane & TC;
          const int pw2 = a.OW >> 1, pohw = (a.OH >> 1) * pw2;
          const size_t pobase = static_cast<size_t>(img) * a.MC * pohw + (oy >> 1) * pw2 + (ox >> 1);
          const int pix = (oy & ~1) * a.OW + (ox & ~1);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float l[2], r2[2];   // this row's two values of channel 2k + right
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const float v0 = v[4 * g + 2 * k], v1 = v[4 * g + 2 * k + 1];
              const float from1 = s1_lane_xor1(v1), from0 = s1_lane_xor1(v0);
              l[k]  = right ? from1 : v0;
              r2[k] = right ? v1 : from0;
            }
            const float l0 = s1_lane_xor<TC>(l[0]), r0 = s1_lane_xor<TC>(r2[0]), l1 = s1_lane_xor<TC>(l[1]), r1 = s1_lane_xor<TC>(r2[1]);
            const float w4[4] = {below ? l1 : l[0], below ? r1 : r2[0], below ? l[1] : l0, below ? r2[1] : r0};
            float best = -3.402823466e+38f;
            int sel    = -1;
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (w4[k] > best) {
                best = w4[k];
                sel  = k;
              }
            const int m = mb + 8 * g + (right ? 1 : 0) + (below ? 2 : 0);
            if (m < a.MC) {
              const size_t at = pobase + static_cast<size_t>(m) * pohw;
              a.pool_out[at]    = best;
              a.pool_argmax[at] = sel < 0 ? 0 : m * ohw + pix + (sel >> 1) * a.OW + (sel & 1);
              if (a.pool_act_out) a.pool_act_out[at] = best > 0.0f ? best : 0.0f;
            }
          }
        }
      }
    }
  }
}

}  // namespace
}  // namespace tdh
