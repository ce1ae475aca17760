// conv_s1.h — what the host side of the stride-1 convolution kernel (conv_s1.hip) and the
// translation units that instantiate the kernel (conv_s1_inst.hip, compiled once per window and
// load width so that they build in parallel) share.
#pragma once
#include "common.h"

namespace tdh {

// Reduction channels per chunk. Tiles of four accumulator blocks a wave take 8 (4 with 25
// taps), tiles of two channel blocks with 25 taps 8: two workgroups share a CU's 512 registers, and
// beside that many accumulators the staged words of 16 channels no longer fit.
constexpr int s1_kch(int RS, int TM, int TN) {
  return TM * TN >= 4 ? (RS >= 25 ? 4 : 8) : (TM == 2 && TN == 1 && RS >= 25 ? 8 : 16);
}

// Input-patch words a thread stages per chunk at most: a tile of 128*TN pixels in rows of TC,
// cut into at most two images (two halos), 256/KCH threads to a channel plane.
constexpr int s1_niq(int R, int S, int TC, int TM, int TN) {
  const int nq  = (3 + TC + S - 1 + 3) / 4;
  const int tpc = 256 / s1_kch(R * S, TM, TN);
  const int n   = ((128 * TN / TC + 2 * (R - 1)) * nq + tpc - 1) / tpc;
  return n > 16 ? 16 : n;
}

// The three-part bf16 kernel (conv_x3_body.h): 16 channels a chunk, words of eight channels that
// a thread stages per chunk at most (32 registers each; 1 x 1: the tile shared by filter taps).
constexpr int X3_KCH = 16;
constexpr int x3_items(int TM, int TN) { return TM * TN >= 4 || TM * TN == 1 ? 1 : 2; }
// rows of the packed filters: whole tiles of either width
constexpr int x3_mc_pad(int MC) { return MC > 32 ? (MC + 63) / 64 * 64 : 32; }
constexpr size_t x3_pack_bytes(int RS, int KC, int MC) {
  return static_cast<size_t>((KC + 15) / 16) * RS * 6 * x3_mc_pad(MC) * 16;
}

// The first pixel, in the workgroup's tile of rows of TC pixels, of accumulator block b = wave * TN + j. Blocks are 32 pixels in
// a row, one after the other; where a row of 64 is two blocks and a wave has two, they are the same columns of two rows, so that a lane
// holds both rows of its column and two lanes a 2x2 pooling window. A wave of four blocks of such rows holds two rows anyway (in any
// other order the instance needs more than the 256 registers there are: 80 of them went to memory, and 24 -> 32 channels, 5x5, 96x96,
// 16 images, tanh and the pool took 105 us instead of 89). (Not in the three-part kernel, whose waves read
// 0.5 % slower that way: 32 -> 64 channels, 3x3, 64x64, batch 64, forward, dX and dW 219.3 us / 220.3.)
template <int TC, int TN>
__host__ __device__ constexpr int s1_block_pixel(const int b) {
  return TC == 64 && TN == 2 ? ((b >> 2) * 2 + (b & 1)) * 64 + ((b >> 1) & 1) * 32 : 32 * b;
}
// how many blocks further on in the wave the one below a block is
constexpr int s1_block_below(const int TC, const int TN) { return TC == 64 && TN == 4 ? 2 : 1; }

// the sign of step u's products (chunk, tap): the packed filters carry it
__host__ __device__ constexpr float x3_sign(int u) { return u & 1 ? -1.0f : 1.0f; }

struct ConvS1Args {
  const float *in;
  const void *wp;              // filters: floats [tap][kc][m], or the parts of conv_x3_inst.hip
  // what wp was packed from, for sums that the three-part kernel computes again: OIHW filters, the
  // connection table they are masked by (or null), and whether this is dX (taps reversed)
  const float *w;
  const uint8_t *tbl;
  int flip;
  const float *bias;
  float *out;
  ActGrad ag;
  float *act_out;              // forward: act(out) of the pointwise activation layer that follows
  int act_kind;
  // forward: the 2x2 / stride-2 max-pool layer behind the convolution (or behind act_out) and
  // the relu behind that pool, all null when the pool runs as a kernel of its own. Only waves
  // whose blocks hold whole pool windows (rows of 8 or 16 pixels, or an even number of blocks in rows of 32 and, in fp32, 64; no split) take it.
  float *pool_out;
  int32_t *pool_argmax;        // flat CHW index inside the sample of the pool's input
  float *pool_act_out;         // max(pool_out, 0), or null
  int batch, KC, MC, IH, IW, OH, OW, ph, pw;
  int pwa;                     // staged column 0 is image column x0 - pwa
  int TR, TI;                  // tile rows, images per tile (TI*TR*TC = PIX), powers of two
  int log_tr, log_ti;
  int tiles_x, tiles_y;        // tiles per image row / column direction
  FastDiv div_rows;            // by the words of one image of the staged patch, (TR+R-1)*NQ
  // split over the reduction channels: workgroup z sums channels [z*kc_split, (z+1)*kc_split)
  // into part[z][...] (laid out like out); part == nullptr: one pass, written to out
  int kc_split;
  int mc_pad;                  // rows of the packed filters (three-part kernel)
  float *part;
  size_t part_stride;
};

struct S1Plan {
  bool ok;
  bool x3;                     // the three-part bf16 kernel
  int tc, tm, tn;
  ConvS1Args args;
  size_t lds_bytes;
  dim3 grid;
  int splits;
};

// the plan of a dX that shares its launch with the weight gradient (conv_bwd_pair.hip)
S1Plan make_s1_pair_plan(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw);
size_t plan_workspace_bytes(const S1Plan &p, int RS);
int finish_s1_split(const S1Plan &p, const float *bias, ActGrad ag, float *out, float *act_out, int act_kind);

// one launcher per translation unit of kernel instances
int s1_launch_3x3_vec(const S1Plan &p);
int s1_launch_3x3_scalar(const S1Plan &p);
int s1_launch_5x5_vec(const S1Plan &p);
int s1_launch_5x5_scalar(const S1Plan &p);
int x3_launch_1_vec(const S1Plan &p);
int x3_launch_1_scalar(const S1Plan &p);
int x3_launch_3_vec(const S1Plan &p);
int x3_launch_3_scalar(const S1Plan &p);
int x3_launch_5_vec(const S1Plan &p);
int x3_launch_5_scalar(const S1Plan &p);
int x3_launch_7_vec(const S1Plan &p);
int x3_launch_7_scalar(const S1Plan &p);

}  // namespace tdh
