// tiny_net.h — plan of the workgroup-per-sample train step of a small net (tiny_net.hip);
// built by net.hip from a network's layers.
#pragma once

#include "common.h"

namespace tdh {

constexpr int TINY_MAX_LAYERS     = 16;
constexpr int TINY_MAX_TENSORS    = 2 * TINY_MAX_LAYERS;
constexpr size_t TINY_LDS_MAX_BYTES = 152u << 10;  // of a compute unit's 160 KiB
constexpr int TINY_SCRATCH_FLOATS = 4096;          // LDS where the partial sums of a split layer meet

struct TinyTensor {
  float *g, *w, *s0, *s1;
  int index;                   // in the optimizer's table
};
struct TinyLayer {
  int kind, act;               // TDH_L_*, TDH_ACT_* (activation layers)
  float p0;                    // leaky relu's slope
  int C, H, W, K, OH, OW;      // input channels / size, output channels / size (conv, pools)
  int R, S, sh, sw, ph, pw;    // window rows / columns, strides, padding in front
  int in_size, out_size, has_bias;
  float scale;                 // average pooling: 1 / (window elements)
  const float *w, *b;
  const uint8_t *tbl;          // conv connection table [C][K], or NULL
  float *out;                  // memory: this layer's output [batch][out_size]
  float *dx;                   // memory: gradient w.r.t. this layer's input [batch][in_size]
  int32_t *argmax;             // memory: max-pool records [batch][out_size]
  float *gw, *gb;              // memory: a gradient slice per group of samples, [group][nw], [group][nb]
  float *pw_part, *pb_part;    // memory, layers in front of TinyPlan::split: what the back kernel leaves per sample
  TinyTensor tw, tb;           // weights and bias, as the optimizer has them
  int dw_chunk, dw_chunk_waves;   // parameter gradients: samples in LDS at a time, with a workgroup or a wave a channel pair (0: not so)
  int nw, nb;
  int lds_in, lds_out;         // where the layer's input and output live in LDS (floats)
  // divisions by the layer's sizes as multiply-high + shift
  FastDiv d_oplane, d_ow, d_quads, d_vquads, d_iplane, d_iplanes, d_cblocks, d_w, d_taps, d_s, d_c, d_out, d_nk;
  // the unrolled input gradient of a stride-1 3x3 / 5x5 convolution reads dY from a zero-framed copy,
  // [K][H + R - 1][W + S - 1] floats in LDS; 0 when the layer takes the general loops
  int dx_framed;
  FastDiv d_pplane, d_pw, d_pw4;
  // A stride-1 convolution's forward product without padding on the matrix cores (conv_mfma in
  // tiny_net.hip): where in LDS the step kernel keeps the filters as [co][k] (k = (ci, tap), rows
  // padded with zeros), the input offset of every k and a copy of the bias; -1: the scalar loops
  int mf_fwd_w, mf_fwd_ko, mf_fwd_b;
  // The input gradient of the layer whose filters wait in registers (TinyPlan::mf_ahead), from the
  // framed dY, as the same kind of product with the filter columns folded into the rows:
  //   D[(ci, wx)][iy][px] = sum over (co, wy) of W[co][ci][wy][wx] * framed[co][iy + R-1-wy][px]
  // (C * S rows, K * R terms a sum, every position of H framed rows a column), then
  //   dX[ci][iy][ix] = sum over wx of D[(ci, wx)][iy][ix + S-1-wx].
  // mf_dx_w / mf_dx_ko: the operand [(ci, wx)][(co, wy)] and its offset table, written into the
  // scratch area in front of the phase; mf_dx_d: D. -1: the scalar loops.
  int mf_dx_w, mf_dx_ko, mf_dx_d;
};

struct TinyPlan {
  TinyLayer l[TINY_MAX_LAYERS];
  int n, in_size;
  // the second convolution, where the layers in front of it run a channel a workgroup (tiny_net.hip), or 0;
  // LDS of those launches: floats behind the input in front, and offsets behind the framed dY
  int split, front_floats, back_scratch, back_planes, back_sample, back_sample_floats, back_floats;
  int lds_g0, lds_g1, lds_w, lds_pad, lds_floats;   // lds_pad: the zero-framed dY
  int n_mfma, mfma_layers[TINY_MAX_LAYERS];   // the layers with operands to stage for the matrix cores
  int mf_ahead;                // the layer (> 0) whose filters wait in registers until the layer in front of it runs, or -1
  // the layer whose filters wait in registers from layer held_from on (held_chain), or 0; how they lie there (Held)
  int held, held_from, held_shift, held_rows;   // (held_from: a convolution on the matrix cores)
  FastDiv d_held_rows;
  float mse_factor;            // 2 / outputs
  float *dloss;                // memory: gradient w.r.t. the net's output [batch][out_size]
  double flop_per_sample;
  int first_dx_as_job;         // the first layer's input gradient is computed beside the parameter gradients,
  float *first_w;              // ... from this copy of its filters (memory), which the step kernel makes
  int by_rows;                 // weight gradients of convolutions sample by sample (a window is not 3x3 or 5x5, or strided)
  int skip_first_dx;           // nobody wants the gradient of the net's input: it is not computed
  int lds_job_floats;          // LDS of the parameter-gradient kernel
};

// the groups' slices of every trainable tensor and the gradient tensor each is added to
struct TinyMerge {
  const float *slices[TINY_MAX_TENSORS];
  float *g[TINY_MAX_TENSORS];
  int len[TINY_MAX_TENSORS], layer[TINY_MAX_TENSORS];
  int count[TINY_MAX_TENSORS];                       // slices (of the batch in use)
  int first_block[TINY_MAX_TENSORS + 1];
  int n;
};

// raises the kernel's LDS limit; once, outside any stream capture
int tiny_prepare();
// dev_plan: the plan in device memory (the kernel walks its layers by index, which a kernel
// argument passed by value would pay for with a private copy per thread); loss, softmax_xent:
// this step's loss and whether the closing softmax folds into it
int launch_tiny_step(const TinyPlan &plan, const TinyPlan *dev_plan, int loss, int softmax_xent, int batch,
                     const float *x, const float *t);
// Decides which layers' input gradients read a zero-framed dY, which products run on the matrix cores and
// which layers the front and back kernels take, and appends what that needs to the plan's LDS (lds_floats
// comes in as the floats in use so far; the caller checks the result against TINY_LDS_MAX_BYTES).
int tiny_layout(TinyPlan &plan);
// the largest batch that runs the front and back kernels (0: none)
int tiny_most_split(const TinyPlan &plan);
// How a batch's parameter gradients are split: samples of a layer's group, each of which leaves a slice; whether there is one group
// everywhere (which may be updated at once)
struct TinyGroups {
  int size[TINY_MAX_LAYERS];
  bool waves[TINY_MAX_LAYERS];   // a wave a channel pair
  bool one;
  int count(int layer, int batch) const { return ceil_div(batch, size[layer]); }
};
TinyGroups tiny_groups(const TinyPlan &plan, int batch);
// Every layer's weight and bias gradients (and the first layer's input gradient) from the outputs and
// gradients that launch_tiny_step left in memory. With `update` (one group everywhere) the optimizer's step
// on all tensors as well (powers_in, powers_out: as in launch_opt_update_multi), else the slices.
int launch_tiny_params(const TinyPlan &plan, const TinyPlan *dev_plan, const TinyGroups &groups, int batch, const float *x,
                       tdh_opt *update, int n_tensors, const float *powers_in, float *powers_out);
int launch_tiny_merge(const TinyMerge &m);

}  // namespace tdh
