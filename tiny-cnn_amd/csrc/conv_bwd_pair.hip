// conv_bwd_pair.hip — dX and dW (and db) of a 5x5 convolution on small images as ONE launch: the
// workgroups of conv_x3_body.h (dX, 32 channels x 128 pixels each) and, behind them, those of
// conv_dw_img.h (dW). Both read dY and neither reads what the other writes.
//
// Each of the two alone is about one workgroup, four waves, per compute unit, and half of its time a
// wave waits: for its first loads, for the other waves between two chunks, for the sums at the end.
// Together two workgroups sit on a compute unit (72 KB of LDS each, 256 registers a wave) and one
// multiplies while the other waits. On two streams the kernels overlap as well, but a fork and a
// join cost a replayed step 5 us each.
//
// dX shares its filter taps out to the waves, because a wave that keeps to 32 pixels of its own
// reads more filter operands than its products cover (alone, 16x16 images, 32 -> 32 channels, batch
// 128: 25 us; in fp32 21). us, two launches / this one with dX in fp32 / as it is, batch 128:
// 16x16, 32 -> 32 channels 42.7 / 36.5 / 31.3; 8x8, 32 -> 64 28.2 / 23.3 / 19.8. Bound: MFMA issue,
// the weight gradient's in fp32.
#include <algorithm>

#include "conv_dw_img.h"
#include "conv_x3_body.h"

namespace tdh {

namespace {

template <int IS>
__global__ void __launch_bounds__(256, 2)
conv_bwd_pair_kernel(const ConvS1Args dx, const DwImgArgs dw, const int dx_blocks, const FastDiv div_tiles,
                     const FastDiv div_m) {
  const int id = blockIdx.x;
  if (id >= dx_blocks) {
    dw_img_workgroup<IS>(dw, id - dx_blocks, gridDim.x - dx_blocks);
    return;
  }
  uint32_t rest, tile, m, split;
  div_tiles.divmod(id, rest, tile);
  div_m.divmod(rest, split, m);
  conv_x3_workgroup<5, 5, IS, 1, 1, true, true>(dx, tile, m, split);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

bool conv_bwd_pair_applicable(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph, int pw) {
  return make_dw_img_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw).ok &&
         make_s1_pair_plan(R, S, batch, Kc, C, OH, OW, H, W, R - 1 - ph, S - 1 - pw).ok;
}

static size_t slices_bytes(const DwImgPlan &im, int Kc, int crs) {
  return ws_align(sizeof(float) * static_cast<size_t>(im.slices) * Kc * crs) +
         ws_align(sizeof(float) * static_cast<size_t>(im.slices) * Kc);
}

size_t conv_bwd_pair_workspace_bytes(int R, int S, int batch, int C, int Kc, int H, int W, int ph, int pw) {
  return plan_workspace_bytes(make_s1_pair_plan(R, S, batch, Kc, C, H, W, H, W, R - 1 - ph, S - 1 - pw), R * S) +
         slices_bytes(make_dw_img_plan(R, S, batch, C, Kc, H, W, H, W, ph, pw), Kc, C * R * S);
}

// The caller has checked conv_bwd_pair_applicable and reserved the workspace of both gradients.
// prepacked: this filter packed for dX (read where it is in three parts), or none.
int conv_bwd_pair_run(int R, int S, int batch, int C, int Kc, int H, int W, int ph, int pw, const float *x, const float *dy,
                      const float *w, PackedFilters prepacked, float *dx, ActGrad dx_act, float *dw, float *db,
                      int accumulate) {
  S1Plan p     = make_s1_pair_plan(R, S, batch, Kc, C, H, W, H, W, R - 1 - ph, S - 1 - pw);
  DwImgPlan im = make_dw_img_plan(R, S, batch, C, Kc, H, W, H, W, ph, pw);
  if (!p.ok || !im.ok || !aligned16(x) || !aligned16(dy))
    return set_error(TDH_ERR_INVALID, "conv_bwd_pair_run: shape not supported");
  const int crs  = C * R * S;
  const void *wp = prepacked.data;
  if (!wp || prepacked.kind != CONV_PACK_X3) {
    void *fresh = nullptr;
    TDH_TRY(ws_take(conv_s1_packed_bytes(CONV_PACK_X3, R * S, Kc, C), &fresh));
    const PackJob job{w, nullptr, fresh, C, Kc, R, S, CONV_PACK_X3, 1};
    TDH_TRY(conv_pack_filters(&job, 1));
    wp = fresh;
  }
  ConvS1Args &a = p.args;
  a.in = dy; a.wp = wp; a.bias = nullptr; a.out = dx; a.ag = dx_act;
  a.w = w; a.tbl = nullptr; a.flip = 1;
  a.act_out = nullptr; a.act_kind = TDH_ACT_NONE;
  a.pool_out = nullptr; a.pool_argmax = nullptr; a.pool_act_out = nullptr;
  if (p.splits > 1) {
    void *part = nullptr;
    TDH_TRY(ws_take(sizeof(float) * p.splits * a.part_stride, &part));
    a.part = static_cast<float *>(part);
  }
  void *part = nullptr, *part_db = nullptr;
  TDH_TRY(ws_take(sizeof(float) * static_cast<size_t>(im.slices) * Kc * crs, &part));
  if (db) TDH_TRY(ws_take(sizeof(float) * static_cast<size_t>(im.slices) * Kc, &part_db));
  im.args.x = x; im.args.dy = dy;
  im.args.partial = static_cast<float *>(part); im.args.partial_db = static_cast<float *>(part_db);
  {
    ProfScope prof("conv_bwd_pair", 2.0 * batch * H * W * Kc * (2.0 * crs + (db ? 1 : 0)), WORK_FLOP);
    static bool raised[2] = {false, false};
    const int which = im.size == 8 ? 0 : 1;
    void (*kernel)(const ConvS1Args, const DwImgArgs, int, FastDiv, FastDiv) =
        which ? conv_bwd_pair_kernel<16> : conv_bwd_pair_kernel<8>;
    if (!raised[which]) {  // (80 KB: two workgroups a compute unit, as the plans promise)
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  80 * 1024));
      raised[which] = true;
    }
    const int dx_blocks = p.grid.x * p.grid.y * p.grid.z;
    TDH_LAUNCH(kernel, dim3(dx_blocks + im.workgroups), dim3(256), std::max(p.lds_bytes, im.lds_bytes), ctx().stream,
               a, im.args, dx_blocks, FastDiv(p.grid.x), FastDiv(p.grid.y));
    TDH_LAUNCH_CHECK();
  }
  if (p.splits > 1) TDH_TRY(finish_s1_split(p, nullptr, dx_act, dx, nullptr, TDH_ACT_NONE));
  return conv_dw_sum_slices(part, part_db, im.slices, Kc, crs, dw, db, accumulate);
}

}  // namespace tdh
