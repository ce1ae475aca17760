// conv_s1.hip — host side of the stride-1 convolution (forward and dX) on the LDS-halo MFMA
// kernel of conv_s1_inst.hip: tile choice, filter repacking, split-K reduction.
#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "conv_pack.h"

namespace tdh {

namespace {

// out = part[0] + part[1] + ... (in this order) (+ bias[m]) (* act'(y)); four elements per
// thread when a channel plane is a multiple of four
template <int VEC>
__global__ void __launch_bounds__(256)
s1_split_reduce_kernel(const SplitSum sum, float *__restrict__ act_out, const int act_kind) {
  const size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * VEC;
  if (i >= sum.stride) return;
  float v[VEC];
  split_sum_values<VEC>(sum, i, v);
  if (act_out) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) act_out[i + e] = act_apply(act_kind, v[e]);
  }
}

int launch_split_reduce(const SplitSum &sum, int plane, float *act_out, int act_kind) {
  const size_t total = sum.stride;
  ProfScope prof("conv_s1_split_reduce", 4.0 * total * (sum.splits + 1 + (sum.ag.kind != TDH_ACT_NONE)),
                 WORK_BYTE);
  if (plane % 4 == 0)
    TDH_LAUNCH((s1_split_reduce_kernel<4>), dim3(static_cast<unsigned>(ceil_div_sz(total / 4, 256))), dim3(256), 0,
               ctx().stream, sum, act_out, act_kind);
  else
    TDH_LAUNCH((s1_split_reduce_kernel<1>), dim3(static_cast<unsigned>(ceil_div_sz(total, 256))), dim3(256), 0,
               ctx().stream, sum, act_out, act_kind);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

__global__ void __launch_bounds__(256) pack_filters_kernel(const PackJobs jobs) { pack_any(jobs, blockIdx.x * 256 + threadIdx.x); }
__global__ void __launch_bounds__(256) pack_filter_kernel(const PackPlan j) { pack_one(j, blockIdx.x * 256 + threadIdx.x); }

int pow2_ceil(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}
int ilog2(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

// Splits the reduction channels over grid.z when the tiles alone leave most of the chip idle.
void choose_split(S1Plan &p, int kch, long blocks) {
  const int nchunks = ceil_div(p.args.KC, kch);
  int splits = 1;
  if (blocks < 384 && nchunks >= 4) {
    splits = static_cast<int>(std::min<long>(8, (512 + blocks - 1) / blocks));
    splits = std::min(splits, nchunks / 2);
    // still under half the chip: one chunk per workgroup
    if (blocks * splits <= 128) splits = static_cast<int>(std::min<long>(nchunks, 256 / blocks));
  } else if (blocks <= 128 && nchunks >= 2) {
    splits = 2;  // half the chip would idle: one chunk per workgroup is still the better deal
  }
  const int per      = ceil_div(nchunks, splits) * kch;
  p.splits           = ceil_div(p.args.KC, per);
  p.args.kc_split    = p.splits > 1 ? per : p.args.KC;
  p.args.part        = nullptr;
  p.args.part_stride = static_cast<size_t>(p.args.batch) * p.args.MC * p.args.OH * p.args.OW;
  p.grid.z           = p.splits;
}

// Shape-only choice of the tile geometry; ok = false sends the caller to the generic GEMM.
// Candidates run from the largest workgroup tile to the smallest; the first one that yields
// at least 256 workgroups wins, else the one with the most workgroups, and shapes that cannot
// even fill a quarter of the chip are left to the split-K GEMM.
// by_taps: the three-part kernel's workgroup of 32 channels x 128 pixels that the waves share by
// filter taps (conv_bwd_pair.hip), however few of them, and split over the reduction channels.
S1Plan make_plan_of(bool x3, int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph,
                    int pw, bool by_taps = false) {
  S1Plan best;
  best.ok = false;
  best.x3 = x3;
  if (R != S || !(R == 3 || R == 5 || (x3 && (R == 1 || R == 7)))) return best;
  if (MC < 16 || KC < 8 || OW < 4 || OH < 1 || pw > 4) return best;
  // offsets inside the input are 32-bit
  if (static_cast<long>(batch) * KC * IH * IW >= (1L << 31)) return best;
  static const int cand_wide[3][2]   = {{2, 2}, {2, 1}, {1, 1}};  // MC > 32
  static const int cand_narrow[3][2] = {{1, 4}, {1, 2}, {1, 1}};  // MC <= 32
  // (three parts: tiles of at least two accumulator blocks a wave, or the filter operands that a
  // wave reads for every tap are more than its products cover: 16x16 images, 32 -> 32 channels, 5x5,
  // batch 128: 25 us with one block, 21 in fp32)
  const int n_cand = !x3 || by_taps ? 3 : MC > 32 ? 2 : 1;
  long best_blocks = 0;
  for (int ci = by_taps ? 2 : 0; ci < n_cand; ++ci) {
    S1Plan p;
    p.ok = false;
    p.x3 = x3;
    const int *narrow = cand_narrow[x3 && !by_taps ? 1 : ci];
    p.tc = OW >= 48 ? 64 : OW >= 24 ? 32 : OW >= 12 ? 16 : 8;
    p.tm = MC > 32 ? cand_wide[ci][0] : narrow[0];
    p.tn = MC > 32 ? cand_wide[ci][1] : narrow[1];
    const int pix = 128 * p.tn;
    if (pix < p.tc) continue;
    int tr = pix / p.tc;
    if (tr > pow2_ceil(OH)) tr = pow2_ceil(OH);
    const int ti = pix / (tr * p.tc);
    ConvS1Args &a = p.args;
    a.batch = batch; a.KC = KC; a.MC = MC; a.IH = IH; a.IW = IW; a.OH = OH; a.OW = OW;
    a.ph = ph; a.pw = pw; a.pwa = (pw + 3) & ~3;
    a.TR = tr; a.TI = ti; a.log_tr = ilog2(tr); a.log_ti = ilog2(ti);
    a.tiles_x = ceil_div(OW, p.tc);
    a.tiles_y = ceil_div(OH, tr);
    const int nq     = (3 + p.tc + S - 1 + 3) / 4;
    const int planeq = ti * (tr + R - 1) * nq;
    a.div_rows = FastDiv((tr + R - 1) * nq);
    const int kch = x3 ? X3_KCH : s1_kch(R * S, p.tm, p.tn);
    if (x3) {
      if (2 * planeq > 256 * x3_items(p.tm, p.tn)) continue;
      p.lds_bytes = 6 * 16 * 4 * static_cast<size_t>(planeq);
      if (p.lds_bytes > 80 * 1024) continue;  // two workgroups a compute unit
      if (static_cast<long>(ti) * KC * IH * IW >= (1L << 29)) continue;  // 32-bit byte offsets inside a tile
      a.mc_pad = x3_mc_pad(MC);
      if (by_taps) p.lds_bytes = std::max<size_t>(p.lds_bytes, 64 * 1024);  // (the waves' sums)
    } else {
      if (ceil_div(planeq, 256 / kch) > s1_niq(R, S, p.tc, p.tm, p.tn)) continue;
      p.lds_bytes = sizeof(float) * kch * (4 * static_cast<size_t>(planeq) + R * S * 32 * p.tm);
      if (p.lds_bytes > 150 * 1024) continue;
    }
    const long tiles  = static_cast<long>(a.tiles_x) * a.tiles_y * ceil_div(batch, ti);
    const long blocks = tiles * ceil_div(MC, 32 * p.tm);
    if (tiles > 2000000000L) continue;
    p.grid = dim3(static_cast<unsigned>(tiles), ceil_div(MC, 32 * p.tm), 1);
    p.ok   = true;
    if (x3) {
      // unsplit, and a workgroup for every compute unit at least; two where a single short chunk has
      // nothing to cover its loads with (32x32 images, 16 -> 32 channels, 3x3, batch 64: 12.6 us with
      // one a unit, 11.2 in fp32)
      if (by_taps) {
        choose_split(p, kch, blocks);
        return p;
      }
      if (blocks < (KC * R * S < 256 ? 512 : 256)) continue;
      p.splits = 1;
      a.kc_split = KC; a.part = nullptr; a.part_stride = 0;
      return p;
    }
    choose_split(p, kch, blocks);
    // short reductions have nothing to overlap their loads with inside a workgroup: ask for
    // more, smaller workgroups then
    if (blocks >= (KC * R * S < 256 ? 1024 : 256)) return p;
    if (blocks > best_blocks) {
      best_blocks = blocks;
      best        = p;
    }
  }
  if (best_blocks * (best.ok ? best.splits : 1) < 128) best.ok = false;
  return best;
}

S1Plan make_plan(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw) {
  if (!ctx().keep_f32) {
    const S1Plan p = make_plan_of(true, R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
    if (p.ok) return p;
  }
  return make_plan_of(false, R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

S1Plan make_s1_pair_plan(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw) {
  S1Plan p;
  p.ok = false;
  if (!ctx().keep_f32) p = make_plan_of(true, R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw, true);
  return p;
}

bool conv_s1_applicable(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW,
                        int ph, int pw) {
  return make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw).ok;
}

// The share of its tiles' outputs that exist, of the fp32 kernel's (1 where another one runs), and the estimated us of that
// kernel with its packing and split sum: whole rounds of the workgroups, fitted to 800 shapes of poorly filled tiles
// (12 % rms).
double conv_s1_fill(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw, double *us) {
  *us = 0.0;
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  if (!p.ok || p.x3) return 1.0;
  const double products = p.args.kc_split * R * S / 2 * p.tm * p.tn * 64 / 2400.0;   // of a workgroup, us of its matrix instructions
  const double full     = static_cast<double>(p.grid.x) * p.grid.y * p.splits / 256;
  const int resident    = p.lds_bytes <= 80 * 1024 ? 2 : 1;
  auto round = [&](double at_once) { return 2.8 + 1.6 * products * at_once; };
  const double whole = std::floor(full / resident), left = std::ceil(full - whole * resident);
  *us = 6.4 + whole * round(resident) + (left > 0 ? round(left) : 0.0) + (p.splits > 1 ? 0.6 : 0.0);
  const double in_tiles = 128.0 * p.tn * p.grid.x * (32.0 * p.tm * p.grid.y);
  return static_cast<double>(batch) * OH * OW * MC / in_tiles;
}

int conv_s1_packed_kind(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw) {
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  return !p.ok ? CONV_PACK_NONE : p.x3 ? CONV_PACK_X3 : CONV_PACK_F32;
}
size_t conv_s1_packed_bytes(int kind, int RS, int KC, int MC) {
  return kind == CONV_PACK_X3 ? x3_pack_bytes(RS, KC, MC) : sizeof(float) * static_cast<size_t>(RS) * KC * MC;
}

bool conv_s1_single_pass(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW,
                         int ph, int pw) {
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  return p.ok && p.splits == 1;
}

// A wave must hold whole 2x2 windows: in a 32-pixel accumulator block (rows of 8 or 16 pixels; tile rows
// come in powers of two and start at even image rows) or in two of them (s1_block_pixel), with even image sizes and
// one pass over the reduction channels (the partial sums of a split have no maximum yet).
bool conv_s1_fuses_pool(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW,
                        int ph, int pw) {
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  return p.ok && p.splits == 1 && (p.tc <= 16 || (p.tn % 2 == 0 && !(p.x3 && p.tc == 64))) && p.args.TR >= 2 && OH % 2 == 0 && OW % 2 == 0 &&
         static_cast<long>(MC) * OH * OW < (1L << 31);
}

// tiles of rows of 8 or 16 pixels
bool conv_s1_short_rows(int R, int S, int batch, int KC, int MC, int IH, int IW, int OH, int OW, int ph, int pw) {
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  return p.ok && p.tc <= 16;
}

// packed filters and the partial sums of a split
size_t plan_workspace_bytes(const S1Plan &p, int RS) {
  const size_t packed = ws_align(conv_s1_packed_bytes(p.x3 ? CONV_PACK_X3 : CONV_PACK_F32, RS, p.args.KC, p.args.MC));
  return packed + (p.splits > 1 ? ws_align(sizeof(float) * p.splits * p.args.part_stride) : 0);
}

size_t conv_s1_workspace_bytes(int R, int S, int batch, int C, int Kc, int flip, int IH, int IW,
                               int OH, int OW, int ph, int pw) {
  const int KC = flip ? Kc : C, MC = flip ? C : Kc;
  size_t most = 0;
  for (int k = 0; k < 3; ++k) {  // (which of the kernels runs is the caller's choice as well)
    const S1Plan p = make_plan_of(k != 0, R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw, /*by_taps=*/k == 2);
    if (p.ok) most = std::max(most, plan_workspace_bytes(p, R * S));
  }
  return most;
}

size_t conv_s1_run_workspace_bytes(int R, int S, int batch, int C, int Kc, int flip, int IH, int IW,
                                   int OH, int OW, int ph, int pw) {
  const int KC = flip ? Kc : C, MC = flip ? C : Kc;
  const S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  return p.ok ? plan_workspace_bytes(p, R * S) : 0;
}

void plan_packs(const PackJob *jobs, int n, PackJobs *p, int *blocks, double *bytes) {
  *blocks = 0;
  *bytes  = 0.0;
  for (int k = 0; k < CONV_PACK_JOBS; ++k) {
    p->first_block[k] = k < n ? *blocks : INT_MAX;
    if (k >= n) continue;
    PackPlan &j = p->job[k];
    static_cast<PackJob &>(j) = jobs[k];
    const bool x3 = j.kind == CONV_PACK_X3;
    const int rs = j.R * j.S, KC = j.flip ? j.Kc : j.C, MC = j.flip ? j.C : j.Kc;
    j.div_rs = FastDiv(rs);
    j.div_m  = FastDiv(x3 ? x3_mc_pad(MC) : MC);
    j.div_kc = FastDiv(KC);
    *blocks += ceil_div(x3 ? ceil_div(KC, 16) * rs * 2 * x3_mc_pad(MC) : rs * KC * MC, 256);
    *bytes += (x3 ? 10.0 : 8.0) * rs * KC * MC;
  }
}

int conv_pack_filters(const PackJob *jobs, int n) {
  for (int at = 0; at < n; at += CONV_PACK_JOBS) {
    PackJobs p;
    const int here = std::min(CONV_PACK_JOBS, n - at);
    int blocks;
    double bytes;
    plan_packs(jobs + at, here, &p, &blocks, &bytes);
    ProfScope prof("conv_repack_weights", bytes, WORK_BYTE);
    if (here == 1)
      TDH_LAUNCH(pack_filter_kernel, dim3(blocks), dim3(256), 0, ctx().stream, p.job[0]);
    else
      TDH_LAUNCH(pack_filters_kernel, dim3(blocks), dim3(256), 0, ctx().stream, p);
    TDH_LAUNCH_CHECK();
  }
  return TDH_OK;
}

// Jobs that the next launch of a first convolution takes along.
static thread_local std::vector<PackJob> left_packs;
void conv_pack_leave(const PackJob *jobs, int n) { left_packs.assign(jobs, jobs + n); }
bool conv_packs_left() { return !left_packs.empty(); }
std::vector<PackJob> take_left_packs() { return std::exchange(left_packs, {}); }
int conv_pack_finish() {
  const std::vector<PackJob> jobs = take_left_packs();
  return conv_pack_filters(jobs.data(), static_cast<int>(jobs.size()));
}

// Runs out = conv(in, repack(w)) (+ bias) (* act'(y)); the caller has checked applicability
// and reserved conv_s1_workspace_bytes of scratch. flip = 0: forward, 1: dX. w: the filters, masked by
// tbl_dev unless null. prepacked: the result of conv_pack_filters for them, when the caller already
// has it in the layout of the kernel that runs.
int conv_s1_run(int R, int S, int batch, int C, int Kc, int flip, const float *in, const float *w,
                const uint8_t *tbl_dev, const float *bias, float *out, int IH, int IW, int OH,
                int OW, int ph, int pw, ActGrad ag, const char *tag, PackedFilters prepacked,
                float *act_out, int act_kind, const PoolFuse *pool) {
  const int KC = flip ? Kc : C, MC = flip ? C : Kc;
  S1Plan p = make_plan(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw);
  if (!p.ok) return set_error(TDH_ERR_INVALID, "conv_s1_run: shape not supported");
  if (pool && (flip || !pool->out || !pool->argmax ||
               (pool->act_out && pool->act_kind != TDH_ACT_RELU) ||
               !conv_s1_fuses_pool(R, S, batch, KC, MC, IH, IW, OH, OW, ph, pw)))
    return set_error(TDH_ERR_INVALID, "conv_s1_run: this shape does not compute the pool layer behind it");
  if (!out && !pool && !(act_out && p.splits == 1))
    return set_error(TDH_ERR_INVALID, "conv_s1_run: no output tensor");
  const void *wp = prepacked.data;
  if (!wp || prepacked.kind != (p.x3 ? CONV_PACK_X3 : CONV_PACK_F32)) {
    void *fresh = nullptr;
    TDH_TRY(ws_take(conv_s1_packed_bytes(p.x3 ? CONV_PACK_X3 : CONV_PACK_F32, R * S, KC, MC), &fresh));
    const PackJob job{w, tbl_dev, fresh, C, Kc, R, S, p.x3 ? CONV_PACK_X3 : CONV_PACK_F32, flip};
    TDH_TRY(conv_pack_filters(&job, 1));
    wp = fresh;
  }
  p.args.in = in; p.args.wp = wp; p.args.bias = bias;
  p.args.w = w; p.args.tbl = tbl_dev; p.args.flip = flip;
  p.args.out = out; p.args.ag = ag;
  p.args.act_out = act_out; p.args.act_kind = act_kind;
  p.args.pool_out     = pool ? pool->out : nullptr;
  p.args.pool_argmax  = pool ? pool->argmax : nullptr;
  p.args.pool_act_out = pool ? pool->act_out : nullptr;
  if (p.splits > 1) {
    void *part = nullptr;
    TDH_TRY(ws_take(sizeof(float) * p.splits * p.args.part_stride, &part));
    p.args.part = static_cast<float *>(part);
  }
  {
    const char *name = !p.x3 ? (pool ? "conv_fwd_s1_pool" : tag) : pool ? "conv_fwd_x3_pool" : flip ? "conv_dx_x3" : "conv_fwd_x3";
    ProfScope prof(name, MC, batch * OH * OW, KC * R * S);
    const bool vec = IW % 4 == 0 && aligned16(in) && (p.x3 || (MC % 4 == 0 && aligned16(wp)));
    if (p.x3 && vec)
      TDH_TRY(R == 1 ? x3_launch_1_vec(p) : R == 3 ? x3_launch_3_vec(p) : R == 5 ? x3_launch_5_vec(p) : x3_launch_7_vec(p));
    else if (p.x3)
      TDH_TRY(R == 1 ? x3_launch_1_scalar(p) : R == 3 ? x3_launch_3_scalar(p) : R == 5 ? x3_launch_5_scalar(p) : x3_launch_7_scalar(p));
    else if (vec) TDH_TRY(R == 3 ? s1_launch_3x3_vec(p) : s1_launch_5x5_vec(p));
    else TDH_TRY(R == 3 ? s1_launch_3x3_scalar(p) : s1_launch_5x5_scalar(p));
  }
  return p.splits > 1 ? finish_s1_split(p, bias, ag, out, act_out, act_kind) : TDH_OK;
}

// out from the partial sums of a split: left to the kernel that reads `out` next, if the caller has
// asked for that (it adds the partials up and writes `out`), or launched here
int finish_s1_split(const S1Plan &p, const float *bias, ActGrad ag, float *out, float *act_out, int act_kind) {
  SplitSum sum;
  sum.part = p.args.part; sum.splits = p.splits; sum.stride = p.args.part_stride;
  sum.bias = bias; sum.MC = p.args.MC; sum.div_plane = FastDiv(p.args.OH * p.args.OW); sum.ag = ag; sum.out = out;
  if (ctx().leave_split_sum && !act_out) {
    left_split_sum()     = sum;
    ctx().split_sum_left = true;
    return TDH_OK;
  }
  return launch_split_reduce(sum, p.args.OH * p.args.OW, act_out, act_kind);
}

SplitSum &left_split_sum() {
  static SplitSum sum;
  return sum;
}

int finish_split_sum() {
  if (!ctx().split_sum_left) return TDH_OK;
  ctx().split_sum_left = false;
  const SplitSum &sum = left_split_sum();
  return launch_split_reduce(sum, static_cast<int>(sum.div_plane.d), nullptr, TDH_ACT_NONE);
}

}  // namespace tdh
