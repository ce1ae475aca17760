// conv_pack.h — filters written into the layouts that the stride-1 kernels read (conv_s1.hip), by a launch of its own
// or by workgroups in front of those of a net's first convolution (conv_fwd_small.hip).
#pragma once
#include <climits>
#include <vector>

#include "conv_s1.h"
#include "split_bf16.h"

namespace tdh {

// The filters of several layers in one launch: job k owns the workgroups [first_block[k],
// first_block[k+1]). A launch of its own in every pass whose caller may have written the weights: bound by
// latency, so nothing is divided and a thread's loads are asked for together. us for 5x5, 32 -> 32 and
// 32 -> 64 channels, both directions' copies: one thread per weight with scattered stores 5.9.
// (A single job goes as a kernel of its own, with a tenth of the arguments and no search.)
struct PackPlan : PackJob {
  FastDiv div_rs, div_m, div_kc;
};
struct PackJobs {
  PackPlan job[CONV_PACK_JOBS];
  int first_block[CONV_PACK_JOBS];   // (past the last job: INT_MAX)
};

namespace {

// wp[t][kc][m]: forward (flip = 0): kc = ci, m = co, t as is; dX (flip = 1): kc = co, m = ci,
// tap reversed. An optional connection table zeroes unconnected (ci, co) pairs. e: element of wp.
__device__ __forceinline__ void pack_f32(const PackPlan &j, const int e) {
  const int rs = j.R * j.S;
  if (e >= j.C * j.Kc * rs) return;
  uint32_t rest, m, t, kc;
  j.div_m.divmod(e, rest, m);
  j.div_kc.divmod(rest, t, kc);
  const int co = j.flip ? kc : m, ci = j.flip ? m : kc;
  const float v = j.w[(static_cast<size_t>(co) * j.C + ci) * rs + (j.flip ? rs - 1 - t : t)];
  static_cast<float *>(j.wp)[e] = j.tbl && !j.tbl[ci * j.Kc + co] ? 0.0f : v;
}

// The filters of the three-part kernel: unit ((g*rs + t)*3 + part)*2 + half)*mc_pad + m holds the
// parts of channels 16g + 8*half .. +7 of row m (zero beyond the tensor), with the sign of step
// g*rs + t. A thread writes the
// three units of eight channels.
__device__ __forceinline__ void pack_x3(const PackPlan &j, const int e) {
  const int rs = j.R * j.S, KC = j.flip ? j.Kc : j.C, MC = j.flip ? j.C : j.Kc, mc_pad = j.div_m.d;
  uint32_t rest, m, g, t;
  j.div_m.divmod(e, rest, m);
  const int half = rest & 1;
  j.div_rs.divmod(rest >> 1, g, t);
  if (static_cast<int>(g) * 16 >= KC) return;
  const int step = (j.flip ? j.C : 1) * rs, kc0 = 16 * g + 8 * half;   // floats from one channel to the next
  const float *src = j.w + static_cast<size_t>(j.flip ? min(static_cast<int>(m), MC - 1) : min(static_cast<int>(m), MC - 1) * j.C) * rs +
                     (j.flip ? rs - 1 - t : t);
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = src[static_cast<size_t>(min(kc0 + k, KC - 1)) * step];
  const float sign = X3_SCALE * x3_sign(g * rs + t);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int kc = kc0 + k, co = j.flip ? kc : m, ci = j.flip ? m : kc;
    const bool in = kc < KC && static_cast<int>(m) < MC && (!j.tbl || j.tbl[ci * j.Kc + co]);
    v[k] = in ? sign * v[k] : 0.0f;
  }
  uint32_t part[X3_PARTS][4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t p3[X3_PARTS];
    split_pair(v[2 * k], v[2 * k + 1], p3);
#pragma unroll
    for (int p = 0; p < X3_PARTS; ++p) part[p][k] = p3[p];
  }
  uint4 *wp = static_cast<uint4 *>(j.wp);
#pragma unroll
  for (int p = 0; p < X3_PARTS; ++p)
    wp[((static_cast<size_t>(g * rs + t) * X3_PARTS + p) * 2 + half) * mc_pad + m] =
      make_uint4(part[p][0], part[p][1], part[p][2], part[p][3]);
}

__device__ __forceinline__ void pack_one(const PackPlan &j, const int e) {
  if (j.kind == CONV_PACK_X3)
    pack_x3(j, e);
  else
    pack_f32(j, e);
}

// thread t of the workgroups of 256 that the jobs take
__device__ __forceinline__ void pack_any(const PackJobs &jobs, const int t) {
  const int block = __builtin_amdgcn_readfirstlane(t >> 8);
  int k = 0;
#pragma unroll
  for (int i = 1; i < CONV_PACK_JOBS; ++i) k += jobs.first_block[i] <= block ? 1 : 0;
  pack_one(jobs.job[k], t - 256 * jobs.first_block[k]);
}

}  // namespace

// the jobs as a kernel takes them; their workgroups and bytes
void plan_packs(const PackJob *jobs, int n, PackJobs *p, int *blocks, double *bytes);
std::vector<PackJob> take_left_packs();

}  // namespace tdh
