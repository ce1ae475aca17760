// conv_any.h — what conv_any.hip (forward and dX of any window, stride and size), conv_dw_any.hip (dW) and the
// convolution's host side share: the packing of filters, and the sums of dW's slices, each of which runs as
// workgroups of the other gradient's launch where one call computes both. A launch of its own takes either
// some 4 us, of which its work is less than one.
#pragma once
#include "gemm_mfma.h"
#include "split_bf16.h"

namespace tdh {

typedef uint32_t uintx4_any __attribute__((ext_vector_type(4)));

// filters [m][kc][tap] (steps wm, wk floats) to parts [group of 8 kc][tap][part][m_pad][8]
struct AnyPack {
  const float *w;
  uintx4_any *wp;
  int M, KC, m_pad, wm, wk, total;
  int blocks, first;     // workgroups; the number of the first of them in a larger launch
  FastDiv div_m, div_rs;
};
// slices [splits][M][N] of a weight gradient, added up by gemm_mfma.h's tree
struct AnySums {
  const float *partial;
  int splits, M, N;
  int blocks, first_x;
  EpiDwDb epi;
};
int conv_any_dx_pack(const ConvShape &c, const float *w, AnyPack *pack);
// whether dX's launch can be that many workgroups larger
bool conv_any_dx_has_room(const ConvShape &c, int blocks);
// packed: the filters are (or will be, by a launch in front) packed; with: sums to take along
int conv_any_dx_run(const ConvShape &c, const float *dy, const float *w, float *dx, ActGrad ag, const AnyPack *packed,
                    const AnySums *with);
// pack: filters to pack along the way
int conv_dw_any_run(const ConvShape &c, const float *x, const float *dy, bool with_db, const float **partial, int *slices,
                    const AnyPack *pack);

namespace {

// thread = (group, tap, m)
__device__ __forceinline__ void any_pack_block(const AnyPack &p, const int block) {
  const int e = block * 256 + threadIdx.x;
  if (e >= p.total) return;
  uint32_t gt, m, g, t;
  p.div_m.divmod(e, gt, m);
  p.div_rs.divmod(gt, g, t);
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int kc  = 8 * static_cast<int>(g) + k;
    const bool on = static_cast<int>(m) < p.M && kc < p.KC;
    const float f = p.w[on ? static_cast<size_t>(m) * p.wm + static_cast<size_t>(kc) * p.wk + t : 0];
    v[k]          = on ? f * X3_SCALE : 0.0f;
  }
  uintx4_any part[X3_PARTS];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    uint32_t p3[X3_PARTS];
    split_pair(v[2 * c], v[2 * c + 1], p3);
#pragma unroll
    for (int q = 0; q < X3_PARTS; ++q) part[q][c] = p3[q];
  }
#pragma unroll
  for (int q = 0; q < X3_PARTS; ++q) p.wp[(static_cast<size_t>(gt) * X3_PARTS + q) * p.m_pad + m] = part[q];
}

// ANY_SUMS outputs a workgroup, four a lane, in splitk_reduce_block's tree. A workgroup of the larger launch holds its
// LDS and registers, so there are few of them, and each asks for up to 32 words at once.
constexpr int ANY_SUMS = 4 * REDUCE_OUTPUTS;
__device__ __forceinline__ void any_sums_block(const AnySums &s, const int block, float (*sm)[ANY_SUMS]) {
  const int o = threadIdx.x & (REDUCE_OUTPUTS - 1), g = threadIdx.x / REDUCE_OUTPUTS, mn = s.M * s.N;
  float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int z0 = g; z0 < s.splits; z0 += 8 * REDUCE_GROUPS) {
    float v[8][4];
#pragma unroll
    for (int u = 0; u < 8; ++u)   // (a slice past the last repeats it and is dropped)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[u][c] = s.partial[static_cast<size_t>(min(z0 + u * REDUCE_GROUPS, s.splits - 1)) * mn +
                            min(block * ANY_SUMS + c * REDUCE_OUTPUTS + o, mn - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (z0 + u * REDUCE_GROUPS < s.splits) {
#pragma unroll
        for (int c = 0; c < 4; ++c) sum[c] += v[u][c];
      }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) sm[g][c * REDUCE_OUTPUTS + o] = sum[c];
  __syncthreads();
  const int idx = block * ANY_SUMS + threadIdx.x;
  if (threadIdx.x < ANY_SUMS && idx < mn) {
    float t = sm[0][threadIdx.x];
#pragma unroll
    for (int i = 1; i < REDUCE_GROUPS; ++i) t += sm[i][threadIdx.x];
    const int m = idx / s.N, n = idx - m * s.N;
    s.epi.store(m, s.epi.col(n), t);
  }
}

}  // namespace
}  // namespace tdh
