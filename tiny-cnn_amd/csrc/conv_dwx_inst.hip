// conv_dwx_inst.hip — weight gradient of a stride-1 convolution on the bf16 matrix cores with
// three-part operands (split_bf16.h):
//
//   dW[co][ci][fy][fx] = sum_{img,oy,ox} dY[img][co][oy][ox] * X[img][ci][oy+fy-ph][ox+fx-pw]
//
// M = output channels, N = input channels, K = output pixels, 16 neighbours of a row per
// v_mfma_f32_32x32x16_bf16 (8 per half wave), one accumulator block per filter tap. Bound: bf16
// MFMA issue.
//
// A workgroup (one a compute unit) owns 32*COB x 32*CIB channels and RW filter rows and walks down columns of TC pixels, 64/TC rows a step. X rows live in a ring in LDS and serve
// every filter row that meets them, so a step brings in only its own rows of X and dY: loaded as
// 16-byte words while the step before is multiplied, split once, stored as
// [row][part][channel][pixel] bf16 (channel rows an odd number of 16-byte words apart: 32 lanes
// reading 16 bytes each hit all banks evenly). A new image, or the start of a slice in the middle of
// one, first runs the steps that only fill the ring.
//
// A lane's eight X values of a tap start fx pixels into the row: it reads two aligned 16-byte words
// per part and filter row and takes the taps out of them with a shift of two bytes where fx is
// odd, so a row's taps cost two reads a part. The waves are RW filter rows x COB x CIB channel blocks x
// KS = 4/(COB*CIB) shares of the step's four 16-pixel groups (12 waves of 3 accumulators each for a
// 3x3 window: all nine in one wave left no registers to read ahead). Shares are added
// through LDS at the end and the workgroup writes one slice [slice][co][ci][tap], which the split
// reduction adds up in order.
// us, fp32 kernel / here (batch 64): 64 -> 64 channels of 128x128 591 / 440, 128 -> 128 of 64x64 581 /
// 391, 64 -> 128 of 64x64 296 / 212, 32 -> 64 of 64x64 88 / 74 (131-110 to 198-130 TFLOP/s).
#include "conv_dwx.h"
#include "split_bf16.h"

namespace tdh {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr unsigned DWX_NOWHERE = 0x80000000u;  // past the end of every tensor's images

// eight consecutive bf16 starting at element AT of the sixteen in w
template <int AT>
__device__ __forceinline__ bf16x8 take8(const uint32_t (&w)[8]) {
  uintx4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = AT % 2 == 0 ? w[AT / 2 + i] : __builtin_amdgcn_alignbit(w[AT / 2 + i + 1 < 8 ? AT / 2 + i + 1 : 7], w[AT / 2 + i], 16);
  return __builtin_bit_cast(bf16x8, r);
}

// acc[fx] += sign * d * (the eight values from AT + fx on of w), tap after tap
template <int AT, int S>
__device__ __forceinline__ void add_taps(floatx16 *acc, const bf16x8 (&d)[X3_PARTS], const uint32_t (&w)[X3_PARTS][8],
                                         const float sign) {
  const bf16x8 x[1][X3_PARTS] = {{take8<AT>(w[0]), take8<AT>(w[1]), take8<AT>(w[2])}};
  const bf16x8 dd[1][X3_PARTS] = {{d[0], d[1], d[2]}};
  mfma_x3<1, 1>(reinterpret_cast<floatx16(&)[1][1]>(*acc), dd, x, sign);
  if constexpr (S > 1) add_taps<AT + 1, S - 1>(acc + 1, d, w, sign);
}

// The wave's infinite and NaN sums once more in fp32 (split_bf16.h), over the slice's rows and its TC
// columns: lane l brings output channel co and input channel ci, l%32 of their blocks, at pixel
// p + l/32. Eight pixels are asked for together.
template <int S, int TC, int RPS>
__device__ __forceinline__ void dwx_redo_exceptional(const DwxArgs &a, floatx16 (&acc)[S], const int lane, const int co,
                                                     const int ci, const int fy, const int x0, const int slice) {
  // (hidden from the compiler, which otherwise keeps the comparisons for the stores behind)
  int rows = a.Kc - (co - (lane & 31)) - 4 * (lane >> 5);   // from this lane's first element
  asm volatile("" : "+v"(rows));
  x3_redo(acc, [&](int, int r) { return ci < a.C && 8 * (r >> 2) + (r & 3) < rows; }, [&](floatx16 (&sum)[S]) {
    const int end = min(a.chunks_total, (slice + 1) * a.chunks_per_slice);
#pragma unroll 1
    for (int chunk = slice * a.chunks_per_slice; chunk < end; ++chunk) {
      const int img = chunk / a.chunks_per_image, y0 = RPS * (chunk % a.chunks_per_image);
      const float *dy = a.dy + (static_cast<size_t>(img) * a.Kc + (co < a.Kc ? co : 0)) * a.OH * a.OW;
      const float *x  = a.x + (static_cast<size_t>(img) * a.C + (ci < a.C ? ci : 0)) * a.H * a.W;
#pragma unroll 1
      for (int p0 = lane >> 5; p0 < 64; p0 += 8) {
        float d[4], v[4][S];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int p = p0 + 2 * k, oy = y0 + p / TC, ox = x0 + p % TC, iy = oy + fy - a.ph;
          const bool on = oy < a.OH && ox < a.OW;
          d[k] = on && co < a.Kc ? dy[oy * a.OW + ox] : 0.0f;
#pragma unroll
          for (int fx = 0; fx < S; ++fx) {
            const int ix  = ox + fx - a.pw;
            const bool in = on && ci < a.C && static_cast<unsigned>(iy) < static_cast<unsigned>(a.H) &&
                            static_cast<unsigned>(ix) < static_cast<unsigned>(a.W);
            v[k][fx] = in ? x[iy * a.W + ix] : 0.0f;
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int fx = 0; fx < S; ++fx) sum[fx] = __builtin_amdgcn_mfma_f32_32x32x2f32(d[k], v[k][fx], sum[fx], 0, 0, 0);
      }
      if (x3_all_nan(sum)) return;
      if (chunk == slice * a.chunks_per_slice) {
        // A NaN anywhere in dY's channel makes NaN of all of that channel's sums: the channels that still
        // have a number are looked through, a step of 64 pixels to a load, as far as an image goes (a
        // few channels with a NaN here and there would take the loop around this one through all
        // of it: 64 images of 64x64, 128 -> 128 channels, 970 us, so 358).
        uint32_t need = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          bool number = false;
#pragma unroll
          for (int fx = 0; fx < S; ++fx) number = number || sum[fx][r] == sum[fx][r];
          const uint64_t lanes = __ballot(number);
          const int row        = 8 * (r >> 2) + (r & 3);   // of lanes 0-31; lanes 32-63 hold row + 4
          need |= (static_cast<uint32_t>(lanes) != 0 ? 1u : 0u) << row | ((lanes >> 32) != 0 ? 1u : 0u) << (row + 4);
        }
        uint32_t nan_rows = 0;
        while (need) {
          const int row = __builtin_ctz(need), channel = co - (lane & 31) + row;
          need &= need - 1;
          for (int c0 = chunk; c0 < min(end, chunk + a.chunks_per_image); c0 += 8) {
            bool nan = false;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              const int c = min(c0 + k, end - 1), i = c / a.chunks_per_image;
              const int oy = RPS * (c - i * a.chunks_per_image) + lane / TC, ox = x0 + lane % TC;
              const float d = oy < a.OH && ox < a.OW && channel < a.Kc
                                ? a.dy[(static_cast<size_t>(i) * a.Kc + channel) * a.OH * a.OW + oy * a.OW + ox] : 0.0f;
              nan = nan || d != d;
            }
            if (__any(nan)) {
              nan_rows |= 1u << row;
              break;
            }
          }
        }
        nan_rows >>= 4 * (lane >> 5);
#pragma unroll
        for (int fx = 0; fx < S; ++fx)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (nan_rows >> (8 * (r >> 2) + (r & 3)) & 1u) sum[fx][r] = __builtin_nanf("");
        if (x3_all_nan(sum)) return;
      }
    }
  });
}

template <int RW, int S, int TC, int COB, int CIB, int SHIFT, bool VEC>
__global__ void __launch_bounds__(dwx_threads(RW), dwx_threads(RW) / 256) conv_dwx_kernel(const DwxArgs a) {
  constexpr int RPS  = 64 / TC;                     // output rows a step
  constexpr int NQ   = dwx_words(TC, S);            // 4-pixel words of a staged X row
  constexpr int XPX  = 4 * NQ;                      // pixels of a staged X row
  constexpr int NR   = RW - 1 + RPS;                // ring rows
  constexpr int NCI  = 32 * CIB, NCO = 32 * COB;
  constexpr int NT   = dwx_threads(RW);
  constexpr int KS   = 4 / (COB * CIB);
  constexpr int GPW  = 4 / KS;                      // 16-pixel groups a wave takes per step
  constexpr int XROW = X3_PARTS * NCI * XPX;        // bf16 elements of a ring row
  constexpr int DYP  = 72;                          // pixels per staged dY channel
  constexpr int XI   = (RPS * NCI * NQ + NT - 1) / NT;  // X words a thread stages per step
  constexpr int DI   = (NCO * 16 + NT - 1) / NT;           // dY words
  constexpr int WARM = (RW - 1 + RPS - 1) / RPS;    // steps that only fill the ring
  static_assert(SHIFT + S - 1 + 8 <= 16, "two words cover all taps of a row");
  static_assert((XPX / 8) % 2 == 1, "channel rows an odd number of 16-byte words apart");

  extern __shared__ __align__(16) uint16_t lds[];
  uint16_t *xl = lds;                               // [NR][part][NCI][XPX]
  uint16_t *dl = lds + NR * XROW;                   // [part][NCO][DYP]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fy = wave % RW, blk = wave / RW % (COB * CIB), ks = wave / (RW * COB * CIB);
  const int cob = blk % COB, cib = blk / COB;
  // neighbours on one XCD: the workgroups of a slice and column, which read the same rows
  int id = xcd_compact_id(blockIdx.x, gridDim.x);
  const int fyg = id % a.fy_groups; id /= a.fy_groups;
  const int ci0 = id % a.ci_tiles * NCI; id /= a.ci_tiles;
  const int co0 = id % a.co_tiles * NCO; id /= a.co_tiles;
  const int x0  = id % a.tiles_x * TC;
  const int part_slice = id;                        // slice * tiles_x + column
  const int slice = id / a.tiles_x;
  const int fy0 = fyg * RW;
  const int hw = a.H * a.W, ohw = a.OH * a.OW;

  // ---- staging plans: a row of X is NQ words per channel, a step of dY 16 words per channel
  unsigned xoff[XI], xlds[XI];
  int xrow[XI];
  unsigned xkeep = 0, dkeep = 0;
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int e = tid + NT * i;
    const int q = e % NQ, rest = e / NQ, c = rest % NCI, r = rest / NCI;
    const int ix = x0 - a.pwa + 4 * q;
    unsigned keep = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (static_cast<unsigned>(ix + k) < static_cast<unsigned>(a.W)) keep |= 1u << k;
    const bool in = r < RPS && ci0 + c < a.C && (VEC ? keep == 15u : keep != 0u);
    xrow[i] = r < RPS ? r : -1;
    xoff[i] = in ? 4u * ((ci0 + c) * hw + ix) : DWX_NOWHERE;
    xlds[i] = c * XPX + 4 * q;
    xkeep |= keep << (4 * i);
  }
  // dY: word tid%16 of channels tid/16 + NT/16*i
  unsigned doff[DI];
  const int dq = tid & 15, drow = 4 * dq / TC, dox = x0 + 4 * dq % TC, dlds = (tid >> 4) * DYP + 4 * dq;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (dox + k < a.OW) dkeep |= 1u << k;
#pragma unroll
  for (int i = 0; i < DI; ++i) {
    const int c = (tid >> 4) + NT / 16 * i;
    doff[i] = c < NCO && co0 + c < a.Kc && (VEC ? dkeep == 15u : dkeep != 0u) ? 4u * ((co0 + c) * ohw + dox) : DWX_NOWHERE;
  }

  // every other 16-pixel group of dY is staged with its sign turned (split_bf16.h); a thread's
  // words lie in groups of the same parity
  const float dsign = (tid & 15) >> 2 & 1 ? -X3_SCALE : X3_SCALE;

  floatx4 rx[XI], rd[DI];
  auto load4 = [](auto desc, unsigned off, unsigned keep) {
    if (VEC) return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(desc, off, 0, 0));
    floatx4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(desc, keep >> k & 1u ? off + 4 * k : DWX_NOWHERE, 0, 0));
    return v;
  };
  // the words of step `t` of image `img`: X rows y+fy0+RW-1-ph .. of the RPS output rows from y
  // = RPS*t on, and those rows of dY (unless the step only fills the ring: t < first)
  auto fetch = [&](int img, int y, bool with_dy) {
    const auto xd = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x + static_cast<size_t>(img) * a.C * hw), 0,
                                                      4u * a.C * hw, 0x00027000);
    const auto dd = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.dy + static_cast<size_t>(img) * a.Kc * ohw), 0,
                                                      4u * a.Kc * ohw, 0x00027000);
    const int iy0 = y + fy0 + RW - 1 - a.ph;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int iy = iy0 + xrow[i];
      const bool in = xrow[i] >= 0 && static_cast<unsigned>(iy) < static_cast<unsigned>(a.H);
      rx[i] = load4(xd, in && xoff[i] != DWX_NOWHERE ? xoff[i] + 4u * iy * a.W : DWX_NOWHERE, xkeep >> (4 * i));
    }
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      const int oy = y + drow;
      const bool in = with_dy && oy < a.OH;
      rd[i] = load4(dd, in && doff[i] != DWX_NOWHERE ? doff[i] + 4u * oy * a.OW : DWX_NOWHERE, dkeep);
    }
  };
  float dbs[DI];
#pragma unroll
  for (int i = 0; i < DI; ++i) dbs[i] = 0.0f;
  auto store4 = [](uint16_t *at, int part_stride, const floatx4 &v) {
    uint32_t lo[X3_PARTS], hi[X3_PARTS];
    split_pair(v.x, v.y, lo);
    split_pair(v.z, v.w, hi);
#pragma unroll
    for (int p = 0; p < X3_PARTS; ++p) *reinterpret_cast<uintx2 *>(at + p * part_stride) = uintx2{lo[p], hi[p]};
  };
  // ring slot of the first row of the step that is staged next
  int head = 0;
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      if (xrow[i] < 0) continue;
      int slot = head + xrow[i];
      slot -= slot >= NR ? NR : 0;
      store4(xl + slot * XROW + xlds[i], NCI * XPX, rx[i] * X3_SCALE);
    }
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      if (NCO * 16 % NT == 0 || tid + NT * i < NCO * 16) store4(dl + dlds + NT / 16 * DYP * i, NCO * DYP, rd[i] * dsign);
      dbs[i] += (rd[i].x + rd[i].y) + (rd[i].z + rd[i].w);
    }
  };

  floatx16 acc[S];
#pragma unroll
  for (int t = 0; t < S; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;

  const int half = lane >> 5, l32 = lane & 31;
  const uint16_t *dlane = dl + (cob * 32 + l32) * DYP + 8 * half;
  const uint16_t *xlane = xl + (cib * 32 + l32) * XPX + 8 * half;
  auto multiply = [&](int oldest) {
#pragma unroll
    for (int gi = 0; gi < GPW; ++gi) {
      const int g = ks * GPW + gi;                  // pixels 16g .. 16g+15 of the step
      const int r = 16 * g / TC, c = 16 * g % TC;
      bf16x8 d[X3_PARTS];
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p)
        d[p] = *reinterpret_cast<const bf16x8 *>(dlane + p * NCO * DYP + 16 * g);
      int slot = oldest + r + fy;
      slot -= slot >= NR ? NR : 0;
      const uint16_t *row = xlane + slot * XROW + c;
      uint32_t w[X3_PARTS][8];
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p) {
        const uintx4 w0 = *reinterpret_cast<const uintx4 *>(row + p * NCI * XPX);
        const uintx4 w1 = *reinterpret_cast<const uintx4 *>(row + p * NCI * XPX + 8);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          w[p][k]     = w0[k];
          w[p][k + 4] = w1[k];
        }
      }
      add_taps<SHIFT, S>(acc, d, w, g & 1 ? -1.0f : 1.0f);
    }
  };

  // ---- the slice's steps: chunks of RPS output rows, [beg, end) counted over the batch
  const int per_image = a.chunks_per_image;
  int chunk = slice * a.chunks_per_slice;
  const int end = min(a.chunks_total, chunk + a.chunks_per_slice);
  int img, t;                                       // the step that is fetched
  img = chunk / per_image;
  t   = chunk - img * per_image - WARM;             // (WARM steps fill the ring first)
  int first = t + WARM;
  if (chunk < end) fetch(img, RPS * t, t >= first);
  while (chunk < end) {
    __syncthreads();                                // everyone is done with the rows that are replaced
    stage();
    __syncthreads();
    const bool product = t >= first;
    head += RPS;
    head -= head >= NR ? NR : 0;
    // the next step
    if (product) ++chunk;
    if (++t >= per_image) {
      ++img;
      t     = -WARM;
      first = 0;
    }
    if (chunk < end) fetch(img, RPS * t, t >= first);
    if (product) multiply(head);
  }

  // ---- shares of a channel block are added in wave order, then the slice is stored: reg r of
  //      lane l holds output channel 8*(r/4) + 4*(l/32) + r%4, input channel l%32
  const int crs = a.C * a.RS;
  float *out    = a.partial + static_cast<size_t>(part_slice) * a.Kc * crs;
  float *red    = reinterpret_cast<float *>(lds);   // [KS-1][COB*CIB*RW][S][16][64]
  const int mine = blk * RW + fy;
  if (KS > 1) {
    __syncthreads();
    if (ks > 0) {
#pragma unroll
      for (int fx = 0; fx < S; ++fx)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          red[((((ks - 1) * COB * CIB * RW + mine) * S + fx) * 16 + r) * 64 + lane] = acc[fx][r];
    }
    __syncthreads();
  }
  if (ks == 0 && fy0 + fy < a.R) {
    if (KS > 1) {
#pragma unroll
      for (int fx = 0; fx < S; ++fx)
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int k = 1; k < KS; ++k)
            acc[fx][r] += red[((((k - 1) * COB * CIB * RW + mine) * S + fx) * 16 + r) * 64 + lane];
    }
    dwx_redo_exceptional<S, TC, RPS>(a, acc, lane, co0 + 32 * cob + l32, ci0 + 32 * cib + l32, fy0 + fy, x0, slice);
#pragma unroll
    for (int fx = 0; fx < S; ++fx)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float v = acc[fx][r];
        const int co = co0 + 32 * cob + 8 * (r >> 2) + 4 * half + (r & 3), ci = ci0 + 32 * cib + l32;
        if (co < a.Kc && ci < a.C) out[static_cast<size_t>(co) * crs + ci * a.RS + (fy0 + fy) * S + fx] = v;
      }
  }
  if (a.partial_db && ci0 == 0 && fyg == 0) {
    // the 16 words of a channel sit in neighbouring lanes: added with a fixed butterfly
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      float v = dbs[i];
      v += __shfl_xor(v, 1, 64);
      v += __shfl_xor(v, 2, 64);
      v += __shfl_xor(v, 4, 64);
      v += __shfl_xor(v, 8, 64);
      const int c = co0 + (tid >> 4) + NT / 16 * i;
      if ((tid & 15) == 0 && c < min(a.Kc, co0 + NCO)) a.partial_db[static_cast<size_t>(part_slice) * a.Kc + c] = v;
    }
  }
}

template <int RW, int S, int TC, int COB, int CIB, int SHIFT, bool VEC>
int launch_dwx_inst(const DwxPlan &p) {
  auto kernel = conv_dwx_kernel<RW, S, TC, COB, CIB, SHIFT, VEC>;
  static bool raised = false;
  if (!raised) {
    TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(p.lds_bytes)));
    raised = true;
  }
  TDH_LAUNCH(kernel, dim3(p.workgroups), dim3(dwx_threads(RW)), p.lds_bytes, ctx().stream, p.args);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

template <int RW, int S, int TC, int SHIFT, bool VEC>
int launch_dwx_blocks(const DwxPlan &p) {
  if (p.cob == 2 && p.cib == 2) return launch_dwx_inst<RW, S, TC, 2, 2, SHIFT, VEC>(p);
  if (p.cob == 2) return launch_dwx_inst<RW, S, TC, 2, 1, SHIFT, VEC>(p);
  return launch_dwx_inst<RW, S, TC, 1, 2, SHIFT, VEC>(p);
}

template <int RW, int S, int SHIFT, bool VEC>
int launch_dwx_tc(const DwxPlan &p) {
  switch (p.tc) {
    case 64: return launch_dwx_blocks<RW, S, 64, SHIFT, VEC>(p);
    case 32: return launch_dwx_blocks<RW, S, 32, SHIFT, VEC>(p);
    default: return launch_dwx_blocks<RW, S, 16, SHIFT, VEC>(p);
  }
}

}  // namespace

// compiled three times, -DTDH_DWX_PART=0..2: 3x3 windows with 16-byte and scalar loads, 5x5 windows with
// scalar loads; each with padding::same (the row starts 4 - pad pixels into the first word) and
// without padding
#if TDH_DWX_PART == 0
int dwx_launch_3_vec(const DwxPlan &p) { return p.shift ? launch_dwx_tc<3, 3, 3, true>(p) : launch_dwx_tc<3, 3, 0, true>(p); }
#elif TDH_DWX_PART == 1
int dwx_launch_3_scalar(const DwxPlan &p) { return p.shift ? launch_dwx_tc<3, 3, 3, false>(p) : launch_dwx_tc<3, 3, 0, false>(p); }
#elif TDH_DWX_PART == 2
int dwx_launch_5_scalar(const DwxPlan &p) { return p.shift ? launch_dwx_blocks<2, 5, 64, 2, false>(p) : launch_dwx_blocks<2, 5, 64, 0, false>(p); }
#else
#error "TDH_DWX_PART must be 0..2"
#endif

}  // namespace tdh
