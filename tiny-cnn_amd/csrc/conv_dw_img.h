// conv_dw_img.h — weight gradient of a 5x5 convolution (padding 2, stride 1) on images of 8x8 or
// 16x16 pixels, every filter row in one workgroup: what a workgroup does. The kernels around it
// are in conv_dw.hip (this gradient alone) and conv_bwd_pair.hip (beside dX).
//
// The kernel of conv_dw.hip gives such a layer workgroups of (one filter row) x (a chunk of
// images): five workgroups stage the same tiles, and a wave's slice leaves as 80 scattered 4-byte
// stores. Here a workgroup owns 32 output channels x 32 input channels x one of FOUR GROUPS OF TAPS
// (7 + 6 + 6 + 6 of the 25, each group lies in two filter rows) for a run of chunks of 128 pixels,
// two images of 8x8 or half an image of 16x16; a wave takes 32 of them as four groups of eight.
// X is staged with its zero frame (12 rows of IS + 4 per image or half image), so the X fragment of
// a row and filter row is two 16-byte reads, eight floats, that serve all five taps of the row; a
// dY fragment (one 16-byte read per group) serves all taps of the group. The pixel pairing is the
// one of conv_dw.hip: k = 0 lanes take the left four pixels of a group, k = 1 lanes the right four.
// The next chunk's words travel while the current one is multiplied. The four waves' sums meet in
// LDS (pairwise), and the whole workgroup stores the slice. The bias gradient comes from the
// workgroups of tap group 0 and input-channel block 0, out of the dY they stage anyway.
//
// A chunk of 128 pixels, and not 256, keeps the footprint (54 KB, and 72 KB for the sums at the end)
// under half a compute unit's LDS: two workgroups share it, one loading or adding up while the other
// multiplies.
#pragma once
#include "common.h"

namespace tdh {

struct DwImgArgs {
  const float *x, *dy;
  float *partial;      // [slices][Kc][C*25]
  float *partial_db;   // [slices][Kc], or null
  int batch, C, Kc;
  int chunks_total, chunks_per_slice;   // chunks of 128 pixels
  int co_blocks, ci_blocks;
};
struct DwImgPlan {
  bool ok;
  int size;            // 8 or 16
  DwImgArgs args;
  int slices, workgroups;
  size_t lds_bytes;
};
DwImgPlan make_dw_img_plan(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph, int pw);
int conv_dw_sum_slices(const void *part, const void *part_db, int slices, int Kc, int crs, float *dw, float *db,
                       int accumulate);

namespace {

constexpr int DWI_NT  = 256;
constexpr int DWI_DYP = 128 + 4;        // floats per staged dY channel (4 mod 32)
constexpr int DWI_SUM = 32 * 32 * 9;    // floats of a pair of waves' sums, [co][ci][tap]
// geometry of a chunk for images of IS x IS pixels
template <int IS> struct DwImgGeom {
  static constexpr int IPC   = IS == 8 ? 2 : 1;       // images a chunk
  static constexpr int FP    = IS + 4;                // framed row
  static constexpr int PLANE = 12 * FP;               // 8 rows and their halo
  static constexpr int XP    = IPC * PLANE + 4;       // floats per staged X channel (4 / 20 mod 32)
  static constexpr int WPR   = IS / 4;                // 16-byte words of an image row
  static constexpr int XW    = IS == 8 ? 4 : 6;       // X words a thread stages per chunk
  static constexpr int LDS_FLOATS = 32 * DWI_DYP + 32 * XP > 2 * DWI_SUM ? 32 * DWI_DYP + 32 * XP : 2 * DWI_SUM;
};

// tap group G: taps T0 .. T0+N-1 of the 25 (tap = 5*fy + fx)
template <int G> struct DwImgTaps {
  static constexpr int T0 = G == 0 ? 0 : G == 1 ? 7 : G == 2 ? 13 : 19;
  static constexpr int N  = G == 0 ? 7 : 6;
  static constexpr int FY0 = T0 / 5, FY1 = (T0 + N - 1) / 5;
};

typedef float dwi_floatx16 __attribute__((ext_vector_type(16)));
typedef float dwi_floatx4 __attribute__((ext_vector_type(4)));

// the products of the wave's 32 pixels (four groups of eight: rows of an image, or halves of two
// rows) for tap group G: acc[t - T0] += dY x X shifted by tap t
template <int G, int IS>
__device__ __forceinline__ void dw_img_products(const float *ap, const float *bp, dwi_floatx16 (&acc)[DwImgTaps<G>::N]) {
  using TG = DwImgTaps<G>;
  constexpr int FP = DwImgGeom<IS>::FP;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int oy = IS == 8 ? u : u >> 1, ox = IS == 8 ? 0 : 8 * (u & 1);
    const dwi_floatx4 a4 = *reinterpret_cast<const dwi_floatx4 *>(ap + u * 8);
    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
    for (int fy = TG::FY0; fy <= TG::FY1; ++fy) {
      const dwi_floatx4 b0 = *reinterpret_cast<const dwi_floatx4 *>(bp + (oy + fy) * FP + ox);
      const dwi_floatx4 b1 = *reinterpret_cast<const dwi_floatx4 *>(bp + (oy + fy) * FP + ox + 4);
      const float bv[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
      for (int fx = 0; fx < 5; ++fx) {
        const int t = 5 * fy + fx - TG::T0;
        if (t < 0 || t >= TG::N) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[j], bv[j + fx], acc[t], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int IS, int G>
__device__ __forceinline__ void dw_img_taps(const DwImgArgs &a, const int cob, const int cib, const int slice) {
  using GE = DwImgGeom<IS>;
  using TG = DwImgTaps<G>;
  constexpr int XP = GE::XP, FP = GE::FP, PIX = IS * IS, WPR = GE::WPR, XW = GE::XW;
  extern __shared__ __align__(16) float smem[];
  float *dy_l = smem;                  // [32][DWI_DYP]
  float *x_l  = smem + 32 * DWI_DYP;   // [32][XP], frames of zeros around the images
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int co0 = cob * 32, ci0 = cib * 32;
  const int kohw = a.Kc * PIX, chw = a.C * PIX;

  dwi_floatx16 acc[TG::N];
#pragma unroll
  for (int t = 0; t < TG::N; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
  const bool sums_dy = G == 0 && a.partial_db != nullptr && cib == 0;
  float dbs = 0.0f;   // this thread's share of the bias gradient of channel tid / 8

  // fragment bases: A lane = (output channel l%32, half l/32), B lane = (input channel l%32, half)
  const float *ap = dy_l + (lane & 31) * DWI_DYP + wave * 32 + 4 * (lane >> 5);
  const float *bp = x_l + (lane & 31) * XP + (IS == 8 ? (wave >> 1) * GE::PLANE + 4 * (wave & 1) * FP : 2 * wave * FP) +
                    4 * (lane >> 5);

  const int c_begin = slice * a.chunks_per_slice;
  const int c_end   = min(a.chunks_total, c_begin + a.chunks_per_slice);
  // ---- staging: a thread moves four 16-byte words of dY and four (six) of X per chunk, all loads
  //      asked for before the first store. dY word e: channel e / 32, words of the 128 pixels. X
  //      word e: the same, or of 16x16 images channel e / 48, word of the twelve rows; rows outside
  //      the image and images past the batch are read from a row of the tensor and stored as zeros.
  dwi_floatx4 rdy[4], rx[XW];
  auto x_row = [&](int chunk, int q) { return (q >> 2) - 2 + 8 * (chunk & 1); };   // (16x16 images)
  auto fetch = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + DWI_NT * i, c = e >> 5, q = e & 31;
      const int img = IS == 8 ? 2 * chunk + (q >> 4) : chunk >> 1;
      const int at  = IS == 8 ? 4 * (q & 15) : 128 * (chunk & 1) + 4 * q;
      const size_t ig = img < a.batch ? img : 0;
      rdy[i] = *reinterpret_cast<const dwi_floatx4 *>(a.dy + ig * kohw + (co0 + c) * PIX + at);
    }
#pragma unroll
    for (int i = 0; i < XW; ++i) {
      const int e = tid + DWI_NT * i;
      if (IS == 8) {
        const int c = e >> 5, q = e & 31, img = 2 * chunk + (q >> 4);
        const size_t ig = img < a.batch ? img : 0;
        rx[i] = *reinterpret_cast<const dwi_floatx4 *>(a.x + ig * chw + (ci0 + c) * PIX + 4 * (q & 15));
      } else {
        const int c = e / 48, q = e - 48 * c, row = min(max(x_row(chunk, q), 0), IS - 1);
        rx[i] = *reinterpret_cast<const dwi_floatx4 *>(a.x + static_cast<size_t>(chunk >> 1) * chw + (ci0 + c) * PIX +
                                                       row * IS + 4 * (q & 3));
      }
    }
  };
  if (c_begin < c_end) fetch(c_begin);
  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    if (chunk == c_begin) {   // the frames of zeros, written while the first loads are on their way
      for (int i = tid; i < 32 * XP / 4; i += DWI_NT) reinterpret_cast<dwi_floatx4 *>(x_l)[i] = dwi_floatx4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();   // (the previous chunk's fragments have been read; the first time: the zeros are in place)
    const dwi_floatx4 z = dwi_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + DWI_NT * i, c = e >> 5, q = e & 31;
      const bool on = IS != 8 || 2 * chunk + (q >> 4) < a.batch;
      *reinterpret_cast<dwi_floatx4 *>(dy_l + c * DWI_DYP + 4 * q) = on ? rdy[i] : z;
    }
#pragma unroll
    for (int i = 0; i < XW; ++i) {
      // X row, word of the row -> framed row, columns 2 + 4 * word .. + 3 (8-byte aligned)
      const int e = tid + DWI_NT * i;
      int at;
      bool on;
      if (IS == 8) {
        const int c = e >> 5, q = e & 31;
        on = 2 * chunk + (q >> 4) < a.batch;
        at = c * XP + (q >> 4) * GE::PLANE + (((q & 15) / WPR) + 2) * FP + 2 + 4 * (q % WPR);
      } else {
        const int c = e / 48, q = e - 48 * c;
        on = static_cast<unsigned>(x_row(chunk, q)) < static_cast<unsigned>(IS);
        at = c * XP + (q >> 2) * FP + 2 + 4 * (q & 3);
      }
      const dwi_floatx4 v = on ? rx[i] : z;
      *reinterpret_cast<float2 *>(x_l + at)     = make_float2(v.x, v.y);
      *reinterpret_cast<float2 *>(x_l + at + 2) = make_float2(v.z, v.w);
    }
    __syncthreads();
    if (chunk + 1 < c_end) fetch(chunk + 1);   // (travels while this chunk is multiplied)
    if (sums_dy) {   // channel tid/8, floats (tid%8)*16 .. +15 of its 128 pixels
      const dwi_floatx4 *row = reinterpret_cast<const dwi_floatx4 *>(dy_l + (tid >> 3) * DWI_DYP + (tid & 7) * 16);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const dwi_floatx4 v = row[k];
        dbs += (v.x + v.y) + (v.z + v.w);
      }
    }
    dw_img_products<G, IS>(ap, bp, acc);
  }

  // ---- the four waves' sums, pairwise: (0 + 2) + (1 + 3). Waves 2 and 3 park
  //      their sums, waves 0 and 1 add them to their own and park the two results transposed,
  //      [output channel][input channel][tap] (rows of nine floats: no two lanes of a store share
  //      a bank), and the whole workgroup adds those two and stores: a lane's neighbours then
  //      write neighbouring taps and input channels, seven cache lines a store instead of 64.
  float *red = smem;   // [2][7*16][64], then [2][32*32][9]
  __syncthreads();
  if (wave >= 2) {
    float *dst = red + (wave - 2) * (7 * 16 * 64) + lane;
#pragma unroll
    for (int t = 0; t < TG::N; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(t * 16 + r) * 64] = acc[t][r];
  }
  __syncthreads();
  if (wave < 2) {
    const float *src = red + wave * (7 * 16 * 64) + lane;
#pragma unroll
    for (int t = 0; t < TG::N; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][r] += src[(t * 16 + r) * 64];
  }
  __syncthreads();
  if (wave < 2) {
    // reg r of lane l: output channel 8*(r/4) + 4*(l/32) + r%4, input channel l%32
    float *dst = red + wave * DWI_SUM + (4 * (lane >> 5) * 32 + (lane & 31)) * 9;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int t = 0; t < TG::N; ++t) dst[(8 * (r >> 2) + (r & 3)) * (32 * 9) + t] = acc[t][r];
  }
  __syncthreads();
  const int crs = a.C * 25;
  float *out = a.partial + (static_cast<size_t>(slice) * a.Kc + co0) * crs + ci0 * 25 + TG::T0;
  for (int e = tid; e < 32 * 32 * 8; e += DWI_NT) {
    const int t = e & 7, pair = e >> 3;   // pair = output channel * 32 + input channel
    if (t < TG::N)
      out[static_cast<size_t>(pair >> 5) * crs + (pair & 31) * 25 + t] = red[pair * 9 + t] + red[DWI_SUM + pair * 9 + t];
  }
  if (sums_dy) {
    // the eight shares of a channel sit in neighbouring lanes: added with a fixed butterfly
    dbs += __shfl_xor(dbs, 1, 64);
    dbs += __shfl_xor(dbs, 2, 64);
    dbs += __shfl_xor(dbs, 4, 64);
    if ((tid & 7) == 0) a.partial_db[static_cast<size_t>(slice) * a.Kc + co0 + (tid >> 3)] = dbs;
  }
}

// workgroup `block` of `blocks`, launched with DwImgGeom<IS>::LDS_FLOATS of LDS
template <int IS>
__device__ __forceinline__ void dw_img_workgroup(const DwImgArgs &a, const int block, const int blocks) {
  // workgroups that read the same tiles (the four tap groups and the output-channel blocks of a
  // slice) are neighbours after the renumbering, and so share an XCD's L2
  int id = xcd_compact_id(block, blocks);
  const int grp = id & 3;
  id >>= 2;
  const int cob = id % a.co_blocks;
  id /= a.co_blocks;
  const int cib = id % a.ci_blocks, slice = id / a.ci_blocks;
  // (one copy of the loop per group: a switch inside it would move every accumulator between the copies)
  switch (grp) {
    case 0: dw_img_taps<IS, 0>(a, cob, cib, slice); break;
    case 1: dw_img_taps<IS, 1>(a, cob, cib, slice); break;
    case 2: dw_img_taps<IS, 2>(a, cob, cib, slice); break;
    default: dw_img_taps<IS, 3>(a, cob, cib, slice); break;
  }
}

}  // namespace
}  // namespace tdh
