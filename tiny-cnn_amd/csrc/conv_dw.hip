// conv_dw.hip — weight gradient of a stride-1 3x3 or 5x5 convolution from LDS-staged tiles.
//
//   dW[co][ci][fy][fx] = sum_{img,oy,ox} dY[img][co][oy][ox] * X[img][ci][oy+fy-ph][ox+fx-pw]
//
// MFMA mapping (v_mfma_f32_32x32x2_f32): M = 32 output channels (A lane: co = l%32), N = 32
// input channels (B lane: ci = l%32), K = output pixels, two per instruction (k = l/32). Every
// filter tap is its own 32x32 accumulator: one dY fragment feeds all taps, and the X fragment
// of tap (fy,fx) is the same staged patch read (fy rows, fx columns) further on.
//
// The two pixels of an instruction are NOT neighbours: within a tile row of TC pixels, k = 0
// lanes walk the left half and k = 1 lanes the right half. A lane therefore needs consecutive
// pixels in consecutive instructions: per four pixels and filter row one 16-byte dY word and
// 4+S-1 X floats serve 4*S instructions. dY channel planes are padded to 4 (mod 32) floats (eight
// lanes' 16-byte words cover all banks), X channel planes to an odd stride (32 lanes' floats
// cover all banks).
//
// Staging is by aligned 16-byte words of the tensors' own rows: the staged X patch starts at
// the image column x0 - pwa, pwa the padding rounded up to 4, so that every word is either
// wholly inside a row or wholly outside; the fragment reads start pwa - pw floats in. A thread
// keeps one relative offset per word; whether the word exists for a given chunk (row inside the
// image, image inside the batch) is ONE unsigned compare of offset + chunk base against a
// limit, and words that do not exist are read from a zero word instead, which keeps the loads
// free of branches. Tensors whose rows are not multiples of four floats take the same words as
// four scalar loads.
//
// A workgroup owns 32*WCO output channels x 32 input channels x its taps for a range of pixel
// chunks (WK row groups of 64/TC output rows x TC columns). Waves: WCO channel blocks x WK row groups of the
// chunk x WFY filter-row groups; a wave keeps (R/WFY)*S accumulators, up to 144 registers, so
// the kernel runs one workgroup per CU with the full register file. The next chunk's global
// loads are issued before the current chunk's MFMAs and parked in registers. At the end the
// WK row-group sums are added pairwise through LDS and the workgroup writes one slice
// [slice][co][ci][tap]; splitk_reduce_kernel adds the slices in order.
//
// 5x5 windows: 25 accumulators do not fit one wave, so the filter rows (of 3x3 windows too, where the
// chip has room for them) go to different
// WORKGROUPS (grid z = channel block x filter row) and the kernel runs as a 1x5 window whose
// input rows are shifted by the filter row. Such a window needs no halo rows, so on small
// images a chunk holds TI whole images stacked as rows.
#include "conv_dw_img.h"
#include "conv_dwx.h"
#include "gemm_mfma.h"

namespace tdh {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int DWH_NDY = 8;   // dY words a thread stages per chunk
constexpr int DWH_NEVER = -(1 << 30);  // relative offset of a word that never exists

// a word that does not exist is loaded from here (not const: the loads must stay in the global
// address space, like those of the tensors)
__device__ __align__(16) float dwh_zero_word[4] = {0.0f, 0.0f, 0.0f, 0.0f};

struct DwHaloArgs {
  const float *x, *dy;
  float *partial;  // [slices][Kc][C*RF*S]
  // Bias gradient on the way (or null): the workgroups of input-channel block 0 / filter row 0
  // add up the dY words they stage anyway; [slices][Kc], reduced like the dW slices.
  float *partial_db;
  int batch, C, Kc, H, W, OH, OW, ph, pw;
  int TI;          // whole images stacked in a chunk (1: a chunk is WK*64/TC rows of one image)
  int tiles_x, chunks_total, chunks_per_slice;
  int plane_p;     // channel stride of the staged X planes (odd)
  int dyp;         // channel stride of the staged dY planes (4 mod 32)
  int pwa;         // staged X column 0 is image column x0 - pwa
  FastDiv div_rowchunks, div_oh;
  FastDiv div_gy, div_gz, div_tiles_x;  // grid y and z, tiles per row: the workgroup's place
};

// R: filter rows one workgroup covers, RF: filter rows of the window (RF/R workgroups share a
// channel block), VEC: the rows of X and dY allow aligned 16-byte loads
template <int R, int S, int TC, int WCO, int WK, int WFY, int RF, bool VEC>
__global__ void __launch_bounds__(64 * WCO * WK * WFY, 1) conv_dw_halo_kernel(const DwHaloArgs a) {
  constexpr int NT    = 64 * WCO * WK * WFY;
  constexpr int FYB   = RF / R;
  constexpr int RPW   = R / WFY;  // filter rows per wave
  constexpr int NACC  = RPW * S;
  constexpr int BCO   = 32 * WCO;
  constexpr int NQ    = (3 + TC + S - 1 + 3) / 4;  // words per staged X row
  constexpr int PITCH = 4 * NQ;
  constexpr int TPC   = NT / 32;  // threads staging one X channel plane
  constexpr int NG    = TC / 8;   // 4-pixel groups per row and half
  constexpr int TRW   = 64 / TC;  // output rows one wave row-group takes per chunk
  constexpr int STEPS = TRW * NG; // (row, group) steps of a chunk's MFMA loop: always 8
  constexpr int TR    = TRW * WK;
  constexpr int PRQ   = (TR + R - 1) * NQ;        // words of a staged X plane
  constexpr int NXI   = (PRQ + TPC - 1) / TPC;    // X words a thread stages per chunk
  static_assert(NXI <= 16, "the keep bits of the scalar loads cover 16 words");
  constexpr int LOG_TC = TC == 64 ? 6 : TC == 32 ? 5 : TC == 16 ? 4 : 3;
  constexpr int DQ    = 16 * WK;  // words per staged dY channel: 64 pixels per row group
  constexpr int DCO   = NT / DQ;  // dY channels one staging trip covers
  static_assert(R % WFY == 0, "filter rows must divide among the waves");
  static_assert(RF % R == 0, "filter rows must divide among the workgroups");
  static_assert(BCO * DQ == NT * DWH_NDY, "dY staging trips");
  static_assert(WFY == 1 || WK == 1, "row groups and filter-row groups are not combined");

  extern __shared__ __align__(16) float smem[];
  float *dy_l = smem;                // [BCO][dyp]
  float *x_l  = smem + BCO * a.dyp;  // [32][plane_p]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wco = wave % WCO, wk = (wave / WCO) % WK, wfy = wave / (WCO * WK);
  // Workgroups are handed to the eight XCDs (each with its own L2) round-robin in launch
  // order. Renumber them so that the workgroups that read the same tiles (the filter rows of a
  // channel block share dY and X, the input-channel blocks share dY, the output-channel blocks
  // share X) are neighbours on one XCD.
  int bx, by, bz;
  {
    const int gy = gridDim.y, gz = gridDim.z;
    const int total = gridDim.x * gy * gz, per = total >> 3;
    int id = blockIdx.x + gridDim.x * (blockIdx.y + gy * blockIdx.z);
    if (id < (per << 3)) id = (id & 7) * per + (id >> 3);
    uint32_t rest, q, m;  // filter row fastest, then input-channel block
    a.div_gz.divmod(static_cast<uint32_t>(id), rest, m);
    bz = static_cast<int>(m);
    a.div_gy.divmod(rest, q, m);
    by = static_cast<int>(m);
    bx = static_cast<int>(q);
  }
  uint32_t slice_u, tx_u;
  a.div_tiles_x.divmod(static_cast<uint32_t>(bx), slice_u, tx_u);
  const int tx = static_cast<int>(tx_u), slice = static_cast<int>(slice_u);
  const int x0 = tx * TC, co0 = by * BCO;
  const int ci0 = (bz / FYB) * 32, fy0 = (bz % FYB) * R;
  const int hw = a.H * a.W, ohw = a.OH * a.OW;
  const int chw = a.C * hw, kohw = a.Kc * ohw;

  // ---- X staging plan: thread -> channel xc, words xl + TPC*i of the plane [rows][NQ]
  const int xc = tid / TPC, xl = tid % TPC;
  int xrel[NXI];            // offset of word i from the chunk's base, or DWH_NEVER
  unsigned long long xkeep = 0; // scalar loads: 4 bits per word, float k lies inside the row
  // (written without branches: the plan runs once, cold, in front of the first load)
  const bool stacked = a.TI > 1;
#pragma unroll
  for (int i = 0; i < NXI; ++i) {
    const int pe = xl + TPC * i;
    const int r = pe / NQ, q = pe - r * NQ;
    const int ix = x0 - a.pwa + 4 * q;
    unsigned keep = 0;
    if (VEC) {
      keep = (ix >= 0 && ix + 3 < a.W) ? 15u : 0u;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) keep |= (static_cast<unsigned>(ix + k) < static_cast<unsigned>(a.W) ? 1u : 0u) << k;
    }
    // stacked whole images: the row inside its image is fixed, the chunk only picks images
    uint32_t il, rr;
    a.div_oh.divmod(static_cast<uint32_t>(r), il, rr);
    const int rs   = static_cast<int>(rr) + fy0 - a.ph;
    const bool in  = !stacked || (static_cast<int>(il) < a.TI && static_cast<unsigned>(rs) < static_cast<unsigned>(a.H));
    const bool ok  = (pe < PRQ) & (ci0 + xc < a.C) & (VEC ? keep == 15u : keep != 0u) & in;
    const int base = stacked ? static_cast<int>(il) * chw : 0;
    xrel[i] = ok ? base + (stacked ? rs : r) * a.W + ix : DWH_NEVER;
    if (!VEC) xkeep |= static_cast<unsigned long long>(ok ? keep : 0u) << (4 * i);
  }
  const float *x_chan = a.x + static_cast<size_t>(ci0 + xc) * hw;

  // ---- dY staging plan: word tid + NT*i -> channel dco + DCO*i, the same row and column for
  //      every i
  const int dq = tid % DQ, dco = tid / DQ;
  const int dcol = x0 + ((4 * dq) & (TC - 1));
  int dyrel = DWH_NEVER;
  {
    int r = (4 * dq) >> LOG_TC, base = 0;
    bool ok = VEC ? dcol + 3 < a.OW : dcol < a.OW;
    if (a.TI > 1) {
      uint32_t il, rr;
      a.div_oh.divmod(static_cast<uint32_t>(r), il, rr);
      ok   = ok && static_cast<int>(il) < a.TI;
      base = static_cast<int>(il) * kohw;
      r    = static_cast<int>(rr);
    }
    if (ok) dyrel = base + r * a.OW + dcol;
  }
  const float *dy_chan = a.dy + static_cast<size_t>(co0 + dco) * ohw;
  const float *zero = dwh_zero_word;

  floatx4 rx[NXI];
  floatx4 rdy[DWH_NDY];
  const bool sums_dy = a.partial_db != nullptr && bz == 0;
  float dbs[DWH_NDY];  // this thread's share of the bias gradient of channels dco + DCO*i
#pragma unroll
  for (int i = 0; i < DWH_NDY; ++i) dbs[i] = 0.0f;

  // The loads of a chunk are issued in STEPS parts, one per step of the MFMA loop of the chunk
  // before: every workgroup of the grid fetches at the same time, and a chunk's words issued
  // in one go wait for HBM while the matrix cores idle.
  const float *xb = nullptr, *dyb = nullptr;  // the chunk's image, this thread's channel
  int xbase = 0, dybase = 0;                  // added to the words' relative offsets
  unsigned xlimit = 0, dylimit = 0;
  auto fetch_begin = [&](int chunk) {
    uint32_t img, rc;
    a.div_rowchunks.divmod(chunk, img, rc);
    img *= a.TI;
    const int y0   = a.TI > 1 ? 0 : rc * TR;
    const int nimg = min(a.TI, a.batch - static_cast<int>(img));
    xb      = x_chan + static_cast<size_t>(img) * chw;
    xbase   = a.TI > 1 ? 0 : (y0 - a.ph + fy0) * a.W;
    xlimit  = a.TI > 1 ? nimg * chw : hw;
    dyb     = dy_chan + static_cast<size_t>(img) * kohw;
    dybase  = y0 * a.OW;
    dylimit = a.TI > 1 ? nimg * kohw : ohw;
  };
  // (in the first half of the steps: a load issued in the last steps has no MFMAs left to hide
  // behind, and the next stage() would wait a whole trip to memory for it)
  constexpr int LOAD_STEPS = STEPS / 2;
  auto fetch_part = [&](int part) {
#pragma unroll
    for (int i = 0; i < NXI; ++i) {
      if (i % LOAD_STEPS != part) continue;
      const int rel = xrel[i] + xbase;
      const bool ok = static_cast<unsigned>(rel) < xlimit;
      if (VEC) {
        rx[i] = *reinterpret_cast<const floatx4 *>(ok ? xb + rel : zero);
      } else {
        const unsigned keep = ok ? static_cast<unsigned>(xkeep >> (4 * (i & 15))) & 15u : 0u;
        rx[i].x = *((keep & 1u) ? xb + rel : zero);
        rx[i].y = *((keep & 2u) ? xb + rel + 1 : zero);
        rx[i].z = *((keep & 4u) ? xb + rel + 2 : zero);
        rx[i].w = *((keep & 8u) ? xb + rel + 3 : zero);
      }
    }
#pragma unroll
    for (int i = 0; i < DWH_NDY; ++i) {
      if (i % LOAD_STEPS != part) continue;
      const int rel  = dyrel + dybase;
      const bool oki = static_cast<unsigned>(rel) < dylimit && co0 + dco + DCO * i < a.Kc;
      const float *p = dyb + static_cast<size_t>(DCO * i) * ohw + rel;
      if (VEC) {
        rdy[i] = *reinterpret_cast<const floatx4 *>(oki ? p : zero);
      } else {
        rdy[i].x = *(oki ? p : zero);
        rdy[i].y = *((oki && dcol + 1 < a.OW) ? p + 1 : zero);
        rdy[i].z = *((oki && dcol + 2 < a.OW) ? p + 2 : zero);
        rdy[i].w = *((oki && dcol + 3 < a.OW) ? p + 3 : zero);
      }
    }
  };
  auto stage = [&]() {
    float *xd = x_l + xc * a.plane_p + 4 * xl;
#pragma unroll
    for (int i = 0; i < NXI; ++i) {
      if (xl + TPC * i < PRQ) {
        float *d = xd + 4 * TPC * i;
        d[0] = rx[i].x; d[1] = rx[i].y; d[2] = rx[i].z; d[3] = rx[i].w;
      }
    }
    float *dd = dy_l + dco * a.dyp + 4 * dq;
#pragma unroll
    for (int i = 0; i < DWH_NDY; ++i) *reinterpret_cast<floatx4 *>(dd + DCO * i * a.dyp) = rdy[i];
    if (sums_dy) {
#pragma unroll
      for (int i = 0; i < DWH_NDY; ++i) dbs[i] += (rdy[i].x + rdy[i].y) + (rdy[i].z + rdy[i].w);
    }
  };

  const int c_begin = slice * a.chunks_per_slice;
  const int c_end   = min(a.chunks_total, c_begin + a.chunks_per_slice);
  if (c_begin < c_end) {
    fetch_begin(c_begin);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) fetch_part(s);
  }

  floatx16 acc[NACC];
#pragma unroll
  for (int t = 0; t < NACC; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;

  // fragment bases of this lane: half k = lane/32 starts TC/2 pixels into the row
  const float *ap = dy_l + (wco * 32 + (lane & 31)) * a.dyp + ((wk * TRW) << LOG_TC) + (lane >> 5) * (TC / 2);
  const float *bp = x_l + (lane & 31) * a.plane_p + (wk * TRW + wfy * RPW) * PITCH + (a.pwa - a.pw) +
                    (lane >> 5) * (TC / 2);

  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    if (chunk > c_begin) __syncthreads();  // everyone is done reading the previous chunk
    stage();
    __syncthreads();
    // (behind the last chunk the same loads run against empty limits and fetch the zero word:
    // a step without branches is one block that the compiler can interleave)
    const bool more = chunk + 1 < c_end;
    fetch_begin(more ? chunk + 1 : chunk);
    if (!more) xlimit = dylimit = 0;
    // The fragments of step s+1 are read from LDS before the products of step s are issued,
    // and the next chunk's global loads between them: with one wave per SIMD nothing else
    // would cover their latencies.
    floatx4 av4[2];
    float bv[2][RPW][4 + S - 1];
    auto read_fragments = [&](int s, int to) {
      const int r = s / NG, g = s % NG;
      av4[to] = *reinterpret_cast<const floatx4 *>(ap + (r << LOG_TC) + 4 * g);
#pragma unroll
      for (int fy = 0; fy < RPW; ++fy)
#pragma unroll
        for (int k = 0; k < 4 + S - 1; ++k) bv[to][fy][k] = bp[(r + fy) * PITCH + 4 * g + k];
    };
    read_fragments(0, 0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int cur = s & 1;
      if (s + 1 < STEPS) read_fragments(s + 1, cur ^ 1);
      const float av[4] = {av4[cur].x, av4[cur].y, av4[cur].z, av4[cur].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int fy = 0; fy < RPW; ++fy)
#pragma unroll
          for (int fx = 0; fx < S; ++fx)
            acc[fy * S + fx] =
              __builtin_amdgcn_mfma_f32_32x32x2f32(av[j], bv[cur][fy][j + fx], acc[fy * S + fx], 0, 0, 0);
        if (j == 0) fetch_part(s);
      }
      __builtin_amdgcn_sched_barrier(0);  // (the loads stay in the step they were written for)
    }
  }

  // ---- add the WK row-group sums pairwise (upper half of the groups onto the lower half)
  if (WK > 1) {
    float *red = smem;  // [WK/2][WCO][NACC*16][64]
    for (int h = WK / 2; h >= 1; h >>= 1) {
      __syncthreads();
      if (wk >= h && wk < 2 * h) {
        float *dst = red + static_cast<size_t>((wk - h) * WCO + wco) * (NACC * 16 * 64) + lane;
#pragma unroll
        for (int t = 0; t < NACC; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) dst[(t * 16 + r) * 64] = acc[t][r];
      }
      __syncthreads();
      if (wk < h) {
        const float *src = red + static_cast<size_t>(wk * WCO + wco) * (NACC * 16 * 64) + lane;
#pragma unroll
        for (int t = 0; t < NACC; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[t][r] += src[(t * 16 + r) * 64];
      }
    }
  }
  if (wk == 0) {
    // reg r of lane l: row (co) 8*(r/4) + 4*(l/32) + r%4, column (ci) l%32
    const int ci = ci0 + (lane & 31);
    const int crs = a.C * RF * S;
    if (ci < a.C) {
      float *dst = a.partial + static_cast<size_t>(bx) * a.Kc * crs + ci * (RF * S) +
                   (fy0 + wfy * RPW) * S;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int co = co0 + wco * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (co >= a.Kc) continue;
#pragma unroll
        for (int t = 0; t < NACC; ++t) dst[static_cast<size_t>(co) * crs + t] = acc[t][r];
      }
    }
  }
  if (sums_dy) {
    // channel c = dco + DCO*i was summed by the DQ threads dco*DQ .. dco*DQ + DQ-1: add their
    // shares in thread order
    float *sh = smem;  // [DWH_NDY][NT]
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DWH_NDY; ++i) sh[i * NT + tid] = dbs[i];
    __syncthreads();
    if (tid < BCO && co0 + tid < a.Kc) {
      const float *src = sh + (tid / DCO) * NT + (tid % DCO) * DQ;
      float s = 0.0f;
      for (int q = 0; q < DQ; ++q) s += src[q];
      a.partial_db[static_cast<size_t>(bx) * a.Kc + co0 + tid] = s;
    }
  }
}


// 5x5 windows on 8x8 and 16x16 images (conv_dw_img.h)
template <int IS>
__global__ void __launch_bounds__(DWI_NT, 2) conv_dw_img_kernel(const DwImgArgs a) {
  dw_img_workgroup<IS>(a, blockIdx.x, gridDim.x);
}

struct DwHaloPlan {
  bool ok;
  int tc, wco, wk, wfy, nt;
  int window;      // filter rows (3 or 5)
  int rows_block;  // filter rows one workgroup covers
  DwHaloArgs args;
  size_t lds_bytes;
  dim3 grid;
  int slices;
};

int pad_to_4_mod_32(int v) {
  while ((v & 31) != 4) ++v;
  return v;
}

DwHaloPlan make_dw_plan(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph,
                        int pw) {
  DwHaloPlan p;
  p.ok = false;
  const bool five = R == 5 && S == 5;
  if (!(R == 3 && S == 3) && !five) return p;
  if (C < 16 || Kc < 16 || OW < 8 || OH < 2 || pw > 4) return p;
  p.tc = OW >= 48 ? 64 : OW >= 24 ? 32 : OW >= 12 ? 16 : 8;
  p.wfy = 1;
  // more than 32 output channels: two channel blocks share a workgroup's staged X patch (half
  // the row groups each), which also keeps the 5x5 kernel's LDS footprint small enough for a
  // convolution workgroup of the main chain to share the compute unit
  p.wco = Kc > 32 ? 2 : 1;
  p.wk  = 4 / p.wco;
  p.nt = 64 * p.wco * p.wk * p.wfy;
  p.window     = R;
  p.rows_block = five ? 1 : R;
  DwHaloArgs &a = p.args;
  a.batch = batch; a.C = C; a.Kc = Kc; a.H = H; a.W = W; a.OH = OH; a.OW = OW; a.ph = ph; a.pw = pw;
  const int tr = (64 / p.tc) * p.wk;
  const int nq = (3 + p.tc + S - 1 + 3) / 4;
  a.pwa = (pw + 3) & ~3;
  a.TI = 1;
  // whole images stacked as rows; rows past the last whole image stay empty
  if (five && tr > OH) a.TI = tr / OH;
  const int prq = (tr + p.rows_block - 1) * nq;
  a.plane_p = (4 * prq) | 1;
  a.dyp     = pad_to_4_mod_32(tr * p.tc);
  // the keep bits of the scalar loads cover 16 words a thread
  if (ceil_div(prq, p.nt / 32) > 16) return p;
  // offsets inside a chunk are 32-bit and must stay clear of the never-exists marker
  if (static_cast<long>(a.TI) * std::max<long>(static_cast<long>(C) * H * W, static_cast<long>(Kc) * OH * OW) >=
      (1L << 29))
    return p;
  a.tiles_x = ceil_div(OW, p.tc);
  const int row_chunks = a.TI > 1 ? 1 : ceil_div(OH, tr);
  a.chunks_total  = a.TI > 1 ? ceil_div(batch, a.TI) : batch * row_chunks;
  a.div_rowchunks = FastDiv(row_chunks);
  a.div_oh        = FastDiv(OH);
  const int co_blocks = ceil_div(Kc, 32 * p.wco);
  int ci_blocks       = ceil_div(C, 32) * (R / p.rows_block);
  const long base = static_cast<long>(a.tiles_x) * co_blocks * ci_blocks;
  // one workgroup per CU; a slice should still cover a few chunks so that its prologue and
  // its partial tile are paid for
  long slices = std::max<long>(1, 256 / base);
  slices = std::min<long>(slices, std::max(1, a.chunks_total / 2));
  a.chunks_per_slice = ceil_div(a.chunks_total, static_cast<int>(slices));
  p.slices           = ceil_div(a.chunks_total, a.chunks_per_slice);
  // A 3x3 window whose slices leave compute units idle: a workgroup per filter row as well, of the same slices (a tap has a
  // sum of its own either way, in the same order). us with the rows together / apart: 15x15, 24 -> 48, batch 37 (37
  // workgroups / 111) 28.5 / 15.6; 24x24, 16 -> 32, batch 16 28.5 / 13.5; 10x10, 32 -> 64, batch 64 29.5 / 16.1.
  if (p.rows_block == 3 && 3 * base * p.slices <= 256) {
    p.rows_block = 1;
    ci_blocks *= 3;
    a.plane_p = (4 * (tr * nq)) | 1;
  }
  const int nacc = (p.rows_block / p.wfy) * S;
  const size_t stage_floats = static_cast<size_t>(32 * p.wco) * a.dyp + 32 * static_cast<size_t>(a.plane_p);
  const size_t red_floats   = static_cast<size_t>(p.wk / 2) * p.wco * nacc * 16 * 64;
  p.lds_bytes = sizeof(float) * std::max(stage_floats, red_floats);
  if (p.lds_bytes > 150 * 1024) return p;
  if (static_cast<long>(a.tiles_x) * p.slices > 65535L * 16) return p;
  p.grid = dim3(a.tiles_x * p.slices, co_blocks, ci_blocks);
  a.div_gy      = FastDiv(co_blocks);
  a.div_gz      = FastDiv(ci_blocks);
  a.div_tiles_x = FastDiv(a.tiles_x);
  p.ok   = true;
  return p;
}

template <int R, int S, int TC, int WCO, int WK, int WFY, int RF, bool VEC>
int launch_dw_inst(const DwHaloPlan &p) {
  auto kernel = conv_dw_halo_kernel<R, S, TC, WCO, WK, WFY, RF, VEC>;
  if (p.lds_bytes > 64 * 1024) {
    // raised once per kernel instance and size: the default dynamic LDS limit is 64 KiB
    static size_t raised = 0;
    if (p.lds_bytes > raised) {
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(p.lds_bytes)));
      raised = p.lds_bytes;
    }
  }
  TDH_LAUNCH(kernel, p.grid, dim3(p.nt), p.lds_bytes, ctx().stream, p.args);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

template <int TC, bool VEC>
int launch_dw_tc(const DwHaloPlan &p) {
  if (p.window == 5)
    return p.wco == 2 ? launch_dw_inst<1, 5, TC, 2, 2, 1, 5, VEC>(p) : launch_dw_inst<1, 5, TC, 1, 4, 1, 5, VEC>(p);
  if (p.wco == 2)
    return p.rows_block == 1 ? launch_dw_inst<1, 3, TC, 2, 2, 1, 3, VEC>(p) : launch_dw_inst<3, 3, TC, 2, 2, 1, 3, VEC>(p);
  // 8 columns x 4 row groups would stage 17 words a thread with the filter rows together; the plan leaves that tile out
  constexpr int TC1 = TC == 8 ? 16 : TC;
  if (TC == 8) return set_error(TDH_ERR_INVALID, "conv_dw_halo_run: tile not built");
  return p.rows_block == 1 ? launch_dw_inst<1, 3, TC1, 1, 4, 1, 3, VEC>(p) : launch_dw_inst<3, 3, TC1, 1, 4, 1, 3, VEC>(p);
}

template <bool VEC>
int launch_dw_vec(const DwHaloPlan &p) {
  switch (p.tc) {
    case 64: return launch_dw_tc<64, VEC>(p);
    case 32: return launch_dw_tc<32, VEC>(p);
    case 16: return launch_dw_tc<16, VEC>(p);
    default: return launch_dw_tc<8, VEC>(p);
  }
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The three-part kernel of conv_dwx_inst.hip. It takes most of a compute unit's LDS, so the channel tiles x columns x filter-row groups x slices are chosen to come out just
// under a whole number of rounds of the 256 units; a slice keeps at least four steps for its
// prologue and partial tile. Two blocks of 32 channels on one side at least: with 32 x 32 half of
// every tile would be empty.
DwxPlan make_dwx_plan(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph, int pw) {
  DwxPlan p;
  p.ok = false;
  if (ctx().keep_f32 || R != S || (R != 3 && R != 5) || ph != pw || (pw != 0 && pw != R / 2)) return p;
  if (C < 16 || Kc < 16 || (C <= 32 && Kc <= 32) || OW < 12) return p;
  if (static_cast<long>(C) * H * W >= (1L << 29) || static_cast<long>(Kc) * OH * OW >= (1L << 29)) return p;
  p.tc  = OW >= 48 ? 64 : OW >= 24 ? 32 : 16;
  // Rows that fill less than four fifths of a narrow tile are better off with the fp32 kernel, whose
  // steps cost less (24x24 images, 64 -> 64, batch 100: 60 us there, 63 here; 28x28, 48 -> 96, batch
  // 50: 68 and 55). A 5x5 window goes through three groups of two filter rows, one of the six rows
  // empty: ahead only where the fp32 kernel has to load float by float (45x45, 33 -> 70, batch 19: 241
  // and 148; 64x64, 32 -> 64, batch 16: 72 and 73).
  if (p.tc < 64 && 5 * OW < 4 * p.tc * ceil_div(OW, p.tc)) return p;
  if (R == 5 && (p.tc < 64 || (W % 4 == 0 && OW % 4 == 0))) return p;
  p.cob = Kc > 32 ? 2 : 1;
  p.cib = C > 32 ? 2 : 1;
  const int rw = R == 3 ? 3 : 2, rps = 64 / p.tc;
  DwxArgs &a = p.args;
  a.batch = batch; a.C = C; a.Kc = Kc; a.H = H; a.W = W; a.OH = OH; a.OW = OW; a.ph = ph; a.pw = pw;
  a.R = R; a.RS = R * S;
  a.pwa   = (pw + 3) & ~3;
  p.shift = a.pwa - pw;
  a.tiles_x   = ceil_div(OW, p.tc);
  a.co_tiles  = ceil_div(Kc, 32 * p.cob);
  a.ci_tiles  = ceil_div(C, 32 * p.cib);
  a.fy_groups = ceil_div(R, rw);
  a.chunks_per_image = ceil_div(OH, rps);
  a.chunks_total     = batch * a.chunks_per_image;
  const int base     = a.tiles_x * a.co_tiles * a.ci_tiles * a.fy_groups;
  const int most     = a.chunks_total / 4;
  if (static_cast<long>(base) * most < 192 || base > 4096) return p;
  int slices = 1;
  double best = 0.0;
  for (int s = 1; s <= most && (s == 1 || base * s <= 512); ++s) {
    const int rounds  = ceil_div(base * s, 256);
    const double fill = base * s / (256.0 * rounds) - 0.02 * rounds;
    if (fill > best) {
      best   = fill;
      slices = s;
    }
  }
  a.chunks_per_slice = ceil_div(a.chunks_total, slices);
  p.slices     = ceil_div(a.chunks_total, a.chunks_per_slice);
  p.workgroups = base * p.slices;
  const size_t stage = 2u * 3 * (static_cast<size_t>(rw - 1 + rps) * 32 * p.cib * 4 * dwx_words(p.tc, S) + 32u * p.cob * 72);
  const int blocks   = p.cob * p.cib, shares = 4 / blocks;
  const size_t sums  = static_cast<size_t>(shares - 1) * blocks * rw * S * 16 * 64 * sizeof(float);
  p.lds_bytes = std::max(stage, sums);
  p.ok = p.lds_bytes <= 160 * 1024;
  return p;
}
int dwx_slices(const DwxPlan &p) { return p.slices * p.args.tiles_x; }

}  // namespace

// One workgroup per compute unit and tap group where the batch allows it. 16x16 images: from the
// batch on where the chunks give every compute unit a workgroup; the kernel above has fewer,
// longer workgroups, which is what a step that runs it beside its main chain wants.
DwImgPlan make_dw_img_plan(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph, int pw) {
  DwImgPlan p;
  p.ok = false;
  const int is = H;
  if (R != 5 || S != 5 || (is != 8 && is != 16) || W != is || OH != is || OW != is || ph != 2 || pw != 2 ||
      C % 32 != 0 || Kc % 32 != 0 || batch < 4 || static_cast<long>(batch) * std::max(C, Kc) * is * is >= (1L << 30))
    return p;
  DwImgArgs &a = p.args;
  p.size = is;
  a.batch = batch; a.C = C; a.Kc = Kc;
  a.co_blocks = Kc / 32; a.ci_blocks = C / 32;
  a.chunks_total = is == 8 ? ceil_div(batch, 2) : 2 * batch;
  const int base   = 4 * a.co_blocks * a.ci_blocks;
  const int slices = std::min(std::max(1, 256 / base), a.chunks_total);
  a.chunks_per_slice = ceil_div(a.chunks_total, slices);
  p.slices     = ceil_div(a.chunks_total, a.chunks_per_slice);
  p.workgroups = base * p.slices;
  p.lds_bytes  = sizeof(float) * (is == 8 ? DwImgGeom<8>::LDS_FLOATS : DwImgGeom<16>::LDS_FLOATS);
  p.ok = true;
  return p;
}

bool conv_dw_halo_applicable(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW,
                             int ph, int pw) {
  return make_dwx_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw).ok ||
         make_dw_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw).ok;
}

// the fp32 kernel's part of it: a shape that has a plan at one batch has one at every smaller batch
bool conv_dw_halo_f32_applicable(int R, int S, int batch, int C, int Kc, int H, int W, int OH, int OW, int ph, int pw) {
  return make_dw_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw).ok;
}

size_t conv_dw_halo_workspace_bytes(int R, int S, int batch, int C, int Kc, int H, int W, int OH,
                                    int OW, int ph, int pw) {
  const DwxPlan x3   = make_dwx_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  const DwHaloPlan p = make_dw_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  const DwImgPlan im = make_dw_img_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  // (which of them runs also depends on the tensors' alignment: room for whichever has more slices)
  size_t slices = 0;
  if (p.ok) slices = p.grid.x;
  if (x3.ok) slices = std::max(slices, static_cast<size_t>(dwx_slices(x3)));
  if (im.ok) slices = std::max(slices, static_cast<size_t>(im.slices));
  return slices == 0 ? 0 : ws_align(sizeof(float) * slices * Kc * C * R * S) + ws_align(sizeof(float) * slices * Kc);
}

// the kernel that runs for these tensors: x3 if ok, else im if ok, else p (slices 0: none does)
struct HaloChoice {
  bool vec;
  DwxPlan x3;
  DwImgPlan im;
  DwHaloPlan p;
  int slices;
};
static HaloChoice choose_halo(int R, int S, int batch, int C, int Kc, const float *x, const float *dy, int H, int W,
                              int OH, int OW, int ph, int pw) {
  HaloChoice h;
  h.vec = W % 4 == 0 && OW % 4 == 0 && aligned16(x) && aligned16(dy);
  h.x3  = make_dwx_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  h.im  = make_dw_img_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  h.p   = make_dw_plan(R, S, batch, C, Kc, H, W, OH, OW, ph, pw);
  h.im.ok  = h.im.ok && h.vec && (h.im.size == 8 || batch >= 96);
  h.slices = h.x3.ok ? dwx_slices(h.x3) : h.im.ok ? h.im.slices : h.p.ok ? static_cast<int>(h.p.grid.x) : 0;
  return h;
}

size_t conv_dw_halo_run_workspace_bytes(int R, int S, int batch, int C, int Kc, const float *x, const float *dy,
                                        int H, int W, int OH, int OW, int ph, int pw) {
  const size_t slices = choose_halo(R, S, batch, C, Kc, x, dy, H, W, OH, OW, ph, pw).slices;
  return ws_align(sizeof(float) * slices * Kc * C * R * S) + ws_align(sizeof(float) * slices * Kc);
}

// dw (+)= the slices of part, db (+)= those of part_db: left to the train step, or launched here
int conv_dw_sum_slices(const void *part, const void *part_db, int slices, int Kc, int crs, float *dw, float *db,
                       int accumulate) {
  EpiRowMajor epi{dw, crs, nullptr, ActGrad(), accumulate};
  EpiRowMajor epi_b{db, 1, nullptr, ActGrad(), accumulate};
  // the two reductions leave as one launch: collected by the train step, or here
  const bool collect_here = !ctx().defer_reduce;
  if (collect_here) flush_deferred_reduces(false);  // nothing may be left from a failed call
  ctx().defer_reduce = true;
  defer_reduce(static_cast<const float *>(part), slices, Kc, crs, epi);
  if (db) defer_reduce(static_cast<const float *>(part_db), slices, Kc, 1, epi_b);
  if (!collect_here) return TDH_OK;
  ctx().defer_reduce = false;
  return flush_deferred_reduces();
}

// dw (+)= sum over the batch; the caller has checked applicability and reserved the workspace
int conv_dw_halo_run(int R, int S, int batch, int C, int Kc, const float *x, const float *dy,
                     float *dw, int H, int W, int OH, int OW, int ph, int pw, int accumulate,
                     float *db) {
  HaloChoice h = choose_halo(R, S, batch, C, Kc, x, dy, H, W, OH, OW, ph, pw);
  DwxPlan &x3   = h.x3;
  DwImgPlan &im = h.im;
  DwHaloPlan &p = h.p;
  const bool vec = h.vec;
  if (!h.slices) return set_error(TDH_ERR_INVALID, "conv_dw_halo_run: shape not supported");
  const int crs = C * R * S, slices = h.slices;
  void *part = nullptr, *part_db = nullptr;
  TDH_TRY(ws_take(sizeof(float) * static_cast<size_t>(slices) * Kc * crs, &part));
  if (db) TDH_TRY(ws_take(sizeof(float) * static_cast<size_t>(slices) * Kc, &part_db));
  if (x3.ok) {
    x3.args.x = x; x3.args.dy = dy;
    x3.args.partial = static_cast<float *>(part); x3.args.partial_db = static_cast<float *>(part_db);
    ProfScope prof(db ? "conv_dw_db_x3" : "conv_dw_x3", Kc, crs, batch * OH * OW);
    TDH_TRY(R == 5 ? dwx_launch_5_scalar(x3) : vec ? dwx_launch_3_vec(x3) : dwx_launch_3_scalar(x3));
  } else {
    const bool rows = !im.ok && p.window == 3 && p.rows_block == 1;
    ProfScope prof(rows ? (db ? "conv_dw_db_rows" : "conv_dw_rows") : db ? "conv_dw_db_halo" : "conv_dw_halo", Kc, crs, batch * OH * OW);
    if (im.ok) {
      im.args.x = x; im.args.dy = dy;
      im.args.partial = static_cast<float *>(part); im.args.partial_db = static_cast<float *>(part_db);
      static bool raised[2] = {false, false};
      const int which = im.size == 8 ? 0 : 1;
      void (*kernel)(const DwImgArgs) = which ? conv_dw_img_kernel<16> : conv_dw_img_kernel<8>;
      if (!raised[which]) {
        TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(im.lds_bytes)));
        raised[which] = true;
      }
      TDH_LAUNCH(kernel, dim3(im.workgroups), dim3(DWI_NT), im.lds_bytes, ctx().stream, im.args);
      TDH_LAUNCH_CHECK();
    } else {
      p.args.x = x; p.args.dy = dy; p.args.partial = static_cast<float *>(part);
      p.args.partial_db = static_cast<float *>(part_db);
      TDH_TRY(vec ? launch_dw_vec<true>(p) : launch_dw_vec<false>(p));
    }
  }
  return conv_dw_sum_slices(part, part_db, slices, Kc, crs, dw, db, accumulate);
}

}  // namespace tdh
