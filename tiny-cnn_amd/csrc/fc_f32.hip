// fc_f32.hip — y[b][o] = x[b][i] W[i][o] of fully-connected layers in fp32, for plain matrices of rows of whole 16-byte
// words: the tiles, slices of the reduction and order of the sums of gemm_mfma_kernel (gemm_mfma.h), so its bits, with a
// loop that carries nothing but this layout.
//
// A tile's words are loaded while the tile before the last is multiplied, through a buffer descriptor (what does not exist
// has an offset behind it), and cross LDS into the other of two buffers while the last is multiplied: one barrier every
// FF_BK indices. us, the general kernel / here: 4096 x 4096, batch 256 93 / 82 (104 TFLOP/s; what is left are the slices' 32 MB,
// the first loads and the barriers), batch 1024 321 / 269, 131072 x 256, batch 64 62 / 51, batch 96 111 / 73, 5376 x 1308, batch
// 278 85 / 57. Sixteen indices a barrier, reads two and four steps ahead, three workgroups a compute unit: no different.
#include "gemm_mfma.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int FF_NT = 256;
constexpr int FF_BK = 32;
constexpr int FF_PAD = 4;
constexpr unsigned FF_NOWHERE = 0x80000000u;   // past the end of every matrix

template <int BM, int BN, int WM, int WN, class Epi>
__global__ void __launch_bounds__(FF_NT, 2)
fc_f32_kernel(const float *__restrict__ A, const float *__restrict__ B, const Epi epi, const int M, const int N, const int K,
              const int k_per_split, float *__restrict__ partial) {
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int QK = FF_BK / 4, QN = BN / 4;        // words of a row of A and of B in a tile
  constexpr int NA = BM * QK / FF_NT, NB = FF_BK * QN / FF_NT;
  static_assert(NA * FF_NT == BM * QK && NB * FF_NT == FF_BK * QN, "whole words to every thread");
  extern __shared__ __align__(16) float ff_lds[];
  constexpr int LDA = BM + FF_PAD, LDB = BN + FF_PAD, BUF = FF_BK * (LDA + LDB);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  // neighbouring tiles, which share rows of A or columns of B, on one XCD
  const int gx = gridDim.x, gy = gridDim.y;
  int id = xcd_compact_id(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * gy * gridDim.z);
  const int bx = id % gx;
  id /= gx;
  const int by = id % gy, bz = id / gy;
  const int m0 = by * BM, n0 = bx * BN;
  const int kbeg = bz * k_per_split, kend = min(K, kbeg + k_per_split);

  const auto da = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, 4u * M * K, 0x00027000);
  const auto db = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, 4u * K * N, 0x00027000);
  unsigned aoff[NA], boff[NB];
  const int aq = tid % QK, ar = tid / QK, bq = tid % QN, bk = tid / QN;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int m = m0 + ar + FF_NT / QK * i;
    aoff[i] = m < M ? 4u * (m * K + 4 * aq) : FF_NOWHERE;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) boff[i] = n0 + 4 * bq < N ? 4u * ((bk + FF_NT / QN * i) * N + n0 + 4 * bq) : FF_NOWHERE;

  floatx4 ra[NA], rb[NB];
  auto fetch = [&](int k0) {
    const int left = kend - k0;
    const int ks = min(k0, K);
#pragma unroll
    for (int i = 0; i < NA; ++i)
      ra[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                              da, left >= FF_BK || 4 * aq < left ? aoff[i] : FF_NOWHERE, 4 * ks, 0));
#pragma unroll
    for (int i = 0; i < NB; ++i)
      rb[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                              db, left >= FF_BK || bk + FF_NT / QN * i < left ? boff[i] : FF_NOWHERE, 4 * ks * N, 0));
  };
  auto stage = [&](int to) {
    float *as = ff_lds + to * BUF + 4 * aq * LDA + ar, *bs = ff_lds + to * BUF + FF_BK * LDA + bk * LDB + 4 * bq;
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) as[j * LDA + FF_NT / QK * i] = ra[i][j];
#pragma unroll
    for (int i = 0; i < NB; ++i) *reinterpret_cast<floatx4 *>(bs + FF_NT / QN * i * LDB) = rb[i];
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int at_a = (lane >> 5) * LDA + wm * (BM / WM) + (lane & 31);
  const int at_b = FF_BK * LDA + (lane >> 5) * LDB + wn * (BN / WN) + (lane & 31);
  fetch(kbeg);
  stage(0);
  fetch(kbeg + FF_BK);
  __syncthreads();
  int cur = 0;
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += FF_BK) {
    stage(cur ^ 1);   // (behind the last tile: zeros that nobody reads)
    fetch(k0 + 2 * FF_BK);
    const float *as = ff_lds + cur * BUF + at_a, *bs = ff_lds + cur * BUF + at_b;
    constexpr int AHEAD = TM * TN == 1 ? 3 : TM * TN == 2 ? 2 : 1;
    float af[AHEAD + 1][TM], bf[AHEAD + 1][TN];
    auto read = [&](int p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[p % (AHEAD + 1)][i] = as[2 * p * LDA + 32 * i];
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[p % (AHEAD + 1)][j] = bs[2 * p * LDB + 32 * j];
    };
#pragma unroll
    for (int p = 0; p < AHEAD; ++p) read(p);
#pragma unroll
    for (int p = 0; p < FF_BK / 2; ++p) {
      if (p + AHEAD < FF_BK / 2) read(p + AHEAD);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[p % (AHEAD + 1)][i], bf[p % (AHEAD + 1)][j], acc[i][j], 0, 0, 0);
      if (TM * TN == 1) __builtin_amdgcn_sched_barrier(0);   // (the reads stay that far ahead)
    }
    __syncthreads();
    cur ^= 1;
  }

  // D[i][j] of a block: reg r of lane l at row 8*(r/4) + 4*(l/32) + r%4, column l%32
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn * (BN / WN) + 32 * j + (lane & 31);
    if (n >= N) continue;
    if (partial) {
      float *dst = partial + static_cast<size_t>(bz) * M * N + n;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + wm * (BM / WM) + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          if (m < M) dst[static_cast<size_t>(m) * N] = acc[i][j][r];
        }
    } else {
      const typename Epi::Col c = epi.col(n);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        float before[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + wm * (BM / WM) + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          before[r]   = m < M ? epi.prior(m, c) : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + wm * (BM / WM) + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          if (m < M) epi.store(m, c, acc[i][j][r], before[r]);
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, class Epi>
int launch_ff(const GemmPlan &p, const float *A, const float *B, const Epi &epi, int M, int N, int K, float *partial) {
  auto kernel = fc_f32_kernel<BM, BN, WM, WN, Epi>;
  constexpr int bytes = 2 * FF_BK * (BM + BN + 2 * FF_PAD) * static_cast<int>(sizeof(float));
  if (bytes > 64 * 1024) {
    static const hipError_t raised =
        hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TDH_HIP(raised);
  }
  TDH_LAUNCH(kernel, dim3(ceil_div(N, BN), ceil_div(M, BM), p.splits), dim3(FF_NT), bytes, ctx().stream, A, B, epi, M, N, K,
             p.k_per_split, partial);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace

bool fc_f32_applies(int M, int N, int K, const float *A, const float *B) {
  if (N % 4 || K % 4 || ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15)) return false;
  if (static_cast<long>(M) * K >= (1L << 29) || static_cast<long>(N) * K >= (1L << 29)) return false;
  const GemmPlan p = plan_gemm(M, N, K, true);
  // (shorter slices are a tile or two: 2352 x 64, batch 37, slices of 16 4.6 / 6.0; 2048 x 512, batch 128, of 64 9.8 / 9.4)
  return p.k_per_split >= 64 && (p.cfg == 0 || (p.cfg >= 2 && p.cfg <= 5));
}

template <class Epi>
static int run_ff(const float *A, const float *B, const Epi &epi, int M, int N, int K, const char *tag, const char *reduce_tag) {
  const GemmPlan p = plan_gemm(M, N, K, true);
  float *partial   = nullptr;
  if (p.splits > 1) {
    void *ws = nullptr;
    TDH_TRY(ws_take(sizeof(float) * p.splits * static_cast<size_t>(M) * N, &ws));
    partial = static_cast<float *>(ws);
  }
  {
    ProfScope prof(tag, M, N, K);
    switch (p.cfg) {
      case 0: TDH_TRY((launch_ff<128, 128, 2, 2>(p, A, B, epi, M, N, K, partial))); break;
      case 2: TDH_TRY((launch_ff<64, 128, 2, 2>(p, A, B, epi, M, N, K, partial))); break;
      case 3: TDH_TRY((launch_ff<64, 64, 2, 2>(p, A, B, epi, M, N, K, partial))); break;
      case 4: TDH_TRY((launch_ff<32, 128, 1, 4>(p, A, B, epi, M, N, K, partial))); break;
      default: TDH_TRY((launch_ff<32, 256, 1, 4>(p, A, B, epi, M, N, K, partial))); break;
    }
  }
  return p.splits > 1 ? launch_splitk_reduce(partial, p.splits, M, N, epi, reduce_tag) : TDH_OK;
}
int fc_f32_run(const float *A, const float *B, const EpiRowMajor &epi, int M, int N, int K, const char *tag, const char *reduce_tag) {
  return run_ff(A, B, epi, M, N, K, tag, reduce_tag);
}
int fc_f32_run_act(const float *A, const float *B, const EpiRowMajorAct &epi, int M, int N, int K, const char *tag,
                   const char *reduce_tag) {
  return run_ff(A, B, epi, M, N, K, tag, reduce_tag);
}

}  // namespace tdh
