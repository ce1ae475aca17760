// fc_x3.hip — products of large fully-connected layers on the bf16 matrix cores with three-part
// operands (split_bf16.h): C[M][N] = sum_k A[m][k] B[k][n] for plain matrices whose fast
// index differs:
//
//   forward  y[b][o]  = x[b][i] W[i][o]     A rows along k, B rows along n
//   dX       dx[b][i] = dy[b][o] W[i][o]    both along k
//   dW       dW[i][o] = x[b][i] dy[b][o]    A rows along m, B rows along n
//
// (Not the forward product of a train step: the bias gradients of a train step hang on the last bits of it
// and of the weights, and Adam makes a full step of one that is nearly zero.)
//
// A workgroup of four wave64 owns 64*WM x 64*WN elements, a wave 64 x 64 of them (four accumulator
// blocks). Per step of 32 reduction indices the tile's 16-byte words are loaded while the step
// before is multiplied, split once and left in LDS as [part][8 indices][row][8] bf16, so a lane's
// operand is one aligned 16-byte read. Words along k go there whole (rows of the eight-index planes are
// two units further apart than there are rows: the four words of a 128-byte line then hit
// different banks); words along m or n are turned in registers, four indices by four rows, and the
// rows of a plane are stored in the order row ^ (row/16 mod 4), which spreads the stores of 16
// neighbouring lanes over all banks. Two workgroups a compute unit cover each other's staging. Bound:
// the vector instructions that split the operands (290 a step and wave beside 48 matrix
// instructions; the two hardly overlap), HBM where one matrix is narrow.
// us, fp32 kernels / here: 4096 x 4096, batch 256 forward 107 / 67, dX 87 / 71; 6000 x 4096, batch 512
// 258 / 161, 234 / 179; 131072 x 256, batch 64 69 / 43, 65 / 47. Loading two steps ahead changed
// nothing, nor did tiles of 256 x 128 whose next step is split between the products of this one (dX of 4096 x 4096, batch 1024 199 and
// 203): what is left is what the chip's power allows.
#include "gemm_mfma.h"
#include "split_bf16.h"

namespace tdh {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr int FX_NT = 256;
constexpr int FX_BK = 32;
constexpr unsigned FX_NOWHERE = 0x80000000u;  // past the end of every matrix

// One operand of a tile: ROWS rows (m or n) x FX_BK indices. KC: the matrix has k as its fast index.
template <int ROWS, bool KC>
struct FxSide {
  static constexpr int PLANE = ROWS + 2;                         // units of an eight-index plane
  static constexpr int UNITS = X3_PARTS * 4 * PLANE;             // 16-byte units in LDS
  // words: KC 2 words (8 k of a row) twice an item, else 4 words (4 k x 4 rows) an item
  static constexpr int ITEMS = KC ? ROWS * 4 : ROWS * 2;
  static constexpr int PER   = (ITEMS + FX_NT - 1) / FX_NT;      // items a thread
  static constexpr int WORDS = KC ? 2 : 4;
  floatx4 reg[PER][WORDS];
  unsigned off[PER];

  __device__ __forceinline__ static int row_of(int e) { return KC ? e >> 2 : 4 * (e % (ROWS / 4)); }
  __device__ __forceinline__ static int k_of(int e) { return KC ? 8 * (e & 3) : 4 * (e / (ROWS / 4)); }
  __device__ __forceinline__ static int unit(int k8, int row) {
    return k8 * PLANE + (KC ? row : row ^ ((row >> 4) & 3));
  }
  // ld: floats from one row of the matrix to the next; rows: rows (KC) or row length (else) in use
  __device__ __forceinline__ void plan(int tid, int first, int extent, int ld) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + FX_NT * i, r = first + row_of(e), k = k_of(e);
      off[i] = e < ITEMS && r < extent ? 4u * (KC ? r * ld + k : k * ld + r) : FX_NOWHERE;
    }
  }
  template <class Desc>
  __device__ __forceinline__ void fetch(Desc desc, int tid, int k0, int left, int ld) {
    const int at = 4 * (KC ? k0 : k0 * ld);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int k = k_of(tid + FX_NT * i);
#pragma unroll
      for (int w = 0; w < WORDS; ++w) {
        const bool in = left >= FX_BK || k + (KC ? 4 * w : w) < left;
        const unsigned o = off[i] + (KC ? 16u * w : 4u * w * ld);
        reg[i][w] = __builtin_bit_cast(
            floatx4, __builtin_amdgcn_raw_buffer_load_b128(desc, in && off[i] != FX_NOWHERE ? o : FX_NOWHERE, at, 0));
      }
    }
  }
  // TURN: with the sign turned (the first operand's words carry the sign of their step)
  template <bool TURN>
  __device__ __forceinline__ void stage(uintx4 *lds, int tid) {
    constexpr float sign = TURN ? -X3_SCALE : X3_SCALE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + FX_NT * i;
      if (ITEMS % FX_NT != 0 && e >= ITEMS) continue;
      const int row = row_of(e), k = k_of(e);
      if (KC) {
        uintx4 part[X3_PARTS];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint32_t p3[X3_PARTS];
          split_pair(sign * reg[i][c / 2][2 * (c & 1)], sign * reg[i][c / 2][2 * (c & 1) + 1], p3);
#pragma unroll
          for (int p = 0; p < X3_PARTS; ++p) part[p][c] = p3[p];
        }
#pragma unroll
        for (int p = 0; p < X3_PARTS; ++p) lds[p * 4 * PLANE + unit(k / 8, row)] = part[p];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t lo[X3_PARTS], hi[X3_PARTS];
          split_pair(sign * reg[i][0][j], sign * reg[i][1][j], lo);
          split_pair(sign * reg[i][2 % WORDS][j], sign * reg[i][3 % WORDS][j], hi);
#pragma unroll
          for (int p = 0; p < X3_PARTS; ++p)
            reinterpret_cast<uintx2 *>(lds + p * 4 * PLANE + unit(k / 8, row + j))[(k >> 2) & 1] = uintx2{lo[p], hi[p]};
        }
      }
    }
  }
  __device__ __forceinline__ static bf16x8 read(const uintx4 *lds, int part, int k8, int row) {
    return __builtin_bit_cast(bf16x8, lds[part * 4 * PLANE + unit(k8, row)]);
  }
};

template <int WM, int WN, bool A_KC, bool B_KC, class Epi>
__global__ void __launch_bounds__(FX_NT, 2)
fc_x3_kernel(const float *__restrict__ A, const float *__restrict__ B, const int lda, const int ldb, const Epi epi,
             const int M, const int N, const int K, const int k_per_split, float *__restrict__ partial) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  using SideA = FxSide<BM, A_KC>;
  using SideB = FxSide<BN, B_KC>;
  __shared__ uintx4 a_lds[SideA::UNITS], b_lds[SideB::UNITS];
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

  const auto da = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, 4u * (A_KC ? M : K) * lda, 0x00027000);
  const auto db = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, 4u * (B_KC ? N : K) * ldb, 0x00027000);
  SideA sa;
  SideB sb;
  sa.plan(tid, m0, M, lda);
  sb.plan(tid, n0, N, ldb);

  floatx16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int half = lane >> 5, l32 = lane & 31;
  auto step = [&](int k0, auto odd) {
    constexpr int T = decltype(odd)::value;
    if (k0 > kbeg) __syncthreads();
    sa.template stage<T == 1>(a_lds, tid);
    sb.template stage<false>(b_lds, tid);
    __syncthreads();
    if (k0 + FX_BK < kend) {
      sa.fetch(da, tid, k0 + FX_BK, kend - k0 - FX_BK, lda);
      sb.fetch(db, tid, k0 + FX_BK, kend - k0 - FX_BK, ldb);
    }
    bf16x8 af[2][2][X3_PARTS], bf[2][2][X3_PARTS];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int p = 0; p < X3_PARTS; ++p)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          af[s][i][p] = SideA::read(a_lds, p, 2 * s + half, 64 * wm + 32 * i + l32);
          bf[s][i][p] = SideB::read(b_lds, p, 2 * s + half, 64 * wn + 32 * i + l32);
        }
    mfma_x3<2, 2, 2>(acc, af, bf, T ? -1.0f : 1.0f);
  };
  sa.fetch(da, tid, kbeg, kend - kbeg, lda);
  sb.fetch(db, tid, kbeg, kend - kbeg, ldb);
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += 2 * FX_BK) {
    step(k0, std::integral_constant<int, 0>());
    if (k0 + FX_BK < kend) step(k0 + FX_BK, std::integral_constant<int, 1>());
  }

  // the wave's infinite and NaN sums once more in fp32 (split_bf16.h): lane l brings row and column l%32
  // of the blocks at index k + l/32; eight indices are asked for together
  {
    // (hidden from the compiler, which otherwise keeps the comparisons for the stores below)
    int rows = M - (m0 + 64 * wm + 4 * half), cols = N - (n0 + 64 * wn + l32);   // from this lane's first element
    asm volatile("" : "+v"(rows), "+v"(cols));
    x3_redo(reinterpret_cast<floatx16(&)[4]>(acc), [&](int b, int r) {
      return 32 * (b % 2) < cols && 32 * (b / 2) + 8 * (r >> 2) + (r & 3) < rows;
    }, [&](floatx16 (&sum)[4]) {
#pragma unroll 1
      for (int k0 = kbeg; k0 < kend; k0 += 8) {
        float av[4][2], bv[4][2];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = k0 + 2 * s + half;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int m = m0 + 64 * wm + 32 * i + l32, n = n0 + 64 * wn + 32 * i + l32;
            av[s][i] = k < kend && m < M ? A[A_KC ? static_cast<size_t>(m) * lda + k : static_cast<size_t>(k) * lda + m] : 0.0f;
            bv[s][i] = k < kend && n < N ? B[B_KC ? static_cast<size_t>(n) * ldb + k : static_cast<size_t>(k) * ldb + n] : 0.0f;
          }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int b = 0; b < 4; ++b) sum[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[s][b / 2], bv[s][b % 2], sum[b], 0, 0, 0);
        if (x3_all_nan(sum)) return;
      }
    });
  }

  // D[i][j] of a block: reg r of lane l at row 8*(r/4) + 4*(l/32) + r%4, column l%32
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + 64 * wn + 32 * j + l32;
    if (n >= N) continue;
    const typename Epi::Col c = epi.col(n);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int mb = m0 + 64 * wm + 32 * i + 4 * half;
      if (partial) {
        float *dst = partial + static_cast<size_t>(bz) * M * N + n;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mb + 8 * (r >> 2) + (r & 3);
          if (m < M) dst[static_cast<size_t>(m) * N] = acc[i][j][r];
        }
      } else {
        float before[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mb + 8 * (r >> 2) + (r & 3);
          before[r]   = m < M ? epi.prior(m, c) : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mb + 8 * (r >> 2) + (r & 3);
          if (m < M) epi.store(m, c, acc[i][j][r], before[r]);
        }
      }
    }
  }
}

struct FxPlan {
  bool ok;
  int wm, wn, splits, k_per_split;
};
// Tiles of 128 x 128 (64 x 256 and 256 x 64 where one side has no more than 64 rows), split along k
// until every compute unit has two workgroups.
FxPlan fx_plan(int M, int N, int K) {
  FxPlan p;
  p.wm = M <= 64 ? 1 : N <= 64 ? 4 : 2;
  p.wn = 4 / p.wm;
  const long tiles = static_cast<long>(ceil_div(M, 64 * p.wm)) * ceil_div(N, 64 * p.wn);
  long splits = tiles < 512 ? 512 / tiles : 1;
  splits = std::max(1L, std::min<long>(splits, K / 128));
  p.k_per_split = ceil_div(ceil_div(K, static_cast<int>(splits)), FX_BK) * FX_BK;
  p.splits      = ceil_div(K, p.k_per_split);
  p.ok = tiles * p.splits >= 192;
  return p;
}

template <bool A_KC, bool B_KC, class Epi>
int launch_fx(const FxPlan &p, const float *A, const float *B, int lda, int ldb, const Epi &epi, int M, int N, int K,
              float *partial) {
  const dim3 grid(ceil_div(N, 64 * p.wn), ceil_div(M, 64 * p.wm), p.splits);
  switch (p.wm) {
    case 1: TDH_LAUNCH((fc_x3_kernel<1, 4, A_KC, B_KC, Epi>), grid, dim3(FX_NT), 0, ctx().stream, A, B, lda, ldb, epi, M, N, K, p.k_per_split, partial); break;
    case 2: TDH_LAUNCH((fc_x3_kernel<2, 2, A_KC, B_KC, Epi>), grid, dim3(FX_NT), 0, ctx().stream, A, B, lda, ldb, epi, M, N, K, p.k_per_split, partial); break;
    default: TDH_LAUNCH((fc_x3_kernel<4, 1, A_KC, B_KC, Epi>), grid, dim3(FX_NT), 0, ctx().stream, A, B, lda, ldb, epi, M, N, K, p.k_per_split, partial); break;
  }
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace

// dW: its result is written once however few samples there are, and the fp32 kernels (fc.hip) have less in front of their
// products. us there / here: 4096 x 4096 of 64 samples 31 / 39, 256 87 / 75 (one after the other for 10 ms, with dX and an
// optimizer between them, no different), 1024 309 / 212; 6000 x 4096 of 512 239 / 177; 784 x 1024 of 512 23 / 21; 512 x 512
// of 4000 37 / 28; 2048 x 2048 of 128 21 / 22; 131072 x 256 of 64 57 / 72.
constexpr int FX_DW_SAMPLES = 384;
bool fc_x3_applies(FxRows rows, int M, int N, int K, const float *A, const float *B, int lda, int ldb) {
  if (ctx().keep_f32 || M % 4 || N % 4 || (rows != FX_A_M_B_N && K % 4) || lda % 4 || ldb % 4 || K < (rows == FX_A_M_B_N ? FX_DW_SAMPLES : 64)) return false;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) return false;
  if (static_cast<long>(M) * K >= (1L << 29) || static_cast<long>(N) * K >= (1L << 29)) return false;
  return fx_plan(M, N, K).ok;
}

size_t fc_x3_workspace_bytes(int M, int N, int K) {
  const FxPlan p = fx_plan(M, N, K);
  return p.ok && p.splits > 1 ? ws_align(sizeof(float) * p.splits * static_cast<size_t>(M) * N) : 0;
}

template <class Epi>
static int run_fx(FxRows rows, const float *A, const float *B, int lda, int ldb, const Epi &epi, int M, int N, int K,
                  const char *tag, const char *reduce_tag, LeftSums *leave = nullptr) {
  const FxPlan p = fx_plan(M, N, K);
  float *partial = nullptr;
  if (p.splits > 1) {
    void *ws = nullptr;
    TDH_TRY(ws_take(sizeof(float) * p.splits * static_cast<size_t>(M) * N, &ws));
    partial = static_cast<float *>(ws);
  }
  {
    ProfScope prof(tag, M, N, K);
    if constexpr (std::is_same<Epi, EpiRowMajorAct>::value)
      TDH_TRY((launch_fx<true, false>(p, A, B, lda, ldb, epi, M, N, K, partial)));
    else
      TDH_TRY(rows == FX_A_K_B_K   ? (launch_fx<true, true>(p, A, B, lda, ldb, epi, M, N, K, partial))
              : rows == FX_A_K_B_N ? (launch_fx<true, false>(p, A, B, lda, ldb, epi, M, N, K, partial))
                                   : (launch_fx<false, false>(p, A, B, lda, ldb, epi, M, N, K, partial)));
  }
  if constexpr (std::is_same<Epi, EpiRowMajor>::value) {
    if (leave && p.splits > 1 && !ctx().defer_reduce && N % 4 == 0 && static_cast<long>(M) * N >= REDUCE_WIDE_MIN) {
      *leave = LeftSums{partial, p.splits, M, N, epi};   // (the order of the wide kernel, which would add them up)
      return TDH_OK;
    }
  }
  return p.splits > 1 ? launch_splitk_reduce(partial, p.splits, M, N, epi, reduce_tag) : TDH_OK;
}
int fc_x3_run(FxRows rows, const float *A, const float *B, int lda, int ldb, const EpiRowMajor &epi, int M, int N, int K,
              const char *tag, const char *reduce_tag, LeftSums *leave) {
  return run_fx(rows, A, B, lda, ldb, epi, M, N, K, tag, reduce_tag, leave);
}
int fc_x3_run_act(const float *A, const float *B, int lda, int ldb, const EpiRowMajorAct &epi, int M, int N, int K,
                  const char *tag, const char *reduce_tag) {
  return run_fx(FX_A_K_B_N, A, B, lda, ldb, epi, M, N, K, tag, reduce_tag);
}

}  // namespace tdh
