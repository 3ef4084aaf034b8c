// FP32-MFMA GEMM for gfx950 on float64 operands:
//   C[m][n] = alpha * sum_k fl32(A[m][k]) * fl32(B[n][k]) + beta * C[m][n]
// (row-major, both operands K-contiguous, C float64).  The contractions of the FP32
// precision mode (force bias, VHS) read the same float64 operands as the float64 path;
// each element is rounded to float32 as it is staged into LDS and the products run on
// v_mfma_f32_16x16x4f32 with float32 accumulation, so the mode needs no extra copies of
// the Cholesky vectors or the Green's function.
//
// v_mfma_f32_16x16x4f32 lane layout (as v_mfma_f64_16x16x4f64 for the operands, as the
// other float32-accumulating 16 x 16 MFMAs for the result):
//   A operand: lane l holds A[l % 16][l / 16]
//   B operand: lane l holds B[l / 16][l % 16]   (B as k x n)
//   D (float4): lane l, element r holds D[4 (l / 16) + r][l % 16]
//
// Tiles of BM x BN with BK = 16, four waves (2 x 2), float operands in LDS (double buffered,
// register prefetch of the next k-tile).  Split-K as in the float64 GEMM: grid.y splits K and
// split z writes alpha * its partial product to C + z * c_split_stride (beta must be 0);
// consumers add the slices in order.
//
// As in the float64 GEMM, operand loads are 16 bytes and unconditional, from clamped rows and
// k at any 8-byte boundary (masked loads waited one by one, and odd K read 8 bytes at a
// time), and k past the range is zeroed as the registers go to LDS.  An LDS row of 16 floats
// is four 16-byte chunks, element e of chunk c being k = 4 e + c, so one read per lane and
// row feeds the four MFMAs of a k-tile, each of four consecutive k; chunk c of row r sits at
// c ^ ((r >> 1) & 3), under which the sixteen rows of a chunk meet no bank twice.
// A step's two, 1200 x 2701 x 301 and 1200 x 301 x 1241: 62 -> 29 us on average.
#include "common.h"

namespace {

constexpr int F32_BK = 16;
constexpr int F32_RCH = F32_BK / 4;  // chunks per LDS row
// 16 bytes at any 8-byte boundary (rows of odd length)
typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef double d2_t __attribute__((ext_vector_type(2)));

template <int BM, int BN, int WM, int WN>
__device__ __forceinline__ void gemm_nt_f32_body(
    int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double beta, double* __restrict__ C, int ldc,
    int tiles_m, int tiles_n, int k_per_split, int64_t c_split_stride, const int bx,
    const int by) {
  constexpr int BK = F32_BK, RCH = F32_RCH;
  constexpr int TM = BM / WM / 16;
  constexpr int TN = BN / WN / 16;
  constexpr int A_LD = BM / 32, B_LD = BN / 32;  // 8 threads to a row
  static_assert(WM * WN == 4, "four waves");

  __shared__ float4_t As[2][BM * RCH];
  __shared__ float4_t Bs[2][BN * RCH];

  int tile_m, tile_n;
  const bool m_major = M > N;
  const int band = xcd_band((int64_t)(m_major ? N : M) * k_per_split * 8,
                            (int64_t)(m_major ? BM : BN) * k_per_split * 8);
  xcd_tile(bx, tiles_m, tiles_n, m_major, band, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int kbeg = by * k_per_split;
  const int kend = (kbeg + k_per_split < K) ? kbeg + k_per_split : K;
  C += (int64_t)by * c_split_stride;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int lch = t & 7, lr = t >> 3;

  // rows past M or N read the last row: their products are never stored
  const double* Ab = A + (int64_t)m0 * lda;
  const double* Bb = B + (int64_t)n0 * ldb;
  int aoff[A_LD], boff[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) aoff[i] = min(lr + i * 32, M - 1 - m0) * lda;
#pragma unroll
  for (int i = 0; i < B_LD; ++i) boff[i] = min(lr + i * 32, N - 1 - n0) * ldb;
  d2_t ra[A_LD], rb[B_LD];
  // pairs past kend read elements kend - 1 and kend (the operands' allocations end with at
  // least one element of padding)
  auto load_tile = [&](int k0) {
    const int k = min(k0 + 2 * lch, kend - 1);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) ra[i] = *reinterpret_cast<const d2u_t*>(Ab + (aoff[i] + k));
#pragma unroll
    for (int i = 0; i < B_LD; ++i) rb[i] = *reinterpret_cast<const d2u_t*>(Bb + (boff[i] + k));
  };
  // the places of k = 2 lch and 2 lch + 1 in a row's floats (32-row steps keep them)
  const int c0 = (2 * lch) & 3, rsw = (lr >> 1) & 3;
  const int s0 = (lr * RCH + (c0 ^ rsw)) * 4 + (lch >> 1);
  const int s1 = (lr * RCH + ((c0 + 1) ^ rsw)) * 4 + (lch >> 1);
  auto store_tile = [&](int buf, int k0) {
    const bool ok0 = k0 + 2 * lch < kend, ok1 = k0 + 2 * lch + 1 < kend;
    float* a = reinterpret_cast<float*>(As[buf]);
    float* b = reinterpret_cast<float*>(Bs[buf]);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      a[s0 + i * 32 * BK] = ok0 ? (float)ra[i].x : 0.f;
      a[s1 + i * 32 * BK] = ok1 ? (float)ra[i].y : 0.f;
    }
#pragma unroll
    for (int i = 0; i < B_LD; ++i) {
      b[s0 + i * 32 * BK] = ok0 ? (float)rb[i].x : 0.f;
      b[s1 + i * 32 * BK] = ok1 ? (float)rb[i].y : 0.f;
    }
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  const int nk = (kend - kbeg + BK - 1) / BK;
  if (nk > 0) {
    load_tile(kbeg);
    store_tile(0, kbeg);
  }
  __syncthreads();
  const int co = (lane >> 4) ^ ((lane >> 1) & 3);
  const int am = (wm * (BM / WM) + (lane & 15)) * RCH + co;
  const int bn = (wn * (BN / WN) + (lane & 15)) * RCH + co;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const int knext = kbeg + (kt + 1) * BK;
    if (kt + 1 < nk) load_tile(knext);
    float4_t af[TM], bf[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = As[cur][am + i * 16 * RCH];
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = Bs[cur][bn + j * 16 * RCH];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][e], bf[j][e], acc[i][j], 0, 0, 0);
    if (kt + 1 < nk) store_tile(cur ^ 1, knext);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * (BN / WN) + j * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * (BM / WM) + i * 16 + 4 * (lane >> 4) + r;
        if (row < M && col < N) {
          double* p = C + (int64_t)row * ldc + col;
          const double v = alpha * (double)acc[i][j][r];
          *p = (beta == 0.0) ? v : v + beta * (*p);
        }
      }
    }
}

template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_nt_f32_kernel(
    int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double beta, double* __restrict__ C, int ldc,
    int tiles_m, int tiles_n, int k_per_split, int64_t c_split_stride) {
  gemm_nt_f32_body<BM, BN, 2, 2>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles_m,
                                      tiles_n, k_per_split, c_split_stride, blockIdx.x,
                                      blockIdx.y);
}

// grouped: problem p owns tiles [start[p], start[p + 1]), no split-K, beta = 0
template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_grouped_kernel(const GemmArgs* __restrict__ args,
                                                               const int* __restrict__ start,
                                                               int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const GemmArgs a = args[p];
  gemm_nt_f32_body<BM, BN, 2, 2>(a.M, a.N, a.K, (double)a.alpha,
                                      static_cast<const double*>(a.A), (int)a.lda,
                                      static_cast<const double*>(a.B), (int)a.ldb, 0.0,
                                      static_cast<double*>(a.C), (int)a.ldc, a.tiles_m, a.tiles_n,
                                      (a.K + F32_BK - 1) / F32_BK * F32_BK, 0,
                                      blockIdx.x - start[p], 0);
}

template <int BM, int BN>
int launch_f32_tiles(hipStream_t s, int M, int N, int K, double alpha, const double* A, int lda,
                     const double* B, int ldb, double beta, double* C, int ldc, int splits,
                     int k_per_split, int64_t c_split_stride) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  dim3 grid(tm * tn, splits);
  hipLaunchKernelGGL((gemm_nt_f32_kernel<BM, BN>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda,
                     B, ldb, beta, C, ldc, tm, tn, k_per_split, c_split_stride);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

}  // namespace

// 128-wide tiles where they make two rounds of the 256 CUs
int gemm_f32_tile(int M, int N, int splits) {
  return (int64_t)((M + 127) / 128) * ((N + 127) / 128) * splits >= 512 ? 128 : 64;
}

int launch_gemm_nt_f32_split(hipStream_t s, int M, int N, int K, double alpha, const double* A,
                             int lda, const double* B, int ldb, double* C, int ldc, int splits,
                             int64_t c_split_stride) {
  if (M <= 0 || N <= 0) return AFQMC_OK;
  if (K <= 0) return afqmc_set_error(AFQMC_ERR_ARG, "gemm: K=%d", K);
  if (splits < 1) splits = 1;
  int kps = (K + splits - 1) / splits;
  kps = (kps + F32_BK - 1) / F32_BK * F32_BK;
  if (gemm_f32_tile(M, N, splits) == 128)
    return launch_f32_tiles<128, 128>(s, M, N, K, alpha, A, lda, B, ldb, 0.0, C, ldc, splits,
                                      kps, c_split_stride);
  return launch_f32_tiles<64, 64>(s, M, N, K, alpha, A, lda, B, ldb, 0.0, C, ldc, splits, kps,
                                  c_split_stride);
}

int launch_gemm_nt_f32(hipStream_t s, int M, int N, int K, double alpha, const double* A,
                       int lda, const double* B, int ldb, double beta, double* C, int ldc) {
  if (M <= 0 || N <= 0) return AFQMC_OK;
  if (K <= 0) return afqmc_set_error(AFQMC_ERR_ARG, "gemm: K=%d", K);
  if (gemm_f32_tile(M, N, 1) == 128)
    return launch_f32_tiles<128, 128>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, 1, K, 0);
  return launch_f32_tiles<64, 64>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, 1, K, 0);
}

int launch_gemm_f32_grouped(hipStream_t s, int bm, const GemmArgs* args, const int* start,
                            int nprob, int nblocks) {
  if (bm == 128)
    hipLaunchKernelGGL((gemm_f32_grouped_kernel<128, 128>), dim3(nblocks), dim3(256), 0, s, args,
                       start, nprob);
  else
    hipLaunchKernelGGL((gemm_f32_grouped_kernel<64, 64>), dim3(nblocks), dim3(256), 0, s, args,
                       start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}
