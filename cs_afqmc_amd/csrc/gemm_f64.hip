// FP64 MFMA GEMM for gfx950:  C[m][n] = alpha * sum_k A[m][k] * B[n][k] + beta * C[m][n]
// (row-major, both operands K-contiguous).  Used for the Cholesky contractions of the
// step: force bias (split Green x rot_chol^T), VHS (i sqrt(dt) x~ x chol) and the
// local-energy f_g matrices (rot_chol x Green^T).
//
// v_mfma_f64_16x16x4f64 lane layout (measured on gfx950):
//   A operand: lane l holds A[l % 16][l / 16]
//   B operand: lane l holds B[l / 16][l % 16]
//   D (double4): lane l, element r holds D[l / 16 + 4 r][l % 16]
//
// Tiles of BM x BN with BK = 16, four waves (2 x 2), double buffered in LDS with the next
// k-tile's loads in flight in registers.  Optional split-K: grid.y splits the K range and
// each split writes alpha * partial product to its own slice C + split * c_split_stride
// (beta must be 0); consumers sum the slices in order.
//
// What bounds it: one 16 x 16 x 4 MFMA takes 64 cycles, so four 4 x 4-tile waves need 4096
// MFMA cycles per k-tile and everything else has to stay off that path.
//   - Operand loads are 16-byte and unconditional, from clamped rows and k (a masked load
//     compiles to a branch with its own wait, which serialised the loads of a k-tile); k
//     past the range is zeroed on both operands when the registers go to LDS.
//   - LDS tiles keep the row-major order of memory (16 doubles = 8 chunks of 16 bytes per
//     row), so staging is one 16-byte store per load instead of a scatter of 8-byte ones,
//     and an operand read is one 16-byte chunk per lane: k = 2 c and 2 c + 1 of chunk
//     c = 4 ks + lane / 16, which feeds two MFMAs (any order of k serves, as long as both
//     operands share it).  Chunk c of row r sits at c ^ ((r >> 1) & 7): the sixteen rows
//     of one chunk then cover all 64 banks once.
#include "common.h"

namespace {

constexpr int GEMM_BK = 16;
// 16 bytes at any 8-byte boundary (rows of odd length)
typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef double d2_t __attribute__((ext_vector_type(2)));

template <int BM, int BN, int WM, int WN>
__device__ __forceinline__ void gemm_nt_f64_body(
    int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double beta, double* __restrict__ C, int ldc,
    int tiles_m, int tiles_n, int k_per_split, int64_t c_split_stride, const int bx,
    const int by) {
  constexpr int NT = 256;
  constexpr int BK = GEMM_BK;
  constexpr int CH = BK / 2;  // 16-byte chunks per row
  constexpr int TM = BM / WM / 16;
  constexpr int TN = BN / WN / 16;
  constexpr int RSTEP = NT / CH;  // rows covered per load pass
  constexpr int A_LD = BM / RSTEP;
  constexpr int B_LD = BN / RSTEP;
  static_assert(WM * WN == 4, "four waves");
  static_assert(A_LD >= 1 && B_LD >= 1, "tile too small");

  __shared__ d2_t As[2][BM * CH];
  __shared__ d2_t Bs[2][BN * CH];

  // XCD-aware block -> tile map (contiguous tile runs per XCD; the larger operand's
  // panels are the shared ones)
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
  const int lch = t % CH, lr = t / CH;

  // rows past M or N read the last row: their products are never stored
  const double* Ab = A + (int64_t)m0 * lda;
  const double* Bb = B + (int64_t)n0 * ldb;
  int aoff[A_LD], boff[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) aoff[i] = min(lr + i * RSTEP, M - 1 - m0) * lda;
#pragma unroll
  for (int i = 0; i < B_LD; ++i) boff[i] = min(lr + i * RSTEP, N - 1 - n0) * ldb;
  d2_t ra[A_LD], rb[B_LD];
  // chunks past kend read elements kend - 1 and kend (the operands' allocations end with
  // at least one element of padding)
  auto load_tile = [&](int k0) {
    const int k = min(k0 + 2 * lch, kend - 1);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) ra[i] = *reinterpret_cast<const d2u_t*>(Ab + (aoff[i] + k));
#pragma unroll
    for (int i = 0; i < B_LD; ++i) rb[i] = *reinterpret_cast<const d2u_t*>(Bb + (boff[i] + k));
  };
  const int sidx = lr * CH + (lch ^ ((lr >> 1) & 7));  // (RSTEP is a multiple of 16 rows)
  auto store_tile = [&](int buf, int k0) {
    const bool ok0 = k0 + 2 * lch < kend, ok1 = k0 + 2 * lch + 1 < kend;
#pragma unroll
    for (int i = 0; i < A_LD; ++i)
      As[buf][sidx + i * RSTEP * CH] = d2_t{ok0 ? ra[i].x : 0.0, ok1 ? ra[i].y : 0.0};
#pragma unroll
    for (int i = 0; i < B_LD; ++i)
      Bs[buf][sidx + i * RSTEP * CH] = d2_t{ok0 ? rb[i].x : 0.0, ok1 ? rb[i].y : 0.0};
  };

  double4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  const int nk = (kend - kbeg + BK - 1) / BK;
  if (nk > 0) {
    load_tile(kbeg);
    store_tile(0, kbeg);
  }
  __syncthreads();
  const int am = (wm * (BM / WM) + (lane & 15)) * CH;
  const int bn = (wn * (BN / WN) + (lane & 15)) * CH;
  const int kq = lane >> 4, sw = (lane >> 1) & 7;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const int knext = kbeg + (kt + 1) * BK;
    if (kt + 1 < nk) load_tile(knext);
#pragma unroll
    for (int ks = 0; ks < BK / 8; ++ks) {
      d2_t af[TM], bf[TN];
      const int co = (ks * 4 + kq) ^ sw;
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = As[cur][am + i * 16 * CH + co];
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = Bs[cur][bn + j * 16 * CH + co];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i].x, bf[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i].y, bf[j].y, acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) store_tile(cur ^ 1, knext);
    __syncthreads();
  }

  // epilogue
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * (BN / WN) + j * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * (BM / WM) + i * 16 + (lane >> 4) + 4 * r;
        if (row < M && col < N) {
          double* p = C + (int64_t)row * ldc + col;
          const double v = alpha * acc[i][j][r];
          *p = (beta == 0.0) ? v : v + beta * (*p);
        }
      }
    }
}

// two waves per SIMD (two 128 x 128 workgroups per CU): without the bound the 128-wide
// tile takes 336 registers
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256, 2) void gemm_nt_f64_kernel(
    int M, int N, int K, double alpha, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double beta, double* __restrict__ C, int ldc,
    int tiles_m, int tiles_n, int k_per_split, int64_t c_split_stride) {
  gemm_nt_f64_body<BM, BN, WM, WN>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles_m,
                                        tiles_n, k_per_split, c_split_stride, blockIdx.x,
                                        blockIdx.y);
}

// grouped: problem p owns tiles [start[p], start[p + 1]), no split-K, beta = 0
template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f64_grouped_kernel(const GemmArgs* __restrict__ args,
                                                               const int* __restrict__ start,
                                                               int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const GemmArgs a = args[p];
  gemm_nt_f64_body<BM, BN, 2, 2>(a.M, a.N, a.K, (double)a.alpha,
                                      static_cast<const double*>(a.A), (int)a.lda,
                                      static_cast<const double*>(a.B), (int)a.ldb, 0.0,
                                      static_cast<double*>(a.C), (int)a.ldc, a.tiles_m, a.tiles_n,
                                      (a.K + GEMM_BK - 1) / GEMM_BK * GEMM_BK, 0,
                                      blockIdx.x - start[p], 0);
}

template <int BM, int BN>
int launch_tiles(hipStream_t s, int M, int N, int K, double alpha, const double* A, int lda,
                 const double* B, int ldb, double beta, double* C, int ldc, int splits,
                 int k_per_split, int64_t c_split_stride) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_nt_f64_kernel<BM, BN, 2, 2>), dim3(tm * tn, splits), dim3(256), 0, s,
                     M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tm, tn, k_per_split,
                     c_split_stride);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

}  // namespace

// Tile edge: a 128-wide tile runs at 65 TFLOP/s against 61 of a 64-wide one (8192 x 4096 x
// 4096), but in rounds of 256 tiles (one per CU) a partly filled last round weighs more.
// 128 where it has two rounds and still does more per round (measured at 2048 x 10000 x
// 400, 4.9 rounds: 280 against 317 us; 2048 x 5050 x 400, 2.5 rounds: 167 against 147).
int gemm_f64_tile(int M, int N, int splits) {
  const int64_t t128 = (int64_t)((M + 127) / 128) * ((N + 127) / 128) * splits;
  const int64_t t64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64) * splits;
  if (t128 < 512) return 64;
  const double e128 = (double)t128 / (double)((t128 + 255) / 256);
  const double e64 = (double)t64 / (double)((t64 + 255) / 256);
  return 65.0 * e128 > 61.0 * e64 ? 128 : 64;
}

int gemm_f64_splits(int M, int N, int K) {
  // split K only when the 64x64 tile grid cannot fill the 256 CUs twice over
  const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
  if (tiles >= 512) return 1;
  int sp = (int)((512 + tiles - 1) / tiles);
  const int max_sp = K / 256;  // keep >= 256 k per split
  if (sp > max_sp) sp = max_sp;
  if (sp > 8) sp = 8;
  return sp < 1 ? 1 : sp;
}

int launch_gemm_nt_f64_split(hipStream_t s, int M, int N, int K, double alpha, const double* A,
                             int lda, const double* B, int ldb, double* C, int ldc, int splits,
                             int64_t c_split_stride) {
  if (M <= 0 || N <= 0) return AFQMC_OK;
  if (K <= 0) return afqmc_set_error(AFQMC_ERR_ARG, "gemm: K=%d", K);
  if (splits < 1) splits = 1;
  int kps = (K + splits - 1) / splits;
  kps = (kps + GEMM_BK - 1) / GEMM_BK * GEMM_BK;
  if (gemm_f64_tile(M, N, splits) == 128)
    return launch_tiles<128, 128>(s, M, N, K, alpha, A, lda, B, ldb, 0.0, C, ldc, splits, kps,
                                  c_split_stride);
  return launch_tiles<64, 64>(s, M, N, K, alpha, A, lda, B, ldb, 0.0, C, ldc, splits, kps,
                              c_split_stride);
}

int launch_gemm_nt_f64(hipStream_t s, int M, int N, int K, double alpha, const double* A,
                       int lda, const double* B, int ldb, double beta, double* C, int ldc) {
  if (M <= 0 || N <= 0) return AFQMC_OK;
  if (K <= 0) return afqmc_set_error(AFQMC_ERR_ARG, "gemm: K=%d", K);
  if (gemm_f64_tile(M, N, 1) == 128)
    return launch_tiles<128, 128>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, 1, K, 0);
  return launch_tiles<64, 64>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, 1, K, 0);
}

int launch_gemm_f64_grouped(hipStream_t s, int bm, const GemmArgs* args, const int* start,
                            int nprob, int nblocks) {
  if (bm == 128)
    hipLaunchKernelGGL((gemm_f64_grouped_kernel<128, 128>), dim3(nblocks), dim3(256), 0, s, args,
                       start, nprob);
  else
    hipLaunchKernelGGL((gemm_f64_grouped_kernel<64, 64>), dim3(nblocks), dim3(256), 0, s, args,
                       start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

namespace {

// dst (cols x rows) = src (rows x cols)^T through 32 x 32 LDS tiles.  With n > 0 (cols =
// n^2) only the columns (p, k), p <= k, of a row's n x n matrix are kept: dst row
// p n - p (p - 1) / 2 + k - p, the upper triangle row by row.
__global__ __launch_bounds__(256) void transpose_f64_kernel(int rows, int cols, int n,
                                                           const double* __restrict__ src,
                                                           double* __restrict__ dst) {
  __shared__ double tile[32][33];
  const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int j = ty; j < 32; j += 8) {
    const int r = r0 + j, c = c0 + tx;
    if (r < rows && c < cols) tile[j][tx] = src[(int64_t)r * cols + c];
  }
  __syncthreads();
  for (int j = ty; j < 32; j += 8) {
    int c = c0 + j;
    const int r = r0 + tx;
    if (r >= rows || c >= cols) continue;
    if (n) {
      const int p = c / n, k = c - p * n;
      if (k < p) continue;
      c = p * n - (p * (p - 1)) / 2 + k - p;
    }
    dst[(int64_t)c * rows + r] = tile[tx][j];
  }
}

// Symmetry of count n x n matrices: out[0] = max |L[p][k] - L[k][p]| and out[1] = max |L|
// as the bit patterns of non-negative doubles (ordered like the values, so integer maxima
// apply, and NaN, which fmax would drop, is the largest: vectors with an entry that is not
// finite never count as symmetric).  A block takes one pair (I, J), I <= J, of 32 x 32 tiles of one matrix, both
// read along rows, the second one compared through LDS.
__global__ __launch_bounds__(256) void sym_check_kernel(int n, int nt,
                                                        const double* __restrict__ L,
                                                        unsigned long long* __restrict__ out) {
  __shared__ double tile[32][33];
  int I = 0, J = blockIdx.x;
  while (J >= nt - I) J -= nt - I++;
  J += I;
  const double* m = L + (int64_t)blockIdx.y * n * n;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  unsigned long long asym = 0ull, amax = 0ull;
  auto bits = [](double x) { return (unsigned long long)__double_as_longlong(fabs(x)); };
  for (int j = ty; j < 32; j += 8) {
    const int r = J * 32 + j, c = I * 32 + tx;
    const double v = (r < n && c < n) ? m[(int64_t)r * n + c] : 0.0;
    tile[j][tx] = v;
    amax = max(amax, bits(v));
  }
  __syncthreads();
  for (int j = ty; j < 32; j += 8) {
    const int r = I * 32 + j, c = J * 32 + tx;
    if (r < n && c < n) {
      const double v = m[(int64_t)r * n + c];
      amax = max(amax, bits(v));
      asym = max(asym, bits(v - tile[tx][j]));
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    asym = max(asym, __shfl_xor(asym, off, 64));
    amax = max(amax, __shfl_xor(amax, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    // (a wave below the maximum so far leaves it alone: 10^5 waves share the two words)
    const unsigned long long v[2] = {asym, amax};
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (v[i] > __atomic_load_n(&out[i], __ATOMIC_RELAXED)) atomicMax(&out[i], v[i]);
  }
}

}  // namespace

int launch_transpose_f64(hipStream_t s, int rows, int cols, int packed_n, const double* src,
                         double* dst) {
  if (rows <= 0 || cols <= 0) return AFQMC_OK;
  dim3 grid((cols + 31) / 32, (rows + 31) / 32);
  if (grid.y > 65535) return afqmc_set_error(AFQMC_ERR_SIZE, "transpose: %d rows", rows);
  hipLaunchKernelGGL(transpose_f64_kernel, grid, dim3(256), 0, s, rows, cols, packed_n, src, dst);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

int launch_sym_check(hipStream_t s, int n, int64_t count, const double* L,
                     unsigned long long* out) {
  const int nt = (n + 31) / 32;
  for (int64_t c0 = 0; c0 < count; c0 += 65535) {
    const unsigned nc = (unsigned)(count - c0 < 65535 ? count - c0 : 65535);
    hipLaunchKernelGGL(sym_check_kernel, dim3(nt * (nt + 1) / 2, nc), dim3(256), 0, s, n, nt,
                       L + c0 * n * n, out);
    LAUNCH_CHECK();
  }
  return AFQMC_OK;
}
