// Split-bf16 ("bf16x3") GEMM for gfx950 on v_mfma_f32_16x16x32_bf16:
//   C[m][n] = alpha * sum_k A[m][k] * B[n][k]   (row-major, both operands K-contiguous)
// Each operand x is stored as two bf16 planes, x = hi + lo with hi = bf16(x) and
// lo = bf16(x - hi) (round to nearest even), so the pair carries 16 mantissa bits.  The
// product keeps the three leading terms  Ah Bh + Ah Bl + Al Bh  (the dropped Al Bl is
// ~2^-16 relative) with float32 accumulation in the MFMA.  Used for the Cholesky
// contractions of the mixed-precision step (VHS, force bias, local-energy f_g).
//
// v_mfma_f32_16x16x32_bf16 lane layout (measured on gfx950):
//   A: lane l holds A[l % 16][8 (l / 16) + e], e = 0..7      (16 bytes, K-contiguous)
//   B: lane l holds B[8 (l / 16) + e][l % 16]                  (= row l%16 of an NT B)
//   D (float4): lane l, element r holds D[4 (l / 16) + r][l % 16]
// Operands have rows of K elements, a multiple of 32 (zero padded), in blocks of 32 hi and 32
// lo values (bf_pos), so K needs no tail handling and an operand row of a k step is one line.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int BK = 32;
// LDS rows of one k step are 128 bytes: the four 16-byte chunks of the hi values, then of
// the lo ones, chunk c of row r at c ^ ((r >> 1) & 7): a wave reading 16 rows x 16 bytes at
// each of four chunks (an MFMA operand) then meets no bank conflicts.
constexpr int RCH = 8;

__device__ inline uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
  return (uint16_t)(u >> 16);
}
__device__ inline float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// x (float64, rows x cols, ld_src) -> hi / lo bf16 planes (rows x ld_dst, zero padded), or a
// split-bf16 operand at hi where lo is null
__global__ void split_bf16_kernel(int rows, int cols, const double* __restrict__ x, int64_t ld_src,
                                  uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                  int64_t ld_dst) {
  const int64_t total = (int64_t)rows * ld_dst;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / ld_dst, c = e - r * ld_dst;
    uint16_t h = 0, l = 0;
    if (c < cols) {
      const double v = x[r * ld_src + c];
      h = f32_to_bf16((float)v);
      l = f32_to_bf16((float)(v - (double)bf16_to_f32(h)));
    }
    if (lo) {
      hi[e] = h;
      lo[e] = l;
    } else {
      hi[bf_pos(e)] = h;
      hi[bf_pos(e) + BF_LO] = l;
    }
  }
}

// What bounds it: the operand lines each tile takes from L2.  Loads are 16 bytes and
// unconditional (rows past M or N read the last row, their products are never stored; a
// masked load compiles to a branch with its own wait), eight lanes to a line.
template <int BM, int BN, typename OutT>
__device__ __forceinline__ void gemm_nt_bf16x3_body(
    int M, int N, int K, float alpha, const uint16_t* __restrict__ A,
    const uint16_t* __restrict__ B, OutT* __restrict__ C, int64_t ldc, int tiles_m, int tiles_n,
    int k_per_split, int64_t c_split_stride, const int bx, const int by) {
  constexpr int TM = BM / 2 / 16, TN = BN / 2 / 16;  // 2 x 2 waves
  constexpr int A_LD = BM / 32, B_LD = BN / 32;      // 16-byte chunks per thread
  __shared__ u32x4_t sA[2][BM * RCH];
  __shared__ u32x4_t sB[2][BN * RCH];

  int tile_m, tile_n;
  // operand bytes: hi and lo values, 4 per element over this split's K
  const bool m_major = M > N;
  const int band = xcd_band((int64_t)(m_major ? N : M) * k_per_split * 4,
                            (int64_t)(m_major ? BM : BN) * k_per_split * 4);
  xcd_tile(bx, tiles_m, tiles_n, m_major, band, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int kbeg = by * k_per_split;
  const int kend = (kbeg + k_per_split < K) ? kbeg + k_per_split : K;
  C += (int64_t)by * c_split_stride;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int lch = t & 7, lr = t >> 3;

  const unsigned char* Ab = reinterpret_cast<const unsigned char*>(A + 2 * (int64_t)m0 * K);
  const unsigned char* Bb = reinterpret_cast<const unsigned char*>(B + 2 * (int64_t)n0 * K);
  uint32_t aoff[A_LD], boff[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) aoff[i] = 4 * min(lr + 32 * i, M - 1 - m0) * K + 16 * lch;
#pragma unroll
  for (int i = 0; i < B_LD; ++i) boff[i] = 4 * min(lr + 32 * i, N - 1 - n0) * K + 16 * lch;
  u32x4_t ra[A_LD], rb[B_LD];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_LD; ++i)
      ra[i] = *reinterpret_cast<const u32x4_t*>(Ab + 4 * k0 + aoff[i]);
#pragma unroll
    for (int i = 0; i < B_LD; ++i)
      rb[i] = *reinterpret_cast<const u32x4_t*>(Bb + 4 * k0 + boff[i]);
  };
  const int sidx = lr * RCH + (lch ^ ((lr >> 1) & 7));  // (32-row steps keep the order)
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_LD; ++i) sA[buf][sidx + i * 32 * RCH] = ra[i];
#pragma unroll
    for (int i = 0; i < B_LD; ++i) sB[buf][sidx + i * 32 * RCH] = rb[i];
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  const int nk = (kend - kbeg) / BK;
  if (nk > 0) {
    load_tile(kbeg);
    store_tile(0);
  }
  __syncthreads();
  // k chunk lane >> 4 of the hi values; of the lo values: chunk ^ 4
  const int koff = (lane >> 4) ^ ((lane >> 1) & 7);
  const int ao = (wm * (BM / 2) + (lane & 15)) * RCH, bo = (wn * (BN / 2) + (lane & 15)) * RCH;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load_tile(kbeg + (kt + 1) * BK);
    bf16x8_t ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      ah[i] = __builtin_bit_cast(bf16x8_t, sA[cur][ao + i * 16 * RCH + koff]);
      al[i] = __builtin_bit_cast(bf16x8_t, sA[cur][ao + i * 16 * RCH + (koff ^ 4)]);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      bh[j] = __builtin_bit_cast(bf16x8_t, sB[cur][bo + j * 16 * RCH + koff]);
      bl[j] = __builtin_bit_cast(bf16x8_t, sB[cur][bo + j * 16 * RCH + (koff ^ 4)]);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
      }
    if (kt + 1 < nk) store_tile(cur ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * (BN / 2) + j * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + r;
        if (row < M && col < N) C[(int64_t)row * ldc + col] = (OutT)(alpha * acc[i][j][r]);
      }
    }
}

template <int BM, int BN, typename OutT>
__global__ __launch_bounds__(256, 2) void gemm_nt_bf16x3_kernel(
    int M, int N, int K, float alpha, const uint16_t* __restrict__ A,
    const uint16_t* __restrict__ B, OutT* __restrict__ C, int64_t ldc, int tiles_m, int tiles_n,
    int k_per_split, int64_t c_split_stride) {
  gemm_nt_bf16x3_body<BM, BN, OutT>(M, N, K, alpha, A, B, C, ldc, tiles_m, tiles_n, k_per_split,
                                    c_split_stride, blockIdx.x, blockIdx.y);
}

// grouped: problem p owns tiles [start[p], start[p + 1]), no split-K
template <int BM, int BN, typename OutT>
__global__ __launch_bounds__(256, 2) void gemm_bf16x3_grouped_kernel(
    const GemmArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const GemmArgs a = args[p];
  gemm_nt_bf16x3_body<BM, BN, OutT>(a.M, a.N, a.K, a.alpha, static_cast<const uint16_t*>(a.A),
                                    static_cast<const uint16_t*>(a.B), static_cast<OutT*>(a.C),
                                    a.ldc, a.tiles_m, a.tiles_n, a.K, 0, blockIdx.x - start[p], 0);
}

template <int BM, int BN, typename OutT>
int launch_bf(hipStream_t s, int M, int N, int K, float alpha, const uint16_t* A,
              const uint16_t* B, OutT* C, int64_t ldc, int splits, int kps,
              int64_t c_split_stride) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_nt_bf16x3_kernel<BM, BN, OutT>), dim3(tm * tn, splits), dim3(256), 0,
                     s, M, N, K, alpha, A, B, C, ldc, tm, tn, kps, c_split_stride);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <typename OutT>
int gemm_bf16x3(hipStream_t s, int M, int N, int K, float alpha, const uint16_t* A,
                const uint16_t* B, OutT* C, int64_t ldc, int splits, int64_t c_split_stride) {
  if (M <= 0 || N <= 0) return AFQMC_OK;
  if (K <= 0 || K % BK) return afqmc_set_error(AFQMC_ERR_ARG, "bf16x3 gemm: K=%d", K);
  if (splits < 1) splits = 1;
  int kps = (K / BK + splits - 1) / splits * BK;
  if (gemm_bf16x3_tile(M, N, splits) == 128)
    return launch_bf<128, 128, OutT>(s, M, N, K, alpha, A, B, C, ldc, splits, kps,
                                     c_split_stride);
  return launch_bf<64, 64, OutT>(s, M, N, K, alpha, A, B, C, ldc, splits, kps, c_split_stride);
}

}  // namespace

// 128-wide tiles where they make two rounds of the 256 CUs
int gemm_bf16x3_tile(int M, int N, int splits) {
  return (int64_t)((M + 127) / 128) * ((N + 127) / 128) * splits >= 512 ? 128 : 64;
}

int launch_split_bf16(hipStream_t s, int rows, int cols, const double* x, int64_t ld_src,
                      uint16_t* hi, uint16_t* lo, int64_t ld_dst) {
  const int64_t total = (int64_t)rows * ld_dst;
  if (total <= 0) return AFQMC_OK;
  const int64_t blocks = (total + 255) / 256 < 65536 ? (total + 255) / 256 : 65536;
  hipLaunchKernelGGL(split_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0, s, rows, cols, x,
                     ld_src, hi, lo, ld_dst);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

int launch_gemm_nt_bf16x3_f32(hipStream_t s, int M, int N, int K, float alpha, const uint16_t* A,
                              const uint16_t* B, float* C, int64_t ldc, int splits,
                              int64_t c_split_stride) {
  return gemm_bf16x3<float>(s, M, N, K, alpha, A, B, C, ldc, splits, c_split_stride);
}

int launch_gemm_nt_bf16x3_f64(hipStream_t s, int M, int N, int K, float alpha, const uint16_t* A,
                              const uint16_t* B, double* C, int64_t ldc, int splits,
                              int64_t c_split_stride) {
  return gemm_bf16x3<double>(s, M, N, K, alpha, A, B, C, ldc, splits, c_split_stride);
}

int launch_gemm_bf16x3_grouped(hipStream_t s, int bm, int out, const GemmArgs* args,
                               const int* start, int nprob, int nblocks) {
  if (bm == 128) {
    if (out)
      hipLaunchKernelGGL((gemm_bf16x3_grouped_kernel<128, 128, float>), dim3(nblocks), dim3(256),
                         0, s, args, start, nprob);
    else
      hipLaunchKernelGGL((gemm_bf16x3_grouped_kernel<128, 128, double>), dim3(nblocks),
                         dim3(256), 0, s, args, start, nprob);
  } else {
    if (out)
      hipLaunchKernelGGL((gemm_bf16x3_grouped_kernel<64, 64, float>), dim3(nblocks), dim3(256), 0,
                         s, args, start, nprob);
    else
      hipLaunchKernelGGL((gemm_bf16x3_grouped_kernel<64, 64, double>), dim3(nblocks), dim3(256),
                         0, s, args, start, nprob);
  }
  LAUNCH_CHECK();
  return AFQMC_OK;
}
