// Local energy, rhf._calc_energy_restricted (wavefunctions.py:529-541) and
// uhf._calc_energy (wavefunctions.py:711-743):
//   f_g = rot_chol_s[g] G_s^T (n x n),  c_g = sum_s m_s tr f_g,  x_g = sum_s m_s tr(f_g f_g)
//   E = sum_g (c_g^2 - x_g) / 2 + sum_s m_s sum G_s * rot_h1_s + h0
// with m_s = 2 for restricted walkers (one spin standing for both) and 1 otherwise;
// for m = 2 this is 2 sum c^2 - exc + 2 sum G rot_h1 + h0, the restricted formula.
//
// c_g equals the force bias of the walker (fb_g = sum_s m_s sum_ip rot_chol_s[g,i,p]
// G_s[i,p], wavefunctions.py:503-511 / :694-709), so it comes from the float64
// force-bias GEMM.  The exchange sums x_g need every f_g: a fused kernel forms a tile
// of F[(g,i)][(w,c,j)] = sum_p rot_chol[g][i][p] green[w][c][j][p] on MFMA (float64, or
// split-bf16 with float32 accumulation in the mixed mode), holding whole (g, w) blocks
// -- g_per_tile = BM / n rows of g and w_per_tile = BN / 2n walkers -- so the tile is
// reduced to sum_g x_g per walker in LDS and F never reaches HBM.  Per-tile partial
// sums are added in tile order by the finishing kernel, so results are deterministic.
// The tile holds whole (g, w) blocks for n <= 64 occupied orbitals per spin, the
// library's limit (AFQMC_MAX_NOCC).
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int ENER_NT = 256;

// (g-tile, walker-tile) of block bx.  Blocks are dealt round-robin to the 8 XCDs (block
// b runs on XCD b % 8), each with its own 4 MB L2, and each XCD takes a contiguous run of
// the pairs in this order: chunks of gc g-tiles (as many Cholesky tiles as fill half an
// L2), within a chunk walker tiles slowest.  The blocks an XCD has in flight then share
// one or two walker tiles and cycle through Cholesky tiles that stay in its L2, so the
// Cholesky operand is fetched about once per XCD and chunk, and the Green's-function
// operand about once per chunk (instead of the whole Cholesky operand once per walker
// tile with g-tiles fastest).
__device__ inline void exchange_tile_of(int bx, int g_tiles, int w_tiles, int gc, int* gt,
                                        int* wt) {
  const int nblk = g_tiles * w_tiles;
  const int q = nblk >> 3, r = nblk & 7, x = bx & 7, i = bx >> 3;
  const int b = x * q + (x < r ? x : r) + i;
  const int per = gc * w_tiles, c = b / per, g0 = c * gc;
  const int gcc = g_tiles - g0 < gc ? g_tiles - g0 : gc;
  const int rem = b - c * per;
  *wt = rem / gcc;
  *gt = g0 + rem - (rem / gcc) * gcc;
}

// g-tiles per chunk of exchange_tile_of: Cholesky tiles of tile_bytes filling half an L2
inline int exchange_chunk(int g_tiles, int64_t tile_bytes) {
  const int64_t fit = (int64_t)(2 << 20) / (tile_bytes > 0 ? tile_bytes : 1);
  return fit < 1 ? 1 : (fit > g_tiles ? g_tiles : (int)fit);
}

// ---------------------------------------------------------------- fused exchange

// Exchange sums of a workgroup's F tile: F row gl*n + i, column wl*2n + 2j + c (the re and
// im of an entry side by side: the operand rows are staged in that order), and x_w =
// sum_g sum_ij f(i,j) f(j,i), taken over the pairs i <= j (weight 2 off the diagonal).  The
// tile goes through LDS in passes of as many whole g as fit EX_FR rows (write(r0, rows)
// stores rows r0 .. r0 + rows - 1 to Fs), so the operand buffers' LDS serves it and two or
// three workgroups share a CU: one reduces while the others multiply.  A wave's vector
// instructions and MFMAs take turns on its SIMD, so the instruction count of this part is
// what it costs: every thread takes (g, pair) items, with the pair from a table, and runs
// over the walkers; its sums stay in registers over the passes, EX_MAXW walkers at a time
// (tiles of more walkers, n <= 7, add up per pass instead).  Sums over threads: wave tree,
// then the waves in order.
constexpr int EX_NT = 256, EX_FR = 64, EX_MAXW = 8, EX_WMAX = 64;
static_assert(2 * EX_MAXW == 16, "exchange_wave_sums");

// (i, j), i <= j, of pair q = j (j + 1) / 2 + i
struct PairTable {
  uint16_t ij[AFQMC_MAX_NOCC * (AFQMC_MAX_NOCC + 1) / 2];
  constexpr PairTable() : ij() {
    int q = 0;
    for (int j = 0; j < AFQMC_MAX_NOCC; ++j)
      for (int i = 0; i <= j; ++i) ij[q++] = (uint16_t)(i | j << 8);
  }
};
__device__ const PairTable exchange_pairs{};

// operand row of F column col: column w*2n + 2j + c holds walker row w*2n + c*n + j
__device__ inline int exchange_col_row(int col, int n) {
  const int w = (int)(((float)col + 0.5f) * (1.0f / (float)(2 * n)));
  const int e = col - w * 2 * n;
  return w * 2 * n + (e & 1) * n + (e >> 1);
}

// Sum over the wave of each of 16 values, value l / 4 in lane l: a lane adds its partner's
// half of the values to its own and passes on the other half, 17 exchanges where a tree for
// each value takes 96, with the same additions in the same order.  Those trees were most of
// the reduction where a thread has few items and a tile many walkers.  Energies, us, with a
// tree for each value and so: one vector, n = 1, 64 walkers, split-bf16, 42.6 -> 27.7; norb
// 40, n = 6, 160 vectors, 512 walkers, split-bf16, 58.1 -> 47.0; norb 100, n = 20, 400
// vectors, 1024 walkers, float64 1649 -> 1591, split-bf16 524 -> 447.
template <int HALF>
__device__ __forceinline__ void exchange_halve(double (&v)[16], int lane) {
  const bool up = lane & (4 * HALF);
#pragma unroll
  for (int k = 0; k < HALF; ++k) {
    const double mine = up ? v[HALF + k] : v[k], give = up ? v[k] : v[HALF + k];
    v[k] = mine + __shfl_xor(give, 4 * HALF, 64);
  }
}
__device__ __forceinline__ double exchange_wave_sums(double (&v)[16], int lane) {
  exchange_halve<8>(v, lane);
  exchange_halve<4>(v, lane);
  exchange_halve<2>(v, lane);
  exchange_halve<1>(v, lane);
  v[0] += __shfl_xor(v[0], 2, 64);
  return v[0] + __shfl_xor(v[0], 1, 64);
}

template <typename T, typename WriteF>
__device__ __forceinline__ void exchange_reduce(T* Fs, int ldf, int n, int g_used, int w_used,
                                                int w0, cplx* __restrict__ xpart, cplx* parts,
                                                WriteF write) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int npairs = n * (n + 1) / 2;
  const float inv_pairs = 1.0f / (float)npairs;
  const int gpp = EX_FR / n;  // g per pass
  const bool persist = w_used <= EX_MAXW;
  double xr[EX_MAXW], xi[EX_MAXW];
#pragma unroll
  for (int k = 0; k < EX_MAXW; ++k) xr[k] = xi[k] = 0.0;
  for (int g0 = 0; g0 < g_used; g0 += gpp) {
    const int gn = min(gpp, g_used - g0);
    __syncthreads();  // the operands, or the last pass, are no longer read
    write(g0 * n, gn * n);
    __syncthreads();
    const bool last = g0 + gpp >= g_used;
    for (int wb = 0; wb < w_used; wb += EX_MAXW) {
      if (!persist) {
#pragma unroll
        for (int k = 0; k < EX_MAXW; ++k) xr[k] = xi[k] = 0.0;
      }
      for (int it = t; it < gn * npairs; it += EX_NT) {
        // (exact: the product is off by less than half of 1 / npairs)
        const int gl = (int)(((float)it + 0.5f) * inv_pairs);
        const int ij = exchange_pairs.ij[it - gl * npairs];
        const int i = ij & 255, j = ij >> 8;
        const T wgt = i == j ? (T)1 : (T)2;
        const T* pa = Fs + (gl * n + i) * ldf + wb * 2 * n + 2 * j;  // f(i, j)
        const T* pb = Fs + (gl * n + j) * ldf + wb * 2 * n + 2 * i;  // f(j, i)
#pragma unroll
        for (int k = 0; k < EX_MAXW; ++k)
          if (wb + k < w_used) {
            const T2 fa = *reinterpret_cast<const T2*>(pa + k * 2 * n);
            const T2 fb = *reinterpret_cast<const T2*>(pb + k * 2 * n);
            const double ar = (double)(wgt * fa.x), ai = (double)(wgt * fa.y);
            const double br = (double)fb.x, bi = (double)fb.y;
            xr[k] = fma(-ai, bi, fma(ar, br, xr[k]));
            xi[k] = fma(ai, br, fma(ar, bi, xi[k]));
          }
      }
      if (!persist || last) {
        double v[2 * EX_MAXW];
#pragma unroll
        for (int k = 0; k < EX_MAXW; ++k) {
          v[k] = xr[k];
          v[EX_MAXW + k] = xi[k];
        }
        const double sum = exchange_wave_sums(v, lane);
        const int k = (lane >> 2) & (EX_MAXW - 1);
        if ((lane & 3) == 0 && wb + k < w_used) {
          double* p = reinterpret_cast<double*>(parts + wave * EX_WMAX + wb + k) + (lane >> 5);
          *p = g0 == 0 || persist ? sum : *p + sum;
        }
      }
    }
  }
  __syncthreads();
  if (t < w_used) {
    cplx x = parts[t];
#pragma unroll
    for (int v = 1; v < 4; ++v) x = cadd(x, parts[v * EX_WMAX + t]);
    xpart[w0 + t] = x;
  }
}

// float64 MFMA tile BM x 16 TN (four waves, BM / 4 rows each), BK = 16, operands row-major
// in LDS as 16-byte chunks, double buffered, loaded 16 bytes at a time without conditions
// (rows past the operands read the last row, their products belong to no (g, w) block; k
// past N is zeroed as the registers go to LDS).  A lane's chunk feeds two float64 MFMAs or
// four float32 ones.  With F32 (the FP32 precision mode) the same tile runs on
// v_mfma_f32_16x16x4f32: operands rounded to float32 as they are staged, float32
// accumulation and F tile (its D rows are 4 (l / 16) + r instead of l / 16 + 4 r); the
// exchange sums still accumulate in float64.
constexpr int EF_BK = 16;
typedef double ef_d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef double ef_d2_t __attribute__((ext_vector_type(2)));
typedef float ef_f4_t __attribute__((ext_vector_type(4)));

template <bool F32, int BM, int TN>
struct EfTile {
  typedef typename std::conditional<F32, float, double>::type T;
  static constexpr int BN = 16 * TN, BNP = (BN + 31) / 32 * 32;  // staged B rows
  // an odd number of entries: reads down a column spread over the banks
  static constexpr int LDF = BN + 2;
  static constexpr int OPS = 2 * (BM + BNP) * EF_BK * (int)sizeof(T);
  static constexpr int F = (EX_FR * LDF * (int)sizeof(T) + 15) / 16 * 16;
  static constexpr int BODY = OPS > F ? OPS : F;
  static constexpr int LDS = BODY + 4 * EX_WMAX * (int)sizeof(cplx);
};

template <bool F32, int BM, int TN>
__device__ __forceinline__ void exchange_f64_body(const ExchArgs& x, const int bx) {
  typedef EfTile<F32, BM, TN> Tile;
  typedef typename Tile::T T;
  typedef typename std::conditional<F32, float4_t, double4_t>::type AccT;
  typedef typename std::conditional<F32, ef_f4_t, ef_d2_t>::type ChunkT;  // 16 bytes
  constexpr int TM = BM / 64, BK = EF_BK;
  constexpr int RCH = F32 ? 4 : 8;  // chunks per row
  constexpr int A_LD = BM / 32, B_LD = Tile::BNP / 32;
  __shared__ __attribute__((aligned(16))) unsigned char lds[Tile::LDS];
  constexpr int BUF = (BM + Tile::BNP) * RCH;
  ChunkT* ops = reinterpret_cast<ChunkT*>(lds);

  const int n = x.n, N = x.K;
  int gt, wt;
  exchange_tile_of(bx, x.g_tiles, (x.W + x.wpt - 1) / x.wpt, x.gc, &gt, &wt);
  const int g0 = gt * x.gpt, w0 = wt * x.wpt;
  const int m0 = g0 * n, n0 = w0 * 2 * n;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lch = t & 7, lr = t >> 3;
  const double* Ab = static_cast<const double*>(x.A) + (int64_t)m0 * N;
  const double* Bb = static_cast<const double*>(x.B) + (int64_t)n0 * N;
  int aoff[A_LD], boff[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) aoff[i] = min(lr + i * 32, x.G * n - 1 - m0) * N;
#pragma unroll
  for (int i = 0; i < B_LD; ++i)
    boff[i] = min(exchange_col_row(lr + i * 32, n), 2 * x.W * n - 1 - n0) * N;
  ef_d2_t ra[A_LD], rb[B_LD];
  // chunks past N read elements N - 1 and N (the operands' allocations end with at least
  // one element of padding)
  auto load_tile = [&](int k0) {
    const int k = min(k0 + 2 * lch, N - 1);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) ra[i] = *reinterpret_cast<const ef_d2u_t*>(Ab + (aoff[i] + k));
#pragma unroll
    for (int i = 0; i < B_LD; ++i) rb[i] = *reinterpret_cast<const ef_d2u_t*>(Bb + (boff[i] + k));
  };
  auto store_tile = [&](int buf, int k0) {
    const bool ok0 = k0 + 2 * lch < N, ok1 = k0 + 2 * lch + 1 < N;
    auto put = [&](int row, ef_d2_t v) {  // (32-row steps leave the swizzle unchanged)
      if constexpr (F32) {
        // element e of chunk c is k = 4 e + c: each MFMA sums four consecutive k
        float* p = reinterpret_cast<float*>(ops + buf * BUF + row * RCH);
        const int c = (2 * lch) & 3, sw = (lr >> 1) & 3;
        p[(c ^ sw) * 4 + (lch >> 1)] = ok0 ? (float)v.x : 0.f;
        p[((c + 1) ^ sw) * 4 + (lch >> 1)] = ok1 ? (float)v.y : 0.f;
      } else {
        ops[buf * BUF + row * RCH + (lch ^ ((lr >> 1) & 7))] =
            ef_d2_t{ok0 ? v.x : 0.0, ok1 ? v.y : 0.0};
      }
    };
#pragma unroll
    for (int i = 0; i < A_LD; ++i) put(lr + i * 32, ra[i]);
#pragma unroll
    for (int i = 0; i < B_LD; ++i) put(BM + lr + i * 32, rb[i]);
  };

  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = AccT{0, 0, 0, 0};

  const int am = wave * (BM / 4) + (lane & 15), bn = BM + (lane & 15);
  const int kq = lane >> 4;
  // one LDS chunk per lane and operand row: 8 (float64) or 16 (float32) k
  auto compute = [&](int cur, int ks) {
    const int co = F32 ? kq ^ ((lane >> 1) & 3) : (ks * 4 + kq) ^ ((lane >> 1) & 7);
    ChunkT af[TM], bf[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = ops[cur * BUF + (am + i * 16) * RCH + co];
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = ops[cur * BUF + (bn + j * 16) * RCH + co];
#pragma unroll
    for (int e = 0; e < (F32 ? 4 : 2); ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (F32)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][e], bf[j][e], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i][e], bf[j][e], acc[i][j], 0, 0, 0);
        }
  };
  const int nk = (N + BK - 1) / BK;
  load_tile(0);
  store_tile(0, 0);
  __syncthreads();
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const int cur = kt & 1;
    load_tile((kt + 1) * BK);
    compute(cur, 0);
    if (!F32) compute(cur, 1);
    store_tile(cur ^ 1, (kt + 1) * BK);
    __syncthreads();
  }
  compute((nk - 1) & 1, 0);
  if (!F32 && N - (nk - 1) * BK > 8) compute((nk - 1) & 1, 1);

  T* Fs = reinterpret_cast<T*>(lds);
  auto write = [&](int r0, int rows) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int rb = wave * (BM / 4) + i * 16 - r0;  // the same in the wave
      if (rb + 16 <= 0 || rb >= rows) continue;
      const int row = rb + (F32 ? 4 * kq : kq);
      T* p = Fs + row * Tile::LDF + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        constexpr int RS = F32 ? 1 : 4;
        if ((unsigned)(row + RS * r) < (unsigned)rows) {
#pragma unroll
          for (int j = 0; j < TN; ++j) p[RS * r * Tile::LDF + j * 16] = acc[i][j][r];
        }
      }
    }
  };
  exchange_reduce<T>(Fs, Tile::LDF, n, min(x.gpt, x.G - g0), min(x.wpt, x.W - w0), w0,
                     x.xpart + (int64_t)gt * x.W, reinterpret_cast<cplx*>(lds + Tile::BODY),
                     write);
}

// split-bf16 tile 128 x 32 TN on v_mfma_f32_16x16x32_bf16 (2 x 2 waves, each 64 x 16 TN),
// BK = 32; operand planes have K = Np32 (zero padded), so there is no k tail.  The operands
// go from memory straight to LDS (16 bytes a lane, 8 rows an instruction), single
// buffered: two or three workgroups share a CU, and one loads or reduces while the others
// multiply.  LDS rows (32 hi, then 32 lo values) have the chunk order c ^ ((r >> 1) & 7), as
// in the split-bf16 GEMM, under which the 16-row operand reads meet no LDS bank conflicts;
// the order is made by the address each lane loads from.
constexpr int EB_BM = 128, EB_BK = 32;
template <int TN>
struct EbTile {
  static constexpr int BN = 32 * TN;
  // an odd number of entries, and rows 4 apart 24 banks apart: neither the reads down a
  // column nor the stores of accumulators meet on a bank
  static constexpr int LDF = BN + 6;
  static constexpr int OPS = 2 * (EB_BM + BN) * EB_BK * 2;
  static constexpr int F = (EX_FR * LDF * 4 + 15) / 16 * 16;
  static constexpr int BODY = OPS > F ? OPS : F;
  static constexpr int LDS = BODY + 4 * EX_WMAX * (int)sizeof(cplx);
  static constexpr int WGS = TN <= 5 ? 3 : 2;  // workgroups per CU
  static_assert(WGS * LDS <= 160 * 1024, "workgroups per CU");
};

template <int TN>
__device__ __forceinline__ void exchange_bf16x3_body(const ExchArgs& x, const int bx) {
  typedef EbTile<TN> Tile;
  constexpr int BM = EB_BM, TM = 4, BK = EB_BK;
  constexpr int LD = 4 + TN;  // loads per wave and k step: 16 + 4 TN row groups
  __shared__ __attribute__((aligned(16))) unsigned char lds[Tile::LDS];

  const int n = x.n, K = x.K;
  int gt, wt;
  exchange_tile_of(bx, x.g_tiles, (x.W + x.wpt - 1) / x.wpt, x.gc, &gt, &wt);
  const int g0 = gt * x.gpt, w0 = wt * x.wpt;
  const int m0 = g0 * n, n0 = w0 * 2 * n;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave & 1, wn = wave >> 1;

  // LDS: the 128 rows of A, then the BN rows of B, 1 KB per group of 8 rows.  The wave's s-th
  // load is group wave + 4 s; rows past the operands read the last row (their products
  // belong to no (g, w) block).
  const unsigned char* Ab = static_cast<const unsigned char*>(x.A) + 4 * (int64_t)m0 * K;
  const unsigned char* Bb = static_cast<const unsigned char*>(x.B) + 4 * (int64_t)n0 * K;
  uint32_t off[LD];
  const int rl = lane >> 3;
#pragma unroll
  for (int s = 0; s < LD; ++s) {
    const int r = (wave + 4 * s) * 8 + rl;
    const int row = s < 4 ? min(r, x.G * n - 1 - m0)
                          : min(exchange_col_row(r - BM, n), 2 * x.W * n - 1 - n0);
    off[s] = 4 * row * K + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // k chunk lane >> 4 of the hi values; of the lo values: chunk ^ 4
  const int koff = ((lane >> 4) ^ ((lane >> 1) & 7)) * 16;
  const unsigned char* pa = lds + (wm * 64 + (lane & 15)) * 128;
  const unsigned char* pb = lds + (BM + wn * 16 * TN + (lane & 15)) * 128;
  for (int k0 = 0; k0 < K; k0 += BK) {
    if (k0) __syncthreads();  // the last step's operands are no longer read
#pragma unroll
    for (int s = 0; s < LD; ++s)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)((s < 4 ? Ab : Bb) + 4 * k0 + off[s]),
          (__attribute__((address_space(3))) void*)(lds + (wave + 4 * s) * 1024), 16, 0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    bf16x8_t ah[TM], al[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      ah[i] = *reinterpret_cast<const bf16x8_t*>(pa + i * 2048 + koff);
      al[i] = *reinterpret_cast<const bf16x8_t*>(pa + i * 2048 + (koff ^ 64));
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const bf16x8_t bh = *reinterpret_cast<const bf16x8_t*>(pb + j * 2048 + koff);
      const bf16x8_t bl = *reinterpret_cast<const bf16x8_t*>(pb + j * 2048 + (koff ^ 64));
#pragma unroll
      for (int i = 0; i < TM; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh, acc[i][j], 0, 0, 0);
    }
  }

  float* Fs = reinterpret_cast<float*>(lds);
  auto write = [&](int r0, int rows) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int rb = wm * 64 + i * 16 - r0;  // the same in the wave
      if (rb + 16 <= 0 || rb >= rows) continue;
      const int row = rb + 4 * (lane >> 4);
      float* p = Fs + row * Tile::LDF + wn * 16 * TN + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if ((unsigned)(row + r) < (unsigned)rows) {
#pragma unroll
          for (int j = 0; j < TN; ++j) p[r * Tile::LDF + j * 16] = acc[i][j][r];
        }
      }
    }
  };
  exchange_reduce<float>(Fs, Tile::LDF, n, min(x.gpt, x.G - g0), min(x.wpt, x.W - w0), w0,
                         x.xpart + (int64_t)gt * x.W,
                         reinterpret_cast<cplx*>(lds + Tile::BODY), write);
}

template <bool F32, int BM, int TN>
__global__ __launch_bounds__(EX_NT, 2) void exchange_f64_kernel(ExchArgs a) {
  exchange_f64_body<F32, BM, TN>(a, blockIdx.x);
}

template <bool F32, int BM, int TN>
__global__ __launch_bounds__(EX_NT, 2) void exchange_f64_grouped_kernel(
    const ExchArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  exchange_f64_body<F32, BM, TN>(args[p], blockIdx.x - start[p]);
}

template <int TN>
__global__ __launch_bounds__(EX_NT, EbTile<TN>::WGS) void exchange_bf16x3_kernel(ExchArgs a) {
  exchange_bf16x3_body<TN>(a, blockIdx.x);
}

template <int TN>
__global__ __launch_bounds__(EX_NT, EbTile<TN>::WGS) void exchange_bf16x3_grouped_kernel(
    const ExchArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  exchange_bf16x3_body<TN>(args[p], blockIdx.x - start[p]);
}

// E_w = sum_g (c_g^2 - x_g) / 2 + sum_s m_s sum G_s rot_h1_s + h0 with c_g the summed
// force-bias slices and x_g = sum over spins and g-tiles (in order) of m_s * xpart.
__device__ __forceinline__ void energy_finish_body(
    int G, int N, int nspin, int mult, int n0, int n1, const double* __restrict__ fb, int nparts,
    int64_t part_stride, const cplx* __restrict__ xpart, int gt0, int gt1, int W,
    const double* __restrict__ green0, const double* __restrict__ green1,
    const double* __restrict__ rot_h1_0, const double* __restrict__ rot_h1_1, double h0,
    cplx* __restrict__ energies, const int bx) {
  __shared__ double red[ENER_NT / 64];
  const int w = bx;
  double c2r = 0.0, c2i = 0.0;
  for (int g = threadIdx.x; g < G; g += ENER_NT) {
    const double* p = fb + (int64_t)w * 2 * G + g;
    double re = p[0], im = p[G];
    for (int s = 1; s < nparts; ++s) {
      re += p[s * part_stride];
      im += p[s * part_stride + G];
    }
    c2r += re * re - im * im;
    c2i += 2.0 * re * im;
  }
  double xr = 0.0, xi = 0.0;
  const int gts[2] = {gt0, gt1};
  const cplx* xs = xpart;
  for (int s = 0; s < nspin; ++s) {
    for (int t = threadIdx.x; t < gts[s]; t += ENER_NT) {
      const cplx v = xs[(int64_t)t * W + w];
      xr += mult * v.re;
      xi += mult * v.im;
    }
    xs += (int64_t)gts[s] * W;
  }
  const int ns[2] = {n0, n1};
  const double* gs[2] = {green0, green1};
  const double* hs[2] = {rot_h1_0, rot_h1_1};
  double e1r = 0.0, e1i = 0.0;
  for (int s = 0; s < nspin; ++s) {
    const int kd = ns[s] * N;
    const double* gr = gs[s] + (int64_t)w * 2 * kd;
    const double* gi = gr + kd;
    for (int e = threadIdx.x; e < kd; e += ENER_NT) {
      e1r += mult * gr[e] * hs[s][e];
      e1i += mult * gi[e] * hs[s][e];
    }
  }
  const double C2r = block_sum<ENER_NT>(c2r, red);
  const double C2i = block_sum<ENER_NT>(c2i, red);
  const double Xr = block_sum<ENER_NT>(xr, red);
  const double Xi = block_sum<ENER_NT>(xi, red);
  const double E1r = block_sum<ENER_NT>(e1r, red);
  const double E1i = block_sum<ENER_NT>(e1i, red);
  if (threadIdx.x == 0)
    energies[w] = cplx{(C2r - Xr) / 2.0 + E1r + h0, (C2i - Xi) / 2.0 + E1i};
}

__global__ __launch_bounds__(ENER_NT) void energy_finish_kernel(
    int G, int N, int nspin, int mult, int n0, int n1, const double* __restrict__ fb, int nparts,
    int64_t part_stride, const cplx* __restrict__ xpart, int gt0, int gt1, int W,
    const double* __restrict__ green0, const double* __restrict__ green1,
    const double* __restrict__ rot_h1_0, const double* __restrict__ rot_h1_1, double h0,
    cplx* __restrict__ energies) {
  energy_finish_body(G, N, nspin, mult, n0, n1, fb, nparts, part_stride, xpart, gt0, gt1, W,
                     green0, green1, rot_h1_0, rot_h1_1, h0, energies, blockIdx.x);
}

__global__ __launch_bounds__(ENER_NT) void energy_finish_grouped_kernel(
    const FinishArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const FinishArgs a = args[p];
  energy_finish_body(a.G, a.N, a.nspin, a.mult, a.n0, a.n1, a.fb, a.nparts, a.part_stride,
                     a.xpart, a.gt0, a.gt1, a.W, a.green0, a.green1, a.rot_h1_0, a.rot_h1_1,
                     a.h0, a.energies, blockIdx.x - start[p]);
}

}  // namespace

namespace {

// Exchange tile of a context and spin: rows bm holding gpt whole g, 16-column tiles tn (per
// workgroup; the split-bf16 one has two waves across, so tn is even there) holding wpt whole
// walkers.  Rows: 128, but 64 for n < 8 and where 128 would leave CUs idle (float64 / FP32).
// Columns: the width of the best filled columns, the wider one at equal fill.
enum { EXCH_BF16 = 0, EXCH_F64 = 1, EXCH_F32 = 2 };
struct ExchTile {
  int family, bm, tn, gpt, wpt;
};
ExchTile exchange_tile_for(const afqmc_ctx* c, int s) {
  const int n = c->nocc[s], W = c->d.n_walkers, G = c->d.nchol;
  ExchTile x;
  x.family = c->mixed ? EXCH_BF16 : (c->f32 ? EXCH_F32 : EXCH_F64);
  const int step = c->mixed ? 2 : 1;
  if (n < 16) {
    x.tn = 8;
  } else {
    const int fixed = c->mixed ? 0 : 2;
    x.tn = 8 * step;
    for (int tn = 8 * step; tn >= (c->mixed ? 4 : 5) * step; tn -= step)
      if ((16 * tn / (2 * n)) * (x.tn + fixed) > (16 * x.tn / (2 * n)) * (tn + fixed)) x.tn = tn;
  }
  x.bm = 128;
  if (!c->mixed) {
    const int gp = 128 / n, wp = 16 * x.tn / (2 * n);
    const int64_t blocks = (int64_t)((G + gp - 1) / gp) * ((W + wp - 1) / wp);
    if (n < 8 || blocks < 512) {
      x.bm = 64;
      x.tn = 8;
    }
  }
  x.gpt = x.bm / n;
  x.wpt = 16 * x.tn / (2 * n);
  return x;
}

template <bool GROUPED, typename Single, typename Grouped>
void launch_exchange_kernel(hipStream_t st, Single one, Grouped many, const ExchArgs& a,
                            const ExchArgs* args, const int* start, int nprob, int nblocks) {
  if constexpr (GROUPED)
    hipLaunchKernelGGL(many, dim3(nblocks), dim3(EX_NT), 0, st, args, start, nprob);
  else
    hipLaunchKernelGGL(one, dim3(nblocks), dim3(EX_NT), 0, st, a);
}

inline int exchange_kind(const ExchTile& x) { return (x.family * 256 + x.bm) * 32 + x.tn; }

template <bool GROUPED>
int launch_exchange(hipStream_t st, int kind, const ExchArgs& a, const ExchArgs* args,
                    const int* start, int nprob, int nblocks) {
#define EXCH_CASE(family, bm, tn, one, many)                                                  \
  case (family * 256 + bm) * 32 + tn:                                                         \
    launch_exchange_kernel<GROUPED>(st, one, many, a, args, start, nprob, nblocks);           \
    break;
#define EXCH_BF(t) \
  EXCH_CASE(EXCH_BF16, 128, 2 * t, exchange_bf16x3_kernel<t>, exchange_bf16x3_grouped_kernel<t>)
#define EXCH_F(family, f32, bm, t)                                     \
  EXCH_CASE(family, bm, t, (exchange_f64_kernel<f32, bm, t>), \
            (exchange_f64_grouped_kernel<f32, bm, t>))
  switch (kind) {
    EXCH_BF(4) EXCH_BF(5) EXCH_BF(6) EXCH_BF(7) EXCH_BF(8)
    EXCH_F(EXCH_F64, false, 128, 5) EXCH_F(EXCH_F64, false, 128, 6)
    EXCH_F(EXCH_F64, false, 128, 7) EXCH_F(EXCH_F64, false, 128, 8)
    EXCH_F(EXCH_F64, false, 64, 8)
    EXCH_F(EXCH_F32, true, 128, 5) EXCH_F(EXCH_F32, true, 128, 6)
    EXCH_F(EXCH_F32, true, 128, 7) EXCH_F(EXCH_F32, true, 128, 8)
    EXCH_F(EXCH_F32, true, 64, 8)
    default:
      return afqmc_set_error(AFQMC_ERR_STATE, "exchange: no kernel for tile %d", kind);
  }
#undef EXCH_F
#undef EXCH_BF
#undef EXCH_CASE
  LAUNCH_CHECK();
  return AFQMC_OK;
}

}  // namespace

int energy_g_tiles(const afqmc_ctx* c, int s) {
  if (c->nocc[s] < 1) return 0;
  const int gpt = exchange_tile_for(c, s).gpt;
  return (c->d.nchol + gpt - 1) / gpt;
}

void exchange_plan(const afqmc_ctx* c, int s, int W, ExchArgs* a, int* kind, int* nblocks) {
  static_assert(AFQMC_MAX_NOCC <= EX_FR && 2 * AFQMC_MAX_NOCC <= 128,
                "a (g, w) block must fit one tile and one pass");
  const int N = c->d.norb, G = c->d.nchol, n = c->nocc[s];
  cplx* xp = c->energy_x;
  for (int t = 0; t < s; ++t) xp += (int64_t)energy_g_tiles(c, t) * W;
  const ExchTile x = exchange_tile_for(c, s);
  *a = ExchArgs{};
  a->G = G;
  a->n = n;
  a->W = W;
  a->xpart = xp;
  a->gpt = x.gpt;
  a->wpt = x.wpt;
  a->g_tiles = (G + x.gpt - 1) / x.gpt;
  if (c->mixed) {
    a->K = c->Np32;
    a->gc = exchange_chunk(a->g_tiles, (int64_t)a->gpt * n * c->Np32 * 4);
    a->A = c->rot_chol_bf[s];
    a->B = c->green_bf[s];
  } else {
    a->K = N;
    a->gc = exchange_chunk(a->g_tiles, (int64_t)a->gpt * n * N * 8);
    a->A = c->rot_chol[s];
    a->B = c->green[s];
  }
  *kind = exchange_kind(x);
  *nblocks = a->g_tiles * ((W + a->wpt - 1) / a->wpt);
}

void energy_finish_args(const afqmc_ctx* c, int W, cplx* energies, FinishArgs* a) {
  *a = FinishArgs{};
  a->G = c->d.nchol;
  a->N = c->d.norb;
  a->nspin = c->nspin;
  a->mult = c->mult;
  a->n0 = c->nocc[0];
  a->n1 = c->nocc[1];
  a->nparts = c->fb_parts;
  a->gt0 = energy_g_tiles(c, 0);
  a->gt1 = c->nspin > 1 ? energy_g_tiles(c, 1) : 0;
  a->W = W;
  a->part_stride = (int64_t)2 * W * c->d.nchol;
  a->fb = c->fb;
  a->xpart = c->energy_x;
  a->green0 = c->green[0];
  a->green1 = c->green[1];
  a->rot_h1_0 = c->rot_h1[0];
  a->rot_h1_1 = c->rot_h1[1];
  a->h0 = c->h0;
  a->energies = energies;
}

int launch_exchange_grouped(hipStream_t st, int kind, const ExchArgs* args, const int* start,
                            int nprob, int nblocks) {
  return launch_exchange<true>(st, kind, ExchArgs{}, args, start, nprob, nblocks);
}

int launch_energy_finish_grouped(hipStream_t st, const FinishArgs* args, const int* start,
                                 int nprob, int nblocks) {
  hipLaunchKernelGGL(energy_finish_grouped_kernel, dim3(nblocks), dim3(ENER_NT), 0, st, args,
                     start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

// Needs the float64 Green's function of every spin in c->green (and, in the mixed mode,
// its split-bf16 planes) and the float64 force bias in c->fb (c->fb_parts slices).
int launch_energy(afqmc_ctx* c, int W, cplx* energies) {
  for (int s = 0; s < c->nspin; ++s) {
    ExchArgs a;
    int kind, nb;
    exchange_plan(c, s, W, &a, &kind, &nb);
    int rc = launch_exchange<false>(c->stream, kind, a, nullptr, nullptr, 0, nb);
    if (rc) return rc;
  }
  FinishArgs f;
  energy_finish_args(c, W, energies, &f);
  hipLaunchKernelGGL(energy_finish_kernel, dim3(W), dim3(ENER_NT), 0, c->stream, f.G, f.N,
                     f.nspin, f.mult, f.n0, f.n1, f.fb, f.nparts, f.part_stride, f.xpart, f.gt0,
                     f.gt1, W, f.green0, f.green1, f.rot_h1_0, f.rot_h1_1, f.h0, energies);
  LAUNCH_CHECK();
  return AFQMC_OK;
}
