// Trotterised propagator on walker tiles:  w <- E (t0 + sum_{k=1}^{K} V^k t0 / k!),
// t0 = E w, with E = exp_h1 (real N x N) and V = VHS (complex N x N, per walker).
// Follows propagator._apply_trotprop_det (propagation.py:67-92): carry_k = V carry_{k-1}
// unscaled, each term divided by k!, summed, then added to t0 (here in Horner form).
// Columns of a walker are independent under left multiplication.
#include <type_traits>

#include "common.h"

namespace {

// x / k for a small integer k, rk = 1 / k: the quotient corrected by its residual
__device__ inline double div_small(double x, double k, double rk) {
  const double q = x * rk;
  return fma(fma(-q, k, x), rk, q);
}

// ------------------------------------------------------------------------------------
// Streaming float64 form (N > 128 or n > 32).  One workgroup per walker of one spin and
// chunk of 16 of its columns; wave r owns output rows [16 r, 16 r + 16).  y = [yr | yi]
// lives in LDS, rows q of 32 doubles.  The rows of V stream from memory (L2 or HBM) once
// per Horner term as the A operand of v_mfma_f64_16x16x4f64: four real products per k
// group,
//   ur = Vr yr - Vi yi,  ui = Vr yi + Vi yr.
//
// What it is shaped by (measured at norb 131, 29 + 26 columns, 777 walkers, both spins:
// 1.89 ms with masked loads of one entry per k group):
//   - a block of 16 k is four MFMAs, number 2 h + e taking k = 16 g + 8 h + 2 s + e in the
//     lanes s = l / 16, so a lane reads two consecutive entries of its row at a time
//     instead of one entry of each of four k groups;
//   - the registers of a pair are refilled with the next block's entries as soon as its
//     MFMAs are issued: loads stay in flight under the other pair's MFMAs and the other
//     waves', without a second set of registers.  Registers decide here: two workgroups
//     have to share a CU to cover each other's barriers, and the dispatcher counts
//     ceil(waves / 4) waves on every SIMD for each;
//   - no copies or avoidable index arithmetic in the loop: VALU instructions take issue
//     slots from float64 MFMA.
// With V kept as its upper triangle, blocks right of the diagonal read rows as before,
// blocks left of it read the stored rows q, 16 consecutive p each, and the block on the
// diagonal reads entry by entry.
typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));

// the BLGP field of a float64 MFMA negates its operands; bit 0: A
constexpr int MFMA_NEG_A = 1;

constexpr int TS_RS = 32;  // doubles per LDS row
// Column c of row q of y sits at c ^ ts_swz(q): the B operands of a wave (rows 2 s + e,
// 16 columns each) and its stores of D tiles (rows s + 4 r) then meet both halves of the
// banks
__device__ inline int ts_swz(int q) { return (((q >> 1) ^ q) & 1) << 4; }

template <bool PACKED>
__device__ __forceinline__ void taylor_stream_body(int N, int n, int n_terms_k,
                                                   cplx* __restrict__ walkers,
                                                   const double* __restrict__ expE,
                                                   const double* __restrict__ vhs, int nv,
                                                   const int w, const int c0) {
  constexpr int RS = TS_RS;
  extern __shared__ double YS[];  // [16 ceil(N / 16)][RS]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = lane >> 4, col = lane & 15;
  const int rb = wave * 16;
  const int nb = (N + 15) >> 4;         // blocks of 16 k
  const int pc = min(rb + col, N - 1);  // A row of this lane (rows >= N are never stored)
  cplx* phi = walkers + (int64_t)w * N * n;
  const double* Vr = vhs + (int64_t)w * 2 * nv;
  const double* Vi = Vr + nv;
  // V planes hold all N^2 entries row-major, or (PACKED: nv = N(N+1)/2, symmetric V) the
  // upper triangle row by row: entry (a, b), a <= b, at a N - a (a - 1) / 2 + b - a

  // the walker's chunk; rows q >= N and columns past n zero
  for (int e = threadIdx.x; e < nb * 256; e += blockDim.x) {
    const int q = e >> 4, j = e & 15;
    const cplx z = phi[min(q, N - 1) * n + min(c0 + j, n - 1)];
    const bool ok = q < N && c0 + j < n;
    double* row = YS + q * RS;
    const int sw = ts_swz(q);
    row[j ^ sw] = ok ? z.re : 0.0;
    row[(16 + j) ^ sw] = ok ? z.im : 0.0;
  }
  __syncthreads();

  auto put = [&](const double4_t& yr, const double4_t& yi) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = rb + s + 4 * r;
      if (q < N) {
        double* row = YS + q * RS;
        const int sw = ts_swz(q);
        row[col ^ sw] = yr[r];
        row[(16 + col) ^ sw] = yi[r];
      }
    }
  };
  // loads at a uniform base plus a 32-bit byte offset
  auto at = [](const double* base, uint32_t o) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + o);
  };
  auto load2 = [](double* a, const double* base, uint32_t o) {
    const d2u_t x = *reinterpret_cast<const d2u_t*>(reinterpret_cast<const char*>(base) + o);
    a[0] = x.x;
    a[1] = x.y;
  };
  // entries past the row's end (of the last block) are zeroed: they meet zero rows of y
  auto mask = [&](double (&a)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      a[u] = 16 * (nb - 1) + 8 * (u >> 1) + 2 * s + (u & 1) < N ? a[u] : 0.0;
  };
  // B of the MFMAs with k = row + 2 s + e: two buffers, one read from LDS while the other
  // is in use
  struct Yop {
    double r, i;
  };
  const int sw0 = (s & 1) << 4;  // ts_swz of even rows 2 s; odd rows: the other half
  const double* y0r = YS + 2 * s * RS + (col ^ sw0);
  const double* y0i = YS + 2 * s * RS + (col ^ sw0 ^ 16);
  auto loady = [&](Yop& y, int row, int e) {
    y.r = (e ? y0i : y0r)[row * RS];
    y.i = (e ? y0r : y0i)[row * RS];
  };
  // One pass over k: mma(y, u) with the operand of MFMA u of each block, refill(g, h) once
  // pair h is free
  auto pass = [&](auto&& mma, auto&& refill, auto&& last) {
    Yop y0, y1;
    loady(y0, 0, 0);
#pragma unroll 1
    for (int g = 0; g < nb; ++g) {
      const int gn = g + 1 < nb ? g + 1 : 0;
      if (g == nb - 1) last();
      loady(y1, 16 * g + 1, 1);
      mma(y0, 0);
      __builtin_amdgcn_sched_barrier(0);
      loady(y0, 16 * g + 8, 0);
      mma(y1, 1);
      __builtin_amdgcn_sched_barrier(0);
      refill(gn, 0);
      loady(y1, 16 * g + 9, 1);
      mma(y0, 2);
      __builtin_amdgcn_sched_barrier(0);
      loady(y0, 16 * gn, 0);
      mma(y1, 3);
      __builtin_amdgcn_sched_barrier(0);
      refill(gn, 1);
    }
  };
  const double4_t z4 = {0.0, 0.0, 0.0, 0.0};
  double vr[4], vi[4];
  // E y, a real operator on both halves (rows of E in vr)
  const uint32_t erow = 8u * (uint32_t)(pc * N + 2 * s);
  auto load_e = [&](int g, int h) { load2(vr + 2 * h, expE, erow + 128u * g + 64u * h); };
  auto e_product = [&](double4_t& ar, double4_t& ai) {
    ar = ai = z4;
    load_e(0, 0);
    load_e(0, 1);
    pass(
        [&](const Yop& y, int u) {
          ar = __builtin_amdgcn_mfma_f64_16x16x4f64(vr[u], y.r, ar, 0, 0, 0);
          ai = __builtin_amdgcn_mfma_f64_16x16x4f64(vr[u], y.i, ai, 0, 0, 0);
        },
        load_e, [&]() { mask(vr); });
  };
  // pair h of block g of V
  const uint32_t vrow =
      8u * (uint32_t)(PACKED ? pc * N - (pc * (pc - 1)) / 2 - pc + 2 * s : pc * N + 2 * s);
  auto load_v = [&](int g, int h) {
    if (!PACKED || g > wave) {
      const uint32_t o = vrow + 128u * g + 64u * h;
      load2(vr + 2 * h, Vr, o);
      load2(vi + 2 * h, Vi, o);
    } else if (g < wave) {  // entries (q, p), q < p: rows q and q + 1 N - q - 1 apart
      const int q = 16 * g + 8 * h + 2 * s;
      const uint32_t o = 8u * (uint32_t)(q * N - (q * (q + 1)) / 2 + pc);
      const uint32_t o1 = o + 8u * (uint32_t)(N - q - 1);
      vr[2 * h] = at(Vr, o);
      vi[2 * h] = at(Vi, o);
      vr[2 * h + 1] = at(Vr, o1);
      vi[2 * h + 1] = at(Vi, o1);
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int q = min(16 * g + 8 * h + 2 * s + e, N - 1);
        const int a = min(pc, q), b = max(pc, q);
        const uint32_t o = 8u * (uint32_t)(a * N - (a * (a - 1)) / 2 + (b - a));
        vr[2 * h + e] = at(Vr, o);
        vi[2 * h + e] = at(Vi, o);
      }
    }
  };

  double4_t t0r, t0i, ur, ui;
  e_product(t0r, t0i);
  load_v(0, 0);
  load_v(0, 1);
  lds_barrier();
  put(t0r, t0i);
  lds_barrier();
#pragma unroll 1
  for (int k = n_terms_k; k >= 1; --k) {
    ur = ui = z4;
    // (the pass ends with block 0 of V loaded for the next term)
    pass(
        [&](const Yop& y, int u) {
          ur = __builtin_amdgcn_mfma_f64_16x16x4f64(vr[u], y.r, ur, 0, 0, 0);
          ui = __builtin_amdgcn_mfma_f64_16x16x4f64(vr[u], y.i, ui, 0, 0, 0);
          ur = __builtin_amdgcn_mfma_f64_16x16x4f64(vi[u], y.i, ur, 0, 0, MFMA_NEG_A);
          ui = __builtin_amdgcn_mfma_f64_16x16x4f64(vi[u], y.r, ui, 0, 0, 0);
        },
        load_v,
        [&]() {
          mask(vr);
          mask(vi);
        });
    lds_barrier();
    const double dk = (double)k, rk = 1.0 / dk;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ur[r] = t0r[r] + div_small(ur[r], dk, rk);
      ui[r] = t0i[r] + div_small(ui[r], dk, rk);
    }
    put(ur, ui);
    lds_barrier();
  }
  e_product(ur, ui);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int p = rb + s + 4 * r, j = c0 + col;
    if (p < N && j < n) phi[p * n + j] = cplx{ur[r], ui[r]};
  }
}

// Blocks are dealt round-robin to the 8 XCDs (block b on XCD b % 8): block
// b = 8 (q units + u) + r takes unit u (a column chunk of one spin) of walker 8 q + r, so
// the units of a walker run on one XCD, one dispatch round apart, and mostly share its V
// (the same one for both spins unless the vectors are spin resolved) through that XCD's
// L2; and the spins of a launch fill its last round together.
__device__ inline bool stream_block(int b, int W, int units, int* w, int* unit) {
  const int g = b >> 3;
  *unit = g % units;
  *w = 8 * (g / units) + (b & 7);
  return *w < W;
}

// column chunks of a spin with n columns
__host__ __device__ inline int stream_chunks(int n) { return (n + 15) / 16; }

// registers for two workgroups per CU up to STREAM_SMALL waves (N <= 192), else one
constexpr int STREAM_SMALL = 12;
constexpr int stream_threads(bool small) { return small ? 64 * STREAM_SMALL : 1024; }
constexpr int stream_wpe(bool small) { return small ? 6 : 4; }

template <bool SMALL>
__global__ __launch_bounds__(stream_threads(SMALL), stream_wpe(SMALL)) void taylor_stream_kernel(
    int N, int n0, int n1, int n_terms_k, int W, cplx* __restrict__ w0, cplx* __restrict__ w1,
    const double* __restrict__ e0, const double* __restrict__ e1, const double* __restrict__ v0,
    const double* __restrict__ v1, int nv) {
  const int u0 = stream_chunks(n0), u1 = n1 ? stream_chunks(n1) : 0;
  int w, u;
  if (!stream_block(blockIdx.x, W, u0 + u1, &w, &u)) return;
  const bool dn = u >= u0;
  const int n = dn ? n1 : n0, c0 = 16 * (dn ? u - u0 : u);
  cplx* wk = dn ? w1 : w0;
  const double *E = dn ? e1 : e0, *V = dn ? v1 : v0;
  if (nv == N * N)
    taylor_stream_body<false>(N, n, n_terms_k, wk, E, V, nv, w, c0);
  else
    taylor_stream_body<true>(N, n, n_terms_k, wk, E, V, nv, w, c0);
}

template <bool SMALL>
__global__ __launch_bounds__(stream_threads(SMALL), stream_wpe(SMALL)) void taylor_stream_grouped_kernel(
    const TaylorArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const TaylorArgs a = args[p];
  int w, u;
  if (!stream_block(blockIdx.x - start[p], a.W, stream_chunks(a.n), &w, &u)) return;
  if (a.nv == a.N * a.N)
    taylor_stream_body<false>(a.N, a.n, a.K, a.walkers, static_cast<const double*>(a.E),
                              static_cast<const double*>(a.vhs), a.nv, w, 16 * u);
  else
    taylor_stream_body<true>(a.N, a.n, a.K, a.walkers, static_cast<const double*>(a.E),
                             static_cast<const double*>(a.vhs), a.nv, w, 16 * u);
}

inline int stream_blocks(int W, int units) { return 8 * ((W + 7) / 8) * units; }
inline size_t stream_shm(int N) { return (size_t)((N + 15) / 16) * 16 * TS_RS * sizeof(double); }

// both spins of the context (or its one)
template <bool SMALL>
int launch_stream(afqmc_ctx* c, int W, cplx* wup, cplx* wdn) {
  const int N = c->d.norb, s1 = c->nspin - 1;
  const size_t shm = stream_shm(N);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)taylor_stream_kernel<SMALL>, shm, &lds_limit);
  if (rc) return rc;
  const int n0 = c->nocc[0], n1 = c->nspin == 2 ? c->nocc[1] : 0;
  const int units = stream_chunks(n0) + (n1 ? stream_chunks(n1) : 0);
  hipLaunchKernelGGL((taylor_stream_kernel<SMALL>), dim3(stream_blocks(W, units)),
                     dim3(64 * ((N + 15) / 16)), shm, c->stream, N, n0, n1, c->d.n_exp_terms - 1,
                     W, wup, wdn, c->exp_h1[0], c->exp_h1[s1], vhs_of(c, 0),
                     vhs_of(c, s1), c->vhs_nv);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

// ------------------------------------------------------------------------------------
// Register-resident form (N <= 128, n <= 32).  One workgroup per (walker, spin) of NW =
// ceil(N / 16) waves; wave r keeps rows [16 r, 16 r + 16) of A = [Vr | Vi] (N x 2Np, Np =
// N rounded up to 4) in registers for the whole series, so V is read from HBM once.  The
// complex product is one real product  [ur | ui] = [Vr | Vi] [[tr, ti], [-ti, tr]]  whose
// B operand lives in LDS as 2Np rows: rows [0, Np) = [tr | ti], rows [Np, 2Np) =
// [-ti | tr] (columns padded to CTP*16), so k-group kg reads rows 4 kg .. 4 kg + 3 of one
// uniform array.  The series is evaluated in Horner form  y <- t0 + V y / k  (k = K..1),
// which equals t0 + sum_k V^k t0 / k! of propagation.py:67-92.
//
// Bound by float64 MFMA once a walker's loads are out of the way, and a CU holds one or
// two walkers only (V fills the registers), so nothing may wait in turn:
//   - every load is unconditional, from a clamped index, and masked after; as masked loads
//     the 2Np / 4 loads of a V row each waited for HBM on their own;
//   - the walker and the rows of E are loaded first and V last, so V arrives while the
//     first product E w runs (the barriers wait for LDS only);
//   - the rows of E are whole in registers before their product, instead of one L2 round
//     trip per k group;
//   - y / k is a multiplication by 1 / k with one correction step, not a division.
template <int CTP>
struct RegTile {
  static constexpr int RS = 16 * CTP + ((CTP % 2 == 0) ? 16 : 0);  // == 16 (mod 32) doubles
};

template <int NW, int CTP>
__device__ __forceinline__ void taylor_reg_body(int N, int n, int n_terms_k,
                                                cplx* __restrict__ walkers,
                                                const double* __restrict__ expE,
                                                const double* __restrict__ vhs, int nv,
                                                const int w) {
  constexpr int NKG = 4 * NW;  // k-groups of one half (of E, Vr or Vi) for N = 16 NW
  constexpr int RS = RegTile<CTP>::RS;
  constexpr int NT = 64 * NW;
  extern __shared__ double TT[];  // [2 Np][RS]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rb = wave * 16;
  const int Np = (N + 3) & ~3;
  const int nkg = Np >> 2;         // k-groups in use: NKG - 3 <= nkg <= NKG
  const int s = lane >> 4, col = lane & 15;
  const int p = rb + col;          // A-operand row of this lane
  const int pc = min(p, N - 1);    // (rows p >= N are never stored)
  const int n2 = 2 * n;
  cplx* phi = walkers + (int64_t)w * N * n;
  const double* Vr = vhs + (int64_t)w * 2 * nv;
  const double* Vi = Vr + nv;
  // V planes hold all N^2 entries row-major, or (nv = N(N+1)/2, symmetric V) the upper
  // triangle row by row: entry (a, b), a <= b, at a N - a (a - 1) / 2 + b - a
  const bool packed = nv != N * N;

  // walker tile: [tr | ti] and [-ti | tr]; rows q >= N zero (whatever A holds there)
  for (int e = threadIdx.x; e < N * n; e += NT) {
    const int q = e / n, j = e - q * n;
    const cplx z = phi[e];
    double* up = TT + q * RS + j;
    double* lo = up + Np * RS;
    up[0] = z.re;
    up[n] = z.im;
    lo[0] = -z.im;
    lo[n] = z.re;
  }
  for (int e = threadIdx.x; e < (Np - N) * RS; e += NT)
    TT[N * RS + e] = TT[(Np + N) * RS + e] = 0.0;

  // rows of E, k-group kg: E[p][4 kg + s]; what is read past the row's end (the next row,
  // or the padding after the matrix) is zeroed before the product
  double ea[NKG];
  auto load_e = [&](const double* erow) {
#pragma unroll
    for (int kg = 0; kg < NKG; ++kg) ea[kg] = erow[4 * kg];
  };
  load_e(expE + (pc * N + s));
  __builtin_amdgcn_sched_barrier(0);
  // rows of V in registers: k-group kg, slot s -> column q = 4 kg + s, of which real and
  // imaginary part share the index.  The scheduling barriers keep the indices of a few
  // loads in registers, not of all.
  double vr[NKG], vi[NKG];
#pragma unroll
  for (int kg = 0; kg < NKG; ++kg) {
    const int qc = min(4 * kg + s, N - 1);
    const int a = min(pc, qc), b = max(pc, qc);
    const int idx = packed ? a * N - (a * (a - 1)) / 2 + (b - a) : pc * N + qc;
    vr[kg] = Vr[idx];
    vi[kg] = Vi[idx];
    if (kg % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();

  const double* bbase = TT + s * RS + col;  // + kg * 4 RS + ct * 16
  const double* blo = bbase + Np * RS;

  // y rows -> both halves (rows q >= N keep their zeros)
  auto put = [&](const double4_t* v) {
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rb + s + 4 * r;
        const int cc = ct * 16 + col;
        if (row < N) {
          TT[row * RS + cc] = v[ct][r];
          if (cc < n)
            TT[(Np + row) * RS + cc + n] = v[ct][r];
          else if (cc < n2)
            TT[(Np + row) * RS + cc - n] = -v[ct][r];
        }
      }
  };
  // acc += A y over the rows a[] of A and one half of y; B of k-group kg + 1 is read from
  // LDS under the MFMAs of kg
  auto product = [&](const double (&a)[NKG], const double* bb, double4_t* acc) {
    double b[CTP];
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) b[ct] = bb[ct * 16];
#pragma unroll
    for (int kg = 0; kg < NKG; ++kg) {
      if (kg < NKG - 3 || kg < nkg) {
        double bn[CTP];
#pragma unroll
        for (int ct = 0; ct < CTP; ++ct)
          bn[ct] = bb[(kg + 1 < NKG - 3 ? kg + 1 : min(kg + 1, nkg - 1)) * 4 * RS + ct * 16];
#pragma unroll
        for (int ct = 0; ct < CTP; ++ct)
          acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kg], b[ct], acc[ct], 0, 0, 0);
#pragma unroll
        for (int ct = 0; ct < CTP; ++ct) b[ct] = bn[ct];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto zero = [&](double4_t* acc) {
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) acc[ct] = double4_t{0.0, 0.0, 0.0, 0.0};
  };

  auto e_product = [&](double4_t* acc) {
#pragma unroll
    for (int kg = NKG - 4; kg < NKG; ++kg) ea[kg] = 4 * kg + s < N ? ea[kg] : 0.0;
    zero(acc);
    product(ea, bbase, acc);
  };

  double4_t t0[CTP], u[CTP];
  e_product(t0);
  lds_barrier();
  put(t0);
  lds_barrier();
#pragma unroll 1
  for (int k = n_terms_k; k >= 1; --k) {
    zero(u);
    product(vr, bbase, u);
    product(vi, blo, u);
    lds_barrier();
    const double dk = (double)k, rk = 1.0 / dk;
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[ct][r] = t0[ct][r] + div_small(u[ct][r], dk, rk);
    put(u);
    lds_barrier();
  }
  int eoff = pc * N + s;
  asm volatile("" : "+v"(eoff));  // (addressed anew: nothing of E stays in registers meanwhile)
  load_e(expE + eoff);
  e_product(u);
#pragma unroll
  for (int ct = 0; ct < CTP; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = rb + s + 4 * r;
      const int cc = ct * 16 + col;
      if (row < N && cc < n2) {
        double* dst = reinterpret_cast<double*>(phi + (int64_t)row * n + (cc < n ? cc : cc - n));
        dst[cc < n ? 0 : 1] = u[ct][r];
      }
    }
}

// waves of a register-form workgroup (a template key) and its column tiles
inline int reg_waves(int N) { return (N + 15) / 16; }
inline int reg_ct(int n) { return (2 * n + 15) / 16; }
inline size_t reg_shm(int N, int ct) {
  return (size_t)2 * ((N + 3) & ~3) * (16 * ct + ((ct % 2 == 0) ? 16 : 0)) * sizeof(double);
}

template <int NW, int CTP>
__global__ __launch_bounds__(64 * NW) void taylor_reg_kernel(
    int N, int n, int n_terms_k, cplx* __restrict__ walkers, const double* __restrict__ expE,
    const double* __restrict__ vhs, int nv) {
  taylor_reg_body<NW, CTP>(N, n, n_terms_k, walkers, expE, vhs, nv, blockIdx.x);
}

template <int NW, int CTP>
__global__ __launch_bounds__(64 * NW) void taylor_reg_grouped_kernel(
    const TaylorArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const TaylorArgs a = args[p];
  taylor_reg_body<NW, CTP>(a.N, a.n, a.K, a.walkers, static_cast<const double*>(a.E),
                           static_cast<const double*>(a.vhs), a.nv, blockIdx.x - start[p]);
}

template <int NW, int CTP>
int launch_reg(afqmc_ctx* c, int W, int n, cplx* wk, const double* E, const double* V) {
  const int N = c->d.norb;
  if (reg_waves(N) != NW || reg_ct(n) != CTP)
    return afqmc_set_error(AFQMC_ERR_ARG, "taylor f64: %d waves do not fit N %d", NW, N);
  const size_t shm = reg_shm(N, CTP);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)taylor_reg_kernel<NW, CTP>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((taylor_reg_kernel<NW, CTP>), dim3(W), dim3(NW * 64), shm, c->stream, N, n,
                     c->d.n_exp_terms - 1, wk, E, V, c->vhs_nv);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

// ------------------------------------------------------------------------------------
// Split-bf16 register-resident form for the mixed mode (N <= 128, n <= 32).  The complex
// product is one real block product [ur | ui] = [Vr | Vi] [[yr, yi], [-yi, yr]] on
// v_mfma_f32_16x16x32_bf16, with each operand x = hi + lo (bf16 planes) and the three
// leading products al bh + ah bl + ah bh accumulated in float32:
//   A (V rows, registers): lane l holds A[l % 16][8 (l / 16) + e] of each 32-wide k block
//   B (y, LDS [column][k], k contiguous): lane l holds B[8 (l / 16) + e][l % 16]
//   D (float4): lane l, element r holds D[4 (l / 16) + r][l % 16]
// The k axis is packed tightly: with Nh = N rounded up to 4, k in [0, Nh) is the real
// part of V (top half of the y column), k in [Nh, 2 Nh) the imaginary part (bottom half),
// and KB = ceil(2 Nh / 32) k blocks cover it.  A lane's four D rows 4 (l / 16) + r are
// consecutive k of one LDS column, so y goes to LDS as 8-byte stores.
// The one-body factor is applied as E y = y + (E - I) y with E - I in split bf16 (rows of
// Np32 = 32 ceil(N / 32) entries, zero beyond N): its entries are O(dt), so the product's
// relative error stays far below float32 rounding of E y itself.  The Horner recursion
// y <- t0 + V y / k and all additions run in float32; the walker is read and written in
// float64.
// LDS rows (one column of y) are 32 KB + 16 bf16 long, 32 bytes past a multiple of 64,
// and 16-byte chunk j of column c is stored at chunk j ^ ((c >> 2) & 1).  With that, the
// sixteen columns a wave's B operand reads (8 consecutive k each) meet no bank conflict,
// and the D-layout stores of put (4 consecutive k) cost no more than with unswizzled
// rows 16 bytes past a multiple of 32, which conflict on the reads.
template <int KB>
struct BfTile {
  static constexpr int LDK = 32 * KB + 16;  // LDS row (one column of y) in bf16 elements
  static constexpr int KH = (KB + 1) / 2;   // 32-wide k blocks of E - I: ceil(N / 32)
};
inline int bf_ldk(int kb) { return 32 * kb + 16; }  // BfTile<kb>::LDK for a runtime kb
// element offset of k (a multiple of 4) in LDS column c
__device__ inline int bf_koff(int c, int k) { return (((k >> 3) ^ ((c >> 2) & 1)) << 3) | (k & 7); }
// y's real part spans k < Nh, its imaginary part k in [Nh, 2 Nh); Nh = N rounded up to 8
// keeps both halves' 4-row groups in the same chunk halves
__host__ __device__ inline int bf_nh(int N) { return (N + 7) & ~7; }

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

// 8 floats -> hi and lo bf16 planes (4 dwords each)
__device__ inline void split8(const float (&v)[8], u32x4_t& ph, u32x4_t& pl) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t h = pack_bf16x2(v[2 * j], v[2 * j + 1]);
    ph[j] = h;
    pl[j] = pack_bf16x2(v[2 * j] - bf16_lo_val(h), v[2 * j + 1] - bf16_hi_val(h));
  }
}

template <int KB, int CTP>
__device__ __forceinline__ void taylor_bf_body(int N, int n, int n_terms_k,
                                               cplx* __restrict__ walkers,
                                               const uint16_t* __restrict__ emi_hi,
                                               const uint16_t* __restrict__ emi_lo,
                                               const float* __restrict__ vhs, int nv,
                                               const int w) {
  constexpr int LDK = BfTile<KB>::LDK;
  constexpr int KH = BfTile<KB>::KH;
  extern __shared__ uint16_t YB[];  // [2 planes][CTP * 16 columns][LDK]
  uint16_t* Yh = YB;
  uint16_t* Yl = YB + CTP * 16 * LDK;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rb = wave * 16;
  const int np32 = 32 * KH;
  const int Nh = bf_nh(N);
  const int q4 = lane >> 4, col = lane & 15;
  const int q4s = q4 ^ ((col >> 2) & 1);  // this lane's B chunk within a 32-wide k block
  const int p = rb + col;  // A row of this lane
  const bool prow = p < N;
  const bool tail = rb + 16 > N;  // the wave holds rows past N
  const int pc = min(p, N - 1);
  const int n2 = 2 * n;
  cplx* phi = walkers + (int64_t)w * N * n;
  const float* Vr = vhs + (int64_t)w * 2 * nv;
  // V planes hold all N^2 entries row-major, or (nv = N(N+1)/2, symmetric V) the upper
  // triangle row by row: entry (a, b), a <= b, at a N - a (a - 1) / 2 + b - a
  const bool packed = nv != N * N;

  // walker -> registers (D layout), issued first so that its round trip overlaps the V
  // loads'; clamped into the walker and masked after, like the V loads below
  float4_t y[CTP], t0[CTP];
  {
    const double* wz = reinterpret_cast<const double*>(phi);
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rb + 4 * q4 + r;
        const int c = ct * 16 + col;
        const bool ok = (row < N) & (c < n2);
        const int rc = min(row, N - 1);
        const int cc = c < n ? c : min(c - n, n - 1);
        const double z = wz[2 * ((int64_t)rc * n + cc) + (c < n ? 0 : 1)];
        y[ct][r] = ok ? (float)z : 0.f;
      }
  }

  // V rows in registers, split once.  A chunk of 8 k lies in one plane (Nh is a multiple of
  // 8); its entries follow from the first: each 1 further from the diagonal on, N - 1 - k
  // left of it in the packed layout (at most 7 past the row's end, which the VHS buffer's
  // tail padding covers; those past N, and rows past N, are zeroed).  Offsets in bytes to a
  // uniform base: an entry costs five instructions besides its split, against 24, two
  // multiplications and a branch for an index from its row and column, and vector
  // instructions and MFMAs share the SIMD (norb 100, n = 20, 1024 walkers: 72 -> 66 us).
  bf16x8_t vh[KB], vl[KB];
  auto load1 = [&](uint32_t o) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(Vr) + o);
  };
  const uint32_t plane = 4 * (uint32_t)nv;
  const int voff = packed ? pc * N - (pc * (pc - 1)) / 2 : pc * N;  // packed: entry (p, p)
  float v[KB][8];
  auto load_v = [&](auto is_packed) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int k = kb * 32 + 8 * q4;
      const bool im = k >= Nh;
      const int kk = im ? k - Nh : k, kc = min(kk, N - 1);
      uint32_t o = im ? plane : 0;
      if constexpr (is_packed) {
        const int left = kc * N - (kc * (kc - 1)) / 2 + pc - kc;
        o += 4 * (uint32_t)(kc <= pc ? left : voff + kc - pc);
        const int d = 4 * (N - 1 - kc), m = pc - kc;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[kb][e] = load1(o);
          o += m > e ? d - 4 * e : 4;
        }
      } else {
        o += 4 * (uint32_t)(voff + kc);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[kb][e] = load1(o + 4 * e);
      }
    }
  };
  if (packed)
    load_v(std::true_type{});
  else
    load_v(std::false_type{});
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const bool ends = (kb * 32 < Nh && kb * 32 + 32 > N) || kb * 32 + 32 > Nh + N;
    if (tail || ends) {
      const int k = kb * 32 + 8 * q4, kk = k >= Nh ? k - Nh : k;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[kb][e] = prow && kk + e < N ? v[kb][e] : 0.f;
    }
    u32x4_t ph, pl;
    split8(v[kb], ph, pl);
    vh[kb] = __builtin_bit_cast(bf16x8_t, ph);
    vl[kb] = __builtin_bit_cast(bf16x8_t, pl);
  }

  {
    u32x4_t* z = reinterpret_cast<u32x4_t*>(YB);
    const int nz = 2 * CTP * 16 * LDK / 8;
    for (int e = threadIdx.x; e < nz; e += blockDim.x) z[e] = u32x4_t{0u, 0u, 0u, 0u};
  }
  __syncthreads();

  // y (D layout, float32) -> LDS planes: column c < n holds [yr_c ; -yi_c], column n + c
  // holds [yi_c ; yr_c] (top half at k = row, bottom half at k = Nh + row)
  auto put = [&](const float4_t* y) {
    const int row0 = rb + 4 * q4;
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) {
      const int c = ct * 16 + col;
      if (row0 < N && c < n2) {
        const uint32_t h01 = pack_bf16x2(y[ct][0], y[ct][1]);
        const uint32_t h23 = pack_bf16x2(y[ct][2], y[ct][3]);
        const uint32_t l01 = pack_bf16x2(y[ct][0] - bf16_lo_val(h01), y[ct][1] - bf16_hi_val(h01));
        const uint32_t l23 = pack_bf16x2(y[ct][2] - bf16_lo_val(h23), y[ct][3] - bf16_hi_val(h23));
        const int ot = c * LDK + bf_koff(c, row0);
        *reinterpret_cast<u32x2_t*>(Yh + ot) = u32x2_t{h01, h23};
        *reinterpret_cast<u32x2_t*>(Yl + ot) = u32x2_t{l01, l23};
        const int cb = c < n ? c + n : c - n;
        const uint32_t sg = c < n ? 0u : 0x80008000u;  // bottom half: +yr, -yi
        const int ob = cb * LDK + bf_koff(cb, Nh + row0);
        *reinterpret_cast<u32x2_t*>(Yh + ob) = u32x2_t{h01 ^ sg, h23 ^ sg};
        *reinterpret_cast<u32x2_t*>(Yl + ob) = u32x2_t{l01 ^ sg, l23 ^ sg};
      }
    }
  };
  auto bload = [&](const uint16_t* plane, int ct, int kb) {
    return __builtin_bit_cast(
        bf16x8_t, *reinterpret_cast<const u32x4_t*>(plane + (ct * 16 + col) * LDK + kb * 32 + 8 * q4s));
  };
  // acc = (E - I) y: A (rows of E - I) streams from L2; k < Np32 reads the top half of
  // each column and, past Nh, bottom-half entries that meet zero columns of E - I
  auto e_product = [&](float4_t* acc) {
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) acc[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    const uint16_t* eh = emi_hi + pc * np32 + 8 * q4;
    const uint16_t* el = emi_lo + pc * np32 + 8 * q4;
    u32x4_t nh = *reinterpret_cast<const u32x4_t*>(eh), nl = *reinterpret_cast<const u32x4_t*>(el);
#pragma unroll
    for (int kb = 0; kb < KH; ++kb) {
      u32x4_t ah = nh, al = nl;
      if (kb + 1 < KH) {
        nh = *reinterpret_cast<const u32x4_t*>(eh + 32 * (kb + 1));
        nl = *reinterpret_cast<const u32x4_t*>(el + 32 * (kb + 1));
      }
      if (tail && !prow) ah = al = u32x4_t{0, 0, 0, 0};
      const bf16x8_t a_h = __builtin_bit_cast(bf16x8_t, ah), a_l = __builtin_bit_cast(bf16x8_t, al);
#pragma unroll
      for (int ct = 0; ct < CTP; ++ct) {
        const bf16x8_t bh = bload(Yh, ct, kb), bl = bload(Yl, ct, kb);
        acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_l, bh, acc[ct], 0, 0, 0);
        acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_h, bl, acc[ct], 0, 0, 0);
        acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_h, bh, acc[ct], 0, 0, 0);
      }
    }
  };

  put(y);
  __syncthreads();
  e_product(t0);
#pragma unroll
  for (int ct = 0; ct < CTP; ++ct) t0[ct] += y[ct];
  __syncthreads();
  put(t0);
  __syncthreads();
  for (int k = n_terms_k; k >= 1; --k) {
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) y[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int ct = 0; ct < CTP; ++ct) {
        const bf16x8_t bh = bload(Yh, ct, kb), bl = bload(Yl, ct, kb);
        y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vl[kb], bh, y[ct], 0, 0, 0);
        y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[kb], bl, y[ct], 0, 0, 0);
        y[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[kb], bh, y[ct], 0, 0, 0);
      }
    }
    __syncthreads();
    const float rk = 1.0f / (float)k;
#pragma unroll
    for (int ct = 0; ct < CTP; ++ct) y[ct] = t0[ct] + y[ct] * rk;
    put(y);
    __syncthreads();
  }
  float4_t acc[CTP];
  e_product(acc);
#pragma unroll
  for (int ct = 0; ct < CTP; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = rb + 4 * q4 + r;
      const int c = ct * 16 + col;
      if (row < N && c < n2) {
        double* dst = reinterpret_cast<double*>(phi + (int64_t)row * n + (c < n ? c : c - n));
        dst[c < n ? 0 : 1] = (double)(y[ct][r] + acc[ct][r]);
      }
    }
}

// Two 7- or 8-wave workgroups per CU need at most 128 VGPRs (4 waves per SIMD); the
// widest tiles (n > 24 with N > 96) would spill inside the series at that budget.
constexpr int bf_waves_per_simd(int KB, int CTP) { return (CTP == 4 && KB >= 7) ? 3 : 4; }

template <int KB, int CTP>
__global__ __launch_bounds__(512, bf_waves_per_simd(KB, CTP)) void taylor_bf_kernel(int N, int n, int n_terms_k,
                                                           cplx* __restrict__ walkers,
                                                           const uint16_t* __restrict__ emi_hi,
                                                           const uint16_t* __restrict__ emi_lo,
                                                           const float* __restrict__ vhs,
                                                           int nv) {
  taylor_bf_body<KB, CTP>(N, n, n_terms_k, walkers, emi_hi, emi_lo, vhs, nv, blockIdx.x);
}

template <int KB, int CTP>
__global__ __launch_bounds__(512, bf_waves_per_simd(KB, CTP)) void taylor_bf_grouped_kernel(
    const TaylorArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int pidx = group_of(start, nprob, blockIdx.x);
  const TaylorArgs a = args[pidx];
  taylor_bf_body<KB, CTP>(a.N, a.n, a.K, a.walkers, static_cast<const uint16_t*>(a.E),
                          static_cast<const uint16_t*>(a.E2), static_cast<const float*>(a.vhs),
                          a.nv, blockIdx.x - start[pidx]);
}

// k blocks of the packed [Vr | Vi] axis
inline int bf_kblocks(int N) { return (2 * bf_nh(N) + 31) / 32; }
// threads of a register-form workgroup: a wave per 16 rows, with 6 or 7 waves rounded up
// to 8 (the extra waves own rows >= N: zero work, but every SIMD then holds two waves of
// the group at its barriers, and at four waves per SIMD two such groups fill a CU either
// way); 5 waves stay 5, which lets three groups share a CU
inline int bf_threads(int N) {
  const int w = (N + 15) / 16;
  return 64 * ((w == 6 || w == 7) ? 8 : w);
}

template <int KB, int CTP>
int launch_bf(afqmc_ctx* c, int W, int n, cplx* wk, int s) {
  const int N = c->d.norb;
  if (BfTile<KB>::KH * 32 != c->Np32 || bf_kblocks(N) != KB)
    return afqmc_set_error(AFQMC_ERR_ARG, "taylor bf16x3: k blocks %d do not fit N %d", KB, N);
  const size_t shm = (size_t)2 * CTP * 16 * BfTile<KB>::LDK * sizeof(uint16_t);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)taylor_bf_kernel<KB, CTP>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((taylor_bf_kernel<KB, CTP>), dim3(W), dim3(bf_threads(N)), shm, c->stream, N,
                     n, c->d.n_exp_terms - 1, wk, c->emi_bf[s][0], c->emi_bf[s][1],
                     vhs_f32_of(c, s), c->vhs_nv);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int KB>
int launch_bf_ct(afqmc_ctx* c, int W, int n, cplx* wk, int s) {
  switch ((2 * n + 15) / 16) {
    case 1: return launch_bf<KB, 1>(c, W, n, wk, s);
    case 2: return launch_bf<KB, 2>(c, W, n, wk, s);
    case 3: return launch_bf<KB, 3>(c, W, n, wk, s);
    default: return launch_bf<KB, 4>(c, W, n, wk, s);
  }
}

// ------------------------------------------------------------------------------------
// Split-bf16 streaming form for the mixed mode beyond the register kernel's range
// (N <= 256, n <= 64).  One workgroup per walker of one spin; wave r owns output rows
// [16 r, 16 r + 16) and every column.  y = [yr | yi] (N x 2 n, each half padded to 16 CT
// columns) lives in LDS as hi / lo bf16 planes stored [column][k] with k contiguous, so a
// lane's B operand (8 consecutive k of one column) is one 16-byte read; k is padded with
// zeros to 32 ceil(N / 32).  V streams from global memory as float32 rows, 32 k at a time
// with the next block in flight while the current one multiplies, and is split into bf16
// planes in registers.  The complex product is four real products,
//   ur = Vr yr - Vi yi,  ui = Vr yi + Vi yr,
// each as three bf16 products (al bh + ah bl + ah bh) on v_mfma_f32_16x16x32_bf16 with
// float32 accumulation; the planes of -Vi are those of Vi with the sign bits flipped
// (round-to-nearest-even is symmetric).  E y = y + (E - I) y uses the split planes of
// E - I (rows of 32 ceil(N / 32) entries) as the register form does, and the Horner
// recursion y <- t0 + V y / k runs in float32 registers.
//
// What it is shaped by: LDS holds one workgroup of up to 16 waves per CU, so a wave has 128
// registers and little else to hide its loads.  The next block's loads must not be touched
// before its split (a select or copy of a loaded value waits for it in the step that
// asked for it), and nothing may spill: constant LDS strides, byte offsets to uniform bases,
// and blocks of one kind per branch.  Masked loads, copied at once, with 25 to 48 registers
// spilled: 2.00 ms for both spins at norb 200, n = 40, 2048 walkers; now 1.50.
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));  // dword-aligned rows

// LDS columns of y: k padded to 32 ceil(N / 32), a stride fixed for N up to 128 or 256 so
// that every operand's place is an immediate offset
constexpr int bfs_ldk(bool small) { return small ? 144 : 272; }
inline bool bfs_small(int N, int ct) { return N <= 128 && ct >= 3; }  // (else N > 128)
inline size_t bfs_shm(int N, int ct) {
  return (size_t)2 * 32 * ct * bfs_ldk(bfs_small(N, ct)) * sizeof(uint16_t);
}
inline int bfs_threads(int N) { return 64 * ((N + 15) / 16); }

template <int CT, bool SMALL>
__device__ __forceinline__ void taylor_bfs_body(int N, int n, int n_terms_k,
                                                cplx* __restrict__ walkers,
                                                const uint16_t* __restrict__ emi_hi,
                                                const uint16_t* __restrict__ emi_lo,
                                                const float* __restrict__ vhs, int nv,
                                                const int w) {
  constexpr int NC = 32 * CT;  // LDS columns: CT tiles of yr, then CT tiles of yi
  constexpr int LDK = bfs_ldk(SMALL);  // rows and chunk swizzle as in the register form
  const int KBk = (N + 31) >> 5;
  const int np32 = 32 * KBk;
  extern __shared__ uint16_t YB[];  // [2 planes][NC][LDK]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rb = wave * 16;
  const int q4 = lane >> 4, col = lane & 15;
  const int sw = (col >> 2) & 1;  // chunk swizzle of this lane's LDS columns
  cplx* phi = walkers + (int64_t)w * N * n;
  // V planes: all N^2 entries row-major, or (nv = N(N+1)/2, symmetric V) the upper
  // triangle row by row, entry (a, b), a <= b, at a N - a (a - 1) / 2 + b - a
  const bool packed = nv != N * N;
  const float* Vr = vhs + (int64_t)w * 2 * nv;
  const float* Vi = Vr + nv;
  const int p = min(rb + col, N - 1);  // A row of this lane
  const bool prow = rb + col < N;
  const bool tail = rb + 16 > N;  // the wave holds rows past N: zeros
  // start of row p (packed: of its upper part, entry (p, p))
  const int voff = packed ? p * N - (p * (p - 1)) / 2 : p * N;

  {
    u32x4_t* z = reinterpret_cast<u32x4_t*>(YB);
    const int nz = 2 * NC * LDK / 8;
    for (int e = threadIdx.x; e < nz; e += blockDim.x) z[e] = u32x4_t{0u, 0u, 0u, 0u};
  }

  // walker (float64) -> float32 D layout, the loads all in flight
  float4_t t0r[CT], t0i[CT], ur[CT], ui[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    cplx z[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      z[r] = phi[min(rb + 4 * q4 + r, N - 1) * n + min(ct * 16 + col, n - 1)];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool ok = rb + 4 * q4 + r < N && ct * 16 + col < n;
      t0r[ct][r] = ok ? (float)z[r].re : 0.f;
      t0i[ct][r] = ok ? (float)z[r].im : 0.f;
    }
  }
  __syncthreads();

  // D layout (rows 4 (l / 16) + r of a tile, column l % 16) -> LDS planes: four
  // consecutive k of one column, 8-byte stores.  Rows >= N and columns >= n carry zeros
  // (their A rows / B columns are zero), which keeps the padding zero.
  uint16_t* yput = YB + col * LDK + rb + 8 * ((q4 >> 1) ^ sw) + 4 * (q4 & 1);
  auto put = [&](const float4_t (&yr)[CT], const float4_t (&yi)[CT]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const float4_t v = h ? yi[ct] : yr[ct];
        const int off = (h * 16 * CT + ct * 16) * LDK;
        const uint32_t h01 = pack_bf16x2(v[0], v[1]);
        const uint32_t h23 = pack_bf16x2(v[2], v[3]);
        const uint32_t l01 = pack_bf16x2(v[0] - bf16_lo_val(h01), v[1] - bf16_hi_val(h01));
        const uint32_t l23 = pack_bf16x2(v[2] - bf16_lo_val(h23), v[3] - bf16_hi_val(h23));
        *reinterpret_cast<u32x2_t*>(yput + off) = u32x2_t{h01, h23};
        *reinterpret_cast<u32x2_t*>(yput + NC * LDK + off) = u32x2_t{l01, l23};
      }
  };
  // B operand: 8 consecutive k of column 16 c + col (c: CT tiles of yr, then of yi)
  const uint16_t* yget = YB + col * LDK + 8 * (q4 ^ sw);
  auto bload = [&](const uint16_t* yk, int plane, int c) {
    return __builtin_bit_cast(
        bf16x8_t, *reinterpret_cast<const u32x4_t*>(yk + (plane * NC + 16 * c) * LDK));
  };
  auto bf = [](const u32x4_t& x) { return __builtin_bit_cast(bf16x8_t, x); };
  // acc = (E - I) y, a real operator on both halves; the next block's E in flight
  auto e_product = [&](float4_t (&ar)[CT], float4_t (&ai)[CT]) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) ar[ct] = ai[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    const uint16_t* eh = emi_hi + p * np32 + 8 * q4;
    const uint16_t* el = emi_lo + p * np32 + 8 * q4;
    u32x4_t nh = *reinterpret_cast<const u32x4_t*>(eh), nl = *reinterpret_cast<const u32x4_t*>(el);
    const uint16_t* yk = yget;
#pragma unroll 1
    for (int kb = 0; kb < KBk; ++kb, yk += 32) {
      u32x4_t ah = nh, al = nl;
      const int kn = kb + 1 < KBk ? 32 * (kb + 1) : 0;
      nh = *reinterpret_cast<const u32x4_t*>(eh + kn);
      nl = *reinterpret_cast<const u32x4_t*>(el + kn);
      if (tail && !prow) ah = al = u32x4_t{0, 0, 0, 0};
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const bf16x8_t rh = bload(yk, 0, ct), rl = bload(yk, 1, ct);
        ar[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(al), rh, ar[ct], 0, 0, 0);
        ar[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ah), rl, ar[ct], 0, 0, 0);
        ar[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ah), rh, ar[ct], 0, 0, 0);
        const bf16x8_t ih = bload(yk, 0, CT + ct), il = bload(yk, 1, CT + ct);
        ai[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(al), ih, ai[ct], 0, 0, 0);
        ai[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ah), il, ai[ct], 0, 0, 0);
        ai[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ah), ih, ai[ct], 0, 0, 0);
      }
    }
  };
  // 8 consecutive k of the lane's V row (those past N, or of a row past N, are zeroed at the
  // split).  Right of the diagonal, or in whole rows, a chunk is contiguous: two 16-byte loads
  // (one that straddles k = N reads at most 7 floats past the row end, into the next row or,
  // for the last row of the last walker, into the 8 floats of tail padding of the VHS
  // buffer).  Left of the diagonal of the packed layout it is the entries (k, p) of rows
  // k < p, each N - 1 - k after the last; for a fixed k the 16 rows of a lane group are
  // consecutive floats of one stored row.  Which of the two a block is holds for the whole
  // wave but for the one or two blocks on the diagonal, so the branches are scalar and the
  // loads unconditional, from clamped k.
  struct Vops {
    f4u_t r0, r1, i0, i1;
  };
  auto load1 = [](const float* base, uint32_t o) {  // uniform base, byte offset
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + o);
  };
  auto load4 = [](const float* base, uint32_t o) {
    return *reinterpret_cast<const f4u_t*>(reinterpret_cast<const char*>(base) + o);
  };
  auto vload = [&](int kb, Vops& v) {
    const int k0 = kb * 32 + 8 * q4;
    if (!packed || 32 * kb >= rb + 15) {
      // (chunks past N: the row's first one)
      const uint32_t o = 4 * (voff + (k0 < N ? (packed ? k0 - p : k0) : 0));
      v.r0 = load4(Vr, o);
      v.r1 = load4(Vr, o + 16);
      v.i0 = load4(Vi, o);
      v.i1 = load4(Vi, o + 16);
    } else if (32 * kb + 31 <= rb) {
      uint32_t x = 4 * (k0 * N - (k0 * (k0 - 1)) / 2 + p - k0);  // entry (k0, p)
      uint32_t d = 4 * (N - 1 - k0);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (e < 4) {
          v.r0[e & 3] = load1(Vr, x);
          v.i0[e & 3] = load1(Vi, x);
        } else {
          v.r1[e & 3] = load1(Vr, x);
          v.i1[e & 3] = load1(Vi, x);
        }
        x += d;
        d -= 4;
      }
    } else {
      const int kc = min(k0, N - 1);
      uint32_t x = 4 * (kc * N - (kc * (kc - 1)) / 2 + p - kc);  // entry (k, p), for k <= p
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = min(k0 + e, N - 1);
        const uint32_t o = k <= p ? x : 4 * (uint32_t)(voff + (k - p));
        if (e < 4) {
          v.r0[e & 3] = load1(Vr, o);
          v.i0[e & 3] = load1(Vi, o);
        } else {
          v.r1[e & 3] = load1(Vr, o);
          v.i1[e & 3] = load1(Vi, o);
        }
        x += 4 * (N - 1 - k);
      }
    }
  };
  auto v_product = [&]() {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) ur[ct] = ui[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    Vops v;
    int first = 0;  // (opaque: the block's 16 addresses would be kept, spilled, across the terms)
    asm volatile("" : "+s"(first));
    vload(first, v);
    const uint16_t* yk = yget;
#pragma unroll 1
    for (int kb = 0; kb < KBk; ++kb, yk += 32) {
      u32x4_t rh, rl, ih, il;
      {
        float r[8], i[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          r[e] = v.r0[e];
          r[4 + e] = v.r1[e];
          i[e] = v.i0[e];
          i[4 + e] = v.i1[e];
        }
        if (tail || 32 * kb + 32 > N) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (!prow || kb * 32 + 8 * q4 + e >= N) r[e] = i[e] = 0.f;
        }
        split8(r, rh, rl);
        split8(i, ih, il);
      }
      if (kb + 1 < KBk) vload(kb + 1, v);  // next block in flight
      // rows of yr: ur += Vr yr, ui += Vi yr
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const bf16x8_t yh = bload(yk, 0, ct), yl = bload(yk, 1, ct);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rl), yh, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(il), yh, ui[ct], 0, 0, 0);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rh), yl, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ih), yl, ui[ct], 0, 0, 0);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rh), yh, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ih), yh, ui[ct], 0, 0, 0);
      }
      // rows of yi: ur += (-Vi) yi, ui += Vr yi (Vi's planes negated in place)
      const u32x4_t sg = {0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
      ih ^= sg;
      il ^= sg;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const bf16x8_t yh = bload(yk, 0, CT + ct), yl = bload(yk, 1, CT + ct);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(il), yh, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rl), yh, ui[ct], 0, 0, 0);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ih), yl, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rh), yl, ui[ct], 0, 0, 0);
        ur[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(ih), yh, ur[ct], 0, 0, 0);
        ui[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf(rh), yh, ui[ct], 0, 0, 0);
      }
    }
  };

  put(t0r, t0i);
  __syncthreads();
  e_product(ur, ui);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    t0r[ct] += ur[ct];
    t0i[ct] += ui[ct];
  }
  __syncthreads();
  put(t0r, t0i);
  __syncthreads();
#pragma unroll 1
  for (int k = n_terms_k; k >= 1; --k) {
    v_product();
    __syncthreads();
    const float rk = 1.0f / (float)k;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      ur[ct] = t0r[ct] + ur[ct] * rk;
      ui[ct] = t0i[ct] + ui[ct] * rk;
    }
    put(ur, ui);
    __syncthreads();
  }
  e_product(t0r, t0i);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = rb + 4 * q4 + r;
      const int c = ct * 16 + col;
      if (row < N && c < n)
        phi[row * n + c] =
            cplx{(double)(ur[ct][r] + t0r[ct][r]), (double)(ui[ct][r] + t0i[ct][r])};
    }
}

template <int CT, bool SMALL>
__global__ __launch_bounds__(SMALL ? 512 : 1024, 4) void taylor_bfs_kernel(
    int N, int n, int n_terms_k, cplx* __restrict__ walkers, const uint16_t* __restrict__ emi_hi,
    const uint16_t* __restrict__ emi_lo, const float* __restrict__ vhs, int nv) {
  taylor_bfs_body<CT, SMALL>(N, n, n_terms_k, walkers, emi_hi, emi_lo, vhs, nv,
                                  blockIdx.x);
}

template <int CT, bool SMALL>
__global__ __launch_bounds__(SMALL ? 512 : 1024, 4) void taylor_bfs_grouped_kernel(
    const TaylorArgs* __restrict__ args, const int* __restrict__ start, int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const TaylorArgs a = args[p];
  taylor_bfs_body<CT, SMALL>(
      a.N, a.n, a.K, a.walkers, static_cast<const uint16_t*>(a.E),
      static_cast<const uint16_t*>(a.E2), static_cast<const float*>(a.vhs), a.nv,
      blockIdx.x - start[p]);
}

// Both spins of an unrestricted walker set that share one V (spin-summed Cholesky
// vectors) in one launch.  Block b = 16 q + 8 s + r takes spin s of walker 8 q + r:
// blocks are dealt round-robin to the 8 XCDs (block b on XCD b % 8), so the two blocks
// of a walker run on the same XCD, one dispatch round apart, and the second one's V
// rows mostly come from that XCD's L2 instead of HBM.
template <int CT, bool SMALL>
__global__ __launch_bounds__(SMALL ? 512 : 1024, 4) void taylor_bfs_spins_kernel(
    int N, int n0, int n1, int n_terms_k, int W, cplx* __restrict__ w0, cplx* __restrict__ w1,
    const uint16_t* __restrict__ e0h, const uint16_t* __restrict__ e0l,
    const uint16_t* __restrict__ e1h, const uint16_t* __restrict__ e1l,
    const float* __restrict__ vhs, int nv) {
  const int b = blockIdx.x;
  const int s = (b >> 3) & 1, w = 8 * (b >> 4) + (b & 7);
  if (w >= W) return;  // (whole workgroup: the tail of the last group of 8 walkers)
  taylor_bfs_body<CT, SMALL>(N, s ? n1 : n0, n_terms_k, s ? w1 : w0, s ? e1h : e0h,
                                  s ? e1l : e0l, vhs, nv, w);
}

template <int CT, bool SMALL>
int launch_bfs_spins(afqmc_ctx* c, int W, cplx* wup, cplx* wdn) {
  const int N = c->d.norb;
  if (N > 256 || c->nocc[0] > 16 * CT || c->nocc[1] > 16 * CT || 32 * ((N + 31) / 32) != c->Np32)
    return afqmc_set_error(AFQMC_ERR_ARG, "taylor bf16x3 streaming: N %d column tiles %d", N, CT);
  const size_t shm = bfs_shm(N, CT);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)taylor_bfs_spins_kernel<CT, SMALL>, shm, &lds_limit);
  if (rc) return rc;
  const int groups = (W + 7) / 8;
  hipLaunchKernelGGL((taylor_bfs_spins_kernel<CT, SMALL>), dim3(16 * groups), dim3(bfs_threads(N)),
                     shm, c->stream, N, c->nocc[0], c->nocc[1], c->d.n_exp_terms - 1, W, wup,
                     wdn, c->emi_bf[0][0], c->emi_bf[0][1], c->emi_bf[1][0], c->emi_bf[1][1],
                     vhs_f32_of(c, 0), c->vhs_nv);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int CT, bool SMALL>
int launch_bfs(afqmc_ctx* c, int W, int n, cplx* wk, int s) {
  const int N = c->d.norb;
  if (N > 256 || n > 16 * CT || 32 * ((N + 31) / 32) != c->Np32)
    return afqmc_set_error(AFQMC_ERR_ARG, "taylor bf16x3 streaming: N %d n %d column tiles %d",
                           N, n, CT);
  const size_t shm = bfs_shm(N, CT);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)taylor_bfs_kernel<CT, SMALL>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((taylor_bfs_kernel<CT, SMALL>), dim3(W), dim3(bfs_threads(N)), shm, c->stream,
                     N, n, c->d.n_exp_terms - 1, wk, c->emi_bf[s][0], c->emi_bf[s][1],
                     vhs_f32_of(c, s), c->vhs_nv);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int NW>
int launch_reg_ct(afqmc_ctx* c, int W, int n, cplx* wk, const double* E, const double* V) {
  switch (reg_ct(n)) {
    case 1: return launch_reg<NW, 1>(c, W, n, wk, E, V);
    case 2: return launch_reg<NW, 2>(c, W, n, wk, E, V);
    case 3: return launch_reg<NW, 3>(c, W, n, wk, E, V);
    default: return launch_reg<NW, 4>(c, W, n, wk, E, V);
  }
}

}  // namespace

// The kernel launch_taylor picks for spin s, as a plan for grouped launches.
void taylor_plan(const afqmc_ctx* c, int s, TaylorPlan* pl) {
  const int N = c->d.norb, n = c->nocc[s];
  const int ctp = (2 * n + 15) / 16 > 4 ? 4 : (2 * n + 15) / 16;
  pl->nthreads = ((N + 15) / 16) * 64;
  pl->nblocks = c->d.n_walkers;
  pl->nkgv = 0;
  pl->ct = 0;
  if (c->taylor_bf) {
    if (N <= 128 && n <= 32) {
      const int kb = bf_kblocks(N);
      pl->kind = TAYLOR_REG_BF16X3;
      pl->nthreads = bf_threads(N);
      pl->nkgv = kb;
      pl->ct = ctp;
      pl->shm = (size_t)2 * ctp * 16 * bf_ldk(kb) * sizeof(uint16_t);
    } else {  // N <= AFQMC_MAX_NORB = 256, n <= AFQMC_MAX_NOCC = 64
      pl->kind = TAYLOR_STREAM_BF16X3;
      const int ct = (n + 15) / 16;
      pl->ct = ct + (bfs_small(N, ct) ? 4 : 0);
      pl->nthreads = bfs_threads(N);
      pl->shm = bfs_shm(N, ct);
    }
  } else if (N <= 128 && c->nocc[0] <= 32 && c->nocc[1] <= 32) {
    pl->kind = TAYLOR_REG_F64;
    pl->nkgv = reg_waves(N);
    pl->ct = ctp;
    pl->shm = reg_shm(N, ctp);
  } else {
    pl->kind = TAYLOR_STREAM_F64;
    pl->nblocks = stream_blocks(c->d.n_walkers, stream_chunks(n));
    pl->shm = stream_shm(N);
  }
}

int launch_taylor(afqmc_ctx* c, int W, cplx* wup, cplx* wdn) {
  const int N = c->d.norb;
  if (c->taylor_bf && c->nspin == 2 && vhs_f32_of(c, 0) == vhs_f32_of(c, 1) &&
      !(N <= 128 && c->nocc[0] <= 32) && !(N <= 128 && c->nocc[1] <= 32) &&
      (c->nocc[0] + 15) / 16 == (c->nocc[1] + 15) / 16) {
    // both spins streaming with one shared V: one launch, the spins of a walker side by side
    switch ((c->nocc[0] + 15) / 16) {
      case 1: return launch_bfs_spins<1, false>(c, W, wup, wdn);
      case 2: return launch_bfs_spins<2, false>(c, W, wup, wdn);
      case 3:
        return N <= 128 ? launch_bfs_spins<3, true>(c, W, wup, wdn)
                        : launch_bfs_spins<3, false>(c, W, wup, wdn);
      default:
        return N <= 128 ? launch_bfs_spins<4, true>(c, W, wup, wdn)
                        : launch_bfs_spins<4, false>(c, W, wup, wdn);
    }
  }
  if (c->taylor_bf) {
    for (int s = 0; s < c->nspin; ++s) {
      const int n = c->nocc[s];
      cplx* wk = (s == 0) ? wup : wdn;
      int rc;
      if (N <= 128 && n <= 32) {
        switch (bf_kblocks(N)) {
          case 1: rc = launch_bf_ct<1>(c, W, n, wk, s); break;
          case 2: rc = launch_bf_ct<2>(c, W, n, wk, s); break;
          case 3: rc = launch_bf_ct<3>(c, W, n, wk, s); break;
          case 4: rc = launch_bf_ct<4>(c, W, n, wk, s); break;
          case 5: rc = launch_bf_ct<5>(c, W, n, wk, s); break;
          case 6: rc = launch_bf_ct<6>(c, W, n, wk, s); break;
          case 7: rc = launch_bf_ct<7>(c, W, n, wk, s); break;
          default: rc = launch_bf_ct<8>(c, W, n, wk, s); break;
        }
      } else {
        switch ((n + 15) / 16) {
          case 1: rc = launch_bfs<1, false>(c, W, n, wk, s); break;
          case 2: rc = launch_bfs<2, false>(c, W, n, wk, s); break;
          case 3:
            rc = N <= 128 ? launch_bfs<3, true>(c, W, n, wk, s)
                          : launch_bfs<3, false>(c, W, n, wk, s);
            break;
          default:
            rc = N <= 128 ? launch_bfs<4, true>(c, W, n, wk, s)
                          : launch_bfs<4, false>(c, W, n, wk, s);
            break;
        }
      }
      if (rc) return rc;
    }
    return AFQMC_OK;
  }
  if (N <= 128 && c->nocc[0] <= 32 && c->nocc[1] <= 32) {
    for (int s = 0; s < c->nspin; ++s) {
      const int n = c->nocc[s];
      cplx* wk = (s == 0) ? wup : wdn;
      const double *E = c->exp_h1[s], *V = vhs_of(c, s);
      int rc;
      switch (reg_waves(N)) {
        case 1: rc = launch_reg_ct<1>(c, W, n, wk, E, V); break;
        case 2: rc = launch_reg_ct<2>(c, W, n, wk, E, V); break;
        case 3: rc = launch_reg_ct<3>(c, W, n, wk, E, V); break;
        case 4: rc = launch_reg_ct<4>(c, W, n, wk, E, V); break;
        case 5: rc = launch_reg_ct<5>(c, W, n, wk, E, V); break;
        case 6: rc = launch_reg_ct<6>(c, W, n, wk, E, V); break;
        case 7: rc = launch_reg_ct<7>(c, W, n, wk, E, V); break;
        default: rc = launch_reg_ct<8>(c, W, n, wk, E, V); break;
      }
      if (rc) return rc;
    }
    return AFQMC_OK;
  }
  return (N + 15) / 16 <= STREAM_SMALL ? launch_stream<true>(c, W, wup, wdn)
                                       : launch_stream<false>(c, W, wup, wdn);
}

namespace {

template <typename KernelFn>
int launch_grouped_fn(KernelFn fn, hipStream_t st, const TaylorArgs* args, const int* start,
                      int nprob, int nblocks, int nthreads, size_t shm, int* lds_limit) {
  const int rc = ensure_dyn_lds((const void*)fn, shm, lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL(fn, dim3(nblocks), dim3(nthreads), shm, st, args, start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int NW>
int reg_grouped(int ct, hipStream_t st, const TaylorArgs* args, const int* start, int nprob,
                int nblocks, int nthreads, size_t shm) {
  static int lim[4] = {};
  const int ci = ct < 1 ? 0 : (ct > 4 ? 3 : ct - 1);
  switch (ct) {
    case 1: return launch_grouped_fn(taylor_reg_grouped_kernel<NW, 1>, st, args, start, nprob, nblocks, nthreads, shm, &lim[ci]);
    case 2: return launch_grouped_fn(taylor_reg_grouped_kernel<NW, 2>, st, args, start, nprob, nblocks, nthreads, shm, &lim[ci]);
    case 3: return launch_grouped_fn(taylor_reg_grouped_kernel<NW, 3>, st, args, start, nprob, nblocks, nthreads, shm, &lim[ci]);
    case 4: return launch_grouped_fn(taylor_reg_grouped_kernel<NW, 4>, st, args, start, nprob, nblocks, nthreads, shm, &lim[ci]);
  }
  return afqmc_set_error(AFQMC_ERR_ARG, "grouped taylor: column tiles %d", ct);
}

}  // namespace

// Grouped Taylor launch for problems of one kernel kind and template key (nkgv, column
// tiles ct) and one block size nthreads = 64 * ceil(N / 16).
int launch_taylor_grouped(hipStream_t st, int kind, int nkgv, int ct, const TaylorArgs* args,
                          const int* start, int nprob, int nblocks, int nthreads, size_t shm) {
  if (kind == TAYLOR_REG_F64) {
    switch (nkgv) {
      case 1: return reg_grouped<1>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 2: return reg_grouped<2>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 3: return reg_grouped<3>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 4: return reg_grouped<4>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 5: return reg_grouped<5>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 6: return reg_grouped<6>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 7: return reg_grouped<7>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      case 8: return reg_grouped<8>(ct, st, args, start, nprob, nblocks, nthreads, shm);
      default: return afqmc_set_error(AFQMC_ERR_ARG, "grouped taylor: %d waves", nkgv);
    }
  }
  if (kind == TAYLOR_REG_BF16X3) {
    static int lim[8][4] = {};
    const int ci = ct < 1 ? 0 : (ct > 4 ? 3 : ct - 1);
#define BF_CASE(KB, C)                                                                      \
  if (nkgv == KB && ct == C)                                                                \
    return launch_grouped_fn(taylor_bf_grouped_kernel<KB, C>, st, args, start, nprob, nblocks, \
                             nthreads, shm, &lim[KB - 1][ci]);
#define BF_CASES(KB) BF_CASE(KB, 1) BF_CASE(KB, 2) BF_CASE(KB, 3) BF_CASE(KB, 4)
    BF_CASES(1) BF_CASES(2) BF_CASES(3) BF_CASES(4)
    BF_CASES(5) BF_CASES(6) BF_CASES(7) BF_CASES(8)
#undef BF_CASES
#undef BF_CASE
    return afqmc_set_error(AFQMC_ERR_ARG, "grouped taylor: k blocks %d, column tiles %d", nkgv, ct);
  }
  if (kind == TAYLOR_STREAM_BF16X3) {
    static int lim[6] = {};
#define BFS_CASE(CASE, C, SMALL, I)                                                            \
  case CASE:                                                                                   \
    return launch_grouped_fn(taylor_bfs_grouped_kernel<C, SMALL>, st, args, start, nprob,      \
                             nblocks, nthreads, shm, &lim[I]);
    switch (ct) {
      BFS_CASE(1, 1, false, 0) BFS_CASE(2, 2, false, 1) BFS_CASE(3, 3, false, 2)
      BFS_CASE(4, 4, false, 3) BFS_CASE(7, 3, true, 4) BFS_CASE(8, 4, true, 5)
      default: return afqmc_set_error(AFQMC_ERR_ARG, "grouped taylor: column tiles %d", ct);
    }
#undef BFS_CASE
  }
  static int lim64[2] = {};
  if (nthreads <= 64 * STREAM_SMALL)
    return launch_grouped_fn(taylor_stream_grouped_kernel<true>, st, args, start, nprob, nblocks,
                             nthreads, shm, &lim64[0]);
  return launch_grouped_fn(taylor_stream_grouped_kernel<false>, st, args, start, nprob, nblocks,
                           nthreads, shm, &lim64[1]);
}
