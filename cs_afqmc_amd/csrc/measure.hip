// Trial measurements per walker and spin: O = C^T w (n x n), O^-1 and det(O) by a blocked
// in-place Gauss-Jordan inversion with partial pivoting (pivot: the largest |re| + |im|
// over the remaining rows, LAPACK's izamax measure), and the half-rotated Green's
// function G = (w O^-1)^T (n x N).
//
// Follows rhf._calc_overlap_restricted / _calc_green (wavefunctions.py:478-501) and
// uhf._calc_overlap / _calc_green (wavefunctions.py:658-692).  The trial C is real.
//
// One workgroup per (walker, spin): two waves for n <= 24, four beyond.  The overlap and
// Green products run on v_mfma_f64_16x16x4f64 in real block form:
//   [Or | Oi]  = C^T [wr | wi]                         (n x 2n,  K = N)
//   [Gr ; Gi]  = [[Xr^T, -Xi^T], [Xi^T, Xr^T]] [wr^T ; wi^T]   (2n x N, K = 2n)
// The second product's rows are exactly the rows of the split Green layout
// green[w][c][i][p] (c = re / im), so results go straight to global memory.
//
// Inversion: O is overwritten in LDS (n x n complex) by a blocked in-place Gauss-Jordan
// elimination with implicit pivoting (rows stay in place), in panels of GJ_PB = 4 pivot
// columns.  The wave that owns a panel's 16-column block factors it with a lane per row
// (pivot search by a wave reduction, the panel's other columns updated in registers); the
// panel columns then hold the panel's transform, and every other column is updated by a
// complex rank-4 product on MFMA (four real MFMAs per 16 x 16 tile), each wave over its
// own column block.  With r_k the pivot row of column k, O^-1[i][j] = S[r_i][r^-1(j)] for
// the stored S; the Green product reads X through these two maps.
#include <algorithm>

#include "common.h"


namespace {

constexpr int MEAS_KC = 4;  // k-groups whose operands are loaded ahead of their MFMAs

constexpr int GJ_PB = 4;  // panel width: the K of one f64 MFMA

// LDS of the inversion: B (n x ld complex), then the state below (256 ints)
__host__ __device__ constexpr int gj_ld(int n) { return n | 1; }
__host__ __device__ constexpr size_t gj_bytes(int n) {
  return (size_t)n * gj_ld(n) * sizeof(cplx) + 256 * sizeof(int);
}
struct GjState {
  int rho[64];     // rho[k]: the pivot row of column k
  int rhoinv[64];  // its inverse (filled at the end)
  int vrow[64];    // row order of the equivalent row-exchanging elimination (for the sign)
  unsigned long long used;      // rows pivoted so far
  unsigned long long pmask[2];  // pivot rows of the current panel (double-buffered)
  unsigned long long pad;
  cplx det;
};
static_assert(sizeof(GjState) <= 256 * sizeof(int), "GjState exceeds its LDS slot");

// Panel [k0, k0 + pb) on one wave, lane = row r < n (n <= 64), rows kept in place
// (implicit pivoting).  Pivot of column k: the largest |re| + |im| over the rows not yet
// pivoted (compared to 2^-17 relative, the first row among near-equal ones).  The pivot row r_k is scaled by 1 / piv (its column-k entry becomes
// 1 / piv) and every other row r loses f_r = A[r][k] times it (its column-k entry
// becomes -f_r / piv), over the panel's columns only.  Updates the state (pivot rows,
// used rows, row order, det).
__device__ __forceinline__ void gj_panel(cplx* B, int ld, int n, int k0, int pb, int panel,
                                         GjState* st, int lane) {
  const bool live = lane < n;
  unsigned long long used = st->used;
  int vr = st->vrow[lane];
  cplx det = st->det;
  unsigned long long pm = 0ull;
  int rk[GJ_PB];
  cplx p[GJ_PB];
  // loads clamped into the matrix and masked after, so they issue back to back
#pragma unroll
  for (int j = 0; j < GJ_PB; ++j) {
    const cplx v = B[(live ? lane : 0) * ld + k0 + (j < pb ? j : 0)];
    p[j] = (live && j < pb) ? v : cplx{0.0, 0.0};
    rk[j] = 0;
  }
#pragma unroll
  for (int j = 0; j < GJ_PB; ++j) {
    if (j >= pb) continue;
    const int k = k0 + j;
    // one 32-bit key per candidate row: |re| + |im| as float32 with its low 6 bits
    // replaced by 63 - row, so an integer wave maximum picks the largest magnitude and,
    // among magnitudes equal to 2^-17 relative, the first row
    const bool cand = live && !((used >> lane) & 1ull);
    const float amag = (float)(fabs(p[j].re) + fabs(p[j].im));
    unsigned key = 0u;
    if (cand) key = (amag == amag ? (__float_as_uint(amag) & ~63u) : 0u) | (unsigned)(63 - lane);
    const unsigned kmax = __ockl_wfred_max_u32(key);
    // (a column of NaN or zeros only: the first remaining row)
    const int pr = kmax ? 63 - (int)(kmax & 63u) : __builtin_ctzll(__ballot(cand));
    used |= 1ull << pr;
    pm |= 1ull << pr;
    rk[j] = pr;
    // the row-exchanging elimination would swap positions k and q (row pr's position)
    const int q = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(vr == pr)));
    const int vk = __builtin_amdgcn_readlane(vr, k);
    vr = lane == k ? pr : (lane == q ? vk : vr);
    const cplx piv = readlane_c(p[j], pr);
    det = cmul(det, piv);
    if (q != k) det = cplx{-det.re, -det.im};
    const double d2 = rcp_f64(piv.re * piv.re + piv.im * piv.im);
    const cplx ipiv = cplx{piv.re * d2, -piv.im * d2};
    cplx qv[GJ_PB];
#pragma unroll
    for (int jj = 0; jj < GJ_PB; ++jj) qv[jj] = jj == j ? ipiv : cmul(readlane_c(p[jj], pr), ipiv);
    const cplx f = p[j];
    const bool pivrow = lane == pr;
#pragma unroll
    for (int jj = 0; jj < GJ_PB; ++jj) {
      if (jj == j) {
        const cplx e = cmul(f, ipiv);
        p[jj] = pivrow ? ipiv : cplx{-e.re, -e.im};
      } else {
        const cplx e = cmul(f, qv[jj]);
        p[jj] = pivrow ? qv[jj] : cplx{p[jj].re - e.re, p[jj].im - e.im};
      }
    }
  }
#pragma unroll
  for (int j = 0; j < GJ_PB; ++j)
    if (live && j < pb) B[lane * ld + k0 + j] = p[j];
  st->vrow[lane] = vr;
  if (lane < pb) st->rho[k0 + lane] = lane == 0 ? rk[0] : lane == 1 ? rk[1] : lane == 2 ? rk[2] : rk[3];
  if (lane == 0) {
    st->used = used;
    st->pmask[panel & 1] = pm;
    st->det = det;
  }
}

// In-place inversion of the n x n complex matrix B (row stride ld, LDS; st right after
// it) by NW >= ceil(n / 16) waves; TT >= ceil(n / 16) row tiles.  Wave w owns column block w (all its row tiles): it
// factors the panels that fall in its block and applies every panel's transform to its
// block, so one barrier per panel orders the factorization before the other blocks'
// updates.  For panel K (pivot rows R_K) and a column x outside it:
//   x <- T x[R_K] + (x with the rows R_K cleared),  T = the panel's columns,
// four real MFMAs per 16 x 16 tile.  On return B holds S with
//   O^-1[i][j] = S[rho[i]][rhoinv[j]],
// and st->det = det(O).  Ends with a barrier.  With det_only, column blocks that no later
// panel reads are left as they are (the same pivots, hence the same det; no inverse).
template <int NW, int TT>
__device__ __forceinline__ void gj_invert(cplx* B, int ld, int n, GjState* st, int lane, int wv,
                                          bool det_only) {
  const int tid = threadIdx.x;
  if (tid < 64) st->vrow[tid] = tid;
  if (tid == 0) {
    st->used = 0ull;
    st->det = cplx{1.0, 0.0};
  }
  const int tt = (n + 15) >> 4;
  const int kk = lane >> 4, c16 = lane & 15;
  const int cb = 16 * wv + c16;  // this wave's column
  const bool mine = wv < tt;
  lds_barrier();
  for (int k0 = 0, panel = 0; k0 < n; k0 += GJ_PB, ++panel) {
    const int pb = min(GJ_PB, n - k0);
    if (wv == (k0 >> 4)) gj_panel(B, ld, n, k0, pb, panel, st, lane);
    lds_barrier();
    if (!mine || (det_only && 16 * (wv + 1) <= k0 + pb)) continue;
    // loads clamped into the matrix and masked after, so they issue back to back
    const unsigned long long pm = st->pmask[panel & 1];
    const bool kok = kk < pb, cok = cb < n;
    const int kc = k0 + (kok ? kk : 0), cbc = cok ? cb : 0;
    const cplx xv = B[st->rho[kc] * ld + cbc];
    const double br = (kok && cok) ? xv.re : 0.0, bi = (kok && cok) ? xv.im : 0.0;
    double4_t dr[TT], di[TT];
#pragma unroll
    for (int tr = 0; tr < TT; ++tr) {
      dr[tr] = di[tr] = double4_t{0.0, 0.0, 0.0, 0.0};
      if (tr >= tt) continue;
      const int ra = 16 * tr + c16;
      const cplx tv = B[(ra < n ? ra : 0) * ld + kc];
      const double ar = (kok && ra < n) ? tv.re : 0.0, ai = (kok && ra < n) ? tv.im : 0.0;
      cplx dv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * tr + kk + 4 * q;
        dv[q] = B[(row < n ? row : 0) * ld + cbc];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * tr + kk + 4 * q;
        const bool ok = row < n && cok && !((pm >> row) & 1ull);
        dr[tr][q] = ok ? dv[q].re : 0.0;
        di[tr][q] = ok ? dv[q].im : 0.0;
      }
      dr[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, dr[tr], 0, 0, 0);
      dr[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, dr[tr], 0, 0, 0);
      di[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, di[tr], 0, 0, 0);
      di[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, di[tr], 0, 0, 0);
    }
    // every read of this block precedes the first write (the wave's LDS operations stay
    // in order); the panel's own columns keep T
    if (cok && (cb < k0 || cb >= k0 + pb)) {
#pragma unroll
      for (int tr = 0; tr < TT; ++tr) {
        if (tr >= tt) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = 16 * tr + kk + 4 * q;
          if (row < n) B[row * ld + cb] = cplx{dr[tr][q], di[tr][q]};
        }
      }
    }
  }
  lds_barrier();
  if (tid < n) st->rhoinv[st->rho[tid]] = tid;
  lds_barrier();
}

// waves per walker (two for n <= 24, four beyond) and the LDS the two-wave kernel's
// cross-wave overlap reduction needs
constexpr int meas_waves(int t2) { return t2 <= 3 ? 2 : 4; }
// waves per SIMD the register budget is compiled for
constexpr int meas_wpe(int t2) { return t2 <= 3 ? 2 : t2 == 4 ? 4 : t2 <= 6 ? 3 : 2; }
constexpr int meas_ti(int t2) { return t2 > 3 ? 1 : (t2 + 1) / 2; }
constexpr size_t meas_red_bytes(int t2) {
  return t2 <= 3 ? (size_t)meas_ti(t2) * t2 * 4 * 64 * sizeof(double) : 0;
}
// walkers up to this size are staged in LDS by the two-wave kernel (four blocks per CU)
constexpr size_t MEAS_STAGE_MAX = 40 * 1024;

// [Or | Oi] = C^T [wr | wi] for the row tiles [tb, tb + TI) of O, into M (complex n x n,
// row stride ldm; K = N).  All TI x T2 accumulators are live, so each B value feeds TI MFMAs; the
// operands of k-group chunk j + NW are loaded while chunk j runs.  With NW = 2 the waves
// take alternate chunks, wave 1's partial sums reach wave 0 through red (summed in the
// order wave 0 + wave 1) and wave 0 writes M; `aliased` adds the barrier that keeps red's
// writes after both waves' last read of a staged walker sharing that LDS.
template <int T2, int TI, int NW>
__device__ __forceinline__ void overlap_tiles(int N, int n, int tb, const double* __restrict__ trial,
                                              const double* __restrict__ wsrc, cplx* M, int ldm,
                                              double* red, bool aliased, int lane, int wv) {
  const int n2 = 2 * n;
  const int s = lane >> 4, col = lane & 15;
  const int nkg = (N + 3) >> 2;
  int boff[T2];
#pragma unroll
  for (int tc = 0; tc < T2; ++tc) {
    const int c = tc * 16 + col;
    boff[tc] = c < n2 ? 2 * (c < n ? c : c - n) + (c < n ? 0 : 1) : -1;
  }
  double4_t acc[TI][T2];
#pragma unroll
  for (int ti = 0; ti < TI; ++ti)
#pragma unroll
    for (int tc = 0; tc < T2; ++tc) acc[ti][tc] = double4_t{0.0, 0.0, 0.0, 0.0};
  // two operand buffers with compile-time names (a runtime buffer index would put them
  // in scratch memory)
  double a0[MEAS_KC][TI], b0[MEAS_KC][T2], a1[MEAS_KC][TI], b1[MEAS_KC][T2];
  // Loads come from clamped (always valid) addresses and issue unconditionally.  Rows
  // i >= n and columns c >= 2n of the product are never stored, so only the k padding
  // p >= N needs a zero, on one operand; it is applied where the MFMA reads the operand,
  // so the wait for a chunk's loads falls just before its MFMAs.
  auto load = [&](double (&a)[MEAS_KC][TI], double (&b)[MEAS_KC][T2], int kg0) {
#pragma unroll
    for (int u = 0; u < MEAS_KC; ++u) {
      const int pc = min(4 * (kg0 + u) + s, N - 1);
#pragma unroll
      for (int ti = 0; ti < TI; ++ti) a[u][ti] = trial[pc * n + min((tb + ti) * 16 + col, n - 1)];
#pragma unroll
      for (int tc = 0; tc < T2; ++tc) b[u][tc] = wsrc[(int64_t)2 * pc * n + max(boff[tc], 0)];
    }
  };
  auto mma = [&](const double (&a)[MEAS_KC][TI], const double (&b)[MEAS_KC][T2], int kg0) {
#pragma unroll
    for (int u = 0; u < MEAS_KC; ++u) {
      const bool pok = 4 * (kg0 + u) + s < N;
#pragma unroll
      for (int ti = 0; ti < TI; ++ti) {
        const double av = __builtin_unpredictable(pok) ? a[u][ti] : 0.0;
#pragma unroll
        for (int tc = 0; tc < T2; ++tc)
          acc[ti][tc] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[u][tc], acc[ti][tc], 0, 0, 0);
      }
    }
  };
  const int nch = (nkg + MEAS_KC - 1) / MEAS_KC;
  if (wv < nch) load(a0, b0, wv * MEAS_KC);
  for (int ch = wv; ch < nch; ch += 2 * NW) {
    if (ch + NW < nch) load(a1, b1, (ch + NW) * MEAS_KC);
    mma(a0, b0, ch * MEAS_KC);
    if (ch + 2 * NW < nch) load(a0, b0, (ch + 2 * NW) * MEAS_KC);
    if (ch + NW < nch) mma(a1, b1, (ch + NW) * MEAS_KC);
  }
  if constexpr (NW > 1) {
    if (aliased) __syncthreads();
    if (wv == 1) {
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int tc = 0; tc < T2; ++tc)
#pragma unroll
          for (int r = 0; r < 4; ++r) red[((ti * T2 + tc) * 4 + r) * 64 + lane] = acc[ti][tc][r];
    }
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
      for (int tc = 0; tc < T2; ++tc)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[ti][tc][r] += red[((ti * T2 + tc) * 4 + r) * 64 + lane];
  }
#pragma unroll
  for (int tc = 0; tc < T2; ++tc) {
    if (boff[tc] < 0) continue;
    const int c = tc * 16 + col;
    const int cj = c < n ? c : c - n, ci = c < n ? 0 : 1;
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = (tb + ti) * 16 + s + 4 * r;
        if (row < n) reinterpret_cast<double*>(&M[row * ldm + cj])[ci] = acc[ti][tc][r];
      }
  }
}

// thread 0: det of this spin and, on the last spin's launch, the walker's weight
__device__ inline void finish_walker(cplx det, cplx* dets, int w, int spin,
                                     const WeightsArgs& tail) {
  dets[(int64_t)w * 2 + spin] = det;
  if (tail.weights) {
    const cplx onew = tail.nspin == 1 ? cmul(det, det) : cmul(dets[(int64_t)w * 2], det);
    walker_weight_update(tail, tail.scalars[1], w, onew);
  }
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// 8 floats -> hi and lo bf16 planes, x ~= hi + lo
__device__ inline void split8_bf(const float (&v)[8], bf16x8_t& h8, bf16x8_t& l8) {
  u32x4_t ph, pl;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t h = pack_bf16x2(v[2 * j], v[2 * j + 1]);
    ph[j] = h;
    pl[j] = pack_bf16x2(v[2 * j] - bf16_lo_val(h), v[2 * j + 1] - bf16_hi_val(h));
  }
  h8 = __builtin_bit_cast(bf16x8_t, ph);
  l8 = __builtin_bit_cast(bf16x8_t, pl);
}

// The mixed mode's Green product, where only the split-bf16 planes are wanted (they are
// the A operand of the split-bf16 force-bias GEMM): [Gr ; Gi] = X' [wr^T ; wi^T] with
// X' = [[Xr^T, -Xi^T], [Xi^T, Xr^T]] (2n x 2n), on v_mfma_f32_16x16x32_bf16 with both
// operands split into hi + lo bf16 planes (al bh + ah bl + ah bh, float32 accumulation)
// rather than on float64 MFMA.  K = 2n runs in KB blocks of 32, zero beyond 2n in A.
//   A (lane l): row r = 16 tr + l % 16, k = 32 kb + 8 (l / 16) + e, read once from X in LDS
//   B (lane l): k = 32 kb + 8 (l / 16) + e, column p = 16 tp + l % 16, from the walker
//   D (lane l, element j): row 16 tr + 4 (l / 16) + j, column 16 tp + l % 16
// bpre holds column tile wv's walker operand, loaded by the caller (it is in flight
// during the inversion).  The waves take alternate column tiles.
template <int T2>
struct GreenBf {
  static constexpr int KB = (T2 + 1) / 2;  // 2n <= 16 T2
};
template <int T2>
__device__ __forceinline__ void green_bf_load_b(const double* __restrict__ phid, int N, int n,
                                                int tp, int lane, double (&b)[GreenBf<T2>::KB][8]) {
  const int s = lane >> 4, col = lane & 15;
  const double* rowp = phid + (int64_t)2 * min(tp * 16 + col, N - 1) * n;
#pragma unroll
  for (int kb = 0; kb < GreenBf<T2>::KB; ++kb)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = kb * 32 + 8 * s + e;  // k >= 2n meets zeros of A: any valid entry
      const int kj = min(k < n ? k : k - n, n - 1);
      b[kb][e] = rowp[2 * kj + (k < n ? 0 : 1)];
    }
}
template <int T2, int NW>
__device__ __forceinline__ void green_bf_tiles(int N, int n, const double* __restrict__ phid,
                                               const cplx* M, int ld, const GjState* st,
                                               uint16_t* __restrict__ gbf, int ld16, int lane,
                                               int wv, double (&bpre)[GreenBf<T2>::KB][8]) {
  constexpr int KB = GreenBf<T2>::KB;
  const int n2 = 2 * n;
  const int s = lane >> 4, col = lane & 15;
  const int tp_n = (N + 15) >> 4;
  bf16x8_t ah[T2][KB], al[T2][KB];
  {
    int xcol[T2];
#pragma unroll
    for (int tr = 0; tr < T2; ++tr) {
      const int r = tr * 16 + col;  // (rows r >= 2n are not stored)
      xcol[tr] = st->rhoinv[min(r < n ? r : r - n, n - 1)];
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float v[T2][8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = kb * 32 + 8 * s + e;
        const int xr = st->rho[min(k < n ? k : k - n, n - 1)] * ld;
#pragma unroll
        for (int tr = 0; tr < T2; ++tr) {
          const int r = tr * 16 + col;
          const cplx x = M[xr + xcol[tr]];  // X[kj][ri]
          // (r < n, k < n): Xr; (r < n, k >= n): -Xi; (r >= n, k < n): Xi; else Xr
          const double d = (r < n) == (k < n) ? x.re : ((r < n) ? -x.im : x.im);
          v[tr][e] = k < n2 ? (float)d : 0.f;
        }
      }
#pragma unroll
      for (int tr = 0; tr < T2; ++tr) split8_bf(v[tr], ah[tr][kb], al[tr][kb]);
    }
  }
  for (int tp = wv; tp < tp_n; tp += NW) {
    bf16x8_t bh[KB], bl[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = (float)bpre[kb][e];
      split8_bf(f, bh[kb], bl[kb]);
    }
    if (tp + NW < tp_n) green_bf_load_b<T2>(phid, N, n, tp + NW, lane, bpre);
    float4_t acc[T2];
#pragma unroll
    for (int tr = 0; tr < T2; ++tr) {
      acc[tr] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        acc[tr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[tr][kb], bh[kb], acc[tr], 0, 0, 0);
        acc[tr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tr][kb], bl[kb], acc[tr], 0, 0, 0);
        acc[tr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[tr][kb], bh[kb], acc[tr], 0, 0, 0);
      }
    }
    const int p = tp * 16 + col;
    if (p >= N) continue;
#pragma unroll
    for (int tr = 0; tr < T2; ++tr)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = tr * 16 + 4 * s + j;
        if (r < n2) {
          const float v = acc[tr][j];
          const uint16_t h = f32_to_bf16_rne(v);
          uint16_t* q = gbf + bf_pos((int64_t)r * ld16 + p);
          q[0] = h;
          q[BF_LO] = f32_to_bf16_rne(v - __uint_as_float((uint32_t)h << 16));
        }
      }
  }
}

// n <= 24 (T2 <= 3): two waves per walker.  STAGE 2: the walker is staged in LDS (one
// round of loads) and stays there for the Green product, with O and the inversion's
// state after it; with two row tiles of O each wave then forms one of them over the whole
// K, else the waves split K and wave 1's partial sums reach wave 0 through LDS.  STAGE 1
// (walker too large to keep beside O): staged for the overlap product only, the region
// then reused for O, the state and the partials, the Green product reading the walker
// from global memory.  STAGE 0: no staging.  Each wave's first Green tile of the walker
// operand loads while the waves invert O; the Green product's A operand (from X) is then
// read into registers once and the walker operand runs two tiles ahead.
template <int T2, int STAGE>
__device__ __forceinline__ void measure_narrow_body(
    int N, int n, const cplx* __restrict__ walkers, const double* __restrict__ trial,
    cplx* __restrict__ dets, int spin, double* __restrict__ green, uint16_t* __restrict__ gbf,
    int ld16, const int w, const WeightsArgs& tail) {
  constexpr int NW = 2, TI = meas_ti(T2);
  constexpr int NKG = 4 * T2;  // k groups of 2n <= 16 T2
  extern __shared__ double smem[];
  const int n2 = 2 * n, ld = gj_ld(n);
  cplx* ph = reinterpret_cast<cplx*>(smem);                   // staged walker (STAGE > 0)
  cplx* M = STAGE == 2 ? ph + N * n : ph;                     // O, then its inverse: n x ld
  GjState* st = reinterpret_cast<GjState*>(M + n * ld);       // the inversion's state
  double* red = reinterpret_cast<double*>(reinterpret_cast<int*>(st) + 256);  // overlap partials
  // wave index as a scalar: the waves' paths below are real branches, so registers that
  // live on one wave's path only can share storage with the other's
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = lane >> 4, col = lane & 15;
  const cplx* phi = walkers + (int64_t)w * N * n;
  const double* phid = reinterpret_cast<const double*>(phi);

  if constexpr (STAGE == 2) {
    for (int e = threadIdx.x; e < N * n; e += 64 * NW) ph[e] = phi[e];
    __syncthreads();
    phid = reinterpret_cast<const double*>(ph);
    if constexpr (TI == 2)
      overlap_tiles<T2, 1, 1>(N, n, wv, trial, phid, M, ld, nullptr, false, lane, 0);
    else
      overlap_tiles<T2, TI, NW>(N, n, 0, trial, phid, M, ld, red, false, lane, wv);
  } else if constexpr (STAGE == 1) {
    for (int e = threadIdx.x; e < N * n; e += 64 * NW) ph[e] = phi[e];
    __syncthreads();
    overlap_tiles<T2, TI, NW>(N, n, 0, trial, reinterpret_cast<const double*>(ph), M, ld,
                              red, true, lane, wv);
  } else {
    overlap_tiles<T2, TI, NW>(N, n, 0, trial, phid, M, ld, red, false, lane, wv);
  }

  // ---- O^-1 and det(O) (blocked in-place Gauss-Jordan, both waves); then
  // [Gr ; Gi] = [[Xr^T, -Xi^T], [Xi^T, Xr^T]] [wr^T ; wi^T], K = 2n, columns p in tiles
  // of 16, tiles split between the waves.
  const bool want_green = green || gbf;
  const int tp_n = (N + 15) >> 4;
  // B[k][p] = re / im of w[p][k mod n]: 32-bit offsets within a walker row (tile
  // invariant), one row base per tile, clamped loads masked after
  int boff[NKG];
#pragma unroll
  for (int kg = 0; kg < NKG; ++kg) {
    const int k = 4 * kg + s;
    boff[kg] = k < n2 ? 2 * (k < n ? k : k - n) + (k < n ? 0 : 1) : -1;
  }
  // (clamped, unmasked: columns p >= N are not stored, and A is zero for k >= 2n)
  auto load_b = [&](double (&b)[NKG], int tp) {
    const double* rowp = phid + (int64_t)2 * min(tp * 16 + col, N - 1) * n;
#pragma unroll
    for (int kg = 0; kg < NKG; ++kg) b[kg] = rowp[max(boff[kg], 0)];
  };
  // each wave's first tile loads while the waves invert O
  double b[NKG];
  double bbf[GreenBf<T2>::KB][8];
  if (green && wv < tp_n) load_b(b, wv);
  if (!green && gbf && wv < tp_n) green_bf_load_b<T2>(phid, N, n, wv, lane, bbf);
  gj_invert<NW, 2>(M, ld, n, st, lane, wv, !want_green);
  if (threadIdx.x == 0) finish_walker(st->det, dets, w, spin, tail);
  if (!want_green) return;
  if (!green) {  // split-bf16 planes only (mixed mode's step)
    green_bf_tiles<T2, NW>(N, n, phid, M, ld, st, gbf + 2 * (int64_t)w * n2 * ld16, ld16, lane, wv, bbf);
    return;
  }

  // A operand of every tile, from X in LDS, read once: the pivot maps of the lane's rows
  // and columns first, then every element, each load from a clamped index
  int xrow[NKG], xcol[T2];
#pragma unroll
  for (int kg = 0; kg < NKG; ++kg) {
    const int k = 4 * kg + s;
    xrow[kg] = st->rho[min(k < n ? k : k - n, n - 1)] * ld;
  }
#pragma unroll
  for (int tr = 0; tr < T2; ++tr) {
    const int r = tr * 16 + col;
    xcol[tr] = st->rhoinv[min(r < n ? r : r - n, n - 1)];
  }
  double a[NKG][T2];
#pragma unroll
  for (int kg = 0; kg < NKG; ++kg)
#pragma unroll
    for (int tr = 0; tr < T2; ++tr) {
      const int k = 4 * kg + s;
      const int r = tr * 16 + col;
      const cplx x = M[xrow[kg] + xcol[tr]];
      // X[kj][ri]: (r < n, k < n): Xr; (r < n, k >= n): -Xi; (r >= n, k < n): Xi; else Xr
      const double v = (r < n) == (k < n) ? x.re : ((r < n) ? -x.im : x.im);
      a[kg][tr] = k < n2 ? v : 0.0;  // (rows r >= 2n are not stored)
    }
  double* gw = green ? green + (int64_t)w * n2 * N : nullptr;
  uint16_t* gb = gbf ? gbf + 2 * (int64_t)w * n2 * ld16 : nullptr;
  // tile tp; the walker operand of tile tp + NW loads into b once the MFMAs have read it
  auto tile = [&](int tp) {
    double4_t acc[T2];
#pragma unroll
    for (int tr = 0; tr < T2; ++tr) acc[tr] = double4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kg = 0; kg < NKG; ++kg)
#pragma unroll
      for (int tr = 0; tr < T2; ++tr)
        acc[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kg][tr], b[kg], acc[tr], 0, 0, 0);
    if (tp + NW < tp_n) load_b(b, tp + NW);
    // row tr * 16 + 4 q + s of column p: one base pointer per lane, wave-uniform offsets
    const int p = tp * 16 + col;
    if (p >= N) return;
    double* gwp = gw ? gw + (int64_t)s * N + p : nullptr;
    uint16_t* gbp = gb ? gb + bf_pos((int64_t)s * ld16 + p) : nullptr;
#pragma unroll
    for (int tr = 0; tr < T2; ++tr)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r0 = tr * 16 + 4 * q;
        if (r0 + s < n2) {
          if (gwp) gwp[(int64_t)r0 * N] = acc[tr][q];
          if (gbp) {
            uint16_t* e = gbp + 2 * (int64_t)r0 * ld16;
            split_bf16(acc[tr][q], e, e + BF_LO);
          }
        }
      }
  };
  for (int tp = wv; tp < tp_n; tp += NW) tile(tp);
}

// n > 24: four waves per walker; four (n <= 32) or three (n <= 48) walkers share a CU.
//   - Overlaps: chunks of 16 rows of the walker and of the trial pass through LDS (loaded
//     once by all waves, two chunks ahead in registers: the walker comes from HBM), and the
//     tiles of O are dealt to the waves one by one.
//   - The inversion on all four waves.
//   - Green's function: X is first laid out in LDS as the A operand, P[k][c] = [Xr | Xi]
//     through the pivot maps (in place of O), so a k group is one read per row tile without
//     maps or selections: rows k < n of A are P[k][r], rows n + k are P[k] with its halves
//     exchanged and the first negated.  One 16-byte load of the walker feeds both.
// Per walker at norb 200, n = 40 and two walkers per CU, in cycles (MFMA alone in brackets):
// overlaps 44k (13k), inversion 82k, Green's function 55k (26k); with the operands read as
// they came (X through both maps for each tile) it was 42k, 83k and 108k.  A launch with the
// float64 Green's function, 2048 walkers: 455 -> 335 us; norb 131, n = 29, 777 walkers: 131 ->
// 75 us; norb 250, n = 50, 512: 321 -> 184 us.
constexpr int MW_KC = 16;  // rows per chunk of the overlap product
// doubles per LDS row: 16 T2 columns, == 16 (mod 32), so rows k and k + 1 meet different
// bank halves
__host__ __device__ constexpr int mw_ps(int t2) { return 16 * t2 + (t2 % 2 ? 0 : 16); }
__host__ __device__ constexpr int mw_ts(int t2) {  // of the trial's rows: ceil(n / 16) tiles
  const int ti = (t2 + 1) / 2;
  return 16 * ti + (ti % 2 ? 0 : 16);
}
// LDS shared in turn by the overlap's chunks (two buffers), O and P
__host__ __device__ constexpr size_t mw_region(int t2, int n) {
  const size_t stage = (size_t)2 * MW_KC * (mw_ps(t2) + mw_ts(t2)) * sizeof(double);
  const size_t o = (size_t)n * gj_ld(n) * sizeof(cplx);
  const size_t p = (size_t)((n + 3) & ~3) * mw_ps(t2) * sizeof(double);
  const size_t m = stage > o ? (stage > p ? stage : p) : (o > p ? o : p);
  return (m + 15) & ~(size_t)15;
}
constexpr size_t mw_bytes(int t2, int n) { return mw_region(t2, n) + 256 * sizeof(int); }

template <int T2>
__device__ __forceinline__ void measure_wide_body(
    int N, int n, const cplx* __restrict__ walkers, const double* __restrict__ trial,
    cplx* __restrict__ dets, int spin, double* __restrict__ green, uint16_t* __restrict__ gbf,
    int ld16, const int w, const WeightsArgs& tail) {
  constexpr int NW = 4, NT = 64 * NW, KC = MW_KC;
  constexpr int PS = mw_ps(T2), TS = mw_ts(T2);
  constexpr int TIM = (T2 + 1) / 2;             // row tiles of O at most
  constexpr int UPW = (TIM * T2 + NW - 1) / NW;  // tiles of O per wave
  constexpr int NE = (8 * T2 * KC + NT - 1) / NT;  // chunk elements per thread (n <= 8 T2)
  extern __shared__ double smem[];
  const int n2 = 2 * n, ld = gj_ld(n);
  cplx* M = reinterpret_cast<cplx*>(smem);  // O, then its inverse: n x ld
  GjState* st = reinterpret_cast<GjState*>(reinterpret_cast<char*>(smem) + mw_region(T2, n));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = lane >> 4, col = lane & 15;
  const cplx* phi = walkers + (int64_t)w * N * n;

  // ---- O = C^T w, [Or | Oi] = C^T [wr | wi] in 16 x 16 tiles, tile u of the wave:
  // number wv + 4 u, row-major over ceil(n / 16) x T2
  const int tiles = ((n + 15) >> 4) * T2;
  {
    double* sb = smem;                 // [2][KC][PS]: [wr | wi]
    double* sa = smem + 2 * KC * PS;   // [2][KC][TS]: C
    // two sets: a chunk's loads are issued two chunks ahead of its products
    cplx rw0[NE], rw1[NE];
    double rt0[NE], rt1[NE];
    int ow[NE], ot[NE];  // LDS offsets of the thread's elements of a chunk
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = tid + NT * i, r = e / n, j = e - r * n;
      ow[i] = r * PS + j;
      ot[i] = r * TS + j;
    }
    // a chunk is contiguous in both arrays; past the last row: any entry, zeros of C
    auto load = [&](cplx (&rw)[NE], double (&rt)[NE], int p0) {
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const int e = min(p0 * n + tid + NT * i, N * n - 1);
        rw[i] = phi[e];
        rt[i] = trial[e];
      }
    };
    auto store = [&](const cplx (&rw)[NE], const double (&rt)[NE], int buf, int p0) {
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const int e = tid + NT * i;
        if (e >= KC * n) continue;
        double* b = sb + buf * KC * PS + ow[i];
        b[0] = rw[i].re;
        b[n] = rw[i].im;
        sa[buf * KC * TS + ot[i]] = p0 * n + e < N * n ? rt[i] : 0.0;
      }
    };
    int aoff[UPW], boff[UPW];
    double4_t acc[UPW];
#pragma unroll
    for (int u = 0; u < UPW; ++u) {
      const int t = min(wv + NW * u, tiles - 1), ti = t / T2;
      aoff[u] = s * TS + ti * 16 + col;  // (rows i >= n and columns c >= 2n are not stored)
      boff[u] = s * PS + (t - ti * T2) * 16 + col;
      acc[u] = double4_t{0.0, 0.0, 0.0, 0.0};
    }
    const int nch = (N + KC - 1) / KC;
    auto product = [&](int buf) {
#pragma unroll
      for (int kg = 0; kg < KC / 4; ++kg)
#pragma unroll
        for (int u = 0; u < UPW; ++u) {
          if (wv + NW * u >= tiles) continue;  // (uniform)
          acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(sa[(buf * KC + 4 * kg) * TS + aoff[u]],
                                                        sb[(buf * KC + 4 * kg) * PS + boff[u]],
                                                        acc[u], 0, 0, 0);
        }
    };
    load(rw0, rt0, 0);
    load(rw1, rt1, KC);
    store(rw0, rt0, 0, 0);
    lds_barrier();
    for (int ch = 0; ch < nch; ch += 2) {
      load(rw0, rt0, (ch + 2) * KC);
      product(0);
      store(rw1, rt1, 1, (ch + 1) * KC);
      lds_barrier();
      if (ch + 1 >= nch) break;
      load(rw1, rt1, (ch + 3) * KC);
      product(1);
      store(rw0, rt0, 0, (ch + 2) * KC);
      lds_barrier();
    }
#pragma unroll
    for (int u = 0; u < UPW; ++u) {
      const int t = wv + NW * u, ti = t / T2, c = (t - ti * T2) * 16 + col;
      if (t >= tiles || c >= n2) continue;
      const int cj = c < n ? c : c - n, ci = c < n ? 0 : 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = ti * 16 + s + 4 * r;
        if (row < n) reinterpret_cast<double*>(&M[row * ld + cj])[ci] = acc[u][r];
      }
    }
  }

  // ---- O^-1 and det(O): blocked in-place Gauss-Jordan on all four waves
  gj_invert<NW, TIM>(M, ld, n, st, lane, wv, !(green || gbf));
  const cplx det = st->det;
  if (!(green || gbf)) {
    if (tid == 0) finish_walker(det, dets, w, spin, tail);
    return;
  }

  // ---- P from X (through registers: P takes the place of M), zero rows up to a k group
  double* P = smem;
  {
    constexpr int NX = T2 * T2 / 4 + (T2 * T2 % 4 ? 1 : 0);  // n^2 / 256 at most
    cplx x[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = min(tid + NT * i, n * n - 1), k = e / n, r = e - k * n;
      x[i] = M[st->rho[k] * ld + st->rhoinv[r]];
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = tid + NT * i, k = e / n, r = e - k * n;
      if (e >= n * n) continue;
      P[k * PS + r] = x[i].re;
      P[k * PS + n + r] = x[i].im;
    }
    for (int e = tid; e < (((n + 3) & ~3) - n) * PS; e += NT) P[n * PS + e] = 0.0;
    lds_barrier();
  }

  // (past the last barrier: only this wave waits for it)
  if (tid == NT - 64) finish_walker(det, dets, w, spin, tail);

  // ---- [Gr ; Gi] = [[Xr^T, -Xi^T], [Xi^T, Xr^T]] [wr^T ; wi^T], K = 2n, columns p; the
  // waves take alternate column tiles
  double* gw = green ? green + (int64_t)w * n2 * N : nullptr;
  uint16_t* gb = gbf ? gbf + 2 * (int64_t)w * n2 * ld16 : nullptr;
  const int tp_n = (N + 15) >> 4, nkg = (n + 3) >> 2;
  const double* P0 = P + s * PS + col;  // + 16 tr: row k < n of A
  const double* P1[T2];                 // row n + k of A, before its sign
  unsigned sgn[T2];
#pragma unroll
  for (int tr = 0; tr < T2; ++tr) {
    const int r = tr * 16 + col;
    P1[tr] = P + s * PS + (r < n ? r + n : min(r - n, n - 1));
    sgn[tr] = r < n ? 0x80000000u : 0u;
  }
  auto flip = [](double v, unsigned m) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    return __longlong_as_double((long long)(u ^ ((unsigned long long)m << 32)));
  };
  auto load_w = [&](int tp, int kg) {
    return phi[min(tp * 16 + col, N - 1) * n + min(4 * kg + s, n - 1)];
  };
  constexpr int PD = 2;  // k groups of the walker in flight
  cplx b[PD];
#pragma unroll
  for (int u = 0; u < PD; ++u) b[u] = load_w(wv, u);  // (clamped: valid past the last group)
  for (int tp = wv; tp < tp_n; tp += NW) {
    double4_t acc[T2];
#pragma unroll
    for (int tr = 0; tr < T2; ++tr) acc[tr] = double4_t{0.0, 0.0, 0.0, 0.0};
    for (int kg0 = 0; kg0 < nkg; kg0 += PD) {
#pragma unroll
      for (int u = 0; u < PD; ++u) {
        const int kg = kg0 + u;
        if (kg < nkg) {  // (uniform)
          const double* p0 = P0 + kg * 4 * PS;
#pragma unroll
          for (int tr = 0; tr < T2; ++tr)
            acc[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(p0[tr * 16], b[u].re, acc[tr], 0, 0, 0);
#pragma unroll
          for (int tr = 0; tr < T2; ++tr)
            acc[tr] = __builtin_amdgcn_mfma_f64_16x16x4f64(flip(P1[tr][kg * 4 * PS], sgn[tr]),
                                                           b[u].im, acc[tr], 0, 0, 0);
        }
        // the group PD ahead, of the next tile past this one's end
        const bool more = kg0 + PD < nkg;
        b[u] = load_w(more ? tp : tp + NW, more ? kg + PD : u);
      }
    }
    const int p = tp * 16 + col;
    if (p >= N) continue;
#pragma unroll
    for (int tr = 0; tr < T2; ++tr)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = tr * 16 + s + 4 * q;
        if (row < n2) {
          if (gw) gw[(int64_t)row * N + p] = acc[tr][q];
          if (gb) store_split_bf16(gb, (int64_t)row * ld16 + p, acc[tr][q]);
        }
      }
  }
}

template <int T2, int TI, int STAGE>
__global__ __launch_bounds__(64 * meas_waves(T2), meas_wpe(T2)) void measure_kernel(
    int N, int n, const cplx* __restrict__ walkers, const double* __restrict__ trial,
    cplx* __restrict__ dets, int spin, double* __restrict__ green, uint16_t* __restrict__ gbf,
    int ld16, WeightsArgs tail) {
  if constexpr (T2 <= 3)
    measure_narrow_body<T2, STAGE>(N, n, walkers, trial, dets, spin, green, gbf, ld16,
                                   blockIdx.x, tail);
  else
    measure_wide_body<T2>(N, n, walkers, trial, dets, spin, green, gbf, ld16, blockIdx.x,
                          tail);
}

template <int T2, int TI, int STAGE>
__global__ __launch_bounds__(64 * meas_waves(T2), meas_wpe(T2)) void measure_grouped_kernel(const MeasureArgs* __restrict__ args,
                                                             const int* __restrict__ start,
                                                             int nprob) {
  const int p = group_of(start, nprob, blockIdx.x);
  const MeasureArgs a = args[p];
  const WeightsArgs none{};
  if constexpr (T2 <= 3)
    measure_narrow_body<T2, STAGE>(a.N, a.n, a.walkers, a.trial, a.dets, a.spin, a.green,
                                   a.gbf, a.ld16, blockIdx.x - start[p], none);
  else
    measure_wide_body<T2>(a.N, a.n, a.walkers, a.trial, a.dets, a.spin, a.green, a.gbf,
                          a.ld16, blockIdx.x - start[p], none);
}

template <int T2, int STAGE>
int launch_measure_grouped_s(hipStream_t st, const MeasureArgs* args, const int* start,
                             int nprob, int nblocks, size_t shm) {
  constexpr int TI = meas_ti(T2);
  static int lds_limit = 0;
  const int rc =
      ensure_dyn_lds((const void*)measure_grouped_kernel<T2, TI, STAGE>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((measure_grouped_kernel<T2, TI, STAGE>), dim3(nblocks),
                     dim3(64 * meas_waves(T2)), shm, st, args, start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int T2>
int launch_measure_grouped_t(hipStream_t st, int stage, const MeasureArgs* args,
                             const int* start, int nprob, int nblocks, size_t shm) {
  if constexpr (T2 <= 3) {
    if (stage == 2) return launch_measure_grouped_s<T2, 2>(st, args, start, nprob, nblocks, shm);
    if (stage == 1) return launch_measure_grouped_s<T2, 1>(st, args, start, nprob, nblocks, shm);
  }
  return launch_measure_grouped_s<T2, 0>(st, args, start, nprob, nblocks, shm);
}

template <int T2, int STAGE>
int launch_measure_s(afqmc_ctx* c, int W, int n, const cplx* wk, int s, bool g64, bool gbf,
                     const WeightsArgs& tail, size_t shm) {
  constexpr int TI = meas_ti(T2);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)measure_kernel<T2, TI, STAGE>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((measure_kernel<T2, TI, STAGE>), dim3(W), dim3(64 * meas_waves(T2)), shm,
                     c->stream, c->d.norb, n, wk, c->trial[s], c->dets, s,
                     g64 ? c->green[s] : nullptr, gbf ? c->green_bf[s] : nullptr,
                     c->Np32, tail);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int T2>
int launch_measure_t(afqmc_ctx* c, int W, int n, const cplx* wk, int s, bool g64, bool gbf,
                     const WeightsArgs& tail) {
  int t2, stage;
  size_t shm;
  measure_plan(c, s, &t2, &stage, &shm);
  if constexpr (T2 <= 3) {
    if (stage == 2) return launch_measure_s<T2, 2>(c, W, n, wk, s, g64, gbf, tail, shm);
    if (stage == 1) return launch_measure_s<T2, 1>(c, W, n, wk, s, g64, gbf, tail, shm);
  }
  return launch_measure_s<T2, 0>(c, W, n, wk, s, g64, gbf, tail, shm);
}

}  // namespace

int launch_measure(afqmc_ctx* c, int W, const cplx* wup, const cplx* wdn, bool g64, bool gbf,
                   const WeightsArgs* tail) {
  for (int sp = 0; sp < c->nspin; ++sp) {
    const int n = c->nocc[sp];
    const cplx* wk = (sp == 0) ? wup : wdn;
    const WeightsArgs t = (tail && sp == c->nspin - 1) ? *tail : WeightsArgs{};
    int rc;
    switch ((2 * n + 15) / 16) {
      case 1: rc = launch_measure_t<1>(c, W, n, wk, sp, g64, gbf, t); break;
      case 2: rc = launch_measure_t<2>(c, W, n, wk, sp, g64, gbf, t); break;
      case 3: rc = launch_measure_t<3>(c, W, n, wk, sp, g64, gbf, t); break;
      case 4: rc = launch_measure_t<4>(c, W, n, wk, sp, g64, gbf, t); break;
      case 5: rc = launch_measure_t<5>(c, W, n, wk, sp, g64, gbf, t); break;
      case 6: rc = launch_measure_t<6>(c, W, n, wk, sp, g64, gbf, t); break;
      case 7: rc = launch_measure_t<7>(c, W, n, wk, sp, g64, gbf, t); break;
      default: rc = launch_measure_t<8>(c, W, n, wk, sp, g64, gbf, t); break;
    }
    if (rc) return rc;
  }
  return AFQMC_OK;
}

// Grouped form: one launch for every (fragment, spin) problem with the same column-tile
// count t2 and staging choice; shm is the largest LDS need among them.
int launch_measure_grouped(hipStream_t st, int t2, int stage, const MeasureArgs* args,
                           const int* start, int nprob, int nblocks, size_t shm) {
  switch (t2) {
    case 1: return launch_measure_grouped_t<1>(st, stage, args, start, nprob, nblocks, shm);
    case 2: return launch_measure_grouped_t<2>(st, stage, args, start, nprob, nblocks, shm);
    case 3: return launch_measure_grouped_t<3>(st, stage, args, start, nprob, nblocks, shm);
    case 4: return launch_measure_grouped_t<4>(st, stage, args, start, nprob, nblocks, shm);
    case 5: return launch_measure_grouped_t<5>(st, stage, args, start, nprob, nblocks, shm);
    case 6: return launch_measure_grouped_t<6>(st, stage, args, start, nprob, nblocks, shm);
    case 7: return launch_measure_grouped_t<7>(st, stage, args, start, nprob, nblocks, shm);
    default: return launch_measure_grouped_t<8>(st, stage, args, start, nprob, nblocks, shm);
  }
}

// The kernel launch_measure picks for spin s, as a plan for grouped launches: column tiles
// t2 of the Green product, the staging mode and the LDS bytes.
void measure_plan(const afqmc_ctx* c, int s, int* t2, int* stage, size_t* shm) {
  const int n = c->nocc[s], N = c->d.norb;
  const int t = (2 * n + 15) / 16;
  *t2 = t > 8 ? 8 : t;
  const size_t walker = (size_t)N * n * sizeof(cplx);
  if (*t2 <= 3) {  // two-wave kernel
    const size_t red = meas_red_bytes(*t2);
    const size_t kept = walker + gj_bytes(n) + (meas_ti(*t2) == 2 ? 0 : red);
    const size_t m_red = gj_bytes(n) + red;
    if (kept <= MEAS_STAGE_MAX) {  // walker kept beside O for the Green product
      *stage = 2;
      *shm = kept;
    } else if (walker <= MEAS_STAGE_MAX) {  // O, state and partials alias the walker
      *stage = 1;
      *shm = std::max(walker, m_red);
    } else {
      *stage = 0;
      *shm = m_red;
    }
    return;
  }
  *stage = 0;
  *shm = mw_bytes(*t2, n);
}

// ------------------------------------------------------------------------------------
// A whole float64 step of small problems, one workgroup per walker: Green's function (unless
// the last step left it), force bias and fields, V, Taylor, the new overlaps and the weight
// update, and in the workgroup that finishes last the population-control shift.
//
// What it is for: an H10 chain's step (norb 10, n = 5, 27 vectors, 200 walkers) is seven
// launches of 3.5 to 9 us, each a chain of dependent loads on a mostly idle chip, plus the
// gaps between them.  Everything but the shift is per walker, and a walker's intermediates
// fit LDS; the price is that every walker reads the Cholesky vectors itself (small_step_fits
// has the line).  The chain is what bounds it, so four lanes share every sum (their partial
// sums meet in the quad), what is read from memory is asked for ahead of its use, and O
// (n <= 8) is inverted in the registers of one wave while the others wait or multiply.
namespace {

struct SmallStep {
  int W, N, G, nspin, chol_spins, terms_k, nv, mult, reuse, keep;
  int n[2];
  double dt, sqdt;
  const double* trial[2];
  const double* rot[2];
  const double* chol_t;
  const double* E[2];
  const cplx* mf;
  cplx* walkers[2];
  double* green[2];
  const double* fields;
  WeightsArgs tail;
  int* arrived;  // workgroups done, 0 between launches
};

constexpr int SMALL_NT = 256, SMALL_MAX_N = 28, SMALL_MAX_OCC = 8;
constexpr int SMALL_R = (SMALL_MAX_N * SMALL_MAX_OCC * 4 + SMALL_NT - 1) / SMALL_NT;  // sums per quad

// lane ^ 1 and lane ^ 2 of a quad
template <int CTRL>
__device__ inline double quad_dpp(double x) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)u, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double quad_sum(double x) {
  x += quad_dpp<0xB1>(x);         // quad_perm [1, 0, 3, 2]
  return x + quad_dpp<0x4E>(x);   // quad_perm [2, 3, 0, 1]
}

// det(O) and, with full, X = O^-1 of the n x n matrix at O (rows of SMALL_MAX_OCC, LDS), by
// one wave: lane j holds column j of O, lane 8 + j column j of the unit matrix; Gauss-Jordan
// with row exchanges, pivots by largest |re| + |im|.
__device__ __forceinline__ cplx small_invert(const cplx* O, cplx* X, int n, bool full, int lane) {
  constexpr int M = SMALL_MAX_OCC;
  cplx c[M];
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const cplx o = O[r * M + (lane & 7)];
    c[r] = lane < M ? o : cplx{lane - M == r ? 1.0 : 0.0, 0.0};
  }
  cplx det = {1.0, 0.0};
#pragma unroll
  for (int k = 0; k < M; ++k) {
    if (k >= n) continue;
    cplx p[M];  // column k, the same in all lanes
#pragma unroll
    for (int r = 0; r < M; ++r)
      if (r >= k || full) p[r] = readlane_c(c[r], k);
    int pr = k;
    double best = fabs(p[k].re) + fabs(p[k].im);
#pragma unroll
    for (int r = k + 1; r < M; ++r) {
      const double a = fabs(p[r].re) + fabs(p[r].im);
      if (r < n && a > best) {
        best = a;
        pr = r;
      }
    }
    pr = __builtin_amdgcn_readfirstlane(pr);
#pragma unroll
    for (int r = k + 1; r < M; ++r)
      if (r == pr) {
        const cplx a = c[k], b = p[k];
        c[k] = c[r];
        c[r] = a;
        p[k] = p[r];
        p[r] = b;
      }
    det = cmul(det, p[k]);
    if (pr != k) det = cplx{-det.re, -det.im};
    const double d2 = rcp_f64(p[k].re * p[k].re + p[k].im * p[k].im);
    c[k] = cmul(c[k], cplx{p[k].re * d2, -p[k].im * d2});
#pragma unroll
    for (int r = 0; r < M; ++r)
      if (r != k && r < n && (r > k || full)) c[r] = csub(c[r], cmul(p[r], c[k]));
  }
  if (full && lane >= M && lane < M + n) {
#pragma unroll
    for (int r = 0; r < M; ++r)
      if (r < n) X[r * M + lane - M] = c[r];
  }
  return det;
}

// walker_weight_update on two lanes: the importance function on even, the phase on odd ones
__device__ __forceinline__ void small_weight(const WeightsArgs& a, double pcs, int w, cplx onew,
                                             cplx st, cplx ft, cplx oold, double wold, int lane) {
  const bool phase = lane & 1;
  const cplx e = phase ? cplx{-a.sqdt * st.re, -a.sqdt * st.im}
                       : cplx{-a.sqdt * st.re + ft.re + a.dt * (pcs + a.h0_prop),
                              -a.sqdt * st.im + ft.im};
  const cplx z = cdiv(cmul(cexp_(e), onew), oold);
  const double f = phase ? cos(atan2(z.im, z.re)) : hypot(z.re, z.im);
  const double g = quad_dpp<0xB1>(f);
  if (lane == 0) {
    double ipl = f * g;
    if (isnan(ipl)) ipl = 0.0;
    if (ipl < 1.0e-3) ipl = 0.0;
    if (ipl > 100.0) ipl = 0.0;
    double wt = ipl * wold;
    if (wt > 100.0) wt = 0.0;
    // (written through: the last workgroup reads it, possibly on another XCD)
    __hip_atomic_store(a.weights + w, wt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    a.overlaps[w] = onew;
  }
}

// doubles of LDS: Green's functions, x, V, walker, E and trial of a spin, O and X
__host__ __device__ inline int small_doubles(int N, int n0, int n1, int G) {
  const int n = n0 > n1 ? n0 : n1;
  return 2 * N * (n0 + n1) + 2 * G + 2 * N * N + 2 * N * n + N * N + N * n +
         4 * SMALL_MAX_OCC * SMALL_MAX_OCC;
}

__global__ __launch_bounds__(SMALL_NT, 2) void small_step_kernel(SmallStep a) {
  constexpr int M = SMALL_MAX_OCC;
  extern __shared__ double smem[];
  __shared__ double red[4 * (SMALL_NT / 64)];
  __shared__ cplx dets[2];
  __shared__ int last;
  const int t = threadIdx.x, lane = t & 63, w = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), q4 = t & 3;
  const int N = a.N, G = a.G, nm = max(a.n[0], a.n[1]);

  // the walker's Green's functions [re / im][i][p]
  auto gl = [&](int s) { return smem + (s ? 2 * N * a.n[0] : 0); };
  cplx* V = reinterpret_cast<cplx*>(gl(1) + 2 * N * a.n[1]);
  cplx* y = V + N * N;
  cplx* O = y + N * nm;
  cplx* X = O + M * M;
  double* E = reinterpret_cast<double*>(X + M * M);
  double* C = E + N * N;
  double* xr = C + N * nm;
  double* xi = xr + G;

  auto stage_walker = [&](int s) {
    const int c = N * a.n[s];
    const cplx* phi = a.walkers[s] + (int64_t)w * c;
    for (int o = t; o < c; o += SMALL_NT) y[o] = phi[o];
  };
  auto stage_trial = [&](int s) {
    const int c = N * a.n[s];
    for (int o = t; o < c; o += SMALL_NT) C[o] = a.trial[s][o];
  };
  // O = C^T y, four lanes per entry (n^2 <= 64 entries)
  auto overlap = [&](int n) {
    const int e = t >> 2, i = e / n, j = e - i * n;
    cplx z = {0.0, 0.0};
    if (i < n)
      for (int p = q4; p < N; p += 4) {
        const double v = C[p * n + i];
        const cplx b = y[p * n + j];
        z.re = fma(v, b.re, z.re);
        z.im = fma(v, b.im, z.im);
      }
    z.re = quad_sum(z.re);
    z.im = quad_sum(z.im);
    if (i < n && q4 == 0) O[i * M + j] = z;
  };
  // entry o = i N + p of the Green's function, (y X)[p][i]
  auto green = [&](int o, int n) {
    const int i = o / N, p = o - i * N;
    cplx z = {0.0, 0.0};
    for (int j = 0; j < n; ++j) z = cadd(z, cmul(y[p * n + j], X[j * M + i]));
    return z;
  };

  // ---- Green's functions of the walker
  for (int s = 0; s < a.nspin; ++s) {
    const int n = a.n[s], c = N * n;
    if (a.reuse) {
      for (int e = t; e < 2 * c; e += SMALL_NT) gl(s)[e] = a.green[s][(int64_t)w * 2 * c + e];
    } else {
      if (s) __syncthreads();
      stage_walker(s);
      stage_trial(s);
      __syncthreads();
      overlap(n);
      __syncthreads();
      if (wave == 0) small_invert(O, X, n, true, lane);
      __syncthreads();
      for (int o = t; o < c; o += SMALL_NT) {
        const cplx z = green(o, n);
        gl(s)[o] = z.re;
        gl(s)[c + o] = z.im;
      }
    }
  }
  __syncthreads();
  // the first spin's walker and E, and what the weight update needs, while the fields form
  if (a.reuse || a.nspin > 1) stage_walker(0);
  for (int e = t; e < N * N; e += SMALL_NT) E[e] = a.E[0][e];
  const cplx oold = a.tail.overlaps[w];
  const double wold = a.tail.weights[w], pcs = a.tail.scalars[1];

  // ---- force bias and fields (fields_kernel's formulas)
  cplx st = {0.0, 0.0}, ft = {0.0, 0.0};
  for (int g0 = 0; g0 < G; g0 += SMALL_NT / 4) {
    const int g = g0 + (t >> 2), gc = min(g, G - 1);
    const cplx m = a.mf[gc];
    const double xv = a.fields[(int64_t)w * G + gc];
    double fr = 0.0, fi = 0.0;
    for (int s = 0; s < a.nspin; ++s) {
      const int c = N * a.n[s];
      const double* r = a.rot[s] + (int64_t)gc * c;
#pragma unroll 8
      for (int e = q4; e < c; e += 4) {
        const double v = r[e];
        fr = fma(v, gl(s)[e], fr);
        fi = fma(v, gl(s)[c + e], fi);
      }
    }
    const cplx f = {a.mult * quad_sum(fr), a.mult * quad_sum(fi)};
    if (g < G && q4 == 0) {
      const cplx fs = {-a.sqdt * (-f.im - m.re), -a.sqdt * (f.re - m.im)};
      const cplx xt = {xv - fs.re, -fs.im};
      const cplx fs2 = cmul(fs, fs);
      st = cadd(st, cmul(xt, m));
      ft = cadd(ft, cplx{xv * fs.re - fs2.re / 2.0, xv * fs.im - fs2.im / 2.0});
      xr[g] = -a.sqdt * xt.im;
      xi[g] = a.sqdt * xt.re;
    }
  }
  {
    double v[4] = {st.re, st.im, ft.re, ft.im};
#pragma unroll
    for (int off = 32; off >= 4; off >>= 1)  // (lanes 4 i carry the sums)
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] += __shfl_down(v[c], off, 64);
    if (lane == 0)
#pragma unroll
      for (int c = 0; c < 4; ++c) red[wave * 4 + c] = v[c];
  }
  __syncthreads();

  for (int s = 0; s < a.nspin; ++s) {
    const int n = a.n[s], c = N * n;
    if (s) {  // (the last spin's Green's function is done with y)
      stage_walker(s);
      for (int e = t; e < N * N; e += SMALL_NT) E[e] = a.E[s][e];
    }
    stage_trial(s);
    // ---- V (as N x N, from the packed upper triangle too)
    if (s == 0 || a.chol_spins == 2) {
      const double* L = a.chol_t + (int64_t)(a.chol_spins == 2 ? s : 0) * a.nv * G;
      const bool packed = a.nv != N * N;
      for (int e0 = 0; e0 < a.nv; e0 += SMALL_NT / 4) {
        const int e = e0 + (t >> 2);
        const double* r = L + (int64_t)min(e, a.nv - 1) * G;
        double vr = 0.0, vi = 0.0;
#pragma unroll 8
        for (int g = q4; g < G; g += 4) {
          const double l = r[g];
          vr = fma(l, xr[g], vr);
          vi = fma(l, xi[g], vi);
        }
        vr = quad_sum(vr);
        vi = quad_sum(vi);
        if (e < a.nv && q4 == 0) {
          if (packed) {
            // row p of the triangle starts at p N - p (p - 1) / 2
            const float b = (float)(2 * N + 1);
            int p = (int)((b - sqrtf(b * b - 8.0f * (float)e)) * 0.5f);
            if (p * N - p * (p - 1) / 2 > e) --p;
            if ((p + 1) * N - (p + 1) * p / 2 <= e) ++p;
            const int k = p + e - (p * N - p * (p - 1) / 2);
            V[p * N + k] = V[k * N + p] = cplx{vr, vi};
          } else {
            V[e] = cplx{vr, vi};
          }
        }
      }
    }
    __syncthreads();
    // ---- w <- E (t0 + V t0 + V V t0 / 2 + ...), t0 = E w, in Horner form; the lane of
    // number j mod 4 of a quad stores its sum j
    int prow[SMALL_R], pcol[SMALL_R];
    cplx t0[SMALL_R], u[SMALL_R];
#pragma unroll
    for (int j = 0; j < SMALL_R; ++j) {
      const int o = min((t >> 2) + SMALL_NT / 4 * j, c - 1);
      prow[j] = o / n;
      pcol[j] = o - prow[j] * n;
      t0[j] = u[j] = cplx{0.0, 0.0};
    }
    auto real_product = [&](cplx (&out)[SMALL_R]) {  // out = E y
#pragma unroll
      for (int j = 0; j < SMALL_R; ++j) {
        if (SMALL_NT / 4 * j >= c) continue;
        cplx x = {0.0, 0.0};
#pragma unroll 4
        for (int q = q4; q < N; q += 4) {
          const double v = E[prow[j] * N + q];
          const cplx z = y[q * n + pcol[j]];
          x.re = fma(v, z.re, x.re);
          x.im = fma(v, z.im, x.im);
        }
        out[j] = cplx{quad_sum(x.re), quad_sum(x.im)};
      }
    };
    auto put = [&](const cplx (&v)[SMALL_R]) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < SMALL_R; ++j) {
        const int o = (t >> 2) + SMALL_NT / 4 * j;
        if (o < c && q4 == (j & 3)) y[o] = v[j];
      }
      __syncthreads();
    };
    real_product(t0);
    put(t0);
    for (int k = a.terms_k; k >= 1; --k) {
      const double dk = (double)k, rk = 1.0 / dk;
#pragma unroll
      for (int j = 0; j < SMALL_R; ++j) {
        if (SMALL_NT / 4 * j >= c) continue;
        cplx x0 = {0.0, 0.0}, x1 = {0.0, 0.0};
#pragma unroll 4
        for (int q = q4; q < N; q += 4) {
          const cplx v = V[prow[j] * N + q], z = y[q * n + pcol[j]];
          x0.re = fma(v.re, z.re, x0.re);
          x0.im = fma(v.re, z.im, x0.im);
          x1.re = fma(-v.im, z.im, x1.re);
          x1.im = fma(v.im, z.re, x1.im);
        }
        // x / k: the product with 1 / k corrected by its residual
        const double sr = quad_sum(x0.re + x1.re), si = quad_sum(x0.im + x1.im);
        const double qr = sr * rk, qi = si * rk;
        u[j] = cplx{t0[j].re + fma(fma(-qr, dk, sr), rk, qr),
                    t0[j].im + fma(fma(-qi, dk, si), rk, qi)};
      }
      put(u);
    }
    real_product(u);
    put(u);
    cplx* phi = a.walkers[s] + (int64_t)w * c;
    for (int o = t; o < c; o += SMALL_NT) phi[o] = y[o];

    // ---- new overlaps; one wave updates the weight, the others form the Green's function
    // for the next step
    overlap(n);
    __syncthreads();
    if (wave == 0) {
      const cplx det = small_invert(O, X, n, a.keep, lane);
      if (lane == 0) dets[s] = det;
    }
    __syncthreads();
    if (wave == 0) {
      if (s + 1 == a.nspin) {
        const cplx onew = cmul(dets[0], dets[s]);
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (red[i] + red[4 + i]) + (red[8 + i] + red[12 + i]);
        small_weight(a.tail, pcs, w, onew, cplx{v[0], v[1]}, cplx{v[2], v[3]}, oold, wold, lane);
      }
    } else if (a.keep) {
      double* gw = a.green[s] + (int64_t)w * 2 * c;
      for (int o = t - 64; o < c; o += SMALL_NT - 64) {
        const cplx z = green(o, n);
        gw[o] = z.re;
        gw[c + o] = z.im;
      }
    }
    __syncthreads();
  }

  // ---- population-control shift (propagation.py:161-164) by the last workgroup to arrive.
  // Nothing but the weights is read across workgroups: they are written through, and the
  // wait puts a weight in place before its workgroup arrives (a release at agent scope would
  // write the whole L2 back: 3 us).  Every workgroup has read the old shift by then.
  if (t == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(a.arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           a.W - 1;
  }
  __syncthreads();
  if (!last) return;
  double part = 0.0;
  for (int i = t; i < a.W; i += SMALL_NT)
    part += __hip_atomic_load(a.tail.weights + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const double total = block_sum<SMALL_NT>(part, red);
  if (t == 0) {
    a.tail.scalars[1] = a.tail.scalars[0] - 0.1 * (log(total / (double)a.W) / a.dt);
    *a.arrived = 0;
  }
}

}  // namespace

// Where one launch is the better step.  A workgroup runs through a walker's sums by itself, on
// vector instructions: the entries of the Cholesky vectors (V's and the half-rotated ones),
// one product each, and the Taylor terms, N^2 n products each on four lanes' chains, which
// weigh four times as much a term.  Separate launches take a spin's part as often as there are
// spins.  Hence the cost per spin, entries + 4 terms N^2 n; separate against one launch, us a
// step (graph of 20 steps), five terms:
//   W <= 256, a CU to a workgroup: norb 10, n = 5, 27 vectors (cost 12800) 31.3 : 19.8; norb
//     24, n = 6, 96 vectors (112000) 40.6 : 37.6; two spins of norb 24, n = 8, 70 vectors
//     (116000) 70.9 : 63.5; norb 26, n = 8, 40 vectors (131000) 43.0 : 42.4; norb 28, n = 7,
//     50 vectors (140000) 43.3 : 43.7; norb 30, n = 8, 5 vectors (148000) 42.4 : 45.8
//   to 512, two workgroups to a CU: norb 16, n = 4, 250 vectors (70500) 44.2 : 41.6; two
//     spins of norb 20, n = 8 + 7, a set of 69 vectors each (84800) 80.9 : 78.7, n = 8 + 8,
//     94 vectors (88900) 75.4 : 78.7; norb 20, n = 5, 100 vectors, V whole (90000) 44.1 : 45.2
//   more walkers: norb 16, n = 4, 64 vectors, five steps 272 : 196 at 500, 289 : 321 at 1000
// Past norb 28 a step may lose below those lines (norb 29, n = 5, 70 vectors, 122000: 41.1 :
// 45.3; norb 31, n = 3, 40 vectors, 512 walkers, 81000: 40.5 : 42.6; two spins of norb 31, n =
// 8 + 1, 60 vectors, 110000: 64.0 : 68.6; norb 30, n = 5 + 5, a set of 30 vectors each,
// 108000: 70.2 : 79.7), past 50000 entries the Cholesky vectors alone are too many (norb 32,
// n = 8, 128 vectors, five steps: 339 : 393).
// LDS grows with the vectors (two doubles each, 400 KB at norb 1 with the 25000 vectors those
// entries allow): what one workgroup can have, or half of a CU's where two have to share it.
constexpr int SMALL_MAX_W = 512;
constexpr int64_t SMALL_MAX_ENTRIES = 50000;
constexpr int64_t SMALL_COST_ONE = 125000, SMALL_COST_TWO = 85000;
constexpr size_t SMALL_LDS_ONE = 156 * 1024, SMALL_LDS_TWO = 78 * 1024;
size_t small_step_lds(const afqmc_ctx* c) {
  return sizeof(double) * (size_t)small_doubles(c->d.norb, c->nocc[0],
                                                c->nspin > 1 ? c->nocc[1] : 0, c->d.nchol);
}
bool small_step_fits(const afqmc_ctx* c, int W) {
  if (c->mixed || c->f32 || W > SMALL_MAX_W || c->d.norb > SMALL_MAX_N) return false;
  int64_t rows = (int64_t)c->chol_spins * c->vhs_nv, taylor = 0;
  for (int s = 0; s < c->nspin; ++s) {
    if (c->nocc[s] < 1 || c->nocc[s] > SMALL_MAX_OCC) return false;
    rows += c->kdim[s];
    taylor += (int64_t)c->kdim[s] * c->d.norb;
  }
  const int64_t entries = rows * c->d.nchol;
  const int64_t cost = (entries + 4 * (c->d.n_exp_terms - 1) * taylor) / c->nspin;
  const bool two = W > 256;  // workgroups on a CU
  return entries <= SMALL_MAX_ENTRIES && cost <= (two ? SMALL_COST_TWO : SMALL_COST_ONE) &&
         small_step_lds(c) <= (two ? SMALL_LDS_TWO : SMALL_LDS_ONE);
}

int launch_small_step(afqmc_ctx* c, int W, cplx* wup, cplx* wdn, const double* fields,
                      const WeightsArgs& tail, bool reuse, bool keep) {
  SmallStep a{};
  a.W = W;
  a.N = c->d.norb;
  a.G = c->d.nchol;
  a.nspin = c->nspin;
  a.chol_spins = c->chol_spins;
  a.terms_k = c->d.n_exp_terms - 1;
  a.nv = c->vhs_nv;
  a.mult = c->mult;
  a.reuse = reuse;
  a.keep = keep;
  a.dt = c->d.dt;
  a.sqdt = sqrt(c->d.dt);
  for (int s = 0; s < c->nspin; ++s) {
    a.n[s] = c->nocc[s];
    a.trial[s] = c->trial[s];
    a.rot[s] = c->rot_chol[s];
    a.E[s] = c->exp_h1[s];
    a.walkers[s] = s ? wdn : wup;
    a.green[s] = c->green[s];
  }
  a.chol_t = c->chol_t;
  a.mf = c->mf_shifts;
  a.fields = fields;
  a.tail = tail;
  a.arrived = c->step_arrived;
  const size_t shm = small_step_lds(c);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)small_step_kernel, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL(small_step_kernel, dim3(W), dim3(SMALL_NT), shm, c->stream, a);
  LAUNCH_CHECK();
  return AFQMC_OK;
}
