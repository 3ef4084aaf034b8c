// Walker re-orthonormalisation: reduced Householder QR, walker <- Q.
// Follows linalg_utils.qr_vmap / qr_vmap_uhf (linalg_utils.py:51-65), i.e.
// jnp.linalg.qr, whose CPU lowering is LAPACK geqrf + orgqr/ungqr.  For the sizes
// here (n <= 64 < the blocked crossover) those are the unblocked zgeqr2 + zung2r:
//   zlarfg: beta = -sign(Re alpha) * |(alpha, x)|, tau = ((beta - Re a)/beta, -Im a/beta),
//           v = [1; x / (alpha - beta)], R[i][i] = beta (real)
//   geqr2 applies H(i)^H = I - conj(tau) v v^H to the trailing columns;
//   ung2r accumulates Q = H(0) ... H(n-1) backwards, in place.
// One workgroup per (walker, spin), the walker's columns in registers.
//
// Bound by the chain of n reflectors, each a norm, a barrier and a round of column updates
// (reductions over the rows), not by flops:
//   - wave w keeps columns w, w + NWV, ... in registers for the whole factorisation (lane l
//     the rows l, l + 64, ...); only the reflectors' vectors go through LDS, written once
//     with their zeros and the leading one;
//   - the owner of column i + 1 updates that column first and forms reflector i + 1 from
//     its registers while the other waves still apply reflector i: one barrier per
//     reflector, reached with the next one ready;
//   - the accumulation of Q needs no barrier where all vectors stay in LDS: a column of Q
//     starts as H(j) e_j and takes H(j - 1) ... H(0) on its own.  Else the vectors return
//     to LDS from their owners' registers in batches.
// Against the walker in LDS, four waves and no look-ahead, per launch: norb 200, 40
// columns, 2048 walkers 2.06 -> 0.90 ms; norb 131, 29 columns, 777 walkers 0.28 -> 0.16;
// norb 100, 20 columns, 1024 walkers 116 -> 90 us; norb 250, 50 columns, 512 walkers (was
// in place in global memory) 3.7 -> 0.39 ms.
#include <type_traits>

#include "common.h"

extern "C" __device__ double __ockl_wfred_add_f64(double);

namespace {

// dynamic LDS: 160 KiB per workgroup less the static arrays below
constexpr size_t QR_LDS_LIMIT = 156 * 1024;
// column stride of LDS (odd: one row's consecutive columns spread over the banks when the
// walker passes through on its way to and from the registers)
__host__ __device__ inline int qr_ldc(int m) { return m | 1; }

// The instances (waves, columns per wave, rows per lane) have to agree to the last bit, as
// a group launches one for its largest member: every product and sum is written as the
// fused or plain operation it is, and nothing is contracted further.
#pragma clang fp contract(off)
__device__ inline cplx qr_mul(cplx a, cplx b) {
  return cplx{fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}

// zlarfg on the column x (lane's rows lane + 64 k; zero past m) for row i: beta =
// -sign(Re alpha) |(alpha, x)|, tau = ((beta - Re alpha) / beta, -Im alpha / beta),
// v = x / (alpha - beta) below row i.  x becomes v, with v_i = 1 and zeros above.
template <int RPL>
__device__ __forceinline__ cplx qr_reflector(cplx (&x)[RPL], int i, int lane) {
  double part = 0.0;
  cplx al = cplx{0.0, 0.0};
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    part = r > i ? fma(x[k].re, x[k].re, fma(x[k].im, x[k].im, part)) : part;
    if (k == (i >> 6)) al = x[k];  // (uniform)
  }
  const double x2 = __ockl_wfred_add_f64(part);
  const cplx alpha = readlane_c(al, i & 63);
  cplx t = cplx{0.0, 0.0}, scal = cplx{1.0, 0.0};
  if (!(x2 == 0.0 && alpha.im == 0.0)) {
    const double n2 = fma(alpha.re, alpha.re, fma(alpha.im, alpha.im, x2));
    double nrm, inrm;
    if (n2 > 0x1p-900 && n2 < 0x1p900) {
      // sqrt and its reciprocal from one estimate: two Newton steps on 1 / sqrt, then the
      // root corrected by its residual
      double y = __builtin_amdgcn_rsq(n2);
#pragma unroll
      for (int it = 0; it < 2; ++it) y = fma(0.5 * y, fma(-n2 * y, y, 1.0), y);
      const double g = n2 * y;
      nrm = fma(fma(-g, g, n2), 0.5 * y, g);
      inrm = y;
    } else {
      // |(alpha, |x|)| scaled by the largest magnitude (dlapy3)
      const double xnorm = sqrt(x2), xa = fabs(alpha.re), ya = fabs(alpha.im);
      const double w = fmax(xa, fmax(ya, xnorm));
      const double iw = 1.0 / w;
      const double a = xa * iw, b = ya * iw, c = xnorm * iw;
      nrm = w * sqrt(fma(a, a, fma(b, b, c * c)));
      inrm = 1.0 / nrm;
    }
    const double sg = alpha.re >= 0.0 ? -1.0 : 1.0;
    const double beta = sg * nrm, ib = sg * inrm;
    const cplx d = cplx{alpha.re - beta, alpha.im};
    t = cplx{-d.re * ib, -alpha.im * ib};
    const double d2 = fma(d.re, d.re, d.im * d.im);
    const double id = d2 > 0x1p-900 && d2 < 0x1p900 ? rcp_f64(d2) : 1.0 / d2;
    scal = cplx{d.re * id, -d.im * id};
  }
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    const cplx v = qr_mul(x[k], scal);
    x[k] = r > i ? v : (r == i ? cplx{1.0, 0.0} : cplx{0.0, 0.0});
  }
  return t;
}

// x <- (I - t v v^H) x for the columns c of a[] with use(c), their reductions side by side
template <int CPW, int RPL, typename F>
__device__ __forceinline__ void qr_apply(cplx (&a)[CPW][RPL], const cplx (&v)[RPL], cplx t,
                                         F&& use) {
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
    if (!use(c)) continue;
    double sr = 0.0, si = 0.0;
#pragma unroll
    for (int k = 0; k < RPL; ++k) {  // conj(v) * a
      sr = fma(v[k].re, a[c][k].re, fma(v[k].im, a[c][k].im, sr));
      si = fma(v[k].re, a[c][k].im, fma(-v[k].im, a[c][k].re, si));
    }
    const cplx ts = qr_mul(t, cplx{__ockl_wfred_add_f64(sr), __ockl_wfred_add_f64(si)});
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      a[c][k].re = fma(-v[k].re, ts.re, fma(v[k].im, ts.im, a[c][k].re));
      a[c][k].im = fma(-v[k].re, ts.im, fma(-v[k].im, ts.re, a[c][k].im));
    }
  }
}

// walker g (m x n, row-major) <- Q.  V: LDS for `slots` vectors of qr_ldc(m); with
// slots == n it also carries the walker between memory and registers.
template <int NWV, int CPW, int RPL>
__device__ __forceinline__ void qr_walker(int m, int n, cplx* __restrict__ g, int slots, cplx* V,
                                          cplx* tau) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ldc = qr_ldc(m);
  const bool whole = slots == n;
  cplx a[CPW][RPL];  // column wave + NWV c, row lane + 64 k

  if (whole) {
    for (int e = threadIdx.x; e < m * n; e += 64 * NWV) {
      const int r = e / n, j = e - r * n;
      V[j * ldc + r] = g[e];
    }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < CPW; ++c)
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int j = wave + NWV * c, r = lane + 64 * k;
      const int jc = min(j, n - 1), rc = min(r, m - 1);
      const cplx x = whole ? V[jc * ldc + rc] : g[rc * n + jc];
      a[c][k] = (j < n && r < m) ? x : cplx{0.0, 0.0};
    }
  if (whole) __syncthreads();  // V now takes the reflectors' vectors

  auto publish = [&](const cplx (&x)[RPL], int slot) {
#pragma unroll
    for (int k = 0; k < RPL; ++k)
      if (lane + 64 * k < m) V[slot * ldc + lane + 64 * k] = x[k];
  };
  auto load_v = [&](cplx (&v)[RPL], int slot) {
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const cplx x = V[slot * ldc + min(lane + 64 * k, m - 1)];
      v[k] = lane + 64 * k < m ? x : cplx{0.0, 0.0};
    }
  };
  // the owner forms reflector i from its column i
  auto form = [&](int i, int slot) {
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      if (i != wave + NWV * c) continue;  // (uniform)
      const cplx t = qr_reflector<RPL>(a[c], i, lane);
      publish(a[c], slot);
      if (lane == 0) tau[i] = t;
    }
  };

  // ---- zgeqr2; vector i in slot i (or alternately in two slots)
  if (wave == 0) form(0, 0);
  lds_barrier();
  for (int i = 0; i + 1 < n; ++i) {
    cplx v[RPL];
    load_v(v, whole ? i : i & 1);
    const cplx tc = cconj(tau[i]);
    const int next = i + 1;
    if (wave == next % NWV) {
      qr_apply<CPW, RPL>(a, v, tc, [&](int c) { return next == wave + NWV * c; });
      form(next, whole ? next : next & 1);
    }
    qr_apply<CPW, RPL>(a, v, tc, [&](int c) {
      const int j = wave + NWV * c;
      return j > next && j < n;
    });
    lds_barrier();
  }

  // ---- zung2r: column j starts as H(j) e_j = e_j - tau_j v_j, then takes H(i), i < j
  auto accumulate = [&](int i, int slot) {
    cplx v[RPL];
    load_v(v, slot);
    const cplx t = tau[i];
    qr_apply<CPW, RPL>(a, v, t, [&](int c) {
      const int j = wave + NWV * c;
      return j > i && j < n;
    });
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      if (i != wave + NWV * c) continue;
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const cplx e = qr_mul(t, v[k]);
        a[c][k] = cplx{(lane + 64 * k == i ? 1.0 : 0.0) - e.re, -e.im};
      }
    }
  };
  if (whole) {
    for (int i = n - 1; i >= 0; --i) accumulate(i, i);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPW; ++c)
      if (wave + NWV * c < n) publish(a[c], wave + NWV * c);
    __syncthreads();
    for (int e = threadIdx.x; e < m * n; e += 64 * NWV) {
      const int r = e / n, j = e - r * n;
      g[e] = V[j * ldc + r];
    }
  } else {
    for (int top = n; top > 0; top -= slots) {  // vectors [lo, top), still in registers
      const int lo = max(0, top - slots);
      lds_barrier();
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        const int j = wave + NWV * c;
        if (j >= lo && j < top) publish(a[c], j - lo);
      }
      lds_barrier();
      for (int i = top - 1; i >= lo; --i) accumulate(i, i - lo);
    }
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int j = wave + NWV * c, r = lane + 64 * k;
        if (j < n && r < m) g[r * n + j] = a[c][k];
      }
  }
}

// waves per SIMD the registers allow for: two workgroups of eight waves where the columns
// fit (norb <= 192)
constexpr int qr_wpe(int nwv, int rpl) { return nwv == 8 && rpl == 3 ? 4 : 1; }

template <int NWV, int CPW, int RPL>
__global__ __launch_bounds__(64 * NWV, qr_wpe(NWV, RPL)) void qr_kernel(int m, int n, cplx* __restrict__ walkers,
                                                      int slots) {
  extern __shared__ double smem[];
  __shared__ cplx tau[AFQMC_MAX_NOCC];
  qr_walker<NWV, CPW, RPL>(m, n, walkers + (int64_t)blockIdx.x * m * n, slots,
                           reinterpret_cast<cplx*>(smem), tau);
}

template <int NWV, int CPW, int RPL>
__global__ __launch_bounds__(64 * NWV, qr_wpe(NWV, RPL)) void qr_grouped_kernel(const QrArgs* __restrict__ args,
                                                              const int* __restrict__ start,
                                                              int nprob) {
  extern __shared__ double smem[];
  __shared__ cplx tau[AFQMC_MAX_NOCC];
  const int p = group_of(start, nprob, blockIdx.x);
  const QrArgs a = args[p];
  qr_walker<NWV, CPW, RPL>(a.m, a.n, a.walkers + (int64_t)(blockIdx.x - start[p]) * a.m * a.n,
                           a.slots, reinterpret_cast<cplx*>(smem), tau);
}

template <int NWV, int CPW, int RPL>
int launch_qr_t(hipStream_t st, int m, int n, cplx* walkers, int W, int slots) {
  const size_t shm = (size_t)qr_ldc(m) * slots * sizeof(cplx);
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)qr_kernel<NWV, CPW, RPL>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((qr_kernel<NWV, CPW, RPL>), dim3(W), dim3(64 * NWV), shm, st, m, n, walkers,
                     slots);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

template <int NWV, int CPW, int RPL>
int launch_qr_grouped_t(hipStream_t st, const QrArgs* args, const int* start, int nprob,
                        int nblocks, size_t shm) {
  static int lds_limit = 0;
  const int rc = ensure_dyn_lds((const void*)qr_grouped_kernel<NWV, CPW, RPL>, shm, &lds_limit);
  if (rc) return rc;
  hipLaunchKernelGGL((qr_grouped_kernel<NWV, CPW, RPL>), dim3(nblocks), dim3(64 * NWV), shm, st,
                     args, start, nprob);
  LAUNCH_CHECK();
  return AFQMC_OK;
}

// f(waves, columns per wave, rows per lane), compile-time constants, for the largest m and
// n of a launch: at most four columns per wave, so that a step's updates stay short beside
// the chain of reflectors
template <int NWV, int CPW, typename F>
int qr_rows(int m, F&& f) {
  constexpr std::integral_constant<int, NWV> nwv{};
  constexpr std::integral_constant<int, CPW> cpw{};
  switch ((m + 63) / 64) {
    case 1: return f(nwv, cpw, std::integral_constant<int, 1>{});
    case 2: return f(nwv, cpw, std::integral_constant<int, 2>{});
    case 3: return f(nwv, cpw, std::integral_constant<int, 3>{});
    default: return f(nwv, cpw, std::integral_constant<int, 4>{});
  }
}
template <typename F>
int qr_select(int m, int n, F&& f) {
  static_assert(AFQMC_MAX_NORB <= 256 && AFQMC_MAX_NOCC <= 64, "rows per lane, columns");
  if (n <= 8) return qr_rows<4, 2>(m, f);
  if (n <= 16) return qr_rows<4, 4>(m, f);
  if (n <= 32) return qr_rows<8, 4>(m, f);
  if (n <= 48) return qr_rows<16, 3>(m, f);
  return qr_rows<16, 4>(m, f);
}

}  // namespace

// vectors the LDS holds: all n, or as many as fit (at least two)
int qr_slots(int m, int n) {
  const int fit = (int)(QR_LDS_LIMIT / (qr_ldc(m) * sizeof(cplx)));
  return fit < n ? fit : n;
}
size_t qr_lds_bytes(int m, int n) { return (size_t)qr_ldc(m) * qr_slots(m, n) * sizeof(cplx); }

// max_m, max_n: over the problems
int launch_qr_grouped(hipStream_t st, const QrArgs* args, const int* start, int nprob,
                      int nblocks, size_t shm, int max_m, int max_n) {
  return qr_select(max_m, max_n, [&](auto nwv, auto cpw, auto rpl) {
    return launch_qr_grouped_t<nwv, cpw, rpl>(st, args, start, nprob, nblocks, shm);
  });
}

int launch_qr(afqmc_ctx* c, int W, cplx* wup, cplx* wdn) {
  const int N = c->d.norb;
  for (int s = 0; s < c->nspin; ++s) {
    const int n = c->nocc[s];
    cplx* walkers = s == 0 ? wup : wdn;
    const int rc =
        qr_in_lds(c) ? launch_qr_lds(c->stream, N, n, walkers, W)
                     : qr_select(N, n, [&](auto nwv, auto cpw, auto rpl) {
                         return launch_qr_t<nwv, cpw, rpl>(c->stream, N, n, walkers, W,
                                                           qr_slots(N, n));
                       });
    if (rc) return rc;
  }
  return AFQMC_OK;
}
