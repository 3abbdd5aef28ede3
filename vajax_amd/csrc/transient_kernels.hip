// Element-wise kernels of the Newton / time-step loop (FP64 throughout).
#include "block_flags.h"
#include "circuit.h"
#include "transient.h"

namespace vjx {

namespace {

__device__ __forceinline__ unsigned long long dbits(double x) {
  return (unsigned long long)__double_as_longlong(x);
}
__device__ __forceinline__ double bitsd(unsigned long long b) {
  return __longlong_as_double((long long)b);
}
// jnp.maximum semantics: NaN propagates.
__device__ __forceinline__ double jmax(double a, double b) {
  if (a != a || b != b) return __longlong_as_double(0x7ff8000000000000LL);
  return a > b ? a : b;
}
__device__ __forceinline__ double jmin(double a, double b) {
  if (a != a || b != b) return __longlong_as_double(0x7ff8000000000000LL);
  return a < b ? a : b;
}

constexpr int kStatusLanes = 1024;  // of the kernels that reduce into a status record

__device__ __forceinline__ unsigned long long max_bits(unsigned long long a,
                                                       unsigned long long b) {
  return b > a ? b : a;
}

// delta test of solver_factories.py:283-299
__global__ void __launch_bounds__(1024) k_delta(int n_unk, int m, int n_total,
                                                const double* __restrict__ delta,
                                                const double* __restrict__ X,
                                                const DevScalars* __restrict__ sc, DevStatus* st) {
  unsigned long long adv = 0, ad = 0;
  unsigned int fail = 0;
  for (int i = (int)(blockIdx.x * kStatusLanes + threadIdx.x); i < n_unk + m;
       i += (int)gridDim.x * kStatusLanes) {
    const double d = delta[i];
    double cd, xr, atol;
    if (i < n_unk) {
      cd = d * sc->nr_damping;
      xr = X[1 + i];
      atol = sc->vntol;
      adv = max_bits(adv, dbits(fabs(d)));
    } else {
      cd = d;
      xr = X[n_total + (i - n_unk)];
      atol = sc->abstol;
    }
    const double tol = jmax(fabs(xr) * sc->reltol, atol);
    fail += !(fabs(cd) < tol);
    ad = max_bits(ad, dbits(fabs(d)));
  }
  block_flags(adv, ad, fail, &st->maxdv_bits, &st->maxdelta_bits, &st->delta_fail);
}

// damped update of solver_factories.py:301-309
__global__ void __launch_bounds__(256) k_update(int n_unk, int m, int n_total,
                                                const double* __restrict__ delta, double* X,
                                                const DevScalars* __restrict__ sc,
                                                const DevStatus* __restrict__ st) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_unk + m) return;
  if (i < n_unk) {
    const double maxdv = bitsd(st->maxdv_bits);
    const double vs = jmin(1.0, sc->max_step / jmax(maxdv, 1e-30));
    X[1 + i] = X[1 + i] + delta[i] * vs * sc->nr_damping;
  } else {
    const int j = n_total + (i - n_unk);
    X[j] = X[j] + delta[i];
  }
}

// k_delta, k_update and k_status_export in one workgroup, for systems of up to
// kFinishMax unknowns: the maxima go through LDS instead of memory, the deltas
// and the iterate stay in registers between test and update, and the same
// thread that has the counts exports the records.
constexpr int kFinishEach = 8;
constexpr int kFinishMax = kStatusLanes * kFinishEach;
__global__ void __launch_bounds__(1024) k_finish(int n_unk, int m, int n_total,
                                                 const double* __restrict__ delta, double* X,
                                                 const DevScalars* __restrict__ sc, DevStatus* st,
                                                 const DevStatus* __restrict__ lu_st,
                                                 DevStatus* out) {
  __shared__ unsigned long long s_adv, s_ad;
  __shared__ unsigned int s_fail;
  const int tid = (int)threadIdx.x;
  if (tid == 0) {
    s_adv = s_ad = 0;
    s_fail = 0;
  }
  const int n = n_unk + m;
  double d[kFinishEach], x[kFinishEach];
#pragma unroll
  for (int u = 0; u < kFinishEach; ++u) {
    const int i = tid + u * kStatusLanes;
    if (i < n) {
      d[u] = delta[i];
      x[u] = X[i < n_unk ? 1 + i : n_total + (i - n_unk)];
    }
  }
  unsigned long long adv = 0, ad = 0;
  unsigned int fail = 0;
#pragma unroll
  for (int u = 0; u < kFinishEach; ++u) {
    const int i = tid + u * kStatusLanes;
    if (i < n) {
      const bool node = i < n_unk;
      const double cd = node ? d[u] * sc->nr_damping : d[u];
      const double tol = jmax(fabs(x[u]) * sc->reltol, node ? sc->vntol : sc->abstol);
      fail += !(fabs(cd) < tol);
      ad = max_bits(ad, dbits(fabs(d[u])));
      if (node) adv = max_bits(adv, dbits(fabs(d[u])));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    adv = max_bits(adv, __shfl_xor(adv, o));
    ad = max_bits(ad, __shfl_xor(ad, o));
    fail += __shfl_xor(fail, o);
  }
  __syncthreads();
  if ((tid & 63) == 0) {
    atomicMax(&s_adv, adv);
    atomicMax(&s_ad, ad);
    atomicAdd(&s_fail, fail);
  }
  __syncthreads();
  const double vs = jmin(1.0, sc->max_step / jmax(bitsd(s_adv), 1e-30));
#pragma unroll
  for (int u = 0; u < kFinishEach; ++u) {
    const int i = tid + u * kStatusLanes;
    if (i < n_unk)
      X[1 + i] = x[u] + d[u] * vs * sc->nr_damping;
    else if (i < n)
      X[n_total + (i - n_unk)] = x[u] + d[u];
  }
  if (tid == 0) {
    DevStatus r = *st;
    r.maxdv_bits = s_adv;
    r.maxdelta_bits = s_ad;
    r.delta_fail = s_fail;
    *st = r;
    out[0] = r;
    out[1] = *lu_st;
  }
}

// Predictor (adaptive.py:94-218) and, for the node rows, the residual
// tolerance floor max(reltol * history max |contribution|, abstol)
// (full_mna.py:1922-1928) of the step, in one launch.
__global__ void k_predict(int n_total, int m, const double* __restrict__ Xa,
                          const double* __restrict__ h0, const double* __restrict__ h1,
                          const double* __restrict__ h2, double a0, double a1, double a2,
                          int can_predict, double* Vp, double* Xw, int n_unk,
                          const double* __restrict__ hmrc, double reltol, double abstol,
                          double* floor) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (floor && i < n_unk) floor[i] = jmax(hmrc[i] * reltol, abstol);
  if (i < n_total) {
    const double v = a0 * h0[i] + a1 * h1[i] + a2 * h2[i];
    Vp[i] = v;
    Xw[i] = can_predict ? v : Xa[i];
  } else if (i < n_total + m) {
    Xw[i] = Xa[i];
  }
}

__global__ void k_fill(int n, double v, double* x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

__global__ void k_copy(int n, const double* __restrict__ a, double* b) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// The fixed-step loop's accepted step in one launch (full_mna.py:1355-1365):
// X_accepted = X_new, and the charge history shifts, Q_prev2 = Q_prev,
// Q_prev = Q_new, dQ/dt_prev = dQ/dt_new (each element read before written).
__global__ void k_fixed_accept(int nx, int n_unk, const double* __restrict__ Xw,
                               double* __restrict__ Xa, const double* __restrict__ Qn,
                               const double* __restrict__ dQn, double* __restrict__ Qp,
                               double* __restrict__ dQ, double* __restrict__ Q2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nx) Xa[i] = Xw[i];
  if (i < n_unk) {
    Q2[i] = Qp[i];
    Qp[i] = Qn[i];
    dQ[i] = dQn[i];
  }
}

// The Newton and LU status records written by one thread straight into
// mapped pinned host memory at the end of an iteration (no copy launches on
// the critical path).
__global__ void k_status_export(const DevStatus* __restrict__ a, const DevStatus* __restrict__ b,
                                DevStatus* out) {
  if (threadIdx.x != 0) return;
  out[0] = *a;
  if (b) out[1] = *b;
}

// Marks the boundaries of a measurement window in kernel traces (a profiler
// keeps the dispatches between two of these); it does no work.
__global__ void k_window_mark(int which) { (void)which; }

__global__ void k_gather(int n, const int32_t* __restrict__ idx, const double* __restrict__ a,
                         double* b) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[idx[i]];
}

__global__ void k_dqdt(int n, double c0, double c1, double d1, double c2,
                       const double* __restrict__ Q, const double* __restrict__ Qp,
                       const double* __restrict__ dQ, const double* __restrict__ Q2, double* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = c0 * Q[i] + c1 * Qp[i] + d1 * dQ[i] + c2 * Q2[i];
}

// LTE ratio of adaptive.py:254-271
__global__ void __launch_bounds__(1024) k_lte(int n, const double* __restrict__ Vn,
                                             const double* __restrict__ Vp,
                                             const double* __restrict__ Vmax, double scale,
                                             double reltol, double abstol, DevStatus* st,
                                             DevStatus* out) {
  unsigned long long top = 0;
  for (int i = (int)(blockIdx.x * kStatusLanes + threadIdx.x); i < n;
       i += (int)gridDim.x * kStatusLanes) {
    const double lte = (Vn[i] - Vp[i]) * scale;
    const double vc = jmax(fabs(Vn[i]), fabs(Vp[i]));
    const double vs = jmax(Vmax[i], vc);
    const double tol = reltol * vs + abstol;
    double r = fabs(lte) / tol;
    if (r != r) r = __longlong_as_double(0x7ff8000000000000LL);
    top = max_bits(top, dbits(r));
  }
  block_flags(top, 0, 0u, &st->maxf_bits, nullptr, nullptr);
  if (out && threadIdx.x == 0) {  // the only workgroup
    DevStatus r = *st;
    r.maxf_bits = __hip_atomic_load(&st->maxf_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *out = r;
  }
}

// state update on use_new_solution (full_mna.py:2078-2113)
__global__ void k_accept(int n_total, int n_unk, int m, const double* __restrict__ Xw, double* Xa,
                         double* hist_new, double* Vmax, const double* __restrict__ Qn,
                         const double* __restrict__ dQn, double* Qp, double* dQ, double* Q2,
                         const double* __restrict__ mrc, double* hmrc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_total) {
    const double v = Xw[i];
    Xa[i] = v;
    hist_new[i] = v;
    Vmax[i] = jmax(Vmax[i], fabs(v));
  }
  if (i < m) Xa[n_total + i] = Xw[n_total + i];
  if (i < n_unk) {
    Q2[i] = Qp[i];
    Qp[i] = Qn[i];
    dQ[i] = dQn[i];
    hmrc[i] = jmax(hmrc[i], mrc[i]);
  }
}

__global__ void k_output(int n_total, int m, const double* __restrict__ Xa,
                         const double* __restrict__ Ivs, int zero_current, double* vrow,
                         double* irow) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_total) vrow[i] = Xa[i];
  if (i < m) irow[i] = zero_current ? 0.0 : Ivs[i];
}

inline int nb(long long n, int b = 256) { return (int)((n + b - 1) / b); }

// A status kernel's workgroups each end with one atomic a value on the same
// cache line, and those run one after another (about 10 ns each), so its
// workgroups have 1024 lanes and there are at most 128 of them: at 130k
// unknowns k_delta 6.8 us and k_lte 4.5 us (14.3 and 8.0 with 509 workgroups of 256).
inline int status_blocks(int n) {
  const int b = (n + kStatusLanes - 1) / kStatusLanes;
  return b < 128 ? b : 128;
}

}  // namespace

void launch_finish(int n_unk, int m, int n_total, const double* delta, double* X,
                   const DevScalars* sc, DevStatus* st, const DevStatus* lu_st, DevStatus* out,
                   int n_noi, const int32_t* noi_rows, hipStream_t s) {
  const int n = n_unk + m;
  // One workgroup up to eight unknowns a lane (noise rows are reset between
  // update and export, so circuits with them keep the launches): the ring of
  // 101 stages 13.0 -> 12.6 ms, even at 4 300 unknowns (14.0 ms); beyond, one
  // compute unit's loads would be the bound.
  if (n <= kFinishMax && n_noi == 0) {
    k_finish<<<1, kStatusLanes, 0, s>>>(n_unk, m, n_total, delta, X, sc, st, lu_st, out);
    return;
  }
  k_delta<<<status_blocks(n), kStatusLanes, 0, s>>>(n_unk, m, n_total, delta, X, sc, st);
  k_update<<<nb(n), 256, 0, s>>>(n_unk, m, n_total, delta, X, sc, st);
  launch_noi_clamp(n_noi, noi_rows, X, s);
  launch_status_export(st, lu_st, out, s);
}
void launch_predict(int n_total, int m, const double* Xa, const double* h0, const double* h1,
                    const double* h2, double a0, double a1, double a2, int can_predict, double* Vp,
                    double* Xw, int n_unk, const double* hmrc, double reltol, double abstol,
                    double* floor, hipStream_t s) {
  // n_unk < n_total: the grid covers the floor rows too
  k_predict<<<nb(n_total + m), 256, 0, s>>>(n_total, m, Xa, h0, h1, h2, a0, a1, a2, can_predict,
                                            Vp, Xw, n_unk, hmrc, reltol, abstol, floor);
}
// Noise-only internal nodes in the Newton solve (solver_factories.py:1268-1276):
// zero their rows and their columns in node rows, put 1 on their diagonals,
// 0 in their right-hand side (three disjoint index sets).
__global__ void k_noi_apply(int nz, const int32_t* __restrict__ zero, int nd,
                            const int32_t* __restrict__ diag, const int32_t* __restrict__ rows,
                            double* csr, double* f) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nz) {
    csr[zero[i]] = 0.0;
  } else if (i < nz + nd) {
    csr[diag[i - nz]] = 1.0;
  } else if (i < nz + 2 * nd) {
    f[rows[i - nz - nd]] = 0.0;
  }
}

// NOI nodes held at 0 V after the update (solver_factories.py:311-313).
__global__ void k_noi_clamp(int nd, const int32_t* __restrict__ rows, double* X) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nd) X[1 + rows[i]] = 0.0;
}

void launch_noi_apply(int nz, const int32_t* zero, int nd, const int32_t* diag,
                      const int32_t* rows, double* csr, double* f, hipStream_t s) {
  const int n = nz + 2 * nd;
  if (n) k_noi_apply<<<nb(n), 256, 0, s>>>(nz, zero, nd, diag, rows, csr, f);
}

void launch_noi_clamp(int nd, const int32_t* rows, double* X, hipStream_t s) {
  if (nd) k_noi_clamp<<<nb(nd), 256, 0, s>>>(nd, rows, X);
}

void launch_fill(int n, double v, double* x, hipStream_t s) {
  if (n) k_fill<<<nb(n), 256, 0, s>>>(n, v, x);
}
void launch_copy(int n, const double* a, double* b, hipStream_t s) {
  if (n) k_copy<<<nb(n), 256, 0, s>>>(n, a, b);
}
void launch_fixed_accept(int nx, int n_unk, const double* Xw, double* Xa, const double* Qn,
                         const double* dQn, double* Qp, double* dQ, double* Q2, hipStream_t s) {
  const int n = nx > n_unk ? nx : n_unk;
  if (n) k_fixed_accept<<<nb(n), 256, 0, s>>>(nx, n_unk, Xw, Xa, Qn, dQn, Qp, dQ, Q2);
}
void launch_window_mark(int which, hipStream_t s) { k_window_mark<<<1, 64, 0, s>>>(which); }
void launch_status_export(const DevStatus* a, const DevStatus* b, DevStatus* out, hipStream_t s) {
  k_status_export<<<1, 64, 0, s>>>(a, b, out);
}
void launch_gather(int n, const int32_t* idx, const double* a, double* b, hipStream_t s) {
  if (n) k_gather<<<nb(n), 256, 0, s>>>(n, idx, a, b);
}
void launch_dqdt(int n, double c0, double c1, double d1, double c2, const double* Q,
                 const double* Qp, const double* dQ, const double* Q2, double* out,
                 hipStream_t s) {
  if (n) k_dqdt<<<nb(n), 256, 0, s>>>(n, c0, c1, d1, c2, Q, Qp, dQ, Q2, out);
}
void launch_lte(int n, const double* Vn, const double* Vp, const double* Vmax, double scale,
                double reltol, double abstol, DevStatus* st, DevStatus* out, hipStream_t s) {
  if (n <= kFinishMax) {
    k_lte<<<1, kStatusLanes, 0, s>>>(n, Vn, Vp, Vmax, scale, reltol, abstol, st, out);
  } else {
    k_lte<<<status_blocks(n), kStatusLanes, 0, s>>>(n, Vn, Vp, Vmax, scale, reltol, abstol, st,
                                                    nullptr);
    launch_status_export(st, nullptr, out, s);
  }
}
void launch_accept(int n_total, int n_unk, int m, const double* Xw, double* Xa, double* hist_new,
                   double* Vmax, const double* Qn, const double* dQn, double* Qp, double* dQ,
                   double* Q2, const double* mrc, double* hmrc, hipStream_t s) {
  k_accept<<<nb(n_total > m ? n_total : m), 256, 0, s>>>(n_total, n_unk, m, Xw, Xa, hist_new, Vmax, Qn, dQn, Qp,
                                           dQ, Q2, mrc, hmrc);
}
void launch_output(int n_total, int m, const double* Xa, const double* Ivs, int zero_current,
                   double* vrow, double* irow, hipStream_t s) {
  k_output<<<nb(n_total + m), 256, 0, s>>>(n_total, m, Xa, Ivs, zero_current, vrow, irow);
}

}  // namespace vjx
