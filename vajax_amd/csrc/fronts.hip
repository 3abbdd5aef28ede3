// Front program on the GPU (fronts.h): refactorisation and solves as dense
// fronts of at most 64 rows, one wavefront per front.
//
// What bounds it: the chain of fronts from the leaves to the root.  Every
// pivot is a dependent step (broadcast, reciprocal, one multiply-add), every
// front a hand-over through L2.  So a front stays in the registers of one
// wavefront -- an 8 x 8 grid of lanes, lane (ti, tj) holding the values
// (ti + 8 a, tj + 8 b) -- where a pivot step needs no barrier: the pivot's row
// and column reach the other lanes through the LDS crossbar (ds_bpermute), no
// memory in between.  A workgroup is four wavefronts walking one piece of the
// tree level by level; pieces that depend on each other are separate launches
// (a 65k-gate circuit: five).
#include "block_flags.h"
#include "internal.h"
#include "lane_value.h"

#include <algorithm>

namespace vjx {

namespace {

constexpr int kWaves = 4;       // wavefronts (small fronts in flight) per workgroup
constexpr int kSmallTiles = 4;  // 8-row tiles of a front for one wavefront (32 rows)

__device__ __forceinline__ unsigned long long dbits(double x) {
  return (unsigned long long)__double_as_longlong(x);
}

// The value of the lane whose number is addr / 4 (any lane per lane).
__device__ __forceinline__ double from_lane(double v, int addr) {
  const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
  const unsigned int lo =
      (unsigned int)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned int)bits);
  const unsigned int hi =
      (unsigned int)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned int)(bits >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float from_lane(float v, int addr) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}

__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// 1 / p to the last bit or two, for quotient(): the hardware's estimate and two
// Newton steps (about 50 cycles of dependent operations; the IEEE division has
// 120 and is on the path of every pivot).  Outside the range where the steps
// neither overflow nor meet denormals, and for zero, infinity and NaN, the
// division itself.
__device__ __forceinline__ double reciprocal(double p) {
  const double a = fabs(p);
  if (!(a > 0x1p-960 && a < 0x1p960)) return 1.0 / p;
  double r = __builtin_amdgcn_rcp(p);
  r = __builtin_fma(r, __builtin_fma(-p, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-p, r, 1.0), r);
}
__device__ __forceinline__ float reciprocal(float p) { return 1.0f / p; }

// a / p from r = reciprocal(p): the correction by the exact remainder leaves
// the rounded quotient (the CPU program divides).  Infinite quotients come out
// as NaN; both count as non-finite factor entries.
template <typename T>
__device__ __forceinline__ T quotient(T a, T p, T r) {
  const T q = a * r;
  const T e = fmadd(-q, p, a);
  return fmadd(e, r, q);
}

// Values one lane of a wavefront wrote to LDS are read by its other lanes
// after this (the LDS executes a wavefront's operations in order; the fence
// only keeps the compiler from reordering or forwarding them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup barrier for data exchanged through LDS only (s_waitcnt immediate
// 0xC07F: lgkmcnt(0), vmcnt and expcnt at their maxima).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

struct Growth {
  double mag = 0.0;      // largest finite |L|
  unsigned int bad = 0;  // non-finite L entries
  __device__ __forceinline__ void add(double x) {
    const double m = fabs(x);
    if (m <= 1.7976931348623157e308)
      mag = fmax(mag, m);
    else
      ++bad;
  }
};

// Where a front's results go: value (i, j) of its pivots' columns and rows to
// the factors, the rest to the update block.
template <typename T>
__device__ __forceinline__ T* front_place(int i, int j, int k, int m, T* fo, T* co) {
  T* const f = fo + (j < k ? j * m + i : k * m + (j - k) * k + i);
  return (j < k || i < k) ? f : co + (j - k) * (m - k) + (i - k);
}

// Elimination of a front's k pivots (at most 32 rows) in the registers of one
// wavefront, an 8 x 8 grid of lanes, from the assembled front in LDS to its
// places.  A front with fewer than four 8-row tiles uses the last ones (off =
// 4 - nt), so that every front runs the same code from pivot block off on.  w
// (RHS): right-hand side, lane = row, before and after.  (Results through LDS
// and column by column took 200 cycles a column; from the registers a 7-row
// front is one store.)
template <bool RHS, typename T>
__device__ __forceinline__ void front_eliminate(int k, int m, int off, int ld, const T* F, int lane,
                                                T* fo, T* co, T& w, Growth& g) {
  constexpr int N = kSmallTiles;
  const int ti = lane & 7, tj = lane >> 3;
  // value (ti + 8 (a - off), tj + 8 (b - off)) at base + 8 a + 8 b ld
  const int base = ti - 8 * off + (tj - 8 * off) * ld;
  T acc[N][N], ww[N];
#pragma unroll
  for (int b = 0; b < N; ++b)
    if (b >= off) {
#pragma unroll
      for (int a = 0; a < N; ++a)
        if (a >= off) acc[a][b] = F[base + 8 * a + 8 * b * ld];
      if constexpr (RHS) ww[b] = from_lane(w, 4 * (ti + 8 * (b - off)));
    }
#pragma unroll
  for (int pb = 0; pb < N; ++pb) {
    const int k0 = k - 8 * (pb - off);  // pivots from this block on
    if (pb < off || k0 <= 0) continue;
    const int pn = k0 < 8 ? k0 : 8;
    for (int pp = 0; pp < pn; ++pp) {
      const T piv = lane_value(acc[pb][pb], 9 * pp);
      const int ca = (ti + 8 * pp) * 4, ra = (pp + 8 * tj) * 4;
      T l[N], u[N];
#pragma unroll
      for (int a = pb; a < N; ++a) {
        l[a] = from_lane(acc[a][pb], ca);
        u[a] = from_lane(acc[pb][a], ra);
      }
      const T r = reciprocal(piv);
#pragma unroll
      for (int a = pb; a < N; ++a) l[a] = quotient<T>(l[a], piv, r);
      const bool below = ti > pp, right = tj > pp, column = tj == pp;
#pragma unroll
      for (int a = pb; a < N; ++a)
        if (column && (a > pb || below)) acc[a][pb] = l[a];
      if (!below) l[pb] = (T)0;
      if (!right) u[pb] = (T)0;
      if constexpr (RHS) {
        const T wp = lane_value(ww[pb], pp);
#pragma unroll
        for (int a = pb; a < N; ++a) ww[a] = fmadd(-l[a], wp, ww[a]);
      }
#pragma unroll
      for (int b = pb; b < N; ++b)
#pragma unroll
        for (int a = pb; a < N; ++a) acc[a][b] = fmadd(-l[a], u[b], acc[a][b]);
    }
  }
#pragma unroll
  for (int b = 0; b < N; ++b)
    if (b >= off) {
      const int j = tj + 8 * (b - off);
#pragma unroll
      for (int a = 0; a < N; ++a)
        if (a >= off) {
          const int i = ti + 8 * (a - off);
          if (i < m && j < m) {
            *front_place(i, j, k, m, fo, co) = acc[a][b];
            if (j < k && i > j) g.add((double)acc[a][b]);
          }
        }
    }
  if constexpr (RHS) {
    // back to lane = row: row i is held by lane i % 8 (any tj) in ww[i / 8]
    const int row = lane & 31;
    T v = (T)0;
#pragma unroll
    for (int a = 0; a < N; ++a)
      if (a >= off) {
        const T x = from_lane(ww[a], 4 * (row & 7));
        if ((row >> 3) == a - off) v = x;
      }
    w = v;
  }
}

struct FrontArgs {
  const FrontDesc* fronts;  // in the order of FrontProgram::order
  const FrontInst* inst;
  const int4* task;
  const int32_t* level;
  const int32_t* idx;
  const uint16_t* apos;
  const uint16_t* cpos;
  const uint16_t* vtab;
  const int32_t* asrc;
  const int32_t* sg_src;
  const int32_t* sg_div;
  const int32_t* rs_ptr;
  const int32_t* rs_rhs;
  const int2* row_single;
  const int4* col_single;
  int n_sg, n_rs, n_cs;
};

__device__ __forceinline__ bool finite(double v) { return fabs(v) <= 1.7976931348623157e308; }

// Right-hand side of one permuted row in the solve's precision.
template <typename T>
__device__ __forceinline__ T rhs_value(const double* __restrict__ rhs, int i, double scale) {
  const T v = (T)rhs[i];
  return scale == -1.0 ? -v : v;
}

// Before a refactorisation that carries a right-hand side along: the
// singletons' values, and every row's right-hand side less the row singletons'
// columns, in permuted order, so that a front reads its part in one step.
template <typename T>
__global__ void __launch_bounds__(256)
    k_front_prep(FrontArgs A, int n, int n_rs_entries, const double* __restrict__ csr, T* sg,
                 const int32_t* __restrict__ p, const double* __restrict__ rhs, double scale, T* y,
                 DevStatus* st) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  Growth g;
  unsigned int bad_in = 0;
  if (i < n) {
    T v = rhs_value<T>(rhs, p[i], scale);
    for (int e = A.rs_ptr[i], e1 = A.rs_ptr[i + 1]; e < e1; ++e) {
      const double a = csr[A.sg_src[e]];
      if (!finite(a)) ++bad_in;
      const T l = (T)a / (T)csr[A.sg_div[e]];
      g.add((double)l);
      sg[e] = l;
      v = fmadd(-l, rhs_value<T>(rhs, A.rs_rhs[e], scale), v);
    }
    y[i] = v;
  }
  // the other singletons' values
  for (int e = n_rs_entries + i; e < A.n_sg; e += (int)gridDim.x * 256) {
    const double a = csr[A.sg_src[e]];
    if (!finite(a)) ++bad_in;
    sg[e] = (T)a;
  }
  if (st) {
    block_flags(dbits(g.mag), 0, g.bad, &st->maxl_bits, nullptr, &st->nonfinite);
    __syncthreads();
    block_flags(0, 0, bad_in, nullptr, nullptr, &st->nonfinite_in);
  }
}

// A front's right-hand side, lane = row: prepared values for its pivots, and
// the children's contributions.
template <typename T>
__device__ __forceinline__ T front_rhs(const FrontArgs& A, const FrontDesc& d, const FrontInst& I,
                                       int lane, int row, const T* y, const T* cv) {
  T v = lane < d.k ? y[row] : (T)0;
  const uint16_t* vt = A.vtab + d.vtab + lane;
  const T* src = cv + I.cv + d.v0;
  for (int c0 = 0; c0 < d.nv; c0 += 4) {
    int at[4];
    T w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      at[u] = (lane < d.m && c0 + u < d.nv) ? vt[(c0 + u) * d.m] : kNoPos;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (at[u] != kNoPos) w[u] = src[at[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (at[u] != kNoPos) v += w[u];
  }
  return v;
}

// Stage 0 of the refactorisation: workgroup = task, one wavefront per front of
// its levels; the workgroups from n_task on take the singletons' values.  RHS:
// the forward solve goes along -- a front's columns of L are in LDS when it
// ends, so its rows of y (k_front_prep's right-hand sides, then the solve's)
// and its contributions cost a multiply-add per pivot and no memory round of
// their own (the forward solve by itself, a launch per stage: 93 us at 65k
// gates).
template <typename T, bool RHS>
__global__ void __launch_bounds__(64 * kWaves)
    k_front_small(FrontArgs A, int task0, int n_task, int lds_wave, const double* __restrict__ csr,
                  T* fac, T* sg, T* cb, DevStatus* st, T* y, T* cv) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  Growth g;
  unsigned int bad_in = 0;
  if ((int)blockIdx.x >= n_task) {
    const int i = ((int)blockIdx.x - n_task) * (64 * kWaves) + (int)threadIdx.x;
    if (i < A.n_sg) {
      const double x = csr[A.sg_src[i]];
      const int dv = A.sg_div[i];
      T v = (T)x;
      if (!finite(x)) bad_in = 1;
      if (dv >= 0) {
        v = v / (T)csr[dv];
        g.add((double)v);
      }
      sg[i] = v;
    }
  } else {
    T* F = reinterpret_cast<T*>(lds_raw) + wave * lds_wave;
    const int4 tk = A.task[task0 + blockIdx.x];
    const FrontInst I = A.inst[tk.x];
    constexpr int NA = 4, NB = 8;
    // the front's description and its entries' indices are loaded while the
    // wavefront's previous front is eliminated, so a front waits for one
    // round of loads: its entries, and its children's values
    FrontDesc d;
    int ix[NA], pa[NA];
    int ready = -1;  // the front that d, ix and pa are for
    auto entries = [&](int e0) {
#pragma unroll
      for (int u = 0; u < NA; ++u)
        if (e0 + 64 * u < d.na) {
          ix[u] = A.asrc[d.a0 + I.asrc + e0 + 64 * u];
          pa[u] = A.apos[d.a0 + e0 + 64 * u];
        }
    };
    const int lend = tk.y + tk.z;
    for (int lv = tk.y; lv < lend; ++lv) {
      const int o1 = A.level[lv + 1];
      for (int o = A.level[lv] + wave; o < o1; o += kWaves) {
        if (ready != o) {
          d = A.fronts[o];
          entries(lane);
        }
        const int k = d.k, m = d.m, nt = d.nt, ld = front_ld(nt);
        const uint16_t* cpos = A.cpos + d.cpos;
        const T* src = cb + I.cb + d.c0;
        T* fo = fac + I.fac + d.fac;
        T* co = cb + I.cb + d.cb;
        int pc[NB];
        T vc[NB];
        auto children = [&](int e0) {
#pragma unroll
          for (int u = 0; u < NB; ++u) {
            pc[u] = kNoPos;
            if (e0 + 64 * u < d.nc) {
              pc[u] = cpos[e0 + 64 * u];
              vc[u] = src[e0 + 64 * u];
            }
          }
        };
        children(lane);
        const int row = I.row + d.r0 + lane;
        T w = (T)0;
        if constexpr (RHS) w = front_rhs<T>(A, d, I, lane, row, y, cv);
        T* cvo = cv + I.cv + d.cv;
        double v[NA];
#pragma unroll
        for (int u = 0; u < NA; ++u)
          if (lane + 64 * u < d.na) v[u] = csr[ix[u]];
        for (int e = lane, tot = front_lds(nt); e < tot; e += 64) F[e] = (T)0;
        for (int e0 = lane; e0 < d.na;) {
#pragma unroll
          for (int u = 0; u < NA; ++u)
            if (e0 + 64 * u < d.na) {
              if (!finite(v[u])) ++bad_in;
              F[pa[u]] = (T)v[u];
            }
          e0 += 64 * NA;
          entries(e0);
#pragma unroll
          for (int u = 0; u < NA; ++u)
            if (e0 + 64 * u < d.na) v[u] = csr[ix[u]];
        }
        // children's update blocks, 64 values at a time in the program's
        // order (no position twice in a group): LDS adds need no round trip,
        // and a wavefront's run in order, so the sums are fixed
        for (int e0 = lane; e0 < d.nc; e0 += 64 * NB) {
#pragma unroll
          for (int u = 0; u < NB; ++u)
            if (pc[u] != kNoPos)
              __hip_atomic_fetch_add(&F[pc[u] & kPosMask], vc[u], __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
          children(e0 + 64 * NB);
        }
        wave_sync();
        // the wavefront's next front: in this level, or first of the next
        int on = o + kWaves;
        if (on >= o1 && lv + 1 < lend) {
          on = o1 + wave;
          if (on >= A.level[lv + 2]) on = -1;
        } else if (on >= o1) {
          on = -1;
        }
        ready = on;
        if (on >= 0) {
          d = A.fronts[on];
          entries(lane);
        }
        front_eliminate<RHS, T>(k, m, kSmallTiles - nt, ld, F, lane, fo, co, w, g);
        if constexpr (RHS) {
          if (lane < k)
            y[row] = w;
          else if (lane < m)
            cvo[lane - k] = w;
        }
        wave_sync();
      }
      __syncthreads();  // the next level reads this one's update blocks
    }
  }
  if (st) {
    block_flags(dbits(g.mag), 0, g.bad, &st->maxl_bits, nullptr, &st->nonfinite);
    __syncthreads();
    block_flags(0, 0, bad_in, nullptr, nullptr, &st->nonfinite_in);
  }
}

// A later stage: one front of up to 64 rows per workgroup (or a chain of
// them).  256 threads hold the front as 32 rows x 8 columns of threads with 2 x
// 8 values each, aligned to the last row and column (the front is the lower
// right corner of a 64 x 64 matrix; rows and columns before it are not
// touched).  A pivot's row and column go through LDS with one barrier; the
// loop over its 8-column block is unrolled so that finished columns drop out.
// One wavefront per front took 0.45 us per pivot at 56 rows (83 FP64
// operations and 28 cross-lane reads in one instruction stream, about 1 000
// cycles); here a thread does at most 33 operations.
template <typename T, bool RHS>
__global__ void __launch_bounds__(256)
    k_front_large(FrontArgs A, int task0, const double* __restrict__ csr, T* fac, T* cb,
                  DevStatus* st, T* y, T* cv) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ __align__(16) T colbuf[2][64][2], rowbuf[2][65][2];  // by pivot of the pair
  __shared__ T vbuf[64];
  T* F = reinterpret_cast<T*>(lds_raw);
  const int tid = (int)threadIdx.x;
  const int ti = tid & 31, tj = tid >> 5;
  Growth g;
  unsigned int bad_in = 0;
  const int4 tk = A.task[task0 + blockIdx.x];
  const FrontInst I = A.inst[tk.x];
  int par = 0;
  const int oend = tk.w + tk.z;  // one front per level
  for (int o = tk.w; o < oend; ++o) {
    const FrontDesc d = A.fronts[o];
    const int k = d.k, m = d.m, ld = front_ld(d.nt), off = 8 - d.nt;
    const int pad = 8 * off;  // rows and columns before the front
    // All loads at once: entries' indices and children's values (about 0.6 us
    // away each), then the entries.  Taking the children one after another,
    // map and values, cost 2.2 us per child.
    constexpr int NB = 8;
    const T* src = cb + I.cb + d.c0;
    int ix = 0, pa0 = 0, pc[NB];
    T vc[NB];
    if (tid < d.na) {
      ix = A.asrc[d.a0 + I.asrc + tid];
      pa0 = A.apos[d.a0 + tid];
    }
#pragma unroll
    for (int u = 0; u < NB; ++u)
      if (tid + 256 * u < d.nc) {
        pc[u] = A.cpos[d.cpos + tid + 256 * u];
        vc[u] = src[tid + 256 * u];
      }
    if constexpr (RHS) {
      if (tid < 64) vbuf[tid] = front_rhs<T>(A, d, I, tid, I.row + d.r0 + tid, y, cv);
    }
    for (int e = tid, tot = front_lds(d.nt); e < tot; e += 256) F[e] = (T)0;
    T v0 = (T)0;
    if (tid < d.na) {
      const double v = csr[ix];
      if (!finite(v)) ++bad_in;
      v0 = (T)v;
    }
    lds_barrier();
    if (tid < d.na) F[pa0] = v0;
    for (int e = tid + 256; e < d.na; e += 256) {
      const double v = csr[A.asrc[d.a0 + I.asrc + e]];
      if (!finite(v)) ++bad_in;
      F[A.apos[d.a0 + e]] = (T)v;
    }
    lds_barrier();
    // A position's values in the children's order: round c adds the c-th of
    // each (its number is in the position's upper bits), so a round meets no
    // position twice and the sums are fixed.  Children one after another, a
    // barrier each, took 1 000 cycles a child; two or three rounds do.
    // (A front with more children on one position than there are numbers, a
    // bus of many blocks, is summed by one wavefront in the program's order.)
    if (d.rounds > kMaxRounds) {
      for (int e = tid; tid < 64 && e < d.nc; e += 64) {
        const int at = A.cpos[d.cpos + e];
        if (at != kNoPos)
          __hip_atomic_fetch_add(&F[at & kPosMask], src[e], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      lds_barrier();
    }
    for (int c = 0; d.rounds <= kMaxRounds && c < d.rounds; ++c) {
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (256 * u < d.nc && tid + 256 * u < d.nc && (pc[u] >> kPosBits) == c)
          __hip_atomic_fetch_add(&F[pc[u] & kPosMask], vc[u], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      for (int e = 256 * NB + tid; e < d.nc; e += 256) {
        const int at = A.cpos[d.cpos + e];
        if ((at >> kPosBits) == c)
          __hip_atomic_fetch_add(&F[at & kPosMask], src[e], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      lds_barrier();
    }
    T acc[2][8];
    const int i0 = ti - pad, i1 = ti + 32 - pad;  // the thread's rows in the front
    T w0 = (T)0, w1 = (T)0;                       // their right-hand sides
    if constexpr (RHS) {
      if (i0 >= 0) w0 = vbuf[i0];
      if (i1 >= 0) w1 = vbuf[i1];
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int j = tj + 8 * b - pad;
      acc[0][b] = (j >= 0 && i0 >= 0) ? F[i0 + j * ld] : (T)0;
      acc[1][b] = (j >= 0 && i1 >= 0) ? F[i1 + j * ld] : (T)0;
    }
#pragma unroll
    for (int pb = 0; pb < 8; ++pb) {
      constexpr int kHalf = 4;  // column blocks per 32 rows
      const int k0 = k - 8 * (pb - off);
      if (pb < off || k0 <= 0) continue;
      const int pn = k0 < 8 ? k0 : 8;
      const int pa = pb / kHalf;  // the pivots' row half
      // Two pivots at a time: one barrier for both; every thread brings the
      // second pivot's row and column up to date for itself (a 41-pivot front's
      // stage 22.2 us one at a time, 20.2 us in pairs; the loop is bound by
      // FP64 issue, about 6 cycles an operation for one wavefront per SIMD).
      for (int pp = 0; pp < pn; pp += 2) {
        const int p = 8 * pb + pp;
        const bool two = pp + 1 < pn;
        if (tj - pp == 0 || tj - pp == 1) {
          T* c = &colbuf[par][0][0] + (tj - pp);
          c[2 * (ti + 32)] = acc[1][pb];
          if (pa == 0) c[2 * ti] = acc[0][pb];
        }
        const int tr = ti - (p & 31);
        if (tr == 0 || tr == 1) {
          T* c = &rowbuf[par][0][0] + tr;
#pragma unroll
          for (int b = pb; b < 8; ++b) c[2 * (tj + 8 * b)] = acc[pa][b];
          if (RHS && tj == 0) c[2 * 64] = pa == 0 ? w0 : w1;
        }
        lds_barrier();
        const T a00 = rowbuf[par][p][0], a10 = rowbuf[par][p][1];
        const T a01 = rowbuf[par][p + 1][0];
        T a11 = rowbuf[par][p + 1][1];
        // columns (rows ti and ti + 32) and rows of the two pivots
        T c0[2], c1[2], u0[8], u1[8];
#pragma unroll
        for (int a = pa; a < 2; ++a) {
          c0[a] = colbuf[par][ti + 32 * a][0];
          c1[a] = colbuf[par][ti + 32 * a][1];
        }
#pragma unroll
        for (int b = pb; b < 8; ++b) {
          u0[b] = rowbuf[par][tj + 8 * b][0];
          u1[b] = rowbuf[par][tj + 8 * b][1];
        }
        const T r0 = reciprocal(a00);
        const T l10 = quotient<T>(a10, a00, r0);
        a11 = fmadd(-l10, a01, a11);
        const T r1 = reciprocal(a11);
#pragma unroll
        for (int a = pa; a < 2; ++a) {
          c0[a] = quotient<T>(c0[a], a00, r0);
          c1[a] = fmadd(-c0[a], a01, c1[a]);
          c1[a] = two ? quotient<T>(c1[a], a11, r1) : (T)0;
        }
#pragma unroll
        for (int b = pb; b < 8; ++b) u1[b] = fmadd(-l10, u0[b], u1[b]);
        // rows up to a pivot and columns up to it stay
        if (tj <= pp) u0[pb] = (T)0;
        if (tj <= pp + 1) u1[pb] = (T)0;
        T wp = (T)0, wq = (T)0;
        if constexpr (RHS) {
          wp = rowbuf[par][64][0];
          wq = fmadd(-l10, wp, rowbuf[par][64][1]);
        }
#pragma unroll
        for (int a = pa; a < 2; ++a) {
          const int i = ti + 32 * a;
          const T l0 = i > p ? c0[a] : (T)0, l1 = i > p + 1 ? c1[a] : (T)0;
#pragma unroll
          for (int b = pb; b < 8; ++b) {
            acc[a][b] = fmadd(-l0, u0[b], acc[a][b]);
            acc[a][b] = fmadd(-l1, u1[b], acc[a][b]);
          }
          if (tj == pp && i > p) acc[a][pb] = c0[a];
          if (two && tj == pp + 1 && i > p + 1) acc[a][pb] = c1[a];
          if constexpr (RHS) {
            T& w = a ? w1 : w0;
            w = fmadd(-l0, wp, w);
            if (two) w = fmadd(-l1, wq, w);
          }
        }
        par ^= 1;
      }
    }
    if constexpr (RHS) {
      if (tj == 0) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const int i = a ? i1 : i0;
          if (i < 0 || i >= m) continue;
          if (i < k)
            y[I.row + d.r0 + i] = a ? w1 : w0;
          else
            cv[I.cv + d.cv + i - k] = a ? w1 : w0;
        }
      }
    }
    T* fo = fac + I.fac + d.fac;
    T* co = cb + I.cb + d.cb;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (b < off) continue;
      const int j = tj + 8 * b - pad;
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        if (a == 0 && off >= 4) continue;  // no rows in the upper half
        const int i = a ? i1 : i0;
        if (i < 0 || i >= m || j >= m) continue;
        *front_place(i, j, k, m, fo, co) = acc[a][b];
        if (j < k && i > j) g.add((double)acc[a][b]);
      }
    }
    if (o + 1 < oend) __syncthreads();  // the chain's next front reads the block
  }
  if (st) {
    block_flags(dbits(g.mag), 0, g.bad, &st->maxl_bits, nullptr, &st->nonfinite);
    __syncthreads();
    block_flags(0, 0, bad_in, nullptr, nullptr, &st->nonfinite_in);
  }
}

// Right-hand side of a permuted row less the row singletons' columns.
template <typename T>
__device__ __forceinline__ T core_rhs(const FrontArgs& A, int row, const T* sg, const int32_t* p,
                                      const double* rhs, double scale) {
  T v = rhs_value<T>(rhs, p[row], scale);
  for (int e = A.rs_ptr[row], e1 = A.rs_ptr[row + 1]; e < e1; ++e)
    v = fmadd(-sg[e], rhs_value<T>(rhs, A.rs_rhs[e], scale), v);
  return v;
}

// The forward solve of one task, lane = row of the front: right-hand side
// (row_rhs), the children's contributions, then the pivots
// one after another (the columns of L are loaded eight at a time, ahead of the
// chain).
template <int W, typename T, typename Rhs>
__device__ __forceinline__ void task_fwd(const FrontArgs& A, const int4& tk, const T* fac,
                                         Rhs row_rhs, T* y, T* cv) {
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const FrontInst I = A.inst[tk.x];
  for (int lv = tk.y; lv < tk.y + tk.z; ++lv) {
    const int o1 = A.level[lv + 1];
    for (int o = A.level[lv] + wave; o < o1; o += W) {
      const FrontDesc d = A.fronts[o];
      const int k = d.k, m = d.m;
      const T* f = fac + I.fac + d.fac;
      const int row = I.row + d.r0 + lane;
      T v = (T)0;
      if (lane < k) v = row_rhs(row);
      const uint16_t* vt = A.vtab + d.vtab + lane;
      const T* src = cv + I.cv + d.v0;
      for (int c0 = 0; c0 < d.nv; c0 += 4) {
        int at[4];
        T w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) at[u] = (lane < m && c0 + u < d.nv) ? vt[(c0 + u) * m] : kNoPos;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (at[u] != kNoPos) w[u] = src[at[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (at[u] != kNoPos) v += w[u];
      }
      for (int p0 = 0; p0 < k; p0 += 8) {
        T l[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          l[u] = (p0 + u < k && lane > p0 + u && lane < m) ? f[(p0 + u) * m + lane] : (T)0;
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (p0 + u < k) v = fmadd(-l[u], lane_value(v, p0 + u), v);
      }
      if (lane < k)
        y[row] = v;
      else if (lane < m)
        cv[I.cv + d.cv + lane - k] = v;
    }
    __syncthreads();
  }
}

// The backward solve of one task: the update rows' solutions first (columns of
// U from the last), then the pivots from the last.
template <int W, typename T>
__device__ __forceinline__ void task_bwd(const FrontArgs& A, const int4& tk, const T* fac,
                                         const int32_t* q, const T* y, T* z, double* x) {
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const FrontInst I = A.inst[tk.x];
  for (int lv = tk.y + tk.z - 1; lv >= tk.y; --lv) {
    const int o1 = A.level[lv + 1];
    for (int o = A.level[lv] + wave; o < o1; o += W) {
      const FrontDesc d = A.fronts[o];
      const int k = d.k, m = d.m;
      const T* f = fac + I.fac + d.fac;
      const int row = I.row + d.r0 + lane;
      T v = (T)0, piv = (T)1;
      int col = 0;
      if (lane < k) {
        v = y[row];
        piv = f[lane * m + lane];
        col = q[row];
      } else if (lane < m) {
        v = z[I.row + A.idx[d.idx + lane - k]];
      }
      const T r = reciprocal(piv);
      const T* f2 = f + k * m;
      // Columns from the last, N at a time; the next N, and at the start the
      // pivots' own last N, are in flight meanwhile (one round of loads after
      // another was most of a large front's 7 us).
      constexpr int N = 8;
      T c[2][N], e[2][N];
      auto load_u = [&](T(&w)[N], int j0) {  // update rows' columns j0, j0 - 1, ...
#pragma unroll
        for (int t = 0; t < N; ++t)
          if (j0 - t >= k) w[t] = lane < k ? f2[(j0 - t - k) * k + lane] : (T)0;
      };
      auto load_p = [&](T(&w)[N], int j0) {  // pivots' columns
#pragma unroll
        for (int t = 0; t < N; ++t)
          if (j0 - t >= 0) w[t] = lane < j0 - t ? f[(j0 - t) * m + lane] : (T)0;
      };
      auto step_u = [&](const T(&w)[N], int j0) {
#pragma unroll
        for (int t = 0; t < N; ++t)
          if (j0 - t >= k) v = fmadd(-w[t], lane_value(v, j0 - t), v);
      };
      auto step_p = [&](const T(&w)[N], int j0) {
#pragma unroll
        for (int t = 0; t < N; ++t)
          if (j0 - t >= 0) {
            const T xq = quotient<T>(v, piv, r);
            const T xj = lane_value(xq, j0 - t);
            v = lane == j0 - t ? xq : fmadd(-w[t], xj, v);
          }
      };
      load_u(c[0], m - 1);
      load_p(e[0], k - 1);
      for (int j0 = m - 1; j0 >= k; j0 -= 2 * N) {
        if (j0 - N >= k) load_u(c[1], j0 - N);
        step_u(c[0], j0);
        if (j0 - N < k) break;
        if (j0 - 2 * N >= k) load_u(c[0], j0 - 2 * N);
        step_u(c[1], j0 - N);
      }
      for (int j0 = k - 1; j0 >= 0; j0 -= 2 * N) {
        if (j0 - N >= 0) load_p(e[1], j0 - N);
        step_p(e[0], j0);
        if (j0 - N < 0) break;
        if (j0 - 2 * N >= 0) load_p(e[0], j0 - 2 * N);
        step_p(e[1], j0 - N);
      }
      if (lane < k) {
        z[row] = v;
        x[col] = (double)v;
      }
    }
    __syncthreads();
  }
}

// One stage of the forward solve; the workgroups from n_task on (first stage)
// keep the singletons' right-hand sides, so that x may be the right-hand
// side's buffer: nothing reads it after the last forward stage, nothing writes
// x before.
template <typename T>
__global__ void __launch_bounds__(64 * kWaves)
    k_front_fwd(FrontArgs A, int task0, int n_task, const T* __restrict__ fac,
                const T* __restrict__ sg, const int32_t* __restrict__ p,
                const double* __restrict__ rhs, double scale, T* y, T* cv) {
  if ((int)blockIdx.x >= n_task) {
    const int i = ((int)blockIdx.x - n_task) * (64 * kWaves) + (int)threadIdx.x;
    if (i < A.n_rs + A.n_cs) {
      const int r = i < A.n_rs ? A.row_single[i].x : A.col_single[i - A.n_rs].x;
      y[r] = rhs_value<T>(rhs, p[r], scale);
    }
    return;
  }
  task_fwd<kWaves, T>(A, A.task[task0 + blockIdx.x], fac,
                      [&](int row) { return core_rhs<T>(A, row, sg, p, rhs, scale); }, y, cv);
}

// One stage of the backward solve; the workgroups from n_task on (last launch)
// solve the row singletons.
template <typename T>
__global__ void __launch_bounds__(64 * kWaves)
    k_front_bwd(FrontArgs A, int task0, int n_task, const T* __restrict__ fac,
                const T* __restrict__ sg, const int32_t* __restrict__ q, const T* __restrict__ y,
                T* z, double* x) {
  if ((int)blockIdx.x >= n_task) {
    const int i = ((int)blockIdx.x - n_task) * (64 * kWaves) + (int)threadIdx.x;
    if (i < A.n_rs) {
      const int2 rs = A.row_single[i];
      x[q[rs.x]] = (double)(y[rs.x] / sg[rs.y]);
    }
    return;
  }
  task_bwd<kWaves, T>(A, A.task[task0 + blockIdx.x], fac, q, y, z, x);
}

// Sum of the U entries [e0, e1) (at most kHubChunk) times x by threads 0 ..
// 255: strided partials, then a halving tree.  Every thread of the workgroup
// calls; the result is thread 0's.
template <typename T>
__device__ __forceinline__ T single_chunk(int b0, int b1, int us_first, const int32_t* us_col,
                                          const T* sg, const double* x, T* red) {
  const int tid = (int)threadIdx.x;
  T acc = (T)0;
  if (tid < 256) {
    for (int e0 = b0 + tid; e0 < b1; e0 += 4 * 256) {
      T a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + 256 * u < b1) {
          a[u] = sg[e0 + 256 * u];
          b[u] = (T)x[us_col[e0 + 256 * u - us_first]];
        }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + 256 * u < b1) acc = fmadd(a[u], b[u], acc);
    }
    red[tid] = acc;
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  return red[0];
}

// The column singletons after the solve: x = (b - sum of the row's U entries
// times x) / pivot, the sums in chunks of kHubChunk entries, one workgroup
// each (256 strided partials, halving tree); the workgroup that finishes a
// row's last chunk adds the chunks in order (the supply rail's row: 32 of
// them on a 65k-gate circuit) and leaves the row's counter at zero.
template <typename T>
__global__ void __launch_bounds__(256)
    k_front_single(const int4* __restrict__ chunk, const int4* __restrict__ single, int us_first,
                   const int32_t* __restrict__ us_col, const T* __restrict__ sg,
                   const int32_t* __restrict__ q, const T* __restrict__ y, T* part,
                   unsigned int* count, double* x) {
  __shared__ T red[256];
  __shared__ int s_last;
  const int tid = (int)threadIdx.x;
  const int4 ch = chunk[blockIdx.x];
  const int4 sn = single[ch.x];
  T total = single_chunk(ch.y, ch.z, us_first, us_col, sg, x, red);
  const int nch = ch.w;
  const int first = (int)blockIdx.x - (ch.y - sn.z) / kHubChunk;  // the row's first chunk
  if (nch > 1) {
    if (tid == 0) {
      __hip_atomic_store(&part[blockIdx.x], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned int old = __hip_atomic_fetch_add(&count[ch.x], 1u, __ATOMIC_ACQ_REL,
                                                      __HIP_MEMORY_SCOPE_AGENT);
      s_last = old == (unsigned int)(nch - 1);
      if (s_last)
        __hip_atomic_store(&count[ch.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;  // uniform across the block
    if (tid < 64) {
      total = (T)0;
      for (int c0 = 0; c0 < nch; c0 += 64) {
        T v = (T)0;
        if (c0 + tid < nch)
          v = __hip_atomic_load(&part[first + c0 + tid], __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
        const int n = nch - c0 < 64 ? nch - c0 : 64;
        for (int c = 0; c < n; ++c) total += lane_value(v, c);
      }
    }
  }
  if (tid == 0) x[q[sn.x]] = (double)((y[sn.x] - total) / sg[sn.y]);
}

// A system with one task in one launch: factors (mode 1), solves (mode 2) or
// both (3) from LDS.  Everything the levels read is loaded first, all at once,
// so the workgroup waits for memory twice (index, value) and not at every
// level.
template <typename T>
__global__ void __launch_bounds__(64 * kTinyWaves)
    k_front_tiny(FrontArgs A, FrontProgram::Tiny S, int mode, const double* __restrict__ csr,
                 T* fac, T* sg, DevStatus* st, const int32_t* __restrict__ p,
                 const int32_t* __restrict__ q, const double* rhs, double scale, double* x,
                 int us_first, const int32_t* __restrict__ us_col) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ T red[256];
  const int tid = (int)threadIdx.x;
  constexpr int nthr = 64 * kTinyWaves;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  FrontDesc* desc = reinterpret_cast<FrontDesc*>(lds_raw + S.desc);
  int32_t* level = reinterpret_cast<int32_t*>(lds_raw + S.level);
  T* lf = reinterpret_cast<T*>(lds_raw + S.fac);
  T* lsg = reinterpret_cast<T*>(lds_raw + S.sg);
  const int4 tk = A.task[0];
  const FrontInst I = A.inst[tk.x];
  Growth g;
  unsigned int bad_in = 0;
  constexpr int kDescInts = (int)(sizeof(FrontDesc) / sizeof(int32_t));
  for (int i = tid; i < S.n_fronts * kDescInts; i += nthr)
    reinterpret_cast<int32_t*>(desc)[i] = reinterpret_cast<const int32_t*>(A.fronts)[i];
  for (int i = tid; i < S.n_level; i += nthr) level[i] = A.level[tk.y + i];
  T* y = reinterpret_cast<T*>(lds_raw + S.y);
  if (mode & 2)  // right-hand sides; the row singletons' part follows below
    for (int r = tid; r < S.n_rows; r += nthr) y[r] = rhs_value<T>(rhs, p[r], scale);
  int32_t* idx = reinterpret_cast<int32_t*>(lds_raw + S.idx);
  uint16_t* vtab = reinterpret_cast<uint16_t*>(lds_raw + S.vtab);
  T* cv = reinterpret_cast<T*>(lds_raw + S.cv);
  T* z = reinterpret_cast<T*>(lds_raw + S.z);
  FrontArgs B = A;  // the tables in LDS
  B.fronts = desc;
  B.level = level - tk.y;
  B.idx = idx;
  B.vtab = vtab;
  if (mode & 2) {
    for (int i = tid; i < S.n_idx; i += nthr) idx[i] = A.idx[i];
    for (int i = tid; i < S.n_vtab; i += nthr) vtab[i] = A.vtab[i];
  }
  auto core = [&]() {  // the row singletons' part of the right-hand sides
    for (int r = tid; r < S.n_rows; r += nthr) {
      T v = y[r];
      for (int e = A.rs_ptr[r], e1 = A.rs_ptr[r + 1]; e < e1; ++e)
        v = fmadd(-lsg[e], rhs_value<T>(rhs, A.rs_rhs[e], scale), v);
      y[r] = v;
    }
    __syncthreads();
  };
  if (mode & 1) {
    double* av = reinterpret_cast<double*>(lds_raw + S.av);
    uint16_t* apos = reinterpret_cast<uint16_t*>(lds_raw + S.apos);
    uint16_t* cpos = reinterpret_cast<uint16_t*>(lds_raw + S.cpos);
    for (int i = tid; i < S.n_a; i += nthr) {
      const double v = csr[A.asrc[i]];
      if (!finite(v)) ++bad_in;
      av[i] = v;
      apos[i] = A.apos[i];
    }
    for (int i = tid; i < S.n_c; i += nthr) cpos[i] = A.cpos[i];
    for (int i = tid; i < A.n_sg; i += nthr) {
      const double v0 = csr[A.sg_src[i]];
      const int dv = A.sg_div[i];
      T v = (T)v0;
      if (!finite(v0)) ++bad_in;
      if (dv >= 0) {
        v = v / (T)csr[dv];
        g.add((double)v);
      }
      lsg[i] = v;
      sg[i] = v;
    }
    T* cb = reinterpret_cast<T*>(lds_raw + S.cb);
    T* F = reinterpret_cast<T*>(lds_raw + S.front) + wave * S.lds_wave;
    __syncthreads();
    if (mode & 2) core();
    for (int lv = 0; lv + 1 < S.n_level; ++lv) {
      for (int o = level[lv] + wave; o < level[lv + 1]; o += kTinyWaves) {
        const FrontDesc& d = desc[o];
        const int k = __builtin_amdgcn_readfirstlane(d.k);
        const int m = __builtin_amdgcn_readfirstlane(d.m);
        const int nt = __builtin_amdgcn_readfirstlane(d.nt);
        const int na = d.na, a0 = d.a0, nc = d.nc, cp = d.cpos, c0 = d.c0;
        const int ld = front_ld(nt);
        for (int e = lane, tot = front_lds(nt); e < tot; e += 64) F[e] = (T)0;
        for (int e = lane; e < na; e += 64) F[apos[a0 + e]] = (T)av[a0 + e];
        for (int e = lane; e < nc; e += 64) {
          const int at = cpos[cp + e];
          if (at != kNoPos)
            __hip_atomic_fetch_add(&F[at & kPosMask], cb[c0 + e], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        wave_sync();
        // a right-hand side in hand goes along, as in k_front_small
        T w = (T)0;
        const int row = I.row + d.r0 + lane;
        if (mode & 2) w = front_rhs<T>(B, d, I, lane, row, y, cv - I.cv);
        front_eliminate<true, T>(k, m, kSmallTiles - nt, ld, F, lane, lf + d.fac, cb + d.cb, w, g);
        if (mode & 2) {
          if (lane < k)
            y[row] = w;
          else if (lane < m)
            cv[d.cv + lane - k] = w;
        }
        wave_sync();
      }
      __syncthreads();
    }
    for (int i = tid; i < S.n_fac; i += nthr) fac[I.fac + i] = lf[i];
  } else {
    for (int i = tid; i < S.n_fac; i += nthr) lf[i] = fac[I.fac + i];
    for (int i = tid; i < A.n_sg; i += nthr) lsg[i] = sg[i];
  }
  if (mode & 2) {
    const T* f0 = lf - I.fac;  // block offsets: one block holds all fronts
    if (!(mode & 1)) {
      __syncthreads();
      core();
      task_fwd<kTinyWaves, T>(B, tk, f0, [&](int row) { return y[row]; }, y, cv - I.cv);
    }
    task_bwd<kTinyWaves, T>(B, tk, f0, q, y, z, x);
    for (int i = tid; i < A.n_rs; i += nthr) {
      const int2 rs = A.row_single[i];
      x[q[rs.x]] = (double)(y[rs.x] / lsg[rs.y]);
    }
    __syncthreads();
    for (int i = 0; i < A.n_cs; ++i) {
      const int4 sn = A.col_single[i];
      const T total = single_chunk(sn.z, sn.w, us_first, us_col, lsg, x, red);
      if (tid == 0) x[q[sn.x]] = (double)((y[sn.x] - total) / lsg[sn.y]);
      __syncthreads();
    }
  }
  if ((mode & 1) && st) {
    block_flags(dbits(g.mag), 0, g.bad, &st->maxl_bits, nullptr, &st->nonfinite);
    __syncthreads();
    block_flags(0, 0, bad_in, nullptr, nullptr, &st->nonfinite_in);
  }
}

inline int nblk(long long n, int b) { return (int)((n + b - 1) / b); }

FrontArgs front_args(const DevLU& L) {
  const DevFronts& D = L.front;
  const FrontProgram& F = L.sym.front;
  FrontArgs a;
  a.fronts = reinterpret_cast<const FrontDesc*>(D.fronts.p);
  a.inst = reinterpret_cast<const FrontInst*>(D.inst.p);
  a.task = reinterpret_cast<const int4*>(D.task.p);
  a.level = D.level.p;
  a.idx = D.idx.p;
  a.apos = D.apos.p;
  a.cpos = D.cpos.p;
  a.vtab = D.vtab.p;
  a.asrc = D.asrc.p;
  a.sg_src = D.sg_src.p;
  a.sg_div = D.sg_div.p;
  a.rs_ptr = D.rs_ptr.p;
  a.rs_rhs = D.rs_rhs.p;
  a.row_single = reinterpret_cast<const int2*>(D.row_single.p);
  a.col_single = reinterpret_cast<const int4*>(D.col_single.p);
  a.n_sg = (int)F.sg_src.size();
  a.n_rs = (int)F.row_single.size() / 2;
  a.n_cs = (int)F.col_single.size() / 4;
  return a;
}

template <typename T>
T* cb_of(DevLU& L);
template <>
double* cb_of<double>(DevLU& L) {
  return L.front.cb.p;
}
template <>
float* cb_of<float>(DevLU& L) {
  return reinterpret_cast<float*>(L.front.cb.p);
}

template <typename T>
void launch_tiny(DevLU& L, int mode, const double* csr, T* fac, DevStatus* st, const double* rhs,
                 double scale, double* x, hipStream_t s) {
  const FrontProgram& F = L.sym.front;
  ktimer_begin(s);
  k_front_tiny<T><<<1, 64 * kTinyWaves, (size_t)F.tiny.total, s>>>(
      front_args(L), F.tiny, mode, csr, fac, fac + F.n_fac, st, L.p.p, L.q.p, rhs, scale, x,
      F.us_first, L.front.us_col.p);
  ktimer_end(mode & 1 ? KC_LU_TASKS : KC_TRI_TASKS, s);
}

}  // namespace

// rhs (may be null): carried along; y then holds the forward solve
template <typename T>
static void run_refactor(DevLU& L, const double* csr, T* fac, DevStatus* st, const double* rhs,
                         double scale, T* y, hipStream_t s) {
  const FrontProgram& F = L.sym.front;
  const FrontArgs A = front_args(L);
  T* sg = fac + F.n_fac;
  T* cb = cb_of<T>(L);
  T* cv = reinterpret_cast<T*>(L.front.cv.p);
  const int ns = (int)F.stage_task.size() - 1;
  const int nsb = rhs ? 0 : nblk(A.n_sg, 64 * kWaves);
  if (rhs) {
    ktimer_begin(s);
    k_front_prep<T><<<nblk(L.sym.n, 256), 256, 0, s>>>(A, L.sym.n, (int)F.rs_rhs.size(), csr, sg,
                                                       L.p.p, rhs, scale, y, st);
    ktimer_end(KC_LU_GATHER, s);
  }
  for (int g = 0; g < std::max(ns, 1); ++g) {
    const int t0 = g < ns ? F.stage_task[g] : 0, nt = g < ns ? F.stage_task[g + 1] - t0 : 0;
    const int grid = nt + (g == 0 ? nsb : 0);
    if (grid == 0) continue;
    const int w = nt > 0 ? front_lds(F.stage_nt[g]) : 0;
    const size_t lds = sizeof(T) * (size_t)w;
    ktimer_begin(s);
    if (g == 0 && rhs)
      k_front_small<T, true><<<grid, 64 * kWaves, lds * kWaves, s>>>(A, t0, nt, w, csr, fac, sg, cb,
                                                                     st, y, cv);
    else if (g == 0)
      k_front_small<T, false><<<grid, 64 * kWaves, lds * kWaves, s>>>(A, t0, nt, w, csr, fac, sg,
                                                                      cb, st, y, cv);
    else if (rhs)
      k_front_large<T, true><<<grid, 256, lds, s>>>(A, t0, csr, fac, cb, st, y, cv);
    else
      k_front_large<T, false><<<grid, 256, lds, s>>>(A, t0, csr, fac, cb, st, y, cv);
    ktimer_end(KC_LU_TASKS, s);
  }
}

// The backward solve and the singletons, from y.
template <typename T>
static void run_backward(DevLU& L, const T* fac, double* x, const T* y, T* z, hipStream_t s) {
  const FrontProgram& F = L.sym.front;
  const FrontArgs A = front_args(L);
  const T* sg = fac + F.n_fac;
  T* part = reinterpret_cast<T*>(L.front.part.p);
  const int ns = (int)F.stage_task.size() - 1;
  const int nrb = nblk(A.n_rs, 64 * kWaves);
  for (int g = std::max(ns, 1) - 1; g >= 0; --g) {
    const int t0 = g < ns ? F.stage_task[g] : 0, nt = g < ns ? F.stage_task[g + 1] - t0 : 0;
    const int grid = nt + (g == 0 ? nrb : 0);
    if (grid == 0) continue;
    ktimer_begin(s);
    k_front_bwd<T><<<grid, 64 * kWaves, 0, s>>>(A, t0, nt, fac, sg, L.q.p, y, z, x);
    ktimer_end(KC_TRI_TASKS, s);
  }
  const int nch = (int)F.us_chunk.size() / 4;
  if (nch > 0) {
    ktimer_begin(s);
    k_front_single<T><<<nch, 256, 0, s>>>(reinterpret_cast<const int4*>(L.front.us_chunk.p),
                                          A.col_single, F.us_first, L.front.us_col.p, sg, L.q.p, y,
                                          part, L.front.count.p, x);
    ktimer_end(KC_TRI_HUB, s);
  }
}

template <typename T>
void launch_front_refactor(DevLU& L, const double* csr, T* fac, DevStatus* st, hipStream_t s) {
  if (L.sym.front.tiny.total) {
    launch_tiny<T>(L, 1, csr, fac, st, nullptr, 1.0, nullptr, s);
    return;
  }
  run_refactor<T>(L, csr, fac, st, nullptr, 1.0, nullptr, s);
}

template <typename T>
void launch_front_solve(DevLU& L, const T* fac, const double* rhs, double scale, double* x, T* y,
                        T* z, hipStream_t s) {
  const FrontProgram& F = L.sym.front;
  if (F.tiny.total) {
    launch_tiny<T>(L, 2, nullptr, const_cast<T*>(fac), nullptr, rhs, scale, x, s);
    return;
  }
  const FrontArgs A = front_args(L);
  const T* sg = fac + F.n_fac;
  T* cv = reinterpret_cast<T*>(L.front.cv.p);
  const int ns = (int)F.stage_task.size() - 1;
  const int nsb = nblk(A.n_rs + A.n_cs, 64 * kWaves);
  for (int g = 0; g < std::max(ns, 1); ++g) {
    const int t0 = g < ns ? F.stage_task[g] : 0, nt = g < ns ? F.stage_task[g + 1] - t0 : 0;
    const int grid = nt + (g == 0 ? nsb : 0);
    if (grid == 0) continue;
    ktimer_begin(s);
    k_front_fwd<T><<<grid, 64 * kWaves, 0, s>>>(A, t0, nt, fac, sg, L.p.p, rhs, scale, y, cv);
    ktimer_end(KC_TRI_TASKS, s);
  }
  run_backward<T>(L, fac, x, y, z, s);
}

template <typename T>
void launch_lu_factor_solve(DevLU& L, const double* csr, T* fac, DevStatus* st, const double* rhs,
                            double scale, double* x, T* y, T* z, hipStream_t s) {
  if (L.sym.front.on() && L.sym.front.tiny.total) {
    launch_tiny<T>(L, 3, csr, fac, st, rhs, scale, x, s);
    return;
  }
  if (L.sym.front.on()) {
    run_refactor<T>(L, csr, fac, st, rhs, scale, y, s);
    run_backward<T>(L, fac, x, y, z, s);
    return;
  }
  launch_lu_refactor<T>(L, csr, fac, st, s);
  launch_lu_solve<T>(L, fac, rhs, scale, x, y, z, s);
}

template void launch_lu_factor_solve<double>(DevLU&, const double*, double*, DevStatus*,
                                             const double*, double, double*, double*, double*,
                                             hipStream_t);
template void launch_lu_factor_solve<float>(DevLU&, const double*, float*, DevStatus*,
                                            const double*, double, double*, float*, float*,
                                            hipStream_t);
template void launch_front_refactor<double>(DevLU&, const double*, double*, DevStatus*, hipStream_t);
template void launch_front_refactor<float>(DevLU&, const double*, float*, DevStatus*, hipStream_t);
template void launch_front_solve<double>(DevLU&, const double*, const double*, double, double*,
                                         double*, double*, hipStream_t);
template void launch_front_solve<float>(DevLU&, const float*, const double*, double, double*,
                                        float*, float*, hipStream_t);

}  // namespace vjx
