/*
 * isk_tri.h -- the 1-D direct Poisson solve of one work-group and the electric
 * field of a node, used by the solver's own kernel and by the time loop's
 * field kernel of 1-D grids.
 */
#ifndef ISK_TRI_H
#define ISK_TRI_H

#include "isk_internal.h"

/* E = -grad phi at node n: central differences inside, one-sided at the ends */
__device__ __forceinline__ void efield_node(const double *phi, float *E, int dim, int nx, int ny,
                                            double dx, double dy, int n) {
  const int i = n % nx, j = n / nx;
  double ex;
  if (nx < 2) ex = 0.0;
  else if (i == 0) ex = (phi[n] - phi[n + 1]) / dx;
  else if (i == nx - 1) ex = (phi[n - 1] - phi[n]) / dx;
  else ex = (phi[n - 1] - phi[n + 1]) / (2.0 * dx);
  if (dim == 1) {
    E[n] = (float)ex;
    return;
  }
  double ey;
  if (ny < 2) ey = 0.0;
  else if (j == 0) ey = (phi[n] - phi[n + nx]) / dy;
  else if (j == ny - 1) ey = (phi[n - nx] - phi[n]) / dy;
  else ey = (phi[n - nx] - phi[n + nx]) / (2.0 * dy);
  E[2 * n] = (float)ex;
  E[2 * n + 1] = (float)ey;
}

struct TriArgs {
  const double *rho;
  const int8_t *tags;
  const double *tagval;
  const double *a, *cp, *inv;
  const double *ma, *ncp; /* the factored maps' slopes: -a inv and -cp */
  double *y, *phi;
  int n;
  double scale; /* dx^2 / eps0 */
  int singular;
};

/* one thread: rhs, forward elimination, back substitution (FP64, explicit fma) */
__device__ __forceinline__ void tri_solve_body(const TriArgs &t) {
  const int n = t.n;
  if (!t.singular) {
    double yprev = 0.0;
    for (int i = 0; i < n; ++i) {
      int tg = t.tags[i];
      double r = tg ? t.tagval[tg] : -(t.rho[i] * t.scale);
      double y = __builtin_fma(-t.a[i], yprev, r) * t.inv[i];
      t.y[i] = y;
      yprev = y;
    }
    double xn = 0.0;
    for (int i = n - 1; i >= 0; --i) {
      double x = __builtin_fma(-t.cp[i], xn, t.y[i]);
      t.phi[i] = x;
      xn = x;
    }
    return;
  }
  /* periodic ring without Dirichlet nodes: project, pin node 0, solve nodes 1..n-1 */
  double sum = 0.0;
  for (int i = 0; i < n; ++i) sum += -(t.rho[i] * t.scale);
  double mean = sum / (double)n;
  double yprev = 0.0;
  for (int i = 1; i < n; ++i) {
    double r = -(t.rho[i] * t.scale) - mean;
    double y = __builtin_fma(-t.a[i], yprev, r) * t.inv[i];
    t.y[i] = y;
    yprev = y;
  }
  double xn = 0.0;
  double s2 = 0.0;
  for (int i = n - 1; i >= 1; --i) {
    double x = __builtin_fma(-t.cp[i], xn, t.y[i]);
    t.phi[i] = x;
    xn = x;
  }
  t.phi[0] = 0.0;
  for (int i = 0; i < n; ++i) s2 += t.phi[i];
  double m2 = s2 / (double)n;
  for (int i = 0; i < n; ++i) t.phi[i] = t.phi[i] - m2;
}

/* The same system solved by a whole work-group for n <= TRI_BLOCK * TRI_K: with
 * Dirichlet nodes all n rows, on the periodic ring (singular) rows 1 .. n - 1 after
 * node 0 is pinned.
 * Both recurrences of the factored system are first-order affine maps,
 * forward y_i = A_i y_(i-1) + B_i with A_i = -a_i inv_i, B_i = r_i inv_i, and
 * backward x_i = C_i x_(i+1) + D_i with C_i = -cp_i, D_i = y_i, so each is a
 * prefix composition of maps, (A2, B2) after (A1, B1) = (A2 A1, fma(A2, B1,
 * B2)): every thread composes its TRI_K consecutive maps, a Hillis-Steele
 * scan over the TRI_BLOCK segment maps gives each segment its incoming value,
 * and every element is then one fma away.  log2(TRI_BLOCK) + 2 TRI_K
 * dependent steps instead of 3n.  The operations are fixed, so the oracle
 * restates them bit for bit.  For larger n thread 0 runs tri_solve_body. */
#define TRI_BLOCK 256
#define TRI_K 8

/* scratch of the scans and sums, two buffers each */
struct TriShared {
  double ga[2][TRI_BLOCK], gb[2][TRI_BLOCK];
};

/* one prefix composition of n affine maps (ma[i], mb[i]) applied to 0;
 * rev != 0 scans from the last element down.  out[i] = value at element i.
 * Up to 65 segments (n <= 520) the Hillis-Steele steps stay in wave 0 as
 * shuffles, the same compositions in the same order (the 65th segment only
 * needs the value that leaves the 64th): two barriers instead of eighteen. */
__device__ __forceinline__ void tri_scan(const double *ma, const double *mb, int n, int rev,
                                         double *out, TriShared &sh) {
  const int tid = threadIdx.x, j0 = tid * TRI_K;
  double la[TRI_K], lb[TRI_K];
  double ca = 1.0, cb = 0.0;
#pragma unroll
  for (int k = 0; k < TRI_K; ++k) {
    const int j = j0 + k;
    if (j < n) {
      const int i = rev ? n - 1 - j : j;
      const double A = ma[i], B = mb[i];
      cb = __builtin_fma(A, cb, B);
      ca = A * ca;
    }
    la[k] = ca;
    lb[k] = cb;
  }
  int cur = 0;
  if (n <= 65 * TRI_K) {
    if (tid < 64) {
      for (int d = 1; d < 64; d <<= 1) {
        const double pa = __shfl_up(ca, d), pb = __shfl_up(cb, d);
        if (tid >= d) {
          cb = __builtin_fma(ca, pb, cb);
          ca = ca * pa;
        }
      }
      sh.gb[0][tid] = cb;
    }
    __syncthreads();
  } else {
    const bool on = tid < TRI_BLOCK; /* the work-group may be wider */
    if (on) {
      sh.ga[0][tid] = ca;
      sh.gb[0][tid] = cb;
    }
    __syncthreads();
    for (int d = 1; d < TRI_BLOCK; d <<= 1) {
      if (on && tid >= d) {
        const double pa = sh.ga[cur][tid - d], pb = sh.gb[cur][tid - d];
        cb = __builtin_fma(ca, pb, cb);
        ca = ca * pa;
      }
      cur ^= 1;
      if (on) {
        sh.ga[cur][tid] = ca;
        sh.gb[cur][tid] = cb;
      }
      __syncthreads();
    }
  }
  const double vin = tid > 0 ? sh.gb[cur][min(tid - 1, n <= 65 * TRI_K ? 63 : TRI_BLOCK - 1)] : 0.0;
#pragma unroll
  for (int k = 0; k < TRI_K; ++k) {
    const int j = j0 + k;
    if (j < n) out[rev ? n - 1 - j : j] = __builtin_fma(la[k], vin, lb[k]);
  }
  __syncthreads(); /* out and the scratch are read or rewritten next */
}

/* sum of v[0..n) in a fixed order: each thread adds its TRI_K consecutive
 * elements, then a pairwise tree over the TRI_BLOCK partials, its last six
 * levels as shuffles of wave 0 (every thread returns the same bits) */
__device__ __forceinline__ double tri_sum(const double *v, int n, TriShared &sh) {
  const int tid = threadIdx.x, j0 = tid * TRI_K;
  double *g = sh.ga[0];
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < TRI_K; ++k)
    if (j0 + k < n) s += v[j0 + k];
  if (tid < TRI_BLOCK) g[tid] = s;
  __syncthreads();
  if (tid < 64) {
    double t = (g[tid] + g[tid + 128]) + (g[tid + 64] + g[tid + 192]);
    for (int d = 32; d > 0; d >>= 1) t += __shfl_down(t, d);
    if (tid == 0) sh.gb[0][0] = t;
  }
  __syncthreads();
  const double r = sh.gb[0][0];
  __syncthreads();
  return r;
}

/* grids the work-group solves; larger ones are one thread's (tri_solve_body) */
#define TRI_MAX (TRI_BLOCK * TRI_K)

/* LDS of the work-group solve */
struct TriWork {
  double A[TRI_MAX], B[TRI_MAX], C[TRI_MAX], y[TRI_MAX];
  TriShared sh;
};

/* the work-group solve of n <= TRI_MAX nodes, phi to t.phi and w.B (no barrier
 * after).  Before, ordered by a barrier: w.A and w.C the slopes of the two
 * scans' maps (ring: entry i - 1 of node i) and
 *  with Dirichlet nodes, w.B = r inv, r the node's value or -rho scale;
 *  on the periodic ring (A1/A2: right-hand side projected to zero mean, node 0
 *  pinned, rows 1..n-1 solved by the two scans, then the mean of phi removed,
 *  sums in tri_sum's order), w.y = -rho scale and w.B[i - 1] = inv of node i. */
__device__ __forceinline__ void tri_solve_lds(const TriArgs &t, TriWork &w) {
  const int n = t.n;
  if (t.singular) {
    const int m = n - 1;
    const double mean = tri_sum(w.y, n, w.sh) / (double)n;
    for (int j = threadIdx.x; j < m; j += blockDim.x) w.B[j] = (w.y[j + 1] - mean) * w.B[j];
    __syncthreads();
    tri_scan(w.A, w.B, m, 0, w.y, w.sh);
    tri_scan(w.C, w.y, m, 1, w.B, w.sh);
    /* phi over all n nodes in y: node 0 pinned at 0 */
    for (int i = threadIdx.x; i < n; i += blockDim.x) w.y[i] = i == 0 ? 0.0 : w.B[i - 1];
    __syncthreads();
    const double m2 = tri_sum(w.y, n, w.sh) / (double)n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      w.B[i] = w.y[i] - m2;
      t.phi[i] = w.B[i];
    }
    return;
  }
  tri_scan(w.A, w.B, n, 0, w.y, w.sh);
  tri_scan(w.C, w.y, n, 1, w.B, w.sh);
  for (int i = threadIdx.x; i < n; i += blockDim.x) t.phi[i] = w.B[i];
}

/* one node's part of that set-up */
__device__ __forceinline__ void tri_load(const TriArgs &t, TriWork &w, int i, double rho,
                                         double inv, double ma, double ncp, int tag) {
  if (t.singular) {
    w.y[i] = -(rho * t.scale);
    if (i > 0) {
      w.A[i - 1] = ma;
      w.B[i - 1] = inv;
      w.C[i - 1] = ncp;
    }
    return;
  }
  const double r = tag ? t.tagval[tag] : -(rho * t.scale);
  w.A[i] = ma;
  w.B[i] = r * inv;
  w.C[i] = ncp;
}

__device__ __forceinline__ void tri_solve_group(const TriArgs &t) {
  __shared__ TriWork w;
  if (t.n > TRI_MAX) {
    if (threadIdx.x == 0) tri_solve_body(t);
    return;
  }
  for (int i = threadIdx.x; i < t.n; i += blockDim.x)
    tri_load(t, w, i, t.rho[i], t.inv[i], t.ma[i], t.ncp[i], t.tags[i]);
  __syncthreads();
  tri_solve_lds(t, w);
}

/* the solve of a context's grid (poisson.hip) */
void isk_tri_prepare(iskra_ctx *c, TriArgs *pt);

#endif /* ISK_TRI_H */
