/*
 * poisson.hip -- finite-difference Poisson solve and E = -grad(phi) on gfx950.
 *
 * System (FiniteDifferenceMethod/src/generalized_poisson.jl:34-68,205-215,
 * 271-324,372-378): A phi = b with b = -rho/eps0 at free nodes, A the
 * natural-edge 3/5-point Laplacian scaled by 1/dx^2 (also along y,
 * generalized_poisson.jl:65), periodic ring links from apply_periodic and
 * Dirichlet rows (phi = value) from apply_dirichlet.  Multiplying by -dx^2
 * gives the symmetric positive form used here,
 *     L phi = f,   (L phi)_i = sum_links c (phi_i - phi_nb),   f = dx^2 rho/eps0,
 * with Dirichlet values moved to the right-hand side (same solution as the
 * reference's non-symmetric A).
 *
 * Solvers:
 *  DIRECT  1-D tridiagonal elimination (the reference's A\b is a direct solve),
 *          FP64, factor built once on the host, substitution on the device.
 *  PCG     Jacobi-preconditioned conjugate gradients: x, r, Ap and all inner
 *          products in FP64, search direction p and z in FP32; a dot product
 *          is per-work-group partials, summed in block order by the kernel
 *          that needs it (every work-group of it gets the same bits).
 *  MG      geometric multigrid V(2,2) cycles with red-black Gauss-Seidel on FP32
 *          levels as a defect correction of the FP64 iterate (residual, norm
 *          and update in FP64); levels <= 65^2 run in one work-group from LDS.
 *  MGPCG   PCG with one symmetric V-cycle as preconditioner.
 * Stopping rule: ||f_elim - L x||_2 / ||f_elim||_2 <= rtol in FP64 (f_elim is
 * f with the Dirichlet contributions moved over).  A system without any
 * Dirichlet node is singular (periodic); its right-hand side is projected to
 * zero mean and the mean-free solution is returned (the reference's A\b fixes
 * the constant by round-off).
 */
#include <math.h>

#include <algorithm>
#include <vector>

#include "isk_internal.h"
#include "isk_tri.h"

#define RED_BLOCK 256
#define PCG_BATCH 32
#define MG_BATCH 4
#define MG_COARSE_MAX 65

/* scalars: S_RZ0/S_RZ1 hold (r,z) of even/odd CG iterations, S_RTOL2 = rtol^2,
 * S_TOL2 = rtol^2 (f,f) */
enum { S_PAP = 0, S_ALPHA, S_BETA, S_RR, S_FF, S_TOL2, S_MEAN, S_RELRES, S_RZ0, S_RZ1, S_RTOL2,
       S_WORDS = 16 };
/* iflag words: [0] done, [1] iterations, [2] singular (PCG/MG); spectral solve:
 * [4] this solve met rtol, [5] sticky: an in-loop solve missed rtol,
 * [6] transform passes of this solve */
enum { IF_SP_DONE = 4, IF_SP_FAIL = 5, IF_SP_PASSES = 6 };


template <typename T>
__device__ __forceinline__ double apply_L(const Sten &s, const T *v, int i, int j,
                                          double *diag_out) {
  int n = j * s.nx + i;
  double acc = 0.0, diag = 0.0;
  if (s.axial) {
    const double cz = isk_rz_w(i, s.nx) * s.az;
    if (i > 0) { acc += ((double)i - 0.5) * (double)v[n - 1]; diag += (double)i - 0.5; }
    if (i < s.nx - 1) { acc += ((double)i + 0.5) * (double)v[n + 1]; diag += (double)i + 0.5; }
    if (j > 0) { acc += cz * (double)v[n - s.nx]; diag += cz; }
    if (j < s.ny - 1) { acc += cz * (double)v[n + s.nx]; diag += cz; }
    if (diag_out) *diag_out = diag;
    return diag * (double)v[n] - acc;
  }
  if (i > 0) { acc += (double)v[n - 1]; diag += 1.0; }
  if (i < s.nx - 1) { acc += (double)v[n + 1]; diag += 1.0; }
  if (s.per_x) {
    if (i == 0) { acc += s.cxp * (double)v[n + s.nx - 1]; diag += s.cxp; }
    if (i == s.nx - 1) { acc += s.cxp * (double)v[n - (s.nx - 1)]; diag += s.cxp; }
  }
  if (s.dim == 2) {
    if (j > 0) { acc += (double)v[n - s.nx]; diag += 1.0; }
    if (j < s.ny - 1) { acc += (double)v[n + s.nx]; diag += 1.0; }
    if (s.per_y) {
      if (j == 0) { acc += s.cyp * (double)v[n + (s.ny - 1) * s.nx]; diag += s.cyp; }
      if (j == s.ny - 1) { acc += s.cyp * (double)v[n - (s.ny - 1) * s.nx]; diag += s.cyp; }
    }
  }
  if (diag_out) *diag_out = diag;
  return diag * (double)v[n] - acc;
}

/* ------------------------------------------------------------------------ */
/* 1-D direct solve                                                          */
/* ------------------------------------------------------------------------ */
__global__ __launch_bounds__(TRI_BLOCK) void k_tri_solve(TriArgs t) {
  if (blockIdx.x != 0) return;
  tri_solve_group(t);
}

/* ------------------------------------------------------------------------ */
/* PCG                                                                       */
/* ------------------------------------------------------------------------ */
struct PcgArgs {
  Sten s;
  const double *rho;
  double *x, *r, *Ap;
  float *z, *p0, *p1; /* search directions of even / odd iterations */
  float *f0;  /* MG preconditioner input (MGPCG) */
  float *e0;  /* MG finest-level correction, zeroed before each V-cycle */
  const float *mz; /* what a V-cycle leaves as its result */
  double *scal, *partials;
  int *iflag;
  double *cgp; /* CG partials, 7 per work-group */
  int nblk;    /* work-groups of the CG kernels */
  double scale;
  int warm;
  const double *phi_in;
  double *phi_out; /* spectral solve: the residual kernels write phi here */
  int mgpre;
  int max_iter;
};

/* x = Dirichlet values / warm start / 0 */
__global__ void k_pcg_setx(PcgArgs a) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= a.s.nx * a.s.ny) return;
  int t = a.s.tags[n];
  a.x[n] = t ? a.s.tagval[t] : (a.warm ? a.phi_in[n] : 0.0);
}

/* scalars and flags of a new solve */
__global__ void k_pcg_init(double *scal, int *iflag, double tol2, int singular) {
  if (threadIdx.x < S_WORDS)
    scal[threadIdx.x] = (threadIdx.x == S_TOL2 || threadIdx.x == S_RTOL2) ? tol2 : 0.0;
  if (threadIdx.x < 4) iflag[threadIdx.x] = threadIdx.x == 2 ? singular : 0;
}

/* CG without device-wide reductions: a kernel that needs a dot product sums
 * the per-work-group partials that the previous kernel wrote, in block order,
 * in every work-group (the same data summed the same way gives the same bits
 * everywhere), so no kernel waits on the others through fences or counters.
 * Partials, RED_BLOCK-node work-groups: two slots by iteration parity of
 * {(r,r), (r,z), (f,f)} per work-group, then one (p,Ap) per work-group.
 * Iteration it: A(it) takes (r,r) and (r,z) of x_it, decides convergence,
 * forms p_it = z + beta p_{it-1} in p[it & 1] and (p, Ap); B(it) updates
 * x, r, z and writes the partials of x_{it+1} into slot (it + 1) & 1. */

/* sums of 3 doubles over the work-group: an xor butterfly within each wave
 * (every lane ends with the same bits), then the waves in index order */
template <int NT = RED_BLOCK>
__device__ __forceinline__ void wg_sum3(double &a, double &b, double &c) {
  __shared__ double w3[3][NT / 64];
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off);
    b += __shfl_xor(b, off);
    c += __shfl_xor(c, off);
  }
  __syncthreads(); /* a previous call's readers are done with w3 */
  if ((threadIdx.x & 63) == 0) {
    const int w = threadIdx.x >> 6;
    w3[0][w] = a;
    w3[1][w] = b;
    w3[2][w] = c;
  }
  __syncthreads();
  double sa = 0.0, sb = 0.0, sc = 0.0;
  for (int k = 0; k < NT / 64; ++k) {
    sa += w3[0][k];
    sb += w3[1][k];
    sc += w3[2][k];
  }
  a = sa;
  b = sb;
  c = sc;
}

__device__ __forceinline__ double *cg_slot(const PcgArgs &a, int q) {
  return a.cgp + (size_t)q * 3 * a.nblk;
}
__device__ __forceinline__ double *cg_pap(const PcgArgs &a) { return a.cgp + (size_t)6 * a.nblk; }

/* this work-group's partials (thread 0 holds the work-group sums) */
__device__ __forceinline__ void cg_put3(double *slot, double x, double y, double z) {
  wg_sum3(x, y, z);
  if (threadIdx.x == 0) {
    slot[3 * blockIdx.x] = x;
    slot[3 * blockIdx.x + 1] = y;
    slot[3 * blockIdx.x + 2] = z;
  }
}

/* singular systems: per-work-group partial sums of the right-hand side (the
 * residual kernel that follows sums them for the zero-mean projection) */
__global__ __launch_bounds__(RED_BLOCK) void k_pcg_mean(PcgArgs a) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  double v = 0.0, d1 = 0.0, d2 = 0.0;
  if (n < a.s.nx * a.s.ny) v = a.rho[n] * a.scale;
  wg_sum3(v, d1, d2);
  if (threadIdx.x == 0) a.partials[blockIdx.x] = v;
}

/* r = f_elim - L x at free nodes; partials of (r,r), (r,z) (Jacobi z = r/diag;
 * the MG preconditioner's z comes later) and (f,f) into slot 0 */
__global__ __launch_bounds__(RED_BLOCK) void k_pcg_resid(PcgArgs a) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  int nn = a.s.nx * a.s.ny;
  double rr = 0.0, rz = 0.0, ff = 0.0;
  /* singular system (flag set by an earlier kernel, the same for every
   * thread): the mean of the right-hand side from k_pcg_mean's partials */
  double mean = 0.0;
  if (a.iflag[2]) {
    double d1 = 0.0, d2 = 0.0;
    for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) mean += a.partials[k];
    wg_sum3(mean, d1, d2);
    mean /= (double)nn;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.scal[S_MEAN] = mean;
  }
  if (n < nn) {
    int i = n % a.s.nx, j = n / a.s.nx;
    if (a.s.tags[n] == 0) {
      double f = a.rho[n] * a.scale;
      if (a.s.axial) f *= isk_rz_w(i, a.s.nx);
      if (a.iflag[2]) f -= mean;
      double diag;
      /* x holds the Dirichlet values, so L x already carries them */
      double Lx = apply_L(a.s, a.x, i, j, &diag);
      double fe = f + dirichlet_rhs(a.s, i, j);
      double r = f - Lx;
      a.r[n] = r;
      if (!a.mgpre) {
        float z = (float)(r / diag);
        a.z[n] = z;
        rz = r * (double)z;
      } else {
        a.f0[n] = (float)r;
        a.e0[n] = 0.0f;
      }
      rr = r * r;
      ff = fe * fe;
    } else {
      a.r[n] = 0.0;
      a.z[n] = 0.0f;
      if (a.mgpre) {
        a.f0[n] = 0.0f;
        a.e0[n] = 0.0f;
      }
    }
    a.p0[n] = 0.0f;
    a.p1[n] = 0.0f;
  }
  cg_put3(cg_slot(a, 0), rr, rz, ff);
}

/* MG-preconditioned CG: z = the V-cycle's finest correction, (r,z) partials
 * into slot q */
__global__ __launch_bounds__(RED_BLOCK) void k_cg_toz(PcgArgs a, int q) {
  if (a.iflag[0]) return;
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  double rz = 0.0, d1 = 0.0, d2 = 0.0;
  if (n < a.s.nx * a.s.ny) {
    float z = a.mz[n];
    a.z[n] = z;
    rz = a.r[n] * (double)z;
  }
  wg_sum3(rz, d1, d2);
  if (threadIdx.x == 0) cg_slot(a, q)[3 * blockIdx.x + 1] = rz;
}

/* A(it): scalars of x_it, convergence, p_it = z + beta p_{it-1} (recomputed
 * at the neighbours), Ap = L p_it, (p, Ap) partials */
__global__ __launch_bounds__(RED_BLOCK) void k_cg_a(PcgArgs a, int it) {
  __shared__ int s_stop;
  if (threadIdx.x == 0) s_stop = a.iflag[0];
  double rr = 0.0, rz = 0.0, ff = 0.0;
  {
    const double *sl = cg_slot(a, it & 1);
    for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) {
      rr += sl[3 * k];
      rz += sl[3 * k + 1];
      ff += sl[3 * k + 2];
    }
  }
  wg_sum3(rr, rz, ff); /* its barriers also publish s_stop */
  if (s_stop) return;
  const double sff = it == 0 ? ff : a.scal[S_FF];
  const double tol2 = it == 0 ? a.scal[S_RTOL2] * ff : a.scal[S_TOL2];
  const bool done = rr <= tol2 || it >= a.max_iter;
  double beta = 0.0;
  if (it > 0) {
    const double old = a.scal[S_RZ0 + ((it - 1) & 1)];
    beta = old != 0.0 ? rz / old : 0.0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (it == 0) {
      a.scal[S_FF] = ff;
      a.scal[S_TOL2] = tol2;
    }
    a.scal[S_RR] = rr;
    a.scal[S_RELRES] = sff > 0.0 ? sqrt(rr / sff) : 0.0;
    a.scal[S_RZ0 + (it & 1)] = rz;
    a.scal[S_BETA] = beta;
    a.iflag[1] = it;
    if (done) a.iflag[0] = 1;
  }
  if (done) return;
  const float *pold = (it & 1) ? a.p0 : a.p1;
  float *pnew = (it & 1) ? a.p1 : a.p0;
  const float fb = (float)beta;
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  int nn = a.s.nx * a.s.ny;
  double pap = 0.0;
  if (n < nn) {
    int i = n % a.s.nx, j = n / a.s.nx;
    if (a.s.tags[n] == 0) {
#define PN(m) (a.s.tags[m] ? 0.0 : (double)fmaf(fb, pold[m], a.z[m]))
      double pc = PN(n);
      double acc = 0.0, diag = 0.0;
      if (a.s.axial) {
        const double cz = isk_rz_w(i, a.s.nx) * a.s.az;
        if (i > 0) { acc += ((double)i - 0.5) * PN(n - 1); diag += (double)i - 0.5; }
        if (i < a.s.nx - 1) { acc += ((double)i + 0.5) * PN(n + 1); diag += (double)i + 0.5; }
        if (j > 0) { acc += cz * PN(n - a.s.nx); diag += cz; }
        if (j < a.s.ny - 1) { acc += cz * PN(n + a.s.nx); diag += cz; }
      } else {
      if (i > 0) { acc += PN(n - 1); diag += 1.0; }
      if (i < a.s.nx - 1) { acc += PN(n + 1); diag += 1.0; }
      if (a.s.per_x) {
        if (i == 0) { acc += a.s.cxp * PN(n + a.s.nx - 1); diag += a.s.cxp; }
        if (i == a.s.nx - 1) { acc += a.s.cxp * PN(n - (a.s.nx - 1)); diag += a.s.cxp; }
      }
      if (a.s.dim == 2) {
        if (j > 0) { acc += PN(n - a.s.nx); diag += 1.0; }
        if (j < a.s.ny - 1) { acc += PN(n + a.s.nx); diag += 1.0; }
        if (a.s.per_y) {
          if (j == 0) { acc += a.s.cyp * PN(n + (a.s.ny - 1) * a.s.nx); diag += a.s.cyp; }
          if (j == a.s.ny - 1) { acc += a.s.cyp * PN(n - (a.s.ny - 1) * a.s.nx); diag += a.s.cyp; }
        }
      }
      }
#undef PN
      double ap = diag * pc - acc;
      pnew[n] = (float)pc;
      a.Ap[n] = ap;
      pap = pc * ap;
    } else {
      pnew[n] = 0.0f;
      a.Ap[n] = 0.0;
    }
  }
  double d1 = 0.0, d2 = 0.0;
  wg_sum3(pap, d1, d2);
  if (threadIdx.x == 0) cg_pap(a)[blockIdx.x] = pap;
}

/* B(it): alpha = (r,z) / (p,Ap); x += alpha p, r -= alpha Ap, z = M^-1 r;
 * partials of x_{it+1} into slot (it + 1) & 1 */
__global__ __launch_bounds__(RED_BLOCK) void k_cg_b(PcgArgs a, int it) {
  if (a.iflag[0]) return; /* set by an earlier kernel: the same for every thread */
  double pap = 0.0, d1 = 0.0, d2 = 0.0;
  {
    const double *pp = cg_pap(a);
    for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) pap += pp[k];
  }
  wg_sum3(pap, d1, d2);
  const double rzc = a.scal[S_RZ0 + (it & 1)];
  const double alpha = pap != 0.0 ? rzc / pap : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.scal[S_PAP] = pap;
    a.scal[S_ALPHA] = alpha;
  }
  const float *pc = (it & 1) ? a.p1 : a.p0;
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  int nn = a.s.nx * a.s.ny;
  double rr = 0.0, rz = 0.0;
  if (n < nn && a.s.tags[n] == 0) {
    int i = n % a.s.nx, j = n / a.s.nx;
    double p = (double)pc[n];
    a.x[n] = __builtin_fma(alpha, p, a.x[n]);
    double r = __builtin_fma(-alpha, a.Ap[n], a.r[n]);
    a.r[n] = r;
    rr = r * r;
    if (!a.mgpre) {
      double diag = 0.0;
      if (a.s.axial) {
        const double cz = isk_rz_w(i, a.s.nx) * a.s.az;
        if (i > 0) diag += (double)i - 0.5;
        if (i < a.s.nx - 1) diag += (double)i + 0.5;
        if (j > 0) diag += cz;
        if (j < a.s.ny - 1) diag += cz;
      } else {
        if (i > 0) diag += 1.0;
        if (i < a.s.nx - 1) diag += 1.0;
        if (a.s.per_x && (i == 0 || i == a.s.nx - 1)) diag += a.s.cxp;
        if (a.s.dim == 2) {
          if (j > 0) diag += 1.0;
          if (j < a.s.ny - 1) diag += 1.0;
          if (a.s.per_y && (j == 0 || j == a.s.ny - 1)) diag += a.s.cyp;
        }
      }
      float z = (float)(r / diag);
      a.z[n] = z;
      rz = r * (double)z;
    } else {
      a.f0[n] = (float)r;
    }
  }
  if (a.mgpre && n < nn) a.e0[n] = 0.0f;
  cg_put3(cg_slot(a, (it + 1) & 1), rr, rz, 0.0);
}

/* final: mean removal for singular systems, copy to phi */
__global__ void k_pcg_out(PcgArgs a, double *phi, double mean_sub) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < a.s.nx * a.s.ny) phi[n] = a.x[n] - mean_sub;
}

/* ------------------------------------------------------------------------ */
/* spectral direct solve: phi = Sy ((Sy F Sx) / lambda) Sx                   */
/* ------------------------------------------------------------------------ */
/* F (interior, row-major [j-1][i-1]) = f_elim = rho scale + Dirichlet
 * neighbours (the time loop's deposit kernel writes the same values) */
__global__ void k_sp_pack(IskSpPack pk, const double *rho) {
  const int mx = pk.s.nx - 2, my = pk.s.ny - 2;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= mx * my) return;
  const int i = e % mx + 1, j = e / mx + 1;
  pk.F[e] = isk_sp_pack_value(pk, rho[j * pk.s.nx + i], i, j);
}

struct SpGemm {
  const double *A, *B, *L; /* L: elementwise factor (mode 1) */
  double *C;               /* modes 0, 1 */
  double *x;               /* modes 2, 3: node array, interior (i, j) = (col+1, row+1) */
  int M, N, K, nx, mode;
  Sten s;                  /* mode 2: the boundary ring's Dirichlet values */
};

typedef double f64x4 __attribute__((ext_vector_type(4)));

/* B operand: the matrix B (RES = 0), or the residual node array read at the
 * interior nodes, row k and column c = node (c+1, k+1) (RES = 1) */
template <int RES>
__device__ __forceinline__ double sp_bload(const SpGemm &g, int k, int col) {
  if (RES) return g.B[(size_t)(k + 1) * g.nx + (col + 1)];
  return g.B[(size_t)k * g.N + col];
}

/* C = A B (row-major FP64) on the matrix cores (v_mfma_f64_16x16x4f64) for
 * one 16 x 16 block of C: the K range is split over 4 waves (w = 0..3) and
 * each wave's partial block goes to red[w]; sp_tile_sum adds them in wave
 * order (deterministic).  Operand lanes: A[row0 + l%16][k + l/16],
 * B[k + l/16][col0 + l%16]; result lane l holds C[row0 + l/16 + 4i][col0 +
 * l%16], i = 0..3 (rows interleaved).  All loads of a 64-wide k block are
 * issued before its MFMAs; the accumulation order is k ascending. */
template <int RES>
__device__ __forceinline__ void sp_tile_mfma(const SpGemm &g, int row0, int col0, int w, int lane,
                                             double (*red)[256]) {
  const int lr = lane & 15, kq = lane >> 4;
  const int arow = row0 + lr, bcol = col0 + lr;
  const int kper = ((g.K + 15) / 16) * 4;
  const int kbeg = w * kper;
  const int kend = min(g.K, kbeg + kper);
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  for (int k0 = kbeg; k0 < kend; k0 += 64) {
    double av[16], bv[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int kk = k0 + 4 * u + kq;
      av[u] = (arow < g.M && kk < kend) ? g.A[(size_t)arow * g.K + kk] : 0.0;
      bv[u] = (kk < kend && bcol < g.N) ? sp_bload<RES>(g, kk, bcol) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (k0 + 4 * u >= kend) break;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u], acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[w][(kq + 4 * i) * 16 + lr] = acc[i];
}
__device__ __forceinline__ double sp_tile_sum(double (*red)[256], int e) {
  return ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
}

/* wave 0 of the group, after a barrier: sum the 4 partials, apply the mode */
__device__ __forceinline__ void sp_tile_store(const SpGemm &g, int row0, int col0, int lane,
                                              double (*red)[256]) {
  const int lr = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = (kq + 4 * i) * 16 + lr;
    const double v = sp_tile_sum(red, e);
    const int row = row0 + kq + 4 * i, col = col0 + lr;
    if (row >= g.M || col >= g.N) continue;
    const size_t o = (size_t)row * g.N + col;
    if (g.mode == 0) g.C[o] = v;
    else if (g.mode == 1) g.C[o] = v * g.L[o];
    else {
      const size_t n = (size_t)(row + 1) * g.nx + (col + 1);
      if (g.mode == 2) g.x[n] = v;
      else g.x[n] += v;
    }
  }
}

/* the boundary ring of x = its Dirichlet values */
__device__ __forceinline__ void sp_ring_setx(const SpGemm &g, int tid, int nthr) {
  const int nx = g.s.nx, ny = g.s.ny;
  const int ring = 2 * nx + 2 * (ny - 2);
  for (int q = tid; q < ring; q += nthr) {
    int n;
    if (q < nx) n = q;                                     /* row 0 */
    else if (q < 2 * nx) n = (ny - 1) * nx + (q - nx);     /* row ny-1 */
    else {
      const int r = q - 2 * nx;                            /* columns 0, nx-1 */
      n = (1 + (r >> 1)) * nx + ((r & 1) ? nx - 1 : 0);
    }
    const int t = g.s.tags[n];
    g.x[n] = t ? g.s.tagval[t] : 0.0;
  }
}

/* one block of C per work-group; mode 2 (first pass, x = result) also sets
 * the boundary ring of x (work-group (0, 0)) */
__global__ __launch_bounds__(256) void k_sp_gemm(SpGemm g) {
  __shared__ double red[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row0 = blockIdx.y * 16, col0 = blockIdx.x * 16;
  sp_tile_mfma<0>(g, row0, col0, w, lane, red);
  __syncthreads();
  if (w == 0) sp_tile_store(g, row0, col0, lane, red);
  if (g.mode == 2 && blockIdx.x == 0 && blockIdx.y == 0) sp_ring_setx(g, threadIdx.x, 256);
}

static SpGemm sp_desc(iskra_ctx *c, const PcgArgs &a, const double *A, const double *B,
                      const double *L, double *C, int M, int N, int K, int mode) {
  SpGemm g;
  g.A = A;
  g.B = B;
  g.L = L;
  g.C = C;
  g.x = a.x;
  g.M = M;
  g.N = N;
  g.K = K;
  g.nx = c->g.nx;
  g.mode = mode;
  g.s = a.s;
  return g;
}

/* the four GEMMs of one transform pass: x = L^-1 F (first, with the
 * boundary ring) or x += L^-1 r (correction, r read at the interior nodes) */
static void sp_pass_desc(iskra_ctx *c, const PcgArgs &a, int correction, SpGemm g[4]) {
  IskPoisson &p = c->ps;
  const int mx = p.sp_nx, my = p.sp_ny;
  g[0] = sp_desc(c, a, p.sp_Sy, correction ? a.r : p.sp_F, nullptr, p.sp_T1, my, mx, my, 0);
  g[1] = sp_desc(c, a, p.sp_T1, p.sp_Sx, p.sp_Li, p.sp_T2, my, mx, mx, 1);
  g[2] = sp_desc(c, a, p.sp_Sy, p.sp_T2, nullptr, p.sp_T1, my, mx, my, 0);
  g[3] = sp_desc(c, a, p.sp_T1, p.sp_Sx, nullptr, nullptr, my, mx, mx, correction ? 3 : 2);
}

/* residual of node n (free nodes: r = f - L x, contributions to ||r||^2 and
 * ||f_elim||^2; Dirichlet nodes: r = 0); also phi = x and, with E, the field
 * of node n from x (the arithmetic of efield_body).  f and fe: the node's f and
 * f_elim */
__device__ __forceinline__ void sp_resid_node(const PcgArgs &a, const double *x, int n, bool free,
                                              double f, double fe, float *E, double dx, double dy,
                                              double *rr, double *ff) {
  if (free) {
    const double r = f - apply_L(a.s, x, n % a.s.nx, n / a.s.nx, nullptr);
    a.r[n] = r;
    *rr += r * r;
    *ff += fe * fe;
  } else {
    a.r[n] = 0.0;
  }
  a.phi_out[n] = x[n];
  if (E) efield_node(x, E, 2, a.s.nx, a.s.ny, dx, dy, n);
}
__device__ __forceinline__ void sp_resid_node(const PcgArgs &a, const double *x, int n, float *E,
                                              double dx, double dy, double *rr, double *ff) {
  const bool free = a.s.tags[n] == 0;
  const double f = free ? a.rho[n] * a.scale : 0.0;
  const double fe = free ? f + dirichlet_rhs(a.s, n % a.s.nx, n / a.s.nx) : 0.0;
  sp_resid_node(a, x, n, free, f, fe, E, dx, dy, rr, ff);
}

/* r = f_elim - L x; phi = x; with E != null also E = -grad phi.  Each
 * work-group writes its sums of r^2 and f_elim^2 to partials[2b], [2b+1]
 * (summed in a fixed order by k_sp_correct, which runs next: no device-wide
 * fence and counter here) */
__global__ __launch_bounds__(RED_BLOCK) void k_sp_resid(PcgArgs a, float *E, double dx,
                                                        double dy) {
  __shared__ double ra[RED_BLOCK], rb[RED_BLOCK];
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  double rr = 0.0, ff = 0.0;
  if (n < a.s.nx * a.s.ny) sp_resid_node(a, a.x, n, E, dx, dy, &rr, &ff);
  ra[threadIdx.x] = rr;
  rb[threadIdx.x] = ff;
  __syncthreads();
  for (int off = RED_BLOCK / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) {
      ra[threadIdx.x] += ra[threadIdx.x + off];
      rb[threadIdx.x] += rb[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.partials[2 * blockIdx.x] = ra[0];
    a.partials[2 * blockIdx.x + 1] = rb[0];
  }
}

/* A correction pass in one work-group of 16 waves (4 groups of 4 waves, each
 * group computing 16 x 16 blocks with the same tile code as k_sp_gemm, so the
 * results are those of the multi-work-group GEMMs), then the residual, phi and
 * E of the corrected x.  It returns at once when iflag[IF_SP_DONE] is set,
 * which is the usual case: one transform pass is exact to FP64 round-off, and
 * a correction is only needed when rtol is below that (then it takes about a
 * millisecond at 257^2).  second != 0: a miss after the correction sets
 * iflag[IF_SP_FAIL]. */
#define SPC_THREADS 1024
struct SpCorrect {
  SpGemm g[4];
  PcgArgs a;
  double rtol, dx, dy;
  float *E;
  int second;
  int nparts; /* > 0: first sum the residual's partials (the first pass's residual) */
};

/* fixed-order sum over the work-group of two values per thread; every
 * thread gets the totals */
__device__ __forceinline__ void spc_sum2(double *x, double *y, double (*sred)[SPC_THREADS / 64]) {
  double rr = *x, ff = *y;
  for (int off = 32; off > 0; off >>= 1) {
    rr += __shfl_xor(rr, off);
    ff += __shfl_xor(ff, off);
  }
  if ((threadIdx.x & 63) == 0) {
    sred[0][threadIdx.x >> 6] = rr;
    sred[1][threadIdx.x >> 6] = ff;
  }
  __syncthreads();
  double srr = 0.0, sff = 0.0;
  for (int k = 0; k < SPC_THREADS / 64; ++k) {
    srr += sred[0][k];
    sff += sred[1][k];
  }
  __syncthreads();
  *x = srr;
  *y = sff;
}

/* Small grids: a transform pass in two launches.  A work-group of 16 waves makes a
 * strip of 16 rows of the first product in LDS (one 16 x 16 block each 4 waves,
 * the contraction split over them as in k_sp_gemm, so x is the same to the last bit)
 * and multiplies it on; the second launch's strips overlap by a row on either side, so
 * that the residual, phi and E of their 14 inner rows follow from LDS as well.  A
 * launch is a chain of waits, so all that depends on nothing, the operands of both
 * products and the nodes' right-hand sides, is requested first.
 * As four products and a residual pass a step of a few particles took 36.8 us on
 * 65 x 65 nodes, 34.5 on 33 x 33 and 38.1 on 65 x 129, with this 32.4, 27.6 and 35.6;
 * on wider grids the strips are too few for the chip (129 x 129: 54.6 us against
 * 40.5), hence the limits. */
#define SPP_ROWS 14
#define SPP_COLS 64 /* interior columns: 4 blocks */
#define SPP_MAXMY 128
#define SPP_LD (SPP_COLS + 1)
struct SpPair {
  const double *Sy, *B, *Sx, *Li; /* B: F, or the first launch's T2 */
  double *T2;
  int mx, my;
  PcgArgs a;
  double dx, dy;
  float *E;
};
static int sp_paired(int mx, int my) { return mx <= SPP_COLS && my <= SPP_MAXMY; }

template <int LAST>
__global__ __launch_bounds__(SPC_THREADS) void k_sp_pair(SpPair c) {
  __shared__ double red[4][4][256];
  __shared__ double T[16 * SPP_LD];
  __shared__ double xs[LAST ? 16 * (SPP_COLS + 2) : 1];
  constexpr int U0 = SPP_MAXMY / 16, U1 = SPP_COLS / 16;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, grp = wv >> 2, w = wv & 3;
  const int lr = lane & 15, kq = lane >> 4;
  const int mx = c.mx, my = c.my, nx = mx + 2, ny = my + 2;
  const int row0 = LAST ? (int)blockIdx.x * SPP_ROWS - 1 : (int)blockIdx.x * 16;
  const int arow = row0 + lr, col = grp * 16 + lr;
  const bool aon = arow >= 0 && arow < my, con = col < mx;
  const int kp0 = ((my + 15) / 16) * 4, kb0 = w * kp0, ke0 = min(my, kb0 + kp0);
  const int kp1 = ((mx + 15) / 16) * 4, kb1 = w * kp1, ke1 = min(mx, kb1 + kp1);
  double av[U0], bv[U0], sv[U1];
#pragma unroll
  for (int u = 0; u < U0; ++u) {
    const int k = kb0 + 4 * u + kq;
    av[u] = aon && k < ke0 ? c.Sy[(size_t)arow * my + k] : 0.0;
    bv[u] = con && k < ke0 ? c.B[(size_t)k * mx + col] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < U1; ++u) {
    const int k = kb1 + 4 * u + kq;
    sv[u] = con && k < ke1 ? c.Sx[(size_t)k * mx + col] : 0.0;
  }
  /* a wave stores the 4 rows kq + 4 w of its block's sum */
  const int sr = kq + 4 * w, srow = row0 + sr;
  const bool son = con && srow >= 0 && srow < my;
  /* LAST: strip row r is node row j0 + r; this group's nodes are rows jb .. je - 1 */
  const int j0 = row0 + 1, jb = j0 == 0 ? 0 : j0 + 1;
  const int je = j0 + SPP_ROWS >= my ? ny : j0 + 1 + SPP_ROWS;
  const int n0 = jb * nx + tid;
  double f0 = 0.0, fe0 = 0.0, li = 0.0;
  bool free0 = false;
  if (LAST) {
    for (int q = tid; q < 16 * nx; q += SPC_THREADS) { /* the ring's Dirichlet values */
      const int j = j0 + q / nx, i = q % nx;
      if (j < ny && (j == 0 || j == ny - 1 || i == 0 || i == nx - 1)) {
        const int t = c.a.s.tags[j * nx + i];
        xs[q] = t ? c.a.s.tagval[t] : 0.0;
      }
    }
    if (n0 < je * nx) {
      free0 = c.a.s.tags[n0] == 0;
      if (free0) {
        f0 = c.a.rho[n0] * c.a.scale;
        fe0 = f0 + dirichlet_rhs(c.a.s, n0 % nx, n0 / nx);
      }
    }
  } else if (son) {
    li = c.Li[(size_t)srow * mx + col];
  }
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < U0; ++u)
    if (kb0 + 4 * u < ke0) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u], acc, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) red[grp][w][(kq + 4 * i) * 16 + lr] = acc[i];
  __syncthreads();
  T[sr * SPP_LD + col] = sp_tile_sum(red[grp], sr * 16 + lr);
  __syncthreads();
  acc = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < U1; ++u)
    if (kb1 + 4 * u < ke1) {
      const int k = kb1 + 4 * u + kq;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k < ke1 ? T[lr * SPP_LD + k] : 0.0, sv[u], acc, 0,
                                                 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[grp][w][(kq + 4 * i) * 16 + lr] = acc[i];
  __syncthreads();
  const double v = sp_tile_sum(red[grp], sr * 16 + lr);
  if (!LAST) {
    if (son) c.T2[(size_t)srow * mx + col] = v * li;
    return;
  }
  if (son) xs[sr * nx + col + 1] = v;
  __syncthreads();
  const double *x = xs - (ptrdiff_t)j0 * nx;
  double rr = 0.0, ff = 0.0;
  if (n0 < je * nx) {
    c.a.x[n0] = x[n0];
    sp_resid_node(c.a, x, n0, free0, f0, fe0, c.E, c.dx, c.dy, &rr, &ff);
  }
  for (int n = n0 + SPC_THREADS; n < je * nx; n += SPC_THREADS) {
    c.a.x[n] = x[n];
    sp_resid_node(c.a, x, n, c.E, c.dx, c.dy, &rr, &ff);
  }
  spc_sum2(&rr, &ff, (double(*)[SPC_THREADS / 64])&red[0][0][0]);
  if (tid == 0) {
    c.a.partials[2 * blockIdx.x] = rr;
    c.a.partials[2 * blockIdx.x + 1] = ff;
  }
}

__global__ __launch_bounds__(SPC_THREADS) void k_sp_correct(SpCorrect c) {
  __shared__ double red[4][4][256];
  __shared__ double sred[2][SPC_THREADS / 64];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6, grp = wv >> 2, w = wv & 3;
  bool done;
  if (c.nparts > 0) {
    double rr = 0.0, ff = 0.0;
    for (int k = tid; k < c.nparts; k += SPC_THREADS) {
      rr += c.a.partials[2 * k];
      ff += c.a.partials[2 * k + 1];
    }
    spc_sum2(&rr, &ff, sred);
    const double rel = ff > 0.0 ? sqrt(rr / ff) : 0.0;
    done = rel <= c.rtol;
    if (tid == 0) {
      c.a.scal[S_RELRES] = rel;
      c.a.iflag[IF_SP_DONE] = done;
      c.a.iflag[IF_SP_PASSES] = 1;
    }
  } else {
    done = c.a.iflag[IF_SP_DONE] != 0;
  }
  if (done) return;
  for (int st = 0; st < 4; ++st) {
    const SpGemm &g = c.g[st];
    const int tx = (g.N + 15) / 16, ntile = tx * ((g.M + 15) / 16);
    for (int t0 = 0; t0 < ntile; t0 += 4) {
      const int t = t0 + grp;
      const bool on = t < ntile;
      const int row0 = (t / tx) * 16, col0 = (t % tx) * 16;
      if (on) {
        if (st == 0) sp_tile_mfma<1>(g, row0, col0, w, lane, red[grp]);
        else sp_tile_mfma<0>(g, row0, col0, w, lane, red[grp]);
      }
      __syncthreads();
      if (on && w == 0) sp_tile_store(g, row0, col0, lane, red[grp]);
      __syncthreads();
    }
    /* the next stage reads what this one wrote (global memory) */
    __threadfence();
    __syncthreads();
  }
  const int nn = c.a.s.nx * c.a.s.ny;
  double rr = 0.0, ff = 0.0;
  for (int n = tid; n < nn; n += SPC_THREADS) sp_resid_node(c.a, c.a.x, n, c.E, c.dx, c.dy, &rr, &ff);
  spc_sum2(&rr, &ff, sred);
  if (tid == 0) {
    const double rel = ff > 0.0 ? sqrt(rr / ff) : 0.0;
    c.a.scal[S_RELRES] = rel;
    const int ok = rel <= c.rtol;
    c.a.iflag[IF_SP_DONE] = ok;
    c.a.iflag[IF_SP_PASSES] += 1;
    if (c.second && !ok) c.a.iflag[IF_SP_FAIL] = 1;
  }
}

/* ------------------------------------------------------------------------ */
/* multigrid                                                                 */
/* ------------------------------------------------------------------------ */
struct MgLevel {
  float *e, *f;
  int nx, ny;
};

/* levels [cl, nlev) as one V-cycle inside one work-group (LDS resident) */
struct MgCoarseArgs {
  float *e_out, *f_in;
  int nlev_c;
  int nx[12], ny[12], off[12];
  int total;
  const int *flag;
  /* decide != 0: this kernel takes the cycle's convergence verdict */
  int decide, nparts, dfirst, max_iter;
  const double *partials;
  double *scal;
  int *iflag;
};

/* defect-correction multigrid: the convergence verdict on the FP64 residual
 * of x, taken by the kernel after the one that wrote the per-work-group
 * (r,r), (f,f) partials, in every work-group alike (the same sums in the
 * same order give the same bits); work-group 0 records it.  Returns true
 * when the cycle stops here.  The iteration limit is applied by work-group 0
 * alone through the flag, which the later kernels of the cycle read. */
template <int NT>
__device__ bool mg_verdict(const double *partials, int nparts, int first, double *scal,
                           int *iflag, int max_iter) {
  double rr = 0.0, ff = 0.0, d = 0.0;
  for (int k = threadIdx.x; k < nparts; k += NT) {
    rr += partials[2 * k];
    ff += partials[2 * k + 1];
  }
  wg_sum3<NT>(rr, ff, d);
  const double sff = first ? ff : scal[S_FF];
  const double tol2 = first ? scal[S_RTOL2] * ff : scal[S_TOL2];
  const bool done = rr <= tol2;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    if (first) {
      scal[S_FF] = ff;
      scal[S_TOL2] = tol2;
    }
    scal[S_RR] = rr;
    scal[S_RELRES] = sff > 0.0 ? sqrt(rr / sff) : 0.0;
    const int it = iflag[1];
    if (done || it >= max_iter) iflag[0] = 1;
    else iflag[1] = it + 1;
  }
  return done;
}

/* threads as a 32 x 32 grid; interior nodes of one colour, no divisions */
__device__ __forceinline__ void lds_rbgs(float *e, const float *f, int nx, int ny, int color) {
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int j = 1 + ty; j < ny - 1; j += 32) {
    int i0 = 2 - ((color + j) & 1);
    for (int i = i0 + 2 * tx; i < nx - 1; i += 64) {
      int m = j * nx + i;
      float s = (e[m - 1] + e[m + 1]) + (e[m - nx] + e[m + nx]);
      e[m] = (f[m] + s) * 0.25f;
    }
  }
  __syncthreads();
}

__global__ __launch_bounds__(1024) void k_mg_coarse(MgCoarseArgs a) {
  if (a.decide) {
    if (mg_verdict<1024>(a.partials, a.nparts, a.dfirst, a.scal, a.iflag, a.max_iter)) return;
  } else if (a.flag[0]) {
    return;
  }
  extern __shared__ float sm[];
  float *E = sm;
  float *Fv = sm + a.total;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  int n0 = a.nx[0] * a.ny[0];
  for (int k = threadIdx.x; k < a.total; k += blockDim.x) {
    E[k] = 0.0f;
    Fv[k] = k < n0 ? a.f_in[k] : 0.0f;
  }
  __syncthreads();
  /* down */
  for (int l = 0; l < a.nlev_c - 1; ++l) {
    float *e = E + a.off[l];
    float *f = Fv + a.off[l];
    int nx = a.nx[l], ny = a.ny[l];
    lds_rbgs(e, f, nx, ny, 0);
    lds_rbgs(e, f, nx, ny, 1);
    lds_rbgs(e, f, nx, ny, 0);
    lds_rbgs(e, f, nx, ny, 1);
    float *fc = Fv + a.off[l + 1];
    int cx = a.nx[l + 1], cy = a.ny[l + 1];
    for (int J = 1 + ty; J < cy - 1; J += 32)
      for (int I = 1 + tx; I < cx - 1; I += 32) {
        int i = 2 * I, j = 2 * J;
        float acc[3][3];
        for (int dj = -1; dj <= 1; ++dj)
          for (int di = -1; di <= 1; ++di) {
            int m = (j + dj) * nx + (i + di);
            float s = (e[m - 1] + e[m + 1]) + (e[m - nx] + e[m + nx]);
            acc[dj + 1][di + 1] = f[m] - (4.0f * e[m] - s);
          }
        float edge = (acc[0][1] + acc[2][1]) + (acc[1][0] + acc[1][2]);
        float corner = (acc[0][0] + acc[0][2]) + (acc[2][0] + acc[2][2]);
        fc[J * cx + I] = (4.0f * acc[1][1] + 2.0f * edge + corner) * 0.25f;
      }
    __syncthreads();
  }
  /* coarsest: exact for one interior node, otherwise Gauss-Seidel sweeps */
  {
    int l = a.nlev_c - 1;
    float *e = E + a.off[l];
    float *f = Fv + a.off[l];
    int nx = a.nx[l], ny = a.ny[l];
    if (nx == 3 && ny == 3) {
      if (threadIdx.x == 0) e[4] = 0.25f * f[4];
      __syncthreads();
    } else {
      for (int it = 0; it < 16; ++it) {
        lds_rbgs(e, f, nx, ny, 0);
        lds_rbgs(e, f, nx, ny, 1);
      }
    }
  }
  /* up */
  for (int l = a.nlev_c - 2; l >= 0; --l) {
    float *e = E + a.off[l];
    float *f = Fv + a.off[l];
    float *ec = E + a.off[l + 1];
    int nx = a.nx[l], ny = a.ny[l], cx = a.nx[l + 1];
    for (int j = 1 + ty; j < ny - 1; j += 32)
      for (int i = 1 + tx; i < nx - 1; i += 32) {
        int I = i >> 1, J = j >> 1;
        int m = J * cx + I;
        float v;
        if (!(i & 1) && !(j & 1)) v = ec[m];
        else if ((i & 1) && !(j & 1)) v = 0.5f * (ec[m] + ec[m + 1]);
        else if (!(i & 1) && (j & 1)) v = 0.5f * (ec[m] + ec[m + cx]);
        else v = 0.25f * ((ec[m] + ec[m + 1]) + (ec[m + cx] + ec[m + cx + 1]));
        e[j * nx + i] += v;
      }
    __syncthreads();
    lds_rbgs(e, f, nx, ny, 1);
    lds_rbgs(e, f, nx, ny, 0);
    lds_rbgs(e, f, nx, ny, 1);
    lds_rbgs(e, f, nx, ny, 0);
  }
  for (int k = threadIdx.x; k < n0; k += blockDim.x) a.e_out[k] = E[k];
}

/* ------------------------------------------------------------------------ */
/* fused fine-level multigrid kernels (temporal blocking in LDS)            */
/* ------------------------------------------------------------------------ */
/* A work-group owns CT x CT coarse nodes and the 2CT x 2CT fine nodes starting
 * at twice their index; it loads a fine tile with a halo of H nodes, runs the
 * four red-black half-sweeps of one smoothing stage there (each half-sweep
 * leaves one fewer halo ring exact), and writes only owned nodes, so the
 * result equals the global red-black Gauss-Seidel sweep. */
#define MGT_NT 512
#define MGT_CT 8
#define MGT_H 6
#define MGT_S (2 * MGT_CT + 2 * MGT_H)

struct MgFused {
  MgLevel F, C;
  float *out;   /* up: the level's new e (not F.e: other work-groups still read its halo) */
  const int *flag;
  /* finest level of the FP64 defect correction */
  int mode_in;  /* down: 0 = f from F.f, 1 = f = dx^2 rho/eps0 - L x (FP64) */
  int mode_out; /* up: 0 = write out, 1 = x += e (FP64) */
  Sten s;
  double *x;
  const double *rho;
  double scale;
  double *scal, *partials;
  int *iflag;
  int first, max_iter;
  /* decide != 0: this kernel takes the cycle's convergence verdict from the
   * nparts partials of the finest residual (dfirst: first cycle of the solve) */
  int decide, nparts, dfirst;
};

/* one colour of a tile: a thread a node of that colour, so a sweep is one pass of
 * MGT_NT threads (a thread a node of either colour, 256 at a time, took four; a cycle
 * on 513 x 513 nodes 83 us, now 71; 256 threads 75, 1024 77; tiles of 24 or 32 nodes
 * 10 to 30 % longer) */
__device__ __forceinline__ void tile_sweep(float *se, const float *sf, int ox0, int oy0, int nx,
                                           int ny, int color) {
  constexpr int HALF = MGT_S / 2; /* nodes of a colour in a row */
  for (int q = threadIdx.x; q < HALF * MGT_S; q += MGT_NT) {
    const int lj = q / HALF, gj = oy0 + lj;
    const int li = 2 * (q - lj * HALF) + ((color ^ ox0 ^ gj) & 1), gi = ox0 + li;
    if (li < 1 || lj < 1 || li > MGT_S - 2 || lj > MGT_S - 2) continue;
    if (gi < 1 || gj < 1 || gi > nx - 2 || gj > ny - 2) continue;
    const int k = lj * MGT_S + li;
    float sum = (se[k - 1] + se[k + 1]) + (se[k - MGT_S] + se[k + MGT_S]);
    se[k] = (sf[k] + sum) * 0.25f;
  }
  __syncthreads();
}

/* pre-smooth from e = 0, restrict the residual, write owned e (and f) */
__global__ __launch_bounds__(MGT_NT) void k_mgf_down(MgFused a) {
  if (a.decide) {
    if (mg_verdict<MGT_NT>(a.partials, a.nparts, a.dfirst, a.scal, a.iflag, a.max_iter)) return;
  } else if (!a.first && a.flag[0]) {
    return;
  }
  __shared__ float se[MGT_S * MGT_S], sf[MGT_S * MGT_S];
  const int nx = a.F.nx, ny = a.F.ny;
  const int I0 = blockIdx.x * MGT_CT, J0 = blockIdx.y * MGT_CT;
  const int ox0 = 2 * I0 - MGT_H, oy0 = 2 * J0 - MGT_H;
  double rr = 0.0, ff = 0.0;
  for (int k = threadIdx.x; k < MGT_S * MGT_S; k += MGT_NT) {
    int lj = k / MGT_S, li = k - lj * MGT_S;
    int gi = ox0 + li, gj = oy0 + lj;
    bool interior = gi >= 1 && gj >= 1 && gi <= nx - 2 && gj <= ny - 2;
    float f = 0.0f;
    if (interior) {
      int m = gj * nx + gi;
      if (a.mode_in == 1) {
        double fs = a.rho[m] * a.scale;
        double r = fs - apply_L(a.s, a.x, gi, gj, nullptr);
        f = (float)r;
        bool owned = li >= MGT_H && lj >= MGT_H && li < MGT_H + 2 * MGT_CT &&
                     lj < MGT_H + 2 * MGT_CT;
        if (owned) {
          double fe = fs + dirichlet_rhs(a.s, gi, gj);
          rr += r * r;
          ff += fe * fe;
        }
      } else {
        f = a.F.f[m];
      }
    }
    sf[k] = f;
    se[k] = 0.0f;
  }
  __syncthreads();
  tile_sweep(se, sf, ox0, oy0, nx, ny, 0);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 1);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 0);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 1);
  /* residual at fine nodes -> full weighting -> coarse rhs (x4) */
  const int cx = a.C.nx, cy = a.C.ny;
  for (int q = threadIdx.x; q < MGT_CT * MGT_CT; q += MGT_NT) {
    int I = I0 + (q % MGT_CT), J = J0 + (q / MGT_CT);
    if (I >= cx || J >= cy) continue;
    int n = J * cx + I;
    a.C.e[n] = 0.0f;
    if (I <= 0 || J <= 0 || I >= cx - 1 || J >= cy - 1) {
      a.C.f[n] = 0.0f;
      continue;
    }
    int lc = (2 * J - oy0) * MGT_S + (2 * I - ox0);
    float acc[3][3];
#pragma unroll
    for (int dj = -1; dj <= 1; ++dj)
#pragma unroll
      for (int di = -1; di <= 1; ++di) {
        int k = lc + dj * MGT_S + di;
        float sum = (se[k - 1] + se[k + 1]) + (se[k - MGT_S] + se[k + MGT_S]);
        acc[dj + 1][di + 1] = sf[k] - (4.0f * se[k] - sum);
      }
    float edge = (acc[0][1] + acc[2][1]) + (acc[1][0] + acc[1][2]);
    float corner = (acc[0][0] + acc[0][2]) + (acc[2][0] + acc[2][2]);
    a.C.f[n] = (4.0f * acc[1][1] + 2.0f * edge + corner) * 0.25f;
  }
  /* owned fine nodes: smoothed e (and, at the finest level, f) */
  for (int q = threadIdx.x; q < 4 * MGT_CT * MGT_CT; q += MGT_NT) {
    int li = MGT_H + (q % (2 * MGT_CT)), lj = MGT_H + (q / (2 * MGT_CT));
    int gi = ox0 + li, gj = oy0 + lj;
    if (gi >= nx || gj >= ny) continue;
    int m = gj * nx + gi;
    int k = lj * MGT_S + li;
    a.F.e[m] = se[k];
    if (a.mode_in == 1) a.F.f[m] = sf[k];
  }
  if (a.mode_in == 1) {
    /* partials of the residual of x; the next kernel takes the verdict */
    double d = 0.0;
    wg_sum3<MGT_NT>(rr, ff, d);
    if (threadIdx.x == 0) {
      const int bid = blockIdx.x + gridDim.x * blockIdx.y;
      a.partials[2 * bid] = rr;
      a.partials[2 * bid + 1] = ff;
    }
  }
}

/* e += P e_coarse, post-smooth, write owned e (or x += e at the finest level) */
__global__ __launch_bounds__(MGT_NT) void k_mgf_up(MgFused a) {
  if (a.flag[0]) return;
  __shared__ float se[MGT_S * MGT_S], sf[MGT_S * MGT_S];
  const int nx = a.F.nx, ny = a.F.ny, cx = a.C.nx;
  const int I0 = blockIdx.x * MGT_CT, J0 = blockIdx.y * MGT_CT;
  const int ox0 = 2 * I0 - MGT_H, oy0 = 2 * J0 - MGT_H;
  for (int k = threadIdx.x; k < MGT_S * MGT_S; k += MGT_NT) {
    int lj = k / MGT_S, li = k - lj * MGT_S;
    int i = ox0 + li, j = oy0 + lj;
    bool interior = i >= 1 && j >= 1 && i <= nx - 2 && j <= ny - 2;
    float e = 0.0f, f = 0.0f;
    if (interior) {
      int m = j * nx + i;
      int I = i >> 1, J = j >> 1;
      const float *ec = a.C.e;
      int mc = J * cx + I;
      float v;
      if (!(i & 1) && !(j & 1)) v = ec[mc];
      else if ((i & 1) && !(j & 1)) v = 0.5f * (ec[mc] + ec[mc + 1]);
      else if (!(i & 1) && (j & 1)) v = 0.5f * (ec[mc] + ec[mc + cx]);
      else v = 0.25f * ((ec[mc] + ec[mc + 1]) + (ec[mc + cx] + ec[mc + cx + 1]));
      e = a.F.e[m] + v;
      f = a.F.f[m];
    }
    se[k] = e;
    sf[k] = f;
  }
  __syncthreads();
  tile_sweep(se, sf, ox0, oy0, nx, ny, 1);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 0);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 1);
  tile_sweep(se, sf, ox0, oy0, nx, ny, 0);
  for (int q = threadIdx.x; q < 4 * MGT_CT * MGT_CT; q += MGT_NT) {
    int li = MGT_H + (q % (2 * MGT_CT)), lj = MGT_H + (q / (2 * MGT_CT));
    int gi = ox0 + li, gj = oy0 + lj;
    if (gi >= nx || gj >= ny) continue;
    int m = gj * nx + gi;
    int k = lj * MGT_S + li;
    if (a.mode_out == 1) {
      if (gi >= 1 && gj >= 1 && gi <= nx - 2 && gj <= ny - 2) a.x[m] += (double)se[k];
    } else {
      a.out[m] = se[k];
    }
  }
}

/* FP64 defect-correction residual: f0 = r = f_elim - L x, e0 = 0 */
__global__ __launch_bounds__(RED_BLOCK) void k_mg_resid0(PcgArgs a, float *e0, int first) {
  if (!first && a.iflag[0]) return;
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  int nn = a.s.nx * a.s.ny;
  double rr = 0.0, ff = 0.0;
  if (n < nn) {
    e0[n] = 0.0f;
    if (a.s.tags[n] == 0) {
      int i = n % a.s.nx, j = n / a.s.nx;
      double f = a.rho[n] * a.scale;
      double fe = f + dirichlet_rhs(a.s, i, j);
      double r = f - apply_L(a.s, a.x, i, j, nullptr);
      a.f0[n] = (float)r;
      rr = r * r;
      ff = fe * fe;
    } else {
      a.f0[n] = 0.0f;
    }
  }
  /* partials of the residual of x; the next kernel takes the verdict */
  double d = 0.0;
  wg_sum3<RED_BLOCK>(rr, ff, d);
  if (threadIdx.x == 0) {
    a.partials[2 * blockIdx.x] = rr;
    a.partials[2 * blockIdx.x + 1] = ff;
  }
}

__global__ void k_mg_update0(PcgArgs a, const float *e0) {
  if (a.iflag[0]) return;
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < a.s.nx * a.s.ny && a.s.tags[n] == 0) a.x[n] += (double)e0[n];
}

/* z = e0 after a preconditioning V-cycle */
/* ------------------------------------------------------------------------ */
/* E = -grad(phi)                                                            */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ void efield_body(const double *phi, float *E, int dim, int nx, int ny,
                                            double dx, double dy, const int blk) {
  int n = blk * blockDim.x + threadIdx.x;
  if (n >= nx * ny) return;
  efield_node(phi, E, dim, nx, ny, dx, dy, n);
}

__global__ void k_efield(const double *phi, float *E, int dim, int nx, int ny, double dx,
                         double dy) {
  efield_body(phi, E, dim, nx, ny, dx, dy, blockIdx.x);
}

int isk_efield(iskra_ctx *c) {
  int nn = isk_nodes(c);
  hipLaunchKernelGGL(k_efield, dim3((nn + 255) / 256), dim3(256), 0, c->stream,
                     c->phi, c->E, c->g.dim, c->g.nx, c->g.ny, c->g.dx, c->g.dy);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* ------------------------------------------------------------------------ */
/* host side                                                                 */
/* ------------------------------------------------------------------------ */
/* ------------------------------------------------------------------------ */
/* BiCGStab for the systems with floating-electrode rows                     */
/* ------------------------------------------------------------------------ */
/* calculate_electric_potential (generalized_poisson.jl:372-378) when
 * apply_neumann has replaced rows (floating electrodes): the system is not
 * symmetric, so it is solved by right-preconditioned BiCGStab (van der
 * Vorst 1992) with the Jacobi preconditioner, FP64 throughout.  Unknowns are
 * the non-Dirichlet nodes; the sigma degrees of freedom are identity rows in
 * the reference (b = sigma), so they enter as known right-hand-side terms.
 * Like the CG kernels, every kernel sums the previous kernel's per-work-group
 * partials in block order itself (no device-wide reduction); iteration it:
 *   B1: beta, p = r + beta (p - omega v), v = A K^-1 p, partials (rh, v)
 *   B2: alpha = rho / (rh, v), s = r - alpha v
 *   B3: t = A K^-1 s, partials (t, s), (t, t)
 *   B4: omega = (t, s) / (t, t), x += alpha K^-1 p + omega K^-1 s,
 *       r = s - omega t, partials (rh, r), (r, r)
 * p and v alternate between two buffers by iteration parity. */
enum { BS_RHO0 = 0, BS_RHO1, BS_ALPHA, BS_OMEGA, BS_BB, BS_RR, BS_RELRES, BS_WORDS = 8 };

static Sten make_sten(iskra_ctx *c);

struct BiArgs {
  Sten s;
  const double *rho;
  double scale;
  const int *srow, *snb, *sdof;
  const double *sd, *sc, *ssig, *sigma, *dg;
  double *x, *r, *rh, *pp[2], *v[2], *sv, *tv;
  double *p0, *pa, *pt; /* partials: 3 x nblk (init / B4), nblk (B1), 2 x nblk (B3) */
  double *scal;
  int *iflag;
  int nblk, max_iter, warm;
  const double *phi_in;
  double rtol2;
};

/* row n of the unknowns' operator applied to get(m) (callers return 0 at
 * Dirichlet nodes, whose values are on the right-hand side) */
template <typename G>
__device__ __forceinline__ double bi_row(const BiArgs &a, int n, G get) {
  const int k = a.srow[n];
  if (k >= 0) {
    double acc = a.sd[k] * get(n);
    for (int q = 0; q < 2; ++q) {
      const int m = a.snb[2 * k + q];
      if (m >= 0) acc -= a.sc[2 * k + q] * get(m);
    }
    return acc;
  }
  const Sten &s = a.s;
  const int i = n % s.nx, j = n / s.nx;
  double acc = 0.0, diag = 0.0;
  if (i > 0) { acc += get(n - 1); diag += 1.0; }
  if (i < s.nx - 1) { acc += get(n + 1); diag += 1.0; }
  if (s.per_x) {
    if (i == 0) { acc += s.cxp * get(n + s.nx - 1); diag += s.cxp; }
    if (i == s.nx - 1) { acc += s.cxp * get(n - (s.nx - 1)); diag += s.cxp; }
  }
  if (s.dim == 2) {
    if (j > 0) { acc += get(n - s.nx); diag += 1.0; }
    if (j < s.ny - 1) { acc += get(n + s.nx); diag += 1.0; }
    if (s.per_y) {
      if (j == 0) { acc += s.cyp * get(n + (s.ny - 1) * s.nx); diag += s.cyp; }
      if (j == s.ny - 1) { acc += s.cyp * get(n - (s.ny - 1) * s.nx); diag += s.cyp; }
    }
  }
  return diag * get(n) - acc;
}

/* right-hand side of unknown n */
__device__ __forceinline__ double bi_rhs(const BiArgs &a, int n) {
  const double f = a.rho[n] * a.scale;
  const int k = a.srow[n];
  if (k >= 0) {
    double b = f + a.ssig[k] * a.sigma[a.sdof[k]];
    for (int q = 0; q < 2; ++q) {
      const int m = a.snb[2 * k + q];
      if (m >= 0 && a.s.tags[m] && a.srow[m] < 0) b += a.sc[2 * k + q] * a.s.tagval[a.s.tags[m]];
    }
    return b;
  }
  return f + dirichlet_rhs(a.s, n % a.s.nx, n / a.s.nx);
}

__global__ __launch_bounds__(RED_BLOCK) void k_bi_init(BiArgs a) {
  const int n = blockIdx.x * RED_BLOCK + threadIdx.x, nn = a.s.nx * a.s.ny;
  double rr = 0.0, bb = 0.0, rhor = 0.0;
  if (blockIdx.x == 0 && threadIdx.x < BS_WORDS) a.scal[threadIdx.x] = 0.0;
  if (n < nn) {
    const int t = a.s.tags[n];
    const bool unk = t == 0 || a.srow[n] >= 0;
    if (!unk) {
      a.x[n] = a.s.tagval[t];
      a.r[n] = a.rh[n] = 0.0;
    } else {
      const double x0 = a.warm ? a.phi_in[n] : 0.0;
      a.x[n] = x0;
      auto gx = [&](int m) -> double {
        return (a.s.tags[m] && a.srow[m] < 0) ? 0.0 : (a.warm ? a.phi_in[m] : 0.0);
      };
      const double b = bi_rhs(a, n);
      const double r = b - bi_row(a, n, gx);
      a.r[n] = r;
      a.rh[n] = r;
      rr = r * r;
      bb = b * b;
      rhor = r * r;
    }
    a.pp[1][n] = 0.0;
    a.v[1][n] = 0.0;
  }
  wg_sum3(rhor, bb, rr);
  if (threadIdx.x == 0) {
    a.p0[3 * blockIdx.x] = rhor;
    a.p0[3 * blockIdx.x + 1] = bb;
    a.p0[3 * blockIdx.x + 2] = rr;
  }
}

__global__ __launch_bounds__(RED_BLOCK) void k_bi_1(BiArgs a, int it) {
  __shared__ int s_stop;
  if (threadIdx.x == 0) s_stop = a.iflag[0];
  double rho = 0.0, bb = 0.0, rr = 0.0;
  for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) {
    rho += a.p0[3 * k];
    bb += a.p0[3 * k + 1];
    rr += a.p0[3 * k + 2];
  }
  wg_sum3(rho, bb, rr);
  if (s_stop) return;
  if (it > 0) bb = a.scal[BS_BB];
  const bool done = rr <= a.rtol2 * bb || it >= a.max_iter || !(rr == rr);
  double beta = 0.0;
  const double omega = a.scal[BS_OMEGA];
  if (it > 0) {
    const double rho_old = a.scal[BS_RHO0 + ((it - 1) & 1)];
    beta = (rho_old != 0.0 && omega != 0.0) ? (rho / rho_old) * (a.scal[BS_ALPHA] / omega) : 0.0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (it == 0) a.scal[BS_BB] = bb;
    a.scal[BS_RR] = rr;
    a.scal[BS_RELRES] = bb > 0.0 ? sqrt(rr / bb) : 0.0;
    a.scal[BS_RHO0 + (it & 1)] = rho;
    a.iflag[1] = it;
    if (done) a.iflag[0] = 1;
  }
  if (done) return;
  const double *pold = a.pp[(it + 1) & 1], *vold = a.v[(it + 1) & 1];
  double *pnew = a.pp[it & 1], *vnew = a.v[it & 1];
  const int n = blockIdx.x * RED_BLOCK + threadIdx.x, nn = a.s.nx * a.s.ny;
  double rv = 0.0, d1 = 0.0, d2 = 0.0;
  if (n < nn) {
    auto unk = [&](int m) { return a.s.tags[m] == 0 || a.srow[m] >= 0; };
    auto gp = [&](int m) -> double {
      if (!unk(m)) return 0.0;
      const double p = a.r[m] + beta * (pold[m] - omega * vold[m]);
      return p / a.dg[m];
    };
    if (unk(n)) {
      const double p = a.r[n] + beta * (pold[n] - omega * vold[n]);
      pnew[n] = p;
      const double v = bi_row(a, n, gp);
      vnew[n] = v;
      rv = a.rh[n] * v;
    } else {
      pnew[n] = 0.0;
      vnew[n] = 0.0;
    }
  }
  wg_sum3(rv, d1, d2);
  if (threadIdx.x == 0) a.pa[blockIdx.x] = rv;
}

__global__ __launch_bounds__(RED_BLOCK) void k_bi_2(BiArgs a, int it) {
  if (a.iflag[0]) return;
  double rv = 0.0, d1 = 0.0, d2 = 0.0;
  for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) rv += a.pa[k];
  wg_sum3(rv, d1, d2);
  const double rho = a.scal[BS_RHO0 + (it & 1)];
  const double alpha = rv != 0.0 ? rho / rv : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.scal[BS_ALPHA] = alpha;
    if (rv == 0.0) a.iflag[3] = 1; /* breakdown */
  }
  const int n = blockIdx.x * RED_BLOCK + threadIdx.x, nn = a.s.nx * a.s.ny;
  if (n < nn) a.sv[n] = a.r[n] - alpha * a.v[it & 1][n];
}

__global__ __launch_bounds__(RED_BLOCK) void k_bi_3(BiArgs a, int it) {
  if (a.iflag[0]) return;
  (void)it;
  const int n = blockIdx.x * RED_BLOCK + threadIdx.x, nn = a.s.nx * a.s.ny;
  double ts = 0.0, tt = 0.0, d2 = 0.0;
  if (n < nn) {
    auto unk = [&](int m) { return a.s.tags[m] == 0 || a.srow[m] >= 0; };
    if (unk(n)) {
      auto gs = [&](int m) -> double { return unk(m) ? a.sv[m] / a.dg[m] : 0.0; };
      const double t = bi_row(a, n, gs);
      a.tv[n] = t;
      ts = t * a.sv[n];
      tt = t * t;
    } else {
      a.tv[n] = 0.0;
    }
  }
  wg_sum3(ts, tt, d2);
  if (threadIdx.x == 0) {
    a.pt[2 * blockIdx.x] = ts;
    a.pt[2 * blockIdx.x + 1] = tt;
  }
}

__global__ __launch_bounds__(RED_BLOCK) void k_bi_4(BiArgs a, int it) {
  if (a.iflag[0]) return;
  double ts = 0.0, tt = 0.0, d2 = 0.0;
  for (int k = threadIdx.x; k < a.nblk; k += RED_BLOCK) {
    ts += a.pt[2 * k];
    tt += a.pt[2 * k + 1];
  }
  wg_sum3(ts, tt, d2);
  const double omega = tt != 0.0 ? ts / tt : 0.0;
  const double alpha = a.scal[BS_ALPHA];
  if (blockIdx.x == 0 && threadIdx.x == 0) a.scal[BS_OMEGA] = omega;
  const int n = blockIdx.x * RED_BLOCK + threadIdx.x, nn = a.s.nx * a.s.ny;
  double rhor = 0.0, rr = 0.0, z = 0.0;
  if (n < nn && (a.s.tags[n] == 0 || a.srow[n] >= 0)) {
    const double dg = a.dg[n];
    a.x[n] += alpha * (a.pp[it & 1][n] / dg) + omega * (a.sv[n] / dg);
    const double r = a.sv[n] - omega * a.tv[n];
    a.r[n] = r;
    rhor = a.rh[n] * r;
    rr = r * r;
  }
  wg_sum3(rhor, z, rr);
  if (threadIdx.x == 0) {
    a.p0[3 * blockIdx.x] = rhor;
    a.p0[3 * blockIdx.x + 1] = 0.0;
    a.p0[3 * blockIdx.x + 2] = rr;
  }
}

__global__ void k_bi_out(const double *x, double *phi, int nn) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < nn) phi[n] = x[n];
}

/* ------------------------------------------------------------------------ */
/* small systems: a whole Krylov solve in one work-group                     */
/* ------------------------------------------------------------------------ */
/* An iteration of the kernels above is bound by its dependent launches (two of
 * CG 10 us, four of BiCGStab 22 us, at any size up to some 60,000 nodes).  A
 * system whose vectors fit one CU is solved by one work-group instead: a thread
 * keeps the vectors of NPT consecutive nodes of one grid column in registers,
 * the vector the operator reads is in LDS with a ring of zeros around the grid,
 * and dot products go through the waves' sums in LDS, so an iteration is three
 * (five) barriers and is bound by one CU's FP64 rate.  Along a column the row
 * coefficients are constants of the thread and two of the five entries are the
 * neighbours just read: 30 instructions a node and iteration of CG, where nodes
 * dealt out by index took 65 (6.2 us an iteration on 12,513 nodes).  The
 * set-up, phi, E and the verdict are part of the same launch; the verdict goes
 * to host memory the host reads after its one wait.  Measured an iteration:
 * CG on 12,513 nodes 5.0 us (10.0 with two launches; 7.6 with the LDS array in
 * FP64, whose reads then bind), BiCGStab on 2401 nodes 5.0 us (21.8 with four;
 * 8.5 with 512 threads and the special rows read from memory).
 * The arithmetic is that of the kernels above (z = the FP32 rounding of an FP64 r / diag),
 * with the division as a product with the FP64 reciprocal; sums in another order. */
#define ONE_WAVES 16
/* LDS of the padded vector and tables; iterations one launch may take (0.1 s) */
#define ONE_LDS 64000
#define ONE_MAX_ITER 32768
/* nodes whose loads are in flight together: scheduled all at once they would
 * not fit the registers */
#define ONE_GROUP 6
#define ONE_STOP(k) \
  if ((k) % ONE_GROUP == ONE_GROUP - 1) __builtin_amdgcn_sched_barrier(0)

/* steps a running index down a column; hoisted out of the iterations, one
 * index per node would take as many registers as a vector */
#define ONE_NEXT(q, px) \
  do {                  \
    (q) += (px);        \
    asm volatile("" : "+v"(q)); \
  } while (0)

/* sum over the wave in the last lane: DPP row shifts and broadcasts (the
 * cross-lane moves of a shuffle butterfly go through LDS) */
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_sum_last(double v) {
  v = dpp_add<0x111, 0xf>(v); /* row_shr:1, 2, 4, 8 */
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v); /* row_bcast:15, 31 */
  return dpp_add<0x143, 0xc>(v);
}

/* sums of N values a thread over the work-group, in a fixed order; every
 * thread gets the totals.  One barrier: consecutive calls use different
 * buffers (part), and two calls of one buffer have another's barrier between. */
template <int BLK, int N>
__device__ __forceinline__ void one_sum(double *v, double (*part)[ONE_WAVES]) {
#pragma unroll
  for (int q = 0; q < N; ++q) {
    const double s = wave_sum_last(v[q]);
    if ((threadIdx.x & 63) == 63) part[q][threadIdx.x >> 6] = s;
  }
  isk_lds_barrier();
#pragma unroll
  for (int q = 0; q < N; ++q) {
    double s = part[q][0];
#pragma unroll
    for (int w = 1; w < BLK / 64; ++w) s += part[q][w];
    v[q] = s;
  }
}

/* a thread's part of the grid: rows j0 .. j0 + NPT - 1 of column i, the entry
 * of its first node in the padded array (rows of px entries, one ring of
 * zeros; rows past the grid are zero and so are their vectors), and the
 * constants of its rows: links lo, hi along x, cz along y, diag with both y
 * links (a missing one is made up for by taking the node's own value there) */
struct OneCol {
  int i, j0, q0, px, klast; /* klast: which of its rows is the grid's last */
  double lo, hi, cz, diag;
};

__host__ __device__ __forceinline__ int one_segs(int ny, int npt) { return (ny + npt - 1) / npt; }
/* entries of the padded array */
__host__ __device__ __forceinline__ int one_entries(int nx, int ny, int npt) {
  return (nx + 2) * (one_segs(ny, npt) * npt + 2);
}

template <int NPT, bool AXIAL>
__device__ __forceinline__ OneCol one_col(const Sten &s) {
  OneCol c;
  const int tid = threadIdx.x;
  c.px = s.nx + 2;
  c.i = tid % s.nx;
  const int seg = tid / s.nx;
  c.j0 = seg * NPT;
  c.klast = s.ny - 1 - c.j0;
  c.q0 = (c.j0 + 1) * c.px + c.i + 1;
  if (seg >= one_segs(s.ny, NPT)) { /* no part: the zero column left of the grid */
    c.i = -1;
    c.j0 = s.ny;
    c.klast = -1;
    c.q0 = c.px;
  }
  if (AXIAL) {
    c.lo = c.i > 0 ? (double)c.i - 0.5 : 0.0;
    c.hi = c.i < s.nx - 1 ? (double)c.i + 0.5 : 0.0;
    c.cz = isk_rz_w(c.i, s.nx) * s.az;
  } else {
    c.lo = c.i > 0 ? 1.0 : 0.0;
    c.hi = c.i < s.nx - 1 ? 1.0 : 0.0;
    c.cz = s.dim == 2 ? 1.0 : 0.0;
  }
  c.diag = c.lo + c.hi + 2.0 * c.cz;
  return c;
}
/* node index of the thread's first row (its row k is in the grid for k <= klast) */
__device__ __forceinline__ int one_node(const OneCol &c, const Sten &s) {
  return c.klast >= 0 ? c.j0 * s.nx + c.i : 0;
}

/* v = L p at the thread's nodes, 0 where bit k of `on` is (Dirichlet nodes and rows
 * past the grid have zero residual and so stay 0 in every vector, with no
 * branch, once their row is dropped); *pv = (p, v) */
template <int NPT, typename T>
__device__ __forceinline__ void one_apply(const OneCol &c, const T *p, unsigned on, double *v,
                                          double *pv) {
  double sum = 0.0;
  int q = c.q0;
  double pc = (double)p[q];
  double pd = c.j0 == 0 ? pc : (double)p[q - c.px];
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    double acc = c.lo * (double)p[q - 1];
    acc = __builtin_fma(c.hi, (double)p[q + 1], acc);
    ONE_NEXT(q, c.px);
    const double up = (double)p[q], pu = k == c.klast ? pc : up;
    acc = __builtin_fma(c.cz, pd + pu, acc);
    acc = __builtin_fma(c.diag, pc, -acc);
    v[k] = on >> k & 1 ? acc : 0.0;
    sum = __builtin_fma(pc, v[k], sum);
    pd = pc;
    pc = up;
    ONE_STOP(k);
  }
  *pv = sum;
}

struct CgOne {
  PcgArgs a;
  float *E;
  double dx, dy, rtol;
  double *mail;
};

/* Jacobi-preconditioned CG (k_pcg_setx ... k_pcg_out, then k_efield) */
template <int NPT, int BLK, bool AXIAL>
__global__ __launch_bounds__(BLK) void k_cg_one(CgOne c) {
  extern __shared__ float lp[];
  __shared__ double part[5][ONE_WAVES];
  const PcgArgs &a = c.a;
  const Sten s = a.s;
  const int nn = s.nx * s.ny, np = one_entries(s.nx, s.ny, NPT);
  const int tid = threadIdx.x;
  for (int k = tid; k < np; k += BLK) lp[k] = 0.0f;
  for (int n = tid; n < nn; n += BLK) {
    const int t = s.tags[n];
    a.x[n] = t ? s.tagval[t] : (a.warm ? a.phi_in[n] : 0.0);
  }
  __syncthreads();
  /* r by a rolled loop through memory */
  double sum[3] = {0.0, 0.0, 0.0}; /* (r,r), (r,z), (f,f) */
#pragma unroll 1
  for (int n = tid; n < nn; n += BLK) {
    double r0 = 0.0;
    if (s.tags[n] == 0) {
      const int i = n % s.nx, j = n / s.nx;
      double f = a.rho[n] * a.scale, diag;
      if (AXIAL) f *= isk_rz_w(i, s.nx);
      /* x holds the Dirichlet values, so L x already carries them */
      r0 = f - apply_L(s, a.x, i, j, &diag);
      const double fe = f + dirichlet_rhs(s, i, j);
      sum[0] += r0 * r0;
      sum[1] += r0 * (double)(float)(r0 / diag);
      sum[2] += fe * fe;
    }
    a.r[n] = r0;
  }
  __syncthreads();
  const OneCol col = one_col<NPT, AXIAL>(s);
  const int px = col.px;
  double x[NPT], r[NPT], ap[NPT];
  unsigned on = 0;
#pragma unroll
  for (int k = 0, n = one_node(col, s); k < NPT; ++k) {
    const bool in = k <= col.klast;
    x[k] = in ? a.x[n] : 0.0;
    r[k] = in ? a.r[n] : 0.0;
    if (in && s.tags[n] == 0) on |= 1u << k;
    ONE_NEXT(n, s.nx);
    ONE_STOP(k);
  }
  one_sum<BLK, 3>(sum, part);
  /* reciprocal diagonals of the column: its first and last row lack a link */
  const double inv = 1.0 / col.diag;
  const double inv0 = 1.0 / (col.j0 == 0 ? col.diag - col.cz : col.diag);
  const double invl = 1.0 / (col.diag - (s.ny > 1 ? col.cz : 2.0 * col.cz));
  /* z waits in ap, which is free between the update of r and the next L p: another
   * array would not fit the registers (kl: klast, and on, opaque so that nothing a row
   * is kept over the iterations) */
  int kl = col.klast;
  auto z = [&](int k) {
    return (double)(float)(r[k] * (k == kl ? invl : k == 0 ? inv0 : inv));
  };
  const double ff = sum[2], tol2 = c.rtol * c.rtol * ff;
  double rr = sum[0], rz = sum[1], rz_old = 0.0;
#pragma unroll
  for (int k = 0; k < NPT; ++k) ap[k] = z(k);
  int it = 0;
  for (; !(rr <= tol2) && it < a.max_iter; ++it) {
    const float beta = (float)(it > 0 && rz_old != 0.0 ? rz / rz_old : 0.0);
#pragma unroll
    for (int k = 0, q = col.q0; k < NPT; ++k) {
      lp[q] = fmaf(beta, lp[q], (float)ap[k]);
      ONE_NEXT(q, px);
      ONE_STOP(k);
    }
    isk_lds_barrier();
    double pap;
    one_apply<NPT>(col, lp, on, ap, &pap);
    one_sum<BLK, 1>(&pap, part + (it & 1 ? 3 : 0));
    const double alpha = pap != 0.0 ? rz / pap : 0.0;
    double t[2] = {0.0, 0.0};
    asm volatile("" : "+v"(kl), "+v"(on));
#pragma unroll
    for (int k = 0, q = col.q0; k < NPT; ++k) {
      x[k] = __builtin_fma(alpha, (double)lp[q], x[k]);
      ONE_NEXT(q, px);
      r[k] = __builtin_fma(-alpha, ap[k], r[k]);
      t[0] = __builtin_fma(r[k], r[k], t[0]);
      ap[k] = z(k);
      t[1] = __builtin_fma(r[k], ap[k], t[1]);
      ONE_STOP(k);
    }
    one_sum<BLK, 2>(t, part + 1);
    rz_old = rz;
    rr = t[0];
    rz = t[1];
  }
#pragma unroll
  for (int k = 0, n = one_node(col, s); k < NPT; ++k) {
    if (k <= col.klast) a.phi_out[n] = x[k];
    ONE_NEXT(n, s.nx);
  }
  const double rel = ff > 0.0 ? sqrt(rr / ff) : 0.0;
  if (tid == 0) {
    c.mail[MAIL_ITERS] = (double)it;
    c.mail[MAIL_RELRES] = rel;
    c.mail[MAIL_BREAK] = 0.0;
  }
  if (!c.E || !(rel <= c.rtol)) return; /* a solve that failed leaves E as it was */
  __syncthreads();
  for (int n = tid; n < nn; n += BLK)
    efield_node(a.phi_out, c.E, s.dim, s.nx, s.ny, c.dx, c.dy, n);
}

struct BiOne {
  BiArgs a;
  int nspec; /* special rows */
  double *phi;
  float *E;
  double dx, dy, rtol;
  double *mail;
};

/* a special row in LDS: its factors, and its neighbours' entries in the padded
 * array (a missing one has factor 0) */
struct BiSpec {
  double sd, sc0, sc1;
  int q0, q1;
};

/* v = A (padded array) at the thread's nodes: the 5-point rows, then the few
 * special ones from their own links (sid: a node's row of the table) */
template <int NPT>
__device__ __forceinline__ void bi_one_apply(const OneCol &c, unsigned on, unsigned spec,
                                             const BiSpec *tab, const unsigned short *sid,
                                             const double *p, double *v) {
  double pv;
  one_apply<NPT>(c, p, on, v, &pv);
  if (spec) {
#pragma unroll
    for (int k = 0; k < NPT; ++k)
      if (spec >> k & 1) {
        const BiSpec &w = tab[sid[c.q0 + k * c.px]];
        v[k] = w.sd * p[c.q0 + k * c.px] - w.sc0 * p[w.q0] - w.sc1 * p[w.q1];
      }
  }
}

/* right-preconditioned BiCGStab (k_bi_init ... k_bi_out, then k_efield) */
template <int NPT, int BLK>
__global__ __launch_bounds__(BLK) void k_bi_one(BiOne c) {
  extern __shared__ double lk[]; /* K^-1 p, then K^-1 s; the special rows' table */
  __shared__ double part[6][ONE_WAVES];
  const BiArgs &a = c.a;
  const Sten s = a.s;
  const int nn = s.nx * s.ny, np = one_entries(s.nx, s.ny, NPT);
  const int tid = threadIdx.x;
  BiSpec *tab = reinterpret_cast<BiSpec *>(lk + np);
  unsigned short *sid = reinterpret_cast<unsigned short *>(tab + c.nspec);
  for (int k = tid; k < np; k += BLK) lk[k] = 0.0;
  for (int k = tid; k < c.nspec; k += BLK) {
    BiSpec w;
    const int m0 = a.snb[2 * k], m1 = a.snb[2 * k + 1];
    w.sd = a.sd[k];
    w.sc0 = m0 >= 0 ? a.sc[2 * k] : 0.0;
    w.sc1 = m1 >= 0 ? a.sc[2 * k + 1] : 0.0;
    w.q0 = m0 >= 0 ? (m0 / s.nx + 1) * (s.nx + 2) + m0 % s.nx + 1 : 0;
    w.q1 = m1 >= 0 ? (m1 / s.nx + 1) * (s.nx + 2) + m1 % s.nx + 1 : 0;
    tab[k] = w;
  }
  __syncthreads();
  /* x into the padded array (Dirichlet nodes stay 0 there: their values are on
   * the right-hand side), the right-hand side through memory */
#pragma unroll 1
  for (int n = tid; n < nn; n += BLK) {
    const int tg = s.tags[n];
    double b = 0.0, iv = 0.0, x0;
    if (tg == 0 || a.srow[n] >= 0) {
      x0 = a.warm ? a.phi_in[n] : 0.0;
      iv = 1.0 / a.dg[n];
      const int q = (n / s.nx + 1) * (s.nx + 2) + n % s.nx + 1;
      lk[q] = x0;
      sid[q] = (unsigned short)max(a.srow[n], 0);
      b = bi_rhs(a, n);
    } else {
      x0 = s.tagval[tg];
    }
    a.x[n] = x0;
    a.r[n] = b;
    a.tv[n] = iv;
  }
  __syncthreads();
  const OneCol col = one_col<NPT, false>(s);
  const int px = col.px;
  double x[NPT], r[NPT], rh[NPT], p[NPT], v[NPT], t[NPT], inv[NPT];
  unsigned spec = 0, on = 0;
#pragma unroll
  for (int k = 0, n = one_node(col, s); k < NPT; ++k) {
    const bool in = k <= col.klast;
    p[k] = v[k] = 0.0;
    x[k] = in ? a.x[n] : 0.0;
    r[k] = in ? a.r[n] : 0.0;
    inv[k] = in ? a.tv[n] : 0.0;
    if (inv[k] != 0.0) on |= 1u << k;
    if (in && a.srow[n] >= 0) spec |= 1u << k;
    ONE_NEXT(n, s.nx);
    ONE_STOP(k);
  }
  bi_one_apply<NPT>(col, on, spec, tab, sid, lk, t);
  double sum[3] = {0.0, 0.0, 0.0}; /* (rh,r), (b,b), (r,r) */
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    sum[1] += r[k] * r[k];
    rh[k] = r[k] = r[k] - t[k];
    sum[2] += r[k] * r[k];
  }
  sum[0] = sum[2];
  one_sum<BLK, 3>(sum, part);
  double rho = sum[0], rho_old = 0.0, rr = sum[2], alpha = 0.0, omega = 0.0;
  const double bb = sum[1];
  int it = 0, broke = 0;
  for (; !(rr <= a.rtol2 * bb) && it < a.max_iter && rr == rr; ++it) {
    const double beta =
        it > 0 && rho_old != 0.0 && omega != 0.0 ? (rho / rho_old) * (alpha / omega) : 0.0;
#pragma unroll
    for (int k = 0, q = col.q0; k < NPT; ++k) {
      p[k] = r[k] + beta * (p[k] - omega * v[k]);
      lk[q] = p[k] * inv[k];
      ONE_NEXT(q, px);
    }
    isk_lds_barrier();
    bi_one_apply<NPT>(col, on, spec, tab, sid, lk, v);
    double rv = 0.0;
#pragma unroll
    for (int k = 0; k < NPT; ++k) rv = __builtin_fma(rh[k], v[k], rv);
    one_sum<BLK, 1>(&rv, part + 5);
    alpha = rv != 0.0 ? rho / rv : 0.0;
    if (rv == 0.0) broke = 1;
    /* s in r; K^-1 s takes K^-1 p's place once x has taken that */
#pragma unroll
    for (int k = 0, q = col.q0; k < NPT; ++k) {
      x[k] = __builtin_fma(alpha, lk[q], x[k]);
      r[k] = r[k] - alpha * v[k];
      lk[q] = r[k] * inv[k];
      ONE_NEXT(q, px);
    }
    isk_lds_barrier();
    bi_one_apply<NPT>(col, on, spec, tab, sid, lk, t);
    double ts[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      ts[0] = __builtin_fma(t[k], r[k], ts[0]);
      ts[1] = __builtin_fma(t[k], t[k], ts[1]);
    }
    one_sum<BLK, 2>(ts, part + 3);
    omega = ts[1] != 0.0 ? ts[0] / ts[1] : 0.0;
    double u[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0, q = col.q0; k < NPT; ++k) {
      x[k] = __builtin_fma(omega, lk[q], x[k]);
      ONE_NEXT(q, px);
      r[k] = r[k] - omega * t[k];
      u[0] = __builtin_fma(rh[k], r[k], u[0]);
      u[1] = __builtin_fma(r[k], r[k], u[1]);
    }
    one_sum<BLK, 2>(u, part);
    rho_old = rho;
    rho = u[0];
    rr = u[1];
  }
#pragma unroll
  for (int k = 0, n = one_node(col, s); k < NPT; ++k) {
    if (k <= col.klast) c.phi[n] = x[k];
    ONE_NEXT(n, s.nx);
  }
  const double rel = bb > 0.0 ? sqrt(rr / bb) : 0.0;
  if (tid == 0) {
    c.mail[MAIL_ITERS] = (double)it;
    c.mail[MAIL_RELRES] = rel;
    c.mail[MAIL_BREAK] = (double)broke;
  }
  if (!c.E || !(rel <= c.rtol)) return; /* a solve that failed leaves E as it was */
  __syncthreads();
  for (int n = tid; n < nn; n += BLK)
    efield_node(c.phi, c.E, s.dim, s.nx, s.ny, c.dx, c.dy, n);
}

/* nodes a thread for a system the one-work-group solvers take, 0 for any other:
 * no periodic link (the ring of zeros stands for the edges), every column
 * segment a thread of its own, and the padded array (`entry` bytes each) and `extra` bytes in LDS.
 * The first shape whose threads cover the grid: 1024 threads while the vectors fit
 * 128 VGPRs (more waves hide the latencies of LDS and FP64), then 512, which cover more
 * than 1024 with 8 (4) nodes only from 17 (9) nodes on */
struct OneShape {
  int npt, block;
};
static const OneShape one_cg_shapes[] = {{2, 1024}, {4, 1024}, {8, 1024}, {19, 512}, {26, 512},
                                         {0, 0}};
static const OneShape one_bi_shapes[] = {{2, 1024}, {4, 1024}, {10, 512}, {0, 0}};

static int one_npt(const iskra_ctx *c, const OneShape *shapes, size_t entry, size_t extra,
                   size_t *shm) {
  const IskPoisson &p = c->ps;
  if (p.per_x || p.per_y || p.singular || p.max_iter > ONE_MAX_ITER) return 0;
  for (; shapes->npt; ++shapes)
    if (c->g.nx * one_segs(c->g.ny, shapes->npt) <= shapes->block) {
      const size_t n = one_entries(c->g.nx, c->g.ny, shapes->npt);
      *shm = n * entry + extra;
      return *shm <= ONE_LDS ? shapes->npt : 0;
    }
  return 0;
}

/* the verdict of a one-work-group solve (waits for the stream) */
static int one_result(iskra_ctx *c, int *iters, double *relres, int *broke) {
  ISK_HIP(hipStreamSynchronize(c->stream));
  *iters = (int)c->mail[MAIL_ITERS];
  *relres = c->mail[MAIL_RELRES];
  *broke = c->mail[MAIL_BREAK] != 0.0;
  return ISKRA_OK;
}

/* E != null: may form E = -grad(phi) too, and then sets *E_done */
int isk_bicgstab_solve(iskra_ctx *c, int warm, int *iters, double *relres, float *E,
                       int *E_done) {
  IskPoisson &p = c->ps;
  const int nn = isk_nodes(c), nblk = (nn + RED_BLOCK - 1) / RED_BLOCK;
  BiArgs a;
  a.s = make_sten(c);
  a.rho = c->rho;
  a.scale = (c->g.dx * c->g.dx) / p.eps0;
  a.srow = p.d_srow;
  a.snb = p.d_snb;
  a.sdof = p.d_sdof;
  a.sd = p.d_sd;
  a.sc = p.d_sc;
  a.ssig = p.d_ssig;
  a.sigma = c->d_elec + EL_SIGMA;
  a.dg = p.d_dg;
  double *b = p.bi;
  a.x = p.x;
  a.r = b;
  a.rh = b + nn;
  a.pp[0] = b + 2 * (size_t)nn;
  a.pp[1] = b + 3 * (size_t)nn;
  a.v[0] = b + 4 * (size_t)nn;
  a.v[1] = b + 5 * (size_t)nn;
  a.sv = b + 6 * (size_t)nn;
  a.tv = b + 7 * (size_t)nn;
  a.p0 = b + 8 * (size_t)nn;
  a.pa = a.p0 + 3 * nblk;
  a.pt = a.pa + nblk;
  a.scal = a.pt + 2 * nblk;
  a.iflag = p.iflag;
  a.nblk = nblk;
  a.max_iter = p.max_iter;
  a.warm = warm == ISKRA_WARM_PREV ? 1 : 0;
  a.phi_in = c->phi;
  a.rtol2 = p.rtol * p.rtol;
  int it = 0, hflag[4] = {0, 0, 0, 0}, n_it = 0, broke = 0;
  double rel = 0.0;
  size_t shm = 0;
  const int nspec = (int)p.h_sd.size();
  const size_t sid_bytes = 2 * (size_t)(c->g.nx + 2) * (c->g.ny + 1); /* read inside the grid only */
  const int npt = one_npt(c, one_bi_shapes, sizeof(double), nspec * sizeof(BiSpec) + sid_bytes, &shm);
  const bool one = npt > 0;
  if (one) {
    BiOne o;
    o.a = a;
    o.nspec = nspec;
    o.phi = c->phi;
    o.E = E;
    o.dx = c->g.dx;
    o.dy = c->g.dy;
    o.rtol = p.rtol;
    o.mail = c->mail;
    auto k = npt == 2 ? k_bi_one<2, 1024> : npt == 4 ? k_bi_one<4, 1024> : k_bi_one<10, 512>;
    hipLaunchKernelGGL(k, dim3(1), dim3(npt <= 4 ? 1024 : 512), shm, c->stream, o);
    ISK_CHECK_LAUNCH();
    if (E) *E_done = 1;
    int rc = one_result(c, &n_it, &rel, &broke);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(64), 0, c->stream, p.scal, p.iflag, 0.0, 0);
    hipLaunchKernelGGL(k_bi_init, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a);
    ISK_CHECK_LAUNCH();
  }
  while (!one) {
    for (int k = 0; k < 8; ++k, ++it) {
      hipLaunchKernelGGL(k_bi_1, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it);
      hipLaunchKernelGGL(k_bi_2, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it);
      hipLaunchKernelGGL(k_bi_3, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it);
      hipLaunchKernelGGL(k_bi_4, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it);
      ISK_CHECK_LAUNCH();
    }
    ISK_HIP(hipMemcpyAsync(hflag, p.iflag, sizeof(hflag), hipMemcpyDeviceToHost, c->stream));
    ISK_HIP(hipStreamSynchronize(c->stream));
    if (hflag[0]) break;
    if (it > p.max_iter + 16) {
      isk_set_error("poisson: BiCGStab stopped after %d host iterations without a verdict", it);
      return ISKRA_E_CONVERGE;
    }
  }
  if (!one) {
    double sc[BS_WORDS];
    ISK_HIP(hipMemcpy(sc, a.scal, sizeof(sc), hipMemcpyDeviceToHost));
    hipLaunchKernelGGL(k_bi_out, dim3((nn + 255) / 256), dim3(256), 0, c->stream, p.x, c->phi,
                       nn);
    ISK_CHECK_LAUNCH();
    n_it = hflag[1];
    broke = hflag[3];
    rel = sc[BS_RELRES];
  }
  p.last_iters = n_it;
  p.last_relres = rel;
  c->stats.poisson_solves++;
  c->stats.poisson_iters += n_it;
  c->stats.last_iters = n_it;
  c->stats.last_relres = rel;
  if (iters) *iters = n_it;
  if (relres) *relres = rel;
  if (!(rel <= p.rtol)) {
    isk_set_error("poisson: BiCGStab reached relative residual %.3g > %.3g after %d iterations%s",
                  rel, p.rtol, n_it, broke ? " (breakdown)" : "");
    return ISKRA_E_CONVERGE;
  }
  return ISKRA_OK;
}

int isk_poisson_free(iskra_ctx *c) {
  IskPoisson &p = c->ps;
  void *ptrs[] = {p.d_tags, p.d_tag_val, p.d_tri_a, p.d_tri_cp, p.d_tri_inv,
                  p.d_tri_ma, p.d_tri_ncp, p.d_work, p.x, p.r, p.Ap, p.z, p.p[0], p.p[1], p.scal,
                  p.partials, p.cgp, p.iflag, p.sp_Sx, p.sp_Sy, p.sp_Li,
                  p.sp_F, p.sp_T1, p.sp_T2, p.d_srow, p.d_snb, p.d_sdof, p.d_sd,
                  p.d_sc, p.d_ssig, p.bi, p.d_dg};
  for (void *q : ptrs) isk_free(q);
  p.d_srow = p.d_snb = p.d_sdof = nullptr;
  p.d_sd = p.d_sc = p.d_ssig = p.bi = p.d_dg = nullptr;
  p.sp_Sx = p.sp_Sy = p.sp_Li = p.sp_F = p.sp_T1 = p.sp_T2 = nullptr;
  p.sp_nx = p.sp_ny = 0;
  for (int l = 0; l < p.nlev; ++l) {
    isk_free(p.me[l]);
    isk_free(p.mo[l]);
    p.mo[l] = nullptr;
    isk_free(p.mf[l]);
  }
  p.d_tags = nullptr;
  p.d_tag_val = nullptr;
  p.d_tri_a = p.d_tri_cp = p.d_tri_inv = p.d_tri_ma = p.d_tri_ncp = p.d_work = nullptr;
  p.x = p.r = p.Ap = nullptr;
  p.z = p.p[0] = p.p[1] = nullptr;
  p.scal = p.partials = p.cgp = nullptr;
  p.iflag = nullptr;
  p.nlev = 0;
  return ISKRA_OK;
}

static Sten make_sten(iskra_ctx *c) {
  Sten s;
  s.dim = c->g.dim;
  s.nx = c->g.nx;
  s.ny = c->g.ny;
  s.per_x = c->ps.per_x;
  s.per_y = c->ps.per_y;
  /* apply_periodic axis labels: wrapping i uses dy^2, wrapping j uses dx^2
   * (generalized_poisson.jl:291-323); in 1-D the ring uses dx^2 (:279-283);
   * all entries were divided by dx^2 at assembly (:65) */
  s.cxp = c->g.dim == 2 ? (c->g.dx * c->g.dx) / (c->g.dy * c->g.dy) : 1.0;
  s.cyp = 1.0;
  s.tags = c->ps.d_tags;
  s.tagval = c->ps.d_tag_val;
  s.axial = c->g.axial;
  s.az = c->g.axial ? (c->g.dx * c->g.dx) / (c->g.dy * c->g.dy) : 1.0;
  return s;
}

int isk_poisson_setup(iskra_ctx *c) {
  IskPoisson &p = c->ps;
  const int nn = isk_nodes(c);
  int ndir = 0, interior_tag = 0;
  for (int k = 0; k < nn; ++k) {
    if (p.tags[k]) {
      ++ndir;
      int i = k % c->g.nx, j = k / c->g.nx;
      bool edge = i == 0 || i == c->g.nx - 1 ||
                  (c->g.dim == 2 && (j == 0 || j == c->g.ny - 1));
      if (!edge) interior_tag = 1;
    }
  }
  p.singular = ndir == 0;
  if (c->g.axial) {
    /* the axisymmetric operator (generalized_poisson.jl:70-199) is solved by
     * CG on its symmetric weighted form only */
    if (p.kind != ISKRA_POISSON_PCG) {
      isk_set_error("poisson: an axial grid is solved by PCG only");
      return ISKRA_E_UNSUPPORTED;
    }
    if (p.per_x || p.per_y) {
      isk_set_error("poisson: no periodic link on an axial grid (the reference's "
                    "apply_periodic for RZ cannot run)");
      return ISKRA_E_UNSUPPORTED;
    }
    if (p.singular) {
      isk_set_error("poisson: an axial grid needs a Dirichlet node (the reference's "
                    "matrix is singular without one)");
      return ISKRA_E_UNSUPPORTED;
    }
  }
  if (isk_alloc((void **)&p.d_tags, nn)) return ISKRA_E_HIP;
  ISK_HIP(hipMemcpy(p.d_tags, p.tags.data(), nn, hipMemcpyHostToDevice));
  if (isk_alloc((void **)&p.d_tag_val, sizeof(double) * (ISK_MAX_TAGS + 1))) return ISKRA_E_HIP;
  ISK_HIP(hipMemcpy(p.d_tag_val, p.tag_val, sizeof(double) * (ISK_MAX_TAGS + 1),
                    hipMemcpyHostToDevice));
  if (p.kind == ISKRA_POISSON_DIRECT) {
    if (c->g.dim != 1) {
      isk_set_error("poisson: DIRECT is the 1-D tridiagonal solver; use PCG/MG in 2-D");
      return ISKRA_E_UNSUPPORTED;
    }
    if (p.per_x && !p.singular) {
      isk_set_error("poisson: periodic ring with Dirichlet nodes is not supported by DIRECT; use PCG");
      return ISKRA_E_UNSUPPORTED;
    }
    const int n = c->g.nx;
    std::vector<double> a(n, 0.0), d(n, 0.0), cc(n, 0.0), cp(n, 0.0), inv(n, 0.0);
    if (!p.singular) {
      for (int i = 0; i < n; ++i) {
        if (p.tags[i]) {
          d[i] = 1.0;
          continue;
        }
        a[i] = i > 0 ? 1.0 : 0.0;
        cc[i] = i < n - 1 ? 1.0 : 0.0;
        d[i] = -(a[i] + cc[i]);
      }
      /* elimination: inv_i = 1/(d_i - a_i cp_{i-1}), cp_i = c_i inv_i */
      double cprev = 0.0;
      for (int i = 0; i < n; ++i) {
        double den = d[i] - a[i] * cprev;
        if (den == 0.0) {
          isk_set_error("poisson: singular tridiagonal system (row %d)", i);
          return ISKRA_E_ARG;
        }
        inv[i] = 1.0 / den;
        cp[i] = cc[i] * inv[i];
        cprev = cp[i];
      }
    } else {
      /* ring, node 0 pinned: rows 1..n-1, each with two neighbours */
      double cprev = 0.0;
      for (int i = 1; i < n; ++i) {
        a[i] = i > 1 ? 1.0 : 0.0;
        cc[i] = i < n - 1 ? 1.0 : 0.0;
        d[i] = -2.0;
        double den = d[i] - a[i] * cprev;
        inv[i] = 1.0 / den;
        cp[i] = cc[i] * inv[i];
        cprev = cp[i];
      }
    }
    std::vector<double> ma(n), ncp(n);
    for (int i = 0; i < n; ++i) {
      ma[i] = -a[i] * inv[i];
      ncp[i] = -cp[i];
    }
    if (isk_alloc((void **)&p.d_tri_a, n * 8) || isk_alloc((void **)&p.d_tri_cp, n * 8) ||
        isk_alloc((void **)&p.d_tri_inv, n * 8) || isk_alloc((void **)&p.d_tri_ma, n * 8) ||
        isk_alloc((void **)&p.d_tri_ncp, n * 8) || isk_alloc((void **)&p.d_work, n * 8))
      return ISKRA_E_HIP;
    ISK_HIP(hipMemcpy(p.d_tri_ma, ma.data(), n * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_tri_ncp, ncp.data(), n * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_tri_a, a.data(), n * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_tri_cp, cp.data(), n * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_tri_inv, inv.data(), n * 8, hipMemcpyHostToDevice));
    return ISKRA_OK;
  }
  /* iterative solvers */
  int nblk = (nn + RED_BLOCK - 1) / RED_BLOCK;
  {
    /* the finest fused multigrid kernel reduces over one block per tile */
    int cx = (c->g.nx - 1) / 2 + 1, cy = c->g.dim == 2 ? (c->g.ny - 1) / 2 + 1 : 1;
    int tiles = ((cx + MGT_CT - 1) / MGT_CT) * ((cy + MGT_CT - 1) / MGT_CT);
    p.partials_blocks = std::max({nblk, tiles, (int)c->g.ny}); /* at most a row each */
  }
  if (isk_alloc((void **)&p.x, nn * 8) || isk_alloc((void **)&p.r, nn * 8) ||
      isk_alloc((void **)&p.Ap, nn * 8) || isk_alloc((void **)&p.z, nn * 4) ||
      isk_alloc((void **)&p.p[0], nn * 4) || isk_alloc((void **)&p.p[1], nn * 4) ||
      isk_alloc((void **)&p.scal, S_WORDS * 8) ||
      isk_alloc((void **)&p.partials, (size_t)p.partials_blocks * 2 * 8) ||
      isk_alloc((void **)&p.cgp, (size_t)nblk * 7 * 8) ||
      isk_alloc((void **)&p.iflag, 64))
    return ISKRA_E_HIP;
  ISK_HIP(hipMemset(p.iflag, 0, 64));
  p.nlev = 0;
  if (!p.h_sd.empty()) {
    /* floating electrodes: apply_neumann rows, solved by BiCGStab */
    if (c->g.dim != 2 || c->g.axial ||
        (p.kind != ISKRA_POISSON_PCG && p.kind != ISKRA_POISSON_MGPCG)) {
      isk_set_error("poisson: floating electrodes need a 2-D Cartesian grid and the PCG kind "
                    "(their rows make the system non-symmetric: BiCGStab solves it)");
      return ISKRA_E_UNSUPPORTED;
    }
    const int ns = (int)p.h_sd.size();
    std::vector<double> dg(nn);
    for (int k = 0; k < nn; ++k) {
      if (p.h_srow[k] >= 0) {
        dg[k] = p.h_sd[p.h_srow[k]];
        continue;
      }
      const int i = k % c->g.nx, j = k / c->g.nx;
      double d = 0.0;
      if (i > 0) d += 1.0;
      if (i < c->g.nx - 1) d += 1.0;
      if (p.per_x && (i == 0 || i == c->g.nx - 1)) d += (c->g.dx * c->g.dx) / (c->g.dy * c->g.dy);
      if (j > 0) d += 1.0;
      if (j < c->g.ny - 1) d += 1.0;
      if (p.per_y && (j == 0 || j == c->g.ny - 1)) d += 1.0;
      dg[k] = d > 0.0 ? d : 1.0;
    }
    const size_t nbuf = (size_t)8 * nn + 6 * (size_t)nblk + 16;
    if (isk_alloc((void **)&p.d_srow, (size_t)nn * 4) ||
        isk_alloc((void **)&p.d_snb, (size_t)2 * ns * 4) ||
        isk_alloc((void **)&p.d_sdof, (size_t)ns * 4) || isk_alloc((void **)&p.d_sd, (size_t)ns * 8) ||
        isk_alloc((void **)&p.d_sc, (size_t)2 * ns * 8) ||
        isk_alloc((void **)&p.d_ssig, (size_t)ns * 8) ||
        isk_alloc((void **)&p.d_dg, (size_t)nn * 8) || isk_alloc((void **)&p.bi, nbuf * 8))
      return ISKRA_E_HIP;
    ISK_HIP(hipMemcpy(p.d_srow, p.h_srow.data(), (size_t)nn * 4, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_snb, p.h_snb.data(), (size_t)2 * ns * 4, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_sdof, p.h_sdof.data(), (size_t)ns * 4, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_sd, p.h_sd.data(), (size_t)ns * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_sc, p.h_sc.data(), (size_t)2 * ns * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_ssig, p.h_ssig.data(), (size_t)ns * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.d_dg, dg.data(), (size_t)nn * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemset(p.bi, 0, nbuf * 8));
    return ISKRA_OK;
  }
  if (p.kind == ISKRA_POISSON_SPECTRAL) {
    if (c->g.dim != 2 || p.per_x || p.per_y || interior_tag) {
      isk_set_error("poisson: the spectral solve needs a 2-D grid with Dirichlet walls only");
      return ISKRA_E_UNSUPPORTED;
    }
    for (int k = 0; k < nn; ++k) {
      int i = k % c->g.nx, j = k / c->g.nx;
      bool edge = i == 0 || i == c->g.nx - 1 || j == 0 || j == c->g.ny - 1;
      if (edge && !p.tags[k]) {
        isk_set_error("poisson: the spectral solve needs Dirichlet values on all four walls");
        return ISKRA_E_UNSUPPORTED;
      }
    }
    const int mx = c->g.nx - 2, my = c->g.ny - 2;
    if (mx < 1 || my < 1) {
      isk_set_error("poisson: the spectral solve needs interior nodes");
      return ISKRA_E_ARG;
    }
    /* S[a][b] = sqrt(2/(m+1)) sin(pi (a+1)(b+1)/(m+1)): symmetric, S S = I;
     * eigenvalues of the unit 5-point operator: (2-2cos pi p/(mx+1)) + (2-2cos pi q/(my+1)) */
    auto basis = [](int m, std::vector<double> &S) {
      S.assign((size_t)m * m, 0.0);
      const double c0 = sqrt(2.0 / (m + 1)), w = M_PI / (m + 1);
      for (int a = 0; a < m; ++a)
        for (int b = 0; b < m; ++b) {
          /* reduce (a+1)(b+1) modulo 2(m+1) so the sine argument stays small */
          long long k = (long long)(a + 1) * (b + 1) % (2ll * (m + 1));
          S[(size_t)a * m + b] = c0 * sin(w * (double)k);
        }
    };
    std::vector<double> Sx, Sy, Li((size_t)mx * my);
    basis(mx, Sx);
    basis(my, Sy);
    for (int q = 0; q < my; ++q)
      for (int pp = 0; pp < mx; ++pp) {
        double lx = 2.0 - 2.0 * cos(M_PI * (pp + 1) / (mx + 1));
        double ly = 2.0 - 2.0 * cos(M_PI * (q + 1) / (my + 1));
        Li[(size_t)q * mx + pp] = 1.0 / (lx + ly);
      }
    size_t m2 = (size_t)mx * my;
    if (isk_alloc((void **)&p.sp_Sx, (size_t)mx * mx * 8) ||
        isk_alloc((void **)&p.sp_Sy, (size_t)my * my * 8) ||
        isk_alloc((void **)&p.sp_Li, m2 * 8) || isk_alloc((void **)&p.sp_F, m2 * 8) ||
        isk_alloc((void **)&p.sp_T1, m2 * 8) || isk_alloc((void **)&p.sp_T2, m2 * 8))
      return ISKRA_E_HIP;
    ISK_HIP(hipMemcpy(p.sp_Sx, Sx.data(), (size_t)mx * mx * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.sp_Sy, Sy.data(), (size_t)my * my * 8, hipMemcpyHostToDevice));
    ISK_HIP(hipMemcpy(p.sp_Li, Li.data(), m2 * 8, hipMemcpyHostToDevice));
    p.sp_nx = mx;
    p.sp_ny = my;
    return ISKRA_OK;
  }
  if (p.kind == ISKRA_POISSON_MG || p.kind == ISKRA_POISSON_MGPCG) {
    if (c->g.dim != 2 || p.per_x || p.per_y || interior_tag) {
      isk_set_error("poisson: multigrid needs a 2-D grid with Dirichlet walls only");
      return ISKRA_E_UNSUPPORTED;
    }
    /* every edge node must be Dirichlet */
    for (int k = 0; k < nn; ++k) {
      int i = k % c->g.nx, j = k / c->g.nx;
      bool edge = i == 0 || i == c->g.nx - 1 || j == 0 || j == c->g.ny - 1;
      if (edge && !p.tags[k]) {
        isk_set_error("poisson: multigrid needs Dirichlet values on all four walls");
        return ISKRA_E_UNSUPPORTED;
      }
    }
    if (fabs(c->g.dx - c->g.dy) > 1e-12 * c->g.dx) {
      /* the reference scales all links by 1/dx^2 (isotropic stencil): fine */
    }
    int nx = c->g.nx, ny = c->g.ny;
    int l = 0;
    p.ln[0] = nx;
    while (true) {
      if (isk_alloc((void **)&p.me[l], (size_t)nx * ny * 4) ||
          isk_alloc((void **)&p.mf[l], (size_t)nx * ny * 4))
        return ISKRA_E_HIP;
      p.ln[l] = nx | (ny << 16);
      ++l;
      if ((nx - 1) % 2 || (ny - 1) % 2 || nx <= 3 || ny <= 3 || l >= 12) break;
      nx = (nx - 1) / 2 + 1;
      ny = (ny - 1) / 2 + 1;
    }
    p.nlev = l;
    /* first level that fits the single work-group coarse solver */
    int cl = 0;
    while (cl < p.nlev) {
      int cx = p.ln[cl] & 0xFFFF, cy = p.ln[cl] >> 16;
      if (cx <= MG_COARSE_MAX && cy <= MG_COARSE_MAX) break;
      ++cl;
    }
    if (cl >= p.nlev) {
      isk_set_error("poisson: grid does not coarsen to <= %d nodes per axis", MG_COARSE_MAX);
      return ISKRA_E_UNSUPPORTED;
    }
    p.coarse_lev = cl;
    for (int k = 0; k < cl; ++k)
      if (isk_alloc((void **)&p.mo[k], (size_t)(p.ln[k] & 0xFFFF) * (p.ln[k] >> 16) * 4))
        return ISKRA_E_HIP;
  }
  return ISKRA_OK;
}

static PcgArgs make_pcg(iskra_ctx *c, int mgpre) {
  IskPoisson &p = c->ps;
  PcgArgs a;
  a.s = make_sten(c);
  a.rho = c->rho;
  a.x = p.x;
  a.r = p.r;
  a.Ap = p.Ap;
  a.z = p.z;
  a.p0 = p.p[0];
  a.p1 = p.p[1];
  a.cgp = p.cgp;
  a.nblk = (isk_nodes(c) + RED_BLOCK - 1) / RED_BLOCK;
  a.f0 = p.nlev ? p.mf[0] : nullptr;
  a.e0 = p.nlev ? p.me[0] : nullptr;
  a.mz = !p.nlev ? nullptr : p.coarse_lev > 0 ? p.mo[0] : p.me[0];
  a.scal = p.scal;
  a.partials = p.partials;
  a.iflag = p.iflag;
  a.scale = (c->g.dx * c->g.dx) / p.eps0;
  a.warm = 0;
  a.phi_in = c->phi;
  a.phi_out = c->phi;
  a.mgpre = mgpre;
  a.max_iter = p.max_iter;
  return a;
}

/* one V-cycle; mode_in0 = 1 makes the finest down-kernel compute the FP64
 * residual of x (defect correction, first = 1 on the solve's first cycle);
 * mode_out0 = 1 adds the correction to x.  part: the whole cycle, only its kernels
 * up to the one that takes the verdict on x, or only those after it. */
enum { MG_WHOLE, MG_HEAD, MG_TAIL };
static int mg_vcycle(iskra_ctx *c, int mode_in0, int mode_out0, int first, int part = MG_WHOLE) {
  IskPoisson &p = c->ps;
  const int *flag = p.iflag;
  auto lev = [&](int l) {
    MgLevel L;
    L.e = p.me[l];
    L.f = p.mf[l];
    L.nx = p.ln[l] & 0xFFFF;
    L.ny = p.ln[l] >> 16;
    return L;
  };
  MgFused a;
  a.flag = flag;
  a.s = make_sten(c);
  a.x = p.x;
  a.rho = c->rho;
  a.scale = (c->g.dx * c->g.dx) / p.eps0;
  a.scal = p.scal;
  a.partials = p.partials;
  a.iflag = p.iflag;
  a.max_iter = p.max_iter;
  const int nn0 = (p.ln[0] & 0xFFFF) * (p.ln[0] >> 16);
  const int nblk0 = (nn0 + RED_BLOCK - 1) / RED_BLOCK;
  PcgArgs pa = make_pcg(c, 0);
  /* with mode_in0 = 1 the finest residual kernel writes per-work-group
   * partials and the kernel after it takes the convergence verdict: the
   * second down kernel, or the single-work-group kernel */
  int nparts = 0;
  a.decide = 0;
  a.nparts = 0;
  a.dfirst = first;
  if (p.coarse_lev == 0 && mode_in0 == 1) {
    /* the whole grid is solved by the single work-group kernel: FP64 residual here */
    if (part != MG_TAIL)
      hipLaunchKernelGGL(k_mg_resid0, dim3(nblk0), dim3(RED_BLOCK), 0, c->stream, pa, p.me[0],
                         first);
    nparts = nblk0;
  }
  for (int l = 0; l < p.coarse_lev; ++l) {
    a.F = lev(l);
    a.C = lev(l + 1);
    a.mode_in = l == 0 ? mode_in0 : 0;
    a.first = l == 0 ? first : 0;
    a.decide = (l == 1 && nparts > 0) ? 1 : 0;
    a.nparts = nparts;
    dim3 g((a.C.nx + MGT_CT - 1) / MGT_CT, (a.C.ny + MGT_CT - 1) / MGT_CT);
    if (a.mode_in == 1 && (int)(g.x * g.y) > p.partials_blocks) {
      isk_set_error("poisson: reduction scratch holds %d blocks, kernel needs %d",
                    p.partials_blocks, (int)(g.x * g.y));
      return ISKRA_E_STATE;
    }
    if (l < 2 ? part != MG_TAIL : part != MG_HEAD)
      hipLaunchKernelGGL(k_mgf_down, g, dim3(MGT_NT), 0, c->stream, a);
    if (a.mode_in == 1) nparts = (int)(g.x * g.y);
  }
  if (p.coarse_lev < 2 ? part != MG_TAIL : part != MG_HEAD) {
    MgCoarseArgs ca;
    int tot = 0;
    ca.nlev_c = p.nlev - p.coarse_lev;
    for (int k = 0; k < ca.nlev_c; ++k) {
      int l = p.coarse_lev + k;
      ca.nx[k] = p.ln[l] & 0xFFFF;
      ca.ny[k] = p.ln[l] >> 16;
      ca.off[k] = tot;
      tot += ca.nx[k] * ca.ny[k];
    }
    ca.total = tot;
    ca.e_out = p.me[p.coarse_lev];
    ca.f_in = p.mf[p.coarse_lev];
    ca.flag = flag;
    /* the verdict here when no second down kernel took it */
    ca.decide = (nparts > 0 && p.coarse_lev <= 1) ? 1 : 0;
    ca.nparts = nparts;
    ca.dfirst = first;
    ca.max_iter = p.max_iter;
    ca.partials = p.partials;
    ca.scal = p.scal;
    ca.iflag = p.iflag;
    hipLaunchKernelGGL(k_mg_coarse, dim3(1), dim3(1024), (size_t)tot * 2 * 4, c->stream, ca);
  }
  for (int l = part == MG_HEAD ? -1 : p.coarse_lev - 1; l >= 0; --l) {
    a.F = lev(l);
    a.C = lev(l + 1);
    if (l + 1 < p.coarse_lev) a.C.e = p.mo[l + 1];
    a.out = p.mo[l];
    a.mode_out = l == 0 ? mode_out0 : 0;
    dim3 g((a.C.nx + MGT_CT - 1) / MGT_CT, (a.C.ny + MGT_CT - 1) / MGT_CT);
    hipLaunchKernelGGL(k_mgf_up, g, dim3(MGT_NT), 0, c->stream, a);
  }
  if (p.coarse_lev == 0 && mode_out0 == 1 && part != MG_HEAD)
    hipLaunchKernelGGL(k_mg_update0, dim3(nblk0), dim3(RED_BLOCK), 0, c->stream, pa, p.me[0]);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

void isk_tri_prepare(iskra_ctx *c, TriArgs *pt) {
  IskPoisson &p = c->ps;
  TriArgs &t = *pt;
  t.rho = c->rho;
  t.tags = p.d_tags;
  t.tagval = p.d_tag_val;
  t.a = p.d_tri_a;
  t.cp = p.d_tri_cp;
  t.inv = p.d_tri_inv;
  t.ma = p.d_tri_ma;
  t.ncp = p.d_tri_ncp;
  t.y = p.d_work;
  t.phi = c->phi;
  t.n = c->g.nx;
  t.scale = (c->g.dx * c->g.dx) / p.eps0;
  t.singular = p.singular;
}

int isk_poisson_solve(iskra_ctx *c, int warm, int *iters, double *relres) {
  return isk_poisson_solve_ex(c, warm, iters, relres, 0, nullptr, 0);
}

/* the spectral right-hand side packing, for the deposit kernel of the time
 * loop; returns 0 (and F = null) for the other solvers */
int isk_poisson_pack_desc(iskra_ctx *c, IskSpPack *pk) {
  IskPoisson &p = c->ps;
  pk->F = nullptr;
  if (p.kind != ISKRA_POISSON_SPECTRAL || !p.sp_F) return 0;
  pk->F = p.sp_F;
  pk->s = make_sten(c);
  pk->scale = (c->g.dx * c->g.dx) / p.eps0;
  return 1;
}

/* the device's verdict on a PCG or MG solve, for the host to look at */
__global__ void k_solve_mail(const double *scal, const int *iflag, double *mail) {
  mail[MAIL_ITERS] = (double)iflag[1];
  mail[MAIL_RELRES] = scal[S_RELRES];
  mail[MAIL_DONE] = (double)iflag[0];
}
static int solve_look(iskra_ctx *c) {
  hipLaunchKernelGGL(k_solve_mail, dim3(1), dim3(1), 0, c->stream, c->ps.scal, c->ps.iflag,
                     c->mail);
  ISK_CHECK_LAUNCH();
  ISK_HIP(hipStreamSynchronize(c->stream));
  return ISKRA_OK;
}

/* bookkeeping of a PCG or MG solve that ended after `it` iterations */
static int pcg_finish(iskra_ctx *c, int it, double rel, int *iters, double *relres) {
  IskPoisson &p = c->ps;
  p.last_iters = it;
  p.last_relres = rel;
  if (iters) *iters = it;
  if (relres) *relres = rel;
  c->stats.poisson_solves++;
  c->stats.poisson_iters += it;
  c->stats.last_iters = it;
  c->stats.last_relres = rel;
  if (!(rel <= p.rtol)) {
    isk_set_error("poisson: relative residual %.3e after %d iterations (rtol %.1e)", rel, it,
                  p.rtol);
    return ISKRA_E_CONVERGE;
  }
  return ISKRA_OK;
}

/* with_E != 0: a solver that can form E in the same pass does so and sets
 * *E_done (the spectral solve and the one-work-group solves); otherwise *E_done stays 0 */
int isk_poisson_solve_ex(iskra_ctx *c, int warm, int *iters, double *relres, int with_E,
                         int *E_done, int packed) {
  IskPoisson &p = c->ps;
  if (E_done) *E_done = 0;
  const int nn = isk_nodes(c);
  if (p.kind == ISKRA_POISSON_DIRECT) {
    TriArgs t;
    isk_tri_prepare(c, &t);
    hipLaunchKernelGGL(k_tri_solve, dim3(1), dim3(TRI_BLOCK), 0, c->stream, t);
    ISK_CHECK_LAUNCH();
    p.last_iters = 1;
    p.last_relres = 0.0;
    if (iters) *iters = 1;
    if (relres) *relres = 0.0;
    c->stats.poisson_solves++;
    c->stats.poisson_iters += 1;
    c->stats.last_iters = 1;
    c->stats.last_relres = 0.0;
    return ISKRA_OK;
  }
  const int nblk = (nn + RED_BLOCK - 1) / RED_BLOCK;
  if (p.kind == ISKRA_POISSON_SPECTRAL) {
    /* transform pass (F packed by the deposit kernel in the time loop, else
     * here; 4 GEMM launches, the last also sets the boundary ring of x),
     * FP64 residual (also phi, and E when asked), then
     * the correction kernel, which does nothing when the pass met rtol.
     * Without iters/relres (the time loop) one correction is enqueued and
     * a miss after it is reported by iskra_sync; with them the residual is
     * read back after each pass and up to 3 corrections are made. */
    PcgArgs a = make_pcg(c, 0);
    float *E = with_E ? c->E : nullptr;
    if (!packed) {
      IskSpPack pk;
      isk_poisson_pack_desc(c, &pk);
      const int m2 = p.sp_nx * p.sp_ny;
      hipLaunchKernelGGL(k_sp_pack, dim3((m2 + 255) / 256), dim3(256), 0, c->stream, pk, c->rho);
      ISK_CHECK_LAUNCH();
    }
    int nparts = nblk;
    if (sp_paired(p.sp_nx, p.sp_ny)) {
      SpPair sp;
      sp.Sy = p.sp_Sy;
      sp.B = p.sp_F;
      sp.Sx = p.sp_Sx;
      sp.Li = p.sp_Li;
      sp.T2 = p.sp_T2;
      sp.mx = p.sp_nx;
      sp.my = p.sp_ny;
      sp.a = a;
      sp.dx = c->g.dx;
      sp.dy = c->g.dy;
      sp.E = E;
      hipLaunchKernelGGL(k_sp_pair<0>, dim3((sp.my + 15) / 16), dim3(SPC_THREADS), 0,
                         c->stream, sp);
      ISK_CHECK_LAUNCH();
      sp.B = p.sp_T2;
      nparts = (sp.my + SPP_ROWS - 1) / SPP_ROWS;
      hipLaunchKernelGGL(k_sp_pair<1>, dim3(nparts), dim3(SPC_THREADS), 0, c->stream, sp);
      ISK_CHECK_LAUNCH();
    } else {
      SpGemm g[4];
      sp_pass_desc(c, a, 0, g);
      for (int k = 0; k < 4; ++k) {
        hipLaunchKernelGGL(k_sp_gemm, dim3((g[k].N + 15) / 16, (g[k].M + 15) / 16), dim3(256), 0,
                           c->stream, g[k]);
        ISK_CHECK_LAUNCH();
      }
      hipLaunchKernelGGL(k_sp_resid, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, E, c->g.dx,
                         c->g.dy);
      ISK_CHECK_LAUNCH();
    }
    SpCorrect sc;
    sp_pass_desc(c, a, 1, sc.g);
    sc.a = a;
    sc.rtol = p.rtol;
    sc.dx = c->g.dx;
    sc.dy = c->g.dy;
    sc.E = E;
    sc.nparts = nparts; /* the first call sums the residual of the first pass */
    sc.second = (!iters && !relres) ? 1 : 0;
    hipLaunchKernelGGL(k_sp_correct, dim3(1), dim3(SPC_THREADS), 0, c->stream, sc);
    ISK_CHECK_LAUNCH();
    int rounds = 1;
    double rel = 0.0;
    if (iters || relres) {
      sc.nparts = 0;
      while (true) {
        double scal[S_WORDS];
        int fl[8];
        ISK_HIP(hipMemcpyAsync(scal, p.scal, sizeof(scal), hipMemcpyDeviceToHost, c->stream));
        ISK_HIP(hipMemcpyAsync(fl, p.iflag, sizeof(fl), hipMemcpyDeviceToHost, c->stream));
        ISK_HIP(hipStreamSynchronize(c->stream));
        rel = scal[S_RELRES];
        rounds = fl[IF_SP_PASSES];
        if (fl[IF_SP_DONE]) break;
        if (rounds >= 4) {
          isk_set_error("poisson: spectral solve reached relative residual %.3g > %.3g", rel,
                        p.rtol);
          return ISKRA_E_CONVERGE;
        }
        hipLaunchKernelGGL(k_sp_correct, dim3(1), dim3(SPC_THREADS), 0, c->stream, sc);
        ISK_CHECK_LAUNCH();
      }
    }
    if (E_done) *E_done = with_E;
    p.last_iters = rounds;
    p.last_relres = rel;
    if (iters) *iters = rounds;
    if (relres) *relres = rel;
    c->stats.poisson_solves++;
    c->stats.poisson_iters += rounds;
    c->stats.last_iters = rounds;
    c->stats.last_relres = rel;
    return ISKRA_OK;
  }
  if (!p.h_sd.empty()) {
    int rc = isk_electrodes_after_push(c, 0.0); /* fold in charge collected since */
    if (rc) return rc;
    return isk_bicgstab_solve(c, warm, iters, relres, with_E ? c->E : nullptr, E_done);
  }
  const int mgpre = p.kind == ISKRA_POISSON_MGPCG;
  PcgArgs a = make_pcg(c, mgpre);
  a.warm = warm;
  size_t shm = 0;
  const int npt = p.kind != ISKRA_POISSON_PCG ? 0 : one_npt(c, one_cg_shapes, sizeof(float), 0, &shm);
  if (npt) {
    CgOne o;
    o.a = a;
    o.E = with_E ? c->E : nullptr;
    o.dx = c->g.dx;
    o.dy = c->g.dy;
    o.rtol = p.rtol;
    o.mail = c->mail;
#define CG_ONE(A)                                                                     \
  (npt == 2 ? k_cg_one<2, 1024, A> : npt == 4 ? k_cg_one<4, 1024, A>                  \
   : npt == 8 ? k_cg_one<8, 1024, A> : npt == 19 ? k_cg_one<19, 512, A>               \
   : k_cg_one<26, 512, A>)
    auto k = c->g.axial ? CG_ONE(true) : CG_ONE(false);
#undef CG_ONE
    hipLaunchKernelGGL(k, dim3(1), dim3(npt <= 8 ? 1024 : 512), shm, c->stream, o);
    ISK_CHECK_LAUNCH();
    if (with_E) *E_done = 1;
    int it = 0, broke = 0;
    double rel = 0.0;
    int rc = one_result(c, &it, &rel, &broke);
    if (rc) return rc;
    return pcg_finish(c, it, rel, iters, relres);
  }
  hipLaunchKernelGGL(k_pcg_setx, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a);
  hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(64), 0, c->stream, p.scal, p.iflag,
                     p.rtol * p.rtol, p.singular ? 1 : 0);
  ISK_CHECK_LAUNCH();
  if (p.singular) {
    hipLaunchKernelGGL(k_pcg_mean, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a);
    ISK_CHECK_LAUNCH();
  }
  if (p.kind == ISKRA_POISSON_MG) {
    /* as many cycles as the last solve needed, the head of one more, which takes
     * the verdict on them, and a look at it; then two cycles a look.  A whole
     * cycle more and another for the verdict, empty as they mostly are, and two
     * copies back took 60 us of 1640 of a solve on 513 x 513 nodes. */
    int batch = p.last_iters > 0 ? p.last_iters : MG_BATCH;
    int first = 1;
    int launched = batch;
    while (true) {
      for (int b = 0; b < batch; ++b) {
        int rc = mg_vcycle(c, 1, 1, first);
        if (rc) return rc;
        first = 0;
      }
      int rc = mg_vcycle(c, 1, 1, 0, MG_HEAD);
      if (rc) return rc;
      if ((rc = solve_look(c))) return rc;
      if (c->mail[MAIL_DONE] != 0.0) break;
      if ((rc = mg_vcycle(c, 1, 1, 0, MG_TAIL))) return rc;
      batch = 1;
      launched += 2;
      if (launched > p.max_iter + 4) {
        isk_set_error("poisson: multigrid stopped after %d host cycles without a device verdict", launched);
        return ISKRA_E_CONVERGE;
      }
    }
  } else {
    hipLaunchKernelGGL(k_pcg_resid, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a);
    ISK_CHECK_LAUNCH();
    if (mgpre) {
      int rc = mg_vcycle(c, 0, 0, 0);
      if (rc) return rc;
      hipLaunchKernelGGL(k_cg_toz, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, 0);
    }
    /* every batch ends with an A kernel, which decides convergence */
    hipLaunchKernelGGL(k_cg_a, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, 0);
    ISK_CHECK_LAUNCH();
    int it = 0;
    while (true) {
      for (int b = 0; b < (mgpre ? MG_BATCH : PCG_BATCH); ++b, ++it) {
        hipLaunchKernelGGL(k_cg_b, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it);
        if (mgpre) {
          int rc = mg_vcycle(c, 0, 0, 0);
          if (rc) return rc;
          hipLaunchKernelGGL(k_cg_toz, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a,
                             (it + 1) & 1);
        }
        hipLaunchKernelGGL(k_cg_a, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, it + 1);
        ISK_CHECK_LAUNCH();
      }
      int rc = solve_look(c);
      if (rc) return rc;
      if (c->mail[MAIL_DONE] != 0.0) break;
      if (it > p.max_iter + 2 * PCG_BATCH) {
        isk_set_error("poisson: CG stopped after %d host iterations without a device verdict", it);
        return ISKRA_E_CONVERGE;
      }
    }
  }
  double mean_sub = 0.0;
  if (p.singular) {
    std::vector<double> hx(nn);
    ISK_HIP(hipMemcpy(hx.data(), p.x, nn * 8, hipMemcpyDeviceToHost));
    double s = 0.0;
    for (int k = 0; k < nn; ++k) s += hx[k];
    mean_sub = s / nn;
  }
  hipLaunchKernelGGL(k_pcg_out, dim3(nblk), dim3(RED_BLOCK), 0, c->stream, a, c->phi, mean_sub);
  ISK_CHECK_LAUNCH();
  return pcg_finish(c, (int)c->mail[MAIL_ITERS], c->mail[MAIL_RELRES], iters, relres);
}

/* where an in-loop spectral solve records a miss and its residual (else null) */
void isk_poisson_status(const iskra_ctx *c, const int **fail, const double **relres) {
  const IskPoisson &p = c->ps;
  const bool sp = p.kind == ISKRA_POISSON_SPECTRAL && p.iflag;
  *fail = sp ? p.iflag + IF_SP_FAIL : nullptr;
  *relres = sp ? p.scal + S_RELRES : nullptr;
}

/* an in-loop spectral solve missed rtol since the last check: clears that and
 * reports it */
int isk_poisson_check(iskra_ctx *c) {
  int zero = 0;
  ISK_HIP(hipMemcpy(c->ps.iflag + IF_SP_FAIL, &zero, 4, hipMemcpyHostToDevice));
  isk_set_error("poisson: a spectral solve in the time loop missed rtol %.3g after "
                "correction (relative residual %.3g)", c->ps.rtol, c->ps.last_relres);
  return ISKRA_E_CONVERGE;
}
