/*
 * particles.hip -- particle kernels of the electrostatic PIC step on gfx950.
 *
 *  k_push<DIM>      fused gather + push + boundary + CIC deposit, one
 *                   work-group per chunk of a tile; E window and deposit
 *                   window in LDS; deposit accumulated as 64-bit fixed point
 *                   (integer adds are associative, so the result does not
 *                   depend on particle order or scheduling).
 *  k_merge<DIM>     per node, sums the chunk windows that cover it in a fixed
 *                   order plus the global fallback accumulator.
 *  k_sort_*         stable counting sort by tile (or by cell in tile):
 *                   strip histograms -> column scans -> stable scatter, a strip
 *                   being the work of one wave.
 *  k_field1         1-D grids: counts, rho, the direct solve, E and the electrode
 *                   waveforms in one launch.
 *  k_rho            rho = sum_s q_s n_s + background,  n_s = deposit / volume.
 *
 * Reference semantics followed (paths relative to the reference tree):
 *  particle_cell            ParticleInCell/src/ParticleInCell.jl:28-35
 *  grid_to_particle (CIC)   ParticleInCell/src/pic/cloud_in_cell.jl:20-36
 *  push_in_cartesian! (B=0) ParticleInCell/src/pic/pushers.jl:37-50
 *  wrap! / discard!         ParticleInCell/src/pic/surfaces/wrap.jl:1-33
 *  particle_to_grid (CIC)   ParticleInCell/src/pic/cloud_in_cell.jl:1-18
 *  density, cell_volume     pic/kinetic.jl:53, RegularGrids/src/RegularGrids.jl:26-38
 *  rho accumulation         ParticleInCell/src/ParticleInCell.jl:118-124
 */
#include <math.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "isk_fp64math.h"
#include "isk_internal.h"
#include "isk_tri.h"

/* push work-group shape: threads, and particles per thread per batch (one
 * batch covers a 2048-particle chunk). 2-D: 512 x 4 keeps the kernel at 59
 * VGPRs (8 waves per SIMD), 2 % faster than 256 x 8 at 96 VGPRs on the
 * 256^2-cell slab; 1-D keeps 256 x 8 */
template <int DIM>
struct PushShape {
  static constexpr int block = DIM == 2 ? 512 : 256;
  static constexpr int unroll = DIM == 2 ? 4 : 8;
};
/* the largest float below 1 (1 - 2^-24): an offset on the upper edge of its cell */
#define ISK_BELOW_ONE 0x1.fffffep-1f
/* counting sort: one wave per strip of particles; rounds of 64 particles,
 * SORT_DEPTH rounds of loads in flight; strips are multiples of SORT_STRIP_MIN */
#define SORT_WAVE 64
#define SORT_DEPTH 4
#define SORT_STRIP_MIN (SORT_WAVE * SORT_DEPTH)
/* rounds of keys the histogram has in flight, and its threads on a long strip */
#define SORT_KEYS 16
#define SORT_HIST 256
#define SORT_STRIP_MAX 8192
/* strips aimed at per sort: 4 waves a CU.  With 4096 a sort of 4 M particles in 1024
 * tiles takes 107 us, of 1 M 54; with 1024 72 and 45, with 512 72 and 43 (and 6 % more
 * than with 1024 for 4 M in 7744 tiles) */
#define SORT_STRIPS 1024
/* entries of the strip x bin table above which strips get longer instead */
#define SORT_TABLE_MAX (8 << 20)
/* column scans: bins and row segments of a work-group (SORT_CB x SORT_CS threads) */
#define SORT_CB 32
#define SORT_CS (1024 / SORT_CB)
/* strips up to which one work-group scans a table of one bin group: 6 us for
 * 80 strips against 4.4 + 4.8 us for the two launches; with three groups of
 * 256 strips it takes 12.4 */
#define SORT_ONE_MAX 512
/* eights of rows a segment may have to be read once: in the column scans' own launch,
 * and in the one work-group's (all its rows) */
#define SORT_CR 8
#define SORT_CR_ONE (SORT_ONE_MAX / SORT_CS / 8)

/* ------------------------------------------------------------------------ */
/* small utility kernels                                                     */
/* ------------------------------------------------------------------------ */
__global__ void k_fill_i64(long long *p, long long n, long long v) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long stride = (long long)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

int isk_fill_i64(iskra_ctx *c, void *p, int64_t n, long long v) {
  if (n <= 0) return ISKRA_OK;
  int blocks = (int)std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_i64, dim3(blocks), dim3(256), 0, c->stream,
                     (long long *)p, (long long)n, v);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* ------------------------------------------------------------------------ */
/* upload (host conversion) and Maxwellian loader                           */
/* ------------------------------------------------------------------------ */
/* particle_cell with the grid origin removed: s = (x - x0)/dh, i = floor(s),
 * offset = s - i rounded to FP32 (an offset that rounds up to 1 moves to the
 * next cell with offset 0). */
static int cell_of(double x, double x0, double dh, int nc, int *i, float *o) {
  double s = (x - x0) / dh;
  double fl = floor(s);
  if (!(fl >= 0.0) || fl >= (double)nc) return -1;
  int ii = (int)fl;
  float of = (float)(s - fl);
  if (of >= 1.0f) {
    of = 0.0f;
    ii += 1;
    if (ii >= nc) return -1;
  }
  *i = ii;
  *o = of;
  return 0;
}

int isk_convert_upload(iskra_ctx *c, int sid, int64_t np, const double *x,
                       const double *v, const uint32_t *id) {
  IskSpecies *s = &c->sp[sid];
  const IskGrid &g = c->g;
  if (np < 0 || np > s->cap) {
    isk_set_error("upload: np=%lld outside [0, capacity=%lld]", (long long)np,
                  (long long)s->cap);
    return ISKRA_E_CAPACITY;
  }
  std::vector<int32_t> cell(np);
  std::vector<float> ox(np), oy(g.dim == 2 ? np : 0), vx(np), vy(np), vz(np);
  std::vector<uint32_t> ids(s->track_ids ? np : 0);
  uint32_t maxid = 0;
  for (int64_t p = 0; p < np; ++p) {
    int i = 0, j = 0;
    float fx = 0.f, fy = 0.f;
    if (cell_of(x[p], g.x0, g.dx, g.ncx, &i, &fx) != 0) {
      isk_set_error("upload: particle %lld has x=%g outside the grid",
                    (long long)p, x[p]);
      return ISKRA_E_ARG;
    }
    if (g.dim == 2) {
      if (cell_of(x[np + p], g.y0, g.dy, g.ncy, &j, &fy) != 0) {
        isk_set_error("upload: particle %lld has y=%g outside the grid",
                      (long long)p, x[np + p]);
        return ISKRA_E_ARG;
      }
      oy[p] = fy;
    }
    cell[p] = i | (j << 16);
    ox[p] = fx;
    vx[p] = (float)v[p];
    vy[p] = (float)v[np + p];
    vz[p] = (float)v[2 * np + p];
    if (s->track_ids) {
      ids[p] = id ? id[p] : (uint32_t)p;
      if (ids[p] > maxid) maxid = ids[p];
    }
  }
  int b = s->cur;
  if (np > 0) {
    ISK_HIP(hipMemcpyAsync(s->cell[b], cell.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    ISK_HIP(hipMemcpyAsync(s->ox[b], ox.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    if (g.dim == 2)
      ISK_HIP(hipMemcpyAsync(s->oy[b], oy.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    ISK_HIP(hipMemcpyAsync(s->vx[b], vx.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    ISK_HIP(hipMemcpyAsync(s->vy[b], vy.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    ISK_HIP(hipMemcpyAsync(s->vz[b], vz.data(), np * 4, hipMemcpyHostToDevice, c->stream));
    if (s->track_ids)
      ISK_HIP(hipMemcpyAsync(s->id[b], ids.data(), np * 4, hipMemcpyHostToDevice, c->stream));
  }
  long long hdr[HDR_WORDS];
  ISK_HIP(hipMemcpyAsync(hdr, s->hdr, sizeof(hdr), hipMemcpyDeviceToHost, c->stream));
  ISK_HIP(hipStreamSynchronize(c->stream));
  hdr[HDR_NP] = np;
  hdr[HDR_NP_SORTED] = 0;
  hdr[HDR_NCHUNKS] = 0;
  hdr[HDR_NEXT_ID] = s->track_ids ? (long long)maxid + 1 : np;
  hdr[HDR_OVERFLOW] = 0;
  ISK_HIP(hipMemcpyAsync(s->hdr, hdr, sizeof(hdr), hipMemcpyHostToDevice, c->stream));
  ISK_HIP(hipStreamSynchronize(c->stream));
  return isk_sort_species(c, sid, 0);
}

/* sample!(::MaxwellianSource): x = U*wx + dx, v = N(0,1)*wv + dv.
 * Draws: Philox4x32-10, key = seed, counter = (k_lo, k_hi, stream, block). */
struct SampleArgs {
  int32_t *cell;
  float *ox, *oy, *vx, *vy, *vz;
  uint32_t *id;
  long long *hdr;
  long long n;
  double wx[2], dxo[2], wv[3], dv[3];
  double x0, y0, dx, dy;
  int ncx, ncy, dim;
  uint32_t k0, k1, stream;
};

__global__ __launch_bounds__(256) void k_sample(SampleArgs a) {
  long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.n) return;
  long long np0 = a.hdr[HDR_NP];
  long long p = np0 + k;
  IskU4 c0 = {(uint32_t)k, (uint32_t)(k >> 32), a.stream, 0u};
  IskU4 r0 = isk_philox(c0, a.k0, a.k1);
  c0.w = 1u;
  IskU4 r1 = isk_philox(c0, a.k0, a.k1);
  c0.w = 2u;
  IskU4 r2 = isk_philox(c0, a.k0, a.k1);
  /* positions */
  double ux = isk_u01(r0.x, r0.y);
  double px = ux * a.wx[0] + a.dxo[0];
  double s = (px - a.x0) / a.dx;
  double fl = floor(s);
  int i = (int)fl;
  float of = (float)(s - fl);
  if (of >= 1.0f) { of = 0.0f; i += 1; }
  /* the host keeps the box inside the grid; these only catch a position
   * that rounding put just past an edge of it */
  if (i < 0) { i = 0; of = 0.0f; }
  if (i > a.ncx - 1) { i = a.ncx - 1; of = ISK_BELOW_ONE; }
  int j = 0;
  if (a.dim == 2) {
    double uy = isk_u01(r0.z, r0.w);
    double py = uy * a.wx[1] + a.dxo[1];
    double sy = (py - a.y0) / a.dy;
    double fly = floor(sy);
    j = (int)fly;
    float ofy = (float)(sy - fly);
    if (ofy >= 1.0f) { ofy = 0.0f; j += 1; }
    if (j < 0) { j = 0; ofy = 0.0f; }
    if (j > a.ncy - 1) { j = a.ncy - 1; ofy = ISK_BELOW_ONE; }
    a.oy[p] = ofy;
  }
  /* velocities: Box-Muller on (r1.xy, r1.zw) and (r2.xy, r2.zw) */
  double u1 = isk_u01(r1.x, r1.y), u2 = isk_u01(r1.z, r1.w);
  double u3 = isk_u01(r2.x, r2.y), u4 = isk_u01(r2.z, r2.w);
  double rad1 = sqrt(-2.0 * isk_log(u1)), rad2 = sqrt(-2.0 * isk_log(u3));
  double s1, c1, s2, c2;
  isk_sincos2pi(u2, &s1, &c1);
  isk_sincos2pi(u4, &s2, &c2);
  a.cell[p] = i | (j << 16);
  a.ox[p] = of;
  a.vx[p] = (float)(rad1 * c1 * a.wv[0] + a.dv[0]);
  a.vy[p] = (float)(rad1 * s1 * a.wv[1] + a.dv[1]);
  a.vz[p] = (float)(rad2 * c2 * a.wv[2] + a.dv[2]);
  if (a.id) a.id[p] = (uint32_t)(a.hdr[HDR_NEXT_ID] + k);
}

__global__ void k_sample_commit(long long *hdr, long long n) {
  hdr[HDR_NP] += n;
  hdr[HDR_NEXT_ID] += n;
}

int isk_sample_maxwellian(iskra_ctx *c, int sid, int64_t n, const double *wx,
                          const double *dx, const double *wv, const double *dv,
                          uint64_t seed, uint32_t stream) {
  IskSpecies *s = &c->sp[sid];
  long long hdr[HDR_WORDS];
  ISK_HIP(hipMemcpyAsync(hdr, s->hdr, sizeof(hdr), hipMemcpyDeviceToHost, c->stream));
  ISK_HIP(hipStreamSynchronize(c->stream));
  int64_t room = s->cap - hdr[HDR_NP];
  if (n > room) n = room; /* sample! truncates to the free capacity (sources.jl:30) */
  if (n <= 0) return ISKRA_OK;
  SampleArgs a;
  int b = s->cur;
  a.cell = s->cell[b];
  a.ox = s->ox[b];
  a.oy = s->oy[b];
  a.vx = s->vx[b];
  a.vy = s->vy[b];
  a.vz = s->vz[b];
  a.id = s->track_ids ? s->id[b] : nullptr;
  a.hdr = s->hdr;
  a.n = n;
  for (int d = 0; d < 2; ++d) {
    a.wx[d] = d < c->g.dim ? wx[d] : 0.0;
    a.dxo[d] = d < c->g.dim ? (dx ? dx[d] : 0.0) : 0.0;
  }
  for (int d = 0; d < 3; ++d) {
    a.wv[d] = wv[d];
    a.dv[d] = dv ? dv[d] : 0.0;
  }
  a.x0 = c->g.x0;
  a.y0 = c->g.y0;
  a.dx = c->g.dx;
  a.dy = c->g.dy;
  a.ncx = c->g.ncx;
  a.ncy = c->g.ncy;
  a.dim = c->g.dim;
  a.k0 = (uint32_t)seed;
  a.k1 = (uint32_t)(seed >> 32);
  a.stream = stream;
  int blocks = (int)((n + 255) / 256);
  hipLaunchKernelGGL(k_sample, dim3(blocks), dim3(256), 0, c->stream, a);
  ISK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_sample_commit, dim3(1), dim3(1), 0, c->stream, s->hdr,
                     (long long)n);
  ISK_CHECK_LAUNCH();
  return isk_sort_species(c, sid, 0);
}

/* ------------------------------------------------------------------------ */
/* counting sort                                                             */
/* ------------------------------------------------------------------------ */
/* Stable counting sort of one species, in three or four launches:
 *   k_sort_hist     per strip of particles, the count of every bin -> H[strip][bin]
 *   k_sort_cols     per bin, the exclusive prefix over the strips, and the total
 *   k_sort_bins     the bins' first positions, the new counts and the chunk table
 *                   (k_sort_table: this and the column scans in one work-group)
 *   k_sort_scatter  every strip writes its particles behind the earlier ones
 * A strip belongs to one wave of its own work-group, which walks it in rounds
 * of 64: ranks come from ballots over the key's bits and the strip's next
 * positions live in LDS that only this wave touches (LDS serves one wave's
 * accesses in order), so no round waits at a barrier.  What bounds a small sort
 * is the chain of rounds of one strip (about 0.5 us each), a large one the
 * memory: the strip length follows the capacity, and short strips are only
 * worth their table rows while the table stays small against the particles.
 * Measured, one sort of an ordered species (before: strips of 8192 shared by four
 * waves that matched keys between barriers): 100,000 particles in 64 tiles 30 us (74), 1 M
 * in 1024 45 (85), 4 M 72 (92), 16 M 243 (261), 4 M in 7744 tiles 117 (130), 16 M 297
 * (326).  An XCD taking neighbouring strips puts its waves on few memory channels
 * at a time: 410 instead of 353 us for 2^24. */
struct KeyDesc {
  int mode; /* 0: tile, 1: cell inside tile, 2: tile, then cell inside it */
  int dim, T, log2T, ntx, nbins;
  int nbits; /* bits of the largest key (nbins, the discarded particles') */
};

__device__ __forceinline__ int sort_key(int c, const KeyDesc &k) {
  if (c < 0) return k.nbins; /* discarded -> last bin */
  int i = c & 0xFFFF;
  int j = c >> 16;
  const int tile = (i >> k.log2T) + k.ntx * (j >> k.log2T);
  if (k.mode == 0) return tile;
  const int in = (i & (k.T - 1)) + (k.dim == 2 ? ((j & (k.T - 1)) << k.log2T) : 0);
  if (k.mode == 1) return in;
  return (tile << (k.dim * k.log2T)) + in;
}

struct ScatterArgs {
  const int32_t *cell;
  const float *ox, *oy, *vx, *vy, *vz;
  const uint32_t *id;
  int32_t *cell_o;
  float *ox_o, *oy_o, *vx_o, *vy_o, *vz_o;
  uint32_t *id_o;
};

/* everything one sort pass of one species needs (single or batched launch) */
struct SortArgs {
  KeyDesc kd;
  ScatterArgs sc;
  long long *hdr;
  int *H, *tot, *start;
  int nb1, nrow, strip, ngrp; /* bins + 1, strips, particles a strip, groups of SORT_CB bins */
  int one;                    /* the table is scanned by one work-group */
  int span;                   /* bins a tile */
  int build, CH;
  IskChunk *chunks;
  int *tcb;
};

/* strips that hold particles */
__device__ __forceinline__ int sort_active(const SortArgs &a, long long np) {
  return min(a.nrow, (int)((np + a.strip - 1) / a.strip));
}

/* orders this wave's LDS accesses (they execute in order; the fence keeps the
 * compiler from moving them) */
__device__ __forceinline__ void sort_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
  __builtin_amdgcn_wave_barrier();
}

/* a strip's counts; its waves (one, or four on a long strip) count together */
__device__ __forceinline__ void sort_hist_body(const SortArgs &a, const int blk) {
  extern __shared__ int sh[];
  const int row = blk, nt = (int)blockDim.x;
  const long long np = a.hdr[HDR_NP];
  const long long base = (long long)row * a.strip;
  const int tid = threadIdx.x;
  if (base >= np) return;
  for (int b = tid; b < a.nb1; b += nt) sh[b] = 0;
  __syncthreads();
  const int32_t *__restrict__ cell = a.sc.cell;
  const KeyDesc kd = a.kd;
  const long long end = min(np, base + a.strip);
  /* SORT_KEYS rounds of keys in flight (index clamped to the last particle,
   * validity applied at use) */
  for (long long r = base; r < end; r += SORT_KEYS * nt) {
    int cv[SORT_KEYS];
#pragma unroll
    for (int u = 0; u < SORT_KEYS; ++u) {
      const long long p = r + u * nt + tid;
      cv[u] = cell[p < np ? p : np - 1];
    }
    /* valid lanes are a prefix of the wave, so its first lane is valid when any
     * is; that lane's key (in tile-ordered data mostly the key of the whole wave) is
     * counted with one ballot, the other lanes add 1 each */
#pragma unroll
    for (int u = 0; u < SORT_KEYS; ++u) {
      const bool valid = r + u * nt + tid < end;
      const int key = valid ? sort_key(cv[u], kd) : -1;
      if (__ballot(valid) == 0ull) break;
      const int k0 = __builtin_amdgcn_readfirstlane(key);
      const unsigned long long m0 = __ballot(key == k0);
      if ((tid & 63) == 0) atomicAdd(&sh[k0], (int)__popcll(m0));
      if (valid && key != k0) atomicAdd(&sh[key], 1);
    }
  }
  __syncthreads();
  int *__restrict__ Hb = a.H + (size_t)row * a.nb1;
#pragma unroll 8
  for (int b = tid; b < a.nb1; b += nt) Hb[b] = sh[b];
}

__global__ __launch_bounds__(SORT_HIST) void k_sort_hist(SortArgs a) {
  sort_hist_body(a, blockIdx.x);
}

/* bins [SORT_CB grp, ...): exclusive prefix of every bin over the strips in
 * place, its total into tot.  Thread (bin, segment) takes a contiguous part
 * of the strips; a row's SORT_CB entries are one 128-byte read. */
template <int CR>
__device__ __forceinline__ void sort_cols_body(const SortArgs &a, const int grp, const int nact) {
  __shared__ int part[SORT_CS][SORT_CB + 1];
  const int lb = threadIdx.x & (SORT_CB - 1), seg = threadIdx.x / SORT_CB;
  const int b = grp * SORT_CB + lb;
  const int per = (nact + SORT_CS - 1) / SORT_CS;
  const int r0 = min(seg * per, nact), r1 = min(r0 + per, nact);
  int *__restrict__ col = a.H + (b < a.nb1 ? b : 0);
  const size_t ld = a.nb1;
  const bool on = b < a.nb1, once = per <= 8 * CR; /* the part stays in registers */
  int sum = 0;
  int v[CR][8];
  if (once) {
#pragma unroll
    for (int k = 0; k < CR; ++k)
      if (8 * k < per)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = r0 + 8 * k + u;
          v[k][u] = on && r < r1 ? col[r * ld] : 0;
        }
#pragma unroll
    for (int k = 0; k < CR; ++k)
      if (8 * k < per)
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += v[k][u];
  } else if (on) {
    int r = r0;
    for (; r + 8 <= r1; r += 8) {
      int w[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) w[u] = col[(r + u) * ld];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += w[u];
    }
    for (; r < r1; ++r) sum += col[r * ld];
  }
  __syncthreads(); /* part may still be read for the previous group */
  part[seg][lb] = sum;
  __syncthreads();
  int run = 0;
  for (int s = 0; s < seg; ++s) run += part[s][lb];
  if (!on) return;
  if (seg == SORT_CS - 1) a.tot[b] = run + sum;
  if (once) {
#pragma unroll
    for (int k = 0; k < CR; ++k)
      if (8 * k < per)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = r0 + 8 * k + u;
          if (r < r1) col[r * ld] = run;
          run += v[k][u];
        }
    return;
  }
  int r = r0;
  for (; r + 8 <= r1; r += 8) {
    int w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = col[(r + u) * ld];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      col[(r + u) * ld] = run;
      run += w[u];
    }
  }
  for (; r < r1; ++r) {
    const int w = col[r * ld];
    col[r * ld] = run;
    run += w;
  }
}

__global__ __launch_bounds__(1024) void k_sort_cols(SortArgs a) {
  sort_cols_body<SORT_CR>(a, blockIdx.x, sort_active(a, a.hdr[HDR_NP]));
}

/* inclusive scan of one value a thread over 1024 threads: within each wave by
 * shuffles, then over the 16 waves' totals */
__device__ __forceinline__ int sort_scan1024(int v, int *total) {
  __shared__ int wsum[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off);
    if (lane >= off) v += u;
  }
  __syncthreads(); /* wsum may still be read by an earlier call */
  if (lane == 63) wsum[w] = v;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    if (k < w) before += wsum[k];
    all += wsum[k];
  }
  *total = all;
  return v + before;
}

/* one work-group of 1024: first position of every bin, the particle counts
 * (the scatter reads the old one from HDR_NP_OLD) and, with build, the chunk
 * table of the tiles (span bins each).  Every thread holds the old count
 * before this is called. */
template <int PB, int PT> /* bins and tiles a thread, at most */
__device__ __forceinline__ void sort_bins_some(const SortArgs &a, const long long np_old) {
  const int nbins = a.nb1 - 1;
  int *__restrict__ start = a.start;
  const int per = (a.nb1 + 1023) / 1024;
  const int lo = min((int)threadIdx.x * per, a.nb1), hi = min(lo + per, a.nb1);
  int sum = 0, all;
  int tot[PB]; /* loaded together (one by one they are a chain of waits) */
#pragma unroll
  for (int k = 0; k < PB; ++k) {
    if (k >= per) break;
    tot[k] = lo + k < hi ? a.tot[lo + k] : 0;
  }
#pragma unroll
  for (int k = 0; k < PB; ++k) {
    if (k >= per) break;
    sum += tot[k];
  }
  int run = sort_scan1024(sum, &all) - sum;
#pragma unroll
  for (int k = 0; k < PB; ++k) {
    if (k >= per) break;
    if (lo + k < hi) start[lo + k] = run;
    run += tot[k];
  }
  if (threadIdx.x == 0) start[a.nb1] = all;
  __syncthreads(); /* start is read across threads below */
  const long long live = start[nbins];
  int nch = 0;
  if (a.build) {
    const int ntile = nbins / a.span, pt = (ntile + 1023) / 1024;
    const int t0 = min((int)threadIdx.x * pt, ntile), t1 = min(t0 + pt, ntile);
    int cs = 0, at[PT + 1];
#pragma unroll
    for (int k = 0; k <= PT; ++k) {
      if (k > pt) break;
      at[k] = t0 + k <= t1 ? start[(t0 + k) * a.span] : 0;
    }
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      if (k >= pt) break;
      if (t0 + k < t1) cs += (at[k + 1] - at[k] + a.CH - 1) / a.CH;
    }
    int c = sort_scan1024(cs, &nch) - cs;
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      if (k >= pt || t0 + k >= t1) break;
      const int n = at[k + 1] - at[k];
      a.tcb[t0 + k] = c;
      for (int q = 0; q * a.CH < n; ++q) {
        IskChunk ch;
        ch.tile = t0 + k;
        ch.start = at[k] + q * a.CH;
        ch.count = min(a.CH, n - q * a.CH);
        ch.pad = 0;
        a.chunks[c++] = ch;
      }
    }
    if (threadIdx.x == 0) a.tcb[ntile] = nch;
  }
  if (threadIdx.x == 0) {
    a.hdr[HDR_NP_OLD] = np_old;
    a.hdr[HDR_NP] = live;
    a.hdr[HDR_NP_SORTED] = a.build ? live : 0;
    a.hdr[HDR_NCHUNKS] = nch;
  }
}

__device__ __forceinline__ void sort_bins_body(const SortArgs &a, const long long np_old) {
  if (a.nb1 <= 1024) sort_bins_some<1, 1>(a, np_old);
  else sort_bins_some<ISK_SORT_BINS / 1024, ISK_MAX_BINS / 1024>(a, np_old);
}

__global__ __launch_bounds__(1024) void k_sort_bins(SortArgs a) {
  const long long np = a.hdr[HDR_NP];
  sort_bins_body(a, np);
}

/* the column scans and the bins in one work-group: one launch instead of two
 * dependent ones while the strips x bin groups are few (SORT_ONE_MAX) */
__device__ __forceinline__ void sort_table_body(const SortArgs &a) {
  const long long np = a.hdr[HDR_NP];
  const int nact = sort_active(a, np);
  for (int g = 0; g < a.ngrp; ++g) sort_cols_body<SORT_CR_ONE>(a, g, nact);
  __syncthreads(); /* tot is read across threads */
  sort_bins_some<1, 1>(a, np); /* one group: SORT_CB bins */
}

__global__ __launch_bounds__(1024) void k_sort_table(SortArgs a) { sort_table_body(a); }

template <int DIM, bool ID>
struct SortPay {
  int c[SORT_DEPTH];
  float ox[SORT_DEPTH], oy[SORT_DEPTH], vx[SORT_DEPTH], vy[SORT_DEPTH], vz[SORT_DEPTH];
  uint32_t id[SORT_DEPTH];
};

/* SORT_DEPTH rounds of records; indices are clamped to the last particle, so
 * the loads carry no condition and stay in flight */
template <int DIM, bool ID>
__device__ __forceinline__ void scatter_load(const ScatterArgs &a, long long p0, long long np,
                                             SortPay<DIM, ID> &q) {
#pragma unroll
  for (int u = 0; u < SORT_DEPTH; ++u) {
    const long long p = p0 + u * SORT_WAVE, pc = p < np ? p : np - 1;
    q.c[u] = a.cell[pc];
    q.ox[u] = a.ox[pc];
    if (DIM == 2) q.oy[u] = a.oy[pc];
    q.vx[u] = a.vx[pc];
    q.vy[u] = a.vy[pc];
    q.vz[u] = a.vz[pc];
    if (ID) q.id[u] = a.id[pc];
  }
}

/* destination of one round's particles: lanes of equal key are found by
 * ballots over the key's bits (one ballot when the whole wave has lane 0's
 * key), ranked in lane order, and the first of them moves the bin's next
 * position on.  Lanes past the end hold key -1 and get no position. */
__device__ __forceinline__ int scatter_rank(const KeyDesc &kd, int key, unsigned long long all,
                                            int *base) {
  const int k0 = __builtin_amdgcn_readfirstlane(key);
  unsigned long long m = __ballot(key == k0);
  if (m != all) {
    m = all;
    for (int bit = 0; bit < kd.nbits; ++bit) {
      const bool one = (key >> bit) & 1;
      const unsigned long long bl = __ballot(one);
      m &= one ? bl : ~bl;
    }
  }
  const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                             __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
  int d0 = 0;
  if (key >= 0) d0 = base[key];
  sort_wave_fence();
  if (key >= 0 && rank == 0) base[key] = d0 + (int)__popcll(m);
  sort_wave_fence();
  return d0 + rank;
}

template <int DIM, bool ID>
__device__ __forceinline__ void scatter_store(const ScatterArgs &a, const SortPay<DIM, ID> &q,
                                              int u, int d) {
  a.cell_o[d] = q.c[u];
  a.ox_o[d] = q.ox[u];
  if (DIM == 2) a.oy_o[d] = q.oy[u];
  a.vx_o[d] = q.vx[u];
  a.vy_o[d] = q.vy[u];
  a.vz_o[d] = q.vz[u];
  if (ID) a.id_o[d] = q.id[u];
}

/* SORT_DEPTH whole rounds.  Nothing here is conditional on a lane, discarded
 * particles are written behind the live ones (nothing reads them there): loads
 * and stores share one counter, and a store that may be skipped makes the
 * compiler wait for loads that are still wanted in flight. */
template <int DIM, bool ID>
__device__ __forceinline__ void scatter_full(const ScatterArgs &sc, const KeyDesc &kd,
                                             const SortPay<DIM, ID> &q, int *base) {
  int d[SORT_DEPTH];
#pragma unroll
  for (int u = 0; u < SORT_DEPTH; ++u) d[u] = scatter_rank(kd, sort_key(q.c[u], kd), ~0ull, base);
#pragma unroll
  for (int u = 0; u < SORT_DEPTH; ++u) scatter_store<DIM, ID>(sc, q, u, d[u]);
}

template <int DIM, bool ID>
__device__ __forceinline__ void sort_scatter_body(const SortArgs &a, const int blk) {
  extern __shared__ int base[];
  const int row = blk;
  const long long np = a.hdr[HDR_NP_OLD];
  const long long b0 = (long long)row * a.strip;
  if (b0 >= np) return;
  const int lane = threadIdx.x;
  const ScatterArgs sc = a.sc;
  const KeyDesc kd = a.kd;
  const long long end = min(np, b0 + a.strip);
  /* two sets of records: the next rounds' loads are issued before the current
   * ones are ranked and written */
  SortPay<DIM, ID> A, B;
  long long p = b0 + lane;
  scatter_load(sc, p, np, A);
  const int *__restrict__ Hb = a.H + (size_t)row * a.nb1;
  const int *__restrict__ st = a.start;
#pragma unroll 8
  for (int b = lane; b < a.nb1; b += SORT_WAVE) base[b] = st[b] + Hb[b];
  sort_wave_fence();
  long long left = end - b0; /* particles not written yet */
  while (left >= 2 * SORT_STRIP_MIN) {
    scatter_load(sc, p + SORT_STRIP_MIN, np, B);
    scatter_full(sc, kd, A, base);
    scatter_load(sc, p + 2 * SORT_STRIP_MIN, np, A);
    scatter_full(sc, kd, B, base);
    p += 2 * SORT_STRIP_MIN;
    left -= 2 * SORT_STRIP_MIN;
  }
  /* the last rounds of the strip, partly filled at the end of the particles */
  while (left > 0) {
    scatter_load(sc, p + SORT_STRIP_MIN, np, B);
#pragma unroll
    for (int u = 0; u < SORT_DEPTH; ++u) {
      const bool valid = u * SORT_WAVE + lane < left;
      const unsigned long long all = __ballot(valid);
      if (all == 0ull) break;
      const int d = scatter_rank(kd, valid ? sort_key(A.c[u], kd) : -1, all, base);
      if (valid) scatter_store<DIM, ID>(sc, A, u, d);
    }
    A = B;
    p += SORT_STRIP_MIN;
    left -= SORT_STRIP_MIN;
  }
}

template <int DIM, bool ID>
__global__ __launch_bounds__(SORT_WAVE) void k_sort_scatter(SortArgs a) {
  sort_scatter_body<DIM, ID>(a, blockIdx.x);
}

/* scratch sizing and arguments of a pass reading buffer `b` */
static int sort_prepare(iskra_ctx *c, int sid, int mode, int build, int b, SortArgs *A) {
  IskSpecies *s = &c->sp[sid];
  KeyDesc kd;
  kd.mode = mode;
  kd.dim = c->g.dim;
  kd.T = c->t.T;
  kd.log2T = c->t.log2T;
  kd.ntx = c->ntx;
  const int cells = c->g.dim == 2 ? c->t.T * c->t.T : c->t.T;
  kd.nbins = mode == 0 ? c->ntiles : mode == 1 ? cells : c->ntiles * cells;
  const int nb1 = kd.nbins + 1;
  kd.nbits = 1;
  while ((1 << kd.nbits) <= kd.nbins) ++kd.nbits;
  if (nb1 > ISK_SORT_BINS) {
    isk_set_error("sort: %d bins exceed %d", kd.nbins, ISK_SORT_BINS - 1);
    return ISKRA_E_UNSUPPORTED;
  }
  /* strip length: SORT_STRIPS strips, none shorter than an eighth of the bins
   * (its table row is written and read once), the table bounded */
  int strip = SORT_STRIP_MIN;
  while (strip < SORT_STRIP_MAX &&
         ((int64_t)strip * SORT_STRIPS < s->cap - s->cap / 8 || strip * 8 < nb1 ||
          (s->cap + strip - 1) / strip * nb1 > SORT_TABLE_MAX))
    strip *= 2;
  const int nrow = std::max(1, (int)((s->cap + strip - 1) / strip));
  const int64_t need_H = (int64_t)nrow * nb1;
  if (need_H > c->sort_H_words) {
    isk_free(c->sort_H);
    c->sort_H = nullptr;
    c->sort_H_words = 0;
    if (isk_alloc((void **)&c->sort_H, need_H * 4)) return ISKRA_E_HIP;
    c->sort_H_words = need_H;
  }
  if (!c->sort_tot && isk_alloc((void **)&c->sort_tot, (int64_t)(ISK_SORT_BINS + 1) * 4))
    return ISKRA_E_HIP;
  if (!c->sort_start && isk_alloc((void **)&c->sort_start, (int64_t)(ISK_SORT_BINS + 1) * 4))
    return ISKRA_E_HIP;
  int o = 1 - b;
  A->kd = kd;
  A->hdr = s->hdr;
  A->H = c->sort_H;
  A->tot = c->sort_tot;
  A->start = c->sort_start;
  A->nb1 = nb1;
  A->nrow = nrow;
  A->strip = strip;
  A->ngrp = (nb1 + SORT_CB - 1) / SORT_CB;
  A->one = A->ngrp == 1 && nrow <= SORT_ONE_MAX;
  A->span = mode == 2 ? cells : 1;
  ScatterArgs &a = A->sc;
  a.cell = s->cell[b];
  a.ox = s->ox[b];
  a.oy = s->oy[b];
  a.vx = s->vx[b];
  a.vy = s->vy[b];
  a.vz = s->vz[b];
  a.id = s->track_ids ? s->id[b] : nullptr;
  a.cell_o = s->cell[o];
  a.ox_o = s->ox[o];
  a.oy_o = s->oy[o];
  a.vx_o = s->vx[o];
  a.vy_o = s->vy[o];
  a.vz_o = s->vz[o];
  a.id_o = s->track_ids ? s->id[o] : nullptr;
  A->build = build;
  A->CH = c->t.CH;
  A->chunks = s->chunks;
  A->tcb = s->tile_chunk_begin;
  return ISKRA_OK;
}

static int sort_pass(iskra_ctx *c, int sid, int mode, int build) {
  IskSpecies *s = &c->sp[sid];
  SortArgs A;
  int rc = sort_prepare(c, sid, mode, build, s->cur, &A);
  if (rc) return rc;
  const size_t shm = (size_t)A.nb1 * sizeof(int);
  const dim3 rows(A.nrow), wave(SORT_WAVE), wide(1024);
  /* four waves count a strip that gives each of them enough loads at once (in a batch
   * one does: most of its work-groups find no particles, and those are what it takes) */
  const dim3 count(A.strip >= SORT_KEYS * SORT_HIST / 4 ? SORT_HIST : SORT_WAVE);
  hipLaunchKernelGGL(k_sort_hist, rows, count, shm, c->stream, A);
  ISK_CHECK_LAUNCH();
  if (A.one) {
    hipLaunchKernelGGL(k_sort_table, dim3(1), wide, 0, c->stream, A);
  } else {
    hipLaunchKernelGGL(k_sort_cols, dim3(A.ngrp), wide, 0, c->stream, A);
    ISK_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_sort_bins, dim3(1), wide, 0, c->stream, A);
  }
  ISK_CHECK_LAUNCH();
  auto scatter = A.kd.dim == 2
                     ? (A.sc.id ? k_sort_scatter<2, true> : k_sort_scatter<2, false>)
                     : (A.sc.id ? k_sort_scatter<1, true> : k_sort_scatter<1, false>);
  hipLaunchKernelGGL(scatter, rows, wave, shm, c->stream, A);
  ISK_CHECK_LAUNCH();
  s->cur = 1 - s->cur;
  return ISKRA_OK;
}

int isk_sort_species(iskra_ctx *c, int sid, int exact_cell) {
  int rc;
  hipEvent_t ev = nullptr;
  if ((rc = isk_prof_begin(c, &ev))) return rc;
  /* by exact cell: one pass over the cells in tile order where their bins fit
   * the sort's table, else by cell inside the tile and then by tile (each
   * pass is stable, so both give the same order) */
  const int cells = c->g.dim == 2 ? c->t.T * c->t.T : c->t.T;
  const bool single = exact_cell && (int64_t)c->ntiles * cells + 1 <= ISK_SORT_BINS;
  if (exact_cell && !single) {
    if ((rc = sort_pass(c, sid, 1, 0))) return rc;
  }
  if ((rc = sort_pass(c, sid, single ? 2 : 0, 1))) return rc;
  return isk_prof_end(c, ev, ISKRA_K_SORT, 0);
}

/* ------------------------------------------------------------------------ */
/* fused gather + push + boundary + deposit                                  */
/* ------------------------------------------------------------------------ */
struct PushArgs {
  int32_t *cell;
  float *ox, *oy, *vx, *vy;
  float *vz;     /* RZ pusher: v_theta, rotated with v_r */
  double dtdr;   /* RZ pusher: dt / dr */
  /* surface tracker (PM_TRACK): edge codes per cell and direction, tracked
   * cells, per-electrode hit counters of this species, dt and the spacing
   * the reference's check uses */
  const uint8_t *surf, *tracked;
  unsigned long long *ehit;
  double dt_d, dh_d;
  long long *hdr;
  const IskChunk *chunks;
  long long *partial;
  unsigned long long *gfall;
  const float *E;
  int nx, ny, ncx, ncy;
  int T, log2T, M, W, CH, ntx;
  float qmdt, dtdx, dtdy;
  int bndx, bndy;
  int do_push;
  int *live_cnt; /* per work-group live particles pushed */
};

/* rn(a 2^32) and rn(a b 2^32) for offsets a, b in [0, 1): the FP64
 * products are exact (24 x 24 bit mantissas), rint rounds half to even, and
 * the results are below 2^32, so they convert to uint32 exactly */
__device__ __forceinline__ long long fix32_dev(float a) {
  return (long long)(unsigned int)__builtin_rint((double)a * 4294967296.0);
}
__device__ __forceinline__ long long fixprod32_dev(float a, float b) {
  return (long long)(unsigned int)__builtin_rint(((double)a * (double)b) * 4294967296.0);
}

/* CIC weights in 2^-32 units: Wx = rn(hx 2^32), Wy = rn(hy 2^32), Wxy =
 * rn(hx hy 2^32); the four corners sum to exactly 2^32 */
__device__ __forceinline__ void fix_weights2(float hx, float hy, long long *w00,
                                             long long *w10, long long *w01,
                                             long long *w11) {
  long long Wx = fix32_dev(hx);
  long long Wy = fix32_dev(hy);
  long long Wxy = fixprod32_dev(hx, hy);
  *w11 = Wxy;
  *w10 = Wx - Wxy;
  *w01 = Wy - Wxy;
  *w00 = (1LL << 32) - Wx - Wy + Wxy;
}

/* one step of a coordinate: o += v*dtd, split off the integer part */
__device__ __forceinline__ int advance_coord(float v, float dtd, float *o) {
  float h = fmaf(v, dtd, *o);
  float f = floorf(h);
  h = h - f;
  if (h >= 1.0f) {
    h = 0.0f;
    f += 1.0f;
  }
  *o = h;
  return (int)f;
}

/* transform_from_cartesian_to_cylindrical! (pushers.jl:52-66) in cell units,
 * after the Cartesian step of the radial coordinate: the particle sits at
 * X = i + hx + v_r dt/dr in the plane through its old position and the axis
 * and has moved Y = v_theta dt/dr out of it; it is rotated back to radius
 * R = sqrt(X^2 + Y^2) with sin = Y/R (0 when R = 0, the reference's
 * r .~ 0 test) and cos = +sqrt(1 - sin^2) (also for X < 0, as the reference
 * takes it), and (v_r, v_theta) rotated by the same angle.  FP64 throughout
 * (correctly rounded sqrt and division); R beyond 2^30 cells maps to a cell
 * index no grid has. */
__device__ __forceinline__ void rz_transform(int *i, float *hx, float *vr, float *vt,
                                             double dtdr) {
  const double X = (double)*i + ((double)*hx + (double)*vr * dtdr);
  const double Y = (double)*vt * dtdr;
  const double R = sqrt(X * X + Y * Y);
  const double sn = R == 0.0 ? 0.0 : Y / R;
  const double cs = sqrt(1.0 - sn * sn);
  const double nvr = cs * (double)*vr + sn * (double)*vt;
  const double nvt = cs * (double)*vt - sn * (double)*vr;
  int ii;
  float h;
  if (R < 1073741824.0) {
    const double fl = floor(R);
    ii = (int)fl;
    h = (float)(R - fl);
    if (h >= 1.0f) {
      h = 0.0f;
      ++ii;
    }
  } else {
    ii = 1 << 30;
    h = 0.0f;
  }
  *i = ii;
  *hx = h;
  *vr = (float)nvr;
  *vt = (float)nvt;
}

/* pusher modes of the push kernels */
enum { PM_XY = 0, PM_RZ = 1, PM_TRACK = 2 };

/* track! + check! + hit! of the reference's surface tracker
 * (pic/surfaces/track.jl:152-161, check.jl:17-68, hit.jl:1-56,
 * circuit_coupling.jl:47-62) for one particle that starts in a tracked cell:
 * from its offsets (hx, hy) before the push it follows the straight path
 * with the pushed velocity (vx, vy) cell by cell for dt, in FP64 and in the
 * reference's operation order (one spacing dh for both axes, as check uses
 * st.dh).  At each edge crossed: no surface -> keep tracing from the next
 * cell; absorbing surface or fixed electrode -> absorbed; floating electrode
 * k -> absorbed and counted on electrode k; reflective surface -> the
 * velocity components along the edge normal flip, the position is corrected
 * by the reflected rest of the path (the reference's px -= v dt' ... px +=
 * v' dt'), and tracing resumes in the cell the particle came from
 * (scattered!); any other surface ends the tracing.  Returns 1 if absorbed;
 * *cx, *cy receive the position corrections in cells. */
#define ISK_TRACK_MAX 64
__device__ __forceinline__ int track_path(const PushArgs &a, int i, int j, float hx0, float hy0,
                                          float *vx, float *vy, double *cx, double *cy) {
  const double h = a.dh_d;
  double T = a.dt_d, hx = hx0, hy = hy0;
  *cx = 0.0;
  *cy = 0.0;
  for (int it = 0; it < ISK_TRACK_MAX; ++it) {
    const double vxd = *vx, vyd = *vy;
    const double dxs = vxd > 0 ? h * (1.0 - hx) : h * hx;
    const double dys = vyd > 0 ? h * (1.0 - hy) : h * hy;
    const double tx = dxs / fabs(vxd), ty = dys / fabs(vyd);
    if (T < tx && T < ty) return 0; /* stays in this cell */
    int ni = i, nj = j, dir;
    double nhx, nhy, Tn;
    if (tx < ty) {
      Tn = T - tx;
      nhy = hy + vyd * tx / h;
      if (vxd > 0) { ni = i + 1; nhx = 0.0; dir = 1; }
      else { ni = i - 1; nhx = 1.0; dir = 0; }
    } else {
      Tn = T - ty;
      nhx = hx + vxd * ty / h;
      if (vyd > 0) { nj = j + 1; nhy = 0.0; dir = 3; }
      else { nj = j - 1; nhy = 1.0; dir = 2; }
    }
    if (i < 0 || i >= a.ncx || j < 0 || j >= a.ncy) return 0; /* left the grid untracked */
    const int code = a.surf[(i + a.ncx * j) * 4 + dir];
    if (code == ISK_SURF_NONE) {
      i = ni;
      j = nj;
      hx = nhx;
      hy = nhy;
      T = Tn;
      continue;
    }
    if (code == ISK_SURF_ABSORB) return 1;
    if (code >= ISK_SURF_ELECTRODE) {
      atomicAdd(&a.ehit[code - ISK_SURF_ELECTRODE], 1ull);
      return 1;
    }
    if (code != ISK_SURF_REFLECT) return 0; /* hit!(::Surface) does nothing */
    if (ni != i) {
      *vx = -*vx;
      *cx += 2.0 * (double)*vx * Tn / h;
    }
    if (nj != j) {
      *vy = -*vy;
      *cy += 2.0 * (double)*vy * Tn / h;
    }
    /* scattered! (hit.jl:13-21) */
    int si = ni, sj = nj;
    double shx = nhx, shy = nhy;
    if (nhx == 0.0) { si = ni - 1; shx = 1.0; }
    if (nhx == 1.0) { si = ni + 1; shx = 0.0; }
    if (nhy == 0.0) { sj = nj - 1; shy = 1.0; }
    if (nhy == 1.0) { sj = nj + 1; shy = 0.0; }
    i = si;
    j = sj;
    hx = shx;
    hy = shy;
    T = Tn;
  }
  return 0;
}

/* a position correction of c cells added to (cell, offset), FP64 */
__device__ __forceinline__ int shift_coord(double c, float *o) {
  const double t = (double)*o + c;
  const double f = floor(t);
  float h = (float)(t - f);
  int k = (int)f;
  if (h >= 1.0f) {
    h = 0.0f;
    ++k;
  }
  *o = h;
  return k;
}

/* boundary on one axis; returns false if the particle is discarded */
__device__ __forceinline__ bool apply_bnd(int *i, int n, int mode) {
  if (*i >= 0 && *i < n) return true;
  if (mode == ISKRA_BND_WRAP) {
    int r = *i % n;
    if (r < 0) r += n;
    *i = r;
    return true;
  }
  return false; /* discard (NONE also removes particles that leave the grid) */
}

template <int DIM>
struct PushRegs {
  static constexpr int U = PushShape<DIM>::unroll;
  int32_t c[U];
  float hx[U], hy[U], vx[U], vy[U];
};

/* pointers are the work-group's first particle (uniform), indices 32-bit */
template <int DIM>
__device__ __forceinline__ void push_load(PushRegs<DIM> &r, const int32_t *__restrict__ cb,
                                          const float *__restrict__ oxb,
                                          const float *__restrict__ oyb,
                                          const float *__restrict__ vxb,
                                          const float *__restrict__ vyb, unsigned count,
                                          unsigned b0) {
  /* branch-free: slots past the end load the first particle (the caller
   * skips them); nothing here consumes a loaded value, so all loads of the
   * batch are in flight together */
#pragma unroll
  for (int u = 0; u < PushShape<DIM>::unroll; ++u) {
    const unsigned k = b0 + u * PushShape<DIM>::block + threadIdx.x;
    __builtin_assume(k < (1u << 24));
    const unsigned q = k < count ? k : 0u;
    r.c[u] = cb[q];
    r.hx[u] = oxb[q];
    r.vx[u] = vxb[q];
    r.hy[u] = DIM == 2 ? oyb[q] : 0.f;
    r.vy[u] = DIM == 2 ? vyb[q] : 0.f;
  }
}

template <int DIM, int PM = PM_XY>
__device__ __forceinline__ void push_body(const PushArgs &a, const int blk) {
  constexpr bool RZ = PM == PM_RZ, TRACK = PM == PM_TRACK;
  constexpr int BLK = PushShape<DIM>::block, UNR = PushShape<DIM>::unroll;
  extern __shared__ unsigned long long sD[]; /* WW deposit counters, then E */
  const int W = a.W;
  const int WW = DIM == 2 ? W * W : W;
  float *sE = reinterpret_cast<float *>(sD + WW);
  int32_t *__restrict__ cellp = a.cell;
  float *__restrict__ oxp = a.ox;
  float *__restrict__ oyp = a.oy;
  float *__restrict__ vxp = a.vx;
  float *__restrict__ vyp = a.vy;
  const long long nch = a.hdr[HDR_NCHUNKS];
  const long long np = a.hdr[HDR_NP];
  const long long nps = a.hdr[HDR_NP_SORTED];
  long long start, count;
  bool windowed;
  int wx0 = 0, wy0 = 0;
  if ((long long)blk < nch) {
    IskChunk ch = a.chunks[blk];
    start = ch.start;
    count = ch.count;
    windowed = true;
    if (DIM == 2) {
      int ti = ch.tile % a.ntx, tj = ch.tile / a.ntx;
      wx0 = ti * a.T - a.M;
      wy0 = tj * a.T - a.M;
    } else {
      wx0 = ch.tile * a.T - a.M;
    }
  } else {
    start = nps + ((long long)blk - nch) * a.CH;
    if (start >= np) {
      if (threadIdx.x == 0) a.live_cnt[blk] = 0;
      return;
    }
    count = min((long long)a.CH, np - start);
    windowed = false;
  }
  /* the first batch of particles is requested before the E window, so the
   * two memory latencies overlap instead of following each other */
  int32_t *__restrict__ cb = cellp + start;
  float *__restrict__ oxb = oxp + start;
  float *__restrict__ oyb = DIM == 2 ? oyp + start : oyp;
  float *__restrict__ vxb = vxp + start;
  float *__restrict__ vyb = DIM == 2 ? vyp + start : vyp;
  const unsigned ucount = (unsigned)count;
  PushRegs<DIM> cur;
  push_load<DIM>(cur, cb, oxb, oyb, vxb, vyb, ucount, 0u);
  if (windowed) {
    for (int k = threadIdx.x; k < WW; k += BLK) {
      sD[k] = 0ull;
      if (a.do_push) {
        int li = DIM == 2 ? k % W : k;
        int lj = DIM == 2 ? k / W : 0;
        int gi = wx0 + li, gj = wy0 + lj;
        bool in = gi >= 0 && gi < a.nx && (DIM == 1 || (gj >= 0 && gj < a.ny));
        if (DIM == 2) {
          float2 e = in ? reinterpret_cast<const float2 *>(a.E)[gj * a.nx + gi]
                        : make_float2(0.f, 0.f);
          sE[2 * k] = e.x;
          sE[2 * k + 1] = e.y;
        } else {
          sE[k] = in ? a.E[gi] : 0.f;
        }
      }
    }
    __syncthreads();
  }
  int live = 0;
  const long long per = (long long)BLK * UNR;
  for (long long b0 = 0; b0 < count; b0 += per) {
    /* a batch of UNR particles per thread: all loads, then compute + stores */
    if (b0 > 0) push_load<DIM>(cur, cb, oxb, oyb, vxb, vyb, ucount, (unsigned)b0);
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const unsigned kslot = (unsigned)b0 + u * BLK + threadIdx.x;
      if (kslot >= ucount) continue;
      int32_t c = cur.c[u];
      if (c < 0) continue;
      int i = c & 0xFFFF;
      int j = c >> 16;
      float hx = cur.hx[u], hy = cur.hy[u], vx = cur.vx[u], vy = cur.vy[u];
      float vt = 0.f;
      bool alive = true;
      if (a.do_push) {
        /* gather (cloud_in_cell.jl:20-36) */
        float ax = 1.0f - hx;
        float Ex, Ey = 0.f;
        if (DIM == 2) {
          float ay = 1.0f - hy;
          float w00 = ax * ay, w10 = hx * ay, w01 = ax * hy, w11 = hx * hy;
          float2 e00, e10, e01, e11;
          int li = i - wx0, lj = j - wy0;
          if (windowed && (unsigned)li < (unsigned)(W - 1) && (unsigned)lj < (unsigned)(W - 1)) {
            int q = lj * W + li;
            e00 = make_float2(sE[2 * q], sE[2 * q + 1]);
            e10 = make_float2(sE[2 * q + 2], sE[2 * q + 3]);
            e01 = make_float2(sE[2 * (q + W)], sE[2 * (q + W) + 1]);
            e11 = make_float2(sE[2 * (q + W) + 2], sE[2 * (q + W) + 3]);
          } else {
            const float2 *E2 = reinterpret_cast<const float2 *>(a.E);
            int q = j * a.nx + i;
            e00 = E2[q];
            e10 = E2[q + 1];
            e01 = E2[q + a.nx];
            e11 = E2[q + a.nx + 1];
          }
          Ex = fmaf(w11, e11.x, fmaf(w01, e01.x, fmaf(w10, e10.x, w00 * e00.x)));
          Ey = fmaf(w11, e11.y, fmaf(w01, e01.y, fmaf(w10, e10.y, w00 * e00.y)));
        } else {
          float e0, e1;
          int li = i - wx0;
          if (windowed && (unsigned)li < (unsigned)(W - 1)) {
            e0 = sE[li];
            e1 = sE[li + 1];
          } else {
            e0 = a.E[i];
            e1 = a.E[i + 1];
          }
          Ex = fmaf(hx, e1, ax * e0);
        }
        /* push with B = 0 (pushers.jl:37-50): v += (q/m) E dt, x += v dt */
        vx = fmaf(a.qmdt, Ex, vx);
        if (TRACK && DIM == 2) {
          /* track! before the push, check! after it (ParticleInCell.jl:55-60) */
          vy = fmaf(a.qmdt, Ey, vy);
          const float vx0 = vx, vy0 = vy;
          double cx = 0.0, cy = 0.0;
          int absorbed = 0;
          if (a.tracked[i + a.ncx * j])
            absorbed = track_path(a, i, j, hx, hy, &vx, &vy, &cx, &cy);
          i += advance_coord(vx0, a.dtdx, &hx);
          j += advance_coord(vy0, a.dtdy, &hy);
          if (cx != 0.0) i += shift_coord(cx, &hx);
          if (cy != 0.0) j += shift_coord(cy, &hy);
          alive = apply_bnd(&i, a.ncx, a.bndx);
          alive = apply_bnd(&j, a.ncy, a.bndy) && alive;
          if (absorbed) alive = false;
        } else {
          if (RZ) {
            vt = a.vz[start + kslot];
            rz_transform(&i, &hx, &vx, &vt, a.dtdr);
          } else {
            i += advance_coord(vx, a.dtdx, &hx);
          }
          alive = apply_bnd(&i, a.ncx, a.bndx);
          if (DIM == 2) {
            vy = fmaf(a.qmdt, Ey, vy);
            j += advance_coord(vy, a.dtdy, &hy);
            alive = apply_bnd(&j, a.ncy, a.bndy) && alive;
          }
        }
      }
      if (alive) {
        ++live;
        /* deposit (cloud_in_cell.jl:1-18) */
        if (DIM == 2) {
          long long w00, w10, w01, w11;
          fix_weights2(hx, hy, &w00, &w10, &w01, &w11);
          int li = i - wx0, lj = j - wy0;
          if (windowed && (unsigned)li < (unsigned)(W - 1) && (unsigned)lj < (unsigned)(W - 1)) {
            int q = lj * W + li;
            atomicAdd(&sD[q], (unsigned long long)w00);
            atomicAdd(&sD[q + 1], (unsigned long long)w10);
            atomicAdd(&sD[q + W], (unsigned long long)w01);
            atomicAdd(&sD[q + W + 1], (unsigned long long)w11);
          } else {
            int q = j * a.nx + i;
            atomicAdd(&a.gfall[q], (unsigned long long)w00);
            atomicAdd(&a.gfall[q + 1], (unsigned long long)w10);
            atomicAdd(&a.gfall[q + a.nx], (unsigned long long)w01);
            atomicAdd(&a.gfall[q + a.nx + 1], (unsigned long long)w11);
          }
        } else {
          long long w1 = fix32_dev(hx);
          long long w0 = (1LL << 32) - w1;
          int li = i - wx0;
          if (windowed && (unsigned)li < (unsigned)(W - 1)) {
            atomicAdd(&sD[li], (unsigned long long)w0);
            atomicAdd(&sD[li + 1], (unsigned long long)w1);
          } else {
            atomicAdd(&a.gfall[i], (unsigned long long)w0);
            atomicAdd(&a.gfall[i + 1], (unsigned long long)w1);
          }
        }
      }
      if (a.do_push) {
        const unsigned k = (unsigned)b0 + u * BLK + threadIdx.x;
        /* the cell is stored only when it changed: slow particles (the ions)
         * then leave whole sectors of the cell array unwritten */
        const int32_t nc = alive ? (i | (j << 16)) : -1;
        if (nc != c) cb[k] = nc;
        oxb[k] = hx;
        vxb[k] = vx;
        if (DIM == 2) {
          oyb[k] = hy;
          vyb[k] = vy;
        }
        if (RZ) a.vz[start + k] = vt;
      }
    }
  }
  /* per-work-group live count (summed by the merge kernel, no atomics) */
  __shared__ int wl[BLK / 64];
  for (int off = 32; off > 0; off >>= 1) live += __shfl_xor(live, off);
  if ((threadIdx.x & 63) == 0) wl[threadIdx.x >> 6] = live;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int k = 0; k < BLK / 64; ++k) t += wl[k];
    a.live_cnt[blk] = t;
  }
  if (windowed) {
    long long *dst = a.partial + (size_t)blk * WW;
    for (int k = threadIdx.x; k < WW; k += BLK) dst[k] = (long long)sD[k];
  }
}

template <int DIM, int PM = PM_XY>
__global__ __launch_bounds__(PushShape<DIM>::block) void k_push(PushArgs a) {
  push_body<DIM, PM>(a, blockIdx.x);
}

/* arguments of one push launch reading buffer `b`; grid and LDS size */
static void push_prepare(iskra_ctx *c, int sid, double dt, int do_push, int b, PushArgs *pa,
                         int *grid, size_t *shm) {
  IskSpecies *s = &c->sp[sid];
  const IskGrid &g = c->g;
  PushArgs &a = *pa;
  a.cell = s->cell[b];
  a.ox = s->ox[b];
  a.oy = s->oy[b];
  a.vx = s->vx[b];
  a.vy = s->vy[b];
  a.vz = s->vz[b];
  a.dtdr = dt / g.dx;
  a.surf = c->trk.surf;
  a.tracked = c->trk.tracked;
  a.ehit = s->ehit;
  a.dt_d = dt;
  a.dh_d = g.dx;
  a.hdr = s->hdr;
  a.chunks = s->chunks;
  a.partial = s->partial;
  a.gfall = s->gfall;
  a.E = c->E;
  a.nx = g.nx;
  a.ny = g.ny;
  a.ncx = g.ncx;
  a.ncy = g.ncy;
  a.T = c->t.T;
  a.log2T = c->t.log2T;
  a.M = isk_sp_margin(c, sid);
  a.W = isk_sp_window(c, sid);
  a.CH = c->t.CH;
  a.ntx = c->ntx;
  a.qmdt = (float)(s->q / s->m * dt);
  a.dtdx = (float)(dt / g.dx);
  a.dtdy = (float)(dt / g.dy);
  a.bndx = s->bnd[0];
  a.bndy = s->bnd[1];
  a.do_push = do_push;
  a.live_cnt = s->live_cnt;
  *grid = (int)s->max_chunks;
  int WW = g.dim == 2 ? a.W * a.W : a.W;
  *shm = (size_t)WW * (8 + 4 * g.dim);
}

/* the push (or deposit-only) launch of one species; fill != 0 clears the
 * fallback grid first (every merge clears it after reading, so a push that
 * follows a merge finds it zero) */
static int push_launch(iskra_ctx *c, int sid, double dt, int do_push, int fill) {
  IskSpecies *s = &c->sp[sid];
  int rc;
  if (fill && (rc = isk_fill_i64(c, s->gfall, isk_nodes(c), 0))) return rc;
  PushArgs a;
  int grid;
  size_t shm;
  push_prepare(c, sid, dt, do_push, s->cur, &a, &grid, &shm);
  hipEvent_t ev = nullptr;
  if (do_push) {
    int rc2 = isk_prof_begin(c, &ev);
    if (rc2) return rc2;
  }
  if (c->g.dim == 2 && c->pusher == ISKRA_PUSHER_RZ && do_push)
    hipLaunchKernelGGL((k_push<2, PM_RZ>), dim3(grid), dim3(PushShape<2>::block), shm, c->stream,
                       a);
  else if (c->g.dim == 2 && c->trk.on && do_push)
    hipLaunchKernelGGL((k_push<2, PM_TRACK>), dim3(grid), dim3(PushShape<2>::block), shm,
                       c->stream, a);
  else if (c->g.dim == 2)
    hipLaunchKernelGGL(k_push<2>, dim3(grid), dim3(PushShape<2>::block), shm, c->stream, a);
  else
    hipLaunchKernelGGL(k_push<1>, dim3(grid), dim3(PushShape<1>::block), shm, c->stream, a);
  ISK_CHECK_LAUNCH();
  if (do_push) {
    int rc2 = isk_prof_end(c, ev, ISKRA_K_PUSH, 0);
    if (rc2) return rc2;
  }
  return ISKRA_OK;
}

/* the pushes of all species in one launch: work-group g belongs to species
 * s with bstart[s] <= g < bstart[s+1] and acts as work-group g - bstart[s]
 * of that species' own launch (one launch boundary less per step, and the
 * tail of one species overlaps the next) */
struct PushMulti {
  PushArgs a[ISK_MAX_SPECIES];
  int bstart[ISK_MAX_SPECIES + 1];
  int n;
};

template <int DIM, int PM = PM_XY>
__global__ __launch_bounds__(PushShape<DIM>::block) void k_push_multi(PushMulti m) {
  int s = 0;
  while (s + 1 < m.n && (int)blockIdx.x >= m.bstart[s + 1]) ++s;
  /* a copy in registers: read through a reference into the argument block,
   * the fields would be re-read from memory after every particle's stores */
  const PushArgs a = m.a[s];
  push_body<DIM, PM>(a, blockIdx.x - m.bstart[s]);
}

static int push_launch_all(iskra_ctx *c, double dt) {
  if (c->nspecies == 0) return ISKRA_OK;
  PushMulti m;
  size_t shm = 0;
  m.n = c->nspecies;
  m.bstart[0] = 0;
  for (int s = 0; s < c->nspecies; ++s) {
    int grid;
    size_t sh;
    push_prepare(c, s, dt, 1, c->sp[s].cur, &m.a[s], &grid, &sh);
    m.bstart[s + 1] = m.bstart[s] + grid;
    shm = std::max(shm, sh);
  }
  if (m.bstart[c->nspecies] == 0) return ISKRA_OK;
  hipEvent_t ev = nullptr;
  int rc = isk_prof_begin(c, &ev);
  if (rc) return rc;
  if (c->g.dim == 2 && c->pusher == ISKRA_PUSHER_RZ)
    hipLaunchKernelGGL((k_push_multi<2, PM_RZ>), dim3(m.bstart[m.n]), dim3(PushShape<2>::block),
                       shm, c->stream, m);
  else if (c->g.dim == 2 && c->trk.on)
    hipLaunchKernelGGL((k_push_multi<2, PM_TRACK>), dim3(m.bstart[m.n]),
                       dim3(PushShape<2>::block), shm, c->stream, m);
  else if (c->g.dim == 2)
    hipLaunchKernelGGL(k_push_multi<2>, dim3(m.bstart[m.n]), dim3(PushShape<2>::block), shm,
                       c->stream, m);
  else
    hipLaunchKernelGGL(k_push_multi<1>, dim3(m.bstart[m.n]), dim3(PushShape<1>::block), shm,
                       c->stream, m);
  ISK_CHECK_LAUNCH();
  return isk_prof_end(c, ev, ISKRA_K_PUSH, 0);
}

int isk_push_species(iskra_ctx *c, int sid, double dt, int do_push) {
  int rc = push_launch(c, sid, dt, do_push, 1);
  if (rc) return rc;
  c->sp[sid].deposited = 1;
  hipEvent_t em = nullptr;
  if ((rc = isk_prof_begin(c, &em))) return rc;
  if ((rc = isk_merge_species(c, sid, do_push))) return rc;
  return isk_prof_end(c, em, ISKRA_K_MERGE, 0);
}

/* ------------------------------------------------------------------------ */
/* deterministic merge of the chunk windows                                  */
/* ------------------------------------------------------------------------ */
struct MergeArgs {
  const long long *tilewin; /* 2-D: per-tile sums of the chunk windows (null: per chunk) */
  const int *live_cnt;
  int nlive; /* entries of live_cnt to add to HDR_PUSHED (0: deposit only) */
  long long *hdr_rw;
  const long long *partial;
  unsigned long long *gfall; /* read, then cleared for the next push */
  const int *tcb;
  const long long *hdr;
  long long *cnt;
  int nx, ny, T, M, W, ntx, nty;
};

/* pushed-particle count of the step: sum of the per-chunk live counts */
__device__ __forceinline__ void merge_live(const MergeArgs &a, const int blk, const int nblk) {
  __shared__ unsigned long long ls[4];
  unsigned long long sum = 0;
  for (int k = blk * blockDim.x + threadIdx.x; k < a.nlive; k += nblk * blockDim.x)
    sum += (unsigned long long)a.live_cnt[k];
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if ((threadIdx.x & 63) == 0) ls[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = ls[0] + ls[1] + ls[2] + ls[3];
    if (t) atomicAdd((unsigned long long *)&a.hdr_rw[HDR_PUSHED], t);
  }
  __syncthreads();
}

/* deposit count of one node: fallback grid + the windows that cover it.
 * Window of tile t spans nodes [tT - M, tT - M + W - 1] per axis, so the
 * covering tiles are t in [ceil((i + M - W + 1) / T), floor((i + M) / T)]:
 * at most 4 per axis because the margin M is at most T.  All terms are
 * int64, so the sum does not depend on the order of the additions. */
__device__ __forceinline__ int merge_tlo(int i, const MergeArgs &a) {
  const int u = i + a.M - a.W + 1;
  return u <= 0 ? 0 : (u + a.T - 1) / a.T;
}

template <int DIM>
__device__ __forceinline__ long long merge_node(const MergeArgs &a, const int node) {
  const int i = node % a.nx, j = node / a.nx;
  const unsigned long long g = a.gfall[node];
  if (g) a.gfall[node] = 0ull;
  long long s = (long long)g;
  if (a.hdr[HDR_NCHUNKS] <= 0) return s;
  const int WW = DIM == 2 ? a.W * a.W : a.W;
  const int tlo = merge_tlo(i, a), thi = min((i + a.M) / a.T, a.ntx - 1);
  const int ulo = DIM == 2 ? merge_tlo(j, a) : 0;
  const int uhi = DIM == 2 ? min((j + a.M) / a.T, a.nty - 1) : 0;
  if (DIM == 1 && a.tilewin) {
    for (int ti = tlo; ti <= thi; ++ti) s += a.tilewin[(size_t)ti * WW + (i - (ti * a.T - a.M))];
    return s;
  }
  if (DIM == 2 && a.tilewin) {
    long long v[16];
#pragma unroll
    for (int dy = 0; dy < 4; ++dy)
#pragma unroll
      for (int dx = 0; dx < 4; ++dx) {
        const int ti = tlo + dx, tj = ulo + dy;
        const int li = i - (ti * a.T - a.M), lj = j - (tj * a.T - a.M);
        v[4 * dy + dx] = (ti <= thi && tj <= uhi)
                             ? a.tilewin[(size_t)(ti + a.ntx * tj) * WW + lj * a.W + li]
                             : 0ll;
      }
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
    return s;
  }
  for (int tj = ulo; tj <= uhi; ++tj) {
    const int lj = j - (tj * a.T - a.M);
    for (int ti = tlo; ti <= thi; ++ti) {
      const int li = i - (ti * a.T - a.M);
      const int t = ti + a.ntx * tj;
      const int q = DIM == 2 ? lj * a.W + li : li;
      const int k1 = a.tcb[t + 1];
      for (int k = a.tcb[t]; k < k1; k += 8) {
        long long v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = k + u < k1 ? a.partial[(size_t)(k + u) * WW + q] : 0ll;
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
      }
    }
  }
  return s;
}

template <int DIM>
__device__ __forceinline__ void merge_body(const MergeArgs &a, const int blk, const int nblk) {
  if (a.nlive > 0) merge_live(a, blk, nblk);
  const int node = blk * blockDim.x + threadIdx.x;
  if (node >= a.nx * a.ny) return;
  a.cnt[node] = merge_node<DIM>(a, node);
}

template <int DIM>
__global__ __launch_bounds__(256) void k_merge(MergeArgs a) {
  merge_body<DIM>(a, blockIdx.x, gridDim.x);
}

/* stage 1 of the 2-D merge: one work-group per tile sums its chunks' windows
 * (contiguous in memory, chunks of a tile are consecutive) */
__device__ __forceinline__ void merge_tile_body(const long long *__restrict__ partial,
                                                const int *__restrict__ tcb,
                                                const long long *__restrict__ hdr,
                                                long long *__restrict__ tilewin, int WW, int t) {
  const int k0 = hdr[HDR_NCHUNKS] > 0 ? tcb[t] : 0, k1 = hdr[HDR_NCHUNKS] > 0 ? tcb[t + 1] : 0;
  if (2 * WW <= (int)blockDim.x) {
    /* narrow (1-D) windows: G = blockDim / WW thread groups take every G-th
     * chunk of the tile, then the G partial sums are added in LDS (integer
     * sums: any grouping gives the same result) */
    __shared__ long long red[256];
    const int G = (int)blockDim.x / WW, q = (int)threadIdx.x % WW, g = (int)threadIdx.x / WW;
    long long s0 = 0, s1 = 0;
    if (g < G) {
      int k = k0 + g;
      for (; k + G < k1; k += 2 * G) {
        s0 += partial[(size_t)k * WW + q];
        s1 += partial[(size_t)(k + G) * WW + q];
      }
      if (k < k1) s0 += partial[(size_t)k * WW + q];
    }
    red[threadIdx.x] = s0 + s1;
    __syncthreads();
    if (g == 0) {
      long long v = red[threadIdx.x];
      for (int h = 1; h < G; ++h) v += red[threadIdx.x + h * WW];
      tilewin[(size_t)t * WW + q] = v;
    }
    return;
  }
  for (int q = threadIdx.x; q < WW; q += blockDim.x) {
    /* four independent partial sums keep four loads in flight (integer
     * sums: the grouping does not change the result) */
    long long s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int k = k0;
    for (; k + 4 <= k1; k += 4) {
      s0 += partial[(size_t)k * WW + q];
      s1 += partial[(size_t)(k + 1) * WW + q];
      s2 += partial[(size_t)(k + 2) * WW + q];
      s3 += partial[(size_t)(k + 3) * WW + q];
    }
    for (; k < k1; ++k) s0 += partial[(size_t)k * WW + q];
    tilewin[(size_t)t * WW + q] = (s0 + s1) + (s2 + s3);
  }
}

__global__ __launch_bounds__(256) void k_merge_tiles(const long long *__restrict__ partial,
                                                     const int *__restrict__ tcb,
                                                     const long long *__restrict__ hdr,
                                                     long long *__restrict__ tilewin, int WW) {
  merge_tile_body(partial, tcb, hdr, tilewin, WW, blockIdx.x);
}

static void merge_prepare(iskra_ctx *c, int sid, int count_live, MergeArgs *pa, int *grid) {
  IskSpecies *s = &c->sp[sid];
  MergeArgs &a = *pa;
  a.live_cnt = s->live_cnt;
  a.nlive = count_live ? (int)s->max_chunks : 0;
  a.hdr_rw = s->hdr;
  a.partial = s->partial;
  a.gfall = s->gfall;
  a.tcb = s->tile_chunk_begin;
  a.hdr = s->hdr;
  a.cnt = s->cnt;
  a.nx = c->g.nx;
  a.ny = c->g.ny;
  a.T = c->t.T;
  a.M = isk_sp_margin(c, sid);
  a.W = isk_sp_window(c, sid);
  a.ntx = c->ntx;
  a.nty = c->nty;
  a.tilewin = nullptr;
  *grid = (isk_nodes(c) + 255) / 256;
}

int isk_merge_species(iskra_ctx *c, int sid, int count_live) {
  MergeArgs a;
  int grid;
  merge_prepare(c, sid, count_live, &a, &grid);
  IskSpecies *s = &c->sp[sid];
  const int W = isk_sp_window(c, sid);
  hipLaunchKernelGGL(k_merge_tiles, dim3(c->ntiles), dim3(256), 0, c->stream,
                     (const long long *)s->partial, (const int *)s->tile_chunk_begin,
                     (const long long *)s->hdr, s->tilewin, c->g.dim == 2 ? W * W : W);
  ISK_CHECK_LAUNCH();
  a.tilewin = s->tilewin;
  if (c->g.dim == 2)
    hipLaunchKernelGGL(k_merge<2>, dim3(grid), dim3(256), 0, c->stream, a);
  else
    hipLaunchKernelGGL(k_merge<1>, dim3(grid), dim3(256), 0, c->stream, a);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* ------------------------------------------------------------------------ */
/* rho = sum_s q_s n_s + background                                          */
/* ------------------------------------------------------------------------ */
struct RhoArgs {
  const long long *cnt[ISK_MAX_SPECIES];
  double qw[ISK_MAX_SPECIES]; /* w0 */
  double q[ISK_MAX_SPECIES];
  int ns;
  const double *vol, *bg;
  double *rho;
  int nn;
};

/* r + q_s n_s with n_s = count * w0 / V (count in 2^-32 units) */
__device__ __forceinline__ double rho_term(double r, long long cnt, double qw, double q, double V) {
  const double n = ((double)cnt * (1.0 / ISK_FIX_ONE)) * qw / V;
  return r + q * n;
}

__device__ __forceinline__ void rho_body(const RhoArgs &a, const int blk) {
  int node = blk * blockDim.x + threadIdx.x;
  if (node >= a.nn) return;
  double V = a.vol[node];
  double r = 0.0;
  for (int s = 0; s < a.ns; ++s) r = rho_term(r, a.cnt[s][node], a.qw[s], a.q[s], V);
  a.rho[node] = r + a.bg[node];
}

__global__ void k_rho(RhoArgs a) { rho_body(a, blockIdx.x); }

/* the time loop's deposit tail for all species in two launches: the tile
 * windows of every species (grid tiles x species), then per node the counts
 * of every species and rho (same arithmetic as k_merge + k_rho) */
struct MergeTilesN {
  const long long *partial[ISK_MAX_SPECIES];
  const int *tcb[ISK_MAX_SPECIES];
  const long long *hdr[ISK_MAX_SPECIES];
  long long *tilewin[ISK_MAX_SPECIES];
  int WW[ISK_MAX_SPECIES]; /* window nodes of each species */
};

__global__ __launch_bounds__(256) void k_merge_tiles_n(MergeTilesN a) {
  const int s = blockIdx.y;
  merge_tile_body(a.partial[s], a.tcb[s], a.hdr[s], a.tilewin[s], a.WW[s], blockIdx.x);
}

struct MergeRhoArgs {
  MergeArgs m[ISK_MAX_SPECIES];
  RhoArgs r;
  IskSpPack pk; /* F != null: also the spectral solve's packed right-hand side */
};

template <int DIM>
__global__ __launch_bounds__(256) void k_merge_rho(MergeRhoArgs a) {
  for (int s = 0; s < a.r.ns; ++s)
    if (a.m[s].nlive > 0) merge_live(a.m[s], blockIdx.x, gridDim.x);
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= a.r.nn) return;
  const double V = a.r.vol[node];
  double r = 0.0;
  for (int s = 0; s < a.r.ns; ++s) {
    const long long cnt = merge_node<DIM>(a.m[s], node);
    a.m[s].cnt[node] = cnt;
    r = rho_term(r, cnt, a.r.qw[s], a.r.q[s], V);
  }
  const double rho = r + a.r.bg[node];
  a.r.rho[node] = rho;
  if (DIM == 2 && a.pk.F) {
    const int nx = a.pk.s.nx, i = node % nx, j = node / nx;
    if (i > 0 && j > 0 && i < nx - 1 && j < a.pk.s.ny - 1)
      a.pk.F[(j - 1) * (nx - 2) + (i - 1)] = isk_sp_pack_value(a.pk, rho, i, j);
  }
}

int isk_rho(iskra_ctx *c) {
  RhoArgs a;
  int ns = 0;
  for (int s = 0; s < c->nspecies; ++s) {
    if (!c->sp[s].deposited) {
      int rc = isk_push_species(c, s, 0.0, 0);
      if (rc) return rc;
    }
    a.cnt[ns] = c->sp[s].cnt;
    a.qw[ns] = c->sp[s].w0;
    a.q[ns] = c->sp[s].q;
    ++ns;
  }
  a.ns = ns;
  a.vol = c->vol;
  a.bg = c->bg;
  a.rho = c->rho;
  a.nn = isk_nodes(c);
  hipLaunchKernelGGL(k_rho, dim3((a.nn + 255) / 256), dim3(256), 0, c->stream, a);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* ------------------------------------------------------------------------ */
/* 1-D grids: everything between the deposit and the next step               */
/* ------------------------------------------------------------------------ */
/* counts, rho, the direct solve, E and the electrode waveforms of a 1-D grid in
 * one work-group.  As four or five launches (merge and rho, solve, E, a waveform a
 * tag) these took 14.8 us a step at 65 nodes and 22 at 513, nearly all of it
 * launches.  What bounds the one launch is its chain of waits: all loads that
 * depend on nothing are requested first (21 us at 513 nodes with 256 threads
 * that loaded as they went), and phi stays in LDS until E is formed.  Measured:
 * 9.2 us at 65 nodes (periodic, 12 chunks merged here), 9.6 at 513. */
struct WaveDesc {
  int tag;
  double off, amp, f, ph; /* ph in turns */
};
struct Field1Args {
  MergeArgs m[ISK_MAX_SPECIES];
  RhoArgs r;
  TriArgs t;
  float *E;
  double dx;
  int nwave;
  WaveDesc wave[ISK_MAX_TAGS];
  double dt; /* waveforms at t = (step0 + *step_dev) dt */
  long long step0;
  const long long *step_dev;
};

#define FIELD1_BLOCK 1024
#define FIELD1_PER ((TRI_MAX + FIELD1_BLOCK - 1) / FIELD1_BLOCK)

/* a node's deposit: fallback grid (cleared for the next push) and the windows
 * that cover it, at most 4; the tile sums are zero where there are no chunks */
__device__ __forceinline__ long long field1_node(const MergeArgs &a, int i) {
  if (!a.tilewin) return merge_node<1>(a, i);
  const int lt = __builtin_ctz(a.T);
  const int u = i + a.M - a.W + 1;
  const int tlo = u <= 0 ? 0 : (u + a.T - 1) >> lt, thi = min((i + a.M) >> lt, a.ntx - 1);
  long long v[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int t = tlo + d;
    v[d] = t <= thi ? a.tilewin[(size_t)t * a.W + (i - ((t << lt) - a.M))] : 0ll;
  }
  const unsigned long long g = a.gfall[i];
  if (g) a.gfall[i] = 0ull;
  return (long long)g + ((v[0] + v[1]) + (v[2] + v[3]));
}

/* work-group 0: the field; work-group 1: the pushed-particle counts */
__device__ __forceinline__ void field1_body(const Field1Args &a, const int blk) {
  if (blk == 1) {
    for (int s = 0; s < a.r.ns; ++s) {
      unsigned long long sum = 0;
      for (int k = threadIdx.x; k < a.m[s].nlive; k += FIELD1_BLOCK)
        sum += (unsigned long long)a.m[s].live_cnt[k];
      for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
      if ((threadIdx.x & 63) == 0 && sum)
        atomicAdd((unsigned long long *)&a.m[s].hdr_rw[HDR_PUSHED], sum);
    }
    return;
  }
  __shared__ TriWork w;
  const int n = a.r.nn;
  if (n <= TRI_MAX) {
    /* everything that does not depend on another load is requested first */
    double V[FIELD1_PER], bg[FIELD1_PER], inv[FIELD1_PER], ma[FIELD1_PER], ncp[FIELD1_PER],
        r[FIELD1_PER];
    int tag[FIELD1_PER];
#pragma unroll
    for (int k = 0; k < FIELD1_PER; ++k) {
      const int i = min((int)threadIdx.x + k * FIELD1_BLOCK, n - 1);
      V[k] = a.r.vol[i];
      bg[k] = a.r.bg[i];
      inv[k] = a.t.inv[i];
      ma[k] = a.t.ma[i];
      ncp[k] = a.t.ncp[i];
      tag[k] = a.t.tags[i];
      r[k] = 0.0;
    }
    for (int s = 0; s < a.r.ns; ++s)
#pragma unroll
      for (int k = 0; k < FIELD1_PER; ++k) {
        const int i = threadIdx.x + k * FIELD1_BLOCK;
        if (i < n) {
          const long long cnt = field1_node(a.m[s], i);
          a.m[s].cnt[i] = cnt;
          r[k] = rho_term(r[k], cnt, a.r.qw[s], a.r.q[s], V[k]);
        }
      }
#pragma unroll
    for (int k = 0; k < FIELD1_PER; ++k) {
      const int i = threadIdx.x + k * FIELD1_BLOCK;
      if (i < n) {
        const double rho = r[k] + bg[k];
        a.r.rho[i] = rho;
        tri_load(a.t, w, i, rho, inv[k], ma[k], ncp[k], tag[k]);
      }
    }
    __syncthreads();
    tri_solve_lds(a.t, w);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += FIELD1_BLOCK)
      efield_node(w.B, a.E, 1, n, 1, a.dx, 1.0, i);
  } else {
    for (int i = threadIdx.x; i < n; i += FIELD1_BLOCK) {
      double r = 0.0;
      for (int s = 0; s < a.r.ns; ++s) {
        const long long cnt = field1_node(a.m[s], i);
        a.m[s].cnt[i] = cnt;
        r = rho_term(r, cnt, a.r.qw[s], a.r.q[s], a.r.vol[i]);
      }
      a.r.rho[i] = r + a.r.bg[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) tri_solve_body(a.t);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += FIELD1_BLOCK)
      efield_node(a.t.phi, a.E, 1, n, 1, a.dx, 1.0, i);
  }
  /* the next step's electrode values (after_loop hook): this step's solve is done */
  if ((int)threadIdx.x < a.nwave) {
    const WaveDesc &d = a.wave[threadIdx.x];
    const double t = (double)(a.step0 + (a.step_dev ? *a.step_dev : 0)) * a.dt;
    double u = d.f * t + d.ph;
    u = u - floor(u);
    double sn, co;
    isk_sincos2pi(u, &sn, &co);
    const_cast<double *>(a.t.tagval)[d.tag] = d.off + d.amp * sn;
  }
}

__global__ __launch_bounds__(FIELD1_BLOCK) void k_field1(Field1Args a) {
  field1_body(a, blockIdx.x);
}

/* chunks up to which the field kernel adds the chunk windows itself (above,
 * k_merge_tiles_n adds them per tile first): 12 chunks cost it about 1 us, the launch
 * 2.6 */
#define FIELD1_CHUNKS 32

static bool field1_direct(const IskSpecies &s) { return s.max_chunks <= FIELD1_CHUNKS; }

static void field1_prepare(iskra_ctx *c, double dt, const long long *step_dev, Field1Args *pa) {
  Field1Args &a = *pa;
  int grid;
  for (int s = 0; s < c->nspecies; ++s) {
    merge_prepare(c, s, 1, &a.m[s], &grid);
    a.m[s].tilewin = field1_direct(c->sp[s]) ? nullptr : c->sp[s].tilewin;
    a.r.cnt[s] = c->sp[s].cnt;
    a.r.qw[s] = c->sp[s].w0;
    a.r.q[s] = c->sp[s].q;
  }
  a.r.ns = c->nspecies;
  a.r.vol = c->vol;
  a.r.bg = c->bg;
  a.r.rho = c->rho;
  a.r.nn = isk_nodes(c);
  isk_tri_prepare(c, &a.t);
  a.E = c->E;
  a.dx = c->g.dx;
  a.nwave = 0;
  for (int k = 1; k <= ISK_MAX_TAGS; ++k)
    if (c->ps.wf_on[k] && c->ps.d_tag_val) {
      WaveDesc &w = a.wave[a.nwave++];
      w.tag = k;
      w.off = c->ps.wf_off[k];
      w.amp = c->ps.wf_amp[k];
      w.f = c->ps.wf_f[k];
      w.ph = c->ps.wf_ph[k];
    }
  a.dt = dt;
  a.step0 = c->step_count;
  a.step_dev = step_dev;
}

static int tiles_launch(iskra_ctx *c) {
  MergeTilesN t;
  for (int s = 0; s < c->nspecies; ++s) {
    t.partial[s] = c->sp[s].partial;
    t.tcb[s] = c->sp[s].tile_chunk_begin;
    t.hdr[s] = c->sp[s].hdr;
    t.tilewin[s] = c->sp[s].tilewin;
    t.WW[s] = c->g.dim == 2 ? isk_sp_window(c, s) * isk_sp_window(c, s) : isk_sp_window(c, s);
  }
  hipLaunchKernelGGL(k_merge_tiles_n, dim3(c->ntiles, c->nspecies), dim3(256), 0, c->stream, t);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* time loop of a 1-D grid with the direct solve: push, deposit, field, electrode
 * values */
int isk_step_tail_1d(iskra_ctx *c, double dt) {
  int rc;
  if ((rc = push_launch_all(c, dt))) return rc;
  hipEvent_t ev = nullptr;
  bool direct = true;
  for (int s = 0; s < c->nspecies; ++s) direct &= field1_direct(c->sp[s]);
  if (!direct) {
    if ((rc = isk_prof_begin(c, &ev))) return rc;
    if ((rc = tiles_launch(c))) return rc;
    if ((rc = isk_prof_end(c, ev, ISKRA_K_MERGE, 0))) return rc;
  }
  Field1Args a;
  field1_prepare(c, dt, nullptr, &a);
  if ((rc = isk_prof_begin(c, &ev))) return rc;
  hipLaunchKernelGGL(k_field1, dim3(2), dim3(FIELD1_BLOCK), 0, c->stream, a);
  ISK_CHECK_LAUNCH();
  for (int s = 0; s < c->nspecies; ++s) c->sp[s].deposited = 1;
  c->ps.last_iters = c->stats.last_iters = 1;
  c->ps.last_relres = c->stats.last_relres = 0.0;
  c->stats.poisson_solves++;
  c->stats.poisson_iters++;
  return isk_prof_end(c, ev, ISKRA_K_POISSON, 0);
}

/* time loop: push every species, then the tile windows of all species in
 * one launch and counts + rho in another */
int isk_push_deposit_all(iskra_ctx *c, double dt) {
  int rc;
  if ((rc = push_launch_all(c, dt))) return rc;
  hipEvent_t em = nullptr;
  if ((rc = isk_prof_begin(c, &em))) return rc;
  MergeRhoArgs a;
  int grid = 0;
  for (int s = 0; s < c->nspecies; ++s) {
    merge_prepare(c, s, 1, &a.m[s], &grid);
    a.m[s].tilewin = c->sp[s].tilewin;
    a.r.cnt[s] = c->sp[s].cnt;
    a.r.qw[s] = c->sp[s].w0;
    a.r.q[s] = c->sp[s].q;
  }
  a.r.ns = c->nspecies;
  a.r.vol = c->vol;
  a.r.bg = c->bg;
  a.r.rho = c->rho;
  a.r.nn = isk_nodes(c);
  isk_poisson_pack_desc(c, &a.pk);
  if (c->nspecies > 0 && (rc = tiles_launch(c))) return rc;
  grid = (a.r.nn + 255) / 256;
  if (c->g.dim == 2)
    hipLaunchKernelGGL(k_merge_rho<2>, dim3(grid), dim3(256), 0, c->stream, a);
  else
    hipLaunchKernelGGL(k_merge_rho<1>, dim3(grid), dim3(256), 0, c->stream, a);
  ISK_CHECK_LAUNCH();
  for (int s = 0; s < c->nspecies; ++s) c->sp[s].deposited = 1;
  return isk_prof_end(c, em, ISKRA_K_MERGE, 0);
}

/* ------------------------------------------------------------------------ */
/* gather only (grid_to_particle), for inspection                           */
/* ------------------------------------------------------------------------ */
template <int DIM>
__global__ void k_gather(const int32_t *cell, const float *ox, const float *oy,
                         const long long *hdr, const float *E, int nx,
                         float *out, long long cap) {
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= hdr[HDR_NP]) return;
  int cc = cell[p];
  float Ex = 0.f, Ey = 0.f;
  if (cc >= 0) {
    int i = cc & 0xFFFF, j = cc >> 16;
    float hx = ox[p];
    float ax = 1.0f - hx;
    if (DIM == 2) {
      float hy = oy[p];
      float ay = 1.0f - hy;
      float w00 = ax * ay, w10 = hx * ay, w01 = ax * hy, w11 = hx * hy;
      const float2 *E2 = reinterpret_cast<const float2 *>(E);
      int q = j * nx + i;
      float2 e00 = E2[q], e10 = E2[q + 1], e01 = E2[q + nx], e11 = E2[q + nx + 1];
      Ex = fmaf(w11, e11.x, fmaf(w01, e01.x, fmaf(w10, e10.x, w00 * e00.x)));
      Ey = fmaf(w11, e11.y, fmaf(w01, e01.y, fmaf(w10, e10.y, w00 * e00.y)));
    } else {
      Ex = fmaf(hx, E[i + 1], ax * E[i]);
    }
  }
  out[p] = Ex;
  out[cap + p] = Ey;
}

int isk_gather_species(iskra_ctx *c, int sid) {
  IskSpecies *s = &c->sp[sid];
  if (c->gather_cap < s->cap) {
    isk_free(c->gather_out);
    c->gather_out = nullptr;
    if (isk_alloc((void **)&c->gather_out, (size_t)s->cap * 2 * sizeof(float))) return ISKRA_E_HIP;
    c->gather_cap = s->cap;
  }
  int b = s->cur;
  int blocks = (int)((s->cap + 255) / 256);
  if (c->g.dim == 2)
    hipLaunchKernelGGL(k_gather<2>, dim3(blocks), dim3(256), 0, c->stream, s->cell[b],
                       s->ox[b], s->oy[b], s->hdr, c->E, c->g.nx, c->gather_out,
                       (long long)s->cap);
  else
    hipLaunchKernelGGL(k_gather<1>, dim3(blocks), dim3(256), 0, c->stream, s->cell[b],
                       s->ox[b], s->oy[b], s->hdr, c->E, c->g.nx, c->gather_out,
                       (long long)s->cap);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* ------------------------------------------------------------------------ */
/* batched launches over instances (one work-group = one work-group of one  */
/* instance's own launch, same device function)                             */
/* ------------------------------------------------------------------------ */
__global__ __launch_bounds__(PushShape<1>::block) void kb_push1(const PushArgs *A, const int *bstart,
                                                        int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  const PushArgs a = A[i]; /* in registers, not re-read after each store */
  push_body<1>(a, blockIdx.x - bstart[i]);
}

struct MergeTile1 {
  const long long *partial;
  const int *tcb;
  const long long *hdr;
  long long *tilewin;
  int WW;
};

__global__ __launch_bounds__(256) void kb_merge_tiles(const MergeTile1 *A, const int *bstart,
                                                      int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  const MergeTile1 a = A[i];
  merge_tile_body(a.partial, a.tcb, a.hdr, a.tilewin, a.WW, blockIdx.x - bstart[i]);
}

__global__ __launch_bounds__(FIELD1_BLOCK) void kb_field1(const Field1Args *A) {
  field1_body(A[blockIdx.x >> 1], blockIdx.x & 1);
}

__global__ __launch_bounds__(SORT_WAVE) void kb_sort_hist(const SortArgs *A, const int *bstart,
                                                           int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  sort_hist_body(A[i], blockIdx.x - bstart[i]);
}

__global__ __launch_bounds__(1024) void kb_sort_cols(const SortArgs *A, const int *bstart, int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  sort_cols_body<SORT_CR>(A[i], blockIdx.x - bstart[i], sort_active(A[i], A[i].hdr[HDR_NP]));
}

__global__ __launch_bounds__(1024) void kb_sort_bins(const SortArgs *A, const int *bstart, int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  if (A[i].one) sort_table_body(A[i]);
  else sort_bins_body(A[i], A[i].hdr[HDR_NP]);
}

__global__ __launch_bounds__(SORT_WAVE) void kb_sort_scatter(const SortArgs *A,
                                                              const int *bstart, int n) {
  const int i = isk_bfind(bstart, n, blockIdx.x);
  if (A[i].sc.id) sort_scatter_body<1, true>(A[i], blockIdx.x - bstart[i]);
  else sort_scatter_body<1, false>(A[i], blockIdx.x - bstart[i]);
}

/* entries (instance, species), species by species of an instance */
int isk_bbuild_push(iskra_ctx **cs, int n, double dt, int phase, IskBLaunch *L) {
  std::vector<PushArgs> A;
  std::vector<int> blocks;
  size_t shm = 0;
  for (int i = 0; i < n; ++i)
    for (int s = 0; s < cs[i]->nspecies; ++s) {
      int grid;
      size_t sh;
      A.emplace_back();
      push_prepare(cs[i], s, dt, 1, cs[i]->sp[s].cur ^ phase, &A.back(), &grid, &sh);
      blocks.push_back(grid);
      shm = std::max(shm, sh);
    }
  return isk_blaunch_upload(L, ISK_B_PUSH1, A.data(), sizeof(PushArgs), blocks, PushShape<1>::block,
                            shm);
}

int isk_bbuild_tiles(iskra_ctx **cs, int n, IskBLaunch *L) {
  std::vector<MergeTile1> A;
  std::vector<int> blocks;
  for (int i = 0; i < n; ++i)
    for (int s = 0; s < cs[i]->nspecies; ++s) {
      const IskSpecies &sp = cs[i]->sp[s];
      A.emplace_back();
      A.back().partial = sp.partial;
      A.back().tcb = sp.tile_chunk_begin;
      A.back().hdr = sp.hdr;
      A.back().tilewin = sp.tilewin;
      A.back().WW = isk_sp_window(cs[i], s);
      blocks.push_back(field1_direct(sp) ? 0 : cs[i]->ntiles);
    }
  return isk_blaunch_upload(L, ISK_B_TILES, A.data(), sizeof(MergeTile1), blocks, 256, 0);
}

int isk_bbuild_field(iskra_ctx **cs, int n, double dt, const long long *step_dev, int64_t advanced,
                     IskBLaunch *L) {
  std::vector<Field1Args> A(n);
  std::vector<int> two(n, 2);
  for (int i = 0; i < n; ++i) {
    if (cs[i]->ps.kind != ISKRA_POISSON_DIRECT) {
      isk_set_error("batch: instance %d does not use the direct 1-D Poisson solve", i);
      return ISKRA_E_UNSUPPORTED;
    }
    field1_prepare(cs[i], dt, step_dev, &A[i]);
    A[i].step0 -= advanced; /* *step_dev counts from the plan's origin */
  }
  return isk_blaunch_upload(L, ISK_B_FIELD, A.data(), sizeof(Field1Args), two, FIELD1_BLOCK, 0);
}

/* the launches of one tile-sort pass (with chunk table); instances whose
 * table one work-group scans have no work-group in the column launch, which is
 * left out when no instance has any */
int isk_bbuild_sort(iskra_ctx **cs, int n, int sid, const int *cur, IskBLaunch L[ISK_SORT_LAUNCHES]) {
  std::vector<SortArgs> A(n);
  std::vector<int> rows(n), cols(n), one(n, 1);
  size_t shm = 0;
  for (int i = 0; i < n; ++i) {
    int rc = sort_prepare(cs[i], sid, 0, 1, cur[i], &A[i]);
    if (rc) return rc;
    rows[i] = A[i].nrow;
    cols[i] = A[i].one ? 0 : A[i].ngrp;
    shm = std::max(shm, (size_t)A[i].nb1 * sizeof(int));
  }
  int rc;
  if ((rc = isk_blaunch_upload(&L[0], ISK_B_SORT_HIST, A.data(), sizeof(SortArgs), rows,
                               SORT_WAVE, shm)))
    return rc;
  if ((rc = isk_blaunch_upload(&L[1], ISK_B_SORT_COLS, A.data(), sizeof(SortArgs), cols, 1024, 0)))
    return rc;
  if ((rc = isk_blaunch_upload(&L[2], ISK_B_SORT_BINS, A.data(), sizeof(SortArgs), one, 1024, 0)))
    return rc;
  return isk_blaunch_upload(&L[3], ISK_B_SORT_SCATTER, A.data(), sizeof(SortArgs), rows,
                            SORT_WAVE, shm);
}

int isk_blaunch_particles(const IskBLaunch &L, hipStream_t st) {
  if (L.total <= 0) return ISKRA_OK;
  dim3 g((unsigned)L.total), b((unsigned)L.block);
  switch (L.kind) {
    case ISK_B_PUSH1:
      hipLaunchKernelGGL(kb_push1, g, b, L.shm, st, (const PushArgs *)L.args, L.bstart, L.n);
      break;
    case ISK_B_TILES:
      hipLaunchKernelGGL(kb_merge_tiles, g, b, 0, st, (const MergeTile1 *)L.args, L.bstart, L.n);
      break;
    case ISK_B_FIELD:
      hipLaunchKernelGGL(kb_field1, g, b, 0, st, (const Field1Args *)L.args);
      break;
    case ISK_B_SORT_HIST:
      hipLaunchKernelGGL(kb_sort_hist, g, b, L.shm, st, (const SortArgs *)L.args, L.bstart, L.n);
      break;
    case ISK_B_SORT_COLS:
      hipLaunchKernelGGL(kb_sort_cols, g, b, 0, st, (const SortArgs *)L.args, L.bstart, L.n);
      break;
    case ISK_B_SORT_BINS:
      hipLaunchKernelGGL(kb_sort_bins, g, b, 0, st, (const SortArgs *)L.args, L.bstart, L.n);
      break;
    case ISK_B_SORT_SCATTER:
      hipLaunchKernelGGL(kb_sort_scatter, g, b, L.shm, st, (const SortArgs *)L.args, L.bstart,
                         L.n);
      break;
    default:
      isk_set_error("batched launch: kind %d is not a particle kernel", L.kind);
      return ISKRA_E_ARG;
  }
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}
