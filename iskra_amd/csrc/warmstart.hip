/*
 * warmstart.hip -- learned warm start for the 2-D Poisson solve on gfx950.
 *
 * A convolutional encoder-decoder maps the right-hand side f = dx^2 rho/eps0
 * of a square grid with phi = 0 on all four walls to phi at the interior
 * nodes; its output seeds the iterative solver (PCG or multigrid), which then
 * iterates to the same FP64 residual as from any other start, so the network
 * can only change the iteration count, never the answer.  Trained with the
 * energy objective (the A-norm of the error left by the network plus one
 * damped Jacobi sweep), the same network preconditions every iteration of a
 * flexible CG on the FP64 residual (iskra_ws_solve).  There is no
 * counterpart in the reference (its Poisson solve is a dense direct solve,
 * FiniteDifferenceMethod/src/generalized_poisson.jl:201-203,372-378).
 *
 * Network (L levels, channels c_l = base * 2^min(l, 3), 3x3 convolutions, zero
 * padding, no biases, so the map is positively homogeneous and inputs are
 * normalised by their RMS):
 *   encoder  l = 0..L-1:  Ea_l = relu(conv(P_l)),  E_l = relu(conv(Ea_l)),
 *                         P_0 = input (8 channels, channel 0 = f / s),
 *                         P_l = avgpool2(E_{l-1})
 *   decoder  l = L-2..0:  U_l = upsample2(D_{l+1}) (D_{L-1} = E_{L-1}),
 *                         Da_l = relu(conv(U_l) + E_l),  D_l = relu(conv(Da_l))
 *   output   o = conv(D_0) channel 0;  phi = o * gain * s.
 * Tensors are NHWC bfloat16 (interior nodes padded to side S = nodes - 1);
 * convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16 with FP32
 * accumulation: forward and input-gradient kernels read 8 consecutive
 * channels per lane (16 bytes) for both operands and pool, mask and add what
 * follows on the way out, the weight-gradient
 * kernel stages segments of pixels in LDS and reduces over pixels in image order
 * (in chunks, which are then added in order).  The order of every sum follows from
 * a layer's shape and batch alone, so training is deterministic and a change of
 * tiles does not change it.
 * Gradients of activations are FP32 until they are masked and rounded for the next
 * layer; Adam keeps FP32 master weights.
 */
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "isk_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define WS_MAX_LEVELS 8
#define WS_IN_CH 8       /* input channels (channel 0 carries f) */
#define WS_OUT_CH 16     /* output channels computed (channel 0 is used) */
#define WS_PART_BYTES (64ll << 20)
#define EW_BLOCK 256
#define WS_MAX_SWEEPS 16
#ifndef WS_CONV_MIN_WG
#define WS_CONV_MIN_WG 512 /* work-groups a convolution should give: two a compute
                            * unit; with 256 or 1024 a forward pass's layers
                            * take 13 % longer */
#endif

__host__ __device__ inline uint16_t ws_f2bf(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ inline float ws_bf2f(uint16_t h) {
  return __builtin_bit_cast(float, (uint32_t)h << 16);
}

#define WRC(x)             \
  do {                     \
    int _rc = (x);         \
    if (_rc) return _rc;   \
  } while (0)

/* ------------------------------------------------------------------------ */
/* convolution: forward, input gradient, network output                       */

/* place of weight (co, k) in an operand's weights: the 16 x 32 block a wave loads
 * for one product is contiguous, 8 values a lane */
__host__ __device__ __forceinline__ long long ws_windex(int co, int k, int Kpad) {
  return (((long long)(co >> 4) * (Kpad >> 5) + (k >> 5)) * 64 + ((k >> 3) & 3) * 16 + (co & 15)) *
             8 + (k & 7);
}
/* length of the contraction, k = tap * Cin + ci, in whole blocks of 32 */
__host__ __device__ __forceinline__ int ws_kpad(int c) { return (9 * c + 31) & ~31; }

/* what becomes of the result v of a pixel (fp32): */
enum {
  WS_ACT,   /* Y = bf16(relu(v + skip)); with P also the 2x2 averages of Y */
  WS_PLANE, /* Yf = channel 0 */
  WS_MASK,  /* g = [act > 0] v: Gm = bf16(g); with Eg also Eg = g */
  WS_UP,    /* gradient of a 2x2 repetition: WS_MASK of the block's sum */
  WS_POOL   /* gradient of a 2x2 average: Gm = bf16([act > 0] (Eg + v / 4)) at its
             * four pixels */
};
struct ConvArgs {
  const uint16_t *X;     /* NHWC, Cin channels; up: of half the side, repeated 2x2 */
  const uint16_t *Wt;    /* ws_windex order, k = tap * Cin + ci, zero padded */
  const uint16_t *skip;  /* NHWC, Cout channels, or null */
  const uint16_t *act;   /* the activation whose gradient this is */
  uint16_t *Y, *P, *Gm;
  float *Yf, *Eg;
  int H, W, Cin, Cout, relu, mode, up;
};

__device__ __forceinline__ u16x8 ws_pack(const float v[8]) {
  u16x8 o;
#pragma unroll
  for (int r = 0; r < 8; ++r) o[r] = ws_f2bf(v[r]);
  return o;
}
/* v where the activation is positive, else 0 */
__device__ __forceinline__ void ws_gate(float v[8], const uint16_t *act) {
  const u16x8 y = *(const u16x8 *)act;
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = ws_bf2f(y[r]) > 0.f ? v[r] : 0.f;
}

/* RW rows x 16 pixels x 16 NJ channels of a wave (image n, first row h1, column w0
 * and channel c1), done with as a's mode says; `out`: this wave's 16 x (16 NJ + 4)
 * floats of LDS, for 16 bytes a lane of consecutive channels.  What follows a layer
 * in the network is done here: pooling, and in the backward pass the activation's
 * mask, the sum or the spread over 2x2 blocks and the skip connection.  As launches
 * of their own these took 36 us of a forward and 350 us of a backward pass on
 * 2^18 pixels. */
template <int NJ, int RW>
__device__ __forceinline__ void ws_conv_out(const ConvArgs &a, const f32x4 (&acc)[RW][NJ],
                                            float *out, int n, int h1, int w0, int c1) {
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  if (a.mode == WS_PLANE) {
#pragma unroll
    for (int g = 0; g < RW; ++g) {
      const int h = h1 + g, x = w0 + col;
      if (h < a.H && x < a.W && c1 + grp == 0)
        a.Yf[((long long)n * a.H + h) * a.W + x] = acc[g][0][0];
    }
    return;
  }
  constexpr int LD = 16 * NJ + 4, QV = 2 * NJ, NV8 = (16 * QV + 63) / 64;
  float up[NV8][8];
#pragma unroll
  for (int g = 0; g < RW; ++g) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) *(f32x4 *)(out + col * LD + j * 16 + grp * 4) = acc[g][j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int h = h1 + g;
#pragma unroll
    for (int i = 0; i < NV8; ++i) {
      const int q = (lane + 64 * i) / QV, x = w0 + q, c = (lane + 64 * i) % QV * 8;
      const bool in = q < 16 && h < a.H && x < a.W;
      const float *src = out + (q & 15) * LD + c;
      const f32x4 lo = *(const f32x4 *)src, hi = *(const f32x4 *)(src + 4);
      float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const long long o = (((long long)n * a.H + h) * a.W + x) * a.Cout + c1 + c;
      const long long o2 =
          (((long long)n * (a.H >> 1) + (h >> 1)) * (a.W >> 1) + (x >> 1)) * a.Cout + c1 + c;
      const bool first = in && !(q & 1); /* of a pair of columns */
      if (a.mode == WS_ACT) {
        if (a.skip && in) {
          const u16x8 sk = *(const u16x8 *)(a.skip + o);
#pragma unroll
          for (int r = 0; r < 8; ++r) v[r] += ws_bf2f(sk[r]);
        }
        if (a.relu) {
#pragma unroll
          for (int r = 0; r < 8; ++r) v[r] = fmaxf(v[r], 0.f);
        }
        const u16x8 y = ws_pack(v);
        if (in) *(u16x8 *)(a.Y + o) = y;
        if (a.P) {
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            const float e = ws_bf2f(y[r]), s = e + __shfl_xor(e, QV);
            if (g & 1) v[r] = 0.25f * (up[i][r] + s);
            else up[i][r] = s;
          }
          if ((g & 1) && first) *(u16x8 *)(a.P + o2) = ws_pack(v);
        }
      } else if (a.mode == WS_MASK) {
        if (!in) continue;
        ws_gate(v, a.act + o);
        *(u16x8 *)(a.Gm + o) = ws_pack(v);
        if (a.Eg) {
          *(f32x4 *)(a.Eg + o) = (f32x4){v[0], v[1], v[2], v[3]};
          *(f32x4 *)(a.Eg + o + 4) = (f32x4){v[4], v[5], v[6], v[7]};
        }
      } else if (a.mode == WS_UP) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const float s = v[r] + __shfl_xor(v[r], QV);
          if (g & 1) v[r] = up[i][r] + s;
          else up[i][r] = s;
        }
        if (!(g & 1) || !first) continue;
        ws_gate(v, a.act + o2);
        *(u16x8 *)(a.Gm + o2) = ws_pack(v);
      } else if (in) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const long long f =
              (((long long)n * 2 * a.H + 2 * h + (k >> 1)) * 2 * a.W + 2 * x + (k & 1)) * a.Cout +
              c1 + c;
          const f32x4 e0 = *(const f32x4 *)(a.Eg + f), e1 = *(const f32x4 *)(a.Eg + f + 4);
          float e[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) e[r] = (r < 4 ? e0[r & 3] : e1[r & 3]) + 0.25f * v[r];
          ws_gate(e, a.act + f);
          *(u16x8 *)(a.Gm + f) = ws_pack(e);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

/* Order of the sums.  Products are added 32 at a time (one matrix instruction), blocks
 * of 32 k's in one chain; the order of the blocks is part of a layer's result (a
 * different one flips roundings to bf16, and a training run ends in another
 * network: the 513^2 learned solve of 1000 snapshots then needs 148 iterations
 * or stalls).  It is fixed by a layer's shape and batch (ws_chunk_major) and does
 * not depend on the tile that computes it: either 32 channels at a time, their 9
 * taps in order (k_ws_conv), or the taps in order, each over all its channels, where
 * a block of 32 spans several taps if there are fewer channels (k_ws_conv_taps). */

/* 32 channels at a time; Cin a multiple of 32 KC, H and W of 16.  A work-group
 * computes a tile of 16 columns x RW WR rows x 16 NJ WC channels, WR = 4 / WC: its four
 * waves are WR groups of RW rows x WC groups of 16 NJ channels.  Per 32 KC input
 * channels the tile with its halo is staged (pixel stride 40 channels, so the 16
 * pixels a quarter-wave reads fall in distinct banks), the next ones' loads in
 * flight during the products.  An input row's three column shifts serve the three
 * taps above and below; a tap row's weights are replaced by the next 32 channels'
 * when the last pixel row has used them.
 *   Coarse planes have few tiles and many channels: there the waves share a tile of
 * 4 rows and several chunks go between two barriers.
 *   The layers of one 512 x 512 plane with 32 to 256 channels (4.8 or 9.7 GFLOP each),
 * on average: 15.8 us at the two finest levels (bound by their memory traffic), 12.3
 * and 10.2 at the next two (bound by the latency of few chunks); the same as with the
 * channels split over the waves, in another order of the sums, and 16 to 44 us with
 * each tap's weights loaded before its products. */
#define WS_LDS_PIX 40
template <int NJ, int RW, int WC, int KC>
__global__ __launch_bounds__(256) void k_ws_conv(ConvArgs a) {
  constexpr int WR = 4 / WC, TR = RW * WR, NPX = 18 * (TR + 2), NV = NPX * 4 * KC;
  constexpr int NR = (NV + 255) / 256, TILE = KC * NPX * WS_LDS_PIX;
  constexpr int OUT = 16 * (16 * NJ + 4); /* floats a wave */
  __shared__ __align__(16) uint16_t tile[TILE > 8 * OUT ? TILE : 8 * OUT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wr = wv / WC, wc = wv % WC;
  const int tw = a.W >> 4, th = a.H / TR;
  int t = blockIdx.x;
  const int w0 = t % tw * 16;
  t /= tw;
  const int h0 = t % th * TR, n = t / th;
  const int c1 = (blockIdx.y * WC + wc) * 16 * NJ;
  const int ncb = a.Cin >> 5, nkb = 9 * ncb;
  const int Hs = a.H >> a.up, Ws = a.W >> a.up;
  f32x4 acc[RW][NJ];
#pragma unroll
  for (int g = 0; g < RW; ++g)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[g][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  u32x4 st[NR], wt[3][3][NJ];
  auto fetch = [&](int cb) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int v = threadIdx.x + 256 * k, px = v / (4 * KC), c = cb * 32 + v % (4 * KC) * 8;
      const int hh = h0 + px / 18 - 1, ww = w0 + px % 18 - 1;
      st[k] = (u32x4){0u, 0u, 0u, 0u};
      if (px < NPX && hh >= 0 && hh < a.H && ww >= 0 && ww < a.W)
        st[k] = *(const u32x4 *)(a.X + ((long long)(n * Hs + (hh >> a.up)) * Ws + (ww >> a.up)) *
                                           a.Cin + c);
    }
  };
  const u32x4 *wp = (const u32x4 *)a.Wt + (long long)(c1 >> 4) * nkb * 64 + lane;
  auto weights = [&](int cb, int dy) {
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        wt[dy][dx][j] = wp[(j * nkb + (dy * 3 + dx) * ncb + cb) * 64];
  };
  fetch(0);
#pragma unroll
  for (int dy = 0; dy < 3; ++dy) weights(0, dy);
  for (int c0 = 0; c0 < ncb; c0 += KC) {
    if (c0) __syncthreads(); /* the previous chunks have been read */
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int v = threadIdx.x + 256 * k, px = v / (4 * KC), q = v % (4 * KC);
      if (v < NV) *(u32x4 *)(tile + (q / 4 * NPX + px) * WS_LDS_PIX + q % 4 * 8) = st[k];
    }
    __syncthreads();
    if (c0 + KC < ncb) fetch(c0 + KC);
    const uint16_t *bt = tile + (wr * RW * 18 + col) * WS_LDS_PIX + grp * 8;
#pragma unroll 1
    for (int kc = 0; kc < KC; ++kc, bt += NPX * WS_LDS_PIX) {
      const int cb = c0 + kc + 1;
#pragma unroll
      for (int r = 0; r < RW + 2; ++r) {
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const bf16x8 bv = *(const bf16x8 *)(bt + (r * 18 + dx) * WS_LDS_PIX);
#pragma unroll
          for (int dy = 0; dy < 3; ++dy) {
            if (r - dy < 0 || r - dy >= RW) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[r - dy][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(bf16x8, wt[dy][dx][j]), bv, acc[r - dy][j], 0, 0, 0);
          }
        }
        if (r >= RW - 1 && cb < ncb) weights(cb, r - (RW - 1));
      }
    }
  }
  __syncthreads();
  ws_conv_out<NJ, RW>(a, acc, (float *)tile + wv * OUT, n, h0 + wr * RW, w0, c1);
}

/* tap by tap; any Cin that is a multiple of 8.  Tiles and waves as in k_ws_conv, but
 * the tile holds all input channels (LDS), or, where those do not fit, a lane reads its
 * 8 channels from memory.  Bound by the latency of a block's operands, hence D blocks
 * in flight: 256 -> 128 channels on 4 planes of 32 x 32 take 27 us, 35 with one block
 * ahead; the first layer of a 512 x 512 plane (8 -> 32) 12 us. */
__host__ __device__ __forceinline__ int ws_taps_stride(int cin) { return cin + 8; }
template <int NJ, int RW, int WC, bool LDS>
__global__ __launch_bounds__(256) void k_ws_conv_taps(ConvArgs a) {
  constexpr int WR = 4 / WC, TR = RW * WR, NPX = 18 * (TR + 2), D = 8 / (RW * NJ);
  constexpr int OUT = 16 * (16 * NJ + 4);
  extern __shared__ __align__(16) uint16_t ws_mem[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wr = wv / WC, wc = wv % WC;
  const int tw = (a.W + 15) >> 4, th = (a.H + TR - 1) / TR;
  int t = blockIdx.x;
  const int w0 = t % tw * 16;
  t /= tw;
  const int h0 = t % th * TR, n = t / th;
  const int c1 = (blockIdx.y * WC + wc) * 16 * NJ;
  const int nkb = ws_kpad(a.Cin) >> 5, ld = ws_taps_stride(a.Cin);
  const int Hs = a.H >> a.up, Ws = a.W >> a.up;
  auto input = [&](int hh, int ww, int c) {
    u32x4 v = (u32x4){0u, 0u, 0u, 0u};
    if (hh >= 0 && hh < a.H && ww >= 0 && ww < a.W)
      v = *(const u32x4 *)(a.X + ((long long)(n * Hs + (hh >> a.up)) * Ws + (ww >> a.up)) *
                                     a.Cin + c);
    return v;
  };
  const u32x4 *wp = (const u32x4 *)a.Wt + (long long)(c1 >> 4) * nkb * 64 + lane;
  if (LDS) {
    const int cv = a.Cin >> 3;
#pragma unroll 8
    for (int v = threadIdx.x; v < NPX * cv; v += 256) {
      const int px = v / cv, c = (v - px * cv) * 8;
      *(u32x4 *)(ws_mem + px * ld + c) = input(h0 + px / 18 - 1, w0 + px % 18 - 1, c);
    }
    __syncthreads();
  }
  f32x4 acc[RW][NJ];
#pragma unroll
  for (int g = 0; g < RW; ++g)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[g][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int tap = grp * 8 / a.Cin, ci = grp * 8 - tap * a.Cin; /* of this lane's 8 k's */
  const int tap32 = 32 / a.Cin, ci32 = 32 - tap32 * a.Cin;
  auto operand = [&](u32x4 *bv) {
    const int dy = tap * 11 >> 5, dx = tap - 3 * dy; /* tap / 3 and its rest */
#pragma unroll
    for (int g = 0; g < RW; ++g) {
      const int row = wr * RW + g;
      bv[g] = (u32x4){0u, 0u, 0u, 0u};
      if (tap < 9) {
        if (LDS) bv[g] = *(const u32x4 *)(ws_mem + ((row + dy) * 18 + col + dx) * ld + ci);
        else bv[g] = input(h0 + row + dy - 1, w0 + col + dx - 1, ci);
      }
    }
    tap += tap32;
    ci += ci32;
    if (ci >= a.Cin) {
      ci -= a.Cin;
      ++tap;
    }
  };
  /* D blocks at a time, the next D's operands in flight during the products (those
   * past the end are read from the last block and not used) */
  u32x4 wt[D][NJ], bv[D][RW];
  auto blocks = [&](int kb, u32x4 (*w)[NJ], u32x4 (*x)[RW]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int k = min(kb + d, nkb - 1);
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[d][j] = wp[(j * nkb + k) * 64];
      operand(x[d]);
    }
  };
  blocks(0, wt, bv);
  for (int kb = 0; kb < nkb; kb += D) {
    u32x4 wn[D][NJ], bn[D][RW];
    blocks(kb + D, wn, bn);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (kb + d < nkb)
#pragma unroll
        for (int g = 0; g < RW; ++g)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[g][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, wt[d][j]), __builtin_bit_cast(bf16x8, bv[d][g]),
                acc[g][j], 0, 0, 0);
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) wt[d][j] = wn[d][j];
#pragma unroll
      for (int g = 0; g < RW; ++g) bv[d][g] = bn[d][g];
    }
  }
  __syncthreads();
  ws_conv_out<NJ, RW>(a, acc, (float *)ws_mem + wv * OUT, n, h0 + wr * RW, w0, c1);
}

/* ------------------------------------------------------------------------ */
/* weight gradient: part[chunk][co][tap*Cin+ci] = sum over the chunk's pixels */
/* of G[p][co] * X[p + tap][ci]                                               */

struct WgradArgs {
  const uint16_t *X;  /* NHWC Cin */
  const uint16_t *G;  /* NHWC Cout (masked output gradient) */
  float *part;
  int H, W, Cin, Cout;
  int up;             /* X has half the side, repeated 2x2 */
  int nseg;           /* segments of 64 pixels */
  int seg_per_chunk;
};

/* widest segment with its halo: 64 pixels of one row */
#define WSG_PX (66 * 3)

/* LDS stride of a pixel of C channels: an odd multiple of 8 banks, so the 8
 * pixels a half-wave reads fall in different banks */
__host__ __device__ constexpr int wsg_stride(int C) {
  return (C / 16) % 2 ? C : C + 16;
}
template <int NC, int CW, int IW>
constexpr size_t wsg_lds() {
  return ((size_t)WSG_PX * wsg_stride(16 * IW) + 64 * wsg_stride(16 * NC * CW)) * 2 * 2;
}

/* the 4 pixels x 16 channels that 16 lanes address (8 bytes each: lane s the
 * pixel s / 4, channels 4 (s % 4) ..) transposed: lane i gets channel i of the
 * 4 pixels */
__device__ __forceinline__ uint2 wsg_tr(const uint16_t *p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) s16x4 *)p));
}
__device__ __forceinline__ bf16x8 wsg_pair(uint2 lo, uint2 hi) {
  return __builtin_bit_cast(bf16x8, (u32x4){lo.x, lo.y, hi.x, hi.y});
}

/* Contraction over pixels on the matrix cores, 32 consecutive ones at a time in
 * image order.  A chunk of seg_per_chunk segments of 64 pixels is one chain of
 * sums, and the chunks are added in order (k_ws_reduce): which pixels make a chunk
 * is part of the result, as the order of a convolution's sums is, and follows
 * from the layer alone.  A work-group takes a chunk for a block of 16 NC CW output
 * x 16 IW input channels; its waves are CW x IW groups of channels x TW groups of
 * taps.  X with its halo and G of a segment lie in LDS once (two buffers: one
 * barrier a segment; the loads of the segment after next are in flight), and the
 * operands, whose 8 values a lane are pixels of one channel, are read with the
 * transposing LDS read.
 *   On 2^18 pixels x 32 channels, or the same work deeper in the network, 18 us on average,
 * bound by the latency of a segment (8 in a row a chunk): 45 with a copy of the
 * segment for every tap and 16-bit LDS reads; 13 with tiles of 16 x 8 pixels, whose rows
 * serve three taps, but those are other chains of sums. */
template <int NC, int CW, int IW, int TW>
__global__ __launch_bounds__(256) void k_ws_wgrad(WgradArgs a) {
  static_assert(CW * IW * TW == 4, "four waves");
  constexpr int XC = 16 * IW, GC = 16 * NC * CW, XS = wsg_stride(XC), GS = wsg_stride(GC);
  constexpr int XV = XC / 8, GV = GC / 8; /* 16-byte vectors a pixel */
  constexpr int XN = (WSG_PX * XV + 255) / 256, GN = (64 * GV + 255) / 256;
  constexpr int TN = (9 + TW - 1) / TW; /* taps of a wave */
  constexpr int BUF = WSG_PX * XS + 64 * GS;
  extern __shared__ __attribute__((aligned(16))) uint16_t ws_mem[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int tg = wv / (CW * IW), cw = wv / IW % CW, iw = wv % IW;
  const int tap0 = tg * TN;
  const int co0 = blockIdx.y * GC, ci0 = blockIdx.z * XC;
  const int s0 = blockIdx.x * a.seg_per_chunk, s1 = min(a.nseg, s0 + a.seg_per_chunk);
  /* a segment is pw - 2 columns of one or more rows (sides are powers of two) */
  const int lw = min(6, 31 - __builtin_clz(a.W)), pw = (1 << lw) + 2, ph = (64 >> lw) + 2;
  const int img = a.H * a.W >> 6; /* segments an image */
  int xh[XN], xw[XN]; /* this thread's pixels of the halo, relative to the segment */
#pragma unroll
  for (int k = 0; k < XN; ++k) {
    const int px = (threadIdx.x + 256 * k) / XV;
    xh[k] = px < pw * ph ? px / pw - 1 : -4;
    xw[k] = px % pw - 1;
  }
  u32x4 rx[XN], rg[GN];
  auto fetch = [&](int s) {
    const int n = s / img, r = (s - n * img) * 64, h0 = r / a.W, w0 = r - h0 * a.W;
#pragma unroll
    for (int k = 0; k < XN; ++k) {
      const int c = ci0 + (threadIdx.x + 256 * k) % XV * 8, hh = h0 + xh[k], ww = w0 + xw[k];
      rx[k] = (u32x4){0u, 0u, 0u, 0u};
      if (xh[k] > -4 && c < a.Cin && hh >= 0 && hh < a.H && ww >= 0 && ww < a.W)
        rx[k] = *(const u32x4 *)(a.X + ((long long)(n * (a.H >> a.up) + (hh >> a.up)) *
                                            (a.W >> a.up) + (ww >> a.up)) * a.Cin + c);
    }
#pragma unroll
    for (int k = 0; k < GN; ++k) {
      const int v = threadIdx.x + 256 * k, px = v / GV, c = co0 + v % GV * 8;
      rg[k] = (u32x4){0u, 0u, 0u, 0u};
      if (px < 64 && c < a.Cout) rg[k] = *(const u32x4 *)(a.G + ((long long)s * 64 + px) * a.Cout + c);
    }
  };
  auto stage = [&](uint16_t *buf) {
#pragma unroll
    for (int k = 0; k < XN; ++k) {
      const int v = threadIdx.x + 256 * k;
      if (v < WSG_PX * XV) *(u32x4 *)(buf + v / XV * XS + v % XV * 8) = rx[k];
    }
#pragma unroll
    for (int k = 0; k < GN; ++k) {
      const int v = threadIdx.x + 256 * k;
      if (v < 64 * GV) *(u32x4 *)(buf + WSG_PX * XS + v / GV * GS + v % GV * 8) = rg[k];
    }
  };
  f32x4 acc[NC][TN];
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[j][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  /* pixels 8 (lane / 16) .. + 3 of 32 (the next four are 4 further), this lane's of them */
  const int px = 8 * (lane >> 4) + ((lane & 15) >> 2), ch = (lane & 3) * 4;
  int bx[2];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc) {
    const int p = 32 * kc + px;
    bx[kc] = ((p >> lw) * pw + (p & ((1 << lw) - 1))) * XS + iw * 16 + ch;
  }
  const int bg = WSG_PX * XS + px * GS + cw * NC * 16 + ch;
  int xt[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) { /* (a tap past the ninth repeats it and is not stored) */
    const int tap = min(tap0 + t, 8);
    xt[t] = (tap / 3 * pw + tap % 3) * XS;
  }
  fetch(s0);
  stage(ws_mem);
  if (s0 + 1 < s1) fetch(s0 + 1);
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const uint16_t *buf = ws_mem + ((s - s0) & 1) * BUF;
    if (s + 1 < s1) {
      stage(ws_mem + ((s - s0 + 1) & 1) * BUF);
      if (s + 2 < s1) fetch(s + 2);
    }
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      bf16x8 A[NC];
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const uint16_t *g = buf + bg + 32 * kc * GS + j * 16;
        A[j] = wsg_pair(wsg_tr(g), wsg_tr(g + 4 * GS));
      }
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const uint16_t *x = buf + bx[kc] + xt[t];
        const bf16x8 B = wsg_pair(wsg_tr(x), wsg_tr(x + 4 * XS));
#pragma unroll
        for (int j = 0; j < NC; ++j)
          acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j], B, acc[j][t], 0, 0, 0);
      }
    }
    __syncthreads(); /* this buffer has been read, the other is written */
  }
  const long long K = 9ll * a.Cin;
  float *out = a.part + (long long)blockIdx.x * a.Cout * K;
  const int ci = ci0 + iw * 16 + (lane & 15);
  if (ci >= a.Cin) return;
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int co = co0 + (cw * NC + j) * 16 + (lane >> 4) * 4;
    if (co >= a.Cout) continue;
#pragma unroll
    for (int t = 0; t < TN; ++t)
      if (tap0 + t < 9)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(co + r) * K + (tap0 + t) * a.Cin + ci] = acc[j][t][r];
  }
}

/* grads[i] = sum_c part[c][i], the chunks in order: a work-group takes 64
 * neighbouring elements, WSR_ROWS rows of 16 lanes bring WSR_DEPTH WSR_ROWS chunks
 * of them to LDS, the next ones in flight, and one wave adds those up: 7 us on
 * average (one thread an element walked 512 chunks of a 32 -> 32 layer in 56 us). */
#define WSR_ROWS 32
#define WSR_DEPTH 4
__global__ __launch_bounds__(16 * WSR_ROWS) void k_ws_reduce(const float *__restrict__ part,
                                                            float *__restrict__ out, long long n,
                                                            int nchunk) {
  __shared__ float4 row[WSR_DEPTH * WSR_ROWS][16];
  const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
  const long long i = ((long long)blockIdx.x * 16 + x) * 4, o = (long long)blockIdx.x * 64;
  float4 v[WSR_DEPTH];
  auto fetch = [&](int c0) {
#pragma unroll
    for (int u = 0; u < WSR_DEPTH; ++u) {
      const int c = c0 + u * WSR_ROWS + y;
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c < nchunk && i < n) v[u] = *(const float4 *)(part + (long long)c * n + i);
    }
  };
  float s = 0.f;
  fetch(0);
  for (int c0 = 0; c0 < nchunk; c0 += WSR_DEPTH * WSR_ROWS) {
    if (c0) __syncthreads(); /* the rows before have been added */
#pragma unroll
    for (int u = 0; u < WSR_DEPTH; ++u) row[u * WSR_ROWS + y][x] = v[u];
    __syncthreads();
    if (c0 + WSR_DEPTH * WSR_ROWS < nchunk) fetch(c0 + WSR_DEPTH * WSR_ROWS);
    if (threadIdx.x < 64) {
      const int m = min(WSR_DEPTH * WSR_ROWS, nchunk - c0);
      const float *col = (const float *)row + threadIdx.x;
#pragma unroll 8
      for (int c = 0; c < m; ++c) s += col[64 * c];
    }
  }
  if (threadIdx.x < 64 && o + threadIdx.x < n) out[o + threadIdx.x] = s;
}

/* ------------------------------------------------------------------------ */
/* elementwise kernels (grid-stride, one element per thread)                  */

__global__ void k_ws_fill(float *p, long long n, float v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

/* loss over interior pixels (h, w < S-1): sum (o - t)^2 per block -> part;
 * Gout[p][0] = bf16(2 (o - t) * inv_count), other output channels 0 */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_loss(const float *o, const float *t,
                                                      uint16_t *Gout, double *part, int S,
                                                      long long npix, float inv_count) {
  __shared__ double red[EW_BLOCK];
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x) {
    const int pix = (int)(i % ((long long)S * S));
    const int h = pix / S, w = pix - (pix / S) * S;
    float d = 0.f;
    if (h < S - 1 && w < S - 1) d = o[i] - t[i];
    acc += (double)d * (double)d;
    if (Gout) {
      uint16_t *g = Gout + i * WS_OUT_CH;
      g[0] = ws_f2bf(2.f * d * inv_count);
      for (int c = 1; c < WS_OUT_CH; ++c) g[c] = 0;
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_ws_adam(float *p, const float *g, float *m, float *v, long long n, float lr,
                          float b1, float b2, float eps, float c1, float c2) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  }
}

/* bf16 weights of one layer: Wt of (co, tap, ci) (forward) and Wtt of (ci, tap, co)
 * (input gradient: taps mirrored, in/out channels swapped), zero in the padding */
__global__ void k_ws_wprep(const float *p, uint16_t *Wt, uint16_t *Wtt, int Cin, int Cout) {
  const int kp = ws_kpad(Cin), kpt = ws_kpad(Cout);
  const long long n1 = (long long)Cout * kp, n2 = Wtt ? (long long)Cin * kpt : 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n1 + n2;
       i += (long long)gridDim.x * blockDim.x) {
    float v = 0.f;
    if (i < n1) {
      const int co = (int)(i / kp), k = (int)(i - (long long)co * kp);
      if (k < 9 * Cin) v = p[(long long)co * 9 * Cin + k];
      Wt[ws_windex(co, k, kp)] = ws_f2bf(v);
    } else {
      const long long j = i - n1;
      const int ci = (int)(j / kpt), k = (int)(j - (long long)ci * kpt);
      const int tp = k / Cout, co = k % Cout;
      if (tp < 9) v = p[((long long)co * 9 + 8 - tp) * Cin + ci];
      Wtt[ws_windex(ci, k, kpt)] = ws_f2bf(v);
    }
  }
}

/* training batch: A0[b][pix][0..7] = (ds_in[idx[b]][pix], 0, ...);
 * tgt[b][pix] = ds_out[idx[b]][pix] * inv_gain */
__global__ void k_ws_batch(const uint16_t *ds_in, const float *ds_out, const long long *idx,
                           uint16_t *A0, float *tgt, int S2, int nb, float inv_gain) {
  const long long n = (long long)nb * S2;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int b = (int)(i / S2);
    const int pix = (int)(i - (long long)b * S2);
    const long long s = idx[b];
    u16x8 v = (u16x8){0, 0, 0, 0, 0, 0, 0, 0};
    v[0] = ds_in[s * S2 + pix];
    *(u16x8 *)(A0 + i * WS_IN_CH) = v;
    if (tgt) tgt[i] = ds_out ? ds_out[s * S2 + pix] * inv_gain : 0.f;
  }
}

/* host-supplied (already normalised) inputs: A0[i][0] = bf16(x[i]) */
__global__ void k_ws_input(const float *x, uint16_t *A0, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    u16x8 v = (u16x8){0, 0, 0, 0, 0, 0, 0, 0};
    v[0] = ws_f2bf(x[i]);
    *(u16x8 *)(A0 + i * WS_IN_CH) = v;
  }
}

/* right-hand side of the context's rho: sum of f^2 over interior nodes per
 * block, f = rho * fscale */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_rhs_sumsq(const double *rho, int nx,
                                                           double fscale, double *part) {
  __shared__ double red[EW_BLOCK];
  const int S = nx - 1;
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
       i < (long long)(S - 1) * (S - 1); i += (long long)gridDim.x * blockDim.x) {
    const int h = (int)(i / (S - 1)), w = (int)(i - (long long)h * (S - 1));
    const double f = rho[(long long)(h + 1) * nx + (w + 1)] * fscale;
    acc += f * f;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

/* scal[0] = s = sqrt(mean f^2) (1 if f == 0), scal[1] = 1/s */
/* sum of part[stride b + v] over b < nb, one work-group of EW_BLOCK threads
 * (thread t takes b = t, t + EW_BLOCK, ... in order, then a fixed tree):
 * deterministic; valid in thread 0 */
__device__ __forceinline__ double ws_group_sum(const double *part, int nb, int stride, int v,
                                               double *red) {
  double t = 0.0;
  for (int b = threadIdx.x; b < nb; b += EW_BLOCK) t += part[(long long)stride * b + v];
  red[threadIdx.x] = t;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

/* launched with one work-group of EW_BLOCK threads */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_rhs_scale(const double *part, int nb,
                                                           long long count, double *scal) {
  __shared__ double red[EW_BLOCK];
  const double t = ws_group_sum(part, nb, 1, 0, red);
  if (threadIdx.x == 0) {
    double s = sqrt(t / (double)count);
    if (!(s > 0.0)) s = 1.0;
    scal[0] = s;
    scal[1] = 1.0 / s;
  }
}

/* normalised input (and, for capture, the normalised target phi / s) */
__global__ void k_ws_rhs_store(const double *rho, const double *phi, int nx, double fscale,
                               const double *scal, uint16_t *in_plane, uint16_t *A0,
                               float *out_plane) {
  const int S = nx - 1;
  const double inv = scal[1];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < (long long)S * S;
       i += (long long)gridDim.x * blockDim.x) {
    const int h = (int)(i / S), w = (int)(i - (long long)h * S);
    const bool in = h < S - 1 && w < S - 1;
    const long long node = (long long)(h + 1) * nx + (w + 1);
    const float x = in ? (float)(rho[node] * fscale * inv) : 0.f;
    if (in_plane) in_plane[i] = ws_f2bf(x);
    if (A0) {
      u16x8 v = (u16x8){0, 0, 0, 0, 0, 0, 0, 0};
      v[0] = ws_f2bf(x);
      *(u16x8 *)(A0 + i * WS_IN_CH) = v;
    }
    if (out_plane) out_plane[i] = in ? (float)(phi[node] * inv) : 0.f;
  }
}

/* phi (interior nodes) = o * gain * s */
__global__ void k_ws_phi_out(const float *o, double *phi, int nx, double gain,
                             const double *scal) {
  const int S = nx - 1;
  const double sc = gain * scal[0];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
       i < (long long)(S - 1) * (S - 1); i += (long long)gridDim.x * blockDim.x) {
    const int h = (int)(i / (S - 1)), w = (int)(i - (long long)h * (S - 1));
    phi[(long long)(h + 1) * nx + (w + 1)] = (double)o[(long long)h * S + w] * sc;
  }
}

/* sum of squares of a float range, per block */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_sumsq(const float *x, long long n,
                                                       double *part) {
  __shared__ double red[EW_BLOCK];
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    acc += (double)x[i] * (double)x[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

/* ------------------------------------------------------------------------ */
/* energy objective: the network (times gain) followed by k damped Jacobi     */
/* sweeps, scored in the A-norm.  Plane pixels (h, w) < S-1 are the interior  */
/* nodes; A v = 4 v - (4 neighbours), neighbours outside the interior are 0.  */

__device__ __forceinline__ float eg_nb(const float *v, long long i, int h, int w, int S) {
  float s = 0.f;
  if (h > 0) s += v[i - S];
  if (h < S - 2) s += v[i + S];
  if (w > 0) s += v[i - 1];
  if (w < S - 2) s += v[i + 1];
  return s;
}

/* one sweep dst = sc src + om4 (x - A sc src), x = the network input (A0
 * channel 0).  last: dst -= gain t (the error e) and part[nb + b] = the
 * block's sum of (gain t).A(gain t) */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_eg_sweep(const float *src, float *dst,
                                                          const uint16_t *A0, const float *t,
                                                          int S, long long npix, float sc,
                                                          float om4, float gain, int last,
                                                          double *part, int nb) {
  __shared__ double red[EW_BLOCK];
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x) {
    const int pix = (int)(i % ((long long)S * S));
    const int h = pix / S, w = pix - (pix / S) * S;
    float v = 0.f;
    if (h < S - 1 && w < S - 1) {
      const float y = sc * src[i];
      const float ay = 4.f * y - sc * eg_nb(src, i, h, w, S);
      const float x = ws_bf2f(A0[i * WS_IN_CH]);
      v = y + om4 * (x - ay);
      if (last) {
        const float tv = gain * t[i];
        v -= tv;
        acc += (double)tv * (double)(4.f * tv - gain * eg_nb(t, i, h, w, S));
      }
    }
    dst[i] = v;
  }
  if (!last) return;
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[nb + blockIdx.x] = red[0];
}

/* ae = A e; part[b] = sum e.Ae */
__global__ __launch_bounds__(EW_BLOCK) void k_ws_eg_ae(const float *e, float *ae, int S,
                                                       long long npix, double *part) {
  __shared__ double red[EW_BLOCK];
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x) {
    const int pix = (int)(i % ((long long)S * S));
    const int h = pix / S, w = pix - (pix / S) * S;
    float a = 0.f;
    if (h < S - 1 && w < S - 1) {
      a = 4.f * e[i] - eg_nb(e, i, h, w, S);
      acc += (double)e[i] * (double)a;
    }
    ae[i] = a;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = EW_BLOCK / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

/* back through one sweep: h' = coef (h - om4 A h); Gout (non-null, the last
 * sweep) receives bf16(h') in channel 0 and 0 in the other channels, else
 * dst = h' */
__global__ void k_ws_eg_back(const float *hsrc, float *dst, uint16_t *Gout, int S,
                             long long npix, float om4, float coef) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x) {
    const int pix = (int)(i % ((long long)S * S));
    const int h = pix / S, w = pix - (pix / S) * S;
    float g = 0.f;
    if (h < S - 1 && w < S - 1) {
      const float a = hsrc[i];
      g = coef * (a - om4 * (4.f * a - eg_nb(hsrc, i, h, w, S)));
    }
    if (Gout) {
      uint16_t *gp = Gout + i * WS_OUT_CH;
      gp[0] = ws_f2bf(g);
      for (int c = 1; c < WS_OUT_CH; ++c) gp[c] = 0;
    } else {
      dst[i] = g;
    }
  }
}

/* dst = src - om4 A src on the interior (0 outside): one factor of the
 * pre-smoothing polynomial P = (I - om4 A)^k that maps a training pair (x, t)
 * to the pair the network meets after k pre-sweeps, (P x, P t) */
__global__ void k_ws_eg_poly(const float *src, float *dst, int S, long long npix, float om4) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x) {
    const int pix = (int)(i % ((long long)S * S));
    const int h = pix / S, w = pix - (pix / S) * S;
    float v = 0.f;
    if (h < S - 1 && w < S - 1) {
      const float a = src[i];
      v = a - om4 * (4.f * a - eg_nb(src, i, h, w, S));
    }
    dst[i] = v;
  }
}

/* plane <-> channel 0 of the network input */
__global__ void k_ws_a0_get(const uint16_t *A0, float *x, long long npix) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < npix;
       i += (long long)gridDim.x * blockDim.x)
    x[i] = ws_bf2f(A0[i * WS_IN_CH]);
}

/* ------------------------------------------------------------------------ */
/* the network inside the iteration: flexible CG on the interior nodes of     */
/* the network's grid, A x = 4 x - (4 neighbours) = f = dx^2 rho / eps0, walls */
/* 0 (the reference system with its Dirichlet columns eliminated and the rows  */
/* multiplied by -dx^2).  Node k = j nx + i; vectors keep 0 on the walls.      */

#define LS_BLOCK 256
enum { LS_FF = 0, LS_RR = 1, LS_ZQ = 2, LS_PQ = 3, LS_RP = 4, LS_NS = 8 };

__device__ __forceinline__ double ls_Ax(const double *x, int nx, long long k) {
  return 4.0 * x[k] - x[k - 1] - x[k + 1] - x[k - nx] - x[k + nx];
}

/* interior node of flat index q < (nx-2)^2 */
__device__ __forceinline__ long long ls_node(long long q, int nx) {
  const int m = nx - 2;
  const long long j = q / m;
  return (j + 1) * nx + (q - j * m) + 1;
}

/* block sum, valid in thread 0 (wave shuffles, then the waves in order) */
__device__ __forceinline__ double ls_block_sum(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int q = 0; q < LS_BLOCK / 64; ++q) s += red[q];
  return s;
}

/* x = phi (or 0), r = f - A x; partials of f.f and r.r */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_init(const double *rho, const double *phi,
                                                      int nx, double fscale, double *x,
                                                      double *r, double *part) {
  __shared__ double red[LS_BLOCK / 64];
  const long long n = (long long)(nx - 2) * (nx - 2);
  double ff = 0.0, rr = 0.0;
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    const double f = rho[k] * fscale;
    const double xv = phi ? phi[k] : 0.0;
    const double rv = phi ? f - ls_Ax(phi, nx, k) : f;
    x[k] = xv;
    r[k] = rv;
    ff += f * f;
    rr += rv * rv;
  }
  ff = ls_block_sum(ff, red);
  rr = ls_block_sum(rr, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = ff;
    part[2 * blockIdx.x + 1] = rr;
  }
}

/* out[v] = sum over blocks of part[nv b + v], v < nv (one work-group of
 * EW_BLOCK threads, fixed order) */
__global__ __launch_bounds__(EW_BLOCK) void k_ls_reduce(const double *part, int nb, int nv,
                                                        double *out) {
  __shared__ double red[EW_BLOCK];
  for (int v = 0; v < nv; ++v) {
    const double t = ws_group_sum(part, nb, nv, v, red);
    if (threadIdx.x == 0) out[v] = t;
  }
}

/* zs = z + om4 (r - A z): one damped Jacobi sweep (z null: from z = 0) */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_smooth(const double *r, const double *z,
                                                        double *zs, int nx, double om4) {
  const long long n = (long long)(nx - 2) * (nx - 2);
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    zs[k] = z ? z[k] + om4 * (r[k] - ls_Ax(z, nx, k)) : om4 * r[k];
  }
}

/* rp = r - A z: what the pre-sweeps left for the network */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_resid(const double *r, const double *z,
                                                       double *rp, int nx) {
  const long long n = (long long)(nx - 2) * (nx - 2);
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    rp[k] = r[k] - ls_Ax(z, nx, k);
  }
}

/* z += c: the network's correction added to the pre-sweeps' iterate */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_add(double *z, const double *c, int nx) {
  const long long n = (long long)(nx - 2) * (nx - 2);
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    z[k] += c[k];
  }
}

/* partials of a.b */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_dot(const double *a, const double *b, int nx,
                                                     double *part) {
  __shared__ double red[LS_BLOCK / 64];
  const long long n = (long long)(nx - 2) * (nx - 2);
  double s = 0.0;
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    s += a[k] * b[k];
  }
  s = ls_block_sum(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

/* p = z + beta p_prev, beta = -(z.q_prev)/(p_prev.q_prev) (none in the first
 * iteration): the new direction A-orthogonal to the previous one */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_dir(const double *z, const double *pprev,
                                                     double *p, int nx, const double *s,
                                                     int first) {
  const long long n = (long long)(nx - 2) * (nx - 2);
  const double beta = first ? 0.0 : -s[LS_ZQ] / s[LS_PQ];
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    p[k] = first ? z[k] : z[k] + beta * pprev[k];
  }
}

/* q = A p; partials of p.q and r.p */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_Ap(const double *p, const double *r, double *qv,
                                                    int nx, double *part) {
  __shared__ double red[LS_BLOCK / 64];
  const long long n = (long long)(nx - 2) * (nx - 2);
  double pq = 0.0, rp = 0.0;
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    const double a = ls_Ax(p, nx, k);
    qv[k] = a;
    pq += p[k] * a;
    rp += r[k] * p[k];
  }
  pq = ls_block_sum(pq, red);
  rp = ls_block_sum(rp, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = pq;
    part[2 * blockIdx.x + 1] = rp;
  }
}

/* alpha = (r.p)/(p.q); x += alpha p, r -= alpha q; partials of r.r */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_xr(double *x, double *r, const double *p,
                                                    const double *qv, int nx, const double *s,
                                                    double *part) {
  __shared__ double red[LS_BLOCK / 64];
  const long long n = (long long)(nx - 2) * (nx - 2);
  const double alpha = s[LS_RP] / s[LS_PQ];
  double rr = 0.0;
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    x[k] = __builtin_fma(alpha, p[k], x[k]);
    const double rv = __builtin_fma(-alpha, qv[k], r[k]);
    r[k] = rv;
    rr += rv * rv;
  }
  rr = ls_block_sum(rr, red);
  if (threadIdx.x == 0) part[blockIdx.x] = rr;
}

/* phi (interior nodes) = x */
__global__ __launch_bounds__(LS_BLOCK) void k_ls_out(const double *x, double *phi, int nx) {
  const long long n = (long long)(nx - 2) * (nx - 2);
  for (long long q = blockIdx.x * (long long)LS_BLOCK + threadIdx.x; q < n;
       q += (long long)gridDim.x * LS_BLOCK) {
    const long long k = ls_node(q, nx);
    phi[k] = x[k];
  }
}

/* a training pair from an FCG iterate: input r / s, target (phi - x) / s at
 * the interior nodes (s = scal[0], the RMS of r), plane layout of capture */
__global__ void k_ws_pair_store(const double *r, const double *phi, const double *x, int nx,
                                const double *scal, uint16_t *in_plane, float *out_plane) {
  const int S = nx - 1;
  const double inv = scal[1];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < (long long)S * S;
       i += (long long)gridDim.x * blockDim.x) {
    const int h = (int)(i / S), w = (int)(i - (long long)h * S);
    const bool in = h < S - 1 && w < S - 1;
    const long long node = (long long)(h + 1) * nx + (w + 1);
    in_plane[i] = ws_f2bf(in ? (float)(r[node] * inv) : 0.f);
    out_plane[i] = in ? (float)((phi[node] - x[node]) * inv) : 0.f;
  }
}

/* ------------------------------------------------------------------------ */
/* host side                                                                  */

struct WsConv {
  int cin, cout, level, relu;
  long long woff;  /* offset in the parameter vector ([co][tap][ci]) */
  uint16_t *wt = nullptr, *wtt = nullptr;
};

struct WsTensor {
  int level = 0, C = 0;
  uint16_t *a = nullptr; /* bf16 activations */
  float *g = nullptr;    /* fp32 gradient */
};

struct iskra_ws {
  iskra_ctx *ctx = nullptr;
  int L = 0, base = 0, S = 0, maxb = 0;
  std::vector<WsConv> conv;
  long long nparam = 0;
  float *params = nullptr, *grads = nullptr, *m = nullptr, *v = nullptr;
  long long adam_t = 0;
  double gain = 1.0;
  WsTensor A0, Ea[WS_MAX_LEVELS], E[WS_MAX_LEVELS], P[WS_MAX_LEVELS],
      Da[WS_MAX_LEVELS], D[WS_MAX_LEVELS];
  float *out = nullptr, *tgt = nullptr;
  uint16_t *gout = nullptr, *gm[2] = {nullptr, nullptr};
  long long gm_elems = 0;
  float *part = nullptr;
  double *dpart = nullptr, *scal = nullptr;
  int dpart_n = 0;
  long long *idx = nullptr;
  float *xin = nullptr;  /* host-input staging */
  /* dataset */
  uint16_t *ds_in = nullptr;
  float *ds_out = nullptr;
  long long ds_cap = 0, ds_n = 0;
  /* training objective (ISKRA_WS_*), its Jacobi weight / 4 and planes */
  int obj = ISKRA_WS_PHI_MSE;
  double om4 = 0.0;
  int sweeps = 1;
  float *eg_e = nullptr, *eg_ae = nullptr;
  /* the network-preconditioned solve (node grid, FP64; walls stay 0) */
  double *lx = nullptr, *lr = nullptr, *lz = nullptr, *lzs = nullptr, *lp[2] = {nullptr, nullptr},
         *lq[2] = {nullptr, nullptr}, *lpart = nullptr, *ls = nullptr, *lpre[2] = {nullptr, nullptr},
         *lrp = nullptr;
};

static int ws_side(const iskra_ws *w, int l) { return w->S >> l; }
static long long ws_npix(const iskra_ws *w, int l, int b) {
  return (long long)b * ws_side(w, l) * ws_side(w, l);
}
static unsigned ws_grid(long long n) {
  long long b = (n + EW_BLOCK - 1) / EW_BLOCK;
  return (unsigned)std::max(1ll, std::min(b, 8192ll));
}

static int ws_tensor(iskra_ws *w, WsTensor *t, int level, int C, bool grad) {
  t->level = level;
  t->C = C;
  const long long n = ws_npix(w, level, w->maxb) * C;
  WRC(isk_alloc((void **)&t->a, n * 2));
  if (grad) WRC(isk_alloc((void **)&t->g, n * 4));
  w->gm_elems = std::max(w->gm_elems, n);
  return ISKRA_OK;
}

static void ws_free_tensor(WsTensor *t) {
  isk_free(t->a);
  isk_free(t->g);
  t->a = nullptr;
  t->g = nullptr;
}

/* channels of level l: base * 2^l, held at base * 8 from level 3 on (so a
 * deep network keeps its coarse levels affordable) */
static int ws_chan(const iskra_ws *w, int l) { return w->base << std::min(l, 3); }

/* layer order: enc0A, enc0B, ..., enc(L-1)B, dec(L-2)A, dec(L-2)B, ..., dec0B, out */
static int ws_enc(int l, int b) { return 2 * l + b; }
static int ws_dec(const iskra_ws *w, int l, int b) { return 2 * w->L + 2 * (w->L - 2 - l) + b; }
static int ws_out(const iskra_ws *w) { return 2 * w->L + 2 * (w->L - 1); }

static void ws_add_conv(iskra_ws *w, int cin, int cout, int level, int relu) {
  WsConv c;
  c.cin = cin;
  c.cout = cout;
  c.level = level;
  c.relu = relu;
  c.woff = w->nparam;
  w->nparam += (long long)cout * 9 * cin;
  w->conv.push_back(c);
}

/* Order of a layer's sums (see k_ws_conv): 32 channels at a time where blocks of 256
 * pixels by 64, 32 or 16 output channels, the first of those that divide the layer and
 * number at least 256, or else the most numerous of them and of blocks of 64
 * pixels, are of 256 pixels, and the channels and the plane divide evenly. */
static bool ws_chunk_major(long long npix, int side, int cin, int cout) {
  static const int blocks[6][2] = {{64, 256}, {32, 256}, {16, 256}, {64, 64}, {32, 64}, {16, 64}};
  int px = 64;
  long long most = -1;
  for (const int *k : blocks) {
    if (cout % k[0] || npix % k[1]) continue;
    const long long nb = (npix / k[1]) * (cout / k[0]);
    if (nb > most) px = k[1];
    most = std::max(most, nb);
    if (nb >= 256) break;
  }
  return px == 256 && cin % 32 == 0 && side % 16 == 0;
}

/* launches the convolution described by a (its H and W are set here) on batch b
 * of a level */
struct WsShape {
  int nj, rw, wc;
  int rows() const { return rw * (4 / wc); }
  int chan() const { return 16 * nj * wc; }
};
static int ws_launch_conv(iskra_ws *w, int level, int b, ConvArgs a) {
  a.H = a.W = ws_side(w, level);
  if (a.Cin % 8 || a.Cout % 16 || a.H % 8) {
    isk_set_error("warm start: conv shape %d->%d on side %d not supported", a.Cin, a.Cout, a.H);
    return ISKRA_E_ARG;
  }
  /* the first of the tiles, in order of fewer loads per product, that gives at least
   * WS_CONV_MIN_WG work-groups; else the one with the most */
  static const WsShape shapes[] = {{2, 4, 1}, {1, 4, 2}, {1, 2, 2}, {1, 4, 1}, {1, 2, 1}};
  const WsShape *s = nullptr;
  long long most = -1, tiles = 0;
  for (const WsShape &k : shapes) {
    if (a.Cout % k.chan()) continue;
    const long long nt = (long long)b * ((a.W + 15) / 16) * ((a.H + k.rows() - 1) / k.rows());
    const long long wg = nt * (a.Cout / k.chan());
    if (wg <= most) continue;
    most = wg;
    tiles = nt;
    s = &k;
    if (wg >= WS_CONV_MIN_WG) break;
  }
  const dim3 grid((unsigned)tiles, (unsigned)(a.Cout / s->chan()));
  hipStream_t st = w->ctx->stream;
  auto is = [&](int nj, int rw, int wc) { return s->nj == nj && s->rw == rw && s->wc == wc; };
  if (ws_chunk_major(ws_npix(w, level, b), a.H, a.Cin, a.Cout)) {
    auto k = is(2, 4, 1) ? k_ws_conv<2, 4, 1, 1>
             : is(1, 4, 2) ? (a.Cin % 64 ? k_ws_conv<1, 4, 2, 1> : k_ws_conv<1, 4, 2, 2>)
             : is(1, 2, 2) ? (a.Cin % 128 ? k_ws_conv<1, 2, 2, 1> : k_ws_conv<1, 2, 2, 4>)
             : is(1, 4, 1) ? k_ws_conv<1, 4, 1, 1>
                           : k_ws_conv<1, 2, 1, 1>;
    hipLaunchKernelGGL(k, grid, dim3(256), 0, st, a);
  } else {
    const size_t out = 4 * 4 * 16 * (16 * s->nj + 4);
    size_t shm = (size_t)18 * (s->rows() + 2) * ws_taps_stride(a.Cin) * 2;
    const bool lds = shm <= 65536;
    shm = lds ? std::max(shm, out) : out;
    auto k = is(2, 4, 1) ? (lds ? k_ws_conv_taps<2, 4, 1, true> : k_ws_conv_taps<2, 4, 1, false>)
             : is(1, 4, 2) ? (lds ? k_ws_conv_taps<1, 4, 2, true> : k_ws_conv_taps<1, 4, 2, false>)
             : is(1, 2, 2) ? (lds ? k_ws_conv_taps<1, 2, 2, true> : k_ws_conv_taps<1, 2, 2, false>)
             : is(1, 4, 1) ? (lds ? k_ws_conv_taps<1, 4, 1, true> : k_ws_conv_taps<1, 4, 1, false>)
                           : (lds ? k_ws_conv_taps<1, 2, 1, true> : k_ws_conv_taps<1, 2, 1, false>);
    hipLaunchKernelGGL(k, grid, dim3(256), shm, st, a);
  }
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* forward of a layer: input X (up: read as its 2x2 repetition) to activations Y
 * (pool: also to their 2x2 averages), or to the output plane (Y = null) */
static int ws_fwd_conv(iskra_ws *w, int layer, int b, const uint16_t *X, const uint16_t *skip,
                       uint16_t *Y, int up, uint16_t *pool) {
  const WsConv &c = w->conv[layer];
  ConvArgs a = {};
  a.X = X;
  a.Wt = c.wt;
  a.Cin = c.cin;
  a.Cout = c.cout;
  a.skip = skip;
  a.Y = Y;
  a.P = pool;
  a.Yf = w->out;
  a.relu = c.relu;
  a.mode = Y ? WS_ACT : WS_PLANE;
  a.up = up;
  return ws_launch_conv(w, c.level, b, a);
}

/* input gradient of a layer: from its masked output gradient G to the masked
 * gradient Gm of the activation act it came from (mode, Eg: see ConvArgs) */
static int ws_dgrad(iskra_ws *w, int layer, int b, const uint16_t *G, int mode,
                    const WsTensor &act, float *Eg, uint16_t *Gm) {
  const WsConv &c = w->conv[layer];
  ConvArgs a = {};
  a.X = G;
  a.Wt = c.wtt;
  a.Cin = c.cout;
  a.Cout = c.cin;
  a.act = act.a;
  a.Gm = Gm;
  a.Eg = Eg;
  a.mode = mode;
  return ws_launch_conv(w, c.level, b, a);
}

/* chunks of a layer's weight gradient: about 1024 work-groups of 32 x 16 channels
 * would take one each, the partial sums within WS_PART_BYTES */
static int ws_chunks(const WsConv &c, long long nseg, int *seg_per_chunk) {
  const long long per_chunk = 9ll * c.cout * c.cin;
  const long long fit = std::max(1ll, WS_PART_BYTES / 4 / per_chunk);
  const long long want = std::max(1, 1024 / (((c.cout + 31) / 32) * ((c.cin + 15) / 16)));
  const long long most = std::min(std::min(fit, want), nseg);
  *seg_per_chunk = (int)((nseg + most - 1) / most);
  return (int)((nseg + *seg_per_chunk - 1) / *seg_per_chunk);
}

template <int NC, int CW, int IW, int TW>
static int ws_launch_wgrad(iskra_ws *w, const WsConv &c, const WgradArgs &a, int nchunk) {
  const int gy = (c.cout + 16 * NC * CW - 1) / (16 * NC * CW), gz = (c.cin + 16 * IW - 1) / (16 * IW);
  hipLaunchKernelGGL((k_ws_wgrad<NC, CW, IW, TW>), dim3((unsigned)nchunk, gy, gz), dim3(256),
                     (wsg_lds<NC, CW, IW>()), w->ctx->stream, a);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

/* The split of the four waves follows the channels that there are: blocks of 32 x 32
 * (output, input) channels, two work-groups a compute unit on a large layer (64 x 32 reads
 * less per product, but there is one then: 22 us against 20), and with 16 channels
 * the waves share the taps instead of computing padding. */
static int ws_wgrad(iskra_ws *w, int layer, int b, const uint16_t *G, const uint16_t *X,
                    int up = 0) {
  const WsConv &c = w->conv[layer];
  WgradArgs a;
  a.X = X;
  a.G = G;
  a.up = up;
  a.part = w->part;
  a.H = a.W = ws_side(w, c.level);
  a.Cin = c.cin;
  a.Cout = c.cout;
  a.nseg = (int)(ws_npix(w, c.level, b) / 64);
  const int nchunk = ws_chunks(c, a.nseg, &a.seg_per_chunk);
  if (c.cin <= 16 && c.cout <= 16) WRC((ws_launch_wgrad<1, 1, 1, 4>(w, c, a, nchunk)));
  else if (c.cin <= 16) WRC((ws_launch_wgrad<1, 2, 1, 2>(w, c, a, nchunk)));
  else if (c.cout <= 16) WRC((ws_launch_wgrad<1, 1, 2, 2>(w, c, a, nchunk)));
  else WRC((ws_launch_wgrad<2, 1, 2, 2>(w, c, a, nchunk)));
  const long long n = (long long)c.cout * 9 * c.cin;
  hipLaunchKernelGGL(k_ws_reduce, dim3((unsigned)((n + 63) / 64)), dim3(16 * WSR_ROWS), 0,
                     w->ctx->stream, (const float *)w->part, w->grads + c.woff, n, nchunk);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

static int ws_zero(iskra_ws *w, float *p, long long n) {
  hipLaunchKernelGGL(k_ws_fill, dim3(ws_grid(n)), dim3(EW_BLOCK), 0, w->ctx->stream, p, n, 0.f);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

static const WsTensor &ws_dec_out(const iskra_ws *w, int l) {
  return l == w->L - 1 ? w->E[l] : w->D[l];
}

/* forward of a batch already in A0; output plane in w->out */
static int ws_forward(iskra_ws *w, int b) {
  const int L = w->L;
  for (int l = 0; l < L; ++l) {
    WRC(ws_fwd_conv(w, ws_enc(l, 0), b, l == 0 ? w->A0.a : w->P[l].a, nullptr, w->Ea[l].a, 0,
                    nullptr));
    WRC(ws_fwd_conv(w, ws_enc(l, 1), b, w->Ea[l].a, nullptr, w->E[l].a, 0,
                    l + 1 < L ? w->P[l + 1].a : nullptr));
  }
  for (int l = L - 2; l >= 0; --l) {
    WRC(ws_fwd_conv(w, ws_dec(w, l, 0), b, ws_dec_out(w, l + 1).a, w->E[l].a, w->Da[l].a, 1,
                    nullptr));
    WRC(ws_fwd_conv(w, ws_dec(w, l, 1), b, w->Da[l].a, nullptr, w->D[l].a, 0, nullptr));
  }
  const WsTensor &last = L > 1 ? w->D[0] : w->E[0];
  return ws_fwd_conv(w, ws_out(w), b, last.a, nullptr, nullptr, 0, nullptr);
}

static int ws_pre(iskra_ws *w, int b);

/* energy objective on a batch (x, t) already mapped to (P x, P t) by
 * ws_pre: z = k post-sweeps from gain * out, e = z - gain t (= P (gain out
 * - gain t), the error of the whole two-level cycle), loss = sum e.Ae /
 * sum (gain t).A(gain t) over the batch; with_grad: Gout = its gradient with
 * respect to the output plane, 2 gain (I - om4 A)^k A e / denominator.
 * Planes ping-pong between eg_e and eg_ae. */
static int ws_energy_loss(iskra_ws *w, int b, bool with_grad, double *loss) {
  hipStream_t st = w->ctx->stream;
  const long long npix = ws_npix(w, 0, b);
  const unsigned nb = std::min(ws_grid(npix), (unsigned)(w->dpart_n / 2));
  /* no post-sweeps (sweeps = 0, or the network's own error scored):
   * one pass with om4 = 0 forms e = gain (o - t) */
  const bool post = w->obj == ISKRA_WS_ENERGY && w->sweeps > 0;
  const int ks = post ? w->sweeps : 1;
  const float gain = (float)w->gain, om4 = post ? (float)w->om4 : 0.f;
  float *buf[2] = {w->eg_e, w->eg_ae};
  const float *src = w->out;
  int cur = 0;
  for (int k = 0; k < ks; ++k) {
    const int last = k == ks - 1;
    hipLaunchKernelGGL(k_ws_eg_sweep, dim3(nb), dim3(EW_BLOCK), 0, st, src, buf[cur],
                       (const uint16_t *)w->A0.a, (const float *)w->tgt, w->S, npix,
                       k == 0 ? gain : 1.f, om4, gain, last, w->dpart, (int)nb);
    ISK_CHECK_LAUNCH();
    src = buf[cur];
    cur ^= 1;
  }
  /* e in buf[cur ^ 1]; A e into buf[cur] */
  hipLaunchKernelGGL(k_ws_eg_ae, dim3(nb), dim3(EW_BLOCK), 0, st, src, buf[cur], w->S, npix,
                     w->dpart);
  ISK_CHECK_LAUNCH();
  std::vector<double> h(2 * nb);
  ISK_HIP(hipMemcpyAsync(h.data(), w->dpart, 2 * nb * 8, hipMemcpyDeviceToHost, st));
  ISK_HIP(hipStreamSynchronize(st));
  double num = 0.0, den = 0.0;
  for (unsigned i = 0; i < nb; ++i) {
    num += h[i];
    den += h[nb + i];
  }
  if (!(den > 0.0)) den = 1.0;
  if (loss) *loss = num / den;
  if (with_grad) {
    /* the sweeps' adjoint, applied k times (A is symmetric); the first
     * carries the factor 2 gain / den */
    for (int k = 0; k < ks; ++k) {
      const int last = k == ks - 1;
      hipLaunchKernelGGL(k_ws_eg_back, dim3(ws_grid(npix)), dim3(EW_BLOCK), 0, st,
                         (const float *)buf[cur], buf[cur ^ 1], last ? w->gout : nullptr, w->S,
                         npix, om4, k == 0 ? (float)(2.0 * w->gain / den) : 1.f);
      ISK_CHECK_LAUNCH();
      cur ^= 1;
    }
  }
  return ISKRA_OK;
}

/* loss of w->out against w->tgt; with_grad: also Gout; returns the mean */
static int ws_loss(iskra_ws *w, int b, bool with_grad, double *loss) {
  if (w->obj != ISKRA_WS_PHI_MSE) return ws_energy_loss(w, b, with_grad, loss);
  const long long npix = ws_npix(w, 0, b);
  const long long count = (long long)b * (w->S - 1) * (w->S - 1);
  const unsigned nb = std::min(ws_grid(npix), (unsigned)w->dpart_n);
  hipLaunchKernelGGL(k_ws_loss, dim3(nb), dim3(EW_BLOCK), 0, w->ctx->stream,
                     (const float *)w->out, (const float *)w->tgt, with_grad ? w->gout : nullptr,
                     w->dpart, w->S, npix, (float)(1.0 / (double)count));
  ISK_CHECK_LAUNCH();
  std::vector<double> h(nb);
  ISK_HIP(hipMemcpyAsync(h.data(), w->dpart, nb * 8, hipMemcpyDeviceToHost, w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  double s = 0.0;
  for (unsigned i = 0; i < nb; ++i) s += h[i];
  if (loss) *loss = s / (double)count;
  return ISKRA_OK;
}

/* backward after ws_forward + ws_loss(with_grad): parameter gradients in w->grads.
 * g is the masked gradient of the layer at hand: Gout (the output layer is linear),
 * then in turn one of two buffers.  The skip connections' gradients wait in E's. */
static int ws_backward(iskra_ws *w, int b) {
  const int L = w->L;
  int cur = 0;
  const uint16_t *g = w->gout;
  auto dgrad = [&](int layer, int mode, const WsTensor &act, float *Eg) {
    const int rc = ws_dgrad(w, layer, b, g, mode, act, Eg, w->gm[cur]);
    g = w->gm[cur];
    cur ^= 1;
    return rc;
  };
  const WsTensor &last = L > 1 ? w->D[0] : w->E[0];
  WRC(ws_wgrad(w, ws_out(w), b, g, last.a));
  WRC(dgrad(ws_out(w), WS_MASK, last, nullptr));
  for (int l = 0; l <= L - 2; ++l) {
    const WsTensor &in = ws_dec_out(w, l + 1);
    WRC(ws_wgrad(w, ws_dec(w, l, 1), b, g, w->Da[l].a));
    WRC(dgrad(ws_dec(w, l, 1), WS_MASK, w->Da[l], w->E[l].g));
    WRC(ws_wgrad(w, ws_dec(w, l, 0), b, g, in.a, 1));
    WRC(dgrad(ws_dec(w, l, 0), WS_UP, in, nullptr));
  }
  for (int l = L - 1; l >= 0; --l) {
    WRC(ws_wgrad(w, ws_enc(l, 1), b, g, w->Ea[l].a));
    WRC(dgrad(ws_enc(l, 1), WS_MASK, w->Ea[l], nullptr));
    WRC(ws_wgrad(w, ws_enc(l, 0), b, g, l == 0 ? w->A0.a : w->P[l].a));
    if (l > 0) WRC(dgrad(ws_enc(l, 0), WS_POOL, w->E[l - 1], w->E[l - 1].g));
  }
  return ISKRA_OK;
}

static int ws_prep_weights(iskra_ws *w) {
  for (size_t i = 0; i < w->conv.size(); ++i) {
    WsConv &c = w->conv[i];
    const long long n =
        (long long)c.cout * ws_kpad(c.cin) + (c.wtt ? (long long)c.cin * ws_kpad(c.cout) : 0);
    hipLaunchKernelGGL(k_ws_wprep, dim3(ws_grid(n)), dim3(EW_BLOCK), 0, w->ctx->stream,
                       (const float *)(w->params + c.woff), c.wt, c.wtt, c.cin, c.cout);
    ISK_CHECK_LAUNCH();
  }
  return ISKRA_OK;
}

static void ws_release(iskra_ws *w) {
  for (WsConv &c : w->conv) {
    isk_free(c.wt);
    isk_free(c.wtt);
  }
  ws_free_tensor(&w->A0);
  for (int l = 0; l < WS_MAX_LEVELS; ++l) {
    ws_free_tensor(&w->Ea[l]);
    ws_free_tensor(&w->E[l]);
    ws_free_tensor(&w->P[l]);
    ws_free_tensor(&w->Da[l]);
    ws_free_tensor(&w->D[l]);
  }
  void *ptrs[] = {w->params, w->grads, w->m,     w->v,     w->out,    w->tgt,   w->gout,
                  w->gm[0],  w->gm[1], w->part,  w->dpart, w->scal,  w->idx,    w->xin,   w->ds_in,
                  w->ds_out, w->eg_e,  w->eg_ae, w->lx,    w->lr,     w->lz,    w->lzs,
                  w->lp[0],  w->lp[1], w->lq[0], w->lq[1], w->lpart,  w->ls,    w->lpre[0],
                  w->lpre[1], w->lrp};
  for (void *p : ptrs) isk_free(p);
}

static int ws_check(iskra_ws *w) {
  if (!w || !w->ctx) {
    isk_set_error("warm start: null network");
    return ISKRA_E_ARG;
  }
  isk_clear_error();
  ISK_HIP(hipSetDevice(w->ctx->device));
  return ISKRA_OK;
}

/* the context's grid must be the network's: square, 2-D, (S+1)^2 nodes */
static int ws_check_grid(iskra_ws *w) {
  const iskra_ctx *c = w->ctx;
  if (!c->have_grid || c->g.dim != 2 || c->g.nx != w->S + 1 || c->g.ny != w->S + 1) {
    isk_set_error("warm start: the context grid must be 2-D with %d x %d nodes", w->S + 1,
                  w->S + 1);
    return ISKRA_E_STATE;
  }
  if (c->g.axial) {
    isk_set_error("warm start: the network maps Cartesian grids, not an axial one");
    return ISKRA_E_UNSUPPORTED;
  }
  return ISKRA_OK;
}

/* f = rho * dx^2 / eps0 of the context -> scale in w->scal */
static int ws_rhs_scale(iskra_ws *w, double *fscale) {
  iskra_ctx *c = w->ctx;
  *fscale = c->g.dx * c->g.dx / c->ps.eps0;
  const long long cnt = (long long)(w->S - 1) * (w->S - 1);
  const unsigned nb = std::min(ws_grid(cnt), (unsigned)w->dpart_n);
  hipLaunchKernelGGL(k_ws_rhs_sumsq, dim3(nb), dim3(EW_BLOCK), 0, c->stream,
                     (const double *)c->rho, c->g.nx, *fscale, w->dpart);
  ISK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_ws_rhs_scale, dim3(1), dim3(EW_BLOCK), 0, c->stream, (const double *)w->dpart,
                     (int)nb, cnt, w->scal);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

extern "C" {

int iskra_ws_create(iskra_ctx *ctx, int levels, int base, int side, int max_batch,
                    iskra_ws **out) {
  if (!ctx || !out) {
    isk_set_error("ws_create: null argument");
    return ISKRA_E_ARG;
  }
  ISK_HIP(hipSetDevice(ctx->device));
  isk_clear_error();
  *out = nullptr;
  if (levels < 1 || levels > WS_MAX_LEVELS || base < 16 || base % 16 || side < 16 ||
      (side & (side - 1)) || (side >> (levels - 1)) < 8 || max_batch < 1 || max_batch > 1024) {
    isk_set_error("ws_create: levels in [1,%d], base a multiple of 16, side a power of two with "
                  "side/2^(levels-1) >= 8, max_batch in [1,1024]", WS_MAX_LEVELS);
    return ISKRA_E_ARG;
  }
  iskra_ws *w = new iskra_ws();
  w->ctx = ctx;
  w->L = levels;
  w->base = base;
  w->S = side;
  w->maxb = max_batch;
  for (int l = 0; l < levels; ++l) {
    ws_add_conv(w, l == 0 ? WS_IN_CH : ws_chan(w, l - 1), ws_chan(w, l), l, 1);
    ws_add_conv(w, ws_chan(w, l), ws_chan(w, l), l, 1);
  }
  for (int l = levels - 2; l >= 0; --l) {
    ws_add_conv(w, ws_chan(w, l + 1), ws_chan(w, l), l, 1);
    ws_add_conv(w, ws_chan(w, l), ws_chan(w, l), l, 1);
  }
  ws_add_conv(w, ws_chan(w, 0), WS_OUT_CH, 0, 0);
  int rc = ISKRA_OK;
#define WTRY(x)                  \
  do {                           \
    rc = (x);                    \
    if (rc) goto fail;           \
  } while (0)
  for (size_t i = 0; i < w->conv.size(); ++i) {
    WsConv &c = w->conv[i];
    WTRY(isk_alloc((void **)&c.wt, (size_t)c.cout * ws_kpad(c.cin) * 2));
    if (i != 0) WTRY(isk_alloc((void **)&c.wtt, (size_t)c.cin * ws_kpad(c.cout) * 2));
  }
  WTRY(isk_alloc((void **)&w->params, w->nparam * 4));
  WTRY(isk_alloc((void **)&w->grads, w->nparam * 4));
  WTRY(isk_alloc((void **)&w->m, w->nparam * 4));
  WTRY(isk_alloc((void **)&w->v, w->nparam * 4));
  WTRY(ws_tensor(w, &w->A0, 0, WS_IN_CH, false));
  for (int l = 0; l < levels; ++l) {
    WTRY(ws_tensor(w, &w->Ea[l], l, ws_chan(w, l), false));
    WTRY(ws_tensor(w, &w->E[l], l, ws_chan(w, l), l <= levels - 2)); /* skip gradients */
    if (l > 0) WTRY(ws_tensor(w, &w->P[l], l, ws_chan(w, l - 1), false));
    if (l <= levels - 2) {
      WTRY(ws_tensor(w, &w->Da[l], l, ws_chan(w, l), false));
      WTRY(ws_tensor(w, &w->D[l], l, ws_chan(w, l), false));
    }
  }
  {
    const long long npix = ws_npix(w, 0, max_batch);
    w->gm_elems = std::max(w->gm_elems, npix * WS_OUT_CH);
    WTRY(isk_alloc((void **)&w->out, npix * 4));
    WTRY(isk_alloc((void **)&w->tgt, npix * 4));
    WTRY(isk_alloc((void **)&w->xin, npix * 4));
    WTRY(isk_alloc((void **)&w->gout, npix * WS_OUT_CH * 2));
    WTRY(isk_alloc((void **)&w->eg_e, npix * 4));
    WTRY(isk_alloc((void **)&w->eg_ae, npix * 4));
    for (uint16_t *&g : w->gm) WTRY(isk_alloc((void **)&g, w->gm_elems * 2));
    long long part_bytes = WS_PART_BYTES; /* at least one chunk of the largest layer */
    for (const WsConv &c : w->conv) part_bytes = std::max(part_bytes, 36ll * c.cin * c.cout);
    WTRY(isk_alloc((void **)&w->part, part_bytes));
    w->dpart_n = 8192;
    WTRY(isk_alloc((void **)&w->dpart, w->dpart_n * 8));
    WTRY(isk_alloc((void **)&w->scal, 64));
    WTRY(isk_alloc((void **)&w->idx, (size_t)max_batch * 8));
  }
  WTRY(ws_zero(w, w->params, w->nparam));
  WTRY(ws_zero(w, w->m, w->nparam));
  WTRY(ws_zero(w, w->v, w->nparam));
  WTRY(ws_zero(w, w->grads, w->nparam));
  WTRY(ws_prep_weights(w));
  {
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
      rc = isk_hip_fail(e, "hipStreamSynchronize", __FILE__, __LINE__);
      goto fail;
    }
  }
#undef WTRY
  *out = w;
  return ISKRA_OK;
fail:
  ws_release(w);
  delete w;
  return rc;
}

int iskra_ws_destroy(iskra_ws *w) {
  if (!w) return ISKRA_OK;
  if (w->ctx) (void)hipSetDevice(w->ctx->device);
  if (w->ctx) (void)hipStreamSynchronize(w->ctx->stream);
  ws_release(w);
  delete w;
  return ISKRA_OK;
}

int iskra_ws_param_count(iskra_ws *w, int64_t *n) {
  WRC(ws_check(w));
  if (!n) return ISKRA_E_ARG;
  *n = w->nparam;
  return ISKRA_OK;
}

int iskra_ws_set_params(iskra_ws *w, const float *p) {
  WRC(ws_check(w));
  if (!p) return ISKRA_E_ARG;
  ISK_HIP(hipMemcpyAsync(w->params, p, w->nparam * 4, hipMemcpyHostToDevice, w->ctx->stream));
  WRC(ws_zero(w, w->m, w->nparam));
  WRC(ws_zero(w, w->v, w->nparam));
  w->adam_t = 0;
  WRC(ws_prep_weights(w));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

int iskra_ws_get_params(iskra_ws *w, float *p) {
  WRC(ws_check(w));
  if (!p) return ISKRA_E_ARG;
  ISK_HIP(hipMemcpyAsync(p, w->params, w->nparam * 4, hipMemcpyDeviceToHost, w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

int iskra_ws_set_gain(iskra_ws *w, double gain) {
  WRC(ws_check(w));
  if (!(gain > 0.0)) {
    isk_set_error("ws_set_gain: gain must be positive");
    return ISKRA_E_ARG;
  }
  w->gain = gain;
  return ISKRA_OK;
}

int iskra_ws_set_objective(iskra_ws *w, int objective, double omega, int sweeps) {
  WRC(ws_check(w));
  if ((objective != ISKRA_WS_PHI_MSE && objective != ISKRA_WS_ENERGY &&
       objective != ISKRA_WS_ENERGY_NET) ||
      !(omega >= 0.0) ||
      omega >= 2.0 || sweeps < 0 || sweeps > WS_MAX_SWEEPS) {
    isk_set_error("ws_set_objective: objective ISKRA_WS_PHI_MSE, _ENERGY or _ENERGY_NET, omega in "
                  "[0, 2), sweeps in [0, %d]", WS_MAX_SWEEPS);
    return ISKRA_E_ARG;
  }
  w->obj = objective;
  w->om4 = 0.25 * omega;
  w->sweeps = sweeps;
  return ISKRA_OK;
}

static int ws_host_input(iskra_ws *w, int batch, const float *in) {
  const long long npix = ws_npix(w, 0, batch);
  ISK_HIP(hipMemcpyAsync(w->xin, in, npix * 4, hipMemcpyHostToDevice, w->ctx->stream));
  hipLaunchKernelGGL(k_ws_input, dim3(ws_grid(npix)), dim3(EW_BLOCK), 0, w->ctx->stream,
                     (const float *)w->xin, w->A0.a, npix);
  ISK_CHECK_LAUNCH();
  return ISKRA_OK;
}

int iskra_ws_forward(iskra_ws *w, int batch, const float *in, float *out) {
  WRC(ws_check(w));
  if (batch < 1 || batch > w->maxb || !in || !out) return ISKRA_E_ARG;
  WRC(ws_host_input(w, batch, in));
  WRC(ws_forward(w, batch));
  ISK_HIP(hipMemcpyAsync(out, w->out, ws_npix(w, 0, batch) * 4, hipMemcpyDeviceToHost,
                         w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

int iskra_ws_backward(iskra_ws *w, int batch, const float *in, const float *target,
                      float *grads, double *loss) {
  WRC(ws_check(w));
  if (batch < 1 || batch > w->maxb || !in || !target) return ISKRA_E_ARG;
  WRC(ws_host_input(w, batch, in));
  ISK_HIP(hipMemcpyAsync(w->tgt, target, ws_npix(w, 0, batch) * 4, hipMemcpyHostToDevice,
                         w->ctx->stream));
  WRC(ws_pre(w, batch));
  WRC(ws_forward(w, batch));
  WRC(ws_loss(w, batch, true, loss));
  WRC(ws_backward(w, batch));
  if (grads)
    ISK_HIP(hipMemcpyAsync(grads, w->grads, w->nparam * 4, hipMemcpyDeviceToHost,
                           w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

int iskra_ws_dataset_reserve(iskra_ws *w, int64_t n) {
  WRC(ws_check(w));
  if (n < 1) return ISKRA_E_ARG;
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  isk_free(w->ds_in);
  isk_free(w->ds_out);
  w->ds_in = nullptr;
  w->ds_out = nullptr;
  w->ds_cap = w->ds_n = 0;
  const long long S2 = (long long)w->S * w->S;
  WRC(isk_alloc((void **)&w->ds_in, (size_t)n * S2 * 2));
  WRC(isk_alloc((void **)&w->ds_out, (size_t)n * S2 * 4));
  w->ds_cap = n;
  return ISKRA_OK;
}

int iskra_ws_capture(iskra_ws *w, int64_t *index) {
  WRC(ws_check(w));
  WRC(ws_check_grid(w));
  if (w->ds_n >= w->ds_cap) {
    isk_set_error("ws_capture: dataset full (%lld samples)", (long long)w->ds_cap);
    return ISKRA_E_CAPACITY;
  }
  double fscale;
  WRC(ws_rhs_scale(w, &fscale));
  const long long S2 = (long long)w->S * w->S;
  iskra_ctx *c = w->ctx;
  hipLaunchKernelGGL(k_ws_rhs_store, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, c->stream,
                     (const double *)c->rho, (const double *)c->phi, c->g.nx, fscale,
                     (const double *)w->scal, w->ds_in + w->ds_n * S2, (uint16_t *)nullptr,
                     w->ds_out + w->ds_n * S2);
  ISK_CHECK_LAUNCH();
  if (index) *index = w->ds_n;
  ++w->ds_n;
  return ISKRA_OK;
}

int iskra_ws_dataset_size(iskra_ws *w, int64_t *n) {
  WRC(ws_check(w));
  if (!n) return ISKRA_E_ARG;
  *n = w->ds_n;
  return ISKRA_OK;
}

/* RMS of the stored (phi / s) targets of samples [first, first+count) */
int iskra_ws_dataset_rms(iskra_ws *w, int64_t first, int64_t count, double *rms) {
  WRC(ws_check(w));
  if (first < 0 || count < 1 || first + count > w->ds_n || !rms) return ISKRA_E_ARG;
  const long long S2 = (long long)w->S * w->S;
  const long long n = count * S2;
  const unsigned nb = std::min(ws_grid(n), (unsigned)w->dpart_n);
  hipLaunchKernelGGL(k_ws_sumsq, dim3(nb), dim3(EW_BLOCK), 0, w->ctx->stream,
                     (const float *)(w->ds_out + first * S2), n, w->dpart);
  ISK_CHECK_LAUNCH();
  std::vector<double> h(nb);
  ISK_HIP(hipMemcpyAsync(h.data(), w->dpart, nb * 8, hipMemcpyDeviceToHost, w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  double s = 0.0;
  for (unsigned i = 0; i < nb; ++i) s += h[i];
  *rms = sqrt(s / (double)(count * (long long)(w->S - 1) * (w->S - 1)));
  return ISKRA_OK;
}

/* energy objective with k > 0 sweeps: the batch pair (x in A0, t in tgt)
 * becomes (P x, P t), P = (I - om4 A)^k, the residual and correction the
 * network meets after k pre-sweeps from zero (A^-1 commutes with P) */
static int ws_pre(iskra_ws *w, int b) {
  if (w->obj == ISKRA_WS_PHI_MSE || w->sweeps == 0) return ISKRA_OK;
  hipStream_t st = w->ctx->stream;
  const long long npix = ws_npix(w, 0, b);
  const unsigned g = ws_grid(npix);
  float *buf[2] = {w->eg_e, w->eg_ae};
  const float om4 = (float)w->om4;
  for (int pass = 0; pass < 2; ++pass) {
    const float *src = w->tgt;
    if (pass == 0) {
      hipLaunchKernelGGL(k_ws_a0_get, dim3(g), dim3(EW_BLOCK), 0, st, (const uint16_t *)w->A0.a,
                         w->eg_ae, npix);
      ISK_CHECK_LAUNCH();
      src = w->eg_ae;
    }
    int cur = 0;
    for (int k = 0; k < w->sweeps; ++k) {
      hipLaunchKernelGGL(k_ws_eg_poly, dim3(g), dim3(EW_BLOCK), 0, st, src, buf[cur], w->S, npix,
                         om4);
      ISK_CHECK_LAUNCH();
      src = buf[cur];
      cur ^= 1;
    }
    if (pass == 0) {
      hipLaunchKernelGGL(k_ws_input, dim3(g), dim3(EW_BLOCK), 0, st, src, w->A0.a, npix);
      ISK_CHECK_LAUNCH();
    } else {
      ISK_HIP(hipMemcpyAsync(w->tgt, src, npix * 4, hipMemcpyDeviceToDevice, st));
    }
  }
  return ISKRA_OK;
}

static int ws_load_batch(iskra_ws *w, const long long *idx, int b) {
  ISK_HIP(hipMemcpyAsync(w->idx, idx, (size_t)b * 8, hipMemcpyHostToDevice, w->ctx->stream));
  const long long S2 = (long long)w->S * w->S;
  hipLaunchKernelGGL(k_ws_batch, dim3(ws_grid(b * S2)), dim3(EW_BLOCK), 0, w->ctx->stream,
                     (const uint16_t *)w->ds_in, (const float *)w->ds_out,
                     (const long long *)w->idx, w->A0.a, w->tgt, (int)S2, b,
                     (float)(1.0 / w->gain));
  ISK_CHECK_LAUNCH();
  WRC(ws_pre(w, b));
  /* the index upload reads host memory of this call: finish before returning */
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

/* steps of Adam on random batches of samples [first, first+count), drawn with
 * Philox4x32-10 keyed by seed; losses[s] (nullable) = batch loss of step s */
int iskra_ws_train(iskra_ws *w, int64_t first, int64_t count, int batch, int steps, float lr,
                   uint64_t seed, double *losses) {
  WRC(ws_check(w));
  if (first < 0 || count < 1 || first + count > w->ds_n || batch < 1 || batch > w->maxb ||
      steps < 0 || !(lr > 0.f)) {
    isk_set_error("ws_train: bad range, batch or learning rate");
    return ISKRA_E_ARG;
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  std::vector<long long> idx(batch);
  for (int s = 0; s < steps; ++s) {
    for (int k = 0; k < batch; ++k) {
      IskU4 r = isk_philox((IskU4){(uint32_t)(w->adam_t + s), (uint32_t)k, 0x57534200u, 0u},
                           (uint32_t)seed, (uint32_t)(seed >> 32));
      idx[k] = first + (long long)(((uint64_t)r.x << 32 | r.y) % (uint64_t)count);
    }
    WRC(ws_load_batch(w, idx.data(), batch));
    WRC(ws_forward(w, batch));
    double loss = 0.0;
    WRC(ws_loss(w, batch, true, &loss));
    if (losses) losses[s] = loss;
    WRC(ws_backward(w, batch));
    const long long t = ++w->adam_t;
    const float c1 = (float)(1.0 / (1.0 - pow(b1, (double)t)));
    const float c2 = (float)(1.0 / (1.0 - pow(b2, (double)t)));
    hipLaunchKernelGGL(k_ws_adam, dim3(ws_grid(w->nparam)), dim3(EW_BLOCK), 0, w->ctx->stream,
                       w->params, (const float *)w->grads, w->m, w->v, w->nparam, lr, b1, b2, eps,
                       c1, c2);
    ISK_CHECK_LAUNCH();
    WRC(ws_prep_weights(w));
  }
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  return ISKRA_OK;
}

/* mean loss over samples [first, first+count), batches of the maximum size */
int iskra_ws_eval(iskra_ws *w, int64_t first, int64_t count, double *mse) {
  WRC(ws_check(w));
  if (first < 0 || count < 1 || first + count > w->ds_n || !mse) return ISKRA_E_ARG;
  double tot = 0.0;
  std::vector<long long> idx(w->maxb);
  for (long long s = 0; s < count; s += w->maxb) {
    const int b = (int)std::min((long long)w->maxb, count - s);
    for (int k = 0; k < b; ++k) idx[k] = first + s + k;
    WRC(ws_load_batch(w, idx.data(), b));
    WRC(ws_forward(w, b));
    double l = 0.0;
    WRC(ws_loss(w, b, false, &l));
    tot += l * b;
  }
  *mse = tot / (double)count;
  return ISKRA_OK;
}

/* z = the two-level cycle applied to the residual r: `sweeps` damped Jacobi
 * sweeps from z = 0, the network's estimate of A^-1 of what they leave
 * (r - A z, scaled by its RMS and the gain) added to z, then `sweeps`
 * sweeps again.  om4 = 0 or sweeps = 0: the network alone. */
static int ls_precond(iskra_ws *w, int nx, double om4, int sweeps, const double **z) {
  iskra_ctx *c = w->ctx;
  hipStream_t st = c->stream;
  const long long n = (long long)(nx - 2) * (nx - 2);
  const unsigned g = (unsigned)std::min((n + LS_BLOCK - 1) / LS_BLOCK, 1024ll);
  const int k = om4 > 0.0 ? sweeps : 0;
  /* pre-sweeps: ping-pong between lpre[0] and lpre[1] */
  const double *zpre = nullptr;
  for (int i = 0; i < k; ++i) {
    hipLaunchKernelGGL(k_ls_smooth, dim3(g), dim3(LS_BLOCK), 0, st, (const double *)w->lr, zpre,
                       w->lpre[i & 1], nx, om4);
    ISK_CHECK_LAUNCH();
    zpre = w->lpre[i & 1];
  }
  const double *rin = w->lr;
  if (zpre) {
    hipLaunchKernelGGL(k_ls_resid, dim3(g), dim3(LS_BLOCK), 0, st, (const double *)w->lr, zpre,
                       w->lrp, nx);
    ISK_CHECK_LAUNCH();
    rin = w->lrp;
  }
  const long long cnt = (long long)(w->S - 1) * (w->S - 1);
  const unsigned nb = std::min(ws_grid(cnt), (unsigned)w->dpart_n);
  hipLaunchKernelGGL(k_ws_rhs_sumsq, dim3(nb), dim3(EW_BLOCK), 0, st, rin, nx, 1.0, w->dpart);
  ISK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_ws_rhs_scale, dim3(1), dim3(EW_BLOCK), 0, st, (const double *)w->dpart, (int)nb,
                     cnt, w->scal);
  ISK_CHECK_LAUNCH();
  const long long S2 = (long long)w->S * w->S;
  hipLaunchKernelGGL(k_ws_rhs_store, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, st, rin,
                     (const double *)nullptr, nx, 1.0, (const double *)w->scal,
                     (uint16_t *)nullptr, w->A0.a, (float *)nullptr);
  ISK_CHECK_LAUNCH();
  WRC(ws_forward(w, 1));
  hipLaunchKernelGGL(k_ws_phi_out, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, st,
                     (const float *)w->out, w->lz, nx, w->gain, (const double *)w->scal);
  ISK_CHECK_LAUNCH();
  if (zpre) {
    hipLaunchKernelGGL(k_ls_add, dim3(g), dim3(LS_BLOCK), 0, st, w->lz, zpre, nx);
    ISK_CHECK_LAUNCH();
  }
  *z = w->lz;
  double *buf[2] = {w->lzs, w->lz};
  for (int i = 0; i < k; ++i) {
    hipLaunchKernelGGL(k_ls_smooth, dim3(g), dim3(LS_BLOCK), 0, st, (const double *)w->lr, *z,
                       buf[i & 1], nx, om4);
    ISK_CHECK_LAUNCH();
    *z = buf[i & 1];
  }
  return ISKRA_OK;
}

/* the context must hold the network's system: a configured solver with
 * phi = 0 on the four walls and no other Dirichlet node or periodic link;
 * allocates the iteration vectors on first use */
static int ls_setup(iskra_ws *w, const char *who, double omega, int sweeps) {
  WRC(ws_check_grid(w));
  iskra_ctx *c = w->ctx;
  IskPoisson &p = c->ps;
  if (p.kind < 0) {
    isk_set_error("%s: no Poisson solver configured", who);
    return ISKRA_E_STATE;
  }
  if (!(omega >= 0.0) || omega >= 2.0 || sweeps < 0 || sweeps > WS_MAX_SWEEPS) {
    isk_set_error("%s: the Jacobi weight must lie in [0, 2), sweeps in [0, %d]", who,
                  WS_MAX_SWEEPS);
    return ISKRA_E_ARG;
  }
  const int nx = c->g.nx;
  bool ok = !p.per_x && !p.per_y && (int)p.tags.size() == nx * nx;
  for (int j = 0; ok && j < nx; ++j)
    for (int i = 0; i < nx; ++i) {
      const int t = p.tags[(size_t)j * nx + i];
      const bool wall = i == 0 || j == 0 || i == nx - 1 || j == nx - 1;
      if (wall ? (t == 0 || p.tag_val[t] != 0.0) : t != 0) {
        ok = false;
        break;
      }
    }
  if (!ok) {
    isk_set_error("%s: the network solves phi = 0 on all four walls with no other Dirichlet "
                  "node or periodic link", who);
    return ISKRA_E_UNSUPPORTED;
  }
  const long long nn = (long long)nx * nx;
  if (!w->lx) {
    double **bufs[] = {&w->lx,    &w->lr,    &w->lz,      &w->lzs,     &w->lp[0], &w->lp[1],
                       &w->lq[0], &w->lq[1], &w->lpre[0], &w->lpre[1], &w->lrp};
    for (double **b : bufs) {
      WRC(isk_alloc((void **)b, nn * 8));
      ISK_HIP(hipMemsetAsync(*b, 0, nn * 8, c->stream));
    }
    WRC(isk_alloc((void **)&w->lpart, 4096 * 8));
    WRC(isk_alloc((void **)&w->ls, LS_NS * 8));
    ISK_HIP(hipMemsetAsync(w->ls, 0, LS_NS * 8, c->stream));
  }
  return ISKRA_OK;
}

/* training pair (r, phi - x) of the current iterate appended to the dataset */
static int ls_capture_pair(iskra_ws *w) {
  iskra_ctx *c = w->ctx;
  const int nx = c->g.nx;
  const long long cnt = (long long)(w->S - 1) * (w->S - 1);
  const unsigned nb = std::min(ws_grid(cnt), (unsigned)w->dpart_n);
  hipLaunchKernelGGL(k_ws_rhs_sumsq, dim3(nb), dim3(EW_BLOCK), 0, c->stream,
                     (const double *)w->lr, nx, 1.0, w->dpart);
  ISK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_ws_rhs_scale, dim3(1), dim3(EW_BLOCK), 0, c->stream, (const double *)w->dpart,
                     (int)nb, cnt, w->scal);
  ISK_CHECK_LAUNCH();
  const long long S2 = (long long)w->S * w->S;
  hipLaunchKernelGGL(k_ws_pair_store, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, c->stream,
                     (const double *)w->lr, (const double *)c->phi, (const double *)w->lx, nx,
                     (const double *)w->scal, w->ds_in + w->ds_n * S2, w->ds_out + w->ds_n * S2);
  ISK_CHECK_LAUNCH();
  ++w->ds_n;
  return ISKRA_OK;
}

/* Flexible CG from phi (warm) or 0 on f = dx^2 rho / eps0 until the relative
 * residual meets rtol or maxit iterations; with caps (ascending), the
 * iteration also stops after the last cap and the pair of every capped
 * iterate is captured.  Iterate in lx, residual in lr. */
static int ls_iterate(iskra_ws *w, int warm, double om4, int sweeps, int maxit, double rtol,
                      const int *caps, int ncaps, int *it_out, double *rr_out) {
  iskra_ctx *c = w->ctx;
  const int nx = c->g.nx;
  const long long n = (long long)(nx - 2) * (nx - 2);
  const int nb = (int)std::min((n + LS_BLOCK - 1) / LS_BLOCK, 1024ll);
  const double fscale = c->g.dx * c->g.dx / c->ps.eps0;
  hipLaunchKernelGGL(k_ls_init, dim3(nb), dim3(LS_BLOCK), 0, c->stream, (const double *)c->rho,
                     warm == ISKRA_WARM_PREV ? (const double *)c->phi : (const double *)nullptr,
                     nx, fscale, w->lx, w->lr, w->lpart);
  ISK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_ls_reduce, dim3(1), dim3(EW_BLOCK), 0, c->stream, (const double *)w->lpart,
                     nb, 2, w->ls + LS_FF);
  ISK_CHECK_LAUNCH();
  double s[2];
  ISK_HIP(hipMemcpyAsync(s, w->ls, 16, hipMemcpyDeviceToHost, c->stream));
  ISK_HIP(hipStreamSynchronize(c->stream));
  double rr = s[0] > 0.0 ? sqrt(s[1] / s[0]) : 0.0;
  int it = 0, cur = 0, next_cap = 0;
  if (caps) maxit = std::min(maxit, caps[ncaps - 1]);
  while (rr > rtol && it < maxit) {
    ++it;
    const double *z = nullptr;
    WRC(ls_precond(w, nx, om4, sweeps, &z));
    const int prev = cur ^ 1;
    if (it > 1) {
      hipLaunchKernelGGL(k_ls_dot, dim3(nb), dim3(LS_BLOCK), 0, c->stream, z,
                         (const double *)w->lq[prev], nx, w->lpart);
      ISK_CHECK_LAUNCH();
      hipLaunchKernelGGL(k_ls_reduce, dim3(1), dim3(EW_BLOCK), 0, c->stream,
                         (const double *)w->lpart, nb, 1, w->ls + LS_ZQ);
      ISK_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_ls_dir, dim3(nb), dim3(LS_BLOCK), 0, c->stream, z,
                       (const double *)w->lp[prev], w->lp[cur], nx, (const double *)w->ls,
                       it == 1 ? 1 : 0);
    ISK_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_ls_Ap, dim3(nb), dim3(LS_BLOCK), 0, c->stream,
                       (const double *)w->lp[cur], (const double *)w->lr, w->lq[cur], nx,
                       w->lpart);
    ISK_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_ls_reduce, dim3(1), dim3(EW_BLOCK), 0, c->stream, (const double *)w->lpart,
                       nb, 2, w->ls + LS_PQ);
    ISK_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_ls_xr, dim3(nb), dim3(LS_BLOCK), 0, c->stream, w->lx, w->lr,
                       (const double *)w->lp[cur], (const double *)w->lq[cur], nx,
                       (const double *)w->ls, w->lpart);
    ISK_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_ls_reduce, dim3(1), dim3(EW_BLOCK), 0, c->stream, (const double *)w->lpart,
                       nb, 1, w->ls + LS_RR);
    ISK_CHECK_LAUNCH();
    if (caps && next_cap < ncaps && it == caps[next_cap]) {
      WRC(ls_capture_pair(w));
      ++next_cap;
    }
    ISK_HIP(hipMemcpyAsync(s, w->ls, 16, hipMemcpyDeviceToHost, c->stream));
    ISK_HIP(hipStreamSynchronize(c->stream));
    rr = s[0] > 0.0 ? sqrt(s[1] / s[0]) : 0.0;
    cur ^= 1;
  }
  *it_out = it;
  *rr_out = rr;
  return ISKRA_OK;
}

int iskra_ws_solve(iskra_ws *w, int warm, double omega, int sweeps, int max_iter, int *iters,
                   double *relres) {
  WRC(ws_check(w));
  if (warm != ISKRA_WARM_ZERO && warm != ISKRA_WARM_PREV) return ISKRA_E_ARG;
  WRC(ls_setup(w, "ws_solve", omega, sweeps));
  iskra_ctx *c = w->ctx;
  IskPoisson &p = c->ps;
  const int nx = c->g.nx;
  hipEvent_t ev = nullptr;
  WRC(isk_prof_begin(c, &ev));
  int it = 0;
  double rr = 0.0;
  WRC(ls_iterate(w, warm, 0.25 * omega, sweeps, max_iter > 0 ? max_iter : p.max_iter, p.rtol,
                 nullptr, 0, &it, &rr));
  const long long n = (long long)(nx - 2) * (nx - 2);
  const int nb = (int)std::min((n + LS_BLOCK - 1) / LS_BLOCK, 1024ll);
  hipLaunchKernelGGL(k_ls_out, dim3(nb), dim3(LS_BLOCK), 0, c->stream, (const double *)w->lx,
                     c->phi, nx);
  ISK_CHECK_LAUNCH();
  WRC(isk_prof_end(c, ev, ISKRA_K_POISSON, 0));
  ISK_HIP(hipStreamSynchronize(c->stream));
  p.last_iters = it;
  p.last_relres = rr;
  c->stats.poisson_solves++;
  c->stats.poisson_iters += it;
  c->stats.last_iters = it;
  c->stats.last_relres = rr;
  if (iters) *iters = it;
  if (relres) *relres = rr;
  if (rr > p.rtol) {
    isk_set_error("ws_solve: relative residual %.3e above %.3e after %d iterations", rr, p.rtol,
                  it);
    return ISKRA_E_CONVERGE;
  }
  return ISKRA_OK;
}

int iskra_ws_capture_iterates(iskra_ws *w, double omega, int sweeps, const int *iters,
                              int n_iters, int64_t *captured) {
  WRC(ws_check(w));
  if (!iters || n_iters < 1 || iters[0] < 1) {
    isk_set_error("ws_capture_iterates: n_iters >= 1 iteration counts, the first >= 1");
    return ISKRA_E_ARG;
  }
  for (int k = 1; k < n_iters; ++k)
    if (iters[k] <= iters[k - 1]) {
      isk_set_error("ws_capture_iterates: iteration counts must increase");
      return ISKRA_E_ARG;
    }
  if (w->ds_n + n_iters > w->ds_cap) {
    isk_set_error("ws_capture_iterates: dataset full (%lld of %lld samples)", (long long)w->ds_n,
                  (long long)w->ds_cap);
    return ISKRA_E_CAPACITY;
  }
  WRC(ls_setup(w, "ws_capture_iterates", omega, sweeps));
  const long long n0 = w->ds_n;
  int it = 0;
  double rr = 0.0;
  WRC(ls_iterate(w, ISKRA_WARM_ZERO, 0.25 * omega, sweeps, iters[n_iters - 1], 0.0, iters,
                 n_iters, &it, &rr));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  if (captured) *captured = w->ds_n - n0;
  return ISKRA_OK;
}

int iskra_ws_dataset_get(iskra_ws *w, int64_t index, float *in, float *out) {
  WRC(ws_check(w));
  if (index < 0 || index >= w->ds_n || !in || !out) {
    isk_set_error("ws_dataset_get: index outside the dataset or null buffer");
    return ISKRA_E_ARG;
  }
  const long long S2 = (long long)w->S * w->S;
  std::vector<uint16_t> h(S2);
  ISK_HIP(hipMemcpyAsync(h.data(), w->ds_in + index * S2, S2 * 2, hipMemcpyDeviceToHost,
                         w->ctx->stream));
  ISK_HIP(hipMemcpyAsync(out, w->ds_out + index * S2, S2 * 4, hipMemcpyDeviceToHost,
                         w->ctx->stream));
  ISK_HIP(hipStreamSynchronize(w->ctx->stream));
  for (long long i = 0; i < S2; ++i) in[i] = ws_bf2f(h[i]);
  return ISKRA_OK;
}

/* phi at the context's interior nodes <- network prediction from its rho */
int iskra_ws_predict(iskra_ws *w) {
  WRC(ws_check(w));
  WRC(ws_check_grid(w));
  iskra_ctx *c = w->ctx;
  hipEvent_t ev = nullptr;
  WRC(isk_prof_begin(c, &ev));
  double fscale;
  WRC(ws_rhs_scale(w, &fscale));
  const long long S2 = (long long)w->S * w->S;
  hipLaunchKernelGGL(k_ws_rhs_store, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, c->stream,
                     (const double *)c->rho, (const double *)nullptr, c->g.nx, fscale,
                     (const double *)w->scal, (uint16_t *)nullptr, w->A0.a, (float *)nullptr);
  ISK_CHECK_LAUNCH();
  WRC(ws_forward(w, 1));
  hipLaunchKernelGGL(k_ws_phi_out, dim3(ws_grid(S2)), dim3(EW_BLOCK), 0, c->stream,
                     (const float *)w->out, c->phi, c->g.nx, w->gain, (const double *)w->scal);
  ISK_CHECK_LAUNCH();
  WRC(isk_prof_end(c, ev, ISKRA_K_WARMSTART, 0));
  return ISKRA_OK;
}

} /* extern "C" */
