// Per-DOF MLP initial guess for transient solves: inference and training kernels.
//
// Network: x in R^4 -> 128 -> 128 -> 128 -> 1 with ReLU, weights stored in bf16,
// every sum accumulated in fp32.  The layers run on MFMA (the two 128x128 ones
// on v_mfma_f32_16x16x32_bf16) in a transposed formulation: a wave holds the
// activations of 32 or 64 rows (DOF samples) as the B operand (K = input feature,
// N = row) and the weight tile as the A operand (M = output feature), so two
// 16x16 fp32 result tiles are, lane for lane, the B operand of a K-block of the
// next layer: activations never leave registers between layers.
//
// Training (one Adam step on a batch of B samples, loss 0.5/B sum (y-t)^2):
//   k_mlp_fwd<1>   forward, stores a1..a3 (bf16)
//   k_mlp_bwd      dz3 = (d4*W4) o [a3>0], dz2 = (W3^T dz3) o [a2>0], dz1 = (W2^T dz2) o [a1>0]
//                  (dz rounded to bf16: they are MFMA operands and are stored)
//   k_mlp_wgrad    gW2 = dz2^T a1, gW3 = dz3^T a2 on MFMA, per-block partials (K = rows)
//   k_mlp_small    gW1, b1..b3, gW4, b4 and the loss, per-block partials (VALU)
//   k_mlp_adam     fixed-order sum of partials, Adam update, bf16 mirror of the weights
// Every reduction has a fixed order, so results are bitwise repeatable.
// This component has no counterpart in the reference (it feeds the initial
// guess of the Oseen/implicit-Euler step, opencmp/models/ins.py:323-359).
#include "internal.h"

#include <algorithm>
#include <cmath>

namespace ocmp {
namespace {

constexpr int H = OCMP_MLP_HIDDEN, NIN = 4;
constexpr int OW1 = 0, OB1 = OW1 + H * NIN, OW2 = OB1 + H, OB2 = OW2 + H * H, OW3 = OB2 + H, OB3 = OW3 + H * H,
              OW4 = OB3 + H, OB4 = OW4 + H, NP = OB4 + 1;
static_assert(NP == OCMP_MLP_NPARAM, "parameter layout");
constexpr int LDW = H + 8;       // padded LDS row of a 128x128 bf16 weight tile (272 B: 16-byte aligned)
constexpr int ROWS_BLK = 128;    // batches are padded to this many rows
constexpr int CH = 64;           // rows per staged chunk of the weight-gradient kernel
constexpr int LDC = CH + 8;      // padded LDS row (144 B)
constexpr int NSMALL = H * NIN + 4 * H + 2;  // gW1, gb1, gb2, gb3, gW4, gb4, loss
constexpr int MAXSEG = OCMP_MLP_MAXSEG;

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 b4 __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16;

__device__ __forceinline__ u16 f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((unsigned)h << 16); }

struct SegArgs {
  int nseg;
  int64_t off[MAXSEG + 1];
  float s[MAXSEG], U[MAXSEG];
};

struct GuessArgs {
  const double *u0, *u1, *u2, *u3;
  double *out;
  int base;  // 1: the network predicts the correction to the linear extrapolation 2 u0 - u1
};

__device__ __forceinline__ int seg_of(const SegArgs &sg, int64_t i) {
  int k = 0;
  while (k + 1 < sg.nseg && i >= sg.off[k + 1]) ++k;
  return k;
}

// features of one DOF from its last four states: scaled increments and the scaled state
__device__ __forceinline__ float4 features(double u0, double u1, double u2, double u3, float s, float U) {
  const double is = 1.0 / (double)s;
  return make_float4((float)((u0 - u1) * is), (float)((u1 - u2) * is), (float)((u2 - u3) * is),
                     (float)(u0 / (double)U));
}

// The K index of a 32-wide block of v_mfma_f32_16x16x32_bf16 is dealt so that a layer's result tiles are
// the next layer's B operand without a move: slot 8 g + j of K-block kb holds feature
// 32 kb + 4 g + j (j < 4: what lane group g has of result tile 2 kb) or 32 kb + 16 + 4 g + j - 4 (tile
// 2 kb + 1). The weights lie in LDS in slot order, one 16-byte read per A operand.
__device__ __forceinline__ b8 pair8(b4 lo, b4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }

// a 128x128 bf16 weight (row-major [out][in]) into LDS rows [out][slot of in]
__device__ void stage_w(u16 *lds, const u16 *__restrict__ w) {
  for (int e = threadIdx.x; e < H * 16; e += blockDim.x) {
    const int o = e / 16, q = e % 16, f = 32 * (q / 4) + 4 * (q % 4);
    const b4 lo = *(const b4 *)(w + o * H + f), hi = *(const b4 *)(w + o * H + f + 16);
    *(b8 *)(lds + o * LDW + 8 * q) = pair8(lo, hi);
  }
}

// its transpose into LDS rows [in][slot of out]; a wave reads along the rows of w
__device__ void stage_wt(u16 *lds, const u16 *__restrict__ w) {
  for (int e = threadIdx.x; e < H * 16; e += blockDim.x) {
    const int i = e % H, q = e / H, f = 32 * (q / 4) + 4 * (q % 4);
    union {
      u16 u[8];
      b8 v;
    } t;
#pragma unroll
    for (int j = 0; j < 8; ++j) t.u[j] = w[(f + (j < 4 ? j : 12 + j)) * H + i];
    *(b8 *)(lds + i * LDW + 8 * q) = t.v;
  }
}

// acc[h][nt] += W[16 (2 mp + h) .., :] * act[:][nt]: two result tiles, the ones of K-block mp of the next layer
template <int NT>
__device__ __forceinline__ void dense_mfma(const u16 *sW, const b8 (&act)[4][NT], int mp, f4 (&acc)[2][NT], int r,
                                           int g) {
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const b8 a = *(const b8 *)(sW + (32 * mp + 16 * h + r) * LDW + 32 * kb + 8 * g);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[h][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, act[kb][nt], acc[h][nt], 0, 0, 0);
    }
}

// (the median with 0 and the largest float, which rounds to bf16 infinity like what lies above it, is one
// instruction and 0 for a NaN, as is fmaxf(v, 0), which costs another one to make v canonical first)
__device__ __forceinline__ b4 relu_bf(f4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_fmed3f(v[i], 0.f, 3.402823466e38f);
  return __builtin_convertvector(v, b4);
}

// MODE 0: Y = f(X); MODE 1: same and store a1..a3;
// MODE 2: out = u0 + base * (u0 - u1) + s * f(features(u0..u3))
// Bound by the matrix pipe (65.5 kFLOP of bf16 a row) and by the roundings between layers, which a SIMD's two
// waves overlap only in part. A wave carries 16 NT rows: every weight read from LDS serves NT products. Lane l
// loads, scales and writes row l of the wave's rows (one feature evaluation a row); layer 1 is
// v_mfma_f32_16x16x4_f32 on the FP32 features, layer 4 one more bf16 tile whose rows 0, 4, 8 and 12 are all
// W4, so that every lane group ends up with every row's result. The guess of 1,594,712 rows: 417 -> 113 us
// (0.92 PFLOP/s; 16x16x16 tiles of 32 rows, layers 1 and 4 and the rounding in scalar code before).
template <int MODE, int NT>
__global__ __launch_bounds__(256, 2) void k_mlp_fwd(const u16 *__restrict__ pb, int64_t n, int64_t npad,
                                                    const float4 *__restrict__ X, float *__restrict__ Y,
                                                    u16 *__restrict__ act, SegArgs sg, GuessArgs ga) {
  __shared__ alignas(16) u16 sW2[H * LDW], sW3[H * LDW], sW4[H];
  __shared__ alignas(16) float sB1[H], sB2[H], sB3[H];
  constexpr int WR = 16 * NT;
  __shared__ alignas(16) float sx[4][WR * NIN];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  stage_w(sW2, pb + OW2);
  stage_w(sW3, pb + OW3);
  for (int e = threadIdx.x; e < H; e += blockDim.x) {
    sB1[e] = bf2f(pb[OB1 + e]);
    sB2[e] = bf2f(pb[OB2 + e]);
    sB3[e] = bf2f(pb[OB3 + e]);
    const int j = e % 8;
    sW4[e] = pb[OW4 + e / 32 * 32 + (e % 32) / 8 * 4 + (j < 4 ? j : 12 + j)];
  }
  const float b4v = bf2f(pb[OB4]);
  float w1[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) w1[m] = bf2f(pb[OW1 + (16 * m + r) * NIN + g]);
  __syncthreads();

  const int64_t step = (int64_t)gridDim.x * 4 * WR;
  int64_t rb = ((int64_t)blockIdx.x * 4 + wv) * WR;
  double u[4] = {0.0, 0.0, 0.0, 0.0};
  float4 xn = make_float4(0.f, 0.f, 0.f, 0.f);
  auto load = [&](int64_t base) {
    const int64_t row = base + lane;
    if (lane < WR && row < n) {
      if (MODE == 2) {
        u[0] = ga.u0[row];
        u[1] = ga.u1[row];
        u[2] = ga.u2[row];
        u[3] = ga.u3[row];
      } else {
        xn = X[row];
      }
    } else {
      xn = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  load(rb);
  for (; rb < npad; rb += step) {
    asm volatile("" ::: "memory");  // the weights are read from LDS each time, not held (and spilled) across rows
    const int64_t row = rb + lane;
    const bool have = lane < WR && row < n;
    float4 x = xn;
    float su = 1.f;
    const double u0 = u[0], u1 = u[1];
    if (MODE == 2) {
      x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (have) {
        const int k = seg_of(sg, row);
        su = sg.s[k];
        x = features(u0, u1, u[2], u[3], sg.s[k], sg.U[k]);
      }
    }
    load(rb + step);  // the next rows, under way meanwhile
    b8 in[4][NT], out[4][NT];
    // layer 1 (4 -> 128)
    if (lane < WR) *(float4 *)(sx[wv] + lane * NIN) = x;  // turned over within the wave
    __builtin_amdgcn_wave_barrier();
    float xb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) xb[nt] = sx[wv][(16 * nt + r) * NIN + g];
#pragma unroll
    for (int mp = 0; mp < 4; ++mp) {
      f4 z[2][NT];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f4 b = *(const f4 *)(sB1 + 32 * mp + 16 * h + 4 * g);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          z[h][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[2 * mp + h], xb[nt], b, 0, 0, 0);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) in[mp][nt] = pair8(relu_bf(z[0][nt]), relu_bf(z[1][nt]));
    }
    auto store = [&](int L, const b8 (&v)[4][NT]) {
      if (MODE != 1) return;
#pragma unroll
      for (int mp = 0; mp < 4; ++mp)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          u16 *q = act + (size_t)L * npad * H + (size_t)(rb + 16 * nt + r) * H + 32 * mp + 4 * g;
          *(b4 *)q = __builtin_shufflevector(v[mp][nt], v[mp][nt], 0, 1, 2, 3);
          *(b4 *)(q + 16) = __builtin_shufflevector(v[mp][nt], v[mp][nt], 4, 5, 6, 7);
        }
    };
    auto layer = [&](const u16 *sW, const float *sB, const b8 (&vi)[4][NT], b8 (&vo)[4][NT]) {
      f4 acc[2][2][NT];
#pragma unroll
      for (int mp = 0; mp < 5; ++mp) {  // the tiles of mp are multiplied while those of mp - 1 are rounded
        if (mp < 4) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f4 b = *(const f4 *)(sB + 32 * mp + 16 * h + 4 * g);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mp & 1][h][nt] = b;
          }
          dense_mfma<NT>(sW, vi, mp, acc[mp & 1], r, g);
        }
        if (mp > 0)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            vo[mp - 1][nt] = pair8(relu_bf(acc[(mp - 1) & 1][0][nt]), relu_bf(acc[(mp - 1) & 1][1][nt]));
      }
    };
    store(0, in);
    layer(sW2, sB2, in, out);
    store(1, out);
    layer(sW3, sB3, out, in);
    store(2, in);
    // layer 4 (128 -> 1)
    f4 y[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) y[nt] = f4{b4v, b4v, b4v, b4v};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      b8 a = *(const b8 *)(sW4 + 32 * kb + 8 * g);
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = (r & 3) == 0 ? a[j] : (__bf16)0.f;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) y[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, in[kb][nt], y[nt], 0, 0, 0);
    }
    float yr = y[0].x;
#pragma unroll
    for (int nt = 1; nt < NT; ++nt) yr = g == nt ? y[nt].x : yr;
    if (have) {
      if (MODE == 2)
        ga.out[row] = u0 + (double)ga.base * (u0 - u1) + (double)su * (double)yr;
      else
        Y[row] = yr;
    }
  }
}

// the entries of v where the activation a of the same features is positive, rounded; 0 elsewhere
__device__ __forceinline__ b4 masked_bf(f4 v, b4 a) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (float)a[i] > 0.f ? v[i] : 0.f;
  return __builtin_convertvector(v, b4);
}

// backward through layers 4..1 for 32 rows per wave; writes dz1..dz3 (bf16) and d4 = dL/dy
// Eight waves share a staging of the two transposed weights, which a batch of 65,536 otherwise pays for
// every 128 rows: 54 -> 27 us.
constexpr int BWD_T = 512, BWD_ROWS = BWD_T / 64 * 32;
__global__ __launch_bounds__(BWD_T) void k_mlp_bwd(const u16 *__restrict__ pb, int64_t n, int64_t npad,
                                                   const float *__restrict__ Y, const float *__restrict__ T,
                                                   float invB, const u16 *__restrict__ act, u16 *__restrict__ dz,
                                                   float *__restrict__ d4) {
  __shared__ alignas(16) u16 sW2T[H * LDW], sW3T[H * LDW];
  __shared__ alignas(16) float sW4[H];
  stage_wt(sW2T, pb + OW2);
  stage_wt(sW3T, pb + OW3);
  for (int e = threadIdx.x; e < H; e += blockDim.x) sW4[e] = bf2f(pb[OW4 + e]);
  __syncthreads();

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const size_t LS = (size_t)npad * H;
  for (int64_t rb = ((int64_t)blockIdx.x * (BWD_T / 64) + wv) * 32; rb < npad; rb += (int64_t)gridDim.x * BWD_ROWS) {
    asm volatile("" ::: "memory");  // as in the forward pass
    b8 d_[4][2], e_[4][2];
    // dz3 = (d4 * W4) o [a3 > 0]
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int64_t row = rb + 16 * nt + r;
      const float d = row < n ? (Y[row] - T[row]) * invB : 0.f;
      if (g == 0) d4[row] = d;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        b4 v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int o = 32 * kb + 16 * h + 4 * g;
          const size_t at = 2 * LS + (size_t)row * H + o;
          v[h] = masked_bf(*(const f4 *)(sW4 + o) * d, *(const b4 *)(act + at));
          *(b4 *)(dz + at) = v[h];
        }
        d_[kb][nt] = pair8(v[0], v[1]);
      }
    }
    // dz2 = (W3^T dz3) o [a2 > 0], then dz1 = (W2^T dz2) o [a1 > 0]
    auto layer = [&](int L, const u16 *sWT, const b8 (&vi)[4][2], b8 (&vo)[4][2]) {
      b4 am[4][2][2];
#pragma unroll
      for (int mp = 0; mp < 4; ++mp)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            am[mp][nt][h] = *(const b4 *)(act + (size_t)L * LS + (size_t)(rb + 16 * nt + r) * H + 32 * mp + 16 * h +
                                          4 * g);
#pragma unroll
      for (int mp = 0; mp < 4; ++mp) {
        f4 acc[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[h][0] = acc[h][1] = f4{0.f, 0.f, 0.f, 0.f};
        dense_mfma<2>(sWT, vi, mp, acc, r, g);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          b4 v[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            v[h] = masked_bf(acc[h][nt], am[mp][nt][h]);
            *(b4 *)(dz + (size_t)L * LS + (size_t)(rb + 16 * nt + r) * H + 32 * mp + 16 * h + 4 * g) = v[h];
          }
          vo[mp][nt] = pair8(v[0], v[1]);
        }
      }
    };
    layer(1, sW3T, d_, e_);
    layer(0, sW2T, e_, d_);
  }
}

// gW_{L} = dz_L^T a_{L-1} for the two 128x128 layers (blockIdx.y = 0: W2, 1: W3); K = rows.
// Block b sums rows [b*rpb, (b+1)*rpb); wave w owns output rows 32w..32w+31. A thread turns 8 rows by 4
// features of each operand in registers, so that LDS is written 16 bytes at a time, and the next chunk's
// loads are under way while this one is multiplied. 65,536 rows: 31 -> 18 us.
__global__ __launch_bounds__(256) void k_mlp_wgrad(int64_t npad, int64_t rpb, const u16 *__restrict__ act,
                                                   const u16 *__restrict__ dz, float *__restrict__ part) {
  __shared__ alignas(16) u16 sD[H * LDC], sA[H * LDC];
  static_assert(CH == 64 && H == 128, "one unit of 8 rows by 4 features per thread");
  const int L = blockIdx.y;
  const size_t LS = (size_t)npad * H;
  const u16 *D = dz + (size_t)(L + 1) * LS;
  const u16 *A = act + (size_t)L * LS;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int fq = (threadIdx.x & 31) * 4, rq = (threadIdx.x >> 5) * 8;
  f4 acc[2][8];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int nn = 0; nn < 8; ++nn) acc[mi][nn] = f4{0.f, 0.f, 0.f, 0.f};
  const int64_t r0 = (int64_t)blockIdx.x * rpb, r1 = r0 + rpb < npad ? r0 + rpb : npad;
  b4 dv[8], av[8];
  auto load = [&](int64_t c0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      dv[i] = *(const b4 *)(D + (size_t)(c0 + rq + i) * H + fq);
      av[i] = *(const b4 *)(A + (size_t)(c0 + rq + i) * H + fq);
    }
  };
  if (r0 < r1) load(r0);
  for (int64_t c0 = r0; c0 < r1; c0 += CH) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      b8 d, a;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        d[i] = dv[i][c];
        a[i] = av[i][c];
      }
      *(b8 *)(sD + (fq + c) * LDC + rq) = d;
      *(b8 *)(sA + (fq + c) * LDC + rq) = a;
    }
    __syncthreads();
    if (c0 + CH < r1) load(c0 + CH);
#pragma unroll
    for (int ks = 0; ks < CH / 32; ++ks) {
      b8 a[2];
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) a[mi] = *(const b8 *)(sD + (32 * wv + 16 * mi + r) * LDC + 32 * ks + 8 * g);
#pragma unroll
      for (int nn = 0; nn < 8; ++nn) {
        const b8 b = *(const b8 *)(sA + (16 * nn + r) * LDC + 32 * ks + 8 * g);
        acc[0][nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b, acc[0][nn], 0, 0, 0);
        acc[1][nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b, acc[1][nn], 0, 0, 0);
      }
    }
  }
  float *P = part + ((size_t)blockIdx.x * 2 + L) * H * H;
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int nn = 0; nn < 8; ++nn) {
      const int o = 32 * wv + 16 * mi + 4 * g, in = 16 * nn + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) P[(o + i) * H + in] = acc[mi][nn][i];
    }
}

// per-block partials of gW1 (dz1 x), gb1..gb3, gW4 (d4 a3), gb4 and sum (y-t)^2: a pass over dz1..dz3 and a3,
// bound by their bytes. A thread holds 8 features (16-byte loads) and every 16th row of the block
// (65,536 rows, 71 MB: 93 -> 18 us; one feature and every other row before).
__global__ __launch_bounds__(256) void k_mlp_small(int64_t n, int64_t npad, int64_t rpb,
                                                   const float4 *__restrict__ X, const float *__restrict__ Y,
                                                   const float *__restrict__ T, const float *__restrict__ d4,
                                                   const u16 *__restrict__ act, const u16 *__restrict__ dz,
                                                   float *__restrict__ part) {
  constexpr int NQ = 8 * 8;  // sums of a thread: w1[4], b1, b2, b3, w4 of 8 features
  __shared__ float sh[4][16][NQ + 1];
  __shared__ float sl[4][2];
  const size_t LS = (size_t)npad * H;
  const int fg = threadIdx.x & 15, rg = threadIdx.x >> 4, wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float s[8][8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int j = 0; j < 8; ++j) s[c][j] = 0.f;
  float b4s = 0.f, ls = 0.f;
  const int64_t r0 = (int64_t)blockIdx.x * rpb, r1 = r0 + rpb < n ? r0 + rpb : n;
#pragma unroll 2
  for (int64_t row = r0 + rg; row < r1; row += 16) {
    const size_t at = (size_t)row * H + 8 * fg;
    const float4 x = X[row];
    const b8 z1 = *(const b8 *)(dz + at), z2 = *(const b8 *)(dz + LS + at), z3 = *(const b8 *)(dz + 2 * LS + at),
             a3 = *(const b8 *)(act + 2 * LS + at);
    const float d = d4[row];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float z = (float)z1[j];
      s[0][j] += z * x.x;
      s[1][j] += z * x.y;
      s[2][j] += z * x.z;
      s[3][j] += z * x.w;
      s[4][j] += z;
      s[5][j] += (float)z2[j];
      s[6][j] += (float)z3[j];
      s[7][j] += d * (float)a3[j];
    }
    if (fg == 0) {
      b4s += d;
      const float e = Y[row] - T[row];
      ls += e * e;
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = s[c][j];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (lane < 16) sh[wv][fg][c * 8 + j] = v;
    }
  b4s += __shfl_xor(b4s, 16);
  b4s += __shfl_xor(b4s, 32);
  ls += __shfl_xor(ls, 16);
  ls += __shfl_xor(ls, 32);
  if (lane == 0) {
    sl[wv][0] = b4s;
    sl[wv][1] = ls;
  }
  __syncthreads();
  float *P = part + (size_t)blockIdx.x * NSMALL;
  for (int e = threadIdx.x; e < 8 * H; e += blockDim.x) {
    // e: gW1 as [o][c], then gb1, gb2, gb3, gW4
    const int c = e < 4 * H ? e % 4 : e / H, o = e < 4 * H ? e / 4 : e % H;
    const int f = o / 8, k = c * 8 + o % 8;
    P[e] = (sh[0][f][k] + sh[1][f][k]) + (sh[2][f][k] + sh[3][f][k]);
  }
  if (threadIdx.x < 2)
    P[8 * H + threadIdx.x] = (sl[0][threadIdx.x] + sl[1][threadIdx.x]) + (sl[2][threadIdx.x] + sl[3][threadIdx.x]);
}

// fixed-order sum of the partials into the gradient, optional Adam step and bf16 mirror. A block takes 64
// parameters and its 8 waves every 8th partial of them (one thread a parameter chained 128 loads on an
// eighth of the chip: 42 us, now 7).
constexpr int ADAM_P = 64, ADAM_S = 8;
__global__ __launch_bounds__(ADAM_P *ADAM_S) void k_mlp_adam(int nbw, int nbs, const float *__restrict__ pw,
                                                  const float *__restrict__ ps, float *__restrict__ grad, float *p,
                                                  float *m, float *v, u16 *pb, float lr, float c1, float c2,
                                                  int update, double *loss, double half_invB) {
  __shared__ float sh[ADAM_S][ADAM_P];
  __shared__ double shl[ADAM_S];
  const int jl = threadIdx.x % ADAM_P, q = threadIdx.x / ADAM_P;
  const int j = blockIdx.x * ADAM_P + jl;
  float s = 0.f;
  if (j < NP) {
    const float *src;
    int nb, ld;
    if (j >= OW2 && j < OB2) {
      src = pw + (j - OW2), nb = nbw, ld = 2 * H * H;
    } else if (j >= OW3 && j < OB3) {
      src = pw + H * H + (j - OW3), nb = nbw, ld = 2 * H * H;
    } else {
      int k;
      if (j < OB1) k = j - OW1;
      else if (j < OW2) k = H * NIN + (j - OB1);
      else if (j < OW3) k = H * NIN + H + (j - OB2);
      else if (j < OW4) k = H * NIN + 2 * H + (j - OB3);
      else if (j < OB4) k = H * NIN + 3 * H + (j - OW4);
      else k = H * NIN + 4 * H;
      src = ps + k, nb = nbs, ld = NSMALL;
    }
#pragma unroll 8
    for (int b = q; b < nb; b += ADAM_S) s += src[(size_t)b * ld];
  } else if (j == NP) {  // loss
    double l = 0.0;
#pragma unroll 8
    for (int b = q; b < nbs; b += ADAM_S) l += (double)ps[(size_t)b * NSMALL + NSMALL - 1];
    shl[q] = l;
  }
  sh[q][jl] = s;
  __syncthreads();
  if (q != 0 || j > NP) return;
  if (j == NP) {
    double l = 0.0;
    for (int i = 0; i < ADAM_S; ++i) l += shl[i];
    *loss = l * half_invB;
    return;
  }
  float gsum = 0.f;
#pragma unroll
  for (int i = 0; i < ADAM_S; ++i) gsum += sh[i][jl];
  if (grad) grad[j] = gsum;
  if (update) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mj = b1 * m[j] + (1.f - b1) * gsum;
    const float vj = b2 * v[j] + (1.f - b2) * gsum * gsum;
    m[j] = mj;
    v[j] = vj;
    const float pj = p[j] - lr * (mj * c1) / (sqrtf(vj * c2) + eps);
    p[j] = pj;
    pb[j] = f2bf(pj);
  }
}

__global__ void k_mlp_mirror(const float *__restrict__ p, u16 *__restrict__ pb) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < NP) pb[j] = f2bf(p[j]);
}

__device__ __forceinline__ uint64_t splitmix(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// random (snapshot j, dof i) samples: X = features of u^j..u^{j-3},
// T = (u^{j+1} - u^j - base (u^j - u^{j-1})) / s
__global__ void k_mlp_sample(const double *__restrict__ snap, int nsnap, int64_t ld, int64_t n, SegArgs sg,
                             uint64_t seed, int batch, int base, float4 *__restrict__ X,
                             float *__restrict__ T) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  const uint64_t h1 = splitmix(seed * 0x2545F4914F6CDD1Dull + (uint64_t)b);
  const uint64_t h2 = splitmix(h1);
  const int j = 3 + (int)(h1 % (uint64_t)(nsnap - 4));
  const int64_t i = (int64_t)(h2 % (uint64_t)n);
  const int k = seg_of(sg, i);
  const double u0 = snap[(size_t)j * ld + i], u1 = snap[(size_t)(j - 1) * ld + i];
  X[b] = features(u0, u1, snap[(size_t)(j - 2) * ld + i], snap[(size_t)(j - 3) * ld + i], sg.s[k], sg.U[k]);
  T[b] = (float)((snap[(size_t)(j + 1) * ld + i] - u0 - (double)base * (u0 - u1)) / (double)sg.s[k]);
}

// per (segment, block) sums of squared increments and squared values over the snapshots
__global__ __launch_bounds__(256) void k_mlp_scales(const double *__restrict__ snap, int nsnap, int64_t ld,
                                                    SegArgs sg, double *__restrict__ part) {
  __shared__ double sh[2][256];
  const int k = blockIdx.y;
  const int64_t o = sg.off[k], len = sg.off[k + 1] - sg.off[k];
  const int64_t tot = (int64_t)(nsnap - 1) * len;
  double si = 0.0, sv = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
    const int j = 1 + (int)(q / len);
    const int64_t i = o + q % len;
    const double u = snap[(size_t)j * ld + i], d = u - snap[(size_t)(j - 1) * ld + i];
    si += d * d;
    sv += u * u;
  }
  sh[0][threadIdx.x] = si;
  sh[1][threadIdx.x] = sv;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
      sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[((size_t)k * gridDim.x + blockIdx.x) * 2 + 0] = sh[0][0];
    part[((size_t)k * gridDim.x + blockIdx.x) * 2 + 1] = sh[1][0];
  }
}

constexpr int FWD_GRID_MAX = 512;  // two blocks of 256 threads a CU (LDS and registers allow no more)
constexpr int WG_BLOCKS_MAX = 128;
constexpr int SMALL_BLOCKS_MAX = 256, SMALL_ROWS_MIN = 64;

// 64 rows a wave where that leaves every SIMD two waves (from 131,072 rows), 32 below. Forward with 64 and 32
// rows: 1,000 rows 7.6 and 6.4 us, 30,000 8.2 and 7.0, 131,072 12.2 and 13.2, 450,000 30.2 and 33.4,
// 1,594,712 92.6 and 101.8
constexpr int64_t FWD_WIDE = (int64_t)FWD_GRID_MAX * 4 * 64;
template <int MODE>
void launch_fwd(hipStream_t st, const u16 *pb, int64_t n, int64_t npad, const float4 *X, float *Y, u16 *act,
                const SegArgs &sg, const GuessArgs &ga) {
  const bool wide = npad >= FWD_WIDE;
  const int64_t rows = wide ? 256 : 128;
  const unsigned grid = (unsigned)std::min<int64_t>((npad + rows - 1) / rows, FWD_GRID_MAX);
  if (wide)
    k_mlp_fwd<MODE, 4><<<grid, 256, 0, st>>>(pb, n, npad, X, Y, act, sg, ga);
  else
    k_mlp_fwd<MODE, 2><<<grid, 256, 0, st>>>(pb, n, npad, X, Y, act, sg, ga);
}

}  // namespace

struct Mlp {
  Ctx *ctx;
  int64_t max_batch = 0, bpad = 0;
  DBuf<float> p, m, v, grad, partw, parts, y, d4;
  DBuf<u16> pb, act, dz;
  DBuf<double> loss, spart;
  int64_t step = 0;
  SegArgs sg{};
  int base = 0;  // guess relative to u0 (0) or to the linear extrapolation 2 u0 - u1 (1)
};

static void mlp_alloc(Mlp *M, int64_t max_batch) {
  M->max_batch = max_batch;
  M->bpad = (max_batch + ROWS_BLK - 1) / ROWS_BLK * ROWS_BLK;
  M->p.alloc(NP);
  M->m.alloc(NP);
  M->v.alloc(NP);
  M->grad.alloc(NP);
  M->pb.alloc(NP + 8);
  M->loss.alloc(1);
  M->act.alloc((size_t)3 * M->bpad * H);
  M->dz.alloc((size_t)3 * M->bpad * H);
  M->y.alloc(M->bpad);
  M->d4.alloc(M->bpad);
  M->partw.alloc((size_t)WG_BLOCKS_MAX * 2 * H * H);
  M->parts.alloc((size_t)SMALL_BLOCKS_MAX * NSMALL);
  M->sg.nseg = 1;
  M->sg.off[0] = 0;
  M->sg.off[1] = INT64_MAX;
  M->sg.s[0] = M->sg.U[0] = 1.f;
}

Mlp *mlp_create(Ctx *ctx, const float *params, int64_t max_batch) {
  OCMP_REQUIRE(max_batch >= 1 && max_batch <= ((int64_t)1 << 26), "mlp: max_batch out of range [1, 2^26]");
  Mlp *M = new Mlp();
  M->ctx = ctx;
  try {
    mlp_alloc(M, max_batch);
    mlp_set_params(M, params);
  } catch (...) {
    delete M;
    throw;
  }
  return M;
}

void mlp_destroy(Mlp *M) { delete M; }

void mlp_set_params(Mlp *M, const float *params) {
  hipStream_t s = M->ctx->stream;
  OCMP_REQUIRE(params, "mlp: null parameter array");
  OCMP_HIP(hipMemcpyAsync(M->p.p, params, NP * sizeof(float), hipMemcpyHostToDevice, s));
  OCMP_HIP(hipMemsetAsync(M->m.p, 0, NP * sizeof(float), s));
  OCMP_HIP(hipMemsetAsync(M->v.p, 0, NP * sizeof(float), s));
  k_mlp_mirror<<<(NP + 255) / 256, 256, 0, s>>>(M->p.p, M->pb.p);
  OCMP_HIP(hipGetLastError());
  OCMP_HIP(hipStreamSynchronize(s));
  M->step = 0;
}

void mlp_get_params(Mlp *M, float *params) {
  OCMP_REQUIRE(params, "mlp: null output array");
  OCMP_HIP(hipMemcpyAsync(params, M->p.p, NP * sizeof(float), hipMemcpyDeviceToHost, M->ctx->stream));
  OCMP_HIP(hipStreamSynchronize(M->ctx->stream));
}

static void set_segments(SegArgs &sg, int nseg, const int64_t *off) {
  OCMP_REQUIRE(nseg >= 1 && nseg <= MAXSEG, "mlp: nseg out of range [1, OCMP_MLP_MAXSEG]");
  OCMP_REQUIRE(off, "mlp: null segment offsets");
  OCMP_REQUIRE(off[0] == 0, "mlp: segment offsets must start at 0");
  for (int k = 0; k < nseg; ++k) OCMP_REQUIRE(off[k + 1] > off[k], "mlp: segment offsets must increase");
  sg.nseg = nseg;
  for (int k = 0; k <= nseg; ++k) sg.off[k] = off[k];
}

void mlp_set_scales(Mlp *M, int nseg, const int64_t *off, const double *s, const double *U) {
  set_segments(M->sg, nseg, off);
  for (int k = 0; k < nseg; ++k) {
    OCMP_REQUIRE(s[k] > 0 && U[k] > 0 && std::isfinite(s[k]) && std::isfinite(U[k]), "mlp: scales must be > 0");
    M->sg.s[k] = (float)s[k];
    M->sg.U[k] = (float)U[k];
  }
}

void mlp_get_scales(Mlp *M, int *nseg, int64_t *off, double *s, double *U) {
  *nseg = M->sg.nseg;
  for (int k = 0; k <= M->sg.nseg; ++k) off[k] = M->sg.off[k];
  for (int k = 0; k < M->sg.nseg; ++k) {
    s[k] = M->sg.s[k];
    U[k] = M->sg.U[k];
  }
}

void mlp_fit_scales(Mlp *M, const double *snap, int nsnap, int64_t ld, int nseg, const int64_t *off) {
  OCMP_REQUIRE(snap && nsnap >= 2, "mlp: need at least two snapshots");
  SegArgs sg{};
  set_segments(sg, nseg, off);
  OCMP_REQUIRE(off[nseg] <= ld, "mlp: segments exceed the snapshot stride");
  const int nb = 256;
  M->spart.alloc((size_t)nseg * nb * 2);
  hipStream_t st = M->ctx->stream;
  k_mlp_scales<<<dim3(nb, nseg), 256, 0, st>>>(snap, nsnap, ld, sg, M->spart.p);
  OCMP_HIP(hipGetLastError());
  std::vector<double> h((size_t)nseg * nb * 2);
  OCMP_HIP(hipMemcpyAsync(h.data(), M->spart.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  OCMP_HIP(hipStreamSynchronize(st));
  std::vector<double> s(nseg), U(nseg);
  for (int k = 0; k < nseg; ++k) {
    double si = 0.0, sv = 0.0;
    for (int b = 0; b < nb; ++b) {
      si += h[((size_t)k * nb + b) * 2];
      sv += h[((size_t)k * nb + b) * 2 + 1];
    }
    const double cnt = (double)(nsnap - 1) * (double)(off[k + 1] - off[k]);
    s[k] = std::sqrt(si / cnt);
    U[k] = std::sqrt(sv / cnt);
    if (!(s[k] > 1e-300)) s[k] = 1.0;  // a component that does not move: features stay 0
    if (!(U[k] > 1e-300)) U[k] = 1.0;
  }
  mlp_set_scales(M, nseg, off, s.data(), U.data());
}

void mlp_sample(Mlp *M, const double *snap, int nsnap, int64_t ld, int64_t n, uint64_t seed, int64_t batch,
                float *X, float *T) {
  OCMP_REQUIRE(snap && X && T, "mlp: null buffer");
  OCMP_REQUIRE(nsnap >= 5, "mlp: sampling needs at least five snapshots");
  OCMP_REQUIRE(n >= 1 && n <= ld, "mlp: n out of range");
  OCMP_REQUIRE(M->sg.off[M->sg.nseg] >= n || M->sg.off[M->sg.nseg] == INT64_MAX,
               "mlp: scale segments do not cover the dofs");
  OCMP_REQUIRE(batch >= 1 && batch <= ((int64_t)1 << 30), "mlp: batch out of range");
  hipStream_t st = M->ctx->stream;
  k_mlp_sample<<<(unsigned)((batch + 255) / 256), 256, 0, st>>>(snap, nsnap, ld, n, M->sg, seed, (int)batch,
                                                               M->base, (float4 *)X, T);
  OCMP_HIP(hipGetLastError());
}

void mlp_forward(Mlp *M, int64_t n, const float *X, float *Y) {
  OCMP_REQUIRE(X && Y, "mlp: null buffer");
  OCMP_REQUIRE(n >= 1, "mlp: empty input");
  OCMP_REQUIRE(((uintptr_t)X & 15) == 0, "mlp: X must be 16-byte aligned (n x 4 float32)");
  const int64_t npad = (n + ROWS_BLK - 1) / ROWS_BLK * ROWS_BLK;
  Ctx *c = M->ctx;
  KTimer t(c, c->cls("mlp_forward"), (double)n * 20.0 + NP * 2.0);
  launch_fwd<0>(c->stream, M->pb.p, n, npad, (const float4 *)X, Y, nullptr, M->sg, GuessArgs{});
  OCMP_HIP(hipGetLastError());
}

void mlp_guess(Mlp *M, int64_t n, const double *u0, const double *u1, const double *u2, const double *u3,
               double *out) {
  OCMP_REQUIRE(u0 && u1 && u2 && u3 && out, "mlp: null history vector");
  OCMP_REQUIRE(n >= 1, "mlp: empty input");
  OCMP_REQUIRE(M->sg.off[M->sg.nseg] >= n || M->sg.off[M->sg.nseg] == INT64_MAX,
               "mlp: scale segments do not cover the dofs");
  const int64_t npad = (n + ROWS_BLK - 1) / ROWS_BLK * ROWS_BLK;
  Ctx *c = M->ctx;
  KTimer t(c, c->cls("mlp_guess"), (double)n * 40.0 + NP * 2.0);
  launch_fwd<2>(c->stream, M->pb.p, n, npad, nullptr, nullptr, nullptr, M->sg,
                GuessArgs{u0, u1, u2, u3, out, M->base});
  OCMP_HIP(hipGetLastError());
}

void mlp_set_base(Mlp *M, int base) {
  OCMP_REQUIRE(base == 0 || base == 1, "mlp: base must be 0 (previous state) or 1 (linear extrapolation)");
  M->base = base;
}

int mlp_get_base(const Mlp *M) { return M->base; }

// gradient of the batch loss (and optionally one Adam step); loss (device) written to M->loss
static void mlp_backprop(Mlp *M, int64_t n, const float *X, const float *T, float *grad, bool update, float lr) {
  OCMP_REQUIRE(X && T, "mlp: null buffer");
  OCMP_REQUIRE(n >= 1 && n <= M->max_batch, "mlp: batch larger than the max_batch given at creation");
  OCMP_REQUIRE(((uintptr_t)X & 15) == 0, "mlp: X must be 16-byte aligned (n x 4 float32)");
  Ctx *c = M->ctx;
  hipStream_t st = c->stream;
  const int64_t npad = (n + ROWS_BLK - 1) / ROWS_BLK * ROWS_BLK;
  const unsigned grid = (unsigned)std::min<int64_t>((npad + BWD_ROWS - 1) / BWD_ROWS, FWD_GRID_MAX);
  const float invB = 1.0f / (float)n;
  {
    KTimer t(c, c->cls("mlp_train_fwd"), (double)n * 20.0 + (double)npad * 3 * H * 2);
    launch_fwd<1>(st, M->pb.p, n, npad, (const float4 *)X, M->y.p, M->act.p, M->sg, GuessArgs{});
    OCMP_HIP(hipGetLastError());
  }
  {
    KTimer t(c, c->cls("mlp_train_bwd"), (double)npad * (8.0 + 6 * H * 2));
    k_mlp_bwd<<<grid, BWD_T, 0, st>>>(M->pb.p, n, npad, M->y.p, T, invB, M->act.p, M->dz.p, M->d4.p);
    OCMP_HIP(hipGetLastError());
  }
  // rows per weight-gradient block: a multiple of the staged chunk, at most WG_BLOCKS_MAX blocks
  int64_t rpb = (npad + WG_BLOCKS_MAX - 1) / WG_BLOCKS_MAX;
  rpb = (rpb + CH - 1) / CH * CH;
  const int nbw = (int)((npad + rpb - 1) / rpb);
  const int64_t rps = std::max<int64_t>((n + SMALL_BLOCKS_MAX - 1) / SMALL_BLOCKS_MAX, SMALL_ROWS_MIN);
  const int nbs = (int)((n + rps - 1) / rps);
  {
    KTimer t(c, c->cls("mlp_train_wgrad"), (double)npad * 4 * H * 2 + (double)nbw * 2 * H * H * 4);
    k_mlp_wgrad<<<dim3(nbw, 2), 256, 0, st>>>(npad, rpb, M->act.p, M->dz.p, M->partw.p);
    OCMP_HIP(hipGetLastError());
    k_mlp_small<<<nbs, 256, 0, st>>>(n, npad, rps, (const float4 *)X, M->y.p, T, M->d4.p, M->act.p, M->dz.p,
                                     M->parts.p);
    OCMP_HIP(hipGetLastError());
  }
  float c1 = 1.f, c2 = 1.f;
  if (update) {
    M->step += 1;
    c1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)M->step)));
    c2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)M->step)));
  }
  {
    KTimer t(c, c->cls("mlp_adam"), (double)nbw * 2 * H * H * 4 + (double)nbs * NSMALL * 4 + NP * 26.0);
    k_mlp_adam<<<(NP + 1 + ADAM_P - 1) / ADAM_P, ADAM_P * ADAM_S, 0, st>>>(nbw, nbs, M->partw.p, M->parts.p, grad ? grad : M->grad.p,
                                                     M->p.p, M->m.p, M->v.p, M->pb.p, lr, c1, c2, update ? 1 : 0,
                                                     M->loss.p, 0.5 / (double)n);
    OCMP_HIP(hipGetLastError());
  }
}

void mlp_grad(Mlp *M, int64_t n, const float *X, const float *T, float *grad, double *loss) {
  mlp_backprop(M, n, X, T, grad, false, 0.f);
  if (loss) {
    OCMP_HIP(hipMemcpyAsync(loss, M->loss.p, sizeof(double), hipMemcpyDeviceToHost, M->ctx->stream));
    OCMP_HIP(hipStreamSynchronize(M->ctx->stream));
  }
}

void mlp_train_step(Mlp *M, int64_t n, const float *X, const float *T, float lr, double *loss) {
  OCMP_REQUIRE(lr > 0.f && std::isfinite(lr), "mlp: learning rate must be > 0");
  mlp_backprop(M, n, X, T, nullptr, true, lr);
  if (loss) {
    OCMP_HIP(hipMemcpyAsync(loss, M->loss.p, sizeof(double), hipMemcpyDeviceToHost, M->ctx->stream));
    OCMP_HIP(hipStreamSynchronize(M->ctx->stream));
  }
}

}  // namespace ocmp
