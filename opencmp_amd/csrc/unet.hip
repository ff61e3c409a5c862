// Learned preconditioner correction: a 3-level U-net on the vertex grid of a
// structured (N^3 cubes x 6 tets) mesh, used inside flexible GMRES.
//
// The correction acts on the vertex dofs of four scalar blocks (the velocity
// components and the pressure of the diffuse-interface Stokes system): a vector
// v is restricted to a 4-channel grid (vertex id = grid index, x fastest), the
// network maps it to a 4-channel grid y, and y is added back onto the same
// vertex dofs. As a preconditioner, M v = D^{-1} v + E U(R v) (D the point-Jacobi
// diagonal). The network is trained on the GPU to minimise
// 0.5 ||v - A M v||^2 over vectors v from plain solves (self-supervised: only
// products with A are needed), by the kernels below and Adam.
//
// Layers (3x3x3 kernels, zero padding), bf16 weights and activations, fp32 sums:
//   a0 = relu(conv (x;  4 -> 8))        a1 = relu(conv2(a0; 8 -> 16))
//   a2 = relu(conv (a1; 16 -> 16))      a3 = relu(conv2(a2; 16 -> 32))
//   a4 = relu(conv (a3; 32 -> 32))      a5 = relu(tconv2(a4; 32 -> 16) + a2)
//   a6 = relu(tconv2(a5; 16 -> 8) + a0) y  = conv (a6; 8 -> 4)
// conv stride s: out[o,z] = b[o] + sum_{i,d} W[o,i,d] in[i, s z + d - 1]
// tconv stride 2: out[o,z] = b[o] + sum_{i,d} W[i,o,d] in[i,y] over 2y + d - 1 = z
// Weight-gradient reductions use fixed partitions and fixed-order sums: bitwise
// repeatable. No counterpart in the reference (its preconditioners are
// opencmp/models/base_model.py:365-383).
#include "internal.h"

#include <cmath>

namespace ocmp {
namespace {

typedef unsigned short u16;

__device__ __forceinline__ u16 f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((unsigned)h << 16); }

constexpr int NL = 8;          // layers
constexpr int NT = 256;

struct LayerDef {
  int cin, cout, stride, transposed, level_in, level_out;
};
// level 0: n0 = N+1, level 1: n1 = N/2+1, level 2: n2 = N/4+1
constexpr LayerDef LD[NL] = {{4, 8, 1, 0, 0, 0},   {8, 16, 2, 0, 0, 1},  {16, 16, 1, 0, 1, 1}, {16, 32, 2, 0, 1, 2},
                             {32, 32, 1, 0, 2, 2}, {32, 16, 2, 1, 2, 1}, {16, 8, 2, 1, 1, 0},  {8, 4, 1, 0, 0, 0}};

constexpr int layer_w(int l) { return LD[l].cin * LD[l].cout * 27; }
constexpr int layer_p(int l) { return layer_w(l) + LD[l].cout; }
constexpr int nparam() {
  int s = 0;
  for (int l = 0; l < NL; ++l) s += layer_p(l);
  return s;
}
constexpr int NP = nparam();
static_assert(NP == OCMP_UNET_NPARAM, "parameter layout");

int param_off(int l) {
  int s = 0;
  for (int k = 0; k < l; ++k) s += layer_p(k);
  return s;
}

// The convolutions' weights as FP32 copies of the bf16 ones in the order the matrix cores read them:
// [tap][input channel][output channel, padded to 16 with zeros], for the forward product (adj 0) and
// for its adjoint (adj 1: input and output channels swapped). Rebuilt when the parameters change.
constexpr int pad16(int c) { return (c + 15) / 16 * 16; }
constexpr int pk_in(int l, int adj) { return adj ? LD[l].cout : LD[l].cin; }
constexpr int pk_out(int l, int adj) { return adj ? LD[l].cin : LD[l].cout; }
constexpr int pk_size(int l, int adj) { return 27 * pk_in(l, adj) * pad16(pk_out(l, adj)); }
constexpr int pk_off(int l, int adj) {
  int s = 0;
  for (int k = 0; k < l; ++k) s += pk_size(k, 0) + pk_size(k, 1);
  return adj ? s + pk_size(l, 0) : s;
}
constexpr int NPACK = pk_off(NL - 1, 1) + pk_size(NL - 1, 1);

struct PackSeg {
  int off, in, out, w, si, so;  // w(o, i, k) = pb[w + (o so + i si) 27 + k]
};
struct PackTable {
  PackSeg s[2 * NL];
};

__global__ void k_pack_weights(PackTable T, const u16 *__restrict__ pb, float *__restrict__ wp) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= NPACK) return;
  int k = 0;
  while (k + 1 < 2 * NL && e >= T.s[k + 1].off) ++k;
  const PackSeg g = T.s[k];
  const int cop = pad16(g.out), r = e - g.off;
  const int o = r % cop, i = (r / cop) % g.in, tap = r / (cop * g.in);
  wp[e] = o < g.out ? bf2f(pb[g.w + (o * g.so + i * g.si) * 27 + tap]) : 0.f;
}

struct Conv {
  const void *in;
  int in_bf16, cin, nin;
  void *out;
  int out_bf16, cout, nout;
  const float *W;           // packed, [tap][cin][cop]
  int cop;
  const u16 *bias;          // may be null
  const void *skip;         // added before the activation, may be null
  int skip_bf16;
  const u16 *mask;          // multiply by [mask > 0] (backward), may be null
  int relu, stride, transposed;
};

__device__ __forceinline__ float ld_any(const void *p, int bf, size_t i) {
  return bf ? bf2f(((const u16 *)p)[i]) : ((const float *)p)[i];
}
__device__ __forceinline__ float ld_f(const u16 *p, int64_t i) { return bf2f(p[i]); }
__device__ __forceinline__ float ld_f(const float *p, int64_t i) { return p[i]; }

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One workgroup per 16 voxels x 16 output channels (blockIdx.y), as v_mfma_f32_16x16x4 over K = 27 taps
// x CIN input channels, the taps dealt to its four wavefronts and their sums added in LDS. FP32
// products of the same bf16 (forward) or fp32 (backward) operands as on the vector units. Lane l
// holds weight (channel l % 16, input l / 16) and input (input l / 16, voxel l % 16): both loads
// are runs of 16, and it receives channels 4 (l / 16) + r, r = 0..3, of voxel l % 16. What bounds the
// coarse levels is one wavefront's chain of dependent loads (9^3 voxels are 46 tiles): hence the split
// of the taps, and all of a wavefront's loads before its first product. 33^3 grid, all 23 products of two
// forwards and a gradient: 192 us (tap after tap 261; one thread per voxel and 8 channels, weights staged in
// LDS by every workgroup: 1745 us).
template <int CIN, typename TI>
__global__ __launch_bounds__(NT) void k_conv3(Conv c) {
  __shared__ float sh[4][256];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int64_t zout = (int64_t)c.nout * c.nout * c.nout;
  const int64_t zin = (int64_t)c.nin * c.nin * c.nin;
  const TI *__restrict__ in = (const TI *)c.in + (int64_t)lk * zin;
  const float *__restrict__ W = c.W + (int64_t)lk * c.cop + blockIdx.y * 16 + li;
  {
    const int64_t z = (int64_t)blockIdx.x * 16 + li;
    const int64_t zr = z < zout ? z : zout - 1;
    const int zx = (int)(zr % c.nout), zq = (int)(zr / c.nout), zy = zq % c.nout, zz = zq / c.nout;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // a wave's seven taps: all loads first, then the matrix instructions
    constexpr int NTAP = 7;
    float x[NTAP][CIN / 4], w[NTAP][CIN / 4];
    bool ok[NTAP], any[NTAP];
#pragma unroll
    for (int j = 0; j < NTAP; ++j) {
      const int k = wv + 4 * j;
      const int dz = k / 9, dy = (k / 3) % 3, dx = k % 3;
      int sx, sy, sz;
      bool in_ = z < zout && k < 27;
      if (!c.transposed) {
        sx = c.stride * zx + dx - 1;
        sy = c.stride * zy + dy - 1;
        sz = c.stride * zz + dz - 1;
      } else {
        const int tx = zx - dx + 1, ty = zy - dy + 1, tz = zz - dz + 1;
        if (c.stride == 2) {
          in_ = in_ && !((tx | ty | tz) & 1);
          sx = tx >> 1;
          sy = ty >> 1;
          sz = tz >> 1;
        } else {
          sx = tx;
          sy = ty;
          sz = tz;
        }
      }
      ok[j] = in_ && sx >= 0 && sy >= 0 && sz >= 0 && sx < c.nin && sy < c.nin && sz < c.nin;
      any[j] = __any(ok[j]);  // whole wavefront: the matrix instructions below run with all lanes
      const int64_t src = ok[j] ? ((int64_t)sz * c.nin + sy) * c.nin + sx : 0;
      if (any[j])
#pragma unroll
        for (int i = 0; i < CIN / 4; ++i) {
          x[j][i] = ld_f(in, (int64_t)(4 * i) * zin + src);
          w[j][i] = W[(int64_t)(k * CIN + 4 * i) * c.cop];
        }
    }
#pragma unroll
    for (int j = 0; j < NTAP; ++j)
      if (any[j])
#pragma unroll
        for (int i = 0; i < CIN / 4; ++i)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][i], ok[j] ? x[j][i] : 0.f, acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) sh[wv][r * 64 + lane] = acc[r];
  }
  __syncthreads();
  const int t = threadIdx.x;
  const int o = blockIdx.y * 16 + 4 * ((t & 63) >> 4) + (t >> 6);
  const int64_t z = (int64_t)blockIdx.x * 16 + (t & 15);
  if (o >= c.cout || z >= zout) return;
  float v = (sh[0][t] + sh[1][t]) + (sh[2][t] + sh[3][t]);
  const size_t at = (size_t)o * zout + z;
  if (c.bias) v += bf2f(c.bias[o]);
  if (c.skip) v += ld_any(c.skip, c.skip_bf16, at);
  if (c.relu) v = fmaxf(v, 0.f);
  if (c.mask && !(bf2f(c.mask[at]) > 0.f)) v = 0.f;
  if (c.out_bf16)
    ((u16 *)c.out)[at] = f2bf(v);
  else
    ((float *)c.out)[at] = v;
}

// Parameter gradients of all layers in one launch, after the backward sweep (every activation and
// gradient is kept). Layer weights: gW[a][b][k] = sum_z P[a][z] Q[b][s z + d_k - 1], with P on the coarser
// grid (the output gradient of a convolution, the input of a transposed one); bias: sum_z G[c][z].
// A workgroup takes one chunk of voxels, one 16 x 16 tile of (a, b) and the nine taps of one dz (or,
// as the fourth such group, the bias), its wavefronts quarters of the chunk: each lane loads four
// consecutive voxels of channel a = l % 16 once and the shifted voxels of channel b = l % 16 for
// every tap, and v_mfma_f32_16x16x4 contracts voxel by voxel. Fixed partitions and order of sums.
// 33^3 grid: 64 us (95 with a branch around each load) and 8 for the sums over the chunks (20 with one load in
// flight), against 426 us in 32 launches (one per layer, operand and stage, on the vector units).
struct WGrad {
  const void *P, *Q, *G;
  int p_bf16, na, np, q_bf16, nb, nq, stride;
  int nc, ng;          // bias: channels and grid of G (fp32)
  int nch, blk0;       // chunks; first workgroup of the layer
  int64_t part;        // its partial sums: [chunk][na nb 27 + nc]
  int off;             // its first parameter
};
struct WGrads {
  WGrad l[NL];
};

// A chunk grows with the grid beyond 256 of them (from 53^3 voxels on): a wavefront's FP32 sums run over at
// most WG_RUN tiles of 16 voxels and are then added up in LDS, so that a sum of 129^3 products is 128 + 17
// additions long and not 2,096; the partial sums of the chunks and the biases are summed in FP64. (Added up in
// registers: two waves a SIMD instead of three, 33^3 203 -> 213 us a gradient; in LDS 192.)
constexpr int WG_RUN = 8;

__device__ __forceinline__ int64_t chunk_len(int64_t n, int nch) { return ((n + nch - 1) / nch + 15) / 16 * 16; }

__global__ __launch_bounds__(NT) void k_conv_wgrad(WGrads T, float *__restrict__ part) {
  __shared__ alignas(16) float sh[4][9 * 256];
  int l = 0;
  while (l + 1 < NL && (int)blockIdx.x >= T.l[l + 1].blk0) ++l;
  const WGrad &g = T.l[l];
  int rem = blockIdx.x - g.blk0;
  const int dz = rem & 3;
  rem >>= 2;
  const int nta = (g.na + 15) / 16, ntb = (g.nb + 15) / 16;
  const int ta = rem % nta, tb = (rem / nta) % ntb, ch = rem / (nta * ntb);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int64_t len = (int64_t)g.na * g.nb * 27 + g.nc;
  float *__restrict__ out = part + g.part + (int64_t)ch * len;
  if (dz == 3) {  // bias: tiles (ta, 0) or (0, tb) cover G's channels 16 at a time
    const int ct = g.nc == g.na ? ta : tb;
    if (g.nc == g.na ? tb != 0 : ta != 0) return;
    const int64_t zg = (int64_t)g.ng * g.ng * g.ng, cl = chunk_len(zg, g.nch);
    const int64_t z0 = ch * cl, z1 = min(zg, z0 + cl);
    const int cch = ct * 16 + li;
    double s = 0.0;
    if (cch < g.nc)
      for (int64_t z = z0 + wv * 4 + lk; z < z1; z += 16) s += (double)((const float *)g.G)[(int64_t)cch * zg + z];
    double *shd = reinterpret_cast<double *>(sh[0]);
    shd[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < 16 && ct * 16 + (int)threadIdx.x < g.nc) {
      double t = 0.0;
      for (int k = 0; k < 16; ++k) t += shd[k * 16 + threadIdx.x];
      out[(int64_t)g.na * g.nb * 27 + ct * 16 + threadIdx.x] = (float)t;
    }
    return;
  }
  const int64_t zp = (int64_t)g.np * g.np * g.np, zq = (int64_t)g.nq * g.nq * g.nq;
  const int64_t cl = chunk_len(zp, g.nch);
  const int64_t z0 = ch * cl, z1 = min(zp, z0 + cl);
  const int a = ta * 16 + li, b = tb * 16 + li;
  const int64_t pa = (int64_t)min(a, g.na - 1) * zp, qb = (int64_t)min(b, g.nb - 1) * zq;
  f32x4 acc[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  int run = 0;
  bool more = false;
  auto put = [&]() {  // to the wavefront's own part of LDS
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float &t = sh[wv][k * 256 + r * 64 + lane];
        t = more ? t + acc[k][r] : acc[k][r];
      }
    more = true;
  };
  // the 40 loads of four voxels go out together: what lies outside reads the channel's first value and counts 0
  auto sweep = [&](auto *P, auto *Q) {
    for (int64_t zb = z0 + wv * 16; zb < z1; zb += 64) {
      const int64_t zl = zb + 4 * lk;
      const int zc = (int)min(zl, zp - 1);
      int zx = zc % g.np, zt = zc / g.np, zy = zt % g.np, zz = zt / g.np;
      float pv[4], qv[4][9];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool in = zl + r < z1;
        const float pr = ld_f(P, pa + (in ? zl + r : 0));
        pv[r] = (in & (a < g.na)) ? pr : 0.f;
        const int sx = g.stride * zx - 1, sy = g.stride * zy - 1, sz = g.stride * zz + dz - 1;
        const bool vz = in & (b < g.nb) & ((unsigned)sz < (unsigned)g.nq);
        const int row = (sz * g.nq + sy) * g.nq + sx;  // a channel has at most 513^3 voxels
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          const int dy = k / 3, dx = k % 3;
          const bool ok = vz & ((unsigned)(sy + dy) < (unsigned)g.nq) & ((unsigned)(sx + dx) < (unsigned)g.nq);
          const float q = ld_f(Q, qb + (ok ? row + dy * g.nq + dx : 0));
          qv[r][k] = ok ? q : 0.f;
        }
        if (++zx == g.np) {
          zx = 0;
          if (++zy == g.np) {
            zy = 0;
            ++zz;
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 9; ++k) acc[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[r], qv[r][k], acc[k], 0, 0, 0);
      if (++run == WG_RUN && zb + 64 < z1) {
        run = 0;
        put();
#pragma unroll
        for (int k = 0; k < 9; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  if (g.p_bf16) {
    if (g.q_bf16)
      sweep((const u16 *)g.P, (const u16 *)g.Q);
    else
      sweep((const u16 *)g.P, (const float *)g.Q);
  } else {
    if (g.q_bf16)
      sweep((const float *)g.P, (const u16 *)g.Q);
    else
      sweep((const float *)g.P, (const float *)g.Q);
  }
  put();
  __syncthreads();
  const int t = threadIdx.x;
  const int ao = ta * 16 + 4 * ((t & 63) >> 4) + (t >> 6), bo = tb * 16 + (t & 15);
  if (ao >= g.na || bo >= g.nb) return;
#pragma unroll
  for (int k = 0; k < 9; ++k)
    out[((int64_t)ao * g.nb + bo) * 27 + dz * 9 + k] =
        (sh[0][k * 256 + t] + sh[1][k * 256 + t]) + (sh[2][k * 256 + t] + sh[3][k * 256 + t]);
}

// grad[j] (+)= sum over its layer's chunks of the partial sums, in chunk order
__global__ void k_chunk_reduce(WGrads T, const float *__restrict__ part, float *__restrict__ grad, int accumulate) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= NP) return;
  int l = 0;
  while (l + 1 < NL && j >= T.l[l + 1].off) ++l;
  const WGrad &g = T.l[l];
  const int64_t len = (int64_t)g.na * g.nb * 27 + g.nc;
  const float *__restrict__ p = part + g.part + (j - g.off);
  double s = 0.0;
#pragma unroll 8
  for (int c = 0; c < g.nch; ++c) s += (double)p[(int64_t)c * len];
  grad[j] = accumulate ? grad[j] + (float)s : (float)s;
}

__global__ void k_adam_step(int n, const float *__restrict__ grad, float gscale, float *p, float *m, float *v,
                            u16 *pb, float lr, float c1, float c2) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const float g = grad[j] * gscale;
  const float mj = 0.9f * m[j] + 0.1f * g;
  const float vj = 0.999f * v[j] + 0.001f * g * g;
  m[j] = mj;
  v[j] = vj;
  const float pj = p[j] - lr * (mj * c1) / (sqrtf(vj * c2) + 1e-8f);
  p[j] = pj;
  pb[j] = f2bf(pj);
}

__global__ void k_mirror_bf16(int n, const float *__restrict__ p, u16 *__restrict__ pb) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) pb[j] = f2bf(p[j]);
}

struct Chan4 {
  int64_t off[4];   // dof offset of each channel's scalar block (its vertex dofs come first)
  float scale[4];
};

// x[c][p] = bf16(sv * v[off_c + p] * scale_c)
template <typename T>
__global__ void k_restrict(const T *__restrict__ v, const double *__restrict__ sv, int64_t nv, Chan4 ch,
                           u16 *__restrict__ x) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nv) return;
  const float s = sv ? (float)sv[0] : 1.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) x[(size_t)c * nv + p] = f2bf((float)v[ch.off[c] + p] * s * ch.scale[c]);
}

// g[c][p] = scale_c * v[off_c + p]   (fp32, gradient path)
__global__ void k_restrict_f32(const double *__restrict__ v, int64_t nv, Chan4 ch, float *__restrict__ g) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nv) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) g[(size_t)c * nv + p] = (float)v[ch.off[c] + p] * ch.scale[c];
}

// z[off_c + p] (+)= scale_c * y[c][p] on free dofs
template <typename T>
__global__ void k_embed(const float *__restrict__ y, int64_t nv, Chan4 ch, const uint8_t *__restrict__ freem,
                        T *__restrict__ z, int accumulate) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nv) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t i = ch.off[c] + p;
    const T v = freem[i] ? (T)(ch.scale[c] * y[(size_t)c * nv + p]) : (T)0;
    z[i] = accumulate ? (T)(z[i] + v) : v;
  }
}

// r = v - A D^{-1} v helpers on FP64 dof vectors
__global__ void k_mul_diag(int64_t n, const double *__restrict__ d, const double *__restrict__ v,
                           double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = d[i] * v[i];
}

__global__ void k_sub_masked(int64_t n, const double *__restrict__ a, const double *__restrict__ b,
                             const uint8_t *__restrict__ freem, double *__restrict__ out, double *__restrict__ part) {
  __shared__ double sh[NT / 64];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double v = freem[i] ? a[i] - b[i] : 0.0;
    out[i] = v;
    s += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < NT / 64; ++w) t += sh[w];
    part[blockIdx.x] = t;
  }
}

__global__ void k_neg_masked(int64_t n, const uint8_t *__restrict__ freem, double *__restrict__ v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = freem[i] ? -v[i] : 0.0;
}

// per-block partial sums over samples and vertex points of (v_c)^2 and (dinv v)_c^2, c < 4
__global__ __launch_bounds__(NT) void k_chan_stats(const double *__restrict__ S, int ns, int64_t ld, int64_t nv,
                                                   Chan4 ch, const double *__restrict__ dinv,
                                                   double *__restrict__ part) {
  __shared__ double sh[8][NT / 64];
  double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const int64_t tot = (int64_t)ns * nv;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < tot; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t s = q / nv, p = q % nv;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int64_t i = ch.off[c] + p;
      const double v = S[(size_t)s * ld + i];
      const double z = dinv[i] * v;
      a[c] += v * v;
      a[4 + c] += z * z;
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    double v = a[c];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[c][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    double t = 0.0;
    for (int w = 0; w < NT / 64; ++w) t += sh[threadIdx.x][w];
    part[(size_t)blockIdx.x * 8 + threadIdx.x] = t;
  }
}

constexpr int SUB_GRID = 1024;

}  // namespace

struct Unet {
  Ctx *ctx;
  int N;
  int64_t n[3], zn[3];
  DBuf<float> p, m, v, grad, part;
  DBuf<u16> pb;
  DBuf<float> wp;               // packed FP32 copies of pb's weights
  DBuf<u16> x, act[7];          // x, a0..a6 (bf16)
  DBuf<float> y, gy, g[7];      // y, dL/dy, gradients of a0..a6 (pre-activation)
  Chan4 in_ch{}, out_ch{};
  int64_t step = 0;
  // training state
  DBuf<double> rj, tmp, res, zf, spart;
};

static void pack_weights(Unet *U, hipStream_t st) {
  PackTable T;
  for (int l = 0; l < NL; ++l)
    for (int adj = 0; adj < 2; ++adj) {
      // layer weights [cout][cin][27], transposed layers [cin][cout][27]
      const int sci = LD[l].transposed ? LD[l].cout : 1, sco = LD[l].transposed ? 1 : LD[l].cin;
      T.s[2 * l + adj] = PackSeg{pk_off(l, adj), pk_in(l, adj), pk_out(l, adj), param_off(l), adj ? sco : sci,
                                 adj ? sci : sco};
    }
  k_pack_weights<<<(NPACK + 255) / 256, 256, 0, st>>>(T, U->pb.p, U->wp.p);
  OCMP_HIP(hipGetLastError());
}

template <typename TI>
static void conv_launch_t(const Conv &c, dim3 grid, hipStream_t st) {
  switch (c.cin) {
    case 4: k_conv3<4, TI><<<grid, NT, 0, st>>>(c); break;
    case 8: k_conv3<8, TI><<<grid, NT, 0, st>>>(c); break;
    case 16: k_conv3<16, TI><<<grid, NT, 0, st>>>(c); break;
    default: k_conv3<32, TI><<<grid, NT, 0, st>>>(c); break;
  }
}
static void conv_launch(const Conv &c, hipStream_t st) {
  const int64_t zout = (int64_t)c.nout * c.nout * c.nout;
  dim3 grid((unsigned)((zout + 15) / 16), (unsigned)(c.cop / 16));
  if (c.in_bf16) conv_launch_t<u16>(c, grid, st);
  else conv_launch_t<float>(c, grid, st);
  OCMP_HIP(hipGetLastError());
}

// forward over the bf16 input U->x; keeps every activation
static void unet_forward(Unet *U, hipStream_t st) {
  for (int l = 0; l < NL; ++l) {
    const LayerDef &L = LD[l];
    Conv c{};
    c.in = (l == 0) ? (const void *)U->x.p : (const void *)U->act[l - 1].p;
    c.in_bf16 = 1;
    c.cin = L.cin;
    c.nin = (int)U->n[L.level_in];
    c.cout = L.cout;
    c.nout = (int)U->n[L.level_out];
    c.W = U->wp.p + pk_off(l, 0);
    c.cop = pad16(L.cout);
    c.bias = U->pb.p + param_off(l) + layer_w(l);
    c.stride = L.stride;
    c.transposed = L.transposed;
    if (l == 5) c.skip = U->act[2].p, c.skip_bf16 = 1;
    if (l == 6) c.skip = U->act[0].p, c.skip_bf16 = 1;
    if (l < NL - 1) {
      c.out = U->act[l].p;
      c.out_bf16 = 1;
      c.relu = 1;
    } else {
      c.out = U->y.p;
      c.out_bf16 = 0;
      c.relu = 0;
    }
    conv_launch(c, st);
  }
}

// what every layer's parameter gradient is formed from, and the partition of its voxels: chunks of
// 512 voxels (a wavefront's share keeps its nine accumulators busy for eight tiles), longer on grids that
// would give more than 256
static WGrads wgrad_table(Unet *U, int64_t *part_len, int *nblocks) {
  WGrads T;
  int64_t po = 0;
  int blk = 0;
  for (int l = 0; l < NL; ++l) {
    const LayerDef &L = LD[l];
    const void *gout = l == NL - 1 ? (const void *)U->gy.p : (const void *)U->g[l].p;
    const void *xin = l == 0 ? (const void *)U->x.p : (const void *)U->act[l - 1].p;
    WGrad &g = T.l[l];
    const int nin = (int)U->n[L.level_in], nout = (int)U->n[L.level_out];
    if (!L.transposed) g = WGrad{gout, xin, gout, 0, L.cout, nout, 1, L.cin, nin, L.stride};
    else g = WGrad{xin, gout, gout, 1, L.cin, nin, 0, L.cout, nout, L.stride};
    g.nc = L.cout;
    g.ng = nout;
    const int64_t zp = (int64_t)g.np * g.np * g.np;
    g.nch = (int)std::min<int64_t>(256, (zp + 511) / 512);
    g.blk0 = blk;
    g.part = po;
    g.off = param_off(l);
    blk += 4 * ((g.na + 15) / 16) * ((g.nb + 15) / 16) * g.nch;
    po += (int64_t)g.nch * layer_p(l);
  }
  *part_len = po;
  *nblocks = blk;
  return T;
}

// backward from U->gy (dL/dy, fp32): parameter gradients into U->grad (accumulated if asked)
static void unet_backward(Unet *U, int accumulate, hipStream_t st) {
  // adjoint (grad-input) of layer l applied to gout, masked by the layer input's activation
  auto adj = [&](int l, const float *gout, float *gin, const float *skipg, const u16 *mask) {
    const LayerDef &L = LD[l];
    Conv c{};
    c.in = gout;
    c.in_bf16 = 0;
    c.cin = L.cout;
    c.nin = (int)U->n[L.level_out];
    c.out = gin;
    c.out_bf16 = 0;
    c.cout = L.cin;
    c.nout = (int)U->n[L.level_in];
    c.W = U->wp.p + pk_off(l, 1);
    c.cop = pad16(L.cin);
    c.transposed = !L.transposed;  // the adjoint of a gather conv is a scatter (transposed) conv
    c.stride = L.stride;
    c.skip = skipg;
    c.skip_bf16 = 0;
    c.mask = mask;
    conv_launch(c, st);
  };
  adj(7, U->gy.p, U->g[6].p, nullptr, U->act[6].p);
  adj(6, U->g[6].p, U->g[5].p, nullptr, U->act[5].p);
  adj(5, U->g[5].p, U->g[4].p, nullptr, U->act[4].p);
  adj(4, U->g[4].p, U->g[3].p, nullptr, U->act[3].p);
  adj(3, U->g[3].p, U->g[2].p, U->g[5].p, U->act[2].p);  // + skip from a5
  adj(2, U->g[2].p, U->g[1].p, nullptr, U->act[1].p);
  adj(1, U->g[1].p, U->g[0].p, U->g[6].p, U->act[0].p);  // + skip from a6
  int64_t plen;
  int nblk;
  const WGrads T = wgrad_table(U, &plen, &nblk);
  OCMP_REQUIRE((size_t)plen <= U->part.n, "unet: weight-gradient scratch too small");
  k_conv_wgrad<<<nblk, NT, 0, st>>>(T, U->part.p);
  OCMP_HIP(hipGetLastError());
  k_chunk_reduce<<<(NP + 255) / 256, 256, 0, st>>>(T, U->part.p, U->grad.p, accumulate);
  OCMP_HIP(hipGetLastError());
}

Unet *unet_create(Ctx *ctx, int N, const float *params) {
  OCMP_REQUIRE(N >= 4 && N % 4 == 0 && N <= 512, "unet: N must be a multiple of 4 in [4, 512]");
  OCMP_REQUIRE(params, "unet: null parameters");
  auto *U = new Unet();
  U->ctx = ctx;
  U->N = N;
  U->n[0] = N + 1;
  U->n[1] = N / 2 + 1;
  U->n[2] = N / 4 + 1;
  for (int l = 0; l < 3; ++l) U->zn[l] = U->n[l] * U->n[l] * U->n[l];
  try {
    U->p.alloc(NP);
    U->m.alloc(NP);
    U->v.alloc(NP);
    U->grad.alloc(NP);
    U->pb.alloc(NP);
    U->x.alloc((size_t)4 * U->zn[0]);
    for (int l = 0; l < 7; ++l) {
      const LayerDef &L = LD[l];
      U->act[l].alloc((size_t)L.cout * U->zn[L.level_out]);
      U->g[l].alloc((size_t)L.cout * U->zn[L.level_out]);
    }
    U->y.alloc((size_t)4 * U->zn[0]);
    U->gy.alloc((size_t)4 * U->zn[0]);
    U->wp.alloc(NPACK);
    int64_t plen;
    int nblk;
    wgrad_table(U, &plen, &nblk);
    U->part.alloc((size_t)plen);  // at most 256 partial sums of every parameter
    unet_set_params(U, params);
  } catch (...) {
    delete U;
    throw;
  }
  for (int c = 0; c < 4; ++c) U->in_ch.scale[c] = U->out_ch.scale[c] = 1.f;
  return U;
}

void unet_destroy(Unet *U) { delete U; }

int64_t unet_grid_points(const Unet *U) { return U->zn[0]; }

void unet_set_params(Unet *U, const float *params) {
  hipStream_t st = U->ctx->stream;
  OCMP_HIP(hipMemcpyAsync(U->p.p, params, NP * sizeof(float), hipMemcpyHostToDevice, st));
  OCMP_HIP(hipMemsetAsync(U->m.p, 0, NP * sizeof(float), st));
  OCMP_HIP(hipMemsetAsync(U->v.p, 0, NP * sizeof(float), st));
  k_mirror_bf16<<<(NP + 255) / 256, 256, 0, st>>>(NP, U->p.p, U->pb.p);
  OCMP_HIP(hipGetLastError());
  pack_weights(U, st);
  OCMP_HIP(hipStreamSynchronize(st));
  U->step = 0;
}

void unet_get_params(Unet *U, float *params) {
  OCMP_HIP(hipMemcpyAsync(params, U->p.p, NP * sizeof(float), hipMemcpyDeviceToHost, U->ctx->stream));
  OCMP_HIP(hipStreamSynchronize(U->ctx->stream));
}

void unet_set_channels(Unet *U, const int64_t *off, const double *in_scale, const double *out_scale) {
  for (int c = 0; c < 4; ++c) {
    OCMP_REQUIRE(off[c] >= 0, "unet: negative channel offset");
    OCMP_REQUIRE(in_scale[c] > 0 && out_scale[c] > 0 && std::isfinite(in_scale[c]) && std::isfinite(out_scale[c]),
                 "unet: channel scales must be positive");
    U->in_ch.off[c] = U->out_ch.off[c] = off[c];
    U->in_ch.scale[c] = (float)in_scale[c];
    U->out_ch.scale[c] = (float)out_scale[c];
  }
}

int64_t unet_max_index(const Unet *U) {
  int64_t m = 0;
  for (int c = 0; c < 4; ++c) m = std::max(m, U->in_ch.off[c] + U->zn[0]);
  return m;
}

// channel scales from samples (device f64 rows, stride ld): in_c = 1/rms(v_c), out_c = rms((D^{-1} v)_c)
void unet_fit_channels(Unet *U, Precond *P, const double *samples, int ns, int64_t ld, const int64_t *off) {
  OCMP_REQUIRE(P && P->kind == OCMP_PRE_JACOBI && P->ready, "unet: needs an updated Jacobi preconditioner");
  for (int c = 0; c < 4; ++c) {
    OCMP_REQUIRE(off[c] >= 0 && off[c] + U->zn[0] <= P->A->n, "unet: channel dofs out of range");
    U->in_ch.off[c] = U->out_ch.off[c] = off[c];
  }
  hipStream_t st = U->ctx->stream;
  const int nb = 512;
  DBuf<double> part;
  part.alloc((size_t)nb * 8);
  k_chan_stats<<<nb, NT, 0, st>>>(samples, ns, ld, U->zn[0], U->in_ch, P->dinv.p, part.p);
  OCMP_HIP(hipGetLastError());
  std::vector<double> h((size_t)nb * 8);
  OCMP_HIP(hipMemcpyAsync(h.data(), part.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  OCMP_HIP(hipStreamSynchronize(st));
  const double cnt = (double)ns * (double)U->zn[0];
  for (int c = 0; c < 4; ++c) {
    double sv = 0.0, sz = 0.0;
    for (int b = 0; b < nb; ++b) {
      sv += h[(size_t)b * 8 + c];
      sz += h[(size_t)b * 8 + 4 + c];
    }
    const double rv = std::sqrt(sv / cnt), rz = std::sqrt(sz / cnt);
    U->in_ch.scale[c] = rv > 0 ? (float)(1.0 / rv) : 1.f;
    U->out_ch.scale[c] = rz > 0 ? (float)rz : 1.f;
  }
}

void unet_get_channels(const Unet *U, int64_t *off, double *in_scale, double *out_scale) {
  for (int c = 0; c < 4; ++c) {
    off[c] = U->in_ch.off[c];
    in_scale[c] = U->in_ch.scale[c];
    out_scale[c] = U->out_ch.scale[c];
  }
}

// copy one stored activation (layer -1: the bf16 input, 0..6: a0..a6, 7: y) as float32
__global__ void k_bf16_to_f32(int64_t n, const u16 *__restrict__ a, float *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = bf2f(a[i]);
}

int64_t unet_activation(Unet *U, int layer, float *out) {
  hipStream_t st = U->ctx->stream;
  if (layer == 7) {
    const int64_t n = 4 * U->zn[0];
    if (out) OCMP_HIP(hipMemcpyAsync(out, U->y.p, n * sizeof(float), hipMemcpyDeviceToDevice, st));
    return n;
  }
  const u16 *src = layer < 0 ? U->x.p : U->act[layer].p;
  const int64_t n = layer < 0 ? 4 * U->zn[0] : (int64_t)LD[layer].cout * U->zn[LD[layer].level_out];
  if (out) {
    k_bf16_to_f32<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(n, src, out);
    OCMP_HIP(hipGetLastError());
  }
  return n;
}

// y = U(x): grid in/out (device, x: float32 [4][n0^3] rounded to bf16 on entry, y: float32)
void unet_forward_grid(Unet *U, const float *x, float *y) {
  hipStream_t st = U->ctx->stream;
  Ctx *c = U->ctx;
  KTimer t(c, c->cls("unet_forward"), 0.0);
  const int64_t n4 = 4 * U->zn[0];
  k_mirror_bf16<<<(unsigned)((n4 + 255) / 256), 256, 0, st>>>((int)n4, x, U->x.p);
  OCMP_HIP(hipGetLastError());
  unet_forward(U, st);
  OCMP_HIP(hipMemcpyAsync(y, U->y.p, n4 * sizeof(float), hipMemcpyDeviceToDevice, st));
}

// parameter gradient of sum(gy * U(x)) (grid, device float32) into grad (device float32[NP])
void unet_grad_grid(Unet *U, const float *x, const float *gy, float *grad) {
  hipStream_t st = U->ctx->stream;
  const int64_t n4 = 4 * U->zn[0];
  k_mirror_bf16<<<(unsigned)((n4 + 255) / 256), 256, 0, st>>>((int)n4, x, U->x.p);
  OCMP_HIP(hipGetLastError());
  unet_forward(U, st);
  OCMP_HIP(hipMemcpyAsync(U->gy.p, gy, n4 * sizeof(float), hipMemcpyDeviceToDevice, st));
  unet_backward(U, 0, st);
  OCMP_HIP(hipMemcpyAsync(grad, U->grad.p, NP * sizeof(float), hipMemcpyDeviceToDevice, st));
}

// z (+)= E U(R (s v)) on the free dofs of A's space (the learned half of the preconditioner)
template <typename T>
void unet_correct(Unet *U, const uint8_t *freem, const T *v, const double *sv, T *z, int accumulate) {
  hipStream_t st = U->ctx->stream;
  Ctx *c = U->ctx;
  KTimer t(c, c->cls(sizeof(T) == 8 ? "unet_correction_f64" : "unet_correction_f32"), 0.0);
  const int64_t nv = U->zn[0];
  k_restrict<T><<<(unsigned)((nv + 255) / 256), 256, 0, st>>>(v, sv, nv, U->in_ch, U->x.p);
  OCMP_HIP(hipGetLastError());
  unet_forward(U, st);
  k_embed<T><<<(unsigned)((nv + 255) / 256), 256, 0, st>>>(U->y.p, nv, U->out_ch, freem, z, accumulate);
  OCMP_HIP(hipGetLastError());
}
template void unet_correct<float>(Unet *, const uint8_t *, const float *, const double *, float *, int);
template void unet_correct<double>(Unet *, const uint8_t *, const double *, const double *, double *, int);

// One Adam step of the self-supervised loss  L = 1/(2B) sum_b ||r_b - A E U(R v_b)||^2,
// r_b = v_b - A D^{-1} v_b, over the batch of samples v_b = samples[idx[b]] (device f64 rows
// of length A->n). Returns the batch loss (host, syncs).
double unet_train_step(Unet *U, Matrix *A, Precond *P, const double *samples, int64_t ld, const int *idx, int nb,
                       float lr) {
  OCMP_REQUIRE(P && P->kind == OCMP_PRE_JACOBI && P->ready, "unet training needs an updated Jacobi preconditioner");
  OCMP_REQUIRE(nb >= 1, "unet: empty batch");
  hipStream_t st = U->ctx->stream;
  const int64_t n = A->n;
  const uint8_t *fm = A->space->d_free.p;
  U->rj.alloc(n);
  U->tmp.alloc(n);
  U->res.alloc(n);
  U->zf.alloc(n);
  U->spart.alloc((size_t)SUB_GRID * (nb + 1));  // row nb: scratch partials of r_J
  const int64_t nv = U->zn[0];
  const unsigned gb = (unsigned)((n + 255) / 256);
  for (int b = 0; b < nb; ++b) {
    const double *vb = samples + (size_t)idx[b] * ld;
    // r_J = v - A D^{-1} v
    k_mul_diag<<<gb, 256, 0, st>>>(n, P->dinv.p, vb, U->tmp.p);
    spmv_f64(A, U->tmp.p, U->res.p);
    k_sub_masked<<<SUB_GRID, 256, 0, st>>>(n, vb, U->res.p, fm, U->rj.p, U->spart.p + (size_t)nb * SUB_GRID);
    // z = E U(R v) (zero elsewhere), res = r_J - A z, loss partials
    OCMP_HIP(hipMemsetAsync(U->zf.p, 0, n * sizeof(double), st));
    unet_correct<double>(U, fm, vb, nullptr, U->zf.p, 1);
    spmv_f64(A, U->zf.p, U->tmp.p);
    k_sub_masked<<<SUB_GRID, 256, 0, st>>>(n, U->rj.p, U->tmp.p, fm, U->res.p, U->spart.p + (size_t)b * SUB_GRID);
    // dL/dz = -A^T res = -A res (the Stokes systems are symmetric); restricted to the grid
    spmv_f64(A, U->res.p, U->tmp.p);
    k_neg_masked<<<gb, 256, 0, st>>>(n, fm, U->tmp.p);
    k_restrict_f32<<<(unsigned)((nv + 255) / 256), 256, 0, st>>>(U->tmp.p, nv, U->out_ch, U->gy.p);
    OCMP_HIP(hipGetLastError());
    // U->x still holds R v of this sample, the activations its forward pass
    unet_backward(U, b > 0 ? 1 : 0, st);
  }
  U->step += 1;
  const float c1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)U->step)));
  const float c2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)U->step)));
  k_adam_step<<<(NP + 255) / 256, 256, 0, st>>>(NP, U->grad.p, 1.f / (float)nb, U->p.p, U->m.p, U->v.p, U->pb.p, lr,
                                                c1, c2);
  OCMP_HIP(hipGetLastError());
  pack_weights(U, st);
  std::vector<double> h((size_t)SUB_GRID * nb);  // rows 0..nb-1: the loss partials
  OCMP_HIP(hipMemcpyAsync(h.data(), U->spart.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  OCMP_HIP(hipStreamSynchronize(st));
  double loss = 0.0;
  for (double v : h) loss += v;
  return 0.5 * loss / nb;
}

}  // namespace ocmp
