// hps_unet.hip -- kernels of the learned SCHEFF field surrogate: a
// one-dimensional convolutional U-Net along the bunch axis z with the source
// rings as channels (network object and C ABI in hps_surrogate.hip): the
// convolutions forward and backward on the BF16 matrix cores, FiLM, loss,
// Adam.
//
// Why this shape: the SCHEFF field is linear in the charge histogram and
// invariant under shifts along z (the Green's table depends on zp - zs only,
// space_charge_kernel.cu:38-100), but not under shifts in r.  So the network
// convolves along z, mixes rings densely in its channels, has no biases and
// no activations (superposition holds exactly), and takes the mesh aspect --
// the one parameter of the normalised Green's function -- through FiLM
// scales 1 + sum_j A[l][c][j] u^j (j = 1..3) on every layer's channels.
// The U-Net levels (z, z/2, z/4, z/8, and dilated convolutions at the
// coarsest level) reach the whole bunch, as the Coulomb field does.
//
// Input x[b][z][rs] = n(zs = z, rs) * nr * nz / Q for z < nz and 0 for the
// padding up to Z0 = nz + 8 (n particles per bin, Q their sum); output
// y[b][z][2 rp + comp] for the field nodes z <= nz; the field (before the
// c1 / dr^2 factor) is y * Q * out_scale.
//
// Precision: weights BF16 (FP32 master copies for Adam), accumulation FP32
// on v_mfma_f32_16x16x16_bf16; activations stay FP32 in memory and enter
// the products as two BF16 terms (hi + lo), so the only rounding of an
// activation is that of FP32.
//
// MFMA 16x16x16 bf16 operand layout (wave64): lane l supplies A[m][k] for
// m = l % 16, k = 4 (l / 16) + j and B[k][n] for n = l % 16, k = 4 (l / 16)
// + j (j = 0..3); the result D[m][n] is held for n = l % 16, m = 4 (l / 16)
// + i in element i.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "hpsim_amd.h"
#include "hps_unet.hpp"

namespace hps {

int fail_msg(const std::string& m);   // hps_engine.hip

namespace unet {

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kMaxFrag = kMaxCout / 16;
// Output positions from which a conv workgroup takes two position tiles: each
// weight fragment then serves two products, but the workgroups are half as
// many.  The line was set without a sweep and lies lower than the sizes below
// ask for: two tiles pay only on a device that is full either way.  The same
// run with two tiles from 4,096 positions on, one tile always, and two from
// 20,000 on: training, 64 samples on 32 x 128 (at most 8,704 positions) 7.8 /
// 7.0 / 7.0 ms, on 64 x 256 (16,896) 9.5 / 8.5 / 8.5; 160 beams of 32 x 128 with
// surrogate fields (21,760) 5.1 / 4.9 / 4.8.  The bits are the same either way.
constexpr int kConvTwoTiles = 4096;

__host__ __device__ inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// float -> bfloat16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ uint16_t f2bf(float f)
{
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// v = hi + lo with hi = bf16(v), lo = bf16(v - hi)
__device__ __forceinline__ void split4(const float4& v, s4& hi, s4& lo)
{
  const float a[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint16_t h = f2bf(a[j]);
    hi[j] = (short)h;
    lo[j] = (short)f2bf(a[j] - bf2f(h));
  }
}

__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// source position of output position zo for tap t (-1: none)
__device__ __forceinline__ int src_of(int mode, int zo, int t, int dil, int zin)
{
  int zi;
  switch (mode) {
    case kSame: zi = zo + (t - 1) * dil; break;
    case kSameFlip: zi = zo + (1 - t) * dil; break;
    case kPoint: zi = zo; break;
    case kDown: zi = 2 * zo + t; break;
    default: zi = (zo & 1) == t ? zo >> 1 : -1; break;   // kUp
  }
  return (zi >= 0 && zi < zin) ? zi : -1;
}

// pre = conv(in); out = pre * scale[b][co] (+ skip).  A workgroup computes
// kMT tiles of 16 output positions, one wave per 16 output channels (Cout / 16
// waves).  Cin % 16 == 0, Cout % 16 == 0, both <= kMaxCout.
//
// What bounds a layer is latency, not the matrix cores: at 6 samples of 136
// positions a layer is 51 position tiles of 18 dependent product steps.  So a
// wave takes one channel tile only (a wave over all channels left 51 waves on
// 1,024 SIMDs), its weights (stored in operand order by k_bf16:
// one contiguous 512-byte load per step) and the epilogue's operands are
// loaded before anything waits, and the activations' split into two BF16
// terms, 3/4 of the arithmetic, is done once per workgroup into LDS instead
// of once per channel tile.  Six 65,536-particle members over 20 periods with
// surrogate fields: 45.9 -> 20.8 ms; a training step of 64 samples, with the
// backward kernels below: 1.90 -> 0.88 ms.  Each output's sum runs over (tap, channel) in
// ascending order, hi term before lo term, whatever the tiling.
// LDS: rows of Cin / 4 16-byte groups (4 hi, 4 lo) plus one group of padding.
constexpr int kMaxSteps = 3 * kMaxCout / 16;   // product steps (16 channels of a tap) of a layer

__host__ __device__ inline size_t conv_lds(int taps, int Cin, int mt)
{
  return (size_t)taps * 16 * mt * (Cin / 4 + 1) * 16;
}

template <int kMT>
__global__ __launch_bounds__(64 * kMaxFrag) void k_conv(ConvArgs a)
{
  extern __shared__ uint4 tile[];
  const int B = a.dyn_b ? (int)a.dyn_b[0] : a.B;
  const int P = B * a.Zout;
  const int p0 = blockIdx.x * 16 * kMT;
  if (p0 >= P) return;
  const int lane = threadIdx.x & 63;
  const int n = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // channel tile
  const int KS = a.taps * a.Cin / 16;
  const uint2* wp = reinterpret_cast<const uint2*>(a.w) + (size_t)n * KS * 64 + lane;
  uint2 wv[kMaxSteps];
#pragma unroll
  for (int s = 0; s < kMaxSteps; ++s)
    if (s < KS) wv[s] = wp[(size_t)s * 64];
  // epilogue operands of this lane's outputs: channel co, positions p0 + 16 mt + 4 (lane / 16) + i
  const int co = n * 16 + (lane & 15);
  float scl[kMT][4], skp[kMT][4];
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = min(p0 + 16 * mt + 4 * (lane >> 4) + i, P - 1);
      scl[mt][i] = a.scale ? a.scale[(size_t)(p / a.Zout) * a.Cout + co] : 1.f;
      skp[mt][i] = a.skip ? a.skip[(size_t)p * a.Cout + co] : 0.f;
    }
  // the tile's source rows, split, into LDS; four groups of loads in flight
  const int G = a.Cin / 4;
  const int total = a.taps * 16 * kMT * G;
  const int nthr = blockDim.x;
  constexpr int kStage = 4;
  for (int e0 = threadIdx.x; e0 < total; e0 += kStage * nthr) {
    float4 v[kStage];
    int at[kStage];
#pragma unroll
    for (int u = 0; u < kStage; ++u) {
      const int e = e0 + u * nthr;
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      at[u] = -1;
      if (e < total) {
        const int row = e / G, g = e - row * G;
        const int t = row / (16 * kMT), p = p0 + row - t * 16 * kMT;
        at[u] = row * (G + 1) + g;
        if (p < P) {
          const int b = p / a.Zout;
          const int zi = src_of(a.mode, p - b * a.Zout, t, a.dil, a.Zin);
          if (zi >= 0)
            v[u] = *reinterpret_cast<const float4*>(a.in + ((size_t)b * a.Zin + zi) * a.Cin +
                                                    4 * g);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kStage; ++u) {
      if (at[u] < 0) continue;
      s4 hi, lo;
      split4(v[u], hi, lo);
      const uint2 h = __builtin_bit_cast(uint2, hi), l = __builtin_bit_cast(uint2, lo);
      tile[at[u]] = make_uint4(h.x, h.y, l.x, l.y);
    }
  }
  __syncthreads();
  f4 acc[kMT];
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt) acc[mt] = f4{0.f, 0.f, 0.f, 0.f};
  const int per = a.Cin / 16;
  int row = lane & 15, c = 0;   // LDS row of (tap, position), 16-channel block in it
#pragma unroll
  for (int s = 0; s < kMaxSteps; ++s) {
    if (s >= KS) continue;
    const s4 b = __builtin_bit_cast(s4, wv[s]);
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt) {
      const uint4 q = tile[(row + 16 * mt) * (G + 1) + 4 * c + (lane >> 4)];
      const s4 hi = __builtin_bit_cast(s4, make_uint2(q.x, q.y));
      const s4 lo = __builtin_bit_cast(s4, make_uint2(q.z, q.w));
      acc[mt] = mfma(hi, b, acc[mt]);
      acc[mt] = mfma(lo, b, acc[mt]);
    }
    if (++c == per) { c = 0; row += 16 * kMT; }
  }
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = p0 + 16 * mt + 4 * (lane >> 4) + i;
      if (p >= P) continue;
      const size_t o = (size_t)p * a.Cout + co;
      float v = acc[mt][i];
      if (a.pre) a.pre[o] = v;
      if (a.scale) v *= scl[mt][i];
      if (a.skip) v += skp[mt][i];
      a.out[o] = v;
    }
}

// dw[co][t][ci] += sum over positions of dpre[p][co] * in[src(p, t)][ci]:
// one workgroup per (tap, 16 co, 16 ci, chunk of 256 positions); FP32 atomics.
__global__ __launch_bounds__(64 * kWaves) void k_wgrad(WgradArgs a)
{
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int P = a.B * a.Zout;
  const int nco = a.Cout / 16, nci = a.Cin / 16;
  const int nchunk = cdiv(P, kWgradChunk);
  const int chunk = blockIdx.x % nchunk;
  int r = blockIdx.x / nchunk;
  const int cit = r % nci; r /= nci;
  const int cot = r % nco;
  const int t = r / nco;
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  const int kq = 4 * (lane >> 4);
  const int co = cot * 16 + (lane & 15), ci = cit * 16 + (lane & 15);
  const int pend = min(P, (chunk + 1) * kWgradChunk);
  // A task is one workgroup: its waves take 64 positions each, whose loads
  // are all issued before the first is used, and meet in LDS, so a weight gets
  // one atomic add per task.  (A wave per task left most SIMDs with one wave
  // or none, whose memory round trips nothing hid: 19.3 us a layer at 64
  // samples, so 9.2; with eight waves and 512 positions 9.9.)
  constexpr int kAhead = 4;
  static_assert(16 * kAhead * kWaves == kWgradChunk, "one step per wave");
  const int q0 = chunk * kWgradChunk + wave * 16 * kAhead;
  if (q0 < pend) {
    float dv[kAhead][4], xv[kAhead][4];
#pragma unroll
    for (int h = 0; h < kAhead; ++h) {
      const int pq = q0 + 16 * h + kq;
      int b = pq / a.Zout, zo = pq - b * a.Zout;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = pq + j;
        dv[h][j] = 0.f;
        xv[h][j] = 0.f;
        if (p < pend) {
          const int zi = src_of(a.mode, zo, t, a.dil, a.Zin);
          if (zi >= 0) {
            dv[h][j] = a.dpre[(size_t)p * a.Cout + co];
            xv[h][j] = a.in[((size_t)b * a.Zin + zi) * a.Cin + ci];
          }
        }
        if (++zo == a.Zout) { zo = 0; ++b; }
      }
    }
#pragma unroll
    for (int h = 0; h < kAhead; ++h) {
      s4 da, xh, xl;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        da[j] = (short)f2bf(dv[h][j]);
        const uint16_t x = f2bf(xv[h][j]);
        xh[j] = (short)x;
        xl[j] = (short)f2bf(xv[h][j] - bf2f(x));
      }
      acc = mfma(da, xh, acc);
      acc = mfma(da, xl, acc);
    }
  }
  // D[m = co][n = ci]: a lane holds ci = cit*16 + lane%16, co rows 4(lane/16)+i;
  // thread 64 i + lane adds element i of its lane over the waves
  __shared__ float part[kWaves][4][64];
#pragma unroll
  for (int i = 0; i < 4; ++i) part[wave][i][lane] = acc[i];
  __syncthreads();
  static_assert(kWaves == 4, "a wave per element of the accumulator");
  float v = part[0][wave][lane];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) v += part[w][wave][lane];
  const int cor = cot * 16 + 4 * (lane >> 4) + wave;
  atomicAdd(&a.dw[((size_t)cor * a.taps + t) * a.Cin + ci], v);
}

// Bounded conditioning v = 2 tanh(u / 2) (the FiLM polynomial stays within
// the range it was trained on)
__device__ __forceinline__ float film_v(float u) { return 2.f * tanhf(0.5f * u); }

// FiLM scales of every layer: scale[l][b][co] = 1 + sum_j A[l][co][j] v_b^j
__global__ void k_film(const float* __restrict__ params, const FilmLayer* __restrict__ layers,
                       int nlayers, const float* __restrict__ u, const uint32_t* dyn_b, int B,
                       float* __restrict__ scale, int max_b)
{
  const int nb = dyn_b ? (int)dyn_b[0] : B;
  const int l = blockIdx.y;
  if (l >= nlayers) return;
  const FilmLayer L = layers[l];
  for (int e = blockIdx.x * 256 + threadIdx.x; e < nb * L.cout; e += gridDim.x * 256) {
    const int b = e / L.cout, co = e % L.cout;
    const float x = film_v(u[b]);
    const float* A = params + L.a_off + (size_t)co * 3;
    scale[L.s_off + (size_t)b * L.cout + co] = 1.f + A[0] * x + A[1] * x * x + A[2] * x * x * x;
  }
}

// dpre = dy * scale; part[b][slab][co] = sum over the slab's z of dy * pre.
// Workgroup (b, slab of z): C / 4 threads take four channels each, the others
// further rows of the slab; the rows' sums meet in LDS.  (One thread per
// (b, co) over all z left the chip idle: 25 us a layer at 64 samples.)  The
// slabs' sums are stored and added up by one k_film_sum for all layers: added
// atomically, three values a channel, they met in the few cache lines of a
// layer's coefficients (12.5 us a layer at 64 samples, so 3.6).
__global__ __launch_bounds__(256) void k_film_bwd(const float* __restrict__ dy,
                                                  const float* __restrict__ pre,
                                                  const float* __restrict__ scale,
                                                  float* __restrict__ dpre,
                                                  float* __restrict__ part, int Z, int C)
{
  __shared__ float4 red[256];
  const int b = blockIdx.x, C4 = C / 4, ng = 256 / C4;
  const int g = threadIdx.x / C4, c = threadIdx.x - g * C4;
  const int z1 = min(Z, (int)(blockIdx.y + 1) * kFilmSlab);
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  if (g < ng) {
    const float4 s = reinterpret_cast<const float4*>(scale + (size_t)b * C)[c];
    for (int z = blockIdx.y * kFilmSlab + g; z < z1; z += ng) {
      const size_t o = ((size_t)b * Z + z) * C4 + c;
      const float4 d = reinterpret_cast<const float4*>(dy)[o];
      const float4 q = reinterpret_cast<const float4*>(pre)[o];
      sum.x += d.x * q.x; sum.y += d.y * q.y; sum.z += d.z * q.z; sum.w += d.w * q.w;
      reinterpret_cast<float4*>(dpre)[o] = make_float4(d.x * s.x, d.y * s.y, d.z * s.z, d.w * s.w);
    }
  }
  red[threadIdx.x] = sum;
  __syncthreads();
  // channel co of the slab: the ng row sums
  if ((int)threadIdx.x < C) {
    float t = 0.f;
    for (int k = 0; k < ng; ++k)
      t += reinterpret_cast<const float*>(red)[4 * k * C4 + threadIdx.x];
    part[((size_t)b * gridDim.y + blockIdx.y) * C + threadIdx.x] = t;
  }
}

// dA[co][j] += sum over samples and slabs of part[b][slab][co] v_b^j, every
// layer: workgroup (16 channels, layer), a thread a channel of every sixteenth
// sample, the sixteen sums of a channel met in LDS.
__global__ __launch_bounds__(256) void k_film_sum(const FilmLayer* __restrict__ layers,
                                                  const float* __restrict__ part,
                                                  const float* __restrict__ u, float* __restrict__ g,
                                                  int B)
{
  __shared__ float red[3][256];
  const FilmLayer L = layers[blockIdx.y];
  const int co = blockIdx.x * 16 + (threadIdx.x & 15);
  float a0 = 0.f, a1 = 0.f, a2 = 0.f;
  if (co < L.cout) {
    const float* p = part + L.p_off + co;
    for (int b = threadIdx.x >> 4; b < B; b += 16) {
      float t = 0.f;
      for (int k = 0; k < L.slabs; ++k) t += p[((size_t)b * L.slabs + k) * L.cout];
      const float x = film_v(u[b]);
      a0 += t * x;
      a1 += t * x * x;
      a2 += t * x * x * x;
    }
  }
  red[0][threadIdx.x] = a0;
  red[1][threadIdx.x] = a1;
  red[2][threadIdx.x] = a2;
  __syncthreads();
  const int j = threadIdx.x >> 4;
  if (j < 3 && co < L.cout) {
    float v = 0.f;
    for (int k = 0; k < 16; ++k) v += red[j][16 * k + (threadIdx.x & 15)];
    g[L.a_off + (size_t)co * 3 + j] += v;
  }
}

// loss_b = |y - t / out_scale|^2 / |t / out_scale|^2 over z < zn, c < cout
// (y [B][Z0][Cpad], t [B][zn][cout]); dy (optional) = d loss_mean / d y
// A workgroup per sample, as wide as it goes: the passes over its rows are
// dependent loads and divisions (64 samples of 129 x 66: 256 threads 25 us,
// 1,024 threads 11).
constexpr int kLossBlock = 1024;

__global__ __launch_bounds__(kLossBlock) void k_loss(
    const float* __restrict__ y, const float* __restrict__ tgt, float* __restrict__ dy,
    float* __restrict__ loss, int Z0, int Cpad, int zn, int cout, float inv_scale, int B)
{
  __shared__ float red[2][kLossBlock];
  const int b = blockIdx.x, t = threadIdx.x;
  float nt = 0.f, nd = 0.f;
  for (int e = t; e < zn * cout; e += kLossBlock) {
    const int z = e / cout, c = e % cout;
    const float tv = tgt[((size_t)b * zn + z) * cout + c] * inv_scale;
    const float d = y[((size_t)b * Z0 + z) * Cpad + c] - tv;
    nt += tv * tv;
    nd += d * d;
  }
  red[0][t] = nt;
  red[1][t] = nd;
  __syncthreads();
  for (int o = kLossBlock / 2; o > 0; o >>= 1) {
    if (t < o) { red[0][t] += red[0][t + o]; red[1][t] += red[1][t + o]; }
    __syncthreads();
  }
  const float ntot = red[0][0] > 0.f ? red[0][0] : 1.f;
  if (t == 0) loss[b] = red[1][0] / ntot;
  if (!dy) return;
  const float k = 2.f / (ntot * (float)B);
  for (int e = t; e < Z0 * Cpad; e += kLossBlock) {
    const int z = e / Cpad, c = e % Cpad;
    float v = 0.f;
    if (z < zn && c < cout)
      v = k * (y[((size_t)b * Z0 + z) * Cpad + c] - tgt[((size_t)b * zn + z) * cout + c] * inv_scale);
    dy[((size_t)b * Z0) * Cpad + e] = v;
  }
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ gr, float* __restrict__ m,
                       float* __restrict__ v, int n, float lr_t, float b1, float b2, float eps)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float g = gr[i];
  const float mi = b1 * m[i] + (1.f - b1) * g;
  const float vi = b2 * v[i] + (1.f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr_t * mi / (sqrtf(vi) + eps);
}

// BF16 copies of the layers' weights W[Cout][taps][Cin] in the operand order
// of k_conv: element j of lane l of step s of output tile n at
// ((n KS + s) 64 + l) 4 + j holds row 16 n + l % 16, column 16 s + 4 (l / 16) + j
// of the [rows][taps * columns] matrix.  wt: rows co, columns (t, ci); wb, for
// the backward data product: rows ci, columns (t, co).  One launch for all
// layers (blockIdx.y).
__global__ void k_bf16(const float* __restrict__ params, uint16_t* __restrict__ wt_all,
                       uint16_t* __restrict__ wb_all, const WeightLayer* __restrict__ layers)
{
  const WeightLayer L = layers[blockIdx.y];
  const float* w = params + L.w_off;
  uint16_t* wt = wt_all + L.w_off;
  uint16_t* wb = wb_all + L.w_off;
  const int total = L.cout * L.taps * L.cin;
  const auto place = [](int row, int col, int ks) {
    const int l = ((col & 15) >> 2) * 16 + (row & 15);
    return (((row >> 4) * ks + (col >> 4)) * 64 + l) * 4 + (col & 3);
  };
  for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    const int ci = i % L.cin, t = (i / L.cin) % L.taps, co = i / (L.cin * L.taps);
    const uint16_t h = f2bf(w[i]);
    wt[place(co, t * L.cin + ci, L.taps * L.cin / 16)] = h;
    wb[place(ci, t * L.cout + co, L.taps * L.cout / 16)] = h;
  }
}

// A training batch: sample idx[b]'s charges into the leading rows of xb[b]
// (its padding rows stay zero), its field into tb[b], its conditioning into ub[b].
__global__ __launch_bounds__(256) void k_stage(BatchArgs a)
{
  const int b = blockIdx.y;
  const size_t i = a.idx[b];
  const float4* x = reinterpret_cast<const float4*>(a.x + i * a.row_x);
  float4* xo = reinterpret_cast<float4*>(a.xb + (size_t)b * a.stride_x);
  for (int e = blockIdx.x * 256 + threadIdx.x; e < a.row_x / 4; e += gridDim.x * 256) xo[e] = x[e];
  const float* y = a.y + i * a.row_y;
  float* yo = a.tb + (size_t)b * a.row_y;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < a.row_y; e += gridDim.x * 256) yo[e] = y[e];
  if (blockIdx.x == 0 && threadIdx.x == 0) a.ub[b] = (a.u[i] - a.mu) * a.inv_sigma;
}

// rows idx[i] of src (row floats each) -> dst[i]
__global__ void k_gather(const float* __restrict__ src, const uint32_t* __restrict__ idx,
                         float* __restrict__ dst, int n, int row)
{
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (size_t)n * row) return;
  const size_t i = e / row, k = e % row;
  dst[e] = src[(size_t)idx[i] * row + k];
}

}  // namespace

hipError_t conv(const ConvArgs& a, hipStream_t s)
{
  const int P = a.B * a.Zout;   // dyn_b <= B: the grid covers the largest count
  const int waves = a.Cout / 16;
  if (P >= kConvTwoTiles)
    hipLaunchKernelGGL(k_conv<2>, dim3(cdiv(P, 32)), dim3(64 * waves), conv_lds(a.taps, a.Cin, 2),
                       s, a);
  else
    hipLaunchKernelGGL(k_conv<1>, dim3(cdiv(P, 16)), dim3(64 * waves), conv_lds(a.taps, a.Cin, 1),
                       s, a);
  return hipGetLastError();
}

hipError_t wgrad(const WgradArgs& a, hipStream_t s)
{
  const int tasks = a.taps * (a.Cout / 16) * (a.Cin / 16) * cdiv(a.B * a.Zout, kWgradChunk);
  hipLaunchKernelGGL(k_wgrad, dim3(tasks), dim3(64 * kWaves), 0, s, a);
  return hipGetLastError();
}

hipError_t film(const float* params, const FilmLayer* layers, int nlayers, const float* u,
                const uint32_t* dyn_b, int B, float* scale, hipStream_t s)
{
  hipLaunchKernelGGL(k_film, dim3(64, nlayers), dim3(256), 0, s, params, layers, nlayers, u, dyn_b,
                     B, scale, B);
  return hipGetLastError();
}

hipError_t film_bwd(const float* dy, const float* pre, const float* scale, float* dpre,
                    float* part, int B, int Z, int C, hipStream_t s)
{
  hipLaunchKernelGGL(k_film_bwd, dim3(B, film_slabs(Z)), dim3(256), 0, s, dy, pre, scale, dpre,
                     part, Z, C);
  return hipGetLastError();
}

hipError_t film_sum(const FilmLayer* layers, int nlayers, const float* part, const float* u,
                    float* g, int B, hipStream_t s)
{
  hipLaunchKernelGGL(k_film_sum, dim3(cdiv(kMaxCout, 16), nlayers), dim3(256), 0, s, layers, part,
                     u, g, B);
  return hipGetLastError();
}

hipError_t loss(const float* y, const float* tgt, float* dy, float* l, int Z0, int Cpad, int zn,
                int cout, float inv_scale, int B, hipStream_t s)
{
  hipLaunchKernelGGL(k_loss, dim3(B), dim3(kLossBlock), 0, s, y, tgt, dy, l, Z0, Cpad, zn, cout,
                     inv_scale, B);
  return hipGetLastError();
}

hipError_t adam(float* w, const float* g, float* m, float* v, int n, float lr_t, float b1,
                float b2, float eps, hipStream_t s)
{
  hipLaunchKernelGGL(k_adam, dim3(cdiv(n, 256)), dim3(256), 0, s, w, g, m, v, n, lr_t, b1, b2,
                     eps);
  return hipGetLastError();
}

hipError_t bf16_copies(const float* params, uint16_t* wt, uint16_t* wb, const WeightLayer* layers,
                       int nlayers, hipStream_t s)
{
  hipLaunchKernelGGL(k_bf16, dim3(16, nlayers), dim3(256), 0, s, params, wt, wb, layers);
  return hipGetLastError();
}

hipError_t stage(const BatchArgs& a, hipStream_t s)
{
  hipLaunchKernelGGL(k_stage, dim3(4, a.B), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t gather(const float* src, const uint32_t* idx, float* dst, int n, int row, hipStream_t s)
{
  const size_t total = (size_t)n * row;
  hipLaunchKernelGGL(k_gather, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, src, idx,
                     dst, n, row);
  return hipGetLastError();
}

}  // namespace unet
}  // namespace hps
