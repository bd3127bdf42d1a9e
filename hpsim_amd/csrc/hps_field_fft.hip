// hps_field_fft.hip -- the grouped field product of a batch in the frequency
// domain along z.
//
// The grouped product (hps_field_gemm.hip) evaluates, for every remeshing
// member's column p and its aspect class c,
//
//   W[p][(rp, comp)][zp] = sum over rs, zs of S_c[rp][rs][comp][zp - zs] q[p][rs][zs]
//
// for zp = 0 .. nz: per pair of rings a convolution along z with the signed
// offset table S (offsets 1 - nz .. nz, the Green's entries of
// UpdateFldTbl1Kernel, space_charge_kernel.cu:38-100).  With L = 2 nz the
// circular convolution of the zero-padded charges with S laid out by offset
// modulo L has no wrap-around for these zp, so
//
//   W[p][row][.] = IDFT_L( sum over rs of S^_c[row][rs][f] q^_p[rs][f] )
//
// with ^ the DFT of length L (row = 2 rp + comp).  Per frequency f the sum
// over rs is a complex matrix product (2 (nr + 1) rows x nr rings x the
// columns of the class), a real product of twice the size, on the FP32 matrix
// cores or, for a class with few columns, on the vector unit; the transforms
// are radix-2 FFTs in LDS.  Per column
// this is about 2 (L/2 + 1) x 2(nr+1) x 2 nr x 2 flops for the product plus
// the transforms, against 2 x 2(nr+1)(nz+1) x nr nz for the direct product:
// 40 times fewer at 64 x 256.
//
// Launch sequence (one "spectral" shape of launch_gemm_product; it writes
// the same w[p][m] layout as the direct product with one K split, so the
// store, audit and capture kernels read it unchanged):
//   k_fft_forward  transforms of the offset tables of the slots in use whose
//                  spectrum is not that of their class, and of the charges of
//                  every member with product columns (straight from its
//                  histogram, once for its three columns)
//   k_fft_product  the complex products; marks the spectra as current
//   k_fft_inverse  inverse transforms, W[p][m] for zp = 0 .. nz
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "hps_internal.hpp"

namespace hps {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kFftThreads = 256;
constexpr int kFftElems = 2048;        // complex entries of a workgroup's rows: eight a thread
constexpr int kFftMaxL = 4096;         // longest transform (then one row per workgroup)
constexpr int kProdVec = 4;            // most columns of a slot for the vector product
constexpr int kProdNT = 32;            // columns per matrix-core tile
constexpr int kProdMaxK = 128;         // 2 nr: the real K of the product (nr <= 64)

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ f4 mfma(float a, float b, f4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t ilog2(uint32_t v) { return 31u - __builtin_clz(v); }

// LDS slot of entry i: a gap after every eighth, so that neither the
// bit-reversed stores nor the strided passes meet on one bank.
__device__ __forceinline__ uint32_t slot_of(uint32_t i) { return i + (i >> 3); }
constexpr int kFftLds = kFftMaxL + kFftMaxL / 8;

// Stages b .. b + B - 1 of the radix-2 transforms on `total` entries (rows of
// L, a power of two): 2^B entries per thread in registers.
template <int B>
__device__ __forceinline__ void fft_pass(float2* x, const float2* tw, uint32_t L, uint32_t total,
                                         uint32_t b)
{
  constexpr int N = 1 << B;
  for (uint32_t g = threadIdx.x; g < total >> B; g += kFftThreads) {
    const uint32_t low = g & ((1u << b) - 1), base = (g >> b << (b + B)) | low;
    float2 v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = x[slot_of(base + ((uint32_t)j << b))];
#pragma unroll
    for (int s = 0; s < B; ++s) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if (j >> s & 1) continue;
        const uint32_t k = low + ((uint32_t)(j & ((1 << s) - 1)) << b);
        const float2 c = cmul(v[j | 1 << s], tw[k * (L >> (b + s + 1))]);
        const float2 a = v[j];
        v[j] = make_float2(a.x + c.x, a.y + c.y);
        v[j | 1 << s] = make_float2(a.x - c.x, a.y - c.y);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) x[slot_of(base + ((uint32_t)j << b))] = v[j];
  }
  __syncthreads();
}

// In-place forward DFT (exponent -2 pi i f k / L) of `cnt` rows of length L
// in LDS, entry k of row r stored at slot_of(r L + bit-reversed k): log2(L)
// radix-2 stages, three to a pass through LDS (a pass a stage took a barrier
// and a dependent LDS round trip for every stage: 18 -> 7 us for 21 columns
// of L = 256); tw[k] = exp(-2 pi i k / L), k < L / 2.  All threads of the
// workgroup take part, after a barrier; the rows are in order on return.
__device__ __forceinline__ void fft_rows(float2* x, const float2* tw, uint32_t L, uint32_t cnt)
{
  const uint32_t lg = ilog2(L), total = cnt * L;
  uint32_t b = 0;
  for (; b + 3 <= lg; b += 3) fft_pass<3>(x, tw, L, total, b);
  if (lg - b == 2) fft_pass<2>(x, tw, L, total, b);
  else if (lg - b == 1) fft_pass<1>(x, tw, L, total, b);
}

__device__ __forceinline__ uint32_t reversed(uint32_t k, uint32_t lg) { return __brev(k) >> (32 - lg); }

__host__ __device__ __forceinline__ uint32_t fft_rows_per_wg(uint32_t L)
{
  return L < (uint32_t)kFftElems ? kFftElems / L : 1;
}

__device__ __forceinline__ void load_twiddles(float2* tw_s, const float2* tw, uint32_t L)
{
  for (uint32_t k = threadIdx.x; k < L / 2; k += blockDim.x) tw_s[k] = tw[k];
}

// Spectra of two real rows transformed together as x = a + i b: for
// f = 0 .. L/2, A[f] = (X[f] + conj X[-f]) / 2 and B[f] = (X[f] - conj X[-f]) / (2 i).
// (row at entry i0)
__device__ __forceinline__ void split_real_pair(const float2* x, uint32_t i0, uint32_t L, uint32_t f,
                                                float2& A, float2& B)
{
  const float2 u = x[slot_of(i0 + f)], v = x[slot_of(i0 + ((L - f) & (L - 1)))];
  A = make_float2(0.5f * (u.x + v.x), 0.5f * (u.y - v.y));
  B = make_float2(0.5f * (u.y + v.y), -0.5f * (u.x - v.x));
}

// Whether slot s is used at this kick point (slot_count > 0) and its spectrum
// is not that of the class it holds.
__device__ __forceinline__ bool stale_slot(const GemmState* gs, const int32_t* spec_class, uint32_t s)
{
  return gs->slot_count[s] > 0 && spec_class[s] != gs->slot_class[s];
}

}  // namespace

// ---- forward transforms ---------------------------------------------------------

// Grid-stride over units of fft_rows_per_wg rows: first the stale slots'
// offset tables, then the members' charges.
//
// Tables: S^[slot][f][rs][row], row = 2 rp + comp: the offset rows of (rp,
// rs), both components transformed together (x = E_r + i E_z), laid out by
// offset modulo L (k <= nz: offset k at o = k + nz - 1; k > nz: offset k - L
// at o = k - nz - 1).  The product reads it along `row`.
//
// Charges: q^[m][f][rs], rings rs and rs + 1 transformed together,
// zero-padded from nz to L; the FP32 charge is the histogram's fixed point
// rounded once (k_gemm_pack's value).
__global__ __launch_bounds__(kFftThreads) void k_fft_forward(
    const GemmState* __restrict__ gs, const GemmMember* __restrict__ mem, uint32_t nmem,
    const int32_t* __restrict__ pos_exact, const int32_t* __restrict__ spec_class,
    const float* __restrict__ tables, float2* __restrict__ shat, float2* __restrict__ qhat,
    const float2* __restrict__ tw, uint32_t nr, uint32_t nz)
{
  __shared__ float2 x[kFftLds];
  __shared__ float2 tw_s[kFftMaxL / 2];
  __shared__ uint32_t slots[kGemmSlots];
  static_assert(kGemmSlots == 64, "one wave lists the slots");
  if (gs->nrem == 0) return;
  const uint32_t t = threadIdx.x;
  uint32_t nlist = 0;
  {   // every wave counts, the first one lists
    const uint32_t s = t & 63;
    const bool need = stale_slot(gs, spec_class, s);
    const uint64_t bal = __ballot(need);
    nlist = (uint32_t)__popcll(bal);
    if (t < 64 && need) slots[__popcll(bal & ((1ull << s) - 1))] = s;
  }
  const uint32_t L = 2 * nz, F = nz + 1, R = 2 * (nr + 1), lg = ilog2(L);
  const uint32_t rows = fft_rows_per_wg(L);
  const uint32_t tpairs = (nr + 1) * nr, tgroups = (tpairs + rows - 1) / rows;
  const uint32_t qpairs = nr / 2, qgroups = (qpairs + rows - 1) / rows;
  const uint32_t tunits = nlist * tgroups, units = tunits + nmem * qgroups;
  const size_t slot_sz = (size_t)(nr + 1) * nr * 4 * nz;
  load_twiddles(tw_s, tw, L);
  for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
    __syncthreads();   // previous unit done with x; twiddles and list in place
    if (u < tunits) {
      // pair pr = rs (nr + 1) + rp: neighbouring rows of S^ in a workgroup
      const uint32_t slot = slots[u / tgroups];
      const uint32_t pr0 = (u % tgroups) * rows, cnt = min(rows, tpairs - pr0);
      for (uint32_t e = t; e < cnt * L; e += kFftThreads) {
        const uint32_t r = e >> lg, k = e & (L - 1), pr = pr0 + r;
        const uint32_t rs = pr / (nr + 1), rp = pr - rs * (nr + 1);
        const float* row = tables + slot * slot_sz + (size_t)(rp * nr + rs) * 4 * nz;
        const uint32_t o = k <= nz ? k + nz - 1 : k - nz - 1;
        x[slot_of((r << lg) + reversed(k, lg))] = make_float2(row[o], row[2 * nz + o]);
      }
      __syncthreads();
      fft_rows(x, tw_s, L, cnt);
      for (uint32_t e = t; e < cnt * F; e += kFftThreads) {
        const uint32_t r = e % cnt, f = e / cnt, pr = pr0 + r;
        const uint32_t rs = pr / (nr + 1), rp = pr - rs * (nr + 1);
        float2 a, b;
        split_real_pair(x, r << lg, L, f, a, b);
        float2* dst = shat + (((size_t)slot * F + f) * nr + rs) * R + 2 * rp;
        dst[0] = a;
        dst[1] = b;
      }
      continue;
    }
    const uint32_t v = u - tunits, m = v / qgroups;
    if (pos_exact[kGemmCols * m] < 0) continue;   // no product columns
    const int64_t* bins = mem[m].bins;
    const uint32_t pr0 = (v % qgroups) * rows, cnt = min(rows, qpairs - pr0);
    for (uint32_t e = t; e < cnt * L; e += kFftThreads) {
      const uint32_t r = e % cnt, k = e / cnt, rs = 2 * (pr0 + r);
      float2 q = make_float2(0.f, 0.f);
      if (k < nz)
        q = make_float2((float)((double)bins[k * nr + rs] * 0x1p-36),
                        (float)((double)bins[k * nr + rs + 1] * 0x1p-36));
      x[slot_of((r << lg) + reversed(k, lg))] = q;
    }
    __syncthreads();
    fft_rows(x, tw_s, L, cnt);
    for (uint32_t e = t; e < cnt * F; e += kFftThreads) {
      const uint32_t r = e % cnt, f = e / cnt, rs = 2 * (pr0 + r);
      float2 a, b;
      split_real_pair(x, r << lg, L, f, a, b);
      float2* dst = qhat + ((size_t)m * F + f) * nr + rs;
      dst[0] = a;
      dst[1] = b;
    }
  }
}

// ---- the product per frequency --------------------------------------------------

// W^[p][f][row] = sum over rs of S^[slot][f][row][rs] q^[m][f][rs] for the
// columns p (of member m = perm[p]) of slot's class, as the real chain
//   Re: fma(Re S, Re q, .) then fma(-Im S, Im q, .),  Im: fma(Im S, Re q, .)
//   then fma(Re S, Im q, .),  rs ascending,
// which is also what v_mfma_f32_16x16x4f32 computes (an ascending chain of
// fused multiply-adds, checked bit for bit on the device), so both forms
// below give the same bits.
//
// A slot of at most kProdVec columns takes the vector form: the product is
// then bound by reading S^ (17 MB a slot at 64 x 256), and a matrix tile
// would multiply 12 to 15 empty columns for it (four members on 64 x 256:
// 111 -> 48 us a kick point; seven on 32 x 128: 32 -> 17 us).  One lane per
// (f, row), S^ coalesced along row, kRing rings in flight; the charges of a
// frequency are the same address for its lanes.  kProdVec of 2 / 4 / 6 / 8: 57 /
// 48 / 54 / 59 us for the former, 17.8 / 16.6 / 16.6 / 16.6 for the latter.
template <int NC>
__device__ __forceinline__ void product_rows(const float2* __restrict__ S,
                                             const float2* __restrict__ qhat,
                                             float2* __restrict__ what,
                                             const uint32_t* __restrict__ perm, uint32_t p0,
                                             uint32_t idx, uint32_t nr, uint32_t R, uint32_t F)
{
  const uint32_t f = idx / R, row = idx - f * R;
  if (f >= F) return;
  S += (size_t)f * nr * R + row;
  const float2* q[NC];
  float2 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    q[c] = qhat + ((size_t)perm[p0 + c] * F + f) * nr;
    acc[c] = make_float2(0.f, 0.f);
  }
  constexpr uint32_t kRing = 8;
  for (uint32_t r0 = 0; r0 < nr; r0 += kRing) {
    float2 a[kRing], b[NC][kRing];
#pragma unroll
    for (uint32_t u = 0; u < kRing; ++u) {
      const uint32_t rs = min(r0 + u, nr - 1);
      a[u] = S[(size_t)rs * R];
#pragma unroll
      for (int c = 0; c < NC; ++c) b[c][u] = q[c][rs];
    }
#pragma unroll
    for (uint32_t u = 0; u < kRing; ++u) {
      if (r0 + u >= nr) break;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        acc[c].x = ::fmaf(a[u].x, b[c][u].x, acc[c].x);
        acc[c].y = ::fmaf(a[u].y, b[c][u].x, acc[c].y);
        acc[c].x = ::fmaf(-a[u].y, b[c][u].y, acc[c].x);
        acc[c].y = ::fmaf(a[u].x, b[c][u].y, acc[c].y);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) what[((size_t)(p0 + c) * F + f) * R + row] = acc[c];
}

// The matrix form of one column tile (p0 .. p0 + nb - 1, kG groups of 16) at
// frequency f: M' = 2 R rows (m' = 2 row + part: part 0 the real, 1 the
// imaginary part) by K' = 2 nr (k' = 2 rs + c: c 0 the real, 1 the imaginary
// part of q^) with A'[2 row][2 rs] = Re S^, A'[2 row][2 rs + 1] = -Im S^,
// A'[2 row + 1][2 rs] = Im S^, A'[2 row + 1][2 rs + 1] = Re S^.  The tile's
// charge spectra are staged in LDS; each wave takes 16-row tiles of M' in
// turn and reads S^ through the caches.
template <int kG>
__device__ __forceinline__ void product_tile(const float2* __restrict__ A,
                                             const float2* __restrict__ qhat,
                                             float2* __restrict__ what,
                                             const uint32_t* __restrict__ perm, uint32_t p0,
                                             uint32_t nb, uint32_t f, uint32_t nr, uint32_t R,
                                             uint32_t F, float* b_lds)
{
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t Kp = 2 * nr, Mp = 2 * R, pitch = Kp + 1, mtiles = (Mp + 15) / 16;
  for (uint32_t e = t; e < 16 * kG * Kp; e += kFftThreads) {
    const uint32_t j = e / Kp, kk = e % Kp;
    float v = 0.f;
    if (j < nb) {
      const float2 c = qhat[((size_t)perm[p0 + j] * F + f) * nr + kk / 2];
      v = (kk & 1) ? c.y : c.x;
    }
    b_lds[j * pitch + kk] = v;
  }
  __syncthreads();
  for (uint32_t mt = wave; mt < mtiles; mt += kFftThreads / 64) {
    f4 acc[kG];
#pragma unroll
    for (int g = 0; g < kG; ++g) acc[g] = f4{0.f, 0.f, 0.f, 0.f};
    const uint32_t m = mt * 16 + (lane & 15);     // this lane's row of A'
    const uint32_t row = m / 2, part = m & 1;
    const bool mrow = m < Mp;
    for (uint32_t k4 = 0; k4 < Kp; k4 += 4) {
      const uint32_t kk = k4 + (lane >> 4);
      float a = 0.f;
      if (mrow) {
        const float2 s = A[(size_t)(kk / 2) * R + row];
        // part 0: (Re, -Im); part 1: (Im, Re) for c = 0, 1
        a = part == 0 ? ((kk & 1) ? -s.y : s.x) : ((kk & 1) ? s.x : s.y);
      }
#pragma unroll
      for (int g = 0; g < kG; ++g)
        acc[g] = mfma(a, b_lds[(g * 16 + (lane & 15)) * pitch + kk], acc[g]);
    }
    // D[m][n]: n = lane % 16, m = 4 (lane / 16) + i
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      const uint32_t j = g * 16 + (lane & 15);
      if (j >= nb) continue;
      float* out = (float*)(what + ((size_t)(p0 + j) * F + f) * R);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t mo = mt * 16 + 4 * (lane >> 4) + i;
        if (mo < Mp) out[mo] = acc[g][i];   // m' = 2 row + part: interleaved complex
      }
    }
  }
}

// Grid-stride over units: a slot of at most kProdVec columns has
// ceil(F R / kFftThreads) of them (lanes of product_rows), any other F per
// tile of kProdNT columns.
__global__ __launch_bounds__(kFftThreads) void k_fft_product(const GemmState* __restrict__ gs,
                                                             const uint32_t* __restrict__ perm,
                                                             int32_t* spec_class,
                                                             const float2* __restrict__ shat,
                                                             const float2* __restrict__ qhat,
                                                             float2* __restrict__ what,
                                                             uint32_t nr, uint32_t nz)
{
  __shared__ uint32_t s_start[kGemmSlots], s_count[kGemmSlots], s_unit[kGemmSlots + 1];
  __shared__ float b_lds[kProdNT * (kProdMaxK + 1)];
  if (gs->nrem == 0) return;
  const uint32_t t = threadIdx.x;
  const uint32_t F = nz + 1, R = 2 * (nr + 1);
  const uint32_t vunits = (F * R + kFftThreads - 1) / kFftThreads;
  if (t < kGemmSlots) {
    const uint32_t c = gs->slot_count[t];
    s_start[t] = gs->slot_start[t];
    s_count[t] = c;
    uint32_t n = c == 0 ? 0 : c <= (uint32_t)kProdVec ? vunits : (c + kProdNT - 1) / kProdNT * F;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {   // inclusive scan over the slots
      const uint32_t v = __shfl_up(n, o, 64);
      if (t >= o) n += v;
    }
    s_unit[t + 1] = n;
    if (t == 0) s_unit[0] = 0;
    // the spectra k_fft_forward brought up to date
    if (blockIdx.x == 0 && c > 0) spec_class[t] = gs->slot_class[t];
  }
  __syncthreads();
  const uint32_t units = s_unit[kGemmSlots];
  uint32_t slot = 0;
  for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
    while (u >= s_unit[slot + 1]) ++slot;
    const uint32_t v = u - s_unit[slot], count = s_count[slot], start = s_start[slot];
    const float2* S = shat + (size_t)slot * F * nr * R;
    if (count <= (uint32_t)kProdVec) {
      const uint32_t idx = v * kFftThreads + t;
      switch (count) {
        case 1: product_rows<1>(S, qhat, what, perm, start, idx, nr, R, F); break;
        case 2: product_rows<2>(S, qhat, what, perm, start, idx, nr, R, F); break;
        case 3: product_rows<3>(S, qhat, what, perm, start, idx, nr, R, F); break;
        default: product_rows<4>(S, qhat, what, perm, start, idx, nr, R, F); break;
      }
      continue;
    }
    const uint32_t f = v % F, p0 = start + v / F * kProdNT;
    const uint32_t nb = min((uint32_t)kProdNT, start + count - p0);
    __syncthreads();   // the previous unit is done with b_lds
    if (nb <= 16)
      product_tile<1>(S + (size_t)f * nr * R, qhat, what, perm, p0, nb, f, nr, R, F, b_lds);
    else
      product_tile<2>(S + (size_t)f * nr * R, qhat, what, perm, p0, nb, f, nr, R, F, b_lds);
  }
}

// ---- inverse transforms -----------------------------------------------------------

// w[p][(2 rp + comp) (nz + 1) + zp] for zp = 0 .. nz: the two components of
// rp transformed back together, z = IDFT(E_r^ + i E_z^) = conj(DFT(conj(.))) / L
// with the spectra extended by Hermitian symmetry.  Grid-stride over (column,
// group of radii).
__global__ __launch_bounds__(kFftThreads) void k_fft_inverse(const GemmState* __restrict__ gs,
                                                             const float2* __restrict__ what,
                                                             float* __restrict__ w,
                                                             const float2* __restrict__ tw,
                                                             uint32_t nr, uint32_t nz)
{
  __shared__ float2 x[kFftLds];
  __shared__ float2 tw_s[kFftMaxL / 2];
  if (gs->nrem == 0) return;
  const uint32_t L = 2 * nz, F = nz + 1, R = 2 * (nr + 1), lg = ilog2(L);
  const uint32_t M = R * (nz + 1);
  const uint32_t rows = fft_rows_per_wg(L);
  const uint32_t groups = (nr + 1 + rows - 1) / rows;
  const uint32_t units = gs->nrem * groups;
  const float inv_l = 1.0f / (float)L;
  load_twiddles(tw_s, tw, L);
  for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
    const uint32_t p = u / groups, rp0 = (u % groups) * rows;
    const uint32_t cnt = min(rows, nr + 1 - rp0);
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < cnt * F; e += kFftThreads) {
      const uint32_t r = e % cnt, f = e / cnt, rp = rp0 + r;
      const float2* src = what + ((size_t)p * F + f) * R + 2 * rp;
      const float2 a = src[0], b = src[1];
      // Z = A + i B, stored conjugated for the forward transform
      x[slot_of((r << lg) + reversed(f, lg))] = make_float2(a.x - b.y, -(a.y + b.x));
      if (f > 0 && f < nz) {                           // X[L - f] = conj X[f]
        const float ay = -a.y, by = -b.y;
        x[slot_of((r << lg) + reversed(L - f, lg))] = make_float2(a.x - by, -(ay + b.x));
      }
    }
    __syncthreads();
    fft_rows(x, tw_s, L, cnt);
    for (uint32_t e = threadIdx.x; e < cnt * (nz + 1); e += kFftThreads) {
      const uint32_t r = e / (nz + 1), zp = e % (nz + 1), rp = rp0 + r;
      const float2 z = x[slot_of((r << lg) + zp)];     // conj of the inverse, times L
      float* out = w + (size_t)p * M;
      out[(rp * 2 + 0) * (nz + 1) + zp] = z.x * inv_l;
      out[(rp * 2 + 1) * (nz + 1) + zp] = -z.y * inv_l;
    }
  }
}

// ---- launcher -----------------------------------------------------------------------

bool fft_product_supported(uint32_t nr, uint32_t nz)
{
  const uint32_t L = 2 * nz;
  return nr >= 2 && nr % 2 == 0 && (L & (L - 1)) == 0 && L >= 8 &&
         L <= (uint32_t)kFftMaxL && 2 * nr <= (uint32_t)kProdMaxK;
}

// Workgroups a CU: the transforms' 52 KB of LDS leave room for three, the
// product's 17 KB for nine.  Four members on 64 x 256, us a kick point: the
// forward transforms 14.3 / 11.7 / 11.5 with one / two / four, the product 57 /
// 48 / 48 with four / eight / sixteen; seven members on 32 x 128 differ by less
// than the runs.
hipError_t launch_fft_product(const GemmMember* mem, uint32_t nmem, const GemmState* gs,
                              const uint32_t* perm, const int32_t* pos_exact,
                              const float* tables, float* w, const FftBufs& fb, uint32_t nr,
                              uint32_t nz, uint32_t cus, hipStream_t s)
{
  hipLaunchKernelGGL(k_fft_forward, dim3(cus * 2), dim3(kFftThreads), 0, s, gs, mem, nmem,
                     pos_exact, fb.spec_class, tables, fb.shat, fb.qhat, fb.tw, nr, nz);
  hipLaunchKernelGGL(k_fft_product, dim3(cus * 8), dim3(kFftThreads), 0, s, gs, perm,
                     fb.spec_class, fb.shat, fb.qhat, fb.what, nr, nz);
  hipLaunchKernelGGL(k_fft_inverse, dim3(cus * 2), dim3(kFftThreads), 0, s, gs, fb.what, w,
                     fb.tw, nr, nz);
  return hipGetLastError();
}

}  // namespace hps
