// hps_kernels.hip -- gfx950 kernels of the tracking engine.
//
// Kernel families (one HBM sweep each):
//   k_segment  SCHEFF kick of the previous kick point + every element map up
//              to the next kick point, fused in registers, + per-chunk beam
//              moments the next kick needs (reference: SimulatePartialDrift/
//              HalfQuad/RFGap kernels, ApplySpchKickKernel, and the
//              reductions of Beam::UpdateStatForSpaceCharge up to the x/y
//              moments); k_seg_final finishes them in one workgroup.
//   k_phase    per-chunk relative-phase moments; k_phase_final finishes them
//              and runs the Scheff::Start control logic on the device (no
//              host round trip per kick).
//   k_sc_build / k_field_wave   the SCHEFF rebuild (Green's table and charge
//              deposit in one launch, then the field sum), run only when the
//              control step asks for a remesh (flag in device memory).
// Reductions follow one canonical order (see kChunk): lane sums of 4
// particles strided by 256, halving tree over 256 lanes, halving tree over
// the chunk partials zero-padded to a power of two.  The grid kernels write
// one partial per chunk; a one-workgroup kernel launched after them performs
// the cross-chunk tree (kernel order makes the partials visible, with no
// device-wide fence per workgroup).
#include "hps_internal.hpp"

namespace hps {

// hps_push_fast.hip builds this file a second time with HPS_FAST_PUSH
// defined and reciprocal division; that build's kernels and launchers live
// in hps::fast.
#ifdef HPS_FAST_PUSH
namespace fast {
#endif

namespace {

constexpr int kBlock = 256;

// Loads and stores through global-address-space pointers.  Pointers that a
// kernel reads from device memory (the per-simulation records of the
// batched launches) are generic to the compiler, which then emits flat
// accesses (64-bit VGPR addresses, waits on both memory counters); every
// buffer of the engine is global memory.
template <class T>
__device__ __forceinline__ T gld(const T* p, size_t i)
{
  return ((const __attribute__((address_space(1))) T*)p)[i];
}

template <class T>
__device__ __forceinline__ void gst(T* p, size_t i, T v)
{
  ((__attribute__((address_space(1))) T*)p)[i] = v;
}

// A barrier for what the workgroup exchanges through LDS: __syncthreads also
// waits for the wave's outstanding global stores.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// --- canonical reductions -------------------------------------------------

// Canonical halving tree over the 256 lane values of Q sums (levels 128 and
// 64 through LDS, 32..1 with wavefront shuffles: lane i adds lane i + o at
// every level, the same pairing as the serial definition), plus an integer
// count and a max carried alongside.  The results are valid in thread 0;
// red must hold Q*256 doubles, ured 256 words.
template <int Q>
__device__ __forceinline__ void block_reduce(double (&v)[Q], uint32_t& cnt, double& mx, double* red,
                                             uint32_t* ured, double* mred, int t)
{
#pragma unroll
  for (int q = 0; q < Q; ++q) red[q * kBlock + t] = v[q];
  ured[t] = cnt;
  mred[t] = mx;
  __syncthreads();
  if (t < 128) {
#pragma unroll
    for (int q = 0; q < Q; ++q) red[q * kBlock + t] = red[q * kBlock + t] + red[q * kBlock + t + 128];
    ured[t] += ured[t + 128];
    mred[t] = ::fmax(mred[t], mred[t + 128]);
  }
  __syncthreads();
  if (t < 64) {
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = red[q * kBlock + t] + red[q * kBlock + t + 64];
    cnt = ured[t] + ured[t + 64];
    mx = ::fmax(mred[t], mred[t + 64]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
      for (int q = 0; q < Q; ++q) v[q] = v[q] + __shfl_down(v[q], o, 64);
      cnt += __shfl_down(cnt, o, 64);
      mx = ::fmax(mx, __shfl_down(mx, o, 64));
    }
  }
  __syncthreads();
}

// Largest of the 256 lane values (valid in thread 0).  The comparison
// a < v keeps a when v is NaN; a maximum does not depend on the order.
// buf holds kBlock / 64 doubles.
__device__ __forceinline__ double block_max(double v, double* buf, int t)
{
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double u = __shfl_down(v, o, 64);
    v = v < u ? u : v;
  }
  if ((t & 63) == 0) buf[t >> 6] = v;
  __syncthreads();
  double r = 0.0;
  if (t == 0) {
    r = buf[0];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) r = r < buf[w] ? buf[w] : r;
  }
  __syncthreads();
  return r;
}

// --- cross-chunk trees ------------------------------------------------------
//
// A quantity's chunk partials P[0, mpad) (zero padded to mpad, a power of two
// of at most 4,096) are summed by one wavefront: lane l holds the entries
// l + 64 m, folds them over m as the upper levels of the halving tree, and the
// lanes' values meet in shuffles.  The waves of the one workgroup take
// different quantities, so the sums need no LDS and no barrier among
// themselves; what bounds them is the memory round trip, so the loads of up
// to 16 entries a lane are issued before the first addition.

// sum of the tree over P (valid in lane 0)
template <int M>
__device__ __forceinline__ double wave_tree(const double* P, uint32_t mpad, int l)
{
  // entries m = g + kG k of batch g fold over k (the upper levels), then the
  // batches over g: (0 + 2) + (1 + 3) of four, 0 + 1 of two
  constexpr int kN = M < 16 ? M : 16, kG = M / kN;
  static_assert(kG <= 4, "at most 4,096 entries");
  const auto batch = [&](int g) {
    double r[kN];
#pragma unroll
    for (int k = 0; k < kN; ++k)
      r[k] = (M > 1 || (uint32_t)l < mpad) ? gld(P, l + 64 * (g + kG * k)) : 0.0;
#pragma unroll
    for (int h = kN / 2; h >= 1; h /= 2) {
#pragma unroll
      for (int k = 0; k < h; ++k) r[k] = r[k] + r[k + h];
    }
    return r[0];
  };
  double s;
  if constexpr (kG == 1) {
    s = batch(0);
  } else {
    constexpr int kH = kG / 2;
    double v[2] = {0.0, 0.0};
#pragma unroll 1
    for (int j = 0; j < kG; ++j) {   // 0, kH, 1, kH + 1: one batch's registers at a time
      const double x = batch((j & 1) * kH + (j >> 1));
      if ((j & 1) == 0) v[1] = x;
      else v[0] = j == 1 ? v[1] + x : v[0] + (v[1] + x);
    }
    s = v[0];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s = s + __shfl_down(s, o, 64);
  return s;
}

__device__ __forceinline__ double wave_tree_sum(const double* P, uint32_t mpad, int l)
{
  switch (mpad > 64 ? mpad / 64 : 1u) {
    case 1: return wave_tree<1>(P, mpad, l);
    case 2: return wave_tree<2>(P, mpad, l);
    case 4: return wave_tree<4>(P, mpad, l);
    case 8: return wave_tree<8>(P, mpad, l);
    case 16: return wave_tree<16>(P, mpad, l);
    case 32: return wave_tree<32>(P, mpad, l);
    default: return wave_tree<64>(P, mpad, l);
  }
}

// sum of the counts C[0, n) (valid in lane 0)
__device__ __forceinline__ uint32_t wave_count(const uint32_t* C, uint32_t n, int l)
{
  uint32_t v = 0;
#pragma unroll 16
  for (uint32_t c = l; c < n; c += 64) v += gld(C, c);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// largest of M[0, n), from v0 up (a NaN entry is never taken; valid in lane 0)
__device__ __forceinline__ double wave_max(const double* M, uint32_t n, double v0, int l)
{
  double v = v0;
#pragma unroll 8
  for (uint32_t c = l; c < n; c += 64) {
    const double u = gld(M, c);
    if (u > v) v = u;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double u = __shfl_down(v, o, 64);
    if (u > v) v = u;
  }
  return v;
}

__device__ __forceinline__ bool is_good(uint32_t loss, uint32_t lloss)
{
  return (uint32_t)(loss + lloss) == 0u;
}

// --- SCHEFF kick (ApplySpchKickKernel, space_charge_kernel.cu:572-706) -----

struct KickConst {
  double phimc, xbar, ybar, epsq, gmg, dr, dzg, hl, c2, c3, xfac, yfac;
  double er_ratio, ez_ratio, cbgcoef, r_beta, phi_ref, pl;
  double repsq, rdr, rdzg;   // rounded reciprocals of epsq, dr, dzg
  uint32_t nx, nz, adj;
  uint32_t mark;   // 0 where these are in Quick's range, else Quick::kOff
};

// The kick constants of ApplySpchKickKernel (space_charge_kernel.cu:578-640):
// the parts fixed by the control step come from ScDev (kick_prepare in
// k_phase_final); the element length, the on-mesh count (k_deposit) and the
// phase references (which a host frequency step may change) are read here.
template <class A>
__device__ __forceinline__ KickConst kick_const(const ScDev* scg, const hps_beam_stats* stg,
                                                double r_length)
{
  // read through the constant address space (scalar loads: neither record
  // changes while k_segment runs)
  typedef const __attribute__((address_space(4))) ScDev CScDev;
  typedef const __attribute__((address_space(4))) hps_beam_stats CStats;
  CScDev* sc = (CScDev*)scg;
  CStats* st = (CStats*)stg;
  KickConst k;
  k.phimc = st->phi_avg_r;
  k.xbar = sc->k_xbar;
  k.ybar = sc->k_ybar;
  k.epsq = sc->k_epsq;
  k.gmg = sc->k_gmg;
  k.dr = sc->k_dr;
  k.dzg = sc->k_dzg;
  k.nx = sc->st.nx;
  k.nz = sc->st.nz;
  k.hl = sc->k_hl;
  k.c2 = sc->k_c2;
  k.c3 = A::div_by(r_length, sc->k_bgmg, sc->k_rbgmg);
  k.repsq = sc->k_repsq;
  k.rdr = sc->k_rdr;
  k.rdzg = sc->k_rdzg;
  k.xfac = sc->k_xfac;
  k.yfac = sc->k_yfac;
  k.er_ratio = sc->k_er_ratio;
  k.ez_ratio = sc->k_ez_ratio;
  k.cbgcoef = sc->k_c1 * k.c3 * PI * 0.5 * sc->st.num_on_mesh;
  k.r_beta = sc->beta;
  k.phi_ref = st->phi_avg_good;
  k.pl = sc->k_pl;
  k.adj = sc->adj_eff;
  k.mark = sc->k_mark;
  return k;
}

// The control-step part of the kick constants, in the expressions of
// ApplySpchKickKernel; r_num_part, r_mass: the beam's size and mass.
// fld_off: of the last remesh.  Returns whether Quick covers them.
__device__ __forceinline__ bool kick_prepare(ScDev* sc, double r_beta, double r_freq,
    double r_current, double x_avg_good, double y_avg_good, double x_sig_good,
    double y_sig_good, double dr, double dz, uint32_t nz, double ratio_r, double ratio_z,
    double ratio_q, double ratio_g, uint32_t r_num_part, double r_mass, bool remesh,
    uint32_t fld_off)
{
  const double epsq = x_sig_good / y_sig_good;
  const double gmg = 1.0 / ::sqrt(1.0 - r_beta * r_beta);
  const double dzg = dz * gmg * ratio_z;
  const double wave_len = CLIGHT / r_freq;
  const double xfac = 2.0 / (epsq + 1.0);
  sc->k_xbar = x_avg_good;
  sc->k_ybar = y_avg_good;
  sc->k_epsq = epsq;
  sc->k_gmg = gmg;
  sc->k_dr = dr * ratio_r;
  sc->k_dzg = dzg;
  sc->k_hl = nz * 0.5 * dzg;
  sc->k_c1 = 5721.67 * r_current / (r_freq * 1e6 * (double)r_num_part * r_mass);
  sc->k_c2 = r_beta * gmg * wave_len / TWOPI;
  sc->k_pl = r_beta * gmg * wave_len;
  sc->k_bgmg = r_beta * gmg;
  sc->k_repsq = 1.0 / epsq;
  sc->k_rdr = 1.0 / (dr * ratio_r);
  sc->k_rdzg = 1.0 / dzg;
  sc->k_rbgmg = 1.0 / (r_beta * gmg);
  sc->k_xfac = xfac;
  sc->k_yfac = epsq * xfac;
  sc->k_er_ratio = ratio_q / (ratio_r * ratio_z * ratio_g * ratio_g);
  sc->k_ez_ratio = ratio_q / (ratio_z * ratio_z);
  if constexpr (!kBounded) return false;
  // The others follow: gmg is 1 at least, c2 and pl are products of two of
  // these, xfac and yfac at most 2.  With c1 and the ratios below 2^64 (they
  // may be 0) the field tables, kept until the next remesh, and the field
  // outside the mesh stay below 2^500.
  const uint32_t m = Quick::mark(epsq) | Quick::mark(sc->k_dr) | Quick::mark(dzg) |
                     Quick::mark(wave_len) | Quick::mark(sc->k_bgmg);
  const uint32_t c1_off = !below_range_end(sc->k_c1), table_off = remesh ? c1_off : fld_off;
  const uint32_t off = (uint32_t)Quick::off(m) | c1_off | table_off |
                       !below_range_end(sc->k_er_ratio) | !below_range_end(sc->k_ez_ratio);
  sc->fld_off = table_off;
  sc->k_mark = off ? Quick::kOff : 0u;
  return off == 0;
}

template <class A>
__device__ __forceinline__ void kick(Particle& p, const KickConst& k, const double* tbl,
                                     double r_mass, double rmass)
{
  const double phi = relative_phi(p.phi, k.phi_ref);   // phi_r of UpdateRelativePhi(true)
  const double gm1 = A::div_by(p.w, r_mass, rmass);
  const double gm = gm1 + 1.0;
  const double bgz = A::sqrt((gm - 1.0) * (gm + 1.0));
  double bgx = bgz * p.xp;
  double bgy = bgz * p.yp;
  double bgzstar = k.gmg * (bgz - k.r_beta * gm);
  const double xxbar = p.x - k.xbar;
  const double yybar = p.y - k.ybar;
  const double r2 = A::div_by(xxbar * xxbar, k.epsq, k.repsq) + yybar * yybar * k.epsq;
  double r = A::sqrt(r2);
  if (r == 0.0) r = 1.0e-8;
  const double rr = A::recip(r);
  const double xovr = A::div_by(xxbar * k.xfac, r, rr);
  const double yovr = A::div_by(yybar * k.yfac, r, rr);
  double ddz = phi - k.phimc;
  for (int guard = 0; (ddz > PI || ddz < -PI) && guard < 4096; ++guard) {
    if (ddz > 0.0) ddz -= TWOPI;
    else ddz += TWOPI;
  }
  double z = -k.c2 * ddz;
  double cbgr, cbgzs;
  if (r > k.nx * k.dr || __builtin_fabs(z) > k.hl) {
    z = -k.c2 * (phi - k.phimc);
    const double d = A::sqrt(z * z + r * r);
    p.mark |= A::mark(d);
    const double invd3 = A::div(1.0, d * d * d);
    double rod3 = r * invd3;
    double zod3 = z * invd3;
    // point charges of the neighbouring bunches (space_charge_kernel.cu:650-662)
    for (uint32_t nb = 1; nb <= k.adj; ++nb) {
      int xi = (int)nb;
      for (int lr = 0; lr < 2; ++lr) {
        const double sz = z + xi * k.pl;
        const double dd = A::sqrt(sz * sz + r * r);
        const double iv = A::div(1.0, dd * dd * dd);
        rod3 += r * iv;
        zod3 += sz * iv;
        xi = -xi;
      }
    }
    cbgr = k.cbgcoef * rod3;
    cbgzs = k.cbgcoef * zod3;
  } else {
    const double ri = A::div_by(r, k.dr, k.rdr), zj = A::div_by(z + k.hl, k.dzg, k.rdzg);
    const uint32_t i = (uint32_t)(1 + to_int(ri));
    const double a = ri - (i - 1.0);
    const double b = 1.0 - a;
    const uint32_t j = (uint32_t)(1 + to_int(zj));
    const double c = zj - (j - 1.0);
    const double d = 1.0 - c;
    const uint32_t tbl_sz = (k.nx + 1) * (k.nz + 1);
    uint32_t l = (j - 1) * (k.nx + 1) + i;
    uint32_t m = l + (k.nx + 1);
    if (m >= tbl_sz) m = tbl_sz - 1;
    if (l >= tbl_sz) l = tbl_sz - 1;
    if constexpr (std::is_same<A, Quick>::value) {   // out of its range i and j are anything
      if (m < 1) m = 1;
      if (l < 1) l = 1;
    }
    const double tl0 = gld(tbl, 2 * l), tl1 = gld(tbl, 2 * l + 1);
    const double tk0 = gld(tbl, 2 * (l - 1)), tk1 = gld(tbl, 2 * (l - 1) + 1);
    const double tm0 = gld(tbl, 2 * m), tm1 = gld(tbl, 2 * m + 1);
    const double tn0 = gld(tbl, 2 * (m - 1)), tn1 = gld(tbl, 2 * (m - 1) + 1);
    cbgr = k.er_ratio * k.c3 * (d * (a * tl0 + b * tk0) + c * (a * tm0 + b * tn0));
    cbgzs = k.ez_ratio * k.c3 * (d * (a * tl1 + b * tk1) + c * (a * tm1 + b * tn1));
  }
  bgx += cbgr * xovr;
  bgy += cbgr * yovr;
  bgzstar += cbgzs;
  const double gstar = 1.0 + 0.5 * bgzstar * bgzstar;
  const double bgzf = k.gmg * (bgzstar + k.r_beta * gstar);
  // Terms that lie below their quotient's range are lost in bgx and bgy, by
  // less than half an ulp, wherever these are in range themselves.
  p.mark |= A::mark(gm1) | A::mark(r2) | A::mark(bgx) | A::mark(bgy) | A::mark(bgzf) | k.mark;
  if (bgzf <= 0.0) {
    p.loss = 9999;
  } else {
    const double rbg = A::recip(bgzf);
    p.xp = A::div_by(bgx, bgzf, rbg);
    p.yp = A::div_by(bgy, bgzf, rbg);
    p.w *= 1.0 + A::div((gm + 1.0) * (bgzf - bgz), gm * bgz);
  }
}

// --- k_segment ---------------------------------------------------------------

// Per-chunk moments of the SCHEFF statistics (quantity order in partials):
//   0 phi, 1 x, 2 x^2, 3 y, 4 y^2, 5 w   over (loss + lloss) == 0
// plus the good count and the largest phi among particles not yet flagged
// as longitudinally lost (the chunks a new lloss flag can appear in).
constexpr int kScQ = 6;

struct RedSmem {
  double red[kMaxQ * kBlock];
  double mred[kBlock];
  uint32_t ured[kBlock];
};

// Sets the longitudinal-loss flag of every particle of chunk c beyond the
// threshold thr and recomputes the chunk's statistics partials with the new
// flags, in one pass over the chunk, on one wavefront: lane L stands for the
// canonical lanes L, L+64, L+128 and L+192 of k_segment's 256-lane order
// (each the same sequential sum over j), then folds them as levels 128 and 64
// of the halving tree before the shuffle levels 32..1 -- the same tree as
// block_reduce, so the partials are identical.  The waves of a workgroup
// rescan different chunks at the same time.
__device__ void chunk_flag_stats_wave(const BeamArrays& b, uint32_t c, double thr, int lane,
                                      const Partials& pr)
{
  static_assert(kBlock == 256, "the folds below are written for 256 canonical lanes");
  uint32_t cnt = 0;
  double mx = -__builtin_huge_val();
  // canonical lanes lane + 64 sl: the sums of one sl from its four particles,
  // all loaded (at clamped indexes) before the first is used
  const auto slot = [&](int sl, double (&acc)[kScQ]) {
    double phi[kPerLane], x[kPerLane], y[kPerLane], w[kPerLane];
    uint32_t loss[kPerLane], lloss[kPerLane];
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j) {
      const uint32_t i = c * kChunk + j * kBlock + sl * 64 + lane;
      const uint32_t k = i < b.n ? i : b.n - 1;
      phi[j] = gld(b.phi, k); x[j] = gld(b.x, k); y[j] = gld(b.y, k); w[j] = gld(b.w, k);
      loss[j] = gld(b.loss, k); lloss[j] = gld(b.lloss, k);
    }
#pragma unroll
    for (int q = 0; q < kScQ; ++q) acc[q] = 0.0;
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j) {
      const uint32_t i = c * kChunk + j * kBlock + sl * 64 + lane;
      const bool in = i < b.n;
      if (in && phi[j] > thr) {
        if (lloss[j] != 1) gst(b.lloss, i, 1u);
        lloss[j] = 1;
      }
      if (in && lloss[j] == 0) mx = ::fmax(mx, phi[j]);
      const bool g = in && is_good(loss[j], lloss[j]);
      const double vphi = g ? phi[j] : 0.0, vx = g ? x[j] : 0.0, vy = g ? y[j] : 0.0,
                   vw = g ? w[j] : 0.0;
      acc[0] = acc[0] + vphi;
      acc[1] = acc[1] + vx;
      acc[2] = acc[2] + vx * vx;
      acc[3] = acc[3] + vy;
      acc[4] = acc[4] + vy * vy;
      acc[5] = acc[5] + vw;
      cnt += g ? 1u : 0u;
    }
  };
  // (lane L + lane L+128) + (lane L+64 + lane L+192): levels 128 and 64
  double v[kScQ], h[kScQ];
#pragma unroll 1
  for (int j = 0; j < 4; ++j) {   // slots 0, 2, 1, 3
    double u[kScQ];
    slot((j & 1) * 2 + (j >> 1), u);
#pragma unroll
    for (int q = 0; q < kScQ; ++q) {
      if ((j & 1) == 0) h[q] = u[q];
      else v[q] = j == 1 ? h[q] + u[q] : v[q] + (h[q] + u[q]);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
    for (int q = 0; q < kScQ; ++q) v[q] = v[q] + __shfl_down(v[q], o, 64);
    cnt += __shfl_down(cnt, o, 64);
    mx = ::fmax(mx, __shfl_down(mx, o, 64));
  }
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < kScQ; ++q) gst(pr.sums, q * pr.mpad + c, v[q]);
    gst(pr.cnt, c, cnt);
    gst(pr.pmax, c, mx);
  }
}

// Particles of one lane in flight at a time in k_segment, per map class.
#ifndef HPS_SEG_GROUP_GAP
#define HPS_SEG_GROUP_GAP 1
#endif
#ifndef HPS_SEG_GROUP_QUAD
#define HPS_SEG_GROUP_QUAD 1
#endif
#ifndef HPS_SEG_GROUP_LIGHT
#define HPS_SEG_GROUP_LIGHT 1
#endif
constexpr int kSegGroupGap = HPS_SEG_GROUP_GAP;
constexpr int kSegGroupQuad = HPS_SEG_GROUP_QUAD;
constexpr int kSegGroupLight = HPS_SEG_GROUP_LIGHT;

// Particle i of the beam, or an excluded placeholder (loss = 1) past the end.
__device__ __forceinline__ Particle load_particle(const BeamArrays& b, uint32_t i,
                                                  uint32_t mark = 0)
{
  Particle p;
  p.loss = 1; p.lloss = 0;
  p.x = p.xp = p.y = p.yp = p.phi = p.w = 0.0;
  p.mark = mark;
  if (i < b.n) {
    p.loss = gld(b.loss, i);
    p.lloss = gld(b.lloss, i);
    p.x = gld(b.x, i); p.xp = gld(b.xp, i); p.y = gld(b.y, i); p.yp = gld(b.yp, i);
    p.phi = gld(b.phi, i); p.w = gld(b.w, i);
  }
  return p;
}

// Writes back a pushed particle that was alive on entry (the map kernels write
// only those); a new loss code is written with it.
__device__ __forceinline__ void store_particle(const BeamArrays& b, uint32_t i, const Particle& q)
{
  gst(b.x, i, q.x); gst(b.xp, i, q.xp); gst(b.y, i, q.y); gst(b.yp, i, q.yp);
  gst(b.phi, i, q.phi); gst(b.w, i, q.w);
  if (q.loss != 0) gst(b.loss, i, q.loss);
}

// The arguments of k_segment_batch, in their order.
struct SegBatchArgs {
  const SegArgs* recs;
  const uint32_t* map;
  const uint64_t* roff;
};

// This workgroup's SegArgs in memory: the one argument of k_segment and
// k_segment_wide, or its record of k_segment_batch.  The empty asm hides where
// the pointer comes from, so nothing read before is kept for what reads here.
typedef const __attribute__((address_space(4))) SegArgs SegArgsConst;

template <bool kBatch>
__device__ __forceinline__ SegArgsConst* own_args()
{
#ifdef __HIP_DEVICE_COMPILE__
  typedef const __attribute__((address_space(4))) SegBatchArgs CArgs;
  typedef const __attribute__((address_space(4))) uint32_t CMap;
  typedef const __attribute__((address_space(4))) uint64_t COff;
  uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm("" : "+s"(at));
  if constexpr (kBatch) {
    const CArgs& k = *(CArgs*)at;
    const uint32_t e = ((CMap*)(uint64_t)k.map)[blockIdx.x];
    at = (uint64_t)k.recs + ((COff*)(uint64_t)k.roff)[0] + (e >> kBatchLocalBits) * sizeof(SegArgs);
  }
  return (SegArgsConst*)at;
#else
  return nullptr;
#endif
}

// The kick and the maps of particle i once more, from memory and through Any,
// where Quick does not cover it.  Nothing is stored between, and the two share
// no value.  (With either form tried at each map k_segment took 82 to 90
// VGPRs, five waves per SIMD instead of seven; with the arguments shared, 40
// more scalar registers were spilled.)
template <int kClass, bool kBatch>
__device__ __forceinline__ void redo(uint32_t i, Particle& p)
{
  if constexpr (kBounded) {
    if (__builtin_expect(!Quick::off(p.mark), 1)) return;
#ifdef __HIP_DEVICE_COMPILE__
    asm("" : "+v"(i));
#endif
    SegArgsConst& a = *own_args<kBatch>();
    BeamArrays b;
    b.x = a.b.x; b.xp = a.b.xp; b.y = a.b.y; b.yp = a.b.yp; b.phi = a.b.phi; b.w = a.b.w;
    b.loss = a.b.loss; b.lloss = a.b.lloss;
    b.n = a.b.n;
    const double mass = a.b.mass, charge = a.b.charge;
    p = load_particle(b, i);
    if (p.loss != 0) return;
    if (a.kick && p.lloss == 0 && (i & a.kick_mask) != 0)
      kick<Any>(p, kick_const<Any>(a.sc, a.st, a.kick_len), a.fld2, mass, 0.0);
    const hps_beam_stats* st = a.st;
    const double xa = st->x_avg, ya = st->y_avg;
    for (int o = a.op_begin; o < a.op_end; ++o) {
      const OpConst& op = ((const OpConst*)a.ops)[o];
      if (p.loss == 0) apply_op<Any, kClass>(op, p, i, mass, 0.0, charge, xa, ya);
    }
  }
}

// One workgroup per 1024-particle chunk; each lane carries its four
// particles (i = chunk*1024 + j*256 + lane) through the kick, the maps and
// the store in groups of kGroup, and accumulates the chunk statistics in the
// canonical lane order (j = 0..3, from +0.0):
//   STAT_SC        0 phi, 1 x, 2 x^2, 3 y, 4 y^2, 5 w over (loss + lloss) == 0,
//                  the good count and the largest phi among particles not yet
//                  flagged as longitudinally lost;
//   STAT_APERTURE  x and y over loss == 0 and the count of loss != 0
//                  (UpdateLoss + UpdateAvgXY, simulation_engine.cu:311-312).
// The group size trades registers (waves per SIMD) against independent
// chains per wave.
template <int kClass, int kGroup, bool kBatch>
__device__ __forceinline__ void segment_body(const SegArgs& a, uint32_t c, RedSmem& sm)
{
  static_assert(kPerLane % kGroup == 0, "group must divide the particles per lane");
  const int t = threadIdx.x;
  const BeamArrays& b = a.b;
  const double xa = a.st->x_avg, ya = a.st->y_avg;
  // per-lane accumulators in LDS rows (lane t owns column t): 0..5 sums,
  // 6 largest r^2, ured count, mred max phi.  Held in LDS rather than
  // registers across the particle loop, they leave the registers to the
  // maps (14 fewer VGPRs in the RF-gap class).
  double* const acc = sm.red + t;
#pragma unroll
  for (int q = 0; q < kScQ + 1; ++q) acc[q * kBlock] = 0.0;
  sm.ured[t] = 0;
  sm.mred[t] = -__builtin_huge_val();
#pragma unroll 1
  for (int j0 = 0; j0 < (int)kPerLane; j0 += kGroup) {
    Particle p[kGroup];
    bool alive_in[kGroup];
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const uint32_t i = c * kChunk + (j0 + g) * kBlock + t;
      p[g] = load_particle(b, i, a.mark);
      alive_in[g] = i < b.n && p[g].loss == 0;
    }
    if (a.kick) {
      // the kick constants are read again for every particle group (scalar
      // loads from the scalar cache) rather than held in SGPRs across the maps
      const ScDev* scp = a.sc;
      const hps_beam_stats* stp = a.st;
      asm volatile("" : "+s"(scp), "+s"(stp));
      const KickConst k = kick_const<Usual>(scp, stp, a.kick_len);
#pragma unroll
      for (int g = 0; g < kGroup; ++g) {
        const uint32_t i = c * kChunk + (j0 + g) * kBlock + t;
        if (alive_in[g] && p[g].lloss == 0 && (i & a.kick_mask) != 0)
          kick<Usual>(p[g], k, a.fld2, b.mass, b.rmass);
      }
    }
    for (int o = a.op_begin; o < a.op_end; ++o) {
      const OpConst& op = ((const OpConst*)a.ops)[o];
#pragma unroll
      for (int g = 0; g < kGroup; ++g) {
        const uint32_t i = c * kChunk + (j0 + g) * kBlock + t;
        if (p[g].loss == 0)
          apply_op<Usual, kClass>(op, p[g], i, b.mass, b.rmass, b.charge, xa, ya);
      }
    }
#pragma unroll
    for (int g = 0; g < kGroup; ++g)
      redo<kClass, kBatch>(c * kChunk + (j0 + g) * kBlock + t, p[g]);
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const uint32_t i = c * kChunk + (j0 + g) * kBlock + t;
      const bool in = i < b.n;
      const Particle& q = p[g];
      if (alive_in[g]) store_particle(b, i, q);
      if (a.stats == STAT_SC) {
        if (in && q.lloss == 0) sm.mred[t] = ::fmax(sm.mred[t], q.phi);
        const bool gd = in && is_good(q.loss, q.lloss);
        const double vphi = gd ? q.phi : 0.0, vx = gd ? q.x : 0.0, vy = gd ? q.y : 0.0,
                     vw = gd ? q.w : 0.0;
        acc[0] = acc[0] + vphi;
        acc[kBlock] = acc[kBlock] + vx;
        acc[2 * kBlock] = acc[2 * kBlock] + vx * vx;
        acc[3 * kBlock] = acc[3 * kBlock] + vy;
        acc[4 * kBlock] = acc[4 * kBlock] + vy * vy;
        acc[5 * kBlock] = acc[5 * kBlock] + vw;
        sm.ured[t] += gd ? 1u : 0u;
        if (a.rmax && in && q.loss == 0) {
          const double tx = q.x - xa, ty = q.y - ya;
          const double r2 = tx * tx + ty * ty;
          const double r2m = acc[6 * kBlock];
          acc[6 * kBlock] = r2m < r2 ? r2 : r2m;
        }
      } else if (a.stats == STAT_APERTURE) {
        const bool ok = in && q.loss == 0;
        acc[0] = acc[0] + (ok ? q.x : 0.0);
        acc[kBlock] = acc[kBlock] + (ok ? q.y : 0.0);
        sm.ured[t] += (in && q.loss != 0) ? 1u : 0u;
      }
    }
  }
  const Partials& pr = a.pr;
  if (a.stats == STAT_SC) {
    double v[kScQ];
#pragma unroll
    for (int q = 0; q < kScQ; ++q) v[q] = acc[q * kBlock];
    const double r2m = acc[6 * kBlock];
    uint32_t cnt = sm.ured[t];
    double mx = sm.mred[t];
    block_reduce<kScQ>(v, cnt, mx, sm.red, sm.ured, sm.mred, t);
    if (t == 0) {
#pragma unroll
      for (int q = 0; q < kScQ; ++q) pr.sums[q * pr.mpad + c] = v[q];
      pr.cnt[c] = cnt;
      pr.pmax[c] = mx;
    }
    if (a.rmax) {
      const double m = block_max(r2m, sm.mred, t);
      if (t == 0) pr.rmax2[c] = m;
    }
  } else if (a.stats == STAT_APERTURE) {
    double ap[2] = {acc[0], acc[kBlock]};
    uint32_t cnt = sm.ured[t];
    double m0 = 0.0;
    block_reduce<2>(ap, cnt, m0, sm.red, sm.ured, sm.mred, t);
    if (t == 0) { pr.sums[c] = ap[0]; pr.sums[pr.mpad + c] = ap[1]; pr.cnt[c] = cnt; }
  }
}

#ifdef HPS_FAST_PUSH
// The batched push of the grouped solve (this file as built by
// hps_push_fast.hip): the same push, moments and chunk partials as
// segment_body, but only over the chunk's live particles.  Particles lost
// before the segment are never pushed.  Scattered at random among the live
// ones, they would otherwise keep their lanes of every wavefront busy (on
// the 64-beam stress batch about half the particles are lost, on average,
// over the lattice).  The workgroup first reads the loss flags of its 1,024
// particles.  A lost particle adds to the loss count (aperture statistics)
// or, when not flagged longitudinally, offers its unchanged phase to the
// largest-phase test.  The live ones are listed in particle order in LDS
// (ballots per 64-particle group, an exclusive scan over the 16 groups),
// and thread t pushes list entries t, t + 256, ...  Each sum then adds its
// terms in another order than the canonical one; that is within this
// build's error bounds, and the counts and maxima are the same.
struct LiveSmem {
  uint16_t list[kChunk];     // chunk offsets (j * 256 + lane) of the live particles
  uint32_t gcnt[kPerLane * (kBlock / 64)];
};

template <int kClass>
__device__ __forceinline__ void segment_body_live(const SegArgs& a, uint32_t c, RedSmem& sm,
                                                  LiveSmem& ls)
{
  static_assert(kBlock == 256 && kPerLane == 4, "16 groups of 64 particles per chunk");
  const int t = threadIdx.x, wave = t >> 6;
  const BeamArrays& b = a.b;
  const double xa = a.st->x_avg, ya = a.st->y_avg;
  double* const acc = sm.red + t;
#pragma unroll
  for (int q = 0; q < kScQ + 1; ++q) acc[q * kBlock] = 0.0;
  // flags of the lane's four particles; lost ones' contributions
  uint32_t nlost = 0;
  double mlost = -__builtin_huge_val();
  bool live[kPerLane];
#pragma unroll
  for (int j = 0; j < (int)kPerLane; ++j) {
    const uint32_t i = c * kChunk + j * kBlock + t;
    live[j] = false;
    if (i < b.n) {
      if (gld(b.loss, i) == 0) {
        live[j] = true;
      } else {
        ++nlost;
        if (a.stats == STAT_SC && gld(b.lloss, i) == 0) mlost = ::fmax(mlost, gld(b.phi, i));
      }
    }
  }
  sm.ured[t] = a.stats == STAT_APERTURE ? nlost : 0u;
  sm.mred[t] = mlost;
  uint64_t bal[kPerLane];
#pragma unroll
  for (int j = 0; j < (int)kPerLane; ++j) {
    bal[j] = __ballot(live[j]);
    if ((t & 63) == 0) ls.gcnt[j * 4 + wave] = (uint32_t)__popcll(bal[j]);
  }
  __syncthreads();
  uint32_t nlive = 0, base[kPerLane] = {0, 0, 0, 0};
#pragma unroll
  for (int g = 0; g < (int)(kPerLane * 4); ++g) {
    const uint32_t n = ls.gcnt[g];
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j)
      if (g < j * 4 + wave) base[j] += n;
    nlive += n;
  }
#pragma unroll
  for (int j = 0; j < (int)kPerLane; ++j) {
    if (live[j]) {
      const uint32_t below = __builtin_amdgcn_mbcnt_hi(
          (uint32_t)(bal[j] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal[j], 0u));
      ls.list[base[j] + below] = (uint16_t)(j * kBlock + t);
    }
  }
  __syncthreads();
#pragma unroll 1
  for (uint32_t sl = (uint32_t)t; sl < nlive; sl += kBlock) {
    const uint32_t i = c * kChunk + ls.list[sl];
    Particle p = load_particle(b, i);
    if (a.kick) {
      const ScDev* scp = a.sc;
      const hps_beam_stats* stp = a.st;
      asm volatile("" : "+s"(scp), "+s"(stp));
      const KickConst k = kick_const<Usual>(scp, stp, a.kick_len);
      if (p.lloss == 0 && (i & a.kick_mask) != 0)
        kick<Usual>(p, k, a.fld2, b.mass, b.rmass);
    }
    for (int o = a.op_begin; o < a.op_end; ++o) {
      const OpConst& op = ((const OpConst*)a.ops)[o];
      if (p.loss == 0) apply_op<Usual, kClass>(op, p, i, b.mass, b.rmass, b.charge, xa, ya);
    }
    store_particle(b, i, p);
    if (a.stats == STAT_SC) {
      if (p.lloss == 0) sm.mred[t] = ::fmax(sm.mred[t], p.phi);
      const bool gd = is_good(p.loss, p.lloss);
      const double vphi = gd ? p.phi : 0.0, vx = gd ? p.x : 0.0, vy = gd ? p.y : 0.0,
                   vw = gd ? p.w : 0.0;
      acc[0] = acc[0] + vphi;
      acc[kBlock] = acc[kBlock] + vx;
      acc[2 * kBlock] = acc[2 * kBlock] + vx * vx;
      acc[3 * kBlock] = acc[3 * kBlock] + vy;
      acc[4 * kBlock] = acc[4 * kBlock] + vy * vy;
      acc[5 * kBlock] = acc[5 * kBlock] + vw;
      sm.ured[t] += gd ? 1u : 0u;
      if (a.rmax && p.loss == 0) {
        const double tx = p.x - xa, ty = p.y - ya;
        const double r2 = tx * tx + ty * ty;
        const double r2m = acc[6 * kBlock];
        acc[6 * kBlock] = r2m < r2 ? r2 : r2m;
      }
    } else if (a.stats == STAT_APERTURE) {
      const bool ok = p.loss == 0;
      acc[0] = acc[0] + (ok ? p.x : 0.0);
      acc[kBlock] = acc[kBlock] + (ok ? p.y : 0.0);
      sm.ured[t] += ok ? 0u : 1u;
    }
  }
  const Partials& pr = a.pr;
  if (a.stats == STAT_SC) {
    double v[kScQ];
#pragma unroll
    for (int q = 0; q < kScQ; ++q) v[q] = acc[q * kBlock];
    const double r2m = acc[6 * kBlock];
    uint32_t cnt = sm.ured[t];
    double mx = sm.mred[t];
    block_reduce<kScQ>(v, cnt, mx, sm.red, sm.ured, sm.mred, t);
    if (t == 0) {
#pragma unroll
      for (int q = 0; q < kScQ; ++q) pr.sums[q * pr.mpad + c] = v[q];
      pr.cnt[c] = cnt;
      pr.pmax[c] = mx;
    }
    if (a.rmax) {
      const double m = block_max(r2m, sm.mred, t);
      if (t == 0) pr.rmax2[c] = m;
    }
  } else if (a.stats == STAT_APERTURE) {
    double ap[2] = {acc[0], acc[kBlock]};
    uint32_t cnt = sm.ured[t];
    double m0 = 0.0;
    block_reduce<2>(ap, cnt, m0, sm.red, sm.ured, sm.mred, t);
    if (t == 0) { pr.sums[c] = ap[0]; pr.sums[pr.mpad + c] = ap[1]; pr.cnt[c] = cnt; }
  }
}
#endif

template <int kClass, int kGroup>
__global__ __launch_bounds__(kBlock) void k_segment(SegArgs a)
{
  __shared__ RedSmem sm;
  segment_body<kClass, kGroup, false>(a, blockIdx.x, sm);
}

// The same over the chunks of several simulations: map[block] packs the
// simulation (high bits) and its chunk (low kBatchLocalBits bits).
// A batched launch finds its records at recs + *roff bytes: 0 for an eager
// launch, the replayed lattice period's offset inside a period graph.
template <class T>
__device__ __forceinline__ const T* period_recs(const T* recs, const uint64_t* roff)
{
  return (const T*)((const char*)recs + roff[0]);
}

// Waves per SIMD: the classes without RF gaps need 66 VGPRs with the second
// pass of redo, two more than eight waves leave (seven members on 32 x 128:
// 59.5 us a launch at seven waves, 56.0 at eight).
template <int kClass>
constexpr int kBatchWaves = kBounded && kClass < OPC_GAP ? 8 : 1;

template <int kClass, int kGroup>
__global__ __launch_bounds__(kBlock, kBatchWaves<kClass>) void k_segment_batch(
    const SegArgs* __restrict__ recs, const uint32_t* __restrict__ map,
    const uint64_t* __restrict__ roff)
{
  __shared__ RedSmem sm;
  const uint32_t e = map[blockIdx.x];
  const SegArgs& a = period_recs(recs, roff)[e >> kBatchLocalBits];
#ifdef HPS_FAST_PUSH
  __shared__ LiveSmem ls;
  segment_body_live<kClass>(a, e & kBatchLocalMask, sm, ls);
#else
  segment_body<kClass, kGroup, true>(a, e & kBatchLocalMask, sm);
#endif
}

// The same push for beams too small to fill the GPU with k_segment's 256-thread
// workgroups: one chunk per 1024-thread workgroup, one particle per thread.
// Thread j*256 + l pushes particle i = chunk*1024 + j*256 + l (the particle
// canonical lane l takes as its j-th) and stores its statistics
// contributions in LDS; lane l (< 256) then adds its four in the canonical
// order j = 0..3 from +0.0, and the 256 lane sums go through block_reduce's
// halving tree -- the chunk partials are k_segment's bit for bit.
constexpr uint32_t kWideBlock = kChunk;
// at most this many chunks (k_segment would run at most two wavefronts per
// SIMD; measured faster up to 512 chunks, slower at 1024)
constexpr uint32_t kWideMaxChunks = 512;
// Batches of at least this many chunks run the phase pass one chunk per
// wavefront (MI355X, 262,144 chunks of the 64-beam stress batch: phase pass
// 189 -> 164 ms per step); a lone beam of 1,024 chunks in that form has one
// wave per SIMD and runs slower (7.3 -> 13.5 ms per step), so lone beams
// keep a workgroup per chunk.
constexpr uint32_t kPhaseWaveMinChunks = 8192;
struct WideSmem {
  double q[kScQ][kWideBlock];   // contributions, then lane sums in [q][0, 256)
  double mx[kWideBlock];        // phi of particles not longitudinally flagged, else -inf
  double r2[kWideBlock];        // r^2 about (x_avg, y_avg), loss == 0
  uint32_t cnt[kWideBlock];     // good (STAT_SC) or lost (STAT_APERTURE) flags
};

template <int kClass>
__device__ __forceinline__ void segment_body_wide(const SegArgs& a, uint32_t c, WideSmem& w)
{
  const int t = threadIdx.x;
  const BeamArrays& b = a.b;
  const uint32_t i = c * kChunk + (uint32_t)t;
  Particle p = load_particle(b, i, a.mark);
  const bool alive_in = i < b.n && p.loss == 0;
  if (a.kick && alive_in && p.lloss == 0 && (i & a.kick_mask) != 0) {
    const KickConst k = kick_const<Usual>(a.sc, a.st, a.kick_len);
    kick<Usual>(p, k, a.fld2, b.mass, b.rmass);
  }
  const double xa = a.st->x_avg, ya = a.st->y_avg;
  for (int o = a.op_begin; o < a.op_end; ++o) {
    const OpConst& op = ((const OpConst*)a.ops)[o];
    if (p.loss == 0) apply_op<Usual, kClass>(op, p, i, b.mass, b.rmass, b.charge, xa, ya);
  }
  redo<kClass, false>(i, p);
  const bool in = i < b.n;
  if (alive_in) store_particle(b, i, p);
  if (a.stats == STAT_NONE) return;
  const Partials& pr = a.pr;
  if (a.stats == STAT_SC) {
    const bool gd = in && is_good(p.loss, p.lloss);
    const double vx = gd ? p.x : 0.0, vy = gd ? p.y : 0.0;
    w.q[0][t] = gd ? p.phi : 0.0;
    w.q[1][t] = vx;
    w.q[2][t] = vx * vx;
    w.q[3][t] = vy;
    w.q[4][t] = vy * vy;
    w.q[5][t] = gd ? p.w : 0.0;
    w.cnt[t] = gd ? 1u : 0u;
    w.mx[t] = (in && p.lloss == 0) ? p.phi : -__builtin_huge_val();
    double r2 = 0.0;
    if (a.rmax && in && p.loss == 0) {
      // MaxR2PhiReduceKernel's first pass (beam_kernel.cu:826-843)
      const double tx = p.x - xa, ty = p.y - ya;
      r2 = tx * tx + ty * ty;
    }
    w.r2[t] = r2;
  } else {
    const bool ok = in && p.loss == 0;
    w.q[0][t] = ok ? p.x : 0.0;
    w.q[1][t] = ok ? p.y : 0.0;
    w.cnt[t] = (in && p.loss != 0) ? 1u : 0u;
    w.mx[t] = -__builtin_huge_val();
    w.r2[t] = 0.0;
  }
  __syncthreads();
  const int nq = a.stats == STAT_SC ? kScQ : 2;
  // lane sums in the canonical order over j, kept in [q][0, 256)
  if (t < (int)kBlock) {
    for (int q = 0; q < nq; ++q) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < (int)kPerLane; ++j) acc = acc + w.q[q][j * kBlock + t];
      w.q[q][t] = acc;
    }
    uint32_t n = 0;
    double m = -__builtin_huge_val(), r = 0.0;
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j) {
      n += w.cnt[j * kBlock + t];
      m = ::fmax(m, w.mx[j * kBlock + t]);
      const double u = w.r2[j * kBlock + t];
      r = r < u ? u : r;
    }
    w.cnt[t] = n;
    w.mx[t] = m;
    w.r2[t] = r;
  }
  __syncthreads();
  // block_reduce's levels over the 256 lane sums
  if (t < 128) {
    for (int q = 0; q < nq; ++q) w.q[q][t] = w.q[q][t] + w.q[q][t + 128];
    w.cnt[t] += w.cnt[t + 128];
    w.mx[t] = ::fmax(w.mx[t], w.mx[t + 128]);
    const double u = w.r2[t + 128];
    w.r2[t] = w.r2[t] < u ? u : w.r2[t];
  }
  __syncthreads();
  if (t < 64) {
    double v[kScQ];
    for (int q = 0; q < kScQ; ++q) v[q] = q < nq ? w.q[q][t] + w.q[q][t + 64] : 0.0;
    uint32_t n = w.cnt[t] + w.cnt[t + 64];
    double m = ::fmax(w.mx[t], w.mx[t + 64]);
    double r = w.r2[t];
    {
      const double u = w.r2[t + 64];
      r = r < u ? u : r;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
      for (int q = 0; q < kScQ; ++q) v[q] = v[q] + __shfl_down(v[q], o, 64);
      n += __shfl_down(n, o, 64);
      m = ::fmax(m, __shfl_down(m, o, 64));
      const double u = __shfl_down(r, o, 64);
      r = r < u ? u : r;
    }
    if (t == 0) {
      if (a.stats == STAT_SC) {
#pragma unroll
        for (int q = 0; q < kScQ; ++q) pr.sums[q * pr.mpad + c] = v[q];
        pr.cnt[c] = n;
        pr.pmax[c] = m;
        if (a.rmax) pr.rmax2[c] = r;
      } else {
        pr.sums[c] = v[0];
        pr.sums[pr.mpad + c] = v[1];
        pr.cnt[c] = n;
      }
    }
  }
}

template <int kClass>
__global__ __launch_bounds__(kWideBlock) void k_segment_wide(SegArgs a)
{
  extern __shared__ double wide_lds[];
  segment_body_wide<kClass>(a, blockIdx.x, *reinterpret_cast<WideSmem*>(wide_lds));
}

// Cross-chunk step of the k_segment statistics in one workgroup, launched
// after k_segment so that kernel order, not a device-wide fence per
// workgroup, makes the partials visible: the aperture loss count and
// centroid (UpdateLoss + UpdateAvgXY), or the longitudinal-loss update and
// good moments of the space-charge statistics.
//
// kFinalBlock threads: the first eight waves reduce a quantity each; all
// sixteen rescan chunks.
constexpr uint32_t kFinalBlock = 1024;
constexpr uint32_t kRescan = 256;   // chunks of one rescan round

__device__ __forceinline__ void seg_final_body(const SegArgs& a)
{
  __shared__ double sum[kScQ];
  __shared__ double pm;
  __shared__ uint32_t good;
  __shared__ uint32_t rescan_list[kRescan];
  __shared__ uint32_t rescan_n;
  const int t = threadIdx.x, l = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const BeamArrays& b = a.b;
  const Partials& pr = a.pr;
  hps_beam_stats* st = a.st;
  if (a.stats == STAT_APERTURE) {
    if (wave < 2) {
      const double v = wave_tree_sum(pr.sums + (size_t)wave * pr.mpad, pr.mpad, l);
      if (l == 0) sum[wave] = v;
    } else if (wave == 2) {
      const uint32_t n = wave_count(pr.cnt, pr.nch, l);
      if (l == 0) good = n;
    }
    __syncthreads();
    if (t == 0) {
      const uint32_t nloss = good;
      st->num_loss = nloss;
      const double surv = (double)(uint32_t)(b.n - nloss);
      st->x_avg = sum[0] / surv;
      st->y_avg = sum[1] / surv;
    }
    return;
  }

  // STAT_SC: the longitudinal-loss update of Beam::UpdateLongitudinalLoss
  // (beam.cpp:776-782), then the good moments of beam.cpp:1008-1014.
  const uint32_t num_loss = st->num_loss;
  const auto moments = [&]() {
    if (wave < kScQ) {
      const double v = wave_tree_sum(pr.sums + (size_t)wave * pr.mpad, pr.mpad, l);
      if (l == 0) sum[wave] = v;
    } else if (wave == kScQ) {
      const uint32_t n = wave_count(pr.cnt, pr.nch, l);
      if (l == 0) good = n;
    } else if (wave == kScQ + 1) {
      const double m = wave_max(pr.pmax, pr.nch, -__builtin_huge_val(), l);
      if (l == 0) pm = m;
    }
    __syncthreads();
  };
  moments();
  const double avg1 = good > 0 ? sum[0] / (double)good : -99999;
  const double thr = avg1 + TWOPI + PI;
  // Chunks where a not-yet-flagged particle is beyond the threshold get their
  // lloss flags set and their partials recomputed (rare: once per particle),
  // a chunk per wave.  Beams that spill out of the bucket have tens to
  // hundreds of such chunks at a kick point, hence the sixteen waves.
  if (pm > thr) {
    for (uint32_t it = 0; it < pr.nch / kRescan + 2; ++it) {
      __syncthreads();
      if (t == 0) rescan_n = 0;
      __syncthreads();
      for (uint32_t cc = t; cc < pr.nch; cc += kFinalBlock) {
        if (gld(pr.pmax, cc) > thr) {
          const uint32_t slot = atomicAdd(&rescan_n, 1u);
          if (slot < kRescan) rescan_list[slot] = cc;
        }
      }
      __syncthreads();
      const uint32_t nfound = rescan_n;
      if (nfound == 0) break;
      const uint32_t take = nfound < kRescan ? nfound : kRescan;
      for (uint32_t r = (uint32_t)wave; r < take; r += kFinalBlock / 64)
        chunk_flag_stats_wave(b, rescan_list[r], thr, l, pr);
    }
    __syncthreads();
    moments();
  }
  if (t == 0) {
    const uint32_t g2 = good;
    st->num_good = g2;
    st->phi_avg_good = g2 > 0 ? sum[0] / (double)g2 : -99999;
    const double surv = (double)(uint32_t)(b.n - num_loss);
    const double xavg = sum[1] / surv, x2avg = sum[2] / surv, yavg = sum[3] / surv,
                 y2avg = sum[4] / surv;
    st->x_avg_good = xavg;
    st->x_sig_good = ::sqrt(x2avg - xavg * xavg);
    st->y_avg_good = yavg;
    st->y_sig_good = ::sqrt(y2avg - yavg * yavg);
    st->w_avg_good = g2 > 0 ? sum[5] / (double)g2 : -99999;
  }
}


__global__ __launch_bounds__(kFinalBlock) void k_seg_final(SegArgs a) { seg_final_body(a); }

// one workgroup per simulation of a batch
__global__ __launch_bounds__(kFinalBlock) void k_seg_final_batch(const SegArgs* recs,
                                                            const uint64_t* roff)
{
  const SegArgs a = period_recs(recs, roff)[blockIdx.x];
  seg_final_body(a);
}

// --- k_phase -------------------------------------------------------------------

// Per-chunk sums of the relative phase (UpdateRelativePhi(true) then the
// phi_r moments of Beam::UpdateStatForSpaceCharge, beam.cpp:1003-1016):
//   0 phi_r over loss == 0, 1 phi_r and 2 phi_r^2 over good particles.
__device__ __forceinline__ void phase_body(const PhaseArgs& a, uint32_t c)
{
  __shared__ RedSmem sm;
  const int t = threadIdx.x;
  const BeamArrays& b = a.b;
  const Partials& pr = a.pr;
  const double ref = a.st->phi_avg_good;
  double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < (int)kPerLane; ++j) {
    const uint32_t i = c * kChunk + j * kBlock + t;
    double pr_ = 0.0;
    uint32_t loss = 1, lloss = 0;
    if (i < b.n) {
      loss = b.loss[i];
      lloss = b.lloss[i];
      // the relative phase enters the sums only for loss == 0; a lost
      // particle keeps its last phase, which falls ever further behind the
      // reference, so its exact remainder would take the longest
      if (loss == 0) pr_ = relative_phi(b.phi[i], ref);
    }
    const bool tg = (i < b.n) && loss == 0;
    const bool g = (i < b.n) && is_good(loss, lloss);
    acc[0] = acc[0] + (tg ? pr_ : 0.0);
    const double vg = g ? pr_ : 0.0;
    acc[1] = acc[1] + vg;
    acc[2] = acc[2] + vg * vg;
  }
  uint32_t cnt = 0;
  double mx = 0.0;
  block_reduce<3>(acc, cnt, mx, sm.red, sm.ured, sm.mred, t);
  if (t == 0) {
    pr.sums[c] = acc[0];
    pr.sums[pr.mpad + c] = acc[1];
    pr.sums[2 * pr.mpad + c] = acc[2];
  }
}

__global__ __launch_bounds__(kBlock) void k_phase(PhaseArgs a) { phase_body(a, blockIdx.x); }

// The same for beams of at most kWideMaxChunks chunks, one particle per
// thread (as k_segment_wide): contributions in LDS, lane l (< 256) adds its
// four in the canonical order, then block_reduce's halving tree.
__global__ __launch_bounds__(kWideBlock) void k_phase_wide(PhaseArgs a)
{
  __shared__ double w[3][kWideBlock];
  const int t = threadIdx.x;
  const BeamArrays& b = a.b;
  const Partials& pr = a.pr;
  const uint32_t c = blockIdx.x;
  const double ref = a.st->phi_avg_good;
  const uint32_t i = c * kChunk + (uint32_t)t;
  double pr_ = 0.0;
  uint32_t loss = 1, lloss = 0;
  if (i < b.n) {
    loss = b.loss[i];
    lloss = b.lloss[i];
    if (loss == 0) pr_ = relative_phi(b.phi[i], ref);   // used only for loss == 0
  }
  const bool tg = (i < b.n) && loss == 0;
  const bool g = (i < b.n) && is_good(loss, lloss);
  const double vg = g ? pr_ : 0.0;
  w[0][t] = tg ? pr_ : 0.0;
  w[1][t] = vg;
  w[2][t] = vg * vg;
  __syncthreads();
  if (t < (int)kBlock) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < (int)kPerLane; ++j) acc = acc + w[q][j * kBlock + t];
      w[q][t] = acc;
    }
  }
  __syncthreads();
  if (t < 128) {
#pragma unroll
    for (int q = 0; q < 3; ++q) w[q][t] = w[q][t] + w[q][t + 128];
  }
  __syncthreads();
  if (t < 64) {
    double v[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) v[q] = w[q][t] + w[q][t + 64];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
      for (int q = 0; q < 3; ++q) v[q] = v[q] + __shfl_down(v[q], o, 64);
    }
    if (t == 0) {
      pr.sums[c] = v[0];
      pr.sums[pr.mpad + c] = v[1];
      pr.sums[2 * pr.mpad + c] = v[2];
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_phase_batch(const PhaseArgs* recs, const uint32_t* map,
                                                        const uint64_t* roff)
{
  const uint32_t e = map[blockIdx.x];
  const PhaseArgs a = period_recs(recs, roff)[e >> kBatchLocalBits];
  phase_body(a, e & kBatchLocalMask);
}

// The same sums with one chunk per wavefront (batches of at least
// kPhaseWaveMinChunks chunks): lane l stands for the canonical
// lanes l, l + 64, l + 128 and l + 192 of phase_body, sums each one's four
// particles in its order and folds them as levels 128 and 64 of
// block_reduce's tree, then the same shuffle levels: the same bits, without
// LDS or barriers, and all sixteen particles' loads issued before the first
// relative phase.
__device__ __forceinline__ void phase_wave_body(const PhaseArgs& a, uint32_t c, int l)
{
  const BeamArrays& b = a.b;
  const Partials& pr = a.pr;
  const double ref = a.st->phi_avg_good;
  double ph[4][kPerLane];
  uint32_t lo[4][kPerLane], ll[4][kPerLane];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j) {
      const uint32_t i = c * kChunk + j * kBlock + q * 64 + l;
      const bool in = i < b.n;
      ph[q][j] = in ? gld(b.phi, i) : 0.0;
      lo[q][j] = in ? gld(b.loss, i) : 1u;
      ll[q][j] = in ? gld(b.lloss, i) : 0u;
    }
  double v[4][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < (int)kPerLane; ++j) {
      // used only for loss == 0 (beyond n, loss reads 1)
      const double pr_ = lo[q][j] == 0 ? relative_phi(ph[q][j], ref) : 0.0;
      const bool tg = lo[q][j] == 0;
      const bool g = is_good(lo[q][j], ll[q][j]);
      acc[0] = acc[0] + (tg ? pr_ : 0.0);
      const double vg = g ? pr_ : 0.0;
      acc[1] = acc[1] + vg;
      acc[2] = acc[2] + vg * vg;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) v[q][k] = acc[k];
  }
  double s[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) s[k] = (v[0][k] + v[2][k]) + (v[1][k] + v[3][k]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) s[k] = s[k] + __shfl_down(s[k], o, 64);
  }
  if (l == 0) {
    gst(pr.sums, c, s[0]);
    gst(pr.sums, pr.mpad + c, s[1]);
    gst(pr.sums, 2 * pr.mpad + c, s[2]);
  }
}

__global__ __launch_bounds__(kBlock) void k_phase_wave_batch(const PhaseArgs* recs,
                                                             const uint32_t* map, uint32_t nch,
                                                             const uint64_t* roff)
{
  // the chunk map deals each member's chunks to one XCD's positions (8 j + x
  // for XCD x); workgroup b runs on XCD b mod 8, so its four waves take
  // positions 32 (b / 8) + 8 w + b mod 8, w < 4: every position once, each
  // on its XCD
  static_assert(kBlock == 256, "four waves per workgroup");
  const uint32_t b = blockIdx.x, w = threadIdx.x >> 6;
  const uint32_t k = __builtin_amdgcn_readfirstlane(32u * (b >> 3) + 8u * w + (b & 7u));
  if (k >= nch) return;
  const uint32_t e = map[k];
  const PhaseArgs a = period_recs(recs, roff)[e >> kBatchLocalBits];
  phase_wave_body(a, e & kBatchLocalMask, threadIdx.x & 63);
}

// One workgroup after k_phase: the phi_r moments, then the Scheff::Start
// control logic of space_charge.cpp:84-138 (mesh_size_cutoff_w = 0) on the
// device, and the cleared charge histogram
// when it decides to remesh.  Thread 0 reads every input into registers
// before it writes any output.  What bounds it is one chain of memory round
// trips and divisions: the decision goes to the other waves through LDS alone,
// so they clear the histogram while thread 0 works on, and wait for none of its
// stores (1,048,576 particles on 32 x 128: 6.2 -> 5.6 us).
constexpr uint32_t kPhaseFinalBlock = 512;

__device__ __forceinline__ void phase_final_body(const PhaseArgs& a)
{
  __shared__ double sum[4];   // the three sums, the largest r^2
  __shared__ int remesh;
  __shared__ uint32_t nbins;
  const int t = threadIdx.x;
  uint32_t fld_off = 0;
  const BeamArrays& b = a.b;
  hps_beam_stats* st = a.st;
  ScDev* sc = a.sc;
  // thread 0's inputs, loaded before the reduction so that both round trips
  // overlap
  uint32_t good_cnt = 0, num_loss = 0;
  double x_sig_good = 0.0, y_sig_good = 0.0, ke = 0.0, phi_sig_good = 0.0;
  double x_avg_good = 0.0, y_avg_good = 0.0;
  hps_spch_state ss{};
  if (t == 0) {
    good_cnt = st->num_good;
    num_loss = st->num_loss;
    x_sig_good = st->x_sig_good;
    y_sig_good = st->y_sig_good;
    x_avg_good = st->x_avg_good;
    y_avg_good = st->y_avg_good;
    ke = st->w_avg_good;
    phi_sig_good = st->phi_sig_good;
    ss = sc->st;
    fld_off = sc->fld_off;
  }
  // waves 0..2: the relative-phase sums; wave 3: Beam::UpdateMaxRPhi
  // (beam.cu:829-851), the largest r^2 about the last all-particle centroid
  // over loss == 0, for the adjacent-bunch mesh, from the segment's chunk
  // maxima, or directly for beams of at most two particles (no segment
  // statistics).
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
  if (wave < 3) {
    const double v =
        a.do_sums ? wave_tree_sum(a.pr.sums + (size_t)wave * a.pr.mpad, a.pr.mpad, l) : 0.0;
    if (l == 0) sum[wave] = v;
  } else if (wave == 3) {
    const double v = a.rmax == 1 ? wave_max(a.pr.rmax2, a.pr.nch, 0.0, l) : 0.0;
    if (l == 0) sum[3] = v;
  }
  __syncthreads();
  const double s[3] = {sum[0], sum[1], sum[2]};
  double r2max = sum[3];
  if (a.rmax == 2 && t == 0) {
    const double xa = st->x_avg, ya = st->y_avg;
    for (uint32_t i = 0; i < b.n; ++i) {
      if (b.loss[i] != 0) continue;
      const double tx = b.x[i] - xa, ty = b.y[i] - ya;
      const double r2 = tx * tx + ty * ty;
      r2max = r2max < r2 ? r2 : r2max;
    }
  }
  // thread 0 decides; then the other waves clear the histogram while it works
  // out and stores the rest
  double avg_r = 0.0, gamma = 0.0, beta = 0.0, sigz = 0.0, sigr = 0.0;
  int rm = 0;
  if (t == 0) {
    if (a.do_sums) {
      const double gd = (double)good_cnt;
      const double avg = s[1] / gd, avg2 = s[2] / gd;
      phi_sig_good = ::sqrt(avg2 - avg * avg);
      avg_r = s[0] / (double)(uint32_t)(b.n - num_loss);
    }
    const double sigphi = b.n < 2 ? 0.0 : phi_sig_good;
    const double sigx = b.n < 2 ? 0.0 : x_sig_good;
    const double sigy = b.n < 2 ? 0.0 : y_sig_good;
    gamma = (double)ke / b.mass + 1.0;
    beta = ::sqrt(1.0 - 1.0 / (gamma * gamma));
    const double lmbd = 299.792458 / a.freq;
    sigz = sigphi * 0.5 / 3.14159265 * beta * lmbd;
    sigr = ::sqrt(sigx * sigx + sigy * sigy);
    const double cratior = sigr * sigz;
    const double cratioz = sigz * sigz * gamma * gamma;
    const double cratior_old = ss.sigr_old * ss.sigz_old;
    const double cratioz_old = ss.sigz_old * ss.sigz_old * ss.gm_old * ss.gm_old;
    rm = cratior_old == 0.0 || cratioz_old == 0.0 ||
         __builtin_fabs(cratior - cratior_old) / cratior_old > ss.remesh_val ||
         __builtin_fabs(cratioz - cratioz_old) / cratioz_old > ss.remesh_val;
    remesh = rm;
    nbins = ss.nx * ss.nz;
  }
  lds_barrier();
  if (wave != 0) {
    if (remesh)
      for (uint32_t i = t - 64; i < nbins; i += kPhaseFinalBlock - 64) gst(a.bins, i, (int64_t)0);
    return;
  }
  if (t == 0) {
    if (a.do_sums) {
      st->phi_avg_r = avg_r;
      st->phi_sig_good = phi_sig_good;
    }
    // adjacent bunches below the cutoff energy only (space_charge.cpp:102-105)
    const uint32_t adj = (ss.adj_bunch_w == 0.0 || ke < ss.adj_bunch_w) ? ss.adj_bunch : 0u;
    double ratio_r = 1.0, ratio_z = 1.0, ratio_q = 1.0, ratio_g = 1.0;
    ss.kick_count += 1;
    if (rm) {
      ss.sigr_old = sigr;
      ss.sigz_old = sigz;
      ss.gm_old = gamma;
      ss.good_cnt_old = good_cnt;
      ss.remesh_count += 1;
      // UpdateScheffMeshSizeKernel via UpdateMeshKernelCall: the reference
      // compares the device pointers x_sig_good > y_sig_good (space_charge.cu:131);
      // x_sig_good is allocated first (beam.cu:51,54), so sigma_y is used.
      const double bl = beta * CLIGHT / a.freq;
      if (adj != 0) {
        // with adjacent bunches the mesh spans the largest radius and one
        // RF period (UpdateScheffMeshSizeKernel with r_coef = 1)
        ss.dr = 1.0 * ::sqrt(r2max) / ss.nx;
        ss.dz = bl / ss.nz;
      } else {
        ss.dr = 3.0 * y_sig_good / ss.nx;
        ss.dz = 3.0 * bl * phi_sig_good / (ss.nz * PI);
      }
      // the aspect the grouped field solve of a batch interpolates its
      // shared Green's tables in (gm as the Green's table computes it)
      sc->log_aspect = log_aspect(ss.dr, ss.dz, 1.0 / ::sqrt(1.0 - beta * beta));
      ss.num_on_mesh = 0;
    } else {
      ratio_r = sigr / ss.sigr_old;
      ratio_z = sigz / ss.sigz_old;
      // uint / uint, space_charge.cpp:137-138
      ratio_q = ss.good_cnt_old ? (double)(good_cnt / ss.good_cnt_old) : 0.0;
      ratio_g = gamma / ss.gm_old;
    }
    sc->st = ss;
    sc->freq = a.freq;
    sc->beta = beta;
    sc->frac = a.frac;
    sc->current = a.current;
    sc->ratio_r = ratio_r;
    sc->ratio_z = ratio_z;
    sc->ratio_q = ratio_q;
    sc->ratio_g = ratio_g;
    sc->adj_eff = adj;
    if (rm) sc->valid = 1;
    const bool usual =
        kick_prepare(sc, beta, a.freq, a.current * a.frac, x_avg_good, y_avg_good, x_sig_good,
                 y_sig_good, ss.dr, ss.dz, ss.nz, ratio_r, ratio_z, ratio_q, ratio_g, b.n,
                 b.mass, rm != 0, fld_off);
    sc->remesh = rm ? (usual ? kRemeshQuick : kRemesh) : 0;
  }
}

__global__ __launch_bounds__(kPhaseFinalBlock) void k_phase_final(PhaseArgs a) { phase_final_body(a); }

__global__ __launch_bounds__(kPhaseFinalBlock) void k_phase_final_batch(const PhaseArgs* recs,
                                                              const uint64_t* roff)
{
  const PhaseArgs a = period_recs(recs, roff)[blockIdx.x];
  phase_final_body(a);
}

// --- SCHEFF rebuild ----------------------------------------------------------------

// One entry of the ring Green's table, UpdateFldTbl1Kernel
// (space_charge_kernel.cu:38-100), stored [rp][dz][rs] so that the field sum
// reads consecutive rs.
template <class A>
__device__ __forceinline__ void greens_entry(const ScDev* sc, double* fld1, uint32_t nr,
                                             uint32_t nz, uint32_t r_num_part, double mass,
                                             uint32_t idx)
{
  uint32_t k, t, rpi;   // source ring rs, dz, field radius rp
  if (((nr & (nr - 1)) | (nz & (nz - 1))) == 0) {
    const uint32_t lr = 31u - __builtin_clz(nr), lz = 31u - __builtin_clz(nz);
    k = idx & (nr - 1);
    t = (idx >> lr) & (nz - 1);
    rpi = idx >> (lr + lz);
  } else {
    const uint32_t row = idx / nr;
    k = idx - row * nr;
    rpi = row / nz;
    t = row - rpi * nz;
  }
  const double r_beta = sc->beta, r_freq = sc->freq;
  const double r_current_ov_mc2 = sc->current * sc->frac / mass;
  const double gm = 1.0 / ::sqrt(1.0 - r_beta * r_beta);
  const double dr = sc->st.dr;
  const double dzg = sc->st.dz * gm;
  const double rs = ::sqrt(0.5 * (k * k + (k + 1) * (k + 1))) * dr;
  const double zs = 0.5 * dzg;
  const double zp = (t + 1) * dzg;
  const double rp = rpi * dr;
  const double d = zp - zs;
  double er1, ez1;
  ring_green<A>(rs, rp, d, er1, ez1);
  // image rings of the neighbouring bunches, one RF period apart in the
  // bunch frame (space_charge_kernel.cu:74-94)
  const uint32_t adj = sc->adj_eff;
  if (adj != 0) {
    const double wave_len = CLIGHT / r_freq;
    const double pl = r_beta * gm * wave_len;
    for (uint32_t i = 1; i <= adj; ++i) {
      double xi = (double)i;
      for (int j = 0; j < 2; ++j) {
        double er, ez;
        ring_green<A>(rs, rp, d - xi * pl, er, ez);
        if (rp != 0.0) er1 += er;
        ez1 += ez;
        xi = -xi;
      }
    }
  }
  const double c1 = 5721.67 * r_current_ov_mc2 / (r_freq * 1e6 * (double)r_num_part);
  fld1[2 * (size_t)idx] = c1 * er1;
  fld1[2 * (size_t)idx + 1] = c1 * ez1;
}

// Charge deposit, DistributeParticleKernel (space_charge_kernel.cu:122-224),
// of workgroup `blk` of `nblk` into an LDS-private int64 fixed-point
// histogram, merged into bins with 64-bit integer atomics: integer sums make
// the result independent of the order.
// Constants of one rebuild's deposit (DistributeParticleKernel's
// prologue, space_charge_kernel.cu:122-150).
struct DepConst {
  uint32_t nx, nz;
  double phimc, xbar, ybar, epsq, ref, dr, dzg, hl, c2, drdr;
  double repsq, rdr, rdzg, rdrdr;   // reciprocals for div_by
};

__device__ __forceinline__ DepConst dep_const(const hps_beam_stats* st, const ScDev* sc)
{
  DepConst d;
  d.nx = sc->st.nx;
  d.nz = sc->st.nz;
  const double r_beta = sc->beta, r_freq = sc->freq;
  d.phimc = st->phi_avg_r;
  d.xbar = st->x_avg_good;
  d.ybar = st->y_avg_good;
  d.epsq = st->x_sig_good / st->y_sig_good;
  d.ref = st->phi_avg_good;
  const double gm = 1.0 / ::sqrt(1.0 - r_beta * r_beta);
  d.dr = sc->st.dr;
  d.dzg = sc->st.dz * gm;
  const double wave_len = CLIGHT / r_freq;
  d.hl = d.nz * 0.5 * d.dzg;
  d.c2 = r_beta * gm * wave_len / TWOPI;
  d.drdr = d.dr * d.dr;
  if constexpr (kBounded) {
    d.repsq = recip(d.epsq);
    d.rdr = recip(d.dr);
    d.rdzg = recip(d.dzg);
    d.rdrdr = recip(d.drdr);
  }
  return d;
}

// The squared radius of a particle scaled to the round beam.
template <class A>
__device__ __forceinline__ double deposit_r2(double x, double y, const DepConst& d)
{
  return A::div_by((x - d.xbar) * (x - d.xbar), d.epsq, d.repsq) +
         (y - d.ybar) * (y - d.ybar) * d.epsq;
}

// One good particle's charge into the LDS histogram: the area weights in r,
// the linear weights in z, as 2^-36 fixed point (DistributeParticleKernel's
// body, space_charge_kernel.cu:151-218); returns whether it landed on the
// mesh.  rsq_sh: the squared radius (deposit_r2).
template <class A>
__device__ __forceinline__ bool deposit_one(double rsq_sh, double phi, const DepConst& d,
                                            unsigned long long* hist)
{
  const uint32_t nx = d.nx, nz = d.nz;
  const double dr = d.dr, dzg = d.dzg, drdr = d.drdr, hl = d.hl;
  double z = relative_phi(phi, d.ref);
  const int i = to_int(A::div_by(A::sqrt(rsq_sh), dr, d.rdr) + 1);
  if (i < 1 || i > (int)nx) return false;
  double ddz = z - d.phimc;
  for (int guard = 0; (ddz > PI || ddz < -PI) && guard < 4096; ++guard) {
    if (ddz > 0.0) ddz -= TWOPI;
    else ddz += TWOPI;
  }
  z = -d.c2 * ddz;
  if (!(__builtin_fabs(z) < hl)) return false;
  const double zz = z + hl;
  const int jm1 = to_int(A::div_by(zz, dzg, d.rdzg) + 1);
  int i1 = i + 1;
  if (rsq_sh < 0.5 * drdr * (double)(i * i + (i - 1) * (i - 1))) i1 = i - 1;
  if (i1 < 1) i1 = 1;
  if (i1 > (int)nx) i1 = (int)nx;
  int j1 = jm1 + 1;
  if (zz < (jm1 - 1 + 0.5) * dzg) j1 = jm1 - 1;
  if (j1 < 1) j1 = 1;
  if (j1 > (int)nz) j1 = (int)nz;
  double a;
  if (i1 == i) {
    a = 1.0;
  } else {
    const double sqrtmp = A::sqrt(A::div_by(4.0 * rsq_sh, drdr, d.rdrdr) - 1.0);
    const double rminsq = 0.25 * drdr * (sqrtmp - 1.0) * (sqrtmp - 1.0);
    const double rmaxsq = rminsq + sqrtmp * drdr;
    if (i1 < i) a = A::div(rmaxsq - (i - 1) * (i - 1) * drdr, rmaxsq - rminsq);
    else a = A::div((i1 - 1) * (i1 - 1) * drdr - rminsq, rmaxsq - rminsq);
  }
  double cc = 1.0;
  if (j1 != jm1) cc = A::div(zz - (j1 - 1 + 0.5) * dzg, (jm1 - j1) * dzg);
  const double bb = 1.0 - a;
  const double dd = 1.0 - cc;
  if (jm1 < 1 || jm1 > (int)nz) return false;
  int k = (jm1 - 1) * (int)nx + i;
  atomicAdd(&hist[k - 1], (unsigned long long)(int64_t)(a * cc * 0x1p36));
  k += i1 - i;
  atomicAdd(&hist[k - 1], (unsigned long long)(int64_t)(bb * cc * 0x1p36));
  k = (j1 - 1) * (int)nx + i;
  atomicAdd(&hist[k - 1], (unsigned long long)(int64_t)(a * dd * 0x1p36));
  k += i1 - i;
  atomicAdd(&hist[k - 1], (unsigned long long)(int64_t)(bb * dd * 0x1p36));
  return true;
}

// The deposit of a workgroup's share of the particles (strided by the
// deposit grid) into its LDS histogram, flushed into the global one with
// 64-bit integer atomics.  Each thread loads its next particle (flags and
// coordinates, unconditionally) before depositing the current one; the
// histogram is the same (integer sums), only the load order differs (the
// 1,048,576-particle beam: 14.7 -> 14.2 ms per 800-element step; 64 beams
// of 4,194,304 particles on 64 x 256: 226 -> 185 ms per 160-element step).
__device__ __forceinline__ void deposit_block(const BeamArrays& b, const hps_beam_stats* st,
                                              ScDev* sc, int64_t* bins, uint32_t blk,
                                              uint32_t nblk, bool usual,
                                              unsigned long long* hist, uint32_t* ured)
{
  const int t = threadIdx.x;
  const DepConst d = dep_const(st, sc);
  const uint32_t nb = d.nx * d.nz;
  for (uint32_t i = t; i < nb; i += kDepositBlock) hist[i] = 0ull;
  if (t == 0) ured[0] = 0;
  __syncthreads();
  uint32_t count = 0;
  bool again = false;
  const uint32_t stride = nblk * kDepositBlock;
  uint32_t np = blk * kDepositBlock + t;
  bool have = np < b.n;
  uint32_t lo = 1, ll = 0;
  double x = 0.0, y = 0.0, ph = 0.0;
  if (have) {
    lo = gld(b.loss, np); ll = gld(b.lloss, np);
    x = gld(b.x, np); y = gld(b.y, np); ph = gld(b.phi, np);
  }
  while (have) {
    const uint32_t clo = lo, cll = ll;
    const double cx = x, cy = y, cph = ph;
    np += stride;
    have = np < b.n;
    if (have) {
      lo = gld(b.loss, np); ll = gld(b.lloss, np);
      x = gld(b.x, np); y = gld(b.y, np); ph = gld(b.phi, np);
    }
    if (clo == 0 && cll == 0) {
      const double r2 = deposit_r2<Usual>(cx, cy, d);
      if (!usual || Usual::off(Usual::mark(r2))) again = true;
      else if (deposit_one<Usual>(r2, cph, d, hist)) ++count;
    }
  }
  if constexpr (kBounded) {
    // the particles that Quick does not cover, in a sweep of their own
    if (__builtin_expect(again, 0)) {
      for (uint32_t i = blk * kDepositBlock + t; i < b.n; i += stride) {
        if (gld(b.loss, i) != 0 || gld(b.lloss, i) != 0) continue;
        const double px = gld(b.x, i), py = gld(b.y, i);
        if (usual && in_range(deposit_r2<Quick>(px, py, d))) continue;
        if (deposit_one<Any>(deposit_r2<Any>(px, py, d), gld(b.phi, i), d, hist)) ++count;
      }
    }
  }
  __syncthreads();
  for (uint32_t i = t; i < nb; i += kDepositBlock) {
    const unsigned long long v = hist[i];
    if (v != 0ull) atomicAdd((unsigned long long*)&bins[i], v);
  }
  // on-mesh count: wave sums, one LDS add a wave
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) count += __shfl_down(count, o, 64);
  if ((t & 63) == 0 && count) atomicAdd(ured, count);
  __syncthreads();
  if (t == 0 && ured[0]) atomicAdd(&sc->st.num_on_mesh, ured[0]);
}

// The SCHEFF rebuild after a remesh decision, one launch of
// sc_build_blocks(a) workgroups per simulation: greens_wgs of them fill the
// Green's table, in turns of a workgroup's threads, dep_blocks deposit; side by
// side (the first greens_wgs, then the others) or, combined, the first
// greens_wgs before they deposit (build_plan).  Both roles read only the
// control step's results; all exit when there is no remesh.

__device__ __forceinline__ void sc_build_body(const BuildArgs& a, uint32_t nr, uint32_t nz,
                                              uint32_t blk, unsigned long long* hist,
                                              uint32_t* ured)
{
  const int remesh = a.sc->remesh;
  if (!remesh) return;
  const bool usual = !kBounded || __builtin_expect(remesh == kRemeshQuick, 1);
  const bool table = blk < a.greens_wgs;
  const uint32_t total = (nr + 1) * nz * nr;
  const uint32_t first = blk * kDepositBlock + threadIdx.x, step = a.greens_wgs * kDepositBlock;
  if (table && usual)
    for (uint32_t i = first; i < total; i += step)
      greens_entry<Usual>(a.sc, a.fld1, nr, nz, a.b.n, a.b.mass, i);
  if (!(table && a.side))
    deposit_block(a.b, a.st, a.sc, a.bins, a.side ? blk - a.greens_wgs : blk, a.dep_blocks, usual,
                  hist, ured);
  // a mesh that Quick does not cover; here, where its loop keeps no register
  // of the usual one's
  if constexpr (kBounded) {
    if (table && !usual) {
      const ScDev* sc = a.sc;
#ifdef __HIP_DEVICE_COMPILE__
      asm volatile("" : "+s"(sc));
#endif
      for (uint32_t i = first; i < total; i += step)
        greens_entry<Any>(sc, a.fld1, nr, nz, a.b.n, a.b.mass, i);
    }
  }
}

__global__ __launch_bounds__(kDepositBlock) void k_sc_build(BuildArgs a, uint32_t nr, uint32_t nz)
{
  extern __shared__ unsigned long long hist[];
  __shared__ uint32_t ured[1];
  sc_build_body(a, nr, nz, blockIdx.x, hist, ured);
}

__global__ __launch_bounds__(kDepositBlock) void k_sc_build_batch(const BuildArgs* recs,
                                                                  const uint32_t* map,
                                                                  uint32_t nr, uint32_t nz)
{
  extern __shared__ unsigned long long hist[];
  __shared__ uint32_t ured[1];
  const uint32_t e = map[blockIdx.x];
  const BuildArgs a = recs[e >> kBatchLocalBits];
  sc_build_body(a, nr, nz, e & kBatchLocalMask, hist, ured);
}

// Field table E(zp, rp) = sum over bins of charge * Green's value,
// UpdateFldTbl2Kernel (space_charge_kernel.cu:230-342), in the canonical
// order: P = min(NextPow2(nr), 64) partial sums, partial p takes the source
// rings rs = p, p + P, ... in ascending order and for each the rows
// zs = 0 .. nz-1 in ascending order (fma), then a halving tree over the P
// partials.  Field point (zp, rp) reads the Green's entry at dz = zs - zp
// (zs >= zp, E_z sign -1) or zp - zs - 1 (zs < zp).
//
// A wave computes K consecutive rows zp0 .. zp0 + K - 1 of 64 / P radii rp
// (wave's lanes = P partials x 64 / P radii).  Along zs the K rows need the
// Green's entries of K consecutive offsets d = zs - zp, so a K-deep window of
// (E_r, signed E_z) values stays in registers and each step takes one new
// entry and one charge for 2 K products.  The window slot of offset d is d
// mod K (zp0 is a multiple of K), so with the zs loop unrolled by K every
// slot index is a compile-time constant.
//
// All lanes of the wave share zp0, hence d: the row an entry is read from and
// the sign of its E_z are scalar, and the vector unit does little but the 2 K
// products.  Lanes of one wave on different rows of one radius cost as many
// vector instructions for index and sign as for the products, and every
// workgroup staged the whole table slice of its radius in LDS first (32 x 128:
// 96 KB per workgroup of four waves, two memory round trips before the first
// product; 64 x 256: sixteen-byte pieces of every line, eight splits and a
// combine launch).  The entries now come straight from L2, coalesced, kDepth
// row blocks ahead of their use; only the charges, shared by all waves, are
// staged.  Workgroups are dealt so that those of neighbouring radii share an
// XCD's L2.  Against the staged form: 300,007 particles on 64 x 256 148 ->
// 109 us a kick point, seven FP64 members on 32 x 128 field 46 -> 24 us.
struct FieldGeom {
  uint32_t P;        // partials
  uint32_t blocks;   // row blocks of K rows
  uint32_t units;    // waves with work: groups of 64 / P radii x row blocks
  uint32_t per_xcd;  // workgroups dealt to an XCD
};

template <int K, int kDepth>
__device__ __forceinline__ void field_wave_body(const FieldArgs& f, uint32_t nr, uint32_t nz,
                                                const FieldGeom& fg, uint32_t blk, double* lq)
{
  if (!f.sc->remesh) return;
  // charges, kStage in flight per thread
  constexpr uint32_t kStage = 8;
  const uint32_t fld_sz = nr * nz;
  for (uint32_t i0 = threadIdx.x; i0 < fld_sz; i0 += kStage * blockDim.x) {
    int64_t qv[kStage];
#pragma unroll
    for (uint32_t u = 0; u < kStage; ++u) qv[u] = gld(f.bins, ::min(i0 + u * blockDim.x, fld_sz - 1));
#pragma unroll
    for (uint32_t u = 0; u < kStage; ++u)
      lq[::min(i0 + u * blockDim.x, fld_sz - 1)] = (double)qv[u] * 0x1p-36;
  }
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wg = (blk & 7u) * fg.per_xcd + (blk >> 3);
  const uint32_t unit = wg * (blockDim.x >> 6) + wave;
  const uint32_t P = fg.P, lane = threadIdx.x & 63u;
  const uint32_t j = lane & (P - 1);
  const uint32_t rp0 = unit / fg.blocks * (64 / P);   // the wave's radii rp0 ...
  const uint32_t rp = rp0 + lane / P;
  const int zp0 = (int)(unit % fg.blocks) * K;
  const int inz = (int)nz;
  __syncthreads();
  if (unit >= fg.units) return;
  // the wave's part of the table as a buffer: entries at a lane offset (radius
  // and ring) plus a scalar row offset
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const uint32_t nrad = ::min(nr + 1 - rp0, 64 / P);
  const __amdgpu_buffer_rsrc_t tab = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(f.fld1) + 2 * (size_t)rp0 * fld_sz, 0, (int)(16 * nrad * fld_sz), 0x00020000);
  const uint32_t lane0 = 16 * ((rp <= nr ? rp : nr) - rp0) * fld_sz;
  const int rb = 16 * (int)nr, last = (inz - 1) * rb;   // bytes of a row, offset of the last
  double tx[K], ty[K];
#pragma unroll
  for (int k = 0; k < K; ++k) { tx[k] = 0.0; ty[k] = 0.0; }
  for (uint32_t rs = j; rs < nr; rs += P) {
    const int at = (int)(lane0 + 16 * rs);
    const auto entry = [&](int so) -> double2 {
      const u4 v = __builtin_amdgcn_raw_buffer_load_b128(tab, at, ::min(so, last), 0);
      return make_double2(double_of((uint64_t)v.y << 32 | v.x), double_of((uint64_t)v.w << 32 | v.z));
    };
    // the entries (E_z unsigned) of source rows zs0 .. zs0 + K - 1 against row
    // zp0: both multiples of K, so all behind or all ahead; rows past the
    // table repeat its last and are not used
    const auto load = [&](double2 (&e)[K], int zs0) {
      const bool ahead = zs0 >= zp0;
      int so = (ahead ? zs0 - zp0 : zp0 - 1 - zs0) * rb;
#pragma unroll
      for (int u = 0; u < K; ++u) {
        e[u] = entry(so);
        so += ahead ? rb : -rb;
      }
    };
    // Ring of kDepth + 1 row blocks: block b sits in ring[b % R], its
    // predecessor (the older half of the window) in the slot before, and when
    // b is done that slot takes block b + kDepth.
    constexpr int R = kDepth + 1;
    double2 ring[R][K];
    ring[R - 1][0] = make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 1; k < K; ++k) {   // offsets -zp0 - k: entry zp0 + k - 1, none past the table
      ring[R - 1][K - k] = entry((zp0 + k - 1) * rb);
      if (zp0 + k > inz) ring[R - 1][K - k] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int h = 0; h < kDepth; ++h) load(ring[h], h * K);
    // the products of block b = zs0 / K in ring[h], n of its K rows
    double c[R][K];
    const auto block = [&](int zs0, int h, int n) {
      const uint64_t flip = zs0 >= zp0 ? 0x8000000000000000ull : 0ull;   // sources ahead
      const int hp = (h + R - 1) % R;
#pragma unroll
      for (int u = 0; u < K; ++u) {
        if (u >= n) continue;
        ring[h][u].y = double_of(bits_of(ring[h][u].y) ^ flip);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const double2 v = k <= u ? ring[h][u - k] : ring[hp][K + u - k];
          tx[k] = ::fma(c[h][u], v.x, tx[k]);
          ty[k] = ::fma(c[h][u], v.y, ty[k]);
        }
      }
    };
    // charges of a whole block, read from LDS one block ahead (past the last
    // whole block it is read again, unused)
    const auto charges = [&](int zs0, int h) {
      const double* q = lq + (uint32_t)::min(zs0, inz - K) * nr + rs;
#pragma unroll
      for (int u = 0; u < K; ++u) c[h][u] = q[(uint32_t)u * nr];
    };
    int zs0 = 0;
    if (R * K <= inz) {
      charges(0, 0);
      for (; zs0 + R * K <= inz; zs0 += R * K) {
#pragma unroll
        for (int h = 0; h < R; ++h) {
          charges(zs0 + (h + 1) * K, (h + 1) % R);
          block(zs0 + h * K, h, K);
          load(ring[(h + R - 1) % R], zs0 + (h + kDepth) * K);
        }
      }
    }
#pragma unroll
    for (int h = 0; h < R; ++h) {
      const int z = zs0 + h * K, n = ::min(K, inz - z);
      if (n <= 0) break;
#pragma unroll
      for (int u = 0; u < K; ++u)
        if (u < n) c[h][u] = lq[(uint32_t)(z + u) * nr + rs];
      block(z, h, n);
      if (h == 0) load(ring[R - 1], zs0 + kDepth * K);
    }
  }
  // halving tree over the partials
  for (uint32_t o = P / 2; o >= 1; o >>= 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const double ox = __shfl_down(tx[k], o, (int)P);
      const double oy = __shfl_down(ty[k], o, (int)P);
      tx[k] = tx[k] + ox;
      ty[k] = ty[k] + oy;
    }
  }
  if (j == 0 && rp <= nr) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int zp = zp0 + k;
      if (zp <= inz) {
        const size_t o = (size_t)zp * (nr + 1) + rp;
        gst(f.fld2, 2 * o, tx[k]);
        gst(f.fld2, 2 * o + 1, ty[k]);
      }
    }
  }
}

constexpr uint32_t kFieldMaxWaves = 9;

template <int K, int kDepth>
__global__ __launch_bounds__(64 * kFieldMaxWaves) void k_field_wave(FieldArgs f, uint32_t nr,
                                                                    uint32_t nz, FieldGeom fg)
{
  extern __shared__ double lds[];
  field_wave_body<K, kDepth>(f, nr, nz, fg, blockIdx.x, lds);
}

// per simulation of a batch: blocks [m * per, (m + 1) * per)
template <int K, int kDepth>
__global__ __launch_bounds__(64 * kFieldMaxWaves) void k_field_wave_batch(
    const FieldArgs* recs, uint32_t per, uint32_t nr, uint32_t nz, FieldGeom fg)
{
  extern __shared__ double lds[];
  const FieldArgs f = recs[blockIdx.x / per];
  field_wave_body<K, kDepth>(f, nr, nz, fg, blockIdx.x % per, lds);
}

// --- getter reductions ---------------------------------------------------------

// With rel_ref given, the first variable is the relative phase of pa
// against rel_ref[0] (what k_relative_phi stores), computed in registers.
__global__ __launch_bounds__(kBlock) void k_sums(BeamArrays b, const double* pa, const double* pb,
                                                 int filter, Partials pr, const double* rel_ref)
{
  __shared__ RedSmem sm;
  const int t = threadIdx.x;
  const uint32_t c = blockIdx.x;
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  uint32_t nloss = 0, ngood = 0, nlloss = 0;
#pragma unroll
  for (int j = 0; j < (int)kPerLane; ++j) {
    const uint32_t i = c * kChunk + j * kBlock + t;
    if (i >= b.n) continue;
    const uint32_t loss = b.loss[i], lloss = b.lloss[i];
    nloss += loss != 0;
    nlloss += lloss != 0;
    ngood += is_good(loss, lloss);
    const bool inc = filter == 0 ? loss == 0 : (filter == 1 ? is_good(loss, lloss) : true);
    double va = (inc && pa) ? pa[i] : 0.0;
    if (inc && pa && rel_ref) va = relative_phi(va, rel_ref[0]);
    const double vb = (inc && pb) ? pb[i] : 0.0;
    acc[0] = acc[0] + va;
    acc[1] = acc[1] + va * va;
    acc[2] = acc[2] + vb;
    acc[3] = acc[3] + vb * vb;
    acc[4] = acc[4] + va * vb;
  }
  // counts are packed 3 x 11 bits (at most 1024 per chunk each)
  uint32_t packed = nloss | (ngood << 11) | (nlloss << 22);
  double mx = 0.0;
  block_reduce<5>(acc, packed, mx, sm.red, sm.ured, sm.mred, t);
  if (t == 0) {
#pragma unroll
    for (int q = 0; q < 5; ++q) pr.sums[q * pr.mpad + c] = acc[q];
    pr.cnt[c] = packed & 0x7ffu;
    pr.cnt[pr.mpad + c] = (packed >> 11) & 0x7ffu;
    pr.cnt[2 * pr.mpad + c] = packed >> 22;
  }
}

// Cross-chunk trees of k_sums in one workgroup.
__global__ __launch_bounds__(576) void k_sums_final(Partials pr, BeamSums* out, Readout* ro,
                                                    const hps_beam_stats* st, const double* w)
{
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  if (wave < 5) {
    const double v = wave_tree_sum(pr.sums + (size_t)wave * pr.mpad, pr.mpad, l);
    if (l == 0) out->s[wave] = v;
  } else if (wave < 8) {
    const int k = wave - 5;
    const uint32_t n = wave_count(pr.cnt + (size_t)k * pr.mpad, pr.nch, l);
    if (l == 0) (&out->nloss)[k] = n;
  } else if (ro) {
    constexpr int kWords = sizeof(hps_beam_stats) / 4;
    for (int i = l; i < kWords; i += 64) ((uint32_t*)&ro->st)[i] = ((const uint32_t*)st)[i];
    if (l == 0) ro->w0 = w[0];
  }
}

__global__ void k_set_stats(hps_beam_stats* st, hps_beam_stats s)
{
  if (threadIdx.x == 0) *st = s;
}

// A particle per thread, 56 bytes in flight each way.
__global__ __launch_bounds__(kBlock) void k_copy_beam(BeamArrays src, BeamArrays dst)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= src.n) return;
  gst(dst.x, i, gld(src.x, i)); gst(dst.xp, i, gld(src.xp, i));
  gst(dst.y, i, gld(src.y, i)); gst(dst.yp, i, gld(src.yp, i));
  gst(dst.phi, i, gld(src.phi, i)); gst(dst.w, i, gld(src.w, i));
  gst(dst.loss, i, gld(src.loss, i)); gst(dst.lloss, i, gld(src.lloss, i));
}

__global__ void k_relative_phi(BeamArrays b, const double* ref)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < b.n) b.phi_r[i] = relative_phi(b.phi[i], ref[0]);
}

// UpdateLongitudinalLossCoordinateKernel, beam_kernel.cu:1549-1559
__global__ void k_lloss_flag(BeamArrays b, const double* avg)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < b.n && b.phi[i] > avg[0] + TWOPI + PI) b.lloss[i] = 1;
}

// ShiftVariableKernel, beam_kernel.cu:1489-1496 (particle 0 untouched)
__global__ void k_shift(double* a, uint32_t n, double v)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i > 0 && i < n) a[i] += v;
}

// ChangeFrequencyKernel, beam_kernel.cu:1531-1537
__global__ void k_scale(double* a, uint32_t n, double v)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) a[i] *= v;
}

// CutBeamKernel, beam_kernel.cu:1464-1480
__global__ void k_cut(const double* a, uint32_t* loss, uint32_t n, double lo, double hi)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i > 0 && i < n && loss[i] == 0) {
    const double x = a[i];
    if (x < hi && x > lo) loss[i] = 99999;
  }
}

__global__ void k_probe(int fn, const double* x, const double* y, double* out, uint32_t n)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double v = x[i];
  double r = 0.0, s, c;
  switch (fn) {
    case 0: r = hps::exp(v); break;
    case 1: r = hps::log(v); break;
    case 2: hps::sincos(v, &s, &c); r = s; break;
    case 3: hps::sincos(v, &s, &c); r = c; break;
    case 4: r = hps::sinh(v); break;
    case 5: r = hps::cosh(v); break;
    case 6: r = ::sqrt(v); break;
    case 7: r = hps::fmod_pos(v, TWOPI); break;
    case 8: r = v / y[i]; break;
    case 9: r = bessi0c(v); break;
    case 10: r = bessi1c(v); break;
    case 11: r = bessi1p(v); break;
    case 12: r = psqrt(v); break;
    case 13: psincos(v, &s, &c); r = s; break;
    case 14: psincos(v, &s, &c); r = c; break;
    case 15: psinhcosh(v, &s, &c); r = s; break;
    case 16: psinhcosh(v, &s, &c); r = c; break;
    case 17: r = pdiv(v, y[i]); break;
    case 18: r = div_by(v, y[i], 1.0 / y[i]); break;
    case 19: r = sqrt_unscaled(v); break;
    default: break;
  }
  out[i] = r;
}

inline uint32_t blocks_for(uint32_t n) { return (n + kBlock - 1) / kBlock; }

}  // namespace

hipError_t launch_segment(const SegArgs& a, hipStream_t s)
{
  const uint32_t nch = (a.b.n + kChunk - 1) / kChunk;
  if (nch <= kWideMaxChunks) {
    const size_t lds = sizeof(WideSmem);
    if (a.op_class >= OPC_GAP)
      hipLaunchKernelGGL((k_segment_wide<OPC_GAP>), dim3(nch), dim3(kWideBlock), lds, s, a);
    else if (a.op_class == OPC_QUAD)
      hipLaunchKernelGGL((k_segment_wide<OPC_QUAD>), dim3(nch), dim3(kWideBlock), lds, s, a);
    else
      hipLaunchKernelGGL((k_segment_wide<OPC_LIGHT>), dim3(nch), dim3(kWideBlock), lds, s, a);
    return hipGetLastError();
  }
  if (a.op_class >= OPC_GAP)
    hipLaunchKernelGGL((k_segment<OPC_GAP, kSegGroupGap>), dim3(nch), dim3(kBlock), 0, s, a);
  else if (a.op_class == OPC_QUAD)
    hipLaunchKernelGGL((k_segment<OPC_QUAD, kSegGroupQuad>), dim3(nch), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL((k_segment<OPC_LIGHT, kSegGroupLight>), dim3(nch), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_segment_batch(const SegArgs* recs, const uint32_t* map, uint32_t nblocks,
                                int op_class, const uint64_t* roff, hipStream_t s)
{
  if (op_class >= OPC_GAP)
    hipLaunchKernelGGL((k_segment_batch<OPC_GAP, kSegGroupGap>), dim3(nblocks), dim3(kBlock), 0,
                       s, recs, map, roff);
  else if (op_class == OPC_QUAD)
    hipLaunchKernelGGL((k_segment_batch<OPC_QUAD, kSegGroupQuad>), dim3(nblocks), dim3(kBlock),
                       0, s, recs, map, roff);
  else
    hipLaunchKernelGGL((k_segment_batch<OPC_LIGHT, kSegGroupLight>), dim3(nblocks),
                       dim3(kBlock), 0, s, recs, map, roff);
  return hipGetLastError();
}

hipError_t launch_seg_final(const SegArgs& a, hipStream_t s)
{
  hipLaunchKernelGGL(k_seg_final, dim3(1), dim3(kFinalBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_seg_final_batch(const SegArgs* recs, uint32_t nmem, const uint64_t* roff,
                                  hipStream_t s)
{
  hipLaunchKernelGGL(k_seg_final_batch, dim3(nmem), dim3(kFinalBlock), 0, s, recs, roff);
  return hipGetLastError();
}

hipError_t launch_phase(const PhaseArgs& a, hipStream_t s)
{
  const uint32_t nch = (a.b.n + kChunk - 1) / kChunk;
  if (nch <= kWideMaxChunks)
    hipLaunchKernelGGL(k_phase_wide, dim3(nch), dim3(kWideBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_phase, dim3(nch), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_phase_final(const PhaseArgs& a, hipStream_t s)
{
  hipLaunchKernelGGL(k_phase_final, dim3(1), dim3(kPhaseFinalBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_phase_batch(const PhaseArgs* recs, const uint32_t* map, uint32_t nblocks,
                              const uint64_t* roff, hipStream_t s)
{
  // nblocks: one per chunk of the batch.  Batches of at least
  // kPhaseWaveMinChunks chunks run a wavefront per chunk (four chunks per
  // workgroup); smaller ones a workgroup per chunk, which keeps more waves in
  // flight when there are few chunks.
  if (nblocks >= kPhaseWaveMinChunks)
    hipLaunchKernelGGL(k_phase_wave_batch, dim3((nblocks + 31) / 32 * 8), dim3(kBlock), 0, s,
                       recs, map, nblocks, roff);
  else
    hipLaunchKernelGGL(k_phase_batch, dim3(nblocks), dim3(kBlock), 0, s, recs, map, roff);
  return hipGetLastError();
}

hipError_t launch_phase_final_batch(const PhaseArgs* recs, uint32_t nmem, const uint64_t* roff,
                                    hipStream_t s)
{
  hipLaunchKernelGGL(k_phase_final_batch, dim3(nmem), dim3(kPhaseFinalBlock), 0, s, recs, roff);
  return hipGetLastError();
}

// roff[0] = v (set) or roff[0] += v (advance): the record offset of the
// next replay of a period graph, as a kernel node (no memset node).
__global__ void k_roff(uint64_t* roff, uint64_t v, int add)
{
  if (threadIdx.x == 0) roff[0] = add ? roff[0] + v : v;
}

hipError_t launch_roff(uint64_t* roff, uint64_t v, bool add, hipStream_t s)
{
  hipLaunchKernelGGL(k_roff, dim3(1), dim3(64), 0, s, roff, v, add ? 1 : 0);
  return hipGetLastError();
}

uint32_t deposit_blocks(uint32_t n, uint32_t per_thread)
{
  uint32_t grid = (n + per_thread * kDepositBlock - 1) / (per_thread * kDepositBlock);
  if (grid < 1) grid = 1;
  if (grid > kDepositMaxBlocks) grid = kDepositMaxBlocks;
  return grid;
}

// Deposit workgroups of a batch member whose rebuild is the deposit alone
// (grouped field solve, no per-beam Green's table): four particles per
// thread, at most kDepositMaxBlocksBatch workgroups, or kDepositMaxBlocksBig
// when the histogram takes more than 64 KB of LDS (one workgroup per CU).
// Fewer, fuller workgroups spread the zeroing and flush of each workgroup's
// histogram over more particles: 64 members of 4,194,304 particles on the
// 64 x 256 mesh, deposit per 160-element step 360 / 294 / 261 / 241 / 233 /
// 227 ms at 1,024 / 512 / 256 / 128 / 64 / 32 workgroups per member; the
// 256-beam scan on 32 x 128 takes 84 ms at 128 and 91 ms at 32.  A batch of
// few members fills the device instead, each with its share, by particles, of
// the workgroups that run at once (four members of 2,097,152 particles on
// 64 x 256: 32 workgroups each, half of the CUs, 120 us a rebuild; 64 each
// 77 us.  Seven members of 16,384 to 1,048,576 on 32 x 128: 24.1 -> 20.8).
uint32_t deposit_blocks_batch(uint32_t n, uint64_t total, uint32_t nr, uint32_t nz, uint32_t cus)
{
  const bool big = (size_t)nr * nz * sizeof(unsigned long long) > 65536;
  const uint32_t share = (uint32_t)((uint64_t)cus * (big ? 1 : 2) * n / total);
  uint32_t cap = big ? kDepositMaxBlocksBig : kDepositMaxBlocksBatch;
  if (cap < share) cap = share;
  uint32_t grid = (n + 4 * kDepositBlock - 1) / (4 * kDepositBlock);
  if (grid < 1) grid = 1;
  if (grid > cap) grid = cap;
  return grid;
}

#ifndef HPS_FAST_PUSH
// The workgroups of one simulation's rebuild: greens (with a Green's table of
// its own) and dep_blocks deposit workgroups.  A deposit of at least as many
// workgroups as the table has turns is combined with it (1,048,576 particles
// on 32 x 128, 256 and 132: 63.7 ms per 800-element step against 65.1 side by
// side); otherwise they run side by side (65,536 particles: 64 and 132,
// sc_build 1.55 ms per step against 1.82 combined) as long as the device
// holds them together: two workgroups a CU, one where the histogram takes
// more than half of its LDS.  Past that they share the room by work, a
// particle's deposit about two table entries, and the table's workgroups take
// several turns (300,007 particles on 64 x 256, 256 and 1,040 workgroups of
// 132 KB LDS in six rounds: 113 us a kick point; all 256 combined 109; 96 and
// 160: 102, 64 and 192 102, 128 and 128 106, 160 and 96 110).
void build_plan(BuildArgs& a, bool greens, uint32_t dep_blocks, uint32_t nr, uint32_t nz,
                uint32_t cus)
{
  const size_t lds = (size_t)nr * nz * sizeof(unsigned long long) + kBlockLdsReserve;
  const uint32_t room = cus * (2 * lds > kCuLds ? 1 : 2);
  const uint32_t entries = greens ? (nr + 1) * nz * nr : 0;
  const uint32_t turns = (entries + kDepositBlock - 1) / kDepositBlock;
  a.dep_blocks = dep_blocks;
  a.greens_wgs = turns;
  a.side = dep_blocks < turns ? 1 : 0;
  if (a.side && dep_blocks + turns > room) {
    const double work = 2.0 * a.b.n;
    const uint32_t share = (uint32_t)(room * (work / (work + entries)));
    if (dep_blocks > share) a.dep_blocks = share > 0 ? share : 1;
    const uint32_t left = room > a.dep_blocks ? room - a.dep_blocks : 1;
    a.greens_wgs = turns < left ? turns : left;
  }
}

hipError_t launch_sc_build(ScDev* sc, double* fld1, uint32_t nr, uint32_t nz, BeamArrays b,
                           const hps_beam_stats* st, int64_t* bins, bool deposit,
                           uint32_t cus, hipStream_t s)
{
  BuildArgs a;
  a.sc = sc; a.fld1 = fld1; a.b = b; a.st = st; a.bins = bins;
  // a lone beam spreads its deposit over up to one particle per thread (65,536
  // particles: 64 workgroups, 9.9 -> 9.0 ms per 160-element step); from
  // 262,144 particles on the 256-workgroup cap holds
  build_plan(a, true, deposit ? deposit_blocks(b.n, 1) : 0, nr, nz, cus);
  const size_t lds = (size_t)nr * nz * sizeof(unsigned long long);
  hipLaunchKernelGGL(k_sc_build, dim3(sc_build_blocks(a)), dim3(kDepositBlock), lds, s, a, nr,
                     nz);
  return hipGetLastError();
}

#endif

hipError_t launch_sc_build_batch(const BuildArgs* recs, const uint32_t* map, uint32_t nblocks,
                                 uint32_t nr, uint32_t nz, hipStream_t s)
{
  const size_t lds = (size_t)nr * nz * sizeof(unsigned long long);
  hipLaunchKernelGGL(k_sc_build_batch, dim3(nblocks), dim3(kDepositBlock), lds, s, recs, map, nr,
                     nz);
  return hipGetLastError();
}

namespace {

// Launch shape of the field sum: rows per wave and waves per workgroup.
struct FieldShape {
  int K;
  FieldGeom g;
  uint32_t threads, blocks;
};

FieldShape field_shape(uint32_t nr, uint32_t nz, int K, uint32_t waves)
{
  FieldShape f{};
  uint32_t P = 1;
  while (P < nr && P < 64) P <<= 1;
  const uint32_t radii = 64 / P;
  f.K = K;
  f.g.P = P;
  f.g.blocks = (nz + 1 + K - 1) / K;
  f.g.units = (nr + 1 + radii - 1) / radii * f.g.blocks;
  f.g.per_xcd = ((f.g.units + waves - 1) / waves + 7) / 8;
  f.threads = 64 * waves;
  f.blocks = 8 * f.g.per_xcd;
  return f;
}

// The launch shapes (every shape computes the same canonical sums): K = 8 / 4
// / 2 rows, 9 / 4 / 2 waves.
constexpr uint32_t kFieldShapes = 9;
constexpr uint32_t kFieldWaves[] = {9, 4, 2};
static_assert(kFieldWaves[0] <= kFieldMaxWaves, "launch bounds");

FieldShape field_shape_of(uint32_t nr, uint32_t nz, uint32_t idx)
{
  return field_shape(nr, nz, 8 >> (idx / 3), kFieldWaves[idx % 3]);
}

template <bool kBatch>
hipError_t launch_field_shape(const FieldShape& f, const FieldArgs* recs, const FieldArgs& one,
                              uint32_t nsim, uint32_t nr, uint32_t nz, hipStream_t s)
{
  const dim3 grid(f.blocks * nsim), block(f.threads);
  const size_t lds = (size_t)nr * nz * sizeof(double);
#define HPS_FIELD_LAUNCH(KK, DD)                                                                \
  if (kBatch)                                                                                   \
    hipLaunchKernelGGL((k_field_wave_batch<KK, DD>), grid, block, lds, s, recs, f.blocks, nr,   \
                       nz, f.g);                                                                \
  else                                                                                          \
    hipLaunchKernelGGL((k_field_wave<KK, DD>), grid, block, lds, s, one, nr, nz, f.g);
  if (f.K == 8) { HPS_FIELD_LAUNCH(8, 1) }
  else if (f.K == 4) { HPS_FIELD_LAUNCH(4, 3) }
  else { HPS_FIELD_LAUNCH(2, 7) }
#undef HPS_FIELD_LAUNCH
  return hipGetLastError();
}

}  // namespace

uint32_t field_batch_shapes() { return kFieldShapes; }

// Eight rows a wave spend 84 % of the vector instructions on products, four
// 80 %, but a table with fewer than one wave of eight rows per SIMD is bound
// by the length of a wave's chain, which four rows halve (65,536 particles on
// 32 x 128: 42.3 us a kick point with K = 4, 43.8 with 8, 44.4 with 2; seven
// members: 153.0 with 8, 153.4 with 4, 166.7 with 2).  Where the charges take
// more than half of the LDS a CU holds one workgroup, so it takes nine waves,
// as many as its registers allow (64 x 256, 2,145 waves on 239 workgroups:
// 109 us a kick point; eight waves are a second round of workgroups, 127;
// four 130; the sum alone, nine and four waves: 44.0 and 64.4 us there, 39.8
// and 42.9 on 48 x 256, 35.4 and 39.8 on 128 x 100); otherwise several small
// ones (four waves; nine 163, two 156 on the seven members).
uint32_t field_batch_default_shape(uint32_t nr, uint32_t nz, uint32_t nmem)
{
  const uint32_t k = field_shape(nr, nz, 8, 1).g.units * (uint64_t)nmem >= 1024 ? 0 : 1;
  const uint32_t w = (size_t)nr * nz * sizeof(double) > kCuLds / 2 ? 0 : 1;
  return 3 * k + w;
}

hipError_t launch_field(const FieldArgs& a, uint32_t nr, uint32_t nz, hipStream_t s)
{
  return launch_field_shape<false>(
      field_shape_of(nr, nz, field_batch_default_shape(nr, nz, 1)), nullptr, a, 1, nr, nz, s);
}

hipError_t launch_field_batch(const FieldArgs* recs, uint32_t nmem, uint32_t nr, uint32_t nz,
                              uint32_t shape, hipStream_t s)
{
  FieldArgs none{};
  if (shape >= kFieldShapes) shape = field_batch_default_shape(nr, nz, nmem);
  return launch_field_shape<true>(field_shape_of(nr, nz, shape), recs, none, nmem, nr, nz, s);
}

hipError_t launch_sums(BeamArrays b, const double* a, const double* bb, int filter, Partials pr,
                       hipStream_t s, const double* rel_ref, BeamSums* out, Readout* ro,
                       const hps_beam_stats* st)
{
  const uint32_t nch = (b.n + kChunk - 1) / kChunk;
  hipLaunchKernelGGL(k_sums, dim3(nch), dim3(kBlock), 0, s, b, a, bb, filter, pr, rel_ref);
  hipLaunchKernelGGL(k_sums_final, dim3(1), dim3(576), 0, s, pr, out, ro, st, b.w);
  return hipGetLastError();
}

hipError_t launch_set_stats(hps_beam_stats* st, const hps_beam_stats& v, hipStream_t s)
{
  hipLaunchKernelGGL(k_set_stats, dim3(1), dim3(64), 0, s, st, v);
  return hipGetLastError();
}

hipError_t launch_copy_beam(const BeamArrays& src, const BeamArrays& dst, hipStream_t s)
{
  hipLaunchKernelGGL(k_copy_beam, dim3(blocks_for(src.n)), dim3(kBlock), 0, s, src, dst);
  return hipGetLastError();
}

hipError_t launch_relative_phi(BeamArrays b, const double* ref, hipStream_t s)
{
  hipLaunchKernelGGL(k_relative_phi, dim3(blocks_for(b.n)), dim3(kBlock), 0, s, b, ref);
  return hipGetLastError();
}

hipError_t launch_lloss_flag(BeamArrays b, const double* avg, hipStream_t s)
{
  hipLaunchKernelGGL(k_lloss_flag, dim3(blocks_for(b.n)), dim3(kBlock), 0, s, b, avg);
  return hipGetLastError();
}

hipError_t launch_shift(double* a, uint32_t n, double v, hipStream_t s)
{
  hipLaunchKernelGGL(k_shift, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, n, v);
  return hipGetLastError();
}

hipError_t launch_scale(double* a, uint32_t n, double v, hipStream_t s)
{
  hipLaunchKernelGGL(k_scale, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, n, v);
  return hipGetLastError();
}

hipError_t launch_cut(const double* a, uint32_t* loss, uint32_t n, double lo, double hi,
                      hipStream_t s)
{
  hipLaunchKernelGGL(k_cut, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, loss, n, lo, hi);
  return hipGetLastError();
}

// --- synthetic beams ---------------------------------------------------------------

// Philox4x32-10 block (Salmon et al., SC'11): counter c, key (k0, k1).
__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t hi0 = __umulhi(0xD2511F53u, c[0]), lo0 = 0xD2511F53u * c[0];
    const uint32_t hi1 = __umulhi(0xCD9E8D57u, c[2]), lo1 = 0xCD9E8D57u * c[2];
    const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

__device__ __forceinline__ double u53(uint32_t a, uint32_t b)
{
  return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) / 9007199254740992.0;
}

// Coordinate c of particle i: center + sigma * z, z a standard normal
// truncated to |z| <= 3 by rejection with the attempt number in the Philox
// counter (i, c, attempt), Box-Muller from two 53-bit uniforms -- the
// sampler of hpsim_amd/configs.py (truncated_normal) with the engine's own
// log and cos.  Particle 0 is the reference particle (on axis, centred).
__global__ void k_sample_gaussian(BeamArrays b, uint32_t seed, GaussSpec g)
{
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= b.n) return;
  double* out[6] = {b.x, b.xp, b.y, b.yp, b.phi, b.w};
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    double z = 0.0;
    for (uint32_t attempt = 0; attempt <= 64; ++attempt) {
      uint32_t r[4] = {i, 0u, (uint32_t)c, attempt};
      philox(r, seed, 0x48505331u);
      const double u1 = 1.0 - u53(r[0], r[1]);
      const double u2 = u53(r[2], r[3]);
      double sn, cs;
      hps::sincos(2.0 * PI * u2, &sn, &cs);
      z = ::sqrt(-2.0 * hps::log(u1)) * cs;
      if (__builtin_fabs(z) <= 3.0) break;
    }
    double v = g.center[c] + g.sigma[c] * z;
    if (i == 0) v = c < 4 ? 0.0 : g.center[c];
    out[c][i] = v;
  }
  b.loss[i] = 0;
  b.lloss[i] = 0;
}

hipError_t launch_sample_gaussian(BeamArrays b, uint32_t seed, const GaussSpec& g, hipStream_t s)
{
  hipLaunchKernelGGL(k_sample_gaussian, dim3(blocks_for(b.n)), dim3(kBlock), 0, s, b, seed, g);
  return hipGetLastError();
}

hipError_t launch_probe(int fn, const double* x, const double* y, double* out, uint32_t n,
                        hipStream_t s)
{
  hipLaunchKernelGGL(k_probe, dim3(blocks_for(n)), dim3(kBlock), 0, s, fn, x, y, out, n);
  return hipGetLastError();
}

#ifdef HPS_FAST_PUSH
}  // namespace fast
#endif

}  // namespace hps
