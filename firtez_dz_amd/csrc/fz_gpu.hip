// MI355X (gfx950) implementation of the FIRTEZ-dz per-column forward synthesis
// and analytic response functions, behind the C ABI of include/firtez_gpu.h.
//
// Kernels
//   saha/rho/opac/tau kernels : FP64 microphysics per (column, height): Saha
//                  factors, the electron-density fixed point (sequential in
//                  height per column, warm start from the height below as in
//                  FORWARD1D, forward.f90:911-960), implicit EOS derivatives,
//                  continuum/line opacity, damping.  Writes a per-height
//                  record [field][z][column] (columns fastest).
//   rt_kernel<RF> : one thread per (column, wavelength).  Pass 1 bottom->top:
//                  propagation matrix, evolution operator, formal solution
//                  I_k = (1-O_k) S_k + O_k I_{k-1} (rtesolver.f90:163-265);
//                  the incoming I of every height goes to a scratch slab.
//                  Pass 2 top->bottom (response functions): recomputes the
//                  propagation matrix with derivatives, the local response
//                  dO(I_in - S) + (1-O) dS, and propagates it to the top with
//                  the running product O_nz...O_{k+1} (forward.f90:511-548).
//   hsra_saha/rho/opac_kernel, gain_kernel : continuum normalisation (normalization.f90).
//   saha_mid/he_rk4 kernels : hydrostatic RK4 from the top
//                  (hydrostatic_tools.f90:150-396), standalone or inside the
//                  forward with HYDROSTATIC: yes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/firtez_gpu.h"
#include "fz_micro.hpp"
#include "fz_rt.hpp"

namespace fz {

constexpr int MAXL = 16, MAXR = 8, MAXS = 32, MAXC = 1024, MAXNZ = 512, MAXBLK = 128;
// internal response set of the inversion forward when neither Pg, rho nor P0
// is inverted and HYDROSTATIC is off: slots T|Pg, Bx, By, Bz, v_z only (the
// Pg|T and rho|T directional derivatives are not formed)
constexpr int RF_CART_TBV = 4;
constexpr int TBV_SLOT[8] = {0, -1, -1, 1, 2, 3, 4, -1};   // slot of an inverted parameter there

constexpr int RT_WAVE = 64;   // wavelengths per radiative-transfer workgroup (one wave)
constexpr int NATM = 12;
enum { A_T = 0, A_PG, A_RHO, A_PEL, A_MU, A_BX, A_BY, A_BZ, A_VX, A_VY, A_VZ, A_TAU };

// Per-height record of a column, rec floats at micro[(k * rncol + col - rcol0) * rec]
// (columns rcol0 .. rcol0 + rncol - 1 are held):
// a head of REC_HEAD floats, then per region REC_REG floats and REC_SLOT per
// line of the region, each part a whole number of float4, so that a wave
// copies the heights it needs next into LDS with 16-byte loads and every lane
// reads them from there.  kappa_5000 is kept apart, [nz][rncol] after the
// records (tau_kernel reads it along the columns).
//   head    flag, T, 1/T, 1/sqrt(T) | v_z, |B|, sgf/2, cgf/4 | qf/2, qf/4, cg/2, sg |
//           cos 2phi, sin 2phi, sg cg, line-optical-depth factor | d|B|/dB (3), d gamma/dB (3), d phi/dBx, dBy
//           (sgf, cgf = 1 -+ cos^2 of the inclination; qf = sgf, 0 without a transverse field, whose frame is unturned)
//   region  kappa_c and its three derivatives
//   slot    kl, a, dkl/dT, da/dT | dkl/dPg, dkl/drho, da/dPg, da/drho | VoigtPoly (13) | 1/Doppler width,
//           -1/(Doppler temperature), Doppler shift (mA)
constexpr int REC_HEAD = 24, REC_REG = 4, REC_SLOT = 24;

struct Cfg {
  int nlines, nreg, nslot, numw, nz;
  int rec;              // floats of a per-height record
  LineConst line[MAXL];
  float dopfac[MAXL];   // Doppler width (mA) = dopfac * sqrt(T)
  float idopfac[MAXL];  // 1 / dopfac
  float vfac[MAXL];     // Doppler shift (mA) = vfac * v_z   (absorption_matrix.f90:1896)
  int reg_nblend[MAXR], reg_slot0[MAXR], reg_pix0[MAXR], reg_nwave[MAXR];
  int reg_rec[MAXR];    // first float of the region in the per-height record
  double reg_wstart[MAXR], reg_wstep[MAXR], reg_l0main[MAXR];
  int slot_line[MAXS];
  float slot_bldiff[MAXS];
  // Zeeman components sorted sigma_r, pi, sigma_b (those of no strength left
  // out): shift from the type's centre, strength and its products with the
  // shift and its square; per type the strength-weighted centre and the sums
  // of strength and strength * shift over sqrt(pi)
  int comp0[MAXL], ntype[MAXL][3];
  float4 comp[MAXC], type[MAXL][3];
  // what the transfer needs of a slot's line, together: the scalar loads of a
  // layer then wait once
  struct SlotRt {
    int comp0, n[3];
    float bldiff, vfac, pad[2];
    float4 type[3];
  } slot_rt[MAXS];
  float dz_cm[MAXNZ];
  double zz[MAXNZ];    // heights in km, rounded through REAL(4) like MODEL(:,13)
  // radiative-transfer workgroups of one column: each covers up to RT_WAVE
  // wavelengths of a single region, so the column and the region (and every
  // per-height quantity read) are uniform across the wave
  int nbpc;
  int blk_reg[MAXBLK], blk_l0[MAXBLK], blk_n[MAXBLK];
  // hydrostatic RK4 steps k+1 -> k (hydrostatic_tools.f90:166-212): step dz
  // and the two weights of the mid-step temperature, with the running height
  // t0 accumulated exactly as the reference does
  double he_dz[MAXNZ], he_a[MAXNZ], he_b[MAXNZ];
  // m_u g dz / k per height (GET_HYD_DERIVATIVES, forward.f90:1033-1061)
  float he_cte[MAXNZ];
  // spectral LSF (MLSF): on/off and LSF_VALID per region
  int lsf_on;
  int reg_lsf[MAXR];
  // microturbulence xi: the Doppler width of line li is that of the
  // temperature T + xi_t[li], xi_t = m xi^2 / (2 k) (xi_on 0: thermal only)
  int xi_on;
  double xi_t[MAXL];
  float xi_tf[MAXL];
};
__constant__ Cfg c_cfg;

// ---------------------------------------------------------------- microphysics
// FORWARD1D's per-height physics (forward.f90:911-1006) over a tile of
// columns.  A column loop with one thread per column would give a few ten
// thousand threads (~1 wave per SIMD); only the electron-density fixed point
// is sequential in height (warm start from the height below), so the work is
// split into:
//   saha_kernel  one thread per (height, column): partition functions and the
//                Saha factors of all 92 elements -> sbuf[k][e][4][column]
//   rho_group_kernel  16 to 64 lanes per column, heights bottom->top: only the
//                warm-started electron-density fixed point (GET_RHO), reading
//                the factors from sbuf -> rho, mu, Pe and (n_e, N_H) per height
//   deriv_kernel, opac_kernel  one thread per (height, column): EOS derivatives,
//                continuum and line opacity, damping -> the per-height record
//   tau_kernel   one thread per column: the REAL(4) log tau5 trapezoid
// FP64 throughout; the fixed point keeps the reference's iteration path
// (stopping rule 1e-4, warm start).
struct MicroTile {
  int ncol, col0, ntile, der;
  int rcol0, rncol;   // columns held in micro
  float* atm;
  float* micro;
  double* sbuf;    // [nz][92][4][ntile]
  double* eos;     // [2][nz][ntile]: n_e, N_H
  double* deriv;   // [8][nz][ntile]: the DERIVVAR scalars (with response functions)
  int32_t* status; // [ncol]
  // NLTE departure coefficients [2][nz][nreg] (POPL, POPU), or null (LTE)
  const double* pop;
};

// The Saha factors of every (height, column), one thread each, all lanes of a
// wave at the same element; with DER their T derivatives too (without
// them those rows are neither written nor read).
// Bounds: with DER the writes (2944 B per height and column), without them the FP64
// issue about as much as the writes.  The partition functions' derivatives, four
// divisions and two general exponentials per element, and the rows of zeros left out
// where nothing reads them: 82944 columns x 96 heights 5.5 -> 2.75 ms; with DER
// 36864 x 96 take 2.15 ms before and after.
template <bool DER>
__global__ void __launch_bounds__(256) saha_kernel(MicroTile a) {
  const int nz = c_cfg.nz;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)nz * a.ntile) return;
  const int k = (int)(t / a.ntile), ct = (int)(t - (long)k * a.ntile);
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  const SahaT s((double)a.atm[A_T * ps + k * cs + a.col0 + ct]);
  double* o = a.sbuf + (long)k * FZ_NELEM * 4 * a.ntile + ct;
  const int per = (FZ_NELEM + gridDim.y - 1) / gridDim.y;   // elements of this workgroup
#pragma unroll 1
  for (int i = blockIdx.y * per; i < min(FZ_NELEM, (int)(blockIdx.y + 1) * per); ++i) {
    double a1, a2, da1, da2;
    saha_element<DER>(i, s, a1, a2, da1, da2);
    o[(long)(i * 4 + 0) * a.ntile] = a1;
    o[(long)(i * 4 + 1) * a.ntile] = a2;
    if constexpr (DER) {
      o[(long)(i * 4 + 2) * a.ntile] = da1;
      o[(long)(i * 4 + 3) * a.ntile] = da2;
    }
  }
}

// GET_RHO (chemical_equilibrium.f90:165-278) for one column by a group of G
// lanes: lane q holds the Saha factors of elements q, q + G, ... of a height
// in registers.  Per iteration an element adds
//   abf (1 + i) / (x + 1 + i),  x = n_e a1, i = 1 / (n_e a2)
// (n_II + n_III over N_H; hydrogen adds n_III - n_I, abf (i - x) / (x + 1 + i)),
// one FP64 reciprocal where the reference's quotients (:1601-1652) take four
// divisions, and no quotient that overflows before the fractions themselves
// underflow.  1 / a2 is formed once per height and 1 / n_e once per iteration.
//
// The terms are summed by one fixed tree whatever G is: elements j and j + 64,
// then residues 32, 16 and 8 apart, then 1, 2 and 4 apart, the levels below G
// by cross-lane moves and the others within the lane.  Every group size thus
// gives the same bits, so a column's result does not depend on the tile it
// is launched in.
//
// Bound: the chain of one iteration (the reciprocals, the tree and the
// stopping test), and with many columns the issue of its FP64 instructions.
// Against the sequential fold of 91 terms through LDS with eight lanes per
// column that this replaces: hydrostatic integration of 16 columns x 64
// heights 8.9 -> 0.55 ms, of 9216 x 96 heights 26.9 -> 2.2 ms; the forward's
// fixed point of 82944 columns x 96 heights 24.4 -> 5.9 ms.
template <int CTRL>
__device__ __forceinline__ double dpp64(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true));
}

// x of a row of 16 lanes (of 32 lanes) plus x of its neighbour
__device__ __forceinline__ double add_swap16(double x) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
__device__ __forceinline__ double add_swap32(double x) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}

// the fixed tree over the lane's terms t[m] of elements q + G m
template <int G, int NS>
__device__ __forceinline__ double group_sum(double (&t)[NS]) {
  constexpr int M = 64 / G;            // residues mod 64 held by a lane
#pragma unroll
  for (int m = 0; m + M < NS; ++m) t[m] += t[m + M];
#pragma unroll
  for (int w = M / 2; w > 0; w /= 2)
#pragma unroll
    for (int m = 0; m < w; ++m) t[m] += t[m + w];
  double s = t[0];
  if constexpr (G >= 64) s = add_swap32(s);
  if constexpr (G >= 32) s = add_swap16(s);
  if constexpr (G >= 16) s += dpp64<0x128>(s);   // row_ror:8
  s += dpp64<0xB1>(s);                           // lanes 1 apart
  s += dpp64<0x4E>(s);                           // 2 apart
  s += dpp64<0x141>(s);                          // row_half_mirror: 4 apart, quads being uniform
  return s;
}

template <int G>
struct RhoGroup {
  static constexpr int NS = (FZ_NELEM + G - 1) / G;
  int q;
  double ab[NS];   // abundances of the lane's elements (0 past the last one)
  __device__ __forceinline__ explicit RhoGroup(int lane) : q(lane & (G - 1)) {
#pragma unroll
    for (int m = 0; m < NS; ++m) ab[m] = q + G * m < FZ_NELEM ? g_c.abfac[q + G * m] : 0.0;
  }
  // a1, a2 of a height; base: [element][4][stride] of the column
  __device__ __forceinline__ void load(const double* __restrict__ base, long stride, double (&a1)[NS],
                                       double (&a2)[NS]) const {
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      const int j = q + G * m;
      a1[m] = j < FZ_NELEM ? base[(long)(j * 4 + 0) * stride] : 1.0;
      a2[m] = j < FZ_NELEM ? base[(long)(j * 4 + 1) * stride] : 1.0;
    }
  }
  static __device__ __forceinline__ void invert(double (&a2)[NS]) {
#pragma unroll
    for (int m = 0; m < NS; ++m) a2[m] = rcp64(a2[m]);
  }
  // the warm-started fixed point on a1 and ia2 = 1 / a2: the reference's
  // iteration path (damping 1/2, stop at 1e-4, at most 100).  ne: start in,
  // result out; pelec is the start's electron pressure, as the reference returns
  __device__ __forceinline__ int solve(const double (&a1)[NS], const double (&ia2)[NS], double T, double PG,
                                       double& ne, double& nh, double& pelec, double& dens, double& mu) const {
    const double kT = KBOL * T;
    double n = ne;
    if (n != n) n = 0.0;
    if (n < 1.0) n = PG / (101.0 * kT);
    pelec = n * kT;
    if (pelec > PG) n = (PG * 0.5) / kT;
    const double isa = 1.0 / (g_c.deno_sa * kT);
    double nnew = n, h = 0.0;
    int iter = 1;
    bool more = true;
    while (more && iter <= 100 && h >= 0.0) {
      const double nold = nnew, ine = rcp64(nold);
      h = fma(-nold, kT, PG) * isa;
      double t[NS];
#pragma unroll
      for (int m = 0; m < NS; ++m) {
        const double x = nold * a1[m], i = ia2[m] * ine;
        const double s = (m == 0 && q == 0) ? -x : 1.0;
        t[m] = fma(ab[m], i, ab[m] * s) * rcp64((x + 1.0) + i);
      }
      const double est = h * group_sum<G, NS>(t);
      nnew = (fmax(est, 0.0) + nold) * 0.5;
      more = fabs(nnew - nold) > 1.0e-4 * fabs(nnew);
      ++iter;
    }
    if (iter >= 100 || h < 0.0) return ERR_EOS;
    n = nnew;
    h = (PG - n * kT) / (g_c.deno_sa * kT);
    dens = h * g_c.deno_sam + n * MELE;
    mu = ((dens * kT) / MAMU) * (1.0 / PG);
    if (h != h || n != n) return ERR_NAN;
    if (n < 0.0 || h <= 0.0) return ERR_EOS;
    ne = n;
    nh = h;
    return ERR_OK;
  }
};

constexpr int RHO_BLOCK = 256;

template <int G>
__global__ void __launch_bounds__(RHO_BLOCK, G == 16 ? 3 : 4) rho_group_kernel(MicroTile a) {
  using R = RhoGroup<G>;
  const R g(threadIdx.x & 63);
  const int ct = (int)(((long)blockIdx.x * blockDim.x + threadIdx.x) / G);
  const bool active = ct < a.ntile;
  // a group past the tile repeats the last column without writing, so that
  // every group of a wave runs the same code
  const int cc = active ? ct : a.ntile - 1;
  const bool wr = active && g.q == 0;
  const int nz = c_cfg.nz, col = a.col0 + cc;
  const long cs = a.ncol, ps = (long)nz * a.ncol, hs = (long)FZ_NELEM * 4 * a.ntile;
  const double* sb = a.sbuf + cc;
  double ne = 0.0;
  int err = ERR_OK;
  // the next height's factors are loaded while this one iterates
  double n1[R::NS], n2[R::NS];
  g.load(sb, a.ntile, n1, n2);
  float Tn = a.atm[A_T * ps + col], Pn = a.atm[A_PG * ps + col];
  for (int k = 0; k < nz; ++k) {
    const double T = (double)Tn, P = (double)Pn;
    double a1[R::NS], ia2[R::NS];
#pragma unroll
    for (int m = 0; m < R::NS; ++m) {
      a1[m] = n1[m];
      ia2[m] = n2[m];
    }
    const int kn = min(k + 1, nz - 1);
    g.load(sb + kn * hs, a.ntile, n1, n2);
    Tn = a.atm[A_T * ps + kn * cs + col];
    Pn = a.atm[A_PG * ps + kn * cs + col];
    R::invert(ia2);
    double nh, pel, dens, mu;
    err = g.solve(a1, ia2, T, P, ne, nh, pel, dens, mu);
    if (err) break;
    if (wr) {
      a.atm[A_RHO * ps + k * cs + col] = (float)dens;
      a.atm[A_MU * ps + k * cs + col] = (float)mu;
      a.atm[A_PEL * ps + k * cs + col] = (float)pel;
      a.eos[(long)k * a.ntile + cc] = ne;
      a.eos[((long)nz + k) * a.ntile + cc] = nh;
    }
  }
  if (wr) a.status[col] = err;
}

// The implicit EOS derivatives (GET_DNHYDDTEMP and its four solves,
// chemical_equilibrium.f90:2008-2052) per (height, column), kept apart from
// the opacities so that neither kernel carries the other's registers.
__global__ void __launch_bounds__(256) deriv_kernel(MicroTile a) {
  const int nz = c_cfg.nz;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)nz * a.ntile) return;
  const int k = (int)(t / a.ntile), ct = (int)(t - (long)k * a.ntile), col = a.col0 + ct;
  if (a.status[col] != 0) return;
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  const double T = (double)a.atm[A_T * ps + k * cs + col], P = (double)a.atm[A_PG * ps + k * cs + col];
  const float rhof = a.atm[A_RHO * ps + k * cs + col];
  const double ne = a.eos[(long)k * a.ntile + ct];
  const SahaView s(a.sbuf + (long)k * FZ_NELEM * 4 * a.ntile + ct, a.ntile);
  Deriv d = {};
  eos_derivatives(s, T, P, (double)rhof, ne, d);
  const long ds = (long)nz * a.ntile, o = (long)k * a.ntile + ct;
  a.deriv[0 * ds + o] = d.nh_T_pg;
  a.deriv[1 * ds + o] = d.nh_T_rho;
  a.deriv[2 * ds + o] = d.nh_pg_T;
  a.deriv[3 * ds + o] = d.nh_rho_T;
  a.deriv[4 * ds + o] = d.ne_pg_T;
  a.deriv[5 * ds + o] = d.ne_T_rho;
  a.deriv[6 * ds + o] = d.ne_T_pg;
  a.deriv[7 * ds + o] = d.ne_rho_T;
}

// Bound by its FP64 chains and their latency: limited to 256 registers (22 of them
// then spill, outside the loops) two waves share a SIMD instead of one: 82944
// columns x 96 heights 2.65 -> 2.15 ms, with response functions 36864 x 96 1.57 -> 1.27 ms.
__global__ void __launch_bounds__(256, 2) opac_kernel(MicroTile a) {
  const int nz = c_cfg.nz;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)nz * a.ntile) return;
  const int k = (int)(t / a.ntile), ct = (int)(t - (long)k * a.ntile), col = a.col0 + ct;
  if (a.status[col] != 0) return;
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  float4* const R = reinterpret_cast<float4*>(a.micro + ((long)k * a.rncol + col - a.rcol0) * c_cfg.rec);
  const float* at = a.atm + k * cs + col;
  const float Tf = at[A_T * ps], vz = at[A_VZ * ps], iT = 1.0f / Tf, rsT = rsqrtf(Tf);
  {
    // FP32 field geometry and the chain rule (|B|, gamma, phi) -> (Bx, By, Bz)
    // for the radiative transfer.  With B = 0 every field derivative is zero,
    // as in the reference (absorption_matrix.f90:1842-1866); with a vertical
    // field the azimuth terms are dropped (the reference's d cos2phi / dBx is
    // 0/0 there).
    const float bx = at[A_BX * ps], by = at[A_BY * ps], bz = at[A_BZ * ps];
    const Geo g = geometry(bx, by, bz);
    const float bt2 = bx * bx + by * by, bt = sqrtf(bt2), B2 = g.B * g.B;
    const bool hasB = g.B > 0.f, hasT = bt2 > 0.f;
    const float iB = hasB ? 1.f / g.B : 0.f, iBt = hasT ? 1.f / (B2 * bt) : 0.f, ibt2 = hasT ? 1.f / bt2 : 0.f;
    const float qf = hasT ? g.sgf : 0.f;
    R[1] = {vz, g.B, 0.5f * g.sgf, 0.25f * g.cgf};
    R[2] = {0.5f * qf, 0.25f * qf, 0.5f * g.cg, g.sg};
    R[4] = {bx * iB, by * iB, bz * iB, bz * bx * iBt};
    R[5] = {bz * by * iBt, hasB ? -bt / B2 : 0.f, -by * ibt2, bx * ibt2};
    // the frame's angle; the line-optical-depth factor follows below
    R[3] = {hasT ? g.c2p : 1.f, hasT ? g.s2p : 0.f, g.sg * g.cg, 0.f};
  }
  const double T = (double)a.atm[A_T * ps + k * cs + col], P = (double)a.atm[A_PG * ps + k * cs + col];
  const float rhof = a.atm[A_RHO * ps + k * cs + col];
  const double ne = a.eos[(long)k * a.ntile + ct], nh = a.eos[((long)nz + k) * a.ntile + ct];
  const SahaView s(a.sbuf + (long)k * FZ_NELEM * 4 * a.ntile + ct, a.ntile);
  Deriv d = {};
  if (a.der) {
    const long ds = (long)nz * a.ntile, o = (long)k * a.ntile + ct;
    d.nh_T_pg = a.deriv[0 * ds + o];
    d.nh_T_rho = a.deriv[1 * ds + o];
    d.nh_pg_T = a.deriv[2 * ds + o];
    d.nh_rho_T = a.deriv[3 * ds + o];
    d.ne_pg_T = a.deriv[4 * ds + o];
    d.ne_T_rho = a.deriv[5 * ds + o];
    d.ne_T_pg = a.deriv[6 * ds + o];
    d.ne_rho_T = a.deriv[7 * ds + o];
  }
  (void)P;
  (void)rhof;
  double kc[4];
  int err = opac_cont(T, 5000.0, ne, nh, d, false, kc);
  if (!err) {
    const double kc5 = kc[0] / nh * (1.0 / MAMU);
    const bool bnd = (k == 0) || (kc5 >= 2.0e10);     // forward.f90:884,931,971
    R[0] = {bnd ? 1.0f : 0.0f, Tf, iT, rsT};
    a.micro[(long)nz * a.rncol * c_cfg.rec + (long)k * a.rncol + col - a.rcol0] = (float)kc5;
    // the opacities are formed wherever kc5 is below the threshold, the
    // bottom height included (its absorption matrix feeds LINE OPTICAL DEPTH,
    // forward.f90:931-968, while the transfer takes it as the boundary)
    const bool opaque = kc5 >= 2.0e10;
    if (opaque) return;
    // 1 / (N_H m_u MW) (LINE OPTICAL DEPTH: KLINTAU = ETAI / N_H / m_u / MW; 0 where opaque)
    R[3].w = (float)(1.0 / (nh * MAMU * (double)a.atm[A_MU * ps + k * cs + col]));
    for (int r = 0; r < c_cfg.nreg && !err; ++r) {
      float4* Q = R + c_cfg.reg_rec[r] / 4;
      err = opac_cont(T, c_cfg.reg_l0main[r], ne, nh, d, a.der != 0, kc);
      *Q++ = {(float)kc[0], (float)kc[1], (float)kc[2], (float)kc[3]};
      for (int b = 0; b < c_cfg.reg_nblend[r] && !err; ++b, Q += REC_SLOT / 4) {
        const int li = c_cfg.slot_line[c_cfg.reg_slot0[r] + b];
        const LineConst& L = c_cfg.line[li];
        double kl[4] = {0, 0, 0, 0}, dm[4] = {0, 0, 0, 0};
        // the region's departure coefficients for every line of the region (forward.f90:949)
        const double bl = a.pop ? a.pop[((long)0 * nz + k) * c_cfg.nreg + r] : 1.0;
        const double bu = a.pop ? a.pop[((long)nz + k) * c_cfg.nreg + r] : 1.0;
        const double Td = T + c_cfg.xi_t[li];
        err = opac_line(L, T, ne, nh, s, d, a.der != 0, kl, bl, bu, Td);
        damping(L, T, nh, d, a.der != 0, dm, Td);
        const float rsd = c_cfg.xi_on ? rsqrtf(Tf + c_cfg.xi_tf[li]) : rsT;   // 1/sqrt(Doppler temperature)
        float v[NVP];
        voigt_poly((double)(float)dm[0], v);
        Q[0] = {(float)kl[0], (float)dm[0], (float)kl[1], (float)dm[1]};
        Q[1] = {(float)kl[2], (float)kl[3], (float)dm[2], (float)dm[3]};
        Q[2] = {v[0], v[1], v[2], v[3]};
        Q[3] = {v[4], v[5], v[6], v[7]};
        Q[4] = {v[8], v[9], v[10], v[11]};
        Q[5] = {v[12], c_cfg.idopfac[li] * rsd, c_cfg.xi_on ? -rsd * rsd : -iT, c_cfg.vfac[li] * vz};
      }
    }
  }
  if (err) atomicMax(&a.status[col], err);
}

__global__ void __launch_bounds__(64) tau_kernel(MicroTile a) {
  const int ct = blockIdx.x * blockDim.x + threadIdx.x;
  if (ct >= a.ntile) return;
  const int nz = c_cfg.nz, col = a.col0 + ct;
  if (a.status[col] != 0) return;
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  const float* kc5 = a.micro + (long)nz * a.rncol * c_cfg.rec + col - a.rcol0;
  const long rs = a.rncol;
  // log tau_5000 by the REAL(4) trapezoid of forward.f90:1000-1006 (z in km)
  float tau = 1e-9f;
  a.atm[A_TAU * ps + (nz - 1) * cs + col] = log10f(tau);
  // eight heights' loads together: the trapezoid is a chain, its terms are not
  float xn = kc5[(nz - 1) * rs] * a.atm[A_RHO * ps + (nz - 1) * cs + col];
  for (int k0 = nz - 2; k0 >= 0; k0 -= 8) {
    float q[8], r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = max(k0 - i, 0);
      q[i] = kc5[k * rs];
      r[i] = a.atm[A_RHO * ps + k * cs + col];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 - i;
      if (k < 0) break;
      const float xk = q[i] * r[i];
      const float x = (xk + xn) / 2.0f;
      tau = (float)((double)tau + (double)x * ((c_cfg.zz[k + 1] - c_cfg.zz[k]) * 1000.0 * 100.0));
      a.atm[A_TAU * ps + k * cs + col] = log10f(tau);
      xn = xk;
    }
  }
}

// ---------------------------------------------------------------- hydrostatic equilibrium
// RK4_INTEGRATION_LOG (hydrostatic_tools.f90:150-222, RK4_LOG :350-396) over
// a tile: the Saha factors at the heights come from saha_kernel, those at the
// RK4 mid-step temperatures from saha_mid_kernel, and he_rk4_group_kernel
// (16 to 64 lanes per column, top -> bottom) runs only the fixed points.
__device__ __forceinline__ double he_tmid(int k, double tm0, double tm1) {
  const double dz = c_cfg.he_dz[k];
  return tm0 / dz * c_cfg.he_a[k] + tm1 / dz * c_cfg.he_b[k];
}

__global__ void __launch_bounds__(256) saha_mid_kernel(MicroTile a, double* __restrict__ smid) {
  const int nz = c_cfg.nz;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)(nz - 1) * a.ntile) return;
  const int k = (int)(t / a.ntile), ct = (int)(t - (long)k * a.ntile);
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  const double tm0 = (double)a.atm[A_T * ps + (k + 1) * cs + a.col0 + ct];
  const double tm1 = (double)a.atm[A_T * ps + k * cs + a.col0 + ct];
  const SahaT s(he_tmid(k, tm0, tm1));
  double* o = smid + (long)k * FZ_NELEM * 4 * a.ntile + ct;
  const int per = (FZ_NELEM + gridDim.y - 1) / gridDim.y;
#pragma unroll 1
  for (int i = blockIdx.y * per; i < min(FZ_NELEM, (int)(blockIdx.y + 1) * per); ++i) {
    double a1, a2, da1, da2;
    saha_element<false>(i, s, a1, a2, da1, da2);
    o[(long)(i * 4 + 0) * a.ntile] = a1;
    o[(long)(i * 4 + 1) * a.ntile] = a2;
  }
}

// RK4_INTEGRATION_LOG by groups of G lanes per column, each fixed point as in
// rho_group_kernel; the integration scalars are identical in the lanes of a
// group.  The factors of height k + 1 (first step) are those of the previous
// height's last two; the mid-step and the new height's are loaded a height
// ahead.  Writes Pg, rho, Pe, mu of every height and, for the forward, (n_e, N_H) with
// n_e = Pe/(k T) from the REAL(4) Pe and T (forward.f90:904).
template <int G>
__global__ void __launch_bounds__(RHO_BLOCK, 2) he_rk4_group_kernel(MicroTile a, const double* __restrict__ smid) {
  using R = RhoGroup<G>;
  const R g(threadIdx.x & 63);
  const int ct = (int)(((long)blockIdx.x * blockDim.x + threadIdx.x) / G);
  const bool active = ct < a.ntile;
  const int cc = active ? ct : a.ntile - 1;
  const bool wr = active && g.q == 0;
  const int nz = c_cfg.nz, col = a.col0 + cc;
  const long cs = a.ncol, ps = (long)nz * a.ncol;
  const long hs = (long)FZ_NELEM * 4 * a.ntile;
  const double* SH = a.sbuf + cc;
  const double* SM = smid + cc;
  auto A = [&](int p, int k) -> float& { return a.atm[p * ps + k * cs + col]; };
  int err = 0;
  const int top = nz - 1;
  double u0 = log((double)A(A_PG, top));
  double nel = (double)A(A_PEL, top) / KBOL / (double)A(A_T, top);
  double nh = 0.0, pel = 0.0, dens = 0.0, mw = 0.0;
  // factors (a1, 1/a2) of the height above, of the mid step and of the new height
  double h1[R::NS], h2[R::NS], m1[R::NS], m2[R::NS], k1a[R::NS], k2a[R::NS];
  double pm1[R::NS], pm2[R::NS], pk1[R::NS], pk2[R::NS];
  g.load(SH + top * hs, a.ntile, h1, h2);
  {
    const int kn = max(top - 1, 0);
    g.load(SM + kn * hs, a.ntile, pm1, pm2);
    g.load(SH + kn * hs, a.ntile, pk1, pk2);
  }
  R::invert(h2);
  double tm0 = (double)A(A_T, top);
  err = g.solve(h1, h2, tm0, exp(u0), nel, nh, pel, dens, mw);
  if (wr) {
    A(A_PG, top) = (float)exp(u0);
    A(A_RHO, top) = (float)dens;
    A(A_PEL, top) = (float)pel;
    A(A_MU, top) = (float)mw;
    if (a.eos) a.eos[((long)nz + top) * a.ntile + cc] = nh;
  }
  // RK4_SOLVE_LOG (hydrostatic_tools.f90:53-71)
  auto rhs = [&](const double (&f1)[R::NS], const double (&f2)[R::NS], double lnp, double tem) -> double {
    double mu = 0.0;
    const int e = g.solve(f1, f2, tem, exp(lnp), nel, nh, pel, dens, mu);
    if (e) err = e;
    return -mu * MAMU * GRAV / (KBOL * tem);
  };
  for (int k = nz - 2; k >= 0 && !err; --k) {
    const double dz = c_cfg.he_dz[k];
    const double tm1 = (double)A(A_T, k), tmid = he_tmid(k, tm0, tm1);
#pragma unroll
    for (int m = 0; m < R::NS; ++m) {
      m1[m] = pm1[m];
      m2[m] = pm2[m];
      k1a[m] = pk1[m];
      k2a[m] = pk2[m];
    }
    const int kn = max(k - 1, 0);
    g.load(SM + kn * hs, a.ntile, pm1, pm2);
    g.load(SH + kn * hs, a.ntile, pk1, pk2);
    const double s1 = rhs(h1, h2, u0, tm0) * dz;
    R::invert(m2);
    const double s2 = rhs(m1, m2, u0 + s1 / 2.0, tmid) * dz;
    const double s3 = rhs(m1, m2, u0 + s2 / 2.0, tmid) * dz;
    R::invert(k2a);
    const double s4 = rhs(k1a, k2a, u0 + s3, tm1) * dz;
    const double u1 = u0 + 1.0 / 6.0 * (s1 + 2.0 * s2 + 2.0 * s3 + s4);
    const double pg = exp(u1);
    const int e = g.solve(k1a, k2a, tm1, pg, nel, nh, pel, dens, mw);
    if (e) err = e;
    if (wr) {
      A(A_PG, k) = (float)pg;
      A(A_RHO, k) = (float)dens;
      A(A_PEL, k) = (float)pel;
      A(A_MU, k) = (float)mw;
      if (a.eos) a.eos[((long)nz + k) * a.ntile + cc] = nh;
    }
#pragma unroll
    for (int m = 0; m < R::NS; ++m) {
      h1[m] = k1a[m];
      h2[m] = k2a[m];
    }
    tm0 = tm1;
    u0 = u1;
  }
  if (a.eos && wr)
    for (int k = 0; k < nz; ++k)
      a.eos[(long)k * a.ntile + cc] = (double)A(A_PEL, k) / KBOL / (double)A(A_T, k);
  if (wr) a.status[col] = err;
}

// ---------------------------------------------------------------- radiative transfer
// Launch description of rt_kernel (host side; the kernel receives the
// pointers as separate restrict-qualified arguments so that loads whose
// address is uniform across the wave become scalar loads).
// One radiative-transfer workgroup of a cube with per-pixel spectral
// windows: column, region, first wavelength (index in the configured grid),
// wavelengths in this workgroup (<= RT_WAVE) and their position in the
// pixel's own spectrum.
struct RtItem {
  int col;
  short r, n;
  int l0, lout;
};

struct RtArgs {
  int ncol;          // columns in the whole cube (strides of atm/micro)
  int col0;          // first column of this launch
  int ntile;         // columns in this launch
  int rcol0, rncol;  // columns held in micro
  const float* atm;
  const float* micro;
  const float* gain; // [numw][4]
  int32_t* status;
  float* stokes;     // [ncol][4][numw]
  float* jac;        // [ncol - jcol0][np][nz][4][numw]
  int jcol0;         // column of jac[0]
  float* scratch;    // [nz][4][ntile*numw]
  int chunk;         // heights of the record that a wave holds in LDS at a time
  // per-pixel windows (items null: every column uses every wavelength)
  const RtItem* items;   // this launch's workgroups
  const int64_t* poff;   // [ncol+1] prefix of the pixels' wavelength counts: Stokes at 4*poff[col]
  const double* pop;     // NLTE departure coefficients [2][nz][nreg], or null (LTE)
  float* fs;             // FULL_STOKES [ncol][nz][4][numw] (Stokes after every height), or null
};

// The record of one (column, height) as the transfer reads it, from LDS or
// from global memory (P: const float4* of either)
template <class P>
struct Rec {
  P h, r;   // head, region
};

// sums over the component types (sigma_r, pi, sigma_b) of one quantity: the
// absorption profiles (h) and the dispersion profiles (f)
struct Sums {
  float h[3], f[3];
};
__device__ __forceinline__ void zero(Sums& x) {
#pragma unroll
  for (int t = 0; t < 3; ++t) x.h[t] = x.f[t] = 0.f;
}

// profile combination of the three types into the frame's five elements
// (absorption_matrix.f90:1946-2230)
struct Mix {
  float i0, i1, q0, q1, v;   // I = i0 pi + i1 (r + b), q = q0 pi - q1 (r + b), V = v (r - b)
};
__device__ __forceinline__ Five mix(const Mix& m, const Sums& x) {
  const float sh = x.h[0] + x.h[2], sf = x.f[0] + x.f[2];
  return {fmaf(m.i0, x.h[1], m.i1 * sh), fmaf(m.q0, x.h[1], -(m.q1 * sh)), m.v * (x.h[0] - x.h[2]),
          fmaf(m.q0, x.f[1], -(m.q1 * sf)), m.v * (x.f[0] - x.f[2])};
}

__device__ __forceinline__ VoigtPoly voigt_load(const float4& a, const float4& b, const float4& c, float d) {
  return {{a.x, a.y, a.z, a.w, b.x, b.y}, {b.z, b.w, c.x, c.y, c.z, c.w, d}};
}

// Profile sums of region r's lines times kl dz at one height
template <class P>
__device__ __forceinline__ Sums absorb(P q, int r, float wave, float B, float dz) {
  Sums X;
  zero(X);
  for (int b = 0; b < c_cfg.reg_nblend[r]; ++b, q += REC_SLOT / 4) {
    const Cfg::SlotRt sc = c_cfg.slot_rt[c_cfg.reg_slot0[r] + b];
    const float4 q0 = q[0], q5 = q[5];
    const VoigtPoly vp = voigt_load(q[2], q[3], q[4], q5.x);
    const float kl = q0.x * dz;
    const float base = (wave - sc.bldiff + q5.w) * q5.y, bsc = B * q5.y;
    const float4* cm = c_cfg.comp + sc.comp0;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const float ut = fmaf(sc.type[t].x, bsc, base);
      const int n = sc.n[t];
      float h = 0.f, f = 0.f;
      // two components at a time: one wait for their constants and two
      // independent profiles
      int j = 0;
      for (; j + 2 <= n; j += 2, cm += 2) {
        const float4 ca = cm[0], cb = cm[1];
        float H, F, H2, F2;
        voigt(vp, fmaf(ca.x, bsc, ut), H, F);
        voigt(vp, fmaf(cb.x, bsc, ut), H2, F2);
        h = fmaf(cb.y, H2, fmaf(ca.y, H, h));
        f = fmaf(cb.y, F2, fmaf(ca.y, F, f));
      }
      if (j < n) {
        float H, F;
        voigt(vp, fmaf(cm->x, bsc, ut), H, F);
        h = fmaf(cm->y, H, h);
        f = fmaf(cm->y, F, f);
        ++cm;
      }
      X.h[t] = fmaf(kl, h, X.h[t]);
      X.f[t] = fmaf(kl, f, X.f[t]);
    }
  }
  return X;
}

// The same with the derivatives along T|Pg, v_z, |B| and, with PR, Pg|T and
// rho|T (absorption_matrix.f90:1717-2642).  With w = H + iF, dH/du = 2 (a F -
// u H) = dF/da and dH/da = 2 (a H + u F - 1/sqrt(pi)) = -dF/du, and the
// components of a type lie at u = ut + bsc delta: every derivative sum of
// the type is a combination of the moments sum st delta^n (H, F), n = 0, 1, 2,
// so a component costs its profile and six multiply-adds.
template <bool PR, class P>
__device__ __forceinline__ void absorb_der(P q, int r, float wave, float B, float dz, Sums& X, Sums& XT, Sums& XV,
                                           Sums& XB, Sums& XP, Sums& XR) {
  zero(X);
  zero(XT);
  zero(XV);
  zero(XB);
  if (PR) {
    zero(XP);
    zero(XR);
  }
  for (int b = 0; b < c_cfg.reg_nblend[r]; ++b, q += REC_SLOT / 4) {
    const Cfg::SlotRt sc = c_cfg.slot_rt[c_cfg.reg_slot0[r] + b];
    const float4 q0 = q[0], q5 = q[5];
    const VoigtPoly vp = voigt_load(q[2], q[3], q[4], q5.x);
    const float a = q0.y, kl = q0.x * dz, dklT = q0.z * dz;
    const float base = (wave - sc.bldiff + q5.w) * q5.y, bsc = B * q5.y;
    // kl times twice the derivatives of u in T (over u), v_z and |B| (over
    // the shift), and of a in T: the factor 2 of dH/du and dH/da
    const float uT = kl * q5.z, uv = 2.f * kl * sc.vfac * q5.y, ub = 2.f * kl * q5.y, aT = 2.f * kl * q0.w;
    float dklP = 0.f, dklR = 0.f, aP = 0.f, aR = 0.f;
    if (PR) {
      const float4 q1 = q[1];
      dklP = q1.x * dz;
      dklR = q1.y * dz;
      aP = 2.f * kl * q1.z;
      aR = 2.f * kl * q1.w;
    }
    const float4* cm = c_cfg.comp + sc.comp0;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const float4 ty = sc.type[t];
      const float ut = fmaf(ty.x, bsc, base);
      const int n = sc.n[t];
      // half dH/du and dH/da summed over the type, and times u and the shift
      float h0 = 0.f, f0 = 0.f, hu, ha, huu, hau, hb, hab;
      if (n == 1) {
        voigt(vp, ut, h0, f0);
        hu = fmaf(a, f0, -(ut * h0));
        ha = fmaf(a, h0, fmaf(ut, f0, -ty.y));
        huu = ut * hu;
        hau = ut * ha;
        hb = ty.x * hu;
        hab = ty.x * ha;
        ++cm;
      } else {
        float h1 = 0.f, f1 = 0.f, h2 = 0.f, f2 = 0.f;
        int j = 0;
        for (; j + 2 <= n; j += 2, cm += 2) {
          const float4 ca = cm[0], cb = cm[1];
          float H, F, H2, F2;
          voigt(vp, fmaf(ca.x, bsc, ut), H, F);
          voigt(vp, fmaf(cb.x, bsc, ut), H2, F2);
          h0 = fmaf(cb.y, H2, fmaf(ca.y, H, h0));
          f0 = fmaf(cb.y, F2, fmaf(ca.y, F, f0));
          h1 = fmaf(cb.z, H2, fmaf(ca.z, H, h1));
          f1 = fmaf(cb.z, F2, fmaf(ca.z, F, f1));
          h2 = fmaf(cb.w, H2, fmaf(ca.w, H, h2));
          f2 = fmaf(cb.w, F2, fmaf(ca.w, F, f2));
        }
        if (j < n) {
          const float4 ca = *cm++;
          float H, F;
          voigt(vp, fmaf(ca.x, bsc, ut), H, F);
          h0 = fmaf(ca.y, H, h0);
          f0 = fmaf(ca.y, F, f0);
          h1 = fmaf(ca.z, H, h1);
          f1 = fmaf(ca.z, F, f1);
          h2 = fmaf(ca.w, H, h2);
          f2 = fmaf(ca.w, F, f2);
        }
        hu = fmaf(a, f0, -fmaf(ut, h0, bsc * h1));
        ha = fmaf(a, h0, fmaf(ut, f0, fmaf(bsc, f1, -ty.y)));
        const float hd = fmaf(a, f1, -fmaf(ut, h1, bsc * h2));
        const float hc = fmaf(a, h1, fmaf(ut, f1, fmaf(bsc, f2, -ty.z)));
        huu = fmaf(ut, hu, bsc * hd);
        hau = fmaf(ut, ha, bsc * hc);
        hb = fmaf(ty.x, hu, hd);
        hab = fmaf(ty.x, ha, hc);
      }
      X.h[t] = fmaf(kl, h0, X.h[t]);
      X.f[t] = fmaf(kl, f0, X.f[t]);
      XT.h[t] = fmaf(dklT, h0, fmaf(uT, huu, fmaf(aT, ha, XT.h[t])));
      XT.f[t] = fmaf(dklT, f0, fmaf(-uT, hau, fmaf(aT, hu, XT.f[t])));
      XV.h[t] = fmaf(uv, hu, XV.h[t]);
      XV.f[t] = fmaf(-uv, ha, XV.f[t]);
      XB.h[t] = fmaf(ub, hb, XB.h[t]);
      XB.f[t] = fmaf(-ub, hab, XB.f[t]);
      if (PR) {
        XP.h[t] = fmaf(dklP, h0, fmaf(aP, ha, XP.h[t]));
        XP.f[t] = fmaf(dklP, f0, fmaf(aP, hu, XP.f[t]));
        XR.h[t] = fmaf(dklR, h0, fmaf(aR, ha, XR.h[t]));
        XR.f[t] = fmaf(dklR, f0, fmaf(aR, hu, XR.f[t]));
      }
    }
  }
}

// LINE OPTICAL DEPTH (forward.f90:966-968, 1008-1015): per (column,
// wavelength) KLINTAU_k = ETAI_k / N_H / m_u / MW_k from the propagation
// matrix of every height whose opacities are formed (0 where the height is
// opaque; the reference keeps the last computed ETAI there), then the REAL(4)
// trapezoid from the top (tau = 1e-9) down, and log10.
// out[((col * nz + k) * numw + l]; one lane per (column, wavelength).
__global__ void __launch_bounds__(256) taulin_kernel(RtArgs a, float* __restrict__ out) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int numw = c_cfg.numw, nz = c_cfg.nz;
  if (g >= (long)a.ntile * numw) return;
  const int ct = (int)(g / numw), l = (int)(g - (long)ct * numw), col = a.col0 + ct;
  if (a.status && a.status[col] != 0) return;
  int r = 0;
  while (r + 1 < c_cfg.nreg && l >= c_cfg.reg_pix0[r + 1]) ++r;
  const float wave = (float)(c_cfg.reg_wstart[r] + c_cfg.reg_wstep[r] * (double)(l - c_cfg.reg_pix0[r]));
  const long ps = (long)nz * a.ncol, cs = a.ncol;
  float* o = out + (long)col * nz * numw + l;
  for (int k = 0; k < nz; ++k) {
    const float4* R = reinterpret_cast<const float4*>(a.micro + ((long)k * a.rncol + col - a.rcol0) * c_cfg.rec);
    const float fac = R[3].w;
    float kl = 0.f;
    if (fac != 0.f) {
      const float4* Q = R + c_cfg.reg_rec[r] / 4;
      const float4 h1 = R[1];
      const Sums X = absorb(Q + 1, r, wave, h1.y, 1.0f);
      kl = (Q[0].x + fmaf(h1.z, X.h[1], h1.w * (X.h[0] + X.h[2]))) * fac;
    }
    o[(long)k * numw] = kl;
  }
  float tau = 1.0e-9f, kln = o[(long)(nz - 1) * numw];
  o[(long)(nz - 1) * numw] = log10f(tau);
  for (int k = nz - 2; k >= 0; --k) {
    const float klk = o[(long)k * numw];
    const float x = (klk * a.atm[A_RHO * ps + k * cs + col] + kln * a.atm[A_RHO * ps + (k + 1) * cs + col]) / 2.0f;
    tau = (float)((double)tau + (double)x * ((c_cfg.zz[k + 1] - c_cfg.zz[k]) * 1000.0 * 100.0));
    o[(long)k * numw] = log10f(tau);
    kln = klk;
  }
}

// a value that is the same in all lanes, in a scalar register
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long uniform(int64_t x) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)x);
  return ((long)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32) | lo;
}

// flags of a raw 32-bit buffer resource
constexpr int RSRC_FLAGS = 0x00027000;

// Node contraction within the transfer (CALCULATE_EQUIVALENT_DSYN,
// forward.f90:552-681) for the five slots of RF_CART_TBV: per height and slot
// the lowest node that still takes heights (free parameter index) and the
// weights of that node and the next (the hat functions overlap pairwise);
// node -1: the slot is not inverted
struct NodeTab {
  double c0, c1;
  int node, pad;
};
struct NodeArgs {
  float* eqv;          // [ncol][np][nstk * numw], ragged with windows
  int np, nstk;
  int blk[4];          // block of each Stokes parameter among the inverted ones, -1: not inverted
  int last[5];         // last node of each slot
};

// bytes of LDS that a transfer wave fills with the records of its next heights
constexpr size_t RT_LDS = 10 * 1024;

// Radiative transfer, one lane per (column, wavelength), one wave per
// workgroup.  Bound: the issue of FP32 operations (no packed FP32 in this
// build), about 600 per height in pass 1 and 1400 in pass 2 for two lines with
// 15 Zeeman components and five parameters.
//
// HE (HYDROSTATIC: yes, response functions on): the T response of height K
// also carries the change of Pg below K through hydrostatic equilibrium,
// dPg_i/dT_K = Pg_i (-mu_K m_u g dz_K / (k T_K^2)) (GET_HYD_DERIVATIVES), i.e.
// g_K * W_K with W_K = sum_{i<K} O_K..O_{i+1} (local Pg|T response of i) Pg_i,
// skipping layers with O_11 <= 1e-5 (rtesolver.f90:218-231).  W is built in
// pass 1 with one extra directional derivative per layer, so the term costs
// O(nz) instead of the reference's O(nz^2).  In that mode the reference
// evaluates the rho, B and v responses with the layer's outgoing Stokes
// vector (STKIN is reset to SYN1D after the hydrostatic block); reproduced.
//
// PACK (no per-pixel windows): the lanes of a launch run over the flattened
// (column, wavelength) pairs of the tile in one region after the other, 64 to a
// wave, so no lane idles when a region's wavelength count is not a multiple of
// 64 (112 = 64 + 48 would leave 16 of 128 lanes idle per column); a wave then
// spans two or more columns, each lane reading its own column's record from
// LDS.  437 columns x 81 heights in three regions of 77 wavelengths, seven
// responses with hydrostatic equilibrium: 1.46 ms with a column per wave, 0.94 packed.
//
// NW (packed launches of few waves): a team of NW waves has the wave's 64
// lanes' layers in turn, NW at a time.  Absorption, evolution operator and local responses,
// nine tenths of the work, do not depend on the neighbouring layers; the step
// of the Stokes vector (pass 1) and of the running product (pass 2) go from wave to
// wave through LDS.  The same operations on the same values: the same bits.
// One column of 64 heights and 112 wavelengths: synthesis 0.32 -> 0.22 ms with its
// microphysics, with five responses 0.61 -> 0.34 ms (where the line lies: launch_rt).
//
// NODES (RF_CART_TBV): the responses are contracted with the node basis as
// they are formed instead of going to memory per height.  Going down, a slot
// feeds the FP64 sums of two nodes; where the lower one's support ends the
// upper node is complete and stored.  The registers of the sums leave two
// waves per SIMD instead of three, which the issue-bound transfer bears:
// forward and contraction of 128x128x64 columns 10.2 -> 7.9 ms against
// responses stored per height (9.4 GB) and read again by eqv_kernel.
template <int RF, bool HE, bool PACK, bool NODES = false, int NW = 1>
__global__ void __launch_bounds__(RT_WAVE * NW) rt_kernel(RtArgs a, NodeArgs nd, const NodeTab* __restrict__ ntab) {
#pragma clang fp contract(off)
  // parameters: 5 spherical, 7 Cartesian, 8 with P0 (the top pressure)
  constexpr int NP = (RF == FZ_RF_SPHERICAL || RF == RF_CART_TBV)
                         ? 5
                         : (RF == FZ_RF_CARTESIAN ? 7 : (RF == FZ_RF_CARTESIAN_P0 ? 8 : 0));
  constexpr int NPL = RF == FZ_RF_CARTESIAN_P0 ? 7 : NP;    // parameters with a local response
  constexpr bool PR = RF == FZ_RF_CARTESIAN || RF == FZ_RF_CARTESIAN_P0;
  constexpr bool HEX = HE && RF != 0;
  extern __shared__ float4 lds[];
  // a team's running Stokes vector (and Ahe) and its running product
  __shared__ float xi[NW > 1 ? 8 : 1][RT_WAVE], xa[NW > 1 && RF != 0 ? 16 : 1][RT_WAVE];
  __shared__ float xo[NW > 1 && NODES ? NW : 1][20][RT_WAVE];   // responses of a team's layers
  const int numw = c_cfg.numw, nz = c_cfg.nz, lane = (int)threadIdx.x & (RT_WAVE - 1);
  const int wv = NW > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  // workgroup -> (column, region, first wavelength); lane -> wavelength.  A
  // lane past the work repeats the last one without storing, so that the
  // whole wave takes part in the copies to LDS.
  bool live = true;
  int ct, ct0, r, l;
  long sbase;        // the column's Stokes: stokes[sbase + s * snumw + lo]
  int snumw, lo;
  // scratch rows of nthr lanes and response functions: the wave's first
  // element (t0, j0, wave-uniform) and the lane's distance from it, so that
  // the accesses take a scalar base and a 32-bit offset
  long t0, nthr, j0;
  unsigned dt, dj;   // jac[j0 + dj + ((p*nz + k)*4 + s)*snumw]
  if constexpr (PACK) {
    int b = (int)blockIdx.x;
    for (r = 0; r + 1 < c_cfg.nreg; ++r) {
      const int nw = (a.ntile * c_cfg.reg_nwave[r] + RT_WAVE - 1) / RT_WAVE;
      if (b < nw) break;
      b -= nw;
    }
    const int n = c_cfg.reg_nwave[r], p0 = c_cfg.reg_pix0[r];
    const int g0 = b * RT_WAVE, last = a.ntile * n - 1;
    live = g0 + lane <= last;
    const int g = min(g0 + lane, last);
    ct = g / n;
    ct0 = uniform(g0 / n);
    l = p0 + g - ct * n;
    sbase = (long)(a.col0 + ct) * 4 * numw;
    snumw = numw;
    lo = l;
    t0 = (long)a.ntile * p0 + g0;
    dt = (unsigned)(g - g0);
    nthr = (long)a.ntile * numw;
    j0 = (long)(a.col0 + ct0 - a.jcol0) * NP * nz * 4 * numw;
    dj = (unsigned)((ct - ct0) * NP * nz * 4 * numw + l);
  } else if (a.items) {
    // per-pixel windows: scratch and response functions are ragged too
    const RtItem it = a.items[blockIdx.x];
    const int icol = uniform(it.col), lout = uniform(it.lout);
    live = lane < it.n;
    const int i = min(lane, it.n - 1);
    ct = ct0 = icol - a.col0;
    r = uniform(it.r);
    l = it.l0 + i;
    const long p0 = uniform(a.poff[icol]), pt = uniform(a.poff[a.col0]);
    sbase = 4 * p0;
    snumw = (int)(uniform(a.poff[icol + 1]) - p0);
    lo = lout + i;
    t0 = (p0 - pt) + lout;
    dt = dj = (unsigned)i;
    nthr = uniform(a.poff[a.col0 + a.ntile]) - pt;
    j0 = (long)NP * nz * 4 * (p0 - uniform(a.poff[a.jcol0])) + lout;
  } else {
    ct = ct0 = uniform((int)(blockIdx.x / (unsigned)c_cfg.nbpc));
    const int bc = (int)(blockIdx.x - (unsigned)ct * (unsigned)c_cfg.nbpc);
    live = lane < c_cfg.blk_n[bc];
    r = c_cfg.blk_reg[bc];
    l = c_cfg.blk_l0[bc] + min(lane, c_cfg.blk_n[bc] - 1);
    sbase = (long)(a.col0 + ct) * 4 * numw;
    snumw = numw;
    lo = l;
    t0 = (long)ct * numw + c_cfg.blk_l0[bc];
    dt = dj = (unsigned)min(lane, c_cfg.blk_n[bc] - 1);
    nthr = (long)a.ntile * numw;
    j0 = (long)(a.col0 + ct - a.jcol0) * NP * nz * 4 * numw + c_cfg.blk_l0[bc];
  }
  const int col = a.col0 + ct;
  // the column's node responses: [np][nstk][snumw] from here
  float* eqv = nullptr;
  if constexpr (NODES)
    eqv = nd.eqv + (a.items ? (long)nd.np * nd.nstk * (sbase / 4) : (long)col * nd.np * nd.nstk * snumw) + lo;
  // Another workgroup of the column may set its status during this launch (below):
  // a team takes its first wave's reading, so that its waves agree on what they do.
  bool failed;
  if constexpr (NW > 1) {
    __shared__ unsigned long long bad;
    if (wv == 0) {
      const unsigned long long m = __ballot(a.status && a.status[col] != 0);
      if (lane == 0) bad = m;
    }
    __syncthreads();
    failed = (bad >> lane) & 1;
  } else {
    failed = a.status && a.status[col] != 0;
  }
  if (failed) {
    if (live && wv == 0) {
      for (int s = 0; s < 4; ++s) a.stokes[sbase + (long)s * snumw + lo] = __builtin_nanf("");
      if constexpr (NODES)
        for (int i = 0; i < nd.np * nd.nstk; ++i) eqv[(long)i * snumw] = 0.f;
    }
    live = false;
  }
  if (__ballot(live) == 0) return;
  // the wave's columns are ct0 .. ct0 + nc - 1
  const int nc = PACK ? uniform(__shfl(ct, 63) - ct0 + 1) : 1;
  const int rs4 = (REC_HEAD + REC_REG + REC_SLOT * c_cfg.reg_nblend[r]) / 4;   // float4 per (height, column) in LDS
  const float4* grec = reinterpret_cast<const float4*>(a.micro);
  const int rc0 = a.col0 + ct0 - a.rcol0;
  const int rec4 = c_cfg.rec / 4, roff4 = (c_cfg.reg_rec[r] - REC_HEAD) / 4;
  // heights k0 .. k0 + n - 1 of the wave's columns into LDS: half a wave per
  // record (rs4 <= 32)
  auto stage = [&](int k0, int n) {
    __syncthreads();
    const int f = lane & 31;
    const int src = f + (f >= REC_HEAD / 4 ? roff4 : 0);
    const int np = n * nc;
    int h = 0, c = 2 * wv + (lane >> 5);
    while (c >= nc) {
      c -= nc;
      ++h;
    }
    for (int p = 2 * wv + (lane >> 5); p < np; p += 2 * NW) {
      if (f < rs4) lds[p * rs4 + f] = grec[((long)(k0 + h) * a.rncol + rc0 + c) * rec4 + src];
      c += 2 * NW;
      while (c >= nc) {
        c -= nc;
        ++h;
      }
    }
    __syncthreads();
  };
  const float4* const mine = lds + (ct - ct0) * rs4;
  const double wd = c_cfg.reg_wstart[r] + c_cfg.reg_wstep[r] * (double)(l - c_cfg.reg_pix0[r]);
  const float wave = (float)wd;
  // Planck function constants (rtesolver.f90:1008-1035): S = c1 / (exp(c2/T) - 1)
  const double lam = (c_cfg.reg_l0main[r] + wd / 1.0e3) * 1.0e-8;
  const float c1 = (float)(2.0 * HPLA * LIGHT * LIGHT / (lam * lam * lam * lam * lam));
  const float c2 = (float)(HPLA * LIGHT / (lam * KBOL));
  const long ps = (long)nz * a.ncol, cs = a.ncol;
  float I[4] = {0.f, 0.f, 0.f, 0.f};
  float Ahe[4] = {0.f, 0.f, 0.f, 0.f};
  // row i of the pass-1 scratch and of the response functions
  // rows of the pass-1 scratch (64 lanes from t0) and of the wave's response
  // functions as buffers: the row is a scalar offset, the lane a 32-bit one
  const unsigned dtb = 4u * dt, djb = 4u * dj;
  auto scr = [&](int i) -> __amdgpu_buffer_rsrc_t {
    return __builtin_amdgcn_make_buffer_rsrc(a.scratch + t0 + (long)i * nthr, 0, 4 * RT_WAVE, RSRC_FLAGS);
  };
  auto scr_store = [&](int i, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), scr(i), dtb, 0, 0);
  };
  auto scr_load = [&](int i) -> float {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(scr(i), dtb, 0, 0));
  };
  const __amdgpu_buffer_rsrc_t jbuf = __builtin_amdgcn_make_buffer_rsrc(
      RF && !NODES ? a.jac + j0 : nullptr, 0, 4 * nc * NP * nz * 4 * snumw, RSRC_FLAGS);
  auto jac_store = [&](int i, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), jbuf, djb, 4 * i * snumw, 0);
  };
  // POPL/POPU of the wavelength's region at height k (SOURCE_FUNCTION,
  // rtesolver.f90:1030-1033): S = c1 / ((POPL/POPU) exp(c2/T) - 1)
  auto depart = [&](int k) -> float {
    return a.pop ? (float)(a.pop[(long)k * c_cfg.nreg + r] / a.pop[((long)nz + k) * c_cfg.nreg + r]) : 1.0f;
  };
  // FULL_STOKES (forward.f90:980-983): the Stokes vector after every
  // height, times GAIN1D, at fs[((col * nz + k) * 4 + s) * numw + l]
  float* fsp = a.fs && live ? a.fs + (long)col * nz * 4 * snumw + lo : nullptr;
  auto store_fs = [&](int k) {
    if (!fsp) return;
#pragma unroll
    for (int s = 0; s < 4; ++s) fsp[(long)(k * 4 + s) * snumw] = I[s] * a.gain[l * 4 + s];
  };
  // into the layer's frame (cos, sin of twice the azimuth) and back
  auto turn = [](float c, float s, const float v[4], float o[4]) {
    o[0] = v[0];
    o[1] = fmaf(c, v[1], s * v[2]);
    o[2] = fmaf(c, v[2], -(s * v[1]));
    o[3] = v[3];
  };
  auto turn_back = [](float c, float s, float v[4]) {
    const float q = fmaf(c, v[1], -(s * v[2])), u = fmaf(s, v[1], c * v[2]);
    v[1] = q;
    v[2] = u;
  };
  // Pass 1, bottom to top.  What of a layer does not depend on the light
  // (form) and the step through it (pass).
  struct Layer {
    Evol E;
    Five fp;
    float S;
  };
  auto form = [&](int k, const float4* R, Layer& Y) {
    const float4 h1 = R[1], h2 = R[2], rg = R[REC_HEAD / 4];
    const float dz = c_cfg.dz_cm[k];
    const Mix mx = {h1.z, h1.w, h2.x, h2.y, h2.z};
    Five f;
    if constexpr (HEX) {
      Sums X, XT, XV, XB, XP, XR;
      absorb_der<true>(R + REC_HEAD / 4 + 1, r, wave, h1.y, dz, X, XT, XV, XB, XP, XR);
      f = mix(mx, X);
      Y.fp = mix(mx, XP);
      Y.fp.I = fmaf(rg.z, dz, Y.fp.I);
    } else {
      f = mix(mx, absorb(R + REC_HEAD / 4 + 1, r, wave, h1.y, dz));
    }
    f.I = fmaf(rg.x, dz, f.I);
    evol_build<HEX>(f, Y.E);
  };
  auto pass = [&](int k, const float4& h3, const Layer& Y) {
    const Evol& E = Y.E;
    const float v[4] = {I[0] - Y.S, I[1], I[2], I[3]};
    float vf[4], dv[4];
    turn(h3.x, h3.y, v, vf);
    const Pieces w = evol_pieces(E, vf);
    evol_apply(E, w, dv);
    if constexpr (HEX) {
      Grad G;
      evol_grad(E, vf, w, G);
      float d2[4], Af[4], W[4];
      grad_dot(G, Y.fp, d2);
      turn_back(h3.x, h3.y, d2);
      turn(h3.x, h3.y, Ahe, Af);
      evol_apply(E, evol_pieces(E, Af), W);
      turn_back(h3.x, h3.y, W);
      const bool thin = fmaf(E.D4, E.s0, E.A) > 1.0e-5f;    // O_11
      const float pg = a.atm[A_PG * ps + k * cs + col];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        W[i] = thin ? fmaf(E.A, Ahe[i], W[i]) : Ahe[i];
        if (live) scr_store((nz + k) * 4 + i, W[i]);
        if (thin) Ahe[i] = fmaf(d2[i], pg, W[i]);
      }
    }
    turn_back(h3.x, h3.y, dv);
#pragma unroll
    for (int i = 0; i < 4; ++i) I[i] = fmaf(E.A, v[i], dv[i]) + (i == 0 ? Y.S : 0.f);
  };
  auto keep = [&](int k) {
    if (RF && live) {
#pragma unroll
      for (int s = 0; s < 4; ++s) scr_store(k * 4 + s, I[s]);
    }
  };
  if constexpr (NW > 1) {
    if (wv == 0)
#pragma unroll
      for (int i = 0; i < 8; ++i) xi[i][lane] = 0.f;
  }
  for (int k0 = 0; k0 < nz; k0 += a.chunk) {
    const int n = min(a.chunk, nz - k0);
    stage(k0, n);
    for (int kb = 0; kb < n; kb += NW) {
      const int kk = kb + wv, k = k0 + kk;
      const bool has = NW == 1 || kk < n;
      const float4* R = mine + (has ? kk : 0) * nc * rs4;
      const float4 h0 = R[0], h3 = R[3];
      Layer Y;
      Y.S = c1 * (1.0f / (depart(has ? k : 0) * expf(c2 * h0.z) - 1.0f));
      if constexpr (NW == 1) {
        keep(k);
        if (h0.x != 0.f) {
          I[0] = Y.S; I[1] = 0.f; I[2] = 0.f; I[3] = 0.f;
        } else {
          form(k, R, Y);
          pass(k, h3, Y);
        }
        store_fs(k);
      } else {
        if (has && h0.x == 0.f) form(k, R, Y);
#pragma unroll 1
        for (int i = 0; i < NW; ++i) {
          if (i == wv && has) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              I[s] = xi[s][lane];
              if (HEX) Ahe[s] = xi[4 + s][lane];
            }
            keep(k);
            if (h0.x != 0.f) {
              I[0] = Y.S; I[1] = 0.f; I[2] = 0.f; I[3] = 0.f;
            } else {
              pass(k, h3, Y);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              xi[s][lane] = I[s];
              if (HEX) xi[4 + s][lane] = Ahe[s];
            }
            store_fs(k);
          }
          __syncthreads();
        }
      }
    }
  }
  if constexpr (NW > 1) {
#pragma unroll
    for (int s = 0; s < 4; ++s) I[s] = xi[s][lane];
  }
  float gn[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    gn[s] = a.gain[l * 4 + s];
    if (live && wv == 0) a.stokes[sbase + (long)s * snumw + lo] = I[s] * gn[s];
  }
  // a non-finite Stokes vector comes from a non-finite profile, propagation
  // matrix or evolution operator, where the reference stops
  // (voigt.f:91-95, absorption_matrix.f90:1882-1889, rtesolver.f90:346-352)
  if (live && wv == 0 && a.status && !(__builtin_isfinite(I[0]) && __builtin_isfinite(I[1]) && __builtin_isfinite(I[2]) &&
                            __builtin_isfinite(I[3])))
    atomicMax(&a.status[col], (int32_t)ERR_NAN);
  if constexpr (RF != 0) {
    // O_nz ... O_{k+1}, its rows times GAIN1D (but for P0, whose response is
    // a product of two propagated ones)
    constexpr bool GACC = RF != FZ_RF_CARTESIAN_P0;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = (i == j) ? (GACC ? gn[i] : 1.f) : 0.f;
    // sums of nodes jl, jl + 1 of a slot (a team's wave keeps those of one Stokes
    // parameter, with eight waves of some slots)
    constexpr int NST = NW > 1 ? 1 : 4;
    double nlo[NODES ? 5 : 1][NST], nhi[NODES ? 5 : 1][NST];
    int jl[5];
    const int st0 = NW > 1 ? wv & 3 : 0;
    auto owned = [&](int p) { return NW <= 4 || (p < 3) == (wv < 4); };
    auto store_node = [&](int p, int j, const double (&x)[NST]) {
      if (!live || j > nd.last[p]) return;
#pragma unroll
      for (int i = 0; i < NST; ++i)
        if (nd.blk[st0 + i] >= 0) eqv[((long)j * nd.nstk + nd.blk[st0 + i]) * snumw] = (float)x[i];
    };
    // a slot's nodes whose support ends above height k are complete
    auto next_node = [&](int p, int k) {
      const int w = ntab[k * 5 + p].node;
      while (w >= 0 && jl[p] > w) {
        store_node(p, jl[p] + 1, nhi[p]);
#pragma unroll
        for (int i = 0; i < NST; ++i) {
          nhi[p][i] = nlo[p][i];
          nlo[p][i] = 0.0;
        }
        --jl[p];
      }
    };
    if constexpr (NODES) {
#pragma unroll
      for (int p = 0; p < 5; ++p) {
        jl[p] = nd.last[p];
#pragma unroll
        for (int i = 0; i < NST; ++i) nlo[p][i] = nhi[p][i] = 0.0;
      }
    }
    // Pass 2, top to bottom.  A layer's local responses in the frame (local: lp[0] =
    // T, then (Pg, rho,) and the field's), the running product (extend) with the row
    // vectors b of acc in the frame, and the propagated responses (emit).
    auto local = [&](int k, const float4* R, const float4& h0, Evol& E, float (&lp)[NPL][4]) {
                const float4 h1 = R[1], h2 = R[2], h3 = R[3], rg = R[REC_HEAD / 4];
                const float dz = c_cfg.dz_cm[k];
                // S = c1 / (ex - 1), dS/dT = S (ex / (ex - 1)) (c2 / T) / T
                const float x = c2 * h0.z;
                const float ex = depart(k) * expf(x);
                const float iem1 = 1.0f / (ex - 1.0f);
                const float S = c1 * iem1;
                const float dS = S * (ex * iem1) * x * h0.z;
                const Mix mx = {h1.z, h1.w, h2.x, h2.y, h2.z};
                Sums X, XT, XV, XB, XP, XR;
                absorb_der<PR>(R + REC_HEAD / 4 + 1, r, wave, h1.y, dz, X, XT, XV, XB, XP, XR);
                Five f = mix(mx, X);
                f.I = fmaf(rg.x, dz, f.I);
                evol_build<true>(f, E);
                float v[4], vf[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) v[s] = scr_load(k * 4 + s) - (s == 0 ? S : 0.f);
                turn(h3.x, h3.y, v, vf);
                // local responses in the frame: lp[0] = T, then (Pg, rho,) and the field's
                float lB[4], lG[4], lF[4];
                constexpr int o = PR ? 2 : 0;
                {
                  const Pieces w = evol_pieces(E, vf);
                  Grad G;
                  evol_grad(E, vf, w, G);
                  Five fd = mix(mx, XT);
                  fd.I = fmaf(rg.y, dz, fd.I);
                  grad_dot(G, fd, lp[0]);
                  if constexpr (PR) {
                    fd = mix(mx, XP);
                    fd.I = fmaf(rg.z, dz, fd.I);
                    grad_dot(G, fd, lp[1]);
                  }
                  if constexpr (HEX) {
                    float vo[4], vof[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                      vo[s] = (k == nz - 1 ? I[s] : scr_load((k + 1) * 4 + s)) - (s == 0 ? S : 0.f);
                    turn(h3.x, h3.y, vo, vof);
                    const Pieces wo = evol_pieces(E, vof);
                    evol_grad(E, vof, wo, G);
                    evol_azimuth(E, vof, wo, lF);
                  } else {
                    evol_azimuth(E, vf, w, lF);
                  }
                  if constexpr (PR) {
                    fd = mix(mx, XR);
                    fd.I = fmaf(rg.w, dz, fd.I);
                    grad_dot(G, fd, lp[2]);
                  }
                  grad_dot(G, mix(mx, XB), lB);
                  grad_dot(G, mix(mx, XV), lp[4 + o]);
                  // the inclination: I and q share their factor, d sin^2 = 2 sg cg
                  const Mix mg = {h3.z, -0.5f * h3.z, h3.z, 0.5f * h3.z, -0.5f * h2.w};
                  grad_dot(G, mix(mg, X), lG);
                }
                // source-function term (1 - O) e0 dS/dT for T; O e0 in the frame
                {
                  const float alx = -fmaf(E.ga, E.ex, E.gb * E.rx), alz = -fmaf(E.ga, E.ez, E.gb * E.rz);
                  lp[0][0] = fmaf(1.f - fmaf(E.D4, E.s0, E.A), dS, lp[0][0]);
                  lp[0][1] = fmaf(-alx, dS, lp[0][1]);
                  lp[0][2] = fmaf(E.D4 * E.cy, dS, lp[0][2]);
                  lp[0][3] = fmaf(-alz, dS, lp[0][3]);
                }
                if constexpr (HEX) {
                  const float mu = a.atm[A_MU * ps + k * cs + col];
                  const float gk = -mu * c_cfg.he_cte[k] * h0.z * h0.z;
                  float W[4], Wf[4];
#pragma unroll
                  for (int i = 0; i < 4; ++i) W[i] = scr_load((nz + k) * 4 + i);
                  turn(h3.x, h3.y, W, Wf);
#pragma unroll
                  for (int i = 0; i < 4; ++i) lp[0][i] = fmaf(gk, Wf[i], lp[0][i]);
                }
                if constexpr (RF == FZ_RF_SPHERICAL) {
#pragma unroll
                  for (int i = 0; i < 4; ++i) {
                    lp[1][i] = lB[i];
                    lp[2][i] = lG[i];
                    lp[3][i] = lF[i];
                  }
                } else {
                  // chain rule (|B|, gamma, phi) -> (Bx, By, Bz)
                  const float4 h4 = R[4], h5 = R[5];
#pragma unroll
                  for (int i = 0; i < 4; ++i) {
                    lp[1 + o][i] = fmaf(h4.x, lB[i], fmaf(h4.w, lG[i], h5.z * lF[i]));
                    lp[2 + o][i] = fmaf(h4.y, lB[i], fmaf(h5.x, lG[i], h5.w * lF[i]));
                    lp[3 + o][i] = fmaf(h4.z, lB[i], h5.y * lG[i]);
                  }
                }
    };
    // the running product O_nz ... O_k = acc (A 1 + turned-back (O - A 1))
    auto extend = [&](const float4& h3, const Evol& E, float (&b)[4][4]) {
      const float M11 = E.D4 * (fmaf(E.ex, E.ex, E.rx * E.rx) - E.s0), M33 = E.D4 * (fmaf(E.ez, E.ez, E.rz * E.rz) - E.s0);
      const float M00 = E.D4 * E.s0, M02 = E.D4 * E.cy, M13 = E.D4 * fmaf(E.ex, E.ez, E.rx * E.rz);
      const float M01 = -fmaf(E.ga, E.ex, E.gb * E.rx), M03 = -fmaf(E.ga, E.ez, E.gb * E.rz);
      const float M12 = fmaf(E.ga, E.rz, -(E.gb * E.ez)), M23 = fmaf(E.ga, E.rx, -(E.gb * E.ex));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        turn(h3.x, h3.y, acc[i], b[i]);
        float m[4];
        m[0] = fmaf(b[i][0], M00, fmaf(b[i][1], M01, fmaf(-b[i][2], M02, b[i][3] * M03)));
        m[1] = fmaf(b[i][0], M01, fmaf(b[i][1], M11, fmaf(-b[i][2], M12, b[i][3] * M13)));
        m[2] = fmaf(b[i][0], M02, fmaf(b[i][1], M12, fmaf(-b[i][2], M00, -(b[i][3] * M23))));
        m[3] = fmaf(b[i][0], M03, fmaf(b[i][1], M13, fmaf(b[i][2], M23, b[i][3] * M33)));
        turn_back(h3.x, h3.y, m);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(E.A, acc[i][j], m[j]);
      }
    };
    // above[i]: sum of row i of acc above the layer (for P0)
    auto emit = [&](int k, const float (&lp)[NPL][4], const float (&b)[4][4], const float (&above)[4]) {
      float outv[NP][4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < NPL; ++p)
          outv[p][i] = fmaf(b[i][0], lp[p][0], fmaf(b[i][1], lp[p][1], fmaf(b[i][2], lp[p][2], b[i][3] * lp[p][3])));
      if constexpr (RF == FZ_RF_CARTESIAN_P0) {
        // P0 (forward.f90:543-545): the local response is 1 in every Stokes
        // parameter; below the top it is propagated and then multiplied,
        // component by component, by PG(K)/PG(NZ) and the propagated Pg|T
        // response of the same height; the top layer keeps 1
        if (k == nz - 1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) outv[7][i] = 1.f;
        } else {
          const float ratio = a.atm[A_PG * ps + k * cs + col] / a.atm[A_PG * ps + (nz - 1) * cs + col];
#pragma unroll
          for (int i = 0; i < 4; ++i) outv[7][i] = above[i] * ratio * outv[1][i];
        }
      }
      if constexpr (NODES && NW > 1) {
#pragma unroll
        for (int p = 0; p < 5; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) xo[wv][p * 4 + i][lane] = outv[p][i];
      } else if constexpr (NODES) {
#pragma unroll
        for (int p = 0; p < 5; ++p) {
          const double c0 = ntab[k * 5 + p].c0, c1 = ntab[k * 5 + p].c1;
#pragma unroll
          for (int i = 0; i < NST; ++i) {
            const double x = (double)outv[p][i];
            nlo[p][i] = fma(x, c0, nlo[p][i]);
            nhi[p][i] = fma(x, c1, nhi[p][i]);
          }
        }
      } else if (live) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int s = 0; s < 4; ++s) jac_store((p * nz + k) * 4 + s, GACC ? outv[p][s] : outv[p][s] * gn[s]);
      }
    };
    auto row_sums = [&](float (&above)[4]) {
      if constexpr (RF == FZ_RF_CARTESIAN_P0)
#pragma unroll
        for (int i = 0; i < 4; ++i) above[i] = acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
    };
    // boundary layer: no local response; layers below cannot reach the top
    auto blank = [&](int k) {
      if constexpr (NODES && NW > 1) {
#pragma unroll
        for (int i = 0; i < 20; ++i) xo[wv][i][lane] = 0.f;
      }
      if (!NODES && live)
#pragma unroll 1
        for (int i = 0; i < 4 * NP; ++i) jac_store(((i >> 2) * nz + k) * 4 + (i & 3), 0.f);
    };
    if constexpr (NW > 1) {
      if (wv == 0)
#pragma unroll
        for (int i = 0; i < 16; ++i) xa[i][lane] = acc[i >> 2][i & 3];
    }
    for (int k0 = (nz - 1) / a.chunk * a.chunk; k0 >= 0; k0 -= a.chunk) {
      const int n = min(a.chunk, nz - k0);
      stage(k0, n);
      for (int kb = (n - 1) / NW * NW; kb >= 0; kb -= NW) {
        const int kk = kb + wv, k = k0 + kk;
        const bool has = NW == 1 || kk < n;
        const float4* R = mine + (has ? kk : 0) * nc * rs4;
        const float4 h0 = R[0];
        if constexpr (NODES && NW == 1) {
#pragma unroll
          for (int p = 0; p < 5; ++p) next_node(p, k);
        }
        Evol E;
        float lp[NPL][4], b[4][4], above[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (NW == 1) {
          if (h0.x != 0.f) {
            blank(k);
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i >> 2][i & 3] = 0.f;
          } else {
            local(k, R, h0, E, lp);
            row_sums(above);
            extend(R[3], E, b);
            emit(k, lp, b, above);
          }
        } else {
          const float4 h3 = R[3];
          if (has && h0.x == 0.f) local(k, R, h0, E, lp);
#pragma unroll 1
          for (int i = NW - 1; i >= 0; --i) {
            if (i == wv && has) {
#pragma unroll
              for (int j = 0; j < 16; ++j) acc[j >> 2][j & 3] = xa[j][lane];
              row_sums(above);
              if (h0.x != 0.f) {
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[j >> 2][j & 3] = 0.f;
              } else {
                extend(h3, E, b);
              }
#pragma unroll
              for (int j = 0; j < 16; ++j) xa[j][lane] = acc[j >> 2][j & 3];
            }
            __syncthreads();
          }
          if (has) {
            if (h0.x != 0.f)
              blank(k);
            else
              emit(k, lp, b, above);
          }
          if constexpr (NODES) {
            __syncthreads();
#pragma unroll 1
            for (int q = min(NW, n - kb) - 1; q >= 0; --q) {
              const int kq = k0 + kb + q;
#pragma unroll
              for (int p = 0; p < 5; ++p) {
                if (!owned(p)) continue;
                next_node(p, kq);
                const double x = (double)xo[q][p * 4 + st0][lane];
                nlo[p][0] = fma(x, ntab[kq * 5 + p].c0, nlo[p][0]);
                nhi[p][0] = fma(x, ntab[kq * 5 + p].c1, nhi[p][0]);
              }
            }
          }
        }
      }
    }
    if constexpr (NODES) {
#pragma unroll
      for (int p = 0; p < 5; ++p) {
        if (nd.last[p] < 0 || !owned(p)) continue;
        store_node(p, jl[p] + 1, nhi[p]);
        store_node(p, jl[p], nlo[p]);
      }
    }
  }
}

// ---------------------------------------------------------------- HSRA normalisation
// Equation of state and continuum opacity along the embedded HSRA model
// (normalization.f90:696-754); one thread, heights in order (warm start).
// HSRA's continuum opacities at the regions' central wavelengths
// (normalization.f90:696-754): the EOS of every HSRA height warm-started
// from the height below, as GET_RHO runs it there.  The Saha factors of all
// heights and elements are independent (one thread each), the fixed point is
// sequential in height (the 64 lanes of one wave), and the
// opacities are independent again (one thread per height and region).
__global__ void __launch_bounds__(256) hsra_saha_kernel(double* __restrict__ sb /*[387][92][4]*/) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= FZ_HSRA_LEN * FZ_NELEM) return;
  const int k = t / FZ_NELEM, i = t - k * FZ_NELEM;
  const SahaT s((double)fz_hsra_t[k]);
  double a1, a2, da1, da2;
  saha_element<false>(i, s, a1, a2, da1, da2);
  double* o = sb + ((long)k * FZ_NELEM + i) * 4;
  o[0] = a1;
  o[1] = a2;
}

__global__ void __launch_bounds__(64) hsra_rho_kernel(const double* __restrict__ sb, double* __restrict__ eos /*[2][387]*/,
                                                      int32_t* __restrict__ err_out /*[2]: code, first bad height*/) {
  using R = RhoGroup<64>;
  const R g(threadIdx.x);
  double ne = 0.0;
  int err = ERR_OK, kbad = FZ_HSRA_LEN;
  double n1[R::NS], n2[R::NS];
  g.load(sb, 1, n1, n2);
  for (int k = 0; k < FZ_HSRA_LEN; ++k) {
    double a1[R::NS], ia2[R::NS];
#pragma unroll
    for (int m = 0; m < R::NS; ++m) {
      a1[m] = n1[m];
      ia2[m] = n2[m];
    }
    g.load(sb + (long)min(k + 1, FZ_HSRA_LEN - 1) * FZ_NELEM * 4, 1, n1, n2);
    R::invert(ia2);
    double nh, pel, dens, mu;
    err = g.solve(a1, ia2, (double)fz_hsra_t[k], (double)fz_hsra_pg[k], ne, nh, pel, dens, mu);
    if (err) {
      kbad = k;
      break;
    }
    if (g.q == 0) {
      eos[k] = ne;
      eos[FZ_HSRA_LEN + k] = nh;
    }
  }
  if (g.q == 0) {
    err_out[0] = err;
    err_out[1] = kbad;
  }
}

__global__ void __launch_bounds__(256) hsra_opac_kernel(const double* __restrict__ eos, int32_t* __restrict__ err,
                                                        double* __restrict__ kc_out /*[387][nreg]*/) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= FZ_HSRA_LEN * c_cfg.nreg) return;
  const int k = t / c_cfg.nreg, r = t - k * c_cfg.nreg;
  if (k >= err[1]) return;
  Deriv d = {};
  double kc[4];
  const int e = opac_cont((double)fz_hsra_t[k], c_cfg.reg_l0main[r], eos[k], eos[FZ_HSRA_LEN + k], d, false, kc);
  kc_out[k * c_cfg.nreg + r] = kc[0];
  if (e) atomicMax(&err[2], e);
}

// Continuum formal solution through HSRA per wavelength; every step is
// rounded to REAL(4) like ANALYTICAL_SOLVER_HSRA (normalization.f90:466-480).
// The source function uses the last region's central wavelength for every
// pixel, which is what SOURCE_FUNCTION_HSRA's region test evaluates to
// (normalization.f90:679-682).
__global__ void gain_kernel(const double* __restrict__ kc, float* __restrict__ gain) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= c_cfg.numw) return;
  int r = 0;
  while (r + 1 < c_cfg.nreg && l >= c_cfg.reg_pix0[r + 1]) ++r;
  const double wave = c_cfg.reg_wstart[r] + c_cfg.reg_wstep[r] * (double)(l - c_cfg.reg_pix0[r]);
  const double lam = (c_cfg.reg_l0main[c_cfg.nreg - 1] + wave / 1.0e3) * 1.0e-8;
  const double c1 = 2.0 * HPLA * LIGHT * LIGHT / (lam * lam * lam * lam * lam), c2 = HPLA * LIGHT / (lam * KBOL);
  double syn = 0.0;
  for (int k = 0; k < FZ_HSRA_LEN; ++k) {
    const double sf = (double)(float)(c1 * (1.0 / (exp(c2 / (double)fz_hsra_t[k]) - 1.0)));
    if (k == 0) {
      syn = sf;
      continue;
    }
    double eta = kc[k * c_cfg.nreg + r];
    const bool imat = (eta == eta + 1.0);
    if (imat) eta = 1.0e15;
    const double dz = (k == FZ_HSRA_LEN - 1) ? 1.0e5 * fabs((double)fz_hsra_z[k] - (double)fz_hsra_z[k - 1])
                                             : 1.0e5 * fabs((double)fz_hsra_z[k + 1] - (double)fz_hsra_z[k]);
    const double ev = imat ? 1.0 : exp(-eta * dz);
    syn = (double)(float)((1.0 - ev) * sf + ev * syn);
  }
  const float g = (float)(1.0 / syn);
  gain[4 * l + 0] = g;
  gain[4 * l + 1] = g;
  gain[4 * l + 2] = g;
  gain[4 * l + 3] = -g;   // V sign convention (normalization.f90:743,751)
}


// ---------------------------------------------------------------- layout transposes for FORWARD3D
// Fortran cube (NZ,NY,NX) -> device SoA [z][col] with col = y + NY*x
__global__ void cube_to_soa(const float* __restrict__ src, float* __restrict__ dst, int nz, int ncol) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)nz * ncol) return;
  const int col = (int)(i / nz), k = (int)(i - (long)col * nz);
  dst[(long)k * ncol + col] = src[i];
}
__global__ void soa_to_cube(const float* __restrict__ src, float* __restrict__ dst, int nz, int ncol) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)nz * ncol) return;
  const int col = (int)(i / nz), k = (int)(i - (long)col * nz);
  dst[i] = src[(long)k * ncol + col];
}

}  // namespace fz

#include "fz_lm.hpp"
#include "fz_pert.hpp"
#include "fz_invert.hpp"
#include "fz_mlp.hpp"
#include "fz_psf.hpp"

namespace fz {
// Spectral line-spread function (MLSF) on rows of numw floats (Stokes rows,
// per-height or per-node response functions).  Per valid region of n pixels
// the reference multiplies the r2c DFT of the row by the DFT of LSF_KERNEL
// and transforms back with an unnormalised c2r (forward.f90:621-657,
// 814-844), i.e. the circular convolution
//     y[i] = sum_t tap[t] x[(i - t) mod n],  tap = n * LSF_KERNEL.
// FP32 sums over the n taps of a unit-sum kernel; the rows are updated in place.
//
// lsf_kernel: a contraction of the rows with the circulant of the taps, on
// v_mfma_f32_16x16x4: a wave has 16 rows of a region in LDS (A operand: row
// lane % 16, four k), the taps are there once for the workgroup, unrolled so
// that tap (i - k) mod n is at te[n4 + i - k] (B operand: output lane % 16);
// up to four tiles of 16 outputs share an A operand.  The matrix cores' FP32
// rate bounds it; the vector units (lsf_wide_kernel) read an LDS word per
// multiply-add and took 4.4 ms for a million rows of 3 x 77 wavelengths where
// this takes 0.69 ms.  n4: n rounded up to 4, x zero from n on.
__host__ __device__ constexpr int lsf_pitch(int n) { return ((n + 3) & ~3) + 2; }
__host__ __device__ constexpr int lsf_taps(int n) { return ((n + 3) & ~3) + ((n + 63) & ~63); }

template <int NT>
__device__ __forceinline__ void lsf_tiles(const float* __restrict__ x, const float* __restrict__ te, int n4,
                                          f32x4* acc) {
#pragma unroll
  for (int g = 0; g < NT; ++g) acc[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < n4; k += 4) {
    const float a = x[k];
#pragma unroll
    for (int g = 0; g < NT; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, te[16 * g - k], acc[g], 0, 0, 0);
  }
}

__global__ void __launch_bounds__(256) lsf_kernel(float* __restrict__ rows, long nrows, const float* __restrict__ taps,
                                                  int tcap, int pcap) {
  extern __shared__ float lsf_lds[];
  const int numw = c_cfg.numw;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const long row0 = ((long)blockIdx.x * (blockDim.x >> 6) + w) * 16;
  float* te = lsf_lds;
  float* x = lsf_lds + tcap + w * 16 * pcap;
  for (int r = 0; r < c_cfg.nreg; ++r) {
    if (!c_cfg.reg_lsf[r]) continue;
    const int p0 = c_cfg.reg_pix0[r], n = c_cfg.reg_nwave[r], n4 = (n + 3) & ~3, pitch = lsf_pitch(n);
    __syncthreads();
    for (int j = threadIdx.x; j < lsf_taps(n); j += blockDim.x) {
      int t = (j - n4) % n;
      if (t < 0) t += n;
      te[j] = taps[p0 + t];
    }
    for (int i = lane; i < n4; i += 64) {
      float v[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) v[q] = i < n && row0 + q < nrows ? rows[(row0 + q) * numw + p0 + i] : 0.f;
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q * pitch + i] = v[q];
    }
    __syncthreads();
    if (row0 >= nrows) continue;
    for (int i0 = 0; i0 < n; i0 += 64) {
      f32x4 acc[4];
      const int nt = min(4, (n - i0 + 15) >> 4);
      const float *xa = x + lr * pitch + lk, *ta = te + n4 + i0 + lr - lk;
      switch (nt) {
        case 1: lsf_tiles<1>(xa, ta, n4, acc); break;
        case 2: lsf_tiles<2>(xa, ta, n4, acc); break;
        case 3: lsf_tiles<3>(xa, ta, n4, acc); break;
        default: lsf_tiles<4>(xa, ta, n4, acc);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int i = i0 + 16 * g + lr;
        if (g >= nt || i >= n) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (row0 + 4 * lk + q < nrows) rows[(row0 + 4 * lk + q) * numw + p0 + i] = acc[g][q];
      }
    }
  }
}

// Regions of more wavelengths than 16 rows of LDS hold: one wave per row, lane
// i accumulates output i over the taps, the tap index is wave-uniform
// (scalar loads) and the LDS reads of consecutive lanes are consecutive.
// blockDim.x / 64 rows per workgroup (up to 4, with numw * rows floats of
// LDS <= 64 KiB).
__global__ void __launch_bounds__(256) lsf_wide_kernel(float* __restrict__ rows, long nrows, const float* __restrict__ taps) {
  extern __shared__ float xs[];
  const int numw = c_cfg.numw;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * (blockDim.x >> 6) + w;
  float* x = xs + w * numw;
  float* out = rows + row * numw;
  if (row < nrows)
    for (int i = lane; i < numw; i += 64) x[i] = out[i];
  __syncthreads();
  if (row >= nrows) return;
  for (int r = 0; r < c_cfg.nreg; ++r) {
    if (!c_cfg.reg_lsf[r]) continue;
    const int p0 = c_cfg.reg_pix0[r], n = c_cfg.reg_nwave[r];
    const float* xr = x + p0;
    const float* tr = taps + p0;
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int i = i0 + lane;
      float acc = 0.f;
      int j = i < n ? i : 0;           // (i - t) mod n for t = 0; lanes past n idle in range
      for (int t = 0; t < n; ++t) {
        acc += tr[t] * xr[j];
        j = j == 0 ? n - 1 : j - 1;
      }
      if (i < n) out[p0 + i] = acc;
    }
  }
}
}  // namespace fz

// ==================================================================== C ABI
using namespace fz;

// Learned initial model: network shape, FP32 master parameters (flat:
// W_0, b_0, W_1, b_1, ...; W_l row-major [out][in]), their BF16 copy, Adam
// moments, gradient, normalisations and the per-batch work buffers.
struct MlpState {
  bool on = false;
  int nin = 0, nh = 0, nl = 0, nj = 0, nout = 0, nz = 0;
  long np = 0;
  long woff[8] = {0}, boff[8] = {0};
  int din[8] = {0}, dout[8] = {0};
  MlpShape shape;           // the same, and where the parameters are, for the kernels
  float *w = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
  bf16* wb = nullptr;       // each W_l and its transpose
  float* norms = nullptr;   // xmean[nin], xstd[nin], tmean[nout], tstd[nout]
  double* pinv = nullptr;   // [nj][nz] least-squares node fit
  double* coefs = nullptr;  // [nz][nj] hat basis
  float* loss = nullptr;
  long step = 0;
  // work buffers of the forward pass for cap rows, and what the gradient needs besides for
  // gcap; each only grows, so that batches of different sizes in turn allocate nothing
  int cap = 0, gcap = 0;
  bf16 *X = nullptr, *act = nullptr;      // act: [nl] of frag_size(cap, nh)
  bf16 *XT = nullptr, *actT = nullptr;
  bf16 *dZ = nullptr, *dZT = nullptr;     // two of the widest layer; every layer's
  float *csum = nullptr, *partial = nullptr;
  size_t act_stride() const { return frag_size(cap, nh); }
  size_t actt_stride() const { return frag_size(nh, gcap); }
  size_t dz_stride() const { return frag_size(gcap, std::max(nh, nout)); }
  size_t dzt_stride() const { return frag_size(std::max(nh, nout), gcap); }
  size_t csum_stride() const { return (size_t)pad32(gcap) / 16 * pad32(std::max(nh, nout)); }
  void release() {
    release_forward();
    release_gradient();
    void* ps[] = {w, g, m1, m2, wb, norms, pinv, coefs, loss};
    for (void* q : ps)
      if (q) (void)hipFree(q);
    *this = MlpState();
  }
  void release_forward() {
    for (void* q : {(void*)X, (void*)act})
      if (q) (void)hipFree(q);
    X = act = nullptr;
    cap = 0;
  }
  void release_gradient() {
    for (void* q : {(void*)XT, (void*)actT, (void*)dZ, (void*)dZT, (void*)csum, (void*)partial})
      if (q) (void)hipFree(q);
    XT = actT = dZ = dZT = nullptr;
    csum = partial = nullptr;
    gcap = 0;
  }
};

struct fz_ctx {
  int device = 0;
  bool configured = false;
  bool have_gain = false;
  Cfg cfg;
  std::string err;
  float* d_gain = nullptr;
  float* d_micro = nullptr;
  size_t micro_cap = 0;
  float* d_scratch = nullptr;
  size_t scratch_cap = 0;
  int tile = 32768;
  int block = 256;
  bool prof = false;
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  int rt_launches = 0;
  // microphysics of the next column tile on a second stream while the
  // radiative transfer of the current one runs (default priority); off by
  // default: on the 288x288x96 forward the concurrent kernels slowed the
  // transfer more than they hid (112.5 ms per step against 108)
  bool overlap = false;
  // STOKES SETUP: AUTO (input_file.f90:1294): per-pixel weights from the
  // observations in fz_invert3d_dev
  bool autow = false;
  hipStream_t aux = nullptr;
  std::vector<hipEvent_t> tev;
  // inversion
  bool inv_set = false;
  LmArgs lm;                  // per-cycle constants; per-call pointers filled at launch
  std::vector<int> slot_of;   // [np] physical parameter (= Cartesian slot) of each free parameter
  std::vector<int> kbeg, kend;  // [np] support of each node's hat function
  float* d_invtab = nullptr;  // one buffer for the tables that follow
  size_t invtab_cap = 0;
  int* d_eqvnode = nullptr;   // [3][np]: kbeg, kend, Cartesian slot
  int* d_eqvtab_j = nullptr;  // [nparam][nz] node table of the pairwise contraction
  double* d_eqvtab_c = nullptr;  // [nparam][nz][2]
  bool eqv_pairs = false;
  NodeTab* d_nodetab = nullptr;  // [nz][5]: the contraction within the transfer (five slots)
  bool lm_big = false;        // more than LM_MAXNP free parameters: work arrays in device memory
  size_t lm_work = 0;         // bytes of one pixel's work arrays (lm_big)
  double* d_lmwork = nullptr;
  size_t lmwork_cap = 0;
  double* d_coefs = nullptr;  // [np][nz]
  double* d_colsum = nullptr; // [np]
  float* d_jtile = nullptr;   // per-height response functions of one tile
  size_t jtile_cap = 0;
  // microphysics tile buffers
  int mtile = 0;               // microphysics columns per tile; 0: from the free memory (auto_mtile)
  float* d_sbuf = nullptr;    // Saha factors [nz][92][4][mtile] (double)
  size_t sbuf_cap = 0;
  float* d_eosb = nullptr;    // n_e, N_H [2][nz][mtile] (double)
  size_t eosb_cap = 0;
  float* d_stat = nullptr;    // per-column status when the caller passes none
  size_t stat_cap = 0;
  float* d_smid = nullptr;    // Saha factors at the RK4 mid-step temperatures (double)
  size_t smid_cap = 0;
  float* d_derb = nullptr;    // EOS derivatives [8][nz][mtile] (double)
  size_t derb_cap = 0;
  bool hydro = false;         // HYDROSTATIC: yes
  double xi = 0.0;            // microturbulence (cm/s); survives fz_configure
  size_t lm_lds = 0;
  bool lm_p0 = false;         // P0 among the inverted parameters
  bool lm_pr = false;         // Pg or rho among the inverted parameters
  // per-pixel spectral windows
  bool win_on = false;
  int win_ncol = 0;
  std::vector<int64_t> h_poff;      // [ncol+1]
  std::vector<int> h_item_first;    // [ncol+1] first RT workgroup of each column
  RtItem* d_items = nullptr;
  int64_t* d_poff = nullptr;
  int32_t* d_win = nullptr;         // [ncol][nreg][3]: first, count, position in the pixel's spectrum
  float* d_lsf = nullptr;     // LSF taps n * LSF_KERNEL [numw]
  double* d_pop = nullptr;    // NLTE departure coefficients [2][nz][nreg]
  bool pop_on = false;
  // GET_PERTURBATION / HESSIAN: normal matrix and solver work arrays, and
  // the device copies of the host-array entry points' inputs
  float* d_pert = nullptr;
  size_t pert_cap = 0;
  float* d_pstage = nullptr;
  size_t pstage_cap = 0;
  MlpState mlp;
  // spatial PSF of the coupled inversion: PSF(NPY, NPX) as given, and its
  // tap tables, made at the first convolution with it
  std::vector<double> h_psf;
  int psf_npx = 0, psf_npy = 0;
  float* d_taps = nullptr;
  size_t taps_cap = 0;
  bf16* d_tapfrag = nullptr;  // behind the taps: these as matrix operands (both directions), where in range
  bool taps_ok = false, taps_split = false;
  int taps_rx = 0, taps_ry = 0, taps_ntx = 0;
  double taps_sq = 0.0;   // sum of the squared taps
};



// the context whose configuration is in a device's constant memory
static const fz_ctx* g_owner[64];

static int set_err(fz_ctx* c, int code, const std::string& msg) {
  if (c) c->err = msg;
  return code;
}

#define HIPCHK(c, x)                                                                     \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) return set_err((c), FZ_EHIP, std::string(#x ": ") + hipGetErrorString(e_)); \
  } while (0)

static int ensure(fz_ctx* c, float** p, size_t* cap, size_t bytes);

// rows of numw floats through the LSF (no-op when it is off)
static int run_lsf(fz_ctx* c, float* d_rows, long nrows, hipStream_t st) {
  if (!c->cfg.lsf_on || nrows <= 0) return FZ_OK;
  int nmax = 0;
  for (int r = 0; r < c->cfg.nreg; ++r)
    if (c->cfg.reg_lsf[r]) nmax = std::max(nmax, c->cfg.reg_nwave[r]);
  if (!nmax) return FZ_OK;
  // 16 rows a wave and the taps in 64 KB; as many waves (up to four) as fit
  const int tcap = lsf_taps(nmax), pcap = lsf_pitch(nmax), waves = std::min(4, (16384 - tcap) / (16 * pcap));
  if (waves >= 1) {
    const long nb = (nrows + 16 * waves - 1) / (16 * waves);
    if (nb > 0x7fffffffL) return set_err(c, FZ_EARG, "too many rows for the LSF launch");
    hipLaunchKernelGGL(lsf_kernel, dim3((unsigned)nb), dim3(64 * waves), sizeof(float) * (tcap + 16 * waves * pcap),
                       st, d_rows, nrows, (const float*)c->d_lsf, tcap, pcap);
    HIPCHK(c, hipGetLastError());
    return FZ_OK;
  }
  const int rpb = std::max(1, std::min(4, 16384 / c->cfg.numw));
  const long nb = (nrows + rpb - 1) / rpb;
  if (nb > 0x7fffffffL) return set_err(c, FZ_EARG, "too many rows for the LSF launch");
  hipLaunchKernelGGL(lsf_wide_kernel, dim3((unsigned)nb), dim3(64 * rpb), sizeof(float) * rpb * c->cfg.numw, st, d_rows,
                     nrows, (const float*)c->d_lsf);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// microturbulence xi (cm/s) into the configuration: Doppler temperature
// offsets m xi^2 / (2 k) per line
static void set_xi(Cfg& g, const double* matom, double xi) {
  g.xi_on = xi > 0.0 ? 1 : 0;
  for (int i = 0; i < g.nlines; ++i) {
    g.xi_t[i] = xi * xi * matom[g.line[i].zn] * MAMU / (2.0 * KBOL);
    g.xi_tf[i] = (float)g.xi_t[i];
  }
}

static int upload_cfg(fz_ctx* c) {
  if (c->device < 64 && g_owner[c->device] == c) return FZ_OK;
  HIPCHK(c, hipMemcpyToSymbol(HIP_SYMBOL(c_cfg), &c->cfg, sizeof(Cfg)));
  if (c->device < 64) g_owner[c->device] = c;
  return FZ_OK;
}

// device allocation released when it goes out of scope (early error returns included)
struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

// per-device address of the fixed scratch array (fz_get_perturbation_dev_noalloc)
static int scratch_setup(int device);

extern "C" {

int fz_create(fz_ctx** out, int device) {
  if (!out) return FZ_EARG;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= device || device < 0) return FZ_EHIP;
  fz_ctx* c = new fz_ctx();
  c->device = device;
  if (hipSetDevice(device) != hipSuccess) {
    delete c;
    return FZ_EHIP;
  }
  hipLaunchKernelGGL(fz_init_constants_kernel, dim3(1), dim3(1), 0, 0);
  if (hipDeviceSynchronize() != hipSuccess || scratch_setup(device) != FZ_OK) {
    delete c;
    return FZ_EHIP;
  }
  *out = c;
  return FZ_OK;
}

void fz_destroy(fz_ctx* c) {
  if (!c) return;
  if (c->device < 64 && g_owner[c->device] == c) g_owner[c->device] = nullptr;
  (void)hipSetDevice(c->device);
  for (hipEvent_t e : c->tev) (void)hipEventDestroy(e);
  if (c->aux) (void)hipStreamDestroy(c->aux);
  if (c->d_gain) (void)hipFree(c->d_gain);
  if (c->d_micro) (void)hipFree(c->d_micro);
  if (c->d_scratch) (void)hipFree(c->d_scratch);
  if (c->d_invtab) (void)hipFree(c->d_invtab);
  if (c->d_lmwork) (void)hipFree(c->d_lmwork);
  if (c->d_jtile) (void)hipFree(c->d_jtile);
  if (c->d_sbuf) (void)hipFree(c->d_sbuf);
  if (c->d_eosb) (void)hipFree(c->d_eosb);
  if (c->d_stat) (void)hipFree(c->d_stat);
  if (c->d_smid) (void)hipFree(c->d_smid);
  if (c->d_derb) (void)hipFree(c->d_derb);
  if (c->d_items) (void)hipFree(c->d_items);
  if (c->d_poff) (void)hipFree(c->d_poff);
  if (c->d_win) (void)hipFree(c->d_win);
  if (c->d_lsf) (void)hipFree(c->d_lsf);
  if (c->d_pop) (void)hipFree(c->d_pop);
  if (c->d_pert) (void)hipFree(c->d_pert);
  if (c->d_pstage) (void)hipFree(c->d_pstage);
  if (c->d_taps) (void)hipFree(c->d_taps);
  c->mlp.release();
  for (int i = 0; i < 3; ++i)
    if (c->ev[i]) (void)hipEventDestroy(c->ev[i]);
  delete c;
}

const char* fz_last_error(const fz_ctx* c) { return c ? c->err.c_str() : "null context"; }

// Zeeman pattern of one line (magsplit.f90:38-187), components grouped by type
static int zeeman_host(const fz_line& L, std::vector<float>& shift, std::vector<float>& str, int ntype[3]) {
  const int dj = (int)(L.ju - L.jl);
  if (std::abs(dj) > 1) return -1;
  double gl = 0.0, gu = 0.0;
  if (L.jl != 0) gl = 1.5 + (L.sl * (L.sl + 1.0) - L.ll * (L.ll + 1.0)) / (2.0 * L.jl * (L.jl + 1.0));
  if (L.ju != 0) gu = 1.5 + (L.su * (L.su + 1.0) - L.lu * (L.lu + 1.0)) / (2.0 * L.ju * (L.ju + 1.0));
  std::vector<double> sh[3], st[3];
  const int nml = (int)(2 * L.jl + 1), nmu = (int)(2 * L.ju + 1);
  for (int j = 0; j < nml; ++j) {
    const double ml = (double)j - L.jl;
    for (int k = 0; k < nmu; ++k) {
      const double mu = (double)k - L.ju;
      const int dm = (int)(mu - ml);
      if (std::abs(dm) > 1) continue;
      const double jl = L.jl, ju = L.ju;
      double s;
      if (dj == -1) s = dm == -1 ? (jl + mu) * (ju + mu + 2.0) : (dm == 0 ? 2.0 * (jl * jl - mu * mu) : (jl - mu) * (ju - mu + 2.0));
      else if (dj == 0) s = dm == -1 ? (ju - mu) * (ju + mu + 1.0) : (dm == 0 ? 2.0 * mu * mu : (ju + mu) * (ju - mu + 1.0));
      else s = dm == -1 ? (ju - mu) * (jl - mu) : (dm == 0 ? 2.0 * (ju * ju - mu * mu) : (ju + mu) * (jl + mu));
      // shift in mA/G rounded to REAL(4) as in the reference
      sh[dm + 1].push_back((double)(float)(4.66685e-10 * (ml * gl - mu * gu) * L.lambda0 * L.lambda0));
      st[dm + 1].push_back(s);
    }
  }
  for (int t = 0; t < 3; ++t) {
    double sum = 0.0;
    for (double v : st[t]) sum += v;
    ntype[t] = 0;
    for (size_t i = 0; i < st[t].size(); ++i) {
      // the pi component 0 -> 0 of a J = J transition has no strength
      if (st[t][i] == 0.0) continue;
      shift.push_back((float)sh[t][i]);
      str.push_back((float)(st[t][i] / sum));
      ++ntype[t];
    }
  }
  return 0;
}

}  // extern "C"

// drops the per-pixel windows (their regions are those of one configuration)
static void clear_windows(fz_ctx* c) {
  if (c->d_items) (void)hipFree(c->d_items);
  if (c->d_poff) (void)hipFree(c->d_poff);
  if (c->d_win) (void)hipFree(c->d_win);
  c->d_items = nullptr;
  c->d_poff = nullptr;
  c->d_win = nullptr;
  c->win_on = false;
  c->win_ncol = 0;
  c->h_poff.clear();
  c->h_item_first.clear();
}

extern "C" {

int fz_configure(fz_ctx* c, const fz_line* lines, int nlines, const fz_region* regs, int nreg, int nz,
                 const double* z_km) {
  if (!c || !lines || !regs || !z_km) return FZ_EARG;
  if (nlines < 1 || nlines > MAXL || nreg < 1 || nreg > MAXR || nz < 2 || nz > MAXNZ)
    return set_err(c, FZ_ECONFIG, "configuration outside limits");
  Cfg& g = c->cfg;
  memset(&g, 0, sizeof(g));
  g.nlines = nlines;
  g.nreg = nreg;
  g.nz = nz;
  std::vector<float> shift, str;
  double matom[FZ_NELEM];
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMemcpyFromSymbol(matom, HIP_SYMBOL(fz_matom), sizeof(matom)));
  for (int i = 0; i < nlines; ++i) {
    const fz_line& L = lines[i];
    if (L.zn < 1 || L.zn > FZ_NELEM || L.ion < 1 || L.ion > 3) return set_err(c, FZ_EION, "bad element/ion");
    g.line[i] = {L.zn - 1, L.ion, L.lambda0, L.loggf, L.eplow, L.sigma, L.alpha};
    g.dopfac[i] = (float)(1.0e3 * L.lambda0 / LIGHT * sqrt(2.0 * KBOL / (matom[L.zn - 1] * MAMU)));
    g.idopfac[i] = (float)(1.0 / (1.0e3 * L.lambda0 / LIGHT * sqrt(2.0 * KBOL / (matom[L.zn - 1] * MAMU))));
    g.vfac[i] = (float)(-1.0e3 * L.lambda0 / LIGHT);
    g.comp0[i] = (int)shift.size();
    if (zeeman_host(L, shift, str, g.ntype[i]) != 0) return set_err(c, FZ_ECONFIG, "|Delta J| > 1");
  }
  if ((int)shift.size() > MAXC) return set_err(c, FZ_ECONFIG, "too many Zeeman components");
  for (int i = 0; i < nlines; ++i) {
    size_t m = (size_t)g.comp0[i];
    for (int t = 0; t < 3; ++t) {
      double c0 = 0.0, w = 0.0, w1 = 0.0;
      for (int j = 0; j < g.ntype[i][t]; ++j) c0 += (double)str[m + j] * (double)shift[m + j];
      const float cen = (float)c0;
      for (int j = 0; j < g.ntype[i][t]; ++j, ++m) {
        const float dl = (float)((double)shift[m] - (double)cen), st = str[m];
        g.comp[m] = {dl, st, (float)((double)st * dl), (float)((double)st * dl * dl)};
        w += (double)st;
        w1 += (double)st * (double)dl;
      }
      const double isp = 0.564189583547756;   // 1/sqrt(pi)
      g.type[i][t] = {cen, (float)(isp * w), (float)(isp * w1), 0.f};
    }
  }
  int numw = 0, ns = 0;
  for (int r = 0; r < nreg; ++r) {
    const fz_region& R = regs[r];
    if (R.nblend < 1 || R.nblend > 4 || R.nwave < 1) return set_err(c, FZ_ECONFIG, "bad region");
    g.reg_nblend[r] = R.nblend;
    g.reg_slot0[r] = ns;
    g.reg_pix0[r] = numw;
    g.reg_nwave[r] = R.nwave;
    g.reg_wstart[r] = R.wave_start;
    g.reg_wstep[r] = R.wave_step;
    g.reg_l0main[r] = lines[R.line[0]].lambda0;
    for (int b = 0; b < R.nblend; ++b) {
      if (R.line[b] < 0 || R.line[b] >= nlines || ns >= MAXS) return set_err(c, FZ_ECONFIG, "bad blend");
      g.slot_line[ns] = R.line[b];
      g.slot_bldiff[ns] = b == 0 ? 0.f : (float)(1.0e3 * (lines[R.line[b]].lambda0 - lines[R.line[0]].lambda0));
      ++ns;
    }
    numw += R.nwave;
  }
  g.nslot = ns;
  g.numw = numw;
  g.nbpc = 0;
  for (int r = 0; r < nreg; ++r)
    for (int l0 = g.reg_pix0[r]; l0 < g.reg_pix0[r] + g.reg_nwave[r]; l0 += RT_WAVE) {
      if (g.nbpc >= MAXBLK) return set_err(c, FZ_ECONFIG, "too many wavelengths");
      g.blk_reg[g.nbpc] = r;
      g.blk_l0[g.nbpc] = l0;
      g.blk_n[g.nbpc] = std::min(RT_WAVE, g.reg_pix0[r] + g.reg_nwave[r] - l0);
      ++g.nbpc;
    }
  for (int sl = 0; sl < ns; ++sl) {
    const int li = g.slot_line[sl];
    Cfg::SlotRt& q = g.slot_rt[sl];
    q.comp0 = g.comp0[li];
    q.bldiff = g.slot_bldiff[sl];
    q.vfac = g.vfac[li];
    for (int t = 0; t < 3; ++t) {
      q.n[t] = g.ntype[li][t];
      q.type[t] = g.type[li][t];
    }
  }
  g.rec = REC_HEAD;
  for (int r = 0; r < nreg; ++r) {
    g.reg_rec[r] = g.rec;
    g.rec += REC_REG + REC_SLOT * g.reg_nblend[r];
  }
  set_xi(g, matom, c->xi);
  // layer thickness uses the spacing to the next height, the top one the
  // spacing below (rtesolver.f90:439-443); z rounded to REAL(4) like MODEL(:,13)
  for (int k = 0; k < nz; ++k) {
    const double zk = (double)(float)z_km[k];
    const double zo = (k == nz - 1) ? (double)(float)z_km[k - 1] : (double)(float)z_km[k + 1];
    g.dz_cm[k] = (float)(1.0e5 * fabs(zo - zk));
    g.zz[k] = zk;
  }
  {
    double t0 = g.zz[nz - 1] * 1000.0 * 100.0;
    for (int k = nz - 2; k >= 0; --k) {
      const double dz = (g.zz[k] - g.zz[k + 1]) * 1000.0 * 100.0;
      const double it1 = t0 + dz / 2.0;
      g.he_dz[k] = dz;
      g.he_a[k] = t0 + dz - it1;
      g.he_b[k] = it1 - t0;
      t0 = t0 + dz;
    }
    g.he_cte[0] = 0.f;
    for (int k = 1; k < nz; ++k) g.he_cte[k] = (float)(MAMU / KBOL * GRAV * (g.zz[k] - g.zz[k - 1]) * 1.0e3 * 1.0e2);
  }
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMemcpyToSymbol(HIP_SYMBOL(c_cfg), &g, sizeof(Cfg)));
  if (c->device < 64) g_owner[c->device] = c;
  if (c->d_gain) (void)hipFree(c->d_gain);
  HIPCHK(c, hipMalloc(&c->d_gain, sizeof(float) * 4 * numw));
  std::vector<float> ones(4 * numw, 1.0f);
  for (int l = 0; l < numw; ++l) ones[4 * l + 3] = -1.0f;
  HIPCHK(c, hipMemcpy(c->d_gain, ones.data(), sizeof(float) * 4 * numw, hipMemcpyHostToDevice));
  clear_windows(c);
  c->pop_on = false;   // LTE until fz_set_departure (input_file.f90:504-508)
  c->configured = true;
  c->have_gain = false;
  return FZ_OK;
}

int fz_numw(const fz_ctx* c) { return (c && c->configured) ? c->cfg.numw : -1; }

int fz_set_gain(fz_ctx* c, const float* gain) {
  if (!c || !c->configured || !gain) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMemcpy(c->d_gain, gain, sizeof(float) * 4 * c->cfg.numw, hipMemcpyHostToDevice));
  c->have_gain = true;
  return FZ_OK;
}

int fz_set_departure(fz_ctx* c, const double* popl, const double* popu) {
  if (!c || !c->configured) return FZ_EARG;
  if (!popl || !popu) {
    c->pop_on = false;
    return FZ_OK;
  }
  const int nz = c->cfg.nz, nreg = c->cfg.nreg;
  const size_t n = (size_t)nz * nreg;
  std::vector<double> h(2 * n);
  for (size_t i = 0; i < n; ++i) {
    // POPL(r, k) at r + k*nreg, the device layout [2][nz][nreg]
    if (!(popl[i] > 0.0) || !(popu[i] > 0.0) || !std::isfinite(popl[i]) || !std::isfinite(popu[i]))
      return set_err(c, FZ_EARG, "departure coefficients must be finite and positive");
    h[i] = popl[i];
    h[n + i] = popu[i];
  }
  HIPCHK(c, hipSetDevice(c->device));
  if (c->d_pop) (void)hipFree(c->d_pop);
  c->d_pop = nullptr;
  HIPCHK(c, hipMalloc(&c->d_pop, sizeof(double) * 2 * n));
  HIPCHK(c, hipMemcpy(c->d_pop, h.data(), sizeof(double) * 2 * n, hipMemcpyHostToDevice));
  c->pop_on = true;
  return FZ_OK;
}

int fz_set_psf(fz_ctx* c, const double* psf, int npy, int npx) {
  if (!c) return FZ_EARG;
  if (!psf) {
    c->h_psf.clear();
    c->psf_npx = c->psf_npy = 0;
    c->taps_ok = false;
    return FZ_OK;
  }
  if (npx < 1 || npy < 1 || npx / 2 > PSF_RMAX || npy / 2 > PSF_RMAX)
    return set_err(c, FZ_EARG, "PSF size outside 1 .. 63 pixels per axis");
  // READ_PSF takes NPX/2 pixels either side of (NPY/2 + 1, NPX/2 + 1): an even
  // side would reach one pixel past the array
  if (npx % 2 == 0 || npy % 2 == 0) return set_err(c, FZ_EARG, "PSF sides must be odd");
  for (long i = 0; i < (long)npx * npy; ++i)
    if (!std::isfinite(psf[i])) return set_err(c, FZ_EARG, "PSF values must be finite");
  c->h_psf.assign(psf, psf + (size_t)npx * npy);
  c->psf_npx = npx;
  c->psf_npy = npy;
  c->taps_ok = false;
  return FZ_OK;
}

}  // extern "C"

// the taps of the PSF (READ_PSF's central part of half-widths NPX/2, NPY/2
// around (NPY/2 + 1, NPX/2 + 1)) for an nx x ny map: the tables do not depend on
// the map, whose periodic sum needs 2 r + 1 <= n along each axis
static int psf_taps(fz_ctx* c, int nx, int ny) {
  if (c->h_psf.empty()) return set_err(c, FZ_ECONFIG, "no PSF set (fz_set_psf)");
  const int rx = c->psf_npx / 2, ry = c->psf_npy / 2;
  if (2 * rx + 1 > nx || 2 * ry + 1 > ny) return set_err(c, FZ_ECONFIG, "PSF wider than the map");
  if (c->taps_ok) return FZ_OK;
  const int x0 = c->psf_npx / 2, y0 = c->psf_npy / 2, nu = 2 * ry + 1;
  const int ntx = (2 * rx + 1 + 7) / 8 * 8;
  // two tap tables [nu][ntx] in the kernel's window order: the convolution's
  // (tap (t, u) = PSF(Y0 + ry - u, X0 + rx - t)) and the adjoint's
  // (PSF(Y0 + u - ry, X0 + t - rx)); zero beyond t = 2 rx
  std::vector<float> t((size_t)2 * nu * ntx, 0.f);
  double sq = 0.0;
  for (int dx = -rx; dx <= rx; ++dx)
    for (int dy = -ry; dy <= ry; ++dy) {
      const float v = (float)c->h_psf[(size_t)(y0 + dy) + (size_t)c->psf_npy * (x0 + dx)];
      t[(size_t)(ry - dy) * ntx + (rx - dx)] = v;
      t[(size_t)nu * ntx + (size_t)(ry + dy) * ntx + (rx + dx)] = v;
      sq += (double)v * (double)v;
    }
  // Sixteen taps and fewer are left to the vector units: the matrix cores' work
  // does not get less below 2 rx + 1 = 32 (ms, vector units / matrix cores, 112
  // maps of 256 x 256: 9 x 9 taps 0.067 / 0.071, 15 x 15 0.089 / 0.092, 17 x 17
  // 0.131 / 0.087; 64 maps, 63 x 63 0.61 / 0.29).
  bool split = ntx > 16;
  for (float v : t)
    if (v != 0.f && !(std::fabs(v) > 0x1p-100f && std::fabs(v) < 0x1p100f)) split = false;
  // taps, then operands: [direction][u][x tile][step][part][lane][8]
  const int ks = psf_steps(ntx), npiece = split ? 2 * nu * 2 * ks * 3 * 64 : 0;
  const size_t off = (sizeof(float) * t.size() + 255) / 256 * 256;
  HIPCHK(c, hipSetDevice(c->device));
  // convolutions with the tables of another PSF may be running
  HIPCHK(c, hipDeviceSynchronize());
  int r = ensure(c, &c->d_taps, &c->taps_cap, off + sizeof(bf16) * 8 * npiece);
  if (r) return r;
  c->d_tapfrag = reinterpret_cast<bf16*>(reinterpret_cast<char*>(c->d_taps) + off);
  HIPCHK(c, hipMemcpy(c->d_taps, t.data(), sizeof(float) * t.size(), hipMemcpyHostToDevice));
  if (split) {
    hipLaunchKernelGGL(psf_operand_kernel, dim3((unsigned)((npiece + 255) / 256)), dim3(256), 0, 0,
                       (const float*)c->d_taps, npiece, ks, ntx, c->d_tapfrag);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(0));   // before a convolution on any stream
  }
  c->taps_rx = rx;
  c->taps_ry = ry;
  c->taps_ntx = ntx;
  c->taps_sq = sq;
  c->taps_split = split;
  c->taps_ok = true;
  return FZ_OK;
}

template <int NTX, int YT>
static void launch_psf_split_y(fz_ctx* c, const PsfArgs& a, int adjoint, hipStream_t st) {
  constexpr int KS = psf_steps(NTX);
  const int ty = 32 * YT, nu = 2 * a.ry + 1;
  const size_t lds = std::max(sizeof(bf16) * 3 * (ty + 2 * a.ry) * (32 * KS + 8),
                              sizeof(float) * (PSF_TX + NTX - 1) * (PSF_TY + 2 * a.ry));
  (void)hipFuncSetAttribute((const void*)psf_split_kernel<NTX, YT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            144 * 1024);
  const dim3 grid((unsigned)((a.ny + ty - 1) / ty), (unsigned)((a.nx + PSF_TX - 1) / PSF_TX), (unsigned)a.nmaps);
  hipLaunchKernelGGL((psf_split_kernel<NTX, YT>), grid, dim3(256), lds, st, a,
                     (const bf16*)c->d_tapfrag + (adjoint ? (size_t)nu * 2 * KS * 3 * 512 : 0));
}

template <int NTX>
static void launch_psf_split(fz_ctx* c, const PsfArgs& a, int adjoint, hipStream_t st) {
  // 128 y a workgroup, 64 where that covers the map with fewer
  if ((a.ny + 127) / 128 * 2 <= (a.ny + 63) / 64)
    launch_psf_split_y<NTX, 4>(c, a, adjoint, st);
  else
    launch_psf_split_y<NTX, 2>(c, a, adjoint, st);
}

static void launch_psf(fz_ctx* c, int nx, int ny, int nmaps, const float* in, float* out, int adjoint, hipStream_t st) {
  PsfArgs a;
  a.nx = nx;
  a.ny = ny;
  a.nmaps = nmaps;
  a.rx = c->taps_rx;
  a.ry = c->taps_ry;
  a.npix = (long)nx * ny;
  const int ntx = c->taps_ntx;
  a.taps = c->d_taps + (adjoint ? (size_t)(2 * a.ry + 1) * ntx : 0);
  a.in = in;
  a.out = out;
  if (c->taps_split) {
    switch (ntx) {
      case 24: launch_psf_split<24>(c, a, adjoint, st); break;
      case 32: launch_psf_split<32>(c, a, adjoint, st); break;
      case 40: launch_psf_split<40>(c, a, adjoint, st); break;
      case 48: launch_psf_split<48>(c, a, adjoint, st); break;
      case 56: launch_psf_split<56>(c, a, adjoint, st); break;
      default: launch_psf_split<64>(c, a, adjoint, st); break;
    }
    return;
  }
  const size_t lds = sizeof(float) * (PSF_TX + ntx - 1) * (PSF_TY + 2 * a.ry);
  const dim3 grid((unsigned)((ny + PSF_TY - 1) / PSF_TY), (unsigned)((nx + PSF_TX - 1) / PSF_TX), (unsigned)nmaps);
  switch (ntx) {
    case 8: hipLaunchKernelGGL(psf_conv_kernel<8>, grid, dim3(256), lds, st, a); break;
    case 16: hipLaunchKernelGGL(psf_conv_kernel<16>, grid, dim3(256), lds, st, a); break;
    case 24: hipLaunchKernelGGL(psf_conv_kernel<24>, grid, dim3(256), lds, st, a); break;
    case 32: hipLaunchKernelGGL(psf_conv_kernel<32>, grid, dim3(256), lds, st, a); break;
    case 40: hipLaunchKernelGGL(psf_conv_kernel<40>, grid, dim3(256), lds, st, a); break;
    case 48: hipLaunchKernelGGL(psf_conv_kernel<48>, grid, dim3(256), lds, st, a); break;
    case 56: hipLaunchKernelGGL(psf_conv_kernel<56>, grid, dim3(256), lds, st, a); break;
    default: hipLaunchKernelGGL(psf_conv_kernel<64>, grid, dim3(256), lds, st, a); break;
  }
}

extern "C" {

int fz_psf_convolve_dev(fz_ctx* c, int nx, int ny, int nmaps, const float* d_in, float* d_out, int adjoint,
                        void* stream) {
  if (!c || nx < 1 || ny < 1 || nmaps < 1 || nmaps > 65535 || !d_in || !d_out || d_in == d_out) return FZ_EARG;
  int r = psf_taps(c, nx, ny);
  if (r) return r;
  HIPCHK(c, hipSetDevice(c->device));
  launch_psf(c, nx, ny, nmaps, d_in, d_out, adjoint != 0, (hipStream_t)stream);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_set_lsf(fz_ctx* c, const double* lsf_kernel, const int32_t* lsf_valid) {
  if (!c || !c->configured) return FZ_EARG;
  Cfg& g = c->cfg;
  HIPCHK(c, hipSetDevice(c->device));
  g.lsf_on = 0;
  for (int r = 0; r < g.nreg; ++r) g.reg_lsf[r] = 0;
  if (lsf_kernel) {
    std::vector<float> taps(g.numw, 0.f);
    for (int r = 0; r < g.nreg; ++r) {
      g.reg_lsf[r] = lsf_valid ? (lsf_valid[r] != 0) : 1;
      const int p0 = g.reg_pix0[r], n = g.reg_nwave[r];
      for (int i = 0; i < n; ++i) {
        if (!std::isfinite(lsf_kernel[p0 + i])) return set_err(c, FZ_EARG, "non-finite LSF kernel");
        taps[p0 + i] = (float)(lsf_kernel[p0 + i] * (double)n);
      }
    }
    if (!c->d_lsf) HIPCHK(c, hipMalloc(&c->d_lsf, sizeof(float) * RT_WAVE * MAXBLK));
    HIPCHK(c, hipMemcpy(c->d_lsf, taps.data(), sizeof(float) * g.numw, hipMemcpyHostToDevice));
    g.lsf_on = 1;
  }
  HIPCHK(c, hipMemcpyToSymbol(HIP_SYMBOL(c_cfg), &g, sizeof(Cfg)));
  if (c->device < 64) g_owner[c->device] = c;
  return FZ_OK;
}

int fz_set_windows(fz_ctx* c, int ncol, const int32_t* windows) {
  if (!c || !c->configured) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  clear_windows(c);
  if (!windows) return FZ_OK;
  if (ncol < 1) return set_err(c, FZ_EARG, "no columns");
  const Cfg& g = c->cfg;
  const int nreg = g.nreg;
  std::vector<int64_t> poff((size_t)ncol + 1, 0);
  std::vector<int> first((size_t)ncol + 1, 0);
  std::vector<RtItem> items;
  std::vector<int32_t> w((size_t)ncol * nreg * 3);
  for (int col = 0; col < ncol; ++col) {
    int pos = 0;
    for (int r = 0; r < nreg; ++r) {
      const int f0 = windows[((size_t)col * nreg + r) * 2], cnt = windows[((size_t)col * nreg + r) * 2 + 1];
      if (cnt < 0 || f0 < 0 || f0 + cnt > g.reg_nwave[r])
        return set_err(c, FZ_EARG, "window outside its region (column " + std::to_string(col) + ")");
      w[((size_t)col * nreg + r) * 3 + 0] = f0;
      w[((size_t)col * nreg + r) * 3 + 1] = cnt;
      w[((size_t)col * nreg + r) * 3 + 2] = pos;
      for (int o = 0; o < cnt; o += RT_WAVE) {
        RtItem it;
        it.col = col;
        it.r = (short)r;
        it.n = (short)std::min(RT_WAVE, cnt - o);
        it.l0 = g.reg_pix0[r] + f0 + o;
        it.lout = pos + o;
        items.push_back(it);
      }
      pos += cnt;
    }
    if (pos == 0) return set_err(c, FZ_EARG, "a pixel without wavelengths (column " + std::to_string(col) + ")");
    poff[col + 1] = poff[col] + pos;
    if (items.size() > (size_t)0x7fffffff) return set_err(c, FZ_EARG, "too many workgroups");
    first[col + 1] = (int)items.size();
  }
  HIPCHK(c, hipMalloc(&c->d_items, sizeof(RtItem) * items.size()));
  HIPCHK(c, hipMalloc(&c->d_poff, sizeof(int64_t) * poff.size()));
  HIPCHK(c, hipMalloc(&c->d_win, sizeof(int32_t) * w.size()));
  HIPCHK(c, hipMemcpy(c->d_items, items.data(), sizeof(RtItem) * items.size(), hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(c->d_poff, poff.data(), sizeof(int64_t) * poff.size(), hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(c->d_win, w.data(), sizeof(int32_t) * w.size(), hipMemcpyHostToDevice));
  c->h_poff = poff;
  c->h_item_first = first;
  c->win_ncol = ncol;
  c->win_on = true;
  return FZ_OK;
}

int fz_window_offsets(const fz_ctx* c, int64_t* offsets) {
  if (!c || !c->win_on || !offsets) return FZ_EARG;
  std::memcpy(offsets, c->h_poff.data(), sizeof(int64_t) * c->h_poff.size());
  return FZ_OK;
}

int fz_gain_hsra(fz_ctx* c, float* gain) {
  if (!c || !c->configured) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  int ru = upload_cfg(c);
  if (ru) return ru;
  DevBuf b_kc, b_err, b_sb, b_eos;
  HIPCHK(c, hipMalloc(&b_kc.p, sizeof(double) * FZ_HSRA_LEN * c->cfg.nreg));
  HIPCHK(c, hipMalloc(&b_err.p, sizeof(int32_t) * 3));
  HIPCHK(c, hipMalloc(&b_sb.p, sizeof(double) * FZ_HSRA_LEN * FZ_NELEM * 4));
  HIPCHK(c, hipMalloc(&b_eos.p, sizeof(double) * 2 * FZ_HSRA_LEN));
  double* kc = (double*)b_kc.p;
  int32_t* derr = (int32_t*)b_err.p;
  const int32_t zero3[3] = {0, 0, 0};
  HIPCHK(c, hipMemcpy(derr, zero3, sizeof(zero3), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(hsra_saha_kernel, dim3((FZ_HSRA_LEN * FZ_NELEM + 255) / 256), dim3(256), 0, 0, (double*)b_sb.p);
  hipLaunchKernelGGL(hsra_rho_kernel, dim3(1), dim3(64), 0, 0, (const double*)b_sb.p, (double*)b_eos.p, derr);
  hipLaunchKernelGGL(hsra_opac_kernel, dim3((FZ_HSRA_LEN * c->cfg.nreg + 255) / 256), dim3(256), 0, 0,
                     (const double*)b_eos.p, derr, kc);
  HIPCHK(c, hipGetLastError());
  int32_t eh[3] = {0, 0, 0};
  HIPCHK(c, hipMemcpy(eh, derr, sizeof(eh), hipMemcpyDeviceToHost));
  // the first failure in height order, as the sequential loop meets it: the
  // EOS of height kbad, or an opacity of a height below it
  const int32_t e = eh[2] ? eh[2] : eh[0];
  if (e == ERR_LAMBDA) return set_err(c, e, "HSRA normalisation: wavelength below 1800 A");
  if (e) return set_err(c, e, "HSRA normalisation: equation of state or opacity failed");
  hipLaunchKernelGGL(gain_kernel, dim3((c->cfg.numw + 63) / 64), dim3(64), 0, 0, kc, c->d_gain);
  HIPCHK(c, hipGetLastError());
  if (gain) HIPCHK(c, hipMemcpy(gain, c->d_gain, sizeof(float) * 4 * c->cfg.numw, hipMemcpyDeviceToHost));
  c->have_gain = true;
  return FZ_OK;
}


static int ensure(fz_ctx* c, float** p, size_t* cap, size_t bytes) {
  if (*cap >= bytes) return FZ_OK;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (hipMalloc((void**)p, bytes) != hipSuccess) return set_err(c, FZ_ENOMEM, "device allocation failed");
  *cap = bytes;
  return FZ_OK;
}

// floats of radiative-transfer scratch per lane (column-wavelength): the
// incoming Stokes vector of every layer (and W_k with HYDROSTATIC)
static size_t rt_scratch_per_lane(const fz_ctx* c, int rf_mode) {
  if (rf_mode == FZ_RF_NONE) return 0;
  const size_t nz = (size_t)c->cfg.nz;
  return nz * (c->hydro ? 8 : 4);
}

// columns of one radiative-transfer launch: the configured tile, at most as many as
// keep its lanes (rounded up to waves) below 2^29, so that the kernel's lane
// numbers and the launch's work-items, four times as many with teams, stay within 32 bits
static int rt_tile(const fz_ctx* c, int ncol) {
  return std::min(std::min(c->tile, ncol), (1 << 29) / (RT_WAVE * c->cfg.nbpc));
}

static int rf_nparam(int rf_mode) {
  return rf_mode == FZ_RF_SPHERICAL ? 5
         : rf_mode == FZ_RF_CARTESIAN ? 7
         : rf_mode == FZ_RF_CARTESIAN_P0 ? 8
         : rf_mode == RF_CART_TBV ? 5
         : 0;
}

static int launch_rt(fz_ctx* c, int rf_mode, RtArgs a, hipStream_t st, int nitems = 0, const NodeArgs* nd = nullptr) {
  if (a.items && nitems == 0) return FZ_OK;
  const Cfg& g = c->cfg;
  // packed lanes without windows, as long as the response functions of a
  // wave's columns stay within 32-bit offsets
  int npar = 0, nmin = g.numw, nb = 0;
  if (rf_mode == FZ_RF_SPHERICAL) npar = 5;
  else if (rf_mode != FZ_RF_NONE) npar = 8;
  long npack = 0;
  for (int r = 0; r < g.nreg; ++r) {
    npack += ((long)a.ntile * g.reg_nwave[r] + RT_WAVE - 1) / RT_WAVE;
    nmin = std::min(nmin, g.reg_nwave[r]);
    nb = std::max(nb, g.reg_nblend[r]);
  }
  int wcols = std::min(a.ntile, 1 + (RT_WAVE - 1 + nmin - 1) / nmin);   // columns that a packed wave spans at most
  const bool pack = !a.items && 16L * wcols * npar * g.nz * g.numw < (1L << 31);
  if (!pack) wcols = 1;
  const dim3 grid(a.items ? (unsigned)nitems : pack ? (unsigned)npack : (unsigned)a.ntile * (unsigned)g.nbpc);
  // a wave's share of LDS: as many heights of its columns' records as 10 KB
  // hold (16 waves per CU), one at least
  const size_t per = sizeof(float) * (REC_HEAD + REC_REG + REC_SLOT * (size_t)nb) * wcols;
  a.chunk = (int)std::max<size_t>(1, std::min<size_t>((size_t)std::min(16, g.nz), RT_LDS / per));
  // Teams while one wave per 64 lanes leaves SIMDs without a wave, for the
  // synthesis always (its tail and its records in LDS gain from them):
  // ms with 8 / 4 / 1 waves, 64 heights: 64 columns x 120 wavelengths, 5
  // responses 0.42 / 0.47 / 0.74; 400 columns 0.65 / 0.55 / 0.80; 1600 columns 1.74 / 1.36 / 1.30;
  // node responses of 256 x 112 0.76 / 0.70 / 0.94, of 1024 x 112 1.52 / 1.23 / 1.14;
  // synthesis of 64 x 112 0.27 / 0.28 / 0.37, of 4096 x 112 1.05 / 0.98 / 1.05.
  int team = 1;
  if (pack || nd) {
    if (grid.x <= 256 && per * 8 <= 16384) team = 8;
    else if ((grid.x <= 1024 || rf_mode == FZ_RF_NONE) && per * 4 <= 16384) team = 4;
  }
  if (team > 1) a.chunk = (int)std::min<size_t>(16, 16384 / per) / team * team;
  const size_t lds = per * a.chunk;
  a.pop = c->pop_on ? c->d_pop : nullptr;
  const NodeArgs nodes = nd ? *nd : NodeArgs();
#define FZ_RT(RF, HE, PK, ND, NW) \
  hipLaunchKernelGGL((rt_kernel<RF, HE, PK, ND, NW>), grid, dim3(RT_WAVE * NW), lds, st, a, nodes, \
                     (const NodeTab*)c->d_nodetab)
#define FZ_RTT(RF, HE, PK, ND) \
  do { \
    if (team == 8) FZ_RT(RF, HE, PK, ND, 8); \
    else if (team == 4) FZ_RT(RF, HE, PK, ND, 4); \
    else FZ_RT(RF, HE, PK, ND, 1); \
  } while (0)
#define FZ_RTP(RF, HE) \
  do { \
    if (pack) FZ_RTT(RF, HE, true, false); \
    else FZ_RT(RF, HE, false, false, 1); \
  } while (0)
  if (nd && pack) FZ_RTT(RF_CART_TBV, false, true, true);
  else if (nd) FZ_RTT(RF_CART_TBV, false, false, true);
  else if (rf_mode == FZ_RF_NONE) FZ_RTP(FZ_RF_NONE, false);
  else if (!c->hydro && rf_mode == FZ_RF_SPHERICAL) FZ_RTP(FZ_RF_SPHERICAL, false);
  else if (!c->hydro && rf_mode == FZ_RF_CARTESIAN_P0) FZ_RTP(FZ_RF_CARTESIAN_P0, false);
  else if (c->hydro && rf_mode == FZ_RF_CARTESIAN_P0) FZ_RTP(FZ_RF_CARTESIAN_P0, true);
  else if (!c->hydro) FZ_RTP(FZ_RF_CARTESIAN, false);
  else if (rf_mode == FZ_RF_SPHERICAL) FZ_RTP(FZ_RF_SPHERICAL, true);
  else FZ_RTP(FZ_RF_CARTESIAN, true);
#undef FZ_RTT
#undef FZ_RTP
#undef FZ_RT
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// Columns whose records are held at a time: all of them, or, where these would
// pass a third of the memory that is free or holds records already, as many
// as that third takes; a larger map is then worked through in slabs of so many
// columns (microphysics and transfer of one after the other).  A record is 308
// bytes per height with two lines, 30 KB per column of 96 heights.
static int record_slab(const fz_ctx* c, int ncol) {
  const size_t per = sizeof(float) * (size_t)(c->cfg.rec + 1) * c->cfg.nz, held = c->micro_cap / per;
  size_t freeb = 0, totb = 0;
  if (held >= (size_t)ncol || hipMemGetInfo(&freeb, &totb) != hipSuccess) return ncol;
  const size_t n = std::max(held, (freeb + c->micro_cap) / 3 / per);
  return (int)std::max<size_t>(1, std::min<size_t>(n, (size_t)ncol));
}

static int ensure_records(fz_ctx* c, int slab) {
  return ensure(c, &c->d_micro, &c->micro_cap, sizeof(float) * (size_t)(c->cfg.rec + 1) * c->cfg.nz * slab);
}

// Microphysics of columns cbeg .. cend - 1, tile by tile; status[ncol] receives each
// column's FZ_E* code (the caller's array, or the context's own).  With
// hydro, Pg is first re-integrated from the top (forward.f90:891-906) and the
// EOS takes N_H and n_e from that integration; with physics == false only the
// hydrostatic integration runs (fz_hydrostatic_dev).
// Microphysics tile when none is set: the electron-density fixed point is
// sequential in height, a few lanes per column, so a tile should hold as many
// columns as memory allows (up to a quarter of the free memory, at most
// 64 GiB, for the Saha factors and the EOS buffers of every column).
static int auto_mtile(fz_ctx* c, bool hydro) {
  size_t freeb = 0, totb = 0;
  if (hipMemGetInfo(&freeb, &totb) != hipSuccess) return 16384;
  const size_t per_col = sizeof(double) * (size_t)c->cfg.nz * (FZ_NELEM * 4 * (hydro ? 2 : 1) + 2 + 8);
  // what this context already holds for the tile counts as available
  const size_t held = c->sbuf_cap + c->eosb_cap + c->derb_cap + c->smid_cap;
  const size_t budget = std::min((freeb + held) / 4, (size_t)64 << 30);
  const size_t m = budget / per_col;
  return (int)std::max<size_t>(4096, std::min<size_t>(m, 1 << 20));
}

// Grid of the Saha kernels over n (height, column) pairs: the 92 elements are
// shared out over up to 46 workgroups where the pairs alone do not give every
// SIMD two waves (one workgroup per pair block takes 80 us for a single
// column, the partition functions of all elements being a chain).
static dim3 saha_grid(long n) {
  const unsigned nb = (unsigned)((n + 255) / 256);
  return dim3(nb, std::max(1u, std::min(46u, 512u / nb)));
}

// Lanes per column of the fixed-point kernels for a tile of n columns: as
// many as keep about one wave per SIMD (1024), since a column's heights are a
// chain and only more columns or more lanes fill the card; beyond, 16, whose
// issue per column is lowest without spilling (8 lanes hold 12 elements each:
// 262 registers).  64 heights, hydrostatic integration / forward without
// response functions, ms:
//   columns   64 lanes      32 lanes      16 lanes
//      1024   0.57 / 0.54   0.59 / 0.54   0.70 / 0.58
//      2048   0.88 / 0.65   0.68 / 0.60   0.79 / 0.65
//      4096   1.49 / 0.95   1.09 / 0.83   0.98 / 0.82
//     16384   5.76 / 3.60   3.88 / 2.33   3.26 / 2.07
static int rho_lanes(int n) { return n <= 1024 ? 64 : n <= 3072 ? 32 : 16; }

// the second stream and n ordering events of the overlapped forward
static int ensure_aux(fz_ctx* c, int n) {
  if (!c->aux) HIPCHK(c, hipStreamCreateWithFlags(&c->aux, hipStreamNonBlocking));
  while ((int)c->tev.size() < n) {
    hipEvent_t e;
    HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    c->tev.push_back(e);
  }
  return FZ_OK;
}

static int run_micro(fz_ctx* c, int ncol, float* d_atm, int32_t** status, bool der, bool hydro, bool physics,
                     hipStream_t st, int cbeg, int cend, int rcol0, int rncol) {
  const int nz = c->cfg.nz;
  int32_t* stv = *status;
  if (!stv) {
    int r = ensure(c, &c->d_stat, &c->stat_cap, sizeof(int32_t) * (size_t)ncol);
    if (r) return r;
    stv = (int32_t*)c->d_stat;
    *status = stv;
  }
  const int mt = std::min(c->mtile > 0 ? c->mtile : auto_mtile(c, hydro), ncol);
  int r = ensure(c, &c->d_sbuf, &c->sbuf_cap, sizeof(double) * (size_t)nz * FZ_NELEM * 4 * mt);
  if (r) return r;
  r = ensure(c, &c->d_eosb, &c->eosb_cap, sizeof(double) * (size_t)2 * nz * mt);
  if (r) return r;
  if (der && physics) {
    r = ensure(c, &c->d_derb, &c->derb_cap, sizeof(double) * (size_t)8 * nz * mt);
    if (r) return r;
  }
  if (hydro) {
    r = ensure(c, &c->d_smid, &c->smid_cap, sizeof(double) * (size_t)(nz - 1) * FZ_NELEM * 4 * mt);
    if (r) return r;
  }
  for (int c0 = cbeg; c0 < cend; c0 += mt) {
    MicroTile a;
    a.ncol = ncol;
    a.col0 = c0;
    a.ntile = std::min(mt, cend - c0);
    a.der = (der && physics) ? 1 : 0;
    a.rcol0 = rcol0;
    a.rncol = rncol;
    a.atm = d_atm;
    a.micro = c->d_micro;
    a.sbuf = (double*)c->d_sbuf;
    a.eos = physics ? (double*)c->d_eosb : nullptr;
    a.deriv = (der && physics) ? (double*)c->d_derb : nullptr;
    a.status = stv;
    a.pop = c->pop_on ? c->d_pop : nullptr;
    const long nkt = (long)nz * a.ntile;
    if (a.der)
      hipLaunchKernelGGL(saha_kernel<true>, saha_grid(nkt), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL(saha_kernel<false>, saha_grid(nkt), dim3(256), 0, st, a);
    if (hydro) {
      const long nmt = (long)(nz - 1) * a.ntile;
      hipLaunchKernelGGL(saha_mid_kernel, saha_grid(nmt), dim3(256), 0, st, a, (double*)c->d_smid);
    }
    const int gl = rho_lanes(a.ntile);
    const dim3 gr((unsigned)(((long)a.ntile * gl + RHO_BLOCK - 1) / RHO_BLOCK)), gb(RHO_BLOCK);
    const double* sm = (const double*)c->d_smid;
    if (hydro) {
      if (gl == 16) hipLaunchKernelGGL(he_rk4_group_kernel<16>, gr, gb, 0, st, a, sm);
      else if (gl == 32) hipLaunchKernelGGL(he_rk4_group_kernel<32>, gr, gb, 0, st, a, sm);
      else hipLaunchKernelGGL(he_rk4_group_kernel<64>, gr, gb, 0, st, a, sm);
    } else {
      if (gl == 16) hipLaunchKernelGGL(rho_group_kernel<16>, gr, gb, 0, st, a);
      else if (gl == 32) hipLaunchKernelGGL(rho_group_kernel<32>, gr, gb, 0, st, a);
      else hipLaunchKernelGGL(rho_group_kernel<64>, gr, gb, 0, st, a);
    }
    if (physics) {
      if (a.der) hipLaunchKernelGGL(deriv_kernel, dim3((unsigned)((nkt + 255) / 256)), dim3(256), 0, st, a);
      hipLaunchKernelGGL(opac_kernel, dim3((unsigned)((nkt + 255) / 256)), dim3(256), 0, st, a);
      hipLaunchKernelGGL(tau_kernel, dim3((a.ntile + 63) / 64), dim3(64), 0, st, a);
    }
    HIPCHK(c, hipGetLastError());
  }
  return FZ_OK;
}

int fz_set_hydrostatic(fz_ctx* c, int on) {
  if (!c) return FZ_EARG;
  c->hydro = on != 0;
  return FZ_OK;
}

int fz_set_microturbulence(fz_ctx* c, double xi_cm_s) {
  if (!c || !std::isfinite(xi_cm_s) || xi_cm_s < 0.0 || xi_cm_s > 1.0e7) return FZ_EARG;
  c->xi = xi_cm_s;
  if (!c->configured) return FZ_OK;
  double matom[FZ_NELEM];
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMemcpyFromSymbol(matom, HIP_SYMBOL(fz_matom), sizeof(matom)));
  set_xi(c->cfg, matom, xi_cm_s);
  HIPCHK(c, hipMemcpyToSymbol(HIP_SYMBOL(c_cfg), &c->cfg, sizeof(Cfg)));
  if (c->device < 64) g_owner[c->device] = c;
  return FZ_OK;
}

int fz_set_tile(fz_ctx* c, int tile, int block) {
  if (!c || tile < 1 || block < 64 || block > 1024 || block % 64) return FZ_EARG;
  c->tile = tile;
  c->block = block;
  return FZ_OK;
}

}  // extern "C"

// FORWARD3D on device data; d_full (or null): the Stokes vector after every
// height, [ncol][nz][4][numw] (FULL_STOKES)
static int forward_impl(fz_ctx* c, int ncol, float* d_atm, int rf_mode, float* d_stokes, float* d_jac,
                        float* d_full, int32_t* d_status, void* stream) {
  if (!c || !c->configured || ncol < 1 || !d_atm || !d_stokes) return FZ_EARG;
  if (d_full && c->win_on) return set_err(c, FZ_EARG, "per-pixel windows: no full Stokes output");
  if (rf_mode != FZ_RF_NONE && !d_jac) return set_err(c, FZ_EARG, "jacobian output missing");
  if (rf_mode < 0 || rf_mode > 3) return FZ_EARG;
  if (c->win_on) {
    if (ncol != c->win_ncol) return set_err(c, FZ_EARG, "column count differs from fz_set_windows");
    if (rf_mode != FZ_RF_NONE)
      return set_err(c, FZ_EARG, "per-pixel windows: response functions come through the inversion only");
    if (c->cfg.lsf_on) return set_err(c, FZ_ECONFIG, "per-pixel windows and an LSF together are not supported");
  }
  const Cfg& g = c->cfg;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  int r = upload_cfg(c);
  if (r) return r;
  // columns per radiative-transfer launch: the configured tile, fewer where
  // its scratch would pass 48 GiB; whole tiles to a slab of records
  const size_t per_col = sizeof(float) * rt_scratch_per_lane(c, rf_mode) * g.numw;
  int slab = record_slab(c, ncol), tile = std::min(rt_tile(c, ncol), slab);
  if (per_col) tile = (int)std::max<size_t>(1, std::min<size_t>((size_t)tile, ((size_t)48 << 30) / per_col));
  if (slab < ncol) slab = slab / tile * tile;
  r = ensure_records(c, slab);
  if (r) return r;
  if (rf_mode != FZ_RF_NONE) {
    r = ensure(c, &c->d_scratch, &c->scratch_cap, per_col * tile);
    if (r) return r;
  }
  const int ntiles = (ncol + tile - 1) / tile;
  const bool ovl = c->overlap && ntiles > 1 && !c->win_on && slab == ncol;
  if (c->prof) HIPCHK(c, hipEventRecord(c->ev[0], st));
  if (ovl) {
    // the microphysics of RT tile i+1 runs on the second stream while tile
    // i's radiative transfer runs on st; tile i's transfer waits for its own
    // microphysics only (the micro scratch is reused tile after tile on the
    // second stream, and the tiles' columns are disjoint)
    r = ensure_aux(c, ntiles + 1);
    if (r) return r;
    if (!d_status) {
      r = ensure(c, &c->d_stat, &c->stat_cap, sizeof(int32_t) * (size_t)ncol);
      if (r) return r;
      d_status = (int32_t*)c->d_stat;
    }
    HIPCHK(c, hipEventRecord(c->tev[0], st));
    HIPCHK(c, hipStreamWaitEvent(c->aux, c->tev[0], 0));
    for (int i = 0; i < ntiles; ++i) {
      r = run_micro(c, ncol, d_atm, &d_status, rf_mode != FZ_RF_NONE, c->hydro, true, c->aux, i * tile,
                    std::min(ncol, (i + 1) * tile), 0, ncol);
      if (r) return r;
      HIPCHK(c, hipEventRecord(c->tev[i + 1], c->aux));
    }
  }
  c->rt_launches = 0;
  for (int s0 = 0; s0 < ncol; s0 += slab) {
    const int s1 = std::min(ncol, s0 + slab);
    if (!ovl) {
      r = run_micro(c, ncol, d_atm, &d_status, rf_mode != FZ_RF_NONE, c->hydro, true, st, s0, s1, s0, slab);
      if (r) return r;
    } else {
      HIPCHK(c, hipStreamWaitEvent(st, c->tev[1], 0));
    }
    // with the overlap, "microphysics" is the first tile's, which nothing
    // hides, and with several slabs the first one's
    if (c->prof && s0 == 0) HIPCHK(c, hipEventRecord(c->ev[1], st));
    for (int c0 = s0; c0 < s1; c0 += tile) {
      if (ovl && c0 > 0) HIPCHK(c, hipStreamWaitEvent(st, c->tev[c0 / tile + 1], 0));
      RtArgs a;
      a.ncol = ncol;
      a.col0 = c0;
      a.ntile = std::min(tile, s1 - c0);
      a.rcol0 = s0;
      a.rncol = slab;
      a.atm = d_atm;
      a.micro = c->d_micro;
      a.gain = c->d_gain;
      a.status = d_status;
      a.stokes = d_stokes;
      a.jac = d_jac;
      a.jcol0 = 0;
      a.scratch = c->d_scratch;
      a.items = nullptr;
      a.poff = nullptr;
      a.fs = d_full;
      int nit = 0;
      if (c->win_on) {
        a.items = c->d_items + c->h_item_first[c0];
        a.poff = c->d_poff;
        nit = c->h_item_first[c0 + a.ntile] - c->h_item_first[c0];
      }
      r = launch_rt(c, rf_mode, a, st, nit);
      if (r) return r;
      HIPCHK(c, hipGetLastError());
      c->rt_launches++;
    }
  }
  r = run_lsf(c, d_stokes, (long)ncol * 4, st);
  if (r) return r;
  if (rf_mode != FZ_RF_NONE) {
    r = run_lsf(c, d_jac, (long)ncol * rf_nparam(rf_mode) * g.nz * 4, st);
    if (r) return r;
  }
  if (c->prof) HIPCHK(c, hipEventRecord(c->ev[2], st));
  return FZ_OK;
}

extern "C" {

int fz_forward_dev(fz_ctx* c, int ncol, float* d_atm, int rf_mode, float* d_stokes, float* d_jac, int32_t* d_status,
                   void* stream) {
  return forward_impl(c, ncol, d_atm, rf_mode, d_stokes, d_jac, nullptr, d_status, stream);
}

int fz_forward_full_dev(fz_ctx* c, int ncol, float* d_atm, int rf_mode, float* d_stokes, float* d_jac, float* d_full,
                        int32_t* d_status, void* stream) {
  if (!d_full) return FZ_EARG;
  return forward_impl(c, ncol, d_atm, rf_mode, d_stokes, d_jac, d_full, d_status, stream);
}

int fz_line_tau_dev(fz_ctx* c, int ncol, float* d_atm, float* d_tau, int32_t* d_status, void* stream) {
  if (!c || !c->configured || ncol < 1 || !d_atm || !d_tau) return FZ_EARG;
  if (c->win_on) return set_err(c, FZ_EARG, "per-pixel windows: no line optical depth");
  const Cfg& g = c->cfg;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  int r = upload_cfg(c);
  if (r) return r;
  const int slab = record_slab(c, ncol);
  r = ensure_records(c, slab);
  if (r) return r;
  for (int s0 = 0; s0 < ncol; s0 += slab) {
    RtArgs a = {};
    a.ncol = ncol;
    a.col0 = a.rcol0 = s0;
    a.ntile = std::min(slab, ncol - s0);
    a.rncol = slab;
    r = run_micro(c, ncol, d_atm, &d_status, false, c->hydro, true, st, s0, s0 + a.ntile, s0, slab);
    if (r) return r;
    a.atm = d_atm;
    a.micro = c->d_micro;
    a.gain = c->d_gain;
    a.status = d_status;
    const long n = (long)a.ntile * g.numw;
    hipLaunchKernelGGL(taulin_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, d_tau);
    HIPCHK(c, hipGetLastError());
  }
  return FZ_OK;
}

int fz_set_overlap(fz_ctx* c, int on) {
  if (!c) return FZ_EARG;
  c->overlap = on != 0;
  return FZ_OK;
}

int fz_set_auto_weights(fz_ctx* c, int on) {
  if (!c) return FZ_EARG;
  c->autow = on != 0;
  return FZ_OK;
}

// SET_WEIGHTS3D's per-pixel work (get_dmodel.f90:2051-2170): SET_WEIGHTS1D
// (:2191-2224) on the pixel's observed row, WSTK = those weights in REAL(4),
// then SET_ISIGMAP (:356-373).  One lane per pixel; the row is nstk blocks of
// numw values, the blocks of the inverted Stokes parameters in I, Q, U, V
// order.  STDDEV (:2228-2251): mean as the sum of x_i / n, then the n - 1
// variance, both in sequence order.
__global__ void auto_weights_kernel(int ncol, int numw, int inv_mask, double isigma, const double* __restrict__ obs,
                                    double* __restrict__ isig) {
  const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= ncol) return;
  int nstk = 0;
  for (int s = 0; s < 4; ++s) nstk += (inv_mask >> s) & 1;
  const int nf = nstk * numw;
  const double* o = obs + col * nf;
  double w[4], minw = 1.0e60;
  const double dn = (double)numw;
  for (int s = 0, b = 0; s < 4; ++s) {
    w[s] = 0.0;
    if (!((inv_mask >> s) & 1)) continue;
    const double* x = o + (long)b * numw;
    double mn = 0.0;
    for (int i = 0; i < numw; ++i) mn += x[i] / dn;
    double v = 0.0;
    for (int i = 0; i < numw; ++i) v += (x[i] - mn) * (x[i] - mn);
    const double sd = sqrt(v / (dn - 1.0));
    w[s] = sqrt(1.0 / (sd * sd));
    if (w[s] < minw) minw = w[s];
    ++b;
  }
  minw *= 10.0;
  double ss = 0.0;
  for (int s = 0; s < 4; ++s) {
    if (w[s] > minw) w[s] = minw;
    ss += w[s] * w[s];
  }
  const double nrm = sqrt(ss) / sqrt((double)nstk);
  double* out = isig + col * nf;
  for (int s = 0, b = 0; s < 4; ++s) {
    if (!((inv_mask >> s) & 1)) continue;
    const float ws = (float)(w[s] / nrm);
    const double v = (double)(ws * ws) / (isigma * isigma);
    for (int i = 0; i < numw; ++i) out[(long)b * numw + i] = v;
    ++b;
  }
}

int fz_auto_weights_dev(fz_ctx* c, int ncol, const double* d_obs, const int32_t* invstk, float noise,
                        double* d_isigmap, void* stream) {
  if (!c || !c->configured || ncol < 1 || !d_obs || !invstk || !d_isigmap) return FZ_EARG;
  if (c->win_on) return set_err(c, FZ_ECONFIG, "automatic Stokes weights take the dense spectral grid");
  if (c->cfg.numw < 2) return set_err(c, FZ_ECONFIG, "automatic Stokes weights need two wavelengths or more");
  int mask = 0;
  for (int s = 0; s < 4; ++s) mask |= invstk[s] ? 1 << s : 0;
  if (!mask) return set_err(c, FZ_ECONFIG, "no Stokes parameter inverted");
  HIPCHK(c, hipSetDevice(c->device));
  const double isigma = (double)(noise > 0 ? noise : 4.0e-3f);
  hipLaunchKernelGGL(auto_weights_kernel, dim3((ncol + 255) / 256), dim3(256), 0, (hipStream_t)stream, ncol,
                     c->cfg.numw, mask, isigma, d_obs, d_isigmap);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_set_profiling(fz_ctx* c, int on) {
  if (!c) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  if (on && !c->ev[0])
    for (int i = 0; i < 3; ++i) HIPCHK(c, hipEventCreate(&c->ev[i]));
  c->prof = on != 0;
  return FZ_OK;
}

int fz_last_timing(fz_ctx* c, float* micro_ms, float* rt_ms, int* launches) {
  if (!c || !c->prof) return FZ_EARG;
  HIPCHK(c, hipEventSynchronize(c->ev[2]));
  float a = 0.f, b = 0.f;
  HIPCHK(c, hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
  HIPCHK(c, hipEventElapsedTime(&b, c->ev[1], c->ev[2]));
  if (micro_ms) *micro_ms = a;
  if (rt_ms) *rt_ms = b;
  if (launches) *launches = c->rt_launches;
  return FZ_OK;
}

int fz_autotune(fz_ctx* c, int ncol, float* d_atm, int rf_mode, float* d_stokes, float* d_jac, int32_t* d_status,
                void* stream, int* tile_out, int* mtile_out) {
  if (!c || !c->configured || ncol < 1 || !d_atm || !d_stokes) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  const bool prof = c->prof;
  const int mtile0 = c->mtile, tile0 = c->tile;
  // on a failed trial the context keeps the caller's tiles and profiling switch
  auto fail = [&](int code) {
    c->mtile = mtile0;
    c->tile = tile0;
    c->prof = prof;
    return code;
  };
  int r = fz_set_profiling(c, 1);
  if (r) return r;
  const int nz = c->cfg.nz, numw = c->cfg.numw;
  size_t freeb = 0, totb = 0;
  if (hipMemGetInfo(&freeb, &totb) != hipSuccess) return fail(set_err(c, FZ_EHIP, "hipMemGetInfo failed"));
  const size_t budget = freeb / 3;
  // microphysics tile: Saha factors, EOS and derivative buffers per column
  const size_t per_mcol = sizeof(double) * (size_t)nz * (FZ_NELEM * 4 * (c->hydro ? 2 : 1) + 2 + 8);
  // radiative-transfer tile: the Stokes scratch per column
  const size_t per_rcol = sizeof(float) * rt_scratch_per_lane(c, rf_mode) * numw;
  const int mcand[] = {4096, 8192, 16384, 32768, 65536, 131072, 262144};
  const int rcand[] = {2048, 4096, 8192, 16384, 32768};
  float best = 1e30f;
  int best_m = c->mtile, best_t = c->tile;
  for (int m : mcand) {
    if (m > 2 * ncol && m != mcand[0]) break;
    if ((size_t)std::min(m, ncol) * per_mcol > budget) break;
    c->mtile = m;
    r = fz_forward_dev(c, ncol, d_atm, rf_mode, d_stokes, d_jac, d_status, stream);
    if (r) return fail(r);
    float ms = 0.f;
    r = fz_last_timing(c, &ms, nullptr, nullptr);
    if (r) return fail(r);
    if (ms < best) {
      best = ms;
      best_m = m;
    }
  }
  c->mtile = best_m;
  best = 1e30f;
  if (rf_mode != FZ_RF_NONE) {
    for (int t : rcand) {
      if (t > 2 * ncol && t != rcand[0]) break;
      if ((size_t)std::min(t, ncol) * per_rcol > budget) break;
      c->tile = t;
      r = fz_forward_dev(c, ncol, d_atm, rf_mode, d_stokes, d_jac, d_status, stream);
      if (r) return fail(r);
      float ms = 0.f;
      r = fz_last_timing(c, nullptr, &ms, nullptr);
      if (r) return fail(r);
      if (ms < best) {
        best = ms;
        best_t = t;
      }
    }
  }
  c->tile = best_t;
  // release what the larger trials left behind; the next call allocates its size
  if (c->d_sbuf) (void)hipFree(c->d_sbuf);
  if (c->d_eosb) (void)hipFree(c->d_eosb);
  if (c->d_derb) (void)hipFree(c->d_derb);
  if (c->d_smid) (void)hipFree(c->d_smid);
  if (c->d_scratch) (void)hipFree(c->d_scratch);
  c->d_sbuf = c->d_eosb = c->d_derb = c->d_smid = c->d_scratch = nullptr;
  c->sbuf_cap = c->eosb_cap = c->derb_cap = c->smid_cap = c->scratch_cap = 0;
  c->prof = prof;
  if (tile_out) *tile_out = c->tile;
  if (mtile_out) *mtile_out = c->mtile;
  return FZ_OK;
}

int fz_hydrostatic_dev(fz_ctx* c, int ncol, float* d_atm, int32_t* d_status, void* stream) {
  if (!c || !c->configured || ncol < 1 || !d_atm) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  int r = upload_cfg(c);
  if (r) return r;
  r = run_micro(c, ncol, d_atm, &d_status, false, true, false, (hipStream_t)stream, 0, ncol, 0, ncol);
  return r;
}

int fz_forward3d(fz_ctx* c, int nx, int ny, float* tem3d, float* pg3d, float* rho3d, float* pel3d, float* mw3d,
                 const float* bx3d, const float* by3d, const float* bz3d, const float* vx3d, const float* vy3d,
                 const float* vz3d, float* tau3d5, const int32_t* am_i_done, int rf_mode, double* syn3d, float* dsyn) {
  if (!c || !c->configured || nx < 1 || ny < 1 || !syn3d) return FZ_EARG;
  const Cfg& g = c->cfg;
  const int nz = g.nz, numw = g.numw;
  const int np = rf_nparam(rf_mode);
  if (np && !dsyn) return FZ_EARG;
  // columns still to be computed (AM_I_DONE == 0, forward.f90:120-140)
  std::vector<int> cols;
  for (int x = 0; x < nx; ++x)
    for (int y = 0; y < ny; ++y)
      if (!am_i_done || am_i_done[y + (size_t)ny * x] == 0) cols.push_back(y + ny * x);
  const int n = (int)cols.size();
  if (n == 0) return FZ_OK;
  const float* cubes[NATM] = {tem3d, pg3d, rho3d, pel3d, mw3d, bx3d, by3d, bz3d, vx3d, vy3d, vz3d, tau3d5};
  const size_t colbytes = sizeof(float) * nz;
  std::vector<float> h(colbytes / sizeof(float) * n);
  DevBuf b_atm, b_tmp, b_st, b_jac, b_status;
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMalloc(&b_atm.p, colbytes * NATM * n));
  HIPCHK(c, hipMalloc(&b_tmp.p, colbytes * n));
  HIPCHK(c, hipMalloc(&b_st.p, sizeof(float) * 4 * numw * n));
  HIPCHK(c, hipMalloc(&b_status.p, sizeof(int32_t) * n));
  if (np) HIPCHK(c, hipMalloc(&b_jac.p, sizeof(float) * (size_t)np * nz * 4 * numw * n));
  float *d_atm = (float*)b_atm.p, *d_tmp = (float*)b_tmp.p, *d_st = (float*)b_st.p, *d_jac = (float*)b_jac.p;
  int32_t* d_status = (int32_t*)b_status.p;
  const unsigned tb = 256, tg = (unsigned)(((long)nz * n + tb - 1) / tb);
  for (int p = 0; p < NATM; ++p) {
    for (int i = 0; i < n; ++i) memcpy(&h[(size_t)i * nz], cubes[p] + (size_t)cols[i] * nz, colbytes);
    HIPCHK(c, hipMemcpy(d_tmp, h.data(), colbytes * n, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(cube_to_soa, dim3(tg), dim3(tb), 0, 0, d_tmp, d_atm + (size_t)p * nz * n, nz, n);
  }
  int rc = fz_forward_dev(c, n, d_atm, rf_mode, d_st, d_jac, d_status, nullptr);
  if (rc == FZ_OK) {
    std::vector<int32_t> stat(n);
    HIPCHK(c, hipMemcpy(stat.data(), d_status, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    for (int i = 0; i < n && rc == FZ_OK; ++i)
      if (stat[i]) rc = set_err(c, stat[i], "column " + std::to_string(cols[i]) + " failed");
  }
  if (rc == FZ_OK) {
    // model updated in place: Pg (re-integrated with HYDROSTATIC), rho, Pe,
    // mu, log tau5 (SPLIT_MODEL3D, forward.f90:1225-1270)
    float* outs[NATM] = {nullptr, pg3d, rho3d, pel3d, mw3d, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, tau3d5};
    for (int p = 0; p < NATM; ++p) {
      if (!outs[p]) continue;
      hipLaunchKernelGGL(soa_to_cube, dim3(tg), dim3(tb), 0, 0, d_atm + (size_t)p * nz * n, d_tmp, nz, n);
      HIPCHK(c, hipMemcpy(h.data(), d_tmp, colbytes * n, hipMemcpyDeviceToHost));
      for (int i = 0; i < n; ++i) memcpy(outs[p] + (size_t)cols[i] * nz, &h[(size_t)i * nz], colbytes);
    }
    std::vector<float> st((size_t)4 * numw * n);
    HIPCHK(c, hipMemcpy(st.data(), d_st, sizeof(float) * st.size(), hipMemcpyDeviceToHost));
    const size_t nf = (size_t)4 * numw;
    for (int i = 0; i < n; ++i)
      for (size_t f = 0; f < nf; ++f) syn3d[(size_t)cols[i] * nf + f] = (double)st[(size_t)i * nf + f];
    if (np) {
      const size_t per = (size_t)np * nz * 4 * numw;
      std::vector<float> jh(per);
      for (int i = 0; i < n; ++i) {
        HIPCHK(c, hipMemcpy(jh.data(), d_jac + (size_t)i * per, sizeof(float) * per, hipMemcpyDeviceToHost));
        // device [np][nz][4][numw] -> DSYN(NFREQ=4*numw, IFREEP=np*nz): same order
        memcpy(dsyn + (size_t)cols[i] * per, jh.data(), sizeof(float) * per);
      }
    }
  }
  return rc;
}

int fz_malloc(fz_ctx* c, void** p, uint64_t bytes) {
  if (!c || !p) return FZ_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  if (hipMalloc(p, bytes) != hipSuccess) return set_err(c, FZ_ENOMEM, "hipMalloc failed");
  return FZ_OK;
}
int fz_free(fz_ctx* c, void* p) {
  if (!c) return FZ_EARG;
  HIPCHK(c, hipFree(p));
  return FZ_OK;
}
int fz_memcpy_h2d(fz_ctx* c, void* d, const void* s, uint64_t b) {
  HIPCHK(c, hipMemcpy(d, s, b, hipMemcpyHostToDevice));
  return FZ_OK;
}
int fz_memcpy_d2h(fz_ctx* c, void* d, const void* s, uint64_t b) {
  HIPCHK(c, hipMemcpy(d, s, b, hipMemcpyDeviceToHost));
  return FZ_OK;
}
int fz_synchronize(fz_ctx* c) {
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipDeviceSynchronize());
  return FZ_OK;
}

// ------------------------------------------------------------------ inversion

// GET_POSITIONS + GET_INT_COEFS (get_dmodel.f90:463-477, 563-644)
int fz_int_coefs(int nz, int nj, double* coefs) {
  if (!coefs || nz < 1 || nj < 1 || nj > nz) return FZ_EARG;
  std::fill(coefs, coefs + (size_t)nz * nj, 0.0);
  if (nj == 1) {
    for (int k = 0; k < nz; ++k) coefs[k] = 1.0;
    return FZ_OK;
  }
  if (nj == nz) {
    for (int k = 0; k < nz; ++k) coefs[(size_t)k * nz + k] = 1.0;
    return FZ_OK;
  }
  std::vector<double> pos(nj);
  const double step = (double)(nz - 1) / (double)(nj - 1);
  for (int j = 0; j < nj; ++j) pos[j] = ((double)(j + 1) - 1.0) * step + 1.0;
  for (int j = 0; j < nj; ++j) {
    const double lo = pos[std::max(j - 1, 0)], hi = pos[std::min(j + 1, nj - 1)], mid = pos[j];
    for (int i = 1; i <= nz; ++i) {
      const double x = (double)i;
      if (x < lo || x > hi) continue;
      double v;
      if (x == mid) v = 1.0;
      else if (x < mid) v = (1.0 - 0.0) / (mid - lo) * (x - lo);
      else v = (1.0 - 0.0) / (hi - mid) * (hi - x);
      coefs[(size_t)j * nz + (i - 1)] = v;
    }
  }
  return FZ_OK;
}

int fz_set_inversion(fz_ctx* c, const fz_inversion* inv, int* ifreep, int* nfreq) {
  if (!c || !inv) return FZ_EARG;
  if (!c->configured) return set_err(c, FZ_ECONFIG, "fz_configure first");
  const int nz = c->cfg.nz, numw = c->cfg.numw;
  LmArgs& L = c->lm;
  c->inv_set = false;   // until every table is there
  L = LmArgs();
  L.nz = nz;
  L.numw = numw;
  int nstk = 0;
  for (int s = 0; s < 4; ++s)
    if (inv->invstk[s]) L.rowstk[nstk++] = s;
  if (nstk == 0) return set_err(c, FZ_ECONFIG, "no Stokes parameter inverted");
  L.nfreq = nstk * numw;
  static const int mcol[8] = {A_T, A_PG, A_RHO, A_BX, A_BY, A_BZ, A_VZ, A_PG};
  std::vector<double> coefs;
  c->slot_of.clear();
  int np = 0, npar = 0;
  for (int p = 0; p < 8; ++p) {
    if (!inv->atmpar[p]) continue;
    const int nj = inv->nodes[p];
    if (nj < 1 || nj > nz) return set_err(c, FZ_ECONFIG, "nodes must be in 1..nz");
    if (np + nj > LM_MAXNP_BIG) return set_err(c, FZ_ECONFIG, "more than 2048 free parameters");
    L.par[npar] = p;
    L.slot[npar] = p;  // Cartesian slots: T|Pg, Pg|T, rho|T, Bx, By, Bz, v_z, P0
    L.mcol[npar] = mcol[p];
    L.j0[npar] = np;
    L.nj[npar] = nj;
    std::vector<double> cf((size_t)nz * nj);
    fz_int_coefs(nz, nj, cf.data());
    coefs.insert(coefs.end(), cf.begin(), cf.end());
    for (int j = 0; j < nj; ++j) c->slot_of.push_back(p);
    np += nj;
    ++npar;
  }
  if (np == 0) return set_err(c, FZ_ECONFIG, "no parameter inverted");
  L.np = np;
  L.nparam = npar;
  // the model columns that a step holds: the inverted ones, then log tau5
  for (int p = 0; p < NATM; ++p) L.rowslot[p] = -1;
  L.nheld = 0;
  for (int ip = 0; ip < npar; ++ip) {
    if (L.rowslot[L.mcol[ip]] < 0) L.rowslot[L.mcol[ip]] = L.nheld++;
    L.mslot[ip] = L.rowslot[L.mcol[ip]];
  }
  L.rowslot[A_TAU] = L.nheld++;
  std::vector<double> colsum(np);
  c->kbeg.assign(np, 0);
  c->kend.assign(np, 0);
  for (int j = 0; j < np; ++j) {
    double w = 0.0;
    int kb = nz, ke = -1;
    for (int k = 0; k < nz; ++k) {
      const double v = coefs[(size_t)j * nz + k];
      w += v;
      if (v != 0.0) {
        kb = std::min(kb, k);
        ke = std::max(ke, k);
      }
    }
    colsum[j] = w;
    c->kbeg[j] = kb;
    c->kend[j] = ke;
  }
  L.regul = inv->regul ? 1 : 0;
  L.solver = inv->solver;
  if (L.solver != 1 && L.solver != 2) return set_err(c, FZ_ECONFIG, "solver must be 1 or 2");
  L.node_expansion = inv->node_expansion;
  if (L.node_expansion != 1 && L.node_expansion != 2) return set_err(c, FZ_ECONFIG, "node_expansion must be 1 or 2");
  for (int p = 0; p < 8; ++p) {
    L.pen_typ[p] = inv->pen_typ[p];
    L.pen_alp[p] = inv->pen_alp[p];
  }
  L.svdtol = inv->svdtol == 0.0 ? 1.0e-4 : inv->svdtol;
  L.inu = inv->inu == 0.0 ? (double)L.nfreq : inv->inu;
  L.mpert = inv->mpert == 0.0 ? 0.15 : inv->mpert;
  L.maxsteps = (double)inv->maxsteps;
  // up to LM_MAXNP free parameters the step's work arrays live in LDS;
  // beyond, in a per-pixel slice of device memory
  c->lm_big = np > LM_MAXNP;
  c->lm_lds = c->lm_big ? 0 : lm_lds_bytes(np, nz, L.regul != 0, LM_THREADS);
  c->lm_work = c->lm_big ? (lm_lds_bytes(np, nz, L.regul != 0, LM_BIG_THREADS) + 255) / 256 * 256 : 0;
  if (c->lm_lds > 160 * 1024 - 512) return set_err(c, FZ_ECONFIG, "inversion set-up exceeds the LDS of one workgroup");
  HIPCHK(c, hipSetDevice(c->device));
  // node table of the contraction: supports, Cartesian slot
  std::vector<int> node((size_t)3 * np);
  for (int j = 0; j < np; ++j) {
    node[j] = c->kbeg[j];
    node[np + j] = c->kend[j];
    node[2 * np + j] = c->slot_of[j];
  }
  // the pairwise contraction applies when every parameter's node supports
  // overlap at most pairwise and move up with the node index (the hat basis
  // of GET_INT_COEFS); its per-height table
  c->eqv_pairs = true;
  for (int ip = 0; ip < npar; ++ip)
    for (int j = L.j0[ip]; j < L.j0[ip] + L.nj[ip]; ++j) {
      const int je = L.j0[ip] + L.nj[ip] - 1;
      if (c->kbeg[j] > c->kend[j]) c->eqv_pairs = false;
      if (j + 1 <= je && (c->kbeg[j + 1] < c->kbeg[j] || c->kend[j + 1] < c->kend[j])) c->eqv_pairs = false;
      if (j + 2 <= je && c->kbeg[j + 2] <= c->kend[j]) c->eqv_pairs = false;
    }
  std::vector<int> tj;
  std::vector<double> tc;
  std::vector<NodeTab> nt;
  if (c->eqv_pairs) {
    tj.assign((size_t)npar * nz, 0);
    tc.assign((size_t)npar * nz * 2, 0.0);
    for (int ip = 0; ip < npar; ++ip) {
      const int jb = L.j0[ip], je = jb + L.nj[ip] - 1;
      int jl = jb;
      for (int k = c->kbeg[jb]; k <= c->kend[je]; ++k) {
        while (k > c->kend[jl]) ++jl;
        int w = jl;
        if (k >= c->kbeg[jl]) {
          w |= 1 << 30;
          tc[((size_t)ip * nz + k) * 2] = coefs[(size_t)jl * nz + k];
        }
        if (jl < je && k >= c->kbeg[jl + 1]) {
          w |= 1 << 29;
          tc[((size_t)ip * nz + k) * 2 + 1] = coefs[(size_t)(jl + 1) * nz + k];
        }
        tj[(size_t)ip * nz + k] = w;
      }
    }
    // the same per height for the five slots T, Bx, By, Bz, v_z
    nt.assign((size_t)nz * 5, NodeTab{0.0, 0.0, -1, 0});
    for (int ip = 0; ip < npar; ++ip) {
      const int sl = TBV_SLOT[L.par[ip]];
      if (sl < 0) continue;
      for (int k = 0; k < nz; ++k) {
        const int w = tj[(size_t)ip * nz + k];
        nt[(size_t)k * 5 + sl] = {tc[((size_t)ip * nz + k) * 2], tc[((size_t)ip * nz + k) * 2 + 1], w & 0xffff, 0};
      }
    }
  }
  // all tables with one copy into one buffer, which is kept (an allocation and a
  // copy each took 96 us for five parameters of four nodes): doubles, then integers
  std::vector<char> tab;
  auto put = [&](const void* src, size_t bytes) {
    const size_t at = tab.size();
    tab.resize(at + bytes);
    if (bytes) memcpy(tab.data() + at, src, bytes);
    return at;
  };
  const size_t o_coefs = put(coefs.data(), sizeof(double) * coefs.size());
  const size_t o_colsum = put(colsum.data(), sizeof(double) * np);
  const size_t o_tc = put(tc.data(), sizeof(double) * tc.size());
  const size_t o_nt = put(nt.data(), sizeof(NodeTab) * nt.size());
  const size_t o_node = put(node.data(), sizeof(int) * node.size());
  const size_t o_tj = put(tj.data(), sizeof(int) * tj.size());
  HIPCHK(c, hipDeviceSynchronize());   // work with the tables of another set-up may be running
  const int re = ensure(c, &c->d_invtab, &c->invtab_cap, tab.size());
  if (re) return re;
  HIPCHK(c, hipMemcpy(c->d_invtab, tab.data(), tab.size(), hipMemcpyHostToDevice));
  char* base = reinterpret_cast<char*>(c->d_invtab);
  c->d_coefs = reinterpret_cast<double*>(base + o_coefs);
  c->d_colsum = reinterpret_cast<double*>(base + o_colsum);
  c->d_eqvtab_c = reinterpret_cast<double*>(base + o_tc);
  c->d_nodetab = reinterpret_cast<NodeTab*>(base + o_nt);
  c->d_eqvnode = reinterpret_cast<int*>(base + o_node);
  c->d_eqvtab_j = reinterpret_cast<int*>(base + o_tj);
  if (!c->lm_big)
    HIPCHK(c, hipFuncSetAttribute((const void*)lm_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)c->lm_lds));
  L.coefs = c->d_coefs;
  L.colsum = c->d_colsum;
  c->inv_set = true;
  c->lm_p0 = inv->atmpar[7] != 0;
  c->lm_pr = inv->atmpar[1] != 0 || inv->atmpar[2] != 0;
  if (ifreep) *ifreep = np;
  if (nfreq) *nfreq = L.nfreq;
  return FZ_OK;
}

int fz_forward_nodes_dev(fz_ctx* c, int ncol, float* d_atm, float* d_stokes, float* d_eqv, int32_t* d_status,
                         void* stream) {
  if (!c || !c->configured || ncol < 1 || !d_atm || !d_stokes || !d_eqv) return FZ_EARG;
  if (!c->inv_set) return set_err(c, FZ_ECONFIG, "fz_set_inversion first");
  if (c->lm.nz != c->cfg.nz || c->lm.numw != c->cfg.numw)
    return set_err(c, FZ_ECONFIG, "heights or wavelengths changed since fz_set_inversion");
  if (c->win_on) {
    if (ncol != c->win_ncol) return set_err(c, FZ_EARG, "column count differs from fz_set_windows");
    if (c->cfg.lsf_on) return set_err(c, FZ_ECONFIG, "per-pixel windows and an LSF together are not supported");
  }
  const Cfg& g = c->cfg;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  int r = upload_cfg(c);
  if (r) return r;
  // the P0 slot is synthesised only when P0 is inverted; the Pg and rho
  // slots only when they are inverted or feed another response (P0, HYDROSTATIC)
  const bool p0 = c->lm_p0;
  // with the five slots T, Bx, By, Bz, v_z the transfer contracts them itself
  const bool tbv = !p0 && !c->lm_pr && !c->hydro && c->eqv_pairs;
  const int rf = p0 ? FZ_RF_CARTESIAN_P0 : (tbv ? RF_CART_TBV : FZ_RF_CARTESIAN);
  const int nslot = tbv ? 0 : rf_nparam(rf);
  // columns per tile: the configured tile, fewer where one tile's response
  // functions and scratch would pass 24 GiB; sized by the widest tile (the
  // wavelengths of its columns: ragged with per-pixel windows)
  const size_t per_w = sizeof(float) * ((size_t)nslot * g.nz * 4 + rt_scratch_per_lane(c, rf));
  const size_t budget = (size_t)24 << 30;
  int slab = record_slab(c, ncol), tile = std::min(rt_tile(c, ncol), slab);
  size_t wmax = 0;
  for (;;) {
    wmax = 0;
    for (int c0 = 0; c0 < ncol; c0 += tile) {
      const int n = std::min(tile, ncol - c0);
      wmax = std::max(wmax, c->win_on ? (size_t)(c->h_poff[c0 + n] - c->h_poff[c0]) : (size_t)n * g.numw);
    }
    if (wmax * per_w <= budget || tile == 1) break;
    tile = std::max(1, (int)((double)tile * (double)budget / (double)(wmax * per_w)));
  }
  if (slab < ncol) slab = slab / tile * tile;
  r = ensure_records(c, slab);
  if (r) return r;
  r = ensure(c, &c->d_scratch, &c->scratch_cap, sizeof(float) * rt_scratch_per_lane(c, rf) * wmax);
  if (r) return r;
  if (nslot) {
    r = ensure(c, &c->d_jtile, &c->jtile_cap, sizeof(float) * (size_t)nslot * g.nz * 4 * wmax);
    if (r) return r;
  }
  if (c->prof) HIPCHK(c, hipEventRecord(c->ev[0], st));
  c->rt_launches = 0;
  EqvArgs e;
  e.nz = g.nz;
  e.numw = g.numw;
  e.nfreq = c->lm.nfreq;
  e.np = c->lm.np;
  e.nstk = c->lm.nfreq / g.numw;
  e.nslot = nslot;
  for (int s = 0; s < 4; ++s) e.rowstk[s] = c->lm.rowstk[s];
  const int np = e.np;
  e.kbeg = c->d_eqvnode;
  e.kend = c->d_eqvnode + np;
  e.slot_of = c->d_eqvnode + 2 * np;
  e.nparam = c->lm.nparam;
  for (int ip = 0; ip < e.nparam; ++ip) {
    e.j0[ip] = c->lm.j0[ip];
    e.nj[ip] = c->lm.nj[ip];
  }
  e.pairs = c->eqv_pairs ? 1 : 0;
  e.tab_j = c->d_eqvtab_j;
  e.tab_c = c->d_eqvtab_c;
  e.coefs = c->d_coefs;
  e.eqv = d_eqv;
  e.poff = c->win_on ? c->d_poff : nullptr;
  NodeArgs nd;
  nd.eqv = d_eqv;
  nd.np = np;
  nd.nstk = e.nstk;
  for (int s = 0; s < 4; ++s) nd.blk[s] = -1;
  for (int b = 0; b < e.nstk; ++b) nd.blk[e.rowstk[b]] = b;
  for (int p = 0; p < 5; ++p) nd.last[p] = -1;
  for (int ip = 0; ip < e.nparam; ++ip)
    if (tbv) nd.last[TBV_SLOT[c->lm.par[ip]]] = e.j0[ip] + e.nj[ip] - 1;
  for (int c0 = 0, s0 = 0; c0 < ncol; c0 += tile) {
    if (c0 % slab == 0) {
      s0 = c0;
      r = run_micro(c, ncol, d_atm, &d_status, true, c->hydro, true, st, s0, std::min(ncol, s0 + slab), s0, slab);
      if (r) return r;
      if (c->prof && s0 == 0) HIPCHK(c, hipEventRecord(c->ev[1], st));
    }
    RtArgs a;
    a.ncol = ncol;
    a.col0 = c0;
    a.ntile = std::min(tile, ncol - c0);
    a.rcol0 = s0;
    a.rncol = slab;
    a.atm = d_atm;
    a.micro = c->d_micro;
    a.gain = c->d_gain;
    a.status = d_status;
    a.stokes = d_stokes;
    a.jac = c->d_jtile;
    a.jcol0 = c0;
    a.scratch = c->d_scratch;
    a.items = nullptr;
    a.poff = nullptr;
    a.fs = nullptr;
    int nit = 0;
    if (c->win_on) {
      a.items = c->d_items + c->h_item_first[c0];
      a.poff = c->d_poff;
      nit = c->h_item_first[c0 + a.ntile] - c->h_item_first[c0];
    }
    r = launch_rt(c, rf, a, st, nit, tbv ? &nd : nullptr);
    if (r) return r;
    c->rt_launches++;
    if (tbv) continue;
    e.ncol_tile = a.ntile;
    e.col0 = c0;
    e.jac = c->d_jtile;
    const long ne = c->win_on ? (long)e.nstk * (c->h_poff[c0 + a.ntile] - c->h_poff[c0]) : (long)a.ntile * e.nfreq;
    hipLaunchKernelGGL(eqv_kernel, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, st, e);
    HIPCHK(c, hipGetLastError());
  }
  // the LSF acts on the node-contracted response functions, after GAIN1D
  // (forward.f90:608-657), and on the Stokes rows (:810-844)
  r = run_lsf(c, d_stokes, (long)ncol * 4, st);
  if (r) return r;
  r = run_lsf(c, d_eqv, (long)ncol * e.np * e.nstk, st);
  if (r) return r;
  if (c->prof) HIPCHK(c, hipEventRecord(c->ev[2], st));
  return FZ_OK;
}

}  // extern "C"

// per-pixel windows: the LM step reads ragged rows and normalises each
// pixel's chi^2 by its own number of wavelengths times inverted Stokes
static void set_lm_windows(const fz_ctx* c, LmArgs& a) {
  a.poff = c->win_on ? c->d_poff : nullptr;
  a.nstk = a.nfreq / a.numw;
  a.inu_pix = c->win_on ? 1 : 0;
}

// lm_kernel over nrows rows: one wave per row with the work arrays in LDS,
// or, beyond LM_MAXNP free parameters, four waves per row with the work
// arrays in device memory, in batches of rows whose slices fit 2 GiB
static int launch_lm(fz_ctx* c, LmArgs a, int nrows, hipStream_t st) {
  if (!c->lm_big) {
    a.work = nullptr;
    a.work_stride = 0;
    a.row0 = 0;
    hipLaunchKernelGGL(lm_kernel<false>, dim3(nrows), dim3(LM_THREADS), c->lm_lds, st, a);
    HIPCHK(c, hipGetLastError());
    return FZ_OK;
  }
  const int batch = (int)std::max<size_t>(1, std::min<size_t>((size_t)nrows, ((size_t)2 << 30) / c->lm_work));
  int r = ensure(c, (float**)&c->d_lmwork, &c->lmwork_cap, c->lm_work * batch);
  if (r) return r;
  a.work = c->d_lmwork;
  a.work_stride = (long)(c->lm_work / sizeof(double));
  for (int r0 = 0; r0 < nrows; r0 += batch) {
    a.row0 = r0;
    hipLaunchKernelGGL(lm_kernel<true>, dim3(std::min(batch, nrows - r0)), dim3(LM_BIG_THREADS), 0, st, a);
    HIPCHK(c, hipGetLastError());
  }
  return FZ_OK;
}

extern "C" {

int fz_lm_step_dev(fz_ctx* c, int ncol, const double* d_obs, const float* d_stokes, double* d_best_syn, double* d_sla,
                   const float* d_eqv, float* d_eqv_best, const double* d_isigmap, float* d_atm, float* d_atm_best,
                   int32_t* d_done, double* d_delta, void* stream) {
  if (!c || ncol < 1 || !d_obs || !d_stokes || !d_best_syn || !d_sla || !d_eqv || !d_eqv_best || !d_isigmap ||
      !d_atm || !d_atm_best)
    return FZ_EARG;
  if (!c->inv_set) return set_err(c, FZ_ECONFIG, "fz_set_inversion first");
  if (c->win_on && ncol != c->win_ncol) return set_err(c, FZ_EARG, "column count differs from fz_set_windows");
  HIPCHK(c, hipSetDevice(c->device));
  LmArgs a = c->lm;
  a.ncol = ncol;
  a.obs = d_obs;
  a.stokes = d_stokes;
  a.best_syn = d_best_syn;
  a.sla = d_sla;
  a.eqv = d_eqv;
  a.eqv_best = d_eqv_best;
  a.isigmap = d_isigmap;
  a.atm = d_atm;
  a.atm_best = d_atm_best;
  a.done = d_done;
  a.delta = d_delta;
  a.pix_of = nullptr;
  set_lm_windows(c, a);
  return launch_lm(c, a, ncol, (hipStream_t)stream);
}

}  // extern "C"

// ------------------------------------------------------------------ GET_PERTURBATION / HESSIAN

// doubles of device memory that run_pert needs beyond its inputs and outputs:
// the normal matrix with the gradient column, and the solver's work arrays
// when they do not fit the LDS
static size_t pert_scratch_doubles(int np) {
  size_t n = (size_t)np * (np + 1);
  if (np > LM_MAXNP) n += pert_work_doubles(np, LM_BIG_THREADS);
  return (n + 31) / 32 * 32;
}

static int pert_check(fz_ctx* c, int np, int nf, int dtype) {
  if (np < 1 || nf < 1) return set_err(c, FZ_EARG, "GET_PERTURBATION: NP and NF must be positive");
  if (np > LM_MAXNP_BIG) return set_err(c, FZ_EARG, "GET_PERTURBATION: more than 2048 parameters");
  // lm.f90:194-201: any other DTYPE stops the reference
  if (dtype != 1 && dtype != 2) return set_err(c, FZ_EARG, "LM does not support DTYPE " + std::to_string(dtype));
  return FZ_OK;
}

// the normal matrix of X (np columns at x[p*sp + f*sf]) and, with y, the
// gradient X^T y into gram[np][np+1] (upper triangle)
static int launch_gram(fz_ctx* c, int np, int nf, const double* x, long sp, long sf, const double* y, double* gram,
                       hipStream_t st) {
  GramArgs g;
  g.np = np;
  g.nf = nf;
  g.x = x;
  g.sp = sp;
  g.sf = sf;
  g.y = y;
  g.gram = gram;
  const unsigned nti = (unsigned)((np + GR_TILE - 1) / GR_TILE), ntj = (unsigned)((np + 1 + GR_TILE - 1) / GR_TILE);
  hipLaunchKernelGGL(gram_kernel, dim3(ntj, nti), dim3(GR_THREADS), 0, st, g);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// GET_PERTURBATION on device arrays with the caller's scratch (at least
// pert_scratch_doubles(np) doubles)
static int run_pert(fz_ctx* c, int np, int nf, const double* d_ijac, const double* d_diff, double lambda,
                    double* d_delta, const double* d_pen, const double* d_hss, int dtype, double svdtol,
                    double* scratch, hipStream_t st) {
  int r = launch_gram(c, np, nf, d_ijac, nf, 1, d_diff, scratch, st);
  if (r) return r;
  PertArgs a;
  a.np = np;
  a.dtype = dtype;
  a.lambda = lambda;
  a.svdtol = svdtol;
  a.gram = scratch;
  a.reg_pen = d_pen;
  a.reg_hss = d_hss;
  a.delta = d_delta;
  if (np <= LM_MAXNP) {
    const size_t lds = pert_work_doubles(np, LM_THREADS) * sizeof(double);
    HIPCHK(c, hipFuncSetAttribute((const void*)pert_solve_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds));
    a.work = nullptr;
    hipLaunchKernelGGL(pert_solve_kernel<false>, dim3(1), dim3(LM_THREADS), lds, st, a);
  } else {
    a.work = scratch + (size_t)np * (np + 1);
    hipLaunchKernelGGL(pert_solve_kernel<true>, dim3(1), dim3(LM_BIG_THREADS), 0, st, a);
  }
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// fz_get_perturbation_dev_noalloc: the normal matrix and the solver's work
// arrays in a fixed device array instead of memory the context allocates.
// Every call on a GPU shares that GPU's copy (calls that overlap on one GPU
// race); each call writes every entry it reads, so nothing is cleared.
constexpr int NOALLOC_MAXNP = 512;
constexpr size_t NOALLOC_DOUBLES = (size_t)NOALLOC_MAXNP * (NOALLOC_MAXNP + 1) +
                                   2 * (size_t)NOALLOC_MAXNP * (NOALLOC_MAXNP + 1) + 8 * (size_t)NOALLOC_MAXNP +
                                   LM_BIG_THREADS + 32;   // 6.3 MB
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];
// the address of each GPU's copy of scratch, from hipGetSymbolAddress with
// that GPU current (the array's name is a host-side stand-in)
static double* g_scratch_dev[64];

static int scratch_setup(int device) {
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  if (device < 0 || device >= 64) return FZ_EARG;
  if (g_scratch_dev[device]) return FZ_OK;
  void* ptr = nullptr;
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return FZ_EHIP;
  g_scratch_dev[device] = (double*)ptr;
  return FZ_OK;
}

extern "C" {

int fz_get_perturbation_dev_noalloc(fz_ctx* c, int np, int nf, const double* d_ijacobian, const double* d_diff,
                                    double lambdap, double* d_delta, const double* d_reg_pen,
                                    const double* d_reg_hss, int dtype, double svdtol, void* stream) {
  if (!c || !d_ijacobian || !d_diff || !d_delta) return FZ_EARG;
  int r = pert_check(c, np, nf, dtype);
  if (r) return r;
  if (np > NOALLOC_MAXNP)
    return set_err(c, FZ_EARG, "fz_get_perturbation_dev_noalloc: at most 512 parameters (fixed scratch)");
  static_assert(NOALLOC_DOUBLES >= (size_t)NOALLOC_MAXNP * (NOALLOC_MAXNP + 1) + 2 * (size_t)NOALLOC_MAXNP *
                                        (NOALLOC_MAXNP + 1) + 8 * (size_t)NOALLOC_MAXNP + LM_BIG_THREADS,
                "scratch holds pert_scratch_doubles(NOALLOC_MAXNP)");
  if (pert_scratch_doubles(np) > NOALLOC_DOUBLES) return set_err(c, FZ_EARG, "scratch too small");
  double* ptr = g_scratch_dev[c->device];
  if (!ptr) return set_err(c, FZ_EHIP, "scratch address of this device not set");
  HIPCHK(c, hipSetDevice(c->device));
  return run_pert(c, np, nf, d_ijacobian, d_diff, lambdap, d_delta, d_reg_pen, d_reg_hss, dtype, svdtol, ptr,
                  (hipStream_t)stream);
}

int fz_get_perturbation_dev(fz_ctx* c, int np, int nf, const double* d_ijacobian, const double* d_diff,
                            double lambdap, double* d_delta, const double* d_reg_pen, const double* d_reg_hss,
                            int dtype, double svdtol, void* stream) {
  if (!c || !d_ijacobian || !d_diff || !d_delta) return FZ_EARG;
  int r = pert_check(c, np, nf, dtype);
  if (r) return r;
  HIPCHK(c, hipSetDevice(c->device));
  r = ensure(c, &c->d_pert, &c->pert_cap, sizeof(double) * pert_scratch_doubles(np));
  if (r) return r;
  return run_pert(c, np, nf, d_ijacobian, d_diff, lambdap, d_delta, d_reg_pen, d_reg_hss, dtype, svdtol,
                  (double*)c->d_pert, (hipStream_t)stream);
}

int fz_get_perturbation(fz_ctx* c, int np, int nf, const double* ijacobian, const double* diff, double lambdap,
                        double* delta, const double* reg_pen, const double* reg_hss, int dtype, double svdtol) {
  if (!c || !ijacobian || !diff || !delta) return FZ_EARG;
  int r = pert_check(c, np, nf, dtype);
  if (r) return r;
  HIPCHK(c, hipSetDevice(c->device));
  const size_t nj = (size_t)np * nf, nh = reg_hss ? (size_t)np * np : 0, npn = reg_pen ? (size_t)np : 0;
  r = ensure(c, &c->d_pstage, &c->pstage_cap, sizeof(double) * (nj + nf + npn + nh + np));
  if (r) return r;
  r = ensure(c, &c->d_pert, &c->pert_cap, sizeof(double) * pert_scratch_doubles(np));
  if (r) return r;
  double* dj = (double*)c->d_pstage;
  double* dd = dj + nj;
  double* dp = dd + nf;
  double* dh = dp + npn;
  double* dl = dh + nh;
  HIPCHK(c, hipMemcpy(dj, ijacobian, sizeof(double) * nj, hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(dd, diff, sizeof(double) * nf, hipMemcpyHostToDevice));
  if (npn) HIPCHK(c, hipMemcpy(dp, reg_pen, sizeof(double) * npn, hipMemcpyHostToDevice));
  if (nh) HIPCHK(c, hipMemcpy(dh, reg_hss, sizeof(double) * nh, hipMemcpyHostToDevice));
  r = run_pert(c, np, nf, dj, dd, lambdap, dl, npn ? dp : nullptr, nh ? dh : nullptr, dtype, svdtol,
               (double*)c->d_pert, nullptr);
  if (r) return r;
  HIPCHK(c, hipMemcpy(delta, dl, sizeof(double) * np, hipMemcpyDeviceToHost));
  return FZ_OK;
}

int fz_hessian(fz_ctx* c, int np, int nf, const double* jacobian, double* hss) {
  if (!c || !jacobian || !hss) return FZ_EARG;
  if (np < 1 || nf < 1 || np > LM_MAXNP_BIG) return set_err(c, FZ_EARG, "HESSIAN: NP in 1..2048 and NF >= 1");
  HIPCHK(c, hipSetDevice(c->device));
  const size_t nj = (size_t)np * nf, ng = (size_t)np * (np + 1);
  int r = ensure(c, &c->d_pstage, &c->pstage_cap, sizeof(double) * (nj + ng));
  if (r) return r;
  double* dj = (double*)c->d_pstage;
  double* dg = dj + nj;
  HIPCHK(c, hipMemcpy(dj, jacobian, sizeof(double) * nj, hipMemcpyHostToDevice));
  // JACOBIAN(NP,NF): parameter p of spectral row f at jacobian[f*np + p]
  r = launch_gram(c, np, nf, dj, 1, np, nullptr, dg, nullptr);
  if (r) return r;
  std::vector<double> g(ng);
  HIPCHK(c, hipMemcpy(g.data(), dg, sizeof(double) * ng, hipMemcpyDeviceToHost));
  for (int j = 0; j < np; ++j)
    for (int i = 0; i < np; ++i) hss[(size_t)j * np + i] = g[(size_t)std::min(i, j) * (np + 1) + std::max(i, j)];
  return FZ_OK;
}

}  // extern "C"

extern "C" {

int fz_get_dmodel3ds(fz_ctx* c, int nx, int ny, const double* obs3d, const double* syn3d, double* best_syn,
                     double* inv_mas, int ld_inv_mas, const float* dsyn, float* best_dsyn, const double* isigmap3d,
                     float* const* model, float* const* best_model, int32_t* am_i_done) {
  if (!c || nx < 1 || ny < 1 || !obs3d || !syn3d || !best_syn || !inv_mas || ld_inv_mas < 9 || !dsyn ||
      !best_dsyn || !isigmap3d || !model || !best_model || !am_i_done)
    return FZ_EARG;
  for (int p = 0; p < NATM; ++p)
    if (!model[p] || !best_model[p]) return FZ_EARG;
  if (!c->inv_set) return set_err(c, FZ_ECONFIG, "fz_set_inversion first");
  if (c->win_on) return set_err(c, FZ_EARG, "per-pixel windows: use fz_lm_step_dev");
  const int nz = c->cfg.nz, nf = c->lm.nfreq, np = c->lm.np;
  // pixels with AM_I_DONE == 0, in the reference's (y fastest) order
  std::vector<int> cols;
  for (int x = 0; x < nx; ++x)
    for (int y = 0; y < ny; ++y)
      if (am_i_done[y + (size_t)ny * x] == 0) cols.push_back(y + ny * x);
  const int n = (int)cols.size();
  if (n == 0) return FZ_OK;
  // one weight vector when ISIGMAP3D is the same in every pixel
  bool shared = true;
  for (int i = 1; i < n && shared; ++i)
    shared = memcmp(isigmap3d + (size_t)cols[i] * nf, isigmap3d + (size_t)cols[0] * nf, sizeof(double) * nf) == 0;
  const size_t nfn = (size_t)nf * n, ne = (size_t)np * nf;
  DevBuf b_obs, b_syn, b_bsyn, b_sla, b_eqv, b_eqvb, b_isig, b_atm, b_best, b_tmp, b_done;
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMalloc(&b_obs.p, sizeof(double) * nfn));
  HIPCHK(c, hipMalloc(&b_syn.p, sizeof(double) * nfn));
  HIPCHK(c, hipMalloc(&b_bsyn.p, sizeof(double) * nfn));
  HIPCHK(c, hipMalloc(&b_sla.p, sizeof(double) * 9 * n));
  HIPCHK(c, hipMalloc(&b_eqv.p, sizeof(float) * ne * n));
  HIPCHK(c, hipMalloc(&b_eqvb.p, sizeof(float) * ne * n));
  HIPCHK(c, hipMalloc(&b_isig.p, sizeof(double) * (shared ? (size_t)nf : nfn)));
  HIPCHK(c, hipMalloc(&b_atm.p, sizeof(float) * NATM * nz * n));
  HIPCHK(c, hipMalloc(&b_best.p, sizeof(float) * NATM * nz * n));
  HIPCHK(c, hipMalloc(&b_tmp.p, sizeof(float) * nz * n));
  HIPCHK(c, hipMalloc(&b_done.p, sizeof(int32_t) * n));
  // gather the active pixels' rows (GET_DMODEL3DS sends the same arrays per pixel)
  auto gather_d = [&](const double* src, size_t len, void* dst) -> int {
    std::vector<double> h(len * n);
    for (int i = 0; i < n; ++i) memcpy(&h[(size_t)i * len], src + (size_t)cols[i] * len, sizeof(double) * len);
    HIPCHK(c, hipMemcpy(dst, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
    return FZ_OK;
  };
  auto gather_f = [&](const float* src, size_t len, void* dst) -> int {
    std::vector<float> h(len * n);
    for (int i = 0; i < n; ++i) memcpy(&h[(size_t)i * len], src + (size_t)cols[i] * len, sizeof(float) * len);
    HIPCHK(c, hipMemcpy(dst, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice));
    return FZ_OK;
  };
  int r;
  if ((r = gather_d(obs3d, nf, b_obs.p)) || (r = gather_d(syn3d, nf, b_syn.p)) ||
      (r = gather_d(best_syn, nf, b_bsyn.p)) || (r = gather_f(dsyn, ne, b_eqv.p)) ||
      (r = gather_f(best_dsyn, ne, b_eqvb.p)))
    return r;
  if (shared) HIPCHK(c, hipMemcpy(b_isig.p, isigmap3d + (size_t)cols[0] * nf, sizeof(double) * nf, hipMemcpyHostToDevice));
  else if ((r = gather_d(isigmap3d, nf, b_isig.p))) return r;
  {
    std::vector<double> h((size_t)9 * n);
    for (int i = 0; i < n; ++i) memcpy(&h[(size_t)i * 9], inv_mas + (size_t)cols[i] * ld_inv_mas, sizeof(double) * 9);
    HIPCHK(c, hipMemcpy(b_sla.p, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
  }
  HIPCHK(c, hipMemset(b_done.p, 0, sizeof(int32_t) * n));
  const unsigned tb = 256, tg = (unsigned)(((long)nz * n + tb - 1) / tb);
  const size_t colbytes = sizeof(float) * nz;
  std::vector<float> h((size_t)nz * n);
  float* d_tmp = (float*)b_tmp.p;
  for (int which = 0; which < 2; ++which) {
    float* const* cubes = which ? best_model : model;
    float* d = (float*)(which ? b_best.p : b_atm.p);
    for (int p = 0; p < NATM; ++p) {
      for (int i = 0; i < n; ++i) memcpy(&h[(size_t)i * nz], cubes[p] + (size_t)cols[i] * nz, colbytes);
      HIPCHK(c, hipMemcpy(d_tmp, h.data(), colbytes * n, hipMemcpyHostToDevice));
      hipLaunchKernelGGL(cube_to_soa, dim3(tg), dim3(tb), 0, 0, d_tmp, d + (size_t)p * nz * n, nz, n);
    }
  }
  LmArgs a = c->lm;
  a.ncol = n;
  a.obs = (const double*)b_obs.p;
  a.syn_d = (const double*)b_syn.p;
  a.stokes = (const float*)b_syn.p;   // not read: the FP64 synthesis replaces it
  a.best_syn = (double*)b_bsyn.p;
  a.sla = (double*)b_sla.p;
  a.eqv = (const float*)b_eqv.p;
  a.eqv_best = (float*)b_eqvb.p;
  a.isigmap = (const double*)b_isig.p;
  a.isig_stride = shared ? 0 : nf;
  a.atm = (float*)b_atm.p;
  a.atm_best = (float*)b_best.p;
  a.done = (int32_t*)b_done.p;
  a.delta = nullptr;
  a.pix_of = nullptr;
  set_lm_windows(c, a);
  r = launch_lm(c, a, n, nullptr);
  if (r) return r;
  HIPCHK(c, hipDeviceSynchronize());
  // scatter back: models, INV_MAS(1:9), BEST_DSYN, BEST_SYN, AM_I_DONE
  for (int which = 0; which < 2; ++which) {
    float* const* cubes = which ? best_model : model;
    const float* d = (const float*)(which ? b_best.p : b_atm.p);
    for (int p = 0; p < NATM; ++p) {
      hipLaunchKernelGGL(soa_to_cube, dim3(tg), dim3(tb), 0, 0, d + (size_t)p * nz * n, d_tmp, nz, n);
      HIPCHK(c, hipMemcpy(h.data(), d_tmp, colbytes * n, hipMemcpyDeviceToHost));
      for (int i = 0; i < n; ++i) memcpy(cubes[p] + (size_t)cols[i] * nz, &h[(size_t)i * nz], colbytes);
    }
  }
  {
    std::vector<double> hs((size_t)9 * n), hb(nfn);
    HIPCHK(c, hipMemcpy(hs.data(), b_sla.p, sizeof(double) * hs.size(), hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(hb.data(), b_bsyn.p, sizeof(double) * nfn, hipMemcpyDeviceToHost));
    std::vector<int32_t> hd(n);
    HIPCHK(c, hipMemcpy(hd.data(), b_done.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) {
      memcpy(inv_mas + (size_t)cols[i] * ld_inv_mas, &hs[(size_t)i * 9], sizeof(double) * 9);
      memcpy(best_syn + (size_t)cols[i] * nf, &hb[(size_t)i * nf], sizeof(double) * nf);
      if (hd[i]) am_i_done[cols[i]] = 1;
    }
    std::vector<float> he(ne * n);
    HIPCHK(c, hipMemcpy(he.data(), b_eqvb.p, sizeof(float) * he.size(), hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) memcpy(best_dsyn + (size_t)cols[i] * ne, &he[(size_t)i * ne], sizeof(float) * ne);
  }
  return FZ_OK;
}

// fz_lm_step_dev over the na active pixels pix_of[0..na): stokes and eqv are
// the compacted rows of those pixels, everything else is in pixel space.
static int lm_step_active(fz_ctx* c, int ncol, int na, const int32_t* pix_of, const double* d_obs,
                          const float* d_stokes_c, double* d_best_syn, double* d_sla, const float* d_eqv_c,
                          float* d_eqv_best, const double* d_isigmap, long isig_stride, float* d_atm,
                          float* d_atm_best, int32_t* d_done, hipStream_t st) {
  LmArgs a = c->lm;
  a.ncol = ncol;
  a.obs = d_obs;
  a.stokes = d_stokes_c;
  a.best_syn = d_best_syn;
  a.sla = d_sla;
  a.eqv = d_eqv_c;
  a.eqv_best = d_eqv_best;
  a.isigmap = d_isigmap;
  a.isig_stride = isig_stride;
  a.atm = d_atm;
  a.atm_best = d_atm_best;
  a.done = d_done;
  a.delta = nullptr;
  a.pix_of = pix_of;
  set_lm_windows(c, a);
  if (c->win_on && (pix_of || ncol != c->win_ncol)) return set_err(c, FZ_EARG, "per-pixel windows: every pixel keeps its row");
  return launch_lm(c, a, na, st);
}

// GET_NJEVALS (get_dmodel.f90:375-407) with TOFFSET = 1 (pre_post_duties.f90:645)
static int njevals(int apar, int curic, int maxiter, int cycpow, int nz) {
  const int toffset = 1;
  if (apar == 1) {
    if (curic == 0 || curic == maxiter) return nz;
    return std::min(nz, (int)std::pow((double)cycpow, (double)(curic + toffset - 1)));
  }
  if (curic == 0) return nz;
  if (curic == 1) return 1;
  if (curic == maxiter) return nz;
  return std::min(nz, (int)std::pow((double)cycpow, (double)(curic - 1)));
}

// SET_TAU's assists on device data (fz_assist_dev, the first cycle of fz_invert3d_dev)
static int run_assist(fz_ctx* c, int ncol, const double* d_obs, int flags, float* d_atm, hipStream_t st) {
  const Cfg& g = c->cfg;
  AssistArgs a;
  a.ncol = ncol;
  a.nz = g.nz;
  a.nfreq = c->lm.nfreq;
  a.numw = g.numw;
  a.itz = g.reg_nwave[0];
  a.nstk = c->lm.nfreq / g.numw;
  a.flags = flags;
  a.kz = (int)std::ceil((double)(float)g.nz / 3.0) - 1;   // CEILING(REAL(NZ)/3.)
  a.lk_hc = (g.reg_l0main[0] * 1.0e-8 * KBOL) / (HPLA * LIGHT);
  a.obs = d_obs;
  a.atm = d_atm;
  DevBuf b_vec, b_pix, b_mx;
  HIPCHK(c, hipMalloc(&b_vec.p, sizeof(double) * (3 * (size_t)a.itz + 1)));
  HIPCHK(c, hipMalloc(&b_pix.p, sizeof(double) * 5 * (size_t)ncol));
  HIPCHK(c, hipMalloc(&b_mx.p, sizeof(double) * 4));
  a.vec = (double*)b_vec.p;
  a.pix = (double*)b_pix.p;
  a.mx = (double*)b_mx.p;
  const unsigned gp = (unsigned)((ncol + 255) / 256);
  if (flags & (ASSIST_B | ASSIST_V)) {
    hipLaunchKernelGGL(assist_sum_kernel, dim3((unsigned)a.itz), dim3(256), 0, st, a);
    hipLaunchKernelGGL(assist_vec_kernel, dim3(1), dim3(64), 0, st, a);
  } else {
    HIPCHK(c, hipMemsetAsync(a.vec, 0, sizeof(double) * (3 * (size_t)a.itz + 1), st));
  }
  hipLaunchKernelGGL(assist_pix_kernel, dim3(gp), dim3(256), 0, st, a);
  hipLaunchKernelGGL(assist_max_kernel, dim3(1), dim3(256), 0, st, a);
  hipLaunchKernelGGL(assist_apply_kernel, dim3(gp), dim3(256), 0, st, a);
  HIPCHK(c, hipGetLastError());
  // the scratch is released at return: wait for the kernels that read it
  HIPCHK(c, hipStreamSynchronize(st));
  return FZ_OK;
}

extern "C" int fz_assist_dev(fz_ctx* c, int ncol, const double* d_obs, int flags, float* d_atm, void* stream) {
  if (!c || ncol < 1 || !d_obs || !d_atm || (flags & ~15)) return FZ_EARG;
  if (!c->inv_set) return set_err(c, FZ_ECONFIG, "fz_set_inversion first");
  if (c->win_on) return set_err(c, FZ_EARG, "per-pixel windows: the assists read a common first region");
  if (flags == 0) return FZ_OK;
  HIPCHK(c, hipSetDevice(c->device));
  return run_assist(c, ncol, d_obs, flags, d_atm, (hipStream_t)stream);
}

int fz_invert3d_dev(fz_ctx* c, int nx, int ny, float* d_atm, const double* d_obs, const fz_invert_control* ctl,
                    float* d_stokes, double* d_chi2, int* iterations, void* stream) {
  if (!c || !c->configured || nx < 1 || ny < 1 || !d_atm || !d_obs || !ctl || !d_stokes) return FZ_EARG;
  const int nz = c->cfg.nz, numw = c->cfg.numw, ncol = nx * ny;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  // MAXITER (pre_post_duties.f90:635-646) from the parameters' maximum nodes
  int nfreev = 0, nfreep = 0, infreepmax = 0;
  for (int p = 0; p < 8; ++p) {
    if (!ctl->atmpar[p]) continue;
    const int vmax = ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
    ++nfreev;
    nfreep += vmax;
    infreepmax = std::max(infreepmax, vmax);
  }
  if (nfreev == 0) return set_err(c, FZ_ECONFIG, "no parameter inverted");
  const int cycpow = ctl->cycpow > 0 ? ctl->cycpow : 2;
  const int maxiter = (nfreep == nfreev) ? 1 : (int)std::floor(std::log((double)infreepmax) / std::log((double)cycpow));
  if (maxiter < 1) return set_err(c, FZ_ECONFIG, "no inversion cycle");
  const int maxsteps = ctl->maxsteps > 0 ? ctl->maxsteps : 5;
  const int itcap = ctl->max_iterations > 0 ? ctl->max_iterations : 1000;
  // Stokes weights WSTK / MINW in REAL(4) (input_file.f90:1298-1303; weights of
  // Stokes parameters not inverted are zero) and ISIGMAP = WSTK^2 / ISIGMA^2
  // with ISIGMA a REAL(8) taken from a REAL(4) value (input_file.f90:181,433)
  int nstk = 0;
  float wsum = 0.f, wst[4];
  for (int s = 0; s < 4; ++s) {
    wst[s] = ctl->invstk[s] ? ctl->wstk[s] : 0.f;
    if (ctl->invstk[s]) ++nstk;
    wsum += wst[s] * wst[s];
  }
  if (nstk == 0) return set_err(c, FZ_ECONFIG, "no Stokes parameter inverted");
  const float minw = sqrtf(wsum) / sqrtf((float)nstk);
  const double isigma = (double)(float)(ctl->noise > 0 ? ctl->noise : 4.0e-3);
  const int nfreq = nstk * numw;
  // per-pixel windows: ragged rows of nstk*numw_pix (obs, best synthesis,
  // response functions), Stokes of 4*numw_pix; every pixel keeps its row
  const bool win = c->win_on;
  if (win && ncol != c->win_ncol) return set_err(c, FZ_EARG, "column count differs from fz_set_windows");
  const size_t nwtot = win ? (size_t)c->h_poff[ncol] : (size_t)ncol * numw;
  std::vector<double> isig(nfreq);
  {
    int b = 0;
    for (int s = 0; s < 4; ++s) {
      if (!ctl->invstk[s]) continue;
      const float w = wst[s] / minw;
      for (int l = 0; l < numw; ++l) isig[b * numw + l] = (double)(w * w) / (isigma * isigma);
      ++b;
    }
  }
  int npmax = 0;
  for (int p = 0; p < 8; ++p)
    if (ctl->atmpar[p]) npmax += ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
  if (npmax > LM_MAXNP_BIG) return set_err(c, FZ_ECONFIG, "more than 2048 free parameters in the last cycle");
  DevBuf b_isig, b_best, b_eqv, b_eqvb, b_bsyn, b_sla, b_done, b_stat, b_t0, b_t1, b_atmc, b_idx, b_cnt;
  const size_t natm = (size_t)12 * nz * ncol;
  // STOKES SETUP: AUTO replaces the map-wide weights by every pixel's own
  // (SET_WEIGHTS, get_dmodel.f90:2024-2047), set once from the observations
  const long isig_stride = c->autow ? nfreq : 0;
  if (c->autow && win) return set_err(c, FZ_ECONFIG, "automatic Stokes weights take the dense spectral grid");
  HIPCHK(c, hipMalloc(&b_isig.p, sizeof(double) * nfreq * (c->autow ? (size_t)ncol : 1)));
  HIPCHK(c, hipMalloc(&b_best.p, sizeof(float) * natm));
  HIPCHK(c, hipMalloc(&b_eqv.p, sizeof(float) * nwtot * npmax * nstk));
  HIPCHK(c, hipMalloc(&b_eqvb.p, sizeof(float) * nwtot * npmax * nstk));
  HIPCHK(c, hipMalloc(&b_bsyn.p, sizeof(double) * nwtot * nstk));
  HIPCHK(c, hipMalloc(&b_sla.p, sizeof(double) * (size_t)ncol * 9));
  HIPCHK(c, hipMalloc(&b_done.p, sizeof(int32_t) * ncol));
  HIPCHK(c, hipMalloc(&b_stat.p, sizeof(double) * 2));
  HIPCHK(c, hipMalloc(&b_t0.p, sizeof(double) * (size_t)nz * ncol));
  HIPCHK(c, hipMalloc(&b_t1.p, sizeof(double) * (size_t)nz * ncol));
  // active pixels: FORWARD3D models only the columns with AM_I_DONE == 0
  // (forward.f90:43-306); they are gathered into a compact cube
  HIPCHK(c, hipMalloc(&b_atmc.p, sizeof(float) * natm));
  HIPCHK(c, hipMalloc(&b_idx.p, sizeof(int32_t) * ncol));
  HIPCHK(c, hipMalloc(&b_cnt.p, sizeof(int32_t)));
  if (c->autow) {
    int r = fz_auto_weights_dev(c, ncol, d_obs, ctl->invstk, ctl->noise, (double*)b_isig.p, stream);
    if (r) return r;
  } else {
    HIPCHK(c, hipMemcpyAsync(b_isig.p, isig.data(), sizeof(double) * nfreq, hipMemcpyHostToDevice, st));
  }
  float* best = (float*)b_best.p;
  double* sla = (double*)b_sla.p;
  int32_t* done = (int32_t*)b_done.p;
  const unsigned gatm = (unsigned)((natm + 255) / 256), grow = (unsigned)(((size_t)nz * ncol + 255) / 256);
  static const int rowof[8] = {A_T, A_PG, A_RHO, A_BX, A_BY, A_BZ, A_VZ, A_PG};
  int total_it = 0;
  const int cyc0 = std::min(std::max(1, ctl->first_cycle), maxiter);
  for (int cyc = cyc0; cyc <= maxiter; ++cyc) {
    // INITIALIZE_CYCLE (invert3d.f90:228-325)
    fz_inversion inv;
    std::memset(&inv, 0, sizeof(inv));
    for (int p = 0; p < 8; ++p) {
      if (!ctl->atmpar[p]) continue;
      const int vmax = ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
      inv.atmpar[p] = 1;
      inv.nodes[p] = std::min(njevals(p + 1, cyc, maxiter, cycpow, nz), vmax);
      inv.pen_typ[p] = ctl->pen_typ[p];
      inv.pen_alp[p] = ctl->pen_alp[p];
    }
    for (int s = 0; s < 4; ++s) inv.invstk[s] = ctl->invstk[s];
    inv.regul = ctl->regul;
    inv.solver = ctl->solver > 0 ? ctl->solver : 1;
    inv.node_expansion = ctl->node_expansion > 0 ? ctl->node_expansion : 1;
    inv.maxsteps = maxsteps;
    inv.svdtol = ctl->svdtol;
    int r = fz_set_inversion(c, &inv, nullptr, nullptr);
    if (r) return r;
    hipLaunchKernelGGL(inv_init_kernel, dim3((ncol + 255) / 256), dim3(256), 0, st, ncol, sla, done);
    // SET_TAU (:492-727): a synthesis updates log tau5 when Pg and P0 are not
    // inverted; in the first cycle the assist initialisers change the start
    // model before it
    if (!ctl->atmpar[1] && !ctl->atmpar[7]) {
      if (cyc == cyc0 && ctl->assist && !c->win_on) {
        r = run_assist(c, ncol, d_obs, ctl->assist & 15, d_atm, st);
        if (r) return r;
      }
      r = fz_forward_dev(c, ncol, d_atm, FZ_RF_NONE, d_stokes, nullptr, nullptr, stream);
      if (r) return r;
    }
    // UPDATE_CURRENT_TO_BEST, then SMOOTHING_B on the best model into both
    hipLaunchKernelGGL(copy_f32_kernel, dim3(gatm), dim3(256), 0, st, d_atm, best, (long)natm);
    if (ctl->smoothing) {
      for (int p = 0; p < 8; ++p) {
        if (!ctl->atmpar[p]) continue;
        float* rb = best + (size_t)rowof[p] * nz * ncol;
        float* rc = d_atm + (size_t)rowof[p] * nz * ncol;
        double *t0 = (double*)b_t0.p, *t1 = (double*)b_t1.p;
        hipLaunchKernelGGL(to_double_kernel, dim3(grow), dim3(256), 0, st, rb, t0, (long)nz * ncol);
        const int ext[3] = {nx, ny, nz};
        for (int ax = 0; ax < 3; ++ax) {
          if (ext[ax] <= 4) continue;
          hipLaunchKernelGGL(smooth_axis_kernel, dim3(grow), dim3(256), 0, st, t0, t1, nz, ny, nx, ax);
          std::swap(t0, t1);
        }
        hipLaunchKernelGGL(from_double_kernel, dim3(grow), dim3(256), 0, st, t0, rc, rb, (long)nz * ncol);
      }
    }
    HIPCHK(c, hipGetLastError());
    const double need = (double)std::max(1, maxsteps - (maxiter - cyc));
    int na = ncol;   // active pixels (every pixel at a cycle start)
    for (int it = 0; it < itcap; ++it) {
      // MODELLING -> SOLVE_DMODEL -> MAKE_DECISION
      if (na == ncol) {
        r = fz_forward_nodes_dev(c, ncol, d_atm, d_stokes, (float*)b_eqv.p, nullptr, stream);
        if (r) return r;
        r = lm_step_active(c, ncol, ncol, nullptr, d_obs, d_stokes, (double*)b_bsyn.p, sla, (const float*)b_eqv.p,
                           (float*)b_eqvb.p, (const double*)b_isig.p, isig_stride, d_atm, best, done, st);
        if (r) return r;
      } else {
        const int32_t* idx = (const int32_t*)b_idx.p;
        float* atmc = (float*)b_atmc.p;
        const unsigned gc = (unsigned)(((long)12 * nz * na + 255) / 256);
        hipLaunchKernelGGL(gather_cols_kernel, dim3(gc), dim3(256), 0, st, (const float*)d_atm, atmc, idx, na, ncol,
                           12 * nz);
        r = fz_forward_nodes_dev(c, na, atmc, d_stokes, (float*)b_eqv.p, nullptr, stream);
        if (r) return r;
        hipLaunchKernelGGL(scatter_cols_kernel, dim3(gc), dim3(256), 0, st, (const float*)atmc, d_atm, idx, na,
                           ncol, 12 * nz);
        r = lm_step_active(c, ncol, na, idx, d_obs, d_stokes, (double*)b_bsyn.p, sla, (const float*)b_eqv.p,
                           (float*)b_eqvb.p, (const double*)b_isig.p, isig_stride, d_atm, best, done, st);
        if (r) return r;
      }
      hipLaunchKernelGGL(stats_kernel, dim3(1), dim3(256), 0, st, ncol, sla, done, (double*)b_stat.p);
      double hs[2];
      HIPCHK(c, hipMemcpyAsync(hs, b_stat.p, sizeof(hs), hipMemcpyDeviceToHost, st));
      HIPCHK(c, hipStreamSynchronize(st));
      ++total_it;
      if (ncol - (int)hs[1] <= 0) break;
      if (hs[0] / (double)ncol >= need) break;
      const int nact = ncol - (int)hs[1];
      if (nact < ncol && !win) {
        hipLaunchKernelGGL(compact_kernel, dim3(1), dim3(1024), 0, st, ncol, (const int32_t*)done, (int32_t*)b_idx.p,
                           (int32_t*)b_cnt.p);
        HIPCHK(c, hipGetLastError());
      }
      na = win ? ncol : nact;
    }
    // END_CYCLE (:328-403): current := best, synthesis without response functions
    hipLaunchKernelGGL(copy_f32_kernel, dim3(gatm), dim3(256), 0, st, best, d_atm, (long)natm);
    r = fz_forward_dev(c, ncol, d_atm, FZ_RF_NONE, d_stokes, nullptr, nullptr, stream);
    if (r) return r;
  }
  if (d_chi2) {
    HIPCHK(c, hipMemcpy2DAsync(d_chi2, sizeof(double), sla + 2, sizeof(double) * 9, sizeof(double), ncol,
                               hipMemcpyDeviceToDevice, st));
  }
  HIPCHK(c, hipStreamSynchronize(st));
  if (iterations) *iterations = total_it;
  return FZ_OK;
}

// INVERT3D with the spatial PSF coupling the pixels (the coupled inversion
// whose buffers coupled_inversion.f90:10-207 allocates; the reference does
// not wire its mathematics, get_dmodel.f90:1707-1711).  The model of every
// pixel is fitted to the observations through the PSF: chi^2 of the map =
// sum over pixels of the weighted squared residual obs - PSF * syn.  A
// Levenberg-Marquardt iteration over the whole map:
//   * forward with node-contracted response functions of the current model,
//     PSF convolution of the synthesis, residual and chi^2 of the map;
//   * acceptance by the map's chi^2 (pixels are coupled, so one pixel's
//     chi^2 does not decide its own step), lambda divided by sqrt(10) on an
//     accepted step and multiplied by 10 on a rejected one (the rules of
//     UPDATE_LAMBDA, get_dmodel.f90:917-956, applied to the map), the best
//     model, response functions and residual kept;
//   * the exact gradient of the map's chi^2 for each pixel, J_q^T W (PSF^T r)_q
//     with the adjoint convolution of the best residual, and the pixel's own
//     block of the coupled Gauss-Newton matrix, (sum PSF^2) J_q^T W J_q; the
//     damped solve and the node-basis update of lm_kernel.
// The cycle schedule, SET_TAU, the 1-2-1 smoothing and the assists are those
// of fz_invert3d_dev.  The cycle ends after MAXSTEPS rejected steps in a row
// with no net gain (the map's step count as INV_SLA(1) counts a pixel's) or
// the iteration cap.
static int coupled_forward(fz_ctx* c, int nx, int ny, float* d_atm, float* d_stokes, float* d_eqv, float* d_t1,
                           float* d_t2, hipStream_t st, bool nodes) {
  const int numw = c->cfg.numw, ncol = nx * ny;
  int r = nodes ? fz_forward_nodes_dev(c, ncol, d_atm, d_stokes, d_eqv, nullptr, st)
                : fz_forward_dev(c, ncol, d_atm, FZ_RF_NONE, d_stokes, nullptr, nullptr, st);
  if (r) return r;
  const long nch = 4L * numw;
  // [ncol][4 numw] -> [4 numw][ncol], convolve
  hipLaunchKernelGGL((transpose_kernel<float, float>), dim3((unsigned)((nch + 31) / 32), (unsigned)((ncol + 31) / 32)),
                     dim3(256), 0, st, (const float*)d_stokes, d_t1, (long)ncol, nch);
  launch_psf(c, nx, ny, (int)nch, d_t1, d_t2, 0, st);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

extern "C" {

int fz_coupled_invert3d_dev(fz_ctx* c, int nx, int ny, float* d_atm, const double* d_obs,
                            const fz_invert_control* ctl, float* d_stokes, double* d_chi2, int* iterations,
                            void* stream) {
  if (!c || !c->configured || nx < 1 || ny < 1 || !d_atm || !d_obs || !ctl || !d_stokes) return FZ_EARG;
  if (c->win_on) return set_err(c, FZ_ECONFIG, "the coupled inversion takes the dense spectral grid");
  if (c->autow) return set_err(c, FZ_ECONFIG, "the coupled inversion takes the map-wide Stokes weights");
  // the map transposes put 32 pixels per workgroup row on the grid's y axis
  if ((long)nx * ny > 32L * 65535) return set_err(c, FZ_EARG, "more than 2097120 pixels in one coupled map");
  const int nz = c->cfg.nz, numw = c->cfg.numw, ncol = nx * ny;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  int r = psf_taps(c, nx, ny);
  if (r) return r;
  int nfreev = 0, nfreep = 0, infreepmax = 0;
  for (int p = 0; p < 8; ++p) {
    if (!ctl->atmpar[p]) continue;
    const int vmax = ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
    ++nfreev;
    nfreep += vmax;
    infreepmax = std::max(infreepmax, vmax);
  }
  if (nfreev == 0) return set_err(c, FZ_ECONFIG, "no parameter inverted");
  const int cycpow = ctl->cycpow > 0 ? ctl->cycpow : 2;
  const int maxiter = (nfreep == nfreev) ? 1 : (int)std::floor(std::log((double)infreepmax) / std::log((double)cycpow));
  if (maxiter < 1) return set_err(c, FZ_ECONFIG, "no inversion cycle");
  const int maxsteps = ctl->maxsteps > 0 ? ctl->maxsteps : 5;
  const int itcap = ctl->max_iterations > 0 ? ctl->max_iterations : 1000;
  int nstk = 0;
  float wsum = 0.f, wst[4];
  for (int s = 0; s < 4; ++s) {
    wst[s] = ctl->invstk[s] ? ctl->wstk[s] : 0.f;
    if (ctl->invstk[s]) ++nstk;
    wsum += wst[s] * wst[s];
  }
  if (nstk == 0) return set_err(c, FZ_ECONFIG, "no Stokes parameter inverted");
  const float minw = sqrtf(wsum) / sqrtf((float)nstk);
  const double isigma = (double)(float)(ctl->noise > 0 ? ctl->noise : 4.0e-3);
  const int nfreq = nstk * numw;
  std::vector<double> isig(nfreq);
  {
    int b = 0;
    for (int s = 0; s < 4; ++s) {
      if (!ctl->invstk[s]) continue;
      const float w = wst[s] / minw;
      for (int l = 0; l < numw; ++l) isig[b * numw + l] = (double)(w * w) / (isigma * isigma);
      ++b;
    }
  }
  int npmax = 0;
  for (int p = 0; p < 8; ++p)
    if (ctl->atmpar[p]) npmax += ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
  if (npmax > LM_MAXNP_BIG) return set_err(c, FZ_ECONFIG, "more than 2048 free parameters in the last cycle");
  const size_t natm = (size_t)12 * nz * ncol, nrow = (size_t)ncol * nfreq, nmap = (size_t)4 * numw * ncol;
  DevBuf b_isig, b_best, b_eqv, b_eqvb, b_syn, b_res, b_resb, b_gres, b_chi, b_sum, b_t1, b_t2, b_s0, b_s1;
  HIPCHK(c, hipMalloc(&b_isig.p, sizeof(double) * nfreq));
  HIPCHK(c, hipMalloc(&b_best.p, sizeof(float) * natm));
  HIPCHK(c, hipMalloc(&b_eqv.p, sizeof(float) * nrow * npmax));
  HIPCHK(c, hipMalloc(&b_eqvb.p, sizeof(float) * nrow * npmax));
  HIPCHK(c, hipMalloc(&b_syn.p, sizeof(double) * nrow));
  HIPCHK(c, hipMalloc(&b_res.p, sizeof(double) * nrow));
  HIPCHK(c, hipMalloc(&b_resb.p, sizeof(double) * nrow));
  HIPCHK(c, hipMalloc(&b_gres.p, sizeof(double) * nrow));
  HIPCHK(c, hipMalloc(&b_chi.p, sizeof(double) * ncol));
  HIPCHK(c, hipMalloc(&b_sum.p, sizeof(double)));
  HIPCHK(c, hipMalloc(&b_t1.p, sizeof(float) * std::max(nmap, nrow)));
  HIPCHK(c, hipMalloc(&b_t2.p, sizeof(float) * std::max(nmap, nrow)));
  HIPCHK(c, hipMalloc(&b_s0.p, sizeof(double) * (size_t)nz * ncol));
  HIPCHK(c, hipMalloc(&b_s1.p, sizeof(double) * (size_t)nz * ncol));
  HIPCHK(c, hipMemcpyAsync(b_isig.p, isig.data(), sizeof(double) * nfreq, hipMemcpyHostToDevice, st));
  float* best = (float*)b_best.p;
  float *eqv = (float*)b_eqv.p, *eqvb = (float*)b_eqvb.p;
  float *t1 = (float*)b_t1.p, *t2 = (float*)b_t2.p;
  double *res = (double*)b_res.p, *resb = (double*)b_resb.p, *gres = (double*)b_gres.p;
  const unsigned gatm = (unsigned)((natm + 255) / 256), grow = (unsigned)(((size_t)nz * ncol + 255) / 256);
  static const int rowof[8] = {A_T, A_PG, A_RHO, A_BX, A_BY, A_BZ, A_VZ, A_PG};
  CoupledArgs ca;
  ca.npix = ncol;
  ca.nfreq = nfreq;
  ca.numw = numw;
  ca.nstk = nstk;
  ca.conv = t2;
  ca.obs = d_obs;
  ca.isig = (const double*)b_isig.p;
  ca.syn_c = (double*)b_syn.p;
  ca.chi = (double*)b_chi.p;
  // the map's chi^2 of the current model (forward, convolution, residual)
  auto map_chi2 = [&](bool nodes, double* rdst, double& chi) -> int {
    int rr = coupled_forward(c, nx, ny, d_atm, d_stokes, eqv, t1, t2, st, nodes);
    if (rr) return rr;
    ca.res = rdst;
    for (int b = 0; b < 4; ++b) ca.rowstk[b] = c->lm.rowstk[b];
    ca.inu = (double)nfreq;
    hipLaunchKernelGGL(coupled_resid_kernel, dim3((unsigned)((ncol + 255) / 256)), dim3(256), 0, st, ca);
    hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(256), 0, st, (const double*)ca.chi, ncol, (double*)b_sum.p);
    HIPCHK(c, hipMemcpyAsync(&chi, b_sum.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(c, hipStreamSynchronize(st));
    chi /= (double)ncol;
    return FZ_OK;
  };
  int total_it = 0;
  const int cyc0 = std::min(std::max(1, ctl->first_cycle), maxiter);
  for (int cyc = cyc0; cyc <= maxiter; ++cyc) {
    fz_inversion inv;
    std::memset(&inv, 0, sizeof(inv));
    for (int p = 0; p < 8; ++p) {
      if (!ctl->atmpar[p]) continue;
      const int vmax = ctl->nslb_max[p] > 0 ? std::min(ctl->nslb_max[p], nz) : nz;
      inv.atmpar[p] = 1;
      inv.nodes[p] = std::min(njevals(p + 1, cyc, maxiter, cycpow, nz), vmax);
      inv.pen_typ[p] = ctl->pen_typ[p];
      inv.pen_alp[p] = ctl->pen_alp[p];
    }
    for (int s = 0; s < 4; ++s) inv.invstk[s] = ctl->invstk[s];
    inv.regul = ctl->regul;
    inv.solver = ctl->solver > 0 ? ctl->solver : 1;
    inv.node_expansion = ctl->node_expansion > 0 ? ctl->node_expansion : 1;
    inv.maxsteps = maxsteps;
    inv.svdtol = ctl->svdtol;
    r = fz_set_inversion(c, &inv, nullptr, nullptr);
    if (r) return r;
    // SET_TAU with its assists, then the smoothing of the start model
    if (!ctl->atmpar[1] && !ctl->atmpar[7]) {
      if (cyc == cyc0 && ctl->assist) {
        r = run_assist(c, ncol, d_obs, ctl->assist & 15, d_atm, st);
        if (r) return r;
      }
      r = fz_forward_dev(c, ncol, d_atm, FZ_RF_NONE, d_stokes, nullptr, nullptr, stream);
      if (r) return r;
    }
    if (ctl->smoothing) {
      for (int p = 0; p < 8; ++p) {
        if (!ctl->atmpar[p]) continue;
        float* rc = d_atm + (size_t)rowof[p] * nz * ncol;
        double *s0 = (double*)b_s0.p, *s1 = (double*)b_s1.p;
        hipLaunchKernelGGL(to_double_kernel, dim3(grow), dim3(256), 0, st, rc, s0, (long)nz * ncol);
        const int ext[3] = {nx, ny, nz};
        for (int ax = 0; ax < 3; ++ax) {
          if (ext[ax] <= 4) continue;
          hipLaunchKernelGGL(smooth_axis_kernel, dim3(grow), dim3(256), 0, st, s0, s1, nz, ny, nx, ax);
          std::swap(s0, s1);
        }
        hipLaunchKernelGGL(from_double_kernel, dim3(grow), dim3(256), 0, st, s0, rc, rc, (long)nz * ncol);
      }
    }
    HIPCHK(c, hipGetLastError());
    const size_t neqv = nrow * (size_t)c->lm.np;
    double chibest = 1.0e29, lam = 10.0, steps = 0.0, precyc = 0.0;
    for (int it = 0; it < itcap; ++it) {
      double chi = 0.0;
      r = map_chi2(true, res, chi);
      if (r) return r;
      ++total_it;
      // UPDATE_LAMBDA on the map's chi^2
      const bool accept = chi < chibest;
      if (accept) {
        if ((chibest - chi) > 0.01 * chibest) steps = std::max(0.0, steps - 1.0);
        else steps = steps + 1.0;
        chibest = chi;
        lam = lam / std::sqrt(10.0);
        hipLaunchKernelGGL(copy_f32_kernel, dim3(gatm), dim3(256), 0, st, (const float*)d_atm, best, (long)natm);
        HIPCHK(c, hipMemcpyAsync(eqvb, eqv, sizeof(float) * neqv, hipMemcpyDeviceToDevice, st));
        HIPCHK(c, hipMemcpyAsync(resb, res, sizeof(double) * nrow, hipMemcpyDeviceToDevice, st));
      } else {
        if (std::fabs(precyc - 1.0) < 1.0e-2) {
          precyc = 0.0;
          lam = lam * 3.0;
        } else {
          lam = lam * 10.0;
        }
        steps = steps + 1.0;
        hipLaunchKernelGGL(copy_f32_kernel, dim3(gatm), dim3(256), 0, st, (const float*)best, d_atm, (long)natm);
      }
      lam = std::max(1.0e-2, lam);
      // MAKE_DECISION (invert3d.f90:820-859) on the map's step count
      if (steps >= (double)std::max(1, maxsteps - (maxiter - cyc))) break;
      // gradient residual: the adjoint PSF convolution of the best residual
      hipLaunchKernelGGL((transpose_kernel<double, float>), dim3((unsigned)((nfreq + 31) / 32), (unsigned)((ncol + 31) / 32)),
                         dim3(256), 0, st, (const double*)resb, t1, (long)ncol, (long)nfreq);
      launch_psf(c, nx, ny, nfreq, t1, t2, 1, st);
      hipLaunchKernelGGL((transpose_kernel<float, double>), dim3((unsigned)((ncol + 31) / 32), (unsigned)((nfreq + 31) / 32)),
                         dim3(256), 0, st, (const float*)t2, gres, (long)nfreq, (long)ncol);
      HIPCHK(c, hipGetLastError());
      LmArgs a = c->lm;
      a.ncol = ncol;
      a.obs = d_obs;
      a.stokes = d_stokes;
      a.syn_d = (const double*)b_syn.p;
      a.best_syn = nullptr;
      a.sla = nullptr;
      a.eqv = eqvb;
      a.eqv_best = nullptr;
      a.isigmap = (const double*)b_isig.p;
      a.isig_stride = 0;
      a.atm = d_atm;
      a.atm_best = nullptr;
      a.done = nullptr;
      a.delta = nullptr;
      a.pix_of = nullptr;
      a.poff = nullptr;
      a.gres = gres;
      a.hscale = c->taps_sq;
      a.ext_lambda = lam;
      r = launch_lm(c, a, ncol, st);
      if (r) return r;
    }
    // END_CYCLE: current := best
    hipLaunchKernelGGL(copy_f32_kernel, dim3(gatm), dim3(256), 0, st, (const float*)best, d_atm, (long)natm);
    HIPCHK(c, hipGetLastError());
  }
  // the convolved synthesis of the final model and each pixel's chi^2
  double chi = 0.0;
  r = map_chi2(false, res, chi);
  if (r) return r;
  hipLaunchKernelGGL((transpose_kernel<float, float>), dim3((unsigned)((ncol + 31) / 32), (unsigned)((4 * numw + 31) / 32)),
                     dim3(256), 0, st, (const float*)t2, d_stokes, (long)(4 * numw), (long)ncol);
  if (d_chi2) HIPCHK(c, hipMemcpyAsync(d_chi2, b_chi.p, sizeof(double) * ncol, hipMemcpyDeviceToDevice, st));
  HIPCHK(c, hipStreamSynchronize(st));
  if (iterations) *iterations = total_it;
  return FZ_OK;
}

}  // extern "C"

}  // extern "C"

// INVERT3D on the host cubes: upload, fz_invert3d_dev or (coupled) fz_coupled_invert3d_dev, download
static int invert3d_host(fz_ctx* c, int nx, int ny, float* tem3d, float* pg3d, float* rho3d, float* pel3d,
                         float* mw3d, float* bx3d, float* by3d, float* bz3d, const float* vx3d, const float* vy3d,
                         float* vz3d, float* tau3d5, const double* obs3d, const fz_invert_control* ctl,
                         double* syn3d, double* chi2, int* iterations, bool coupled) {
  if (!c || !c->configured || nx < 1 || ny < 1 || !obs3d || !ctl || !syn3d) return FZ_EARG;
  if (c->win_on) return set_err(c, FZ_ECONFIG, "per-pixel windows: the cubes of fz_invert3d are dense");
  const int nz = c->cfg.nz, numw = c->cfg.numw, ncol = nx * ny;
  int nstk = 0;
  for (int s = 0; s < 4; ++s) nstk += ctl->invstk[s] != 0;
  const size_t nfreq = (size_t)nstk * numw;
  float* cubes[NATM] = {tem3d, pg3d, rho3d, pel3d, mw3d, bx3d, by3d, bz3d, (float*)vx3d, (float*)vy3d, vz3d, tau3d5};
  HIPCHK(c, hipSetDevice(c->device));
  DevBuf b_atm, b_tmp, b_obs, b_st, b_chi;
  const size_t cube = sizeof(float) * (size_t)nz * ncol;
  HIPCHK(c, hipMalloc(&b_atm.p, cube * NATM));
  HIPCHK(c, hipMalloc(&b_tmp.p, cube));
  HIPCHK(c, hipMalloc(&b_obs.p, sizeof(double) * nfreq * ncol));
  HIPCHK(c, hipMalloc(&b_st.p, sizeof(float) * 4 * numw * (size_t)ncol));
  HIPCHK(c, hipMalloc(&b_chi.p, sizeof(double) * ncol));
  float* d_atm = (float*)b_atm.p;
  const unsigned tb = 256, tg = (unsigned)(((long)nz * ncol + tb - 1) / tb);
  // the cubes (NZ,NY,NX) are column-major with column index y + ny*x, the
  // same column order as the device layout [parameter][height][column]
  for (int p = 0; p < NATM; ++p) {
    HIPCHK(c, hipMemcpy(b_tmp.p, cubes[p], cube, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(cube_to_soa, dim3(tg), dim3(tb), 0, 0, (const float*)b_tmp.p, d_atm + (size_t)p * nz * ncol,
                       nz, ncol);
  }
  // OBS3D(NFREQ,NY,NX) is already [column][NFREQ]
  HIPCHK(c, hipMemcpy(b_obs.p, obs3d, sizeof(double) * nfreq * ncol, hipMemcpyHostToDevice));
  const int rc = coupled ? fz_coupled_invert3d_dev(c, nx, ny, d_atm, (const double*)b_obs.p, ctl, (float*)b_st.p,
                                                    (double*)b_chi.p, iterations, nullptr)
                         : fz_invert3d_dev(c, nx, ny, d_atm, (const double*)b_obs.p, ctl, (float*)b_st.p,
                                           (double*)b_chi.p, iterations, nullptr);
  if (rc) return rc;
  // the model (every parameter the inversion or the EOS changed) back to the cubes
  const int outp[] = {A_T, A_PG, A_RHO, A_PEL, A_MU, A_BX, A_BY, A_BZ, A_VZ, A_TAU};
  for (int p : outp) {
    hipLaunchKernelGGL(soa_to_cube, dim3(tg), dim3(tb), 0, 0, d_atm + (size_t)p * nz * ncol, (float*)b_tmp.p, nz,
                       ncol);
    HIPCHK(c, hipMemcpy(cubes[p], b_tmp.p, cube, hipMemcpyDeviceToHost));
  }
  std::vector<float> st((size_t)4 * numw * ncol);
  HIPCHK(c, hipMemcpy(st.data(), b_st.p, sizeof(float) * st.size(), hipMemcpyDeviceToHost));
  for (size_t i = 0; i < (size_t)4 * numw * ncol; ++i) syn3d[i] = (double)st[i];
  if (chi2) HIPCHK(c, hipMemcpy(chi2, b_chi.p, sizeof(double) * ncol, hipMemcpyDeviceToHost));
  return FZ_OK;
}

extern "C" {

int fz_invert3d(fz_ctx* c, int nx, int ny, float* tem3d, float* pg3d, float* rho3d, float* pel3d, float* mw3d,
                float* bx3d, float* by3d, float* bz3d, const float* vx3d, const float* vy3d, float* vz3d,
                float* tau3d5, const double* obs3d, const fz_invert_control* ctl, double* syn3d, double* chi2,
                int* iterations) {
  return invert3d_host(c, nx, ny, tem3d, pg3d, rho3d, pel3d, mw3d, bx3d, by3d, bz3d, vx3d, vy3d, vz3d, tau3d5, obs3d,
                       ctl, syn3d, chi2, iterations, false);
}

int fz_coupled_invert3d(fz_ctx* c, int nx, int ny, float* tem3d, float* pg3d, float* rho3d, float* pel3d,
                        float* mw3d, float* bx3d, float* by3d, float* bz3d, const float* vx3d, const float* vy3d,
                        float* vz3d, float* tau3d5, const double* obs3d, const fz_invert_control* ctl, double* syn3d,
                        double* chi2, int* iterations) {
  return invert3d_host(c, nx, ny, tem3d, pg3d, rho3d, pel3d, mw3d, bx3d, by3d, bz3d, vx3d, vy3d, vz3d, tau3d5, obs3d,
                       ctl, syn3d, chi2, iterations, true);
}

}  // extern "C"

// ---------------------------------------------------------------- learned initial model
namespace {

uint64_t splitmix64(uint64_t& x) {
  uint64_t z = (x += 0x9e3779b97f4a7c15ULL);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

// Work buffers for n rows of the forward pass and, with grad, of the gradient.
int mlp_work(fz_ctx* c, int n, bool grad) {
  MlpState& M = c->mlp;
  bool ok = true;
  if (M.cap < n) {
    M.release_forward();
    M.cap = n;
    ok = hipMalloc(&M.X, sizeof(bf16) * frag_size(n, M.nin)) == hipSuccess &&
         hipMalloc(&M.act, sizeof(bf16) * M.act_stride() * M.nl) == hipSuccess;
    if (!ok) M.release_forward();
  }
  if (ok && grad && M.gcap < n) {
    M.release_gradient();
    M.gcap = n;
    ok = hipMalloc(&M.XT, sizeof(bf16) * frag_size(M.nin, n)) == hipSuccess &&
         hipMalloc(&M.actT, sizeof(bf16) * M.actt_stride() * M.nl) == hipSuccess &&
         hipMalloc(&M.dZ, sizeof(bf16) * 2 * M.dz_stride()) == hipSuccess &&
         hipMalloc(&M.dZT, sizeof(bf16) * M.dzt_stride() * (M.nl + 1)) == hipSuccess &&
         hipMalloc(&M.csum, sizeof(float) * M.csum_stride() * (M.nl + 1)) == hipSuccess &&
         hipMalloc(&M.partial, sizeof(float) * 4 * (pad32(n) / 32) * (pad32(M.nout) / 32)) == hipSuccess;
    if (!ok) M.release_gradient();
  }
  return ok ? FZ_OK : set_err(c, FZ_ENOMEM, "device allocation failed (network work buffers)");
}

// A product of the network: D[m][n], A [N][K] and B [M][K] in operand order
GemmArgs mlp_gemm(const bf16* A, const bf16* B, int M, int N, int K) {
  GemmArgs g;
  memset(&g, 0, sizeof(g));
  g.A = A;
  g.B = B;
  g.M = M;
  g.N = N;
  g.ks = pad32(K) / 32;
  g.tn = pad32(N) / 32;
  return g;
}

template <int MODE>
void mlp_layer(GemmArgs g, const LossArgs& ls, hipStream_t st) {
  const long m64 = (g.M + 63) / 64, n64 = (g.N + 63) / 64;
  if (MODE != MLP_LOSS && m64 * n64 >= 512) {
    g.tn = (int)n64;
    hipLaunchKernelGGL((mlp_layer_kernel<MODE, 2>), dim3((unsigned)(m64 * n64)), dim3(256), 0, st, g, ls);
  } else {
    hipLaunchKernelGGL((mlp_layer_kernel<MODE, 1>), dim3((unsigned)(pad32(g.M) / 32 * g.tn)), dim3(256), 0, st, g, ls);
  }
}

// Forward pass of n rows already in M.X: the hidden layers (with their
// transposes for the gradient) and, when y is given, the output (standardised).
void mlp_forward_rows(MlpState& M, int n, float* y, bool grad, hipStream_t st) {
  const LossArgs none = {};
  for (int l = 0; l < M.nl + (y ? 1 : 0); ++l) {
    GemmArgs g = mlp_gemm(M.wb + M.shape.wb[l], l == 0 ? M.X : M.act + (l - 1) * M.act_stride(), n, M.dout[l],
                          M.din[l]);
    g.bias = M.w + M.boff[l];
    if (l < M.nl) {
      g.Cb = M.act + l * M.act_stride();
      if (grad) g.CbT = M.actT + l * M.actt_stride();
      mlp_layer<MLP_HIDDEN>(g, none, st);
    } else {
      g.Cf = y;
      mlp_layer<MLP_OUT>(g, none, st);
    }
  }
}

// Output layer, loss and gradient of the parameters for n of a batch's rows
// (targets t, rows gathered by idx when given): their part of the mean squared
// error into loss[0], or added to it.
void mlp_backward_rows(MlpState& M, int n, int rows, bool add, const float* d_t, const int32_t* d_idx, float* loss,
                       float* grad, hipStream_t st) {
  const float* tmean = M.norms + 2 * M.nin;
  LossArgs ls = {d_t, tmean, tmean + M.nout, d_idx, M.partial, rows};
  DwArgs dw;
  memset(&dw, 0, sizeof(dw));
  const bf16* dz = nullptr;
  for (int l = M.nl; l >= 0; --l) {
    bf16* out = M.dZ + (l & 1) * M.dz_stride();
    bf16* outT = M.dZT + l * M.dzt_stride();
    GemmArgs g;
    if (l == M.nl)         // Y = A W^T + b and dY from it
      g = mlp_gemm(M.wb + M.shape.wb[l], M.act + (l - 1) * M.act_stride(), n, M.dout[l], M.din[l]);
    else                   // dZ_l[m][k] = sum_o dZ_(l+1)[m][o] W_(l+1)[o][k], times ReLU'
      g = mlp_gemm(M.wb + M.shape.wt[l + 1], dz, n, M.dout[l], M.dout[l + 1]);
    g.bias = M.w + M.boff[l];
    g.mask = l < M.nl ? M.act + l * M.act_stride() : nullptr;
    g.Cb = out;
    g.CbT = outT;
    g.csum = M.csum + l * M.csum_stride();
    if (l == M.nl)
      mlp_layer<MLP_LOSS>(g, ls, st);
    else
      mlp_layer<MLP_DACT>(g, ls, st);
    dz = out;
    // dW_l[o][k] = sum_m dZ_l[m][o] A_l[m][k]
    GemmArgs& h = dw.g[l];
    h = mlp_gemm(l == 0 ? M.XT : M.actT + (l - 1) * M.actt_stride(), outT, M.dout[l], M.din[l], n);
    h.Cf = grad + M.woff[l];
    dw.csum[l] = g.csum;
    dw.bg[l] = grad + M.boff[l];
  }
  dw.n = M.nl + 1;
  dw.nparts = pad32(n) / 16;
  int nb = 0;
  for (int l = 0; l <= M.nl; ++l) {
    dw.g[l].tile0 = nb;
    nb += pad32(M.dout[l]) / 32 * dw.g[l].tn;
  }
  for (int l = 0; l <= M.nl; ++l) {
    dw.blk0[l] = nb;
    nb += (M.dout[l] + 15) / 16;
  }
  dw.loss_blk = nb;
  dw.nloss = 4 * (pad32(n) / 32) * (pad32(M.nout) / 32);
  dw.lpart = M.partial;
  dw.lscale = (float)((long)rows * M.nout);
  dw.loss = loss;
  dw.add = add;
  hipLaunchKernelGGL(mlp_dw_kernel, dim3((unsigned)(nb + 1)), dim3(256), 0, st, dw);
}

int mlp_input(fz_ctx* c, int n, const float* d_x, const double* d_xd, const int32_t* d_idx, bool grad,
              hipStream_t st) {
  MlpState& M = c->mlp;
  const size_t np = frag_size(n, M.nin) / 8 * (grad ? 2 : 1);
  hipLaunchKernelGGL(mlp_input_kernel, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, st, n, M.nin, d_x, d_xd,
                     d_idx, (const float*)M.norms, (const float*)(M.norms + M.nin), M.X, grad ? M.XT : nullptr);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// Bytes of LDS of mlp_infer_kernel for tiles of R rows
size_t mlp_infer_lds(const MlpState& M, int R) {
  const size_t pitch = std::max(pad32(M.nin), pad32(M.nh)) + 8;
  return std::max(sizeof(bf16) * R * pitch, sizeof(float) * 2 * R * M.nout);
}

constexpr size_t MLP_LDS = 144 * 1024;

template <int MF>
int mlp_infer_launch(fz_ctx* c, const InferArgs& a, hipStream_t st) {
  const size_t lds = mlp_infer_lds(c->mlp, 16 * MF);
  HIPCHK(c, hipFuncSetAttribute((const void*)mlp_infer_kernel<MF>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)MLP_LDS));
  hipLaunchKernelGGL((mlp_infer_kernel<MF>), dim3((unsigned)((a.n + 16 * MF - 1) / (16 * MF))), dim3(512), lds, st,
                     c->mlp.shape, a);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

// All layers in one launch, where the network fits the kernel (widest layer
// and LDS): 16 rows a workgroup while these fill no more than the chip, else 32, else
// 64, so that the weights are read through as few CUs' ports as keep all busy.
bool mlp_infer_fits(const MlpState& M) { return M.nh <= MLP_INFER_NH && mlp_infer_lds(M, 16) <= MLP_LDS; }

int mlp_infer(fz_ctx* c, int n, const float* d_x, const double* d_xd, float* d_y, float* d_atm, hipStream_t st) {
  MlpState& M = c->mlp;
  InferArgs a;
  a.n = n;
  a.pitch = std::max(pad32(M.nin), pad32(M.nh)) + 8;
  a.xf = d_x;
  a.xd = d_xd;
  a.mean = M.norms;
  a.sdev = M.norms + M.nin;
  a.tmean = M.norms + 2 * M.nin;
  a.tstd = a.tmean + M.nout;
  a.w = M.w;
  a.wb = M.wb;
  a.y = d_y;
  a.coefs = M.coefs;
  a.atm = d_atm;
  if (n > 8192 && mlp_infer_lds(M, 64) <= MLP_LDS) return mlp_infer_launch<4>(c, a, st);
  if (n > 4096 && mlp_infer_lds(M, 32) <= MLP_LDS) return mlp_infer_launch<2>(c, a, st);
  return mlp_infer_launch<1>(c, a, st);
}

}  // namespace

extern "C" {

int fz_mlp_create(fz_ctx* c, int nin, int nhidden, int nlayers, int nodes, uint64_t seed) {
  if (!c || !c->configured || nin < 1 || nhidden < 1 || nlayers < 1 || nlayers > 6 || nodes < 1 ||
      nodes > MLP_MAXNODE || nodes > c->cfg.nz)
    return set_err(c, FZ_EARG, "network shape outside limits");
  HIPCHK(c, hipSetDevice(c->device));
  c->mlp.release();
  MlpState& M = c->mlp;
  M.nin = nin;
  M.nh = nhidden;
  M.nl = nlayers;
  M.nj = nodes;
  M.nout = MLP_NQ * nodes;
  M.nz = c->cfg.nz;
  long off = 0;
  for (int l = 0; l <= nlayers; ++l) {
    M.din[l] = l == 0 ? nin : nhidden;
    M.dout[l] = l == nlayers ? M.nout : nhidden;
    M.woff[l] = off;
    off += (long)M.din[l] * M.dout[l];
    M.boff[l] = off;
    off += M.dout[l];
  }
  M.np = off;
  size_t nwb = 0;
  MlpShape& S = M.shape;
  memset(&S, 0, sizeof(S));
  S.nl = nlayers;
  S.nin = nin;
  S.nout = M.nout;
  S.nj = nodes;
  S.nz = M.nz;
  for (int l = 0; l <= nlayers; ++l) {
    S.din[l] = M.din[l];
    S.dout[l] = M.dout[l];
    S.woff[l] = M.woff[l];
    S.boff[l] = M.boff[l];
    S.wb[l] = (long)nwb;
    nwb += frag_size(M.dout[l], M.din[l]);
    S.wt[l] = (long)nwb;
    nwb += frag_size(M.din[l], M.dout[l]);
  }
  // He-uniform weights for ReLU layers (bound sqrt(6 / fan_in)), the output
  // layer scaled by 1/4; zero biases
  std::vector<float> w(off, 0.f);
  uint64_t s = seed;
  for (int l = 0; l <= nlayers; ++l) {
    const double b = std::sqrt(6.0 / M.din[l]) * (l == nlayers ? 0.25 : 1.0);
    for (long i = 0; i < (long)M.din[l] * M.dout[l]; ++i)
      w[M.woff[l] + i] = (float)(b * (2.0 * ((splitmix64(s) >> 11) * (1.0 / 9007199254740992.0)) - 1.0));
  }
  bool ok = hipMalloc(&M.w, sizeof(float) * off) == hipSuccess && hipMalloc(&M.g, sizeof(float) * off) == hipSuccess &&
            hipMalloc(&M.m1, sizeof(float) * off) == hipSuccess &&
            hipMalloc(&M.m2, sizeof(float) * off) == hipSuccess && hipMalloc(&M.wb, sizeof(bf16) * nwb) == hipSuccess &&
            hipMalloc(&M.norms, sizeof(float) * 2 * (nin + M.nout)) == hipSuccess &&
            hipMalloc(&M.pinv, sizeof(double) * nodes * M.nz) == hipSuccess &&
            hipMalloc(&M.coefs, sizeof(double) * nodes * M.nz) == hipSuccess &&
            hipMalloc(&M.loss, sizeof(float) * 4) == hipSuccess;
  if (!ok) {
    M.release();
    return set_err(c, FZ_ENOMEM, "device allocation failed (network)");
  }
  HIPCHK(c, hipMemcpy(M.w, w.data(), sizeof(float) * off, hipMemcpyHostToDevice));
  HIPCHK(c, hipMemset(M.m1, 0, sizeof(float) * off));
  HIPCHK(c, hipMemset(M.m2, 0, sizeof(float) * off));
  HIPCHK(c, hipMemset(M.g, 0, sizeof(float) * off));
  HIPCHK(c, hipMemset(M.wb, 0, sizeof(bf16) * nwb));   // the padding of K stays zero
  hipLaunchKernelGGL(mlp_to_bf16_kernel, dim3((unsigned)((off + 255) / 256)), dim3(256), 0, 0, off, S,
                     (const float*)M.w, M.wb);
  HIPCHK(c, hipGetLastError());
  std::vector<float> nrm(2 * (nin + M.nout));
  for (int i = 0; i < nin; ++i) {
    nrm[i] = 0.f;
    nrm[nin + i] = 1.f;
  }
  for (int i = 0; i < M.nout; ++i) {
    nrm[2 * nin + i] = 0.f;
    nrm[2 * nin + M.nout + i] = 1.f;
  }
  HIPCHK(c, hipMemcpy(M.norms, nrm.data(), sizeof(float) * nrm.size(), hipMemcpyHostToDevice));
  // hat basis of GET_INT_COEFS (fz_int_coefs: node-major [nj][nz]) as
  // cf[k * nj + j], and its least-squares pseudo-inverse pv[j * nz + k]
  std::vector<double> cf((size_t)M.nz * nodes), pv((size_t)nodes * M.nz);
  {
    std::vector<double> cj((size_t)M.nz * nodes);
    const int r0 = fz_int_coefs(M.nz, nodes, cj.data());
    if (r0) return set_err(c, r0, "node basis");
    for (int j = 0; j < nodes; ++j)
      for (int k = 0; k < M.nz; ++k) cf[(size_t)k * nodes + j] = cj[(size_t)j * M.nz + k];
  }
  {
    // normal equations (C^T C) P = C^T, solved by Gauss-Jordan on nodes x nodes
    const int nj = nodes, nz = M.nz;
    std::vector<double> a((size_t)nj * nj, 0.0), inv((size_t)nj * nj, 0.0);
    for (int i = 0; i < nj; ++i)
      for (int j = 0; j < nj; ++j)
        for (int k = 0; k < nz; ++k) a[i * nj + j] += cf[(size_t)k * nj + i] * cf[(size_t)k * nj + j];
    for (int i = 0; i < nj; ++i) inv[i * nj + i] = 1.0;
    for (int p = 0; p < nj; ++p) {
      int piv = p;
      for (int i = p + 1; i < nj; ++i)
        if (std::fabs(a[i * nj + p]) > std::fabs(a[piv * nj + p])) piv = i;
      if (a[piv * nj + p] == 0.0) return set_err(c, FZ_ECONFIG, "singular node basis");
      for (int j = 0; j < nj; ++j) {
        std::swap(a[p * nj + j], a[piv * nj + j]);
        std::swap(inv[p * nj + j], inv[piv * nj + j]);
      }
      const double d = a[p * nj + p];
      for (int j = 0; j < nj; ++j) {
        a[p * nj + j] /= d;
        inv[p * nj + j] /= d;
      }
      for (int i = 0; i < nj; ++i) {
        if (i == p) continue;
        const double f = a[i * nj + p];
        for (int j = 0; j < nj; ++j) {
          a[i * nj + j] -= f * a[p * nj + j];
          inv[i * nj + j] -= f * inv[p * nj + j];
        }
      }
    }
    for (int j = 0; j < nj; ++j)
      for (int k = 0; k < nz; ++k) {
        double v = 0.0;
        for (int i = 0; i < nj; ++i) v += inv[j * nj + i] * cf[(size_t)k * nj + i];
        pv[(size_t)j * nz + k] = v;
      }
  }
  HIPCHK(c, hipMemcpy(M.coefs, cf.data(), sizeof(double) * cf.size(), hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(M.pinv, pv.data(), sizeof(double) * pv.size(), hipMemcpyHostToDevice));
  M.on = true;
  return FZ_OK;
}

int64_t fz_mlp_size(const fz_ctx* c) {
  if (!c || !c->mlp.on) return -1;
  return c->mlp.np + 2 * (c->mlp.nin + c->mlp.nout);
}

int fz_mlp_get_params(fz_ctx* c, float* params) {
  if (!c || !c->mlp.on || !params) return FZ_EARG;
  MlpState& M = c->mlp;
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipMemcpy(params, M.w, sizeof(float) * M.np, hipMemcpyDeviceToHost));
  HIPCHK(c, hipMemcpy(params + M.np, M.norms, sizeof(float) * 2 * (M.nin + M.nout), hipMemcpyDeviceToHost));
  return FZ_OK;
}

int fz_mlp_set_params(fz_ctx* c, const float* params) {
  if (!c || !c->mlp.on || !params) return FZ_EARG;
  MlpState& M = c->mlp;
  HIPCHK(c, hipSetDevice(c->device));
  for (long i = 0; i < M.np + 2 * (M.nin + M.nout); ++i)
    if (!std::isfinite(params[i])) return set_err(c, FZ_EARG, "non-finite network parameter");
  HIPCHK(c, hipMemcpy(M.w, params, sizeof(float) * M.np, hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(M.norms, params + M.np, sizeof(float) * 2 * (M.nin + M.nout), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(mlp_to_bf16_kernel, dim3((unsigned)((M.np + 255) / 256)), dim3(256), 0, 0, M.np,
                     M.shape, (const float*)M.w, M.wb);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipMemset(M.m1, 0, sizeof(float) * M.np));
  HIPCHK(c, hipMemset(M.m2, 0, sizeof(float) * M.np));
  M.step = 0;
  return FZ_OK;
}

int fz_mlp_fit_norms_dev(fz_ctx* c, int n, const float* d_x, const float* d_t, void* stream) {
  if (!c || !c->mlp.on || n < 2 || !d_x || !d_t) return FZ_EARG;
  MlpState& M = c->mlp;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  hipLaunchKernelGGL(mlp_stats_kernel, dim3((unsigned)((M.nin + 63) / 64)), dim3(64), 0, st, n, M.nin, d_x, M.norms,
                     M.norms + M.nin);
  hipLaunchKernelGGL(mlp_stats_kernel, dim3((unsigned)((M.nout + 63) / 64)), dim3(64), 0, st, n, M.nout, d_t,
                     M.norms + 2 * M.nin, M.norms + 2 * M.nin + M.nout);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_mlp_targets_dev(fz_ctx* c, int ncol, const float* d_atm, float* d_t, void* stream) {
  if (!c || !c->mlp.on || ncol < 1 || !d_atm || !d_t) return FZ_EARG;
  if (c->cfg.nz != c->mlp.nz) return set_err(c, FZ_ECONFIG, "height grid changed since fz_mlp_create");
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  hipLaunchKernelGGL(mlp_targets_kernel, dim3((unsigned)((ncol + 127) / 128)), dim3(128), 0, st, ncol, c->mlp.nz,
                     c->mlp.nj, d_atm, (const double*)c->mlp.pinv, d_t);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_mlp_forward_dev(fz_ctx* c, int n, const float* d_x, const double* d_xd, float* d_y, void* stream) {
  if (!c || !c->mlp.on || n < 1 || (!d_x && !d_xd) || !d_y) return FZ_EARG;
  MlpState& M = c->mlp;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  // (one launch reads some rows after it has written others: outputs in the place of
  // inputs go by layers, whose first takes every row)
  const char *x = d_x ? (const char*)d_x : (const char*)d_xd, *y = (const char*)d_y;
  const bool apart = y + sizeof(float) * (size_t)n * M.nout <= x ||
                     x + (d_x ? sizeof(float) : sizeof(double)) * (size_t)n * M.nin <= y;
  if (apart && mlp_infer_fits(M)) return mlp_infer(c, n, d_x, d_xd, d_y, nullptr, st);
  const int chunk = 65536;
  int r = mlp_work(c, std::min(n, chunk), false);
  if (r) return r;
  for (int r0 = 0; r0 < n; r0 += M.cap) {
    const int nr = std::min(M.cap, n - r0);
    r = mlp_input(c, nr, d_x ? d_x + (size_t)r0 * M.nin : nullptr, d_xd ? d_xd + (size_t)r0 * M.nin : nullptr,
                  nullptr, false, st);
    if (r) return r;
    mlp_forward_rows(M, nr, d_y + (size_t)r0 * M.nout, false, st);
  }
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_mlp_gradient_dev(fz_ctx* c, int n, const float* d_x, const float* d_t, const int32_t* d_idx, float* d_loss,
                        float* d_grad, void* stream) {
  if (!c || !c->mlp.on || n < 1 || !d_x || !d_t) return FZ_EARG;
  MlpState& M = c->mlp;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  // a million rows at a time (15 GB of work buffers for 448-512-512-512-20),
  // their sums added up
  const int chunk = 1 << 20;
  int r = mlp_work(c, std::min(n, chunk), true);
  if (r) return r;
  for (int r0 = 0; r0 < n; r0 += std::min(chunk, n - r0)) {
    const int nr = std::min(chunk, n - r0);
    const float *x = d_idx ? d_x : d_x + (size_t)r0 * M.nin, *t = d_idx ? d_t : d_t + (size_t)r0 * M.nout;
    const int32_t* idx = d_idx ? d_idx + r0 : nullptr;
    r = mlp_input(c, nr, x, nullptr, idx, true, st);
    if (r) return r;
    mlp_forward_rows(M, nr, nullptr, true, st);
    mlp_backward_rows(M, nr, n, r0 > 0, t, idx, d_loss ? d_loss : M.loss, d_grad ? d_grad : M.g, st);
  }
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_mlp_train_step_dev(fz_ctx* c, int n, const float* d_x, const float* d_t, const int32_t* d_idx, float lr,
                          float* d_loss, void* stream) {
  int r = fz_mlp_gradient_dev(c, n, d_x, d_t, d_idx, d_loss, nullptr, stream);
  if (r) return r;
  MlpState& M = c->mlp;
  const float b1 = 0.9f, b2 = 0.999f;
  ++M.step;
  const float c1 = (float)(1.0 - std::pow((double)b1, (double)M.step));
  const float c2 = (float)(1.0 - std::pow((double)b2, (double)M.step));
  hipLaunchKernelGGL(mlp_adam_kernel, dim3((unsigned)((M.np + 255) / 256)), dim3(256), 0, (hipStream_t)stream, M.np,
                     M.shape, M.w, (const float*)M.g, M.m1, M.m2, M.wb, lr, b1, b2, 1e-8f, c1, c2);
  HIPCHK(c, hipGetLastError());
  return FZ_OK;
}

int fz_learned_init_dev(fz_ctx* c, int ncol, const double* d_obs, float* d_atm, void* stream) {
  if (!c || !c->mlp.on || ncol < 1 || !d_obs || !d_atm) return FZ_EARG;
  if (c->cfg.nz != c->mlp.nz) return set_err(c, FZ_ECONFIG, "height grid changed since fz_mlp_create");
  MlpState& M = c->mlp;
  hipStream_t st = (hipStream_t)stream;
  HIPCHK(c, hipSetDevice(c->device));
  if (mlp_infer_fits(M)) {
    const int r = mlp_infer(c, ncol, nullptr, d_obs, nullptr, d_atm, st);
    if (r) return r;
    HIPCHK(c, hipStreamSynchronize(st));
    return FZ_OK;
  }
  DevBuf y;
  HIPCHK(c, hipMalloc(&y.p, sizeof(float) * (size_t)ncol * M.nout));
  int r = fz_mlp_forward_dev(c, ncol, nullptr, d_obs, (float*)y.p, stream);
  if (r) return r;
  hipLaunchKernelGGL(mlp_decode_kernel, dim3((unsigned)((ncol + 31) / 32)), dim3(256), 0, st, M.shape, ncol,
                     (const float*)y.p, (const float*)(M.norms + 2 * M.nin), (const float*)(M.norms + 2 * M.nin + M.nout),
                     (const double*)M.coefs, d_atm);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(st));
  return FZ_OK;
}

}  // extern "C"
