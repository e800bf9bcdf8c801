// FP32 per-(column, wavelength) radiative transfer pieces: Faraday-Voigt
// profiles, the evolution operator of a layer in the frame of its field and
// the gradient of the operator's action.
#pragma once
#include <hip/hip_runtime.h>

namespace fz {

// Voigt H(a,u) and Faraday-Voigt L(a,u) = Re, Im of w(u + i a) with the
// Hui, Armstrong & Wray (1978) 7/7 rational form in z = a - iu (voigt.f:17-98;
// the coefficients are real, so H is even and L odd in u without |u|).  a > 0
// always here (radiative damping is positive).  Both polynomials are expanded
// about a, P(a - iu) = sum_j P^(j)(a)/j! (-iu)^j: even powers of u give the
// real part, odd ones the imaginary part, as polynomials in u^2 with
// coefficients of the height and line alone.  opac_kernel forms those in FP64
// (VoigtPoly); a profile then takes 22 operations and a reciprocal, where
// evaluating the polynomials at the complex point takes 40.  FP32 error against
// FP64, emulated at 4e6 points of a = 1e-4 .. 30, |u| < 60: 3.3e-7 at most and 2.2e-8 rms
// (that evaluation 3.1e-7 and 2.1e-8), relative to |w| 1.0e-6 at most (2.1e-6).
constexpr int NVP = 13;   // p0..p5, q0..q6; p6 and q7 are constants
constexpr float VOIGT_A6 = .564189583562615f;

struct VoigtPoly {
  float p[6], q[7];
};

__device__ inline void voigt_poly(double a, float* v /*[NVP]*/) {
  double P[7] = {122.607931777104326, 214.382388694706425, 181.928533092181549, 93.155580458138441,
                 30.180142196210589, 5.912626209773153, .564189583562615};
  double Q[8] = {122.60793177387535, 352.730625110963558, 457.334478783897737, 348.703917719495792,
                 170.354001821091472, 53.992906912940207, 10.479857114260399, 1.0};
  // Taylor coefficients about a by repeated synthetic division
#pragma unroll
  for (int j = 0; j < 6; ++j) {
#pragma unroll
    for (int k = 5; k >= j; --k) P[k] = fma(a, P[k + 1], P[k]);
  }
#pragma unroll
  for (int j = 0; j < 7; ++j) {
#pragma unroll
    for (int k = 6; k >= j; --k) Q[k] = fma(a, Q[k + 1], Q[k]);
  }
#pragma unroll
  for (int j = 0; j < 6; ++j) v[j] = (float)P[j];
#pragma unroll
  for (int j = 0; j < 7; ++j) v[6 + j] = (float)Q[j];
}

__device__ __forceinline__ void voigt(const VoigtPoly& c, float u, float& H, float& F) {
  const float s = u * u;
  const float nr = fmaf(fmaf(fmaf(-VOIGT_A6, s, c.p[4]), s, -c.p[2]), s, c.p[0]);
  const float ni = fmaf(fmaf(c.p[5], s, -c.p[3]), s, c.p[1]);             // Im P = -u ni
  const float dr = fmaf(fmaf(fmaf(-c.q[6], s, c.q[4]), s, -c.q[2]), s, c.q[0]);
  const float di = fmaf(fmaf(c.q[5] - s, s, -c.q[3]), s, c.q[1]);         // Im Q = -u di
  const float sd = s * di;
  const float inv = __builtin_amdgcn_rcpf(fmaf(dr, dr, sd * di));
  H = fmaf(nr, dr, ni * sd) * inv;
  F = (u * inv) * fmaf(nr, di, -(ni * dr));
}

// Field geometry of one height (absorption_matrix.f90:1800-1871): |B|,
// cos and sin of the inclination, 1 +- cos^2, cos 2phi, sin 2phi.  Formed
// once per (height, column) with the opacities and stored in the per-height
// record, so the radiative transfer reads it instead of forming it in
// every lane of the column.
struct Geo {
  float B, cg, sg, sgf, cgf, c2p, s2p;
};

__device__ __forceinline__ Geo geometry(float bx, float by, float bz) {
  // absorption_matrix.f90:1800-1871
  Geo g;
  const float bt2 = bx * bx + by * by, b2 = bt2 + bz * bz;
  g.B = sqrtf(b2);
  if (g.B > 0.f) {
    g.cg = bz / g.B;
    g.sg = sqrtf(bt2) / g.B;
    g.cgf = 1.f + bz * bz / b2;
    g.sgf = 1.f - bz * bz / b2;
  } else {
    g.cg = 0.f; g.sg = 0.f; g.cgf = 1.f; g.sgf = 1.f;
  }
  if (bt2 > 0.f) {
    g.c2p = (bx * bx - by * by) / bt2;
    g.s2p = 2.f * bx * by / bt2;
  } else {
    g.c2p = 0.f; g.s2p = 0.f;
  }
  return g;
}

// Frame of a layer.  Every line and every direction but the azimuth moves Q
// and U along (cos 2phi, sin 2phi), so in the (Q, U) axes turned by 2phi the
// propagation matrix has five elements, (eta_I, eta_q, eta_V, rho_q, rho_V),
// and the vectors e = (eta_q, 0, eta_V), r = (rho_q, 0, rho_V) no second
// component.  Stokes vectors are turned into the frame, the operator's part
// beyond A times the identity is applied there, and the result turned back;
// the part A * 1 is applied unturned, so that a transparent layer does not
// pick up the rounding of cos^2 + sin^2.
struct Five {
  float I, q, V, qF, VF;
};

// Evolution operator of a constant-property layer, O = exp(-K dz), in the
// closed form of Landi Degl'Innocenti & Landi Degl'Innocenti (1985)
// (rtesolver.f90:269-473).  Written for FP32: all propagation-matrix elements
// are scaled by dz first (optical thicknesses), the two eigen-parameters are
// formed without cancellation (lambda1*lambda2 = |eta.rho|), and the
// exp(-eta_I dz) factor is folded into cosh/sinh so nothing overflows.
//   O = A*1 + P(alpha, omega) + D4 * M4raw
// with alpha = -(ga e + gb r), omega = -(gb e - ga r).
//
// Near-degenerate polarisation eigenvalues.  The closed form divides by
// th = sqrt(d^2 + 4 (e.r)^2) and by l1, l2; when th is small the terms of
// the directional derivatives grow like 1/th^1.5 and cancel, and in FP32 the
// error grows like eps (s0/th)^2 (s0 = (e.e + r.r)/2).  The four coefficient
// functions the operator needs are entire functions of d and q = (e.r)^2:
// with x, y the roots of z^2 - d z - q (x = l1^2, y = -l2^2),
//   A  e^ei = (cosh l1 + cos l2)/2            = 1/2 sum_n P_n / (2n)!
//   D4 e^ei = (cosh l1 - cos l2)/th           = sum_{n>=1} H_{n-1} / (2n)!
//   ga e^ei = (l1 sinh l1 + l2 sin l2)/th     = sum_n H_n / (2n+1)!
//   gb e^ei = e.r (sinh l1/l1 - sin l2/l2)/th = e.r sum_{n>=1} H_{n-1} / (2n+1)!
// where H_n = sum_{i<=n} x^i y^(n-i) follows H_n = d H_{n-1} + q H_{n-2}
// (H_0 = 1, H_1 = d) and P_n = x^n + y^n = 2 H_n - d H_{n-1}.  With
// dP_n/dd = n H_{n-1}, dP_n/dq = n H_{n-2} and dH_n/dq = dH_{n-1}/dd (from
// the generating functions) the d- and q-derivatives need one more recurrence,
// H'_n = dH_n/dd, and those of A are the ga and gb series over 4.  For
// th < TH_SER the operator and its derivatives use these series (terms below
// NSER; |x|, |y| <= 2, truncation below 2e-10); the closed form is kept above,
// where th is not small against s0 unless the layer is optically thick and
// e^-ei removes it.
constexpr float TH_SER = 2.0f;
constexpr int NSER = 8;

// (From here on, and in the transfer kernel, the multiply-adds are written out: what
// else the compiler would join could differ between the kernel's instances, whose
// results are the same bits.)
#pragma clang fp contract(off)
struct Evol {
  float ex, ez, rx, rz;        // e and r in the frame of the field
  float A, D4, ga, gb, s0, cy; // cy: (e x r) along the second axis
  // partial derivatives of A, D4, ga, gb in d and e.r (with DER)
  float Ad, Ae, Dd, De, gad, gae, gbd, gbe;
};

template <bool DER>
__device__ __forceinline__ void evol_build(const Five& f, Evol& E) {
  // 1/k! for k = 0 .. 2 NSER - 1
  constexpr float IF[2 * NSER] = {1.f, 1.f, 1.f / 2.f, 1.f / 6.f, 1.f / 24.f, 1.f / 120.f, 1.f / 720.f,
                                  1.f / 5040.f, 1.f / 40320.f, 1.f / 362880.f, 1.f / 3628800.f,
                                  1.f / 39916800.f, 1.f / 479001600.f, 1.f / 6227020800.f,
                                  1.f / 87178291200.f, 1.f / 1307674368000.f};
  E.ex = f.q;
  E.ez = f.V;
  E.rx = f.qF;
  E.rz = f.VF;
  const float e2 = fmaf(E.ex, E.ex, E.ez * E.ez), r2 = fmaf(E.rx, E.rx, E.rz * E.rz);
  const float er = fmaf(E.ex, E.rx, E.ez * E.rz), d = e2 - r2;
  E.s0 = 0.5f * (e2 + r2);
  E.cy = fmaf(E.ez, E.rx, -(E.ex * E.rz));
  // hypot without its scaling unless the squares could overflow
  const float th = (fabsf(d) < 1.0e18f && fabsf(er) < 1.0e18f) ? sqrtf(fmaf(d, d, 4.0f * er * er)) : hypotf(d, 2.0f * er);
  const float ex = expf(-f.I);
  if (th < TH_SER) {
    const float q = er * er;
    float h0 = 1.f, h1 = d, g0 = 0.f, g1 = 1.f, gm = 0.f;     // H_{n-1}, H_n, H'_{n-1}, H'_n, H'_{n-2}
    float C = 1.f, G = 1.f, D = 0.f, B = 0.f;
    float Dd = 0.f, Dq = 0.f, Gd = 0.f, Bd = 0.f, Bq = 0.f;
#pragma unroll
    for (int n = 1; n < NSER; ++n) {
      C = fmaf(h1, IF[2 * n], C);
      G = fmaf(h1, IF[2 * n + 1], G);
      D = fmaf(h0, IF[2 * n], D);
      B = fmaf(h0, IF[2 * n + 1], B);
      if (DER) {
        if (n > 1) {
          Dd = fmaf(g0, IF[2 * n], Dd);
          Bd = fmaf(g0, IF[2 * n + 1], Bd);
        }
        if (n > 2) {
          Dq = fmaf(gm, IF[2 * n], Dq);
          Bq = fmaf(gm, IF[2 * n + 1], Bq);
        }
        Gd = fmaf(g1, IF[2 * n + 1], Gd);
        gm = g0;
        const float g2 = fmaf(d, g1, fmaf(q, g0, h1));
        g0 = g1;
        g1 = g2;
      }
      const float h2 = fmaf(d, h1, q * h0);
      h0 = h1;
      h1 = h2;
    }
    E.A = ex * fmaf(-0.5f * d, D, C);
    E.D4 = ex * D;
    E.ga = ex * G;
    E.gb = ex * (er * B);
    if (DER) {
      const float er2 = 2.f * er;
      E.Ad = 0.25f * E.ga;
      E.Ae = (0.25f * er2) * (ex * B);
      E.Dd = ex * Dd;
      E.De = ex * (er2 * Dq);
      E.gad = ex * Gd;
      E.gae = ex * (er2 * Bd);
      E.gbd = ex * (er * Bd);
      E.gbe = ex * fmaf(er * er2, Bq, B);
    }
  } else {
    float l1, l2, il;
    const bool dp = d >= 0.f;
    if (dp) {
      l1 = sqrtf(0.5f * (th + d));
      il = 1.0f / l1;
      l2 = fabsf(er) * il;
    } else {
      l2 = sqrtf(0.5f * (th - d));
      il = 1.0f / l2;
      l1 = fabsf(er) * il;
    }
    const float sig = er > 0.f ? 1.f : (er < 0.f ? -1.f : 0.f);
    float che, she;
    if (l1 < 40.f) {
      // cosh and sinh from one exponential; sinh by its Taylor series below
      // 0.5 (truncation 1e-11 relative), where E - 1/E would cancel
      const float El = expf(l1), iEl = 1.0f / El;
      const float x2 = l1 * l1;
      const float shs = l1 * fmaf(x2 * (1.f / 6.f), fmaf(x2 * (1.f / 20.f), fmaf(x2 * (1.f / 42.f), fmaf(x2, 1.f / 72.f, 1.f), 1.f), 1.f), 1.f);
      che = ex * (0.5f * (El + iEl));
      she = ex * (l1 < 0.5f ? shs : 0.5f * (El - iEl));
    } else {
      const float p = expf(l1 - f.I), m = expf(-l1 - f.I);
      che = 0.5f * (p + m);
      she = 0.5f * (p - m);
    }
    float sn, cs;
    sincosf(l2, &sn, &cs);
    const float ce = ex * cs, se = ex * sn;
    const float ith = 1.0f / th;
    const float C2 = se * ith, B3 = she * ith;
    E.A = 0.5f * (che + ce);
    E.D4 = (che - ce) * ith;
    // With a2 = l2 e - s l1 r, a3 = l1 e + s l2 r, w2 = -(s l1 e + l2 r) and
    // w3 = s l2 e - l1 r, the vectors al = -(C2 a2 + B3 a3) and
    // om = -(C2 w2 + B3 w3) take two scalars: ga = C2 l2 + B3 l1 and
    // gb = s (B3 l2 - C2 l1).
    E.ga = fmaf(C2, l2, B3 * l1);
    E.gb = sig * fmaf(B3, l2, -(C2 * l1));
    if (DER) {
      // one pass per variable: dth, dl1, dl2 for a unit change of d, then of e.r
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const float dd = v == 0 ? 1.f : 0.f, der = v == 0 ? 0.f : 1.f;
        const float dth = (v == 0 ? d : 4.f * er) * ith;
        float dl1, dl2;
        if (dp) {
          dl1 = (dth + dd) * (0.25f * il);
          dl2 = fmaf(-l2, dl1, sig * der) * il;
        } else {
          dl2 = (dth - dd) * (0.25f * il);
          dl1 = fmaf(-l1, dl2, sig * der) * il;
        }
        const float dA = 0.5f * fmaf(she, dl1, -(se * dl2));
        const float dC2 = fmaf(ce, dl2, -(C2 * dth)) * ith;
        const float dB3 = fmaf(che, dl1, -(B3 * dth)) * ith;
        const float dD = fmaf(she, dl1, fmaf(se, dl2, -(E.D4 * dth))) * ith;
        const float dga = fmaf(dC2, l2, fmaf(C2, dl2, fmaf(dB3, l1, B3 * dl1)));
        const float dgb = sig * fmaf(dB3, l2, fmaf(B3, dl2, -fmaf(dC2, l1, C2 * dl1)));
        if (v == 0) {
          E.Ad = dA; E.Dd = dD; E.gad = dga; E.gbd = dgb;
        } else {
          E.Ae = dA; E.De = dD; E.gae = dga; E.gbe = dgb;
        }
      }
    }
  }
}

// The pieces of (O - A 1) v for a vector v in the frame: M4raw v, P(e, -r) v
// and P(r, e) v, where P(a, w) = [[0,a1,a2,a3],[a1,0,w3,-w2],[a2,-w3,0,w1],[a3,w2,-w1,0]]
struct Pieces {
  float m4[4], p1[4], p2[4];   // p1[0] = e.v, p2[0] = r.v
};

__device__ __forceinline__ Pieces evol_pieces(const Evol& E, const float v[4]) {
  Pieces w;
  const float ev = fmaf(E.ex, v[1], E.ez * v[3]), rv = fmaf(E.rx, v[1], E.rz * v[3]);
  w.m4[0] = fmaf(E.s0, v[0], E.cy * v[2]);
  w.m4[1] = fmaf(E.ex, ev, fmaf(E.rx, rv, -(E.s0 * v[1])));
  w.m4[2] = -fmaf(E.cy, v[0], E.s0 * v[2]);
  w.m4[3] = fmaf(E.ez, ev, fmaf(E.rz, rv, -(E.s0 * v[3])));
  w.p1[0] = ev;
  w.p1[1] = fmaf(E.ex, v[0], -(E.rz * v[2]));
  w.p1[2] = fmaf(E.rz, v[1], -(E.rx * v[3]));
  w.p1[3] = fmaf(E.ez, v[0], E.rx * v[2]);
  w.p2[0] = rv;
  w.p2[1] = fmaf(E.rx, v[0], E.ez * v[2]);
  w.p2[2] = fmaf(E.ex, v[3], -(E.ez * v[1]));
  w.p2[3] = fmaf(E.rz, v[0], -(E.ex * v[2]));
  return w;
}

// (O - A 1) v
__device__ __forceinline__ void evol_apply(const Evol& E, const Pieces& w, float o[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = fmaf(E.D4, w.m4[i], -fmaf(E.ga, w.p1[i], E.gb * w.p2[i]));
}

// Gradient of O v in the five elements of the frame (columns I, q, V, qF, VF)
// and, for the azimuth, the directional derivative itself.  The reference
// forms the partial derivatives of O as matrices (rtesolver.f90:476-1002);
// here the gradient of its action on one vector serves every direction, 20
// operations each, where a directional derivative by itself took 200.
struct Grad {
  float g[5][4];
};

__device__ __forceinline__ void evol_grad(const Evol& E, const float v[4], const Pieces& w, Grad& G) {
  float xd[4], xe[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    xd[i] = fmaf(E.Ad, v[i], fmaf(E.Dd, w.m4[i], -fmaf(E.gad, w.p1[i], E.gbd * w.p2[i])));
    xe[i] = fmaf(E.Ae, v[i], fmaf(E.De, w.m4[i], -fmaf(E.gae, w.p1[i], E.gbe * w.p2[i])));
    G.g[0][i] = -fmaf(E.A, v[i], fmaf(E.D4, w.m4[i], -fmaf(E.ga, w.p1[i], E.gb * w.p2[i])));
  }
  const float ev = w.p1[0], rv = w.p2[0];
  const float ex = E.ex, ez = E.ez, rx = E.rx, rz = E.rz, D4 = E.D4, ga = E.ga, gb = E.gb;
  const float ex2 = 2.f * ex, ez2 = 2.f * ez, rx2 = -2.f * rx, rz2 = -2.f * rz;
  // d(M4raw) v of a unit change of e along the first axis is (ex v0 - rz v2,
  // e.v, rz v0 - ex v2, ez v1 - ex v3), and so on
  const float a02 = fmaf(ex, v[0], -(rz * v[2])), a13 = fmaf(ez, v[1], -(ex * v[3]));
  const float b02 = fmaf(ez, v[0], rx * v[2]);
  const float c02 = fmaf(rx, v[0], ez * v[2]), c13 = fmaf(rz, v[1], -(rx * v[3]));
  const float d02 = fmaf(rz, v[0], -(ex * v[2]));
  G.g[1][0] = fmaf(ex2, xd[0], fmaf(rx, xe[0], fmaf(D4, a02, -(ga * v[1]))));
  G.g[1][1] = fmaf(ex2, xd[1], fmaf(rx, xe[1], fmaf(D4, ev, -(ga * v[0]))));
  G.g[1][2] = fmaf(ex2, xd[2], fmaf(rx, xe[2], fmaf(D4, d02, -(gb * v[3]))));
  G.g[1][3] = fmaf(ex2, xd[3], fmaf(rx, xe[3], fmaf(D4, a13, gb * v[2])));
  G.g[2][0] = fmaf(ez2, xd[0], fmaf(rz, xe[0], fmaf(D4, b02, -(ga * v[3]))));
  G.g[2][1] = fmaf(ez2, xd[1], fmaf(rz, xe[1], -fmaf(D4, a13, gb * v[2])));
  G.g[2][2] = fmaf(ez2, xd[2], fmaf(rz, xe[2], fmaf(-D4, c02, gb * v[1])));
  G.g[2][3] = fmaf(ez2, xd[3], fmaf(rz, xe[3], fmaf(D4, ev, -(ga * v[0]))));
  G.g[3][0] = fmaf(rx2, xd[0], fmaf(ex, xe[0], fmaf(D4, c02, -(gb * v[1]))));
  G.g[3][1] = fmaf(rx2, xd[1], fmaf(ex, xe[1], fmaf(D4, rv, -(gb * v[0]))));
  G.g[3][2] = fmaf(rx2, xd[2], fmaf(ex, xe[2], fmaf(-D4, b02, ga * v[3])));
  G.g[3][3] = fmaf(rx2, xd[3], fmaf(ex, xe[3], fmaf(D4, c13, -(ga * v[2]))));
  G.g[4][0] = fmaf(rz2, xd[0], fmaf(ez, xe[0], fmaf(D4, d02, -(gb * v[3]))));
  G.g[4][1] = fmaf(rz2, xd[1], fmaf(ez, xe[1], fmaf(-D4, c13, ga * v[2])));
  G.g[4][2] = fmaf(rz2, xd[2], fmaf(ez, xe[2], fmaf(D4, a02, -(ga * v[1]))));
  G.g[4][3] = fmaf(rz2, xd[3], fmaf(ez, xe[3], fmaf(D4, rv, -(gb * v[0]))));
}

// the directional derivative (dO) v for the change f of the five elements
__device__ __forceinline__ void grad_dot(const Grad& G, const Five& f, float o[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = fmaf(f.I, G.g[0][i],
                fmaf(f.q, G.g[1][i], fmaf(f.V, G.g[2][i], fmaf(f.qF, G.g[3][i], f.VF * G.g[4][i]))));
}

// the derivative in the azimuth, which moves e and r along the frame's second
// axis by twice their first component; every term carries that component, so
// nothing cancels in a weak transverse field
__device__ __forceinline__ void evol_azimuth(const Evol& E, const float v[4], const Pieces& w, float o[4]) {
  const float alx = -fmaf(E.ga, E.ex, E.gb * E.rx), omx = fmaf(E.ga, E.rx, -(E.gb * E.ex));
  const float t2 = fmaf(E.ex, E.ex, E.rx * E.rx), g = fmaf(E.ex, E.ez, E.rx * E.rz);
  o[0] = 2.f * fmaf(alx, v[2], -(E.D4 * (E.cy * v[1])));
  o[1] = 2.f * fmaf(E.D4, fmaf(E.cy, v[0], t2 * v[2]), -(omx * v[3]));
  o[2] = 2.f * fmaf(E.D4, fmaf(E.ex, w.p1[0], E.rx * w.p2[0]), alx * v[0]);
  o[3] = 2.f * fmaf(E.D4, g * v[2], omx * v[1]);
}

#pragma clang fp contract(fast)

}  // namespace fz
