// Per-pixel Levenberg-Marquardt step of the FIRTEZ-dz inversion on the GPU.
//
//   eqv_kernel : node contraction of the per-height response functions where
//                rt_kernel does not form it (Pg, rho, P0, HYDROSTATIC)
//                (CALCULATE_EQUIVALENT_DSYN, forward.f90:552-681): one thread
//                per (pixel, spectral row), FP64 accumulation over the support
//                of each node's hat function, REAL(4) store.
//   lm_kernel  : one wave per pixel (four beyond LM_MAXNP free parameters),
//                FP64 throughout except the REAL(4) model (GET_PERT_1D,
//                get_dmodel.f90:1201-1244): chi^2 and accept/reject
//                (:960-1032), lambda update (:917-956), Jacobian
//                normalisation (:725-770), Gauss-Newton normal matrix and
//                gradient streamed through LDS in chunks of 32 spectral rows,
//                damped pseudo-inverse by a parallel cyclic Jacobi
//                eigen-decomposition in LDS (the symmetric form of the
//                truncated SVD of lm.f90:61-133), and the limited
//                perturbation applied through the node basis (:1715-2016).
#pragma once

namespace fz {

constexpr int LM_MAXNP = 64;     // free parameters per pixel with the work arrays in LDS
// one wave per pixel: the Jacobi rounds and reductions are wave-local, so
// the barriers are cheap and a CU holds many pixels at once
constexpr int LM_THREADS = 64;
constexpr int LM_CH = 32;        // spectral rows per chunk of the normal matrix
constexpr int LM_PF = 10;        // responses that a lane loads together
// more free parameters (up to NZ nodes per parameter, the reference's
// default): the same step with its work arrays in a per-pixel slice of
// device memory, four waves per pixel
constexpr int LM_MAXNP_BIG = 2048;
constexpr int LM_BIG_THREADS = 256;

// get_dmodel.f90:31 (PARAM_NORMS) and :1903-1919 (hard bounds)
__constant__ double c_lm_norm[8] = {6000.0, 1.0e5, 1.0e-5, 1.0e3, 1.0e3, 1.0e3, 1.0e6, 6.0e2};
__constant__ double c_lm_low[8] = {2500.0, 1.0e-2, 1.0e-10, -5.0e4, -5.0e4, -5.0e4, -1.0e7, 1.0e-8};
__constant__ double c_lm_upp[8] = {1.8e4, 1.0e12, 1.0e10, 5.0e4, 5.0e4, 5.0e4, 1.0e7, 1.0e12};

struct LmArgs {
  int ncol, nz, numw, nfreq, np;
  int nparam;                  // inverted physical parameters
  int par[8];                  // physical index 0..7 (T, Pg, rho, Bx, By, Bz, vz, P0)
  int slot[8];                 // response-function slot in the Cartesian per-height output
  int mcol[8];                 // model column
  int mslot[8];                // its place among the pixel's columns in LDS (Pg and P0 share theirs)
  int rowslot[12];             // place of each model row there (log tau5 last), -1: not held
  int nheld;                   // columns held, log tau5 included
  int j0[8], nj[8];            // first free parameter, nodes
  int rowstk[4];               // Stokes index of each inverted Stokes block
  int regul, solver, node_expansion, pen_typ[8];
  double pen_alp[8];
  double svdtol, inu, mpert, maxsteps;
  const double* coefs;         // [np][nz]
  const double* colsum;        // [np] column sums of the node basis
  // per pixel
  const double* obs;           // [ncol][nfreq]
  const float* stokes;         // [ncol][4][numw] current synthesis (times GAIN1D)
  const double* syn_d;
  double* best_syn;            // [ncol][nfreq]
  double* sla;                 // [ncol][9]
  const float* eqv;            // [ncol][np][nfreq] current equivalent response functions
  float* eqv_best;             // [ncol][np][nfreq]
  const double* isigmap;       // [nfreq], or [ncol][nfreq] with isig_stride = nfreq
  long isig_stride;            // 0: one weight vector for every pixel (ISIGMAP3D equal over the map)
  // synthesis of the inverted Stokes parameters in FP64, [ncol][nfreq] like
  // obs (SYN3D of the host-array entry point), or null: the float Stokes rows
  float* atm;                  // [12][nz][ncol] current model (in: model of eqv; out: new trial)
  float* atm_best;             // [12][nz][ncol]
  int32_t* done;               // [ncol] AM_I_DONE
  double* delta;               // [ncol][np] applied node perturbation, or null
  // active-pixel launch: workgroup b handles pixel pix_of[b], and stokes/eqv
  // hold the compacted rows (row b); null: workgroup b is pixel b
  const int32_t* pix_of;
  // per-pixel windows (poff null: none): pixel pix has numw_pix =
  // poff[pix+1]-poff[pix] wavelengths; its obs/best_syn rows start at
  // nstk*poff[pix], its Stokes at 4*poff[pix], its eqv/eqv_best at
  // np*nstk*poff[pix]; isigmap is read per Stokes block (isigmap[b*numw]);
  // inu_pix: chi^2 normalised by the pixel's own NFREQ
  const int64_t* poff;
  int nstk, inu_pix;
  // work arrays in device memory (more than LM_MAXNP free parameters):
  // workgroup b handles row row0 + b and uses work[b * work_stride ...]
  double* work;
  long work_stride;
  int row0;
  // externally controlled step (the PSF-coupled inversion, whose acceptance
  // and damping are decided over the whole map): gres non-null gives the
  // residual of the gradient J^T W gres per pixel ([ncol][nfreq], the
  // adjoint-convolved residual), hscale multiplies J^T W J (the sum of the
  // squared PSF taps: the pixel's own block of the coupled normal matrix) and
  // ext_lambda is the damping; chi^2, acceptance, INV_SLA, the best model
  // and AM_I_DONE are left to the caller, eqv is the Jacobian of the model
  // in atm
  const double* gres = nullptr;
  double hscale = 1.0, ext_lambda = 0.0;
};

// ---------------------------------------------------------------- node contraction
struct EqvArgs {
  int ncol_tile, col0, nz, numw, nfreq, np, nstk;
  int nslot;                   // response-function slots per column in the tile (7, or 8 with P0)
  int rowstk[4];
  const int* slot_of;          // [np] response-function slot of each free parameter
  const int* kbeg;             // [np] support of each node's hat function
  const int* kend;             // [np]
  // per parameter and height (pairs): the lowest unfinished node in bits
  // 0-15, bit 30 set when it takes height k, bit 29 when the next node does;
  // tab_c the two coefficients, so each height's loads are independent of
  // the running node index
  const int* tab_j;            // [nparam][nz]
  const double* tab_c;         // [nparam][nz][2]
  // the nodes of inverted parameter ip are j0[ip] .. j0[ip]+nj[ip]-1; pairs:
  // every height lies in the support of at most two consecutive nodes of a
  // parameter and the supports move up with the node index (hat functions),
  // so one pass over the heights feeds two running sums
  int nparam, pairs;
  int j0[8], nj[8];
  const double* coefs;         // [np][nz]
  const float* jac;            // tile: [ntile][nslot][nz][4][numw], ragged with windows
  float* eqv;                  // [ncol][np][nfreq], ragged with windows
  // per-pixel windows (poff null: none): the tile's response functions are
  // [nslot][nz][4][numw_col] per column from nslot*nz*4*(poff[col]-poff[col0]);
  // the output block of pixel col is [np][nstk][numw_col] from np*nstk*poff[col]
  const int64_t* poff;
};

// the column of the tile [c0, c0+n) whose ragged range [poff[c], poff[c+1]) holds g
__device__ __forceinline__ int ragged_column(const int64_t* poff, int c0, int n, int64_t g) {
  int lo = c0, hi = c0 + n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (poff[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// EQVDSYN (forward.f90:552-681): one thread per (column, inverted Stokes row,
// wavelength), all free parameters; FP64 sums over the node's heights
__global__ void __launch_bounds__(256) eqv_kernel(EqvArgs a) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const float* jc;
  float* out;
  long cs, fstride;
  if (a.poff) {
    const int64_t base = a.poff[a.col0];
    if (t >= (long)a.nstk * (a.poff[a.col0 + a.ncol_tile] - base)) return;
    const int col = ragged_column(a.poff, a.col0, a.ncol_tile, base + t / a.nstk);
    const int64_t p0 = a.poff[col];
    const int nw = (int)(a.poff[col + 1] - p0);
    const int f = (int)(t - (long)a.nstk * (p0 - base));
    const int b = f / nw, l = f - b * nw;
    cs = (long)4 * nw;
    jc = a.jac + (long)a.nslot * a.nz * 4 * (p0 - base) + (long)a.rowstk[b] * nw + l;
    fstride = (long)a.nstk * nw;
    out = a.eqv + (long)a.np * a.nstk * p0 + f;
  } else {
    if (t >= (long)a.ncol_tile * a.nfreq) return;
    const int ct = (int)(t / a.nfreq);
    const int f = (int)(t - (long)ct * a.nfreq);
    const int b = f / a.numw, l = f - b * a.numw;
    cs = (long)4 * a.numw;
    jc = a.jac + (long)ct * a.nslot * a.nz * cs + a.rowstk[b] * a.numw + l;
    fstride = a.nfreq;
    out = a.eqv + ((long)(a.col0 + ct) * a.np) * a.nfreq + f;
  }
  if (a.pairs) {
    // each node's sum is formed in the same order (heights ascending from
    // its support's start) as the per-node loop below: identical results,
    // half the reads where the hat supports overlap
    for (int ip = 0; ip < a.nparam; ++ip) {
      const int jb = a.j0[ip], je = jb + a.nj[ip] - 1;
      const float* jp = jc + (long)a.slot_of[jb] * a.nz * cs;
      const int* tj = a.tab_j + (long)ip * a.nz;
      const double* tc = a.tab_c + (long)ip * a.nz * 2;
      int jl = jb;                                   // lowest unfinished node
      double alo = 0.0, ahi = 0.0;                   // sums of nodes jl, jl+1
      const int k0 = a.kbeg[jb], k1 = a.kend[je];
      // the loads of eight heights are issued together (one strided read per
      // height and lane: eight in flight instead of one), the sums then take
      // them in height order as before
      for (int kb = k0; kb <= k1; kb += 8) {
        float vb[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) vb[i] = (kb + i <= k1) ? jp[(long)(kb + i) * cs] : 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int k = kb + i;
          if (k > k1) break;
          const int w = tj[k];
          while (jl < (w & 0xffff)) {
            out[(long)jl * fstride] = (float)alo;
            alo = ahi;
            ahi = 0.0;
            ++jl;
          }
          const double v = (double)vb[i];
          if (w & (1 << 30)) alo += v * tc[2 * k];
          if (w & (1 << 29)) ahi += v * tc[2 * k + 1];
        }
      }
      out[(long)jl * fstride] = (float)alo;
      if (jl < je) out[(long)(jl + 1) * fstride] = (float)ahi;
    }
    return;
  }
  for (int j = 0; j < a.np; ++j) {
    const float* jp = jc + (long)a.slot_of[j] * a.nz * cs;
    const double* cf = a.coefs + (long)j * a.nz;
    double acc = 0.0;
    for (int k = a.kbeg[j]; k <= a.kend[j]; ++k) acc += (double)jp[k * cs] * cf[k];
    out[(long)j * fstride] = (float)acc;
  }
}

// ---------------------------------------------------------------- LM step
// rows of a chunk in LDS: np normalised responses and the residual, padded to
// a multiple of four doubles and to a stride that spreads the banks
constexpr size_t lm_ldj(int np) { return (size_t)(np + 4) / 4 * 4 + 2; }
// the normal matrix and the gradient (column np) in blocks of two rows by
// four columns, those with an entry on or above the diagonal
constexpr size_t lm_blocks(int np) {
  size_t n = 0;
  for (int i = 0; i < np; i += 2) n += (np + 4) / 4 - i / 4;
  return n;
}
constexpr int LM_MAXHELD = 8;    // model columns of a pixel in LDS: seven inverted ones and log tau5

template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
  const int t = threadIdx.x;
  red[t] = v;
  __syncthreads();
  for (int s = NT / 2; s > 0; s >>= 1) {
    if (t < s) red[t] += red[t + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// sum over a wave (every lane gets it) by the fixed tree of cross-lane moves,
// and over a workgroup of NT threads
__device__ __forceinline__ double wave_sum(double x) {
  x = add_swap32(x);
  x = add_swap16(x);
  x += dpp64<0x128>(x);
  x += dpp64<0xB1>(x);
  x += dpp64<0x4E>(x);
  return x + dpp64<0x141>(x);
}
template <int NT>
__device__ __forceinline__ double team_sum(double v, double* red) {
  v = wave_sum(v);
  if constexpr (NT == 64) return v;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) s += red[w];
  return s;
}

// 1 / sqrt(x) for x of ordinary size
__device__ __forceinline__ double rsq64(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-(x * r), r, 1.0), r);
  return fma(0.5 * r, fma(-(x * r), r, 1.0), r);
}

// GET_IT_PENALTIES (get_dmodel.f90:1041-1197) by one thread: pen_res[np],
// pen_hss[np*np] (row-major, block diagonal) from the model columns in LDS;
// sm and pen are LDS work vectors of np entries.
__device__ void lm_penalties(const LmArgs& a, const float* mod, double* pen_res, double* pen_hss, double* sm,
                             double* pen) {
  const int np = a.np, nz = a.nz;
  for (int i = 0; i < np; ++i) pen_res[i] = 0.0;
  for (int i = 0; i < np * np; ++i) pen_hss[i] = 0.0;
  for (int ip = 0; ip < a.nparam; ++ip) {
    const int p = a.par[ip], ji = a.j0[ip], jd = a.nj[ip];
    const float* col = mod + a.mslot[ip] * nz;
    const double alp = sqrt(a.pen_alp[p] / (double)np);
    for (int j = 0; j < jd; ++j) {
      const double* cf = a.coefs + (long)(ji + j) * nz;
      double s = 0.0;
      for (int k = 0; k < nz; ++k) s = s + (double)col[k] * cf[k];
      sm[j] = s / a.colsum[ji + j] / c_lm_norm[p];
    }
    // L: type 0 -> diag(1/jd), type 1 -> first differences (first row empty)
    for (int k = 0; k < jd; ++k) {
      double v = 0.0;
      if (a.pen_typ[p] == 0) v = (1.0 * (1.0 / (double)jd)) * alp * sm[k];
      else if (a.pen_typ[p] == 1 && k > 0) v = (1.0 * 1.0) * alp * sm[k] + (-1.0 * 1.0) * alp * sm[k - 1];
      pen[k] = v;
    }
    for (int j = 0; j < jd; ++j) {
      double s = 0.0;
      if (a.pen_typ[p] == 0) s = (1.0 / (double)jd) * alp * pen[j];
      else if (a.pen_typ[p] == 1) {
        if (j > 0) s += alp * pen[j];
        if (j + 1 < jd) s += -alp * pen[j + 1];
      }
      pen_res[ji + j] = s;
    }
    // L^T L into the zeroed block: type 0 is diagonal; type 1, with
    // L_kk = alp (k>0) and L_k,k-1 = -alp, is tridiagonal:
    // (L^T L)_ii = sum over k = i (i>0), then k = i+1 (i+1<jd) of alp^2,
    // (L^T L)_i,i+-1 = -alp^2 from the single k = max(i, j)
    for (int i = 0; i < jd; ++i) {
      double* row = pen_hss + (long)(ji + i) * np + ji;
      if (a.pen_typ[p] == 0) {
        row[i] = ((1.0 / (double)jd) * alp) * ((1.0 / (double)jd) * alp);
      } else if (a.pen_typ[p] == 1) {
        double d = 0.0;
        if (i > 0) d += alp * alp;
        if (i + 1 < jd) d += (-alp) * (-alp);
        row[i] = d;
        if (i > 0) row[i - 1] = alp * -alp;
        if (i + 1 < jd) row[i + 1] = -alp * alp;
      }
    }
  }
}

// The Jacobi rotation that clears a_pq: cs, sn with a reciprocal and two
// reciprocal square roots where the entries' squares are of ordinary size
// (the chain of one rotation is what a round waits for)
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double apq, double& cs, double& sn) {
  const double d = aqq - app, b = 2.0 * apq, h = fma(d, d, b * b);
  double t;
  if (h > 1.0e-280 && h < 1.0e280) {
    t = (d >= 0.0 ? b : -b) * rcp64(fabs(d) + h * rsq64(h));
    cs = rsq64(fma(t, t, 1.0));
  } else {
    const double th = d / b;
    t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(1.0 + th * th));
    cs = 1.0 / sqrt(1.0 + t * t);
  }
  sn = t * cs;
}

// Damped solve of GET_PERTURBATION (lm.f90:137-204) on a symmetric matrix
// A[np][ld] (ld = np + 1; rows up to np + (np & 1) zero-padded) and the
// right-hand side g, by all NT threads of the workgroup; V must hold the
// identity.  solver 1: parallel cyclic Jacobi (tournament order) and the
// truncated pseudo-inverse of GET_INVERSE (lm.f90:61-133: values below
// svdtol * max dropped); solver 2: the CG iteration of
// NEW_CALCULATE_DELTA_UBICGSTAB (lm.f90:375-453).  Work vectors: dv[np],
// red[NT], rot[np + 1], nod[4 np].  Result in del[np]; A and V are destroyed.
//
// A round of the Jacobi sweep turns npe/2 disjoint pairs at once.  Each lane
// takes one 2 x 2 block of A that two pairs share (the blocks above the
// diagonal, mirrored on store) and applies both rotations to it, so A is read
// and written once per round; V takes one rotation per pair and row.  Bound:
// the latency of a round, so a lane loads its block and its rows of V before
// the rotations are formed (by the lanes of the diagonal blocks, from those
// blocks) and one exchange through LDS hands the rotations out.  A round of 20
// parameters took 1.3 us with the loads behind the exchange.
//
// Inlined into its kernels: as a function it could not know that its arrays are in
// LDS, and its kernels took 197 registers and a stack (here 174 and 88): the step of 4096
// pixels with 20 parameters 0.85 -> 0.65 ms (CG the same), with 64 parameters of 1024
// 7.0 -> 6.1 ms; a single CG solve of 20 parameters 44.4 -> 42.1 us.
template <int NT>
__device__ __forceinline__ void damped_solve(int solver, double svdtol, int np, double* A, double* V, const double* g,
                             double* dv, double* del, double* red, double* rot, double* nod) {
  const int t = threadIdx.x;
  const int ld = np + 1;
  const int npe = np + (np & 1);
  if (solver == 1) {
    const int half = npe / 2;
    // pair i of a round: players L[i], L[npe-1-i] with L = [0, (rnd+k)%(npe-1)+1 ...]
    auto pair = [&](int rnd, int i, int& p, int& q) {
      int x = rnd + i - 1, y = rnd + npe - 2 - i;
      if (x >= npe - 1) x -= npe - 1;
      if (y >= npe - 1) y -= npe - 1;
      const int p0 = i == 0 ? 0 : x + 1, q0 = y + 1;
      p = min(p0, q0);
      q = max(p0, q0);
    };
    // blocks (i1 <= i2): the diagonal ones first, then row by row (NT == 64:
    // listed once in LDS; else found again for each)
    const int nblk = half * (half + 1) / 2;
    unsigned short* blk = reinterpret_cast<unsigned short*>(nod);
    if constexpr (NT == 64) {
      for (int i = t; i < half; i += NT) {
        blk[i] = (unsigned short)(i << 8 | i);
        int o = half + i * (half - 1) - i * (i - 1) / 2;
        for (int j = i + 1; j < half; ++j) blk[o++] = (unsigned short)(i << 8 | j);
      }
      __syncthreads();
    }
    // V: NG lanes to a pair, each every NG-th row
    const int ng = max(1, NT / half), vi0 = t / ng, vr = t - vi0 * ng, vstep = max(1, NT / ng);
    auto turn = [&](double c1, double s1, double c2, double s2, double& app, double& apq, double& aqp, double& aqq) {
      const double bpp = c2 * app - s2 * apq, bpq = s2 * app + c2 * apq;
      const double bqp = c2 * aqp - s2 * aqq, bqq = s2 * aqp + c2 * aqq;
      app = c1 * bpp - s1 * bqp;
      apq = c1 * bpq - s1 * bqq;
      aqp = s1 * bpp + c1 * bqp;
      aqq = s1 * bpq + c1 * bqq;
    };
    auto put = [&](int i1, int i2, int p1, int q1, int p2, int q2, double app, double apq, double aqp, double aqq) {
      A[p1 * ld + p2] = app;
      A[p1 * ld + q2] = apq;
      A[q1 * ld + p2] = aqp;
      A[q1 * ld + q2] = aqq;
      if (i1 != i2) {
        A[p2 * ld + p1] = app;
        A[q2 * ld + p1] = apq;
        A[p2 * ld + q1] = aqp;
        A[q2 * ld + q1] = aqq;
      }
    };
    // the lane's first block
    int j1 = -1, j2 = 0;
    if constexpr (NT == 64) {
      if (t < nblk) {
        j1 = blk[t] >> 8;
        j2 = blk[t] & 255;
      }
    }
    const int ei0 = t / np, ek0 = t - ei0 * np, edi = NT / np, edk = NT - edi * np;
    for (int sweep = 0; sweep < 60; ++sweep) {
      double o = 0.0, tt = 0.0;
      for (int i = ei0, k = ek0; i < np;) {
        const double x = A[i * ld + k];
        tt += x * x;
        if (i != k) o += x * x;
        i += edi;
        k += edk;
        if (k >= np) {
          k -= np;
          ++i;
        }
      }
      const double off = team_sum<NT>(o, red), tot = team_sum<NT>(tt, red);
      if (off <= 1e-30 * tot || off == 0.0) break;
      for (int rnd = 0; rnd < npe - 1; ++rnd) {
        int p1 = 0, q1 = 0, p2 = 0, q2 = 0;
        double app = 0.0, apq = 0.0, aqp = 0.0, aqq = 0.0;
        if (j1 >= 0) {
          pair(rnd, j1, p1, q1);
          pair(rnd, j2, p2, q2);
          app = A[p1 * ld + p2];
          apq = A[p1 * ld + q2];
          aqp = A[q1 * ld + p2];
          aqq = A[q1 * ld + q2];
        }
        int pv = 0, qv = 0;
        const bool hasv = vi0 < half;
        double vp[4], vq[4];
        if (hasv) pair(rnd, vi0, pv, qv);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = vr + u * ng;
          const bool in = hasv && k < np && qv < np;
          vp[u] = in ? V[k * ld + pv] : 0.0;
          vq[u] = in ? V[k * ld + qv] : 0.0;
        }
        for (int i = t; i < half; i += NT) {
          int p, q;
          pair(rnd, i, p, q);
          double cs = 1.0, sn = 0.0;
          if (q < np) {
            // (NT == 64: block (i, i) is the lane's own)
            const double bpp = NT == 64 ? app : A[p * ld + p], bqq = NT == 64 ? aqq : A[q * ld + q];
            const double bpq = NT == 64 ? apq : A[p * ld + q];
            if (bpq != 0.0) jacobi_rotation(bpp, bqq, bpq, cs, sn);
          }
          rot[2 * i] = cs;
          rot[2 * i + 1] = sn;
        }
        __syncthreads();
        // A <- J^T A J
        if (j1 >= 0) {
          turn(rot[2 * j1], rot[2 * j1 + 1], rot[2 * j2], rot[2 * j2 + 1], app, apq, aqp, aqq);
          put(j1, j2, p1, q1, p2, q2, app, apq, aqp, aqq);
        }
        auto block = [&](int i1, int i2) {
          pair(rnd, i1, p1, q1);
          pair(rnd, i2, p2, q2);
          app = A[p1 * ld + p2];
          apq = A[p1 * ld + q2];
          aqp = A[q1 * ld + p2];
          aqq = A[q1 * ld + q2];
          turn(rot[2 * i1], rot[2 * i1 + 1], rot[2 * i2], rot[2 * i2 + 1], app, apq, aqp, aqq);
          put(i1, i2, p1, q1, p2, q2, app, apq, aqp, aqq);
        };
        if constexpr (NT == 64) {
          for (int e = t + NT; e < nblk; e += NT) block(blk[e] >> 8, blk[e] & 255);
        } else {
          for (int e = t; e < half * half; e += NT) {
            const int i1 = e / half, i2 = e - i1 * half;
            if (i1 <= i2) block(i1, i2);
          }
        }
        // V <- V J
        for (int i = vi0; i < half; i += vstep) {
          if (i != vi0) pair(rnd, i, pv, qv);
          const double cs = rot[2 * i], sn = rot[2 * i + 1];
          for (int k0 = vr; k0 < np; k0 += 4 * ng) {
            if (i != vi0 || k0 != vr) {
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const int k = k0 + u * ng;
                const bool in = k < np && qv < np;
                vp[u] = in ? V[k * ld + pv] : 0.0;
                vq[u] = in ? V[k * ld + qv] : 0.0;
              }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int k = k0 + u * ng;
              if (k < np && qv < np) {
                V[k * ld + pv] = cs * vp[u] - sn * vq[u];
                V[k * ld + qv] = sn * vp[u] + cs * vq[u];
              }
            }
          }
        }
        __syncthreads();
      }
    }
    // truncated pseudo-inverse: keep |d| >= svdtol * max|d|
    double mx = 0.0;
    for (int i = 0; i < np; ++i) mx = fmax(mx, fabs(A[i * ld + i]));
    const double thr = mx * (svdtol > 0 ? svdtol : 10.0e-4);
    for (int e = t; e < np; e += NT) {
      const double d = A[e * ld + e];
      double pr = 0.0;
      if (!(fabs(d) < thr)) {
        for (int i = 0; i < np; ++i) pr += V[i * ld + e] * g[i];
        pr /= d;
      }
      dv[e] = pr;
    }
    __syncthreads();
    for (int i = t; i < np; i += NT) {
      double s = 0.0;
      for (int e = 0; e < np; ++e) s += V[i * ld + e] * dv[e];
      del[i] = s;
    }
  } else {
    // NEW_CALCULATE_DELTA_UBICGSTAB (lm.f90:375-453): the matrix-vector and
    // dot products spread over the workgroup; every thread holds the same
    // scalars, so the iteration and its stopping test are uniform
    double* xv = nod;
    double* pv = nod + np;
    double* rv = nod + 2 * np;
    double* qv = nod + 3 * np;
    auto dot = [&](const double* x, const double* y) {
      double s = 0.0;
      for (int i = t; i < np; i += NT) s += x[i] * y[i];
      return block_sum<NT>(s, red);
    };
    // A is exactly symmetric here (its lower triangle mirrored, a symmetric
    // penalty Hessian, the diagonal scaled): row i is read as column i, so
    // the lanes of a wave read consecutive entries
    auto matvec = [&](const double* x, double* y) {
      for (int i = t; i < np; i += NT) {
        double s = 0.0;
        for (int j = 0; j < np; ++j) s += A[j * ld + i] * x[j];
        y[i] = s;
      }
      __syncthreads();
    };
    for (int i = t; i < np; i += NT) {
      xv[i] = 0.0;
      pv[i] = g[i];
      rv[i] = g[i];   // bet - alp x with x = 0
    }
    __syncthreads();
    double crho = dot(rv, rv);
    matvec(pv, qv);
    double calpha = crho / dot(pv, qv);
    for (int i = t; i < np; i += NT) {
      xv[i] = xv[i] + calpha * pv[i];
      rv[i] = rv[i] - calpha * qv[i];
    }
    __syncthreads();
    double pcond = 1.0e29, dcond = -1.0e29;
    bool conv = false;
    // each iteration forms the next direction before its stopping test, so
    // one pass over A gives both A x (the test) and A p (the next step);
    // each of the two sums keeps the order of a separate product
    {
      const double crho0 = crho;
      crho = dot(rv, rv);
      const double cbeta = crho / crho0;
      for (int i = t; i < np; i += NT) pv[i] = rv[i] + cbeta * pv[i];
      __syncthreads();
      matvec(pv, qv);
    }
    for (int it = 1; it <= 100000; ++it) {
      calpha = crho / dot(pv, qv);
      for (int i = t; i < np; i += NT) {
        xv[i] = xv[i] + calpha * pv[i];
        rv[i] = rv[i] - calpha * qv[i];
      }
      __syncthreads();
      const double crho0 = crho;
      crho = dot(rv, rv);
      const double cbeta = crho / crho0;
      for (int i = t; i < np; i += NT) pv[i] = rv[i] + cbeta * pv[i];
      __syncthreads();
      double cs = 0.0;
      for (int i = t; i < np; i += NT) {
        double s = 0.0, sq = 0.0;
        for (int j = 0; j < np; ++j) {
          const double aij = A[j * ld + i];
          s += aij * xv[j];
          sq += aij * pv[j];
        }
        qv[i] = sq;
        const double e = (s - g[i]) / (fabs(g[i]) + 1.0e-5);
        cs += e * e;
      }
      const double cond = block_sum<NT>(cs, red) / (double)np;
      if (cond < 1.0e-3 || dcond > 1.0e30) {
        for (int i = t; i < np; i += NT) del[i] = xv[i];
        conv = true;
        break;
      }
      dcond = cond - pcond;
      pcond = cond;
    }
    if (!conv)
      for (int i = t; i < np; i += NT) del[i] = xv[i] / 10.0;
  }
}

template <bool BIG>
__global__ void __launch_bounds__(BIG ? LM_BIG_THREADS : LM_THREADS) lm_kernel(LmArgs a) {
  constexpr int NT = BIG ? LM_BIG_THREADS : LM_THREADS;
  extern __shared__ __align__(16) double smem_dyn[];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  // consecutive rows to one XCD (workgroups go round the eight of them), so
  // that the lines of the model, a pixel's width each, meet in one L2
  const int bid = (int)blockIdx.x, per = (int)gridDim.x / 8;
  const int brow = bid < 8 * per ? (bid & 7) * per + (bid >> 3) : bid;
  const int row = a.row0 + brow;
  double* smem = BIG ? a.work + (long)brow * a.work_stride : smem_dyn;
  const int pix = a.pix_of ? uniform(a.pix_of[row]) : row;
  if (a.done && a.done[pix] != 0) return;
  const int np = a.np, nz = a.nz;
  int nf = a.nfreq, numw = a.numw;
  long o_obs = (long)pix * a.nfreq, o_stk = (long)row * 4 * a.numw;
  long o_ecur = (long)row * np * a.nfreq, o_ebest = (long)pix * np * a.nfreq;
  double inu = a.inu;
  if (a.poff) {
    const long p0 = uniform(a.poff[pix]);
    numw = (int)(uniform(a.poff[pix + 1]) - p0);
    nf = a.nstk * numw;
    o_obs = (long)a.nstk * p0;
    o_stk = 4 * p0;
    o_ecur = o_ebest = (long)np * a.nstk * p0;
    if (a.inu_pix) inu = (double)nf;
  }
  // inverse noise weight of row f (one value per Stokes block with windows)
  const double* isg = a.isigmap + (long)pix * a.isig_stride;
  auto isig = [&](int f) -> double {
    return a.poff ? isg[(long)(f / numw) * a.numw] : isg[f];
  };
  const int ld = np + 1;                       // LDS row stride of A and V
  const int npe = np + (np & 1);               // even size for the tournament ordering
  const int ldj = (int)lm_ldj(np), nblk = (int)lm_blocks(np), nquad = (np + 4) / 4;
  // LDS carve-up
  double* A = smem;                            // [npe][ld]  (ld >= npe when np odd: ld = np+1 = npe)
  double* V = A + npe * ld;                    // [npe][ld], in the place of Jn once that is contracted
  double* Jn = V;                              // [LM_CH][ldj]
  double* g = V + max(npe * ld, LM_CH * ldj);  // [np]
  double* dv = g + np;                         // [np] eigenvalues / projections
  double* del = dv + np;                       // [np]
  double* red = del + np;                      // [NT]
  double* rot = red + NT;                      // [npe/2][2]
  double* nzp = rot + npe;                     // [nz]
  double* nod = nzp + nz;                      // [4][np] node work vectors
  double* nrm = nod + 4 * np;                  // [np] PARAM_NORM of each free parameter
  double* pen_res = nrm + np;                  // [np]
  double* pen_hss = pen_res + np;              // [np*np] (only when regularising)
  float* mod = (float*)(pen_hss + (a.regul ? np * np : 0));   // [nheld][nz] current model
  float* bum = mod + LM_MAXHELD * nz;          // [nz]
  float* ftmp = bum + nz;                      // [nz]
  int* izero = (int*)(ftmp + nz);              // [np] zeroed response columns
  int* btab = izero + np;                      // [nblk] (first row << 16 | first column) of each block
  __shared__ double s_sla[9];
  __shared__ int s_accept;

  const long ncol = a.ncol;
  const bool ext = a.gres != nullptr;
  // ---- the pixel's model columns and scalars
  auto load_model = [&](const float* src, float* copy) {
    for (int k = t; k < nz; k += NT) {
      float v[12];
#pragma unroll
      for (int p = 0; p < 12; ++p)
        v[p] = a.rowslot[p] >= 0 || copy ? src[((long)p * nz + k) * ncol + pix] : 0.f;
#pragma unroll
      for (int p = 0; p < 12; ++p) {
        if (a.rowslot[p] >= 0) mod[a.rowslot[p] * nz + k] = v[p];
        if (copy) copy[((long)p * nz + k) * ncol + pix] = v[p];
      }
    }
  };
  load_model(a.atm, nullptr);
  if (t < 9) s_sla[t] = a.sla ? a.sla[(long)pix * 9 + t] : 0.0;
  for (int ip = 0; ip < a.nparam; ++ip)
    for (int j = t; j < a.nj[ip]; j += NT) nrm[a.j0[ip] + j] = c_lm_norm[a.par[ip]];
  const float* ecur = a.eqv + o_ecur;
  __syncthreads();

  // ---- NEW_CALCULATE_CHI2 (get_dmodel.f90:960-1032)
  const double* obs = a.obs + o_obs;
  const float* stk = a.stokes + o_stk;
  const double* sd = a.syn_d ? a.syn_d + o_obs : nullptr;
  // current synthesis of row f
  auto syn = [&](int f) -> double {
    if (sd) return sd[f];
    const int b = f / numw, l = f - b * numw;
    return (double)stk[a.rowstk[b] * numw + l];
  };
  double part = 0.0;
#pragma unroll 4
  for (int f = t; f < nf; f += NT) {
    const double d = obs[f] - syn(f);
    part += d * d * isig(f);
  }
  double chi = team_sum<NT>(part, red) / inu;
  if (a.regul) {
    if (t == 0) lm_penalties(a, mod, pen_res, pen_hss, nod, nod + np);
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < np; ++i) s += pen_res[i] * 1.0 * 1.0 * pen_res[i];
    chi = chi + s;
  }
  if (t == 0) s_accept = (ext || chi < s_sla[2]) ? 1 : 0;
  __syncthreads();
  const bool accept = uniform(s_accept) != 0;
  double* bsyn = ext ? nullptr : a.best_syn + o_obs;
  float* ebest = ext ? nullptr : a.eqv_best + o_ebest;
  const bool tobest = accept && !ext;
  if (ext) {
    // the caller keeps the best model; the step starts from atm
  } else if (accept) {
    // best := current (model and synthesis here, the equivalent response
    // functions as they are read below)
    load_model(a.atm, a.atm_best);
    for (int f = t; f < nf; f += NT) bsyn[f] = syn(f);
  } else {
    // current := best
    load_model(a.atm_best, a.atm);
  }
  __syncthreads();
  if (!accept && a.regul) {
    if (t == 0) lm_penalties(a, mod, pen_res, pen_hss, nod, nod + np);
  }
  if (t == 0 && ext) {
    s_sla[1] = chi;
    s_sla[8] = a.ext_lambda;
  } else if (t == 0) {
    // UPDATE_LAMBDA (get_dmodel.f90:917-956) with INV_SLA(2,3,9,1,4), factor 0.01
    double chicur = chi, chipre = s_sla[2], lam = s_sla[8], steps = s_sla[0], precyc = s_sla[3];
    if ((chipre - chicur) > 0) {
      if ((chipre - chicur) > 0.01 * chipre) steps = fmax(0.0, steps - 1.0);
      else steps = steps + 1.0;
      chipre = chicur;
      lam = lam / sqrt(10.0);
    } else {
      if (fabs(precyc - 1.0) < 1.0e-2) {
        precyc = 0.0;
        lam = lam * 3.0;
      } else {
        lam = lam * 10.0;
      }
      steps = steps + 1.0;
    }
    lam = fmax(1.0e-2, lam);
    s_sla[0] = steps;
    s_sla[1] = chicur;
    s_sla[2] = chipre;
    s_sla[3] = precyc;
    s_sla[8] = lam;
  }
  __syncthreads();

  // ---- normal matrix and gradient of the normalised problem
  //      J_n = J sqrt(w) / sqrt(nu) * PARAM_NORM,  r = (obs - best) sqrt(w) / sqrt(nu)
  // Rows go to LDS in chunks, read along the spectrum; a lane sums blocks of
  // two rows by four columns of [J_n | r]^T J_n, three 16-byte reads for eight
  // products.  The block of the lane's own number stays in registers over the
  // chunks, further ones (more than NT blocks) are summed in A.
  const float* jsrc = accept ? ecur : ebest;
  const double isnu = 1.0 / sqrt(inu);
  for (int i = 2 * t; i < np; i += 2 * NT) {
    int o = 0;
    for (int m = 0; m < i; m += 2) o += nquad - m / 4;
    for (int j = i / 4; j < nquad; ++j) btab[o++] = i << 16 | 4 * j;
  }
  for (int j = t; j < np; j += NT) izero[j] = 0;
  for (int e = t; e < LM_CH * ldj; e += NT) Jn[e] = 0.0;
  auto add_block = [&](int w, const double (&acc)[2][4]) {
    const int i0 = w >> 16, j0 = w & 0xffff;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = i0 + r, j = j0 + c;
        if (i >= np || j < i || j > np) continue;
        if (j < np) A[i * ld + j] += acc[r][c];
        else g[i] += acc[r][c];
      }
  };
  auto sum_block = [&](int w, double (&acc)[2][4]) {
    const double* pi = Jn + (w >> 16);
    const double* pj = Jn + (w & 0xffff);
#pragma unroll 4
    for (int c = 0; c < LM_CH; ++c) {
      const double2 x = *reinterpret_cast<const double2*>(pi + c * ldj);
      const double2 y0 = *reinterpret_cast<const double2*>(pj + c * ldj);
      const double2 y1 = *reinterpret_cast<const double2*>(pj + c * ldj + 2);
      acc[0][0] = fma(x.x, y0.x, acc[0][0]);
      acc[0][1] = fma(x.x, y0.y, acc[0][1]);
      acc[0][2] = fma(x.x, y1.x, acc[0][2]);
      acc[0][3] = fma(x.x, y1.y, acc[0][3]);
      acc[1][0] = fma(x.y, y0.x, acc[1][0]);
      acc[1][1] = fma(x.y, y0.y, acc[1][1]);
      acc[1][2] = fma(x.y, y1.x, acc[1][2]);
      acc[1][3] = fma(x.y, y1.y, acc[1][3]);
    }
  };
  // Columns whose absolute sum overflows REAL(4) are zeroed (forward.f90:672-678).
  // The sum of nf < 1e8 values cannot overflow where none passes 1e30, so a
  // first pass takes every column and notes whether one does; only then are
  // the columns' sums formed and, where one overflows, the pass repeated.
  for (int pass = 0; pass < 2; ++pass) {
    for (int e = t; e < npe * ld; e += NT) A[e] = 0.0;
    for (int i = t; i < np; i += NT) g[i] = 0.0;
    __syncthreads();
    double own[2][4] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
    const int wown = t < nblk ? btab[t] : -1;
    bool large = false;
    // the lane's responses of a chunk, LM_PF columns at a time loaded
    // together and, for the first of them and the row's residual and weight,
    // a chunk ahead: the loads of a chunk would otherwise wait for one another
    // behind its stores
    constexpr int S = NT / LM_CH;
    const int c = t & (LM_CH - 1), jg = t / LM_CH;
    float pf[LM_PF];
    double pw = 0.0, po = 0.0, pb = 0.0;
    auto fetch = [&](int f, int jb, float (&v)[LM_PF]) {
#pragma unroll
      for (int u = 0; u < LM_PF; ++u) {
        const int j = jb + S * u;
        v[u] = f < nf && j < np ? jsrc[(unsigned)(j * nf + f)] : 0.f;
      }
    };
    auto fetch_row = [&](int f) {
      if (f >= nf) return;
      pw = isig(f);
      if (jg == 0) {
        po = ext ? a.gres[o_obs + f] : obs[f];
        pb = ext ? 0.0 : bsyn[f];
      }
    };
    fetch_row(c);
    fetch(c, jg, pf);
    for (int f0 = 0; f0 < nf; f0 += LM_CH) {
      const int f = f0 + c;
      const bool in = f < nf;
      const double w = in ? sqrt(pw) * isnu : 0.0;
      asm volatile("" ::: "memory");   // the columns' norms stay in LDS
      for (int jb = jg; jb < np; jb += S * LM_PF) {
        float v[LM_PF];
        if (jb == jg) {
#pragma unroll
          for (int u = 0; u < LM_PF; ++u) v[u] = pf[u];
        } else {
          fetch(f, jb, v);
        }
#pragma unroll
        for (int u = 0; u < LM_PF; ++u) {
          const int j = jb + S * u;
          if (j >= np) break;
          large = large || fabsf(v[u]) > 1.0e30f;
          if (pass && izero[j]) v[u] = 0.f;
          if (tobest && in) ebest[(unsigned)(j * nf + f)] = v[u];
          Jn[c * ldj + j] = (double)v[u] * w * nrm[j];
        }
      }
      if (jg == 0) Jn[c * ldj + np] = in ? (po - pb) * w : 0.0;
      if (f0 + LM_CH < nf) {
        fetch_row(f + LM_CH);
        fetch(f + LM_CH, jg, pf);
      }
      __syncthreads();
      if (wown >= 0) sum_block(wown, own);
      for (int q = t + NT; q < nblk; q += NT) {
        double acc[2][4] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
        sum_block(btab[q], acc);
        add_block(btab[q], acc);
      }
      __syncthreads();
    }
    if (wown >= 0) add_block(wown, own);
    if (pass || !accept || !__syncthreads_or(large)) break;
    bool over = false;
    for (int j = wv; j < np; j += NT / 64) {
      float s = 0.f;
      for (int f = lane; f < nf; f += 64) s += fabsf(ecur[(long)j * nf + f]);
      const bool z = wave_sum((double)s) > (double)3.40282347e38f;
      if (lane == 0) izero[j] = z ? 1 : 0;
      over = over || z;
    }
    if (!__syncthreads_or(over)) break;
  }
  __syncthreads();
  const double lam = s_sla[8];
  if (ext && a.hscale != 1.0) {
    for (int e = t; e < np * np; e += NT) {
      const int i = e / np, j = e - i * np;
      if (j >= i) A[i * ld + j] *= a.hscale;
    }
    __syncthreads();
  }
  // A = H + REG_HSS, diag += diag * lambda; g = J^T r - REG_PEN
  for (int e = t; e < np * np; e += NT) {
    const int i = e / np, j = e - i * np;
    if (j < i) A[i * ld + j] = A[j * ld + i];
  }
  for (int i = t; i < np; i += NT)
    if (a.regul) g[i] -= pen_res[i];
  __syncthreads();
  if (a.regul)
    for (int e = t; e < np * np; e += NT) {
      const int i = e / np, j = e - i * np;
      A[i * ld + j] += pen_hss[e];
    }
  __syncthreads();
  for (int i = t; i < np; i += NT) A[i * ld + i] = A[i * ld + i] + A[i * ld + i] * lam;
  for (int e = t; e < npe * ld; e += NT) V[e] = 0.0;
  __syncthreads();
  for (int i = t; i < np; i += NT) V[i * ld + i] = 1.0;
  __syncthreads();

  // ---- damped solve (symmetric eigen-decomposition or CG)
  damped_solve<NT>(a.solver, a.svdtol, np, A, V, g, dv, del, red, rot, nod);
  __syncthreads();
  // NaN filter (get_dmodel.f90:806-822)
  if (t == 0) {
    double s = 0.0;
    for (int i = 0; i < np; ++i) s += del[i];
    if (s != s)
      for (int i = 0; i < np; ++i)
        if (del[i] != del[i]) del[i] = 0.0;
  }
  __syncthreads();

  // ---- LIMIT_PERTURBATION -> REARANGE_DA_MODEL -> SORT_DELTA_TO_ATMOSPHERE
  double* itd = nod;            // [np] scaled / limited node perturbation
  double* sumv = nod + 2 * np;  // [np]
  // node mean of a column: a wave per node, its lanes along the heights
  auto node_mean = [&](const float* x, int j) -> double {
    const double* cf = a.coefs + (long)j * nz;
    const double cs = a.colsum[j];
    double s = 0.0;
    for (int k = lane; k < nz; k += 64) s = fma((double)x[k], cf[k], s);
    return wave_sum(s) / cs;
  };
  for (int ip = 0; ip < a.nparam; ++ip) {
    const int p = a.par[ip], j0 = a.j0[ip], nj = a.nj[ip];
    float* col = mod + a.mslot[ip] * nz;
    const double factor = c_lm_norm[p], inf = c_lm_low[p], sup = c_lm_upp[p];
    const double absolute = c_lm_norm[p] * a.mpert;
    for (int k = t; k < nz; k += NT) bum[k] = col[k];
    for (int j = wv; j < nj; j += NT / 64) {
      const double av = node_mean(col, j0 + j);
      double lim;
      if (absolute > 0) lim = fmax(absolute, fabs(a.mpert * av));
      else lim = fabs(a.mpert * av);
      if (av == 0) lim = absolute;
      double x = del[j0 + j] * factor;
      if (fabs(x) > lim) x = x / fabs(x) * lim;
      if (lane == 0) {
        itd[j] = x;
        sumv[j] = av + x;
        del[j0 + j] = x;
      }
    }
    __syncthreads();
    for (int k = t; k < nz; k += NT) {
      double s = 0.0;
      for (int j = 0; j < nj; ++j) s = s + sumv[j] * a.coefs[(long)(j0 + j) * nz + k];
      nzp[k] = s;
    }
    __syncthreads();
    if (a.node_expansion == 2) {
      for (int k = t; k < nz; k += NT) {
        float o = (float)nzp[k];
        if ((double)o < inf) o = (float)inf;
        if ((double)o > sup) o = (float)sup;
        col[k] = o - col[k];
      }
    } else if (a.node_expansion == 1) {
      for (int k = t; k < nz; k += NT) {
        nzp[k] = nzp[k] - (double)col[k];
        ftmp[k] = (float)nzp[k];
      }
      __syncthreads();
      for (int j = wv; j < nj; j += NT / 64) {
        const double x = node_mean(ftmp, j0 + j);
        if (lane == 0) {
          itd[j] = x;
          del[j0 + j] = x;
        }
      }
      __syncthreads();
      for (int k = t; k < nz; k += NT) {
        double s = 0.0;
        for (int j = 0; j < nj; ++j) s = s + itd[j] * a.coefs[(long)(j0 + j) * nz + k];
        const float o = col[k] + (float)s;
        if ((double)o < inf) s = inf - (double)col[k];
        if ((double)o > sup) s = sup - (double)col[k];
        col[k] = (float)s;
      }
    }
    __syncthreads();
    if (p == 0 && t < 64) {
      // temperature tail rule in log tau5 (get_dmodel.f90:1970-1984), top
      // down: damped above tllim, and below tulim the value of the height
      // above, so of the nearest height above that does not take another's
      const float* tau = mod + a.rowslot[A_TAU] * nz;
      const float tllim = -11.5f, tulim = 0.5f;
      float carry = 0.f;
      for (int kb = (nz - 1) / 64 * 64; kb >= 0; kb -= 64) {
        const int k = kb + lane;
        const bool in = k < nz;
        const float tk = in ? tau[k] : 0.f;
        float v = in ? col[k] : 0.f;
        if (tk < tllim) {
          const float x = fabsf(tk - tllim) / 0.5f;
          v = expf(-(x * x)) * v;
        }
        const unsigned long long keep = __ballot(in && (!(tk > tulim) || k == nz - 1)) >> lane;
        const float from = __shfl(v, keep ? lane + __builtin_ctzll(keep) : lane);
        if (in && tk > tulim && k != nz - 1) v = keep ? from : carry;
        if (in) col[k] = v;
        carry = __shfl(v, 0);
      }
    }
    __syncthreads();
    for (int k = t; k < nz; k += NT) col[k] = col[k] + bum[k];
    __syncthreads();
  }

  // ---- write back the inverted columns (the others are in place)
#pragma unroll 1
  for (int p = 0; p < 12; ++p) {
    const int sl = a.rowslot[p];
    if (sl < 0 || p == A_TAU) continue;
    for (int k = t; k < nz; k += NT) a.atm[((long)p * nz + k) * ncol + pix] = mod[sl * nz + k];
  }
  if (t < 9 && a.sla) a.sla[(long)pix * 9 + t] = s_sla[t];
  if (a.delta)
    for (int i = t; i < np; i += NT) a.delta[(long)pix * np + i] = del[i];
  if (t == 0 && !ext && a.done && s_sla[0] > a.maxsteps) a.done[pix] = 1;
}

// bytes of lm_kernel's work arrays (LDS, or the device-memory slice of one
// pixel) for np free parameters, nz heights and nt threads
inline size_t lm_lds_bytes(int np, int nz, bool regul, int nt) {
  const size_t npe = np + (np & 1), ld = np + 1;
  const size_t d = npe * ld + std::max(npe * ld, LM_CH * lm_ldj(np)) + 3 * (size_t)np + nt + npe + nz + 4 * (size_t)np +
                   2 * (size_t)np + (regul ? (size_t)np * np : 0);
  const size_t f = (size_t)(LM_MAXHELD + 2) * nz + np + lm_blocks(np);   // floats + ints
  return d * 8 + f * 4;
}

}  // namespace fz
