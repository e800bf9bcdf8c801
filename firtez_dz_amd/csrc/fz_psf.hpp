// Spatial PSF of the coupled inversion: a periodic 2-D convolution of maps on
// the (x, y) grid, and its adjoint.
//
// The reference reads the PSF (READ_PSF, pre_post_duties.f90:488-555), embeds
// the central (2 YS + 1) x (2 XS + 1) part in an NY x NX array centred at
// (NY/2 + 1, NX/2 + 1), shifts the centre to (1, 1) and multiplies Fourier
// transforms (SPATIAL_CONV_INIT :559-588, SMOOTH_MODEL invert3d.f90:412-488):
// a circular convolution,
//   out(y, x) = sum_{dy, dx} PSF(Y0 + dy, X0 + dx) in(y - dy mod NY, x - dx mod NX).
// Here the same sum is formed directly (a 31 x 31 PSF is 961 taps per
// output), which needs no FFT library and keeps the result exact to FP32
// summation: psf_split_kernel on the matrix cores, psf_conv_kernel on the
// vector units for PSFs of up to 16 pixels in x and taps outside the range of the
// former.  The adjoint (the transpose
// of the convolution, used for the gradient of the coupled chi^2) is the
// correlation out(y, x) = sum PSF(Y0 + dy, X0 + dx) in(y + dy, x + dx).
//
// psf_conv_kernel: maps channel-major, map m at in[m * npix + col] with
// col = y + ny * x (the cube's column order), so a map is an nx x ny image
// with y contiguous.  One workgroup of four waves computes a 32 (x) x 64 (y)
// output tile of one map: the lanes of a wave take 64 consecutive y, and
// each lane 8 consecutive x.  The (32 + NTX - 1) x (64 + 2 ry) input tile is
// staged in LDS with the periodic wrap applied at load.  For each of the
// 2 ry + 1 tap rows along y, a lane reads the strip of 8 + NTX - 1 inputs
// along x that its 8 outputs need into registers (conflict-free: the 64
// lanes read 64 consecutive words) and applies the NTX taps of that row,
// wave-uniform scalar loads, to all 8 outputs: 8 NTX FMAs per
// 8 + NTX - 1 LDS reads, which keeps the FP32 VALU, not LDS bandwidth, the
// bound.  NTX is the x-tap count 2 rx + 1 rounded up to a multiple of 8;
// the padding taps are zero and the padding rows of the tile hold wrapped
// (finite) inputs.
#pragma once

namespace fz {

constexpr int PSF_OX = 8;                  // outputs per lane along x
constexpr int PSF_TX = 4 * PSF_OX;         // output tile along x (four waves)
constexpr int PSF_TY = 64;                 // output tile along y (the lanes of a wave)
constexpr int PSF_RMAX = 31;               // largest tap radius (63 x 63 PSF)

// K steps of 32 that the band of 32 outputs and ntx taps takes
constexpr int psf_steps(int ntx) { return ntx > 32 ? 3 : 2; }

struct PsfArgs {
  int nx, ny, nmaps, rx, ry;
  long npix;
  // [2 ry + 1][NTX] taps in the tile's order: taps[u * NTX + t] multiplies
  // tile row (x) offset t and column (y) offset u of the output's window
  // (the PSF reversed for the convolution, as given for the adjoint)
  const float* taps;
  const float* in;
  float* out;
};

// One 32 x 64 tile from (x0, y0), by all 256 threads; tile: LDS
template <int NTX>
__device__ __forceinline__ void psf_vector(const PsfArgs& a, int x0, int y0, const float* __restrict__ src,
                                           float* __restrict__ dst, float* tile) {
  constexpr int NW = PSF_OX + NTX - 1;     // register strip along x
  constexpr int ROWS = PSF_TX + NTX - 1;   // tile rows (x)
  const int cols = PSF_TY + 2 * a.ry;      // tile columns (y)
  // tile[i][j] = in(x0 - rx + i, y0 - ry + j), periodic in x and y
  for (int e = threadIdx.x; e < ROWS * cols; e += 256) {
    const int i = e / cols, j = e - i * cols;
    int x = (x0 - a.rx + i) % a.nx;
    if (x < 0) x += a.nx;
    int y = (y0 - a.ry + j) % a.ny;
    if (y < 0) y += a.ny;
    tile[e] = src[(long)x * a.ny + y];
  }
  __syncthreads();
  const int ty = threadIdx.x & 63, xw = (threadIdx.x >> 6) * PSF_OX;
  float acc[PSF_OX];
#pragma unroll
  for (int i = 0; i < PSF_OX; ++i) acc[i] = 0.f;
  const int nu = 2 * a.ry + 1;
  for (int u = 0; u < nu; ++u) {
    // output (xw + i, ty) reads tile row xw + i + t, column ty + u
    const float* colp = tile + xw * cols + ty + u;
    float v[NW];
#pragma unroll
    for (int j = 0; j < NW; ++j) v[j] = colp[j * cols];
    const float* k = a.taps + u * NTX;
#pragma unroll
    for (int t = 0; t < NTX; ++t) {
      const float kt = k[t];
#pragma unroll
      for (int i = 0; i < PSF_OX; ++i) acc[i] = fmaf(kt, v[i + t], acc[i]);
    }
  }
  const int y = y0 + ty;
  if (y >= a.ny) return;
#pragma unroll
  for (int i = 0; i < PSF_OX; ++i) {
    const int x = x0 + xw + i;
    if (x < a.nx) dst[(long)x * a.ny + y] = acc[i];
  }
}

template <int NTX>
__global__ void __launch_bounds__(256) psf_conv_kernel(PsfArgs a) {
  extern __shared__ float tile[];
  psf_vector<NTX>(a, blockIdx.y * PSF_TX, blockIdx.x * PSF_TY, a.in + (long)blockIdx.z * a.npix,
                  a.out + (long)blockIdx.z * a.npix, tile);
}

// The convolution on the matrix cores.  Inputs and taps are split into three BF16
// parts each (8 + 8 + 8 bits: x = hi + mid + lo exactly), and six of the nine
// products of parts are summed in FP32; the three left out are below 2^-24 of
// the product.  For a tap row u the outputs of 32 x are a banded Toeplitz matrix of the
// taps (two 16 x (32 KS) operands, in operand order from memory, the same for
// every tile) times the strip of 32 + 2 rx inputs, which lies in LDS with x contiguous
// so that 16 y and 32 x are one operand at any row y + u.
//
// A workgroup has 32 x and 32 YT y of one map: of its four waves two have
// half the y each, two the even and two the odd tap rows, added at the end.  Per tap row
// a wave reads 6 KS tap operands (a row ahead) and 3 KS YT input operands for
// 12 KS YT MFMAs.  Bound: these, (2 rx + 1) / (32 KS) of whose products are taps.
// Error against 64 bits (448 maps of 256 x 256, 31 x 31 taps): 1.6e-7 of the
// result, with the vector units' sums 4.7e-7; time 0.49 ms for 0.97.
//
// A tile with an input that is not finite, beyond 2^120 or, not being zero,
// below 2^-100, where the parts would leave BF16's range, takes psf_vector.  All
// tiles there, ms for psf_conv_kernel's: 448 maps of 256 x 256, 31 x 31 taps 0.96 (0.96);
// 4 maps of 64 x 64, 63 x 63 0.112 (0.108); 64 maps of 256 x 256, 63 x 63, where the
// operands' LDS leaves one workgroup to a CU, 0.88 (0.56).  (With the tap count at run
// time 1.14, 0.147 and 1.06; a row's inputs a row ahead 1.10, 0.118 and 1.02.)
template <int NTX, int YT>
__global__ void __launch_bounds__(256) psf_split_kernel(PsfArgs a, const bf16* __restrict__ frag) {
  extern __shared__ __attribute__((aligned(16))) char psf_lds[];
  __shared__ int flag[4];
  constexpr int KS = psf_steps(NTX), XP = 32 * KS + 8, TY = 32 * YT;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int x0 = blockIdx.y * PSF_TX, y0 = blockIdx.x * TY;
  const int rows = TY + 2 * a.ry, nk = PSF_TX + 2 * a.rx, nu = 2 * a.ry + 1;
  const float* src = a.in + (long)blockIdx.z * a.npix;
  float* dst = a.out + (long)blockIdx.z * a.npix;
  bf16* plane = reinterpret_cast<bf16*>(psf_lds);
  const int ps = rows * XP;
  bool bad = false;
  for (int e = threadIdx.x; e < rows * 4 * KS; e += 256) {
    const int g = e / rows, j = e - g * rows;
    // (rx < nx, ry < ny; small maps go round more than once)
    int y = y0 - a.ry + j, x = x0 - a.rx + 8 * g;
    y += y < 0 ? a.ny : 0;
    x += x < 0 ? a.nx : 0;
    while (y >= a.ny) y -= a.ny;
    while (x >= a.nx) x -= a.nx;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = 8 * g + i < nk ? src[(long)x * a.ny + y] : 0.f;
      x = x + 1 == a.nx ? 0 : x + 1;
    }
    bf16x8 p0, p1, p2;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned b = __float_as_uint(v[i]) & 0x7fffffffu;
      bad |= b > 0x7b800000u || (b != 0 && b < 0x0d800000u);
      p0[i] = (bf16)v[i];
      const float r = v[i] - (float)p0[i];
      p1[i] = (bf16)r;
      p2[i] = (bf16)(r - (float)p1[i]);
    }
    bf16* o = plane + j * XP + 8 * g;
    *reinterpret_cast<bf16x8*>(o) = p0;
    *reinterpret_cast<bf16x8*>(o + ps) = p1;
    *reinterpret_cast<bf16x8*>(o + 2 * ps) = p2;
  }
  const bool any = __ballot(bad) != 0;
  if (lane == 0) flag[wave] = any;
  __syncthreads();
  if (flag[0] | flag[1] | flag[2] | flag[3]) {
#pragma unroll 1
    for (int h = 0; h < TY && y0 + h < a.ny; h += PSF_TY) {
      __syncthreads();
      psf_vector<NTX>(a, x0, y0 + h, src, dst, reinterpret_cast<float*>(psf_lds));
    }
    return;
  }
  f32x4 acc[2][YT];
#pragma unroll
  for (int i = 0; i < 2 * YT; ++i) acc[i & 1][i >> 1] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int yb = (wave & 1) * 16 * YT;
  const bf16x8* F = reinterpret_cast<const bf16x8*>(frag) + lane;
  constexpr int NF = 6 * KS;     // tap operands of a row: [x tile][step][part]
  bf16x8 t[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) t[i] = F[(min(wave >> 1, nu - 1) * NF + i) * 64];
  for (int u = wave >> 1; u < nu; u += 2) {
    bf16x8 n[NF];
    const int un = min(u + 2, nu - 1);
#pragma unroll
    for (int i = 0; i < NF; ++i) n[i] = F[(un * NF + i) * 64];
    __builtin_amdgcn_sched_barrier(0);   // keeps the loads here, a row ahead
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int yt = 0; yt < YT; ++yt) {
        const bf16* b = plane + (yb + 16 * yt + lr + u) * XP + 32 * s + 8 * lg;
        const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(b), b1 = *reinterpret_cast<const bf16x8*>(b + ps),
                     b2 = *reinterpret_cast<const bf16x8*>(b + 2 * ps);
#pragma unroll
        for (int xt = 0; xt < 2; ++xt) {
          const bf16x8 *c = t + (xt * KS + s) * 3;
          f32x4 d = acc[xt][yt];
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[0], b2, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[2], b0, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[1], b1, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[0], b1, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[1], b0, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[0], b0, d, 0, 0, 0);
          acc[xt][yt] = d;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) t[i] = n[i];
  }
  // the odd rows' sums to the waves of the even ones
  f32x4* red = reinterpret_cast<f32x4*>(psf_lds);
  __syncthreads();
  if (wave >= 2)
#pragma unroll
    for (int i = 0; i < 2 * YT; ++i) red[((wave & 1) * 2 * YT + i) * 64 + lane] = acc[i & 1][i >> 1];
  __syncthreads();
  if (wave >= 2) return;
#pragma unroll
  for (int i = 0; i < 2 * YT; ++i) {
    const f32x4 d = acc[i & 1][i >> 1] + red[(wave * 2 * YT + i) * 64 + lane];
    const int y = y0 + yb + 16 * (i >> 1) + lr, x = x0 + 16 * (i & 1) + 4 * lg;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (y < a.ny && x + q < a.nx) dst[(long)(x + q) * a.ny + y] = d[q];
  }
}

// Operands of psf_split_kernel from the taps [direction, u][ntx], a lane's
// eight k (16 bytes) per thread: tap t of output i of the 32 is at input k = i + t,
// its parts as the kernel splits its inputs.  A new PSF and its first convolution
// (4 maps of 64 x 64) took 250 us for 31 x 31 taps and 880 for 63 x 63 when the host
// built and copied these 0.8 and 2.3 MB, and take 51 and 71.
__global__ void __launch_bounds__(256) psf_operand_kernel(const float* __restrict__ taps, int npiece, int ks, int ntx,
                                                          bf16* __restrict__ frag) {
  const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (e >= npiece) return;
  int q = e >> 6;
  const int lane = e & 63, part = q % 3;
  q /= 3;
  const int s = q % ks;
  q /= ks;
  const int i = 16 * (q & 1) + (lane & 15), k0 = 32 * s + 8 * (lane >> 4), du = q >> 1;
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t = k0 + j - i;
    const float v = t >= 0 && t < ntx ? taps[du * ntx + t] : 0.f;
    const bf16 p0 = (bf16)v;
    const float r = v - (float)p0;
    const bf16 p1 = (bf16)r;
    o[j] = part == 0 ? p0 : part == 1 ? p1 : (bf16)(r - (float)p1);
  }
  reinterpret_cast<bf16x8*>(frag)[e] = o;
}

// 32 x 32 transpose through LDS: out[c][r] = in[r][c] for an R x C matrix
// (in row stride C, out row stride R), converting the element type
template <class Tin, class Tout>
__global__ void __launch_bounds__(256) transpose_kernel(const Tin* __restrict__ in, Tout* __restrict__ out, long R,
                                                        long C) {
  __shared__ Tin t[32][33];
  const long r0 = (long)blockIdx.y * 32, c0 = (long)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8 threads
  for (int k = ty; k < 32; k += 8) {
    const long r = r0 + k, c = c0 + tx;
    if (r < R && c < C) t[k][tx] = in[r * C + c];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const long c = c0 + k, r = r0 + tx;
    if (r < R && c < C) out[c * R + r] = (Tout)t[tx][k];
  }
}

}  // namespace fz

namespace fz {

// The coupled residual: from the PSF-convolved synthesis maps conv
// ([4 numw][npix], channel-major) take the inverted Stokes rows, and per
// pixel write syn_c and r = obs - syn_c ([npix][nfreq]) and its chi^2 (the
// weighted sum over the rows / inu).  One thread per pixel.
struct CoupledArgs {
  int npix, nfreq, numw, nstk;
  int rowstk[4];
  double inu;
  const float* conv;
  const double* obs;
  const double* isig;   // [nfreq]
  double* syn_c;
  double* res;
  double* chi;          // [npix]
};

__global__ void __launch_bounds__(256) coupled_resid_kernel(CoupledArgs a) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.npix) return;
  double s = 0.0;
  for (int f = 0; f < a.nfreq; ++f) {
    const int b = f / a.numw, l = f - b * a.numw;
    const double sy = (double)a.conv[(long)(a.rowstk[b] * a.numw + l) * a.npix + p];
    const double r = a.obs[(long)p * a.nfreq + f] - sy;
    a.syn_c[(long)p * a.nfreq + f] = sy;
    a.res[(long)p * a.nfreq + f] = r;
    s += r * r * a.isig[f];
  }
  a.chi[p] = s / a.inu;
}

// sum of n doubles by one workgroup (fixed order for a given n)
__global__ void __launch_bounds__(256) sum_kernel(const double* __restrict__ x, int n, double* __restrict__ out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += x[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

}  // namespace fz
