// Learned initial model for the inversion: a small fully connected network
// (Stokes profiles -> node values of T, Bz, B_perp cos 2phi, B_perp sin 2phi,
// v_z) with BF16 weights and activations and FP32 accumulation on the MFMA
// units.  The reference has no counterpart: its initial model is the input
// model file (invert3d.f90:57-178); the inversion itself is unchanged.
//
// Every BF16 matrix R x K is stored in the order in which the MFMA operands
// are read (frag_at): 16 rows x 32 k are one kilobyte, a lane's eight k
// together, so that an operand is one 16-byte load per lane from consecutive
// addresses, without LDS.  Rows and K are padded to multiples of 32, the K
// padding with zeros; padding rows hold anything.  What a later product
// contracts over the batch is stored transposed as well by the kernel that
// makes it, so that every product is D[m][n] = sum_k B[m][k] A[n][k].
//
//   mlp_infer_kernel     all layers of 16, 32 or 64 rows in one workgroup, from
//                        the observed profiles to the network output or the
//                        initial model
//   mlp_layer_kernel     one layer of a batch with its epilogue (bias, ReLU;
//                        loss and its gradient; ReLU' mask and column sums)
//   mlp_dw_kernel        all weight gradients, bias gradients and the loss
//   mlp_input_kernel     standardised BF16 inputs (optionally gathered by a
//                        permutation of the training set)
//   mlp_adam_kernel      Adam on FP32 master weights, refreshing the BF16 copies
//   mlp_targets_kernel   training targets from a model cube (least-squares
//                        node values through a pseudo-inverse of the node basis)
//   mlp_decode_kernel    network output -> initial model rows (node expansion)
#pragma once

namespace fz {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int MLP_MAXNODE = 8;
constexpr int MLP_NQ = 5;      // quantities per node: T, Bz, Bp cos2phi, Bp sin2phi, vz
constexpr int MLP_MAXLAYER = 7;

__host__ __device__ inline int pad32(int n) { return (n + 31) & ~31; }
__host__ __device__ inline size_t frag_size(int rows, int k) { return (size_t)pad32(rows) * pad32(k); }
// element (r, k) of a matrix of ks = pad32(K) / 32 steps
__host__ __device__ inline size_t frag_at(int r, int k, int ks) {
  return (((size_t)(r >> 4) * ks + (k >> 5)) * 64 + (r & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

// network shape and where its parameters are: W_l row-major [out][in] and b_l
// in the flat FP32 vector, wb / wt the BF16 copies [out][in] and [in][out]
struct MlpShape {
  int nl;                              // hidden layers
  int nin, nout, nj, nz;
  int din[MLP_MAXLAYER], dout[MLP_MAXLAYER];
  long woff[MLP_MAXLAYER], boff[MLP_MAXLAYER];
  long wb[MLP_MAXLAYER], wt[MLP_MAXLAYER];
};

// D[m][n] = sum over ks steps of 32 of B[m][k] A[n][k], m < M, n < N; tn tiles along n
struct GemmArgs {
  const bf16 *A, *B;
  int ks, M, N, tn, tile0;
  const float* bias;      // [N]
  const bf16* mask;       // like Cb: the result is zeroed where the mask is not positive
  float* Cf;              // FP32 result [M][N]
  bf16 *Cb, *CbT;         // BF16 result and its transpose (optional)
  float* csum;            // [pad32(M) / 16][pad32(N)] column sums of 16 rows
};

// acc[i][j] += the products of steps s0 .. s1 of FA fragments of A and FB of B
// (their first operands at A and B, ks steps apart): the loads of CH steps together
// and a chunk ahead, the additions in the order of the steps.  MFMA operand
// layout (16x16x32, BF16): lane l holds row l % 16 with 8 consecutive k of
// the lane group l / 16; the accumulator holds D[row of A 4 (l / 16) + q][row
// of B l % 16], q = 0..3: here four consecutive n of one m.
template <int FA, int FB, int CH>
__device__ __forceinline__ void gemm_steps(const bf16x8* __restrict__ A, const bf16x8* __restrict__ B, int ks, int s0,
                                           int s1, f32x4 (&acc)[FA][FB]) {
  if (s0 >= s1) return;
  bf16x8 a[CH][FA], b[CH][FB];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int s = min(s0 + u, s1 - 1);
#pragma unroll
    for (int i = 0; i < FA; ++i) a[u][i] = A[((size_t)i * ks + s) * 64];
#pragma unroll
    for (int j = 0; j < FB; ++j) b[u][j] = B[((size_t)j * ks + s) * 64];
  }
  for (int s = s0; s < s1; s += CH) {
    bf16x8 an[CH][FA], bn[CH][FB];
    const bool more = s + CH < s1;
    if (more) {
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int t = min(s + CH + u, s1 - 1);
#pragma unroll
        for (int i = 0; i < FA; ++i) an[u][i] = A[((size_t)i * ks + t) * 64];
#pragma unroll
        for (int j = 0; j < FB; ++j) bn[u][j] = B[((size_t)j * ks + t) * 64];
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (s + u >= s1) break;
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
    }
    if (!more) break;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
#pragma unroll
      for (int i = 0; i < FA; ++i) a[u][i] = an[u][i];
#pragma unroll
      for (int j = 0; j < FB; ++j) b[u][j] = bn[u][j];
    }
  }
}

__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

struct LossArgs {
  const float *T, *tmean, *tstd;
  const int32_t* idx;
  float* part;              // [4 tiles] sums of the squares
  int rows;                 // of the whole batch, whose mean the loss is
};

enum { MLP_HIDDEN = 0, MLP_OUT = 1, MLP_LOSS = 2, MLP_DACT = 3 };

// HIDDEN: Cb = ReLU(D + bias).  OUT: Cf = D + bias.  LOSS: the squared
// differences of D + bias from the standardised targets, and their gradient
// dY = 2 (Y - (T - tmean) / tstd) / (rows N) into Cb.  DACT: Cb = D where the mask is
// positive.  CbT gets Cb's transpose, csum the column sums of the FP32 values.
// The sums over K run in one order whatever the tile (a regrouped sum
// rounds some activations the other way).  Each of the four waves has FR x FR
// fragments of a tile of 32 FR rows and columns.  FR = 1 is bounded by the
// latency of two or three rounds of loads: 1024 x 512 x 512 takes 5.3 us,
// where 64 x 64 tiles staged through LDS with a barrier per K step took 25.  FR
// = 2 halves the operands' traffic and is taken once its tiles fill the chip twice.
template <int MODE, int FR>
__global__ void __launch_bounds__(256) mlp_layer_kernel(GemmArgs g, LossArgs ls) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tm = (int)blockIdx.x / g.tn, tn = (int)blockIdx.x - tm * g.tn;
  const int fm = (2 * tm + (wave & 1)) * FR, fn = (2 * tn + (wave >> 1)) * FR;   // first fragments
  float e2 = 0.f;
  if (16 * fm < pad32(g.M) && 16 * fn < pad32(g.N)) {
    f32x4 acc[FR][FR];
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
      for (int j = 0; j < FR; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    gemm_steps<FR, FR, FR == 1 ? 8 : 4>(reinterpret_cast<const bf16x8*>(g.A) + (size_t)fn * g.ks * 64 + lane,
                                        reinterpret_cast<const bf16x8*>(g.B) + (size_t)fm * g.ks * 64 + lane, g.ks, 0,
                                        g.ks, acc);
#pragma unroll
    for (int j = 0; j < FR; ++j) {
      const int m = 16 * (fm + j) + (lane & 15);
      const long row = MODE == MLP_LOSS && m < g.M ? (ls.idx ? (long)ls.idx[m] : (long)m) : 0;
#pragma unroll
      for (int i = 0; i < FR; ++i) {
        const int n = 16 * (fn + i) + 4 * (lane >> 4);
        const size_t at = frag_at(m, n, pad32(g.N) >> 5);
        float v[4];
        bf16x4 mk;
        if constexpr (MODE == MLP_DACT) mk = *reinterpret_cast<const bf16x4*>(g.mask + at);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool in = m < g.M && n + q < g.N;
          v[q] = acc[i][j][q];
          if constexpr (MODE != MLP_DACT) v[q] += in ? g.bias[n + q] : 0.f;
          if constexpr (MODE == MLP_HIDDEN) v[q] = v[q] > 0.f ? v[q] : 0.f;
          if constexpr (MODE == MLP_DACT)
            if (!((float)mk[q] > 0.f)) v[q] = 0.f;
          if constexpr (MODE == MLP_LOSS) {
            if (in) {
              const float tn = (ls.T[row * g.N + n + q] - ls.tmean[n + q]) / ls.tstd[n + q];
              const float df = v[q] - tn;
              e2 += df * df;
              v[q] = 2.f * df / ((float)ls.rows * (float)g.N);
            }
          }
          if (!in) v[q] = 0.f;
          if constexpr (MODE == MLP_OUT)
            if (in) g.Cf[(size_t)m * g.N + n + q] = v[q];
        }
        if constexpr (MODE != MLP_OUT) {
          bf16x4 w;
#pragma unroll
          for (int q = 0; q < 4; ++q) w[q] = (bf16)v[q];
          *reinterpret_cast<bf16x4*>(g.Cb + at) = w;
          if (g.CbT)
#pragma unroll
            for (int q = 0; q < 4; ++q) g.CbT[frag_at(n + q, m, pad32(g.M) >> 5)] = w[q];
        }
        if constexpr (MODE == MLP_LOSS || MODE == MLP_DACT) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = sum16(v[q]);
          if ((lane & 15) == 0)
            *reinterpret_cast<float4*>(g.csum + (size_t)(fm + j) * pad32(g.N) + n) =
                make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    }
  }
  if constexpr (MODE == MLP_LOSS) {
    e2 = sum16(e2);
    e2 += __shfl_xor(e2, 16, 64);
    e2 += __shfl_xor(e2, 32, 64);
    if (lane == 0) ls.part[blockIdx.x * 4 + wave] = e2;
  }
}

// One 32 x 32 tile of a weight gradient, whose K is the batch: the four waves of a
// workgroup share out the steps and then own one 16 x 16 quarter each, the
// partial sums added in a fixed order.
__device__ __forceinline__ f32x4 gemm_tile(const GemmArgs& g, int tile, f32x4* __restrict__ red, int& m, int& n) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tm = tile / g.tn, tn = tile - tm * g.tn, ks = g.ks;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = (f32x4){0.f, 0.f, 0.f, 0.f};
  gemm_steps<2, 2, 4>(reinterpret_cast<const bf16x8*>(g.A) + (size_t)(2 * tn) * ks * 64 + lane,
                      reinterpret_cast<const bf16x8*>(g.B) + (size_t)(2 * tm) * ks * 64 + lane, ks,
                      (int)((long)wave * ks / 4), (int)((long)(wave + 1) * ks / 4), acc);
#pragma unroll
  for (int i = 0; i < 4; ++i) red[(wave * 4 + i) * 64 + lane] = acc[i >> 1][i & 1];
  __syncthreads();
  m = 32 * tm + 16 * (wave & 1) + (lane & 15);
  n = 32 * tn + 16 * (wave >> 1) + 4 * (lane >> 4);
  return (red[wave * 64 + lane] + red[(4 + wave) * 64 + lane]) +
         (red[(8 + wave) * 64 + lane] + red[(12 + wave) * 64 + lane]);
}

// All of a batch's sums over its rows in one launch: the weight gradients
// dW_l[o][k] = sum_m dZ_l[m][o] A_l[m][k] (a tile per workgroup), the bias gradients
// from the column sums (16 of one layer per workgroup), the loss (one).
struct DwArgs {
  int n;                             // layers
  GemmArgs g[MLP_MAXLAYER];          // M = dout, N = din, Cf = the layer's gradient
  int nparts;                        // partial column sums
  int blk0[MLP_MAXLAYER];            // first workgroup of the layer's biases
  const float* csum[MLP_MAXLAYER];
  float* bg[MLP_MAXLAYER];
  int loss_blk, nloss;
  const float* lpart;
  float lscale;
  float* loss;
  int add;                           // to what the rows before this launch's gave
};

__global__ void __launch_bounds__(256) mlp_dw_kernel(DwArgs a) {
  __shared__ f32x4 red[16 * 64];
  const int blk = (int)blockIdx.x, t = threadIdx.x;
  float* fr = reinterpret_cast<float*>(red);
  if (blk < a.blk0[0]) {
    int l = 0;
    while (l + 1 < a.n && blk >= a.g[l + 1].tile0) ++l;
    const GemmArgs& g = a.g[l];
    int m, n;
    f32x4 d = gemm_tile(g, blk - g.tile0, red, m, n);
    if (m >= g.M) return;
    float* o = g.Cf + (size_t)m * g.N + n;
    if (a.add)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < g.N) d[q] += o[q];
    if (n + 3 < g.N && ((uintptr_t)o & 15) == 0)
      *reinterpret_cast<f32x4*>(o) = d;
    else
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < g.N) o[q] = d[q];
    return;
  }
  if (blk < a.loss_blk) {
    int l = 0;
    while (l + 1 < a.n && blk >= a.blk0[l + 1]) ++l;
    const int o = (blk - a.blk0[l]) * 16 + (t & 15), no = a.g[l].M, p = pad32(no);
    const float* c = a.csum[l] + o;
    float s = 0.f;
    if (o < no)
      for (int i = t >> 4; i < a.nparts; i += 16) s += c[(size_t)i * p];
    fr[t] = s;
    __syncthreads();
    for (int h = 128; h >= 16; h >>= 1) {
      if (t < h) fr[t] += fr[t + h];
      __syncthreads();
    }
    if (t < 16 && o < no) a.bg[l][o] = a.add ? a.bg[l][o] + fr[t] : fr[t];
    return;
  }
  float s = 0.f;
  for (int i = t; i < a.nloss; i += 256) s += a.lpart[i];
  fr[t] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) fr[t] += fr[t + h];
    __syncthreads();
  }
  if (t == 0) a.loss[0] = a.add ? a.loss[0] + fr[0] / a.lscale : fr[0] / a.lscale;
}

// X(m, i) = bf16((x[row][i] - mean[i]) / std[i]), row = idx ? idx[m] : m, and
// the transpose when XT is given; x is float (xf) or double (xd).  A lane
// makes one 16-byte piece; the four lanes of a row read 32 consecutive
// inputs, in the transpose 16 lanes read 16.
__global__ void __launch_bounds__(256) mlp_input_kernel(int n, int nin, const float* __restrict__ xf,
                                                        const double* __restrict__ xd, const int32_t* __restrict__ idx,
                                                        const float* __restrict__ mean, const float* __restrict__ sdev,
                                                        bf16* __restrict__ X, bf16* __restrict__ XT) {
  const int ks = pad32(nin) >> 5, kt = pad32(n) >> 5;
  const size_t np = (size_t)pad32(n) * ks * 4;          // pieces of X, and of XT
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool tr = t >= np;
  if (tr) t -= np;
  if (t >= (tr ? (size_t)pad32(nin) * kt * 4 : np) || (tr && !XT)) return;
  const int lane = (int)(t & 63), steps = tr ? kt : ks;
  const size_t f = t >> 6;
  const int r = (int)(f / steps) * 16 + (lane & 15), k0 = (int)(f % steps) * 32 + 8 * (lane >> 4);
  bf16x8 v;
  // (one type per loop, so that the eight loads are in flight together)
  auto fill = [&](const auto* x) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = tr ? k0 + j : r, i = tr ? r : k0 + j;
      const int mc = min(m, n - 1), ic = min(i, nin - 1);
      const long row = idx ? (long)idx[mc] : (long)mc;
      const float e = ((float)x[row * nin + ic] - mean[ic]) / sdev[ic];
      v[j] = (bf16)(m < n && i < nin ? e : 0.f);
    }
  };
  if (xf)
    fill(xf);
  else
    fill(xd);
  reinterpret_cast<bf16x8*>(tr ? XT : X)[t] = v;
}

// Parameter i's places in the BF16 copies (biases have none).
__device__ __forceinline__ void mlp_put(const MlpShape& S, long i, float v, bf16* __restrict__ wb) {
  int l = 0;
  while (l < S.nl && i >= S.woff[l + 1]) ++l;
  if (i >= S.boff[l]) return;
  const long e = i - S.woff[l];
  const int o = (int)(e / S.din[l]), k = (int)(e - (long)o * S.din[l]);
  const bf16 b = (bf16)v;
  wb[S.wb[l] + frag_at(o, k, pad32(S.din[l]) >> 5)] = b;
  wb[S.wt[l] + frag_at(k, o, pad32(S.dout[l]) >> 5)] = b;
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters; the weights are
// copied to BF16.
__global__ void mlp_adam_kernel(long np, MlpShape S, float* __restrict__ w, const float* __restrict__ g,
                                float* __restrict__ m1, float* __restrict__ m2, bf16* __restrict__ wb, float lr,
                                float b1, float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float v = w[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
  w[i] = v;
  mlp_put(S, i, v, wb);
}

__global__ void mlp_to_bf16_kernel(long np, MlpShape S, const float* __restrict__ w, bf16* __restrict__ wb) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) mlp_put(S, i, w[i], wb);
}

// Per-feature mean and standard deviation of x[n][nf] (FP64 sums); a
// feature with no spread gets a unit scale.
__global__ void mlp_stats_kernel(int n, int nf, const float* __restrict__ x, float* __restrict__ mean,
                                 float* __restrict__ sdev) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nf) return;
  double s = 0.0, s2 = 0.0;
  for (long m = 0; m < n; ++m) {
    const double v = x[m * nf + f];
    s += v;
    s2 += v * v;
  }
  const double mu = s / n;
  const double var = fmax(s2 / n - mu * mu, 0.0);
  const double sd = sqrt(var);
  mean[f] = (float)mu;
  sdev[f] = sd > 1e-6 * fmax(fabs(mu), 1e-30) && sd > 0.0 ? (float)sd : 1.0f;
}

// Node values of a model cube atm[12][nz][ncol]: per quantity the least-
// squares fit x_j = sum_k pinv[j][k] q(z_k) through the hat basis; B_perp and
// its azimuth enter as (B_perp cos 2phi, B_perp sin 2phi), invariant under the
// 180-degree ambiguity of Q and U.  t[col][q * nj + j].
__global__ void mlp_targets_kernel(int ncol, int nz, int nj, const float* __restrict__ atm,
                                   const double* __restrict__ pinv, float* __restrict__ t) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncol) return;
  const long cs = (long)nz * ncol;
  for (int j = 0; j < nj; ++j) {
    double T = 0.0, bx = 0.0, by = 0.0, bz = 0.0, vz = 0.0;
    for (int k = 0; k < nz; ++k) {
      const double p = pinv[j * nz + k];
      const long o = (long)k * ncol + c;
      T += p * atm[0 * cs + o];
      bx += p * atm[5 * cs + o];
      by += p * atm[6 * cs + o];
      bz += p * atm[7 * cs + o];
      vz += p * atm[10 * cs + o];
    }
    const double bp = sqrt(bx * bx + by * by);
    const double ph2 = 2.0 * atan2(by, bx);
    float* o = t + (long)c * MLP_NQ * nj;
    o[0 * nj + j] = (float)T;
    o[1 * nj + j] = (float)bz;
    o[2 * nj + j] = (float)(bp * cos(ph2));
    o[3 * nj + j] = (float)(bp * sin(ph2));
    o[4 * nj + j] = (float)vz;
  }
}

// Network output (standardised, y[R][nout] in LDS) -> node values -> heights
// through the hat basis coefs[k][j]; writes T, Bx, By, Bz, vz of columns
// c0 .. c0 + R - 1 of atm (other rows untouched).  T is kept inside the
// inversion's bounds (2500-18000 K, get_dmodel.f90 LOWLIM/UPPLIM).  All
// threads of the workgroup take part; a lane has one column and every
// (blockDim / R)-th height.  node: R * nout floats of LDS.
__device__ __forceinline__ void mlp_decode(const MlpShape& S, int R, int c0, int ncol, const float* y, float* node,
                                           const float* __restrict__ tmean, const float* __restrict__ tstd,
                                           const double* __restrict__ coefs, float* __restrict__ atm) {
  const int nj = S.nj, no = S.nout;
  for (int e = threadIdx.x; e < R * nj; e += blockDim.x) {
    const int j = e / R, c = e - j * R;
    float q[MLP_NQ];
#pragma unroll
    for (int i = 0; i < MLP_NQ; ++i) q[i] = y[c * no + i * nj + j] * tstd[i * nj + j] + tmean[i * nj + j];
    const float bp = sqrtf(q[2] * q[2] + q[3] * q[3]);
    const float ph = 0.5f * atan2f(q[3], q[2]);
    float* o = node + j * MLP_NQ * R + c;
    o[0] = q[0];
    o[R] = bp * cosf(ph);
    o[2 * R] = bp * sinf(ph);
    o[3 * R] = q[1];
    o[4 * R] = q[4];
  }
  __syncthreads();
  const int c = threadIdx.x % R;
  if (c0 + c >= ncol) return;
  const size_t cs = (size_t)S.nz * ncol;
  // with 64 columns the height is the wave's: the basis comes through scalar loads
  for (int k = R == 64 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64) : (int)threadIdx.x / R; k < S.nz;
       k += blockDim.x / R) {
    double T = 0.0, X = 0.0, Y = 0.0, Z = 0.0, V = 0.0;
    for (int j = 0; j < nj; ++j) {
      const double w = coefs[k * nj + j];
      const float* q = node + j * MLP_NQ * R + c;
      T += w * q[0];
      X += w * q[R];
      Y += w * q[2 * R];
      Z += w * q[3 * R];
      V += w * q[4 * R];
    }
    float* o = atm + (size_t)k * ncol + c0 + c;
    o[0] = (float)fmin(fmax(T, 2500.0), 18000.0);
    o[5 * cs] = (float)X;
    o[6 * cs] = (float)Y;
    o[7 * cs] = (float)Z;
    o[10 * cs] = (float)V;
  }
}

__global__ void __launch_bounds__(256) mlp_decode_kernel(MlpShape S, int ncol, const float* __restrict__ y,
                                                         const float* __restrict__ tmean,
                                                         const float* __restrict__ tstd,
                                                         const double* __restrict__ coefs, float* __restrict__ atm) {
  __shared__ float ys[32 * MLP_NQ * MLP_MAXNODE], node[32 * MLP_NQ * MLP_MAXNODE];
  const int c0 = (int)blockIdx.x * 32, ne = min(32, ncol - c0) * S.nout;
  for (int e = threadIdx.x; e < ne; e += 256) ys[e] = y[(size_t)c0 * S.nout + e];
  for (int e = ne + threadIdx.x; e < 32 * S.nout; e += 256) ys[e] = 0.f;
  __syncthreads();
  mlp_decode(S, 32, c0, ncol, ys, node, tmean, tstd, coefs, atm);
}

// All layers of R = 16 MF rows in one workgroup of eight waves: the
// activations stay in LDS (one buffer: a layer's results wait in the
// accumulators until every wave has read its inputs), the weights come
// from L2 straight into the MFMA operands, two steps ahead, wave w taking
// the output fragments w, w + 8, w + 16 and w + 24 of 16.  Bounded by the weights' way
// into a CU (64 B per cycle: 11 us for the 1.5 MB of 448-512-512-512-20) and by
// the inputs from memory.  Layer by layer, with activations in
// memory, inputs and decoding apart, 16384 rows of 448 took 210 us in kernels, here 53.
// y [n][nout] or, when atm is given, the initial model.
struct InferArgs {
  int n, pitch;
  const float* xf;
  const double* xd;
  const float *mean, *sdev, *tmean, *tstd;
  const float* w;
  const bf16* wb;
  float* y;
  const double* coefs;
  float* atm;
};

constexpr int MLP_INFER_NH = 512;   // widest layer: 8 waves x 4 fragments

template <int MF>
__global__ void __launch_bounds__(512) mlp_infer_kernel(MlpShape S, InferArgs a) {
  extern __shared__ __attribute__((aligned(16))) char mlp_lds[];
  bf16* act = reinterpret_cast<bf16*>(mlp_lds);
  constexpr int R = 16 * MF;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4, pitch = a.pitch;
  const int c0 = (int)blockIdx.x * R;
  // inputs: wave w standardises rows w, w + 8, ..., the loads of all its rows in
  // flight (one at a time, as a choice of the type at each load makes them, 16384 rows
  // took 63 us in all instead of 53)
  auto inputs = [&](const auto* x) {
    const int nin = S.nin, np = pad32(nin);
    constexpr int U = R / 8, V = 2;
    for (int i0 = lane; i0 < np; i0 += 64 * V) {
      auto v = [&](int q, int u) {
        return x[(size_t)min(c0 + wave + 8 * u, a.n - 1) * nin + min(i0 + 64 * q, nin - 1)];
      };
      decltype(v(0, 0)) w[V][U];
      float mu[V], sd[V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        mu[q] = a.mean[min(i0 + 64 * q, nin - 1)];
        sd[q] = a.sdev[min(i0 + 64 * q, nin - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) w[q][u] = v(q, u);
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const int i = i0 + 64 * q;
        if (i >= np) break;
#pragma unroll
        for (int u = 0; u < U; ++u)
          act[(wave + 8 * u) * pitch + i] = (bf16)(i < nin ? ((float)w[q][u] - mu[q]) / sd[q] : 0.f);
      }
    }
  };
  if (a.xf)
    inputs(a.xf);
  else
    inputs(a.xd);
  __syncthreads();
  for (int l = 0; l <= S.nl; ++l) {
    const int N = S.dout[l], nfr = pad32(N) >> 4, ks = pad32(S.din[l]) >> 5;
    const bf16x8* W = reinterpret_cast<const bf16x8*>(a.wb + S.wb[l]) + (size_t)wave * ks * 64 + lane;
    f32x4 acc[4][MF];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < MF; ++i) acc[j][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int nf = wave < nfr ? (nfr - wave + 7) >> 3 : 0;   // this wave's fragments
    if (nf > 0) {
      bf16x8 w[2][4];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < nf) w[p][j] = W[((size_t)(8 * j) * ks + min(p, ks - 1)) * 64];
      for (int s = 0; s < ks; s += 2) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          if (s + p >= ks) break;
          bf16x8 x[MF];
#pragma unroll
          for (int i = 0; i < MF; ++i)
            x[i] = *reinterpret_cast<const bf16x8*>(act + (16 * i + lr) * pitch + 32 * (s + p) + 8 * lg);
          const int t = min(s + p + 2, ks - 1);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (j >= nf) break;
#pragma unroll
            for (int i = 0; i < MF; ++i)
              acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[p][j], x[i], acc[j][i], 0, 0, 0);
            w[p][j] = W[((size_t)(8 * j) * ks + t) * 64];
          }
        }
      }
    }
    __syncthreads();
    const float* bias = a.w + S.boff[l];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j >= nf) break;
      const int n = 16 * (wave + 8 * j) + 4 * lg;
      float b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) b[q] = n + q < N ? bias[n + q] : 0.f;
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int m = 16 * i + lr;
        if (l == S.nl) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (n + q < N) reinterpret_cast<float*>(mlp_lds)[m * N + n + q] = acc[j][i][q] + b[q];
        } else {
          bf16x4 o;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float v = acc[j][i][q] + b[q];
            o[q] = (bf16)(n + q < N && v > 0.f ? v : 0.f);
          }
          *reinterpret_cast<bf16x4*>(act + m * pitch + n) = o;
        }
      }
    }
    __syncthreads();
  }
  const float* ys = reinterpret_cast<const float*>(mlp_lds);
  if (a.atm) {
    mlp_decode(S, R, c0, a.n, ys, reinterpret_cast<float*>(mlp_lds) + R * S.nout, a.tmean, a.tstd, a.coefs, a.atm);
    return;
  }
  for (int e = threadIdx.x; e < min(R, a.n - c0) * S.nout; e += 512) a.y[(size_t)c0 * S.nout + e] = ys[e];
}

}  // namespace fz
