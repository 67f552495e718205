// The learned subgrid closure (no counterpart in the reference):
//
//   k_filter     spectral box in x, z and a y top-hat: fine spectra -> coarse
//   k_czinv      z inverse transform of coarse fields, d/dx and d/dz fused
//                into the load (FP64)
//   k_cxc2r      x inverse real transform to physical values (FP64)
//   k_samples    (9 gradients, 6 stresses) per coarse grid point
//   k_mlp_train  forward + backward of the 9-64-64-6 tanh network for 128
//                samples per block on the matrix cores (bfloat16 operands,
//                FP32 accumulation), per-block partial gradients
//   k_adam       ordered reduction of the partial gradients and the Adam step
//   k_mlp_infer  the network on samples or on the physical gradient fields
//   k_cxr2c      x forward real transform of the modelled stresses (FP64),
//                then the solver's own z forward transform and ghost rows
//   k_add_stress P += tau-hat on the live state's products
//
// Matrix-core layout (v_mfma_f32_16x16x32_bf16, one wavefront): lane l holds
// A[l%16][8(l/16)+v] and B[8(l/16)+v][l%16], v < 8, and D[4(l/16)+v][l%16],
// v < 4.  Samples run along the 16 columns; a layer's D fragments of two
// consecutive 16-row tiles are the B operand of the next layer once the K
// slots are renamed (kfeat): slot v of lane group q is row 4q+v of the first
// tile for v < 4 and of the second for v >= 4, and the weights are staged in
// LDS in the same order.  Weight gradients contract over samples, so the
// activations and errors are also staged as [feature][sample] in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "hst_cx.h"
#include "hst_fft_dev.h"
#include "hst_internal.h"
#include "../../include/hst_closure.h"

namespace hst {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f4;

constexpr int NP = HST_MLP_NPARAM;
constexpr int NPP = NP + 2;  // row of the partial-gradient buffer: the parameters, the loss
constexpr int OW1 = 0, OB1 = 64 * 9, OW2 = OB1 + 64, OB2 = OW2 + 64 * 64, OW3 = OB2 + 64, OB3 = OW3 + 6 * 64;
static_assert(OB3 + 6 == NP, "parameter layout");
constexpr int SPB = 128;        // samples per training block
constexpr int SP = 72;          // LDS row stride (bf16) of the [feature][64 samples] staging
constexpr int MAX_PART = 2048;  // partial-gradient rows: at most SPB * MAX_PART samples per launch

// ================================================================== transforms

struct FilterArgs {
  const void *src[9];
  double2 *dst[9];
};

// One lane per coarse column; coarse row k = sum_t w[8k+t] * fine row j0[k]+t.
template <typename RS>
__global__ void __launch_bounds__(256)
    k_filter(FilterArgs a, int ncol_f, int NZm_f, int nz_f, Dims Dc, const int *__restrict__ j0,
             const double *__restrict__ w) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= Dc.ncol) return;
  const int ixc = c / Dc.NZm, izc = c % Dc.NZm - Dc.nz;
  const size_t fcol = (size_t)ixc * NZm_f + izc + nz_f;
  const Cx<RS> *src = (const Cx<RS> *)a.src[blockIdx.y];
  double2 *dst = a.dst[blockIdx.y];
  for (int k = 0; k < Dc.ny; k++) {
    double sx = 0.0, sy = 0.0;
    const int r0 = j0[k] + 2;
    for (int t = 0; t < 8; t++) {
      const double wt = w[k * 8 + t];
      if (wt == 0.0) continue;
      const Cx<RS> v = src[(size_t)(r0 + t) * ncol_f + fcol];
      sx += wt * (double)v.x;
      sy += wt * (double)v.y;
    }
    dst[(size_t)(k + 2) * Dc.ncol + c] = make_double2(sx, sy);
  }
}

struct ZSrc {
  const double2 *p[18];
  int op[18];  // 0 the field, 1 d/dx, 2 d/dz
};

constexpr int ZG = 8;  // z lines (x modes) per block
constexpr int XG = 8;  // x lines (z points) per block

// z inverse transform of the interior rows of nf coarse fields into
// Hc[f][row][zp][ix] (ix < NXp), the padding and the derivative factor fused
// into the load.
template <int NZD>
__global__ void __launch_bounds__(ZG * fft_threads(NZD))
    k_czinv(ZSrc s, Cx<double> *__restrict__ Hc, Dims D, const Cx<double> *__restrict__ tw) {
  constexpr int T = fft_threads(NZD), LS = NZD + 1;
  __shared__ Cx<double> lds[ZG * LS];
  __shared__ Cx<double> twl[NZD];
  for (int k = threadIdx.x; k < NZD; k += blockDim.x) twl[k] = tw[k];
  const int f = blockIdx.z, rowc = blockIdx.y, ix0 = blockIdx.x * ZG, nz = D.nz;
  const double2 *src = s.p[f] + (size_t)(rowc + 2) * D.ncol;
  const int op = s.op[f];
  for (int e = threadIdx.x; e < ZG * NZD; e += blockDim.x) {
    const int j = e / NZD, k = e % NZD, ix = ix0 + j;
    const int iz = k <= nz ? k : (k >= NZD - nz ? k - NZD : INT_MAX);
    Cx<double> v{0.0, 0.0};
    if (ix < D.NXm && iz != INT_MAX) {
      const double2 a = src[(size_t)ix * D.NZm + iz + nz];
      v = Cx<double>{a.x, a.y};
      if (op) {
        const double kk = op == 1 ? D.alfa0 * ix : D.beta0 * iz;
        v = Cx<double>{-kk * a.y, kk * a.x};
      }
    }
    lds[j * LS + k] = v;
  }
  __syncthreads();
  const int g = threadIdx.x / T, t = threadIdx.x % T;
  fft_line<double, NZD, T, +1>(lds + g * LS, t, twl);
  Cx<double> *dst = Hc + ((size_t)f * D.ny + rowc) * NZD * D.NXp;
  for (int e = threadIdx.x; e < ZG * NZD; e += blockDim.x) {
    const int j = e % ZG, zp = e / ZG;
    if (ix0 + j < D.NXm) dst[(size_t)zp * D.NXp + ix0 + j] = lds[j * LS + zp];
  }
}

// x inverse real transform of one (field, row, z point) line per T threads:
// phys[f][row][zp][x], x < 2M.  The half-length complex form of the
// reference's c2r, the imaginary part of the kx = 0 bin ignored.
template <int M>
__global__ void __launch_bounds__(XG * fft_threads(M))
    k_cxc2r(const Cx<double> *__restrict__ Hc, double *__restrict__ phys, Dims D,
            const Cx<double> *__restrict__ twx, const Cx<double> *__restrict__ twh) {
  constexpr int T = fft_threads(M), LS = M + 1;
  __shared__ Cx<double> lin[XG * LS], wk[XG * LS];
  const int f = blockIdx.z, rowc = blockIdx.y, g = threadIdx.x / T, t = threadIdx.x % T;
  const int zp = blockIdx.x * XG + g, nx = D.nx;
  const Cx<double> *src = Hc + (((size_t)f * D.ny + rowc) * D.nzd + zp) * D.NXp;
  Cx<double> *wl = wk + g * LS, *vl = lin + g * LS;
  for (int k = t; k <= nx; k += T) wl[k] = src[k];
  __syncthreads();
  for (int k = t; k < M; k += T) {
    Cx<double> a = (k <= nx) ? wl[k] : Cx<double>{0.0, 0.0};
    if (k == 0) a.y = 0.0;
    const int j = M - k;
    const Cx<double> b = (k > 0 && j <= nx) ? conj(wl[j]) : Cx<double>{0.0, 0.0};
    const Cx<double> e = conj(twh[k]);
    vl[k] = (a + b) + mul_i(e * (a - b));
  }
  __syncthreads();
  fft_line<double, M, T, +1>(vl, t, twx);
  double *out = phys + (((size_t)f * D.ny + rowc) * D.nzd + zp) * (2 * M);
  for (int m = t; m < M; m += T) {
    out[2 * m] = vl[m].x;
    out[2 * m + 1] = vl[m].y;
  }
}

// x forward real transform (times factor) of six physical fields into the
// product buffer in the tiled layout the z forward transform reads (hoff).
template <int M>
__global__ void __launch_bounds__(XG * fft_threads(M))
    k_cxr2c(const double *__restrict__ phys, Cx<double> *__restrict__ Hp, Dims D,
            const Cx<double> *__restrict__ twx, const Cx<double> *__restrict__ twh) {
  constexpr int T = fft_threads(M), LS = M + 1;
  __shared__ Cx<double> lin[XG * LS];
  const int p = blockIdx.z, rowc = blockIdx.y, g = threadIdx.x / T, t = threadIdx.x % T;
  const int zp = blockIdx.x * XG + g, nx = D.nx;
  const double *in = phys + (((size_t)p * D.ny + rowc) * D.nzd + zp) * (2 * M);
  Cx<double> *vl = lin + g * LS;
  for (int m = t; m < M; m += T) vl[m] = Cx<double>{in[2 * m] * D.factor, in[2 * m + 1] * D.factor};
  __syncthreads();
  fft_line<double, M, T, -1>(vl, t, twx);
  Cx<double> *dst = Hp + ((size_t)p * D.ny + rowc) * D.nzd * D.NXp;
  for (int k = t; k <= nx; k += T) {
    const Cx<double> Z = vl[k], Zc = conj(vl[(M - k) % M]);
    const Cx<double> e = twh[k];
    const Cx<double> s = (Z + Zc) * 0.5, d = (Z - Zc) * 0.5;
    dst[hoff<double>(D.nzd, D.NXp, zp, k)] = s - mul_i(e * d);
  }
}

// (gradients, stresses) of every point: phys fields 0..8 the gradients
// (i-major), 9..11 u v w, 12..17 the filtered products.
__global__ void __launch_bounds__(256)
    k_samples(const double *__restrict__ phys, size_t fs, int64_t npts, float *__restrict__ X,
              float *__restrict__ Y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npts) return;
#pragma unroll
  for (int k = 0; k < 9; k++) X[i * 9 + k] = (float)phys[k * fs + i];
  const double u = phys[9 * fs + i], v = phys[10 * fs + i], w = phys[11 * fs + i];
  const double uu[6] = {u * u, v * v, w * w, u * v, v * w, u * w};
#pragma unroll
  for (int p = 0; p < 6; p++) Y[i * 6 + p] = (float)(phys[(12 + p) * fs + i] - uu[p]);
}

// P[p] += T[p] over all rows of the six products
template <typename R>
__global__ void __launch_bounds__(256) k_add_stress(Cx<R> *__restrict__ P, const double2 *__restrict__ T, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double2 t = T[i];
  Cx<R> p = P[i];
  p.x = (R)((double)p.x + t.x);
  p.y = (R)((double)p.y + t.y);
  P[i] = p;
}

// ================================================================== the network

struct Norm {
  float mx[9], rx[9], my[6], ry[6], sy[6];
};

__device__ __forceinline__ f4 mfma(const bf8 &a, const bf8 &b, const f4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// feature of K slot v of lane group q in K block kb, when the B operand is
// formed from the D fragments of output tiles 2kb and 2kb+1
__device__ __forceinline__ int kfeat(int kb, int q, int v) { return 32 * kb + (v < 4 ? 4 * q + v : 12 + 4 * q + v); }

// The weights as the instruction's operands: those of the forward pass, and
// behind them (training) the transposed ones of the backward pass.  One image
// of them per context is kept in global memory beside the FP32 parameters, so
// that a block copies it to LDS in whole cache lines (gathered from the
// parameters by every block it took 5 of the training kernel's 29 us); k_pack
// writes it for given parameters and k_adam with each update.
struct WFwd {
  bf8 A1[4][64];     // W1[16m+i][8q+v], K padded 9 -> 32
  bf8 A2[4][2][64];  // W2[16m+i][kfeat]
  bf8 A3[2][64];     // W3[i][kfeat], rows 6..15 zero
  float b1[64], b2[64], b3[16];
};
struct WBwd {
  bf8 B3[4][64];     // W3[4q+v][16m+i] (v < 4): W3^T against the output errors
  bf8 B2[4][2][64];  // W2[kfeat][16m+i]: W2^T
};
struct WImage {
  WFwd f;
  WBwd b;
};

// parameter p (of value x) into its places of the image
__device__ __forceinline__ void pack_param(int p, float x, WImage &w) {
  const __bf16 h = (__bf16)x;
  // K block, lane group and slot of feature f (the inverse of kfeat)
  auto slot = [](int f, int &kb, int &q, int &v) {
    const int g = f & 31;
    kb = f >> 5;
    q = (g & 15) >> 2;
    v = (g & 3) + (g < 16 ? 0 : 4);
  };
  int kb, q, v;
  if (p < OB1) {
    const int r = p / 9, k = p - r * 9;
    w.f.A1[r >> 4][(r & 15) + 16 * (k >> 3)][k & 7] = h;
  } else if (p < OW2) {
    w.f.b1[p - OB1] = x;
  } else if (p < OB2) {
    const int r = (p - OW2) >> 6, f = (p - OW2) & 63;
    slot(f, kb, q, v);
    w.f.A2[r >> 4][kb][(r & 15) + 16 * q][v] = h;
    slot(r, kb, q, v);
    w.b.B2[f >> 4][kb][(f & 15) + 16 * q][v] = h;
  } else if (p < OW3) {
    w.f.b2[p - OB2] = x;
  } else if (p < OB3) {
    const int o = (p - OW3) >> 6, f = (p - OW3) & 63;
    slot(f, kb, q, v);
    w.f.A3[kb][o + 16 * q][v] = h;
    w.b.B3[f >> 4][(f & 15) + 16 * (o >> 2)][o & 3] = h;
  } else {
    w.f.b3[p - OB3] = x;
  }
}

// The image of the parameters; one block: the padding zero, then the entries.
__global__ void __launch_bounds__(1024) k_pack(const float *__restrict__ par, WImage *__restrict__ img) {
  for (int k = threadIdx.x; k < (int)(sizeof(WImage) / 4); k += 1024) ((float *)img)[k] = 0.0f;
  __syncthreads();
  for (int p = threadIdx.x; p < NP; p += 1024) pack_param(p, par[p], *img);
}

// a part of the image to LDS by the NT threads of a block, every load before the first store
template <int NT, class T>
__device__ __forceinline__ void stage_weights(const T &g, T &lds) {
  typedef __attribute__((__vector_size__(16))) float v4;
  constexpr int N = sizeof(T) / 16, PER = (N + NT - 1) / NT;
  static_assert(sizeof(T) % 16 == 0, "whole vectors");
  const v4 *src = (const v4 *)&g;
  v4 t[PER];
#pragma unroll
  for (int u = 0; u < PER; u++) t[u] = src[min(u * NT + (int)threadIdx.x, N - 1)];
#pragma unroll
  for (int u = 0; u < PER; u++)
    if (u * NT + (int)threadIdx.x < N) ((v4 *)&lds)[u * NT + threadIdx.x] = t[u];
}

// B operands of the next layer from the D fragments of four 16-row tiles
__device__ __forceinline__ void to_operands(const f4 h[4], bf8 B[2]) {
#pragma unroll
  for (int kb = 0; kb < 2; kb++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      B[kb][v] = (__bf16)h[2 * kb][v];
      B[kb][4 + v] = (__bf16)h[2 * kb + 1][v];
    }
}

// tanh x without a branch: below one, x - x^3 (45045 + 2772 x^2 + 27 x^4) / D,
// D = 135135 + 62370 x^2 + 3150 x^4 + 28 x^6 (the seventh convergent of Lambert's
// continued fraction, 7e-11 off at one, written as a correction to x); above,
// +-1 -+ 2 / (exp(2 |x|) + 1), |x| cut at 10 where the correction is 4e-9.  One
// reciprocal serves both, and since the correction is at most 0.24 of what it corrects
// (31 % of the result, at one) its rounding hardly shows: over 4 M arguments of
// 1e-8 .. 12 the largest error against 64 bits is 1.33 units of the last place and
// the rms 0.238 (tanhf: 1.35 and 0.240).  A wavefront evaluates 32 a tile, most of
// the network's instructions: k_mlp_infer 116 -> 90 us on 798,720 points.
__device__ __forceinline__ float tanh_f(float x) {
  const float a = fabsf(x), c = a > 10.0f ? 10.0f : a, x2 = x * x;
  const bool small = a < 1.0f;
  const float e = __builtin_amdgcn_exp2f(c * 2.88539008f);  // 2 / ln 2
  const float p = -x * x2 * fmaf(x2, fmaf(x2, 27.0f, 2772.0f), 45045.0f);
  const float q = fmaf(x2, fmaf(x2, fmaf(x2, 28.0f, 3150.0f), 62370.0f), 135135.0f);
  const float num = small ? p : copysignf(2.0f, -x), den = small ? q : e + 1.0f;
  return fmaf(num, __builtin_amdgcn_rcpf(den), small ? x : copysignf(1.0f, x));
}

// Forward pass of one 16-sample tile: x the input operand; h1, h2 the hidden
// activations (FP32 D fragments), y the outputs (rows 4q+v, valid below 6).
// The biases start the accumulators.
__device__ __forceinline__ void forward(const WFwd &W, int l, const bf8 &x, f4 h1[4], f4 h2[4], f4 &y) {
  const int q = l >> 4;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const f4 z = mfma(W.A1[m][l], x, *(const f4 *)(W.b1 + 16 * m + 4 * q));
#pragma unroll
    for (int v = 0; v < 4; v++) h1[m][v] = tanh_f(z[v]);
  }
  bf8 B[2];
  to_operands(h1, B);
#pragma unroll
  for (int m = 0; m < 4; m++) {
    f4 z = mfma(W.A2[m][0][l], B[0], *(const f4 *)(W.b2 + 16 * m + 4 * q));
    z = mfma(W.A2[m][1][l], B[1], z);
#pragma unroll
    for (int v = 0; v < 4; v++) h2[m][v] = tanh_f(z[v]);
  }
  to_operands(h2, B);
  y = mfma(W.A3[0][l], B[0], *(const f4 *)(W.b3 + 4 * q));
  y = mfma(W.A3[1][l], B[1], y);
}

// The standardisation of a lane's inputs: features 8q .. 8q+7 in lane group q,
// the ninth for those past it (whose operand entries are zero).
struct LaneNorm {
  float m[8], r[8];
  __device__ __forceinline__ LaneNorm(const Norm &nm, int q) {
#pragma unroll
    for (int v = 0; v < 8; v++) {
      const int k = min(8 * q + v, 8);
      m[v] = nm.mx[k];
      r[v] = nm.rx[k];
    }
  }
  // the input operand of the sample whose features raw holds
  template <typename In>
  __device__ __forceinline__ bf8 operand(int q, bool valid, const In (&raw)[8]) const {
    bf8 x;
#pragma unroll
    for (int v = 0; v < 8; v++)
      x[v] = (__bf16)((valid && 8 * q + v < 9) ? ((float)raw[v] - m[v]) * r[v] : 0.0f);
    return x;
  }
};

struct TrainArgs {
  const float *X, *Y;
  int64_t n;              // samples of this launch
  int64_t base;           // first position
  int64_t mul, add, mod;  // sample index = (mul * (base + b) + add) % mod
  float scale;            // 2 / (samples of the loss * 6)
};

// GRAD: forward, backward and the per-block partial gradients (part[blk][NPP],
// the last two entries the sum of squared errors); otherwise the sum of
// squared errors alone into lossp[blk].
//
// A block of four wavefronts takes SPB samples in passes of 64.  In a pass every
// wavefront runs forward and backward of a 16-sample tile of its own and stages
// activations and errors [feature][sample]; then it forms the 16 rows of the
// weight gradients that are its own over all 64 samples, so no gradient is
// summed across wavefronts and a wavefront holds a quarter of them.  The kernel
// is bound by the latency of this chain (tanh, LDS, barriers) and not by the
// matrix cores: a batch of 65,536 on one wavefront per 128 samples left half of
// the SIMDs without work, 65 -> 32 us (25.5 with
// tanh_f and the operand image).
constexpr int TNT = 256, TPS = 64;  // threads; samples per pass
static_assert(SPB % TPS == 0 && TPS == TNT / 4, "a tile of 16 samples per wavefront and pass");

template <bool GRAD>
__global__ void __launch_bounds__(TNT)
    k_mlp_train(const WImage *__restrict__ img, Norm nm, TrainArgs ta, float *__restrict__ part,
                double *__restrict__ lossp) {
  constexpr int NPASS = SPB / TPS, ROWS = GRAD ? 1 : 0;  // (the arrays of the backward pass are its own)
  __shared__ WFwd W;
  __shared__ WBwd WB[1];
  __shared__ __attribute__((aligned(16))) __bf16 Xs[ROWS * 16 + 1][SP], H1s[ROWS * 64 + 1][SP],
      H2s[ROWS * 64 + 1][SP], DYs[ROWS * 16 + 1][SP], DZ2s[ROWS * 64 + 1][SP], DZ1s[ROWS * 64 + 1][SP];
  __shared__ float red[4][2 * 64 + 8];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, j = l & 15, q = l >> 4;
  // the samples of every pass: index, inputs and targets, in flight while the weights are staged
  bool valid[NPASS];
  float xr[NPASS][8], yr[NPASS][4];
#pragma unroll
  for (int p = 0; p < NPASS; p++) {
    const int64_t b = (int64_t)blockIdx.x * SPB + p * TPS + w * 16 + j;
    valid[p] = b < ta.n;
    const int64_t idx = (ta.mul * (ta.base + (valid[p] ? b : 0)) + ta.add) % ta.mod;
#pragma unroll
    for (int v = 0; v < 8; v++) xr[p][v] = ta.X[idx * 9 + min(8 * q + v, 8)];
#pragma unroll
    for (int v = 0; v < 4; v++) yr[p][v] = ta.Y[idx * 6 + min(4 * q + v, 5)];
  }
  const LaneNorm ln(nm, q);
  float my[4], ry[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    my[v] = nm.my[min(4 * q + v, 5)];
    ry[v] = nm.ry[min(4 * q + v, 5)];
  }
  stage_weights<TNT>(img->f, W);
  if constexpr (GRAD) {
    stage_weights<TNT>(img->b, WB[0]);
    for (int r = 9 + w; r < 16; r += 4)
      if (l < TPS) Xs[r][l] = (__bf16)0.0f;
  }
  __syncthreads();
  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  f4 gW2[4], gW1 = zero, gW3 = zero;
  float gb1[4][4], gb2[4][4], gb3[4];
#pragma unroll
  for (int a = 0; a < 4; a++) {
    gW2[a] = zero;
    gb3[a] = 0.f;
#pragma unroll
    for (int v = 0; v < 4; v++) { gb1[a][v] = 0.f; gb2[a][v] = 0.f; }
  }
  float lsum = 0.0f;
#pragma unroll
  for (int p = 0; p < NPASS; p++) {
    const bf8 x = ln.operand(q, valid[p], xr[p]);
    f4 h1[4], h2[4], y;
    forward(W, l, x, h1, h2, y);
    f4 dy = zero;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      if (valid[p] && 4 * q + v < 6) {
        const float e = y[v] - (yr[p][v] - my[v]) * ry[v];
        lsum += e * e;
        dy[v] = ta.scale * e;
      }
    }
    if constexpr (GRAD) {
      bf8 Bd;
#pragma unroll
      for (int v = 0; v < 4; v++) { Bd[v] = (__bf16)dy[v]; Bd[4 + v] = (__bf16)0.0f; }
      f4 dz2[4], dz1[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const f4 a = mfma(WB[0].B3[m][l], Bd, zero);
#pragma unroll
        for (int v = 0; v < 4; v++) dz2[m][v] = a[v] * (1.0f - h2[m][v] * h2[m][v]);
      }
      bf8 Bz[2];
      to_operands(dz2, Bz);
#pragma unroll
      for (int m = 0; m < 4; m++) {
        f4 a = mfma(WB[0].B2[m][0][l], Bz[0], zero);
        a = mfma(WB[0].B2[m][1][l], Bz[1], a);
#pragma unroll
        for (int v = 0; v < 4; v++) dz1[m][v] = a[v] * (1.0f - h1[m][v] * h1[m][v]);
      }
      // stage [feature][sample] for the weight gradients; bias gradients in FP32
      const int col = w * 16 + j;
#pragma unroll
      for (int v = 0; v < 8; v++)
        if (8 * q + v < 9) Xs[8 * q + v][col] = x[v];
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = 16 * m + 4 * q + v;
          H1s[r][col] = (__bf16)h1[m][v];
          H2s[r][col] = (__bf16)h2[m][v];
          DZ2s[r][col] = (__bf16)dz2[m][v];
          DZ1s[r][col] = (__bf16)dz1[m][v];
          gb1[m][v] += dz1[m][v];
          gb2[m][v] += dz2[m][v];
        }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        DYs[4 * q + v][col] = Bd[v];
        gb3[v] += dy[v];
      }
      __syncthreads();
      // K = 32 samples at a time: the wavefront's A rows from one array, B columns from another
#pragma unroll
      for (int k = 0; k < TPS / 32; k++) {
        auto rd = [&](const __bf16 *row) { return *(const bf8 *)(row + 32 * k + 8 * q); };
        const bf8 dz2r = rd(DZ2s[16 * w + j]);
#pragma unroll
        for (int mk = 0; mk < 4; mk++) gW2[mk] = mfma(dz2r, rd(H1s[16 * mk + j]), gW2[mk]);
        gW1 = mfma(rd(DZ1s[16 * w + j]), rd(Xs[j]), gW1);
        gW3 = mfma(rd(DYs[j]), rd(H2s[16 * w + j]), gW3);
      }
      if (p + 1 < NPASS) __syncthreads();
    }
  }
  // sums over the wavefront, then over the four wavefronts in order
  for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
  if (l == 0) red[w][134] = lsum;
  if constexpr (!GRAD) {
    __syncthreads();
    if (threadIdx.x == 0)
      lossp[blockIdx.x] = (double)red[0][134] + (double)red[1][134] + (double)red[2][134] + (double)red[3][134];
    return;
  }
  float *pr = part + (size_t)blockIdx.x * NPP;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int r = 16 * w + 4 * q + v;
#pragma unroll
    for (int mk = 0; mk < 4; mk++) pr[OW2 + r * 64 + 16 * mk + j] = gW2[mk][v];
    if (j < 9) pr[OW1 + r * 9 + j] = gW1[v];
    if (4 * q + v < 6) pr[OW3 + (4 * q + v) * 64 + 16 * w + j] = gW3[v];
  }
  // bias gradients: the 16 sample columns of the wavefront, then the wavefronts
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int v = 0; v < 4; v++)
      for (int o = 1; o < 16; o <<= 1) {
        gb1[m][v] += __shfl_xor(gb1[m][v], o);
        gb2[m][v] += __shfl_xor(gb2[m][v], o);
      }
#pragma unroll
  for (int v = 0; v < 4; v++)
    for (int o = 1; o < 16; o <<= 1) gb3[v] += __shfl_xor(gb3[v], o);
  if (j == 0) {
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        red[w][16 * m + 4 * q + v] = gb1[m][v];
        red[w][64 + 16 * m + 4 * q + v] = gb2[m][v];
      }
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (4 * q + v < 6) red[w][128 + 4 * q + v] = gb3[v];
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < 135) {
    const float g = red[0][t] + red[1][t] + red[2][t] + red[3][t];
    pr[t < 64 ? OB1 + t : (t < 128 ? OB2 + t - 64 : (t < 134 ? OB3 + t - 128 : NP))] = g;
  }
}

// Ordered sum of nblk partial rows per parameter, then (update) the Adam step
// or (!update) the gradient into grad; slot NP: the summed squared error.
// A block holds 64 parameters (one per lane of a wavefront, so every row read
// is 256 contiguous bytes) and AR row groups (one per wavefront); the group
// sums are added in a fixed order, so the result does not depend on timing.
constexpr int AR = 8;
__global__ void __launch_bounds__(64 * AR)
    k_adam(float *__restrict__ par, float *__restrict__ m1, float *__restrict__ m2, const float *__restrict__ part,
           int nblk, int update, float lr, float c1, float c2, float *__restrict__ grad, double *__restrict__ sse,
           WImage *__restrict__ img) {
  __shared__ double red[AR][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + l;
  double g = 0.0;
  if (p <= NP) {
#pragma unroll 8
    for (int b = w; b < nblk; b += AR) g += (double)part[(size_t)b * NPP + p];
  }
  red[w][l] = g;
  __syncthreads();
  if (w != 0 || p > NP) return;
  g = 0.0;
  for (int k = 0; k < AR; k++) g += red[k][l];
  if (p == NP) {
    *sse = g;
    return;
  }
  if (!update) {
    grad[p] = (float)g;
    return;
  }
  const float gf = (float)g;
  const float a = 0.9f * m1[p] + 0.1f * gf, s = 0.999f * m2[p] + 0.001f * gf * gf;
  m1[p] = a;
  m2[p] = s;
  const float x = par[p] - lr * (a * c1) / (sqrtf(s * c2) + 1e-8f);
  par[p] = x;
  pack_param(p, x, *img);
}

struct InferIO {
  const float *X;      // mode 0: x[n][9]
  float *Y;            // mode 0: y[n][6]
  const double *gin;   // mode 1: 9 gradient fields of stride fs
  double *tout;        // mode 1: 6 stress fields of stride fs
  size_t fs;
  int64_t n;
  int mode;
};

// One 16-sample tile per wavefront at a time, the next tile's inputs loaded
// while this one is computed.  The weights stay in registers, which leaves two
// wavefronts a SIMD: two blocks of four a CU (three blocks, without: 5 % slower).
// The vector ALU bounds it (about 900 instructions a tile, two thirds of them
// tanh): 798,720 points take 82 us against 405 with one wavefront a block, 32
// tiles each, tanhf and the weights gathered by every block.
constexpr int INFER_NT = 256, INFER_BLOCKS = 256 * 2;

template <int MODE>
__global__ void __launch_bounds__(INFER_NT) k_mlp_infer(const WImage *__restrict__ img, Norm nm, InferIO io) {
  __shared__ WFwd W;
  const int l = threadIdx.x & 63, j = l & 15, q = l >> 4;
  stage_weights<INFER_NT>(img->f, W);
  __syncthreads();
  const int64_t ntile = (io.n + 15) / 16, step = (int64_t)gridDim.x * (INFER_NT / 64);
  typedef typename std::conditional<MODE == 0, float, double>::type In;
  const LaneNorm ln(nm, q);
  float my[4], sy[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    my[v] = nm.my[min(4 * q + v, 5)];
    sy[v] = nm.sy[min(4 * q + v, 5)];
  }
  // a tile's inputs, without a branch (past the last feature or sample: the last again)
  auto fetch = [&](int64_t tile, In (&raw)[8]) {
    const int64_t s = min(tile * 16 + j, io.n - 1);
#pragma unroll
    for (int v = 0; v < 8; v++) {
      const int k = min(8 * q + v, 8);
      if constexpr (MODE == 0) raw[v] = io.X[s * 9 + k];
      else raw[v] = io.gin[(size_t)k * io.fs + s];
    }
  };
  int64_t tile = (int64_t)blockIdx.x * (INFER_NT / 64) + (threadIdx.x >> 6);
  if (tile >= ntile) return;
  In cur[8], nxt[8];
  fetch(tile, cur);
  for (; tile < ntile; tile += step) {
    fetch(min(tile + step, ntile - 1), nxt);
    const int64_t s = tile * 16 + j;
    const bool valid = s < io.n;
    const bf8 x = ln.operand(q, valid, cur);
    f4 h1[4], h2[4], y;
    forward(W, l, x, h1, h2, y);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int o = 4 * q + v;
      if (!valid || o >= 6) continue;
      const float t = y[v] * sy[v] + my[v];
      if constexpr (MODE == 0) io.Y[s * 6 + o] = t;
      else io.tout[(size_t)o * io.fs + s] = (double)t;
    }
#pragma unroll
    for (int v = 0; v < 8; v++) cur[v] = nxt[v];
  }
}

static void run_infer(const WImage *img, const Norm &nm, const InferIO &io, hipStream_t st) {
  const int64_t tiles = (io.n + 15) / 16, per = INFER_NT / 64;
  dim3 grid((unsigned)std::min<int64_t>((tiles + per - 1) / per, INFER_BLOCKS));
  if (io.mode == 0) hipLaunchKernelGGL(k_mlp_infer<0>, grid, dim3(INFER_NT), 0, st, img, nm, io);
  else hipLaunchKernelGGL(k_mlp_infer<1>, grid, dim3(INFER_NT), 0, st, img, nm, io);
}

// sums (pass 0) or sums of squared deviations (pass 1) of the 15 columns, per block
__global__ void __launch_bounds__(256)
    k_moments(const float *__restrict__ X, const float *__restrict__ Y, int64_t n, const double *__restrict__ mean,
              int pass, double *__restrict__ part) {
  __shared__ double red[15][4];
  double acc[15];
  for (int k = 0; k < 15; k++) acc[k] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    for (int k = 0; k < 15; k++) {
      double v = k < 9 ? (double)X[i * 9 + k] : (double)Y[i * 6 + k - 9];
      if (pass) {
        v -= mean[k];
        v *= v;
      }
      acc[k] += v;
    }
  }
  for (int k = 0; k < 15; k++) {
    double v = acc[k];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x < 15) {
    const int k = threadIdx.x;
    part[(size_t)blockIdx.x * 15 + k] = red[k][0] + red[k][1] + red[k][2] + red[k][3];
  }
}

// ================================================================== host side

template <int NZD>
static void run_czinv(const Dims &D, const ZSrc &s, int nf, Cx<double> *Hc, const Cx<double> *tw, hipStream_t st) {
  dim3 grid((D.NXm + ZG - 1) / ZG, D.ny, nf);
  hipLaunchKernelGGL(k_czinv<NZD>, grid, dim3(ZG * fft_threads(NZD)), 0, st, s, Hc, D, tw);
}
template <int M>
static void run_cxc2r(const Dims &D, int nf, const Cx<double> *Hc, double *phys, const Cx<double> *twx,
                      const Cx<double> *twh, hipStream_t st) {
  dim3 grid(D.nzd / XG, D.ny, nf);
  hipLaunchKernelGGL(k_cxc2r<M>, grid, dim3(XG * fft_threads(M)), 0, st, Hc, phys, D, twx, twh);
}
template <int M>
static void run_cxr2c(const Dims &D, const double *phys, Cx<double> *Hp, const Cx<double> *twx,
                      const Cx<double> *twh, hipStream_t st) {
  dim3 grid(D.nzd / XG, D.ny, 6);
  hipLaunchKernelGGL(k_cxr2c<M>, grid, dim3(XG * fft_threads(M)), 0, st, phys, Hp, D, twx, twh);
}

#define CLOSURE_Z_SIZES(X) X(48) X(64) X(96) X(128) X(192)
#define CLOSURE_X_SIZES(X) X(32) X(48) X(64) X(96) X(128)

static bool closure_size_ok(const Dims &D) {
  bool z = false, x = false;
#define ZC(n) z = z || D.nzd == n;
#define XC(n) x = x || D.nxd == n;
  CLOSURE_Z_SIZES(ZC)
  CLOSURE_X_SIZES(XC)
#undef ZC
#undef XC
  return z && x && D.nzd % XG == 0;
}

}  // namespace hst

using namespace hst;

struct hst_closure {
  hst_deck deck;
  hst_grid_info g;
  Dims D;
  std::vector<double> y, dyl, der;
  D0Factor f0;
  D0Const fc;
  double *d_der = nullptr, *d_dyl = nullptr, *d_f0 = nullptr;
  Cx<double> *twz = nullptr, *twx = nullptr, *twh = nullptr;
  void *tables = nullptr;  // FP64 tables of the solver's z forward transform
  double2 *fields = nullptr;  // 15 coarse fields: U[3], Pbar[6], Tau[6]
  double2 *Gy = nullptr;      // 3 y derivatives
  double2 *XR = nullptr;      // the workspaces of the three D0 solves
  Cx<double> *Hc = nullptr;   // z-inverse output, 18 fields
  double *phys = nullptr;     // 18 physical fields of the interior rows
  double2 *stage = nullptr;   // layout staging, one field
  int *d_j0 = nullptr;
  double *d_w = nullptr;
  int fine_ny = 0;
  int64_t cap = 0, count = 0;
  float *X = nullptr, *Yd = nullptr;
  WImage *img = nullptr;  // the parameters as the matrix cores' operands
  float *par = nullptr, *m1 = nullptr, *m2 = nullptr, *part = nullptr, *gradd = nullptr;
  double *sse = nullptr, *lossp = nullptr, *mom = nullptr, *meand = nullptr;
  int64_t adam_t = 0;
  double norm[HST_CLOSURE_NORM];
  bool have_norm = false, have_params = false, attached = false;
  hipStream_t own = nullptr;
  size_t nf() const { return (size_t)D.NYg * D.ncol; }
  double2 *field(int k) { return fields + (size_t)k * nf(); }
  size_t fs() const { return (size_t)D.ny * D.nzd * 2 * D.nxd; }
};

namespace {

int cfail(const std::string &m, int rc = 1) {
  set_error("closure: " + m);
  return rc ? rc : 1;
}

#define CHK(call)                                                                               \
  do {                                                                                          \
    hipError_t _e = (call);                                                                     \
    if (_e != hipSuccess) return cfail(std::string(#call) + ": " + hipGetErrorString(_e), (int)_e); \
  } while (0)

hst_closure *g_attached = nullptr;

// the stream: the live state's when there is one (its data are read), else the context's
hipStream_t stream_of(hst_closure *c) {
  StateView v;
  if (state_view(v)) return v.stream;
  return c->own;
}

Norm make_norm(const double *n) {
  Norm nm;
  for (int k = 0; k < 9; k++) {
    nm.mx[k] = (float)n[k];
    nm.rx[k] = 1.0f / (float)n[9 + k];
  }
  for (int k = 0; k < 6; k++) {
    nm.my[k] = (float)n[18 + k];
    nm.ry[k] = 1.0f / (float)n[24 + k];
    nm.sy[k] = (float)n[24 + k];
  }
  return nm;
}

int filter_weights(int nyf, int nyc, std::vector<int> &j0, std::vector<double> &w) {
  if (nyc < 4 || nyf < nyc) return 1;
  j0.assign(nyc, 0);
  w.assign((size_t)nyc * 8, 0.0);
  const double r = 0.5 * (double)nyf / (double)nyc;
  auto cdf = [](double x) {  // integral of the unit hat function up to x
    if (x <= -1.0) return 0.0;
    if (x <= 0.0) return 0.5 * (x + 1.0) * (x + 1.0);
    if (x <= 1.0) return 1.0 - 0.5 * (1.0 - x) * (1.0 - x);
    return 1.0;
  };
  for (int k = 0; k < nyc; k++) {
    const double cen = (double)k * nyf / nyc, a = cen - r, b = cen + r;
    const int lo = (int)std::floor(a), hi = (int)std::ceil(b);
    if (hi - lo + 1 > 8) return 2;
    j0[k] = lo;
    for (int t = 0; t <= hi - lo; t++) w[(size_t)k * 8 + t] = (cdf(b - (lo + t)) - cdf(a - (lo + t))) / (b - a);
  }
  return 0;
}

// gradients (and, with sample, u and the filtered products) of the context's
// fields to physical values: phys fields 0..8 (and 9..17)
int to_physical(hst_closure *c, const double2 *const U[3], bool sample, double sx, double sz, hipStream_t st) {
  const Dims &D = c->D;
  double2 *Gy[3], *XR[3];
  for (int i = 0; i < 3; i++) {
    Gy[i] = c->Gy + (size_t)i * c->nf();
    XR[i] = c->XR + (size_t)i * (D.ny - 2) * D.ncol;
  }
  if (int rc = launch_d0solve(D, 1, 0, 3, U, Gy, nullptr, XR, c->d_f0, c->fc, c->d_der, c->d_dyl, sx, sz, nullptr,
                              nullptr, st))
    return cfail("y derivatives", rc);
  ZSrc zs;
  int nf = 0;
  for (int i = 0; i < 3; i++) {
    zs.p[nf] = U[i]; zs.op[nf++] = 1;
    zs.p[nf] = c->Gy + (size_t)i * c->nf(); zs.op[nf++] = 0;
    zs.p[nf] = U[i]; zs.op[nf++] = 2;
  }
  if (sample) {
    for (int i = 0; i < 3; i++) { zs.p[nf] = U[i]; zs.op[nf++] = 0; }
    for (int p = 0; p < 6; p++) { zs.p[nf] = c->field(HST_CLOSURE_PBAR + p); zs.op[nf++] = 0; }
  }
  switch (D.nzd) {
#define ZC(n) case n: run_czinv<n>(D, zs, nf, c->Hc, c->twz, st); break;
    CLOSURE_Z_SIZES(ZC)
#undef ZC
    default: return cfail("z size");
  }
  switch (D.nxd) {
#define XC(n) case n: run_cxc2r<n>(D, nf, c->Hc, c->phys, c->twx, c->twh, st); break;
    CLOSURE_X_SIZES(XC)
#undef XC
    default: return cfail("x size");
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cfail(std::string("transform launch: ") + hipGetErrorString(e), (int)e);
  return 0;
}

// modelled stress spectra of U into the Tau fields (ghosts at sx, sz)
int stress(hst_closure *c, const double2 *const U[3], double sx, double sz, hipStream_t st) {
  if (!c->have_norm || !c->have_params) return cfail("the network has no parameters or no standardisation");
  const Dims &D = c->D;
  if (int rc = to_physical(c, U, false, sx, sz, st)) return rc;
  InferIO io;
  io.X = nullptr; io.Y = nullptr;
  io.gin = c->phys;
  io.tout = c->phys + 9 * c->fs();
  io.fs = c->fs();
  io.n = (int64_t)c->fs();
  io.mode = 1;
  run_infer(c->img, make_norm(c->norm), io, st);
  Cx<double> *Hp = c->Hc;  // the z-inverse output is free again
  switch (D.nxd) {
#define XC(n) case n: run_cxr2c<n>(D, c->phys + 9 * c->fs(), Hp, c->twx, c->twh, st); break;
    CLOSURE_X_SIZES(XC)
#undef XC
    default: return cfail("x size");
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cfail(std::string("stress launch: ") + hipGetErrorString(e), (int)e);
  int rc = launch_zfft(D, 0, 6, Hp, c->field(HST_CLOSURE_TAU), c->nf(), 2, D.ny, c->tables, st);
  if (rc) return cfail("z forward transform", rc);
  double2 *T[6];
  for (int p = 0; p < 6; p++) T[p] = c->field(HST_CLOSURE_TAU + p);
  rc = launch_ghosts(D, 6, T, sx, sz, st);
  if (rc) return cfail("ghost rows", rc);
  return 0;
}

// the live state has the grid and box of the context (the sizes its kernels assume)
bool same_grid(const StateView &v, const hst_closure *c) {
  const Dims &F = v.D, &D = c->D;
  return F.nx == D.nx && F.ny == D.ny && F.nz == D.nz && v.deck.alfa0 == c->deck.alfa0 &&
         v.deck.beta0 == c->deck.beta0 && v.deck.ly == c->deck.ly && v.deck.S == c->deck.S &&
         v.deck.ystretch == c->deck.ystretch;
}

// the timestep hook: stresses of the live state's velocity added to its products
int hook(void *ctx, double time) {
  hst_closure *c = (hst_closure *)ctx;
  StateView v;
  if (!state_view(v)) return cfail("no live state");
  // the state may have been freed and set up again on another grid since the attach
  if (!same_grid(v, c)) return cfail("the live state's grid is no longer the attached context's");
  double sx, sz;
  deck_shifts(c->deck, c->g.lx, c->g.lz, time, sx, sz);
  const double2 *U[3] = {v.F[HST_V1], v.F[HST_V2], v.F[HST_V3]};
  return profiled("closure", 0.0, [&]() -> int {
    if (int rc = stress(c, U, sx, sz, v.stream)) return rc;
    const size_t n = 6 * c->nf();
    if (v.mixed)
      hipLaunchKernelGGL(k_add_stress<float>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, v.stream,
                         (Cx<float> *)v.P, (const double2 *)c->field(HST_CLOSURE_TAU), n);
    else
      hipLaunchKernelGGL(k_add_stress<double>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, v.stream,
                         (Cx<double> *)v.P, (const double2 *)c->field(HST_CLOSURE_TAU), n);
    return (int)hipGetLastError();
  });
}

void release(hst_closure *c) {
  if (c->own) (void)hipStreamSynchronize(c->own);
  void *ptrs[] = {c->d_der, c->d_dyl, c->d_f0, c->twz, c->twx, c->twh, c->fields, c->Gy, c->XR, c->Hc, c->phys,
                  c->stage, c->d_j0, c->d_w, c->X, c->Yd, c->par, c->m1, c->m2, c->part, c->gradd, c->sse,
                  c->lossp, c->mom, c->meand, c->img};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (c->tables) free_fft_tables(c->tables);
  if (c->own) (void)hipStreamDestroy(c->own);
}

int fill_tw(Cx<double> **dst, int n, double den) {
  std::vector<Cx<double>> h(n);
  for (int k = 0; k < n; k++) {
    const double a = -2.0 * M_PI * (double)k / den;
    h[k] = Cx<double>{std::cos(a), std::sin(a)};
  }
  if (hipMalloc(dst, sizeof(Cx<double>) * n) != hipSuccess) return 1;
  return hipMemcpy(*dst, h.data(), sizeof(Cx<double>) * n, hipMemcpyHostToDevice) != hipSuccess;
}

}  // namespace

extern "C" {

int hst_closure_filter_weights(int ny_fine, int ny_coarse, int32_t *first_row, double *weights) {
  std::vector<int> j0;
  std::vector<double> w;
  if (filter_weights(ny_fine, ny_coarse, j0, w)) return cfail("filter: need 4 <= ny_coarse <= ny_fine, ratio below 6");
  for (int k = 0; k < ny_coarse; k++) first_row[k] = j0[k];
  std::memcpy(weights, w.data(), sizeof(double) * w.size());
  return 0;
}

int hst_closure_create(const hst_deck *coarse, int64_t capacity, hst_closure **out) {
  if (!coarse || !out) return cfail("NULL argument");
  *out = nullptr;
  std::string err = check_deck(*coarse);
  if (!err.empty()) return cfail(err);
  if (capacity < 0) return cfail("negative capacity");
  hst_closure *c = new hst_closure();
  c->deck = *coarse;
  grid_setup(c->deck, c->g, c->y, c->dyl, c->der);
  c->D = make_dims(c->deck, c->g);
  const Dims &D = c->D;
  if (!closure_size_ok(D)) {
    delete c;
    return cfail("coarse grid transform sizes nxd = " + std::to_string(D.nxd) + ", nzd = " + std::to_string(D.nzd) +
                 " are not built for the closure (nxd 32..128, nzd 48..192)");
  }
  d0_factor(c->der, D.ny, c->f0);
  c->fc = d0_const(c->f0);
  auto bad = [&](const char *what, hipError_t e) {
    release(c);
    delete c;
    return cfail(std::string(what) + ": " + hipGetErrorString(e), (int)e);
  };
#define MAL(p, bytes)                                    \
  do {                                                   \
    hipError_t _e = hipMalloc(&(p), (bytes));            \
    if (_e != hipSuccess) return bad("allocation", _e); \
  } while (0)
  hipError_t e = hipStreamCreate(&c->own);
  if (e != hipSuccess) return bad("stream", e);
  std::vector<double> derd((size_t)D.ny * 20);
  for (int iy = 0; iy < D.ny; iy++)
    for (int n = 0; n < 4; n++)
      for (int j = 0; j < 5; j++) derd[(size_t)iy * 20 + n * 5 + j] = c->der[(size_t)iy + (size_t)D.ny * (n + 4 * j)];
  MAL(c->d_der, derd.size() * sizeof(double));
  MAL(c->d_dyl, c->dyl.size() * sizeof(double));
  MAL(c->d_f0, c->f0.rows.size() * sizeof(double));
  (void)hipMemcpy(c->d_der, derd.data(), derd.size() * sizeof(double), hipMemcpyHostToDevice);
  (void)hipMemcpy(c->d_dyl, c->dyl.data(), c->dyl.size() * sizeof(double), hipMemcpyHostToDevice);
  (void)hipMemcpy(c->d_f0, c->f0.rows.data(), c->f0.rows.size() * sizeof(double), hipMemcpyHostToDevice);
  if (fill_tw(&c->twz, D.nzd, D.nzd) || fill_tw(&c->twx, D.nxd, D.nxd) || fill_tw(&c->twh, D.nxd, 2.0 * D.nxd))
    return bad("twiddles", hipErrorOutOfMemory);
  if (make_fft_tables(D, 0, &c->tables)) return bad("tables", hipErrorOutOfMemory);
  MAL(c->fields, 15 * c->nf() * sizeof(double2));
  MAL(c->Gy, 3 * c->nf() * sizeof(double2));
  MAL(c->stage, c->nf() * sizeof(double2));
  MAL(c->XR, 3 * (size_t)(D.ny - 2) * D.ncol * sizeof(double2));
  MAL(c->Hc, 18 * (size_t)D.ny * D.nzd * D.NXp * sizeof(Cx<double>));
  MAL(c->phys, 18 * c->fs() * sizeof(double));
  (void)hipMemset(c->fields, 0, 15 * c->nf() * sizeof(double2));
  (void)hipMemset(c->Gy, 0, 3 * c->nf() * sizeof(double2));
  c->cap = capacity;
  if (capacity > 0) {
    MAL(c->X, (size_t)capacity * 9 * sizeof(float));
    MAL(c->Yd, (size_t)capacity * 6 * sizeof(float));
  }
  MAL(c->img, sizeof(WImage));
  MAL(c->par, NP * sizeof(float));
  MAL(c->m1, NP * sizeof(float));
  MAL(c->m2, NP * sizeof(float));
  MAL(c->gradd, NP * sizeof(float));
  MAL(c->part, (size_t)MAX_PART * NPP * sizeof(float));
  MAL(c->sse, sizeof(double) * 1);
  MAL(c->lossp, sizeof(double) * 4096);
  MAL(c->mom, sizeof(double) * 15 * 1024);
  MAL(c->meand, sizeof(double) * 15);
  (void)hipMemset(c->m1, 0, NP * sizeof(float));
  (void)hipMemset(c->m2, 0, NP * sizeof(float));
#undef MAL
  *out = c;
  return 0;
}

int hst_closure_free(hst_closure *c) {
  if (!c) return 0;
  if (g_attached == c) {
    set_stress_hook(nullptr, nullptr);
    g_attached = nullptr;
  }
  release(c);
  delete c;
  return 0;
}

int hst_closure_filter(hst_closure *c, double time) {
  if (!c) return cfail("NULL context");
  StateView v;
  if (!state_view(v)) return cfail("filter: no live state (hst_gpu_init)");
  const Dims &F = v.D, &D = c->D;
  if (F.nx < D.nx || F.nz < D.nz || F.ny < D.ny || v.deck.alfa0 != c->deck.alfa0 || v.deck.beta0 != c->deck.beta0 ||
      v.deck.ly != c->deck.ly || v.deck.ystretch != 0.0 || c->deck.ystretch != 0.0)
    return cfail("filter: the state's grid must be finer, uniform in y, with the same alfa0, beta0, ly");
  if (c->fine_ny != F.ny) {
    std::vector<int> j0;
    std::vector<double> w;
    if (filter_weights(F.ny, D.ny, j0, w)) return cfail("filter: y ratio not supported (at most 6)");
    for (int k = 0; k < D.ny; k++)
      for (int t = 0; t < 8; t++)
        if (w[(size_t)k * 8 + t] != 0.0 && (j0[k] + t < -2 || j0[k] + t > F.ny + 1))
          return cfail("filter: a weight falls outside the fine rows");
    if (c->d_j0) (void)hipFree(c->d_j0);
    if (c->d_w) (void)hipFree(c->d_w);
    c->d_j0 = nullptr;
    c->d_w = nullptr;
    CHK(hipMalloc(&c->d_j0, sizeof(int) * D.ny));
    CHK(hipMalloc(&c->d_w, sizeof(double) * 8 * D.ny));
    CHK(hipMemcpy(c->d_j0, j0.data(), sizeof(int) * D.ny, hipMemcpyHostToDevice));
    CHK(hipMemcpy(c->d_w, w.data(), sizeof(double) * 8 * D.ny, hipMemcpyHostToDevice));
    c->fine_ny = F.ny;
  }
  hipStream_t st = v.stream;
  const size_t cs = v.mixed ? sizeof(float2) : sizeof(double2);
  FilterArgs fv, fp;
  for (int i = 0; i < 3; i++) {
    fv.src[i] = v.F[HST_V1 + i];
    fv.dst[i] = c->field(HST_CLOSURE_U + i);
  }
  for (int p = 0; p < 6; p++) {
    fp.src[p] = (const char *)v.P + (size_t)p * F.NYg * F.ncol * cs;
    fp.dst[p] = c->field(HST_CLOSURE_PBAR + p);
  }
  const unsigned gx = (unsigned)((D.ncol + 255) / 256);
  hipLaunchKernelGGL(k_filter<double>, dim3(gx, 3), dim3(256), 0, st, fv, F.ncol, F.NZm, F.nz, D, c->d_j0, c->d_w);
  if (v.mixed)
    hipLaunchKernelGGL(k_filter<float>, dim3(gx, 6), dim3(256), 0, st, fp, F.ncol, F.NZm, F.nz, D, c->d_j0, c->d_w);
  else
    hipLaunchKernelGGL(k_filter<double>, dim3(gx, 6), dim3(256), 0, st, fp, F.ncol, F.NZm, F.nz, D, c->d_j0, c->d_w);
  CHK(hipGetLastError());
  double sx, sz;
  deck_shifts(c->deck, c->g.lx, c->g.lz, time, sx, sz);
  double2 *f[8];
  for (int i = 0; i < 8; i++) f[i] = c->field(i);
  int rc = launch_ghosts(D, 8, f, sx, sz, st);
  if (!rc) {
    double2 *last[1] = {c->field(8)};
    rc = launch_ghosts(D, 1, last, sx, sz, st);
  }
  if (rc) return cfail("ghost rows", rc);
  CHK(hipStreamSynchronize(st));
  return 0;
}

int hst_closure_get_field(hst_closure *c, int which, double *host) {
  if (!c || !host) return cfail("NULL argument");
  if (which < 0 || which > 14) return cfail("field index out of range (0..14)");
  hipStream_t st = stream_of(c);
  int rc = launch_to_ref_layout(c->D, c->field(which), c->stage, st);
  if (rc) return cfail("layout", rc);
  CHK(hipMemcpyAsync(host, c->stage, c->nf() * sizeof(double2), hipMemcpyDeviceToHost, st));
  CHK(hipStreamSynchronize(st));
  return 0;
}

int hst_closure_set_field(hst_closure *c, int which, const double *host) {
  if (!c || !host) return cfail("NULL argument");
  if (which < 0 || which > 14) return cfail("field index out of range (0..14)");
  hipStream_t st = stream_of(c);
  CHK(hipMemcpyAsync(c->stage, host, c->nf() * sizeof(double2), hipMemcpyHostToDevice, st));
  int rc = launch_to_device_layout(c->D, c->stage, c->field(which), st);
  if (rc) return cfail("layout", rc);
  CHK(hipStreamSynchronize(st));
  return 0;
}

int hst_closure_sample(hst_closure *c, double time, int64_t *count) {
  if (!c) return cfail("NULL context");
  const int64_t npts = (int64_t)c->fs();
  if (c->count + npts > c->cap)
    return cfail("data set full: " + std::to_string(c->count) + " + " + std::to_string(npts) + " > capacity " +
                 std::to_string(c->cap));
  hipStream_t st = stream_of(c);
  double sx, sz;
  deck_shifts(c->deck, c->g.lx, c->g.lz, time, sx, sz);
  const double2 *U[3] = {c->field(0), c->field(1), c->field(2)};
  if (int rc = to_physical(c, U, true, sx, sz, st)) return rc;
  hipLaunchKernelGGL(k_samples, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, st, c->phys, c->fs(), npts,
                     c->X + (size_t)c->count * 9, c->Yd + (size_t)c->count * 6);
  CHK(hipGetLastError());
  CHK(hipStreamSynchronize(st));
  c->count += npts;
  if (count) *count = c->count;
  return 0;
}

int hst_closure_set_dataset(hst_closure *c, int64_t n, const float *x, const float *y) {
  if (!c || !x || !y) return cfail("NULL argument");
  if (n < 0 || n > c->cap) return cfail("data set size beyond capacity");
  CHK(hipMemcpy(c->X, x, (size_t)n * 9 * sizeof(float), hipMemcpyHostToDevice));
  CHK(hipMemcpy(c->Yd, y, (size_t)n * 6 * sizeof(float), hipMemcpyHostToDevice));
  c->count = n;
  return 0;
}

int hst_closure_get_dataset(hst_closure *c, int64_t first, int64_t n, float *x, float *y) {
  if (!c) return cfail("NULL context");
  if (first < 0 || n < 0 || first + n > c->count) return cfail("range beyond the data set");
  if (x) CHK(hipMemcpy(x, c->X + (size_t)first * 9, (size_t)n * 9 * sizeof(float), hipMemcpyDeviceToHost));
  if (y) CHK(hipMemcpy(y, c->Yd + (size_t)first * 6, (size_t)n * 6 * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int hst_closure_count(hst_closure *c, int64_t *count) {
  if (!c || !count) return cfail("NULL argument");
  *count = c->count;
  return 0;
}

int hst_closure_normalise(hst_closure *c, double *norm) {
  if (!c) return cfail("NULL context");
  if (c->count < 2) return cfail("normalise: fewer than two samples");
  hipStream_t st = c->own;
  const int nblk = 1024;
  double s[15], q[15];
  std::vector<double> h((size_t)nblk * 15);
  for (int pass = 0; pass < 2; pass++) {
    hipLaunchKernelGGL(k_moments, dim3(nblk), dim3(256), 0, st, c->X, c->Yd, c->count, c->meand, pass, c->mom);
    CHK(hipGetLastError());
    CHK(hipMemcpyAsync(h.data(), c->mom, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    CHK(hipStreamSynchronize(st));
    double *acc = pass ? q : s;
    for (int k = 0; k < 15; k++) {
      acc[k] = 0.0;
      for (int b = 0; b < nblk; b++) acc[k] += h[(size_t)b * 15 + k];
    }
    if (pass == 0) {
      double mean[15];
      for (int k = 0; k < 15; k++) mean[k] = s[k] / (double)c->count;
      CHK(hipMemcpy(c->meand, mean, sizeof(mean), hipMemcpyHostToDevice));
    }
  }
  for (int k = 0; k < 15; k++) {
    const double mean = s[k] / (double)c->count, sd = std::sqrt(q[k] / (double)c->count);
    const int mi = k < 9 ? k : 18 + (k - 9), si = k < 9 ? 9 + k : 24 + (k - 9);
    c->norm[mi] = mean;
    c->norm[si] = sd > 0.0 ? sd : 1.0;
  }
  c->have_norm = true;
  if (norm) std::memcpy(norm, c->norm, sizeof(c->norm));
  return 0;
}

int hst_closure_set_norm(hst_closure *c, const double *norm) {
  if (!c || !norm) return cfail("NULL argument");
  for (int k = 0; k < 9; k++)
    if (!(norm[9 + k] > 0.0)) return cfail("standard deviations must be positive");
  for (int k = 0; k < 6; k++)
    if (!(norm[24 + k] > 0.0)) return cfail("standard deviations must be positive");
  std::memcpy(c->norm, norm, sizeof(c->norm));
  c->have_norm = true;
  return 0;
}

int hst_closure_get_norm(hst_closure *c, double *norm) {
  if (!c || !norm) return cfail("NULL argument");
  if (!c->have_norm) return cfail("no standardisation yet");
  std::memcpy(norm, c->norm, sizeof(c->norm));
  return 0;
}

int hst_closure_init_params(hst_closure *c, uint64_t seed) {
  if (!c) return cfail("NULL context");
  std::mt19937_64 gen(seed);
  std::vector<float> p(NP, 0.0f);
  auto fill = [&](int off, int fan_out, int fan_in) {
    const double a = std::sqrt(6.0 / (fan_in + fan_out));
    std::uniform_real_distribution<double> u(-a, a);
    for (int i = 0; i < fan_out * fan_in; i++) p[off + i] = (float)u(gen);
  };
  fill(OW1, 64, 9);
  fill(OW2, 64, 64);
  fill(OW3, 6, 64);
  return hst_closure_set_params(c, p.data());
}

int hst_closure_set_params(hst_closure *c, const float *params) {
  if (!c || !params) return cfail("NULL argument");
  CHK(hipMemcpy(c->par, params, NP * sizeof(float), hipMemcpyHostToDevice));
  CHK(hipMemset(c->m1, 0, NP * sizeof(float)));
  CHK(hipMemset(c->m2, 0, NP * sizeof(float)));
  hipLaunchKernelGGL(k_pack, dim3(1), dim3(1024), 0, c->own, c->par, c->img);
  CHK(hipGetLastError());
  CHK(hipStreamSynchronize(c->own));  // the image is read on the live state's stream too
  c->adam_t = 0;
  c->have_params = true;
  return 0;
}

int hst_closure_get_params(hst_closure *c, float *params) {
  if (!c || !params) return cfail("NULL argument");
  CHK(hipMemcpy(params, c->par, NP * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int hst_closure_grad(hst_closure *c, int64_t first, int64_t n, float *grad, double *loss) {
  if (!c) return cfail("NULL context");
  if (!c->have_norm || !c->have_params) return cfail("grad: parameters and standardisation needed");
  if (first < 0 || n < 1 || first + n > c->count) return cfail("grad: range beyond the data set");
  if (n > (int64_t)SPB * MAX_PART) return cfail("grad: at most " + std::to_string(SPB * MAX_PART) + " samples");
  hipStream_t st = c->own;
  TrainArgs ta{c->X, c->Yd, n, first, 1, 0, INT64_MAX, (float)(2.0 / ((double)n * 6.0))};
  const int nblk = (int)((n + SPB - 1) / SPB);
  hipLaunchKernelGGL(k_mlp_train<true>, dim3(nblk), dim3(TNT), 0, st, c->img, make_norm(c->norm), ta, c->part,
                     c->lossp);
  hipLaunchKernelGGL(k_adam, dim3((NP + 1 + 63) / 64), dim3(64 * AR), 0, st, c->par, c->m1, c->m2, c->part, nblk, 0,
                     0.0f, 0.0f, 0.0f, c->gradd, c->sse, c->img);
  CHK(hipGetLastError());
  double sse = 0.0;
  if (grad) CHK(hipMemcpyAsync(grad, c->gradd, NP * sizeof(float), hipMemcpyDeviceToHost, st));
  CHK(hipMemcpyAsync(&sse, c->sse, sizeof(double), hipMemcpyDeviceToHost, st));
  CHK(hipStreamSynchronize(st));
  if (loss) *loss = sse / ((double)n * 6.0);
  return 0;
}

// loss over [first, first + n) without gradients
static int eval_loss(hst_closure *c, int64_t first, int64_t n, double *loss) {
  hipStream_t st = c->own;
  double total = 0.0;
  const int64_t chunk = (int64_t)SPB * 4096;
  std::vector<double> h(4096);
  for (int64_t b0 = 0; b0 < n; b0 += chunk) {
    const int64_t m = std::min(chunk, n - b0);
    TrainArgs ta{c->X, c->Yd, m, first + b0, 1, 0, INT64_MAX, 0.0f};
    const int nblk = (int)((m + SPB - 1) / SPB);
    hipLaunchKernelGGL(k_mlp_train<false>, dim3(nblk), dim3(TNT), 0, st, c->img, make_norm(c->norm), ta, c->part,
                       c->lossp);
    CHK(hipGetLastError());
    CHK(hipMemcpyAsync(h.data(), c->lossp, nblk * sizeof(double), hipMemcpyDeviceToHost, st));
    CHK(hipStreamSynchronize(st));
    for (int b = 0; b < nblk; b++) total += h[b];
  }
  *loss = total / ((double)n * 6.0);
  return 0;
}

int hst_closure_train(hst_closure *c, int epochs, int batch, double lr, uint64_t seed, int64_t n_train,
                      double *loss, double *val_loss) {
  if (!c) return cfail("NULL context");
  if (!c->have_norm || !c->have_params) return cfail("train: parameters and standardisation needed");
  if (n_train <= 0 || n_train > c->count) n_train = c->count;
  if (batch < SPB || batch % SPB || batch > n_train || batch > SPB * MAX_PART)
    return cfail("train: batch must be a multiple of 128, at most the training samples and " +
                 std::to_string(SPB * MAX_PART));
  if (epochs < 1) return cfail("train: epochs < 1");
  hipStream_t st = c->own;
  const Norm nm = make_norm(c->norm);
  const int64_t nb = n_train / batch;
  const int nblk = batch / SPB;
  std::mt19937_64 gen(seed);
  double *dsse = nullptr;
  CHK(hipMalloc(&dsse, sizeof(double) * nb));
  std::vector<double> h(nb);
  for (int e = 0; e < epochs; e++) {
    // this epoch's order: sample = (mul * position + add) mod n_train, mul coprime to n_train
    std::uniform_int_distribution<int64_t> um(1, std::max<int64_t>(1, n_train - 1)), ua(0, n_train - 1);
    int64_t mul = um(gen);
    while (std::gcd(mul, n_train) != 1) mul = um(gen);
    const int64_t add = ua(gen);
    for (int64_t b = 0; b < nb; b++) {
      c->adam_t++;
      const double t = (double)c->adam_t;
      const float c1 = (float)(1.0 / (1.0 - std::pow(0.9, t))), c2 = (float)(1.0 / (1.0 - std::pow(0.999, t)));
      TrainArgs ta{c->X, c->Yd, batch, b * batch, mul, add, n_train, (float)(2.0 / ((double)batch * 6.0))};
      hipLaunchKernelGGL(k_mlp_train<true>, dim3(nblk), dim3(TNT), 0, st, c->img, nm, ta, c->part, c->lossp);
      hipLaunchKernelGGL(k_adam, dim3((NP + 1 + 63) / 64), dim3(64 * AR), 0, st, c->par, c->m1, c->m2, c->part, nblk,
                         1, (float)lr, c1, c2, c->gradd, dsse + b, c->img);
    }
    hipError_t err = hipGetLastError();
    if (err == hipSuccess) err = hipMemcpyAsync(h.data(), dsse, sizeof(double) * nb, hipMemcpyDeviceToHost, st);
    if (err == hipSuccess) err = hipStreamSynchronize(st);
    if (err != hipSuccess) {
      (void)hipFree(dsse);
      return cfail(std::string("train: ") + hipGetErrorString(err), (int)err);
    }
    double s = 0.0;
    for (int64_t b = 0; b < nb; b++) s += h[b] / ((double)batch * 6.0);
    if (loss) loss[e] = s / (double)nb;
    if (val_loss) {
      val_loss[e] = 0.0;
      if (n_train < c->count) {
        int rc = eval_loss(c, n_train, c->count - n_train, &val_loss[e]);
        if (rc) {
          (void)hipFree(dsse);
          return rc;
        }
      }
    }
  }
  (void)hipFree(dsse);
  return 0;
}

int hst_closure_predict(hst_closure *c, int64_t n, const float *x, float *y) {
  if (!c || !x || !y) return cfail("NULL argument");
  if (!c->have_norm || !c->have_params) return cfail("predict: parameters and standardisation needed");
  if (n < 1) return 0;
  hipStream_t st = c->own;
  float *dx = nullptr, *dy = nullptr;
  CHK(hipMalloc(&dx, (size_t)n * 9 * sizeof(float)));
  if (hipMalloc(&dy, (size_t)n * 6 * sizeof(float)) != hipSuccess) {
    (void)hipFree(dx);
    return cfail("predict: allocation");
  }
  InferIO io{dx, dy, nullptr, nullptr, 0, n, 0};
  hipError_t e = hipMemcpyAsync(dx, x, (size_t)n * 9 * sizeof(float), hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    run_infer(c->img, make_norm(c->norm), io, st);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(y, dy, (size_t)n * 6 * sizeof(float), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(dx);
  (void)hipFree(dy);
  if (e != hipSuccess) return cfail(std::string("predict: ") + hipGetErrorString(e), (int)e);
  return 0;
}

int hst_closure_stress(hst_closure *c, double time) {
  if (!c) return cfail("NULL context");
  hipStream_t st = stream_of(c);
  double sx, sz;
  deck_shifts(c->deck, c->g.lx, c->g.lz, time, sx, sz);
  const double2 *U[3] = {c->field(0), c->field(1), c->field(2)};
  if (int rc = stress(c, U, sx, sz, st)) return rc;
  CHK(hipStreamSynchronize(st));
  return 0;
}

int hst_closure_attach(hst_closure *c, int on) {
  if (!c) return cfail("NULL context");
  if (!on) {
    if (g_attached == c) {
      set_stress_hook(nullptr, nullptr);
      g_attached = nullptr;
    }
    return 0;
  }
  StateView v;
  if (!state_view(v)) return cfail("attach: no live state");
  if (!same_grid(v, c)) return cfail("attach: the live state's grid is not the context's");
  if (!c->have_norm || !c->have_params) return cfail("attach: the network has no parameters or no standardisation");
  set_stress_hook(hook, c);
  g_attached = c;
  return 0;
}

}  // extern "C"
