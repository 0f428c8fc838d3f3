// Learned block preconditioner (see mlp.h): feature extraction, the network
// (bf16 weights, fp32 activations and accumulation on the fp32 matrix
// cores), its backward pass and Adam training, inference inside the local
// GMRES, and the collection of training pairs from block-Jacobi solves.
//
// Network: y = W3^T relu(W2^T relu(W1^T x + b1) + b2) + b3 + jac(x) on
// columns x of the feature matrix X (kMlpIn x M, column-major, one column
// per block), where jac(x) = residual features / diagonal features is the
// point-Jacobi solution of the block that the layers correct.
// Features of block b = (b1, b2) of the local vector v (rx1, n, rx2):
//   [diag(B_b), superdiag(B_b), subdiag(B_b)] / s_b and r_b / |r_b|,
// with B_b(i,j) = sum_{a1,a2} Phi1(b1,b1,a1) A(a1,i,j,a2) Phi2(b2,a2,b2)
// (the block of djac_gen 'c', tt_linalg.f90:412-416), r_b = v(b1, :, b2)
// and s_b = mean |diag(B_b)|; the block correction is y_b |r_b| / s_b.
#include "mlp.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace ttf {

namespace {

struct MlpModel {
  bool ready = false;
  float* master = nullptr;    // fp32 parameters (what Adam updates)
  uint16_t* wbf = nullptr;    // bf16 copy read by the forward kernels
  float* wr = nullptr;        // fp32 values of the bf16 weights (backward GEMMs)
  float* am = nullptr;        // Adam moments
  float* av = nullptr;
  long step = 0;
};
MlpModel g_model;

struct MlpSink {
  bool active = false;
  int64_t cap = 0, count = 0;
  int per_apply = 0;
  uint64_t counter = 0;
  float* X = nullptr;   // kMlpIn x cap
  float* T = nullptr;   // kMlpOut x cap
  float* inv = nullptr; // per-sample s_b / |r_b| staging
  int64_t inv_cap = 0;
};
MlpSink g_sink;

void ensure_model() {
  if (g_model.master) return;
  const size_t nb = sizeof(float) * (size_t)kMlpParams;
  TTF_HIP(hipMalloc(&g_model.master, nb));
  TTF_HIP(hipMalloc(&g_model.wbf, sizeof(uint16_t) * (size_t)kMlpParams));
  TTF_HIP(hipMalloc(&g_model.wr, nb));
  TTF_HIP(hipMalloc(&g_model.am, nb));
  TTF_HIP(hipMalloc(&g_model.av, nb));
}

__device__ __forceinline__ uint16_t to_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);   // inf / nan kept
  u += 0x7fffu + ((u >> 16) & 1u);                                      // nearest, ties to even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// master -> bf16 copy and its fp32 value
__global__ void round_params_kernel(int64_t np, const float* __restrict__ master, uint16_t* __restrict__ wbf,
                                    float* __restrict__ wr) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < np; e += (int64_t)gridDim.x * blockDim.x) {
    const uint16_t h = to_bf16(master[e]);
    wbf[e] = h;
    wr[e] = from_bf16(h);
  }
}

// One wave per output column c; block b = (b_start + c * b_stride) mod nb.
// Writes X(:, c), scale(c) = |r_b| / s_b and, if inv is given,
// inv(c) = s_b / |r_b| (0 for a zero slice).
__global__ __launch_bounds__(256) void features_kernel(int rx1, int n, int rx2, int ra1, int ra2,
                                                       const double* __restrict__ phi1, const double* __restrict__ A,
                                                       const double* __restrict__ phi2, const double* __restrict__ v,
                                                       int ncols, int64_t b_start, int64_t b_stride,
                                                       float* __restrict__ X, float* __restrict__ scale,
                                                       float* __restrict__ inv) {
  const int lane = threadIdx.x & 63;
  const int64_t col = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  if (col >= ncols) return;
  const int64_t nb = (int64_t)rx1 * rx2;
  const int64_t b = (b_start + col * b_stride) % nb;
  const int b1 = (int)(b % rx1), b2 = (int)(b / rx1);
  const int i = lane;   // n == 64
  double dg = 0.0, up = 0.0, lo = 0.0;
  for (int a1 = 0; a1 < ra1; ++a1) {
    const double d1 = phi1[b1 + (int64_t)rx1 * (b1 + (int64_t)rx1 * a1)];
    for (int a2 = 0; a2 < ra2; ++a2) {
      const double c = d1 * phi2[b2 + (int64_t)rx2 * (a2 + (int64_t)ra2 * b2)];
      const int64_t base = a1 + (int64_t)ra1 * n * n * a2;
      dg += c * A[base + (int64_t)ra1 * (i + (int64_t)n * i)];
      if (i < n - 1) {
        up += c * A[base + (int64_t)ra1 * (i + (int64_t)n * (i + 1))];
        lo += c * A[base + (int64_t)ra1 * ((i + 1) + (int64_t)n * i)];
      }
    }
  }
  const double r = v[b1 + (int64_t)rx1 * (i + (int64_t)n * b2)];
  const double s = wave_sum(fabs(dg)) / n;
  const double rn = sqrt(wave_sum(r * r));
  const double sinv = s > 0.0 ? 1.0 / s : 0.0;
  const double rinv = rn > 0.0 ? 1.0 / rn : 0.0;
  float* x = X + (int64_t)kMlpIn * col;
  x[i] = (float)(dg * sinv);
  x[n + i] = (float)(up * sinv);
  x[2 * n + i] = (float)(lo * sinv);
  x[3 * n + i] = (float)(r * rinv);
  if (lane == 0) {
    scale[col] = (float)(rn * sinv);
    if (inv) inv[col] = (float)(rn > 0.0 ? s * rinv : 0.0);
  }
}

// ---- training: the forward and backward products on the f32 matrix cores,
// through the GEMM engine's tiles with the elementwise work in their
// epilogues.  A batch of 1024 columns is a few tens of MFLOP, so what counts
// is launches and how many work-groups each one has: seven launches of 32 x
// 32 or 64 x 64 tiles, in place of seventeen whose bias sums ran one thread
// per row.  Loss and gradient of 1024 columns: 873 -> 128 us, 52 us of it in
// these kernels and the rest in bringing 0.6 MB of gradient to the host.
//
// Y (N x M, ld N) = act(W^T X + b) for W (K x N, ld K; the fp32 values of
// the bf16 weights) and X (K x M, ld K).  MODE 0: act = ReLU, Y = H.  MODE 1
// (the output layer): the point-Jacobi term X0(3 kMlpBlock + n, m) /
// X0(n, m) of the input features X0 is added, Y = dL/dY = f (y - T) with the
// targets T, and part[work-group] = the sum of (y - T)^2.
typedef GemmTile<float, 32, 32, 64, 2, 2, true, kVecBoth> LayerTile;

template <int MODE>
__global__ __launch_bounds__(256, 2) void train_layer_kernel(GemmOp<float> op, const float* __restrict__ bias,
                                                             const float* __restrict__ X0,
                                                             const float* __restrict__ T, float f,
                                                             double* __restrict__ part) {
  const int tilesN = (op.N + 31) / 32;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int tm = wg / tilesN, tn = wg - tm * tilesN;
  LayerTile t;
  t.sums(op, op.A, op.B, tm * 32, tn * 32, 0, op.K);
  // the epilogue's operands, from clamped in-range indices before any is
  // used: loaded under each output's own condition they become a branch
  // with a full wait apiece
  float eb[4], ed[4], ex[4], et[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = min(tm * 32 + LayerTile::row(0, r), op.M - 1);
    const int m = min(tn * 32 + LayerTile::col(0, r), op.N - 1);
    eb[r] = bias[n];
    if (MODE == 1) {
      ed[r] = X0[n + (int64_t)kMlpIn * m];
      ex[r] = X0[3 * kMlpBlock + n + (int64_t)kMlpIn * m];
      et[r] = T[n + (int64_t)op.M * m];
    }
  }
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = tm * 32 + LayerTile::row(0, r), m = tn * 32 + LayerTile::col(0, r);
    if (n < op.M && m < op.N) {
      float val = t.acc[0][0][r] + eb[r];
      if (MODE == 0) {
        val = fmaxf(val, 0.f);
      } else {
        val += ed[r] != 0.f ? ex[r] / ed[r] : 0.f;
        const float d = val - et[r];
        s += (double)d * d;
        val = f * d;
      }
      op.C[n + (int64_t)op.M * m] = val;
    }
  }
  if (MODE == 1) {
    __shared__ double red[4];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
  }
}

// The backward sums are folded per chunk of 64 (the split sums that they
// replace were); the forward ones stay one chain, so that the loss keeps its
// bits.
typedef GemmTile<float, 32, 32, 64, 2, 2, true, kVecBoth, true> BackTile;

// dH (kMlpHid x M) = W D with the ReLU derivative from the activation H
// itself: zero where H is not positive.
__global__ __launch_bounds__(256, 2) void train_back_kernel(GemmOp<float> op, const float* __restrict__ H) {
  const int tilesN = (op.N + 31) / 32;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int tm = wg / tilesN, tn = wg - tm * tilesN;
  BackTile t;
  t.sums(op, op.A, op.B, tm * 32, tn * 32, 0, op.K);
  float h[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    h[r] = H[min(tm * 32 + BackTile::row(0, r), op.M - 1) +
             (int64_t)op.M * min(tn * 32 + BackTile::col(0, r), op.N - 1)];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = tm * 32 + BackTile::row(0, r), m = tn * 32 + BackTile::col(0, r);
    if (n < op.M && m < op.N) op.C[n + (int64_t)op.M * m] = h[r] > 0.f ? t.acc[0][0][r] : 0.f;
  }
}

// All gradients over one slice of columns per group of work-groups, into
// the slice's own parameter vector part + slice kMlpParams: the tiles of the
// three weight gradients In_l D_l^T (64 x 64, four rows of tiles each), then
// the bias gradients, 64 rows of D_l per work-group.
constexpr int kGradSlices = 16;
constexpr int kGradTiles = 4 * (kMlpHid + kMlpHid + kMlpOut) / 64;   // 36 weight tiles
constexpr int kGradRows = (kMlpHid + kMlpHid + kMlpOut) / 64;        // 9 bias groups
static_assert(kMlpIn == 256 && kMlpHid == 256 && kMlpOut == 64, "gradient tiles");
typedef GemmTile<float, 64, 64, 32, 2, 2, true, kVecBoth, true> GradTile;

struct WeightGrads {
  const float* in[3];   // X, H1, H2 (256 x M)
  const float* d[3];    // dH1, dH2, dY (256, 256, 64 rows x M)
  int M, slice, nslices;
};

__global__ __launch_bounds__(256, 2) void weight_grad_kernel(WeightGrads a, float* __restrict__ part) {
  const int per = kGradTiles + kGradRows;
  const int s = blockIdx.x / per;
  int u = blockIdx.x - s * per;
  const int m0 = s * a.slice, m1 = min(a.M, m0 + a.slice);
  float* out = part + (int64_t)kMlpParams * s;
  const bool weight = u < kGradTiles;
  if (!weight) u = 4 * (u - kGradTiles);
  const int l = u < 16 ? 0 : (u < 32 ? 1 : 2);   // 16, 16 and 4 tiles
  u -= 16 * l;
  const int tn = u >> 2, tm = u & 3, cols = l == 2 ? kMlpOut : kMlpHid;
  const float* D = a.d[l];
  if (weight) {
    out += l == 0 ? kMlpOffW1 : (l == 1 ? kMlpOffW2 : kMlpOffW3);
    GemmOp<float> op{};
    op.M = kMlpIn; op.N = cols; op.K = a.M;
    op.sAi = 1; op.sAk = kMlpIn;
    op.sBj = 1; op.sBk = cols;
    GradTile t;
    t.sums(op, a.in[l], D, 64 * tm, 64 * tn, m0, m1);
#pragma unroll
    for (int i = 0; i < GradTile::FM; ++i)
#pragma unroll
      for (int j = 0; j < GradTile::FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[64 * tm + GradTile::row(i, r) + kMlpIn * (64 * tn + GradTile::col(j, r))] = t.acc[i][j][r];
  } else {
    __shared__ float red[4][64];
    const int r = threadIdx.x & 63, g = threadIdx.x >> 6, row = 64 * tn + r;
    float sum = 0.f;
    for (int m = m0 + g; m < m1; m += 32) {   // eight columns of this thread in flight
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = D[row + (int64_t)cols * min(m + 4 * q, m1 - 1)];
#pragma unroll
      for (int q = 0; q < 8; ++q) sum += m + 4 * q < m1 ? v[q] : 0.f;
    }
    red[g][r] = sum;
    __syncthreads();
    if (g == 0)
      out[(l == 0 ? kMlpOffB1 : (l == 1 ? kMlpOffB2 : kMlpOffB3)) + row] =
          (red[0][r] + red[1][r]) + (red[2][r] + red[3][r]);
  }
}

// g = the sum of the slices in order; the last work-group adds the loss
// partials instead: loss = scale * their sum.
__global__ __launch_bounds__(256) void grad_reduce_kernel(int nslices, const float* __restrict__ part,
                                                          float* __restrict__ g, int nloss,
                                                          const double* __restrict__ lpart, double scale,
                                                          double* __restrict__ loss) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ double red[4];
    double s = 0.0;
    for (int i = threadIdx.x; i < nloss; i += 256) s += lpart[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *loss = ((red[0] + red[1]) + (red[2] + red[3])) * scale;
    return;
  }
  const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (e >= kMlpParams) return;
  float v[kGradSlices];
#pragma unroll
  for (int s = 0; s < kGradSlices; ++s) v[s] = part[e + kMlpParams * (int64_t)min(s, nslices - 1)];
  float sum = 0.f;
#pragma unroll
  for (int s = 0; s < kGradSlices; ++s) sum += s < nslices ? v[s] : 0.f;
  g[e] = sum;
}

// ---- inference: the whole network in one launch on gfx950's bf16 matrix
// cores, with the activations rounded to bf16 (round to nearest even) at
// each layer's input and the products accumulated in fp32 by
// v_mfma_f32_16x16x32_bf16.  Lane l feeds row (or column) l % 16 and the
// eight consecutive k = 8 (l / 16) .. +7 of each 32-deep step to both
// operands, so the A and B elements it supplies meet at the same k.
//
// A work-group of eight waves takes 16 columns through all three layers,
// the activations in LDS and the weights (288 KB in bf16) from L2: 16
// columns make 256 work-groups of the 4096 blocks of a rank 64 x 64 problem.
// What bounds it is latency, so each layer's weights are requested a phase
// before they are used.  Separate feature, layer and scatter kernels took 43
// + 32 + 5 us for those blocks (the features' strided reads of A's diagonals
// most of it); with the diagonals packed first and everything in one kernel
// the apply takes 22 us instead of 78.
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf4_t __attribute__((ext_vector_type(4)));
constexpr int kBfK = 256;
static_assert(kMlpIn == kBfK && kMlpHid == kBfK && kMlpOut == 64, "the inference kernel's layer sizes");
constexpr int kInfCols = 16, kInfWaves = 8, kInfThreads = 64 * kInfWaves;
constexpr int kActLd = kBfK + 8;   // bf16 per column of activations: 16-byte rows, spread over the banks

// The three central diagonals of A's bond slices: Ad[k][q][i], k = a1 ra2 +
// a2, q = diagonal, super-, subdiagonal (zero past the edge).
__global__ __launch_bounds__(192) void diagonals_kernel(int n, int ra1, int ra2, const double* __restrict__ A,
                                                        double* __restrict__ Ad) {
  const int a1 = blockIdx.x / ra2, a2 = blockIdx.x - a1 * ra2;
  const int q = threadIdx.x >> 6, i = threadIdx.x & 63;
  const int row = q == 2 ? i + 1 : i, col = q == 1 ? i + 1 : i;
  const bool in = row < n && col < n;
  const double v = A[a1 + ra1 * (min(row, n - 1) + (int64_t)n * (min(col, n - 1) + (int64_t)n * a2))];
  Ad[192 * (int64_t)blockIdx.x + threadIdx.x] = in ? v : 0.0;
}

struct InferArgs {
  int ncols;
  const uint16_t* w;     // bf16 parameters
  const float* master;   // fp32 parameters (biases)
  // columns from X (kMlpIn x ncols) to Y (kMlpOut x ncols)
  const float* X;
  float* Y;
  // or the blocks of the local vector v (rx1, 64, rx2), corrections to z
  int rx1, rx2, ra1, ra2;
  const double* phi1;
  const double* Ad;
  const double* phi2;
  const double* v;
  double* z;
};

// One 16-row group of W^T act(:, 16 columns): fragments from registers (w)
// and LDS.
__device__ __forceinline__ f4_t infer_rows(const uint4 (&w)[kBfK / 32], const __bf16* act) {
  f4_t acc = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kBfK / 32; ++s)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, w[s]),
                                                  *reinterpret_cast<const bf8_t*>(act + 32 * s), acc, 0, 0, 0);
  return acc;
}

template <bool BLOCKS>
__global__ __launch_bounds__(kInfThreads, 2) void infer_kernel(InferArgs a) {
  __shared__ __attribute__((aligned(16))) __bf16 act[2][kInfCols * kActLd];
  __shared__ float skip_d[kInfCols][kMlpBlock + 1], skip_r[kInfCols][kMlpBlock + 1];
  __shared__ float scale[kInfCols];
  __shared__ double rs[BLOCKS ? kInfCols : 1][kMlpBlock + 1];
  __shared__ double cs[BLOCKS ? kInfCols : 1][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * kInfCols;
  // wave w owns rows 32 w .. 32 w + 31 of the hidden layers
  auto weights = [&](int64_t off, int row, uint4 (&w)[kBfK / 32]) {
    const uint16_t* p = a.w + off + 8 * g + (int64_t)kBfK * (row + c);
#pragma unroll
    for (int s = 0; s < kBfK / 32; ++s) w[s] = *reinterpret_cast<const uint4*>(p + 32 * s);
  };
  uint4 w1[2][kBfK / 32];
  weights(kMlpOffW1, 32 * wave, w1[0]);
  weights(kMlpOffW1, 32 * wave + 16, w1[1]);

  if constexpr (BLOCKS) {
    // residual slices: consecutive columns are consecutive in memory
    const int64_t nblk = (int64_t)a.rx1 * a.rx2;
    for (int e = tid; e < kInfCols * kMlpBlock; e += kInfThreads) {
      const int cc = e & (kInfCols - 1), i = e / kInfCols;
      const int64_t b = min((int64_t)col0 + cc, nblk - 1);
      const int64_t b2 = b / a.rx1, b1 = b - b2 * a.rx1;
      rs[cc][i] = a.v[b1 + a.rx1 * (i + (int64_t)kMlpBlock * b2)];
    }
    // the blocks' diagonals: this wave's two columns, bond pairs in the order
    // of k, 64 coefficients at a time through LDS
    const int nk = a.ra1 * a.ra2, q0 = 2 * wave;
    double dg[2] = {0.0, 0.0}, up[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    for (int k0 = 0; k0 < nk; k0 += 64) {
      const int k = min(k0 + lane, nk - 1), a1 = k / a.ra2, a2 = k - a1 * a.ra2;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int64_t b = min((int64_t)col0 + q0 + u, nblk - 1);
        const int64_t b2 = b / a.rx1, b1 = b - b2 * a.rx1;
        cs[q0 + u][lane] = a.phi1[b1 + a.rx1 * (b1 + a.rx1 * (int64_t)a1)] *
                           a.phi2[b2 + a.rx2 * (a2 + a.ra2 * b2)];
      }
      __syncthreads();
      const double* ad = a.Ad + 192 * (int64_t)k0 + lane;
      const int kn = min(64, nk - k0);
      for (int k4 = 0; k4 < kn; k4 += 4) {   // four bond pairs' loads in flight
        double d[4][3];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int q = 0; q < 3; ++q) d[t][q] = ad[192 * min(k4 + t, kn - 1) + 64 * q];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (k4 + t < kn) {   // uniform
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const double cc = cs[q0 + u][k4 + t];
              dg[u] += cc * d[t][0];
              up[u] += cc * d[t][1];
              lo[u] += cc * d[t][2];
            }
          }
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int q = q0 + u;
      const double r = rs[q][lane];
      const double sm = wave_sum(fabs(dg[u])) / kMlpBlock;
      const double rn = sqrt(wave_sum(r * r));
      const double sinv = sm > 0.0 ? 1.0 / sm : 0.0;
      const double rinv = rn > 0.0 ? 1.0 / rn : 0.0;
      const float fd = (float)(dg[u] * sinv), fr = (float)(r * rinv);
      __bf16* x = act[0] + q * kActLd + lane;
      x[0] = (__bf16)fd;
      x[kMlpBlock] = (__bf16)(float)(up[u] * sinv);
      x[2 * kMlpBlock] = (__bf16)(float)(lo[u] * sinv);
      x[3 * kMlpBlock] = (__bf16)fr;
      skip_d[q][lane] = fd;
      skip_r[q][lane] = fr;
      if (lane == 0) scale[q] = (float)(rn * sinv);
    }
  } else {
    // two columns per wave, four features per lane
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int q = 2 * wave + u;
      const float* x = a.X + (int64_t)kMlpIn * min(col0 + q, a.ncols - 1) + lane;
      float f[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) f[t] = x[64 * t];
#pragma unroll
      for (int t = 0; t < 4; ++t) act[0][q * kActLd + 64 * t + lane] = (__bf16)f[t];
      skip_d[q][lane] = f[0];
      skip_r[q][lane] = f[3];
    }
  }

  // hidden layers: rows 32 wave + 16 i + 4 g + r, column c
  auto hidden = [&](const uint4 (&w)[2][kBfK / 32], int64_t bias, const __bf16* in, __bf16* out) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 32 * wave + 16 * i + 4 * g;
      const float* pb = a.master + bias + row;
      const float b[4] = {pb[0], pb[1], pb[2], pb[3]};
      const f4_t acc = infer_rows(w[i], in + c * kActLd + 8 * g);
      bf4_t h;
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = (__bf16)fmaxf(acc[r] + b[r], 0.f);
      *reinterpret_cast<bf4_t*>(out + c * kActLd + row) = h;
    }
  };
  uint4 w2[2][kBfK / 32];
  weights(kMlpOffW2, 32 * wave, w2[0]);
  weights(kMlpOffW2, 32 * wave + 16, w2[1]);
  __syncthreads();
  hidden(w1, kMlpOffB1, act[0], act[1]);
  uint4 w3[kBfK / 32];
  weights(kMlpOffW3, 16 * (wave & 3), w3);
  __syncthreads();
  hidden(w2, kMlpOffB2, act[1], act[0]);
  __syncthreads();
  // output layer: waves 0..3, 16 rows each
  float y[4];
  const int row = 16 * (wave & 3) + 4 * g;
  if (wave < 4) {   // uniform
    const float* pb = a.master + kMlpOffB3 + row;
    const f4_t acc = infer_rows(w3, act[0] + c * kActLd + 8 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float d = skip_d[c][row + r];
      y[r] = acc[r] + pb[r];
      y[r] += d != 0.f ? skip_r[c][row + r] / d : 0.f;
    }
  }
  if constexpr (BLOCKS) {
    const int64_t b = (int64_t)col0 + c;
    if (wave < 4 && b < a.ncols) {
      const int64_t b2 = b / a.rx1, b1 = b - b2 * a.rx1;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        a.z[b1 + a.rx1 * (row + r + (int64_t)kMlpBlock * b2)] = (double)y[r] * (double)scale[c];
    }
  } else {
    if (wave < 4 && col0 + c < a.ncols) {
      float* dst = a.Y + (int64_t)kMlpOut * (col0 + c) + row;
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[r] = y[r];
    }
  }
}

// T(i, c) = z(b1, i, b2) * inv(c) for the sampled blocks
__global__ __launch_bounds__(256) void targets_kernel(int rx1, int n, int rx2, const double* __restrict__ z,
                                                      int ncols, int64_t b_start, int64_t b_stride,
                                                      const float* __restrict__ inv, float* __restrict__ T) {
  const int lane = threadIdx.x & 63;
  const int64_t col = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  if (col >= ncols) return;
  const int64_t nb = (int64_t)rx1 * rx2;
  const int64_t b = (b_start + col * b_stride) % nb;
  const int b1 = (int)(b % rx1), b2 = (int)(b / rx1);
  T[lane + (int64_t)kMlpOut * col] = (float)(z[b1 + (int64_t)rx1 * (lane + (int64_t)n * b2)] * (double)inv[col]);
}

__global__ void gather_cols_kernel(int rows, int ncols, const int* __restrict__ idx, const float* __restrict__ src,
                                   float* __restrict__ dst) {
  const int64_t total = (int64_t)rows * ncols;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(e % rows);
    const int64_t c = e / rows;
    dst[e] = src[r + (int64_t)rows * idx[c]];
  }
}

__global__ void adam_kernel(int64_t np, float* __restrict__ master, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, float lr, float beta1, float beta2, float eps, float c1, float c2,
                            uint16_t* __restrict__ wbf, float* __restrict__ wr) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < np; e += (int64_t)gridDim.x * blockDim.x) {
    const float ge = g[e];
    const float me = beta1 * m[e] + (1.f - beta1) * ge;
    const float ve = beta2 * v[e] + (1.f - beta2) * ge * ge;
    m[e] = me;
    v[e] = ve;
    const float th = master[e] - lr * (me / c1) / (sqrtf(ve / c2) + eps);
    master[e] = th;
    const uint16_t h = to_bf16(th);
    wbf[e] = h;
    wr[e] = from_bf16(h);
  }
}

int grid_of(int64_t n, int per = 256) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, 4096)); }

void features(int rx1, int n, int rx2, int ra1, int ra2, const double* phi1, const double* A, const double* phi2,
              const double* v, int ncols, int64_t b_start, int64_t b_stride, float* X, float* scale, float* inv,
              hipStream_t st) {
  if (ncols <= 0) return;
  hipLaunchKernelGGL(features_kernel, dim3((unsigned)((ncols + 3) / 4)), dim3(256), 0, st, rx1, n, rx2, ra1, ra2, phi1,
                     A, phi2, v, ncols, b_start, b_stride, X, scale, inv);
  TTF_HIP(hipGetLastError());
}

// Columns per slice of the gradient sums: at most kGradSlices slices, at
// least 128 columns each and whole multiples of 64.
int grad_slice(int M) {
  const int64_t per = std::max<int64_t>(128, ((int64_t)M + kGradSlices - 1) / kGradSlices);
  return (int)((per + 63) / 64 * 64);
}

// Work-groups (and loss partials) of the output layer.
int64_t loss_parts(int M) { return kMlpOut / 32 * (((int64_t)M + 31) / 32); }

// Training workspace for M columns: the loss partials, the gradient slices
// and (floats) X | H1 | H2 | dY | dH2 | dH1.
struct MlpWork {
  float *X, *H1, *H2, *dY, *dH2, *dH1, *slices;
  double* lpart;
};
MlpWork work_for(int M) {
  const size_t per = (size_t)kMlpIn + 4 * kMlpHid + kMlpOut;
  const size_t nl = ((size_t)loss_parts(M) + 1) / 2 * 2;   // keeps what follows on 16 bytes
  const size_t ns = (size_t)kMlpParams * kGradSlices;
  char* base = (char*)arena(kArenaMlp, sizeof(double) * nl + sizeof(float) * (ns + per * (size_t)M));
  MlpWork w{};
  w.lpart = (double*)base;
  w.slices = (float*)(base + sizeof(double) * nl);
  w.X = w.slices + ns;
  w.H1 = w.X + (size_t)kMlpIn * M;
  w.H2 = w.H1 + (size_t)kMlpHid * M;
  w.dY = w.H2 + (size_t)kMlpHid * M;
  w.dH2 = w.dY + (size_t)kMlpOut * M;
  w.dH1 = w.dH2 + (size_t)kMlpHid * M;
  return w;
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

void set_params_device(const float* host) {
  ensure_model();
  hipStream_t st = stream();
  TTF_HIP(hipMemcpyAsync(g_model.master, host, sizeof(float) * (size_t)kMlpParams, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(round_params_kernel, dim3(grid_of(kMlpParams)), dim3(256), 0, st, (int64_t)kMlpParams,
                     g_model.master, g_model.wbf, g_model.wr);
  TTF_HIP(hipGetLastError());
  TTF_HIP(hipMemsetAsync(g_model.am, 0, sizeof(float) * (size_t)kMlpParams, st));
  TTF_HIP(hipMemsetAsync(g_model.av, 0, sizeof(float) * (size_t)kMlpParams, st));
  TTF_HIP(hipStreamSynchronize(st));
  g_model.step = 0;
  g_model.ready = true;
}

// Loss (device) and gradient g of the batch (X, T); X on a 16-byte boundary.
void batch_loss_grad(int M, const float* X, const float* T, MlpWork& w, float* g, double* loss, hipStream_t st) {
  const float* p = g_model.master;
  const float* wr = g_model.wr;
  const double count = (double)kMlpOut * M;
  auto op = [&](int rows, int K, const float* A, int64_t sAi, int64_t sAk, const float* B, float* C) {
    GemmOp<float> o{};
    o.M = rows; o.N = M; o.K = K;
    o.A = A; o.sAi = sAi; o.sAk = sAk;
    o.B = B; o.sBk = 1; o.sBj = K;
    o.C = C;
    return o;
  };
  auto grid = [&](int rows) { return dim3((unsigned)((int64_t)(rows / 32) * (((int64_t)M + 31) / 32))); };
  const dim3 blk(256);
  const float* no = nullptr;
  double* nop = nullptr;
  // forward: H = relu(W^T In + b), and the output layer with the loss
  hipLaunchKernelGGL(train_layer_kernel<0>, grid(kMlpHid), blk, 0, st,
                     op(kMlpHid, kMlpIn, wr + kMlpOffW1, kMlpIn, 1, X, w.H1), p + kMlpOffB1, no, no, 0.f, nop);
  hipLaunchKernelGGL(train_layer_kernel<0>, grid(kMlpHid), blk, 0, st,
                     op(kMlpHid, kMlpHid, wr + kMlpOffW2, kMlpHid, 1, w.H1, w.H2), p + kMlpOffB2, no, no, 0.f, nop);
  hipLaunchKernelGGL(train_layer_kernel<1>, grid(kMlpOut), blk, 0, st,
                     op(kMlpOut, kMlpHid, wr + kMlpOffW3, kMlpHid, 1, w.H2, w.dY), p + kMlpOffB3, X, T,
                     2.0f / ((float)M * (float)kMlpOut), w.lpart);
  // backward: dH = (W D) masked
  hipLaunchKernelGGL(train_back_kernel, grid(kMlpHid), blk, 0, st,
                     op(kMlpHid, kMlpOut, wr + kMlpOffW3, 1, kMlpHid, w.dY, w.dH2), (const float*)w.H2);
  hipLaunchKernelGGL(train_back_kernel, grid(kMlpHid), blk, 0, st,
                     op(kMlpHid, kMlpHid, wr + kMlpOffW2, 1, kMlpHid, w.dH2, w.dH1), (const float*)w.H1);
  WeightGrads a{};
  a.in[0] = X; a.in[1] = w.H1; a.in[2] = w.H2;
  a.d[0] = w.dH1; a.d[1] = w.dH2; a.d[2] = w.dY;
  a.M = M;
  a.slice = grad_slice(M);
  a.nslices = (int)(((int64_t)M + a.slice - 1) / a.slice);
  hipLaunchKernelGGL(weight_grad_kernel, dim3((unsigned)(a.nslices * (kGradTiles + kGradRows))), blk, 0, st, a,
                     w.slices);
  hipLaunchKernelGGL(grad_reduce_kernel, dim3((unsigned)((kMlpParams + 255) / 256 + 1)), blk, 0, st, a.nslices,
                     (const float*)w.slices, g, (int)loss_parts(M), (const double*)w.lpart, 1.0 / count, loss);
  TTF_HIP(hipGetLastError());
}

}  // namespace

bool mlp_ready() { return g_model.ready; }

void mlp_precond(int rx1, int n, int rx2, int ra1, int ra2, const double* phi1, const double* A, const double* phi2,
                 const double* v, double* z, hipStream_t st) {
  TTF_REQUIRE(g_model.ready, "learned preconditioner: no parameters set (ttf_mlp_init / ttf_mlp_set_params)");
  TTF_REQUIRE(n == kMlpBlock, "learned preconditioner: mode size %d, the network is built for %d", n, kMlpBlock);
  const int64_t nb64 = (int64_t)rx1 * rx2;
  TTF_REQUIRE(nb64 <= (1 << 24), "learned preconditioner: %lld blocks", (long long)nb64);
  const int nb = (int)nb64;
  double* Ad = (double*)arena(kArenaMlp, sizeof(double) * 192 * (size_t)ra1 * ra2);
  hipLaunchKernelGGL(diagonals_kernel, dim3((unsigned)(ra1 * ra2)), dim3(192), 0, st, n, ra1, ra2, A, Ad);
  InferArgs a{};
  a.ncols = nb;
  a.w = g_model.wbf;
  a.master = g_model.master;
  a.rx1 = rx1; a.rx2 = rx2; a.ra1 = ra1; a.ra2 = ra2;
  a.phi1 = phi1; a.Ad = Ad; a.phi2 = phi2; a.v = v; a.z = z;
  hipLaunchKernelGGL(infer_kernel<true>, dim3((unsigned)((nb + kInfCols - 1) / kInfCols)), dim3(kInfThreads), 0, st,
                     a);
  TTF_HIP(hipGetLastError());
}

bool mlp_collecting() { return g_sink.active; }

void mlp_collect_pair(int rx1, int n, int rx2, int ra1, int ra2, const double* phi1, const double* A,
                      const double* phi2, const double* v, const double* z, hipStream_t st) {
  if (!g_sink.active || n != kMlpBlock || g_sink.count >= g_sink.cap) return;
  const int64_t nb = (int64_t)rx1 * rx2;
  const int64_t take = std::min<int64_t>({(int64_t)g_sink.per_apply, nb, g_sink.cap - g_sink.count});
  if (take <= 0) return;
  const int64_t stride = std::max<int64_t>(1, nb / take);
  const int64_t start = (int64_t)(splitmix(g_sink.counter) % (uint64_t)nb);
  if (g_sink.inv_cap < take) {
    if (g_sink.inv) TTF_HIP(hipFree(g_sink.inv));
    TTF_HIP(hipMalloc(&g_sink.inv, sizeof(float) * 2 * (size_t)take));
    g_sink.inv_cap = take;
  }
  float* X = g_sink.X + (size_t)kMlpIn * g_sink.count;
  float* T = g_sink.T + (size_t)kMlpOut * g_sink.count;
  features(rx1, n, rx2, ra1, ra2, phi1, A, phi2, v, (int)take, start, stride, X, g_sink.inv + take, g_sink.inv, st);
  hipLaunchKernelGGL(targets_kernel, dim3((unsigned)((take + 3) / 4)), dim3(256), 0, st, rx1, n, rx2, z, (int)take,
                     start, stride, g_sink.inv, T);
  TTF_HIP(hipGetLastError());
  g_sink.count += take;
}

}  // namespace ttf

using namespace ttf;

extern "C" {

long ttf_mlp_param_count(void) { return (long)kMlpParams; }

int ttf_mlp_init(unsigned seed) {
  return guarded([&] {
    std::vector<float> p((size_t)kMlpParams, 0.f);
    uint64_t s = 0x1234abcdull ^ ((uint64_t)seed << 17);
    auto fill = [&](int64_t off, int fan_in, int64_t cnt) {
      const double lim = 1.0 / std::sqrt((double)fan_in);
      for (int64_t e = 0; e < cnt; ++e) {
        const double u = (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
        p[(size_t)(off + e)] = (float)((2.0 * u - 1.0) * lim);
      }
    };
    fill(kMlpOffW1, kMlpIn, (int64_t)kMlpIn * kMlpHid);
    fill(kMlpOffW2, kMlpHid, (int64_t)kMlpHid * kMlpHid);
    // W3 and all biases start at zero: the untrained network is the
    // point-Jacobi solve of each block
    set_params_device(p.data());
  });
}

int ttf_mlp_set_params(const float* params) {
  return guarded([&] {
    TTF_REQUIRE(params != nullptr, "ttf_mlp_set_params: null parameters");
    set_params_device(params);
  });
}

int ttf_mlp_get_params(float* params) {
  return guarded([&] {
    TTF_REQUIRE(g_model.ready, "ttf_mlp_get_params: no parameters set");
    hipStream_t st = stream();
    read_back(params, g_model.master, sizeof(float) * (size_t)kMlpParams, st);
  });
}

int ttf_mlp_forward(int M, const float* X, float* Y) {
  return guarded([&] {
    TTF_REQUIRE(g_model.ready, "ttf_mlp_forward: no parameters set");
    TTF_REQUIRE(M >= 0, "ttf_mlp_forward: M=%d", M);
    if (M == 0) return;
    InferArgs a{};
    a.ncols = M;
    a.w = g_model.wbf;
    a.master = g_model.master;
    a.X = X;
    a.Y = Y;
    hipLaunchKernelGGL(infer_kernel<false>, dim3((unsigned)(((int64_t)M + kInfCols - 1) / kInfCols)),
                       dim3(kInfThreads), 0, stream(), a);
    TTF_HIP(hipGetLastError());
  });
}

int ttf_mlp_loss_grad(int M, const float* X, const float* T, double* loss, float* grad) {
  return guarded([&] {
    TTF_REQUIRE(g_model.ready, "ttf_mlp_loss_grad: no parameters set");
    TTF_REQUIRE(M > 0, "ttf_mlp_loss_grad: M=%d", M);
    hipStream_t st = stream();
    MlpWork w = work_for(M);
    float* g = (float*)arena(kArenaMlp2, sizeof(float) * (size_t)kMlpParams + sizeof(double) * 2);
    double* out = (double*)(g + kMlpParams + (kMlpParams & 1));
    if ((reinterpret_cast<uintptr_t>(X) & 15) != 0) {
      TTF_HIP(hipMemcpyAsync(w.X, X, sizeof(float) * (size_t)kMlpIn * M, hipMemcpyDeviceToDevice, st));
      X = w.X;
    }
    batch_loss_grad(M, X, T, w, g, out, st);
    TTF_HIP(hipMemcpyAsync(loss, out, sizeof(double), hipMemcpyDeviceToHost, st));
    if (grad) read_back(grad, g, sizeof(float) * (size_t)kMlpParams, st);
  });
}

int ttf_mlp_train(long nsamples, const float* X, const float* T, int epochs, int batch, float lr, unsigned seed,
                  double* loss_hist, int hist_cap, int* hist_len) {
  return guarded([&] {
    TTF_REQUIRE(g_model.ready, "ttf_mlp_train: no parameters set (ttf_mlp_init first)");
    TTF_REQUIRE(nsamples > 0 && epochs >= 0 && batch > 0 && lr > 0.f, "ttf_mlp_train: bad arguments");
    TTF_REQUIRE(nsamples <= (1L << 30), "ttf_mlp_train: %ld samples", nsamples);
    hipStream_t st = stream();
    const int B = (int)std::min<long>(batch, nsamples);
    const long nbat = nsamples / B;
    MlpWork w = work_for(B);
    float* g = (float*)arena(kArenaMlp2, sizeof(float) * (size_t)kMlpParams + sizeof(double) * (nbat + 1) +
                                             sizeof(int) * (size_t)nsamples + 64);
    double* losses = (double*)(g + kMlpParams + (kMlpParams & 1));
    int* idx = (int*)(losses + nbat + 1);
    float* Tb = (float*)arena(kArenaMlp3, sizeof(float) * (size_t)kMlpOut * B);   // batch targets
    std::vector<int> perm((size_t)nsamples);
    for (long i = 0; i < nsamples; ++i) perm[(size_t)i] = (int)i;
    uint64_t s = 0x5eedull ^ ((uint64_t)seed << 21);
    std::vector<double> hl((size_t)nbat);
    if (hist_len) *hist_len = 0;
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    for (int e = 0; e < epochs; ++e) {
      for (long i = nsamples - 1; i > 0; --i) std::swap(perm[(size_t)i], perm[(size_t)(splitmix(s) % (uint64_t)(i + 1))]);
      TTF_HIP(hipMemcpyAsync(idx, perm.data(), sizeof(int) * (size_t)nsamples, hipMemcpyHostToDevice, st));
      for (long bi = 0; bi < nbat; ++bi) {
        const int* ib = idx + bi * B;
        hipLaunchKernelGGL(gather_cols_kernel, dim3(grid_of((int64_t)kMlpIn * B)), dim3(256), 0, st, kMlpIn, B, ib, X, w.X);
        hipLaunchKernelGGL(gather_cols_kernel, dim3(grid_of((int64_t)kMlpOut * B)), dim3(256), 0, st, kMlpOut, B, ib, T,
                           Tb);
        batch_loss_grad(B, w.X, Tb, w, g, losses + bi, st);
        ++g_model.step;
        const float c1 = 1.f - std::pow(beta1, (float)g_model.step);
        const float c2 = 1.f - std::pow(beta2, (float)g_model.step);
        hipLaunchKernelGGL(adam_kernel, dim3(grid_of(kMlpParams)), dim3(256), 0, st, (int64_t)kMlpParams, g_model.master,
                           g, g_model.am, g_model.av, lr, beta1, beta2, eps, c1, c2, g_model.wbf, g_model.wr);
        TTF_HIP(hipGetLastError());
      }
      read_back(hl.data(), losses, sizeof(double) * (size_t)nbat, st);   // idx is rewritten by the next epoch
      if (loss_hist && hist_len && *hist_len < hist_cap) {
        double m = 0.0;
        for (double v : hl) m += v;
        loss_hist[(*hist_len)++] = m / (double)std::max<long>(nbat, 1);
      }
    }
    TTF_HIP(hipStreamSynchronize(st));
  });
}

int ttf_mlp_features(int rx1, int n, int rx2, int ra1, int ra2, const double* phi1, const double* A,
                     const double* phi2, const double* v, float* X, float* scale) {
  return guarded([&] {
    TTF_REQUIRE(n == kMlpBlock, "ttf_mlp_features: mode size %d, features are built for %d", n, kMlpBlock);
    TTF_REQUIRE(rx1 > 0 && rx2 > 0 && ra1 > 0 && ra2 > 0, "ttf_mlp_features: invalid sizes");
    features(rx1, n, rx2, ra1, ra2, phi1, A, phi2, v, rx1 * rx2, 0, 1, X, scale, nullptr, stream());
  });
}

int ttf_mlp_precond(int rx1, int n, int rx2, int ra1, int ra2, const double* phi1, const double* A,
                    const double* phi2, const double* v, double* z) {
  return guarded([&] {
    TTF_REQUIRE(rx1 > 0 && rx2 > 0 && ra1 > 0 && ra2 > 0, "ttf_mlp_precond: invalid sizes");
    mlp_precond(rx1, n, rx2, ra1, ra2, phi1, A, phi2, v, z, stream());
  });
}

int ttf_mlp_collect_begin(long capacity, int per_apply) {
  return guarded([&] {
    TTF_REQUIRE(capacity > 0 && per_apply > 0, "ttf_mlp_collect_begin: bad arguments");
    if (g_sink.X) TTF_HIP(hipFree(g_sink.X));
    if (g_sink.T) TTF_HIP(hipFree(g_sink.T));
    g_sink.X = g_sink.T = nullptr;
    TTF_HIP(hipMalloc(&g_sink.X, sizeof(float) * (size_t)kMlpIn * capacity));
    TTF_HIP(hipMalloc(&g_sink.T, sizeof(float) * (size_t)kMlpOut * capacity));
    g_sink.cap = capacity;
    g_sink.count = 0;
    g_sink.per_apply = per_apply;
    g_sink.counter = 0x9e37ull;
    g_sink.active = true;
  });
}

int ttf_mlp_collect_end(long* count) {
  return guarded([&] {
    g_sink.active = false;
    TTF_HIP(hipStreamSynchronize(stream()));
    if (count) *count = (long)g_sink.count;
  });
}

int ttf_mlp_collected(float** X, float** T, long* count) {
  return guarded([&] {
    TTF_REQUIRE(X && T && count, "ttf_mlp_collected: null arguments");
    *X = g_sink.X;
    *T = g_sink.T;
    *count = (long)g_sink.count;
  });
}

}  // extern "C"
