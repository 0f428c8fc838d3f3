// The local matvec (ttals.f90:9-83) of small and middle ranks with narrow
// modes in one launch, in all four element types:
//   T1(b1,j,a2)  = sum_b2 x(b1,j,b2) phi2(b2,a2,c2)
//   T2(b1,a1,i)  = sum_{j,a2} A(a1,i,j,a2) T1(b1,j,a2)
//   y(c1,i,c2)   = sum_{b1,a1} phi1(c1,b1,a1) T2(b1,a1,i)
// One work-group of eight waves per (vector, right-interface index c2), the
// intermediates in LDS.  For one c2 the products have only ra2 and n
// columns, which would fill a fraction of a 16-column matrix-core tile, and
// the vector units multiply f64 at the matrix cores' rate: a thread keeps
// one row's ra2 (or n) sums in registers, the narrow operand reaches all
// lanes of a wave at once (phi2 by scalar loads, T2 by LDS broadcasts), and
// the waves left over by the rows split the sum, their parts added in a
// fixed order.
#include "contract.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace ttf {

namespace {

constexpr int kNT = 512;
constexpr int kMaxCols = 8;          // ra2 and n at most
constexpr int kInFlight = 8;         // loads of the wide operand per round trip
constexpr size_t kLdsBytes = 96 * 1024;

template <typename T>
struct SmallArgs {
  int rx1, m, rx2, ry1, n, ry2, ra1, ra2;
  const T* phi1;
  const T* A;      // nullptr: T2 = T1 (m = n = 1, ra1 = ra2)
  const T* phi2;
  const T* x;
  int64_t ldx;
  T* y;
  int64_t ldy;
};

__device__ __forceinline__ double mac(double c, double a, double b) { return fma(a, b, c); }
__device__ __forceinline__ float mac(float c, float a, float b) { return fmaf(a, b, c); }
__device__ __forceinline__ hipDoubleComplex mac(hipDoubleComplex c, hipDoubleComplex a, hipDoubleComplex b) {
  return make_hipDoubleComplex(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ hipFloatComplex mac(hipFloatComplex c, hipFloatComplex a, hipFloatComplex b) {
  return make_hipFloatComplex(fmaf(a.x, b.x, fmaf(-a.y, b.y, c.x)), fmaf(a.x, b.y, fmaf(a.y, b.x, c.y)));
}
__device__ __forceinline__ double plus(double a, double b) { return a + b; }
__device__ __forceinline__ float plus(float a, float b) { return a + b; }
__device__ __forceinline__ hipDoubleComplex plus(hipDoubleComplex a, hipDoubleComplex b) {
  return make_hipDoubleComplex(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ hipFloatComplex plus(hipFloatComplex a, hipFloatComplex b) {
  return make_hipFloatComplex(a.x + b.x, a.y + b.y);
}
template <typename T> __device__ __forceinline__ T zero() { return T(0); }
template <> __device__ __forceinline__ hipDoubleComplex zero() { return make_hipDoubleComplex(0.0, 0.0); }
template <> __device__ __forceinline__ hipFloatComplex zero() { return make_hipFloatComplex(0.f, 0.f); }

// Threads per group of the rows x K split: whole waves, at most the block.
__host__ __device__ inline int row_threads(int rows) {
  const int r = (rows + 63) / 64 * 64;
  return r < kNT ? r : kNT;
}

// part[(kg C + c) rows + r] = sum over group kg's share of k of W(r, k)
// B(k, c), c < C, for the wide W (rows x K, ld rows, global) and the narrow
// B given by at(k, c); groups of row_threads(rows) threads.
template <int C, typename T, typename At>
__device__ __forceinline__ void narrow_product(const T* __restrict__ W, int rows, int K, T* part, At at) {
  const int rt = row_threads(rows), groups = kNT / rt;
  const int kg = __builtin_amdgcn_readfirstlane((int)threadIdx.x / rt);
  if (kg >= groups) return;   // uniform over the wave
  const int per = (K + groups - 1) / groups;
  const int k0 = kg * per, k1 = min(K, k0 + per);
  for (int r = (int)threadIdx.x - kg * rt; r < (rows + rt - 1) / rt * rt; r += rt) {
    const T* w = W + min(r, rows - 1);
    T acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = zero<T>();
    int k = k0;
    for (; k + kInFlight <= k1; k += kInFlight) {
      T v[kInFlight];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) v[u] = w[(int64_t)rows * (k + u)];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = mac(acc[c], v[u], at(k + u, c));
    }
    if (k < k1) {   // the rest, its loads clamped and its products skipped
      T v[kInFlight];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) v[u] = w[(int64_t)rows * min(k + u, k1 - 1)];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u)
        if (k + u < k1) {   // uniform
#pragma unroll
          for (int c = 0; c < C; ++c) acc[c] = mac(acc[c], v[u], at(k + u, c));
        }
    }
    if (r < rows) {
#pragma unroll
      for (int c = 0; c < C; ++c) part[((int64_t)kg * C + c) * rows + r] = acc[c];
    }
  }
}

template <int C, typename T>
__device__ __forceinline__ T group_sum(const T* part, int rows, int groups, int c, int r) {
  T s = part[(int64_t)c * rows + r];
  for (int g = 1; g < groups; ++g) s = plus(s, part[((int64_t)g * C + c) * rows + r]);
  return s;
}

// A2 >= ra2 and N >= n columns; columns past them repeat the last one and
// are dropped.
template <typename T, int A2, int N>
__global__ __launch_bounds__(kNT) void bfun3_small_kernel(SmallArgs<T> a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x;
  const int c2 = blockIdx.x % a.ry2, v = blockIdx.x / a.ry2;
  const int R1 = a.rx1 * a.m, K3 = a.rx1 * a.ra1;
  T* T1 = reinterpret_cast<T*>(lds);       // (b1, j, a2)
  T* T2 = T1 + R1 * a.ra2;                 // T2[(b1 + rx1 a1) N + i]
  T* part = T2 + K3 * N;
  {
    const T* __restrict__ p2 = a.phi2 + (int64_t)a.rx2 * a.ra2 * c2;
    const int rx2 = a.rx2, last = a.ra2 - 1;
    narrow_product<A2>(a.x + v * a.ldx, R1, a.rx2, part,
                       [&](int k, int c) { return p2[k + rx2 * (c < last ? c : last)]; });
  }
  __syncthreads();
  {
    const int groups = kNT / row_threads(R1);
    for (int e = tid; e < R1 * a.ra2; e += kNT) {
      const int c = e / R1;
      T1[e] = group_sum<A2>(part, R1, groups, c, e - c * R1);
    }
  }
  __syncthreads();
  for (int e = tid; e < K3 * N; e += kNT) {
    const int i = e / K3, k = e - i * K3;
    T s = zero<T>();
    if (i < a.n) {
      if (a.A == nullptr) {
        s = T1[k];
      } else {
        const int a1 = k / a.rx1, b1 = k - a1 * a.rx1;
        const T* Ai = a.A + a1 + a.ra1 * i;
        for (int q = 0; q < a.m * a.ra2; ++q) s = mac(s, Ai[(int64_t)a.ra1 * a.n * q], T1[b1 + a.rx1 * q]);
      }
    }
    T2[k * N + i] = s;
  }
  __syncthreads();
  narrow_product<N>(a.phi1, a.ry1, K3, part, [&](int k, int c) { return T2[k * N + c]; });
  __syncthreads();
  {
    T* y = a.y + v * a.ldy + (int64_t)a.ry1 * a.n * c2;
    const int groups = kNT / row_threads(a.ry1);
    for (int e = tid; e < a.ry1 * a.n; e += kNT) {
      const int i = e / a.ry1;
      y[e] = group_sum<N>(part, a.ry1, groups, i, e - i * a.ry1);
    }
  }
}

int bucket(int c) { return c <= 2 ? 2 : c <= 3 ? 3 : c <= 5 ? 5 : 8; }

template <typename T>
size_t lds_need(const Shape& s, int A2, int N) {
  const int64_t R1 = (int64_t)s.rx1 * s.m, K3 = (int64_t)s.rx1 * s.ra1;
  const int64_t g1 = kNT / row_threads((int)std::min<int64_t>(R1, kNT)), g3 = kNT / row_threads(s.ry1);
  return sizeof(T) * (size_t)(R1 * s.ra2 + K3 * N + std::max(g1 * A2 * R1, g3 * N * s.ry1));
}

bool small_enabled() {
  static const bool on = [] {
    const char* e = std::getenv("TTF_BFUN3_SMALL");
    return !(e && std::atoi(e) == 0);
  }();
  return on;
}

// Where the one launch is the faster way: both ways' times estimated in us.
//
// A work-group streams its vector and all of phi1 through one CU, so its
// time goes with the elements it loads, its multiply-adds (columns as padded)
// and those of the middle stage, whose operands come one by one; with more
// than 256 work-groups times the rounds.  A limit on the launch's total alone
// let work-groups of any size through: (left rank, n, right rank, operator
// rank) = (512, 2, 2, 3) in f64 took 92 us where the other way takes 18, (512,
// 2, 1, 5) in f32 135 against 17.
//
// The other way in real types is the fused kernel or a chain of tuned
// products: a few launches, and more with the total of multiply-adds.  In
// complex types it is three products of fixed tiles (zgemm_plan), each the
// chain of its K or rounds of it.
//
// The constants are least squares over 4300 shapes of the four types (ranks
// 1 to 512, both sides equal or not, modes and operator ranks 1 to 8, 1 to 8
// vectors; rms error 14 to 17 % for this kernel, 6 % for the complex chains)
// and hold up to a total of multiply-adds, past which the matrix cores' tiles
// are the rule.  Against the faster way of each shape below it the choice
// loses 0.4 % on average in f64, 0.3 in f32, 0.1 in c128 and 0.4 in c64 (the
// total alone: 22, 25, 3 and 11 %); at worst it takes 1.3 times the other
// way's time in real types, 1.2 in c128 and 1.6 in c64.  Measured (us, other way
// -> this), operator rank 5, n = 2, one vector unless said, ranks on both
// sides or left x right:
//   f64   2: 11.9 -> 4.6; 64: 16.5 -> 8.5; 128: 29.2 -> 18.6; 128 x 4: 22.8 ->
//         15.0; 4 x 400, operator rank 3: 24.3 -> 11.4; other way: 256 x 4: 27.1
//         against 42.8
//   f32   64: 23.6 -> 7.0; 128: 27.8 -> 13.5; 128 x 4: 23.0 -> 10.3; other way:
//         400 x 4, operator rank 3: 21.0 against 41.1
//   c128  64: 21.9 -> 10.2; 128 x 4: 19.8 -> 15.7; other way: 256 x 1, operator
//         rank 3: 19.6 against 27.1
//   c64   64: 17.9 -> 9.3; 128 x 64: 23.7 -> 18.4; other way: 512 x 2, operator
//         rank 3: 29.6 against 101
struct SmallCost {
  double start, load, mac, mid, round;
};
template <typename T> constexpr SmallCost kSmall = {5.3, 7.3e-5, 1.5e-5, 1.2e-4, 1.9};
template <> constexpr SmallCost kSmall<float> = {5.2, 3.3e-5, 1.4e-5, 5.7e-5, 1.3};
template <> constexpr SmallCost kSmall<hipDoubleComplex> = {5.7, 0.0, 5.7e-5, 1.6e-4, 2.4};
template <> constexpr SmallCost kSmall<hipFloatComplex> = {5.6, 3.7e-5, 3.2e-5, 1.1e-4, 2.0};

// A complex product: `k32` per k of a 32-wide tile's chain, `more32` of it for
// each further round, `k64` per k and round of 64-wide tiles, `split` for a
// second launch, `wgs` per 256 work-groups.
struct ZCost {
  double start, k32, more32, k64, split, wgs;
};
template <typename T> constexpr ZCost kZ = {3.0, 0.068, 0.068, 0.16, 3.2, 2.2};
template <> constexpr ZCost kZ<hipFloatComplex> = {3.0, 0.046, 0.024, 0.10, 2.7, 1.1};

template <typename T>
double zgemm_us(int M, int N, int K, int nbatch) {
  const ZCost c = kZ<T>;
  const ZPlan p = zgemm_plan(M, N, K, nbatch);
  const double per = std::ceil((double)K / p.ks), rounds = (double)p.tiles * nbatch * p.ks / 256;
  const double sums = p.bm == 32 ? (c.k32 + c.more32 * std::max(0.0, rounds - 1)) * per : c.k64 * per * std::ceil(rounds);
  return c.start + sums + (p.ks > 1 ? c.split : 0.0) + c.wgs * rounds;
}

template <typename T> constexpr double kMostMacs = 1.2e8;
template <> constexpr double kMostMacs<double> = 5e7;
template <> constexpr double kMostMacs<hipDoubleComplex> = 6e7;

template <typename T>
bool faster_small(const Shape& s, int nvec, bool core, int A2, int N) {
  const double groups = (double)s.ry2 * nvec, K3 = (double)s.rx1 * s.ra1;
  const double wide1 = (double)s.rx1 * s.m * s.rx2, wide3 = s.ry1 * K3, macs = wide1 * A2 + wide3 * N;
  if (macs * groups > kMostMacs<T>) return false;
  if (groups > 65535) return true;   // the chains take no more products in one batch
  const SmallCost c = kSmall<T>;
  const double own = c.load * (wide1 + wide3) + c.mac * macs + (core ? c.mid * K3 * N * s.m * s.ra2 : 0.0);
  const double rounds = std::max(1.0, groups / 256);
  const double small = c.start + own * rounds + c.round * (rounds - 1);
  if (std::is_same<T, double>::value) return small <= 17.5 + 1.5e-7 * macs * groups;
  if (std::is_same<T, float>::value) return small <= 14.5 + 8e-8 * macs * groups;
  double other = zgemm_us<T>(s.rx1 * s.m, s.ra2 * s.ry2, s.rx2, nvec);
  if (core) other += zgemm_us<T>(s.rx1, s.ra1 * s.n, s.m * s.ra2, s.ry2 * nvec);
  return small <= other + zgemm_us<T>(s.ry1, s.n * s.ry2, s.rx1 * s.ra1, nvec);
}

template <typename T, int A2, int N>
void launch_n(const SmallArgs<T>& a, unsigned grid, size_t lds, hipStream_t st) {
  static std::atomic<bool> attr{false};   // concurrent first calls only repeat the call
  if (!attr) {
    TTF_HIP(hipFuncSetAttribute((const void*)bfun3_small_kernel<T, A2, N>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes));
    attr = true;
  }
  hipLaunchKernelGGL((bfun3_small_kernel<T, A2, N>), dim3(grid), dim3(kNT), lds, st, a);
}

template <typename T, int A2>
void launch(const SmallArgs<T>& a, int N, unsigned grid, size_t lds, hipStream_t st) {
  switch (N) {
    case 2: launch_n<T, A2, 2>(a, grid, lds, st); break;
    case 3: launch_n<T, A2, 3>(a, grid, lds, st); break;
    case 5: launch_n<T, A2, 5>(a, grid, lds, st); break;
    default: launch_n<T, A2, 8>(a, grid, lds, st); break;
  }
}

}  // namespace

template <typename T>
bool bfun3_small_fits(const Shape& s, int nvec, bool core) {
  if (!small_enabled() || nvec < 1 || s.ra2 > kMaxCols || s.n > kMaxCols) return false;
  const int64_t R1 = (int64_t)s.rx1 * s.m, K3 = (int64_t)s.rx1 * s.ra1;
  if (R1 > 2048 || K3 > 4096 || s.ry1 > 2048) return false;
  const int A2 = bucket(s.ra2), N = bucket(s.n);
  return (int64_t)s.ry2 * nvec <= 0x7fffffff / kNT && lds_need<T>(s, A2, N) <= kLdsBytes &&
         faster_small<T>(s, nvec, core, A2, N);
}

template <typename T>
bool bfun3_small(const Shape& s, int nvec, const T* phi1, const T* A, const T* phi2, const T* x, int64_t ldx, T* y,
                 int64_t ldy, hipStream_t st) {
  if (!bfun3_small_fits<T>(s, nvec, A != nullptr)) return false;
  const int A2 = bucket(s.ra2), N = bucket(s.n);
  const size_t lds = lds_need<T>(s, A2, N);
  SmallArgs<T> a{s.rx1, s.m, s.rx2, s.ry1, s.n, s.ry2, s.ra1, s.ra2, phi1, A, phi2, x, ldx, y, ldy};
  const unsigned grid = (unsigned)(s.ry2 * nvec);
  switch (A2) {
    case 2: launch<T, 2>(a, N, grid, lds, st); break;
    case 3: launch<T, 3>(a, N, grid, lds, st); break;
    case 5: launch<T, 5>(a, N, grid, lds, st); break;
    default: launch<T, 8>(a, N, grid, lds, st); break;
  }
  TTF_HIP(hipGetLastError());
  return true;
}

template bool bfun3_small_fits<double>(const Shape&, int, bool);
template bool bfun3_small_fits<float>(const Shape&, int, bool);
template bool bfun3_small_fits<hipDoubleComplex>(const Shape&, int, bool);
template bool bfun3_small_fits<hipFloatComplex>(const Shape&, int, bool);
template bool bfun3_small<double>(const Shape&, int, const double*, const double*, const double*, const double*,
                                  int64_t, double*, int64_t, hipStream_t);
template bool bfun3_small<float>(const Shape&, int, const float*, const float*, const float*, const float*, int64_t,
                                 float*, int64_t, hipStream_t);
template bool bfun3_small<hipDoubleComplex>(const Shape&, int, const hipDoubleComplex*, const hipDoubleComplex*,
                                            const hipDoubleComplex*, const hipDoubleComplex*, int64_t,
                                            hipDoubleComplex*, int64_t, hipStream_t);
template bool bfun3_small<hipFloatComplex>(const Shape&, int, const hipFloatComplex*, const hipFloatComplex*,
                                           const hipFloatComplex*, const hipFloatComplex*, int64_t,
                                           hipFloatComplex*, int64_t, hipStream_t);

}  // namespace ttf
