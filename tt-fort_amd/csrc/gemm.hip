// GEMM launchers: runtime autotuning of tile shape and split-K, and the
// small-panel kernel for products with a short K and a narrow shared B.
#include "gemm_mfma.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace ttf {

// ---------------------------------------------------------------- small panel
// C[b](i,j) = alpha sum_k A[b](i,k) B(k,j) + beta C[b](i,j) with K <= 64,
// N <= 32, B shared by all batches and A, C row-contiguous (sAi = sCi = 1).
// This is the shape of the middle bfun3 / phi stage for small mode sizes
// (K = m*ra2, N = ra1*n): memory-bound, so one thread per row i of one batch
// accumulates all N outputs while B sits in LDS.
// NN is N rounded up to the kernel's column bucket; B is zero-padded in LDS
// to (64 x NN) so the inner loops carry no guards.
template <typename T, int NN>
__global__ __launch_bounds__(256) void panel_kernel(GemmOp<T> op) {
  __shared__ T Bs[64][NN];
  const int K = op.K, N = op.N;
  for (int t = threadIdx.x; t < 64 * NN; t += blockDim.x) {
    int k = t / NN, j = t % NN;
    Bs[k][j] = (k < K && j < N) ? op.B[k * op.sBk + j * op.sBj] : T(0);
  }
  __syncthreads();
  const int64_t total = (int64_t)op.M * op.nbatch;
  // 32-bit unsigned index arithmetic whenever it fits (a 64-bit division is
  // a long instruction sequence on the vector ALU)
  const bool narrow = total <= 0x7fffffff;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < total;
       g += (int64_t)gridDim.x * blockDim.x) {
    int i, b;
    if (narrow) {
      i = (int)((unsigned)g % (unsigned)op.M);
      b = (int)((unsigned)g / (unsigned)op.M);
    } else {
      i = (int)(g % op.M);
      b = (int)(g / op.M);
    }
    int b0 = 0, b1 = b;
    if (op.nb0 != 1) {
      b0 = (int)((unsigned)b % (unsigned)op.nb0);
      b1 = (int)((unsigned)b / (unsigned)op.nb0);
    }
    const T* a = op.A + b0 * op.sAb0 + b1 * op.sAb1 + i;
    T* c = op.C + b0 * op.sCb0 + b1 * op.sCb1 + i;
    T acc[NN];
#pragma unroll
    for (int j = 0; j < NN; ++j) acc[j] = T(0);
    // the kernel is bound by memory latency: each chunk issues its 8 loads
    // together before the arithmetic that consumes them
    for (int k0 = 0; k0 < K; k0 += 8) {
      T av[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) av[u] = (k0 + u < K) ? a[(k0 + u) * op.sAk] : T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int j = 0; j < NN; ++j) acc[j] += av[u] * Bs[k0 + u][j];
    }
    // with beta != 0 every C element of the row is loaded before any is
    // used (one load under its own condition, used inside it, becomes a
    // branch with a full wait per column); columns past N read column 0
    T cv[NN];
    if (op.beta != T(0)) {
#pragma unroll
      for (int j = 0; j < NN; ++j) cv[j] = c[(j < N ? j : 0) * op.sCj];
    }
#pragma unroll
    for (int j = 0; j < NN; ++j)
      if (j < N) {
        T v = op.alpha * acc[j];
        if (op.beta != T(0)) v += op.beta * cv[j];
        c[j * op.sCj] = v;
      }
  }
}

template <typename T>
static bool panel_eligible(const GemmOp<T>& op) {
  return op.K <= 64 && op.N <= 32 && op.sAi == 1 && op.sCi == 1 && op.sBb0 == 0 &&
         op.sBb1 == 0 && (int64_t)op.M * op.nbatch >= 256;
}

// ---------------------------------------------------------------- autotuner
// Set while this thread records a stream capture: untuned shapes then take
// the heuristic configuration instead of timing runs (not recorded, so a
// later eager call still tunes them).
static thread_local bool t_no_tune = false;
void gemm_no_tuning(bool on) { t_no_tune = on; }

// A tile shape (kTiles below) and the split-K factor ks.
struct Cfg {
  int bm, bn, ks;
};

// The tile shapes that launch_tiles instantiates.  `rate`: the share of the
// matrix cores' rate that a chip full of such work-groups reaches with a
// long K, in hundredths (f64, 16-byte loads), which orders the candidates;
// the best three are timed, so the order need only be about right.  It is
// used for f32 and for element-wise loads too.  Measured there, a product of
// 8192 x 1024 x 1024, TFLOP/s in the order of the table:
//   f64, 16 bytes   55.5 48.8 51.3 55.6 54.0 44.4 32.9
//   f64, elements   52.5 50.0 47.9 53.5 52.6 47.8 36.3
//   f32, 16 bytes   85.6 89.5 90.0 92.3 87.9 59.4 45.6
//   f32, elements   85.1 79.6 79.2 84.3 75.8 70.1 54.1
struct Tile {
  int bm, bn, threads, rate;
};
static const Tile kTiles[] = {{128, 64, 256, 92}, {64, 96, 512, 90}, {64, 80, 256, 84}, {64, 64, 256, 86},
                              {64, 32, 256, 82},  {32, 32, 256, 70}, {32, 16, 64, 45}};

// Whether an operand's offsets inside a tile (at most 128 rows and 64 of k)
// fit 32 bits.
template <typename T>
static bool operand_near(int64_t s_row, int64_t s_k) {
  const int64_t most = ((int64_t)1 << 32) / (int64_t)sizeof(T);
  return s_row >= 0 && s_k >= 0 && s_row < most && s_k < most && 128 * s_row + 64 * s_k < most;
}

// Whether an operand (rows x K, strides s_row, s_k, batch strides) can be
// read 16 bytes at a time along its contiguous direction: pointer, other
// strides and the extent of that direction all whole multiples of 16 bytes.
template <typename T>
static bool operand_aligned(const T* p, int64_t s_row, int64_t s_k, int64_t sb0, int64_t sb1, int rows, int K) {
  constexpr int V = 16 / (int)sizeof(T);
  if ((reinterpret_cast<uintptr_t>(p) & 15) != 0 || sb0 % V != 0 || sb1 % V != 0) return false;
  if (s_row == 1) return s_k % V == 0 && rows % V == 0;
  return s_k == 1 && s_row % V == 0 && K % V == 0;
}

template <typename T>
static LoadMode load_mode(const GemmOp<T>& op) {
  if (!operand_near<T>(op.sAi, op.sAk) || !operand_near<T>(op.sBj, op.sBk)) return kWide;
  const bool va = operand_aligned(op.A, op.sAi, op.sAk, op.sAb0, op.sAb1, op.M, op.K);
  const bool vb = operand_aligned(op.B, op.sBj, op.sBk, op.sBb0, op.sBb1, op.N, op.K);
  return va && vb ? kVecBoth : (va ? kVecA : (vb ? kVecB : kScalar));
}

struct Key {
  int type, M, N, K, nbatch, flags;
  bool operator==(const Key& o) const {
    return type == o.type && M == o.M && N == o.N && K == o.K && nbatch == o.nbatch &&
           flags == o.flags;
  }
};
struct KeyHash {
  size_t operator()(const Key& k) const {
    size_t h = 1469598103934665603ull;
    for (int v : {k.type, k.M, k.N, k.K, k.nbatch, k.flags}) h = (h ^ (size_t)v) * 1099511628211ull;
    return h;
  }
};

template <typename T> static int type_id();
template <> int type_id<double>() { return 0; }
template <> int type_id<float>() { return 1; }

// A product's key: sizes, which directions are contiguous, and how its tiles
// read their operands, since one tile's time differs between the modes (both
// operands in 16-byte loads is 0, the mode of tables without one).
template <typename T>
static Key key_of(const GemmOp<T>& op) {
  const LoadMode m = load_mode(op);
  const int mode = m == kVecBoth ? 0 : (m == kVecA ? 1 : (m == kVecB ? 2 : (m == kScalar ? 3 : 4)));
  return {type_id<T>(), op.M, op.N, op.K, op.nbatch,
          (op.sAi == 1 ? 1 : 0) | (op.sBj == 1 ? 2 : 0) | (op.sCi == 1 ? 4 : 0) | (mode << 3)};
}

namespace {
std::mutex g_tune_mu;
std::unordered_map<Key, Cfg, KeyHash> g_tuned;
std::atomic<int> g_autotune{-1};   // -1: read TTF_AUTOTUNE on first use
long g_tune_count = 0;
bool g_table_loaded = false;
}  // namespace

// Persistent tuning table: when TTF_TUNE_FILE names a file, its entries
// ("type M N K nbatch flags bm bk ks bn" per line; a line without bn, or
// with bn 0, means square tiles, and bk is kept for older tables and not
// used) are loaded on first use and
// every newly tuned shape is appended, so that separate processes (a timed
// run and its counter-collection reruns, or successive jobs) launch the same
// configuration for the same product.  Called with g_tune_mu held.
static const char* tune_file() {
  const char* f = std::getenv("TTF_TUNE_FILE");
  return (f && f[0]) ? f : nullptr;
}

static int splitk_rule(int M, int N, int K, int nbatch);

static void load_tune_table() {
  if (g_table_loaded) return;
  g_table_loaded = true;
  const char* path = tune_file();
  if (!path) return;
  FILE* fp = std::fopen(path, "r");
  if (!fp) return;
  char line[256];
  while (std::fgets(line, sizeof(line), fp)) {
    Key k{};
    Cfg c{};
    int bk = 0;
    const int got = std::sscanf(line, "%d %d %d %d %d %d %d %d %d %d", &k.type, &k.M, &k.N, &k.K, &k.nbatch,
                                &k.flags, &c.bm, &bk, &c.ks, &c.bn);
    if (got == 9 || (got == 10 && c.bn == 0)) c.bn = c.bm;
    bool valid = false;
    for (const Tile& t : kTiles) valid = valid || (t.bm == c.bm && t.bn == c.bn);
    if ((got == 9 || got == 10) && valid) {
      c.ks = splitk_rule(k.M, k.N, k.K, k.nbatch);   // the split is never tuned
      g_tuned[k] = c;
    }
  }
  std::fclose(fp);
}

static void record_tuned(const Key& k, const Cfg& c) {
  const char* path = tune_file();
  if (!path) return;
  FILE* fp = std::fopen(path, "a");
  if (!fp) return;
  std::fprintf(fp, "%d %d %d %d %d %d %d %d %d %d\n", k.type, k.M, k.N, k.K, k.nbatch, k.flags, c.bm, 16,
               c.ks, c.bn);
  std::fclose(fp);
}

static bool autotune_enabled() {
  if (g_autotune.load() < 0) {
    const char* e = std::getenv("TTF_AUTOTUNE");
    g_autotune.store((e && e[0] == '0') ? 0 : 1);
  }
  return g_autotune.load() == 1;
}

// Split-K factor of a product, a function of its shape alone: the tuner
// varies tiles and K chunks, which leave every sum's order unchanged, but
// never the split, so one shape gives the same bits in every process and
// on every stream whatever the tuning found.  Products with fewer than 128
// 64 x 64 tiles split K into power-of-two ranges of at least 64 until about
// 512 work-groups are in flight.
static int splitk_rule(int M, int N, int K, int nbatch) {
  const int64_t t64 = ceil_div(M, 64) * ceil_div(N, 64) * (int64_t)nbatch;
  if (t64 >= 128 || K < 128) return 1;
  int ks = 1;
  while (ks < 8 && K / (2 * ks) >= 64 && t64 * ks < 512) ks *= 2;
  return ks;
}

// Estimated cost of a tile shape: rounds of work-groups over the 256 CUs
// times a work-group's matrix-core time at its rate.  A work-group of one
// wave shares its CU with three others.
static double tile_cost(const Tile& t, int M, int N, int nbatch, int ks) {
  const int64_t wgs = ceil_div(M, t.bm) * ceil_div(N, t.bn) * nbatch * ks;
  const int64_t percu = t.threads == 64 ? 4 : 1;
  const double rounds = (double)ceil_div(wgs, 256 * percu);
  return rounds * percu * t.bm * t.bn / t.rate;
}

static Cfg heuristic(int M, int N, int K, int nbatch) {
  const int ks = splitk_rule(M, N, K, nbatch);
  const Tile* best = nullptr;
  double cost = 0.0;
  for (const Tile& t : kTiles) {
    const double c = tile_cost(t, M, N, nbatch, ks);
    if (!best || c < cost) { best = &t; cost = c; }
  }
  return {best->bm, best->bn, ks};
}

template <typename T, bool CT, int MODE>
static void launch_tiles(const GemmOp<T>& op, const Cfg& c, hipStream_t st) {
  const unsigned wgs = (unsigned)(ceil_div(op.M, c.bm) * ceil_div(op.N, c.bn) * op.nbatch * op.ksplit);
  // K chunk: 16 for f64, 32 for f32 (a 16-byte load covers four k); the
  // small tiles, latency-bound on each chunk, take twice as much
  constexpr int BK = sizeof(T) == 8 ? 16 : 32, BK1 = MODE == kVecBoth ? 2 * BK : BK;
  switch (1000 * c.bm + c.bn) {
    case 128064:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 128, 64, BK, 2, 2, CT, MODE>), dim3(wgs), dim3(256), 0, st, op);
      break;
    case 64096:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 64, 96, BK, 4, 2, CT, MODE>), dim3(wgs), dim3(512), 0, st, op);
      break;
    case 64080:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 64, 80, BK, 4, 1, CT, MODE>), dim3(wgs), dim3(256), 0, st, op);
      break;
    case 64064:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 64, 64, BK, 2, 2, CT, MODE>), dim3(wgs), dim3(256), 0, st, op);
      break;
    case 64032:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 64, 32, BK, 4, 1, CT, MODE>), dim3(wgs), dim3(256), 0, st, op);
      break;
    case 32032:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 32, 32, BK1, 2, 2, CT, MODE>), dim3(wgs), dim3(256), 0, st, op);
      break;
    default:
      hipLaunchKernelGGL((gemm_mfma_kernel<T, 32, 16, BK1, 1, 1, CT, MODE>), dim3(wgs), dim3(64), 0, st, op);
      break;
  }
}

template <typename T>
static void launch_cfg(GemmOp<T> op, const Cfg& c, hipStream_t st) {
  op.ksplit = c.ks;
  // column-contiguous outputs (and the column-major split-K slices) take the
  // swapped-fragment variant, whose lanes store consecutive rows; the other
  // outputs are few, and small, and read element by element
  if (op.ksplit == 1 && op.sCi != 1) {
    launch_tiles<T, false, kWide>(op, c, st);
  } else {
    switch (load_mode(op)) {
      case kWide: launch_tiles<T, true, kWide>(op, c, st); break;
      case kVecBoth: launch_tiles<T, true, kVecBoth>(op, c, st); break;
      case kVecA: launch_tiles<T, true, kVecA>(op, c, st); break;
      case kVecB: launch_tiles<T, true, kVecB>(op, c, st); break;
      default: launch_tiles<T, true, kScalar>(op, c, st); break;
    }
  }
  TTF_HIP(hipGetLastError());
  if (op.ksplit > 1) {
    int64_t total = (int64_t)op.M * op.N * op.nbatch;
    int blocks = (int)std::min<int64_t>(ceil_div(total, 256), 4096);
    hipLaunchKernelGGL((gemm_splitk_reduce<T>), dim3(blocks), dim3(256), 0, st, op);
    TTF_HIP(hipGetLastError());
  }
}

template <typename T>
static T* splitk_work(const GemmOp<T>& op, int ks) {
  size_t need = sizeof(T) * (size_t)ks * op.nbatch * (size_t)op.M * op.N;
  return (T*)arena(kArenaSplitK, need);
}

// Times the three tile shapes that tile_cost ranks first twice with events
// and keeps the fastest; the split-K factor is fixed by splitk_rule.  Only
// products that overwrite C (beta == 0) are tuned, since the candidates run
// the product several times.
template <typename T>
static Cfg tune(const GemmOp<T>& op0, hipStream_t st) {
  const int ks = splitk_rule(op0.M, op0.N, op0.K, op0.nbatch);
  std::vector<std::pair<double, Cfg>> ranked;
  for (const Tile& t : kTiles)
    ranked.push_back({tile_cost(t, op0.M, op0.N, op0.nbatch, ks), Cfg{t.bm, t.bn, ks}});
  std::stable_sort(ranked.begin(), ranked.end(),
                   [](const std::pair<double, Cfg>& x, const std::pair<double, Cfg>& y) { return x.first < y.first; });
  std::vector<Cfg> cands;
  for (size_t i = 0; i < ranked.size() && i < 3; ++i) cands.push_back(ranked[i].second);
  hipEvent_t e0, e1;
  TTF_HIP(hipEventCreate(&e0));
  TTF_HIP(hipEventCreate(&e1));
  Cfg best = heuristic(op0.M, op0.N, op0.K, op0.nbatch);
  float best_ms = 1e30f;
  for (const Cfg& c : cands) {
    GemmOp<T> op = op0;
    if (c.ks > 1) op.work = splitk_work(op, c.ks);
    launch_cfg(op, c, st);   // warm-up (code object load, caches)
    TTF_HIP(hipEventRecord(e0, st));
    launch_cfg(op, c, st);
    launch_cfg(op, c, st);
    TTF_HIP(hipEventRecord(e1, st));
    TTF_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    TTF_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (ms < best_ms) { best_ms = ms; best = c; }
  }
  TTF_HIP(hipEventDestroy(e0));
  TTF_HIP(hipEventDestroy(e1));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    ++g_tune_count;
  }
  return best;
}

template <typename T>
void gemm_launch(GemmOp<T> op, hipStream_t st) {
  if (op.M <= 0 || op.N <= 0 || op.nbatch <= 0) return;
  if (op.nb0 <= 0) op.nb0 = 1;
  TTF_REQUIRE(op.nbatch <= 65535, "gemm: batch count %d exceeds the grid limit", op.nbatch);
  if (op.K <= 0) {
    // empty sum: C = beta*C (alpha*0)
    op.K = 0;
  }
  if (panel_eligible(op)) {
    int64_t total = (int64_t)op.M * op.nbatch;
    int blocks = (int)std::min<int64_t>(ceil_div(total, 256), 65535);
    if (op.N <= 4)
      hipLaunchKernelGGL((panel_kernel<T, 4>), dim3(blocks), dim3(256), 0, st, op);
    else if (op.N <= 8)
      hipLaunchKernelGGL((panel_kernel<T, 8>), dim3(blocks), dim3(256), 0, st, op);
    else if (op.N <= 16)
      hipLaunchKernelGGL((panel_kernel<T, 16>), dim3(blocks), dim3(256), 0, st, op);
    else
      hipLaunchKernelGGL((panel_kernel<T, 32>), dim3(blocks), dim3(256), 0, st, op);
    TTF_HIP(hipGetLastError());
    return;
  }
  const double flops = 2.0 * op.M * op.N * (double)op.K * op.nbatch;
  const Key key = key_of(op);
  Cfg c;
  bool have = false;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    load_tune_table();
    auto it = g_tuned.find(key);
    if (it != g_tuned.end()) { c = it->second; have = true; }
  }
  if (!have) {
    const bool alias = (const void*)op.C == (const void*)op.A || (const void*)op.C == (const void*)op.B;
    // no timing runs while a stream capture records this thread's launches
    const bool tuned = autotune_enabled() && !t_no_tune && op.beta == T(0) && !alias && flops >= 4e6;
    c = tuned ? tune(op, st) : heuristic(op.M, op.N, op.K, op.nbatch);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    if (!t_no_tune) g_tuned[key] = c;
    if (tuned) record_tuned(key, c);
  }
  if (c.ks > 1) op.work = splitk_work(op, c.ks);
  launch_cfg(op, c, st);
}

template <typename T>
size_t gemm_workspace(const GemmOp<T>& op) {
  if (op.M <= 0 || op.N <= 0 || op.nbatch <= 0 || panel_eligible(op)) return 0;
  const int ks = splitk_rule(op.M, op.N, op.K, op.nbatch);
  return ks > 1 ? (size_t)ks * op.nbatch * (size_t)op.M * op.N : 0;
}

template <typename T>
void gemm_launch_ws(GemmOp<T> op, T* ws, size_t ws_cap, hipStream_t st) {
  if (op.M <= 0 || op.N <= 0 || op.nbatch <= 0) return;
  if (op.nb0 <= 0) op.nb0 = 1;
  TTF_REQUIRE(op.nbatch <= 65535, "gemm: batch count %d exceeds the grid limit", op.nbatch);
  if (op.K <= 0) op.K = 0;
  if (panel_eligible(op)) {
    gemm_launch(op, st);   // the panel kernel needs no workspace and is never tuned
    return;
  }
  const Key key = key_of(op);
  Cfg c = heuristic(op.M, op.N, op.K, op.nbatch);
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(key);
    if (it != g_tuned.end()) c = it->second;
  }
  if (c.ks > 1) {
    const size_t need = (size_t)c.ks * op.nbatch * (size_t)op.M * op.N;
    TTF_REQUIRE(ws != nullptr && need <= ws_cap, "gemm: split-K workspace of %zu elements exceeds the %zu given",
                need, ws_cap);
    op.work = ws;
  }
  launch_cfg(op, c, st);
}

template void gemm_launch<double>(GemmOp<double>, hipStream_t);
template void gemm_launch<float>(GemmOp<float>, hipStream_t);
template size_t gemm_workspace<double>(const GemmOp<double>&);
template size_t gemm_workspace<float>(const GemmOp<float>&);
template void gemm_launch_ws<double>(GemmOp<double>, double*, size_t, hipStream_t);
template void gemm_launch_ws<float>(GemmOp<float>, float*, size_t, hipStream_t);

ZPlan zgemm_plan(int M, int N, int K, int nbatch) {
  ZPlan p;
  p.bm = ceil_div(M, 64) * ceil_div(N, 64) * (int64_t)nbatch >= 128 ? 64 : 32;
  p.tiles = ceil_div(M, p.bm) * ceil_div(N, p.bm);
  // few work-groups with a long K: slices of K in parallel (at least 48 deep
  // each), summed by a second launch
  p.ks = 1;
  if (p.bm == 32 && p.tiles * nbatch < 32 && K >= 128)
    p.ks = std::max(1, (int)std::min<int64_t>({8, K / 48, ceil_div(64, p.tiles * nbatch)}));
  return p;
}

template <typename R>
static void zgemm_launch_t(ZGemmOpT<R> op, hipStream_t st) {
  typedef typename CplxT<R>::type C_t;
  if (op.M <= 0 || op.N <= 0 || op.nbatch <= 0) return;
  if (op.nb0 <= 0) op.nb0 = 1;
  TTF_REQUIRE(op.nbatch <= 65535, "zgemm: batch count %d exceeds the grid limit", op.nbatch);
  const ZPlan p = zgemm_plan(op.M, op.N, op.K, op.nbatch);
  op.ksplit = p.ks;
  op.work = p.ks > 1 ? (C_t*)arena(kArenaSplitK, sizeof(C_t) * (size_t)p.ks * op.nbatch * (size_t)op.M * op.N) : nullptr;
  dim3 grid((unsigned)p.tiles, (unsigned)op.nbatch, (unsigned)op.ksplit);
  // 32x32 tiles come with few work-groups, each one's K loop latency-bound
  // on its global loads: a 32-deep K chunk halves the trips
  if (p.bm == 64)
    hipLaunchKernelGGL((zgemm_mfma_kernel<R, 64, 64>), grid, dim3(256), 0, st, op);
  else if (op.K > 16)
    hipLaunchKernelGGL((zgemm_mfma_kernel<R, 32, 32, 32>), grid, dim3(256), 0, st, op);
  else
    hipLaunchKernelGGL((zgemm_mfma_kernel<R, 32, 32>), grid, dim3(256), 0, st, op);
  TTF_HIP(hipGetLastError());
  if (op.ksplit > 1) {
    const int64_t total = (int64_t)op.M * op.N * op.nbatch;
    hipLaunchKernelGGL(zgemm_splitk_reduce<R>, dim3((unsigned)std::min<int64_t>(ceil_div(total, 256), 4096)),
                       dim3(256), 0, st, op);
    TTF_HIP(hipGetLastError());
  }
}

void zgemm_launch(ZGemmOp op, hipStream_t st) { zgemm_launch_t<double>(op, st); }
void cgemm_launch(CGemmOp op, hipStream_t st) { zgemm_launch_t<float>(op, st); }

long gemm_tuned_shapes() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  return (long)g_tuned.size();
}

}  // namespace ttf

extern "C" {

int ttf_set_autotune(int enable) {
  std::lock_guard<std::mutex> lk(ttf::g_tune_mu);
  ttf::g_autotune = enable ? 1 : 0;
  if (!enable) ttf::g_tuned.clear();
  return 0;
}

long ttf_autotune_count(void) {
  std::lock_guard<std::mutex> lk(ttf::g_tune_mu);
  return ttf::g_tune_count;
}

}  // extern "C"
