// Two-sided cyclic Jacobi for small symmetric matrices held in LDS, shared by
// the small eigensolver, SVQB orthonormalisation and Rayleigh-Ritz kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "wave.h"

namespace ttf {

constexpr int kJacobiMaxN = 64;   // largest order (rows are indexed by lanes)

// Pair k of round r of the circle schedule over nn (even) indices: index
// nn-1 stays fixed and the others rotate, so every pair meets once in the
// nn-1 rounds of a sweep.
__device__ inline void jacobi_pair(int r, int k, int nn, int& p, int& q) {
  int a, b;
  if (k == 0) {
    a = r;
    b = nn - 1;
  } else {
    a = r + k;
    if (a >= nn - 1) a -= nn - 1;
    b = r - k;
    if (b < 0) b += nn - 1;
  }
  p = min(a, b);
  q = max(a, b);
}

// Rotation parameters (J = [[c, s], [-s, c]] on rows and columns p, q) that
// annihilate a_pq of the 2x2 block [[app, apq], [apq, aqq]] when `go`, else
// the identity.  t = tan(theta) is the smaller root of
// t^2 + 2 cot(2 theta) t - 1 = 0, t = sign(d) 2 a_pq / (|d| + sqrt(d^2 + 4 a_pq^2))
// with d = a_qq - a_pp, evaluated from the hardware reciprocal (square
// root) estimates refined by Newton steps: t to about 2^-46 (it only sets
// how well a_pq is annihilated), c = (1 + t^2)^(-1/2) by two steps so that
// c^2 + s^2 = 1 to rounding whatever the error of t (the rotation stays
// orthogonal).  `go` selects the results, so its own comparison is off the
// chain.  The half-angle form, c^2 = (1 + |d| w) / 2 and s = sign(d) a_pq w / c
// with w = (d^2 + 4 a_pq^2)^(-1/2), has one estimate less, but the rounding of
// w goes into c^2 + s^2: it doubled ||Q^T Q - I||_F (order 64, 2.5e-14 ->
// 5.0e-14), lost orthogonality where d^2 + 4 a_pq^2 is subnormal, and was no
// faster (left factor of 256 x 640: 4630 us against 4612).
__device__ __forceinline__ void jacobi_cs(double apq, double app, double aqq, bool go, double& c, double& s) {
  const double d = aqq - app;
  const double q = d * d + 4.0 * apq * apq;
  double rq = __builtin_amdgcn_rsq(q);
  rq = rq * (1.5 - 0.5 * q * rq * rq);
  const double den = fabs(d) + q * rq;
  double ri = __builtin_amdgcn_rcp(den);
  ri = ri * (2.0 - den * ri);
  const double t = (d >= 0.0 ? 2.0 : -2.0) * apq * ri;
  const double x = 1.0 + t * t;
  double cc = __builtin_amdgcn_rsq(x);
  cc = cc * (1.5 - 0.5 * x * cc * cc);
  cc = cc * (1.5 - 0.5 * x * cc * cc);
  c = go ? cc : 1.0;
  s = go ? t * cc : 0.0;
}

// Whether pair (p, q) of the current matrix is rotated: |a_pq| above the
// caller's rounding floor tol_abs and above eps * sqrt(|a_pp a_qq|).
__device__ __forceinline__ bool jacobi_go(double apq, double app, double aqq, double tol_abs) {
  const double eps = 2.220446049250313e-16;
  return fabs(apq) > tol_abs && apq * apq > eps * eps * fabs(app * aqq);
}

// Rotations with |sin| at most this are "small": a sweep whose rotations
// are all small leaves off-diagonal entries of order n * kJacobiSmall^2 *
// ||A|| (quadratic convergence), below the rounding floor for n <= 64, so
// the next sweep would not change the result and is skipped.
constexpr double kJacobiSmall = 1e-9;

// The double-buffered form, for any n <= 64: diagonalises the symmetric
// n x n matrix held in A (row stride LD) and accumulates the rotations into
// V (V <- V J).  B is a second buffer: each round of the circle schedule reads one buffer and writes the other,
// so one barrier per round suffices.  Odd n is padded with a zero row and
// column n (in A, B and V; the buffers hold at least n + 1 rows), so every
// pair is real and no load is conditional; rotations involving the pad are
// the identity.  Thread t owns the 2x2 block (rows of pair kp) x (columns of
// pair kq), t = kp + half * kq, derives both rotations from the round's
// input itself (no phase publishes rotations) and also rotates rows kp and
// kp + half of V in the columns of pair kq.  All of a task's loads are
// issued before its arithmetic so that one LDS round trip and the two
// interleaved rotation computations make up the round.  The 2x2 blocks are
// updated in full (annihilated entries keep their rounding-level values).
// go(a_pq, a_pp, a_qq) decides whether a pair is rotated.  The loop ends
// after a sweep with no rotation above `small` or after max_sweeps; a thread takes at most 4 tasks, so the
// block needs 4 blockDim.x >= (n / 2 + 1)^2.  `flags` is 3 ints of LDS.  All threads
// of the block call it; the returned pointer (A or B) holds the diagonalised
// matrix.
template <int LD, class Go>
__device__ double (*jacobi_sym_circle(double (*A)[LD], double (*B)[LD], double (*V)[LD], int n, int max_sweeps,
                                      const Go& go, int* flags, double small))[LD] {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nn = n + (n & 1);
  const int half = nn / 2;
  if (n <= 1) return A;
  if (n & 1) {
    for (int j = tid; j <= n; j += nt) {
      A[n][j] = 0.0;
      A[j][n] = 0.0;
      B[n][j] = 0.0;
      B[j][n] = 0.0;
      V[n][j] = 0.0;
      V[j][n] = 0.0;
    }
  }
  const int ntask = half * half;   // at most 1024 = 4 x 256 tasks
  double(*cur)[LD] = A;
  double(*nxt)[LD] = B;
  if (tid < 3) flags[tid] = 0;
  // each thread's tasks (pair indices kp, kq), once: the rounds then have no
  // division on their critical path
  int kps[4], kqs[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int t = tid + w * nt;
    kps[w] = t % half;
    kqs[w] = t / half;
  }
  __syncthreads();
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    int* moved = flags + sweep % 3;
    // flags[(sweep+1) % 3] was last read before the previous sweep's barriers
    if (tid == 0) flags[(sweep + 1) % 3] = 0;
    for (int r = 0; r < nn - 1; ++r) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (tid + w * nt >= ntask) break;
        const int kp = kps[w], kq = kqs[w];
        int p, q, u, v;
        jacobi_pair(r, kp, nn, p, q);
        jacobi_pair(r, kq, nn, u, v);
        const double app = cur[p][p], aqq = cur[q][q], apq = cur[p][q];
        const double auu = cur[u][u], avv = cur[v][v], auv = cur[u][v];
        const double apu = cur[p][u], apv = cur[p][v], aqu = cur[q][u], aqv = cur[q][v];
        const int i1 = kp + half;
        const double x0 = V[kp][u], y0 = V[kp][v], x1 = V[i1][u], y1 = V[i1][v];
        double c1, s1, c2, s2;
        jacobi_cs(apq, app, aqq, go(apq, app, aqq), c1, s1);
        jacobi_cs(auv, auu, avv, go(auv, auu, avv), c2, s2);
        if (kq == 0 && fabs(s1) > small) *moved = 1;
        // columns u, v
        const double t0 = c2 * apu - s2 * apv, t1 = s2 * apu + c2 * apv;
        const double t2 = c2 * aqu - s2 * aqv, t3 = s2 * aqu + c2 * aqv;
        // rows p, q
        nxt[p][u] = c1 * t0 - s1 * t2;
        nxt[p][v] = c1 * t1 - s1 * t3;
        nxt[q][u] = s1 * t0 + c1 * t2;
        nxt[q][v] = s1 * t1 + c1 * t3;
        // rows kp and kp + half of V, columns of pair kq
        V[kp][u] = c2 * x0 - s2 * y0;
        V[kp][v] = s2 * x0 + c2 * y0;
        V[i1][u] = c2 * x1 - s2 * y1;
        V[i1][v] = s2 * x1 + c2 * y1;
      }
      __syncthreads();
      double(*tt)[LD] = cur;
      cur = nxt;
      nxt = tt;
    }
    if (!*moved) break;
  }
  return cur;
}

// The same circle schedule with the matrix kept in slot order: slots 2k and
// 2k+1 hold the pair that round's rotation k acts on, and between rounds the
// contents move by one fixed permutation of the slots (the circle's
// rotation), so that after the nn - 1 rounds of a sweep every index is back
// in its starting slot.  Slot s starts with index jacobi_slot_index(s).
__device__ inline int jacobi_slot_index(int s, int nn) {
  return (s & 1) == 0 ? s >> 1 : (s == 1 ? nn - 1 : nn - 1 - (s >> 1));
}

// The slot that the contents of slot s move to between two rounds (half =
// nn / 2 pairs).
__device__ inline int jacobi_slot_next(int s, int half) {
  if (half == 1 || s == 1) return s;
  if (s == 0) return 3;
  if ((s & 1) == 0) return s - 2;
  if (s == 2 * half - 1) return 2 * half - 2;
  return s + 2;
}

// The slot whose contents move to slot s.
__device__ inline int jacobi_slot_prev(int s, int half) {
  if (half == 1 || s == 1) return s;
  if (s == 3) return 0;
  if (s == 2 * half - 2) return 2 * half - 1;
  return (s & 1) == 0 ? s + 2 : s - 2;
}

// jacobi_sym for n >= 3 and (n + 1) / 2 squared <= blockDim.x - 64: thread
// (kp, kq) owns the 2x2 block of slot pairs kp x kq for the whole solve, with
// every address fixed once.  One barrier a round: the matrix alternates
// between two buffers (both in slot order), each round applies rotations
// that the round before published, and beside it a thread per pair takes the
// next round's rotation from the entries of the old matrix that meet in that
// pair: two diagonal entries and one coupling, each brought up to date by the
// current rotations.  The chain of a round is then loads, one 2x2 update,
// the rotation and a barrier, where it was that with a second barrier and a
// reload of the rotations between them.  The pairs' threads are the block's
// last wave, which owns no 2x2 block, and the vectors (V, in index order;
// a thread rotates its own two columns of a row, in place) go to threads
// without blocks when there are enough of them.  Working copies: the matrix
// in slot order in B and A; at the end A's diagonal holds the eigenvalues,
// and A is returned.  One sweep of order 32 on 512 threads: 43500 clocks with
// two barriers a round -> 37800; the rest of a round is its LDS traffic (two
// loads and two stores of every entry of both matrices).
template <int LD, class Go>
__device__ double (*jacobi_sym_slots(double (*A)[LD], double (*B)[LD], double (*V)[LD], int n, int max_sweeps,
                                     const Go& go, int* flags, double small))[LD] {
  __shared__ double2 csb[2][kJacobiMaxN / 2];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nn = n + (n & 1);
  const int half = nn / 2, ntask = half * half;
  if (n & 1) {
    for (int j = tid; j <= n; j += nt) {
      A[n][j] = 0.0;
      A[j][n] = 0.0;
      V[n][j] = 0.0;
      V[j][n] = 0.0;
    }
  }
  if (tid < 3) flags[tid] = 0;
  __syncthreads();
  for (int e = tid; e < nn * nn; e += nt) {
    const int s = e % nn, t = e / nn;
    B[s][t] = A[jacobi_slot_index(s, nn)][jacobi_slot_index(t, nn)];
  }
  __syncthreads();
  double(*cur)[LD] = B;
  double(*nxt)[LD] = A;
  // matrix blocks
  const bool task = tid < ntask;
  const int kp = task ? tid % half : 0, kq = task ? tid / half : 0;
  const int p0 = 2 * kp, q0 = 2 * kq;
  const int np0 = jacobi_slot_next(p0, half), np1 = jacobi_slot_next(p0 + 1, half);
  const int nq0 = jacobi_slot_next(q0, half), nq1 = jacobi_slot_next(q0 + 1, half);
  // rotations: pair k of the next round joins the contents of slots sa and sb
  const int last = nt - 64;
  const int k = tid - last;
  const bool rot = k >= 0 && k < half;
  const int sa = jacobi_slot_prev(2 * (rot ? k : 0), half), sb = jacobi_slot_prev(2 * (rot ? k : 0) + 1, half);
  const int ka = sa >> 1, kb = sb >> 1;
  // vectors: rows i and i + half in the columns of pair kv; up to two tasks
  const int vfirst = (ntask + 63) / 64 * 64, vcount = max(0, last - vfirst);
  const bool vsplit = 2 * vcount >= ntask;
  const int v0 = vsplit ? tid - vfirst : tid, vstep = vsplit ? vcount : nt;
  int vi[2], vk[2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int t = v0 + w * vstep;
    const bool on = v0 >= 0 && (!vsplit || v0 < vcount) && t < ntask;
    vi[w] = on ? t % half : -1;
    vk[w] = on ? t / half : 0;
  }
  if (rot) {
    const double app = cur[2 * k][2 * k], apq = cur[2 * k][2 * k + 1], aqq = cur[2 * k + 1][2 * k + 1];
    double c, s;
    jacobi_cs(apq, app, aqq, go(apq, app, aqq), c, s);
    csb[0][k] = make_double2(c, s);
    if (fabs(s) > small) flags[0] = 1;
  }
  __syncthreads();
  int par = 0;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    // flags[(sweep+1) % 3] was last read before the previous sweep's barriers
    // and is next set in this sweep's last round (n >= 3: not its first)
    if (tid == 0) flags[(sweep + 1) % 3] = 0;
    for (int r = 0; r < nn - 1; ++r) {
      if (rot) {
        const double2 ra = csb[par][ka], rb = csb[par][kb];
        const double* a0 = &cur[2 * ka][2 * ka];
        const double* a1 = &cur[2 * ka + 1][2 * ka];
        const double* b0 = &cur[2 * kb][2 * kb];
        const double* b1 = &cur[2 * kb + 1][2 * kb];
        const double* c0 = &cur[2 * ka][2 * kb];
        const double* c1 = &cur[2 * ka + 1][2 * kb];
        const double aa = a0[0], ab = a0[1], ad = a1[1], ba = b0[0], bb = b0[1], bd = b1[1];
        const double m00 = c0[0], m01 = c0[1], m10 = c1[0], m11 = c1[1];
        // entry (ea, eb) of a rotated block: rows (c, -s) or (s, c)
        const bool ea = sa & 1, eb = sb & 1;
        const double ua = ea ? ra.y : ra.x, va = ea ? ra.x : -ra.y;
        const double ub = eb ? rb.y : rb.x, vb = eb ? rb.x : -rb.y;
        const double app = ua * (ua * aa + va * ab) + va * (ua * ab + va * ad);
        const double aqq = ub * (ub * ba + vb * bb) + vb * (ub * bb + vb * bd);
        const double apq = ua * (ub * m00 + vb * m01) + va * (ub * m10 + vb * m11);
        double c, s;
        jacobi_cs(apq, app, aqq, go(apq, app, aqq), c, s);
        csb[par ^ 1][k] = make_double2(c, s);
        if (fabs(s) > small) flags[(r + 1 < nn - 1 ? sweep : sweep + 1) % 3] = 1;
      }
      if (task) {
        const double m00 = cur[p0][q0], m01 = cur[p0][q0 + 1], m10 = cur[p0 + 1][q0], m11 = cur[p0 + 1][q0 + 1];
        const double2 rp = csb[par][kp], rq = csb[par][kq];
        const double c1 = rp.x, s1 = rp.y, c2 = rq.x, s2 = rq.y;
        // columns of pair kq, then rows of pair kp
        const double t0 = c2 * m00 - s2 * m01, t1 = s2 * m00 + c2 * m01;
        const double t2 = c2 * m10 - s2 * m11, t3 = s2 * m10 + c2 * m11;
        nxt[np0][nq0] = c1 * t0 - s1 * t2;
        nxt[np0][nq1] = c1 * t1 - s1 * t3;
        nxt[np1][nq0] = s1 * t0 + c1 * t2;
        nxt[np1][nq1] = s1 * t1 + c1 * t3;
      }
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if (vi[w] < 0) break;
        // slots 2 kv and 2 kv + 1 hold indices (kv + r) mod (nn - 1) and
        // (-kv + r) mod (nn - 1), pair 0's second the fixed index nn - 1
        int u = vk[w] + r, v = r - vk[w];
        if (u >= nn - 1) u -= nn - 1;
        if (v < 0) v += nn - 1;
        if (vk[w] == 0) v = nn - 1;
        const int i0 = vi[w], i1 = vi[w] + half;
        const double2 rq = csb[par][vk[w]];
        const double w00 = V[i0][u], w01 = V[i0][v], w10 = V[i1][u], w11 = V[i1][v];
        V[i0][u] = rq.x * w00 - rq.y * w01;
        V[i0][v] = rq.y * w00 + rq.x * w01;
        V[i1][u] = rq.x * w10 - rq.y * w11;
        V[i1][v] = rq.y * w10 + rq.x * w11;
      }
      __syncthreads();
      double(*tt)[LD] = cur;
      cur = nxt;
      nxt = tt;
      par ^= 1;
    }
    if (!flags[sweep % 3]) break;
  }
  // a sweep ends with every index in its starting slot (nn <= 64 <= nt)
  const double d = tid < nn ? cur[tid][tid] : 0.0;
  __syncthreads();
  if (tid < nn) {
    const int i = jacobi_slot_index(tid, nn);
    A[i][i] = d;
  }
  __syncthreads();
  return A;
}

// The slot-ordered form for a block that has no wave left for the rotations
// (orders 61 to 64 on 1024 threads, 27 to 32 on 256): two barriers a round,
// updates in place.  Thread (kp, kq) owns the 2x2 block of slot pairs kp x kq; a
// round: each thread loads its block and its two rows of the vectors' slot
// pair kq; the diagonal-block threads compute the round's rotations and
// publish them; after a barrier every thread applies its two rotations and
// stores the block at the slots its contents move to.  Rotations taken a round
// ahead by waves that own blocks as well took 818 us against 534 for a solve
// of order 64.  Where a wave is free the form above is the faster one or equal:
// on 1024 threads order 60 takes 654 us in place and 547 with it, 48 303 and
// 274, 44 251 and 254, 33 164 and 144.  Working copies: the matrix in slot
// order in B, the vectors (V with columns in slot order) in A; at the end V
// receives the vectors in index order and A's diagonal the eigenvalues, and A
// is returned.
template <int LD, class Go>
__device__ double (*jacobi_sym_slots_inplace(double (*A)[LD], double (*B)[LD], double (*V)[LD], int n, int max_sweeps,
                                     const Go& go, int* flags, double small))[LD] {
  __shared__ double2 csb[kJacobiMaxN / 2];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nn = n + (n & 1);
  const int half = nn / 2;
  if (n & 1) {
    for (int j = tid; j <= n; j += nt) {
      A[n][j] = 0.0;
      A[j][n] = 0.0;
      V[n][j] = 0.0;
      V[j][n] = 0.0;
    }
  }
  __syncthreads();
  for (int e = tid; e < nn * nn; e += nt) {
    const int s = e % nn, t = e / nn;
    B[s][t] = A[jacobi_slot_index(s, nn)][jacobi_slot_index(t, nn)];
  }
  __syncthreads();
  for (int e = tid; e < nn * nn; e += nt) {
    const int r = e % nn, s = e / nn;
    A[r][s] = V[r][jacobi_slot_index(s, nn)];
  }
  if (tid < 3) flags[tid] = 0;
  __syncthreads();
  double(*M)[LD] = B;
  double(*W)[LD] = A;
  const bool task = tid < half * half;
  const int kp = task ? tid % half : 0, kq = task ? tid / half : 0;
  const int p0 = 2 * kp, p1 = p0 + 1, q0 = 2 * kq, q1 = q0 + 1;
  const int np0 = jacobi_slot_next(p0, half), np1 = jacobi_slot_next(p1, half);
  const int nq0 = jacobi_slot_next(q0, half), nq1 = jacobi_slot_next(q1, half);
  const int r0 = kp, r1 = kp + half;   // the rows of W this thread rotates
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    int* moved = flags + sweep % 3;
    // flags[(sweep+1) % 3] was last read before the previous sweep's barriers
    if (tid == 0) flags[(sweep + 1) % 3] = 0;
    for (int r = 0; r < nn - 1; ++r) {
      double m00 = 0.0, m01 = 0.0, m10 = 0.0, m11 = 0.0, w00 = 0.0, w01 = 0.0, w10 = 0.0, w11 = 0.0;
      if (task) {
        m00 = M[p0][q0]; m01 = M[p0][q1]; m10 = M[p1][q0]; m11 = M[p1][q1];
        w00 = W[r0][q0]; w01 = W[r0][q1]; w10 = W[r1][q0]; w11 = W[r1][q1];
        if (kp == kq) {   // a diagonal block: [[a_pp, a_pq], [a_pq, a_qq]]
          double c, s;
          jacobi_cs(m01, m00, m11, go(m01, m00, m11), c, s);
          csb[kp] = make_double2(c, s);
          if (fabs(s) > small) *moved = 1;
        }
      }
      __syncthreads();
      if (task) {
        const double2 rp = csb[kp], rq = csb[kq];
        const double c1 = rp.x, s1 = rp.y, c2 = rq.x, s2 = rq.y;
        // columns of pair kq, then rows of pair kp
        const double t0 = c2 * m00 - s2 * m01, t1 = s2 * m00 + c2 * m01;
        const double t2 = c2 * m10 - s2 * m11, t3 = s2 * m10 + c2 * m11;
        M[np0][nq0] = c1 * t0 - s1 * t2;
        M[np0][nq1] = c1 * t1 - s1 * t3;
        M[np1][nq0] = s1 * t0 + c1 * t2;
        M[np1][nq1] = s1 * t1 + c1 * t3;
        W[r0][nq0] = c2 * w00 - s2 * w01;
        W[r0][nq1] = s2 * w00 + c2 * w01;
        W[r1][nq0] = c2 * w10 - s2 * w11;
        W[r1][nq1] = s2 * w10 + c2 * w11;
      }
      __syncthreads();
    }
    if (!*moved) break;
  }
  // a sweep ends with every index in its starting slot
  for (int e = tid; e < nn * nn; e += nt) {
    const int r = e % nn, s = e / nn;
    V[r][jacobi_slot_index(s, nn)] = W[r][s];
  }
  __syncthreads();
  for (int s = tid; s < nn; s += nt) {
    const int i = jacobi_slot_index(s, nn);
    A[i][i] = M[s][s];
  }
  __syncthreads();
  return A;
}

// Diagonalises the symmetric n x n matrix held in A (row stride LD, n <= 64)
// and accumulates the rotations into V (V <- V J); B is a second buffer of
// the same shape.  Returns the matrix (A or B) whose diagonal holds the
// eigenvalues, in the order of V's columns.  Orders from 3 with (n + 1) / 2 squared
// <= blockDim.x - 64 take the slot-ordered form with a wave for the
// rotations, up to blockDim.x the one in place, larger ones the
// double-buffered one.
template <int LD>
__device__ double (*jacobi_sym(double (*A)[LD], double (*B)[LD], double (*V)[LD], int n, int max_sweeps,
                               double tol_abs, int* flags, double small = kJacobiSmall))[LD] {
  const auto go = [tol_abs](double apq, double app, double aqq) { return jacobi_go(apq, app, aqq, tol_abs); };
  const int half = (n + 1) / 2;
  if (n >= 3 && half * half <= (int)blockDim.x - 64)
    return jacobi_sym_slots<LD>(A, B, V, n, max_sweeps, go, flags, small);
  if (n >= 2 && half * half <= (int)blockDim.x)
    return jacobi_sym_slots_inplace<LD>(A, B, V, n, max_sweeps, go, flags, small);
  return jacobi_sym_circle<LD>(A, B, V, n, max_sweeps, go, flags, small);
}

// Block-wide sum of v over all threads (blockDim.x a multiple of 64, at most
// 1024); `red` holds one double per wave.  Every thread receives the sum.
__device__ inline double block_sum(double v, double* red) {
  v = wave_sum64(v);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

// Block-wide maximum, same contract as block_sum.
__device__ inline double block_max(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = red[0];
  for (int i = 1; i < nw; ++i) s = fmax(s, red[i]);
  return s;
}

}  // namespace ttf
