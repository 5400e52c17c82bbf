// jacobi.hpp -- one-workgroup parallel cyclic Jacobi eigensolver for the
// small symmetric projected matrices of the Lanczos solvers (FP64, in LDS).
// Call from a kernel launched with 256 threads per block.
#pragma once

#include <hip/hip_runtime.h>

namespace spined {

constexpr int kJacobiMax = 64;
constexpr int kJacobiThreads = 256;

// Rotation (c, s) that annihilates a_pq of the pair with diagonal a_pp, a_qq.
__device__ inline void jacobi_rotation(double app, double aqq, double apq, double &c, double &s) {
  c = 1.0;
  s = 0.0;
  if (apq != 0.0) {
    const double tau = (aqq - app) / (2.0 * apq);
    const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
    c = 1.0 / sqrt(1.0 + t * t);
    s = t * c;
  }
}

// Parallel cyclic Jacobi (round-robin pairing) for the symmetric m x m
// projected matrix, m <= MAXM (even, <= 64), in LDS.  evals ascending; S
// column-major.  MAXM sizes the LDS workspace (2 MAXM (MAXM + 1) doubles).
//
// Bound: the latency of one round's chain -- the rotation's two divisions and
// two square roots, LDS, barriers -- about m - 1 rounds a sweep and 7 sweeps.
// The 2 x 2 blocks A[pair k][pair l] are independent, so after the rotations
// one step updates columns and rows together and V with them.  Every ordered
// pair (k, l) is computed from its own four entries, columns first, then rows:
// the rounding of a pass over all columns followed by one over all rows.  (The
// mirror image of a block has another rounding, and the sign of an eigenvector
// of the block solver hangs on the last bit.)  Up to m = 32 that is one block a
// thread.  The closing sort and copy run on all threads (one thread took a third
// of the call).  Rotations by every block's thread itself, without the barrier
// between, were slower (223 us against 177 for three steps a round, m <= 24): the
// divisions then compete for issue.
template <int MAXM = kJacobiMax>
__device__ inline void jacobi_eigh_device(const double *__restrict__ T, int ldt, int m,
                                          double *__restrict__ evals, double *__restrict__ S,
                                          int max_sweeps) {
  static_assert(MAXM % 2 == 0 && MAXM <= kJacobiMax, "even size up to kJacobiMax");
  constexpr int kHalf = MAXM / 2;
  constexpr int kBlocks = (kHalf * kHalf + kJacobiThreads - 1) / kJacobiThreads;
  __shared__ double A[MAXM][MAXM + 1];
  __shared__ double V[MAXM][MAXM + 1];
  __shared__ double cs[kHalf], sn[kHalf];
  __shared__ double red[2][kJacobiThreads / 64]; // per-wave sums of (off, dia)
  const int tid = threadIdx.x;
  const int mp = m + (m & 1);
  const int half = mp / 2;
  for (int e = tid; e < mp * mp; e += kJacobiThreads) {
    const int i = e / mp, j = e % mp;
    double a = 0.0;
    if (i < m && j < m) a = 0.5 * (T[i * ldt + j] + T[j * ldt + i]);
    A[i][j] = a;
    V[i][j] = i == j ? 1.0 : 0.0;
  }
  // the pairs (k, l) of this thread's blocks
  int bk[kBlocks], bl[kBlocks];
#pragma unroll
  for (int z = 0; z < kBlocks; ++z) {
    const int e = tid + z * kJacobiThreads;
    bk[z] = e < half * half ? e / half : -1;
    bl[z] = e % half;
  }
  __syncthreads();
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    // convergence: off-diagonal mass vs diagonal mass
    double off = 0.0, dia = 0.0;
    for (int e = tid; e < mp * mp; e += kJacobiThreads) {
      const int i = e / mp, j = e % mp;
      const double a = A[i][j];
      if (i == j)
        dia += a * a;
      else
        off += a * a;
    }
    // wave sums, then the four waves in order
    for (int off2 = 32; off2 > 0; off2 >>= 1) {
      off += __shfl_down(off, off2, 64);
      dia += __shfl_down(dia, off2, 64);
    }
    if ((tid & 63) == 0) {
      red[0][tid >> 6] = off;
      red[1][tid >> 6] = dia;
    }
    __syncthreads();
    const double off_tot = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    const double dia_tot = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    if (off_tot <= 1e-30 * (dia_tot + off_tot) || off_tot == 0.0) break; // the same in all threads
    for (int step = 0; step < mp - 1; ++step) {
      // round robin: position 0 holds player 0, others rotate
      auto player = [&](int pos) {
        int v = pos - 1 + step;
        v = v >= mp - 1 ? v - (mp - 1) : v;
        return pos == 0 ? 0 : 1 + v;
      };
      auto pair = [&](int k, int &p, int &q) {
        const int a = player(k), b = player(mp - 1 - k);
        p = a < b ? a : b;
        q = a < b ? b : a;
      };
      if (tid < half) {
        int p, q;
        pair(tid, p, q);
        double c, sk;
        jacobi_rotation(A[p][p], A[q][q], A[p][q], c, sk);
        cs[tid] = c;
        sn[tid] = sk;
      }
      __syncthreads();
#pragma unroll
      for (int z = 0; z < kBlocks; ++z) {
        if (bk[z] < 0) continue;
        int p, q, r, t;
        pair(bk[z], p, q);
        pair(bl[z], r, t);
        const double ck = cs[bk[z]], sk = sn[bk[z]], cl = cs[bl[z]], sl = sn[bl[z]];
        // block rows p, q and columns r, t: columns by (cl, sl), then rows
        const double a0 = A[p][r], a1 = A[p][t], a2 = A[q][r], a3 = A[q][t];
        const double b0 = cl * a0 - sl * a1, b1 = sl * a0 + cl * a1;
        const double b2 = cl * a2 - sl * a3, b3 = sl * a2 + cl * a3;
        const double w0 = ck * b0 - sk * b2, w1 = ck * b1 - sk * b3;
        const double w2 = sk * b0 + ck * b2, w3 = sk * b1 + ck * b3;
        A[p][r] = w0;
        A[p][t] = w1;
        A[q][r] = w2;
        A[q][t] = w3;
      }
      // V <- V J (columns p, q)
      for (int e = tid; e < half * mp; e += kJacobiThreads) {
        const int k = e / mp, i = e % mp;
        int p, q;
        pair(k, p, q);
        const double c = cs[k], sk = sn[k];
        const double vp = V[i][p], vq = V[i][q];
        V[i][p] = c * vp - sk * vq;
        V[i][q] = sk * vp + c * vq;
      }
      __syncthreads();
    }
  }
  __syncthreads();
  // ascending order of the m real eigenpairs (the padding index is dropped): a
  // pair's place is the number of smaller ones; equal or unordered values take
  // the order that a selection sort with exchanges leaves them in
  __shared__ int order[MAXM];
  __shared__ int serial;
  if (tid == 0) serial = 0;
  __syncthreads();
  for (int i = tid; i < m; i += kJacobiThreads) {
    const double a = A[i][i];
    int at = 0;
    bool tie = false;
    for (int j = 0; j < m; ++j) {
      const double b = A[j][j];
      at += b < a ? 1 : 0;
      tie = tie || (j != i && !(b < a) && !(a < b));
    }
    order[at] = i;
    if (tie) serial = 1;
  }
  __syncthreads();
  if (serial && tid == 0) {
    for (int i = 0; i < m; ++i) order[i] = i;
    for (int i = 0; i < m; ++i) {
      int best = i;
      for (int j = i + 1; j < m; ++j)
        if (A[order[j]][order[j]] < A[order[best]][order[best]]) best = j;
      const int t = order[i];
      order[i] = order[best];
      order[best] = t;
    }
  }
  __syncthreads();
  for (int i = tid; i < m; i += kJacobiThreads) evals[i] = A[order[i]][order[i]];
  for (int e = tid; e < m * m; e += kJacobiThreads) S[e] = V[e % m][order[e / m]];
}

} // namespace spined
