// f64 orthogonalisations of MPS tensors: Householder QR (gauge moves), the
// Cholesky factor of CholeskyQR3 and one-sided Jacobi (Hestenes) SVD
// (entanglement spectrum moves).  One workgroup per matrix.
#include "tnx_common.h"
#include "jacobi_rot.h"

namespace {

constexpr int NQ = 1024;    // lanes of the QR and SVD kernels
constexpr int KMAX = 4096;  // max columns of a gauge-move matrix

__device__ __forceinline__ double src_at(const double TNX_GLOBAL* src, int ld, int trans, int r, int c) {
  return trans ? src[(int64_t)c * ld + r] : src[(int64_t)r * ld + c];
}

// ------------------------------------------------------ Householder QR
// Three ways, by the number of rows:
// - m <= 16 (chain ends): a lane holds a column in registers; the reflectors
//   of the first columns are formed one after the other, every lane applies
//   them to its own column.
// - m <= 512 with at least 16 reflectors (the wide panels of a random MPS
//   that is brought into canonical form: 32 x chi .. chi/2 x chi): blocks of
//   16 columns, factored in LDS with one barrier per column, then applied to
//   the columns right of them as I - V T V^T on f64 MFMA; Q the same way in
//   reverse.
// - otherwise (tall panels of less than 8 columns, where CholeskyQR3 is not
//   used) column by column in global memory.
// Bound: a serial chain of reflectors (about 700 cycles each) in the panels,
// the f64 MFMA rate of the one CU in the products.  us (MI355X), one wave per
// column in global memory -> this: 16 matrices of 4 x 128 74 -> 8, of 16 x 128
// 327 -> 24, of 64 x 128 1387 -> 167; one of 32 x 512 2440 -> 106, of 256 x
// 512 37200 -> 2040.
constexpr int QS = 16;       // rows of the small path, columns of a block
constexpr int QB_MAX = 512;  // rows of the blocked path

struct QrLds {
  double tau[KMAX];
  double P[QS * (QB_MAX + 1)];   // the block's columns, then its V, stride m + 1
  double S[QS][QS + 1], T[QS][QS + 1];
  double beta[QS], scal[QS];
};

// Reflector of (x0, x) with s = |x|^2: beta, tau and the scale of x
__device__ __forceinline__ void reflector(double x0, double s, double& beta, double& tau, double& scal) {
  if (s == 0.0) {
    beta = x0;
    tau = 0.0;
    scal = 0.0;
  } else {
    const double nrm = sqrt(x0 * x0 + s);
    beta = x0 >= 0.0 ? -nrm : nrm;
    tau = (beta - x0) / beta;
    scal = 1.0 / (x0 - beta);
  }
}

template <int MR>   // m <= MR
__device__ __forceinline__ void qr_small(const tnx_qr_job& J, QrLds& L) {
  const int m = J.m, n = J.n, k = m < n ? m : n, t = threadIdx.x;
  const int w0 = t & ~63;   // first column of the wave: waves without columns only keep the barriers
  const double TNX_GLOBAL* src = as_global<const double>(J.src);
  int ld = J.ld, trans = J.trans;
  // More columns than lanes: R is written before the last ones are read, so src
  // is copied first if R may lie in it.
  const uint64_t len = 8 * (trans ? (uint64_t)(n - 1) * ld + m : (uint64_t)(m - 1) * ld + n);
  if (n > NQ && J.r < J.src + len && J.src < J.r + 8 * (uint64_t)k * n) {
    double TNX_GLOBAL* W = as_global<double>(J.work);
    for (int e = t; e < m * n; e += NQ) {
      const int c = e / m;
      W[e] = src_at(src, ld, trans, e - c * m, c);
    }
    __syncthreads();
    src = W;
    ld = m;
    trans = 1;
  }
  double TNX_GLOBAL* R = as_global<double>(J.r);
  double TNX_GLOBAL* q = as_global<double>(J.q);
  double (*V)[QS + 1] = L.S;   // V[j]: zeros, V[j][j] = 1, the reflector, zeros past m
  double x[MR];
  auto load = [&](int c) {
#pragma unroll
    for (int r = 0; r < MR; ++r) x[r] = (r < m && c < n) ? src_at(src, ld, trans, r, c) : 0.0;
  };
  auto apply = [&](int j) {   // (I - tau v v^T) x
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int r = 0; r < MR; ++r) s[r & 1] += V[j][r] * x[r];
    const double f = (s[0] + s[1]) * L.tau[j];
#pragma unroll
    for (int r = 0; r < MR; ++r) x[r] -= f * V[j][r];
  };
  auto store_r = [&](int c) {
#pragma unroll
    for (int i = 0; i < MR; ++i)
      if (i < k && c < n) R[(int64_t)i * n + c] = i <= c ? x[i] : 0.0;
  };
  if (w0 < n) load(t);
#pragma unroll 1
  for (int j = 0; j < k; ++j) {
    if (t == j) {
      double s = 0.0, x0 = 0.0, beta, tau, scal;
#pragma unroll
      for (int r = 0; r < MR; ++r) {
        s += r > j ? x[r] * x[r] : 0.0;
        x0 = r == j ? x[r] : x0;
      }
      reflector(x0, s, beta, tau, scal);
      L.tau[j] = tau;
#pragma unroll
      for (int r = 0; r < MR; ++r) {
        V[j][r] = r > j ? x[r] * scal : (r == j ? 1.0 : 0.0);
        x[r] = r == j ? beta : x[r];
      }
    }
    __syncthreads();
    if (t > j && w0 < n) apply(j);
  }
  if (w0 < n) store_r(t);
#pragma unroll 1
  for (int c = t + NQ; c < n; c += NQ) {
    load(c);
#pragma unroll 1
    for (int j = 0; j < k; ++j) apply(j);
    store_r(c);
  }
  __syncthreads();   // src is read before q, which may be the same memory, is written
  if (t < k) {
#pragma unroll
    for (int r = 0; r < MR; ++r) x[r] = r == t ? 1.0 : 0.0;
#pragma unroll 1
    for (int j = k - 1; j >= 0; --j) apply(j);
#pragma unroll
    for (int r = 0; r < MR; ++r)
      if (r < m) q[J.q_trans ? (int64_t)t * m + r : (int64_t)r * k + t] = x[r];
  }
}

// C[:, c0 .. c1) <- (I - V op(T) V^T) C over rows j0 .. m - 1 (C column-major,
// leading dimension m; op(T) = T^T if trans); each wave takes 16 columns.
__device__ __forceinline__ void qr_apply(double TNX_GLOBAL* C, int c0, int c1, int j0, int m, QrLds& L,
                                         bool trans) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4, ldp = m + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int ct = c0 + 16 * wave; ct < c1; ct += 16 * (NQ / 64)) {
    const bool ok = ct + i < c1;
    double TNX_GLOBAL* col = C + (int64_t)(ok ? ct + i : ct) * m;
    tnx_d4 w1 = {0, 0, 0, 0}, w2 = {0, 0, 0, 0};
    for (int r0 = j0; r0 < m; r0 += 8) {   // V^T C, lane group g: rows 2 g, 2 g + 1
      const int r = r0 + 2 * g;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int rr = min(r + h, m - 1);
        const double a = L.P[i * ldp + rr], b = col[rr];
        const bool in = r + h < m;
        w1 = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? a : 0.0, in && ok ? b : 0.0, w1, 0, 0, 0);
      }
    }
    // w1's register s holds rows 4 s + g: the k of MFMA s as it is
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w2 = __builtin_amdgcn_mfma_f64_16x16x4f64(trans ? L.T[4 * s + g][i] : L.T[i][4 * s + g], -w1[s],
                                                w2, 0, 0, 0);
    for (int r0 = j0; r0 < m; r0 += 16) {
      tnx_d4 d;
#pragma unroll
      for (int r = 0; r < 4; ++r) d[r] = col[min(r0 + g + 4 * r, m - 1)];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const double a = L.P[(4 * s + g) * ldp + min(r0 + i, m - 1)];
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(a, w2[s], d, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (ok && r0 + g + 4 * r < m) col[r0 + g + 4 * r] = d[r];
    }
  }
}

// T of the block reflector H_0 ... H_15 = I - V T V^T from V (L.P) and tau
// (columns past the block have V = 0 and tau = 0)
__device__ __forceinline__ void qr_form_t(int j0, int jb, int m, QrLds& L) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4, ldp = m + 1;
  if (threadIdx.x < 64) {
    tnx_d4 s4 = {0, 0, 0, 0};
    for (int r0 = j0; r0 < m; r0 += 4) {
      const double v = L.P[i * ldp + min(r0 + g, m - 1)];
      const double x = r0 + g < m ? v : 0.0;
      s4 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, x, s4, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) L.S[g + 4 * r][i] = s4[r];
    __builtin_amdgcn_wave_barrier();
    // column c of T: T[a][c] = -tau_c sum_b T[a][b] S[b][c] (b < c); lane a
    // holds row a in LDS (only it reads that row)
    if (g == 0) {
#pragma unroll 1
      for (int c = 0; c < QS; ++c) {
        const double tc = c < jb ? L.tau[j0 + c] : 0.0;
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int b = 0; b < QS; ++b) s[b & 3] += b < c ? L.T[i][b] * L.S[b][c] : 0.0;
        L.T[i][c] = i == c ? tc : (i < c ? -tc * ((s[0] + s[1]) + (s[2] + s[3])) : 0.0);
      }
    }
  }
}

// column-major m x n work matrix W (ld = m); Q scratch m x k after it.
__device__ __forceinline__ void qr_blocked(const tnx_qr_job& J, QrLds& L) {
  const int m = J.m, n = J.n, k = m < n ? m : n, t = threadIdx.x, ldp = m + 1;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  double TNX_GLOBAL* W = as_global<double>(J.work);
  double TNX_GLOBAL* Q = W + (int64_t)m * n;
  for (int j0 = 0; j0 < k; j0 += QS) {
    const int jb = min(QS, k - j0), rows = m - j0;
    for (int e = t; e < QS * rows; e += NQ) {
      const int c = e / rows, r = j0 + e - c * rows;
      L.P[c * ldp + r] = c < jb ? W[(int64_t)(j0 + c) * m + r] : 0.0;
    }
    __syncthreads();
    // column jj: every wave forms the reflector from the unscaled column and
    // applies it to one column right of it
    for (int jj = 0; jj < jb; ++jj) {
      const int j = j0 + jj, c = jj + 1 + wave;
      const double* x = L.P + jj * ldp;
      if (c < jb || wave == 0) {
        double* y = L.P + (c < jb ? c : jj) * ldp;
        double s = 0.0, d = 0.0;
        for (int r = j + 1 + lane; r < m; r += 64) {
          const double xr = x[r];
          s += xr * xr;
          d += xr * y[r];
        }
        s = tnx_wave_sum(s);
        d = tnx_wave_sum(d);
        double beta, tau, scal;
        reflector(x[j], s, beta, tau, scal);
        if (t == 0) {
          L.beta[jj] = beta;
          L.scal[jj] = scal;
          L.tau[j] = tau;
        }
        if (c < jb && tau != 0.0) {
          const double f = (y[j] + scal * d) * tau, fs = f * scal;
          for (int r = j + 1 + lane; r < m; r += 64) y[r] -= fs * x[r];
          if (lane == 0) y[j] -= f;
        }
      }
      __syncthreads();
    }
    // R and V to W, V (unit lower trapezoidal) in P
    for (int e = t; e < QS * rows; e += NQ) {
      const int c = e / rows, r = j0 + e - c * rows;
      if (c >= jb) continue;
      double v = L.P[c * ldp + r];
      if (r == j0 + c) {
        W[(int64_t)(j0 + c) * m + r] = L.beta[c];
        v = 1.0;
      } else {
        if (r > j0 + c) v *= L.scal[c];
        W[(int64_t)(j0 + c) * m + r] = v;
        if (r < j0 + c) v = 0.0;
      }
      L.P[c * ldp + r] = v;
    }
    __syncthreads();
    qr_form_t(j0, jb, m, L);
    __syncthreads();
    qr_apply(W, j0 + jb, n, j0, m, L, true);
    __syncthreads();
  }
  double TNX_GLOBAL* R = as_global<double>(J.r);
  for (int64_t e = t; e < (int64_t)k * n; e += NQ) {
    const int i = (int)(e / n), c = (int)(e - (int64_t)i * n);
    R[e] = (i <= c) ? W[(int64_t)c * m + i] : 0.0;
  }
  // Q = H_0 ... H_{k-1} [I_k; 0], the blocks in reverse
  for (int64_t e = t; e < (int64_t)m * k; e += NQ) {
    const int c = (int)(e / m), r = (int)(e - (int64_t)c * m);
    Q[e] = (r == c) ? 1.0 : 0.0;
  }
  for (int j0 = (k - 1) / QS * QS; j0 >= 0; j0 -= QS) {
    const int jb = min(QS, k - j0), rows = m - j0;
    for (int e = t; e < QS * rows; e += NQ) {
      const int c = e / rows, r = j0 + e - c * rows;
      L.P[c * ldp + r] = c >= jb || r < j0 + c ? 0.0 : r == j0 + c ? 1.0 : W[(int64_t)(j0 + c) * m + r];
    }
    __syncthreads();
    qr_form_t(j0, jb, m, L);
    __syncthreads();
    qr_apply(Q, j0, k, j0, m, L, false);
    __syncthreads();
  }
}

// column by column: each reflector by one wave, its columns by all of them
__device__ __forceinline__ void qr_columns(const tnx_qr_job& J, QrLds& L) {
  const int m = J.m, n = J.n, k = m < n ? m : n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double TNX_GLOBAL* W = as_global<double>(J.work);
  double TNX_GLOBAL* Q = W + (int64_t)m * n;
  for (int j = 0; j < k; ++j) {
    double TNX_GLOBAL* wj = W + (int64_t)j * m;
    if (wave == 0) {
      double s = 0.0;
      for (int r = j + 1 + lane; r < m; r += 64) s += wj[r] * wj[r];
      s = tnx_wave_sum(s);
      double beta, t, scal;
      reflector(wj[j], s, beta, t, scal);
      for (int r = j + 1 + lane; r < m; r += 64) wj[r] *= scal;
      if (lane == 0) {
        wj[j] = beta;
        L.tau[j] = t;
      }
    }
    __syncthreads();
    const double tj = L.tau[j];
    if (tj != 0.0) {
      for (int c = j + 1 + wave; c < n; c += NQ / 64) {
        double TNX_GLOBAL* wc = W + (int64_t)c * m;
        double s = (lane == 0) ? wc[j] : 0.0;
        for (int r = j + 1 + lane; r < m; r += 64) s += wj[r] * wc[r];
        s = tnx_wave_sum(s) * tj;
        if (lane == 0) wc[j] -= s;
        for (int r = j + 1 + lane; r < m; r += 64) wc[r] -= s * wj[r];
      }
    }
    __syncthreads();
  }
  // R (k x n, row-major): upper triangle of W
  double TNX_GLOBAL* R = as_global<double>(J.r);
  for (int64_t e = threadIdx.x; e < (int64_t)k * n; e += NQ) {
    int i = (int)(e / n), c = (int)(e - (int64_t)i * n);
    R[e] = (i <= c) ? W[(int64_t)c * m + i] : 0.0;
  }
  // Q = H_0 ... H_{k-1} [I_k; 0], column-major m x k, backward accumulation
  for (int64_t e = threadIdx.x; e < (int64_t)m * k; e += NQ) {
    int c = (int)(e / m), r = (int)(e - (int64_t)c * m);
    Q[e] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int j = k - 1; j >= 0; --j) {
    const double tj = L.tau[j];
    if (tj != 0.0) {
      const double TNX_GLOBAL* v = W + (int64_t)j * m;  // v[j] = 1 implicit, v[r>j] stored
      for (int c = j + wave; c < k; c += NQ / 64) {
        double TNX_GLOBAL* qc = Q + (int64_t)c * m;
        double s = (lane == 0) ? qc[j] : 0.0;
        for (int r = j + 1 + lane; r < m; r += 64) s += v[r] * qc[r];
        s = tnx_wave_sum(s) * tj;
        if (lane == 0) qc[j] -= s;
        for (int r = j + 1 + lane; r < m; r += 64) qc[r] -= s * v[r];
      }
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(NQ) void qr_kernel(const tnx_qr_job* __restrict__ jobs) {
  extern __shared__ double lds[];
  QrLds& L = *(QrLds*)lds;
  const tnx_qr_job J = jobs[blockIdx.x];
  const int m = J.m, n = J.n, k = m < n ? m : n;
  if (k > KMAX || m <= 0 || n <= 0) return;  // rejected on the host
  if (m <= QS) {
    if (m <= 4) qr_small<4>(J, L);
    else if (m <= 8) qr_small<8>(J, L);
    else qr_small<QS>(J, L);
    return;
  }
  const double TNX_GLOBAL* src = as_global<const double>(J.src);
  double TNX_GLOBAL* W = as_global<double>(J.work);
  const double TNX_GLOBAL* Q = W + (int64_t)m * n;
  for (int64_t e = threadIdx.x; e < (int64_t)m * n; e += NQ) {
    int r, c;
    if (J.trans) { c = (int)(e / m); r = (int)(e - (int64_t)c * m); }   // src[c*ld+r] contiguous in r
    else { r = (int)(e / n); c = (int)(e - (int64_t)r * n); }           // src[r*ld+c] contiguous in c
    W[(int64_t)c * m + r] = src_at(src, J.ld, J.trans, r, c);
  }
  __syncthreads();
  if (m <= QB_MAX && k >= QS) qr_blocked(J, L);
  else qr_columns(J, L);
  double TNX_GLOBAL* q = as_global<double>(J.q);
  if (J.q_trans) {
    for (int64_t e = threadIdx.x; e < (int64_t)m * k; e += NQ) q[e] = Q[e];
  } else {
    for (int64_t e = threadIdx.x; e < (int64_t)m * k; e += NQ) {
      int r = (int)(e / k), c = (int)(e - (int64_t)r * k);
      q[e] = Q[(int64_t)c * m + r];
    }
  }
}

// ------------------------------------------------ one-sided Jacobi SVD
// W (m x n) and V (n x n), both column-major, in LDS when they fit
// (SVD_LDS bytes: n = 80 for a square matrix) and in the job's work area
// otherwise.  SVD_T = 16 lanes rotate a column pair, so the pairs of a round
// run side by side up to n = 128; more lanes only repeat the scalar part of a
// rotation, which is most of it (order 64: 64 lanes a pair 2.0 ms, 16 0.85).
// Bound: a rotation's reductions and angle (latency).  ms (MI355X), four
// wavefronts on columns in global memory -> this: order 16 0.32 -> 0.08, 32
// 1.5 -> 0.24, 64 6.5 -> 0.85, with singular values over 20 decades 17.3 ->
// 2.4, 128 (not in LDS) 37 -> 12.  Putting the larger column of a pair first,
// as the block Jacobi does, costs sweeps here (1.2 ms at 64).
constexpr size_t SVD_LDS = 100 * 1024;
constexpr int SVD_T = 16;
// the SVD by way of a QR: rows, and columns, at most (SVD_LDS holds m n + 2 n^2
// doubles, m >= n)
constexpr int SVD_QR_M = 256;
constexpr int SVD_QR_N = 65;
static_assert(3 * 8 * SVD_QR_N * SVD_QR_N <= (int)SVD_LDS &&
                  3 * 8 * (SVD_QR_N + 1) * (SVD_QR_N + 1) > (int)SVD_LDS, "the largest square");
constexpr int SVD_TOP = 240;

// sum over the 16 lanes of a row
__device__ __forceinline__ double row_sum(double v) {
  v += tnx_row_get<0x128>(v);
  v += tnx_row_get<0x124>(v);
  v += tnx_row_get<0x122>(v);
  return v + tnx_row_get<0x121>(v);
}

// and over T lanes, a row or the wavefront
template <int T> __device__ __forceinline__ double lane_sum(double v) {
  static_assert(T == 16 || T == 64, "a row or a wavefront");
  if constexpr (T == 64) return tnx_wave_sum(v);
  else return row_sum(v);
}

// Rotates the columns of W (m x n) until they are orthogonal, V (n x n) along; T
// (16 or 64) lanes a pair.  64 where the 16 wavefronts hold all pairs of a round
// at once (n <= 32): 300 x 20 over 10 decades 676 us with 16 and 416 with 64,
// 1024 x 7 269 and 93 (230 by four wavefronts on columns in global memory), 280 x
// 30 534 and 440.
template <int T, typename PW>
__device__ __forceinline__ void jacobi_sweeps(PW W, int m, PW V, int n, double eps, int max_sweeps,
                                              int& rotated) {
  const int l = threadIdx.x & (T - 1);
  const int np = (n + 1) & ~1;  // players in the round-robin tournament
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    if (threadIdx.x == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      for (int p = threadIdx.x / T; p < np / 2; p += NQ / T) {
        // circle method: player np-1 fixed, others rotate
        int a = (p == 0) ? np - 1 : (round + p) % (np - 1);
        int b = (round + np - 1 - p) % (np - 1);
        if (p == 0) b = round % (np - 1);
        if (a >= n || b >= n || a == b) continue;
        if (a > b) { int t = a; a = b; b = t; }
        const PW wa = W + (int64_t)a * m, wb = W + (int64_t)b * m;
        double al = 0.0, be = 0.0, ga = 0.0;
        for (int r = l; r < m; r += T) {
          const double x = wa[r], y = wb[r];
          al += x * x;
          be += y * y;
          ga += x * y;
        }
        al = lane_sum<T>(al);
        be = lane_sum<T>(be);
        ga = lane_sum<T>(ga);
        const double ab = al * be;
        const bool rot = ga != 0.0 && fabs(ga) > eps * (ab > 0.0 ? ab * __builtin_amdgcn_rsq(ab) : 0.0);
        if (rot) {
          const JacobiRot jr = jacobi_rot(al, be, ga, rot, false);
          if (l == 0) rotated = 1;
          for (int r = l; r < m; r += T) {
            double x = wa[r], y = wb[r];
            jacobi_apply(jr, x, y);
            wa[r] = x;
            wb[r] = y;
          }
          const PW va = V + (int64_t)a * n, vb = V + (int64_t)b * n;
          for (int r = l; r < n; r += T) {
            double x = va[r], y = vb[r];
            jacobi_apply(jr, x, y);
            va[r] = x;
            vb[r] = y;
          }
        }
      }
      __syncthreads();
    }
    if (rotated == 0) break;
    __syncthreads();
  }
}

// The same by the sums and rotations of a job with `in_order`: 64 lanes a pair,
// a lane's rows 64 apart, the angle by divisions and roots, and which product of
// a sum is fused said.  In LDS where it fits: order 64 with values down to rounding
// 13.5 ms in global memory, 4 ms in LDS (0.77 by way of a QR).
template <typename PW>
__device__ __forceinline__ void jacobi_sweeps_in_order(PW W, int m, PW V, int n, double eps,
                                                       int max_sweeps, int& rotated) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int np = (n + 1) & ~1;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    if (threadIdx.x == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      for (int p = wave; p < np / 2; p += NQ / 64) {
        int a = (p == 0) ? np - 1 : (round + p) % (np - 1);
        int b = (p == 0) ? round % (np - 1) : (round + np - 1 - p) % (np - 1);
        if (a >= n || b >= n || a == b) continue;
        if (a > b) { int t = a; a = b; b = t; }
        const PW wa = W + (int64_t)a * m, wb = W + (int64_t)b * m;
        double al = 0.0, be = 0.0, ga = 0.0;
        for (int r = lane; r < m; r += 64) {
          const double x = wa[r], y = wb[r];
          al = fma(x, x, al);
          be = fma(y, y, be);
          ga = fma(x, y, ga);
        }
        al = tnx_wave_sum(al);
        be = tnx_wave_sum(be);
        ga = tnx_wave_sum(ga);
        if (ga != 0.0 && fabs(ga) > eps * sqrt(al * be)) {
          if (lane == 0) rotated = 1;
          const double zeta = (be - al) / (2.0 * ga);
          const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(fma(zeta, zeta, 1.0)));
          const double cs = 1.0 / sqrt(fma(t, t, 1.0)), sn = cs * t;
          for (int r = lane; r < m; r += 64) {
            const double x = wa[r], y = wb[r];
            wa[r] = fma(cs, x, -(sn * y));
            wb[r] = fma(sn, x, cs * y);
          }
          const PW va = V + (int64_t)a * n, vb = V + (int64_t)b * n;
          for (int r = lane; r < n; r += 64) {
            const double x = va[r], y = vb[r];
            va[r] = fma(cs, x, -(sn * y));
            vb[r] = fma(sn, x, cs * y);
          }
        }
      }
      __syncthreads();
    }
    if (rotated == 0) break;
    __syncthreads();
  }
}

// The same for two n x n matrices in LDS, n <= 16 NE: a lane's NE elements of the
// pair's columns of W and V stay in registers from the dot products to the
// store, all reads ahead of the angle.  Bound: latency, one such chain a round
// (order 64 over 10 decades 659 us in all, some 180 more with the elements read again for
// each use and the pair found by remainders; 8 or 32 lanes a pair 980 and 890).
template <int NE>
__device__ __forceinline__ void jacobi_sweeps_lds(double* W, double* V, int n, double eps,
                                                  int max_sweeps, int& rotated) {
  const int l = threadIdx.x & (SVD_T - 1), p = threadIdx.x / SVD_T;
  const int np = (n + 1) & ~1;   // players in the round-robin tournament
  static_assert(NQ / SVD_T >= SVD_QR_N / 2, "every pair of a round at once");
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    if (threadIdx.x == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      // circle method: player np-1 fixed, others rotate
      int a = round + p, b = round + np - 1 - p;
      a = p == 0 ? np - 1 : a >= np - 1 ? a - (np - 1) : a;
      b = p == 0 ? round : b >= np - 1 ? b - (np - 1) : b;
      if (p < np / 2 && max(a, b) < n) {
        const int u = min(a, b), v = max(a, b);
        double* wa = W + u * n;
        double* wb = W + v * n;
        double* va = V + u * n;
        double* vb = V + v * n;
        double x[NE], y[NE], xv[NE], yv[NE];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
          const int r = min(l + SVD_T * e, n - 1);
          x[e] = wa[r];
          y[e] = wb[r];
          xv[e] = va[r];
          yv[e] = vb[r];
        }
        double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
        for (int e = 0; e < NE; ++e)
          if (l + SVD_T * e < n) {
            al += x[e] * x[e];
            be += y[e] * y[e];
            ga += x[e] * y[e];
          }
        al = row_sum(al);
        be = row_sum(be);
        ga = row_sum(ga);
        const double ab = al * be;
        const bool rot = ga != 0.0 && fabs(ga) > eps * (ab > 0.0 ? ab * __builtin_amdgcn_rsq(ab) : 0.0);
        if (rot) {
          const JacobiRot jr = jacobi_rot(al, be, ga, rot, false);
          if (l == 0) rotated = 1;
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            jacobi_apply(jr, x[e], y[e]);
            jacobi_apply(jr, xv[e], yv[e]);
            if (l + SVD_T * e < n) {
              const int r = l + SVD_T * e;
              wa[r] = x[e];
              wb[r] = y[e];
              va[r] = xv[e];
              vb[r] = yv[e];
            }
          }
        }
      }
      __syncthreads();
    }
    if (rotated == 0) break;
    __syncthreads();
  }
}

// Squares of entries below a norm^2 of SQ_SMALL lose bits to underflow: such a
// norm is formed from the entries over a power of two near the largest.
constexpr double SQ_SMALL = 1e-280;

// Exponent of the largest entry of a wavefront's vector, ROWS a lane.
template <int ROWS> __device__ __forceinline__ int column_exp(const double (&v)[ROWS]) {
  double big = 0.0;
#pragma unroll
  for (int t = 0; t < ROWS; ++t) big = fmax(big, fabs(v[t]));
  return __builtin_amdgcn_frexp_exp(
      tnx_wave_fold(big, [](double x, double y) { return fmax(x, y); }));
}

// What stands for the norm^2 of such a vector: below SQ_SMALL, above zero if any
// entry is, rising with the norm (its logarithm, linear between powers of two).
template <int ROWS> __device__ __forceinline__ double small_key(const double (&v)[ROWS]) {
  const int e = column_exp(v);
  double s = 0.0;
#pragma unroll
  for (int t = 0; t < ROWS; ++t) {
    const double x = __builtin_amdgcn_ldexp(v[t], -e);
    s += x * x;
  }
  s = sqrt(tnx_wave_sum(s));
  if (s == 0.0) return 0.0;
  const int e2 = __builtin_amdgcn_frexp_exp(s);
  const double f = (double)(e + e2) + 2.0 * __builtin_amdgcn_ldexp(s, -e2);
  return SQ_SMALL * (0.5 + f * (1.0 / 4096.0));
}

// Singular values sv (LDS) = column norms of W, order = their descending order.
template <bool SCALE, typename PW>
__device__ __forceinline__ void sort_columns(PW W, int m, int n, double* sv, int* order) {
  const int lane = threadIdx.x & 63;
  for (int c = threadIdx.x >> 6; c < n; c += NQ / 64) {
    const PW wc = W + (int64_t)c * m;
    double s = 0.0;
    for (int r = lane; r < m; r += 64) s += wc[r] * wc[r];
    s = tnx_wave_sum(s);
    int ex = 0;
    if constexpr (SCALE) {
      if (s < SQ_SMALL) {
        double big = 0.0;
        for (int r = lane; r < m; r += 64) big = fmax(big, fabs(wc[r]));
        ex = __builtin_amdgcn_frexp_exp(
            tnx_wave_fold(big, [](double x, double y) { return fmax(x, y); }));
        s = 0.0;
        for (int r = lane; r < m; r += 64) {
          const double x = __builtin_amdgcn_ldexp(wc[r], -ex);
          s += x * x;
        }
        s = tnx_wave_sum(s);
      }
    }
    if (lane == 0) {
      sv[c] = SCALE ? __builtin_amdgcn_ldexp(sqrt(s), ex) : sqrt(s);
      order[c] = c;   // (values that do not compare leave entries unset below)
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < n; c += NQ) {
    int rank = 0;
    const double x = sv[c];
    for (int o = 0; o < n; ++o) rank += (sv[o] > x) || (sv[o] == x && o < c);
    order[rank] = c;
  }
  __syncthreads();
}

template <bool IN_ORDER, typename PW>
__device__ __forceinline__ void svd_body(const tnx_svd_job& J, int max_sweeps, PW W, PW V, double* sv,
                                         int* order, int& rotated) {
  const int m = J.m, n = J.n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int NW = NQ / 64;
  const double TNX_GLOBAL* src = as_global<const double>(J.src);

  for (int64_t e = threadIdx.x; e < (int64_t)m * n; e += NQ) {
    int r, c;
    if (J.trans) { c = (int)(e / m); r = (int)(e - (int64_t)c * m); }
    else { r = (int)(e / n); c = (int)(e - (int64_t)r * n); }
    W[(int64_t)c * m + r] = src_at(src, J.ld, J.trans, r, c);
  }
  for (int64_t e = threadIdx.x; e < (int64_t)n * n; e += NQ) {
    int c = (int)(e / n), r = (int)(e - (int64_t)c * n);
    V[e] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();

  // rotate while |a.b| > m*eps*|a||b| (columns orthogonal to working accuracy)
  const double eps = 2.220446049250313e-16 * (double)(m > 8 ? m : 8);
  if constexpr (IN_ORDER) jacobi_sweeps_in_order(W, m, V, n, eps, max_sweeps, rotated);
  else if (n <= 2 * (NQ / 64)) jacobi_sweeps<64>(W, m, V, n, eps, max_sweeps, rotated);
  else jacobi_sweeps<SVD_T>(W, m, V, n, eps, max_sweeps, rotated);
  sort_columns<false>(W, m, n, sv, order);
  double TNX_GLOBAL* s_out = as_global<double>(J.s);
  double TNX_GLOBAL* u = as_global<double>(J.u);
  double TNX_GLOBAL* svt = as_global<double>(J.svt);
  for (int i = threadIdx.x; i < n; i += NQ) s_out[i] = sv[order[i]];
  // U columns (normalised), sorted; zero columns are completed afterwards
  for (int i = wave; i < n; i += NW) {
    const int c = order[i];
    const double sc = sv[c] > 0.0 ? 1.0 / sv[c] : 0.0;
    const PW wc = W + (int64_t)c * m;
    for (int r = lane; r < m; r += 64) {
      const double v = wc[r] * sc;
      if (J.u_trans) u[(int64_t)i * m + r] = v;
      else u[(int64_t)r * n + i] = v;
    }
  }
  // svt[i][col] = s_i * V[col][order i]
  for (int64_t e = threadIdx.x; e < (int64_t)n * n; e += NQ) {
    int i = (int)(e / n), col = (int)(e - (int64_t)i * n);
    const int c = order[i];
    svt[e] = sv[c] * V[(int64_t)c * n + col];
  }
  __syncthreads();
  // complete null columns of U (singular value exactly 0) by Gram-Schmidt
  if (wave == 0) {
    int next_unit = 0;
    for (int i = 0; i < n; ++i) {
      if (sv[order[i]] > 0.0) continue;
      for (; next_unit < m; ++next_unit) {
        // candidate e_{next_unit}, orthogonalised twice against columns != i
        for (int r = lane; r < m; r += 64) {
          const double v = (r == next_unit) ? 1.0 : 0.0;
          if (J.u_trans) u[(int64_t)i * m + r] = v; else u[(int64_t)r * n + i] = v;
        }
        for (int pass = 0; pass < 2; ++pass) {
          for (int o = 0; o < n; ++o) {
            if (o == i || (sv[order[o]] == 0.0 && o > i)) continue;
            double d = 0.0;
            for (int r = lane; r < m; r += 64) {
              const double uo = J.u_trans ? u[(int64_t)o * m + r] : u[(int64_t)r * n + o];
              const double ui = J.u_trans ? u[(int64_t)i * m + r] : u[(int64_t)r * n + i];
              d += uo * ui;
            }
            d = tnx_wave_sum(d);
            for (int r = lane; r < m; r += 64) {
              const double uo = J.u_trans ? u[(int64_t)o * m + r] : u[(int64_t)r * n + o];
              if (J.u_trans) u[(int64_t)i * m + r] -= d * uo; else u[(int64_t)r * n + i] -= d * uo;
            }
          }
        }
        double nn = 0.0;
        for (int r = lane; r < m; r += 64) {
          const double ui = J.u_trans ? u[(int64_t)i * m + r] : u[(int64_t)r * n + i];
          nn += ui * ui;
        }
        nn = tnx_wave_sum(nn);
        if (nn > 0.25) {
          const double sc = 1.0 / sqrt(nn);
          for (int r = lane; r < m; r += 64) {
            if (J.u_trans) u[(int64_t)i * m + r] *= sc; else u[(int64_t)r * n + i] *= sc;
          }
          ++next_unit;
          break;
        }
      }
    }
  }
}

// The same by way of M P = Q R (Householder, the largest remaining column
// first): the columns of X = R^T are rotated, X W = B, so that M = Q W B^T P^T,
// u = Q W, diag(s) vt = B^T P^T.  With singular values that decay the columns of
// X start nearly sorted and nearly orthogonal, those of M do not: 24 sweeps
// become 7 (order 64, values over 10 or 16 decades), 10 of a random matrix 9,
// and a tall M is rotated as an n x n matrix.  u comes out orthonormal whatever
// the rank.  A (m x n), X and V (n x n) in LDS, m <= 64 ROWS.  M is scaled by a
// power of two, its largest entry to 2^SVD_TOP: products of two columns' norms^2
// (n <= 65, m <= 256) stay below 2^1024, and squares keep their bits down to
// columns 1e-210 of the largest.  A reflector is formed from its column over a
// power of two of its own, so that its products with any other column stay in range.
// us (MI355X), columns of M -> this: order 64 with values over 10 decades 2030 ->
// 659, random 840 -> 699; 128 x 40 over 10 decades 1150 -> 312, random 550 ->
// 351; order 16 132 -> 68, random 84 -> 73; order 8 41 -> 31.
template <int ROWS>
__device__ __forceinline__ void svd_body_qr(const tnx_svd_job& J, int max_sweeps, double* A, double* X,
                                            double* V, double* sv, int* order, int& rotated) {
  const int m = J.m, n = J.n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int NW = NQ / 64;
  // nrm: norms^2 of the remaining columns, two copies.  Step k reads one and
  // writes the other, so that a wave which comes to its choice late chooses
  // from the same norms as the rest (the waves' orders must not differ).
  __shared__ double nrm[2][SVD_QR_N], v0s[SVD_QR_N], fs[SVD_QR_N], beta[SVD_QR_N];
  __shared__ int vex[SVD_QR_N];   // power of two of reflector k
  const double TNX_GLOBAL* src = as_global<const double>(J.src);
  double big = 0.0;
  for (int64_t e = threadIdx.x; e < (int64_t)m * n; e += NQ) {
    int r, c;
    if (J.trans) { c = (int)(e / m); r = (int)(e - (int64_t)c * m); }
    else { r = (int)(e / n); c = (int)(e - (int64_t)r * n); }
    const double x = src_at(src, J.ld, J.trans, r, c);
    A[(int64_t)c * m + r] = x;
    big = fmax(big, fabs(x));
  }
  big = tnx_wave_fold(big, [](double x, double y) { return fmax(x, y); });
  if (lane == 0) sv[wave] = big;
  __syncthreads();
  big = sv[lane & (NW - 1)];
  big = tnx_wave_fold(big, [](double x, double y) { return fmax(x, y); });
  const int ex = __builtin_amdgcn_frexp_exp(big) - SVD_TOP;
  for (int e = threadIdx.x; e < m * n; e += NQ) A[e] = __builtin_amdgcn_ldexp(A[e], -ex);
  for (int e = threadIdx.x; e < n * n; e += NQ) {
    const int c = e / n;
    V[e] = (e - c * n == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int c = wave; c < n; c += NW) {
    double y[ROWS], t = 0.0;
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      y[q] = lane + 64 * q < m ? A[c * m + lane + 64 * q] : 0.0;
      t += y[q] * y[q];
    }
    t = tnx_wave_sum(t);
    if (t < SQ_SMALL) t = small_key<ROWS>(y);
    if (lane == 0) nrm[0][c] = t;
  }
  __syncthreads();
  // pivoted order, a copy per wave: lane j has the column at position j, and
  // that at 64 + j
  int p0 = lane, p1 = 64 + lane;
  auto at = [&](int j) {
    return j < 64 ? __builtin_amdgcn_readlane(p0, j) : __builtin_amdgcn_readlane(p1, j - 64);
  };
  for (int k = 0; k < n; ++k) {
    // position of the largest remaining column (the first of equal ones)
    const double* now = nrm[k & 1];
    const bool in0 = lane >= k && lane < n, in1 = 64 + lane >= k && 64 + lane < n;
    const double n0 = in0 ? now[p0] : -1.0;
    const double n1 = in1 ? now[p1] : -1.0;
    const double top = tnx_wave_fold(fmax(n0, n1), [](double x, double y) { return fmax(x, y); });
    // (only positions that remain: where all of their norms are NaN, top is the
    // -1 of the others)
    const unsigned long long m0 = __ballot(in0 && n0 == top), m1 = __ballot(in1 && n1 == top);
    const int best = m0 ? __builtin_ctzll(m0) : m1 ? 64 + __builtin_ctzll(m1) : k;   // (NaN: k)
    const int ck = at(k), cb = at(best);
    if (lane == (k & 63)) (k < 64 ? p0 : p1) = cb;
    if (lane == (best & 63)) (best < 64 ? p0 : p1) = ck;
    // reflector I - f v v^T, v = (x_k - beta, x_{k+1}, ...)
    const double* x = A + cb * m;
    double v[ROWS], ss = 0.0;
#pragma unroll
    for (int t = 0; t < ROWS; ++t) {
      const int r = lane + 64 * t;
      v[t] = r >= k && r < m ? x[r] : 0.0;
      ss += v[t] * v[t];
    }
    ss = tnx_wave_sum(ss);
    int e = __builtin_amdgcn_frexp_exp(ss) >> 1;
    const bool small = ss < SQ_SMALL;   // (the same in every lane)
    if (small) e = column_exp(v);
    ss = __builtin_amdgcn_ldexp(ss, -2 * e);
#pragma unroll
    for (int t = 0; t < ROWS; ++t) v[t] = __builtin_amdgcn_ldexp(v[t], -e);
    if (small) {
      ss = 0.0;
#pragma unroll
      for (int t = 0; t < ROWS; ++t) ss += v[t] * v[t];
      ss = tnx_wave_sum(ss);
    }
    const double xk = __builtin_amdgcn_ldexp(x[k], -e), nx = sqrt(ss);
    const double b = xk > 0.0 ? -nx : nx, v0 = xk - b;
    const double f = nx > 0.0 ? 1.0 / (nx * (nx + fabs(xk))) : 0.0;
#pragma unroll
    for (int t = 0; t < ROWS; ++t)
      if (lane + 64 * t == k) v[t] = v0;
    if (threadIdx.x == 0) {
      v0s[k] = v0;
      fs[k] = f;
      beta[k] = __builtin_amdgcn_ldexp(b, e);
      vex[k] = e;
    }
    for (int j = k + 1 + wave; j < n; j += NW) {
      double* a = A + at(j) * m;
      double y[ROWS], d = 0.0, t2 = 0.0;
#pragma unroll
      for (int t = 0; t < ROWS; ++t) {
        const int r = lane + 64 * t;
        y[t] = r < m ? a[r] : 0.0;
        d += v[t] * y[t];
      }
      d = f * tnx_wave_sum(d);
#pragma unroll
      for (int t = 0; t < ROWS; ++t) {
        const int r = lane + 64 * t;
        y[t] -= d * v[t];
        if (r >= k && r < m) a[r] = y[t];
        if (r > k) t2 += y[t] * y[t];
      }
      t2 = tnx_wave_sum(t2);
      if (t2 < SQ_SMALL) {
#pragma unroll
        for (int t = 0; t < ROWS; ++t)
          if (lane + 64 * t <= k || lane + 64 * t >= m) y[t] = 0.0;
        t2 = small_key<ROWS>(y);
      }
      if (lane == 0) nrm[(k & 1) ^ 1][at(j)] = t2;
    }
    __syncthreads();
  }
  // X: column i is row i of R; the reflectors (rows below) over their powers
  for (int i = wave; i < n; i += NW) {
    for (int c = lane; c < n; c += 64) {
      const int pc = c < 64 ? p0 : p1;   // (c = lane or 64 + lane)
      X[i * n + c] = c > i ? A[pc * m + i] : c == i ? beta[i] : 0.0;
    }
    double* x = A + at(i) * m;
    for (int r = i + 1 + lane; r < m; r += 64) x[r] = __builtin_amdgcn_ldexp(x[r], -vex[i]);
  }
  __syncthreads();
  const double eps = 2.220446049250313e-16 * (double)(m > 8 ? m : 8);
  if (n <= 16) jacobi_sweeps_lds<1>(X, V, n, eps, max_sweeps, rotated);
  else if (n <= 32) jacobi_sweeps_lds<2>(X, V, n, eps, max_sweeps, rotated);
  else if (n <= 48) jacobi_sweeps_lds<3>(X, V, n, eps, max_sweeps, rotated);
  else if (n <= 64) jacobi_sweeps_lds<4>(X, V, n, eps, max_sweeps, rotated);
  else jacobi_sweeps_lds<5>(X, V, n, eps, max_sweeps, rotated);
  sort_columns<true>(X, n, n, sv, order);
  double TNX_GLOBAL* s_out = as_global<double>(J.s);
  double TNX_GLOBAL* u = as_global<double>(J.u);
  double TNX_GLOBAL* svt = as_global<double>(J.svt);
  for (int i = threadIdx.x; i < n; i += NQ) s_out[i] = __builtin_amdgcn_ldexp(sv[order[i]], ex);
  for (int i = wave; i < n; i += NW) {
    const int c = order[i];
    for (int q = lane; q < n; q += 64) 
      svt[(int64_t)i * n + (q < 64 ? p0 : p1)] = __builtin_amdgcn_ldexp(X[c * n + q], ex);
    double z[ROWS];
#pragma unroll
    for (int t = 0; t < ROWS; ++t) {
      const int r = lane + 64 * t;
      z[t] = r < n ? V[c * n + r] : 0.0;
    }
    for (int k = n - 1; k >= 0; --k) {
      const double* x = A + at(k) * m;
      const double v0 = v0s[k];
      double v[ROWS], d = 0.0;
#pragma unroll
      for (int t = 0; t < ROWS; ++t) {
        const int r = lane + 64 * t;
        v[t] = r > k && r < m ? x[r] : r == k ? v0 : 0.0;
        d += v[t] * z[t];
      }
      d = fs[k] * tnx_wave_sum(d);
#pragma unroll
      for (int t = 0; t < ROWS; ++t) z[t] -= d * v[t];
    }
#pragma unroll
    for (int t = 0; t < ROWS; ++t) {
      const int r = lane + 64 * t;
      if (r < m) {
        if (J.u_trans) u[(int64_t)i * m + r] = z[t];
        else u[(int64_t)r * n + i] = z[t];
      }
    }
  }
}

__global__ __launch_bounds__(NQ) void svd_kernel(const tnx_svd_job* __restrict__ jobs, int max_sweeps) {
  extern __shared__ double lds[];
  __shared__ int rotated;
  __shared__ double sv[KMAX];
  __shared__ int order[KMAX];
  const tnx_svd_job J = jobs[blockIdx.x];
  const int m = J.m, n = J.n;
  if (n > KMAX || m < n || n <= 0) return;  // rejected on the host
  const int64_t wn = (int64_t)m * n;
  const bool columns_fit = (wn + (int64_t)n * n) * (int64_t)sizeof(double) <= (int64_t)SVD_LDS;
  double TNX_GLOBAL* W = as_global<double>(J.work);
  if (J.in_order) {
    if (columns_fit) svd_body<true>(J, max_sweeps, lds, lds + wn, sv, order, rotated);
    else svd_body<true>(J, max_sweeps, W, W + wn, sv, order, rotated);
  } else if (m <= SVD_QR_M && n <= SVD_QR_N &&
      (wn + 2 * (int64_t)n * n) * (int64_t)sizeof(double) <= (int64_t)SVD_LDS) {
    double *X = lds + wn, *V = X + n * n;
    if (m <= 64) svd_body_qr<1>(J, max_sweeps, lds, X, V, sv, order, rotated);
    else if (m <= 128) svd_body_qr<2>(J, max_sweeps, lds, X, V, sv, order, rotated);
    else svd_body_qr<4>(J, max_sweeps, lds, X, V, sv, order, rotated);
  } else if (columns_fit) {
    svd_body<false>(J, max_sweeps, lds, lds + wn, sv, order, rotated);
  } else {
    svd_body<false>(J, max_sweeps, W, W + wn, sv, order, rotated);
  }
}

// Cholesky factor + inverse of one n x n SPD matrix (n <= 128), 1024 lanes,
// in 16 x 16 blocks (nb = ceil(n / 16) block rows; the padding is the
// identity).  Right-looking, with the inverse carried along: eliminating
// [S | I] = R^T [R | F] gives R and F = R^{-T}, so R^{-1} = F^T comes out of
// the same steps.  Per panel p:
//   1. the owner wave of the diagonal block factors S_pp = R_pp^T R_pp in
//      registers, a column a lane, F_pp = R_pp^{-T} from the same steps;
//   2. row panel p on MFMA: R_pb = F_pp S_pb (b > p), F_pe = F_pp E_pe (e < p);
//   3. trailing update on MFMA: S_ab -= R_pa^T R_pb (p < a <= b) and
//      E_ae -= R_pa^T F_pe (a > p, e <= p).
// The 8 x 8 blocks (the upper part S -> R, the strictly lower one E -> F) are
// dealt to the 4 x 4 waves cyclically, four accumulator blocks a wave.  The
// owner of the next diagonal block updates it first and factors it while the
// other waves finish the trailing update; two barriers per panel.  An
// accumulator block is in the layout of the MFMA's B operand, so the row panel
// is formed in its owners' registers.  LDS holds the row panels as they are
// formed (R above the diagonal, F below it, F_pp in its own buffer), which are
// the operands of the later phases and the output at the end.
// Bound: the serial chain of the diagonal blocks, 16 pivots each.  us (MI355X),
// with 256 lanes and the diagonal block in the MFMA layout, its rows moved by
// lane shuffles, and now: n = 128 57 and 30, the chains of a run at chi 64
// (n <= 128) 18.9 and 12.7, at chi 16 (n <= 32) 6.3 and 4.8.
constexpr int NC = 1024;
constexpr int CHOL_NMAX = 128;
constexpr double CHOL_NEAR_ID = 1e-10;  // largest |S - I| entry of the first-order path
constexpr int CB_LD = CHOL_NMAX + 1;    // LDS row stride: row and column reads hit distinct banks
constexpr int CB_XLD = 17;              // row stride of the F_pp blocks
constexpr size_t CHOL_LDS = sizeof(double) * (CHOL_NMAX * CB_LD + 8 * 16 * CB_XLD);

// 16 x 16 block in the MFMA output layout: row (lane / 16) + 4 r, column lane % 16
__device__ __forceinline__ tnx_d4 chol_ld(const double* p, int ld, int lane) {
  tnx_d4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = p[((lane >> 4) + 4 * r) * ld + (lane & 15)];
  return v;
}
__device__ __forceinline__ void chol_st(double* p, int ld, int lane, tnx_d4 v) {
#pragma unroll
  for (int r = 0; r < 4; ++r) p[((lane >> 4) + 4 * r) * ld + (lane & 15)] = v[r];
}

// acc += sgn * A B over K = 16, A[m][k] = pa[m * sam + k * sak], B[k][n] = pb[k * sbk + n]
__device__ __forceinline__ tnx_d4 chol_mma(tnx_d4 acc, const double* pa, int sam, int sak,
                                           const double* pb, int sbk, int lane, double sgn) {
  const int mn = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < 16; kk += 4) {
    const double av = sgn * pa[mn * sam + (kk + kq) * sak];
    const double bv = pb[(kk + kq) * sbk + mn];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc, 0, 0, 0);
  }
  return acc;
}

__device__ __forceinline__ double chol_readlane(double v, int l) {
  const long long x = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)x, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(x >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// What a pivot that is not positive (or NaN) is replaced by: the smallest normal
// number, so that fmax leaves every other pivot as it is (a compare and selects
// instead of it take 4% of the kernel).
constexpr double CHOL_TINY = 2.2250738585072014e-308;

// The diagonal block D (LDS, 16 rows of CB_LD) -> R_pp with zeros below the
// diagonal; F (16 rows of CB_XLD) = R_pp^{-T}.  One wave: lane j < 16 holds
// column j of D, lane 16 + j that of E (the identity at first).  Step k: row k
// of both times 1 / sqrt(D[k][k]); rows i > k lose R[k][i], a lane's value read
// into a scalar, times row k.  Row k + 1 goes first, so that the root of its
// pivot is under way while the others are updated.
__device__ __forceinline__ void chol_diag(double* D, double* F, int lane, int& bad) {
  const int j = lane & 15;
  const bool inv = lane & 16;
  double d[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) d[i] = inv ? (i == j ? 1.0 : 0.0) : D[i * CB_LD + j];
  double piv = chol_readlane(d[0], 0);
  double x = fmax(piv, CHOL_TINY), y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    bad |= !(piv > 0.0);
    // sqrt(piv) = piv / sqrt(piv): one root on the serial chain
    d[k] = (lane == k ? x : d[k]) * tnx_rsqrt_step(x, y);
    if (k == 15) break;
    d[k + 1] = fma(-chol_readlane(d[k], k + 1), d[k], d[k + 1]);
    piv = chol_readlane(d[k + 1], k + 1);
    x = fmax(piv, CHOL_TINY);
    y = __builtin_amdgcn_rsq(x);
    __builtin_amdgcn_sched_barrier(0);
    double r[16];
#pragma unroll
    for (int i = k + 2; i < 16; ++i) r[i] = chol_readlane(d[k], i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = k + 2; i < 16; ++i) d[i] = fma(-r[i], d[k], d[i]);
  }
  if (lane < 32) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (inv) F[i * CB_XLD + j] = d[i];
      else D[i * CB_LD + j] = i <= j ? d[i] : 0.0;
    }
  }
}

__global__ __launch_bounds__(NC) void chol_inv_kernel(const tnx_chol_job* __restrict__ jobs) {
  extern __shared__ double lds[];
  double* Sl = lds;                          // CHOL_NMAX rows of CB_LD
  double* Xd = lds + CHOL_NMAX * CB_LD;      // F_pp, 16 rows of CB_XLD per panel
  const tnx_chol_job J = jobs[blockIdx.x];
  const int n = J.n;
  if (n <= 0 || n > CHOL_NMAX) return;  // rejected on the host
  const int ld = J.ld > 0 ? J.ld : n;
  const int nb = (n + 15) >> 4, np = 16 * nb;
  __shared__ double red[2][NC / 64];
  __shared__ int bad_s;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // G padded with the identity; trace (shift) and largest |G - I| entry
  constexpr int NR = CHOL_NMAX / (NC / 64);   // rows of a wave
  double trace = 0.0, emax = 0.0;
  {
    const double TNX_GLOBAL* G = as_global<const double>(J.g);
    double v[NR][2];
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      if (NC / 64 * t >= np) break;
      const double TNX_GLOBAL* row = G + (int64_t)min(wave + NC / 64 * t, n - 1) * ld;
#pragma unroll
      for (int c = 0; c < 2; ++c) v[t][c] = row[(unsigned)min(lane + 64 * c, n - 1)];
    }
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      if (NC / 64 * t >= np) break;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int i = wave + NC / 64 * t, j = lane + 64 * c;
        const double id = i == j ? 1.0 : 0.0;
        if (i < n && j < n) {
          if (i == j) trace += v[t][c];
          emax = fmax(emax, fabs(v[t][c] - id));
        } else {
          v[t][c] = id;
        }
        if (i < np && j < np) Sl[i * CB_LD + j] = v[t][c];
      }
    }
  }
  trace = tnx_wave_sum(trace);
  emax = tnx_wave_fold(emax, [](double x, double y) { return fmax(x, y); });
  if (lane == 0) {
    red[0][wave] = trace;
    red[1][wave] = emax;
  }
  if (threadIdx.x == 0) bad_s = 0;
  __syncthreads();
  double tsum = 0.0, em = 0.0;
#pragma unroll
  for (int w = 0; w < NC / 64; ++w) {
    tsum += red[0][w];
    em = fmax(em, red[1][w]);
  }
  const double shift =
      J.shift_scale * (J.shift_ref ? *as_global<const double>(J.shift_ref) : tsum);
  double TNX_GLOBAL* R = as_global<double>(J.r);
  double TNX_GLOBAL* Ri = as_global<double>(J.rinv);
  // Near-identity Gram matrix (the last pass of CholeskyQR3, whose panel is
  // already orthonormal to working accuracy): with S = I + E, ||E||_max <=
  // CHOL_NEAR_ID and no shift, R = I + U (U = strict upper part of E plus
  // half its diagonal) and R^{-1} = I - U hold up to O(E^2) <= 1e-20, below
  // the rounding of the factorisation, and need no sequential steps.
  if (shift == 0.0 && em <= CHOL_NEAR_ID) {
    for (int i = wave; i < n; i += NC / 64)
      for (int j = lane; j < n; j += 64) {
        const double sv = Sl[i * CB_LD + j];
        const double u = j > i ? sv : (j == i ? 0.5 * (sv - 1.0) : 0.0);
        const double id = (i == j) ? 1.0 : 0.0;
        R[(int64_t)i * ld + j] = id + u;
        Ri[(int64_t)i * ld + j] = id - u;
      }
    if (threadIdx.x == 0 && J.status != 0) *(int32_t*)J.status = 0;
    return;
  }
  // block (sa, sb) of slot s: slot 0 or 3 is a diagonal block of waves 0, 5, 10, 15
  const int wa = wave >> 2, wb = wave & 3;
  tnx_d4 acc[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int sa = wa + 4 * (s >> 1), sb = wb + 4 * (s & 1);
    acc[s] = tnx_d4{0.0, 0.0, 0.0, 0.0};
    if (sa <= sb && sb < nb) {
      acc[s] = chol_ld(Sl + 16 * sa * CB_LD + 16 * sb, CB_LD, lane);
      if (sa == sb) {   // the shift on the diagonal (not on the padding)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * sa + (lane >> 4) + 4 * r;
          if ((lane >> 4) + 4 * r == (lane & 15) && i < n) acc[s][r] += shift;
        }
      }
    }
  }
  int bad = 0;
#pragma unroll 1
  for (int p = 0; p < nb; ++p) {
    int ln = lane;   // opaque: what follows from the lane is formed anew, not
    asm volatile("" : "+v"(ln));   // kept in registers (and spilled) across panels
    double* Pp = Sl + 16 * p * CB_LD;             // row panel p
    double* Fp = Xd + 16 * p * CB_XLD;
    const double* Pq = Pp - 16 * CB_LD;           // and p - 1 (p > 0)
    const double* Fq = Fp - 16 * CB_XLD;
    if (wave == 5 * (p & 3)) {   // the diagonal block: trailing update, then its factor
      __builtin_amdgcn_s_setprio(3);
      tnx_d4 dd = p < 4 ? acc[0] : acc[3];
      if (p > 0) dd = chol_mma(dd, Pq + 16 * p, 1, CB_LD, Pq + 16 * p, CB_LD, ln, -1.0);
      chol_st(Pp + 16 * p, CB_LD, ln, dd);
      __builtin_amdgcn_wave_barrier();
      chol_diag(Pp + 16 * p, Fp, ln, bad);
      __builtin_amdgcn_s_setprio(0);
    }
    if (p > 0) {   // trailing update of panel p - 1
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int sa = wa + 4 * (s >> 1), sb = wb + 4 * (s & 1);
        if (sa < p || sa >= nb || sb >= nb || (sa == p && sb == p)) continue;
        if (sb < sa && sb >= p) continue;   // E_ab starts with panel b
        const bool diag = sb == p - 1;
        acc[s] = chol_mma(acc[s], Pq + 16 * sa, 1, CB_LD, diag ? Fq : Pq + 16 * sb,
                          diag ? CB_XLD : CB_LD, ln, -1.0);
      }
    }
    __syncthreads();
    // R_pb = F_pp S_pb, F_pe = F_pp E_pe
    if (wa == (p & 3)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int sa = wa + 4 * (s >> 1), sb = wb + 4 * (s & 1);
        if (sa != p || sb == p || sb >= nb) continue;
        tnx_d4 c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          c = __builtin_amdgcn_mfma_f64_16x16x4f64(Fp[(ln & 15) * CB_XLD + 4 * r + (ln >> 4)],
                                                   acc[s][r], c, 0, 0, 0);
        chol_st(Pp + 16 * sb, CB_LD, ln, c);
      }
    }
    __syncthreads();
  }
  if (bad && lane == 0) bad_s = 1;
  __syncthreads();
  // R (upper) and R^{-1} = F^T: F_pp from its buffer, the blocks below the
  // diagonal of F from the lower part of Sl
  for (int i = wave; i < n; i += NC / 64)
    for (int j = lane; j < n; j += 64) {
      double rv = 0.0, xv = 0.0;
      if (j >= i) {
        rv = Sl[i * CB_LD + j];
        xv = ((i >> 4) == (j >> 4)) ? Xd[16 * (j >> 4) * CB_XLD + (j & 15) * CB_XLD + (i & 15)]
                                    : Sl[j * CB_LD + i];
      }
      R[(int64_t)i * ld + j] = rv;
      Ri[(int64_t)i * ld + j] = xv;
    }
  if (threadIdx.x == 0 && J.status != 0) *(int32_t*)J.status = bad_s;
}

}  // namespace

extern "C" int tnx_chol_inv_f64(const tnx_chol_job* jobs, int njob, tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || njob < 0) {
    tnx_set_error("tnx_chol_inv_f64: bad arguments");
    return TNX_EINVAL;
  }
  static std::atomic<uint64_t> lds_set{0};
  if (int rc = tnx_dynamic_lds((const void*)chol_inv_kernel, CHOL_LDS, lds_set)) return rc;
  hipLaunchKernelGGL(chol_inv_kernel, dim3(njob), dim3(NC), CHOL_LDS, (hipStream_t)stream, jobs);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

extern "C" int tnx_qr_f64(const tnx_qr_job* jobs, int njob, tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || njob < 0) {
    tnx_set_error("tnx_qr_f64: bad arguments");
    return TNX_EINVAL;
  }
  static std::atomic<uint64_t> lds_set{0};
  if (int rc = tnx_dynamic_lds((const void*)qr_kernel, sizeof(QrLds), lds_set)) return rc;
  hipLaunchKernelGGL(qr_kernel, dim3(njob), dim3(NQ), sizeof(QrLds), (hipStream_t)stream, jobs);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

extern "C" int tnx_svd_jacobi_f64(const tnx_svd_job* jobs, int njob, int max_sweeps,
                                  tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || njob < 0 || max_sweeps < 1) {
    tnx_set_error("tnx_svd_jacobi_f64: bad arguments");
    return TNX_EINVAL;
  }
  static std::atomic<uint64_t> lds_set{0};
  if (int rc = tnx_dynamic_lds((const void*)svd_kernel, SVD_LDS, lds_set)) return rc;
  hipLaunchKernelGGL(svd_kernel, dim3(njob), dim3(NQ), SVD_LDS, (hipStream_t)stream, jobs, max_sweeps);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}
