// Singular value decomposition of the n x n factor R of an SVD gauge move
// (n <= 1024), by block one-sided Jacobi over many workgroups.
//
// The columns of M = R^T (the rows of R, contiguous in the row-major R) are
// rotated until they are mutually orthogonal: M W = B with W orthogonal, so
// R = W S U^T with S = column norms of B and U = B S^-1.  The outputs avoid
// S^-1: row k of `u` is the k-th left singular vector of R (a column of W)
// and row k of `v` is s_k times the k-th right singular vector (a column of
// B), in descending order of s_k, so R = u^T v exactly.  A gauge move
// A = Q R then keeps A_new = Q u^T (an isometry even when R is rank
// deficient) and hands v to the neighbour.
//
// Columns are grouped into blocks of bw; one launch is one round of the
// round-robin over block pairs, rounds repeat until a sweep rotates nothing.
// A workgroup takes its pair in panels of 16 + 16 columns (all of it for
// bw <= 16): the 32 x 32 Gram matrix of the columns by f64 MFMA, one sweep of
// plane rotations on that matrix (16 disjoint ones at a time, from both
// sides) accumulated into an orthogonal Q, and B and W times Q by MFMA.  The
// columns cross the memory once per round instead of LDS once per rotation,
// and a panel whose Gram matrix needs no rotation is not written.  What ends
// the sweeps is decided on Gram matrices formed anew from B.
// A rotation puts the larger column first, which sorts the columns as they
// converge, and is applied as x - s (y + t x), whose rounding errors are
// those of the small numbers s and t: relative error of the singular values
// 1.5e-15 (n = 128, 200) where c x - s y on the columns had 1.5e-14 to 4e-14.
// ms (MI355X), rotations of columns in LDS -> this: one matrix of order 64 1.8
// -> 0.8, 128 6.6 -> 1.6, 256 21.9 -> 5.0, 1024 195 -> 58; 16 of order 256
// 23.1 -> 5.9, with singular values over 10 decades in rows of any size 75.9
// -> 15.5; values only, 500 of order 128 16.0 -> 8.7.
// Bound: latency.  A round (n = 128 about 21 us; 25 with the rows' angles
// formed anew instead of taken from the lane that has them, and the reads of a
// step behind its angle) is 31 steps of one barrier, each a chain of some 30
// dependent f64 operations for the angle; Gram matrix
// and products are the rest.  Tried and not kept: two sweeps over a Gram
// matrix (fewer rounds, more steps: 128 2.7 ms), two for panels whose column
// norms differ by 1e4 (10 decades 5.4 -> 8.9 ms), angles in f32 (no gain), 256
// lanes for both G and Q (10% slower; faster only for many values-only jobs).
// A column whose norm is at most n eps ||R||_F is numerical zero (rounding
// residue of a rank-deficient R) and takes part in no rotation: rotating
// pairs of such columns never settles, and leaving them alone keeps
// R = u^T v exact and u orthogonal.
//
// A job with u == 0 asks for the singular values only (the entanglement
// spectrum of a bond whose gauge move was a QR): W is neither formed nor
// rotated, and the work area is n^2 + n + 1 doubles (B, column norms, scale).
// R may then be the work area itself (r == work, ld_r == n): forming B is a
// copy onto itself.
#include "tnx_common.h"
#include "jacobi_rot.h"

namespace {

constexpr int NT = 256;
constexpr int SJ_NMAX = 1024;
constexpr int SB = 16;         // columns of a sub-block; a panel is two
constexpr int PW = 2 * SB;
constexpr int GLD = PW + 2;    // LDS row stride of G and Q (with 33 the pairs of a round, u + v
                               // constant, would share a bank)
constexpr int RT = 512;        // lanes of a round's workgroup

// values-only job: no W (see the header)
__device__ __forceinline__ bool values_only(const tnx_svdj_job& J) { return J.u == 0; }
// column norms and the scale ||R||_F^2 follow B (and W, when formed)
__device__ __forceinline__ double* norms_of(const tnx_svdj_job& J) {
  return (double*)J.work + (values_only(J) ? 1 : 2) * (int64_t)J.n * J.n;
}

// pair p of round `round` (< players - 1) of the round-robin, a < b
__device__ __forceinline__ void pair_of(int players, int round, int p, int& a, int& b) {
  const int last = players - 1;
  const int x = round + p, y = round + last - p;
  const int u = p == 0 ? last : (x >= last ? x - last : x);
  const int v = p == 0 ? round : (y >= last ? y - last : y);
  a = min(u, v);
  b = max(u, v);
}

// B (column j = row j of R) and W = I, both column-major n x n in the work area.
__global__ __launch_bounds__(NT) void k_svdj_init(const tnx_svdj_job* __restrict__ jobs) {
  const tnx_svdj_job J = jobs[blockIdx.y];
  const int n = J.n;
  const double* R = (const double*)J.r;
  double* B = (double*)J.work;
  double* W = B + (int64_t)n * n;
  const bool vo = values_only(J);
  for (int j = blockIdx.x; j < n; j += gridDim.x)
    for (int i = threadIdx.x; i < n; i += NT) {
      B[(int64_t)j * n + i] = R[(int64_t)j * J.ld_r + i];
      if (!vo) W[(int64_t)j * n + i] = (i == j) ? 1.0 : 0.0;
    }
}

// ||R||_F^2 of each job into work[2 n^2 + n] (one workgroup per job, a fixed
// summation order, so the zero test below does not depend on the batch); the
// sweeps' flag cleared.
constexpr int NS = 1024;
__global__ __launch_bounds__(NS) void k_svdj_scale(const tnx_svdj_job* __restrict__ jobs,
                                                   int32_t* flag) {
  const tnx_svdj_job J = jobs[blockIdx.x];
  const int64_t nn = (int64_t)J.n * J.n;
  const double TNX_GLOBAL* B = as_global<const double>(J.work);
  double s = 0.0;
#pragma unroll 4
  for (int64_t i = threadIdx.x; i < nn; i += NS) {
    const double b = B[i];
    s += b * b;
  }
  s = tnx_wave_sum(s);
  __shared__ double red[NS / 64];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < NS / 64; ++w) t += red[w];
    norms_of(J)[J.n] = t;
    if (blockIdx.x == 0) *flag = 0;
  }
}

// The flag of a sweep to the host (pinned memory, read after an event), cleared
// for the next one.  (A copy and a clear were two launches of 3.7 us.)
__global__ void k_svdj_publish(int32_t* flag, volatile int32_t* host) {
  if (threadIdx.x == 0) {
    *host = *flag;
    *flag = 0;
  }
}

// Column c (0..31) of a panel: sub-blocks starting at columns ca and cb, cnt
// columns each; -1 past them or past n.
__device__ __forceinline__ int panel_col(int c, int ca, int cb, int cnt, int n) {
  const int l = c & (SB - 1), g = (c < SB ? ca : cb) + l;
  return l < cnt && g < n ? g : -1;
}

// P <- Q^T P for the panel's columns of the column-major n x n matrix P: wave
// `wave` of `waves` takes 32 rows at a time, reads them whole and writes them
// back.
__device__ __forceinline__ void apply_q(double TNX_GLOBAL* P, const double (*Q)[GLD], int n, int ca,
                                        int cb, int cnt, int wave, int waves) {
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
#pragma unroll 1
  for (int r0 = 32 * wave; r0 < n; r0 += 32 * waves) {
    const int row = r0 + 2 * m;
    const bool ok0 = row < n, ok1 = row + 1 < n;
    double b[8][2];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int col = panel_col(4 * s + g, ca, cb, cnt, n);
      const int off = max(col, 0) * n + row;
      b[s][0] = (col >= 0 && ok0) ? P[off] : 0.0;
      b[s][1] = (col >= 0 && ok1) ? P[off + 1] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      tnx_d4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const double qa = Q[4 * s + g][16 * i + m];
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(qa, b[s][0], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(qa, b[s][1], acc[1], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = panel_col(16 * i + g + 4 * r, ca, cb, cnt, n);
        const int off = col * n + row;
        if (col >= 0 && ok0) P[off] = acc[0][r];
        if (col >= 0 && ok1) P[off + 1] = acc[1][r];
      }
      __builtin_amdgcn_sched_barrier(0);   // one half of the columns at a time: registers
    }
  }
}

// One round: block pair p of every job that has that many rounds.  Of the 512
// lanes, the first half owns the 2 x 2 blocks of the Gram matrix, the second
// half those of Q, so that the two updates of a step run side by side.
__global__ __launch_bounds__(RT, 4) void k_svdj_round(const tnx_svdj_job* __restrict__ jobs, int njob,
                                                   int round, int32_t* flag) {
  // the partial Gram matrices of the waves, then G and Q, two copies of each
  // (a step reads one and writes the other)
  __shared__ union {
    double part[RT / 64][3][256];
    struct { double G[2][PW][GLD], Q[2][PW][GLD]; } m;
  } L;
  __shared__ int turned;
  const int ji = tnx_find_owner(jobs, sizeof(tnx_svdj_job), offsetof(tnx_svdj_job, pair_begin),
                                njob, blockIdx.x);
  const tnx_svdj_job J = jobs[ji];
  const int nb = J.nblk, n = J.n, bw = J.bw;
  if (round >= nb - 1) return;  // this job has fewer blocks than the largest one
  int ba, bb;
  pair_of(nb, round, blockIdx.x - J.pair_begin, ba, bb);
  double TNX_GLOBAL* B = as_global<double>(J.work);
  double TNX_GLOBAL* W = B + (int64_t)n * n;
  const bool vo = values_only(J);
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool q_half = wave >= RT / 128;
  const int t = threadIdx.x & (RT / 2 - 1);
  const int pi = t >> 4, qi = t & 15;   // the lane's 2 x 2 block: rotations pi (rows), qi (columns)
  // Gram entries are scaled by a power of two near 1 / ||R||_F^2, so that
  // products of them neither over- nor underflow
  const double fro2 = norms_of(J)[n];
  const double scale = (fro2 > 1e-300 && fro2 < 1.7e308) ? ldexp(1.0, -ilogb(fro2)) : 1.0;
  const double eps = 2.220446049250313e-16 * (double)(n > 8 ? n : 8), eps2 = eps * eps;
  const double zero2 = eps2 * fro2 * scale;  // column norm^2 of numerical zero
  const int cnt = bw < SB ? bw : SB, nsub = bw < SB ? 1 : bw / SB;
  int any = 0;
  // the pair's sub-blocks (one per block for bw <= 16), every two of them
  for (int sr = 0; sr < 2 * nsub - 1; ++sr)
    for (int sp = 0; sp < nsub; ++sp) {
      int sa, sb;
      pair_of(2 * nsub, sr, sp, sa, sb);
      const int ca = (sa < nsub ? ba : bb) * bw + (sa % nsub) * SB;
      const int cb = (sb < nsub ? ba : bb) * bw + (sb % nsub) * SB;
      if (ca >= n) continue;
      if (sr + sp > 0) __syncthreads();   // the last panel is written
      // Gram matrix: blocks (0, 0), (0, 1), (1, 1), each wave every eighth
      // 8 rows; lane group g holds rows 2 g, 2 g + 1 of them
      {
        const int c0 = panel_col(m, ca, cb, cnt, n), c1 = panel_col(16 + m, ca, cb, cnt, n);
        const double TNX_GLOBAL* p0 = B + (int64_t)max(c0, 0) * n;
        const double TNX_GLOBAL* p1 = B + (int64_t)max(c1, 0) * n;
        tnx_d4 g00 = {0, 0, 0, 0}, g01 = {0, 0, 0, 0}, g11 = {0, 0, 0, 0};
#pragma unroll 1
        for (int r0 = 8 * wave; r0 < n; r0 += 8 * (RT / 64)) {
          const int r = r0 + 2 * g;
          double x[2], y[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int rr = min(r + k, n - 1);
            const double xv = p0[rr], yv = p1[rr];
            x[k] = (c0 >= 0 && r + k < n) ? xv : 0.0;
            y[k] = (c1 >= 0 && r + k < n) ? yv : 0.0;
          }
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            g00 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], x[k], g00, 0, 0, 0);
            g01 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], y[k], g01, 0, 0, 0);
            g11 = __builtin_amdgcn_mfma_f64_16x16x4f64(y[k], y[k], g11, 0, 0, 0);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          L.part[wave][0][(g + 4 * r) * 16 + m] = g00[r];
          L.part[wave][1][(g + 4 * r) * 16 + m] = g01[r];
          L.part[wave][2][(g + 4 * r) * 16 + m] = g11[r];
        }
      }
      if (threadIdx.x == 0) turned = 0;
      __syncthreads();
      double v[3];
      if (!q_half) {
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          v[x] = 0.0;
#pragma unroll
          for (int w = 0; w < RT / 64; ++w) v[x] += L.part[w][x][t];
          v[x] *= scale;
        }
      }
      __syncthreads();
      if (!q_half) {
        L.m.G[0][pi][qi] = v[0];
        L.m.G[0][pi][16 + qi] = v[1];
        L.m.G[0][16 + qi][pi] = v[1];
        L.m.G[0][16 + pi][16 + qi] = v[2];
      } else {
        L.m.Q[0][pi][qi] = pi == qi ? 1.0 : 0.0;
        L.m.Q[0][pi][16 + qi] = 0.0;
        L.m.Q[0][16 + pi][qi] = 0.0;
        L.m.Q[0][16 + pi][16 + qi] = pi == qi ? 1.0 : 0.0;
      }
      __syncthreads();
      // a pair that the Gram matrix has to rotate?
      if (!q_half) {
        bool need = false;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int i = pi + 16 * (x >> 1), j = qi + 16 * (x & 1);
          if (i < j) {
            const double a = L.m.G[0][i][i], c = L.m.G[0][j][j], gg = L.m.G[0][i][j];
            need = need || (gg != 0.0 && a > zero2 && c > zero2 && gg * gg > eps2 * (a * c));
          }
        }
        if (need) turned = 1;
      }
      __syncthreads();
      if (turned == 0) continue;
      any = 1;
      // A lane holds elements (r1, r2) x (uq, vq): of G, rows and columns of two
      // rotations, or of Q, rows 2 pi and 2 pi + 1.  The indices of the next
      // step are formed ahead of the barrier, all LDS reads ahead of the angle.
      static_assert(offsetof(decltype(L.m), Q) == sizeof(L.m.G), "Q follows G");
      double* const M = &L.m.G[0][0][0];
      constexpr int COPY = PW * GLD;          // elements of one copy of G or Q
      const int half = q_half ? 2 * COPY : 0;
      int uq, vq, r1 = 2 * pi, r2 = 2 * pi + 1;
      pair_of(PW, 0, qi, uq, vq);
      if (!q_half) pair_of(PW, 0, pi, r1, r2);
#pragma unroll 1
      for (int ir = 0; ir < PW - 1; ++ir) {
        const double* G = M + (ir & 1) * COPY;
        const double* S = G + half;
        double* D = M + ((ir & 1) ^ 1) * COPY + half;
        const int ru = (int)__umul24(uq, GLD), rv = (int)__umul24(vq, GLD);
        const int o1 = (int)__umul24(r1, GLD), o2 = (int)__umul24(r2, GLD);
        const double a = G[ru + uq], c = G[rv + vq], gg = G[ru + vq];
        double x11 = S[o1 + uq], x12 = S[o1 + vq], x21 = S[o2 + uq], x22 = S[o2 + vq];
        const bool live = a > zero2 && c > zero2;   // no zero column (the padding among them)
        // (entries of a live pair are above 1e-45: the squares stay in range)
        const JacobiRot rq = jacobi_rot<false>(a, c, gg, live && gg * gg > eps2 * (a * c), live);
        jacobi_apply(rq, x11, x12);
        jacobi_apply(rq, x21, x22);
        if (!q_half) {
          // the rows' rotation: the one lane pi has for its column
          JacobiRot rp;
          rp.s = __shfl(rq.s, pi, 64);
          rp.tau = __shfl(rq.tau, pi, 64);
          rp.swap = (__ballot(rq.swap) >> pi) & 1;
          jacobi_apply(rp, x11, x21);
          jacobi_apply(rp, x12, x22);
        }
        D[o1 + uq] = x11;
        D[o1 + vq] = x12;
        D[o2 + uq] = x21;
        D[o2 + vq] = x22;
        pair_of(PW, ir + 1, qi, uq, vq);
        if (!q_half) pair_of(PW, ir + 1, pi, r1, r2);
        __syncthreads();
      }
      const double (*Q)[GLD] = L.m.Q[(PW - 1) & 1];
      const bool w_half = q_half && !vo;
      const int waves = vo ? RT / 64 : RT / 128;
      apply_q(w_half ? W : B, Q, n, ca, cb, cnt, w_half ? wave - RT / 128 : wave, waves);
    }
  if (any && threadIdx.x == 0) atomicOr(flag, 1);
}

// su[j] = ||B_j|| (one wavefront per column)
__global__ __launch_bounds__(NT) void k_svdj_norms(const tnx_svdj_job* __restrict__ jobs) {
  const tnx_svdj_job J = jobs[blockIdx.y];
  const int n = J.n;
  const int j = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  if (j >= n) return;
  const double* B = (const double*)J.work;
  double* su = norms_of(J);
  double s = 0.0;
  for (int i = threadIdx.x & 63; i < n; i += 64) {
    const double b = B[(int64_t)j * n + i];
    s += b * b;
  }
  s = tnx_wave_sum(s);
  if ((threadIdx.x & 63) == 0) su[j] = sqrt(s);
}

// Rank of column j in descending order (ties by index); row rank of u and v
// gets column j of W and of B, s[rank] = su[j].
__global__ __launch_bounds__(NT) void k_svdj_sort(const tnx_svdj_job* __restrict__ jobs) {
  const tnx_svdj_job J = jobs[blockIdx.y];
  const int n = J.n, j = blockIdx.x;
  if (j >= n) return;
  const double* B = (const double*)J.work;
  const double* W = B + (int64_t)n * n;
  const double* su = norms_of(J);
  const double sj = su[j];
  int cnt = 0;
  for (int q = threadIdx.x; q < n; q += NT) {
    const double sq = su[q];
    cnt += (sq > sj || (sq == sj && q < j)) ? 1 : 0;
  }
  __shared__ int red[NT / 64];
  for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = cnt;
  __syncthreads();
  const int rank = red[0] + red[1] + red[2] + red[3];
  if (!values_only(J)) {
    double* u = (double*)J.u;
    double* v = (double*)J.v;
    for (int i = threadIdx.x; i < n; i += NT) {
      u[(int64_t)rank * n + i] = W[(int64_t)j * n + i];
      v[(int64_t)rank * n + i] = B[(int64_t)j * n + i];
    }
  }
  if (threadIdx.x == 0) ((double*)J.s)[rank] = sj;
}

thread_local int32_t* g_flag_pin = nullptr;   // two slots: sweeps alternate

}  // namespace

extern "C" int tnx_svd_block_jacobi(const tnx_svdj_job* jobs, int njob, int npairs, int max_nblk,
                                    int max_n, int32_t* flag, int max_sweeps,
                                    tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || flag == nullptr || njob < 0 || npairs <= 0 || max_nblk < 2 ||
      max_n <= 0 || max_n > SJ_NMAX || max_sweeps < 1) {
    tnx_set_error("tnx_svd_block_jacobi: bad arguments (njob=%d npairs=%d nblk=%d n=%d)", njob,
                  npairs, max_nblk, max_n);
    return TNX_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  if (g_flag_pin == nullptr)
    TNX_CHECK_HIP(hipHostMalloc((void**)&g_flag_pin, 64, hipHostMallocDefault));
  hipLaunchKernelGGL(k_svdj_init, dim3(max_n < 1024 ? max_n : 1024, njob), dim3(NT), 0, s, jobs);
  hipLaunchKernelGGL(k_svdj_scale, dim3(njob), dim3(NS), 0, s, jobs, flag);
  TNX_CHECK_LAUNCH();
  // The flag of a sweep is read while the next one runs: a sweep after the
  // last is a Gram matrix per panel and nothing else (n = 128: 30 us for one
  // job), less than the stop after every sweep that it saves.
  hipEvent_t ev[2];
  TNX_CHECK_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
  if (hipEventCreateWithFlags(&ev[1], hipEventDisableTiming) != hipSuccess) {
    (void)hipEventDestroy(ev[0]);
    tnx_set_error("tnx_svd_block_jacobi: no event");
    return TNX_EHIP;
  }
  bool converged = false;
  int recorded = 0;   // sweeps with a recorded event
  hipError_t err = hipSuccess;
  for (int sweep = 0; sweep < max_sweeps && !converged && err == hipSuccess; ++sweep) {
    for (int r = 0; r < max_nblk - 1; ++r)
      hipLaunchKernelGGL(k_svdj_round, dim3(npairs), dim3(RT), 0, s, jobs, njob, r, flag);
    hipLaunchKernelGGL(k_svdj_publish, dim3(1), dim3(64), 0, s, flag,
                       (volatile int32_t*)g_flag_pin + (sweep & 1));
    err = hipGetLastError();
    if (err == hipSuccess) err = hipEventRecord(ev[sweep & 1], s);
    if (err == hipSuccess) ++recorded;
    // the previous sweep's flag, or after the last allowed sweep its own too
    for (int k = sweep > 0 ? sweep - 1 : 0; err == hipSuccess && !converged && k <= sweep; ++k) {
      if (k == sweep && sweep + 1 < max_sweeps) break;
      err = hipEventSynchronize(ev[k & 1]);
      converged = err == hipSuccess && ((volatile int32_t*)g_flag_pin)[k & 1] == 0;
    }
  }
  if (err == hipSuccess) {
    hipLaunchKernelGGL(k_svdj_norms, dim3((max_n + 3) / 4, njob), dim3(NT), 0, s, jobs);
    hipLaunchKernelGGL(k_svdj_sort, dim3(max_n, njob), dim3(NT), 0, s, jobs);
    err = hipGetLastError();
  }
  // The sweep queued past the last one publishes too: its write must be over
  // before this thread's next call, which may be on another stream, reads the
  // slots (the wait is for that sweep; norms and order run meanwhile).
  const hipError_t last =
      err == hipSuccess ? hipEventSynchronize(ev[(recorded - 1) & 1]) : hipStreamSynchronize(s);
  if (err == hipSuccess) err = last;
  (void)hipEventDestroy(ev[0]);
  (void)hipEventDestroy(ev[1]);
  if (err != hipSuccess) {
    tnx_set_error("tnx_svd_block_jacobi: %s", hipGetErrorString(err));
    return TNX_EHIP;
  }
  return converged ? TNX_OK : TNX_ENOCONV;
}
