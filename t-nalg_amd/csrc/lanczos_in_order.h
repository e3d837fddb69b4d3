// The passes of a Lanczos call whose plan asks for sums in a fixed order
// (TNX_GEMM_IN_ORDER in its mode), part of lanczos.hip.
//
// The infinite-size driver cuts its centre between Schmidt values that can be
// equal to rounding (with symmetric environments and an odd bond dimension they
// always are), so which combination of a degenerate pair is kept, and with it
// every later number of the run, hangs on the last bit of each product, sum and
// eigenvector before it.  What such a run returns is therefore defined by the
// arithmetic, and this file is that definition: 256 lanes a chunk of 1024, a
// butterfly per sum, the tridiagonal problem by Sturm counts with divisions and
// inverse iteration, the restart by QR steps on the tridiagonal matrix.  Nothing
// in it may be regrouped, and a sum of products says which of them are fused (the
// compiler's own choice is another one in another loop).  k_irl_apply and k_final,
// which add the rows in order, serve both.  The passes of lanczos.hip give the same results to
// rounding, faster: us for the three passes of a step of a 64 x 64 problem (4
// chunks, mean over the cycles of 20, MI355X) 35 here (24 of them the tridiagonal
// problem), 18 there; a restart 162 and 15.
#pragma once

constexpr int IT = 256;           // lanes
constexpr int IE = CHUNK / IT;    // elements of a lane: i0 + t + IT q
constexpr int IW = IT / 64;

__device__ __forceinline__ int io_elem(const ChunkInfo& ci, int q) {
  return min(ci.i0 + q * IT + (int)threadIdx.x, ci.i1 - 1);
}
__device__ __forceinline__ bool io_inside(const ChunkInfo& ci, int q) {
  return ci.i0 + q * IT + (int)threadIdx.x < ci.i1;
}
__device__ __forceinline__ double io_total(const double (*red)[NCV_MAX + 1], int k) {
  return (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
}

// reduce_partials by 256 lanes and a butterfly per sum
__device__ __forceinline__ void io_reduce(const double* part, int nchunks, int chunk_begin, int nch,
                                          int nk, int npad, double* dst) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double TNX_GLOBAL* p = as_global<const double>((uint64_t)part) + chunk_begin;
  for (int k0 = wave; k0 < npad; k0 += 4 * IW) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = lane; c < nch; c += 64) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * IW;
        if (k < nk) s[u] += p[(int64_t)k * nchunks + c];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double v = tnx_wave_sum(s[u]);
      if (lane == 0 && k0 + u * IW < npad) dst[k0 + u * IW] = v;
    }
  }
}

__global__ __launch_bounds__(IT) void io_init_norm(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                   void* state, int nchunks) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  const double TNX_GLOBAL* v = as_global<const double>(S[ci.s].init);
  double acc = 0.0;
  for (int i = ci.i0 + threadIdx.x; i < ci.i1; i += IT) acc = fma(v[i], v[i], acc);
  __shared__ double red[IW][NCV_MAX + 1];
  acc = tnx_wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][0] = acc;
  __syncthreads();
  if (threadIdx.x == 0) L.partA[blockIdx.x] = io_total(red, 0);
}

// k_init_scale
__global__ __launch_bounds__(IT) void io_init_scale(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                    void* state, int nchunks, int x_dtype) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  const tnx_lanczos_solve D = S[ci.s];
  __shared__ double tot;
  io_reduce(L.partA, nchunks, D.chunk_begin, ci.nch, 1, 1, &tot);
  __syncthreads();
  const double sc = tot > 0.0 ? 1.0 / sqrt(tot) : -1.0;
  if (ci.c == 0 && threadIdx.x == 0) {   // the rest of the state is zero
    L.st[ci.s].scale = sc;
    L.st[ci.s].y[0] = 1.0;
    L.act[ci.s] = 1;
  }
  const double TNX_GLOBAL* v = as_global<const double>(D.init);
  const double flat = 1.0 / sqrt((double)D.n);
  const int xd = dtype_of(x_dtype, D.x_dtype);
  for (int i = ci.i0 + threadIdx.x; i < ci.i1; i += IT) {
    double val = sc > 0.0 ? v[i] * sc : flat;
    if (D.v_dtype == TNX_F32) {
      const float vv = (float)val;
      as_global<float>(D.V)[i] = vv;
      val = (double)vv;
    } else {
      as_global<double>(D.V)[i] = val;
    }
    tnx_store((void*)D.x, xd, i, val);
  }
}

// This chunk's elements of the rows min(u, j), u < LV
template <typename VT, int LV>
__device__ __forceinline__ void io_rows(const VT TNX_GLOBAL* V, int ldv, int j, const ChunkInfo& ci,
                                        VT (&v)[LV][IE]) {
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const VT TNX_GLOBAL* row = V + (int64_t)min(u, j) * ldv;
#pragma unroll
    for (int q = 0; q < IE; ++q) v[u][q] = row[io_elem(ci, q)];
  }
}
// Their dots with x (zero past the chunk's end), wave sums into red[wave]
template <typename VT, int LV>
__device__ __forceinline__ void io_dots(const VT (&v)[LV][IE], const double (&x)[IE],
                                        double (*red)[NCV_MAX + 1]) {
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < IE; ++q) s = fma((double)v[u][q], x[q], s);
    s = tnx_wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][u] = s;
  }
}
__device__ __forceinline__ void io_load_w(const tnx_lanczos_solve& D, int wd, const ChunkInfo& ci,
                                          double (&w)[IE]) {
#pragma unroll
  for (int q = 0; q < IE; ++q) {
    w[q] = tnx_load((const void*)D.w, wd, io_elem(ci, q));
    if (!io_inside(ci, q)) w[q] = 0.0;
  }
}

template <typename VT, int LV>
__device__ __forceinline__ void io_dots_body(const tnx_lanczos_solve& D, const LzLayout& L,
                                             const ChunkInfo& ci, int nchunks, int j, int wd) {
  __shared__ double red[IW][NCV_MAX + 1];
  VT v[LV][IE];
  io_rows(as_global<const VT>(D.V), D.ldv, j, ci, v);
  double w[IE];
  io_load_w(D, wd, ci, w);
  io_dots(v, w, red);
  __syncthreads();
  if ((int)threadIdx.x <= j)
    L.partA[(int64_t)threadIdx.x * nchunks + blockIdx.x] = io_total(red, threadIdx.x);
}

// k_dots
template <int LV>
__global__ __launch_bounds__(IT) void io_pass1(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                               void* state, int nchunks, int j, int w_dtype,
                                               unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  if (L.act[ci.s] == 0) return;
  const tnx_lanczos_solve D = S[ci.s];
  const int wd = dtype_of(w_dtype, D.w_dtype);
  if (D.v_dtype == TNX_F32) io_dots_body<float, LV>(D, L, ci, nchunks, j, wd);
  else io_dots_body<double, LV>(D, L, ci, nchunks, j, wd);
  tnx_stamp_end(ts);
}

template <typename VT, int LV>
__device__ __forceinline__ void io_update_body(const tnx_lanczos_solve& D, const LzLayout& L,
                                               const ChunkInfo& ci, int nchunks, int j, int wd) {
  __shared__ double red[IW][NCV_MAX + 1];
  __shared__ double h[NCV_MAX + 1];
  VT v[LV][IE];
  io_rows(as_global<const VT>(D.V), D.ldv, j, ci, v);
  double r[IE];
  io_load_w(D, wd, ci, r);
  io_reduce(L.partA, nchunks, D.chunk_begin, ci.nch, j + 1, LV, h);   // zero from j + 1 on
  __syncthreads();
  if (ci.c == 0 && (int)threadIdx.x <= j) L.st[ci.s].h1[threadIdx.x] = h[threadIdx.x];
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double hu = h[u];
#pragma unroll
    for (int q = 0; q < IE; ++q) r[q] = fma(-hu, (double)v[u][q], r[q]);
  }
  VT TNX_GLOBAL* Vn = as_global<VT>(D.V) + (int64_t)(j + 1) * D.ldv;
#pragma unroll
  for (int q = 0; q < IE; ++q) {
    if (io_inside(ci, q)) Vn[io_elem(ci, q)] = (VT)r[q];
    else r[q] = 0.0;
  }
  io_dots(v, r, red);
  static_assert(IE == 4, "the order of a lane's squares");
  double nn = fma(r[3], r[3], fma(r[2], r[2], fma(r[0], r[0], r[1] * r[1])));
  nn = tnx_wave_sum(nn);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][j + 1] = nn;
  __syncthreads();
  if ((int)threadIdx.x <= j + 1)
    L.partB[(int64_t)threadIdx.x * nchunks + blockIdx.x] = io_total(red, threadIdx.x);
}

// k_update_dots
template <int LV>
__global__ __launch_bounds__(IT) void io_pass2(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                               void* state, int nchunks, int j, int w_dtype,
                                               unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  if (L.act[ci.s] == 0) return;
  const tnx_lanczos_solve D = S[ci.s];
  const int wd = dtype_of(w_dtype, D.w_dtype);
  if (D.v_dtype == TNX_F32) io_update_body<float, LV>(D, L, ci, nchunks, j, wd);
  else io_update_body<double, LV>(D, L, ci, nchunks, j, wd);
  tnx_stamp_end(ts);
}

// Number of eigenvalues of the symmetric tridiagonal (a, b) below x.
__device__ inline int sturm_count(const double* a, const double* b, int k, double x) {
  const double tiny = 1e-300;
  int cnt = 0;
  double q = a[0] - x;
  if (q < 0) cnt++;
  for (int i = 1; i < k; ++i) {
    if (fabs(q) < tiny) q = -tiny;
    q = (a[i] - x) - b[i - 1] * b[i - 1] / q;
    if (q < 0) cnt++;
  }
  return cnt;
}

// Lowest eigenpair of the k x k tridiagonal (a, b) in LDS, all IT lanes of the
// block; thread 0 writes y[0..k) and *theta.  work: LDS scratch of 5 * NCV_MAX
// doubles for the inverse iteration.  The bracket shrinks 257-fold per round:
// lane t evaluates the Sturm count at the (t + 1)-th of 256 interior points and
// the first point with a count >= 1 bounds the lowest eigenvalue.
__device__ void io_tridiag(const double* a, const double* b, int k, double* y, double* theta,
                           double* work) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (k == 1) {
    if (threadIdx.x == 0) {
      y[0] = 1.0;
      *theta = a[0];
    }
    return;
  }
  __shared__ unsigned long long masks[IW];
  double lo = a[0], hi = a[0];
  for (int i = 0; i < k; ++i) {
    const double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < k - 1 ? fabs(b[i]) : 0.0);
    lo = fmin(lo, a[i] - r);
    hi = fmax(hi, a[i] + r);
  }
  const double span = fmax(hi - lo, 1e-300);
  lo -= 1e-12 * span;
  hi += 1e-12 * span;
  constexpr double NSUB = IT + 1;
  for (int round = 0; round < 16; ++round) {
    const double w = hi - lo;  // identical in every lane
    if (w <= 4.0 * 2.220446049250313e-16 * fmax(fabs(lo), fabs(hi)) + 1e-300) break;
    const double x = lo + w * (double)(threadIdx.x + 1) / NSUB;
    const int cnt = sturm_count(a, b, k, x);
    const unsigned long long m = __ballot(cnt >= 1);
    if (lane == 0) masks[wave] = m;
    __syncthreads();
    int f = -1;
    for (int q = 0; q < IW; ++q)
      if (masks[q] != 0ull) {
        f = q * 64 + __ffsll((long long)masks[q]) - 1;
        break;
      }
    __syncthreads();  // masks are rewritten next round
    if (f < 0) {
      lo = lo + w * (double)IT / NSUB;
    } else {
      const double xf = lo + w * (double)(f + 1) / NSUB;
      const double xp = lo + w * (double)f / NSUB;
      hi = xf;
      lo = xp;
    }
  }
  if (threadIdx.x != 0) return;
  const double th = 0.5 * (lo + hi);
  *theta = th;
  // inverse iteration with partial pivoting on (T - th I)
  double* z = work;
  double* rhs = work + NCV_MAX;
  double* u0 = work + 2 * NCV_MAX;
  double* u1 = work + 3 * NCV_MAX;
  double* u2 = work + 4 * NCV_MAX;
  const double tiny = 2.220446049250313e-16 * span;
  for (int i = 0; i < k; ++i) z[i] = 1.0 / sqrt((double)k);
  for (int it = 0; it < 2; ++it) {
    for (int i = 0; i < k; ++i) rhs[i] = z[i];
    // current pivot-row candidate (cols i, i+1, i+2)
    double p0 = a[0] - th, p1 = b[0], p2 = 0.0, pr = rhs[0];
    for (int i = 0; i < k - 1; ++i) {
      const double n0 = b[i], n1 = a[i + 1] - th, n2 = (i + 1 < k - 1) ? b[i + 1] : 0.0;
      const double nr = rhs[i + 1];
      if (fabs(p0) >= fabs(n0)) {
        if (fabs(p0) < tiny) p0 = (p0 < 0 ? -tiny : tiny);
        const double f = n0 / p0;
        u0[i] = p0; u1[i] = p1; u2[i] = p2; rhs[i] = pr;
        p0 = fma(-f, p1, n1); p1 = fma(-f, p2, n2); p2 = 0.0; pr = fma(-f, pr, nr);
      } else {
        const double f = p0 / n0;
        u0[i] = n0; u1[i] = n1; u2[i] = n2; rhs[i] = nr;
        const double q0 = fma(-f, n1, p1), q1 = fma(-f, n2, p2);
        p0 = q0; p1 = q1; p2 = 0.0; pr = fma(-f, nr, pr);
      }
    }
    if (fabs(p0) < tiny) p0 = (p0 < 0 ? -tiny : tiny);
    u0[k - 1] = p0; u1[k - 1] = 0.0; u2[k - 1] = 0.0; rhs[k - 1] = pr;
    for (int i = k - 1; i >= 0; --i) {
      double s = rhs[i];
      if (i + 1 < k) s = fma(-u1[i], z[i + 1], s);
      if (i + 2 < k) s = fma(-u2[i], z[i + 2], s);
      z[i] = s / u0[i];
    }
    double nrm = 0.0;
    for (int i = 0; i < k; ++i) nrm = fma(z[i], z[i], nrm);
    nrm = 1.0 / sqrt(nrm);
    for (int i = 0; i < k; ++i) z[i] *= nrm;
  }
  for (int i = 0; i < k; ++i) y[i] = z[i];
}

template <typename VT>
__device__ __forceinline__ void io_normalize_body(const tnx_lanczos_solve& D, const ChunkInfo& ci,
                                                  int j, int xd, const double* h, double beta,
                                                  bool skip) {
  const VT TNX_GLOBAL* V = as_global<const VT>(D.V);
  VT TNX_GLOBAL* Vn = as_global<VT>(D.V) + (int64_t)(j + 1) * D.ldv;
  const double inv = 1.0 / beta;
  double r[IE];
#pragma unroll
  for (int q = 0; q < IE; ++q) r[q] = (double)Vn[io_elem(ci, q)];
  if (!skip)
    for (int k = 0; k <= j; ++k) {
      const double hk = h[k];
#pragma unroll
      for (int q = 0; q < IE; ++q)
        r[q] = fma(-hk, (double)V[(int64_t)k * D.ldv + io_elem(ci, q)], r[q]);
    }
#pragma unroll
  for (int q = 0; q < IE; ++q)
    if (io_inside(ci, q)) {
      const VT v = (VT)(r[q] * inv);
      Vn[io_elem(ci, q)] = v;
      tnx_store((void*)D.x, xd, io_elem(ci, q), (double)v);
    }
}

// k_update_norm (the same blocks and decisions)
__global__ __launch_bounds__(IT) void io_pass3(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                               void* state, int nchunks, int j, int x_dtype,
                                               int min_iters, int32_t* nact_host,
                                               unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  const bool solver = (int)blockIdx.x < nsolve;
  ChunkInfo ci;
  int s = (int)blockIdx.x;
  if (!solver) {
    ci = chunk_of(S, nsolve, (int)blockIdx.x - nsolve);
    s = ci.s;
  }
  if (!solve_active(L.act, s)) {
    if (solver) publish_nact(L, nsolve, false, nact_host);
    return;
  }
  const tnx_lanczos_solve D = S[s];
  __shared__ double h[NCV_MAX + 1];
  __shared__ double beta_s;
  __shared__ int skip_s;
  io_reduce(L.partB, nchunks, D.chunk_begin, (D.n + CHUNK - 1) / CHUNK, j + 2, j + 2, h);
  __syncthreads();
  if (threadIdx.x == 0) {
    double hh = 0.0;
    for (int k = 0; k <= j; ++k) hh = fma(h[k], h[k], hh);
    const double bb = fmax(h[j + 1] - hh, 0.0);
    beta_s = sqrt(bb);
    const double sk = D.v_dtype == TNX_F32 ? LZ_REORTH_SKIP_F32 : LZ_REORTH_SKIP;
    skip_s = hh <= sk * sk * bb;
  }
  __syncthreads();
  const double beta = beta_s;
  if (!solver) {
    const int xd = dtype_of(x_dtype, D.x_dtype);
    if (D.v_dtype == TNX_F32) io_normalize_body<float>(D, ci, j, xd, h, beta, skip_s != 0);
    else io_normalize_body<double>(D, ci, j, xd, h, beta, skip_s != 0);
    tnx_stamp_end(ts);
    return;
  }
  LzState& st = L.st[s];
  __shared__ double a_s[NCV_MAX], b_s[NCV_MAX], y_s[NCV_MAX], th_s;
  __shared__ double work[5 * NCV_MAX];
  for (int k = threadIdx.x; k < j; k += IT) {
    a_s[k] = st.alpha[k];
    b_s[k] = st.beta[k];
  }
  for (int k = threadIdx.x; k <= j; k += IT) st.h2[k] = h[k];
  if (threadIdx.x == 0) {
    const double alpha = st.h1[j] + h[j];
    st.alpha[j] = alpha;
    st.beta[j] = beta;
    st.iters += 1;
    a_s[j] = alpha;
    b_s[j] = beta;
  }
  __syncthreads();
  io_tridiag(a_s, b_s, j + 1, y_s, &th_s, work);
  __syncthreads();
  for (int k = threadIdx.x; k <= j; k += IT) st.y[k] = y_s[k];
  bool conv = false;
  if (threadIdx.x == 0) {
    const double th = th_s;
    const double res = fabs(beta * y_s[j]);
    st.theta = th;
    st.resid = res;
    st.jlast = j;
    const double thr = fmax(D.tol_scale * fabs(1.0 - D.tau * th), D.floor_rel * fabs(th));
    double anorm = 0.0;
    for (int k = 0; k <= j; ++k) anorm = fmax(anorm, fabs(a_s[k]) + (k > 0 ? fabs(b_s[k - 1]) : 0.0));
    const bool breakdown = beta <= 1e-14 * fmax(anorm, 1e-300);
    const bool full = (j + 1 >= D.n);
    conv = full || breakdown || ((j + 1 >= min_iters) && res <= thr);
    if (conv) {
      st.converged = 1;
      __hip_atomic_store(L.act + s, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  publish_nact(L, nsolve, conv, nact_host);
  tnx_stamp_end(ts);
}

// Sturm count (eigenvalues below x) of the m x m tridiagonal held in
// registers: a[i] diagonal, e[i] = b[i]^2 the squared coupling of i, i+1.
__device__ __forceinline__ int sturm_count_reg(const double (&a)[NCV_MAX],
                                               const double (&e)[NCV_MAX], int m, double x) {
  const double tiny = 1e-300;
  int cnt = 0;
  double q = 1.0;
#pragma unroll
  for (int i = 0; i < NCV_MAX; ++i) {
    if (i < m) {
      q = (i == 0) ? (a[0] - x) : (a[i] - x) - e[i - 1] / q;
      if (q < 0) cnt++;
      if (fabs(q) < tiny) q = -tiny;
    }
  }
  return cnt;
}

// k_irl_solve by the QR steps alone: lane i bisects the Sturm count for
// eigenvalue k + i, lane 0 applies the shifts, lane r accumulates row r of Q.
__global__ __launch_bounds__(IT) void io_irl_solve(const tnx_lanczos_solve* __restrict__ S,
                                                   int nsolve, void* state, int nchunks, int m,
                                                   int k) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  const int s = blockIdx.x;
  if (!solve_active(L.act, s)) return;
  LzState& st = L.st[s];
  __shared__ double a_l[NCV_MAX], b_l[NCV_MAX], sh[NCV_MAX];
  __shared__ double rc[NCV_MAX][NCV_MAX], rs[NCV_MAX][NCV_MAX];
  __shared__ int nrot[NCV_MAX];
  __shared__ double qmk, rho_s, bhat_s;
  __shared__ double ak[LZ_KEEP], bk[LZ_KEEP];
  const int t = threadIdx.x;
  if (t < m) {
    a_l[t] = st.alpha[t];
    b_l[t] = st.beta[t];   // b[m-1]: coefficient of V[m]
  }
  __syncthreads();
  const int np = m - k;
  if (t < np) {
    double a[NCV_MAX], e[NCV_MAX];
    double lo = a_l[0], hi = a_l[0];
#pragma unroll
    for (int i = 0; i < NCV_MAX; ++i) {
      a[i] = (i < m) ? a_l[i] : 0.0;
      const double bi = (i < m - 1) ? b_l[i] : 0.0;
      e[i] = bi * bi;
      if (i < m) {
        const double r = fabs(bi) + (i > 0 ? fabs(b_l[i - 1]) : 0.0);
        lo = fmin(lo, a[i] - r);
        hi = fmax(hi, a[i] + r);
      }
    }
    const int idx = k + t;
    for (int it = 0; it < 64; ++it) {
      if (hi - lo <= 1e-13 * fmax(fabs(lo), fabs(hi)) + 1e-300) break;
      const double mid = 0.5 * (lo + hi);
      if (sturm_count_reg(a, e, m, mid) >= idx + 1) hi = mid;
      else lo = mid;
    }
    sh[t] = 0.5 * (lo + hi);
  }
  __syncthreads();
  if (t == 0) {
    double a[NCV_MAX], b[NCV_MAX];
#pragma unroll
    for (int i = 0; i < NCV_MAX; ++i) {
      a[i] = (i < m) ? a_l[i] : 0.0;
      b[i] = (i < m - 1) ? b_l[i] : 0.0;
    }
    for (int p = 0; p < np; ++p) {
      int iend = m - 1;   // chase rows/cols 0..iend
#pragma unroll
      for (int u = NCV_MAX - 2; u >= 0; --u)
        if (u < m - 1 && fabs(b[u]) <= 2.220446049250313e-16 * (fabs(a[u]) + fabs(a[u + 1])))
          iend = u;   // the first negligible coupling from the top
#pragma unroll
      for (int u = 0; u < NCV_MAX - 1; ++u)
        if (u == iend) b[u] = 0.0;
      nrot[p] = iend;
      double x = a[0] - sh[p], z = b[0], bulge = 0.0;
#pragma unroll
      for (int u = 0; u < NCV_MAX - 1; ++u) {
        if (u < iend) {
          double c = 1.0, sn = 0.0;
          if (z != 0.0) {
            const double ri = rsqrt(fma(z, z, x * x));
            c = x * ri;
            sn = z * ri;
          }
          rc[p][u] = c;
          rs[p][u] = sn;
          if (u > 0) b[u - 1] = fma(sn, bulge, c * b[u - 1]);
          const double au = a[u], au1 = a[u + 1], bu = b[u];
          const double cc = c * c, ss = sn * sn, off = 2.0 * c * sn * bu;
          a[u] = fma(ss, au1, fma(cc, au, off));
          a[u + 1] = fma(cc, au1, fma(ss, au, -off));
          b[u] = fma(c * sn, au1 - au, fma(c, c, -ss) * bu);
          if (u + 1 < iend) {
            bulge = sn * b[u + 1];
            b[u + 1] = c * b[u + 1];
            x = b[u];
            z = bulge;
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < LZ_KEEP; ++i) {
      ak[i] = a[i];
      bk[i] = b[i];
    }
  }
  __syncthreads();
  double q[NCV_MAX];   // row t of Q (static indices: kept in registers)
#pragma unroll
  for (int c = 0; c < NCV_MAX; ++c) q[c] = (c == t) ? 1.0 : 0.0;
  if (t < m) {
    for (int p = 0; p < np; ++p) {
      const int n = nrot[p];
#pragma unroll
      for (int u = 0; u < NCV_MAX - 1; ++u) {
        if (u < n) {
          const double c = rc[p][u], sn = rs[p][u];
          const double q0 = q[u], q1 = q[u + 1];
          q[u] = fma(c, q0, sn * q1);
          q[u + 1] = fma(c, q1, -(sn * q0));
        }
      }
    }
    if (t == m - 1) {
#pragma unroll
      for (int c = 0; c < NCV_MAX; ++c)
        if (c == k - 1) qmk = q[c];
    }
  }
  __syncthreads();
  if (t == 0) {
    const double bhat = bk[k - 1];
    const double sigma = st.beta[m - 1] * qmk;
    const double rho = hypot(bhat, sigma);
    bhat_s = bhat;
    rho_s = rho;
    double anorm = 0.0;
    for (int u = 0; u < m; ++u) anorm = fmax(anorm, fabs(a_l[u]) + fabs(b_l[u]));
    for (int u = 0; u < k; ++u) st.alpha[u] = ak[u];
    for (int u = 0; u + 1 < k; ++u) st.beta[u] = bk[u];
    st.beta[k - 1] = rho;
    st.restarts += 1;
    for (int u = 0; u <= k; ++u) st.C[m][u] = 0.0;
    if (rho > 0.0) st.C[m][k] = sigma / rho;
    if (!(rho > 1e-14 * fmax(anorm, 1e-300))) {
      // invariant subspace: the current Ritz pair is exact
      st.converged = 1;
      __hip_atomic_store(L.act + s, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      atomicSub(L.nact, 1);
    }
  }
  __syncthreads();
  if (t < m) {
    const double f = rho_s > 0.0 ? bhat_s / rho_s : 0.0;
#pragma unroll
    for (int c = 0; c < NCV_MAX; ++c) {
      if (c < k) st.C[t][c] = q[c];
      else if (c == k) st.C[t][c] = f * q[c];
    }
  }
}
