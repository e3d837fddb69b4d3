// Batched Lanczos eigensolver for the lowest eigenpair of every solve's
// effective Hamiltonian (the local problem of one-site DMRG).
//
// All solves of a batch advance in lockstep over Krylov index j; a solve
// that has converged is masked out (its active flag is 0) so the matvec and
// the kernels below skip it.  Vectors are cut into 1024-element chunks, one
// workgroup per chunk.  A per-solve reduction never synchronises blocks
// inside a kernel: each kernel leaves one partial sum per chunk, and every
// block of the next kernel on the stream (ordered after it) sums the
// partials of its own solve in the same fixed order.  A Lanczos step is
//   matvec (3 launches) + dots + update/dots/norm
//   + update/normalise (plus one block per solve: tridiagonal solve,
//     convergence).
// All reductions are f64 (two-pass classical Gram-Schmidt against the full
// basis); the basis is stored in f64, or in f32 for a solve whose matvec
// runs in f32 or bf16 (v_dtype: the basis passes then move half the bytes).
// The matvec may run in f32 or bf16.
// The (j+1)x(j+1) tridiagonal eigenproblem is solved on the device by one
// wavefront: multisection with secant steps, then a twisted factorisation.
// (A call whose plan asks for sums in a fixed order takes the passes of
// lanczos_in_order.h.)
// A solve that has not converged after ncv steps is restarted implicitly
// (Sorensen's implicitly restarted Lanczos with exact shifts, as ARPACK's
// dsaupd does for eigsh): the ncv - k largest Ritz values are applied as
// shifts to the tridiagonal matrix, which compresses the factorisation to
// k = min(LZ_KEEP, ncv - 1) vectors spanning the k lowest Ritz vectors; the next cycle continues the Lanczos recurrence from step k.
#include <mutex>

#include "tnx_common.h"

namespace {

constexpr int NCV_MAX = 32;
constexpr int CHUNK = 1024;
constexpr int NP = 512;           // lanes of the kernels over a chunk
constexpr int EPT = CHUNK / NP;   // elements of a lane
constexpr int NW = NP / 64;
constexpr int NT = 256;           // lanes of the restart's solve
constexpr int LZ_KEEP = 4;   // vectors kept by an implicit restart (at most)
constexpr double LZ_REORTH_SKIP = 1e-12;   // second projection left out below this (relative)
constexpr double LZ_REORTH_SKIP_F32 = 1e-6;  // the same for an f32 basis (its rounding level)

struct LzState {
  double alpha[NCV_MAX];
  double beta[NCV_MAX];
  double h1[NCV_MAX + 1];
  double h2[NCV_MAX + 1];
  double y[NCV_MAX];
  // restart: row t of the new basis row u is C[t][u] (t <= ncv, u <= k)
  double C[NCV_MAX + 1][LZ_KEEP + 1];
  double theta, resid, scale, spare;
  int32_t converged, iters, jlast, restarts;
};

// Vectors an implicit restart keeps for a call with ncv Krylov vectors.
__host__ __device__ inline int lz_keep(int ncv) { return ncv - 1 < LZ_KEEP ? ncv - 1 : LZ_KEEP; }

// partA / partB: per-chunk partial sums, [NCV_MAX + 1][nchunks] (a solve's
// partials of one sum are consecutive).  Passes that follow each other
// alternate between them (a kernel reads one while it writes the other).
// nact[0]: active solves; nact[1]: eigensolve blocks of the running
// k_update_norm that are done.
struct LzLayout {
  LzState* st;
  int32_t* act;
  double* partA;
  double* partB;
  int32_t* nact;
};

__host__ __device__ inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

__host__ __device__ inline LzLayout lz_layout(void* state, int nsolve, int nchunks) {
  char* p = (char*)state;
  LzLayout L;
  L.st = (LzState*)p;
  p += align256(sizeof(LzState) * (size_t)nsolve);
  L.act = (int32_t*)p;
  p += align256(sizeof(int32_t) * (size_t)nsolve);
  L.partA = (double*)p;
  p += align256(sizeof(double) * (size_t)nchunks * (NCV_MAX + 1));
  L.partB = (double*)p;
  p += align256(sizeof(double) * (size_t)nchunks * (NCV_MAX + 1));
  L.nact = (int32_t*)p;
  return L;
}

struct ChunkInfo {
  int s;        // solve index
  int c;        // chunk within solve
  int nch;      // chunks of this solve
  int i0, i1;   // element range
};

__device__ __forceinline__ ChunkInfo chunk_of(const tnx_lanczos_solve* solves, int nsolve,
                                           int b = -1) {
  if (b < 0) b = blockIdx.x;   // chunk index (the block index unless offset)
  ChunkInfo ci;
  ci.s = tnx_find_owner(solves, sizeof(tnx_lanczos_solve), offsetof(tnx_lanczos_solve, chunk_begin),
                        nsolve, b);
  const int n = solves[ci.s].n;
  ci.c = b - solves[ci.s].chunk_begin;
  ci.nch = (n + CHUNK - 1) / CHUNK;
  ci.i0 = ci.c * CHUNK;
  ci.i1 = min(n, ci.i0 + CHUNK);
  return ci;
}

typedef double (*Red)[NCV_MAX + 1];   // wavefront sums, red[wave][k]

// R = 4, 8 or 16 sums over the wavefront at once, of v[0..R), into
// red[k0..k0 + R).  Each step of the butterfly halves the sums a lane carries
// as well as the lanes that share one: the exchange moves one value of a pair
// each way.  63 instructions for 16 sums, where 16 butterflies take 288.
template <int R> __device__ __forceinline__ void wave_sums(const double* v, int k0, double* red) {
  const int lane = threadIdx.x & 63;
  double s[R / 2];
#pragma unroll
  for (int u = 0; u < R / 2; ++u) {
    double p = v[u], q = v[u + R / 2];
    tnx_swap<true>(p, q);
    s[u] = p + q;
  }
#pragma unroll
  for (int u = 0; u < R / 4; ++u) {
    double p = s[u], q = s[u + R / 4];
    tnx_swap<false>(p, q);
    s[u] = p + q;
  }
  int k = (lane >> 5) * (R / 2) + ((lane >> 4) & 1) * (R / 4);
  if constexpr (R >= 8) {
    const bool up = lane & 8;
#pragma unroll
    for (int u = 0; u < R / 8; ++u) {
      const double keep = up ? s[u + R / 8] : s[u], give = up ? s[u] : s[u + R / 8];
      s[u] = keep + tnx_row_get<0x128>(give);
    }
    k += up ? R / 8 : 0;
  } else {
    s[0] += tnx_row_get<0x128>(s[0]);
  }
  if constexpr (R == 16) {   // 0x141: lane ^ 7, the other half of the 8 lanes
    const bool up = lane & 4;
    const double keep = up ? s[1] : s[0], give = up ? s[0] : s[1];
    s[0] = keep + tnx_row_get<0x141>(give);
    k += up ? 1 : 0;
  } else {
    s[0] += tnx_row_get<0x141>(s[0]);
  }
  s[0] += tnx_row_get<0x4e>(s[0]);   // lane ^ 2, then lane ^ 1
  s[0] += tnx_row_get<0xb1>(s[0]);
  if ((lane & (64 / R - 1)) == 0) red[k0 + k] = s[0];
}
// L sums (a multiple of 4, up to 32)
template <int L> __device__ __forceinline__ void wave_sums_all(const double (&v)[L], double* red) {
  constexpr int A = L & 16, B = L & 8;
  if constexpr (L == 32) wave_sums<16>(v + 16, 16, red);
  if constexpr (L >= 16) wave_sums<16>(v, 0, red);
  if constexpr (L < 32 && B != 0) wave_sums<8>(v + A, A, red);
  if constexpr ((L & 4) != 0) wave_sums<4>(v + A + B, A + B, red);
}

// sum of the NW wavefronts' entries k
__device__ __forceinline__ double red_total(const double (*red)[NCV_MAX + 1], int k) {
  return ((red[0][k] + red[1][k]) + (red[2][k] + red[3][k])) +
         ((red[4][k] + red[5][k]) + (red[6][k] + red[7][k]));
}

// Elements of lane t of a chunk: i0 + t, i0 + t + NP.  elem: the element's
// index, that of the chunk's last element past its end.
__device__ __forceinline__ int elem(const ChunkInfo& ci, int q) {
  return min(ci.i0 + q * NP + (int)threadIdx.x, ci.i1 - 1);
}
__device__ __forceinline__ bool inside(const ChunkInfo& ci, int q) {
  return ci.i0 + q * NP + (int)threadIdx.x < ci.i1;
}

// This chunk's elements of L basis rows, row min(u, j) for u = 0..L - 1, all
// loads in flight together.
template <typename VT, int L>
__device__ __forceinline__ void load_rows(const VT TNX_GLOBAL* V, int ldv, int j,
                                          const ChunkInfo& ci, VT (&v)[L][EPT]) {
#pragma unroll
  for (int u = 0; u < L; ++u) {
    const VT TNX_GLOBAL* row = V + (int64_t)min(u, j) * ldv;
#pragma unroll
    for (int q = 0; q < EPT; ++q) v[u][q] = row[elem(ci, q)];
  }
}

// Dots of the L rows with x (zero past the chunk's end), wavefront sums into
// red[wave].
template <typename VT, int L>
__device__ __forceinline__ void rows_dots(const VT (&v)[L][EPT], const double (&x)[EPT], Red red) {
  double s[L];
#pragma unroll
  for (int u = 0; u < L; ++u) {
    s[u] = 0.0;
#pragma unroll
    for (int q = 0; q < EPT; ++q) s[u] += (double)v[u][q] * x[q];
  }
  wave_sums_all(s, red[threadIdx.x >> 6]);
}

// x -= sum_{k<=j} h[k] V[k] over this chunk (rows four at a time).
template <typename VT>
__device__ __forceinline__ void chunk_axpy(const VT TNX_GLOBAL* V, int ldv, int j,
                                           const ChunkInfo& ci, const double* h,
                                           double (&x)[EPT]) {
  for (int k0 = 0; k0 <= j; k0 += 4) {
    double v[4][EPT];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < EPT; ++q)
        v[u][q] = (double)V[(int64_t)min(k0 + u, j) * ldv + elem(ci, q)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double hk = k0 + u <= j ? h[min(k0 + u, j)] : 0.0;
#pragma unroll
      for (int q = 0; q < EPT; ++q) x[q] -= hk * v[u][q];
    }
  }
}

// Sum the partials of one solve (chunks [chunk_begin, chunk_begin + nch))
// for k in [0, nk) into dst[k], zeros for k in [nk, npad) (all NP lanes; dst
// is read after a barrier).  The partials were written by the previous kernel
// on the stream.  Wave w sums the entries k = w, w + NW, ...: its 64 lanes
// stride over the chunks and four entries are read per pass, so the loads are
// in flight together.  The summation order depends only on nch, so every
// block of a solve gets the same bits.
__device__ __forceinline__ void reduce_partials(const double* part, int nchunks, int chunk_begin,
                                                int nch, int nk, int npad, double* dst) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __shared__ double out[NW][4];
  const double TNX_GLOBAL* p = as_global<const double>((uint64_t)part) + chunk_begin;
  for (int k0 = wave; k0 < npad; k0 += 4 * NW) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = lane; c < nch; c += 64) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * NW;
        s[u] += k < nk ? p[(int64_t)min(k, nk - 1) * nchunks + c] : 0.0;
      }
    }
    wave_sums<4>(s, 0, out[wave]);
    __builtin_amdgcn_wave_barrier();
    if (lane < 4 && k0 + lane * NW < npad) dst[k0 + lane * NW] = out[wave][lane];
  }
}

// A symmetric tridiagonal problem in LDS, scaled: rows 0..pad_rows(k) - 1 with
// diagonal a[i] and squared couplings c2[i] of rows i - 1 and i (c2[0] = 0),
// entries of order one or less; rows from k on are decoupled, above the
// spectrum.
constexpr int MINOR_ROWS = 8;   // rows whose LDS reads are issued together
__device__ __forceinline__ int pad_rows(int k) { return (k + MINOR_ROWS - 1) & -MINOR_ROWS; }
constexpr double PAD_DIAG = 4.0;

// MINOR_ROWS more leading minors p_i = (a_i - x) p_{i-1} - c2_i p_{i-2} from
// row i0: one dependent operation a row, where the ratios of the minors
// (Sturm's sequence) need a division.  The pair is then scaled up if both
// have got small: MINOR_ROWS rows cannot take them from there to underflow,
// short of an x within rounding of an eigenvalue, where any count will do.
// CHANGES: *acc += the sign changes (a zero takes either sign); else the sign
// bit of *acc is set once a minor is negative.
template <bool CHANGES>
__device__ __forceinline__ void minors(const double* a, const double* c2, int i0, double x,
                                       double& p0, double& p1, int& acc, int& scaled) {
  double ar[MINOR_ROWS], cr[MINOR_ROWS];
#pragma unroll
  for (int u = 0; u < MINOR_ROWS; ++u) {
    ar[u] = a[i0 + u] - x;
    cr[u] = c2[i0 + u];
  }
#pragma unroll
  for (int u = 0; u < MINOR_ROWS; ++u) {
    const double p2 = fma(ar[u], p1, -cr[u] * p0);
    if constexpr (CHANGES) acc += (unsigned)(__double2hiint(p1) ^ __double2hiint(p2)) >> 31;
    else acc |= __double2hiint(p2);
    p0 = p1;
    p1 = p2;
  }
  const bool small = fmax(fabs(p0), fabs(p1)) < 1e-100;
  const double sc = small ? 1e100 : 1.0;
  scaled += small;
  p0 *= sc;
  p1 *= sc;
}

// Number of eigenvalues below x of the problem's k rows.
__device__ __forceinline__ int count_below(const double* a, const double* c2, int k, double x) {
  double p0 = 0.0, p1 = 1.0;
  int cnt = 0, scaled = 0;
  for (int i0 = 0; i0 < pad_rows(k); i0 += MINOR_ROWS)
    minors<true>(a, c2, i0, x, p0, p1, cnt, scaled);
  return cnt;
}

// Eigenvalue idx of the problem's k rows in [lo, hi], to `stop`, by one
// wavefront: each round 64 points, one a lane, the bracket being the
// neighbouring points around the eigenvalue.  The points are evenly spaced
// (65-fold per round), or, once the determinant has opposite signs at the
// ends of the bracket, at distances halving towards the secant's zero from
// both ends: its error is of second order in the bracket, so four or five
// rounds take the place of nine.  A secant round that gains less than an even
// one is followed by an even one.  g: a first guess in the place of the
// secant's zero, if it lies inside the bracket.  LOWEST: idx = 0.
template <bool LOWEST>
__device__ __forceinline__ double multisect(const double* a, const double* c2, int k, int idx,
                                            double lo, double hi, double stop, double g) {
  const int lane = threadIdx.x & 63;
  bool secant = g > lo && g < hi;
  for (int round = 0; round < 24; ++round) {
    const double w = hi - lo;  // all of these identical in every lane
    if (w <= stop) break;
    const double even = lo + w * (1.0 / 65.0) * (double)(lane + 1);
    const double near = lane < 32 ? g - __builtin_amdgcn_ldexp(g - lo, -(lane + 1))
                                  : g + __builtin_amdgcn_ldexp(hi - g, lane - 64);
    const double x = secant ? near : even;
    double p0 = 0.0, p1 = 1.0;
    int acc = 0, scaled = 0;
    for (int i0 = 0; i0 < pad_rows(k); i0 += MINOR_ROWS)
      minors<!LOWEST>(a, c2, i0, x, p0, p1, acc, scaled);
    const unsigned long long m = __ballot(LOWEST ? acc < 0 : acc > idx);
    const int f = m != 0ull ? __builtin_ctzll(m) : 64;   // first lane above it
    const int lu = min(f, 63), ll = max(f, 1) - 1;
    auto from = [](double v, int l) {
      const long long b = __double_as_longlong(v);
      const int lo32 = __builtin_amdgcn_readlane((int)b, l);
      const int hi32 = __builtin_amdgcn_readlane((int)(b >> 32), l);
      return __longlong_as_double(((long long)hi32 << 32) | (unsigned)lo32);
    };
    const double xu = from(x, lu), xl = from(x, ll), vu = from(p1, lu), vl = from(p1, ll);
    const bool both = f > 0 && f < 64 && __builtin_amdgcn_readlane(scaled, lu) ==
                                             __builtin_amdgcn_readlane(scaled, ll);
    if (f < 64) hi = xu;
    if (f > 0) lo = xl;
    const bool gained = 65.0 * (hi - lo) <= w;
    g = lo + (hi - lo) * vl * tnx_rcp(vl - vu);
    secant = both && (gained || !secant) && g > lo && g < hi && ((vl < 0.0) != (vu < 0.0));
  }
  return 0.5 * (lo + hi);
}

// Eigenpair idx (0: the lowest) of the k x k tridiagonal (a, b) in LDS, by one
// wavefront (all 64 lanes): *theta and y[0..k) (LDS).  work: LDS scratch of
// TRI_WORK doubles of the wavefront's own; guess: of the eigenvalue, or NaN.
// The eigenvalue is searched between the Gershgorin bounds (the smallest
// diagonal entry bounds the lowest).  The vector is that of the twisted
// factorisation: the pivots of T - theta from the top (D+) and from the bottom
// (D-), each the ratio of neighbouring minors, meet at the row r of smallest
// gamma_r = D+_r + D-_r - (a_r - theta), and z_r = 1 is continued by z_i = -b
// z_{i+1} / D+_i above and -b z_{i-1} / D-_i below it: products of ratios,
// accurate for the small components, the last of which is the residual
// estimate.  A vanishing pivot is replaced by a tiny one and one over a
// vanishing minor by a huge one (their ratios cancel).  The vector's sign is
// that of a positive component sum (as inverse iteration from a constant
// vector gives).
// Bound: the serial chains over k rows.  k_update_norm, most of which this is
// (mean over k = 1..20, one solve, MI355X): 16.1 us with Sturm sequences by
// division in 256 lanes and inverse iteration by one lane, 12.2 with minors and
// even rounds only, 8.3 with secant points, 7.9 from the last eigenvalue on.
constexpr int TRI_WORK = 6 * NCV_MAX + 2;
template <bool LOWEST>
__device__ __forceinline__ void tridiag_pair(const double* a, const double* b, int k, int idx,
                                             double* y, double* theta, double* work,
                                             double guess) {
  const int lane = threadIdx.x & 63;
  if (k == 1) {
    if (lane == 0) {
      y[0] = 1.0;
      *theta = a[0];
    }
    return;
  }
  double* as = work;
  double* c2 = work + NCV_MAX;             // NCV_MAX + 1 entries
  double* mn = work + 2 * NCV_MAX + 2;     // minors: top, top before, bottom, bottom before
  const bool in = lane < k;
  const double al = in ? a[lane] : 0.0;
  const double bl = lane + 1 < k ? b[lane] : 0.0;   // coupling of rows lane, lane + 1
  const double bm = in && lane > 0 ? b[lane - 1] : 0.0;
  const double inf = __builtin_huge_val();
  double base = tnx_wave_min(in ? al - fabs(bl) - fabs(bm) : inf);
  const double most = -tnx_wave_min(in ? -(al + fabs(bl) + fabs(bm)) : inf);
  const double top = LOWEST ? tnx_wave_min(in ? al : inf) : most;
  base -= 1e-12 * fmax(most - base, 1e-300);
  // entries relative to `base`, over a power of two near the spectrum's width
  const int ex = __builtin_amdgcn_frexp_exp(most - base);
  if (lane <= NCV_MAX) {
    const double bs = __builtin_amdgcn_ldexp(bm, -ex);
    if (lane < NCV_MAX) as[lane] = in ? __builtin_amdgcn_ldexp(al - base, -ex) : PAD_DIAG;
    c2[lane] = bs * bs;
  }
  __builtin_amdgcn_wave_barrier();
  const double stop = __builtin_amdgcn_ldexp(
      4.0 * 2.220446049250313e-16 * fmax(fabs(base), fabs(top)), -ex) + 1e-300;
  const double th = multisect<LOWEST>(
      as, c2, k, idx, 0.0, __builtin_amdgcn_ldexp(top - base, -ex) * (1.0 + 1e-12), stop,
      __builtin_amdgcn_ldexp(guess - base, -ex));
  // minors: lane 0 from the top, lane 1 from the bottom, with the one before
  // each at the same scale
  const bool up = lane & 1;
  const int kk = pad_rows(k);
  double* mw = mn + (up ? 2 * NCV_MAX : 0);
  double p0 = 0.0, p1 = 1.0;
  for (int i0 = 0; i0 < kk; i0 += MINOR_ROWS) {
    double ar[MINOR_ROWS], cr[MINOR_ROWS], p[MINOR_ROWS + 1];
#pragma unroll
    for (int u = 0; u < MINOR_ROWS; ++u) {
      ar[u] = as[up ? kk - 1 - (i0 + u) : i0 + u] - th;
      cr[u] = c2[up ? kk - (i0 + u) : i0 + u];
    }
    p[0] = p1;
#pragma unroll
    for (int u = 0; u < MINOR_ROWS; ++u) {
      const double p2 = fma(ar[u], p1, -cr[u] * p0);
      p0 = p1;
      p[u + 1] = p1 = p2;
    }
    if (lane < 2) {
#pragma unroll
      for (int u = 0; u < MINOR_ROWS; ++u) {
        const int row = up ? kk - 1 - (i0 + u) : i0 + u;
        mw[row] = p[u + 1];
        mw[NCV_MAX + row] = p[u];
      }
    }
    const double sc = fmax(fabs(p0), fabs(p1)) < 1e-100 ? 1e100 : 1.0;
    p0 *= sc;
    p1 *= sc;
  }
  __builtin_amdgcn_wave_barrier();
  const double tiny = 1e-150;
  double dt = 1.0, db = 1.0;   // pivots of row `lane`
  if (in) {
    const double t1 = mn[lane], t0 = mn[NCV_MAX + lane];
    const double u1 = mn[2 * NCV_MAX + lane], u0 = mn[3 * NCV_MAX + lane];
    dt = fabs(t0) < 1e-290 ? 1e150 : t1 * tnx_rcp(t0);
    db = fabs(u0) < 1e-290 ? 1e150 : u1 * tnx_rcp(u0);
    if (fabs(dt) < tiny) dt = tiny;
    if (fabs(db) < tiny) db = tiny;
  }
  const double gam = in ? fabs(dt + db - (as[lane] - th)) : inf;
  const double gmin = tnx_wave_min(gam);
  const int r = __ffsll((long long)__ballot(gam == gmin)) - 1;
  // ratio of z_lane to its neighbour on the side of r, then running products
  double z = 1.0;
  if (in && lane < r) z = -__builtin_amdgcn_ldexp(bl, -ex) * tnx_rcp(dt);
  else if (in && lane > r) z = -__builtin_amdgcn_ldexp(bm, -ex) * tnx_rcp(db);
#pragma unroll
  for (int o = 1; o < NCV_MAX; o <<= 1) {
    const int from = lane < r ? lane + o : lane - o;
    const double v = __shfl(z, from, 64);
    if (lane < r ? from < r : from > r) z *= v;
  }
  z = in ? z : 0.0;
  double f = tnx_rsqrt(tnx_wave_sum(z * z));
  if (tnx_wave_sum(z) < 0.0) f = -f;
  if (in) y[lane] = z * f;
  if (lane == 0) *theta = base + __builtin_amdgcn_ldexp(th, ex);
}

// dtype of a solve's x or w: the call's, or the solve's own field when the
// call passes TNX_DTYPE_PER_SOLVE
__device__ __forceinline__ int dtype_of(int call_dtype, int32_t own) {
  return call_dtype >= 0 ? call_dtype : own;
}

// ---------------------------------------------------------------- kernels

// act[s], read once per block through LDS, so that every lane of a block
// takes the same early return whenever another block clears it.
__device__ __forceinline__ bool solve_active(const int32_t* act, int s) {
  __shared__ int a;
  if (threadIdx.x == 0) a = __hip_atomic_load(act + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return a != 0;
}

// chunk partial of ||init||^2 -> partA[0][chunk]
__global__ __launch_bounds__(NP) void k_init_norm(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                  void* state, int nchunks) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  const tnx_lanczos_solve D = S[ci.s];
  const double TNX_GLOBAL* v = as_global<const double>(D.init);
  double acc = 0.0;
  for (int q = 0; q < EPT; ++q)
    if (inside(ci, q)) acc += v[elem(ci, q)] * v[elem(ci, q)];
  __shared__ double red[NW][NCV_MAX + 1];
  acc = tnx_wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][0] = acc;
  __syncthreads();
  if (threadIdx.x == 0) L.partA[blockIdx.x] = red_total(red, 0);
}

// scale = 1 / ||init|| (summed by every block); V[0] = init * scale (a flat
// vector when init == 0); x = cast(V[0]).  Block 0 of the solve resets the
// solve's state and marks it active.
__global__ __launch_bounds__(NP) void k_init_scale(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                   void* state, int nchunks, int x_dtype) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  const tnx_lanczos_solve D = S[ci.s];
  __shared__ double tot;
  reduce_partials(L.partA, nchunks, D.chunk_begin, ci.nch, 1, 1, &tot);
  __syncthreads();
  const double sc = tot > 0.0 ? 1.0 / sqrt(tot) : -1.0;
  if (ci.c == 0 && threadIdx.x < NCV_MAX) {
    LzState& st = L.st[ci.s];
    st.y[threadIdx.x] = threadIdx.x == 0 ? 1.0 : 0.0;
    if (threadIdx.x == 0) {
      st.scale = sc;
      st.converged = 0;
      st.iters = 0;
      st.jlast = 0;
      st.restarts = 0;
      st.theta = 0.0;
      st.resid = 0.0;
      L.act[ci.s] = 1;
    }
  }
  const double TNX_GLOBAL* v = as_global<const double>(D.init);
  const double flat = 1.0 / sqrt((double)D.n);
  const int xd = dtype_of(x_dtype, D.x_dtype);
  const bool vf = D.v_dtype == TNX_F32;
  for (int q = 0; q < EPT; ++q) {
    if (!inside(ci, q)) continue;
    const int i = elem(ci, q);
    double val = sc > 0.0 ? v[i] * sc : flat;
    if (vf) {
      // the basis row as stored: the start vector rounded to f32
      const float vv = (float)val;
      as_global<float>(D.V)[i] = vv;
      val = (double)vv;
    } else {
      as_global<double>(D.V)[i] = val;
    }
    tnx_store((void*)D.x, xd, i, val);
  }
}

// The two projections of a Krylov step (k_dots, k_update_dots) hold the
// chunk's part of all basis rows in registers: LV >= j + 1 rows (a multiple
// of 4, chosen by the host), so every load is issued before the first is
// used, and the second projection reads nothing again.
// Bound: latency at a few chunks, else the basis rows' bandwidth.
// us a call, dots and update/dots, f64 basis, mean over the cycles of 20
// (MI355X): one solve of 2 chunks 8.7 + 11.3 with 256 lanes, generic pointers,
// rows four at a time and a butterfly per sum, now 3.5 + 4.7; 16 solves of 32
// chunks 21 + 27, now 9 + 11.

// chunk partials of V[k] . w, k <= j -> partA
template <typename VT, int LV>
__device__ __forceinline__ void dots_body(const tnx_lanczos_solve& D, const LzLayout& L,
                                          const ChunkInfo& ci, int nchunks, int j, int wd) {
  __shared__ double red[NW][NCV_MAX + 1];
  VT v[LV][EPT];
  load_rows(as_global<const VT>(D.V), D.ldv, j, ci, v);
  double w[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    w[q] = tnx_load((const void*)D.w, wd, elem(ci, q));
    if (!inside(ci, q)) w[q] = 0.0;
  }
  rows_dots(v, w, red);
  __syncthreads();
  if ((int)threadIdx.x <= j)
    L.partA[(int64_t)threadIdx.x * nchunks + blockIdx.x] = red_total(red, threadIdx.x);
}

// pass 1
template <int LV>
__global__ __launch_bounds__(NP) void k_dots(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                             void* state, int nchunks, int j, int w_dtype,
                                             unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  if (L.act[ci.s] == 0) return;
  const tnx_lanczos_solve D = S[ci.s];
  const int wd = dtype_of(w_dtype, D.w_dtype);
  if (D.v_dtype == TNX_F32) dots_body<float, LV>(D, L, ci, nchunks, j, wd);
  else dots_body<double, LV>(D, L, ci, nchunks, j, wd);
  tnx_stamp_end(ts);
}

// h1 = sum of the pass-1 partials; r = w - sum h1[k] V[k] -> V[j+1];
// pass 2: chunk partials of V[k] . r (k <= j) and of ||r||^2 (slot j+1) -> partB.
// With an f32 basis r (kept in f64 registers for its dots and norm) is parked
// in row j+1 rounded to f32; the next pass normalises the parked row.
template <typename VT, int LV>
__device__ __forceinline__ void update_dots_body(const tnx_lanczos_solve& D, const LzLayout& L,
                                                 const ChunkInfo& ci, int nchunks, int j, int wd) {
  __shared__ double red[NW][NCV_MAX + 1];
  __shared__ double h[NCV_MAX + 1];
  VT v[LV][EPT];
  load_rows(as_global<const VT>(D.V), D.ldv, j, ci, v);
  double r[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    r[q] = tnx_load((const void*)D.w, wd, elem(ci, q));
    if (!inside(ci, q)) r[q] = 0.0;
  }
  reduce_partials(L.partA, nchunks, D.chunk_begin, ci.nch, j + 1, LV, h);
  __syncthreads();
  if (ci.c == 0 && (int)threadIdx.x <= j) L.st[ci.s].h1[threadIdx.x] = h[threadIdx.x];
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double hu = h[u];
#pragma unroll
    for (int q = 0; q < EPT; ++q) r[q] -= hu * (double)v[u][q];
  }
  VT TNX_GLOBAL* Vn = as_global<VT>(D.V) + (int64_t)(j + 1) * D.ldv;
  double nn = 0.0;  // ||r||^2
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    if (inside(ci, q)) Vn[elem(ci, q)] = (VT)r[q];
    else r[q] = 0.0;
    nn += r[q] * r[q];
  }
  rows_dots(v, r, red);
  nn = tnx_wave_sum(nn);
  __shared__ double rn[NW];
  if ((threadIdx.x & 63) == 0) rn[threadIdx.x >> 6] = nn;
  __syncthreads();
  if ((int)threadIdx.x <= j) {
    L.partB[(int64_t)threadIdx.x * nchunks + blockIdx.x] = red_total(red, threadIdx.x);
  } else if ((int)threadIdx.x == j + 1) {
    L.partB[(int64_t)threadIdx.x * nchunks + blockIdx.x] =
        ((rn[0] + rn[1]) + (rn[2] + rn[3])) + ((rn[4] + rn[5]) + (rn[6] + rn[7]));
  }
}

template <int LV>
__global__ __launch_bounds__(NP) void k_update_dots(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                    void* state, int nchunks, int j, int w_dtype,
                                                    unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  if (L.act[ci.s] == 0) return;
  const tnx_lanczos_solve D = S[ci.s];
  const int wd = dtype_of(w_dtype, D.w_dtype);
  if (D.v_dtype == TNX_F32) update_dots_body<float, LV>(D, L, ci, nchunks, j, wd);
  else update_dots_body<double, LV>(D, L, ci, nchunks, j, wd);
  tnx_stamp_end(ts);
}

// The active count after a step, written to the host by the last eigensolve
// block of k_update_norm to finish (every block has made its convergence
// decision by then): each block adds itself to the done count nact[1] and, if
// its solve converged, takes it off the active count nact[0], in one 64-bit
// atomic; the one that completes the count writes the active count to `host`
// (pinned memory the host reads after the launch's event) and clears the done
// count for the next launch.  No block waits for another.
__device__ __forceinline__ void publish_nact(const LzLayout& L, int nsolve, bool converged,
                                             int32_t* host) {
  if (threadIdx.x != 0) return;
  unsigned long long* both = (unsigned long long*)L.nact;
  const unsigned long long add = (1ull << 32) - (converged ? 1 : 0);
  const unsigned long long now =
      __hip_atomic_fetch_add(both, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
  if ((now >> 32) == (unsigned long long)nsolve) {
    if (host != nullptr) *(volatile int32_t*)host = (int32_t)(unsigned)now;
    __hip_atomic_store(both, now & 0xffffffffull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// beta_j = sqrt(||r||^2 - ||h2||^2) from the sums h[0..j] = h2, h[j+1] =
// ||r||^2 (LDS), the same bits in every wavefront; *skip: the second
// projection is negligible.
__device__ __forceinline__ double new_coupling(const double* h, int j, int v_dtype, bool* skip) {
  const int lane = threadIdx.x & 63;
  const double hl = lane <= j ? h[lane] : 0.0;
  const double hh = tnx_wave_sum(hl * hl);
  const double bb = fmax(h[j + 1] - hh, 0.0);
  const double sk = v_dtype == TNX_F32 ? LZ_REORTH_SKIP_F32 : LZ_REORTH_SKIP;
  *skip = hh <= sk * sk * bb;
  return sqrt(bb);
}

// alpha_j and beta_j of a solve, the tridiagonal eigenproblem and the
// convergence test, by one wavefront (LDS: a, b with entries 0..j-1 loaded,
// y, work).  True if the solve converged (its active flag is cleared).
__device__ __forceinline__ bool finish_step(const tnx_lanczos_solve& D, const LzLayout& L, int s,
                                            int j, double alpha, double beta, double last_theta,
                                            int min_iters, double* a, double* b, double* y,
                                            double* work) {
  const int lane = threadIdx.x & 63;
  LzState& st = L.st[s];
  __shared__ double th_s;
  if (lane == 0) {
    a[j] = alpha;
    b[j] = beta;
  }
  __builtin_amdgcn_wave_barrier();
  // the lowest eigenvalue only falls as the matrix grows: the last one is a
  // close guess
  tridiag_pair<true>(a, b, j + 1, 0, y, &th_s, work, last_theta);
  __builtin_amdgcn_wave_barrier();
  if (lane <= j) st.y[lane] = y[lane];
  const double anorm = -tnx_wave_min(
      lane <= j ? -(fabs(a[lane]) + (lane > 0 ? fabs(b[lane - 1]) : 0.0)) : 0.0);
  const double th = th_s;
  const double res = fabs(beta * y[j]);
  const double thr = fmax(D.tol_scale * fabs(1.0 - D.tau * th), D.floor_rel * fabs(th));
  const bool breakdown = beta <= 1e-14 * fmax(anorm, 1e-300);
  const bool full = (j + 1 >= D.n);
  const bool conv = full || breakdown || ((j + 1 >= min_iters) && res <= thr);
  if (lane == 0) {
    st.alpha[j] = alpha;
    st.beta[j] = beta;
    st.iters += 1;
    st.theta = th;
    st.resid = res;
    st.jlast = j;
    if (conv) {
      st.converged = 1;
      __hip_atomic_store(L.act + s, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  return conv;
}

// h2 = sum of the pass-2 partials (slots 0..j), ||r||^2 = slot j+1;
// beta_j = sqrt(||r||^2 - ||h2||^2), the norm of r - V h2 (V^T r = h2 and
// V is orthonormal; ||h2|| is at rounding level next to ||r|| except at a
// Lanczos breakdown, which the test below catches).
// Chunk blocks: V[j+1] = (r - V h2) / beta_j and x = cast(V[j+1]) over
// their chunk.  When the second
// projection is below LZ_REORTH_SKIP relative to beta_j (the usual case:
// r is already orthogonal to V to that level after the first pass), the
// correction is left out and V is not read: V[j+1] = r / beta_j, whose
// overlap with every earlier basis vector is then at most LZ_REORTH_SKIP,
// far below the semi-orthogonality (sqrt of the unit roundoff) that keeps
// the Ritz values of the tridiagonal matrix accurate to rounding.  Every
// block of a solve takes the same decision from the same sums.
// Blocks [0, nsolve), one per solve: alpha_j = h1[j] + h2[j] and beta_j (the
// same reduction, so the same bits), the tridiagonal eigenproblem and the
// convergence test (clearing act[s]; the solve's chunk blocks, which read
// act[s] when they start, then skip V[j+1] and x, unused after
// convergence).  They come first in the grid, so the serial eigensolve
// starts with the chunks' pass (blocks [nsolve, nsolve + nchunks)) instead
// of after it.
template <typename VT>
__device__ __forceinline__ void normalize_body(const tnx_lanczos_solve& D, const ChunkInfo& ci,
                                               int j, int xd, const LzLayout& L, int nchunks) {
  __shared__ double h[NCV_MAX + 1];
  __shared__ int active;
  if (threadIdx.x == 0)
    active = __hip_atomic_load(L.act + ci.s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const VT TNX_GLOBAL* V = as_global<const VT>(D.V);
  VT TNX_GLOBAL* Vn = as_global<VT>(D.V) + (int64_t)(j + 1) * D.ldv;
  double r[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) r[q] = (double)Vn[elem(ci, q)];
  reduce_partials(L.partB, nchunks, D.chunk_begin, ci.nch, j + 2, j + 2, h);
  __syncthreads();
  if (active == 0) return;
  bool skip;
  const double beta = new_coupling(h, j, D.v_dtype, &skip);
  const double inv = 1.0 / beta;
  if (!skip) chunk_axpy(V, D.ldv, j, ci, h, r);
#pragma unroll
  for (int q = 0; q < EPT; ++q)
    if (inside(ci, q)) {
      // x is the basis row as stored, so the next matvec acts on it
      const VT v = (VT)(r[q] * inv);
      Vn[elem(ci, q)] = v;
      tnx_store((void*)D.x, xd, elem(ci, q), (double)v);
    }
}

__global__ __launch_bounds__(NP) void k_update_norm(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                                    void* state, int nchunks, int j, int x_dtype,
                                                    int min_iters, int32_t* nact_host,
                                                    unsigned long long* ts) {
  tnx_stamp_begin(ts);
  LzLayout L = lz_layout(state, nsolve, nchunks);
  if ((int)blockIdx.x >= nsolve) {
    const ChunkInfo ci = chunk_of(S, nsolve, (int)blockIdx.x - nsolve);
    const tnx_lanczos_solve D = S[ci.s];
    const int xd = dtype_of(x_dtype, D.x_dtype);
    if (D.v_dtype == TNX_F32) normalize_body<float>(D, ci, j, xd, L, nchunks);
    else normalize_body<double>(D, ci, j, xd, L, nchunks);
    tnx_stamp_end(ts);
    return;
  }
  const int s = (int)blockIdx.x;
  // (only this block clears the flag in this launch; all loads are issued
  // before it is looked at)
  const int active =
      __hip_atomic_load(L.act + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const tnx_lanczos_solve D = S[s];
  LzState& st = L.st[s];
  __shared__ double h[NCV_MAX + 1];
  __shared__ double a_s[NCV_MAX], b_s[NCV_MAX], y_s[NCV_MAX], work[TRI_WORK];
  // alpha[0..j-1], beta[0..j-1] were written by earlier launches: every lane
  // loads its share (one round trip instead of a serial loop of j loads)
  if ((int)threadIdx.x < j) {
    a_s[threadIdx.x] = st.alpha[threadIdx.x];
    b_s[threadIdx.x] = st.beta[threadIdx.x];
  }
  const double h1j = st.h1[j], last = st.theta;
  reduce_partials(L.partB, nchunks, D.chunk_begin, (D.n + CHUNK - 1) / CHUNK, j + 2, j + 2, h);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  if (active == 0) {
    publish_nact(L, nsolve, false, nact_host);
    return;
  }
  if ((int)threadIdx.x <= j) st.h2[threadIdx.x] = h[threadIdx.x];
  bool skip;
  const double beta = new_coupling(h, j, D.v_dtype, &skip);
  const bool conv = finish_step(D, L, s, j, h1j + h[j], beta, last, min_iters, a_s, b_s, y_s, work);
  publish_nact(L, nsolve, conv, nact_host);
  tnx_stamp_end(ts);
}

// k_dots, k_update_dots and k_update_norm of one Krylov step in one launch, for
// solves of at most NG chunks: a workgroup per solve, NP lanes per chunk, the
// basis rows and r in registers throughout and the sums through LDS.  The
// sums are those of the three passes in the same order (a solve's result does
// not depend on what it shares a call with).
// Bound: latency, mostly the eigensolve's, and one CU's loads of the basis rows.
// us a step, mean over the cycles of 20 (MI355X), and two launches fewer: one
// chunk 8.3, two 13.3, the three passes 17.  More chunks in a workgroup would
// read their rows (650 KB for four) at one CU's rate.
template <typename VT, int LV, int NG>
__device__ __forceinline__ void step_small_body(const tnx_lanczos_solve& D, const LzLayout& L,
                                                int s, int nsolve, int j, int wd, int xd,
                                                int min_iters, int32_t* nact_host) {
  __shared__ double red[NG * NW][NCV_MAX + 1], rn[NG * NW];
  __shared__ double h[NCV_MAX + 1];
  __shared__ double a_s[NCV_MAX], b_s[NCV_MAX], y_s[NCV_MAX], work[TRI_WORK];
  const int t = threadIdx.x, g = t / NP;
  // lanes g NP .. g NP + NP - 1 have chunk g (elem, inside add the lane)
  ChunkInfo ci;
  ci.i0 = g * (CHUNK - NP);
  ci.i1 = min(D.n, (g + 1) * CHUNK);
  LzState& st = L.st[s];
  VT v[LV][EPT];
  load_rows(as_global<const VT>(D.V), D.ldv, j, ci, v);
  double r[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    r[q] = tnx_load((const void*)D.w, wd, elem(ci, q));
    if (!inside(ci, q)) r[q] = 0.0;
  }
  const double last = st.theta;
  if (t < j) {
    a_s[t] = st.alpha[t];
    b_s[t] = st.beta[t];
  }
  rows_dots(v, r, red);
  __syncthreads();
  auto total = [&](int k) {
    double x = red_total(red, k);
    if constexpr (NG == 2) x += red_total(red + NW, k);
    return x;
  };
  if (t < LV) {
    const double x = t <= j ? total(t) : 0.0;
    h[t] = x;
    if (t <= j) st.h1[t] = x;
  }
  __syncthreads();
  const double h1j = h[j];
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double hu = h[u];
#pragma unroll
    for (int q = 0; q < EPT; ++q) r[q] -= hu * (double)v[u][q];
  }
  double nn = 0.0;
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    if (!inside(ci, q)) r[q] = 0.0;
    nn += r[q] * r[q];
  }
  rows_dots(v, r, red);
  nn = tnx_wave_sum(nn);
  if ((t & 63) == 0) rn[t >> 6] = nn;
  __syncthreads();
  if (t <= j) {
    h[t] = total(t);
  } else if (t == j + 1) {
    double x = ((rn[0] + rn[1]) + (rn[2] + rn[3])) + ((rn[4] + rn[5]) + (rn[6] + rn[7]));
    if constexpr (NG == 2)
      x += ((rn[8] + rn[9]) + (rn[10] + rn[11])) + ((rn[12] + rn[13]) + (rn[14] + rn[15]));
    h[t] = x;
  }
  __syncthreads();
  bool skip;
  const double beta = new_coupling(h, j, D.v_dtype, &skip);
  const double inv = 1.0 / beta;
#pragma unroll
  for (int q = 0; q < EPT; ++q) r[q] = (double)(VT)r[q];   // as the three passes park it
  if (!skip) {
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const double hu = u <= j ? h[u] : 0.0;
#pragma unroll
      for (int q = 0; q < EPT; ++q) r[q] -= hu * (double)v[u][q];
    }
  }
  VT TNX_GLOBAL* Vn = as_global<VT>(D.V) + (int64_t)(j + 1) * D.ldv;
#pragma unroll
  for (int q = 0; q < EPT; ++q)
    if (inside(ci, q)) {
      const VT x = (VT)(r[q] * inv);
      Vn[elem(ci, q)] = x;
      tnx_store((void*)D.x, xd, elem(ci, q), (double)x);
    }
  if (t >= 64) return;
  if (t <= j) st.h2[t] = h[t];
  const bool conv = finish_step(D, L, s, j, h1j + h[j], beta, last, min_iters, a_s, b_s, y_s, work);
  publish_nact(L, nsolve, conv, nact_host);
}

template <int LV, int NG>
__global__ __launch_bounds__(NG * NP) void k_step_small(const tnx_lanczos_solve* __restrict__ S,
                                                        int nsolve, void* state, int nchunks,
                                                        int j, int w_dtype, int x_dtype,
                                                        int min_iters, int32_t* nact_host) {
  const LzLayout L = lz_layout(state, nsolve, nchunks);
  const int s = (int)blockIdx.x;
  // (only this block clears the flag in this launch, and not before the first
  // barrier, which every lane passes after it has read the flag)
  if (__hip_atomic_load(L.act + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
    publish_nact(L, nsolve, false, nact_host);
    return;
  }
  const tnx_lanczos_solve D = S[s];
  const int wd = dtype_of(w_dtype, D.w_dtype), xd = dtype_of(x_dtype, D.x_dtype);
  if (D.v_dtype == TNX_F32)
    step_small_body<float, LV, NG>(D, L, s, nsolve, j, wd, xd, min_iters, nact_host);
  else
    step_small_body<double, LV, NG>(D, L, s, nsolve, j, wd, xd, min_iters, nact_host);
}

// Implicit restart with the m - k largest Ritz values as shifts, from the k
// lowest Ritz pairs (one wavefront; the pairs' vectors y[i][0..m) and values
// th[i] in LDS).  What the shifted QR steps leave is determined by them: the
// new basis spans V Y, its tridiagonal matrix has their values, and only its
// last vector couples to V[m].  So in the coordinates of the Ritz vectors the
// basis is the Lanczos basis of diag(th) built backwards: the last vector is
// s / |s|, s_i = y_i[m-1], and a Lanczos recurrence from it gives the others
// down to the first and the couplings (positive, as the QR steps leave them).
// The one sign left is that of the first vector, prod (T - shift) e_1 in the
// QR steps: (-1)^(m-k) along each Ritz vector, as the shifts lie above.
// False, with nothing written, if two Ritz values are so close that their
// vectors are not independent: those vectors are each accurate to rounding
// over the gap only.
// Writes the new alpha, beta[0..k-2], the coefficients C[0..m-1] and sigma,
// the coupling of the new last vector to V[m].
__device__ __forceinline__ bool restart_from_pairs(double (*y)[NCV_MAX], const double* th, int m,
                                                   int k, double beta_m, LzState& st,
                                                   double* sigma) {
  const int lane = threadIdx.x & 63;
  double v[LZ_KEEP];
#pragma unroll
  for (int i = 0; i < LZ_KEEP; ++i) v[i] = i < k && lane < m ? y[i][lane] : 0.0;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass)
#pragma unroll
    for (int i = 1; i < LZ_KEEP; ++i)
      if (i < k) {
#pragma unroll
        for (int q = 0; q < i; ++q) v[i] -= tnx_wave_sum(v[q] * v[i]) * v[q];
        const double nn = tnx_wave_sum(v[i] * v[i]);
        if (!(nn > 1e-4)) return false;
        v[i] *= tnx_rsqrt(nn);
      }
  // From here every lane computes the same k x k numbers: z[c][i] is the
  // component of new vector c along Ritz vector i.
  double z[LZ_KEEP][LZ_KEEP], d[LZ_KEEP], s2 = 0.0;
#pragma unroll
  for (int i = 0; i < LZ_KEEP; ++i) {
    const double si = __shfl(v[i], m - 1, 64);
    d[i] = i < k ? th[i] - th[0] : 0.0;
    s2 += si * si;
#pragma unroll
    for (int c = 0; c < LZ_KEEP; ++c) z[c][i] = c == k - 1 ? si : 0.0;
  }
  const double spread = d[0] + fmax(fmax(d[1], d[2]), d[3]);
  const double sn = sqrt(s2);
  double al[LZ_KEEP], be[LZ_KEEP];
#pragma unroll
  for (int c = LZ_KEEP - 1; c >= 0; --c) {
    if (c >= k) continue;
    double w[LZ_KEEP], wn = 0.0;
    if (c == k - 1) {
#pragma unroll
      for (int i = 0; i < LZ_KEEP; ++i) w[i] = sn > 0.0 ? z[c][i] : (i == 0 ? 1.0 : 0.0);
      wn = sn > 0.0 ? s2 : 1.0;
    } else {
      // Theta z of the vector above, orthogonalised twice.  If nothing is left
      // (an invariant subspace) any orthogonal vector will do: from the unit
      // vector with the most room, and its coupling is zero to rounding.
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (u == 1 && wn > 1e-28 * spread * spread) continue;
        int row = 0;
        double room = 2.0;
#pragma unroll
        for (int i = 0; i < LZ_KEEP; ++i) {
          double q = 0.0;
#pragma unroll
          for (int l = c + 1; l < LZ_KEEP; ++l) q += l < k ? z[l][i] * z[l][i] : 0.0;
          if (i < k && q < room) {
            room = q;
            row = i;
          }
        }
#pragma unroll
        for (int i = 0; i < LZ_KEEP; ++i)
          w[i] = u == 0 ? d[i] * z[c + 1 < LZ_KEEP ? c + 1 : c][i] : (i == row ? 1.0 : 0.0);
#pragma unroll
        for (int pass = 0; pass < 2; ++pass)
#pragma unroll
          for (int l = c + 1; l < LZ_KEEP; ++l)
            if (l < k) {
              double dot = 0.0;
#pragma unroll
              for (int i = 0; i < LZ_KEEP; ++i) dot += z[l][i] * w[i];
#pragma unroll
              for (int i = 0; i < LZ_KEEP; ++i) w[i] -= dot * z[l][i];
            }
        wn = 0.0;
#pragma unroll
        for (int i = 0; i < LZ_KEEP; ++i) wn += w[i] * w[i];
        if (u == 0) be[c] = sqrt(wn);
      }
    }
    const double f = 1.0 / sqrt(wn);
    al[c] = 0.0;
#pragma unroll
    for (int i = 0; i < LZ_KEEP; ++i) {
      z[c][i] = w[i] * f;
      if (i < k) al[c] += th[i] * z[c][i] * z[c][i];
    }
  }
  // the sign, from the largest component of the first vector
  double big = 0.0, sg = 1.0;
#pragma unroll
  for (int i = 0; i < LZ_KEEP; ++i) {
    const double y0 = __shfl(v[i], 0, 64);
    if (i < k && fabs(z[0][i]) > big) {
      big = fabs(z[0][i]);
      sg = ((z[0][i] < 0.0) != (y0 < 0.0)) != (((m - k) & 1) != 0) ? -1.0 : 1.0;
    }
  }
#pragma unroll
  for (int c = 0; c < LZ_KEEP; ++c)
    if (c < k) {
      double q = 0.0;
#pragma unroll
      for (int i = 0; i < LZ_KEEP; ++i) q += v[i] * z[c][i];
      if (lane < m) st.C[lane][c] = sg * q;
      if (lane == 0) {
        st.alpha[c] = al[c];
        if (c + 1 < k) st.beta[c] = be[c];
      }
    }
  if (lane < m) st.C[lane][k] = 0.0;
  if (lane == 0) *sigma = beta_m * sg * sn;
  return true;
}

// Implicit restart, solve part (one workgroup per solve, active solves
// only), after a full cycle of m = ncv steps (V[m] is the normalised next
// Lanczos vector, beta[m-1] its coefficient): the factorisation of length k
// that implicit QR steps with the m - k largest Ritz values as shifts leave.
//  1. wavefronts 0..k-1 find the k lowest Ritz pairs, and the new basis
//     follows from them (restart_from_pairs);
//  2. when Ritz values coincide to rounding, by the QR steps themselves:
//     SH_LANES lanes search for eigenvalue k + i together, that many + 1
//     parts a round (a shift needs no more than ~1e-13 relative accuracy: any
//     shift gives a valid compressed factorisation); lane 0 applies the
//     shifts to T = tridiag(alpha, beta) (a Givens bulge chase per shift,
//     within the leading block when a subdiagonal entry has become
//     negligible) in registers (statically indexed unrolled loops) and
//     records the rotations; lane r (r < m) applies them to row r of the
//     identity: the transformation Q;
//  3. the new T (k x k) and the residual of the compressed factorisation
//        r = bhat * V Q[:, k] + beta[m-1] Q[m-1, k-1] V[m],  beta[k-1] = |r|,
//     (bhat = 0 in case 1) give the coefficients C of the new basis rows
//     0..k (k_irl_apply).
// A residual that vanishes (an invariant subspace) ends the solve as
// converged with its current Ritz pair.
// Bound: latency, a few serial chains over m rows.  us for m = 20 (MI355X):
// the QR steps with a library square root and one lane's bisection per shift
// 164, with tnx_rsqrt and SH_LANES lanes 103, from the Ritz pairs 14.4.
constexpr int SH_LANES = 8;   // NT / NCV_MAX: every shift at once
__global__ __launch_bounds__(NT) void k_irl_solve(const tnx_lanczos_solve* __restrict__ S,
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
  __shared__ double yk[LZ_KEEP][NCV_MAX], thk[LZ_KEEP], tw[LZ_KEEP][TRI_WORK], sigma_s;
  __shared__ int pairs_s;
  static_assert(NT / 64 >= LZ_KEEP, "a wavefront per kept Ritz pair");
  if (t / 64 < k) 
    tridiag_pair<false>(a_l, b_l, m, t / 64, yk[t / 64], &thk[t / 64], tw[t / 64],
                        __builtin_nan(""));
  __syncthreads();
  if (t < 64) {
    const bool ok = restart_from_pairs(yk, thk, m, k, b_l[m - 1], st, &sigma_s);
    if (t == 0) pairs_s = ok;
  }
  __syncthreads();
  const bool pairs = pairs_s != 0;
  double q[NCV_MAX];   // row t of Q (static indices: kept in registers)
  if (!pairs) {
    const int np = m - k;
    __shared__ double as_l[NCV_MAX], c2_l[NCV_MAX];
    double lo = a_l[0], hi = a_l[0];
    for (int i = 0; i < m; ++i) {
      const double r = (i < m - 1 ? fabs(b_l[i]) : 0.0) + (i > 0 ? fabs(b_l[i - 1]) : 0.0);
      lo = fmin(lo, a_l[i] - r);
      hi = fmax(hi, a_l[i] + r);
    }
    // entries relative to the lower bound, over a power of two near the span
    const int ex = __builtin_amdgcn_frexp_exp(fmax(hi - lo, 1e-300));
    const double base = lo, amax = fmax(fabs(lo), fabs(hi));
    if (t < NCV_MAX) {
      as_l[t] = t < m ? __builtin_amdgcn_ldexp(a_l[t] - base, -ex) : PAD_DIAG;
      const double bs = t > 0 && t < m ? __builtin_amdgcn_ldexp(b_l[t - 1], -ex) : 0.0;
      c2_l[t] = bs * bs;
    }
    __syncthreads();
    {
      const int i = t / SH_LANES, l = t % SH_LANES, idx = k + i;
      const double stop = __builtin_amdgcn_ldexp(1e-13 * amax, -ex) + 1e-300;
      double x0 = 0.0, x1 = __builtin_amdgcn_ldexp(hi - base, -ex);
      if (i < np) {
        for (int it = 0; it < 20 && x1 - x0 > stop; ++it) {
          const double w = (x1 - x0) * (1.0 / (SH_LANES + 1));
          const bool above = count_below(as_l, c2_l, m, x0 + w * (double)(l + 1)) >= idx + 1;
          // the group's lanes of the ballot: points from the first `above` on
          const unsigned msk = (unsigned)(__ballot(above) >> ((t & 63) - l)) & ((1u << SH_LANES) - 1);
          const int f = msk ? __ffs((int)msk) : SH_LANES + 1;
          const double o = x0;
          x0 = o + w * (double)(f - 1);
          if (f <= SH_LANES) x1 = o + w * (double)f;
        }
        if (l == 0) sh[i] = base + __builtin_amdgcn_ldexp(0.5 * (x0 + x1), ex);
      }
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
            // one reciprocal square root per rotation: the chase is a serial
            // chain, and its entries are O(|T|), far from over- or underflow
            double c = 1.0, sn = 0.0;
            if (z != 0.0) {
              const double ri = tnx_rsqrt(x * x + z * z);
              c = x * ri;
              sn = z * ri;
            }
            rc[p][u] = c;
            rs[p][u] = sn;
            if (u > 0) b[u - 1] = c * b[u - 1] + sn * bulge;
            const double au = a[u], au1 = a[u + 1], bu = b[u];
            a[u] = c * c * au + 2.0 * c * sn * bu + sn * sn * au1;
            a[u + 1] = sn * sn * au - 2.0 * c * sn * bu + c * c * au1;
            b[u] = c * sn * (au1 - au) + (c * c - sn * sn) * bu;
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
            q[u] = c * q0 + sn * q1;
            q[u + 1] = -sn * q0 + c * q1;
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
  }
  if (t == 0) {
    const double bhat = pairs ? 0.0 : bk[k - 1];
    const double sigma = pairs ? sigma_s : b_l[m - 1] * qmk;
    const double rho = hypot(bhat, sigma);
    bhat_s = bhat;
    rho_s = rho;
    double anorm = 0.0;
    for (int u = 0; u < m; ++u) anorm = fmax(anorm, fabs(a_l[u]) + fabs(b_l[u]));
    for (int u = 0; u < k && !pairs; ++u) st.alpha[u] = ak[u];
    for (int u = 0; u + 1 < k && !pairs; ++u) st.beta[u] = bk[u];
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
  if (t < m && !pairs) {
    const double f = rho_s > 0.0 ? bhat_s / rho_s : 0.0;
#pragma unroll
    for (int c = 0; c < NCV_MAX; ++c) {
      if (c < k) st.C[t][c] = q[c];
      else if (c == k) st.C[t][c] = f * q[c];
    }
  }
}

// Rows V'[u] = sum_t C[t][u] V[t] (u <= k, t <= m) of this chunk in place,
// x = cast(V'[k]) as stored.  Rows are read eight at a time, so their loads
// are in flight together.
template <typename VT>
__device__ __forceinline__ void irl_apply_rows(const tnx_lanczos_solve& D,
                                               const double (*C)[LZ_KEEP + 1],
                                               const ChunkInfo& ci, int m, int k, int xd) {
  VT TNX_GLOBAL* V = as_global<VT>(D.V);
  double acc[EPT][LZ_KEEP + 1];
#pragma unroll
  for (int q = 0; q < EPT; ++q)
#pragma unroll
    for (int u = 0; u <= LZ_KEEP; ++u) acc[q][u] = 0.0;
  for (int t0 = 0; t0 <= m; t0 += 8) {
    VT v[8][EPT];
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int q = 0; q < EPT; ++q) v[r][q] = V[(int64_t)min(t0 + r, m) * D.ldv + elem(ci, q)];
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (t0 + r <= m) {
#pragma unroll
        for (int u = 0; u <= LZ_KEEP; ++u)
          if (u <= k) {
            const double c = C[t0 + r][u];
#pragma unroll
            for (int q = 0; q < EPT; ++q) acc[q][u] += c * (double)v[r][q];
          }
      }
  }
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    if (!inside(ci, q)) continue;
    double xk = 0.0;
#pragma unroll
    for (int u = 0; u <= LZ_KEEP; ++u)
      if (u <= k) {
        const VT st = (VT)acc[q][u];
        V[(int64_t)u * D.ldv + elem(ci, q)] = st;
        if (u == k) xk = (double)st;
      }
    tnx_store((void*)D.x, xd, elem(ci, q), xk);
  }
}

// Implicit restart, basis part (chunk workgroups of the active solves): the
// new rows V'[u] = sum_t C[t][u] V[t] (u <= k, t <= m) in place (every
// element is read in full before it is written), x = cast(V'[k]).
__global__ __launch_bounds__(NP) void k_irl_apply(const tnx_lanczos_solve* __restrict__ S,
                                                  int nsolve, void* state, int nchunks, int m,
                                                  int k, int x_dtype) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  if (!solve_active(L.act, ci.s)) return;
  const tnx_lanczos_solve D = S[ci.s];
  const LzState& st = L.st[ci.s];
  __shared__ double C[NCV_MAX + 1][LZ_KEEP + 1];
  for (int e = threadIdx.x; e < (m + 1) * (LZ_KEEP + 1); e += NP)
    C[e / (LZ_KEEP + 1)][e % (LZ_KEEP + 1)] = st.C[e / (LZ_KEEP + 1)][e % (LZ_KEEP + 1)];
  __syncthreads();
  const int xd = dtype_of(x_dtype, D.x_dtype);
  if (D.v_dtype == TNX_F32) irl_apply_rows<float>(D, C, ci, m, k, xd);
  else irl_apply_rows<double>(D, C, ci, m, k, xd);
}

// out = sum_k y[k] V[k] of a chunk, eight rows' loads in flight at a time
template <typename VT>
__device__ __forceinline__ void final_rows(const tnx_lanczos_solve& D, const ChunkInfo& ci,
                                           const double* y, int kk) {
  const VT TNX_GLOBAL* V = as_global<const VT>(D.V);
  double acc[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) acc[q] = 0.0;
  for (int t0 = 0; t0 < kk; t0 += 8) {
    VT v[8][EPT];
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int q = 0; q < EPT; ++q)
        v[r][q] = V[(int64_t)min(t0 + r, kk - 1) * D.ldv + elem(ci, q)];
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (t0 + r < kk) {
#pragma unroll
        for (int q = 0; q < EPT; ++q) acc[q] += y[t0 + r] * (double)v[r][q];
      }
  }
#pragma unroll
  for (int q = 0; q < EPT; ++q)
    if (inside(ci, q)) as_global<double>(D.out)[elem(ci, q)] = acc[q];
}

// out = sum_k y[k] V[k] for every solve; the first chunk's block of each
// solve also writes its result record to `res`
__global__ __launch_bounds__(NP) void k_final(const tnx_lanczos_solve* __restrict__ S, int nsolve,
                                              void* state, int nchunks,
                                              tnx_lanczos_result* res) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  ChunkInfo ci = chunk_of(S, nsolve);
  const tnx_lanczos_solve D = S[ci.s];
  const LzState& st = L.st[ci.s];
  if (ci.c == 0 && threadIdx.x == 0) {
    res[ci.s].theta = st.theta;
    res[ci.s].resid = st.resid;
    res[ci.s].iters = st.iters;
    res[ci.s].converged = st.converged;
  }
  __shared__ double y[NCV_MAX];
  if (threadIdx.x < NCV_MAX) y[threadIdx.x] = st.y[threadIdx.x];
  __syncthreads();
  if (D.v_dtype == TNX_F32) final_rows<float>(D, ci, y, st.jlast + 1);
  else final_rows<double>(D, ci, y, st.jlast + 1);
}

#include "lanczos_in_order.h"

// pinned staging for the polled active count and the results
struct Pinned {
  int32_t* nact = nullptr;
  tnx_lanczos_result* res = nullptr;
  int res_cap = 0;
};
thread_local Pinned g_pin;

int ensure_pinned(int nsolve) {
  if (g_pin.nact == nullptr) {
    TNX_CHECK_HIP(hipHostMalloc((void**)&g_pin.nact, 64 * sizeof(int32_t), hipHostMallocDefault));
  }
  if (g_pin.res_cap < nsolve) {
    if (g_pin.res) (void)hipHostFree(g_pin.res);
    g_pin.res = nullptr;
    int cap = nsolve < 256 ? 256 : nsolve;
    TNX_CHECK_HIP(hipHostMalloc((void**)&g_pin.res, sizeof(tnx_lanczos_result) * cap, hipHostMallocDefault));
    g_pin.res_cap = cap;
  }
  return TNX_OK;
}

}  // namespace

extern "C" size_t tnx_lanczos_state_bytes(int nsolve, int nchunks, int ncv) {
  (void)ncv;
  return align256(sizeof(LzState) * (size_t)nsolve) + align256(sizeof(int32_t) * (size_t)nsolve) +
         2 * align256(sizeof(double) * (size_t)nchunks * (NCV_MAX + 1)) + 256;
}

namespace {

// Zeroes n 8-byte words (the solves' state at the start of a call; a kernel
// rather than a memset node, so the launch sequence is plain kernels) and
// sets the active count.
__global__ void k_zero_words(uint64_t* p, size_t n, int32_t* nact, int nsolve) {
  // every solve active; no block of a k_update_norm launch counted done yet
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    nact[0] = nsolve;
    nact[1] = 0;
  }
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

int check_args(const char* who, const tnx_matvec_plan* plans, int nplan,
               const tnx_lanczos_solve* solves, int nsolve, int nchunks, int ncv,
               int max_restarts, int x_dtype, int w_dtype) {
  if (plans == nullptr || nplan <= 0 || solves == nullptr || nsolve <= 0 || nchunks <= 0 ||
      ncv < 2 || ncv > NCV_MAX || max_restarts < 0 || x_dtype < -1 || x_dtype > TNX_BF16 ||
      w_dtype < -1 || w_dtype > TNX_BF16) {
    tnx_set_error("%s: bad arguments (nplan=%d nsolve=%d nchunks=%d ncv=%d)", who, nplan, nsolve,
                  nchunks, ncv);
    return TNX_EINVAL;
  }
  return TNX_OK;
}

// The launches of a call before its first Krylov step: state zeroed, every
// solve active, start vectors normalised into V[0] and x.
int issue_start(const tnx_lanczos_solve* solves, int nsolve, void* state, int nchunks,
                int x_dtype, bool in_order, hipStream_t s) {
  LzLayout L = lz_layout(state, nsolve, nchunks);
  const size_t words = sizeof(LzState) * (size_t)nsolve / sizeof(uint64_t);
  static_assert(sizeof(LzState) % sizeof(uint64_t) == 0, "LzState is whole words");
  hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((words + 255) / 256 < 1024 ? (words + 255) / 256 : 1024)),
                     dim3(256), 0, s, (uint64_t*)L.st, words, L.nact, nsolve);
  const dim3 grid(nchunks), block(in_order ? IT : NP);
  hipLaunchKernelGGL(in_order ? io_init_norm : k_init_norm, grid, block, 0, s, solves, nsolve, state,
                     nchunks);
  hipLaunchKernelGGL(in_order ? io_init_scale : k_init_scale, grid, block, 0, s, solves, nsolve,
                     state, nchunks, x_dtype);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

// The projections' instances for Krylov index j: the next multiple of 4 above
// j rows in registers.
typedef void (*BasisKernel)(const tnx_lanczos_solve*, int, void*, int, int, int,
                            unsigned long long*);
struct BasisPass {
  BasisKernel dots, update_dots;
};
typedef void (*SmallKernel)(const tnx_lanczos_solve*, int, void*, int, int, int, int, int,
                            int32_t*);
// The one-launch step for solves of at most `chunks` chunks, or null: two
// chunks are 1024 lanes, whose registers hold 20 basis rows.
SmallKernel small_pass(int j, int chunks) {
  static const SmallKernel one[NCV_MAX / 4] = {
      k_step_small<4, 1>,  k_step_small<8, 1>,  k_step_small<12, 1>, k_step_small<16, 1>,
      k_step_small<20, 1>, k_step_small<24, 1>, k_step_small<28, 1>, k_step_small<32, 1>};
  static const SmallKernel two[5] = {k_step_small<4, 2>, k_step_small<8, 2>, k_step_small<12, 2>,
                                     k_step_small<16, 2>, k_step_small<20, 2>};
  if (chunks == 1) return one[j / 4];
  return chunks == 2 && j < 20 ? two[j / 4] : nullptr;
}

// whether a call's passes keep to the fixed order of sums
bool call_in_order(const tnx_matvec_plan* plans) {
  return (plans[0].mode & TNX_GEMM_IN_ORDER) != 0;
}

BasisPass basis_pass(int j, bool in_order) {
  static const BasisPass fixed[NCV_MAX / 4] = {
      {io_pass1<4>, io_pass2<4>},   {io_pass1<8>, io_pass2<8>},   {io_pass1<12>, io_pass2<12>},
      {io_pass1<16>, io_pass2<16>}, {io_pass1<20>, io_pass2<20>}, {io_pass1<24>, io_pass2<24>},
      {io_pass1<28>, io_pass2<28>}, {io_pass1<32>, io_pass2<32>}};
  if (in_order) return fixed[j / 4];
  static const BasisPass table[NCV_MAX / 4] = {
      {k_dots<4>, k_update_dots<4>},   {k_dots<8>, k_update_dots<8>},
      {k_dots<12>, k_update_dots<12>}, {k_dots<16>, k_update_dots<16>},
      {k_dots<20>, k_update_dots<20>}, {k_dots<24>, k_update_dots<24>},
      {k_dots<28>, k_update_dots<28>}, {k_dots<32>, k_update_dots<32>}};
  return table[j / 4];
}

// Krylov step j of every active solve: each plan's matvec, then the dots,
// the update with its dots and norm, and the normalisation with the
// tridiagonal solve and the convergence test.
int issue_step(const tnx_matvec_plan* plans, int nplan, const tnx_lanczos_solve* solves,
               int nsolve, void* state, int nchunks, int j, int ncv, int min_iters, int x_dtype,
               int w_dtype, tnx_stream_t stream, int32_t* nact_host = nullptr) {
  hipStream_t s = (hipStream_t)stream;
  LzLayout L = lz_layout(state, nsolve, nchunks);
  for (int p = 0; p < nplan; ++p)
    if (int rc = tnx_heff_matvec(plans + p, L.act, stream)) return rc;
  const bool in_order = call_in_order(plans);
  const dim3 grid(nchunks), block(in_order ? IT : NP);
  // sampled timing (one plan: its modes give the x and w element sizes, and
  // the basis element size under the policy that a low-precision matvec
  // has an f32 basis); algorithmic bytes over the nchunks * CHUNK
  // elements: basis rows 0..j read once, w / r / x read or written once
  const bool prof = tnx_prof_on() && nplan == 1;
  const double E = (double)nchunks * CHUNK;
  const int m1 = plans[0].mode & 0xff, m2 = plans[0].mode2 & 0xff;
  const double xs = m1 == TNX_GEMM_F64 ? 8.0 : m1 == TNX_GEMM_F32 ? 4.0 : 2.0;
  const double ws = m2 == TNX_GEMM_F64 ? 8.0 : m2 == TNX_GEMM_BF16_BF16 ? 2.0 : 4.0;
  const double vs = m1 == TNX_GEMM_F64 ? 8.0 : 4.0;
  const double vrows = vs * (j + 1);
  tnx_prof_count(TNX_PC_DOTS, E * (vrows + ws));
  tnx_prof_count(TNX_PC_UPDATE_DOTS, E * (vrows + ws + vs));
  tnx_prof_count(TNX_PC_UPDATE_NORM, E * (2.0 * vs + xs));
  // Every solve has a chunk at least, so none has more than this.  (Sampled
  // timing keeps the three passes, which it reports one by one.)
  const int most = nchunks - nsolve + 1;
  if (const SmallKernel small = prof || in_order ? nullptr : small_pass(j, most)) {
    hipLaunchKernelGGL(small, dim3(nsolve), dim3(most * NP), 0, s, solves, nsolve, state, nchunks,
                       j, w_dtype, x_dtype, min_iters, nact_host);
    TNX_CHECK_LAUNCH();
    return TNX_OK;
  }
  int mk = prof ? tnx_prof_mark(TNX_PC_DOTS, s) : -1;
  const BasisPass pass = basis_pass(j, in_order);
  hipLaunchKernelGGL(pass.dots, grid, block, 0, s, solves, nsolve, state, nchunks, j, w_dtype,
                     tnx_prof_ts(mk));
  tnx_prof_done(mk, s, E * (vrows + ws));
  mk = prof ? tnx_prof_mark(TNX_PC_UPDATE_DOTS, s) : -1;
  hipLaunchKernelGGL(pass.update_dots, grid, block, 0, s, solves, nsolve, state, nchunks, j,
                     w_dtype, tnx_prof_ts(mk));
  tnx_prof_done(mk, s, E * (vrows + ws + vs));
  // the chunk blocks normalise V[j+1] at every step, the last of a cycle
  // included (an implicit restart combines V[ncv] into the new basis)
  (void)ncv;
  mk = prof ? tnx_prof_mark(TNX_PC_UPDATE_NORM, s) : -1;
  hipLaunchKernelGGL(in_order ? io_pass3 : k_update_norm, dim3(nchunks + nsolve), block, 0, s,
                     solves, nsolve, state, nchunks, j, x_dtype, min_iters, nact_host, tnx_prof_ts(mk));
  // (r read, V[j+1] and x written; the basis rows of the second correction,
  // read only when it is not negligible, are not counted)
  tnx_prof_done(mk, s, E * (2.0 * vs + xs));
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

// Implicit restart of the still-active solves after a full cycle: the next
// cycle continues from Krylov step lz_keep(ncv).
int issue_restart(const tnx_lanczos_solve* solves, int nsolve, void* state, int nchunks, int ncv,
                  int x_dtype, bool in_order, hipStream_t s) {
  const int k = lz_keep(ncv);
  static_assert(IT == NT, "one block size for both");
  hipLaunchKernelGGL(in_order ? io_irl_solve : k_irl_solve, dim3(nsolve), dim3(NT), 0, s, solves,
                     nsolve, state, nchunks, ncv, k);
  hipLaunchKernelGGL(k_irl_apply, dim3(nchunks), dim3(NP), 0, s, solves, nsolve, state, nchunks,
                     ncv, k, x_dtype);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

// Eigenvectors into every solve's `out`, results into `res` (device-visible).
int issue_finish(const tnx_lanczos_solve* solves, int nsolve, void* state, int nchunks,
                 tnx_lanczos_result* res, hipStream_t s) {
  hipLaunchKernelGGL(k_final, dim3(nchunks), dim3(NP), 0, s, solves, nsolve, state, nchunks, res);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

// The Lanczos loop of the entry points below: each Krylov step applies the
// nplan matvec plans in turn (one per precision of the batch), then the
// shared orthogonalisation kernels over all solves.  The host polls the
// active count one step behind the device, so one step stays queued.
// With `next` (nnext recorded launches), those launches are queued behind
// the result copies and the call returns once the results are on the host,
// while the queued launches may still run; *next_rc receives their
// tnx_run_ops code.
int lanczos_run(const tnx_matvec_plan* plans, int nplan, const tnx_lanczos_solve* solves,
                int nsolve, int nchunks, int ncv, int max_restarts, int min_iters, int x_dtype,
                int w_dtype, void* state, tnx_lanczos_result* results, tnx_stream_t stream,
                const tnx_op* next = nullptr, int nnext = 0, int32_t* next_rc = nullptr) {
  if (int rc = check_args("tnx_lanczos_run", plans, nplan, solves, nsolve, nchunks, ncv,
                          max_restarts, x_dtype, w_dtype))
    return rc;
  if (state == nullptr) {
    tnx_set_error("tnx_lanczos_run: null state");
    return TNX_EINVAL;
  }
  if (int rc = ensure_pinned(nsolve)) return rc;
  hipStream_t s = (hipStream_t)stream;
  LzLayout L = lz_layout(state, nsolve, nchunks);
  if (int rc = issue_start(solves, nsolve, state, nchunks, x_dtype, call_in_order(plans), s)) return rc;

  hipEvent_t ev[2];
  TNX_CHECK_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
  TNX_CHECK_HIP(hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
  volatile int32_t* pin = g_pin.nact;
  pin[0] = nsolve;
  pin[1] = nsolve;
  bool done = false;
  int rc = TNX_OK;
  int issued = 0;  // events recorded so far
  const bool sampled = tnx_prof_call_begin();
  for (int r = 0; r <= max_restarts && !done && !rc; ++r) {
    if (r > 0 && (rc = issue_restart(solves, nsolve, state, nchunks, ncv, x_dtype,
                                     call_in_order(plans), s))) break;
    for (int j = (r > 0 ? lz_keep(ncv) : 0); j < ncv && !done; ++j) {
      tnx_prof_set(sampled && r == 0 && j == 0);
      // lagged poll: the step writes its active count to pin[slot], then
      // wait for the previous step (the device keeps one step queued)
      const int slot = issued & 1;
      rc = issue_step(plans, nplan, solves, nsolve, state, nchunks, j, ncv, min_iters, x_dtype,
                      w_dtype, stream, (int32_t*)(pin + slot));
      tnx_prof_set(false);
      if (rc) break;
      TNX_CHECK_HIP(hipEventRecord(ev[slot], s));
      ++issued;
      if (issued >= 2) {
        const int prev = (issued - 2) & 1;
        TNX_CHECK_HIP(hipEventSynchronize(ev[prev]));
        if (pin[prev] <= 0) done = true;
      }
    }
    if (rc) break;
    if (!done) {
      // end of a Krylov cycle: make the restart decision on fresh data
      const int slot = (issued - 1) & 1;
      TNX_CHECK_HIP(hipEventSynchronize(ev[slot]));
      if (pin[slot] <= 0) done = true;
    }
  }
  (void)hipEventDestroy(ev[0]);
  (void)hipEventDestroy(ev[1]);
  if (rc) return rc;
  if ((rc = issue_finish(solves, nsolve, state, nchunks, g_pin.res, s))) return rc;
  int orc = TNX_OK;
  if (nnext > 0) {
    hipEvent_t fin;
    TNX_CHECK_HIP(hipEventCreateWithFlags(&fin, hipEventDisableTiming));
    TNX_CHECK_HIP(hipEventRecord(fin, s));
    orc = tnx_run_ops(next, nnext, stream);   // sets the message of a failure
    if (next_rc) *next_rc = orc;
    const hipError_t e = hipEventSynchronize(fin);
    (void)hipEventDestroy(fin);
    if (e != hipSuccess) {
      tnx_set_error("tnx_lanczos_run_multi_then: %s", hipGetErrorString(e));
      return TNX_EHIP;
    }
  } else {
    TNX_CHECK_HIP(hipStreamSynchronize(s));
  }
  int nconv = 0;
  for (int i = 0; i < nsolve; ++i) {
    if (results) results[i] = g_pin.res[i];
    nconv += g_pin.res[i].converged;
  }
  if (orc != TNX_OK && orc != TNX_ENOCONV) return orc;
  return nconv == nsolve ? TNX_OK : TNX_ENOCONV;
}

}  // namespace

extern "C" int tnx_lanczos_run_ex(const tnx_matvec_plan* plan, const tnx_lanczos_solve* solves,
                                  int nsolve, int nchunks, int ncv, int max_restarts,
                                  int min_iters, int x_dtype, int w_dtype, void* state,
                                  tnx_lanczos_result* results, tnx_stream_t stream) {
  return lanczos_run(plan, 1, solves, nsolve, nchunks, ncv, max_restarts, min_iters, x_dtype,
                     w_dtype, state, results, stream);
}

extern "C" int tnx_lanczos_run_multi(const tnx_matvec_plan* plans, int nplan,
                                     const tnx_lanczos_solve* solves, int nsolve, int nchunks,
                                     int ncv, int max_restarts, int min_iters, void* state,
                                     tnx_lanczos_result* results, tnx_stream_t stream) {
  return lanczos_run(plans, nplan, solves, nsolve, nchunks, ncv, max_restarts, min_iters,
                     TNX_DTYPE_PER_SOLVE, TNX_DTYPE_PER_SOLVE, state, results, stream);
}

extern "C" int tnx_lanczos_run_multi_then(const tnx_matvec_plan* plans, int nplan,
                                          const tnx_lanczos_solve* solves, int nsolve,
                                          int nchunks, int ncv, int max_restarts, int min_iters,
                                          void* state, tnx_lanczos_result* results,
                                          const tnx_op* next, int nnext, int32_t* next_rc,
                                          tnx_stream_t stream) {
  if (next_rc) *next_rc = TNX_OK;
  if (nnext < 0 || (nnext > 0 && next == nullptr)) {
    tnx_set_error("tnx_lanczos_run_multi_then: bad launch list (nnext=%d)", nnext);
    return TNX_EINVAL;
  }
  return lanczos_run(plans, nplan, solves, nsolve, nchunks, ncv, max_restarts, min_iters,
                     TNX_DTYPE_PER_SOLVE, TNX_DTYPE_PER_SOLVE, state, results, stream, next,
                     nnext, next_rc);
}

extern "C" int tnx_lanczos_run(const tnx_matvec_plan* plan, const tnx_lanczos_solve* solves,
                               int nsolve, int nchunks, int ncv, int max_restarts, int x_dtype,
                               int w_dtype, void* state, tnx_lanczos_result* results,
                               tnx_stream_t stream) {
  return tnx_lanczos_run_ex(plan, solves, nsolve, nchunks, ncv, max_restarts, 1, x_dtype, w_dtype,
                            state, results, stream);
}

// ------------------------------------------------- no-allocation entry point
//
// tnx_lanczos_run_multi_static: the same Lanczos loop with its state in a
// library-owned device array instead of a caller workspace, and no host
// staging memory: it allocates nothing on any call.  Each GPU the library
// runs on holds one copy of `scratch` until the process ends; every call on
// that GPU shares it, so calls that overlap on one GPU race.  The state is
// re-initialised by every call (nothing carries over from the last call).
namespace {

constexpr size_t LZ_STATIC_BYTES = TNX_LANCZOS_STATIC_BYTES;
static __device__ __align__(256) unsigned char scratch[LZ_STATIC_BYTES];

constexpr int MAX_DEVICES = 64;
void* g_scratch_ptr[MAX_DEVICES];   // device address of `scratch` per GPU
std::mutex g_scratch_mu;

// Device address of the current GPU's `scratch` (looked up once per GPU,
// with that GPU current).
int scratch_of_current_device(void** out) {
  int dev = -1;
  TNX_CHECK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) {
    tnx_set_error("tnx_lanczos_run_multi_static: device %d out of range", dev);
    return TNX_EINVAL;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    TNX_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TNX_OK;
}

}  // namespace

extern "C" int tnx_lanczos_run_multi_static(const tnx_matvec_plan* plans, int nplan,
                                            const tnx_lanczos_solve* solves, int nsolve,
                                            int nchunks, int ncv, int max_restarts, int min_iters,
                                            tnx_lanczos_result* results, tnx_stream_t stream) {
  const char* who = "tnx_lanczos_run_multi_static";
  if (int rc = check_args(who, plans, nplan, solves, nsolve, nchunks, ncv, max_restarts,
                          TNX_DTYPE_PER_SOLVE, TNX_DTYPE_PER_SOLVE))
    return rc;
  const size_t state_bytes = tnx_lanczos_state_bytes(nsolve, nchunks, ncv);
  const size_t need = state_bytes + align256(sizeof(tnx_lanczos_result) * (size_t)nsolve);
  if (need > LZ_STATIC_BYTES) {
    tnx_set_error("%s: %d solves over %d chunks need %zu bytes of state, more than the %zu of "
                  "the library's scratch (use tnx_lanczos_run_multi with a workspace)",
                  who, nsolve, nchunks, need, LZ_STATIC_BYTES);
    return TNX_EINVAL;
  }
  void* base = nullptr;
  if (int rc = scratch_of_current_device(&base)) return rc;
  void* state = base;
  tnx_lanczos_result* dres = (tnx_lanczos_result*)((char*)base + state_bytes);
  hipStream_t s = (hipStream_t)stream;
  LzLayout L = lz_layout(state, nsolve, nchunks);
  const bool in_order = call_in_order(plans);
  if (int rc = issue_start(solves, nsolve, state, nchunks, TNX_DTYPE_PER_SOLVE, in_order, s))
    return rc;
  // Every Krylov step of a cycle is queued without polling: a solve that has
  // converged is masked on the device, so its arithmetic, and the result,
  // are those of tnx_lanczos_run_multi.  The active count is read at the end
  // of each cycle (the restart decision).
  bool done = false;
  const bool sampled = tnx_prof_call_begin();
  for (int r = 0; r <= max_restarts && !done; ++r) {
    if (r > 0)
      if (int rc = issue_restart(solves, nsolve, state, nchunks, ncv, TNX_DTYPE_PER_SOLVE,
                                 in_order, s))
        return rc;
    for (int j = (r > 0 ? lz_keep(ncv) : 0); j < ncv; ++j) {
      tnx_prof_set(sampled && r == 0 && j == 0);
      const int rc = issue_step(plans, nplan, solves, nsolve, state, nchunks, j, ncv, min_iters,
                                TNX_DTYPE_PER_SOLVE, TNX_DTYPE_PER_SOLVE, stream);
      tnx_prof_set(false);
      if (rc) return rc;
    }
    int32_t nact = 0;
    TNX_CHECK_HIP(hipMemcpyAsync(&nact, L.nact, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    TNX_CHECK_HIP(hipStreamSynchronize(s));
    done = nact <= 0;
  }
  if (int rc = issue_finish(solves, nsolve, state, nchunks, dres, s)) return rc;
  tnx_lanczos_result* host = results;
  int nconv = 0;
  for (int i0 = 0; i0 < nsolve; i0 += 64) {   // results through a bounded stack buffer
    tnx_lanczos_result buf[64];
    const int k = nsolve - i0 < 64 ? nsolve - i0 : 64;
    TNX_CHECK_HIP(hipMemcpyAsync(buf, dres + i0, sizeof(tnx_lanczos_result) * (size_t)k,
                                 hipMemcpyDeviceToHost, s));
    TNX_CHECK_HIP(hipStreamSynchronize(s));
    for (int i = 0; i < k; ++i) {
      if (host) host[i0 + i] = buf[i];
      nconv += buf[i].converged;
    }
  }
  return nconv == nsolve ? TNX_OK : TNX_ENOCONV;
}
