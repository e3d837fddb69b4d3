// Elementwise kernels of the DMRG step: the physical-index mixer
//   dst[a,s,b] (=|+=) sum_terms coef * sum_t O[s,t] src[a,t,b]
// (which is also the linear combination of environment matrices and the
// dtype cast), batched traces / Frobenius products, the matvec composition
// and the library's error/version entry points.
#include <stdarg.h>

#include <type_traits>

#include "tnx_common.h"

static thread_local std::string g_last_error;

void tnx_set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
}

namespace {

constexpr int MIX_DMAX = 4;   // largest physical dimension (the operator table holds 4 x 4)

// (a, b) pairs per lane and per workgroup of a job of physical dimension d:
// jobs with d <= 2 (spin-1/2 sites) take 4 pairs per lane, larger d 2 (the
// registers of a lane hold PPT x d sources and PPT x d sums either way).
__host__ __device__ constexpr int mix_ppt(int d) { return d <= 2 ? 4 : 2; }

template <int DT> struct Elem { typedef double T; };
template <> struct Elem<TNX_F32> { typedef float T; };
template <> struct Elem<TNX_BF16> { typedef __bf16 T; };
template <typename TI> __device__ __forceinline__ double widen(TI v) { return (double)v; }
template <> __device__ __forceinline__ double widen<__bf16>(__bf16 v) { return (double)(float)v; }

// a buffer whose groups of 4 elements are one piece
__device__ __forceinline__ bool aligned4(uint64_t p, int dtype) {
  const int isz = dtype == TNX_F64 ? 8 : dtype == TNX_F32 ? 4 : 2;
  return (p & (uint64_t)(4 * isz - 1)) == 0;
}

// Four consecutive elements at e (a multiple of 4) of an aligned4 buffer.
template <int DT>
__device__ __forceinline__ void store4(uint64_t p, int64_t e, const double (&v)[4], bool add) {
  typedef typename Elem<DT>::T TI;
  typedef TI V4 __attribute__((ext_vector_type(4)));
  V4 TNX_GLOBAL* d = as_global<V4>(p) + e / 4;
  V4 o;
  if (add) o = *d;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double x = add ? v[q] + widen<TI>(o[q]) : v[q];
    if constexpr (DT == TNX_BF16) o[q] = (TI)(float)x;
    else o[q] = (TI)x;
  }
  *d = o;
}

// Element e of a destination of dtype DT (+)= v.
template <int DT>
__device__ __forceinline__ void store1(uint64_t p, int64_t e, double v, bool add) {
  typedef typename Elem<DT>::T TI;
  TI TNX_GLOBAL* d = as_global<TI>(p) + e;
  if (add) v += widen<TI>(*d);
  if constexpr (DT == TNX_BF16) *d = (TI)(float)v;
  else *d = (TI)v;
}

// One workgroup of a job whose sources all have dtype DT: 256 lanes, PPT
// (a, b) pairs each; the D source values of a term and pair are mixed by the
// D x D operator in registers, so each output element costs one load per term.
// TB terms at a time: their records, then their operators (scalar loads) and
// every source element, before the first is used.  An element gets its terms in order, whichever instance runs
// it (the same bits).
// VEC (d <= 2, Dr % 4 == 0, everything aligned4): the lane's 4 pairs are
// consecutive, in one row, and a row is one load or store; otherwise the pairs
// are 256 apart.
// Bound: latency for a few blocks (owner, job, terms and sources follow each
// other), else memory.  us a matvec's launch (MI355X), by terms one at a time,
// a record and an operator waited for in each, and now: a 30 x 27 problem 6.3
// and 4.9; 64 of 128 x 128 in bf16 (41 MB) 20.1 and 16.4, in f64 (147 MB) 25.9
// and 24.2.
template <int D, bool VEC, int DT, int TB>
__device__ __forceinline__ void mix_body(const tnx_mix_job TNX_CONST& J, int blk,
                                         const tnx_mix_term TNX_CONST* T,
                                         const double TNX_CONST* ops) {
  constexpr int PPT = mix_ppt(D);
  static_assert(!VEC || PPT == 4, "a row's piece is 4 elements");
  typedef typename Elem<DT>::T TI;
  typedef TI V4 __attribute__((ext_vector_type(4)));
  const int Dr = J.Dr, count = J.term_count;
  const int npairs = J.Dl * Dr;
  int64_t e0[PPT];  // element (a, 0, b) of each pair (past the end: of the last one)
  bool ok[PPT];
#pragma unroll
  for (int q = 0; q < PPT; ++q) {
    const int p = blk * 256 * PPT + (VEC ? 4 * (int)threadIdx.x + q : q * 256 + (int)threadIdx.x);
    ok[q] = p < npairs;
    if (VEC && q > 0) {
      e0[q] = e0[0] + q;
    } else {
      const int pc = min(p, npairs - (VEC ? 4 : 1));
      const int a = pc / Dr;
      e0[q] = (int64_t)a * D * Dr + (pc - a * Dr);
    }
  }
  double acc[D][PPT];
#pragma unroll
  for (int s = 0; s < D; ++s)
#pragma unroll
    for (int q = 0; q < PPT; ++q) acc[s][q] = 0.0;
  for (int t0 = 0; t0 < count; t0 += TB) {
    const int n = count - t0;
    uint64_t src[TB];
    double coef[TB], O[TB][D * D];
    int op[TB];
    TI x[TB][D][PPT];
#pragma unroll
    for (int u = 0; u < TB; ++u) {
      const tnx_mix_term TNX_CONST& t = T[min(t0 + u, count - 1)];
      src[u] = t.src;
      coef[u] = t.coef;
      op[u] = t.op;
    }
#pragma unroll
    for (int u = 0; u < TB; ++u) {
      const double TNX_CONST* Op = ops + (int64_t)max(op[u], 0) * (D * D);
      if (op[u] >= 0) {
#pragma unroll
        for (int k = 0; k < D * D; ++k) O[u][k] = Op[k];
      }
    }
#pragma unroll
    for (int u = 0; u < TB; ++u)
      if (u < n) {
        const TI TNX_GLOBAL* sp = as_global<const TI>(src[u]);
#pragma unroll
        for (int t = 0; t < D; ++t) {
          const int64_t row = (int64_t)t * Dr;
          if constexpr (VEC) {
            const V4 v = *(const V4 TNX_GLOBAL*)(sp + e0[0] + row);
#pragma unroll
            for (int q = 0; q < 4; ++q) x[u][t][q] = v[q];
          } else {
#pragma unroll
            for (int q = 0; q < PPT; ++q) x[u][t][q] = sp[e0[q] + row];
          }
        }
      }
#pragma unroll
    for (int u = 0; u < TB; ++u)
      if (u < n) {
        double w[D][PPT];
#pragma unroll
        for (int t = 0; t < D; ++t)
#pragma unroll
          for (int q = 0; q < PPT; ++q) w[t][q] = widen<TI>(x[u][t][q]);
        if (op[u] < 0) {
#pragma unroll
          for (int s = 0; s < D; ++s)
#pragma unroll
            for (int q = 0; q < PPT; ++q) acc[s][q] += coef[u] * w[s][q];
        } else {
#pragma unroll
          for (int s = 0; s < D; ++s)
#pragma unroll
            for (int q = 0; q < PPT; ++q) {
              double m = 0.0;
#pragma unroll
              for (int t = 0; t < D; ++t) m += O[u][s * D + t] * w[t][q];
              acc[s][q] += coef[u] * m;
            }
        }
      }
  }
  const bool add = J.accumulate != 0;
  auto store = [&](auto tag) {
    constexpr int DD = decltype(tag)::value;
#pragma unroll
    for (int s = 0; s < D; ++s) {
      const int64_t row = (int64_t)s * Dr;
      if constexpr (VEC) {
        if (ok[0]) store4<DD>(J.dst, e0[0] + row, acc[s], add);
      } else {
#pragma unroll
        for (int q = 0; q < PPT; ++q)
          if (ok[q]) store1<DD>(J.dst, e0[q] + row, acc[s][q], add);
      }
    }
  };
  if (J.dst_dtype == TNX_F64) store(std::integral_constant<int, TNX_F64>());
  else if (J.dst_dtype == TNX_F32) store(std::integral_constant<int, TNX_F32>());
  else store(std::integral_constant<int, TNX_BF16>());
}

// The same for a job whose sources differ in dtype: element by element.
__device__ __forceinline__ void mix_mixed(const tnx_mix_job TNX_CONST& J, int blk,
                                          const tnx_mix_term TNX_CONST* T,
                                          const double TNX_CONST* ops) {
  const int d = J.d, Dr = J.Dr, per = 256 * mix_ppt(d);
  const int end = min(J.Dl * Dr, (blk + 1) * per);
  for (int p = blk * per + (int)threadIdx.x; p < end; p += 256) {
    const int a = p / Dr;
    const int64_t e0 = (int64_t)a * d * Dr + (p - a * Dr);
    double acc[MIX_DMAX] = {0.0, 0.0, 0.0, 0.0};
    for (int u = 0; u < J.term_count; ++u) {
      const double coef = T[u].coef;
      double x[MIX_DMAX];
#pragma unroll
      for (int t = 0; t < MIX_DMAX; ++t)
        x[t] = tnx_load((const void*)T[u].src, T[u].src_dtype, e0 + (int64_t)min(t, d - 1) * Dr);
      const double TNX_CONST* O = ops + (int64_t)max(T[u].op, 0) * d * d;
#pragma unroll
      for (int s = 0; s < MIX_DMAX; ++s) {
        double m = x[s];
        if (T[u].op >= 0) {
          m = 0.0;
#pragma unroll
          for (int t = 0; t < MIX_DMAX; ++t)
            if (s < d && t < d) m += O[s * d + t] * x[t];
        }
        acc[s] += coef * m;
      }
    }
#pragma unroll
    for (int s = 0; s < MIX_DMAX; ++s)
      if (s < d) {
        const int64_t e = e0 + (int64_t)s * Dr;
        if (J.accumulate) acc[s] += tnx_load((const void*)J.dst, J.dst_dtype, e);
        tnx_store((void*)J.dst, J.dst_dtype, e, acc[s]);
      }
  }
}

// The job that owns block `bid`: jobs of a launch are mostly of one size, so
// the record at its share of the range is tried first, then the search.
__device__ __forceinline__ int find_job(const tnx_mix_job* jobs, int njob, int bid, int nblocks) {
  const tnx_mix_job TNX_CONST* J = (const tnx_mix_job TNX_CONST*)(uint64_t)jobs;
  const int guess = __builtin_amdgcn_readfirstlane((int)((int64_t)bid * njob / nblocks));
  const int lo = J[guess].block_begin;
  const int hi = guess + 1 < njob ? J[min(guess + 1, njob - 1)].block_begin : nblocks;
  if (bid >= lo && bid < hi) return guess;
  return tnx_find_owner(jobs, sizeof(tnx_mix_job), offsetof(tnx_mix_job, block_begin), njob, bid);
}

// DT: the matvec's mixer, whose sources have the dtype of its first GEMM's
// operands (a job with others goes element by element); -1: any mix.  With
// one dtype's bodies the bf16 instance needs 77 registers instead of 99, and
// more workgroups are in flight.
template <int DT>
__global__ __launch_bounds__(256) void mix_kernel(const tnx_mix_job* __restrict__ jobs, int njob,
                                                  const tnx_mix_term* __restrict__ terms,
                                                  const double* __restrict__ ops,
                                                  const int32_t* __restrict__ active,
                                                  unsigned long long* ts) {
  tnx_stamp_begin(ts);
  const int bid = tnx_xcd_remap(blockIdx.x, gridDim.x);
  const int ji = __builtin_amdgcn_readfirstlane(find_job(jobs, njob, bid, gridDim.x));
  const tnx_mix_job TNX_CONST& J = ((const tnx_mix_job TNX_CONST*)(uint64_t)jobs)[ji];
  const int on = J.active >= 0 && active != nullptr
                     ? ((const int32_t TNX_CONST*)(uint64_t)active)[J.active] : 1;
  if (on == 0) return;
  const double TNX_CONST* O = (const double TNX_CONST*)(uint64_t)ops;
  const int blk = bid - J.block_begin;
  // the sources' dtype and alignments
  const tnx_mix_term TNX_CONST* T = (const tnx_mix_term TNX_CONST*)(uint64_t)terms + J.term_begin;
  const int count = J.term_count, dt = count > 0 ? T[0].src_dtype : TNX_F64;
  bool same = true, vec = J.d <= 2 && J.Dr % 4 == 0 && aligned4(J.dst, J.dst_dtype);
  for (int u0 = 0; u0 < count; u0 += 4)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const tnx_mix_term TNX_CONST& t = T[min(u0 + u, count - 1)];
      same = same && t.src_dtype == dt;
      vec = vec && aligned4(t.src, t.src_dtype);
    }
#define TNX_MIX(DT)                                                  \
  if (vec && J.d == 2) mix_body<2, true, DT, 4>(J, blk, T, O);       \
  else if (vec) mix_body<1, true, DT, 4>(J, blk, T, O);              \
  else if (J.d == 1) mix_body<1, false, DT, 4>(J, blk, T, O);        \
  else if (J.d == 2) mix_body<2, false, DT, 2>(J, blk, T, O);        \
  else if (J.d == 3) mix_body<3, false, DT, 1>(J, blk, T, O);        \
  else mix_body<4, false, DT, 1>(J, blk, T, O)
  if constexpr (DT >= 0) {
    if (same && dt == DT) {
      TNX_MIX(DT);
    } else {
      mix_mixed(J, blk, T, O);
    }
  } else if (!same) {
    mix_mixed(J, blk, T, O);
  } else if (dt == TNX_F64) {
    TNX_MIX(TNX_F64);
  } else if (dt == TNX_F32) {
    TNX_MIX(TNX_F32);
  } else {
    TNX_MIX(TNX_BF16);
  }
#undef TNX_MIX
  tnx_stamp_end(ts);
}

__global__ __launch_bounds__(256) void trace_dot_kernel(const tnx_dot_job* __restrict__ jobs,
                                                        double* __restrict__ out) {
  const tnx_dot_job J = jobs[blockIdx.x];
  const double* X = (const double*)J.x;
  const double* Y = (const double*)J.y;
  double acc = 0.0;
  if (Y == nullptr) {
    const int nd = J.rows < J.cols ? J.rows : J.cols;
    for (int i = threadIdx.x; i < nd; i += 256) acc += X[(int64_t)i * J.ldx + i];
  } else {
    const int64_t tot = (int64_t)J.rows * J.cols;
    for (int64_t e = threadIdx.x; e < tot; e += 256) {
      int64_t r = e / J.cols, c = e - r * J.cols;
      acc += X[r * J.ldx + c] * Y[r * J.ldy + c];
    }
  }
  __shared__ double red[4];
  acc = tnx_wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// x /= ||x|| for one job per workgroup: the sum of squares in a fixed order
// (lane-strided partials, then the wave and workgroup sums), then the scale.
__global__ __launch_bounds__(1024) void normalize_kernel(const tnx_norm_job* __restrict__ jobs) {
  const tnx_norm_job J = jobs[blockIdx.x];
  double* x = (double*)J.x;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < J.n; i += 1024) acc += x[i] * x[i];
  __shared__ double red[16];
  __shared__ double scale;
  acc = tnx_wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < 16; ++w) t += red[w];
    scale = t > 0.0 ? 1.0 / sqrt(t) : 1.0;
  }
  __syncthreads();
  const double sc = scale;
  for (int64_t i = threadIdx.x; i < J.n; i += 1024) x[i] *= sc;
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC 2011): ten rounds of two 32 x 32 -> 64 multiplies on
// a 128-bit counter under a 64-bit key bumped by the Weyl constants.
__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// dst[i] = normal number (offset + i) of the stream of `seed`: pair q =
// (offset + i) / 2 comes from Philox of counter (q, 0) -> two 53-bit
// uniforms in (0, 1) -> Box-Muller (cos, sin).
__global__ __launch_bounds__(256) void fill_normal_kernel(const tnx_fill_job* __restrict__ jobs) {
  const tnx_fill_job J = jobs[blockIdx.x];
  double* x = (double*)J.dst;
  const uint32_t k0 = (uint32_t)J.seed, k1 = (uint32_t)(J.seed >> 32);
  for (int64_t i = threadIdx.x; i < J.n; i += 256) {
    const uint64_t g = (uint64_t)(J.offset + i);
    const uint64_t q = g >> 1;
    uint32_t c[4] = {(uint32_t)q, (uint32_t)(q >> 32), 0u, 0u};
    philox4x32_10(c, k0, k1);
    const uint64_t a = ((uint64_t)c[0] << 32) | c[1];
    const uint64_t b = ((uint64_t)c[2] << 32) | c[3];
    const double u1 = ((double)(a >> 11) + 0.5) * 1.1102230246251565e-16;   // 2^-53
    const double u2 = ((double)(b >> 11) + 0.5) * 1.1102230246251565e-16;
    const double r = sqrt(-2.0 * log(u1));
    double sn, cs;
    sincospi(2.0 * u2, &sn, &cs);
    x[i] = (g & 1) ? r * sn : r * cs;
  }
}

}  // namespace

extern "C" int tnx_fill_normal_f64(const tnx_fill_job* jobs, int njob, tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || njob < 0) {
    tnx_set_error("tnx_fill_normal_f64: bad arguments (njob=%d)", njob);
    return TNX_EINVAL;
  }
  hipLaunchKernelGGL(fill_normal_kernel, dim3(njob), dim3(256), 0, (hipStream_t)stream, jobs);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

extern "C" int tnx_normalize_f64(const tnx_norm_job* jobs, int njob, tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || njob < 0) {
    tnx_set_error("tnx_normalize_f64: bad arguments (njob=%d)", njob);
    return TNX_EINVAL;
  }
  hipLaunchKernelGGL(normalize_kernel, dim3(njob), dim3(1024), 0, (hipStream_t)stream, jobs);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

extern "C" int tnx_version(void) { return TNX_VERSION; }

extern "C" const char* tnx_last_error(void) { return g_last_error.c_str(); }

extern "C" int tnx_abi_sizes(int32_t* sizes, int n) {
  const int32_t all[] = {(int32_t)sizeof(tnx_gemm_seg),      (int32_t)sizeof(tnx_gemm_problem),
                         (int32_t)sizeof(tnx_mix_job),       (int32_t)sizeof(tnx_mix_term),
                         (int32_t)sizeof(tnx_matvec_plan),   (int32_t)sizeof(tnx_lanczos_solve),
                         (int32_t)sizeof(tnx_lanczos_result), (int32_t)sizeof(tnx_qr_job),
                         (int32_t)sizeof(tnx_svd_job),       (int32_t)sizeof(tnx_dot_job),
                         (int32_t)sizeof(tnx_chol_job),      (int32_t)sizeof(tnx_svdj_job),
                         (int32_t)sizeof(tnx_prof_stat),     (int32_t)sizeof(tnx_norm_job),
                         (int32_t)sizeof(tnx_fill_job),      (int32_t)sizeof(tnx_kron_term),
                         (int32_t)sizeof(tnx_kron_job),      (int32_t)sizeof(tnx_sym_job),
                         (int32_t)sizeof(tnx_op)};
  const int na = (int)(sizeof(all) / sizeof(all[0]));
  if (sizes == nullptr) return na;
  for (int i = 0; i < n && i < na; ++i) sizes[i] = all[i];
  return na;
}

static int launch_mix(const tnx_mix_job* job, int njob, const tnx_mix_term* term, int nblocks,
                      const double* ops, const int32_t* active, tnx_stream_t stream, int dt,
                      unsigned long long* ts = nullptr) {
  if (nblocks == 0 || njob == 0) return TNX_OK;
  if (job == nullptr || term == nullptr || nblocks < 0 || njob < 0) {
    tnx_set_error("tnx_mix: bad arguments (njob=%d nblocks=%d)", njob, nblocks);
    return TNX_EINVAL;
  }
  auto kernel = dt == TNX_F64    ? mix_kernel<TNX_F64>
                : dt == TNX_F32  ? mix_kernel<TNX_F32>
                : dt == TNX_BF16 ? mix_kernel<TNX_BF16>
                                 : mix_kernel<-1>;
  hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(256), 0, (hipStream_t)stream, job, njob, term, ops,
                     active, ts);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

extern "C" int tnx_mix(const tnx_mix_job* job, int njob, const tnx_mix_term* term, int nblocks,
                       const double* ops, const int32_t* active, tnx_stream_t stream) {
  return launch_mix(job, njob, term, nblocks, ops, active, stream, -1);
}

extern "C" int tnx_trace_dot(const tnx_dot_job* jobs, int njob, double* out, tnx_stream_t stream) {
  if (njob == 0) return TNX_OK;
  if (jobs == nullptr || out == nullptr || njob < 0) {
    tnx_set_error("tnx_trace_dot: bad arguments");
    return TNX_EINVAL;
  }
  hipLaunchKernelGGL(trace_dot_kernel, dim3(njob), dim3(256), 0, (hipStream_t)stream, jobs, out);
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}

// Timing class of a matvec GEMM launch (the variant byte of the mode aside).
static int gemm_class(int mode, int second) {
  switch (mode & 0xff) {
    case TNX_GEMM_F64: return TNX_PC_GEMM_F64_1 + second;
    case TNX_GEMM_F32: return TNX_PC_GEMM_F32_1 + second;
    default: return TNX_PC_GEMM_BF16_1 + second;
  }
}

extern "C" int tnx_heff_matvec(const tnx_matvec_plan* plan, const int32_t* active,
                               tnx_stream_t stream) {
  if (plan == nullptr) {
    tnx_set_error("tnx_heff_matvec: null plan");
    return TNX_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  const bool prof = tnx_prof_on();
  tnx_prof_count(gemm_class(plan->mode, 0), plan->work[0]);
  if (plan->mix_nblocks > 0) tnx_prof_count(TNX_PC_MIX, plan->work[1]);
  tnx_prof_count(gemm_class(plan->mode2, 1), plan->work[2]);
  int mk = prof ? tnx_prof_mark(gemm_class(plan->mode, 0), s) : -1;
  int rc = tnx_gemm_grouped_ts(plan->mode, plan->g1_prob, plan->g1_nprob, plan->g1_seg,
                               plan->g1_ntiles, active, stream, tnx_prof_ts(mk));
  if (rc) return rc;
  tnx_prof_done(mk, s, plan->work[0]);
  mk = (prof && plan->mix_nblocks > 0) ? tnx_prof_mark(TNX_PC_MIX, s) : -1;
  const int m1 = plan->mode & 0xff;
  rc = launch_mix(plan->mix_job, plan->mix_njob, plan->mix_term, plan->mix_nblocks, plan->ops, active,
                  stream, m1 == TNX_GEMM_F64 ? TNX_F64 : m1 == TNX_GEMM_F32 ? TNX_F32 : TNX_BF16,
                  tnx_prof_ts(mk));
  if (rc) return rc;
  tnx_prof_done(mk, s, plan->work[1]);
  mk = prof ? tnx_prof_mark(gemm_class(plan->mode2, 1), s) : -1;
  rc = tnx_gemm_grouped_ts(plan->mode2, plan->g2_prob, plan->g2_nprob, plan->g2_seg,
                           plan->g2_ntiles, active, stream, tnx_prof_ts(mk));
  if (rc) return rc;
  tnx_prof_done(mk, s, plan->work[2]);
  return TNX_OK;
}
