// Grouped, K-concatenated GEMM on CDNA4 matrix cores (MFMA), the contraction
// engine of the DMRG effective-Hamiltonian matvec and environment updates.
//
// One launch covers every output matrix ("problem") of a sweep step for all
// solves of a batch; problem p owns the 64x64 output tiles
// [tile_begin_p, tile_begin_{p+1}).  A problem sums several K-segments, each
// an (optionally transposed) A x B product with its own alpha, so the whole
// sum_k L_k x_k or sum_r U_r R_r^T of one local step is one accumulation in
// registers.
//   f64 : v_mfma_f64_16x16x4_f64    f32: v_mfma_f32_16x16x4_f32
//   bf16: v_mfma_f32_16x16x32_bf16 (f32 accumulate)
#include <type_traits>

#include "tnx_common.h"

namespace {

template <int MODE> struct Tr;
template <> struct Tr<TNX_GEMM_F64> {
  typedef double TI; typedef double TC; typedef tnx_d4 V4;
};
template <> struct Tr<TNX_GEMM_F32> {
  typedef float TI; typedef float TC; typedef tnx_f4 V4;
};
template <> struct Tr<TNX_GEMM_BF16_F32> {
  typedef __bf16 TI; typedef float TC; typedef tnx_f4 V4;
};
template <> struct Tr<TNX_GEMM_BF16_BF16> {
  typedef __bf16 TI; typedef __bf16 TC; typedef tnx_f4 V4;
};

template <typename T> __device__ __forceinline__ double to_d(T v) { return (double)v; }
template <> __device__ __forceinline__ double to_d<__bf16>(__bf16 v) { return (double)(float)v; }
template <typename T> __device__ __forceinline__ T from_d(double v) { return (T)v; }
template <> __device__ __forceinline__ __bf16 from_d<__bf16>(double v) { return (__bf16)(float)v; }

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// A K chunk is 128 bytes deep (KB = 16, 32 or 64 elements) and is staged
// through LDS in the layout of its source, 16 bytes at a time:
// - an operand contiguous in k as rows of 128 bytes, [row][k], the 16-byte
//   pieces of a row permuted by (row / MB) % 8 so that the 16 rows an MFMA
//   reads at one k lie in distinct banks;
// - an operand contiguous along its rows (A) or columns (B) as [k][row].
// Lane group g = lane / 16 holds k = KL g .. KL g + KL - 1 of each half
// chunk (KL elements are 16 bytes) and MFMA t takes element t of every
// group; block i of a wave has rows MB m + i.  So every access to LDS and
// to global memory, the stores of C included, is as wide as the layout lets
// it be, and the k order of an element is the same for every tile shape:
// the shape never changes the bits.
template <typename TI, int TT, int MB> struct Operand {
  static constexpr int E = 16 / (int)sizeof(TI);      // elements per piece
  static constexpr int KL = E;
  static constexpr int KB = 128 / (int)sizeof(TI);
  static constexpr int NP = TT * 8 / 256;             // pieces per lane and chunk
  static constexpr int PR = TT / E;                   // pieces per k row of the [k][row] layout
  static constexpr bool HALF = sizeof(TI) == 2;

  // The lane's pieces of the chunk at k0, without a branch (the waits then
  // count loads and leave the later ones in flight).  Rows past `lim` repeat
  // earlier ones (their products are not stored) and k past K earlier k,
  // which clear() zeroes when the chunk is staged.  WIDE: one 16-byte load a
  // piece, for sizes that pieces divide, and of 16-bit elements for all of a piece
  // at least (wide_ok): the piece that such a size ends in is loaded up to that
  // end, and clear() or align() moves its elements to their places.  Otherwise by
  // elements.  (Eight loads a piece are too many: 64 products of 100 x 200 x 400 in
  // bf16 30 us by elements, 12 so.  Two or four are not: 8-byte elements lose up to
  // 10% of a small launch to the moves.)
  template <bool KC> static __device__ __forceinline__ bool wide_ok(int lim, int K) {
    const int n = KC ? K : lim;
    return HALF ? n >= E : n % E == 0;
  }
  // the elements of r from the `sh`-th on, zeros behind them (sh >= E: zeros)
  static __device__ __forceinline__ u4 from_element(u4 r, int sh) {
    unsigned __int128 v = __builtin_bit_cast(unsigned __int128, r);
    v = sh < E ? v >> (8 * (int)sizeof(TI) * sh) : (unsigned __int128)0;
    return __builtin_bit_cast(u4, v);
  }
  // [k][row], WIDE: whether the rows of the tile end within a piece, and its place
  static __device__ __forceinline__ bool ragged(int row0, int lim) {
    return HALF && row0 + TT > lim && lim % E != 0;
  }
  static __device__ __forceinline__ void align(u4 (&r)[NP], int row0, int lim) {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));   // formed in the branch, not ahead of the stream
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int sh = row0 + ((t + 256 * q) % PR) * E + E - lim;
      if (sh > 0) r[q] = from_element(r[q], sh);
    }
  }
  template <bool KC, bool WIDE>
  static __device__ __forceinline__ void fetch(u4 (&r)[NP], uint64_t b, int64_t ld, int row0,
                                               int lim, int k0, int K) {
    typedef TI V __attribute__((ext_vector_type(E), aligned(sizeof(TI))));
    const TI TNX_GLOBAL* base = as_global<const TI>(b);
    if constexpr (!WIDE && HALF && TT == 64) {
      // an operand of less than a piece: pieces that reach into its next rows, the
      // last ones up to the operand's end and then moved; what is not its own k is
      // zero, other rows' elements belong to outputs that are not stored (in the
      // 32x32 shape the loads by elements are the faster ones)
      const int n = KC ? K : lim, rows = KC ? lim : K;
      const int64_t span = (rows - 1) * ld + n;
      if (span >= E) {
        int at[NP], sh[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const int c = threadIdx.x + 256 * q;
          const int row = row0 + (KC ? c >> 3 : (c % PR) * E);
          const int k = k0 + (KC ? (c & 7) * E : c / PR);
          at[q] = KC ? k : row;
          const int64_t want = min(KC ? row : k, rows - 1) * ld + (at[q] < n ? at[q] : 0);
          const int64_t off = min(want, span - E);
          sh[q] = (int)(want - off);
          r[q] = __builtin_bit_cast(u4, *(const V TNX_GLOBAL*)(base + off));
        }
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          r[q] = from_element(r[q], sh[q]);
          if constexpr (KC) {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              const uint32_t lo = at[q] + 2 * x < n ? 0xffffu : 0u, hi = at[q] + 2 * x + 1 < n ? 0xffff0000u : 0u;
              r[q][x] &= lo | hi;
            }
          }
        }
        return;
      }
    }
    if constexpr (!WIDE && HALF && TT == 64) {
      // a matrix of less than a piece: by elements in a loop, as all eight loads
      // cost every launch of the kernel 3%, in registers and code
#pragma unroll
      for (int q = 0; q < NP; ++q) r[q] = u4{0, 0, 0, 0};
#pragma unroll 2
      for (int x = 0; x < E; ++x) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const int c = threadIdx.x + 256 * q;
          const int row = row0 + (KC ? c >> 3 : (c % PR) * E + x);
          const int k = k0 + (KC ? (c & 7) * E + x : c / PR);
          const int64_t off = KC ? min(row, lim - 1) * ld + min(k, K - 1)
                                 : min(k, K - 1) * ld + min(row, lim - 1);
          const uint32_t e = __builtin_bit_cast(uint16_t, (TI)base[off]);
          // the elements so far move down, this one comes last
          r[q] = u4{r[q][0] >> 16 | r[q][1] << 16, r[q][1] >> 16 | r[q][2] << 16,
                    r[q][2] >> 16 | r[q][3] << 16, r[q][3] >> 16 | e << 16};
        }
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int c = threadIdx.x + 256 * q;
      const int row = row0 + (KC ? c >> 3 : (c % PR) * E);
      const int k = k0 + (KC ? (c & 7) * E : c / PR);
      if constexpr (WIDE) {
        const int64_t off = KC ? min(row, lim - 1) * ld + min(k, K - E)
                               : min(k, K - 1) * ld + min(row, lim - E);
        r[q] = __builtin_bit_cast(u4, *(const V TNX_GLOBAL*)(base + off));
      } else {
        TI e[E];
#pragma unroll
        for (int x = 0; x < E; ++x)
          e[x] = KC ? base[min(row, lim - 1) * ld + min(k + x, K - 1)]
                    : base[min(k, K - 1) * ld + min(row + x, lim - 1)];
        __builtin_memcpy(&r[q], e, 16);
        // piece by piece: the addresses of all of them would cost occupancy
        if constexpr (HALF) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  static __device__ __forceinline__ int swz(int row) { return (row / MB) & 7; }

  template <bool KC> static __device__ __forceinline__ void commit(const u4 (&r)[NP], u4* lds) {
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int c = t + 256 * q;
      lds[KC ? (c & ~7) | ((c & 7) ^ swz(c >> 3)) : c] = r[q];
    }
  }

  // zero the pieces' elements from k index `valid` of the chunk on
  template <bool KC, bool WIDE> static __device__ __forceinline__ void clear(u4 (&r)[NP], int valid) {
    int t = threadIdx.x;
    if constexpr (HALF) asm volatile("" : "+v"(t));
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int c = t + 256 * q;
      if constexpr (KC && WIDE && HALF) {
        const int sh = (c & 7) * E + E - valid;
        if (sh > 0) r[q] = from_element(r[q], sh);
        continue;
      }
      TI e[E];
      __builtin_memcpy(e, &r[q], 16);
#pragma unroll
      for (int x = 0; x < E; ++x)
        if ((KC ? (c & 7) * E + x : c / PR) >= valid) e[x] = (TI)0.0f;
      __builtin_memcpy(&r[q], e, 16);
    }
  }

  static __device__ __forceinline__ void scale(u4 (&r)[NP], double alpha) {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      TI e[E];
      __builtin_memcpy(e, &r[q], 16);
#pragma unroll
      for (int x = 0; x < E; ++x) {
        if constexpr (HALF) e[x] = (TI)((float)alpha * (float)e[x]);
        else e[x] = (TI)(alpha * (double)e[x]);
      }
      __builtin_memcpy(&r[q], e, 16);
    }
  }

  // Half chunk h of the wave's rows from `row` (within the tile).  SEQ (f64):
  // MFMA t takes k = 4 t + g of the half chunk from lane group g, so that the
  // sum over k runs in the order of the index (8-byte instead of 16-byte LDS
  // reads: GEMM 2 of an order-64 problem and its like 10.1 instead of 9.5 us).
  template <bool KC, bool SEQ> struct Raw {
    static_assert(!SEQ || sizeof(TI) == 8, "in-order sums are f64");
    // [k][row]: KL loads of MB elements (16-bit ones as whole words)
    static constexpr int W = KC ? 4 : (MB * (int)sizeof(TI) + 3) / 4;
    uint32_t w[KC ? MB : KL][W];

    __device__ __forceinline__ void read(const u4* lds, int row, int h) {
      const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
      if constexpr (KC) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const int rr = row + MB * m + i;
          if constexpr (SEQ) {
#pragma unroll
            for (int t = 0; t < KL; ++t) {
              const u4* p = lds + rr * 8 + ((4 * h + 2 * t + (g >> 1)) ^ swz(rr));
              const double v = ((const double*)p)[g & 1];
              __builtin_memcpy(&w[i][2 * t], &v, 8);
            }
          } else {
            const u4 v = lds[rr * 8 + ((4 * h + g) ^ swz(rr))];
#pragma unroll
            for (int x = 0; x < 4; ++x) w[i][x] = v[x];
          }
        }
      } else {
        const char* p = (const char*)lds +
                        ((h * (KB / 2) + (SEQ ? 1 : KL) * g) * TT + row + MB * m) * (int)sizeof(TI);
#pragma unroll
        for (int s = 0; s < KL; ++s) {
          const char* q = p + s * (SEQ ? 4 : 1) * TT * (int)sizeof(TI);
          if constexpr (MB * sizeof(TI) == 2) w[s][0] = *(const uint16_t*)q;
          else {
            typedef uint32_t V __attribute__((ext_vector_type(W)));
            const V v = *(const V*)q;
#pragma unroll
            for (int x = 0; x < W; ++x) w[s][x] = v[x];
          }
        }
      }
    }
    // element s of block i (f64, f32)
    __device__ __forceinline__ TI get(int i, int s) const {
      TI v;
      constexpr int WE = sizeof(TI) >= 4 ? (int)sizeof(TI) / 4 : 1;
      __builtin_memcpy(&v, KC ? &w[KC ? i : 0][WE * s] : &w[KC ? 0 : s][KC ? 0 : WE * i], sizeof(TI));
      return v;
    }
    // the 8 k of block i (bf16)
    __device__ __forceinline__ tnx_bf8 get8(int i) const {
      uint32_t x[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (KC) x[t] = w[i][t];
        else x[t] = __builtin_amdgcn_perm(w[2 * t + 1][i / 2], w[2 * t][i / 2],
                                          (i & 1) ? 0x07060302u : 0x05040100u);
      }
      tnx_bf8 v;
      __builtin_memcpy(&v, x, 16);
      return v;
    }
  };
};

// acc += the staged chunk's A B, the wave's rows from wr and columns from wc
template <int MODE, bool SEQ, int TT, int MB, bool KA, bool KBc>
__device__ __forceinline__ void mma_chunk(typename Tr<MODE>::V4 (&acc)[MB][MB], const u4* As,
                                          const u4* Bs, int wr, int wc) {
  typedef typename Tr<MODE>::TI TI;
  typedef Operand<TI, TT, MB> O;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    typename O::template Raw<KA, SEQ> a;
    typename O::template Raw<KBc, SEQ> b;
    a.read(As, wr, h);
    b.read(Bs, wc, h);
    if constexpr (O::HALF) {
      tnx_bf8 av[MB], bv[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) av[i] = a.get8(i);
#pragma unroll
      for (int i = 0; i < MB; ++i) bv[i] = b.get8(i);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
    } else {
#pragma unroll
      for (int t = 0; t < O::KL; ++t)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < MB; ++j) {
            if constexpr (MODE == TNX_GEMM_F64)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.get(i, t), b.get(j, t), acc[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.get(i, t), b.get(j, t), acc[i][j], 0, 0, 0);
          }
    }
  }
}

// The problem that owns 64x64 tile `bid`: problems of a launch are mostly of
// one size, so the record at its share of the range is tried first (one
// round of loads, scalar ones, as the whole record is then mostly in the
// cache), then the search.
__device__ __forceinline__ int find_problem(const tnx_gemm_problem* __restrict__ probs, int nprob,
                                            int bid, int ntiles) {
  const tnx_gemm_problem TNX_CONST* P = (const tnx_gemm_problem TNX_CONST*)(uint64_t)probs;
  const int guess = __builtin_amdgcn_readfirstlane((int)((int64_t)bid * nprob / ntiles));
  const int lo = P[guess].tile_begin;
  const int hi = guess + 1 < nprob ? P[min(guess + 1, nprob - 1)].tile_begin : ntiles;
  if (bid >= lo && bid < hi) return guess;
  return tnx_find_owner(probs, sizeof(tnx_gemm_problem), offsetof(tnx_gemm_problem, tile_begin),
                        nprob, bid);
}

// Barrier of the LDS stages: LDS accesses only are ordered (the loads from
// global memory of the chunks ahead stay in flight across it).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// whether a segment's operands can be fetched by 16-byte pieces
template <typename O, bool KA, bool KBc>
__device__ __forceinline__ bool wide(int M, int N, int K) {
  return O::template wide_ok<KA>(M, K) && O::template wide_ok<KBc>(N, K);
}

// acc += the products of the segments [s, ...) with the same layouts as
// segment s (KA: A contiguous in k, KBc: B) and the same WIDE; returns the
// first segment after them.  Their chunks form one stream: PD chunks are in flight in registers
// ahead of the staged one, across the segments; past the last chunk it is
// fetched again, unused (no branch around the loads, so that the waits count
// them and never drain them).
template <int MODE, bool SEQ, int TT, int PD, bool KA, bool KBc, bool WIDE>
__device__ __forceinline__ int run_stream(typename Tr<MODE>::V4 (&acc)[TT / 32][TT / 32],
                                          const tnx_gemm_seg TNX_CONST* segs, int s, int s_end,
                                          int M, int N, int row0, int col0, int wr, int wc,
                                          u4 (*As)[TT * 8], u4 (*Bs)[TT * 8]) {
  constexpr int MB = TT / 32;
  typedef Operand<typename Tr<MODE>::TI, TT, MB> O;
  u4 ra[PD][O::NP], rb[PD][O::NP];
  double al[PD];
  // k of the chunk that exist; where the tile ends within a piece, so much less
  // that every chunk of it takes the branch of the ends below
  int kv[PD];
  const bool edge_a = WIDE && !KA && O::ragged(row0, M), edge_b = WIDE && !KBc && O::ragged(col0, N);
  const int less = edge_a || edge_b ? 1 << 30 : 0;
  // the stream's extent: its segments and chunks
  int chunks = 0, end = s;
  for (; end < s_end; ++end) {
    const int K = segs[end].K;
    if (K <= 0) continue;
    if ((segs[end].transA == 0) != KA || (segs[end].transB != 0) != KBc ||
        wide<O, KA, KBc>(M, N, K) != WIDE)
      break;
    chunks += (K + O::KB - 1) / O::KB;
  }
  uint64_t A = segs[s].a, B = segs[s].b;
  int lda = segs[s].lda, ldb = segs[s].ldb, K = segs[s].K, k0 = 0;
  double alpha = segs[s].alpha;
  auto fetch = [&](int d) {
    O::template fetch<KA, WIDE>(ra[d], A, lda, row0, M, k0, K);
    O::template fetch<KBc, WIDE>(rb[d], B, ldb, col0, N, k0, K);
    al[d] = alpha;
    kv[d] = K - k0 - less;
    if (k0 + O::KB < K) {
      k0 += O::KB;
    } else {
      int n = s + 1;
      while (n < end && segs[n].K <= 0) ++n;
      if (n < end) {
        s = n;
        A = segs[n].a;
        B = segs[n].b;
        lda = segs[n].lda;
        ldb = segs[n].ldb;
        K = segs[n].K;
        alpha = segs[n].alpha;
        k0 = 0;
      }
    }
  };
  auto commit = [&](int d, int stage) {
    if (kv[d] < O::KB) {
      asm volatile("");   // a branch, not selects on every chunk
      const int valid = kv[d] + less;
      if (edge_a) O::align(ra[d], row0, M);
      if (edge_b) O::align(rb[d], col0, N);
      O::template clear<KA, WIDE>(ra[d], valid);
      O::template clear<KBc, WIDE>(rb[d], valid);
    }
    if (__double_as_longlong(al[d]) != 0x3FF0000000000000ll) {
      asm volatile("");
      O::scale(ra[d], al[d]);
    }
    O::template commit<KA>(ra[d], As[stage]);
    O::template commit<KBc>(rb[d], Bs[stage]);
  };
#pragma unroll
  for (int d = 0; d < PD; ++d) fetch(d);
  commit(0, 0);
  fetch(0);
  lds_barrier();
  // each step: the MFMAs of the staged chunk, then the next one into the
  // other stage (read by all before the last barrier) and its registers
  // refilled
  auto step = [&](int u) {
    const int d = (u + 1) % PD, stage = u & 1;
    mma_chunk<MODE, SEQ, TT, MB, KA, KBc>(acc, As[stage], Bs[stage], wr, wc);
    commit(d, stage ^ 1);
    fetch(d);
    lds_barrier();
  };
  for (int t = chunks / (2 * PD); t > 0; --t) {
#pragma unroll
    for (int u = 0; u < 2 * PD; ++u) step(u);
  }
  const int rest = chunks % (2 * PD);
#pragma unroll
  for (int u = 0; u < 2 * PD - 1; ++u)
    if (u < rest) step(u);
  return end;
}

// Workgroup of 4 wavefronts (2 x 2) over a TT x TT part of the problem: a
// quarter of a 64x64 tile (TT = 32) or one tile (64).  Two LDS stages (16 or
// 32 KB), W waves per SIMD at least.
// Bound: the f64 and f32 MFMA rate where the chip is full (28 problems of
// 1024 x 2048 x 1024: f64 64 of the 73 TFLOP/s a library product reaches,
// f32 117 of 153; 53 and 92 with scalar LDS accesses, flat loads and the
// loads drained at every barrier), latency for the K of 64 to 512 and the few
// tiles of a chain's step: there a workgroup lives for a handful of chunks
// and descriptor, first loads and barriers are most of it (64 products of
// 256 x 128 x 512 f64 64 -> 45 us; 16 of 128 x 64 x 256 21 -> 8.4 us; bf16 15
// -> 11 us).  PD: three (32) f64 chunks in flight hide a cold load behind
// MFMAs of 256 cycles; one is enough behind the 1024 of the 64x64 shape.
// Tried and not kept: operands straight from global memory to the MFMA
// registers (an operand contiguous in k then touches 16 lines per load: f64
// 58 of 73 and 42 where both are), 128 x 128 workgroups (f64 32, f32 63).
template <int MODE, bool SEQ, int TT, int PD, int W>
__global__ __launch_bounds__(256, W) void gemm_grouped_kernel(const tnx_gemm_problem* __restrict__ probs,
                                                           int nprob,
                                                           const tnx_gemm_seg* __restrict__ segs,
                                                           int ntiles,
                                                           const int32_t* __restrict__ active,
                                                           unsigned long long* ts) {
  tnx_stamp_begin(ts);
  constexpr int MB = TT / 32, NB = MB;
  typedef Tr<MODE> T;
  typedef typename T::TC TC;
  typedef typename T::V4 V4;
  __shared__ u4 As[2][TT * 8], Bs[2][TT * 8];
  int bid = tnx_xcd_remap(blockIdx.x, gridDim.x), sub = 0;
  if constexpr (TT == 32) {
    sub = bid & 3;
    bid >>= 2;
  }
  const int pi = __builtin_amdgcn_readfirstlane(find_problem(probs, nprob, bid, ntiles));
  const tnx_gemm_problem TNX_CONST* cp = (const tnx_gemm_problem TNX_CONST*)(uint64_t)probs + pi;
  const tnx_gemm_seg TNX_CONST* cs = (const tnx_gemm_seg TNX_CONST*)(uint64_t)segs;
  const tnx_gemm_problem TNX_CONST& P = *cp;
  // (flags change between launches only: a scalar load, waited for with the
  // records)
  const int on = P.active >= 0 && active != nullptr
                     ? ((const int32_t TNX_CONST*)(uint64_t)active)[P.active] : 1;
  if (on == 0) return;
  const int tiles_n = (P.N + 63) / 64;
  const int t_local = bid - P.tile_begin;
  const int tr = t_local / tiles_n, tc = t_local - tr * tiles_n;
  const int row0 = tr * 64 + (TT == 32 ? 32 * (sub >> 1) : 0);
  const int col0 = tc * 64 + (TT == 32 ? 32 * (sub & 1) : 0);
  if (row0 >= P.M || col0 >= P.N) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = (wave >> 1) * 16 * MB, wc = (wave & 1) * 16 * NB;
  // C: lane % 16 is the column index of a block; the row index of
  // accumulator element r is 4 (lane / 16) + r for the f32-output MFMAs
  // and lane / 16 + 4 r for v_mfma_f64_16x16x4_f64 (measured on gfx950)
  TC TNX_GLOBAL* Cp = as_global<TC>(P.c);
  const TC TNX_GLOBAL* C0 = as_global<const TC>(P.c0);
  const int gj = col0 + wc + NB * (lane & 15);
  const bool full = gj + NB <= P.N;   // the lane's columns all exist
  typedef TC VC __attribute__((ext_vector_type(NB), aligned(sizeof(TC))));
  auto row_of = [&](int i, int r) {
    const int rr = (MODE == TNX_GEMM_F64) ? ((lane >> 4) + 4 * r) : ((lane >> 4) * 4 + r);
    return row0 + wr + MB * rr + i;
  };
  // All of C0 before the first store (no load can pass a store it might
  // alias; elements past the edges: of the last row or column), and before the
  // products where the registers allow it.
  TC c0[MB][4][NB];
  auto load_c0 = [&]() {
    if (C0 == nullptr) return;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const TC TNX_GLOBAL* row = C0 + (int64_t)min(row_of(i, r), P.M - 1) * P.ldc0;
        if (full) {
          if constexpr (NB == 1) c0[i][r][0] = row[gj];
          else {
            const VC c = *(const VC TNX_GLOBAL*)(row + gj);
#pragma unroll
            for (int j = 0; j < NB; ++j) c0[i][r][j] = c[j];
          }
        } else {
#pragma unroll
          for (int j = 0; j < NB; ++j) c0[i][r][j] = row[min(gj + j, P.N - 1)];
        }
      }
  };
  if constexpr (MB == 1) load_c0();
  V4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = V4{0, 0, 0, 0};

  int s = P.seg_begin;
  const int s_end = s + P.seg_count;
  while (s < s_end) {
    if (cs[s].K <= 0) {
      ++s;
      continue;
    }
    const bool ta = cs[s].transA != 0, tb = cs[s].transB != 0;
    const int K = cs[s].K;
    typedef Operand<typename T::TI, TT, MB> O;
#define TNX_STREAM(KA, KBc)                                                                 \
  s = wide<O, KA, KBc>(P.M, P.N, K)                                                         \
          ? run_stream<MODE, SEQ, TT, PD, KA, KBc, true>(acc, cs, s, s_end, P.M, P.N, row0, col0, wr, \
                                                    wc, As, Bs)                             \
          : run_stream<MODE, SEQ, TT, O::HALF ? 1 : PD, KA, KBc, false>(acc, cs, s, s_end, P.M, P.N, row0, col0, wr, \
                                                     wc, As, Bs)
    if (!ta && tb) TNX_STREAM(true, true);
    else if (!ta) TNX_STREAM(true, false);
    else if (tb) TNX_STREAM(false, true);
    else TNX_STREAM(false, false);
#undef TNX_STREAM
  }

  if constexpr (MB > 1) load_c0();
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gi = row_of(i, r);
      if (gi >= P.M) continue;
      TC v[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        double x = (double)acc[i][j][r];
        if (C0 != nullptr) x += P.beta * to_d(c0[i][r][j]);
        v[j] = from_d<TC>(x);
      }
      TC TNX_GLOBAL* row = Cp + (int64_t)gi * P.ldc;
      if (full) {
        if constexpr (NB == 1) row[gj] = v[0];
        else {
          VC c;
#pragma unroll
          for (int j = 0; j < NB; ++j) c[j] = v[j];
          *(VC TNX_GLOBAL*)(row + gj) = c;
        }
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (gj + j < P.N) row[gj + j] = v[j];
      }
    }
  if (ts != nullptr) {
    __syncthreads();
    tnx_stamp_end(ts);
  }
}

}  // namespace

// Both shapes give the same bits; which is faster depends on whether the 64x64
// tiles fill the 256 CUs: a tile's MFMAs take their time on the one CU that
// holds it, so below one tile per CU the 32x32 shape spreads a tile over four,
// above it the larger shape reads its operands half as often (f64, us, 32x32
// against 64x64: 128 tiles of K = 512 18 / 27, 256 tiles 28 / 29, 512 tiles
// 52 / 46, 2048 tiles of K = 128 67 / 51; f32 11 / 16, 17 / 17, 33 / 28, 48 /
// 32).  The bf16 MFMAs are fast enough for the line to lie at half that (128
// tiles of K = 512 7.4 / 7.8 and of K = 3584 21 / 26, 192 tiles 8.6 / 8.0,
// 256 tiles 12.5 / 8.3).
static int gemm_small_tiles(int mode) { return mode <= TNX_GEMM_F32 ? 256 : 128; }

template <int MODE, bool SEQ, int TT, int PD, int W>
static void launch_gemm(const tnx_gemm_problem* prob, int nprob, const tnx_gemm_seg* seg, int ntiles,
                        const int32_t* active, hipStream_t s, unsigned long long* ts) {
  hipLaunchKernelGGL((gemm_grouped_kernel<MODE, SEQ, TT, PD, W>), dim3(TT == 32 ? 4 * ntiles : ntiles),
                     dim3(256), 0, s, prob, nprob, seg, ntiles, active, ts);
}

extern "C" int tnx_gemm_variants(int mode) {
  switch (mode) {
    case TNX_GEMM_F64:
    case TNX_GEMM_F32:
    case TNX_GEMM_BF16_F32:
    case TNX_GEMM_BF16_BF16: return 2;
    default:
      tnx_set_error("tnx_gemm_variants: unknown mode %d", mode);
      return TNX_EINVAL;
  }
}

extern "C" int tnx_gemm_grouped(int mode, const tnx_gemm_problem* prob, int nprob,
                                const tnx_gemm_seg* seg, int ntiles, const int32_t* active,
                                tnx_stream_t stream) {
  return tnx_gemm_grouped_ts(mode, prob, nprob, seg, ntiles, active, stream, nullptr);
}

int tnx_gemm_grouped_ts(int mode, const tnx_gemm_problem* prob, int nprob,
                        const tnx_gemm_seg* seg, int ntiles, const int32_t* active,
                        tnx_stream_t stream, unsigned long long* ts) {
  if (nprob == 0 && ntiles == 0) return TNX_OK;
  if (nprob < 0 || ntiles < 0 || prob == nullptr || seg == nullptr) {
    tnx_set_error("tnx_gemm_grouped: bad arguments (nprob=%d ntiles=%d)", nprob, ntiles);
    return TNX_EINVAL;
  }
  const int base = mode & 0xFF, var = (mode >> 8) & 0xFF;
  const int nvar = tnx_gemm_variants(base);
  const bool in_order = (mode & TNX_GEMM_IN_ORDER) != 0;
  if (nvar < 0 || (mode & ~(TNX_GEMM_IN_ORDER | 0xFFFF)) != 0 || var >= nvar ||
      (in_order && base != TNX_GEMM_F64)) {
    tnx_set_error("tnx_gemm_grouped: unknown mode %d (variant %d)", base, var);
    return TNX_EINVAL;
  }
  if (ntiles == 0) return TNX_OK;
  hipStream_t s = (hipStream_t)stream;
  // variant 0 takes the shape of the rule, variant 1 the other one; the 32x32
  // grid has four workgroups a tile, which a launch's x extent must hold
  const bool small = ((ntiles <= gemm_small_tiles(base)) != (var == 1)) && ntiles < (1 << 29);
#define TNX_GEMM_LAUNCH(MODE, SEQ, PDS, WS, PDL, WL)                                          \
  if (small) launch_gemm<MODE, SEQ, 32, PDS, WS>(prob, nprob, seg, ntiles, active, s, ts);     \
  else launch_gemm<MODE, SEQ, 64, PDL, WL>(prob, nprob, seg, ntiles, active, s, ts)
  switch (base) {
    case TNX_GEMM_F64:
      if (in_order) {
        TNX_GEMM_LAUNCH(TNX_GEMM_F64, true, 3, 4, 1, 3);
      } else {
        TNX_GEMM_LAUNCH(TNX_GEMM_F64, false, 3, 4, 1, 3);
      }
      break;
    case TNX_GEMM_F32: TNX_GEMM_LAUNCH(TNX_GEMM_F32, false, 3, 4, 1, 3); break;
    case TNX_GEMM_BF16_F32: TNX_GEMM_LAUNCH(TNX_GEMM_BF16_F32, false, 4, 3, 1, 2); break;
    default: TNX_GEMM_LAUNCH(TNX_GEMM_BF16_BF16, false, 4, 3, 1, 2); break;
  }
#undef TNX_GEMM_LAUNCH
  TNX_CHECK_LAUNCH();
  return TNX_OK;
}
