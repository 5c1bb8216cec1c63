// Dense semiring batched matmul: the arg-max backward kernels (gfx950).
#include <type_traits>

#include "common.h"

namespace GENBMM_NS {
namespace {

// ===================================================== argmax backward
//
// maxbmm / samplebmm:  grad_a[m,k] = sum_n [k == idx[m,n]] g[m,n]
//                      grad_b[k,n] = sum_m [k == idx[m,n]] g[m,n]
// prodmaxbmm: the terms are b[k,n]*g[m,n] and a[m,k]*g[m,n].
// (reference matmul_cuda_kernel.cu:336-456: one thread per gradient cell
// scanning the whole reduction axis, O(M*K*N).)  Here a lane owns a row m (resp.
// column n) and a range of k, walks the row once in ascending n (resp. the column
// in ascending m) and adds each term whose idx falls into its range to that
// cell of an LDS-resident accumulator; the additions hitting a given cell
// therefore happen in the reference's order, so the result is bit-identical, in
// O(M*N) work.  Products are rounded before the add (the build uses
// -ffp-contract=on: no fusion across statements).
constexpr int kKC = 128;  // cells of the reduction axis per lane, at most (KC: those of an instantiation)

// The 64 lanes of a workgroup are (line, part): 64 >> ps lines (rows m of grad_a,
// columns n of grad_b) times 2^ps parts of kKC consecutive k, so that one workgroup
// covers every k of its lines (up to 64 * kKC; longer K: further workgroups) and idx
// and g are read from memory once - the lanes of a line read the same addresses.
// Each lane walks its whole line and adds the terms whose k falls into its part.
//
// A lane's cells are its own and lie at [k][lane]: whatever k each lane adds to, the 64 lanes
// stay in 64 different banks, and nothing is exchanged between lanes (no barrier).  33 KB per
// wave leave four waves on a compute unit, one per SIMD, so nothing but a lane's own loads
// hides the latency of memory: the walk is double-buffered in registers, the next chunk of the
// line is in flight while one is added.  Bound by the chains of ordered additions, one LDS round
// trip per four cells.  Measured (both gradients, max product; before: loads waited for 16 cells at a
// time, cells of a row side by side so that the lanes' additions met in banks, rows of unaligned
// length one cell at a time): (256, 256^3) 104 -> 87 us, (64, 512^3) 141 -> 123, (8192, 32^3) 79 -> 54,
// (40, 251, 173, 301) 111 -> 37.  A row's partial last chunk too is read in pieces of four, the last one cell by
// cell (all 32 cell by cell cost forward and backward of float16 draws at (64, 20^3) 32.7 -> 33.5 us, now 32.3;
// prodmaxbmm (814, 76, 51, 83) 165 -> 153; clamped addresses in the place of the uniform tests: 5 % slower).
// One wave on a SIMD issues everything itself, so instructions count: a slot by one unsigned minimum and a column's
// addresses carried along (two chunks of a column 687 -> 482 instructions, of a row 950 -> 760): max and
// sample, again and again on one set of buffers, which the Infinity Cache holds in part, and (in brackets) on other
// buffers each time, as behind a forward: (256, 256^3) 74 -> 65 us (85 -> 78), (64, 512^3) 124 -> 99 (133 -> 111),
// (40, 251, 173, 301) 21.6 -> 17.9 (22.5 -> 20.7), (100, 500, 300, 510) 198 -> 160 (200 -> 163), (512, 128^3) 34
// (43) either way (memory).  With the product semiring's factors the same took more registers
// than a wave's 256 ((512, 128^3) 47 -> 51, (64, 512^3) 158 -> 139): it keeps the longer form.
//
// A K of 96, 64 or 32 and less takes as many cells per lane: what bounds the waves of a compute unit is their LDS,
// and six, nine or nineteen waves hide each other's chains (chunks are shorter then, for the registers).  On other
// buffers each time, max and (in brackets) product semiring, from 128 cells: (5753, 54^3) 95 -> 85 us (138 -> 132),
// (2048, 48^3) 33.5 -> 23.6 (39.6 -> 33.6), (814, 76, 51, 83) 45 -> 34 (68 -> 64), (1000, 90^3) 58 -> 52 (100 -> 88),
// (8192, 32^3) 60 -> 49 (75 -> 72).
static_assert(kKC == 128, "the shifts of the write-out");
constexpr int kChB = 16;  // cells of a column per chunk (single loads, and at most 63 loads can be in flight)
template <int KC>
constexpr int kArgAcc = 64 * KC + 64;  // floats of LDS: the cells, one spare cell per lane
template <int KC>
constexpr int kChA = KC == kKC ? 32 : 16;  // cells of a row per chunk

// Chunks of a line as they come from memory - indices, gradients and for PROD == 2 the other factor;
// nothing is converted before it is added, which would wait for the load - of a row (pieces of four
// cells, any alignment) and of a column (single cells).
typedef int argmax_i4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float argmax_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef elem_t argmax_e4 __attribute__((ext_vector_type(4), aligned(sizeof(elem_t))));
// (typed as global memory: a pointer carried around the loop was taken for one of unknown address space, whose
// loads are flat and drain all others)
template <class E>
using argmax_global = const __attribute__((address_space(1))) E*;
template <int PROD, int KC>
struct ArgRow {
  static constexpr int CH = kChA<KC>;
  argmax_i4 i4[CH / 4];
  argmax_e4 g4[CH / 4];
  argmax_f4 f4[PROD == 2 ? CH / 4 : 1];
  __device__ __forceinline__ int iv(int q) const { return i4[q >> 2][q & 3]; }
  __device__ __forceinline__ float gv(int q) const { return (float)g4[q >> 2][q & 3]; }
  __device__ __forceinline__ float fv(int q) const { return f4[q >> 2][q & 3]; }
};
template <int PROD>
struct ArgCol {
  static constexpr int CH = kChB;
  int i[CH];
  elem_t g[CH];
  float f[PROD == 2 ? CH : 1];
  __device__ __forceinline__ int iv(int q) const { return i[q]; }
  __device__ __forceinline__ float gv(int q) const { return (float)g[q]; }
  __device__ __forceinline__ float fv(int q) const { return f[q]; }
};
// Compiler-level ordering point for a wave's own LDS traffic (one wave's LDS instructions execute in order).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The lane's cells cleared; then the line's `cells` cells through load(chunk, number), tail(chunk, number)
// (the cells of a partial last chunk, index -1 behind them) and add(chunk, number).  No load stands
// under a branch in the loop - the last chunk is asked for again instead -: behind a branch the compiler
// can no longer tell which loads are younger than the chunk it waits for, and waits for all of them.
template <int KC, class Chunk, class Load, class Tail, class Add>
__device__ __forceinline__ void argmax_walk(float* __restrict__ accs, int cells, int kcap, Load load, Tail tail, Add add) {
  const int lane = threadIdx.x, full = cells / Chunk::CH;
  Chunk x, y;
  if (full > 0) load(x, 0);
#pragma unroll 16
  for (int kk = 0; kk < kcap; ++kk) accs[kk * 64 + lane] = 0.f;
  accs[KC * 64 + lane] = 0.f;
  int c = 0;
  for (; c + 1 < full; c += 2) {
    load(y, c + 1);
    add(x, c);
    load(x, min(c + 2, full - 1));
    add(y, c + 1);
  }
  if (c < full) add(x, c);
  if (full * Chunk::CH < cells) {
    tail(y, full);
    add(y, full);
  }
}
// The chunk's terms (g, times the other factor for the product semiring) in order.  other(cell, k):
// that factor read from its matrix (PROD == 1), only when the index falls into the lane's part.
template <int PROD, int KC, class Chunk, class Other>
__device__ __forceinline__ void argmax_add(float* __restrict__ accs, const Chunk& x, int c0, int kc, Other other) {
  constexpr int CH = Chunk::CH;
  const int lane = threadIdx.x;
  unsigned kr[CH];
  float tv[CH];
#pragma unroll
  for (int q = 0; q < CH; ++q) {
    if constexpr (PROD == 2) {
      const int k = x.iv(q) - c0;
      kr[q] = k >= 0 && k < kc ? k : KC;  // [KC]: the spare cells
      tv[q] = __fmul_rn(x.fv(q), x.gv(q));
    } else {
      // the lane's cell, or its spare one: an index below the part wraps around, one of K or beyond (none that the
      // library writes) may fall to a cell of the last part that is not written out.  Its factor does not exist.
      const unsigned k = min((unsigned)x.iv(q) - (unsigned)c0, (unsigned)KC);
      kr[q] = k;
      tv[q] = x.gv(q);
      if (PROD == 1 && (int)k < kc) tv[q] = __fmul_rn(other(q, x.iv(q)), tv[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < CH; q += 4) {
    const unsigned k4[4] = {kr[q], kr[q + 1], kr[q + 2], kr[q + 3]};
    const float t4[4] = {tv[q], tv[q + 1], tv[q + 2], tv[q + 3]};
    add4_ordered(accs + lane, k4, t4);
  }
}

// grad_a: line = row m, read in pieces of four cells (any alignment).
// (blk: the workgroup's number among those of grad_a; accs: kArgAcc<KC> floats of LDS)
template <int PROD, int KC>
__device__ __forceinline__ void argmax_bwd_a_block(float* __restrict__ accs, int blk,
                                                   const elem_t* __restrict__ bmat,
                                                   const float* __restrict__ fac,
                                                   const int32_t* __restrict__ idx,
                                                   const elem_t* __restrict__ g,
                                                   elem_t* __restrict__ grad_a, int M, int K,
                                                   int N, int row_tiles, int k_chunks, int ps) {
  const int lane = threadIdx.x, parts = 1 << ps, lines = 64 >> ps;
  const int part = lane & (parts - 1), line = lane >> ps;
  const int kc_id = blk % k_chunks, rt = blk / k_chunks;
  const int batch = rt / row_tiles;
  const int m = (rt - batch * row_tiles) * lines + line;
  const int c0 = kc_id * (parts * KC) + part * KC;  // first k of this lane
  const int kc = min(KC, K - c0);                    // <= 0: the part lies beyond K
  const long row = (long)batch * M + min(m, M - 1);   // lanes beyond the matrix walk the last row
  const int32_t* irow = idx + row * N;
  const elem_t* grow = g + row * N;
  const elem_t* bb = PROD == 1 ? bmat + (long)batch * K * N : nullptr;
  const float* frow = PROD == 2 ? fac + row * N : nullptr;
  const int kcap = min(KC, K);  // no lane has more cells
  using Chunk = ArgRow<PROD, KC>;
  auto load = [&](Chunk& x, int c) __attribute__((always_inline)) {
    const int n0 = c * Chunk::CH;
#pragma unroll
    for (int q = 0; q < Chunk::CH / 4; ++q) {
      x.i4[q] = *reinterpret_cast<const argmax_i4*>(irow + n0 + 4 * q);
      x.g4[q] = *reinterpret_cast<const argmax_e4*>(grow + n0 + 4 * q);
      if constexpr (PROD == 2) x.f4[q] = *reinterpret_cast<const argmax_f4*>(frow + n0 + 4 * q);
    }
  };
  auto tail = [&](Chunk& x, int c) __attribute__((always_inline)) {
    const int n0 = c * Chunk::CH;
#pragma unroll
    for (int q = 0; q < Chunk::CH / 4; ++q) {
      const int nq = n0 + 4 * q;
      if (nq + 4 <= N) {  // uniform
        x.i4[q] = *reinterpret_cast<const argmax_i4*>(irow + nq);
        x.g4[q] = *reinterpret_cast<const argmax_e4*>(grow + nq);
        if constexpr (PROD == 2) x.f4[q] = *reinterpret_cast<const argmax_f4*>(frow + nq);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool in = nq + j < N;
          x.i4[q][j] = in ? irow[nq + j] : -1;
          x.g4[q][j] = in ? grow[nq + j] : (elem_t)0.f;
          if constexpr (PROD == 2) x.f4[q][j] = in ? frow[nq + j] : 0.f;
        }
      }
    }
  };
  argmax_walk<KC, Chunk>(accs, N, kcap, load, tail, [&](const Chunk& x, int c) __attribute__((always_inline)) {
    argmax_add<PROD, KC>(accs, x, c0, kc, [&](int q, int k) { return (float)bb[(long)k * N + c * Chunk::CH + q]; });
  });
  // The cells change places, through registers, to [lane][KC + 1] - a row's parts one after the other -
  // so that the rows leave in runs (a lane storing its own cells, 16 bytes at a time and 512 apart, took
  // longer than the walk).
  wave_lds_sync();
  {
    float cell[KC];
#pragma unroll
    for (int k0 = 0; k0 < KC; k0 += 32)
      if (k0 < kcap) {  // uniform
#pragma unroll
        for (int kk = k0; kk < k0 + 32; ++kk) cell[kk] = accs[kk * 64 + lane];
      }
    wave_lds_sync();
#pragma unroll
    for (int k0 = 0; k0 < KC; k0 += 32)
      if (k0 < kcap) {
#pragma unroll
        for (int kk = k0; kk < k0 + 32; ++kk) accs[lane * (KC + 1) + kk] = cell[kk];
      }
  }
  wave_lds_sync();
  const int kw = parts * KC, w0 = kc_id * kw, kn = min(kw, K - w0);
  const int m0 = (rt - batch * row_tiles) * lines, rows = min(lines, M - m0);
  elem_t* dst = grad_a + ((long)batch * M + m0) * K + w0;
  auto cell_of = [&](int kk) { return KC < kKC ? accs + kk : accs + (kk >> 7) * (kKC + 1) + (kk & (kKC - 1)); };
  if (lines >= 8) {
    for (int kk = lane; kk < kn; kk += 64) {
      const float* src = cell_of(kk);
#pragma unroll 8
      for (int r = 0; r < rows; ++r) dst[(long)r * K + kk] = to_elem<elem_t>(src[r * parts * (KC + 1)]);
    }
  } else {
    // K beyond 1024, a few long rows: the loads of a row overlap, not those of a column of four rows or fewer
    // (maxbmm forward and backward (1, 16, 4096, 16) 92 -> 83.5 us, (1, 8, 8192, 8) 98 -> 86)
    for (int r = 0; r < rows; ++r) {
      const int off = r * parts * (KC + 1), whole = kn >> 6;
      elem_t* row = dst + (long)r * K;
#pragma unroll 8
      for (int i = 0; i < whole; ++i) row[64 * i + lane] = to_elem<elem_t>(cell_of(64 * i + lane)[off]);
      if (64 * whole + lane < kn) row[64 * whole + lane] = to_elem<elem_t>(cell_of(64 * whole + lane)[off]);
    }
  }
}

// grad_b: line = column n.
// (blk: the workgroup's number among those of grad_b; accs: kArgAcc<KC> floats of LDS)
template <int PROD, int KC>
__device__ __forceinline__ void argmax_bwd_b_block(float* __restrict__ accs, int blk,
                                                   const elem_t* __restrict__ amat,
                                                   const float* __restrict__ fac,
                                                   const int32_t* __restrict__ idx,
                                                   const elem_t* __restrict__ g,
                                                   elem_t* __restrict__ grad_b, int M, int K,
                                                   int N, int col_tiles, int k_chunks, int ps) {
  const int lane = threadIdx.x, parts = 1 << ps, lines = 64 >> ps;
  const int part = lane / lines, line = lane & (lines - 1);  // the lanes of a part: adjacent columns
  const int kc_id = blk % k_chunks, ct = blk / k_chunks;
  const int batch = ct / col_tiles;
  const int n = (ct - batch * col_tiles) * lines + line, nn = min(n, N - 1);
  const int c0 = kc_id * (parts * KC) + part * KC;
  const int kc = min(KC, K - c0);
  const int32_t* icol = idx + (long)batch * M * N + nn;
  const elem_t* gcol = g + (long)batch * M * N + nn;
  const elem_t* ab = PROD == 1 ? amat + (long)batch * M * K : nullptr;
  const float* fcol = PROD == 2 ? fac + (long)batch * M * N + nn : nullptr;
  const int kcap = min(KC, K);  // no lane has more cells
  using Chunk = ArgCol<PROD>;
  // HOLD: where a lane's cells of a chunk lie, one address each, a chunk on at a time.  Formed anew from the row's
  // number they take three scalar instructions a load, which a lone wave issues in the place of everything else.
  constexpr bool HOLD = PROD != 2;
  argmax_global<int32_t> ip[HOLD ? kChB : 1];
  argmax_global<elem_t> gp[HOLD ? kChB : 1];
  if constexpr (HOLD) {
#pragma unroll
    for (int q = 0; q < kChB; ++q) {
      ip[q] = (argmax_global<int32_t>)(icol + (long)q * N);
      gp[q] = (argmax_global<elem_t>)(gcol + (long)q * N);
    }
  }
  int reached = 0;  // the chunk they point at
  auto load = [&](Chunk& x, int c) __attribute__((always_inline)) {
    const int m0 = c * kChB;
    const long on = (long)((c - reached) * kChB) * N;  // none where the last chunk is asked for again
    reached = c;
#pragma unroll
    for (int q = 0; q < kChB; ++q) {
      if constexpr (HOLD) {
        x.i[q] = *(ip[q] += on);
        x.g[q] = *(gp[q] += on);
      } else {
        x.i[q] = icol[(long)(m0 + q) * N];
        x.g[q] = gcol[(long)(m0 + q) * N];
        x.f[q] = fcol[(long)(m0 + q) * N];
      }
    }
  };
  auto tail = [&](Chunk& x, int c) __attribute__((always_inline)) {
    const int m0 = c * kChB;
#pragma unroll
    for (int q = 0; q < kChB; ++q) {
      const bool in = m0 + q < M;
      x.i[q] = in ? icol[(long)(m0 + q) * N] : -1;
      x.g[q] = in ? gcol[(long)(m0 + q) * N] : (elem_t)0.f;
      if constexpr (PROD == 2) x.f[q] = in ? fcol[(long)(m0 + q) * N] : 0.f;
    }
  };
  argmax_walk<KC, Chunk>(accs, M, kcap, load, tail, [&](const Chunk& x, int c) __attribute__((always_inline)) {
    argmax_add<PROD, KC>(accs, x, c0, kc, [&](int q, int k) { return (float)ab[(long)(c * kChB + q) * K + k]; });
  });
  if (n < N)
#pragma unroll 16
    for (int kk = 0; kk < kc; ++kk)
      grad_b[((long)batch * K + c0 + kk) * N + n] = to_elem<elem_t>(accs[kk * 64 + lane]);
}

// Both gradients in one launch, batch item by batch item (ta workgroups of grad_a, then tb of
// grad_b, per item; XCD-aware numbering): both read the item's idx and g, which then come from
// memory once.
// KC: below kKC where K is no larger (one part per line).
template <int PROD, int KC>
__global__ __launch_bounds__(64, KC == 32 ? 3 : KC < kKC ? 2 : 1) void k_argmax_bwd_both(const elem_t* __restrict__ amat,
                                                       const elem_t* __restrict__ bmat,
                                                       const float* __restrict__ fac_a,
                                                       const float* __restrict__ fac_b,
                                                       const int32_t* __restrict__ idx,
                                                       const elem_t* __restrict__ g,
                                                       elem_t* __restrict__ grad_a,
                                                       elem_t* __restrict__ grad_b, int M, int K, int N,
                                                       int row_tiles, int kc_a, int ps_a,
                                                       int col_tiles, int kc_b, int ps_b) {
  __shared__ float accs[kArgAcc<KC>];
  const int ta = row_tiles * kc_a, tb = col_tiles * kc_b;
  const int v = xcd_renumber(blockIdx.x, gridDim.x);
  const int item = v / (ta + tb), r = v - item * (ta + tb);
  if (r < ta)
    argmax_bwd_a_block<PROD, KC>(accs, item * ta + r, bmat, fac_a, idx, g, grad_a, M, K, N, row_tiles, kc_a, ps_a);
  else
    argmax_bwd_b_block<PROD, KC>(accs, item * tb + r - ta, amat, fac_b, idx, g, grad_b, M, K, N, col_tiles, kc_b, ps_b);
}

// Parts per workgroup for a reduction axis of K cells: the smallest power of two that
// covers it (at most 64).
inline int argmax_parts_shift(int K) {
  int ps = 0;
  while (ps < 6 && (kKC << ps) < K) ++ps;
  return ps;
}

template <bool PROD>
int run_argmax_bwd(const elem_t* a, const elem_t* b, const int32_t* idx, const float* factors,
                   const elem_t* g, elem_t* grad_a, elem_t* grad_b, int B, int M, int K, int N,
                   void* stream) {
  if (int e = check_dense_dims(B, M, K, N)) return e;
  const int64_t mk = (int64_t)B * M * K, kn = (int64_t)B * K * N, mn = (int64_t)B * M * N;
  if (missing(idx, mn) || missing(g, mn) || missing(grad_a, mk) || missing(grad_b, kn) ||
      (PROD && !factors && (missing(a, mk) || missing(b, kn))))
    return GENBMM_E_NULLPTR;
  // factors = [a[m, idx] | b[idx, n]], each B*M*N: grad_a needs the second, grad_b the first
  constexpr int kGather = PROD ? 1 : 0;
  hipStream_t s = (hipStream_t)stream;
  if (mk == 0 && kn == 0) return GENBMM_OK;
  // (an empty M or N leaves one gradient without workgroups; the other is then all zeros)
  const int ps_a = argmax_parts_shift(K);
  const int row_tiles = ceil_div(M, 64 >> ps_a), kc_a = ceil_div(K, kKC << ps_a);
  // columns: two parts at most - narrower groups of columns cost more in the strided
  // reads of idx and g than reading them again saves
  const int ps_b = min(argmax_parts_shift(K), 1);
  const int col_tiles = ceil_div(N, 64 >> ps_b), kc_b = ceil_div(K, kKC << ps_b);
  const int64_t total = (int64_t)B * ((int64_t)row_tiles * kc_a + (int64_t)col_tiles * kc_b);
  if (total > 0x7fffffffLL) return GENBMM_E_SHAPE;
  auto go = [&](auto kern, const float* fa, const float* fb) {
    hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(64), 0, s, a, b, fa, fb, idx, g, grad_a, grad_b, M, K, N, row_tiles,
                       kc_a, ps_a, col_tiles, kc_b, ps_b);
  };
  auto pick = [&](auto kc) {
    constexpr int KC = decltype(kc)::value;
    if (PROD && factors) go(k_argmax_bwd_both<2, KC>, factors + mn, factors);
    else go(k_argmax_bwd_both<kGather, KC>, (const float*)nullptr, (const float*)nullptr);
  };
  if (K <= 32) pick(std::integral_constant<int, 32>{});
  else if (K <= 64) pick(std::integral_constant<int, 64>{});
  else if (K <= 96) pick(std::integral_constant<int, 96>{});
  else pick(std::integral_constant<int, kKC>{});
  if (int e = launch_status()) return e;
  return GENBMM_OK;
}

}  // namespace
}  // namespace GENBMM_NS

extern "C" {

// One set per element type: genbmm_argmax_bwd, genbmm_argmax_bwd_f16, ..._bf16, ...
int GENBMM_API(argmax_bwd)(const int32_t* idx, const GENBMM_NS::abi_t* g, GENBMM_NS::abi_t* grad_a,
                           GENBMM_NS::abi_t* grad_b, int B, int M, int K, int N, void* stream) {
  using namespace GENBMM_NS;
  return run_argmax_bwd<false>(nullptr, nullptr, idx, nullptr, el(g), el(grad_a), el(grad_b), B, M, K, N,
                               stream);
}

int GENBMM_API(prodmax_bwd)(const GENBMM_NS::abi_t* a, const GENBMM_NS::abi_t* b, const int32_t* idx,
                            const float* factors, const GENBMM_NS::abi_t* g, GENBMM_NS::abi_t* grad_a,
                            GENBMM_NS::abi_t* grad_b, int B, int M, int K, int N, void* stream) {
  using namespace GENBMM_NS;
  return run_argmax_bwd<true>(el(a), el(b), idx, factors, el(g), el(grad_a), el(grad_b), B, M, K, N,
                              stream);
}

}  // extern "C"
