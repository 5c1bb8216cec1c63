// logbmm second order (gfx950): gradients with respect to (a, b, g) of
// <u_a, grad_a> + <u_b, grad_b>, where (grad_a, grad_b) are the first-order gradients for the
// incoming gradient g.  Replaces _genbmm.backbackward (matmul_cuda.cpp:94-109,
// matmul_cuda_kernel.cu:547-622, kernels :220-331).
//
// With p = exp(a[m,k] + b[k,n] - out[m,n]), w = u_a[m,k] + u_b[k,n] (a missing u counts as 0):
//   t[m,n]      = sum_k p * w                        (gradient w.r.t. g)
//   grad_a[m,k] = sum_n g[m,n] * p * (w - t[m,n])
//   grad_b[k,n] = sum_m g[m,n] * p * (w - t[m,n])
// With u_b = 0 these are the reference's three quartic kernels (inner = sum_k2 (delta*s -
// s*s2)*u[k2] = s*(u[k] - t)) in O(M K N).
//
// Two implementations.
//  * Exact, on the vector ALU: three passes (t, grad_a, grad_b), one exponential per (m,k,n)
//    in each.  Any shape; the whole computation for small problems, and the recompute of
//    batch items that the factored form cannot take.
//  * Factored, on the matrix cores (needs the caller's workspace): with the row maxima
//    alpha of a and column maxima beta of b, EA = exp(a - alpha), EB = exp(b - beta),
//    R = exp(alpha + beta - out), H = g R, X = EA u_a, Y = EB u_b:
//      t      = R (X EB + EA Y)
//      grad_a = X (H EB^T) + EA (H Y^T - (H t) EB^T)
//      grad_b = Y (EA^T H) + EB (X^T H - EA^T (H t))
//    eight products (five when u_b is absent) of batched GEMM shape.  The operands are laid out
//    once, zero-padded to multiples of 128 in every extent: EA, X, EB, Y by an elementwise launch, H and
//    H t by the epilogue of t; one GEMM kernel (128 x 128 tiles, three-part operands on v_mfma_f32_32x32x16_bf16, 16-deep slabs
//    through two LDS buffers) then runs without any edge handling in its loop, sums up to two products into one
//    accumulator and applies the epilogue of its role.  A batch item with a cell whose
//    alpha + beta - out is beyond 40 ln 2 or not finite (a factor could underflow against a
//    term that matters), or with an X, Y, H or -H t beyond the largest bfloat16 (an infinite operand has
//    no three parts), is flagged where they are formed and redone by the exact kernels, which run
//    behind the factored ones on the flagged items only.
#include <algorithm>
#include <type_traits>

#include "logbmm_split.h"

namespace GENBMM_NS {
namespace {

// ------------------------------------------------------------------ exact passes
// tt: t per output cell as float (grad_g itself for float tensors; a buffer of the workspace for
// the half types, whose grad_g holds t rounded).  only: NULL, or one word per batch item - items
// whose word is 0 are skipped.
struct BB {
  const elem_t* a; const elem_t* b; const elem_t* out; const elem_t* g;
  const elem_t* ua; const elem_t* ub;
  elem_t* ga; elem_t* gb; elem_t* gg;
  float* tt;
  const int* only;
  int M, K, N;
  int B;
};

// The blocks of a pass.  A block is `per_block` consecutive units (cells or rows) starting at `base`
// and ending before `limit`; f(base, limit) works on one.  Without `only`: one block per workgroup
// over all units (numbered so that an item's workgroups share an XCD).  With it - the pass over
// flagged items, which usually finds none - a small grid looks all flags over at once (a round trip to
// memory per 64 of them took 6 to 7 us a launch at 512 items); if there are any, its workgroups
// form groups of one item's blocks (or one group that strides, for items of more blocks than the
// grid), and the flagged items go to the groups in turn: tens of thousands of workgroups that look
// up a flag and exit cost 60 us a launch.  blk of nblk: the workgroup's number in its pass.
constexpr int kBBOnlyGrid = 2048;
template <bool ONLY, class F>
__device__ __forceinline__ void bb_blocks(const BB& p, unsigned blk, unsigned nblk, long total, long per_item,
                                          int per_block, F&& f) {
  if constexpr (!ONLY) {
    f((long)xcd_renumber(blk, nblk) * per_block, total);
    return;
  }
  int any = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < p.B; i += 256) any |= p.only[i];
  if (!__syncthreads_or(any)) return;
  const int lane = threadIdx.x & 63;
  const long bpi = (per_item + per_block - 1) / per_block;  // blocks per item
  const bool fits = bpi <= (long)nblk;
  const long groups = fits ? (long)nblk / bpi : 1;
  const long grp = fits ? (long)blk / bpi : 0;
  if (grp >= groups) return;
  const long first = fits ? (long)blk - grp * bpi : (long)blk;
  const long stride = fits ? bpi : (long)nblk;
  long seen = 0;
  for (int b0 = 0; b0 < p.B; b0 += 64) {
    unsigned long long live = __ballot(b0 + lane < p.B && p.only[b0 + lane] != 0);
    while (live) {
      const long batch = b0 + __builtin_ctzll(live);
      live &= live - 1;
      if (seen++ % groups != grp) continue;
      for (long u = first * per_block; u < per_item; u += stride * per_block)
        f(batch * per_item + u, (batch + 1) * per_item);
    }
  }
}
inline dim3 bb_grid(const BB& p, long nblocks) {
  return dim3((unsigned)(p.only ? std::min<long>(nblocks, kBBOnlyGrid) : nblocks));
}

template <bool ONLY>
__global__ __launch_bounds__(256) void k_log_bwdbwd_t(const BB p, long total) {
  bb_blocks<ONLY>(p, blockIdx.x, gridDim.x, total, (long)p.M * p.N, 256, [&](long base, long limit) __attribute__((always_inline)) {
  const long e = base + threadIdx.x;
  if (e >= limit) return;
  const int n = (int)(e % p.N);
  const long bm = e / p.N;  // batch*M + m
  const long batch = bm / p.M;
  if (p.only && !p.only[batch]) return;
  const elem_t* arow = p.a + bm * p.K;
  const elem_t* uarow = p.ua ? p.ua + bm * p.K : nullptr;
  const elem_t* bcol = p.b + batch * p.K * p.N + n;
  const elem_t* ubcol = p.ub ? p.ub + batch * p.K * p.N + n : nullptr;
  const float o = p.out[e];
  float t = 0.f;
  for (int k = 0; k < p.K; ++k) {
    const float pr = fast_exp((float)arow[k] + (float)bcol[(long)k * p.N] - o);
    const float w = (uarow ? (float)uarow[k] : 0.f) + (ubcol ? (float)ubcol[(long)k * p.N] : 0.f);
    t = __builtin_fmaf(pr, w, t);
  }
  p.tt[e] = t;
  if constexpr (!kElemF32) p.gg[e] = to_elem<elem_t>(t);
  });
}

// grad_a: a wave per row (batch, m), its lanes along n - the one axis on which b, u_b, out, g and
// t are all contiguous (with a lane per cell (m, k) the reads of b run down a column, one cache
// line per lane).  The row's out, g and t stay in registers for N <= 256; per k the lanes'
// partial sums are added across the wave and 64 finished cells are written at once.
constexpr int kBBChunks = 4;  // n chunks of 64 a lane keeps in registers
template <bool ONLY>
__device__ __forceinline__ void bb_grad_a(const BB& p, unsigned blk, unsigned nblk, long rows) {
  bb_blocks<ONLY>(p, blk, nblk, rows, (long)p.M, 4, [&](long base, long limit) __attribute__((always_inline)) {
  const int lane = threadIdx.x & 63;
  const long bm = base + (threadIdx.x >> 6);
  if (bm >= limit) return;
  const long batch = bm / p.M;
  if (p.only && !p.only[batch]) return;
  const int K = p.K, N = p.N;
  const elem_t* arow = p.a + bm * K;
  const elem_t* uarow = p.ua ? p.ua + bm * K : nullptr;
  const elem_t* bmat = p.b + batch * K * N;
  const elem_t* ubmat = p.ub ? p.ub + batch * K * N : nullptr;
  const elem_t* orow = p.out + bm * N;
  const elem_t* grow = p.g + bm * N;
  const float* trow = p.tt + bm * N;
  const bool cached = N <= 64 * kBBChunks;
  float oc[kBBChunks], gc[kBBChunks], tc[kBBChunks];
#pragma unroll
  for (int j = 0; j < kBBChunks; ++j) {
    const int n = lane + 64 * j;
    const bool in = cached && n < N;
    oc[j] = in ? (float)orow[n] : 0.f;
    gc[j] = in ? (float)grow[n] : 0.f;
    tc[j] = in ? trow[n] : 0.f;
  }
  float mine = 0.f;  // the finished cell k with k % 64 == lane
  for (int k = 0; k < K; ++k) {
    const float av = arow[k], uav = uarow ? (float)uarow[k] : 0.f;
    const elem_t* brow = bmat + (long)k * N;
    const elem_t* ubrow = ubmat ? ubmat + (long)k * N : nullptr;
    float acc = 0.f;
    if (cached) {
#pragma unroll
      for (int j = 0; j < kBBChunks; ++j) {
        const int n = lane + 64 * j;
        if (n < N) {
          const float pr = fast_exp(av + (float)brow[n] - oc[j]);
          const float w = uav + (ubrow ? (float)ubrow[n] : 0.f) - tc[j];
          acc = __builtin_fmaf(gc[j] * pr, w, acc);
        }
      }
    } else {
      for (int n = lane; n < N; n += 64) {
        const float pr = fast_exp(av + (float)brow[n] - (float)orow[n]);
        const float w = uav + (ubrow ? (float)ubrow[n] : 0.f) - trow[n];
        acc = __builtin_fmaf((float)grow[n] * pr, w, acc);
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((k & 63) == lane) mine = acc;
    if ((k & 63) == 63 || k == K - 1) {
      const int k0 = k & ~63;
      if (k0 + lane <= k) p.ga[bm * K + k0 + lane] = to_elem<elem_t>(mine);
    }
  }
  });
}

template <bool ONLY>
__device__ __forceinline__ void bb_grad_b(const BB& p, unsigned blk, unsigned nblk, long total) {
  bb_blocks<ONLY>(p, blk, nblk, total, (long)p.K * p.N, 256, [&](long base, long limit) __attribute__((always_inline)) {
  const long e = base + threadIdx.x;
  if (e >= limit) return;
  const int n = (int)(e % p.N);
  const long bk = e / p.N;  // batch*K + k
  const long batch = bk / p.K;
  if (p.only && !p.only[batch]) return;
  const int k = (int)(bk - batch * p.K);
  const float bv = p.b[e];
  const float ubv = p.ub ? (float)p.ub[e] : 0.f;
  const elem_t* acol = p.a + batch * p.M * p.K + k;
  const elem_t* uacol = p.ua ? p.ua + batch * p.M * p.K + k : nullptr;
  const elem_t* ocol = p.out + batch * p.M * p.N + n;
  const elem_t* gcol = p.g + batch * p.M * p.N + n;
  const float* tcol = p.tt + batch * p.M * p.N + n;
  float acc = 0.f;
  for (int m = 0; m < p.M; ++m) {
    const long mn = (long)m * p.N;
    const float pr = fast_exp((float)acol[(long)m * p.K] + bv - (float)ocol[mn]);
    const float w = (uacol ? (float)uacol[(long)m * p.K] : 0.f) + ubv - tcol[mn];
    acc = __builtin_fmaf((float)gcol[mn] * pr, w, acc);
  }
  p.gb[e] = to_elem<elem_t>(acc);
  });
}

// Both gradients need t and not each other.  Over flagged items, of which there are hardly ever any, they are one
// launch, workgroups [0, split) grad_a's; over all items a launch each, which has each pass's own registers
// (a whole (512, 128^3): 1.86 ms, in one launch 1.99).
__global__ __launch_bounds__(256) void k_log_bwdbwd_ab(const BB p, unsigned split, long rows, long total) {
  if (blockIdx.x < split) bb_grad_a<true>(p, blockIdx.x, split, rows);
  else bb_grad_b<true>(p, blockIdx.x - split, gridDim.x - split, total);
}
__global__ __launch_bounds__(256) void k_log_bwdbwd_a(const BB p, long rows) {
  bb_grad_a<false>(p, blockIdx.x, gridDim.x, rows);
}
__global__ __launch_bounds__(256) void k_log_bwdbwd_b(const BB p, long total) {
  bb_grad_b<false>(p, blockIdx.x, gridDim.x, total);
}

// Two passes' workgroups in one launch of go(grid, split), the first pass's in front; in two launches where the
// sum of their work-items is beyond what one may have.
template <class F>
void launch_pair(dim3 first, dim3 second, F&& go) {
  if (((int64_t)first.x + second.x) * 256 <= 0xffffffffLL) {
    if (first.x + second.x > 0) go(dim3(first.x + second.x), first.x);
    return;
  }
  if (first.x > 0) go(first, first.x);
  if (second.x > 0) go(second, 0u);
}

int launch_exact(const BB& p, int B, hipStream_t s) {
  auto blocks = [&](long total) { return bb_grid(p, (total + 255) / 256); };
  const long tmn = (long)B * p.M * p.N, tmk = (long)B * p.M * p.K, tkn = (long)B * p.K * p.N;
  if (tmn > 0) {
    hipLaunchKernelGGL(p.only ? k_log_bwdbwd_t<true> : k_log_bwdbwd_t<false>, blocks(tmn), dim3(256), 0, s, p, tmn);
    if (int e = launch_status()) return e;
  }
  const long rows = tmk > 0 ? (long)B * p.M : 0;  // four rows per workgroup
  const dim3 grid_a = bb_grid(p, (rows + 3) / 4), grid_b = blocks(tkn);
  if (p.only) {
    if (grid_a.x + grid_b.x > 0)
      hipLaunchKernelGGL(k_log_bwdbwd_ab, dim3(grid_a.x + grid_b.x), dim3(256), 0, s, p, grid_a.x, rows, tkn);
    return launch_status();
  }
  if (grid_a.x > 0) {
    hipLaunchKernelGGL(k_log_bwdbwd_a, grid_a, dim3(256), 0, s, p, rows);
    if (int e = launch_status()) return e;
  }
  if (grid_b.x > 0) hipLaunchKernelGGL(k_log_bwdbwd_b, grid_b, dim3(256), 0, s, p, tkn);
  return launch_status();
}

// ------------------------------------------------------------------ factored form
constexpr int kBBPad = 128;  // every extent of the workspace's arrays is a multiple of this
inline int bb_pad(int x) { return (x + kBBPad - 1) / kBBPad * kBBPad; }
// The factored form pays from here on (padding to 128 at most doubles an extent of 64).
inline bool bb_factored_ok(int B, int M, int K, int N) {
  return min(M, min(K, N)) >= 64 && (int64_t)B * M * K * N >= ((int64_t)1 << 21);
}

struct BBWs {
  float* t_exact;  // (B, M, N): t for the exact passes (and unrounded for the half types)
  float* alpha;    // (B, Mp)
  float* beta;     // (B, Np)
  int* flags;      // (B): items to redo exactly
  float *ea, *x;   // (B, Mp, Kp): exp(a - alpha), ea * u_a
  float *eb, *y;   // (B, Kp, Np)
  float *h, *nht;  // (B, Mp, Np): g exp(alpha + beta - out), -h t
};
inline size_t bb_ws_floats(int B, int M, int K, int N, BBWs* w, float* base) {
  size_t off = 0;
  auto take = [&](size_t n) {
    float* p = base ? base + off : nullptr;
    off += (n + 3) & ~(size_t)3;
    return p;
  };
  BBWs t{};
  t.t_exact = take((size_t)B * M * N);
  if (bb_factored_ok(B, M, K, N)) {
    const size_t Mp = bb_pad(M), Kp = bb_pad(K), Np = bb_pad(N);
    t.alpha = take(B * Mp);
    t.beta = take(B * Np);
    t.flags = reinterpret_cast<int*>(take(B));
    t.ea = take(B * Mp * Kp); t.x = take(B * Mp * Kp);
    t.eb = take(B * Kp * Np); t.y = take(B * Kp * Np);
    t.h = take(B * Mp * Np); t.nht = take(B * Mp * Np);
  }
  if (w) *w = t;
  return off;
}

// The passes move four cells per lane and instruction (the padded extents are multiples of
// 128; rows of the caller's tensors start at any element, which the loads take).
__device__ __forceinline__ float4 exp4_st(float4 v, float m) {
  return make_float4(exp_st(v.x - m), exp_st(v.y - m), exp_st(v.z - m), exp_st(v.w - m));
}
__device__ __forceinline__ float4 mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float max4(float m, float4 v) { return fmaxf(fmaxf(m, fmaxf(v.x, v.y)), fmaxf(v.z, v.w)); }

// every value has three bfloat16 parts (NaN, infinities and what rounds to one do not)
__device__ __forceinline__ bool splits(float v) { return fabsf(v) <= 0x1.fep127f; }
__device__ __forceinline__ bool splits4(float4 v) { return splits(v.x) && splits(v.y) && splits(v.z) && splits(v.w); }

// alpha, EA, X: a wave per padded row (b, mp) - half a wave where a row is 128 cells, 32 lanes' worth;
// rows and columns of the padding hold zeros.
__device__ __forceinline__ void bb_prep_a(unsigned blk, const elem_t* __restrict__ a, const elem_t* __restrict__ ua,
                                          float* __restrict__ alpha, float* __restrict__ ea, float* __restrict__ x,
                                          int* __restrict__ flags, int M, int K, int Mp, int Kp, long rows) {
  const int lpr = Kp == 128 ? 32 : 64;  // lanes per row
  const int lane = threadIdx.x & (lpr - 1);
  const long row = ((long)blk * 256 + threadIdx.x) / lpr;
  if (row >= rows) return;
  const long batch = row / Mp;
  const int m = (int)(row - batch * Mp);
  if (row < (rows / Mp) && lane == 0) flags[row] = 0;  // (rows / Mp = B words, cleared by the first B rows)
  float* er = ea + row * Kp;
  float* xr = x + row * Kp;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const int step = lpr * 4;
  if (m >= M) {
    for (int k = lane * 4; k < Kp; k += step) { st4(er + k, zero); st4(xr + k, zero); }
    if (lane == 0) alpha[row] = 0.f;
    return;
  }
  const elem_t* ar = a + (batch * M + m) * K;
  const elem_t* ur = ua ? ua + (batch * M + m) * K : nullptr;
  float mx = -INFINITY;
  for (int k = lane * 4; k < K; k += step) mx = max4(mx, ld4m(ar + k, K - k, -INFINITY));
  // (the exchange stays within the row's own lanes, all of which are here)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    if (off < lpr) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  bool bad = false;
  for (int k = lane * 4; k < Kp; k += step) {
    // (the fill -inf gives exp = 0 in the padding; a row of -inf has mx = -inf and NaN here, and is
    //  flagged where H is formed)
    const float4 e = k < K ? exp4_st(ld4m(ar + k, K - k, -INFINITY), mx) : zero;
    const float4 xv = (ur && k < K) ? mul4(e, ld4m(ur + k, K - k, 0.f)) : zero;
    bad = bad || !splits4(xv);
    st4(er + k, e);
    st4(xr + k, xv);
  }
  // (the flags are being cleared here: a row that does not split has no maximum, and its item
  //  is flagged where H is formed)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    if (off < lpr) bad = bad | (bool)__shfl_xor((int)bad, off, 64);
  if (lane == 0) alpha[row] = bad ? NAN : mx;
}

// beta, EB, Y: a workgroup per (batch item, 64 columns): 16 lanes x 4 columns across, the 16 lane
// groups of the four waves split the rows of b.
__device__ __forceinline__ void bb_prep_b(unsigned blk, const elem_t* __restrict__ b, const elem_t* __restrict__ ub,
                                          float* __restrict__ beta, float* __restrict__ eb, float* __restrict__ y,
                                          int K, int N, int Kp, int Np) {
  __shared__ __attribute__((aligned(16))) float part[16][64];
  const int cq = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int cblocks = Np / 64;
  const long batch = blk / cblocks;
  const int n = (int)(blk - batch * cblocks) * 64 + cq * 4;
  const int cnt = N - n;  // live columns of this lane's four (<= 0: none)
  const elem_t* bc = b + batch * K * N + (cnt > 0 ? n : 0);
  const elem_t* uc = ub ? ub + batch * K * N + (cnt > 0 ? n : 0) : nullptr;
  float4 mx = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
  for (int k = rg; k < K; k += 16) {
    const float4 v = ld4m(bc + (long)k * N, cnt, -INFINITY);
    mx = make_float4(fmaxf(mx.x, v.x), fmaxf(mx.y, v.y), fmaxf(mx.z, v.z), fmaxf(mx.w, v.w));
  }
  st4a(&part[rg][cq * 4], mx);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float4 v = ld4a(&part[r][cq * 4]);
    mx = make_float4(fmaxf(mx.x, v.x), fmaxf(mx.y, v.y), fmaxf(mx.z, v.z), fmaxf(mx.w, v.w));
  }
  float* ec = eb + batch * Kp * Np + n;
  float* yc = y + batch * Kp * Np + n;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  bool bad = false;
  for (int k = rg; k < Kp; k += 16) {
    const bool in = cnt > 0 && k < K;
    float4 e = zero;
    if (in) {
      const float4 v = ld4m(bc + (long)k * N, cnt, -INFINITY);
      e = make_float4(exp_st(v.x - mx.x), cnt > 1 ? exp_st(v.y - mx.y) : 0.f, cnt > 2 ? exp_st(v.z - mx.z) : 0.f,
                      cnt > 3 ? exp_st(v.w - mx.w) : 0.f);
    }
    const float4 yv = (uc && in) ? mul4(e, ld4m(uc + (long)k * N, cnt, 0.f)) : zero;
    bad = bad || !splits4(yv);
    st4(ec + (long)k * Np, e);
    st4(yc + (long)k * Np, yv);
  }
  // (a column that does not split has no maximum, as a row above)
  bad = __syncthreads_or(bad);
  if (rg == 0)
    st4(beta + batch * Np + n, bad ? make_float4(NAN, NAN, NAN, NAN)
                                   : make_float4(cnt > 0 ? mx.x : 0.f, cnt > 1 ? mx.y : 0.f, cnt > 2 ? mx.z : 0.f,
                                                 cnt > 3 ? mx.w : 0.f));
}

// Both operands' passes in one launch, workgroups [0, split) the columns'.
__global__ __launch_bounds__(256) void k_bb_prep_ab(const elem_t* __restrict__ a, const elem_t* __restrict__ ua,
                                                    const elem_t* __restrict__ b, const elem_t* __restrict__ ub,
                                                    const BBWs w, unsigned split, int M, int K, int N, int Mp, int Kp,
                                                    int Np, long rows) {
  if (blockIdx.x < split) bb_prep_b(blockIdx.x, b, ub, w.beta, w.eb, w.y, K, N, Kp, Np);
  else bb_prep_a(blockIdx.x - split, a, ua, w.alpha, w.ea, w.x, w.flags, M, K, Mp, Kp, rows);
}

// One tile of C = P1 Q1 (+ P2 Q2) and its epilogue; for a gradient also of C0 = P3 Q3.  Operands are padded workspace arrays:
//   RT: the rows operand is stored [row][red] (staged transposed), else [red][row];
//   CT: the columns operand is stored [col][red], else [red][col].
constexpr int kEpiT = 0, kEpiGrad = 1;
struct BBMM {
  const float* rows[2];
  const float* cols[2];
  int pairs;
  const float* rows0;   // kEpiGrad: C0's operands, or NULL
  const float* cols0;
  int Rp, Cp, Qp;       // padded extents: output rows, output columns, reduction
  // epilogue
  const float* f_acc;   // kEpiGrad: EA / EB, the factor of the accumulator
  const float* f0;      // kEpiGrad: X / Y, the factor of C0
  const elem_t* out;    // kEpiT: what R and H are formed from
  const elem_t* g;
  const float* alpha;
  const float* beta;
  float* h;             // kEpiT: H
  float* nht;           // kEpiT: -H t
  int* flags;           // kEpiT: per item, set beyond the guard and where H or -H t does not split
  float* tt;            // kEpiT: t unrounded, (B, R, C) unpadded
  elem_t* dst;          // kEpiT: grad_g; kEpiGrad: grad_a / grad_b; (B, R, C) unpadded
  int R, C;             // true extents of the output
};

// The products run on the bf16 matrix instruction, every operand cut into three parts while it is staged
// (split_bf16.h; logbmm_split.h has the staging and the inner loop): on the fp32 instruction, which does a
// sixteenth of the reduction steps in the same time, the five launches of (512, 128^3) took 245 us; three-part
// 240, and 205 (178 with steps of one line staged) with H EB^T and EA^T H formed in the launches that use them (a second set of accumulators)
// instead of written out and read back.
// Bound by what the workspace arrays move (two or four in, one to three more in the epilogue).
using BBTile = MTile<128, 128, 2>;
template <bool RT, bool CT, int EPI>
__global__ __launch_bounds__(BBTile::NT) __attribute__((amdgpu_waves_per_eu(BBTile::WPE, BBTile::WPE)))
void k_bb_mm(const BBMM p) {
  using T = BBTile;
  constexpr int NT = T::NT;
  using SR = std::conditional_t<RT, SplitT<T::TR, NT>, SplitL<T::TR, NT>>;
  using SC = std::conditional_t<CT, SplitT<T::TC, NT>, SplitL<T::TC, NT>>;
  constexpr int PER = 2, ST = 8;  // a thread's pieces of an operand: four steps of two lines, or eight steps of one
  __shared__ __attribute__((aligned(16))) unsigned smem[split_lds_words<SR, SC>()];
  static_assert(split_lds_words<SR, SC>() >= (NT / 64) * kStripFloats, "");
  auto Rs = [&](int buf) __attribute__((always_inline)) { return smem + buf * SR::BUF; };
  auto Cs = [&](int buf) __attribute__((always_inline)) { return smem + 2 * SR::BUF + buf * SC::BUF; };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr0 = (wave / T::WC) * 64, wc0 = (wave % T::WC) * 64;
  const int tiles_c = p.Cp / T::TC, per = (p.Rp / T::TR) * tiles_c;
  const int tile = xcd_tile_id();
  const int batch = tile / per, rem = tile - batch * per;
  const int r0 = (rem / tiles_c) * T::TR, c0 = (rem % tiles_c) * T::TC;
  const int Qp = p.Qp, slabs = Qp / kMS;

  floatx16 acc[2][2], acc0[2][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[x >> 1][x & 1][i] = acc0[x >> 1][x & 1][i] = 0.f;

  // where this thread's pieces of the first slab lie in an operand of either layout: uniform base, lane offsets
  long rbase, cbase;
  unsigned ro[PER], co[PER];
  if constexpr (RT) {
    rbase = ((long)batch * p.Rp + r0) * Qp;
#pragma unroll
    for (int l = 0; l < PER; ++l) ro[l] = SR::line(tid, l) * Qp + SR::quad(tid) * 4;
  } else {
    rbase = ((long)batch * Qp + SR::step0(tid)) * p.Rp + r0;
    ro[0] = SR::line(tid);
  }
  if constexpr (CT) {
    cbase = ((long)batch * p.Cp + c0) * Qp;
#pragma unroll
    for (int l = 0; l < PER; ++l) co[l] = SC::line(tid, l) * Qp + SC::quad(tid) * 4;
  } else {
    cbase = ((long)batch * Qp + SC::step0(tid)) * p.Cp + c0;
    co[0] = SC::line(tid);
  }
  // the slabs of both products are one loop: the second's first slab is in flight under the first's last
  const float *rb = p.rows[0] + rbase, *cb = p.cols[0] + cbase;
  const long rstep = RT ? (long)kMS : (long)kMS * p.Rp, cstep = CT ? (long)kMS : (long)kMS * p.Cp;
  int s_load = 0;
  float4 rr[RT ? PER : 1], rc[CT ? PER : 1];
  float sr[RT ? 1 : ST], sc[CT ? 1 : ST];
  auto load = [&]() __attribute__((always_inline)) {
    if constexpr (RT) {
#pragma unroll
      for (int l = 0; l < PER; ++l) rr[l] = ld4a(rb + ro[l]);
    } else {
#pragma unroll
      for (int j = 0; j < ST; ++j) sr[j] = (rb + (long)j * p.Rp)[ro[0]];
    }
    if constexpr (CT) {
#pragma unroll
      for (int l = 0; l < PER; ++l) rc[l] = ld4a(cb + co[l]);
    } else {
#pragma unroll
      for (int j = 0; j < ST; ++j) sc[j] = (cb + (long)j * p.Cp)[co[0]];
    }
    const bool next = ++s_load == slabs;  // uniform
    rb = next ? p.rows[1] + rbase : rb + rstep;
    cb = next ? p.cols[1] + cbase : cb + cstep;
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
    if constexpr (RT) {
#pragma unroll
      for (int l = 0; l < PER; ++l) SR::put(Rs(buf), tid, l, rr[l]);
    } else {
      SR::put(Rs(buf), tid, sr);
    }
    if constexpr (CT) {
#pragma unroll
      for (int l = 0; l < PER; ++l) SC::put(Cs(buf), tid, l, rc[l]);
    } else {
      SC::put(Cs(buf), tid, sc);
    }
  };
  load();
  stage(0);
  split_loop(slabs * p.pairs, split_early<NT>(wave), load, stage, [&](int buf) __attribute__((always_inline)) {
    split_slab<SR, SC>(Rs(buf), Cs(buf), wr0, wc0, wave & (NT / 64 - 1), lane, acc);
  });
  if (EPI == kEpiGrad && p.rows0) {  // uniform
    rb = p.rows0 + rbase;
    cb = p.cols0 + cbase;
    load();
    stage(0);
    split_loop(slabs, split_early<NT>(wave), load, stage, [&](int buf) __attribute__((always_inline)) {
      split_slab<SR, SC>(Rs(buf), Cs(buf), wr0, wc0, wave & (NT / 64 - 1), lane, acc0);
    });
  }

  // epilogue, row-wise: f(q, t, v) = four columns lc .. lc + 3 of block row 16 q + 4 t + lr
  const int lr = lane >> 4, lc = (lane & 15) * 4;
  const int row0 = r0 + wr0 + lr, col = c0 + wc0 + lc;
  const long pbase = ((long)batch * p.Rp + row0) * p.Cp + col;   // padded arrays
  const int cc = clamp4(p.C - col);                              // columns of the piece that exist
  float* strip = reinterpret_cast<float*>(smem) + wave * kStripFloats;
  if constexpr (EPI == kEpiT) {
    // R = exp(alpha + beta - out), H = g R (zeros in the padding): formed here, where R is used and H first is.
    // (512, 128^3): a pass of its own that wrote both took 25 us, this launch 56 with R and H read and 56 so.
    bool bad = false;
    const float lim = kMfmaGuardBits * kLn2 + 1e-3f;
    const int pc = min(col, p.C - 4), shift = col - pc;  // a piece over the right edge reads the last four columns
    const float4 be4 = ld4(p.beta + (long)batch * p.Cp + col);
    const float be[4] = {be4.x, be4.y, be4.z, be4.w};
    auto columns = [&](float4 v, float (&x)[4]) __attribute__((always_inline)) {
      if (shift & 1) v = make_float4(v.y, v.z, v.w, 0.f);
      if (shift & 2) v = make_float4(v.z, v.w, 0.f, 0.f);
      x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    };
    float4 o4[4], g4[4];
    float al[4];
    acc_rows(acc, strip, lane,
             [&](int q) __attribute__((always_inline)) {
#pragma unroll
               for (int t = 0; t < 4; ++t) {
                 const int row = row0 + 16 * q + 4 * t;
                 const long src = ((long)batch * p.R + min(row, p.R - 1)) * p.C + pc;
                 o4[t] = ld4(p.out + src);
                 g4[t] = ld4(p.g + src);
                 al[t] = p.alpha[(long)batch * p.Rp + row];
               }
             },
             [&](int q, int t, float4 v) __attribute__((always_inline)) {
               const int ru = 16 * q + 4 * t;
               const long pu = pbase + (long)ru * p.Cp;
               const long du = ((long)batch * p.R + row0 + ru) * p.C + col;  // unpadded arrays
               const int live = row0 + ru < p.R ? cc : 0;
               float o[4], gv[4], rv[4], hv[4];
               columns(o4[t], o);
               columns(g4[t], gv);
               bad = bad || (live > 0 && !(al[t] > -INFINITY));
#pragma unroll
               for (int i = 0; i < 4; ++i) {
                 const float ex = al[t] + be[i] - o[i], r = exp_st(ex), h = gv[i] * r;
                 const bool in = i < live;
                 // (a negated comparison: NaN and +inf fail it; alpha, beta not finite make ex not finite or NaN)
                 bad = bad || (in && (!(ex <= lim) || !(be[i] > -INFINITY) || !splits(h)));
                 rv[i] = in ? r : 0.f;
                 hv[i] = in ? h : 0.f;
               }
               const float4 tv = make_float4(rv[0] * v.x, rv[1] * v.y, rv[2] * v.z, rv[3] * v.w);
               const float4 nv = make_float4(-hv[0] * tv.x, -hv[1] * tv.y, -hv[2] * tv.z, -hv[3] * tv.w);
               bad = bad || !splits4(nv);
               st4a(p.h + pu, make_float4(hv[0], hv[1], hv[2], hv[3]));
               st4a(p.nht + pu, nv);
               if (live > 0) {
                 st4m(p.tt + du, cc, tv);
                 if constexpr (!kElemF32) st4m(p.dst + du, cc, tv);
               }
             });
    if (bad) p.flags[batch] = 1;
  } else {
    // C0 scaled by its factor first, kept in registers as rows; then the other product joins it
    float4 o[16];
    if (p.rows0)
      acc_rows(acc0, strip, lane, [](int) {}, [&](int q, int t, float4 v) __attribute__((always_inline)) {
        const float4 x = ld4a(p.f0 + pbase + (long)(16 * q + 4 * t) * p.Cp);
        o[4 * q + t] = make_float4(x.x * v.x, x.y * v.y, x.z * v.z, x.w * v.w);
      });
    else
#pragma unroll
      for (int x = 0; x < 16; ++x) o[x] = make_float4(0.f, 0.f, 0.f, 0.f);
    acc_rows(acc, strip, lane, [](int) {}, [&](int q, int t, float4 v) __attribute__((always_inline)) {
      const int ru = 16 * q + 4 * t;
      const float4 fa = ld4a(p.f_acc + pbase + (long)ru * p.Cp), c0v = o[4 * q + t];
      if (row0 + ru < p.R && cc > 0)
        st4m(p.dst + ((long)batch * p.R + row0 + ru) * p.C + col, cc,
             make_float4(__builtin_fmaf(fa.x, v.x, c0v.x), __builtin_fmaf(fa.y, v.y, c0v.y),
                         __builtin_fmaf(fa.z, v.z, c0v.z), __builtin_fmaf(fa.w, v.w, c0v.w)));
    });
  }
}

template <bool RT, bool CT, int EPI>
int launch_mm(const BBMM& p, int B, hipStream_t s) {
  const int64_t tiles = (int64_t)B * (p.Rp / 128) * (p.Cp / 128);
  if (tiles > 0x7fffffffLL) return GENBMM_E_SHAPE;
  hipLaunchKernelGGL((k_bb_mm<RT, CT, EPI>), dim3((unsigned)tiles), dim3(256), 0, s, p);
  return launch_status();
}

int bwdbwd_factored(const BB& p, const BBWs& w, int B, hipStream_t s) {
  const int M = p.M, K = p.K, N = p.N, Mp = bb_pad(M), Kp = bb_pad(K), Np = bb_pad(N);
  {
    const long rows = (long)B * Mp;
    const long per_wg = Kp == 128 ? 8 : 4;  // rows per workgroup: 32 or 64 lanes each
    launch_pair(dim3((unsigned)(B * (Np / 64))), dim3((unsigned)((rows + per_wg - 1) / per_wg)),
                [&](dim3 grid, unsigned split) {
      hipLaunchKernelGGL(k_bb_prep_ab, grid, dim3(256), 0, s, p.a, p.ua, p.b, p.ub, w, split, M, K, N, Mp, Kp, Np, rows);
    });
    if (int e = launch_status()) return e;
  }
  const bool has_a = p.ua != nullptr, has_b = p.ub != nullptr;
  {  // t = R (X EB + EA Y); also -H t and grad_g
    BBMM q{};
    int n = 0;
    if (has_a) { q.rows[n] = w.x; q.cols[n] = w.eb; ++n; }
    if (has_b) { q.rows[n] = w.ea; q.cols[n] = w.y; ++n; }
    q.pairs = n; q.Rp = Mp; q.Cp = Np; q.Qp = Kp; q.R = M; q.C = N;
    q.out = p.out; q.g = p.g; q.alpha = w.alpha; q.beta = w.beta; q.h = w.h; q.nht = w.nht; q.flags = w.flags; q.tt = p.tt; q.dst = p.gg;
    if (int e = launch_mm<true, false, kEpiT>(q, B, s)) return e;
  }
  {  // grad_a = X (H EB^T) + EA (H Y^T - (H t) EB^T)
    BBMM q{};
    int n = 0;
    if (has_b) { q.rows[n] = w.h; q.cols[n] = w.y; ++n; }
    q.rows[n] = w.nht; q.cols[n] = w.eb; ++n;
    q.pairs = n; q.Rp = Mp; q.Cp = Kp; q.Qp = Np; q.R = M; q.C = K;
    q.f_acc = w.ea; q.dst = p.ga;
    if (has_a) { q.rows0 = w.h; q.cols0 = w.eb; q.f0 = w.x; }
    if (int e = launch_mm<true, true, kEpiGrad>(q, B, s)) return e;
  }
  {  // grad_b = Y (EA^T H) + EB (X^T H - EA^T (H t))
    BBMM q{};
    int n = 0;
    if (has_a) { q.rows[n] = w.x; q.cols[n] = w.h; ++n; }
    q.rows[n] = w.ea; q.cols[n] = w.nht; ++n;
    q.pairs = n; q.Rp = Kp; q.Cp = Np; q.Qp = Mp; q.R = K; q.C = N;
    q.f_acc = w.eb; q.dst = p.gb;
    if (has_b) { q.rows0 = w.ea; q.cols0 = w.h; q.f0 = w.y; }
    if (int e = launch_mm<false, false, kEpiGrad>(q, B, s)) return e;
  }
  // items beyond the guard: the exact passes, on those items only
  BB ex = p;
  ex.only = w.flags;
  return launch_exact(ex, B, s);
}

int bwdbwd(const elem_t* a, const elem_t* b, const elem_t* out, const elem_t* g, const elem_t* u_a,
           const elem_t* u_b, elem_t* grad_a, elem_t* grad_b, elem_t* grad_g, float* workspace, int B, int M,
           int K, int N, void* stream) {
  if (int e = check_dense_dims(B, M, K, N)) return e;
  {
    const int64_t mk = (int64_t)B * M * K, kn = (int64_t)B * K * N, mn = (int64_t)B * M * N;
    if (missing(a, mk) || missing(b, kn) || missing(out, mn) || missing(g, mn) ||
        missing(grad_a, mk) || missing(grad_b, kn) || missing(grad_g, mn) ||
        (missing(u_a, mk) && missing(u_b, kn)))
      return GENBMM_E_NULLPTR;
    if (!kElemF32 && missing(workspace, mn)) return GENBMM_E_NULLPTR;  // t must stay unrounded somewhere
  }
  hipStream_t s = (hipStream_t)stream;
  BB p{a, b, out, g, u_a, u_b, grad_a, grad_b, grad_g, nullptr, nullptr, M, K, N, B};
  BBWs w{};
  if (workspace) bb_ws_floats(B, M, K, N, &w, workspace);
  if constexpr (kElemF32) p.tt = reinterpret_cast<float*>(grad_g);
  else p.tt = w.t_exact;
  if (workspace && bb_factored_ok(B, M, K, N) && (int64_t)B * M * K > 0 && (int64_t)B * K * N > 0)
    return bwdbwd_factored(p, w, B, s);
  return launch_exact(p, B, s);
}

}  // namespace
}  // namespace GENBMM_NS

extern "C" {

#if GENBMM_ELEM == 0
size_t genbmm_logbmm_bwdbwd_ws_size(int B, int M, int K, int N) {
  using namespace GENBMM_NS;
  if (check_dense_dims(B, M, K, N)) return 0;
  return bb_ws_floats(B, M, K, N, nullptr, nullptr);
}

int genbmm_logbmm_bwdbwd(const float* a, const float* b, const float* out, const float* g,
                         const float* u_a, const float* u_b, float* grad_a, float* grad_b,
                         float* grad_g, int B, int M, int K, int N, void* stream) {
  return GENBMM_NS::bwdbwd(a, b, out, g, u_a, u_b, grad_a, grad_b, grad_g, nullptr, B, M, K, N, stream);
}
#endif

// One per element type: genbmm_logbmm_bwdbwd_ws, ..._ws_f16, ..._ws_bf16
int GENBMM_API(logbmm_bwdbwd_ws)(const GENBMM_NS::abi_t* a, const GENBMM_NS::abi_t* b, const GENBMM_NS::abi_t* out,
                                 const GENBMM_NS::abi_t* g, const GENBMM_NS::abi_t* u_a, const GENBMM_NS::abi_t* u_b,
                                 GENBMM_NS::abi_t* grad_a, GENBMM_NS::abi_t* grad_b, GENBMM_NS::abi_t* grad_g,
                                 float* workspace, int B, int M, int K, int N, void* stream) {
  using namespace GENBMM_NS;
  return bwdbwd(el(a), el(b), el(out), el(g), el(u_a), el(u_b), el(grad_a), el(grad_b), el(grad_g), workspace, B, M, K,
                N, stream);
}

}  // extern "C"
