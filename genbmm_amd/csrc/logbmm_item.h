// logbmm for small matrices (extents of at most 128, and their LDS below): one workgroup per batch item, the
// whole item in LDS, one launch for the forward and one for both gradients, the
// contractions on v_mfma_f32_16x16x4_f32.
//
// Same factored form as the large kernels: alpha[m] = max_k a, beta[n] = max_k b
// are taken inside the workgroup, EA = exp(a - alpha), EB = exp(b - beta),
// S = EA * EB, out = log S + alpha + beta, H = g * exp(alpha + beta - out),
// grad_a = EA .* (H * EB^T), grad_b = EB .* (EA^T * H).  Rows of the result, rows of grad_a
// and columns of grad_b with a cell for which the factoring is not exact to fp32 - S < 2^-40,
// anything non-finite, in the forward a shift below the reference's -1e9 floor - are formed again
// at the end of the same kernel in the reference's own two-pass form (item_fwd_rows, item_bwd_exact).
//
// Staging: a wave takes groups of four neighbouring rows of an array, its lanes the columns (a row is
// contiguous in memory; all loads of the item are issued before the first is waited for).  A row's
// maximum is then one wave's reduction and a scalar, a column's is joined through LDS, and a lane's
// four rows are four neighbouring steps of an operand whose lines are the columns: one 16-byte store.
// Arrays are padded to multiples of 16 with zeros, lines are 16 j + 4 words apart: the 16-byte reads of
// a matrix operand (16 lines x 4 steps each) and the stores across lines meet every bank evenly.
//
// Why 16 x 16 tiles of the fp32 instruction: padding to 16 instead of 32 or 64 is what sizes in between
// cost ((8192,39^3): 2.4 times fewer products than with 32), and at these extents an item's products take no longer
// than its memory traffic, so the three-part form of the larger kernels would pay its cuts for nothing.
//
// Measured, forward + both gradients (before: the item on the vector ALU up to 64^3, the factored vector-ALU kernels or one
// 128 x 128 tile beyond): (2048,64^3) 44 + 73 -> 33 + 53 us, (8192,39^3) 99 + 158 -> 55 + 83 (bfloat16 112 + 220 -> 51 + 77),
// (5163,57^3) float16 113 + 245 -> 65 + 104, (1806,69,53,54) 76 + 151 -> 35 + 58, (512,64,128,64) 27 + 47 -> 18 + 38,
// (948,88^3) 46 + 109 -> 41 + 84, (500,96^3) 26 + 61 -> 25 + 49, (16,64^3) 9.6 + 14.1 -> 8.1 + 10.3.  (2048,64^3) moves 302 MB:
// 3.5 TB/s; what it spends beside memory is issue slots, some 700 of them a wave and direction on staging.
#pragma once

#include "common.h"
#include "logbmm_ws.h"

namespace GENBMM_NS {

constexpr float kItemGuardBits = 40.f;
constexpr int kItemMax = 128;  // largest extent these kernels take
// Of the backward's workgroup, at most; beyond, one 128 x 128 tile per item (two workgroups of three-part products: (500,100^3)
// 29 + 70 us against 36 + 63 in one workgroup of 160 KB).
constexpr int kItemLds = 136 * 1024;

// log-sum-exp of a[m,:] + b[:,n] the way the reference's kernel does it
// (matmul_cuda_kernel.cu:27-41): running maximum from -1e9, then the sum.
__device__ __forceinline__ float item_exact_out(const elem_t* __restrict__ arow,
                                                const elem_t* __restrict__ bcol, int K, int N) {
  float mx = kFloor;
  for (int k = 0; k < K; ++k) mx = fmaxf(mx, (float)arow[k] + (float)bcol[(long)k * N]);
  const float nm = -mx * kLog2e;
  float s = 0.f;
  for (int k = 0; k < K; ++k)
    s += fast_exp2(__builtin_fmaf((float)arow[k] + (float)bcol[(long)k * N], kLog2e, nm));
  return logf(s) + mx;
}

// Sums of shifts from which on every term lies so far below the reference's floor that its exponential is 0.
constexpr float kItemDead = kFloor - 1024.f;

// exp(x - shift), with the all -inf row / column (shift = -inf) giving zeros
__device__ __forceinline__ float item_exp(float x, float shift) {
  return fast_exp2((x - (shift == -INFINITY ? 0.f : shift)) * kLog2e);
}

// The larger of two values that are no numbers of a computation yet (fmaxf would quiet each of them in an instruction
// of its own first); of a NaN and a number the number.
__device__ __forceinline__ float item_max(float x, float y) { return __builtin_amdgcn_fmed3f(x, y, INFINITY); }

// Maxima over the wave of four registers, as scalars: two registers become one at each exchange between the halves
// and quarters of the wave, then four rotations within a quarter serve all four (18 instructions; a reduction
// of each takes 50).
__device__ __forceinline__ void item_wave_max4(float (&v)[4], float (&m)[4]) {
  auto u = [](float x) { return __float_as_uint(x); };
  auto f = [](unsigned x) { return __uint_as_float(x); };
  const auto p = __builtin_amdgcn_permlane32_swap(u(v[0]), u(v[1]), false, false);  // halves: of v0, of v1
  const auto q = __builtin_amdgcn_permlane32_swap(u(v[2]), u(v[3]), false, false);
  const float x = item_max(f(p[0]), f(p[1])), y = item_max(f(q[0]), f(q[1]));
  const auto r = __builtin_amdgcn_permlane16_swap(u(x), u(y), false, false);  // quarters: of v0, v2, v1, v3
  float z = item_max(f(r[0]), f(r[1]));
  auto turn = [&](auto ctrl) __attribute__((always_inline)) {
    z = item_max(z, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(z), decltype(ctrl)::value, 0xf, 0xf, true)));
  };
  turn(std::integral_constant<int, 0x128>{});  // row_ror:8
  turn(std::integral_constant<int, 0x124>{});
  turn(std::integral_constant<int, 0x122>{});
  turn(std::integral_constant<int, 0x121>{});
  const int at[4] = {0, 32, 16, 48};
#pragma unroll
  for (int t = 0; t < 4; ++t) m[t] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), at[t]));
}

// Of an R x C array, the rows 4 (wave + W u) + t and the columns lane + 64 h that a wave stages.  `raw` is as
// loaded: always the same loads (rows and columns beyond the matrix read its last ones), none waited for
// before it is used.  Rows beyond the matrix may stay its last one's copies: what they meet is zero.
template <int W, int U, int H>
struct ItemRows {
  elem_t raw[U][4][H];
  float v[U][4][H];
  __device__ __forceinline__ void load(const elem_t* __restrict__ x, int R, int C, int wave, int lane) {
    constexpr int kSize = sizeof(elem_t);
    const buf_t src = buf_of(x, (unsigned)(R * C * kSize));
    const int pitch = C * kSize, last = (R - 1) * pitch;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int at = min(lane + 64 * h, C - 1) * kSize;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int first = 4 * (wave + W * u) * pitch;  // uniform
#pragma unroll
        for (int t = 0; t < 4; ++t) raw[u][t][h] = buf_ld<elem_t>(src, at, min(first + t * pitch, last));
      }
    }
  }
  // v: the loaded cells, -infinity in columns beyond the matrix
  __device__ __forceinline__ void settle(int C, int lane) {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t) v[u][t][h] = lane + 64 * h < C ? (float)raw[u][t][h] : -INFINITY;
  }
  // f(u, first row, column chunk) for every group within Rp rows, in the lanes inside Cp columns
  template <class F>
  static __device__ __forceinline__ void each(int Rp, int Cp, int wave, int lane, F&& f) {
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (lane + 64 * h < Cp) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int r0 = 4 * (wave + W * u);
          if (r0 < Rp) f(u, r0, h);  // uniform
        }
      }
  }
  __device__ __forceinline__ void put_rows(float* __restrict__ dst, int ld, int Rp, int Cp, int wave, int lane) const {
    each(Rp, Cp, wave, lane, [&](int u, int r0, int h) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 4; ++t) dst[(r0 + t) * ld + lane + 64 * h] = v[u][t][h];
    });
  }
  // transposed: [column][row]
  __device__ __forceinline__ void put_cols(float* __restrict__ dst, int ld, int Rp, int Cp, int wave, int lane) const {
    each(Rp, Cp, wave, lane, [&](int u, int r0, int h) __attribute__((always_inline)) {
      *reinterpret_cast<float4*>(dst + (lane + 64 * h) * ld + r0) =
          make_float4(v[u][0][h], v[u][1][h], v[u][2][h], v[u][3][h]);
    });
  }
};

// The maxima of a's rows (left in al[u][t], scalars) and a becomes exp(a - alpha).
template <int W, int U, int H>
__device__ __forceinline__ void item_rows_exp(ItemRows<W, U, H>& x, float (&al)[U][4]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float m[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      m[t] = x.v[u][t][0];
#pragma unroll
      for (int h = 1; h < H; ++h) m[t] = item_max(m[t], x.v[u][t][h]);
    }
    item_wave_max4(m, al[u]);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float sh = al[u][t] == -INFINITY ? 0.f : al[u][t];
#pragma unroll
      for (int h = 0; h < H; ++h) x.v[u][t][h] = fast_exp2((x.v[u][t][h] - sh) * kLog2e);
    }
  }
}
// A wave's part of the maxima of b's columns into part[wave][64 H]; after a barrier item_cols_join has them.
template <int W, int U, int H>
__device__ __forceinline__ void item_cols_part(const ItemRows<W, U, H>& x, float* __restrict__ part, int wave, int lane) {
#pragma unroll
  for (int h = 0; h < H; ++h) {
    float m = x.v[0][0][h];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) m = item_max(m, x.v[u][t][h]);
    part[(wave * H + h) * 64 + lane] = m;
  }
}
template <int W, int H>
__device__ __forceinline__ void item_cols_join(const float* __restrict__ part, int lane, float (&be)[H]) {
#pragma unroll
  for (int h = 0; h < H; ++h) {
    be[h] = part[h * 64 + lane];
#pragma unroll
    for (int w = 1; w < W; ++w) be[h] = item_max(be[h], part[(w * H + h) * 64 + lane]);
  }
}
template <int W, int U, int H>
__device__ __forceinline__ void item_cols_exp(ItemRows<W, U, H>& x, const float (&be)[H]) {
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const float sh = be[h] == -INFINITY ? 0.f : be[h];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) x.v[u][t][h] = fast_exp2((x.v[u][t][h] - sh) * kLog2e);
  }
}

typedef float item_f4 __attribute__((ext_vector_type(4)));
// Four steps of a line: neighbours in LDS, or ld words apart.
__device__ __forceinline__ item_f4 item_frag(const float* p) { return *reinterpret_cast<const item_f4*>(p); }
__device__ __forceinline__ item_f4 item_frag(const float* p, int ld) {
  item_f4 r;
  r[0] = p[0]; r[1] = p[ld]; r[2] = p[2 * ld]; r[3] = p[3 * ld];
  return r;
}
// A 16 x 16 tile over `chunks` times 16 steps: result element r of lane (l15, q) is line 4 q + r of x,
// line l15 of y.  x(c), y(c): the lane's four steps 16 c + 4 q ... of its line l15 of either operand.
// (Which four steps an instruction sums is free as long as both operands agree.)
template <class X, class Y>
__device__ __forceinline__ item_f4 item_tile(int chunks, X&& x, Y&& y) {
  item_f4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
  item_f4 xv = x(0), yv = y(0);
  for (int c = 1; c <= chunks; ++c) {
    const int nx = c < chunks ? c : c - 1;
    const item_f4 xn = x(nx), yn = y(nx);
    c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[0], yv[0], c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[1], yv[1], c1, 0, 0, 0);
    c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[2], yv[2], c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[3], yv[3], c1, 0, 0, 0);
    xv = xn; yv = yn;
  }
  return c0 + c1;
}

// Tile `at`, at + step, ... of a list of rows of C tiles.
struct ItemTiles {
  int r, c, C;
  __device__ __forceinline__ ItemTiles(int at, int C_) : r(0), c(at), C(C_) { wrap(); }
  __device__ __forceinline__ void wrap() {
    while (c >= C) {
      c -= C;
      ++r;
    }
  }
  __device__ __forceinline__ void next(int step) {
    c += step;
    wrap();
  }
};

// The padded extents and LDS (floats) of an item.
struct ItemPad {
  int M, K, N;
};
__host__ __device__ inline ItemPad item_pad(int M, int K, int N) {
  return ItemPad{(M + 15) & ~15, (K + 15) & ~15, (N + 15) & ~15};
}
__host__ __device__ inline int item_bwd_arrays(int M, int K, int N) {
  const ItemPad p = item_pad(M, K, N);
  return p.K * (p.M + 4) + p.K * (p.N + 4) + p.M * (p.N + 4);
}
// (H: column chunks of N)
inline int item_fwd_floats(int M, int K, int N, int W, int H) {
  const ItemPad p = item_pad(M, K, N);
  return (p.M + p.N) * (p.K + 4) + W * H * 64 + p.M + p.N;
}
inline int item_bwd_floats(int M, int K, int N, int W, int H) {
  return item_bwd_arrays(M, K, N) + W * H * 64;
}

typedef elem_t item_e4 __attribute__((ext_vector_type(4), aligned(sizeof(elem_t))));

// R rows (row: their numbers; the last ones may repeat) of a 16-column tile the way the reference's kernel forms them
// (matmul_cuda_kernel.cu:27-41): running maximum from -1e9, then the sum.  The wave's lanes are the columns times
// quarters of 16 terms: of a row they read four neighbours at a time.  The reads and one exponential a term bound it.
// (500,96^3), 24 us where every cell factors: one such cell an item 26, nearly all cells 156 (each in the lane that found
// it, from memory: 52 and 1325); (512,128,100,64) 29, 33 and 214.  Nearly all cells of thin products cost more than
// tiles staged in LDS did ((512,100,40,100) 135 us, 93), the gradients then less (128, 135).
template <int R>
__device__ __forceinline__ void item_fwd_rows(const elem_t* __restrict__ ab, const elem_t* __restrict__ bb,
                                              elem_t* __restrict__ ob, const int (&row)[R], int n0, int M, int K, int N,
                                              int lane) {
  const int n = n0 + (lane & 15), q = lane >> 4;
  const elem_t* const bq = bb + min(n, N - 1);
  float mx[R], nm[R], s[R];
  auto walk = [&](auto add) __attribute__((always_inline)) {
    float t[R];
    int k0 = 0;
    for (; k0 + 16 <= K; k0 += 16) {
      item_e4 av[R];
      float bv[4];
#pragma unroll
      for (int r = 0; r < R; ++r) av[r] = *reinterpret_cast<const item_e4*>(ab + row[r] * K + k0 + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) bv[i] = (float)bq[(k0 + 4 * q + i) * N];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int r = 0; r < R; ++r) t[r] = (float)av[r][i] + bv[i];
        add(t);
      }
    }
    for (; k0 < K; k0 += 4) {
      const int k = min(k0 + q, K - 1);
      const float bv = (float)bq[k * N];
#pragma unroll
      for (int r = 0; r < R; ++r) t[r] = k0 + q < K ? (float)ab[row[r] * K + k] + bv : -INFINITY;
      add(t);
    }
  };
#pragma unroll
  for (int r = 0; r < R; ++r) {
    mx[r] = kFloor;
    s[r] = 0.f;
  }
  walk([&](const float (&t)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) mx[r] = fmaxf(mx[r], t[r]);
  });
#pragma unroll
  for (int r = 0; r < R; ++r) {
    mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], 16, 64));
    mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], 32, 64));
    nm[r] = -mx[r] * kLog2e;
  }
  walk([&](const float (&t)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] += fast_exp2(__builtin_fmaf(t[r], kLog2e, nm[r]));
  });
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s[r] += __shfl_xor(s[r], 16, 64);
    s[r] += __shfl_xor(s[r], 32, 64);
    if (q == 0 && n < N) ob[row[r] * N + n] = to_elem<elem_t>(logf(s[r]) + mx[r]);
  }
}

// W waves; UM, UK groups of four rows per wave (4 W UM >= M, 4 W UK >= K), HK, HN column chunks of 64 of K and N.
template <int W, int UM, int UK, int HK, int HN>
__global__ __launch_bounds__(64 * W, UM <= 2 && UK <= 2 ? 8 : W == 4 && UM == 3 ? 7 : 1) void k_log_item_fwd(const elem_t* __restrict__ a, const elem_t* __restrict__ b,
                                                         elem_t* __restrict__ out, float* __restrict__ stats,
                                                         int* __restrict__ hdr, int M, int K, int N) {
  extern __shared__ __attribute__((aligned(16))) float item_smem[];
  const ItemPad pad = item_pad(M, K, N);
  const int ldk = pad.K + 4;
  float* const Ea = item_smem;             // [m][k]
  float* const Eb = Ea + pad.M * ldk;      // [n][k]
  float* const part = Eb + pad.N * ldk;    // [wave][column]
  float* const s_al = part + W * HN * 64;
  float* const s_be = s_al + pad.M;
  const int tid = threadIdx.x;
  int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int batch = blockIdx.x;
  if (hdr && batch == 0 && tid == 0) hdr[0] = kWsNone;  // no per-tile flags in this workspace
  const elem_t* ab = a + (long)batch * M * K;
  const elem_t* bb = b + (long)batch * K * N;
  ItemRows<W, UM, HK> xa;
  ItemRows<W, UK, HN> xb;
  xa.load(ab, M, K, wave, lane);
  xb.load(bb, K, N, wave, lane);

  float al[UM][4], be[HN];
  xa.settle(K, lane);
  item_rows_exp(xa, al);
  xa.put_rows(Ea, ldk, pad.M, pad.K, wave, lane);
  xb.settle(N, lane);
  item_cols_part(xb, part, wave, lane);
  float* st = stats ? stats + (long)batch * (M + N) : nullptr;
  if (lane == 0) {
#pragma unroll
    for (int u = 0; u < UM; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int m = 4 * (wave + W * u) + t;
        if (m < pad.M) s_al[m] = al[u][t];
        if (st && m < M) st[m] = al[u][t];
      }
  }
  __syncthreads();
  item_cols_join<W, HN>(part, lane, be);
  item_cols_exp(xb, be);
  xb.put_cols(Eb, ldk, pad.K, pad.N, wave, lane);
  if (wave == 0) {
#pragma unroll
    for (int h = 0; h < HN; ++h) {
      const int n = lane + 64 * h;
      if (n < pad.N) s_be[n] = be[h];
      if (st && n < N) st[M + n] = be[h];
    }
  }
  __syncthreads();

  const int l15 = lane & 15, q4 = 4 * (lane >> 4);
  const int tm = pad.M >> 4, tn = pad.N >> 4, chunks = pad.K >> 4;
  const float thr = fast_exp2(-kItemGuardBits);
  elem_t* ob = out + (long)batch * M * N;
  int* const marks = reinterpret_cast<int*>(part) + 64 * HN * wave;  // of this wave's tiles: rows to be formed again
  unsigned flagged = 0;                                             // tiles with such rows
  ItemTiles w(wave, tn);
  for (int at = 0; w.r < tm; w.next(W), ++at) {  // uniform; at most 8 tiles
    const int m0 = w.r * 16, n0 = w.c * 16;
    const float* xl = Eb + (n0 + l15) * ldk + q4;
    const float* yl = Ea + (m0 + l15) * ldk + q4;
    const item_f4 s = item_tile(chunks, [&](int c) { return item_frag(xl + 16 * c); },
                                [&](int c) { return item_frag(yl + 16 * c); });
    const int m = m0 + l15, n = n0 + q4;
    const float am = s_al[m];
    const item_f4 bn = item_frag(s_be + n);
    float o[4];
    int redo = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float shift = am + bn[r];
      const bool ok = (s[r] >= thr) && (s[r] < INFINITY) && (shift >= kFloor) && (shift < INFINITY);
      if (!ok && m < M && n + r < N) redo |= 1 << r;
      o[r] = __builtin_fmaf(fast_log2(s[r]), kLn2, shift);
    }
    bool store = m < M;
    if (__builtin_amdgcn_ballot_w64(redo != 0) != 0) {  // rare
#pragma unroll
      for (int r = 0; r < 4; ++r)  // no term reaches the floor (a masked row or column), so none has mass beside it
        if (am + bn[r] <= kItemDead && s[r] >= 0.f) {
          o[r] = -INFINITY;
          redo &= ~(1 << r);
        }
      const unsigned long long cells = __builtin_amdgcn_ballot_w64(redo != 0);
      const int again = (int)((cells | cells >> 16 | cells >> 32 | cells >> 48) & 0xffff);
      marks[at] = again;
      flagged |= again != 0 ? 1u << at : 0u;
      store = store && !(again >> l15 & 1);
    }
    if (store) st4m(ob + m * N + n, N - n, make_float4(o[0], o[1], o[2], o[3]));
  }
  if (flagged) {  // uniform
    // (values of their own: nothing of this block is formed ahead of it)
    asm volatile("" : "+s"(M), "+s"(K), "+s"(N), "+v"(lane));
    for (; flagged; flagged &= flagged - 1) {
      const int i = __builtin_ctz(flagged), tile = wave + W * i, m0 = tile / tn * 16, n0 = (tile - tile / tn * tn) * 16;
      unsigned again = __builtin_amdgcn_readfirstlane(marks[i]);
      while (again) {  // uniform
        constexpr int R = UM <= 2 ? 2 : 4;  // (registers of eight waves a SIMD)
        if (__builtin_popcount(again) < R / 2 + 1) {
          const int row[1] = {m0 + __builtin_ctz(again)};
          again &= again - 1;
          item_fwd_rows<1>(ab, bb, ob, row, n0, M, K, N, lane);
        } else {
          int row[R];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            row[r] = again ? m0 + __builtin_ctz(again) : row[r > 0 ? r - 1 : 0];
            again &= again - 1;
          }
          item_fwd_rows<R>(ab, bb, ob, row, n0, M, K, N, lane);
        }
      }
    }
  }
}

// What marks a row or column to be formed again.  (Nothing clears the marks' place in LDS first: should what was there
// look like one, a row more is formed so.)
constexpr int kItemMark = 0x7fa5c3e1;

// The marks of `count` rows (columns) become the list of their numbers, in place; by one wave.  Returns how many.
__device__ __forceinline__ int item_list(int* __restrict__ marks, int count, int lane) {
  unsigned long long set[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    set[h] = __builtin_amdgcn_ballot_w64(lane + 64 * h < count && marks[min(lane + 64 * h, count - 1)] == kItemMark);
  const unsigned long long below = (1ULL << lane) - 1;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (set[h] >> lane & 1) marks[(h ? __builtin_popcountll(set[0]) : 0) + __builtin_popcountll(set[h] & below)] = lane + 64 * h;
  return __builtin_popcountll(set[0]) + __builtin_popcountll(set[1]);
}

// Gradients of listed rows (grad_a) and columns (grad_b) in the reference's form (matmul_cuda_kernel.cu:159-184),
// exp(a + b - out) * g summed over n and over m; Al [k][m], Bl [k][n] and Ol [m][n]: the operands and out in LDS.  A
// lane takes four rows m of a k, or four rows k of a column, over the whole list: 16 terms for every ten reads.
// One exponential a term bounds it.  Both gradients of (500,96^3), 48 us where every cell factors: one such cell an item
// 91, one masked row 162, nearly all cells 221 (the whole item again, every cell in a thread of its own that read all
// it needed from memory: 1480 each; by tiles staged in LDS 265 each); (2048,64^3) 53, then 116, 191 and 298 (1836).
template <int W>
__device__ __forceinline__ void item_bwd_exact(const elem_t* __restrict__ gb, const float* __restrict__ Al, int ldm,
                                               const float* __restrict__ Bl, int ldn, const float* __restrict__ Ol,
                                               const int* __restrict__ rows, int nr, const int* __restrict__ cols, int nc,
                                               elem_t* __restrict__ gab, elem_t* __restrict__ gbb, int M, int K, int N,
                                               int tid) {
  constexpr int R = 4;
  if (gab)
    for (int e = tid; e < (nr + R - 1) / R * K; e += 64 * W) {
      const int group = e / K, k = e - group * K;
      const float* bl = Bl + k * ldn;
      float av[R], s[R];
      int m[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        m[r] = rows[min(R * group + r, nr - 1)];
        av[r] = Al[k * ldm + m[r]];
        s[r] = 0.f;
      }
      int n = 0;
      for (; n + 3 < N; n += 4) {
        const item_f4 b4 = item_frag(bl + n);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const item_f4 o4 = item_frag(Ol + m[r] * ldn + n);
          const item_e4 g4 = *reinterpret_cast<const item_e4*>(gb + m[r] * N + n);
#pragma unroll
          for (int q = 0; q < 4; ++q) s[r] = __builtin_fmaf(fast_exp(av[r] + b4[q] - o4[q]), (float)g4[q], s[r]);
        }
      }
      for (; n < N; ++n)
#pragma unroll
        for (int r = 0; r < R; ++r)
          s[r] = __builtin_fmaf(fast_exp(av[r] + bl[n] - Ol[m[r] * ldn + n]), (float)gb[m[r] * N + n], s[r]);
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (R * group + r < nr) gab[m[r] * K + k] = to_elem<elem_t>(s[r]);
    }
  if (gbb)
    for (int e = tid; e < (K + R - 1) / R * nc; e += 64 * W) {
      const int group = e / nc, n = cols[e - group * nc];
      float bv[R], s[R];
      const float* al[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int k = min(R * group + r, K - 1);
        al[r] = Al + k * ldm;
        bv[r] = Bl[k * ldn + n];
        s[r] = 0.f;
      }
      int m = 0;
      for (; m + 3 < M; m += 4) {
        float ov[4], gv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          ov[q] = Ol[(m + q) * ldn + n];
          gv[q] = (float)gb[(m + q) * N + n];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const item_f4 a4 = item_frag(al[r] + m);
#pragma unroll
          for (int q = 0; q < 4; ++q) s[r] = __builtin_fmaf(fast_exp(a4[q] + bv[r] - ov[q]), gv[q], s[r]);
        }
      }
      for (; m < M; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r)
          s[r] = __builtin_fmaf(fast_exp(al[r][m] + bv[r] - Ol[m * ldn + n]), (float)gb[m * N + n], s[r]);
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (R * group + r < K) gbb[(R * group + r) * N + n] = to_elem<elem_t>(s[r]);
    }
}

template <int W, int UM, int UK, int HK, int HN>
__global__ __launch_bounds__(64 * W, UM <= 2 && UK <= 2 ? 8 : W == 8 && (UM == 3 || UM != UK) ? 4 : 1) void k_log_item_bwd(const elem_t* __restrict__ a, const elem_t* __restrict__ b,
                                                         const elem_t* __restrict__ outp, const elem_t* __restrict__ g,
                                                         elem_t* __restrict__ grad_a, elem_t* __restrict__ grad_b,
                                                         int M, int K, int N) {
  extern __shared__ __attribute__((aligned(16))) float item_smem[];
  const ItemPad pad = item_pad(M, K, N);
  const int ldm = pad.M + 4, ldn = pad.N + 4;
  float* const EaT = item_smem;           // [k][m]
  float* const Eb = EaT + pad.K * ldm;    // [k][n]
  float* const Hs = Eb + pad.K * ldn;     // [m][n]
  float* const part = Hs + pad.M * ldn;   // [wave][column]
  const int tid = threadIdx.x;
  int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int batch = blockIdx.x;
  const elem_t* ab = a + (long)batch * M * K;
  const elem_t* bb = b + (long)batch * K * N;
  const elem_t* ob = outp + (long)batch * M * N;
  const elem_t* gb = g + (long)batch * M * N;
  elem_t* gab = grad_a ? grad_a + (long)batch * M * K : nullptr;
  elem_t* gbb = grad_b ? grad_b + (long)batch * K * N : nullptr;
  ItemRows<W, UM, HK> xa;
  ItemRows<W, UK, HN> xb;
  ItemRows<W, UM, HN> xo, xg;
  xb.load(bb, K, N, wave, lane);
  xa.load(ab, M, K, wave, lane);
  xo.load(ob, M, N, wave, lane);
  xg.load(gb, M, N, wave, lane);

  float al[UM][4], be[HN];
  xb.settle(N, lane);
  item_cols_part(xb, part, wave, lane);
  xa.settle(K, lane);
  item_rows_exp(xa, al);
  xa.put_cols(EaT, ldm, pad.M, pad.K, wave, lane);
  __syncthreads();
  item_cols_join<W, HN>(part, lane, be);
  item_cols_exp(xb, be);
  xb.put_rows(Eb, ldn, pad.K, pad.N, wave, lane);
  // H, and whether the factoring is exact for every cell: S < 2^-40, NaN or infinities anywhere are not
  const float lim = kItemGuardBits * kLn2 + 1e-3f;
  float most = 0.f, worst = 0.f;  // worst stays 0 while every exponent is finite
#pragma unroll
  for (int h = 0; h < HN; ++h)
#pragma unroll
    for (int u = 0; u < UM; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bool in = 4 * (wave + W * u) + t < M && lane + 64 * h < N;
        const float ex = in ? al[u][t] + be[h] - (float)xo.raw[u][t][h] : 0.f;
        most = fmaxf(most, ex);
        worst = __builtin_fmaf(ex, 0.f, worst);
        xg.v[u][t][h] = (in ? (float)xg.raw[u][t][h] : 0.f) * fast_exp2(ex * kLog2e);
      }
  const int bad = !(most <= lim) || !(worst == 0.f);
  xg.put_rows(Hs, ldn, pad.M, pad.N, wave, lane);
  // Rows of grad_a and columns of grad_b that such a cell takes part in are formed again below, the rows together with
  // those of its wave; the others need none of its H.
  int* const rows = reinterpret_cast<int*>(part);  // marks, then lists (every wave has joined the columns' maxima)
  int* const cols = rows + 4 * W * UM;
  const int redo = __syncthreads_or(bad);
  if (redo) {  // rare
#pragma unroll
    for (int h = 0; h < HN; ++h)
      if (bad && lane + 64 * h < N) cols[lane + 64 * h] = kItemMark;
    const int m = 4 * (wave + W * (lane >> 2)) + (lane & 3);
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane < 4 * UM && m < M) rows[m] = kItemMark;
  }

  const int l15 = lane & 15, q4 = 4 * (lane >> 4);
  const int tk = pad.K >> 4, tn = pad.N >> 4, tm = pad.M >> 4;
  // grad_a's tiles, then grad_b's: a wave that is done with the former goes on in the latter's list
  ItemTiles w(wave, tk);
  if (gab) {
    for (; w.r < tm; w.next(W)) {  // uniform; four k of a row m: sum over n
      const int m0 = w.r * 16, k0 = w.c * 16;
      const float* xl = Eb + (k0 + l15) * ldn + q4;
      const float* yl = Hs + (m0 + l15) * ldn + q4;
      const item_f4 s = item_tile(tn, [&](int c) { return item_frag(xl + 16 * c); },
                                  [&](int c) { return item_frag(yl + 16 * c); });
      const int m = m0 + l15, k = k0 + q4;
      const item_f4 e = item_frag(EaT + k * ldm + m, ldm);
      if (m < M) st4m(gab + m * K + k, K - k, make_float4(e[0] * s[0], e[1] * s[1], e[2] * s[2], e[3] * s[3]));
    }
    w = ItemTiles((w.r - tm) * tk + w.c, tn);
  } else {
    w = ItemTiles(wave, tn);
  }
  if (gbb) {
    for (; w.r < tk; w.next(W)) {  // uniform; four n of a row k: sum over m
      const int k0 = w.r * 16, n0 = w.c * 16;
      const float* xl = Hs + q4 * ldn + n0 + l15;
      const float* yl = EaT + (k0 + l15) * ldm + q4;
      const item_f4 s = item_tile(tm, [&](int c) { return item_frag(xl + 16 * c * ldn, ldn); },
                                  [&](int c) { return item_frag(yl + 16 * c); });
      const int k = k0 + l15, n = n0 + q4;
      const item_f4 e = item_frag(Eb + k * ldn + n);
      if (k < K) st4m(gbb + k * N + n, N - n, make_float4(e[0] * s[0], e[1] * s[1], e[2] * s[2], e[3] * s[3]));
    }
  }
  if (redo) {
    // (values of their own: nothing of this block is formed ahead of it)
    asm volatile("" : "+s"(M), "+s"(K), "+s"(N), "+v"(lane), "+s"(wave));
    int* const counts = cols + 64 * HN;
    __syncthreads();  // the tiles' results are on their way, LDS is free
    if (wave < 2) {
      const int c = wave == 0 ? item_list(rows, M, lane) : item_list(cols, N, lane);
      if (lane == 0) counts[wave] = c;
    }
    xa.load(ab, M, K, wave, lane);
    xb.load(bb, K, N, wave, lane);
    xo.load(ob, M, N, wave, lane);
    xa.settle(K, lane);
    xa.put_cols(EaT, ldm, pad.M, pad.K, wave, lane);
    xb.settle(N, lane);
    xb.put_rows(Eb, ldn, pad.K, pad.N, wave, lane);
    xo.settle(N, lane);
    xo.put_rows(Hs, ldn, pad.M, pad.N, wave, lane);
    __syncthreads();
    item_bwd_exact<W>(gb, EaT, ldm, Eb, ldn, Hs, rows, counts[0], cols, counts[1], gab, gbb, M, K, N, tid);
  }
}

// ---------------------------------------------------------------- samplebmm's forward, extents of at most 64
// The vector-ALU sweep forms its targets from S = exp(out - alpha - beta), so the draws of a pinned (seed, offset)
// follow the last bit of `out`.  The sums of this forward are taken in the order of k, the one that those draws are
// defined by (in k_log_item_fwd's order one draw in some 10^5 moves to a neighbouring term); (2048,64^3) 44 us against
// 33 there.  TB x TB outputs per thread on a G x G thread grid, G = 16: TB = 2 covers items up to 32 x 32, TB = 4 up
// to 64 x 64.  FULL: M = K = N = G * TB, known to the compiler, whose index arithmetic is most of the instructions.
// (row, column) of elements tid, tid + nt, tid + 2 nt, ... of a row-major array
// with C columns, without a division per element.
struct RowMajorWalk {
  int r, c, dr, dc, C;
  __device__ __forceinline__ RowMajorWalk(int tid, int nt, int cols) : C(cols) {
    r = tid / C;
    c = tid - r * C;
    dr = nt / C;
    dc = nt - dr * C;
  }
  __device__ __forceinline__ void next() {
    r += dr;
    c += dc;
    if (c >= C) {
      c -= C;
      ++r;
    }
  }
};

template <int G, int TB, bool FULL = false>
__global__ __launch_bounds__(G * G, TB == 2 ? 8 : 1) void k_log_item_seq(const elem_t* __restrict__ a,
                                                      const elem_t* __restrict__ b,
                                                      elem_t* __restrict__ out,
                                                      float* __restrict__ stats,
                                                      int* __restrict__ hdr, int M_, int K_,
                                                      int N_) {
  constexpr int NT = G * G, S = G * TB, LD = S + 1;
  const int M = FULL ? S : M_, K = FULL ? S : K_, N = FULL ? S : N_;
  static_assert(2 * S <= NT, "row and column scans use 2*S threads");
  if (hdr && blockIdx.x == 0 && threadIdx.x == 0) hdr[0] = kWsNone;  // no per-tile flags in this workspace
  __shared__ float At[S * LD];  // [k][m]: a, then EA; finally the output tile [m][n]
  __shared__ float Bs[S * LD];  // [k][n]: b, then EB
  __shared__ float al[S], be[S];
  const int tid = threadIdx.x, batch = blockIdx.x;
  const elem_t* ab = a + (long)batch * M * K;
  const elem_t* bb = b + (long)batch * K * N;
  // All reads of the item are issued before the first one is waited for (a thread owns
  // elements tid, tid + NT, ... of each operand): one trip to memory, not one per element.
  constexpr int PER = TB * TB;  // S * S / NT
  float ra[PER], rb[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + u * NT;
    ra[u] = e < M * K ? ab[e] : 0.f;
    rb[u] = e < K * N ? bb[e] : 0.f;
  }
  {
    RowMajorWalk w(tid, NT, K);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (w.r < M) At[w.c * LD + w.r] = ra[u];
      w.next();
    }
  }
  {
    RowMajorWalk w(tid, NT, N);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (w.r < K) Bs[w.r * LD + w.c] = rb[u];
      w.next();
    }
  }
  __syncthreads();
  // row / column maxima: one thread per row, one per column (LDS atomics on the
  // shared maximum while loading measured slower: 32 lanes on one address)
  if (tid < M) {
    float mx = -INFINITY;
    for (int k = 0; k < K; ++k) mx = fmaxf(mx, At[k * LD + tid]);
    al[tid] = mx;
  } else if (tid >= S && tid - S < N) {
    float mx = -INFINITY;
    for (int k = 0; k < K; ++k) mx = fmaxf(mx, Bs[k * LD + tid - S]);
    be[tid - S] = mx;
  }
  __syncthreads();
  for (RowMajorWalk w(tid, NT, K); w.r < M; w.next()) {
    const int m = w.r, k = w.c;
    At[k * LD + m] = item_exp(At[k * LD + m], al[m]);
  }
  for (RowMajorWalk w(tid, NT, N); w.r < K; w.next()) {
    const int k = w.r, n = w.c, e = w.r * N + w.c;
    Bs[k * LD + n] = item_exp(Bs[k * LD + n], be[n]);
  }
  if (stats) {
    float* st = stats + (long)batch * (M + N);
    if (tid < M) st[tid] = al[tid];
    else if (tid >= S && tid - S < N) st[M + tid - S] = be[tid - S];
  }
  __syncthreads();

  const int ty = tid / G, tx = tid % G;
  float acc[TB][TB];
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) acc[i][j] = 0.f;
#pragma unroll 4
  for (int k = 0; k < K; ++k) {
    float av[TB], bv[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) av[i] = At[k * LD + ty * TB + i];
#pragma unroll
    for (int j = 0; j < TB; ++j) bv[j] = Bs[k * LD + tx * TB + j];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
      for (int j = 0; j < TB; ++j) acc[i][j] = __builtin_fmaf(av[i], bv[j], acc[i][j]);
  }
  __syncthreads();  // At becomes the output tile
  const float thr = fast_exp2(-kItemGuardBits);
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      const int m = ty * TB + i, n = tx * TB + j;
      if (m < M && n < N) {
        const float shift = al[m] + be[n], s = acc[i][j];
        const bool ok = (s >= thr) && (s < INFINITY) && (shift >= kFloor) && (shift < INFINITY);
        At[m * LD + n] = ok ? __builtin_fmaf(fast_log2(s), kLn2, shift)
                            : item_exact_out(ab + (long)m * K, bb + n, K, N);
      }
    }
  __syncthreads();
  elem_t* ob = out + (long)batch * M * N;
  for (RowMajorWalk w(tid, NT, N); w.r < M; w.next()) {
    const int m = w.r, n = w.c, e = w.r * N + w.c;
    ob[e] = to_elem<elem_t>(At[m * LD + n]);
  }
}

}  // namespace GENBMM_NS
