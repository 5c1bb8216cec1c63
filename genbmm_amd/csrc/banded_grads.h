// Both gradients of banded (+,*) products as block-banded matrix products on the matrix cores, operands staged
// through LDS as three bfloat16 parts (split_bf16.h): the plain product and the log product on the forward's
// workspace.  Same view of a band as a dense matrix as banded_block.h, the same staged form of a 32 x 32 block.
//
//   grad_b   R[y, z] = sum_x G[x, y] A[x, z]      s = x, lines = y     G[x, y] = g[x][y - x + r_lu]
//   grad_a   R[x, z] = sum_y G[x, y] B[y, z]      s = y, lines = x
//
// Either way a workgroup walks down 32-wide blocks of the reduction axis s.  Block s meets NP blocks of z (the other
// operand's rows s, a contiguous piece of memory) and NG blocks of lines (g's rows s for grad_b; for grad_a 32 columns
// of g, 128 contiguous bytes of each row, the next 128 a step later).  A block of the result, (z block Z, line block
// Z + d), takes its share of steps Z - NP + 1 ... Z and is complete then.  A wave keeps the accumulators of (Z, d) from
// the first of these steps to the last, writes them out and goes on with (Z + NP, d): nothing of an operand is needed for
// longer than one step, so LDS holds two steps' blocks and no ring of rows, which is what the 129 cells of a row of
// g would not leave room for.  NP + NG waves only stage, one block each, their loads two steps ahead; the
// others multiply (a step's products, NP ND of them, over up to eight waves) and write; one barrier per step.
//
// Every cell is staged times 2^26, which makes the three parts of any normal float exact (bfloat16 denormals start
// below 2^-126, a third part 24 bits below its value); sums leave times 2^-52.  What is not finite in a sum - an operand
// that is not, a part that overflowed (2^102), an H that is marked unusable - is recomputed by the per-cell routine.
// Rows of s beyond the matrix read as zeros (the buffer ends with the item); cells of g there meet those zeros.
//
// Measured, both gradients, against the memory-fed kernels (banded_direct.h), which walk 16-row tiles on the fp32 instruction
// with a trip to memory at either end of each: 64 x 4096, 65 diagonals per operand 215 -> 114 us (3.6 TB/s of 408 MB), the log
// product 245 -> 163, bfloat16 164 -> 90 and 225 -> 146; 49 diagonals 135 -> 94 and 165 -> 137; 33: 89 -> 66 and 120 -> 92;
// 8 x 2000, 65 diagonals, log 23.5 -> 19.8.  Error against float64 1.17e-7 (1.45e-7 before).  What bounds it: a step takes 1.67 us
// with eight blocks, of which staging fills about a third of the issue slots; the rest is memory, two steps of loads in flight.
#pragma once

#include "banded_block.h"

namespace GENBMM_NS {

constexpr int kGradProducers = 8;  // blocks of operands per step (and staging waves), at most
constexpr int kGradConsumers = 8;  // multiplying waves, at most
constexpr int kGradTasks = 2;      // blocks of results per multiplying wave, at most
constexpr int kGradBlockWords = 2 * kBlkSlabWords;
constexpr float kGradScale = 67108864.f;                      // 2^26
constexpr float kGradUnscale = 1.f / kGradScale / kGradScale;  // 2^-52

struct GradSide {
  int Wp, Wr;    // cells per row: of the operand beside g, of the result
  int lu_p;      // z = s - lu_p is the first column of the operand's row s
  int lo;        // lines of block s begin at 32 s - lo
  int NP, NG, ND;
  int z_lo, z_hi, z_per, chunks;  // blocks Z of an item, per workgroup, workgroups per item
  int consumers;
  long steps;  // the chip takes for both gradients
};

inline int grad_waves(const GradSide& g) { return g.consumers + g.NP + g.NG; }
inline size_t grad_lds_bytes(const GradSide& g) { return sizeof(unsigned) * 2 * kGradBlockWords * (size_t)(g.NP + g.NG); }
// grad_a: the operand beside g is b; grad_b: a.  lu_*: of that operand and of the result's band.
inline bool grad_side(GradSide& g, int lu_p, int Wp, int lo, int Wr, int Wo, int n, int B) {
  g.Wp = Wp; g.Wr = Wr; g.lu_p = lu_p; g.lo = lo;
  g.NP = (31 + Wp + 31) / 32;
  g.NG = (31 + Wo + 31) / 32;
  g.ND = (Wr - 1 + 31) / 32 + 1;
  const int tasks = g.NP * g.ND;
  if (g.NP + g.NG > kGradProducers || tasks > kGradTasks * kGradConsumers) return false;
  g.consumers = min(tasks, kGradConsumers);
  g.z_lo = lo / 32 - (g.ND - 1);
  g.z_hi = (n - 1 + lo) / 32;
  // One workgroup per compute unit.  Cut an item into the number of pieces that takes the chip the fewest steps:
  // rounds of workgroups times a piece's own blocks, those it walks for a neighbour's sake and its start.
  const int blocks = g.z_hi - g.z_lo + 1;
  int chunks = 1;
  long best = 0;
  for (int c = 1; c <= min(blocks, 256); ++c) {
    const long cost = ((2L * B * c + 255) / 256) * ((blocks + c - 1) / c + g.NP - 1 + 2);
    if (c == 1 || cost < best) {
      best = cost;
      chunks = c;
    }
  }
  g.steps = best;
  g.z_per = (blocks + chunks - 1) / chunks;
  g.chunks = (blocks + g.z_per - 1) / g.z_per;
  return true;
}
inline bool grad_plan(GradSide& ga, GradSide& gb, const BandArgs& p, int B) {
  const int a_ld = p.Wa - 1 - p.a_lu, b_ld = p.Wb - 1 - p.b_lu;
  return grad_side(ga, p.b_lu, p.Wb, a_ld + p.b_lu, p.Wa, p.Wo, p.n, B) &&
         grad_side(gb, p.a_lu, p.Wa, p.a_lu + b_ld, p.Wb, p.Wo, p.n, B) &&
         max(grad_lds_bytes(ga), grad_lds_bytes(gb)) <= kBlkLdsLimit && (long)p.n * p.Wo * 4 < (1L << 30) && p.n * p.Wo >= 4;
}

// Whether these kernels are the faster ones, in microseconds of the plain product: a step takes 0.2 a block and 0.03
// (measured 1.67 with 8 blocks, 1.38 with 7, 0.95 with 5, 0.81 with 4), the memory-fed kernels 1.45 a diagonal of the
// result at 64 x 4096 rows and 8 at the least.  (Both take 1.4 times that for the log product.)
inline bool grad_pays(const GradSide& ga, const GradSide& gb, const BandArgs& p, int B) {
  const int blocks = max(ga.NP + ga.NG, gb.NP + gb.NG);
  return max(ga.steps, gb.steps) * (0.2 * blocks + 0.03) < 1.45 * p.Wo * ((double)B * p.n / 262144.0) + 8.0;
}

// ------------------------------------------------------------------ staging
// Four or eight neighbouring steps of a line as the three planes' words.
__device__ __forceinline__ void grad_put4(unsigned* __restrict__ dst, float x0, float x1, float x2, float x3) {
  uintx2 h, m, l;
  unsigned a, b, c;
  split2(x0, x1, a, b, c);
  h.x = a; m.x = b; l.x = c;
  split2(x2, x3, a, b, c);
  h.y = a; m.y = b; l.y = c;
  *reinterpret_cast<uintx2*>(dst) = h;
  *reinterpret_cast<uintx2*>(dst + kBlkPlaneWords) = m;
  *reinterpret_cast<uintx2*>(dst + 2 * kBlkPlaneWords) = l;
}
__device__ __forceinline__ void grad_put8(unsigned* __restrict__ dst, const float (&x)[8]) {
  uintx4 h, m, l;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    unsigned a, b, c;
    split2(x[2 * q], x[2 * q + 1], a, b, c);
    h[q] = a; m[q] = b; l[q] = c;
  }
  *reinterpret_cast<uintx4*>(dst) = h;
  *reinterpret_cast<uintx4*>(dst + kBlkPlaneWords) = m;
  *reinterpret_cast<uintx4*>(dst + 2 * kBlkPlaneWords) = l;
}
// H = g / S (R = 1 / S; NaN where R is marked unusable), 0 outside the band
__device__ __forceinline__ float grad_h(float g, float r, unsigned inside) {
  float h = (g * kGradScale) * r;
  h = r < 0.f ? __builtin_nanf("") : h;
  return __uint_as_float(__float_as_uint(h) & inside);
}

// A staging wave's block whose rows of memory are steps of s (the operand beside g, and g for grad_b): two slabs of 16
// steps, a lane eight steps of one line of each, a load each (32 lanes read 128 contiguous bytes).
template <class E, bool HASR>
struct GradCols {
  struct Regs {
    E x[2][8];
    float r[HASR ? 2 : 1][HASR ? 8 : 1];
  };
  const E* src;       // of the item
  const float* rsrc;
  int W, steps;       // steps of 32 rows that hold rows of the matrix
  int cells;          // of the item
  int off[2][8];      // from the first cell of the step's first row
  unsigned in[2][8];  // HASR: inside the band (~0 or 0); else the factor kGradScale or 0
  unsigned* dst;
  __device__ __forceinline__ GradCols(const E* src_, const float* rsrc_, int W_, int n, int block, unsigned* lds, int lane)
      : src(src_), rsrc(rsrc_), W(W_), steps((n + 31) >> 5), cells(n * W_) {
    const int line = lane & 31, half = lane >> 5, col = 32 * block + line;
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ds = 16 * sl + 8 * half + e;
        const bool inside = (unsigned)(col - ds) < (unsigned)W;
        off[sl][e] = ds * (W - 1) + col;
        in[sl][e] = inside ? (HASR ? ~0u : __float_as_uint(kGradScale)) : 0u;
      }
    dst = lds + half * 128 + ((line ^ (half << 2)) << 2);
  }
  __device__ __forceinline__ void load(int s, Regs& v) const {
    // (the buffers begin with the step's first row and end with the item; steps without rows: empty)
    const bool any = s >= 0 && s < steps;
    const int first = any ? 32 * s * W : 0, left = any ? cells - first : 0;
    const buf_t bx = buf_of(src + first, (unsigned)(left * (int)sizeof(E)));
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int e = 0; e < 8; ++e) v.x[sl][e] = buf_ld<E>(bx, off[sl][e] * (int)sizeof(E), 0);
    if constexpr (HASR) {
      const buf_t br = buf_of(rsrc + first, (unsigned)(left * 4));
#pragma unroll
      for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int e = 0; e < 8; ++e) v.r[sl][e] = buf_ld<float>(br, off[sl][e] * 4, 0);
    }
  }
  __device__ __forceinline__ void stage(int, const Regs& v, unsigned buf) const {
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (HASR) x[e] = grad_h((float)v.x[sl][e], v.r[sl][e], in[sl][e]);
        else x[e] = (float)v.x[sl][e] * __uint_as_float(in[sl][e]);
      }
      grad_put8(dst + buf + sl * kBlkSlabWords, x);
    }
  }
};

// A staging wave's block of g for grad_a: s runs along the rows of memory, a line is a row.  Four neighbouring lanes take
// the 16 steps of a slab of one row (four steps each), the wave 16 rows at a time.
template <class E, bool HASR>
struct GradRows {
  struct Regs {
    float4 x[2][2], r[HASR ? 2 : 1][HASR ? 2 : 1];
  };
  const E* src;
  const float* rsrc;
  int W, last;         // the last cell to read four from
  int lowest, highest;  // of the block's offsets
  int off[2][2];       // from the first cell of row 32 s: [slab][rows]
  unsigned in[2][2][4];
  unsigned* dst;
  __device__ __forceinline__ GradRows(const E* src_, const float* rsrc_, int W_, int n, int lo, int block, unsigned* lds,
                                      int lane)
      : src(src_), rsrc(rsrc_), W(W_), last(n * W_ - 4) {
    const int quad = lane & 3;
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int line = (lane >> 2) + 16 * u, ds = 16 * sl + 4 * quad, cell = ds + W - 1 - 32 * block - line;
        off[sl][u] = (32 * block + line - lo) * W + cell;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          in[sl][u][e] = (unsigned)(cell + e) < (unsigned)W ? (HASR ? ~0u : __float_as_uint(kGradScale)) : 0u;
      }
    lowest = (32 * block - lo) * W + W - 1 - 32 * block;
    highest = lowest + 31 * (W - 1) + 28;
    // (lines of the second half of a slab's steps swapped in fours, as blk_frag reads them; 16 u keeps the swap)
    dst = lds + (quad >> 1) * 128 + (((lane >> 2) ^ ((quad >> 1) << 2)) << 2) + (quad & 1) * 2;
  }
  __device__ __forceinline__ void load(int s, Regs& v) const {
    const int first = 32 * s * W;
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const unsigned at = (unsigned)min(max(first + off[sl][u], 0), last);
        v.x[sl][u] = ld4(src + at);
        if constexpr (HASR) v.r[sl][u] = ld4(rsrc + at);
      }
  }
  // a piece as it was meant, from what was read `shift` cells before it (cells that were not read lie outside the item)
  static __device__ __forceinline__ float4 moved(float4 v, int shift) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = 0.f;
#pragma unroll
      for (int f = 0; f < 4; ++f) y[e] = f - e == shift ? x[f] : y[e];
    }
    return make_float4(y[0], y[1], y[2], y[3]);
  }
  __device__ __forceinline__ void stage(int s, const Regs& v, unsigned buf) const {
    const int first = 32 * s * W;
    const bool plain = first + lowest >= 0 && first + highest <= last;  // uniform
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float4 x = v.x[sl][u], r = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (HASR) r = v.r[sl][u];
        if (!plain) {
          const int at = first + off[sl][u], shift = at - min(max(at, 0), last);
          x = moved(x, shift);
          if constexpr (HASR) r = moved(r, shift);
        }
        const unsigned(&m)[4] = in[sl][u];
        if constexpr (HASR) x = make_float4(grad_h(x.x, r.x, m[0]), grad_h(x.y, r.y, m[1]), grad_h(x.z, r.z, m[2]), grad_h(x.w, r.w, m[3]));
        else x = make_float4(x.x * __uint_as_float(m[0]), x.y * __uint_as_float(m[1]), x.z * __uint_as_float(m[2]), x.w * __uint_as_float(m[3]));
        grad_put4(dst + buf + sl * kBlkSlabWords + 64 * u, x.x, x.y, x.z, x.w);
      }
  }
};

// The staging waves' walk over steps [s0, s1): loads two steps ahead, a step staged while the one before is multiplied.
template <class Block>
__device__ __forceinline__ void grad_produce(const Block& b, int s0, int s1, unsigned buf_words) {
  typename Block::Regs v0, v1;
  b.load(s0, v0);
  b.load(s0 + 1, v1);
  b.stage(s0, v0, 0u);
  __syncthreads();
  int s = s0;
  for (; s + 1 < s1; s += 2) {  // (steps beyond the last are staged where no step looks any more)
    b.load(s + 2, v0);
    b.stage(s + 1, v1, buf_words);
    __syncthreads();
    b.load(s + 3, v1);
    b.stage(s + 2, v0, 0u);
    __syncthreads();
  }
  if (s < s1) __syncthreads();
}

// ------------------------------------------------------------------ products
template <bool PREP, bool GA>
__device__ __forceinline__ void grad_consume(const BandArgs& p, const GradSide& g, long bn, int wave, int lane, int s0, int s1,
                                             int z0, const unsigned* lds, unsigned buf_words) {
  // the multiplying waves are what a step waits for: they issue ahead of the staging waves
  __builtin_amdgcn_s_setprio(3);
  const int n = p.n, Wr = g.Wr, col = lane & 31, hi32 = lane >> 5;
  const int frag_off = hi32 * 128 + ((col ^ (hi32 << 2)) << 2);  // the lane's 16 bytes of a plane
  const int tasks = wave < g.consumers ? (g.NP * g.ND - wave + g.consumers - 1) / g.consumers : 0;
  constexpr int ES = sizeof(elem_t);
  const buf_t dst = buf_of((GA ? p.o0 : p.o1) + bn * Wr, (unsigned)(n * Wr * ES));
  const buf_t fac = buf_of(PREP ? (GA ? p.ws_ea : p.ws_eb) + bn * Wr : nullptr, PREP ? (unsigned)(n * Wr * 4) : 0u);
  int d[kGradTasks], turn[kGradTasks];  // turn: the block of z that (Z, d) is at this step
  floatx16 acc[kGradTasks];
#pragma unroll
  for (int k = 0; k < kGradTasks; ++k) {
    const int t = wave + k * g.consumers;
    d[k] = t % g.ND;
    turn[k] = ((t / g.ND - s0) % g.NP + g.NP) % g.NP;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
  }
  const int lane_cell = 4 * hi32 * (Wr - 1) + col;
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const unsigned* buf = lds + ((s - s0) & 1) * buf_words + frag_off;
#pragma unroll
    for (int k = 0; k < kGradTasks; ++k) {
      if (k >= tasks) break;  // uniform
      const int i = turn[k], j = i + d[k];
      const bool done = i == 0;
      // element e of the finished block: line row(e) = 4 hi32 + 8 (e / 4) + e % 4 of the block, cell Wr - 1 - 32 d + col - row(e)
      const int l0 = 32 * (s + d[k]) - g.lo, cell0 = Wr - 1 - 32 * d[k] + col - 4 * hi32;
      const int first = l0 * Wr + Wr - 1 - 32 * d[k];
      const bool whole = 32 * d[k] + 31 <= Wr - 1 && 32 * d[k] - 31 >= 0;  // uniform: every cell is one of the band
      auto at = [&](int e) __attribute__((always_inline)) {  // cell of the item; -1: none
        const int ru = 8 * (e >> 2) + (e & 3), o = lane_cell + (first + ru * (Wr - 1));
        return whole || (unsigned)(cell0 - ru) < (unsigned)Wr ? o : -1;
      };
      float f[16];
      if (PREP && done) {
#pragma unroll
        for (int e = 0; e < 16; ++e) f[e] = buf_ld<float>(fac, at(e) << 2, 0);
      }
      if (j < g.NG) {
        const unsigned* gl = buf + j * kGradBlockWords;
        const unsigned* pl = buf + (g.NG + i) * kGradBlockWords;
        BlkFrags f0, f1;
        f0.read(gl, pl);
        f1.read(gl + kBlkSlabWords, pl + kBlkSlabWords);
        f0.mul(acc[k], acc[k]);
        f1.mul(acc[k], acc[k]);
      }
      turn[k] = done ? g.NP - 1 : i - 1;
      if (!done) continue;
      if (s >= z0) {  // (before: a block of the workgroup above)
        const bool z_in = (unsigned)(32 * s - g.lu_p + col) < (unsigned)n;
        float worst = 0.f;  // stays 0 while every sum is finite
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float v = acc[k][e] * kGradUnscale;
          worst = __builtin_fmaf(v, 0.f, worst);  // 0 * v is NaN exactly when v is not finite
          if (PREP) v *= f[e];
          v = z_in ? v : 0.f;  // outside the matrix: the reference's zero fill
          buf_st(dst, at(e) * ES, to_elem<elem_t>(v));
        }
        if (!(worst == 0.f)) {  // rare: those sums alone; the stores above came from this lane: they stay in order
          unsigned bad = 0;
#pragma unroll
          for (int e = 0; e < 16; ++e) bad |= acc[k][e] * kGradUnscale * 0.f == 0.f ? 0u : 1u << e;
          for (; bad; bad &= bad - 1) {
            const int e = __builtin_ctz(bad);
            const int ro = 8 * (e >> 2) + 4 * hi32 + (e & 3), line = l0 + ro, cell = Wr - 1 - 32 * d[k] + col - ro;
            if ((unsigned)line < (unsigned)n && (unsigned)cell < (unsigned)Wr) {
              constexpr int MODE = PREP ? GENBMM_BAND_LOG : GENBMM_BAND_MUL;
              if (GA) band_bwd_a_cell<MODE>(p, bn + line, line, cell);
              else band_bwd_b_cell<MODE>(p, bn + line, line, cell);
            }
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
    }
    __syncthreads();
  }
}

// GA: grad_a; the workgroup `blk` of that gradient
template <bool PREP, bool GA>
__device__ __forceinline__ void grad_block(const BandArgs& p, const GradSide& g, int blk, unsigned* lds) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int batch = blk / g.chunks, n = p.n;
  const long bn = (long)batch * n;
  const int z0 = g.z_lo + (blk - batch * g.chunks) * g.z_per, s1 = min(z0 + g.z_per, g.z_hi + 1), s0 = z0 - (g.NP - 1);
  const unsigned buf_words = (unsigned)((g.NP + g.NG) * kGradBlockWords);
  const int prod = wave - g.consumers;
  if (prod >= 0 && prod < g.NG + g.NP) {
    unsigned* mine = lds + prod * kGradBlockWords;
    if (prod < g.NG) {
      if constexpr (GA) grad_produce(GradRows<elem_t, PREP>(p.g + bn * p.Wo, PREP ? p.ws_r + bn * p.Wo : nullptr, p.Wo, n, g.lo, prod, mine, lane), s0, s1, buf_words);
      else grad_produce(GradCols<elem_t, PREP>(p.g + bn * p.Wo, PREP ? p.ws_r + bn * p.Wo : nullptr, p.Wo, n, prod, mine, lane), s0, s1, buf_words);
    } else if constexpr (PREP) {
      grad_produce(GradCols<float, false>((GA ? p.ws_eb : p.ws_ea) + bn * g.Wp, nullptr, g.Wp, n, prod - g.NG, mine, lane), s0, s1, buf_words);
    } else {
      grad_produce(GradCols<elem_t, false>((GA ? p.b : p.a) + bn * g.Wp, nullptr, g.Wp, n, prod - g.NG, mine, lane), s0, s1, buf_words);
    }
  } else {
    grad_consume<PREP, GA>(p, g, bn, prod < 0 ? wave : g.consumers, lane, s0, s1, z0, lds, buf_words);
  }
}

// A workgroup of grad_a and one of grad_b in turn: those of one item read the same rows of g, neighbours on one XCD.
template <bool PREP>
__global__ __launch_bounds__(64 * (kGradProducers + kGradConsumers)) void k_band_blk_grads(const BandArgs p, const GradSide ga,
                                                                                          const GradSide gb, int na, int nb) {
  extern __shared__ __attribute__((aligned(16))) unsigned blk_smem[];
  const int v = xcd_renumber(blockIdx.x, na + nb), both = 2 * min(na, nb);
  const bool first = v < both ? (v & 1) == 0 : na > nb;
  const int blk = v < both ? v >> 1 : v - both / 2;
  if (first) grad_block<PREP, true>(p, ga, blk, blk_smem);
  else grad_block<PREP, false>(p, gb, blk, blk_smem);
}

}  // namespace GENBMM_NS
