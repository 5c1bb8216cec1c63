// Backward of the banded max product as two scatters: every output cell (i, j)
// hands its incoming gradient to the one a-cell and the one b-cell its argmax
// names, so the work is one pass over g and idx (n * Wo cells per batch item)
// instead of one pass per gradient cell.
//
//   grad_a[i, k]  += g[i, j]   for k  = idx[i, j],                 j ascending
//   grad_b[o, k2] += g[i, j]   for k2 = idx[i, j] - j + Wb - 1,    i ascending
//                                    (o = i + j - r_lu, i.e. j descending)
//
// which are the reference's summation orders (banded_cuda_kernel.cu:104-152 and
// the transposed call of sparse.py:625-635), so the sums come out bit for bit.
// Cells outside the matrix carry index 0 from the forward and are masked here.
//
// A workgroup is one wave on 64 rows of one gradient and up to kArgKC of its diagonals (wider bands:
// further workgroups, each walking only the j that can meet its diagonals).  A lane owns a row and walks
// its cells in that order, accumulating in LDS at [k][lane]: whatever k each lane adds to, the 64 lanes
// stay in 64 different banks, and no cell is shared, so there is no barrier.  grad_b's lanes, at one i,
// take 64 adjacent cells of row i straight from memory; grad_a's cells pass through a tile of LDS (lanes
// that read their own rows fetch a cache line for every 16 bytes: 220 us).  The next chunks are in flight
// while one is added, and no load stands under a branch: behind one the compiler waits for every load.
// Both gradients are one launch, strip by strip, so that the second use of g and idx comes from a cache.
//
// g and idx once and both gradients are 406 MB at 64 x 4096, 65 diagonals each: 180 -> 149 us there (behind a
// forward, as a step runs them).  Of the 31, 7 are addresses and slots that no longer follow clamped rows (grad_b), the rest
// pieces of four cells a load and a store (grad_a) and results that leave as one run instead of 32 diagonals at a time.
// What it waits for now: timed in parts, 55 us are the walk over LDS without loads, additions and results; the ordered
// additions (add4_ordered: one LDS round trip per four cells) and the loads then share two waves a SIMD, which LDS
// bounds.  More loads in flight change nothing; chunks of 8 cells in grad_a, whose tile would leave room for an eighth wave on
// a compute unit, 172 us, of 32 185 (five waves); of 8 rows in grad_b 153, of 4 about 10 more.
#pragma once

#include "banded_cells.h"

namespace GENBMM_NS {

constexpr int kArgRows = 64;  // rows per workgroup: the lanes
constexpr int kArgKC = 128;   // diagonals per workgroup
constexpr int kArgCh = 16;    // cells of a row per chunk (grad_a)
constexpr int kArgChB = 16;   // rows per chunk (grad_b)

// diagonals of a gradient per workgroup, and the workgroups that all W of them take
inline int argmax_kw(int W) { return min(W, kArgKC); }
inline int argmax_parts(int W) { return (W + kArgKC - 1) / kArgKC; }
// the cells and one spare cell per lane (terms that are not the lane's); grad_a: the tile
__host__ __device__ inline int argmax_cells(int kw) { return kArgRows * (kw + 1); }
inline size_t argmax_bwd_bytes(int Wa, int Wb) {
  return max(sizeof(float) * (argmax_cells(argmax_kw(Wa)) + kArgRows * kArgCh) + kArgRows * kArgCh,
             sizeof(float) * (size_t)argmax_cells(argmax_kw(Wb)));
}

typedef int arg_i4 __attribute__((ext_vector_type(4), aligned(4)));
typedef elem_t arg_e4 __attribute__((ext_vector_type(4), aligned(sizeof(elem_t))));
struct ArgRowChunk {  // four cells of each of four rows
  arg_i4 i[4];
  arg_e4 g[4];
};
struct ArgColChunk {  // one cell of each of CH rows
  static constexpr int CH = kArgChB;
  int i[CH];
  elem_t g[CH];
};

// Compiler-level ordering point for a wave's own LDS traffic (one wave's LDS instructions execute in order).
__device__ __forceinline__ void argmax_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The lane's cells cleared, then `chunks` chunks: load(chunk, number), slots(chunk, number, cells' numbers, values)
template <class Chunk, class Load, class Slots>
__device__ __forceinline__ void argmax_walk(float* __restrict__ accs, int kw, int chunks, Load load, Slots slots) {
  constexpr int CH = Chunk::CH;
  const int lane = threadIdx.x;
  // Two chunks, 2 x 32 loads, ahead: about the 63 that a wave can leave in flight.  (A third's wait took part of the second
  // with it, and its registers: 64 x 4096 with 5 diagonals an operand 29 us for 25, bfloat16 33 57 for 53, 65 the same;
  // one ahead is slower from 17 on, 65 138 us for 131.)
  Chunk v0, v1, v2;
  auto add = [&](const Chunk& ch, int c) __attribute__((always_inline)) {
    if (c >= chunks) return;  // uniform
    unsigned kr[CH];
    float tv[CH];
    slots(ch, c, kr, tv);
#pragma unroll
    for (int q = 0; q < CH; q += 4) {
      const unsigned k4[4] = {kr[q], kr[q + 1], kr[q + 2], kr[q + 3]};
      const float t4[4] = {tv[q], tv[q + 1], tv[q + 2], tv[q + 3]};
      add4_ordered(accs + lane, k4, t4);
    }
  };
  if (chunks > 0) {
    load(v0, 0);
    load(v1, 1);
  }
#pragma unroll 16
  for (int k = 0; k <= kw; ++k) accs[k * kArgRows + lane] = 0.f;
  for (int c = 0; c < chunks; c += 3) {
    load(v2, c + 2);
    add(v0, c);
    load(v0, c + 3);
    add(v1, c + 1);
    load(v1, c + 4);
    add(v2, c + 2);
  }
}

// The sums leave as rows: they change places in LDS, through registers, from [k][lane] to [row][k], rows an odd number
// of cells apart, and where a row has no other diagonals go to memory as the one run that they are there, 16 bytes a
// lane.  (Runs of 32 diagonals, each in its own pass over the rows: a third of the kernel's time.)
__device__ __forceinline__ void argmax_write_out(float* __restrict__ accs, int kw, elem_t* __restrict__ out, int W,
                                                 int rows) {
  const int lane = threadIdx.x, pitch = kw | 1;
  float v[kArgKC];
  argmax_lds_sync();
#pragma unroll
  for (int k0 = 0; k0 < kArgKC; k0 += 32)
    if (k0 < kw) {  // uniform
#pragma unroll
      for (int q = k0; q < k0 + 32; ++q) v[q] = accs[min(q, kw - 1) * kArgRows + lane];
    }
  argmax_lds_sync();
#pragma unroll
  for (int k0 = 0; k0 < kArgKC; k0 += 32)
    if (k0 < kw) {
#pragma unroll
      for (int q = k0; q < k0 + 32; ++q) accs[lane * pitch + min(q, kw - 1)] = v[q];  // (beyond kw: the last again)
    }
  argmax_lds_sync();
  const int cells = rows * kw;
  // e < 2^13: e / kw = e inv / 2^32 (kw > 1).  Rows of even length have a gap behind each.
  const unsigned inv = 0xffffffffu / (unsigned)kw + 1, gaps = (kw & 1) ? 0u : inv;
  if (W == kw) {  // uniform
    int e = 4 * lane;
#pragma unroll 4
    for (; e + 3 < cells; e += 256) {
      float4 x;
      if (kw & 1) {  // uniform
        x = *reinterpret_cast<const float4*>(accs + e);
      } else {
        const int r = (int)__umulhi(e, gaps), c = e - r * kw;
        const float* s = accs + e + r;
        x = make_float4(s[0], s[1 + (c + 1 >= kw)], s[2 + (c + 2 >= kw)], s[3 + (c + 3 >= kw)]);
      }
      arg_e4 y;
      y[0] = to_elem<elem_t>(x.x); y[1] = to_elem<elem_t>(x.y); y[2] = to_elem<elem_t>(x.z); y[3] = to_elem<elem_t>(x.w);
      *reinterpret_cast<arg_e4*>(out + e) = y;
    }
    for (int t = (cells & ~3) + lane; t < cells; t += 64) out[t] = to_elem<elem_t>(accs[t + (int)__umulhi(t, gaps)]);
  } else {
    for (int e = lane; e < cells; e += 64) {
      const int r = kw == 1 ? e : (int)__umulhi(e, inv);
      out[(long)r * W + e - r * kw] = to_elem<elem_t>(accs[r * pitch + e - r * kw]);
    }
  }
}

// grad_a, rows [i0, i0 + 64), diagonals [w0, w0 + kw).  A lane loads four cells of a row, four lanes the sixteen
// of a chunk; their terms and the cells they go to (a byte: kw <= 128 marks the spare) change places to the
// lane of their row through a tile of LDS (pieces of four turned by their row: sixteen lanes meet all banks either
// way).  Loads three chunks ahead.  NARROW: rows shorter than a chunk, read cell by cell.
template <bool NARROW>
__device__ __forceinline__ void argmax_band_a(float* __restrict__ accs, const BandArgs& p, int batch, int i0, int w0) {
  const int n = p.n, Wa = p.Wa, Wb = p.Wb, Wo = p.Wo, lane = threadIdx.x;
  const int kw = min(kArgKC, Wa - w0);
  float* const gt = accs + argmax_cells(kw);
  unsigned* const st = reinterpret_cast<unsigned*>(gt + kArgRows * kArgCh);
  const int jlo = w0, jhi = min(w0 + kw - 1 + Wb - 1, Wo - 1);  // cells with a term on these diagonals
  const int lr = lane >> 2, lq = lane & 3;
  const long base = ((long)batch * n + i0) * Wo;
  const elem_t* gb = p.g + base;
  const int32_t* ib = p.idx + base;
  const int last = n - 1 - i0;  // rows behind the matrix re-read its last row (nothing of them is stored)
  // every cell of the strip inside the matrix: o = i + j - r_lu in [0, n)
  const bool inner = i0 >= p.r_lu && (long)i0 + kArgRows - 1 + Wo - 1 - p.r_lu < n;
  ArgRowChunk x, y, z;
  long row[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) row[u] = (long)min(16 * u + lr, last) * Wo + (NARROW ? 0 : 4 * lq);
  // the last chunk of a row starts inside the row, the cells that the chunk before it held are masked
  auto start = [&](int j0) __attribute__((always_inline)) { return max(min(j0, Wo - kArgCh), 0); };
  auto load = [&](ArgRowChunk& v, int j0) __attribute__((always_inline)) {
    const elem_t* gs = gb + start(j0);
    const int32_t* is = ib + start(j0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (NARROW) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = min(4 * lq + e, Wo - 1);
          v.g[u][e] = gs[row[u] + j];
          v.i[u][e] = is[row[u] + j];
        }
      } else {
        // (a chunk past the band asks for one line: every row's last cells again cost 14 us of 83 with 33 diagonals an
        // operand, 7 of 139 with 65)
        const long at = j0 <= jhi ? row[u] : 0;
        v.g[u] = *reinterpret_cast<const arg_e4*>(gs + at);
        v.i[u] = *reinterpret_cast<const arg_i4*>(is + at);
      }
    }
  };
  float4* const gput = reinterpret_cast<float4*>(gt) + lr * 4 + (lq ^ (lr >> 2 & 3));  // (16 u keeps the turn)
  const float4* const gget = reinterpret_cast<const float4*>(gt) + lane * 4;
  auto stage = [&](const ArgRowChunk& v, int j0) __attribute__((always_inline)) {
    argmax_lds_sync();  // the tile has been read
    const bool whole = inner && j0 + kArgCh <= Wo && j0 + kArgCh - 1 <= jhi;  // uniform: sixteen new cells of every row
    const int j = start(j0) + 4 * lq, o = i0 + lr + j - p.r_lu;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      gput[64 * u] = make_float4((float)v.g[u][0], (float)v.g[u][1], (float)v.g[u][2], (float)v.g[u][3]);
      unsigned k[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) k[e] = min((unsigned)(v.i[u][e] - w0), (unsigned)kw);
      if (!whole) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned lim = j + e >= j0 && j + e <= jhi ? n : 0;
          k[e] = (unsigned)(o + 16 * u + e) < lim ? k[e] : kw;
        }
      }
      st[64 * u + lane] = k[0] | k[1] << 8 | k[2] << 16 | k[3] << 24;
    }
    argmax_lds_sync();
  };
  auto add = [&]() __attribute__((always_inline)) {
    float4 t[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) t[q] = gget[q ^ (lane >> 2 & 3)];
    const uint4 w4 = reinterpret_cast<const uint4*>(st)[lane];
    const unsigned w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned k4[4] = {w[q] & 255, w[q] >> 8 & 255, w[q] >> 16 & 255, w[q] >> 24};
      const float t4[4] = {t[q].x, t[q].y, t[q].z, t[q].w};
      add4_ordered(accs + lane, k4, t4);
    }
  };
  auto turn = [&](ArgRowChunk& v, int j0) __attribute__((always_inline)) {
    if (j0 <= jhi) stage(v, j0);  // uniform
    load(v, j0 + 3 * kArgCh);
    if (j0 <= jhi) add();
  };
  if constexpr (NARROW) {  // one chunk
    load(x, 0);
#pragma unroll 16
    for (int k = 0; k <= kw; ++k) accs[k * kArgRows + lane] = 0.f;
    stage(x, 0);
    add();
    argmax_write_out(accs, kw, p.o0 + ((long)batch * n + i0) * Wa + w0, Wa, min(kArgRows, n - i0));
    return;
  }
  // (in this order, as the loop's: the waits for x in its first turn are those of every turn)
  load(x, jlo);
  __builtin_amdgcn_sched_barrier(0);
  load(y, jlo + kArgCh);
  __builtin_amdgcn_sched_barrier(0);
  load(z, jlo + 2 * kArgCh);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll 16
  for (int k = 0; k <= kw; ++k) accs[k * kArgRows + lane] = 0.f;
  for (int j0 = jlo; j0 <= jhi; j0 += 3 * kArgCh) {
    turn(x, j0);
    turn(y, j0 + kArgCh);
    turn(z, j0 + 2 * kArgCh);
  }
  argmax_write_out(accs, kw, p.o0 + ((long)batch * n + i0) * Wa + w0, Wa, min(kArgRows, n - i0));
}

// grad_b, rows [o0, o0 + 64), diagonals [w0, w0 + kw).  A lane's cell of row i is j = o - i + r_lu, one less a row
// further down: in memory row i + 1's lies Wo - 1 cells behind row i's for every lane, so a chunk's addresses are
// a base and offsets that never change.  A lane whose j lies outside the row reads a cell of a row t before or
// behind; k2 of that cell, in [0, Wb) or none, is t Wo away from what its index says for this lane, and Wo >= Wb.
// (Formed from clamped j and row numbers, addresses and slots took 25 of a cell's 34 instructions, now 8 of 17.)
__device__ __forceinline__ void argmax_band_b(float* __restrict__ accs, const BandArgs& p, int batch, int o0, int w0) {
  constexpr int ES = sizeof(elem_t);
  const int n = p.n, Wa = p.Wa, Wb = p.Wb, Wo = p.Wo, lane = threadIdx.x;
  const int kw = min(kArgKC, Wb - w0);
  const elem_t* gb = p.g + (long)batch * n * Wo;
  const int32_t* ib = p.idx + (long)batch * n * Wo;
  // cells with a term on these diagonals, and the rows i that hold them for some lane
  const int jlo = max(0, Wb - w0 - kw), jhi = min(Wo - 1, Wa + Wb - 2 - w0);
  const int ilo = max(0, o0 + p.r_lu - jhi), ihi = min(n - 1, o0 + kArgRows - 1 + p.r_lu - jlo);
  const int jof = o0 + lane + p.r_lu;  // j = jof - i
  const int rows = Wo < (1 << 25) ? kArgChB : 1;  // of a chunk: its offsets fit 32 bits (cells behind them read as 0)
  int off[kArgChB];
#pragma unroll
  for (int q = 0; q < kArgChB; ++q) off[q] = q < rows ? lane + q * (Wo - 1) : -16;
  const int chunks = ihi < ilo ? 0 : (ihi - ilo + rows) / rows;
  argmax_walk<ArgColChunk>(
      accs, kw, chunks,
      [&](ArgColChunk& x, int c) __attribute__((always_inline)) {
        // lane 0's cell of the chunk's first row; the buffers end with the item, a chunk past the rows has none
        const long first = (long)(ilo + min(c, chunks - 1) * rows) * (Wo - 1) + (o0 + p.r_lu);
        const unsigned left = c < chunks ? (unsigned)min((long)n * Wo - first, 1L << 29) : 0;
        const buf_t bi = buf_of(ib + first, left * 4), bg = buf_of(gb + first, left * ES);
#pragma unroll
        for (int q = 0; q < kArgChB; ++q) {
          x.i[q] = buf_ld<int32_t>(bi, off[q] * 4, 0);
          x.g[q] = buf_ld<elem_t>(bg, off[q] * ES, 0);
        }
      },
      [&](const ArgColChunk& x, int c, unsigned (&kr)[kArgChB], float (&tv)[kArgChB]) __attribute__((always_inline)) {
        const unsigned at = (unsigned)(Wb - 1 - w0 + ilo + c * rows) - (unsigned)jof;
#pragma unroll
        for (int q = 0; q < kArgChB; ++q) {
          // An index is a k of its cell, 0 (a cell outside the matrix) or -1 (no term; becomes far too
          // large).  What lies behind the item reads as 0, a term of 0 wherever it falls.
          kr[q] = min(((unsigned)x.i[q] & 0x7fffffffu) + (at + q), (unsigned)kw);  // kw: the spare cells
          tv[q] = (float)x.g[q];
        }
      });
  argmax_write_out(accs, kw, p.o1 + ((long)batch * n + o0) * Wb + w0, Wb, min(kArgRows, n - o0));
}

__global__ __launch_bounds__(64) void k_band_argmax_bwd(const BandArgs p, int strips, int parts_a, int parts_b) {
  extern __shared__ __attribute__((aligned(16))) float accs[];
  const int parts = parts_a + parts_b, wg = xcd_renumber(blockIdx.x, gridDim.x);
  const int strip = wg / parts, part = wg - strip * parts;
  const int batch = strip / strips, r0 = (strip - batch * strips) * kArgRows;
  if (part < parts_a && p.Wo >= kArgCh) argmax_band_a<false>(accs, p, batch, r0, part * kArgKC);
  else if (part < parts_a) argmax_band_a<true>(accs, p, batch, r0, part * kArgKC);
  else argmax_band_b(accs, p, batch, r0, (part - parts_a) * kArgKC);
}

}  // namespace GENBMM_NS
