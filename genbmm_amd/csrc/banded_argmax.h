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
// that read their own rows fetch a cache line for every 16 bytes: 220 us).  The next chunk is in flight
// while one is added, and no load stands under a branch: behind one the compiler waits for every load.
// Both gradients are one launch, strip by strip, so that the second use of g and idx comes from a cache.
//
// Bound by the loads in flight and the ordered additions (add4_ordered: one LDS round trip per four
// cells); g and idx once and both gradients are 406 MB at 64 x 4096, 65 diagonals each.  Measured there:
// 255 us as two launches of four-wave workgroups that passed g and idx through LDS tiles behind two
// barriers each, 175 us now (bfloat16 335 -> 137; 512 x 512, 17 diagonals 92 -> 45).
#pragma once

#include "banded_cells.h"

namespace GENBMM_NS {

constexpr int kArgRows = 64;  // rows per workgroup: the lanes
constexpr int kArgKC = 128;   // diagonals per workgroup
constexpr int kArgCh = 16;    // cells of a row (grad_a), rows (grad_b) per chunk
constexpr int kArgTile = kArgCh + 1;   // grad_a's tile: floats per row
constexpr int kArgSlots = kArgCh + 4;  // and bytes per row (odd strides in banks)

// diagonals of a gradient per workgroup, and the workgroups that all W of them take
inline int argmax_kw(int W) { return min(W, kArgKC); }
inline int argmax_parts(int W) { return (W + kArgKC - 1) / kArgKC; }
// the cells and one spare cell per lane (terms that are not the lane's); grad_a: the tile
__host__ __device__ inline int argmax_cells(int kw) { return kArgRows * (kw + 1); }
inline size_t argmax_bwd_bytes(int Wa, int Wb) {
  return max(sizeof(float) * (argmax_cells(argmax_kw(Wa)) + kArgRows * kArgTile) + kArgRows * kArgSlots,
             sizeof(float) * (size_t)argmax_cells(argmax_kw(Wb)));
}

struct ArgColChunk {  // one cell of each of CH rows
  static constexpr int CH = kArgCh;
  int i[CH];
  elem_t g[CH];
};

// Compiler-level ordering point for a wave's own LDS traffic (one wave's LDS instructions execute in order).
__device__ __forceinline__ void argmax_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The lane's cells cleared, then `chunks` chunks: load(chunk, number), slots(chunk, number, slot, value)
template <class Chunk, class Load, class Slots>
__device__ __forceinline__ void argmax_walk(float* __restrict__ accs, int kw, int chunks, Load load, Slots slots) {
  constexpr int CH = Chunk::CH;
  const int lane = threadIdx.x;
  Chunk x, y;
  auto add = [&](const Chunk& ch, int c) __attribute__((always_inline)) {
    int sl[CH];
    float tv[CH];
    slots(ch, c, sl, tv);
#pragma unroll
    for (int q = 0; q < CH; q += 4) {
      const int s4[4] = {sl[q], sl[q + 1], sl[q + 2], sl[q + 3]};
      const float t4[4] = {tv[q], tv[q + 1], tv[q + 2], tv[q + 3]};
      add4_ordered(accs, s4, t4);
    }
  };
  if (chunks > 0) load(x, 0);
#pragma unroll 16
  for (int k = 0; k <= kw; ++k) accs[k * kArgRows + lane] = 0.f;
  int c = 0;
  for (; c + 1 < chunks; c += 2) {
    load(y, c + 1);
    add(x, c);
    load(x, min(c + 2, chunks - 1));
    add(y, c + 1);
  }
  if (c < chunks) add(x, c);
}

// The sums leave as rows, 32 diagonals at a time: they change places in LDS, through registers, from
// [k][lane] to [row][k] (32 whole diagonals: the k of a row permuted by its row number, which keeps both
// sides clear of bank conflicts), and go to memory in runs along the band.
__device__ __forceinline__ void argmax_write_out(float* __restrict__ accs, int kw, elem_t* __restrict__ out, int W,
                                                 int rows) {
  const int lane = threadIdx.x;
  for (int k0 = 0; k0 < kw; k0 += 32) {
    const int cw = min(32, kw - k0);
    float* t = accs + k0 * kArgRows;
    float v[32];
    argmax_lds_sync();
#pragma unroll
    for (int q = 0; q < 32; ++q) v[q] = t[min(q, cw) * kArgRows + lane];  // (row kw: the spare cells)
    argmax_lds_sync();
    if (cw == 32) {  // uniform
#pragma unroll
      for (int q = 0; q < 32; ++q) t[lane * 32 + (q ^ (lane & 31))] = v[q];
      argmax_lds_sync();
      const int c = lane & 31;
#pragma unroll 8
      for (int r = lane >> 5; r < rows; r += 2) out[(long)r * W + k0 + c] = to_elem<elem_t>(t[r * 32 + (c ^ (r & 31))]);
    } else {
#pragma unroll
      for (int q = 0; q < 32; ++q)
        if (q < cw) t[lane * cw + q] = v[q];
      argmax_lds_sync();
      for (int e = lane; e < rows * cw; e += 64) {
        const int r = e / cw, c = e - r * cw;
        out[(long)r * W + k0 + c] = to_elem<elem_t>(t[e]);
      }
    }
  }
}

// grad_a, rows [i0, i0 + 64), diagonals [w0, w0 + kw).  Sixteen cells of four rows per load; their terms
// and the slots they go to (a byte: kw <= 128 marks the spare) change places to the lane of their row
// through a tile of LDS.
__device__ __forceinline__ void argmax_band_a(float* __restrict__ accs, const BandArgs& p, int batch, int i0, int w0) {
  const int n = p.n, Wa = p.Wa, Wb = p.Wb, Wo = p.Wo, lane = threadIdx.x;
  const int kw = min(kArgKC, Wa - w0);
  float* gt = accs + argmax_cells(kw);
  unsigned char* st = reinterpret_cast<unsigned char*>(gt + kArgRows * kArgTile);
  const int jlo = w0, jhi = min(w0 + kw - 1 + Wb - 1, Wo - 1);  // cells with a term on these diagonals
  const int lr = lane >> 4, lj = lane & 15;
  const long base = ((long)batch * n + i0) * Wo;
  const elem_t* gb = p.g + base;
  const int32_t* ib = p.idx + base;
  const int last = n - 1 - i0;  // rows behind the matrix re-read its last row (nothing of them is stored)
  elem_t gv[kArgCh];
  int iv[kArgCh];
  unsigned ro[kArgCh];
#pragma unroll
  for (int u = 0; u < kArgCh; ++u) ro[u] = (unsigned)(min(4 * u + lr, last) * Wo + min(lj, Wo - 1));
  // the last chunk of a row starts inside the row, the cells that the chunk before it held are masked
  auto start = [&](int j0) __attribute__((always_inline)) { return max(min(j0, Wo - kArgCh), 0); };
  auto load = [&](int j0) __attribute__((always_inline)) {
    const elem_t* gs = gb + start(j0);
    const int32_t* is = ib + start(j0);
#pragma unroll
    for (int u = 0; u < kArgCh; ++u) {
      gv[u] = gs[ro[u]];
      iv[u] = is[ro[u]];
    }
  };
  load(jlo);
#pragma unroll 16
  for (int k = 0; k <= kw; ++k) accs[k * kArgRows + lane] = 0.f;
  for (int j0 = jlo; j0 <= jhi; j0 += kArgCh) {
    argmax_lds_sync();  // the tile has been read
    const int j = start(j0) + lj, o = i0 + lr + j - p.r_lu;
    const unsigned lim = j >= j0 && j <= jhi ? n : 0;  // inside the matrix: o = i + j - r_lu in [0, n)
#pragma unroll
    for (int u = 0; u < kArgCh; ++u) {
      const unsigned kr = (unsigned)(iv[u] - w0);
      const bool ok = kr < (unsigned)kw && (unsigned)(o + 4 * u) < lim;
      gt[(4 * u + lr) * kArgTile + lj] = (float)gv[u];
      st[(4 * u + lr) * kArgSlots + lj] = (unsigned char)(ok ? kr : kw);
    }
    argmax_lds_sync();
    load(j0 + kArgCh);  // (past the band: the row's last cells again)
    float tv[kArgCh];
    unsigned sw[kArgCh / 4];
#pragma unroll
    for (int q = 0; q < kArgCh; ++q) tv[q] = gt[lane * kArgTile + q];
#pragma unroll
    for (int q = 0; q < kArgCh / 4; ++q) sw[q] = *reinterpret_cast<const unsigned*>(st + lane * kArgSlots + 4 * q);
#pragma unroll
    for (int q = 0; q < kArgCh; q += 4) {
      const unsigned w = sw[q >> 2];
      const int s4[4] = {(int)(w & 255) * kArgRows + lane, (int)(w >> 8 & 255) * kArgRows + lane,
                         (int)(w >> 16 & 255) * kArgRows + lane, (int)(w >> 24) * kArgRows + lane};
      const float t4[4] = {tv[q], tv[q + 1], tv[q + 2], tv[q + 3]};
      add4_ordered(accs, s4, t4);
    }
  }
  argmax_write_out(accs, kw, p.o0 + ((long)batch * n + i0) * Wa + w0, Wa, min(kArgRows, n - i0));
}

// grad_b, rows [o0, o0 + 64), diagonals [w0, w0 + kw)
__device__ __forceinline__ void argmax_band_b(float* __restrict__ accs, const BandArgs& p, int batch, int o0, int w0) {
  const int n = p.n, Wa = p.Wa, Wb = p.Wb, Wo = p.Wo, lane = threadIdx.x;
  const int kw = min(kArgKC, Wb - w0), spare = kw * kArgRows + lane;
  const elem_t* gb = p.g + (long)batch * n * Wo;
  const int32_t* ib = p.idx + (long)batch * n * Wo;
  // cells with a term on these diagonals, and the rows i that hold them for some lane
  const int jlo = max(0, Wb - w0 - kw), jhi = min(Wo - 1, Wa + Wb - 2 - w0);
  const int ilo = max(0, o0 + p.r_lu - jhi), ihi = min(n - 1, o0 + kArgRows - 1 + p.r_lu - jlo);
  const int jof = o0 + lane + p.r_lu;  // j = jof - i
  argmax_walk<ArgColChunk>(
      accs, kw, ihi < ilo ? 0 : (ihi - ilo + kArgCh) / kArgCh,
      [&](ArgColChunk& x, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kArgCh; ++q) {
          const int i = min(ilo + c * kArgCh + q, ihi);  // uniform
          const unsigned j = (unsigned)min(max(jof - i, 0), Wo - 1);
          x.i[q] = (ib + (long)i * Wo)[j];
          x.g[q] = (gb + (long)i * Wo)[j];
        }
      },
      [&](const ArgColChunk& x, int c, int (&sl)[kArgCh], float (&tv)[kArgCh]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kArgCh; ++q) {
          // An index is a k of its cell, 0 (a cell outside the matrix) or -1 (no term; becomes far too
          // large).  Where j was clamped it is 0 or at most Wa - 1, and k2 falls outside [0, Wb) by itself.
          const int i = ilo + c * kArgCh + q;
          const unsigned kr = ((unsigned)x.i[q] & 0x7fffffffu) + (unsigned)(Wb - 1 - w0 + i) - (unsigned)jof;
          const unsigned lim = i <= ihi ? kw : 0;  // uniform
          sl[q] = kr < lim ? (int)kr * kArgRows + lane : spare;
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
  if (part < parts_a) argmax_band_a(accs, p, batch, r0, part * kArgKC);
  else argmax_band_b(accs, p, batch, r0, (part - parts_a) * kArgKC);
}

}  // namespace GENBMM_NS
