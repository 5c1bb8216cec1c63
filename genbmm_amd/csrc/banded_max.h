// Banded max-plus forward on whole strips: out[i,j] = max_k a[i,k] + b[o,k2] with its
// arg-max k (lowest k on ties, strict '>' from the reference's -1e9 floor, -1 if no k),
// o = i + j - lu_out, k2 = k - j + Wb - 1.
//
// A workgroup owns 64 rows i.  Their rows of a and the 64 + Wo - 1 rows of b that they
// meet are copied to LDS once, as they lie in memory (16-byte pieces, odd row strides: the
// 64 lanes of a wave are 64 consecutive rows and fall in different banks).  A lane owns
// one row; a wave walks blocks of 8 adjacent result diagonals j (blocks w, w + WAVES, ...
// - their sum lengths pair up, so the waves get equal work), reading one value of
// its own row per k and 8 values of b on an anti-diagonal.  The 8 cells walk the union of
// their k ranges without predicates: the rows of b lie at least 7 cells apart in LDS, with
// -inf between them, and a strip at the matrix's edge has -inf in the cells of a and the rows
// of b that lie outside it.  Values and indices go through LDS so that the strip's rows are
// written as one contiguous run.
//
// Compared with the chunked strip kernel (banded_strip.h) the sliding operand is staged
// once instead of once per 32 diagonals, and the result leaves in 16-byte stores.
//
// Wide results are cut into segments of Wseg <= 160 adjacent diagonals, one workgroup per strip
// and segment: a segment needs only the 64 + Wseg - 1 rows of b that its diagonals meet, so the
// tiles fit in LDS whatever the band width; its cells leave as one run of Wseg per row.
#pragma once

#include "banded_flat.h"

namespace GENBMM_NS {

constexpr int kMaxRows = 64;

struct MaxDims {
  int pp, qp, q_off, ops_floats, q_rows;
  size_t bytes;
};

// Wo: the diagonals one workgroup takes (the whole result or a segment of it)
inline MaxDims max_dims(int Wa, int Wb, int Wo) {
  MaxDims d;
  d.pp = Wa | 1;
  d.qp = (Wb + 7) | 1;  // at least 7 cells of -inf between two rows of b
  d.q_rows = kMaxRows + Wo - 1;
  d.q_off = (kMmSlack + kMaxRows * d.pp + 2 * (d.pp - Wa) + kMmSlack + 3) & ~3;
  // 8 rows more than staged: the last block of diagonals reaches past Wo
  d.ops_floats = (d.q_off + (d.q_rows + 8) * d.qp + 2 * (d.qp - Wb) + kMmSlack + 3) & ~3;
  // operands | values [64][Wo] and indices [64][Wo]
  const int tile = max(d.ops_floats, 2 * ((kMaxRows * Wo + 3) & ~3));
  d.bytes = sizeof(float) * (size_t)tile;
  return d;
}

// PAIRS: the walk takes two k at a time - their sums and the running maximum meet in one three-operand
// maximum, and one compare and one select keep the pair that raised it last: 2.5 instructions per term
// instead of 4 - and which k of its pair it was is found behind the walk, by forming the first one's sum
// again.  The first pair that attains the maximum and the first k inside it are what the walk with a
// strict comparison keeps (16 x 4096, 129 diagonals each 536 -> 497 us).
//
// Eight waves where LDS leaves a compute unit three workgroups or fewer (four waves each kept 1.8 on a SIMD, which
// issued in 63 % of its cycles), and for grids of one round.  With that, and strips at the matrix's edge on the same
// walk as the others instead of a loop of predicated single terms that the launch's end waited for:
// 64 x 4096, 65 diagonals each 272 -> 177 us, bfloat16 291 -> 165, 49 diagonals 153 -> 125; 2 x 500, 65 diagonals
// 72 -> 16; 57 x 366, 20 and 22 diagonals 17.3 -> 11.5.  (Eight waves on narrow bands: 17 diagonals 47 -> 60.)
template <bool PAIRS, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES == 8 ? 4 : 2) void k_band_max_fwd(const BandArgs p, int strips, const MaxDims d,
                                                         long cells_a, long cells_b, int nseg, int Wseg) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  constexpr int NT = 64 * WAVES, BLOCKS = (160 / 8 + WAVES - 1) / WAVES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int wg = xcd_strip_id();
  const int seg = wg % nseg;  // the segments of a strip run side by side: they share its rows of a
  wg /= nseg;
  const int batch = wg / strips, x0 = (wg - batch * strips) * kMaxRows;
  const int n = p.n, Wa = p.Wa, Wb = p.Wb, Wo = p.Wo, r_lu = p.r_lu;
  const int j_lo = seg * Wseg, Ws = min(Wseg, Wo - j_lo);  // this workgroup's diagonals [j_lo, j_lo + Ws)
  const long bn = (long)batch * n;
  float* PL = smem + kMmSlack;
  float* QL = smem + d.q_off;

  // ---- staging
  const int q0 = x0 - r_lu + j_lo;  // first row of b that the segment's cells meet
  const int qr0 = max(q0, 0), qr1 = min(q0 + d.q_rows, n);
  const int pr1 = min(x0 + kMaxRows, n);
  MmFlat<14 * 256 / NT, elem_t, NT> sq;
  MmFlat<6 * 256 / NT, elem_t, NT> sp;
  sq.init(p.b, p.b + cells_b, (bn + qr0) * Wb, (qr1 - qr0) * Wb, Wb, d.qp);
  sq.load(p.b, p.b + cells_b, 0, tid);
  sp.init(p.a, p.a + cells_a, (bn + x0) * Wa, (pr1 - x0) * Wa, Wa, d.pp);
  sp.load(p.a, p.a + cells_a, 0, tid);
  const int qp = d.qp, pp = d.pp;
  float* QR = QL + (qr0 - q0) * qp;  // (row q0 of b, inside the matrix or not, lies at QL)
  sq.store(QR, 0, tid);
  for (int b = 1; sq.more(b); ++b) {
    sq.load(p.b, p.b + cells_b, b, tid);
    sq.store(QR, b, tid);
  }
  sp.store(PL, 0, tid);
  for (int b = 1; sp.more(b); ++b) {
    sp.load(p.a, p.a + cells_a, b, tid);
    sp.store(PL, b, tid);
  }
  float* Pt = PL + sp.origin();  // a[x0 + r][k] = Pt[r * pp + k]
  float* Qt = QL + sq.origin();  // b[q0 + r][k2] = Qt[r * qp + k2]
  {  // -inf between the rows of b (and before the first): cells that are no k of a cell
    const int gap = qp - Wb;
    for (int e = tid; e < (d.q_rows + 1) * gap; e += NT) {
      const int r = e / gap, c = e - r * gap, at = sq.origin() + (r - 1) * qp + Wb + c;
      if (at >= 0) QL[at] = -INFINITY;
    }
  }
  // A strip at the matrix's edge: rows of b outside it, and cells of a in rows outside it, are no terms either.
  const bool interior = x0 >= max(p.a_lu, r_lu) && x0 + kMaxRows - 1 <= n - 1 - max(Wa - 1 - p.a_lu, Wo - 1 - r_lu);
  if (!interior) {  // uniform
    __syncthreads();  // the operands' cells are staged (and, in the first and last piece, cells beyond them)
    const int above = min(qr0 - q0, d.q_rows), below = min(max(q0 + d.q_rows - qr1, 0), d.q_rows - above);
    for (int e = tid; e < (above + below) * Wb; e += NT) {
      const int r = e / Wb, c = e - r * Wb;
      Qt[(r < above ? r : d.q_rows - below + r - above) * qp + c] = -INFINITY;
    }
    for (int e = tid; e < kMaxRows * Wa; e += NT) {
      const int r = e / Wa, k = e - r * Wa;
      if ((unsigned)(x0 + r + k - p.a_lu) >= (unsigned)n) Pt[r * pp + k] = -INFINITY;
    }
  }
  __syncthreads();

  // ---- products
  const int x = x0 + lane;
  const float* ap = Pt + lane * pp;
  const int nblocks = (Ws + 7) >> 3;
  float val[BLOCKS][8];  // blocks wave, wave + WAVES, ... (Ws <= 160)
  int ind[BLOCKS][8];
#pragma unroll
  for (int s = 0; s < BLOCKS; ++s) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      val[s][t] = kFloor;
      ind[s][t] = -1;
    }
    const int jb = wave + WAVES * s;
    if (jb < nblocks) {
      const int j0 = j_lo + 8 * jb;
      // b[o][k2] of cell t at step k: Qt[(lane + j0 - j_lo + t) * qp + k - j0 - t + Wb - 1]
      const float* bp = Qt + (lane + j0 - j_lo) * qp + (Wb - 1 - j0);
      const int dt = qp - 1;
      auto fold = [&](int t, float av, float bv, int k) __attribute__((always_inline)) {
        const float v = av + bv;
        if (v > val[s][t]) {
          val[s][t] = v;
          ind[s][t] = k;
        }
      };
      {
        // all 8 cells walk the union of their k ranges: where a cell has no such k it reads
        // -inf from between the rows
        const int klo = max(0, j0 - (Wb - 1)), khi = min(Wa - 1, j0 + 7);
        // four cells at a time: their compares, then their selects
        auto fold4 = [&](int t, float a0, const float (&b0)[8], int k) __attribute__((always_inline)) {
          const float v[4] = {a0 + b0[t], a0 + b0[t + 1], a0 + b0[t + 2], a0 + b0[t + 3]};
          const Mask4 up(v[0] > val[s][t], v[1] > val[s][t + 1], v[2] > val[s][t + 2], v[3] > val[s][t + 3]);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            val[s][t + q] = up[q] ? v[q] : val[s][t + q];
            ind[s][t + q] = up[q] ? k : ind[s][t + q];
          }
        };
        auto pairs4 = [&](int t, float a0, float a1, const float (&b0)[8], const float (&b1)[8], int k) __attribute__((always_inline)) {
          float m[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) m[q] = __builtin_fmaxf(__builtin_fmaxf(val[s][t + q], a0 + b0[t + q]), a1 + b1[t + q]);
          const Mask4 up(m[0] > val[s][t], m[1] > val[s][t + 1], m[2] > val[s][t + 2], m[3] > val[s][t + 3]);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            ind[s][t + q] = up[q] ? k : ind[s][t + q];
            val[s][t + q] = m[q];
          }
        };
        int k = klo;
        for (; k + 3 <= khi; k += 4) {
          float av[4], bv[4][8];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            av[u] = ap[k + u];
#pragma unroll
            for (int t = 0; t < 8; ++t) bv[u][t] = bp[t * dt + k + u];
          }
#pragma unroll
          for (int u = 0; u < 4; u += 2)
#pragma unroll
            for (int t = 0; t < 8; t += 4) {
              if (PAIRS) {
                pairs4(t, av[u], av[u + 1], bv[u], bv[u + 1], k + u);
              } else {
                fold4(t, av[u], bv[u], k + u);
                fold4(t, av[u + 1], bv[u + 1], k + u + 1);
              }
            }
        }
        for (; k <= khi; ++k) {
          const float av = ap[k];
#pragma unroll
          for (int t = 0; t < 8; ++t) fold(t, av, bp[t * dt + k], k);
        }
        if (PAIRS) {  // which k of its pair: the first whose sum is the maximum
          bool zero = false;
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            const int at = max(ind[s][t], klo);  // (no term: any cell)
            const bool second = ap[at] + bp[t * dt + at] != val[s][t];
            ind[s][t] += ind[s][t] >= 0 && second;
            zero |= val[s][t] == 0.f;
          }
          if (zero) {  // +0 and -0 compare equal: the value is the term's
#pragma unroll
            for (int t = 0; t < 8; ++t)
              if (val[s][t] == 0.f) val[s][t] = ap[ind[s][t]] + bp[t * dt + ind[s][t]];
          }
        }
      }
    }
  }
  __syncthreads();  // the operands are consumed: their place becomes the result tiles

  float* Sv = smem;
  int* Si = reinterpret_cast<int*>(smem + ((kMaxRows * Ws + 3) & ~3));
#pragma unroll
  for (int s = 0; s < BLOCKS; ++s) {
    const int jb = wave + WAVES * s;
    if (jb < nblocks) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int js = 8 * jb + t, o = x + j_lo + js - r_lu;
        if (js < Ws) {
          const bool inside = x < n && o >= 0 && o < n;  // outside: the reference's zero fill
          Sv[lane * Ws + js] = inside ? val[s][t] : 0.f;
          Si[lane * Ws + js] = inside ? ind[s][t] : 0;
        }
      }
    }
  }
  __syncthreads();

  const int rows = min(kMaxRows, n - x0), cells = rows * Ws;
  elem_t* ob = p.o0 + (bn + x0) * Wo + j_lo;
  int32_t* ib = p.oidx + (bn + x0) * Wo + j_lo;
  typedef int mm_i4 __attribute__((ext_vector_type(4)));
  if (Ws == Wo && (cells & 3) == 0 &&
      ((reinterpret_cast<uintptr_t>(ob) | reinterpret_cast<uintptr_t>(ib)) & 15) == 0) {
    for (int e = 4 * tid; e < cells; e += 4 * NT) {  // the strip's rows are one contiguous run
      st4a(ob + e, *reinterpret_cast<const float4*>(Sv + e));
      *reinterpret_cast<mm_i4*>(ib + e) = *reinterpret_cast<const mm_i4*>(Si + e);
    }
  } else {
    for (int e = tid; e < cells; e += NT) {  // runs of Ws cells, one per row
      const int r = e / Ws, c = e - r * Ws;
      ob[(long)r * Wo + c] = to_elem<elem_t>(Sv[e]);
      ib[(long)r * Wo + c] = Si[e];
    }
  }
}

}  // namespace GENBMM_NS
