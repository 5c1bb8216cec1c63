// Factored logbmm on the bf16 matrix instruction with fp32 accuracy: every staged factor
// x (fp32) is cut into three bfloat16 parts h + m + l = x exactly (h = x rounded to bf16,
// m = x - h rounded, l = the rest: 8 + 8 + 8 significant bits), and a product x y is taken
// as the six partial products h h, h m, m h, m m, h l, l h on v_mfma_f32_32x32x16_bf16
// (fp32 accumulate; bf16 x bf16 is exact in fp32).  What is left out - m l, l m, l l - is
// below 2^-23 of x y, the size of one fp32 rounding of the product itself.  The
// instruction does 16 reduction steps in the time the fp32 one (v_mfma_f32_32x32x2_f32)
// needs for one, so six of them per 16 steps are 2.7 times less matrix-pipe time, and -
// unlike the fp32 matrix instruction on this part - vector instructions of other waves can
// execute beside them (the counters show it for about a third of the pipe's busy cycles).
//
// Same tiles, guards, flags, epilogues and fix-up launches as the fp32 kernels of
// logbmm_mfma.h (a 64 x 64 block per wave as 2 x 2 accumulators, whose layout is that of
// the fp32 instruction; reduction in slabs of 16 through two LDS buffers); what differs is
// the staged form and the inner loop.  Ragged edges are a second instantiation of each
// kernel (RAGGED), handled as in logbmm_mfma.h: lines of a tile beyond the matrix re-read
// the last line (under a shift that makes the factor vanish where the line feeds stored
// results), stores are masked.  Any sizes: where the reduction is contiguous a thread reads four
// steps of a line, where the lines are, some steps of one line - lines beyond the matrix are the
// last one again -, so nothing is astride an edge, and the partial last slab of the forward and the
// backward is a step of its own behind the loop, with a loader of its own.  The sampling sweep reads
// its last slab whole and zeroes what lies beyond K; its targets alone come in pieces of four
// columns, of which one astride the right edge is moved down (shift_down).  (Backward of
// (64, 511, 509, 510): 368 us on the fp32 instruction, 256 here.)
//
// LDS layouts, three planes (h, m, l) per operand, words of two bf16:
//  * an operand whose source is [line][reduction] (reduction contiguous): plane[line][8
//    words]; a lane stages four consecutive reduction steps of a line (one 8-byte store
//    per plane) and reads the eight steps of its line that the instruction wants from it
//    as one 16-byte load.
//  * an operand whose source is [reduction][line], staged by a line's own threads (SplitL): plane[half of the
//    slab][line][4 words], an operand one 16-byte read.
//  * the same for the one-tile kernels of logbmm_self.h, whose threads hold four lines (SplitS): plane[8 step
//    pairs][lines + 8]; a thread stages a pair of reduction steps of its four lines (the pair shares a word; one
//    16-byte store per plane) and the instruction's eight steps are four words a row apart.  The compiler pairs
//    these four reads across operands and then moves them apart (24 moves and a wait for each pair per slab, ahead
//    of the products): (64, 512^3) forward 108 us and both gradients 229 in this form, 102 and 210 by SplitL;
//    (48, 251, 173, 301) 33.8 -> 28.8 and 49.8 -> 46.6, results bit for bit.
#pragma once

#include "logbmm_mfma.h"
#include "split_bf16.h"

namespace GENBMM_NS {

// source [line][reduction]
template <int OUT, int NT>
struct SplitT {
  static constexpr int PLANE = OUT * 8;      // words
  static constexpr int BUF = 3 * PLANE;
  static constexpr int PER = OUT * 4 / NT;   // pieces (a line, four reduction steps) per thread
  static_assert(PER >= 1 && OUT * 4 % NT == 0, "");
  static __device__ __forceinline__ int line(int tid, int l) { return (tid >> 2) + l * (NT / 4); }
  static __device__ __forceinline__ int quad(int tid) { return tid & 3; }
  static __device__ __forceinline__ void put(unsigned* __restrict__ buf, int tid, int l, float4 v) {
    unsigned h0, m0, l0, h1, m1, l1;
    split2(v.x, v.y, h0, m0, l0);
    split2(v.z, v.w, h1, m1, l1);
    unsigned* p = buf + line(tid, l) * 8 + quad(tid) * 2;
    uintx2 w;
    w.x = h0; w.y = h1; *reinterpret_cast<uintx2*>(p) = w;
    w.x = m0; w.y = m1; *reinterpret_cast<uintx2*>(p + PLANE) = w;
    w.x = l0; w.y = l1; *reinterpret_cast<uintx2*>(p + 2 * PLANE) = w;
  }
  // the lane's operand of one 32-line block: line0 + lane % 32, reduction steps 8 (lane / 32) .. + 7
  static __device__ __forceinline__ bf16x8 frag(const unsigned* __restrict__ buf, int plane, int line0, int lane) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4*>(buf + plane * PLANE + (line0 + (lane & 31)) * 8 +
                                                                       (lane >> 5) * 4));
  }
};

// source [reduction][line], a thread stages a pair of reduction steps of four lines
template <int OUT, int NT>
struct SplitS {
  static constexpr int LD = OUT + 8;         // words per step pair (lanes 32.. read four rows on: other banks)
  static constexpr int PLANE = 8 * LD;
  static constexpr int BUF = 3 * PLANE;
  static_assert(OUT * 2 == NT, "one piece of a pair and four lines per thread");
  static __device__ __forceinline__ int pair(int tid) { return tid / (OUT / 4); }  // reduction steps 2 pair, 2 pair + 1
  static __device__ __forceinline__ int line0(int tid) { return (tid % (OUT / 4)) * 4; }
  static __device__ __forceinline__ void put(unsigned* __restrict__ buf, int tid, float4 even, float4 odd) {
    const float e[4] = {even.x, even.y, even.z, even.w}, o[4] = {odd.x, odd.y, odd.z, odd.w};
    unsigned h[4], m[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) split2(e[j], o[j], h[j], m[j], l[j]);
    unsigned* p = buf + pair(tid) * LD + line0(tid);
    uintx4 w;
    w.x = h[0]; w.y = h[1]; w.z = h[2]; w.w = h[3]; *reinterpret_cast<uintx4*>(p) = w;
    w.x = m[0]; w.y = m[1]; w.z = m[2]; w.w = m[3]; *reinterpret_cast<uintx4*>(p + PLANE) = w;
    w.x = l[0]; w.y = l[1]; w.z = l[2]; w.w = l[3]; *reinterpret_cast<uintx4*>(p + 2 * PLANE) = w;
  }
  static __device__ __forceinline__ bf16x8 frag(const unsigned* __restrict__ buf, int plane, int line0, int lane) {
    const unsigned* p = buf + plane * PLANE + (lane >> 5) * 4 * LD + line0 + (lane & 31);
    uintx4 w;
    w.x = p[0]; w.y = p[LD]; w.z = p[2 * LD]; w.w = p[3 * LD];
    return __builtin_bit_cast(bf16x8, w);
  }
};

// source [reduction][line], a thread stages ST consecutive reduction steps of one line: plane[half of the
// slab][line][4 words].  The loads of a step run along the lines, a wave's steps are its own (uniform row
// addresses), the staged words leave in one store per plane and an operand is one 16-byte read of
// neighbouring lanes side by side.
template <int OUT, int NT>
struct SplitL {
  static constexpr int PLANE = 8 * OUT;      // words
  static constexpr int BUF = 3 * PLANE;
  static constexpr int ST = 16 * OUT / NT;   // steps per thread
  static_assert((ST == 4 || ST == 8) && OUT % 64 == 0, "");
  static __device__ __forceinline__ int line(int tid) { return tid % OUT; }
  static __device__ __forceinline__ int step0(int tid) { return __builtin_amdgcn_readfirstlane(tid / OUT) * ST; }
  static __device__ __forceinline__ void put(unsigned* __restrict__ buf, int tid, const float (&v)[ST]) {
    unsigned h[ST / 2], m[ST / 2], l[ST / 2];
#pragma unroll
    for (int j = 0; j < ST / 2; ++j) split2(v[2 * j], v[2 * j + 1], h[j], m[j], l[j]);
    const int s0 = step0(tid);
    unsigned* p = buf + (s0 >> 3) * (4 * OUT) + line(tid) * 4 + (ST == 4 ? (s0 & 4) >> 1 : 0);
    if constexpr (ST == 8) {
      uintx4 w;
      w.x = h[0]; w.y = h[1]; w.z = h[2]; w.w = h[3]; *reinterpret_cast<uintx4*>(p) = w;
      w.x = m[0]; w.y = m[1]; w.z = m[2]; w.w = m[3]; *reinterpret_cast<uintx4*>(p + PLANE) = w;
      w.x = l[0]; w.y = l[1]; w.z = l[2]; w.w = l[3]; *reinterpret_cast<uintx4*>(p + 2 * PLANE) = w;
    } else {
      uintx2 w;
      w.x = h[0]; w.y = h[1]; *reinterpret_cast<uintx2*>(p) = w;
      w.x = m[0]; w.y = m[1]; *reinterpret_cast<uintx2*>(p + PLANE) = w;
      w.x = l[0]; w.y = l[1]; *reinterpret_cast<uintx2*>(p + 2 * PLANE) = w;
    }
  }
  static __device__ __forceinline__ bf16x8 frag(const unsigned* __restrict__ buf, int plane, int line0, int lane) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4*>(buf + plane * PLANE + (lane >> 5) * (4 * OUT) +
                                                                       (line0 + (lane & 31)) * 4));
  }
};

// v[j] <- v[j + by] for 0 < by < 4 (the places behind keep what they hold); other `by`: nothing
__device__ __forceinline__ void shift_down(float (&v)[4], int by) {
  if (by == 1) { v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; }
  if (by == 2) { v[0] = v[2]; v[1] = v[3]; }
  if (by == 3) v[0] = v[3];
}

// The waves of a SIMD (waves i, i + 4, ... of the workgroup) run their matrix instructions at
// different priorities, all above the priority of staging: behind a barrier they would otherwise
// take turns instruction by instruction, finish their products together and then all stage at
// once with the matrix pipe idle; this way the first is through early and stages - vector work,
// which issues beside the others' matrix instructions - while the next one multiplies.
__device__ __forceinline__ void mfma_prio(int wave) {
  switch ((wave >> 2) & 3) {
    case 0: __builtin_amdgcn_s_setprio(3); break;
    case 1: __builtin_amdgcn_s_setprio(2); break;
    case 2: __builtin_amdgcn_s_setprio(1); break;
    default: __builtin_amdgcn_s_setprio(1); break;
  }
}

// The six partial products of one staged slab, for the wave's 2 x 2 blocks.  Products of one
// kind go to the four accumulators in turn (no instruction waits for the one before it);
// the small ones first.
template <class SR, class SC>
__device__ __forceinline__ void split_slab(const unsigned* __restrict__ R, const unsigned* __restrict__ Cs, int wr0,
                                           int wc0, int wave, int lane, floatx16 (&acc)[2][2]) {
  // Operand registers are asked for a phase ahead of their products and given up after them
  // (at most 40 of them live beside the 64 accumulators; the fences keep the compiler from
  // asking for all twelve operands up front).
  bf16x8 rh[2], ch[2], cl[2], rl[2], rm[2], cm[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rh[i] = SR::frag(R, 0, wr0 + 32 * i, lane);
    cl[i] = SC::frag(Cs, 2, wc0 + 32 * i, lane);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    ch[i] = SC::frag(Cs, 0, wc0 + 32 * i, lane);
    rl[i] = SR::frag(R, 2, wr0 + 32 * i, lane);
  }
  __builtin_amdgcn_sched_barrier(0);
  mfma_prio(wave);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rh[x >> 1], cl[x & 1], acc[x >> 1][x & 1]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 2; ++i) cm[i] = SC::frag(Cs, 1, wc0 + 32 * i, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rl[x >> 1], ch[x & 1], acc[x >> 1][x & 1]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 2; ++i) rm[i] = SR::frag(R, 1, wr0 + 32 * i, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rh[x >> 1], cm[x & 1], acc[x >> 1][x & 1]);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rm[x >> 1], cm[x & 1], acc[x >> 1][x & 1]);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rm[x >> 1], ch[x & 1], acc[x >> 1][x & 1]);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = mfma_bf16(rh[x >> 1], ch[x & 1], acc[x >> 1][x & 1]);
  __builtin_amdgcn_s_setprio(0);
  __builtin_amdgcn_sched_barrier(0);
}

// LDS words of a kernel on tile T whose row operand is staged by SR and column operand by SC
template <class SR, class SC>
constexpr int split_lds_words() { return 2 * (SR::BUF + SC::BUF); }

// The slab loop.  On entry slab 0 is loaded and staged (no barrier yet).
// The four waves of a SIMD (waves i, i + 4, i + 8, i + 12 of a workgroup of sixteen) issue their
// matrix instructions at descending priority (mfma_prio), so behind the barrier the first is
// through its products early and the last late.  The first half ("late" waves) stages the next
// slab behind its products, while the others still multiply; the second half ("early" waves),
// which must wait for the matrix pipe anyway, stages the next slab AHEAD of its products - from
// registers loaded a whole slab before - while the first half multiplies.  Nobody's staging is
// left for the end of the slab with the matrix pipe idle.  One load in flight per wave either way.
template <class Load, class Stage, class Mma>
__device__ __forceinline__ void split_loop(int slabs, bool early, Load&& load, Stage&& stage, Mma&& mma) {
  if (early && slabs > 1) load();
  __syncthreads();
  for (int s = 0; s < slabs; ++s) {
    const bool more = s + 1 < slabs;
    if (early) {
      if (more) stage((s + 1) & 1);
      if (s + 2 < slabs) load();
    } else {
      if (more) load();
    }
    mma(s & 1);
    if (!early && more) stage((s + 1) & 1);
    __syncthreads();
  }
}
// the second half of a workgroup's waves
template <int NT>
__device__ __forceinline__ bool split_early(int wave) { return wave >= NT / 128; }
// ----------------------------------------------------------------- forward
// rows <- EA from a[m][k] ([line][reduction]), columns <- EB from b[k][n] ([reduction][line]).
// Leaves the maxima, the tile flags and the header; KEEP: also the factors EA, EB (fp32, written
// by the tiles that stage them anyway: slab s of a row block's EA by its column block s mod
// tiles_n, likewise EB) and 1 / S, as k_log_fwd_mfma<T, RAGGED, true> does - what the sampling
// sweep reads.
// PIECES: the reduction axis is cut into `pieces` runs of slabs, each a workgroup of its own
// (workgroup = tile * pieces + piece); a piece leaves its sums S for its tile in ws_r
// ([piece][batch][M][N]) and k_log_fwd_join adds them, tests the guard and takes the logarithm.
// For problems with few output tiles and a long reduction, which would otherwise run on a few
// compute units.
template <class T, bool RAGGED, int KEEPS, bool PIECES = false>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(T::WPE, T::WPE)))
void k_log_fwd_split(const elem_t* __restrict__ a, const elem_t* __restrict__ b, elem_t* __restrict__ out,
                     const float* __restrict__ stats, int* __restrict__ flags, float* __restrict__ ws_ea,
                     float* __restrict__ ws_eb, float* __restrict__ ws_r, int* __restrict__ ws_hdr, int M, int K,
                     int N, int tiles_m, int tiles_n, int pieces = 1) {
  static_assert(!PIECES || (RAGGED && KEEPS == kKeepNone), "");
  constexpr bool KEEP = KEEPS == kKeepFactors;
  constexpr int NT = T::NT;
  using SA = SplitT<T::TR, NT>;
  using SB = SplitL<T::TC, NT>;
  constexpr int ST = SB::ST;
  extern __shared__ __attribute__((aligned(16))) unsigned split_smem[];
  static_assert(split_lds_words<SA, SB>() >= (NT / 64) * kStripFloats, "");
  auto As = [&](int buf) __attribute__((always_inline)) { return split_smem + buf * SA::BUF; };
  auto Bs = [&](int buf) __attribute__((always_inline)) { return split_smem + 2 * SA::BUF + buf * SB::BUF; };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / T::WC) * 64, wn0 = (wave % T::WC) * 64;
  const int per = tiles_m * tiles_n, wg = xcd_tile_id();
  const int tile = PIECES ? wg / pieces : wg, piece = PIECES ? wg - tile * pieces : 0;
  const int batch = tile / per, rem = tile - batch * per;
  const int m0 = (rem / tiles_n) * T::TR, n0 = (rem % tiles_n) * T::TC;
  const float* st = stats + (long)batch * (M + N);
  // the slabs of this workgroup: all of them, or the piece's run (no piece is empty)
  const int slabs_all = RAGGED ? (K + kMS - 1) / kMS : K / kMS;
  const int slabs_piece = PIECES ? (slabs_all + pieces - 1) / pieces : slabs_all;
  const int slab0 = piece * slabs_piece;

  // a pieces: line m0 + line(l), four k from quad * 4;  b: ST steps of one column
  const elem_t* pa[SA::PER];
  float al[SA::PER];
  bool va[SA::PER];
#pragma unroll
  for (int l = 0; l < SA::PER; ++l) {
    const int line = m0 + SA::line(tid, l);
    va[l] = !RAGGED || line < M;
    pa[l] = a + ((long)batch * M + (va[l] ? line : M - 1)) * K + SA::quad(tid) * 4 + (long)slab0 * kMS;
    al[l] = va[l] ? st[line] : INFINITY;  // lines beyond the matrix: exp -> 0
  }
  // the factors live at the same offsets in their own arrays (the source pointers run one slab
  // ahead of what is being staged, whichever side of its products a wave stages on)
  const int nblk = rem % tiles_n, mblk = rem / tiles_n;
  const long da = KEEP ? ws_distance(ws_ea, a) - 4l * kMS : 0, db = KEEP ? ws_distance(ws_eb, b) - 4l * kMS * N : 0;
  int sa = 0, sb = 0;  // the slab the next stage() forms, mod tiles_n and mod tiles_m
  const int brow = SB::step0(tid);  // uniform
  const bool vb = !RAGGED || n0 + SB::line(tid) < N;
  const unsigned bcol = vb ? n0 + SB::line(tid) : N - 1;
  const elem_t* pb = b + ((long)batch * K + brow + (long)slab0 * kMS) * N;
  const float be = vb ? st[M + bcol] : INFINITY;
  if (!PIECES && tile == 0 && tid == 0) {
    ws_hdr[1] = T::TR;
    ws_hdr[2] = T::TC;
    ws_hdr[0] = KEEP ? kWsMfma : KEEPS == kKeepRecip ? kWsRecip : kWsFast;
  }

  floatx16 acc[2][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[x >> 1][x & 1][i] = 0.f;

  const int slabs = PIECES ? min(slabs_piece, slabs_all - slab0) : slabs_all;
  // reduction steps of a partial last slab (of the last piece): one more step behind the loop, with a loader of
  // its own - the loads of the loop stand under no branch, where they would be waited for ahead of the products
  const int ktail = RAGGED && (!PIECES || slab0 + slabs == slabs_all) ? K % kMS : 0;
  const int whole = slabs - (RAGGED && ktail != 0 ? 1 : 0);
  float4 ra[SA::PER];
  elem_t rb[ST];
  auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) ra[l] = ld4(pa[l]);
#pragma unroll
    for (int j = 0; j < ST; ++j) rb[j] = (pb + (long)j * N)[bcol];
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) pa[l] += kMS;
    pb += (long)kMS * N;
  };
  auto stage_to = [&](int buf, int steps) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) {
      const float4 e = exp4(ra[l], al[l]);
      SA::put(As(buf), tid, l, e);
      if (KEEP && sa == nblk) {
        if (!RAGGED) st4(ws_twin(pa[l], da), e);
        else if (va[l]) st4m(ws_twin(pa[l], da), clamp4(steps - SA::quad(tid) * 4), e);
      }
    }
    float eb[ST];
#pragma unroll
    for (int j = 0; j < ST; ++j) eb[j] = exp_st((float)rb[j] - be);
    SB::put(Bs(buf), tid, eb);
    if (KEEP && sb == mblk) {
      float* we = ws_twin(pb, db);
#pragma unroll
      for (int j = 0; j < ST; ++j)
        if (vb && brow + j < steps) (we + (long)j * N)[bcol] = eb[j];
    }
    if (KEEP) {
      sa = sa + 1 == tiles_n ? 0 : sa + 1;
      sb = sb + 1 == tiles_m ? 0 : sb + 1;
    }
  };
  auto stage = [&](int buf) __attribute__((always_inline)) { stage_to(buf, kMS); };

  if (!PIECES || whole > 0) {
    load();
    stage(0);
    split_loop(whole, split_early<NT>(wave), load, stage, [&](int buf) __attribute__((always_inline)) {
      split_slab<SA, SB>(As(buf), Bs(buf), wm0, wn0, wave & (NT / 64 - 1), lane, acc);
    });
  }
  if (RAGGED && ktail != 0) {  // uniform
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) {
      ra[l] = ld4m(pa[l], clamp4(ktail - SA::quad(tid) * 4), -INFINITY);
      pa[l] += kMS;
    }
#pragma unroll
    for (int j = 0; j < ST; ++j) rb[j] = brow + j < ktail ? (pb + (long)j * N)[bcol] : (elem_t)-INFINITY;
    pb += (long)kMS * N;
    stage_to(0, ktail);
    __syncthreads();
    split_slab<SA, SB>(As(0), Bs(0), wm0, wn0, wave & (NT / 64 - 1), lane, acc);
    __syncthreads();
  }

  if constexpr (PIECES) {  // the piece's sums, row-wise; the guard is k_log_fwd_join's
    __syncthreads();       // every wave is done with the staging buffers
    const int lr = lane >> 4, lc = (lane & 15) * 4;
    const int cc = clamp4(N - (n0 + wn0 + lc));
    const long ubase = (((long)piece * (gridDim.x / (pieces * per)) + batch) * M + m0 + wm0) * N + n0 + wn0;
    const int voff = lr * N + lc, rows_left = M - (m0 + wm0) - lr;
    acc_rows(acc, reinterpret_cast<float*>(split_smem) + wave * kStripFloats, lane, [](int) {},
             [&](int q, int t, float4 sv) __attribute__((always_inline)) {
               const int ru = 16 * q + 4 * t;
               if (cc > 0 && ru < rows_left) st4m(ws_r + ubase + (long)ru * N + voff, cc, sv);
             });
    return;
  }
  // guard (as k_log_fwd_mfma): S >= 2^-40 and finite; every shift finite and not below the floor;
  // no shift below -30 opposite a row or column at the floor
  const float thr = fast_exp2(-kMfmaGuardBits);
  int bad = 0;
  {
    const int rlim = M - (m0 + wm0) - mfma_row_l(lane);   // rows of this lane below rlim exist
    const int clim = N - (n0 + wn0) - (lane & 31);        // column blocks at offset < clim exist
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float s = acc[x >> 1][x & 1][i];
        const bool here = !RAGGED || ((x >> 1) * 32 + mfma_row_u(i) < rlim && (x & 1) * 32 < clim);
        if (here && !((s >= thr) && (s < INFINITY))) bad = 1;
      }
  }
  static_assert(T::TR + T::TC <= NT, "one shift per thread");
  int low = 0, neg = 0;  // bit 0: of a row, bit 1: of a column
  {
    const bool row = tid < T::TR;
    const bool here = tid < T::TR + T::TC && (!RAGGED || (row ? m0 + tid < M : n0 + tid - T::TR < N));
    if (here) {
      const float sh = row ? st[m0 + tid] : st[M + n0 + tid - T::TR];
      if (!((sh >= kFloor) && (sh < INFINITY))) bad = 1;
      if (sh <= 0.45f * kFloor) low = row ? 1 : 2;
      if (sh < -30.f) neg = row ? 1 : 2;
    }
  }
  const int row_low = __syncthreads_or(low & 1), col_low = __syncthreads_or(low & 2);
  if (row_low | col_low) {  // uniform, and rare
    const int row_neg = __syncthreads_or(neg & 1), col_neg = __syncthreads_or(neg & 2);
    if ((row_low && col_neg) || (col_low && row_neg)) bad = 1;
  }
  bad = __syncthreads_or(bad);  // also: every wave is done with the staging buffers
  if (tid == 0) flags[tile] = bad;
  if (bad) return;  // the fix-up launch recomputes this tile

  // out = log S + alpha + beta, written row-wise
  const int lr = lane >> 4, lc = (lane & 15) * 4;
  const int cc = RAGGED ? clamp4(N - (n0 + wn0 + lc)) : 4;  // columns of this lane's pieces that exist
  const bool cok = cc > 0;
  const float4 be4 = RAGGED ? ld4m(st + M + (cok ? n0 + wn0 + lc : 0), cc, 0.f) : ld4(st + M + n0 + wn0 + lc);
  const float* alw = st + m0 + wm0 + lr;
  const long ubase = ((long)batch * M + m0 + wm0) * N + n0 + wn0;
  const int voff = lr * N + lc;
  const int rows_left = M - (m0 + wm0) - lr;
  acc_rows(acc, reinterpret_cast<float*>(split_smem) + wave * kStripFloats, lane, [](int) {},
           [&](int q, int t, float4 sv) __attribute__((always_inline)) {
             const int ru = 16 * q + 4 * t;
             if (RAGGED && !(cok && ru < rows_left)) return;
             const float alr = alw[ru];
             const float4 ov = make_float4(__builtin_fmaf(fast_log2(sv.x), kLn2, alr + be4.x),
                                           __builtin_fmaf(fast_log2(sv.y), kLn2, alr + be4.y),
                                           __builtin_fmaf(fast_log2(sv.z), kLn2, alr + be4.z),
                                           __builtin_fmaf(fast_log2(sv.w), kLn2, alr + be4.w));
             if (RAGGED) st4m(out + ubase + (long)ru * N + voff, cc, ov);
             else st4(out + ubase + (long)ru * N + voff, ov);
             if constexpr (KEEPS != kKeepNone) {
               const float4 rv = make_float4(__builtin_amdgcn_rcpf(sv.x), __builtin_amdgcn_rcpf(sv.y),
                                             __builtin_amdgcn_rcpf(sv.z), __builtin_amdgcn_rcpf(sv.w));
               if (RAGGED) st4m(ws_r + ubase + (long)ru * N + voff, cc, rv);
               else st4(ws_r + ubase + (long)ru * N + voff, rv);
             }
           });
}

// The pieces of k_log_fwd_split<.., PIECES> joined: S = the sum of the pieces' sums for a cell, then
// the forward's guard - per tile of TR x TC cells, the tile shape that the flags, the header and the
// exact fix-up launch behind this kernel go by - and out = log S + alpha + beta.  One workgroup per tile.
template <int TR, int TC>
__global__ __launch_bounds__(256) void k_log_fwd_join(const float* __restrict__ parts, elem_t* __restrict__ out,
                                                      const float* __restrict__ stats, int* __restrict__ flags,
                                                      int* __restrict__ ws_hdr, int B, int M, int N, int tiles_m,
                                                      int tiles_n, int pieces) {
  const int tid = threadIdx.x, tile = blockIdx.x, per = tiles_m * tiles_n;
  const int batch = tile / per, rem = tile - batch * per;
  const int m0 = (rem / tiles_n) * TR, n0 = (rem % tiles_n) * TC;
  const float* st = stats + (long)batch * (M + N);
  const long piece_stride = (long)B * M * N;
  const float thr = fast_exp2(-kMfmaGuardBits);
  int bad = 0, low = 0, neg = 0;  // bit 0: of a row, bit 1: of a column
  for (int c = tid; c < TR * (TC / 4); c += 256) {
    const int m = m0 + c / (TC / 4), n = n0 + (c % (TC / 4)) * 4;
    const int cc = clamp4(N - n);
    if (m >= M || cc <= 0) continue;
    const long at = ((long)batch * M + m) * N + n;
    float4 sv = ld4m(parts + at, cc, 0.f);
    int p = 1;
    for (; p + 8 <= pieces; p += 8) {  // eight pieces' loads in flight; added in the pieces' order
      float4 x[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = ld4m(parts + (p + q) * piece_stride + at, cc, 0.f);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        sv.x += x[q].x; sv.y += x[q].y; sv.z += x[q].z; sv.w += x[q].w;
      }
    }
    for (; p < pieces; ++p) {
      const float4 x = ld4m(parts + p * piece_stride + at, cc, 0.f);
      sv.x += x.x; sv.y += x.y; sv.z += x.z; sv.w += x.w;
    }
    const float alr = st[m];
    const float4 be4 = ld4m(st + M + n, cc, 0.f);
    const float s4[4] = {sv.x, sv.y, sv.z, sv.w}, b4[4] = {be4.x, be4.y, be4.z, be4.w};
    if (!((alr >= kFloor) && (alr < INFINITY))) bad = 1;
    if (alr <= 0.45f * kFloor) low |= 1;
    if (alr < -30.f) neg |= 1;
    float o4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o4[j] = 0.f;
      if (j < cc) {
        if (!((s4[j] >= thr) && (s4[j] < INFINITY)) || !((b4[j] >= kFloor) && (b4[j] < INFINITY))) bad = 1;
        if (b4[j] <= 0.45f * kFloor) low |= 2;
        if (b4[j] < -30.f) neg |= 2;
        o4[j] = __builtin_fmaf(fast_log2(s4[j]), kLn2, alr + b4[j]);
      }
    }
    st4m(out + at, cc, make_float4(o4[0], o4[1], o4[2], o4[3]));
  }
  const int row_low = __syncthreads_or(low & 1), col_low = __syncthreads_or(low & 2);
  const int row_neg = __syncthreads_or(neg & 1), col_neg = __syncthreads_or(neg & 2);
  if ((row_low && col_neg) || (col_low && row_neg)) bad = 1;
  bad = __syncthreads_or(bad);
  if (tid == 0) flags[tile] = bad;  // the fix-up launch recomputes a flagged tile
  if (tile == 0 && tid == 0) {
    ws_hdr[1] = TR;
    ws_hdr[2] = TC;
    ws_hdr[0] = kWsFast;
  }
}

// ------------------------------------------------------- sampling sweep
// split_slab with the four accumulators finished two at a time: block row 0's products, then block row
// 1's with done(0) - vector work on the finished accumulators, 64 instructions - spread between them.
// done(1) is left to the caller, beside its staging.  Every accumulator takes its products in
// split_slab's order.
template <class SR, class SC, class Done>
__device__ __forceinline__ void split_slab_rows(const unsigned* __restrict__ R, const unsigned* __restrict__ Cs, int wr0,
                                                int wc0, int lane, floatx16 (&acc)[2][2], Done&& done) {
  bf16x8 rh[2], rm[2], rl[2], ch[2], cm[2], cl[2];
  rh[0] = SR::frag(R, 0, wr0, lane);
#pragma unroll
  for (int i = 0; i < 2; ++i) cl[i] = SC::frag(Cs, 2, wc0 + 32 * i, lane);
  rl[0] = SR::frag(R, 2, wr0, lane);
#pragma unroll
  for (int i = 0; i < 2; ++i) ch[i] = SC::frag(Cs, 0, wc0 + 32 * i, lane);
#pragma unroll
  for (int i = 0; i < 2; ++i) cm[i] = SC::frag(Cs, 1, wc0 + 32 * i, lane);
  rm[0] = SR::frag(R, 1, wr0, lane);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_setprio(3);
  auto products = [&](int r) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rh[r], cl[x], acc[r][x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rl[r], ch[x], acc[r][x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rh[r], cm[x], acc[r][x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rm[r], cm[x], acc[r][x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rm[r], ch[x], acc[r][x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[r][x] = mfma_bf16(rh[r], ch[x], acc[r][x]);
  };
  products(0);
  rh[1] = SR::frag(R, 0, wr0 + 32, lane);
  rl[1] = SR::frag(R, 2, wr0 + 32, lane);
  rm[1] = SR::frag(R, 1, wr0 + 32, lane);
  __builtin_amdgcn_sched_barrier(0);
  products(1);
  done(0);
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);
  }
  __builtin_amdgcn_s_setprio(0);
  __builtin_amdgcn_sched_barrier(0);
}

// The sampling sweep described in logbmm_mfma.h: the forward's contraction again on its fp32
// factors EA, EB - cut into their three parts while they are staged, no exponential - with the
// accumulators started at -t, t = u S the cell's target; after every slab of 16 terms a
// register per cell keeps, by a signed-integer minimum over (value with its low six bits
// replaced by 62 - slab; seven bits and 126 - slab for more than 62 slabs: `tmask` = 63 or 127),
// the slab in which the prefix sum passes t and -rem at the start of that slab.  S is the reciprocal of the forward's 1 / S, the targets are shrunk by 2^-22;
// results: that register in idx (negative; its bits of rem and its tag are all that the resolve needs).  The partial products are added in the
// forward's order, so the sums the sweep compares with its targets are the forward's.  A tile
// with a cell whose S is below 2^-40 or not finite, or that lies in a tile the forward
// flagged, sets that flag and leaves: the forward's tile is redone exactly.  128 x 128 tiles of
// four waves with 256 registers (64 accumulators and 64 history registers per lane); any sizes, N >= 4.
//
// What bounds it: matrix instructions (24 a slab and wave) and the vector instructions beside them (128 for the
// history, about 100 to cut and stage) with two waves on a SIMD.  So half of the history is spread between the
// slab's second twelve matrix instructions, no load stands under a branch of a lane's own (pieces beyond an
// edge are read from the last lines and feed cells that are not stored), targets and results change
// places with the accumulator layout in a wave's own LDS strip.  Forward and draw, both gradients of (64, 512^3):
// 642 -> 537 us against loads, targets and stores under a branch per lane or cell - the loads of a slab were
// waited for ahead of the products, a tile's targets formed one trip to memory after the other -, operands put
// together word by word (SplitS) and the history behind all products.
template <class T>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_sample_sweep_split(const float* __restrict__ ws_ea, const float* __restrict__ ws_eb,
                          const elem_t* __restrict__ out, const float* __restrict__ stats,
                          int* __restrict__ flags, const float* __restrict__ ws_r, int32_t* __restrict__ idx,
                          uint64_t seed, uint64_t offset, int M, int K, int N, int tiles_m, int tiles_n, int ftr,
                          int ftc, int ftiles_m, int ftiles_n, int tmask) {
  constexpr int NT = T::NT;
  using SA = SplitT<T::TR, NT>;
  using SB = SplitL<T::TC, NT>;
  constexpr int ST = SB::ST;
  static_assert(T::TR + T::TC == NT, "one shift per thread");
  static_assert(split_lds_words<SA, SB>() >= (NT / 64) * kStripFloats, "");
  __shared__ __attribute__((aligned(16))) unsigned smem[split_lds_words<SA, SB>()];
  auto As = [&](int buf) __attribute__((always_inline)) { return smem + buf * SA::BUF; };
  auto Bs = [&](int buf) __attribute__((always_inline)) { return smem + 2 * SA::BUF + buf * SB::BUF; };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / T::WC) * 64, wn0 = (wave % T::WC) * 64;
  const int per = tiles_m * tiles_n, tile = xcd_tile_id();
  const int batch = tile / per, rem = tile - batch * per;
  const int m0 = (rem / tiles_n) * T::TR, n0 = (rem % tiles_n) * T::TC;
  const float* st = stats + (long)batch * (M + N);

  // ---- the guard.  The flags are the forward's, one per tile of ITS shape (ftr x ftc): S >= 2^-40 and finite
  // wherever a flag is clear.  What `out` adds is its rounding: a cell passes where alpha + beta - out, i.e.
  // -log S as `out` tells it, is at most 40 ln 2 + 1e-3.  While no shift of the tile exceeds 2048 both roundings
  // together stay below 2.5e-4 and no cell can fail; otherwise, and for half types, the cells are looked at.
  int* flag = flags + (batch * ftiles_m + m0 / ftr) * ftiles_n + n0 / ftc;
  int bad = *flag;
  {
    const int line = tid < T::TR ? min(m0 + tid, M - 1) : M + min(n0 + tid - T::TR, N - 1);
    const int look = !kElemF32 || !(__builtin_fabsf(st[line]) <= 2048.f);
    if (__syncthreads_or(look)) {  // uniform
      constexpr int QR = T::TC / 4;  // quads per tile row
      const float lim = kMfmaGuardBits * kLn2 + 1e-3f;
      for (int q = tid; q < T::TR * QR; q += NT) {
        const int r = q / QR, m = m0 + r, n = n0 + (q - r * QR) * 4;
        if (m >= M || n >= N) continue;
        const int cn = clamp4(N - n);
        const float alr = st[m];
        const float4 be4 = ld4m(st + M + n, cn, 0.f), o4 = ld4m(out + ((long)batch * M + m) * N + n, cn, 0.f);
        const float bev[4] = {be4.x, be4.y, be4.z, be4.w}, ov[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = alr + bev[j] - ov[j];  // -log S
          if (j < cn && (!(e <= lim) || !(e > -INFINITY))) bad = 1;
        }
      }
    }
  }
  if (__syncthreads_or(bad)) {
    if (tid == 0) *flag = 1;
    return;
  }

  // ---- targets: -t = -u S for the wave's 64 x 64 cells, a lane four adjacent cells of sixteen rows (they share
  // one Philox block when rows are a multiple of four cells), and on to the accumulator layout through the
  // wave's strip.  Pieces beyond an edge are read from the last lines, a piece astride the right one moved down.
  floatx16 acc[2][2];
  int low[2][2][16];
  float* strip = reinterpret_cast<float*>(smem) + wave * kStripFloats;
  const int lr = lane >> 4, lc = (lane & 15) * 4;
  const long cell0 = (long)batch * M * N;
  {
    const int n = n0 + wn0 + lc, nc = min(n, N - 4), by = n - nc;
    const bool blocks = (N & 3) == 0;
    float4 r4[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) r4[t] = ld4(ws_r + cell0 + (long)min(m0 + wm0 + lr + 4 * t, M - 1) * N + nc);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float u[4], rv[4] = {r4[4 * q + t].x, r4[4 * q + t].y, r4[4 * q + t].z, r4[4 * q + t].w};
        shift_down(rv, by);
        philox_uniform4((uint64_t)(cell0 + (long)(m0 + wm0 + 16 * q + 4 * t + lr) * N + n), blocks, seed, offset, u);
        float tv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) tv[j] = -(u[j] * kSampleShrink) * __builtin_amdgcn_rcpf(rv[j]);
        *reinterpret_cast<float4*>(strip + (lr + 4 * t) * 64 + lc) = make_float4(tv[0], tv[1], tv[2], tv[3]);
      }
      wave_lds_sync();
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float nt = strip[(mfma_row_u(i) + mfma_row_l(lane)) * 64 + c * 32 + (lane & 31)];
          acc[q >> 1][c][(q & 1) * 8 + i] = nt;
          low[q >> 1][c][(q & 1) * 8 + i] = __float_as_int(nt) | tmask;  // all tag bits: no slab has ended below t
        }
      wave_lds_sync();
    }
  }
  __syncthreads();  // the strips make way for the staged slabs

  // ---- staging of EA ([line][reduction]) and EB ([reduction][line]).  A slab's loads are the same whatever it
  // meets - behind a branch the compiler waits for them ahead of the products they should hide behind - so the
  // last slab of a ragged K reads on past the end of its rows (into the workspace array that follows, at the very
  // end) and what lies beyond K is zeroed when it is staged.
  const float* pa[SA::PER];
#pragma unroll
  for (int l = 0; l < SA::PER; ++l)
    pa[l] = ws_ea + ((long)batch * M + min(m0 + SA::line(tid, l), M - 1)) * K + SA::quad(tid) * 4;
  const int brow = SB::step0(tid), bcol = min(n0 + SB::line(tid), N - 1);
  const float* pb = ws_eb + ((long)batch * K + brow) * N;  // uniform
  const int ktail = K % kMS, slabs = (K + kMS - 1) / kMS;
  float4 ra[SA::PER];
  float rb[ST];
  auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) {
      ra[l] = ld4(pa[l]);
      pa[l] += kMS;
    }
#pragma unroll
    for (int j = 0; j < ST; ++j) rb[j] = pb[(long)j * N + bcol];
    pb += (long)kMS * N;
  };
  auto stage = [&](int slab) __attribute__((always_inline)) {
    if (ktail != 0 && slab == slabs - 1) {  // uniform
      const int ca = ktail - SA::quad(tid) * 4;
#pragma unroll
      for (int l = 0; l < SA::PER; ++l)
        ra[l] = make_float4(ca > 0 ? ra[l].x : 0.f, ca > 1 ? ra[l].y : 0.f, ca > 2 ? ra[l].z : 0.f, ca > 3 ? ra[l].w : 0.f);
#pragma unroll
      for (int j = 0; j < ST; ++j) rb[j] = brow + j < ktail ? rb[j] : 0.f;
    }
#pragma unroll
    for (int l = 0; l < SA::PER; ++l) SA::put(As(slab & 1), tid, l, ra[l]);
    SB::put(Bs(slab & 1), tid, rb);
  };
  int keep = ~tmask;
  asm("" : "+v"(keep));  // a vector register: with the tag one v_and_or_b32 per cell (one scalar operand at most)
  auto multiply = [&](int slab) __attribute__((always_inline)) {
    const int tag = (tmask - 1 - slab) & tmask;
    auto history = [&](int r) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          low[r][x][i] = min(low[r][x][i], (__float_as_int(acc[r][x][i]) & keep) | tag);
          asm volatile("" : "+v"(low[r][x][i]));  // here, not sunk behind the staging
        }
    };
    split_slab_rows<SA, SB>(As(slab & 1), Bs(slab & 1), wm0, wn0, lane, acc, history);
    history(1);
  };
  load();
  stage(0);
  __syncthreads();
  for (int s = 0; s + 1 < slabs; ++s) {
    load();
    multiply(s);
    stage(s + 1);
    __syncthreads();
  }
  multiply(slabs - 1);
  __syncthreads();  // every wave is done with the staged slabs

  // ---- the slab in which the prefix passes t, and rem at its start, row by row
  const int cc = clamp4(N - (n0 + wn0 + lc)), rows_left = M - (m0 + wm0) - lr;
  float* dst = reinterpret_cast<float*>(idx) + cell0 + (long)(m0 + wm0) * N + n0 + wn0 + lr * N + lc;  // bit patterns
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int v = low[x >> 1][x & 1][i], below = tmask - (v & tmask);
      // a target that the sums never reach lies within their rounding of the total: the last term
      acc[x >> 1][x & 1][i] = __int_as_float(below >= slabs ? K - 1 : v);
    }
  acc_rows(acc, strip, lane, [](int) {}, [&](int q, int t, float4 v) __attribute__((always_inline)) {
    const int ru = 16 * q + 4 * t;
    if (cc > 0 && ru < rows_left) st4m(dst + (long)ru * N, cc, v);
  });
}

// ---------------------------------------------------------------- backward
// Operands formed from a, b, out, g and the maxima while they are staged (as
// log_bwd_mfma_tile_lean): EA = exp(a - alpha), EB = exp(b - beta), H = g exp(alpha + beta - out).
// GRAD_A: tile (m,k) of grad_a = EA * sum_n H[m][n] EB[k][n]; rows <- H, columns <- EB, both
//         sources [line][reduction].
// GRAD_B: tile (k,n) of grad_b = EB * sum_m EA[m][k] H[m][n]; rows <- EA, columns <- H, both
//         sources [reduction][line].
template <class T, bool GRAD_A>
struct SplitBwd {
  static constexpr int NT = T::NT;
  using SR = std::conditional_t<GRAD_A, SplitT<T::TR, NT>, SplitL<T::TR, NT>>;
  using SC = std::conditional_t<GRAD_A, SplitT<T::TC, NT>, SplitL<T::TC, NT>>;
  static constexpr int WORDS = split_lds_words<SR, SC>();
};

// One cell of a gradient on plain fp32 products, a lane by itself: (r, c) = (m, k) of grad_a, (k, n) of grad_b.
// The sum ends where it is NaN for good.
template <bool GRAD_A, bool RECIP, class W_t>
__device__ __forceinline__ float log_bwd_cell(const elem_t* __restrict__ ab, const elem_t* __restrict__ bb,
                                              const W_t* __restrict__ wb, const elem_t* __restrict__ gb,
                                              const float* __restrict__ al, const float* __restrict__ be, int M, int K,
                                              int N, int r, int c) {
  const int Q = GRAD_A ? N : M;
  float s = 0.f;
  for (int q0 = 0; q0 < Q && s == s; q0 += 16) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int q = min(q0 + u, Q - 1), m = GRAD_A ? r : q, n = GRAD_A ? q : c;
      const long at = (long)m * N + n;
      const float w = (float)wb[at], h = (float)gb[at] * (RECIP ? w : exp_st(al[m] + be[n] - w));
      const float y = GRAD_A ? exp_st((float)bb[(long)c * N + n] - be[n]) : exp_st((float)ab[(long)m * K + r] - al[m]);
      s = q0 + u < Q ? __builtin_fmaf(h, y, s) : s;
    }
  }
  return s * (GRAD_A ? exp_st((float)ab[(long)r * K + c] - al[r]) : exp_st((float)bb[(long)r * N + c] - be[c]));
}

// RECIP: H = g R with the forward's R = 1 / S (fp32, in the workspace) in the place of out and an
// exponential - for float16 / bfloat16 tensors, whose `out` is stored rounded.  The header is read before
// anything else: a workspace of another forward need not hold R.
//
// An infinite H, or one that rounds to an infinite bfloat16 (beyond 0x1.fep127), has no three parts: inf - inf
// makes every sum of its line NaN.  A wave that stores a NaN sum forms such cells again on fp32 products
// (log_bwd_cell), which leaves infinities where they belong and every other cell alone.
template <class T, bool GRAD_A, bool RAGGED, bool RECIP>
__device__ __forceinline__ void log_bwd_split_tile(unsigned* __restrict__ smem, int tile, const elem_t* __restrict__ g,
                                                   const LeanSrc src, const int* __restrict__ ws_hdr,
                                                   const int* __restrict__ fwd_flags, elem_t* __restrict__ grad, int M,
                                                   int K, int N, int tiles_r, int tiles_c) {
  using W = SplitBwd<T, GRAD_A>;
  using SR = typename W::SR;
  using SC = typename W::SC;
  constexpr int NT = T::NT;
  static_assert(W::WORDS >= (NT / 64) * kStripFloats, "");
  auto Rs = [&](int buf) __attribute__((always_inline)) { return smem + buf * SR::BUF; };
  auto Cs = [&](int buf) __attribute__((always_inline)) { return smem + 2 * SR::BUF + buf * SC::BUF; };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr0 = (wave / T::WC) * 64, wc0 = (wave % T::WC) * 64;
  const int per = tiles_r * tiles_c;
  const int batch = tile / per, rem = tile - batch * per;
  const int r0 = (rem / tiles_c) * T::TR, c0 = (rem % tiles_c) * T::TC;
  const int Q = GRAD_A ? N : M;
  const int R = GRAD_A ? M : K, Cc = GRAD_A ? K : N;
  const float* al = src.stats + (long)batch * (M + N);
  const float* be = al + M;
  using W_t = std::conditional_t<RECIP, float, elem_t>;
  const W_t* wsrc;  // what H is formed from beside g: R, or out
  if constexpr (RECIP) wsrc = src.r;
  else wsrc = src.out;
  constexpr int kNeed = RECIP ? kKeepRecip : kKeepNone;
  floatx16 acc[2][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[x >> 1][x & 1][i] = 0.f;
  const int slabs = Q / kMS;                // whole slabs: the loop
  const int qtail = RAGGED ? Q % kMS : 0;   // reduction steps of a partial last slab: one more step behind the
                                            // loop, with a loader of its own (inside the loop's loader it cost
                                            // 19 spilled registers and the kernel ran 1.7 times slower)

  // Addresses are a base per workgroup (scalar registers, stepped slab by slab) plus a fixed
  // 32-bit offset per thread: the vector registers go to operands and accumulators.
  // RAGGED: any sizes (every extent at least a piece).  Fills of the partial last slab make a factor
  // vanish: -inf for a and b, +inf for out, 0 for g.
  if constexpr (GRAD_A) {
    // rows: H pieces (line m, four n); columns: EB pieces (line k, four n); beta of the slab's four
    // columns is the same for every piece of a thread (all share their quad).  Lines beyond the
    // matrix re-read the last line: they only feed results that are not stored.
    const W_t* ob = wsrc + (long)batch * M * N;
    const elem_t* gb = g + (long)batch * M * N;
    const elem_t* bb = src.b + (long)batch * K * N;
    const float* beb = be;
    int oo[SR::PER], yo[SC::PER];
    float alh[SR::PER];
#pragma unroll
    for (int l = 0; l < SR::PER; ++l) {
      const int m = RAGGED ? min(r0 + SR::line(tid, l), M - 1) : r0 + SR::line(tid, l);
      oo[l] = m * N + SR::quad(tid) * 4;
      alh[l] = al[m];
    }
#pragma unroll
    for (int l = 0; l < SC::PER; ++l) {
      const int k = RAGGED ? min(c0 + SC::line(tid, l), K - 1) : c0 + SC::line(tid, l);
      yo[l] = k * N + SC::quad(tid) * 4;
    }
    const int beo = SR::quad(tid) * 4;
    float4 ro[SR::PER], rg[SR::PER], ry[SC::PER], bslab;
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int l = 0; l < SC::PER; ++l) ry[l] = ld4(bb + yo[l]);
#pragma unroll
      for (int l = 0; l < SR::PER; ++l) {
        ro[l] = ld4(ob + oo[l]);
        rg[l] = ld4(gb + oo[l]);
      }
      bslab = ld4(beb + beo);
      ob += kMS; gb += kMS; bb += kMS; beb += kMS;
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int l = 0; l < SC::PER; ++l) SC::put(Cs(buf), tid, l, exp4(ry[l], bslab));
#pragma unroll
      for (int l = 0; l < SR::PER; ++l) {
        if constexpr (RECIP) {
          SR::put(Rs(buf), tid, l, make_float4(rg[l].x * ro[l].x, rg[l].y * ro[l].y, rg[l].z * ro[l].z, rg[l].w * ro[l].w));
        } else {
          const float4 sh = make_float4(alh[l] + bslab.x, alh[l] + bslab.y, alh[l] + bslab.z, alh[l] + bslab.w);
          SR::put(Rs(buf), tid, l, mul_exp4(rg[l], sh, ro[l]));
        }
      }
    };
    if (RECIP && ws_hdr[0] != kWsRecip) return;  // uniform
    load();
    if (bwd_tile_flagged(ws_hdr, fwd_flags, kNeed, true, r0, T::TR, batch, M, N, tid, NT)) return;
    stage(0);
    split_loop(slabs, split_early<NT>(wave), load, stage, [&](int buf) __attribute__((always_inline)) {
      split_slab<SR, SC>(Rs(buf), Cs(buf), wr0, wc0, wave & (NT / 64 - 1), lane, acc);
    });
    if (RAGGED && qtail != 0) {  // uniform
      const int left = qtail - beo;  // all pieces of a thread share their quad
#pragma unroll
      for (int l = 0; l < SC::PER; ++l) ry[l] = ld4m(bb + yo[l], left, -INFINITY);
#pragma unroll
      for (int l = 0; l < SR::PER; ++l) {
        ro[l] = ld4m(ob + oo[l], left, RECIP ? 0.f : INFINITY);
        rg[l] = ld4m(gb + oo[l], left, 0.f);
      }
      bslab = ld4m(beb + beo, left, 0.f);
      stage(0);
      __syncthreads();
      split_slab<SR, SC>(Rs(0), Cs(0), wr0, wc0, wave & (NT / 64 - 1), lane, acc);
      __syncthreads();
    }
  } else {
    // rows: EA, SR::ST steps m of one line k; columns: H, SC::ST steps m of one line n.  Lines beyond the matrix
    // re-read the last one: they only feed results that are not stored.  alpha of the slab's sixteen steps is one
    // load of the wave's, read lane by lane.
    constexpr int NR = SR::ST, NC = SC::ST;
    const int r_s = SR::step0(tid), c_s = SC::step0(tid);  // uniform
    const elem_t* ab = src.a + (long)batch * M * K;
    const W_t* ob = wsrc + (long)batch * M * N;
    const elem_t* gb = g + (long)batch * M * N;
    const float* alb = al;
    const unsigned kc = RAGGED ? min(r0 + SR::line(tid), K - 1) : r0 + SR::line(tid);
    const unsigned nc = RAGGED ? min(c0 + SC::line(tid), N - 1) : c0 + SC::line(tid);
    const unsigned step = lane & (kMS - 1);
    const float bec = be[nc];
    elem_t ry[NR], rg[NC];
    W_t ro[NC];
    float als;
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < NR; ++j) ry[j] = (ab + (long)(r_s + j) * K)[kc];
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        ro[j] = (ob + (long)(c_s + j) * N)[nc];
        rg[j] = (gb + (long)(c_s + j) * N)[nc];
      }
      als = alb[step];
      ab += (long)kMS * K;
      ob += (long)kMS * N;
      gb += (long)kMS * N;
      alb += kMS;
    };
    auto alpha = [&](int m) __attribute__((always_inline)) {
      return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(als), m));
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
      float e[NR], h[NC];
#pragma unroll
      for (int j = 0; j < NR; ++j) e[j] = exp_st((float)ry[j] - alpha(r_s + j));
#pragma unroll
      for (int j = 0; j < NC; ++j)
        h[j] = (float)rg[j] * (RECIP ? (float)ro[j] : exp_st(alpha(c_s + j) + bec - (float)ro[j]));
      SR::put(Rs(buf), tid, e);
      SC::put(Cs(buf), tid, h);
    };
    if (RECIP && ws_hdr[0] != kWsRecip) return;  // uniform
    load();
    if (bwd_tile_flagged(ws_hdr, fwd_flags, kNeed, false, c0, T::TC, batch, M, N, tid, NT)) return;
    stage(0);
    split_loop(slabs, split_early<NT>(wave), load, stage, [&](int buf) __attribute__((always_inline)) {
      split_slab<SR, SC>(Rs(buf), Cs(buf), wr0, wc0, wave & (NT / 64 - 1), lane, acc);
    });
    if (RAGGED && qtail != 0) {  // uniform; steps beyond M re-read row M - 1 and are replaced by the fills
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        ry[j] = (ab + (long)min(r_s + j, qtail - 1) * K)[kc];
        ry[j] = r_s + j < qtail ? ry[j] : (elem_t)-INFINITY;
      }
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const long at = (long)min(c_s + j, qtail - 1) * N;
        ro[j] = (ob + at)[nc];
        rg[j] = (gb + at)[nc];
        rg[j] = c_s + j < qtail ? rg[j] : (elem_t)0.f;
      }
      als = alb[min((int)step, qtail - 1)];
      stage(0);
      __syncthreads();
      split_slab<SR, SC>(Rs(0), Cs(0), wr0, wc0, wave & (NT / 64 - 1), lane, acc);
      __syncthreads();
    }
  }

  // grad = EX * acc with EX = exp(a - alpha) (grad_a) or exp(b - beta) (grad_b), row-wise
  const int lr = lane >> 4, lc = (lane & 15) * 4;
  const int voff = lr * Cc + lc;
  const long ubase = ((long)batch * R + r0 + wr0) * Cc + c0 + wc0;
  const elem_t* xb = (GRAD_A ? src.a : src.b) + ubase + voff;
  elem_t* gp = grad + ubase + voff;
  const int cc = RAGGED ? clamp4(Cc - (c0 + wc0 + lc)) : 4;
  const bool cok = cc > 0;
  const int rows_left = R - (r0 + wr0) - lr;
  float4 becol = make_float4(0.f, 0.f, 0.f, 0.f);
  if constexpr (!GRAD_A) becol = RAGGED ? ld4m(be + (cok ? c0 + wc0 + lc : 0), cc, 0.f) : ld4(be + c0 + wc0 + lc);
  const float* alrow = al + r0 + wr0 + lr;
  float4 xq[2][4];
  float xa[2][4];
  auto fetch = [&](int q) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool live = !RAGGED || (cok && 16 * q + 4 * t < rows_left);
      if (live) {
        xq[q & 1][t] = RAGGED ? ld4m(xb + (long)(16 * q + 4 * t) * Cc, cc, -INFINITY) : ld4(xb + (long)(16 * q + 4 * t) * Cc);
        if constexpr (GRAD_A) xa[q & 1][t] = alrow[16 * q + 4 * t];
      }
    }
  };
  fetch(0);
  bool lost = false;  // a NaN among the sums (or, without harm, two infinities side by side)
  acc_rows(acc, reinterpret_cast<float*>(smem) + wave * kStripFloats, lane,
           [&](int q) __attribute__((always_inline)) { if (q + 1 < 4) fetch(q + 1); },
           [&](int q, int t, float4 v) __attribute__((always_inline)) {
             if (RAGGED && !(cok && 16 * q + 4 * t < rows_left)) return;
             const float any = (v.x + v.y) + (v.z + v.w);
             lost = lost || any != any;
             float4 x;
             if constexpr (GRAD_A) x = exp4(xq[q & 1][t], xa[q & 1][t]);
             else x = exp4(xq[q & 1][t], becol);
             const float4 r = make_float4(x.x * v.x, x.y * v.y, x.z * v.z, x.w * v.w);
             if (RAGGED) st4m(gp + (long)(16 * q + 4 * t) * Cc, cc, r);
             else st4(gp + (long)(16 * q + 4 * t) * Cc, r);
           });
  if (!__any(lost)) return;
  // The wave's NaN cells are listed in its strip of LDS, half a block at a time, and shared out to the lanes: a
  // line's worth would otherwise fall to four of them.  (Where the cells lie is worked out anew: kept from above
  // it cost the largest tile spilled registers.)
  unsigned short* list = reinterpret_cast<unsigned short*>(smem + wave * kStripFloats);
  static_assert(sizeof(float) * kStripFloats >= 2 * 32 * 64, "");
  const int me = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  elem_t* block = grad + ((long)batch * R + r0 + wr0) * Cc + c0 + wc0;
  const int rows = R - r0 - wr0, cols = Cc - c0 - wc0;
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    int count = 0;
    wave_lds_sync();
#pragma unroll 1
    for (int e = 32 * half; e < 32 * half + 32; ++e) {  // the cells this lane has stored: four of every fourth row
      const int r = (me >> 4) + (e & ~3), c = (me & 15) * 4 + (e & 3);
      const float was = r < rows && c < cols ? settled((float)block[(long)r * Cc + c]) : 0.f;
      const unsigned long long hits = __ballot(was != was);
      if (was != was) list[count + __builtin_popcountll(hits & ((1ull << me) - 1))] = (unsigned short)(r * 64 + c);
      count += __builtin_popcountll(hits);
    }
    wave_lds_sync();
#pragma unroll 1
    for (int i = me; i < count; i += 64) {
      const int r = list[i] >> 6, c = list[i] & 63;
      block[(long)r * Cc + c] = to_elem<elem_t>(
          log_bwd_cell<GRAD_A, RECIP>(src.a + (long)batch * M * K, src.b + (long)batch * K * N, wsrc + (long)batch * M * N,
                                      g + (long)batch * M * N, al, be, M, K, N, r0 + wr0 + r, c0 + wc0 + c));
    }
  }
}

// Both gradients in one launch, item by item, a tile of each in turn (see k_log_bwd_mfma_both).
template <class TA, class TB, bool RAGGED, bool RECIP>
__global__ __launch_bounds__(TA::NT) __attribute__((amdgpu_waves_per_eu(TA::WPE, TA::WPE)))
void k_log_bwd_split_both(const elem_t* __restrict__ g, const LeanSrc src, const int* __restrict__ ws_hdr,
                          const int* __restrict__ fwd_flags, elem_t* __restrict__ grad_a,
                          elem_t* __restrict__ grad_b, int M, int K, int N, int ar, int ac, int br, int bc) {
  static_assert(TA::NT == TB::NT && TA::WPE == TB::WPE, "");
  extern __shared__ __attribute__((aligned(16))) unsigned split_smem[];
  const int per_a = ar * ac, per_b = br * bc;
  const int v = xcd_renumber(blockIdx.x, gridDim.x);
  const int item = v / (per_a + per_b), r = v - item * (per_a + per_b);
  const bool alt = per_a == per_b;
  const bool is_a = alt ? (r & 1) == 0 : r < per_a;
  const int idx = alt ? r >> 1 : (r < per_a ? r : r - per_a);
  if (is_a)
    log_bwd_split_tile<TA, true, RAGGED, RECIP>(split_smem, item * per_a + idx, g, src, ws_hdr, fwd_flags, grad_a, M, K, N, ar, ac);
  else
    log_bwd_split_tile<TB, false, RAGGED, RECIP>(split_smem, item * per_b + idx, g, src, ws_hdr, fwd_flags, grad_b, M, K, N, br, bc);
}

template <class TA, class TB>
constexpr int split_bwd_lds_bytes() {
  constexpr int a = SplitBwd<TA, true>::WORDS, b = SplitBwd<TB, false>::WORDS;
  return 4 * (a > b ? a : b);
}

}  // namespace GENBMM_NS
