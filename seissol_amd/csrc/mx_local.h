// The cell-local pass on the matrix cores in the engine's real type
// (v_mfma_f64_16x16x4_f64 / v_mfma_f32_16x16x4_f32): Cauchy-Kowalevski
// predictor and time integral, face traces, volume and local flux
// (Time.cpp:65-140, Local.cpp:124-160; spec codegen/kernels/aderdg.py:321-537).
//
// A workgroup handles a tile of 16 elements.  Every contraction with a global
// matrix is a GEMM Y(M x 16 c) += A(M x K) X(K x 16 c) whose 16 columns of one
// quantity are the 16 elements: lane l holds rows 4g .. 4g + 3 (g = l / 16) of
// element e = l % 16, so the 9 x 9 products that mix quantities are register
// arithmetic.  X lies in LDS ([column][row]); the fragments of A are coalesced
// loads from L2, shared by all workgroups.
//
// What bounds it: the matrix instructions (64 cycles per 16 x 16 x 4 and SIMD
// in FP64, 32 in FP32) would take a third of its time, HBM less.  The rest is
// the serial chain of a tile (O - 1 derivatives, volume, traces, flux with
// barriers between them) at two to four waves per SIMD, so the pass lives from
// workgroups overlapping their phases, from few instructions, and from waits
// taken out of the chain:
//  * The elastic star matrices couple velocities with stresses only.  Stresses
//    are formed as sum_q (A_j X_q) star_j(q, p): 9 products per k-step and row
//    tile (3 directions, 3 velocities).  Velocities are formed as
//    A_j (sum_q X_q star_j(q, p)), mixed on the way from LDS to the operand: 9
//    products as well, where contracting afterwards needs 18.
//  * The basis is hierarchical: a derivative matrix has zeros left (predictor)
//    or right (volume) of a degree, so each row tile multiplies only the
//    k-steps that hold its non-zeros (host-computed ranges, so that a caller's
//    own matrices give their own ranges): 51 of 69 k-steps of the predictor, 26
//    of 56 of the volume, 68 of 84 of the traces at ORDER 6.
//  * Fragments come from L2, 700 cycles away even on an idle chip: each wave
//    reads them as one stream that runs ahead over row tiles, directions and
//    barriers; the last three derivatives' block is kept in LDS.  The star
//    values and, in FP32, the AplusT columns are read ahead of their use.
//    60k cells, before -> after these: FP32 ORDER 4 116 -> 100 us, ORDER 5 246
//    -> 210, ORDER 6 360 -> 333, ORDER 7 959 -> 769; FP64 ORDER 3 193 -> 169,
//    ORDER 4 283 -> 264, ORDER 5 511 -> 467, ORDER 6 827 -> 737, ORDER 7 1507
//    -> 1457; 500 cells at ORDER 4 (FP64) 25.3 -> 21.1.
//  * dQ_1 and dQ_2 share the X area, later derivatives alternate between the
//    two places: one barrier per derivative from dQ_2 on.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "dpp_rows.h"
#include "mx_common.h"

namespace sdg {
namespace mx {
namespace {

// the block of the predictor matrices kept in LDS (see lateStress)
constexpr int kLateRows = 10, kLateSteps = 5, kLate = 3 * kLateSteps * 4 * kLateRows;

// Waves of the local pass: a pair has one or two row tiles, pair and
// 2 PAIRS - 1 - pair (low tiles have the long products of the predictor, high
// ones those of the volume); its first wave forms the stresses, its second the
// velocities, which cost the same.  Two tiles share a velocity wave's mixing
// and operand reads: one tile per wave, with twice the waves in flight, was
// slower (FP32 60k cells: ORDER 5 219 -> 257 us, ORDER 6 340 -> 359) except
// for FP32 at ORDER 7, where one workgroup's waves fill the CU (892 -> 816).
template <int O, typename real>
struct Waves {
  using G = Geo<O>;
  static constexpr int PAIRS = O == 3 ? 1 : (O == 7 ? (sizeof(real) == 8 ? 4 : 6) : 2);
  static constexpr int WAVES = 2 * PAIRS, THREADS = 64 * WAVES;
  static constexpr int TW = G::MT > PAIRS ? 2 : 1;   // row tiles per wave
  static constexpr int TT = G::MTF > WAVES ? 2 : 1;  // trace tiles per wave
};

// LDS of the local kernel, in reals
template <int O, typename real>
struct LocalLds {
  using G = Geo<O>;
  using N = Waves<O, real>;
  static constexpr int LD = columnStride<real>(G::XROWS);
  static constexpr int X = maxOf(kCols * LD, kElems * kAplusLd<real>);
  static constexpr int bytes = (X + kElems * kStarLd + kLate) * static_cast<int>(sizeof(real));
  static constexpr int GROUPS = 163840 / bytes;  // workgroups per CU that the LDS allows
  // waves per SIMD asked of the register allocator
  static constexpr int wanted = GROUPS * N::WAVES / 4;
  static constexpr int cap = sizeof(real) == 8 ? 2 : (N::TW == 1 ? 4 : 3);
  static constexpr int SIMD_WAVES = wanted < 1 ? 1 : (wanted < cap ? wanted : cap);
};

// a run of fragments [j][KS][64] of one row tile: k-steps [lo, hi) of the three directions
template <typename real>
struct Run {
  const real* fr;
  int lo, hi;
};

// k-steps of fragments loaded ahead by the products below (FP64 has no
// registers for more)
template <typename real>
struct Ahead {
  static constexpr int stress = sizeof(real) == 8 ? 4 : 8, velocity = 2, trace = sizeof(real) == 8 ? 2 : 4;
};

// registers to spare: FP32, and FP64 at low orders
template <int O, typename real>
constexpr bool kRoomy = sizeof(real) == 4 || O <= 4;

// the star values of one direction that feed the stresses, read ahead of the
// direction's products (ROOMY) or two quantities ahead of their use
template <typename real, bool ROOMY>
struct StressStar {
  static constexpr int AHEAD = ROOMY ? 6 : 2;
  real v[6][3];
  const real* at;
  __device__ inline void read(int p) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < kStarCnt[p]) v[p][k] = at[kStarOff[p] + k];
  }
  __device__ inline StressStar(const real* sS, int j) {
    int off = 24 * j;
    asm volatile("" : "+v"(off));  // else the compiler reads the three directions' values at once
    at = sS + off;
    if (AHEAD == 6)
#pragma unroll
      for (int p = 0; p < 6; ++p) read(p);
  }
  // y[p] += sum_q acc_q star_j(q, p), acc_q = A_j X_q of the velocities q = 6 .. 8;
  // the sums are finished before the next direction's products start (else
  // three directions' accumulators stay live)
  __device__ inline void add(const typename Vec<real>::V4 (&acc)[3], typename Vec<real>::V4 (&y)[6]) {
    if (AHEAD < 6)
#pragma unroll
      for (int p = 0; p < AHEAD; ++p) read(p);
#pragma unroll
    for (int p = 0; p < 6; ++p) {
      if (p + AHEAD < 6) read(p + AHEAD);
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (k < kStarCnt[p]) y[p] += acc[kStarQ[p][k] - 6] * v[p][k];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        real t = y[p][r];
        asm volatile("" : "+v"(t));
        y[p][r] = t;
      }
    }
  }
};

template <typename real>
__device__ inline void loadStress(const Run<real>& run, int lane, real (&cur)[Ahead<real>::stress]) {
#pragma unroll
  for (int u = 0; u < Ahead<real>::stress; ++u) cur[u] = run.fr[min(run.lo + u, run.hi - 1) * 64 + lane];
}

// y[p][.] += sum_j sum_q (A_j X_q) star_j(q, p) for the stresses p < 6 of one
// row tile.  x: the lane's column of quantity 0 at row g.  The fragments form
// one stream over the directions and on into the next run: `cur` holds this
// run's first k-steps on entry and the next run's on return, so that their
// latency passes behind the products and the barrier between the runs.
template <int KS, int LD, bool ROOMY, typename real>
__device__ inline void starStress(const Run<real>& run, const Run<real>& next, const real* x, const real* sS, int lane,
                                  typename Vec<real>::V4 (&y)[6], real (&cur)[Ahead<real>::stress]) {
  using V4 = typename Vec<real>::V4;
  constexpr int U = Ahead<real>::stress;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    StressStar<real, ROOMY> star(sS, j);
    V4 acc[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] = V4{0, 0, 0, 0};
#pragma unroll 1
    for (int k = run.lo; k < run.hi; k += U) {
      const bool last = k + U >= run.hi;
      const real* const fr = last ? (j < 2 ? run.fr + (j + 1) * KS * 64 : next.fr) : run.fr + j * KS * 64;
      const int at = last ? (j < 2 ? run.lo : next.lo) : k + U, end = last && j == 2 ? next.hi : run.hi;
      real nxt[U];
#pragma unroll
      for (int u = 0; u < U; ++u) nxt[u] = fr[min(at + u, end - 1) * 64 + lane];
      // operands of XU k-steps at a time, read ahead of the branches
      constexpr int XU = sizeof(real) == 8 ? 1 : 4;
#pragma unroll
      for (int u0 = 0; u0 < U; u0 += XU) {
        real v[XU][3];
#pragma unroll
        for (int u = 0; u < XU; ++u)
#pragma unroll
          for (int i = 0; i < 3; ++i) v[u][i] = x[(6 + i) * 16 * LD + 4 * min(k + u0 + u, run.hi - 1)];
#pragma unroll
        for (int u = 0; u < XU; ++u)
          if (k + u0 + u < run.hi) {
#pragma unroll
            for (int i = 0; i < 3; ++i) acc[i] = mma(cur[u0 + u], v[u][i], acc[i]);
          }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = nxt[u];
    }
    star.add(acc, y);
  }
}

// the velocities' operand sum_q X_q star_j(q, 6 + i) of one k-step
template <typename real>
__device__ inline void mixVelocity(const real (&s)[9], const real (&v)[6], real (&m)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
    m[i] = s[3 * i] * v[kStarQ[6 + i][0]] + s[3 * i + 1] * v[kStarQ[6 + i][1]] + s[3 * i + 2] * v[kStarQ[6 + i][2]];
}

// the union of the tiles' k-steps (lo >= hi: no work)
template <int KS, int TW, typename real>
__device__ inline void velocityRange(const Run<real> (&run)[TW], int& k0, int& k1) {
  k0 = KS;
  k1 = 0;
#pragma unroll
  for (int t = 0; t < TW; ++t)
    if (run[t].lo < run[t].hi) {
      k0 = min(k0, run[t].lo);
      k1 = max(k1, run[t].hi);
    }
}

template <int KS, int TW, typename real>
__device__ inline void loadVelocity(const Run<real> (&run)[TW], int k, int k1, int lane,
                                    real (&cur)[Ahead<real>::velocity][TW][3]) {
#pragma unroll
  for (int u = 0; u < Ahead<real>::velocity; ++u)
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) cur[u][t][j] = run[t].fr[(j * KS + max(min(k + u, k1 - 1), 0)) * 64 + lane];
}

// y[t][i][.] += sum_j A_j (sum_q X_q star_j(q, 6 + i)) for the velocities of
// up to TW row tiles (lo >= hi: none); `cur` and `next` as above
template <int KS, int LD, int TW, typename real>
__device__ inline void starVelocity(const Run<real> (&run)[TW], const Run<real> (&next)[TW], const real* x,
                                    const real* sS, int lane, typename Vec<real>::V4 (&y)[TW][3],
                                    real (&cur)[Ahead<real>::velocity][TW][3]) {
  using V4 = typename Vec<real>::V4;
  constexpr int U = Ahead<real>::velocity;
  int k0, k1, n0, n1;
  velocityRange<KS, TW, real>(run, k0, k1);
  velocityRange<KS, TW, real>(next, n0, n1);
  if (k0 >= k1) return;
  real s[3][9];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 9; ++i) s[j][i] = sS[24 * j + kStarOff[6] + i];
  V4 acc[TW][3];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[t][i] = y[t][i];
#pragma unroll 1
  for (int k = k0; k < k1; k += U) {
    const bool last = k + U >= k1;
    Run<real> ahead[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) ahead[t].fr = last ? next[t].fr : run[t].fr;
    real nxt[U][TW][3];
    loadVelocity<KS, TW, real>(ahead, last ? n0 : k + U, last ? n1 : k1, lane, nxt);
    real v[U][6];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < 6; ++q) v[u][q] = x[q * 16 * LD + 4 * min(k + u, k1 - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k + u < k1) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          real m[3];
          mixVelocity<real>(s[j], v[u], m);
#pragma unroll
          for (int t = 0; t < TW; ++t)
            if (k + u >= run[t].lo && k + u < run[t].hi) {
#pragma unroll
              for (int i = 0; i < 3; ++i) acc[t][i] = mma(cur[u][t][j], m[i], acc[t][i]);
            }
        }
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int j = 0; j < 3; ++j) cur[u][t][j] = nxt[u][t][j];
  }
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int i = 0; i < 3; ++i) y[t][i] = acc[t][i];
}

// The last three derivatives have at most 10 rows and come from at most 20:
// one row tile, so one pair of waves works while the others wait.  Their
// products are too short to hide a fragment's way from L2, so the leading
// 10 x 20 block of the three matrices is kept in LDS, [direction][k-step][g][row].
// KL: k-steps; a: the lane's entry of the block
template <int KL, int LD, bool ROOMY, typename real>
__device__ inline void lateStress(const real* a, const real* x, const real* sS, typename Vec<real>::V4 (&y)[6]) {
  using V4 = typename Vec<real>::V4;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    StressStar<real, ROOMY> star(sS, j);
    V4 acc[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] = V4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < KL; ++k)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        acc[i] = mma(a[(j * kLateSteps + k) * 4 * kLateRows], x[(6 + i) * 16 * LD + 4 * k], acc[i]);
    star.add(acc, y);
  }
}
template <int KL, int LD, typename real>
__device__ inline void lateVelocity(const real* a, const real* x, const real* sS, typename Vec<real>::V4 (&y)[3]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    real s[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) s[i] = sS[24 * j + kStarOff[6] + i];
#pragma unroll
    for (int k = 0; k < KL; ++k) {
      real v[6], m[3];
#pragma unroll
      for (int q = 0; q < 6; ++q) v[q] = x[q * 16 * LD + 4 * k];
      mixVelocity<real>(s, v, m);
#pragma unroll
      for (int i = 0; i < 3; ++i) y[i] = mma(a[(j * kLateSteps + k) * 4 * kLateRows], m[i], y[i]);
    }
  }
}

// acc[q] += A(tile) X_q, q < NQ, over the k-steps of `run`, which are stored
// from the last rows of X to the first: the high degrees, small in a smooth
// solution and with many columns that feed few rows, are summed first, so that
// a matrix instruction, which rounds every product it adds, has smaller sums to
// round (error of the traces' products at ORDER 6 1.9e-7 -> 1.1e-7 in FP32); x:
// the lane's column of the first quantity at row g; `cur` and `next` as above
template <int KS, int LD, int NQ, int U, typename real>
__device__ inline void gemm(typename Vec<real>::V4 (&acc)[NQ], const Run<real>& run, const Run<real>& next,
                            const real* x, int lane, real (&cur)[U]) {
#pragma unroll 1
  for (int k = run.lo; k < run.hi; k += U) {
    const bool last = k + U >= run.hi;
    const real* const fr = last ? next.fr : run.fr;
    const int at = last ? next.lo : k + U, end = last ? next.hi : run.hi;
    real nxt[U];
#pragma unroll
    for (int u = 0; u < U; ++u) nxt[u] = fr[min(at + u, end - 1) * 64 + lane];
    constexpr int XU = sizeof(real) == 8 ? 1 : 2;
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += XU) {
      real v[XU][NQ];
#pragma unroll
      for (int u = 0; u < XU; ++u)
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[u][q] = x[q * 16 * LD + 4 * (KS - 1 - min(k + u0 + u, run.hi - 1))];
#pragma unroll
      for (int u = 0; u < XU; ++u)
        if (k + u0 + u < run.hi) {
#pragma unroll
          for (int q = 0; q < NQ; ++q) acc[q] = mma(cur[u0 + u], v[u][q], acc[q]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) cur[u] = nxt[u];
  }
}

// W = T A for the four rows of a lane's quad, two rows at a time (more
// outgrow the registers); A is read at lds[at + 9 p + q], one column at a
// time (else all 81 entries are loaded at once), ahead of its use (ROOMY)
template <typename real, bool ROOMY>
__device__ inline void mixRows(typename Vec<real>::V4 (&t)[9], const real* lds, int at, bool zero) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    constexpr int N = ROOMY ? 2 : 1;  // columns in flight
    real w0[9], w1[9], a[N][9];
    auto column = [&](int p, real(&c)[9]) {
      int col = at + 9 * p;
      asm volatile("" : "+v"(col));
#pragma unroll
      for (int q = 0; q < 9; ++q) c[q] = lds[col + q];
    };
    if (N == 2) column(0, a[0]);
#pragma unroll
    for (int p = 0; p < 9; ++p) {
      if (p + N - 1 < 9) column(p + N - 1, a[(p + N - 1) % N]);
      real s0 = real(0), s1 = real(0);
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        s0 += t[q][2 * h] * a[p % N][q];
        s1 += t[q][2 * h + 1] * a[p % N][q];
      }
      w0[p] = zero ? real(0) : s0;
      w1[p] = zero ? real(0) : s1;
      asm volatile("" : "+v"(w0[p]), "+v"(w1[p]));
    }
#pragma unroll
    for (int p = 0; p < 9; ++p) {
      t[p][2 * h] = w0[p];
      t[p][2 * h + 1] = w1[p];
    }
  }
}

template <typename real, int O>
struct LocalArgs {
  int64_t E0;  // the tile's first cell
  int cells;   // its cells: columns beyond load zeros and store nothing
  int reset;
  const real* frag;
  const int* ranges;
  const real (&c)[O];
  real* dofs;
  real* integ;
  real* traces;
  const real* star;
  const real* aplus;
  const uint8_t* faceTypes;
  const CellLayout& lay;
  const LtsOut& lts;
};

// Into LDS: the compact star values of the tile, [element][3][24], and with
// LATE the leading block of the predictor matrices; all loads of a thread are
// in flight before its first store
template <typename real, int O, bool LATE>
__device__ inline void stage(const LocalArgs<real, O>& A, real* const sStar, real* const sLate) {
  using G = Geo<O>;
  constexpr int THREADS = Waves<O, real>::THREADS, N = cdiv(kElems * 72, THREADS), NL = LATE ? cdiv(kLate, THREADS) : 1;
  const int64_t E0 = A.E0;
  const int cells = A.cells;
  const CellLayout& lay = A.lay;
  const Buffer<real> star(A.star + E0 * lay.starStride, (cells - 1) * lay.starStride + (lay.starCompact ? 72 : 243));
  const int stride = static_cast<int>(lay.starStride) * static_cast<int>(sizeof(real));
  real v[N], l[NL];
  auto offset = [&](int u, bool compact) {
    const int i = threadIdx.x + u * THREADS, r = i % 72;
    const int at = compact ? r : 81 * (r / 24) + kStarPos[r % 24];
    return i / 72 < cells ? (i / 72) * stride + at * static_cast<int>(sizeof(real)) : kNowhere;
  };
  if (lay.starCompact) {  // uniform: the compact format needs no position table
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = star.load1(offset(u, true), 0);
  } else {
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = star.load1(offset(u, false), 0);
  }
  if constexpr (LATE) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int i = min(static_cast<int>(threadIdx.x) + u * THREADS, kLate - 1);
      const int row = i % kLateRows, g = i / kLateRows % 4, k = i / (4 * kLateRows) % kLateSteps;
      const int j = i / (4 * kLateRows * kLateSteps);
      l[u] = A.frag[G::ck + (j * G::KS + min(k, G::KS - 1)) * 64 + 16 * g + fragRow<real>(row)];
    }
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int i = threadIdx.x + u * THREADS;
    if (i < kElems * 72) sStar[(i / 72) * kStarLd + i % 72] = v[u];
  }
  if constexpr (LATE) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int i = threadIdx.x + u * THREADS;
      if (i < kLate) sLate[i] = l[u];
    }
  }
}

// One wave's share of a tile: the stresses (VEL = false) or the velocities of
// its row tiles.  Both instantiations run the same sequence of barriers, each
// wave of the workgroup one of them.
template <typename real, int O, int PARTS, bool LTS, bool VEL>
__device__ inline void localWave(const LocalArgs<real, O>& A, real* const xs, real* const sStar, real* const sLate,
                                 const int w) {
  using G = Geo<O>;
  using V4 = typename Vec<real>::V4;
  constexpr int B = G::B, LD = LocalLds<O, real>::LD, KS = G::KS, B2P = G::B2P;
  constexpr int THREADS = Waves<O, real>::THREADS, TW = Waves<O, real>::TW, PAIRS = Waves<O, real>::PAIRS;
  constexpr int NP = VEL ? 3 : 6, P0 = VEL ? 6 : 0, RS = sizeof(real);
  const CellLayout& lay = A.lay;
  const int lane = threadIdx.x & 63, g = lane >> 4, e = lane & 15;
  int tile[TW];
  tile[0] = w >> 1;
  if constexpr (TW == 2) tile[1] = 2 * PAIRS - 1 - (w >> 1);
  const int64_t E0 = A.E0;
  const int cells = A.cells;
  const Buffer<real> dofs(A.dofs + E0 * lay.qStride, cells * lay.qStride);
  const Buffer<real> integ(A.integ + E0 * lay.qStride, A.integ != nullptr ? cells * lay.qStride : 0);
  const int cell = e < cells ? e * static_cast<int>(lay.qStride) * RS : kNowhere;
  const int ldq = lay.ldq * RS;  // bytes between quantities

  real* const xq = xs + (P0 * 16 + e) * LD;  // the wave's first quantity, the lane's element
  const real* const xr = xs + e * LD + g;    // operand reads: quantity 0, row g
  const real* const sS = sStar + e * kStarLd;
  auto toX = [&](const V4(&v)[TW][NP]) {
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int row = 16 * tile[t] + 4 * g;
      if (row < G::KB)
#pragma unroll
        for (int p = 0; p < NP; ++p) *reinterpret_cast<V4*>(xq + p * 16 * LD + row) = v[t][p];
    }
  };

  // fragments of the wave's row tiles in step d of the predictor (d = 0: the volume)
  auto run = [&](int d, int t) {
    const bool has = d == 0 ? tile[t] < G::MT : 16 * tile[t] < basis3(O - d);
    const int row = has ? tile[t] : 0, at = d == 0 ? G::rVol + 2 * row : G::rCk + 2 * ((d - 1) * G::MT + row);
    const int hi = A.ranges[at + 1];
    return Run<real>{A.frag + (d == 0 ? G::vol : G::ck) + static_cast<int64_t>(row) * 3 * KS * 64,
                     has ? A.ranges[at] : hi, hi};
  };
  real ahead[VEL ? Ahead<real>::velocity * TW * 3 : Ahead<real>::stress];
  auto& aheadS = reinterpret_cast<real(&)[Ahead<real>::stress]>(ahead);
  auto& aheadV = reinterpret_cast<real(&)[Ahead<real>::velocity][TW][3]>(ahead);
  // the first fragments of `runs`
  auto preload = [&](const Run<real>(&runs)[TW]) {
    if constexpr (VEL) {
      int k0, k1;
      velocityRange<KS, TW, real>(runs, k0, k1);
      loadVelocity<KS, TW, real>(runs, k0, k1, lane, aheadV);
    } else {
      loadStress<real>(runs[0], lane, aheadS);
    }
  };
  // y += the star products of `runs`, then on to the fragments of `next`
  auto product = [&](const Run<real>(&runs)[TW], const Run<real>(&next)[TW], const real* x, V4(&y)[TW][NP]) {
    if constexpr (VEL) {
      starVelocity<KS, LD, TW, real>(runs, next, x, sS, lane, y, aheadV);
    } else {
#pragma unroll
      for (int t = 0; t < TW; ++t)
        if (runs[t].lo < runs[t].hi) {
          if (TW == 2 && t == 0)
            starStress<KS, LD, kRoomy<O, real>, real>(runs[0], runs[1].lo < runs[1].hi ? runs[1] : next[0], x, sS, lane, y[0], aheadS);
          else
            starStress<KS, LD, kRoomy<O, real>, real>(runs[t], next[0], x, sS, lane, y[t], aheadS);
        }
    }
  };

  // ia: the time integral of the wave's rows and quantities
  V4 ia[TW][NP];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int p = 0; p < NP; ++p)
      ia[t][p] = ((PARTS & kPredict) ? dofs : integ).template loadQuad<B>(cell, 16 * tile[t] + 4 * g, (P0 + p) * ldq);
  stage<real, O, (PARTS & kPredict) != 0>(A, sStar, sLate);
  Run<real> runs[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t) runs[t] = run((PARTS & kPredict) && O > 4 ? 1 : 0, t);
  if constexpr ((PARTS & kPredict) == 0 || O > 4) preload(runs);
  toX(ia);

  if constexpr ((PARTS & kPredict) != 0) {
    [[maybe_unused]] unsigned setup = 0;
    [[maybe_unused]] int myDeriv = kNowhere;
    const Buffer<real> deriv(static_cast<real*>(A.lts.deriv) + E0 * lay.dsize,
                             A.lts.deriv != nullptr ? cells * lay.dsize : 0);
    if constexpr (LTS) {
      setup = A.lts.setup != nullptr ? A.lts.setup[E0 + min(e, cells - 1)] : SDG_LTS_HAS_BUFFERS | SDG_LTS_HAS_DERIVATIVES;
      if (e < cells && (setup & SDG_LTS_HAS_DERIVATIVES)) myDeriv = e * static_cast<int>(lay.dsize) * RS;
      if (A.lts.deriv != nullptr) {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
          for (int p = 0; p < NP; ++p) deriv.storeQuad(ia[t][p], myDeriv, 16 * tile[t] + 4 * g, B, (P0 + p) * ldq);
      }
    }
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int p = 0; p < NP; ++p) ia[t][p] *= A.c[0];
    __syncthreads();
    [[maybe_unused]] int doff = 9 * ldq;
    // dQ_{d-1} is read at row source(d), dQ_d stored at row target(d)
    auto source = [](int d) { return d >= 3 && (d & 1) ? G::R1 : 0; };
    auto target = [](int d) { return d & 1 ? 0 : G::R1; };
    // dQ_d of row tile t: into X, the time integral and the derivatives
    auto finish = [&](int d, int m, int t, V4(&y)[NP]) {
      const int row = 16 * tile[t] + 4 * g, ldm = lay.rows(m) * RS;
      const real cd = A.c[d];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int r = 0; r < 4; ++r) y[p][r] = row + r < m ? y[p][r] : real(0);
        ia[t][p] += cd * y[p];
      }
      if (row < m)
#pragma unroll
        for (int p = 0; p < NP; ++p) *reinterpret_cast<V4*>(xq + p * 16 * LD + target(d) + row) = y[p];
      if constexpr (LTS) {
        if (A.lts.deriv != nullptr)
#pragma unroll
          for (int p = 0; p < NP; ++p) deriv.storeQuad(y[p], myDeriv, row, m, doff + (P0 + p) * ldm);
      }
    };
#pragma unroll 1
    for (int d = 1; d < O - 3; ++d) {
      const int m = basis3(O - d);
      Run<real> next[TW];
#pragma unroll
      for (int t = 0; t < TW; ++t) next[t] = run(d + 1 < O - 3 ? d + 1 : d, t);
      V4 y[TW][NP];
#pragma unroll
      for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int p = 0; p < NP; ++p) y[t][p] = V4{0, 0, 0, 0};
      product(runs, next, xr + source(d), y);
      if (d == 1) __syncthreads();  // dQ_1 takes the place of Q
#pragma unroll
      for (int t = 0; t < TW; ++t)
        if (16 * tile[t] < m) finish(d, m, t, y[t]);
      if constexpr (LTS) doff += 9 * lay.rows(m) * RS;
#pragma unroll
      for (int t = 0; t < TW; ++t) runs[t] = next[t];
      __syncthreads();
    }
    // the last derivatives: row tile 0 only
    const real* const late = sLate + g * kLateRows + min(fragRow<real>(e), kLateRows - 1);
    staticFor<3>([&](auto dI) {
      constexpr int d = O - 3 + decltype(dI)::value;
      if constexpr (d >= 1) {
        constexpr int m = basis3(O - d), KL = cdiv(basis3(O - d + 1), 4);
        V4 y[NP];
        if (w < 2) {
#pragma unroll
          for (int p = 0; p < NP; ++p) y[p] = V4{0, 0, 0, 0};
          if constexpr (VEL) lateVelocity<KL, LD, real>(late, xr + source(d), sS, y);
          else lateStress<KL, LD, kRoomy<O, real>, real>(late, xr + source(d), sS, y);
        }
        if constexpr (d == 1) __syncthreads();  // dQ_1 takes the place of Q
        if (w < 2) finish(d, m, 0, y);
        if constexpr (LTS) doff += 9 * lay.rows(m) * RS;
        __syncthreads();
      }
    });
    // the time integral: output (LTS: the buffer, stored or accumulated)
    if (A.integ != nullptr) {
      int mine = cell;
      if constexpr (LTS) mine = (setup & SDG_LTS_HAS_BUFFERS) ? cell : kNowhere;
      [[maybe_unused]] int before = kNowhere;  // the old buffer, where it accumulates (else zeros are loaded)
      if constexpr (LTS)
        before = A.lts.setup != nullptr && !A.reset && (setup & SDG_LTS_ACCUMULATE_BUFFERS) ? mine : kNowhere;
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const int row = 16 * tile[t] + 4 * g;
        V4 out[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          out[p] = V4{0, 0, 0, 0};
          if constexpr (LTS) out[p] = integ.template loadQuad<B>(before, row, (P0 + p) * ldq);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) integ.storeQuad(out[p] + ia[t][p], mine, row, B, (P0 + p) * ldq);
      }
    }
    if constexpr ((PARTS & kFlux) != 0) toX(ia);  // the barrier after the last derivative freed the area
  }
  if constexpr ((PARTS & kFlux) != 0) {
    if constexpr ((PARTS & kPredict) != 0) {
#pragma unroll
      for (int t = 0; t < TW; ++t) runs[t] = run(0, t);
      preload(runs);
    }
    __syncthreads();
    // volume: sum_j kDivM_j I star_j, the initial value of the flux accumulators
    V4 acc[TW][NP];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int p = 0; p < NP; ++p) acc[t][p] = V4{0, 0, 0, 0};
    // the wave's trace tiles (the second, where there is one, goes to the
    // velocity waves, which hold fewer registers), their first fragments loaded
    // ahead of the volume products
    constexpr int TT = VEL ? Waves<O, real>::TT : 1, U = Ahead<real>::trace;
    int tt[TT];
    tt[0] = w;
    if constexpr (TT == 2) tt[1] = 2 * PAIRS + (w >> 1);
    Run<real> trace[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const int row = min(tt[t], G::MTF - 1);
      trace[t] = {A.frag + G::trace + static_cast<int64_t>(row) * KS * 64, A.ranges[G::rTrace + 2 * row],
                  A.ranges[G::rTrace + 2 * row + 1]};
    }
    real aheadT[U];
#pragma unroll
    for (int u = 0; u < U; ++u) aheadT[u] = trace[0].fr[min(trace[0].lo + u, trace[0].hi - 1) * 64 + lane];
    // one value of each 128-byte line of the tile's AplusT, to have it in L2
    // when it is staged (1M cells in FP32 at ORDER 6: 5.00 -> 4.93 ms, 400k in
    // FP64: 4.58 -> 4.46; at the lower FP32 orders, which have more workgroups
    // in flight, it cost 1 %)
    constexpr int LINES = RS == 8 || O >= 6 ? cdiv(324 * RS, 128) : 0, NT = cdiv(kElems * LINES, THREADS);
    const Buffer<real> aplus(A.aplus + E0 * lay.aplusStride, (cells - 1) * lay.aplusStride + 324);
    real touch[NT > 0 ? NT : 1];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int i = threadIdx.x + u * THREADS, el = i / maxOf(LINES, 1);
      touch[u] = aplus.load1(el < cells ? el * static_cast<int>(lay.aplusStride) * RS + i % maxOf(LINES, 1) * 128 : kNowhere, 0);
    }
    product(runs, runs, xr, acc);
    // face traces rT_f I
    V4 tr[TT][9];
    const Buffer<real> traces(A.traces + E0 * 36 * B2P, A.traces != nullptr ? cells * 36 * B2P : 0);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int q = 0; q < 9; ++q) tr[t][q] = V4{0, 0, 0, 0};
      if (tt[t] < G::MTF) {
        gemm<KS, LD, 9, U, real>(tr[t], trace[t], trace[t + 1 < TT ? t + 1 : t], xr, lane, aheadT);
        const int f = G::traceFace(tt[t], g), row = G::traceRow(tt[t], g);
        if (A.traces != nullptr) {
          const int at = e < cells && row < B2P ? ((e * 4 + f) * 9 * B2P + row) * RS : kNowhere;
#pragma unroll
          for (int q = 0; q < 9; ++q) traces.store4(tr[t][q], at, q * B2P * RS);
        }
      }
    }
    // AplusT of the four faces takes the X area, in 16-byte pieces and two
    // batches: the first is in flight across the barrier, and a whole one would
    // outgrow the registers
    {
      typedef real VP __attribute__((ext_vector_type(16 / RS)));
      constexpr int W = 16 / RS, PIECES = 324 / W, N = cdiv(kElems * PIECES, THREADS), N1 = N / 2;
#pragma unroll
      for (int u = 0; u < NT; ++u) asm volatile("" ::"v"(touch[u]));
      const int stride = static_cast<int>(lay.aplusStride);
      auto load = [&](int u) {
        const int i = threadIdx.x + u * THREADS, el = i / PIECES;
        return aplus.load16(el < cells ? (el * stride + i % PIECES * W) * RS : kNowhere);
      };
      auto store = [&](int u, const VP& v) {
        const int i = threadIdx.x + u * THREADS;
        if (i < kElems * PIECES) *reinterpret_cast<VP*>(xs + (i / PIECES) * kAplusLd<real> + i % PIECES * W) = v;
      };
      VP v[N - N1];
#pragma unroll
      for (int u = 0; u < N1; ++u) v[u] = load(u);
      __syncthreads();  // I is no longer read
#pragma unroll
      for (int u = 0; u < N1; ++u) store(u, v[u]);
#pragma unroll
      for (int u = N1; u < N; ++u) v[u - N1] = load(u);
#pragma unroll
      for (int u = N1; u < N; ++u) store(u, v[u - N1]);
    }
    __syncthreads();
    // W = traces AplusT_f, a quad's rows with its own face's matrix; DR faces give none
#pragma unroll
    for (int t = 0; t < TT; ++t)
      if (tt[t] < G::MTF) {
        const int f = G::traceFace(tt[t], g) & 3;
        bool dr = false;
        if (A.faceTypes != nullptr) dr = A.faceTypes[(E0 + min(e, cells - 1)) * 4 + f] == SDG_FACE_DYNAMIC_RUPTURE;
        mixRows<real, kRoomy<O, real>>(tr[t], xs, e * kAplusLd<real> + f * 81, dr);
      }
    // local flux, two faces at a time: Q += rDivM_f diag(M2) W_f, in units of
    // (row tile, face), each unit's fragments loaded during the ones before
    // In FP32 two faces' flux is summed on its own before it joins the rest: a
    // matrix instruction rounds every product it adds, and on top of the volume's
    // sum, twice the result, every one of these roundings would be larger (error
    // of the local pass against 64 bits at ORDER 6 3.9e-7 -> 3.1e-7, with the
    // traces' order of summation 2.7e-7; 1M cells 7.24 -> 7.26 ms a step, four
    // LTS clusters of 600k cells at ORDER 5 22.70 -> 22.84)
    constexpr bool OWN = sizeof(real) == 4;
    constexpr int KSF = G::KSF, UNITS = 2 * TW, FAR = VEL && sizeof(real) == 4 ? 2 : 1;
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      real a[FAR + 1][KSF];
      int lo[UNITS], hi[UNITS];
      auto load = [&](int u) {
        const int row = min(tile[u / 2], G::MT - 1), f = 2 * half + u % 2;
        const real* const fr = A.frag + G::flux + (static_cast<int64_t>(row) * 4 + f) * KSF * 64;
#pragma unroll
        for (int k = 0; k < KSF; ++k) a[u % (FAR + 1)][k] = fr[k * 64 + lane];
      };
#pragma unroll
      for (int u = 0; u < FAR; ++u) load(u);
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        const int at = G::rFlux + 2 * (min(tile[u / 2], G::MT - 1) * 4 + 2 * half + u % 2);
        lo[u] = A.ranges[at];
        hi[u] = tile[u / 2] < G::MT ? A.ranges[at + 1] : 0;
      }
      __syncthreads();  // AplusT, or the first two faces' W, is no longer read
#pragma unroll
      for (int t = 0; t < TT; ++t)
        if (tt[t] < G::MTF) {
          const int f = G::traceFace(tt[t], g), row = G::traceRow(tt[t], g);
          if (f >> 1 == half && row < B2P)
#pragma unroll
            for (int p = 0; p < 9; ++p)
              *reinterpret_cast<V4*>(xs + (p * 16 + e) * LD + (f & 1) * B2P + row) = tr[t][p];
        }
      __syncthreads();
      [[maybe_unused]] V4 pair[NP];
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        if (u + FAR < UNITS) load(u + FAR);
        if (OWN && u % 2 == 0)
#pragma unroll
          for (int p = 0; p < NP; ++p) pair[p] = V4{0, 0, 0, 0};
        const real* const x = xr + P0 * 16 * LD + u % 2 * B2P;
#pragma unroll
        for (int k = 0; k < KSF; ++k)
          if (k >= lo[u] && k < hi[u]) {  // uniform
#pragma unroll
            for (int p = 0; p < NP; ++p) {
              V4& sum = OWN ? pair[p] : acc[u / 2][p];
              sum = mma(a[u % (FAR + 1)][k], x[p * 16 * LD + 4 * k], sum);
            }
          }
        if (OWN && u % 2 == 1)
#pragma unroll
          for (int p = 0; p < NP; ++p) acc[u / 2][p] += pair[p];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // Q += volume + flux: a row tile's old values are loaded before its first store
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      V4 old[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p)
        old[p] = dofs.template loadQuad<B>(cell, 16 * tile[t] + 4 * g, (P0 + p) * ldq);
#pragma unroll
      for (int p = 0; p < NP; ++p)
        dofs.storeQuad(old[p] + acc[t][p], cell, 16 * tile[t] + 4 * g, B, (P0 + p) * ldq);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// PARTS: kPredict (predictor: buffer and derivatives), kFlux (volume and local
// flux from the predictor's time integral, or without it from `integ`)
template <typename real, int O, int PARTS, bool LTS>
__global__ __launch_bounds__((Waves<O, real>::THREADS), (LocalLds<O, real>::SIMD_WAVES)) void kLocalMx(
    Segments<O, real, 1> seg, const real* __restrict__ frag, const int* __restrict__ ranges, real* __restrict__ dofs, real* __restrict__ integ, real* __restrict__ traces, const real* __restrict__ starAll,
    const real* __restrict__ aplus, const uint8_t* __restrict__ faceTypes, CellLayout lay, LtsOut lts) {
  __shared__ __attribute__((aligned(16))) real xs[LocalLds<O, real>::X];
  __shared__ real sStar[kElems * kStarLd];
  __shared__ real sLate[kLate];
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int s = LTS ? seg.find() : 0;
  const int64_t E0 = seg.start[s] + static_cast<int64_t>(static_cast<int>(blockIdx.x) - (LTS ? seg.firstBlock[s] : 0)) * kElems;
  const int cells = static_cast<int>(min(seg.end[s] - E0, int64_t(kElems)));
  const LocalArgs<real, O> A{E0, cells, seg.reset[s], frag, ranges, seg.c[s][0], dofs, integ, traces, starAll, aplus, faceTypes, lay, lts};
  if (w & 1) localWave<real, O, PARTS, LTS, true>(A, xs, sStar, sLate, w);
  else localWave<real, O, PARTS, LTS, false>(A, xs, sStar, sLate, w);
}

template <typename real, int O>
int launchTiles(const EngineState& st, int parts, const ClusterStep* steps, int clusters, const sdg_layer* L,
                const CellLayout& lay, bool writeTraces, const LtsOut* lts, hipStream_t stream) {
  Segments<O, real, 1> seg;
  const int64_t blocks = seg.fill(steps, clusters);
  if (blocks == 0) return SDG_OK;
  const dim3 grid(static_cast<unsigned>(blocks));
  auto launch = [&](auto partsI, auto ltsI) {
    kLocalMx<real, O, decltype(partsI)::value, decltype(ltsI)::value><<<grid, Waves<O, real>::THREADS, 0, stream>>>(
        seg, static_cast<const real*>(st.mxFrags), st.mxRanges, static_cast<real*>(L->dofs),
        static_cast<real*>(L->time_integrated), writeTraces ? static_cast<real*>(L->face_traces) : nullptr,
        static_cast<const real*>(L->star), static_cast<const real*>(L->aplus), L->face_types, lay,
        lts != nullptr ? *lts : LtsOut{});
  };
  if (parts == kPredict) launch(std::integral_constant<int, kPredict>{}, std::true_type{});
  else if (parts == kFlux) launch(std::integral_constant<int, kFlux>{}, std::false_type{});
  else if (lts != nullptr) launch(std::integral_constant<int, kPredict | kFlux>{}, std::true_type{});
  else launch(std::integral_constant<int, kPredict | kFlux>{}, std::false_type{});
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

template <typename real, int O>
int localImpl(const EngineState& st, int parts, const ClusterStep* steps, int clusters, const sdg_layer* L,
              bool writeTraces, const LtsOut* lts, hipStream_t stream) {
  const CellLayout lay = cellLayout(st, L);
  // a tile reaches its cells' operators by 32-bit offsets: where 16 cells are
  // further apart than that, launches of as many cells as are not
  const int64_t apart = std::max(lay.starStride, lay.aplusStride) * static_cast<int64_t>(sizeof(real));
  const int64_t near = 1 + (0x7ff00000 - 324 * static_cast<int64_t>(sizeof(real))) / apart;
  if (near >= kElems) return launchTiles<real, O>(st, parts, steps, clusters, L, lay, writeTraces, lts, stream);
  for (int i = 0; i < clusters; ++i)
    for (ClusterStep part = steps[i]; part.start < steps[i].end; part.start = part.end) {
      part.end = std::min(part.start + near, steps[i].end);
      if (const int rc = launchTiles<real, O>(st, parts, &part, 1, L, lay, writeTraces, lts, stream); rc != SDG_OK)
        return rc;
    }
  return SDG_OK;
}

}  // namespace

template <int O>
int Order<O>::local(const EngineState& e, int parts, const ClusterStep* steps, int clusters, const sdg_layer* layer,
                    bool traces, const LtsOut* lts, hipStream_t stream) {
  return e.arithmetic == SDG_FP64 ? localImpl<double, O>(e, parts, steps, clusters, layer, traces, lts, stream)
                                  : localImpl<float, O>(e, parts, steps, clusters, layer, traces, lts, stream);
}

}  // namespace mx
}  // namespace sdg
