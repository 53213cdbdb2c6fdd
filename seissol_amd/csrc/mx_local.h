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
// What bounds it: the matrix instructions (FP64: 64 cycles per 16 x 16 x 4 and
// SIMD) and HBM come to about the same time, so the pass lives from several
// workgroups per CU overlapping their phases, and from few instructions:
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
//  * dQ_1 and dQ_2 share the X area, later derivatives alternate between the
//    two places: one barrier per derivative from dQ_2 on.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "mx_common.h"

namespace sdg {
namespace mx {
namespace {

template <int O, typename real>
struct Coeffs {
  real c[O];
};

// LDS of the local kernel, in reals
template <int O, typename real>
struct LocalLds {
  using G = Geo<O>;
  static constexpr int LD = columnStride<real>(G::XROWS);
  static constexpr int X = maxOf(kCols * LD, kElems * kAplusLd);
  static constexpr int bytes = (X + kElems * kStarLd) * static_cast<int>(sizeof(real));
  static constexpr int GROUPS = 163840 / bytes;  // workgroups per CU that the LDS allows
  // waves per SIMD asked of the register allocator
  static constexpr int wanted = GROUPS * G::WAVES / 4;
  static constexpr int cap = sizeof(real) == 8 ? 2 : 3;
  static constexpr int SIMD_WAVES = wanted < 1 ? 1 : (wanted < cap ? wanted : cap);
};

// y[p][.] += sum_j sum_q (A_j X_q) star_j(q, p) for the stresses p < 6 of one
// row tile.  fr: its fragments [j][KS][64]; x: the lane's column of quantity 0
// at row g.  Fragments are loaded four k-steps ahead, across the directions.
template <int KS, int LD, typename real>
__device__ inline void starStress(const real* __restrict__ fr, int lo, int hi, const real* x, const real* sS,
                                  int lane, typename Vec<real>::V4 (&y)[6]) {
  using V4 = typename Vec<real>::V4;
  real cur[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) cur[u] = fr[min(lo + u, hi - 1) * 64 + lane];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    V4 acc[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] = V4{0, 0, 0, 0};
#pragma unroll 1
    for (int k = lo; k < hi; k += 4) {
      const bool last = k + 4 >= hi;
      const int nj = last ? (j < 2 ? j + 1 : 2) : j, nk = last ? lo : k + 4;
      real nxt[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) nxt[u] = fr[(nj * KS + min(nk + u, hi - 1)) * 64 + lane];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k + u < hi) {
#pragma unroll
          for (int i = 0; i < 3; ++i) acc[i] = mma(cur[u], x[(6 + i) * 16 * LD + 4 * (k + u)], acc[i]);
        }
#pragma unroll
      for (int u = 0; u < 4; ++u) cur[u] = nxt[u];
    }
    // the star values are read where they are used, and the sums finished
    // before the next direction's products start (else the compiler keeps all
    // 45 values and three directions' accumulators live)
    int at = 24 * j;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int p = 0; p < 6; ++p) {
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (k < kStarCnt[p]) y[p] += acc[kStarQ[p][k] - 6] * sS[at + kStarOff[p] + k];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        real v = y[p][r];
        asm volatile("" : "+v"(v));
        y[p][r] = v;
      }
    }
  }
}

// y[t][i][.] += sum_j A_j (sum_q X_q star_j(q, 6 + i)) for the velocities of
// up to TW row tiles (lo[t] >= hi[t]: none)
template <int KS, int LD, int TW, typename real>
__device__ inline void starVelocity(const real* const (&fr)[TW], const int (&lo)[TW], const int (&hi)[TW],
                                    const real* x, const real* sS, int lane,
                                    typename Vec<real>::V4 (&y)[TW][3]) {
  using V4 = typename Vec<real>::V4;
  int k0 = KS, k1 = 0;
#pragma unroll
  for (int t = 0; t < TW; ++t)
    if (lo[t] < hi[t]) {
      k0 = min(k0, lo[t]);
      k1 = max(k1, hi[t]);
    }
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
  real cur[TW][3];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int j = 0; j < 3; ++j) cur[t][j] = fr[t][(j * KS + k0) * 64 + lane];
#pragma unroll 1
  for (int k = k0; k < k1; ++k) {
    real nxt[TW][3];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) nxt[t][j] = fr[t][(j * KS + min(k + 1, k1 - 1)) * 64 + lane];
    real v[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = x[q * 16 * LD + 4 * k];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      real m[3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
        m[i] = s[j][3 * i] * v[kStarQ[6 + i][0]] + s[j][3 * i + 1] * v[kStarQ[6 + i][1]] +
               s[j][3 * i + 2] * v[kStarQ[6 + i][2]];
#pragma unroll
      for (int t = 0; t < TW; ++t)
        if (k >= lo[t] && k < hi[t]) {
#pragma unroll
          for (int i = 0; i < 3; ++i) acc[t][i] = mma(cur[t][j], m[i], acc[t][i]);
        }
    }
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) cur[t][j] = nxt[t][j];
  }
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int i = 0; i < 3; ++i) y[t][i] = acc[t][i];
}

// acc[q] += A(tile) X_q, q < NQ, over the k-steps [lo, hi); x: the lane's
// column of the first quantity at row g; fragments two k-steps ahead
template <int LD, int NQ, typename real>
__device__ inline void gemm(typename Vec<real>::V4 (&acc)[NQ], const real* __restrict__ fr, int lo, int hi,
                            const real* x, int lane) {
  if (lo >= hi) return;
  real a0 = fr[lo * 64 + lane], a1 = fr[min(lo + 1, hi - 1) * 64 + lane];
#pragma unroll 1
  for (int k = lo; k < hi; k += 2) {
    const real b0 = fr[min(k + 2, hi - 1) * 64 + lane], b1 = fr[min(k + 3, hi - 1) * 64 + lane];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = mma(a0, x[q * 16 * LD + 4 * k], acc[q]);
    if (k + 1 < hi) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[q] = mma(a1, x[q * 16 * LD + 4 * k + 4], acc[q]);
    }
    a0 = b0;
    a1 = b1;
  }
}

// W = T A for the four rows of a lane's quad, two rows at a time (more
// outgrow the registers); A is read at lds[at + 9 p + q], one column at a time
// (else all 81 entries are loaded at once)
template <typename real>
__device__ inline void mixRows(typename Vec<real>::V4 (&t)[9], const real* lds, int at, bool zero) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    real w0[9], w1[9];
#pragma unroll
    for (int p = 0; p < 9; ++p) {
      int col = at + 9 * p;
      asm volatile("" : "+v"(col));
      real s0 = real(0), s1 = real(0);
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        const real a = lds[col + q];
        s0 += t[q][2 * h] * a;
        s1 += t[q][2 * h + 1] * a;
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
  int64_t n;
  const real* frag;
  const int* ranges;
  const Coeffs<O, real>& cf;
  real* dofs;
  real* integ;
  real* traces;
  const real* aplus;
  const uint8_t* faceTypes;
  const CellLayout& lay;
  const LtsOut& lts;
};

// One wave's share of a tile: the stresses (VEL = false) or the velocities of
// its row tiles.  Both instantiations run the same sequence of barriers, each
// wave of the workgroup one of them.
template <typename real, int O, int PARTS, bool LTS, bool VEL>
__device__ inline void localWave(const LocalArgs<real, O>& A, real* const xs, const real* const sStar, const int w) {
  using G = Geo<O>;
  using V4 = typename Vec<real>::V4;
  constexpr int B = G::B, LD = LocalLds<O, real>::LD, TW = G::TW, KS = G::KS, B2P = G::B2P, THREADS = G::THREADS;
  constexpr int NP = VEL ? 3 : 6, P0 = VEL ? 6 : 0, RS = sizeof(real);
  const CellLayout& lay = A.lay;
  const int lane = threadIdx.x & 63, g = lane >> 4, e = lane & 15;
  int tile[TW];
  tile[0] = w >> 1;
  if constexpr (TW == 2) tile[1] = 2 * G::PAIRS - 1 - (w >> 1);
  // the tile's cells: columns beyond the last cell load zeros and store nothing
  const int64_t E0 = static_cast<int64_t>(blockIdx.x) * kElems;
  const int cells = static_cast<int>(min(A.n - E0, int64_t(kElems)));
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

  // ia: the time integral of the wave's rows and quantities
  V4 ia[TW][NP];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int p = 0; p < NP; ++p)
      ia[t][p] = ((PARTS & kPredict) ? dofs : integ).template loadQuad<B>(cell, 16 * tile[t] + 4 * g, (P0 + p) * ldq);
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
      for (int p = 0; p < NP; ++p) ia[t][p] *= A.cf.c[0];
    __syncthreads();
    [[maybe_unused]] int doff = 9 * ldq;
#pragma unroll 1
    for (int d = 1; d < O; ++d) {
      const int m = basis3(O - d);
      // dQ_{d-1} is read at row `src`, dQ_d stored at row `dst`
      const int src = (d >= 3 && (d & 1)) ? G::R1 : 0, dst = (d & 1) ? 0 : G::R1;
      const real cd = A.cf.c[d];
      V4 y[TW][NP];
      const real* fr[TW];
      int lo[TW], hi[TW];
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const bool has = 16 * tile[t] < m;
        const int at = G::rCk + 2 * ((d - 1) * G::MT + (has ? tile[t] : 0));
        lo[t] = A.ranges[at];
        hi[t] = has ? A.ranges[at + 1] : 0;
        fr[t] = A.frag + G::ck + static_cast<int64_t>(has ? tile[t] : 0) * 3 * KS * 64;
#pragma unroll
        for (int p = 0; p < NP; ++p) y[t][p] = V4{0, 0, 0, 0};
      }
      if constexpr (VEL) {
        starVelocity<KS, LD, TW, real>(fr, lo, hi, xr + src, sS, lane, y);
      } else {
#pragma unroll
        for (int t = 0; t < TW; ++t)
          if (lo[t] < hi[t]) starStress<KS, LD, real>(fr[t], lo[t], hi[t], xr + src, sS, lane, y[t]);
      }
      if (d == 1) __syncthreads();  // dQ_1 takes the place of Q
      const int ldm = lay.rows(m) * RS;
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const int row = 16 * tile[t] + 4 * g;
        if (16 * tile[t] < m) {
#pragma unroll
          for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int r = 0; r < 4; ++r) y[t][p][r] = row + r < m ? y[t][p][r] : real(0);
            ia[t][p] += cd * y[t][p];
          }
          if (row < m)
#pragma unroll
            for (int p = 0; p < NP; ++p) *reinterpret_cast<V4*>(xq + p * 16 * LD + dst + row) = y[t][p];
          if constexpr (LTS) {
            if (A.lts.deriv != nullptr)
#pragma unroll
              for (int p = 0; p < NP; ++p) deriv.storeQuad(y[t][p], myDeriv, row, m, doff + (P0 + p) * ldm);
          }
        }
      }
      if constexpr (LTS) doff += 9 * ldm;
      __syncthreads();
    }
    // the time integral: output (LTS: the buffer, stored or accumulated)
    if (A.integ != nullptr) {
      int mine = cell;
      if constexpr (LTS) mine = (setup & SDG_LTS_HAS_BUFFERS) ? cell : kNowhere;
      [[maybe_unused]] int before = kNowhere;  // the old buffer, where it accumulates (else zeros are loaded)
      if constexpr (LTS)
        before = A.lts.setup != nullptr && !A.lts.reset && (setup & SDG_LTS_ACCUMULATE_BUFFERS) ? mine : kNowhere;
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
    __syncthreads();
    // volume: sum_j kDivM_j I star_j, the initial value of the flux accumulators
    V4 acc[TW][NP];
    {
      const real* fr[TW];
      int lo[TW], hi[TW];
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const bool has = tile[t] < G::MT;
        const int at = G::rVol + 2 * (has ? tile[t] : 0);
        lo[t] = A.ranges[at];
        hi[t] = has ? A.ranges[at + 1] : 0;
        fr[t] = A.frag + G::vol + static_cast<int64_t>(has ? tile[t] : 0) * 3 * KS * 64;
#pragma unroll
        for (int p = 0; p < NP; ++p) acc[t][p] = V4{0, 0, 0, 0};
      }
      if constexpr (VEL) {
        starVelocity<KS, LD, TW, real>(fr, lo, hi, xr, sS, lane, acc);
      } else {
#pragma unroll
        for (int t = 0; t < TW; ++t)
          if (lo[t] < hi[t]) starStress<KS, LD, real>(fr[t], lo[t], hi[t], xr, sS, lane, acc[t]);
      }
    }
    // face traces rT_f I of the wave's trace tiles (the second, where there is
    // one, goes to the velocity waves, which hold fewer registers)
    constexpr int TT = VEL ? G::TT : 1;
    V4 tr[TT][9];
    int tt[TT];
    tt[0] = w;
    if constexpr (TT == 2) tt[1] = G::WAVES + (w >> 1);
    const Buffer<real> traces(A.traces + E0 * 36 * B2P, A.traces != nullptr ? cells * 36 * B2P : 0);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int q = 0; q < 9; ++q) tr[t][q] = V4{0, 0, 0, 0};
      if (tt[t] < G::MTF) {
        gemm<LD, 9>(tr[t], A.frag + G::trace + static_cast<int64_t>(tt[t]) * KS * 64, A.ranges[G::rTrace + 2 * tt[t]],
                    A.ranges[G::rTrace + 2 * tt[t] + 1], xr, lane);
        const int f = G::traceFace(tt[t], g), row = G::traceRow(tt[t], g);
        if (A.traces != nullptr) {
          const int at = e < cells && row < B2P ? ((e * 4 + f) * 9 * B2P + row) * RS : kNowhere;
#pragma unroll
          for (int q = 0; q < 9; ++q) traces.store4(tr[t][q], at, q * B2P * RS);
        }
      }
    }
    // AplusT of the four faces takes the X area, in two batches: the first is
    // in flight across the barrier, and a whole one would outgrow the registers
    {
      constexpr int N = cdiv(kElems * 324, THREADS), N1 = N / 2;
      const Buffer<real> aplus(A.aplus + E0 * lay.aplusStride, (cells - 1) * lay.aplusStride + 324);
      const int stride = static_cast<int>(lay.aplusStride);
      auto load = [&](int u) {
        const int i = threadIdx.x + u * THREADS;
        return aplus.load1(i / 324 < cells ? ((i / 324) * stride + i % 324) * RS : kNowhere, 0);
      };
      auto store = [&](int u, real v) {
        const int i = threadIdx.x + u * THREADS;
        if (i < kElems * 324) xs[(i / 324) * kAplusLd + i % 324] = v;
      };
      real v[N - N1];
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
        mixRows<real>(tr[t], xs, e * kAplusLd + f * 81, dr);
      }
    // local flux, two faces at a time: Q += rDivM_f diag(M2) W_f
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
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
#pragma unroll
      for (int t = 0; t < TW; ++t)
        if (tile[t] < G::MT) {
#pragma unroll 1
          for (int fi = 0; fi < 2; ++fi) {
            const int f = 2 * half + fi;
            const int at = G::rFlux + 2 * (tile[t] * 4 + f);
            gemm<LD, NP>(acc[t], A.frag + G::flux + (static_cast<int64_t>(tile[t]) * 4 + f) * G::KSF * 64,
                         A.ranges[at], A.ranges[at + 1], xr + P0 * 16 * LD + fi * B2P, lane);
          }
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
__global__ __launch_bounds__(Geo<O>::THREADS, (LocalLds<O, real>::SIMD_WAVES)) void kLocalMx(
    int64_t n, const real* __restrict__ frag, const int* __restrict__ ranges, Coeffs<O, real> cf,
    real* __restrict__ dofs, real* __restrict__ integ, real* __restrict__ traces, const real* __restrict__ starAll,
    const real* __restrict__ aplus, const uint8_t* __restrict__ faceTypes, CellLayout lay, LtsOut lts) {
  constexpr int THREADS = Geo<O>::THREADS;
  __shared__ __attribute__((aligned(16))) real xs[LocalLds<O, real>::X];
  __shared__ real sStar[kElems * kStarLd];
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  // the compact star values of the tile, [element][3][24]; all loads of a
  // thread are in flight before its first store
  {
    constexpr int N = cdiv(kElems * 72, THREADS);
    const int64_t E0 = static_cast<int64_t>(blockIdx.x) * kElems;
    const int cells = static_cast<int>(min(n - E0, int64_t(kElems)));
    const Buffer<real> star(starAll + E0 * lay.starStride, (cells - 1) * lay.starStride + (lay.starCompact ? 72 : 243));
    const int stride = static_cast<int>(lay.starStride) * static_cast<int>(sizeof(real));
    real v[N];
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
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = threadIdx.x + u * THREADS;
      if (i < kElems * 72) sStar[(i / 72) * kStarLd + i % 72] = v[u];
    }
  }
  const LocalArgs<real, O> A{n, frag, ranges, cf, dofs, integ, traces, aplus, faceTypes, lay, lts};
  if (w & 1) localWave<real, O, PARTS, LTS, true>(A, xs, sStar, w);
  else localWave<real, O, PARTS, LTS, false>(A, xs, sStar, w);
}

template <typename real, int O>
int localImpl(const EngineState& st, int parts, const double* coeffs, const sdg_layer* L, bool writeTraces,
              const LtsOut* lts, hipStream_t stream) {
  using G = Geo<O>;
  const int64_t n = L->num_elements;
  if (n == 0) return SDG_OK;
  Coeffs<O, real> cf{};
  if (coeffs != nullptr)
    for (int i = 0; i < O; ++i) cf.c[i] = static_cast<real>(coeffs[i]);
  const CellLayout lay = cellLayout(st, L);
  const dim3 grid(static_cast<unsigned>((n + kElems - 1) / kElems));
  auto launch = [&](auto partsI, auto ltsI) {
    kLocalMx<real, O, decltype(partsI)::value, decltype(ltsI)::value><<<grid, G::THREADS, 0, stream>>>(
        n, static_cast<const real*>(st.mxFrags), st.mxRanges, cf, static_cast<real*>(L->dofs),
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

}  // namespace

template <int O>
int Order<O>::local(const EngineState& e, int parts, const double* coeffs, const sdg_layer* layer, bool traces,
                    const LtsOut* lts, hipStream_t stream) {
  return e.arithmetic == SDG_FP64 ? localImpl<double, O>(e, parts, coeffs, layer, traces, lts, stream)
                                  : localImpl<float, O>(e, parts, coeffs, layer, traces, lts, stream);
}

}  // namespace mx
}  // namespace sdg
