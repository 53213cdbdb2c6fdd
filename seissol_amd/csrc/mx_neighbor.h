// Neighbour flux on the matrix cores in the engine's real type
// (Neighbor.cpp:66-109, TimeCommon.cpp:40-87; spec
// codegen/kernels/aderdg.py:414-431), global and local time stepping:
// Q += sum_f rDivM_f ((fP_h U_f) AminusT_f) with U_f = rT_j I_nb, formed here
// from the neighbours' time-integrated DOFs or read as the face traces that
// the local pass wrote.
//
// A workgroup handles a tile of 16 elements, that is 64 tasks (element, face),
// in three phases:
//  1. U.  From DOFs: the tasks are sorted by the side j of their neighbour
//     into groups of 16 with one j each, so that rT_j is the stationary
//     operand of a matrix instruction whose 16 columns are one quantity of
//     16 tasks.  The neighbours' DOFs go from global memory straight into the
//     operand registers (each value feeds one or two row tiles only, LDS would
//     not be reused); a group is split over three waves by quantities.
//     From traces: copied to LDS, every load of the tile in flight at once.
//  2. W = (fP_h U) AminusT_f per task on 16 lanes, in place of U: fP_h as rows
//     of at most ORDER non-zeros, AminusT read once per task and broadcast
//     across its lanes (DPP row_newbcast).
//  3. Q += rDivM_f W_f, a GEMM over the tile with K = the four faces' rows.
// All four faces' operands stay in LDS (110 KB in FP64 at ORDER 6, one
// workgroup of eight waves per CU; 56 KB in FP32), which leaves two barriers
// per tile.  Bound by the matrix instructions (FP64) or, on random links, by
// the gather of four neighbours' DOFs per element; AminusT and the old DOFs are
// loaded across the barriers (400k cells in FP64 at ORDER 6 from traces 2.04 ->
// 1.93 ms, 350k in FP32 at ORDER 5 with LTS 1.09 -> 1.05, 100k in FP32 at ORDER
// 6 from DOFs 537 -> 514 us).
// From traces this replaced a kernel that went face by face, nine barriers a
// tile, one wave per row tile: FP64 steps of 60k cells 608 -> 286 us at ORDER
// 3, 487 -> 428 at 4, 793 -> 721 at 5, 2148 -> 1952 at 7; 400k cells at ORDER
// 6 7.34 -> 7.11 ms; 500 cells at ORDER 4 52 -> 35 us.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dpp_rows.h"
#include "mx_common.h"

namespace sdg {
namespace mx {
namespace {

// what the neighbour pass reads: the neighbours' buffers, buffers or
// derivatives (local time stepping), or the face traces rT_j I of the local pass
constexpr int kFromDofs = 0, kFromLts = 1, kFromTraces = 2;

// geometry and LDS of the neighbour kernel
template <int O, typename real>
struct NeighborGeo {
  using G = Geo<O>;
  static constexpr int WAVES = 2 * G::MT, THREADS = 64 * WAVES;
  static constexpr int FS = 9 * G::B2P;  // reals of one task's operand [quantity][B2P]
  // element stride: the 16 elements' operand reads conflict-free, quads aligned
  static constexpr int ES = columnStride<real>(4 * FS);
  static constexpr int bytes = kElems * ES * static_cast<int>(sizeof(real)) +
                               3 * G::B2 * O * (static_cast<int>(sizeof(real)) + 4) + 1024;
  static constexpr int wanted = (163840 / bytes) * WAVES / 4;  // waves per SIMD that the LDS allows
  // waves per SIMD asked of the register allocator: all that the LDS allows,
  // but no more than two or four for the sums over derivatives (LTS) and the
  // DOF operands of the high orders, which would spill
  static constexpr int simdWaves(bool lean) {
    const int cap = sizeof(real) == 8 ? (lean ? 3 : 2) : (lean ? 6 : 4);
    return maxOf(cdiv(WAVES, 4), wanted < cap ? wanted : cap);
  }
  static constexpr int MAXGROUPS = 7;  // sum over four sides of ceil(tasks / 16), 64 tasks
};

// rows row, row + 1 of quantity block q (B rows), zero from B on; in bounds
// for every row (a last single row is taken from the pair that ends the block)
template <int B, typename real>
__device__ inline void loadPair(const real* __restrict__ q, int row, real (&v)[2]) {
  typedef real V2 __attribute__((ext_vector_type(2), aligned(sizeof(real))));
  const V2 raw = *reinterpret_cast<const V2*>(q + min(row, B - 2));
  v[0] = row < B ? raw[0] : real(0);
  v[1] = row + 1 < B ? raw[1] : real(0);
  if constexpr (B % 2 != 0) {
    if (row == B - 1) v[0] = raw[1];
  }
}

template <typename real, int O, int SRC>
__global__ __launch_bounds__((NeighborGeo<O, real>::THREADS),
                             (NeighborGeo<O, real>::simdWaves(SRC == kFromTraces || (SRC == kFromDofs && O <= 5)))) void kNeighborMx(
    Segments<O, real, 2> seg, const real* __restrict__ frag, const int* __restrict__ ranges, real* __restrict__ dofs,
    const real* __restrict__ integ, const real* __restrict__ deriv, const int32_t* __restrict__ neighbors,
    const uint8_t* __restrict__ faceRel, const real* __restrict__ aminus, const uint8_t* __restrict__ faceTypes,
    const uint16_t* __restrict__ setups, CellLayout lay) {
  using G = Geo<O>;
  using N = NeighborGeo<O, real>;
  using V4 = typename Vec<real>::V4;
  constexpr int B = G::B, B2 = G::B2, B2P = G::B2P, FS = N::FS, ES = N::ES, RS = sizeof(real);
  constexpr bool LTS = SRC == kFromLts;
  // AminusT and the old DOFs ahead across the barriers, unless the registers for
  // it cost waves (FP32 at ORDER 5 from traces, 60k cells: 101 us, 109 ahead)
  constexpr bool AHEAD = LTS || N::wanted < 6;
  __shared__ __attribute__((aligned(16))) real sU[kElems * ES];  // U, then W: [element][face][quantity][B2P]
  __shared__ real sFP[3 * B2 * O];
  __shared__ int sFPCol[3 * B2 * O];
  __shared__ int sNb[64], sMeta[64];  // per task: neighbour; regular | h << 1 | derivatives << 3 | gts << 4
  __shared__ int sSlot[N::MAXGROUPS * 16];  // tasks in group order, -1: none
  __shared__ int sSide[N::MAXGROUPS + 1];   // side of each group; last: number of groups

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int g = lane >> 4, c = lane & 15;
  const int s = LTS ? seg.find() : 0;
  const int64_t E0 = seg.start[s] + static_cast<int64_t>(static_cast<int>(blockIdx.x) - (LTS ? seg.firstBlock[s] : 0)) * kElems;
  const int cells = static_cast<int>(min(seg.end[s] - E0, int64_t(kElems)));

  for (int i = threadIdx.x; i < 3 * B2 * O; i += N::THREADS) {
    sFP[i] = frag[G::fP + i];
    sFPCol[i] = static_cast<int>(frag[G::fPCol + i]);
  }
  if (w == 0) {
    // one lane per task: element lane / 4, face lane % 4
    const int el = min(lane >> 2, cells - 1);
    const int64_t at = (E0 + el) * 4 + (lane & 3);
    const int type = faceTypes != nullptr ? faceTypes[at] : SDG_FACE_REGULAR;
    const int nb = neighbors[at];
    const int side = min(static_cast<int>(faceRel[2 * at]), 3), h = min(static_cast<int>(faceRel[2 * at + 1]), 2);
    const bool regular = (lane >> 2) < cells && type == SDG_FACE_REGULAR;
    int meta = (regular ? 1 : 0) | h << 1;
    if constexpr (LTS) {
      const unsigned setup = setups[E0 + el];
      meta |= ((setup >> (lane & 3)) & 1u) << 3 | ((setup >> (4 + (lane & 3))) & 1u) << 4;
    }
    sNb[lane] = regular ? nb : 0;
    sMeta[lane] = meta;
    if constexpr (SRC == kFromTraces) {
      sSlot[lane] = regular ? side : -1;
    } else {
      sSlot[lane] = -1;
      if (lane < N::MAXGROUPS * 16 - 64) sSlot[64 + lane] = -1;
      waveSync();
      int group = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint64_t mask = __ballot(regular && side == j);
        const int before = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                                     __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u));
        if (regular && side == j) sSlot[16 * group + before] = lane;
        const int groups = (__popcll(mask) + 15) / 16;
        if (lane < groups) sSide[group + lane] = j;
        group += groups;
      }
      if (lane == 0) sSide[N::MAXGROUPS] = group;
    }
  }
  __syncthreads();

  if constexpr (SRC == kFromTraces) {
    // phase 1: the traces [neighbour][side][quantity][B2P], every load of a
    // thread in flight before its first store
    constexpr int TR4 = FS / 4, N4 = cdiv(64 * TR4, N::THREADS);
    V4 v[N4];
#pragma unroll
    for (int u = 0; u < N4; ++u) {
      const int i = min(static_cast<int>(threadIdx.x) + u * N::THREADS, 64 * TR4 - 1), t = i / TR4;
      const int side = max(sSlot[t], 0);  // a task without a neighbour reads cell 0's first trace; its W is zero
      v[u] = *reinterpret_cast<const V4*>(integ + (static_cast<int64_t>(sNb[t]) * 4 + side) * FS + 4 * (i % TR4));
    }
#pragma unroll
    for (int u = 0; u < N4; ++u) {
      const int i = threadIdx.x + u * N::THREADS, t = i / TR4;
      if (i < 64 * TR4) *reinterpret_cast<V4*>(sU + (t >> 2) * ES + (t & 3) * FS + 4 * (i % TR4)) = v[u];
    }
  } else {
    // phase 1: units of (group, three quantities)
    const int units = 3 * __builtin_amdgcn_readfirstlane(sSide[N::MAXGROUPS]);
#pragma unroll 1
    for (int u = w; u < units; u += N::WAVES) {
      const int group = u / 3, q0 = 3 * (u % 3);
      const int j = __builtin_amdgcn_readfirstlane(sSide[group]);
      const int task = sSlot[16 * group + c];
      const int t = task < 0 ? 0 : task;
      const int64_t nb = task < 0 ? 0 : sNb[t];
      // the neighbour's time integral: its buffer, or its derivatives integrated
      // over this step (GTS relation: time coefficients, else the sub-interval's)
      [[maybe_unused]] bool fromDeriv = false;
      [[maybe_unused]] bool gts = false;
      if constexpr (LTS) {
        const int meta = sMeta[t];
        fromDeriv = task >= 0 && (meta >> 3 & 1);
        gts = meta >> 4 & 1;
      }
      real x[G::KB8][3][2];
      {
        const real* const src = integ + nb * lay.qStride + q0 * lay.ldq;
#pragma unroll
        for (int k = 0; k < G::KB8; ++k)
#pragma unroll
          for (int q = 0; q < 3; ++q) loadPair<B>(src + q * lay.ldq, 8 * k + 2 * g, x[k][q]);
      }
      if constexpr (LTS) {
        if (__ballot(fromDeriv) != 0) {
          const real* src = deriv + nb * lay.dsize;
          real y[G::KB8][3][2];
#pragma unroll
          for (int k = 0; k < G::KB8; ++k)
#pragma unroll
            for (int q = 0; q < 3; ++q) y[k][q][0] = y[k][q][1] = real(0);
          staticFor<O>([&](auto dI) {
            constexpr int d = decltype(dI)::value, m = basis3(O - d);
            const int ldm = lay.rows(m);
            const real cd = gts ? seg.c[s][0][d] : seg.c[s][1][d];  // GTS relation, sub-interval of a larger step
#pragma unroll
            for (int k = 0; k < cdiv(m, 8); ++k)
#pragma unroll
              for (int q = 0; q < 3; ++q) {
                real v[2];
                if constexpr (m >= 2) {
                  loadPair<m>(src + (q0 + q) * ldm, 8 * k + 2 * g, v);
                } else {
                  const real v0 = src[(q0 + q) * ldm];
                  v[0] = g == 0 ? v0 : real(0);
                  v[1] = real(0);
                }
                y[k][q][0] += cd * v[0];
                y[k][q][1] += cd * v[1];
              }
            src += 9LL * ldm;
          });
#pragma unroll
          for (int k = 0; k < G::KB8; ++k)
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
              for (int i = 0; i < 2; ++i) x[k][q][i] = fromDeriv ? y[k][q][i] : x[k][q][i];
        }
      }
      V4 acc[G::RT][3];
#pragma unroll
      for (int r = 0; r < G::RT; ++r)
#pragma unroll
        for (int q = 0; q < 3; ++q) acc[r][q] = V4{0, 0, 0, 0};
      typedef real V2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int r = 0; r < G::RT; ++r) {
        const V2* const fr =
            reinterpret_cast<const V2*>(frag + G::rt + (static_cast<int64_t>(j) * G::RT + r) * G::KB8 * 128) + lane;
        const int lo = ranges[G::rRt + 2 * (j * G::RT + r)], hi = ranges[G::rRt + 2 * (j * G::RT + r) + 1];
#pragma unroll
        for (int k = 0; k < G::KB8; ++k)
          if (k >= lo && k < hi) {  // uniform
            const V2 a = fr[k * 64];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
              for (int q = 0; q < 3; ++q) acc[r][q] = mma(a[i], x[k][q][i], acc[r][q]);
          }
      }
      if (task >= 0) {
        real* const out = sU + (task >> 2) * ES + (task & 3) * FS + q0 * B2P + 4 * g;
#pragma unroll
        for (int r = 0; r < G::RT; ++r)
          if (16 * r + 4 * g < B2P)
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<V4*>(out + q * B2P + 16 * r) = acc[r][q];
      }
    }
  }
  // phase 2: a task per 16-lane row, lane c its face rows c (and c + 16).
  constexpr int RF = cdiv(B2P, 16);
  real rowA[9];  // lane c: row min(c, 8) of AminusT
  auto loadA = [&](int t, real(&a)[9]) {
    const real* const A = aminus + (E0 + min(t >> 2, cells - 1)) * lay.aminusStride + 81 * (t & 3) + min(c, 8);
#pragma unroll
    for (int p = 0; p < 9; ++p) a[p] = A[9 * p];
  };
  if constexpr (AHEAD) loadA(4 * w + g, rowA);
  __syncthreads();
#pragma unroll 1
  for (int t0 = 4 * w; t0 < 64; t0 += 4 * N::WAVES) {
    const int t = t0 + g;
    const int meta = sMeta[t], h = meta >> 1 & 3;
    const bool regular = meta & 1;
    real nextA[9];
    if constexpr (AHEAD) loadA(min(t + 4 * N::WAVES, 63), nextA);
    else loadA(t, rowA);
    real* const us = sU + (t >> 2) * ES + (t & 3) * FS;
    real u[RF][9];
#pragma unroll
    for (int r = 0; r < RF; ++r) {
#pragma unroll
      for (int q = 0; q < 9; ++q) u[r][q] = real(0);
      const int list = (h * B2 + min(c + 16 * r, B2 - 1)) * O;
#pragma unroll
      for (int k = 0; k < O; ++k) {
        const real f = sFP[list + k];
        const real* const col = us + sFPCol[list + k];
#pragma unroll
        for (int q = 0; q < 9; ++q) u[r][q] += f * col[q * B2P];
      }
    }
    real wv[RF][9];
#pragma unroll
    for (int r = 0; r < RF; ++r) {
#pragma unroll
      for (int p = 0; p < 9; ++p) wv[r][p] = real(0);
      staticFor<9>([&](auto qI) {
        constexpr int q = decltype(qI)::value;
        fmacRowBcast9<q>(wv[r], rowA, u[r][q]);
      });
    }
    waveSync();  // every lane of the task has read U
#pragma unroll
    for (int r = 0; r < RF; ++r)
      if (c + 16 * r < B2P)
#pragma unroll
        for (int p = 0; p < 9; ++p) us[p * B2P + c + 16 * r] = regular && c + 16 * r < B2 ? wv[r][p] : real(0);
    if constexpr (AHEAD)
#pragma unroll
      for (int p = 0; p < 9; ++p) rowA[p] = nextA[p];
  }

  // phase 3: wave (row tile, quantities 0-4 or 5-8)
  const int tile = w >> 1, p0 = 5 * (w & 1), np = (w & 1) ? 4 : 5;
  const Buffer<real> q(dofs + E0 * lay.qStride, cells * lay.qStride);
  const int cell = c < cells ? c * static_cast<int>(lay.qStride) * RS : kNowhere;
  const int row = 16 * tile + 4 * g;
  V4 old[5];
  auto loadOld = [&] {
#pragma unroll
    for (int p = 0; p < 5; ++p)
      old[p] = q.template loadQuad<B>(p < np ? cell : kNowhere, row, (p0 + p) * lay.ldq * RS);
  };
  if constexpr (AHEAD) loadOld();
  __syncthreads();

  V4 acc[5];
#pragma unroll
  for (int p = 0; p < 5; ++p) acc[p] = V4{0, 0, 0, 0};
  const real* const xr = sU + c * ES + p0 * B2P + g;
#pragma unroll 1
  for (int f = 0; f < 4; ++f) {
    const int lo = ranges[G::rFlux + 2 * (tile * 4 + f)], hi = ranges[G::rFlux + 2 * (tile * 4 + f) + 1];
    const real* const fr = frag + G::rdm + (static_cast<int64_t>(tile) * 4 + f) * G::KSF * 64 + lane;
    real a[G::KSF];
#pragma unroll
    for (int k = 0; k < G::KSF; ++k) a[k] = fr[k * 64];
#pragma unroll
    for (int k = 0; k < G::KSF; ++k)
      if (k >= lo && k < hi) {  // uniform
#pragma unroll
        for (int p = 0; p < 5; ++p)
          if (p < np) acc[p] = mma(a[k], xr[f * FS + p * B2P + 4 * k], acc[p]);
      }
  }
  if constexpr (!AHEAD) loadOld();
#pragma unroll
  for (int p = 0; p < 5; ++p)
    q.storeQuad(old[p] + acc[p], p < np ? cell : kNowhere, row, B, (p0 + p) * lay.ldq * RS);
}

template <typename real, int O>
int neighborImpl(const EngineState& st, const sdg_layer* L, const ClusterStep* steps, int clusters, bool traces,
                 hipStream_t stream) {
  using N = NeighborGeo<O, real>;
  Segments<O, real, 2> seg;
  const int64_t blocks = seg.fill(steps, clusters);
  if (blocks == 0) return SDG_OK;
  const CellLayout lay = cellLayout(st, L);
  const dim3 grid(static_cast<unsigned>(blocks));
  auto launch = [&](auto srcI) {
    kNeighborMx<real, O, decltype(srcI)::value><<<grid, N::THREADS, 0, stream>>>(
        seg, static_cast<const real*>(st.mxFrags), st.mxRanges, static_cast<real*>(L->dofs),
        static_cast<const real*>(traces ? L->face_traces : L->time_integrated),
        static_cast<const real*>(L->derivatives), L->face_neighbors, L->face_relations,
        static_cast<const real*>(L->aminus), L->face_types, L->lts_setup, lay);
  };
  if (traces) launch(std::integral_constant<int, kFromTraces>{});
  else if (steps[0].coeffs != nullptr && L->lts_setup != nullptr) launch(std::integral_constant<int, kFromLts>{});
  else if constexpr (O > 3 || sizeof(real) == 8) launch(std::integral_constant<int, kFromDofs>{});
  else {  // prefersNeighborMx sends these to the VALU
    setError("the matrix-core neighbour pass from DOFs starts at ORDER 4 in FP32");
    return SDG_ERR_UNSUPPORTED;
  }
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

}  // namespace

template <int O>
int Order<O>::neighbor(const EngineState& e, const sdg_layer* layer, const ClusterStep* steps, int clusters, bool traces,
                       hipStream_t stream) {
  return e.arithmetic == SDG_FP64 ? neighborImpl<double, O>(e, layer, steps, clusters, traces, stream)
                                  : neighborImpl<float, O>(e, layer, steps, clusters, traces, stream);
}

}  // namespace mx
}  // namespace sdg
