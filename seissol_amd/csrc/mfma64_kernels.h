// Plain FP64 neighbour flux on the matrix cores (v_mfma_f64_16x16x4_f64) from
// the FP64 face traces the local pass wrote (mx_local.h).  Included by the
// per-order sources kernels_mfma64_o<O>.hip.
//
// The contraction with rDivM_f is a GEMM over a tile of 16 elements, the 144
// columns being (quantity p, element e) -> 16 p + e, in k-steps of 4.  One
// wave owns one 16-row tile of the basis index for all 9 quantities: lane l
// holds rows g, g + 4, g + 8, g + 12 (g = l / 16) of the tile for element
// e = l % 16 (the accumulator layout of v_mfma_f64_16x16x4).  The operand lies
// in LDS column-major ([column][k], k contiguous); A is pre-swizzled in global
// memory so one k-step's fragment is one coalesced 8-byte load per lane
// (L2-resident, shared by all workgroups).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "engine.h"
#include "mfma_common.h"

namespace sdg {
namespace mfma64 {

using mfma::basis3;
using mfma::cdiv;
using mfma::kCols;
using mfma::kTileElems;

typedef double doublex4 __attribute__((ext_vector_type(4)));

__device__ inline doublex4 mma(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// q[p * ld + row0 + 4 j] += acc[p][j] for the lane's rows below B: all 36 old
// values are loaded first, unconditionally from in-bounds (clamped) rows, then
// stored where real (a read-modify-write under a branch waits on every load)
template <int B>
__device__ inline void addRows(double* q, int ld, int row0, bool live, const doublex4 (&acc)[9]) {
  double old[9][4];
#pragma unroll
  for (int p = 0; p < 9; ++p)
#pragma unroll
    for (int j = 0; j < 4; ++j) old[p][j] = q[p * ld + min(row0 + 4 * j, B - 1)];
  if (live)
#pragma unroll
    for (int p = 0; p < 9; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (row0 + 4 * j < B) q[p * ld + row0 + 4 * j] = old[p][j] + acc[p][j];
}

// acc[q] += A_tile X(:, quantity q) over `ksteps` k-steps, q < 9
template <int LD>
__device__ inline void gemm9(doublex4 (&acc)[9], const double* __restrict__ a, int ksteps, const double* xs,
                             int lane) {
  const int g = lane >> 4, e = lane & 15;
  double an = a[lane];
  for (int kk = 0; kk < ksteps; ++kk) {
    const double ac = an;
    if (kk + 1 < ksteps) an = a[(kk + 1) * 64 + lane];
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q] = mma(ac, xs[(q * 16 + e) * LD + 4 * kk + g], acc[q]);
  }
}

// Neighbour flux from the neighbours' face traces (Neighbor.cpp:66-109; spec
// aderdg.py:414-431): face by face, the 16 neighbours' traces rT_j I of the
// shared side are gathered, W_f = (fP_h Tr) AminusT_f is formed by 16-lane
// groups (one element, two rows per lane), and Q += rDivM_f W_f on the
// matrix cores; the next face's traces and AminusT are loaded into registers
// while the current face is computed.
template <int O, bool DEF>
__global__ __launch_bounds__(Shape64<O>::NTHREADS, 2) void kNeighborMfma64(
    int64_t n, const double* __restrict__ frag, double* __restrict__ dofs, const double* __restrict__ traces,
    const int32_t* __restrict__ neighbors, const uint8_t* __restrict__ faceRel, const double* __restrict__ aminus,
    const uint8_t* __restrict__ faceTypes, CellLayout lay) {
  using S = Shape64<O>;
  constexpr int B = S::B, B2 = S::B2, B2P = S::B2P, LDW = S::LDW, THREADS = S::NTHREADS;
  constexpr int HALF = B2P / 2;                 // row pairs of one (padded) face
  static_assert(HALF <= 16, "a face's row pairs fit a 16-lane group");
  constexpr int GROUPS = THREADS / 16;          // 16-lane groups per pass, one element each
  constexpr int PASSES = cdiv(kTileElems, GROUPS);
  constexpr int TR = 9 * B2P;                   // doubles of one face trace
  constexpr int TR2 = TR / 2;                   // 16-byte pieces of one face trace
  constexpr int GPT = cdiv(kTileElems * TR2, THREADS);
  constexpr int APT = cdiv(kTileElems * 81, THREADS);
  __shared__ __attribute__((aligned(16))) double xs[kCols * LDW];  // face operand, rows [0, B2P)
  __shared__ __attribute__((aligned(16))) double sTr[kTileElems * TR];
  __shared__ double sAm[kTileElems * 81];
  __shared__ double sFP[3 * B2 * O];
  __shared__ int sFPCol[3 * B2 * O];
  __shared__ int sLink[kTileElems * 4];  // trace index nb * 4 + side of (element, face), -1: none
  __shared__ int sRel[kTileElems * 4];   // orientation h of (element, face)

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int g = lane >> 4, e = lane & 15;
  const int64_t E0 = static_cast<int64_t>(blockIdx.x) * kTileElems;
  const bool valid = E0 + e < n;
  const int ldq = DEF ? B : lay.ldq;
  const int64_t qStride = DEF ? 9 * B : lay.qStride;
  const int row0 = 16 * w + g;  // the lane's rows row0 + 4 r

  // the fP tables and the neighbour links, every load issued unconditionally
  // from an in-bounds (clamped) address before the first store
  {
    constexpr int FPN = 3 * B2 * O, FPI = cdiv(FPN, THREADS);
    double fv[FPI], fc[FPI];
#pragma unroll
    for (int u = 0; u < FPI; ++u) {
      const int i = min(static_cast<int>(threadIdx.x) + u * THREADS, FPN - 1);
      fv[u] = frag[S::tFP + i];
      fc[u] = frag[S::tFPCol + i];
    }
    static_assert(kTileElems * 4 <= THREADS, "one thread per (element, face) link");
    const int s = threadIdx.x >> 2 & (kTileElems - 1), f = threadIdx.x & 3;
    const int64_t el = E0 + s < n ? E0 + s : n - 1;
    const int type = faceTypes != nullptr ? faceTypes[el * 4 + f] : SDG_FACE_REGULAR;
    const int nb = neighbors[el * 4 + f];
    const int side = faceRel[(el * 4 + f) * 2 + 0], rel = faceRel[(el * 4 + f) * 2 + 1];
#pragma unroll
    for (int u = 0; u < FPI; ++u) {
      const int i = threadIdx.x + u * THREADS;
      if (i < FPN) {
        sFP[i] = fv[u];
        sFPCol[i] = static_cast<int>(fc[u]);
      }
    }
    if (threadIdx.x < kTileElems * 4) {
      const bool use = E0 + s < n && type == SDG_FACE_REGULAR;
      sLink[threadIdx.x] = use ? nb * 4 + min(side, 3) : -1;
      sRel[threadIdx.x] = use ? min(rel, 2) : 0;
    }
  }
  __syncthreads();
  double2 gv[GPT];
  double av[APT];
  auto gather = [&](int f) {
#pragma unroll
    for (int i = 0; i < GPT; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      double2 v{0.0, 0.0};
      if (idx < kTileElems * TR2) {
        const int link = sLink[(idx / TR2) * 4 + f];
        if (link >= 0) v = *reinterpret_cast<const double2*>(traces + static_cast<int64_t>(link) * TR + 2 * (idx % TR2));
      }
      gv[i] = v;
    }
#pragma unroll
    for (int i = 0; i < APT; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      const int64_t at = (E0 + idx / 81) * (DEF ? 324 : lay.aminusStride) + f * 81 + idx % 81;
      av[i] = (idx < kTileElems * 81 && E0 + idx / 81 < n) ? aminus[at] : 0.0;
    }
  };
  gather(0);
  doublex4 acc[9];
#pragma unroll
  for (int p = 0; p < 9; ++p) acc[p] = doublex4{0, 0, 0, 0};
#pragma unroll 1
  for (int f = 0; f < 4; ++f) {
    // the previous face's items have read sTr / sAm and its product xs
#pragma unroll
    for (int i = 0; i < GPT; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      if (idx < kTileElems * TR2) *reinterpret_cast<double2*>(sTr + 2 * idx) = gv[i];
    }
#pragma unroll
    for (int i = 0; i < APT; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      if (idx < kTileElems * 81) sAm[idx] = av[i];
    }
    if (f < 3) gather(f + 1);
    __syncthreads();
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      // rows 2 rp and 2 rp + 1 of face f of element s (rows >= B2 are padding: zero)
      const int s = static_cast<int>(threadIdx.x >> 4) + ps * GROUPS;
      const int rp = static_cast<int>(threadIdx.x & 15);
      const int r0 = 2 * rp;
      const bool act = s < kTileElems && rp < HALF;
      const int sl = s < kTileElems ? s : 0;
      const bool regular = act && sLink[sl * 4 + f] >= 0;
      const int h = sRel[sl * 4 + f];
      const double* tr = sTr + sl * TR;
      double u[2][9];
#pragma unroll
      for (int ri = 0; ri < 2; ++ri) {
#pragma unroll
        for (int qq = 0; qq < 9; ++qq) u[ri][qq] = 0.0;
        const int row = r0 + ri;
        if (regular && row < B2) {
          const double* fp = sFP + (h * B2 + row) * O;
          const int* fc = sFPCol + (h * B2 + row) * O;
#pragma unroll
          for (int kk = 0; kk < O; ++kk) {
            const double c = fp[kk];
            const int mm = fc[kk];
#pragma unroll
            for (int qq = 0; qq < 9; ++qq) u[ri][qq] += c * tr[qq * B2P + mm];
          }
        }
      }
      const double* A = sAm + sl * 81;
#pragma unroll
      for (int p = 0; p < 9; ++p) {
        double w0 = 0.0, w1 = 0.0;
        if (regular)
#pragma unroll
          for (int qq = 0; qq < 9; ++qq) {
            const double a = A[qq + 9 * p];
            w0 += u[0][qq] * a;
            w1 += u[1][qq] * a;
          }
        if (act) *reinterpret_cast<double2*>(xs + (p * 16 + s) * LDW + r0) = double2{w0, w1};
      }
    }
    __syncthreads();
    gemm9<LDW>(acc, frag + S::rdmN + (static_cast<int64_t>(w) * 4 + f) * S::KSF * 64, S::KSF, xs, lane);
  }
  addRows<B>(dofs + (valid ? E0 + e : 0) * qStride, ldq, row0, valid, acc);
}

template <int B>
bool defaultLayout64(const CellLayout& lay) {
  return lay.ldq == B && lay.qStride == 9 * B && lay.aplusStride == 324 && lay.starStride == (lay.starCompact ? 72 : 243);
}

template <int O>
int MfmaOrder64<O>::neighbor(const EngineState& st, const sdg_layer* L, hipStream_t stream) {
  using S = Shape64<O>;
  const int64_t n = L->num_elements;
  if (n == 0) return SDG_OK;
  const CellLayout lay = cellLayout(st, L);
  const dim3 grid(static_cast<unsigned>((n + kTileElems - 1) / kTileElems));
  auto launch = [&](auto defFlag) {
    kNeighborMfma64<O, decltype(defFlag)::value><<<grid, S::NTHREADS, 0, stream>>>(
        n, static_cast<const double*>(st.mfma64Frags), static_cast<double*>(L->dofs),
        static_cast<const double*>(L->face_traces), L->face_neighbors, L->face_relations,
        static_cast<const double*>(L->aminus), L->face_types, lay);
  };
  if (defaultLayout64<S::B>(lay) && lay.aminusStride == 324) launch(std::true_type{});
  else launch(std::false_type{});
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

}  // namespace mfma64
}  // namespace sdg
