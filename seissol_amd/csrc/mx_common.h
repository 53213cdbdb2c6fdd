// Tile geometry and device helpers of the element update on the matrix cores
// in the engine's own real type (FP64 or FP32, one product per contraction):
// kernels in mx_local.h and mx_neighbor.h, host data in kernels_mx.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "engine.h"

namespace sdg {
namespace mx {

constexpr int basis3(int o) { return o * (o + 1) * (o + 2) / 6; }
constexpr int basis2(int o) { return o * (o + 1) / 2; }
constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }
constexpr int ceil4(int a) { return (a + 3) / 4 * 4; }
constexpr int maxOf(int a, int b) { return a > b ? a : b; }

constexpr int kElems = 16;         // elements per tile: the columns of one matrix instruction
constexpr int kCols = 9 * kElems;  // GEMM columns (quantity, element) -> 16 q + e
constexpr int kStarLd = 73;        // an element's 72 star values, padded against bank conflicts
// an element's 4 x 81 AplusT values: 16-byte pieces aligned, conflict-free
template <typename real>
constexpr int kAplusLd = sizeof(real) == 8 ? 326 : 324;

// where the compact star values (24 per direction) of output quantity p lie,
// and the input quantities they multiply
__device__ constexpr int kStarQ[9][3] = {{6, 7, 8}, {6, 7, 8}, {6, 7, 8}, {6, 7, -1}, {7, 8, -1},
                                         {6, 8, -1}, {0, 3, 5}, {1, 3, 4}, {2, 4, 5}};
__device__ constexpr int kStarOff[9] = {0, 3, 6, 9, 11, 13, 15, 18, 21};
__device__ constexpr int kStarCnt[9] = {3, 3, 3, 2, 2, 2, 3, 3, 3};
// entry z of a compact star matrix: its column-major position q + 9 p
__device__ constexpr int kStarPos[24] = {6 + 0,  7 + 0,  8 + 0,  6 + 9,  7 + 9,  8 + 9,  6 + 18, 7 + 18,
                                         8 + 18, 6 + 27, 7 + 27, 7 + 36, 8 + 36, 6 + 45, 8 + 45, 0 + 54,
                                         3 + 54, 5 + 54, 1 + 63, 3 + 63, 4 + 63, 2 + 72, 4 + 72, 5 + 72};

// Geometry per order.  Fragments are stored per (row tile, k-step of 4), 64
// reals each in the lane order of the A operand (lane l: row l % 16, column
// l / 16 of the 16 x 4 block), the rows permuted so that a lane's four results
// are the consecutive rows 4g .. 4g + 3 (g = l / 16) in both real types.
template <int O>
struct Geo {
  static constexpr int B = basis3(O), B2 = basis2(O);
  static constexpr int MT = cdiv(B, 16);  // row tiles of the basis index
  static constexpr int KB = ceil4(B), KS = KB / 4;
  static constexpr int B2P = ceil4(B2);  // face rows padded to a multiple of 4
  static constexpr int KSF = B2P / 4;
  // Row tiles of the four faces' traces.  A face's first 16 rows form a tile;
  // its remaining rows need only the columns of the highest degrees, so they
  // get tiles of their own (two faces to a tile where they fit).
  static constexpr int MTF = B2P <= 8 ? 2 : (B2P <= 16 ? 4 : (B2P <= 24 ? 6 : 8));
  // the quad g (four rows) of trace tile t: its face, and its first row (B2P or more: none)
  static constexpr int traceFace(int t, int g) {
    return B2P <= 8 ? 2 * t + g / 2 : (t < 4 ? t : (B2P <= 24 ? 2 * (t - 4) + g / 2 : t - 4));
  }
  static constexpr int traceRow(int t, int g) {
    return B2P <= 8 ? 4 * (g % 2) : (t < 4 ? 4 * g : (B2P <= 24 ? 16 + 4 * (g % 2) : 16 + 4 * g));
  }
  // rows of the X area: the DOFs; dQ_1 and, behind it, dQ_2; two faces' W
  static constexpr int R1 = ceil4(basis3(O - 1)), R2 = O > 2 ? ceil4(basis3(O - 2)) : 0;
  static constexpr int XROWS = maxOf(maxOf(KB, R1 + R2), 2 * B2P);
  // fragment offsets (reals)
  static constexpr int64_t ck = 0;                               // [MT][3][KS]
  static constexpr int64_t vol = ck + 3LL * MT * KS * 64;        // [MT][3][KS]
  static constexpr int64_t trace = vol + 3LL * MT * KS * 64;     // [MTF][KS]     rT_f = fMrT_f / M2, last k-step first
  static constexpr int64_t flux = trace + 1LL * MTF * KS * 64;   // [MT][4][KSF]  rDivM_f diag(M2)
  // neighbour pass: rT_j in blocks of 8 columns (a lane's two consecutive
  // ones in one load), rDivM_f, and fP_h as rows of O (value, column) entries
  static constexpr int RT = cdiv(B2, 16), KB8 = cdiv(B, 8);
  static constexpr int64_t rt = flux + 4LL * MT * KSF * 64;      // [4][RT][KB8][64][2]
  static constexpr int64_t rdm = rt + 4LL * RT * KB8 * 128;      // [MT][4][KSF]
  static constexpr int64_t fP = rdm + 4LL * MT * KSF * 64;       // [3][B2][O] values
  static constexpr int64_t fPCol = fP + 3LL * B2 * O;            // [3][B2][O] columns (exact integers)
  static constexpr int64_t total = fPCol + 3LL * B2 * O;
  // k-step ranges [lo, hi) that hold a row tile's non-zeros, as (lo, hi) pairs
  static constexpr int rCk = 0;                       // [O - 1][MT]
  static constexpr int rVol = rCk + 2 * (O - 1) * MT; // [MT]
  static constexpr int rTrace = rVol + 2 * MT;        // [MTF]
  static constexpr int rFlux = rTrace + 2 * MTF;      // [MT][4]
  static constexpr int rRt = rFlux + 2 * 4 * MT;      // [4][RT], in blocks of 8 columns
  static constexpr int rTotal = rRt + 2 * 4 * RT;
};

// column stride of X: quads aligned to 16 bytes, and the 16 elements' columns
// (a multiple of 16 strides apart from each other's banks) conflict-free for
// the operand reads
template <typename real>
constexpr int columnStride(int rows) {
  if (sizeof(real) == 8) {
    while (rows % 4 != 2) ++rows;
  } else {
    while (rows % 8 != 4) ++rows;
  }
  return rows;
}

// logical row of physical A row i: FP64's accumulator register j of lane group
// g holds row g + 4 j, FP32's row 4 g + j
template <typename real>
constexpr int fragRow(int i) {
  return sizeof(real) == 8 ? 4 * (i % 4) + i / 4 : i;
}

template <typename real>
struct Vec;
template <>
struct Vec<double> {
  typedef double V4 __attribute__((ext_vector_type(4)));
};
template <>
struct Vec<float> {
  typedef float V4 __attribute__((ext_vector_type(4)));
};

__device__ inline Vec<double>::V4 mma(double a, double b, Vec<double>::V4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline Vec<float>::V4 mma(float a, float b, Vec<float>::V4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Global memory through buffer instructions: a uniform base, a 32-bit byte
// offset per lane, and a hardware range check that gives zero for loads and
// drops stores beyond `bytes`.  Lanes without work pass kNowhere, so that the
// kernels need no divergent branches around their accesses (a block of guarded
// loads waits on each in turn, and under register pressure the compiler has
// placed copies of live registers inside such blocks, where the inactive lanes
// lose them).
constexpr int kNowhere = 0x7fff0000;  // (no 32-bit sum with the small offsets added to it wraps)

template <typename real>
struct Buffer {
  __amdgpu_buffer_rsrc_t rsrc;
  using V4 = typename Vec<real>::V4;

  __device__ inline Buffer(const real* base, int64_t reals)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<real*>(base), 0,
                                               static_cast<int>(min(reals * static_cast<int64_t>(sizeof(real)),
                                                                    int64_t(0x7ff00000))),
                                               0x00027000)) {}
  // four consecutive reals at byte offset `off` (per lane) + `s` (uniform)
  __device__ inline V4 load4(int off, int s) const {
    typedef unsigned U4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(real) == 8) {
      union {
        U4 u[2];
        V4 v;
      } x;
      x.u[0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, s, 0);
      x.u[1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 16, s, 0);
      return x.v;
    } else {
      union {
        U4 u;
        V4 v;
      } x;
      x.u = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, s, 0);
      return x.v;
    }
  }
  // stores keep the scalar offset field zero: with a register there, stores of
  // 16 bytes have lost their last lanes' data to the next write of the data
  // registers (the compiler adds the wait state of that hazard only without)
  __device__ inline void store4(const V4& v, int off, int s) const {
    off += s;
    typedef unsigned U4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(real) == 8) {
      union {
        V4 v;
        U4 u[2];
      } x;
      x.v = v;
      __builtin_amdgcn_raw_buffer_store_b128(x.u[0], rsrc, off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(x.u[1], rsrc, off + 16, 0, 0);
    } else {
      union {
        V4 v;
        U4 u;
      } x;
      x.v = v;
      __builtin_amdgcn_raw_buffer_store_b128(x.u, rsrc, off, 0, 0);
    }
  }
  // 16 bytes at byte offset `off`
  __device__ inline auto load16(int off) const {
    typedef unsigned U4 __attribute__((ext_vector_type(4)));
    typedef real VP __attribute__((ext_vector_type(16 / sizeof(real))));
    union {
      U4 u;
      VP v;
    } x;
    x.u = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
    return x.v;
  }
  __device__ inline real load1(int off, int s) const {
    if constexpr (sizeof(real) == 8) {
      typedef unsigned U2 __attribute__((ext_vector_type(2)));
      union {
        U2 u;
        real v;
      } x;
      x.u = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, s, 0);
      return x.v;
    } else {
      return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, off, s, 0));
    }
  }
  __device__ inline void store1(real v, int off, int s) const {
    if constexpr (sizeof(real) == 8) {
      typedef unsigned U2 __attribute__((ext_vector_type(2)));
      union {
        real v;
        U2 u;
      } x;
      x.v = v;
      __builtin_amdgcn_raw_buffer_store_b64(x.u, rsrc, off + s, 0, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, off + s, 0, 0);
    }
  }
  // the quad of rows row .. row + 3 of a block of B rows (zero from B on) at
  // byte offset `block` + `s`
  template <int B>
  __device__ inline V4 loadQuad(int block, int row, int s) const {
    V4 v = load4(row < B ? block + row * static_cast<int>(sizeof(real)) : kNowhere, s);
    if constexpr (B % 4 != 0) {
#pragma unroll
      for (int j = B % 4; j < 4; ++j)
        if (row + j >= B) v[j] = real(0);
    }
    return v;
  }
  // the rows below m of that quad
  __device__ inline void storeQuad(const V4& v, int block, int row, int m, int s) const {
    const int at = block + row * static_cast<int>(sizeof(real));
    store4(v, row + 3 < m ? at : kNowhere, s);
    if (m % 4 != 0) {  // uniform
#pragma unroll
      for (int j = 0; j < 3; ++j)
        store1(v[j], row + 3 >= m && row + j < m ? at + j * static_cast<int>(sizeof(real)) : kNowhere, s);
    }
  }
};

// local-time-stepping outputs of the local pass (TimeCluster.cpp:380-434):
// per cell its LtsSetup bits say whether it stores its buffer (accumulated
// over the sub-steps a slower neighbour sees unless its cluster resets it) and its
// derivatives; setup == nullptr: the buffer and (if any) the derivatives of
// every cell
struct LtsOut {
  const uint16_t* setup = nullptr;
  void* deriv = nullptr;
};

// One launch over several clusters of a layer (local time stepping: the
// clusters that step at the same time), each with its own range of cells, time
// coefficients and reset flag; tiles do not cross the ranges.  Small clusters
// are bound by the chain of one tile, 20 us whatever their size, so they run
// beside the others.
struct ClusterStep {
  int64_t start = 0, end = 0;  // cells of the layer
  const double* coeffs = nullptr;  // time integral over the cluster's step
  const double* sub = nullptr;     // neighbour pass: over the sub-interval of a larger step
  int reset = 1;
};
constexpr int kMaxClusters = 16;

template <int O, typename real, int SETS>
struct Segments {
  int count = 0;
  int firstBlock[kMaxClusters] = {};
  int reset[kMaxClusters] = {};
  int64_t start[kMaxClusters] = {}, end[kMaxClusters] = {};
  real c[kMaxClusters][SETS][O] = {};

  // the number of blocks
  int64_t fill(const ClusterStep* steps, int n) {
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
      if (steps[i].end <= steps[i].start) continue;
      firstBlock[count] = static_cast<int>(blocks);
      start[count] = steps[i].start;
      end[count] = steps[i].end;
      reset[count] = steps[i].reset;
      for (int d = 0; d < O; ++d) {
        c[count][0][d] = steps[i].coeffs != nullptr ? static_cast<real>(steps[i].coeffs[d]) : real(0);
        if (SETS == 2) c[count][SETS - 1][d] = steps[i].sub != nullptr ? static_cast<real>(steps[i].sub[d]) : real(0);
      }
      blocks += (steps[i].end - steps[i].start + kElems - 1) / kElems;
      ++count;
    }
    return blocks;
  }
  // the segment of this block (uniform)
  __device__ inline int find() const {
    int s = 0;
    for (int i = 1; i < count; ++i) s = static_cast<int>(blockIdx.x) >= firstBlock[i] ? i : s;
    return s;
  }
};

// parts of the local pass
constexpr int kPredict = 1, kFlux = 2;

// host entry points of one order (explicitly instantiated per order)
template <int O>
struct Order {
  static int local(const EngineState& e, int parts, const ClusterStep* steps, int clusters, const sdg_layer* layer,
                   bool traces, const LtsOut* lts, hipStream_t stream);
  // neighbour flux; steps without coefficients: global time stepping; traces: from the layer's face traces
  // instead of the neighbours' DOFs
  static int neighbor(const EngineState& e, const sdg_layer* layer, const ClusterStep* steps, int clusters, bool traces,
                      hipStream_t stream);
};

}  // namespace mx

// the fused local pass in FP32 or FP64 writing the layer's face traces, with
// the outputs of `lts` (nullptr: neither derivatives nor LTS setup; a layer
// without time_integrated: no buffer)
int launchLocalTracesMx(const EngineState& e, const double* coeffs, int reset, const sdg_layer* layer,
                        const mx::LtsOut* lts, hipStream_t stream);
// the LTS passes of several clusters of a layer at once (its arrays whole)
int launchLocalClustersMx(const EngineState& e, const mx::ClusterStep* steps, int clusters, const sdg_layer* layer,
                          hipStream_t stream);
int launchNeighborClustersMx(const EngineState& e, const mx::ClusterStep* steps, int clusters, const sdg_layer* layer,
                             hipStream_t stream);
}  // namespace sdg
