// Tile geometry shared by the matrix-core kernels and the host code that
// prepares their pre-split, pre-swizzled matrix fragments.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "engine.h"

namespace sdg {
namespace mfma {

constexpr int basis3(int o) { return o * (o + 1) * (o + 2) / 6; }
constexpr int basis2(int o) { return o * (o + 1) / 2; }
constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }

// bf16 elements of one (m-tile, k-step) fragment set: 64 lanes x 8 values for
// each of the two planes, one plane after the other.
constexpr int kFragPlane = 512;
constexpr int kFragPair = 2 * kFragPlane;
constexpr int kTileElems = 16;        // elements per workgroup tile
constexpr int kCols = 9 * kTileElems; // GEMM columns (quantity, element)

template <int O>
struct MShape {
  static constexpr int B = basis3(O);
  static constexpr int B2 = basis2(O);
  static constexpr int MT = cdiv(B, 16);            // row tiles of the basis index
  static constexpr int KPB = cdiv(B, 32) * 32;      // padded K over the basis index
  static constexpr int KSB = KPB / 32;
  static constexpr int B2P = (B2 + 3) / 4 * 4;      // face rows padded to a multiple of 4
  static constexpr int FR = 4 * B2P;                // rows of the four stacked (padded) face operands
  static constexpr int MTF = cdiv(FR, 16);
  static constexpr int KPF = cdiv(FR, 32) * 32;
  static constexpr int KSF = KPF / 32;
  static constexpr int KMAX = KPB > KPF ? KPB : KPF;
  static constexpr int LDX = KMAX + 8;              // bf16 stride of one X column (bank spread)
  static constexpr int THREADS = 64 * MT;
  // fragment offsets (bf16 elements)
  static constexpr int64_t ck = 0;                                   // [3][MT][KSB]
  static constexpr int64_t vol = ck + 3LL * MT * KSB * kFragPair;    // [3][MT][KSB]
  static constexpr int64_t fmrt = vol + 3LL * MT * KSB * kFragPair;  // [MTF][KSB]
  static constexpr int64_t rdm = fmrt + 1LL * MTF * KSB * kFragPair; // [MT][KSF]
  // rDivM_f one face at a time: k-step f holds face f's B2 columns, zero-padded to 32
  static constexpr int64_t rdmF = rdm + 1LL * MT * KSF * kFragPair;  // [MT][4]
  static constexpr int64_t total = rdmF + 4LL * MT * kFragPair;
  // float tables: fP[3][B2][B2] as at most O non-zeros per row (every fP_h row has at most O)
  static constexpr int tFP = 0;                   // fP_h rows as O (value) entries: [3][B2][O]
  static constexpr int tFPCol = tFP + 3 * B2 * O; // their columns (exact small integers): [3][B2][O]
  static constexpr int tTotal = tFPCol + 3 * B2 * O;
};

// local-time-stepping outputs of the local pass (TimeCluster.cpp:380-434):
// per cell its LtsSetup bits say whether it stores its buffer (accumulated
// over the sub-steps a slower neighbour sees unless `reset`) and its
// derivatives; setup == nullptr: buffer (if any) stored, derivatives (if any)
// stored for every cell
struct LtsOut {
  const uint16_t* setup = nullptr;
  float* deriv = nullptr;
  int reset = 1;
  int pad_ = 0;
};

// 16-byte DOF accesses: every block starts on a multiple of 4 reals and the
// arrays are 16-byte aligned (always so for B a multiple of 4 on aligned arrays)
inline bool vectorAccess(const CellLayout& lay, const void* dofs, const void* integ, const char* who, bool& v4) {
  const bool aligned = (reinterpret_cast<uintptr_t>(dofs) % 16 == 0) &&
                       (integ == nullptr || reinterpret_cast<uintptr_t>(integ) % 16 == 0);
  v4 = lay.ldq % 4 == 0 && aligned;
  if (lay.ldq % 4 == 0 && !aligned) {
    setError(std::string(who) + ": dofs and time_integrated must be 16-byte aligned");
    return false;
  }
  return true;
}

// Which engines run on split products: the two-plane form, whose three bf16
// products per contraction beat the FP32 pass of mx_local.h where the row
// tiles are full.  Every other matrix-core form runs the FP32 passes, which
// are at least as accurate (error of a step's DOFs against 64 bits on random
// links, split -> FP32, orders 3 to 7: f16x3 1.75, 1.97, 2.12, 2.34, 2.55e-7 ->
// 1.41, 1.64, 1.82, 2.04, 2.31e-7; bf16x6 1.66, 1.90, 2.12, 2.37, 2.71e-7 -> the
// same): their 4-row k-steps skip the matrices' zeros
// (32-row steps are mostly padding at low orders), they need no column scales
// (f16x3) and half the products of three planes (bf16x6).  Whole step, random
// links, split -> FP32 local pass: f16x3 ORDER 6 1M cells 7.93 -> 7.42 ms, 10k
// 119 -> 106 us, 1k 59.3 -> 58.8; ORDER 7 120k 1965 -> 1917; f16x3 60k ORDER 3
// 171 -> 121, ORDER 4 280 -> 189, ORDER 5 448 -> 326; bf16x6 ORDER 6 60k 784 ->
// 529, ORDER 7 120k 2225 -> 1914; bf16x3 60k ORDER 5 403 -> 326, but ORDER 6
// 200k 1335 -> 1392 and ORDER 7 120k 1677 -> 1914.
constexpr bool splitProducts(int arithmetic, int order) { return arithmetic == SDG_BF16X3 && order >= 6; }
inline bool splitProducts(const EngineState& e) { return splitProducts(e.arithmetic, e.order); }
// Their neighbour pass: at ORDER 7 the FP32 pass from the traces is faster (60k
// cells 921 -> 862 us a step), at ORDER 6 it is not (459 -> 478).
constexpr int kSplitNeighborOrder = 6;

// host entry points of one order's kernels
template <int O>
struct MfmaOrder {
  // local pass; lts == nullptr: the GTS pass (face traces, no derivatives)
  static int local(const EngineState& e, const double* coeffs, const sdg_layer* layer, bool writeIntegrated,
                   hipStream_t stream, const LtsOut* lts);
  static int neighbor(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
};

}  // namespace mfma
}  // namespace sdg
