// Internal engine state and kernel entry points shared by the HIP sources.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/seissol_amd.h"

namespace sdg {

void setError(const std::string& msg);
int hipFail(hipError_t err, const char* what);
#define SDG_HIP_CHECK(call)                                  \
  do {                                                       \
    hipError_t err_ = (call);                                \
    if (err_ != hipSuccess) return ::sdg::hipFail(err_, #call); \
  } while (0)

constexpr int kMaxOrder = 8;
constexpr int kMinOrder = 2;

// Offsets (in reals) of the device copies of the global matrices.  All
// matrices are stored transposed relative to the generator output so that
// consecutive output rows are consecutive in memory:
//   ck  [3][B][B]    ck[j][l][k]   = -kDivMT_j[k][l]
//   vol [3][B][B]    vol[j][l][k]  =  kDivM_j[k][l]
//   fmrt[4][B][B2]   fmrt[f][l][m] =  fMrT_f[m][l]
//   rt  [4][B][B2]   rt[j][l][m]   =  rT_j[m][l]
//   fp  [3][B2][B2]  fp[h][n][m]   =  fP_h[m][n]
//   rdm [4*B2][B]    rdm[f*B2+m][k] = rDivM_f[k][m]
struct DeviceMatrixLayout {
  int64_t ck, vol, fmrt, rt, fp, rdm, total;
};
DeviceMatrixLayout deviceMatrixLayout(int order);

inline bool matrixCore(int arithmetic) {
  return arithmetic == SDG_BF16X3 || arithmetic == SDG_BF16X6 || arithmetic == SDG_F16X3;
}

// Storage layout of a layer's per-cell arrays as the kernels see them.
// DOF-like blocks (dofs, buffers, Taylor outputs) are [9][ldq] per cell, a
// derivative block of m rows is [9][rows(m)], the blocks one after another;
// the per-cell operators sit starStride / aplusStride / aminusStride reals
// apart, the star matrices as 3 x 81 dense or 3 x 24 non-zeros.
struct CellLayout {
  int32_t ldq = 0;
  int32_t align = 1;      // rows of a block are rounded up to a multiple of this (a power of two)
  int64_t qStride = 0;    // 9 * ldq
  int64_t dsize = 0;      // reals of one cell's derivatives
  int64_t starStride = 0, aplusStride = 324, aminusStride = 324;
  int32_t starCompact = 0;
  int32_t pad_ = 0;
  __host__ __device__ int rows(int m) const { return (m + align - 1) & ~(align - 1); }
};

struct EngineState {
  int order = 0;
  int arithmetic = SDG_FP64;
  // layout of the cells' arrays (sdg_engine_set_layout): alignment in bytes
  // (0 = packed) and the star format
  int alignment = 0;
  int starFormat = SDG_STAR_DENSE;
  void* matrices = nullptr;  // device, real type of the engine
  DeviceMatrixLayout layout{};
  // split-product engines: pre-split bf16 fragments and FP32 tables
  void* mfmaFrags = nullptr;
  void* mfmaTables = nullptr;
  // dynamic rupture face matrices (V3mTo2n, V3mTo2nTWDivM), on first use
  void* drMatrices = nullptr;
  // SDG_KERNELS_AUTO: the matrix-core passes where the engine has them;
  // SDG_KERNELS_VALU: the VALU kernels only (sdg_engine_set_kernels)
  int kernels = SDG_KERNELS_AUTO;
  // orders 3-7: fragments in the real type and k-step ranges of the
  // matrix-core passes of mx_local.h
  void* mxFrags = nullptr;
  int* mxRanges = nullptr;
  bool mxNeighbor = false;  // the fP_h are sparse enough for the neighbour pass of mx_neighbor.h
};

// the layout of `layer` (its strides, 0 = the dense defaults) under the engine's settings
CellLayout cellLayout(const EngineState& e, const sdg_layer* layer);
// proxy kernels 0-4 on a validated layer (sdg_proxy_run); allocates nothing
int proxyRun(const EngineState& st, int kernelId, int steps, double dt, const sdg_layer* layer, hipStream_t s);
// the same for arrays handed over without a layer (derivatives, Taylor outputs)
CellLayout engineLayout(const EngineState& e);
// checks the per-cell strides of `layer` against the minimum sizes; sets the error text
bool layerStridesOk(const EngineState& e, const sdg_layer* layer, const char* who);

}  // namespace sdg

struct sdg_engine {
  sdg::EngineState s;
};

namespace sdg {
// kernels_valu.hip
int launchAder(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream);
int launchAderLocal(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream);
int launchLocal(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
int launchNeighbor(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
int launchTaylor(const EngineState& e, const double* coeffs, const void* derivatives, void* out, int64_t n,
                 hipStream_t stream);
// local time stepping kernels; `variant` selects a tile shape (0..3, 0 = default)
constexpr int kTileVariants = 4;
// neighbour pass: the kTileVariants tiles of kNeighbor, then kNeighborRows
// (one element per 16-lane row)
constexpr int kNeighborRowsVariant = kTileVariants;
constexpr int kNeighborVariants = kTileVariants + 1;
int launchLocalIntegration(const EngineState& e, const double* coeffs, const sdg_layer* layer, int resetBuffers,
                           hipStream_t stream, int variant = 0);
int launchNeighboringIntegration(const EngineState& e, const double* timeCoeffs, const double* subtimeCoeffs,
                                 const sdg_layer* layer, hipStream_t stream, int variant = 0);
// kernels_mfma.hip
int launchLocalMfma(const EngineState& e, const double* coeffs, const sdg_layer* layer, bool writeIntegrated,
                    hipStream_t stream);
int launchNeighborMfma(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
// kernels_mx.hip: the cell-local pass on the matrix cores in the engine's real
// type (orders 3-7, kernel family AUTO): predictor alone, volume and local
// flux from a given time integral, both fused (FP64: with face traces when the
// layer has them), and the LTS local pass
bool hasMx(const EngineState& e);
// `own`: the generated matrices, which tell a caller's zeros from its small entries
int uploadMx(EngineState& s, const double* globalMatrices, const double* own);
int launchAderMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream);
int launchLocalMx(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
int launchAderLocalMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream);
int launchLocalIntegrationMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, int resetBuffers,
                             hipStream_t stream);
// the neighbour pass from the neighbours' buffers (LTS: with the time
// coefficients, else nullptr: global time stepping)
bool hasNeighborMx(const EngineState& e);
// whether one call over `cells` cells, from DOFs or from LTS buffers and
// derivatives, is faster with it than on the VALU.  Not at ORDER 3 in FP32, nor
// in FP64 from DOFs up to 24 cells per CU: a tile's two barriers and its groups
// padded to 16 tasks outweigh 10 x 6 products (periodic and random links, VALU
// / matrix cores: FP32 300 cells 8.8 / 14.8 and 16.2 us, 5,000 11.2 / 17.6 and
// 19.3, 50,000 48 / 53 and 57, LTS 2,560 12.6 / 19.0; FP64 5,000 22 / 23 and
// 26, 6,500 27 / 24 and 27; LTS 2,560 25.9 / 23.0).  The clusters of a layer
// share its launch, which is faster there as well (a macro step of 51,200 cells
// in FP32 803 / 779 us).
bool prefersNeighborMx(const EngineState& e, int64_t cells, bool lts);
int launchNeighborMx(const EngineState& e, const sdg_layer* layer, const double* timeCoeffs,
                     const double* subtimeCoeffs, hipStream_t stream);
// the same from the face traces the local pass wrote (layer->face_traces,
// [n][4][9][B2P] in the real type)
int launchNeighborTracesMx(const EngineState& e, const sdg_layer* layer, hipStream_t stream);
// the LTS local pass on the matrix cores: buffers and derivatives per the
// layer's lts_setup (TimeCluster::computeLocalIntegration), no face traces
int launchLocalIntegrationMfma(const EngineState& e, const double* coeffs, const sdg_layer* layer, int resetBuffers,
                               hipStream_t stream);
}  // namespace sdg
