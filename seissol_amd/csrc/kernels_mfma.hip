// Host dispatch of the matrix-core arithmetics (orders 3-7): the split-product
// kernels (built by kernels_mfma_o<O>.hip) or the FP32 passes.
#include <hip/hip_runtime.h>

#include "engine.h"
#include "mfma_common.h"
#include "mx_common.h"

namespace sdg {

namespace {
int localPass(const EngineState& e, const double* coeffs, const sdg_layer* layer, bool writeIntegrated,
              hipStream_t stream, const mfma::LtsOut* lts) {
  if (e.order < 3 || e.order > 7) {
    setError("matrix-core path supports orders 3..7");
    return SDG_ERR_UNSUPPORTED;
  }
  if (mfma::splitProducts(e))
    return e.order == 6 ? mfma::MfmaOrder<6>::local(e, coeffs, layer, writeIntegrated, stream, lts)
                        : mfma::MfmaOrder<7>::local(e, coeffs, layer, writeIntegrated, stream, lts);
  sdg_layer own = *layer;
  if (!writeIntegrated) own.time_integrated = nullptr;
  bool v4 = false;
  if (own.num_elements > 0 &&
      !mfma::vectorAccess(cellLayout(e, &own), own.dofs, own.time_integrated, "matrix-core local pass", v4))
    return SDG_ERR_INVALID;
  mx::LtsOut out{};
  if (lts != nullptr) out = {lts->setup, lts->deriv};
  return launchLocalTracesMx(e, coeffs, lts != nullptr ? lts->reset : 1, &own, lts != nullptr ? &out : nullptr, stream);
}
}  // namespace

int launchLocalMfma(const EngineState& e, const double* coeffs, const sdg_layer* layer, bool writeIntegrated,
                    hipStream_t stream) {
  if (layer->derivatives != nullptr) {
    // the fused ader + local pass with derivatives (every cell stores them)
    const mfma::LtsOut lts{nullptr, static_cast<float*>(layer->derivatives), 1, 0};
    return localPass(e, coeffs, layer, writeIntegrated, stream, &lts);
  }
  return localPass(e, coeffs, layer, writeIntegrated, stream, nullptr);
}

int launchLocalIntegrationMfma(const EngineState& e, const double* coeffs, const sdg_layer* layer, int resetBuffers,
                               hipStream_t stream) {
  const mfma::LtsOut lts{layer->lts_setup, static_cast<float*>(layer->derivatives), resetBuffers, 0};
  return localPass(e, coeffs, layer, layer->time_integrated != nullptr, stream, &lts);
}

int launchNeighborMfma(const EngineState& e, const sdg_layer* layer, hipStream_t stream) {
  if (mfma::splitProducts(e) && e.order == mfma::kSplitNeighborOrder)
    return mfma::MfmaOrder<mfma::kSplitNeighborOrder>::neighbor(e, layer, stream);
  bool v4 = false;
  if (!mfma::vectorAccess(cellLayout(e, layer), layer->dofs, nullptr, "matrix-core neighbour pass", v4) &&
      layer->num_elements > 0)
    return SDG_ERR_INVALID;
  return launchNeighborTracesMx(e, layer, stream);
}

}  // namespace sdg
