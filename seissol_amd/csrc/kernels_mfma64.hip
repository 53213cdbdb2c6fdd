// Host side of the FP64 engines' matrix-core neighbour pass: the FP64 fragments of
// the global matrices and the dispatch over the orders 3-7 (the kernels of one
// order are built by kernels_mfma64_o<O>.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>

#include "engine.h"
#include "global_matrices.h"
#include "mfma_common.h"

namespace sdg {
namespace {

template <int O>
int uploadData64(EngineState& s, const double* gm) {
  using S = mfma64::Shape64<O>;
  const auto g = globalMatrixLayout(O);
  const int B = S::B, B2 = S::B2;
  std::vector<double> frags(S::total, 0.0);
  // rDivM_f per face, and fP_h as rows of at most O non-zeros
  for (int mt = 0; mt < S::MT; ++mt)
    for (int f = 0; f < 4; ++f)
      for (int ks = 0; ks < S::KSF; ++ks) {
        double* base = frags.data() + S::rdmN + ((static_cast<int64_t>(mt) * 4 + f) * S::KSF + ks) * 64;
        for (int l = 0; l < 64; ++l) {
          const int r = 16 * mt + l % 16, m = 4 * ks + l / 16;
          base[l] = (r < B && m < B2) ? gm[g.rDivM + (f * B + r) * B2 + m] : 0.0;
        }
      }
  for (int h = 0; h < 3; ++h) {
    double mx = 0.0;
    for (int i = 0; i < B2 * B2; ++i) mx = std::max(mx, std::fabs(gm[g.fP + h * B2 * B2 + i]));
    for (int r = 0; r < B2; ++r) {
      int cnt = 0;
      for (int c = 0; c < B2; ++c) {
        const double v = gm[g.fP + (h * B2 + r) * B2 + c];
        if (std::fabs(v) <= 1e-13 * mx) continue;
        if (cnt == O) {
          setError("face permutation matrix with more than `order` non-zeros in a row");
          return SDG_ERR_INVALID;
        }
        frags[S::tFP + (h * B2 + r) * O + cnt] = v;
        frags[S::tFPCol + (h * B2 + r) * O + cnt] = static_cast<double>(c);
        ++cnt;
      }
    }
  }
  if (s.mfma64Frags == nullptr) SDG_HIP_CHECK(hipMalloc(&s.mfma64Frags, frags.size() * sizeof(double)));
  SDG_HIP_CHECK(hipMemcpy(s.mfma64Frags, frags.data(), frags.size() * sizeof(double), hipMemcpyHostToDevice));
  return SDG_OK;
}

}  // namespace

int64_t mfma64::fragmentCount(int order) {
  switch (order) {
    case 3: return Shape64<3>::total;
    case 4: return Shape64<4>::total;
    case 5: return Shape64<5>::total;
    case 6: return Shape64<6>::total;
    case 7: return Shape64<7>::total;
    default: return 0;
  }
}

int uploadMfma64(EngineState& s, const double* gm) {
  switch (s.order) {
    case 3: return uploadData64<3>(s, gm);
    case 4: return uploadData64<4>(s, gm);
    case 5: return uploadData64<5>(s, gm);
    case 6: return uploadData64<6>(s, gm);
    case 7: return uploadData64<7>(s, gm);
    default: return SDG_OK;  // no FP64 matrix-core pass at this order
  }
}

bool hasMfma64(const EngineState& e) {
  return e.arithmetic == SDG_FP64 && e.mfma64Frags != nullptr && e.kernels == SDG_KERNELS_AUTO;
}

int launchNeighborMfma64(const EngineState& e, const sdg_layer* layer, hipStream_t stream) {
  switch (e.order) {
    case 3: return mfma64::MfmaOrder64<3>::neighbor(e, layer, stream);
    case 4: return mfma64::MfmaOrder64<4>::neighbor(e, layer, stream);
    case 5: return mfma64::MfmaOrder64<5>::neighbor(e, layer, stream);
    case 6: return mfma64::MfmaOrder64<6>::neighbor(e, layer, stream);
    case 7: return mfma64::MfmaOrder64<7>::neighbor(e, layer, stream);
    default: setError("the FP64 matrix-core pass supports orders 3..7"); return SDG_ERR_UNSUPPORTED;
  }
}

}  // namespace sdg
