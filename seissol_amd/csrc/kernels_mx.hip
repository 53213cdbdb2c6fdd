// Host side of the matrix-core passes in the engine's real type: the fragments
// of the global matrices, the k-step ranges that hold each row tile's
// non-zeros, and the dispatch over the orders 3-7 (the kernels of one order
// are built by kernels_mx_o<O>.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>

#include "engine.h"
#include "global_matrices.h"
#include "mfma_common.h"
#include "mx_common.h"

namespace sdg {
namespace {

using Matrix = std::function<double(int, int)>;

// One row tile (16 rows) of A: fragments over k-steps [0, ksteps) in the lane
// order of the A operand, and the range of k-steps that holds its non-zeros
template <typename real>
void tileFragments(const Matrix& A, int ksteps, real* out) {
  for (int ks = 0; ks < ksteps; ++ks)
    for (int l = 0; l < 64; ++l) out[ks * 64 + l] = static_cast<real>(A(mx::fragRow<real>(l % 16), 4 * ks + l / 16));
}
// rows < rowEnd, columns < colEnd, in steps of `step` columns; lo < hi always (a zero tile keeps k-step 0)
void tileRange(const std::vector<Matrix>& As, int rowEnd, int colEnd, int step, int* out) {
  int lo = 1 << 20, hi = 0;
  for (const Matrix& A : As)
    for (int r = 0; r < rowEnd && r < 16; ++r)
      for (int c = 0; c < colEnd; ++c)
        if (A(r, c) != 0.0) {
          lo = std::min(lo, c / step);
          hi = std::max(hi, c / step + 1);
        }
  out[0] = hi == 0 ? 0 : lo;
  out[1] = hi == 0 ? 1 : hi;
}
double largest(const double* p, int64_t n) {
  double m = 0.0;
  for (int64_t i = 0; i < n; ++i) m = std::max(m, std::fabs(p[i]));
  return m;
}

// The matrices `gm` with the rounding noise of their quadrature set to zero:
// entries at places where the basis makes the exact value zero (there the
// generated matrices `own` have nothing but noise, up to 3e-15 of their
// largest entry, and nothing below 2e-6 elsewhere) that are no larger than such
// noise.  Every other entry of a caller's matrices counts, however small.
std::vector<double> withoutNoise(int order, const double* gm, const double* own) {
  const auto g = globalMatrixLayout(order);
  const int64_t B = numBasis3(order), B2 = numBasis2(order);
  std::vector<double> out(gm, gm + g.total);
  auto clean = [&](size_t at, int64_t n) {
    const double exact = 1e-13 * largest(own + at, n), noise = 1e-14 * largest(gm + at, n);
    for (size_t i = at; i < at + n; ++i)
      if (std::fabs(own[i]) <= exact && std::fabs(gm[i]) <= noise) out[i] = 0.0;
  };
  clean(g.kDivMT, 3 * B * B);
  clean(g.kDivM, 3 * B * B);
  clean(g.fMrT, 4 * B2 * B);
  clean(g.rDivM, 4 * B * B2);
  clean(g.rT, 4 * B2 * B);
  for (int h = 0; h < 3; ++h) clean(g.fP + h * B2 * B2, B2 * B2);
  return out;
}

template <typename real, int O>
int uploadOrder(EngineState& s, const double* gm, const double* own) {
  using G = mx::Geo<O>;
  const auto g = globalMatrixLayout(O);
  constexpr int B = G::B, B2 = G::B2, B2P = G::B2P, KS = G::KS;
  std::vector<real> frags(G::total, real(0));
  std::vector<int> ranges(G::rTotal, 0);
  const std::vector<double> nz = withoutNoise(O, gm, own);  // for the ranges
  // a caller's own matrices may have fuller rows: an FP32 engine has no
  // neighbour pass here then, every other one refuses them; with entries that the
  // lists below leave out, no engine has it
  bool sparseFP = true;
  for (int t = 0; t < G::MT; ++t) {
    std::vector<Matrix> ck, vol;
    for (int j = 0; j < 3; ++j) {
      auto block = [=](const double* m, size_t at) {
        return Matrix([=](int r, int c) {
          r += 16 * t;
          return r < B && c < B ? m[at + (j * B + r) * B + c] : 0.0;
        });
      };
      const Matrix T = block(gm, g.kDivMT);
      tileFragments<real>([&](int r, int c) { return -T(r, c); }, KS,
                          frags.data() + G::ck + (static_cast<int64_t>(t) * 3 + j) * KS * 64);
      tileFragments<real>(block(gm, g.kDivM), KS, frags.data() + G::vol + (static_cast<int64_t>(t) * 3 + j) * KS * 64);
      ck.push_back(block(nz.data(), g.kDivMT));
      vol.push_back(block(nz.data(), g.kDivM));
    }
    // derivative d has basis3(O - d) rows of basis3(O - d + 1) columns
    for (int d = 1; d < O; ++d)
      tileRange(ck, mx::basis3(O - d) - 16 * t, mx::basis3(O - d + 1), 4,
                ranges.data() + G::rCk + 2 * ((d - 1) * G::MT + t));
    tileRange(vol, 16, B, 4, ranges.data() + G::rVol + 2 * t);
    for (int f = 0; f < 4; ++f) {
      auto block = [=](const double* m) {
        return Matrix([=](int r, int c) {
          r += 16 * t;
          return r < B && c < B2 ? m[g.rDivM + (f * B + r) * B2 + c] : 0.0;
        });
      };
      const Matrix R = block(gm);
      tileFragments<real>([&](int r, int c) { return c < B2 ? R(r, c) * gm[g.mass2 + c] : 0.0; }, G::KSF,
                          frags.data() + G::flux + (static_cast<int64_t>(t) * 4 + f) * G::KSF * 64);
      tileFragments<real>(R, G::KSF, frags.data() + G::rdm + (static_cast<int64_t>(t) * 4 + f) * G::KSF * 64);
      tileRange({block(nz.data())}, 16, B2, 4, ranges.data() + G::rFlux + 2 * (t * 4 + f));
    }
  }
  for (int t = 0; t < G::MTF; ++t) {
    // k-steps from the last columns to the first (see gemm, mx_local.h)
    auto block = [=](const double* matrices) {
      return Matrix([=](int r, int c) {
        c = 4 * (KS - 1 - c / 4) + c % 4;
        const int f = G::traceFace(t, r / 4), m = G::traceRow(t, r / 4) + r % 4;
        return m < B2 && c < B ? matrices[g.fMrT + (f * B2 + m) * B + c] : 0.0;
      });
    };
    const Matrix F = block(gm);
    tileFragments<real>(
        [&](int r, int c) {
          const int m = G::traceRow(t, r / 4) + r % 4;
          return m < B2 ? F(r, c) / gm[g.mass2 + m] : 0.0;
        },
        KS, frags.data() + G::trace + static_cast<int64_t>(t) * KS * 64);
    tileRange({block(nz.data())}, 16, G::KB, 4, ranges.data() + G::rTrace + 2 * t);
  }
  // rT_j of the neighbour pass: lane l of block k holds columns 8 k + 2 (l / 16) + {0, 1}
  for (int j = 0; j < 4; ++j)
    for (int r = 0; r < G::RT; ++r) {
      auto block = [=](const double* m) {
        return Matrix([=](int i, int c) {
          i += 16 * r;
          return i < B2 && c < B ? m[g.rT + (j * B2 + i) * B + c] : 0.0;
        });
      };
      const Matrix U = block(gm);
      real* const out = frags.data() + G::rt + (static_cast<int64_t>(j) * G::RT + r) * G::KB8 * 128;
      for (int k = 0; k < G::KB8; ++k)
        for (int l = 0; l < 64; ++l)
          for (int i = 0; i < 2; ++i)
            out[(k * 64 + l) * 2 + i] = static_cast<real>(U(mx::fragRow<real>(l % 16), 8 * k + 2 * (l / 16) + i));
      tileRange({block(nz.data())}, 16, B, 8, ranges.data() + G::rRt + 2 * (j * G::RT + r));
    }
  // fP_h as rows of at most O non-zeros, padded with zeros
  for (int h = 0; h < 3; ++h) {
    const double tolP = 1e-13 * largest(gm + g.fP + h * B2 * B2, int64_t(B2) * B2);
    for (int r = 0; r < B2; ++r) {
      int cnt = 0;
      for (int c = 0; c < B2; ++c) {
        const double v = gm[g.fP + (h * B2 + r) * B2 + c];
        if (std::fabs(v) <= tolP) {
          if (nz[g.fP + (h * B2 + r) * B2 + c] != 0.0) sparseFP = false;
          continue;
        }
        if (cnt == O) {
          if (sizeof(real) == 8 || matrixCore(s.arithmetic)) {
            setError("face permutation matrix with more than `order` non-zeros in a row");
            return SDG_ERR_INVALID;
          }
          sparseFP = false;
          break;
        }
        frags[G::fP + (h * B2 + r) * O + cnt] = static_cast<real>(v);
        frags[G::fPCol + (h * B2 + r) * O + cnt] = static_cast<real>(c);
        ++cnt;
      }
    }
  }
  s.mxNeighbor = sparseFP;
  if (s.mxFrags == nullptr) SDG_HIP_CHECK(hipMalloc(&s.mxFrags, frags.size() * sizeof(real)));
  if (s.mxRanges == nullptr)
    SDG_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&s.mxRanges), ranges.size() * sizeof(int)));
  SDG_HIP_CHECK(hipMemcpy(s.mxFrags, frags.data(), frags.size() * sizeof(real), hipMemcpyHostToDevice));
  SDG_HIP_CHECK(hipMemcpy(s.mxRanges, ranges.data(), ranges.size() * sizeof(int), hipMemcpyHostToDevice));
  return SDG_OK;
}

template <typename F>
int orders(const EngineState& e, F&& f) {
  switch (e.order) {
    case 3: return f(mx::Order<3>{});
    case 4: return f(mx::Order<4>{});
    case 5: return f(mx::Order<5>{});
    case 6: return f(mx::Order<6>{});
    case 7: return f(mx::Order<7>{});
    default: setError("the matrix-core passes support orders 3..7"); return SDG_ERR_UNSUPPORTED;
  }
}

}  // namespace

int uploadMx(EngineState& s, const double* gm, const double* own) {
  const bool dbl = s.arithmetic == SDG_FP64;
  switch (s.order) {
    case 3: return dbl ? uploadOrder<double, 3>(s, gm, own) : uploadOrder<float, 3>(s, gm, own);
    case 4: return dbl ? uploadOrder<double, 4>(s, gm, own) : uploadOrder<float, 4>(s, gm, own);
    case 5: return dbl ? uploadOrder<double, 5>(s, gm, own) : uploadOrder<float, 5>(s, gm, own);
    case 6: return dbl ? uploadOrder<double, 6>(s, gm, own) : uploadOrder<float, 6>(s, gm, own);
    case 7: return dbl ? uploadOrder<double, 7>(s, gm, own) : uploadOrder<float, 7>(s, gm, own);
    default: return SDG_OK;  // orders 2 and 8: the VALU kernels
  }
}

bool hasMx(const EngineState& e) { return e.mxFrags != nullptr && e.kernels == SDG_KERNELS_AUTO; }

bool hasNeighborMx(const EngineState& e) { return hasMx(e) && e.mxNeighbor; }

bool prefersNeighborMx(const EngineState& e, int64_t cells, bool lts) {
  return hasNeighborMx(e) && (e.order > 3 || (e.arithmetic == SDG_FP64 && (lts || cells > 24 * 256)));
}

namespace {
// every cell of the layer in one step
mx::ClusterStep whole(const sdg_layer* layer, const double* coeffs, const double* sub, int reset) {
  return {0, layer->num_elements, coeffs, sub, reset};
}
}  // namespace

int launchNeighborMx(const EngineState& e, const sdg_layer* layer, const double* timeCoeffs,
                     const double* subtimeCoeffs, hipStream_t stream) {
  const mx::ClusterStep step = whole(layer, timeCoeffs, subtimeCoeffs, 1);
  return orders(e, [&](auto o) { return o.neighbor(e, layer, &step, 1, false, stream); });
}

int launchNeighborClustersMx(const EngineState& e, const mx::ClusterStep* steps, int clusters, const sdg_layer* layer,
                             hipStream_t stream) {
  return orders(e, [&](auto o) { return o.neighbor(e, layer, steps, clusters, false, stream); });
}

int launchNeighborTracesMx(const EngineState& e, const sdg_layer* layer, hipStream_t stream) {
  const mx::ClusterStep step = whole(layer, nullptr, nullptr, 1);
  return orders(e, [&](auto o) { return o.neighbor(e, layer, &step, 1, true, stream); });
}

int launchAderMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream) {
  const mx::LtsOut lts{layer->lts_setup, layer->derivatives};
  const mx::ClusterStep step = whole(layer, coeffs, nullptr, 1);
  return orders(e, [&](auto o) { return o.local(e, mx::kPredict, &step, 1, layer, false, &lts, stream); });
}

int launchLocalMx(const EngineState& e, const sdg_layer* layer, hipStream_t stream) {
  const mx::ClusterStep step = whole(layer, nullptr, nullptr, 1);
  return orders(e, [&](auto o) { return o.local(e, mx::kFlux, &step, 1, layer, false, nullptr, stream); });
}

int launchAderLocalMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, hipStream_t stream) {
  // only the FP64 neighbour pass reads traces of this kernel
  const bool fp64 = e.arithmetic == SDG_FP64;
  // FP64: the buffer and derivatives of every cell; FP32: per the layer's LTS setup where it has one
  const mx::LtsOut lts{fp64 ? nullptr : layer->lts_setup, layer->derivatives};
  const bool some = lts.deriv != nullptr || lts.setup != nullptr;
  const mx::ClusterStep step = whole(layer, coeffs, nullptr, 1);
  return orders(e, [&](auto o) {
    return o.local(e, mx::kPredict | mx::kFlux, &step, 1, layer, fp64, some ? &lts : nullptr, stream);
  });
}

int launchLocalTracesMx(const EngineState& e, const double* coeffs, int reset, const sdg_layer* layer,
                        const mx::LtsOut* lts, hipStream_t stream) {
  const mx::ClusterStep step = whole(layer, coeffs, nullptr, reset);
  return orders(e, [&](auto o) { return o.local(e, mx::kPredict | mx::kFlux, &step, 1, layer, true, lts, stream); });
}

int launchLocalClustersMx(const EngineState& e, const mx::ClusterStep* steps, int clusters, const sdg_layer* layer,
                          hipStream_t stream) {
  bool v4 = false;
  if (matrixCore(e.arithmetic) &&
      !mfma::vectorAccess(cellLayout(e, layer), layer->dofs, layer->time_integrated, "matrix-core local pass", v4))
    return SDG_ERR_INVALID;
  const mx::LtsOut lts{layer->lts_setup, layer->derivatives};
  return orders(e, [&](auto o) {
    return o.local(e, mx::kPredict | mx::kFlux, steps, clusters, layer, false, &lts, stream);
  });
}

int launchLocalIntegrationMx(const EngineState& e, const double* coeffs, const sdg_layer* layer, int resetBuffers,
                             hipStream_t stream) {
  const mx::LtsOut lts{layer->lts_setup, layer->derivatives};
  const mx::ClusterStep step = whole(layer, coeffs, nullptr, resetBuffers);
  return orders(e, [&](auto o) {
    return o.local(e, mx::kPredict | mx::kFlux, &step, 1, layer, e.arithmetic == SDG_FP64, &lts, stream);
  });
}

}  // namespace sdg
