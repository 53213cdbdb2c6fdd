// Local time stepping (rate 2): the per-cell LTS setup, the cluster-wise
// local and neighbour integration, and the macro step of all clusters,
// enqueued directly or replayed from a captured hipGraph.
//
// Clusters: cluster c advances with dt_c = dt0 * 2^c; its cells are the
// contiguous range [start[c], start[c+1]) of one layer whose arrays hold all
// clusters, so neighbour indices are global.  One macro step (dt of the
// slowest cluster) runs, per cluster step,
//   predict(c, t)  - ader + local integral (TimeCluster::computeLocalIntegration,
//                    TimeCluster.cpp:358-434): buffer (stored or accumulated
//                    over the two sub-steps a slower neighbour sees) and
//                    derivatives of the cells that provide them,
//   step(c-1, t), step(c-1, t + dt_{c-1})  - the two steps of the faster cluster,
//   correct(c, t)  - neighbour integral (TimeCluster::computeNeighboringIntegration,
//                    TimeCluster.cpp:540-628) from buffers or from derivatives
//                    over [t, t + dt_c] (TimeCommon.cpp:40-87).
// A faster cluster reads a slower neighbour's derivatives, expanded at the
// start T of that neighbour's step, over [t - T, t - T + dt_c] (the
// subTimeStart of TimeCluster.cpp:799); the slower cluster reads the faster
// cluster's buffer summed over its two steps.
#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "engine.h"
#include "mfma_common.h"
#include "mx_common.h"

using namespace sdg;

namespace {

constexpr uint16_t kNHD0 = 1u << 0;  // neighbour on face 0 provides derivatives
constexpr uint16_t kGTS0 = 1u << 4;  // neighbour on face 0 is in the same cluster
constexpr uint16_t kBuffers = SDG_LTS_HAS_BUFFERS;
constexpr uint16_t kDerivatives = SDG_LTS_HAS_DERIVATIVES;
constexpr uint16_t kAccumulate = SDG_LTS_ACCUMULATE_BUFFERS;

bool ltsLayerOk(const sdg_layer* L, bool neighbors, const char* who) {
  if (L == nullptr || L->num_elements < 0) {
    setError(std::string(who) + ": invalid layer");
    return false;
  }
  if (L->num_elements == 0) return true;
  if (L->dofs == nullptr || L->time_integrated == nullptr || L->star == nullptr || L->aplus == nullptr ||
      L->lts_setup == nullptr || L->derivatives == nullptr) {
    setError(std::string(who) + ": dofs, buffers, derivatives, star, aplus and lts_setup are required");
    return false;
  }
  if (neighbors && (L->face_neighbors == nullptr || L->face_relations == nullptr || L->aminus == nullptr)) {
    setError(std::string(who) + ": neighbour data missing");
    return false;
  }
  return true;
}

// Kernels of the two passes.  A variant is a number of the public interface:
// the kTileVariants VALU tile shapes (FP32 ones for the matrix-core forms), for
// the neighbour pass the one-element-per-row kernel after them
// (kNeighborRowsVariant), and for the local pass of the matrix-core forms and
// the FP64 engine (orders 3-7, kernel family AUTO) the matrix-core pass before
// them (variant 0).  The FP32 engine's local pass and every engine's neighbour
// pass at orders 3-7 have their matrix-core pass beside the numbers
// (Tile::matrixCore); it is faster than any VALU variant in all but the
// smallest clusters and is what runs untuned.
bool numberedLocal(const EngineState& e) { return matrixCore(e.arithmetic) || (e.arithmetic == SDG_FP64 && hasMx(e)); }
int localVariants(const EngineState& e) { return numberedLocal(e) ? 1 + kTileVariants : kTileVariants; }

// Default VALU variant of the neighbour pass: one element per 16-lane row for
// the FP32 kernel at orders 3-6 and the FP64 kernel at orders 4-5 (where the
// autotuner picked it on every cluster), else tile 0.
int defaultNeighborVariant(const EngineState& e) {
  const bool fp64 = e.arithmetic == SDG_FP64;
  const bool rows = fp64 ? (e.order >= 4 && e.order <= 5) : (e.order >= 3 && e.order <= 6);
  return rows ? kNeighborRowsVariant : 0;
}

struct Tile {
  int variant = 0;
  bool matrixCore = false;  // beside the variants: the matrix-core pass, where the engine has it
};
Tile defaultTile(const EngineState& e, int kernel) {
  if (kernel == 0) return {0, !numberedLocal(e)};
  return {defaultNeighborVariant(e), true};
}
bool runsMx(const EngineState& e, int kernel, const Tile& t) {
  if (kernel == 1) return t.matrixCore && hasNeighborMx(e);
  return numberedLocal(e) ? t.variant == 0 : t.matrixCore && hasMx(e);
}

int runLocal(const EngineState& e, const double* coeffs, const sdg_layer* own, int reset, hipStream_t s,
             const Tile& t) {
  if (!runsMx(e, 0, t)) return launchLocalIntegration(e, coeffs, own, reset, s, t.variant - (numberedLocal(e) ? 1 : 0));
  return matrixCore(e.arithmetic) ? launchLocalIntegrationMfma(e, coeffs, own, reset, s)
                                  : launchLocalIntegrationMx(e, coeffs, own, reset, s);
}

int runNeighbor(const EngineState& e, const double* coeffs, const double* sub, const sdg_layer* nbv, hipStream_t s,
                const Tile& t) {
  return runsMx(e, 1, t) ? launchNeighborMx(e, nbv, coeffs, sub, s)
                         : launchNeighboringIntegration(e, coeffs, sub, nbv, s, t.variant);
}

bool ltsArithmetic(const sdg_engine* e, const char* who) {
  if (matrixCore(e->s.arithmetic) && (e->s.order < 3 || e->s.order > 7)) {
    setError(std::string(who) + ": the matrix-core forms run orders 3..7");
    return false;
  }
  return true;
}

}  // namespace

extern "C" int sdg_derive_lts_setups(int64_t n, const int32_t* cluster_ids, const int32_t* neighbors,
                                     const uint8_t* face_types, uint16_t* setups) {
  if (n < 0 || (n > 0 && (cluster_ids == nullptr || neighbors == nullptr || setups == nullptr))) {
    setError("sdg_derive_lts_setups: invalid arguments");
    return SDG_ERR_INVALID;
  }
  for (int64_t e = 0; e < n * 4; ++e)
    if (neighbors[e] < 0 || neighbors[e] >= n) {
      setError("sdg_derive_lts_setups: neighbour index out of range");
      return SDG_ERR_INVALID;
    }
  // getLtsSetup (LtsSetup.cpp:97-182)
  for (int64_t e = 0; e < n; ++e) {
    uint16_t s = 0;
    const int own = cluster_ids[e];
    for (int f = 0; f < 4; ++f) {
      const uint8_t type = face_types != nullptr ? face_types[e * 4 + f] : SDG_FACE_REGULAR;
      if (type == SDG_FACE_DYNAMIC_RUPTURE) {
        s |= (kNHD0 << f) | (kGTS0 << f) | kDerivatives;
        continue;
      }
      const int nc = cluster_ids[neighbors[e * 4 + f]];
      if (nc > own + 1 || own > nc + 1) {
        // the neighbour integral takes the sub-interval of the next cluster only
        setError("sdg_derive_lts_setups: face neighbours must be at most one cluster apart");
        return SDG_ERR_INVALID;
      }
      if (own < nc) s |= (kNHD0 << f) | kAccumulate;
      else if (own == nc) s |= (kGTS0 << f);
      s |= own > nc ? kDerivatives : kBuffers;
    }
    if ((s & kAccumulate) && (s & (0xfu << 4))) s |= kDerivatives;
    setups[e] = s;
  }
  // normalizeLtsSetup (LtsSetup.cpp:205-217): a same-cluster neighbour whose
  // buffer accumulates over several steps provides derivatives instead
  std::vector<uint16_t> first(setups, setups + n);
  for (int64_t e = 0; e < n; ++e)
    for (int f = 0; f < 4; ++f)
      if ((first[e] & (kGTS0 << f)) && (first[neighbors[e * 4 + f]] & kAccumulate)) setups[e] |= (kNHD0 << f);
  return SDG_OK;
}

extern "C" int sdg_compute_local_integration(sdg_engine* engine, const double* coeffs, double /*time_step_width*/,
                                             const sdg_layer* layer, int reset_buffers, void* stream) {
  if (engine == nullptr || coeffs == nullptr) {
    setError("sdg_compute_local_integration: NULL argument");
    return SDG_ERR_INVALID;
  }
  if (!ltsArithmetic(engine, "sdg_compute_local_integration") ||
      !ltsLayerOk(layer, false, "sdg_compute_local_integration") ||
      !layerStridesOk(engine->s, layer, "sdg_compute_local_integration"))
    return SDG_ERR_INVALID;
  return runLocal(engine->s, coeffs, layer, reset_buffers != 0, static_cast<hipStream_t>(stream),
                  defaultTile(engine->s, 0));
}

extern "C" int sdg_compute_neighboring_integration(sdg_engine* engine, const double* time_coeffs,
                                                   const double* subtime_coeffs, const sdg_layer* layer,
                                                   void* stream) {
  if (engine == nullptr || time_coeffs == nullptr || subtime_coeffs == nullptr) {
    setError("sdg_compute_neighboring_integration: NULL argument");
    return SDG_ERR_INVALID;
  }
  if (!ltsArithmetic(engine, "sdg_compute_neighboring_integration") ||
      !ltsLayerOk(layer, true, "sdg_compute_neighboring_integration") ||
      !layerStridesOk(engine->s, layer, "sdg_compute_neighboring_integration"))
    return SDG_ERR_INVALID;
  Tile tile = defaultTile(engine->s, 1);
  tile.matrixCore = prefersNeighborMx(engine->s, layer->num_elements, true);
  return runNeighbor(engine->s, time_coeffs, subtime_coeffs, layer, static_cast<hipStream_t>(stream), tile);
}

struct sdg_lts {
  sdg_engine* engine = nullptr;
  sdg_layer layer{};
  std::vector<int64_t> start;
  double dt0 = 0.0;
  std::vector<Tile> tile[2];  // per kernel (local, neighbour) and cluster
  hipStream_t captureStream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace {

// view of cluster c: own arrays offset to the cluster, neighbour sources global
sdg_layer clusterView(const sdg_lts& L, int c, bool neighborPass) {
  const int64_t rs = L.engine->s.arithmetic == SDG_FP64 ? 8 : 4;
  const CellLayout lay = cellLayout(L.engine->s, &L.layer);
  const int64_t q = lay.qStride;
  const int64_t off = L.start[c];
  const sdg_layer& g = L.layer;
  sdg_layer v = g;
  auto shift = [&](const void* p, int64_t bytes) -> char* {
    return p == nullptr ? nullptr : const_cast<char*>(static_cast<const char*>(p)) + off * bytes;
  };
  v.num_elements = L.start[c + 1] - L.start[c];
  v.dofs = shift(g.dofs, q * rs);
  v.star = shift(g.star, lay.starStride * rs);
  v.aplus = shift(g.aplus, lay.aplusStride * rs);
  v.aminus = shift(g.aminus, lay.aminusStride * rs);
  v.face_neighbors = reinterpret_cast<const int32_t*>(shift(g.face_neighbors, 16));
  v.face_relations = reinterpret_cast<const uint8_t*>(shift(g.face_relations, 8));
  v.face_types = reinterpret_cast<const uint8_t*>(shift(g.face_types, 4));
  v.lts_setup = reinterpret_cast<const uint16_t*>(shift(g.lts_setup, 2));
  v.face_traces = nullptr;
  if (!neighborPass) {
    v.time_integrated = shift(g.time_integrated, q * rs);
    v.derivatives = shift(g.derivatives, lay.dsize * rs);
  }
  return v;
}

// whether the matrix-core local pass takes several clusters in one launch (the neighbour pass does)
bool mergedLocal(const EngineState& e) { return hasMx(e) && !mfma::splitProducts(e); }

// The passes of clusters 0 .. top that start (local) or end (neighbour) a step
// at the same time.  They are independent: a local pass touches its own cells
// only, a neighbour pass reads buffers and derivatives and writes its own DOFs.
// So the clusters on the matrix-core pass share a launch: a small cluster
// takes 20 us for one tile's chain whatever its size (four clusters of 9k cells
// in FP64 at ORDER 4, a macro step of 30 launches -> 16: 801 -> 614 us).
int localPasses(const sdg_lts& L, int top, int64_t k, hipStream_t s) {
  const EngineState& e = L.engine->s;
  double coeffs[mx::kMaxClusters][kMaxOrder];
  mx::ClusterStep steps[mx::kMaxClusters];
  int merged = 0;
  for (int c = top; c >= 0; --c) {
    const sdg_layer own = clusterView(L, c, false);
    if (own.num_elements == 0) continue;
    const int reset = ((k >> c) & 1) == 0;
    sdg_monomial_integrate(e.order, 0.0, L.dt0 * static_cast<double>(int64_t(1) << c), coeffs[c]);
    if (mergedLocal(e) && runsMx(e, 0, L.tile[0][c])) {
      steps[merged++] = {L.start[c], L.start[c + 1], coeffs[c], nullptr, reset};
    } else if (const int rc = runLocal(e, coeffs[c], &own, reset, s, L.tile[0][c]); rc != SDG_OK) {
      return rc;
    }
  }
  return merged > 0 ? launchLocalClustersMx(e, steps, merged, &L.layer, s) : SDG_OK;
}

int neighborPasses(const sdg_lts& L, int top, int64_t k, hipStream_t s) {
  const EngineState& e = L.engine->s;
  const int C = static_cast<int>(L.start.size()) - 1;
  double coeffs[mx::kMaxClusters][kMaxOrder], sub[mx::kMaxClusters][kMaxOrder];
  mx::ClusterStep steps[mx::kMaxClusters];
  int merged = 0;
  for (int c = 0; c <= top; ++c) {
    const sdg_layer nbv = clusterView(L, c, true);
    if (nbv.num_elements == 0) continue;
    const double dtc = L.dt0 * static_cast<double>(int64_t(1) << c);
    const int64_t begin = k + 1 - (int64_t(1) << c);  // of the cluster's step, in steps of the fastest
    sdg_monomial_integrate(e.order, 0.0, dtc, coeffs[c]);
    // sub-interval of the slower cluster's step
    const double t = c + 1 < C ? L.dt0 * static_cast<double>(begin - ((begin >> (c + 1)) << (c + 1))) : 0.0;
    sdg_monomial_integrate(e.order, t, t + dtc, sub[c]);
    if (runsMx(e, 1, L.tile[1][c])) {
      steps[merged++] = {L.start[c], L.start[c + 1], coeffs[c], sub[c], 1};
    } else if (const int rc = runNeighbor(e, coeffs[c], sub[c], &nbv, s, L.tile[1][c]); rc != SDG_OK) {
      return rc;
    }
  }
  return merged > 0 ? launchNeighborClustersMx(e, steps, merged, &L.layer, s) : SDG_OK;
}

// the clusters' steps in order of time, in units of the fastest's
int macroStep(const sdg_lts& L, hipStream_t s) {
  const int C = static_cast<int>(L.start.size()) - 1;
  auto slowest = [&](int64_t k) {  // of the clusters whose steps divide k
    int c = 0;
    while (c + 1 < C && (k & ((int64_t(2) << c) - 1)) == 0) ++c;
    return c;
  };
  for (int64_t k = 0; k < int64_t(1) << (C - 1); ++k) {
    int rc = localPasses(L, slowest(k), k, s);
    if (rc == SDG_OK) rc = neighborPasses(L, slowest(k + 1), k, s);
    if (rc != SDG_OK) return rc;
  }
  return SDG_OK;
}

}  // namespace

extern "C" int sdg_lts_create(sdg_lts** out, sdg_engine* engine, const sdg_layer* layer, int num_clusters,
                              const int64_t* cluster_start, double dt0) {
  if (out == nullptr || engine == nullptr || cluster_start == nullptr || num_clusters < 1 || num_clusters > 16 ||
      !(dt0 > 0.0)) {
    setError("sdg_lts_create: invalid arguments (1..16 clusters, dt0 > 0)");
    return SDG_ERR_INVALID;
  }
  if (!ltsArithmetic(engine, "sdg_lts_create") || !ltsLayerOk(layer, true, "sdg_lts_create") ||
      !layerStridesOk(engine->s, layer, "sdg_lts_create"))
    return SDG_ERR_INVALID;
  if (cluster_start[0] != 0 || cluster_start[num_clusters] != layer->num_elements) {
    setError("sdg_lts_create: cluster_start must run from 0 to num_elements");
    return SDG_ERR_INVALID;
  }
  for (int c = 0; c < num_clusters; ++c)
    if (cluster_start[c + 1] < cluster_start[c]) {
      setError("sdg_lts_create: cluster_start must not decrease");
      return SDG_ERR_INVALID;
    }
  auto* L = new sdg_lts;
  L->engine = engine;
  L->layer = *layer;
  L->start.assign(cluster_start, cluster_start + num_clusters + 1);
  L->dt0 = dt0;
  for (int k = 0; k < 2; ++k) L->tile[k].assign(num_clusters, defaultTile(engine->s, k));
  *out = L;
  return SDG_OK;
}

namespace {
bool tileArguments(const sdg_lts* lts, int cluster, int kernel, const char* who) {
  if (lts != nullptr && cluster >= 0 && cluster < static_cast<int>(lts->tile[0].size()) && (kernel == 0 || kernel == 1))
    return true;
  setError(std::string(who) + ": invalid arguments");
  return false;
}
// a captured macro step used the previous tiles
void dropGraph(sdg_lts* lts) {
  if (lts->exec != nullptr) (void)hipGraphExecDestroy(lts->exec);
  if (lts->graph != nullptr) (void)hipGraphDestroy(lts->graph);
  lts->exec = nullptr;
  lts->graph = nullptr;
}
}  // namespace

// Tile autotuner: times every tile variant of both kernels on every cluster
// (`repeats` launches each, HIP events on `stream`) and keeps the fastest;
// the cells' state is saved before and restored afterwards.  A variant that
// is faster alone than a matrix-core pass takes its cluster out of the launch
// that the clusters of that pass share, so it has to make the whole macro step
// faster as well (2,560 cells in FP64 at ORDER 3: variants picked alone 357 ->
// 440 us a step; small clusters are where they win).
extern "C" int sdg_lts_autotune(sdg_lts* lts, int repeats, void* stream) {
  if (lts == nullptr || repeats < 1) {
    setError("sdg_lts_autotune: invalid arguments");
    return SDG_ERR_INVALID;
  }
  const auto st = static_cast<hipStream_t>(stream);
  const EngineState& e = lts->engine->s;
  const int order = e.order;
  const int64_t n = lts->layer.num_elements;
  const int64_t rs = e.arithmetic == SDG_FP64 ? 8 : 4;
  const CellLayout lay = cellLayout(e, &lts->layer);
  const int64_t qBytes = n * lay.qStride * rs;
  const int64_t dBytes = n * lay.dsize * rs;
  void* saved[3] = {nullptr, nullptr, nullptr};
  void* live[3] = {lts->layer.dofs, lts->layer.time_integrated, lts->layer.derivatives};
  const int64_t bytes[3] = {qBytes, qBytes, dBytes};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = SDG_OK;
  // every failure from here on goes through the one cleanup path below: the
  // state is restored if it was saved, and what was allocated is released
  for (int i = 0; i < 3 && rc == SDG_OK; ++i) {
    hipError_t err = hipMalloc(&saved[i], bytes[i]);
    if (err != hipSuccess) saved[i] = nullptr;
    if (err == hipSuccess) err = hipMemcpyAsync(saved[i], live[i], bytes[i], hipMemcpyDeviceToDevice, st);
    if (err != hipSuccess) rc = hipFail(err, "sdg_lts_autotune: saving the state");
  }
  if (rc == SDG_OK) {
    hipError_t err = hipEventCreate(&e0);
    if (err == hipSuccess) err = hipEventCreate(&e1);
    if (err != hipSuccess) rc = hipFail(err, "sdg_lts_autotune: events");
  }
  const bool stateSaved = rc == SDG_OK;
  // milliseconds of `repeats` calls of `run`, which returns a status, after an
  // untimed one (the first launch of a kernel loads it)
  auto timed = [&](auto&& run) {
    float ms = 0.0f;
    if (rc == SDG_OK) rc = run();
    (void)hipEventRecord(e0, st);
    for (int r = 0; r < repeats && rc == SDG_OK; ++r) rc = run();
    (void)hipEventRecord(e1, st);
    if (rc != SDG_OK) return ms;
    const hipError_t err = hipEventSynchronize(e1);
    if (err != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
      rc = hipFail(err != hipSuccess ? err : hipErrorUnknown, "sdg_lts_autotune timing");
    return ms;
  };
  const int C = static_cast<int>(lts->start.size()) - 1;
  if (rc == SDG_OK)
    for (int kind = 0; kind < 2; ++kind) lts->tile[kind].assign(C, defaultTile(e, kind));
  for (int c = 0; c < C && rc == SDG_OK; ++c) {
    const double dtc = lts->dt0 * static_cast<double>(int64_t(1) << c);
    std::vector<double> coeffs(order);
    sdg_monomial_integrate(order, 0.0, dtc, coeffs.data());
    const sdg_layer own = clusterView(*lts, c, false), nbv = clusterView(*lts, c, true);
    if (own.num_elements == 0) continue;
    for (int kind = 0; kind < 2 && rc == SDG_OK; ++kind) {
      auto alone = [&](const Tile& t) {
        return timed([&] {
          return kind == 0 ? runLocal(e, coeffs.data(), &own, 1, st, t)
                           : runNeighbor(e, coeffs.data(), coeffs.data(), &nbv, st, t);
        });
      };
      const Tile first = defaultTile(e, kind);
      const bool shared = runsMx(e, kind, first) && (kind == 1 || mergedLocal(e));
      Tile best = first;
      float bestMs = alone(first);
      for (int v = 0; v < (kind == 0 ? localVariants(e) : kNeighborVariants) && rc == SDG_OK; ++v) {
        const Tile t{v, false};
        if (v == first.variant && !first.matrixCore) continue;
        const float ms = alone(t);
        if (ms < bestMs) {
          bestMs = ms;
          best = t;
        }
      }
      if (rc != SDG_OK) break;
      Tile& tile = lts->tile[kind][c];
      if (shared && !runsMx(e, kind, best)) {
        auto step = [&] { return macroStep(*lts, st); };
        const float together = timed(step);
        tile = best;
        // one per cent: what two timings of the same step differ by
        if (!(timed(step) < 0.99f * together)) tile = first;
      } else {
        tile = best;
      }
    }
  }
  // restore whenever the state was saved, also after a failed tuning launch
  // (the first error is the one reported)
  if (stateSaved)
    for (int i = 0; i < 3; ++i) {
      const hipError_t err = hipMemcpyAsync(live[i], saved[i], bytes[i], hipMemcpyDeviceToDevice, st);
      if (err != hipSuccess && rc == SDG_OK) rc = hipFail(err, "sdg_lts_autotune restore");
    }
  (void)hipStreamSynchronize(st);
  for (int i = 0; i < 3; ++i)
    if (saved[i] != nullptr) (void)hipFree(saved[i]);
  if (e0 != nullptr) (void)hipEventDestroy(e0);
  if (e1 != nullptr) (void)hipEventDestroy(e1);
  dropGraph(lts);
  return rc;
}

extern "C" int sdg_lts_set_tile_variant(sdg_lts* lts, int cluster, int kernel, int variant) {
  if (!tileArguments(lts, cluster, kernel, "sdg_lts_set_tile_variant")) return SDG_ERR_INVALID;
  if (variant < 0 || variant >= (kernel == 0 ? localVariants(lts->engine->s) : kNeighborVariants)) {
    setError("sdg_lts_set_tile_variant: invalid arguments");
    return SDG_ERR_INVALID;
  }
  lts->tile[kernel][cluster] = {variant, false};
  dropGraph(lts);
  return SDG_OK;
}

extern "C" int sdg_lts_tile_variant(const sdg_lts* lts, int cluster, int kernel) {
  if (!tileArguments(lts, cluster, kernel, "sdg_lts_tile_variant")) return SDG_ERR_INVALID;
  return lts->tile[kernel][cluster].variant;
}

extern "C" int sdg_lts_matrix_core(const sdg_lts* lts, int cluster, int kernel) {
  if (!tileArguments(lts, cluster, kernel, "sdg_lts_matrix_core")) return SDG_ERR_INVALID;
  return runsMx(lts->engine->s, kernel, lts->tile[kernel][cluster]) ? 1 : 0;
}

extern "C" int sdg_lts_use_matrix_core(sdg_lts* lts, int cluster, int kernel) {
  if (!tileArguments(lts, cluster, kernel, "sdg_lts_use_matrix_core")) return SDG_ERR_INVALID;
  const Tile tile = defaultTile(lts->engine->s, kernel);
  if (!runsMx(lts->engine->s, kernel, tile)) {
    setError("sdg_lts_use_matrix_core: the engine has no matrix-core pass for this kernel");
    return SDG_ERR_UNSUPPORTED;
  }
  lts->tile[kernel][cluster] = tile;
  dropGraph(lts);
  return SDG_OK;
}

extern "C" int sdg_lts_advance(sdg_lts* lts, int macro_steps, void* stream) {
  if (lts == nullptr || macro_steps < 0) {
    setError("sdg_lts_advance: invalid arguments");
    return SDG_ERR_INVALID;
  }
  for (int m = 0; m < macro_steps; ++m) {
    const int rc = macroStep(*lts, static_cast<hipStream_t>(stream));
    if (rc != SDG_OK) return rc;
  }
  return SDG_OK;
}

extern "C" int sdg_lts_graph_advance(sdg_lts* lts, int macro_steps, void* stream) {
  if (lts == nullptr || macro_steps < 0) {
    setError("sdg_lts_graph_advance: invalid arguments");
    return SDG_ERR_INVALID;
  }
  if (lts->exec == nullptr) {
    // capture one macro step on a private stream (default priority)
    if (lts->captureStream == nullptr) SDG_HIP_CHECK(hipStreamCreateWithFlags(&lts->captureStream, hipStreamNonBlocking));
    SDG_HIP_CHECK(hipStreamBeginCapture(lts->captureStream, hipStreamCaptureModeThreadLocal));
    const int rc = macroStep(*lts, lts->captureStream);
    hipGraph_t g = nullptr;
    const hipError_t end = hipStreamEndCapture(lts->captureStream, &g);
    if (rc != SDG_OK) {
      if (g != nullptr) (void)hipGraphDestroy(g);
      return rc;
    }
    SDG_HIP_CHECK(end);
    lts->graph = g;
    SDG_HIP_CHECK(hipGraphInstantiate(&lts->exec, lts->graph, nullptr, nullptr, 0));
  }
  for (int m = 0; m < macro_steps; ++m) SDG_HIP_CHECK(hipGraphLaunch(lts->exec, static_cast<hipStream_t>(stream)));
  return SDG_OK;
}

extern "C" int sdg_lts_destroy(sdg_lts* lts) {
  if (lts == nullptr) return SDG_OK;
  if (lts->exec != nullptr) (void)hipGraphExecDestroy(lts->exec);
  if (lts->graph != nullptr) (void)hipGraphDestroy(lts->graph);
  if (lts->captureStream != nullptr) (void)hipStreamDestroy(lts->captureStream);
  delete lts;
  return SDG_OK;
}
