// Rate-and-state fast-velocity-weakening friction (law 103) on the GPU, FP64.
//
// One lane per (face, Gauss point); the lanes of a face form a contiguous
// power-of-two group inside a wave so the face-wide convergence decisions of
// the CPU implementation (CpuImpl/RateAndState.h:209-222, 375-386) are wave
// ballots restricted to the face's lanes.  Per time point: stresses from the
// interpolated DOFs, nucleation, fixed-point state update around a Newton
// solve for the slip rate, slip/traction update and outputs; afterwards the
// state resampling and the imposed states (FrictionSolverCommon.h:146-631,
// FastVelocityWeakeningLaw.h:43-165, RateAndStateCommon.h:22-139).
//
// Optional warm start of the first slip-rate solve of each time point, before
// its first residual test: a point whose closed-form creep root V_c (the root
// of g(V) + V = 0, so g(V_c) = -V_c) lies below half the tolerance starts at
// V_c and passes that test at once; with a 6-32-32-1 MLP (FP32) every other
// point starts at the network's predicted root when it lies more than a decade
// from the previous slip rate.  No evaluation is added and the residual test
// is unchanged; g is strictly decreasing in V, so a converged solve returns
// the plain solver's root up to the tolerance.
//
// Bound by the FP64 instructions of the Newton steps and state updates at one
// or two waves per SIMD.  So the kernel is lean in both: one pass over the time
// points without per-point arrays, 32-bit offsets, the network's code in an
// instantiation of its own (with it 390 registers, one wave per SIMD), one
// exponential per state instead of two per step, one square root and one
// division per step, the eighth root as three square roots.  20k faces of 25
// points, ORDER 4: 1376 -> 638 us, with the closed-form start 1246 -> 552; 5k
// faces of 49 points, ORDER 6: 952 -> 480; 1k faces of 16 points: 125 -> 107.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "engine.h"
#include "friction_common.h"

namespace sdg {
namespace friction {
namespace {

constexpr double kAlmostZero = 1e-45;
constexpr int kMaxOrder = 8;
constexpr double kMovedDecades = 0.30103;  // log10(2)
constexpr double kJumpDecades = 1.0;
constexpr double kLn10 = 2.30258509299404568402;

// The network's forward pass, kept out of line: inlined into kFriction, its
// unrolled products and LDS weight loads pushed the kernel past its registers
// (916 B of spills per lane); as a call it costs the warm-start branch only.
__device__ __noinline__ float mlpEvaluateCall(const float* prm, const float (&x)[kMlpInputs]) {
  return mlpEvaluate(prm, x);
}

// natural log of the closed-form creep root V_c = 2 V0 exp(-psi/a) sinh(S/N),
// which solves N asinh(V exp(psi/a) / (2 V0)) = S; -inf when S or N is not positive
__device__ __noinline__ double creepLogRoot(double S, double N, double psiOverA, double sr0) {
  if (!(S > 0.0) || !(N > 0.0)) return -INFINITY;
  const double c = S / N;
  return log(2.0 * sr0) - psiOverA + c + log(-0.5 * expm1(-2.0 * c));
}

// mu(V) = a asinh(x e^c), x = V / (2 V0), c = psi / a, of one state psi: what
// depends on the state alone is formed once and kept over the Newton steps.
// e^c overflows where c is large: there asinh(x e^c) = c + log(x + sqrt(x^2 + e^-2c)).
struct MuCurve {
  double a, half, c, grow, decay;  // half = 1 / (2 V0), grow = e^c, decay = e^-c
  __device__ inline MuCurve(double a_, double sr0, double psi) : a(a_), half(0.5 / sr0), c(psi / a_) {
    const double small = c > 0 ? exp(-c) : exp(c);
    const double large = 1.0 / small;
    grow = c > 0 ? large : small;
    decay = c > 0 ? small : large;
  }
  // mu(V), and its derivative as a half num / root
  __device__ inline double eval(double V, double& num, double& root) const {
    const double sw = 10.0, threshold = 50.0, log2 = 0.69314718055994530943;
    const double x = half * V;
    int xexp = 0;
    (void)frexp(x, &xexp);
    if (c + (xexp > 0 ? xexp : 0) * log2 > sw || c >= threshold) {
      const double xa = fabs(x);
      const double xs = x >= 0 ? 1.0 : -1.0;
      root = sqrt(x * x + decay * decay);
      num = 1.0;
      return a * (xs * (c + log(xa + root)));
    }
    const double v = grow * x;
    root = sqrt(1.0 + v * v);
    num = grow;
    return a * asinh(v);
  }
};

__device__ inline double logsinh(double x, double c) {
  const double sign = c >= 0 ? 1.0 : -1.0;
  const double ac = fabs(c);
  return ac + log(x / 2 * -sign * expm1(-2 * ac));
}

__device__ inline double smoothStep(double t, double t0) {
  if (t <= 0) return 0.0;
  if (t < t0) {
    const double tau = t - t0;
    return exp(tau * tau / (t * (t - 2.0 * t0)));
  }
  return 1.0;
}

__device__ __noinline__ double features(double logVc, double S, double N, double psiOverA, double vPrev, double a,
                                        float (&x)[kMlpInputs]) {
  return mlpFeatures(logVc, S, N, psiOverA, vPrev, a, x);
}

struct PointParams {
  double a, sl0, f0, muw, b, srw;
};

__device__ inline double updateStateVariable(const PointParams& pp, double sr0, double svRef, double dt, double V) {
  const double lowV = fmax(0.0, pp.f0 - (pp.b - pp.a) * log(V / sr0));
  const double r = V / pp.srw;
  const double r2 = r * r, r4 = r2 * r2, r8 = r4 * r4;
  const double muSS = pp.muw + (lowV - pp.muw) / sqrt(sqrt(sqrt(1.0 + r8)));
  const double psiSS = pp.a * logsinh(sr0 / V * 2, muSS / pp.a);
  const double pre = -V * (dt / pp.sl0);
  // 1 + rise is e^pre to an ulp of 1, not of itself: the term is off by up to
  // 1e-16 |svRef|, as the stored state is (it changes by the difference from
  // svRef) and as the friction sees it (through e^(state / a))
  const double rise = expm1(pre);
  return psiSS * (-rise) + (1.0 + rise) * svRef;
}

// true if pred holds on every real point of this lane's face
template <int TPF>
__device__ inline bool faceAll(bool pred, int numPoints) {
  const unsigned long long b = __ballot(pred);
  const int lane = threadIdx.x & 63;
  const int seg = (lane / TPF) * TPF;
  const unsigned long long full = numPoints >= 64 ? ~0ULL : ((1ULL << numPoints) - 1ULL);
  return ((b >> seg) & full) == full;
}

// element i of an array with a uniform base; I: unsigned where i * sizeof(T) stays below 2^32
template <typename T, typename I>
__device__ inline T& lane(T* base, I i) {
  typedef std::conditional_t<std::is_const_v<T>, const char, char> Byte;
  return *reinterpret_cast<T*>(reinterpret_cast<Byte*>(base) + i * static_cast<I>(sizeof(T)));
}

// how the first solve of a time point starts: from the previous slip rate, at
// the closed-form creep root where it applies, or by the network (which also
// covers the recording of its samples)
enum Start { kPlain, kClosedForm, kNetwork };

// threads per block: one wave, so that small faults reach every CU and a face's
// long solve holds up nothing but its wave (20k faces of 25 points: 726 us with
// 256 threads, 628 with 64); with the network the block shares its parameters
template <Start S>
constexpr int kBlock = S == kNetwork ? 256 : 64;

struct StepArgs {
  double deltaT[kMaxOrder];
  double timeWeights[kMaxOrder];
};

template <int TPF, Start S, typename I>
__global__ __launch_bounds__((kBlock<S>), 2) void kFriction(sdg_friction_params prm, sdg_fault_layer L, double fullUpdateTime,
                                                 StepArgs args, const double* __restrict__ resample,
                                                 sdg_friction_options opt) {
  constexpr int FPB = kBlock<S> / TPF;
  __shared__ double sDelta[kBlock<S>];
  __shared__ float sMlp[S == kNetwork ? kMlpParams : 1];
  const bool useMlp = S == kNetwork && opt.mlp_params != nullptr;
  if (useMlp)
    for (int i = threadIdx.x; i < kMlpParams; i += blockDim.x) sMlp[i] = opt.mlp_params[i];
  __syncthreads();

  const int pnt = threadIdx.x % TPF;
  const int64_t face = static_cast<int64_t>(blockIdx.x) * FPB + threadIdx.x / TPF;
  const int NP = L.num_points, P = L.points, O = L.order;
  const bool active = face < L.num_faces && pnt < NP;
  // per-point arrays as a uniform base (the block's first face) and a 32-bit
  // byte offset per lane: 64-bit addresses of the 30 arrays, live from their
  // loads to their stores, would take a register pair each
  const int64_t f0 = static_cast<int64_t>(blockIdx.x) * FPB;
  const I fl = active ? threadIdx.x / TPF : 0u;
  const int p = active ? pnt : 0;
  const I k = fl * P + p;
  auto at = [&](auto* array) -> decltype(*array)& { return lane(array + f0 * P, k); };
  auto stress = [&](auto* array, int c) -> decltype(*array)& { return lane(array + f0 * 6 * P, (fl * 6 + c) * P + p); };

  const double* ie = L.imp_and_eta + (f0 + fl) * 11;
  const double etaS = ie[5], invEtaS = ie[6], invZp = ie[7], invZs = ie[8], invZpN = ie[9], invZsN = ie[10];
  const double etaP = ie[4] * (prm.eta_damp_end > fullUpdateTime ? prm.eta_damp : 1.0);
  const PointParams pp{at(L.rs_a), at(L.rs_sl0), at(L.rs_f0), at(L.rs_muw), at(L.rs_b), at(L.rs_srw)};
  auto qp = [&](int o, int q) { return lane(L.q_interpolated_plus + f0 * O * 9 * P, ((fl * O + o) * 9 + q) * P + p); };
  auto qm = [&](int o, int q) { return lane(L.q_interpolated_minus + f0 * O * 9 * P, ((fl * O + o) * 9 + q) * P + p); };

  double trT1 = 0.0, trT2 = 0.0;  // tractions of the last time point
  // imposed states, summed over the time points (quantities 0, 3, 5 are the same on both sides)
  double sumN = 0.0, sumT1 = 0.0, sumT2 = 0.0, minusV[3] = {0.0, 0.0, 0.0}, plusV[3] = {0.0, 0.0, 0.0};
  double sv = at(L.state_variable);
  double slipRate1 = at(L.slip_rate1), slipRate2 = at(L.slip_rate2);
  double srm = at(L.slip_rate_magnitude);
  double muv = at(L.mu);
  uint8_t convInner = at(L.convergence_inner), convOuter = at(L.convergence_outer);
  // the per-point outputs accumulated over the time points, read once here and
  // written once after the time loop (a read-modify-write per time point
  // waited on each load in turn)
  double accSlip = at(L.accumulated_slip), slip1 = at(L.slip1), slip2 = at(L.slip2);
  double peakSr = at(L.peak_slip_rate), ruptureTime = at(L.rupture_time), dynStressTime = at(L.dyn_stress_time);
  uint8_t rupturePending = at(L.rupture_time_pending), dynStressPending = at(L.dyn_stress_time_pending);
  int newtonEvals = 0, newtonSteps = 0;
  const bool closedForm = S != kPlain && opt.closed_form_start != 0;
  const bool record = S == kNetwork && opt.samples != nullptr;

  double updateTime = fullUpdateTime;
  for (int o = 0; o < O; ++o) {
    const double dt = args.deltaT[o];
    const double startTime = updateTime;
    const double m0 = qm(o, 0), m3 = qm(o, 3), m5 = qm(o, 5), m6 = qm(o, 6), m7 = qm(o, 7), m8 = qm(o, 8);
    const double p0 = qp(o, 0), p3 = qp(o, 3), p5 = qp(o, 5), p6 = qp(o, 6), p7 = qp(o, 7), p8 = qp(o, 8);
    const double fsN = etaP * (m6 - p6 + p0 * invZp + m0 * invZpN);
    const double fsT1 = etaS * (m7 - p7 + p3 * invZs + m3 * invZsN);
    const double fsT2 = etaS * (m8 - p8 + p5 * invZs + m5 * invZsN);
    updateTime += dt;
    if (prm.nucleation_count > 0 && L.nucleation_stress != nullptr && updateTime <= prm.t0 + prm.s0 &&
        updateTime >= prm.s0) {
      const double gNuc = smoothStep(updateTime - prm.s0, prm.t0) - smoothStep(updateTime - prm.s0 - dt, prm.t0);
      if (active) {
        for (int c = 0; c < 6; ++c) stress(L.initial_stress, c) += stress(L.nucleation_stress, c) * gNuc;
        if (L.nucleation_pressure != nullptr) at(L.initial_pressure) += at(L.nucleation_pressure) * gNuc;
      }
    }
    const double pressure = at(L.initial_pressure);
    const double s3 = stress(L.initial_stress, 3), s5 = stress(L.initial_stress, 5);
    const double normal = fmin(0.0, fsN + stress(L.initial_stress, 0) + pressure);
    const double svRef = sv;
    const double absShear = sqrt((s3 + fsT1) * (s3 + fsT1) + (s5 + fsT2) * (s5 + fsT2));
    srm = fmax(kAlmostZero, sqrt(slipRate1 * slipRate1 + slipRate2 * slipRate2));
    const double vPrev = srm;
    const double upper = fmax(kAlmostZero, invEtaS * absShear);  // g(upper) <= 0: the root lies below
    const double nScale = invEtaS * fabs(normal) * pp.a;
    double localSR = srm;
    bool convOuterPre = true;
    for (int j = 0; j < prm.rs_state_variable_updates; ++j) {
      sv = active ? updateStateVariable(pp, prm.rs_sr0, svRef, dt, localSR) : 0.0;
      double test = srm;
      // warm start of the first solve; lvc, base, feat also feed the sample recording
      double lvc = -INFINITY, base = 0.0;
      float feat[kMlpInputs];
      if (j == 0 && active && (closedForm || useMlp || record)) {
        lvc = creepLogRoot(invEtaS * absShear, nScale, sv / pp.a, prm.rs_sr0);
        const bool creeping = lvc < log(0.5 * prm.rs_slip_rate_tolerance);
        if (closedForm && creeping) {
          test = fmax(kAlmostZero, exp(lvc));
        } else if (useMlp && !creeping) {
          base = features(lvc, upper, nScale, sv / pp.a, vPrev, pp.a, feat);
          // the root lies in (0, min(V_c, S)]
          const double lg = fmin(base + static_cast<double>(mlpEvaluateCall(sMlp, feat)), fmin(lvc / kLn10, log10(upper)));
          if (isfinite(lg) && fabs(lg - log10(vPrev)) > kJumpDecades) test = fmax(kAlmostZero, pow(10.0, lg));
        }
      }
      double g = 0.0, muF = muv, num = 1.0, root = 1.0;
      const MuCurve curve(pp.a, prm.rs_sr0, sv);
      const double slope = invEtaS * fabs(normal) * (pp.a * curve.half);
      bool converged = false;
      // Newton on g(V) = -invEtaS (|sigma_n| mu(V) - tau) - V from the
      // previous slip rate (RateAndState.h:339-416)
      for (int it = 0; it < prm.rs_max_slip_rate_updates; ++it) {
        if (active) {
          muF = curve.eval(test, num, root);
          g = -invEtaS * (fabs(normal) * muF - absShear) - test;
          ++newtonEvals;
        }
        converged = faceAll<TPF>(!active || fabs(g) < prm.rs_slip_rate_tolerance, NP);
        if (converged) break;
        if (active) {
          // - g / g' with g' = -slope num / root - 1
          test = fmax(kAlmostZero, test + g * root / (slope * num + root));
          ++newtonSteps;
        }
      }
      if (converged) muv = muF;
      else convInner &= (fabs(g) < prm.rs_slip_rate_tolerance) ? 1 : 0;
      if (record && !useMlp && j == 0 && active && converged &&
          !(lvc < log(0.5 * prm.rs_slip_rate_tolerance))) {
        // (features, log10 root - base) of the first solve of the time point
        // where the closed form does not apply; solves that move the slip rate
        // by more than a factor of two are all kept, the others thinned by a
        // hash to 1 in sample_stride
        base = features(lvc, upper, nScale, sv / pp.a, vPrev, pp.a, feat);
        const uint64_t h = (static_cast<uint64_t>(face) * 2654435761ULL) ^ (static_cast<uint64_t>(p) * 40503ULL) ^
                           (static_cast<uint64_t>(o) * 97ULL) ^ static_cast<uint64_t>(fullUpdateTime * 1e9);
        const bool moved = fabs(log10(test) - log10(vPrev)) > kMovedDecades;
        if (moved || opt.sample_stride <= 1 || (h % static_cast<uint64_t>(opt.sample_stride)) == 0) {
          const unsigned long long idx = atomicAdd(opt.sample_count, 1ULL);
          if (static_cast<int64_t>(idx) < opt.capacity) {
            for (int i = 0; i < kMlpInputs; ++i) opt.samples[idx * (kMlpInputs + 1) + i] = feat[i];
            opt.samples[idx * (kMlpInputs + 1) + kMlpInputs] = static_cast<float>(log10(test) - base);
          }
        }
      }
      const double old = srm;
      localSR = 0.5 * (old + test);
      convOuterPre = fabs(test - old) < prm.rs_state_tolerance;
      srm = test;
      if (faceAll<TPF>(!active || convOuterPre, NP)) break;
    }
    convOuter &= convOuterPre ? 1 : 0;
    // final state, friction, slip rates and tractions
    sv = active ? updateStateVariable(pp, prm.rs_sr0, svRef, dt, localSR) : 0.0;
    if (active) {
      double num, root;
      muv = MuCurve(pp.a, prm.rs_sr0, sv).eval(srm, num, root);
      const double strength = -muv * normal;
      const double t1 = s3 + fsT1, t2 = s5 + fsT2;
      const double divisor = strength + etaS * srm;
      slipRate1 = srm * t1 / divisor;
      slipRate2 = srm * t2 / divisor;
      trT1 = fsT1 - etaS * slipRate1;
      trT2 = fsT2 - etaS * slipRate2;
      accSlip += srm * dt;
      slip1 += slipRate1 * dt;
      slip2 += slipRate2 * dt;
      if (rupturePending && srm > 0.001) {
        ruptureTime = startTime;
        rupturePending = 0;
      }
      if (ruptureTime > 0.0 && ruptureTime <= startTime && dynStressPending &&
          muv <= pp.muw + 0.05 * (pp.f0 - pp.muw)) {
        dynStressTime = startTime;
        dynStressPending = 0;
      }
      peakSr = fmax(peakSr, srm);
      // imposed states (FrictionSolverCommon.h:333-401)
      const double w = args.timeWeights[o];
      sumN += w * fsN;
      sumT1 += w * trT1;
      sumT2 += w * trT2;
      minusV[0] += w * (m6 - invZpN * (fsN - m0));
      minusV[1] += w * (m7 - invZsN * (trT1 - m3));
      minusV[2] += w * (m8 - invZsN * (trT2 - m5));
      plusV[0] += w * (p6 + invZp * (fsN - p0));
      plusV[1] += w * (p7 + invZs * (trT1 - p3));
      plusV[2] += w * (p8 + invZs * (trT2 - p5));
    }
  }
  if (active) {
    at(L.accumulated_slip) = accSlip;
    at(L.slip1) = slip1;
    at(L.slip2) = slip2;
    at(L.peak_slip_rate) = peakSr;
    at(L.rupture_time) = ruptureTime;
    at(L.rupture_time_pending) = rupturePending;
    at(L.dyn_stress_time) = dynStressTime;
    at(L.dyn_stress_time_pending) = dynStressPending;
  }
  // state resampling over the face's points (postHook)
  __syncthreads();
  const double delta = active ? sv - at(L.state_variable) : 0.0;
  sDelta[threadIdx.x] = delta;
  __syncthreads();
  if (active) {
    const int base = (threadIdx.x / TPF) * TPF;
    double acc = 0.0;
    for (int q = 0; q < NP; ++q) acc += resample[p * NP + q] * sDelta[base + q];
    at(L.state_variable) += acc;
    at(L.slip_rate1) = slipRate1;
    at(L.slip_rate2) = slipRate2;
    at(L.slip_rate_magnitude) = srm;
    at(L.mu) = muv;
    at(L.traction1) = trT1;
    at(L.traction2) = trT2;
    at(L.convergence_inner) = convInner;
    at(L.convergence_outer) = convOuter;
    if (L.newton_iterations != nullptr) at(L.newton_iterations) += newtonEvals;
    if (L.slip_rate_updates != nullptr) at(L.slip_rate_updates) += newtonSteps;
    const double m[9] = {sumN, 0.0, 0.0, sumT1, 0.0, sumT2, minusV[0], minusV[1], minusV[2]};
    const double pl[9] = {sumN, 0.0, 0.0, sumT1, 0.0, sumT2, plusV[0], plusV[1], plusV[2]};
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      lane(L.imposed_state_minus + f0 * 9 * P, (fl * 9 + q) * P + p) = m[q];
      lane(L.imposed_state_plus + f0 * 9 * P, (fl * 9 + q) * P + p) = pl[q];
    }
  }
}

}  // namespace
}  // namespace friction
}  // namespace sdg

using namespace sdg;

extern "C" int sdg_friction_evaluate(const sdg_friction_params* params, const sdg_fault_layer* layer,
                                     double full_update_time, const double* delta_t, const double* time_weights,
                                     const double* resample, const sdg_friction_options* options, void* stream) {
  if (params == nullptr || layer == nullptr || delta_t == nullptr || time_weights == nullptr) {
    setError("sdg_friction_evaluate: NULL argument");
    return SDG_ERR_INVALID;
  }
  const sdg_fault_layer& L = *layer;
  if (L.num_faces < 0 || L.num_points < 1 || L.num_points > 64 || L.points < L.num_points || L.order < 1 ||
      L.order > friction::kMaxOrder) {
    setError("sdg_friction_evaluate: invalid layer sizes (num_points in [1, 64], order in [1, 8])");
    return SDG_ERR_INVALID;
  }
  if (L.num_faces == 0) return SDG_OK;
  if (resample == nullptr || L.imp_and_eta == nullptr || L.q_interpolated_plus == nullptr ||
      L.q_interpolated_minus == nullptr || L.initial_stress == nullptr || L.initial_pressure == nullptr ||
      L.rs_a == nullptr || L.rs_sl0 == nullptr || L.rs_f0 == nullptr || L.rs_muw == nullptr || L.rs_b == nullptr ||
      L.rs_srw == nullptr || L.state_variable == nullptr || L.slip_rate1 == nullptr || L.slip_rate2 == nullptr ||
      L.slip_rate_magnitude == nullptr || L.mu == nullptr || L.traction1 == nullptr || L.traction2 == nullptr ||
      L.slip1 == nullptr || L.slip2 == nullptr || L.accumulated_slip == nullptr || L.rupture_time == nullptr ||
      L.peak_slip_rate == nullptr || L.dyn_stress_time == nullptr || L.rupture_time_pending == nullptr ||
      L.dyn_stress_time_pending == nullptr || L.convergence_inner == nullptr || L.convergence_outer == nullptr ||
      L.imposed_state_plus == nullptr || L.imposed_state_minus == nullptr) {
    setError("sdg_friction_evaluate: missing fault-layer array");
    return SDG_ERR_INVALID;
  }
  if (params->nucleation_count > 1) {
    setError("sdg_friction_evaluate: at most one nucleation");
    return SDG_ERR_UNSUPPORTED;
  }
  sdg_friction_options opt{};
  if (options != nullptr) opt = *options;
  if (opt.samples != nullptr && opt.sample_count == nullptr) {
    setError("sdg_friction_evaluate: sample recording needs sample_count");
    return SDG_ERR_INVALID;
  }
  friction::StepArgs args{};
  for (int o = 0; o < L.order; ++o) {
    args.deltaT[o] = delta_t[o];
    args.timeWeights[o] = time_weights[o];
  }
  auto st = static_cast<hipStream_t>(stream);
  using friction::Start;
  auto launch = [&](auto tpf, auto start, auto index) {
    constexpr int TPF = decltype(tpf)::value, BLOCK = friction::kBlock<decltype(start)::value>, FPB = BLOCK / TPF;
    const unsigned grid = static_cast<unsigned>((L.num_faces + FPB - 1) / FPB);
    friction::kFriction<TPF, decltype(start)::value, decltype(index)>
        <<<grid, BLOCK, 0, st>>>(*params, L, full_update_time, args, resample, opt);
  };
  auto points = [&](auto start, auto index) {
    if (L.num_points <= 32) launch(std::integral_constant<int, 32>{}, start, index);
    else launch(std::integral_constant<int, 64>{}, start, index);
  };
  // 32-bit byte offsets reach the interpolated states of a block's faces, the
  // largest array, up to some 900,000 points (with the network's larger blocks)
  // or 3.7 million; beyond, 64-bit ones, in the one instantiation that has every start
  const auto narrow = [&](auto start) {
    const int fpb = friction::kBlock<decltype(start)::value> / (L.num_points <= 32 ? 32 : 64);
    return int64_t(fpb) * L.order * 9 * L.points * int64_t(sizeof(double)) <= int64_t(1) << 32;
  };
  constexpr std::integral_constant<Start, friction::kPlain> plain;
  constexpr std::integral_constant<Start, friction::kClosedForm> closedForm;
  constexpr std::integral_constant<Start, friction::kNetwork> network;
  auto run = [&](auto start) {
    if (narrow(start)) points(start, 0u);
    else points(network, uint64_t(0));
  };
  if (opt.mlp_params != nullptr || opt.samples != nullptr) run(network);
  else if (opt.closed_form_start != 0) run(closedForm);
  else run(plain);
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}
