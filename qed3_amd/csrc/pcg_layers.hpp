// The network's layers as the preconditioned CG launches them (pcg.hip): their epilogues, and
// the launchers' instantiations, which are compiled in pcg_layers_*.hip side by side (each
// is some thirty kernels).
#pragma once
#include "cg_epi.hpp"
#include "horner_kernels.hpp"

namespace qed3 {
namespace pcgl {

// the network's layers wait, like K1 and K2, for a pending reliable update
struct EpiSkip {
  static constexpr bool kReduce = false;
  const CGScalars* sc;
  __device__ bool skip() const { return sc->done != 0 || sc->need_ru != 0; }
  __device__ void operator()(size_t, const Spin<float>&, double2&) const {}
  __device__ void operator()(double2) const {}
};

// Last layer of K, injecting H = K^dagger r as stored beside H_old (hk::SrcDots), which
// reduces t = (|H|^2, <H_old, H>) = (<r, z>, <r_old, z>): the FCG scalars.  After a reliable
// update r is the true residual at the new scale while H_old and p_old are at the old one
// (rfac = old / new): beta = (|H|^2 - rfac <H_old, H>) / (rfac rho_old).
struct EpiFcg {
  static constexpr bool kReduce = true;
  CGScalars* sc;
  __device__ bool skip() const { return sc->done != 0 || sc->need_ru != 0; }
  __device__ void operator()(size_t, const Spin<float>&, double2&) const {}
  __device__ void operator()(double2 t) const {
    const double A = t.x, Bv = t.y;
    if (!(A > 0.0 && A < 1e300) || (!sc->fresh && !(fabs(Bv) < 1e300))) {
      sc->done = 2;  // M r must be a descent direction: <r, M r> > 0
      return;
    }
    double beta = 0.0;
    if (!sc->fresh) {
      const double f = sc->rescale ? sc->rfac : 1.0;
      beta = (A - f * Bv) / (f * sc->rho);
    }
    sc->beta = beta;
    sc->rho = A;
    sc->mu = A;  // K1: alpha = mu / |D p|^2
    sc->fresh = 0;
  }
};

}  // namespace pcgl

// every (layer, source, epilogue) the solver and the checked application launch
#define QED3_TC_LAUNCH(ADJ, FIRST, SRC, EPI)                                                                   \
  template void hk::launch_horner_layer_tc<ADJ, FIRST, SRC, EPI>(                                              \
      const HornerView&, const DiracView<float, phasepair_t>&, const HaloView&, const SRC&, const SpinH*, SpinH*, \
      float2, const EPI&, GridReduce, hipStream_t, const hipEvent_t*, SpinH*, float2);
#define QED3_TC_KDAG(X)                 \
  X(true, true, hk::SrcFS, pcgl::EpiSkip) \
  X(true, false, hk::SrcFS, pcgl::EpiSkip)
#define QED3_TC_K(X)                                \
  X(false, true, hk::SrcF<SpinH>, pcgl::EpiSkip)    \
  X(false, false, hk::SrcF<SpinH>, pcgl::EpiSkip)   \
  X(false, true, hk::SrcDots, pcgl::EpiFcg)         \
  X(false, false, hk::SrcDots, pcgl::EpiFcg)
#define QED3_TC_CHECK(X)                        \
  X(true, true, hk::SrcF<SpinH>, hk::EpiNone)   \
  X(true, false, hk::SrcF<SpinH>, hk::EpiNone)  \
  X(false, true, hk::SrcF<SpinH>, hk::EpiNone)  \
  X(false, false, hk::SrcF<SpinH>, hk::EpiNone)
}  // namespace qed3
