// Launches of the small models' largest kernels. Their instantiations take most of
// a library's compile time, so fms_parts.hip compiles them in several objects
// beside the host runtime (fms_lib.hip), one per gate type and exponential.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "fms_adjoint.h"
#include "fms_fibre.h"
#include "fms_model.h"

namespace fms {

struct FibreLaunch {
  DevFibers fb;
  FibreStim st;
  double *vm;
  void *gates;
  const double *steps;
  int nmax, K, n0D, ie;
  const int *order;
  DevSpikes spk;
  DevTrace tr;
  hipStream_t stream;
  hipEvent_t start, stop;   // bound to the launch, or null
};

// T threads per fibre: 128, 256 or (without the tape) 512
template <class G, class E, bool TAPE> void fibre_launch(int T, const FibreLaunch &l);

extern template void fibre_launch<double, ExpApproxFma, false>(int, const FibreLaunch &);
extern template void fibre_launch<double, ExpLibmFma, false>(int, const FibreLaunch &);
extern template void fibre_launch<float, ExpApproxFma, false>(int, const FibreLaunch &);
extern template void fibre_launch<float, ExpLibmFma, false>(int, const FibreLaunch &);
extern template void fibre_launch<double, ExpApproxFma, true>(int, const FibreLaunch &);
extern template void fibre_launch<double, ExpLibmFma, true>(int, const FibreLaunch &);

// the reverse sweep of one segment (Hodgkin-Huxley only), T threads per fibre: 256 or 512
template <class E> void adjoint_launch(int T, int nmax, const AdjArgs &a, hipStream_t stream);

extern template void adjoint_launch<ExpApproxFma>(int, int, const AdjArgs &, hipStream_t);
extern template void adjoint_launch<ExpLibmFma>(int, int, const AdjArgs &, hipStream_t);

}  // namespace fms
