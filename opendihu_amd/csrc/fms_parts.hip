// One object per FMS_PART (fms_parts.h).
#include "fms_parts.h"

namespace fms {

template <class G, class E, int T, int C, bool TAPE> void fibre_launch_shape(const FibreLaunch &l) {
  const auto kernel = k_fibre<Model, G, E, T, C, TAPE>;
  const size_t lds = chunk_lds_doubles<T>((l.nmax + T - 1) / T) * sizeof(double);
  G *gates = static_cast<G *>(l.gates);
  if (l.start)
    hipExtLaunchKernelGGL(kernel, dim3(l.fb.n_fibers), dim3(T), lds, l.stream, l.start, l.stop, 0, l.fb, l.st, l.vm,
                          gates, l.steps, l.K, l.n0D, l.ie, l.order, l.spk, l.tr);
  else
    hipLaunchKernelGGL(kernel, dim3(l.fb.n_fibers), dim3(T), lds, l.stream, l.fb, l.st, l.vm, gates, l.steps, l.K,
                       l.n0D, l.ie, l.order, l.spk, l.tr);
}

template <class G, class E, bool TAPE> void fibre_launch(int T, const FibreLaunch &l) {
  // 512 threads are for fibres of more than 2048 nodes, which the adjoint does not take
  if constexpr (!TAPE)
    if (T == 512) return fibre_launch_shape<G, E, 512, 8, TAPE>(l);
  if (T == 128) fibre_launch_shape<G, E, 128, 8, TAPE>(l);
  else fibre_launch_shape<G, E, 256, 8, TAPE>(l);
}

template <class E, int T, int CMAX> void adjoint_launch_threads(int nmax, const AdjArgs &a, hipStream_t stream) {
  const size_t lds = chunk_lds_doubles<T>((nmax + T - 1) / T) * sizeof(double);
  hipLaunchKernelGGL((k_adj_steps<E, T, CMAX>), dim3(a.fb.n_fibers), dim3(T), lds, stream, a);
}

template <class E> void adjoint_launch(int T, int nmax, const AdjArgs &a, hipStream_t stream) {
  if (T == 256) adjoint_launch_threads<E, 256, 4>(nmax, a, stream);
  else adjoint_launch_threads<E, 512, 4>(nmax, a, stream);
}

#if FMS_PART == 0
template void fibre_launch<double, ExpApproxFma, false>(int, const FibreLaunch &);
#elif FMS_PART == 1
template void fibre_launch<double, ExpLibmFma, false>(int, const FibreLaunch &);
#elif FMS_PART == 2
template void fibre_launch<float, ExpApproxFma, false>(int, const FibreLaunch &);
#elif FMS_PART == 3
template void fibre_launch<float, ExpLibmFma, false>(int, const FibreLaunch &);
#elif FMS_PART == 4
template void fibre_launch<double, ExpApproxFma, true>(int, const FibreLaunch &);
#elif FMS_PART == 5
template void fibre_launch<double, ExpLibmFma, true>(int, const FibreLaunch &);
#elif FMS_PART == 6
template void adjoint_launch<ExpApproxFma>(int, int, const AdjArgs &, hipStream_t);
#elif FMS_PART == 7
template void adjoint_launch<ExpLibmFma>(int, int, const AdjArgs &, hipStream_t);
#endif

}  // namespace fms
