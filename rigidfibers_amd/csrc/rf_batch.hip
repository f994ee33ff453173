// rf_batch.hip -- the assembly of a served batch: workgroup = (suspension, target
// fiber), all of its sources in one group.
//
// A file of its own, like rf_near.hip: a process that serves loads these kernels
// and not the single suspension's.
#include "rf_near.h"
#include "rf_theta.h"

namespace rf {

// Serving: workgroup = (suspension, target fiber), all sources in one group, so
// b and the velocity constants are written directly, and with them the first
// GMRES residual (into the basis' first vector) and its norms.
template <int N, int NQI, bool ANALYTIC>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(
    theta_min_waves<N, NQI, ANALYTIC>(0), 8))) void assemble_theta_batch_kernel(
    const SusDev* __restrict__ sus, const int2* __restrict__ targets, PhysConsts pc) {
  const int2 e = targets[blockIdx.x];
  const SusDev& d = sus[e.x];
  assemble_theta_block<N, NQI, ANALYTIC, false, true>(e.y, 0, d.M, d.Lp, d.pos, d.ori, d.T, d.b, d.M, pc, d.Tv,
                                                      d.cpart, nullptr, nullptr, nullptr, nullptr, &d);
}

// Serving: workgroup = (suspension, target fiber), all sources in one group, after
// the far kernel, whose sums are added, so b and the velocity constants are complete
// here, and with them the first GMRES residual (into the basis' first vector) and
// its norms.
template <int N, int NQI, bool ANALYTIC>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(
    theta_min_waves<N, NQI, ANALYTIC>(kProductBytes<N, NQI> + kListBytes<N, NQI>), 8))) void assemble_near_batch_kernel(
    const SusDev* __restrict__ sus, const int2* __restrict__ targets, PhysConsts pc) {
  const int2 e = targets[blockIdx.x];
  const SusDev& d = sus[e.x];
  assemble_near_block<N, NQI, ANALYTIC>(e.y, 0, d.M, d.Lp, d.pos, d.ori, d.T, d.b, d.M, pc, d.Tv, d.cpart, nullptr,
                                        nullptr, nullptr, nullptr, &d);
}

template <int N, int NQI, bool AN>
static hipError_t launch_theta_batch_t(int nfar, int ntargets, const SusDev* sus, const int2* targets,
                                       const PhysConsts& pc, hipStream_t s) {
  if (nfar > 0) {
    const hipError_t e = launch_assemble_far_batch(N, NQI, AN, nfar, sus, targets, pc, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((assemble_near_batch_kernel<N, NQI, AN>), dim3(nfar), dim3(kPairThreads), 0, s, sus, targets,
                       pc);
  }
  if (ntargets > nfar)
    hipLaunchKernelGGL((assemble_theta_batch_kernel<N, NQI, AN>), dim3(ntargets - nfar), dim3(kPairThreads), 0, s,
                       sus, targets + nfar, pc);
  return hipGetLastError();
}

template <int N, int NQI>
static hipError_t launch_theta_batch_n(bool an, int nfar, int ntargets, const SusDev* sus, const int2* targets,
                                       const PhysConsts& pc, hipStream_t s) {
  return an ? launch_theta_batch_t<N, NQI, true>(nfar, ntargets, sus, targets, pc, s)
            : launch_theta_batch_t<N, NQI, false>(nfar, ntargets, sus, targets, pc, s);
}

hipError_t launch_assemble_theta_batch(int N, int NQI, bool analytical, int nfar, int ntargets, const SusDev* sus,
                                       const int2* targets, const PhysConsts& pc, hipStream_t s) {
  if (ntargets <= 0) return hipSuccess;
  switch (N) {
#define RF_TB(NN)                                                                                 \
  case NN:                                                                                        \
    if (NQI == 4) return launch_theta_batch_n<NN, 4>(analytical, nfar, ntargets, sus, targets, pc, s);   \
    if (NQI == 8) return launch_theta_batch_n<NN, 8>(analytical, nfar, ntargets, sus, targets, pc, s);   \
    if (NQI == 16) return launch_theta_batch_n<NN, 16>(analytical, nfar, ntargets, sus, targets, pc, s); \
    return hipErrorInvalidValue;
    RF_TB(1)
    RF_TB(2)
    RF_TB(3)
    RF_TB(4)
    RF_TB(5)
    RF_TB(6)
    RF_TB(7)
    RF_TB(8)
#undef RF_TB
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace rf
