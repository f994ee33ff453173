// rf_near.hip -- the near pairs of the theta-form assembly, beside the far pairs'
// kernel (rf_far.hip), of one suspension.
//
// A file of its own: a program's first launch of any of a file's kernels loads all
// of them, about 2 ms per MB, and suspensions without a far kernel need none of
// these.
#include "rf_near.h"

namespace rf {

template <int N, int NQI, bool ANALYTIC, bool HALF>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(
    theta_min_waves<N, NQI, ANALYTIC>(kProductBytes<N, NQI> + kListBytes<N, NQI>), 8))) void assemble_near_kernel(
    int M, int64_t Lp, const double* __restrict__ pos, const double* __restrict__ ori, float* __restrict__ T,
    double* __restrict__ bpart, int jgroup, PhysConsts pc, float* __restrict__ Tv, double* __restrict__ cpart,
    const double* __restrict__ x0, double* __restrict__ apart, _Float16* __restrict__ T16, float* __restrict__ S16) {
  assemble_near_block<N, NQI, ANALYTIC, HALF>(blockIdx.x, blockIdx.y, M, Lp, pos, ori, T, bpart, jgroup, pc, Tv,
                                              cpart, x0, apart, T16, S16);
}

template <int N, int NQI, bool AN>
static hipError_t launch_near_t(int M, int64_t Lp, const double* pos, const double* ori, float* T, double* bpart,
                                const PairGrid& g, float* Tv, double* cpart, const double* x0, double* apart,
                                const PhysConsts& pc, hipStream_t s, _Float16* T16, float* S16) {
  const dim3 grid(M, g.groups), block(kPairThreads);
  if (T16)
    hipLaunchKernelGGL((assemble_near_kernel<N, NQI, AN, true>), grid, block, 0, s, M, Lp, pos, ori, T, bpart,
                       g.jgroup, pc, Tv, cpart, x0, apart, T16, S16);
  else
    hipLaunchKernelGGL((assemble_near_kernel<N, NQI, AN, false>), grid, block, 0, s, M, Lp, pos, ori, T, bpart,
                       g.jgroup, pc, Tv, cpart, x0, apart, nullptr, nullptr);
  return hipGetLastError();
}

template <int N, int NQI>
static hipError_t launch_near_n(bool an, int M, int64_t Lp, const double* pos, const double* ori, float* T,
                                double* bpart, const PairGrid& g, float* Tv, double* cpart, const double* x0,
                                double* apart, const PhysConsts& pc, hipStream_t s, _Float16* T16, float* S16) {
  return an ? launch_near_t<N, NQI, true>(M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16)
            : launch_near_t<N, NQI, false>(M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16);
}

hipError_t launch_assemble_near(int N, int NQI, bool analytical, int M, int64_t Lp, const double* pos,
                                const double* ori, float* T, double* bpart, const PairGrid& g, float* Tv,
                                double* cpart, const double* x0, double* apart, const PhysConsts& pc, hipStream_t s,
                                _Float16* T16, float* S16) {
  switch (N) {
#define RF_NEAR(NN)                                                                                              \
  case NN:                                                                                                       \
    if (NQI == 4)                                                                                                \
      return launch_near_n<NN, 4>(analytical, M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16);  \
    if (NQI == 8)                                                                                                \
      return launch_near_n<NN, 8>(analytical, M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16);  \
    if (NQI == 16)                                                                                               \
      return launch_near_n<NN, 16>(analytical, M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16); \
    return hipErrorInvalidValue;
    RF_NEAR(1)
    RF_NEAR(2)
    RF_NEAR(3)
    RF_NEAR(4)
    RF_NEAR(5)
    RF_NEAR(6)
    RF_NEAR(7)
    RF_NEAR(8)
#undef RF_NEAR
    default:
      return hipErrorInvalidValue;
  }
}


}  // namespace rf
