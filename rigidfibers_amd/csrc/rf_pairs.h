// rf_pairs.h -- what the assembly kernels that form pairs by their target nodes
// share (rf_assemble.hip, rf_theta.h, rf_near.h): the inner integrals of one pair at one
// node, and the register budget.
#pragma once

#include "rf_internal.h"

namespace rf {

constexpr int kPairThreads = 192;

// Modes from the highest down: mode m is the last reader of the moments
// I3_{m+2}, I5_{m+2}, so they die as the sweep goes.
template <int N, int NQI, int M_>
__device__ __forceinline__ void analytic_modes(const NodeProducts& q, double eps2, const double* I1, const double* I3,
                                               const double* I5, float acc[N + 1][6]) {
  if constexpr (M_ >= 0) {
    double G[6];
    analytic_g<M_>(q, eps2, I1, I3, I5, G);
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[M_][c] = static_cast<float>(G[c]);
    analytic_modes<N, NQI, M_ - 1>(q, eps2, I1, I3, I5, acc);
  }
}

// G_m(q_i) for m = 0..N of one ordered pair (i, j) at the lane's target node:
// quadrature over q_j (mirror-paired nodes) or the exact FP64 integral.
template <int N, int NQI, bool ANALYTIC>
__device__ __forceinline__ void inner_integrals(const double xi[3], const double tid_[3], const float ti[3], double sq_d,
                                                float sq, double xj0, double xj1, double xj2, double tj0, double tj1,
                                                double tj2, const PhysConsts& pc, float acc[N + 1][6]) {
  constexpr Quad<N, NQI> quad{};
  constexpr int Q = 3 * NQI;
  constexpr int NM = N + 1;
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[m][c] = 0.0f;
  if constexpr (!ANALYTIC) {
    // R(q_i, q_j) = (x_i - x_j) + s_i t_i - s_j t_j; the centre difference is
    // formed in FP64 and rounded once.
    const float ax = fmaf(sq, ti[0], static_cast<float>(xi[0] - xj0));
    const float ay = fmaf(sq, ti[1], static_cast<float>(xi[1] - xj1));
    const float az = fmaf(sq, ti[2], static_cast<float>(xi[2] - xj2));
    const float tx = static_cast<float>(tj0), ty = static_cast<float>(tj1), tz = static_cast<float>(tj2);
#pragma unroll
    for (int h = 0; h < Q / 2; ++h) {
      const float s = quad.s[h];
      const float ux = s * tx, uy = s * ty, uz = s * tz;
      float Kp[6], Km[6];
      stokes_kernel(ax - ux, ay - uy, az - uz, pc.eps2, Kp);  // node h (s)
      stokes_kernel(ax + ux, ay + uy, az + uz, pc.eps2, Km);  // node Q-1-h (-s)
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const float E = Kp[c] + Km[c];
        const float O = Kp[c] - Km[c];
#pragma unroll
        for (int m = 0; m < NM; ++m) acc[m][c] = fmaf(quad.W[m][h], (m & 1) ? O : E, acc[m][c]);
      }
    }
  } else {
    const double R0[3] = {xi[0] - xj0 + sq_d * tid_[0], xi[1] - xj1 + sq_d * tid_[1], xi[2] - xj2 + sq_d * tid_[2]};
    const double ll = R0[0] * R0[0] + R0[1] * R0[1] + R0[2] * R0[2];
    if (ll >= kFarField[N] * kFarField[N]) {
      // far field: 8-point Gauss-Legendre over the source fiber (FP32)
      constexpr FarQuad<N> far{};
      const float rx = static_cast<float>(R0[0]), ry = static_cast<float>(R0[1]), rz = static_cast<float>(R0[2]);
      const float tx = static_cast<float>(tj0), ty = static_cast<float>(tj1), tz = static_cast<float>(tj2);
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float s = far.s[h];
        const float ux = s * tx, uy = s * ty, uz = s * tz;
        float Kp[6], Km[6];
        stokes_kernel(rx - ux, ry - uy, rz - uz, pc.eps2, Kp);  // node +s
        stokes_kernel(rx + ux, ry + uy, rz + uz, pc.eps2, Km);  // node -s
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          const float E = Kp[c] + Km[c];
          const float O = Kp[c] - Km[c];
#pragma unroll
          for (int m = 0; m < NM; ++m) acc[m][c] = fmaf(far.W[m][h], (m & 1) ? O : E, acc[m][c]);
        }
      }
    } else {
      const double tjd[3] = {tj0, tj1, tj2};
      const double bb = -2.0 * (R0[0] * tj0 + R0[1] * tj1 + R0[2] * tj2);
      double I1[N + 3], I3[N + 3], I5[N + 3];
      moments<N>(bb, ll, I1, I3, I5);
      analytic_modes<N, NQI, N>(node_products(R0, tjd), pc.eps2_d, I1, I3, I5, acc);
    }
  }
}

// Waves per SIMD a kernel asks the register allocator for: as many as the
// workgroups whose LDS (the sweeps' and `extra` bytes) fits a CU's 160 KB can use,
// at most 3 for the analytical form (its FP64 moments need more than the 128
// registers of 4 waves; 3 waves allow 168).
template <int N, int NQI, bool ANALYTIC>
constexpr int theta_min_waves(int extra) {
  constexpr int Q = 3 * NQI, PAIRS = kPairThreads / Q, NM = N + 1;
  constexpr int RP = 6 * PAIRS * NM;
  const int bytes = 4 * (RP * Q + NM * RP) + 8 * PAIRS * (3 * N + 6) + 8 * kMaxTerms + extra;
  const int blocks = (160 * 1024) / bytes;
  return (blocks >= 5 && !ANALYTIC) ? 4 : (blocks >= 4 ? 3 : (blocks >= 3 ? 2 : 1));
}
// The product sums of the source slots, and the near kernel's lists.
template <int N, int NQI>
constexpr int kProductBytes = 8 * (kPairThreads / (3 * NQI)) * (3 * N - 2);
template <int N, int NQI>
constexpr int kListBytes = 4 * (2 * kPairThreads + 2 * (kPairThreads / (3 * NQI)) + 6);

}  // namespace rf
