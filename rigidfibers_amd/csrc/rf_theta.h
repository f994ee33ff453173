// rf_theta.h -- the theta form, and the kernel body that forms every pair of it
// (rf_assemble.hip for one suspension, rf_batch.hip for a served batch).
#pragma once

#include "rf_pairs.h"

namespace rf {

// Theta form of the system, for the iterative solvers.
//
// Every off-diagonal 3x3 block of A is fixed by t_i and the symmetric
// projection Theta_{k_i,k_j} (fortran/assemble_matrix.incl:59-79,117-137):
//   k_i = 0:  A_blk = D1 t_i Q0^T,  Q0 = Theta_{0,k_j} t_i            (3 numbers)
//   k_i > 0:  A_blk = gamma_k (Theta - eigen_k t_i (Theta t_i)^T)     (6 numbers)
// so 3 + 6(N-1) numbers per (i, j, k_j) carry the 9N entries of a block
// column (27 instead of 45 for N = 5).  They are stored as component arrays
//   T[(i * NC + c) * Lp + j * N + k_j],  NC = 3 + 6(N-1),  Lp >= M*N,
// c = b for Q0_b, c = 3 + 6(k_i-1) + s for Theta_{k_i}[s] (s = xx yy zz xy xz yz),
// zero for j == i (the identity diagonal blocks are implicit).

// Velocity operator (when the velocities integrate like the system): the
// reference's velocity sums (fortran/update_velocities.incl:29-86) are
// projections of the same inner integrals G_m(q_i) the assembly forms,
//   sum_j TFA0_ij = sum_j [Phi0_{ij,0} F/2 + sum_k Phi0_{ij,k+1} x_{j,k}]   (weights w)
//   sum_j TFA1_ij = sum_j [Theta_{ij,0,P0} F/2 + sum_k Theta_{ij,0,k} x_{j,k}] (weights w P_1)
// so with Tv != nullptr the kernel also stores, per (i, j, k_j), the
// symmetric Theta_{0,k_j} and Phi0_{k_j+1} = sum_{q_i} w G_{k_j+1}(q_i)
//   Tv[(i * 12 + c) * Lp + j * N + k_j],  c = s (Theta_0), 6 + s (Phi0),
// and in cpart[group][i][6] the constant sums of Phi0_{ij,0} F/2 and
// Theta_{ij,0,P0} F/2 over its sources.

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Every pair of one workgroup: target fiber i, source group gy.  For suspensions
// below far_min_fibers and the direct solvers; the near kernel (rf_near.h), which
// lists its sources, took 12 to 15% longer at this with exact integrals (M = 437: 147
// against 130 us, 5000: 14.0 against 12.0 ms) and 2.5% with numerical ones in a
// served batch (24 suspensions, 1.143 against 1.085 ms).
//   phase 1  lane (p, q_i) writes G_m(q_i) of source slot p into LDS as row
//            r = c*CB + (m == 0 ? p : PAIRS + p*N + m-1) of a GEMM operand
//            (c = symmetric component; the mode-0 rows feed the RHS).
//   phase 2  lane r forms C[r][kk] = sum_q W[kk][q] G[r][q] (kk = 0..N: the
//            projections onto w P_kk) for all kk from the mirror sums
//            E = G(q) + G(-q) and differences O = G(q) - G(-q): the weights
//            satisfy W[kk][-q] = (-1)^kk W[kk][q] exactly, so even kk take E,
//            odd kk take O, and the table entries are immediate operands.
//   phase 3  each lane writes 4 consecutive (source, mode) columns of one
//            component array (16-byte stores); the k_i = 0 components
//            (Theta_0 t_i) and the RHS of each source slot are formed here.
// With x0, the workgroup also forms its share of the off-diagonal product,
// sum_{j in group} A_ij x0_j, into apart[gy n + row] (FP32 values times FP64 x0,
// FP64 sums), in one of two ways.  A single suspension's launch is latency: the
// lanes of the RHS take it from the projections in LDS (warm assembly with
// numerical / exact integrals, in us, against the read-back: M = 100 22.2 / 19.6
// against 28.6 / 26.2, 310 104.5 / 79.2 against 109 / 83.7).  A served batch fills
// the chip, and there those few lanes hold up the workgroup (1.144 against 1.09 ms
// for 24 suspensions): the rows are read back after the sweeps, which is memory
// traffic while the other workgroups of the CU keep its VALUs busy.
// HALF (GMRES-IR's FP16 copy T16, S16): phase 2 also takes each (target,
// source) block's largest |projection|, phase 3 stores the block scales, and
// the read-back (run then with or without x0) converts the stored values.
template <int N, int NQI, bool ANALYTIC, bool HALF, bool SERVING>
__device__ __forceinline__ void assemble_theta_block(int i, int gy, int M, int64_t Lp, const double* __restrict__ pos,
                                                     const double* __restrict__ ori, float* __restrict__ T,
                                                     double* __restrict__ bpart, int jgroup, const PhysConsts& pc,
                                                     float* __restrict__ Tv, double* __restrict__ cpart,
                                                     const double* __restrict__ x0, double* __restrict__ apart,
                                                     _Float16* __restrict__ T16, float* __restrict__ S16,
                                                     const SusDev* __restrict__ serving) {
  constexpr Quad<N, NQI> quad{};
  constexpr int Q = 3 * NQI;
  constexpr int PAIRS = kPairThreads / Q;
  constexpr int NM = N + 1;
  constexpr int ROWS = 3 * N;
  constexpr int NC = 3 + 6 * (N - 1);
  constexpr int NR = ROWS + 6;  // RHS rows + the two velocity constants
  constexpr int NACC = 1 + 3 * (N - 1);  // s0 = Q0 . x0, then U_k = Theta_k x0 (k >= 1)
  constexpr bool kReadBack = SERVING || HALF;
  constexpr int PN = PAIRS * N;  // (source, mode) columns of one sweep
  constexpr int CB = PAIRS + PN;  // GEMM rows per component
  constexpr int RP = 6 * CB;  // GEMM rows
  constexpr int NV = PN / 4;  // float4 chunks per component and sweep
  static_assert(kPairThreads % Q == 0 && Q % 2 == 0 && PAIRS % 4 == 0, "sweep shapes");

  __shared__ __align__(16) float G[RP * Q];
  __shared__ __align__(16) float Pj[NM * RP];
  __shared__ double bred[PAIRS][NR];
  __shared__ double ared[kReadBack ? 1 : PAIRS][NACC];
  __shared__ float modes[2 * kMaxTerms];  // gamma_k, then eigen_k
  // FP16 copy: each source slot's largest |projection| (float bits), one
  // buffer per sweep parity
  __shared__ unsigned smax[2][PAIRS];

  const int tid = threadIdx.x;
  const int p = tid / Q;
  const int qi = tid - p * Q;
  const int jb = gy * jgroup;
  const int je = min(M, jb + jgroup);
  const int64_t n = static_cast<int64_t>(ROWS) * M;

  const double xi[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
  const double tid_[3] = {ori[3 * i], ori[3 * i + 1], ori[3 * i + 2]};
  const float ti[3] = {static_cast<float>(tid_[0]), static_cast<float>(tid_[1]), static_cast<float>(tid_[2])};
  const double sq_d = node_fp64<NQI>(qi);
  const float sq = static_cast<float>(sq_d);
  float* Ti = T + static_cast<int64_t>(i) * NC * Lp;
  float* Vi = Tv ? Tv + static_cast<int64_t>(i) * 12 * Lp : nullptr;

  // RHS (and velocity-constant) and product sums of each source slot, kept in
  // LDS; the mode factors gamma_k, eigen_k as a table the RHS lanes index by k
  for (int r = tid; r < PAIRS * NR; r += kPairThreads) bred[r / NR][r % NR] = 0.0;
  if constexpr (!kReadBack) {
    for (int r = tid; r < PAIRS * NACC; r += kPairThreads) ared[r / NACC][r % NACC] = 0.0;
  }
  if (tid < 2 * PAIRS) smax[tid / PAIRS][tid % PAIRS] = 0u;
#pragma unroll
  for (int t = 0; t < kMaxTerms; ++t)
    if (tid == t) {
      modes[t] = pc.gamma[t];
      modes[kMaxTerms + t] = pc.eigen[t];
    }
  __syncthreads();

  for (int j0 = jb; j0 < je; j0 += PAIRS) {
    const int j = j0 + p;
    if (j < je && j != i) {
      float acc[NM][6];
      inner_integrals<N, NQI, ANALYTIC>(xi, tid_, ti, sq_d, sq, pos[3 * j], pos[3 * j + 1], pos[3 * j + 2],
                                        ori[3 * j], ori[3 * j + 1], ori[3 * j + 2], pc, acc);
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int c = 0; c < 6; ++c) G[(c * CB + (m == 0 ? p : PAIRS + p * N + m - 1)) * Q + qi] = acc[m][c];
    }
    __syncthreads();
    // FP16 copy: this sweep's block maxima go to smax[par]; the other buffer,
    // last read in the previous sweep's phase 3 (before the barrier above), is
    // cleared for the next sweep
    const int par = ((j0 - jb) / PAIRS) & 1;
    if constexpr (HALF) {
      if (tid < PAIRS) smax[par ^ 1][tid] = 0u;
    }
    for (int r = tid; r < RP; r += kPairThreads) {
      const float* gr = G + r * Q;
      float E[Q / 2], O[Q / 2];
#pragma unroll
      for (int h = 0; h < Q / 2; ++h) {
        const float x = gr[h], y = gr[Q - 1 - h];
        E[h] = x + y;
        O[h] = x - y;
      }
      float g = 0.0f;
#pragma unroll
      for (int kk = 0; kk < NM; ++kk) {
        float acc = 0.0f;
#pragma unroll
        for (int h = 0; h < Q / 2; ++h) acc = fmaf(quad.W[kk][h], (kk & 1) ? O[h] : E[h], acc);
        Pj[kk * RP + r] = acc;
        if (kk > 0) g = fmaxf(g, fabsf(acc));
      }
      if constexpr (HALF) {  // rows of the modes m >= 1 feed the system components
        const int e = r % CB;
        if (e >= PAIRS) atomicMax(&smax[par][(e - PAIRS) / N], __float_as_uint(g));
      }
    }
    __syncthreads();
    const int npm = min(PAIRS, je - j0) * N;  // valid columns of this sweep
    const bool full = npm == PN;                // every sweep but possibly the last
    const bool self_here = i >= j0 && i < j0 + PAIRS;  // the self pair's columns are in this sweep
    const int sself = (i - j0) * N;
    float* const Tcol = Ti + static_cast<int64_t>(j0) * N;  // this sweep's first column, component 0
    // 4 consecutive columns of one component array (offset `off` from the
    // sweep's first column of component 0): self-pair columns zeroed, columns
    // past the sweep's last source not written.  The conditions are uniform
    // over the workgroup except in the sweep that holds them.
    auto put = [&](float* base, uint32_t off, int pm0, floatx4& val) {
      if (self_here) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (static_cast<unsigned>(pm0 + e - sself) < static_cast<unsigned>(N)) val[e] = 0.0f;
      }
      float* dst = base + off;
      if (full || pm0 + 3 < npm) {
        *reinterpret_cast<floatx4*>(dst) = val;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (pm0 + e < npm) dst[e] = val[e];
      }
    };
    const uint32_t lp32 = static_cast<uint32_t>(Lp);
    // system components: u < 3 Q0_u = (Theta_0 t_i)_u (Theta_0 = the P_1
    // projection), then Theta_{k_i} for k_i = 1..N-1 (projection k_i + 1)
    auto sys_val = [&](int u, int pm0) {
      floatx4 val;
      if (u < 3) {
        const float* b1 = Pj + RP + PAIRS + pm0;
        const floatx4 x0 = *reinterpret_cast<const floatx4*>(b1 + sym_index(0, u) * CB);
        const floatx4 x1 = *reinterpret_cast<const floatx4*>(b1 + sym_index(1, u) * CB);
        const floatx4 x2 = *reinterpret_cast<const floatx4*>(b1 + sym_index(2, u) * CB);
#pragma unroll
        for (int e = 0; e < 4; ++e) val[e] = x0[e] * ti[0] + x1[e] * ti[1] + x2[e] * ti[2];
      } else {
        const int kk = 2 + (u - 3) / 6;
        const int c = (u - 3) - 6 * (kk - 2);
        val = *reinterpret_cast<const floatx4*>(Pj + kk * RP + c * CB + PAIRS + pm0);
      }
      return val;
    };
    // FP16 copy: the sweep's block scales (S16); the values are converted
    // when the workgroup reads its rows back after the sweeps
    if constexpr (HALF) {
      if (tid < PAIRS && j0 + tid < je) {
        float sv, iv;
        // the self pair's slot holds no projections: its block is zero
        half_block_scale(j0 + tid == i ? 0u : smax[par][tid], sv, iv);
        S16[static_cast<int64_t>(i) * M + j0 + tid] = sv;
      }
    }
    for (int job = tid; job < NC * NV; job += kPairThreads) {
      const int u = job / NV;
      const int pm0 = 4 * (job - u * NV);
      floatx4 val = sys_val(u, pm0);
      put(Tcol, static_cast<uint32_t>(u) * lp32 + static_cast<uint32_t>(pm0), pm0, val);
    }
    // velocity operator: Theta_0 (projection 1), then Phi_0 (projection 0).
    // Analytical form: its jobs start on the lanes after the system
    // components' last partial pass and the RHS jobs sit on the top lanes,
    // so the three waves get the same number of passes (measured faster
    // there, slower for the numerical form, which keeps the plain order).
    if (Vi) {
      float* const Vcol = Vi + static_cast<int64_t>(j0) * N;
      constexpr int kVShift = ANALYTIC ? kPairThreads - (NC * NV) % kPairThreads : 0;
      for (int job = (tid + kVShift) % kPairThreads; job < 12 * NV; job += kPairThreads) {
        const int w = job / NV;
        const int pm0 = 4 * (job - w * NV);
        const int kk = w < 6 ? 1 : 0;
        const int c = w < 6 ? w : w - 6;
        floatx4 val = *reinterpret_cast<const floatx4*>(Pj + kk * RP + c * CB + PAIRS + pm0);
        put(Vcol, static_cast<uint32_t>(w) * lp32 + static_cast<uint32_t>(pm0), pm0, val);
      }
    }
    // RHS (source slot p2, row block k): k < N forms rows 3k..3k+2 of b from
    // the projection of G_0 F/2 onto w P_{k+1}; k = N the velocity constants
    // sum_q w G_0 F/2 and sum_q w P_1 G_0 F/2.  Without the read-back, row
    // block k < N of A x0 too.
    constexpr int kRShift = ANALYTIC ? PAIRS * (N + 1) % kPairThreads : 0;
    for (int rj = (tid + kRShift) % kPairThreads; rj < PAIRS * (N + 1); rj += kPairThreads) {
      const int p2 = rj / (N + 1), k = rj - p2 * (N + 1), j2 = j0 + p2;
      if (j2 >= je || j2 == i) continue;
      auto proj = [&](int kk, float f[3]) {  // sum_b Theta^(0)_kk[a][b] F_b / 2
        const float* b0 = Pj + kk * RP + p2;
        const float g0 = b0[0 * CB], g1 = b0[1 * CB], g2 = b0[2 * CB];
        const float g3 = b0[3 * CB], g4 = b0[4 * CB], g5 = b0[5 * CB];
        f[0] = g0 * pc.Fh[0] + g3 * pc.Fh[1] + g4 * pc.Fh[2];
        f[1] = g3 * pc.Fh[0] + g1 * pc.Fh[1] + g5 * pc.Fh[2];
        f[2] = g4 * pc.Fh[0] + g5 * pc.Fh[1] + g2 * pc.Fh[2];
      };
      double* br = bred[p2];
      if (k < N) {
        float TF[3];
        proj(k + 1, TF);
        const float gam = modes[k], eig = modes[kMaxTerms + k];
        const float QF = TF[0] * ti[0] + TF[1] * ti[1] + TF[2] * ti[2];
        double v[3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
          v[a] = static_cast<double>((k == 0) ? pc.D1 * ti[a] * QF : gam * (TF[a] - eig * ti[a] * QF));
#pragma unroll
        for (int a = 0; a < 3; ++a) br[3 * k + a] -= v[a];
        if constexpr (!kReadBack) {
          if (x0 != nullptr) {
            const double* x = x0 + static_cast<int64_t>(ROWS) * j2;
            double* ar = ared[p2];
            if (k == 0) {
              const float* th = Pj + RP + PAIRS + p2 * N;  // Theta_0
              double s0 = ar[0];
              for (int m = 0; m < N; ++m)
                for (int u = 0; u < 3; ++u) {
                  const float q0 = th[sym_index(0, u) * CB + m] * ti[0] + th[sym_index(1, u) * CB + m] * ti[1] +
                                   th[sym_index(2, u) * CB + m] * ti[2];
                  s0 = fma(static_cast<double>(q0), x[3 * m + u], s0);
                }
              ar[0] = s0;
            } else {
              double* U = ar + 1 + 3 * (k - 1);
              for (int m = 0; m < N; ++m) {
                const float* q = Pj + (k + 1) * RP + PAIRS + p2 * N + m;
                const double xx = q[0], yy = q[CB], zz = q[2 * CB], xy = q[3 * CB], xz = q[4 * CB], yz = q[5 * CB];
                const double xa = x[3 * m], xb = x[3 * m + 1], xc = x[3 * m + 2];
                U[0] = fma(xx, xa, fma(xy, xb, fma(xz, xc, U[0])));
                U[1] = fma(xy, xa, fma(yy, xb, fma(yz, xc, U[1])));
                U[2] = fma(xz, xa, fma(yz, xb, fma(zz, xc, U[2])));
              }
            }
          }
        }
      } else {
        float TV[3], T1[3];
        proj(0, TV);
        proj(1, T1);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          br[ROWS + a] += static_cast<double>(TV[a]);
          br[ROWS + 3 + a] += static_cast<double>(T1[a]);
        }
      }
    }
  }
  __syncthreads();  // bred complete

  if (tid < ROWS) {
    double s = 0.0;
    for (int q = 0; q < PAIRS; ++q) s += bred[q][tid];
    bpart[static_cast<int64_t>(gy) * n + static_cast<int64_t>(ROWS) * i + tid] = s;
  } else if (cpart && tid < NR) {
    double s = 0.0;
    for (int q = 0; q < PAIRS; ++q) s += bred[q][tid];
    cpart[(static_cast<int64_t>(gy) * M + i) * 6 + (tid - ROWS)] = s;
  }

  // Serving: the suspension's fields are read only here, after the sweeps,
  // so that they hold no registers during them.
  if constexpr (SERVING) x0 = serving->x0;
  double out = 0.0;  // lane tid < ROWS: row tid of the off-diagonal product A x0
  const bool have_x = x0 != nullptr;
  if constexpr (!kReadBack) {
    if (have_x && tid < ROWS) {
      const int k = tid / 3, a = tid - 3 * k;
      auto sum = [&](int idx) {
        double t = 0.0;
        for (int q = 0; q < PAIRS; ++q) t += ared[q][idx];
        return t;
      };
      if (k == 0) {
        out = static_cast<double>(pc.D1) * tid_[a] * sum(0);
      } else {
        const double U[3] = {sum(1 + 3 * (k - 1)), sum(2 + 3 * (k - 1)), sum(3 + 3 * (k - 1))};
        const double tU = tid_[0] * U[0] + tid_[1] * U[1] + tid_[2] * U[2];
        out = static_cast<double>(modes[k]) * (U[a] - static_cast<double>(modes[kMaxTerms + k]) * tid_[a] * tU);
      }
      if (apart) apart[static_cast<int64_t>(gy) * n + static_cast<int64_t>(ROWS) * i + tid] = out;
    }
    return;
  }
  // The workgroup reads back the rows it stored (visible to it after the
  // barrier above): for the product with x0, and for the FP16 copy, which
  // converts them with the block scales the sweeps stored (the values the
  // sweeps wrote, so the copy is theirs bit for bit; the self pair's columns
  // are zero already).
  double acc[NACC];
#pragma unroll
  for (int a = 0; a < NACC; ++a) acc[a] = 0.0;
  if (have_x || HALF) {
    // column (i-row block, e): s0 += Q0 . x_e, U_k += Theta_k x_e
    auto add_column = [&](const float* q, double xa, double xb, double xc) {
      acc[0] = fma(static_cast<double>(q[0]), xa,
                   fma(static_cast<double>(q[Lp]), xb, fma(static_cast<double>(q[2 * Lp]), xc, acc[0])));
#pragma unroll
      for (int k = 1; k < N; ++k) {
        const float* qk = q + (3 + 6 * (k - 1)) * Lp;
        const double txx = qk[0], tyy = qk[Lp], tzz = qk[2 * Lp], txy = qk[3 * Lp], txz = qk[4 * Lp],
                     tyz = qk[5 * Lp];
        double* u = acc + 1 + 3 * (k - 1);
        u[0] = fma(txx, xa, fma(txy, xb, fma(txz, xc, u[0])));
        u[1] = fma(txy, xa, fma(tyy, xb, fma(tyz, xc, u[1])));
        u[2] = fma(txz, xa, fma(tyz, xb, fma(tzz, xc, u[2])));
      }
    };
    // Pairs of consecutive columns per lane with 8-byte loads (the group's
    // first column jb N is even -- jgroup is a multiple of the sources per
    // sweep, a multiple of 4 -- and Lp a multiple of 64, so the loads are
    // aligned), then the remaining column one per lane.
    const int ebeg = jb * N, eend = je * N;
    const int efull = ebeg + (eend - ebeg) / 2 * 2;
    // FP16 copy: the inverse of column e's block scale (1 / sv exactly, sv a
    // power of two; 0 for a zero or non-finite scale, as half_block_scale)
    _Float16* const Hi = HALF ? T16 + static_cast<int64_t>(i) * NC * Lp : nullptr;
    auto inv_scale = [&](int e) {
      const unsigned es = (__float_as_uint(S16[static_cast<int64_t>(i) * M + e / N]) >> 23) & 0xffu;
      return (es >= 1u && es < 255u) ? __uint_as_float((254u - es) << 23) : 0.0f;
    };
    for (int e0 = ebeg + 2 * tid; e0 < efull; e0 += 2 * kPairThreads) {
      const float* q = Ti + e0;
      auto ld = [&](int comp) { return *reinterpret_cast<const floatx2*>(q + static_cast<int64_t>(comp) * Lp); };
      if constexpr (HALF) {
        typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
        const float iv0 = inv_scale(e0), iv1 = inv_scale(e0 + 1);
#pragma unroll
        for (int comp = 0; comp < NC; ++comp) {
          const floatx2 v = ld(comp);
          halfx2 h;
          h[0] = static_cast<_Float16>(v[0] * iv0);
          h[1] = static_cast<_Float16>(v[1] * iv1);
          *reinterpret_cast<halfx2*>(Hi + static_cast<int64_t>(comp) * Lp + e0) = h;
        }
        if (!have_x) continue;
      }
      double xv[2][3];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int a = 0; a < 3; ++a) xv[c][a] = x0[3 * static_cast<int64_t>(e0 + c) + a];
      {
        const floatx2 q0 = ld(0), q1 = ld(1), q2 = ld(2);
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[0] = fma(static_cast<double>(q0[c]), xv[c][0],
                       fma(static_cast<double>(q1[c]), xv[c][1], fma(static_cast<double>(q2[c]), xv[c][2], acc[0])));
      }
#pragma unroll
      for (int k = 1; k < N; ++k) {
        const int base = 3 + 6 * (k - 1);
        const floatx2 vxx = ld(base), vyy = ld(base + 1), vzz = ld(base + 2), vxy = ld(base + 3),
                      vxz = ld(base + 4), vyz = ld(base + 5);
        double* u = acc + 1 + 3 * (k - 1);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const double txx = vxx[c], tyy = vyy[c], tzz = vzz[c], txy = vxy[c], txz = vxz[c], tyz = vyz[c];
          const double xa = xv[c][0], xb = xv[c][1], xc = xv[c][2];
          u[0] = fma(txx, xa, fma(txy, xb, fma(txz, xc, u[0])));
          u[1] = fma(txy, xa, fma(tyy, xb, fma(tyz, xc, u[1])));
          u[2] = fma(txz, xa, fma(tyz, xb, fma(tzz, xc, u[2])));
        }
      }
    }
    for (int e = efull + tid; e < eend; e += kPairThreads) {
      if constexpr (HALF) {
        const float iv = inv_scale(e);
#pragma unroll
        for (int comp = 0; comp < NC; ++comp)
          Hi[static_cast<int64_t>(comp) * Lp + e] = static_cast<_Float16>(Ti[static_cast<int64_t>(comp) * Lp + e] * iv);
      }
      if (have_x)
        add_column(Ti + e, x0[3 * static_cast<int64_t>(e)], x0[3 * static_cast<int64_t>(e) + 1],
                   x0[3 * static_cast<int64_t>(e) + 2]);
    }
  }
  if (have_x) {  // uniform over the workgroup: the barrier below is reached by all or none
    constexpr int WAVES = kPairThreads / 64;
    static_assert(WAVES * NACC * sizeof(double) <= RP * Q * sizeof(float), "partials fit the freed G");
    double* red = reinterpret_cast<double*>(G);  // G is free after the last sweep
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int a = 0; a < NACC; ++a) {
      double v = acc[a];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
      if (lane == 0) red[wave * NACC + a] = v;
    }
    __syncthreads();
    if (tid < ROWS) {
      const int k = tid / 3, a = tid - 3 * k;
      auto sum = [&](int idx) {
        double t = 0.0;
        for (int w = 0; w < WAVES; ++w) t += red[w * NACC + idx];
        return t;
      };
      if (k == 0) {
        out = static_cast<double>(pc.D1) * tid_[a] * sum(0);
      } else {
        const double U[3] = {sum(1 + 3 * (k - 1)), sum(2 + 3 * (k - 1)), sum(3 + 3 * (k - 1))};
        const double tU = tid_[0] * U[0] + tid_[1] * U[1] + tid_[2] * U[2];
        out = static_cast<double>(pc.gamma[k]) * (U[a] - static_cast<double>(pc.eigen[k]) * tid_[a] * tU);
      }
      if (apart) apart[static_cast<int64_t>(gy) * n + static_cast<int64_t>(ROWS) * i + tid] = out;
    }
  }
  // Serving (all sources in this workgroup, b written directly): the first
  // residual r0 = b - (x0 + A_offdiag x0) (r0 = b without x0) into V_0 and
  // the target's squared norms of b and r0 into npart[2 i], npart[2 i + 1].
  if constexpr (SERVING) {
    static_assert(2 * ROWS * sizeof(double) <= NM * RP * sizeof(float), "norm partials fit the freed Pj");
    double* nred = reinterpret_cast<double*>(Pj);  // Pj is free after the last sweep
    if (tid < ROWS) {
      double sb = 0.0;
      for (int q = 0; q < PAIRS; ++q) sb += bred[q][tid];  // this row of b, as stored above
      const int64_t row = static_cast<int64_t>(ROWS) * i + tid;
      const double r = (x0 != nullptr) ? sb - (out + x0[row]) : sb;
      serving->V[row] = r;
      nred[tid] = sb * sb;
      nred[ROWS + tid] = r * r;
    }
    __syncthreads();
    if (tid == 0) {
      double b2 = 0.0, r2 = 0.0;
      for (int t = 0; t < ROWS; ++t) {
        b2 += nred[t];
        r2 += nred[ROWS + t];
      }
      serving->npart[2 * i] = b2;
      serving->npart[2 * i + 1] = r2;
    }
  }
}

}  // namespace rf
