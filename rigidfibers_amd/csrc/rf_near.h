// rf_near.h -- the near pairs of the theta form: of the assembly beside the far
// kernel (rf_near.hip), and the segments that the operator form stores
// (rf_operator.hip).
#pragma once

#include "rf_pairs.h"

namespace rf {

// The near pairs of one workgroup: target fiber i, source group gy (the far
// pairs, by far_class, are assemble_far_block's).  The workgroup scans its sources
// kScan at a time, lists the near ones in LDS in their order, and forms them PAIRS
// at a sweep:
//   phase 1  lane (p, q_i) writes G_m(q_i) of source slot p into LDS as row
//            r = c*CB + (m == 0 ? p : PAIRS + p*N + m-1) of a GEMM operand
//            (c = symmetric component; the mode-0 rows feed the RHS).
//   phase 2  lane r forms C[r][kk] = sum_q W[kk][q] G[r][q] (kk = 0..N: the
//            projections onto w P_kk) for all kk from the mirror sums
//            E = G(q) + G(-q) and differences O = G(q) - G(-q): the weights
//            satisfy W[kk][-q] = (-1)^kk W[kk][q] exactly, so even kk take E,
//            odd kk take O, and the table entries are immediate operands.
//   phase 3  each lane writes (source, mode) columns of the component arrays;
//            the k_i = 0 components (Theta_0 t_i), the RHS of each source slot
//            and, with x0, its share of the off-diagonal product A x0 (FP32
//            values times FP64 x0, FP64 sums) are formed here.
// The self pair's columns are zeroed.  HALF (GMRES-IR's FP16 copy T16, S16):
// phase 2 also takes each (target, source) block's largest |projection|,
// phase 3 stores the block scales and the scaled FP16 values.
// Beside the far kernel a target has few near sources (8 of 5000 in a ball at 0.028
// fibers per unit volume, about 20 at 0.1), so the sweeps are few and the scan, one
// distance per source, is most of the launch.  SEGMENTS takes every source within
// the first radius (46 and about 180 there).
template <int N, int NQI, bool ANALYTIC, bool HALF = false, bool SEGMENTS = false>
__device__ __forceinline__ void assemble_near_block(int i, int gy, int M, int64_t Lp, const double* __restrict__ pos,
                                                    const double* __restrict__ ori, float* __restrict__ T,
                                                    double* __restrict__ bpart, int jgroup, const PhysConsts& pc,
                                                    float* __restrict__ Tv, double* __restrict__ cpart,
                                                    const double* __restrict__ x0, double* __restrict__ apart,
                                                    _Float16* __restrict__ T16 = nullptr,
                                                    float* __restrict__ S16 = nullptr,
                                                    const SusDev* __restrict__ serving = nullptr,
                                                    const NearStore* __restrict__ store = nullptr) {
  constexpr Quad<N, NQI> quad{};
  constexpr FarRule rule = far_rule(N, NQI);
  constexpr int Q = 3 * NQI;
  constexpr int PAIRS = kPairThreads / Q;
  constexpr int NM = N + 1;
  constexpr int ROWS = 3 * N;
  constexpr int NC = 3 + 6 * (N - 1);
  constexpr int NR = ROWS + 6;  // RHS rows + the two velocity constants
  constexpr int NACC = 1 + 3 * (N - 1);  // s0 = Q0 . x0, then U_k = Theta_k x0 (k >= 1)
  constexpr int PN = PAIRS * N;  // (source, mode) columns of one sweep
  constexpr int CB = PAIRS + PN;  // GEMM rows per component
  constexpr int RP = 6 * CB;  // GEMM rows
  constexpr int WAVES = kPairThreads / 64;
  constexpr int kPer = 2, kScan = kPer * kPairThreads;  // sources per scan
  static_assert(kPairThreads % Q == 0 && Q % 2 == 0 && PAIRS % 4 == 0, "sweep shapes");

  __shared__ __align__(16) float G[RP * Q];
  __shared__ __align__(16) float Pj[NM * RP];
  __shared__ double bred[PAIRS][NR];
  __shared__ double ared[PAIRS][NACC];
  __shared__ float modes[2 * kMaxTerms];  // gamma_k, then eigen_k
  __shared__ unsigned smax[PAIRS];  // FP16 copy: each source slot's largest |projection| (float bits)
  __shared__ int nlist[kScan + PAIRS];
  __shared__ int ncount[kPer][WAVES];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int p = tid / Q;
  const int qi = tid - p * Q;
  const int jb = gy * jgroup;
  const int je = min(M, jb + jgroup);
  const int64_t n = static_cast<int64_t>(ROWS) * M;

  const double xi[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
  const double tid_[3] = {ori[3 * i], ori[3 * i + 1], ori[3 * i + 2]};
  const float ti[3] = {static_cast<float>(tid_[0]), static_cast<float>(tid_[1]), static_cast<float>(tid_[2])};
  const double ti2 = fma(tid_[2], tid_[2], fma(tid_[1], tid_[1], tid_[0] * tid_[0]));
  const double sq_d = node_fp64<NQI>(qi);
  const float sq = static_cast<float>(sq_d);
  float* Ti = SEGMENTS ? nullptr : T + static_cast<int64_t>(i) * NC * Lp;
  float* Vi = Tv ? Tv + static_cast<int64_t>(i) * 12 * Lp : nullptr;
  _Float16* const Hi = HALF ? T16 + static_cast<int64_t>(i) * NC * Lp : nullptr;
  if (serving != nullptr) x0 = serving->x0;
  uint32_t lp32 = static_cast<uint32_t>(Lp);
  auto is_near = [&](int j) {
    if (j >= je || j == i) return false;
    const double t0 = ori[3 * j], t1 = ori[3 * j + 1], t2 = ori[3 * j + 2];
    const int c = far_class(rule, xi[0] - pos[3 * j], xi[1] - pos[3 * j + 1], xi[2] - pos[3 * j + 2], ti2,
                            fma(t2, t2, fma(t1, t1, t0 * t0)));
    return SEGMENTS ? c != 0 : c < 0;
  };
  // The target's segment: counted, then taken from the store.  Where it starts
  // depends on the order the workgroups come in, what it holds does not.
  int* seg = nullptr;  // its sources
  int formed = 0;      // pairs of the segment formed so far
  if constexpr (SEGMENTS) {
    __shared__ long long seg_base;
    int mine = 0;
    for (int j = jb + tid; j < je; j += kPairThreads) mine += is_near(j) ? 1 : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
    if (lane == 0) ncount[0][wave] = mine;
    __syncthreads();
    int cnt = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) cnt += ncount[0][w];
    lp32 = static_cast<uint32_t>(near_stride(cnt, N));
    if (tid < 3) {
      store->pos[3 * i + tid] = pos[3 * i + tid];
      store->ori[3 * i + tid] = ori[3 * i + tid];
    }
    if (tid == 0) {
      const int64_t size = near_ints(cnt) + static_cast<int64_t>(NC + (store->velocity ? 12 : 0)) * lp32;
      const int64_t at = static_cast<int64_t>(atomicAdd(store->used, static_cast<unsigned long long>(size)));
      seg_base = at + size <= store->capacity ? at : -1;
      store->base[i] = seg_base;
      store->count[i] = cnt;
    }
    __syncthreads();
    if (seg_base < 0) return;  // no room: the host takes more and repeats the launch
    seg = reinterpret_cast<int*>(store->data + seg_base);
    Ti = store->data + seg_base + near_ints(cnt);
    Vi = store->velocity ? Ti + static_cast<int64_t>(NC) * lp32 : nullptr;
  }

  // RHS (and velocity-constant) and product sums of each source slot, kept in
  // LDS; the mode factors gamma_k, eigen_k as a table the lanes index by k
  for (int r = tid; r < PAIRS * NR; r += kPairThreads) bred[r / NR][r % NR] = 0.0;
  for (int r = tid; r < PAIRS * NACC; r += kPairThreads) ared[r / NACC][r % NACC] = 0.0;
#pragma unroll
  for (int t = 0; t < kMaxTerms; ++t)
    if (tid == t) {
      modes[t] = pc.gamma[t];
      modes[kMaxTerms + t] = pc.eigen[t];
    }
  // the self pair
  if (!SEGMENTS && i >= jb && i < je) {
    const uint32_t col = static_cast<uint32_t>(i) * N;
    for (int r = tid; r < NC * N; r += kPairThreads) {
      const uint32_t u = r / N, k = r - (r / N) * N;
      Ti[u * lp32 + col + k] = 0.0f;
      if constexpr (HALF) Hi[u * lp32 + col + k] = static_cast<_Float16>(0.0f);
    }
    if (Vi)
      for (int r = tid; r < 12 * N; r += kPairThreads) {
        const uint32_t u = r / N, k = r - (r / N) * N;
        Vi[u * lp32 + col + k] = 0.0f;
      }
    if constexpr (HALF) {
      if (tid == 0) S16[static_cast<int64_t>(i) * M + i] = 0.0f;
    }
  }

  int pend = 0;  // near sources listed and not yet formed
  for (int js = jb;; js += kScan) {
    const bool last = js + kScan >= je;
    bool near[kPer];
    int before[kPer];
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
      near[t] = is_near(js + t * kPairThreads + tid);
      const unsigned long long mask = __ballot(near[t]);
      before[t] = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                            __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u));
      if (lane == 0) ncount[t][wave] = __popcll(mask);
    }
    // every lane is past the last sweep's reads of nlist here, and past the
    // set-up above the first time
    __syncthreads();
    int found = 0;
#pragma unroll
    for (int t = 0; t < kPer; ++t)
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        if (w == wave && near[t]) nlist[pend + found + before[t]] = js + t * kPairThreads + tid;
        found += ncount[t][w];
      }
    pend += found;
    __syncthreads();
    while (pend >= PAIRS || (last && pend > 0)) {
      const int take = min(pend, PAIRS);
      pend -= take;
      const int* const js_ = nlist + pend;  // this sweep's sources
      // first column of source slot q
      auto col0 = [&](int q) { return SEGMENTS ? (formed + q) * N : js_[q] * N; };
      if constexpr (SEGMENTS) {
        if (tid < take) seg[formed + tid] = js_[tid];
      }
      if (tid < PAIRS) smax[tid] = 0u;
      if (p < take) {
        const int j = js_[p];
        float acc[NM][6] = {};
        // i itself is never listed: without this test the compiler's schedule of the
        // exact integrals is slower (segments at M = 5000: 437 us, with it 391)
        if (j != i)
          inner_integrals<N, NQI, ANALYTIC>(xi, tid_, ti, sq_d, sq, pos[3 * j], pos[3 * j + 1], pos[3 * j + 2],
                                            ori[3 * j], ori[3 * j + 1], ori[3 * j + 2], pc, acc);
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int c = 0; c < 6; ++c) G[(c * CB + (m == 0 ? p : PAIRS + p * N + m - 1)) * Q + qi] = acc[m][c];
      }
      __syncthreads();
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
          if (e >= PAIRS) atomicMax(&smax[(e - PAIRS) / N], __float_as_uint(g));
        }
      }
      __syncthreads();
      if constexpr (HALF) {
        if (tid < take) {
          float sv, iv;
          half_block_scale(smax[tid], sv, iv);
          S16[static_cast<int64_t>(i) * M + js_[tid]] = sv;
        }
      }
      // system components: u < 3 Q0_u = (Theta_0 t_i)_u (Theta_0 = the P_1
      // projection), then Theta_{k_i} for k_i = 1..N-1 (projection k_i + 1)
      auto sys_val = [&](int u, int pm) {
        if (u < 3) {
          const float* b1 = Pj + RP + PAIRS + pm;
          return b1[sym_index(0, u) * CB] * ti[0] + b1[sym_index(1, u) * CB] * ti[1] + b1[sym_index(2, u) * CB] * ti[2];
        }
        const int kk = 2 + (u - 3) / 6;
        const int c = (u - 3) - 6 * (kk - 2);
        return Pj[kk * RP + c * CB + PAIRS + pm];
      };
      for (int job = tid; job < NC * PN; job += kPairThreads) {
        const int u = job / PN, pm = job - u * PN, s = pm / N;
        if (s >= take) continue;
        const float val = sys_val(u, pm);
        const uint32_t at = static_cast<uint32_t>(u) * lp32 + static_cast<uint32_t>(col0(s) + (pm - s * N));
        Ti[at] = val;
        if constexpr (HALF) {
          float sv, iv;
          half_block_scale(smax[s], sv, iv);
          Hi[at] = static_cast<_Float16>(val * iv);
        }
      }
      // velocity operator: Theta_0 (projection 1), then Phi_0 (projection 0)
      if (Vi) {
        for (int job = tid; job < 12 * PN; job += kPairThreads) {
          const int w = job / PN, pm = job - w * PN, s = pm / N;
          if (s >= take) continue;
          const int kk = w < 6 ? 1 : 0;
          const int c = w < 6 ? w : w - 6;
          Vi[static_cast<uint32_t>(w) * lp32 + static_cast<uint32_t>(col0(s) + (pm - s * N))] =
              Pj[kk * RP + c * CB + PAIRS + pm];
        }
      }
      // RHS (source slot p2, row block k): k < N forms rows 3k..3k+2 of b from
      // the projection of G_0 F/2 onto w P_{k+1}; k = N the velocity constants
      // sum_q w G_0 F/2 and sum_q w P_1 G_0 F/2.  Row block k < N of A x0 too.
      for (int rj = tid; rj < PAIRS * (N + 1); rj += kPairThreads) {
        const int p2 = rj / (N + 1), k = rj - p2 * (N + 1);
        if (p2 >= take) continue;
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
          if (x0 != nullptr) {
            const double* x = x0 + static_cast<int64_t>(ROWS) * js_[p2];
            double* ar = ared[p2];
            if (k == 0) {
              double s0 = ar[0];
              for (int m = 0; m < N; ++m)
                for (int u = 0; u < 3; ++u) s0 = fma(static_cast<double>(sys_val(u, p2 * N + m)), x[3 * m + u], s0);
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
      __syncthreads();  // the sweep's LDS is free
      if constexpr (SEGMENTS) formed += take;
    }
    if (last) break;
  }

  // Row tid of b, of the off-diagonal product A x0, and the velocity constants:
  // the slots' sums in order.  Serving adds the far pairs' sums, which the far
  // kernel left in b, cpart and V_0.
  auto slots = [&](const double* first, int stride) {
    double s = 0.0;
    for (int q = 0; q < PAIRS; ++q) s += first[q * stride];
    return s;
  };
  double sb = 0.0, out = 0.0;
  const int64_t row = static_cast<int64_t>(ROWS) * i + tid;
  if (tid < ROWS) {
    sb = slots(&bred[0][tid], NR);
    if (x0 != nullptr) {
      const int k = tid / 3, a = tid - 3 * k;
      if (k == 0) {
        out = static_cast<double>(pc.D1) * tid_[a] * slots(&ared[0][0], NACC);
      } else {
        double U[3];
        for (int c = 0; c < 3; ++c) U[c] = slots(&ared[0][1 + 3 * (k - 1) + c], NACC);
        const double tU = tid_[0] * U[0] + tid_[1] * U[1] + tid_[2] * U[2];
        out = static_cast<double>(modes[k]) * (U[a] - static_cast<double>(modes[kMaxTerms + k]) * tid_[a] * tU);
      }
    }
    if (serving == nullptr) {
      bpart[static_cast<int64_t>(gy) * n + row] = sb;
      if (apart && x0 != nullptr) apart[static_cast<int64_t>(gy) * n + row] = out;
    } else {
      sb += bpart[row];
      bpart[row] = sb;
    }
  } else if (cpart && tid < NR) {
    double s = slots(&bred[0][tid], NR);
    double* c = cpart + (static_cast<int64_t>(gy) * M + i) * 6 + (tid - ROWS);
    if (serving != nullptr) s += *c;
    *c = s;
  }
  // Serving (all sources in this workgroup): the first residual r0 = b - (x0 +
  // A_offdiag x0) (r0 = b without x0) into V_0 and the target's squared norms
  // of b and r0 into npart[2 i], npart[2 i + 1].
  if (serving != nullptr) {
    static_assert(2 * ROWS * sizeof(double) <= NM * RP * sizeof(float), "norm partials fit the freed Pj");
    double* nred = reinterpret_cast<double*>(Pj);  // Pj is free after the last sweep
    double* const r0v = serving->V;
    if (tid < ROWS) {
      const double r = (x0 != nullptr) ? sb - ((out + r0v[row]) + x0[row]) : sb;
      r0v[row] = r;
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
