// rf_assemble.hip -- assembly of the dense fiber-fiber system A x = b.
//
// Reference: fortran/assemble_matrix.incl:1-161 (block formulas),
// fortran/compute_inner_integral_numerically.incl:1-40 and
// fortran/compute_inner_integral_analytically.incl:1-338 (inner integrals),
// src/kernels/assemble_system_2D.cu:8-367 (the GPU layout of the same system).
//
// Work decomposition.  One workgroup = PAIRS consecutive target fibers i times
// Q target nodes q_i (192 lanes), looping over a group of source fibers j.
//   phase 1  lane (i, q_i) forms G_m(q_i) = sum_{q_j} w P_m(s_{q_j}) K(X_i(q_i) - X_j(q_j))
//            for all modes m = 0..N at once (the reference recomputes K for each
//            source mode), pairing q_j with its mirror -s_{q_j} so even modes use
//            K(q) + K(-q) and odd modes K(q) - K(-q).  Analytical mode forms the
//            same G_m exactly from FP64 moments, once per (i, j, q_i) for all m.
//   phase 2  jobs (i, m, column b) read G_m(.)[(a,b)] from LDS, project over q_i
//            (Theta_{k_i} = sum_{q_i} w P_{k_i+1}(s_{q_i}) G) and write the
//            15-row column segment of A; jobs (i, m = 0) accumulate the RHS.
// A is column-major with leading dimension lda; the workgroup's 8 target
// fibers own 8*15 consecutive rows, so each column segment it writes is
// contiguous.  Diagonal blocks are written as the identity, so A needs no
// memset.  RHS partial sums go to bpart[group][row] (FP64), summed afterwards
// in a fixed order: no atomics, bitwise reproducible.
#include "rf_theta.h"

namespace rf {

template <int N, int NQI, bool ANALYTIC>
__global__ __launch_bounds__(kPairThreads) void assemble_kernel(int M, int64_t lda, const double* __restrict__ pos,
                                                                const double* __restrict__ ori,
                                                                float* __restrict__ A, double* __restrict__ bpart,
                                                                int jgroup, PhysConsts pc, int jfirst, int jend) {
  constexpr Quad<N, NQI> quad{};
  constexpr int Q = 3 * NQI;
  constexpr int PAIRS = kPairThreads / Q;
  constexpr int NM = N + 1;
  constexpr int ROWS = 3 * N;
  static_assert(kPairThreads % Q == 0, "Q must divide the workgroup");
  static_assert(Q % 2 == 0, "mirror pairing needs an even node count");

  __shared__ float lds[PAIRS][NM][6][Q];
  __shared__ float ti_lds[PAIRS][3];

  const int tid = threadIdx.x;
  const int p = tid / Q;
  const int qi = tid - p * Q;
  const int i = blockIdx.x * PAIRS + p;
  const bool ivalid = i < M;
  const int j0 = jfirst + blockIdx.y * jgroup;
  const int j1 = min(jend, j0 + jgroup);
  const int64_t n = static_cast<int64_t>(ROWS) * M;

  double xi[3] = {0, 0, 0}, tid_[3] = {0, 0, 0};
  if (ivalid) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      xi[a] = pos[3 * i + a];
      tid_[a] = ori[3 * i + a];
    }
  }
  if (qi == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) ti_lds[p][a] = static_cast<float>(tid_[a]);
  }
  const double sq_d = node_fp64<NQI>(qi);
  const float sq = static_cast<float>(sq_d);
  const float ti[3] = {static_cast<float>(tid_[0]), static_cast<float>(tid_[1]), static_cast<float>(tid_[2])};

  // RHS accumulators of the jobs (i, m = 0); thread tid < PAIRS owns pair tid.
  double bacc[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) bacc[r] = 0.0;

  constexpr int kJobs = PAIRS * (3 * N + 1);

  for (int j = j0; j < j1; ++j) {
    // ---------------- phase 1: inner integrals G_m(q_i) ----------------
    if (ivalid && i != j) {
      const double xj0 = pos[3 * j + 0], xj1 = pos[3 * j + 1], xj2 = pos[3 * j + 2];
      const double tj0 = ori[3 * j + 0], tj1 = ori[3 * j + 1], tj2 = ori[3 * j + 2];
      float acc[NM][6];
      inner_integrals<N, NQI, ANALYTIC>(xi, tid_, ti, sq_d, sq, xj0, xj1, xj2, tj0, tj1, tj2, pc, acc);
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int c = 0; c < 6; ++c) lds[p][m][c][qi] = acc[m][c];
    }
    __syncthreads();

    // ---------------- phase 2: projections and stores ----------------
    for (int job = tid; job < kJobs; job += kPairThreads) {
      int p2, m, bcol;
      if (job < PAIRS) {
        p2 = job;
        m = 0;
        bcol = 0;
      } else {
        const int jj = job - PAIRS;
        p2 = jj % PAIRS;
        const int rest = jj / PAIRS;
        m = 1 + rest / 3;
        bcol = rest - 3 * (rest / 3);
      }
      const int i2 = blockIdx.x * PAIRS + p2;
      if (i2 >= M) continue;
      const float t0 = ti_lds[p2][0], t1 = ti_lds[p2][1], t2 = ti_lds[p2][2];
      if (m == 0) {
        if (i2 == j) continue;
        // TF_{k_i} = sum_{q_i} w P_{k_i+1} (G_0(q_i) F/2)
        float TF[N][3];
#pragma unroll
        for (int k = 0; k < N; ++k) TF[k][0] = TF[k][1] = TF[k][2] = 0.0f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const float g0 = lds[p2][0][0][q], g1 = lds[p2][0][1][q], g2 = lds[p2][0][2][q];
          const float g3 = lds[p2][0][3][q], g4 = lds[p2][0][4][q], g5 = lds[p2][0][5][q];
          const float f0 = g0 * pc.Fh[0] + g3 * pc.Fh[1] + g4 * pc.Fh[2];
          const float f1 = g3 * pc.Fh[0] + g1 * pc.Fh[1] + g5 * pc.Fh[2];
          const float f2 = g4 * pc.Fh[0] + g5 * pc.Fh[1] + g2 * pc.Fh[2];
#pragma unroll
          for (int k = 0; k < N; ++k) {
            TF[k][0] = fmaf(quad.W[k + 1][q], f0, TF[k][0]);
            TF[k][1] = fmaf(quad.W[k + 1][q], f1, TF[k][1]);
            TF[k][2] = fmaf(quad.W[k + 1][q], f2, TF[k][2]);
          }
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const float QF = TF[k][0] * t0 + TF[k][1] * t1 + TF[k][2] * t2;
          const float tt[3] = {t0, t1, t2};
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const float v = (k == 0) ? pc.D1 * tt[a] * QF : pc.gamma[k] * (TF[k][a] - pc.eigen[k] * tt[a] * QF);
            bacc[3 * k + a] -= static_cast<double>(v);
          }
        }
        continue;
      }
      const int kj = m - 1;
      const int64_t col = static_cast<int64_t>(ROWS) * (j - jfirst) + 3 * kj + bcol;
      float* out = A + col * lda + static_cast<int64_t>(ROWS) * i2;
      if (i2 == j) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) out[r] = (r == 3 * kj + bcol) ? 1.0f : 0.0f;
        continue;
      }
      // Theta_{k_i}[(a, bcol)] for a = 0..2
      const int c0 = sym_index(0, bcol), c1 = sym_index(1, bcol), c2 = sym_index(2, bcol);
      float T[N][3];
#pragma unroll
      for (int k = 0; k < N; ++k) T[k][0] = T[k][1] = T[k][2] = 0.0f;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const float g0 = lds[p2][m][c0][q], g1 = lds[p2][m][c1][q], g2 = lds[p2][m][c2][q];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          T[k][0] = fmaf(quad.W[k + 1][q], g0, T[k][0]);
          T[k][1] = fmaf(quad.W[k + 1][q], g1, T[k][1]);
          T[k][2] = fmaf(quad.W[k + 1][q], g2, T[k][2]);
        }
      }
      const float tt[3] = {t0, t1, t2};
#pragma unroll
      for (int k = 0; k < N; ++k) {
        // (Theta t_i)_bcol, Theta symmetric
        const float Qb = T[k][0] * t0 + T[k][1] * t1 + T[k][2] * t2;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const float v = (k == 0) ? pc.D1 * tt[a] * Qb : pc.gamma[k] * (T[k][a] - pc.eigen[k] * tt[a] * Qb);
          out[3 * k + a] = v;
        }
      }
    }
    __syncthreads();
  }

  if (tid < PAIRS && bpart != nullptr) {
    const int i2 = blockIdx.x * PAIRS + tid;
    if (i2 < M) {
      double* dst = bpart + static_cast<int64_t>(blockIdx.y) * n + static_cast<int64_t>(ROWS) * i2;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) dst[r] = bacc[r];
    }
  }
}

// ---------------------------------------------------------------------------
// Theta form (rf_theta.h).

template <int N, int NQI, bool ANALYTIC, bool HALF>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(
    theta_min_waves<N, NQI, ANALYTIC>(HALF ? 0 : kProductBytes<N, NQI>), 8))) void assemble_theta_kernel(
    int M, int64_t Lp, const double* __restrict__ pos, const double* __restrict__ ori, float* __restrict__ T,
    double* __restrict__ bpart, int jgroup, PhysConsts pc, float* __restrict__ Tv, double* __restrict__ cpart,
    const double* __restrict__ x0, double* __restrict__ apart, _Float16* __restrict__ T16, float* __restrict__ S16) {
  assemble_theta_block<N, NQI, ANALYTIC, HALF, false>(blockIdx.x, blockIdx.y, M, Lp, pos, ori, T, bpart, jgroup, pc,
                                                      Tv, cpart, x0, apart, T16, S16, nullptr);
}

// Dense A (column-major, leading dimension n) from the theta form; identity
// diagonal blocks.  One lane per (i, j, k_j).  Only the columns of source
// fibers j0 .. j0 + jcount - 1 (all n rows) are written, the column of source
// fiber j0's first unknown at A[0].
template <int N>
__global__ void expand_theta_kernel(int M, int64_t Lp, const float* __restrict__ T, const double* __restrict__ ori,
                                    PhysConsts pc, int j0, int jcount, float* __restrict__ A) {
  constexpr int NC = 3 + 6 * (N - 1);
  constexpr int ROWS = 3 * N;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(M) * jcount * N;
  if (id >= total) return;
  const int kj = static_cast<int>(id % N);
  const int64_t ij = id / N;
  const int jl = static_cast<int>(ij % jcount), i = static_cast<int>(ij / jcount);
  const int j = j0 + jl;
  const int64_t n = static_cast<int64_t>(ROWS) * M;
  const int64_t e = static_cast<int64_t>(j) * N + kj;
  const float* Ti = T + static_cast<int64_t>(i) * NC * Lp;
  const float t[3] = {static_cast<float>(ori[3 * i]), static_cast<float>(ori[3 * i + 1]),
                      static_cast<float>(ori[3 * i + 2])};
  for (int b = 0; b < 3; ++b) {
    float* col = A + (static_cast<int64_t>(ROWS) * jl + 3 * kj + b) * n + static_cast<int64_t>(ROWS) * i;
    if (i == j) {
      for (int r = 0; r < ROWS; ++r) col[r] = (r == 3 * kj + b) ? 1.0f : 0.0f;
      continue;
    }
    const float q0 = Ti[b * Lp + e];
    for (int a = 0; a < 3; ++a) col[a] = pc.D1 * t[a] * q0;
    for (int k = 1; k < N; ++k) {
      const float* Tk = Ti + (3 + 6 * (k - 1)) * Lp + e;
      float th[3], tht[3];
      for (int a = 0; a < 3; ++a) th[a] = Tk[sym_index(a, b) * Lp];
      // (Theta t)_b
      float qb = 0.0f;
      for (int a = 0; a < 3; ++a) {
        tht[a] = Tk[sym_index(a, b) * Lp];
        qb += tht[a] * t[a];
      }
      for (int a = 0; a < 3; ++a) col[3 * k + a] = pc.gamma[k] * (th[a] - pc.eigen[k] * t[a] * qb);
    }
  }
}

PairGrid pair_grid(int M, int pairs_per_tile) {
  PairGrid g;
  g.tiles = (M + pairs_per_tile - 1) / pairs_per_tile;
  // aim at ~16 workgroups per CU over 256 CUs
  int groups = (4096 + g.tiles - 1) / g.tiles;
  if (groups > M) groups = M;
  if (groups < 1) groups = 1;
  g.jgroup = (M + groups - 1) / groups;
  g.groups = (M + g.jgroup - 1) / g.jgroup;
  return g;
}

// Grid of the near pairs: blockIdx.x = target fiber, blockIdx.y = group of
// source fibers (a multiple of the 8 / 16 / 4 sources one sweep covers).
PairGrid theta_grid(int M, int sources_per_iteration) {
  PairGrid g;
  g.tiles = M;
  int groups = (4096 + M - 1) / M;
  const int max_groups = (M + sources_per_iteration - 1) / sources_per_iteration;
  if (groups > max_groups) groups = max_groups;
  if (groups < 1) groups = 1;
  int jg = (M + groups - 1) / groups;
  jg = (jg + sources_per_iteration - 1) / sources_per_iteration * sources_per_iteration;
  g.jgroup = jg;
  g.groups = (M + jg - 1) / jg;
  return g;
}

int max_pair_groups(int M) {
  int best = 1;
  for (int pairs : {4, 8, 16}) {
    const PairGrid g = pair_grid(M, pairs);
    if (g.groups > best) best = g.groups;
    const int t = theta_grid(M, pairs).groups + far_grid(M).groups;
    if (t > best) best = t;
  }
  return best;
}

int64_t theta_stride(int M, int N) { return (static_cast<int64_t>(M) * N + 63) / 64 * 64; }

template <int N, int NQI, bool AN>
static hipError_t launch_asm_t(int M, int64_t lda, const double* pos, const double* ori, float* A, double* bpart,
                               const PhysConsts& pc, hipStream_t s, int j0, int jcount) {
  constexpr int PAIRS = kPairThreads / (3 * NQI);
  PairGrid g = pair_grid(M, PAIRS);
  if (bpart == nullptr) g.groups = (jcount + g.jgroup - 1) / g.jgroup;
  hipLaunchKernelGGL((assemble_kernel<N, NQI, AN>), dim3(g.tiles, g.groups), dim3(kPairThreads), 0, s, M, lda, pos,
                     ori, A, bpart, g.jgroup, pc, j0, j0 + jcount);
  return hipGetLastError();
}

template <int N, int NQI>
static hipError_t launch_asm_n(bool an, int M, int64_t lda, const double* pos, const double* ori, float* A,
                               double* bpart, const PhysConsts& pc, hipStream_t s, int j0, int jcount) {
  return an ? launch_asm_t<N, NQI, true>(M, lda, pos, ori, A, bpart, pc, s, j0, jcount)
            : launch_asm_t<N, NQI, false>(M, lda, pos, ori, A, bpart, pc, s, j0, jcount);
}

bool assemble_supported(int N, int NQI) { return N >= 1 && N <= kMaxTerms && (NQI == 4 || NQI == 8 || NQI == 16); }

#define RF_ASM_CASE(NN)                                                                      \
  case NN:                                                                                   \
    if (NQI == 4) return launch_asm_n<NN, 4>(analytical, M, lda, pos, ori, A, bpart, pc, s, j0, jcount); \
    if (NQI == 8) return launch_asm_n<NN, 8>(analytical, M, lda, pos, ori, A, bpart, pc, s, j0, jcount); \
    if (NQI == 16) return launch_asm_n<NN, 16>(analytical, M, lda, pos, ori, A, bpart, pc, s, j0, jcount); \
    return hipErrorInvalidValue;

static hipError_t launch_asm(int N, int NQI, bool analytical, int M, int64_t lda, const double* pos,
                             const double* ori, float* A, double* bpart, const PhysConsts& pc, hipStream_t s, int j0,
                             int jcount) {
  switch (N) {
    RF_ASM_CASE(1)
    RF_ASM_CASE(2)
    RF_ASM_CASE(3)
    RF_ASM_CASE(4)
    RF_ASM_CASE(5)
    RF_ASM_CASE(6)
    RF_ASM_CASE(7)
    RF_ASM_CASE(8)
    default:
      return hipErrorInvalidValue;
  }
}
#undef RF_ASM_CASE

hipError_t launch_assemble(int N, int NQI, bool analytical, int M, int64_t lda, const double* pos,
                           const double* ori, float* A, double* bpart, const PhysConsts& pc, hipStream_t s) {
  return launch_asm(N, NQI, analytical, M, lda, pos, ori, A, bpart, pc, s, 0, M);
}

hipError_t launch_assemble_columns(int N, int NQI, bool analytical, int M, int64_t lda, const double* pos,
                                   const double* ori, float* A, const PhysConsts& pc, hipStream_t s, int j0,
                                   int jcount) {
  if (j0 < 0 || jcount < 1 || j0 + jcount > M) return hipErrorInvalidValue;
  return launch_asm(N, NQI, analytical, M, lda, pos, ori, A, nullptr, pc, s, j0, jcount);
}

template <int N, int NQI, bool AN>
static hipError_t launch_theta_t(int M, int64_t Lp, const double* pos, const double* ori, float* T, double* bpart,
                                 float* Tv, double* cpart, const double* x0, double* apart, bool far,
                                 const PhysConsts& pc, hipStream_t s, int* groups, _Float16* T16, float* S16) {
  constexpr int PAIRS = kPairThreads / (3 * NQI);
  const PairGrid g = theta_grid(M, PAIRS);
  *groups = g.groups;
  if (far) {
    *groups += far_grid(M).groups;
    const hipError_t e =
        launch_assemble_far(N, NQI, AN, M, Lp, pos, ori, T, bpart, g.groups, Tv, cpart, x0, apart, pc, s, T16, S16);
    if (e != hipSuccess) return e;
    return launch_assemble_near(N, NQI, AN, M, Lp, pos, ori, T, bpart, g, Tv, cpart, x0, apart, pc, s, T16, S16);
  }
  const dim3 grid(M, g.groups), block(kPairThreads);
  if (T16)  // the FP16 copy of GMRES-IR (a separate instantiation: the plain kernel keeps its registers)
    hipLaunchKernelGGL((assemble_theta_kernel<N, NQI, AN, true>), grid, block, 0, s, M, Lp, pos, ori, T, bpart,
                       g.jgroup, pc, Tv, cpart, x0, apart, T16, S16);
  else
    hipLaunchKernelGGL((assemble_theta_kernel<N, NQI, AN, false>), grid, block, 0, s, M, Lp, pos, ori, T, bpart,
                       g.jgroup, pc, Tv, cpart, x0, apart, nullptr, nullptr);
  return hipGetLastError();
}

template <int N, int NQI>
static hipError_t launch_theta_n(bool an, int M, int64_t Lp, const double* pos, const double* ori, float* T,
                                 double* bpart, float* Tv, double* cpart, const double* x0, double* apart, bool far,
                                 const PhysConsts& pc, hipStream_t s, int* groups, _Float16* T16, float* S16) {
  return an ? launch_theta_t<N, NQI, true>(M, Lp, pos, ori, T, bpart, Tv, cpart, x0, apart, far, pc, s, groups, T16, S16)
            : launch_theta_t<N, NQI, false>(M, Lp, pos, ori, T, bpart, Tv, cpart, x0, apart, far, pc, s, groups, T16, S16);
}

#define RF_TH_CASE(NN)                                                                             \
  case NN:                                                                                         \
    if (NQI == 4) return launch_theta_n<NN, 4>(analytical, M, Lp, pos, ori, T, bpart, Tv, cpart, x0, apart, far, pc, s, groups, T16, S16); \
    if (NQI == 8) return launch_theta_n<NN, 8>(analytical, M, Lp, pos, ori, T, bpart, Tv, cpart, x0, apart, far, pc, s, groups, T16, S16); \
    if (NQI == 16) return launch_theta_n<NN, 16>(analytical, M, Lp, pos, ori, T, bpart, Tv, cpart, x0, apart, far, pc, s, groups, T16, S16); \
    return hipErrorInvalidValue;

hipError_t launch_assemble_theta(int N, int NQI, bool analytical, int M, int64_t Lp, const double* pos,
                                 const double* ori, float* T, double* bpart, float* Tv, double* cpart,
                                 const double* x0, double* apart, bool far, const PhysConsts& pc, hipStream_t s, int* groups,
                                 _Float16* T16, float* S16) {
  switch (N) {
    RF_TH_CASE(1)
    RF_TH_CASE(2)
    RF_TH_CASE(3)
    RF_TH_CASE(4)
    RF_TH_CASE(5)
    RF_TH_CASE(6)
    RF_TH_CASE(7)
    RF_TH_CASE(8)
    default:
      return hipErrorInvalidValue;
  }
}
#undef RF_TH_CASE

// The whole dense A from the theta form, for the LU's factor storage
// (leading dimension lda), with the arithmetic of expand_theta_kernel (the
// identity for i == j).  A workgroup takes TI = 256 / 3N targets x 32 entries
// (entry e: source j = e / N, mode k_j = e % N): it stages their 3 + 6(N-1)
// numbers in LDS, one 128-byte row per (target, component), then writes the
// tile's 96 columns 3 e + b, each a run of TI x 3N contiguous rows 3N i + r,
// one row per lane.
template <int N>
constexpr int exp_targets() { return 256 / (3 * N); }
constexpr int kExpEntries = 32;
constexpr int kExpRow = kExpEntries + 4;  // padded LDS row (16-byte aligned, banks spread)

template <int N>
__global__ __launch_bounds__(256) void expand_theta_dense_kernel(int M, int64_t Lp, const float* __restrict__ T,
                                                                 const double* __restrict__ ori, PhysConsts pc,
                                                                 float* __restrict__ A, int64_t lda) {
  constexpr int NC = 3 + 6 * (N - 1);
  constexpr int ROWS = 3 * N;
  constexpr int TI = exp_targets<N>();
  constexpr int TROWS = TI * ROWS;  // rows of a column in the tile, <= 256
  constexpr int kChunks = TI * NC * (kExpEntries / 4);  // 16-byte chunks of the tile
  constexpr int kPer = (kChunks + 255) / 256;           // per thread
  // the tile's rows, then rows for the last round's chunks past the tile
  __shared__ __align__(16) float Ts[kPer * 256 / (kExpEntries / 4) * kExpRow];
  const int tid = threadIdx.x;
  const int64_t L = static_cast<int64_t>(M) * N;
  // Tile order: workgroup w runs on XCD w % 8; each XCD takes a contiguous
  // run of tiles, target groups fastest, so the column runs that continue
  // each other (and share their first and last 128-byte lines) are written
  // one after another through the same L2.
  const int ny = (M + TI - 1) / TI;
  const int tiles = static_cast<int>((L + kExpEntries - 1) / kExpEntries) * ny;
  const int per = (tiles + 7) / 8;
  const int v = (static_cast<int>(blockIdx.x) & 7) * per + (static_cast<int>(blockIdx.x) >> 3);
  if (v >= tiles) return;  // uniform over the workgroup, before any barrier
  const int64_t e0 = static_cast<int64_t>(v / ny) * kExpEntries;
  const int i0 = (v % ny) * TI;
  // stage: row (ti, c) holds T[i0 + ti][c][e0 .. e0 + 31] (within the padded
  // row of Lp >= e0 + 32 numbers).  Every load of the thread is in flight
  // before the LDS stores, which are unconditional (a guarded store would let
  // the compiler sink each load to it): chunks past the tile, and rows of
  // targets past M, load the tile's first chunk and store it where nothing
  // reads it.
  float4 sv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    int q = tid + 256 * u;
    int row = q / (kExpEntries / 4);
    if (q >= kChunks || i0 + row / NC >= M) q = 0, row = 0;
    const int part = q - row * (kExpEntries / 4);
    const int ti = row / NC, c = row - ti * NC;
    sv[u] = *reinterpret_cast<const float4*>(T + (static_cast<int64_t>(i0 + ti) * NC + c) * Lp + e0 + 4 * part);
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int q = tid + 256 * u;
    const int row = q / (kExpEntries / 4), part = q - row * (kExpEntries / 4);
    *reinterpret_cast<float4*>(&Ts[row * kExpRow + 4 * part]) = sv[u];
  }
  __syncthreads();
  if (tid >= TROWS) return;  // no barrier follows
  const int ti = tid / ROWS, r = tid - ti * ROWS;
  const int i = i0 + ti;
  if (i >= M) return;
  const int k = r / 3, a = r - 3 * k;
  const float t[3] = {static_cast<float>(ori[3 * i]), static_cast<float>(ori[3 * i + 1]),
                      static_cast<float>(ori[3 * i + 2])};
  float gk = 0.0f, ek = 0.0f;
#pragma unroll
  for (int kk = 1; kk < N; ++kk)
    if (k == kk) {
      gk = pc.gamma[kk];
      ek = pc.eigen[kk];
    }
  const float* Tr = Ts + ti * NC * kExpRow;  // this target's rows
  const int cbase = (k == 0) ? 0 : 3 + 6 * (k - 1);
  const int ecount = static_cast<int>(min(static_cast<int64_t>(kExpEntries), L - e0));
  float* const out = A + static_cast<int64_t>(ROWS) * i0 + tid;
  for (int ee = 0; ee < ecount; ++ee) {
    const int64_t e = e0 + ee;
    const int j = static_cast<int>(e / N), kj = static_cast<int>(e - static_cast<int64_t>(j) * N);
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      float v;
      if (i == j) {
        v = (r == 3 * kj + b) ? 1.0f : 0.0f;
      } else if (k == 0) {
        v = pc.D1 * t[a] * Tr[b * kExpRow + ee];
      } else {
        float qb = 0.0f;
#pragma unroll
        for (int a2 = 0; a2 < 3; ++a2) qb += Tr[(cbase + sym_index(a2, b)) * kExpRow + ee] * t[a2];
        v = gk * (Tr[(cbase + sym_index(a, b)) * kExpRow + ee] - ek * t[a] * qb);
      }
      out[(3 * e + b) * lda] = v;
    }
  }
}

hipError_t launch_expand_theta_dense(int N, int M, int64_t Lp, const float* T, const double* ori,
                                     const PhysConsts& pc, float* A, int64_t lda, hipStream_t s) {
  if (M < 1 || lda < static_cast<int64_t>(3) * N * M || Lp % kExpEntries != 0) return hipErrorInvalidValue;
  const int64_t ex = (static_cast<int64_t>(M) * N + kExpEntries - 1) / kExpEntries;
  switch (N) {
#define RF_EXD(NN)                                                                                          \
  case NN: {                                                                                                \
    const int64_t tiles = ex * ((M + exp_targets<NN>() - 1) / exp_targets<NN>());                          \
    if (tiles > INT32_MAX - 8) return hipErrorInvalidValue;                                                 \
    hipLaunchKernelGGL(expand_theta_dense_kernel<NN>, dim3(static_cast<unsigned>((tiles + 7) / 8 * 8)),     \
                       dim3(256), 0, s, M, Lp, T, ori, pc, A, lda);                                         \
    break;                                                                                                  \
  }
    RF_EXD(1)
    RF_EXD(2)
    RF_EXD(3)
    RF_EXD(4)
    RF_EXD(5)
    RF_EXD(6)
    RF_EXD(7)
    RF_EXD(8)
#undef RF_EXD
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_expand_theta(int N, int M, int64_t Lp, const float* T, const double* ori, const PhysConsts& pc,
                               float* A, hipStream_t s, int j0, int jcount) {
  if (jcount < 0) jcount = M - j0;
  if (j0 < 0 || jcount < 1 || j0 + jcount > M) return hipErrorInvalidValue;
  const int64_t total = static_cast<int64_t>(M) * jcount * N;
  const unsigned blocks = static_cast<unsigned>((total + 255) / 256);
  switch (N) {
#define RF_EX(NN) \
  case NN:        \
    hipLaunchKernelGGL(expand_theta_kernel<NN>, dim3(blocks), dim3(256), 0, s, M, Lp, T, ori, pc, j0, jcount, A); \
    break;
    RF_EX(1)
    RF_EX(2)
    RF_EX(3)
    RF_EX(4)
    RF_EX(5)
    RF_EX(6)
    RF_EX(7)
    RF_EX(8)
#undef RF_EX
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace rf
