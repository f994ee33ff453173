// rf_operator.hip -- the system of a large suspension as an operator: products
// with A that form the far pairs' kernel values where they are used.
//
// Reference: fortran/assemble_matrix.incl:1-161 (the system), the product of
// fortran/solve_system.incl:36 and lib/viennacl/linalg/gmres.hpp; the velocity
// sums of fortran/update_velocities.incl:29-86.
//
// Stored in theta form the system is read once per product: 540 bytes per pair
// of fibers (N = 5), 13.5 GB and 2.05 ms at M = 5000, 6.6 TB/s.  A far pair
// (far_rule's first radius and beyond, rf_device.h) is the tensor rule on 6 x 6
// nodes, and its share of a product is
//   g_i(s_p) += sum_q K(x_i + s_p t_i - x_j - s_q t_j) f_j(s_q),
// f_j(s_q) = sum_m W_m(s_q) x_{j,m} formed once per source, the projections
// TF_k = sum_p W_k(s_p) g_i(s_p) once per target: 926 instructions of a lane
// per pair and no memory, 0.70 ms a product at M = 5000.  So far
// pairs are not stored at all, the assembly forms only the others (46 of 5000
// sources there, kept in theta form per target), and the right-hand side, the
// first residual and the velocities are the same sums.
//
// Precision as in the stored form: kernel values in FP32 from centre
// differences in FP64, everything they multiply and all sums in FP64.
#include "rf_near.h"

namespace rf {

constexpr int kOpThreads = 256;
constexpr int kOpWaves = kOpThreads / 64;
constexpr int kOpTile = 64;  // target fibers of a workgroup, one per lane

template <int N>
constexpr int op_nodes() { return far_rule(N, 8).np[0]; }

// Weights in FP64: the composite functional for 4, 8, 16 intervals and the
// exact integral's.
template <int N>
struct OpTables {
  static constexpr int NP = op_nodes<N>();
  FarWeights<N, NP, double> composite[3], exact;
  constexpr OpTables()
      : composite{FarWeights<N, NP, double>(4, false), FarWeights<N, NP, double>(8, false),
                  FarWeights<N, NP, double>(16, false)},
        exact(0, true) {}
};

// Node q of NP: +s_0, -s_0, +s_1, ...
__host__ __device__ constexpr double op_node(int NP, int q) { return (q & 1) ? -gl_node(NP, q >> 1) : gl_node(NP, q >> 1); }

// f_j(s_q) and s_q t_j . f_j(s_q) of every source node, 4 doubles each: of the
// density x (mode m of x is P_{m+1}), or without x of the force F/2 (P_0).
template <int N>
__global__ void op_nodes_kernel(int M, int variant, const double* __restrict__ ori, const double* __restrict__ x,
                                PhysConsts pc, double* __restrict__ nodes, const int* __restrict__ skip) {
  static constexpr OpTables<N> tab{};
  constexpr int NP = op_nodes<N>();
  if (skip != nullptr && *skip) return;
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= M * NP) return;
  const int j = id / NP, q = id - j * NP, h = q >> 1;
  const auto& src = (variant & 1) ? tab.exact : tab.composite[variant >> 1];
  double f[3];
  if (x == nullptr) {
#pragma unroll
    for (int a = 0; a < 3; ++a) f[a] = src.W[h][0] * pc.Fh_d[a];
  } else {
    f[0] = f[1] = f[2] = 0.0;
    const double* xj = x + 3 * static_cast<int64_t>(N) * j;
#pragma unroll
    for (int m = 1; m <= N; ++m) {
      const double w = ((m & 1) && (q & 1)) ? -src.W[h][m] : src.W[h][m];
#pragma unroll
      for (int a = 0; a < 3; ++a) f[a] = fma(w, xj[3 * (m - 1) + a], f[a]);
    }
  }
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < NP / 2; ++r)
    if (h == r) s = gl_node(NP, r);
  if (q & 1) s = -s;
  double* out = nodes + 4 * static_cast<int64_t>(id);
  out[0] = f[0];
  out[1] = f[1];
  out[2] = f[2];
  out[3] = s * fma(ori[3 * j], f[0], fma(ori[3 * j + 1], f[1], ori[3 * j + 2] * f[2]));
}

// g_i(s_p) over the sources of one group: lane = target fiber, the wavefront's
// source j the same in every lane, so its centre, direction and node densities
// come through scalar registers.  With R = b_p - s_q t_j (b_p = x_i + s_p t_i -
// x_j) and K f = a f + c (R . f) R, the sums over q are
//   sum a_q f_q + b_p sum h_q - t_j sum s_q h_q,   h_q = c_q (b_p . f_q - s_q t_j . f_q):
// two conversions and nine FP64 operations per kernel value, 926 instructions
// per pair of fibers in all, VALU instructions active in 98% of the cycles (counters;
// 0.64 ms at M = 5000).
// RHS = 2 sums two densities over the same kernel values (1.13 ms).  Tried:
// centre differences kept in FP64 up to r^2 (0.70 ms) and the reciprocal square
// root refined to FP64 (0.79 ms) left the system's error against FP64 where it
// was: the near pairs' FP32 sums set it.
template <int N, int RHS>
__global__ __launch_bounds__(kOpThreads) void op_far_kernel(int M, double r, const double* __restrict__ pos,
                                                            const double* __restrict__ ori,
                                                            const double* __restrict__ nodes0,
                                                            const double* __restrict__ nodes1,
                                                            double* __restrict__ part, int jgroup, PhysConsts pc,
                                                            const int* __restrict__ skip) {
  constexpr int NP = op_nodes<N>(), H = NP / 2;
  if (skip != nullptr && *skip) return;
  __shared__ double red[kOpWaves - 1][kOpTile][3 * NP + 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = blockIdx.x * kOpTile + lane;
  const int ii = min(i, M - 1);
  // the wavefront's sources
  const int sub = (jgroup + kOpWaves - 1) / kOpWaves;
  const int je = min(M, static_cast<int>(blockIdx.y + 1) * jgroup);
  const int jb = static_cast<int>(blockIdx.y) * jgroup + wave * sub;
  const int jw = min(je, jb + sub);

  double x[3], t[3], ti2 = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    x[a] = pos[3 * ii + a];
    t[a] = ori[3 * ii + a];
    ti2 = fma(t[a], t[a], ti2);
  }
  const float two_eps2 = 2.0f * pc.eps2, six_eps2 = 6.0f * pc.eps2;
  const double r2 = r * r;
  double g[RHS][NP][3];
#pragma unroll
  for (int q = 0; q < RHS; ++q)
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int a = 0; a < 3; ++a) g[q][p][a] = 0.0;

  for (int j = jb; j < jw; ++j) {
    const double tj[3] = {ori[3 * j], ori[3 * j + 1], ori[3 * j + 2]};
    const double tj2 = fma(tj[2], tj[2], fma(tj[1], tj[1], tj[0] * tj[0]));
    const double d[3] = {x[0] - pos[3 * j], x[1] - pos[3 * j + 1], x[2] - pos[3 * j + 2]};
    const double d2 = fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2]));
    // far_class == 0, in the same arithmetic
    if (!(j != ii && d2 >= r2 * fmax(1.0, fmax(ti2, tj2)))) continue;
    float u[H][3];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int a = 0; a < 3; ++a) u[h][a] = static_cast<float>(gl_node(NP, h)) * static_cast<float>(tj[a]);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      double b[3];
      float bf[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        b[a] = fma(op_node(NP, p), t[a], d[a]);
        bf[a] = static_cast<float>(b[a]);
      }
      double H0[RHS], H1[RHS];
#pragma unroll
      for (int q = 0; q < RHS; ++q) H0[q] = H1[q] = 0.0;
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        const int h = s >> 1;
        const float sg = (s & 1) ? 1.0f : -1.0f;
        const float rx = fmaf(sg, u[h][0], bf[0]), ry = fmaf(sg, u[h][1], bf[1]), rz = fmaf(sg, u[h][2], bf[2]);
        const float inv = __builtin_amdgcn_rsqf(fmaf(rx, rx, fmaf(ry, ry, rz * rz)));
        const float inv2 = inv * inv;
        const float inv3 = inv2 * inv;
        const double a = fmaf(two_eps2, inv3, inv);
        const double c = inv3 * fmaf(-six_eps2, inv2, 1.0f);
#pragma unroll
        for (int q = 0; q < RHS; ++q) {
          const double* f = (q == 0 ? nodes0 : nodes1) + 4 * (static_cast<int64_t>(j) * NP + s);
          const double hq = c * fma(b[0], f[0], fma(b[1], f[1], fma(b[2], f[2], -f[3])));
          g[q][p][0] = fma(a, f[0], g[q][p][0]);
          g[q][p][1] = fma(a, f[1], g[q][p][1]);
          g[q][p][2] = fma(a, f[2], g[q][p][2]);
          H0[q] += hq;
          H1[q] = fma(op_node(NP, s), hq, H1[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < RHS; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) g[q][p][a] = fma(b[a], H0[q], fma(-tj[a], H1[q], g[q][p][a]));
    }
  }

  // the wavefronts' sums in order; part[(group RHS + q) M + i][3 NP]
#pragma unroll
  for (int q = 0; q < RHS; ++q) {
    if (wave > 0) {
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int a = 0; a < 3; ++a) red[wave - 1][lane][3 * p + a] = g[q][p][a];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          double s = g[q][p][a];
#pragma unroll
          for (int w = 0; w < kOpWaves - 1; ++w) s += red[w][lane][3 * p + a];
          red[0][lane][3 * p + a] = s;
        }
    }
    __syncthreads();
    const int rows = min(kOpTile, M - static_cast<int>(blockIdx.x) * kOpTile);
    double* out = part + ((static_cast<int64_t>(blockIdx.y) * RHS + q) * M + static_cast<int64_t>(blockIdx.x) * kOpTile) *
                             (3 * NP);
    for (int e = threadIdx.x; e < rows * 3 * NP; e += kOpThreads) out[e] = red[0][e / (3 * NP)][e % (3 * NP)];
    __syncthreads();
  }
}

// Projections TF[k][a] = sum_p W_k(s_p) g_i(s_p)[a], k = 0..N, of target i from
// the groups' partials, into LDS (a barrier follows in the caller).
template <int N>
__device__ __forceinline__ void op_project(int i, int M, int variant, int groups, int rhs, int nrhs,
                                           const double* __restrict__ part, double* gs, double (*TF)[3]) {
  static constexpr OpTables<N> tab{};
  constexpr int NP = op_nodes<N>();
  const int tid = threadIdx.x;
  if (tid < 3 * NP) {
    double s = 0.0;
    for (int q = 0; q < groups; ++q)
      s += part[((static_cast<int64_t>(q) * nrhs + rhs) * M + i) * (3 * NP) + tid];
    gs[tid] = s;
  }
  __syncthreads();
  if (tid < 3 * (N + 1)) {
    const auto& w = tab.composite[variant >> 1];
    const int k = tid / 3, a = tid - 3 * k;
    double s = 0.0;
    for (int h = 0; h < NP / 2; ++h) {
      const double gp = gs[3 * (2 * h) + a], gm = gs[3 * (2 * h + 1) + a];
      s = fma(w.W[h][k], (k & 1) ? gp - gm : gp + gm, s);
    }
    TF[k][a] = s;
  }
}

constexpr int kOpRowThreads = 128;
constexpr int kOpRowWaves = kOpRowThreads / 64;

// Sum of v over the workgroup in lane 0 of each wavefront's red[wave][slot].
template <int S>
__device__ __forceinline__ void op_reduce(const double (&v)[S], double (*red)[S]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < S; ++q) {
    double s = v[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) red[wave][q] = s;
  }
}

// y = A x or b - A x: workgroup = target fiber.  The stored pairs stream their
// segment (the theta product's arithmetic), the far ones come from the partials.
template <int N>
__global__ __launch_bounds__(kOpRowThreads) void op_rows_kernel(int M, int variant, int groups, NearStore near,
                                                                const double* __restrict__ part,
                                                                const double* __restrict__ ori,
                                                                const double* __restrict__ x, double* __restrict__ y,
                                                                const double* __restrict__ b, int mode, PhysConsts pc,
                                                                const int* __restrict__ skip) {
  constexpr int NP = op_nodes<N>();
  constexpr int S = 1 + 3 * (N - 1);
  if (skip != nullptr && *skip) return;
  __shared__ double gs[3 * NP], TF[N + 1][3];
  __shared__ double red[kOpRowWaves][S];
  const int i = blockIdx.x;
  op_project<N>(i, M, variant, groups, 0, 1, part, gs, TF);
  const int cnt = near.count[i];
  const int64_t Lp = near_stride(cnt, N);
  const float* seg = near.data + near.base[i];
  const int* src = reinterpret_cast<const int*>(seg);
  const float* T = seg + near_ints(cnt);
  double acc[S];
#pragma unroll
  for (int q = 0; q < S; ++q) acc[q] = 0.0;
  for (int e = threadIdx.x; e < cnt * N; e += kOpRowThreads) {
    const int slot = e / N;
    const double* xe = x + 3 * (static_cast<int64_t>(src[slot]) * N + (e - slot * N));
    const double x0 = xe[0], x1 = xe[1], x2 = xe[2];
    const float* p = T + e;
    acc[0] = fma(static_cast<double>(p[0]), x0,
                 fma(static_cast<double>(p[Lp]), x1, fma(static_cast<double>(p[2 * Lp]), x2, acc[0])));
#pragma unroll
    for (int k = 1; k < N; ++k) {
      const float* pk = p + (3 + 6 * (k - 1)) * Lp;
      const double xx = pk[0], yy = pk[Lp], zz = pk[2 * Lp], xy = pk[3 * Lp], xz = pk[4 * Lp], yz = pk[5 * Lp];
      double* u = acc + 1 + 3 * (k - 1);
      u[0] = fma(xx, x0, fma(xy, x1, fma(xz, x2, u[0])));
      u[1] = fma(xy, x0, fma(yy, x1, fma(yz, x2, u[1])));
      u[2] = fma(xz, x0, fma(yz, x1, fma(zz, x2, u[2])));
    }
  }
  op_reduce<S>(acc, red);
  __syncthreads();
  const int tid = threadIdx.x;
  if (tid < 3 * N) {
    const int k = tid / 3, a = tid - 3 * k;
    const double t[3] = {ori[3 * i], ori[3 * i + 1], ori[3 * i + 2]};
    auto stored = [&](int q) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kOpRowWaves; ++w) s += red[w][q];
      return s;
    };
    double out;
    if (k == 0) {
      out = static_cast<double>(pc.D1) * t[a] * (stored(0) + (t[0] * TF[1][0] + t[1] * TF[1][1] + t[2] * TF[1][2]));
    } else {
      double U[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) U[c] = stored(1 + 3 * (k - 1) + c) + TF[k + 1][c];
      const double tU = t[0] * U[0] + t[1] * U[1] + t[2] * U[2];
      out = static_cast<double>(pc.gamma[k]) * (U[a] - static_cast<double>(pc.eigen[k]) * t[a] * tU);
    }
    const int64_t row = static_cast<int64_t>(3 * N) * i + tid;
    out += x[row];  // identity diagonal block
    y[row] = mode == 1 ? b[row] - out : out;
  }
}

// The far pairs' rows of b and the velocity constants (density 0: the force)
// and of the off-diagonal product with x0 (density 1).
template <int N>
__global__ __launch_bounds__(64) void op_assemble_rows_kernel(int M, int variant, int groups, int nrhs,
                                                              const double* __restrict__ part,
                                                              const double* __restrict__ ori,
                                                              double* __restrict__ b, double* __restrict__ c,
                                                              double* __restrict__ ax, PhysConsts pc) {
  constexpr int NP = op_nodes<N>();
  __shared__ double gs[3 * NP], TF[N + 1][3];
  const int i = blockIdx.x, tid = threadIdx.x;
  const double t[3] = {ori[3 * i], ori[3 * i + 1], ori[3 * i + 2]};
  for (int q = 0; q < nrhs; ++q) {
    op_project<N>(i, M, variant, groups, q, nrhs, part, gs, TF);
    __syncthreads();
    if (tid < 3 * N) {
      const int k = tid / 3, a = tid - 3 * k;
      const double* U = TF[k + 1];
      const double tU = t[0] * U[0] + t[1] * U[1] + t[2] * U[2];
      const double v = k == 0 ? static_cast<double>(pc.D1) * t[a] * tU
                              : static_cast<double>(pc.gamma[k]) *
                                    (U[a] - static_cast<double>(pc.eigen[k]) * t[a] * tU);
      const int64_t row = static_cast<int64_t>(3 * N) * i + tid;
      if (q == 0)
        b[row] = -v;
      else
        ax[row] = v;
    } else if (q == 0 && c != nullptr && tid < 3 * N + 6) {
      const int e = tid - 3 * N;
      c[static_cast<int64_t>(i) * 6 + e] = TF[e / 3][e % 3];
    }
    __syncthreads();
  }
}

// Velocities: workgroup = target fiber (velocity_stored_block's formulas).
template <int N>
__global__ __launch_bounds__(kOpRowThreads) void op_velocity_kernel(int M, int variant, int groups, NearStore near,
                                                                    const double* __restrict__ part,
                                                                    const double* __restrict__ cpart,
                                                                    const double* __restrict__ ori,
                                                                    const double* __restrict__ x, PhysConsts pc,
                                                                    double* __restrict__ tvel,
                                                                    double* __restrict__ rvel) {
  constexpr int NP = op_nodes<N>();
  constexpr int NC = 3 + 6 * (N - 1);
  __shared__ double gs[3 * NP], TF[N + 1][3];
  __shared__ double red[kOpRowWaves][6];
  const int i = blockIdx.x;
  op_project<N>(i, M, variant, groups, 0, 1, part, gs, TF);
  const int cnt = near.count[i];
  const int64_t Lp = near_stride(cnt, N);
  const float* seg = near.data + near.base[i];
  const int* src = reinterpret_cast<const int*>(seg);
  const float* V = seg + near_ints(cnt) + NC * Lp;
  double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // Phi_0 x, Theta_0 x
  for (int e = threadIdx.x; e < cnt * N; e += kOpRowThreads) {
    const int slot = e / N;
    const double* xe = x + 3 * (static_cast<int64_t>(src[slot]) * N + (e - slot * N));
    const double x0 = xe[0], x1 = xe[1], x2 = xe[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float* p = V + (h == 0 ? 6 : 0) * Lp + e;
      const double xx = p[0], yy = p[Lp], zz = p[2 * Lp], xy = p[3 * Lp], xz = p[4 * Lp], yz = p[5 * Lp];
      double* u = acc + 3 * h;
      u[0] = fma(xx, x0, fma(xy, x1, fma(xz, x2, u[0])));
      u[1] = fma(xy, x0, fma(yy, x1, fma(yz, x2, u[1])));
      u[2] = fma(xz, x0, fma(yz, x1, fma(zz, x2, u[2])));
    }
  }
  op_reduce<6>(acc, red);
  __syncthreads();
  if (threadIdx.x != 0) return;
  double Sv[6];
  for (int c = 0; c < 6; ++c) {
    double s = cpart[static_cast<int64_t>(i) * 6 + c] + cpart[(static_cast<int64_t>(M) + i) * 6 + c] + TF[c / 3][c % 3];
#pragma unroll
    for (int w = 0; w < kOpRowWaves; ++w) s += red[w][c];
    Sv[c] = s;
  }
  const double t[3] = {ori[3 * i], ori[3 * i + 1], ori[3 * i + 2]};
  const double F[3] = {2.0 * pc.Fh_d[0], 2.0 * pc.Fh_d[1], 2.0 * pc.Fh_d[2]};
  const double d = pc.d;
  const double tF = t[0] * F[0] + t[1] * F[1] + t[2] * F[2];
  const double tS = t[0] * Sv[3] + t[1] * Sv[4] + t[2] * Sv[5];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    tvel[3 * i + a] = (0.5 / d) * ((d + 2.0) * F[a] + (d - 2.0) * tF * t[a] + Sv[a]);
    rvel[3 * i + a] = (1.5 / d) * (Sv[3 + a] - t[a] * tS);
  }
}

// The pairs of a large suspension that a product does not form again: workgroup
// = target fiber, every source.
template <int N, int NQI, bool ANALYTIC>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(
    theta_min_waves<N, NQI, ANALYTIC>(kProductBytes<N, NQI> + kListBytes<N, NQI>), 8))) void assemble_segments_kernel(
    int M, const double* __restrict__ pos, const double* __restrict__ ori, NearStore store,
    double* __restrict__ bpart, PhysConsts pc, double* __restrict__ cpart, const double* __restrict__ x0,
    double* __restrict__ apart) {
  assemble_near_block<N, NQI, ANALYTIC, false, true>(blockIdx.x, 0, M, 0, pos, ori, nullptr, bpart, M, pc, nullptr,
                                                     cpart, x0, apart, nullptr, nullptr, nullptr, &store);
}

hipError_t launch_assemble_segments(int N, int NQI, bool analytical, int M, const double* pos, const double* ori,
                                    const NearStore& near, double* bpart, double* cpart, const double* x0,
                                    double* apart, const PhysConsts& pc, hipStream_t s) {
  const dim3 grid(M), block(kPairThreads);
#define RF_SEG(NN, QQ)                                                                                              \
  if (NQI == QQ) {                                                                                                  \
    if (analytical)                                                                                                 \
      hipLaunchKernelGGL((assemble_segments_kernel<NN, QQ, true>), grid, block, 0, s, M, pos, ori, near, bpart, pc,  \
                         cpart, x0, apart);                                                                         \
    else                                                                                                            \
      hipLaunchKernelGGL((assemble_segments_kernel<NN, QQ, false>), grid, block, 0, s, M, pos, ori, near, bpart, pc, \
                         cpart, x0, apart);                                                                         \
    return hipGetLastError();                                                                                       \
  }
#define RF_SEG_N(NN) \
  case NN:           \
    RF_SEG(NN, 4)    \
    RF_SEG(NN, 8)    \
    RF_SEG(NN, 16)   \
    break;
  switch (N) {
    RF_SEG_N(3)  // operator_form is for N >= 3
    RF_SEG_N(4)
    RF_SEG_N(5)
    RF_SEG_N(6)
    RF_SEG_N(7)
    RF_SEG_N(8)
  }
#undef RF_SEG_N
#undef RF_SEG
  return hipErrorInvalidValue;
}

// Source groups: a workgroup is (64 targets, one group), four wavefronts on
// quarters of the group.  Among the counts that leave a wavefront at least 8
// sources, the one that fills whole rounds of the 256 CUs best, more than three
// workgroups per CU if the targets allow it (four are resident).
static PairGrid op_grid(int M) {
  PairGrid best{};
  best.tiles = (M + kOpTile - 1) / kOpTile;
  double score = -1.0;
  for (int g = 1; g <= 64; ++g) {
    const int jg = (M + g - 1) / g;
    if (g > 1 && jg < 8 * kOpWaves) break;
    const int groups = (M + jg - 1) / jg;
    const double wgs = static_cast<double>(best.tiles) * groups;
    const double rounds = static_cast<double>((static_cast<int64_t>(wgs) + 255) / 256);
    const double s = (wgs / (256.0 * rounds)) * (wgs >= 768.0 ? 1.0 : 0.5 + wgs / 1536.0) - 0.002 * groups;
    if (s > score) {
      score = s;
      best.groups = groups;
      best.jgroup = jg;
    }
  }
  return best;
}

static int op_variant(int NQI, bool analytical) {
  return (NQI == 4 ? 0 : (NQI == 8 ? 2 : 4)) + (analytical ? 1 : 0);
}

// Two sets: the force's and x0's.
size_t op_node_doubles(int M, int N) { return 2 * 4 * static_cast<size_t>(M) * (N <= 5 ? 6 : 8); }

size_t op_part_doubles(int M, int N) {
  return 2 * static_cast<size_t>(op_grid(M).groups) * static_cast<size_t>(M) * 3 * (N <= 5 ? 6 : 8);
}

template <int N, int RHS>
static hipError_t op_far(int NQI, bool analytical, int M, const Operator& op, const double* x0, const double* x1,
                         const PhysConsts& pc, hipStream_t s, const int* skip) {
  constexpr int NP = op_nodes<N>();
  const PairGrid g = op_grid(M);
  const int variant = op_variant(NQI, analytical);
  const dim3 nb((M * NP + 255) / 256);
  const double *pos = op.near.pos, *ori = op.near.ori;
  double* n1 = op.nodes + 4 * static_cast<int64_t>(M) * NP;
  hipLaunchKernelGGL(op_nodes_kernel<N>, nb, dim3(256), 0, s, M, variant, ori, x0, pc, op.nodes, skip);
  if (RHS > 1)
    hipLaunchKernelGGL(op_nodes_kernel<N>, nb, dim3(256), 0, s, M, variant, ori, x1, pc, n1, skip);
  hipLaunchKernelGGL((op_far_kernel<N, RHS>), dim3(g.tiles, g.groups), dim3(kOpThreads), 0, s, M,
                     far_rule(N, NQI).r[0], pos, ori, op.nodes, n1, op.part, g.jgroup, pc, skip);
  return hipGetLastError();
}

template <int N>
static hipError_t op_assemble_far_n(int NQI, bool analytical, int M, const Operator& op, double* b,
                                    double* c, const double* x0, double* ax, const PhysConsts& pc, hipStream_t s) {
  const hipError_t e = x0 ? op_far<N, 2>(NQI, analytical, M, op, nullptr, x0, pc, s, nullptr)
                          : op_far<N, 1>(NQI, analytical, M, op, nullptr, nullptr, pc, s, nullptr);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(op_assemble_rows_kernel<N>, dim3(M), dim3(64), 0, s, M, op_variant(NQI, analytical),
                     op_grid(M).groups, x0 ? 2 : 1, op.part, op.near.ori, b, c, ax, pc);
  return hipGetLastError();
}

// operator_form is for N >= 3
#define RF_OP_SIZES(CALL)  \
  switch (N) {             \
    case 3: return CALL(3); \
    case 4: return CALL(4); \
    case 5: return CALL(5); \
    case 6: return CALL(6); \
    case 7: return CALL(7); \
    case 8: return CALL(8); \
    default: return hipErrorInvalidValue; \
  }

hipError_t op_assemble_far(int N, int NQI, bool analytical, int M, const Operator& op, double* bpart, double* cpart,
                           const double* x0, double* apart, const PhysConsts& pc, hipStream_t s) {
  const int64_t n = 3LL * N * M;
  double* c = cpart ? cpart + static_cast<int64_t>(M) * 6 : nullptr;
  double* ax = apart ? apart + n : nullptr;
#define RF_CALL(NN) op_assemble_far_n<NN>(NQI, analytical, M, op, bpart + n, c, x0, ax, pc, s)
  RF_OP_SIZES(RF_CALL)
#undef RF_CALL
}

template <int N>
static hipError_t op_product_n(int NQI, bool analytical, int M, const Operator& op, const double* x, double* y,
                               const double* b, int mode, const PhysConsts& pc, hipStream_t s, const int* skip) {
  const hipError_t e = op_far<N, 1>(NQI, analytical, M, op, x, nullptr, pc, s, skip);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(op_rows_kernel<N>, dim3(M), dim3(kOpRowThreads), 0, s, M, op_variant(NQI, analytical),
                     op_grid(M).groups, op.near, op.part, op.near.ori, x, y, b, mode, pc, skip);
  return hipGetLastError();
}

static hipError_t op_product_any(int N, int NQI, bool analytical, int M, const Operator& op, const double* x,
                                 double* y, const double* b, int mode, const PhysConsts& pc, hipStream_t s,
                                 const int* skip) {
#define RF_CALL(NN) op_product_n<NN>(NQI, analytical, M, op, x, y, b, mode, pc, s, skip)
  RF_OP_SIZES(RF_CALL)
#undef RF_CALL
}

hipError_t op_product(int N, int NQI, bool analytical, int M, const Operator& op, const double* x, double* y,
                      const double* b, int mode, const PhysConsts& pc, hipStream_t s, hipEvent_t ev_begin, hipEvent_t ev_end, const int* skip) {
  if (ev_begin) (void)hipEventRecord(ev_begin, s);
  const hipError_t e = op_product_any(N, NQI, analytical, M, op, x, y, b, mode, pc, s, skip);
  if (ev_end) (void)hipEventRecord(ev_end, s);
  return e;
}

template <int N>
static hipError_t op_velocities_n(int NQI, bool analytical, int M, const Operator& op, const double* cpart,
                                  const double* x, const PhysConsts& pc, double* tvel, double* rvel, hipStream_t s) {
  const hipError_t e = op_far<N, 1>(NQI, analytical, M, op, x, nullptr, pc, s, nullptr);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(op_velocity_kernel<N>, dim3(M), dim3(kOpRowThreads), 0, s, M, op_variant(NQI, analytical),
                     op_grid(M).groups, op.near, op.part, cpart, op.near.ori, x, pc, tvel, rvel);
  return hipGetLastError();
}

hipError_t op_velocities(int N, int NQI, bool analytical, int M, const Operator& op, const double* cpart,
                         const double* x, const PhysConsts& pc, double* tvel, double* rvel, hipStream_t s) {
#define RF_CALL(NN) op_velocities_n<NN>(NQI, analytical, M, op, cpart, x, pc, tvel, rvel, s)
  RF_OP_SIZES(RF_CALL)
#undef RF_CALL
}

}  // namespace rf
