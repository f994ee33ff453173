// rf_far.hip -- the far pairs of the theta-form assembly.
//
// Reference: fortran/assemble_matrix.incl:1-161 forms the projections of every
// pair through its Q target nodes; for fibers whose centres lie far_rule's
// radii apart (rf_device.h) the same projections follow from NP x NP kernel
// values with NP = 6 or 8 (8 or 10 for N >= 6).  The near pairs are
// assemble_near_block's (rf_near.h): both select by far_class, so every
// pair is formed by exactly one of the two.
//
// Work decomposition.  Workgroup = one target fiber i, four wavefronts.  Each
// step classifies 256 sources, one per lane, as eight aligned blocks of 32.  A
// block that is almost all far is formed as it is, by one wavefront, its other
// sources masked; the far sources of the rest, and the closer ones of a block
// formed with the smaller rule, are appended to two lists in LDS (by node
// count) that the wavefronts form 32 at a time.  So no lanes idle in a dense
// suspension, and in a dilute one the rows leave as whole 128-byte lines.
// In a batch lanes 2k and 2k + 1 share the pair (i, j_k): the even
// lane takes the target nodes +s, the odd lane -s, they exchange kernel values
// through a cross-lane move, and each keeps the projections of one parity (even
// lane kk = 0, 2, 4, odd lane 1, 3, 5) of every source mode in registers: each
// kernel value is formed once, without LDS or barriers.  The rows then go
// through the wavefront's own LDS buffer, so that 64 lanes store 64 consecutive
// floats of a component array; the right-hand side, the velocity constants and
// the products with x0 are summed over the sources in FP64 registers.
//
// Bound: VALU issue and the stores, one after the other more than beside each
// other: a wavefront's next batch starts when the stores of its last one have
// left, and 245 registers allow two wavefronts per SIMD.  At M = 5000 (N = 5, 8
// intervals, a ball at 0.028 fibers per unit volume) the launch takes 6.2 ms;
// without its stores 2.7 ms (a batch of 6 x 6 nodes is 1 750 instructions for
// 32 pairs, 3 500 per pair and lane against the 16 400 of 24 x 8 nodes), and a
// kernel that only writes the same 19.5 GB 3.6 ms.  The assembly, near pairs,
// sums and first residual included, went from 13.5 to 6.4 ms there, from 3.65
// to 1.19 ms at M = 2000 and from 85 to 22 ms at M = 10 000 (numerical, 24 x 24
// nodes before).
#include <type_traits>

#include "rf_internal.h"

namespace rf {

constexpr int kFarThreads = 256;
constexpr int kFarWaves = kFarThreads / 64;
constexpr int kFarBatch = 32;              // pairs of a batch: two lanes each
constexpr int kFarRound = kFarWaves * kFarBatch;  // a full batch for each wavefront
constexpr int kFarBlocks = kFarThreads / kFarBatch;  // blocks of one step
// Listed sources at most: less than a round of either kind, plus one step's.
// One list grows from the first entry up, the other from the last down.
constexpr int kFarEntries = 2 * kFarRound + kFarThreads;
// Far sources from which a block of 32 is formed as it is.
constexpr int kFarDirect = 24;

// The other lane of the pair.
__device__ __forceinline__ float swap_pair(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
}

// K(R) as stokes_kernel forms it; R is not small here, so the reciprocal square
// root needs no range handling.
__device__ __forceinline__ void stokes_kernel_far(float rx, float ry, float rz, float two_eps2, float six_eps2,
                                                  float K[6]) {
  const float r2 = fmaf(rx, rx, fmaf(ry, ry, rz * rz));
  const float inv = __builtin_amdgcn_rsqf(r2);
  const float inv2 = inv * inv;
  const float inv3 = inv2 * inv;
  const float a = fmaf(two_eps2, inv3, inv);
  const float c = inv3 * fmaf(-six_eps2, inv2, 1.0f);
  const float cx = c * rx, cy = c * ry, cz = c * rz;
  K[0] = fmaf(cx, rx, a);
  K[1] = fmaf(cy, ry, a);
  K[2] = fmaf(cz, rz, a);
  K[3] = cx * ry;
  K[4] = cx * rz;
  K[5] = cy * rz;
}

// Everything a target's batches need: uniform over the wavefront but sgn and odd.
struct FarTarget {
  double x[3];    // centre
  double st[3];   // sgn t_i: the lane's target nodes are x + s_h st
  float t[3];     // t_i
  bool odd;
  float sgn;      // +1 on even lanes, -1 on odd
};

// FP64 sums over the sources that one lane keeps, by its target slots kg (kk =
// 2 kg + odd): TF of the mode-0 projections dotted with F/2, U = sum_m Theta x0
// (slots kg >= 1), and s0 = Q0 . x0 (odd lanes, kk = 1).
template <int N>
struct FarSums {
  static constexpr int KS = N / 2 + 1;
  double TF[KS][3];
  double U[KS][3];
  double s0;
};

// Target slots of one sweep over the nodes.  Three (N <= 5: every slot at once)
// hold 3 (N + 1) 6 sums per lane; larger N takes two at a time and forms the
// kernel values again for the next two.
template <int N>
constexpr int far_slots() { return N <= 5 ? N / 2 + 1 : 2; }

// The rules' weights for NQI = 4, 8, 16 (variant 2 x index + exact): the target
// functional is the composite rule's, the source functional that or the exact
// integral's.
template <int N, int NP>
struct FarTables {
  FarWeights<N, NP> composite[3], exact;
  constexpr FarTables()
      : composite{FarWeights<N, NP>(4, false), FarWeights<N, NP>(8, false), FarWeights<N, NP>(16, false)},
        exact(0, true) {}
};

// Projections C[k][m][c] of slots K0 .. K0 + KN - 1 for the lane's pair:
// d = x_i - x_j, tj the source's direction.  The loop over the source's node
// pairs stays rolled: its weights come through scalar registers, and a single
// copy keeps C, the node pair's sums and the kernel values within 256 registers.
template <int N, int NP, int K0, int KN>
__device__ __forceinline__ void far_projections(const FarTarget& T, int variant, const double d[3], const float tj[3],
                                                float two_eps2, float six_eps2, float C[KN][N + 1][6]) {
  static constexpr FarTables<N, NP> tab{};
  constexpr int H = NP / 2;
  static constexpr double node[5] = {gl_node(NP, 0), gl_node(NP, 1), gl_node(NP, 2), gl_node(NP, H > 3 ? 3 : 0),
                                     gl_node(NP, H > 4 ? 4 : 0)};
  const FarWeights<N, NP>& tgt = tab.composite[variant >> 1];
  const FarWeights<N, NP>& src = (variant & 1) ? tab.exact : tgt;
  float rb[H][3], wt[KN][H];
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int a = 0; a < 3; ++a) rb[h][a] = static_cast<float>(fma(node[h], T.st[a], d[a]));
#pragma unroll
  for (int k = 0; k < KN; ++k)
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int ke = 2 * (K0 + k), ko = ke + 1;
      const float we = ke <= N ? tgt.W[h][ke <= N ? ke : 0] : 0.0f, wo = ko <= N ? tgt.W[h][ko <= N ? ko : 0] : 0.0f;
      wt[k][h] = T.odd ? wo : we;
    }
#pragma unroll
  for (int k = 0; k < KN; ++k)
#pragma unroll
    for (int m = 0; m <= N; ++m)
#pragma unroll
      for (int c = 0; c < 6; ++c) C[k][m][c] = 0.0f;
#pragma unroll 1
  for (int g = 0; g < H; ++g) {
    const float s = static_cast<float>(node[g]);
    const float ux = s * tj[0], uy = s * tj[1], uz = s * tj[2];
    float Gp[KN][6], Gm[KN][6];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      float K[6];
      // source node +s: even lanes sum the two target nodes, odd lanes take
      // their difference, K(+s_h) +- K(-s_h)
      stokes_kernel_far(rb[h][0] - ux, rb[h][1] - uy, rb[h][2] - uz, two_eps2, six_eps2, K);
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const float e = fmaf(K[c], T.sgn, swap_pair(K[c]));
#pragma unroll
        for (int k = 0; k < KN; ++k) Gp[k][c] = h == 0 ? wt[k][h] * e : fmaf(wt[k][h], e, Gp[k][c]);
      }
      // source node -s
      stokes_kernel_far(rb[h][0] + ux, rb[h][1] + uy, rb[h][2] + uz, two_eps2, six_eps2, K);
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const float e = fmaf(K[c], T.sgn, swap_pair(K[c]));
#pragma unroll
        for (int k = 0; k < KN; ++k) Gm[k][c] = h == 0 ? wt[k][h] * e : fmaf(wt[k][h], e, Gm[k][c]);
      }
    }
#pragma unroll
    for (int k = 0; k < KN; ++k)
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const float E = Gp[k][c] + Gm[k][c], O = Gp[k][c] - Gm[k][c];
#pragma unroll
        for (int m = 0; m <= N; ++m) C[k][m][c] = fmaf(src.W[g][m], (m & 1) ? O : E, C[k][m][c]);
      }
  }
}

// Where a batch's rows go.
struct FarOut {
  float* T;          // target i's system rows (component stride Lp)
  float* Tv;         // its velocity-operator rows, or null
  _Float16* T16;     // its FP16 rows (HALF)
  float* S16;        // its FP16 block scales, by source (HALF)
  const double* x0;  // or null
  uint32_t Lp;
};

// A batch as the store side sees it: its 32 N (source, mode) columns are moved 64
// at a time, lane l those with index l + 64 t of every row, which belong to
// column col[t] of the component arrays.  What the store costs is whether it
// covers whole 128-byte lines (a write kernel of this pattern: 5.4 TB/s, 3.3 -
// 3.7 with runs that start anywhere else, 4 or 16 bytes per lane alike): a full
// block's runs are 32 N floats from a multiple of 32.
template <int N>
struct FarColumns {
  static constexpr int kT = (N + 1) / 2;
  uint32_t col[kT];
  float iv[kT];  // HALF: the inverse scales of their blocks
  bool in[kT];   // within the batch
};

// Rows 0 .. R - 1 of the wavefront's buffer to dst(r) (and, scaled, to dst16(r)).
template <int N, int R, bool HALF, class Dst, class Dst16>
__device__ __forceinline__ void far_flush(const FarColumns<N>& c, const float* buf, Dst dst, Dst16 dst16) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < FarColumns<N>::kT; ++t) {
    if (!c.in[t]) continue;
    float v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = buf[r * kFarBatch * N + lane + 64 * t];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      dst(r)[c.col[t]] = v[r];
      if constexpr (HALF) dst16(r)[c.col[t]] = static_cast<_Float16>(v[r] * c.iv[t]);
    }
  }
}

// Slots K0 .. K0 + KN - 1 of one batch: add to the sums (the active lanes, whose
// pair is (i, j)), then store (every lane of the wavefront takes part).  The
// loads of x0 come before the stores: a load is complete only with every store
// issued before it.
template <int N, int KN, int K0, bool HALF>
__device__ __forceinline__ void far_emit(const FarTarget& T, const FarOut& out, const PhysConsts& pc, bool active,
                                         int j, const FarColumns<N>& cols, float* buf, const float C[KN][N + 1][6],
                                         FarSums<N>& sums) {
  constexpr int ia[3][3] = {{0, 3, 4}, {3, 1, 5}, {4, 5, 2}};  // sym_index
  constexpr bool kOddLast = N % 2 == 1;  // the odd lanes' last slot exists (kk = 2 kg + 1 <= N)
  const int lane = threadIdx.x & 63;
  float* const mine = buf + (lane >> 1) * N;  // the lane's columns of row 0
  auto ordered = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  auto q0 = [&](int u, int m) {  // Q0_u = (Theta_0 t_i)_u, kk = 1: the odd lanes'
    return C[0][m + 1][ia[0][u]] * T.t[0] + C[0][m + 1][ia[1][u]] * T.t[1] + C[0][m + 1][ia[2][u]] * T.t[2];
  };
  if (active) {
#pragma unroll
    for (int k = 0; k < KN; ++k)  // mode 0: the force
#pragma unroll
      for (int a = 0; a < 3; ++a)
        sums.TF[K0 + k][a] += static_cast<double>(C[k][0][ia[a][0]] * pc.Fh[0] + C[k][0][ia[a][1]] * pc.Fh[1] +
                                                  C[k][0][ia[a][2]] * pc.Fh[2]);
    if (out.x0) {
      const double* const x = out.x0 + 3 * static_cast<int64_t>(N) * j;
#pragma unroll
      for (int m = 0; m < N; ++m) {
        const double xm[3] = {x[3 * m], x[3 * m + 1], x[3 * m + 2]};
#pragma unroll
        for (int k = 0; k < KN; ++k) {
          const int kg = K0 + k;
          if (kg == 0) {
#pragma unroll
            for (int u = 0; u < 3; ++u) sums.s0 = fma(static_cast<double>(q0(u, m)), xm[u], sums.s0);
          } else if (kg < N / 2 || kOddLast || !T.odd) {
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
              for (int b = 0; b < 3; ++b)
                sums.U[kg][a] = fma(static_cast<double>(C[k][m + 1][ia[a][b]]), xm[b], sums.U[kg][a]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    const int kg = K0 + k;
    if (kg == 0) {
      if (T.odd) {
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
          for (int m = 0; m < N; ++m) mine[u * kFarBatch * N + m] = q0(u, m);
      }
      ordered();
      far_flush<N, 3, HALF>(
          cols, buf, [&](int u) { return out.T + static_cast<size_t>(u) * out.Lp; },
          [&](int u) { return out.T16 + static_cast<size_t>(u) * out.Lp; });
      ordered();
      if (!out.Tv) continue;
    }
    // kg = 0: Phi_0 (kk = 0) is the velocity operator's components 6..11,
    // Theta_0 (kk = 1) its 0..5.  Else Theta_{kk-1} at component 3 + 6 (kk - 2):
    // even lanes kk = 2 kg, odd lanes 2 kg + 1.
#pragma unroll
    for (int c = 0; c < 6; ++c)
#pragma unroll
      for (int m = 0; m < N; ++m) mine[((T.odd ? 6 : 0) + c) * kFarBatch * N + m] = C[k][m + 1][c];
    ordered();
    if (kg == 0) {
      far_flush<N, 12, false>(
          cols, buf, [&](int r) { return out.Tv + static_cast<size_t>(r < 6 ? 6 + r : r - 6) * out.Lp; },
          [&](int) { return out.T16; });
    } else {
      auto t32 = [&](int r) { return out.T + static_cast<size_t>(3 + 12 * (kg - 1) + r) * out.Lp; };
      auto t16 = [&](int r) { return out.T16 + static_cast<size_t>(3 + 12 * (kg - 1) + r) * out.Lp; };
      if (kg < N / 2 || kOddLast)
        far_flush<N, 12, HALF>(cols, buf, t32, t16);
      else
        far_flush<N, 6, HALF>(cols, buf, t32, t16);
    }
    ordered();
  }
}

// Largest |projection| (kk >= 1, m >= 1) of the lane's slots.
template <int N, int KN, int K0>
__device__ __forceinline__ float far_max(const FarTarget& T, const float C[KN][N + 1][6]) {
  float g = 0.0f;
#pragma unroll
  for (int k = 0; k < KN; ++k) {
    if (K0 + k == 0 && !T.odd) continue;  // kk = 0
#pragma unroll
    for (int m = 1; m <= N; ++m)
#pragma unroll
      for (int c = 0; c < 6; ++c) g = fmaxf(g, fabsf(C[k][m][c]));
  }
  return g;
}

// The lane's largest |projection| over every slot: the FP16 block scale needs it
// before the first row is stored, so more slots than one sweep holds (N >= 6)
// are swept once more for it.
template <int N, int NP, int K0>
__device__ __forceinline__ float far_scan_max(const FarTarget& T, const PhysConsts& pc, int variant, const double d[3],
                                              const float tj[3]) {
  constexpr int KS = N / 2 + 1;
  if constexpr (K0 < KS) {
    constexpr int KN = (KS - K0) < far_slots<N>() ? (KS - K0) : far_slots<N>();
    float C[KN][N + 1][6];
    far_projections<N, NP, K0, KN>(T, variant, d, tj, 2.0f * pc.eps2, 6.0f * pc.eps2, C);
    return fmaxf(far_max<N, KN, K0>(T, C), far_scan_max<N, NP, K0 + KN>(T, pc, variant, d, tj));
  } else {
    return 0.0f;
  }
}

// Block scale of the lane's pair to S16, and the inverse scales of the lane's
// columns.
template <int N>
__device__ __forceinline__ void far_scales(const FarTarget& T, const FarOut& out, bool active, int j, float gmax,
                                           FarColumns<N>& cols) {
  const int lane = threadIdx.x & 63;
  gmax = fmaxf(gmax, swap_pair(gmax));
  float sv, iv;
  half_block_scale(__float_as_uint(gmax), sv, iv);
  if (active && !T.odd) out.S16[j] = sv;
#pragma unroll
  for (int t = 0; t < FarColumns<N>::kT; ++t)
    cols.iv[t] = __shfl(iv, 2 * min((lane + 64 * t) / N, kFarBatch - 1), 64);
}

template <int N, int NP, int K0, bool HALF>
__device__ __forceinline__ void far_passes(const FarTarget& T, const FarOut& out, const PhysConsts& pc, int variant,
                                           bool active, int j, const double d[3], const float tj[3],
                                           FarColumns<N>& cols, float* buf, FarSums<N>& sums) {
  constexpr int KS = N / 2 + 1;
  if constexpr (K0 < KS) {
    constexpr int KN = (KS - K0) < far_slots<N>() ? (KS - K0) : far_slots<N>();
    float C[KN][N + 1][6];
    far_projections<N, NP, K0, KN>(T, variant, d, tj, 2.0f * pc.eps2, 6.0f * pc.eps2, C);
    if constexpr (HALF && KN == KS) far_scales<N>(T, out, active, j, far_max<N, KN, K0>(T, C), cols);
    far_emit<N, KN, K0, HALF>(T, out, pc, active, j, cols, buf, C, sums);
    far_passes<N, NP, K0 + KN, HALF>(T, out, pc, variant, active, j, d, tj, cols, buf, sums);
  }
}

// Target fiber i, sources [jb, je): rows to `out`; the sums of the workgroup to
// bsum (the 3 N rows of b), csum (the 6 velocity constants, or null) and, with
// out.x0, asum (the 3 N rows of the off-diagonal product A x0).
template <int N, bool HALF>
__device__ __forceinline__ void assemble_far_block(int i, int jb, int je, int variant, const double* __restrict__ pos,
                                                   const double* __restrict__ ori, const FarOut& out,
                                                   const PhysConsts& pc, double* __restrict__ bsum,
                                                   double* __restrict__ csum, double* __restrict__ asum) {
  constexpr FarRule fine = far_rule(N, 8), coarse = far_rule(N, 4);
  FarRule rule = fine;
  if (variant < 2) rule = coarse;
  constexpr int KS = N / 2 + 1;
  constexpr int NS = 6 * KS + 1;  // sums of one lane
  // x_i - x_j, t_j and j of the listed sources, then those of the step's sources
  // (a source's entry after kFarEntries is its place in the step)
  __shared__ double ld[3][kFarEntries + kFarThreads];
  __shared__ float lt[3][kFarEntries + kFarThreads];
  __shared__ int lj[kFarEntries];
  __shared__ unsigned masks[2][kFarBlocks];  // the step's far sources, by class
  __shared__ __align__(16) float rows[kFarWaves][12 * kFarBatch * N];
  __shared__ double red[kFarWaves][2][NS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  FarTarget T;
  T.odd = lane & 1;
  T.sgn = T.odd ? -1.0f : 1.0f;
  double ti2 = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    T.x[a] = pos[3 * i + a];
    const double t = ori[3 * i + a];
    T.t[a] = static_cast<float>(t);
    T.st[a] = T.odd ? -t : t;
    ti2 = fma(t, t, ti2);
  }
  FarSums<N> sums;
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) sums.TF[k][a] = sums.U[k][a] = 0.0;
  sums.s0 = 0.0;

  // entry e of list c
  auto entry = [](int c, int e) { return c == 0 ? e : kFarEntries - 1 - e; };
  int pend[2] = {0, 0};  // listed and not yet formed: the same in every wavefront
  int tail = wave;       // the wavefront's next batch of what is left after the last step
  for (int js = jb;; js += kFarThreads) {
    const bool last = js + kFarThreads >= je;
    double d0[3];
    float t0[3];
    int cls = -1;
    {
      const int j = js + static_cast<int>(threadIdx.x);
      if (j < je && j != i) {
        double t[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          t[a] = ori[3 * j + a];
          t0[a] = static_cast<float>(t[a]);
          d0[a] = T.x[a] - pos[3 * j + a];
        }
        cls = far_class(rule, d0[0], d0[1], d0[2], ti2, fma(t[2], t[2], fma(t[1], t[1], t[0] * t[0])));
      }
    }
    const unsigned long long m0 = __ballot(cls == 0), m1 = __ballot(cls == 1);
    __syncthreads();  // the end of the last step's reads
    if (lane < 2) {
      masks[0][2 * wave + lane] = static_cast<unsigned>(m0 >> (32 * lane));
      masks[1][2 * wave + lane] = static_cast<unsigned>(m1 >> (32 * lane));
    }
    if (cls >= 0) {
      const int e = kFarEntries + static_cast<int>(threadIdx.x);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ld[a][e] = d0[a];
        lt[a][e] = t0[a];
      }
    }
    __syncthreads();
    // what becomes of each block, and of this lane's source
    unsigned direct[2] = {0, 0};  // blocks formed as they are with np[0], np[1] nodes
    int mine = -1, place = 0;     // the lane's list and entry
    {
      int found[2] = {pend[0], pend[1]};
      const int myblock = static_cast<int>(threadIdx.x) / kFarBatch;
      const unsigned below = (1u << (lane & 31)) - 1u;
#pragma unroll
      for (int b = 0; b < kFarBlocks; ++b) {
        const unsigned c0 = __builtin_amdgcn_readfirstlane(masks[0][b]);
        const unsigned c1 = __builtin_amdgcn_readfirstlane(masks[1][b]);
        const int n0 = __popc(c0), n1 = __popc(c1);
        const bool small = n0 >= kFarDirect, large = !small && n0 + n1 >= kFarDirect;
        if (small) direct[0] |= 1u << b;
        if (large) direct[1] |= 1u << b;
        const bool list0 = !small && !large, list1 = !large;
        if (b == myblock) {
          if (cls == 0 && list0) mine = 0, place = found[0] + __popc(c0 & below);
          if (cls == 1 && list1) mine = 1, place = found[1] + __popc(c1 & below);
        }
        if (list0) found[0] += n0;
        if (list1) found[1] += n1;
      }
      pend[0] = found[0];
      pend[1] = found[1];
    }
    if (mine >= 0) {
      const int e = entry(mine, place);
      lj[e] = js + static_cast<int>(threadIdx.x);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        ld[a][e] = d0[a];
        lt[a][e] = t0[a];
      }
    }
    __syncthreads();
    // The wavefront's blocks, then rounds of one batch per wavefront while a
    // list fills one, and after the last step the rest of both lists.
    const int n0 = __popc(direct[0]), n1 = __popc(direct[1]);
    for (int id = wave;;) {
      int c;               // rule
      bool active;         // the lane's pair counts
      int src, j;          // its entry and source
      FarColumns<N> cols;
      if (id < n0 + n1) {
        c = id < n0 ? 0 : 1;
        unsigned rest = direct[c];
        for (int q = c == 0 ? id : id - n0; q > 0; --q) rest &= rest - 1u;
        const int b = __ffs(rest) - 1;
        unsigned m = masks[0][b];
        if (c == 1) m |= masks[1][b];
        m = __builtin_amdgcn_readfirstlane(m);
        const int slot = lane >> 1, first = js + kFarBatch * b;
        active = (m >> slot) & 1u;
        j = first + slot;
        src = kFarEntries + kFarBatch * b + slot;
#pragma unroll
        for (int t = 0; t < FarColumns<N>::kT; ++t) {
          const int q = lane + 64 * t;
          cols.in[t] = q < kFarBatch * N && ((m >> (q / N & 31)) & 1u);
          cols.col[t] = static_cast<uint32_t>(first * N + q);
          cols.iv[t] = 0.0f;
        }
        id += kFarWaves;
      } else {
        int at, take = kFarBatch;
        if (pend[0] >= kFarRound || pend[1] >= kFarRound) {
          c = pend[0] >= kFarRound ? 0 : 1;
          pend[c] -= kFarRound;
          at = pend[c] + kFarBatch * wave;
        } else if (last) {
          const int b0 = (pend[0] + kFarBatch - 1) / kFarBatch, b1 = (pend[1] + kFarBatch - 1) / kFarBatch;
          if (tail >= b0 + b1) break;
          c = tail < b0 ? 0 : 1;
          at = kFarBatch * (c == 0 ? tail : tail - b0);
          take = min(kFarBatch, pend[c] - at);
          tail += kFarWaves;
        } else {
          break;
        }
        // the lanes past the batch's end repeat its last pair
        active = (lane >> 1) < take;
        src = entry(c, at + min(lane >> 1, take - 1));
        j = lj[src];
#pragma unroll
        for (int t = 0; t < FarColumns<N>::kT; ++t) {
          const int q = lane + 64 * t;
          cols.in[t] = q < take * N;
          cols.col[t] = static_cast<uint32_t>(lj[entry(c, at + min(q / N, take - 1))] * N + q % N);
          cols.iv[t] = 0.0f;
        }
      }
      const double d[3] = {ld[0][src], ld[1][src], ld[2][src]};
      const float tj[3] = {lt[0][src], lt[1][src], lt[2][src]};
      auto form = [&](auto np) {
        constexpr int NP = decltype(np)::value;
        if constexpr (HALF && KS > far_slots<N>())
          far_scales<N>(T, out, active, j, far_scan_max<N, NP, 0>(T, pc, variant, d, tj), cols);
        far_passes<N, NP, 0, HALF>(T, out, pc, variant, active, j, d, tj, cols, rows[wave], sums);
      };
      if (c == 0)
        form(std::integral_constant<int, fine.np[0]>{});
      else
        form(std::integral_constant<int, fine.np[1]>{});
    }
    if (last) break;
  }

  // sums over the lanes of one parity, then over the wavefronts
  double v[NS];
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      v[3 * k + a] = sums.TF[k][a];
      v[3 * (KS + k) + a] = sums.U[k][a];
    }
  v[NS - 1] = sums.s0;
#pragma unroll
  for (int q = 0; q < NS; ++q) {
#pragma unroll
    for (int off = 32; off > 1; off >>= 1) v[q] += __shfl_xor(v[q], off, 64);
  }
  if (lane < 2) {
#pragma unroll
    for (int q = 0; q < NS; ++q) red[wave][lane][q] = v[q];
  }
  __syncthreads();
  const int tid = threadIdx.x;
  if (tid >= 3 * N + 6) return;
  auto total = [&](int parity, int q) {
    double t = 0.0;
    for (int w = 0; w < kFarWaves; ++w) t += red[w][parity][q];
    return t;
  };
  double t[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) t[a] = ori[3 * i + a];
  if (tid < 3 * N) {  // row 3 k + a: projection kk = k + 1
    const int k = tid / 3, a = tid - 3 * k, kk = k + 1;
    double F[3], U[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      F[b] = total(kk & 1, 3 * (kk >> 1) + b);
      U[b] = total(kk & 1, 3 * (KS + (kk >> 1)) + b);
    }
    double gam = 0.0, eig = 0.0;
#pragma unroll
    for (int q = 1; q < N; ++q)
      if (k == q) {
        gam = pc.gamma[q];
        eig = pc.eigen[q];
      }
    const double tF = t[0] * F[0] + t[1] * F[1] + t[2] * F[2];
    const double ta = tid - 3 * k == 0 ? t[0] : (a == 1 ? t[1] : t[2]);
    const double Fa = a == 0 ? F[0] : (a == 1 ? F[1] : F[2]);
    const double Ua = a == 0 ? U[0] : (a == 1 ? U[1] : U[2]);
    bsum[tid] = -(k == 0 ? static_cast<double>(pc.D1) * ta * tF : gam * (Fa - eig * ta * tF));
    if (out.x0) {
      const double tU = t[0] * U[0] + t[1] * U[1] + t[2] * U[2];
      asum[tid] = k == 0 ? static_cast<double>(pc.D1) * ta * total(1, NS - 1) : gam * (Ua - eig * ta * tU);
    }
  } else if (csum) {  // sums of Phi_0 F/2 (kk = 0), then Theta_0 F/2 (kk = 1)
    const int q = tid - 3 * N;
    csum[q] = q < 3 ? total(0, q) : total(1, q - 3);
  }
}

template <int N, bool HALF>
__global__ __launch_bounds__(kFarThreads, 2) void assemble_far_kernel(
    int M, int64_t Lp, int variant, const double* __restrict__ pos, const double* __restrict__ ori, float* __restrict__ T,
    double* __restrict__ bpart, int jgroup, int slot0, PhysConsts pc, float* __restrict__ Tv,
    double* __restrict__ cpart, const double* __restrict__ x0, double* __restrict__ apart,
    _Float16* __restrict__ T16, float* __restrict__ S16) {
  constexpr int NC = 3 + 6 * (N - 1);
  const int i = blockIdx.x, slot = slot0 + blockIdx.y;
  const int jb = blockIdx.y * jgroup, je = min(M, jb + jgroup);
  const int64_t base = static_cast<int64_t>(i) * NC * Lp;
  const int64_t row = (static_cast<int64_t>(slot) * M + i) * 3 * N;
  FarOut out{T + base,
             Tv ? Tv + static_cast<int64_t>(i) * 12 * Lp : nullptr,
             HALF ? T16 + base : nullptr,
             HALF ? S16 + static_cast<int64_t>(i) * M : nullptr,
             x0,
             static_cast<uint32_t>(Lp)};
  assemble_far_block<N, HALF>(i, jb, je, variant, pos, ori, out, pc, bpart + row,
                              cpart ? cpart + (static_cast<int64_t>(slot) * M + i) * 6 : nullptr,
                              apart ? apart + row : nullptr);
}

// Serving: workgroup = (suspension, target fiber), every source.  The far sums
// go where the near kernel, which follows, reads them: b, cpart, and the
// target's rows of V_0 for the product with x0.
template <int N>
__global__ __launch_bounds__(kFarThreads, 2) void assemble_far_batch_kernel(const SusDev* __restrict__ sus,
                                                                            const int2* __restrict__ targets,
                                                                            int variant, PhysConsts pc) {
  constexpr int NC = 3 + 6 * (N - 1);
  const int2 e = targets[blockIdx.x];
  const SusDev& d = sus[e.x];
  const int i = e.y;
  FarOut out{d.T + static_cast<int64_t>(i) * NC * d.Lp, d.Tv + static_cast<int64_t>(i) * 12 * d.Lp, nullptr, nullptr,
             d.x0, static_cast<uint32_t>(d.Lp)};
  assemble_far_block<N, false>(i, 0, d.M, variant, d.pos, d.ori, out, pc, d.b + static_cast<int64_t>(i) * 3 * N,
                               d.cpart + static_cast<int64_t>(i) * 6, d.V + static_cast<int64_t>(i) * 3 * N);
}

// Sources per workgroup: all of them once the targets alone give the chip two
// rounds (two workgroups of a CU at a time), else a multiple of the 256 that
// one step classifies.
PairGrid far_grid(int M) {
  PairGrid g;
  g.tiles = M;
  int groups = (1024 + M - 1) / M;
  const int most = (M + kFarThreads - 1) / kFarThreads;
  if (groups > most) groups = most;
  int jg = (M + groups - 1) / groups;
  jg = (jg + kFarThreads - 1) / kFarThreads * kFarThreads;
  g.jgroup = jg;
  g.groups = (M + jg - 1) / jg;
  return g;
}

static int far_variant(int NQI, bool analytical) {
  return (NQI == 4 ? 0 : (NQI == 8 ? 2 : 4)) + (analytical ? 1 : 0);
}

hipError_t launch_assemble_far(int N, int NQI, bool analytical, int M, int64_t Lp, const double* pos,
                               const double* ori, float* T, double* bpart, int slot0, float* Tv, double* cpart,
                               const double* x0, double* apart, const PhysConsts& pc, hipStream_t s, _Float16* T16,
                               float* S16) {
  if (!assemble_supported(N, NQI)) return hipErrorInvalidValue;
  const PairGrid g = far_grid(M);
  const dim3 grid(M, g.groups), block(kFarThreads);
  const int variant = far_variant(NQI, analytical);
  switch (N) {
#define RF_FAR(NN)                                                                                                  \
  case NN:                                                                                                          \
    if (T16)                                                                                                        \
      hipLaunchKernelGGL((assemble_far_kernel<NN, true>), grid, block, 0, s, M, Lp, variant, pos, ori, T, bpart,     \
                         g.jgroup, slot0, pc, Tv, cpart, x0, apart, T16, S16);                                      \
    else                                                                                                            \
      hipLaunchKernelGGL((assemble_far_kernel<NN, false>), grid, block, 0, s, M, Lp, variant, pos, ori, T, bpart,    \
                         g.jgroup, slot0, pc, Tv, cpart, x0, apart, T16, S16);                                      \
    break;
    RF_FAR(1)
    RF_FAR(2)
    RF_FAR(3)
    RF_FAR(4)
    RF_FAR(5)
    RF_FAR(6)
    RF_FAR(7)
    RF_FAR(8)
#undef RF_FAR
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_assemble_far_batch(int N, int NQI, bool analytical, int ntargets, const SusDev* sus,
                                     const int2* targets, const PhysConsts& pc, hipStream_t s) {
  if (!assemble_supported(N, NQI)) return hipErrorInvalidValue;
  const int variant = far_variant(NQI, analytical);
  switch (N) {
#define RF_FAR(NN)                                                                                              \
  case NN:                                                                                                      \
    hipLaunchKernelGGL((assemble_far_batch_kernel<NN>), dim3(ntargets), dim3(kFarThreads), 0, s, sus, targets, \
                       variant, pc);                                                                            \
    break;
    RF_FAR(1)
    RF_FAR(2)
    RF_FAR(3)
    RF_FAR(4)
    RF_FAR(5)
    RF_FAR(6)
    RF_FAR(7)
    RF_FAR(8)
#undef RF_FAR
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace rf
