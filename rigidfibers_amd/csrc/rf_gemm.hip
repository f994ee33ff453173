// rf_gemm.hip -- C -= A B (or C = A B) on MFMA for the LU factorisation.
//
// The operands are packed K-contiguous: row r of At holds A[r][0..K) and row c
// of Bt holds B[0..K)[c] (the LU writes these packs while it solves its
// triangular blocks), in the element type of the mode:
//   float    v_mfma_f32_32x32x2_f32    (the plain FP32 --magma path)
//   __bf16   v_mfma_f32_32x32x16_bf16
//   _Float16 v_mfma_f32_32x32x16_f16
// always with FP32 accumulation into the FP32 C (column-major, ldc).
//
// Per-block scaling: the packs of the mixed modes may hold each 32-row block
// of A (32-column block of B) multiplied by a power of two, sa[r / 32]
// (sb[c / 32]); the epilogue multiplies each 32 x 32 accumulator block by
// 1 / (sa sb), exactly, before it updates C.
//
// Tiling: a workgroup of 2 x 2 wavefronts owns a TILE x TILE tile of C (256,
// 128 or 64, see launch_gemm); each wavefront computes (TILE / 2)^2 of it as
// 32x32 MFMA blocks.  K advances in stages of 128 bytes per row (64 BF16/FP16
// or 32 FP32 values).  What bounds the 2-byte types at TILE = 256 is the LDS
// (128 bytes per clock and CU): a stage is 2048 clocks of MFMA; four wavefronts
// of 128x128 read 128 KB of fragments and have 64 KB written, 1536 clocks (eight
// of 128x64, as before: 192 + 64 KB, all 2048).  Therefore:
//   - a stage goes from memory to LDS without registers (16 bytes per lane, a
//     wavefront instruction filling 8 whole 128-byte rows), two buffers, issued
//     for stage s + 2 as soon as every wavefront has read stage s: four
//     fragment steps, 2048 clocks, before it is needed;
//   - the fragments of the next step are read while the MFMAs of this one run
//     (two register sets; reads and loads placed between the MFMAs, since there
//     is one wavefront per SIMD to hide them);
//   - row r holds its 16-byte chunk c in slot c ^ (r / 2) % 8: no padding (which
//     the direct loads cannot write) and no bank conflicts in the reads of 16
//     consecutive rows.
//   - the products are formed transposed (B's fragment first), so that a lane
//     holds rows of C: a wavefront instruction of the epilogue reads or writes
//     two whole 128-byte lines, non-temporally.  C passes the chip once per
//     update; kept out of L2, it no longer evicts the panels: TFLOP/s at
//     m = n = 16 384, K = 3072, BF16: 965 without, 1117 with.
// Measured (BF16 TFLOP/s, eight wavefronts staging through registers before ->
// now): m = n = 24 576, K = 3072: 930 -> 1136; 27 000 x 3072: 948 -> 1061; the
// plain library product (no C read, BF16 result) reaches 1490 there.  FP32: 142
// -> 149 of the 157 peak.
//
// MFMA operand layouts (per lane l):
//   32x32x16 (2-byte types): A[i = l % 32][k = 8 (l / 32) .. +8], likewise B;
//   32x32x2  (FP32): A[i = l % 32][k = l / 32]; a 16-byte read of k = 4 (l / 32)
//            .. +4 feeds four MFMAs, the j-th pairing k = j and k = 4 + j.
//   Output accumulator i: column l % 32, row 8 (i / 4) + 4 (l / 32) + i % 4 (of
//   the transposed product: row of C l % 32, column 8 (i / 4) + ...).
#include <algorithm>
#include <type_traits>

#include "rf_lu.h"

namespace rf {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Tile order: the grid is one-dimensional and each of the 8 XCDs (workgroup w
// runs on XCD w % 8) takes a contiguous run of the tiles ordered in groups of
// kGemmGroupRows row tiles (rows fastest inside a group, then columns), so that
// the workgroups resident on an XCD share a few A and B panels (with K = 3072,
// each 256-row tile's A and B panels are 1.5 MB each: row tiles fastest, the 32
// workgroups on an XCD read 32 different A panels, ~400 MB over the chip, more
// than the 256 MB MALL; groups of 4 rows keep them in it).
constexpr int kGemmGroupRows = 4;
constexpr int kStageBytes = 128;
constexpr int kGemmThreads = 256;
constexpr int kNonTemporal = 2;  // cache policy of the buffer instructions

// s_waitcnt operand: at most n vector-memory operations outstanding, and no LDS
// reads (LGKM0) or any number of them
template <int N, bool LGKM0>
constexpr int wait_vm() {
  return (N & 15) | ((N >> 4) << 14) | 0x70 | (LGKM0 ? 0 : 0xf00);
}

// PERSIST: a grid smaller than the tile count; workgroup b takes the tiles of
// the virtual workgroups b, b + gridDim.x, ... (gridDim.x a multiple of 8, so
// that every one of them runs on b's XCD), with a barrier between tiles.
template <typename T, int TILE, bool STORE, bool PERSIST = false>
__global__ __launch_bounds__(kGemmThreads) void gemm_packed_kernel(int m, int n, int K, const T* __restrict__ At,
                                                                  int64_t ldak, const T* __restrict__ Bt,
                                                                  int64_t ldbk, float* __restrict__ C, int64_t ldc,
                                                                  const float* __restrict__ sa,
                                                                  const float* __restrict__ sb) {
  constexpr int TM = TILE / 64;                     // 32x32 blocks per wavefront along m and n
  constexpr int OP = TILE * kStageBytes;            // bytes per operand and stage
  constexpr int IW = OP / 1024 / 4;                 // direct loads per wavefront, operand and stage
  constexpr int SK = kStageBytes / sizeof(T);       // K per stage
  constexpr int NR = 2 * TM;                        // fragments per step
  constexpr int KJ = std::is_same<T, float>::value ? 4 : 1;
  constexpr int MF = TM * TM * KJ;                  // MFMAs per step
  __shared__ __attribute__((aligned(1024))) char lds[2][2][OP];  // [buffer][operand]

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave & 1) * (TILE / 2), wn = (wave >> 1) * (TILE / 2);
  for (int vw = static_cast<int>(blockIdx.x);; vw += static_cast<int>(gridDim.x)) {  // virtual workgroup
    const int mt = (m + TILE - 1) / TILE, nt = (n + TILE - 1) / TILE, tiles = mt * nt;
    const int per = (tiles + 7) / 8;
    if constexpr (PERSIST) {
      if (vw >= 8 * per) return;                                // every virtual workgroup done
      if (vw != static_cast<int>(blockIdx.x)) __syncthreads();  // the previous tile's LDS reads are done
    }
    const int v = (vw & 7) * per + (vw >> 3);  // this XCD's run of the grouped order
    if (v >= tiles) {                          // padding of the grid (the whole workgroup)
      if constexpr (PERSIST) continue;
      return;
    }
    const int first = v / (kGemmGroupRows * nt) * kGemmGroupRows;
    const int rows = min(kGemmGroupRows, mt - first);
    const int within = v - first * nt;
    const int64_t m0 = static_cast<int64_t>(first + within % rows) * TILE;
    const int64_t n0 = static_cast<int64_t>(within / rows) * TILE;

    v16f acc[TM][TM];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

    // Direct loads: wavefront instruction i fills rows 8 (wave IW + i) .. +8, lane l
    // the slot l % 8 of row l / 8.  Rows past m (columns past n) of a ragged edge
    // tile load the last valid row (column) instead: they only feed accumulators
    // that the epilogue does not store.  Offsets from the tile's first row: below
    // 2^31 (the launch checks it).
    int ao[IW], bo[IW];
#pragma unroll
    for (int i = 0; i < IW; ++i) {
      const int row = 8 * (wave * IW + i) + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
      ao[i] = static_cast<int>(min(static_cast<int64_t>(row), m - m0 - 1) * ldak * sizeof(T)) + 16 * ch;
      bo[i] = static_cast<int>(min(static_cast<int64_t>(row), n - n0 - 1) * ldbk * sizeof(T)) + 16 * ch;
    }
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t ar =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(At) + m0 * ldak, 0, 0x7fffffff, 0x00027000);
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t br =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(Bt) + n0 * ldbk, 0, 0x7fffffff, 0x00027000);
    // load q of 2 IW of stage s into buffer buf
    auto load = [&](int buf, int s, int q) {
#if defined(__HIP_DEVICE_COMPILE__)  // the 16-byte form does not exist for the host pass
      const int i = q >> 1;
      auto* dst = (__attribute__((address_space(3))) void*)&lds[buf][q & 1][1024 * (wave * IW + i)];
      if (q & 1)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(br, dst, 16, bo[i], s * kStageBytes, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, dst, 16, ao[i], s * kStageBytes, 0, 0);
#endif
    };
    using Frag = typename std::conditional<
        std::is_same<T, float>::value, v4f,
        typename std::conditional<std::is_same<T, __bf16>::value, v8bf, v8h>::type>::type;
    Frag fa[2][TM], fb[2][TM];
    // fragment q of step kk (32 bytes of K) into register set `set`
    auto read = [&](auto set, int buf, int kk, int q) {
      constexpr int st = decltype(set)::value;
      const int op = q < TM ? 1 : 0;
      const int r = (op ? wn + 32 * q : wm + 32 * (q - TM)) + (lane & 31), ch = 2 * kk + (lane >> 5);
      const Frag f = *reinterpret_cast<const Frag*>(&lds[buf][op][r * kStageBytes + 16 * (ch ^ ((r >> 1) & 7))]);
      if (q < TM)
        fb[st][q] = f;
      else
        fa[st][q - TM] = f;
    };
    auto mma = [&](auto set, int q) {
      constexpr int st = decltype(set)::value;
      const int j = q / (TM * TM), ta = q / TM % TM, tb = q % TM;
      if constexpr (std::is_same<T, float>::value)
        acc[ta][tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[st][tb][j], fa[st][ta][j], acc[ta][tb], 0, 0, 0);
      else if constexpr (std::is_same<T, __bf16>::value)
        acc[ta][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[st][tb], fa[st][ta], acc[ta][tb], 0, 0, 0);
      else
        acc[ta][tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[st][tb], fa[st][ta], acc[ta][tb], 0, 0, 0);
    };
    // one step: the MFMAs of set `use`; between them the reads of step kk (buffer
    // rbuf) into the other set and, with LOADS, the loads of stage ls into lbuf
    auto step = [&](auto use, auto next, auto loads, int rbuf, int kk, int lbuf, int ls) {
#pragma unroll
      for (int g = 0; g < NR; ++g) {
        read(next, rbuf, kk, g);
        if constexpr (decltype(loads)::value)
#pragma unroll
          for (int q = g * 2 * IW / NR; q < (g + 1) * 2 * IW / NR; ++q) load(lbuf, ls, q);
#pragma unroll
        for (int q = g * MF / NR; q < (g + 1) * MF / NR; ++q) mma(use, q);
        __builtin_amdgcn_sched_barrier(0);  // keep the interleaving
      }
    };
    auto barrier = [&]() {  // nothing moves across it in either compiler layer
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    constexpr std::true_type kLoads{};
    constexpr std::false_type kNoLoads{};
    const int stages = K / SK;
#pragma unroll
    for (int q = 0; q < 2 * IW; ++q) load(0, 0, q);
#pragma unroll
    for (int q = 0; q < 2 * IW; ++q) load(1, min(1, stages - 1), q);
    __builtin_amdgcn_s_waitcnt(wait_vm<2 * IW, false>());  // stage 0 has landed
    barrier();
#pragma unroll
    for (int q = 0; q < NR; ++q) read(S0{}, 0, 0, q);
    for (int s = 0; s < stages; ++s) {
      const int cur = s & 1;
      step(S0{}, S1{}, kNoLoads, cur, 1, 0, 0);
      step(S1{}, S0{}, kNoLoads, cur, 2, 0, 0);
      step(S0{}, S1{}, kNoLoads, cur, 3, 0, 0);
      // this wavefront's loads of stage s + 1 have landed and its reads of stage s
      // are done; after the barrier, every wavefront's
      __builtin_amdgcn_s_waitcnt(wait_vm<0, true>());
      barrier();
      // past the last stage: loads of the last one again and reads that nothing
      // uses (one form of the loop body; a peeled one spills registers)
      step(S1{}, S0{}, kLoads, cur ^ 1, 0, cur, min(s + 2, stages - 1));
    }
    __builtin_amdgcn_s_waitcnt(wait_vm<0, true>());

    // C -= acc / (sa sb), or C = acc (STORE), one 32x32 block pair per round, the
    // reads two rounds ahead.  In a ragged tile the accesses past m and n get an
    // offset past the buffer's end: the hardware's bounds check drops them.
    const int64_t um = m0 + wm, un = n0 + wn;
    if (um < m && un < n) {
      float w[TM][TM];
#pragma unroll
      for (int ta = 0; ta < TM; ++ta)
#pragma unroll
        for (int tb = 0; tb < TM; ++tb) w[ta][tb] = 1.0f;
      if (!STORE && sa) {
        float ra[TM], rb[TM];
#pragma unroll
        for (int ta = 0; ta < TM; ++ta) ra[ta] = sa[min(um + 32 * ta, static_cast<int64_t>(m) - 1) >> 5];
#pragma unroll
        for (int tb = 0; tb < TM; ++tb) rb[tb] = sb[min(un + 32 * tb, static_cast<int64_t>(n) - 1) >> 5];
#pragma unroll
        for (int ta = 0; ta < TM; ++ta)
#pragma unroll
          for (int tb = 0; tb < TM; ++tb) w[ta][tb] = 1.0f / (ra[ta] * rb[tb]);  // exact: powers of two
      }
      const __amdgpu_buffer_rsrc_t cr =
          __builtin_amdgcn_make_buffer_rsrc(C + (un * ldc + um), 0, 0x7fffffff, 0x00027000);
      const int ld4 = static_cast<int>(ldc) * 4;
      const int loff = (4 * (lane >> 5)) * ld4 + 4 * (lane & 31);
      const int mrow = static_cast<int>(min(static_cast<int64_t>(TILE), m - um)) - (lane & 31);
      const int ncol = static_cast<int>(min(static_cast<int64_t>(TILE), n - un)) - 4 * (lane >> 5);
      constexpr int PB = TM * TM >= 2 ? 2 : 1, ROUNDS = TM * TM / PB;  // blocks per round
      float cv[2][PB][16];
      auto finish = [&](auto whole_tile) {
        constexpr bool whole = decltype(whole_tile)::value;
        auto offset = [&](int row, int col) {
          return whole || (row < mrow && col < ncol) ? loff + 4 * row : static_cast<int>(0x80000000u);
        };
        auto fetch = [&](int r) {
#pragma unroll
          for (int b = 0; b < PB; ++b) {
            const int ta = (r * PB + b) % TM, tb = (r * PB + b) / TM;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int col = 32 * tb + 8 * (i >> 2) + (i & 3);
              cv[r & 1][b][i] = __builtin_bit_cast(
                  float, __builtin_amdgcn_raw_buffer_load_b32(cr, offset(32 * ta, col), col * ld4, kNonTemporal));
            }
          }
        };
        if constexpr (!STORE) {
          fetch(0);
          if (ROUNDS > 1) fetch(1);
        }
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
#pragma unroll
          for (int b = 0; b < PB; ++b) {
            const int ta = (r * PB + b) % TM, tb = (r * PB + b) / TM;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int col = 32 * tb + 8 * (i >> 2) + (i & 3);
              const float x = acc[ta][tb][i];
              const float y = STORE ? x : fmaf(-w[ta][tb], x, cv[r & 1][b][i]);
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, y), cr, offset(32 * ta, col),
                                                    col * ld4, kNonTemporal);
            }
          }
          if constexpr (!STORE)
            if (r + 2 < ROUNDS) fetch(r + 2);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (m0 + TILE <= m && n0 + TILE <= n)
        finish(std::true_type{});
      else
        finish(std::false_type{});
    }
    if constexpr (!PERSIST) return;
  }
}

int gemm_stage_k(LuMode mode) { return mode == LuMode::kFP32 ? kStageBytes / 4 : kStageBytes / 2; }

static int64_t tiles_of(int64_t m, int64_t n, int tile) { return ((m + tile - 1) / tile) * ((n + tile - 1) / tile); }

template <typename T, int TILE, bool STORE, bool PERSIST>
static void launch_tile(int64_t workgroups, int64_t m, int64_t n, int64_t K, const void* At, int64_t ldak,
                        const void* Bt, int64_t ldbk, float* C, int64_t ldc, const float* sa, const float* sb,
                        hipStream_t s) {
  hipLaunchKernelGGL((gemm_packed_kernel<T, TILE, STORE, PERSIST>), dim3(static_cast<unsigned>(workgroups)),
                     dim3(kGemmThreads), 0, s, static_cast<int>(m), static_cast<int>(n), static_cast<int>(K),
                     static_cast<const T*>(At), ldak, static_cast<const T*>(Bt), ldbk, C, ldc, sa, sb);
}

// The tile.  256 reads the operands the least, but leaves CUs idle while there
// are few tiles and takes a CU for itself (128 KB of LDS), so that nothing runs
// beside its epilogue; two workgroups of 128 share a CU; 64 is for sizes whose
// 128-tiles do not fill the chip.  Measured, us at 64 / 128 / 256:
//   FP32   476 x 476, K = 1024 25 / 68 / 243; 1976^2, 1024 78 / 84 / 265;
//          6000 x 1024, 1024 113 / 138 / 262 (376 tiles of 128: the second round of
//          512 is nearly empty); 3000^2, 3072 452 / 536 / 706 (576); 12 000 x 1024,
//          1024 211 / 212 / 257 (752); 6000^2, 3072 1665 / 1570 / 2115 (2209);
//          24 576^2, 3072 25 677 / 24 919 / 25 101: 64 below 704 tiles of 128,
//          256 from 16 384 tiles of 256 (32 768^2), where the panels outgrow the
//          MALL (the LU at n = 75 000: 2207 ms with 128, 2115 with 256), else 128;
//   BF16   476^2, 1024 10 / 15 / 36; 1976 x 1024, 1024 11.0 / 12.6 / 27 (128 tiles
//          of 128); 3976 x 1024, 1024 17.2 / 15.3 / 27.5 (256); 72 000 x 1024, 1024
//          227 / 162 / 186; 27 000 x 1024, 2048 188 / 140 / 164; 6000^2, 3072 354 /
//          248 / 290 (576 tiles of 256); 27 000 x 3072, 3072 766 / 497 / 480
//          (1272); 24 576^2, 3072 5871 / 3640 / 3266: 64 below 192 tiles of 128, 256
//          from 1024 tiles of 256 at a K of 3072 (a longer loop per epilogue), else
//          128.  A capped grid (one workgroup per CU) takes 256.
template <typename T>
static void launch_gemm(bool store, int64_t m, int64_t n, int64_t K, const void* At, int64_t ldak, const void* Bt,
                        int64_t ldbk, float* C, int64_t ldc, const float* sa, const float* sb, hipStream_t s,
                        int64_t cap) {
  auto go = [&](auto tile_c) {
    constexpr int TILE = decltype(tile_c)::value;
    const int64_t grid = (tiles_of(m, n, TILE) + 7) / 8 * 8;
    if (store)
      launch_tile<T, TILE, true, false>(grid, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s);
    else
      launch_tile<T, TILE, false, false>(grid, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s);
  };
  using Tile64 = std::integral_constant<int, 64>;
  using Tile128 = std::integral_constant<int, 128>;
  const int64_t t128 = tiles_of(m, n, 128);
  if constexpr (std::is_same<T, float>::value) {
    if (t128 < 704)
      go(Tile64{});
    else if (tiles_of(m, n, 256) >= 16384)
      go(std::integral_constant<int, 256>{});
    else
      go(Tile128{});
  } else {
    const int64_t t256 = tiles_of(m, n, 256);
    if (cap > 0 && !store && t256 > cap)  // the persistent form
      launch_tile<T, 256, false, true>(cap, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s);
    else if (t128 < 192)
      go(Tile64{});
    else if (K >= 3072 && t256 >= 1024)
      go(std::integral_constant<int, 256>{});
    else
      go(Tile128{});
  }
}

hipError_t gemm_packed(LuMode mode, bool store, int64_t m, int64_t n, int64_t K, const void* At, int64_t ldak,
                       const void* Bt, int64_t ldbk, float* C, int64_t ldc, hipStream_t s, const float* sa,
                       const float* sb, int max_workgroups) {
  if (m <= 0 || n <= 0 || K <= 0) return hipSuccess;
  const int bk = gemm_stage_k(mode);
  const int64_t esz = mode == LuMode::kFP32 ? 4 : 2;
  // K a whole number of stages; 16-byte aligned operand rows; offsets inside a
  // tile (of 256 rows of a pack, 256 columns of C) below 2^31 bytes
  if (K % bk != 0 || (ldak * esz) % 16 != 0 || (ldbk * esz) % 16 != 0 ||
      (reinterpret_cast<uintptr_t>(At) & 15) != 0 || (reinterpret_cast<uintptr_t>(Bt) & 15) != 0 ||
      m > INT32_MAX || n > INT32_MAX || 256 * std::max(ldak, ldbk) * esz > INT32_MAX || 256 * ldc * 4 > INT32_MAX)
    return hipErrorInvalidValue;
  if ((sa == nullptr) != (sb == nullptr)) return hipErrorInvalidValue;
  const int64_t cap = max_workgroups / 8 * 8;  // a whole number of workgroups per XCD
  switch (mode) {
    case LuMode::kFP32:
      launch_gemm<float>(store, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s, cap);
      break;
    case LuMode::kBF16:
      launch_gemm<__bf16>(store, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s, cap);
      break;
    case LuMode::kFP16:
      launch_gemm<_Float16>(store, m, n, K, At, ldak, Bt, ldbk, C, ldc, sa, sb, s, cap);
      break;
  }
  return hipGetLastError();
}

}  // namespace rf
