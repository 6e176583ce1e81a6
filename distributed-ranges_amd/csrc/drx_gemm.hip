// drx_gemm.hip -- dense row-major product C = alpha * A * B + beta * C on the
// CDNA4 matrix cores: the local tile product behind dr::sp::gemm
// (include/dr/sp/algorithms/matrix/local_gemm.hpp:15-41 custom_gemm,
// c[i][j] += a[i][k] * b[k][j]; :45-60 mkl_gemm, a row-major gemm with
// alpha = beta = 1 and the views' leading dimensions).
//
// Each workgroup owns a BM x BN tile of C; its waves form a WM x WN grid and
// each wave owns (BM/WM) x (BN/WN) as 16 x 16 MFMA tiles
// (v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64). K advances in BK-deep
// stages through two LDS buffers: while the waves multiply out of one buffer,
// the next stage's A and B slices are in flight to registers and are written
// to the other buffer, so each stage costs one barrier.
//
// MFMA 16x16x4 operand layout (64 lanes, g = lane / 16, r = lane % 16):
//   A operand  lane -> A[r][g],   B operand lane -> B[g][r],
//   result     lane, element v -> D[4 g + v][r] (f32), D[g + 4 v][r] (f64).
// The k index the hardware calls g is free to map to any real k as long as A
// and B agree, so lane group g takes the KK consecutive k of its slot: its A
// operands for KK successive instructions come from one 16-byte LDS read.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "drx_common.hpp"
#include "drx_internal.hpp"
#include "drx_spmv.h"

namespace drx {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<float> {
  using acc_t = f32x4;
  static __device__ __forceinline__ acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // Row of the 16 x 16 result that element v of lane group g holds.
  static __device__ __forceinline__ int row(int g, int v) { return 4 * g + v; }
};
template <> struct Mfma<double> {
  using acc_t = f64x4;
  static __device__ __forceinline__ acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int v) { return g + 4 * v; }
};

template <typename T, int BM, int BN, int BK, int WM, int WN>
struct GemmCfg {
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr int V = 16 / static_cast<int>(sizeof(T));  // elements per 16-byte access
  static constexpr int KK = V;                                 // k per lane per A read
  static constexpr int SK = 4 * KK;                            // k per LDS sub-step
  static constexpr int LDA_S = BK + V;  // A tile row stride (elements): one 16-byte pad
  static constexpr int LDB_S = BN + V;  // B tile row stride
  static constexpr int TM = BM / WM, TN = BN / WN;
  static constexpr int FM = TM / 16, FN = TN / 16;
  static constexpr int A_TPR = BK / V, B_TPR = BN / V;  // 16-byte slots per tile row
  static constexpr int A_VECS = BM * BK / V / kThreads;
  static constexpr int B_VECS = BK * BN / V / kThreads;
  static constexpr int STAGE = BM * LDA_S + BK * LDB_S;  // elements per buffer
  static_assert(BK % SK == 0, "BK must hold whole sub-steps");
  static_assert(TM % 16 == 0 && TN % 16 == 0, "wave tile must be whole MFMA tiles");
  static_assert(A_VECS * V * kThreads == BM * BK, "A stage must split evenly");
  static_assert(B_VECS * V * kThreads == BK * BN, "B stage must split evenly");
  static constexpr int ACC_REGS = FM * FN * 4 * static_cast<int>(sizeof(T)) / 4;
  static_assert(2 * STAGE * sizeof(T) <= 160 * 1024, "two stages must fit 160 KB of LDS");
};

// Tile rows are taken GROUP_M at a time and swept column by column, so the
// workgroups resident on one XCD share A row panels and B column panels in
// that XCD's L2.
constexpr int kGroupM = 8;

// Which part of the product a workgroup computes. The first `main` tiles
// (a multiple of the CUs) are computed whole. The rest would leave most CUs
// idle for the time of a whole tile, so each of them is cut into `parts`
// ranges of k stages: a workgroup writes its range's sums to slot u of a
// workspace (BM x BN elements each), and k_gemm_reduce adds the parts in
// order. FP32, whole tiles only -> cut (us): 2000^3 262 -> 164, 1000^3 144 -> 41,
// 203 x 295 x 4502 703 -> 36, 96 x 5000 x 5000 653 -> 78; FP64 540 -> 287, 292 ->
// 61, 1375 -> 44, 1280 -> 131.
struct GemmGrid {
  int64_t tiles_m, tiles_n;
  int64_t main, main_xcd;  // whole tiles; per XCD
  int64_t tail_xcd;        // parts of the other tiles per XCD
  int parts;
};
struct GemmPart {
  int64_t m0, n0;     // first row and column of the tile
  int64_t kt0, kt1;   // stages
  int64_t slot;       // workspace slot, -1: the whole tile goes to C
};
template <int BM, int BN>
__device__ __forceinline__ void gemm_tile_at(const GemmGrid &g, int64_t tile, int64_t &m0,
                                             int64_t &n0) {
  const int64_t per_group = int64_t(kGroupM) * g.tiles_n;
  const int64_t first = tile / per_group * kGroupM;
  const int64_t gsz = g.tiles_m - first < kGroupM ? g.tiles_m - first : kGroupM;
  const int64_t in_g = tile % per_group;
  m0 = (first + in_g % gsz) * BM;
  n0 = (in_g / gsz) * BN;
}
// false: nothing to do (the whole workgroup leaves together).
template <int BM, int BN>
__device__ __forceinline__ bool gemm_part(const GemmGrid &g, int64_t nk, GemmPart &p) {
  const int64_t whole = g.main_xcd * kXcds;
  int64_t tile;
  if (blockIdx.x < whole) {
    tile = map_block(blockIdx.x, g.main_xcd);
    if (tile >= g.main) return false;
    p.kt0 = 0;
    p.kt1 = nk;
    p.slot = -1;
  } else {
    p.slot = map_block(blockIdx.x - whole, g.tail_xcd);
    tile = g.main + p.slot / g.parts;
    if (tile >= g.tiles_m * g.tiles_n) return false;
    const int64_t part = p.slot % g.parts;
    p.kt0 = nk * part / g.parts;
    p.kt1 = nk * (part + 1) / g.parts;
  }
  gemm_tile_at<BM, BN>(g, tile, p.m0, p.n0);
  return true;
}

// C of the tiles that were cut: the parts' sums in order, then alpha and beta
// as in the kernels' own epilogue. A wave reads 64 consecutive elements of a
// tile row.
template <typename T, int BM, int BN>
__global__ void k_gemm_reduce(int64_t m, int64_t n, T alpha, T beta, T *__restrict__ C,
                              int64_t ldc, GemmGrid g, const T *__restrict__ ws) {
  const int64_t tiles = g.tiles_m * g.tiles_n - g.main;
  const int64_t total = tiles * BM * BN;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = i / (BM * BN), e = i % (BM * BN);
    int64_t m0, n0;
    gemm_tile_at<BM, BN>(g, g.main + t, m0, n0);
    const int64_t gi = m0 + e / BN, gj = n0 + e % BN;
    if (gi >= m || gj >= n) continue;
    const T *p = ws + t * g.parts * (BM * BN) + e;
    T sum = p[0];
    for (int q = 1; q < g.parts; q++) sum += p[static_cast<int64_t>(q) * (BM * BN)];
    T &c = C[gi * ldc + gj];
    const T prod = alpha * sum;
    c = beta == T(0) ? prod : prod + beta * c;
  }
}

// Waves per SIMD the register budget is held to, from the accumulator
// registers per lane: 64 -> 4 waves with eight-wave workgroups, 3 with
// four-wave ones (their lanes carry more of each stage's loads; 4 would
// spill); 128 -> 2; more -> 1.
template <int ACC_REGS, int THREADS> constexpr int gemm_waves() {
  return ACC_REGS <= 64 ? (THREADS >= 512 ? 4 : 3) : ACC_REGS <= 128 ? 2 : 1;
}

template <typename T, int BM, int BN, int BK, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN)
    __attribute__((amdgpu_waves_per_eu(
        gemm_waves<GemmCfg<T, BM, BN, BK, WM, WN>::ACC_REGS, 64 * WM * WN>())))
    k_gemm(int64_t m, int64_t n, int64_t K, T alpha, const T *__restrict__ A,
           int64_t lda, const T *__restrict__ B, int64_t ldb, T beta,
           T *__restrict__ C, int64_t ldc, GemmGrid grid, T *__restrict__ ws) {
  using Cfg = GemmCfg<T, BM, BN, BK, WM, WN>;
  using vec_t = T __attribute__((ext_vector_type(Cfg::V)));
  // Rows of A and B start anywhere (any leading dimension): 16-byte loads at
  // element alignment, which global memory serves. Loading rows that are not
  // 16-byte aligned element by element ran 4099 x 3001 x 2050 FP32 at 53
  // TFLOP/s.
  typedef vec_t mem_t __attribute__((aligned(sizeof(T))));
  using acc_t = typename Mfma<T>::acc_t;
  __shared__ __attribute__((aligned(16))) T smem[2 * Cfg::STAGE];

  const int64_t nk = (K + BK - 1) / BK;
  GemmPart part;
  if (!gemm_part<BM, BN>(grid, nk, part)) return;
  const int64_t m0 = part.m0, n0 = part.n0;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int wm = wave / WN, wn = wave % WN;
  // Full stages load 16 bytes per slot wherever the tile lies: rows of A past
  // m read row m - 1, slots of B past n the row's last whole slot (their
  // products are never stored), and a slot across column n reads on into the
  // next row -- so not in the stage that holds B's last row, which like a
  // partial last stage is loaded with a check per slot. (With a check per
  // slot in every stage of the edge tiles 4100 x 3004 x 2052 FP32 took 585 us
  // where 4096 x 3072 x 2048 took 425; now 446.)
  const bool n_inner = n0 + BN <= n;
  const T *a_src[Cfg::A_VECS], *b_src[Cfg::B_VECS];
#pragma unroll
  for (int p = 0; p < Cfg::A_VECS; ++p) {
    const int q = tid + p * Cfg::kThreads;
    const int64_t gi = m0 + q / Cfg::A_TPR;
    a_src[p] = A + (gi < m ? gi : m - 1) * lda + (q % Cfg::A_TPR) * Cfg::V;
  }
#pragma unroll
  for (int p = 0; p < Cfg::B_VECS; ++p) {
    const int q = tid + p * Cfg::kThreads;
    const int64_t gj = n0 + (q % Cfg::B_TPR) * Cfg::V;
    b_src[p] = B + (q / Cfg::B_TPR) * ldb + (gj < n ? gj : n - Cfg::V);
  }
  // stages [0, nwhole) load whole slots
  const int64_t nwhole = n < Cfg::V ? 0 : n_inner ? K / BK : (K - 1) / BK;
  vec_t ra[Cfg::A_VECS], rb[Cfg::B_VECS];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int p = 0; p < Cfg::A_VECS; ++p)
      ra[p] = *reinterpret_cast<const mem_t *>(a_src[p] + k0);
#pragma unroll
    for (int p = 0; p < Cfg::B_VECS; ++p)
      rb[p] = *reinterpret_cast<const mem_t *>(b_src[p] + k0 * ldb);
  };
  auto a_at = [&](T *st, int q) {
    return reinterpret_cast<vec_t *>(st + (q / Cfg::A_TPR) * Cfg::LDA_S + (q % Cfg::A_TPR) * Cfg::V);
  };
  auto b_at = [&](T *st, int q) {
    return reinterpret_cast<vec_t *>(st + BM * Cfg::LDA_S + (q / Cfg::B_TPR) * Cfg::LDB_S +
                                     (q % Cfg::B_TPR) * Cfg::V);
  };
  auto store = [&](T *st) {
#pragma unroll
    for (int p = 0; p < Cfg::A_VECS; ++p) *a_at(st, tid + p * Cfg::kThreads) = ra[p];
#pragma unroll
    for (int p = 0; p < Cfg::B_VECS; ++p) *b_at(st, tid + p * Cfg::kThreads) = rb[p];
  };
  // A stage with a check per slot, straight to LDS.
  auto load_checked = [&](int64_t k0, T *st) {
#pragma unroll
    for (int p = 0; p < Cfg::A_VECS; ++p) {
      const int q = tid + p * Cfg::kThreads;
      const int64_t gi = m0 + q / Cfg::A_TPR, gk = k0 + (q % Cfg::A_TPR) * Cfg::V;
      vec_t v;
      if (gi < m && gk + Cfg::V <= K) {
        v = *reinterpret_cast<const mem_t *>(A + gi * lda + gk);
      } else {
#pragma unroll
        for (int e = 0; e < Cfg::V; ++e) v[e] = (gi < m && gk + e < K) ? A[gi * lda + gk + e] : T(0);
      }
      *a_at(st, q) = v;
    }
#pragma unroll
    for (int p = 0; p < Cfg::B_VECS; ++p) {
      const int q = tid + p * Cfg::kThreads;
      const int64_t gk = k0 + q / Cfg::B_TPR, gj = n0 + (q % Cfg::B_TPR) * Cfg::V;
      vec_t v;
      if (gk < K && gj + Cfg::V <= n) {
        v = *reinterpret_cast<const mem_t *>(B + gk * ldb + gj);
      } else {
#pragma unroll
        for (int e = 0; e < Cfg::V; ++e) v[e] = (gk < K && gj + e < n) ? B[gk * ldb + gj + e] : T(0);
      }
      *b_at(st, q) = v;
    }
  };

  acc_t acc[Cfg::FM][Cfg::FN];
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j) acc[i][j] = acc_t{};

  if (part.kt0 < part.kt1) {
    T *st = smem + (part.kt0 & 1) * Cfg::STAGE;
    if (part.kt0 < nwhole) {
      load(part.kt0 * BK);
      store(st);
    } else {
      load_checked(part.kt0 * BK, st);
    }
  }
  __syncthreads();
  auto products = [&](int64_t kt) {
    const T *As = smem + (kt & 1) * Cfg::STAGE;
    const T *Bs = As + BM * Cfg::LDA_S;
#pragma unroll
    for (int s = 0; s < BK / Cfg::SK; ++s) {
      vec_t a[Cfg::FM];
      T b[Cfg::FN][Cfg::KK];
#pragma unroll
      for (int i = 0; i < Cfg::FM; ++i)
        a[i] = *reinterpret_cast<const vec_t *>(
            As + (wm * Cfg::TM + i * 16 + r) * Cfg::LDA_S + s * Cfg::SK + g * Cfg::KK);
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int kk = 0; kk < Cfg::KK; ++kk)
          b[j][kk] = Bs[(s * Cfg::SK + g * Cfg::KK + kk) * Cfg::LDB_S + wn * Cfg::TN + j * 16 + r];
#pragma unroll
      for (int kk = 0; kk < Cfg::KK; ++kk)
#pragma unroll
        for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
          for (int j = 0; j < Cfg::FN; ++j)
            acc[i][j] = Mfma<T>::op(a[i][kk], b[j][kk], acc[i][j]);
    }
  };
  // The stages whose successor loads whole slots, then the rest: with the
  // checked loads in the same loop, every stage waited for its loads before
  // its products (4096^3: FP32 1161 -> 1042 us, FP64 2234 -> 2081).
  int64_t kt = part.kt0;
  for (; kt + 1 < (part.kt1 < nwhole ? part.kt1 : nwhole); ++kt) {
    load((kt + 1) * BK);
    products(kt);
    store(smem + ((kt + 1) & 1) * Cfg::STAGE);
    __syncthreads();
  }
  for (; kt < part.kt1; ++kt) {
    products(kt);
    if (kt + 1 < part.kt1) load_checked((kt + 1) * BK, smem + ((kt + 1) & 1) * Cfg::STAGE);
    __syncthreads();
  }

  // A part of a tile: its sums, to the workspace.
  if (part.slot >= 0) {
    T *p = ws + part.slot * (BM * BN);
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int j = 0; j < Cfg::FN; ++j)
          p[(wm * Cfg::TM + i * 16 + Mfma<T>::row(g, v)) * BN + wn * Cfg::TN + j * 16 + r] =
              acc[i][j][v];
    return;
  }
  // Epilogue: element v of the lane holds D[Mfma<T>::row(g, v)][r] of each
  // MFMA tile. beta == 0 does not read C (so C may hold anything, NaN
  // included), as in BLAS.
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t gi = m0 + wm * Cfg::TM + i * 16 + Mfma<T>::row(g, v);
      if (gi >= m) continue;
      T *crow = C + gi * ldc;
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j) {
        const int64_t gj = n0 + wn * Cfg::TN + j * 16 + r;
        if (gj >= n) continue;
        const T prod = alpha * acc[i][j][v];
        crow[gj] = beta == T(0) ? prod : prod + beta * crow[gj];
      }
    }
  }
}

// Direct-to-LDS variant for FP32, BK = 16, BN = 128 (A stage rows of 64
// bytes, B stage rows of 512 bytes). global_load_lds_dwordx4 writes lane i of
// a wave's instruction to 16 bytes at (wave's 1 KB block) + 16 i, so the LDS
// image is unpadded and each lane picks the global slot that belongs at its
// position. Slot c of a 16-row A block's row r sits at c ^ fa(r); slot c of B
// stage row k at c ^ hb(k). Both swizzles keep the MFMA operand reads free of
// bank conflicts (16 lanes per 256 bytes or 8 per 128 bytes for the 16-byte A
// reads; 64 lanes per 256 bytes for the 4-byte B reads). Full stages load
// this way, with no register round trip; rows past m read row m - 1 instead
// (their products are never stored). Tiles on the n edge and a partial last
// stage load through registers into the same positions, after the stage's
// products, so that those registers are never live beside the operands.
__device__ __forceinline__ int dl_fa(int r) { return ((r >> 1) ^ (r >> 3)) & 3; }
// One 16-byte global -> LDS copy per lane into the wave's 1 KB block at lds.
__device__ __forceinline__ void lds_dma16(const void *src, char *lds) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
__device__ __forceinline__ int dl_hb(int k) { return 4 * ((k >> 2) & 3); }

// Register budget: 3 waves per SIMD (the kernel needs about 136 VGPRs; at
// 128 it spills).
template <int BM, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(3)))
    k_gemm_dl(int64_t m, int64_t n, int64_t K, float alpha, const float *__restrict__ A,
              int64_t lda, const float *__restrict__ B, int64_t ldb, float beta,
              float *__restrict__ C, int64_t ldc, GemmGrid grid, float *__restrict__ ws,
              int vec_ok) {
  constexpr int BN = 128, BK = 16, NW = WM * WN;
  constexpr int A_BYTES = BM * BK * 4, B_BYTES = BK * BN * 4, STAGE = A_BYTES + B_BYTES;
  constexpr int A_INSTR = A_BYTES / 1024 / NW, B_INSTR = B_BYTES / 1024 / NW;
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  static_assert(A_INSTR * NW * 1024 == A_BYTES && B_INSTR * NW * 1024 == B_BYTES,
                "stages must split into whole 1 KB wave blocks");
  static_assert(TM % 16 == 0 && TN % 16 == 0, "wave tile must be whole MFMA tiles");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int64_t nk = (K + BK - 1) / BK;
  GemmPart part;
  if (!gemm_part<BM, BN>(grid, nk, part)) return;
  const int64_t m0 = part.m0, n0 = part.n0;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int wm = wave / WN, wn = wave % WN;
  const bool n_inner = n0 + BN <= n;
  // stage kt straight into LDS (which slots may not: see k_gemm)
  auto direct_ok = [&](int64_t kt) {
    return vec_ok && n >= 4 && ((kt + 1) * BK < K || (n_inner && (kt + 1) * BK == K));
  };

  // The (row, slot) each lane moves: A block p * NW + wave, row block*16 +
  // lane/4, slot (lane%4) ^ fa(lane/4); B block p * NW + wave, row
  // 2 block + lane/32, slot (lane%32) ^ hb(row).
  auto a_row = [&](int p) { return (p * NW + wave) * 16 + (lane >> 2); };
  auto a_col = [&](int) { return 4 * ((lane & 3) ^ dl_fa(lane >> 2)); };
  auto b_row = [&](int p) { return (p * NW + wave) * 2 + (lane >> 5); };
  auto b_col = [&](int p) { return 4 * ((lane & 31) ^ dl_hb(b_row(p))); };
  const float *a_src[A_INSTR];
  const float *b_src[B_INSTR];
#pragma unroll
  for (int p = 0; p < A_INSTR; ++p) {
    const int64_t gi = m0 + a_row(p) < m ? m0 + a_row(p) : m - 1;
    a_src[p] = A + gi * lda + a_col(p);
  }
#pragma unroll
  for (int p = 0; p < B_INSTR; ++p) {
    const int64_t gj = n0 + b_col(p);
    b_src[p] = B + b_row(p) * ldb + (gj < n ? gj : (n - 4) / 4 * 4);
  }

  auto issue_direct = [&](int64_t k0, char *st) {
#pragma unroll
    for (int p = 0; p < A_INSTR; ++p)
      lds_dma16(a_src[p] + k0, st + (p * NW + wave) * 1024);
#pragma unroll
    for (int p = 0; p < B_INSTR; ++p)
      lds_dma16(b_src[p] + k0 * ldb, st + A_BYTES + (p * NW + wave) * 1024);
  };

  f32x4 ra[A_INSTR], rb[B_INSTR];
  auto load_regs = [&](int64_t k0) {
#pragma unroll
    for (int p = 0; p < A_INSTR; ++p) {
      const int64_t gi = m0 + a_row(p), gk = k0 + a_col(p);
      if (vec_ok && gi < m && gk + 4 <= K) {
        ra[p] = *reinterpret_cast<const f32x4 *>(A + gi * lda + gk);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) ra[p][e] = (gi < m && gk + e < K) ? A[gi * lda + gk + e] : 0.f;
      }
    }
#pragma unroll
    for (int p = 0; p < B_INSTR; ++p) {
      const int64_t gk = k0 + b_row(p), gj = n0 + b_col(p);
      if (vec_ok && gk < K && gj + 4 <= n) {
        rb[p] = *reinterpret_cast<const f32x4 *>(B + gk * ldb + gj);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) rb[p][e] = (gk < K && gj + e < n) ? B[gk * ldb + gj + e] : 0.f;
      }
    }
  };
  auto store_regs = [&](char *st) {
#pragma unroll
    for (int p = 0; p < A_INSTR; ++p)
      *reinterpret_cast<f32x4 *>(st + (p * NW + wave) * 1024 + lane * 16) = ra[p];
#pragma unroll
    for (int p = 0; p < B_INSTR; ++p)
      *reinterpret_cast<f32x4 *>(st + A_BYTES + (p * NW + wave) * 1024 + lane * 16) = rb[p];
  };

  // Operand offsets (bytes within a stage) of this lane. Row block i of the
  // wave's A tile is a_off + 1024 i; B row 4 g + kk of column tile j is
  // b_off[j] + 512 kk (hb is the same for the four rows of lane group g).
  const int a_off = wm * TM / 16 * 1024 + r * 64 + (g ^ dl_fa(r)) * 16;
  int b_off[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = wn * TN + j * 16 + r;
    b_off[j] = A_BYTES + 4 * g * 512 + (((col >> 2) ^ dl_hb(4 * g)) * 16) + (col & 3) * 4;
  }

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{};

  if (part.kt0 < part.kt1) {
    char *st = smem + (part.kt0 & 1) * STAGE;
    if (direct_ok(part.kt0)) {
      issue_direct(part.kt0 * BK, st);
    } else {
      load_regs(part.kt0 * BK);
      store_regs(st);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int64_t kt = part.kt0; kt < part.kt1; ++kt) {
    const char *cur = smem + (kt & 1) * STAGE;
    char *nxt = smem + ((kt + 1) & 1) * STAGE;
    const bool more = kt + 1 < part.kt1;
    const bool direct = more && direct_ok(kt + 1);
    if (direct) issue_direct((kt + 1) * BK, nxt);
    f32x4 a[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) a[i] = *reinterpret_cast<const f32x4 *>(cur + a_off + i * 1024);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      float b[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = *reinterpret_cast<const float *>(cur + b_off[j] + kk * 512);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<float>::op(a[i][kk], b[j], acc[i][j]);
    }
    if (more && !direct) {
      load_regs((kt + 1) * BK);
      store_regs(nxt);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  if (part.slot >= 0) {
    float *p = ws + part.slot * (BM * BN);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          p[(wm * TM + i * 16 + Mfma<float>::row(g, v)) * BN + wn * TN + j * 16 + r] =
              acc[i][j][v];
    return;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t gi = m0 + wm * TM + i * 16 + Mfma<float>::row(g, v);
      if (gi >= m) continue;
      float *crow = C + gi * ldc;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int64_t gj = n0 + wn * TN + j * 16 + r;
        if (gj >= n) continue;
        const float prod = alpha * acc[i][j][v];
        crow[gj] = beta == 0.f ? prod : prod + beta * crow[gj];
      }
    }
  }
}

// FP64 direct-to-LDS variant, BK = 16, BN = 128: A stage rows of 128 bytes
// (8 slots; a wave's 1 KB block holds 8 rows), B stage rows of 1 KB (one per
// block). Slot c of A row r (r mod 16 within its MFMA tile) sits at
// c ^ fa64(r); slot c of B row k at c ^ hb64(k). The 16-byte A reads (two
// k per lane) and the 8-byte B reads stay free of bank conflicts for 8 or
// 16 lanes per 128 or 256 bytes.
__device__ __forceinline__ int dl64_fa(int r) { return (r ^ (r >> 3)) & 7; }
__device__ __forceinline__ int dl64_hb(int k) { return 8 * ((k >> 1) & 1); }

template <int BM, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2)))
    k_gemm_dl64(int64_t m, int64_t n, int64_t K, double alpha, const double *__restrict__ A,
                int64_t lda, const double *__restrict__ B, int64_t ldb, double beta,
                double *__restrict__ C, int64_t ldc, GemmGrid grid, double *__restrict__ ws,
                int vec_ok) {
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  constexpr int BN = 128, BK = 16, NW = WM * WN;
  constexpr int A_BYTES = BM * BK * 8, B_BYTES = BK * BN * 8, STAGE = A_BYTES + B_BYTES;
  constexpr int A_INSTR = A_BYTES / 1024 / NW, B_INSTR = B_BYTES / 1024 / NW;
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  static_assert(A_INSTR * NW * 1024 == A_BYTES && B_INSTR * NW * 1024 == B_BYTES,
                "stages must split into whole 1 KB wave blocks");
  static_assert(TM % 16 == 0 && TN % 16 == 0, "wave tile must be whole MFMA tiles");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int64_t nk = (K + BK - 1) / BK;
  GemmPart part;
  if (!gemm_part<BM, BN>(grid, nk, part)) return;
  const int64_t m0 = part.m0, n0 = part.n0;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int wm = wave / WN, wn = wave % WN;
  const bool n_inner = n0 + BN <= n;
  // stage kt straight into LDS (which slots may not: see k_gemm)
  auto direct_ok = [&](int64_t kt) {
    return vec_ok && n >= 2 && ((kt + 1) * BK < K || (n_inner && (kt + 1) * BK == K));
  };

  // A block p * NW + wave: rows block*8 + lane/8, slot (lane%8) ^ fa64(row);
  // B block p * NW + wave: row = block, slot lane ^ hb64(row).
  auto a_row = [&](int p) { return (p * NW + wave) * 8 + (lane >> 3); };
  auto a_col = [&](int p) { return 2 * ((lane & 7) ^ dl64_fa(a_row(p) & 15)); };
  auto b_row = [&](int p) { return p * NW + wave; };
  auto b_col = [&](int p) { return 2 * (lane ^ dl64_hb(b_row(p))); };
  const double *a_src[A_INSTR];
  const double *b_src[B_INSTR];
#pragma unroll
  for (int p = 0; p < A_INSTR; ++p) {
    const int64_t gi = m0 + a_row(p) < m ? m0 + a_row(p) : m - 1;
    a_src[p] = A + gi * lda + a_col(p);
  }
#pragma unroll
  for (int p = 0; p < B_INSTR; ++p) {
    const int64_t gj = n0 + b_col(p);
    b_src[p] = B + b_row(p) * ldb + (gj < n ? gj : (n - 2) / 2 * 2);
  }

  auto issue_direct = [&](int64_t k0, char *st) {
#pragma unroll
    for (int p = 0; p < A_INSTR; ++p) lds_dma16(a_src[p] + k0, st + (p * NW + wave) * 1024);
#pragma unroll
    for (int p = 0; p < B_INSTR; ++p)
      lds_dma16(b_src[p] + k0 * ldb, st + A_BYTES + (p * NW + wave) * 1024);
  };
  auto load_store_regs = [&](int64_t k0, char *st) {
#pragma unroll
    for (int p = 0; p < A_INSTR; ++p) {
      const int64_t gi = m0 + a_row(p), gk = k0 + a_col(p);
      f64x2 v;
      if (vec_ok && gi < m && gk + 2 <= K) {
        v = *reinterpret_cast<const f64x2 *>(A + gi * lda + gk);
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e) v[e] = (gi < m && gk + e < K) ? A[gi * lda + gk + e] : 0.0;
      }
      *reinterpret_cast<f64x2 *>(st + (p * NW + wave) * 1024 + lane * 16) = v;
    }
#pragma unroll
    for (int p = 0; p < B_INSTR; ++p) {
      const int64_t gk = k0 + b_row(p), gj = n0 + b_col(p);
      f64x2 v;
      if (vec_ok && gk < K && gj + 2 <= n) {
        v = *reinterpret_cast<const f64x2 *>(B + gk * ldb + gj);
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e) v[e] = (gk < K && gj + e < n) ? B[gk * ldb + gj + e] : 0.0;
      }
      *reinterpret_cast<f64x2 *>(st + A_BYTES + (p * NW + wave) * 1024 + lane * 16) = v;
    }
  };

  // Operand offsets (bytes within a stage). A row block i of the wave at
  // a_off[s] + 2048 i for sub-step s (slot 4 s + g, i.e. bit 2 flipped for
  // s = 1); B row 8 s + 2 g + kk of column tile j at b_off[j] + 1024 (8 s + kk)
  // (hb64 is the same for all of lane group g's rows).
  const int a_base = (wm * TM + r) * 128;
  const int a_off0 = a_base + ((g ^ dl64_fa(r)) * 16);
  const int a_off1 = a_base + (((g ^ dl64_fa(r)) ^ 4) * 16);
  int b_off[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = wn * TN + j * 16 + r;
    b_off[j] = A_BYTES + 2 * g * 1024 + (((col >> 1) ^ dl64_hb(2 * g)) * 16) + (col & 1) * 8;
  }

  f64x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{};

  if (part.kt0 < part.kt1) {
    char *st = smem + (part.kt0 & 1) * STAGE;
    if (direct_ok(part.kt0))
      issue_direct(part.kt0 * BK, st);
    else
      load_store_regs(part.kt0 * BK, st);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int64_t kt = part.kt0; kt < part.kt1; ++kt) {
    const char *cur = smem + (kt & 1) * STAGE;
    char *nxt = smem + ((kt + 1) & 1) * STAGE;
    const bool more = kt + 1 < part.kt1;
    const bool direct = more && direct_ok(kt + 1);
    if (direct) issue_direct((kt + 1) * BK, nxt);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      f64x2 a[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i)
        a[i] = *reinterpret_cast<const f64x2 *>(cur + (s2 ? a_off1 : a_off0) + i * 2048);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        double b[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j)
          b[j] = *reinterpret_cast<const double *>(cur + b_off[j] + (8 * s2 + kk) * 1024);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<double>::op(a[i][kk], b[j], acc[i][j]);
      }
    }
    if (more && !direct) load_store_regs((kt + 1) * BK, nxt);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  if (part.slot >= 0) {
    double *p = ws + part.slot * (BM * BN);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          p[(wm * TM + i * 16 + Mfma<double>::row(g, v)) * BN + wn * TN + j * 16 + r] =
              acc[i][j][v];
    return;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t gi = m0 + wm * TM + i * 16 + Mfma<double>::row(g, v);
      if (gi >= m) continue;
      double *crow = C + gi * ldc;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int64_t gj = n0 + wn * TN + j * 16 + r;
        if (gj >= n) continue;
        const double prod = alpha * acc[i][j][v];
        crow[gj] = beta == 0.0 ? prod : prod + beta * crow[gj];
      }
    }
  }
}

// Tiles whole and in parts: the parts of the tiles beyond the last full round
// of resident workgroups that cost least by this model. A CU works its tiles
// off at one rate, less while few waves share a SIMD (measured: 2000^3, one
// four-wave workgroup per CU, 0.45 of the rate of three), and the cut tiles'
// sums are written and read once more.
constexpr int64_t kLeastStages = 4;
// A product with cut tiles takes at least kCutLeast: two launches and a
// workspace from the pool take the host 29..33 us, a single launch 18 (one call
// after another; the model overstates tiles this small). Tiles across column n
// take their last stage with checks, kEdge more. us per call, one after another,
// before cuts / all that the model without these two cut / now: FP32 512 x 512 x 128
// 22 / 34 / 21, x 224 29 / 33 / 28, x 400 42 / 32 / 32, 500 x 499 x 200 47 / 32 / 34;
// FP64 512 x 512 x 96 27 / 33 / 27, x 160 36 / 33 / 30. Over 15 sizes and 15 k no
// call is slower than before cuts by more than 3 % (kCutLeast 45: FP64 128 x 128 x
// 160 36 us where cut tiles take 29). Single calls that are waited for, whose time
// on the GPU counts too, would gain from cutting earlier: 41.5 us whatever k, against
// 45 for 512 x 512 x 96 FP64 and 39 for x 128 FP32 in one launch.
constexpr double kCutLeast = 40.0, kEdge = 12.0;
struct GemmCost {
  int waves;     // per SIMD and workgroup
  int resident;  // workgroups per CU
  double rate;   // of a busy CU, Tflop/s
};
inline double gemm_time_us(int64_t units, int64_t parts, double tile_us, int64_t cus,
                           const GemmCost &c) {
  constexpr double kEff[5] = {0.45, 0.45, 0.75, 0.95, 1.0};
  const int64_t per_cu = (units + cus - 1) / cus;
  const int64_t waves = std::min<int64_t>(4, std::min<int64_t>(per_cu, c.resident) * c.waves);
  return static_cast<double>(per_cu) / static_cast<double>(parts) * tile_us / kEff[waves];
}
inline void fill_grid(GemmGrid &g) {
  g.main_xcd = (g.main + kXcds - 1) / kXcds;
  g.tail_xcd = ((g.tiles_m * g.tiles_n - g.main) * g.parts + kXcds - 1) / kXcds;
  DRX_REQUIRE((g.main_xcd + g.tail_xcd) * kXcds <= int64_t(0xffffffff),
              "product too large for one launch");
}
inline GemmGrid gemm_grid(int64_t m, int64_t n, int64_t k, int bm, int bn, int bk, size_t esz,
                          int64_t cus, const GemmCost &c) {
  GemmGrid g{};
  g.tiles_m = (m + bm - 1) / bm;
  g.tiles_n = (n + bn - 1) / bn;
  const int64_t tiles = g.tiles_m * g.tiles_n, nk = (k + bk - 1) / bk;
  const int64_t whole = tiles / (c.resident * cus) * (c.resident * cus), rest = tiles - whole;
  const double tile_us = 2e-6 * bm * bn * static_cast<double>(nk * bk) / c.rate;
  g.main = tiles;
  g.parts = 1;
  const double uncut = gemm_time_us(tiles, 1, tile_us, cus, c) + (n % bn != 0 ? kEdge : 0.0);
  const double before = static_cast<double>(whole) / static_cast<double>(cus) * tile_us;
  // the best number of parts first, then whether to cut at all: kCutLeast says
  // nothing about the parts
  double best = 0;
  int parts = 1;
  for (int64_t p = 2; rest > 0 && p <= std::min<int64_t>(64, nk / kLeastStages); p++) {
    const double bytes = 2.0 * static_cast<double>(rest * p) * bm * bn * static_cast<double>(esz);
    const double t = before + gemm_time_us(rest * p, p, tile_us, cus, c) + 6.0 + bytes / 4e6;
    if (parts == 1 || t < best) {
      best = t;
      parts = static_cast<int>(p);
    }
  }
  if (parts > 1 && std::max(kCutLeast, best) < uncut) {
    g.main = whole;
    g.parts = parts;
  }
  fill_grid(g);
  return g;
}
// The same product without cut tiles.
inline GemmGrid whole_grid(GemmGrid g) {
  g.main = g.tiles_m * g.tiles_n;
  g.parts = 1;
  fill_grid(g);
  return g;
}

// Resident workgroups follow from the register budgets (gemm_waves) and the
// 512 registers of a SIMD lane.
template <typename T> constexpr double gemm_rate() { return sizeof(T) == 8 ? 0.26 : 0.52; }
template <typename T, int BM, int BN, int WM, int WN> constexpr GemmCost gemm_cost() {
  constexpr int acc = BM / WM * (BN / WN) / 64 * static_cast<int>(sizeof(T)) / 4;
  constexpr int waves = gemm_waves<acc, 64 * WM * WN>();
  return GemmCost{WM * WN / 4, waves * 4 / (WM * WN) > 0 ? waves * 4 / (WM * WN) : 1,
                  gemm_rate<T>()};
}

inline int gemm_cus() {
  int dev = 0, cus = 0;
  DRX_HIP(hipGetDevice(&dev));
  DRX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return std::max(cus, 1);
}

// Launches `kernel(grid, threads, g, ws)` over the tiles, then the reduction of
// those that were cut.
template <typename T, int BM, int BN, int BK, typename Launch>
void launch_tiles(int64_t m, int64_t n, int64_t k, T alpha, T beta, T *c, int64_t ldc,
                  const GemmCost &cost, hipStream_t s, Launch &&kernel) {
  GemmGrid g = gemm_grid(m, n, k, BM, BN, BK, sizeof(T), gemm_cus(), cost);
  int64_t cut = g.tiles_m * g.tiles_n - g.main;
  T *ws = nullptr;
  if (cut > 0) {
    ws = static_cast<T *>(
        scratch_try(static_cast<size_t>(cut) * g.parts * BM * BN * sizeof(T), s));
    if (ws == nullptr) {  // no memory: all tiles whole
      g = whole_grid(g);
      cut = 0;
    }
  }
  const dim3 grid(static_cast<unsigned>((g.main_xcd + g.tail_xcd) * kXcds));
  if (cut == 0) {
    kernel(grid, g, ws);
    DRX_HIP(hipGetLastError());
    return;
  }
  try {
    kernel(grid, g, ws);
    const int64_t blocks = std::min<int64_t>(cut * (BM * BN / 256), 8192);
    hipLaunchKernelGGL((k_gemm_reduce<T, BM, BN>), dim3(static_cast<unsigned>(blocks)), dim3(256),
                       0, s, m, n, alpha, beta, c, ldc, g, ws);
    DRX_HIP(hipGetLastError());
  } catch (...) {
    scratch_free(ws, s);
    throw;
  }
  scratch_free(ws, s);
}

inline void launch_gemm_dl64(int64_t m, int64_t n, int64_t k, double alpha, const double *a,
                             int64_t lda, const double *b, int64_t ldb, double beta, double *c,
                             int64_t ldc, hipStream_t s) {
  const bool aligned = reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(b) % 16 == 0 && lda % 2 == 0 && ldb % 2 == 0;
  launch_tiles<double, 128, 128, 16>(
      m, n, k, alpha, beta, c, ldc, GemmCost{1, 2, gemm_rate<double>()}, s,
      [&](dim3 grid, const GemmGrid &g, double *ws) {
        hipLaunchKernelGGL((k_gemm_dl64<128, 2, 2>), grid, dim3(256), 0, s, m, n, k, alpha, a, lda,
                           b, ldb, beta, c, ldc, g, ws, aligned ? 1 : 0);
      });
}

template <int BM, int WM, int WN>
void launch_gemm_dl(int64_t m, int64_t n, int64_t k, float alpha, const float *a, int64_t lda,
                    const float *b, int64_t ldb, float beta, float *c, int64_t ldc,
                    hipStream_t s) {
  const bool aligned = reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(b) % 16 == 0 && lda % 4 == 0 && ldb % 4 == 0;
  launch_tiles<float, BM, 128, 16>(
      m, n, k, alpha, beta, c, ldc, GemmCost{WM * WN / 4, 12 / (WM * WN), gemm_rate<float>()}, s,
      [&](dim3 grid, const GemmGrid &g, float *ws) {
        hipLaunchKernelGGL((k_gemm_dl<BM, WM, WN>), grid, dim3(64 * WM * WN), 0, s, m, n, k, alpha,
                           a, lda, b, ldb, beta, c, ldc, g, ws, aligned ? 1 : 0);
      });
}

template <typename T, int BM, int BN, int BK, int WM, int WN>
void launch_gemm(int64_t m, int64_t n, int64_t k, T alpha, const T *a, int64_t lda,
                 const T *b, int64_t ldb, T beta, T *c, int64_t ldc, hipStream_t s) {
  launch_tiles<T, BM, BN, BK>(
      m, n, k, alpha, beta, c, ldc, gemm_cost<T, BM, BN, WM, WN>(), s,
      [&](dim3 grid, const GemmGrid &g, T *ws) {
        hipLaunchKernelGGL((k_gemm<T, BM, BN, BK, WM, WN>), grid,
                           dim3(GemmCfg<T, BM, BN, BK, WM, WN>::kThreads), 0, s, m, n, k, alpha, a,
                           lda, b, ldb, beta, c, ldc, g, ws);
      });
}

// Workgroup tiles (gemm_tile knob):
//   1: 128 x 128, four waves of 64 x 64, BK = 16 (FP32) / 8 (FP64)
//   2: 256 x 128, eight waves of 64 x 64, same depth
//   3: 128 x 128, twice the depth          4: 256 x 128, twice the depth
//   5: 256 x 256, eight waves of 64 x 128 (FP32 only; FP64 takes 4)
//   6, 7: 128 x 128 and 256 x 128 loading stages straight into LDS (FP32;
//      FP64 has the 128 x 128 one, BK 16, and takes 4 for 7)
// 0 picks by type and size (us for n^3, tiles 1 / 2 / 6): FP64 takes 1 (4096:
// 2081 / 2118 / 2105, 999: 62 / 62 / 78); FP32 takes 2 once C holds 4096 tiles
// of 128 x 128 (8192: 8064 / 7935 / 8373), else 1 (5000: 2000 / 2022 / 2063,
// 999: 40.3 / 40.7 / 48.5; rows that are not 16-byte aligned load element by
// element in 6).
inline int default_gemm_tile(bool fp64, int64_t m, int64_t n) {
  return !fp64 && ((m + 127) / 128) * ((n + 127) / 128) >= 4096 ? 2 : 1;
}

template <typename T>
void run_gemm(int64_t m, int64_t n, int64_t k, T alpha, const T *a, int64_t lda,
              const T *b, int64_t ldb, T beta, T *c, int64_t ldc, hipStream_t s) {
  constexpr int BK = sizeof(T) == 4 ? 16 : 8;
  int t = tuned_gemm_tile();
  if (t == 0) t = default_gemm_tile(sizeof(T) == 8, m, n);
  switch (t) {
    case 1: launch_gemm<T, 128, 128, BK, 2, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s); break;
    case 2: launch_gemm<T, 256, 128, BK, 4, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s); break;
    case 3: launch_gemm<T, 128, 128, 2 * BK, 2, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s); break;
    case 6:
    case 7:
      if constexpr (sizeof(T) == 4) {
        if (t == 6)
          launch_gemm_dl<128, 2, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s);
        else
          launch_gemm_dl<256, 4, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s);
      } else if (t == 6) {
        launch_gemm_dl64(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s);
      } else {
        launch_gemm<T, 256, 128, 2 * BK, 4, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s);
      }
      break;
    case 5:
      if constexpr (sizeof(T) == 4) {
        launch_gemm<T, 256, 256, BK, 4, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s);
        break;
      }
      [[fallthrough]];
    default: launch_gemm<T, 256, 128, 2 * BK, 4, 2>(m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s); break;
  }
}

}  // namespace
}  // namespace drx

using namespace drx;

extern "C" int drx_gemm(int vtype, int64_t m, int64_t n, int64_t k, double alpha,
                        const void *a, int64_t lda, const void *b, int64_t ldb,
                        double beta, void *c, int64_t ldc, drx_stream_t stream) {
  return guarded([&] {
    DRX_REQUIRE(m >= 0 && n >= 0 && k >= 0, "negative dimension");
    DRX_REQUIRE(vtype == DRX_F32 || vtype == DRX_F64, "vtype must be DRX_F32 or DRX_F64");
    DRX_REQUIRE(lda >= std::max<int64_t>(k, 1) && ldb >= std::max<int64_t>(n, 1) &&
                    ldc >= std::max<int64_t>(n, 1),
                "leading dimension below the row length");
    if (m == 0 || n == 0) return;
    DRX_REQUIRE(c != nullptr && (k == 0 || (a != nullptr && b != nullptr)), "null operand");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (vtype == DRX_F32)
      run_gemm<float>(m, n, k, static_cast<float>(alpha), static_cast<const float *>(a), lda,
                      static_cast<const float *>(b), ldb, static_cast<float>(beta),
                      static_cast<float *>(c), ldc, s);
    else
      run_gemm<double>(m, n, k, alpha, static_cast<const double *>(a), lda,
                       static_cast<const double *>(b), ldb, beta, static_cast<double *>(c),
                       ldc, s);
  });
}
