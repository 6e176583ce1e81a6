// drx_mrhs.hip -- products with several right-hand sides (k >= 2), and the
// library's stream-ordered scratch pool.
//
// x (column-major, k columns of ldx) is copied into row-major chunks of KP
// columns (KP = 2, 4, 8 or 16 by k, at most 8 for FP64), then the multi-RHS block body of
// drx_fwd.hpp gathers one contiguous KP-vector per entry. With column-major
// x each entry costs k gathers from k separate columns; the copy costs one
// streaming pass over x. A plan's column panels serve k = 1 only: for k >= 2
// the product runs over the share's own CSR arrays.
//
// Reference kernels replaced: the k-column loops of
// csr_row_distribution.hpp:84-115 and csr_eq_distribution.hpp:62-111 (slim
// matrix right-hand sides, broadcasted_slim_matrix.hpp:10-83).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <set>
#include <vector>

#include "drx_blocks.hpp"
#include "drx_common.hpp"
#include "drx_fwd.hpp"
#include "drx_internal.hpp"

namespace drx {

// ---------------------------------------------------------------------------
// Scratch: one memory pool per device, created on first use, that keeps up to
// kPoolKeep bytes across calls (plus the largest reserve), so that steady-state
// calls reuse it without reaching the driver's allocator. Allocation and release
// are ordered on the caller's stream.
// ---------------------------------------------------------------------------
constexpr int kMaxDevices = 64;
constexpr size_t kPoolKeep = size_t(8) << 30;
constexpr size_t kBlocksKeep = size_t(4) << 30;
static std::mutex g_pool_mu;
static hipMemPool_t g_pools[kMaxDevices];
static std::multiset<size_t> g_reserved[kMaxDevices];

static bool blocks_release(int dev);  // gives the kept blocks back; whether any

static hipMemPool_t pool_for(int dev) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  DRX_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal out of range");
  if (!g_pools[dev]) {
    hipMemPoolProps props{};
    props.allocType = hipMemAllocationTypePinned;
    props.handleTypes = hipMemHandleTypeNone;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    hipMemPool_t pool = nullptr;
    DRX_HIP(hipMemPoolCreate(&pool, &props));
    uint64_t keep = kPoolKeep;
    DRX_HIP(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
    g_pools[dev] = pool;
  }
  return g_pools[dev];
}

// null: out of memory (a limit of the caller's choice, or the device's).
static void *pool_alloc(size_t bytes, hipStream_t s) {
  int dev = 0;
  DRX_HIP(hipGetDevice(&dev));
  const hipMemPool_t pool = pool_for(dev);
  bytes = std::max<size_t>(bytes, 256);
  void *p = nullptr;
  hipError_t e = hipMallocFromPoolAsync(&p, bytes, pool, s);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    // blocks that nobody uses go back to the driver first (not under capture,
    // where this allocation takes no memory yet)
    if (blocks_release(dev)) e = hipMallocFromPoolAsync(&p, bytes, pool, s);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  DRX_HIP(e);
  return p;
}

void *scratch_alloc(size_t bytes, hipStream_t s) {
  void *p = pool_alloc(bytes, s);
  if (p == nullptr) throw Error(DRX_ERR_NOMEM, "no device memory for a product's scratch");
  return p;
}

void *scratch_try(size_t bytes, hipStream_t s) {
  const int64_t most = tuned_scratch_max();
  if (most > 0 && bytes > static_cast<size_t>(most)) return nullptr;
  return pool_alloc(bytes, s);
}

void scratch_free(void *p, hipStream_t s) {
  if (p) (void)hipFreeAsync(p, s);
}

// What device dev's pool keeps when it releases memory (with g_pool_mu held).
static size_t set_keep(int dev) {
  const auto &r = g_reserved[dev];
  uint64_t keep = kPoolKeep + (r.empty() ? size_t(0) : *r.rbegin());
  if (g_pools[dev])
    (void)hipMemPoolSetAttribute(g_pools[dev], hipMemPoolAttrReleaseThreshold, &keep);
  return static_cast<size_t>(keep);
}

void scratch_reserve(int dev, size_t bytes, hipStream_t s) {
  scratch_free(scratch_alloc(bytes, s), s);
  std::lock_guard<std::mutex> lk(g_pool_mu);
  g_reserved[dev].insert(bytes);
  set_keep(dev);
}

void scratch_unreserve(int dev, size_t bytes) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  auto &r = g_reserved[dev];
  const auto at = r.find(bytes);
  if (at != r.end()) r.erase(at);
  if (g_pools[dev]) (void)hipMemPoolTrimTo(g_pools[dev], set_keep(dev));
}

// ---------------------------------------------------------------------------
// Blocks (block_alloc): mapping and unmapping the 0.5 GB that the plan and the
// transpose of 20M entries take cost 9 to 14 ms (two boxes) beside 1.2 ms of
// kernels, and the pool above unmaps freed memory whenever it holds more of it
// than is in use.
// ---------------------------------------------------------------------------
struct HipMemory {
  static constexpr int kOutOfMemory = hipErrorOutOfMemory;
  // (a refused call leaves no error behind for the next launch check)
  static hipError_t cleared(hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
  }
  static int alloc(void **p, size_t bytes) { return cleared(hipMalloc(p, bytes)); }
  static bool free(void *p) { return cleared(hipFree(p)) == hipSuccess; }
  static bool wait() { return cleared(hipDeviceSynchronize()) == hipSuccess; }
};
static BlockCache<HipMemory, kBlocksKeep> g_blocks[kMaxDevices];

// Makes dev the current device while it lives.
struct OnDevice {
  int cur, dev;
  explicit OnDevice(int d) : cur(d), dev(d) {
    (void)hipGetDevice(&cur);
    if (cur != dev) (void)hipSetDevice(dev);
  }
  ~OnDevice() {
    if (cur != dev) (void)hipSetDevice(cur);
  }
};

void *block_alloc(size_t bytes, int dev) {
  if (dev < 0) DRX_HIP(hipGetDevice(&dev));
  DRX_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal out of range");
  const OnDevice on(dev);
  void *p = nullptr;
  DRX_HIP(static_cast<hipError_t>(g_blocks[dev].take(bytes, &p)));
  return p;
}

static bool blocks_release(int dev) { return g_blocks[dev].release(); }
size_t blocks_kept(int dev) { return g_blocks[dev].kept(); }

void block_free(int dev, void *p) {
  if (p == nullptr || dev < 0 || dev >= kMaxDevices) return;
  g_blocks[dev].give(p);
}

bool owned_free(int dev, const std::vector<void *> &ptrs) {
  if (dev < 0 || dev >= kMaxDevices) return false;
  bool any = false;
  for (void *p : ptrs) any = any || p != nullptr;
  if (!any) return false;
  const OnDevice on(dev);
  return g_blocks[dev].retire(ptrs);
}

// ---------------------------------------------------------------------------
// Slots: 64 bytes each of pinned memory, out of pieces of 64 KB that stay
// allocated (a slot is used again by later plans).
// ---------------------------------------------------------------------------
struct PinnedSlots {
  static constexpr int kOutOfMemory = -1;
  static constexpr size_t kPiece = 65536, kSlot = 64;
  static int alloc(void **p, size_t) {
    static std::mutex mu;
    static char *piece = nullptr;
    static size_t used = kPiece;
    std::lock_guard<std::mutex> lk(mu);
    if (used == kPiece) {
      void *q = nullptr;
      const hipError_t e = HipMemory::cleared(
          hipHostMalloc(&q, kPiece, hipHostMallocMapped | hipHostMallocCoherent));
      if (e != hipSuccess) return e;
      piece = static_cast<char *>(q);
      used = 0;
    }
    *p = piece + used;
    used += kSlot;
    return 0;
  }
  static bool free(void *) { return false; }
  static bool wait() { return HipMemory::wait(); }
};
static BlockCache<PinnedSlots, SIZE_MAX, PinnedSlots::kSlot> g_slots[kMaxDevices];

uint64_t *slot_alloc(int dev) {
  void *p = nullptr;
  if (dev < 0 || dev >= kMaxDevices || g_slots[dev].take(PinnedSlots::kSlot, &p) != 0)
    return nullptr;
  *static_cast<volatile uint64_t *>(p) = 0;
  return static_cast<uint64_t *>(p);
}

void slot_free(int dev, uint64_t *slot, bool waited) {
  if (slot == nullptr) return;
  if (waited) {
    g_slots[dev].give(slot);
    return;
  }
  const OnDevice on(dev);
  g_slots[dev].retire(std::initializer_list<void *>{slot});
}

// Samples up to 4096 row blocks: the span between the first and the last
// column index of each window, against its entry count (tight: at most
// 4 n + 64) and against ncols / 16 (loose). out = {tight, loose, sampled}. One
// workgroup, bound by the chain record, column.
template <typename TI>
__global__ __launch_bounds__(256) void k_col_local(const BlockRec *rec, int64_t nblocks,
                                                    int64_t ncols, const TI *colind, int *out) {
  __shared__ int cnt[3];
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t S = nblocks < 4096 ? nblocks : 4096;
  int tight = 0, loose = 0, seen = 0;
  for (int64_t i = threadIdx.x; i < S; i += blockDim.x) {
    const BlockRec b = rec[i * nblocks / S];
    const int64_t n = b.es - b.e0;
    if (n >= 2) {
      const int64_t lo = static_cast<int64_t>(colind[b.e0]);
      const int64_t hi = static_cast<int64_t>(colind[b.es - 1]);
      const int64_t span = hi > lo ? hi - lo : lo - hi;
      seen++;
      if (span <= 4 * n + 64) tight++;
      if (span <= 4 * n + 64 || span <= ncols / 16) loose++;
    }
  }
  atomicAdd(&cnt[0], tight);
  atomicAdd(&cnt[1], loose);
  atomicAdd(&cnt[2], seen);
  __syncthreads();
  if (threadIdx.x < 3) out[threadIdx.x] = cnt[threadIdx.x];
}

// The cached locality of a column array, -1 where it is not known.
static int locality_known(const Plan &p, const void *colind) {
  const int cached = p.loc_local.load(std::memory_order_acquire);
  return p.loc_colind.load(std::memory_order_acquire) == colind ? cached : -1;
}

int column_locality(const Plan &p, const void *colind, hipStream_t s) {
  if (p.nnz == 0 || p.nblocks == 0 || colind == nullptr) return 0;
  if (const int cached = locality_known(p, colind); cached >= 0) return cached;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  DRX_HIP(hipStreamIsCapturing(s, &st));
  if (st != hipStreamCaptureStatusNone) return 0;
  // (the counts straight into the plan's host memory, where it has some: scratch
  // and a copy back take 10 us more)
  int h[3] = {0, 0, 0};
  int *d = p.slot ? reinterpret_cast<int *>(p.slot + 1)
                  : static_cast<int *>(scratch_alloc(sizeof(h), s));
  try {
    if (p.itype == DRX_I32)
      hipLaunchKernelGGL(k_col_local<int32_t>, dim3(1), dim3(256), 0, s, p.rec, p.nblocks,
                         p.ncols, static_cast<const int32_t *>(colind), d);
    else
      hipLaunchKernelGGL(k_col_local<int64_t>, dim3(1), dim3(256), 0, s, p.rec, p.nblocks,
                         p.ncols, static_cast<const int64_t *>(colind), d);
    DRX_HIP(hipGetLastError());
    if (!p.slot) DRX_HIP(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s));
    DRX_HIP(hipStreamSynchronize(s));
  } catch (...) {
    if (!p.slot) scratch_free(d, s);
    throw;
  }
  if (!p.slot)
    scratch_free(d, s);
  else
    for (int i = 0; i < 3; i++) h[i] = static_cast<volatile int *>(d)[i];
  int loc = 0;
  if (h[2] > 0 && 10 * h[0] >= 9 * h[2]) loc |= 1;
  if (h[2] > 0 && 10 * h[1] >= 9 * h[2]) loc |= 2;
  // Invalidate, then publish pointer and value.
  p.loc_local.store(-1, std::memory_order_release);
  p.loc_colind.store(colind, std::memory_order_release);
  p.loc_local.store(loc, std::memory_order_release);
  return loc;
}

// ---------------------------------------------------------------------------
// k >= 2 over long rows whose neighbours hold neighbouring columns (wide
// bands). Gathered one row at a time, each entry reads its x row (KP values)
// from L2, 64 bytes per 16 of the matrix in FP64 and k = 8: that bounds the
// row-block kernel, though eight neighbouring rows read almost the same x.
// Here a workgroup takes eight rows and copies the columns that they span into
// LDS piece by piece, straight from x as the caller holds it (no row-major copy,
// no scratch, one launch). A wave sums two rows, a lane every 64th entry; a row's
// next U * 64 entries wait in registers until the piece with their columns is
// there (so their loads are in flight while x is copied, and no entry is read
// twice), and are summed from memory where columns are out of order.
// Bound by the matrix stream: 50000 rows of 2001 entries, k = 8, FP64 values and
// 64-bit columns 315 us (5.1 TB/s; with its launch in a loop 345, the row-block
// kernel 518; entries read again
// in the next piece instead of kept: 390), FP32 and 32-bit columns 190 (315).
// U: FP64 2 / 4 / 8 batches 362 / 345 / 457 us, FP32 260 / 223 / 201.
// ---------------------------------------------------------------------------
constexpr int kBandRows = 8;                 // rows of a workgroup, two per wave
constexpr int kBandLds = 38 * 1024;          // x of one piece (four workgroups per CU)

// Bytes between the x rows of neighbouring columns in LDS: rows of more than 16
// bytes are padded by 16, so that 16 lanes' 16-byte reads of neighbouring
// columns fall into different banks.
template <int KP, typename TX> constexpr int band_stride() {
  constexpr int b = KP * static_cast<int>(sizeof(TX));
  return b <= 16 ? b : b + 16;
}

// x of column c (KP columns from j0 on, kk of them there) in storage type;
// zeros past the last column.
template <int KP, typename TX>
__device__ __forceinline__ void band_xcol(const TX *x, int64_t ldx, int64_t ncols, int64_t j0,
                                          int kk, int64_t c, TX (&t)[KP]) {
  if (static_cast<uint64_t>(c) >= static_cast<uint64_t>(ncols)) kk = 0;
#pragma unroll
  for (int j = 0; j < KP; j++) t[j] = j < kk ? x[(j0 + j) * ldx + c] : TX{};
}

// CH partial sums per lane, row and column, of every CH-th entry of the lane,
// which are added at the end: W * CH chains of additions per row, as many as
// the row-block kernel has at most (wg_row_sums), for rows that give each at
// least 2.5 entries (see mrhs_lanes). With one, rows of 2001 entries had 1.28
// (k <= 4) and 1.17 (k = 8) times that kernel's error; sixteen FP64 sums take one.
template <int KP, typename TX, typename TA> constexpr int band_chains() {
  constexpr int b = KP * static_cast<int>(sizeof(TA));
  return b <= 16 ? 4 : (b <= 32 || (b == 64 && sizeof(TX) == 4) ? 2 : 1);
}

// Rows of fewer than 160 entries are summed by W = 32 lanes of their wave, for the
// same reason (rows of 97: 0.6 % more error with 64 lanes than before, now less).
template <int KP, int CH, int W, typename TV, typename TX, typename TY, typename TA, typename TI>
__global__ __launch_bounds__(256) void k_spmv_band(FwdArgs a, int64_t j0) {
  constexpr int STRIDE = band_stride<KP, TX>(), PC = kBandLds / STRIDE / 64 * 64;
  constexpr int ALIGN = STRIDE < 16 ? STRIDE : 16;
  constexpr int RW = kBandRows / 4, U = sizeof(TA) == 4 ? 8 : 4;
  constexpr uint32_t kDone = 0xffffffffu;
  __shared__ __attribute__((aligned(16))) char xs[PC * STRIDE];
  __shared__ int64_t row_at[kBandRows + 1];
  __shared__ uint32_t range[2];
  __shared__ TA ys[kBandRows * (KP + 1)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (a.gate != nullptr && *a.gate == 0) return;
  const int64_t blk = map_block(blockIdx.x, a.per_xcd);
  if (blk >= a.nblocks) return;  // the whole workgroup
  const int64_t r0 = blk * kBandRows;
  const TI *rowptr = static_cast<const TI *>(a.rowptr);
  const TI *colind = static_cast<const TI *>(a.colind);
  const TV *vals = static_cast<const TV *>(a.vals);
  const TX *x = static_cast<const TX *>(a.x);
  const int kk = a.k - j0 < KP ? static_cast<int>(a.k - j0) : KP;
  if (tid <= kBandRows) {
    const int64_t r = r0 + tid < a.nrows ? r0 + tid : a.nrows;
    row_at[tid] = row_begin(rowptr, a.base, a.nrows, a.nnz, a.sent, r);
  }
  if (tid == 0) {
    range[0] = kDone;
    range[1] = 0;
  }
  __syncthreads();
  int64_t at[RW], end[RW];
  uint32_t c[RW][U];
  TV w[RW][U];
  TA acc[RW][CH][KP];
  // The next U * W entries of a row of the wave; lanes past its end are done.
  auto load = [&](int r) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t e = at[r] + u * W + lane;
      const int64_t ee = e < end[r] ? e : end[r] - 1;
      c[r][u] = col32(ld_stream(colind + ee));
      w[r][u] = ld_stream(vals + ee);
      if (e >= end[r] || (W < 64 && lane >= W)) c[r][u] = kDone;
    }
    at[r] += U * W;
  };
#pragma unroll
  for (int r = 0; r < RW; r++) {
    at[r] = row_at[wave * RW + r];
    end[r] = row_at[wave * RW + r + 1];
#pragma unroll
    for (int t = 0; t < CH; t++)
#pragma unroll
      for (int j = 0; j < KP; j++) acc[r][t][j] = 0;
    if (at[r] < end[r]) {
      load(r);
    } else {
#pragma unroll
      for (int u = 0; u < U; u++) {
        c[r][u] = kDone;
        w[r][u] = TV{};
      }
    }
  }
  if (tid < kBandRows && row_at[tid] < row_at[tid + 1]) {
    atomicMin(&range[0], col32(colind[row_at[tid]]));
    atomicMax(&range[1], col32(colind[row_at[tid + 1] - 1]));
  }
  __syncthreads();
  const uint32_t lo = range[0], ncols = static_cast<uint32_t>(a.ncols);
  const uint32_t past = range[1] < ncols ? range[1] + 1 : ncols;
  const int64_t held = row_at[kBandRows] - row_at[0];
  // The entries held of the wave's rows with columns below p1: x from LDS from
  // column p0 on, from memory below.
  auto sum_below = [&](uint32_t p0, uint32_t p1) {
#pragma unroll
    for (int r = 0; r < RW; r++) {
      for (;;) {
        bool rest = false;
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (c[r][u] < p1) {
            TX t[KP];
            if (c[r][u] >= p0)
              __builtin_memcpy(t, __builtin_assume_aligned(xs + (c[r][u] - p0) * STRIDE, ALIGN),
                               sizeof(t));
            else
              band_xcol<KP>(x, a.ldx, a.ncols, j0, kk, c[r][u], t);
            const TA v = to_acc<TA>(w[r][u]);
#pragma unroll
            for (int j = 0; j < KP; j++)
              acc[r][u % CH][j] = fma_acc(v, to_acc<TA>(t[j]), acc[r][u % CH][j]);
            c[r][u] = kDone;
          }
          rest |= c[r][u] != kDone;
        }
        if (__ballot(rest) != 0 || at[r] >= end[r]) break;
        load(r);
      }
    }
  };
  // Pieces of the columns that the rows span, unless they span far more than
  // the rows hold.
  if (lo < past && past - lo < 2 * held + PC) {
    for (uint32_t p0 = lo; p0 < past; p0 += PC) {
      const uint32_t p1 = past - p0 > PC ? p0 + PC : past;
      __syncthreads();
      for (uint32_t i = tid; i < p1 - p0; i += 256) {
        TX t[KP];
        band_xcol<KP>(x, a.ldx, a.ncols, j0, kk, p0 + i, t);
        __builtin_memcpy(__builtin_assume_aligned(xs + i * STRIDE, ALIGN), t, sizeof(t));
      }
      __syncthreads();
      sum_below(p0, p1);
    }
  }
  // What is left (columns out of order, or no pieces).
  sum_below(kDone, kDone);
#pragma unroll
  for (int r = 0; r < RW; r++) {
#pragma unroll
    for (int j = 0; j < KP; j++) {
      TA sum = acc[r][0][j];
      if constexpr (CH >= 2) sum += acc[r][1][j];
      if constexpr (CH == 4) sum += acc[r][2][j] + acc[r][3][j];
      sum = group_sum<64>(sum);
      if (lane == 0) ys[(wave * RW + r) * (KP + 1) + j] = sum;
    }
  }
  __syncthreads();
  TY *y = static_cast<TY *>(a.y);
  const TA alpha = static_cast<TA>(a.alpha), beta = static_cast<TA>(a.beta);
  for (int t = tid; t < kBandRows * kk; t += 256) {
    const int j = t / kBandRows, i = t % kBandRows;
    if (r0 + i >= a.nrows) continue;
    TY *yp = y + (j0 + j) * a.ldy + r0 + i;
    TA out = alpha * ys[i * (KP + 1) + j];
    if (beta != TA(0)) out += beta * to_acc<TA>(*yp);
    *yp = from_acc<TY>(out);
  }
}

template <int KP, int CH, int W, typename TV, typename TX, typename TY, typename TA>
static void launch_band_ch(const Plan &p, const FwdArgs &a, int64_t j0, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.grid));
  if (p.itype == DRX_I32)
    hipLaunchKernelGGL((k_spmv_band<KP, CH, W, TV, TX, TY, TA, int32_t>), grid, dim3(256), 0, s, a,
                       j0);
  else
    hipLaunchKernelGGL((k_spmv_band<KP, CH, W, TV, TX, TY, TA, int64_t>), grid, dim3(256), 0, s, a,
                       j0);
}

template <int KP, typename TV, typename TX, typename TY, typename TA>
static void launch_band(const Plan &p, const FwdArgs &a, int64_t j0, hipStream_t s) {
  constexpr int MOST = band_chains<KP, TX, TA>();
  if (MOST >= 4 && p.nnz >= 640 * p.nrows)
    launch_band_ch<KP, MOST, 64, TV, TX, TY, TA>(p, a, j0, s);
  else if (MOST >= 2 && p.nnz >= 320 * p.nrows)
    launch_band_ch<KP, MOST < 2 ? MOST : 2, 64, TV, TX, TY, TA>(p, a, j0, s);
  else if (p.nnz >= 160 * p.nrows)
    launch_band_ch<KP, 1, 64, TV, TX, TY, TA>(p, a, j0, s);
  else
    launch_band_ch<KP, 1, 32, TV, TX, TY, TA>(p, a, j0, s);
}

template <typename TV, typename TX, typename TY, typename TA>
static void launch_band_t(const Plan &p, const FwdArgs &a, hipStream_t s) {
  // Up to 16 right-hand sides per pass over the matrix (FP64, rows of 600, 16
  // of them: 183 us, in two passes of 8 228).
  for (int64_t j0 = 0; j0 < a.k; j0 += 16) {
    const int64_t left = a.k - j0;
    if (left <= 2)
      launch_band<2, TV, TX, TY, TA>(p, a, j0, s);
    else if (left <= 4)
      launch_band<4, TV, TX, TY, TA>(p, a, j0, s);
    else if (left <= 8)
      launch_band<8, TV, TX, TY, TA>(p, a, j0, s);
    else
      launch_band<16, TV, TX, TY, TA>(p, a, j0, s);
  }
}

// Whether eight neighbouring rows hold the columns that they span at least
// twice, for nine in ten of up to 128 groups of rows: *gate, and with colind's
// address the plan's slot. One workgroup, eight lanes per group, all loads of
// a lane in two steps. The answer steers the kernels that follow it on the
// stream (first call on a column array: either these or the row blocks run,
// the others leave at once), so the host does not wait for it; later calls find
// it in the slot. (With a host wait, as one workgroup over 4096 samples, the first
// product of 8000 rows of 97..400 entries took 75..110 us instead of 37..40.)
constexpr int kBandGroups = 128;
template <typename TI>
__global__ __launch_bounds__(8 * kBandGroups) void k_band_probe(const TI *rowptr, int64_t base,
                                                                int64_t nrows, int64_t nnz,
                                                                int sent, const TI *colind,
                                                                int *gate, uint64_t *slot) {
  __shared__ int cnt[2];
  if (threadIdx.x < 2) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t groups = (nrows + 7) / 8, S = groups < kBandGroups ? groups : kBandGroups;
  const int64_t i = threadIdx.x / 8;
  const int64_t r = i < S ? i * groups / S * 8 + threadIdx.x % 8 : nrows;
  int64_t at = 0, end = 0;
  if (r < nrows) {
    at = row_begin(rowptr, base, nrows, nnz, sent, r);
    end = row_begin(rowptr, base, nrows, nnz, sent, r + 1);
  }
  int64_t first = INT64_MAX, last = 0, held = 0;
  if (at < end) {
    first = static_cast<int64_t>(colind[at]);
    last = static_cast<int64_t>(colind[end - 1]);
    held = end - at;
  }
#pragma unroll
  for (int o = 1; o < 8; o *= 2) {
    const int64_t f = __shfl_xor(first, o, 64), l = __shfl_xor(last, o, 64);
    first = f < first ? f : first;
    last = l > last ? l : last;
    held += __shfl_xor(held, o, 64);
  }
  if (threadIdx.x % 8 == 0 && held > 0) {
    atomicAdd(&cnt[0], 1);
    if (2 * (last - first) <= held) atomicAdd(&cnt[1], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int band = cnt[0] > 0 && 10 * cnt[1] >= 9 * cnt[0];
    if (gate != nullptr) *gate = band;
    __hip_atomic_store(slot, (reinterpret_cast<uint64_t>(colind) << 1) | band, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

static void launch_band_probe(const Plan &p, const FwdArgs &a, int *gate, hipStream_t s) {
  p.band_colind.store(a.colind, std::memory_order_relaxed);
  if (p.itype == DRX_I32)
    hipLaunchKernelGGL(k_band_probe<int32_t>, dim3(1), dim3(8 * kBandGroups), 0, s,
                       static_cast<const int32_t *>(p.rowptr), p.base, p.nrows, p.nnz,
                       p.has_sentinel, static_cast<const int32_t *>(a.colind), gate, p.slot);
  else
    hipLaunchKernelGGL(k_band_probe<int64_t>, dim3(1), dim3(8 * kBandGroups), 0, s,
                       static_cast<const int64_t *>(p.rowptr), p.base, p.nrows, p.nnz,
                       p.has_sentinel, static_cast<const int64_t *>(a.colind), gate, p.slot);
  DRX_HIP(hipGetLastError());
}

// What the plan's slot says of a column array: kBandProbe, nothing.
static BandChoice band_known(const Plan &p, const void *colind) {
  const uint64_t v = __atomic_load_n(p.slot, __ATOMIC_RELAXED);
  if (v == 0 || v >> 1 != reinterpret_cast<uint64_t>(colind)) return kBandProbe;
  return v & 1 ? kBandYes : kBandNo;
}

// Whether run_mrhs takes its chunk width from the columns' locality: 8-wide
// chunks for k > 8 when the columns are loosely local (measured on the 3-D
// Laplacian 128^3 FP32, k = 16: 2293 vs 1982 GB/s, while a matrix of random
// columns runs half as fast with them: 323 vs 618 GB/s).
static bool mrhs_asks_locality(int64_t k, int xtype) {
  return k > 8 && dtype_size(xtype) == 4 && tuned_mrhs_kp_max() == 0;
}

// Plain shares of rows of much the same length whose neighbours hold
// neighbouring columns (k_band_probe): long rows, where the matrix
// stream covers the steps a workgroup takes one after the other (50000 rows, row
// blocks / here: 401 entries FP32 k = 2 / 8 59 / 54, 73 / 69 us, FP64 k = 2 / 8 / 16
// 75 / 70, 102 / 94, 154 / 156; 301 entries 47 / 48, 55 / 63 and 60 / 63, 83 / 84,
// 122 / 168), longer ones still for more than eight FP32 right-hand sides (whose
// sums leave three waves per SIMD: 401 entries k = 16 102 / 109, 501 167 / 122),
// and shorter ones where all workgroups are resident at once (8192 rows) and one
// launch without scratch counts for more (8000 rows of 97 entries FP64 k = 2 / 8 /
// 16: 36 / 14, 34 / 15, 31 / 24 us).
BandChoice band_mrhs(const Plan &p, const FwdArgs &a, int xtype, hipStream_t s) {
  const int knob = tuned_mrhs_band();
  if (knob == 0 || a.xbytes == 0) return kBandNo;
  if (knob == 2) return kBandYes;
  const int64_t least =
      p.nrows <= 8192 ? kBandLeast : (xtype == DRX_F32 && a.k > 8 ? 5 : 4) * kBandLeast;
  if (p.slot == nullptr || p.nnz < least * p.nrows || p.lmax * p.nrows > 4 * p.nnz)
    return kBandNo;
  const BandChoice known = band_known(p, a.colind);
  if (known != kBandProbe) return known;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  DRX_HIP(hipStreamIsCapturing(s, &st));
  // A capture asks only where a probe was launched before (whose answer may be
  // on its way), so that what it records does not hang on timing.
  if (st != hipStreamCaptureStatusNone)
    return p.band_colind.load(std::memory_order_relaxed) == a.colind ? kBandProbe : kBandNo;
  if (mrhs_asks_locality(a.k, xtype) && locality_known(p, a.colind) < 0) {
    // the chunk width hangs on a probe that the host waits for: one wait
    launch_band_probe(p, a, nullptr, s);
    (void)column_locality(p, a.colind, s);
    return band_known(p, a.colind);
  }
  return kBandProbe;
}

void run_band(const Plan &p, FwdArgs a, int vtype, int xtype, int ytype, hipStream_t s) {
  a.nblocks = (p.nrows + kBandRows - 1) / kBandRows;
  a.per_xcd = (a.nblocks + kXcds - 1) / kXcds;
  a.grid = a.per_xcd * kXcds;
  DRX_REQUIRE(a.grid <= int64_t(0xffffffff), "too many rows for one launch");
  if (vtype == DRX_F64 && xtype == DRX_F64 && ytype == DRX_F64)
    launch_band_t<double, double, double, double>(p, a, s);
  else if (vtype == DRX_F32 && xtype == DRX_F32 && ytype == DRX_F32)
    launch_band_t<float, float, float, float>(p, a, s);
  else if (vtype == DRX_BF16 && xtype == DRX_BF16 && ytype == DRX_F32)
    launch_band_t<bf16, bf16, float, float>(p, a, s);
  else if (vtype == DRX_F16 && xtype == DRX_F16 && ytype == DRX_F32)
    launch_band_t<f16, f16, float, float>(p, a, s);
  else if (vtype == DRX_BF16 && xtype == DRX_F32 && ytype == DRX_F32)
    launch_band_t<bf16, float, float, float>(p, a, s);
  else if (vtype == DRX_F16 && xtype == DRX_F32 && ytype == DRX_F32)
    launch_band_t<f16, float, float, float>(p, a, s);
  else
    throw Error(DRX_ERR_UNSUPPORTED, "unsupported (vtype, xtype, ytype)");
  DRX_HIP(hipGetLastError());
}

int mrhs_kp(int64_t k, int xtype, bool loose_local) {
  if (k <= 2) return 2;
  if (k <= 4) return 4;
  if (k <= 8 || dtype_size(xtype) == 8) return 8;
  const int cap = tuned_mrhs_kp_max();
  return (cap == 8 || (cap == 0 && loose_local)) ? 8 : 16;
}

size_t mrhs_xr_bytes(int64_t ncols, int64_t k, int kp, int xtype) {
  const int64_t nchunk = (k + kp - 1) / kp;
  return static_cast<size_t>(nchunk) * static_cast<size_t>(std::max<int64_t>(ncols, 1)) *
         kp * dtype_size(xtype);
}

// x -> xr on stream s (only the element size matters: the zero padding is
// all-zero bits, +0 in every floating type).
void launch_x_rowmajor(int xtype, const void *x, int64_t ldx, int64_t ncols,
                       int64_t k, int kp, void *xr, const int *gate, hipStream_t s) {
  const int64_t total = ((k + kp - 1) / kp) * ncols;
  if (total == 0) return;
  const dim3 g(static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 1 << 16)));
#define DRX_XR(KP, T)                                                          \
  hipLaunchKernelGGL((k_x_rowmajor<KP, T>), g, dim3(256), 0, s,                \
                     static_cast<const T *>(x), ldx, ncols, k, static_cast<T *>(xr), gate)
#define DRX_XR_T(T)                                                            \
  do {                                                                         \
    if (kp == 2)                                                               \
      DRX_XR(2, T);                                                            \
    else if (kp == 4)                                                          \
      DRX_XR(4, T);                                                            \
    else if (kp == 8)                                                          \
      DRX_XR(8, T);                                                            \
    else                                                                       \
      DRX_XR(16, T);                                                           \
  } while (0)
  const size_t xs = dtype_size(xtype);
  if (xs == 8)
    DRX_XR_T(uint64_t);
  else if (xs == 4)
    DRX_XR_T(uint32_t);
  else
    DRX_XR_T(uint16_t);
#undef DRX_XR_T
#undef DRX_XR
  DRX_HIP(hipGetLastError());
}

template <int KP, int MODE, typename TV, typename TX, typename TY, typename TA,
          typename TI>
static void launch_mrhs(const Plan &p, const FwdArgs &a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.grid));
  if (p.cap <= 2048)
    hipLaunchKernelGGL((k_spmv_mrhs<256, 2048, KP, MODE, TV, TX, TY, TA, TI>),
                       grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_spmv_mrhs<512, 8192, KP, MODE, TV, TX, TY, TA, TI>),
                       grid, dim3(512), 0, s, a);
}

template <int KP, int MODE, typename TV, typename TX, typename TY, typename TA>
static void launch_mrhs_i(const Plan &p, const FwdArgs &a, hipStream_t s) {
  if (p.itype == DRX_I32)
    launch_mrhs<KP, MODE, TV, TX, TY, TA, int32_t>(p, a, s);
  else
    launch_mrhs<KP, MODE, TV, TX, TY, TA, int64_t>(p, a, s);
}

template <typename TV, typename TX, typename TY, typename TA>
static void launch_mrhs_t(const Plan &p, const FwdArgs &a, int mode, int kp,
                          hipStream_t s) {
#define DRX_KP(MODE)                                                           \
  do {                                                                         \
    if (kp == 2)                                                               \
      launch_mrhs_i<2, MODE, TV, TX, TY, TA>(p, a, s);                         \
    else if (kp == 4)                                                          \
      launch_mrhs_i<4, MODE, TV, TX, TY, TA>(p, a, s);                         \
    else if (kp == 8)                                                          \
      launch_mrhs_i<8, MODE, TV, TX, TY, TA>(p, a, s);                         \
    else                                                                       \
      launch_mrhs_i<16, MODE, TV, TX, TY, TA>(p, a, s);                        \
  } while (0)
  if (mode == kPerm)
    DRX_KP(kPerm);
  else
    DRX_KP(kPlain);
#undef DRX_KP
}

void run_mrhs(const Plan &p, FwdArgs a, int mode, int vtype, int xtype,
              int ytype, bool probe, hipStream_t s) {
  DRX_REQUIRE(mode == kPlain || mode == kPerm, "bad mode for k >= 2");
  // one chunk width for the copy and the kernel (the knob may change)
  const bool loose =
      mrhs_asks_locality(a.k, xtype) && (column_locality(p, a.colind, s) & 2) != 0;
  const int kp = mrhs_kp(a.k, xtype, loose);
  const size_t xr_bytes = (mrhs_xr_bytes(p.ncols, a.k, kp, xtype) + 255) & ~size_t(255);
  void *xr = scratch_alloc(xr_bytes + (probe ? 256 : 0), s);
  try {
    if (probe) {
      int *gate = reinterpret_cast<int *>(static_cast<char *>(xr) + xr_bytes);
      launch_band_probe(p, a, gate, s);
      a.gate = gate;
      run_band(p, a, vtype, xtype, ytype, s);
    }
    launch_x_rowmajor(xtype, a.x, a.ldx, p.ncols, a.k, kp, xr, a.gate, s);
    a.xr = xr;
    a.ncols = p.ncols;
    a.gshift = tuned_mrhs_gshift();
    if (vtype == DRX_F64 && xtype == DRX_F64 && ytype == DRX_F64)
      launch_mrhs_t<double, double, double, double>(p, a, mode, kp, s);
    else if (vtype == DRX_F32 && xtype == DRX_F32 && ytype == DRX_F32)
      launch_mrhs_t<float, float, float, float>(p, a, mode, kp, s);
    else if (vtype == DRX_BF16 && xtype == DRX_BF16 && ytype == DRX_F32)
      launch_mrhs_t<bf16, bf16, float, float>(p, a, mode, kp, s);
    else if (vtype == DRX_F16 && xtype == DRX_F16 && ytype == DRX_F32)
      launch_mrhs_t<f16, f16, float, float>(p, a, mode, kp, s);
    else if (vtype == DRX_BF16 && xtype == DRX_F32 && ytype == DRX_F32)
      launch_mrhs_t<bf16, float, float, float>(p, a, mode, kp, s);
    else if (vtype == DRX_F16 && xtype == DRX_F32 && ytype == DRX_F32)
      launch_mrhs_t<f16, float, float, float>(p, a, mode, kp, s);
    else
      throw Error(DRX_ERR_UNSUPPORTED, "unsupported (vtype, xtype, ytype)");
    DRX_HIP(hipGetLastError());
  } catch (...) {
    scratch_free(xr, s);
    throw;
  }
  scratch_free(xr, s);
}

}  // namespace drx
