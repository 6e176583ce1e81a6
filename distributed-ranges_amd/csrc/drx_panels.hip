// drx_panels.hip -- column-panel layout of a plan, for matrices whose x does
// not fit the L2 of an XCD (4 MB) and whose columns are irregular.
//
// Random 4-byte gathers on MI355X run at about 58 G/s from memory, 78 G/s
// from the MALL, 235 G/s from L2 and 280 G/s with a 128 KB range (each gather
// moves a whole cache line into a CU's L1), but a CU's LDS serves a wave's 64
// random 4-byte reads in a few cycles. So the layout cuts the columns into
// slices whose x fits the LDS of one CU (128 KB: 32768 columns of 4-byte
// sums, 16384 of FP64) and keeps a copy of the entries in slice order (a
// stable radix sort by slice: rows, and columns within rows, stay in order).
// The entries of one row in one slice form a segment. A product runs two
// kernels:
//   1. k_slice_sums: each workgroup takes a share of the entries, loads the
//      x slice into LDS, and streams (value, 15-bit column, segment flag) --
//      6 bytes per FP32 entry -- into one sum per segment, in segment order;
//   2. k_slice_rows: each wave owns a run of rows and adds their segments'
//      sums, slice after slice, into FP64 sums in LDS (compensated for FP64),
//      and writes y = alpha * sum + beta * y once.
// Both stream memory; nothing is gathered from beyond LDS. Each segment is
// summed by one wave in entry order and each row's segments are added in
// slice order, so results are deterministic (no floating-point atomics
// between waves).
//
// Measured (16M x 16M Zipf FP32, 1.56e9 entries, 5.4e8 segments): 2.85 ms per
// product -- k_slice_sums 2.15 ms (9.4 GB read, 2.2 GB written: 5.4 TB/s) and
// k_slice_rows 0.75 ms (3.2 GB) -- where one L2-gathering launch per 2 MB
// panel took 8.09 ms (235 G gathers/s). 1M x 4M Zipf BF16 145 us (538 us);
// 5M x 6M FP64 1.64 ms (3.34 ms). Error against 64-bit sums 5.7e-8 (1.4e-7).
//
// Panels of the public interface group slices: a panel wider than a slice is
// cut into equal slices, narrower panels share one.
//
// The copy is tied to the colind/vals given to drx_plan_set_panels; new
// values are re-packed through the kept permutation by
// drx_plan_update_values.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "drx_common.hpp"
#include "drx_internal.hpp"

namespace drx {

// Columns of one slice: 128 KB of x in the sum type; the local column takes
// the upper 15 bits of a 16-bit word, the lowest bit is clear where a segment
// starts (set: the entry continues its predecessor's segment).
template <typename TA> constexpr int64_t slice_cols() { return sizeof(TA) == 8 ? 16384 : 32768; }
// Entries a wave handles per step (8 per lane); the copies' arrays are padded
// to whole steps.
constexpr int64_t kStep = 512;
constexpr int kStepsAhead = 3;  // steps whose loads a wave has in flight (2: 6 % slower, 4 equal)
constexpr int kSumWaves = 16;  // waves of a k_slice_sums workgroup

struct PanelSet {
  int64_t width = 0, npanels = 0, nseg = 0;
  int vtype = 0, device = 0;
  size_t scratch = 0;  // bytes of a product's segment sums (reserved in the pool)
  const void *src_colind = nullptr, *src_vals = nullptr;
  // slices: groups of `group` columns, each of spg slices of sw columns
  int64_t group = 0, spg = 1, sw = 0, ns = 0;
  uint16_t *pcol = nullptr;  // local column << 1 | continues
  void *pval = nullptr;      // values (value_slot order within a step)
  void *perm = nullptr;      // source entry of each entry in slice order
  uint16_t *seg_row = nullptr;  // a segment's row within its row group
  uint32_t *seg_at = nullptr;   // [row group][slice]: first segment
  int64_t rows_per = 0, ngroups = 0;  // rows of a group, groups
  int group_waves = 1;                // waves that own one group
  // k_slice_sums: workgroup g takes tiles [wg_tile[g], wg_tile[g + 1]); a
  // tile is a part of one slice, cut into kSumWaves ranges at segment starts
  // (kSumWaves + 1 first entries and first segments per tile).
  int64_t nwg = 0;
  uint32_t *wg_tile = nullptr, *tile_slice = nullptr, *tile_e = nullptr, *tile_s = nullptr;
};

void free_panels(PanelSet *ps) {
  if (!ps) return;
  owned_free(ps->device, {ps->pcol, ps->pval, ps->perm, ps->seg_row, ps->seg_at, ps->wg_tile,
                          ps->tile_slice, ps->tile_e, ps->tile_s});
  if (ps->scratch > 0) scratch_unreserve(ps->device, ps->scratch);
  delete ps;
}

static dim3 grid_of(int64_t n, int tpb = 256) {
  int64_t b = (n + tpb - 1) / tpb;
  if (b > (int64_t(1) << 20)) b = int64_t(1) << 20;
  return dim3(static_cast<unsigned>(b < 1 ? 1 : b));
}

#define DRX_GRID_LOOP(i, n)                                                    \
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; \
       i < (n); i += static_cast<int64_t>(gridDim.x) * blockDim.x)

// Position of entry i's value within the copy: inside each step of 512
// entries the 16-byte groups that a lane's 8 values make are laid so that
// every 16-byte load of a wave reads 1 KB in lane order.
template <typename TV> __host__ __device__ __forceinline__ int64_t value_slot(int64_t i) {
  constexpr int V = 16 / static_cast<int>(sizeof(TV)) < 8 ? 16 / static_cast<int>(sizeof(TV)) : 8;
  const int64_t step = i & ~(kStep - 1);
  const int k = static_cast<int>(i & 7), lane = static_cast<int>(i >> 3) & 63;
  return step + (k / V) * (64 * V) + lane * V + k % V;
}

// ---------------------------------------------------------------------------
// Products
// ---------------------------------------------------------------------------
struct SliceArgs {
  const uint16_t *pcol;
  const void *pval, *x;
  const uint32_t *wg_tile, *tile_slice, *tile_e, *tile_s;
  int64_t group, spg, sw, ncols;
  void *sums;  // one per segment
};

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t dpp_shift(uint32_t v, uint32_t old = 0) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
      static_cast<int>(old), static_cast<int>(v), CTRL, ROWS, 0xf, false));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp_shift(float v, float old = 0) {
  return __uint_as_float(dpp_shift<CTRL, ROWS>(__float_as_uint(v), __float_as_uint(old)));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_shift(double v, double old = 0) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
  const uint64_t o = static_cast<uint64_t>(__double_as_longlong(old));
  const uint32_t lo = dpp_shift<CTRL, ROWS>(static_cast<uint32_t>(b), static_cast<uint32_t>(o));
  const uint32_t hi =
      dpp_shift<CTRL, ROWS>(static_cast<uint32_t>(b >> 32), static_cast<uint32_t>(o >> 32));
  return __longlong_as_double(static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo));
}
// DPP controls (GFX9 encoding): lane i takes lane i - n of its 16-lane row;
// lane 15 of a row to the next row; lane 31 to the upper half; lane i - 1.
constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;

__device__ __forceinline__ float last_lane(float v) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ double last_lane(double v) {
  const int64_t b = __double_as_longlong(v);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b), 63));
  const uint32_t hi =
      static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b >> 32), 63));
  return __longlong_as_double((static_cast<int64_t>(hi) << 32) | lo);
}

// v where keep is all ones, +0 where it is 0.
__device__ __forceinline__ float and_mask(float v, uint32_t keep) {
  return __uint_as_float(__float_as_uint(v) & keep);
}
__device__ __forceinline__ double and_mask(double v, uint32_t keep) {
  const uint64_t m = (static_cast<uint64_t>(keep) << 32) | keep;
  return __longlong_as_double(
      static_cast<int64_t>(static_cast<uint64_t>(__double_as_longlong(v)) & m));
}

__device__ __forceinline__ void store_sum(rsrc_t r, float v, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, 0, 0);
}
__device__ __forceinline__ void store_sum(rsrc_t r, double v, uint32_t off) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
}

// Sums that a wave stages in LDS at once (2 KB): a whole step's, or for 8-byte
// sums those of half of its lanes.
template <typename TA> constexpr int staged_sums() { return 2048 / static_cast<int>(sizeof(TA)); }

// One lane's 8 entries of a step, as loaded.
template <typename TV> struct StepRegs {
  static constexpr int NV = static_cast<int>(8 * sizeof(TV) / 16);
  Words<4> c;
  Words<4> v[NV];
};

template <typename TV>
__device__ __forceinline__ void load_step(StepRegs<TV> &r, const uint16_t *pcol, const TV *pval,
                                          int64_t at, int lane) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  constexpr int V = 16 / static_cast<int>(sizeof(TV));
  r.c = __builtin_bit_cast(Words<4>, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(
                                         pcol + at + lane * 8)));
#pragma unroll
  for (int i = 0; i < StepRegs<TV>::NV; i++)
    r.v[i] = __builtin_bit_cast(
        Words<4>, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(
                      pval + at + i * 64 * V + lane * V)));
}

// Sums of the segments that start in a wave's range, one step after another.
// Lanes hold 8 consecutive entries each. Sums that run across lanes come from
// a segmented scan over the lanes' tails (DPP, six steps), those that run
// across steps from `open`, the last lane's. `open` belongs to segment
// `seg` - 1 (relative to the range).
template <typename TV, typename TA>
__device__ __forceinline__ void sum_step(const StepRegs<TV> &r, const TA *xs, int lane, int64_t at,
                                         int64_t ea, int64_t eb, rsrc_t out, TA *staged,
                                         TA &open, uint32_t &seg) {
  constexpr uint32_t SZ = sizeof(TA);
  TV tv[8];
  __builtin_memcpy(tv, r.v, sizeof(tv));
  TA v[8], xv[8];
  uint32_t cont[8];  // all ones: continues the entry before it
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint32_t w = r.c.w[k / 2];
    const uint32_t byte = (k & 1) ? (w >> 17) * SZ : ((w & 0xfffeu) >> 1) * SZ;
    xv[k] = *reinterpret_cast<const TA *>(reinterpret_cast<const char *>(xs) + byte);
    cont[k] = static_cast<uint32_t>(
        static_cast<int32_t>((k & 1) ? w << 15 : w << 31) >> 31);
    v[k] = to_acc<TA>(tv[k]);
  }
  if (at < ea || at + kStep > eb) {
    // entries outside [ea, eb): nothing starts there and nothing is added
    // (both factors cleared: the other may be infinite)
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int64_t e = at + lane * 8 + k;
      if (e < ea || e >= eb) {
        cont[k] = 0xffffffffu;
        v[k] = 0;
        xv[k] = 0;
      }
    }
  }
  // starts in this lane, and in the lanes before it
  uint32_t starts = 8;
  TA tail = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    starts += cont[k];
    tail = and_mask(tail, cont[k]) + v[k] * xv[k];
  }
  uint32_t before = starts;
  before += dpp_shift<kRowShr + 1>(before);
  before += dpp_shift<kRowShr + 2>(before);
  before += dpp_shift<kRowShr + 4>(before);
  before += dpp_shift<kRowShr + 8>(before);
  before += dpp_shift<kRowBcast15, 0xa>(before);
  before += dpp_shift<kRowBcast31, 0xc>(before);
  const uint32_t total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(before), 63));
  before -= starts;
  // lanes since the last one (this lane included) in which a segment starts;
  // lane + 1 where there is none
  const uint64_t has = __ballot(starts != 0);
  const uint64_t upto = has & (~uint64_t(0) >> (63 - lane));
  const int dist = lane - (63 - __clzll(static_cast<long long>(upto)));  // clz(0) = 64
  TA s = tail, t;
  t = dpp_shift<kRowShr + 1>(s);
  s = dist >= 1 ? s + t : s;
  t = dpp_shift<kRowShr + 2>(s);
  s = dist >= 2 ? s + t : s;
  t = dpp_shift<kRowShr + 4>(s);
  s = dist >= 4 ? s + t : s;
  t = dpp_shift<kRowShr + 8>(s);
  s = dist >= 8 ? s + t : s;
  t = dpp_shift<kRowBcast15, 0xa>(s);
  s = dist > (lane & 15) ? s + t : s;
  t = dpp_shift<kRowBcast31, 0xc>(s);
  s = dist > (lane & 31) ? s + t : s;
  s = upto == 0 ? s + open : s;
  // the sum that is open before this lane; each start in the lane closes one
  TA acc = dpp_shift<kWaveShr1>(s, open);
  // The sums closed by the step's starts, in LDS in segment order, then
  // stored 64 at a time: stored from the lanes that close them, each of the
  // 8 stores touched the lines of most of the step's sums.
  constexpr int PARTS = static_cast<int>(kStep) / staged_sums<TA>(), LANES = 64 / PARTS;
#pragma unroll
  for (int h = 0; h < PARTS; h++) {
    const uint32_t from = h == 0 ? 0u : static_cast<uint32_t>(__builtin_amdgcn_readlane(
                                            static_cast<int>(before), h * LANES));
    const uint32_t to = h == PARTS - 1 ? total : static_cast<uint32_t>(__builtin_amdgcn_readlane(
                                                     static_cast<int>(before), (h + 1) * LANES));
    if (PARTS == 1 || lane / LANES == h) {
      uint32_t i = before - from;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (cont[k] == 0) staged[i] = acc;
        i += 1 + cont[k];
        acc = and_mask(acc, cont[k]) + v[k] * xv[k];
      }
    }
    // (a range's first start closes nothing: its offset is out of range)
    for (uint32_t i = from; i < to; i += 64)
      if (i + lane < to) store_sum(out, staged[i + lane - from], (seg + i + lane - 1) * SZ);
  }
  open = last_lane(s);
  seg += total;
}

// One workgroup per CU (the x slice and the staged sums fill its 160 KB of
// LDS): 16 waves, each streaming a contiguous range of entries with the loads
// of kStepsAhead steps in flight (3 KB each for FP32, 144 KB per CU). Without
// its stores the kernel streams at 6.4 TB/s; storing each sum from the lane
// that closes its segment cost 1.1 ms of the Zipf product, staged in LDS and
// stored 64 at a time 0.6 ms.
template <typename TV, typename TX, typename TA>
__global__ __launch_bounds__(64 * kSumWaves) void k_slice_sums(SliceArgs a) {
  __shared__ __attribute__((aligned(16))) TA xs[slice_cols<TA>()];
  __shared__ TA staged[kSumWaves * staged_sums<TA>()];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TV *pval = static_cast<const TV *>(a.pval);
  const TX *x = static_cast<const TX *>(a.x);
  for (uint32_t t = a.wg_tile[blockIdx.x]; t < a.wg_tile[blockIdx.x + 1]; t++) {
    const int64_t q = a.tile_slice[t];
    const int64_t in_group = (q % a.spg) * a.sw;
    const int64_t c0 = q / a.spg * a.group + in_group;
    int64_t n = a.sw < a.group - in_group ? a.sw : a.group - in_group;
    n = n < a.ncols - c0 ? n : a.ncols - c0;
    __syncthreads();  // the previous tile's gathers are done
#pragma unroll 8
    for (int i = tid; i < static_cast<int>(n); i += 64 * kSumWaves) xs[i] = to_acc<TA>(x[c0 + i]);
    __syncthreads();
    const uint32_t *te = a.tile_e + t * (kSumWaves + 1) + wave;
    const uint32_t *ts = a.tile_s + t * (kSumWaves + 1) + wave;
    const int64_t ea = te[0], eb = te[1];
    const uint32_t s0 = ts[0], nseg = ts[1] - s0;
    if (ea >= eb) continue;
    const rsrc_t out = make_rsrc(static_cast<TA *>(a.sums) + s0,
                                 static_cast<uint32_t>(nseg * sizeof(TA)));
    int64_t at = ea & ~(kStep - 1);
    TA open = 0;
    uint32_t seg = 0;
    StepRegs<TV> r[kStepsAhead];
#pragma unroll
    for (int j = 0; j < kStepsAhead; j++)
      if (at + j * kStep < eb) load_step<TV>(r[j], a.pcol, pval, at + j * kStep, lane);
    while (at < eb) {
#pragma unroll
      for (int j = 0; j < kStepsAhead; j++) {
        if (at < eb) {
          sum_step<TV, TA>(r[j], xs, lane, at, ea, eb, out, staged + wave * staged_sums<TA>(), open, seg);
          if (at + kStepsAhead * kStep < eb)
            load_step<TV>(r[j], a.pcol, pval, at + kStepsAhead * kStep, lane);
          at += kStep;
        }
      }
    }
    if (lane == 0) store_sum(out, open, (nseg - 1) * static_cast<uint32_t>(sizeof(TA)));
  }
}

struct RowsArgs {
  const void *sums;
  const uint16_t *seg_row;
  const uint32_t *seg_at;
  int64_t ns, rows_per, ngroups, nrows;
  void *y;
  double alpha, beta;
};

// Rows of a group per wave, at most: 5 KB of LDS (FP64 sums of segments in a
// 4-byte type; 1024 rows left 20 waves per CU and took 5 % longer) or 8 KB
// (FP64 sums with their compensation).
template <typename TA> constexpr int rows_per_wave() { return sizeof(TA) == 8 ? 512 : 640; }
constexpr int kRowsAhead = 16;  // slices whose sums are loaded together

// Bound by the latency of its loads: 16 slices' sums are loaded before they
// are added, from 32 waves per CU (Zipf FP32: 8 slices and 20 waves 1.14 ms,
// 16 and 32 0.75 ms).
// A group of rows is owned by GW waves (one, or the 16 waves of a large
// workgroup, with a barrier between slices). A row has at most one segment
// in a slice, so the lanes that add one slice's sums touch different rows,
// and LDS operations of a wave stay in order: the sums come in slice order.
template <typename TA, int GW>
__global__ __launch_bounds__(GW == 1 ? 256 : 64 * GW) void k_slice_rows(RowsArgs a) {
  constexpr bool kComp = sizeof(TA) == 8;
  constexpr int RW = rows_per_wave<TA>() * GW, GROUPS = GW == 1 ? 4 : 1, NL = 64 * GW;
  __shared__ double sm[GROUPS * RW * (kComp ? 2 : 1)];
  const int l = GW == 1 ? threadIdx.x & 63 : threadIdx.x, lane = threadIdx.x & 63;
  const int w = GW == 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  // (neighbouring groups, whose sums share cache lines, stay on one XCD)
  const int64_t b = map_block(blockIdx.x, gridDim.x / kXcds) * GROUPS + w;
  if (b >= a.ngroups) return;  // GW > 1: the whole workgroup
  double *acc = sm + w * RW * (kComp ? 2 : 1);
  [[maybe_unused]] double *low = acc + RW;
  const int64_t row0 = b * a.rows_per;
  const int nr = static_cast<int>(a.nrows - row0 < a.rows_per ? a.nrows - row0 : a.rows_per);
  for (int i = l; i < nr; i += NL) {
    acc[i] = 0;
    if constexpr (kComp) low[i] = 0;
  }
  if constexpr (GW > 1)
    __syncthreads();
  else
    __builtin_amdgcn_wave_barrier();
  const TA *sums = static_cast<const TA *>(a.sums);
  auto add = [&](uint32_t row, TA p) {
    if constexpr (kComp) {
      const double h = acc[row], s = h + p, bb = s - h;
      low[row] += (h - (s - bb)) + (p - bb);
      acc[row] = s;
    } else {
      __hip_atomic_fetch_add(acc + row, static_cast<double>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  for (int64_t q0 = 0; q0 < a.ns; q0 += 64) {
    const int64_t q = q0 + lane;
    const bool in = q < a.ns;
    const uint32_t st = in ? a.seg_at[b * a.ns + q] : 0u;
    const uint32_t en = in ? a.seg_at[(b + 1) * a.ns + q] : 0u;
    const int n = a.ns - q0 < 64 ? static_cast<int>(a.ns - q0) : 64;
    for (int i0 = 0; i0 < n; i0 += kRowsAhead) {
      // (lanes past the last slice hold empty ranges)
      TA p[kRowsAhead];
      uint32_t row[kRowsAhead];
#pragma unroll
      for (int d = 0; d < kRowsAhead; d++) {
        const uint32_t s = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(st), i0 + d));
        const uint32_t len =
            static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(en), i0 + d)) - s;
        p[d] = buf_load<TA>(make_rsrc(sums + s, len * static_cast<uint32_t>(sizeof(TA))),
                                 l * static_cast<uint32_t>(sizeof(TA)));
        row[d] = buf_load<uint16_t>(make_rsrc(a.seg_row + s, len * 2u), l * 2u);
      }
#pragma unroll
      for (int d = 0; d < kRowsAhead; d++) {
        const uint32_t s = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(st), i0 + d));
        const uint32_t e = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(en), i0 + d));
        if (static_cast<uint32_t>(l) < e - s) add(row[d], p[d]);
        for (uint32_t i = s + l + NL; i < e; i += NL) add(a.seg_row[i], sums[i]);
        if constexpr (GW > 1) __syncthreads();
      }
    }
  }
  if constexpr (GW == 1) __builtin_amdgcn_wave_barrier();
  TA *y = static_cast<TA *>(a.y) + row0;
  for (int i = l; i < nr; i += NL) {
    double s = acc[i];
    if constexpr (kComp) {
      // (an infinite sum leaves NaN in its compensation)
      if (__builtin_isfinite(s)) s += low[i];
    }
    double out = a.alpha * s;
    if (a.beta != 0) out += a.beta * static_cast<double>(y[i]);
    y[i] = static_cast<TA>(out);
  }
}

template <typename TY>
__global__ void k_scale_y(TY *y, int64_t nrows, int64_t ldy, int64_t k,
                          double beta) {
  DRX_GRID_LOOP(i, nrows * k) {
    const int64_t r = i % nrows, j = i / nrows;
    TY &v = y[r + j * ldy];
    if (beta == 0.0)
      v = TY(0);
    else
      v = static_cast<TY>(static_cast<double>(v) * beta);
  }
}

void check_panel_operands(const Plan &p, int vtype, const void *colind,
                          const void *vals) {
  const PanelSet &ps = *p.panels;
  DRX_REQUIRE(vtype == ps.vtype, "vtype differs from the panel layout's");
  DRX_REQUIRE(vals == ps.src_vals && colind == ps.src_colind,
              "the panel layout holds a copy of the colind/vals it was built "
              "from: pass those pointers (drx_plan_update_values re-packs new values)");
}

// false: no memory for the sums (nothing is launched then).
template <typename TV, typename TX, typename TA>
static bool run_slices(const Plan &p, const PanelSet &ps, const TX *x, int64_t ldx, TA *y,
                       int64_t ldy, int64_t k, double alpha, double beta, hipStream_t s) {
  SliceArgs a{};
  a.pcol = ps.pcol;
  a.pval = ps.pval;
  a.wg_tile = ps.wg_tile;
  a.tile_slice = ps.tile_slice;
  a.tile_e = ps.tile_e;
  a.tile_s = ps.tile_s;
  a.group = ps.group;
  a.spg = ps.spg;
  a.sw = ps.sw;
  a.ncols = p.ncols;
  RowsArgs b{};
  b.seg_row = ps.seg_row;
  b.seg_at = ps.seg_at;
  b.ns = ps.ns;
  b.rows_per = ps.rows_per;
  b.ngroups = ps.ngroups;
  b.nrows = p.nrows;
  // in the type that the sums have, as the other products take them
  b.alpha = static_cast<double>(static_cast<TA>(alpha));
  b.beta = static_cast<double>(static_cast<TA>(beta));
  void *sums = scratch_try(static_cast<size_t>(ps.nseg) * sizeof(TA), s);
  if (sums == nullptr) return false;
  try {
    a.sums = sums;
    b.sums = sums;
    for (int64_t j = 0; j < k; j++) {
      a.x = x + j * ldx;
      b.y = y + j * ldy;
      hipLaunchKernelGGL((k_slice_sums<TV, TX, TA>), dim3(static_cast<unsigned>(ps.nwg)),
                         dim3(64 * kSumWaves), 0, s, a);
      if (ps.group_waves == 1)
        hipLaunchKernelGGL((k_slice_rows<TA, 1>),
                           dim3(static_cast<unsigned>(((ps.ngroups + 3) / 4 + 7) / 8 * 8)), dim3(256), 0, s, b);
      else
        hipLaunchKernelGGL((k_slice_rows<TA, 16>), dim3(static_cast<unsigned>((ps.ngroups + 7) / 8 * 8)),
                           dim3(1024), 0, s, b);
      DRX_HIP(hipGetLastError());
    }
  } catch (...) {
    scratch_free(sums, s);
    throw;
  }
  scratch_free(sums, s);
  return true;
}

bool run_spmv_panels(const Plan &p, int vtype, const void *colind,
                     const void *vals, int xtype, const void *x, int64_t ldx,
                     int ytype, void *y, int64_t ldy, int64_t k, double alpha,
                     double beta, hipStream_t s) {
  const PanelSet &ps = *p.panels;
  check_panel_operands(p, vtype, colind, vals);
  DRX_REQUIRE(k >= 1 && y != nullptr, "bad output");
  DRX_REQUIRE(k == 1 || (ldx >= p.ncols && ldy >= p.nrows), "ldx/ldy too small");
  DRX_REQUIRE(static_cast<uint64_t>(p.ncols) * dtype_size(xtype) < (uint64_t(1) << 32),
              "the panel layout needs ncols * sizeof(x) < 4 GiB");
  if (p.nrows == 0) return true;
  DRX_REQUIRE(ytype == DRX_F64 || ytype == DRX_F32, "unsupported ytype");
  if (p.nnz == 0) {
    if (beta == 1.0) return true;
    if (ytype == DRX_F64)
      hipLaunchKernelGGL(k_scale_y<double>, grid_of(p.nrows * k), dim3(256), 0, s,
                         static_cast<double *>(y), p.nrows, ldy, k, beta);
    else
      hipLaunchKernelGGL(k_scale_y<float>, grid_of(p.nrows * k), dim3(256), 0, s,
                         static_cast<float *>(y), p.nrows, ldy, k, beta);
    DRX_HIP(hipGetLastError());
    return true;
  }
  DRX_REQUIRE(x != nullptr, "colind/vals/x is null");
#define DRX_RS(TV, TX, TA)                                                     \
  return run_slices<TV, TX, TA>(p, ps, static_cast<const TX *>(x), ldx,               \
                         static_cast<TA *>(y), ldy, k, alpha, beta, s)
  if (vtype == DRX_F64 && xtype == DRX_F64 && ytype == DRX_F64)
    DRX_RS(double, double, double);
  if (vtype == DRX_F32 && xtype == DRX_F32 && ytype == DRX_F32)
    DRX_RS(float, float, float);
  if (vtype == DRX_BF16 && xtype == DRX_BF16 && ytype == DRX_F32)
    DRX_RS(bf16, bf16, float);
  if (vtype == DRX_F16 && xtype == DRX_F16 && ytype == DRX_F32)
    DRX_RS(f16, f16, float);
  if (vtype == DRX_BF16 && xtype == DRX_F32 && ytype == DRX_F32)
    DRX_RS(bf16, float, float);
  if (vtype == DRX_F16 && xtype == DRX_F32 && ytype == DRX_F32)
    DRX_RS(f16, float, float);
  throw Error(DRX_ERR_UNSUPPORTED, "unsupported (vtype, xtype, ytype)");
#undef DRX_RS
}

// ---------------------------------------------------------------------------
// Building the layout
// ---------------------------------------------------------------------------
template <typename T> static T *dmalloc(int64_t n) {
  return static_cast<T *>(block_alloc(static_cast<size_t>(n) * sizeof(T)));
}

// Slice of every entry.
template <typename TI, typename TK>
__global__ void k_slice_key(const TI *colind, int64_t nnz, int64_t group, int64_t spg, int64_t sw,
                            TK *key, TI *iota) {
  DRX_GRID_LOOP(e, nnz) {
    const int64_t c = static_cast<int64_t>(colind[e]);
    int64_t q;
    if ((c | group) >> 32 == 0) {
      const uint32_t g = static_cast<uint32_t>(c) / static_cast<uint32_t>(group);
      const uint32_t in = static_cast<uint32_t>(c) - g * static_cast<uint32_t>(group);
      q = static_cast<int64_t>(g) * spg + in / static_cast<uint32_t>(sw);
    } else {
      q = c / group * spg + c % group / sw;
    }
    key[e] = static_cast<TK>(q);
    iota[e] = static_cast<TI>(e);
  }
}

// Each non-empty row's number at its first entry (the rest stays 0); a
// running maximum then gives every entry's row.
template <typename TI>
__global__ void k_row_marks(const TI *rowptr, int64_t base, int64_t nrows, int64_t nnz, int sent,
                            TI *mark) {
  DRX_GRID_LOOP(r, nrows) {
    const int64_t s = row_begin(rowptr, base, nrows, nnz, sent, r);
    if (row_begin(rowptr, base, nrows, nnz, sent, r + 1) > s) mark[s] = static_cast<TI>(r);
  }
}

// The copies in slice order, and each entry's row.
template <typename TI, typename TV, typename TK>
__global__ void k_gather_entries(const TI *perm, const TK *key, const TI *colind, const TV *vals,
                                 const TI *rowid, int64_t nnz, int64_t group, int64_t spg,
                                 int64_t sw, uint16_t *pcol, TV *pval, TI *prow) {
  DRX_GRID_LOOP(i, nnz) {
    const int64_t e = static_cast<int64_t>(perm[i]);
    const int64_t q = static_cast<int64_t>(key[i]);
    const int64_t g = spg == 1 ? q : q / spg;
    const int64_t c0 = g * group + (q - g * spg) * sw;
    pcol[i] = static_cast<uint16_t>((static_cast<int64_t>(colind[e]) - c0) << 1);
    pval[value_slot<TV>(i)] = vals[e];
    prow[i] = rowid[e];
  }
}

// Where segments start; entries that continue one are marked in pcol.
template <typename TI, typename TK>
__global__ void k_seg_flags(const TK *key, const TI *prow, int64_t nnz, uint16_t *pcol,
                            int32_t *flag) {
  DRX_GRID_LOOP(i, nnz) {
    const bool first = i == 0 || key[i] != key[i - 1] || prow[i] != prow[i - 1];
    flag[i] = first ? 1 : 0;
    if (!first) pcol[i] = static_cast<uint16_t>(pcol[i] | 1);
  }
}

template <typename TI>
__global__ void k_seg_fill(const int32_t *flag, const int32_t *segid, const TI *prow, int64_t nnz,
                           int64_t nseg, int64_t rows_per, TI *seg_prow, uint16_t *seg_row,
                           uint32_t *seg_ptr) {
  DRX_GRID_LOOP(i, nnz) {
    if (flag[i]) {
      const int64_t s = segid[i] - 1;
      const int64_t r = static_cast<int64_t>(prow[i]);
      seg_prow[s] = prow[i];
      seg_row[s] = static_cast<uint16_t>(r % rows_per);
      seg_ptr[s] = static_cast<uint32_t>(i);
    }
    if (i == 0) seg_ptr[nseg] = static_cast<uint32_t>(nnz);
  }
}

// First entry and first segment of every slice.
template <typename TK>
__global__ void k_slice_bounds(const TK *key, const int32_t *segid, int64_t nnz, int64_t nseg,
                               int64_t ns, uint32_t *entry, uint32_t *seg) {
  DRX_GRID_LOOP(q, ns + 1) {
    int64_t lo = 0, hi = nnz;  // first i with key[i] >= q
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo) / 2;
      if (static_cast<int64_t>(key[mid]) >= q)
        hi = mid;
      else
        lo = mid + 1;
    }
    entry[q] = static_cast<uint32_t>(lo);
    seg[q] = static_cast<uint32_t>(lo < nnz ? segid[lo] - 1 : nseg);
  }
}

// First segment of row group b (b <= ngroups) in every slice.
template <typename TI>
__global__ void k_group_bounds(const TI *seg_prow, const uint32_t *slice_seg, int64_t ns,
                               int64_t ngroups, int64_t rows_per, uint32_t *seg_at) {
  DRX_GRID_LOOP(i, ns * (ngroups + 1)) {
    const int64_t b = i / ns, q = i - b * ns;
    int64_t lo = slice_seg[q], hi = slice_seg[q + 1];  // first segment of a row >= b * rows_per
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo) / 2;
      if (static_cast<int64_t>(seg_prow[mid]) >= b * rows_per)
        hi = mid;
      else
        lo = mid + 1;
    }
    seg_at[i] = static_cast<uint32_t>(lo);
  }
}

// The ranges of a tile's waves: equal parts, moved up to segment starts.
// bounds = first and last entry of every tile.
__global__ void k_tile_ranges(const uint32_t *bounds, int64_t ntiles, const int32_t *segid,
                              const uint32_t *seg_ptr, uint32_t *tile_e, uint32_t *tile_s) {
  DRX_GRID_LOOP(i, ntiles * (kSumWaves + 1)) {
    const int64_t t = i / (kSumWaves + 1), w = i % (kSumWaves + 1);
    const int64_t a = bounds[2 * t], b = bounds[2 * t + 1];
    const int64_t pos = a + (b - a) * w / kSumWaves;
    const uint32_t s = pos == 0 ? 0u : static_cast<uint32_t>(segid[pos - 1]);
    tile_s[i] = s;
    tile_e[i] = seg_ptr[s];
  }
}

template <typename TI, typename TV>
__global__ void k_repack(const TI *perm, const TV *vals, int64_t nnz, TV *pval) {
  DRX_GRID_LOOP(i, nnz) { pval[value_slot<TV>(i)] = vals[static_cast<int64_t>(perm[i])]; }
}

// Tiles: the entries (slice_e: first entry of every slice) dealt to nwg
// workgroups in order, each taking about the same number of entries plus the
// cost of the x slices it loads.
struct Tiles {
  std::vector<uint32_t> wg_tile, slice, bounds;
};
static Tiles deal_tiles(const std::vector<uint32_t> &slice_e, int64_t nwg) {
  // an x slice (128 KB) costs about as much as 20000 entries of 6 bytes; a
  // workgroup does not start on a slice for less than this many entries
  constexpr int64_t kLoad = 20000, kLeast = 8192;
  const int64_t ns = static_cast<int64_t>(slice_e.size()) - 1;
  int64_t used = 0;
  for (int64_t q = 0; q < ns; q++) used += slice_e[q + 1] > slice_e[q];
  // (a workgroup that starts inside a slice loads it again)
  const int64_t share = (static_cast<int64_t>(slice_e[ns]) + (used + nwg) * kLoad) / nwg + 1;
  Tiles t;
  t.wg_tile.push_back(0);
  int64_t left = share;  // (what a workgroup leaves or takes too much, the next one gets)
  bool fresh = true;
  for (int64_t q = 0; q < ns; q++) {
    int64_t at = slice_e[q];
    const int64_t end = slice_e[q + 1];
    while (at < end) {
      const bool last = static_cast<int64_t>(t.wg_tile.size()) == nwg;
      if (!last && !fresh && left - kLoad < kLeast) {
        t.wg_tile.push_back(static_cast<uint32_t>(t.slice.size()));
        left += share;
        fresh = true;
      }
      const bool now_last = static_cast<int64_t>(t.wg_tile.size()) == nwg;
      int64_t take = std::max<int64_t>(left - kLoad, kLeast);
      if (now_last || end - at - take < kLeast) take = end - at;
      take = std::min(take, end - at);
      t.slice.push_back(static_cast<uint32_t>(q));
      t.bounds.push_back(static_cast<uint32_t>(at));
      t.bounds.push_back(static_cast<uint32_t>(at + take));
      at += take;
      left -= kLoad + take;
      fresh = false;
    }
  }
  while (static_cast<int64_t>(t.wg_tile.size()) <= nwg)
    t.wg_tile.push_back(static_cast<uint32_t>(t.slice.size()));
  return t;
}

template <typename TI, typename TV, typename TK>
static void build_panels(Plan &p, PanelSet &ps, const TI *colind, const TV *vals, int num_cus,
                         hipStream_t s) {
  const int64_t nnz = p.nnz;
  const int64_t padded = (nnz + kStep - 1) / kStep * kStep;
  std::vector<void *> tmp;
  auto temp = [&](auto *&ptr, int64_t n) {
    ptr = dmalloc<std::remove_reference_t<decltype(*ptr)>>(n);
    tmp.push_back(ptr);
  };
  auto release = [&](void *ptr) {
    block_free(ps.device, ptr);
    tmp.erase(std::find(tmp.begin(), tmp.end(), ptr));
  };
  try {
    TI *iota, *rowid, *mark, *prow, *seg_prow;
    TK *key, *key_sorted;
    int32_t *flag, *segid;
    uint32_t *seg_ptr, *slice_e, *slice_s, *bounds;
    char *work;
    temp(iota, nnz);
    temp(key, nnz);
    temp(key_sorted, nnz);
    ps.perm = dmalloc<TI>(nnz);
    hipLaunchKernelGGL((k_slice_key<TI, TK>), grid_of(nnz), dim3(256), 0, s, colind, nnz, ps.group,
                       ps.spg, ps.sw, key, iota);
    DRX_HIP(hipGetLastError());
    int end_bit = 1;
    while ((int64_t(1) << end_bit) < std::max<int64_t>(ps.ns, 2)) end_bit++;
    size_t tb = 0;
    DRX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, key, key_sorted, iota,
                                               static_cast<TI *>(ps.perm),
                                               static_cast<int>(nnz), 0, end_bit, s));
    temp(work, static_cast<int64_t>(tb));
    DRX_HIP(hipcub::DeviceRadixSort::SortPairs(work, tb, key, key_sorted, iota,
                                               static_cast<TI *>(ps.perm),
                                               static_cast<int>(nnz), 0, end_bit, s));
    DRX_HIP(hipStreamSynchronize(s));
    release(work);
    release(key);
    // every entry's row
    mark = iota;
    temp(rowid, nnz);
    DRX_HIP(hipMemsetAsync(mark, 0, static_cast<size_t>(nnz) * sizeof(TI), s));
    hipLaunchKernelGGL(k_row_marks<TI>, grid_of(p.nrows), dim3(256), 0, s,
                       static_cast<const TI *>(p.rowptr), p.base, p.nrows, nnz, p.has_sentinel,
                       mark);
    DRX_HIP(hipGetLastError());
    tb = 0;
    DRX_HIP(hipcub::DeviceScan::InclusiveScan(nullptr, tb, mark, rowid, hipcub::Max(),
                                              static_cast<int>(nnz), s));
    temp(work, static_cast<int64_t>(tb));
    DRX_HIP(hipcub::DeviceScan::InclusiveScan(work, tb, mark, rowid, hipcub::Max(),
                                              static_cast<int>(nnz), s));
    prow = iota;  // (the marks are read: the stream is in order)
    ps.pcol = dmalloc<uint16_t>(padded);
    ps.pval = dmalloc<TV>(padded);
    DRX_HIP(hipMemsetAsync(ps.pcol + (padded - kStep), 0, kStep * sizeof(uint16_t), s));
    hipLaunchKernelGGL((k_gather_entries<TI, TV, TK>), grid_of(nnz), dim3(256), 0, s,
                       static_cast<const TI *>(ps.perm), key_sorted, colind, vals, rowid, nnz,
                       ps.group, ps.spg, ps.sw, ps.pcol, static_cast<TV *>(ps.pval), prow);
    DRX_HIP(hipGetLastError());
    DRX_HIP(hipStreamSynchronize(s));
    release(work);
    release(rowid);
    temp(flag, nnz);
    temp(segid, nnz);
    hipLaunchKernelGGL((k_seg_flags<TI, TK>), grid_of(nnz), dim3(256), 0, s, key_sorted, prow, nnz,
                       ps.pcol, flag);
    DRX_HIP(hipGetLastError());
    tb = 0;
    DRX_HIP(hipcub::DeviceScan::InclusiveSum(nullptr, tb, flag, segid, static_cast<int>(nnz), s));
    temp(work, static_cast<int64_t>(tb));
    DRX_HIP(hipcub::DeviceScan::InclusiveSum(work, tb, flag, segid, static_cast<int>(nnz), s));
    int32_t nseg32 = 0;
    DRX_HIP(hipMemcpyAsync(&nseg32, segid + nnz - 1, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    DRX_HIP(hipStreamSynchronize(s));
    ps.nseg = nseg32;

    // Row groups: about 52 segments of a slice per wave (a wave adds 64 at
    // once; lengths vary around the mean), at least 64 rows, at most what
    // the LDS share holds, and enough groups for 20 waves on every CU.
    // Where the table of groups would outgrow the entries, groups of 16
    // waves.
    const int64_t most = sizeof(TV) == 8 ? rows_per_wave<double>() : rows_per_wave<float>();
    int64_t rp = static_cast<int64_t>(52.0 * static_cast<double>(ps.ns) *
                                      static_cast<double>(p.nrows) / static_cast<double>(ps.nseg));
    rp = std::min(rp, p.nrows / (20 * int64_t(num_cus)));
    rp = std::min(std::max<int64_t>(rp & ~int64_t(63), 64), most);
    if ((p.nrows + rp - 1) / rp * ps.ns > std::max<int64_t>(nnz, int64_t(1) << 22)) rp = most;
    ps.group_waves = 1;
    if ((p.nrows + rp - 1) / rp * ps.ns > std::max<int64_t>(nnz, int64_t(1) << 22)) {
      rp = most * 16;
      ps.group_waves = 16;
    }
    ps.rows_per = rp;
    ps.ngroups = (p.nrows + rp - 1) / rp;

    ps.seg_row = dmalloc<uint16_t>(ps.nseg);
    temp(seg_prow, ps.nseg);
    temp(seg_ptr, ps.nseg + 1);
    hipLaunchKernelGGL(k_seg_fill<TI>, grid_of(nnz), dim3(256), 0, s, flag, segid, prow, nnz,
                       ps.nseg, ps.rows_per, seg_prow, ps.seg_row, seg_ptr);
    temp(slice_e, ps.ns + 1);
    temp(slice_s, ps.ns + 1);
    hipLaunchKernelGGL(k_slice_bounds<TK>, grid_of(ps.ns + 1), dim3(256), 0, s, key_sorted, segid,
                       nnz, ps.nseg, ps.ns, slice_e, slice_s);
    ps.seg_at = dmalloc<uint32_t>(ps.ns * (ps.ngroups + 1));
    hipLaunchKernelGGL(k_group_bounds<TI>, grid_of(ps.ns * (ps.ngroups + 1)), dim3(256), 0, s,
                       seg_prow, slice_s, ps.ns, ps.ngroups, ps.rows_per, ps.seg_at);
    DRX_HIP(hipGetLastError());
    std::vector<uint32_t> h_slice_e(ps.ns + 1);
    DRX_HIP(hipMemcpyAsync(h_slice_e.data(), slice_e, (ps.ns + 1) * sizeof(uint32_t),
                           hipMemcpyDeviceToHost, s));
    DRX_HIP(hipStreamSynchronize(s));
    // Two workgroups for every CU (one runs at a time), fewer when they
    // would get less than 16384 entries each.
    ps.nwg = std::max<int64_t>(1, std::min<int64_t>(2 * int64_t(num_cus), nnz / 16384));
    const Tiles t = deal_tiles(h_slice_e, ps.nwg);
    const int64_t nt = static_cast<int64_t>(t.slice.size());
    temp(bounds, 2 * nt);
    ps.wg_tile = dmalloc<uint32_t>(ps.nwg + 1);
    ps.tile_slice = dmalloc<uint32_t>(nt);
    ps.tile_e = dmalloc<uint32_t>(nt * (kSumWaves + 1));
    ps.tile_s = dmalloc<uint32_t>(nt * (kSumWaves + 1));
    DRX_HIP(hipMemcpyAsync(bounds, t.bounds.data(), 2 * nt * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    DRX_HIP(hipMemcpyAsync(ps.tile_slice, t.slice.data(), nt * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    DRX_HIP(hipMemcpyAsync(ps.wg_tile, t.wg_tile.data(), (ps.nwg + 1) * sizeof(uint32_t),
                           hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_tile_ranges, grid_of(nt * (kSumWaves + 1)), dim3(256), 0, s, bounds, nt,
                       segid, seg_ptr, ps.tile_e, ps.tile_s);
    DRX_HIP(hipGetLastError());
    DRX_HIP(hipStreamSynchronize(s));
  } catch (...) {
    owned_free(ps.device, tmp);
    throw;
  }
  for (void *q : tmp) block_free(ps.device, q);
}

// Slices of panels of `width` columns over ncols columns: groups, and how many
// slices hold columns (the last panel's may be fewer).
static void cut_slices(PanelSet &ps, int64_t ncols) {
  const int64_t slice = ps.vtype == DRX_F64 ? slice_cols<double>() : slice_cols<float>();
  if (ps.width <= slice) {  // whole panels share a slice
    ps.group = ps.sw = slice / ps.width * ps.width;
    ps.spg = 1;
  } else {  // a panel is cut into equal slices
    ps.group = ps.width;
    ps.spg = (ps.width + slice - 1) / slice;
    ps.sw = (ps.width + ps.spg - 1) / ps.spg;
  }
  const int64_t full = ncols / ps.group;
  ps.ns = std::max<int64_t>(1, full * ps.spg + (ncols - full * ps.group + ps.sw - 1) / ps.sw);
}

// Whether products are faster over slices than over the share's own arrays.
// Below some 8M entries the slice kernels' own steps (33 us however few entries)
// outweigh the gathers, and where a wave's rows hold only a few entries of a
// slice k_slice_rows reads mostly empty ranges. us per product, random columns,
// n x n and fewer rows, own arrays / slices:
//   FP32 n = 600K, 12 and 16 entries per row 46 / 48, 85 / 53; 1.2M, 5 and 8: 43 /
//   53, 64 / 58; 4M, 4: 236 / 99; 30M, 2 (1.4 entries per wave and slice), 3 (2.1)
//   and 4 (2.8): 1147 / 1527, 1148 / 1112, 1217 / 893
//   FP64 n = 1.2M, 5 and 8: 75 / 93, 115 / 103; 12M, 6 (4.2) and 8 (5.6): 1150 /
//   1196, 1147 / 989; 30M, 2 (0.6) and 16 (4.5): 1212 / 8411, 1147 / 1256
//   BF16 n = 2M, 3 and 4: 41 / 51, 59 / 54; 30M, 3 (2.1) and 4 (2.8): 1079 / 1088,
//   1123 / 867
static bool slices_pay(int vtype, int64_t nnz, int64_t nrows, int64_t ns) {
  const int64_t rows = vtype == DRX_F64 ? rows_per_wave<double>() : rows_per_wave<float>();
  const double cells = static_cast<double>((nrows + rows - 1) / rows) * static_cast<double>(ns);
  return nnz >= 8000000 && static_cast<double>(nnz) >= (vtype == DRX_F64 ? 5.0 : 2.5) * cells;
}

static int64_t default_width(int vtype) {
  return std::max<int64_t>(4096, (int64_t(2) << 20) / static_cast<int64_t>(dtype_size(vtype)));
}

// Builds the panel layout of p (drx_plan_set_panels).
static void set_panels(Plan &p, int vtype, const void *colind, const void *vals,
                     int64_t panel_cols, hipStream_t s) {
  DRX_REQUIRE(p.panels == nullptr, "the plan already has a panel layout");
  DRX_REQUIRE(p.nnz == 0 || (colind && vals), "colind/vals is null");
  DRX_REQUIRE(p.nnz <= INT32_MAX, "the panel layout is limited to 2^31-1 entries");
  DRX_REQUIRE(vtype >= DRX_F64 && vtype <= DRX_F16, "bad vtype");
  PanelSet *ps = new PanelSet();
  ps->vtype = vtype;
  ps->src_colind = colind;
  ps->src_vals = vals;
  ps->width = panel_cols > 0 ? panel_cols : default_width(vtype);
  ps->npanels = std::max<int64_t>(1, (p.ncols + ps->width - 1) / ps->width);
  try {
    DRX_REQUIRE(ps->npanels <= (int64_t(1) << 20), "too many panels");
    cut_slices(*ps, p.ncols);
    if (p.nnz > 0) {
      int cus = 0;
      DRX_HIP(hipGetDevice(&ps->device));
      DRX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ps->device));
#define DRX_BPK(TI, TV, TK)                                                    \
  build_panels<TI, TV, TK>(p, *ps, static_cast<const TI *>(colind),            \
                           static_cast<const TV *>(vals), cus, s)
#define DRX_BP(TI, TV)                                                         \
  do {                                                                         \
    if (ps->ns <= 65536)                                                       \
      DRX_BPK(TI, TV, uint16_t);                                               \
    else                                                                       \
      DRX_BPK(TI, TV, uint32_t);                                               \
  } while (0)
      const bool i32 = p.itype == DRX_I32;
      switch (vtype) {
        case DRX_F64: if (i32) DRX_BP(int32_t, double); else DRX_BP(int64_t, double); break;
        case DRX_F32: if (i32) DRX_BP(int32_t, float); else DRX_BP(int64_t, float); break;
        default: if (i32) DRX_BP(int32_t, uint16_t); else DRX_BP(int64_t, uint16_t); break;
      }
#undef DRX_BP
#undef DRX_BPK
      const size_t sums = static_cast<size_t>(ps->nseg) * (vtype == DRX_F64 ? 8 : 4);
      scratch_reserve(ps->device, sums, s);
      ps->scratch = sums;
    } else {
      ps->npanels = 0;
    }
  } catch (...) {
    free_panels(ps);
    throw;
  }
  p.panels = ps;
}

// Column profile of a share for the automatic panel choice: up to 2048 row
// blocks spread over the share, one wave each; a wave compares up to 256
// entries of its block's window with the window's middle column and counts
// those within `near` columns of it. out = {near, sampled}.
template <typename TI>
__global__ void k_col_profile(const BlockRec *rec, int64_t nblocks, const TI *colind,
                              int64_t near, unsigned long long *out) {
  const int64_t S = nblocks < 2048 ? nblocks : 2048;
  const int lane = threadIdx.x & 63;
  unsigned long long n_near = 0, n_seen = 0;
  for (int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / 64; i < S;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x / 64) {
    const BlockRec b = rec[i * nblocks / S];
    const int64_t n = b.es - b.e0;
    if (n < 2) continue;
    const int64_t mid = static_cast<int64_t>(colind[b.e0 + n / 2]);
    const int64_t step = n > 256 ? n / 256 : 1;
    for (int64_t j = lane; j < 256 && j * step < n; j += 64) {
      const int64_t c = static_cast<int64_t>(colind[b.e0 + j * step]);
      const int64_t d = c > mid ? c - mid : mid - c;
      n_near += d <= near ? 1 : 0;
      n_seen += 1;
    }
  }
  atomicAdd(&out[0], n_near);
  atomicAdd(&out[1], n_seen);
}

// Whether the panel layout pays for plan p (see drx_plan_auto_panels).
static bool panels_pay(const Plan &p, int vtype, const void *colind, hipStream_t s) {
  const int64_t sx = static_cast<int64_t>(dtype_size(vtype));
  if (tuned_auto_panels() == 0) return false;
  if (p.panels != nullptr || p.nnz == 0 || p.nnz > INT32_MAX) return false;
  if (p.ncols * sx <= (int64_t(4) << 20)) return false;          // x fits one XCD's L2
  if (p.nnz < 4 * p.nrows) return false;  // too few gathers for a copy of the entries
  if (static_cast<uint64_t>(p.ncols) * sx >= (uint64_t(1) << 32)) return false;
  PanelSet shape;
  shape.vtype = vtype;
  shape.width = default_width(vtype);
  cut_slices(shape, p.ncols);
  if (!slices_pay(vtype, p.nnz, p.nrows, shape.ns)) return false;
  // device memory for the most that building holds at once, with columns so
  // scattered that every entry is a segment: positions, sorted slices,
  // permutation, copies, flags, segment numbers, rows and first entries (34
  // bytes per entry beside the value with 32-bit indices)
  const int64_t si = p.itype == DRX_I32 ? 4 : 8;
  size_t free_b = 0, total_b = 0;
  DRX_HIP(hipMemGetInfo(&free_b, &total_b));
  free_b += blocks_kept(p.device);
  if (static_cast<double>(free_b) < 1.1 * static_cast<double>(p.nnz) * (3 * si + 22 + sx))
    return false;
  unsigned long long *d = static_cast<unsigned long long *>(
      scratch_alloc(2 * sizeof(unsigned long long), s));
  unsigned long long h[2] = {0, 0};
  try {
    DRX_HIP(hipMemsetAsync(d, 0, 2 * sizeof(unsigned long long), s));
    const int64_t near = (int64_t(1) << 20) / sx;  // 1 MiB of x either side
    if (p.itype == DRX_I32)
      hipLaunchKernelGGL(k_col_profile<int32_t>, dim3(32), dim3(256), 0, s, p.rec, p.nblocks,
                         static_cast<const int32_t *>(colind), near, d);
    else
      hipLaunchKernelGGL(k_col_profile<int64_t>, dim3(32), dim3(256), 0, s, p.rec, p.nblocks,
                         static_cast<const int64_t *>(colind), near, d);
    DRX_HIP(hipGetLastError());
    DRX_HIP(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s));
    DRX_HIP(hipStreamSynchronize(s));
  } catch (...) {
    scratch_free(d, s);
    throw;
  }
  scratch_free(d, s);
  // scattered: fewer than half of the sampled entries near their block's
  // middle column
  return h[1] > 0 && 2 * h[0] < h[1];
}

}  // namespace drx

using namespace drx;

extern "C" {

int drx_plan_set_panels(drx_plan plan, int vtype, const void *colind,
                        const void *vals, int64_t panel_cols,
                        drx_stream_t stream) {
  return guarded([&] {
    DRX_REQUIRE(plan != nullptr, "plan is null");
    set_panels(*reinterpret_cast<Plan *>(plan), vtype, colind, vals, panel_cols,
               static_cast<hipStream_t>(stream));
  });
}

int drx_plan_auto_panels(drx_plan plan, int vtype, const void *colind,
                         const void *vals, drx_stream_t stream, int *built) {
  return guarded([&] {
    if (built) *built = 0;
    DRX_REQUIRE(plan != nullptr, "plan is null");
    Plan &p = *reinterpret_cast<Plan *>(plan);
    DRX_REQUIRE(vtype >= DRX_F64 && vtype <= DRX_F16, "bad vtype");
    DRX_REQUIRE(p.nnz == 0 || (colind && vals), "colind/vals is null");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    DRX_HIP(hipStreamIsCapturing(s, &cs));
    DRX_REQUIRE(cs == hipStreamCaptureStatusNone, "the stream is being captured");
    if (!panels_pay(p, vtype, colind, s)) return;
    try {
      set_panels(p, vtype, colind, vals, 0, s);
    } catch (const Error &e) {
      if (e.status != DRX_ERR_NOMEM) throw;
      return;  // (another user of the device was faster)
    }
    if (built) *built = 1;
  });
}

int drx_plan_update_values(drx_plan plan, const void *vals, drx_stream_t stream) {
  return guarded([&] {
    DRX_REQUIRE(plan != nullptr, "plan is null");
    Plan &p = *reinterpret_cast<Plan *>(plan);
    DRX_REQUIRE(p.panels != nullptr, "the plan has no panel layout");
    DRX_REQUIRE(p.nnz == 0 || vals != nullptr, "vals is null");
    PanelSet &ps = *p.panels;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (p.nnz > 0) {
      const bool i32 = p.itype == DRX_I32;
#define DRX_RP(TI, TV)                                                         \
  hipLaunchKernelGGL((k_repack<TI, TV>), grid_of(p.nnz), dim3(256), 0, s,      \
                     static_cast<const TI *>(ps.perm),                         \
                     static_cast<const TV *>(vals), p.nnz,                     \
                     static_cast<TV *>(ps.pval))
      switch (ps.vtype) {
        case DRX_F64: if (i32) DRX_RP(int32_t, double); else DRX_RP(int64_t, double); break;
        case DRX_F32: if (i32) DRX_RP(int32_t, float); else DRX_RP(int64_t, float); break;
        default: if (i32) DRX_RP(int32_t, uint16_t); else DRX_RP(int64_t, uint16_t); break;
      }
#undef DRX_RP
      DRX_HIP(hipGetLastError());
    }
    ps.src_vals = vals;
  });
}

int drx_plan_panels(drx_plan plan, int64_t *npanels, int64_t *panel_cols,
                    int64_t *segments) {
  return guarded([&] {
    DRX_REQUIRE(plan != nullptr, "plan is null");
    const Plan &p = *reinterpret_cast<Plan *>(plan);
    const PanelSet *ps = p.panels;
    if (npanels) *npanels = ps ? ps->npanels : 0;
    if (panel_cols) *panel_cols = ps ? ps->width : 0;
    if (segments) *segments = ps ? ps->nseg : 0;
  });
}

}  // extern "C"
