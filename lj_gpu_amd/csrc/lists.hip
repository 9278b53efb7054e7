// lists.hip — neighbour lists on the device (see lists.h).
//
// The Verlet-list build follows the reference's makepair()/sortpair()
// (cpu_ref/force_aos.cpp:100-140; full list cuda/force_cuda.cu:122-163): the
// same pair predicate, evaluated unfused so every pair decision is
// bit-identical to the reference's, and the same CSR (rows ascending in i,
// partners ascending in j). The O(N^2) pair scan is replaced by a cell list:
//   1. bin particles into cells at least half the search length wide (a
//      radius-2 stencil; the search length and radius 1 for small boxes);
//   2. search each cell's stencil with one wavefront per cell, writing rows
//      into a per-row slab (an exact count-then-fill pass when a row
//      overflows it), and scan the row lengths into row pointers;
//   3. sort every row into place (or, for the MD loop, copy rows in the
//      build's own, position-determined order).
// Derived layouts (full list from a half list, ELL, LDS tiles, and the
// spatial particle order the tiles may follow) are built here from the
// device CSR, so a list never round-trips through the host.
#include "lists.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

namespace ljgpu {

namespace {

int hip_err(hipError_t e, const char* what) {
  return set_error(e == hipErrorOutOfMemory ? LJGPU_ERR_OUT_OF_MEMORY : LJGPU_ERR_HIP,
                   std::string(what) + ": " + hipGetErrorString(e));
}

#define LTRY(expr, what)                          \
  do {                                            \
    hipError_t e_ = (expr);                       \
    if (e_ != hipSuccess) return hip_err(e_, what); \
  } while (0)

#define LCHECK(call)        \
  do {                      \
    int rc_ = (call);       \
    if (rc_) return rc_;    \
  } while (0)

constexpr int kBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;
constexpr int64_t kScanSmall = 16384;  // values scanned by one workgroup
constexpr int64_t kScanTiles = 1024;   // tiles whose sums every workgroup adds up itself

int grid_for(int64_t items, int block, int cap = 65535 * 8) {
  const int64_t g = (items + block - 1) / block;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(g, cap)));
}

// ---------------------------------------------------------------------------
// Small kernels
// ---------------------------------------------------------------------------
template <class T>
__global__ void k_fill(T* __restrict__ a, int64_t n, T v) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    a[t] = v;
}

template <class T>
int fill(hipStream_t s, T* a, int64_t n, T v) {
  if (n <= 0) return LJGPU_OK;
  k_fill<T><<<grid_for(n, kBlock), kBlock, 0, s>>>(a, n, v);
  LTRY(hipGetLastError(), "fill kernel");
  return LJGPU_OK;
}

// Exclusive scan of one value per thread over the workgroup; *total receives
// the sum. `sh` holds one value per wavefront.
template <class T>
__device__ __forceinline__ T block_exclusive(T v, T* total, T* sh) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  T inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T t = __shfl_up(inc, d, 64);
    if (lane >= d) inc += t;
  }
  if (lane == 63) sh[wid] = inc;
  __syncthreads();
  T off = 0, tot = 0;
  for (int w = 0; w < static_cast<int>(blockDim.x) / 64; w++) {
    const T x = sh[w];
    off += w < wid ? x : 0;
    tot += x;
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

// Smallest and largest of one pair per thread over the workgroup, for thread 0.
__device__ __forceinline__ void block_extrema(int32_t& lo, int32_t& hi, int32_t* slo,
                                              int32_t* shi) {
  for (int d = 32; d > 0; d >>= 1) {
    lo = min(lo, __shfl_xor(lo, d, 64));
    hi = max(hi, __shfl_xor(hi, d, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    slo[threadIdx.x >> 6] = lo;
    shi[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  for (int w = 0; w < static_cast<int>(blockDim.x) / 64; w++) {
    lo = min(lo, slo[w]);
    hi = max(hi, shi[w]);
  }
  __syncthreads();
}

__device__ __forceinline__ int32_t clamp_i32(int64_t v) {
  return static_cast<int32_t>(std::min<int64_t>(v, INT32_MAX));
}

// Exclusive scan (values clamped to int32; the host rejects totals above
// INT32_MAX), out[n] = total, with the sum and extrema of the input in *res
// (null: not wanted). Up to kScanSmall values: one workgroup, a contiguous
// piece per thread. More: a pass that sums tiles of kScanTile values, and one that scans
// each tile from the sum of the tiles before it, which every workgroup adds
// up itself (SUMS: taken from sums scanned by k_scan_sums, for lists of many
// tiles).
__global__ __launch_bounds__(1024) void k_scan_small(const int32_t* __restrict__ in, int32_t n,
                                                     int32_t* __restrict__ out,
                                                     ScanStats* __restrict__ res) {
  __shared__ int64_t sh[16];
  __shared__ int32_t slo[16], shi[16];
  const int32_t piece = ((n + 1023) / 1024 + 3) / 4 * 4;
  const int32_t t0 = threadIdx.x * piece, t1 = min(t0 + piece, n);
  int64_t v = 0;
  int32_t lo = INT32_MAX, hi = INT32_MIN;
#pragma unroll 4
  for (int32_t t = t0; t < t1; t++) {
    const int32_t x = in[t];
    v += x;
    lo = min(lo, x);
    hi = max(hi, x);
  }
  int64_t total;
  int64_t run = block_exclusive<int64_t>(v, &total, sh);
#pragma unroll 4
  for (int32_t t = t0; t < t1; t++) {
    out[t] = clamp_i32(run);
    run += in[t];
  }
  if (threadIdx.x == 0) out[n] = clamp_i32(total);
  if (!res) return;
  block_extrema(lo, hi, slo, shi);
  if (threadIdx.x == 0) *res = ScanStats{total, lo, hi};
}

struct ScanTile {
  int64_t sum;
  int32_t lo, hi;
};

// The kScanItems values of this thread in its tile (0 past the end).
__device__ __forceinline__ void scan_load(const int32_t* __restrict__ in, int64_t n, int64_t base,
                                          int32_t (&v)[kScanItems]) {
  if (base + kScanItems <= n) {
#pragma unroll
    for (int q = 0; q < kScanItems / 4; q++) {
      const int4 x = reinterpret_cast<const int4*>(in + base)[q];
      v[4 * q] = x.x;
      v[4 * q + 1] = x.y;
      v[4 * q + 2] = x.z;
      v[4 * q + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int r = 0; r < kScanItems; r++) v[r] = base + r < n ? in[base + r] : 0;
  }
}

__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int32_t* __restrict__ in, int64_t n,
                                                        ScanTile* __restrict__ tiles) {
  __shared__ int64_t sh[kBlock / 64];
  __shared__ int32_t slo[kBlock / 64], shi[kBlock / 64];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int32_t v[kScanItems];
  scan_load(in, n, base, v);
  int64_t sum = 0;
  int32_t lo = INT32_MAX, hi = INT32_MIN;
#pragma unroll
  for (int r = 0; r < kScanItems; r++) {
    sum += v[r];
    if (base + r < n) {
      lo = min(lo, v[r]);
      hi = max(hi, v[r]);
    }
  }
  int64_t total;
  (void)block_exclusive<int64_t>(sum, &total, sh);
  block_extrema(lo, hi, slo, shi);
  if (threadIdx.x == 0) tiles[blockIdx.x] = ScanTile{total, lo, hi};
}

// Exclusive scan of the tile sums in place (one workgroup).
__global__ __launch_bounds__(kBlock) void k_scan_sums(ScanTile* __restrict__ tiles, int64_t nb) {
  __shared__ int64_t sh[kBlock / 64];
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += kBlock) {
    const int64_t t = b0 + threadIdx.x;
    const int64_t v = t < nb ? tiles[t].sum : 0;
    int64_t tot;
    const int64_t ex = block_exclusive<int64_t>(v, &tot, sh);
    if (t < nb) tiles[t].sum = carry + ex;
    carry += tot;
  }
}

template <bool SUMS>
__global__ __launch_bounds__(kBlock) void k_scan_apply(const int32_t* __restrict__ in, int64_t n,
                                                       const ScanTile* __restrict__ tiles,
                                                       int32_t* __restrict__ out,
                                                       ScanStats* __restrict__ res) {
  __shared__ int64_t sh[kBlock / 64];
  __shared__ int32_t slo[kBlock / 64], shi[kBlock / 64];
  int64_t carry = 0;
  if (SUMS) {
    carry = tiles[blockIdx.x].sum;
  } else {
    int64_t before = 0;
    for (int t = threadIdx.x; t < static_cast<int>(blockIdx.x); t += kBlock) before += tiles[t].sum;
    (void)block_exclusive<int64_t>(before, &carry, sh);
  }
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int32_t v[kScanItems];
  scan_load(in, n, base, v);
  int64_t sum = 0;
#pragma unroll
  for (int r = 0; r < kScanItems; r++) sum += v[r];
  int64_t tot;
  int64_t run = carry + block_exclusive<int64_t>(sum, &tot, sh);
  int32_t o[kScanItems];
#pragma unroll
  for (int r = 0; r < kScanItems; r++) {
    o[r] = clamp_i32(run);
    run += v[r];
  }
  if (base + kScanItems <= n) {
#pragma unroll
    for (int q = 0; q < kScanItems / 4; q++)
      reinterpret_cast<int4*>(out + base)[q] =
          make_int4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
  } else {
#pragma unroll
    for (int r = 0; r < kScanItems; r++)
      if (base + r < n) out[base + r] = o[r];
  }
  if (blockIdx.x != gridDim.x - 1) return;
  if (threadIdx.x == 0) out[n] = clamp_i32(carry + tot);
  if (!res) return;
  int32_t lo = INT32_MAX, hi = INT32_MIN;
  for (int t = threadIdx.x; t < static_cast<int>(gridDim.x); t += kBlock) {
    lo = min(lo, tiles[t].lo);
    hi = max(hi, tiles[t].hi);
  }
  block_extrema(lo, hi, slo, shi);
  if (threadIdx.x == 0) *res = ScanStats{carry + tot, lo, hi};
}

// ---------------------------------------------------------------------------
// Validation (validate_csr's rules; reason codes name the defect)
// ---------------------------------------------------------------------------
enum : int { kBadCount = 1, kBadPointer = 2, kBadIndex = 3, kSelf = 4, kHalfOrder = 5 };

__global__ void k_validate(int32_t n, const int32_t* __restrict__ nop,
                           const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                           int64_t e, int half, unsigned long long* __restrict__ bad) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t i = static_cast<int32_t>(t);
    const int64_t np = nop[i], kp = ptr[i];
    int reason = 0;
    if (np < 0 || np >= (n > 1 ? n : 1)) reason = kBadCount;
    else if (kp < 0 || kp + np > e) reason = kBadPointer;
    else
      for (int64_t k = 0; k < np; k++) {
        const int32_t j = list[kp + k];
        if (j < 0 || j >= n) { reason = kBadIndex; break; }
        if (j == i) { reason = kSelf; break; }
        if (half && j < i) { reason = kHalfOrder; break; }
      }
    if (reason) atomicMin(bad, static_cast<unsigned long long>(i) * 8ull + reason);
  }
}

// ---------------------------------------------------------------------------
// Row operations
// ---------------------------------------------------------------------------
// Copy row i of (ptr, list) to dst[dptr[i] ..): one wavefront per row.
__global__ __launch_bounds__(kBlock) void k_copy_rows(int32_t n, const int32_t* __restrict__ nop,
                                                      const int32_t* __restrict__ ptr,
                                                      const int32_t* __restrict__ list,
                                                      const int32_t* __restrict__ dptr,
                                                      int32_t* __restrict__ dst) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (kBlock / 64);
  for (int64_t r = blockIdx.x * static_cast<int64_t>(kBlock / 64) + (threadIdx.x >> 6); r < n;
       r += waves) {
    const int32_t m = nop[r];
    const int64_t s = ptr[r], d = dptr[r];
    for (int32_t k = lane; k < m; k += 64) dst[d + k] = list[s + k];
  }
}

// Sort of each segment [start[r], start[r] + len[r]) of src into the same
// positions of dst, ascending, one wavefront per segment. Segments of up to
// 512 elements are sorted in registers by a bitonic network (element e = r*64 +
// lane in register r of that lane; partners closer than 64 are exchanged
// across lanes, farther ones between a lane's own registers), padded with
// INT32_MAX. Longer segments fall back to a rank sort from memory: each
// element goes to the number of smaller elements plus the equal ones before
// it.
//   Exchanges across lanes are DPP moves and permlane swaps; through shuffles
// the sort was bound by the LDS pipe (132 passes for a row of 150: 175 us at
// 119,000 particles, density 1). What bounds it now is VALU issue, so a row of
// 129 to 192 sorts three registers, not four.

// The lanes that keep the smaller value where lanes J apart are exchanged
// within sorted runs of K (64: all one run).
constexpr uint64_t keep_min_lanes(int K, int J, bool descending) {
  uint64_t m = 0;
  for (int l = 0; l < 64; l++) {
    const bool up = ((K < 64 && (l & K)) != 0) == descending;
    if (((l & J) == 0) == up) m |= uint64_t{1} << l;
  }
  return m;
}

template <int CTRL>
__device__ __forceinline__ int32_t dpp_i32(int32_t v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}

// One exchange between the lanes l and l ^ J.
template <int K, int J, bool DESC>
__device__ __forceinline__ void exchange(int32_t& v) {
  int32_t a = v, b;
  if constexpr (J == 16 || J == 32) {
    // The swap leaves each pair's two values in a and b of both its lanes.
    const auto ab = J == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                            : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = static_cast<int32_t>(ab[0]);
    b = static_cast<int32_t>(ab[1]);
  } else if constexpr (J == 8) {
    b = dpp_i32<0x128>(v);  // row_ror:8
  } else if constexpr (J == 4) {
    b = dpp_i32<0x1B>(dpp_i32<0x141>(v));  // row_half_mirror, then each quad reversed
  } else if constexpr (J == 2) {
    b = dpp_i32<0x4E>(v);  // quad_perm [2, 3, 0, 1]
  } else {
    static_assert(J == 1, "lanes up to 32 apart");
    b = dpp_i32<0xB1>(v);  // quad_perm [1, 0, 3, 2]
  }
  const bool low = __builtin_amdgcn_inverse_ballot_w64(keep_min_lanes(K, J, DESC));
  v = low ? min(a, b) : max(a, b);
}

// Runs of K in v, each one bitonic, sorted in alternating directions.
template <int K, int J, bool DESC>
__device__ __forceinline__ void merge_lanes(int32_t& v) {
  exchange<K, J, DESC>(v);
  if constexpr (J > 1) merge_lanes<K, J / 2, DESC>(v);
}

// v[0..R), bitonic, sorted.
template <int R, bool DESC>
__device__ __forceinline__ void merge_regs(int32_t* v) {
  if constexpr (R == 1) {
    merge_lanes<64, 32, DESC>(v[0]);
  } else {
#pragma unroll
    for (int r = 0; r < R / 2; r++) {
      const int32_t lo = min(v[r], v[r + R / 2]), hi = max(v[r], v[r + R / 2]);
      v[r] = DESC ? hi : lo;
      v[r + R / 2] = DESC ? lo : hi;
    }
    merge_regs<R / 2, DESC>(v);
    merge_regs<R / 2, DESC>(v + R / 2);
  }
}

template <int R, bool DESC>
__device__ __forceinline__ void sort_regs(int32_t* v) {
  if constexpr (R == 1) {
    merge_lanes<2, 1, DESC>(v[0]);
    merge_lanes<4, 2, DESC>(v[0]);
    merge_lanes<8, 4, DESC>(v[0]);
    merge_lanes<16, 8, DESC>(v[0]);
    merge_lanes<32, 16, DESC>(v[0]);
    merge_lanes<64, 32, DESC>(v[0]);
  } else if constexpr (R == 3) {
    static_assert(!DESC, "ascending only");
    // As four registers with one of padding after the third: that one stays
    // where it is, and the steps with it vanish.
    sort_regs<2, false>(v);
    sort_regs<1, true>(v + 2);
    const int32_t lo = min(v[1], v[2]);
    v[2] = max(v[1], v[2]);
    v[1] = lo;
    merge_regs<2, false>(v);
    merge_regs<1, false>(v + 2);
  } else {
    sort_regs<R / 2, false>(v);
    sort_regs<R / 2, true>(v + R / 2);
    merge_regs<R, DESC>(v);
  }
}

template <int R>
__device__ __forceinline__ void sort_segment(const int32_t* __restrict__ src,
                                             int32_t* __restrict__ dst, int32_t m, int lane) {
  int32_t v[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int e = r * 64 + lane;
    v[r] = e < m ? src[e] : INT32_MAX;
  }
  sort_regs<R, false>(v);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int e = r * 64 + lane;
    if (e < m) dst[e] = v[r];
  }
}

// Row r is read from src + r * src_stride (src_stride > 0, a slab) or from
// src + start[r], and written to dst + start[r].
__global__ __launch_bounds__(kBlock) void k_row_sort(int32_t n, const int32_t* __restrict__ len,
                                                     const int32_t* __restrict__ start,
                                                     const int32_t* __restrict__ src,
                                                     int64_t src_stride,
                                                     int32_t* __restrict__ dst) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (kBlock / 64);
  for (int64_t r = blockIdx.x * static_cast<int64_t>(kBlock / 64) + (threadIdx.x >> 6); r < n;
       r += waves) {
    const int32_t m = len[r];
    const int64_t d = start[r];
    const int32_t* in = src + (src_stride > 0 ? r * src_stride : d);
    int32_t* o = dst + d;
    if (m <= 1) {
      if (m == 1 && lane == 0) o[0] = in[0];
    } else if (m <= 64) {
      sort_segment<1>(in, o, m, lane);
    } else if (m <= 128) {
      sort_segment<2>(in, o, m, lane);
    } else if (m <= 192) {
      sort_segment<3>(in, o, m, lane);
    } else if (m <= 256) {
      sort_segment<4>(in, o, m, lane);
    } else if (m <= 512) {
      sort_segment<8>(in, o, m, lane);
    } else {
      for (int32_t a = lane; a < m; a += 64) {
        const int32_t x = in[a];
        int32_t rank = 0;
        for (int32_t b = 0; b < m; b++) {
          const int32_t y = in[b];
          rank += (y < x) | ((y == x) & (b < a));
        }
        o[rank] = x;
      }
    }
  }
}

int row_sort(hipStream_t s, int32_t n, const int32_t* len, const int32_t* start,
             const int32_t* src, int32_t* dst, int64_t src_stride = 0) {
  if (n <= 0) return LJGPU_OK;
  k_row_sort<<<grid_for(n, kBlock / 64), kBlock, 0, s>>>(n, len, start, src, src_stride, dst);
  LTRY(hipGetLastError(), "row sort kernel");
  return LJGPU_OK;
}

// Half-to-full expansion.
__global__ void k_count_lower(int32_t n, const int32_t* __restrict__ nop,
                              const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                              int32_t* __restrict__ lower) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t kp = ptr[t];
    for (int32_t k = 0; k < nop[t]; k++) atomicAdd(&lower[list[kp + k]], 1);
  }
}

__global__ void k_add(int32_t n, const int32_t* __restrict__ a, const int32_t* __restrict__ b,
                      int32_t* __restrict__ c) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    c[t] = a[t] + b[t];
}

__global__ void k_fill_expanded(int32_t n, const int32_t* __restrict__ nop,
                                const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                                const int32_t* __restrict__ lower,
                                const int32_t* __restrict__ fptr, int32_t* __restrict__ fill,
                                int32_t* __restrict__ lower_tmp, int32_t* __restrict__ flist) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t r = static_cast<int32_t>(t);
    const int64_t kp = ptr[r];
    const int64_t own = static_cast<int64_t>(fptr[r]) + lower[r];
    for (int32_t k = 0; k < nop[r]; k++) {
      const int32_t j = list[kp + k];
      const int32_t pos = atomicAdd(&fill[j], 1);
      lower_tmp[static_cast<int64_t>(fptr[j]) + pos] = r;
      flist[own + k] = j;
    }
  }
}

// Row-length extrema (int32 atomics on small[0] = min, small[1] = max).
__global__ void k_minmax(int32_t n, const int32_t* __restrict__ a, int32_t* __restrict__ mm) {
  int32_t lo = INT32_MAX, hi = INT32_MIN;
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    lo = min(lo, a[t]);
    hi = max(hi, a[t]);
  }
  for (int d = 32; d > 0; d >>= 1) {
    lo = min(lo, __shfl_xor(lo, d, 64));
    hi = max(hi, __shfl_xor(hi, d, 64));
  }
  // One atomic pair per workgroup: atomics on one address serialise.
  __shared__ int32_t slo[kBlock / 64], shi[kBlock / 64];
  if ((threadIdx.x & 63) == 0) {
    slo[threadIdx.x >> 6] = lo;
    shi[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; w++) {
      lo = min(lo, slo[w]);
      hi = max(hi, shi[w]);
    }
    atomicMin(&mm[0], lo);
    atomicMax(&mm[1], hi);
  }
}

// Partners j > i in each ascending full row.
__global__ void k_upper_counts(int32_t n, const int32_t* __restrict__ nop,
                               const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                               int32_t* __restrict__ out) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t i = static_cast<int32_t>(t);
    const int32_t* row = list + ptr[i];
    int32_t lo = 0, hi = nop[i];
    while (lo < hi) {  // first position with row[pos] > i
      const int32_t mid = (lo + hi) >> 1;
      if (row[mid] <= i) lo = mid + 1;
      else hi = mid;
    }
    out[i] = nop[i] - lo;
  }
}

__global__ void k_ell(int32_t n, int32_t width, const int32_t* __restrict__ nop,
                      const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                      int32_t* __restrict__ ell) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t kp = ptr[t];
    const int32_t m = nop[t];
    for (int32_t k = 0; k < width; k++) ell[t + static_cast<int64_t>(k) * n] = k < m ? list[kp + k] : 0;
  }
}

// Minimum and maximum of a strided coordinate stream (one workgroup).
__global__ __launch_bounds__(kBlock) void k_extrema(int32_t n, const double* __restrict__ a,
                                                    int stride, double* __restrict__ out) {
  __shared__ double smin[kBlock], smax[kBlock];
  double mn = INFINITY, mx = -INFINITY;
  for (int64_t t = threadIdx.x; t < n; t += kBlock) {
    const double v = a[t * stride];
    mn = fmin(mn, v);
    mx = fmax(mx, v);
  }
  smin[threadIdx.x] = mn;
  smax[threadIdx.x] = mx;
  __syncthreads();
  for (int d = kBlock / 2; d > 0; d >>= 1) {
    if (threadIdx.x < d) {
      smin[threadIdx.x] = fmin(smin[threadIdx.x], smin[threadIdx.x + d]);
      smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + d]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = smin[0];
    out[1] = smax[0];
  }
}

// ---------------------------------------------------------------------------
// Cell list and pair passes
// ---------------------------------------------------------------------------
struct GridArgs {
  int nc0, nc1, nc2;
  double o0, o1, o2;
  double w0, w1, w2;
  double box;
};

__device__ __forceinline__ int cell_coord(double x, double origin, double width, int m, double box) {
  x -= origin;
  // The wrapped image's cell (no division for the positions inside: their
  // quotient is below 1).
  if (box > 0.0 && !(x >= 0.0 && x < box)) x -= box * floor(x / box);
  const int v = static_cast<int>(floor(x / width));
  return min(max(v, 0), m - 1);
}

// A particle's cell; sets *outside when a periodic box has a coordinate outside
// [0, box) (the pair search then applies the minimum image in every cell).
struct CellKey {
  PosIn q;
  GridArgs g;
  __device__ __forceinline__ int32_t operator()(int64_t t, int32_t* outside) const {
    const int64_t o = t * q.stride;
    const double x = q.x[o], y = q.y[o], z = q.z[o];
    // Written as negations so that NaN counts as outside.
    if (g.box > 0.0 &&
        !(x >= 0.0 && x < g.box && y >= 0.0 && y < g.box && z >= 0.0 && z < g.box))
      atomicOr(outside, 1);
    const int cx = cell_coord(x, g.o0, g.w0, g.nc0, g.box);
    const int cy = cell_coord(y, g.o1, g.w1, g.nc1, g.box);
    const int cz = cell_coord(z, g.o2, g.w2, g.nc2, g.box);
    return (cz * g.nc1 + cy) * g.nc0 + cx;
  }
};

__global__ void k_cell_assign(int32_t n, CellKey key, int32_t* __restrict__ count,
                              int32_t* __restrict__ slot, int32_t* __restrict__ cell_of,
                              int32_t* __restrict__ outside) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t c = key(t, outside);
    cell_of[t] = c;
    slot[t] = atomicAdd(&count[c], 1);
  }
}

__global__ void k_cell_scatter(int32_t n, PosIn q, const int32_t* __restrict__ cell_of,
                               const int32_t* __restrict__ slot,
                               const int32_t* __restrict__ cell_start,
                               double4* __restrict__ cpos, int32_t* __restrict__ cell_sorted) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t o = t * q.stride;
    const int32_t c = cell_of[t];
    const int64_t d = static_cast<int64_t>(cell_start[c]) + slot[t];
    cpos[d] = make_double4(q.x[o], q.y[o], q.z[o], static_cast<double>(t));
    cell_sorted[d] = c;
  }
}

// Cells (or bins) in a fixed order: the particles of each by ascending index.
// Their atomic slots leave them in arrival order (k_bin_index); each then takes the rank of
// its index among its bin's, which cost a few loads that do not wait for
// each other where a sort by one thread per bin waits for each exchange. Bins of
// more than kCellOrderMax particles keep the arrival order; the callers look
// at the largest bin.
constexpr int32_t kCellOrderMax = 256;
__global__ void k_bin_index(int32_t n, const int32_t* __restrict__ bin_of,
                            const int32_t* __restrict__ slot, const int32_t* __restrict__ start,
                            int32_t* __restrict__ arrival) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    arrival[start[bin_of[t]] + slot[t]] = static_cast<int32_t>(t);
}

// The place of arrival t, whose particle is i.
__device__ __forceinline__ int32_t bin_place(int64_t t, int32_t i, const int32_t* __restrict__ bin_of,
                                             const int32_t* __restrict__ start,
                                             const int32_t* __restrict__ arrival) {
  const int32_t c = bin_of[i];
  const int32_t a = start[c], b = start[c + 1];
  if (b - a > kCellOrderMax) return static_cast<int32_t>(t);
  int32_t r = a;
  for (int32_t u = a; u < b; u++) r += arrival[u] < i ? 1 : 0;
  return r;
}

__global__ void k_order_place(int32_t n, const int32_t* __restrict__ bin_of,
                              const int32_t* __restrict__ start,
                              const int32_t* __restrict__ arrival, int32_t* __restrict__ order) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t i = arrival[t];
    order[bin_place(t, i, bin_of, start, arrival)] = i;
  }
}

__global__ void k_cell_place(int32_t n, PosIn q, const int32_t* __restrict__ cell_of,
                             const int32_t* __restrict__ start,
                             const int32_t* __restrict__ arrival, double4* __restrict__ cpos) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t i = arrival[t];
    const int64_t o = static_cast<int64_t>(i) * q.stride;
    cpos[bin_place(t, i, cell_of, start, arrival)] =
        make_double4(q.x[o], q.y[o], q.z[o], static_cast<double>(i));
  }
}

// What a binned particle leaves at its place: its cell-ordered position and
// cell, or its index.
struct CellPut {
  PosIn q;
  double4* cpos;
  int32_t* cell;
  __device__ __forceinline__ void operator()(int32_t place, int32_t i, int32_t c) const {
    const int64_t o = static_cast<int64_t>(i) * q.stride;
    cpos[place] = make_double4(q.x[o], q.y[o], q.z[o], static_cast<double>(i));
    cell[place] = c;
  }
};
struct OrderPut {
  int32_t* order;
  __device__ __forceinline__ void operator()(int32_t place, int32_t i, int32_t) const {
    order[place] = i;
  }
};

// Spatial tile order: bins of one system (dev_tile_order).
struct OrderGrid {
  double w[3];     // bin widths: x bins, y and z columns
  double box;      // period
  int32_t nc[3];   // x bins, y columns, z columns
  int32_t key0;    // first key of the system
};

struct OrderKey {
  PosIn q;
  OrderGrid one;
  const OrderGrid* grids;
  const int32_t* rep_of;
  __device__ __forceinline__ int32_t operator()(int64_t t, int32_t*) const {
    const OrderGrid g = rep_of ? grids[rep_of[t]] : one;
    const int64_t o = t * q.stride;
    const int cx = cell_coord(q.x[o], 0.0, g.w[0], g.nc[0], g.box);
    const int cy = cell_coord(q.y[o], 0.0, g.w[1], g.nc[1], g.box);
    const int cz = cell_coord(q.z[o], 0.0, g.w[2], g.nc[2], g.box);
    return g.key0 + (cz * g.nc[1] + cy) * g.nc[0] + cx;
  }
};

// Few particles binned by one workgroup, counts and arrival order in LDS: what
// k_cell_assign or k_order_key, a scan, k_bin_index and a placing kernel do for
// more, whose five launches took 16 us and the gaps between them at 2,048
// particles; this one takes 9 to 11 there and 12 to 15 at 4,000, bound by one
// compute unit's latencies, and twice as many particles would cost what the
// launches do. start (null: not wanted) takes the bins' starts, *flag what the
// keys' flag gathered.
constexpr int32_t kBinSmall = 4096;   // particles
constexpr int32_t kBinsSmall = 8192;  // bins
constexpr int kBinThreads = 1024;

template <class Key, class Put>
struct BinJob {
  int32_t n, nbins;
  Key key;
  Put put;
  int32_t* start;
  int32_t* flag;
  ScanStats* res;
};
struct NoBinJob {};
using CellJob = BinJob<CellKey, CellPut>;
using OrderJob = BinJob<OrderKey, OrderPut>;

template <class Key, class Put>
__device__ __forceinline__ void bin_small(const BinJob<Key, Put>& job, int32_t* bin,
                                          uint16_t* arrival) {
  const int32_t n = job.n, nbins = job.nbins;
  const Key& key = job.key;
  const Put& put = job.put;
  int32_t* const start = job.start;
  int32_t* const flag = job.flag;
  ScanStats* const res = job.res;
  __shared__ int32_t sh[kBinThreads / 64], slo[kBinThreads / 64], shi[kBinThreads / 64];
  __shared__ int32_t gathered;
  constexpr int kPer = kBinSmall / kBinThreads;
  const int32_t tid = static_cast<int32_t>(threadIdx.x);
  for (int32_t c = tid; c <= nbins; c += kBinThreads) bin[c] = 0;
  if (tid == 0) gathered = 0;
  __syncthreads();
  int32_t mine[kPer], slot[kPer];
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int32_t t = u * kBinThreads + tid;
    if (t >= n) break;
    mine[u] = key(t, &gathered);
    slot[u] = atomicAdd(&bin[mine[u]], 1);
  }
  __syncthreads();
  const int32_t piece = (nbins + kBinThreads - 1) / kBinThreads;
  const int32_t c0 = min(tid * piece, nbins), c1 = min(c0 + piece, nbins);
  int32_t v = 0, lo = INT32_MAX, hi = INT32_MIN, total;
  for (int32_t c = c0; c < c1; c++) {
    const int32_t x = bin[c];
    v += x;
    lo = min(lo, x);
    hi = max(hi, x);
  }
  int32_t run = block_exclusive<int32_t>(v, &total, sh);
  for (int32_t c = c0; c < c1; c++) {
    const int32_t x = bin[c];
    bin[c] = run;
    if (start) start[c] = run;
    run += x;
  }
  if (tid == 0) {
    bin[nbins] = n;
    if (start) start[nbins] = n;
    if (flag) *flag = gathered;
  }
  block_extrema(lo, hi, slo, shi);
  if (tid == 0) *res = ScanStats{n, lo, hi};
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int32_t t = u * kBinThreads + tid;
    if (t < n) arrival[bin[mine[u]] + slot[u]] = static_cast<uint16_t>(t);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int32_t t = u * kBinThreads + tid;
    if (t >= n) break;
    const int32_t a = bin[mine[u]], b = bin[mine[u] + 1];
    int32_t place = a;
    if (b - a > kCellOrderMax) place += slot[u];
    else
      for (int32_t k = a; k < b; k++) place += arrival[k] < t ? 1 : 0;
    put(place, t, mine[u]);
  }
}

// A second job runs beside the first, on a workgroup of its own.
template <class A, class B>
__global__ __launch_bounds__(kBinThreads) void k_bin_small(A a, B b) {
  __shared__ int32_t bin[kBinsSmall + 1];
  __shared__ uint16_t arrival[kBinSmall];
  if (std::is_same<B, NoBinJob>::value || blockIdx.x == 0) {
    bin_small(a, bin, arrival);
  } else if constexpr (!std::is_same<B, NoBinJob>::value) {
    bin_small(b, bin, arrival);
  }
}

// Row r of a slab (src + r * stride, len[r] entries) to dst + start[r], in
// order. One wavefront copies kSlabRows rows at a time, 128 entries of each
// per pass, every load of a pass issued before its stores (rows are about
// as long as the search sphere holds partners, so one or two passes).
constexpr int kSlabRows = 4;
__global__ __launch_bounds__(kBlock) void k_copy_slab(int32_t n, const int32_t* __restrict__ len,
                                                      const int32_t* __restrict__ start,
                                                      const int32_t* __restrict__ src,
                                                      int64_t stride, int32_t* __restrict__ dst) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (kBlock / 64);
  for (int64_t r0 = (blockIdx.x * static_cast<int64_t>(kBlock / 64) + (threadIdx.x >> 6)) *
                    kSlabRows;
       r0 < n; r0 += waves * kSlabRows) {
    int32_t m[kSlabRows], mx = 0;
#pragma unroll
    for (int k = 0; k < kSlabRows; k++) {
      m[k] = r0 + k < n ? len[r0 + k] : 0;
      mx = max(mx, m[k]);
    }
    for (int32_t e0 = 0; e0 < mx; e0 += 2 * 64) {
      int32_t v[kSlabRows][2];
#pragma unroll
      for (int k = 0; k < kSlabRows; k++) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int32_t e = e0 + u * 64 + lane;
          v[k][u] = e < m[k] ? src[(r0 + k) * stride + e] : 0;
        }
      }
#pragma unroll
      for (int k = 0; k < kSlabRows; k++) {
        if (e0 >= m[k]) continue;
        int32_t* o = dst + start[r0 + k];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int32_t e = e0 + u * 64 + lane;
          if (e < m[k]) o[e] = v[k][u];
        }
      }
    }
  }
}

// The reference's pair predicate (cpu_ref/force_aos.cpp:131-135) with the
// minimum image of the periodic box: every operation rounded separately, in
// the reference's order, (dx*dx + dy*dy) + dz*dz < SL2.
template <bool IMAGE = true>
__device__ __forceinline__ bool within_search(const double4& a, const double4& b, double box,
                                              double half_box, double sl2) {
#pragma clang fp contract(off)
  double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  if (IMAGE && box > 0.0) {
    if (dx > half_box) dx -= box;
    else if (dx < -half_box) dx += box;
    if (dy > half_box) dy -= box;
    else if (dy < -half_box) dy += box;
    if (dz > half_box) dz -= box;
    else if (dz < -half_box) dz += box;
  }
  const double r2 = dx * dx + dy * dy + dz * dz;
  return r2 < sl2;
}

// One thread per particle in cell order (lanes of a wavefront share their
// home cell, so candidate loads are mostly broadcasts), over the cells within
// R of its own (R = 1 for cells at least the search length wide, 2 for cells
// at least half of it; R = 0: one cell holding every particle). MODE 0 counts
// each row's partners into nop[i]; MODE 1 writes them to out[ptr[i] ..) in
// candidate order; MODE 2 does both, writing at most `cap` of them to the
// row's slab out[i * cap ..).
template <int MODE, bool HALF, int R>
__global__ __launch_bounds__(kBlock) void k_pairs(int32_t n, const double4* __restrict__ cpos,
                                                  const int32_t* __restrict__ cell_sorted,
                                                  const int32_t* __restrict__ cell_start,
                                                  GridArgs g, double sl2, int32_t cap,
                                                  int32_t* __restrict__ nop,
                                                  const int32_t* __restrict__ ptr,
                                                  int32_t* __restrict__ out) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (t >= n) return;
  const double4 pi = cpos[t];
  const int32_t i = static_cast<int32_t>(pi.w);
  const int32_t c = cell_sorted[t];
  const int cx = c % g.nc0, cy = (c / g.nc0) % g.nc1, cz = c / (g.nc0 * g.nc1);
  const bool periodic = g.box > 0.0;
  const double half_box = 0.5 * g.box;
  int64_t base = 0;
  if (MODE == 1) base = ptr[i];
  if (MODE == 2) base = static_cast<int64_t>(i) * cap;
  int32_t cnt = 0;
  for (int dz = -R; dz <= R; dz++) {
    int z = cz + dz;
    if (periodic) z = (z + g.nc2) % g.nc2;
    else if (z < 0 || z >= g.nc2) continue;
    for (int dy = -R; dy <= R; dy++) {
      int y = cy + dy;
      if (periodic) y = (y + g.nc1) % g.nc1;
      else if (y < 0 || y >= g.nc1) continue;
      for (int dx = -R; dx <= R; dx++) {
        int x = cx + dx;
        if (periodic) x = (x + g.nc0) % g.nc0;
        else if (x < 0 || x >= g.nc0) continue;
        const int32_t cc = (z * g.nc1 + y) * g.nc0 + x;
        const int32_t u1 = cell_start[cc + 1];
        auto visit = [&](const double4& pj) {
          const int32_t j = static_cast<int32_t>(pj.w);
          if (HALF ? (j <= i) : (j == i)) return;
          if (within_search(pi, pj, g.box, half_box, sl2)) {
            if (MODE == 1 || (MODE == 2 && cnt < cap)) out[base + cnt] = j;
            cnt++;
          }
        };
        int32_t u = cell_start[cc];
        // Four candidates loaded before any is tested, so their loads overlap.
        for (; u + 4 <= u1; u += 4) {
          const double4 a = cpos[u], b = cpos[u + 1], c4 = cpos[u + 2], d = cpos[u + 3];
          visit(a);
          visit(b);
          visit(c4);
          visit(d);
        }
        for (; u < u1; u++) visit(cpos[u]);
      }
    }
  }
  if (MODE != 1) nop[i] = cnt;
}

__device__ __forceinline__ double readlane_d(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// The candidates of one cell (see k_pairs_wave), with the minimum image
// (IMAGE) or without it: a cell whose stencil does not wrap around the box,
// with every position inside [0, box), has no pair that the image would
// shift, so the predicate without it gives the same result. at(f) is the
// place in cpos of candidate f < total.
constexpr int kPairGroup = 5;     // particles of a cell tested together
constexpr int kPairCand = 1024;   // candidates whose places are kept in LDS
// Up to this many cells, four or two wavefronts share a cell's particles: so few
// wavefronts leave the SIMDs idle, and the search takes as long as one cell's
// rounds. List refresh with one force evaluation, one / two / four: 2,048 particles
// (343 cells) 157 / 149 / 147 us, 4,000 (1,000) 175 / 167 / 163, 6,912 (1,728) 179 /
// 174 / 174, 16,384 (4,096) 210 / 206 / 211, 32,000 (8,000) 247 / 246 / 255.
constexpr int64_t kPairCellsFour = 1024;
constexpr int64_t kPairCellsTwo = 4096;

template <int MODE, bool HALF, bool IMAGE, class At>
__device__ __forceinline__ void pairs_cell(int32_t p0, int32_t p1, int32_t per, int32_t step,
                                           int32_t total, At&& at,
                                           const double4* __restrict__ cpos, const GridArgs& g,
                                           double half_box, double sl2, int32_t cap,
                                           int32_t* __restrict__ nop,
                                           const int32_t* __restrict__ ptr,
                                           int32_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  for (int32_t g0 = p0; g0 < p1; g0 += step) {
    const int32_t mg = min(per, p1 - g0);
    double4 pi = make_double4(0.0, 0.0, 0.0, 0.0);
    if (lane < mg) pi = cpos[g0 + lane];
    const int32_t iv = static_cast<int32_t>(pi.w);
    int32_t pv = 0;
    if (MODE == 1) pv = lane < mg ? ptr[iv] : 0;
    // The group's particles as scalars.
    double4 a[kPairGroup];
    int32_t id[kPairGroup], cnt[kPairGroup];
    char* row[kPairGroup];
#pragma unroll
    for (int k = 0; k < kPairGroup; k++) {
      a[k] = make_double4(readlane_d(pi.x, k), readlane_d(pi.y, k), readlane_d(pi.z, k), 0.0);
      id[k] = __builtin_amdgcn_readlane(iv, k);
      cnt[k] = 0;
      if (MODE == 1) row[k] = reinterpret_cast<char*>(out + __builtin_amdgcn_readlane(pv, k));
      if (MODE == 2) row[k] = reinterpret_cast<char*>(out + static_cast<int64_t>(id[k]) * cap);
    }
    for (int32_t f0 = 0; f0 < total; f0 += 64) {
      const bool live = f0 + lane < total;
      // Lanes past the end read the last candidate, moved out of reach.
      double4 pj = cpos[at(min(f0 + lane, total - 1))];
      pj.x = live ? pj.x : INFINITY;
      const int32_t j = static_cast<int32_t>(pj.w);
#pragma unroll
      for (int k = 0; k < kPairGroup; k++) {
        if (k >= mg) break;  // the whole wavefront
        const uint64_t mask =
            __builtin_amdgcn_ballot_w64(within_search<IMAGE>(a[k], pj, g.box, half_box, sl2)) &
            __builtin_amdgcn_ballot_w64(HALF ? j > id[k] : j != id[k]);
        if (MODE != 0) {
          // The place after the row's hits so far and the lower lanes' ones.
          const uint32_t to = __builtin_amdgcn_mbcnt_hi(
              static_cast<uint32_t>(mask >> 32),
              __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), static_cast<uint32_t>(cnt[k])));
          const bool hit = __builtin_amdgcn_inverse_ballot_w64(mask);
          if (hit & (MODE == 1 || to < static_cast<uint32_t>(cap)))
            __builtin_nontemporal_store(j, reinterpret_cast<int32_t*>(row[k] + to * 4u));
        }
        cnt[k] += __popcll(mask);
      }
    }
    if (MODE != 1) {
      int32_t n = 0;
#pragma unroll
      for (int k = 0; k < kPairGroup; k++) n = lane == k ? cnt[k] : n;
      if (lane < mg) nop[iv] = n;
    }
  }
}

// One wavefront per cell (2^split of them in small systems), for cell grids
// with a stencil (R >= 1). The candidates of the (2R+1)^3 cells around it are
// walked as one flattened sequence, 64 per round, and tested against kPairGroup
// of the cell's particles at a time (about four to five of a fine cell's, so
// mostly one group), whose coordinates, counts and row addresses are scalars: a
// pair costs the eight FP64 operations of the predicate and a handful for the
// place of a hit. A round's hits for one particle go to consecutive addresses of its row
// (ballot, then each hit's rank among them), so the stores coalesce; they are
// read much later, hence non-temporal (580 -> 570 us at 1,048,576 particles). The
// runs of the flattened sequence are the x-rows of the stencil, contiguous
// in cell order: (2R+1)^2 rows, each split at most once where it wraps around
// a periodic box (the grid has at least 2R+1 cells per side); their places
// are written out in LDS once per cell (found by a search over the runs
// where a cell has more than kPairCand). Same predicate (within_search, in the same argument
// order), exclusions and MODEs as k_pairs; a row's entries come out in
// candidate order and are sorted afterwards. *outside (from k_cell_assign)
// keeps the minimum image on in every cell. Bound by VALU issue: 572 us at
// 1,048,576 particles (density 0.8, search length 3.3); one particle per
// step with its coordinates fetched from a lane each round took 1007.
template <int MODE, bool HALF, int R>
__global__ __launch_bounds__(kBlock) void k_pairs_wave(int32_t ncell,
                                                       const double4* __restrict__ cpos,
                                                       const int32_t* __restrict__ cell_start,
                                                       GridArgs g, double sl2, int32_t cap,
                                                       int32_t* __restrict__ nop,
                                                       const int32_t* __restrict__ ptr,
                                                       int32_t* __restrict__ out,
                                                       const int32_t* __restrict__ outside,
                                                       int32_t split) {
  __shared__ int32_t cand_lds[kBlock / 64][kPairCand];
  int32_t* cand = cand_lds[threadIdx.x >> 6];
  constexpr int kSpan = 2 * R + 1;
  constexpr int kRuns = 2 * kSpan * kSpan;
  static_assert(kRuns <= 64, "one run per lane");
  const int lane = threadIdx.x & 63;
  const bool periodic = g.box > 0.0;
  const bool all_inside = *outside == 0;
  const double half_box = 0.5 * g.box;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (kBlock / 64);
  // The wavefront's cell and all that follows from it are scalars.
  const int64_t first = blockIdx.x * static_cast<int64_t>(kBlock / 64) +
                        __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / 64);
  for (int64_t w64 = first; w64 < int64_t{ncell} << split; w64 += waves) {
    const int32_t c = static_cast<int32_t>(w64 >> split);
    const int32_t cell0 = cell_start[c], p1 = cell_start[c + 1];
    // This wavefront's groups: `per` particles each, from p0 on.
    const int32_t per = min(kPairGroup, (p1 - cell0 + (1 << split) - 1) >> split);
    const int32_t p0 = cell0 + per * static_cast<int32_t>(w64 & ((1 << split) - 1));
    if (p0 >= p1) continue;  // the whole wavefront
    const int cx = c % g.nc0, cy = (c / g.nc0) % g.nc1, cz = c / (g.nc0 * g.nc1);
    // Lane r < kRuns: run r of the stencil as [rs, rs + rl) in cpos. An x-row's
    // two runs are its parts before and behind the box's face where it
    // wraps, else its halves.
    int32_t rs = 0, rl = 0;
    if (lane < kRuns) {
      const int yz = lane >> 1;
      int z = cz + yz / kSpan - R, y = cy + yz % kSpan - R;
      bool ok = true;
      if (periodic) {
        z += z < 0 ? g.nc2 : z >= g.nc2 ? -g.nc2 : 0;
        y += y < 0 ? g.nc1 : y >= g.nc1 ? -g.nc1 : 0;
      } else {
        ok = z >= 0 && z < g.nc2 && y >= 0 && y < g.nc1;
      }
      const int x0 = cx - R, x1 = cx + R;
      const bool first = (lane & 1) == 0;
      int a = max(x0, 0), b = min(x1, g.nc0 - 1);  // inclusive x range of cells
      if (periodic && x0 < 0) {
        if (!first) a = x0 + g.nc0, b = g.nc0 - 1;
      } else if (periodic && x1 >= g.nc0) {
        if (!first) a = 0, b = x1 - g.nc0;
      } else {
        const int mid = (a + b) >> 1;
        if (first) b = mid;
        else a = mid + 1;
      }
      if (ok && a <= b) {
        const int32_t rowc = (z * g.nc1 + y) * g.nc0;
        rs = cell_start[rowc + a];
        rl = cell_start[rowc + b + 1] - rs;
      }
    }
    int32_t pre = rl;  // inclusive prefix of the run lengths
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t v = __shfl_up(pre, o, 64);
      if (lane >= o) pre += v;
    }
    const int32_t excl = pre - rl;
    const int32_t total = __builtin_amdgcn_readlane(pre, 63);
    const bool wraps = periodic && (!all_inside || cx < R || cx + R >= g.nc0 || cy < R ||
                                    cy + R >= g.nc1 || cz < R || cz + R >= g.nc2);
    auto walk = [&](auto&& at) {
      if (wraps)
        pairs_cell<MODE, HALF, true>(p0, p1, per, per << split, total, at, cpos, g, half_box, sl2,
                                     cap, nop, ptr, out);
      else
        pairs_cell<MODE, HALF, false>(p0, p1, per, per << split, total, at, cpos, g, half_box, sl2,
                                      cap, nop, ptr, out);
    };
    if (total <= kPairCand) {
      for (int32_t k = 0; k < rl; k++) cand[excl + k] = rs + k;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // one wavefront's own
      walk([&](int32_t f) { return cand[f]; });
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
      walk([&](int32_t f) {
        // The run holding f: the number of runs ending at or before f.
        int r = 0;
#pragma unroll
        for (int bit = 32; bit > 0; bit >>= 1) {
          const int t = r + bit;
          const int32_t v = __shfl(pre, min(t, 64) - 1, 64);
          if (t <= kRuns && v <= f) r = t;
        }
        const int rr = min(r, kRuns - 1);
        return __shfl(rs, rr, 64) + (f - __shfl(excl, rr, 64));
      });
    }
  }
}

// ---------------------------------------------------------------------------
// LDS tiles
// ---------------------------------------------------------------------------
constexpr int kTileMaxStage = kTileLdsBudget / 24 + 1; // staged positions that can fit
constexpr int64_t kTileOnePassBytes = int64_t{4} << 30;  // staging slots of the one-pass build
// Wavefronts per tile of the sliced offsets: at most 1024 threads.
constexpr int kSliceWavesMax = 16;
constexpr int kTileRowsMax = 1024;  // rows of a tile
constexpr int kSliceRows = 64;      // rows whose slices are made together
constexpr size_t kTileLdsMax = 64000;  // dynamic LDS of the row-order kernels

// The set of a tile's partners, kept in LDS as a hash table of words: word
// w stands for the 16 slots [16 w, 16 w + 16), its entry holds the key w and
// a 16-bit mask of the slots present (later also the rank of its first
// slot). Partners of a compact tile are runs of consecutive slots, so a tile
// of about 750 partners and 9,000 entries has some 100 to 200 words: nearly
// every entry finds its bit set already, and the words are few enough to be
// ranked by comparing all pairs. A tile that fits the LDS budget has at most
// kTileMaxStage words, below kWordLimit.
constexpr int kWordBits = 12;
constexpr int kWords = 1 << kWordBits;
constexpr int kWordLimit = 3000;
constexpr int kWordLanes = 16;  // lanes that walk one row together
constexpr int kWordBatch = 4;   // entries per lane in flight
constexpr int kSeedRows = 8;    // one row in so many fills the set first
constexpr int kWordPairs = 192;  // more words are ranked by a sort
constexpr int32_t kTileCodeMax = 12160;  // entry codes kept in LDS, 64 KB with the set
static_assert(kTileMaxStage <= kWordLimit, "the word limit must cover every tile that fits");
static_assert(kWordLimit + 1024 < kWords, "probing must always find a free entry");

// The table entries words[0, nw) by ascending key, the others of words[0, p) (p
// the power of two from nw on) as 0xffff behind them.
__device__ __forceinline__ void sort_words(uint16_t* words, int nw, int p, const int32_t* keys) {
  const int tid = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
  for (int t = nw + tid; t < p; t += nt) words[t] = 0xffff;
  __syncthreads();
  auto key = [&](uint16_t x) { return x == 0xffff ? INT32_MAX : keys[x]; };
  for (int k = 2; k <= p; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = tid; t < p / 2; t += nt) {
        const int a = 2 * t - (t & (j - 1)), b = a + j;
        const uint16_t x = words[a], y = words[b];
        if ((key(x) > key(y)) == ((a & k) == 0)) {
          words[a] = y;
          words[b] = x;
        }
      }
      __syncthreads();
    }
}

__device__ __forceinline__ uint32_t word_hash(int32_t w) {
  return (static_cast<uint32_t>(w) * 2654435761u) >> (32 - kWordBits);
}

template <class T>
__device__ __forceinline__ T lds_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The blocks of a tiling: geo (`step` ints per block: first slot, count, and
// in replicas' four the replica), else (null) blocks of T consecutive slots
// of n.
struct TileSpans {
  const int32_t* geo;
  int32_t T, n, step;
};
struct TileSpan {
  int32_t i0, ni, rid;
};
__device__ __forceinline__ TileSpan tile_span(const TileSpans& g, int32_t b) {
  if (g.geo) {
    const int32_t* d = g.geo + static_cast<int64_t>(g.step) * b;
    return TileSpan{d[0], d[1], d[2]};
  }
  return TileSpan{b * g.T, min(g.T, g.n - b * g.T), 0};
}

struct TileGeom {
  int32_t i0, ni, ne, rid;
  int64_t e0;
};

// Where a particle's row starts: in a list by row pointers, or (stride > 0) in
// the pair search's slab.
struct RowSource {
  const int32_t* list;
  const int32_t* ptr;
  int64_t stride;
  __device__ __forceinline__ const int32_t* row(int32_t i) const {
    return list + (stride > 0 ? i * stride : static_cast<int64_t>(ptr[i]));
  }
};

// Block b's entries are [slot_ptr[i0], slot_ptr[i0 + ni]) of the slot-ordered
// rows.
__device__ __forceinline__ TileGeom tile_geom(const TileSpans& spans, int32_t b,
                                              const int32_t* __restrict__ slot_ptr) {
  const TileSpan t = tile_span(spans, b);
  TileGeom g;
  g.i0 = t.i0;
  g.ni = t.ni;
  g.rid = t.rid;
  g.e0 = slot_ptr[g.i0];
  g.ne = slot_ptr[g.i0 + g.ni] - static_cast<int32_t>(g.e0);
  return g;
}

// Add one slot (its word w, hashed to h, and bit) to the set. Returns the
// word's table entry; once more than kWordLimit words are present the tile
// cannot fit, and the search ends at any entry.
__device__ __forceinline__ uint32_t word_add(int32_t w, uint32_t h, uint32_t bit, int32_t* keys,
                                             uint32_t* masks, int32_t* counter) {
  while (lds_load(counter) <= kWordLimit) {
    const int32_t prev = atomicCAS(&keys[h], -1, w);
    if (prev == -1) atomicAdd(counter, 1);
    if (prev == -1 || prev == w) {
      atomicOr(&masks[h], 1u << bit);
      break;
    }
    h = (h + 1) & (kWords - 1);
  }
  return h;
}

// One workgroup per tile. Every partner's slot (and the tile's own slots)
// enters the word set; the words are ranked, each slot's rank being its
// word's base plus the set bits below it, which is the ascending order of
// slots; the staged particles are written in that order and each entry's LDS
// offset 24 * rank in row order. What an entry needs to find its rank (table
// entry and bit, 16 bits) stays in LDS between the two, so the list and
// slot_of are read once; entries beyond `ecap` are looked up again. The words of
// a compact tile are ranked against each other, up to kWordPairs of them; those of
// scattered partners (hardly two to a word) are sorted. List builds by pairs / by
// sort: 135 words 2840 / 2836 us, 184 words 819 / 817, 270 words 3401 / 2634, 540
// words 3458 / 1507, 2145 words 7258 / 1028; compact tiles (100 to 200
// words, on this kernel) 513 / 561 us at 119,164 particles.
//   Sixteen lanes share a row (no search for the row of an entry), four
// entries per lane in flight, with every first probe of a batch issued
// before any is used. soff null: tile b stages at b * kTileMaxStage, and
// nothing more is done for a tile over the LDS budget; else at soff[b].
// COUNT stops after the set: ns_out[b] distinct slots. stats[b]: distinct
// slots (-1: too many words), LDS bytes, longest row (k_tile_stats reduces
// them: an atomic per tile on one address costs more than the tile).
template <bool COUNT>
__global__ __launch_bounds__(1024) void k_tile_fill(
    TileSpans spans, int32_t nblocks, const int32_t* __restrict__ member,
    const int32_t* __restrict__ slot_of, const int32_t* __restrict__ slot_ptr,
    RowSource rows,
    const int32_t* __restrict__ soff, int32_t ecap, int32_t* __restrict__ ns_out,
    int32_t* __restrict__ desc, int32_t* __restrict__ stage, int32_t* __restrict__ stage_slot,
    uint16_t* __restrict__ local, int4* __restrict__ stats) {
  __shared__ int32_t keys[kWords];
  __shared__ uint32_t masks[kWords];  // slots present, then also the base rank << 16
  __shared__ uint16_t words[kWords];  // table entries in use
  __shared__ int32_t counter, nwords, total, longest;
  __shared__ int32_t sh[16];
  extern __shared__ uint16_t code[];  // ecap: table entry << 4 | bit of each entry
  const int nt = static_cast<int>(blockDim.x), tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kWordLanes - 1), group = tid / kWordLanes, groups = nt / kWordLanes;
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const TileGeom g = tile_geom(spans, b, slot_ptr);
    for (int t = tid; t < kWords; t += nt) {
      keys[t] = -1;
      masks[t] = 0;
    }
    if (tid == 0) counter = nwords = total = longest = 0;
    __syncthreads();
    for (int t = tid; t < g.ni; t += nt) {
      const int32_t key = g.i0 + t;
      (void)word_add(key >> 4, word_hash(key >> 4), key & 15, keys, masks, &counter);
    }
    // One row in kSeedRows first, spread over all the groups: it brings in most
    // of the words and bits, so that the other rows nearly always find theirs
    // (all rows at once would all meet the empty table).
    auto walk = [&](int r, int32_t k0, int32_t step) {
      const int32_t a = slot_ptr[g.i0 + r];
      const int32_t m = slot_ptr[g.i0 + r + 1] - a;
      const int32_t* src = rows.row(member ? member[g.i0 + r] : g.i0 + r);
      const int32_t eoff = a - static_cast<int32_t>(g.e0);
      if (k0 == 0) atomicMax(&longest, m);
      for (; k0 < m; k0 += step * kWordBatch) {
        int32_t key[kWordBatch], w0[kWordBatch];
        uint32_t h[kWordBatch], m0[kWordBatch];
#pragma unroll
        for (int u = 0; u < kWordBatch; u++) {
          const int32_t k = k0 + u * step;
          key[u] = k < m ? src[k] : -1;
        }
        if (slot_of) {
#pragma unroll
          for (int u = 0; u < kWordBatch; u++)
            if (key[u] >= 0) key[u] = slot_of[key[u]];
        }
#pragma unroll
        for (int u = 0; u < kWordBatch; u++) {
          h[u] = word_hash(key[u] >> 4);
          w0[u] = lds_load(&keys[h[u]]);
          m0[u] = lds_load(&masks[h[u]]);
        }
#pragma unroll
        for (int u = 0; u < kWordBatch; u++) {
          if (key[u] < 0) continue;
          const uint32_t bit = key[u] & 15;
          if (w0[u] != key[u] >> 4)
            h[u] = word_add(key[u] >> 4, h[u], bit, keys, masks, &counter);
          else if (!((m0[u] >> bit) & 1))
            atomicOr(&masks[h[u]], 1u << bit);
          const int32_t e = eoff + k0 + u * step;
          if (!COUNT && e < ecap) code[e] = static_cast<uint16_t>(h[u] << 4 | bit);
        }
      }
    };
    const int seeds = (g.ni + kSeedRows - 1) / kSeedRows;
    const int share = max(1, groups / seeds);  // groups to a seed row
    for (int q = group; q < seeds * share; q += groups)
      walk(q / share * kSeedRows, (q % share) * kWordLanes + lane, share * kWordLanes);
    __syncthreads();
    for (int q = group; q < g.ni - seeds; q += groups)
      walk(q / (kSeedRows - 1) * kSeedRows + q % (kSeedRows - 1) + 1, lane, kWordLanes);
    __syncthreads();
    const bool full = counter > kWordLimit;
    // The table entries in use, in any order, and the distinct slots.
    if (!full) {
      int32_t cnt = 0;
      for (int t = tid; t < kWords; t += nt) {
        if (keys[t] == -1) continue;
        words[atomicAdd(&nwords, 1)] = static_cast<uint16_t>(t);
        cnt += __popc(masks[t]);
      }
      if (cnt) atomicAdd(&total, cnt);
    }
    __syncthreads();
    const int32_t nw = nwords;
    const int32_t ns = full ? -1 : total;
    const int64_t bytes = full ? INT32_MAX : tile_lds_bytes(ns, g.ne);
    const bool over = bytes > kTileLdsBudget;
    if (tid == 0) {
      if (COUNT) ns_out[b] = full ? 0 : ns;
      stats[b] = make_int4(ns, static_cast<int32_t>(std::min<int64_t>(bytes, INT32_MAX)), longest, 0);
    }
    if (COUNT || (over && !soff)) {  // uniform over the workgroup
      __syncthreads();
      continue;
    }
    // Base rank of each word: the slots of all smaller words, a scan over the
    // sorted words or eight lanes to a word.
    if (nw > kWordPairs) {
      sort_words(words, nw, 1 << (32 - __clz(nw - 1)), keys);
      const int piece = (nw + nt - 1) / nt;
      const int t0 = min(tid * piece, nw), t1 = min(t0 + piece, nw);
      int32_t n = 0, all;
      for (int t = t0; t < t1; t++) n += __popc(masks[words[t]]);
      int32_t base = block_exclusive<int32_t>(n, &all, sh);
      for (int t = t0; t < t1; t++) {
        const int x = words[t];
        const uint32_t v = masks[x];
        masks[x] = v | static_cast<uint32_t>(base) << 16;
        base += __popc(v);
      }
    } else for (int t0 = 0; t0 < nw; t0 += nt / 8) {
      const int t = t0 + tid / 8;
      int32_t base = 0;
      if (t < nw) {
        const int32_t w = keys[words[t]];
        for (int v = tid & 7; v < nw; v += 8) {
          const int x = words[v];
          base += keys[x] < w ? __popc(masks[x] & 0xffffu) : 0;
        }
      }
#pragma unroll
      for (int d = 4; d > 0; d >>= 1) base += __shfl_xor(base, d, 8);
      // Only the low halves are read above, so the base can go in at once.
      if (t < nw && (tid & 7) == 0) atomicOr(&masks[words[t]], static_cast<uint32_t>(base) << 16);
    }
    __syncthreads();
    const int64_t s0 = soff ? soff[b] : static_cast<int64_t>(b) * kTileMaxStage;
    // Staged particles in slot order: stage holds the particles, stage_slot
    // (spatial order only) their slots.
    for (int t = tid; t < nw * 16; t += nt) {
      const int x = words[t >> 4];
      const uint32_t v = masks[x], bit = t & 15;
      if (!((v >> bit) & 1)) continue;
      const int32_t key = keys[x] << 4 | bit;
      const int64_t d = s0 + (v >> 16) + __popc(v & ((1u << bit) - 1));
      stage[d] = member ? member[key] : key;
      if (stage_slot) stage_slot[d] = key;
    }
    if (tid == 0) {
      int32_t* d = desc + static_cast<int64_t>(b) * 8;
      const int32_t mid = g.i0 + g.ni / 2;
      d[0] = g.i0;
      d[1] = g.ni;
      d[2] = static_cast<int32_t>(s0);
      d[3] = ns;
      d[4] = static_cast<int32_t>(g.e0);
      d[5] = g.ne;
      d[6] = g.rid;
      d[7] = member ? member[mid] : mid;  // middle particle: the periodic unwrap's reference
    }
    const int32_t ncode = min(g.ne, ecap);
    for (int32_t e = tid; e < ncode; e += nt) {
      const uint32_t v = masks[code[e] >> 4], bit = code[e] & 15;
      local[g.e0 + e] = static_cast<uint16_t>(((v >> 16) + __popc(v & ((1u << bit) - 1))) * 24);
    }
    if (g.ne > ecap) {
      for (int r = group; r < g.ni; r += groups) {
        const int32_t a = slot_ptr[g.i0 + r];
        const int32_t m = slot_ptr[g.i0 + r + 1] - a;
        const int32_t* src = rows.row(member ? member[g.i0 + r] : g.i0 + r);
        const int32_t eoff = a - static_cast<int32_t>(g.e0);
        for (int32_t k = lane; k < m; k += kWordLanes) {
          if (eoff + k < ecap) continue;
          int32_t key = src[k];
          if (slot_of) key = slot_of[key];
          uint32_t h = word_hash(key >> 4);
          while (keys[h] != key >> 4) h = (h + 1) & (kWords - 1);
          const uint32_t v = masks[h], bit = key & 15;
          local[a + k] = static_cast<uint16_t>(((v >> 16) + __popc(v & ((1u << bit) - 1))) * 24);
        }
      }
    }
    __syncthreads();
  }
}

// The tiles' stats in one: out[0] a tile over the LDS budget, [1] most staged,
// [2] most LDS bytes, [3] longest row, [4] tiles with too many pages, [6..7]
// the total staged (64 bits), as far as counted. One workgroup.
__global__ __launch_bounds__(1024) void k_tile_stats(int32_t nblocks, const int4* __restrict__ stats,
                                                     uint16_t* __restrict__ pad,
                                                     int32_t* __restrict__ out) {
  // The offsets' padding, too (the force kernels read past the last row).
  for (int t = threadIdx.x; pad && t < kTileLocalPad; t += blockDim.x) pad[t] = 0;
  __shared__ int32_t mx[5];
  __shared__ unsigned long long sum;
  if (threadIdx.x < 5) mx[threadIdx.x] = threadIdx.x == 1 ? -1 : 0;
  if (threadIdx.x == 5) sum = 0;
  __syncthreads();
  int32_t v[5] = {0, -1, 0, 0, 0};
  unsigned long long n = 0;
  for (int32_t b = threadIdx.x; b < nblocks; b += blockDim.x) {
    const int4 t = stats[b];
    v[0] |= t.y > kTileLdsBudget;
    v[1] = max(v[1], t.x);
    v[2] = max(v[2], t.y);
    v[3] = max(v[3], t.z);
    v[4] += t.w;
    n += max(t.x, 0);
  }
  for (int d = 32; d > 0; d >>= 1) {
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = max(v[k], __shfl_xor(v[k], d, 64));
    v[4] += __shfl_xor(v[4], d, 64);
    n += __shfl_xor(n, d, 64);
  }
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < 4; k++) atomicMax(&mx[k], v[k]);
    atomicAdd(&mx[4], v[4]);
    atomicAdd(&sum, n);
  }
  __syncthreads();
  if (threadIdx.x < 5) out[threadIdx.x] = mx[threadIdx.x];
  if (threadIdx.x == 5) *reinterpret_cast<unsigned long long*>(out + 6) = sum;
}

// The same tiles as k_tile_fill<false>, for tiles whose partners lie in few
// pages of 2^pshift consecutive slots (any spatially ordered list: a column's
// slots are consecutive, and a tile meets about 25 columns). The set is
// then a byte per slot of the pages in use, filled by plain stores, with no atomics
// and no search:
//   1. every entry marks its page in a directory of all pages;
//   2. a scan numbers the marked pages in ascending order;
//   3. every entry marks its slot in its page's bytes;
//   4. a scan over the bytes, 16 at a time, leaves a 16-bit mask and a base rank
//      for each sixteen slots, from which every entry takes its rank.
// A row's entries stay in registers (kPageLanes lanes to a row, up to
// kPageKeys of them each; more are loaded again). What a tile takes is mostly
// the latency of its dependent loads and barriers, so the workgroup is sized
// for three of them to a CU (80 VGPRs; at four the 24 spilled registers cost
// more: 87 against 64 us at 119,000 particles, 521 against 364 us at a
// million). The hashed set of k_tile_fill takes 119 and 742 us there. A tile with more pages
// than fit kPageBytes says so in stats[b].w, and the caller uses k_tile_fill.
//   With slices.out the wavefront slices of the rows as they stand (see
// k_tile_slices) leave from LDS as well, and local may be null.
struct SliceDev {
  uint16_t* out;            // null: no slices
  const int32_t* wave_off;
  int32_t lanes, wpb, stride, pad;
};
constexpr int kPageLanes = 8;
constexpr int kPageKeys = 16;
constexpr int kPageBytes = 24576;
constexpr int kPageDir = 32768;  // most pages of a list
static_assert(kPageBytes / 128 < 255, "a page number fits a byte");

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(6))) void k_tile_pages(
    TileSpans spans, int32_t nblocks, const int32_t* __restrict__ member,
    const int32_t* __restrict__ slot_of, const int32_t* __restrict__ slot_ptr,
    RowSource rows, int32_t pshift, int32_t npages, SliceDev slices,
    int32_t* __restrict__ desc, int32_t* __restrict__ stage, int32_t* __restrict__ stage_slot, uint16_t* __restrict__ local, int4* __restrict__ stats) {
  extern __shared__ uint32_t page_lds[];
  __shared__ uint32_t table[kPageBytes / 16];  // slots present, base rank << 16
  __shared__ uint32_t used[kPageBytes / 4];    // a byte per slot of the pages in use
  __shared__ int32_t page_of[256];
  __shared__ int32_t sh[16];
  __shared__ int32_t longest;
  uint8_t* dir = reinterpret_cast<uint8_t*>(page_lds);  // npages, a multiple of 4 bytes
  uint8_t* mark = reinterpret_cast<uint8_t*>(used);
  const int nt = static_cast<int>(blockDim.x), tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kPageLanes - 1), group = tid / kPageLanes, groups = nt / kPageLanes;
  const int32_t low = (1 << pshift) - 1;
  const int32_t chunk = ((npages + nt - 1) / nt + 3) / 4;  // directory words per thread
  if (slices.out && blockIdx.x == 0)
    for (int t = tid; t < slices.pad; t += nt)
      slices.out[slices.wave_off[static_cast<int64_t>(nblocks) * slices.wpb] + t] = 0;
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const TileGeom g = tile_geom(spans, b, slot_ptr);
    for (int t = tid; t < (npages + 3) / 4; t += nt) page_lds[t] = 0;
    if (tid == 0) longest = 0;
    // The group's first row, in registers; places past its end hold the tile's
    // first slot, which belongs to the set anyway.
    int32_t key[kPageKeys];
    int32_t mine = 0;  // the row's entries from this lane's first on
    const int32_t* row = rows.list;
    int32_t a0 = 0;
    if (group < g.ni) {
      a0 = slot_ptr[g.i0 + group];
      mine = slot_ptr[g.i0 + group + 1] - a0 - lane;
      row = rows.row(member ? member[g.i0 + group] : g.i0 + group) + lane;
    }
#pragma unroll
    for (int u = 0; u < kPageKeys; u++) {
      key[u] = slot_of ? -1 : g.i0;
      if (u * kPageLanes < mine) key[u] = row[u * kPageLanes];
    }
    if (slot_of) {
#pragma unroll
      for (int u = 0; u < kPageKeys; u++)
        key[u] = key[u] >= 0 ? slot_of[static_cast<uint32_t>(key[u])] : g.i0;
    }
    // f(slot, row, its start, place) of every other entry of the block.
    auto others = [&](auto&& f) {
      for (int r = group; r < g.ni; r += groups) {
        const int32_t a = slot_ptr[g.i0 + r];
        const int32_t m = slot_ptr[g.i0 + r + 1] - a;
        const int32_t* src = rows.row(member ? member[g.i0 + r] : g.i0 + r);
        for (int32_t k = lane + (r == group ? kPageKeys * kPageLanes : 0); k < m; k += kPageLanes) {
          const int32_t j = src[k];
          f(slot_of ? slot_of[j] : j, r, a, k);
        }
        if (lane == 0) atomicMax(&longest, m);
      }
    };
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPageKeys; u++) dir[key[u] >> pshift] = 1;
    others([&](int32_t s, int, int32_t, int32_t) { dir[s >> pshift] = 1; });
    for (int t = tid; t < g.ni; t += nt) dir[(g.i0 + t) >> pshift] = 1;
    __syncthreads();
    int32_t pages = 0;
    {
      int32_t c = 0;
      for (int w = tid * chunk; w < min((tid + 1) * chunk, (npages + 3) / 4); w++)
        c += __popc(page_lds[w]);
      int32_t p = block_exclusive<int32_t>(c, &pages, sh);
      if ((pages << pshift) <= kPageBytes && c > 0)
        for (int t = tid * chunk * 4; t < min((tid + 1) * chunk * 4, npages); t++)
          if (dir[t]) {
            page_of[p] = t;
            dir[t] = static_cast<uint8_t>(p++);
          }
    }
    if ((pages << pshift) > kPageBytes) {  // uniform over the workgroup
      if (tid == 0) stats[b] = make_int4(0, 0, 0, 1);
      __syncthreads();
      continue;
    }
    const int nwords = (pages << pshift) / 16;
    for (int t = tid; t < nwords * 4; t += nt) used[t] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPageKeys; u++) {
      key[u] = dir[key[u] >> pshift] << pshift | (key[u] & low);  // its byte from here on
      mark[key[u]] = 1;
    }
    others([&](int32_t s, int, int32_t, int32_t) { mark[dir[s >> pshift] << pshift | (s & low)] = 1; });
    for (int t = tid; t < g.ni; t += nt) {
      const int32_t s = g.i0 + t;
      mark[dir[s >> pshift] << pshift | (s & low)] = 1;
    }
    __syncthreads();
    int32_t ns = 0;
    for (int w0 = 0; w0 < nwords; w0 += nt) {
      const int w = w0 + tid;
      uint32_t mask = 0;
      if (w < nwords) {
#pragma unroll
        for (int q = 0; q < 4; q++)  // four bytes of 0 or 1 to four bits
          mask |= ((used[4 * w + q] * 0x01020408u) >> 24 & 15u) << (4 * q);
      }
      int32_t n = 0;
      const int32_t base = ns + block_exclusive<int32_t>(__popc(mask), &n, sh);
      if (w < nwords) table[w] = mask | static_cast<uint32_t>(base) << 16;
      ns += n;
    }
    __syncthreads();
    const int64_t bytes = tile_lds_bytes(ns, g.ne);
    const bool over = bytes > kTileLdsBudget;
    if (tid == 0)
      stats[b] = make_int4(ns, static_cast<int32_t>(std::min<int64_t>(bytes, INT32_MAX)), longest, 0);
    if (over) {  // uniform; the caller retries smaller
      __syncthreads();
      continue;
    }
    const int64_t s0 = static_cast<int64_t>(b) * kTileMaxStage;
    for (int t = tid; t < nwords * 16; t += nt) {
      const uint32_t v = table[t >> 4], bit = t & 15;
      if (!((v >> bit) & 1)) continue;
      const int32_t slot = page_of[t >> pshift] << pshift | (t & low);
      const int64_t d = s0 + (v >> 16) + __popc(v & ((1u << bit) - 1));
      stage[d] = member ? member[slot] : slot;
      if (stage_slot) stage_slot[d] = slot;
    }
    if (tid == 0) {
      int32_t* d = desc + static_cast<int64_t>(b) * 8;
      const int32_t mid = g.i0 + g.ni / 2;
      d[0] = g.i0;
      d[1] = g.ni;
      d[2] = static_cast<int32_t>(s0);
      d[3] = ns;
      d[4] = static_cast<int32_t>(g.e0);
      d[5] = g.ne;
      d[6] = g.rid;
      d[7] = member ? member[mid] : mid;  // middle particle: the periodic unwrap's reference
    }
    auto offset = [&](int32_t at) {
      const uint32_t v = table[at >> 4];
      return static_cast<uint16_t>(((v >> 16) + __popc(v & ((1u << (at & 15)) - 1))) * 24);
    };
    // The rows in LDS too, where the directory's bytes were, if their slices
    // are made here.
    uint16_t* lds_rows = reinterpret_cast<uint16_t*>(used);
    auto put = [&](uint16_t v, int r, int32_t a, int32_t k) {
      if (local) local[a + k] = v;
      if (slices.out) lds_rows[r * slices.stride + k] = v;
    };
#pragma unroll
    for (int u = 0; u < kPageKeys; u++) {
      const uint16_t v = offset(key[u]);
      if (u * kPageLanes < mine) put(v, group, a0, lane + u * kPageLanes);
    }
    others([&](int32_t s, int r, int32_t a, int32_t k) {
      put(offset(dir[s >> pshift] << pshift | (s & low)), r, a, k);
    });
    __syncthreads();
    if (slices.out) {
      const int lsh = 31 - __clz(slices.lanes);
      const int rpw = 64 >> lsh;  // rows per wavefront
      for (int w = tid / 64; w < slices.wpb; w += nt / 64) {
        const int32_t* wo = slices.wave_off + static_cast<int64_t>(b) * slices.wpb + w;
        const int32_t p0 = wo[0], n = wo[1] - wo[0];
        const int r = w * rpw + ((tid & 63) >> lsh);
        const int32_t m = r < g.ni ? slot_ptr[g.i0 + r + 1] - slot_ptr[g.i0 + r] : 0;
        const uint16_t* src = lds_rows + (r < g.ni ? r : 0) * slices.stride;
        int k = tid & (slices.lanes - 1);
#pragma unroll 4
        for (int32_t p = tid & 63; p < n; p += 64, k += slices.lanes)
          slices.out[p0 + p] = k < m ? src[k] : uint16_t{0};
      }
      __syncthreads();
    }
  }
}

// The bank-class order (bank_class_order) of rows in cutoff classes, for the
// layouts that read `local` itself. One wavefront per tile, one row per
// lane, each lane's buffers in LDS.
constexpr int kBankBlock = 64;
__global__ __launch_bounds__(kBankBlock) void k_bank_order(const int32_t* __restrict__ desc,
                                                           int32_t nblocks,
                                                           const int32_t* __restrict__ slot_ptr,
                                                           const int32_t* __restrict__ inner,
                                                           uint16_t* __restrict__ local) {
  __shared__ uint16_t buf[kBankBlock][kBankRowMax];
  __shared__ uint16_t cnt[kBankBlock][kBankClasses];
  __shared__ uint16_t nxt[kBankBlock][kBankClasses];
  const int t = static_cast<int>(threadIdx.x);
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const int32_t i0 = desc[8 * static_cast<int64_t>(b)], ni = desc[8 * static_cast<int64_t>(b) + 1];
    for (int32_t r = t; r < ni; r += kBankBlock) {
      const int32_t a = slot_ptr[i0 + r];
      const int m = slot_ptr[i0 + r + 1] - a;
      const int nin = inner ? inner[i0 + r] : m;
      uint16_t* row = local + a;
      bank_class_order(row, nin, r, 0, buf[t], cnt[t], nxt[t]);
      bank_class_order(row + nin, m - nin, r, nin, buf[t], cnt[t], nxt[t]);
    }
  }
}

// Slice lengths: per (block, wavefront slot), 64 * unroll offsets for each
// batch its longest row needs (0 for slots past the block's rows).
__global__ void k_wave_slices(TileSpans spans, int32_t nblocks, int32_t wpb,
                              const int32_t* __restrict__ slot_ptr, int32_t lanes, int32_t unroll,
                              int32_t* __restrict__ len) {
  const int64_t id = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (id >= static_cast<int64_t>(nblocks) * wpb) return;
  const int32_t b = static_cast<int32_t>(id / wpb), w = static_cast<int32_t>(id % wpb);
  const TileSpan g = tile_span(spans, b);
  const int32_t i0 = g.i0, ni = g.ni;
  const int32_t rpw = 64 / lanes, kb = lanes * unroll;
  int32_t batches = 0;
  for (int32_t r = w * rpw; r < min(ni, (w + 1) * rpw); r++) {
    const int32_t np = slot_ptr[i0 + r + 1] - slot_ptr[i0 + r];
    batches = max(batches, (np + kb - 1) / kb);
  }
  len[id] = batches * 64 * unroll;
}

constexpr int kRowLanes = 8;  // lanes that walk one row together
constexpr int kRowBatch = 3;  // entries per lane in flight

// LDS of one wavefront's order_part: class counts, a byte each, four classes to
// a word, a column of words per lane; and the free places of its rows.
struct OrderLds {
  uint32_t cnt[kBankClasses / 4][64];
  uint8_t hole[64 / kRowLanes][kBankRowMax];
};
static_assert(kBankRowMax / kRowLanes * (kRowLanes - 1) <= 255 && kBankRowMax / kRowLanes <= 128,
              "numbers within a class fit a byte");
static_assert(kBankClasses == 4 * kRowLanes, "one lane per word of counts, four steps a level");

// The places of one part of each row (its inner entries, or the others),
// kRowLanes lanes to a row, a wavefront's rows together: n ranks from[0],
// from[step], ... (of at most nmax in any of its rows) take the places
// to[0 .. n), the same memory, whose first one has target class `phase`. Each
// lane counts its own entries by class; a sum over the row's lanes leaves the
// number of each lane's first one, from which its entries take their numbers
// q, and the q-th entry of a class takes the q-th place that has the class as
// its target. The entries beyond those fill, in order, the places whose class
// ran out. One lane per row and the seven other wavefronts idle took 182 us with the rest of k_tile_slices at
// 119,000 particles (density 1), 35 at 2,000; this way 122 and 25.
__device__ __forceinline__ void order_part(const uint16_t* from, int step, uint16_t* to, int phase,
                                           int n, int nmax, OrderLds& lds) {
  constexpr int kSteps = kBankRowMax / kRowLanes, kGroup = 8;
  const int wl = static_cast<int>(threadIdx.x) & 63;
  int lane = wl & (kRowLanes - 1);
  const int seg = wl - lane;
  asm volatile("" : "+v"(lane));  // places and comparisons again, not held in registers
  const uint32_t below = (1u << lane) - 1;
  uint32_t* cnt = &lds.cnt[0][wl];
  uint8_t* holes = lds.hole[seg / kRowLanes];
  // This row's lanes for which `c` holds.
  auto row_bits = [&](bool c) {
    const uint64_t v = __ballot(c);
    const uint32_t h = wl < 32 ? static_cast<uint32_t>(v) : static_cast<uint32_t>(v >> 32);
    return h >> (seg & 31) & ((1u << kRowLanes) - 1);
  };
#pragma unroll
  for (int w = 0; w < kBankClasses / 4; w++) cnt[w * 64] = 0;
  uint32_t entry[kSteps / 2];  // two ranks each
#pragma unroll
  for (int g = 0; g < kSteps; g += kGroup) {
    if (g * kRowLanes >= nmax) break;  // the whole wavefront
#pragma unroll
    for (int u = g; u < g + kGroup; u++) {
      const int t = u * kRowLanes + lane;
      const uint32_t x = from[(t < n ? t : 0) * step];
      entry[u / 2] = u % 2 ? entry[u / 2] | x << 16 : x;
    }
#pragma unroll
    for (int u = g; u < g + kGroup; u++) {
      const uint32_t x = entry[u / 2] >> 16 * (u % 2) & 0xffffu;
      if (u * kRowLanes + lane < n) atomicAdd(&cnt[(x >> 2 & 7) * 64], 1u << (x & 3) * 8);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wavefront's own, in order
  // Lane w sums word w of the row's counts: each lane's first number. A list
  // may repeat a partner, so a class can hold all of a row's 256 entries, one
  // more than a byte: counts of the first seven lanes stop at 127 in the total,
  // of which only whether it exceeds a level (at most 7) matters.
  uint32_t total = 0;
  {
    uint32_t* word = &lds.cnt[lane][seg];
    uint32_t v[kRowLanes];
#pragma unroll
    for (int j = 0; j < kRowLanes; j++) v[j] = word[j];
#pragma unroll
    for (int j = 0; j < kRowLanes; j++) {
      word[j] = total;
      if (j == kRowLanes - 1)
        total = (total | (total >> 7 & 0x01010101u) * 0x7fu) & 0x7f7f7f7fu;
      total += v[j];
    }
  }
  // Place k has the class (phase + k) % 32, and it is the (k / 32)-th of it.
  uint32_t of_class[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int c = (phase + j * kRowLanes + lane) & (kBankClasses - 1);
    of_class[j] = __shfl(total, seg + c / 4, 64) >> (c & 3) * 8 & 255u;
  }
  int free = 0;
  for (int level = 0; level * kBankClasses < nmax; level++) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int k = level * kBankClasses + j * kRowLanes + lane;
      const bool hole = k < n && level >= static_cast<int>(of_class[j]);
      const uint32_t bits = row_bits(hole);
      if (hole) holes[free + __popc(bits & below)] = static_cast<uint8_t>(k);
      free += __popc(bits);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int left = 0;
  asm volatile("" : "+v"(n), "+v"(lane));
#pragma unroll
  for (int g = 0; g < kSteps; g += kGroup) {
    if (g * kRowLanes >= nmax) break;
    uint32_t q[kGroup];
#pragma unroll
    for (int u = g; u < g + kGroup; u++) {
      const uint32_t x = entry[u / 2] >> 16 * (u % 2) & 0xffffu;
      q[u - g] = atomicAdd(&cnt[(x >> 2 & 7) * 64],
                           u * kRowLanes + lane < n ? 1u << (x & 3) * 8 : 0u) >> (x & 3) * 8 & 255u;
    }
#pragma unroll
    for (int u = g; u < g + kGroup; u++) {
      const uint32_t x = entry[u / 2] >> 16 * (u % 2) & 0xffffu;
      int d = static_cast<int>(((x - phase) & (kBankClasses - 1)) + kBankClasses * q[u - g]);
      const bool valid = u * kRowLanes + lane < n, over = valid && d >= n;
      const uint32_t bits = row_bits(over);
      if (over) d = holes[left + __popc(bits & below)];
      left += __popc(bits);
      if (valid) to[d] = static_cast<uint16_t>(x);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The wavefront's largest v.
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

struct CutDev {
  PosIn q;
  const int32_t* stage;
  const int32_t* member;
  double box;
  const double* rep_box;
  double cl2;
};

// The slices of one block per workgroup, rows in groups of `grows` (at most
// kSliceRows, a multiple of a wavefront's rows): slice position p of
// wavefront w (batch j = p / (64 unroll), slot u, lane l) holds place k = j
// * lanes * unroll + u * lanes + l % lanes of the block's row w * (64 /
// lanes) + l / lanes as `scale` times its rank, or 0 past the row's end
// (padding).
//   CUT first puts the rows in cutoff classes (cut_partition over cut_inner):
// inner entries first, the others behind them, both in list order, in
// `local` as well; inner[s] receives the inner count of slot s's row. The
// partners' positions are staged in LDS (POS_LDS) or, where they do not fit,
// read from memory.
//   ORDER gives the places of each class out by order_part, so that the 32
// lanes that read LDS together mostly read different banks (the row's phase
// is its first lane's place among them), on ranks in LDS, rows `stride` (an odd
// number of dwords) apart, inner entries forward from the row's start, the
// others backward from its end. At density 1 a half-wavefront's read then takes 2.3 passes over the
// banks (modelled on the tiles of 119,164 particles) against 2.6 in the
// bank-class order: FP64 forces 2.4 %, mixed 4 % faster.
//   Rows of more than kBankRowMax entries, and all rows without ORDER, keep
// the order of `local`. Three workgroups fit a CU's LDS, hence the 80 VGPRs
// (a dozen spilled in the CUT form; at 167 registers one workgroup fits).
constexpr int kSliceThreads = 512;
static_assert(kSliceThreads == kSliceRows * kRowLanes, "order_part takes a group's rows at once");

template <bool CUT, bool POS_LDS, bool ORDER>
__global__ __launch_bounds__(kSliceThreads) __attribute__((amdgpu_waves_per_eu(6))) void k_tile_slices(
    const int32_t* __restrict__ desc, int32_t nblocks, const int32_t* __restrict__ slot_ptr,
    int32_t* __restrict__ inner, uint16_t* __restrict__ local, CutDev cut, int32_t grows,
    int32_t stride, int32_t lanes, int32_t wpb, int32_t scale, int32_t pad,
    const int32_t* __restrict__ wave_off, uint16_t* __restrict__ sliced) {
  extern __shared__ double slice_lds[];
  __shared__ int32_t start[kSliceRows], len[kSliceRows];
  // The rows; then the staged positions, whose place order_part's memory takes
  // afterwards.
  uint16_t* in = reinterpret_cast<uint16_t*>(slice_lds);
  double* pos = slice_lds + (grows * stride + 3) / 4;
  OrderLds* order = reinterpret_cast<OrderLds*>(pos);
  const int tid = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
  const int lane = tid & (kRowLanes - 1), seg = (tid & 63) & ~(kRowLanes - 1);
  const int lsh = 31 - __clz(lanes);
  const int rpw = 64 >> lsh;  // rows per wavefront
  const int64_t st = cut.q.stride;
  // The kernels' offset prefetch reads past the last slice.
  if (blockIdx.x == 0)
    for (int t = tid; t < pad; t += nt)
      sliced[wave_off[static_cast<int64_t>(nblocks) * wpb] + t] = 0;
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const int32_t* d = desc + 8 * static_cast<int64_t>(b);
    const int32_t i0 = d[0], ni = d[1], soff = d[2], ns = d[3];
    double box = cut.box;
    if (CUT && cut.rep_box) box = cut.rep_box[2 * d[6]];
    for (int32_t g0 = 0; g0 < ni; g0 += grows) {
      const int nr = min(grows, ni - g0);
      if (tid < nr) {
        const int32_t a = slot_ptr[i0 + g0 + tid];
        const int32_t m = slot_ptr[i0 + g0 + tid + 1] - a;
        start[tid] = a;
        len[tid] = m;
      }
      // The row of these lanes, its particle's position and its first entries,
      // requested before the staging so that their latencies overlap it.
      const int r = tid / kRowLanes;
      const int32_t slot = i0 + g0 + min(r, nr - 1);
      const int32_t a = slot_ptr[slot];
      const int all = slot_ptr[slot + 1] - a;
      const int m = r < nr && all <= kBankRowMax ? all : 0;
      if (CUT && r < nr && all > kBankRowMax && lane == 0) inner[slot] = all;
      int nin = CUT || m == 0 ? 0 : inner ? inner[slot] : m, nout = 0;
      double xi = 0.0, yi = 0.0, zi = 0.0;
      if (CUT) {
        const int64_t i = static_cast<int64_t>(cut.member ? cut.member[slot] : slot) * st;
        xi = cut.q.x[i];
        yi = cut.q.y[i];
        zi = cut.q.z[i];
      }
      constexpr int kStep = kRowBatch * kRowLanes;
      int next[kRowBatch];
      auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < kRowBatch; u++) {
          const int k = k0 + u * kRowLanes + lane;
          next[u] = local[a + (k < m ? k : 0)];
        }
      };
      if (m > 0) load(0);
      if (CUT && POS_LDS) {
#pragma unroll 2
        for (int t = tid; t < ns; t += nt) {
          const int64_t j = static_cast<int64_t>(cut.stage[soff + t]) * st;
          pos[3 * t] = cut.q.x[j];
          pos[3 * t + 1] = cut.q.y[j];
          pos[3 * t + 2] = cut.q.z[j];
        }
      }
      __syncthreads();
      uint16_t* row = in + min(r, grows - 1) * stride;
      for (int k0 = 0; k0 < m; k0 += kStep) {
        int rank[kRowBatch];
#pragma unroll
        for (int u = 0; u < kRowBatch; u++)
          rank[u] = k0 + u * kRowLanes + lane < m ? next[u] / 24 : -1;
        if (k0 + kStep < m) load(k0 + kStep);
        if (!CUT) {
#pragma unroll
          for (int u = 0; u < kRowBatch; u++) {
            const int k = k0 + u * kRowLanes + lane;
            if (rank[u] >= 0)
              row[ORDER && k >= nin ? m - 1 - (k - nin) : k] = static_cast<uint16_t>(rank[u]);
          }
          continue;
        }
        bool in_u[kRowBatch];
#pragma unroll
        for (int u = 0; u < kRowBatch; u++) {
          const int t = max(rank[u], 0);
          double xj, yj, zj;
          if (POS_LDS) {
            xj = pos[3 * t];
            yj = pos[3 * t + 1];
            zj = pos[3 * t + 2];
          } else {
            const int64_t j = static_cast<int64_t>(cut.stage[soff + t]) * st;
            xj = cut.q.x[j];
            yj = cut.q.y[j];
            zj = cut.q.z[j];
          }
          in_u[u] = cut_inner(xi, yi, zi, xj, yj, zj, box, cut.cl2);
        }
#pragma unroll
        for (int u = 0; u < kRowBatch; u++) {
          const bool valid = rank[u] >= 0;
          constexpr uint32_t kSeg = (1u << kRowLanes) - 1;
          const uint32_t vm = kSeg & static_cast<uint32_t>(__ballot(valid) >> seg);
          const uint32_t im = kSeg & static_cast<uint32_t>(__ballot(valid && in_u[u]) >> seg);
          const uint32_t below = (1u << lane) - 1;
          if (valid)
            row[in_u[u] ? nin + __popc(im & below) : m - 1 - nout - __popc(vm & ~im & below)] =
                static_cast<uint16_t>(rank[u]);
          nin += __popc(im);
          nout += __popc(vm & ~im);
        }
      }
      if (CUT && m > 0) {
        if (lane == 0) inner[slot] = nin;
        // The row goes back in its new order (its lanes belong to one
        // wavefront, so their LDS writes come before these reads).
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (nout > 0)
          for (int k = lane; k < m; k += kRowLanes)
            local[a + k] = static_cast<uint16_t>(row[k < nin ? k : m - 1 - (k - nin)] * 24);
      }
      __syncthreads();
      if (ORDER) {
        const int phase = (g0 + r) << lsh;
#pragma nounroll
        for (int part = 0; part < 2; part++) {
          const int n = part ? m - nin : nin, most = wave_max(n);
          if (most == 0) continue;  // the whole wavefront
          const int skip = part ? nin : 0;
          order_part(part ? row + max(m - 1, 0) : row, part ? -1 : 1, row + skip, phase + skip, n,
                     most, order[tid / 64]);
        }
        __syncthreads();
      }
      for (int w = g0 / rpw + tid / 64; w < min(wpb, (g0 + grows) / rpw); w += nt / 64) {
        const int32_t p0 = wave_off[static_cast<int64_t>(b) * wpb + w];
        const int32_t n = wave_off[static_cast<int64_t>(b) * wpb + w + 1] - p0;
        const int r = w * rpw + ((tid & 63) >> lsh) - g0;
        const int m = r < nr ? len[r] : 0;
        const bool direct = m > kBankRowMax;
        const uint16_t* src = direct ? local + start[r] : in + min(r, grows - 1) * stride;
        int k = tid & (lanes - 1);
#pragma unroll 4
        for (int32_t p = tid & 63; p < n; p += 64, k += lanes)
          sliced[p0 + p] =
              k < m ? static_cast<uint16_t>((direct ? src[k] / 24 : src[k]) * scale) : uint16_t{0};
      }
      __syncthreads();
    }
  }
}

// Half lists over tiles. Staged counts of the tiles; then per tile its first
// row of force sums and the rank of its own first slot (keys: the staged
// slots, ascending), and the number of staged places of each slot.
__global__ void k_half_counts(int32_t nblocks, const int32_t* __restrict__ desc,
                              int32_t* __restrict__ ns) {
  const int64_t b = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (b < nblocks) ns[b] = desc[8 * b + 3];
}

__global__ __launch_bounds__(kBlock) void k_half_places(
    int32_t nblocks, const int32_t* __restrict__ desc, const int32_t* __restrict__ keys,
    const int32_t* __restrict__ first_row, int2* __restrict__ tile, int32_t* __restrict__ count) {
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const int32_t* d = desc + 8 * static_cast<int64_t>(b);
    const int32_t i0 = d[0], soff = d[2], ns = d[3];
    for (int t = threadIdx.x; t < ns; t += kBlock) {
      const int32_t s = keys[soff + t];
      atomicAdd(&count[s], 1);
      if (s == i0) tile[b] = make_int2(first_row[b], t);
    }
  }
}

// The rows of each slot, in arrival order, then ascending (k_half_sort, a few rows each).
__global__ __launch_bounds__(kBlock) void k_half_fill(
    int32_t nblocks, const int32_t* __restrict__ desc, const int32_t* __restrict__ keys,
    const int32_t* __restrict__ first_row, const int32_t* __restrict__ first,
    int32_t* __restrict__ used, int32_t* __restrict__ at) {
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const int32_t* d = desc + 8 * static_cast<int64_t>(b);
    const int32_t soff = d[2], ns = d[3];
    for (int t = threadIdx.x; t < ns; t += kBlock) {
      const int32_t s = keys[soff + t];
      at[first[s] + atomicAdd(&used[s], 1)] = first_row[b] + t;
    }
  }
}

// Batched replicas.
__global__ void k_copy_add(int64_t n, const int32_t* __restrict__ src, int32_t* __restrict__ dst,
                           int32_t add) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    dst[t] = src[t] + add;
}

__global__ void k_replica_of(int32_t n, const int32_t* __restrict__ off, int32_t nrep,
                             int32_t* __restrict__ rep) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    int32_t lo = 0, hi = nrep;  // last r with off[r] <= t
    while (hi - lo > 1) {
      const int32_t mid = (lo + hi) >> 1;
      if (off[mid] <= t) lo = mid;
      else hi = mid;
    }
    rep[t] = lo;
  }
}

__global__ void k_check_replicas(int32_t n, const int32_t* __restrict__ nop,
                                 const int32_t* __restrict__ ptr, const int32_t* __restrict__ list,
                                 const int32_t* __restrict__ rep,
                                 unsigned long long* __restrict__ bad) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t kp = ptr[t];
    for (int32_t k = 0; k < nop[t]; k++)
      if (rep[list[kp + k]] != rep[t]) {
        atomicMin(bad, static_cast<unsigned long long>(t));
        break;
      }
  }
}

// at[0 .. m), m <= M distinct values, ascending: every load before the first use.
template <int M>
__device__ __forceinline__ void sort_few(int32_t* __restrict__ at, int32_t m) {
  int32_t v[M];
#pragma unroll
  for (int k = 0; k < M; k++) v[k] = k < m ? at[k] : INT32_MAX;
#pragma unroll
  for (int k = 0; k < M; k++) {
    int32_t r = 0;
#pragma unroll
    for (int j = 0; j < M; j++) r += v[j] < v[k] ? 1 : 0;
    if (k < m) at[r] = v[k];
  }
}

// About seven rows a slot at density 0.8, at a tile's corner some twenty (14 us at
// 62,463 particles; by insertion in memory 39).
__global__ void k_half_sort(int32_t n, const int32_t* __restrict__ first,
                            int32_t* __restrict__ at) {
  const int64_t c = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (c >= n) return;
  const int32_t a = first[c], b = first[c + 1];
  if (b - a <= 8) return sort_few<8>(at + a, b - a);
  if (b - a <= 16) return sort_few<16>(at + a, b - a);
  if (b - a <= 32) return sort_few<32>(at + a, b - a);
  for (int32_t k = a + 1; k < b; k++) {
    const int32_t v = at[k];
    int32_t m = k;
    for (; m > a && at[m - 1] > v; m--) at[m] = at[m - 1];
    at[m] = v;
  }
}

__global__ void k_order_key(int32_t n, OrderKey key, int32_t* __restrict__ count,
                            int32_t* __restrict__ slot, int32_t* __restrict__ key_of) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t k = key(t, nullptr);
    key_of[t] = k;
    slot[t] = atomicAdd(&count[k], 1);
  }
}

// The slots of a spatial order: each block's particles (tile_span) reordered
// by row length, longest first, ties in the order given (the wavefronts of a
// tile then hold rows of similar length, which need similar numbers of
// batches); the particle of each slot, the slot of each particle and each
// slot's row length.
__global__ __launch_bounds__(kBlock) void k_tile_slots(TileSpans spans, int32_t nblocks,
                                                       const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ nop,
                                                       int32_t* __restrict__ member,
                                                       int32_t* __restrict__ slot_of,
                                                       int32_t* __restrict__ slot_len) {
  __shared__ int32_t mem[kTileRowsMax];
  __shared__ int32_t len[kTileRowsMax];
  for (int32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const TileSpan g = tile_span(spans, b);
    for (int32_t t = threadIdx.x; t < g.ni; t += blockDim.x) {
      const int32_t i = order[g.i0 + t];
      mem[t] = i;
      len[t] = nop[i];
    }
    __syncthreads();
    for (int32_t t = threadIdx.x; t < g.ni; t += blockDim.x) {
      const int32_t l = len[t];
      int32_t r = g.i0;
      for (int32_t u = 0; u < g.ni; u++) r += len[u] > l || (len[u] == l && u < t);
      member[r] = mem[t];
      slot_of[mem[t]] = r;
      slot_len[r] = l;
    }
    __syncthreads();
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
int dev_reserve(DevMem& m, size_t bytes, hipStream_t stream) {
  bytes = std::max<size_t>(bytes, 16);
  if (m.p && m.bytes >= bytes) return LJGPU_OK;
  if (m.p) {
    LTRY(hipStreamSynchronize(stream), "hipStreamSynchronize");
    (void)hipFree(m.p);
    m.p = nullptr;
    m.bytes = 0;
  }
  const size_t grow = bytes + bytes / 8;  // headroom for the next, slightly larger build
  if (grow > m.limit) return hip_err(hipErrorOutOfMemory, "hipMalloc (list buffer)");
  LTRY(hipMalloc(&m.p, grow), "hipMalloc (list buffer)");
  m.bytes = grow;
  return LJGPU_OK;
}

void dev_release(DevMem& m) {
  if (m.p) (void)hipFree(m.p);
  m.p = nullptr;
  m.bytes = 0;
}

void dev_release(DevCSR& c) {
  dev_release(c.nop);
  dev_release(c.ptr);
  dev_release(c.list);
  c.n = 0;
  c.e = 0;
}

void dev_release(DevTiles& t) {
  dev_release(t.desc);
  dev_release(t.stage);
  dev_release(t.local);
  dev_release(t.sliced);
  t.bank_rows = false;
  t.bank_lanes = t.bank_unroll = 0;
  t.slice_elems = 0;
  dev_release(t.wave_off);
  t.sliced_lanes = t.sliced_unroll = t.waves_per_block = 0;
  dev_release(t.member);
  dev_release(t.slot_ptr);
  dev_release(t.stage_slot);
  dev_release(t.inner);
  for (DevMem* m : {&t.half_tile, &t.half_first, &t.half_at, &t.half_part}) dev_release(*m);
  t.half_ready = false;
  t.cut = false;
  t.tile_particles = 0;
  t.blocks = 0;
  t.staged = 0;
  t.max_stage = 0;
  t.lds_bytes = 0;
}

void dev_release(ListWork& w) {
  for (DevMem* m : {&w.scan_sums, &w.small, &w.cell_count, &w.cell_start, &w.cell_slot, &w.cell_of,
                    &w.cell_sorted, &w.cpos, &w.counts, &w.tmp, &w.tile_ns, &w.tile_soff, &w.tile_stats,
                    &w.tile_geo, &w.rep_of, &w.order, &w.order_grid, &w.slot_of})
    dev_release(*m);
  dev_release(w.part);
  if (w.results) (void)hipHostFree(w.results);
  w.results = nullptr;
}

// The host-visible results (pinned memory that kernels write): a result is
// valid once the stream has been synchronised after its kernel.
int results(ListWork& w) {
  if (!w.results)
    LTRY(hipHostMalloc(reinterpret_cast<void**>(&w.results), sizeof(ListResults), hipHostMallocDefault),
         "hipHostMalloc");
  return LJGPU_OK;
}

int dev_scan_async(hipStream_t s, const int32_t* in, int32_t* out, int64_t n, ListWork& w,
                   ScanStats* res) {
  if (n <= kScanSmall) {
    k_scan_small<<<1, 1024, 0, s>>>(in, static_cast<int32_t>(n), out, res);
    LTRY(hipGetLastError(), "scan kernel");
    return LJGPU_OK;
  }
  const int64_t nb = (n + kScanTile - 1) / kScanTile;
  LCHECK(dev_reserve(w.scan_sums, sizeof(ScanTile) * nb, s));
  ScanTile* tiles = w.scan_sums.as<ScanTile>();
  k_scan_reduce<<<static_cast<int>(nb), kBlock, 0, s>>>(in, n, tiles);
  if (nb > kScanTiles) {
    k_scan_sums<<<1, kBlock, 0, s>>>(tiles, nb);
    k_scan_apply<true><<<static_cast<int>(nb), kBlock, 0, s>>>(in, n, tiles, out, res);
  } else {
    k_scan_apply<false><<<static_cast<int>(nb), kBlock, 0, s>>>(in, n, tiles, out, res);
  }
  LTRY(hipGetLastError(), "scan kernels");
  return LJGPU_OK;
}

int dev_scan(hipStream_t s, const int32_t* in, int32_t* out, int64_t n, ListWork& w,
             int64_t* total) {
  *total = 0;
  LCHECK(results(w));
  LCHECK(dev_scan_async(s, in, out, std::max<int64_t>(n, 0), w, &w.results->scan));
  LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  *total = w.results->scan.total;
  return LJGPU_OK;
}

int dev_validate(hipStream_t s, int32_t n, const int32_t* nop, const int32_t* ptr,
                 const int32_t* list, int64_t e, int kind, ListWork& w) {
  if (n <= 0) return LJGPU_OK;
  LCHECK(dev_reserve(w.small, sizeof(int64_t) * 8, s));
  unsigned long long* bad = w.small.as<unsigned long long>();
  LCHECK(fill<unsigned long long>(s, bad, 1, ~0ull));
  k_validate<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, nop, ptr, list, e,
                                                   kind == LJGPU_LIST_HALF ? 1 : 0, bad);
  LTRY(hipGetLastError(), "validate kernel");
  unsigned long long h = 0;
  LTRY(hipMemcpyAsync(&h, bad, sizeof(h), hipMemcpyDeviceToHost, s), "hipMemcpyAsync");
  LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  if (h == ~0ull) return LJGPU_OK;
  const int64_t row = static_cast<int64_t>(h / 8);
  static const char* what[] = {"", "number_of_partners out of range", "row leaves the list",
                               "partner index out of range", "row lists itself",
                               "half list holds j < i"};
  return set_error(LJGPU_ERR_BAD_LIST,
                   "row " + std::to_string(row) + ": " + what[std::min<unsigned long long>(h % 8, 5)]);
}

int dev_copy_row_ordered(hipStream_t s, int32_t n, const int32_t* nop, const int32_t* ptr,
                         const int32_t* list, int64_t e, ListWork& w, DevCSR& out) {
  (void)e;
  out.n = n;
  LCHECK(dev_reserve(out.nop, sizeof(int32_t) * std::max(n, 1), s));
  LCHECK(dev_reserve(out.ptr, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  if (n > 0)
    LTRY(hipMemcpyAsync(out.nop.p, nop, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, s),
         "hipMemcpyAsync");
  int64_t total = 0;
  LCHECK(dev_scan(s, out.nop.as<int32_t>(), out.ptr.as<int32_t>(), n, w, &total));
  if (total > INT32_MAX) return set_error(LJGPU_ERR_CAPACITY, "list longer than 2^31-1 entries");
  out.e = total;
  LCHECK(dev_reserve(out.list, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  if (n > 0) {
    k_copy_rows<<<grid_for(n, kBlock / 64), kBlock, 0, s>>>(n, nop, ptr, list, out.ptr.as<int32_t>(),
                                                           out.list.as<int32_t>());
    LTRY(hipGetLastError(), "copy rows kernel");
  }
  return LJGPU_OK;
}

int dev_expand_half(hipStream_t s, int32_t n, const int32_t* hnop, const int32_t* hptr,
                    const int32_t* hlist, ListWork& w, DevCSR& full) {
  full.n = n;
  LCHECK(dev_reserve(w.counts, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  LCHECK(dev_reserve(w.cell_slot, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  LCHECK(dev_reserve(full.nop, sizeof(int32_t) * std::max(n, 1), s));
  LCHECK(dev_reserve(full.ptr, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  int32_t* lower = w.counts.as<int32_t>();
  int32_t* fillc = w.cell_slot.as<int32_t>();
  LCHECK(fill<int32_t>(s, lower, n, 0));
  LCHECK(fill<int32_t>(s, fillc, n, 0));
  if (n > 0) {
    k_count_lower<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, hnop, hptr, hlist, lower);
    k_add<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, lower, hnop, full.nop.as<int32_t>());
    LTRY(hipGetLastError(), "expand kernels");
  }
  int64_t total = 0;
  LCHECK(dev_scan(s, full.nop.as<int32_t>(), full.ptr.as<int32_t>(), n, w, &total));
  if (total > INT32_MAX) return set_error(LJGPU_ERR_CAPACITY, "full list longer than 2^31-1 entries");
  full.e = total;
  LCHECK(dev_reserve(full.list, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  LCHECK(dev_reserve(w.tmp, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  if (n > 0) {
    k_fill_expanded<<<grid_for(n, kBlock), kBlock, 0, s>>>(
        n, hnop, hptr, hlist, lower, full.ptr.as<int32_t>(), fillc, w.tmp.as<int32_t>(),
        full.list.as<int32_t>());
    LTRY(hipGetLastError(), "expand fill kernel");
    // Lower partners ascending (the order in which the reference's rows
    // r < i list i).
    LCHECK(row_sort(s, n, lower, full.ptr.as<int32_t>(), w.tmp.as<int32_t>(),
                    full.list.as<int32_t>()));
  }
  return LJGPU_OK;
}

// The tile order's job that dev_tile_order_begin left for this list build.
bool take_order_job(ListWork& w, OrderJob* job) {
  static_assert(std::is_trivially_copyable<OrderJob>::value, "kept as bytes");
  if (w.order_job.size() != sizeof(*job)) return false;
  std::memcpy(static_cast<void*>(job), w.order_job.data(), sizeof(*job));
  w.order_job.clear();
  return true;
}

int dev_makepair(hipStream_t s, const PosIn& q, int32_t n, double box, double search_length,
                 int kind, ListWork& w, DevCSR& out, bool sort_rows) {
  const double sl2 = search_length * search_length;
  out.n = n;
  LCHECK(dev_reserve(out.nop, sizeof(int32_t) * std::max(n, 1), s));
  LCHECK(dev_reserve(out.ptr, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  w.row_min = w.row_max = 0;
  out.slab_stride = 0;
  if (n == 0) {
    out.e = 0;
    LCHECK(dev_reserve(out.list, sizeof(int32_t), s));
    return fill<int32_t>(s, out.ptr.as<int32_t>(), 1, 0);
  }
  double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  if (box <= 0.0) {
    // Bounding box of the open system, reduced on the device.
    std::vector<double> ext(6);
    DevMem& m = w.scan_sums;
    LCHECK(dev_reserve(m, sizeof(double) * 6, s));
    const double* comp[3] = {q.x, q.y, q.z};
    for (int c = 0; c < 3; c++)
      k_extrema<<<1, kBlock, 0, s>>>(n, comp[c], q.stride, m.as<double>() + 2 * c);
    LTRY(hipGetLastError(), "bounding box kernel");
    LTRY(hipMemcpyAsync(ext.data(), m.p, sizeof(double) * 6, hipMemcpyDeviceToHost, s),
         "hipMemcpyAsync");
    LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
    for (int c = 0; c < 3; c++) {
      lo[c] = ext[2 * c];
      hi[c] = ext[2 * c + 1];
      if (!std::isfinite(lo[c]) || !std::isfinite(hi[c]))
        return set_error(LJGPU_ERR_INVALID_ARGUMENT, "positions are not finite");
    }
  }
  // Cells at least half the search length wide with a radius-2 stencil
  // visit about 45 % fewer candidates than search-length cells with a
  // radius-1 stencil; a periodic box needs 5 such cells per side (each cell
  // visited once), else the coarser grid is used.
  CellGrid cg;
  make_cell_grid(n, lo, hi, box, 0.5 * search_length, &cg);
  bool fine = !cg.brute;
  for (int c = 0; c < 3; c++)
    if (box > 0.0 && cg.nc[c] < 5) fine = false;
  if (!fine) make_cell_grid(n, lo, hi, box, search_length, &cg);
  GridArgs g{cg.nc[0], cg.nc[1], cg.nc[2], cg.origin[0], cg.origin[1], cg.origin[2],
             cg.width[0], cg.width[1], cg.width[2], box};
  const int64_t ncell = cg.ncell;
  LCHECK(dev_reserve(w.cell_count, sizeof(int32_t) * (ncell + 1), s));
  LCHECK(dev_reserve(w.cell_start, sizeof(int32_t) * (ncell + 1), s));
  LCHECK(dev_reserve(w.cell_slot, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.cell_of, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.cell_sorted, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.cpos, sizeof(double4) * n, s));
  int32_t* count = w.cell_count.as<int32_t>();
  int32_t* cstart = w.cell_start.as<int32_t>();
  int32_t* outside = count + ncell;
  LCHECK(results(w));
  const CellKey key{q, g};
  const bool few = n <= kBinSmall && ncell <= kBinsSmall;
  if (few) {
    const CellJob job{n, static_cast<int32_t>(ncell), key,
                      CellPut{q, w.cpos.as<double4>(), w.cell_sorted.as<int32_t>()}, cstart, outside,
                      &w.results->cells};
    OrderJob order;
    if (take_order_job(w, &order)) k_bin_small<<<2, kBinThreads, 0, s>>>(job, order);
    else k_bin_small<<<1, kBinThreads, 0, s>>>(job, NoBinJob{});
    LTRY(hipGetLastError(), "cell kernel");
  } else {
    OrderJob order;
    if (take_order_job(w, &order)) k_bin_small<<<1, kBinThreads, 0, s>>>(order, NoBinJob{});
    LTRY(hipGetLastError(), "tile order kernel");
    LCHECK(fill<int32_t>(s, count, ncell + 1, 0));
    k_cell_assign<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, key, count, w.cell_slot.as<int32_t>(),
                                                         w.cell_of.as<int32_t>(), outside);
    LTRY(hipGetLastError(), "cell assign kernel");
    LCHECK(dev_scan_async(s, count, cstart, ncell, w, &w.results->cells));
  }
  const bool half = kind == LJGPU_LIST_HALF;
  const int R = cg.brute ? 0 : (fine ? 2 : 1);
  // Unsorted rows need a candidate order fixed by the positions alone: the
  // stencil kernel's run order with each cell's particles by index. The
  // single-cell kernel has no such order, so it always sorts.
  if (R == 0) sort_rows = true;
  if (few) {
    // Placed already, each cell's particles by index.
  } else if (sort_rows) {
    k_cell_scatter<<<grid_for(n, kBlock), kBlock, 0, s>>>(
        n, q, w.cell_of.as<int32_t>(), w.cell_slot.as<int32_t>(), cstart, w.cpos.as<double4>(),
        w.cell_sorted.as<int32_t>());
  } else {
    int32_t* arrival = w.cell_sorted.as<int32_t>();
    k_bin_index<<<grid_for(n, kBlock), kBlock, 0, s>>>(
        n, w.cell_of.as<int32_t>(), w.cell_slot.as<int32_t>(), cstart, arrival);
    k_cell_place<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, q, w.cell_of.as<int32_t>(), cstart,
                                                        arrival, w.cpos.as<double4>());
  }
  LTRY(hipGetLastError(), "cell scatter kernels");
  const int grid = grid_for(n, kBlock, INT32_MAX);
  // One wavefront per cell, grid-stride; in small systems several, which share
  // its particles.
  const int split = ncell <= kPairCellsFour ? 2 : ncell <= kPairCellsTwo ? 1 : 0;
  const int wave_grid = grid_for((ncell << split) * 64, kBlock);
  auto pairs = [&](auto mode_tag, int32_t cap, int32_t* nop, const int32_t* ptr, int32_t* outl) {
    constexpr int M = decltype(mode_tag)::value;
    const double4* cp = w.cpos.as<double4>();
    const int32_t* cs = w.cell_sorted.as<int32_t>();
    // A single all-particle cell (R = 0) runs one thread per particle; a
    // stencil grid one wavefront per cell.
#define LJ_PAIRS(H) \
  k_pairs<M, H, 0><<<grid, kBlock, 0, s>>>(n, cp, cs, cstart, g, sl2, cap, nop, ptr, outl)
#define LJ_PAIRS_WAVE(H, RR)                                                                     \
  k_pairs_wave<M, H, RR><<<wave_grid, kBlock, 0, s>>>(static_cast<int32_t>(ncell), cp, cstart, g, \
                                                      sl2, cap, nop, ptr, outl, outside, split)
    if (half) {
      if (R == 0) LJ_PAIRS(true);
      else if (R == 1) LJ_PAIRS_WAVE(true, 1);
      else LJ_PAIRS_WAVE(true, 2);
    } else {
      if (R == 0) LJ_PAIRS(false);
      else if (R == 1) LJ_PAIRS_WAVE(false, 1);
      else LJ_PAIRS_WAVE(false, 2);
    }
#undef LJ_PAIRS
#undef LJ_PAIRS_WAVE
  };
  // Single pass into a slab of `cap` entries per row, sized from the last
  // build's longest row (or from the mean density), then one sort from the
  // slab into place; a row longer than the slab falls back to a second,
  // exact-size pass. Without room for a slab: count pass, then fill pass.
  int32_t cap = 0;
  {
    double vol = 1.0;
    for (int c = 0; c < 3; c++) vol *= std::max(cg.extent[c], search_length);
    const double expect = 4.18879020478639 * search_length * search_length * search_length *
                          (static_cast<double>(n) / vol) * (half ? 0.5 : 1.0);
    const double want = w.last_max_row > 0 ? 1.2 * w.last_max_row + 16 : 1.5 * expect + 32;
    cap = static_cast<int32_t>(std::min(4096.0, std::max(64.0, want)));
    cap = (cap + 31) / 32 * 32;
    if (static_cast<double>(n) * cap * 4.0 > 16.0 * (1u << 30)) cap = 0;
  }
  if (cap > 0) {
    LCHECK(dev_reserve(w.tmp, sizeof(int32_t) * static_cast<size_t>(n) * cap, s));
    pairs(std::integral_constant<int, 2>{}, cap, out.nop.as<int32_t>(), nullptr,
          w.tmp.as<int32_t>());
    LTRY(hipGetLastError(), "pair kernel");
  } else {
    pairs(std::integral_constant<int, 0>{}, 0, out.nop.as<int32_t>(), nullptr, nullptr);
    LTRY(hipGetLastError(), "pair count kernel");
  }
  int64_t total = 0;
  LCHECK(dev_scan(s, out.nop.as<int32_t>(), out.ptr.as<int32_t>(), n, w, &total));
  const int32_t mx = w.results->scan.hi;
  w.row_min = w.results->scan.lo;
  w.row_max = mx;
  // Crowded cells (a collapsed or clustered system) are not in index order.
  if (w.results->cells.hi > kCellOrderMax) sort_rows = true;
  if (total > INT32_MAX) return set_error(LJGPU_ERR_CAPACITY, "list longer than 2^31-1 entries");
  out.e = total;
  if (cap > 0 && mx <= cap) {
    w.last_max_row = mx;
    if (!sort_rows) {
      out.slab_stride = cap;  // the rows stay in w.tmp: dev_copy_slab
      return LJGPU_OK;
    }
    LCHECK(dev_reserve(out.list, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
    return row_sort(s, n, out.nop.as<int32_t>(), out.ptr.as<int32_t>(), w.tmp.as<int32_t>(),
                    out.list.as<int32_t>(), cap);
  }
  LCHECK(dev_reserve(out.list, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  if (cap > 0) w.last_max_row = mx;
  if (!sort_rows) {
    pairs(std::integral_constant<int, 1>{}, 0, out.nop.as<int32_t>(), out.ptr.as<int32_t>(),
          out.list.as<int32_t>());
    LTRY(hipGetLastError(), "pair fill kernel");
    return LJGPU_OK;
  }
  LCHECK(dev_reserve(w.tmp, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  pairs(std::integral_constant<int, 1>{}, 0, out.nop.as<int32_t>(), out.ptr.as<int32_t>(),
        w.tmp.as<int32_t>());
  LTRY(hipGetLastError(), "pair fill kernel");
  return row_sort(s, n, out.nop.as<int32_t>(), out.ptr.as<int32_t>(), w.tmp.as<int32_t>(),
                  out.list.as<int32_t>());
}

int dev_copy_slab(hipStream_t s, ListWork& w, DevCSR& c) {
  if (c.slab_stride == 0) return LJGPU_OK;
  LCHECK(dev_reserve(c.list, sizeof(int32_t) * std::max<int64_t>(c.e, 1), s));
  k_copy_slab<<<grid_for((c.n + kSlabRows - 1) / kSlabRows, kBlock / 64), kBlock, 0, s>>>(
      c.n, c.nop.as<int32_t>(), c.ptr.as<int32_t>(), w.tmp.as<int32_t>(), c.slab_stride,
      c.list.as<int32_t>());
  LTRY(hipGetLastError(), "slab copy kernel");
  c.slab_stride = 0;
  return LJGPU_OK;
}

int dev_minmax(hipStream_t s, const int32_t* a, int32_t n, ListWork& w, int32_t* mn,
               int32_t* mx) {
  *mn = 0;
  *mx = 0;
  if (n <= 0) return LJGPU_OK;
  LCHECK(dev_reserve(w.small, sizeof(int64_t) * 8, s));
  int32_t* mm = w.small.as<int32_t>();
  LCHECK(fill<int32_t>(s, mm, 1, INT32_MAX));
  LCHECK(fill<int32_t>(s, mm + 1, 1, INT32_MIN));
  k_minmax<<<grid_for(n, kBlock, 256), kBlock, 0, s>>>(n, a, mm);
  LTRY(hipGetLastError(), "minmax kernel");
  int32_t h[2];
  LTRY(hipMemcpyAsync(h, mm, sizeof(h), hipMemcpyDeviceToHost, s), "hipMemcpyAsync");
  LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  *mn = h[0];
  *mx = h[1];
  return LJGPU_OK;
}

int dev_half_row_stats(hipStream_t s, const DevCSR& full, ListWork& w, int32_t* min_np,
                       int32_t* max_np) {
  if (full.n <= 0) return dev_minmax(s, nullptr, 0, w, min_np, max_np);
  LCHECK(dev_reserve(w.counts, sizeof(int32_t) * (static_cast<size_t>(full.n) + 1), s));
  k_upper_counts<<<grid_for(full.n, kBlock), kBlock, 0, s>>>(
      full.n, full.nop.as<int32_t>(), full.ptr.as<int32_t>(), full.list.as<int32_t>(),
      w.counts.as<int32_t>());
  LTRY(hipGetLastError(), "upper count kernel");
  return dev_minmax(s, w.counts.as<int32_t>(), full.n, w, min_np, max_np);
}

int dev_make_ell(hipStream_t s, const DevCSR& c, int32_t width, DevMem& ell) {
  width = std::max(width, 1);
  const int64_t cells = static_cast<int64_t>(c.n) * width;
  LCHECK(dev_reserve(ell, sizeof(int32_t) * std::max<int64_t>(cells, 1), s));
  if (c.n > 0) {
    k_ell<<<grid_for(c.n, kBlock), kBlock, 0, s>>>(c.n, width, c.nop.as<int32_t>(),
                                                   c.ptr.as<int32_t>(), c.list.as<int32_t>(),
                                                   ell.as<int32_t>());
    LTRY(hipGetLastError(), "ELL kernel");
  }
  return LJGPU_OK;
}

int dev_tile_order_begin(hipStream_t s, const PosIn& q, int32_t n, double box,
                         const std::vector<int32_t>& replicas, const std::vector<double>& boxes,
                         int32_t T, ListWork& w, bool* begun, bool defer) {
  *begun = false;
  w.order_job.clear();
  if (n <= 0 || T <= 0) return LJGPU_OK;
  const std::vector<int32_t> single = {0, n};
  const std::vector<int32_t>& off = replicas.empty() ? single : replicas;
  const int32_t nsys = static_cast<int32_t>(off.size()) - 1;
  // Kept: the upload below reads it after this returns. One not yet read (of a
  // build that failed before it synchronised) must not be written over.
  std::vector<char>& store = w.order_host;
  if (!replicas.empty() && !store.empty()) LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  const size_t gbytes = (sizeof(OrderGrid) * nsys + 255) / 256 * 256;
  store.resize(gbytes + sizeof(int32_t) * off.size());
  OrderGrid* grids = reinterpret_cast<OrderGrid*>(store.data());
  int64_t keys = 0;
  for (int32_t r = 0; r < nsys; r++) {
    const double L = replicas.empty() ? box : boxes[r];
    if (!(L > 0.0) || !std::isfinite(L)) return LJGPU_OK;  // open systems keep index order
    const int32_t m = std::max(off[r + 1] - off[r], 1);
    OrderGrid& g = grids[r];
    g.box = L;
    const double rho = m / (L * L * L);
    const double side = 0.75 * std::cbrt(T / rho);
    // Rounded to the nearest count: for lattices of 4k^3 particles L / side
    // often lands exactly on an integer, where truncation would follow
    // last-bit rounding.
    for (int c = 1; c < 3; c++) {
      const double v = std::floor(L / side + 0.5);
      g.nc[c] = v >= 1024.0 ? 1024 : std::max(1, static_cast<int>(v));
    }
    // A few particles in a large box: at most about 2 columns per particle,
    // so the key arrays stay proportional to N.
    while (static_cast<int64_t>(g.nc[1]) * g.nc[2] > 2 * static_cast<int64_t>(m) + 16) {
      int& big = g.nc[1] >= g.nc[2] ? g.nc[1] : g.nc[2];
      big = (big + 1) / 2;
    }
    g.nc[0] = std::max<int32_t>(1, m / (g.nc[1] * g.nc[2]));
    for (int c = 0; c < 3; c++) g.w[c] = L / g.nc[c];
    g.key0 = static_cast<int32_t>(keys);
    keys += static_cast<int64_t>(g.nc[0]) * g.nc[1] * g.nc[2];
    if (keys > INT32_MAX - 1) return LJGPU_OK;
  }
  const int32_t* rep_of = nullptr;
  const OrderGrid* dgrids = nullptr;
  if (!replicas.empty()) {
    std::memcpy(store.data() + gbytes, off.data(), sizeof(int32_t) * off.size());
    LCHECK(dev_reserve(w.order_grid, store.size(), s));
    LTRY(hipMemcpyAsync(w.order_grid.p, store.data(), store.size(), hipMemcpyHostToDevice, s),
         "hipMemcpyAsync");
    dgrids = static_cast<const OrderGrid*>(w.order_grid.p);
    const int32_t* doff =
        reinterpret_cast<const int32_t*>(static_cast<const char*>(w.order_grid.p) + gbytes);
    LCHECK(dev_reserve(w.rep_of, sizeof(int32_t) * n, s));
    k_replica_of<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, doff, nsys, w.rep_of.as<int32_t>());
    LTRY(hipGetLastError(), "replica index kernel");
    rep_of = w.rep_of.as<int32_t>();
  }
  LCHECK(dev_reserve(w.cell_count, sizeof(int32_t) * (keys + 1), s));
  LCHECK(dev_reserve(w.cell_start, sizeof(int32_t) * (keys + 1), s));
  LCHECK(dev_reserve(w.cell_slot, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.cell_of, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.cell_sorted, sizeof(int32_t) * n, s));
  LCHECK(dev_reserve(w.order, sizeof(int32_t) * n, s));
  LCHECK(results(w));
  int32_t* count = w.cell_count.as<int32_t>();
  int32_t* start = w.cell_start.as<int32_t>();
  int32_t* arrival = w.cell_sorted.as<int32_t>();
  const int32_t* key_of = w.cell_of.as<int32_t>();
  const OrderKey key{q, grids[0], dgrids, rep_of};
  if (n <= kBinSmall && keys <= kBinsSmall) {
    const OrderJob job{n, static_cast<int32_t>(keys), key, OrderPut{w.order.as<int32_t>()}, nullptr,
                       nullptr, &w.results->order};
    if (defer) {
      w.order_job.resize(sizeof(job));
      std::memcpy(w.order_job.data(), &job, sizeof(job));
    } else {
      k_bin_small<<<1, kBinThreads, 0, s>>>(job, NoBinJob{});
    }
  } else {
    LCHECK(fill<int32_t>(s, count, keys, 0));
    k_order_key<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, key, count, w.cell_slot.as<int32_t>(),
                                                       w.cell_of.as<int32_t>());
    LTRY(hipGetLastError(), "tile order key kernel");
    LCHECK(dev_scan_async(s, count, start, keys, w, &w.results->order));
    k_bin_index<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, key_of, w.cell_slot.as<int32_t>(), start,
                                                       arrival);
    k_order_place<<<grid_for(n, kBlock), kBlock, 0, s>>>(n, key_of, start, arrival,
                                                         w.order.as<int32_t>());
  }
  LTRY(hipGetLastError(), "tile order kernels");
  *begun = true;
  return LJGPU_OK;
}

bool dev_tile_order_end(const ListWork& w) {
  return w.results->order.hi <= kCellOrderMax;  // a crowded bin: keep index order
}

int dev_tile_order(hipStream_t s, const PosIn& q, int32_t n, double box,
                   const std::vector<int32_t>& replicas, const std::vector<double>& boxes,
                   int32_t T, ListWork& w, bool* ok) {
  LCHECK(dev_tile_order_begin(s, q, n, box, replicas, boxes, T, w, ok));
  if (!*ok) return LJGPU_OK;
  LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  *ok = dev_tile_order_end(w);
  return LJGPU_OK;
}

// The blocks of T consecutive slots, restarted at every replica boundary.
int tile_spans(hipStream_t s, int32_t n, int32_t T, const std::vector<int32_t>& reps, ListWork& w,
               TileSpans* spans, int32_t* nblocks) {
  *spans = TileSpans{nullptr, T, n, 4};
  *nblocks = (n + T - 1) / T;
  if (reps.empty()) return LJGPU_OK;
  // Kept: the upload reads it after this returns. One not yet read must not
  // be written over.
  std::vector<int32_t>& geo = w.geo_host;
  if (!geo.empty()) LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  geo.clear();
  for (size_t r = 0; r + 1 < reps.size(); r++)
    for (int32_t i0 = reps[r]; i0 < reps[r + 1]; i0 += T)
      geo.insert(geo.end(), {i0, std::min(T, reps[r + 1] - i0), static_cast<int32_t>(r), 0});
  *nblocks = static_cast<int32_t>(geo.size() / 4);
  LCHECK(dev_reserve(w.tile_geo, sizeof(int32_t) * std::max<size_t>(geo.size(), 1), s));
  if (!geo.empty())
    LTRY(hipMemcpyAsync(w.tile_geo.p, geo.data(), sizeof(int32_t) * geo.size(),
                        hipMemcpyHostToDevice, s), "hipMemcpyAsync");
  spans->geo = w.tile_geo.as<int32_t>();
  return LJGPU_OK;
}

int dev_tile_slots(hipStream_t s, const DevCSR& c, int32_t T, const std::vector<int32_t>& reps,
                   ListWork& w, DevTiles& out) {
  TileSpans spans;
  int32_t nb = 0;
  LCHECK(tile_spans(s, c.n, T, reps, w, &spans, &nb));
  LCHECK(dev_reserve(out.member, sizeof(int32_t) * c.n, s));
  LCHECK(dev_reserve(out.slot_ptr, sizeof(int32_t) * (static_cast<size_t>(c.n) + 1), s));
  LCHECK(dev_reserve(w.slot_of, sizeof(int32_t) * c.n, s));
  LCHECK(dev_reserve(w.counts, sizeof(int32_t) * (static_cast<size_t>(c.n) + 1), s));
  k_tile_slots<<<std::max(1, std::min(nb, 65535)), kBlock, 0, s>>>(
      spans, nb, w.order.as<int32_t>(), c.nop.as<int32_t>(), out.member.as<int32_t>(),
      w.slot_of.as<int32_t>(), w.counts.as<int32_t>());
  LTRY(hipGetLastError(), "tile slot kernel");
  return dev_scan_async(s, w.counts.as<int32_t>(), out.slot_ptr.as<int32_t>(), c.n, w, nullptr);
}

// Entries past the last slice that the kernels' offset prefetch reads: two
// batches.
int32_t slice_pad(int32_t unroll) { return 2 * 64 * unroll + 64; }

// Lengths and starts of the slices (t.wave_off) and room for them (t.sliced);
// *wpb: wavefronts per block, 0 where slices cannot be made.
int plan_slices(hipStream_t s, const TileSpans& spans, int32_t nblocks, int32_t T,
                const int32_t* slot_ptr, int32_t lanes, int32_t unroll, int32_t longest,
                ListWork& w, DevTiles& t, int32_t* wpb) {
  *wpb = 0;
  if (lanes < 1 || lanes > 64 || (64 % lanes) != 0 || unroll < 1 || (unroll & (unroll - 1)) != 0)
    return LJGPU_OK;
  const int32_t waves = (T * lanes + 63) / 64;
  if (waves > kSliceWavesMax) return LJGPU_OK;
  const int64_t nw = static_cast<int64_t>(nblocks) * waves;
  LCHECK(dev_reserve(w.counts, sizeof(int32_t) * (static_cast<size_t>(nw) + 1), s));
  LCHECK(dev_reserve(t.wave_off, sizeof(int32_t) * (static_cast<size_t>(nw) + 1), s));
  k_wave_slices<<<grid_for(nw, kBlock), kBlock, 0, s>>>(spans, nblocks, waves, slot_ptr, lanes,
                                                        unroll, w.counts.as<int32_t>());
  LTRY(hipGetLastError(), "slice length kernel");
  // The slices' length is at most every wavefront's with the longest row; read
  // back only where that would be a waste.
  const int64_t kb = static_cast<int64_t>(lanes) * unroll;
  int64_t total = nw * 64 * unroll * ((longest + kb - 1) / kb);
  if (total <= int64_t{1} << 26)
    LCHECK(dev_scan_async(s, w.counts.as<int32_t>(), t.wave_off.as<int32_t>(), nw, w, nullptr));
  else
    LCHECK(dev_scan(s, w.counts.as<int32_t>(), t.wave_off.as<int32_t>(), nw, w, &total));
  const int32_t pad = slice_pad(unroll);
  if (total + pad > INT32_MAX) return LJGPU_OK;
  LCHECK(dev_reserve(t.sliced, sizeof(uint16_t) * (total + pad), s));
  t.slice_elems = total + pad;
  *wpb = waves;
  return LJGPU_OK;
}

int dev_make_tiles(hipStream_t s, const DevCSR& c, int32_t T, const std::vector<int32_t>& reps,
                   bool spatial, bool half, const SliceReq* req, ListWork& w, DevTiles& out) {
  out.tile_particles = 0;
  out.blocks = 0;
  out.shared = true;
  out.half_ready = false;
  if (T <= 0 || T > kTileRowsMax || c.n <= 0) return LJGPU_OK;
  // The slot order and each slot's row start in the slot-ordered rows.
  // Index order: slot = particle and the list's own row starts. Otherwise
  // dev_tile_slots's (blocks key their particles by slot).
  out.order = spatial ? LJGPU_TILE_ORDER_SPATIAL : LJGPU_TILE_ORDER_INDEX;
  const int32_t* member = spatial ? out.member.as<int32_t>() : nullptr;
  const int32_t* slot_of = spatial ? w.slot_of.as<int32_t>() : nullptr;
  const int32_t* sptr = spatial ? out.slot_ptr.as<int32_t>() : c.ptr.as<int32_t>();
  TileSpans spans;
  int32_t nb = 0;
  LCHECK(tile_spans(s, c.n, T, reps, w, &spans, &nb));
  if (nb == 0) return LJGPU_OK;
  const RowSource source{c.slab_stride > 0 ? w.tmp.as<int32_t>() : c.list.as<int32_t>(),
                         c.ptr.as<int32_t>(), c.slab_stride};
  // Slices of the rows as they stand, where the tiles' rows fit LDS.
  SliceDev slices{};
  const int32_t stride = req ? 2 * ((req->longest + 1) / 2 | 1) : 0;
  if (req && req->lanes > 1 && static_cast<int64_t>(T) * stride * 2 <= kPageBytes) {
    LCHECK(plan_slices(s, spans, nb, T, sptr, req->lanes, req->unroll, req->longest, w, out,
                       &slices.wpb));
    if (slices.wpb > 0) {
      slices.out = out.sliced.as<uint16_t>();
      slices.wave_off = out.wave_off.as<int32_t>();
      slices.lanes = req->lanes;
      slices.stride = stride;
      slices.pad = slice_pad(req->unroll);
    }
  }
  LCHECK(results(w));
  LCHECK(dev_reserve(w.tile_stats, sizeof(int4) * static_cast<size_t>(nb), s));
  int4* stats = w.tile_stats.as<int4>();
  const int grid = std::min(nb, 65535);
  // The force kernel copies entry offsets in whole 16-byte chunks: pad.
  const int64_t nlocal = c.e + kTileLocalPad;
  LCHECK(dev_reserve(out.local, sizeof(uint16_t) * nlocal, s));
  LCHECK(dev_reserve(out.desc, sizeof(int32_t) * 8 * static_cast<size_t>(nb), s));
  // One pass when every block can own kTileMaxStage staging slots within
  // kTileOnePassBytes (and the offsets fit int32); otherwise count, scan, fill.
  const int64_t slots = static_cast<int64_t>(nb) * kTileMaxStage;
  const bool one_pass =
      slots * static_cast<int64_t>(sizeof(int32_t)) * (member ? 2 : 1) <= kTileOnePassBytes &&
      slots <= INT32_MAX;
  int64_t staged = 0;
  int32_t h[4];
  // Sixteen lanes to a row, all rows of a tile of 64 at once; entry codes in
  // LDS for tiles up to a quarter longer than the average row makes them.
  const int threads = std::min(1024, std::max(256, T * kWordLanes));
  const int32_t ecap = static_cast<int32_t>(std::min<int64_t>(
      kTileCodeMax, (c.e / c.n + 1) * T * 5 / 4 + 64));
  const size_t code_bytes = sizeof(uint16_t) * ecap;
  auto read_stats = [&](int32_t (&back)[8]) -> int {
    k_tile_stats<<<1, 1024, 0, s>>>(nb, stats, out.local.as<uint16_t>() + c.e, w.results->tiles);
    LTRY(hipGetLastError(), "tile stats kernel");
    LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
    std::copy(w.results->tiles, w.results->tiles + 8, back);
    return LJGPU_OK;
  };
  if (one_pass) {
    LCHECK(dev_reserve(out.stage, sizeof(int32_t) * slots, s));
    if (member) LCHECK(dev_reserve(out.stage_slot, sizeof(int32_t) * slots, s));
    // Pages of 128 slots or more, so that the directory of a large system
    // fits LDS too.
    int32_t pshift = 7;
    while ((c.n >> pshift) >= kPageDir) pshift++;
    const int32_t npages = (c.n >> pshift) + 1;
    unsigned long long st = 0;
    for (int pass = 0; pass < 2; pass++) {
      if (pass == 0)
        k_tile_pages<<<grid, std::min(512, std::max(256, T * kPageLanes)), (npages + 15) / 16 * 16, s>>>(
            spans, nb, member, slot_of, sptr, source, pshift,
            npages, slices, out.desc.as<int32_t>(), out.stage.as<int32_t>(),
            member ? out.stage_slot.as<int32_t>() : nullptr,
            slices.out && !req->local ? nullptr : out.local.as<uint16_t>(), stats);
      else
        k_tile_fill<false><<<grid, threads, code_bytes, s>>>(
            spans, nb, member, slot_of, sptr, source, nullptr, ecap,
            nullptr, out.desc.as<int32_t>(), out.stage.as<int32_t>(),
            member ? out.stage_slot.as<int32_t>() : nullptr, out.local.as<uint16_t>(), stats);
      LTRY(hipGetLastError(), "tile fill kernel");
      int32_t back[8];
      LCHECK(read_stats(back));
      std::copy(back, back + 4, h);
      std::memcpy(&st, back + 6, sizeof(st));
      if (half && (back[4] > nb / 8 || 2 * static_cast<int64_t>(st) > c.e)) {
        out.shared = false;
        return LJGPU_OK;
      }
      if (back[4] == 0) {
        if (pass == 0 && slices.out && back[0] == 0) {
          out.sliced_lanes = req->lanes;
          out.sliced_unroll = req->unroll;
          out.waves_per_block = slices.wpb;
        }
        break;
      }  // else partners over too many pages: the hashed set
    }
    if (h[0] != 0) return LJGPU_OK;  // does not fit: caller retries smaller or runs untiled
    staged = static_cast<int64_t>(st);
    out.stage_stride = kTileMaxStage;
  } else {
    LCHECK(dev_reserve(w.tile_ns, sizeof(int32_t) * (static_cast<size_t>(nb) + 1), s));
    LCHECK(dev_reserve(w.tile_soff, sizeof(int32_t) * (static_cast<size_t>(nb) + 1), s));
    k_tile_fill<true><<<grid, threads, 0, s>>>(
        spans, nb, member, slot_of, sptr, source, nullptr, 0,
        w.tile_ns.as<int32_t>(), nullptr, nullptr, nullptr, nullptr, stats);
    LTRY(hipGetLastError(), "tile count kernel");
    int32_t back[8];
    LCHECK(read_stats(back));
    std::copy(back, back + 4, h);
    unsigned long long st = 0;
    std::memcpy(&st, back + 6, sizeof(st));
    if (half && 2 * static_cast<int64_t>(st) > c.e) {
      out.shared = false;
      return LJGPU_OK;
    }
    if (h[0] != 0) return LJGPU_OK;  // does not fit: caller retries smaller or runs untiled
    LCHECK(dev_scan(s, w.tile_ns.as<int32_t>(), w.tile_soff.as<int32_t>(), nb, w, &staged));
    if (staged > INT32_MAX) return LJGPU_OK;
    LCHECK(dev_reserve(out.stage, sizeof(int32_t) * std::max<int64_t>(staged, 1), s));
    // The staged particles as slots too, for evaluations over copies of the
    // positions and momenta in slot order.
    if (member)
      LCHECK(dev_reserve(out.stage_slot, sizeof(int32_t) * std::max<int64_t>(staged, 1), s));
    k_tile_fill<false><<<grid, threads, code_bytes, s>>>(
        spans, nb, member, slot_of, sptr, source,
        w.tile_soff.as<int32_t>(), ecap, nullptr, out.desc.as<int32_t>(),
        out.stage.as<int32_t>(), member ? out.stage_slot.as<int32_t>() : nullptr,
        out.local.as<uint16_t>(), stats);
    LTRY(hipGetLastError(), "tile fill kernel");
    out.stage_stride = 0;
  }
  out.cut = false;
  out.bank_rows = false;
  out.bank_lanes = out.bank_unroll = 0;
  out.longest = h[3];
  out.tile_particles = T;
  out.blocks = nb;
  out.staged = staged;
  out.max_stage = h[1];
  out.lds_bytes = h[2];
  return LJGPU_OK;
}

// The slices of `local` in `sliced` (k_tile_slices), lengths and starts from
// plan_slices.
int fill_slices(hipStream_t s, const int32_t* slot_ptr, int32_t lanes, int32_t unroll,
                int32_t scale, bool bank_order, const CutDev* cut, uint16_t* local,
                const DevTiles& t, int32_t wpb, uint16_t* sliced) {
  // Rows an odd number of dwords apart, so that lanes walking one row each
  // read different banks; fewer rows at a time where long ones would not fit.
  const int32_t longest = std::min(std::max(t.longest, 2), kBankRowMax);
  const int32_t stride = 2 * ((longest + 1) / 2 | 1);
  int32_t grows = kSliceRows;
  size_t rows = 0, order = 0;
  for (;; grows /= 2) {
    rows = (sizeof(uint16_t) * stride * grows + 7) / 8 * 8;
    order = bank_order ? sizeof(OrderLds) * kSliceThreads / 64 : 0;
    if (grows == kSliceRows / 2 || rows + order <= kTileLdsMax) break;
  }
  const size_t pos = cut ? sizeof(double) * 3 * static_cast<size_t>(t.max_stage) : 0;
  const bool pos_lds = rows + pos <= kTileLdsMax;
  auto kernel = !bank_order ? k_tile_slices<false, false, false>
                : !cut      ? k_tile_slices<false, false, true>
                : pos_lds   ? k_tile_slices<true, true, true>
                            : k_tile_slices<true, false, true>;
  kernel<<<std::min(t.blocks, 65535), kSliceThreads, rows + std::max(order, pos_lds ? pos : 0), s>>>(
      t.desc.as<int32_t>(), t.blocks, slot_ptr, t.cut || cut ? t.inner.as<int32_t>() : nullptr,
      local, cut ? *cut : CutDev{}, grows, stride, lanes, wpb, scale, slice_pad(unroll),
      t.wave_off.as<int32_t>(), sliced);
  LTRY(hipGetLastError(), "tile slice kernel");
  return LJGPU_OK;
}

int dev_slice_tiles(hipStream_t s, const int32_t* slot_ptr, int32_t lanes, int32_t unroll,
                    int32_t scale, bool bank_order, int32_t n, const CutHint* hint, ListWork& w,
                    DevTiles& t) {
  t.sliced_lanes = t.sliced_unroll = t.waves_per_block = 0;
  t.bank_lanes = t.bank_unroll = 0;
  if (t.blocks <= 0) return LJGPU_OK;
  int32_t wpb = 0;
  LCHECK(plan_slices(s, TileSpans{t.desc.as<int32_t>(), 0, 0, 8}, t.blocks, t.tile_particles,
                     slot_ptr, lanes, unroll, t.longest, w, t, &wpb));
  if (wpb == 0) return LJGPU_OK;
  CutDev cd{};
  const bool cut = bank_order && hint && hint->q.x && !t.cut;
  if (cut) {
    cd.q = hint->q;
    cd.stage = t.stage.as<int32_t>();
    cd.member = t.order == LJGPU_TILE_ORDER_SPATIAL ? t.member.as<int32_t>() : nullptr;
    cd.box = hint->box;
    cd.rep_box = hint->rep_box;
    cd.cl2 = hint->cl2;
    LCHECK(dev_reserve(t.inner, sizeof(int32_t) * n, s));
  }
  LCHECK(fill_slices(s, slot_ptr, lanes, unroll, scale, bank_order, cut ? &cd : nullptr,
                     t.local.as<uint16_t>(), t, wpb, t.sliced.as<uint16_t>()));
  if (cut) t.cut = true;
  t.sliced_lanes = lanes;
  t.sliced_unroll = unroll;
  t.waves_per_block = wpb;
  return LJGPU_OK;
}

int dev_half_tiles(hipStream_t s, int32_t n, ListWork& w, DevTiles& t) {
  t.half_ready = false;
  if (t.blocks <= 0) return LJGPU_OK;
  const int32_t nb = t.blocks;
  LCHECK(dev_reserve(w.tile_ns, sizeof(int32_t) * (static_cast<size_t>(nb) + 1), s));
  LCHECK(dev_reserve(w.tile_soff, sizeof(int32_t) * (static_cast<size_t>(nb) + 1), s));
  LCHECK(dev_reserve(w.counts, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  LCHECK(dev_reserve(t.half_tile, sizeof(int2) * static_cast<size_t>(nb), s));
  LCHECK(dev_reserve(t.half_first, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  const int32_t* desc = t.desc.as<int32_t>();
  const int32_t* keys = t.order == LJGPU_TILE_ORDER_SPATIAL ? t.stage_slot.as<int32_t>()
                                                            : t.stage.as<int32_t>();
  int32_t* count = w.counts.as<int32_t>();
  int32_t* first = t.half_first.as<int32_t>();
  k_half_counts<<<grid_for(nb, kBlock), kBlock, 0, s>>>(nb, desc, w.tile_ns.as<int32_t>());
  LTRY(hipGetLastError(), "half tile count kernel");
  const int64_t total = t.staged;
  if (total > INT32_MAX) return set_error(LJGPU_ERR_CAPACITY, "half list: too many staged partners");
  LCHECK(dev_scan_async(s, w.tile_ns.as<int32_t>(), w.tile_soff.as<int32_t>(), nb, w, nullptr));
  LCHECK(dev_reserve(t.half_at, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  LCHECK(dev_reserve(t.half_part, sizeof(double) * 3 * std::max<int64_t>(total, 1), s));
  const int grid = std::min(nb, 65535);
  LCHECK(fill<int32_t>(s, count, n, 0));
  k_half_places<<<grid, kBlock, 0, s>>>(nb, desc, keys, w.tile_soff.as<int32_t>(),
                                        t.half_tile.as<int2>(), count);
  LTRY(hipGetLastError(), "half tile place kernel");
  LCHECK(dev_scan_async(s, count, first, n, w, nullptr));
  LCHECK(fill<int32_t>(s, count, n, 0));
  k_half_fill<<<grid, kBlock, 0, s>>>(nb, desc, keys, w.tile_soff.as<int32_t>(), first, count,
                                      t.half_at.as<int32_t>());
  k_half_sort<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(n, first, t.half_at.as<int32_t>());
  LTRY(hipGetLastError(), "half tile fill kernels");
  t.half_ready = true;
  return LJGPU_OK;
}

// ListWork::tmp between builds: the rows with their padding, then the slices, whose
// wavefront loads are 128-byte lines (256-byte places: one Kahan evaluation of
// 4,000,000 particles 0.61 ms, off the lines 0.71).
size_t bank_rows_bytes(int64_t e) {
  return (sizeof(uint16_t) * static_cast<size_t>(e + kTileLocalPad) + 255) / 256 * 256;
}
const uint16_t* bank_rows(const ListWork& w) { return w.tmp.as<uint16_t>(); }
const uint16_t* bank_slices(const ListWork& w, int64_t e) {
  return w.tmp.as<uint16_t>() + bank_rows_bytes(e) / sizeof(uint16_t);
}

int bank_room(hipStream_t s, int64_t e, bool slices, ListWork& w, DevTiles& t) {
  const size_t need = bank_rows_bytes(e) + (slices ? sizeof(uint16_t) * t.slice_elems : 0);
  if (w.tmp.p && w.tmp.bytes >= need) return LJGPU_OK;
  t.bank_rows = false;  // the buffer is replaced
  t.bank_lanes = t.bank_unroll = 0;
  return dev_reserve(w.tmp, need, s);
}

int dev_bank_reserve(hipStream_t s, int64_t e, ListWork& w, DevTiles& t) {
  const int rc = bank_room(s, e, true, w, t);
  if (rc != LJGPU_ERR_OUT_OF_MEMORY) return rc;
  (void)hipGetLastError();
  clear_error();
  return LJGPU_OK;
}

int dev_bank_rows(hipStream_t s, const int32_t* slot_ptr, int64_t e, ListWork& w, DevTiles& t) {
  if (t.blocks <= 0 || t.bank_rows) return LJGPU_OK;
  LCHECK(bank_room(s, e, false, w, t));
  uint16_t* rows = w.tmp.as<uint16_t>();
  LTRY(hipMemcpyAsync(rows, t.local.p, sizeof(uint16_t) * (e + kTileLocalPad),
                      hipMemcpyDeviceToDevice, s), "hipMemcpyAsync");
  k_bank_order<<<std::min(t.blocks, 65535), kBankBlock, 0, s>>>(
      t.desc.as<int32_t>(), t.blocks, slot_ptr, t.cut ? t.inner.as<int32_t>() : nullptr, rows);
  LTRY(hipGetLastError(), "tile bank order kernel");
  t.bank_rows = true;
  return LJGPU_OK;
}

int dev_bank_slices(hipStream_t s, const int32_t* slot_ptr, int64_t e, ListWork& w, DevTiles& t) {
  if (t.blocks <= 0 || t.sliced_lanes == 0 ||
      (t.bank_lanes == t.sliced_lanes && t.bank_unroll == t.sliced_unroll))
    return LJGPU_OK;
  LCHECK(bank_room(s, e, true, w, t));
  LCHECK(dev_bank_rows(s, slot_ptr, e, w, t));
  // Lengths and starts of the slices do not depend on the order of a row.
  uint16_t* rows = w.tmp.as<uint16_t>();
  LCHECK(fill_slices(s, slot_ptr, t.sliced_lanes, t.sliced_unroll, 24, false, nullptr, rows, t,
                     t.waves_per_block, rows + bank_rows_bytes(e) / sizeof(uint16_t)));
  t.bank_lanes = t.sliced_lanes;
  t.bank_unroll = t.sliced_unroll;
  return LJGPU_OK;
}

int dev_makepair_batch(hipStream_t s, const PosIn& q, const std::vector<int32_t>& off,
                       const std::vector<double>& boxes, double search_length, int kind,
                       ListWork& w, DevCSR& out) {
  const int32_t nrep = static_cast<int32_t>(off.size()) - 1;
  const int32_t n = off.back();
  out.n = n;
  LCHECK(dev_reserve(out.nop, sizeof(int32_t) * std::max(n, 1), s));
  LCHECK(dev_reserve(out.ptr, sizeof(int32_t) * (static_cast<size_t>(n) + 1), s));
  auto part_of = [&](int32_t r) {
    PosIn qr = q;
    const int64_t shift = static_cast<int64_t>(off[r]) * q.stride;
    qr.x += shift;
    qr.y += shift;
    qr.z += shift;
    return qr;
  };
  // Pass 1: row counts of every replica; pass 2 (after the scan) rebuilds
  // each replica's list and stores it at its place with global indices.
  std::vector<int64_t> e(nrep, 0);
  for (int32_t r = 0; r < nrep; r++) {
    const int32_t nr = off[r + 1] - off[r];
    if (nr == 0) continue;
    LCHECK(dev_makepair(s, part_of(r), nr, boxes[r], search_length, kind, w, w.part));
    e[r] = w.part.e;
    LTRY(hipMemcpyAsync(out.nop.as<int32_t>() + off[r], w.part.nop.p, sizeof(int32_t) * nr,
                        hipMemcpyDeviceToDevice, s), "hipMemcpyAsync");
  }
  int64_t total = 0;
  LCHECK(dev_scan(s, out.nop.as<int32_t>(), out.ptr.as<int32_t>(), n, w, &total));
  if (total > INT32_MAX) return set_error(LJGPU_ERR_CAPACITY, "list longer than 2^31-1 entries");
  out.e = total;
  LCHECK(dev_reserve(out.list, sizeof(int32_t) * std::max<int64_t>(total, 1), s));
  int64_t pos = 0;
  for (int32_t r = 0; r < nrep; r++) {
    const int32_t nr = off[r + 1] - off[r];
    if (nr == 0) continue;
    LCHECK(dev_makepair(s, part_of(r), nr, boxes[r], search_length, kind, w, w.part));
    if (w.part.e != e[r]) return set_error(LJGPU_ERR_HIP, "batched list build: replica changed size");
    if (e[r] > 0) {
      k_copy_add<<<grid_for(e[r], kBlock), kBlock, 0, s>>>(e[r], w.part.list.as<int32_t>(),
                                                           out.list.as<int32_t>() + pos, off[r]);
      LTRY(hipGetLastError(), "copy kernel");
    }
    pos += e[r];
  }
  return LJGPU_OK;
}

int dev_check_replicas(hipStream_t s, const DevCSR& c, const std::vector<int32_t>& off,
                       ListWork& w) {
  if (c.n <= 0) return LJGPU_OK;
  const int32_t nrep = static_cast<int32_t>(off.size()) - 1;
  LCHECK(dev_reserve(w.rep_of, sizeof(int32_t) * c.n, s));
  LCHECK(dev_reserve(w.tile_geo, sizeof(int32_t) * off.size(), s));
  LTRY(hipMemcpyAsync(w.tile_geo.p, off.data(), sizeof(int32_t) * off.size(),
                      hipMemcpyHostToDevice, s), "hipMemcpyAsync");
  k_replica_of<<<grid_for(c.n, kBlock), kBlock, 0, s>>>(c.n, w.tile_geo.as<int32_t>(), nrep,
                                                        w.rep_of.as<int32_t>());
  LCHECK(dev_reserve(w.small, sizeof(int64_t) * 8, s));
  unsigned long long* bad = w.small.as<unsigned long long>();
  LCHECK(fill<unsigned long long>(s, bad, 1, ~0ull));
  k_check_replicas<<<grid_for(c.n, kBlock), kBlock, 0, s>>>(
      c.n, c.nop.as<int32_t>(), c.ptr.as<int32_t>(), c.list.as<int32_t>(), w.rep_of.as<int32_t>(),
      bad);
  LTRY(hipGetLastError(), "replica check kernels");
  unsigned long long h = 0;
  LTRY(hipMemcpyAsync(&h, bad, sizeof(h), hipMemcpyDeviceToHost, s), "hipMemcpyAsync");
  LTRY(hipStreamSynchronize(s), "hipStreamSynchronize");
  if (h == ~0ull) return LJGPU_OK;
  return set_error(LJGPU_ERR_BAD_LIST,
                   "row " + std::to_string(h) + " lists a particle of another replica");
}

}  // namespace ljgpu
