// prims.hip -- device-wide exclusive scan and stable LSD radix sort.
//
// Radix sort: reduce-then-scan with 8-bit digits.  Each block owns a tile of
// 1024 items (256 threads x 4 items, striped so loads are coalesced).  The
// scatter kernel ranks the tile stably in LDS (per-wave digit match via 8
// ballots), sorts it locally, then writes runs of equal digits contiguously.
#include "prims.h"

#include <algorithm>
#include "common.h"

namespace gmpt {

namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;
constexpr size_t kScanDirectTiles = 2048;  // up to this many tiles: two launches per scan

// With range (a device pair lo, hi), entries outside [lo, hi) count as zero
// and are neither read nor written (tiles outside the range touch no memory).
struct ScanRange {
  size_t lo, hi;
  __device__ __forceinline__ ScanRange(const uint32_t *range, size_t n)
      : lo(range ? range[0] : 0), hi(range ? (range[1] < n ? range[1] : n) : n) {}
  __device__ __forceinline__ bool in(size_t j) const { return j >= lo && j < hi; }
};

template <typename T>
__global__ __launch_bounds__(256) void k_scan_reduce(const T *__restrict__ in, size_t n, T *__restrict__ sums,
                                                     const uint32_t *skip, const uint32_t *range) {
  if (skip && *skip) return;  // uniform over the grid
  __shared__ T sh[4];
  const ScanRange rg(range, n);
  size_t base = (size_t)blockIdx.x * kScanTile;
  T acc = 0;
  if (base < rg.hi && base + kScanTile > rg.lo) {
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      size_t j = base + (size_t)i * kScanBlock + threadIdx.x;
      if (rg.in(j)) acc += in[j];
    }
  }
  T tot;
  block_exclusive_scan_256<T>(acc, sh, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Scans one tile; its offset is offsets[blockIdx.x] (already scanned), or,
// with tile_sums, the sum of tile_sums[0 .. blockIdx.x) computed here (used
// when there are few tiles: saves the launch that scans the tile sums).
template <typename T>
__global__ __launch_bounds__(256) void k_scan_down(const T *__restrict__ in, T *__restrict__ out, size_t n,
                                                   const T *__restrict__ offsets, const T *__restrict__ tile_sums,
                                                   T *__restrict__ total, const uint32_t *skip,
                                                   const uint32_t *range) {
  if (skip && *skip) return;  // uniform over the grid
  __shared__ T tile[kScanTile];
  __shared__ T sh[4];
  const ScanRange rg(range, n);
  size_t base = (size_t)blockIdx.x * kScanTile;
  const bool touch = base < rg.hi && base + kScanTile > rg.lo;  // uniform over the block
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    size_t j = base + (size_t)i * kScanBlock + threadIdx.x;
    tile[i * kScanBlock + threadIdx.x] = touch && rg.in(j) ? in[j] : T(0);
  }
  T off = 0;
  if (tile_sums) {
    T part = 0;
    for (uint32_t j = threadIdx.x; j < blockIdx.x; j += kScanBlock) part += tile_sums[j];
    block_exclusive_scan_256<T>(part, sh, &off);
  } else if (offsets) {
    off = offsets[blockIdx.x];
  }
  __syncthreads();
  T v[kScanItems];
  T acc = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    v[i] = tile[threadIdx.x * kScanItems + i];
    acc += v[i];
  }
  T tot;
  T pre = block_exclusive_scan_256<T>(acc, sh, &tot);
  pre += off;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    tile[threadIdx.x * kScanItems + i] = pre;
    pre += v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    size_t j = base + (size_t)i * kScanBlock + threadIdx.x;
    if (touch && rg.in(j)) out[j] = tile[i * kScanBlock + threadIdx.x];
  }
  if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = off + tot;
}

// A scan of at most kScanSmallTiles tiles in one workgroup: each tile as
// k_scan_down scans it, offset by the tiles before (one launch in place of
// the reduce + scan pair).
constexpr size_t kScanSmallTiles = 4;
template <typename T>
__global__ __launch_bounds__(256) void k_scan_small(const T *__restrict__ in, T *__restrict__ out, size_t n,
                                                    T *__restrict__ total, const uint32_t *skip,
                                                    const uint32_t *range, uint32_t ntiles) {
  if (skip && *skip) return;  // uniform over the grid
  __shared__ T tile[kScanTile];
  __shared__ T sh[4];
  const ScanRange rg(range, n);
  T off = 0;
  for (uint32_t b = 0; b < ntiles; b++) {
    const size_t base = (size_t)b * kScanTile;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      const size_t j = base + (size_t)i * kScanBlock + threadIdx.x;
      tile[i * kScanBlock + threadIdx.x] = rg.in(j) ? in[j] : T(0);
    }
    __syncthreads();
    T v[kScanItems];
    T acc = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      v[i] = tile[threadIdx.x * kScanItems + i];
      acc += v[i];
    }
    T tot;
    T pre = block_exclusive_scan_256<T>(acc, sh, &tot) + off;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      tile[threadIdx.x * kScanItems + i] = pre;
      pre += v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      const size_t j = base + (size_t)i * kScanBlock + threadIdx.x;
      if (rg.in(j)) out[j] = tile[i * kScanBlock + threadIdx.x];
    }
    __syncthreads();  // the tile buffer is refilled next
    off += tot;
  }
  if (total && threadIdx.x == 0) *total = off;
}

template <typename T>
size_t scan_temp_elems(size_t n) {
  size_t e = 0;
  while (n > (size_t)kScanTile) {
    n = (n + kScanTile - 1) / kScanTile;
    e += n + 1;
  }
  return e + 1;
}

template <typename T>
hipError_t scan_impl(const T *in, T *out, size_t n, T *total, T *temp, hipStream_t s,
                     const uint32_t *skip = nullptr, const uint32_t *range = nullptr) {
  if (n == 0) {
    if (total) return hipMemsetAsync(total, 0, sizeof(T), s);
    return hipSuccess;
  }
  size_t nb = (n + kScanTile - 1) / kScanTile;
  if (nb <= kScanSmallTiles) {  // one workgroup, tile after tile
    k_scan_small<T><<<1, kScanBlock, 0, s>>>(in, out, n, total, skip, range, (uint32_t)nb);
    return hipGetLastError();
  }
  T *sums = temp;
  T *rest = temp + nb + 1;
  k_scan_reduce<T><<<(unsigned)nb, kScanBlock, 0, s>>>(in, n, sums, skip, range);
  GMPT_LAUNCH_CHECK();
  if (nb <= kScanDirectTiles) {  // each tile adds up the sums before it
    k_scan_down<T><<<(unsigned)nb, kScanBlock, 0, s>>>(in, out, n, nullptr, sums, total, skip, range);
    return hipGetLastError();
  }
  hipError_t e = scan_impl<T>(sums, sums, nb, nullptr, rest, s, skip);
  if (e != hipSuccess) return e;
  k_scan_down<T><<<(unsigned)nb, kScanBlock, 0, s>>>(in, out, n, sums, nullptr, total, skip, range);
  return hipGetLastError();
}

// ------------------------------------------------------------ radix sort --

constexpr int kRsBlock = 256;
constexpr int kRsItems = 4;
constexpr int kRsTile = kRsBlock * kRsItems;
constexpr int kRsWaves = kRsBlock / 64;

// The digit of a pass: eight bits from `shift` on, or, with a mask of the bits
// that vary among the keys (in device memory; 0: not known), the eight highest
// of those.  Keys with constant bits between the varying ones (ASCII digits:
// every other nibble) then fill as many buckets as their values allow.
struct Digit {
  uint64_t m = 0;  // scattered bits to gather, or 0: eight in a row from shift
  int shift;
  __device__ __forceinline__ Digit(int s, const uint64_t *mask) : shift(s) {
    if (mask) {
      uint64_t v = *mask;
      for (uint32_t k = 0; k < 8 && v; k++) {  // the same on every lane
        const uint64_t b = 1ull << (63 - __clzll((long long)v));
        m |= b;
        v ^= b;
      }
      if (m == 0) return;  // not known: the top eight
      const int lo = __ffsll((unsigned long long)m) - 1;
      if (m >> lo == 255) {
        shift = lo;
        m = 0;
      }
    }
  }
  template <typename K>
  __device__ __forceinline__ uint32_t of(K k) const {
    if (m == 0) return (uint32_t)(k >> shift) & 255u;
    uint32_t d = 0;
    for (uint64_t v = m; v;) {
      const int p = 63 - __clzll((long long)v);
      d = d << 1 | ((uint32_t)((uint64_t)k >> p) & 1u);
      v ^= 1ull << p;
    }
    return d;
  }
};

template <typename K>
__global__ __launch_bounds__(256) void k_rs_hist(const K *__restrict__ keys, size_t n, int shift,
                                                 uint32_t *__restrict__ hist, uint32_t nblocks,
                                                 const uint64_t *mask = nullptr) {
  __shared__ uint32_t h[256];
  const Digit digit(shift, mask);
  h[threadIdx.x] = 0;
  __syncthreads();
  size_t base = (size_t)blockIdx.x * kRsTile;
#pragma unroll
  for (int r = 0; r < kRsItems; r++) {
    size_t j = base + (size_t)r * kRsBlock + threadIdx.x;
    if (j < n) atomicAdd(&h[digit.of(keys[j])], 1u);
  }
  __syncthreads();
  hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

template <typename K>
__global__ __launch_bounds__(256) void k_rs_scatter(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                    K *__restrict__ kout, uint32_t *__restrict__ vout, size_t n,
                                                    int shift, const uint32_t *__restrict__ goff,
                                                    uint32_t nblocks, const uint64_t *mask = nullptr) {
  const Digit digit(shift, mask);
  __shared__ uint16_t cnt[kRsItems][kRsWaves][256];
  __shared__ K sk[kRsTile];
  __shared__ uint32_t sv[kRsTile];
  __shared__ uint32_t tstart[256];
  __shared__ uint32_t shs[4];

  const int t = threadIdx.x;
  const int lane = __lane_id();
  const int w = t >> 6;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  size_t base = (size_t)blockIdx.x * kRsTile;

  for (int i = t; i < kRsItems * kRsWaves * 256; i += kRsBlock) (&cnt[0][0][0])[i] = 0;
  __syncthreads();

  K key[kRsItems];
  uint32_t val[kRsItems], dig[kRsItems], wrank[kRsItems];
  bool valid[kRsItems];
#pragma unroll
  for (int r = 0; r < kRsItems; r++) {
    size_t j = base + (size_t)r * kRsBlock + t;
    valid[r] = j < n;
    key[r] = valid[r] ? kin[j] : K(0);
    val[r] = valid[r] ? vin[j] : 0u;
    dig[r] = digit.of(key[r]);
    uint64_t m = __ballot(valid[r]);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      uint64_t bb = __ballot((dig[r] >> b) & 1u);
      m &= ((dig[r] >> b) & 1u) ? bb : ~bb;
    }
    wrank[r] = (uint32_t)__popcll(m & lt_mask);
    // the lowest lane of each digit group records the group's size
    if (valid[r] && (m & lt_mask) == 0) cnt[r][w][dig[r]] = (uint16_t)__popcll(m);
  }
  __syncthreads();
  // per digit: exclusive prefix over (round, wave) in stable order
  {
    const int d = t;
    uint32_t run = 0;
#pragma unroll
    for (int r = 0; r < kRsItems; r++)
#pragma unroll
      for (int ww = 0; ww < kRsWaves; ww++) {
        uint32_t c = cnt[r][ww][d];
        cnt[r][ww][d] = (uint16_t)run;
        run += c;
      }
    uint32_t tot;
    uint32_t st = block_exclusive_scan_256<uint32_t>(run, shs, &tot);
    tstart[d] = st;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRsItems; r++) {
    if (valid[r]) {
      uint32_t pos = tstart[dig[r]] + cnt[r][w][dig[r]] + wrank[r];
      sk[pos] = key[r];
      sv[pos] = val[r];
    }
  }
  __syncthreads();
  size_t valid_n = n - base < (size_t)kRsTile ? n - base : (size_t)kRsTile;
#pragma unroll
  for (int r = 0; r < kRsItems; r++) {
    uint32_t i = r * kRsBlock + t;
    if (i < valid_n) {
      K k = sk[i];
      uint32_t d = digit.of(k);
      size_t dst = (size_t)goff[(size_t)d * nblocks + blockIdx.x] + (i - tstart[d]);
      kout[dst] = k;
      vout[dst] = sv[i];
    }
  }
}

template <typename K>
hipError_t radix_impl(K *k0, uint32_t *v0, K *k1, uint32_t *v1, size_t n, int begin_bit, int end_bit, int *which,
                      void *temp, hipStream_t s) {
  *which = 0;
  if (n <= 1) return hipSuccess;
  uint32_t nb = (uint32_t)((n + kRsTile - 1) / kRsTile);
  uint32_t *hist = (uint32_t *)temp;
  uint32_t *scan_tmp = hist + (size_t)256 * nb + 16;
  K *kin = k0, *kout = k1;
  uint32_t *vin = v0, *vout = v1;
  for (int shift = begin_bit; shift < end_bit; shift += 8) {
    k_rs_hist<K><<<nb, kRsBlock, 0, s>>>(kin, n, shift, hist, nb);
    GMPT_LAUNCH_CHECK();
    hipError_t e = scan_impl<uint32_t>(hist, hist, (size_t)256 * nb, nullptr, scan_tmp, s);
    if (e != hipSuccess) return e;
    k_rs_scatter<K><<<nb, kRsBlock, 0, s>>>(kin, vin, kout, vout, n, shift, hist, nb);
    GMPT_LAUNCH_CHECK();
    K *tk = kin;
    kin = kout;
    kout = tk;
    uint32_t *tv = vin;
    vin = vout;
    vout = tv;
    *which ^= 1;
  }
  return hipSuccess;
}

// One bucket of the first pass per workgroup: bucket d spans
// [goff[d * nblocks], goff[(d + 1) * nblocks]) of the pass's output (the
// exclusive scan of the digit-major per-tile counts), or the whole array
// without goff.  The bucket is counting-sorted in LDS by the 12 highest bits
// that vary among its keys (4,096 sub-buckets: about one entry each for keys
// that spread evenly over those bits' values, constant bits between them or
// not); then each entry counts the entries of its sub-bucket's run that are
// smaller by (key, value), which is its place in the run.  With a run longer
// than kSubMaxRun (a key repeated hundreds of times, keys that share a long
// stretch) the counting would cost its square: the bucket is sorted instead by
// all its varying bits, six at a time from the lowest, stably (it came in
// value order), at about 4 us per six bits.  Only a bucket above kBucketCap
// entries is left as it came, setting bit 1 of *overflow.
constexpr int kBkThreads = 1024;
constexpr uint32_t kBkPer = (uint32_t)(kBucketCap / kBkThreads);  // entries per thread
constexpr uint32_t kBkWaves = kBkThreads / 64;
constexpr uint32_t kSubs = 4096;
constexpr uint32_t kSubPer = kSubs / kBkThreads;                    // sub-buckets per thread
constexpr uint32_t kSubMaxRun = 64;
constexpr uint32_t kLsdBits = 6;
constexpr uint32_t kLsdCnts = (1u << kLsdBits) * kBkPer * kBkWaves;  // a count per digit, round and wave
static_assert(kBucketCap % kBkThreads == 0 && kSubs % kBkThreads == 0, "bucket tiling");
static_assert(kLsdCnts * sizeof(uint16_t) <= kSubs * sizeof(uint32_t) && kLsdCnts == 8 * kBkThreads,
              "the counts fit the sub-bucket starts, eight per thread");

// Exclusive scan of one value per thread over the block.
__device__ __forceinline__ uint32_t bk_scan(uint32_t sum, uint32_t *wsum) {
  const uint32_t t = threadIdx.x, incl = wave_inclusive_scan(sum);
  if (__lane_id() == 63) wsum[t >> 6] = incl;
  __syncthreads();
  uint32_t base = 0;
  for (uint32_t w = 0; w < (t >> 6); w++) base += wsum[w];
  return base + incl - sum;
}

// The c entries (k, v in registers, entry t + q * kBkThreads of the bucket in
// round q) sorted stably by the bits of var, in place.  Every thread of the
// block calls it; the sorted entries end in sk, sv (after its last barrier).
__device__ __forceinline__ void bk_lsd(uint64_t *k, uint32_t *v, uint32_t c, uint64_t var, uint64_t *sk, uint32_t *sv,
                                       uint16_t *cnt, uint32_t *wsum) {
  const uint32_t t = threadIdx.x, lane = __lane_id(), w = t >> 6;
  const uint64_t below = (1ull << lane) - 1;
  do {
    uint64_t m = 0;  // this pass's bits: the lowest left (the same on every lane)
    for (uint32_t j = 0; j < kLsdBits && var; j++) {
      m |= var & (0ull - var);
      var &= var - 1;
    }
    for (uint32_t j = t; j < kLsdCnts / 2; j += kBkThreads) ((uint32_t *)cnt)[j] = 0;
    __syncthreads();
    uint32_t dig[kBkPer], rank[kBkPer];
#pragma unroll
    for (uint32_t q = 0; q < kBkPer; q++) {
      const bool in = t + q * kBkThreads < c;
      uint64_t same = __ballot(in);
      uint32_t d = 0, j = 0;
      for (uint64_t x = m; x; x &= x - 1, j++) {
        const bool bit = in && (k[q] & x & (0ull - x)) != 0;
        const uint64_t bb = __ballot(bit);
        same &= bit ? bb : ~bb;
        d |= (uint32_t)bit << j;
      }
      dig[q] = (d * kBkPer + q) * kBkWaves + w;
      rank[q] = (uint32_t)__popcll(same & below);
      if (in && rank[q] == 0) cnt[dig[q]] = (uint16_t)__popcll(same);
    }
    __syncthreads();
    uint32_t own[8], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
      own[j] = cnt[8 * t + j];
      sum += own[j];
    }
    uint32_t x = bk_scan(sum, wsum);
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
      cnt[8 * t + j] = (uint16_t)x;
      x += own[j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kBkPer; q++)
      if (t + q * kBkThreads < c) {
        const uint32_t p = cnt[dig[q]] + rank[q];
        sk[p] = k[q];
        sv[p] = v[q];
      }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kBkPer; q++)
      if (t + q * kBkThreads < c) {
        k[q] = sk[t + q * kBkThreads];
        v[q] = sv[t + q * kBkThreads];
      }
  } while (var);
}

__global__ __launch_bounds__(1024) void k_bucket_sort(uint64_t *__restrict__ keys, uint32_t *__restrict__ vals,
                                                      uint32_t n, const uint32_t *__restrict__ goff,
                                                      uint32_t nblocks, uint32_t *overflow) {
  __shared__ uint64_t sk[kBucketCap];
  __shared__ uint32_t sv[kBucketCap];
  __shared__ uint32_t start[kSubs + 1];
  __shared__ uint32_t wsum[kBkWaves];
  __shared__ uint64_t wvar[kBkWaves];
  const uint32_t d = blockIdx.x;
  const uint32_t lo = goff ? goff[(size_t)d * nblocks] : 0u;
  const uint32_t hi = goff && d + 1 < 256 ? goff[(size_t)(d + 1) * nblocks] : n;
  const uint32_t c = hi - lo;  // uniform over the block
  if (c <= 1) return;
  if (c > kBucketCap) {
    if (threadIdx.x == 0) atomicOr(overflow, 2u);
    return;
  }
  const uint32_t t = threadIdx.x;
#pragma unroll
  for (uint32_t j = 0; j < kSubPer; j++) start[t + j * kBkThreads] = 0;
  uint64_t k[kBkPer];
  uint32_t v[kBkPer], sub[kBkPer], pos[kBkPer];
  // the bits that vary: those in which some key differs from the first
  const uint64_t k0 = keys[lo];
  uint64_t var = 0;
#pragma unroll
  for (uint32_t q = 0; q < kBkPer; q++) {
    const uint32_t e = t + q * kBkThreads;
    if (e < c) {
      k[q] = keys[lo + e];
      v[q] = vals[lo + e];
      var |= k[q] ^ k0;
    }
  }
  for (int off = 32; off > 0; off >>= 1) var |= (uint64_t)__shfl_xor((unsigned long long)var, off);
  if (__lane_id() == 0) wvar[t >> 6] = var;
  __syncthreads();  // and the counts cleared
  var = 0;
#pragma unroll
  for (uint32_t w = 0; w < kBkWaves; w++) var |= wvar[w];
  // the 12 highest of them (the same on every lane): in a row from sub_shift,
  // as for uniform keys, or gathered
  uint64_t top = 0;
  for (uint32_t j = 0; j < 12 && (var ^ top); j++) top |= 1ull << (63 - __clzll((long long)(var ^ top)));
  const int sub_shift = top ? __ffsll((unsigned long long)top) - 1 : 0;
  const bool row = ((top >> sub_shift) & ((top >> sub_shift) + 1)) == 0;
#pragma unroll
  for (uint32_t q = 0; q < kBkPer; q++) {
    const uint32_t e = t + q * kBkThreads;
    if (e < c) {
      if (row) {
        sub[q] = (uint32_t)((k[q] & top) >> sub_shift);
      } else {
        uint32_t x = 0;
        for (uint64_t m = top; m;) {
          const int p = 63 - __clzll((long long)m);
          x = x << 1 | ((uint32_t)(k[q] >> p) & 1u);
          m ^= 1ull << p;
        }
        sub[q] = x;
      }
      pos[q] = atomicAdd(&start[sub[q]], 1u);
    }
  }
  __syncthreads();
  // exclusive scan of the counts; thread t owns sub-buckets kSubPer t ..
  uint32_t cnt[kSubPer], sum = 0;
#pragma unroll
  for (uint32_t j = 0; j < kSubPer; j++) {
    cnt[j] = start[kSubPer * t + j];
    sum += cnt[j];
  }
  bool long_run = false;
  {
    uint32_t x = bk_scan(sum, wsum);
#pragma unroll
    for (uint32_t j = 0; j < kSubPer; j++) {
      start[kSubPer * t + j] = x;  // only this thread reads or writes these entries here
      x += cnt[j];
      long_run |= cnt[j] > kSubMaxRun;
    }
    if (t + 1 == kBkThreads) start[kSubs] = x;
  }
  if (__syncthreads_or(long_run)) {
    bk_lsd(k, v, c, var, sk, sv, (uint16_t *)start, wsum);
#pragma unroll
    for (uint32_t q = 0; q < kBkPer; q++) {
      const uint32_t e = t + q * kBkThreads;
      if (e < c) {
        keys[lo + e] = k[q];
        vals[lo + e] = v[q];
      }
    }
    return;
  }
#pragma unroll
  for (uint32_t q = 0; q < kBkPer; q++) {
    const uint32_t e = t + q * kBkThreads;
    if (e < c) {
      const uint32_t p = start[sub[q]] + pos[q];
      sk[p] = k[q];
      sv[p] = v[q];
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t q = 0; q < kBkPer; q++) {
    const uint32_t e = t + q * kBkThreads;
    if (e < c) {
      const uint32_t f = start[sub[q]], g = start[sub[q] + 1];
      uint32_t less = 0;
      for (uint32_t p = f; g - f > 1 && p < g; p++) {
        const uint64_t kk = sk[p];
        less += kk < k[q] || (kk == k[q] && sv[p] < v[q]) ? 1u : 0u;
      }
      pos[q] = f + less;
    }
  }
  __syncthreads();  // every run ranked
#pragma unroll
  for (uint32_t q = 0; q < kBkPer; q++) {
    const uint32_t e = t + q * kBkThreads;
    if (e < c) {
      sk[pos[q]] = k[q];
      sv[pos[q]] = v[q];
    }
  }
  __syncthreads();
  for (uint32_t e = t; e < c; e += kBkThreads) {
    keys[lo + e] = sk[e];
    vals[lo + e] = sv[e];
  }
}

}  // namespace

hipError_t bucket_sort_u64(uint64_t *k0, uint32_t *v0, uint64_t *k1, uint32_t *v1, size_t n, int *which, void *temp,
                           hipStream_t s, uint32_t *overflow, const uint64_t *varying) {
  *which = 0;
  if (n <= 1) return hipSuccess;
  if (n > kBucketSortMaxN) return hipErrorInvalidValue;
  if (n <= kBucketCap) {
    k_bucket_sort<<<1, kBkThreads, 0, s>>>(k0, v0, (uint32_t)n, nullptr, 0, overflow);
    return hipGetLastError();
  }
  const uint32_t nb = (uint32_t)((n + kRsTile - 1) / kRsTile);
  uint32_t *hist = (uint32_t *)temp;
  uint32_t *scan_tmp = hist + (size_t)256 * nb + 16;
  k_rs_hist<uint64_t><<<nb, kRsBlock, 0, s>>>(k0, n, 56, hist, nb, varying);
  GMPT_LAUNCH_CHECK();
  hipError_t e = scan_impl<uint32_t>(hist, hist, (size_t)256 * nb, nullptr, scan_tmp, s);
  if (e != hipSuccess) return e;
  k_rs_scatter<uint64_t><<<nb, kRsBlock, 0, s>>>(k0, v0, k1, v1, n, 56, hist, nb, varying);
  GMPT_LAUNCH_CHECK();
  k_bucket_sort<<<256, kBkThreads, 0, s>>>(k1, v1, (uint32_t)n, hist, nb, overflow);
  GMPT_LAUNCH_CHECK();
  *which = 1;
  return hipSuccess;
}

size_t scan_temp_bytes(size_t n) { return scan_temp_elems<uint64_t>(n) * sizeof(uint64_t) + 64; }

size_t radix_temp_bytes(size_t n) {
  size_t nb = (n + kRsTile - 1) / kRsTile + 1;
  return (256 * nb + 16) * sizeof(uint32_t) + scan_temp_bytes(256 * nb) + 256;
}

hipError_t scan_exclusive_u32(const uint32_t *in, uint32_t *out, size_t n, uint32_t *total, void *temp,
                              hipStream_t s) {
  return scan_impl<uint32_t>(in, out, n, total, (uint32_t *)temp, s);
}

hipError_t scan_exclusive_u64(const uint64_t *in, uint64_t *out, size_t n, uint64_t *total, void *temp,
                              hipStream_t s, const uint32_t *skip, const uint32_t *range) {
  return scan_impl<uint64_t>(in, out, n, total, (uint64_t *)temp, s, skip, range);
}

hipError_t radix_sort_u64(uint64_t *k0, uint32_t *v0, uint64_t *k1, uint32_t *v1, size_t n, int begin_bit,
                          int end_bit, int *which, void *temp, hipStream_t s) {
  return radix_impl<uint64_t>(k0, v0, k1, v1, n, begin_bit, end_bit, which, temp, s);
}

hipError_t radix_sort_u32(uint32_t *k0, uint32_t *v0, uint32_t *k1, uint32_t *v1, size_t n, int begin_bit,
                          int end_bit, int *which, void *temp, hipStream_t s) {
  return radix_impl<uint32_t>(k0, v0, k1, v1, n, begin_bit, end_bit, which, temp, s);
}

namespace {
__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
}  // namespace

hipError_t device_copy16(void *dst, const void *src, size_t bytes, hipStream_t s) {
  size_t n16 = bytes / 16;
  if (n16 == 0) return hipSuccess;
  size_t blocks = std::min<size_t>((n16 + 255) / 256, 8192);
  k_copy16<<<(unsigned)blocks, 256, 0, s>>>((const uint4 *)src, (uint4 *)dst, n16);
  return hipGetLastError();
}

}  // namespace gmpt
