// get.hip -- point lookups (gets_parallel) and path node export.
//
// Reference: gets_parallel / get (mpt-with-compress/include/mpt/
// gpu_mpt_kernels.cuh:2267-2340) returns the caller's host pointer recorded at
// insert and the value size; flush_dirty_nodes (gpu_mpt.cuh:1039-1122,
// kernels :2342-2588) exports (hash, encoding) of every node on the given
// keys' paths.

#include "get.h"
#include "phasehc.h"
#include "prims.h"

namespace gmpt {

namespace {

constexpr int kB = 256;
__device__ __forceinline__ uint32_t grid_tid() { return blockIdx.x * blockDim.x + threadIdx.x; }
inline unsigned nblk(size_t n) { return (unsigned)((n + kB - 1) / kB); }

struct HexKey {
  const uint8_t *k;
  uint32_t len;
};

// The key's hex nibbles, or len 0 when its index pair is out of range.
__device__ __forceinline__ HexKey hex_key(const GetArgs &g, uint32_t i) {
  HexKey k;
  int32_t s = g.kidx[2 * i], e = g.kidx[2 * i + 1];
  bool ok = s >= 0 && e >= s && (uint64_t)e < g.kh_bytes;
  k.k = g.kh + (ok ? s : 0);
  k.len = ok ? (uint32_t)(e - s + 1) : 0u;
  return k;
}

// Bytes [0, c) at p (c <= 8), upper bytes zero; reads only the aligned words
// that hold them.
__device__ __forceinline__ uint64_t hex_bytes(const uint8_t *p, uint32_t c) {
  const uintptr_t a = (uintptr_t)p;
  const uint32_t sh = (uint32_t)(a & 7);
  const uint64_t *q = (const uint64_t *)(a - sh);
  uint64_t v = q[0] >> (8 * sh);
  if (sh + c > 8) v |= q[1] << (64 - 8 * sh);
  return c >= 8 ? v : v & ((1ull << (8 * c)) - 1);
}

// 16 hex bytes (h0 first) against the first c nibbles of w: 0 if they agree.
__device__ __forceinline__ uint64_t nibbles_differ(uint64_t w, uint64_t h0, uint64_t h1, uint32_t c) {
  if ((h0 | h1) & 0xF0F0F0F0F0F0F0F0ull) return 1;  // a hex byte above 15 matches nothing
  // bytes 0x0a 0x0b -> one byte 0xab, big-endian nibble order
  uint64_t b0 = __builtin_bswap64(h0), b1 = __builtin_bswap64(h1);
  b0 = (b0 | (b0 >> 4)) & 0x00FF00FF00FF00FFull;
  b1 = (b1 | (b1 >> 4)) & 0x00FF00FF00FF00FFull;
  b0 = (b0 | (b0 >> 8)) & 0x0000FFFF0000FFFFull;
  b1 = (b1 | (b1 >> 8)) & 0x0000FFFF0000FFFFull;
  b0 = (b0 | (b0 >> 16)) & 0xFFFFFFFFull;
  b1 = (b1 | (b1 >> 16)) & 0xFFFFFFFFull;
  const uint64_t x = w ^ (b0 << 32 | b1);
  return c < 16 ? x & ~0ull << (64u - 4u * c) : x;
}

// Nibbles [s, s + m) of the packed key at kp (8-byte aligned) against the m
// hex bytes at h.  The first 64 nibbles' words are all in flight at once, so a
// leaf remainder of ~60 takes one memory round trip (byte by byte it took 60:
// 95 us for 20,000 reads of a 200,000-key trie; a word after the other 24).
__device__ __forceinline__ bool nibbles_equal(const uint8_t *kp, uint32_t s, uint32_t m, const uint8_t *h) {
  if (m == 0) return true;
  // words past the keys' last nibbles are read as the last one instead
  const uint64_t *wk = (const uint64_t *)kp, *wh = (const uint64_t *)((uintptr_t)h & ~(uintptr_t)7);
  const uint32_t ik = s >> 4, ek = (s + m - 1) >> 4, hh = (uint32_t)((uintptr_t)h & 7), eh = (hh + m - 1) >> 3;
  uint64_t a[5], b[9];
#pragma unroll
  for (uint32_t q = 0; q < 5; q++) a[q] = wk[min(ik + q, ek)];
#pragma unroll
  for (uint32_t q = 0; q < 9; q++) b[q] = wh[min(q, eh)];
  const auto hex8 = [&](uint32_t q, uint32_t left) {  // hex bytes 8q .. 8q + 7, the first `left` of them
    uint64_t v = b[q] >> (8 * hh);
    if (hh) v |= b[q + 1] << (64 - 8 * hh);
    return left >= 8 ? v : left ? v & ((1ull << (8 * left)) - 1) : 0ull;
  };
  const uint32_t sh = 4 * (s & 15);
  uint64_t x = 0;
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    uint64_t w = __builtin_bswap64(a[q]) << sh;
    if (sh) w |= __builtin_bswap64(a[q + 1]) >> (64 - sh);
    const uint32_t c = m > 16 * q ? m - 16 * q : 0u;
    if (c) x |= nibbles_differ(w, hex8(2 * q, c), hex8(2 * q + 1, c > 8 ? c - 8 : 0u), c);
  }
  if (x) return false;
  for (uint32_t q = 64; q < m; q += 16) {
    const uint32_t c = min(16u, m - q);
    if (nibbles_differ(nib_word(kp, s + q, s + m), hex_bytes(h + q, min(8u, c)), c > 8 ? hex_bytes(h + q + 8, c - 8) : 0ull, c))
      return false;
  }
  return true;
}

// Walks the key's path; calls visit(ref) for every branch / short node and
// returns the value node reached (REF_NULL when the key is absent).
template <typename F>
__device__ ref_t walk(const Pools &P, ref_t node, HexKey k, F visit) {
  uint32_t pos = 0;
  // the key's hex bytes from a multiple of 16 on, loaded 16 at a time: a branch
  // costs one round trip (its child), not two
  uint64_t b0 = 0, b1 = 0;
  uint32_t at = ~0u;
  for (int guard = 0; guard < 2 * kMaxKeyNibbles + 4; guard++) {
    uint32_t t = ref_type(node);
    if (node == REF_NULL) return REF_NULL;
    if (t == T_VALUE) return pos == k.len ? node : REF_NULL;
    visit(node);
    if (t == T_BRANCH) {
      if (pos >= k.len) return REF_NULL;
      if (pos / 16 != at) {
        at = pos / 16;
        const uint32_t left = k.len - 16 * at;
        b0 = hex_bytes(k.k + 16 * at, min(8u, left));
        b1 = left > 8 ? hex_bytes(k.k + 16 * at + 8, min(8u, left - 8)) : 0ull;
      }
      const uint32_t nib = (uint32_t)((pos & 8 ? b1 : b0) >> (8 * (pos & 7))) & 255u;
      if (nib > 16) return REF_NULL;
      node = P.branch[ref_idx(node)].child[nib];
      pos++;
    } else {
      const Short &S = P.shrt[ref_idx(node)];
      const uint32_t len = S.key_len, term = S.term, real = len - term;
      const ref_t child = S.child;
      if (k.len - pos < len) return REF_NULL;
      if (!nibbles_equal(P.keys + S.key_off, S.key_start, real, k.k + pos)) return REF_NULL;
      if (term && k.k[pos + real] != kNibbleT) return REF_NULL;
      pos += len;
      node = child;
    }
  }
  return REF_NULL;
}

// Threads per block of a walk: some ten thousand keys go a wave per block, so
// that more CUs share their loads.
inline unsigned walk_threads(uint32_t n) { return n <= 65536 ? 64 : kB; }

__global__ __launch_bounds__(256) void k_gets(GetArgs g) {
  uint32_t i = grid_tid();
  if (i >= g.n) return;
  HexKey k = hex_key(g, i);
  uint32_t t = g.tid ? (uint32_t)g.tid[i] : 0u;
  ref_t v = REF_NULL;
  if (t < g.ntries && k.len > 0) v = walk(g.P, g.P.tries[t].root, k, [](ref_t) {});
  if (v == REF_NULL) {
    g.hp[i] = 0;
    g.addr[i] = 0;
    g.size[i] = -1;
  } else {
    const Value &V = g.P.value[ref_idx(v)];
    g.hp[i] = V.hp;
    g.addr[i] = V.addr;
    g.size[i] = (int32_t)V.size;
  }
}

__global__ __launch_bounds__(256) void k_gather_values(const uint64_t *addr, const int32_t *size,
                                                       const uint64_t *off, uint32_t n, uint8_t *out) {
  uint32_t i = blockIdx.x;
  if (i >= n || size[i] <= 0) return;
  const uint8_t *src = (const uint8_t *)addr[i];
  for (int32_t q = threadIdx.x; q < size[i]; q += blockDim.x) out[off[i] + q] = src[q];
}

// The nodes on the keys' paths as a bitmap over the pools' slots (branches,
// then short nodes from word branch_words on): their references come out of it
// in order and once each, with no list per key and no sort.  (Counting and
// writing every key's path, a radix sort and a compaction took 17 launches,
// 250 us for 2,000 keys; marking takes one descent, 21 us, and the pass over
// the bitmap of 340,000 slots 8 us.)  The upper levels' bits are set by the
// first keys to arrive: the others see them and issue no atomic.
__global__ __launch_bounds__(256) void k_path_mark(GetArgs g, unsigned long long *map, uint32_t branch_words,
                                                   uint32_t words) {
  uint32_t i = grid_tid();
  if (i >= g.n) return;
  HexKey k = hex_key(g, i);
  uint32_t t = g.tid ? (uint32_t)g.tid[i] : 0u;
  if (t < g.ntries && k.len > 0)
    walk(g.P, g.P.tries[t].root, k, [&](ref_t r) {
      const uint32_t s = ref_idx(r), w = (ref_type(r) == T_SHORT ? branch_words : 0u) + s / 64;
      const unsigned long long bit = 1ull << (s % 64);
      if (w < words && !(__hip_atomic_load(map + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit))
        atomicOr(map + w, bit);
    });
}

__global__ __launch_bounds__(256) void k_mark_count(const uint64_t *map, uint32_t words, uint32_t *bcnt) {
  __shared__ uint32_t sh[4];
  const uint32_t i = grid_tid();
  uint32_t tot;
  (void)block_exclusive_scan_256<uint32_t>(i < words ? (uint32_t)__popcll(map[i]) : 0u, sh, &tot);
  if (threadIdx.x == 0) bcnt[blockIdx.x] = tot;
}

// bcnt holds the exclusive scan of the blocks' counts.  The map is left clear.
__global__ __launch_bounds__(256) void k_mark_emit(uint64_t *map, uint32_t words, uint32_t branch_words,
                                                   const uint32_t *bcnt, ref_t *out) {
  __shared__ uint32_t sh[4];
  const uint32_t i = grid_tid();
  uint64_t m = i < words ? map[i] : 0ull;
  if (m) map[i] = 0;
  uint32_t tot;
  uint32_t o = bcnt[blockIdx.x] + block_exclusive_scan_256<uint32_t>((uint32_t)__popcll(m), sh, &tot);
  const bool branch = i < branch_words;
  const uint32_t type = branch ? T_BRANCH : T_SHORT, s0 = 64 * (branch ? i : i - branch_words);
  for (; m; m &= m - 1) out[o++] = make_ref(type, s0 + (uint32_t)__ffsll((unsigned long long)m) - 1);
}

}  // namespace

hipError_t launch_gets(const GetArgs &g, hipStream_t s) {
  if (g.n == 0) return hipSuccess;
  const unsigned th = walk_threads(g.n);
  k_gets<<<(g.n + th - 1) / th, th, 0, s>>>(g);
  return hipGetLastError();
}

hipError_t launch_gather_values(const uint64_t *addr, const int32_t *size, const uint64_t *off, uint32_t n,
                                uint8_t *out, hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_gather_values<<<n, 128, 0, s>>>(addr, size, off, n, out);
  return hipGetLastError();
}

hipError_t path_mark(const GetArgs &g, uint64_t *map, uint32_t words, uint32_t branch_words, uint32_t *bcnt,
                     uint32_t *total, void *temp, hipStream_t s) {
  if (g.n == 0 || words == 0) return hipErrorInvalidValue;
  const unsigned th = walk_threads(g.n);
  k_path_mark<<<(g.n + th - 1) / th, th, 0, s>>>(g, (unsigned long long *)map, branch_words, words);
  GMPT_LAUNCH_CHECK();
  k_mark_count<<<nblk(words), kB, 0, s>>>(map, words, bcnt);
  GMPT_LAUNCH_CHECK();
  return scan_exclusive_u32(bcnt, bcnt, nblk(words), total, temp, s);
}

hipError_t mark_emit(uint64_t *map, uint32_t words, uint32_t branch_words, const uint32_t *bcnt, ref_t *out,
                     hipStream_t s) {
  k_mark_emit<<<nblk(words), kB, 0, s>>>(map, words, branch_words, bcnt, out);
  return hipGetLastError();
}

namespace {

__global__ __launch_bounds__(256) void k_rw_mark(const uint8_t *flags, uint32_t n, uint32_t *isr, uint32_t *err) {
  uint32_t i = grid_tid();
  if (i >= n) return;
  uint8_t f = flags[i];
  if (f > 1) atomicCAS(err, 0u, (uint32_t)ERR_BAD_KEY);
  isr[i] = f == 0 ? 1u : 0u;
}

__global__ __launch_bounds__(256) void k_rw_scatter(const uint8_t *flags, uint32_t n, const int32_t *kidx,
                                                    const int64_t *vidx, const uint64_t *hps, const int32_t *tid,
                                                    const uint32_t *pos, int32_t *rk, int32_t *rtid, int32_t *wk,
                                                    int64_t *wv, uint64_t *whp, int32_t *wtid) {
  uint32_t i = grid_tid();
  if (i >= n) return;
  uint32_t r = pos[i];
  if (flags[i] == 0) {
    rk[2 * r] = kidx[2 * i];
    rk[2 * r + 1] = kidx[2 * i + 1];
    if (tid) rtid[r] = tid[i];
  } else {
    uint32_t w = i - r;
    wk[2 * w] = kidx[2 * i];
    wk[2 * w + 1] = kidx[2 * i + 1];
    wv[2 * w] = vidx[2 * i];
    wv[2 * w + 1] = vidx[2 * i + 1];
    if (hps) whp[w] = hps[i];
    if (tid) wtid[w] = tid[i];
  }
}

}  // namespace

hipError_t rw_split(const uint8_t *flags, uint32_t n, const int32_t *kidx, const int64_t *vidx, const uint64_t *hps,
                    const int32_t *tid, uint32_t *isr, uint32_t *pos, uint32_t *nread, int32_t *rk, int32_t *rtid,
                    int32_t *wk, int64_t *wv, uint64_t *whp, int32_t *wtid, uint32_t *err, void *temp,
                    hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_rw_mark<<<nblk(n), kB, 0, s>>>(flags, n, isr, err);
  GMPT_LAUNCH_CHECK();
  hipError_t e = scan_exclusive_u32(isr, pos, n, nread, temp, s);
  if (e != hipSuccess) return e;
  k_rw_scatter<<<nblk(n), kB, 0, s>>>(flags, n, kidx, vidx, hps, tid, pos, rk, rtid, wk, wv, whp, wtid);
  return hipGetLastError();
}

}  // namespace gmpt
