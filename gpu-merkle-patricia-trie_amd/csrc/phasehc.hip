// phasehc.hip -- PhaseHC: bottom-up one-pass hashing of the dirty nodes.
//
// Reference: hash_onepass_v2 (mpt-with-compress/include/mpt/gpu_mpt.cuh:1162-1191)
// counts children per node (mark phase, gpu_mpt_kernels.cuh:2696-2728) and
// lets the last-arriving warp encode and hash each node (update phase,
// :2885-3241).  Here every dirty node carries its nibble depth, so the hash
// order is fixed without counters: all leaf short nodes first (they depend on
// nothing), then non-leaf nodes by decreasing depth (a child is always deeper
// than its parent).  Nodes are binned by (level, estimated Keccak blocks), so
// the lanes of a wave run similar numbers of permutations.
//
// Per level two kernels run:
//  - encode: one thread per node writes the node's RLP encoding, Keccak
//    padding included, into its slot of an HBM scratch buffer (slot sizes are
//    the binning's upper bound).  An encoding shorter than 32 bytes becomes
//    the node's "hash" directly.  The kernel holds few registers, so many
//    waves overlap the pointer chasing to children and values.
//  - permute: Keccak-f[1600] over the slots.  Large levels keep one 25-word
//    state per GPU lane (VGPRs, no communication); small levels are latency
//    bound, so there one state is spread over a wave (40 lanes, a plane per
//    8-lane half-row) and theta, pi and chi exchange words across lanes.
//
// Node encoding follows the reference's encoders exactly
// (FullNode::encode node.cuh:414-452, ShortNode::encode node.cuh:526-559,
// rlp.cuh:118-155): every child is written with write_bytes, i.e. a child
// whose encoding is shorter than 32 bytes is string-wrapped (not inlined),
// a value node contributes its raw bytes, and a node whose own encoding is
// shorter than 32 bytes keeps the raw encoding instead of a digest.
#include "phasehc.h"

#include <algorithm>

#include "hc_leaf.h"
#include "keccak.h"
#include "prims.h"

namespace gmpt {

namespace {

constexpr int kB = 256;
constexpr uint32_t kHcTile = 2048;  // dirty nodes per binning block

__device__ __forceinline__ uint32_t grid_tid() { return blockIdx.x * blockDim.x + threadIdx.x; }
inline unsigned nblk(size_t n) { return (unsigned)((n + kB - 1) / kB); }


// header bytes packed little-endian into a u64 (first byte lowest)
__device__ __forceinline__ uint64_t rlp_hdr(uint32_t L, uint32_t small, uint32_t large, uint32_t *n) {
  if (L < 56) {
    *n = 1;
    return small + L;
  }
  uint32_t nb = be_bytes(L);
  uint64_t h = large + nb;
  for (uint32_t q = 0; q < nb; q++) h |= (uint64_t)((L >> (8 * (nb - 1 - q))) & 255u) << (8 * (q + 1));
  *n = nb + 1;
  return h;
}


// ---------------------------------------------------------- classification --

// Keccak blocks of a node's message, bounded from above before its children
// are hashed: a hashed child counts as a 32-byte digest, and an embedded
// child (encoding < 32 bytes) is never longer than that.
__device__ uint32_t estimate_blocks(const Pools &P, ref_t r, bool *leaf) {
  uint32_t t = ref_type(r), i = ref_idx(r);
  uint32_t len;
  *leaf = false;
  if (t == T_SHORT) {
    const Short &S = P.shrt[i];
    if (ref_type(S.child) == T_VALUE) {
      *leaf = true;
      return leaf_blocks((uint32_t)S.key_len - S.term, P.value[ref_idx(S.child)].size);
    }
    const uint32_t pay = rlp_item_len(((uint32_t)S.key_len - S.term) / 2 + 1, 0) + 33;
    len = rlp_hdr_len(pay) + pay;
  } else {
    const Branch &B = P.branch[i];
    uint32_t pay = 0;
#pragma unroll
    for (int s = 0; s < 17; s++) {
      ref_t c = B.child[s];
      if (c == REF_NULL)
        pay += 1;
      else if (ref_type(c) == T_VALUE)
        pay += rlp_item_len(P.value[ref_idx(c)].size, 0x80);
      else
        pay += 33;
    }
    len = rlp_hdr_len(pay) + pay;
  }
  return keccak_blocks(len);
}

// Inner nodes have at most 5 blocks, so an inner level's last class is free
// for the extensions k_hc_ext_direct hashes: a short node over a branch with
// a key of 1 .. 64 nibbles.
constexpr uint32_t kExtClass = kHcClasses - 1;
__device__ __forceinline__ bool is_direct_ext(const Short &S) {
  return !S.term && ref_type(S.child) == T_BRANCH && S.key_len >= 1 && S.key_len <= kLeafFastNibbles;
}

__device__ __forceinline__ uint32_t bin_of(const Pools &P, ref_t r, uint32_t *blocks) {
  bool leaf;
  uint32_t nb = estimate_blocks(P, r, &leaf);
  *blocks = nb;
  uint32_t cls = nb > kHcClasses ? kHcClasses - 1 : nb - 1;
  if (!leaf && ref_type(r) == T_SHORT && is_direct_ext(P.shrt[ref_idx(r)])) cls = kExtClass;
  uint32_t level;
  if (leaf) {
    level = 0;
  } else {
    uint32_t depth = ref_type(r) == T_SHORT ? P.shrt[ref_idx(r)].depth : P.branch[ref_idx(r)].depth;
    level = 1 + (kHcMaxDepth - min(depth, (uint32_t)kHcMaxDepth));
  }
  return level * kHcClasses + cls;
}

// Leaf metadata (leaf_meta_words) for the leaf-level kernel, recorded by the
// classification in sorted order so that kernel's loads do not chase
// list -> short -> value.
__device__ __forceinline__ void leaf_meta(const Pools &P, ref_t r, uint64_t *m) {
  const Short &S = P.shrt[ref_idx(r)];
  const Value &V = P.value[ref_idx(S.child)];
  leaf_meta_words(S.key_off, S.key_start, (uint32_t)S.key_len - S.term, S.term, V.size, V.addr, m);
}
// Level 0 holds the leaves k_hc_leaf_direct hashes (key remainder <= 64
// nibbles, value < 16,383 bytes); other leaves go to level 1, which no inner
// node uses (a node at nibble depth 255 cannot exist), and take the encode +
// scratch + permutation kernels.
constexpr uint32_t kLdsLeafBins = kHcClasses;  // the bins of level 0

__global__ __launch_bounds__(256) void k_hc_zero(uint32_t *p, uint32_t n, uint32_t *p2 = nullptr, uint32_t n2 = 0) {
  uint32_t i = grid_tid();
  if (i < n) p[i] = 0;
  if (i < n2) p2[i] = 0;
}

// Counting sort of the dirty list by bin.  The first pass computes each
// entry's bin and block estimate once (pointer chasing) and keeps them packed
// in `packed` (bin | blocks << 12, blocks saturated at 2^20 - 1); counts are
// aggregated per block in LDS so each block issues one global atomic per bin
// it touches (a global atomic per node serialises on the few hot bins).

// A leaf whose key remainder or value is beyond the word builder's reach
// (metadata word m0) needs the generic encoder and a scratch slot.
__device__ __forceinline__ bool leaf_too_long(uint64_t m0) {
  return ((m0 >> 41) & 255u) > kLeafFastNibbles || (m0 >> 50) > kLeafDirectMaxValue;
}

// Each thread takes kHcTile / 256 entries; their list and leaf-record loads
// are issued together before any is used (the block count is kept low for
// the global histogram, so each thread's loads must overlap).
constexpr int kHcPer = (int)(kHcTile / 256);
// `packed` entries: bin | blocks << 12 (saturated at kPackedNbMax), and
// kPackedRecorded for a leaf the last build recorded: its metadata is read
// from the build's records, not from lmeta_tmp.
constexpr uint32_t kPackedRecorded = 1u << 31;

__global__ __launch_bounds__(256) void k_hc_hist(Pools P, const ref_t *__restrict__ list, uint32_t n,
                                                 uint32_t *__restrict__ hist, uint32_t *__restrict__ packed,
                                                 uint64_t *__restrict__ lmeta_tmp, LeafRecords rec) {
  __shared__ uint32_t h[kHcBins];
  for (uint32_t b = threadIdx.x; b < kHcBins; b += blockDim.x) h[b] = 0;
  const uint32_t i0 = blockIdx.x * kHcTile + threadIdx.x;
  ref_t r[kHcPer];
  uint32_t rpk[kHcPer];
#pragma unroll
  for (int q = 0; q < kHcPer; q++) {
    const uint32_t i = i0 + 256u * q;
    const uint32_t ri = i - rec.lo;
    r[q] = i < n ? list[i] : REF_NULL;  // builds leave null holes
    // a leaf the last build created: its bin (level 1 when the word builder
    // cannot take it) and metadata were recorded then
    rpk[q] = i < n && rec.pk && ri < rec.n ? rec.pk[ri] : kLeafPackedNone;
  }
  // a branch the last build created: its bin from the depth and child count
  // recorded then (or kLeafPackedNone: read the node)
  uint32_t bpk[kHcPer];
#pragma unroll
  for (int q = 0; q < kHcPer; q++) {
    const uint32_t i = i0 + 256u * q;
    const uint32_t bi = i - rec.blo;
    bpk[q] = i < n && rec.bdesc && bi < rec.bn ? branch_packed(rec.bdesc[bi]) : kLeafPackedNone;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kHcPer; q++) {
    const uint32_t i = i0 + 256u * q;
    if (i >= n) break;
    uint32_t pk = 0xffffffffu;
    if (r[q] != REF_NULL) {
      uint32_t nb, bin, flag = 0;
      if (rpk[q] != kLeafPackedNone) {
        bin = rpk[q] & 0xfff;
        nb = (rpk[q] >> 12) & kPackedNbMax;
        flag = kPackedRecorded;
        // without the word builder every leaf is hashed at level 0
        if (!lmeta_tmp && bin >= kHcClasses) bin -= kHcClasses;
      } else if (bpk[q] != kLeafPackedNone) {
        bin = bpk[q] & 0xfff;
        nb = (bpk[q] >> 12) & kPackedNbMax;
      } else {
        bin = bin_of(P, r[q], &nb);
        if (lmeta_tmp && bin < kLdsLeafBins) {
          uint64_t *m = lmeta_tmp + 2 * (size_t)i;
          leaf_meta(P, r[q], m);
          if (leaf_too_long(m[0])) bin += kHcClasses;
        }
      }
      atomicAdd(&h[bin], 1u);
      pk = bin | (min(nb, kPackedNbMax) << 12) | flag;
    }
    packed[i] = pk;
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < kHcBins; b += blockDim.x)
    if (h[b]) atomicAdd(&hist[b], h[b]);
}

// Scatters each node to its bin and records its scratch slot size
// (136 bytes per estimated block) at the same sorted position.
__global__ __launch_bounds__(256) void k_hc_scatter(Pools P, const ref_t *__restrict__ list,
                                                    const uint32_t *__restrict__ packed, uint32_t n,
                                                    uint32_t *__restrict__ cursor, ref_t *__restrict__ out,
                                                    uint64_t *__restrict__ slot,
                                                    const uint64_t *__restrict__ lmeta_tmp,
                                                    uint64_t *__restrict__ lmeta, LeafRecords rec, HcMeta *meta) {
  __shared__ uint32_t cnt[kHcBins];
  __shared__ uint32_t base[kHcBins];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // the slot scan's range starts past the level-0 leaves hashed without a slot
    uint32_t lo = 0;
    if (lmeta)
      for (uint32_t c = 0; c < kLdsLeafBins; c++) lo += meta->hist[c];
    meta->slot_lo = lo;
  }
  for (uint32_t b = threadIdx.x; b < kHcBins; b += blockDim.x) cnt[b] = 0;
  __syncthreads();
  constexpr int kPer = kHcTile / 256;
  uint32_t pk[kPer], rank[kPer];
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    uint32_t i = blockIdx.x * kHcTile + q * 256 + threadIdx.x;
    pk[q] = i < n ? packed[i] : 0xffffffffu;
    if (pk[q] != 0xffffffffu) rank[q] = atomicAdd(&cnt[pk[q] & 0xfff], 1u);
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < kHcBins; b += blockDim.x)
    if (cnt[b]) base[b] = atomicAdd(&cursor[b], cnt[b]);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; q++)
    if (pk[q] != 0xffffffffu) {
      uint32_t i = blockIdx.x * kHcTile + q * 256 + threadIdx.x;
      uint32_t pos = base[pk[q] & 0xfff] + rank[q];
      ref_t r = list[i];
      uint32_t nb = (pk[q] >> 12) & kPackedNbMax;
      if (nb == kPackedNbMax) bin_of(P, r, &nb);  // saturated: recompute exactly
      out[pos] = r;
      if (lmeta && (pk[q] & 0xfff) < kLdsLeafBins) {  // hashed by k_hc_leaf_direct: no scratch slot
        const uint64_t *m = (pk[q] & kPackedRecorded) ? rec.meta + 2 * (size_t)(i - rec.lo) : lmeta_tmp + 2 * (size_t)i;
        *(uint4 *)(lmeta + 2 * (size_t)pos) = *(const uint4 *)m;
        nb = 0;
      }
      slot[pos] = 136ull * nb;
    }
}


// ------------------------------------------------------------------ encode --

// Unaligned 8-byte read as aligned loads plus a byte funnel shift.
__device__ __forceinline__ uint64_t load8(const uint8_t *p) {
  uintptr_t a = (uintptr_t)p;
  uint32_t sh = (uint32_t)(a & 7);
  const uint64_t *q = (const uint64_t *)(a - sh);
  uint64_t w0 = q[0];
  if (sh == 0) return w0;
  return (w0 >> (8 * sh)) | (q[1] << (64 - 8 * sh));
}
// The first c (1..7) bytes at p, upper bytes zero; reads only words holding them.
__device__ __forceinline__ uint64_t load_part(const uint8_t *p, uint32_t c) {
  uintptr_t a = (uintptr_t)p;
  uint32_t sh = (uint32_t)(a & 7);
  const uint64_t *q = (const uint64_t *)(a - sh);
  uint64_t v = q[0] >> (8 * sh);
  if (sh + c > 8) v |= q[1] << (64 - 8 * sh);
  return v & ((1ull << (8 * c)) - 1);
}

// Writes a byte stream as aligned little-endian 64-bit words.
struct WordWriter {
  uint64_t *out;
  uint64_t acc = 0;   // pending bytes
  uint32_t accn = 0;  // number of pending bytes (0..7)
  uint32_t nw = 0;    // words written
  __device__ __forceinline__ explicit WordWriter(uint64_t *o) : out(o) {}
  // appends the low n (1..8) bytes of v; v's bytes above n must be zero
  __device__ __forceinline__ void push(uint64_t v, uint32_t n) {
    acc |= v << (8 * accn);
    uint32_t tot = accn + n;
    if (tot >= 8) {
      out[nw++] = acc;
      uint32_t used = 8 - accn;
      acc = used >= 8 ? 0ull : (v >> (8 * used));
      accn = tot - 8;
    } else {
      accn = tot;
    }
  }
  __device__ __forceinline__ void inline_bytes(uint64_t b, uint32_t len) {  // len 1..8
    push(len < 8 ? b & ((1ull << (8 * len)) - 1) : b, len);
  }
  __device__ __forceinline__ void mem_bytes(const uint8_t *src, uint32_t len) {
    for (; len >= 8; len -= 8, src += 8) push(load8(src), 8);
    if (len) push(load_part(src, len), len);
  }
  // write_bytes (rlp.cuh:132-155) of a memory string
  __device__ __forceinline__ void rlp_mem(const uint8_t *src, uint32_t len) {
    if (len == 1 && src[0] <= 0x7f) {
      inline_bytes(src[0], 1);
      return;
    }
    uint32_t hn;
    uint64_t h = rlp_hdr(len, 0x80, 0xB7, &hn);
    inline_bytes(h, hn);
    mem_bytes(src, len);
  }
  // write_bytes of the hex-prefix form (utils.cuh:372-396) of nibbles
  // [s, s + cnt) of a packed key (high nibble first) with the leaf flag term
  __device__ __forceinline__ void rlp_compact(const uint8_t *key, uint32_t s, uint32_t cnt, uint32_t term) {
    uint32_t kc = cnt / 2 + 1;
    uint32_t flag = (term << 5) | ((cnt & 1) << 4) | ((cnt & 1) ? packed_nibble(key, s) : 0u);
    if (kc == 1) {  // a single byte <= 0x3f is written raw
      inline_bytes(flag, 1);
      return;
    }
    uint32_t hn;
    uint64_t h = rlp_hdr(kc, 0x80, 0xB7, &hn);
    inline_bytes(h, hn);
    inline_bytes(flag, 1);
    uint32_t first = s + (cnt & 1);
    uint32_t c = kc - 1;
    if ((first & 1) == 0) {
      mem_bytes(key + first / 2, c);
      return;
    }
    // pairs straddle bytes: out byte i = low nibble of b[i], high nibble of b[i+1]
    const uint8_t *sp = key + first / 2;
    for (; c > 0; sp += 8) {
      uint64_t x = load8(sp), y = load8(sp + 1);
      uint64_t v = ((x << 4) & 0xF0F0F0F0F0F0F0F0ull) | ((y >> 4) & 0x0F0F0F0F0F0F0F0Full);
      uint32_t t = c < 8 ? c : 8;
      if (t < 8) v &= (1ull << (8 * t)) - 1;
      push(v, t);
      c -= t;
    }
  }
  // Keccak padding (0x01 after the message, 0x80 in the last byte of the
  // last block) and zero fill up to total_words.
  __device__ __forceinline__ void finish_keccak(uint32_t total_words) {
    push(0x01, 1);
    if (nw == total_words) {  // the 0x01 byte was the last byte of the block
      out[total_words - 1] |= 0x80ull << 56;
      return;
    }
    for (uint32_t w = nw; w < total_words; w++) {
      uint64_t v = w == nw ? acc : 0ull;
      if (w + 1 == total_words) v |= 0x80ull << 56;
      out[w] = v;
    }
  }
  // flush and zero fill up to total_words
  __device__ __forceinline__ void finish_raw(uint32_t total_words) {
    for (uint32_t w = nw; w < total_words; w++) out[w] = w == nw ? acc : 0ull;
  }
};

struct ChildRef {
  const uint8_t *p;
  uint32_t len;
};

__device__ __forceinline__ ChildRef child_bytes(const Pools &P, ref_t c) {
  ChildRef cr;
  uint32_t t = ref_type(c), i = ref_idx(c);
  if (t == T_VALUE) {
    const Value &V = P.value[i];
    cr.p = (const uint8_t *)V.addr;
    cr.len = V.size;
  } else if (t == T_BRANCH) {
    cr.p = P.branch[i].hash;
    cr.len = P.branch[i].hash_size;
  } else {
    cr.p = P.shrt[i].hash;
    cr.len = P.shrt[i].hash_size;
  }
  return cr;
}

__device__ __forceinline__ uint32_t child_item_len(const ChildRef &c) {
  return rlp_item_len(c.len, c.len == 1 ? c.p[0] : 0x80u);
}

// Emits the node's full encoding (list header, then items) into a writer.
template <typename W>
__device__ __forceinline__ void emit_node(const Pools &P, ref_t r, uint32_t payload, W &w) {
  uint32_t hn;
  uint64_t h = rlp_hdr(payload, 0xC0, 0xF7, &hn);
  w.inline_bytes(h, hn);
  if (ref_type(r) == T_SHORT) {
    const Short &S = P.shrt[ref_idx(r)];
    w.rlp_compact(P.keys + S.key_off, S.key_start, S.key_len - S.term, S.term);
    ChildRef c = child_bytes(P, S.child);
    w.rlp_mem(c.p, c.len);
  } else {
    const Branch &B = P.branch[ref_idx(r)];
#pragma unroll
    for (int s = 0; s < 17; s++) {
      ref_t c = B.child[s];
      if (c == REF_NULL) {
        w.inline_bytes(0x80, 1);
      } else {
        ChildRef cb = child_bytes(P, c);
        w.rlp_mem(cb.p, cb.len);
      }
    }
  }
}

__device__ __forceinline__ uint32_t node_payload(const Pools &P, ref_t r) {
  if (ref_type(r) == T_SHORT) {
    const Short &S = P.shrt[ref_idx(r)];
    uint32_t kc = (S.key_len - S.term) / 2 + 1;
    ChildRef c = child_bytes(P, S.child);
    return rlp_item_len(kc, 0) + child_item_len(c);
  }
  const Branch &B = P.branch[ref_idx(r)];
  uint32_t pay = 0;
#pragma unroll
  for (int s = 0; s < 17; s++) {
    ref_t c = B.child[s];
    pay += c == REF_NULL ? 1u : child_item_len(child_bytes(P, c));
  }
  return pay;
}

__device__ __forceinline__ uint8_t *node_hash(const Pools &P, ref_t r) {
  return ref_type(r) == T_SHORT ? P.shrt[ref_idx(r)].hash : P.branch[ref_idx(r)].hash;
}
__device__ __forceinline__ uint32_t node_hash_size(const Pools &P, ref_t r) {
  return ref_type(r) == T_SHORT ? P.shrt[ref_idx(r)].hash_size : P.branch[ref_idx(r)].hash_size;
}
__device__ __forceinline__ void node_done(const Pools &P, ref_t r, uint32_t hs) {
  if (ref_type(r) == T_SHORT) {
    P.shrt[ref_idx(r)].hash_size = (uint8_t)hs;
    P.shrt[ref_idx(r)].dirty = 0;
  } else {
    P.branch[ref_idx(r)].hash_size = (uint8_t)hs;
    P.branch[ref_idx(r)].dirty = 0;
  }
}

// Generic encoder of node r (loads interleaved with stores): enc_len[i], and
// the padded message in out (>= 32 bytes) or the raw encoding as the node's
// "hash" (< 32 bytes, cpu_mpt.cuh:413-418).  Returns the permutations needed.
__device__ __forceinline__ uint32_t encode_generic(const Pools &P, ref_t r, uint64_t *out, uint32_t *enc_out) {
  uint32_t payload = node_payload(P, r);
  uint32_t enc = rlp_hdr_len(payload) + payload;
  *enc_out = enc;
  if (enc < 32) {
    WordWriter w((uint64_t *)node_hash(P, r));
    emit_node(P, r, payload, w);
    w.finish_raw(4);
    node_done(P, r, enc);
    return 0;
  }
  uint32_t nb = keccak_blocks(enc);
  WordWriter w(out);
  emit_node(P, r, payload, w);
  w.finish_keccak(nb * 17);
  return nb;
}

// bytes [off, off + 8) of the little-endian 16-byte pair (a, b), off in 0..7
__device__ __forceinline__ uint64_t funnel8(uint64_t a, uint64_t b, uint32_t off) {
  return off ? (a >> (8 * off)) | (b << (64 - 8 * off)) : a;
}
__device__ __forceinline__ uint64_t low_bytes(uint64_t v, uint32_t n) { return n >= 8 ? v : v & ((1ull << (8 * n)) - 1); }


// Work counters of a hash pass: one reduction over the encoding lengths
// after the last level (per-wave atomics on one counter serialise when waves
// are many).
// (one partial per block: atomics from every block on four counters
// serialise)
__global__ __launch_bounds__(256) void k_hc_count(unsigned long long *parts, const uint32_t *__restrict__ enc_len,
                                                  const uint32_t *__restrict__ nvalid, uint32_t n_leaf) {
  __shared__ unsigned long long sh[4][4];
  const uint32_t n = *nvalid;
  // perms, bytes over all entries; perms, bytes over the leaf entries
  unsigned long long v[4] = {0, 0, 0, 0};
  // four entries per load (enc_len is 16-byte aligned)
  const uint32_t stride = 4 * gridDim.x * blockDim.x;
  for (uint32_t i0 = 4 * grid_tid(); i0 < n; i0 += stride) {
    uint32_t e4[4];
    if (i0 + 4 <= n) {
      const uint4 q = *(const uint4 *)(enc_len + i0);
      e4[0] = q.x, e4[1] = q.y, e4[2] = q.z, e4[3] = q.w;
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) e4[k] = i0 + k < n ? enc_len[i0 + k] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      const uint32_t e = e4[k];
      const uint32_t p = e >= 32 ? keccak_blocks(e) : 0u;
      v[0] += p;
      v[1] += e;
      if (i0 + k < n_leaf) {
        v[2] += p;
        v[3] += e;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++)
    for (int off = 32; off > 0; off >>= 1) v[q] += (unsigned long long)__shfl_xor((long long)v[q], off);
  if (__lane_id() == 0)
#pragma unroll
    for (int q = 0; q < 4; q++) sh[threadIdx.x >> 6][q] = v[q];
  __syncthreads();
  if (threadIdx.x < 4)
    parts[4 * blockIdx.x + threadIdx.x] =
        sh[0][threadIdx.x] + sh[1][threadIdx.x] + sh[2][threadIdx.x] + sh[3][threadIdx.x];
}

// Writes the list header, the compact-key item and the value header (or a
// single raw value byte) of a leaf [compact key, value] from registers into
// `out` as whole little-endian words; the bytes past the head are zero.
__device__ __forceinline__ void leaf_head(uint64_t *out, uint32_t payload, const uint64_t kw[6], uint32_t koff,
                                          uint32_t ks, uint32_t cnt, uint32_t term, uint32_t vsz, bool v_raw,
                                          uint32_t vb0) {
  WordWriter w(out);
  uint32_t hn;
  uint64_t h = rlp_hdr(payload, 0xC0, 0xF7, &hn);
  w.inline_bytes(h, hn);
  const uint32_t kc = cnt / 2 + 1;
  uint64_t b0 = funnel8(kw[0], kw[1], koff);
  uint32_t first_nib = (ks & 1) ? (uint32_t)(b0 & 15) : (uint32_t)((b0 >> 4) & 15);
  uint32_t flag = (term << 5) | ((cnt & 1) << 4) | ((cnt & 1) ? first_nib : 0u);
  if (kc == 1) {
    w.inline_bytes(flag, 1);
  } else {
    w.inline_bytes(0x80 + kc, 1);
    w.inline_bytes(flag, 1);
    const uint32_t first = ks + (cnt & 1);
    const uint32_t d = first / 2 - ks / 2;  // 0 or 1
    uint64_t bs[5];
#pragma unroll
    for (int k = 0; k < 5; k++) bs[k] = funnel8(kw[k], kw[k + 1], koff);
    uint32_t c = kc - 1;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if ((uint32_t)(8 * k) < c) {
        uint64_t v;
        if (first & 1) {  // pairs straddle bytes
          uint64_t x = bs[k], y = (bs[k] >> 8) | (bs[k + 1] << 56);
          v = ((x << 4) & 0xF0F0F0F0F0F0F0F0ull) | ((y >> 4) & 0x0F0F0F0F0F0F0F0Full);
        } else {
          v = d ? (bs[k] >> 8) | (bs[k + 1] << 56) : bs[k];
        }
        uint32_t t = min(8u, c - 8 * k);
        w.push(low_bytes(v, t), t);
      }
    }
  }
  if (v_raw) {
    w.inline_bytes(vb0, 1);
  } else {
    h = rlp_hdr(vsz, 0x80, 0xB7, &hn);
    w.inline_bytes(h, hn);
  }
  if (w.accn) out[w.nw] = w.acc;
}

// Bytes [o, o + 8) of the value at va (vsz bytes), zero outside [0, vsz),
// little-endian; reads only aligned words that hold value bytes.
__device__ __forceinline__ uint64_t value_word(uint64_t va, uint32_t vsz, int64_t o) {
  const int64_t lo = o > 0 ? o : 0, hi = o + 8 < (int64_t)vsz ? o + 8 : (int64_t)vsz;
  if (lo >= hi) return 0ull;
  const uint64_t a_lo = va + (uint64_t)lo;
  const uint64_t *q = (const uint64_t *)(a_lo & ~7ull);
  const uint32_t sh = (uint32_t)(a_lo & 7);
  const uint32_t nbytes = (uint32_t)(hi - lo);
  uint64_t v = q[0] >> (8 * sh);
  if (sh + nbytes > 8) v |= q[1] << (64 - 8 * sh);
  v = low_bytes(v, nbytes);
  return v << (8 * (uint32_t)(lo - o));
}

constexpr uint32_t kLeafGroup = 8;                 // lanes per leaf
constexpr uint32_t kLeafNodes = 256 / kLeafGroup;  // leaves per block
constexpr uint32_t kLeafHeadWords = 6;             // list header + compact key + value header <= 44 bytes
constexpr uint32_t kLeafChunk = 5;                 // message words per lane per load/store round

// Leaf level: 8 lanes per leaf short node [compact key, value] whose key
// remainder has <= 64 nibbles.  Lane s computes message words s, s + 8, ...
// of the padded message -- head bytes, value bytes (two aligned loads per
// word, consecutive across the group) and padding -- and stores them, so the
// group's loads and stores are contiguous and no store waits on a later load.
// Lane 0 builds the head (list header, compact key, value header) in LDS.
// The dependent loads are kept short: the key words are loaded with the value
// node, the value's first byte only for a 1-byte value (which may be raw), and
// the first chunk of value words before the block waits for the heads.
// Other leaves take the generic encoder on lane 0.
__global__ __launch_bounds__(256) void k_hc_encode_leaf(Pools P, const ref_t *__restrict__ list,
                                                        const uint64_t *__restrict__ slot, uint32_t n,
                                                        uint64_t *__restrict__ scratch,
                                                        uint32_t *__restrict__ enc_len) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __shared__ uint64_t head[kLeafNodes][kLeafHeadWords];
  const uint32_t g = threadIdx.x / kLeafGroup, s = threadIdx.x % kLeafGroup;
  const uint32_t i = blockIdx.x * kLeafNodes + g;
  const bool active = i < n;
  const ref_t r = active ? list[i] : REF_NULL;
  uint64_t key_off = 0, va = 0;
  uint32_t ks = 0, cnt = 0, term = 0, vsz = 0;
  ref_t ch = REF_NULL;
  if (active) {
    const Short &S = P.shrt[ref_idx(r)];
    ch = S.child;
    key_off = S.key_off;
    ks = S.key_start;
    cnt = (uint32_t)S.key_len - S.term;
    term = S.term;
  }
  bool fast = ref_type(ch) == T_VALUE && cnt <= kLeafFastNibbles;
  // packed key bytes from byte ks / 2: up to 33 bytes, 6 aligned words
  uint64_t kw[6] = {0, 0, 0, 0, 0, 0};
  uint32_t koff = 0;
  if (fast && s == 0) {
    const uintptr_t ka = (uintptr_t)(P.keys + key_off + ks / 2);
    koff = (uint32_t)(ka & 7);
    const uint64_t *kw_p = (const uint64_t *)(ka - koff);
    const uint32_t kbytes = cnt ? (ks + cnt - 1) / 2 - ks / 2 + 1 : 1;
    const uint32_t nkw = (koff + kbytes + 1 + 7) / 8;
#pragma unroll
    for (int q = 0; q < 6; q++) kw[q] = (uint32_t)q < nkw ? kw_p[q] : 0ull;
  }
  if (fast) {
    const Value &V = P.value[ref_idx(ch)];
    va = V.addr;
    vsz = V.size;
  }
  const uint32_t vb0 = fast && vsz == 1 ? (uint32_t)(value_word(va, 1, 0) & 0xff) : 0u;
  const uint32_t kc = cnt / 2 + 1;
  const uint32_t key_item = kc == 1 ? 1u : 1u + kc;
  const bool v_raw = vsz == 1 && vb0 <= 0x7f;
  const uint32_t vh = v_raw ? 0u : rlp_hdr_len(vsz);
  const uint32_t payload = key_item + (v_raw ? 1u : vh + vsz);
  const uint32_t enc = rlp_hdr_len(payload) + payload;
  fast = fast && enc >= 32;
  const uint32_t nw = fast ? 17 * keccak_blocks(enc) : 0u;
  const uint32_t vstart = enc - vsz;  // message offset of the value bytes (unless raw, in the head)
  // this lane's words in chunks of kLeafChunk: every load of a chunk is
  // issued before its stores (a load after a store waits for the store)
  uint64_t word[kLeafChunk];
  auto chunk = [&](uint32_t w0) {
#pragma unroll
    for (uint32_t q = 0; q < kLeafChunk; q++) {
      const uint32_t w = w0 + q * kLeafGroup, x0 = 8 * w;
      uint64_t v = 0;
      if (w < nw && !v_raw && x0 + 8 > vstart && x0 < enc) v = value_word(va, vsz, (int64_t)x0 - (int64_t)vstart);
      if (enc >= x0 && enc < x0 + 8) v |= 0x01ull << (8 * (enc - x0));  // Keccak padding
      if (w + 1 == nw) v |= 0x80ull << 56;
      word[q] = v;
    }
  };
  chunk(s);
  if (fast && s == 0) {
#pragma unroll
    for (uint32_t q = 0; q < kLeafHeadWords; q++) head[g][q] = 0;
    leaf_head(head[g], payload, kw, koff, ks, cnt, term, vsz, v_raw, vb0);
  }
  __syncthreads();
  if (fast) {
    static_assert(kLeafHeadWords <= kLeafGroup, "head words are in every lane's first word");
    uint64_t *out = scratch + slot[i] / 8;
    if (s < kLeafHeadWords) word[0] |= head[g][s];
    for (uint32_t w0 = s;;) {
#pragma unroll
      for (uint32_t q = 0; q < kLeafChunk; q++)
        if (w0 + q * kLeafGroup < nw) out[w0 + q * kLeafGroup] = word[q];
      w0 += kLeafGroup * kLeafChunk;
      if (w0 >= nw) break;
      chunk(w0);
    }
    if (s == 0) enc_len[i] = enc;
  } else if (active && s == 0) {
    uint32_t e;
    encode_generic(P, r, scratch + slot[i] / 8, &e);
    enc_len[i] = e;
  }
}

// An extension (is_direct_ext) encodes like a leaf whose value is its child's
// hash buffer: [compact key, string of the child's digest, or of its raw
// encoding when that is under 32 bytes].  Fills that leaf's metadata words
// (the string's bytes are read from the child node) and returns true for
// such a node.
__device__ __forceinline__ bool ext_direct_meta(const Pools &P, ref_t r, uint64_t m[2]) {
  if (ref_type(r) != T_SHORT) return false;
  const Short &S = P.shrt[ref_idx(r)];
  if (!is_direct_ext(S)) return false;
  const Branch &B = P.branch[ref_idx(S.child)];
  leaf_meta_words(S.key_off, S.key_start, S.key_len, 0, B.hash_size, (uint64_t)(uintptr_t)B.hash, m);
  return true;
}

constexpr uint32_t kInnerGroup = 16;              // lanes per node (one per nibble slot)
constexpr uint32_t kInnerNodes = 256 / kInnerGroup;
constexpr uint32_t kInnerWords = 80;              // 640 LDS bytes per node >= 4 Keccak blocks

// Encodes inner node r with 16 lanes (s = 0..15 of a 16-lane-aligned segment,
// part = this thread is one of them).  For a branch whose 16 nibble slots hold
// only empty slots and hashed (32-byte) children, and whose slot 16 is empty
// (every branch of fixed-length keys), lane s loads child s's digest, the
// segment prefix-sums the item lengths, each lane writes its item into the
// node's LDS copy of the padded message (lds, kInnerWords words), and the
// segment streams the message words to out.  Other nodes (extension short
// nodes, branches with embedded children or a value) take the generic encoder
// on lane 0.  Every thread of the block calls this (it synchronises the
// block); lane 0 returns the encoding length.  With in_lds, the LDS copy of
// a fast node's message stands (*in_lds set on the segment's lanes) and out
// is not written; the generic encoder still writes out.
__device__ __forceinline__ uint32_t encode_inner_node(const Pools &P, ref_t r, bool active, bool part, uint32_t s,
                                                      uint64_t *lds, uint64_t *out, bool *in_lds = nullptr) {
  const bool is_branch = part && active && ref_type(r) == T_BRANCH;
  ref_t c = REF_NULL, c16 = REF_NULL;
  if (is_branch) {
    const Branch &B = P.branch[ref_idx(r)];
    c = B.child[s];
    c16 = B.child[16];
  }
  const uint32_t ct = ref_type(c);
  const bool node_child = ct == T_BRANCH || ct == T_SHORT;
  uint64_t h[4] = {0, 0, 0, 0};
  uint32_t hs = 0;
  if (node_child) {
    const uint64_t *hp = (const uint64_t *)node_hash(P, c);
#pragma unroll
    for (int q = 0; q < 4; q++) h[q] = hp[q];
    hs = node_hash_size(P, c);
  }
  const bool ok = c == REF_NULL || (node_child && hs == 32);
  const uint64_t bad = __ballot(!ok);
  const uint32_t gbase = __lane_id() & ~(kInnerGroup - 1);
  const bool fast = is_branch && c16 == REF_NULL && ((bad >> gbase) & 0xffffull) == 0;
  if (part) {
#pragma unroll
    for (uint32_t q = 0; q < kInnerWords / kInnerGroup; q++) lds[s + kInnerGroup * q] = 0;
  }
  __syncthreads();
  uint32_t enc = 0, nb = 0;
  if (fast) {
    const uint32_t len = c == REF_NULL ? 1u : 33u;
    uint32_t incl = len;
#pragma unroll
    for (uint32_t d = 1; d < kInnerGroup; d <<= 1) {
      uint32_t t = (uint32_t)__shfl_up((int)incl, d, kInnerGroup);
      if (s >= d) incl += t;
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, kInnerGroup - 1, kInnerGroup);
    const uint32_t payload = total + 1;  // slot 16 is empty: one 0x80 byte
    uint32_t hn;
    const uint64_t hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
    enc = hn + payload;
    nb = keccak_blocks(enc);
    uint8_t *b = (uint8_t *)lds;
    const uint32_t pos = hn + incl - len;
    if (c == REF_NULL) {
      b[pos] = 0x80;
    } else {
      b[pos] = 0xa0;
#pragma unroll
      for (int q = 0; q < 32; q++) b[pos + 1 + q] = (uint8_t)(h[q >> 3] >> (8 * (q & 7)));
    }
    if (s == 0) {
      for (uint32_t q = 0; q < hn; q++) b[q] = (uint8_t)(hdr >> (8 * q));
      b[enc - 1] = 0x80;  // slot 16
      b[enc] = 0x01;      // Keccak padding
      b[136 * nb - 1] |= 0x80;
    }
  }
  __syncthreads();
  if (in_lds) *in_lds = fast;
  if (fast) {
    if (!in_lds)
      for (uint32_t w = s; w < 17 * nb; w += kInnerGroup) out[w] = lds[w];
  } else if (part && active && s == 0) {
    encode_generic(P, r, out, &enc);
  }
  return enc;
}

// Inner levels: 16 lanes per node.
__global__ __launch_bounds__(256) void k_hc_encode_inner(Pools P, const ref_t *__restrict__ list,
                                                         const uint64_t *__restrict__ slot, uint32_t n,
                                                         uint64_t *__restrict__ scratch,
                                                         uint32_t *__restrict__ enc_len) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __shared__ uint64_t lds[kInnerNodes][kInnerWords];
  const uint32_t g = threadIdx.x / kInnerGroup, s = threadIdx.x % kInnerGroup;
  const uint32_t i = blockIdx.x * kInnerNodes + g;
  const bool active = i < n;
  const ref_t r = active ? list[i] : REF_NULL;
  const uint32_t enc = encode_inner_node(P, r, active, true, s, lds[g], active ? scratch + slot[i] / 8 : scratch);
  if (active && s == 0) enc_len[i] = enc;
}

// ----------------------------------------------------------------- permute --

// Sponge over nb padded blocks with one state per lane.
__device__ __forceinline__ void keccak_lane(const uint64_t *m, uint32_t nb, uint64_t s[25]) {
#pragma unroll
  for (int q = 0; q < 25; q++) s[q] = 0;
  for (uint32_t b = 0; b < nb; b++) {
#pragma unroll
    for (int q = 0; q < 17; q++) s[q] ^= m[17 * b + q];
    keccak_f1600(s);
  }
}

// Writes the item 0xa0 + digest (33 bytes; digest words d0, d1 as stored)
// into a zeroed LDS row at byte offset off.  With r = off mod 4 the item
// covers bytes [r, r + 33) of dwords off / 4 + 0 .. 8: dwords 1 .. 7 lie
// inside it and are stored plainly; dwords 0 and 8 may hold a neighbour's
// bytes (the previous or next item, an empty slot's 0x80, the list header)
// and are ORed in, so neighbouring children need no ordering.
__device__ __forceinline__ void or_child_item(uint32_t *row32, uint32_t off, const uint4 &d0, const uint4 &d1) {
  // the item's dwords (byte 0 = 0xa0, bytes 1 .. 32 = the digest)
  uint32_t it[9];
  it[0] = 0xa0u | (d0.x << 8);
  it[1] = __builtin_amdgcn_alignbyte(d0.y, d0.x, 3);
  it[2] = __builtin_amdgcn_alignbyte(d0.z, d0.y, 3);
  it[3] = __builtin_amdgcn_alignbyte(d0.w, d0.z, 3);
  it[4] = __builtin_amdgcn_alignbyte(d1.x, d0.w, 3);
  it[5] = __builtin_amdgcn_alignbyte(d1.y, d1.x, 3);
  it[6] = __builtin_amdgcn_alignbyte(d1.z, d1.y, 3);
  it[7] = __builtin_amdgcn_alignbyte(d1.w, d1.z, 3);
  it[8] = d1.w >> 24;
  const uint32_t r = off & 3u, w0 = off >> 2;
  uint32_t *p = row32 + w0;
  // shifted by r bytes: dword m takes item bytes [4m - r, 4m - r + 4)
#pragma unroll
  for (int m = 0; m < 9; m++) {
    const uint32_t prev = m ? it[m - 1] : 0u;
    const uint32_t v = r ? __builtin_amdgcn_alignbyte(it[m], prev, 4 - r) : it[m];
    if (m == 0 || m == 8)
      atomicOr(p + m, v);
    else
      p[m] = v;
  }
}

// Inner levels above the spread threshold whose nodes are branches of at
// most NB Keccak blocks and extensions (all but a sixteenth of them),
// encoded and hashed in one launch with the messages in LDS: one wave per
// block, one node per lane for the permutation, but the encoding's memory
// work spread over the whole wave:
//  1. Each lane reads its branch's 16 child references (one 64-byte load),
//     keeps them in LDS and writes the bytes that depend on the branch alone
//     into its LDS row: list header, 0x80 for each empty slot, 0x80 for slot
//     16, Keccak padding.  An extension (a short node over a branch) is
//     written whole by its lane: [compact key, 0xa0 + the child's digest].
//  2. The wave's children are dealt out to the lanes: for rows of 1 or 2
//     blocks (a few children per node) the present children, numbered by a
//     prefix sum of the lanes' child counts, round robin; for rows of 4
//     blocks all 64 x 16 (node, slot) pairs, 16 per lane, four at a time so
//     their loads overlap.  Each present child's digest is loaded and ORed,
//     as 0xa0 + digest, into its parent's row at the child's offset (the
//     rank of its slot among the node's present children).
//  3. Each lane absorbs its row and permutes.
// A node whose message would be taller than the rows (NB blocks), a branch
// with a value in slot 16 or an embedded child, and any other short node
// take the generic encoder and their scratch slot.  Blocks run in reverse
// order: the level's nodes are sorted by block count with the extensions
// last, so the larger nodes and extensions start first and finish under the
// bulk.  Entries [skip_lo, skip_hi), the level's nodes taller than the rows
// (classes above NB blocks, before the extensions), are hashed one per block
// by the launch's first nx blocks in the spread layout (hash_spread):
// dispatched first, they run beside the bulk instead of holding the launch
// open after it.
__device__ __forceinline__ void hash_spread(const Pools &P, const ref_t *__restrict__ list,
                                            const uint64_t *__restrict__ slot, uint32_t n,
                                            uint64_t *__restrict__ scratch, uint32_t *__restrict__ enc_len, uint32_t i,
                                            uint64_t *lds);
template <int NB>
struct RowsLds {
  static constexpr uint32_t kStride = 17 * NB + 1;  // words (odd: lane-strided reads spread over the banks)
  static constexpr bool kDense = NB >= 4;           // many children per node: (node, slot) pairs dealt out directly
  uint64_t rows[64 * kStride];
  ref_t cref[kDense ? 64 * 16 : 1];  // the lanes' branches' child references (dense dealing)
  ref_t nref[64];                    // the lanes' nodes
  uint32_t nbase[64];                // first child number of each node (compact dealing)
  uint32_t ninfo[64];                // child mask (0 unless the row path encodes the node) | header length << 16
  uint32_t bad[64];                  // 1: the node takes the generic encoder
};

// An extension's message, [compact key, string of the child's digest d], whole
// into its lane's row, if it takes at most NB blocks.
template <int NB>
__device__ __forceinline__ bool ext_row(const Pools &P, const Short &X, const uint64_t *d, uint64_t *row, uint32_t &enc,
                                        uint32_t &nb) {
  const uint32_t cnt = (uint32_t)X.key_len - X.term;
  const uint32_t payload = rlp_item_len(cnt / 2 + 1, 0) + 33;
  uint32_t hn;
  const uint64_t hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
  if (keccak_blocks(hn + payload) > (uint32_t)NB) return false;
  enc = hn + payload;
  nb = keccak_blocks(enc);
  WordWriter w(row);
  w.inline_bytes(hdr, hn);
  w.rlp_compact(P.keys + X.key_off, X.key_start, cnt, X.term);
  w.inline_bytes(0xa0, 1);
#pragma unroll
  for (int q = 0; q < 4; q++) w.push(d[q], 8);
  w.finish_keccak(17 * nb);
  return true;
}

// Steps 1 and 2 for the wave's nodes, one per lane (r on active lanes): true
// where the lane's row holds its node's message of nb blocks, enc bytes.
// Every lane of the one-wave block calls it (it synchronises the block).
template <int NB>
__device__ __forceinline__ bool rows_encode(const Pools &P, ref_t r, bool active, RowsLds<NB> &S, uint32_t &enc,
                                            uint32_t &nb) {
  constexpr uint32_t RS = RowsLds<NB>::kStride;
  constexpr bool kDense = RowsLds<NB>::kDense;
  const uint32_t lane = threadIdx.x;
  const bool branch = active && ref_type(r) == T_BRANCH;
  bool fast = branch, ext = false;
  uint32_t mask = 0, hn = 0;
  enc = nb = 0;
  uint64_t hdr = 0;
  if (branch) {
    const Branch &B = P.branch[ref_idx(r)];
    const uint4 *cw = (const uint4 *)B.child;  // child[0 .. 15]: 64 bytes, 16-byte aligned
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint4 v = cw[q];
      if (kDense) ((uint4 *)(S.cref + 16 * lane))[q] = v;
      mask |= (v.x != REF_NULL ? 1u : 0u) << (4 * q);
      mask |= (v.y != REF_NULL ? 2u : 0u) << (4 * q);
      mask |= (v.z != REF_NULL ? 4u : 0u) << (4 * q);
      mask |= (v.w != REF_NULL ? 8u : 0u) << (4 * q);
    }
    const uint32_t k = __popc(mask);
    const uint32_t payload = 33 * k + (16 - k) + 1;
    hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
    enc = hn + payload;
    nb = keccak_blocks(enc);
    fast = B.child[16] == REF_NULL && nb <= (uint32_t)NB && enc >= 32;
  } else if (active && ref_type(r) == T_SHORT) {
    ext = is_direct_ext(P.shrt[ref_idx(r)]);
  }
  const uint32_t kc = fast ? (uint32_t)__popc(mask) : 0u;
  const uint32_t incl = wave_inclusive_scan(kc);
  const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);  // the wave's row-path children
  S.nref[lane] = r;
  S.nbase[lane] = incl - kc;
  S.ninfo[lane] = (fast ? mask : 0u) | (hn << 16);
  S.bad[lane] = fast ? 0u : 1u;
  uint64_t *row = S.rows + lane * RS;
  if (fast)
    for (uint32_t w = 0; w < 17 * nb; w++) row[w] = 0;
  __syncthreads();  // rows zeroed; child references, masks visible to the wave
  if (fast) {
    uint8_t *rb = (uint8_t *)row;
    for (uint32_t q = 0; q < hn; q++) rb[q] = (uint8_t)(hdr >> (8 * q));
    uint32_t rank = 0;  // present children below slot s
#pragma unroll
    for (uint32_t s = 0; s < 16; s++) {
      const bool has = (mask >> s) & 1u;
      if (!has) rb[hn + 33 * rank + (s - rank)] = 0x80;
      rank += has ? 1u : 0u;
    }
    rb[enc - 1] = 0x80;  // slot 16: empty
    rb[enc] = 0x01;      // Keccak padding; enc < 136 * nb, so this byte is the message's own
    rb[136 * nb - 1] |= 0x80;
  } else if (ext) {
    const Short &X = P.shrt[ref_idx(r)];
    const Branch &C = P.branch[ref_idx(X.child)];
    uint64_t d[4];
    const uint4 d0 = ((const uint4 *)C.hash)[0], d1 = ((const uint4 *)C.hash)[1];
    d[0] = ((uint64_t)d0.y << 32) | d0.x;
    d[1] = ((uint64_t)d0.w << 32) | d0.z;
    d[2] = ((uint64_t)d1.y << 32) | d1.x;
    d[3] = ((uint64_t)d1.w << 32) | d1.z;
    fast = C.hash_size == 32 && ext_row<NB>(P, X, d, row, enc, nb);
    if (fast) S.bad[lane] = 0;
  }
  if (!kDense) {
    // the wave's present children, numbered node by node, dealt out round
    // robin (a few per lane)
    for (uint32_t t = lane; t < total; t += 64) {
      uint32_t lo = 0, hi = 63;  // the node: the last with S.nbase <= t (it has children)
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) / 2;
        if (S.nbase[mid] <= t)
          lo = mid;
        else
          hi = mid - 1;
      }
      const uint32_t j = lo, info = S.ninfo[j];
      const uint32_t o = t - S.nbase[j];  // the child's rank among the node's present children
      uint32_t mm = info & 0xffffu;     // its slot: the o-th set bit of the mask
      for (uint32_t q = 0; q < o; q++) mm &= mm - 1;
      const uint32_t sl = __ffs(mm) - 1;
      const ref_t c = P.branch[ref_idx(S.nref[j])].child[sl];
      const bool sh = ref_type(c) == T_SHORT;
      const uint8_t *h = sh ? P.shrt[ref_idx(c)].hash : P.branch[ref_idx(c)].hash;
      const uint4 d0 = ((const uint4 *)h)[0], d1 = ((const uint4 *)h)[1];
      const uint32_t hs = sh ? P.shrt[ref_idx(c)].hash_size : P.branch[ref_idx(c)].hash_size;
      if (hs != 32) {
        S.bad[j] = 1;  // an embedded child: the node's own lane encodes it generically
        continue;
      }
      or_child_item((uint32_t *)(S.rows + j * RS), (info >> 16) + 33 * o + (sl - o), d0, d1);
    }
  }
  // (dense) the wave's (node, slot) pairs: pair p = node p / 16, slot p % 16;
  // lane l takes pairs l + 64 q, four at a time so their digest loads overlap
#pragma unroll 1
  for (uint32_t q0 = 0; kDense && q0 < 16; q0 += 4) {
    uint4 d0[4], d1[4];
    uint32_t hs[4], off[4], jj[4];
    bool has[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t p = lane + 64 * (q0 + u);
      const uint32_t j = p >> 4, s = p & 15u;
      const uint32_t info = S.ninfo[j];
      const uint32_t m = info & 0xffffu;
      const uint32_t o = __popc(m & ((1u << s) - 1u));  // the child's rank among the node's present children
      has[u] = (m >> s) & 1u;
      jj[u] = j;
      off[u] = (info >> 16) + 33 * o + (s - o);
      hs[u] = 0;
      d0[u] = d1[u] = make_uint4(0, 0, 0, 0);
      if (has[u]) {
        const ref_t c = S.cref[16 * j + s];
        const bool sh = ref_type(c) == T_SHORT;
        const uint8_t *h = sh ? P.shrt[ref_idx(c)].hash : P.branch[ref_idx(c)].hash;
        d0[u] = ((const uint4 *)h)[0];
        d1[u] = ((const uint4 *)h)[1];
        hs[u] = sh ? P.shrt[ref_idx(c)].hash_size : P.branch[ref_idx(c)].hash_size;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (!has[u]) continue;
      if (hs[u] != 32) {
        S.bad[jj[u]] = 1;  // an embedded child: the node's own lane encodes it generically
        continue;
      }
      or_child_item((uint32_t *)(S.rows + jj[u] * RS), off[u], d0[u], d1[u]);
    }
  }
  __syncthreads();  // every row complete
  return fast && S.bad[lane] == 0;
}

// A digest into its node, and the node clean.
__device__ __forceinline__ void store_digest(const Pools &P, ref_t r, const uint64_t *st) {
  uint64_t *hp = (uint64_t *)node_hash(P, r);
  hp[0] = st[0];
  hp[1] = st[1];
  hp[2] = st[2];
  hp[3] = st[3];
  node_done(P, r, 32);
}

template <int NB>
__global__ __launch_bounds__(64) void k_hc_inner_wave(Pools P, const ref_t *__restrict__ list,
                                                      const uint64_t *__restrict__ slot, uint32_t n,
                                                      uint64_t *__restrict__ scratch, uint32_t *__restrict__ enc_len,
                                                      uint32_t skip_lo, uint32_t skip_hi, uint32_t nx) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __shared__ RowsLds<NB> S;
  static_assert(64 * RowsLds<NB>::kStride >= kInnerWords, "a node's message fits the rows");
  if (blockIdx.x < nx) {  // uniform over the block
    __builtin_amdgcn_s_setprio(2);  // latency-bound waves beside the bulk's permutations
    hash_spread(P, list + skip_lo, slot + skip_lo, skip_hi - skip_lo, scratch, enc_len + skip_lo, blockIdx.x, S.rows);
    return;
  }
  const uint32_t lane = threadIdx.x;
  const uint32_t i = (gridDim.x - 1 - blockIdx.x) * 64 + lane;
  const bool active = i < n && (i < skip_lo || i >= skip_hi);
  const ref_t r = active ? list[i] : REF_NULL;
  uint32_t enc, nb;
  const bool use_row = rows_encode<NB>(P, r, active, S, enc, nb);
  if (!active) return;
  const uint64_t *row = S.rows + lane * RowsLds<NB>::kStride;
  uint64_t *out = scratch + slot[i] / 8;
  if (!use_row) {
    encode_generic(P, r, out, &enc);
    nb = enc >= 32 ? keccak_blocks(enc) : 0u;
  }
  enc_len[i] = enc;
  if (enc < 32) return;  // the raw encoding is the node's "hash", stored by the encoder
  uint64_t st[25];
#pragma unroll
  for (int q = 0; q < 25; q++) st[q] = 0;
  for (uint32_t b = 0; b < nb; b++) {
    if (use_row) {
#pragma unroll
      for (int q = 0; q < 17; q++) st[q] ^= row[17 * b + q];
    } else {
#pragma unroll
      for (int q = 0; q < 17; q++) st[q] ^= out[17 * b + q];
    }
    keccak_f1600(st);
  }
  store_digest(P, r, st);
}

__global__ __launch_bounds__(256) void k_hc_perm_lane(Pools P, const ref_t *list, const uint64_t *slot,
                                                      const uint32_t *enc_len, uint32_t n,
                                                      const uint64_t *scratch) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  uint32_t i = grid_tid();
  if (i >= n) return;
  uint32_t enc = enc_len[i];
  if (enc < 32) return;
  uint64_t s[25];
  keccak_lane(scratch + slot[i] / 8, keccak_blocks(enc), s);
  ref_t r = list[i];
  uint64_t *h = (uint64_t *)node_hash(P, r);
  h[0] = s[0];
  h[1] = s[1];
  h[2] = s[2];
  h[3] = s[3];
  node_done(P, r, 32);
}

// Leaf level 0 (key remainder <= 64 nibbles, value < 16,383 bytes, any
// number of Keccak blocks): encode and hash in one launch, one thread per
// leaf, without a scratch message.  The leaf's
// metadata comes from the classification (leaf_meta, sorted order), so the
// loads are at most two deep; the thread builds the message head (list
// header, compact key, value header) once, then computes each 8-byte message
// word as it absorbs it: head word, value bytes (aligned value words shifted
// by the value's offset in the message and masked to the value's bytes),
// Keccak padding.  The state stays in registers as in k_hc_perm_lane.
// The kernel reads its leaf count (level 0's bins) from the classification
// on the device, so it can be launched before the host has read the bins
// back.  Other leaves are binned at level 1; the only leaves here off the
// word builder's path are those whose encoding is under 32 bytes (raw
// "hash", no permutation).

// Aligned 8-byte load from global memory.
typedef const __attribute__((address_space(1))) uint64_t gword_t;
__device__ __forceinline__ uint64_t gload(uint64_t a) { return *(gword_t *)a; }

// Message layout of a leaf from its metadata word m0 (leaf_meta) and the
// value's first byte (used only for a 1-byte value, which may be raw).
struct LeafLayout {
  uint32_t cnt, vsz, payload, enc, nb;
  bool raw, fast;
};
__device__ __forceinline__ LeafLayout leaf_layout(uint64_t m0, uint32_t vb0) {
  LeafLayout l;
  l.cnt = (uint32_t)(m0 >> 41) & 255u;
  l.vsz = (uint32_t)(m0 >> 50);
  const uint32_t kc = l.cnt / 2 + 1;
  const uint32_t key_item = kc == 1 ? 1u : 1u + kc;
  l.raw = l.vsz == 1 && vb0 <= 0x7f;
  l.payload = key_item + (l.raw ? 1u : rlp_hdr_len(l.vsz) + l.vsz);
  l.enc = rlp_hdr_len(l.payload) + l.payload;
  l.nb = keccak_blocks(l.enc);
  l.fast = l.cnt <= kLeafFastNibbles && l.enc >= 32 && l.vsz <= kLeafDirectMaxValue;
  return l;
}

__device__ __forceinline__ int32_t clamp_i(int32_t x, int32_t lo, int32_t hi) { return max(lo, min(x, hi)); }

// Bytes [sh, sh + 8) of the little-endian 16-byte pair (lo, hi), sh in 0..7.
__device__ __forceinline__ uint64_t funnel_bytes(uint64_t lo, uint64_t hi, uint32_t sh) {
  const uint32_t d0 = (uint32_t)lo, d1 = (uint32_t)(lo >> 32), d2 = (uint32_t)hi, d3 = (uint32_t)(hi >> 32);
  const bool s4 = sh >= 4;
  const uint32_t x = s4 ? d1 : d0, y = s4 ? d2 : d1, z = s4 ? d3 : d2;
  const uint32_t r0 = __builtin_amdgcn_alignbyte(y, x, sh & 3);
  const uint32_t r1 = __builtin_amdgcn_alignbyte(z, y, sh & 3);
  return ((uint64_t)r1 << 32) | r0;
}

// A leaf whose encoding is under 32 bytes: the generic encoder writes the raw
// encoding as its hash.  Returns the encoding length.  Kept out of line: it
// is rare and large.
__device__ __noinline__ uint32_t leaf_raw(const Pools &P, ref_t r) {
  const uint32_t pay = node_payload(P, r);
  const uint32_t e = rlp_hdr_len(pay) + pay;
  if (e >= 32) {  // the binning keeps such leaves out of this kernel
    raise_error(P.cnt, ERR_INTERNAL, 5);
    return e;
  }
  uint32_t enc;
  encode_generic(P, r, nullptr, &enc);
  return enc;
}

constexpr uint32_t kLeafDirectHead = 7;  // LDS words per thread for the head (6 used; odd spreads banks)

// Message words [wlo, whi] that can hold a leaf's string bytes or its 0x01
// padding byte, from its metadata word m0 alone (a superset: the encoding
// length is taken as if the string had a header, the string's start one byte
// earlier than that).
__device__ __forceinline__ void leaf_value_words(uint64_t m0, uint32_t &wlo, uint32_t &whi) {
  const uint32_t cnt = (uint32_t)(m0 >> 41) & 255u, vsz = (uint32_t)(m0 >> 50);
  const uint32_t kc = cnt / 2 + 1;
  const uint32_t payload = (kc == 1 ? 1u : 1u + kc) + rlp_hdr_len(vsz) + vsz;
  const uint32_t enc = rlp_hdr_len(payload) + payload;
  wlo = (enc - vsz - 1) / 8;
  whi = enc / 8;
}

// Encodes and hashes one node shaped [compact key, string] from its metadata
// words m0 (leaf_meta_words) and va (the string's bytes), building each
// message word in registers; hp is the thread's LDS row for the message head.
// Only message words [wlo, whi] (the same on every lane of the wave, and
// covering each lane's leaf_value_words) are built from the string: the
// others hold head bytes or zeros.  Returns the encoding length.
__device__ __forceinline__ uint32_t hash_leaf_shaped(const Pools &P, ref_t r, uint64_t m0, uint64_t va, uint64_t *hp,
                                                     uint32_t wlo = 0, uint32_t whi = 1u << 30) {
  const uint32_t vsz = (uint32_t)(m0 >> 50);
  const uint32_t vb0 = vsz == 1 ? (uint32_t)(gload(va & ~7ull) >> (8 * (va & 7))) & 0xffu : 0u;
  const LeafLayout l = leaf_layout(m0, vb0);
  if (!l.fast) return leaf_raw(P, r);
  const uint32_t enc = l.enc, nb = l.nb;
  uint64_t hw[kLeafHeadWords] = {0, 0, 0, 0, 0, 0};
  {
    const uint64_t ka = (uint64_t)(uintptr_t)P.keys + (m0 & ((1ull << 40) - 1));
    const uint32_t koff = (uint32_t)(ka & 7);
    const uint32_t ks1 = (uint32_t)(m0 >> 40) & 1u, term = (uint32_t)(m0 >> 49) & 1u;
    const uint32_t kbytes = l.cnt ? (ks1 + l.cnt - 1) / 2 + 1 : 1;
    const uint32_t nkw = (koff + kbytes + 1 + 7) / 8;
    uint64_t kw[6];
#pragma unroll
    for (int q = 0; q < 6; q++) kw[q] = (uint32_t)q < nkw ? gload(ka - koff + 8 * q) : 0ull;
#pragma unroll
    for (uint32_t q = 0; q < kLeafHeadWords; q++) hp[q] = 0;
    leaf_head(hp, l.payload, kw, koff, ks1, l.cnt, term, vsz, l.raw, vb0);
#pragma unroll
    for (uint32_t q = 0; q < kLeafHeadWords; q++) hw[q] = hp[q];
  }
  // value geometry: message byte x is value byte x - vstart, i.e. byte
  // x + t0 from the aligned base V0; word w takes aligned words
  // jbase + w and jbase + w + 1 shifted by sh bytes
  const bool hasv = !l.raw && vsz > 0;
  const uint32_t vstart = enc - vsz;
  const uint64_t V0 = va & ~7ull;
  const uint32_t u = (uint32_t)(va & 7);
  const int32_t J = hasv ? (int32_t)((u + vsz - 1) >> 3) : 0;  // last aligned word holding value bytes
  const int32_t t0 = (int32_t)u - (int32_t)vstart;
  const uint32_t sh = (uint32_t)t0 & 7u;
  const int32_t jbase = (t0 - (int32_t)sh) >> 3;
  // the head lies in the first block, on bytes no value byte or padding
  // shares: the state starts as it
  uint64_t st[25];
#pragma unroll
  for (int q = 0; q < 25; q++) st[q] = q < (int)kLeafHeadWords ? hw[q] : 0ull;
#pragma unroll 1
  for (uint32_t b = 0; b < nb; b++) {
    {
      // this block's words of the window (wave-uniform bounds: the word
      // loops below branch over the words outside it)
      const int32_t qlo = max((int32_t)wlo - (int32_t)(17 * b), 0);
      const int32_t qhi = min((int32_t)whi - (int32_t)(17 * b), 16);
      uint64_t W[18];
#pragma unroll
      for (int q = 0; q < 18; q++) {
        W[q] = 0;
        if (q >= qlo && q <= qhi + 1) {
          const int32_t j = clamp_i(jbase + (int32_t)(17 * b) + q, 0, J);  // clamped into the value
          W[q] = hasv ? gload(V0 + 8 * (uint64_t)(uint32_t)j) : 0ull;
        }
      }
#pragma unroll
      for (int q = 0; q < 17; q++) {
        if (q < qlo || q > qhi) continue;
        const int32_t w = 17 * (int32_t)b + q;
        // value bytes: message bytes [max(vstart, 8w), min(enc, 8w + 8)) of this word
        const int32_t lo_b = clamp_i((int32_t)vstart - 8 * w, 0, 8);
        const int32_t hi_b = clamp_i((int32_t)enc - 8 * w, 0, 8);
        const uint64_t f = funnel_bytes(W[q], W[q + 1], sh);
        const uint64_t mk = hasv && hi_b > lo_b ? (~0ull << (8 * lo_b)) & (~0ull >> (64 - 8 * hi_b)) : 0ull;
        uint64_t v = f & mk;
        if ((int32_t)(enc >> 3) == w) v |= 0x01ull << (8 * (enc & 7));  // Keccak padding
        st[q] ^= v;
      }
      if (b + 1 == nb) st[16] ^= 0x80ull << 56;  // the last byte of the last block
    }
    keccak_f1600(st);
  }
  uint64_t *h = (uint64_t *)node_hash(P, r);
  h[0] = st[0];
  h[1] = st[1];
  h[2] = st[2];
  h[3] = st[3];
  node_done(P, r, 32);
  return enc;
}

__global__ __launch_bounds__(256) void k_hc_leaf_direct(Pools P, const ref_t *__restrict__ list,
                                                        const uint64_t *__restrict__ lmeta,
                                                        const uint32_t *__restrict__ hist,
                                                        uint32_t *__restrict__ enc_len) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __shared__ uint64_t head[256][kLeafDirectHead];
  const uint32_t j = grid_tid();
  uint32_t n = 0;  // the leaves of level 0, sorted first
#pragma unroll
  for (uint32_t c = 0; c < kLdsLeafBins; c++) n += hist[c];
  // the leaves from the last: the level is sorted by block count, so the
  // longest leaves start first and the 1-block ones fill the end of the launch
  const bool act = j < n;
  const uint32_t i = act ? n - 1 - j : 0u;
  const uint64_t m0 = act ? lmeta[2 * (size_t)i] : 0ull;
  // the wave's window of string words, reduced while every lane is active
  uint32_t wlo = 0xffffu, whi = 0;
  if (act) leaf_value_words(m0, wlo, whi);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    wlo = min(wlo, (uint32_t)__shfl_xor((int)wlo, off));
    whi = max(whi, (uint32_t)__shfl_xor((int)whi, off));
  }
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  whi = __builtin_amdgcn_readfirstlane(whi);
  if (!act) return;  // no block barrier below
  enc_len[i] = hash_leaf_shaped(P, list[i], m0, lmeta[2 * (size_t)i + 1], head[threadIdx.x], wlo, whi);
}

// The leaf children of list[0 .. n) (inner nodes of the deepest levels),
// one thread per (node, slot): hashed here, on a second stream, so that
// those levels can be hashed beside the leaf-level launch, which hashes the
// same leaves again and stores the same bytes (a reader sees equal old and
// new values).  A child the word builder cannot take is a clean leaf, hashed
// by an earlier pass (the host runs no tail while such a leaf is dirty), and
// is left as it is.
__global__ __launch_bounds__(256) void k_hc_tail_leaves(Pools P, const ref_t *__restrict__ list, uint32_t n) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __builtin_amdgcn_s_setprio(2);  // ahead of the leaf-level launch's waves on a shared SIMD
  __shared__ uint64_t head[256][kLeafDirectHead];
  __shared__ ref_t job[256];
  __shared__ uint32_t sh[4];
  const uint32_t t = grid_tid(), i = t / 16, s = t % 16;
  ref_t leaf = REF_NULL;
  if (i < n) {
    const ref_t r = list[i];
    if (ref_type(r) == T_BRANCH) {  // an extension's child is a branch
      const ref_t c = P.branch[ref_idx(r)].child[s];
      if (ref_type(c) == T_SHORT && ref_type(P.shrt[ref_idx(c)].child) == T_VALUE) leaf = c;
    }
  }
  // the block's leaves packed into its first lanes (a few per node): the
  // waves left without one exit
  uint32_t tot;
  const uint32_t pos = block_exclusive_scan_256<uint32_t>(leaf != REF_NULL ? 1u : 0u, sh, &tot);
  if (leaf != REF_NULL) job[pos] = leaf;
  __syncthreads();
  if (threadIdx.x >= tot) return;  // no block barrier below
  const ref_t c = job[threadIdx.x];
  uint64_t m[2];
  leaf_meta(P, c, m);
  if (leaf_too_long(m[0])) return;  // clean: its hash stands
  (void)hash_leaf_shaped(P, c, m[0], m[1], head[threadIdx.x]);
}

// The extension class of an inner level (kExtClass): each extension encodes
// like a leaf (ext_direct_meta), so the leaf word builder hashes it with no
// scratch message.  A node that is not such an extension (none is binned
// here) would take the generic encoder and its scratch slot.
__global__ __launch_bounds__(256) void k_hc_ext_direct(Pools P, const ref_t *__restrict__ list,
                                                       const uint64_t *__restrict__ slot, uint32_t n,
                                                       uint64_t *__restrict__ scratch,
                                                       uint32_t *__restrict__ enc_len) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  __shared__ uint64_t head[256][kLeafDirectHead];
  const uint32_t i = grid_tid();
  if (i >= n) return;  // no block barrier below
  const ref_t r = list[i];
  uint64_t m[2];
  if (ext_direct_meta(P, r, m)) {
    enc_len[i] = hash_leaf_shaped(P, r, m[0], m[1], head[threadIdx.x]);
    return;
  }
  uint32_t enc;
  uint64_t *msg = scratch + slot[i] / 8;
  encode_generic(P, r, msg, &enc);
  enc_len[i] = enc;
  if (enc < 32) return;
  uint64_t st[25];
  keccak_lane(msg, keccak_blocks(enc), st);
  uint64_t *h = (uint64_t *)node_hash(P, r);
  h[0] = st[0];
  h[1] = st[1];
  h[2] = st[2];
  h[3] = st[3];
  node_done(P, r, 32);
}

// Keccak-f[1600] with one state spread over a wave: lane 8y + p (y < 5) holds
// word A[x, y], x = (p + 4) mod 5, as (l, h) halves; lanes 40 .. 63 hold zero.
// A plane sits in one 8-lane half-row with its ends repeated (p = 0 and 5 hold
// x = 4, p = 1 and 6 x = 0, p = 2 and 7 x = 1), so that a round takes one trip
// through LDS:
//   theta  the column parities by a DPP xor of the half-rows and lane swaps of
//          rows, C[x - 1] and C[x + 1] by DPP from the lanes beside (at
//          p = 1 .. 5, the lanes that are a later source)
//   pi     one gather (ds_bpermute) per half for B[x, y] at every p, one for
//          B[x + 2, y]
//   chi    B[x + 1, y] by DPP from the next lane (at p = 0 .. 6; p = 7 holds
//          anything, and only p = 6 takes anything from it)
// Bound by latency: 2.4 us a permutation on an idle CU, 5.2 with four waves on
// every SIMD.  (A column per half-row, parities and their neighbours gathered
// and all three of chi's operands too, took 3.05 and 10.9: ten gathers a
// round in two trips.)
struct SpreadLane {
  uint32_t ok, iota, flip, t, s0, s2;  // s0, s2: source byte addresses for ds_bpermute
  // pi moves A[x', y'] to B[y', 2x' + 3y']: B[x, y] comes from A[3y + x, x].
  // Lanes 40 .. 63 read themselves, which are zero.
  static __device__ __forceinline__ uint32_t pi_src(uint32_t x, uint32_t y, uint32_t lane) {
    return 4 * (y < 5 ? 8 * x + 1 + (3 * y + x) % 5 : lane);
  }
  __device__ __forceinline__ explicit SpreadLane(uint32_t lane) {
    const uint32_t x = ((lane & 7) + 4) % 5, y = lane >> 3;
    ok = y < 5 ? ~0u : 0u;
    iota = x == 0 && y == 0 ? ~0u : 0u;
    // rho as two funnel shifts by t = (32 - r) mod 32 of the halves, swapped
    // first when flip: rotations by 0 and 32 need no other case
    const uint32_t rho = ok ? (uint32_t)kKeccak.rho[x + 5 * y] : 0u, rr = rho & 31;
    flip = (rho >= 32) != (rr == 0) ? ~0u : 0u;
    t = (32 - rr) & 31;
    s0 = pi_src(x, y, lane);
    s2 = pi_src((x + 2) % 5, y, lane);
  }
  // message word this lane absorbs (x + 5y < 17), or -1
  __device__ __forceinline__ static int word_of(uint32_t lane) {
    const uint32_t w = ((lane & 7) + 4) % 5 + 5 * (lane >> 3);
    return lane < 40 && w < 17 ? (int)w : -1;
  }
  // digest word q is A[q, 0]
  __device__ __forceinline__ static bool digest(uint32_t lane) { return lane - 1 < 4; }
};

__device__ __forceinline__ uint32_t bperm(uint32_t addr, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)addr, (int)v);
}
template <int C>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, C, 0xF, 0xF, true);
}
constexpr int kDppNext = 0x101;  // row_shl 1: the value of lane + 1
constexpr int kDppPrev = 0x111;  // row_shr 1
constexpr int kDppHalf = 0x128;  // row_ror 8: of the row's other half
// a ^ (b & c)
__device__ __forceinline__ uint32_t xor_and(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x78);
}

__device__ __forceinline__ void keccak_spread(uint32_t &l, uint32_t &h, const SpreadLane &c) {
#pragma unroll
  for (int ir = 0; ir < 24; ir++) {
    // theta: A ^= C[x - 1] ^ rotl(C[x + 1], 1).  Both halves' parities in one
    // reduction: after the first swap of 32 lanes the lower lanes hold l's and
    // the upper ones h's, and the last one gives every lane both.
    const auto u = __builtin_amdgcn_permlane32_swap(l ^ dpp<kDppHalf>(l), h ^ dpp<kDppHalf>(h), false, false);
    const uint32_t r = u[0] ^ u[1];
    const auto v = __builtin_amdgcn_permlane16_swap(r, r, false, false);
    const uint32_t q = v[0] ^ v[1];
    const auto p = __builtin_amdgcn_permlane32_swap(q, q, false, false);
    const uint32_t nxl = dpp<kDppNext>(p[0]), nxh = dpp<kDppNext>(p[1]);
    l = xor_and(l, dpp<kDppPrev>(p[0]) ^ __builtin_amdgcn_alignbit(nxl, nxh, 31), c.ok);
    h = xor_and(h, dpp<kDppPrev>(p[1]) ^ __builtin_amdgcn_alignbit(nxh, nxl, 31), c.ok);
    // rho: rotate this lane's word by its own offset
    const uint32_t a = c.flip ? h : l, b = c.flip ? l : h;
    const uint32_t nl = __builtin_amdgcn_alignbit(a, b, c.t);
    const uint32_t nh = __builtin_amdgcn_alignbit(b, a, c.t);
    // pi + chi: B[x, y] ^ (~B[x + 1, y] & B[x + 2, y])
    const uint32_t b0l = bperm(c.s0, nl), b0h = bperm(c.s0, nh);
    const uint32_t b2l = bperm(c.s2, nl), b2h = bperm(c.s2, nh);
    l = chi3(b0l, dpp<kDppNext>(b0l), b2l);
    h = chi3(b0h, dpp<kDppNext>(b0h), b2h);
    // iota (unrolled: the constants are immediates)
    if ((uint32_t)kKeccak.rc[ir]) l = xor_and(l, (uint32_t)kKeccak.rc[ir], c.iota);
    if ((uint32_t)(kKeccak.rc[ir] >> 32)) h = xor_and(h, (uint32_t)(kKeccak.rc[ir] >> 32), c.iota);
  }
}

// Sponge over nb padded blocks, state spread over the wave; every lane must
// call it with the same m and nb.  Digest word q ends on lane q + 1 (q < 4).
__device__ __forceinline__ void sponge_spread(const uint64_t *m, uint32_t nb, uint32_t lane, const SpreadLane &c,
                                              uint32_t &l, uint32_t &h) {
  l = 0;
  h = 0;
  const int w = SpreadLane::word_of(lane);
  for (uint32_t b = 0; b < nb; b++) {
    if (w >= 0) {
      const uint64_t v = m[17 * b + (uint32_t)w];
      l ^= (uint32_t)v;
      h ^= (uint32_t)(v >> 32);
    }
    keccak_spread(l, h, c);
  }
}
__global__ __launch_bounds__(256) void k_hc_perm_spread(Pools P, const ref_t *list, const uint64_t *slot,
                                                        const uint32_t *enc_len, uint32_t n,
                                                        const uint64_t *scratch) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  const uint32_t lane = __lane_id();
  const uint32_t i = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  uint32_t enc = i < n ? enc_len[i] : 0;
  uint32_t nb = enc >= 32 ? keccak_blocks(enc) : 0;  // uniform over the wave
  SpreadLane c(lane);
  uint32_t l, h;
  sponge_spread(nb ? scratch + slot[i] / 8 : scratch, nb, lane, c, l, h);
  if (nb == 0) return;
  ref_t r = list[i];
  if (SpreadLane::digest(lane)) ((uint64_t *)node_hash(P, r))[lane - 1] = ((uint64_t)h << 32) | l;
  if (lane == 0) node_done(P, r, 32);
}

// Node list[i] (if i < n) by one wave: lanes 0..15 encode it
// (encode_inner_node), then the wave runs the sponge with the state spread
// over it, reading the message from the node's LDS copy lds (a generic-encoded
// node's from its scratch slot, which the block barrier makes visible).  Every
// thread of the block calls it (it holds a barrier).
__device__ __forceinline__ void hash_spread(const Pools &P, const ref_t *__restrict__ list,
                                            const uint64_t *__restrict__ slot, uint32_t n,
                                            uint64_t *__restrict__ scratch, uint32_t *__restrict__ enc_len, uint32_t i,
                                            uint64_t *lds) {
  const uint32_t lane = __lane_id();
  const bool active = i < n;
  const ref_t r = active ? list[i] : REF_NULL;
  uint64_t *out = active ? scratch + slot[i] / 8 : scratch;
  bool in_lds = false;
  uint32_t enc = encode_inner_node(P, r, active, lane < kInnerGroup, lane & (kInnerGroup - 1), lds, out, &in_lds);
  enc = (uint32_t)__shfl((int)enc, 0, 64);
  in_lds = __shfl((int)in_lds, 0, 64) != 0;
  if (active && lane == 0) enc_len[i] = enc;
  __syncthreads();  // the node's message words are visible to all its lanes
  const uint32_t nb = active && enc >= 32 ? keccak_blocks(enc) : 0u;  // uniform over the wave
  SpreadLane c(lane);
  uint32_t l, h;
  // a fast node's message stays in LDS (at most 4 blocks: 68 of the 80 words)
  sponge_spread(in_lds ? lds : out, nb, lane, c, l, h);
  if (nb == 0) return;
  if (SpreadLane::digest(lane)) ((uint64_t *)node_hash(P, r))[lane - 1] = ((uint64_t)h << 32) | l;
  if (lane == 0) node_done(P, r, 32);
}

// Small inner levels in one launch, a node per wave.
__global__ __launch_bounds__(256) void k_hc_small(Pools P, const ref_t *__restrict__ list,
                                                  const uint64_t *__restrict__ slot, uint32_t n,
                                                  uint64_t *__restrict__ scratch, uint32_t *__restrict__ enc_len) {
  if (P.cnt->graph_bad) return;  // a replayed pass whose batch is unlike the captured one
  // latency-bound waves: ahead of a concurrent launch's permutations (the
  // leaf level's, or a level's bulk) on a shared SIMD
  __builtin_amdgcn_s_setprio(2);
  __shared__ uint64_t lds[256 / 64][kInnerWords];
  const uint32_t g = threadIdx.x / 64;
  hash_spread(P, list, slot, n, scratch, enc_len, blockIdx.x * (256 / 64) + g, lds[g]);
}

// ------------------------------------------------- small passes: one climb --
//
// A pass over a short dirty list is bound by latency: a classification (five
// launches), a copy of its bins to the host, and one launch per level, each
// waiting for the one before, hash a few hundred nodes in ten times what
// their permutations take.  Such a pass runs as one climb instead:
//   k_tree_link    every dirty node gets its dirty parent (in its own dirty
//                  word) and a branch the number of its dirty children; the
//                  nodes without one are ready
//   k_tree_leaves  (longer lists only) the leaves the word builder takes, one
//                  per lane
//   k_tree_long    (lists that may hold many only) the other leaves, one per
//                  lane while they are many, else ready
//   k_tree_rows    (lists of many inner nodes only, a few launches) while many
//                  nodes are ready, one per lane; those without a row of a few
//                  blocks, and parents that became ready, make the next list
//   k_tree_climb   one wave per ready node hashes it in the spread layout and
//                  counts it off at its parent; the wave that was last goes on
//                  with the parent.  No wave waits for another, and no level
//                  for the slowest node of the one below.
// The host reads nothing back in between.
//
// A dirty word: 1 = dirty without a dirty parent, else 1 | (parent is a short
// node) << 1 | (parent's slot + 1) << 2.
__device__ __forceinline__ uint32_t tree_parent_word(ref_t parent) {
  return 1u | (ref_type(parent) == T_SHORT ? 2u : 0u) | (ref_idx(parent) + 1) << 2;
}

// TreeState::lists: ready entries, leaf entries and listed nodes, 21 bits each
// (one atomic gives a block its place in both lists).
constexpr uint32_t kTreeListBits = 21;
constexpr unsigned long long kTreeListMask = (1ull << kTreeListBits) - 1;
static_assert(kTreeMax < (1u << kTreeListBits), "the lists' counts are packed");

// Words 4 (hash size, depth, dirty) of a branch and 6 (depth, hash size,
// terminator flag, dirty) of a short node.
static_assert(offsetof(Branch, hash_size) == 32 && offsetof(Branch, depth) == 34 && offsetof(Branch, dirty) == 36 &&
                  offsetof(Branch, pad1) == 116,
              "branch words");
static_assert(offsetof(Short, depth) == 48 && offsetof(Short, hash_size) == 50 && offsetof(Short, term) == 51 &&
                  offsetof(Short, dirty) == 52,
              "short node words");

__device__ __forceinline__ unsigned long long tree_reserve(unsigned long long *at, unsigned long long mine,
                                                           uint32_t lane) {
  unsigned long long base = 0;
  if (lane == 0) base = atomicAdd(at, mine);
  return (unsigned long long)__shfl((long long)base, 0);
}

// Entries of ready list k: the links' and leaves' (0), or the ones row launch
// k left.  Row launch k takes list k when it is long enough for lanes (and
// then makes list k + 1); the climb takes the first list that is not.
__device__ __forceinline__ uint32_t tree_ready(const TreeState *T, int k) {
  return (uint32_t)(k == 0 ? T->lists & kTreeListMask : T->rows[k - 1]);
}

// One thread per dirty-list entry (W waves per block: one, to spread the loads
// of a few thousand nodes over the CUs, or four, since blocks take their places
// in the lists by an atomic on one address each).  With kLeafLanes the leaves
// the word builder takes go to the leaf list, those of one block from its front
// and the others from its back (a wave of both would take the longer's time),
// with kLongLeaves the long ones to a list of their own; other leaves are ready.
constexpr int kLeafLanes = 1, kLongLeaves = 2;
template <int W>
__global__ __launch_bounds__(64 * W) void k_tree_link(Pools P, const ref_t *__restrict__ list, uint32_t n,
                                                  ref_t *__restrict__ ready, ref_t *__restrict__ leaves,
                                                  ref_t *__restrict__ longs, TreeState *T, int mode) {
  const uint32_t lane = __lane_id(), i = grid_tid();
  const ref_t r = i < n ? list[i] : REF_NULL;  // builds leave null holes
  bool rdy = false, leaf = false, tall = false, lng = false, listed = false;
  if (ref_type(r) == T_BRANCH) {
    Branch &B = P.branch[ref_idx(r)];
    ref_t c[16];
    const uint4 *cw = (const uint4 *)B.child;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint4 v = cw[q];
      c[4 * q] = v.x;
      c[4 * q + 1] = v.y;
      c[4 * q + 2] = v.z;
      c[4 * q + 3] = v.w;
    }
    uint32_t f[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const uint32_t t = ref_type(c[q]);
      f[q] = t == T_BRANCH || t == T_SHORT ? *node_dirty_flag(P, c[q]) : 0u;
    }
    const uint32_t me = tree_parent_word(r);
    uint32_t k = 0;
#pragma unroll
    for (int q = 0; q < 16; q++)
      if (f[q]) {
        *node_dirty_flag(P, c[q]) = me;
        k++;
      }
    B.pad1 = k;  // dirty children still to be hashed
    rdy = k == 0;
    listed = true;
  } else if (ref_type(r) == T_SHORT) {
    Short &S = P.shrt[ref_idx(r)];
    const ref_t c = S.child;
    if (ref_type(c) == T_VALUE) {
      listed = true;
      if (mode) {
        const uint32_t cnt = (uint32_t)S.key_len - S.term, vsz = P.value[ref_idx(c)].size;
        leaf = cnt <= kLeafFastNibbles && vsz <= kLeafDirectMaxValue;
        lng = !leaf && (mode & kLongLeaves);
        leaf = leaf && (mode & kLeafLanes);
        tall = leaf && leaf_blocks(cnt, vsz) > 1;
        leaf = leaf && !tall;
      }
      rdy = !leaf && !tall && !lng;
    } else if (S.lock & 1) {
      S.dirty = 0;  // replaced by a split since it was listed: no node's child any more, and its child another's
    } else {
      listed = true;
      uint32_t *f = node_dirty_flag(P, c);
      rdy = *f == 0;
      if (!rdy) *f = tree_parent_word(r);
    }
  }
  const uint64_t mr = __ballot(rdy), ml = __ballot(leaf), mt = __ballot(tall), ma = __ballot(listed);
  const uint64_t mo = __ballot(lng);
  const unsigned long long mine = (unsigned long long)__popcll(mr) | (unsigned long long)__popcll(ml) << kTreeListBits |
                                  (unsigned long long)__popcll(ma) << (2 * kTreeListBits);
  unsigned long long base, tbase = 0, obase = 0;
  if (W == 1) {
    if (ma == 0) return;
    base = tree_reserve(&T->lists, mine, lane);
    if (mt) tbase = tree_reserve(&T->tall, (unsigned long long)__popcll(mt), lane);
    if (mo) obase = tree_reserve(&T->longs, (unsigned long long)__popcll(mo), lane);
  } else {
    __shared__ unsigned long long sums[W][3], place[3];
    const uint32_t g = threadIdx.x / 64;
    if (lane == 0) {
      sums[g][0] = mine;
      sums[g][1] = (unsigned long long)__popcll(mt);
      sums[g][2] = (unsigned long long)__popcll(mo);
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      unsigned long long all = 0;
      for (int q = 0; q < W; q++) all += sums[q][threadIdx.x];
      unsigned long long *at = threadIdx.x == 0 ? &T->lists : threadIdx.x == 1 ? &T->tall : &T->longs;
      place[threadIdx.x] = all ? atomicAdd(at, all) : 0ull;
    }
    __syncthreads();
    base = place[0];
    tbase = place[1];
    obase = place[2];
    for (uint32_t q = 0; q < g; q++) {
      base += sums[q][0];
      tbase += sums[q][1];
      obase += sums[q][2];
    }
  }
  const uint64_t below = (1ull << lane) - 1;
  if (rdy) ready[(uint32_t)(base & kTreeListMask) + (uint32_t)__popcll(mr & below)] = r;
  if (leaf) leaves[(uint32_t)(base >> kTreeListBits & kTreeListMask) + (uint32_t)__popcll(ml & below)] = r;
  if (tall) leaves[n - 1 - ((uint32_t)tbase + (uint32_t)__popcll(mt & below))] = r;
  if (lng) longs[(uint32_t)obase + (uint32_t)__popcll(mo & below)] = r;
}

// Adds the wave's work counts (v on lanes 0 .. 6 as TreeState::parts' words).
__device__ __forceinline__ void tree_count(TreeState *T, uint32_t wave, uint32_t lane, unsigned long long v) {
  if (lane < 7 && v) atomicAdd(&T->parts[wave % kTreeParts][lane], v);
}

// A hashed node counts off at its parent word par: the parent if that was its
// last dirty child, or null.
__device__ __forceinline__ ref_t tree_up(const Pools &P, uint32_t par) {
  if (par >> 2 == 0) return REF_NULL;  // a root
  if (par & 2) return make_ref(T_SHORT, (par >> 2) - 1);  // an extension's only child
  return __hip_atomic_fetch_add(&P.branch[(par >> 2) - 1].pad1, ~0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 1u
             ? make_ref(T_BRANCH, (par >> 2) - 1)
             : REF_NULL;
}
// Appends the lanes' nodes (null: none) to a list with its length at `at`.
__device__ __forceinline__ void tree_append(unsigned long long *at, ref_t *list, ref_t r, uint32_t lane) {
  const uint64_t m = __ballot(r != REF_NULL);
  if (m == 0) return;
  const uint32_t base = (uint32_t)(tree_reserve(at, (unsigned long long)__popcll(m), lane) & kTreeListMask);
  if (r != REF_NULL) list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = r;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  for (int off = 32; off > 0; off >>= 1) v += (uint32_t)__shfl_xor((int)v, off);
  return v;
}

// The leaf list, one leaf per lane (as k_hc_leaf_direct), the waves of longer
// leaves first; a node whose last dirty child was one of them becomes ready.
__global__ __launch_bounds__(256) void k_tree_leaves(Pools P, const ref_t *__restrict__ leaves, uint32_t n_list,
                                                     ref_t *ready, TreeState *T) {
  __shared__ uint64_t head[256][kLeafDirectHead];
  const uint32_t i = grid_tid(), lane = __lane_id();
  const uint32_t nt = (uint32_t)T->tall, wt = (nt + 63) / 64 * 64;                 // the longer ones' lanes
  const uint32_t n1 = (uint32_t)(T->lists >> kTreeListBits & kTreeListMask);  // only the ready count moves here
  const bool tall = i < wt;                                                        // uniform over the wave
  const uint32_t k = tall ? i : i - wt, n = tall ? nt : n1;
  if (k - lane >= n) return;
  const bool act = k < n;
  const ref_t r = act ? leaves[tall ? n_list - 1 - k : k] : REF_NULL;
  uint64_t m[2] = {0, 0};
  uint32_t wlo = 0xffffu, whi = 0;  // the wave's window of string words (hash_leaf_shaped)
  if (act) {
    leaf_meta(P, r, m);
    leaf_value_words(m[0], wlo, whi);
  }
  for (int off = 32; off > 0; off >>= 1) {
    wlo = min(wlo, (uint32_t)__shfl_xor((int)wlo, off));
    whi = max(whi, (uint32_t)__shfl_xor((int)whi, off));
  }
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  whi = __builtin_amdgcn_readfirstlane(whi);
  uint32_t enc = 0;
  ref_t up = REF_NULL;
  if (act) {
    const uint32_t par = P.shrt[ref_idx(r)].dirty;
    enc = hash_leaf_shaped(P, r, m[0], m[1], head[threadIdx.x], wlo, whi);
    up = tree_up(P, par);
  }
  tree_append(&T->lists, ready, up, lane);
  const uint32_t bytes = wave_sum(enc), perms = wave_sum(enc >= 32 ? keccak_blocks(enc) : 0u);
  const uint32_t nodes = min(n - (k - lane), 64u);
  tree_count(T, i / 64, lane,
             lane == 0 || lane == 2 ? perms : lane == 1 || lane == 3 ? bytes : lane < 6 ? nodes : 0u);
}

// Ready list k (in) one node per lane, with the messages in LDS rows of NB
// blocks (rows_encode), if it is long enough; an extension whose child a lane
// has just hashed follows in the same lane.  What the rows do not take (taller
// nodes, values in branches, embedded children, leaves) and the parents that
// became ready make list k + 1 (out).
template <int NB>
__global__ __launch_bounds__(64) void k_tree_rows(Pools P, const ref_t *__restrict__ in, ref_t *__restrict__ out,
                                                  TreeState *T, int k) {
  const uint32_t n = tree_ready(T, k), lane = threadIdx.x;
  if (n < kTreeRowsMin) return;
  __shared__ RowsLds<NB> S;
  uint64_t *row = S.rows + lane * RowsLds<NB>::kStride;
  uint32_t perms = 0, bytes = 0, nodes = 0, exts = 0;
  for (uint32_t b = blockIdx.x * 64; b < n; b += gridDim.x * 64) {
    const bool active = b + lane < n;
    const ref_t r = active ? in[b + lane] : REF_NULL;
    uint32_t par = active ? *node_dirty_flag(P, r) : 0u;
    uint32_t enc, nb;
    const bool use = rows_encode<NB>(P, r, active, S, enc, nb) && active;
    ref_t up = r;  // not taken
    if (use) {
      ref_t me = r;
      uint64_t st[25];
      for (;;) {
#pragma unroll
        for (int q = 0; q < 25; q++) st[q] = 0;
        for (uint32_t j = 0; j < nb; j++) {
#pragma unroll
          for (int q = 0; q < 17; q++) st[q] ^= row[17 * j + q];
          keccak_f1600(st);
        }
        store_digest(P, me, st);
        perms += nb;
        bytes += enc;
        nodes++;
        exts += ref_type(me) == T_SHORT ? 1u : 0u;
        up = tree_up(P, par);
        if (up == REF_NULL || ref_type(up) == T_BRANCH) break;
        const Short &X = P.shrt[ref_idx(up)];
        if (!is_direct_ext(X) || !ext_row<NB>(P, X, st, row, enc, nb)) break;
        par = X.dirty;
        me = up;
      }
    }
    tree_append(&T->rows[k], out, up, lane);
    __syncthreads();  // the rows are reused
  }
  perms = wave_sum(perms);
  bytes = wave_sum(bytes);
  nodes = wave_sum(nodes);
  exts = wave_sum(exts);
  tree_count(T, blockIdx.x, lane,
             lane == 0 ? perms : lane == 1 ? bytes : lane == 4 ? nodes : lane == 6 ? exts : 0u);
}

// Agent-scope accesses for what waves on other dies write in the same launch.
template <typename T>
__device__ __forceinline__ T ld_agent(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A wave's LDS operations complete in order: only the compiler must not move
// them across.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A child's digest word q and its size, as another wave may just have stored them.
__device__ __forceinline__ void tree_child(const Pools &P, ref_t c, uint32_t q, uint64_t &h, uint32_t &hs) {
  if (ref_type(c) == T_BRANCH) {
    const uint64_t *w = (const uint64_t *)&P.branch[ref_idx(c)];
    h = ld_agent(w + q);
    hs = (uint32_t)ld_agent(w + 4) & 255u;
  } else {
    const uint64_t *w = (const uint64_t *)&P.shrt[ref_idx(c)];
    h = ld_agent(w + q);
    hs = (uint32_t)(ld_agent(w + 6) >> 16) & 255u;
  }
}

// A node's message: plen bytes in LDS, then the vsz bytes at va; enc = both.
struct TreeMsg {
  uint32_t plen, vsz, enc;
  uint64_t va;
};

// The size and place of a value's string item; its first byte for a 1-byte
// value (raw when <= 0x7f).
struct TreeStr {
  uint64_t va = 0;
  uint32_t vsz = 0, b0 = 0x80;
  __device__ __forceinline__ void load(const Pools &P, ref_t v) {
    const Value &V = P.value[ref_idx(v)];
    va = V.addr;
    vsz = V.size;
    if (vsz == 1) b0 = (uint32_t)value_word(va, 1, 0) & 255u;
  }
  __device__ __forceinline__ bool raw() const { return vsz == 1 && b0 <= 0x7f; }
};

// Ends a message at LDS offset p with the string item: its header (or raw
// byte) in LDS, its bytes left where they are.
__device__ __forceinline__ void tree_tail(uint8_t *b, uint32_t p, uint32_t lane, const TreeStr &s, TreeMsg &m) {
  uint32_t n = 1;
  const uint64_t h = s.raw() ? (uint64_t)s.b0 : rlp_hdr(s.vsz, 0x80, 0xB7, &n);
  if (lane < n) b[p + lane] = (uint8_t)(h >> (8 * lane));
  m.plen = p + n;
  m.va = s.va;
  m.vsz = s.raw() ? 0u : s.vsz;
}

// Four lanes per nibble slot: each takes 8 bytes of the child's digest (or raw
// encoding, written as a string like the digest).
__device__ __forceinline__ void tree_branch(const Pools &P, const Branch &B, uint32_t lane, uint8_t *b, TreeMsg &m) {
  const uint32_t s = lane >> 2, q = lane & 3;
  const ref_t c = B.child[s], c16 = B.child[16];
  uint64_t h = 0;
  uint32_t hs = 0;
  if (c != REF_NULL) tree_child(P, c, q, h, hs);
  TreeStr v;
  if (c16 != REF_NULL) v.load(P, c16);
  const uint32_t len = c == REF_NULL ? 1u : 1u + hs;
  uint32_t incl = len;  // over the slots (the same in a slot's four lanes)
#pragma unroll
  for (uint32_t d = 4; d < 64; d <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)incl, d);
    if (lane >= d) incl += t;
  }
  const uint32_t total = (uint32_t)__shfl((int)incl, 63);
  const uint32_t payload = total + (v.raw() || c16 == REF_NULL ? 1u : rlp_hdr_len(v.vsz) + v.vsz);
  uint32_t hn;
  const uint64_t hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
  if (lane < hn) b[lane] = (uint8_t)(hdr >> (8 * lane));
  const uint32_t pos = hn + incl - len;
  if (q == 0) b[pos] = (uint8_t)(0x80 + hs);  // an empty slot is an empty string
  if (hs == 32) {
#pragma unroll
    for (uint32_t t = 0; t < 8; t++) b[pos + 1 + 8 * q + t] = (uint8_t)(h >> (8 * t));
  } else {
    for (uint32_t t = 0; t < 8 && 8 * q + t < hs; t++) b[pos + 1 + 8 * q + t] = (uint8_t)(h >> (8 * t));
  }
  m.enc = hn + payload;
  if (c16 != REF_NULL) {
    tree_tail(b, hn + total, lane, v, m);
  } else {
    if (lane == 0) b[hn + total] = 0x80;
    m.plen = hn + total + 1;
    m.va = 0;
    m.vsz = 0;
  }
}

// One lane per byte of the compact key.
__device__ __forceinline__ void tree_short(const Pools &P, const Short &S, uint32_t lane, uint8_t *b, TreeMsg &m) {
  const ref_t c = S.child;
  const uint32_t term = S.term, cnt = (uint32_t)S.key_len - term, kc = cnt / 2 + 1, ks = S.key_start;
  const uint8_t *key = P.keys + S.key_off;
  const bool leaf = ref_type(c) == T_VALUE;
  TreeStr v;
  uint64_t h = 0;
  uint32_t hs = 0;
  if (leaf)
    v.load(P, c);
  else
    tree_child(P, c, lane & 3, h, hs);
  uint32_t khn = 0, hn;
  const uint64_t khdr = kc == 1 ? 0ull : rlp_hdr(kc, 0x80, 0xB7, &khn);  // a lone byte is <= 0x3f: raw
  const uint32_t payload = khn + kc + (!leaf ? 1u + hs : v.raw() ? 1u : rlp_hdr_len(v.vsz) + v.vsz);
  const uint64_t hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
  if (lane < hn) b[lane] = (uint8_t)(hdr >> (8 * lane));
  if (lane < khn) b[hn + lane] = (uint8_t)(khdr >> (8 * lane));
  const uint32_t odd = cnt & 1;
  for (uint32_t k = lane; k < kc; k += 64) {
    uint32_t x;
    if (k == 0) {
      x = (term << 5) | (odd << 4) | (odd ? packed_nibble(key, ks) : 0u);
    } else {
      const uint32_t j = ks + odd + 2 * (k - 1);
      x = (packed_nibble(key, j) << 4) | packed_nibble(key, j + 1);
    }
    b[hn + khn + k] = (uint8_t)x;
  }
  m.enc = hn + payload;
  const uint32_t p = hn + khn + kc;
  if (leaf) {
    tree_tail(b, p, lane, v, m);
  } else {
    if (lane == 0) b[p] = (uint8_t)(0x80 + hs);
    for (uint32_t t = 0; lane < 4 && t < 8 && 8 * lane + t < hs; t++) b[p + 1 + 8 * lane + t] = (uint8_t)(h >> (8 * t));
    m.plen = p + 1 + hs;
    m.va = 0;
    m.vsz = 0;
  }
}

// Message word w: LDS bytes, value bytes and, with nb, Keccak padding.
__device__ __forceinline__ uint64_t tree_word(const uint64_t *b, const TreeMsg &m, uint32_t nb, uint32_t w) {
  const uint32_t x0 = 8 * w;
  uint64_t v = 0;
  if (x0 < m.plen) v = low_bytes(b[w], m.plen - x0);
  if (m.vsz && x0 + 8 > m.plen && x0 < m.enc) v |= value_word(m.va, m.vsz, (int64_t)x0 - (int64_t)m.plen);
  if (nb) {
    if (m.enc >= x0 && m.enc < x0 + 8) v |= 0x01ull << (8 * (m.enc - x0));
    if (w + 1 == 17 * nb) v |= 0x80ull << 56;
  }
  return v;
}

// The long leaves (a key remainder past 64 nibbles or a value past 16 KB: the
// word builder takes neither), one per lane: the bytes before the value in LDS,
// the value's words from where they are, 8 to 9 us a block.  Few of them are
// left to the climb, where a wave each costs 3 ns a leaf and 1.14 a block: both
// take as long for about 7,000, whatever their blocks (whole builds, by lane /
// in the climb: 10,000 leaves of 1 block 231 / 244 us, 4,000 233 / 229; 9,000 of
// 16 416 / 460, 4,000 414 / 364; 8,000 of 126 1,423 / 1,534, 6,000 1,420 / 1,273).
// Insert and hash of 150,000 36-byte keys: 1,268 us with all in the climb, 437 so,
// 441 by levels; of 17,000 values of 17,000 bytes 2,897, 1,395 and 1,819.
constexpr uint32_t kLongHead = 19;  // words: headers and a compact key of 128 bytes; odd, so that lanes' rows spread
__global__ __launch_bounds__(64) void k_tree_long(Pools P, const ref_t *__restrict__ longs, ref_t *ready, TreeState *T) {
  const uint32_t n = (uint32_t)T->longs, lane = threadIdx.x;
  if (n == 0) return;
  __shared__ uint64_t heads[64][kLongHead];
  uint64_t *head = heads[lane];
  const bool lanes = n > kTreeLongLanes;
  uint32_t perms = 0, nodes = 0;
  unsigned long long bytes = 0;
  for (uint32_t b = blockIdx.x * 64; b < n; b += gridDim.x * 64) {
    const bool act = b + lane < n;
    const ref_t r = act ? longs[b + lane] : REF_NULL;
    if (!lanes) {
      tree_append(&T->lists, ready, r, lane);
      continue;
    }
    ref_t up = REF_NULL;
    if (act) {
      const Short &S = P.shrt[ref_idx(r)];
      const uint32_t par = S.dirty, term = S.term, cnt = (uint32_t)S.key_len - term;
      TreeStr v;
      v.load(P, S.child);
      const uint32_t payload = rlp_item_len(cnt / 2 + 1, 0) + (v.raw() ? 1u : rlp_hdr_len(v.vsz) + v.vsz);
      uint32_t hn, sn = 1;
      const uint64_t hdr = rlp_hdr(payload, 0xC0, 0xF7, &hn);
      const uint64_t sh = v.raw() ? (uint64_t)v.b0 : rlp_hdr(v.vsz, 0x80, 0xB7, &sn);
      WordWriter w(head);
      w.inline_bytes(hdr, hn);
      w.rlp_compact(P.keys + S.key_off, S.key_start, cnt, term);
      w.inline_bytes(sh, sn);
      head[w.nw] = w.acc;
      TreeMsg m;
      m.plen = 8 * w.nw + w.accn;
      m.va = v.va;
      m.vsz = v.raw() ? 0u : v.vsz;
      m.enc = hn + payload;
      const uint32_t nb = keccak_blocks(m.enc);
      uint64_t st[25];
#pragma unroll
      for (int q = 0; q < 25; q++) st[q] = 0;
      // A block of value bytes only is loaded (its aligned words) before the
      // permutation ahead of it, which hides the loads.
      uint64_t word[18];
      uint32_t off = 0;  // of the block's first byte in word[0]
      bool loaded = false;
      for (uint32_t k = 0; k < nb; k++) {
        if (loaded) {
#pragma unroll
          for (uint32_t q = 0; q < 17; q++) st[q] ^= funnel8(word[q], word[q + 1], off);
        } else {
#pragma unroll
          for (uint32_t q = 0; q < 17; q++) st[q] ^= tree_word(head, m, nb, 17 * k + q);
        }
        const uint32_t x = 136 * (k + 1);
        loaded = x >= m.plen && m.vsz >= 136 && x - m.plen <= m.vsz - 136;
        if (loaded) {
          const uint64_t at = m.va + (x - m.plen);
          const uint64_t *src = (const uint64_t *)(at & ~7ull);
          off = (uint32_t)(at & 7);
#pragma unroll
          for (uint32_t q = 0; q < 17; q++) word[q] = src[q];
          word[17] = src[off ? 17 : 16];  // no word past the value's last byte
        }
        keccak_f1600(st);
      }
      store_digest(P, r, st);
      up = tree_up(P, par);
      perms += nb;
      bytes += m.enc;
      nodes++;
    }
    tree_append(&T->lists, ready, up, lane);
  }
  perms = wave_sum(perms);
  nodes = wave_sum(nodes);
  for (int off = 32; off > 0; off >>= 1) bytes += (unsigned long long)__shfl_xor((long long)bytes, off);
  tree_count(T, blockIdx.x, lane, lane == 0 || lane == 2 ? perms : lane == 1 || lane == 3 ? bytes : lane < 6 ? nodes : 0ull);
}

// One wave per ready node; the wave climbs as long as it hashed its node's
// parent's last dirty child.  Its stores of a node (digest, then the word with
// the size) are written through and complete before the parent's count goes
// down; the last wave's loads of its siblings' nodes start after its own count
// came back.  Every wave ends: a step goes one node up.
// Bound by latency: a level costs its permutations (2.5 us each in the spread
// layout) and about 2.5 us of dependent loads, stores and the count.
constexpr uint32_t kTreeMsgWords = 80;  // a branch's items and value header take at most 536 bytes
__global__ __launch_bounds__(256) void k_tree_climb(Pools P, const ref_t *__restrict__ ready,
                                                    const ref_t *__restrict__ ready1, TreeState *T, int passes) {
  __shared__ uint64_t lds[256 / 64][kTreeMsgWords];
  const uint32_t lane = __lane_id(), g = threadIdx.x / 64;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (256 / 64) + g);
  int pass = 0;  // the list left by the row launches
  while (pass < passes && tree_ready(T, pass) >= kTreeRowsMin) pass++;
  const uint32_t n = tree_ready(T, pass);
  if (pass & 1) ready = ready1;
  if (wave >= n) return;
  uint64_t *msg = lds[g];
  uint8_t *b = (uint8_t *)msg;
  const SpreadLane sl(lane);
  const int w = SpreadLane::word_of(lane);
  uint32_t perms = 0, bytes = 0, lperms = 0, lbytes = 0, nodes = 0, lnodes = 0;
  uint32_t exts = 0;
  for (uint32_t i = wave; i < n; i += gridDim.x * (256 / 64)) {
    ref_t r = __builtin_amdgcn_readfirstlane(ready[i]);
    for (;;) {
      const bool branch = ref_type(r) == T_BRANCH;
      const uint32_t idx = ref_idx(r);
      uint64_t *node = branch ? (uint64_t *)&P.branch[idx] : (uint64_t *)&P.shrt[idx];
      const uint64_t meta = node[branch ? 4 : 6];  // dirty word in the upper half: the parent
      bool leaf = false;
      TreeMsg m;
      if (branch) {
        tree_branch(P, P.branch[idx], lane, b, m);
      } else {
        leaf = ref_type(P.shrt[idx].child) == T_VALUE;
        tree_short(P, P.shrt[idx], lane, b, m);
      }
      wave_lds_order();
      m.enc = __builtin_amdgcn_readfirstlane(m.enc);
      const uint32_t nb = m.enc >= 32 ? keccak_blocks(m.enc) : 0u;
      uint32_t hs = 32;
      if (nb == 0) {  // shorter than a digest: the raw encoding is the "hash"
        hs = m.enc;
        if (lane < 4) st_agent(node + lane, tree_word(msg, m, 0, lane));
      } else {
        uint32_t l = 0, h = 0;
        // the words of two blocks are in flight before the first permutation
        uint64_t cur = w >= 0 ? tree_word(msg, m, nb, (uint32_t)w) : 0ull;
        uint64_t nxt = w >= 0 && nb > 1 ? tree_word(msg, m, nb, 17 + (uint32_t)w) : 0ull;
        for (uint32_t k = 0; k < nb; k++) {
          l ^= (uint32_t)cur;
          h ^= (uint32_t)(cur >> 32);
          cur = nxt;
          if (k + 2 < nb && w >= 0) nxt = tree_word(msg, m, nb, 17 * (k + 2) + (uint32_t)w);
          keccak_spread(l, h, sl);
        }
        if (SpreadLane::digest(lane)) st_agent(node + (lane - 1), ((uint64_t)h << 32) | l);
      }
      if (lane == 0) {
        const uint32_t lo = (uint32_t)meta;
        if (branch)
          st_agent(node + 4, (uint64_t)((lo & 0xffffff00u) | hs));
        else
          st_agent(node + 6, (uint64_t)((lo & 0xff00ffffu) | hs << 16));
      }
      perms += nb;
      bytes += m.enc;
      nodes++;
      if (leaf) {
        lperms += nb;
        lbytes += m.enc;
        lnodes++;
      } else if (!branch) {
        exts++;
      }
      const uint32_t par = __builtin_amdgcn_readfirstlane((uint32_t)(meta >> 32));
      if (par >> 2 == 0) break;  // a root
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0);  // the node's stores have completed
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      if (par & 2) {
        r = make_ref(T_SHORT, (par >> 2) - 1);  // an extension's only child
      } else {
        uint32_t left = 0;
        if (lane == 0)
          left = __hip_atomic_fetch_add(&P.branch[(par >> 2) - 1].pad1, ~0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        left = __builtin_amdgcn_readfirstlane(left);
        if (left != 1) break;  // another child's wave goes on
        r = make_ref(T_BRANCH, (par >> 2) - 1);
      }
      wave_lds_order();
    }
    wave_lds_order();
  }
  tree_count(T, wave, lane,
             lane == 0 ? perms : lane == 1 ? bytes : lane == 2 ? lperms : lane == 3 ? lbytes : lane == 4 ? nodes : lane == 5 ? lnodes : exts);
}

// One wave: the counters, then (once those stores have completed) the number.
__device__ __forceinline__ void publish_wave(const Counters *cnt, const Publish &pub, uint32_t lane) {
  constexpr uint32_t kWords = sizeof(Counters) / 4;
  for (uint32_t q = lane; q < kWords; q += 64)
    __hip_atomic_store((uint32_t *)pub.host + q, ((const uint32_t *)cnt)[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");  // system scope; the wave's lanes store and wait as one
  if (lane == 0) __hip_atomic_store(pub.seq, pub.val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__global__ __launch_bounds__(64) void k_publish(const Counters *cnt, Publish pub) {
  publish_wave(cnt, pub, threadIdx.x);
}

__device__ __forceinline__ void roots_body(const Pools &P, uint32_t ntries, const unsigned long long *parts,
                                           TreeState *tree);
__global__ __launch_bounds__(256) void k_hc_roots(Pools P, uint32_t ntries, const unsigned long long *parts,
                                                  TreeState *tree, Publish pub) {
  roots_body(P, ntries, parts, tree);
  if (grid_tid() < sizeof(P.cnt->scal) / 4) P.cnt->scal[grid_tid()] = 0;
  if (!pub.host) return;
  __syncthreads();  // one block: its counters are complete
  if (threadIdx.x < 64) publish_wave(P.cnt, pub, threadIdx.x);
}
__device__ __forceinline__ void roots_body(const Pools &P, uint32_t ntries, const unsigned long long *parts,
                                           TreeState *tree) {
  uint32_t t = grid_tid();
  // the root's hash first: its two dependent loads overlap the counts' reduction
  uint32_t hs = 0;
  bool left = false;  // a climb left the root out (see hc_tree): its trie keeps the root hash it had
  uint4 h[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
  if (t < ntries) {
    const ref_t r = P.tries[t].root;
    if (ref_type(r) == T_SHORT || ref_type(r) == T_BRANCH) {
      left = tree && *node_dirty_flag(P, r) != 0;
      hs = node_hash_size(P, r);
      const uint4 *src = (const uint4 *)node_hash(P, r);  // offset 0 of a 64- or 128-byte node
      h[0] = src[0];
      h[1] = src[1];
    }
  }
  if (t == 0 && !tree) P.cnt->n_dirty = 0;  // every listed node has been hashed
  if (parts && blockIdx.x == 0) {  // the pass's work counts (uniform branch)
    static_assert(kHcCountParts == 256, "one partial per thread");
    __shared__ unsigned long long sh[4][4];
    unsigned long long v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = parts[4 * threadIdx.x + q];
#pragma unroll
    for (int q = 0; q < 4; q++)
      for (int off = 32; off > 0; off >>= 1) v[q] += (unsigned long long)__shfl_xor((long long)v[q], off);
    if (__lane_id() == 0)
#pragma unroll
      for (int q = 0; q < 4; q++) sh[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
    if (threadIdx.x < 4) {
      unsigned long long *dst = threadIdx.x == 0 ? &P.cnt->n_perms
                                : threadIdx.x == 1 ? &P.cnt->enc_bytes
                                : threadIdx.x == 2 ? &P.cnt->leaf_perms
                                                   : &P.cnt->leaf_bytes;
      *dst += sh[0][threadIdx.x] + sh[1][threadIdx.x] + sh[2][threadIdx.x] + sh[3][threadIdx.x];
    }
  }
  if (tree && blockIdx.x == 0) {  // a climb's counts (uniform branch); its state is left zero for the next one
    static_assert(kTreeParts == 256, "one partial per thread");
    __shared__ unsigned long long st[4][7];
    unsigned long long v[7];
#pragma unroll
    for (int q = 0; q < 7; q++) {
      v[q] = tree->parts[threadIdx.x][q];
      tree->parts[threadIdx.x][q] = 0;
    }
#pragma unroll
    for (int q = 0; q < 7; q++)
      for (int off = 32; off > 0; off >>= 1) v[q] += (unsigned long long)__shfl_xor((long long)v[q], off);
    if (__lane_id() == 0)
#pragma unroll
      for (int q = 0; q < 7; q++) st[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int q = 0; q < 7; q++) v[q] = st[0][q] + st[1][q] + st[2][q] + st[3][q];
      P.cnt->n_perms = v[0];
      P.cnt->enc_bytes = v[1];
      P.cnt->leaf_perms = v[2];
      P.cnt->leaf_bytes = v[3];
      P.cnt->hc_nodes = (uint32_t)v[4];
      P.cnt->hc_leaves = (uint32_t)v[5];
      P.cnt->hc_exts = (uint32_t)v[6];
      P.cnt->hc_listed = (uint32_t)(tree->lists >> (2 * kTreeListBits));
      if (P.cnt->hc_nodes == P.cnt->hc_listed) P.cnt->n_dirty = 0;  // otherwise the list stands for the levels
      tree->lists = tree->tall = tree->longs = 0;
      for (uint32_t q = 0; q < kTreeRowPasses; q++) tree->rows[q] = 0;
    }
  }
  if (t >= ntries || left) return;
  // bytes past the hash size (a root encoding under 32 bytes) read as zero
  uint32_t w[8] = {h[0].x, h[0].y, h[0].z, h[0].w, h[1].x, h[1].y, h[1].z, h[1].w};
#pragma unroll
  for (uint32_t q = 0; q < 8; q++) {
    const uint32_t keep = hs >= 4 * q + 4 ? 4u : hs > 4 * q ? hs - 4 * q : 0u;
    w[q] = keep == 4 ? w[q] : keep ? w[q] & ((1u << (8 * keep)) - 1) : 0u;
  }
  TrieHdr &T = P.tries[t];
  uint64_t *dst = (uint64_t *)T.root_hash;  // offset 16 of the header
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) dst[q] = ((uint64_t)w[2 * q + 1] << 32) | w[2 * q];
  T.root_hash_size = hs;
  if (t == 0) {
    uint32_t *d0 = (uint32_t *)P.cnt->root0;
#pragma unroll
    for (uint32_t q = 0; q < 8; q++) d0[q] = w[q];
    P.cnt->root0_size = hs;
  }
}

// ---------------------------------------------- standalone Keccak (test hook) --

__global__ __launch_bounds__(256) void k_kb_slots(const uint32_t *len, uint32_t n, uint64_t *slot) {
  uint32_t i = grid_tid();
  if (i < n) slot[i] = 136ull * keccak_blocks(len[i]);
}

__global__ __launch_bounds__(256) void k_kb_pad(const uint8_t *data, const uint64_t *off, const uint32_t *len,
                                                uint32_t n, const uint64_t *slot, uint64_t *scratch) {
  uint32_t i = grid_tid();
  if (i >= n) return;
  uint32_t L = len[i];
  WordWriter w(scratch + slot[i] / 8);
  if (L) w.mem_bytes(data + off[i], L);
  w.finish_keccak(keccak_blocks(L) * 17);
}

__global__ __launch_bounds__(256) void k_kb_lane(const uint64_t *slot, const uint32_t *len, uint32_t n,
                                                 const uint64_t *scratch, uint8_t *out) {
  uint32_t i = grid_tid();
  if (i >= n) return;
  uint64_t s[25];
  keccak_lane(scratch + slot[i] / 8, keccak_blocks(len[i]), s);
  for (int q = 0; q < 4; q++) ((uint64_t *)(out + 32 * (size_t)i))[q] = s[q];
}

__global__ __launch_bounds__(256) void k_kb_spread(const uint64_t *slot, const uint32_t *len, uint32_t n,
                                                   const uint64_t *scratch, uint8_t *out) {
  const uint32_t lane = __lane_id();
  const uint32_t i = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  uint32_t nb = i < n ? keccak_blocks(len[i]) : 0;
  SpreadLane c(lane);
  uint32_t l, h;
  sponge_spread(nb ? scratch + slot[i] / 8 : scratch, nb, lane, c, l, h);
  if (nb && SpreadLane::digest(lane)) ((uint64_t *)(out + 32 * (size_t)i))[lane - 1] = ((uint64_t)h << 32) | l;
}

// ------------------------------------------------------------- node export --

// (64 threads a block: a few thousand nodes' dependent loads spread over the CUs)
__global__ __launch_bounds__(64) void k_enc_len(Pools P, const ref_t *refs, uint32_t m, uint64_t *len) {
  uint32_t i = grid_tid();
  if (i >= m) return;
  uint32_t pay = node_payload(P, refs[i]);
  len[i] = rlp_hdr_len(pay) + pay;
}

// Node export: RLP encoding at offs[i], the 32-byte hash slot and the index
// pair of node i.  One wave per node: the message as the climb builds it (in
// LDS, a value's bytes where they are), stored a byte per lane, so a wave's
// stores fill whole lines.  (One thread per node wrote its encoding byte after
// byte: 126 us for 6,000 nodes, 12 now.)
__global__ __launch_bounds__(256) void k_enc_write(Pools P, const ref_t *refs, uint32_t m, const uint64_t *offs,
                                                   uint8_t *encs, uint64_t *hashes, uint64_t *pairs) {
  __shared__ uint64_t lds[256 / 64][kTreeMsgWords];
  const uint32_t lane = __lane_id(), g = threadIdx.x / 64;
  const uint32_t i = blockIdx.x * (256 / 64) + g;
  if (i >= m) return;  // no block barrier below
  uint8_t *b = (uint8_t *)lds[g];
  const ref_t r = refs[i];
  TreeMsg msg;
  if (ref_type(r) == T_BRANCH)
    tree_branch(P, P.branch[ref_idx(r)], lane, b, msg);
  else
    tree_short(P, P.shrt[ref_idx(r)], lane, b, msg);
  wave_lds_order();
  const uint64_t off = offs[i];
  uint8_t *out = encs + off;
  for (uint32_t p = lane; p < msg.plen; p += 64) out[p] = b[p];
  const uint8_t *v = (const uint8_t *)msg.va;
  for (uint32_t p = lane; p < msg.vsz; p += 64) out[msg.plen + p] = v[p];
  if (lane < 4) {
    const uint32_t hs = node_hash_size(P, r);
    const uint64_t h = ((const uint64_t *)node_hash(P, r))[lane];
    hashes[4 * (size_t)i + lane] = hs <= 8 * lane ? 0ull : low_bytes(h, hs - 8 * lane);
  }
  if (lane == 0) {
    pairs[2 * (size_t)i] = off;
    pairs[2 * (size_t)i + 1] = off + msg.enc - 1;
  }
}

}  // namespace

size_t hc_temp_bytes(uint32_t n) { return scan_temp_bytes(n > kHcBins ? n : kHcBins); }

hipError_t hc_classify(const Pools &P, const ref_t *list, uint32_t n, HcMeta *meta, uint32_t *cursor, ref_t *out,
                       uint64_t *slot, uint32_t *packed, void *temp, hipStream_t s, uint64_t *lmeta_tmp,
                       uint64_t *lmeta, LeafRecords rec) {
  // the bins, and the pass's work counters (permutations, bytes, leaf
  // permutations, leaf bytes)
  static_assert(kHcBins >= 8, "one launch clears both");
  k_hc_zero<<<nblk(kHcBins), kB, 0, s>>>(meta->hist, kHcBins, (uint32_t *)&P.cnt->n_perms, 8);
  GMPT_LAUNCH_CHECK();
  if (n == 0) {
    k_hc_zero<<<1, kB, 0, s>>>(&meta->slot_lo, 4);  // slot_lo, nvalid, scratch_bytes
    return hipGetLastError();
  }
  unsigned tiles = (unsigned)((n + kHcTile - 1) / kHcTile);
  k_hc_hist<<<tiles, kB, 0, s>>>(P, list, n, meta->hist, packed, lmeta ? lmeta_tmp : nullptr, rec);
  GMPT_LAUNCH_CHECK();
  hipError_t e = scan_exclusive_u32(meta->hist, cursor, kHcBins, &meta->nvalid, temp, s);
  if (e != hipSuccess) return e;
  k_hc_scatter<<<tiles, kB, 0, s>>>(P, list, packed, n, cursor, out, slot, lmeta_tmp, lmeta, rec, meta);
  GMPT_LAUNCH_CHECK();
  // slot offsets of the sorted nodes that have a slot: [slot_lo, nvalid)
  return scan_exclusive_u64(slot, slot, n, &meta->scratch_bytes, temp, s, nullptr, &meta->slot_lo);
}

hipError_t hc_hash_range(const Pools &P, const ref_t *list, const uint64_t *slot, uint32_t n, uint64_t *scratch,
                         uint32_t *enc_len, bool leaves, uint32_t spread_max, hipStream_t s, hipEvent_t perm_begin,
                         hipEvent_t perm_end, uint32_t n_ext, const uint32_t *cls) {
  if (n == 0) return hipSuccess;
  if (!leaves && n <= spread_max) {  // small inner level: encode and hash in one launch
    if (perm_begin) {
      hipError_t e = hipEventRecord(perm_begin, s);
      if (e != hipSuccess) return e;
    }
    k_hc_small<<<(n + 3) / 4, kB, 0, s>>>(P, list, slot, n, scratch, enc_len);
    GMPT_LAUNCH_CHECK();
    if (perm_end) return hipEventRecord(perm_end, s);
    return hipSuccess;
  }
  // a level of branches of at most 4 blocks and extensions (all but a
  // sixteenth of its nodes): one launch with the messages in LDS, the rest
  // generic inside it; rows as tall as the level's tallest class needs (1, 2
  // or 4 blocks: taller rows leave fewer waves per CU)
  const uint32_t c01 = cls ? cls[0] + cls[1] : 0u, c23 = cls ? cls[2] + cls[3] : 0u;
  const uint32_t cext = cls ? cls[kExtClass] : 0u;
  const int rows_nb = !cls || leaves ? 0
                      : 16ull * ((uint64_t)c01 + cext) >= 15ull * n       ? (cls[1] ? 2 : 1)
                      : 16ull * ((uint64_t)c01 + c23 + cext) >= 15ull * n ? 4
                                                                            : 0;
  // Rows of 4 blocks leave a SIMD one wave, which issues at little more than
  // half its rate: where most of a level fits rows of 2, those nodes get a
  // launch of their own first (the nodes are sorted by class).  1,194,800 nodes,
  // 88 in 100 of them such: 451 -> 376 us; 432,200 nodes, 68 in 100: 246 -> 241.
  if (rows_nb == 4 && c01 >= kRowsSplitMin && 2ull * c01 >= n) {
    const uint32_t low[kHcClasses] = {cls[0], cls[1]};
    hipError_t e = hc_hash_range(P, list, slot, c01, scratch, enc_len, false, spread_max, s, perm_begin, nullptr, 0, low);
    if (e != hipSuccess) return e;
    uint32_t rest[kHcClasses] = {};
    std::copy(cls + 2, cls + kHcClasses, rest + 2);
    return hc_hash_range(P, list + c01, slot + c01, n - c01, scratch, enc_len + c01, false, spread_max, s, nullptr,
                         perm_end, n_ext, rest);
  }
  if (rows_nb) {
    // the few nodes taller than the rows (classes rows_nb .. 6, between the
    // row classes and the extensions) would take the generic encoder and hold
    // the launch open long after the bulk: the launch's first blocks, which
    // are dispatched first, encode and hash them concurrently with the bulk
    const uint32_t cov = std::min(n, rows_nb == 4 ? c01 + c23 : rows_nb == 2 ? c01 : cls[0]);
    const uint32_t multi = n - std::min(n, cov + cext);
    const uint32_t lo = multi ? cov : 0u, hi = lo + multi;
    const uint32_t nx = multi;  // the launch's first blocks: one of them per block
    const unsigned grid = (unsigned)((n + 63) / 64 + nx);
    if (rows_nb == 4)
      k_hc_inner_wave<4><<<grid, 64, 0, s>>>(P, list, slot, n, scratch, enc_len, lo, hi, nx);
    else if (rows_nb == 2)
      k_hc_inner_wave<2><<<grid, 64, 0, s>>>(P, list, slot, n, scratch, enc_len, lo, hi, nx);
    else
      k_hc_inner_wave<1><<<grid, 64, 0, s>>>(P, list, slot, n, scratch, enc_len, lo, hi, nx);
    GMPT_LAUNCH_CHECK();
    return hipSuccess;
  }
  // the level's extension class, sorted last: its own launch when it is large
  // enough to fill the GPU (a few thousand ride along in the branch kernels
  // at no cost, but would pay a launch's latency)
  if (!leaves && n_ext >= kExtDirectMin) {
    const uint32_t m = n - n_ext;
    k_hc_ext_direct<<<nblk(n_ext), kB, 0, s>>>(P, list + m, slot + m, n_ext, scratch, enc_len + m);
    GMPT_LAUNCH_CHECK();
    n = m;
    if (n == 0) return hipSuccess;
  }
  if (leaves)
    k_hc_encode_leaf<<<(n + kLeafNodes - 1) / kLeafNodes, kB, 0, s>>>(P, list, slot, n, scratch, enc_len);
  else
    k_hc_encode_inner<<<(n + kInnerNodes - 1) / kInnerNodes, kB, 0, s>>>(P, list, slot, n, scratch, enc_len);
  GMPT_LAUNCH_CHECK();
  if (perm_begin) {
    hipError_t e = hipEventRecord(perm_begin, s);
    if (e != hipSuccess) return e;
  }
  if (n <= spread_max)
    k_hc_perm_spread<<<(n + 3) / 4, kB, 0, s>>>(P, list, slot, enc_len, n, scratch);
  else
    k_hc_perm_lane<<<nblk(n), kB, 0, s>>>(P, list, slot, enc_len, n, scratch);
  GMPT_LAUNCH_CHECK();
  if (perm_end) return hipEventRecord(perm_end, s);
  return hipSuccess;
}

hipError_t hc_hash_leaves_direct(const Pools &P, const ref_t *list, const uint64_t *lmeta, const HcMeta *meta,
                                 uint32_t n_upper, uint32_t *enc_len, hipStream_t s) {
  if (n_upper == 0) return hipSuccess;
  k_hc_leaf_direct<<<nblk(n_upper), kB, 0, s>>>(P, list, lmeta, meta->hist, enc_len);
  return hipGetLastError();
}

hipError_t hc_tail_leaves(const Pools &P, const ref_t *list, uint32_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_hc_tail_leaves<<<(unsigned)((16ull * n + 255) / 256), kB, 0, s>>>(P, list, n);
  return hipGetLastError();
}

hipError_t hc_count(const uint32_t *enc_len, const HcMeta *meta, uint32_t n, uint32_t n_leaf,
                    unsigned long long *parts, hipStream_t s) {
  k_hc_count<<<kHcCountParts, kB, 0, s>>>(parts, enc_len, &meta->nvalid, n_leaf);
  return hipGetLastError();
}

namespace {
__global__ __launch_bounds__(256) void k_clear(Counters *cnt, TrieHdr *tries, uint32_t ntries) {
  uint32_t t = grid_tid();
  if (t < sizeof(Counters) / 4) ((uint32_t *)cnt)[t] = 0;
  for (uint32_t q = t; q < ntries * (uint32_t)(sizeof(TrieHdr) / 4); q += gridDim.x * blockDim.x)
    ((uint32_t *)tries)[q] = 0;
}
}  // namespace

namespace {
// A replayed pass is valid when the batch sorted without fallback, raised no
// error, and produced the captured pass's dirty-list length, element count
// and hash bins; otherwise it marks the pass bad (the hash kernels, which
// launch with the captured level ranges, then skip).
__global__ __launch_bounds__(256) void k_graph_check(Pools P, const uint32_t *__restrict__ hist,
                                                     const uint32_t *__restrict__ plan, uint32_t nbins,
                                                     uint32_t n_dirty, uint32_t ne, const uint32_t *scal) {
  __shared__ uint32_t bad;
  if (threadIdx.x == 0)
    bad = P.cnt->err != 0 || P.cnt->flag_fallback != 0 || P.cnt->n_dirty != n_dirty || scal[SC_NE_INDEX] != ne;
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < nbins; b += blockDim.x)
    if (hist[b] != plan[b]) bad = 1;
  __syncthreads();
  if (threadIdx.x == 0 && bad) P.cnt->graph_bad = 1;
}
}  // namespace

hipError_t hc_graph_check(const Pools &P, const HcMeta *meta, const uint32_t *plan_hist, uint32_t n_dirty, uint32_t ne,
                          const uint32_t *scal, hipStream_t s) {
  k_graph_check<<<1, kB, 0, s>>>(P, meta->hist, plan_hist, kHcBins, n_dirty, ne, scal);
  return hipGetLastError();
}

hipError_t hc_clear(Counters *cnt, TrieHdr *tries, uint32_t ntries, hipStream_t s) {
  size_t words = std::max<size_t>(sizeof(Counters) / 4, (size_t)ntries * sizeof(TrieHdr) / 4);
  k_clear<<<(unsigned)std::min<size_t>(nblk(words), 1024), kB, 0, s>>>(cnt, tries, ntries);
  return hipGetLastError();
}

hipError_t hc_roots(const Pools &P, uint32_t ntries, const unsigned long long *parts, hipStream_t s, TreeState *tree,
                    Publish pub) {
  const bool one = nblk(ntries) == 1;
  k_hc_roots<<<nblk(ntries), kB, 0, s>>>(P, ntries, parts, tree, one ? pub : Publish());
  GMPT_LAUNCH_CHECK();
  return one || !pub.host ? hipSuccess : publish_counters(P.cnt, pub, s);
}

namespace {
__global__ __launch_bounds__(256) void k_roots_out(const TrieHdr *tries, uint32_t count, uint64_t *hash, int32_t *size) {
  const uint32_t i = grid_tid(), t = i / 4, q = i % 4;  // 8 bytes per thread: the slots are written in a row
  if (t >= count) return;
  hash[i] = ((const uint64_t *)tries[t].root_hash)[q];
  if (q == 0) size[t] = (int32_t)tries[t].root_hash_size;
}
}  // namespace

hipError_t gather_roots(const TrieHdr *tries, uint32_t count, uint8_t *hash, int32_t *size, hipStream_t s) {
  k_roots_out<<<nblk(4 * (size_t)count), kB, 0, s>>>(tries, count, (uint64_t *)hash, size);
  return hipGetLastError();
}

hipError_t publish_counters(const Counters *cnt, Publish pub, hipStream_t s) {
  k_publish<<<1, 64, 0, s>>>(cnt, pub);
  return hipGetLastError();
}

hipError_t hc_tree(const Pools &P, const ref_t *list, uint32_t n, ref_t *ready, ref_t *ready1, ref_t *leaves,
                   TreeState *tree, int passes, bool longs, hipStream_t s) {
  if (n == 0 || n > kTreeMax) return hipErrorInvalidValue;
  const bool lanes = n > kTreeSpreadLeaves;
  const int mode = (lanes ? kLeafLanes : 0) | (longs ? kLongLeaves : 0);
  if (passes)
    k_tree_link<4><<<nblk(n), kB, 0, s>>>(P, list, n, ready, leaves, ready1, tree, mode);
  else
    k_tree_link<1><<<(n + 63) / 64, 64, 0, s>>>(P, list, n, ready, leaves, ready1, tree, mode);
  GMPT_LAUNCH_CHECK();
  if (lanes) {
    k_tree_leaves<<<nblk(n + 63), kB, 0, s>>>(P, leaves, n, ready, tree);
    GMPT_LAUNCH_CHECK();
  }
  if (longs) {
    k_tree_long<<<std::min<uint32_t>((n + 63) / 64, 2048), 64, 0, s>>>(P, ready1, ready, tree);
    GMPT_LAUNCH_CHECK();
  }
  // (one more block than the CUs hold at a time gains nothing: blocks loop)
  const unsigned grid = std::min<uint32_t>((n + 63) / 64, 4096);
  for (int k = 0; k < passes; k++) {
    const ref_t *in = k & 1 ? ready1 : ready;
    ref_t *out = k & 1 ? ready : ready1;
    if (k == 0)
      k_tree_rows<2><<<grid, 64, 0, s>>>(P, in, out, tree, k);
    else
      k_tree_rows<4><<<grid, 64, 0, s>>>(P, in, out, tree, k);
    GMPT_LAUNCH_CHECK();
  }
  k_tree_climb<<<std::min<uint32_t>((n + 3) / 4, passes ? 2048 : ~0u), kB, 0, s>>>(P, ready, ready1, tree, passes);
  return hipGetLastError();
}

hipError_t hc_enc_len(const Pools &P, const ref_t *refs, uint32_t m, uint64_t *len, hipStream_t s) {
  if (m == 0) return hipSuccess;
  k_enc_len<<<(m + 63) / 64, 64, 0, s>>>(P, refs, m, len);
  return hipGetLastError();
}

hipError_t hc_enc_write(const Pools &P, const ref_t *refs, uint32_t m, const uint64_t *offs, uint8_t *encs,
                        uint64_t *hashes, uint64_t *pairs, hipStream_t s) {
  if (m == 0) return hipSuccess;
  k_enc_write<<<(m + 3) / 4, kB, 0, s>>>(P, refs, m, offs, encs, hashes, pairs);
  return hipGetLastError();
}

uint64_t keccak_scratch_bytes(const uint32_t *len, uint32_t n) {
  uint64_t t = 0;
  for (uint32_t i = 0; i < n; i++) t += 136ull * (len[i] / 136 + 1);
  return t;
}

hipError_t keccak_batch(const uint8_t *data, const uint64_t *off, const uint32_t *len, uint32_t n, uint8_t *out,
                        uint64_t *slot, uint64_t *scratch, void *temp, int spread, hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_kb_slots<<<nblk(n), kB, 0, s>>>(len, n, slot);
  GMPT_LAUNCH_CHECK();
  hipError_t e = scan_exclusive_u64(slot, slot, n, nullptr, temp, s);
  if (e != hipSuccess) return e;
  k_kb_pad<<<nblk(n), kB, 0, s>>>(data, off, len, n, slot, scratch);
  GMPT_LAUNCH_CHECK();
  if (spread)
    k_kb_spread<<<(n + 3) / 4, kB, 0, s>>>(slot, len, n, scratch, out);
  else
    k_kb_lane<<<nblk(n), kB, 0, s>>>(slot, len, n, scratch, out);
  return hipGetLastError();
}

}  // namespace gmpt
