// pk_device.hip -- MI355X (gfx950) k-mer counting, histogram cutoff and
// macro-node construction behind the C ABI of include/pakhip.h.
//
// Pipeline of pk_count (one HIP stream per context, everything resident in HBM):
//   1. packing        k_pack reads the FASTA once: two bits per input byte
//                     (plus one exact low bit), the '\n' bits, and their count
//                     per block.
//   2. windows        k_lines / k_valid: which bytes end a k-mer, from the '\n'
//                     bits: record r = header line j0+2r, sequence line
//                     j0+2r+1, with the record rules and the format check of
//                     the reference's Sliding_window (src/kmer_counting.cpp:
//                     2890-2945).  A rank share keeps the ends its owner rule
//                     gives the rank (k_own, k_own_walk, k_own_key); the
//                     builder API's come from k_bld_bits, or
//                     as a read table from k_bld_flags / k_bld_write.
//   3. partition      k_split_main, k_split: tiles of k-mers sorted by a digit of the key's
//                     top bits, one tile per block, each tile written back
//                     as one contiguous piece with a table of where its
//                     digits start.  Level 1 cuts the k-mers out of the packed
//                     bases (the reference's rolling 3-bit update,
//                     kmer_shift, distribute_kmers.h:798-805, read off a
//                     window of bits), further levels gather a bucket's runs
//                     from the tiles of the level before.  This is the
//                     on-device stand-in for the reference's owner routing +
//                     MPI_Alltoallv (kmer_counting.cpp:254-352).
//   4. bucket count   k_bucket_hash: one workgroup per bucket counts
//                     the bucket's distinct keys in an LDS hash table, then
//                     counting-sorts them by the next bits and writes the
//                     ascending (key, count) pairs (the reference's sort + RLE
//                     + merge + aggregate, kmer_counting.cpp:3057-3086,
//                     169-250).  Buckets with more distinct keys than a table
//                     holds take extra passes, then the host-driven split
//                     k_part_hist / k_part_scatter.
//   5. compaction     k_compact: bucket results -> dense sorted table.
// pk_cutoff: per-block LDS histograms of counts < t, k_min_bucket, ordered
//   stream compaction (kmer_histogram.cpp:84-140).
// pk_macro_nodes: range-partitioned 5-way merge of the kept table seen as
//   pred keys (ascending) and, per first base a, succ keys (ascending within
//   the quarter): ranges ranked in LDS, then written (mn_construct.cpp:212-477).

#include <hip/hip_runtime.h>

#include <fcntl.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <cerrno>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "pakhip.h"

typedef unsigned __int128 u128;
typedef unsigned long long ull;

// ---------------------------------------------------------------------------
// Key helpers (Key = uint64_t for k <= 32, u128 for 32 < k <= 64).

template <class Key>
__host__ __device__ __forceinline__ Key key_mask(int nbits) {
  const int bits = (int)sizeof(Key) * 8;
  if (nbits >= bits) return ~Key(0);
  return (Key(1) << nbits) - Key(1);
}

// bits [pos, pos+nbits) of x; bits below 0 read as 0.  nbits <= 16.
template <class Key>
__device__ __forceinline__ uint32_t key_digit(Key x, int pos, int nbits) {
  if (nbits <= 0) return 0;
  Key y;
  if (pos >= 0) {
    if (pos >= (int)sizeof(Key) * 8) return 0;
    y = x >> pos;
  } else {
    y = x << (-pos);
  }
  return (uint32_t)y & ((1u << nbits) - 1u);
}

// u128 keys: the digit from a 32-bit funnel shift of the two 32-bit words
// around pos (v_alignbit), the words picked by a uniform pos without
// branches; same value as the generic form for nbits <= 32.
template <>
__device__ __forceinline__ uint32_t key_digit<unsigned __int128>(unsigned __int128 x, int pos, int nbits) {
  if (nbits <= 0) return 0;
  if (pos < 0) return (uint32_t)(x << (-pos)) & ((1u << nbits) - 1u);
  if (pos >= 128) return 0;
  const uint64_t lo = (uint64_t)x, hi = (uint64_t)(x >> 64);
  const uint32_t w0 = (uint32_t)lo, w1 = (uint32_t)(lo >> 32), w2 = (uint32_t)hi, w3 = (uint32_t)(hi >> 32);
  const int wi = pos >> 5;
  const uint32_t a = wi == 0 ? w0 : wi == 1 ? w1 : wi == 2 ? w2 : w3;
  const uint32_t b = wi == 0 ? w1 : wi == 1 ? w2 : wi == 2 ? w3 : 0u;
  return __builtin_amdgcn_alignbit(b, a, (uint32_t)(pos & 31)) & ((1u << nbits) - 1u);
}

// ---------------------------------------------------------------------------
// Block-wide primitives (wave64).

// Exclusive prefix sum of v over the block (all NT threads must call it).
template <int NT>
__device__ __forceinline__ ull block_excl_scan(ull v) {
  constexpr int NW = NT / 64;
  __shared__ ull wsum[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  ull x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    ull y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  if (w == 0) {
    const ull s = lane < NW ? wsum[lane] : 0ull;
    ull inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      ull y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane < NW) wsum[lane] = inc - s;
  }
  __syncthreads();
  const ull r = x - v + wsum[w];
  __syncthreads();
  return r;
}

// Exclusive prefix sum of v over the block and the block total, without a
// trailing barrier: the caller must pass a barrier before the next call.
template <int NT>
__device__ __forceinline__ ull block_scan_total(ull v, ull* total) {
  constexpr int NW = NT / 64;
  __shared__ ull wsum[NW + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  ull x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    ull y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  if (w == 0) {
    const ull s = lane < NW ? wsum[lane] : 0ull;
    ull inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      ull y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane < NW) wsum[lane] = inc - s;
    if (lane == NW - 1) wsum[NW] = inc;
  }
  __syncthreads();
  *total = wsum[NW];
  return x - v + wsum[w];
}

template <int NT>
__device__ __forceinline__ ull block_sum(ull v) {
  constexpr int NW = NT / 64;
  __shared__ ull ws[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) ws[w] = v;
  __syncthreads();
  ull s = 0;
#pragma unroll
  for (int i = 0; i < NW; i++) s += ws[i];
  __syncthreads();
  return s;
}

template <int NT>
__device__ __forceinline__ ull block_min(ull v) {
  constexpr int NW = NT / 64;
  __shared__ ull ws[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ull y = __shfl_xor(v, o, 64);
    v = y < v ? y : v;
  }
  if (lane == 0) ws[w] = v;
  __syncthreads();
  ull s = ~0ull;
#pragma unroll
  for (int i = 0; i < NW; i++) s = ws[i] < s ? ws[i] : s;
  __syncthreads();
  return s;
}

// ---------------------------------------------------------------------------
// Small utility kernels.

__global__ void k_fill_u64(ull* p, ull v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Results on their way to the host: up to four pieces of 8-byte words, one
// after another into the context's pinned words (box).
constexpr int BOX_WORDS = 512;
struct Post {
  const ull* src[4];
  int n[4];
};

__device__ __forceinline__ void post_words(const Post& p, ull* box) {
  int i = (int)threadIdx.x;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (i >= 0 && i < p.n[q]) box[threadIdx.x] = p.src[q][i];
    i -= p.n[q];
  }
}

__global__ __launch_bounds__(BOX_WORDS) void k_post(Post p, ull* box) { post_words(p, box); }

// ---------------------------------------------------------------------------
// Exclusive scan (u32 or u64 in, u64 out, out[n] = total).  SCAN_PER
// elements per 1024-thread block, SCAN_EPT consecutive ones per thread
// (read and written as 16-byte vectors where aligned, so a thread's loads
// are in flight together).  Up to SCAN_ADD blocks add up the block sums before
// their own themselves (8 KB at most); more scan them first.

constexpr int SCAN_NT = 1024;
constexpr int SCAN_EPT = 16;
constexpr int SCAN_PER = SCAN_NT * SCAN_EPT;
constexpr uint64_t SCAN_ADD = 1024;

// elements [base, base + SCAN_EPT) of in, zero past n
template <class T>
__device__ __forceinline__ void scan_load(const T* in, uint64_t n, uint64_t base, ull* v) {
  if (base + SCAN_EPT <= n && (reinterpret_cast<uintptr_t>(in + base) & 15) == 0) {
    constexpr int PV = 16 / (int)sizeof(T);  // elements per 16-byte vector
    const uint4* p = reinterpret_cast<const uint4*>(in + base);
    uint4 q[SCAN_EPT / PV];
#pragma unroll
    for (int j = 0; j < SCAN_EPT / PV; j++) q[j] = p[j];
#pragma unroll
    for (int j = 0; j < SCAN_EPT / PV; j++) {
      const T* e = reinterpret_cast<const T*>(&q[j]);
#pragma unroll
      for (int i = 0; i < PV; i++) v[j * PV + i] = (ull)e[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_EPT; i++) v[i] = base + i < n ? (ull)in[base + i] : 0ull;
  }
}

template <class T>
__global__ __launch_bounds__(SCAN_NT) void k_scan_reduce(const T* in, ull* sums, uint64_t n) {
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_PER + (uint64_t)threadIdx.x * SCAN_EPT;
  ull v[SCAN_EPT];
  scan_load<T>(in, n, base, v);
  ull s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_EPT; i++) s += v[i];
  s = block_sum<SCAN_NT>(s);
  if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// offs: null (one block), the block sums (sums), or their scan.  box: the total
// and the pieces of p go there too (the last block's).
template <class T>
__global__ __launch_bounds__(SCAN_NT) void k_scan_apply(const T* in, ull* out, const ull* offs, bool sums,
                                                        uint64_t n, Post p, ull* box) {
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_PER + (uint64_t)threadIdx.x * SCAN_EPT;
  ull v[SCAN_EPT];
  scan_load<T>(in, n, base, v);
  ull s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_EPT; i++) s += v[i];
  ull before = 0;
  if (sums) {
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += SCAN_NT) before += offs[i];
    before = block_sum<SCAN_NT>(before);
  } else if (offs) {
    before = offs[blockIdx.x];
  }
  const ull ex = block_excl_scan<SCAN_NT>(s);
  ull o = before + ex;
  if (base + SCAN_EPT <= n && (reinterpret_cast<uintptr_t>(out + base) & 15) == 0) {
    ulonglong2* q = reinterpret_cast<ulonglong2*>(out + base);
#pragma unroll
    for (int j = 0; j < SCAN_EPT / 2; j++) {
      const ull a = o;
      o += v[2 * j];
      q[j] = make_ulonglong2(a, o);
      o += v[2 * j + 1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_EPT; i++) {
      if (base + i < n) out[base + i] = o;
      o += v[i];
    }
  }
  // the thread owning element n-1 writes the total
  if (n > 0 && base <= n - 1 && n - 1 < base + SCAN_EPT) {
    out[n] = o;
    if (box) box[0] = o;
  }
  if (box && blockIdx.x == gridDim.x - 1) post_words(p, box + 1);
}

// ---------------------------------------------------------------------------
// Line index.

constexpr int NL_NT = 256;
// A block covers NL_SLABS slabs of NL_SLAB bytes; in slab j lane t reads the
// 16 bytes at 16 t (one coalesced 16-byte load per lane and slab).
constexpr int NL_SLABS = 4;
constexpr uint64_t NL_SLAB = (uint64_t)NL_NT * 16;
constexpr uint64_t NL_PER_BLOCK = NL_SLAB * NL_SLABS;

// 4-bit mask of the bytes of w equal to e (bit i = byte i): a byte is zero
// in t = w ^ eeee exactly when bit 7 of ((t & 7f..) + 7f..) | t is clear.
__device__ __forceinline__ uint32_t match4(uint32_t w, uint32_t e) {
  const uint32_t t = w ^ (e * 0x01010101u);
  const uint32_t z = ~(((t & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | t) & 0x80808080u;
  return ((z >> 7) & 1u) | ((z >> 14) & 2u) | ((z >> 21) & 4u) | ((z >> 28) & 8u);
}

// Masks (bit i = byte base + i) of the event bytes (e0 or e1) and, when
// want_gt, of the '>' bytes among the 16 bytes at base (bytes at or past n
// never match); returns the 16 bytes (zero past n).  The kernels are bound
// by these byte matches, so a second match runs only when e0 != e1 (the
// builder's delimiter and skip symbol; the main path looks for '\n' alone)
// and the '>' match only where a caller needs it.
__device__ __forceinline__ uint4 scan16(const uint8_t* fa, uint64_t n, uint64_t base, uint32_t e0, uint32_t e1,
                                        bool want_gt, uint32_t& ev, uint32_t& gt) {
  ev = 0;
  gt = 0;
  if (base + 16 <= n && ((reinterpret_cast<uintptr_t>(fa + base) & 15) == 0)) {
    const uint4 v = *reinterpret_cast<const uint4*>(fa + base);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t m = match4(w[i], e0);
      if (e1 != e0) m |= match4(w[i], e1);
      ev |= m << (4 * i);
      if (want_gt) gt |= match4(w[i], '>') << (4 * i);
    }
    return v;
  }
  uint32_t w[4] = {0, 0, 0, 0};
  for (int i = 0; i < 16; i++) {
    if (base + i >= n) break;
    const uint32_t b = fa[base + i];
    w[i >> 2] |= b << (8 * (i & 3));
    ev |= (uint32_t)(b == e0 || b == e1) << i;
    gt |= (uint32_t)(b == '>') << i;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ uint8_t byte_of(const uint4& v, int i) {
  const uint32_t w = i < 8 ? (i < 4 ? v.x : v.y) : (i < 12 ? v.z : v.w);
  return (uint8_t)(w >> (8 * (i & 3)));
}

// Event bytes of the index: bytes equal to e0 or e1 ('\n' and '\n' for the
// line index of the main path; delimiter and skip symbol for the builder).
// Per block: the number of event bytes and the first '>'.  Only the input's
// first '>' is wanted, so only block 0 looks for it unless gt_all is set
// (the host asks for that pass when block 0 holds no '>').
__global__ __launch_bounds__(NL_NT) void k_nl_count(const uint8_t* fa, uint64_t n, uint8_t e0,
                                                    uint8_t e1, ull* blk_cnt, ull* blk_gt, int gt_all) {
  const uint64_t b0 = (uint64_t)blockIdx.x * NL_PER_BLOCK + (uint64_t)threadIdx.x * 16;
  const bool want_gt = gt_all || blockIdx.x == 0;
  uint32_t ev[NL_SLABS], gm[NL_SLABS];
#pragma unroll
  for (int j = 0; j < NL_SLABS; j++) scan16(fa, n, b0 + j * NL_SLAB, e0, e1, want_gt, ev[j], gm[j]);
  ull c = 0, gt = ~0ull;
#pragma unroll
  for (int j = NL_SLABS - 1; j >= 0; j--) {
    c += __popc(ev[j]);
    if (gm[j]) gt = b0 + j * NL_SLAB + __ffs(gm[j]) - 1;
  }
  c = block_sum<NL_NT>(c);
  gt = block_min<NL_NT>(gt);
  if (threadIdx.x == 0) {
    blk_cnt[blockIdx.x] = c;
    blk_gt[blockIdx.x] = gt;
  }
}

// out[0] = min(in[0..n)) (one block).
__global__ __launch_bounds__(1024) void k_min_reduce(const ull* in, uint64_t n, ull* out) {
  ull m = ~0ull;
  for (uint64_t i = threadIdx.x; i < n; i += 1024) m = in[i] < m ? in[i] : m;
  m = block_min<1024>(m);
  if (threadIdx.x == 0) *out = m;
}

// Positions of the event bytes, ascending, from the block's base blk_off.
// The four slab counts of a thread travel through one block scan packed in
// 16-bit fields (a slab holds at most 4096 events, so no field carries).
// With follow = 1, bits 62-63 of each entry tell what follows the event: 1
// a '>', 2 the end of the input, 0 anything else (the record check would
// otherwise read that byte per record, one scattered line each).
constexpr int NL_FLAG_SHIFT = 62;
constexpr ull NL_POS_MASK = (1ull << NL_FLAG_SHIFT) - 1;

__global__ __launch_bounds__(NL_NT) void k_nl_write(const uint8_t* fa, uint64_t n, uint8_t e0,
                                                    uint8_t e1, const ull* blk_off, ull* nl, int follow) {
  const uint64_t b0 = (uint64_t)blockIdx.x * NL_PER_BLOCK + (uint64_t)threadIdx.x * 16;
  uint32_t ev[NL_SLABS];
  uint4 by[NL_SLABS];
  ull packed = 0;
#pragma unroll
  for (int j = 0; j < NL_SLABS; j++) {
    uint32_t gm;
    by[j] = scan16(fa, n, b0 + j * NL_SLAB, e0, e1, false, ev[j], gm);
    packed |= (ull)__popc(ev[j]) << (16 * j);
  }
  ull tot;
  const ull ex = block_scan_total<NL_NT>(packed, &tot);
  ull slab_base = blk_off[blockIdx.x];
#pragma unroll
  for (int j = 0; j < NL_SLABS; j++) {
    ull o = slab_base + ((ex >> (16 * j)) & 0xFFFFull);
    const uint64_t pos = b0 + j * NL_SLAB;
    for (uint32_t m = ev[j]; m; m &= m - 1) {
      const int i = __ffs(m) - 1;
      const uint64_t p = pos + i;
      ull f = 0;
      if (follow) {
        // the next byte: in this thread's 16 bytes, else the next chunk's
        // first (the neighbour's load, usually still in cache)
        f = p + 1 >= n ? 2ull : i < 15 ? (ull)(byte_of(by[j], i + 1) == '>') : (ull)(fa[p + 1] == '>');
      }
      nl[o++] = p | (f << NL_FLAG_SHIFT);
    }
    slab_base += (tot >> (16 * j)) & 0xFFFFull;
  }
}

// Base encodings of the two counting front ends.
//   ENC_MAIN:    char_to_el, (c >> 1) & 7 (distribute_kmers.h:784-786): the
//                3-bit code ORs into the previous base's low bit, and the
//                word is masked to 2k bits (kmer_shift, :798-805).
//   ENC_BUILDER: symbol_to_kmer (concurrent_kmer_counter.hpp:2097-2110):
//                A C T G -> 0 1 2 3, every other byte -> 0; the word is not
//                masked and keeps the last 4*sizeof(kmer_t) bases.
constexpr int ENC_MAIN = 0;
constexpr int ENC_BUILDER = 1;

__device__ __forceinline__ bool base_is_acgt(uint32_t c) { return c == 'A' || c == 'C' || c == 'G' || c == 'T'; }

// char_to_el
__device__ __forceinline__ uint32_t base_code(uint32_t c) { return (c >> 1) & 7u; }

// ---------------------------------------------------------------------------
// Packed input.  The counting path reads the input's bytes once and works on
// two bits per byte from then on: bases, headers and line ends alike, so that
// a k-mer of the read at byte p is the bit window of bytes [p, p + K).
//
//   E   one 32-bit word per 16 bytes, the first byte's field in the top two
//       bits: the two low bits of the byte's base code, the low one ORed with
//       the third code bit of the next byte (ENC_MAIN, the rolling update's
//       spill into the older base; without it for ENC_BUILDER).
//   RX  one word per 16 bytes, byte i at bit i: bits 0-15 the exact low bit
//       of the code (a window's last base has not seen the next byte: its
//       low bit comes from here), bits 16-31 the event bytes.  At an event
//       byte, which is no base, bit i says instead that a '>' follows it.
//
// One pass over the bytes at 16 per lane, half a byte written per byte; the
// valid window ends then come from RX (a quarter of the input) and the first
// partition level reads E, RX and those: 2.5 bytes of traffic per input byte,
// where the byte-wise line index, its second pass, the level-1 histogram and
// the level-1 scatter each read the input (4 bytes).

constexpr int PK_PAD = 8;  // E words before the input's first (windows reach four words back)

// four 2-bit fields, one per byte of t, first byte highest
__device__ __forceinline__ uint32_t pack_crumbs(uint32_t t) { return (t * 0x40100401u) >> 24; }
// bit 0 of each byte of t, first byte lowest
__device__ __forceinline__ uint32_t pack_bits(uint32_t t) { return ((t * 0x01020408u) >> 24) & 15u; }

template <int ENC>
__global__ __launch_bounds__(NL_NT) void k_pack(const uint8_t* fa, uint64_t n, uint8_t e0, uint8_t e1,
                                                ull* blk_cnt, ull* blk_gt, int gt_all, uint32_t* E, uint32_t* RX, ull* small) {
  const uint64_t b0 = (uint64_t)blockIdx.x * NL_PER_BLOCK + (uint64_t)threadIdx.x * 16;
  // the main path's flags (windows_main), before the kernels that set them
  if (small && blockIdx.x == 0 && threadIdx.x < 4) small[2 + threadIdx.x] = threadIdx.x == 0 ? ~0ull : 0ull;
  const bool want_gt = gt_all || blockIdx.x == 0;
  const int lane = threadIdx.x & 63;
  uint32_t ev[NL_SLABS], gm[NL_SLABS];
  uint4 by[NL_SLABS];
#pragma unroll
  for (int j = 0; j < NL_SLABS; j++) by[j] = scan16(fa, n, b0 + j * NL_SLAB, e0, e1, want_gt, ev[j], gm[j]);
  ull c = 0, gt = ~0ull;
#pragma unroll
  for (int j = NL_SLABS - 1; j >= 0; j--) {
    const uint64_t base = b0 + j * NL_SLAB;
    // the byte after these 16: the next lane's first (0 past the end)
    uint32_t nx = __shfl_down(by[j].x, 1, 64) & 0xFFu;
    if (lane == 63) nx = base + 16 < n ? fa[base + 16] : 0u;
    if (base < n) {
      const uint32_t w[5] = {by[j].x, by[j].y, by[j].z, by[j].w, nx};
      uint32_t e = 0, r = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint32_t t = (w[i] >> 1) & 0x03030303u;
        if (ENC == ENC_MAIN) {
          r |= pack_bits(t & 0x01010101u) << (4 * i);
          const uint32_t b = (w[i] >> 3) & 0x01010101u;  // third code bits
          t |= (b >> 8) | (((w[i + 1] >> 3) & 1u) << 24);
        } else {
          // every byte but A, C, G, T counts as 0
          uint32_t ok = 0;
#pragma unroll
          for (int q = 0; q < 4; q++) ok |= (uint32_t)(base_is_acgt((w[i] >> (8 * q)) & 0xFFu)) << (8 * q);
          t &= ok * 3u;
          r |= pack_bits(t & 0x01010101u) << (4 * i);
        }
        e |= pack_crumbs(t) << (24 - 8 * i);
      }
      if (ev[j]) {
        // which event bytes a '>' follows
        uint32_t g = (uint32_t)(nx == '>') << 16;
#pragma unroll
        for (int i = 0; i < 4; i++) g |= match4(w[i], '>') << (4 * i);
        r = (r & ~ev[j]) | ((g >> 1) & ev[j]);
      }
      E[PK_PAD + base / 16] = e;
      RX[base / 16] = r | (ev[j] << 16);
    }
    c += __popc(ev[j]);
    if (gm[j]) gt = base + __ffs(gm[j]) - 1;
  }
  c = block_sum<NL_NT>(c);
  gt = block_min<NL_NT>(gt);
  if (threadIdx.x == 0) {
    blk_cnt[blockIdx.x] = c;
    blk_gt[blockIdx.x] = gt;
  }
}

// Positions of the event bytes from RX (k_nl_write's, without flags): block b covers
// the same NL_PER_BLOCK bytes as k_pack's, a thread 64 consecutive ones.
__global__ __launch_bounds__(NL_NT) void k_nl_write_rx(const uint32_t* RX, uint64_t n, const ull* blk_off, ull* nl) {
  static_assert(NL_PER_BLOCK == (uint64_t)NL_NT * 64, "64 bytes per thread");
  const uint64_t nw = (n + 15) / 16;
  const uint64_t w0 = (uint64_t)blockIdx.x * (NL_PER_BLOCK / 16) + (uint64_t)threadIdx.x * 4;
  uint32_t w[4] = {0, 0, 0, 0};
  if (w0 + 4 <= nw) {
    const uint4 q = *reinterpret_cast<const uint4*>(RX + w0);
    w[0] = q.x;
    w[1] = q.y;
    w[2] = q.z;
    w[3] = q.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = w0 + i < nw ? RX[w0 + i] : 0u;
  }
  ull c = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) c += __popc(w[i] >> 16);
  ull tot;
  ull o = blk_off[blockIdx.x] + block_scan_total<NL_NT>(c, &tot);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    for (uint32_t m = w[i] >> 16; m; m &= m - 1) {
      const int b = __ffs(m) - 1;
      const uint64_t p = (w0 + i) * 16 + b;
      nl[o++] = p;
    }
  }
}

// The main path's records without a list of lines.  With j0 = the '\n's
// before the first '>' (p0), record r's sequence is the bytes that j0 + 2r + 1
// '\n's come before, and it is taken when its header's '\n' (number j0 + 2r)
// lies at least K + 1 bytes before the end of the input (k_reads' rules, from
// counts instead of positions).  lines: [0] j0, [1] R = records taken, [2]
// '\n's of the input, [3] p0 (n when there is none).  K2 > 0: *R2 = R of that
// window length.  One block.
// blk (with nb <= SCAN_PER): the '\n's per block, scanned into blk_off first.
__global__ __launch_bounds__(1024) void k_lines(const uint32_t* RX, uint64_t n, const ull* blk, ull* blk_off,
                                                uint64_t nb, const ull* gt, int K, int K2, ull* lines, ull* R2) {
  static_assert(SCAN_NT == 1024, "the scan's block");
  if (blk) {
    const uint64_t base = (uint64_t)threadIdx.x * SCAN_EPT;
    ull v[SCAN_EPT], s = 0;
    scan_load<ull>(blk, nb, base, v);
#pragma unroll
    for (int i = 0; i < SCAN_EPT; i++) s += v[i];
    ull o = block_excl_scan<SCAN_NT>(s);
#pragma unroll
    for (int i = 0; i < SCAN_EPT; i++) {
      if (base + i < nb) blk_off[base + i] = o;
      o += v[i];
      if (base + i + 1 == nb) blk_off[nb] = o;
    }
    __syncthreads();
  }
  const ull p0 = *gt < n ? *gt : n;
  const uint64_t nw = (n + 15) / 16;
  const ull m = blk_off[nb];
  // '\n's in [a, b) of one block's bytes or less
  auto count = [&](uint64_t a, uint64_t b) -> ull {
    ull c = 0;
    for (uint64_t w = a / 16 + threadIdx.x; w < nw && w * 16 < b; w += 1024) {
      uint32_t x = RX[w] >> 16;
      if (w * 16 < a) x &= 0xFFFFu << (a - w * 16);
      if (w * 16 + 16 > b) x &= (1u << (b - w * 16)) - 1u;
      c += (ull)__popc(x & 0xFFFFu);
    }
    return block_sum<1024>(c);
  };
  const uint64_t pb = p0 / NL_PER_BLOCK;
  const ull j0 = p0 < n ? blk_off[pb] + count(pb * NL_PER_BLOCK, p0) : m;
  auto records = [&](int k) -> ull {
    const ull c = m - count(n > (uint64_t)k ? n - (uint64_t)k : 0, n);  // '\n's at least k + 1 bytes before the end
    return p0 < n && c > j0 ? (c - j0 + 1) / 2 : 0;
  };
  const ull R = records(K);
  if (threadIdx.x == 0) {
    lines[0] = j0;
    lines[1] = R;
    lines[2] = m;
    lines[3] = p0;
  }
  if (K2 > 0) {
    const ull r2 = records(K2);
    if (threadIdx.x == 0) *R2 = r2;
  }
}

// Valid window ends: bit i of W[w] says that the K bytes up to byte 64 w + i
// are a k-mer's, i.e. that byte lies in the sequence of a record that is
// taken and no '\n' is among them.  A thread covers 64 bytes, a block the
// same bytes as k_pack's; cnt[block] = its valid ends.  first_err = the first
// record r >= 1 that does not start with '>' (the reference's assert).  All from
// the '\n' bits: a quarter byte read and an eighth written per input byte.  W2:
// the same bits for windows of K2 <= K bytes (a share's L-mers: 26 us less than
// a launch of their own for 0.21 GB).
__global__ __launch_bounds__(NL_NT) void k_valid(const uint32_t* RX, uint64_t n, const ull* blk_off,
                                                 const ull* lines, int K, ull* W, uint32_t* cnt, ull* first_err, int K2,
                                                 const ull* R2, ull* W2) {
  const uint64_t nw = (n + 15) / 16;
  const uint64_t w0 = (uint64_t)blockIdx.x * (NL_PER_BLOCK / 16) + (uint64_t)threadIdx.x * 4;
  const uint64_t base = w0 * 16;
  const int lane = threadIdx.x & 63;
  const ull j0 = lines[0], R = lines[1];
  ull x = 0, g = 0;  // '\n's; at a '\n': a '>' follows
  if (w0 + 4 <= nw) {
    const uint4 q = *reinterpret_cast<const uint4*>(RX + w0);
    x = (ull)(q.x >> 16) | (ull)(q.y >> 16) << 16 | (ull)(q.z >> 16) << 32 | (ull)(q.w >> 16) << 48;
    g = (ull)(q.x & 0xFFFFu) | (ull)(q.y & 0xFFFFu) << 16 | (ull)(q.z & 0xFFFFu) << 32 | (ull)(q.w & 0xFFFFu) << 48;
  } else {
    for (int i = 0; i < 4 && w0 + i < nw; i++) {
      x |= (ull)(RX[w0 + i] >> 16) << (16 * i);
      g |= (ull)(RX[w0 + i] & 0xFFFFu) << (16 * i);
    }
  }
  // the 64 bytes before: the previous lane's
  ull px = __shfl_up(x, 1, 64);
  if (lane == 0) {
    px = 0;
    if (w0 >= 4) {
      const uint4 q = *reinterpret_cast<const uint4*>(RX + w0 - 4);
      px = (ull)(q.x >> 16) | (ull)(q.y >> 16) << 16 | (ull)(q.z >> 16) << 32 | (ull)(q.w >> 16) << 48;
    }
  }
  // a '\n' among the last K bytes, up to and with this one
  u128 near = (u128)x << 64 | (u128)px;
  int c = 1;
  auto widen = [&](int k) -> ull {
    while (c < k) {
      const int sh = c < k - c ? c : k - c;
      near |= near << sh;
      c += sh;
    }
    return (ull)(near >> 64);
  };
  const ull near2 = W2 ? widen(K2) : 0;
  const ull near1 = widen(K);
  ull tot;
  const ull cb = blk_off[blockIdx.x] + block_scan_total<NL_NT>((ull)__popcll(x), &tot);
  // parity of the '\n's before each byte, relative to j0: odd in sequences
  ull par = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) par ^= par << o;
  ull seq = par ^ x;
  if ((cb ^ j0) & 1) seq = ~seq;
  const ull ce = cb + (ull)__popcll(x);
  // bytes up to the (j0)-th '\n' are before the first sequence, bytes after
  // the (j0 + 2R)-th belong to records not taken
  auto nth = [&](ull k) {  // bit of the k-th '\n' of these bytes
    ull t = x;
    for (; k; k--) t &= t - 1;
    return __ffsll((long long)t) - 1;
  };
  auto taken = [&](ull ok, ull R) -> ull {
    const ull last = j0 + 2 * R;
    if (ce <= j0 || cb > last) return 0;
    if (cb <= j0) {
      const int b = nth(j0 - cb);
      ok &= b == 63 ? 0ull : ~0ull << (b + 1);
    }
    if (ce > last) ok &= (1ull << nth(last - cb)) - 1;
    if (base >= n) return 0;
    if (base + 64 > n) ok &= (1ull << (n - base)) - 1;
    return ok;
  };
  const ull ok = taken(seq & ~near1, R);
  if (W2) W2[w0 / 4] = taken(seq & ~near2, *R2);
  // sequence ends that no '>' follows
  ull bad = x & seq & ~g;
  if (base + 64 >= n && n > base) bad &= ~(1ull << (n - 1 - base));
  for (; bad; bad &= bad - 1) {
    const int b = __ffsll((long long)bad) - 1;
    const ull c = cb + (ull)__popcll(x & ((1ull << b) - 1));
    if (c > j0) {
      atomicMin(first_err, (c - j0 + 1) / 2);
      break;
    }
  }
  W[w0 / 4] = ok;
  const ull sum = block_sum<NL_NT>((ull)__popcll(ok));
  if (threadIdx.x == 0) cnt[blockIdx.x] = (uint32_t)sum;
}

// Inputs beyond 4 GiB: flag set when some 2^32 - 16 bytes in a row may hold no
// '\n' (whole blocks without one), i.e. when a read may be too long.
__global__ void k_long_lines(const ull* blk_off, uint64_t nb, ull* flag) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  constexpr uint64_t span = 0xFFFFFFF0ull / NL_PER_BLOCK - 1;
  if (i + span <= nb && blk_off[i + span] == blk_off[i]) *flag = 1;
}

// a value that is the same in every lane, moved to scalar registers
__device__ __forceinline__ ull uniform(ull x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return (ull)hi << 32 | lo;
}

// Number of x[0..n) (ascending) that are <= key, found by the whole block:
// NT samples per step instead of a chain of log2(n) dependent loads.
template <int NT>
__device__ __forceinline__ ull block_upper(const ull* x, ull n, ull key) {
  ull lo = 0;
  while (n > (ull)NT) {
    const ull step = (n + NT - 1) / NT;
    const ull o = (ull)threadIdx.x * step;
    const int c = __syncthreads_count(o < n && x[lo + o] <= key);
    if (c == 0) return lo;
    // sample c - 1 is <= key, sample c (if any) is not
    const ull skip = (ull)(c - 1) * step;
    lo += skip;
    n = n - skip < step ? n - skip : step;
  }
  return lo + (ull)__syncthreads_count((ull)threadIdx.x < n && x[lo + threadIdx.x] <= key);
}

// ---------------------------------------------------------------------------
// Input formats: multi-line FASTA and four-line FASTQ (either with '\r\n'
// line ends) rewritten into the strict single-line FASTA the counting path
// reads.  Line j of the input is [a, b): a = 0 or one past the (j-1)-th
// '\n', b = the j-th '\n' or the end; a '\r' at b - 1 is dropped.  One
// thread per line computes the line's output length, a scan places the
// lines, and a pass over the output (k_fmt_copy) fetches the bytes.

constexpr int FMT_FASTA = 1;
constexpr int FMT_FASTQ = 2;

__device__ __forceinline__ void fmt_line(const uint8_t* in, uint64_t n, const ull* nl, uint64_t m, uint64_t j,
                                         ull& a, ull& b) {
  a = j ? nl[j - 1] + 1 : 0;
  b = j < m ? nl[j] : n;
  if (b > a && in[b - 1] == '\r') b--;
}

// Multi-line FASTA: *hmin = the first line that starts with '>'.
__global__ void k_fmt_first_record(const uint8_t* in, uint64_t n, const ull* nl, uint64_t m, uint64_t L,
                                   ull* hmin) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= L) return;
  const ull a = j ? nl[j - 1] + 1 : 0;
  if (a < n && in[a] == '>') atomicMin(hmin, (ull)j);
}

// Output bytes of every line.  FASTA: nothing before the first record; a
// header line gives itself + '\n'; a sequence line gives itself; the last
// line of a record adds the '\n' that ends the read (a header with no
// sequence line gives an empty read).  FASTQ: header (its '@' becomes '>')
// and sequence lines give themselves + '\n'; the '+' and quality lines give
// nothing.  bad receives the first malformed FASTQ line, too_long the first
// line whose output exceeds 32 bits.
template <int FMT>
__global__ void k_fmt_lines(const uint8_t* in, uint64_t n, const ull* nl, uint64_t m, uint64_t L,
                            const ull* hmin, uint32_t* olen, ull* lstart, uint32_t* llen, ull* bad,
                            ull* too_long) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= L) return;
  ull a, b;
  fmt_line(in, n, nl, m, j, a, b);
  const ull len = b - a;
  lstart[j] = a;
  llen[j] = (uint32_t)(len < 0xFFFFFFFFull ? len : 0xFFFFFFFFull);
  ull out;
  if (FMT == FMT_FASTA) {
    if (j < *hmin) {
      out = 0;
    } else {
      const bool header = len > 0 && in[a] == '>';
      bool last = j + 1 >= L;
      if (!last) {
        const ull a2 = nl[j] + 1;
        last = a2 < n && in[a2] == '>';
      }
      out = len + (header ? 1 : 0) + (last ? 1 : 0);
    }
  } else {
    const int role = (int)(j & 3);
    if ((role == 0 && !(len > 0 && in[a] == '@')) || (role == 2 && !(len > 0 && in[a] == '+')))
      atomicMin(bad, (ull)j);
    out = role < 2 ? len + 1 : 0;
  }
  if (out > 0xFFFFFFFFull) {
    atomicMin(too_long, (ull)j);
    out = 0;
  }
  olen[j] = (uint32_t)out;
}

// The copy, by output: a block writes FC_BYTES of it, a thread 16 bytes at a
// time, aligned.  The fields of the block's lines lie in LDS (FC_LINES of them;
// lines beyond come from memory), so that a chunk waits for memory only for
// its bytes: one unaligned load for each line it holds, shifted into place.
// Bound by issue: a wave goes through as many lines as its chunk of the most
// (0.21 GB of FASTQ, 0.11 GB written: 134 us; with the fields read per chunk
// 176; by input bytes, with a store of 16 bytes at any address, 371; blocks of
// 32 or 64 KiB and of 512 or 1024 threads within 5 %).
constexpr int FC_NT = 256;
constexpr uint32_t FC_BYTES = 16384;
constexpr uint32_t FC_LINES = 1024;

__device__ __forceinline__ u128 load16(const uint8_t* in, uint64_t n, uint64_t a) {
  u128 v = 0;
  if (a + 16 <= n) {
    __builtin_memcpy(&v, in + a, 16);
  } else {
    for (int i = 0; i < 16; i++)
      if (a + i < n) v |= (u128)in[a + i] << (8 * i);
  }
  return v;
}

// Blank lines a thread steps over one by one before it looks for the end of
// their run: a set with one blank line per read takes the steps, a run of three
// million lines would be 0.6 s of them.
constexpr uint32_t FC_BLANK = 16;

// The line from j on (which starts at or before o) that byte o of the output
// comes from: the last one that starts at or before it, by doubling steps.
__device__ __forceinline__ ull fmt_skip(const ull* ooff, ull L, ull j, ull o) {
  ull step = FC_BLANK;
  while (j + step < L && ooff[j + step] <= o) {
    j += step;
    step *= 2;
  }
  ull hi = j + step < L ? j + step : L;
  while (hi - j > 1) {
    const ull mid = (j + hi) >> 1;
    if (ooff[mid] <= o) j = mid; else hi = mid;
  }
  return j;
}

template <int FMT>
__global__ __launch_bounds__(FC_NT) void k_fmt_copy(const uint8_t* __restrict__ in, uint64_t n,
                                                    const ull* __restrict__ lstart,
                                                    const uint32_t* __restrict__ llen,
                                                    const uint32_t* __restrict__ olen,
                                                    const ull* __restrict__ ooff, ull L, uint8_t* __restrict__ out) {
  // line i of the block: its output starts at rel[i] (the first one's before)
  __shared__ uint32_t rel[FC_LINES], len[FC_LINES], ol[FC_LINES];
  __shared__ ull src[FC_LINES];
  const ull total = ooff[L];
  const ull o0 = (ull)blockIdx.x * FC_BYTES;
  if (o0 >= total) return;
  const uint32_t m = total - o0 < FC_BYTES ? (uint32_t)(total - o0) : FC_BYTES;
  // the last line that starts at or before the block's first byte
  const ull j0 = uniform(block_upper<FC_NT>(ooff, L, o0) - 1);
  const uint32_t q0 = (uint32_t)uniform(o0 - ooff[j0]);  // place in it
  const uint32_t nl = L - j0 < FC_LINES ? (uint32_t)(L - j0) : FC_LINES;
  for (uint32_t i = threadIdx.x; i < nl; i += FC_NT) {
    const ull d = i ? ooff[j0 + i] - o0 : 0;
    rel[i] = d < FC_BYTES ? (uint32_t)d : FC_BYTES;
    len[i] = llen[j0 + i];
    ol[i] = olen[j0 + i];
    src[i] = lstart[j0 + i];
  }
  __syncthreads();
  const bool fits = nl < FC_LINES || rel[FC_LINES - 1] >= m;
  for (uint32_t b = threadIdx.x * 16; b < m; b += FC_NT * 16) {
    ull i;  // the line of the chunk's first byte, from j0
    uint32_t q;
    if (fits) {
      uint32_t lo = 1, hi = nl;  // lines after the first that start at or before b
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (rel[mid] <= b) lo = mid + 1; else hi = mid;
      }
      i = lo - 1;
      q = i ? b - rel[i] : q0 + b;
    } else {
      ull lo = j0, hi = L;
      while (hi - lo > 1) {
        const ull mid = (lo + hi) >> 1;
        if (ooff[mid] <= o0 + b) lo = mid; else hi = mid;
      }
      i = lo - j0;
      q = (uint32_t)(o0 + b - ooff[lo]);
    }
    const uint32_t cnt = m - b < 16 ? m - b : 16;
    u128 v = 0;
    // (FASTQ: the lines after a read's have no output)
    uint32_t blank = 0;
    for (uint32_t p = 0; p < cnt && j0 + i < L; i += FMT == FMT_FASTQ && ((j0 + i) & 3) == 1 ? 3 : 1) {
      const bool in_lds = i < (ull)FC_LINES;
      const uint32_t n0 = in_lds ? len[i] : llen[j0 + i], n1 = in_lds ? ol[i] : olen[j0 + i];
      if (FMT == FMT_FASTA && n1 == 0 && ++blank == FC_BLANK) {
        // the line before the next one with output
        i = fmt_skip(ooff, L, j0 + i, o0 + b + p) - 1 - j0;
        blank = 0;
        continue;
      }
      if (q < n0 && n1) {
        const uint32_t t = n0 - q < cnt - p ? n0 - q : cnt - p;
        u128 x = load16(in, n, (in_lds ? src[i] : lstart[j0 + i]) + q);
        if (FMT == FMT_FASTQ && q == 0 && ((j0 + i) & 3) == 0) x = (x & ~(u128)0xFF) | '>';
        if (t < 16) x &= ((u128)1 << (8 * t)) - 1;
        v |= x << (8 * p);
        p += t;
        q += t;
      }
      // (a line without output adds nothing)
      for (; p < cnt && q < n1; q++, p++) v |= (u128)'\n' << (8 * p);
      q = 0;
    }
    if (cnt == 16) {
      *reinterpret_cast<uint4*>(out + o0 + b) =
          make_uint4((uint32_t)v, (uint32_t)(v >> 32), (uint32_t)(v >> 64), (uint32_t)(v >> 96));
    } else {
      for (uint32_t i = 0; i < cnt; i++) out[o0 + b + i] = (uint8_t)(v >> (8 * i));
    }
  }
}

// Builder-API records (Concurrent_Kmer_Partial_Counter::
// default_count_and_process, concurrent_kmer_counter.hpp:2018-2082): from
// the current position the scan finds the next skip symbol ('>'), skips to
// the delimiter ('\n') that ends the header, and takes read_len bytes from
// there (fewer at the end of the buffer) as the read; the next scan starts
// at the read's first byte.  The records are therefore the first skip symbol
// after every delimiter (and the first one of the buffer): with ev = the
// positions of all delimiter and skip bytes in order, event e is a record
// when it is a skip symbol and event e-1 is not.  A record whose header has
// no delimiter ends the scan; a record is counted when its read holds >=
// klen bytes.  The two symbols differ (checked on the host).
struct BldSyms {
  uint8_t delim, skip;
};

__device__ __forceinline__ bool bld_record(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m,
                                           uint64_t e, int klen, uint64_t read_len, BldSyms sy,
                                           uint64_t* rb, uint64_t* rl) {
  if (fa[ev[e]] != sy.skip || (e > 0 && fa[ev[e - 1]] == sy.skip)) return false;
  uint64_t e2 = e + 1;
  while (e2 < m && fa[ev[e2]] != sy.delim) e2++;
  if (e2 >= m) return false;
  *rb = ev[e2] + 1;
  *rl = read_len < n - *rb ? read_len : n - *rb;
  return *rl >= (uint64_t)klen;
}

// Window ends of the records as k_valid's bitmap (W, cleared before), where a
// key is its window alone (klen >= the word's bases): a thread per event sets
// the ends of its record, two words for a read of 100 bytes, and no list of
// reads is made.  stat[0] = records, stat[1] set when a read runs on into the
// next event: its windows can then end where another's do, which one bit
// cannot say, and the read table takes its place (2 Mbp at 60x, klen = 32: the
// table and level 1 from it 520 us, the ends and k_split_main 240; blocks that
// loop, because one counter takes an add per block: 184 -> 62 us).
__global__ __launch_bounds__(256) void k_bld_bits(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m, int klen,
                                                  uint64_t read_len, BldSyms sy, ull* W, ull* stat) {
  ull rec = 0;
  for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < m; e += (uint64_t)gridDim.x * 256) {
    uint64_t rb, rl;
    if (!bld_record(fa, n, ev, m, e, klen, read_len, sy, &rb, &rl)) continue;
    rec++;
    // the header's delimiter lies right before the read
    uint64_t e2 = e + 1;
    while (e2 < m && ev[e2] < rb) e2++;
    if (e2 < m && ev[e2] < rb + rl) {
      // (no ends: reads that all run to the input's end would set n^2 of them)
      stat[1] = 1;
      continue;
    }
    const ull a = rb + (uint64_t)klen - 1, b = rb + rl;  // ends [a, b)
    for (ull w = a >> 6; w * 64 < b; w++) {
      ull bits = ~0ull;
      if (w * 64 < a) bits &= ~0ull << (a & 63);
      if (w * 64 + 64 > b) bits &= (1ull << (b & 63)) - 1;
      atomicOr(&W[w], bits);
    }
  }
  rec = block_sum<256>(rec);
  if (threadIdx.x == 0 && rec) atomicAdd(&stat[0], rec);
}

__global__ void k_bld_flags(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m, int klen,
                            uint64_t read_len, BldSyms sy, uint32_t* flag) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  uint64_t rb, rl;
  flag[e] = bld_record(fa, n, ev, m, e, klen, read_len, sy, &rb, &rl) ? 1u : 0u;
}

__global__ void k_bld_write(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m, int klen,
                            uint64_t read_len, BldSyms sy, const ull* idx, ull* rstart,
                            uint32_t* rlen, uint32_t* kc) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  uint64_t rb, rl;
  if (!bld_record(fa, n, ev, m, e, klen, read_len, sy, &rb, &rl)) return;
  const ull r = idx[e];
  rstart[r] = rb;
  rlen[r] = (uint32_t)rl;
  kc[r] = (uint32_t)(rl - (uint64_t)klen + 1);
}

// Window records of the implicit builder counters
// (Concurrent_Kmer_Partial_Counter::concurrent_count_and_process_omp_implicit_v0
// / _v1, src/concurrent_kmer_counter.hpp:910-1022,1363-1578): the records of
// bld_record (same scan), every one counted, whatever its length.  flag[e] =
// event e starts a record; bad[0] = a read shorter than read_len (cut at the
// end of the buffer), bad[1] = a read shorter than klen.
__global__ void k_win_flags(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m, int klen,
                            uint64_t read_len, BldSyms sy, uint32_t* flag, uint32_t* bad) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  uint64_t rb, rl;
  const bool rec = bld_record(fa, n, ev, m, e, 0, read_len, sy, &rb, &rl);
  flag[e] = rec ? 1u : 0u;
  if (rec && rl != read_len) atomicOr(&bad[0], 1u);
  if (rec && rl < (uint64_t)klen) atomicOr(&bad[1], 1u);
}

// Writes the window records: start, length and windows (len - klen + 1, or 0).
__global__ void k_win_write(const uint8_t* fa, uint64_t n, const ull* ev, uint64_t m, int klen,
                            uint64_t read_len, BldSyms sy, const ull* idx, ull* rstart, uint32_t* rlen,
                            uint32_t* wc) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  uint64_t rb, rl;
  if (!bld_record(fa, n, ev, m, e, 0, read_len, sy, &rb, &rl)) return;
  const ull r = idx[e];
  rstart[r] = rb;
  rlen[r] = (uint32_t)rl;
  wc[r] = rl >= (uint64_t)klen ? (uint32_t)(rl - (uint64_t)klen + 1) : 0u;
}

// The byte values present in the reads: bit v of present[v / 32].
__global__ void k_win_alpha(const uint8_t* fa, const ull* rstart, const uint32_t* rlen, uint64_t R,
                            uint32_t* present) {
  __shared__ uint32_t p[8];
  if (threadIdx.x < 8) p[threadIdx.x] = 0;
  __syncthreads();
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.y + threadIdx.y; r < R; r += (uint64_t)gridDim.x * blockDim.y) {
    const ull s = rstart[r];
    const uint32_t len = rlen[r];
    for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) {
      const uint32_t v = fa[s + i];
      atomicOr(&p[v >> 5], 1u << (v & 31));
    }
  }
  __syncthreads();
  if (threadIdx.x < 8 && threadIdx.y == 0 && p[threadIdx.x]) atomicOr(&present[threadIdx.x], p[threadIdx.x]);
}

// Window keys: the klen bytes of each window as codes of `bits` bits (code =
// rank of the byte value among the values present, so equal windows, and
// only those, get equal keys), first byte highest.  strncmp compares up to the
// first NUL: with NUL present (code 0) every code after a window's first NUL
// is 0.  One thread per read, windows in read order at woff[r].
template <class Key>
__global__ void k_win_keys(const uint8_t* fa, const ull* rstart, const uint32_t* rlen, const ull* woff,
                           uint64_t R, int klen, int bits, const uint8_t* lut, int has_nul, Key* S) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  const ull s = rstart[r];
  const uint32_t len = rlen[r];
  if (len < (uint32_t)klen) return;
  const uint32_t nw = len - (uint32_t)klen + 1;
  const int kb = klen * bits;
  const Key mask = kb >= (int)(8 * sizeof(Key)) ? ~Key(0) : ((Key(1) << kb) - 1);
  Key* out = S + woff[r];
  if (!has_nul) {
    Key km = 0;
    for (uint32_t i = 0; i < len; i++) {
      km = ((km << bits) | (Key)lut[fa[s + i]]) & mask;
      if (i + 1 >= (uint32_t)klen) out[i + 1 - (uint32_t)klen] = km;
    }
    return;
  }
  for (uint32_t w = 0; w < nw; w++) {
    Key km = 0;
    bool nul = false;
    for (int j = 0; j < klen; j++) {
      const uint8_t v = fa[s + w + j];
      const uint32_t code = nul ? 0u : (uint32_t)lut[v];
      nul = nul || v == 0;
      km = (km << bits) | (Key)code;
    }
    out[w] = km;
  }
}

// Records (kmer_counting.cpp:2920-2945).  Candidate r uses header newline
// nl[j0+2r] and sequence newline nl[j0+2r+1] (or the end of the buffer).
__global__ void k_reads(uint64_t n, const ull* nl, uint64_t m, uint64_t p0,
                        int K, uint64_t ncand, ull* rstart, uint32_t* rlen, uint32_t* kc,
                        ull* first_unproc, ull* first_err, ull* too_long) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // j0 = first newline at or after p0 (one search per block)
  __shared__ uint64_t sj0;
  if (threadIdx.x == 0) {
    uint64_t lo = 0, hi = m;
    while (lo < hi) {
      uint64_t mid = (lo + hi) >> 1;
      if ((nl[mid] & NL_POS_MASK) < p0) lo = mid + 1; else hi = mid;
    }
    sj0 = lo;
  }
  __syncthreads();
  if (r >= ncand) return;
  const uint64_t j0 = sj0;
  const uint64_t h = j0 + 2 * r;
  bool processed = false;
  if (p0 < n && h < m) {
    const uint64_t hdr_nl = nl[h] & NL_POS_MASK;
    processed = hdr_nl + 1 + (uint64_t)K <= n;
    if (processed) {
      const uint64_t s = hdr_nl + 1;
      const uint64_t e = (h + 1 < m) ? nl[h + 1] & NL_POS_MASK : n;
      const uint64_t len = e - s;
      rstart[r] = s;
      if (len > 0xFFFFFFF0ull) {
        atomicMin(too_long, (ull)r);
        rlen[r] = 0;
        kc[r] = 0;
      } else {
        rlen[r] = (uint32_t)len;
        kc[r] = len >= (uint64_t)K ? (uint32_t)(len - K + 1) : 0u;
      }
    }
  }
  if (!processed) {
    rstart[r] = 0;
    rlen[r] = 0;
    kc[r] = 0;
    atomicMin(first_unproc, (ull)r);
  }
  // assert(ptr[p] == '>') at the start of record r >= 1 when it is reached
  if (r >= 1 && p0 < n) {
    const uint64_t hp = j0 + 2 * r - 1;
    if (hp < m && (nl[hp] >> NL_FLAG_SHIFT) == 0) atomicMin(first_err, (ull)r);
  }
}

// ---------------------------------------------------------------------------
// Per-read rolling k-mer parse (one thread per read).

__device__ __forceinline__ uint64_t load_word8(const uint8_t* fa, uint64_t n, uint64_t a) {
  if (a + 8 <= n) return *reinterpret_cast<const uint64_t*>(fa + a);
  uint64_t w = 0;
  for (int i = 0; i < 8; i++)
    if (a + i < n) w |= (uint64_t)fa[a + i] << (8 * i);
  return w;
}

// ---------------------------------------------------------------------------
// Partition (multisplit) into buckets by the top bits of the key.
//   k_split    every level of the main and builder paths and the further
//              levels of the others: tiles sorted in registers and LDS
//   k_l1_hist / k_l1_scatter  level 1 where the packed input has no room
//              (pk_count_noalloc's smaller scratches): a walk over the bytes of
//              every read, each key straight to its slot

constexpr int L1_NT = 512;  // level-1 histogram blocks
constexpr int L1_MAX_BITS = PK_TUNING_L1_BITS_MAX;  // level-1 digit width
constexpr int L1_DEFAULT_BITS = 8;  // wider digits keep more partial lines open (k_l1_scatter)
constexpr int PK_MS_TILES = 4;      // pk_timing's form of a k_split level
constexpr int MS_TIMED_LEVELS = 4;  // further levels with their own timing events
static_assert(sizeof(pk_timing::ms_level_form) / sizeof(int32_t) == MS_TIMED_LEVELS, "per-level timing slots");

// Level-1 producer of the walk.  A block owns rpb consecutive reads and
// walks them in chunks: a chunk is the longest run of <= NT consecutive reads
// (NT threads per block) whose bytes fit in the LDS staging buffer; thread t
// then walks read t of the chunk from LDS with the rolling update (a read too
// long for the buffer is walked from global memory, alone in its chunk).
// Records are in file order, so a chunk's bytes are one contiguous range.
// The buffer holds the base code of every byte, not the byte: bits 0-1 of the
// code in plane A (32 bytes per word) and bit 2 in plane B
// (32 bytes per word), 3/8 of the raw size.  Its size (sb bytes, in dynamic
// LDS) is chosen per input so that NT typical records fit.
constexpr int L1_SB_MIN = 8192, L1_SB_MAX = 98304;  // staged bytes per chunk

struct ChunkLds {
  ull base;  // first staged byte (32-byte aligned)
  int m;     // reads in the chunk
  int lds;   // bytes are staged
};

struct Stage {
  ull* A;       // code bits 0-1 of byte 32 w + i at bits 2i, 2i+1 of A[w]
  uint32_t* B;  // code bit 2 of byte 32 w + i at bit i of B[w]
  int sb;       // capacity in bytes (a multiple of 32)
};

// Bytes of dynamic LDS of a level-1 kernel: the two planes, then nd digit
// entries of dig_bytes each.
__host__ __device__ constexpr uint32_t l1_lds_bytes(int sb, int nd, int dig_bytes) {
  return (uint32_t)(sb / 32) * 12u + (uint32_t)nd * (uint32_t)dig_bytes;
}

// Sets up the chunk starting at read c0 (< r1) and stages its codes.
template <int NT>
__device__ __forceinline__ void stage_chunk(ChunkLds& C, Stage sg, const uint8_t* fa, uint64_t n,
                                            const ull* rstart, const uint32_t* rlen, uint64_t c0,
                                            uint64_t r1) {
  const uint64_t r = c0 + threadIdx.x;
  const ull first = rstart[c0] & ~31ull;
  int fits = 0;
  if (r < r1 && (int)threadIdx.x < NT) fits = rstart[r] + rlen[r] - first <= (ull)sg.sb;
  // records ascend in the file: the reads that fit are a prefix
  const int m = (int)block_sum<NT>((ull)fits);
  if (threadIdx.x == 0) {
    C.base = first;
    C.m = m > 0 ? m : 1;
    C.lds = m > 0;
  }
  __syncthreads();
  if (C.lds) {
    const uint64_t last = c0 + C.m - 1;
    const ull end = rstart[last] + rlen[last];
    const ull nw = (end - first + 31) / 32;
    for (ull i = threadIdx.x; i < nw; i += NT) {
      ull a = 0;
      uint32_t b = 0;
#pragma unroll
      for (int h = 0; h < 4; h++) {
        const ull w = load_word8(fa, n, first + 32 * i + 8 * h);
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const uint32_t el = base_code((uint32_t)(w >> (8 * k)) & 0xFFu);
          a |= (ull)(el & 3u) << (16 * h + 2 * k);
          b |= (el >> 2) << (8 * h + k);
        }
      }
      sg.A[i] = a;
      sg.B[i] = b;
    }
  }
  __syncthreads();
}

// Walks up to Q more k-mers of the thread's read (state s, i, km): emits
// through emit(q, key); returns how many.
// km rolls unmasked (bits above the key shift out of the word, and the
// key's own bits are the same either way): the mask is applied to the keys
// handed out, once per k-mer instead of once per base.
template <class Key, class Emit>
__device__ __forceinline__ int walk_read(const ChunkLds& C, Stage sg, const uint8_t* fa, ull s, uint32_t len,
                                         uint32_t& i,
                                         Key& km, int K, Key mask, int Q,
                                         Emit&& emit) {
  int q = 0;
  if (C.lds) {
    // 32 staged codes at a time from the read's own position (two words
    // shifted together), so every lane runs the same count but on its last
    // piece (pieces ending at word boundaries differ per read and diverge)
    while (q < Q && i < len) {
      const ull off = s + i - C.base;
      const ull w = off >> 5;
      const uint32_t sh = (uint32_t)(off & 31);
      const uint32_t cnt = len - i < 32u ? len - i : 32u;
      ull a = sg.A[w] >> (2 * sh);
      uint32_t b = sg.B[w] >> sh;
      if (sh + cnt > 32u) {
        // the piece runs into the next word, which holds bases of this read
        a |= sg.A[w + 1] << (64 - 2 * sh);
        b |= sg.B[w + 1] << (32 - sh);
      }
      for (uint32_t t = 0; t < cnt && q < Q; t++) {
        const uint32_t el = ((uint32_t)a & 3u) | ((b & 1u) << 2);
        km = (km << 2) | (Key)el;
        a >>= 2;
        b >>= 1;
        i++;
        if (i >= (uint32_t)K) emit(q++, km & mask);
      }
    }
    return q;
  }
  while (q < Q && i < len) {
    const uint32_t el = base_code(fa[s + i]);
    km = (km << 2) | (Key)el;
    i++;
    if (i >= (uint32_t)K) emit(q++, km & mask);
  }
  return q;
}

// Level-1 histogram of the walk: digit = bits [KB - d1, KB) of each key.  Block b's count of digit d goes to H[d * nblk + b] (digit-major),
// so an exclusive scan of H gives every block the output base of each of its
// digit runs.
template <class Key>
__global__ __launch_bounds__(L1_NT) void k_l1_hist(const uint8_t* fa, uint64_t n, const ull* rstart,
                                                   const uint32_t* rlen, uint64_t R, int K, int KB,
                                                   Key mask, int d1, int rpb, int sb, uint32_t* H) {
  __shared__ ChunkLds C;
  // dynamic LDS: plane A, plane B, 2^d1 digit counts
  extern __shared__ ull l1_dyn[];
  const Stage sg{l1_dyn, reinterpret_cast<uint32_t*>(l1_dyn + sb / 32), sb};
  uint32_t* h = sg.B + sb / 32;
  const int nb = 1 << d1;
  for (int i = threadIdx.x; i < nb; i += L1_NT) h[i] = 0;
  const uint64_t r0 = (uint64_t)blockIdx.x * rpb;
  const uint64_t r1 = r0 + rpb < R ? r0 + rpb : R;
  const int bpos = KB - d1;
  for (uint64_t c0 = r0; c0 < r1;) {
    stage_chunk<L1_NT>(C, sg, fa, n, rstart, rlen, c0, r1);
    const int m = C.m;
    if ((int)threadIdx.x < m) {
      const uint64_t r = c0 + threadIdx.x;
      uint32_t i = 0;
      Key km = 0;
      walk_read<Key>(C, sg, fa, rstart[r], rlen[r], i, km, K, mask, 0x7fffffff,
                               [&](int, Key x) { atomicAdd(&h[key_digit<Key>(x, bpos, d1)], 1u); });
    }
    c0 += m;
    __syncthreads();
  }
  for (int i = threadIdx.x; i < nb; i += L1_NT) H[(ull)i * gridDim.x + blockIdx.x] = h[i];
}

// Level-1 scatter of the walk: the same chunked walk as k_l1_hist over
// the same reads per block; every key takes the next slot of its digit from
// the block's LDS cursor (the return value of one 64-bit atomic) and is
// stored at once.  The order of keys inside a bucket is arbitrary, which the
// bucket count does not depend on.
template <class Key>
__global__ __launch_bounds__(L1_NT) void k_l1_scatter(const uint8_t* fa, uint64_t n, const ull* rstart,
                                                      const uint32_t* rlen, uint64_t R, int K, int KB, Key mask,
                                                      int d1, int rpb, int sb, const ull* O,
                                                      uint64_t nblk, Key* S1) {
  __shared__ ChunkLds C;
  // dynamic LDS: plane A, 2^d1 output cursors, plane B
  extern __shared__ ull l1_dyn[];
  const int nb = 1 << d1;
  ull* cur = l1_dyn + sb / 32;
  const Stage sg{l1_dyn, reinterpret_cast<uint32_t*>(cur + nb), sb};
  for (int i = threadIdx.x; i < nb; i += L1_NT) cur[i] = O[(ull)i * nblk + blockIdx.x];
  const uint64_t r0 = (uint64_t)blockIdx.x * rpb;
  const uint64_t r1 = r0 + rpb < R ? r0 + rpb : R;
  const int bpos = KB - d1;
  // stage_chunk's barriers order the set-up above before the first walk
  for (uint64_t c0 = r0; c0 < r1;) {
    stage_chunk<L1_NT>(C, sg, fa, n, rstart, rlen, c0, r1);
    const int m = C.m;
    if ((int)threadIdx.x < m) {
      const uint64_t r = c0 + threadIdx.x;
      uint32_t i = 0;
      Key km = 0;
      walk_read<Key>(C, sg, fa, rstart[r], rlen[r], i, km, K, mask, 0x7fffffff,
                               [&](int, Key x) {
                                 const uint32_t d = key_digit<Key>(x, bpos, d1);
                                 S1[atomicAdd(&cur[d], 1ull)] = x;
                               });
    }
    c0 += m;
    __syncthreads();
  }
}

// bucket offsets of the walk's level 1 from its scanned histogram
__global__ void k_l1_boff(const ull* O, int nb, uint64_t nblk, ull total, ull* boff) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d < nb) boff[d] = O[(ull)d * nblk];
  if (d == nb) boff[nb] = total;
}

// ---------------------------------------------------------------------------
// Tiled partition.  A level splits every bucket of its input by db more key
// bits.  A bucket's keys are cut into tiles of tk; a block takes one tile into
// registers, ranks its keys by digit with LDS atomics, orders them through
// LDS and writes the tile back as one contiguous piece, at the place in the
// output array that the tile has in its bucket (tile t of bucket a starts at
// boff[a] + t * tk), with one table entry per digit: start << 16 | count.
// A bucket of the next level is then a list of runs, one per tile of its
// parent, which its reader gathers; no level needs a histogram pass over its
// input, and all writes are whole lines.
//
// What bounds it: memory.  Per level the keys are read and written once (a
// run of tk / 2^db keys costs up to one extra line), the run table is 12
// bytes per tile and digit, and no store leaves a partly written line but at
// a tile's ends.  Two 512-thread blocks per CU (64 KB of tile buffer and at
// most 128 VGPRs each) overlap one's loads with the other's LDS work.

constexpr int SP_NT = 512;
constexpr int SP_MAX_BITS = 10;  // digit width of a level
constexpr int SP_TILE_BYTES = 65536;

template <class Key>
struct SplitCfg {
  // keys per thread: 64 VGPRs of keys; tiles of 16384 one-word or 8192
  // two-word keys go through the tile buffer in two rounds
  static constexpr int Q = sizeof(Key) == 8 ? 32 : 16;
  static constexpr int TK_MAX = SP_NT * Q;
  static constexpr int ROUND = SP_TILE_BYTES / (int)sizeof(Key);
};

// The buckets of a level's output, as the next reader finds them.
//   M == nullptr: contiguous, bucket b is [boff[b], boff[b + 1]) of the array.
//   else: bucket b = a << db | s, of parent bucket a (tiles tp[a] ..
//   tp[a + 1], keys from boff[a] on), is the runs of digit s in the tiles of
//   a: entry e = (tp[a] << db) + s * ntiles(a) + t of the run table M (start
//   in the tile << 16 | count) and of V, the exclusive scan of the counts.  V
//   gives every key a place in key order of the buckets, the "virtual" index
//   that buckets and tiles are counted in; run e holds the indexes V[e] ..
//   V[e + 1] at array positions boff[a] + t * tk + start (with tb, whose
//   tiles vary in size: tb[t << ts] + start).
struct Runs {
  const uint32_t* M;
  const ull* V;
  const ull* tp;
  const ull* boff;
  int db;
  int tk;
  const ull* tb;  // level 1 of the main path: tile t starts at tb[t << ts]
  int ts;
};

// Array position of tile t of a bucket, from the bucket's first (base).
__device__ __forceinline__ ull tile_place(const Runs& in, ull t) { return in.tb ? in.tb[t << in.ts] : t * (ull)in.tk; }

// count field of a run-table entry, for the scan
struct RunCount {
  uint32_t v;
  __host__ __device__ operator ull() const { return (ull)(v & 0xFFFFu); }
};

struct RunBucket {
  ull v0, n;   // virtual start and key count
  ull e0, nt;  // first run-table entry and number of entries
  ull base;    // array position of the parent's first tile
};

__device__ __forceinline__ RunBucket uniform(const RunBucket& r) {
  return RunBucket{uniform(r.v0), uniform(r.n), uniform(r.e0), uniform(r.nt), uniform(r.base)};
}

// (called with one bucket per lane or per block)
__device__ __forceinline__ RunBucket run_bucket(const Runs& in, ull b) {
  RunBucket r;
  if (!in.M) {
    r.v0 = in.boff[b];
    r.n = in.boff[b + 1] - r.v0;
    r.e0 = r.nt = r.base = 0;
    return r;
  }
  const ull a = b >> in.db, s = b & ((1ull << in.db) - 1);
  const ull t0 = in.tp[a];
  r.nt = in.tp[a + 1] - t0;
  r.e0 = (t0 << in.db) + s * r.nt;
  r.v0 = in.V[r.e0];
  r.n = in.V[r.e0 + r.nt] - r.v0;
  r.base = in.boff[a];
  return r;
}

// Inclusive scan of a u32 over the wave by DPP moves (no LDS traffic, where
// shuffles take one LDS operation per step).
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);   // row_shr 1
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);   // row_shr 2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);   // row_shr 4
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);   // row_shr 8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);  // row_bcast 15 into rows 1, 3
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);  // row_bcast 31 into rows 2, 3
  return x;
}

// Exclusive scan of a u32 over the block through nw[NT / 64 + 1] (LDS); the
// total in *tot.  The caller passes a barrier before nw is used again.
template <int NT>
__device__ __forceinline__ uint32_t block_scan_u32(uint32_t v, uint32_t* nw, uint32_t* tot) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t x = wave_scan_u32(v);
  if (lane == 63) nw[w] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const uint32_t t = nw[i];
    before += i < w ? t : 0u;
    all += t;
  }
  *tot = all;
  return before + x - v;
}

// Map of the m places [v0, v0 + m) onto the pieces of a list that cover them:
// piece idx holds the places V[idx] .. V[idx + 1], its first at source
// position src(idx).  mw[w].x has bit i set when place 32 w + i starts a
// piece, mw[w].y counts the pieces that start before word w, and piece r of
// the map has put(r, source position - place, piece) called once; map_piece
// gives a place's r.  Pieces without places leave no trace.  The list is read
// from piece f (which covers v0 or ends before it) and has no piece past
// `end`.  Returns the number of pieces (put is only called for r < cap).
template <int NT, class Src, class Put>
__device__ __forceinline__ int map_pieces(uint2* mw, uint32_t* nw, int cap, const ull* V, ull f, ull end, ull v0,
                                          int m, Src&& src, Put&& put) {
  const int nwords = (m + 31) >> 5;
  const ull v1 = v0 + (ull)m;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < nwords; i += NT) mw[i].x = 0;
  uint32_t cnt = 0;
  for (ull c0 = f;; c0 += NT) {
    const ull idx = c0 + threadIdx.x;
    const bool in = idx < end;
    ull vs = 0, ve = 0;
    if (in) {
      vs = V[idx];
      ve = V[idx + 1];
    }
    const bool part = in && ve > vs && vs < v1 && ve > v0;
    const ull bal = __ballot(part);
    if (lane == 0) nw[w] = (uint32_t)__popcll(bal);
    // the list goes on inside the places when the chunk's last piece ends there
    const int more = __syncthreads_or(threadIdx.x == NT - 1 && in && ve < v1);
    uint32_t before = cnt, all = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) {
      before += i < w ? nw[i] : 0u;
      all += nw[i];
    }
    if (part) {
      const uint32_t r = before + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
      const uint32_t ls = vs > v0 ? (uint32_t)(vs - v0) : 0u;
      if (r < (uint32_t)cap) put(r, src(idx) - vs + v0, idx);
      atomicOr(&mw[ls >> 5].x, 1u << (ls & 31));
    }
    cnt += all;
    __syncthreads();
    if (!more) break;
  }
  // pieces before each word
  uint32_t carry = 0;
  for (int b = 0; b < nwords; b += NT) {
    const int i = b + (int)threadIdx.x;
    uint32_t tot;
    const uint32_t ex = block_scan_u32<NT>(i < nwords ? (uint32_t)__popc(mw[i].x) : 0u, nw, &tot);
    if (i < nwords) mw[i].y = carry + ex;
    carry += tot;
    __syncthreads();
  }
  return (int)cnt;
}

__device__ __forceinline__ uint32_t map_piece(const uint2* mw, int i) {
  const uint2 q = mw[i >> 5];
  return q.y + (uint32_t)__popc(q.x & (0xFFFFFFFFu >> (31 - (i & 31)))) - 1u;
}

// The same for places tid, tid + NT, ... of thread tid: the word is mt[j *
// NT / 32] with mt = mw + tid / 32, and the bits up to the place are the
// same for all (one LDS address per thread instead of one per place).
__device__ __forceinline__ uint32_t map_low(int tid) { return 0xFFFFFFFFu >> (31 - (tid & 31)); }
__device__ __forceinline__ uint32_t map_piece(uint2 q, uint32_t low) { return q.y + (uint32_t)__popc(q.x & low) - 1u; }

// Piece of place v by binary search (a map that did not fit): the last one in
// [f, end) that starts at or before v.
__device__ __forceinline__ ull find_piece(const ull* V, ull f, ull end, ull v) {
  ull lo = f, hi = end;  // V[lo] <= v, hi past the last
  while (hi - lo > 1) {
    const ull mid = (lo + hi) >> 1;
    if (V[mid] <= v) lo = mid; else hi = mid;
  }
  return lo;
}

// Tiles of a level: bucket offsets boff[0..B] of its input and tile prefix
// tp[0..B] (one block).
__global__ __launch_bounds__(1024) void k_tiles(Runs in, ull B, int tk, ull total, ull* boff, ull* tp) {
  __shared__ uint32_t nw[17];
  ull acc = 0;
  for (ull base = 0; base < B; base += 1024) {
    const ull b = base + threadIdx.x;
    RunBucket r{};
    if (b < B) r = run_bucket(in, b);
    uint32_t tot;
    const uint32_t nt = (uint32_t)((r.n + tk - 1) / tk);
    const uint32_t ex = block_scan_u32<1024>(nt, nw, &tot);
    if (b < B) {
      boff[b] = r.v0;
      tp[b] = acc + ex;
    }
    acc += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    boff[B] = total;
    tp[B] = acc;
  }
}

// One bucket over all windows (level 1's input).
__global__ void k_tiles_one(ull ntiles, ull total, ull* boff, ull* tp) {
  if (threadIdx.x || blockIdx.x) return;
  boff[0] = 0;
  boff[1] = total;
  tp[0] = 0;
  tp[1] = ntiles;
}

// Source of the builder's level 1: window i (of all reads' windows in order) belongs to
// the last read with kofs[r] <= i and starts at byte rstart[r] + i - kofs[r].
struct WinSrc {
  const uint32_t* E;
  const ull* kofs;    // R + 1 offsets
  const ull* rstart;
  ull R;
  int K;
};

enum { SPLIT_RUNS, SPLIT_BUILDER };

// Low 32-bit words of the window that ends at byte e, nw of them, low first.
template <int NWORDS>
__device__ __forceinline__ void window_words(const uint32_t* E, ull e, uint32_t* out) {
  const uint32_t* p = E + (PK_PAD + (e >> 4) - NWORDS);
  const uint32_t sh = 30u - 2u * (uint32_t)(e & 15);
  uint32_t w[NWORDS + 1];
#pragma unroll
  for (int i = 0; i <= NWORDS; i++) w[i] = p[i];
#pragma unroll
  for (int i = 0; i < NWORDS; i++)
    out[i] = __builtin_amdgcn_alignbit(w[NWORDS - 1 - i], w[NWORDS - i], sh);
}

template <class Key>
__device__ __forceinline__ Key window_key(const WinSrc& s, ull e) {
  uint32_t o[sizeof(Key) / 4];
  window_words<(int)sizeof(Key) / 4>(s.E, e, o);
  Key k = 0;
#pragma unroll
  for (int i = (int)sizeof(Key) / 4 - 1; i >= 0; i--) k = (k << 31 << 1) | (Key)o[i];
  return k;
}

template <class Key, int SRC>
__global__ __launch_bounds__(SP_NT, 4) void k_split(const Key* __restrict__ Sin, WinSrc ws, Runs in, int nb, int tk,
                                                    int dpos, int db, const ull* __restrict__ boff,
                                                    const ull* __restrict__ tp, uint32_t* __restrict__ M,
                                                    Key* __restrict__ Sout) {
  constexpr int Q = SplitCfg<Key>::Q;
  constexpr int ROUND = SplitCfg<Key>::ROUND;
  // the tile buffer; before the keys are loaded, the map's piece table
  __shared__ __align__(16) unsigned char buf[SP_TILE_BYTES];
  // digit counts, then starts; before, the map's words
  __shared__ uint32_t h[1 << SP_MAX_BITS];
  __shared__ uint32_t nw[SP_NT / 64 + 1];
  static_assert(SplitCfg<Key>::TK_MAX / 32 * sizeof(uint2) <= sizeof(h), "map words fit the digit counts");
  uint2* mw = reinterpret_cast<uint2*>(h);
  Key* T = reinterpret_cast<Key*>(buf);
  const int tid = (int)threadIdx.x;
  const uint2* mt = mw + (tid >> 5);
  const uint32_t low = map_low(tid);
  const ull blk = blockIdx.x;
  if (blk >= tp[nb]) return;
  const ull a = nb == 1 ? 0 : uniform(block_upper<SP_NT>(tp, (ull)nb, blk) - 1);
  const ull t0 = uniform(tp[a]), nt = uniform(tp[a + 1]) - t0, t = blk - t0;
  const ull v0 = uniform(boff[a]) + t * (ull)tk;
  const ull left = uniform(boff[a + 1]) - v0;
  const int m = left < (ull)tk ? (int)left : tk;
  Key kr[Q];
  if (SRC == SPLIT_RUNS) {
    if (!in.M) {
#pragma unroll
      for (int j = 0; j < Q; j++) {
        const int i = tid + j * SP_NT;
        if (i < m) kr[j] = Sin[v0 + i];
      }
    } else {
      const RunBucket rb = uniform(run_bucket(in, a));
      const ull f = rb.e0 + (rb.nt > SP_NT ? block_upper<SP_NT>(in.V + rb.e0, rb.nt, v0) - 1 : 0);
      constexpr int CAP = SP_TILE_BYTES / 8;
      ull* delta = reinterpret_cast<ull*>(buf);
      auto src = [&](ull e) { return rb.base + tile_place(in, e - rb.e0) + (in.M[e] >> 16); };
      const int np = map_pieces<SP_NT>(mw, nw, CAP, in.V, f, rb.e0 + rb.nt, v0, m, src,
                                       [&](uint32_t r, ull d, ull) { delta[r] = d; });
#pragma unroll
      for (int j = 0; j < Q; j++) {
        const int i = tid + j * SP_NT;
        if (i < m) {
          ull p;
          if (np <= CAP) {
            p = delta[map_piece(mt[j * (SP_NT / 32)], low)] + (ull)i;
          } else {
            const ull e = find_piece(in.V, f, rb.e0 + rb.nt, v0 + i);
            p = src(e) + (v0 + i - in.V[e]);
          }
          kr[j] = Sin[p];
        }
      }
    }
  } else {
    // level 1: the reads of these windows
    const ull f = block_upper<SP_NT>(ws.kofs, ws.R, v0) - 1;
    constexpr int CAP = SP_TILE_BYTES / 12;
    ull* delta = reinterpret_cast<ull*>(buf);
    uint32_t* aux = reinterpret_cast<uint32_t*>(buf + 8 * CAP);  // v0 - kofs (mod 2^32)
    auto src = [&](ull r) { return ws.rstart[r]; };
    const int np = map_pieces<SP_NT>(mw, nw, CAP, ws.kofs, f, ws.R, v0, m, src, [&](uint32_t r, ull d, ull idx) {
      delta[r] = d;
      aux[r] = (uint32_t)(v0 - ws.kofs[idx]);
    });
#pragma unroll
    for (int j = 0; j < Q; j++) {
      const int i = tid + j * SP_NT;
      if (i < m) {
        ull p;
        uint32_t wi;  // index of the window in its read
        if (np <= CAP) {
          const uint32_t r = map_piece(mt[j * (SP_NT / 32)], low);
          p = delta[r] + (ull)i;
          wi = aux[r] + (uint32_t)i;
        } else {
          const ull r = find_piece(ws.kofs, f, ws.R, v0 + i);
          p = ws.rstart[r] + (v0 + i - ws.kofs[r]);
          wi = (uint32_t)(v0 + i - ws.kofs[r]);
        }
        Key k = window_key<Key>(ws, p + (ull)(ws.K - 1));
        // the word holds the last 4 * sizeof(kmer_t) bases since the read's
        // start
        const uint32_t bases = wi + (uint32_t)ws.K;
        if (bases < 4u * (uint32_t)sizeof(Key)) k &= (Key(1) << (2 * bases)) - 1;
        kr[j] = k;
      }
    }
  }
  __syncthreads();
  const int ns = 1 << db;
  for (int i = tid; i < ns; i += SP_NT) h[i] = 0;
  __syncthreads();
  // each key's rank inside its digit, two 16-bit ranks per register
  uint32_t rk[Q / 2] = {};
#pragma unroll
  for (int j = 0; j < Q; j++)
    if (tid + j * SP_NT < m) rk[j / 2] |= atomicAdd(&h[key_digit<Key>(kr[j], dpos, db)], 1u) << (16 * (j & 1));
  __syncthreads();
  {
    static_assert((1 << SP_MAX_BITS) == 2 * SP_NT, "two digits per thread");
    const int d = 2 * tid;
    const uint32_t c0 = d < ns ? h[d] : 0u, c1 = d + 1 < ns ? h[d + 1] : 0u;
    uint32_t tot;
    const uint32_t ex = block_scan_u32<SP_NT>(c0 + c1, nw, &tot);
    const ull mo = (t0 << db) + (ull)d * nt + t;
    if (d < ns) {
      h[d] = ex;
      M[mo] = ex << 16 | c0;
    }
    if (d + 1 < ns) {
      h[d + 1] = ex + c0;
      M[mo + nt] = (ex + c0) << 16 | c1;
    }
  }
  __syncthreads();
  // place of every key in the sorted tile
#pragma unroll
  for (int j = 0; j < Q; j++)
    if (tid + j * SP_NT < m) rk[j / 2] += h[key_digit<Key>(kr[j], dpos, db)] << (16 * (j & 1));
  for (int r0 = 0; r0 < m; r0 += ROUND) {
#pragma unroll
    for (int j = 0; j < Q; j++) {
      if (tid + j * SP_NT < m) {
        const uint32_t p = ((rk[j / 2] >> (16 * (j & 1))) & 0xFFFFu) - (uint32_t)r0;
        if (p < (uint32_t)ROUND) T[p] = kr[j];
      }
    }
    __syncthreads();
    const int c = m - r0 < ROUND ? m - r0 : ROUND;
    Key* o = Sout + v0 + r0;
    for (int p = tid; p < c; p += SP_NT) o[p] = T[p];
    __syncthreads();
  }
}

// Level 1 of the main path: tile t is the bytes [t * 16384 * WPT, ...), its
// keys the k-mers that end there (bits of W).  Three passes: a thread ranks
// the k-mers that end at its own 16 * WPT bytes by digit, cut from WPT words
// of E and the words before them at constant shifts; it notes each one's end
// (15 bits, and the exact low bit) at its place in the sorted order; then
// consecutive threads cut consecutive keys of that order out of the tile's
// packed bases (in LDS) and store them.  The order takes two bytes per key
// instead of the key, so one round covers the tile, and bytes that end no
// k-mer cost only the first two passes.  Bound by VALU: with whole keys
// exchanged through LDS in rounds it issued 115 lane instructions per one-word
// key and took 783 us for 2.5e8 keys, now 498.  (WPT = 2 at eight waves spills one
// vector register.)
constexpr int SM_NT = 1024;

template <class Key, int WPT>
__global__ __launch_bounds__(SM_NT, 8) void k_split_main(const uint32_t* __restrict__ E,
                                                         const uint32_t* __restrict__ RX,
                                                         const uint16_t* __restrict__ W, const ull* __restrict__ tb,
                                                         ull nblk, ull nwords, Key mask, int dpos, int db,
                                                         uint32_t* __restrict__ M, Key* __restrict__ Sout,
                                                         ull* __restrict__ boff, ull* __restrict__ tp) {
  constexpr int NW = (int)sizeof(Key) / 4;
  constexpr int P = 16 * WPT;
  static_assert(NL_PER_BLOCK == 16ull * SM_NT, "a word of E per thread and index block");
  static_assert(SM_NT == 1 << SP_MAX_BITS, "a digit per thread");
  static_assert(SM_NT * P <= 32768, "15 bits of place");
  __shared__ uint16_t order[SM_NT * P];
  __shared__ uint32_t es[SM_NT * WPT + NW];  // E from NW words before the tile
  __shared__ uint32_t h[1 << SP_MAX_BITS];
  __shared__ uint32_t nw[SM_NT / 64 + 1];
  const int tid = (int)threadIdx.x;
  const ull t = blockIdx.x, nt = gridDim.x;
  const ull v0 = uniform(tb[t * WPT]);
  if (t == 0 && tid < 2) {
    // one parent bucket (k_tiles_one's facts)
    boff[tid] = tid ? tb[nblk] : 0;
    tp[tid] = tid ? nt : 0;
  }
  const ull t1 = (t + 1) * WPT < nblk ? (t + 1) * WPT : nblk;
  const int m = (int)(uniform(tb[t1]) - v0);
  const ull w0 = t * (SM_NT * WPT);  // the tile's first word
  const ull w = w0 + (ull)(tid * WPT);
  uint32_t val = 0, rx = 0;
  if (w < nblk * SM_NT) val = W[w];
  if (WPT == 2 && w + 1 < nblk * SM_NT) val |= (uint32_t)W[w + 1] << 16;
  uint32_t ew[NW + WPT] = {};
  if (val) {
#pragma unroll
    for (int i = 0; i < NW + WPT; i++) ew[i] = E[PK_PAD + w - NW + i];
    rx = RX[w] & 0xFFFFu;
    if (WPT == 2) rx |= RX[w + 1] << 16;
  }
  const int ns = 1 << db;
  if (tid < ns) h[tid] = 0;
  // the tile's words for the last pass (a k-mer that ends here may start in
  // words whose own bytes end none)
  for (int i = tid; i < SM_NT * WPT + NW; i += SM_NT)
    if (w0 + i < nwords + NW) es[i] = E[PK_PAD + w0 - NW + i];
  // digit words: dw holds the stream E shifted down by dpos bits, so that the
  // digit of the k-mer that ends at byte j lies at the constant bit position
  // of byte j in it
  uint32_t dw[WPT + 1];
  {
    const int q = dpos >> 5, sh = dpos & 31;
#pragma unroll
    for (int i = 0; i <= WPT; i++) {
      // dw[i] = bits of words c - q - 1, c - q for c = NW + WPT - 1 - i
      const int c = NW + WPT - 1 - i;
      uint32_t hi = 0, lo = 0;
#pragma unroll
      for (int x = 0; x < NW; x++) {
        if (x == q) {
          if (c - x >= 0) lo = ew[c - x];
          if (c - x - 1 >= 0) hi = ew[c - x - 1];
        }
      }
      dw[i] = __builtin_amdgcn_alignbit(hi, lo, (uint32_t)sh);
    }
  }
  const uint32_t dm = (1u << db) - 1u;
  auto digit = [&](int j) -> uint32_t {
    const int i = WPT - 1 - (j >> 4);
    return __builtin_amdgcn_alignbit(dw[i + 1], dw[i], 30u - 2u * (uint32_t)(j & 15)) & dm;
  };
  __syncthreads();
  uint32_t rk[P / 2] = {};
#pragma unroll
  for (int j = 0; j < P; j++)
    if ((val >> j) & 1u) rk[j / 2] |= atomicAdd(&h[digit(j)], 1u) << (16 * (j & 1));
  __syncthreads();
  {
    const uint32_t c = tid < ns ? h[tid] : 0u;
    uint32_t tot;
    const uint32_t ex = block_scan_u32<SM_NT>(c, nw, &tot);
    if (tid < ns) {
      h[tid] = ex;
      M[(ull)tid * nt + t] = ex << 16 | c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < P; j++) {
    if ((val >> j) & 1u)
      order[h[digit(j)] + ((rk[j / 2] >> (16 * (j & 1))) & 0xFFFFu)] =
          (uint16_t)((uint32_t)(tid * P + j) | ((rx >> j) & 1u) << 15);
  }
  __syncthreads();
  Key* o = Sout + v0;
  for (int p = tid; p < m; p += SM_NT) {
    const uint32_t s = order[p];
    const uint32_t e = s & 0x7FFFu;
    const uint32_t* x = es + (e >> 4);
    const uint32_t sh = 30u - 2u * (e & 15u);
    Key k = 0;
#pragma unroll
    for (int i = NW - 1; i >= 0; i--) {
      uint32_t u = __builtin_amdgcn_alignbit(x[NW - 1 - i], x[NW - i], sh);
      // the last base's low bit, without the next byte's spill
      if (i == 0) u = (u & ~1u) | s >> 15;
      k = (k << 31 << 1) | (Key)u;
    }
    o[p] = k & mask;
  }
}

// ---------------------------------------------------------------------------
// Rank-share routing of the reference's Sliding_window (kmer_counting.cpp:
// 2950-3050): a k-mer belongs to rank hash31(m) % P (retrieve_proc_id,
// distribute_kmers.cpp:95-105) of its leftmost minimum-frequency L-mer m
// (L = 8, frequencies of the whole input).  The reference tracks the minimum
// as the window slides: a new L-mer replaces it only when strictly rarer, and
// when it leaves the window every L-mer of the current k-mer is re-read from
// the packed k-mer (recalculate_min_lmer, :355-388).  The rolling L-mer that
// ends at byte e, A(e), has e's exact code; re-read, B(e), its last low bit
// also holds the next byte's third code bit.  So, with w = K - L + 1 and an end
// "dirty" when A != B:
//   - the first window of a read has the leftmost minimum of A over its w ends;
//   - a window without a dirty end but its own has the same, whatever came
//     before (the reference's state is the leftmost minimum over A or B of its
//     ends): k_own, all windows at once;
//   - the other windows depend on where the minimum was last re-read: from the
//     window before a run of them, which k_own gives, k_own_walk follows the
//     reference window by window.  Reads of A, C, G, T have none.
// The result is a bitmap of window ends like k_valid's, and the count goes on
// as on the main path.

constexpr int LMER_L = 8;
constexpr uint32_t LMER_BINS = 1u << (2 * LMER_L);
constexpr int LM_NT = 1024;
// index blocks whose L-mers a block adds before it looks for counters of
// 2^14 or more: three add less than 2^16 - 2^14 to any
constexpr int LM_FLUSH = 3;

// retrieve_proc_id before its % P (src/distribute_kmers.cpp:95-120): hash31
// (includes/distribute_kmers.h:856-873, signed 64-bit) and uhash31 (:836-854,
// unsigned 128-bit) both come to bits 0-30 plus bits 31-61 of a * x + b, which
// depend on x's low 64 bits alone.
__device__ __forceinline__ uint32_t owner_hash(ull x) {
  const ull v = 68111ull * x + 105929ull;
  return (uint32_t)((v >> 31) + v) & 2147483647u;
}

// h % P for h < 2^31 as h - ((h * m) >> s) * P.
struct OwnerMod {
  ull m;
  int s;
  uint32_t P, rank;
};

__device__ __forceinline__ bool owner_is(uint32_t h, const OwnerMod& o) {
  return h - (uint32_t)((ull)h * o.m >> o.s) * o.P == o.rank;
}

// A(e) for byte i of a word e1 of E (e0: the word before; rx: exact low bits)
__device__ __forceinline__ uint32_t lmer_at(uint32_t e0, uint32_t e1, uint32_t rx, int i) {
  const uint32_t b = __builtin_amdgcn_alignbit(e0, e1, 30u - 2u * (uint32_t)i) & 0xFFFFu;
  return (b & ~1u) | ((rx >> i) & 1u);
}

// L-mer frequencies (Sliding_window_l, kmer_counting.cpp:391-438): the L-mers
// that end at the set bits of W (k_valid's at K = L).  A block counts in LDS, 16
// bits per L-mer, and leaves its table in part; counters that grow past 2^14
// move to freq.  Bound by LDS atomics, one per
// L-mer (0.19 GB of reads of 100 bases: 83 us; a global atomic per L-mer took 7.7 ms).
__global__ __launch_bounds__(LM_NT) void k_lmer_count(const uint32_t* __restrict__ E, const uint32_t* __restrict__ RX,
                                                      const uint16_t* __restrict__ W, ull nb, uint32_t* part,
                                                      ull* freq) {
  static_assert(NL_PER_BLOCK == 16ull * LM_NT, "a word of E per thread and index block");
  static_assert(LM_FLUSH * NL_PER_BLOCK + (1u << 14) <= 1u << 16, "16-bit counters");
  __shared__ __align__(16) uint32_t h[LMER_BINS / 2];
  const int tid = (int)threadIdx.x;
  uint4* hv = reinterpret_cast<uint4*>(h);
  for (int i = tid; i < (int)LMER_BINS / 8; i += LM_NT) hv[i] = uint4{0, 0, 0, 0};
  __syncthreads();
  int since = 0;
  // an index block's words, loaded while the one before is counted
  uint32_t n0 = 0, n1 = 0, nr = 0, nv = 0;
  auto fetch = [&](ull b) {
    const ull w = b * LM_NT + tid;
    nv = b < nb ? W[w] : 0u;
    if (nv) {
      n0 = E[PK_PAD + w - 1];
      n1 = E[PK_PAD + w];
      nr = RX[w];
    }
  };
  fetch(blockIdx.x);
  for (ull b = blockIdx.x; b < nb; b += gridDim.x) {
    if (since == LM_FLUSH) {
      since = 0;
      __syncthreads();
      for (int i = tid; i < (int)LMER_BINS / 8; i += LM_NT) {
        const uint4 q = hv[i];
        if ((q.x | q.y | q.z | q.w) & 0xC000C000u) {
          const uint32_t v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
          for (int j = 0; j < 4; j++) {
            uint32_t keep = v[j];
            if (keep & 0xC000u) {
              atomicAdd(&freq[8 * i + 2 * j], (ull)(keep & 0xFFFFu));
              keep &= 0xFFFF0000u;
            }
            if (keep & 0xC0000000u) {
              atomicAdd(&freq[8 * i + 2 * j + 1], (ull)(keep >> 16));
              keep &= 0xFFFFu;
            }
            h[4 * i + j] = keep;
          }
        }
      }
      __syncthreads();
    }
    since++;
    const uint32_t val = nv, e0 = n0, e1 = n1, rx = nr;
    fetch(b + gridDim.x);
    if (val) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        if ((val >> i) & 1u) {
          const uint32_t l = lmer_at(e0, e1, rx, i);
          atomicAdd(&h[l >> 1], 1u << (16u * (l & 1u)));
        }
      }
    }
  }
  __syncthreads();
  uint4* o = reinterpret_cast<uint4*>(part + (ull)blockIdx.x * (LMER_BINS / 2));
  for (int i = tid; i < (int)LMER_BINS / 8; i += LM_NT) o[i] = hv[i];
}

// freq += the np tables of k_lmer_count: a block takes 64 words of each, its
// waves every sixteenth table.
__global__ __launch_bounds__(1024) void k_lmer_sum(const uint32_t* __restrict__ part, int np, ull* freq) {
  __shared__ uint32_t lo[16][64], hi[16][64];
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
  const uint32_t i = blockIdx.x * 64u + (uint32_t)lane;
  uint32_t a = 0, b = 0;  // at most np * 2^16
  for (int t = wv; t < np; t += 16) {
    const uint32_t v = part[(ull)t * (LMER_BINS / 2) + i];
    a += v & 0xFFFFu;
    b += v >> 16;
  }
  lo[wv][lane] = a;
  hi[wv][lane] = b;
  __syncthreads();
  if (wv < 2) {
    ull s = 0;
    for (int t = 0; t < 16; t++) s += wv ? hi[t][lane] : lo[t][lane];
    freq[2 * i + wv] += s;
  }
}

// The same from the bytes and a read table, where a budget has no room for the
// packed input: a thread per read, one global atomic per L-mer (0.19 GB: 7.7 ms).
__global__ void k_lmer_walk(const uint8_t* fa, const ull* rstart, const uint32_t* rlen, uint64_t R, ull* freq) {
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < R; r += (uint64_t)gridDim.x * blockDim.x) {
    const ull s = rstart[r];
    const uint32_t len = rlen[r];
    uint32_t lm = 0;
    for (uint32_t i = 0; i < len; i++) {
      lm = ((lm << 2) | base_code(fa[s + i])) & (LMER_BINS - 1);
      if (i >= (uint32_t)(LMER_L - 1)) atomicAdd(&freq[lm], 1ull);
    }
  }
}

// The routing compares frequencies only with each other, so k_own takes their
// ranks (the number of smaller ones, 16 bits) and holds all of them in LDS.
// Frequencies below 2^16 - 1 rank by a histogram of their values in one block's
// LDS, 16 bits a value (65536 equal ones carry into a value that none has);
// the others, few below 10^8 bases, are listed in big and compared by
// k_freq_big.  One block takes 47 us for the 65536, all of it latency; with the
// histogram by global atomics and a scan it was five launches and 60 us.
// own: bit l = L-mer l's k-mers are this rank's.
__global__ __launch_bounds__(1024) void k_freq_rank(const ull* __restrict__ freq, OwnerMod om, ull* big, ull* nbig,
                                                    uint16_t* __restrict__ rank, ull* __restrict__ own) {
  constexpr int PER = (int)LMER_BINS / 1024, WW = (int)LMER_BINS / 2 / 16;  // words per wave
  __shared__ __align__(16) uint32_t h[LMER_BINS / 2];
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t nb;
  const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int i = tid; i < (int)LMER_BINS / 8; i += 1024) reinterpret_cast<uint4*>(h)[i] = uint4{0, 0, 0, 0};
  if (tid == 0) nb = 0;
  __syncthreads();
  uint32_t z = 0;  // values of 0, small inputs' most frequent one
#pragma unroll 8
  for (int r = 0; r < PER; r++) {
    const ull f = freq[r * 1024 + tid];
    if (f == 0)
      z++;
    else if (f < LMER_BINS - 1)
      atomicAdd(&h[f >> 1], 1u << (16u * (uint32_t)(f & 1)));
    else
      big[atomicAdd(&nb, 1u)] = f;
  }
  const uint32_t zeros = (uint32_t)block_sum<1024>((ull)z);
  __syncthreads();
  // counts -> the number of smaller values, wave by wave
  uint32_t s = 0;
  for (int i = 0; i < WW; i += 64) {
    const uint32_t v = h[wv * WW + i + lane];
    s += (v & 0xFFFFu) + (v >> 16);
  }
  s = wave_scan_u32(s);
  if (lane == 63) wsum[wv] = s;
  __syncthreads();
  uint32_t carry = zeros;
  for (int i = 0; i < wv; i++) carry += wsum[i];
  for (int i = 0; i < WW; i += 64) {
    const uint32_t v = h[wv * WW + i + lane];
    const uint32_t t = (v & 0xFFFFu) + (v >> 16);
    const uint32_t x = wave_scan_u32(t);
    const uint32_t a = carry + x - t;
    h[wv * WW + i + lane] = (a & 0xFFFFu) | (a + (v & 0xFFFFu)) << 16;
    carry += __shfl(x, 63, 64);
  }
  __syncthreads();
#pragma unroll 8
  for (int r = 0; r < PER; r++) {
    const uint32_t l = (uint32_t)(r * 1024 + tid);
    const ull f = freq[l];
    if (f < LMER_BINS - 1) rank[l] = f ? (uint16_t)(h[f >> 1] >> (16u * (uint32_t)(f & 1))) : (uint16_t)0;
    const ull b = __ballot(owner_is(owner_hash(l), om));
    if (lane == 0) own[l / 64] = b;
  }
  if (tid == 0) *nbig = nb;
}

// ranks of the frequencies of 2^16 - 1 and more
__global__ void k_freq_big(const ull* freq, const ull* big, const ull* nbig, uint16_t* rank) {
  const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
  const ull m = *nbig;
  if (m == 0 || freq[l] < LMER_BINS - 1) return;
  const ull f = freq[l];
  ull r = LMER_BINS - m;
  for (ull i = 0; i < m; i++) r += big[i] < f;
  rank[l] = (uint16_t)r;
}

constexpr int OWN_NT = 512;
constexpr int OWN_HALO = 4;  // words before a window end's own that its ends reach
constexpr int OWN_EX = 9;    // exchanged words per thread
constexpr int OWN_TAB = (int)LMER_BINS / 2 + (int)LMER_BINS / 32;  // ranks, then owner bits
constexpr int own_lds = 4 * (OWN_TAB + OWN_NT * OWN_EX);

// Windows [e - w + 1, e] of L-mer ends, w = K - L + 1 in [BS, 2 BS) (BS = 16:
// up to 57): a thread takes the 16 ends of one word of E, looks their ranks up
// in LDS and takes minima from both ends of each block of BS of them.  A
// window's minimum is that of the rest of its first block (from the thread
// that holds it, through LDS), the whole blocks between and the first part of
// its last.  One block of 512 threads per CU holds the tables and stays for
// all its tiles; 4 threads of 512 only feed the next ones.  Bound by VALU, 33
// instructions per byte of input (0.19 GB of reads of 100 bases, w = 25: 272 us,
// 0.69 TB/s of input; a thread per read, walking twice, took 3.96 ms; 640
// threads or tiles of one wave gain nothing).
//   Wout: W without the ends of other ranks and the undecided ones; D: those.
template <int BS>
__global__ __launch_bounds__(OWN_NT) void k_own(const uint32_t* __restrict__ E, const uint32_t* __restrict__ RX,
                                                const uint16_t* __restrict__ W, ull words, ull nwords, int w,
                                                const uint4* __restrict__ tab, uint16_t* __restrict__ Wout,
                                                uint16_t* __restrict__ D) {
  extern __shared__ __align__(16) uint32_t own_dyn[];
  const uint16_t* rk = reinterpret_cast<const uint16_t*>(own_dyn);
  const uint32_t* ob = own_dyn + LMER_BINS / 2;
  uint32_t* ex = own_dyn + OWN_TAB;
  const int tid = (int)threadIdx.x;
  for (int i = tid; i < OWN_TAB / 4; i += OWN_NT) reinterpret_cast<uint4*>(own_dyn)[i] = tab[i];
  constexpr int OUT = OWN_NT - OWN_HALO;
  // a tile's words, loaded while the tile before is worked on
  uint32_t n0 = 0, n1 = 0, nr = 0, nv = 0;
  auto fetch = [&](ull t0) {
    const long long x = (long long)t0 + tid - OWN_HALO;
    if (x >= 0 && (ull)x < nwords) {
      n0 = E[PK_PAD + x - 1];
      n1 = E[PK_PAD + x];
      nr = RX[x];
    }
    nv = tid >= OWN_HALO && (ull)x < words ? W[x] : 0u;
  };
  fetch((ull)blockIdx.x * OUT);
  for (ull t0 = (ull)blockIdx.x * OUT; t0 < words; t0 += (ull)gridDim.x * OUT) {
    __syncthreads();  // the tables; the last tile's reads of ex
    const long long x = (long long)t0 + tid - OWN_HALO;
    const uint32_t e0 = n0, e1 = n1, rx = nr, val = nv;
    fetch(t0 + (ull)gridDim.x * OUT);
    // rank << 16 | place << 1 | owned, places from 2: the least is the
    // leftmost minimum (place 0: the window's first block, 1: those between)
    uint32_t pre[16], suf[16];
    uint32_t dirty = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const uint32_t b = __builtin_amdgcn_alignbit(e0, e1, 30u - 2u * (uint32_t)i);
      const uint32_t l = (b & 0xFFFEu) | ((rx >> i) & 1u);
      dirty = __builtin_amdgcn_alignbit(b ^ l, dirty, 1);
      pre[i] = (uint32_t)rk[l] << 16 | (((ob[l >> 5] >> (l & 31u)) & 1u) | (uint32_t)((i + 2) << 1));
      suf[i] = pre[i];
    }
    // (no window reaches past a line's end, so that the ends before one need not
    // be followed; the last lane, which does not see the next word, keeps its)
    const uint32_t rn = __shfl_down(rx, 1, 64);
    const uint32_t nl = (rx >> 16 | ((tid & 63) == 63 ? 0u : rn & 0x10000u)) >> 1;
    dirty = dirty >> 16 & ~nl;
#pragma unroll
    for (int i = 14; i >= 0; i--)
      if (i % BS != BS - 1) suf[i] = suf[i] < suf[i + 1] ? suf[i] : suf[i + 1];
#pragma unroll
    for (int i = 1; i < 16; i++)
      if (i % BS != 0) pre[i] = pre[i] < pre[i - 1] ? pre[i] : pre[i - 1];
    uint32_t* mine = ex + tid * OWN_EX;
    uint32_t om = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) om = __builtin_amdgcn_alignbit(suf[i], om, 1);
    om = om >> 16 | dirty << 16;
#pragma unroll
    for (int i = 0; i < 8; i++) mine[i] = __builtin_amdgcn_perm(suf[2 * i + 1], suf[2 * i], 0x07060302u);
    mine[8] = om;
    __syncthreads();
    if (tid < OWN_HALO || (ull)x >= words) continue;
    uint32_t out = 0, und = 0;
    if (val) {
      const uint16_t* exh = reinterpret_cast<const uint16_t*>(ex);
      // the windows start in place sh + q of the thread `far` before
      const int far = (w + 14) >> 4, sh = 16 * far - (w - 1);
      const uint16_t* xf = exh + (tid - far) * (2 * OWN_EX);
      uint32_t oms = ex[(tid - far) * OWN_EX + 8] & 0xFFFFu;
      if (far) oms |= ex[(tid - far + 1) * OWN_EX + 8] << 16;
      oms >>= sh;
      // first place of the thread o before, as a block between
      auto head = [&](int o) -> uint32_t {
        const uint32_t* y = ex + (tid - o) * OWN_EX;
        return y[0] << 16 | 2u | (y[8] & 1u);
      };
      // BS = 16: the whole words between, for starts in the thread `far`
      // before (mf) and in the next (mn)
      uint32_t mf = ~0u, mn = ~0u;
      if (BS == 16) {
        for (int o = 1; o < far; o++) {
          const uint32_t c = head(o);
          mn = mf;
          // an earlier word wins ties
          mf = mf >> 16 < c >> 16 ? mf : c;
        }
      }
      uint32_t mp = ~0u;  // BS < 16: the last whole block of the thread before
      if (BS < 16) {
        const uint32_t* y = ex + (tid - 1) * OWN_EX;
        const int i = 16 - BS;
        mp = ((i & 1) ? y[i / 2] & 0xFFFF0000u : y[i / 2] << 16) | 2u | ((y[8] >> i) & 1u);
      }
#pragma unroll
      for (int q = 0; q < 16; q++) {
        const int i = sh + q;
        const uint32_t c = (uint32_t)xf[i + (i < 16 ? 0 : 2 * OWN_EX - 16)] << 16 | ((oms >> q) & 1u);
        uint32_t m = ~0u;
        if (BS == 16) {
          m = i < 16 ? mf : mn;
        } else if (q - (w - 1) < (q / BS - 1) * BS) {
          const int b = (q / BS - 1) * BS;
          m = b < 0 ? mp : ((suf[b < 0 ? 0 : b] & 0xFFFF0001u) | 2u);
        }
        uint32_t v = pre[q] < c ? pre[q] : c;
        v = m < v ? m : v;
        out = __builtin_amdgcn_alignbit(v, out, 1);
      }
      out >>= 16;
      out &= val;
      // dirty ends among the w - 1 before a window's last
      u128 dm = (u128)(om >> 16) << 64;
      for (int o = 1; o <= OWN_HALO; o++) dm |= (u128)(ex[(tid - o) * OWN_EX + 8] >> 16) << (64 - 16 * o);
      const bool edge = w == 1;
      if (dm || edge) {
        const uint32_t before = x > 0 ? W[x - 1] >> 15 : 0u;
        const uint32_t first = val & ~(val << 1 | before);
        u128 near = w > 1 ? dm << 1 : 0;
        for (int c = 1; c < w - 1;) {
          const int sh = c < w - 1 - c ? c : w - 1 - c;
          near |= near << sh;
          c += sh;
        }
        und = (uint32_t)(near >> 64) & 0xFFFFu & val & ~first;
        out &= ~und;
        // K = L: the reference's first window has no L-mer yet but 0
        if (edge) out = (out & ~first) | ((ob[0] & 1u) ? first : 0u);
      }
    }
    Wout[x] = (uint16_t)out;
    D[x] = (uint16_t)und;
  }
}

// The undecided windows (see above): a thread follows the runs that start in
// its word, one after another.
__global__ void k_own_walk(const uint32_t* E, const uint32_t* RX, const uint16_t* D, ull words, int w,
                           const uint16_t* rank, const uint32_t* own, uint32_t* Wout) {
  const ull x = (ull)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= words) return;
  const uint32_t d = D[x];
  if (!d) return;
  const uint32_t before = x ? D[x - 1] >> 15 : 0u;
  auto lmer = [&](ull e, bool exact) -> uint32_t {
    const ull i = e >> 4;
    const uint32_t b =
        __builtin_amdgcn_alignbit(E[PK_PAD + i - 1], E[PK_PAD + i], 30u - 2u * (uint32_t)(e & 15)) & 0xFFFFu;
    return exact ? (b & ~1u) | ((RX[i] >> (e & 15)) & 1u) : b;
  };
  for (uint32_t st = d & ~(d << 1 | before); st; st &= st - 1) {
    ull j = x * 16 + (ull)(__ffs(st) - 1);
    // the window before: leftmost minimum of the rolling L-mers
    uint32_t ml = 0, mr = ~0u;
    int mp = 0;
    for (int i = 0; i < w; i++) {
      const uint32_t l = lmer(j - (ull)w + (ull)i, true), r = rank[l];
      if (r < mr) {
        mr = r;
        ml = l;
        mp = i - 1;
      }
    }
    for (; j < words * 16 && (D[j >> 4] >> (j & 15) & 1u); j++) {
      const uint32_t a = lmer(j, true), r = rank[a];
      if (mp < 0) {
        mr = ~0u;
        for (int i = 0; i < w; i++) {
          const uint32_t l = i == w - 1 ? a : lmer(j - (ull)(w - 1 - i), false), g = rank[l];
          if (g < mr) {
            mr = g;
            ml = l;
            mp = i;
          }
        }
      }
      if (r < mr) {
        mr = r;
        ml = a;
        mp = w - 1;
      }
      mp--;
      if (own[ml >> 5] >> (ml & 31u) & 1u) atomicOr(&Wout[j >> 5], 1u << (j & 31));
    }
  }
}

// The -p counters' rule (kmer_counting.cpp:1949-1950): the owner of a hash of
// the whole k-mer.
__global__ void k_own_key(const uint32_t* __restrict__ E, const uint32_t* __restrict__ RX,
                          const uint16_t* __restrict__ W, ull words, ull mask, OwnerMod om, uint16_t* __restrict__ Wout) {
  const ull x = (ull)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= words) return;
  const uint32_t val = W[x];
  uint32_t out = 0;
  if (val) {
    const uint32_t e0 = E[PK_PAD + x - 2], e1 = E[PK_PAD + x - 1], e2 = E[PK_PAD + x], rx = RX[x];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const uint32_t lo = __builtin_amdgcn_alignbit(e1, e2, 30u - 2u * (uint32_t)i);
      const uint32_t hi = __builtin_amdgcn_alignbit(e0, e1, 30u - 2u * (uint32_t)i);
      const ull key = ((ull)hi << 32 | (lo & ~1u) | ((rx >> i) & 1u)) & mask;
      out |= (uint32_t)owner_is(owner_hash(key), om) << i;
    }
  }
  Wout[x] = (uint16_t)(out & val);
}

// window ends per index block
__global__ __launch_bounds__(256) void k_bits_count(const ull* W, uint32_t* cnt) {
  static_assert(NL_PER_BLOCK == 64 * 256, "a word per thread");
  const ull s = block_sum<256>((ull)__popcll(W[(ull)blockIdx.x * 256 + threadIdx.x]));
  if (threadIdx.x == 0) cnt[blockIdx.x] = (uint32_t)s;
}


// ---------------------------------------------------------------------------
// Per-bucket count: LDS hash table of the bucket's distinct keys (64-bit CAS,
// double hashing; duplicates cost one atomic add), then a counting sort of
// the distinct keys by a 12-bit sub-digit into LDS, a per-sub-bin insertion
// sort (sub-bins hold ~1-2 distinct keys) and a coalesced write of the
// bucket's (key, count) pairs.  This is the reference's sort + run-length +
// merge + aggregate (kmer_counting.cpp:3057-3086, 254-352, 169-250) for the
// keys of one bucket.

// Blocks of 512 threads, as many waves per CU as the keys' registers allow.
// Batches of a whole bucket: a second batch costs a second run map and its
// barriers (k = 63, 1.5e8 keys: 2.46 ms with batches of 2048 against 1.41; k =
// 32, 2.5e8 keys of 3900 a bucket: 1.30 with 4096, 1.17 with 5120, both before
// double hashing).  Buckets up
// to a batch: fewer of them for the same keys (7.6e7 keys: 0.32 ms with 2300 a
// bucket, 0.26 with 4600), and two partition levels instead of three more often
// (2.9e9 two-word keys: 88.7 -> 82.4 ms).
template <class Key>
struct HashCfg;
template <>
struct HashCfg<uint64_t> {
  static constexpr int NT = 512;      // threads per block
  static constexpr int WAVES = 8;     // waves per SIMD the LDS allows (register cap follows)
  static constexpr int T = 2560;      // table slots (12 bytes each)
  static constexpr int LIMIT = 1920;  // distinct keys per task (load 0.75)
  static constexpr int SUB = 11;      // sub-bin bits of the ordering
  static constexpr int HB = 10;       // keys per thread and batch
  static constexpr float FILL = 2.6f;  // built-in instances per bucket: FILL * LIMIT at most, one batch
};
template <>
struct HashCfg<u128> {
  static constexpr int NT = 512;
  static constexpr int WAVES = 8;
  static constexpr int T = 1536;   // 20 bytes each
  static constexpr int LIMIT = 1152;
  static constexpr int SUB = 10;
  static constexpr int HB = 6;
  static constexpr float FILL = 2.6f;
};

// a 32-bit hash scaled to T slots
template <int T>
__device__ __forceinline__ uint32_t slot_of(uint32_t h) {
  return __umulhi(h, (uint32_t)T);
}
// Probes step by an odd number from the hash's low bits, so that keys that
// meet in a slot part ways (steps of one run into each other: 6.2e7 keys in
// tables 0.9 full 0.73 ms, with steps of one 2.6).  A step divisible by T's odd
// factor is back after T / 3 or T / 5 = 512 probes.
template <int T>
__device__ __forceinline__ uint32_t next_slot(uint32_t slot, uint32_t step) {
  const uint32_t s = slot + step;
  return s < (uint32_t)T ? s : s - (uint32_t)T;
}
__device__ __forceinline__ uint32_t probe_step(uint32_t h) { return (h & 255u) | 1u; }
// instances of a task that one block goes through more than once
constexpr uint64_t TASK_MAX_INSTANCES = 1u << 18;
// probe bound of an insert: a table too full to place a key within it sends the
// task to more passes.  48 places all keys of a table 0.8 full; a table that
// cannot hold its keys costs up to twice one that can (six times with steps of
// one and a bound of 256: 1.3e8 keys, 0.72 of them distinct, 3.1 ms; now 0.9).
// The bound of a pass that is one of several is longer: it may be the last.
constexpr int HASH_PROBES = 48, HASH_PROBES_MULTI = 128;
// a probe chain longer than STOP_AFTER slots re-reads the task's overflow
// flag every 8 probes: once one thread has found the table full, the others
// stop probing it (short chains, the usual case, never read it)
constexpr int STOP_AFTER = 8;

template <class Key>
struct HashTable;

// u64 keys are stored as themselves; EMPTY is a key outside the task.
template <>
struct HashTable<uint64_t> {
  static constexpr int T = HashCfg<uint64_t>::T;
  ull* hk;
  uint32_t* hc;
  ull empty;
  __device__ __forceinline__ void init(int tid, int nt) {
    for (int i = tid; i < T / 2; i += nt) reinterpret_cast<ulonglong2*>(hk)[i] = make_ulonglong2(empty, empty);
    for (int i = tid; i < T / 4; i += nt) reinterpret_cast<uint4*>(hc)[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  // returns false when no free slot is found within PROBES probes, or when a
  // long chain finds the table already reported full (*stop)
  // (a read before the CAS, as for u128 keys, was slower here: a new key
  // then waits on two LDS round trips)
  // one 32-bit product: the kernel is bound by issue, and a 64-bit one is
  // three quarter-rate instructions
  __device__ __forceinline__ static uint32_t hash(uint64_t k) {
    const uint32_t lo = (uint32_t)k, hi = (uint32_t)(k >> 32);
    return (lo ^ __builtin_amdgcn_alignbit(hi, hi, 13)) * 0x9E3779B1u;
  }
  __device__ __forceinline__ bool try_slot(uint32_t slot, uint64_t k) {
    const ull prev = atomicCAS(&hk[slot], empty, (ull)k);
    if (prev == empty || prev == (ull)k) {
      atomicAdd(&hc[slot], 1u);
      return true;
    }
    return false;
  }
  template <int PROBES>
  __device__ __forceinline__ bool insert(uint64_t k, const volatile int* stop) {
    const uint32_t h = hash(k), step = probe_step(h);
    uint32_t slot = slot_of<T>(h);
    for (int probe = 0; probe < STOP_AFTER; probe++) {
      if (try_slot(slot, k)) return true;
      slot = next_slot<T>(slot, step);
    }
#pragma unroll 1
    for (int probe = STOP_AFTER; probe < PROBES; probe++) {
      if ((probe & 7) == 0 && *stop) return false;
      if (try_slot(slot, k)) return true;
      slot = next_slot<T>(slot, step);
    }
    return false;
  }
  __device__ __forceinline__ bool used(int i) const { return hc[i] != 0u; }
  __device__ __forceinline__ uint64_t key(int i) const { return hk[i]; }
};

// u128 keys: claim by a 64-bit fingerprint that gives the low word back when
// the high word is known; the high word is stored beside it (20 bytes per
// slot with the count) and checked after the inserts (a fingerprint collision
// sends the task to the split path, which separates the two keys).
template <>
struct HashTable<u128> {
  static constexpr int T = HashCfg<u128>::T;
  static constexpr ull EMPTY = ~0ull;
  ull* hf;
  ull* hh;
  uint32_t* hc;
  // spread of the high word: two 32 x 32 -> 64 products.  Keys of a task that
  // differ in a few bases of the high word differ in about half the bits of
  // the products, which the low words of such keys do not match; other pairs
  // collide with probability ~2^-64.  A collision only costs time.
  __device__ __forceinline__ static ull spread(ull hi) {
    const ull a = (ull)(uint32_t)hi * 0x9e3779b1ull;
    const ull b = (ull)(uint32_t)(hi >> 32) * 0x85ebca77ull;
    return a ^ (b << 32 | b >> 32) ^ 0x2545f4914f6cdd1dull;
  }
  __device__ __forceinline__ static ull fp(u128 k) { return (ull)k ^ spread((ull)(k >> 64)); }
  __device__ __forceinline__ void init(int tid, int nt) {
    for (int i = tid; i < T / 2; i += nt) reinterpret_cast<ulonglong2*>(hf)[i] = make_ulonglong2(EMPTY, EMPTY);
    for (int i = tid; i < T / 4; i += nt) reinterpret_cast<uint4*>(hc)[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  // one more 32-bit product
  __device__ __forceinline__ static uint32_t hash(ull f) { return ((uint32_t)f ^ (uint32_t)(f >> 32)) * 0x9E3779B1u; }
  __device__ __forceinline__ static uint32_t home(ull f) { return slot_of<T>(hash(f)); }
  // a slot changes only once, from EMPTY to its fingerprint: a plain read
  // finds a repeated key or steps over another one without an atomic, and
  // only an empty slot is claimed by CAS (k = 64 bacterial: 2.73 -> 2.56 ms)
  __device__ __forceinline__ bool try_slot(uint32_t slot, ull f, u128 k) {
    ull prev = __hip_atomic_load(&hf[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (prev == EMPTY) {
      prev = atomicCAS(&hf[slot], EMPTY, f);
      if (prev == EMPTY) hh[slot] = (ull)(k >> 64);
    }
    if (prev == EMPTY || prev == f) {
      atomicAdd(&hc[slot], 1u);
      return true;
    }
    return false;
  }
  // the first probe: the home slot if it holds f or is claimed for it, else
  // -1 (the slot holds another fingerprint)
  __device__ __forceinline__ int try_home(u128 k, ull f) {
    const uint32_t slot = home(f);
    return try_slot(slot, f, k) ? (int)slot : -1;
  }
  // the rest, for a key whose home slot holds another fingerprint: the slot
  // that counts k, or -1 (table full, or reported full by another thread)
  template <int PROBES>
  __device__ __forceinline__ int insert_after_home(u128 k, ull f, const volatile int* stop) {
    const uint32_t h = hash(f), step = probe_step(h);
    uint32_t slot = next_slot<T>(slot_of<T>(h), step);
    for (int probe = 1; probe < STOP_AFTER; probe++) {
      if (try_slot(slot, f, k)) return (int)slot;
      slot = next_slot<T>(slot, step);
    }
#pragma unroll 1
    for (int probe = STOP_AFTER; probe < PROBES; probe++) {
      if ((probe & 7) == 0 && *stop) return -1;
      if (try_slot(slot, f, k)) return (int)slot;
      slot = next_slot<T>(slot, step);
    }
    return -1;
  }
  // after a barrier: does the slot that counted k hold k?
  __device__ __forceinline__ bool verify(int slot, u128 k) const { return hh[slot] == (ull)(k >> 64); }
  __device__ __forceinline__ u128 key(int i) const {
    const ull hi = hh[i];
    return (u128)hi << 64 | (u128)(hf[i] ^ spread(hi));
  }
};

template <class Key>
struct HashLds;
template <>
struct HashLds<uint64_t> {
  alignas(16) ull hk[HashCfg<uint64_t>::T];
  alignas(16) uint32_t hc[HashCfg<uint64_t>::T];
  __device__ __forceinline__ HashTable<uint64_t> table(ull empty) {
    HashTable<uint64_t> t;
    t.hk = hk;
    t.hc = hc;
    t.empty = empty;
    return t;
  }
  __device__ __forceinline__ uint64_t* out_keys() { return reinterpret_cast<uint64_t*>(hk); }
};
template <>
struct HashLds<u128> {
  alignas(16) ull hf[HashCfg<u128>::T];
  ull hh[HashCfg<u128>::T];  // with hf: room for T whole keys in the ordering
  alignas(16) uint32_t hc[HashCfg<u128>::T];
  __device__ __forceinline__ HashTable<u128> table(ull) {
    HashTable<u128> t;
    t.hf = hf;
    t.hh = hh;
    t.hc = hc;
    return t;
  }
  __device__ __forceinline__ u128* out_keys() { return reinterpret_cast<u128*>(hf); }
};

// A batch of a task's keys is gathered from its runs through a map (see
// map_pieces) that lies in the idle sub-bin array: a word pair per 32 places
// and RUN_CAP 32-bit run offsets from the parent's first tile (a task whose
// parent has 2^32 keys or more goes to the split path).  A batch with more
// runs than that is cut down to as many places as there is room.
constexpr int MAX_PASS_BITS = 4;
constexpr int RUN_CAP = 512;
constexpr int HASH_QUEUE = 1024;

constexpr int map_words(int batch) { return batch / 32 * 2 + RUN_CAP; }

template <class Key, bool MULTI>
struct HashShared {
  HashLds<Key> lds;
  // sub-bin starts of the ordering (and the end of the last); a batch's run map
  // before, which several passes over one batch keep apart
  alignas(16) uint32_t hs[(1 << HashCfg<Key>::SUB) + 4];
  alignas(8) uint32_t keep[MULTI ? map_words(HashCfg<Key>::NT * HashCfg<Key>::HB) : 2];
  __device__ __forceinline__ uint32_t* map() { return MULTI ? keep : hs; }
  uint32_t nw[HashCfg<Key>::NT / 64 + 1];
  int over;
  // u128: keys of the batch queued for their probe chains (place in the batch,
  // then the slot found, 0xFFFF for none)
  int qn;
  uint16_t hq[sizeof(Key) == 16 ? HASH_QUEUE : 1];
};

// The map of a batch built by the block's first wave alone (the others clear
// the hash table meanwhile): LDS operations of one wave stay in order, so it
// needs no barrier of its own.  The places are [b, b + m) of the task, offsets
// are from the parent's first tile.  Returns false when the runs do not fit;
// the map then points at the parent's first keys.
constexpr ull WAVE_MAP_RUNS = 4096;  // entries a wave looks through

__device__ __forceinline__ bool wave_map(uint2* mw, int nwords, uint32_t* off, const Runs& in, const RunBucket& rb,
                                         uint32_t b, int m) {
  const int lane = (int)threadIdx.x;
  const uint32_t nt = (uint32_t)rb.nt;
  const ull* V = in.V + rb.e0;
  const uint32_t* M = in.M + rb.e0;
  for (int w = lane; w < nwords; w += 64) mw[w].x = 0;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  uint32_t cnt = 0;
  // four chunks of 64 entries at a time, their loads in flight together
  for (uint32_t c4 = 0; c4 < nt; c4 += 256) {
    uint32_t vs[4], ve[4], so[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint32_t idx = c4 + 64 * q + lane;
      vs[q] = ve[q] = so[q] = 0;
      if (idx < nt) {
        vs[q] = (uint32_t)(V[idx] - rb.v0);
        ve[q] = (uint32_t)(V[idx + 1] - rb.v0);
        so[q] = (uint32_t)tile_place(in, idx) + (M[idx] >> 16) - vs[q];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const bool part = ve[q] > vs[q] && vs[q] < b + (uint32_t)m && ve[q] > b;
      const ull bal = __ballot(part);
      const uint32_t r = cnt + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
      if (part && r < (uint32_t)RUN_CAP) {
        off[r] = so[q] + b;
        const uint32_t ls = vs[q] > b ? vs[q] - b : 0u;
        atomicOr(&mw[ls >> 5].x, 1u << (ls & 31));
      }
      cnt += (uint32_t)__popcll(bal);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  // pieces before each word: consecutive words per lane
  const int wpl = (nwords + 63) / 64;
  uint32_t sum = 0;
  for (int i = 0; i < wpl; i++) {
    const int w = lane * wpl + i;
    if (w < nwords) sum += (uint32_t)__popc(mw[w].x);
  }
  uint32_t x = wave_scan_u32(sum) - sum;
  for (int i = 0; i < wpl; i++) {
    const int w = lane * wpl + i;
    if (w < nwords) {
      mw[w].y = x;
      x += (uint32_t)__popc(mw[w].x);
    }
  }
  if (cnt <= (uint32_t)RUN_CAP) return true;
  for (int w = lane; w < nwords; w += 64) mw[w] = make_uint2(1u, 0u);
  if (lane == 0) off[0] = 0;
  return false;
}

// Loads the keys at [b, b + m) of the task into kb (thread t: t, t + BS_NT,
// ...); returns m.  LIGHT (a task of at most TASK_MAX_INSTANCES keys and
// WAVE_MAP_RUNS runs): the map by the first wave, which sets over to 3 when the
// runs do not fit (kb then holds other keys of the parent).
template <class Key, bool RUNS, bool LIGHT, int HB>
__device__ __forceinline__ int load_batch(HashShared<Key, !LIGHT>& L, const Key* Sb, const Runs& in, const RunBucket& rb,
                                          ull b, Key (&kb)[HB]) {
  constexpr int BS_NT = HashCfg<Key>::NT;
  constexpr int BATCH = BS_NT * HB;
  static_assert(BATCH % 32 == 0 && map_words(BATCH) * 4 <= sizeof(L.hs), "the run map fits the sub-bins");
  if constexpr (!RUNS) {
#pragma unroll
    for (int j = 0; j < HB; j++) {
      const uint64_t idx = b + threadIdx.x + (uint64_t)j * BS_NT;
      kb[j] = idx < rb.n ? Sb[idx] : Key(0);
    }
    return rb.n - b < (ull)BATCH ? (int)(rb.n - b) : BATCH;
  } else {
    int m = rb.n - b < (ull)BATCH ? (int)(rb.n - b) : BATCH;
    uint2* mw = reinterpret_cast<uint2*>(L.map());
    uint32_t* off = L.map() + BATCH / 32 * 2;
    if constexpr (LIGHT) {
      if (threadIdx.x < 64 && !wave_map(mw, (m + 31) >> 5, off, in, rb, (uint32_t)b, m)) L.over = 3;
      __syncthreads();
    } else {
      const ull end = rb.e0 + rb.nt, vb = rb.v0 + b;
      const ull f = rb.e0 + (rb.nt > BS_NT ? block_upper<BS_NT>(in.V + rb.e0, rb.nt, vb) - 1 : 0);
      auto src = [&](ull e) { return tile_place(in, e - rb.e0) + (in.M[e] >> 16); };
      for (;;) {
        __syncthreads();  // the last map may still be read
        const int np = map_pieces<BS_NT>(mw, L.nw, RUN_CAP, in.V, f, end, vb, m, src,
                                         [&](uint32_t r, ull d, ull) { off[r] = (uint32_t)d; });
        if (np <= RUN_CAP) break;
        m = RUN_CAP;
      }
    }
    const uint2* mt = mw + (threadIdx.x >> 5);
    const uint32_t low = map_low((int)threadIdx.x);
#pragma unroll
    for (int j = 0; j < HB; j++) {
      const int i = (int)threadIdx.x + j * BS_NT;
      kb[j] = i < m ? Sb[off[map_piece(mt[j * (BS_NT / 32)], low)] + (uint32_t)i] : Key(0);
    }
    return m;
  }
}

// Counts one task: keys rb of S, which share their top `fixed` bits (fixed >=
// 1; top = the first of them).  Writes the task's unique (key, count) pairs
// in ascending order to R / C at rb.v0 and their number to *out_n, returns 0;
// 1 when the table is too small for the distinct keys, 2 on a u128
// fingerprint collision, 3 when a batch has too many runs, 4 when the task is
// left to MULTI untried.  With MULTI a task with too many distinct keys is
// processed in 2^s passes, pass p taking the keys whose next s bits equal p
// (s = 1, 2, ... up to MAX_PASS_BITS).  A task of more instances than
// TASK_MAX_INSTANCES takes all keys at once first, which costs a batch or two
// where they are distinct, and then as many passes as leave that number to each
// (1.4e7 equal keys of one bucket: 190 ms in 16 passes, 32 in one).  full: a
// table has been too small for it already, so that it starts with two passes or,
// if its keys fit one batch, with as many as leave a table 0.85 full if all are
// distinct; such a task's keys stay in registers over its passes.
template <class Key, bool RUNS, bool MULTI>
__device__ __forceinline__ int count_task(HashShared<Key, MULTI>& L, const Key* S, Key* R, int32_t* C, const Runs& in,
                                          const RunBucket& rb, bool top, int K, int fixed, bool full, ull* out_n) {
  constexpr int BS_NT = HashCfg<Key>::NT;
  constexpr int T = HashCfg<Key>::T;
  constexpr int PER = T / BS_NT;  // table slots per thread
  constexpr int HB = HashCfg<Key>::HB;
  constexpr int PROBES = MULTI ? HASH_PROBES_MULTI : HASH_PROBES;
  uint32_t* hs = L.hs;
  const uint32_t* map = L.map();
  const ull start = rb.v0, n = rb.n;
  const int rem = 2 * K - fixed;
  // EMPTY for u64 tables: a key whose top bit differs from the task's (all
  // keys of the task share that bit, so this value is not in the task)
  HashTable<Key> ht = L.lds.table((ull)(top ? Key(0) : Key(1) << (2 * K - 1)));
  const Key* Sb = S + (RUNS ? rb.base : start);
  const int max_s = !MULTI ? 0 : rem < MAX_PASS_BITS ? rem : MAX_PASS_BITS;
  ull out = 0;
  int s = 0, fail = 0;
  // a first try with all keys is pointless when there are too many of them
  if (!MULTI && (n > (ull)TASK_MAX_INSTANCES || rb.nt > WAVE_MAP_RUNS)) return 4;
  if (MULTI && full && max_s) {
    s = 1;
    while (n <= (ull)(BS_NT * HB) && s < max_s && (n >> s) > (ull)(T * 17 / 20)) s++;
  }
  // keys are loaded HB at a time into registers so that the global-load
  // latency is paid once per batch, not once per insert
  Key kb[HB];
  int m = 0;
  for (; s <= max_s; s++) {
    while (MULTI && s > 0 && s < max_s && (n >> s) > (ull)TASK_MAX_INSTANCES) s++;
    out = 0;
    fail = 0;
    for (int pass = 0; pass < (MULTI ? 1 << s : 1) && !fail; pass++) {
      auto mine = [&](Key k) { return !MULTI || (int)key_digit<Key>(k, rem - s, s) == pass; };
      if (threadIdx.x == 0) L.over = 0;
      ht.init(threadIdx.x, BS_NT);
      // (the first batch's map is built before the barrier that ends the
      // clearing)
      if (!RUNS || MULTI) __syncthreads();
      int ksl[HB];  // u128: the slot each key of the batch landed in, or -1 - its place in the queue
      bool clash = false;
      // over as read between two barriers of the last batch (the first wave
      // writes it while it makes the next batch's map): all threads leave
      // together
      int ov = 0;
      for (ull b = 0; b < n && !ov; b += m) {
        // (one batch: the keys are still there)
        if (!MULTI || (ull)m != n) m = load_batch<Key, RUNS, !MULTI, HB>(L, Sb, in, rb, b, kb);
        if constexpr (sizeof(Key) == 16) {
          // A wave runs each probe step as long as its slowest lane needs
          // it, so a batch goes in two phases: every key tries its home slot
          // (one probe, the common case), and the keys whose home slot holds
          // another fingerprint queue up and are then probed by all lanes
          // together, so a long chain holds up one queue round instead of
          // each of its lane's keys.
          if (threadIdx.x == 0) L.qn = 0;
          __syncthreads();
#pragma unroll
          for (int j = 0; j < HB; j++) {
            const int i = (int)threadIdx.x + j * BS_NT;
            if (i < m && mine(kb[j])) {
              const ull f = HashTable<u128>::fp(kb[j]);
              ksl[j] = 0;
              if (f == HashTable<u128>::EMPTY) {
                L.over = 1;
              } else {
                ksl[j] = ht.try_home(kb[j], f);
                if (ksl[j] < 0) {
                  const int q = atomicAdd(&L.qn, 1);
                  if (q < HASH_QUEUE) {
                    L.hq[q] = (uint16_t)i;
                    ksl[j] = -1 - q;
                  } else {
                    ksl[j] = ht.template insert_after_home<PROBES>(kb[j], f, &L.over);
                    if (ksl[j] < 0) L.over = 1;
                  }
                }
              }
            }
          }
          __syncthreads();
          const int nq = L.qn < HASH_QUEUE ? L.qn : HASH_QUEUE;
          for (int q = threadIdx.x; q < nq; q += BS_NT) {
            const int i = L.hq[q];
            ull o = b + (ull)i;
            if constexpr (RUNS)
              o = (ull)(map[BS_NT * HB / 32 * 2 + map_piece(reinterpret_cast<const uint2*>(map), i)] + (uint32_t)i);
            const u128 k = Sb[o];
            const int sl = ht.template insert_after_home<PROBES>(k, HashTable<u128>::fp(k), &L.over);
            if (sl < 0) L.over = 1;
            L.hq[q] = (uint16_t)sl;
          }
          __syncthreads();
          ov = L.over;
          // a key counted in a slot that holds another high word shares its
          // fingerprint with that key (ov == 0: every key has a slot)
          if (!ov) {
#pragma unroll
            for (int j = 0; j < HB; j++) {
              const int i = (int)threadIdx.x + j * BS_NT;
              if (i < m && mine(kb[j])) {
                const int sl = ksl[j] < 0 ? (int)L.hq[-1 - ksl[j]] : ksl[j];
                if (!ht.verify(sl, kb[j])) clash = true;
              }
            }
          }
          if (b + m < n) __syncthreads();
        } else {
#pragma unroll
          for (int j = 0; j < HB; j++) {
            const int i = (int)threadIdx.x + j * BS_NT;
            if (i < m && mine(kb[j]) && !ht.template insert<PROBES>(kb[j], &L.over)) L.over = 1;
          }
          if (b + m < n) {
            __syncthreads();
            ov = L.over;
            __syncthreads();
          }
        }
      }
      __syncthreads();
      if constexpr (sizeof(Key) == 16) {
        if (clash) L.over = 2;
        __syncthreads();
      }
      fail = L.over;
      __syncthreads();
      if (fail) break;
      // order the distinct keys: counting sort by the sub-digit below the
      // pass bits, then rank inside each sub-bin (one key on average)
      constexpr int SUB = HashCfg<Key>::SUB;
      const int r2 = rem - s;
      const int dbits = r2 < SUB ? r2 : SUB;
      const int dpos = r2 - dbits;
      const uint32_t dm = (1u << dbits) - 1u;
      auto sub_bin = [&](Key k) -> uint32_t {
        if constexpr (sizeof(Key) == 8) return (uint32_t)(k >> dpos) & dm;
        else return key_digit<Key>(k, dpos, dbits);
      };
      for (int i = threadIdx.x; i < (1 << SUB) / 4; i += BS_NT)
        reinterpret_cast<uint4*>(hs)[i] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
      Key rk[PER];
      uint32_t rc[PER], rd[PER];  // rd: sub-bin, index of the key inside it << 16
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const int slot = threadIdx.x + j * BS_NT;
        rc[j] = L.lds.hc[slot];
        if (rc[j]) {
          rk[j] = ht.key(slot);
          const uint32_t d = sub_bin(rk[j]);
          rd[j] = d | atomicAdd(&hs[d], 1u) << 16;
        }
      }
      __syncthreads();
      uint32_t nd;  // distinct keys of the pass
      {
        constexpr int BPT = (1 << SUB) / BS_NT;
        static_assert(BPT == 2 || BPT == 4, "bins per thread as one vector");
        uint32_t v[BPT];
        if constexpr (BPT == 4) {
          const uint4 q = reinterpret_cast<const uint4*>(hs)[threadIdx.x];
          v[0] = q.x;
          v[1] = q.y;
          v[2] = q.z;
          v[3] = q.w;
        } else {
          const uint2 q = reinterpret_cast<const uint2*>(hs)[threadIdx.x];
          v[0] = q.x;
          v[1] = q.y;
        }
        uint32_t sm = 0;
#pragma unroll
        for (int i = 0; i < BPT; i++) {
          const uint32_t t = v[i];
          v[i] = sm;
          sm += t;
        }
        const uint32_t ex = block_scan_u32<BS_NT>(sm, L.nw, &nd);
        if constexpr (BPT == 4)
          reinterpret_cast<uint4*>(hs)[threadIdx.x] = make_uint4(ex, ex + v[1], ex + v[2], ex + v[3]);
        else
          reinterpret_cast<uint2*>(hs)[threadIdx.x] = make_uint2(ex, ex + v[1]);
        if (threadIdx.x == 0) hs[1 << SUB] = nd;
      }
      __syncthreads();
      Key* ok = L.lds.out_keys();
      uint32_t* oc = L.lds.hc;
#pragma unroll
      for (int j = 0; j < PER; j++) {
        if (rc[j]) {
          const uint32_t pos = hs[rd[j] & 0xFFFFu] + (rd[j] >> 16);
          ok[pos] = rk[j];
          oc[pos] = rc[j];
        }
      }
      __syncthreads();
      char* Ro = reinterpret_cast<char*>(R + start + out);
      char* Co = reinterpret_cast<char*>(C + start + out);
      for (uint32_t i = threadIdx.x; i < nd; i += BS_NT) {
        const Key v = ok[i];
        const uint32_t d = sub_bin(v);
        // the sub-bin's slots: from its start to the next one's (the bins past
        // dm start at nd)
        const uint32_t a = hs[d], e = hs[d + 1];
        // the sub-bin's first three slots read at once (most hold one key),
        // the rest of a longer one one by one.  a < nd <= T, so a read past
        // the key array lands in the counts that follow it in the same LDS
        // struct, and only slots below e count.
        const Key w0 = ok[a], w1 = ok[a + 1], w2 = ok[a + 2];
        uint32_t p = a + (uint32_t)(w0 < v) + (uint32_t)(a + 1 < e && w1 < v) + (uint32_t)(a + 2 < e && w2 < v);
        for (uint32_t j = a + 3; j < e; j++) p += ok[j] < v;
        *reinterpret_cast<Key*>(Ro + p * (uint32_t)sizeof(Key)) = v;
        *reinterpret_cast<int32_t*>(Co + p * 4u) = (int32_t)oc[i];
      }
      out += nd;
      if (!MULTI) break;
      __syncthreads();
    }
    // too many distinct keys: once more with one more split bit; splitting
    // does not help a fingerprint collision
    if (!MULTI || fail != 1) break;
  }
  *out_n = out;
  return fail;
}

// What bounds it: VALU and LDS are each busy half of the time, and barriers
// between the phases hold the rest.  Of 1.35 ms for 2.5e8 one-word keys, 7.7e7
// distinct (timing copies): loads and map 0.69, inserts 0.23, ordering 0.27,
// writes 0.16.  Sub-bins, vector clears, a DPP scan and one packed register for
// (bin, index) took it from 1.51 to 1.34 ms; without the pass loops around the
// single pass no vector register spills (that moved 2.3 of 5.3 GB), which with
// larger batches gave 1.14, and probes by double hashing 1.00.  84 scalar registers
// are kept in vector lanes (66 for two-word keys): masks of the first eight
// probes, which are unrolled; without that there are 5, and it is slower (1.3e8
// keys, 0.72 distinct: 3.4 against 2.8 ms with the retry).  Two-word keys (1.5e8):
// 2.83 ms with 28-byte slots, 1.42 at 6 waves per SIMD, 1.14 at the 8 that fit,
// now 1.05.  256 or 1024 threads and 2048 to 6144 slots were within 10 % of each
// other; resident blocks that load the next bucket's keys early, or a map built by
// all waves, were slower.
//
// One block per bucket of `in`: tu[b] = the bucket's distinct keys, bstart[b]
// = where they are.  Buckets the table is too small for are left to the retry
// (a single pass needs fewer registers): tu = RETRY_FULL, or RETRY_UNTRIED.
constexpr long long RETRY_FULL = -2, RETRY_UNTRIED = -3;

template <class Key, bool RUNS>
__global__ __launch_bounds__(HashCfg<Key>::NT, HashCfg<Key>::WAVES) void k_bucket_hash(const Key* S, Key* R, int32_t* C,
                                                                            Runs in, int K, int fixed, long long* tu,
                                                                            ull* bstart) {
  __shared__ HashShared<Key, false> L;
  const ull task = blockIdx.x;
  const RunBucket rb = uniform(run_bucket(in, task));
  ull out = 0;
  int fail = 0;
  if (rb.n) {
    fail = 4;
    // (runs are reached by 32-bit offsets from the parent's first tile)
    if (!RUNS || in.boff[(task >> in.db) + 1] - rb.base < (1ull << 32))
      fail = count_task<Key, RUNS, false>(L, S, R, C, in, rb, (bool)((task >> (fixed - 1)) & 1), K, fixed, false,
                                          &out);
  }
  if (threadIdx.x == 0) {
    bstart[task] = rb.v0;
    tu[task] = fail == 0 ? (long long)out : fail == 1 ? RETRY_FULL : RETRY_UNTRIED;
  }
}

// The buckets left to it in several passes, every gridDim.x-th of the B buckets
// to a block (a list of them by atomics on one counter took 50 ns a bucket; eight
// neighbours to a block read their counts in whole lines, 20 us less for 2^20
// buckets, but the heavy buckets are neighbours: 8.8 ms against 1.3 for 2.1e7
// builder words); what still fails goes to ovf_list with tu = -1 for the
// host-driven split.  Bound by
// latency: two blocks per CU, 112 to 128 VGPRs with a batch's keys in registers.
// Bucket count of distinct-rich input, first try and this (before the tiled
// partition; loading the keys for every pass, the first of them the one that had
// failed already; now): 1.3e8 keys of 32 bases, 0.72 distinct, 3.3 / 8.7 / 2.8 ms;
// 6.9e7, all distinct, 2.7 / 5.6 / 1.8; 1.1e8 of 64 bases, 0.95 distinct, 6.5 /
// 12.4 / 4.6; 8.7e7, all distinct, 4.5 / 11.7 / 3.8.
template <class Key, bool RUNS>
__global__ __launch_bounds__(HashCfg<Key>::NT, 4) void k_bucket_retry(const Key* S, Key* R, int32_t* C, Runs in, ull B,
                                                                   int K, int fixed, long long* tu, ull* ovf_count,
                                                                   ull* ovf_list) {
  constexpr int NT = HashCfg<Key>::NT;
  __shared__ HashShared<Key, true> L;
  __shared__ uint32_t left[NT];  // place among the block's buckets << 1 | full
  __shared__ uint32_t nleft;
  for (ull c0 = 0; c0 * gridDim.x + blockIdx.x < B; c0 += NT) {
    if (threadIdx.x == 0) nleft = 0;
    __syncthreads();
    const ull t = (c0 + threadIdx.x) * gridDim.x + blockIdx.x;
    const long long u = t < B ? tu[t] : 0;
    if (u < -1) left[atomicAdd(&nleft, 1u)] = threadIdx.x << 1 | (u == RETRY_FULL ? 1u : 0u);
    __syncthreads();
    const uint32_t nq = nleft;
    for (uint32_t q = 0; q < nq; q++) {
      const uint32_t e = __builtin_amdgcn_readfirstlane(left[q]);
      const ull task = (c0 + (e >> 1)) * gridDim.x + blockIdx.x;
      const RunBucket rb = uniform(run_bucket(in, task));
      ull out = 0;
      int fail = 1;
      if (!RUNS || in.boff[(task >> in.db) + 1] - rb.base < (1ull << 32))
        fail = count_task<Key, RUNS, true>(L, S, R, C, in, rb, (bool)((task >> (fixed - 1)) & 1), K, fixed, e & 1u,
                                           &out);
      if (threadIdx.x == 0) {
        tu[task] = fail ? -1 : (long long)out;
        if (fail) ovf_list[atomicAdd(ovf_count, 1ull)] = task;
      }
    }
    __syncthreads();
  }
}

// Tasks of the split path: [tstart[i], tstart[i] + tcount[i]) of S.
template <class Key>
__global__ __launch_bounds__(HashCfg<Key>::NT) void k_task_hash(const Key* S, Key* R, int32_t* C, const ull* tstart,
                                                     const ull* tcount, int K, int fixed, long long* tu) {
  __shared__ HashShared<Key, true> L;
  const ull task = blockIdx.x;
  RunBucket rb{};
  rb.v0 = tstart[task];
  rb.n = tcount[task];
  ull out = 0;
  int fail = 0;
  if (rb.n) {
    const bool top = (bool)((uint32_t)(S[rb.v0] >> (2 * K - 1)) & 1u);
    fail = count_task<Key, false, true>(L, S, R, C, Runs{}, rb, top, K, fixed, false, &out);
  }
  if (threadIdx.x == 0) tu[task] = fail ? -1 : (long long)out;
}

// All keys of the task are identical (no bits left to split on).
template <class Key>
__global__ void k_single_key(const Key* S, Key* R, int32_t* C, const ull* tstart, const ull* tcount,
                             uint64_t ntasks, long long* tu) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ntasks) return;
  if (tcount[i] == 0) {
    tu[i] = 0;
    return;
  }
  R[tstart[i]] = S[tstart[i]];
  C[tstart[i]] = (int32_t)(uint32_t)tcount[i];
  tu[i] = 1;
}

// Split oversize tasks by the pbits-wide digit at bit pos (host-driven).
constexpr int PT_NT = 256;
constexpr int PT_PER = 4096;

template <class Key>
__global__ __launch_bounds__(PT_NT) void k_part_hist(const Key* S, const ull* tstart,
                                                     const ull* tcount, const uint32_t* blk_task,
                                                     const ull* blk_off, int pos, int pbits,
                                                     ull* th) {
  __shared__ uint32_t h[256];
  const int nb = 1 << pbits;
  for (int i = threadIdx.x; i < nb; i += PT_NT) h[i] = 0;
  __syncthreads();
  const uint32_t t = blk_task[blockIdx.x];
  const uint64_t s = tstart[t], n = tcount[t];
  const uint64_t off = blk_off[blockIdx.x];
  for (uint64_t i = off + threadIdx.x; i < n && i < off + PT_PER; i += PT_NT)
    atomicAdd(&h[key_digit<Key>(S[s + i], pos, pbits)], 1u);
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += PT_NT)
    if (h[i]) atomicAdd(&th[(uint64_t)t * 256 + i], (ull)h[i]);
}

template <class Key>
__global__ __launch_bounds__(PT_NT) void k_part_scatter(const Key* S, const ull* tstart,
                                                        const ull* tcount, const uint32_t* blk_task,
                                                        const ull* blk_off, int pos, int pbits,
                                                        ull* tcur, Key* T) {
  __shared__ uint32_t h[256];
  __shared__ ull base[256];
  const int nb = 1 << pbits;
  for (int i = threadIdx.x; i < nb; i += PT_NT) h[i] = 0;
  __syncthreads();
  const uint32_t t = blk_task[blockIdx.x];
  const uint64_t s = tstart[t], n = tcount[t];
  const uint64_t off = blk_off[blockIdx.x];
  for (uint64_t i = off + threadIdx.x; i < n && i < off + PT_PER; i += PT_NT)
    atomicAdd(&h[key_digit<Key>(S[s + i], pos, pbits)], 1u);
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += PT_NT)
    base[i] = h[i] ? atomicAdd(&tcur[(uint64_t)t * 256 + i], (ull)h[i]) : 0ull;
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += PT_NT) h[i] = 0;
  __syncthreads();
  for (uint64_t i = off + threadIdx.x; i < n && i < off + PT_PER; i += PT_NT) {
    const Key k = S[s + i];
    const uint32_t d = key_digit<Key>(k, pos, pbits);
    const uint32_t r = atomicAdd(&h[d], 1u);
    T[s + base[d] + r] = k;
  }
}

template <class Key>
__global__ void k_copy_tasks(Key* S, const Key* T, const ull* tstart, const ull* tcount,
                             const uint32_t* blk_task, const ull* blk_off) {
  const uint32_t t = blk_task[blockIdx.x];
  const uint64_t s = tstart[t], n = tcount[t];
  const uint64_t off = blk_off[blockIdx.x];
  for (uint64_t i = off + threadIdx.x; i < n && i < off + PT_PER; i += blockDim.x) S[s + i] = T[s + i];
}

// The runs of the listed buckets gathered at their virtual places: gridDim.x
// blocks per bucket (blockIdx.y), each every gridDim.x-th run.  Bound by the
// reads of the runs (3.6e7 builder words of 11 bases and more, 8 oversize buckets
// of 1300 runs: the whole split 3.4 ms, with one block per bucket 13.5).
constexpr unsigned GATHER_BLOCKS = 256;

template <class Key>
__global__ void k_gather_buckets(const Key* S, Runs in, const ull* buckets, Key* out) {
  const RunBucket rb = run_bucket(in, buckets[blockIdx.y]);
  for (ull t = blockIdx.x; t < rb.nt; t += gridDim.x) {
    const ull e = rb.e0 + t, v = in.V[e], c = in.V[e + 1] - v;
    const Key* src = S + rb.base + tile_place(in, t) + (in.M[e] >> 16);
    for (ull i = threadIdx.x; i < c; i += blockDim.x) out[v + i] = src[i];
  }
}

// Dense table from per-leaf results (leaves in key order).
template <class Key>
__global__ void k_compact(const Key* S, const int32_t* C, const ull* lstart, const long long* lu,
                          const ull* loff, uint64_t nleaves, Key* TK, int32_t* TC) {
  const uint64_t b = blockIdx.x;
  if (b >= nleaves) return;
  const long long u = lu[b];
  const uint64_t s = lstart[b], o = loff[b];
  for (long long i = threadIdx.x; i < u; i += blockDim.x) {
    TK[o + i] = S[s + i];
    TC[o + i] = C[s + i];
  }
}

// ---------------------------------------------------------------------------
// Cutoff (kmer_histogram.cpp:84-140).

constexpr int CUT_NT = 1024;
constexpr int T_MAX = 4096;
// A cutoff block covers CUT_R rounds of CUT_NT * 4 counts: in round r thread
// t reads the four at r * CUT_NT * 4 + 4 t (one 16-byte load, coalesced),
// and its loads of all rounds are in flight together.
constexpr int CUT_R = 4;
constexpr uint64_t CUT_PER = (uint64_t)CUT_R * CUT_NT * 4;

__device__ __forceinline__ void cut_load4(const int32_t* TC, uint64_t U, uint64_t base, int32_t fill,
                                          int32_t* v) {
  if (base + 4 <= U) {
    const int4 q = *reinterpret_cast<const int4*>(TC + base);
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    v[3] = q.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = base + i < U ? TC[base + i] : fill;
  }
}

__global__ __launch_bounds__(CUT_NT) void k_count_hist(const int32_t* TC, uint64_t U, int t, ull* hist) {
  __shared__ uint32_t h[T_MAX];
  for (int i = threadIdx.x; i < t; i += CUT_NT) h[i] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * CUT_PER;
  for (uint64_t i = base + threadIdx.x; i < U && i < base + CUT_PER; i += CUT_NT) {
    const int v = TC[i];
    if (v >= 0 && v < t) atomicAdd(&h[v], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < t; i += CUT_NT)
    if (h[i]) atomicAdd(&hist[i], (ull)h[i]);
}

// Small-t path (t <= CUT_SMALL_T): per-wave LDS sub-histograms (no
// contention between waves), the block's histogram stored to BH[b * t + c]
// without global atomics; column sums give hist, and the kept count of block
// b is its size minus its entries with count < min_bucket.
constexpr int CUT_SMALL_T = 64;

__global__ __launch_bounds__(CUT_NT) void k_count_hist_blocks(const int32_t* TC, uint64_t U, int t,
                                                             uint32_t* BH) {
  constexpr int NW = CUT_NT / 64;
  __shared__ uint32_t h[NW * CUT_SMALL_T];
  const int w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < NW * t; i += CUT_NT) h[i] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * CUT_PER + (uint64_t)threadIdx.x * 4;
  int32_t v[CUT_R * 4];
#pragma unroll
  for (int r = 0; r < CUT_R; r++) cut_load4(TC, U, base + (uint64_t)r * CUT_NT * 4, -1, v + 4 * r);
  // count 1 (the k-mers seen once, most of the table) is summed per wave by
  // ballot instead of 64 lanes hitting one LDS word
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < CUT_R * 4; i++) {
    const bool one = v[i] == 1 && t > 1;
    const unsigned long long m = __ballot(one);
    if (lane == 0 && m) atomicAdd(&h[w * t + 1], (uint32_t)__popcll(m));
    if (!one && v[i] >= 0 && v[i] < t) atomicAdd(&h[w * t + v[i]], 1u);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < t; c += CUT_NT) {
    uint32_t sum = 0;
#pragma unroll
    for (int q = 0; q < NW; q++) sum += h[q * t + c];
    BH[(uint64_t)blockIdx.x * t + c] = sum;
  }
}

// hist[c] = sum over blocks of BH[b * t + c]; one block per column
__global__ __launch_bounds__(1024) void k_hist_columns(const uint32_t* BH, uint64_t nb, int t, ull* hist) {
  const int c = blockIdx.x;
  ull s = 0;
  for (uint64_t b = threadIdx.x; b < nb; b += 1024) s += BH[b * t + c];
  s = block_sum<1024>(s);
  if (threadIdx.x == 0) hist[c] = s;
}

// kept[b] = block size - entries with count < min_bucket
__global__ void k_kept_from_hist(const uint32_t* BH, uint64_t nb, uint64_t U, int t, const int* mb,
                                 ull* kept) {
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int m = *mb;
  const uint64_t size = (b + 1) * CUT_PER <= U ? CUT_PER : U - b * CUT_PER;
  uint64_t below = 0;
  for (int c = 0; c < m && c < t; c++) below += BH[b * t + c];
  kept[b] = size - below;
}

// min_bucket = first argmin over hist[1..t-1]; an empty range gives t.
__device__ __forceinline__ int first_min(const ull* hist, int t) {
  int best = t;
  if (t > 1) {
    best = 1;
    for (int i = 2; i < t; i++)
      if (hist[i] < hist[best]) best = i;
  }
  return best;
}

__global__ void k_min_bucket(const ull* hist, int t, int* mb) {
  if (threadIdx.x || blockIdx.x) return;
  *mb = first_min(hist, t);
}

// The four steps from the blocks' histograms to their kept entries' places in
// one block, for up to CUT_PLAN blocks (a plasmid's cutoff is launches: each of
// the four is 2 to 3 us of work and as much of gap).  The threshold, the kept
// number and hn words of the histogram also go to box.
constexpr uint64_t CUT_PLAN = 1024;
__global__ __launch_bounds__(1024) void k_cut_plan(const uint32_t* __restrict__ BH, uint64_t nb, uint64_t U, int t,
                                                   ull* __restrict__ hist, int* __restrict__ mb,
                                                   ull* __restrict__ boffs, int hn, ull* __restrict__ box) {
  __shared__ ull h[CUT_SMALL_T];
  __shared__ int m;
  const int lane = threadIdx.x & 63;
  for (int c = (int)threadIdx.x >> 6; c < t; c += 16) {
    ull s = 0;
    for (uint64_t b = lane; b < nb; b += 64) s += BH[b * t + c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) {
      h[c] = s;
      hist[c] = s;
      if (c < hn) box[2 + c] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    m = first_min(h, t);
    *mb = m;
    box[1] = (ull)(uint32_t)m;
  }
  __syncthreads();
  const uint64_t b = threadIdx.x;
  ull kept = 0;
  if (b < nb) {
    kept = (b + 1) * CUT_PER <= U ? CUT_PER : U - b * CUT_PER;
    for (int c = 0; c < m && c < t; c++) kept -= BH[b * t + c];
  }
  const ull ex = block_excl_scan<1024>(kept);
  if (b < nb) boffs[b] = ex;
  if (b + 1 == nb) boffs[nb] = box[0] = ex + kept;
}

__global__ __launch_bounds__(CUT_NT) void k_kept_count(const int32_t* TC, uint64_t U, const int* mb,
                                                      ull* bsum) {
  const int thr = *mb;
  const uint64_t base = (uint64_t)blockIdx.x * CUT_PER + (uint64_t)threadIdx.x * 4;
  int32_t v[CUT_R * 4];
#pragma unroll
  for (int r = 0; r < CUT_R; r++) cut_load4(TC, U, base + (uint64_t)r * CUT_NT * 4, INT32_MIN, v + 4 * r);
  ull c = 0;
#pragma unroll
  for (int i = 0; i < CUT_R * 4; i++) c += v[i] >= thr;
  c = block_sum<CUT_NT>(c);
  if (threadIdx.x == 0) bsum[blockIdx.x] = c;
}

template <class Key>
__global__ __launch_bounds__(CUT_NT) void k_kept_write(const Key* TK, const int32_t* TC, uint64_t U,
                                                      const int* mb, const ull* boffs, Key* KK,
                                                      int32_t* KC) {
  // a block with no kept entry reads nothing (high cutoffs keep a few
  // thousand of a billion k-mers); the test is the same for every thread
  if (boffs[blockIdx.x + 1] == boffs[blockIdx.x]) return;
  const int thr = *mb;
  const uint64_t base = (uint64_t)blockIdx.x * CUT_PER + (uint64_t)threadIdx.x * 4;
  int32_t cv[CUT_R * 4];
#pragma unroll
  for (int r = 0; r < CUT_R; r++) cut_load4(TC, U, base + (uint64_t)r * CUT_NT * 4, INT32_MIN, cv + 4 * r);
  // the block's kept entries go out in index order: round by round, and in
  // a round by thread.  A thread's four round counts (<= 4 each, <= 4096
  // per round over the block) travel through one scan in 16-bit fields.
  ull packed = 0;
#pragma unroll
  for (int r = 0; r < CUT_R; r++) {
    ull c = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) c += cv[4 * r + i] >= thr;
    packed |= c << (16 * r);
  }
  ull tot;
  const ull ex = block_scan_total<CUT_NT>(packed, &tot);
  ull rbase = boffs[blockIdx.x];
#pragma unroll
  for (int r = 0; r < CUT_R; r++) {
    ull o = rbase + ((ex >> (16 * r)) & 0xFFFFull);
    const uint64_t b = base + (uint64_t)r * CUT_NT * 4;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (cv[4 * r + i] >= thr) {
        KK[o] = TK[b + i];
        KC[o] = cv[4 * r + i];
        o++;
      }
    }
    rbase += (tot >> (16 * r)) & 0xFFFFull;
  }
}

// ---------------------------------------------------------------------------
// Macro nodes (mn_construct.cpp:212-477).
//
// The kept table KK[0..V) is ascending.  pred(x) = x >> 2 is non-decreasing
// over it; within quarter a (first base a) succ(x) = x without its first base
// is ascending.  Node keys are the union of these five sorted lists (list 0:
// pred, lists 1..4: succ of the quarters), so every kept k-mer is one element
// of list 0 and one of its quarter's.
//
// Ranges of node keys go to blocks: range g starts at the node key of list
// 0's element g * MN_PC, and k_mn_bounds finds where it starts in each list.
// k_mn_rank puts a range's elements into sub-bins of its key span (a monotone
// map, about one node per bin), finds which element of equal ones comes first
// and ranks the nodes inside each bin; it stores every element's rank and the
// range's node count.  After the scan of the counts k_mn_write assembles each
// range's records in LDS at their ranks and stores them densely (4.6 Mbp, k =
// 32, 9.2e6 nodes, against a five-way merge by binary searches and a copy: 730
// -> 330 us, 12 + 162 + 152
// for the three kernels; k_mn_write moves 0.22 + 0.44 GB, 4.3 TB/s, k_mn_rank is
// bound by its chain of LDS phases).

constexpr int MN_NT = 512;
constexpr int MN_PC = 640;     // pred elements per range
constexpr int MN_PER = 3;      // elements per thread of a sub-range
constexpr int MN_CAP = MN_NT * MN_PER;
constexpr int MN_STEP = 256;   // elements per list of a sub-range that was cut down
constexpr int MN_BIN_BITS = 10;
constexpr int MN_BINS = 1 << MN_BIN_BITS;
constexpr int MN_ROUND = 640;  // records assembled at a time
static_assert(5 * MN_STEP <= MN_CAP, "a cut sub-range fits");
static_assert(MN_BINS == 2 * MN_NT, "two bins per thread");

template <class Key>
__device__ __forceinline__ Key mn_pred(Key x) { return x >> 2; }

// node key of element i of list l
template <class Key>
__device__ __forceinline__ Key mn_key(const Key* KK, int l, ull i, Key msk) {
  const Key x = KK[i];
  return l == 0 ? mn_pred(x) : (x & msk);
}

template <class Key>
__device__ __forceinline__ ull mn_lower(const Key* KK, ull lo, ull hi, Key x) {
  while (lo < hi) {
    const ull mid = (lo + hi) >> 1;
    if (KK[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// bd[l * (G + 1) + g] = where range g starts in list l (as an index of KK);
// one search per thread.
template <class Key>
__global__ __launch_bounds__(256) void k_mn_bounds(const Key* KK, ull V, int K, ull G, ull* bd) {
  const ull t = (ull)blockIdx.x * 256 + threadIdx.x;
  if (t >= 5 * (G + 1)) return;
  const int l = (int)(t / (G + 1));
  const ull g = t - (ull)l * (G + 1);
  ull r;
  if (l == 0) {
    r = g == G ? V : g * MN_PC;
    if (g > 0 && g < G) {
      // the first of the (up to four) elements of this node
      const Key s = mn_pred(KK[r]);
      while (r > 0 && mn_pred(KK[r - 1]) == s) r--;
    }
  } else if (g == G) {
    r = l == 4 ? V : mn_lower<Key>(KK, 0, V, Key(l) << (2 * K - 2));
  } else {
    const Key s = g == 0 ? Key(0) : mn_pred(KK[g * MN_PC]);
    r = mn_lower<Key>(KK, 0, V, (Key(l - 1) << (2 * K - 2)) | s);
  }
  bd[t] = r;
}

// The sub-ranges of a block's range, in key order: [lo[l], hi[l]) of the five
// lists, at most MN_CAP elements each; a range that fits is one sub-range.
struct MnSub {
  ull lo[5], hi[5], end[5];
};

// Advances to the next sub-range; false when there is none.  Called by the
// whole block with the same m; sh: five words of LDS.
template <class Key>
__device__ __forceinline__ bool mn_next(const Key* KK, Key msk, MnSub& m, ull* sh) {
  ull e = 0;
#pragma unroll
  for (int l = 0; l < 5; l++) {
    m.lo[l] = m.hi[l];
    e += m.end[l] - m.lo[l];
  }
  if (e == 0) return false;
  if (e <= (ull)MN_CAP) {
#pragma unroll
    for (int l = 0; l < 5; l++) m.hi[l] = m.end[l];
    return true;
  }
  // too many: up to the smallest of the keys MN_STEP further in the lists that
  // have more (at most MN_STEP elements of each list lie below it, and at
  // least MN_STEP - 3 of the list it comes from)
  Key cut = ~Key(0);
#pragma unroll
  for (int l = 0; l < 5; l++) {
    if (m.end[l] - m.lo[l] > (ull)MN_STEP) {
      const Key x = mn_key<Key>(KK, l, m.lo[l] + MN_STEP, msk);
      cut = x < cut ? x : cut;
    }
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < 5; l++) {
    if ((int)threadIdx.x == l) {
      ull a = m.lo[l], b = m.end[l] - a > (ull)MN_STEP ? a + MN_STEP : m.end[l];
      while (a < b) {
        const ull mid = (a + b) >> 1;
        if (mn_key<Key>(KK, l, mid, msk) < cut) a = mid + 1; else b = mid;
      }
      sh[l] = a;
    }
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < 5; l++) m.hi[l] = uniform(sh[l]);
  return true;
}

__device__ __forceinline__ MnSub mn_range(const ull* bd, ull G, ull g) {
  MnSub m;
#pragma unroll
  for (int l = 0; l < 5; l++) {
    m.lo[l] = m.hi[l] = uniform(bd[(ull)l * (G + 1) + g]);
    m.end[l] = uniform(bd[(ull)l * (G + 1) + g + 1]);
  }
  return m;
}

// Element e of a sub-range: its list and index of KK.
__device__ __forceinline__ void mn_element(const MnSub& m, uint32_t e, int& l, ull& i) {
  l = 0;
  uint32_t o = e, n = (uint32_t)(m.hi[0] - m.lo[0]);
  ull lo = m.lo[0];
#pragma unroll
  for (int q = 1; q < 5; q++) {
    if (l == q - 1 && o >= n) {
      o -= n;
      n = (uint32_t)(m.hi[q] - m.lo[q]);
      lo = m.lo[q];
      l = q;
    }
  }
  i = lo + o;
}

__device__ __forceinline__ uint32_t mn_size(const MnSub& m) {
  uint32_t e = 0;
#pragma unroll
  for (int l = 0; l < 5; l++) e += (uint32_t)(m.hi[l] - m.lo[l]);
  return e;
}

template <class Key>
__device__ __forceinline__ int bit_length(Key x) {
  if (sizeof(Key) == 16) {
    const ull hi = (ull)((u128)x >> 64);
    return hi ? 128 - __clzll((long long)hi) : 64 - __clzll((long long)(ull)x);
  }
  return 64 - __clzll((long long)(ull)x);
}

// Ranks: rkp[i] / rks[i] = place of KK[i]'s pred / succ node among its
// sub-range's nodes; ng[g] = nodes of range g.
template <class Key>
__global__ __launch_bounds__(MN_NT, 8) void k_mn_rank(const Key* KK, int K, const ull* bd, ull G, uint16_t* rkp,
                                                      uint16_t* rks, ull* ng) {
  __shared__ Key ok[MN_CAP];          // node keys, by bin
  __shared__ __align__(8) uint32_t h[MN_BINS + 1];  // elements per bin, then starts
  __shared__ __align__(8) uint32_t hd[MN_BINS];     // nodes per bin, then starts
  __shared__ uint8_t lead[MN_CAP];     // first of its equals
  __shared__ Key ext[10];
  __shared__ uint32_t nw[MN_NT / 64 + 1];
  __shared__ ull sh[5];
  const ull g = blockIdx.x;
  const Key msk = key_mask<Key>(2 * (K - 1));
  const int tid = (int)threadIdx.x;
  MnSub m = mn_range(bd, G, g);
  ull nodes = 0;
  while (mn_next<Key>(KK, msk, m, sh)) {
    const uint32_t E = mn_size(m);
    Key x[MN_PER];
    int l[MN_PER];
    ull idx[MN_PER];
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      const uint32_t e = (uint32_t)(tid + j * MN_NT);
      l[j] = 0;
      idx[j] = 0;
      x[j] = Key(0);
      if (e < E) {
        mn_element(m, e, l[j], idx[j]);
        x[j] = mn_key<Key>(KK, l[j], idx[j], msk);
      }
    }
    // the key span
#pragma unroll
    for (int q = 0; q < 5; q++) {
      if (tid == q) {
        const bool any = m.hi[q] > m.lo[q];
        ext[q] = any ? mn_key<Key>(KK, q, m.lo[q], msk) : ~Key(0);
        ext[5 + q] = any ? mn_key<Key>(KK, q, m.hi[q] - 1, msk) : Key(0);
      }
    }
    reinterpret_cast<uint2*>(h)[tid] = make_uint2(0u, 0u);
    reinterpret_cast<uint2*>(hd)[tid] = make_uint2(0u, 0u);
    __syncthreads();
    Key lo = ext[0], hi = ext[5];
#pragma unroll
    for (int q = 1; q < 5; q++) {
      lo = ext[q] < lo ? ext[q] : lo;
      hi = ext[5 + q] > hi ? ext[5 + q] : hi;
    }
    const int bl = bit_length<Key>(hi - lo);
    const int shift = bl > MN_BIN_BITS ? bl - MN_BIN_BITS : 0;
    uint32_t d[MN_PER], pos[MN_PER];
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      d[j] = 0;
      pos[j] = 0;
      if ((uint32_t)(tid + j * MN_NT) < E) {
        d[j] = (uint32_t)((x[j] - lo) >> shift);
        pos[j] = atomicAdd(&h[d[j]], 1u);
      }
    }
    __syncthreads();
    uint32_t tot;
    {
      const uint2 c = reinterpret_cast<const uint2*>(h)[tid];
      const uint32_t ex = block_scan_u32<MN_NT>(c.x + c.y, nw, &tot);
      reinterpret_cast<uint2*>(h)[tid] = make_uint2(ex, ex + c.x);
      if (tid == 0) h[MN_BINS] = E;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      if ((uint32_t)(tid + j * MN_NT) < E) {
        pos[j] += h[d[j]];
        ok[pos[j]] = x[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      if ((uint32_t)(tid + j * MN_NT) < E) {
        bool first = true;
        for (uint32_t q = h[d[j]]; q < pos[j]; q++) first = first && ok[q] != x[j];
        lead[pos[j]] = first ? 1 : 0;
        if (first) atomicAdd(&hd[d[j]], 1u);
      }
    }
    __syncthreads();
    {
      const uint2 c = reinterpret_cast<const uint2*>(hd)[tid];
      const uint32_t ex = block_scan_u32<MN_NT>(c.x + c.y, nw, &tot);
      reinterpret_cast<uint2*>(hd)[tid] = make_uint2(ex, ex + c.x);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      if ((uint32_t)(tid + j * MN_NT) < E) {
        uint32_t r = hd[d[j]];
        const uint32_t e = h[d[j] + 1];
        for (uint32_t q = h[d[j]]; q < e; q++) r += (uint32_t)(lead[q] && ok[q] < x[j]);
        (l[j] == 0 ? rkp : rks)[idx[j]] = (uint16_t)r;
      }
    }
    nodes += tot;
    __syncthreads();
  }
  if (tid == 0) ng[g] = nodes;
}

// Node record as written to memory (matches pk_mnode).
struct MnRec {
  ull key_lo, key_hi;
  int32_t pre[4];
  int32_t suf[4];
};

static_assert(sizeof(MnRec) == 48, "three 16-byte words");

// Records of range g at out + noff[g], from the elements' ranks.
template <class Key>
__global__ __launch_bounds__(MN_NT, 8) void k_mn_write(const Key* KK, const int32_t* KC, int K, const ull* bd, ull G,
                                                       const uint16_t* rkp, const uint16_t* rks, const ull* noff,
                                                       MnRec* out) {
  __shared__ ulonglong2 key[MN_ROUND];
  __shared__ uint4 cnt[MN_ROUND * 2];  // pre[4], suf[4] per record
  __shared__ uint32_t top;
  __shared__ ull sh[5];
  const ull g = blockIdx.x;
  const Key msk = key_mask<Key>(2 * (K - 1));
  const int tid = (int)threadIdx.x;
  MnSub m = mn_range(bd, G, g);
  ull base = uniform(noff[g]);
  while (mn_next<Key>(KK, msk, m, sh)) {
    const uint32_t E = mn_size(m);
    Key x[MN_PER];
    int32_t c[MN_PER];
    uint32_t r[MN_PER], f[MN_PER];
    if (tid == 0) top = 0;
    __syncthreads();
    uint32_t rmax = 0;
#pragma unroll
    for (int j = 0; j < MN_PER; j++) {
      const uint32_t e = (uint32_t)(tid + j * MN_NT);
      r[j] = 0xFFFFFFFFu;
      x[j] = Key(0);
      c[j] = 0;
      f[j] = 0;
      if (e < E) {
        int l;
        ull i;
        mn_element(m, e, l, i);
        const Key k = KK[i];
        c[j] = KC[i];
        r[j] = (l == 0 ? rkp : rks)[i];
        f[j] = l == 0 ? 4u + (uint32_t)(k & Key(3)) : (uint32_t)(l - 1);
        x[j] = l == 0 ? mn_pred(k) : (k & msk);
        rmax = r[j] + 1 > rmax ? r[j] + 1 : rmax;
      }
    }
    atomicMax(&top, rmax);
    __syncthreads();
    const uint32_t n = top;
    for (uint32_t r0 = 0; r0 < n; r0 += MN_ROUND) {
      for (int i = tid; i < 2 * MN_ROUND; i += MN_NT) cnt[i] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < MN_PER; j++) {
        const uint32_t p = r[j] - r0;
        if (r[j] != 0xFFFFFFFFu && p < (uint32_t)MN_ROUND) {
          key[p] = make_ulonglong2((ull)x[j], sizeof(Key) == 16 ? (ull)((u128)x[j] >> 64) : 0ull);
          reinterpret_cast<int32_t*>(cnt)[p * 8 + f[j]] = c[j];
        }
      }
      __syncthreads();
      const uint32_t w3 = 3 * (n - r0 < (uint32_t)MN_ROUND ? n - r0 : (uint32_t)MN_ROUND);
      uint4* o = reinterpret_cast<uint4*>(out + base + r0);
      for (uint32_t w = tid; w < w3; w += MN_NT) {
        const uint32_t q = w / 3, part = w - 3 * q;
        o[w] = part == 0 ? reinterpret_cast<const uint4*>(key)[q] : cnt[2 * q + part - 1];
      }
      __syncthreads();
    }
    base += n;
  }
}

// Initial wiring of one macro node per thread (MacroNode::setup_wiring,
// includes/distribute_kmers.h:550-656, after initiate_mnode_wiring appends
// the terminals, src/wire.cpp:84-96).  Entry lists: prefixes in the given
// base order, suffixes ascending, each followed by its terminal; counts are
// (count, visit) pairs.  The index sorts (Comp_rev: visit, then count,
// descending) run on at most five entries, where libstdc++'s std::sort is an
// insertion sort, i.e. stable -- so is the insertion sort here.
__device__ __forceinline__ void wire_sort(int* idx, int n, const int (*cnt)[2]) {
  for (int i = 1; i < n; i++) {
    const int v = idx[i];
    int j = i;
    while (j > 0) {
      const int u = idx[j - 1];
      const bool before = cnt[v][1] > cnt[u][1] || (cnt[v][1] == cnt[u][1] && cnt[v][0] > cnt[u][0]);
      if (!before) break;
      idx[j] = u;
      j--;
    }
    idx[j] = v;
  }
}

__global__ void k_mn_wire(const MnRec* nodes, uint64_t M, const uint8_t* pre_order, int cov,
                          pk_mnwire* out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  const MnRec r = nodes[i];
  int pc_[6][2], sc_[6][2];
  int np = 0, ns = 0;
  for (int q = 0; q < 4; q++) {
    int b = q;
    if (pre_order) {
      const uint8_t o = pre_order[i * 4 + q];
      if (o > 3) continue;
      b = o;
    }
    if (r.pre[b]) {
      pc_[np][0] = r.pre[b];
      pc_[np][1] = (r.pre[b] + cov - 1) / cov;
      np++;
    }
  }
  for (int b = 0; b < 4; b++)
    if (r.suf[b]) {
      sc_[ns][0] = r.suf[b];
      sc_[ns][1] = (r.suf[b] + cov - 1) / cov;
      ns++;
    }
  int pc = 0, sc = 0;
  for (int a = 0; a < np; a++) pc += pc_[a][1];
  for (int a = 0; a < ns; a++) sc += sc_[a][1];
  // terminals (count -1 in the reference until setup_wiring balances them)
  pc_[np][0] = 1;
  pc_[np][1] = sc - pc > 0 ? sc - pc : 0;
  sc_[ns][0] = 1;
  sc_[ns][1] = pc - sc > 0 ? pc - sc : 0;
  np++;
  ns++;
  int ip[6], is[6];
  for (int a = 0; a < np; a++) ip[a] = a;
  for (int a = 0; a < ns; a++) is[a] = a;
  wire_sort(ip, np, pc_);
  wire_sort(is, ns, sc_);
  pk_mnwire w;
  w.n_prefix = np;
  w.n_suffix = ns;
  w.pre_terminal_count[0] = pc_[np - 1][0];
  w.pre_terminal_count[1] = pc_[np - 1][1];
  w.suf_terminal_count[0] = sc_[ns - 1][0];
  w.suf_terminal_count[1] = sc_[ns - 1][1];
  for (int a = 0; a < 11; a++) w.wire[a] = pk_wire_info{0, 0, 0};
  for (int a = 0; a < 5; a++) w.prefix_begin[a][0] = w.prefix_begin[a][1] = 0;
  int off[6] = {0, 0, 0, 0, 0, 0};
  int leftover = sc + sc_[ns - 1][1];
  int top_p = 0, top_s = 0, var_p = 0, var_s = 0, wi = 0, p_size = 0, last_pid = -1, begin = -1;
  while (leftover > 0 && wi < 11 && top_p < np && top_s < ns) {
    const int sid = is[top_s], pid = ip[top_p];
    const int a = pc_[pid][1] - var_p, b = sc_[sid][1] - var_s;
    const int c = a < b ? a : b;
    w.wire[wi] = pk_wire_info{sid, off[sid], c};
    if (last_pid != pid) {
      begin = wi;
      last_pid = pid;
    }
    p_size++;
    wi++;
    leftover -= c;
    var_p += c;
    var_s += c;
    off[sid] += c;
    if (var_p == pc_[pid][1]) {
      var_p = 0;
      top_p++;
      if (pid < 5) {
        w.prefix_begin[pid][0] = begin;
        w.prefix_begin[pid][1] = p_size;
      }
      p_size = 0;
    }
    if (var_s == sc_[sid][1]) {
      var_s = 0;
      top_s++;
    }
  }
  w.n_wire = wi;
  out[i] = w;
}

// Macro-node share of rank `rank` at P ranks: nodes whose (k-1)-mer key is
// owned by the rank (retrieve_proc_id(pred / succ), mn_construct.cpp:
// 234-247; the rank receives every kept k-mer of its nodes,
// kmer_histogram.cpp:140-170, so its records are the one-rank records).
template <class Key>
__global__ void k_node_share_flags(const MnRec* nodes, uint64_t M, int P, int rank, uint32_t* flag) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  Key key;
  if (sizeof(Key) == 8) key = (Key)nodes[i].key_lo;
  else key = (Key)(((u128)nodes[i].key_hi << 64) | (u128)nodes[i].key_lo);
  flag[i] = (int)(owner_hash((ull)key) % (uint32_t)P) == rank ? 1u : 0u;
}

__global__ void k_node_share_write(const MnRec* nodes, uint64_t M, const uint32_t* flag, const ull* pos,
                                   MnRec* out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M || !flag[i]) return;
  out[pos[i]] = nodes[i];
}

// ---------------------------------------------------------------------------
// Host side.

namespace {

struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
};

enum BufId {
  B_FASTA, B_BLK, B_BLKOFF, B_NL, B_RSTART, B_RLEN, B_KC, B_KOFS, B_SMALL, B_BCNT, B_BOFF,
  B_S, B_C, B_TU, B_UOFF, B_TK, B_TC, B_HIST, B_KBS, B_KBOFF, B_KK, B_KC2, B_MNPLAN,
  B_MNNT, B_MNNG, B_MNNOFF, B_MNFLAG, B_NODES, B_TMP, B_OVF, B_PT0, B_PT1, B_PT2, B_PT3, B_PT4,
  B_PT5, B_PT6, B_BLKGT, B_S2, B_BOFF2, B_TP, B_TP2, B_HIST1, B_OFF1, B_HIST2, B_OFF2, B_PACK, B_WCNT, B_WOFF, B_CUTBH, B_LFREQ, B_LPART, B_LBIG, B_LRANK, B_LW, B_OWNW, B_OWNCNT, B_OWNOFF, B_WORDER, B_WIRE, B_NORM, B_NORMNL, B_NORMLEN, B_NORMOFF, B_NORMLS, B_NORMLL, B_SCAN0, B_SCAN1 = B_SCAN0 + 8, B_COUNT = B_SCAN0 + 16
};

}  // namespace

struct pk_ctx {
  int device = 0;
  int ncu = 256;  // compute units of the device
  hipStream_t stream = nullptr;
  uint64_t budget = 0;
  uint64_t held = 0;
  std::string err;
  DevBuf buf[B_COUNT];
  // buffers whose contents no work to come will read: given back when a
  // budget (or the device) has no room for another one
  bool idle[B_COUNT] = {};
  // 0-19: stage boundaries; 20 + 2 L, 21 + 2 L: around k_split of further
  // partition level L for the first MS_TIMED_LEVELS levels
  hipEvent_t ev[20 + 2 * MS_TIMED_LEVELS] = {};
  int ev_parsed = 1;  // the event at which the last count had its windows
  bool have_hist = false;  // the last count ran k_l1_hist
  int ms_levels = 0;  // further partition levels of the last count
  int ms_form[MS_TIMED_LEVELS] = {};  // their scatter forms (timed levels)
  pk_timing timing{};
  // state of the current table
  int k = 0;
  int words = 1;
  uint64_t U = 0, V = 0, M = 0, N = 0, R = 0;
  bool have_table = false, have_kept = false, have_nodes = false;
  int t = 0, mb = 0;
  int key_bits = 0;  // bits of a table key: 2k (main path) or the word (builder)
  // stages whose event times have not been read yet
  bool pend_count = false, pend_split = false, pend_cutoff = false, pend_mn = false;
  // BOX_WORDS words of pinned host memory that kernels leave results in
  ull* box = nullptr;
  // pinned staging of host input: PIN_THREADS host threads, two buffers each
  void* pin[8] = {};
  hipEvent_t pin_ev[8] = {};
  bool pin_used[8] = {};
  bool pend_norm = false;  // normalize_ms of the last pk_count_format
  uint64_t norm_n = 0;     // bytes of the last rewritten input (B_NORM)
  bool have_norm = false;
  pk_tuning tuning{};  // zeros: built-in choices
  // Scratch mode of pk_count_noalloc: need() carves buffers from `arena`
  // (the device's static scratch array) instead of allocating; the caller's
  // output arrays stand in for the table (ids marked in arena_fixed).
  bool arena_mode = false;
  char* arena = nullptr;
  uint64_t arena_cap = 0, arena_used = 0;
  bool arena_fixed[B_COUNT] = {};
  // the packed input sits at the top end of the arena until level 1 has read
  // it; arena_lim is where the other buffers must end meanwhile
  uint64_t arena_lim = 0;
  bool out_short = false;  // the caller's output arrays were too small
  bool no_pack = false;  // the packed input does not fit: level 1 walks the bytes
  uint8_t win_lut[256] = {};  // byte -> code of the last pk_builder_count_windows
  // buffers from the device's stream-ordered pool (pk_ctx_set_alloc_mode)
  bool stream_alloc = false;

  int fail(int code, const std::string& what) {
    err = what;
    return code;
  }
  int hip_fail(hipError_t e, const char* what) {
    err = std::string(what) + ": " + hipGetErrorString(e);
    return PK_EHIP;
  }
};

#define PK_HIP(ctx, x)                                   \
  do {                                                   \
    hipError_t e_ = (x);                                 \
    if (e_ != hipSuccess) return (ctx)->hip_fail(e_, #x); \
  } while (0)

#define PK_TRY(x)          \
  do {                     \
    int rc_ = (x);         \
    if (rc_) return rc_;   \
  } while (0)

namespace {

// Frees idle buffers until `bytes` more fit the budget (all of them without
// one); false when there were none.
bool reclaim(pk_ctx* c, uint64_t bytes) {
  bool any = false;
  for (int i = 0; i < B_COUNT; i++) {
    if (!c->idle[i] || !c->buf[i].p) continue;
    if (any && c->budget && c->held + bytes <= c->budget) break;
    if (!any) (void)hipStreamSynchronize(c->stream);
    any = true;
    (void)(c->stream_alloc ? hipFreeAsync(c->buf[i].p, c->stream) : hipFree(c->buf[i].p));
    c->held -= c->buf[i].cap;
    c->buf[i] = DevBuf{};
  }
  return any;
}

// A new count begins: the last results are void, and every buffer but its
// input is idle until the count asks for it.
void begin_buffers(pk_ctx* c) {
  for (int i = 0; i < B_COUNT; i++) c->idle[i] = i != B_FASTA && i != B_NORM;
}

template <class T>
int need(pk_ctx* c, int id, uint64_t count, T** out) {
  DevBuf& b = c->buf[id];
  c->idle[id] = false;
  const uint64_t bytes = count * sizeof(T) + 256;
  if (c->arena_mode) {
    if (c->arena_fixed[id]) {
      // a caller's output array: it must hold count entries (an empty
      // table asks for one entry and writes none)
      if (count * sizeof(T) > b.cap && !(count == 1 && c->U == 0)) {
        c->out_short = true;
        return c->fail(PK_ENOMEM, "output arrays hold fewer entries than the table (" + std::to_string(count) +
                                      " needed)");
      }
    } else if (b.cap < bytes) {
      const uint64_t take = (bytes + 255) & ~255ull;
      if (c->arena_used + take > c->arena_lim)
        return c->fail(PK_ENOMEM, "input needs more than the " + std::to_string(c->arena_cap >> 20) +
                                      " MiB scratch of pk_count_noalloc");
      b.p = c->arena + c->arena_used;
      b.cap = take;
      c->arena_used += take;
    }
    *out = reinterpret_cast<T*>(b.p);
    return PK_OK;
  }
  if (b.cap < bytes) {
    if (b.p) {
      // stream-ordered contexts free on their own stream: no device-wide wait
      hipError_t e = c->stream_alloc ? hipFreeAsync(b.p, c->stream) : hipFree(b.p);
      (void)e;
      c->held -= b.cap;
      b.p = nullptr;
      b.cap = 0;
    }
    if (c->budget && c->held + bytes > c->budget) {
      (void)reclaim(c, bytes);
      if (c->held + bytes > c->budget) return c->fail(PK_ENOMEM, "device budget exceeded");
    }
    void* p = nullptr;
    hipError_t e = c->stream_alloc ? hipMallocAsync(&p, bytes, c->stream) : hipMalloc(&p, bytes);
    if (e != hipSuccess && reclaim(c, bytes)) {
      (void)hipGetLastError();
      e = c->stream_alloc ? hipMallocAsync(&p, bytes, c->stream) : hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return c->fail(PK_ENOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    }
    b.p = p;
    b.cap = bytes;
    c->held += bytes;
  }
  *out = reinterpret_cast<T*>(b.p);
  return PK_OK;
}

inline unsigned grid_for(uint64_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

int fill_u64(pk_ctx* c, ull* p, ull v, uint64_t n) {
  if (!n) return PK_OK;
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, p, v, n);
  PK_HIP(c, hipGetLastError());
  return PK_OK;
}

// out[0..n) = exclusive scan of in, out[n] = total.  level selects scratch.
// With p the total and p's pieces (BOX_WORDS - 1 words at most, made by
// earlier work) are left in c->box; the caller waits.
template <class T>
int scan_excl(pk_ctx* c, const T* in, ull* out, uint64_t n, int level = 0, const Post* p = nullptr) {
  const Post none{};
  ull* box = p ? c->box : nullptr;
  if (n == 0) {
    PK_TRY(fill_u64(c, out, 0, 1));
    if (p) {
      c->box[0] = 0;
      hipLaunchKernelGGL(k_post, dim3(1), dim3(BOX_WORDS), 0, c->stream, *p, c->box + 1);
      PK_HIP(c, hipGetLastError());
    }
    return PK_OK;
  }
  if (level >= 8) return c->fail(PK_EINVAL, "scan too deep");
  const uint64_t nb = (n + SCAN_PER - 1) / SCAN_PER;
  ull* sums = nullptr;
  if (nb > 1) {
    PK_TRY(need(c, B_SCAN0 + level, nb + 1, &sums));
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_scan_reduce<T>), dim3((unsigned)nb), dim3(SCAN_NT), 0,
                       c->stream, in, sums, n);
    PK_HIP(c, hipGetLastError());
    if (nb > SCAN_ADD) PK_TRY(scan_excl<ull>(c, sums, sums, nb, level + 1));
  }
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_scan_apply<T>), dim3((unsigned)nb), dim3(SCAN_NT), 0, c->stream, in, out,
                     (const ull*)sums, nb > 1 && nb <= SCAN_ADD, n, p ? *p : none, box);
  PK_HIP(c, hipGetLastError());
  return PK_OK;
}

// Waits for the stream's work and then has the pieces' words in c->box.  One
// kernel that writes pinned memory: a copy into the caller's own (pageable)
// memory is a transfer and a wait of its own for each piece (a plasmid's
// count, cutoff and nodes: 542 us with eight copies, 419 without).
int fetch(pk_ctx* c, const Post& p) {
  int n = 0;
  for (int q = 0; q < 4; q++) n += p.n[q];
  if (n > BOX_WORDS) return c->fail(PK_EINVAL, "too many result words");
  hipLaunchKernelGGL(k_post, dim3(1), dim3((unsigned)((n + 63) / 64 * 64)), 0, c->stream, p, c->box);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipStreamSynchronize(c->stream));
  return PK_OK;
}

// scan_excl, then a wait: the total in c->box[0], p's pieces after it.
template <class T>
int scan_fetch(pk_ctx* c, const T* in, ull* out, uint64_t n, const Post& p) {
  PK_TRY(scan_excl<T>(c, in, out, n, 0, &p));
  PK_HIP(c, hipStreamSynchronize(c->stream));
  return PK_OK;
}

int d2h(pk_ctx* c, void* dst, const void* src, size_t bytes) {
  if (bytes && bytes <= BOX_WORDS * sizeof(ull) && bytes % 8 == 0 && reinterpret_cast<uintptr_t>(src) % 8 == 0) {
    PK_TRY(fetch(c, Post{{static_cast<const ull*>(src)}, {(int)(bytes / 8)}}));
    memcpy(dst, c->box, bytes);
    return PK_OK;
  }
  PK_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
  PK_HIP(c, hipStreamSynchronize(c->stream));
  return PK_OK;
}

// Bucket bits: at least 1 (the hash table's EMPTY value flips the top key
// bit), and enough that a bucket holds at most `factor` times cap_keys
// instances (a bucket with more distinct keys than a table holds takes extra
// passes).
int choose_bits(uint64_t N, int K, int cap_keys, float factor) {
  int b = 1;
  const uint64_t target = (uint64_t)((double)cap_keys * factor);
  while (b < 24 && b < 2 * K && (N >> b) > target) b++;
  return b;
}


struct Leaf {
  ull start;
  long long u;
};

// Recursively split oversize tasks (contiguous ranges of S; T is scratch of
// S's size); returns the leaves (in key order) for
// each input task.
template <class Key>
int resolve_overflow(pk_ctx* c, Key* S, Key* T, Key* R, int32_t* C, int K, int fixed_bits,
                     const std::vector<ull>& starts, const std::vector<ull>& counts,
                     std::vector<std::vector<Leaf>>& leaves) {
  constexpr int CAP = HashCfg<Key>::LIMIT;
  leaves.assign(starts.size(), {});
  const int rem = 2 * K - fixed_bits;
  if (rem <= 0) {
    // all keys of every task are identical
    const uint64_t nt = starts.size();
    ull *ts, *tc;
    long long* tu;
    PK_TRY(need(c, B_PT0, nt, &ts));
    PK_TRY(need(c, B_PT1, nt, &tc));
    PK_TRY(need(c, B_PT2, nt, &tu));
    PK_HIP(c, hipMemcpyAsync(ts, starts.data(), nt * 8, hipMemcpyHostToDevice, c->stream));
    PK_HIP(c, hipMemcpyAsync(tc, counts.data(), nt * 8, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_single_key<Key>), dim3(grid_for(nt, 256)), dim3(256), 0,
                       c->stream, S, R, C, ts, tc, nt, tu);
    PK_HIP(c, hipGetLastError());
    std::vector<long long> hu(nt);
    PK_TRY(d2h(c, hu.data(), tu, nt * 8));
    for (size_t i = 0; i < nt; i++) leaves[i].push_back(Leaf{starts[i], hu[i]});
    return PK_OK;
  }
  // digit width for this level
  ull maxn = 0;
  for (auto n : counts) maxn = std::max<ull>(maxn, n);
  int pbits = 1;
  while (pbits < 8 && (maxn >> pbits) > (ull)(CAP / 2)) pbits++;
  if (pbits > rem) pbits = rem;
  const int pos = rem - pbits;
  // block map
  std::vector<uint32_t> bt;
  std::vector<ull> bo;
  for (size_t t = 0; t < starts.size(); t++)
    for (ull o = 0; o < counts[t]; o += PT_PER) {
      bt.push_back((uint32_t)t);
      bo.push_back(o);
    }
  const uint64_t nt = starts.size(), nblk = bt.size();
  ull *ts, *tc, *bo_d, *th;
  uint32_t* bt_d;
  PK_TRY(need(c, B_PT0, nt, &ts));
  PK_TRY(need(c, B_PT1, nt, &tc));
  PK_TRY(need(c, B_PT3, nblk, &bt_d));
  PK_TRY(need(c, B_PT4, nblk, &bo_d));
  PK_TRY(need(c, B_PT5, nt * 256, &th));
  PK_HIP(c, hipMemcpyAsync(ts, starts.data(), nt * 8, hipMemcpyHostToDevice, c->stream));
  PK_HIP(c, hipMemcpyAsync(tc, counts.data(), nt * 8, hipMemcpyHostToDevice, c->stream));
  PK_HIP(c, hipMemcpyAsync(bt_d, bt.data(), nblk * 4, hipMemcpyHostToDevice, c->stream));
  PK_HIP(c, hipMemcpyAsync(bo_d, bo.data(), nblk * 8, hipMemcpyHostToDevice, c->stream));
  PK_TRY(fill_u64(c, th, 0, nt * 256));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_part_hist<Key>), dim3((unsigned)nblk), dim3(PT_NT), 0,
                     c->stream, S, ts, tc, bt_d, bo_d, pos, pbits, th);
  PK_HIP(c, hipGetLastError());
  std::vector<ull> hh(nt * 256);
  PK_TRY(d2h(c, hh.data(), th, nt * 256 * 8));
  std::vector<ull> cur(nt * 256, 0);
  std::vector<ull> sub_start, sub_count;
  std::vector<std::pair<size_t, int>> owner;  // (task, digit)
  for (size_t t = 0; t < nt; t++) {
    ull o = 0;
    for (int d = 0; d < (1 << pbits); d++) {
      cur[t * 256 + d] = o;
      if (hh[t * 256 + d]) {
        sub_start.push_back(starts[t] + o);
        sub_count.push_back(hh[t * 256 + d]);
        owner.push_back({t, d});
      }
      o += hh[t * 256 + d];
    }
  }
  PK_HIP(c, hipMemcpyAsync(th, cur.data(), nt * 256 * 8, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_part_scatter<Key>), dim3((unsigned)nblk), dim3(PT_NT), 0,
                     c->stream, S, ts, tc, bt_d, bo_d, pos, pbits, th, T);
  PK_HIP(c, hipGetLastError());
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_copy_tasks<Key>), dim3((unsigned)nblk), dim3(PT_NT), 0,
                     c->stream, S, T, ts, tc, bt_d, bo_d);
  PK_HIP(c, hipGetLastError());
  // sort the sub-tasks that fit
  const int fixed2 = fixed_bits + pbits;
  const uint64_t ns = sub_start.size();
  ull *ss, *sc;
  long long* su;
  PK_TRY(need(c, B_PT6, ns * 3 + 2, &ss));
  sc = ss + ns;
  su = reinterpret_cast<long long*>(ss + 2 * ns);
  PK_HIP(c, hipMemcpyAsync(ss, sub_start.data(), ns * 8, hipMemcpyHostToDevice, c->stream));
  PK_HIP(c, hipMemcpyAsync(sc, sub_count.data(), ns * 8, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_task_hash<Key>), dim3((unsigned)ns), dim3(HashCfg<Key>::NT), 0, c->stream, S, R, C, ss,
                     sc, K, fixed2, su);
  PK_HIP(c, hipGetLastError());
  std::vector<long long> hu(ns);
  PK_TRY(d2h(c, hu.data(), su, ns * 8));
  std::vector<ull> o_start, o_count;
  std::vector<size_t> o_idx;
  for (size_t i = 0; i < ns; i++)
    if (hu[i] < 0) {
      o_start.push_back(sub_start[i]);
      o_count.push_back(sub_count[i]);
      o_idx.push_back(i);
    }
  std::vector<std::vector<Leaf>> sub_leaves(ns);
  if (!o_start.empty()) {
    std::vector<std::vector<Leaf>> rec;
    PK_TRY(resolve_overflow<Key>(c, S, T, R, C, K, fixed2, o_start, o_count, rec));
    for (size_t j = 0; j < o_idx.size(); j++) sub_leaves[o_idx[j]] = rec[j];
  }
  for (size_t i = 0; i < ns; i++) {
    auto& dst = leaves[owner[i].first];
    if (hu[i] >= 0) dst.push_back(Leaf{sub_start[i], hu[i]});
    else dst.insert(dst.end(), sub_leaves[i].begin(), sub_leaves[i].end());
  }
  return PK_OK;
}

// Index of the event bytes ('\n', or '\n' and '>') of fa: *m events at
// *ev_out; *p0_out = the position of the first '>' (n when there is none).
// small[0] is scratch for the pass that looks for it in every block.
// With pk the input is packed on the way (builder encoding).
struct Packed {
  uint32_t* E = nullptr;
  uint32_t* RX = nullptr;
  ull* W = nullptr;  // main path: valid window ends
};

int event_index(pk_ctx* c, const uint8_t* fa, uint64_t n, uint8_t e0, uint8_t e1, ull* small,
                ull** ev_out, uint64_t* m_out, uint64_t* p0_out, int ev_buf = B_NL, int follow = 0,
                const Packed* pk = nullptr) {
  hipStream_t st = c->stream;
  const uint64_t nb = (n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
  ull *blk, *blkoff, *nl, *blkgt;
  PK_TRY(need(c, B_BLK, nb, &blk));
  PK_TRY(need(c, B_BLKGT, nb + 1, &blkgt));
  PK_TRY(need(c, B_BLKOFF, nb + 1, &blkoff));
  if (nb) {
    if (pk)
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pack<ENC_BUILDER>), dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, e0, e1,
                         blk, blkgt, 0, pk->E, pk->RX, (ull*)nullptr);
    else
      hipLaunchKernelGGL(k_nl_count, dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, e0, e1, blk, blkgt, 0);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<ull>(c, blk, blkoff, nb));
  // a '>' in the first block is the input's first one (other blocks report
  // one only from their byte-wise tail, which comes after it)
  ull hm[2] = {0, ~0ull};
  PK_TRY(fetch(c, Post{{blkoff + nb, blkgt}, {1, nb ? 1 : 0}}));
  hm[0] = c->box[0];
  if (nb) hm[1] = c->box[1];
  if (hm[1] == ~0ull && nb > 1) {
    // no '>' in the first block: the first one anywhere (same counts again)
    hipLaunchKernelGGL(k_nl_count, dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, e0, e1, blk, blkgt, 1);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_min_reduce, dim3(1), dim3(1024), 0, st, blkgt, nb, small);
    PK_HIP(c, hipGetLastError());
    PK_TRY(d2h(c, &hm[1], small, 8));
  }
  const uint64_t m = hm[0];
  PK_TRY(need(c, ev_buf, m + 1, &nl));
  if (nb) {
    if (pk)
      hipLaunchKernelGGL(k_nl_write_rx, dim3((unsigned)nb), dim3(NL_NT), 0, st, pk->RX, n, blkoff, nl);
    else
      hipLaunchKernelGGL(k_nl_write, dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, e0, e1, blkoff, nl, follow);
    PK_HIP(c, hipGetLastError());
  }
  *ev_out = nl;
  *m_out = m;
  *p0_out = hm[1] == ~0ull ? n : hm[1];
  return PK_OK;
}

// The input rewritten into strict single-line FASTA (B_NORM, *out_n bytes).
int normalize_impl(pk_ctx* c, const uint8_t* in, uint64_t n, int fmt, const uint8_t** out_p, uint64_t* out_n) {
  hipStream_t st = c->stream;
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  // small[8] = first '>' (unused), [9] = first record line, [10] = first
  // malformed line, [11] = first over-long line
  PK_TRY(fill_u64(c, small + 8, ~0ull, 4));
  ull* nl;
  uint64_t m, p0;
  PK_TRY(event_index(c, in, n, '\n', '\n', small + 8, &nl, &m, &p0, B_NORMNL));
  // a last line without '\n' is a line; the empty tail after a final '\n' is not
  ull last_nl = 0;
  if (m) PK_TRY(d2h(c, &last_nl, nl + m - 1, 8));
  const uint64_t L = m + ((n > 0 && (m == 0 || last_nl + 1 < n)) ? 1 : 0);
  if (fmt == FMT_FASTQ && L % 4 != 0)
    return c->fail(PK_EFORMAT, "FASTQ input has " + std::to_string(L) + " lines, not a multiple of 4");
  uint32_t *olen, *llen;
  ull *ooff, *lstart;
  uint8_t* out;
  PK_TRY(need(c, B_NORMLEN, L + 1, &olen));
  PK_TRY(need(c, B_NORMOFF, L + 1, &ooff));
  PK_TRY(need(c, B_NORMLS, L + 1, &lstart));
  PK_TRY(need(c, B_NORMLL, L + 1, &llen));
  PK_TRY(need(c, B_NORM, n + L + 64, &out));
  if (L) {
    if (fmt == FMT_FASTA) {
      hipLaunchKernelGGL(k_fmt_first_record, dim3(grid_for(L, 256)), dim3(256), 0, st, in, n, nl, m, L, small + 9);
      PK_HIP(c, hipGetLastError());
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fmt_lines<FMT_FASTA>), dim3(grid_for(L, 256)), dim3(256), 0, st, in, n,
                         nl, m, L, small + 9, olen, lstart, llen, small + 10, small + 11);
    } else {
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fmt_lines<FMT_FASTQ>), dim3(grid_for(L, 256)), dim3(256), 0, st, in, n,
                         nl, m, L, small + 9, olen, lstart, llen, small + 10, small + 11);
    }
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, olen, ooff, L));
  PK_TRY(fetch(c, Post{{ooff + L, small + 10}, {1, 2}}));
  const ull hv[3] = {c->box[0], c->box[1], c->box[2]};
  if (hv[1] != ~0ull)
    return c->fail(PK_EFORMAT, "FASTQ record line " + std::to_string(hv[1]) +
                                   (hv[1] % 4 == 0 ? " does not start with '@'" : " does not start with '+'"));
  if (hv[2] != ~0ull) return c->fail(PK_EINVAL, "line " + std::to_string(hv[2]) + " longer than 4 GiB");
  if (hv[0]) {
    const unsigned ob = (unsigned)((hv[0] + FC_BYTES - 1) / FC_BYTES);
    if (fmt == FMT_FASTA)
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fmt_copy<FMT_FASTA>), dim3(ob), dim3(FC_NT), 0, st, in, n, lstart, llen,
                         olen, ooff, (ull)L, out);
    else
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fmt_copy<FMT_FASTQ>), dim3(ob), dim3(FC_NT), 0, st, in, n, lstart, llen,
                         olen, ooff, (ull)L, out);
    PK_HIP(c, hipGetLastError());
  }
  *out_p = out;
  *out_n = hv[0];
  return PK_OK;
}

// Where the packed input goes (pk stays empty when the scratch of
// pk_count_noalloc has no room for it).
int pack_buffers(pk_ctx* c, uint64_t n, bool valid, Packed* pk) {
  const uint64_t words = (n + 15) / 16, nb = (n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
  const uint64_t ew = (PK_PAD + words + 67) & ~63ull, rw = (words + 64 + 63) & ~63ull;
  const uint64_t vw = valid ? nb * (NL_PER_BLOCK / 64) * 2 : 0;  // W in 32-bit words
  const uint64_t bytes = 4 * (ew + rw + vw);
  uint32_t* p;
  if (c->arena_mode) {
    const uint64_t take = (bytes + 255) & ~255ull;
    if (c->no_pack || c->arena_used + take > c->arena_cap) {
      c->no_pack = true;
      return PK_OK;
    }
    c->arena_lim = c->arena_cap - take;
    p = reinterpret_cast<uint32_t*>(c->arena + c->arena_lim);
  } else {
    PK_TRY(need(c, B_PACK, bytes / 4, &p));
  }
  pk->E = p;
  pk->RX = p + ew;
  if (valid) pk->W = reinterpret_cast<ull*>(p + ew + rw);
  return PK_OK;
}

// The read table of a count: start byte, length (rlen: only where a walk needs
// it), offsets of the reads' windows, and the packed input.
struct Records {
  ull* rstart = nullptr;
  uint32_t* rlen = nullptr;
  ull* kofs = nullptr;
  const ull* tb = nullptr;  // main path: window ends before each index block
  uint64_t n = 0;  // input bytes
  uint64_t R = 0, N = 0;
  bool part = false;  // one rank's windows only
  Packed pk;
};

int format_error(pk_ctx* c, ull r) {
  return c->fail(PK_EFORMAT,
                 "input is not strict single-line FASTA (record " + std::to_string(r) + " does not start with '>')");
}

int records_main(pk_ctx* c, const uint8_t* fa, uint64_t n, int K, Records* rec);

// The windows of the main path from the packed input: valid ends and their
// number per index block, no list of lines or reads.  W2: also the window ends
// of the L-mers.
int windows_main(pk_ctx* c, const uint8_t* fa, uint64_t n, int K, Records* rec, ull* W2 = nullptr) {
  hipStream_t st = c->stream;
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  // small[2] = first format error, [3] = a line may be too long, [4] = overflow
  // count, [6] .. [9] = k_lines' facts, [10] = first '>',
  // [11] = records of the L-mers
  const uint64_t nb = (n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
  if (!nb) {
    PK_TRY(fill_u64(c, small + 2, ~0ull, 1));
    PK_TRY(fill_u64(c, small + 3, 0, 3));
  }
  const Packed& pk = rec->pk;
  ull *blk, *blkoff, *blkgt, *tb;
  uint32_t* cnt;
  PK_TRY(need(c, B_BLK, nb, &blk));
  PK_TRY(need(c, B_BLKGT, nb + 1, &blkgt));
  PK_TRY(need(c, B_BLKOFF, nb + 1, &blkoff));
  PK_TRY(need(c, B_WCNT, nb, &cnt));
  PK_TRY(need(c, B_WOFF, nb + 1, &tb));
  rec->tb = tb;
  if (!nb) return PK_OK;
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pack<ENC_MAIN>), dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, (uint8_t)'\n',
                     (uint8_t)'\n', blk, blkgt, 0, pk.E, pk.RX, small);
  PK_HIP(c, hipGetLastError());
  if (nb > SCAN_PER) PK_TRY(scan_excl<ull>(c, blk, blkoff, nb));
  const bool check_long = n > 0xFFFFFFF0ull;
  if (check_long) {
    hipLaunchKernelGGL(k_long_lines, dim3(grid_for(nb, 256)), dim3(256), 0, st, blkoff, nb, small + 3);
    PK_HIP(c, hipGetLastError());
  }
  ull hs[8], N = 0, R2 = 0;
  // the first '>' is nearly always in the first block (blkgt[0]); else a
  // second pass looks for it everywhere
  const ull* gt = blkgt;
  for (int pass = 0;; pass++) {
    hipLaunchKernelGGL(k_lines, dim3(1), dim3(1024), 0, st, pk.RX, n,
                       (const ull*)(nb <= SCAN_PER && pass == 0 ? blk : nullptr), blkoff, nb, gt, K, W2 ? LMER_L : 0, small + 6,
                       small + 11);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_valid, dim3((unsigned)nb), dim3(NL_NT), 0, st, pk.RX, n, blkoff, small + 6, K, pk.W, cnt,
                       small + 2, LMER_L, (const ull*)(small + 11), W2);
    PK_HIP(c, hipGetLastError());
    PK_TRY(scan_fetch<uint32_t>(c, cnt, tb, nb, Post{{small + 2, small + 11}, {8, W2 ? 1 : 0}}));
    N = c->box[0];
    memcpy(hs, c->box + 1, sizeof(hs));
    R2 = W2 ? c->box[9] : 0;
    if (hs[7] < n || pass || nb == 1) break;
    hipLaunchKernelGGL(k_nl_count, dim3((unsigned)nb), dim3(NL_NT), 0, st, fa, n, (uint8_t)'\n', (uint8_t)'\n', blk,
                       blkgt, 1);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_min_reduce, dim3(1), dim3(1024), 0, st, blkgt, nb, small + 10);
    PK_HIP(c, hipGetLastError());
    gt = small + 10;
  }
  rec->R = hs[5];
  rec->N = N;
  // (the L-mers' records, if asked for, include the windows')
  if (hs[0] != ~0ull && hs[0] <= std::max<uint64_t>(rec->R, R2)) return format_error(c, hs[0]);
  if (check_long && hs[1]) {
    // the read table measures every line
    Records full;
    PK_TRY(records_main(c, fa, n, K, &full));
    PK_TRY(fill_u64(c, small + 4, 0, 2));
  }
  return PK_OK;
}

// Read table of the main path: records of the reference's Sliding_window.
int records_main(pk_ctx* c, const uint8_t* fa, uint64_t n, int K, Records* rec) {
  hipStream_t st = c->stream;
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  // small[0] = first '>', [1] = first unprocessed, [2] = first format error,
  // [3] = first over-long read, [4] = overflow count
  PK_TRY(fill_u64(c, small, ~0ull, 4));
  PK_TRY(fill_u64(c, small + 4, 0, 2));
  if (n >> NL_FLAG_SHIFT) return c->fail(PK_EINVAL, "input larger than 2^62 bytes");
  ull* nl;
  uint64_t m, p0;
  // entries carry what follows each '\n' (bits 62-63): only k_reads reads them
  PK_TRY(event_index(c, fa, n, '\n', '\n', small, &nl, &m, &p0, B_NL, 1));
  const uint64_t ncand = m / 2 + 2;
  ull *rstart, *kofs;
  uint32_t *rlen, *kc;
  PK_TRY(need(c, B_RSTART, ncand, &rstart));
  PK_TRY(need(c, B_RLEN, ncand, &rlen));
  PK_TRY(need(c, B_KC, ncand, &kc));
  PK_TRY(need(c, B_KOFS, ncand + 1, &kofs));
  hipLaunchKernelGGL(k_reads, dim3(grid_for(ncand, 256)), dim3(256), 0, st, n, nl, m, p0, K,
                     ncand, rstart, rlen, kc, small + 1, small + 2, small + 3);
  PK_HIP(c, hipGetLastError());
  PK_TRY(scan_excl<uint32_t>(c, kc, kofs, ncand));
  ull hs[4];
  PK_TRY(fetch(c, Post{{small + 1, kofs + ncand}, {3, 1}}));
  memcpy(hs, c->box, sizeof(hs));
  const uint64_t R = std::min<uint64_t>(hs[0], ncand);
  if (hs[1] != ~0ull && hs[1] <= R) return format_error(c, hs[1]);
  if (hs[2] != ~0ull && hs[2] < R) return c->fail(PK_EINVAL, "read longer than 4 GiB");
  rec->rstart = rstart;
  rec->rlen = rlen;
  rec->kofs = kofs;
  rec->R = R;
  rec->N = hs[3];
  return PK_OK;
}

// Read table of the builder API (bld_record).
// key_bases: bases of a key.
int records_builder(pk_ctx* c, const uint8_t* fa, uint64_t n, int klen, uint64_t read_len, BldSyms sy, int key_bases,
                    Records* rec) {
  hipStream_t st = c->stream;
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  PK_TRY(fill_u64(c, small, ~0ull, 4));
  PK_TRY(fill_u64(c, small + 4, 0, 2));
  ull* ev;
  uint64_t m, p0;
  const bool ends = klen >= key_bases;
  PK_TRY(pack_buffers(c, n, ends, &rec->pk));
  PK_TRY(event_index(c, fa, n, sy.delim, sy.skip, small, &ev, &m, &p0, B_NL, 0, &rec->pk));
  rec->n = n;
  if (ends && m) {
    const uint64_t nb = (n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
    uint32_t* cnt;
    ull* tb;
    PK_TRY(need(c, B_WCNT, nb, &cnt));
    PK_TRY(need(c, B_WOFF, nb + 1, &tb));
    PK_TRY(fill_u64(c, rec->pk.W, 0, nb * (NL_PER_BLOCK / 64)));
    PK_TRY(fill_u64(c, small + 6, 0, 2));
    hipLaunchKernelGGL(k_bld_bits, dim3(std::min<unsigned>(grid_for(m, 256), 8u * (unsigned)c->ncu)), dim3(256), 0, st, fa, n, ev, m, klen, read_len, sy,
                       rec->pk.W, small + 6);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_bits_count, dim3((unsigned)nb), dim3(256), 0, st, (const ull*)rec->pk.W, cnt);
    PK_HIP(c, hipGetLastError());
    PK_TRY(scan_fetch<uint32_t>(c, cnt, tb, nb, Post{{small + 6}, {2}}));
    if (!c->box[2]) {
      rec->N = c->box[0];
      rec->R = c->box[1];
      rec->tb = tb;
      return PK_OK;
    }
  }
  ull *rstart, *kofs, *idx;
  uint32_t *rlen, *kc, *flag;
  PK_TRY(need(c, B_RSTART, m + 1, &rstart));
  PK_TRY(need(c, B_RLEN, m + 1, &rlen));
  PK_TRY(need(c, B_KC, m + 1, &kc));
  PK_TRY(need(c, B_KOFS, m + 2, &kofs));
  PK_TRY(need(c, B_TU, m + 1, &flag));
  PK_TRY(need(c, B_UOFF, m + 2, &idx));
  if (m) {
    hipLaunchKernelGGL(k_bld_flags, dim3(grid_for(m, 256)), dim3(256), 0, st, fa, n, ev, m, klen,
                       read_len, sy, flag);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, flag, idx, m));
  ull R = 0;
  PK_TRY(d2h(c, &R, idx + m, 8));
  if (m) {
    hipLaunchKernelGGL(k_bld_write, dim3(grid_for(m, 256)), dim3(256), 0, st, fa, n, ev, m, klen,
                       read_len, sy, idx, rstart, rlen, kc);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, kc, kofs, R));
  ull N = 0;
  PK_TRY(d2h(c, &N, kofs + R, 8));
  rec->rstart = rstart;
  rec->rlen = rlen;
  rec->kofs = kofs;
  rec->R = R;
  rec->N = N;
  return PK_OK;
}

// Input of a partition level or of the bucket count: B buckets that share
// their top `fixed` key bits, found through `in`.
struct Part {
  Runs in;
  uint64_t B;
  int fixed;
  int set;  // which of the two sets of run-table buffers `in` sits in
};

// Buffers of a level's tiles and run table, in set 0 or 1 (a level reads the
// other set): tiles is an upper bound on the level's tile count.
struct LevelBufs {
  ull *boff, *tp, *V;
  uint32_t* M;
};

int level_buffers(pk_ctx* c, int set, uint64_t B, uint64_t tiles, int db, LevelBufs* l) {
  PK_TRY(need(c, set ? B_BOFF2 : B_BOFF, B + 1, &l->boff));
  PK_TRY(need(c, set ? B_TP2 : B_TP, B + 1, &l->tp));
  PK_TRY(need(c, set ? B_HIST2 : B_HIST1, tiles << db, &l->M));
  PK_TRY(need(c, set ? B_OFF2 : B_OFF1, (tiles << db) + 1, &l->V));
  return PK_OK;
}

// The scan of a level's run table (slots past the level's last tile hold
// anything: they come after every offset that is read).
int level_runs(pk_ctx* c, const LevelBufs& l, uint64_t tiles, int db, int tk, Runs* out) {
  PK_TRY(scan_excl<RunCount>(c, reinterpret_cast<const RunCount*>(l.M), l.V, tiles << db));
  out->M = l.M;
  out->V = l.V;
  out->tp = l.tp;
  out->boff = l.boff;
  out->db = db;
  out->tk = tk;
  return PK_OK;
}

// Bits of the next level when `left` remain: as few levels as possible, the
// bits spread evenly.  A level reads and writes every key once, so one level
// less beats longer runs until a run is down to about a line: 10 bits leave 16
// one-word (8 two-word) keys per run of a full tile.
int level_bits(int left) {
  const int nlev = (left + SP_MAX_BITS - 1) / SP_MAX_BITS;
  return (left + nlev - 1) / nlev;
}

// Further partition levels, the per-bucket count and the dense table.  S
// holds the N keys (KB key bits) as p says; levels follow until btot bits are
// fixed.  S2 is the other instance array, C the per-instance counts;
// small[4] (the overflow count) starts at zero.
template <class Key>
int count_partitioned(pk_ctx* c, Key* S, Key* S2, int32_t* C, Part p, int btot, int KB, uint64_t N) {
  Key* TK;
  int32_t* TC;
  hipStream_t st = c->stream;
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  Key* Sin = S;
  Key* Sout = S2;
  const int tk = SplitCfg<Key>::TK_MAX;
  while (p.fixed < btot) {
    const int db = level_bits(btot - p.fixed);
    const uint64_t tiles = N / tk + p.B + 1;  // upper bound
    const int set = p.set ^ 1;
    LevelBufs l;
    PK_TRY(level_buffers(c, set, p.B, tiles, db, &l));
    hipLaunchKernelGGL(k_tiles, dim3(1), dim3(1024), 0, st, p.in, (ull)p.B, tk, (ull)N, l.boff, l.tp);
    PK_HIP(c, hipGetLastError());
    const int lv = c->ms_levels < MS_TIMED_LEVELS ? c->ms_levels : -1;
    if (lv >= 0) PK_HIP(c, hipEventRecord(c->ev[20 + 2 * lv], st));
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_split<Key, SPLIT_RUNS>), dim3((unsigned)tiles), dim3(SP_NT), 0, st, Sin,
                       WinSrc{}, p.in, (int)p.B, tk, KB - p.fixed - db, db, l.boff, l.tp, l.M, Sout);
    PK_HIP(c, hipGetLastError());
    if (lv >= 0) PK_HIP(c, hipEventRecord(c->ev[21 + 2 * lv], st));
    if (lv >= 0) c->ms_form[lv] = PK_MS_TILES;
    c->timing.ms_scatter_form = PK_MS_TILES;
    c->ms_levels++;
    p.in.tb = nullptr;
    PK_TRY(level_runs(c, l, tiles, db, tk, &p.in));
    p.B <<= db;
    p.fixed += db;
    p.set = set;
    std::swap(Sin, Sout);
  }
  S = Sin;
  Key* Res = Sout;  // the other array receives the (key, count) results
  const uint64_t B = p.B;
  const Runs in = p.in;
  PK_HIP(c, hipEventRecord(c->ev[5], st));
  // 4. per-bucket count
  long long* tu;
  ull *ovl, *uoff, *bstart;
  PK_TRY(need(c, B_BCNT, B, &bstart));
  PK_TRY(need(c, B_TU, B, &tu));
  PK_TRY(need(c, B_OVF, B + 1, &ovl));
  PK_TRY(need(c, B_UOFF, B + 1, &uoff));
  const unsigned rgrid = (unsigned)std::min<uint64_t>(B, 4ull * (uint64_t)c->ncu);
  if (in.M) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_bucket_hash<Key, true>), dim3((unsigned)B), dim3(HashCfg<Key>::NT), 0, st, S, Res, C,
                       in, KB / 2, btot, tu, bstart);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_bucket_retry<Key, true>), dim3(rgrid), dim3(HashCfg<Key>::NT), 0, st, S, Res, C, in,
                       (ull)B, KB / 2, btot, tu, small + 4, ovl);
  } else {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_bucket_hash<Key, false>), dim3((unsigned)B), dim3(HashCfg<Key>::NT), 0, st, S, Res, C,
                       in, KB / 2, btot, tu, bstart);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_bucket_retry<Key, false>), dim3(rgrid), dim3(HashCfg<Key>::NT), 0, st, S, Res, C, in,
                       (ull)B, KB / 2, btot, tu, small + 4, ovl);
  }
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[7], st));
  // the scan of the distinct counts goes ahead of the overflow check: with
  // no oversize bucket (the usual case) one synchronisation yields both
  PK_TRY(scan_fetch<long long>(c, tu, uoff, B, Post{{small + 4}, {1}}));
  const ull hv[2] = {c->box[1], c->box[0]};
  const ull novf = hv[0];
  c->timing.n_split = (int32_t)novf;
  if (novf) PK_HIP(c, hipEventRecord(c->ev[8], st));
  const ull* lstart = bstart;
  const long long* lu = tu;
  uint64_t nleaves = B;
  if (novf) {
    // leaves = buckets, with each oversize bucket replaced by its split
    std::vector<ull> hbo(B + 1);
    std::vector<long long> htu(B);
    PK_TRY(d2h(c, hbo.data(), bstart, B * 8));
    hbo[B] = N;
    PK_TRY(d2h(c, htu.data(), tu, B * 8));
    std::vector<ull> os, oc;
    std::vector<size_t> ob;
    for (uint64_t b = 0; b < B; b++)
      if (htu[b] < 0) {
        os.push_back(hbo[b]);
        oc.push_back(hbo[b + 1] - hbo[b]);
        ob.push_back(b);
      }
    // the split works in place on contiguous keys: gather the runs of the
    // oversize buckets at their virtual places in a second array, and use
    // the first as the split's scratch
    Key* tmp;
    PK_TRY(need(c, B_TMP, N, &tmp));
    if (in.M) {
      std::vector<ull> oi(ob.begin(), ob.end());
      ull* od;
      PK_TRY(need(c, B_PT0, oi.size(), &od));
      PK_HIP(c, hipMemcpyAsync(od, oi.data(), oi.size() * 8, hipMemcpyHostToDevice, st));
      for (size_t q = 0; q < oi.size(); q += 32768) {
        const unsigned nq = (unsigned)std::min<size_t>(32768, oi.size() - q);
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_gather_buckets<Key>), dim3(GATHER_BLOCKS, nq), dim3(256), 0, st, S, in,
                           od + q, tmp);
        PK_HIP(c, hipGetLastError());
      }
      PK_HIP(c, hipStreamSynchronize(st));  // od's buffer is used again below
      std::swap(S, tmp);
    }
    std::vector<std::vector<Leaf>> rec;
    PK_TRY(resolve_overflow<Key>(c, S, tmp, Res, C, KB / 2, btot, os, oc, rec));
    std::vector<ull> ls;
    std::vector<long long> lus;
    size_t j = 0;
    for (uint64_t b = 0; b < B; b++) {
      if (j < ob.size() && ob[j] == b) {
        for (auto& lf : rec[j]) {
          ls.push_back(lf.start);
          lus.push_back(lf.u);
        }
        j++;
      } else {
        ls.push_back(hbo[b]);
        lus.push_back(htu[b]);
      }
    }
    nleaves = ls.size();
    ull* lsd;
    long long* lud;
    PK_TRY(need(c, B_PT0, nleaves, &lsd));
    PK_TRY(need(c, B_PT1, nleaves, &lud));
    PK_TRY(need(c, B_UOFF, nleaves + 1, &uoff));
    PK_HIP(c, hipMemcpyAsync(lsd, ls.data(), nleaves * 8, hipMemcpyHostToDevice, st));
    PK_HIP(c, hipMemcpyAsync(lud, lus.data(), nleaves * 8, hipMemcpyHostToDevice, st));
    lstart = lsd;
    lu = lud;
  }
  if (novf) PK_HIP(c, hipEventRecord(c->ev[9], st));
  ull U = hv[1];
  if (novf) {
    PK_TRY(scan_excl<long long>(c, lu, uoff, nleaves));
    PK_TRY(d2h(c, &U, uoff + nleaves, 8));
  }
  c->U = U;
  // what is left to do reads the buckets' results and their places only
  for (int id : {B_BOFF, B_TP, B_HIST1, B_OFF1, B_BOFF2, B_TP2, B_HIST2, B_OFF2, B_OVF, B_WOFF, B_OWNOFF})
    c->idle[id] = true;
  for (int id : {B_S, B_S2, B_TMP})
    if (c->buf[id].p != static_cast<const void*>(Res)) c->idle[id] = true;
  PK_TRY(need(c, B_TK, U, &TK));
  PK_TRY(need(c, B_TC, U, &TC));
  PK_HIP(c, hipEventRecord(c->ev[10], st));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_compact<Key>), dim3((unsigned)nleaves), dim3(256), 0, st, Res,
                     C, lstart, lu, uoff, nleaves, TK, TC);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[11], st));
  // stage times are read from the events when asked for (pk_last_timing):
  // no wait here, the compaction runs on while the caller goes on
  c->pend_count = true;
  c->pend_split = novf != 0;
  c->have_table = true;
  return PK_OK;
}

// What every count notes about its input; N == 0 ends it with an empty table
// (*empty).
template <class Key>
int begin_count(pk_ctx* c, uint64_t R, uint64_t N, int K, bool* empty) {
  c->R = R;
  c->N = N;
  c->k = K;
  c->words = sizeof(Key) / 8;
  c->timing.n_instances = N;
  c->timing.n_reads = R;
  c->ms_levels = 0;
  c->have_hist = false;
  *empty = N == 0;
  if (N == 0) {
    Key* TK;
    int32_t* TC;
    c->U = 0;
    PK_TRY(need(c, B_TK, 1, &TK));
    PK_TRY(need(c, B_TC, 1, &TC));
    c->have_table = true;
  }
  return PK_OK;
}

// Count the windows of the read table's reads (in file order) from the packed
// input.  K = window length, KB = key bits (2K on the main path, the whole
// word for the builder encoding), mask = the key's bits.
template <class Key, int ENC>
int count_records(pk_ctx* c, const Records& rec, int K, int KB, Key mask) {
  constexpr int CAP = HashCfg<Key>::LIMIT;
  hipStream_t st = c->stream;
  c->ev_parsed = 4;
  const uint64_t N = rec.N;
  bool empty;
  PK_TRY(begin_count<Key>(c, rec.R, N, K, &empty));
  if (empty) return PK_OK;
  const pk_tuning& tun = c->tuning;
  const float bf = tun.bucket_factor > 0.f ? tun.bucket_factor : HashCfg<Key>::FILL;
  const int btot = choose_bits(N, KB / 2, CAP, bf);
  c->timing.bucket_bits = btot;
  Key *S, *S2;
  int32_t* C;
  PK_TRY(need(c, B_S, N, &S));
  LevelBufs l;
  Part p{Runs{}, 0, 0, 0};
  uint64_t tiles;
  int d1, tk = 0;
  auto level1_bits = [&]() {
    if (tun.l1_bits > 0 && tun.l1_bits <= L1_MAX_BITS) return std::min(btot, tun.l1_bits);
    // one level of up to 10 bits while a bucket's runs fit the hash's map
    if (btot <= SP_MAX_BITS && tiles <= (uint64_t)RUN_CAP) return btot;
    int b = level_bits(btot);
    if (rec.part) {
      // a share's tiles hold few keys (1 in P of their windows): a narrower
      // first digit keeps its runs at 32 keys or so, two lines and more each,
      // if the further levels can take the rest
      const int nlev = (btot + SP_MAX_BITS - 1) / SP_MAX_BITS;
      int f = 0;
      while (f < b && (N / tiles) >> (f + 6)) f++;
      b = std::min(b, std::max({1, f, btot - SP_MAX_BITS * (nlev - 1)}));
    }
    return b;
  };
  if (ENC == ENC_MAIN || rec.tb) {
    // tiles of 16 or 32 KiB of the input: the larger ones' runs are twice as
    // long, the smaller ones spread an input over more CUs
    const uint64_t nblk = (rec.n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
    const int wpt = nblk >= 4096 ? 2 : 1;
    tiles = (nblk + wpt - 1) / wpt;
    d1 = level1_bits();
    PK_TRY(level_buffers(c, 0, 1, tiles, d1, &l));
    PK_HIP(c, hipEventRecord(c->ev[4], st));
    const uint16_t* W = reinterpret_cast<const uint16_t*>(rec.pk.W);
    if (wpt == 2)
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_split_main<Key, 2>), dim3((unsigned)tiles), dim3(SM_NT), 0, st, rec.pk.E,
                         rec.pk.RX, W, rec.tb, (ull)nblk, (ull)((rec.n + 15) / 16), mask, KB - d1, d1, l.M, S, l.boff, l.tp);
    else
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_split_main<Key, 1>), dim3((unsigned)tiles), dim3(SM_NT), 0, st, rec.pk.E,
                         rec.pk.RX, W, rec.tb, (ull)nblk, (ull)((rec.n + 15) / 16), mask, KB - d1, d1, l.M, S, l.boff, l.tp);
    p.in.tb = rec.tb;
    p.in.ts = wpt - 1;
  } else if constexpr (ENC == ENC_BUILDER) {
    // tiles of N / 512 windows (so that a small input spreads over the CUs and
    // a bucket has at most RUN_CAP runs), within 4096 and a full tile
    const uint64_t per = (N + RUN_CAP - 1) / RUN_CAP;
    tk = (int)std::min<uint64_t>(SplitCfg<Key>::TK_MAX, std::max<uint64_t>(4096, (per + SP_NT - 1) / SP_NT * SP_NT));
    tiles = (N + tk - 1) / tk;
    d1 = level1_bits();
    PK_TRY(level_buffers(c, 0, 1, tiles, d1, &l));
    hipLaunchKernelGGL(k_tiles_one, dim3(1), dim3(1), 0, st, (ull)tiles, (ull)N, l.boff, l.tp);
    PK_HIP(c, hipGetLastError());
    PK_HIP(c, hipEventRecord(c->ev[4], st));
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_split<Key, SPLIT_BUILDER>), dim3((unsigned)tiles), dim3(SP_NT), 0, st,
                       (const Key*)nullptr, WinSrc{rec.pk.E, rec.kofs, rec.rstart, rec.R, K}, Runs{}, 1, tk, KB - d1,
                       d1, l.boff, l.tp, l.M, S);
  }
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[16], st));
  // the packed input has been read: its scratch is free for what follows
  // in stream order
  c->arena_lim = c->arena_cap;
  c->idle[B_PACK] = c->idle[B_OWNW] = c->idle[B_LW] = c->idle[B_WCNT] = true;
  c->idle[B_RSTART] = c->idle[B_RLEN] = c->idle[B_KC] = c->idle[B_KOFS] = c->idle[B_NL] = true;
  PK_TRY(need(c, B_S2, N, &S2));
  PK_TRY(need(c, B_C, N, &C));
  p.B = 1ull << d1;
  p.fixed = d1;
  PK_TRY(level_runs(c, l, tiles, d1, tk, &p.in));
  return count_partitioned<Key>(c, S, S2, C, p, btot, KB, N);
}

// The count without the packed input: level 1 walks every read and scatters its
// keys into contiguous buckets.
template <class Key>
int count_walk(pk_ctx* c, const uint8_t* fa, uint64_t n, const Records& rec, int K) {
  constexpr int CAP = HashCfg<Key>::LIMIT;
  hipStream_t st = c->stream;
  const uint64_t R = rec.R;
  const uint64_t N = rec.N;
  const int KB = 2 * K;
  const Key mask = key_mask<Key>(KB);
  PK_HIP(c, hipEventRecord(c->ev[1], st));
  c->ev_parsed = 1;
  bool empty;
  PK_TRY(begin_count<Key>(c, R, N, K, &empty));
  if (empty) return PK_OK;
  const pk_tuning& tun = c->tuning;
  const float bf = tun.bucket_factor > 0.f ? tun.bucket_factor : HashCfg<Key>::FILL;
  const int btot = choose_bits(N, K, CAP, bf);
  c->timing.bucket_bits = btot;
  const int d1 = std::min(btot, tun.l1_bits > 0 && tun.l1_bits <= L1_MAX_BITS ? tun.l1_bits : L1_DEFAULT_BITS);
  const uint64_t B1 = 1ull << d1;
  // reads per block: up to 8 chunks of L1_NT, fewer for small inputs so that
  // the grid still spreads over the CUs
  const int rpb = L1_NT * (tun.l1_chunks > 0 && tun.l1_chunks <= 64
                               ? tun.l1_chunks
                               : (int)std::min<uint64_t>(8, std::max<uint64_t>(1, R / (L1_NT * 1024ull))));
  const uint64_t nblk = (R + rpb - 1) / rpb;
  // LDS staging: room for one record per thread of the input's mean size,
  // + 25 %
  const double want = (double)L1_NT * ((double)n / (double)R) * 1.25;
  const int sb = ((int)std::min<double>(L1_SB_MAX, std::max<double>(L1_SB_MIN, want)) + 1023) & ~1023;
  ull *boff, *O;
  uint32_t* H;
  Key *S, *S2;
  int32_t* C;
  PK_TRY(need(c, B_BOFF, B1 + 1, &boff));
  PK_TRY(need(c, B_HIST1, B1 * nblk, &H));
  PK_TRY(need(c, B_OFF1, B1 * nblk + 1, &O));
  PK_TRY(need(c, B_S, N, &S));
  PK_TRY(need(c, B_S2, N, &S2));
  PK_TRY(need(c, B_C, N, &C));
  c->have_hist = true;
  PK_HIP(c, hipEventRecord(c->ev[2], st));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_l1_hist<Key>), dim3((unsigned)nblk), dim3(L1_NT),
                     l1_lds_bytes(sb, (int)B1, 4), st, fa, n, rec.rstart, rec.rlen, R, K, KB, mask, d1, rpb, sb, H);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[3], st));
  PK_TRY(scan_excl<uint32_t>(c, H, O, B1 * nblk));
  hipLaunchKernelGGL(k_l1_boff, dim3(grid_for(B1 + 1, 256)), dim3(256), 0, st, O, (int)B1, nblk, (ull)N,
                     boff);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[4], st));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_l1_scatter<Key>), dim3((unsigned)nblk), dim3(L1_NT),
                     l1_lds_bytes(sb, (int)B1, 8), st, fa, n, rec.rstart, rec.rlen, R, K, KB, mask, d1, rpb, sb, O,
                     nblk, S);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[16], st));
  return count_partitioned<Key>(c, S, S2, C, Part{Runs{nullptr, nullptr, nullptr, boff, 0, 0, nullptr, 0}, B1, d1, 0}, btot, KB,
                                N);
}

// Distinct klen-byte windows of the implicit builder counters: keys from
// k_win_keys (KB bits, even), then the partition and count from memory.
template <class Key>
int windows_count_impl(pk_ctx* c, const uint8_t* fa, const ull* rstart, const uint32_t* rlen, const ull* woff,
                       uint64_t R, uint64_t N, int klen, int bits, const uint8_t* lut, int has_nul, int KB) {
  hipStream_t st = c->stream;
  c->key_bits = -1;  // byte-rank codes: no macro nodes on this table
  PK_HIP(c, hipEventRecord(c->ev[1], st));
  c->ev_parsed = 1;
  bool empty;
  PK_TRY(begin_count<Key>(c, R, N, klen, &empty));
  if (empty) return PK_OK;
  Key *S, *S2;
  int32_t* C;
  ull *boff, *small;
  PK_TRY(need(c, B_S, N, &S));
  PK_TRY(need(c, B_S2, N, &S2));
  PK_TRY(need(c, B_C, N, &C));
  PK_TRY(need(c, B_BOFF, 2, &boff));
  PK_TRY(need(c, B_SMALL, 16, &small));
  PK_TRY(fill_u64(c, small + 4, 0, 2));
  PK_TRY(fill_u64(c, boff, 0, 1));
  PK_TRY(fill_u64(c, boff + 1, N, 1));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_win_keys<Key>), dim3(grid_for(R, 256)), dim3(256), 0, st, fa, rstart, rlen,
                     woff, R, klen, bits, lut, has_nul, S);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[4], st));
  PK_HIP(c, hipEventRecord(c->ev[16], st));
  const float bf = c->tuning.bucket_factor > 0.f ? c->tuning.bucket_factor : HashCfg<Key>::FILL;
  const int btot = choose_bits(N, KB / 2, HashCfg<Key>::LIMIT, bf);
  c->timing.bucket_bits = btot;
  return count_partitioned<Key>(c, S, S2, C, Part{Runs{nullptr, nullptr, nullptr, boff, 0, 0, nullptr, 0}, 1, 0, 0}, btot, KB, N);
}

template <class Key>
int count_impl(pk_ctx* c, const uint8_t* fa, uint64_t n, int K) {
  c->have_table = c->have_kept = c->have_nodes = false;
  begin_buffers(c);
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = c->pend_cutoff = c->pend_mn = c->pend_norm = false;
  c->key_bits = 2 * K;
  PK_HIP(c, hipEventRecord(c->ev[0], c->stream));
  Records rec;
  rec.n = n;
  PK_TRY(pack_buffers(c, n, true, &rec.pk));
  if (!rec.pk.E) {
    // pk_count_noalloc's scratch is short of the packed input
    PK_TRY(records_main(c, fa, n, K, &rec));
    return count_walk<Key>(c, fa, n, rec, K);
  }
  PK_TRY(windows_main(c, fa, n, K, &rec));
  return count_records<Key, ENC_MAIN>(c, rec, K, 2 * K, key_mask<Key>(2 * K));
}

// L-mer frequencies (device, LMER_BINS u64) from the packed input and the
// L-mers' ends W.
int lmer_frequency_impl(pk_ctx* c, const Records& rec, const ull* W, ull** freq_out) {
  hipStream_t st = c->stream;
  ull* freq;
  PK_TRY(need(c, B_LFREQ, LMER_BINS, &freq));
  PK_TRY(fill_u64(c, freq, 0, LMER_BINS));
  const uint64_t nb = (rec.n + NL_PER_BLOCK - 1) / NL_PER_BLOCK;
  if (nb) {
    uint64_t np64 = std::min<uint64_t>(nb, (uint64_t)c->ncu);
    // (fewer blocks where a budget has no room for their tables)
    while (c->budget && np64 > 1 && c->held + np64 * (LMER_BINS / 2) * 4 > c->budget) np64 = (np64 + 1) / 2;
    const int np = (int)np64;
    uint32_t* part;
    PK_TRY(need(c, B_LPART, (uint64_t)np * (LMER_BINS / 2), &part));
    hipLaunchKernelGGL(k_lmer_count, dim3((unsigned)np), dim3(LM_NT), 0, st, rec.pk.E, rec.pk.RX,
                       reinterpret_cast<const uint16_t*>(W), (ull)nb, part, freq);
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_lmer_sum, dim3(LMER_BINS / 128), dim3(1024), 0, st, part, np, freq);
    PK_HIP(c, hipGetLastError());
  }
  *freq_out = freq;
  return PK_OK;
}

OwnerMod owner_mod(int P, int rank) {
  int l = 0;
  while ((1ull << l) < (ull)P) l++;
  return OwnerMod{(1ull << (31 + l)) / (ull)P + 1, 31 + l, (uint32_t)P, (uint32_t)rank};
}

template <int BS>
int launch_own(pk_ctx* c, const Records& rec, uint64_t words, int w, const uint4* tab, uint16_t* Wout, uint16_t* D) {
  PK_HIP(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_own<BS>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, own_lds));
  const uint64_t tiles = (words + (OWN_NT - OWN_HALO) - 1) / (OWN_NT - OWN_HALO);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_own<BS>), dim3((unsigned)std::min<uint64_t>(tiles, (uint64_t)c->ncu)),
                     dim3(OWN_NT), own_lds, c->stream, rec.pk.E, rec.pk.RX, reinterpret_cast<const uint16_t*>(rec.pk.W),
                     (ull)words, (ull)((rec.n + 15) / 16), w, tab, Wout, D);
  PK_HIP(c, hipGetLastError());
  return PK_OK;
}

// Leaves in rec only the window ends of one rank: of the minimum L-mer's owner
// (freq), or of the whole k-mer's (freq null).
int own_windows(pk_ctx* c, int K, const ull* freq, int P, int rank, Records* rec) {
  hipStream_t st = c->stream;
  const uint64_t nb = (rec->n + NL_PER_BLOCK - 1) / NL_PER_BLOCK, words = nb * (NL_PER_BLOCK / 16);
  const OwnerMod om = owner_mod(P, rank);
  uint16_t* wo;
  PK_TRY(need(c, B_OWNW, 2 * words, &wo));
  uint32_t* cnt;
  ull* tb;
  PK_TRY(need(c, B_OWNCNT, nb, &cnt));
  PK_TRY(need(c, B_OWNOFF, nb + 1, &tb));
  if (freq) {
    uint32_t* tab;
    ull* big;  // then their number
    PK_TRY(need(c, B_LBIG, LMER_BINS + 1, &big));
    PK_TRY(need(c, B_LRANK, OWN_TAB, &tab));
    uint16_t* rk = reinterpret_cast<uint16_t*>(tab);
    uint32_t* ob = tab + LMER_BINS / 2;
    hipLaunchKernelGGL(k_freq_rank, dim3(1), dim3(1024), 0, st, freq, om, big, big + LMER_BINS, rk,
                       reinterpret_cast<ull*>(ob));
    PK_HIP(c, hipGetLastError());
    hipLaunchKernelGGL(k_freq_big, dim3(LMER_BINS / 64), dim3(64), 0, st, freq, big, big + LMER_BINS, rk);
    PK_HIP(c, hipGetLastError());
    uint16_t* D = wo + words;
    const uint4* t4 = reinterpret_cast<const uint4*>(tab);
    const int w = K - LMER_L + 1;
    if (w >= 16)
      PK_TRY(launch_own<16>(c, *rec, words, w, t4, wo, D));
    else if (w >= 8)
      PK_TRY(launch_own<8>(c, *rec, words, w, t4, wo, D));
    else if (w >= 4)
      PK_TRY(launch_own<4>(c, *rec, words, w, t4, wo, D));
    else if (w >= 2)
      PK_TRY(launch_own<2>(c, *rec, words, w, t4, wo, D));
    else
      PK_TRY(launch_own<1>(c, *rec, words, w, t4, wo, D));
    hipLaunchKernelGGL(k_own_walk, dim3(grid_for(words, 256)), dim3(256), 0, st, rec->pk.E, rec->pk.RX, D, (ull)words,
                       w, rk, ob, reinterpret_cast<uint32_t*>(wo));
    PK_HIP(c, hipGetLastError());
  } else {
    hipLaunchKernelGGL(k_own_key, dim3(grid_for(words, 256)), dim3(256), 0, st, rec->pk.E, rec->pk.RX,
                       reinterpret_cast<const uint16_t*>(rec->pk.W), (ull)words, key_mask<uint64_t>(2 * K), om, wo);
    PK_HIP(c, hipGetLastError());
  }
  hipLaunchKernelGGL(k_bits_count, dim3((unsigned)nb), dim3(256), 0, st, reinterpret_cast<const ull*>(wo), cnt);
  PK_HIP(c, hipGetLastError());
  PK_TRY(scan_fetch<uint32_t>(c, cnt, tb, nb, Post{}));
  rec->N = c->box[0];
  rec->pk.W = reinterpret_cast<ull*>(wo);
  rec->tb = tb;
  rec->part = true;
  return PK_OK;
}

// One rank's share of the counted table at P ranks (the table rank `rank`
// holds after the reference's all-to-all): the k-mers whose owner is rank, by
// the minimum L-mer or (by_key) retrieve_proc_id(kmer) (the -p counters,
// kmer_counting.cpp:1825-2091, 2095-2271).
template <class Key>
int rank_share_impl(pk_ctx* c, const uint8_t* fa, uint64_t n, int K, int P, int rank, bool by_key) {
  c->have_table = c->have_kept = c->have_nodes = false;
  begin_buffers(c);
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = c->pend_cutoff = c->pend_mn = c->pend_norm = false;
  c->key_bits = 2 * K;
  PK_HIP(c, hipEventRecord(c->ev[0], c->stream));
  Records rec;
  ull *freq = nullptr, *W2 = nullptr;
  rec.n = n;
  PK_TRY(pack_buffers(c, n, true, &rec.pk));
  if (!by_key) PK_TRY(need(c, B_LW, (n + NL_PER_BLOCK - 1) / NL_PER_BLOCK * (NL_PER_BLOCK / 64), &W2));
  PK_TRY(windows_main(c, fa, n, K, &rec, W2));
  if (!by_key && rec.N) PK_TRY(lmer_frequency_impl(c, rec, W2, &freq));
  if (rec.N) PK_TRY(own_windows(c, K, freq, P, rank, &rec));
  return count_records<Key, ENC_MAIN>(c, rec, K, 2 * K, key_mask<Key>(2 * K));
}

template <class Key>
int builder_count_impl(pk_ctx* c, const uint8_t* fa, uint64_t n, int klen, uint64_t read_len,
                       BldSyms sy) {
  c->have_table = c->have_kept = c->have_nodes = false;
  begin_buffers(c);
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = c->pend_cutoff = c->pend_mn = c->pend_norm = false;
  c->key_bits = (int)sizeof(Key) * 8;
  PK_HIP(c, hipEventRecord(c->ev[0], c->stream));
  Records rec;
  PK_TRY(records_builder(c, fa, n, klen, read_len, sy, (int)sizeof(Key) * 4, &rec));
  return count_records<Key, ENC_BUILDER>(c, rec, klen, (int)sizeof(Key) * 8, ~Key(0));
}

__global__ void k_set_int(int* p, int v) { *p = v; }

// fixed_mb > 0: keep count >= fixed_mb with no histogram (the PaK-graph
// builder's threshold rule); else the histogram cutoff with t buckets.
template <class Key>
int cutoff_impl(pk_ctx* c, int t, uint64_t* hist_out, int* mb_out, uint64_t* nk_out, int fixed_mb = 0) {
  hipStream_t st = c->stream;
  PK_HIP(c, hipEventRecord(c->ev[12], st));
  Key* TK = reinterpret_cast<Key*>(c->buf[B_TK].p);
  int32_t* TC = reinterpret_cast<int32_t*>(c->buf[B_TC].p);
  const uint64_t U = c->U;
  ull* hist;
  ull* small;
  PK_TRY(need(c, B_HIST, (uint64_t)t + 8, &hist));
  PK_TRY(need(c, B_SMALL, 16, &small));
  const uint64_t nb = (U + CUT_PER - 1) / CUT_PER;
  const bool want_hist = hist_out && fixed_mb <= 0;
  const int hn = want_hist && t <= BOX_WORDS - 3 ? t : 0;  // histogram words that fit the box
  const bool plan = fixed_mb <= 0 && t <= CUT_SMALL_T && nb && nb <= CUT_PLAN;
  if (!plan) PK_TRY(fill_u64(c, hist, 0, (uint64_t)t));
  int* mbd = reinterpret_cast<int*>(small + 8);
  ull *bs, *boffs;
  PK_TRY(need(c, B_KBS, nb + 1, &bs));
  PK_TRY(need(c, B_KBOFF, nb + 1, &boffs));
  if (fixed_mb > 0) {
    hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, mbd, fixed_mb);
    PK_HIP(c, hipGetLastError());
    if (nb) {
      hipLaunchKernelGGL(k_kept_count, dim3((unsigned)nb), dim3(CUT_NT), 0, st, TC, U, mbd, bs);
      PK_HIP(c, hipGetLastError());
    }
  } else if (t <= CUT_SMALL_T) {
    uint32_t* BH;
    PK_TRY(need(c, B_CUTBH, nb * (uint64_t)t + 1, &BH));
    if (nb) {
      hipLaunchKernelGGL(k_count_hist_blocks, dim3((unsigned)nb), dim3(CUT_NT), 0, st, TC, U, t, BH);
      PK_HIP(c, hipGetLastError());
    }
    if (plan) {
      hipLaunchKernelGGL(k_cut_plan, dim3(1), dim3(1024), 0, st, BH, nb, U, t, hist, mbd, boffs, hn, c->box);
      PK_HIP(c, hipGetLastError());
      PK_HIP(c, hipStreamSynchronize(st));
    } else if (nb) {
      hipLaunchKernelGGL(k_hist_columns, dim3((unsigned)t), dim3(1024), 0, st, BH, nb, t, hist);
      PK_HIP(c, hipGetLastError());
    }
    if (!plan) {
      hipLaunchKernelGGL(k_min_bucket, dim3(1), dim3(1), 0, st, hist, t, mbd);
      PK_HIP(c, hipGetLastError());
    }
    if (nb && !plan) {
      hipLaunchKernelGGL(k_kept_from_hist, dim3(grid_for(nb, 256)), dim3(256), 0, st, BH, nb, U, t,
                         mbd, bs);
      PK_HIP(c, hipGetLastError());
    }
  } else {
    if (nb) {
      hipLaunchKernelGGL(k_count_hist, dim3((unsigned)nb), dim3(CUT_NT), 0, st, TC, U, t, hist);
      PK_HIP(c, hipGetLastError());
    }
    hipLaunchKernelGGL(k_min_bucket, dim3(1), dim3(1), 0, st, hist, t, mbd);
    PK_HIP(c, hipGetLastError());
    if (nb) {
      hipLaunchKernelGGL(k_kept_count, dim3((unsigned)nb), dim3(CUT_NT), 0, st, TC, U, mbd, bs);
      PK_HIP(c, hipGetLastError());
    }
  }
  if (!plan) {
    if (want_hist && !hn) PK_HIP(c, hipMemcpyAsync(hist_out, hist, (size_t)t * 8, hipMemcpyDeviceToHost, st));
    PK_TRY(scan_fetch<ull>(c, bs, boffs, nb, Post{{small + 8, hist}, {1, hn}}));
  }
  const ull V = c->box[0];
  const int mb = (int)(uint32_t)c->box[1];
  if (hn) memcpy(hist_out, c->box + 2, (size_t)t * 8);
  Key* KK;
  int32_t* KC;
  PK_TRY(need(c, B_KK, V, &KK));
  PK_TRY(need(c, B_KC2, V, &KC));
  if (nb && V) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_kept_write<Key>), dim3((unsigned)nb), dim3(CUT_NT), 0, st,
                       TK, TC, U, mbd, boffs, KK, KC);
    PK_HIP(c, hipGetLastError());
  }
  PK_HIP(c, hipEventRecord(c->ev[13], st));
  c->pend_cutoff = true;
  c->V = V;
  c->t = t;
  c->mb = mb;
  c->have_kept = true;
  c->have_nodes = false;
  *mb_out = mb;
  *nk_out = V;
  if (V == 0 && fixed_mb <= 0)
    return c->fail(PK_EEMPTY, "no k-mer has count >= min_bucket(" + std::to_string(mb) + ")");
  return PK_OK;
}

template <class Key>
int mn_impl(pk_ctx* c) {
  hipStream_t st = c->stream;
  PK_HIP(c, hipEventRecord(c->ev[14], st));
  const Key* KK = reinterpret_cast<const Key*>(c->buf[B_KK].p);
  const int32_t* KC = reinterpret_cast<const int32_t*>(c->buf[B_KC2].p);
  const uint64_t V = c->V;
  const int K = c->k;
  const uint64_t G = (V + MN_PC - 1) / MN_PC;
  ull *bd, *ng, *noff;
  MnRec* nodes;
  uint16_t* rk;
  PK_TRY(need(c, B_MNPLAN, 5 * (G + 1), &bd));
  PK_TRY(need(c, B_MNNG, G, &ng));
  PK_TRY(need(c, B_MNNOFF, G + 1, &noff));
  PK_TRY(need(c, B_MNFLAG, 2 * V, &rk));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_mn_bounds<Key>), dim3(grid_for(5 * (G + 1), 256)), dim3(256), 0, st, KK, (ull)V,
                     K, (ull)G, bd);
  PK_HIP(c, hipGetLastError());
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_mn_rank<Key>), dim3((unsigned)G), dim3(MN_NT), 0, st, KK, K, bd, (ull)G, rk,
                     rk + V, ng);
  PK_HIP(c, hipGetLastError());
  PK_TRY(scan_fetch<ull>(c, ng, noff, G, Post{}));
  const ull M = c->box[0];
  PK_TRY(need(c, B_NODES, M, &nodes));
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_mn_write<Key>), dim3((unsigned)G), dim3(MN_NT), 0, st, KK, KC, K, bd, (ull)G,
                     rk, rk + V, noff, nodes);
  PK_HIP(c, hipGetLastError());
  PK_HIP(c, hipEventRecord(c->ev[15], st));
  c->pend_mn = true;
  c->M = M;
  c->have_nodes = true;
  return PK_OK;
}

// Keeps the rank's share of the node table (in place, key order kept).
template <class Key>
int node_share_impl(pk_ctx* c, int P, int rank) {
  hipStream_t st = c->stream;
  const uint64_t M = c->M;
  MnRec* nodes = reinterpret_cast<MnRec*>(c->buf[B_NODES].p);
  uint32_t* flag;
  ull* pos;
  MnRec* tmp;
  PK_TRY(need(c, B_TU, M + 1, &flag));
  PK_TRY(need(c, B_UOFF, M + 2, &pos));
  PK_TRY(need(c, B_MNNT, M + 1, &tmp));
  if (M) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_node_share_flags<Key>), dim3(grid_for(M, 256)), dim3(256), 0, st, nodes,
                       M, P, rank, flag);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, flag, pos, M));
  ull M2 = 0;
  PK_TRY(d2h(c, &M2, pos + M, 8));
  if (M) {
    hipLaunchKernelGGL(k_node_share_write, dim3(grid_for(M, 256)), dim3(256), 0, st, nodes, M, flag, pos, tmp);
    PK_HIP(c, hipGetLastError());
  }
  if (M2) PK_HIP(c, hipMemcpyAsync(nodes, tmp, M2 * sizeof(MnRec), hipMemcpyDeviceToDevice, st));
  c->M = M2;
  return PK_OK;
}

}  // namespace

// Host input to the device through pinned staging: PIN_THREADS host threads
// each take a contiguous slice and copy it PIN_CHUNK bytes at a time into
// one of their two pinned buffers, then queue the DMA copy on the context
// stream; a buffer is refilled once the event after its last copy has
// completed.  A DMA copy from pageable memory runs at about half the rate of
// one from pinned memory (27 against 56 GB/s measured on an MI355X host), so
// the staging pays for its host memcpy.  Small inputs and pinned inputs take
// one direct copy.
constexpr int PIN_THREADS = 4;
constexpr uint64_t PIN_CHUNK = 8ull << 20;
constexpr uint64_t PIN_MIN = 16ull << 20;

// Pinned staging shared by host-memory input and file input: fill(buf, off,
// len) puts bytes [off, off + len) of the input into the pinned buffer
// (returns false on a read error).
template <class Fill>
static int h2d_pinned(pk_ctx* c, uint8_t* dst, uint64_t n, Fill&& fill, bool* read_failed);
static bool pin_buffers(pk_ctx* c);

static int h2d_staged(pk_ctx* c, uint8_t* dst, const char* src, uint64_t n) {
  // pinned (page-locked) input is copied as it is
  hipPointerAttribute_t attr{};
  const bool pinned = hipPointerGetAttributes(&attr, src) == hipSuccess && attr.type == hipMemoryTypeHost;
  (void)hipGetLastError();  // an unregistered pointer may leave an error behind
  if (n < PIN_MIN || pinned) {
    PK_HIP(c, hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, c->stream));
    return PK_OK;
  }
  if (!pin_buffers(c)) {
    // no pinned memory to be had: one direct copy
    PK_HIP(c, hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, c->stream));
    return PK_OK;
  }
  bool bad = false;
  return h2d_pinned(
      c, dst, n,
      [src](void* buf, uint64_t off, uint64_t len) {
        std::memcpy(buf, src + off, len);
        return true;
      },
      &bad);
}

static bool pin_buffers(pk_ctx* c) {
  bool ready = true;
  for (int i = 0; i < 2 * PIN_THREADS && ready; i++) {
    if (!c->pin[i] && hipHostMalloc(&c->pin[i], PIN_CHUNK, hipHostMallocDefault) != hipSuccess) {
      c->pin[i] = nullptr;
      ready = false;
    }
    if (ready && !c->pin_ev[i] && hipEventCreateWithFlags(&c->pin_ev[i], hipEventDisableTiming) != hipSuccess) {
      c->pin_ev[i] = nullptr;
      ready = false;
    }
  }
  if (!ready) (void)hipGetLastError();
  return ready;
}

template <class Fill>
static int h2d_pinned(pk_ctx* c, uint8_t* dst, uint64_t n, Fill&& fill, bool* read_failed) {
  *read_failed = false;
  if (!pin_buffers(c)) return c->fail(PK_ENOMEM, "pinned staging buffers could not be allocated");
  const uint64_t slice = ((n + PIN_THREADS - 1) / PIN_THREADS + 63) & ~63ull;
  hipError_t err[PIN_THREADS];
  bool rerr[PIN_THREADS];
  auto work = [&](int t) {
    err[t] = hipSuccess;
    rerr[t] = false;
    const uint64_t lo = std::min<uint64_t>(n, (uint64_t)t * slice), hi = std::min<uint64_t>(n, lo + slice);
    hipError_t e = hipSetDevice(c->device);
    int k = 0;
    for (uint64_t off = lo; off < hi && e == hipSuccess; off += PIN_CHUNK, k ^= 1) {
      const int b = 2 * t + k;
      const uint64_t len = std::min<uint64_t>(PIN_CHUNK, hi - off);
      if (c->pin_used[b]) e = hipEventSynchronize(c->pin_ev[b]);
      if (e != hipSuccess) break;
      if (!fill(c->pin[b], off, len)) {
        rerr[t] = true;
        break;
      }
      e = hipMemcpyAsync(dst + off, c->pin[b], len, hipMemcpyHostToDevice, c->stream);
      if (e == hipSuccess) e = hipEventRecord(c->pin_ev[b], c->stream);
      c->pin_used[b] = true;
    }
    err[t] = e;
  };
  std::vector<std::thread> th;
  for (int t = 1; t < PIN_THREADS; t++) th.emplace_back(work, t);
  work(0);
  for (auto& x : th) x.join();
  for (int t = 0; t < PIN_THREADS; t++) {
    if (rerr[t]) *read_failed = true;
    if (err[t] != hipSuccess) return c->hip_fail(err[t], "staged host-to-device copy");
  }
  return PK_OK;
}

// ---- File input (pk_count_file) ----------------------------------------------
// The reference reads its rank's byte range of the FASTA file with MPI-IO
// (DivideReads, src/input_reading.cpp:69-243); one GPU takes the whole file:
// PIN_THREADS host threads pread their slices chunk by chunk into pinned
// buffers while the DMA engine drains the previous chunk into HBM.
static int file_to_device(pk_ctx* c, const char* path, const uint8_t** fa, uint64_t* nbytes) {
  const int fd = ::open(path, O_RDONLY);
  if (fd < 0) return c->fail(PK_EINVAL, std::string("cannot open ") + path + ": " + std::strerror(errno));
  struct stat st {};
  if (::fstat(fd, &st) != 0 || !S_ISREG(st.st_mode)) {
    ::close(fd);
    return c->fail(PK_EINVAL, std::string(path) + " is not a regular file");
  }
  const uint64_t n = (uint64_t)st.st_size;
  uint8_t* d;
  int rc = need(c, B_FASTA, n + 64, &d);
  bool bad = false;
  if (rc == PK_OK && n) {
    rc = h2d_pinned(
        c, d, n,
        [fd](void* buf, uint64_t off, uint64_t len) {
          uint64_t got = 0;
          while (got < len) {
            const ssize_t r = ::pread(fd, (char*)buf + got, len - got, (off_t)(off + got));
            if (r <= 0) {
              if (r < 0 && errno == EINTR) continue;
              return false;
            }
            got += (uint64_t)r;
          }
          return true;
        },
        &bad);
  }
  ::close(fd);
  if (rc) return rc;
  if (bad) return c->fail(PK_EINVAL, std::string("read error in ") + path);
  *fa = d;
  *nbytes = n;
  return PK_OK;
}

// ---------------------------------------------------------------------------
// C ABI.

extern "C" {

int pk_ctx_create(pk_ctx** out, int device, uint64_t hbm_budget_bytes) {
  if (!out) return PK_EINVAL;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PK_EHIP;
  if (device < 0 || device >= ndev) return PK_EINVAL;
  if (hipSetDevice(device) != hipSuccess) return PK_EHIP;
  pk_ctx* c = new pk_ctx();
  c->device = device;
  c->budget = hbm_budget_bytes;
  int ncu = 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && ncu > 0)
    c->ncu = ncu;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return PK_EHIP;
  }
  for (auto& e : c->ev) {
    if (hipEventCreate(&e) != hipSuccess) {
      delete c;
      return PK_EHIP;
    }
  }
  void* box = nullptr;
  if (hipHostMalloc(&box, BOX_WORDS * sizeof(ull), hipHostMallocDefault) != hipSuccess) {
    pk_ctx_destroy(c);
    return PK_EHIP;
  }
  c->box = static_cast<ull*>(box);
  *out = c;
  return PK_OK;
}

void pk_ctx_destroy(pk_ctx* c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& b : c->buf)
    if (b.p) (void)(c->stream_alloc ? hipFreeAsync(b.p, c->stream) : hipFree(b.p));
  if (c->stream_alloc && c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& e : c->ev)
    if (e) (void)hipEventDestroy(e);
  for (int i = 0; i < 8; i++) {
    if (c->pin[i]) (void)hipHostFree(c->pin[i]);
    if (c->pin_ev[i]) (void)hipEventDestroy(c->pin_ev[i]);
  }
  if (c->box) (void)hipHostFree(c->box);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char* pk_last_error(const pk_ctx* c) { return c ? c->err.c_str() : "null context"; }
void* pk_ctx_stream(pk_ctx* c) { return c ? (void*)c->stream : nullptr; }
uint64_t pk_ctx_device_bytes(const pk_ctx* c) { return c ? c->held : 0; }

int pk_ctx_set_tuning(pk_ctx* c, const pk_tuning* t) {
  if (!c) return PK_EINVAL;
  if (!t) {
    c->tuning = pk_tuning{};
    return PK_OK;
  }
  if (t->l1_chunks < 0 || t->l1_chunks > 64 || t->l1_bits < 0 || t->l1_bits > L1_MAX_BITS ||
      !(t->bucket_factor >= 0.f && t->bucket_factor <= 64.f) || t->ms_scatter < 0 || t->ms_scatter > 2 ||
      t->ms_fold < 0 || t->ms_fold > 2)
    return c->fail(PK_EINVAL, "tuning values out of range");
  c->tuning = *t;
  return PK_OK;
}

int pk_ctx_set_alloc_mode(pk_ctx* c, int mode) {
  if (!c || (mode != PK_ALLOC_DEVICE && mode != PK_ALLOC_STREAM_ORDERED)) return PK_EINVAL;
  const bool want = mode == PK_ALLOC_STREAM_ORDERED;
  if (want == c->stream_alloc) return PK_OK;
  PK_HIP(c, hipSetDevice(c->device));
  if (want) {
    int pools = 0;
    if (hipDeviceGetAttribute(&pools, hipDeviceAttributeMemoryPoolsSupported, c->device) != hipSuccess || !pools)
      return c->fail(PK_EINVAL, "the device has no stream-ordered memory pools");
  }
  // buffers are freed the way they were allocated
  PK_TRY(pk_ctx_release_buffers(c));
  c->stream_alloc = want;
  return PK_OK;
}

int pk_ctx_release_buffers(pk_ctx* c) {
  if (!c) return PK_EINVAL;
  PK_HIP(c, hipSetDevice(c->device));
  PK_HIP(c, hipStreamSynchronize(c->stream));
  for (auto& b : c->buf) {
    if (b.p) PK_HIP(c, c->stream_alloc ? hipFreeAsync(b.p, c->stream) : hipFree(b.p));
    b.p = nullptr;
    b.cap = 0;
  }
  if (c->stream_alloc) PK_HIP(c, hipStreamSynchronize(c->stream));
  c->held = 0;
  c->have_table = c->have_kept = c->have_nodes = false;
  c->have_norm = false;
  c->norm_n = 0;
  c->pend_count = c->pend_split = c->pend_cutoff = c->pend_mn = c->pend_norm = false;
  return PK_OK;
}

static int fasta_to_device(pk_ctx* c, const char* fasta, uint64_t nbytes, int fasta_on_device,
                           const uint8_t** fa);

int pk_count(pk_ctx* c, const char* fasta, uint64_t nbytes, int k, int fasta_on_device,
             pk_table* out) {
  if (!c || !out || (!fasta && nbytes)) return PK_EINVAL;
  // a failure before the count itself leaves no stale figures behind
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  int rc = (k <= 32) ? count_impl<uint64_t>(c, fa, nbytes, k) : count_impl<u128>(c, fa, nbytes, k);
  if (rc) return rc;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  return PK_OK;
}

// ---- File input (pk_count_file): file_to_device above the C ABI --------------

int pk_count_file(pk_ctx* c, const char* path, int k, pk_table* out) {
  if (!c || !out || !path) return PK_EINVAL;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  uint64_t n = 0;
  PK_TRY(file_to_device(c, path, &fa, &n));
  int rc = (k <= 32) ? count_impl<uint64_t>(c, fa, n, k) : count_impl<u128>(c, fa, n, k);
  if (rc) return rc;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  return PK_OK;
}

// ---- Allocation-free count (pk_count_noalloc) --------------------------------
// Every intermediate buffer of the count lives in one file-scope device array
// per GPU; its address is taken once per device with hipGetSymbolAddress and
// only that address is handed to kernels and copies.
constexpr uint64_t NOALLOC_SCRATCH = PK_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH];
constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[MAX_DEVICES] = {};

static int scratch_address(pk_ctx* c, char** out) {
  if (c->device < 0 || c->device >= MAX_DEVICES) return c->fail(PK_EINVAL, "device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[c->device]) {
    void* p = nullptr;
    // the calling thread has made c->device current
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return c->hip_fail(e, "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[c->device] = p;
  }
  *out = static_cast<char*>(g_scratch_ptr[c->device]);
  return PK_OK;
}

int pk_count_noalloc(pk_ctx* c, const char* fasta_dev, uint64_t nbytes, int k, uint64_t* keys_dev,
                     int32_t* counts_dev, uint64_t capacity, uint64_t* n_out) {
  if (!c || !n_out || (!fasta_dev && nbytes) || (capacity && (!keys_dev || !counts_dev))) return PK_EINVAL;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  *n_out = 0;
  PK_HIP(c, hipSetDevice(c->device));
  char* arena = nullptr;
  PK_TRY(scratch_address(c, &arena));
  // the scratch array is shared by every call on this device: a call still
  // running on this context's stream finishes before its contents change
  PK_HIP(c, hipStreamSynchronize(c->stream));
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  const int words = k <= 32 ? 1 : 2;
  // the context's own buffers step aside for the call
  DevBuf saved[B_COUNT];
  for (int i = 0; i < B_COUNT; i++) {
    saved[i] = c->buf[i];
    c->buf[i] = DevBuf{};
    c->arena_fixed[i] = false;
  }
  c->buf[B_TK] = DevBuf{keys_dev, capacity * (uint64_t)words * 8};
  c->buf[B_TC] = DevBuf{counts_dev, capacity * 4};
  c->arena_fixed[B_TK] = c->arena_fixed[B_TC] = true;
  c->arena = arena;
  c->arena_cap = NOALLOC_SCRATCH;
  c->arena_mode = true;
  const uint8_t* fa = reinterpret_cast<const uint8_t*>(fasta_dev);
  int rc = PK_OK;
  for (int attempt = 0; attempt < 2; attempt++) {
    c->arena_used = 0;
    c->arena_lim = c->arena_cap;
    c->no_pack = attempt == 1;
    c->out_short = false;
    c->U = 0;
    rc = (k <= 32) ? count_impl<uint64_t>(c, fa, nbytes, k) : count_impl<u128>(c, fa, nbytes, k);
    // the scratch ran out with the packed input in it: once more without
    if (rc != PK_ENOMEM || c->no_pack || c->out_short) break;
    for (int i = 0; i < B_COUNT; i++)
      if (!c->arena_fixed[i]) c->buf[i] = DevBuf{};
    if (hipStreamSynchronize(c->stream) != hipSuccess) break;
  }
  c->no_pack = false;
  c->arena_mode = false;
  for (int i = 0; i < B_COUNT; i++) {
    c->buf[i] = saved[i];
    c->arena_fixed[i] = false;
  }
  // the table lives in the caller's arrays, not in the context
  c->have_table = c->have_kept = c->have_nodes = false;
  if (rc) return rc;
  *n_out = c->U;
  return PK_OK;
}


static int fasta_to_device(pk_ctx* c, const char* fasta, uint64_t nbytes, int fasta_on_device,
                           const uint8_t** fa) {
  if (fasta_on_device) {
    *fa = reinterpret_cast<const uint8_t*>(fasta);
    return PK_OK;
  }
  uint8_t* d;
  PK_TRY(need(c, B_FASTA, nbytes + 64, &d));
  if (nbytes) PK_TRY(h2d_staged(c, d, fasta, nbytes));
  *fa = d;
  return PK_OK;
}

// The rewrite of pk_normalize / pk_count_format; events 17-18 bracket it.
static int normalize_input(pk_ctx* c, const char* data, uint64_t nbytes, int format, int on_device,
                           const uint8_t** out, uint64_t* out_n) {
  if (format != PK_FMT_FASTA_STRICT && format != PK_FMT_FASTA && format != PK_FMT_FASTQ)
    return c->fail(PK_EINVAL, "unknown input format " + std::to_string(format));
  const uint8_t* in;
  PK_TRY(fasta_to_device(c, data, nbytes, on_device, &in));
  c->have_norm = false;
  PK_HIP(c, hipEventRecord(c->ev[17], c->stream));
  if (format == PK_FMT_FASTA_STRICT) {
    uint8_t* d;
    PK_TRY(need(c, B_NORM, nbytes + 64, &d));
    if (nbytes) PK_HIP(c, hipMemcpyAsync(d, in, nbytes, hipMemcpyDeviceToDevice, c->stream));
    *out = d;
    *out_n = nbytes;
  } else {
    PK_TRY(normalize_impl(c, in, nbytes, format, out, out_n));
  }
  PK_HIP(c, hipEventRecord(c->ev[18], c->stream));
  c->norm_n = *out_n;
  c->have_norm = true;
  return PK_OK;
}

int pk_normalize(pk_ctx* c, const char* data, uint64_t nbytes, int format, int data_on_device,
                 uint64_t* out_bytes) {
  if (!c || !out_bytes || (!data && nbytes)) return PK_EINVAL;
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* norm;
  uint64_t nn;
  PK_TRY(normalize_input(c, data, nbytes, format, data_on_device, &norm, &nn));
  c->timing.normalize_ms = 0.f;
  c->pend_norm = true;
  *out_bytes = nn;
  return PK_OK;
}

int pk_download_normalized(pk_ctx* c, char* host_out) {
  if (!c || !host_out) return PK_EINVAL;
  if (!c->have_norm) return c->fail(PK_ESTATE, "no rewritten input");
  if (c->norm_n == 0) return PK_OK;
  return d2h(c, host_out, c->buf[B_NORM].p, c->norm_n);
}

int pk_count_format(pk_ctx* c, const char* data, uint64_t nbytes, int k, int format, int data_on_device,
                    pk_table* out) {
  if (!c || !out || (!data && nbytes)) return PK_EINVAL;
  // a failure before the count itself leaves no stale figures behind
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  PK_HIP(c, hipSetDevice(c->device));
  if (format == PK_FMT_FASTA_STRICT) return pk_count(c, data, nbytes, k, data_on_device, out);
  const uint8_t* norm;
  uint64_t nn;
  PK_TRY(normalize_input(c, data, nbytes, format, data_on_device, &norm, &nn));
  int rc = (k <= 32) ? count_impl<uint64_t>(c, norm, nn, k) : count_impl<u128>(c, norm, nn, k);
  if (rc) return rc;
  c->pend_norm = true;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  return PK_OK;
}

int pk_count_rank_share(pk_ctx* c, const char* fasta, uint64_t nbytes, int k, int nranks, int rank,
                        int fasta_on_device, pk_table* out) {
  if (!c || !out || (!fasta && nbytes)) return PK_EINVAL;
  // a failure before the count itself leaves no stale figures behind
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  if (nranks < 1 || rank < 0 || rank >= nranks) return c->fail(PK_EINVAL, "need 0 <= rank < nranks");
  if (nranks == 1) return pk_count(c, fasta, nbytes, k, fasta_on_device, out);
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  int rc = (k <= 32) ? rank_share_impl<uint64_t>(c, fa, nbytes, k, nranks, rank, false)
                     : rank_share_impl<u128>(c, fa, nbytes, k, nranks, rank, false);
  if (rc) return rc;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  return PK_OK;
}

int pk_count_rank_share_by_key(pk_ctx* c, const char* fasta, uint64_t nbytes, int k, int nranks, int rank,
                               int fasta_on_device, pk_table* out) {
  if (!c || !out || (!fasta && nbytes)) return PK_EINVAL;
  if (k < 8 || k > 64) return c->fail(PK_EINVAL, "k must be in [8, 64]");
  if (nranks < 1 || rank < 0 || rank >= nranks) return c->fail(PK_EINVAL, "need 0 <= rank < nranks");
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  if (nranks == 1) return pk_count(c, fasta, nbytes, k, fasta_on_device, out);
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  int rc = (k <= 32) ? rank_share_impl<uint64_t>(c, fa, nbytes, k, nranks, rank, true)
                     : rank_share_impl<u128>(c, fa, nbytes, k, nranks, rank, true);
  if (rc) return rc;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  return PK_OK;
}

int pk_lmer_frequency(pk_ctx* c, const char* fasta, uint64_t nbytes, int fasta_on_device,
                      uint64_t* freq_host) {
  if (!c || !freq_host || (!fasta && nbytes)) return PK_EINVAL;
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  ull* freq;
  auto packed = [&]() -> int {
    Records rec;
    rec.n = nbytes;
    PK_TRY(pack_buffers(c, nbytes, true, &rec.pk));
    PK_TRY(windows_main(c, fa, nbytes, LMER_L, &rec));
    return lmer_frequency_impl(c, rec, rec.pk.W, &freq);
  };
  int rc = packed();
  if (rc == PK_ENOMEM) {
    c->idle[B_PACK] = c->idle[B_LPART] = c->idle[B_WCNT] = c->idle[B_WOFF] = true;
    Records rec;
    PK_TRY(records_main(c, fa, nbytes, LMER_L, &rec));
    PK_TRY(need(c, B_LFREQ, LMER_BINS, &freq));
    PK_TRY(fill_u64(c, freq, 0, LMER_BINS));
    if (rec.R) {
      hipLaunchKernelGGL(k_lmer_walk, dim3((unsigned)std::min<uint64_t>(grid_for(rec.R, 256), 4096)), dim3(256), 0,
                         c->stream, fa, rec.rstart, rec.rlen, rec.R, freq);
      PK_HIP(c, hipGetLastError());
    }
    rc = PK_OK;
  }
  if (rc) return rc;
  return d2h(c, freq_host, freq, LMER_BINS * 8);
}

int pk_builder_count(pk_ctx* c, const char* fasta, uint64_t nbytes, int klen, uint64_t read_len,
                     int kmer_bits, char delimiter, char skip_symbol, int fasta_on_device,
                     pk_table* out, uint64_t* n_reads) {
  if (!c || !out || (!fasta && nbytes)) return PK_EINVAL;
  if (kmer_bits != 64 && kmer_bits != 128) return c->fail(PK_EINVAL, "kmer_bits must be 64 or 128");
  if (klen < 1) return c->fail(PK_EINVAL, "klen must be >= 1");
  if (read_len > 0xFFFFFFF0ull) return c->fail(PK_EINVAL, "read_len must be < 2^32 - 16");
  if (delimiter == skip_symbol) return c->fail(PK_EINVAL, "delimiter and skip_symbol must differ");
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = false;
  const BldSyms sy{(uint8_t)delimiter, (uint8_t)skip_symbol};
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  int rc = kmer_bits == 64 ? builder_count_impl<uint64_t>(c, fa, nbytes, klen, read_len, sy)
                           : builder_count_impl<u128>(c, fa, nbytes, klen, read_len, sy);
  if (rc) return rc;
  out->n = c->U;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_TK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_TC].p);
  if (n_reads) *n_reads = c->R;
  return PK_OK;
}

int pk_builder_count_windows(pk_ctx* c, const char* fasta, uint64_t nbytes, int klen, uint64_t read_len,
                             char delimiter, char skip_symbol, int mode, int fasta_on_device, uint64_t* n_reads,
                             uint64_t* n_windows, uint64_t* n_distinct) {
  if (!c || !n_reads || !n_windows || !n_distinct || (!fasta && nbytes)) return PK_EINVAL;
  if (mode != PK_WINDOWS_V0 && mode != PK_WINDOWS_V1) return c->fail(PK_EINVAL, "unknown window mode");
  if (klen < 1 || klen > 128) return c->fail(PK_EINVAL, "klen must be in [1, 128]");
  if (read_len > 0xFFFFFFF0ull) return c->fail(PK_EINVAL, "read_len must be < 2^32 - 16");
  if (read_len < (uint64_t)klen)
    return c->fail(PK_EINVAL, "read_len < klen: the reference's window count wraps below zero");
  if (delimiter == skip_symbol) return c->fail(PK_EINVAL, "delimiter and skip_symbol must differ");
  c->timing = pk_timing{};
  c->pend_count = c->pend_split = c->pend_cutoff = c->pend_mn = c->pend_norm = false;
  c->have_table = c->have_kept = c->have_nodes = false;
  begin_buffers(c);
  const BldSyms sy{(uint8_t)delimiter, (uint8_t)skip_symbol};
  PK_HIP(c, hipSetDevice(c->device));
  const uint8_t* fa;
  PK_TRY(fasta_to_device(c, fasta, nbytes, fasta_on_device, &fa));
  hipStream_t st = c->stream;
  PK_HIP(c, hipEventRecord(c->ev[0], st));
  ull* small;
  PK_TRY(need(c, B_SMALL, 16, &small));
  PK_TRY(fill_u64(c, small, ~0ull, 4));
  PK_TRY(fill_u64(c, small + 12, 0, 2));
  ull* ev;
  uint64_t m, p0;
  PK_TRY(event_index(c, fa, nbytes, sy.delim, sy.skip, small, &ev, &m, &p0));
  ull *rstart, *woff, *idx;
  uint32_t *rlen, *wc, *flag;
  uint32_t* bad = reinterpret_cast<uint32_t*>(small + 12);
  uint32_t* present = reinterpret_cast<uint32_t*>(small + 8);  // 8 words = small[8..11]
  PK_TRY(need(c, B_TU, m + 1, &flag));
  PK_TRY(need(c, B_UOFF, m + 2, &idx));
  if (m) {
    hipLaunchKernelGGL(k_win_flags, dim3(grid_for(m, 256)), dim3(256), 0, st, fa, nbytes, ev, m, klen, read_len, sy,
                       flag, bad);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, flag, idx, m));
  PK_TRY(fetch(c, Post{{idx + m, reinterpret_cast<const ull*>(bad)}, {1, 1}}));
  const ull hv[2] = {c->box[0], c->box[1]};
  const uint64_t R = hv[0];
  const bool cut = (hv[1] & 0xFFFFFFFFull) != 0, shorter = (hv[1] >> 32) != 0;
  // concurrent_kmer_counter.hpp:965-967 throws on a read cut short; _v1
  // sizes its window array with read_len - klen + 1 (:1427), which wraps
  // for a read shorter than klen
  if (mode == PK_WINDOWS_V0 && cut) return c->fail(PK_EFORMAT, "Variable size read");
  if (mode == PK_WINDOWS_V1 && shorter) return c->fail(PK_EFORMAT, "a read is shorter than klen");
  PK_TRY(need(c, B_RSTART, R + 1, &rstart));
  PK_TRY(need(c, B_RLEN, R + 1, &rlen));
  PK_TRY(need(c, B_KC, R + 1, &wc));
  PK_TRY(need(c, B_KOFS, R + 2, &woff));
  if (m) {
    hipLaunchKernelGGL(k_win_write, dim3(grid_for(m, 256)), dim3(256), 0, st, fa, nbytes, ev, m, klen, read_len, sy,
                       idx, rstart, rlen, wc);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(scan_excl<uint32_t>(c, wc, woff, R));
  PK_TRY(fill_u64(c, small + 8, 0, 4));
  if (R) {
    hipLaunchKernelGGL(k_win_alpha, dim3((unsigned)std::min<uint64_t>((R + 3) / 4, 4096)), dim3(64, 4), 0, st, fa,
                       rstart, rlen, R, present);
    PK_HIP(c, hipGetLastError());
  }
  PK_TRY(fetch(c, Post{{small + 8, woff + R}, {4, 1}}));
  ull hp[5];
  memcpy(hp, c->box, sizeof(hp));
  const uint64_t N = hp[4];
  // byte value -> rank among the values present
  const uint32_t* pw = reinterpret_cast<const uint32_t*>(hp);
  int nval = 0;
  for (int v = 0; v < 256; v++) {
    c->win_lut[v] = 0;
    if (pw[v >> 5] >> (v & 31) & 1u) c->win_lut[v] = (uint8_t)nval++;
  }
  int bits = 1;
  while ((1 << bits) < nval) bits++;
  int KB = klen * bits;
  if (KB > 128)
    return c->fail(PK_EINVAL, "the reads hold " + std::to_string(nval) + " byte values: " + std::to_string(klen) +
                                  " x " + std::to_string(bits) + " bits exceed a 128-bit window key");
  KB += KB & 1;
  const int has_nul = (pw[0] & 1u) ? 1 : 0;
  uint8_t* lut;
  PK_TRY(need(c, B_WORDER, 256, &lut));
  PK_HIP(c, hipMemcpyAsync(lut, c->win_lut, 256, hipMemcpyHostToDevice, st));
  int rc = KB <= 64 ? windows_count_impl<uint64_t>(c, fa, rstart, rlen, woff, R, N, klen, bits, lut, has_nul, KB)
                    : windows_count_impl<u128>(c, fa, rstart, rlen, woff, R, N, klen, bits, lut, has_nul, KB);
  if (rc) return rc;
  *n_reads = R;
  *n_windows = N;
  *n_distinct = c->U;
  return PK_OK;
}

int pk_cutoff(pk_ctx* c, int t, uint64_t* hist_t, int* min_bucket, uint64_t* n_kept) {
  if (!c || !min_bucket || !n_kept) return PK_EINVAL;
  if (!c->have_table) return c->fail(PK_ESTATE, "pk_cutoff before pk_count");
  if (t == 0) t = 21;
  if (t < 0 || t > T_MAX) return c->fail(PK_EINVAL, "t must be in [0, 4096]");
  PK_HIP(c, hipSetDevice(c->device));
  return c->words == 1 ? cutoff_impl<uint64_t>(c, t, hist_t, min_bucket, n_kept)
                       : cutoff_impl<u128>(c, t, hist_t, min_bucket, n_kept);
}

int pk_cutoff_threshold(pk_ctx* c, uint64_t threshold, uint64_t* n_kept) {
  if (!c || !n_kept) return PK_EINVAL;
  if (!c->have_table) return c->fail(PK_ESTATE, "pk_cutoff_threshold before a count");
  PK_HIP(c, hipSetDevice(c->device));
  if (threshold >= 0x7FFFFFFFull) {
    // counts are int32: no count exceeds such a threshold, the kept table is empty
    PK_HIP(c, hipStreamSynchronize(c->stream));
    int32_t* KC;
    uint64_t* KK;
    PK_TRY(need(c, B_KK, c->words, &KK));
    PK_TRY(need(c, B_KC2, 1, &KC));
    c->V = 0;
    c->t = 1;
    c->mb = 0;
    c->have_kept = true;
    c->have_nodes = false;
    c->pend_cutoff = false;
    c->timing.cutoff_ms = 0.f;
    *n_kept = 0;
    return PK_OK;
  }
  const int mb = (int)threshold + 1;
  int mbo = 0;
  return c->words == 1 ? cutoff_impl<uint64_t>(c, 1, nullptr, &mbo, n_kept, mb)
                       : cutoff_impl<u128>(c, 1, nullptr, &mbo, n_kept, mb);
}

int pk_kept_table(pk_ctx* c, pk_table* out) {
  if (!c || !out) return PK_EINVAL;
  if (!c->have_kept) return c->fail(PK_ESTATE, "no kept table");
  out->n = c->V;
  out->words = c->words;
  out->k = c->k;
  out->keys = reinterpret_cast<const uint64_t*>(c->buf[B_KK].p);
  out->counts = reinterpret_cast<const int32_t*>(c->buf[B_KC2].p);
  return PK_OK;
}

int pk_macro_nodes(pk_ctx* c, pk_mn_table* out) {
  if (!c || !out) return PK_EINVAL;
  if (!c->have_kept || c->V == 0) return c->fail(PK_ESTATE, "pk_macro_nodes needs a non-empty kept table");
  if (c->key_bits != 2 * c->k)
    return c->fail(PK_ESTATE, "macro nodes need k-mer keys of exactly 2k bits (builder tables with "
                              "klen != 4 * sizeof(kmer_t) keep extra bases)");
  PK_HIP(c, hipSetDevice(c->device));
  int rc = c->words == 1 ? mn_impl<uint64_t>(c) : mn_impl<u128>(c);
  if (rc) return rc;
  out->n = c->M;
  out->k = c->k;
  out->nodes = reinterpret_cast<const pk_mnode*>(c->buf[B_NODES].p);
  return PK_OK;
}

int pk_macro_nodes_rank_share(pk_ctx* c, int nranks, int rank, pk_mn_table* out) {
  if (!c || !out) return PK_EINVAL;
  if (nranks < 1 || rank < 0 || rank >= nranks) return c->fail(PK_EINVAL, "need 0 <= rank < nranks");
  PK_TRY(pk_macro_nodes(c, out));
  if (nranks == 1) return PK_OK;
  int rc = c->words == 1 ? node_share_impl<uint64_t>(c, nranks, rank) : node_share_impl<u128>(c, nranks, rank);
  if (rc) return rc;
  out->n = c->M;
  return PK_OK;
}

int pk_mn_wiring(pk_ctx* c, int coverage, const uint8_t* pre_order, pk_mnwire* out) {
  if (!c || !out || coverage < 1) return PK_EINVAL;
  if (!c->have_nodes) return c->fail(PK_ESTATE, "pk_mn_wiring before pk_macro_nodes");
  if (c->M == 0) return PK_OK;
  PK_HIP(c, hipSetDevice(c->device));
  uint8_t* ord = nullptr;
  if (pre_order) {
    PK_TRY(need(c, B_WORDER, c->M * 4, &ord));
    PK_HIP(c, hipMemcpyAsync(ord, pre_order, c->M * 4, hipMemcpyHostToDevice, c->stream));
  }
  pk_mnwire* w;
  PK_TRY(need(c, B_WIRE, c->M, &w));
  hipLaunchKernelGGL(k_mn_wire, dim3(grid_for(c->M, 256)), dim3(256), 0, c->stream,
                     reinterpret_cast<const MnRec*>(c->buf[B_NODES].p), c->M, ord, coverage, w);
  PK_HIP(c, hipGetLastError());
  return d2h(c, out, w, c->M * sizeof(pk_mnwire));
}

int pk_download_table(pk_ctx* c, uint64_t* keys, int32_t* counts) {
  if (!c) return PK_EINVAL;
  if (!c->have_table) return c->fail(PK_ESTATE, "no table");
  if (c->U == 0) return PK_OK;
  if (keys) PK_TRY(d2h(c, keys, c->buf[B_TK].p, c->U * c->words * 8));
  if (counts) PK_TRY(d2h(c, counts, c->buf[B_TC].p, c->U * 4));
  return PK_OK;
}

int pk_download_kept(pk_ctx* c, uint64_t* keys, int32_t* counts) {
  if (!c) return PK_EINVAL;
  if (!c->have_kept) return c->fail(PK_ESTATE, "no kept table");
  if (c->V == 0) return PK_OK;
  if (keys) PK_TRY(d2h(c, keys, c->buf[B_KK].p, c->V * c->words * 8));
  if (counts) PK_TRY(d2h(c, counts, c->buf[B_KC2].p, c->V * 4));
  return PK_OK;
}

int pk_download_nodes(pk_ctx* c, pk_mnode* nodes) {
  if (!c || !nodes) return PK_EINVAL;
  if (!c->have_nodes) return c->fail(PK_ESTATE, "no macro nodes");
  if (c->M == 0) return PK_OK;
  return d2h(c, nodes, c->buf[B_NODES].p, c->M * sizeof(pk_mnode));
}

int pk_last_timing(const pk_ctx* cc, pk_timing* out) {
  if (!cc || !out) return PK_EINVAL;
  pk_ctx* c = const_cast<pk_ctx*>(cc);
  auto el = [&](int a, int b) {
    float v = 0;
    (void)hipEventElapsedTime(&v, c->ev[a], c->ev[b]);
    return v;
  };
  if (c->pend_count || c->pend_cutoff || c->pend_mn || c->pend_norm) {
    PK_HIP(c, hipSetDevice(c->device));
    PK_HIP(c, hipStreamSynchronize(c->stream));
  }
  if (c->pend_count) {
    c->timing.parse_ms = el(0, c->ev_parsed);
    c->timing.hist_ms = c->have_hist ? el(2, 3) : 0.f;
    c->timing.scatter_ms = el(4, 5);
    c->timing.l1_scatter_ms = el(4, 16);
    c->timing.sort_ms = el(5, 7);
    c->timing.split_ms = c->pend_split ? el(8, 9) : 0.f;
    c->timing.compact_ms = el(10, 11);
    const int nl = c->ms_levels < MS_TIMED_LEVELS ? c->ms_levels : MS_TIMED_LEVELS;
    c->timing.ms_hist_ms = c->timing.ms_scatter_ms = 0.f;
    for (int l = 0; l < MS_TIMED_LEVELS; l++) {
      const bool on = l < nl;
      c->timing.ms_level_hist_ms[l] = 0.f;  // no level has a histogram pass
      c->timing.ms_level_scatter_ms[l] = on ? el(20 + 2 * l, 21 + 2 * l) : 0.f;
      c->timing.ms_level_form[l] = on ? c->ms_form[l] : 0;
      c->timing.ms_scatter_ms += c->timing.ms_level_scatter_ms[l];
    }
    c->timing.ms_levels = c->ms_levels;
    c->pend_count = false;
  }
  if (c->pend_cutoff) {
    c->timing.cutoff_ms = el(12, 13);
    c->pend_cutoff = false;
  }
  if (c->pend_mn) {
    c->timing.mn_ms = el(14, 15);
    c->pend_mn = false;
  }
  if (c->pend_norm) {
    c->timing.normalize_ms = el(17, 18);
    c->pend_norm = false;
  }
  *out = c->timing;
  return PK_OK;
}

}  // extern "C"
