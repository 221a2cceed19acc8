// sxc_kmatch_unique.h -- KMatch's device path for max_freq = 1 (SatsumaSynteny2's setting): the
// k-mers that occur once in each genome, joined without sorting the tables, and the blocks
// chained and ordered on the device.
//
// The general path (sxc_kmatch.hip) sorts each genome's table by k-mer, six to eight radix
// passes over 16-byte entries, then filters, compacts, and searches one table for every entry
// of the other.  With max_freq = 1 none of that order is needed: a k-mer matters when exactly
// one entry of either genome has it.  So both genomes' entries {hashed k-mer, position} go into
// one array, two radix passes (three above 26 M entries) bring equal k-mers into the same bucket
// of about 200 .. 400 entries, and one wave per bucket counts them in an LDS hash table.  Bound
// by HBM: 12 bytes per position written once, and read and written once per radix pass.
// Measured, host bytes in and records out, in a loop over the same genomes: two 12-Mbp genomes, K = 21,
// 13.4 -> 2.3 ms (device phase 6.3 -> 2.1 ms, most of it the upload; chaining 1.7 ms on the host
// before), with other genomes at each call 21 to 23 -> 3.1 ms; two 1.2-Mbp genomes 5.2 -> 0.6 ms.
//
// Chaining (dump_matching_blocks, kmatch/KMatch.cc:196-318).  A joined position extends the open
// block on its diagonal if that block's end lies at most max_jump before it, and as positions
// are sorted by query and unique, that end is the nearest earlier position on the diagonal and
// at most max_jump entries back.  So links are found by looking back a few entries, a block is
// a chain of links, its first entry is found through per-tile roots, and its place in the output
// -- the step that closes it, then creation order -- follows from its last entry, blocks closed
// by the same step being neighbours among the last entries.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/sxc_kmatch.h"

namespace sxc {
namespace km {

constexpr int64_t kStride = 10000000000LL;  // KMATCH_POSITION_CHR_CNST (KMatch.h:18)
constexpr uint32_t kNone = 0xffffffffu;     // no entry of this k-mer on a side
constexpr uint32_t kMulti = 0xfffffffeu;    // more than one
constexpr uint32_t kNeg = 0x80000000u;      // the reverse complement was the smaller
// A bijection of the 64-bit words (a product, its upper half folded into the lower, twice): the low bits
// spread the k-mers over the buckets, the top bits over a bucket's table.  (Once leaves bits 52 and up out
// of the low 20: the first five bases of 31, whose 1024 variants before one 26-mer, as before the
// homopolymer runs of two 200-Mbp genomes, then shared a bucket and filled its table.)  (The radix sort is given
// low bits, as no call ends at bit 64: see sort_pairs.)
constexpr uint64_t kMul = 0x9E3779B97F4A7C15ull;
constexpr uint64_t inverse(uint64_t a) {
  uint64_t x = a;  // correct to 3 bits, doubled by each step
  for (int i = 0; i < 6; ++i) x *= 2 - a * x;
  return x;
}
constexpr uint64_t kInv = inverse(kMul);
static_assert(kMul * kInv == 1, "");
__host__ __device__ constexpr uint64_t fold(uint64_t x) { return x ^ (x >> 32); }  // its own inverse
__host__ __device__ constexpr uint64_t mix(uint64_t kmer) { return fold(fold(kmer * kMul) * kMul); }
__host__ __device__ constexpr uint64_t unmix(uint64_t h) { return fold(fold(h) * kInv) * kInv; }
static_assert(unmix(mix(0x123456789abcdefull)) == 0x123456789abcdefull, "");
constexpr uint64_t kFree = mix(1ull << 63);  // the image of 2^63, which no k-mer is (K <= 31)

constexpr int kTable = 1024;        // hash slots of a bucket
constexpr int kHeavy = 16384;       // buckets above this are counted by several workgroups
constexpr int kBucketGroups = 2048; // workgroups of one wave: 8 per CU
constexpr int kTile = 1024;         // entries per workgroup of the compactions and the chaining
constexpr int kDense = 4096;        // positions per workgroup of the first compaction

// Control words in device memory.
struct Ctl {
  unsigned long long n;         // entries written
  unsigned long long filled[2]; // k-mers of the query and of the target
  unsigned long long kept[2];   // k-mers that occur once
  unsigned long long joined, blocks;
  uint32_t drop[2];             // position of the entry with the largest kept k-mer
  uint32_t heavy;               // buckets above kHeavy
  uint32_t overflow;            // a bucket held more than kTable k-mers: the general path decides
};

__device__ inline uint32_t code_of(uint32_t b) {  // 2-bit code of A/C/G/T in either case
  return ((b >> 1) ^ (b >> 2)) & 3u;
}
__device__ inline bool is_acgt(uint32_t b) {
  const uint32_t u = b & 0xdfu;
  return u == 'A' || u == 'C' || u == 'G' || u == 'T';
}

// Canonical k-mers of 16 positions per thread.  The workgroup's 4096 + K - 1 bytes are read once,
// 16 at a time, and packed to 2-bit codes and a bit per letter other than A/C/G/T in LDS; a thread
// then builds the first window from three words and rolls it.  Entries are written position
// round by position round, so that a wave's stores are one contiguous run each; their order does
// not matter.
__global__ __launch_bounds__(256) void k_unique_kmers(const unsigned char* buf, int64_t len, int64_t len_q, int K,
                                                      uint64_t* keys, uint32_t* vals, Ctl* ctl) {
  __shared__ uint32_t pk[258], bad[258];
  __shared__ uint32_t wsum[4], wq[4];
  __shared__ unsigned long long base;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t w0 = (int64_t)blockIdx.x * 4096;  // the group's positions: windows that end there
  // words -2 .. 255 of 16 positions: two words of read-behind hold the K - 1 <= 30 before w0
  for (int w = t; w < 258; w += 256) {
    const int64_t p = w0 + 16 * (int64_t)(w - 2);
    uint32_t c = 0, m = 0xffffu;
    if (p >= 0 && p < len) {
      const uint4 v = *(const uint4*)(buf + p);  // the buffer is padded to a multiple of 16
      const uint32_t x[4] = {v.x, v.y, v.z, v.w};
      m = 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t b = (x[i >> 2] >> (8 * (i & 3))) & 255u;
        c |= code_of(b) << (2 * i);
        m |= (is_acgt(b) && p + i < len ? 0u : 1u) << i;
      }
    }
    pk[w] = c;
    bad[w] = m;
  }
  __syncthreads();
  // bit j of ok: the window ending at position p0 + j holds K letters A/C/G/T
  const uint64_t bm = (uint64_t)bad[t] | ((uint64_t)bad[t + 1] << 16) | ((uint64_t)bad[t + 2] << 32);
  uint64_t any = bm;
  for (int have = 1; have < K;) {
    const int step = have < K - have ? have : K - have;
    any |= any << step;
    have += step;
  }
  const uint32_t ok = ~(uint32_t)(any >> 32) & 0xffffu;
  const uint32_t total = __popc(ok);
  const int64_t p0 = w0 + 16 * (int64_t)t;
  // entries of the wave and of the group, and how many of them are the query's
  uint32_t nq = 0;
  if (p0 < len_q) nq = __popc(p0 + 16 <= len_q ? ok : ok & ((1u << (int)(len_q - p0)) - 1));
  uint32_t ws = total, wqs = nq;
  for (int d = 32; d > 0; d >>= 1) {
    ws += __shfl_xor(ws, d, 64);
    wqs += __shfl_xor(wqs, d, 64);
  }
  if (lane == 0) {
    wsum[wave] = ws;
    wq[wave] = wqs;
  }
  __syncthreads();
  if (t == 0) {
    const uint32_t s = wsum[0] + wsum[1] + wsum[2] + wsum[3], q = wq[0] + wq[1] + wq[2] + wq[3];
    base = s ? atomicAdd(&ctl->n, (unsigned long long)s) : 0;
    if (q) atomicAdd(&ctl->filled[0], (unsigned long long)q);
    if (s > q) atomicAdd(&ctl->filled[1], (unsigned long long)(s - q));
  }
  __syncthreads();
  uint64_t at = base;
  for (int w = 0; w < wave; ++w) at += wsum[w];
  // codes of positions p0 - 32 .. p0 + 15, 2 bits each: lo the first 32, hi the thread's own
  const uint64_t lo = (uint64_t)pk[t] | ((uint64_t)pk[t + 1] << 32);
  const uint32_t hi = pk[t + 2];
  const uint64_t mask = (1ull << (2 * K)) - 1;
  const int top = 2 * (K - 1);
  // the K - 1 bases before p0: f has the first base in its top bits, r the complements reversed
  uint64_t f = 0, r = 0;
  if (K > 1) {
    const uint64_t w = lo >> (64 - top);  // first base in the low bits
    uint64_t rev = __brevll(w);
    rev = ((rev >> 1) & 0x5555555555555555ull) | ((rev & 0x5555555555555555ull) << 1);
    f = rev >> (64 - top);
    r = (~w & (mask >> 2)) << 2;
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const uint64_t code = (hi >> (2 * j)) & 3u;
    f = ((f << 2) + code) & mask;
    r = (r >> 2) + ((3 - code) << top);
    const bool v = (ok >> j) & 1u;
    const unsigned long long lanes = __ballot(v);
    if (v) {
      const uint64_t o = at + (uint64_t)__popcll(lanes & ((1ull << lane) - 1));
      const uint32_t start = (uint32_t)(p0 + j - (K - 1));
      keys[o] = mix(f <= r ? f : r);
      vals[o] = f <= r ? start : start | kNeg;
    }
    at += (uint64_t)__popcll(lanes);
  }
}

// Table slots no k-mer fills are entries {0, 0} in the reference.  One is an entry of k-mer 0 like
// any other; two or more only have to make it occur more than once.  Their position is the 'N'
// before the first sequence, which no k-mer starts at.
__global__ void k_unique_unfilled(uint64_t* keys, uint32_t* vals, int64_t slots_q, int64_t slots_t, uint32_t len_q,
                                  Ctl* ctl) {
  unsigned long long n = ctl->n;
  for (int s = 0; s < 2; ++s) {
    const int64_t z = (s ? slots_t : slots_q) - (int64_t)ctl->filled[s];
    for (int64_t k = 0; k < (z < 2 ? z : 2); ++k, ++n) {
      keys[n] = 0;
      vals[n] = (s ? len_q : 0u) | kNeg;
    }
  }
  ctl->n = n;
}

// First entry of every bucket.
__global__ __launch_bounds__(256) void k_bounds(const uint64_t* keys, uint32_t n, uint32_t buckets, uint32_t* start) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i > n) return;
  const uint32_t b1 = i < n ? (uint32_t)keys[i] & (buckets - 1) : buckets;
  const uint32_t b0 = i > 0 ? ((uint32_t)keys[i - 1] & (buckets - 1)) + 1 : 0;
  for (uint32_t b = b0; b <= b1; ++b) start[b] = i;
}

// The buckets above kHeavy.
__global__ __launch_bounds__(256) void k_heavy_list(const uint32_t* start, uint32_t buckets, uint32_t* list, Ctl* ctl) {
  const uint32_t b = blockIdx.x * 256u + threadIdx.x;
  if (b < buckets && start[b + 1] - start[b] > kHeavy) list[atomicAdd(&ctl->heavy, 1u)] = b;
}

struct Table {
  uint64_t* key;
  uint32_t* pos;  // kTable of the query, then kTable of the target
};

// Counts one entry: v is a position, or kMulti for several.  False if the table is full.
__device__ inline bool put(const Table& T, uint64_t h, uint32_t slot, int side, uint32_t v) {
  for (int k = 0; k < kTable; ++k) {
    const uint64_t was = atomicCAS((unsigned long long*)&T.key[slot], (unsigned long long)kFree, (unsigned long long)h);
    if (was == kFree || was == h) {
      uint32_t* p = &T.pos[side * kTable + (int)slot];
      if (v == kMulti || atomicCAS(p, kNone, v) != kNone) atomicExch(p, kMulti);
      return true;
    }
    slot = (slot + 1) & (kTable - 1);
  }
  return false;
}

static_assert(kTable == 1 << 10, "");
__device__ inline uint32_t slot_of(uint64_t h) { return (uint32_t)(h >> 54); }

__device__ inline void clear(const Table& T, int t, int nt) {
  for (int i = t; i < kTable; i += nt) {
    T.key[i] = kFree;
    T.pos[i] = kNone;
    T.pos[kTable + i] = kNone;
  }
}

// What a lane has seen of the kept k-mers.
struct Seen {
  unsigned long long kept[2] = {0, 0};
  uint64_t best[2] = {0, 0};
  uint32_t at[2] = {kNone, kNone};
};

__device__ inline void look(const Table& T, int i, uint32_t len_q, uint32_t* dense, Seen& s) {
  const uint64_t h = T.key[i];
  if (h == kFree) return;
  const uint64_t kmer = unmix(h);
  const uint32_t v[2] = {T.pos[i], T.pos[kTable + i]};
#pragma unroll
  for (int side = 0; side < 2; ++side)
    if (v[side] < kMulti) {
      ++s.kept[side];
      if (s.at[side] == kNone || kmer > s.best[side]) {
        s.best[side] = kmer;
        s.at[side] = v[side] & ~kNeg;
      }
    }
  // orientation = sign of the query position xor the target's (KMatch.cc:141-177)
  if (v[0] < kMulti && v[1] < kMulti)
    dense[v[0] & ~kNeg] = ((v[1] & ~kNeg) - len_q + 1) | ((v[0] ^ v[1]) & kNeg);
}

// The wave's Seen into slot `w` of the per-wave results.
__device__ inline void store_seen(Seen s, int w, uint64_t* best, uint32_t* at, Ctl* ctl) {
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    for (int d = 32; d > 0; d >>= 1) {
      s.kept[side] += __shfl_xor(s.kept[side], d, 64);
      const uint64_t b = __shfl_xor((unsigned long long)s.best[side], d, 64);
      const uint32_t a = __shfl_xor(s.at[side], d, 64);
      if (a != kNone && (s.at[side] == kNone || b > s.best[side])) {
        s.best[side] = b;
        s.at[side] = a;
      }
    }
    if ((threadIdx.x & 63) == 0) {
      best[2 * w + side] = s.best[side];
      at[2 * w + side] = s.at[side];
      if (s.kept[side]) atomicAdd(&ctl->kept[side], s.kept[side]);
    }
  }
}

// One wave per workgroup, walking buckets: 16 KB of LDS each, ten to a CU.
__global__ __launch_bounds__(64) void k_buckets(const uint64_t* keys, const uint32_t* vals, const uint32_t* start,
                                                uint32_t buckets, uint32_t len_q, uint32_t* dense, uint64_t* best,
                                                uint32_t* at, Ctl* ctl) {
  __shared__ uint64_t skey[kTable];
  __shared__ uint32_t spos[2 * kTable];
  const Table T{skey, spos};
  const int t = threadIdx.x;
  Seen s;
  bool full = false;
  for (uint32_t b = blockIdx.x; b < buckets; b += gridDim.x) {
    const uint32_t lo = start[b], hi = start[b + 1];
    if (hi == lo || hi - lo > kHeavy) continue;
    clear(T, t, 64);
    __syncthreads();
    for (uint32_t i = lo + t; i < hi; i += 64) {
      const uint64_t h = keys[i];
      const uint32_t v = vals[i];
      full |= !put(T, h, slot_of(h), (v & ~kNeg) >= len_q, v);
    }
    __syncthreads();
    for (int i = t; i < kTable; i += 64) look(T, i, len_q, dense, s);
    __syncthreads();
  }
  if (full) ctl->overflow = 1;
  store_seen(s, (int)blockIdx.x, best, at, ctl);
}

// Heavy buckets (a k-mer repeated very often): shares of kHeavy entries are counted in LDS by a
// workgroup each and added into the bucket's table in global memory.
__global__ __launch_bounds__(256) void k_heavy_clear(const Ctl* ctl, uint64_t* gkey, uint32_t* gpos) {
  for (uint32_t h = blockIdx.x; h < ctl->heavy; h += gridDim.x) {
    const Table G{gkey + (size_t)h * kTable, gpos + (size_t)h * 2 * kTable};
    clear(G, threadIdx.x, 256);
  }
}

__global__ __launch_bounds__(256) void k_heavy_count(const uint64_t* keys, const uint32_t* vals, const uint32_t* start,
                                                     const uint32_t* list, uint32_t len_q, uint64_t* gkey,
                                                     uint32_t* gpos, Ctl* ctl) {
  __shared__ uint64_t skey[kTable];
  __shared__ uint32_t spos[2 * kTable];
  const Table T{skey, spos};
  const int t = threadIdx.x;
  bool full = false;
  for (uint32_t h = 0; h < ctl->heavy; ++h) {
    const uint32_t b = list[h];
    const uint64_t lo = start[b], hi = start[b + 1];
    const Table G{gkey + (size_t)h * kTable, gpos + (size_t)h * 2 * kTable};
    for (uint64_t c = lo + (uint64_t)blockIdx.x * kHeavy; c < hi; c += (uint64_t)gridDim.x * kHeavy) {
      const uint64_t e = c + kHeavy < hi ? c + kHeavy : hi;
      clear(T, t, 256);
      __syncthreads();
      for (uint64_t i = c + t; i < e; i += 256) {
        const uint64_t k = keys[i];
        const uint32_t v = vals[i];
        full |= !put(T, k, slot_of(k), (v & ~kNeg) >= len_q, v);
      }
      __syncthreads();
      for (int i = t; i < kTable; i += 256) {
        const uint64_t k = skey[i];
        if (k == kFree) continue;
        for (int side = 0; side < 2; ++side)
          if (spos[side * kTable + i] != kNone) full |= !put(G, k, slot_of(k), side, spos[side * kTable + i]);
      }
      __syncthreads();
    }
  }
  if (full) ctl->overflow = 1;
}

__global__ __launch_bounds__(64) void k_heavy_look(uint32_t len_q, uint64_t* gkey, uint32_t* gpos, uint32_t* dense,
                                                   uint64_t* best, uint32_t* at, Ctl* ctl) {
  Seen s;
  for (uint32_t h = blockIdx.x; h < ctl->heavy; h += gridDim.x) {
    const Table G{gkey + (size_t)h * kTable, gpos + (size_t)h * 2 * kTable};
    for (int i = threadIdx.x; i < kTable; i += 64) look(G, i, len_q, dense, s);
  }
  store_seen(s, (int)blockIdx.x, best, at, ctl);
}

// The entry with the largest kept k-mer of each genome, which the reference drops with the last
// slot of its table (kposv.resize(wi - 1), KMatch.cc:124-129).  One wave.
__global__ __launch_bounds__(64) void k_last(const uint64_t* best, const uint32_t* at, int waves, Ctl* ctl) {
  for (int side = 0; side < 2; ++side) {
    uint64_t b = 0;
    uint32_t a = kNone;
    for (int w = threadIdx.x; w < waves; w += 64)
      if (at[2 * w + side] != kNone && (a == kNone || best[2 * w + side] > b)) {
        b = best[2 * w + side];
        a = at[2 * w + side];
      }
    for (int d = 32; d > 0; d >>= 1) {
      const uint64_t ob = __shfl_xor((unsigned long long)b, d, 64);
      const uint32_t oa = __shfl_xor(a, d, 64);
      if (oa != kNone && (a == kNone || ob > b)) {
        b = ob;
        a = oa;
      }
    }
    if (threadIdx.x == 0) ctl->drop[side] = a;
  }
}

// ---- order-preserving compaction: counts per workgroup, one exclusive scan of them, writes

// Exclusive scan over a 256-thread workgroup; *total gets the sum.
__device__ inline uint32_t group_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t ws[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc = v;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = __shfl_up(inc, d, 64);
    if (lane >= d) inc += o;
  }
  if (lane == 63) ws[wave] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += ws[w];
    all += ws[w];
  }
  __syncthreads();
  *total = all;
  return before + inc - v;
}

// Exclusive scan of n group counts in place; the sum goes to *total.  One workgroup.
__global__ __launch_bounds__(1024) void k_scan_groups(uint32_t* count, int n, unsigned long long* total) {
  __shared__ uint32_t ws[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  uint32_t carry = 0;
  for (int base = 0; base < n; base += 1024) {
    const uint32_t v = base + t < n ? count[base + t] : 0;
    uint32_t inc = v;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = __shfl_up(inc, d, 64);
      if (lane >= d) inc += o;
    }
    if (lane == 63) ws[wave] = inc;
    __syncthreads();
    uint32_t before = carry, all = carry;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before += ws[w];
      all += ws[w];
    }
    if (base + t < n) count[base + t] = before + inc - v;
    carry = all;
    __syncthreads();
  }
  if (t == 0) *total = carry;
}

struct Seqs {  // sequence starts (in the concatenated buffer) and indices of one genome
  const int64_t* off;
  const int64_t* index;
  int n;
};

// The reference's position of buffer position p: 1-based plus index * 10^10; 0 for an unfilled slot.
__device__ inline int64_t position_of(const Seqs& s, int64_t p) {
  int lo = 0, hi = s.n - 1;  // the last sequence starting at or before p
  if (p < s.off[0]) return 0;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s.off[mid] <= p) lo = mid; else hi = mid - 1;
  }
  return p - s.off[lo] + 1 + s.index[lo] * kStride;
}

// The joined positions in query order out of the dense array; WRITE false counts them.
template <bool WRITE>
__global__ __launch_bounds__(256) void k_joined(const uint32_t* dense, uint32_t len_q, uint32_t* count, Seqs qs,
                                                Seqs ts, uint64_t* q, int64_t* t, uint8_t* rev, const Ctl* ctl) {
  const uint32_t p0 = blockIdx.x * (uint32_t)kDense + 16u * threadIdx.x;
  const uint32_t dq = ctl->drop[0], dt = ctl->drop[1];
  uint32_t v[16];
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint4 x = p0 + 4 * k < len_q ? *(const uint4*)(dense + p0 + 4 * k) : uint4{0, 0, 0, 0};
    v[4 * k] = x.x;
    v[4 * k + 1] = x.y;
    v[4 * k + 2] = x.z;
    v[4 * k + 3] = x.w;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (p0 + i >= len_q || p0 + i == dq || (v[i] & ~kNeg) - 1 + len_q == dt) v[i] = 0;
    n += v[i] != 0;
  }
  uint32_t all;
  uint32_t at = group_scan(n, &all);
  if (!WRITE) {
    if (threadIdx.x == 0) count[blockIdx.x] = all;
    return;
  }
  at += count[blockIdx.x];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (v[i]) {
      q[at] = (uint64_t)position_of(qs, (int64_t)p0 + i);
      t[at] = position_of(ts, (int64_t)(v[i] & ~kNeg) - 1 + len_q);
      rev[at] = v[i] & kNeg ? 1 : 0;
      ++at;
    }
}

// Links every joined position to the one it extends (the first joined position is skipped, as
// the reference starts at the second), and reduces the links within a tile of kTile entries to
// their first entry: up[i] is i for a block's first entry, else an earlier entry of its block.
__global__ __launch_bounds__(kTile) void k_link(const uint64_t* q, const int64_t* t, const uint8_t* rev, uint32_t n,
                                                int64_t jump, uint32_t* up, uint8_t* extended) {
  __shared__ uint32_t root[kTile];
  const uint32_t i0 = blockIdx.x * (uint32_t)kTile, i = i0 + threadIdx.x;
  uint32_t pred = i;
  if (i > 1 && i < n) {
    const int64_t qi = (int64_t)q[i], ti = t[i];
    const uint8_t ri = rev[i];
    for (uint32_t j = i - 1; j >= 1; --j) {
      const int64_t gap = qi - (int64_t)q[j];
      if (gap > jump) break;
      if (rev[j] == ri && (ri ? t[j] - ti : ti - t[j]) == gap) {
        pred = j;
        extended[j] = 1;
        break;
      }
    }
  }
  // within the tile: double the links until they rest on an entry whose link leaves the tile
  uint32_t r = pred >= i0 ? pred : i;
  root[threadIdx.x] = r;
  __syncthreads();
  for (int d = 0; d < 11; ++d) {
    const uint32_t nr = root[r - i0];
    const int moved = nr != r;
    r = nr;
    if (!__syncthreads_or(moved)) break;
    root[threadIdx.x] = r;
    __syncthreads();
  }
  if (i < n) up[i] = r != i ? r : pred;
}

// The blocks' last entries, in order: first[i] is the block's first entry if entry i ends a block
// of at least min_length bases, else kNone.
__global__ __launch_bounds__(256) void k_ends(const uint64_t* q, const uint32_t* up, const uint8_t* extended,
                                              uint32_t n, int K, int min_length, uint32_t* first, uint32_t* count) {
  uint32_t m = 0;
  for (int k = 0; k < kTile / 256; ++k) {
    const uint32_t i = blockIdx.x * (uint32_t)kTile + (uint32_t)(kTile / 256) * threadIdx.x + k;
    if (i >= n) break;
    uint32_t f = kNone;
    if (i >= 1 && !extended[i]) {
      uint32_t x = i;
      while (up[x] != x) x = up[x];
      if ((int64_t)(q[i] - q[x]) + K >= min_length) {
        f = x;
        ++m;
      }
    }
    first[i] = f;
  }
  uint32_t all;
  group_scan(m, &all);
  if (threadIdx.x == 0) count[blockIdx.x] = all;
}

// {first entry, last entry, the step that closes it} of every block, by last entry.
__global__ __launch_bounds__(256) void k_blocks(const uint64_t* q, const uint32_t* first, uint32_t n, int64_t jump,
                                                const uint32_t* count, uint32_t* bf, uint32_t* bl, uint32_t* bc) {
  uint32_t f[kTile / 256];
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < kTile / 256; ++k) {
    const uint32_t i = blockIdx.x * (uint32_t)kTile + (uint32_t)(kTile / 256) * threadIdx.x + k;
    f[k] = i < n ? first[i] : kNone;
    m += f[k] != kNone;
  }
  uint32_t all;
  uint32_t at = count[blockIdx.x] + group_scan(m, &all);
#pragma unroll
  for (int k = 0; k < kTile / 256; ++k) {
    if (f[k] == kNone) continue;
    const uint32_t i = blockIdx.x * (uint32_t)kTile + (uint32_t)(kTile / 256) * threadIdx.x + k;
    uint32_t c = i + 1;
    while (c < n && (int64_t)(q[c] - q[i]) <= jump) ++c;
    bf[at] = f[k];
    bl[at] = i;
    bc[at] = c;
    ++at;
  }
}

// Every block's t_result at its place in the reference's order: by closing step, then by first entry.
__global__ __launch_bounds__(256) void k_records(const uint32_t* bf, const uint32_t* bl, const uint32_t* bc, uint32_t n,
                                                 const uint64_t* q, const int64_t* t, const uint8_t* rev, int K,
                                                 const uint64_t* lengths, int nlengths, sxc_result* out) {
  const uint32_t k = blockIdx.x * 256u + threadIdx.x;
  if (k >= n) return;
  const uint32_t f = bf[k], c = bc[k];
  uint32_t lo = k, rank = 0;
  while (lo > 0 && bc[lo - 1] == c) rank += bf[--lo] < f;
  for (uint32_t j = k + 1; j < n && bc[j] == c; ++j) rank += bf[j] < f;
  const int64_t qs = (int64_t)q[f], tt = t[f], length = (int64_t)(q[bl[k]] - q[f]);
  const bool r = rev[f] != 0;
  sxc_result x;
  x.query_id = (uint64_t)(qs / kStride - 1);
  x.target_id = (uint64_t)(tt / kStride - 1);
  // query_seqs[query_id] (a record skipped as empty shifts this lookup, as there)
  x.query_size = x.query_id < (uint64_t)nlengths ? lengths[x.query_id] : 0;
  x.qstart = (uint64_t)(qs % kStride - 1);
  x.tstart = r ? (uint64_t)((tt - length) % kStride - 1) : (uint64_t)(tt % kStride - 1);
  x.len = (uint64_t)(length + K);
  x.reverse = r ? 1 : 0;
  for (int z = 0; z < 7; ++z) x.pad_[z] = 0;
  x.prob = 1;
  x.ident = 1;
  out[lo + rank] = x;
}

}  // namespace km
}  // namespace sxc
