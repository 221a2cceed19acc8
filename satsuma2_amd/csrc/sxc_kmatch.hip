// sxc_kmatch.hip -- KMatch (kmatch/KMatch.cc) on the GPU (include/sxc_kmatch.h).  With max_freq = 1
// the path of sxc_kmatch_unique.h runs; this file holds its host side and the general path, whose
// k-mer tables are built, sorted, filtered and joined on the GPU and chained on the host.
//
// Per genome (KMatch::kmer_array_from_fasta, KMatch.cc:21-132): every position whose K
// bases are all A/C/G/T (either case) gives its canonical k-mer -- the smaller of the
// forward 2-bit code and the reverse complement's -- with its 1-based start plus the
// sequence index times 10^10, negated when the reverse complement was the smaller.  The
// table has len + 1 - K slots per sequence; slots no k-mer fills stay {0, 0} and are sorted
// and counted with the rest.  The table is sorted by k-mer, k-mers occurring more than
// max_freq times are dropped, and the last surviving entry is dropped as well
// (kposv.resize(wi - 1), :124-129).  Joining (merge_positions, :141-177) pairs each query
// entry with the target entries of its k-mer, orientation = query sign xor target sign.
//
// Device layout: both genomes' sequences in one byte buffer per genome, each sequence
// preceded by one 'N' so no k-mer window spans two sequences; 64 positions per thread, the
// window kept rolling in registers (two passes: count per thread, exclusive scan, write in
// position order).  Sorting and scans are rocPRIM's device radix sort and scan; the
// frequency filter tests, for each entry, the max_freq + 1 windows of the sorted table that
// contain it (a group is longer than max_freq iff one such window has equal ends), so it
// reads O(max_freq) neighbours instead of the group.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <chrono>
#include <deque>
#include <fstream>
#include <memory>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <string>
#include <vector>

#include "../../include/sxc_kmatch.h"
#include "sxc_api_internal.h"
#include "sxc_kmatch_unique.h"

using sxc::fail;

namespace {

constexpr int64_t kRecordStride = 10000000000LL;  // KMATCH_POSITION_CHR_CNST (KMatch.h:18)
constexpr int kSpan = 16;                          // positions per lane
constexpr int kChunk = 64 * kSpan;                 // positions per chunk (one wave)
constexpr int kBlock = 256;

// One genome's sequences as the table builder walks them: in device memory they follow each
// other, each preceded by one 'N'.
struct Side {
  std::deque<std::string> owned;   // sequences read from a file
  std::vector<const char*> seq;    // each sequence's bytes (owned, or the caller's)
  int64_t len = 0;                 // bytes of the device buffer
  std::vector<int64_t> off;        // start of each sequence in it
  std::vector<int64_t> index;      // its sequence index (headers seen when it was processed)
  std::vector<uint64_t> lengths;   // seqnames[].length, in processing order
  int64_t slots = 0;               // table size: sum of len + 1 - K
};

int add_sequence(Side* s, const char* p, int64_t len, int64_t index, int K, const std::string& what) {
  if (len == 0) return SXC_OK;  // an empty record is not processed (KMatch.cc:50)
  if (len + 1 < K)
    return fail(SXC_ERR_ARG, what + ": a record of " + std::to_string(len) + " bases is shorter than K - 1");
  s->slots += len + 1 - K;
  s->lengths.push_back((uint64_t)len);
  s->off.push_back(s->len + 1);
  s->len += 1 + len;
  s->seq.push_back(p);
  s->index.push_back(index);
  return SXC_OK;
}

// kmer_array_from_fasta's reading (KMatch.cc:32-103): std::getline lines, '>' starts a
// record, and at end of file the pending sequence is processed before the last line read
// is appended, so a final line without a newline is not part of it.
int read_side(const char* path, int K, Side* s) {
  std::ifstream f(path);
  if (!f.is_open()) return fail(SXC_ERR_ARG, std::string("cannot open ") + path);
  std::string line, seq;
  int64_t index = 0;
  for (;;) {
    std::getline(f, line);
    if ((!line.empty() && line[0] == '>') || f.eof()) {
      s->owned.push_back(std::move(seq));
      const int rc = add_sequence(s, s->owned.back().data(), (int64_t)s->owned.back().size(), index, K, path);
      if (rc != SXC_OK) return rc;
      if (f.eof()) break;
      seq = std::string();
      ++index;
    } else {
      if (f.fail()) return fail(SXC_ERR_ARG, std::string("read error in ") + path);
      seq += line;
    }
  }
  return SXC_OK;
}

__device__ inline int base2(unsigned char c) {
  switch (c) {
    case 'A': case 'a': return 0;
    case 'C': case 'c': return 1;
    case 'G': case 'g': return 2;
    case 'T': case 't': return 3;
    default: return -1;
  }
}

// Canonical k-mers of chunk c, positions [1024 c, 1024 c + 1024): one wave per chunk, each lane
// rolling its window over 16 positions.  Pass 0 counts a chunk's k-mers; pass 1 puts each
// lane's k-mers into its 16 LDS slots and the wave then copies the chunk's k-mers, in position
// order, to base[c] on as one contiguous run.  off/index: sequence starts and indices (binary
// search).
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void k_kmers(const unsigned char* buf, int64_t n, int K, int64_t chunks,
                                                  uint64_t* count, const uint64_t* base, const int64_t* off,
                                                  const int64_t* index, int nseq, uint64_t* keys, int64_t* vals) {
  constexpr int kWaves = kBlock / 64;
  static_assert(kBlock % 64 == 0, "");
  __shared__ uint64_t skey[WRITE ? kWaves * kChunk : 1];
  __shared__ int64_t sval[WRITE ? kWaves * kChunk : 1];
  __shared__ int pre[kWaves][65];
  const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64;
  const int64_t c = (int64_t)blockIdx.x * kWaves + wave;
  const bool active = c < chunks;  // every wave reaches the barriers
  int got = 0;
  if (active) {
    const int64_t start = c * kChunk + (int64_t)lane * kSpan;
    const int64_t end = start + kSpan < n ? start + kSpan : n;
    const uint64_t mask = (1ull << (2 * K)) - 1;
    const int top = 2 * (K - 1);
    const int64_t s0 = start - (K - 1) > 0 ? start - (K - 1) : 0;
    int64_t last_unknown = s0 - 1;
    uint64_t f = 0, r = 0;
    for (int64_t p = s0; p < end; ++p) {
      const int b = base2(buf[p]);
      const uint64_t code = b < 0 ? 0 : (uint64_t)b;  // any other letter acts as A and breaks the window
      f = ((f << 2) + code) & mask;
      r = (r >> 2) + ((3 - code) << top);
      if (b < 0) last_unknown = p;
      if (p >= start && last_unknown + K <= p) {
        if (WRITE) {
          int lo = 0, hi = nseq - 1;  // the last sequence starting at or before p
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (off[mid] <= p) lo = mid; else hi = mid - 1;
          }
          const int64_t pos = (p - off[lo]) - K + 2 + index[lo] * kRecordStride;  // 1-based start
          const int slot = wave * kChunk + lane * kSpan + got;
          skey[slot] = f <= r ? f : r;
          sval[slot] = f <= r ? pos : -pos;
        }
        ++got;
      }
    }
  }
  pre[wave][lane + 1] = got;
  __syncthreads();
  if (lane == 0) {
    pre[wave][0] = 0;
    for (int l = 1; l <= 64; ++l) pre[wave][l] += pre[wave][l - 1];
    if (!WRITE && active) count[c] = (uint64_t)pre[wave][64];
  }
  __syncthreads();
  if (!WRITE || !active) return;
  const int total = pre[wave][64];
  const uint64_t at = base[c];
  for (int i = lane; i < total; i += 64) {
    int lo = 0, hi = 63;  // the lane whose k-mers hold entry i: pre[lo] <= i < pre[lo + 1]
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (pre[wave][mid] <= i) lo = mid; else hi = mid - 1;
    }
    const int slot = wave * kChunk + lo * kSpan + (i - pre[wave][lo]);
    keys[at + (uint64_t)i] = skey[slot];
    vals[at + (uint64_t)i] = sval[slot];
  }
}

// keep[i] = 1 unless entry i lies in a run of more than F equal k-mers.
__global__ __launch_bounds__(kBlock) void k_keep(const uint64_t* keys, int64_t n, int F, uint64_t* keep) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  bool drop = false;
  for (int64_t j = i - F > 0 ? i - F : 0; j <= i && j + F < n; ++j)
    if (keys[j] == keys[j + F]) {
      drop = true;
      break;
    }
  keep[i] = drop ? 0 : 1;
}

__global__ __launch_bounds__(kBlock) void k_scatter(const uint64_t* keys, const int64_t* vals, const uint64_t* keep,
                                                    const uint64_t* at, int64_t n, uint64_t* okeys, int64_t* ovals) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n || !keep[i]) return;
  okeys[at[i]] = keys[i];
  ovals[at[i]] = vals[i];
}

__device__ inline int64_t lower_bound(const uint64_t* a, int64_t n, uint64_t v) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (a[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Join: per query entry, the target entries of its k-mer (pass 0 counts, pass 1 writes
// {|query position|, |target position|, orientation} in query-table order).
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void k_join(const uint64_t* qk, const int64_t* qv, int64_t nq,
                                                 const uint64_t* tk, const int64_t* tv, int64_t nt, uint64_t* count,
                                                 const uint64_t* base, uint64_t* jq, int64_t* jt, uint8_t* jrev) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= nq) return;
  const uint64_t k = qk[i];
  const int64_t lb = lower_bound(tk, nt, k);
  if (!WRITE) {
    int64_t c = 0;
    while (lb + c < nt && tk[lb + c] == k) ++c;
    count[i] = (uint64_t)c;
    return;
  }
  uint64_t at = base[i];
  const int64_t q = qv[i];
  for (int64_t j = lb; j < nt && tk[j] == k; ++j, ++at) {
    // the reference tests position > 0: a {0, 0} slot counts as reverse
    bool rev = !(q > 0);
    const int64_t t = tv[j];
    if (!(t > 0)) rev = !rev;
    jq[at] = (uint64_t)(q > 0 ? q : -q);
    jt[at] = t > 0 ? t : -t;
    jrev[at] = rev ? 1 : 0;
  }
}

__global__ __launch_bounds__(kBlock) void k_iota(uint64_t* v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) v[i] = (uint64_t)i;
}

// The sweep's inputs in query order: the target position and strand of each sorted entry
// (order is a permutation of 0 .. n - 1).
__global__ __launch_bounds__(kBlock) void k_gather(const uint64_t* order, const int64_t* t, const uint8_t* r,
                                                   int64_t* t_out, uint8_t* r_out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    const uint64_t j = order[i];
    t_out[i] = t[j];
    r_out[i] = r[j];
  }
}

inline unsigned grid_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// Device buffers of one run, freed on return.
struct Buffers {
  std::vector<void*> ptrs;
  ~Buffers() {
    for (void* p : ptrs) (void)hipFree(p);
  }
  template <class T>
  hipError_t get(T** p, int64_t n) {
    void* q = nullptr;
    const hipError_t e = hipMalloc(&q, (size_t)(n > 0 ? n : 1) * sizeof(T));
    if (e == hipSuccess) ptrs.push_back(q);
    *p = (T*)q;
    return e;
  }
};

#define KCHK(expr)                                                                                          \
  do {                                                                                                      \
    hipError_t e_ = (expr);                                                                                 \
    if (e_ != hipSuccess) return fail(SXC_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));      \
  } while (0)

// Pairs sorted by key bits [0, end).  Asked once for bits [63, 64) of 100 such keys, the library's sort
// had not returned after 60 s; the cause is not known, so no call goes to it with an end of 64.
template <class V>
hipError_t sort_pairs(void* tmp, size_t& bytes, uint64_t* k0, uint64_t* k1, V* v0, V* v1, size_t n, int end, hipStream_t s) {
  if (end < 1 || end > 63) return hipErrorInvalidValue;
  return rocprim::radix_sort_pairs(tmp, bytes, k0, k1, v0, v1, n, 0, end, s);
}

// A genome's buffer into device memory at d.  Long sequences are copied from where they lie,
// runs of short ones, each with the 'N' before it, through `stage` (which has to live until the stream is
// synchronised).
int upload(const Side& side, unsigned char* d, std::vector<std::string>& stage, hipStream_t s) {
  constexpr int64_t kLong = 65536, kStage = 1 << 22;
  bool any_long = false;
  for (uint64_t n : side.lengths) any_long |= (int64_t)n >= kLong;
  if (any_long) KCHK(hipMemsetAsync(d, 'N', (size_t)side.len, s));
  for (size_t k = 0; k < side.seq.size();) {
    const int64_t n = (int64_t)side.lengths[k];
    if (n >= kLong) {
      KCHK(hipMemcpyAsync(d + side.off[k], side.seq[k], (size_t)n, hipMemcpyHostToDevice, s));
      ++k;
      continue;
    }
    const int64_t at = side.off[k] - 1;
    size_t e = k;
    while (e < side.seq.size() && (int64_t)side.lengths[e] < kLong && side.off[e] - at < kStage) ++e;
    std::string run((size_t)(side.off[e - 1] + (int64_t)side.lengths[e - 1] - at), 'N');
    for (; k < e; ++k) memcpy(&run[(size_t)(side.off[k] - at)], side.seq[k], (size_t)side.lengths[k]);
    stage.push_back(std::move(run));
    KCHK(hipMemcpyAsync(d + at, stage.back().data(), stage.back().size(), hipMemcpyHostToDevice, s));
  }
  return SXC_OK;
}

// exclusive scan of n uint64 values; returns the total in *total
int scan(Buffers& B, const uint64_t* in, uint64_t* out, int64_t n, uint64_t* total, hipStream_t s) {
  if (n == 0) {
    *total = 0;
    return SXC_OK;
  }
  size_t bytes = 0;
  KCHK(rocprim::exclusive_scan(nullptr, bytes, in, out, (uint64_t)0, (size_t)n, rocprim::plus<uint64_t>(), s));
  void* tmp = nullptr;
  KCHK(B.get((char**)&tmp, (int64_t)bytes));
  KCHK(rocprim::exclusive_scan(tmp, bytes, in, out, (uint64_t)0, (size_t)n, rocprim::plus<uint64_t>(), s));
  uint64_t last_out = 0, last_in = 0;
  KCHK(hipMemcpyAsync(&last_out, out + n - 1, 8, hipMemcpyDeviceToHost, s));
  KCHK(hipMemcpyAsync(&last_in, in + n - 1, 8, hipMemcpyDeviceToHost, s));
  KCHK(hipStreamSynchronize(s));
  *total = last_out + last_in;
  return SXC_OK;
}

// One genome's table: built, sorted by k-mer, filtered; the sorted kept entries are left in
// (*keys, *vals), *n of them.
int build_table(Buffers& B, const Side& side, int K, int F, hipStream_t s, uint64_t** keys, int64_t** vals,
                int64_t* n, int64_t* kept, std::vector<std::string>& stage) {
  const int64_t len = side.len;
  const int64_t slots = side.slots;
  const int nseq = (int)side.off.size();
  *n = 0;
  *kept = 0;
  if (slots == 0) return SXC_OK;
  unsigned char* dbuf;
  int64_t *doff, *didx;
  KCHK(B.get(&dbuf, len));
  KCHK(B.get(&doff, nseq));
  KCHK(B.get(&didx, nseq));
  int rc = upload(side, dbuf, stage, s);
  if (rc != SXC_OK) return rc;
  KCHK(hipMemcpyAsync(doff, side.off.data(), sizeof(int64_t) * nseq, hipMemcpyHostToDevice, s));
  KCHK(hipMemcpyAsync(didx, side.index.data(), sizeof(int64_t) * nseq, hipMemcpyHostToDevice, s));
  const int64_t chunks = (len + kChunk - 1) / kChunk;
  uint64_t *cnt, *base;
  KCHK(B.get(&cnt, chunks));
  KCHK(B.get(&base, chunks));
  hipLaunchKernelGGL(k_kmers<false>, dim3(grid_of(chunks * 64)), dim3(kBlock), 0, s, dbuf, len, K, chunks, cnt,
                     nullptr, doff, didx, nseq, nullptr, nullptr);
  KCHK(hipGetLastError());
  uint64_t filled = 0;
  rc = scan(B, cnt, base, chunks, &filled, s);
  if (rc != SXC_OK) return rc;
  if ((int64_t)filled > slots) return fail(SXC_ERR_ARG, "k-mer table overflow");  // cannot happen: one per slot
  uint64_t *k0, *k1;
  int64_t *v0, *v1;
  KCHK(B.get(&k0, slots));
  KCHK(B.get(&v0, slots));
  KCHK(B.get(&k1, slots));
  KCHK(B.get(&v1, slots));
  // slots no k-mer fills stay {0, 0}
  KCHK(hipMemsetAsync(k0, 0, sizeof(uint64_t) * slots, s));
  KCHK(hipMemsetAsync(v0, 0, sizeof(int64_t) * slots, s));
  hipLaunchKernelGGL(k_kmers<true>, dim3(grid_of(chunks * 64)), dim3(kBlock), 0, s, dbuf, len, K, chunks, nullptr,
                     base, doff, didx, nseq, k0, v0);
  KCHK(hipGetLastError());
  size_t bytes = 0;
  KCHK(sort_pairs(nullptr, bytes, k0, k1, v0, v1, (size_t)slots, 2 * K, s));
  void* tmp;
  KCHK(B.get((char**)&tmp, (int64_t)bytes));
  KCHK(sort_pairs(tmp, bytes, k0, k1, v0, v1, (size_t)slots, 2 * K, s));
  uint64_t *keep, *at;
  KCHK(B.get(&keep, slots));
  KCHK(B.get(&at, slots));
  hipLaunchKernelGGL(k_keep, dim3(grid_of(slots)), dim3(kBlock), 0, s, k1, slots, F, keep);
  KCHK(hipGetLastError());
  uint64_t nk = 0;
  rc = scan(B, keep, at, slots, &nk, s);
  if (rc != SXC_OK) return rc;
  hipLaunchKernelGGL(k_scatter, dim3(grid_of(slots)), dim3(kBlock), 0, s, k1, v1, keep, at, slots, k0, v0);
  KCHK(hipGetLastError());
  *kept = (int64_t)nk;
  *n = nk > 0 ? (int64_t)nk - 1 : 0;  // kposv.resize(wi - 1)
  *keys = k0;
  *vals = v0;
  return SXC_OK;
}

}  // namespace

struct sxc_kmatch {
  std::vector<sxc_result> out;        // the general path's records
  sxc_result* raw = nullptr;          // or the unique path's, as they came from the device
  int64_t n_raw = 0;
  sxc_kmatch_stats st{};
  const sxc_result* data() const { return raw ? raw : out.data(); }
  int64_t size() const { return raw ? n_raw : (int64_t)out.size(); }
  ~sxc_kmatch() { free(raw); }
};

namespace {

// dump_matching_blocks (KMatch.cc:196-318) over the joined positions sorted by query
// position: a block grows while the next joined position on its diagonal (anti-diagonal
// for reverse) lies within max_jump of its end; blocks are reported when the sweep passes
// their end by more than max_jump, in the order they finish (then creation order), if they
// span at least min_length bases.  The reference starts at the second joined position and
// ends with one read past the table; the first is skipped here too and the last step only
// closes the open blocks.
void sweep(const std::vector<uint64_t>& q, const std::vector<int64_t>& t, const std::vector<uint8_t>& rev,
           const sxc_kmatch_params& p, const Side& qs, const Side& ts, std::vector<sxc_result>* out) {
  struct Block {
    int64_t q_start, t_start;
    bool reverse;
    int64_t length;
  };
  // the open blocks in creation order, kept in a vector (compacted in place each step)
  std::vector<Block> active;
  const uint64_t n = q.size();
  for (uint64_t i = 1; i <= n; ++i) {
    const bool last = i == n;
    bool used = false;
    int64_t qd = 0;
    size_t w = 0;
    for (size_t r = 0; r < active.size(); ++r) {
      Block b = active[r];
      if (!last) {
        qd = (int64_t)q[i] - b.q_start;
        const int64_t td = b.reverse ? b.t_start - t[i] : t[i] - b.t_start;
        if (qd == td && qd - b.length <= p.max_jump && b.reverse == (rev[i] != 0)) {
          b.length = qd;
          used = true;
        }
      }
      if (last || qd - b.length > p.max_jump) {
        if (b.length + p.K >= p.min_length) {
          sxc_result res{};
          res.query_id = (uint64_t)(b.q_start / kRecordStride - 1);
          res.target_id = (uint64_t)(b.t_start / kRecordStride - 1);
          // query_seqs[query_id] (a record skipped as empty shifts this lookup, as there)
          res.query_size = res.query_id < qs.lengths.size() ? qs.lengths[res.query_id] : 0;
          res.qstart = (uint64_t)(b.q_start % kRecordStride - 1);
          res.tstart = b.reverse ? (uint64_t)((b.t_start - b.length) % kRecordStride - 1)
                                 : (uint64_t)(b.t_start % kRecordStride - 1);
          res.len = (uint64_t)(b.length + p.K);
          res.reverse = b.reverse ? 1 : 0;
          res.prob = 1;
          res.ident = 1;
          out->push_back(res);
        }
      } else {
        active[w++] = b;
      }
    }
    active.resize(w);
    if (!used && !last) active.push_back(Block{(int64_t)q[i], t[i], rev[i] != 0, 0});
  }
  (void)ts;
}

// Memory for records that come back from the device; large blocks ask for huge pages, whose first
// touch costs a copy into fresh memory far less.  Given back with free().
void* result_memory(size_t bytes) {
  constexpr size_t kHuge = 2u << 20;
  if (bytes < 2 * kHuge) return malloc(bytes);
  const size_t n = (bytes + kHuge - 1) / kHuge * kHuge;
  void* p = aligned_alloc(kHuge, n);
  if (p) (void)madvise(p, n, MADV_HUGEPAGE);
  return p;
}

// Device buffers of the unique path, kept by the context between calls.
enum { KM_BUF, KM_KEYS, KM_KEYS2, KM_VALS, KM_VALS2, KM_TMP, KM_START, KM_DENSE, KM_SEEN, KM_JOINED, KM_LINKS, KM_SEQS,
       KM_OUT };
static_assert(KM_OUT < SXC_KMATCH_BUFS, "");

// What the unique path takes: every k-mer at most once, gaps the neighbour searches can bridge
// (SatsumaSynteny2 asks for K - 1 <= 30; both searches read up to max_jump entries), positions
// in 31 bits.
bool unique_path(const Side& qs, const Side& ts, const sxc_kmatch_params& p) {
  return p.max_freq == 1 && p.max_jump <= 64 && qs.slots > 0 && ts.slots > 0 &&
         qs.len + ts.len < (1ll << 31) - 65536;
}

// KMatch for max_freq = 1 on the device (sxc_kmatch_unique.h).  *done is false if a bucket held
// more k-mers than its table takes; the general path then runs.
int run_unique(sxc_ctx* ctx, const Side& qs, const Side& ts, const sxc_kmatch_params& p, sxc_kmatch* res, bool* done) {
  using namespace sxc::km;
  hipStream_t s = ctx->stream;
  DevBuf* W = ctx->km;
  std::vector<std::string> stage;
  *done = false;
  const int64_t len = qs.len + ts.len, slots = qs.slots + ts.slots;
  const int nq = (int)qs.off.size(), nt = (int)ts.off.size();
  // buckets of 200 .. 400 entries: half full tables
  int bits = 1;
  while (bits < 24 && (slots >> bits) > 400) ++bits;
  const uint32_t buckets = 1u << bits;
  const size_t heavy_max = (size_t)(slots / kHeavy) + 1;
  constexpr int kHeavyGroups = 1024, kLook = 64, kWaves = kBucketGroups + kLook;
  // sequence starts (in the joint buffer) and indices of both genomes, then the query's lengths
  std::vector<int64_t> seqs;
  seqs.insert(seqs.end(), qs.off.begin(), qs.off.end());
  seqs.insert(seqs.end(), qs.index.begin(), qs.index.end());
  for (int64_t o : ts.off) seqs.push_back(o + qs.len);
  seqs.insert(seqs.end(), ts.index.begin(), ts.index.end());
  for (uint64_t l : qs.lengths) seqs.push_back((int64_t)l);
  KCHK(W[KM_BUF].ensure((size_t)((len + 15) / 16 * 16)));
  KCHK(W[KM_SEQS].ensure(seqs.size() * sizeof(int64_t)));
  KCHK(W[KM_KEYS].ensure((size_t)slots * sizeof(uint64_t)));
  KCHK(W[KM_KEYS2].ensure((size_t)slots * sizeof(uint64_t)));
  KCHK(W[KM_VALS].ensure((size_t)slots * sizeof(uint32_t)));
  KCHK(W[KM_VALS2].ensure((size_t)slots * sizeof(uint32_t)));
  KCHK(W[KM_DENSE].ensure((size_t)(qs.len + 16) * sizeof(uint32_t)));
  // bucket starts, heavy list
  KCHK(W[KM_START].ensure(((size_t)buckets + 1 + heavy_max) * sizeof(uint32_t)));
  const uint32_t dense_groups = (uint32_t)((qs.len + kDense - 1) / kDense);
  // control words, per-wave results, group counts; the heavy tables behind them
  const size_t seen_bytes = 256 + (size_t)kWaves * 2 * (sizeof(uint64_t) + sizeof(uint32_t)) +
                            (((size_t)dense_groups * sizeof(uint32_t) + 255) & ~(size_t)255);
  KCHK(W[KM_SEEN].ensure(seen_bytes + heavy_max * kTable * (sizeof(uint64_t) + 2 * sizeof(uint32_t))));
  unsigned char* dbuf = W[KM_BUF].as<unsigned char>();
  uint64_t *k0 = W[KM_KEYS].as<uint64_t>(), *k1 = W[KM_KEYS2].as<uint64_t>();
  uint32_t *v0 = W[KM_VALS].as<uint32_t>(), *v1 = W[KM_VALS2].as<uint32_t>();
  uint32_t* dense = W[KM_DENSE].as<uint32_t>();
  uint32_t *start = W[KM_START].as<uint32_t>(), *list = start + buckets + 1;
  char* seen = W[KM_SEEN].as<char>();
  Ctl* ctl = (Ctl*)seen;
  static_assert(sizeof(Ctl) <= 256, "");
  uint64_t* best = (uint64_t*)(seen + 256);
  uint32_t* at = (uint32_t*)(best + 2 * kWaves);
  uint32_t* groups = at + 2 * kWaves;
  uint64_t* gkey = (uint64_t*)(seen + seen_bytes);
  uint32_t* gpos = (uint32_t*)(gkey + heavy_max * kTable);
  const int64_t* dseq = W[KM_SEQS].as<int64_t>();
  const Seqs dq{dseq, dseq + nq, nq}, dt{dseq + 2 * nq, dseq + 2 * nq + nt, nt};
  const uint64_t* dlen = (const uint64_t*)(dseq + 2 * nq + 2 * nt);
  const uint32_t len_q = (uint32_t)qs.len;
  Ctl host{};

  KCHK(hipMemsetAsync(ctl, 0, sizeof(Ctl), s));
  int rc = upload(qs, dbuf, stage, s);
  if (rc == SXC_OK) rc = upload(ts, dbuf + qs.len, stage, s);
  if (rc != SXC_OK) return rc;
  KCHK(hipMemcpyAsync(W[KM_SEQS].p, seqs.data(), seqs.size() * sizeof(int64_t), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_unique_kmers, dim3((unsigned)((len + 4095) / 4096)), dim3(256), 0, s, dbuf, len, qs.len, p.K, k0,
                     v0, ctl);
  hipLaunchKernelGGL(k_unique_unfilled, dim3(1), dim3(1), 0, s, k0, v0, qs.slots, ts.slots, len_q, ctl);
  KCHK(hipGetLastError());
  KCHK(hipMemcpyAsync(&host, ctl, sizeof host, hipMemcpyDeviceToHost, s));
  KCHK(hipStreamSynchronize(s));
  const uint32_t n = (uint32_t)host.n;
  if ((int64_t)host.n > slots) return fail(SXC_ERR_ARG, "k-mer table overflow");  // cannot happen: one per slot
  if (n > 0) {
    size_t bytes = 0;
    KCHK(sort_pairs(nullptr, bytes, k0, k1, v0, v1, (size_t)n, bits, s));
    KCHK(W[KM_TMP].ensure(bytes));
    KCHK(sort_pairs(W[KM_TMP].p, bytes, k0, k1, v0, v1, (size_t)n, bits, s));
    KCHK(hipMemsetAsync(dense, 0, (size_t)(qs.len + 16) * sizeof(uint32_t), s));
    hipLaunchKernelGGL(k_bounds, dim3(n / 256 + 1), dim3(256), 0, s, k1, n, buckets, start);
    hipLaunchKernelGGL(k_heavy_list, dim3((buckets + 255) / 256), dim3(256), 0, s, start, buckets, list, ctl);
    hipLaunchKernelGGL(k_buckets, dim3(kBucketGroups), dim3(64), 0, s, k1, v1, start, buckets, len_q, dense, best, at, ctl);
    // (these exit at once where no bucket is heavy)
    hipLaunchKernelGGL(k_heavy_clear, dim3(kLook), dim3(256), 0, s, ctl, gkey, gpos);
    hipLaunchKernelGGL(k_heavy_count, dim3(kHeavyGroups), dim3(256), 0, s, k1, v1, start, list, len_q, gkey, gpos, ctl);
    hipLaunchKernelGGL(k_heavy_look, dim3(kLook), dim3(64), 0, s, len_q, gkey, gpos, dense, best + 2 * kBucketGroups,
                       at + 2 * kBucketGroups, ctl);
    hipLaunchKernelGGL(k_last, dim3(1), dim3(64), 0, s, best, at, kWaves, ctl);
    hipLaunchKernelGGL(k_joined<false>, dim3(dense_groups), dim3(256), 0, s, dense, len_q, groups, dq, dt, nullptr,
                       nullptr, nullptr, ctl);
    hipLaunchKernelGGL(k_scan_groups, dim3(1), dim3(1024), 0, s, groups, (int)dense_groups, &ctl->joined);
    KCHK(hipGetLastError());
    KCHK(hipMemcpyAsync(&host, ctl, sizeof host, hipMemcpyDeviceToHost, s));
    KCHK(hipStreamSynchronize(s));
    if (host.overflow) return SXC_OK;
  }
  const uint32_t nj = (uint32_t)host.joined;
  uint32_t nb = 0;
  if (nj > 0) {
    const uint32_t tiles = (nj + kTile - 1) / kTile;
    const size_t m = ((size_t)nj + 15) / 16 * 16;
    KCHK(W[KM_JOINED].ensure(m * (sizeof(uint64_t) + sizeof(int64_t) + 1)));
    KCHK(W[KM_LINKS].ensure(m * (5 * sizeof(uint32_t) + 1) + (size_t)tiles * sizeof(uint32_t)));
    uint64_t* jq = W[KM_JOINED].as<uint64_t>();
    int64_t* jt = (int64_t*)(jq + m);
    uint8_t* jr = (uint8_t*)(jt + m);
    uint32_t *up = W[KM_LINKS].as<uint32_t>(), *first = up + m, *bf = first + m, *bl = bf + m, *bc = bl + m;
    uint32_t* tile_count = bc + m;
    uint8_t* extended = (uint8_t*)(tile_count + tiles);
    KCHK(hipMemsetAsync(extended, 0, nj, s));
    hipLaunchKernelGGL(k_joined<true>, dim3(dense_groups), dim3(256), 0, s, dense, len_q, groups, dq, dt, jq, jt, jr,
                       ctl);
    hipLaunchKernelGGL(k_link, dim3(tiles), dim3(kTile), 0, s, jq, jt, jr, nj, (int64_t)p.max_jump, up, extended);
    hipLaunchKernelGGL(k_ends, dim3(tiles), dim3(256), 0, s, jq, up, extended, nj, p.K, p.min_length, first, tile_count);
    hipLaunchKernelGGL(k_scan_groups, dim3(1), dim3(1024), 0, s, tile_count, (int)tiles, &ctl->blocks);
    hipLaunchKernelGGL(k_blocks, dim3(tiles), dim3(256), 0, s, jq, first, nj, (int64_t)p.max_jump, tile_count, bf, bl, bc);
    KCHK(hipGetLastError());
    KCHK(hipMemcpyAsync(&host, ctl, sizeof host, hipMemcpyDeviceToHost, s));
    KCHK(hipStreamSynchronize(s));
    nb = (uint32_t)host.blocks;
    if (nb > 0) {
      KCHK(W[KM_OUT].ensure((size_t)nb * sizeof(sxc_result)));
      const size_t bytes = (size_t)nb * sizeof(sxc_result);
      res->raw = (sxc_result*)result_memory(bytes);
      if (!res->raw) return fail(SXC_ERR_NOMEM, "sxc_kmatch: out of memory");
      hipLaunchKernelGGL(k_records, dim3((nb + 255) / 256), dim3(256), 0, s, bf, bl, bc, nb, jq, jt, jr, p.K, dlen,
                         (int)qs.lengths.size(), W[KM_OUT].as<sxc_result>());
      KCHK(hipGetLastError());
      KCHK(hipMemcpyAsync(res->raw, W[KM_OUT].p, (size_t)nb * sizeof(sxc_result), hipMemcpyDeviceToHost, s));
      KCHK(hipStreamSynchronize(s));
    }
  }
  res->n_raw = nb;
  res->st.query_kept = (int64_t)host.kept[0];
  res->st.target_kept = (int64_t)host.kept[1];
  res->st.joined = nj;
  *done = true;
  return SXC_OK;
}

int run_general(sxc_ctx* ctx, const Side& qs, const Side& ts, const sxc_kmatch_params& p, sxc_kmatch* res);

int run(sxc_ctx* ctx, const Side& qs, const Side& ts, const sxc_kmatch_params& p, double read_ms, sxc_kmatch** out) {
  std::lock_guard<std::mutex> lock(ctx->mu);
  KCHK(hipSetDevice(ctx->device));
  sxc_kmatch* res = new (std::nothrow) sxc_kmatch;
  if (!res) return fail(SXC_ERR_NOMEM, "sxc_kmatch: out of memory");
  std::unique_ptr<sxc_kmatch> hold(res);
  res->st.read_ms = read_ms;
  res->st.query_kmers = qs.slots;
  res->st.target_kmers = ts.slots;
  bool done = false;
  if (unique_path(qs, ts, p)) {
    const auto t0 = std::chrono::steady_clock::now();
    const int rc = run_unique(ctx, qs, ts, p, res, &done);
    res->st.device_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    // the buffers stay for the next call while they are small beside the device's memory
    size_t held = 0;
    for (const DevBuf& b : ctx->km) held += b.cap;
    if (held > ((size_t)1 << 30) || rc != SXC_OK)
      for (DevBuf& b : ctx->km) b.release();
    if (rc != SXC_OK) return rc;
  }
  if (!done) {
    const int rc = run_general(ctx, qs, ts, p, res);
    if (rc != SXC_OK) return rc;
  }
  res->st.blocks = res->size();
  *out = hold.release();
  return SXC_OK;
}

// Any max_freq and max_jump: tables sorted, filtered and joined on the device, chained on the host.
int run_general(sxc_ctx* ctx, const Side& qs, const Side& ts, const sxc_kmatch_params& p, sxc_kmatch* res) {
  hipStream_t s = ctx->stream;
  std::vector<std::string> stage;
  hipEvent_t e0, e1;
  KCHK(hipEventCreate(&e0));
  KCHK(hipEventCreate(&e1));
  std::vector<uint64_t> hq;
  std::vector<int64_t> ht;
  std::vector<uint8_t> hr;
  {
    Buffers B;
    KCHK(hipEventRecord(e0, s));
    uint64_t *qk = nullptr, *tk = nullptr;
    int64_t *qv = nullptr, *tv = nullptr, nq = 0, nt = 0;
    int rc = build_table(B, qs, p.K, p.max_freq, s, &qk, &qv, &nq, &res->st.query_kept, stage);
    if (rc != SXC_OK) return rc;
    rc = build_table(B, ts, p.K, p.max_freq, s, &tk, &tv, &nt, &res->st.target_kept, stage);
    if (rc != SXC_OK) return rc;
    uint64_t nj = 0;
    uint64_t* base = nullptr;  // each query entry's first joined slot
    if (nq > 0 && nt > 0) {
      uint64_t* cnt;
      KCHK(B.get(&cnt, nq));
      KCHK(B.get(&base, nq));
      hipLaunchKernelGGL(k_join<false>, dim3(grid_of(nq)), dim3(kBlock), 0, s, qk, qv, nq, tk, tv, nt, cnt, nullptr,
                         nullptr, nullptr, nullptr);
      KCHK(hipGetLastError());
      rc = scan(B, cnt, base, nq, &nj, s);
      if (rc != SXC_OK) return rc;
    }
    res->st.joined = (int64_t)nj;
    if (nj > 0) {
      uint64_t *jq, *jq2, *ix, *ix2;
      int64_t* jt;
      uint8_t* jr;
      KCHK(B.get(&jq, (int64_t)nj));
      KCHK(B.get(&jq2, (int64_t)nj));
      KCHK(B.get(&ix, (int64_t)nj));
      KCHK(B.get(&ix2, (int64_t)nj));
      KCHK(B.get(&jt, (int64_t)nj));
      KCHK(B.get(&jr, (int64_t)nj));
      hipLaunchKernelGGL(k_join<true>, dim3(grid_of(nq)), dim3(kBlock), 0, s, qk, qv, nq, tk, tv, nt, nullptr, base,
                         jq, jt, jr);
      KCHK(hipGetLastError());
      hipLaunchKernelGGL(k_iota, dim3(grid_of((int64_t)nj)), dim3(kBlock), 0, s, ix, (int64_t)nj);
      KCHK(hipGetLastError());
      // by query position; stable, so a query position's target entries keep table order
      int bits = 1;
      const uint64_t maxq = (uint64_t)(qs.index.empty() ? 1 : qs.index.back() + 1) * (uint64_t)kRecordStride;
      while (bits < 64 && (maxq >> bits)) ++bits;
      size_t bytes = 0;
      KCHK(sort_pairs(nullptr, bytes, jq, jq2, ix, ix2, (size_t)nj, bits, s));
      void* tmp;
      KCHK(B.get((char**)&tmp, (int64_t)bytes));
      KCHK(sort_pairs(tmp, bytes, jq, jq2, ix, ix2, (size_t)nj, bits, s));
      int64_t* gt;
      uint8_t* gr;
      KCHK(B.get(&gt, (int64_t)nj));
      KCHK(B.get(&gr, (int64_t)nj));
      hipLaunchKernelGGL(k_gather, dim3(grid_of((int64_t)nj)), dim3(kBlock), 0, s, ix2, jt, jr, gt, gr, (int64_t)nj);
      KCHK(hipGetLastError());
      hq.resize(nj);
      ht.resize(nj);
      hr.resize(nj);
      KCHK(hipMemcpyAsync(hq.data(), jq2, 8 * nj, hipMemcpyDeviceToHost, s));
      KCHK(hipMemcpyAsync(ht.data(), gt, 8 * nj, hipMemcpyDeviceToHost, s));
      KCHK(hipMemcpyAsync(hr.data(), gr, nj, hipMemcpyDeviceToHost, s));
      KCHK(hipStreamSynchronize(s));
    }
    KCHK(hipEventRecord(e1, s));
    KCHK(hipEventSynchronize(e1));
  }
  float ms = 0;
  KCHK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  res->st.device_ms = ms;
  const auto t0 = std::chrono::steady_clock::now();
  sweep(hq, ht, hr, p, qs, ts, &res->out);
  res->st.sweep_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return SXC_OK;
}

int check_params(const sxc_kmatch_params* p) {
  if (!p || p->K < 1 || p->K > 31 || p->K % 2 == 0 || p->max_freq < 0 || p->max_jump < 0)
    return fail(SXC_ERR_ARG, "sxc_kmatch: K must be odd and in 1..31, max_freq and max_jump >= 0");
  return SXC_OK;
}

}  // namespace

extern "C" {

int sxc_kmatch_files(sxc_ctx* ctx, const char* query_fasta, const char* target_fasta, const sxc_kmatch_params* p,
                     sxc_kmatch** out) {
  if (!ctx || !query_fasta || !target_fasta || !out) return fail(SXC_ERR_ARG, "sxc_kmatch_files: null argument");
  int rc = check_params(p);
  if (rc != SXC_OK) return rc;
  const auto t0 = std::chrono::steady_clock::now();
  Side qs, ts;
  rc = read_side(query_fasta, p->K, &qs);
  if (rc != SXC_OK) return rc;
  rc = read_side(target_fasta, p->K, &ts);
  if (rc != SXC_OK) return rc;
  const double read_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return run(ctx, qs, ts, *p, read_ms, out);
}

int sxc_kmatch_records(sxc_ctx* ctx, int32_t n_queries, const char* const* query_seqs, const int64_t* query_lens,
                       int32_t n_targets, const char* const* target_seqs, const int64_t* target_lens,
                       const sxc_kmatch_params* p, sxc_kmatch** out) {
  if (!ctx || !out || n_queries < 0 || n_targets < 0 || (n_queries && (!query_seqs || !query_lens)) ||
      (n_targets && (!target_seqs || !target_lens)))
    return fail(SXC_ERR_ARG, "sxc_kmatch_records: bad arguments");
  int rc = check_params(p);
  if (rc != SXC_OK) return rc;
  Side qs, ts;
  for (int i = 0; i < n_queries && rc == SXC_OK; ++i)
    rc = (!query_seqs[i] || query_lens[i] < 0) ? fail(SXC_ERR_ARG, "sxc_kmatch_records: bad query record")
                                              : add_sequence(&qs, query_seqs[i], query_lens[i], i + 1, p->K, "query");
  for (int i = 0; i < n_targets && rc == SXC_OK; ++i)
    rc = (!target_seqs[i] || target_lens[i] < 0)
             ? fail(SXC_ERR_ARG, "sxc_kmatch_records: bad target record")
             : add_sequence(&ts, target_seqs[i], target_lens[i], i + 1, p->K, "target");
  if (rc != SXC_OK) return rc;
  return run(ctx, qs, ts, *p, 0., out);
}

int sxc_kmatch_results(const sxc_kmatch* k, sxc_result* out, int64_t cap, int64_t* n) {
  if (!k || !n || cap < 0 || (cap && !out)) return fail(SXC_ERR_ARG, "sxc_kmatch_results: bad arguments");
  *n = k->size();
  if (const int64_t m = *n < cap ? *n : cap) memcpy(out, k->data(), (size_t)m * sizeof(sxc_result));
  return *n > cap ? fail(SXC_ERR_CAPACITY, "sxc_kmatch_results: more records than cap") : SXC_OK;
}

int sxc_kmatch_get_stats(const sxc_kmatch* k, sxc_kmatch_stats* st) {
  if (!k || !st) return fail(SXC_ERR_ARG, "sxc_kmatch_get_stats: bad arguments");
  *st = k->st;
  return SXC_OK;
}

void sxc_kmatch_destroy(sxc_kmatch* k) { delete k; }

}  // extern "C"
