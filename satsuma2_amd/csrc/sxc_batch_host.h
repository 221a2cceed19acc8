// sxc_batch_host.h -- packs caller chunk pairs into the flat device layout.
//
// HBM layout of a batch (uploaded once, then read by every kernel):
//   seq      all distinct chunk byte strings back to back (1 byte per base)
//   tchunks  {offset, length, flags} per distinct target chunk; the target spectra
//            buffer holds 4*N floats per entry in the same order
//   qchunks  the same for distinct query chunks
//   pairs    one sxc_pair_dev per chunk pair (indices into the chunk tables + the
//            chunk metadata FilterMatches writes into t_result)
//   ent      window entropies of the chunks with B/D/H/V letters, computed here with the
//            host's log (SXC_ENT_ROW floats per such chunk; sxc_chunk flags bits 8-31)
// Chunks are deduplicated by (pointer, length), so a target shared by many pairs, as in
// the slave's align_target blocks (analysis/HomologyByXCorrSlave.cc:290-299), is
// transformed once.
#pragma once
#include <string.h>

#include <algorithm>
#include <map>
#include <memory>
#include <string>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

#include "../../include/sxc.h"
#include "sxc_tables.h"
#include "sxc_types.h"

namespace sxc {

// Bytes that a resize leaves as they are (every one of them is written afterwards).
template <class T>
struct UnsetAllocator : std::allocator<T> {
  template <class U>
  struct rebind {
    using other = UnsetAllocator<U>;
  };
  template <class U>
  void construct(U* p) {
    ::new ((void*)p) U;
  }
  template <class U, class... A>
  void construct(U* p, A&&... a) {
    ::new ((void*)p) U(std::forward<A>(a)...);
  }
};

struct HostBatch {
  std::vector<unsigned char, UnsetAllocator<unsigned char>> seq;
  std::vector<sxc_chunk> tchunks, qchunks;
  std::vector<sxc_pair_dev> pairs;
  std::vector<float> ent;
  int max_len = 0;
  // signal tails (sxc_batch_create_tails): source sequences, their strands, the tail and
  // segment tables, and the tail of each target chunk (-1: none)
  std::vector<sxc_chunk> schunks;
  std::vector<int32_t> sstrand;
  std::vector<sxc_tail_dev> tails;
  std::vector<sxc_tail_seg_dev> segs;
  std::vector<int32_t> ttail;
  // Empties the tables; their memory stays for the next batch.
  void reset() {
    seq.clear();
    tchunks.clear();
    qchunks.clear();
    pairs.clear();
    ent.clear();
    max_len = 0;
    schunks.clear();
    sstrand.clear();
    tails.clear();
    segs.clear();
    ttail.clear();
  }
};

// Copies n bytes and returns their chunk flags (chunk_flags).  Chunks are almost always pure
// A/C/G/T, which a loop without a table decides 16 bytes at a time; the others look their
// bytes up.
inline int copy_chunk(unsigned char* out, const unsigned char* in, int n) {
  unsigned char other = 0;
  for (int i = 0; i < n; ++i) {
    const unsigned char c = in[i];
    out[i] = c;
    other |= (unsigned char)!((c == 'A') | (c == 'C') | (c == 'G') | (c == 'T'));
  }
  return other ? chunk_flags(in, n) : 6;
}

// Returns an empty string on success, else the reason the input is rejected.
// t_tail / q_tail (optional, n entries each) are the signal tails of include/sxc.h.
// Two passes: the distinct chunks and their places, then their bytes and flags, which large
// batches copy on several threads (2048 pairs of 4096 bp, 16.8 MB, this container's CPU: 21 ms
// with one growing vector, an ordered map and a table lookup per byte, 4.5 ms now).
inline std::string pack_batch(const sxc_pair* in, int n, int N, HostBatch& hb,
                              const sxc_signal_tail* t_tail = nullptr, const sxc_signal_tail* q_tail = nullptr) {
  hb.reset();
  struct Key {
    const char* s;
    int len, tail;
    bool operator==(const Key& o) const { return s == o.s && len == o.len && tail == o.tail; }
  };
  struct Hash {
    size_t operator()(const Key& k) const {
      uint64_t h = (uint64_t)(uintptr_t)k.s * 0x9E3779B97F4A7C15ull;
      h ^= ((uint64_t)(uint32_t)k.len << 32 | (uint32_t)k.tail) * 0xC2B2AE3D27D4EB4Full;
      return (size_t)(h ^ (h >> 29));
    }
  };
  using Map = std::unordered_map<Key, int, Hash>;
  Map tmap((size_t)n * 2), qmap((size_t)n * 2), smap;
  std::map<std::pair<const sxc_tail_seg*, int>, int> tailmap;
  struct Source {  // where a chunk's bytes come from, and its table
    const char* s;
    std::vector<sxc_chunk>* tab;
    int idx;
  };
  std::vector<Source> src;
  int64_t end = 0;
  auto place = [&](const char* s, int len, std::vector<sxc_chunk>& tab, int& idx) -> std::string {
    if (len < 0 || (len > 0 && !s)) return "negative length or null sequence";
    if (len > N) return "sequence longer than the FFT length N";
    idx = (int)tab.size();
    tab.push_back(sxc_chunk{end, len, 0});
    src.push_back(Source{s, &tab, idx});
    end += (len + 15) & ~15;  // next chunk 16-byte aligned
    if (len > hb.max_len) hb.max_len = len;
    return "";
  };
  auto add = [&](const char* s, int len, int tail, std::vector<sxc_chunk>& tab, Map& m, int& idx) -> std::string {
    const auto it = m.try_emplace(Key{s, len, tail}, -1);
    if (!it.second) {
      idx = it.first->second;
      return "";
    }
    const std::string e = place(s, len, tab, idx);
    it.first->second = idx;
    return e;
  };
  // A tail for a chunk of length L: segments must tile [L, end) upwards within each
  // source's length and N.  Returns the tail index (-1 for none) through idx.
  auto add_tail = [&](const sxc_signal_tail* t, int L, int& idx) -> std::string {
    idx = -1;
    if (!t || t->nseg == 0) return "";
    if (t->nseg < 0 || !t->segs) return "bad signal tail";
    int start = L;
    for (int k = 0; k < t->nseg; ++k) {
      const sxc_tail_seg& g = t->segs[k];
      if (g.end <= start || g.end > g.len || g.end > N || (g.strand != 0 && g.strand != 1))
        return "signal tail segments must tile [chunk length, end) within their sources";
      start = g.end;
    }
    const auto key = std::make_pair(t->segs, t->nseg);
    auto it = tailmap.find(key);
    if (it != tailmap.end()) {
      idx = it->second;
      return "";
    }
    sxc_tail_dev td{(int32_t)hb.segs.size(), t->nseg};
    for (int k = 0; k < t->nseg; ++k) {
      const sxc_tail_seg& g = t->segs[k];
      const auto si = smap.try_emplace(Key{g.seq, g.len, g.strand}, -1);
      if (si.second) {
        int at;
        std::string e = place(g.seq, g.len, hb.schunks, at);
        if (!e.empty()) return e;
        si.first->second = at;
        hb.sstrand.push_back(g.strand);
      }
      hb.segs.push_back(sxc_tail_seg_dev{g.end, si.first->second});
    }
    idx = (int)hb.tails.size();
    hb.tails.push_back(td);
    tailmap[key] = idx;
    return "";
  };
  hb.pairs.resize(n);
  for (int k = 0; k < n; ++k) {
    const sxc_pair& p = in[k];
    sxc_pair_dev& d = hb.pairs[k];
    // lags span +-N/2: the shorter chunk must fit in half the transform (the slave uses
    // N = 2 * t_chunk, so every chunk does)
    if (p.tlen > N / 2 && p.qlen > N / 2) return "both chunks longer than N/2";
    int tt, qt;
    std::string e = add_tail(t_tail ? &t_tail[k] : nullptr, p.tlen, tt);
    if (!e.empty()) return e;
    e = add_tail(q_tail ? &q_tail[k] : nullptr, p.qlen, qt);
    if (!e.empty()) return e;
    const size_t before = hb.tchunks.size();
    e = add(p.tseq, p.tlen, tt, hb.tchunks, tmap, d.t_chunk);
    if (!e.empty()) return e;
    if (hb.tchunks.size() > before) hb.ttail.push_back(tt);
    e = add(p.qseq, p.qlen, 0, hb.qchunks, qmap, d.q_chunk);
    if (!e.empty()) return e;
    d.t_chunk_start = p.t_chunk_start;
    d.q_chunk_start = p.q_chunk_start;
    d.t_record = p.t_record;
    d.q_record = p.q_record;
    d.q_record_len = p.q_record_len;
    d.fast = p.fast;
    d.q_tail = qt;
  }
  if (hb.tails.empty()) hb.ttail.clear();  // no tails at all: kernels skip the lookups
  // the bytes, each chunk padded with zeros, and 16 more for the read-ahead of aligned word copies
  hb.seq.resize((size_t)end + 16);
  memset(hb.seq.data() + end, 0, 16);
  auto copy = [&](size_t lo, size_t hi) {
    for (size_t i = lo; i < hi; ++i) {
      sxc_chunk& c = (*src[i].tab)[(size_t)src[i].idx];
      unsigned char* to = hb.seq.data() + c.off;
      // bit 1: only A, C, G, T (scores are 100 or 0); bit 2: only A, C, G, T, N
      c.flags = c.len ? copy_chunk(to, (const unsigned char*)src[i].s, c.len) : chunk_flags(nullptr, 0);
      memset(to + c.len, 0, (size_t)(((c.len + 15) & ~15) - c.len));
    }
  };
  const size_t jobs = end < (4 << 20) ? 1 : std::min<size_t>(8, (size_t)(end >> 21));
  std::vector<std::thread> team;
  for (size_t j = 1; j < jobs; ++j) {
    const size_t lo = src.size() * j / jobs, hi = src.size() * (j + 1) / jobs;
    try {
      team.emplace_back(copy, lo, hi);
    } catch (...) {  // no thread to be had
      copy(lo, hi);
    }
  }
  copy(0, src.size() / jobs);
  for (std::thread& t : team) t.join();
  for (const Source& x : src) {
    sxc_chunk& c = (*x.tab)[(size_t)x.idx];
    if (c.flags < 0) return "sequence byte >= 128";
    if (c.flags & 1) {  // window entropies with the host's log
      const size_t row = hb.ent.size() / SXC_ENT_ROW;
      if (row >= (1u << 24)) return "too many chunks with B, D, H or V letters";
      c.flags |= (int32_t)(row << 8);
      hb.ent.resize(hb.ent.size() + SXC_ENT_ROW);
      window_entropy_row(hb.seq.data() + c.off, c.len, N, hb.ent.data() + row * SXC_ENT_ROW);
    }
  }
  return "";
}

inline int nb_of(int N) {
  int nb = 0;
  while ((1 << nb) < N) ++nb;
  return ((1 << nb) == N) ? nb : -1;
}

}  // namespace sxc
