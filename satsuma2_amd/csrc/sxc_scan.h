// sxc_scan.h -- diagonal scan of every accepted lag and the FP64 match tail.
//
// One workgroup per (pair, strand).  SeqAnalyzer::DoOne (OPTIM_DOONE,
// analysis/CrossCorr.cc:667-724) slides a 46-wide window of integer scores
// (int)(100 * DNA_EqualAmb + 0.5) along the diagonal of each lag FindTop accepted and
// opens a run while the window sum exceeds 1889.
// Pairs of pure A/C/G/T chunks (scan_sliced): a thread moves 32 blocks of a lag by one position
// per operation, one block in each bit of a word, and names the blocks whose runs may be kept;
// those are scanned again position by position.  Pairs with a few letters other than A/C/G/T/N are
// scanned the same way, those letters taken as identical in the first pass.  Other pairs take
// their lags in epochs of 8 or 16.  A/C/G/T/N (scan_epoch_bitmap): threads take whole 32-position blocks of a lag, keep the
// window's flags in an LDS bitmap, and a second pass turns each rising edge into a run.  The
// rest (scan_epoch_segments): a lag's diagonal is split into contiguous
// segments, one per thread; each thread recomputes the window at its segment start,
// records the runs that open and close inside its segment, and a second phase closes runs
// that cross segment boundaries.  Runs go to an LDS queue; the queue is drained by all
// threads at once, one run per thread, through GetMatchProbabilityEx
// (analysis/AlignProbability.cc:62-127) and FilterMatches
// (analysis/HomologyByXCorrSlave.cc:168-219).  Kept records carry the key
// (lag rank, run start) so the finalize kernel restores the reference's order.
//
// Queue capacity: the segment scans' queue holds every run one lag can produce (runs need
// a below-threshold gap, so at most npos/2 + 1 per lag, npos <= N/2), and an epoch of
// several lags that overflows is discarded and redone one lag at a time; the bitmap scan
// re-extracts an overflowing epoch's runs in rounds that each fit its queue, and the sliced scan
// scans slices whose blocks overflow it again, as many as always fit.
#pragma once
#include <math.h>

#include <type_traits>

#include "sxc_fft.h"
#include "sxc_tables.h"

namespace sxc {

struct ScanArgs {
  const sxc_tables* tab;
  const unsigned char* seq;
  const sxc_chunk* tchunks;
  const sxc_chunk* qchunks;
  const sxc_pair_dev* pairs;
  const uint16_t* cands;     // accepted lags, N slots per (pair, strand)
  const int32_t* ncand;      // accepted lags per (pair, strand)
  int32_t n_fft;             // N
  int32_t strands;
  int32_t min_len;
  int32_t q_chunk;
  double min_prob;
  double target_total;
  double z_skip;             // runs with (m - x) / s / 1.414213562 >= z_skip have prob < min_prob
  // shortest flagged stretch (ne - ns) a kept run can have, by the kernel that finds it (pure
  // A/C/G/T, with N, general): keep_min_run.  0 or 1: every run reaches the tail.
  int32_t min_run[3];
  // keep band (keep_band): runs with prob >= keep_lo are written; those with prob < flag_hi
  // are flagged SXC_REC_NEAR for the host to decide, and counted in *nflag (optional)
  double keep_lo;
  double flag_hi;
  int32_t* nflag;
  int32_t mode;              // 0: filter runs into t_results; 1: write runs (MatchUp)
  sxc_result_dev* out;       // mode 0: cap records per (pair, strand)
  int32_t* runs;             // mode 1: cap x {start_target, start_query, len} per (pair, strand)
  uint64_t* keys;
  int32_t* counts;
  int32_t cap;
  int32_t* stats;            // optional {candidates, runs} per (pair, strand)
  const double* ptable;      // optional ProbTable thresholds (SXC_PT_ROWS x SXC_PT_LEN): -prob_table
  double table_prob;         // what a table hit reports (the table's cutoff)
  // workgroups per (pair, strand), each scanning a contiguous share of its accepted lags
  // (0 or 1: one).  With more than one, records take their slots through a global atomic
  // on counts[ps], which must be zero at launch (the pair kernel clears it), and stats
  // runs are added atomically.
  int32_t split;
  const int32_t* list;       // optional: the (pair, strand)s to scan (null: 0 on)
};

// The kinds of chunk pairs the scan has a kernel of its own for, and how many of a launch's
// pairs are of each.
enum { SCAN_PURE = 0, SCAN_N = 1, SCAN_GENERAL = 2 };
SXC_HD inline int scan_kind(int32_t tflags, int32_t qflags) {
  return (tflags & qflags & 2) ? SCAN_PURE : (tflags & qflags & 4) ? SCAN_N : SCAN_GENERAL;
}
struct ScanKinds {
  int32_t pairs[3] = {0, 0, 0};
  bool mixed() const { return (pairs[0] > 0) + (pairs[1] > 0) + (pairs[2] > 0) > 1; }
  int32_t all() const { return pairs[0] + pairs[1] + pairs[2]; }
  // Of a mixed launch, the (pair, strand)s grouped by kind: a kind's launch covers its own only.  (Over
  // all pairs, with the others' workgroups leaving at once, the shares of a rare kind's strands
  // multiplied the whole grid: one pure pair among 100000 with N at N = 512 took 3.2 M workgroups,
  // 9.27 ms against 7.54, and one among 524297 lost its records, as a grid of 2^32 threads or more
  // wraps.  One pair with N among 4096 of 4096 bp: 0.615 and 0.598 ms.)
  template <class KindOf>
  void list(KindOf&& kind_of, int strands, int32_t* out) const {
    int32_t at[3] = {0, strands * pairs[0], strands * (pairs[0] + pairs[1])};
    for (int32_t k = 0; k < all(); ++k) {
      int32_t& to = at[kind_of(k)];
      for (int s = 0; s < strands; ++s) out[to++] = strands * k + s;
    }
  }
};

// Host: the keep decision's parameters for min_prob and the target size -- the float
// pre-filter's z bound and the keep band (sxc_tables.h).
inline void set_keep(ScanArgs& a, double min_prob, double target_total) {
  a.min_prob = min_prob;
  a.target_total = target_total;
  a.z_skip = keep_z_bound(min_prob, target_total);
  // a window that rises to its threshold holds at most this much identity (in bases): 19
  // identical bases; 4 M + K in [76, 79] quarters with N; a score in (1889, 1989] whose
  // hundredths are rounded by at most half a point per position
  a.min_run[0] = keep_min_run(a.z_skip, 19.);
  a.min_run[1] = keep_min_run(a.z_skip, 79. / 4.);
  a.min_run[2] = keep_min_run(a.z_skip, 19.89 + 46. * 0.005);
  keep_band(min_prob, target_total, &a.keep_lo, &a.flag_hi);
}

constexpr int SCAN_NT = 256;  // threads per scan workgroup
// smallest count c of identical A/C/G/T bases with 100 * c > 1889 (19 of 46)
constexpr int SXC_MIN_MATCHES = SXC_WIN_THRESHOLD / 100 + 1;
static_assert(100 * SXC_MIN_MATCHES > SXC_WIN_THRESHOLD && 100 * (SXC_MIN_MATCHES - 1) <= SXC_WIN_THRESHOLD, "");
// With N: a position involving an N scores 25 (N:N and N against A/C/G/T), so a window of M
// identical A/C/G/T bases and K positions with an N exceeds 1889 <=> 4 M + K >= 76.
constexpr int SXC_MIN_QUARTERS = SXC_WIN_THRESHOLD / 25 + 1;
static_assert(25 * SXC_MIN_QUARTERS > SXC_WIN_THRESHOLD && 25 * (SXC_MIN_QUARTERS - 1) <= SXC_WIN_THRESHOLD, "");

// NB: log2 N in bits 0-4; bit 5 selects the kernel for pairs whose two chunks are pure
// A/C/G/T (SLICED); bit 6 the one for pairs of A/C/G/T/N chunks with an N (HASN), whose LDS plan
// holds the packed bases, the N masks, the run queue and the counters (the accepted lags are read
// from global memory).  The general kernel takes every other pair.
template <int NB>
struct ScanSmem {
  static constexpr int LOG = NB & 31;
  static constexpr bool HASN = (NB & 64) != 0;
  static constexpr bool PURE = (NB & 96) != 0;
  static constexpr int N = 1 << LOG;
  // The pure kernel (SLICED) scans 32 blocks of a lag in the bits of a word (scan_sliced) and needs
  // no bitmap: bit planes of the bases instead of the packed words, the staged lags, the queue
  // of blocks and a run count per thread.
  static constexpr bool SLICED = PURE && !HASN;
  // The general kernel scans pairs with few other letters the same way, with a plane of those
  // letters beside the bases; its area for that lies over the segment scan's.
  static constexpr bool AMB = !PURE;
  // The segment scans' queue holds every run one lag can produce (npos / 2 + 1, npos <= N / 2);
  // the bitmap scan and the sliced scan flush theirs whenever it would overflow (the sliced scan's
  // also holds the query's planes while they are turned around).
  static constexpr int QCAP = (SLICED ? (N / 16 < 1024 ? 1024 : N / 16) : PURE ? 896 : N / 4 + 64);
  static constexpr int PKW = SLICED ? 0 : N / 16 + 4;   // 2-bit packed words (+3 words of read-ahead)
  static constexpr int TCODE = 0;                       // uchar[N] (general kernel)
  static constexpr int QCODE = TCODE + (PURE ? 0 : N);  // uchar[N] (general kernel)
  static constexpr int TPK = QCODE + (PURE ? 0 : N);    // uint32[PKW]: 16 bases per word (HASN)
  static constexpr int QPK = TPK + 4 * PKW;             // uint32[PKW]
  // The kernel with N (BMRUNS) keeps each epoch's flags in a bitmap of WPL words per lag and
  // turns its rising edges into runs afterwards; the general kernel scans contiguous
  // segments per thread and stitches runs across them.  BMRUNS, and the general kernel from
  // N = 8192 (4 of its workgroups per CU instead of 3: 200 strands 0.54 ms instead of 0.74; at
  // N = 2048 0.57 instead of 0.44), take one epoch at a time (drained after every epoch) in
  // 4-byte queue entries {lag - first lag of the epoch (RB bits), ns (NSB = LOG - 1), ne
  // (LOG)}; otherwise 16-lag epochs accumulate in 8-byte entries {lag rank, ns | ne << 16}
  // until the queue is half full.
  static constexpr bool BMRUNS = HASN;
  static constexpr bool COMPACT = PURE || LOG >= 13;
  static constexpr int CE = LOG >= 14 ? 8 : 16;         // lags per epoch
  static constexpr int GSZ = SCAN_NT / CE;              // threads per lag in an epoch
  static constexpr int NSB = LOG - 1;                   // ns < N / 2
  static constexpr int RB = 32 - NSB - LOG;             // ne <= N / 2 takes LOG bits
  static_assert(!COMPACT || (RB > 0 && (1 << RB) >= CE), "compact queue entries");
  static constexpr int QE = COMPACT ? 4 : 8;            // bytes per queue entry
  static constexpr int WPL = N / 64;                    // bitmap words per lag: npos <= N / 2
  static constexpr int TNK = QPK + 4 * PKW;             // uint32[PKW]: bit 2b set where base b of a word is N (HASN)
  static constexpr int QNK = TNK + (HASN ? 4 * PKW : 0);
  static constexpr int QUEUE = QNK + (HASN ? 4 * PKW : 0);  // queue entries [QCAP]
  static constexpr int SUMM = QUEUE + QE * QCAP;        // int2[SCAN_NT] (segments)
  static constexpr int BITMAP = SUMM;                   // uint32[CE][WPL] (BMRUNS)
  static constexpr int RLIST = BITMAP + 4 * CE * WPL;   // uint16[CE * WPL]: blocks with a rising edge (BMRUNS)
  static constexpr int PLW = N / 32 + 2 + 34;           // plane words: blocks -2 .. of a scan that runs past the end
  static constexpr int SQCAP = SLICED ? QCAP : 928;     // queue entries of the sliced scan
  static constexpr int TPL = (QUEUE + 4 * SQCAP + 7) & ~7;  // uint32[PLW][2]: low and high bits of 32 bases (SLICED, AMB)
  static constexpr int QPL = TPL + 8 * PLW;
  static constexpr int TAM = QPL + 8 * PLW;             // uint32[PLW]: letters other than A/C/G/T (AMB)
  static constexpr int QAM = TAM + (AMB ? 4 * PLW : 0);
  static constexpr int RPL = QUEUE;                     // uint32[N/32][2]: the query, reversed (before the scan)
  static constexpr int LAGS = QAM + (AMB ? 4 * PLW : 0);  // uint16[SLICE_LAGS]
  static constexpr int RUNS = LAGS + 2 * 512;           // int32[SCAN_NT]
  static constexpr int RANGE = RUNS + 4 * SCAN_NT;      // int32[2 * 32]: first lag with a slice, and how many have it
  static constexpr int SEND = (RANGE + 4 * 64 + 7) & ~7;
  static constexpr int EEND = (SUMM + (BMRUNS ? 6 * CE * WPL : 8 * SCAN_NT) + 7) & ~7;
  static constexpr int EQUAL = SLICED ? SEND : BMRUNS || EEND > SEND ? EEND : SEND;  // double[18][18]
  static constexpr int NTAB = PURE ? 0 : 1;             // the score tables (general kernel)
  static constexpr int GC = EQUAL + NTAB * 8 * SXC_NCLASS * SXC_NCLASS;  // double[18]
  static constexpr int SCORE = GC + NTAB * 8 * SXC_NCLASS;              // uchar[18][18]
  static constexpr int CLS = SCORE + NTAB * SXC_NCLASS * SXC_NCLASS;     // uchar[128]
  static constexpr int RC = CLS + NTAB * 128;                           // uchar[128]
  static constexpr int MISC = (RC + NTAB * 128 + 15) & ~15;             // int[16 + CE]
  static constexpr int BYTES = MISC + 64 + 4 * CE;
};

enum { SM_QN = 0, SM_KEPT = 1, SM_RUNS = 2, SM_NCAND = 3, SM_LT = 4, SM_LQ = 5, SM_NRB = 7, SM_AMB = 8, SM_BASES = 9 /* 4 ints */,
       SM_NPOS = 16 };

// Base code: class id (0..16) of a codec letter, or 128 | byte for a byte whose codec
// row is zero.  Two bases are identical bytes iff their codes are equal.
SXC_HD inline unsigned char base_code(const sxc_tables* tab, unsigned char b) {
  const unsigned char c = tab->cls[b & 127];
  return c < SXC_CLASS_ZERO ? c : (unsigned char)(128 | b);
}

// (int)(100 * DNA_EqualAmb(a, b) + 0.5): identical letters other than 'N' score 100
// (analysis/DNAVector.cc:372-387), 'N':'N' scores 25, a zero-row byte scores 0 against
// any different byte.
SXC_HD inline int code_score(const unsigned char* score, unsigned ca, unsigned cb) {
  if (ca == cb) return ca == SXC_CLASS_N ? 25 : 100;
  if ((ca | cb) & 128) return 0;
  return score[ca * SXC_NCLASS + cb];
}

SXC_HD inline int code_class(unsigned c) { return c < 128 ? (int)c : SXC_CLASS_ZERO; }

// ---- bit-parallel window counts for pure A/C/G/T diagonals
//
// Bases are packed 2 bits each, 16 per 32-bit word.  32 bases of the target and of the
// query diagonal XOR to 32 2-bit groups; a group is zero exactly where the bases match.
// Block k of a diagonal holds the match bits of positions [32k, 32k + 32) at even bit
// positions; the 46-wide window count at position n = 32k + r reads blocks k, k-1, k-2.

SXC_HD inline uint64_t load32(const uint32_t* pk, int p) {  // 32 bases starting at base p >= 0
  const int w = p >> 4, b = (p & 15) * 2;
  const uint64_t lo = (uint64_t)pk[w] | ((uint64_t)pk[w + 1] << 32);
  if (!b) return lo;
  return (lo >> b) | ((uint64_t)pk[w + 2] << (64 - b));
}

SXC_HD inline int popc64(uint64_t v) { return __builtin_popcountll(v); }

// bits [s, s + 32) of hi:lo, 0 <= s < 32 (a funnel shift: one v_alignbit)
SXC_HD inline uint32_t funnel32(uint32_t hi, uint32_t lo, int s) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_alignbit(hi, lo, (unsigned)s);
#else
  return (lo >> s) | ((hi << 1) << (31 - s));
#endif
}

// Bytes of hi:lo chosen by the selector bytes of sel (0-3: lo's bytes, 4-7: hi's; v_perm_b32).
SXC_HD inline uint32_t byte_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_perm(hi, lo, sel);
#else
  const uint64_t v = ((uint64_t)hi << 32) | lo;
  uint32_t r = 0;
  for (int b = 0; b < 4; ++b) r |= (uint32_t)((v >> (8 * ((sel >> (8 * b)) & 7))) & 0xffu) << (8 * b);
  return r;
#endif
}

// Hides x's value from the optimizer (no instruction).
SXC_HD inline void opaque(uint32_t& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(x));
#else
  (void)x;
#endif
}

// Nothing is moved across this point by the instruction scheduler (no instruction).
SXC_HD inline void keep_order() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// a where mask is set, b elsewhere (v_bfi_b32)
SXC_HD inline uint32_t bit_select(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// Window flags of 16 consecutive positions, four at a time in the bytes of a word.  Group p
// (bits 2p, 2p + 1) of z holds m(n) + 1 - m(n - 46) in {0, 1, 2} for the half's position p;
// byte i covers positions 4i .. 4i + 3 and carries u = C - 19 + 128, C the window count.  As
// 0 <= C <= 46, every u below lies in [109, 155]: no add carries and no subtraction borrows
// across a byte, and bit 7 of u is the flag C >= 19.  ub holds u of the position before the
// half in every byte and is advanced to the half's last position.  The flag of position
// 4i + r is returned at bit 8i + 4 + r (bits 8i .. 8i + 3 are not defined).
SXC_HD inline uint32_t half_flags(uint32_t z, uint32_t& ub) {
  const uint32_t A = z & 0x33333333u;               // per byte: z0 | z2 << 4
  const uint32_t P = A + ((z >> 2) & 0x33333333u);  // z0 + z1 | (z2 + z3) << 4
  const uint32_t P01 = P & 0x0F0F0F0Fu;
  const uint32_t s = P01 + ((P >> 4) & 0x0F0F0F0Fu);  // the byte's four z, <= 8
  // the earlier bytes' s (<= 24): shift-adds, kept from being folded into a quarter-rate multiply
  uint32_t x = s + (s << 8);
  opaque(x);
  x = x + (x << 16);
  opaque(x);
  x <<= 8;
  const uint32_t u0 = ub + x - 0x0C080400u;  // u at position 4i - 1
  const uint32_t u1 = u0 + (A & 0x03030303u) - 0x01010101u;
  const uint32_t u2 = u0 + P01 - 0x02020202u;
  const uint32_t u3 = u2 + ((A >> 4) & 0x03030303u) - 0x01010101u;
  const uint32_t u4 = u0 + s - 0x04040404u;
  ub = byte_perm(u4, u4, 0x03030303u);
  return bit_select(0x80808080u, u4, bit_select(0x40404040u, u3 >> 1, bit_select(0x20202020u, u2 >> 2, u1 >> 3)));
}

// Window flags of a 32-position block (bit r: position r) from its z groups (positions 0-15
// in zl, 16-31 in zh); ub as in half_flags.
SXC_HD inline uint32_t window_flags(uint32_t zl, uint32_t zh, uint32_t& ub) {
  const uint32_t n0 = half_flags(zl, ub);
  const uint32_t n1 = half_flags(zh, ub);
  // bytes 0 and 2 of c gather the half's positions 0-7 and 8-15
  const uint32_t c0 = bit_select(0x0F0F0F0Fu, n0 >> 4, n0 >> 8);
  const uint32_t c1 = bit_select(0x0F0F0F0Fu, n1 >> 4, n1 >> 8);
  return byte_perm(c1, c0, 0x06040200u);
}

// half_flags' four u words (byte i of u[t]: u at position 4i + t) for any count that changes
// by z - 1 per position and stays within [0, 255] at every position; ub as in half_flags.
SXC_HD inline void half_values(uint32_t z, uint32_t& ub, uint32_t* u) {
  const uint32_t A = z & 0x33333333u;
  const uint32_t P = A + ((z >> 2) & 0x33333333u);
  const uint32_t P01 = P & 0x0F0F0F0Fu;
  const uint32_t s = P01 + ((P >> 4) & 0x0F0F0F0Fu);
  uint32_t x = s + (s << 8);
  opaque(x);
  x = x + (x << 16);
  opaque(x);
  x <<= 8;
  const uint32_t u0 = ub + x - 0x0C080400u;
  u[0] = u0 + (A & 0x03030303u) - 0x01010101u;
  u[1] = u0 + P01 - 0x02020202u;
  u[2] = u[1] + ((A >> 4) & 0x03030303u) - 0x01010101u;
  u[3] = u0 + s - 0x04040404u;
  ub = byte_perm(u[3], u[3], 0x03030303u);
}

// Window flags of a 32-position block of an A/C/G/T/N pair (bit r: position r).  The window
// holds M identical A/C/G/T bases and K positions with an N (M + K <= 46); its score
// 100 M + 25 K exceeds 1889 iff 4 M + K >= 76.  zm* and zk* hold m(n) + 1 - m(n - 46) and
// k(n) + 1 - k(n - 46) per position as z of half_flags (positions 0-15 in *l, 16-31 in *h);
// ubm carries M and ubk K + 128 - 76 in every byte, advanced as ub of half_flags.  Per byte
// 4 M + (K + 52) <= 3 M + 98 <= 236 (4 M < 256 keeps M's bits in its byte), so bit 7 of the
// combined byte is the flag.
SXC_HD inline uint32_t window_flags_mk(uint32_t zml, uint32_t zmh, uint32_t zkl, uint32_t zkh, uint32_t& ubm,
                                       uint32_t& ubk) {
  auto half = [&](uint32_t zm, uint32_t zk) {
    uint32_t um[4], uk[4], c[4];
    half_values(zm, ubm, um);
    half_values(zk, ubk, uk);
    for (int t = 0; t < 4; ++t) c[t] = (um[t] << 2) + uk[t];
    return bit_select(0x80808080u, c[3], bit_select(0x40404040u, c[2] >> 1, bit_select(0x20202020u, c[1] >> 2, c[0] >> 3)));
  };
  const uint32_t n0 = half(zml, zkl);
  const uint32_t n1 = half(zmh, zkh);
  const uint32_t c0 = bit_select(0x0F0F0F0Fu, n0 >> 4, n0 >> 8);
  const uint32_t c1 = bit_select(0x0F0F0F0Fu, n1 >> 4, n1 >> 8);
  return byte_perm(c1, c0, 0x06040200u);
}

// matches in the window [n - 45, n], n = 32k + r
SXC_HD inline int window_count(uint64_t e0, uint64_t e1, uint64_t e2, int r) {
  const uint64_t low = (r == 31) ? ~0ull : ((1ull << (2 * r + 2)) - 1);
  int c = popc64(e0 & low);
  if (r >= 13) {
    c += popc64(e1 & ~((1ull << (2 * (r - 13))) - 1));
  } else {
    c += popc64(e1) + popc64(e2 & ~((1ull << (2 * (r + 19))) - 1));
  }
  return c;
}

// Counts over a run of bases that may be N (bit 2b of the N mask words set): identical A/C/G/T
// bases, positions with an N on either side, C/G bases and N bases of each side.
SXC_HD inline void packed_counts_n(const uint32_t* tpk, const uint32_t* qpk, const uint32_t* tnk,
                                   const uint32_t* qnk, int st, int sq, int len, int& match, int& nk, int& gct,
                                   int& ntn, int& gcq, int& nqn) {
  match = nk = gct = ntn = gcq = nqn = 0;
  for (int off = 0; off < len; off += 32) {
    const int m = (len - off < 32) ? len - off : 32;
    const uint64_t keep = ((m == 32) ? ~0ull : ((1ull << (2 * m)) - 1)) & 0x5555555555555555ull;
    const uint64_t tv = load32(tpk, st + off), qv = load32(qpk, sq + off);
    const uint64_t tn = load32(tnk, st + off) & keep, qn = load32(qnk, sq + off) & keep;
    const uint64_t x = tv ^ qv;
    match += popc64(~(x | (x >> 1)) & keep & ~(tn | qn));
    nk += popc64(tn | qn);
    gct += popc64((tv ^ (tv >> 1)) & keep & ~tn);
    gcq += popc64((qv ^ (qv >> 1)) & keep & ~qn);
    ntn += popc64(tn);
    nqn += popc64(qn);
  }
}

// The tail after the sums (GCAdjustExpect, Sigma, CDF; analysis/AlignProbability.cc:11-40,
// 107-126).  Returns false, without evaluating erf/exp, when z >= z_skip guarantees the
// probability is below the keep threshold.
SXC_HD inline bool tail_from_sums(double matches, double gct, double gcq, int len, double target_size, double z_skip,
                                  double& prob, double& ident) {
  ident = matches / (double)len;
  const double gc_target = gct / (double)len;
  const double at_target = 1. - gc_target;
  double r = gcq * gc_target;
  r += ((double)len - gcq) * at_target;
  const double p = r / (double)len / 2.;
  const double s = sqrt(p * (1. - p) * (double)len);
  const double m = p * (double)len;
  const double x = (double)len * ident;
  const double z = (m - x) / s / 1.414213562;
  if (z >= z_skip) return false;
  const double cdf = 0.5 * (1. + erf(z));
  const double expect = cdf * target_size;
  prob = exp(-expect);
  return true;
}

// The z of tail_from_sums estimated in float from the integer sums: its error (|m - x| off
// by at most ~5e-7 * len, s by a few ulp) is far below the margin, so a true result implies
// z >= z_skip in FP64 as well and the run can be dropped without the FP64 divisions.
SXC_HD inline bool z_clearly_skipped(int matches, int gct, int gcq, int len, double z_skip) {
  const float fl = (float)len;
  const float gt = (float)gct / fl;
  const float r = (float)gcq * gt + (float)(len - gcq) * (1.f - gt);
  const float p = r / fl * 0.5f;
  const float s = sqrtf(p * (1.f - p) * fl);
  const float z = (p * fl - (float)matches) / s * 0.70710678f;
  const float margin = 1e-5f * (fl / s + fabsf(z) + 1.f);
  return z - margin >= (float)z_skip;  // false for NaN (s = 0) and for z_skip = inf
}

// ProbTable::GetMatchProbability after the sums (analysis/ProbTable.cc:118-141): the table's
// cutoff if the identity reaches the threshold for (expected identity, length), else 0.  An
// expectation below 1/511 selects row 0, which the reference leaves empty; it reports 0.
SXC_HD inline double table_from_sums(double matches, double gct, double gcq, int len, const double* ptable,
                                     double table_prob, double& ident) {
  ident = matches / (double)len;
  const double gc_target = gct / (double)len;
  const double at_target = 1. - gc_target;
  double r = gcq * gc_target;
  r += ((double)len - gcq) * at_target;
  const double p = r / (double)len / 2.;
  const int index = (int)(p * (SXC_PT_ROWS - 1));
  if (index < 1) return 0.;
  const int l = len >= SXC_PT_LEN ? SXC_PT_LEN - 1 : len;
  return ident >= ptable[(size_t)index * SXC_PT_LEN + l] ? table_prob : 0.;
}

struct Lag {
  int shift, i0, npos;
};

SXC_HD inline Lag lag_geometry(int idx, int H, int Lq, int Lt) {
  // SeqAnalyzer::DoOne loop bounds: i from max(0, -shift) while j = i + shift < Lq and
  // i + 1 < Lt (analysis/CrossCorr.cc:685-696)
  Lag g;
  g.shift = idx - H;
  g.i0 = g.shift < 0 ? -g.shift : 0;
  int iend = Lq - g.shift;
  if (Lt - 1 < iend) iend = Lt - 1;
  g.npos = (g.i0 < Lt && iend > g.i0) ? iend - g.i0 : 0;
  return g;
}

// Queue entry of a run (both kernels): compact {lag - first lag of the epoch, ns, ne}
// or the 8-byte {lag rank, ns | ne << 16}.
template <int NB, class Ex>
SXC_HD inline void push_run(Ex& ex, char* sm, int c0, int rank, int ns, int ne) {
  using SS = ScanSmem<NB>;
  int* misc = (int*)(sm + SS::MISC);
  int* queue = (int*)(sm + SS::QUEUE);
  const int k = ex.atomic_add_shared(&misc[SM_QN], 1);
  if (k < SS::QCAP) {
    if constexpr (SS::COMPACT) {
      queue[k] = (int)((unsigned)(rank - c0) | ((unsigned)ns << SS::RB) | ((unsigned)ne << (SS::RB + SS::NSB)));
    } else {
      queue[2 * k] = rank;
      queue[2 * k + 1] = ns | (ne << 16);
    }
  }
}

// A/C/G/T/N lags [c0, c1), gsz threads per lag.  The window's counts are running sums with
// m(< 0) = 0, as the reference's `match` (analysis/CrossCorr.cc:700-705).  Each thread takes whole
// 32-position blocks of one lag, updates every position branch-free and stores the block's
// flags (window above the threshold, positions >= 46 and < npos) in the epoch's LDS
// bitmap.  A second pass over the bitmap words, spread over all threads, turns every rising
// edge at ns and the first clear flag after it at ne (or npos, where the loop ends) into
// the run [ns, ne) -- the runs DoOne opens and closes.
template <int NB, class Ex, class Flush>
SXC_HD inline void scan_epoch_bitmap(Ex& ex, char* sm, const uint16_t* cands, int c0, int c1, int gsz, int min_run,
                                     bool count, Flush&& flush) {
  using SS = ScanSmem<NB>;
  constexpr int H = SS::N / 2;
  constexpr int WPL = SS::WPL;
  int* misc = (int*)(sm + SS::MISC);
  int* npos_of = misc + SM_NPOS;
  uint32_t* bm = (uint32_t*)(sm + SS::BITMAP);
  const uint32_t* tpk = (const uint32_t*)(sm + SS::TPK);
  const uint32_t* qpk = (const uint32_t*)(sm + SS::QPK);
  const int Lt = misc[SM_LT], Lq = misc[SM_LQ];
  const int nl = c1 - c0;
  ex.each([&](int tid) {
    const int j = tid / gsz;
    const int l = tid % gsz;
    if (j >= nl) return;
    const Lag g = lag_geometry(cands[c0 + j], H, Lq, Lt);
    if (l == 0) npos_of[j] = g.npos;
    // whole blocks per thread: no block is written by two threads
    const int S = ((g.npos + gsz - 1) / gsz + 31) & ~31;
    const int na = l * S;
    const int nb = (na + S < g.npos) ? na + S : g.npos;
    if (na >= nb) return;
    uint32_t* row = bm + j * WPL;
    const int ti = g.i0, qj = g.i0 + g.shift;
    const int k0 = na >> 5, klast = (nb - 1) >> 5;
    uint16_t* rl = (uint16_t*)(sm + SS::RLIST);
    {
      // the window test 4 M + K >= 76 over M identical A/C/G/T bases (m bits) and K positions
      // with an N (k bits), byte-parallel from the 2-bit groups m(n) + 1 - m(n - 46) and
      // k(n) + 1 - k(n - 46) (window_flags_mk)
      const uint32_t* tnk = (const uint32_t*)(sm + SS::TNK);
      const uint32_t* qnk = (const uint32_t*)(sm + SS::QNK);
      auto mk_at = [&](int kb, uint64_t& m, uint64_t& kk) {
        if (kb < 0) {
          m = kk = 0;
          return;
        }
        const uint64_t x = load32(tpk, ti + 32 * kb) ^ load32(qpk, qj + 32 * kb);
        kk = (load32(tnk, ti + 32 * kb) | load32(qnk, qj + 32 * kb)) & 0x5555555555555555ull;
        m = ~(x | (x >> 1)) & 0x5555555555555555ull & ~kk;
      };
      uint64_t m3, k3, m2, k2, m1, k1;
      mk_at(k0 - 3, m3, k3);
      mk_at(k0 - 2, m2, k2);
      mk_at(k0 - 1, m1, k1);
      const int M0 = window_count(m1, m2, m3, 31), K0 = window_count(k1, k2, k3, 31);  // at 32 k0 - 1
      uint32_t prev = (na - 1 >= 46 && 4 * M0 + K0 >= SXC_MIN_QUARTERS) ? 1u : 0u;
      uint32_t ubm = byte_perm(0u, (uint32_t)M0, 0u);
      uint32_t ubk = byte_perm(0u, (uint32_t)(K0 + 128 - SXC_MIN_QUARTERS), 0u);
      for (int k = k0; k <= klast; ++k) {
        uint64_t m0, kk0;
        mk_at(k, m0, kk0);
        const uint64_t mm = (m2 >> 36) | (m1 << 28), km = (k2 >> 36) | (k1 << 28);  // at n - 46
        const uint32_t zml = (uint32_t)m0 + (~(uint32_t)mm & 0x55555555u);
        const uint32_t zmh = (uint32_t)(m0 >> 32) + (~(uint32_t)(mm >> 32) & 0x55555555u);
        const uint32_t zkl = (uint32_t)kk0 + (~(uint32_t)km & 0x55555555u);
        const uint32_t zkh = (uint32_t)(kk0 >> 32) + (~(uint32_t)(km >> 32) & 0x55555555u);
        uint32_t f = window_flags_mk(zml, zmh, zkl, zkh, ubm, ubk);
        if (32 * k < 46) f &= (46 - 32 * k >= 32) ? 0u : ~((1u << (46 - 32 * k)) - 1);  // flags from n = 46
        if (k == klast && nb - 32 * k < 32) f &= (1u << (nb - 32 * k)) - 1;
        row[k] = f;
        if (f & ~((f << 1) | prev)) rl[ex.atomic_add_shared(&misc[SM_NRB], 1)] = (uint16_t)(j * WPL + k);
        prev = f >> 31;
        m2 = m1;
        m1 = m0;
        k2 = k1;
        k1 = kk0;
      }
    }
  });
  ex.sync();
  int* queue = (int*)(sm + SS::QUEUE);
  const uint16_t* rlist = (const uint16_t*)(sm + SS::RLIST);
  // All listed blocks at once; if their runs overflowed the queue, again in rounds of blocks
  // that fit it (a word holds at most 16 rising edges), the queue flushed after each round.
  const int nrb = misc[SM_NRB];
  auto extract = [&](int x0, int x1, bool count_runs) {
    ex.each([&](int tid) {
      for (int x = x0 + tid; x < x1; x += SCAN_NT) {
        const int e = rlist[x];
        const int j = e / WPL, w = e % WPL;
        const int npos = npos_of[j];
        const int W = (npos + 31) >> 5;
        const uint32_t* row = bm + j * WPL;
        const uint32_t f = row[w];
        const uint32_t carry = w > 0 ? row[w - 1] >> 31 : 0u;
        uint32_t rises = f & ~((f << 1) | carry);
        while (rises) {
          const int r = __builtin_ctz(rises);
          rises &= rises - 1;
          if (count_runs) ex.atomic_add_shared(&misc[SM_RUNS], 1);  // (one atomic per wave)
          const uint32_t clear = ~f & (~0u << r);  // bit r is set: the first clear bit is above it
          int ne;
          if (clear) {
            ne = 32 * w + __builtin_ctz(clear);
          } else {
            int w2 = w + 1;
            while (w2 < W && row[w2] == ~0u) ++w2;
            ne = w2 < W ? 32 * w2 + __builtin_ctz(~row[w2]) : npos;
          }
          // Too short to be kept (keep_min_run).  A run that starts at 46, where DoOne's test
          // begins, may have been above the threshold before, so the bound does not hold for it.
          if (ne - (32 * w + r) < min_run && 32 * w + r != 46) continue;
          const int at = ex.atomic_add_shared(&misc[SM_QN], 1);  // one atomic per wave
          if (at < SS::QCAP)
            queue[at] = (int)((unsigned)j | ((unsigned)(32 * w + r) << SS::RB) | ((unsigned)ne << (SS::RB + SS::NSB)));
        }
      }
    });
    ex.sync();
  };
  extract(0, nrb, count);
  const int qn = misc[SM_QN];
  if (qn <= SS::QCAP) {
    flush(qn);
  } else {
    ex.sync();  // every thread has read the count
    ex.each([&](int tid) {
      if (tid == 0) misc[SM_QN] = 0;
    });
    ex.sync();
    for (int x0 = 0; x0 < nrb; x0 += SS::QCAP / 16) {
      extract(x0, (x0 + SS::QCAP / 16 < nrb) ? x0 + SS::QCAP / 16 : nrb, false);
      flush(misc[SM_QN]);
    }
  }
  ex.each([&](int tid) {
    if (tid == 0) misc[SM_NRB] = 0;
  });
  ex.sync();
}

// Lags [c0, c1) with gsz threads per lag, each thread scanning a contiguous segment: it
// recomputes the window at its segment start, records the runs that open and close inside
// its segment, and a second phase closes runs that cross segment boundaries.
template <int NB, class Ex>
SXC_HD inline void scan_epoch_segments(Ex& ex, char* sm, const uint16_t* cands, int c0, int c1, int gsz, int min_run) {
  using SS = ScanSmem<NB>;
  constexpr int INF = 0x7fffffff;
  constexpr int H = SS::N / 2;
  const unsigned char* tc = (const unsigned char*)(sm + SS::TCODE);
  const unsigned char* qc = (const unsigned char*)(sm + SS::QCODE);
  const unsigned char* score = (const unsigned char*)(sm + SS::SCORE);
  int* misc = (int*)(sm + SS::MISC);
  int* summ = (int*)(sm + SS::SUMM);
  const int Lt = misc[SM_LT], Lq = misc[SM_LQ];
  auto push = [&](int rank, int ns, int ne) {
    ex.atomic_add_shared(&misc[SM_RUNS], 1);
    if (ne - ns < min_run && ns != 46) return;  // too short to be kept (see scan_epoch_bitmap)
    push_run<NB>(ex, sm, c0, rank, ns, ne);
  };
  ex.each([&](int tid) {
    const int c = c0 + tid / gsz;
    const int l = tid % gsz;
    int first_end = INF, open = -1;
    if (c < c1) {
      const Lag g = lag_geometry(cands[c], H, Lq, Lt);
      const int S = (g.npos + gsz - 1) / gsz;
      const int na = l * S;
      const int nb = (na + S < g.npos) ? na + S : g.npos;
      if (na < nb) {
        const unsigned char* tp = tc + g.i0;
        const unsigned char* qp = qc + g.i0 + g.shift;
        auto sc = [&](int n) -> int { return code_score(score, tp[n], qp[n]); };
        int W = 0;
        for (int m = (na - 46 > 0 ? na - 46 : 0); m < na; ++m) W += sc(m);
        bool prev = (na - 1 >= 46) && W > SXC_WIN_THRESHOLD;
        for (int n = na; n < nb; ++n) {
          W += sc(n);
          if (n >= 46) W -= sc(n - 46);
          const bool on = (n >= 46) && W > SXC_WIN_THRESHOLD;
          if (on && !prev) {
            open = n;
          } else if (!on && prev) {
            if (open >= 0) {
              push(c, open, n);
              open = -1;
            } else if (first_end == INF) {
              first_end = n;
            }
          }
          prev = on;
        }
      }
    }
    summ[2 * tid] = first_end;
    summ[2 * tid + 1] = open;
  });
  ex.sync();
  ex.each([&](int tid) {
    const int c = c0 + tid / gsz;
    const int l = tid % gsz;
    const int open = summ[2 * tid + 1];
    if (c >= c1 || open < 0) return;
    int end = INF;
    const int g0 = tid - l;
    for (int k = l + 1; k < gsz; ++k) {
      const int fe = summ[2 * (g0 + k)];
      if (fe < end) end = fe;
    }
    if (end == INF) end = lag_geometry(cands[c], H, Lq, Lt).npos;  // open where the loop breaks
    push(c, open, end);
  });
  ex.sync();
}

// Two bit planes of 32 bases (bit b: the low and the high bit of base b's 2-bit code).
struct alignas(8) BasePlanes {
  uint32_t lo, hi;
};

// The low half's bits to the even positions, the high half's to the odd ones.
SXC_HD inline uint32_t interleave16(uint32_t v) {
  v = byte_perm(v, v, 0x03010200u);
  uint32_t t = (v ^ (v >> 4)) & 0x00F000F0u;
  v ^= t ^ (t << 4);
  t = (v ^ (v >> 2)) & 0x0C0C0C0Cu;
  v ^= t ^ (t << 2);
  t = (v ^ (v >> 1)) & 0x22222222u;
  return v ^ t ^ (t << 1);
}

SXC_HD inline uint32_t reverse_bits(uint32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bitreverse32(x);
#else
  uint32_t r = 0;
  for (int b = 0; b < 32; ++b) r |= ((x >> b) & 1u) << (31 - b);
  return r;
#endif
}

// Bases [32 w, 32 w + 32) of a chunk of A/C/G/T letters (zeros from len on), read 16 bytes at a
// time: chunks start 16-byte aligned and are padded to whole 16 bytes.
SXC_HD inline BasePlanes planes_of(const unsigned char* seq, int len, int w) {
  struct alignas(16) Quad {
    uint32_t v[4];
  };
  const Quad* p = (const Quad*)seq + 2 * w;
  const int left = len - 32 * w;
  BasePlanes r = {0, 0};
  if (left <= 0) return r;
  const Quad z = {{0, 0, 0, 0}};
  const Quad a = p[0], b = left > 16 ? p[1] : z;
  // code bits 0 and 1 of letter x are x1 ^ x2 and x2 ^ x3; byte i of word j goes to bit 8 i + j
  static_for<0, 8>([&](auto J) {
    constexpr int j = decltype(J)::value;
    const uint32_t v = j < 4 ? a.v[j & 3] : b.v[j & 3];
    const uint32_t y = v ^ (v >> 1);
    r.lo |= ((y >> 1) & 0x01010101u) << j;
    r.hi |= ((y >> 2) & 0x01010101u) << j;
  });
  // bit 8 i + j to bit 4 j + i: the bit's index turned by two places
  const uint32_t keep = left >= 32 ? ~0u : (1u << left) - 1;
  r.lo = interleave16(interleave16(r.lo)) & keep;
  r.hi = interleave16(interleave16(r.hi)) & keep;
  return r;
}

// The same of base codes (class ids 0 to 3 are A/C/G/T), and the bases that are another letter.
SXC_HD inline BasePlanes planes_of_codes(const unsigned char* code, int len, int w, uint32_t& other) {
  const uint32_t* p = (const uint32_t*)code + 8 * w;
  const int left = len - 32 * w;
  BasePlanes r = {0, 0};
  other = 0;
  if (left <= 0) return r;
  static_for<0, 8>([&](auto J) {
    constexpr int j = decltype(J)::value;
    const uint32_t v = p[j];
    r.lo |= (v & 0x01010101u) << j;
    r.hi |= ((v >> 1) & 0x01010101u) << j;
    other |= (((((v >> 2) & 0x3F3F3F3Fu) + 0x3F3F3F3Fu) >> 6) & 0x01010101u) << j;  // bit 6: not 0
  });
  const uint32_t keep = left >= 32 ? ~0u : (1u << left) - 1;
  r.lo = interleave16(interleave16(r.lo)) & keep;
  r.hi = interleave16(interleave16(r.hi)) & keep;
  other = interleave16(interleave16(other)) & keep;
  return r;
}

// 32 bits from base p >= -64 on of a plane that starts two words before base 0
SXC_HD inline uint32_t bits_at(const uint32_t* pl, int p) {
  const uint32_t* w = pl + 2 + (p >> 5);
  return funnel32(w[1], w[0], p & 31);
}

// 32 bases from base p >= -64 on (the planes start two words before base 0)
SXC_HD inline BasePlanes planes_at(const BasePlanes* pl, int p) {
  const BasePlanes* w = pl + 2 + (p >> 5);
  const BasePlanes a = w[0], b = w[1];
  return BasePlanes{funnel32(b.lo, a.lo, p & 31), funnel32(b.hi, a.hi, p & 31)};
}

// Counts over a run of pure A/C/G/T bases: identical positions and C/G bases of each side.  The
// reference's double sums of 0/1 terms equal these counts exactly.
SXC_HD inline void plane_counts(const BasePlanes* tpl, const BasePlanes* qpl, int st, int sq, int len, int& match,
                                int& gct, int& gcq) {
  match = gct = gcq = 0;
  for (int off = 0; off < len; off += 32) {
    const uint32_t keep = len - off < 32 ? (1u << (len - off)) - 1 : ~0u;
    const BasePlanes t = planes_at(tpl, st + off), q = planes_at(qpl, sq + off);
    match += popc64(keep & ~((t.lo ^ q.lo) | (t.hi ^ q.hi)));
    gct += popc64(keep & (t.lo ^ t.hi));  // codes 1 (C), 2 (G)
    gcq += popc64(keep & (q.lo ^ q.hi));
  }
}

// One run through the tail: mode 0 filters it into t_results, mode 1 writes it.
template <int NB, class Ex>
SXC_HD inline void drain_run(Ex& ex, char* sm, const ScanArgs& a, const sxc_pair_dev& pr, const uint16_t* cands, int ps,
                             int rank, int ns, int ne) {
  using SS = ScanSmem<NB>;
  constexpr int H = SS::N / 2;
  const unsigned char* tc = (const unsigned char*)(sm + SS::TCODE);
  const unsigned char* qc = (const unsigned char*)(sm + SS::QCODE);
  const double* equal = (const double*)(sm + SS::EQUAL);
  const double* gcv = (const double*)(sm + SS::GC);
  int* misc = (int*)(sm + SS::MISC);
  const int strand = ps % a.strands;
  const int shift = (int)cands[rank] - H;
  const int i0 = shift < 0 ? -shift : 0;
  const int start_t = i0 + ns - SXC_MIN_LEN;
  const int len = ne - ns + SXC_MIN_LEN;
  const int start_q = start_t + shift;
  const uint64_t key = ((uint64_t)(uint32_t)rank << 32) | (uint32_t)ns;
  if (a.mode == 1) {
    const int slot = a.split > 1 ? ex.atomic_add_global(&a.counts[ps], 1) : ex.atomic_add_shared(&misc[SM_KEPT], 1);
    if (slot >= a.cap) return;
    const size_t at = (size_t)ps * a.cap + slot;
    a.runs[3 * at] = start_t;
    a.runs[3 * at + 1] = start_q;
    a.runs[3 * at + 2] = len;
    a.keys[at] = key;
    return;
  }
  if (len < a.min_len) return;  // FilterMatches: GetLength() < m_minLen
  double ident, prob = 0.;
  if constexpr (SS::HASN) {
    int cm, nk, ct, ntn, cq, nqn;
    packed_counts_n((const uint32_t*)(sm + SS::TPK), (const uint32_t*)(sm + SS::QPK),
                    (const uint32_t*)(sm + SS::TNK), (const uint32_t*)(sm + SS::QNK), start_t, start_q, len, cm,
                    nk, ct, ntn, cq, nqn);
    // DNA_Equal of N against any base or N, and N's GC weight, are quarter multiples, so
    // the reference's running sums equal these products exactly
    const double matches = (double)cm + a.tab->equal[SXC_CLASS_N][0] * (double)nk;
    const double gct = (double)ct + a.tab->gc[SXC_CLASS_N] * (double)ntn;
    const double gcq = (double)cq + a.tab->gc[SXC_CLASS_N] * (double)nqn;
    if (a.ptable) {
      prob = table_from_sums(matches, gct, gcq, len, a.ptable, a.table_prob, ident);
    } else if ((nk == 0 && z_clearly_skipped(cm, ct, cq, len, a.z_skip)) ||
               !tail_from_sums(matches, gct, gcq, len, a.target_total, a.z_skip, prob, ident)) {
      return;
    }
  } else if constexpr (SS::PURE) {
    int cm, ct, cq;
    plane_counts((const BasePlanes*)(sm + SS::TPL), (const BasePlanes*)(sm + SS::QPL), start_t, start_q, len, cm, ct,
                 cq);
    if (a.ptable) {
      prob = table_from_sums((double)cm, (double)ct, (double)cq, len, a.ptable, a.table_prob, ident);
    } else if (z_clearly_skipped(cm, ct, cq, len, a.z_skip) ||
               !tail_from_sums((double)cm, (double)ct, (double)cq, len, a.target_total, a.z_skip, prob, ident)) {
      return;
    }
  } else {
    double matches = 0, gct = 0, gcq = 0;
    for (int i = 0; i < len; ++i) {
      const int ca = code_class(tc[start_t + i]), cb = code_class(qc[start_q + i]);
      matches += equal[ca * SXC_NCLASS + cb];
      gct += gcv[ca];
      gcq += gcv[cb];
    }
    if (a.ptable) {
      prob = table_from_sums(matches, gct, gcq, len, a.ptable, a.table_prob, ident);
    } else if (!tail_from_sums(matches, gct, gcq, len, a.target_total, a.z_skip, prob, ident)) {
      return;
    }
  }
  // FilterMatches keeps prob >= m_minProb.  The table's decision is exact; the device's
  // erf/exp may differ from glibc's by a few ulp, so a probability within the keep band
  // of min_prob is written flagged and decided on the host with glibc.
  bool near = false;
  if (a.ptable) {
    if (prob < a.min_prob) return;
  } else {
    if (prob < a.keep_lo) return;
    near = prob < a.flag_hi;
  }
  const int slot = a.split > 1 ? ex.atomic_add_global(&a.counts[ps], 1) : ex.atomic_add_shared(&misc[SM_KEPT], 1);
  if (slot >= a.cap) return;
  const int tstart = pr.t_chunk_start + start_t;
  // RCQuery (analysis/HomologyByXCorrSlave.cc:56-60) on the reverse strand, with the
  // -q_chunk size (slave) or, for q_chunk == 0, the query chunk's own length (the
  // standalone aligner, tools/analysis/HomologyByXCorr.cc:226-228, 793-798)
  const int rc_chunk = a.q_chunk > 0 ? a.q_chunk : a.qchunks[pr.q_chunk].len;
  const int qstart =
      strand == 0 ? pr.q_chunk_start + start_q : start_q + pr.q_record_len - pr.q_chunk_start - rc_chunk;
  sxc_result_dev r;
  r.query_id = (uint64_t)(int64_t)pr.q_record;
  r.target_id = (uint64_t)(int64_t)pr.t_record;
  r.query_size = (uint64_t)(int64_t)pr.q_record_len;
  r.qstart = (uint64_t)(int64_t)qstart;
  r.tstart = (uint64_t)(int64_t)tstart;
  r.len = (uint64_t)(int64_t)len;
  r.reverse = (uint8_t)(strand == 1);
  for (int z = 0; z < 7; ++z) r.pad_[z] = 0;
  if (near) {
    const uint32_t pi = (uint32_t)(ps / a.strands);  // the pair, for the host's decision
    r.pad_[0] = SXC_REC_NEAR;
    r.pad_[1] = (uint8_t)pi;
    r.pad_[2] = (uint8_t)(pi >> 8);
    r.pad_[3] = (uint8_t)(pi >> 16);
    r.pad_[4] = (uint8_t)(pi >> 24);
    if (a.nflag) ex.atomic_add_global(a.nflag, 1);
  }
  r.prob = prob;
  r.ident = ident;
  const size_t at = (size_t)ps * a.cap + slot;
  a.out[at] = r;
  a.keys[at] = key;
}

// Drains queue entries [0, n): mode 0 filters into t_results, mode 1 writes runs.
// rank_base: the first lag of the epoch the entries come from (compact queue).
template <int NB, class Ex>
SXC_HD inline void drain(Ex& ex, char* sm, const ScanArgs& a, const sxc_pair_dev& pr, const uint16_t* cands, int ps,
                         int n, int rank_base) {
  using SS = ScanSmem<NB>;
  const int* queue = (const int*)(sm + SS::QUEUE);
  ex.each([&](int tid) {
    for (int k = tid; k < n; k += SCAN_NT) {
      int rank, ns, ne;
      if constexpr (SS::COMPACT) {
        const unsigned v = (unsigned)queue[k];
        rank = rank_base + (int)(v & ((1u << SS::RB) - 1));
        ns = (int)((v >> SS::RB) & ((1u << SS::NSB) - 1));
        ne = (int)(v >> (SS::RB + SS::NSB));
      } else {
        rank = queue[2 * k];
        ns = queue[2 * k + 1] & 0xffff;
        ne = (queue[2 * k + 1] >> 16) & 0xffff;
      }
      drain_run<NB>(ex, sm, a, pr, cands, ps, rank, ns, ne);
    }
  });
  ex.sync();
}

// ---- pairs of pure A/C/G/T chunks: 32 blocks of a lag in the bits of a word (scan_sliced)

// Bit i of word j becomes bit j of word i.
SXC_HD inline void transpose32(uint32_t* x) {
  static_for<0, 16>([&](auto K) {
    constexpr int k = decltype(K)::value;
    const uint32_t p = x[k], q = x[k + 16];
    x[k] = byte_perm(q, p, 0x05040100u);
    x[k + 16] = byte_perm(q, p, 0x07060302u);
    if constexpr (k % 4 == 3) keep_order();
  });
  static_for<0, 16>([&](auto K) {
    constexpr int k = (decltype(K)::value & 7) | ((decltype(K)::value & 8) << 1);
    const uint32_t p = x[k], q = x[k + 8];
    x[k] = byte_perm(q, p, 0x06020400u);
    x[k + 8] = byte_perm(q, p, 0x07030501u);
    if constexpr (decltype(K)::value % 4 == 3) keep_order();
  });
  auto stage = [&](auto S, uint32_t low) {
    constexpr int s = decltype(S)::value;
    static_for<0, 16>([&](auto K) {
      constexpr int k = (decltype(K)::value & (s - 1)) | ((decltype(K)::value & ~(s - 1)) << 1);
      const uint32_t p = x[k], q = x[k + s];
      x[k] = bit_select(low, p, q << s);
      x[k + s] = bit_select(low, p >> s, q);
      opaque(x[k]);  // (else the masked halves are kept apart for the next stage, and spilled)
      opaque(x[k + s]);
      if constexpr (decltype(K)::value % 4 == 3) keep_order();
    });
  };
  stage(std::integral_constant<int, 4>{}, 0x0F0F0F0Fu);
  stage(std::integral_constant<int, 2>{}, 0x33333333u);
  stage(std::integral_constant<int, 1>{}, 0x55555555u);
}

// s + 2 c = x + y + z in every bit position
SXC_HD inline void add3(uint32_t x, uint32_t y, uint32_t z, uint32_t& s, uint32_t& c) {
  s = x ^ y ^ z;
  c = (x & y) | (z & (x | y));
}

// The sum of x[0 .. 7] in every bit position: digits s[0 .. 3].
SXC_HD inline void sum8(const uint32_t* x, uint32_t* s) {
  uint32_t a, A, b, B, c, C, D, e, E, F;
  add3(x[0], x[1], x[2], a, A);
  add3(x[3], x[4], x[5], b, B);
  add3(x[6], x[7], a, c, C);
  s[0] = b ^ c;
  D = b & c;
  add3(A, B, C, e, E);
  s[1] = e ^ D;
  F = e & D;
  s[2] = E ^ F;
  s[3] = E & F;
}

// r = x + y over W digits (what does not fit is known to be zero)
template <int W>
SXC_HD inline void sum_digits(const uint32_t* x, const uint32_t* y, uint32_t* r) {
  uint32_t carry = 0;
  static_for<0, W>([&](auto I) {
    constexpr int i = decltype(I)::value;
    uint32_t s, c;
    add3(x[i], y[i], carry, s, c);
    r[i] = s;
    carry = c;
  });
}

// The scan's gate: flags set that many times in a row name a block.
SXC_HD inline int scan_gate(int min_run) { return min_run >= 8 ? 8 : min_run >= 4 ? 4 : min_run >= 2 ? 2 : 1; }

// Whether slices pay for a general pair's `lags` (else segments).  What slices save on most blocks they
// lose on the named ones, found again position by position, by table lookups where the windows hold
// another letter.  How many are named follows from the gate and from how often a base of one chunk
// equals one of the other (by their counts).  The limits are where both took the same time, fitted to
// 1300 measured launches (0 to 6 such letters in 1000, G/C 0.2 to 0.5, N = 512 to 32768, 8 to 4000
// strands); never with another letter in more than one word (32 bases) in 8.  ms sliced and by segments,
// gates 1, 4 and 8, one such letter in the target / 2 / 6 in 1000:
//   512 strands of 16384 bases, G/C 0.41 (equal 0.258): 15.6 7.4 4.8 and 34.8 32.6 32.1 / 24.8 14.5 9.9 and
//   34.2 32.2 31.7 / 30.9 18.9 14.2 and 33.8 31.7 31.4; 0.35 (0.273): 26.5 11.2 7.0 and 36.9 33.3 32.6 / 42.1
//   22.6 15.5 and 36.8 33.3 32.6 / 49.9 31.6 22.6 and 37.2 33.8 33.2; 0.25 (0.313): 64.7 33.2 22.3 and 47.8 40.0
//   36.9 / 100.2 60.2 44.1 and 47.4 39.8 36.8 / 122 78.5 58.1 and 47.8 40.4 37.4;
//   4000 strands of 2048 bases, whose segments are the fastest: 0.41: 1.19 0.81 0.68 and 1.64 1.45 1.43 / 1.52
//   1.11 0.89 and 1.63 1.43 1.42; 0.35: 1.79 0.99 0.78 and 1.74 1.51 1.45; 0.25: 3.70 2.30 1.70 and 2.26 1.91 1.72.
// A share of few blocks leaves most threads of a slice idle: 8 strands in 16 shares, G/C 0.41, gate 1, us:
// 256 bases (about 80 blocks) 104 and 38, 512 (330) 133 and 68, 2048 (420) 179 and 119, 1024 (1300) 142 and 156,
// 4096 (2300) 209 and 322.
SXC_HD inline bool slices_pay(const int* misc, int log_n, int gate, int split, int lags) {
  const float lt = (float)misc[SM_LT], lq = (float)misc[SM_LQ];
  const float wt = (float)(misc[SM_AMB] & 0xffff), wq = (float)(misc[SM_AMB] >> 16);
  if (8.f * 32.f * (wt + wq) > lt + lq) return false;
  const int shorter = misc[SM_LT] < misc[SM_LQ] ? misc[SM_LT] : misc[SM_LQ];
  if (split > 1 && lags * (shorter >> 5) < (log_n == 12 ? 1400 : 800)) return false;
  float equal = 0.f;
  for (int k = 0; k < 4; ++k) {
    const unsigned t = (unsigned)misc[SM_BASES + k / 2], q = (unsigned)misc[SM_BASES + 2 + k / 2];
    equal += (float)((k & 1) ? t >> 16 : t & 0xffffu) * (float)((k & 1) ? q >> 16 : q & 0xffffu);
  }
  // the share of blocks with another letter in their windows, which span three words
  const float dirty = fminf(96.f * (wt / lt + wq / lq), 0.6f);
  const float limit = gate == 8 ? 0.320f : gate == 4 ? 0.315f : gate == 2 ? 0.295f : 0.283f;
  const float slope = (log_n <= 11 ? 0.01f : log_n == 12 ? 0.035f : 0.04f) * (gate >= 4 ? 1.8f : gate == 2 ? 1.3f : 1.f);
  return equal <= (limit - slope * dirty - (log_n == 12 ? 0.018f : 0.f)) * lt * lq;
}
constexpr int SLICE_LAGS = 512;    // lags staged at a time
constexpr int SLICE_BLOCKS = 29;   // blocks a slice decides (of the 32 it computes)

// Slice t of a lag: bit b of a word stands for block 29 t + b - 2.  Bits 0 and 1 are the windows'
// history, bit 2 the flags before the slice; bits 3 to 31 are the blocks the slice decides (block 0
// has no flags, DoOne's test begins at n = 46).  Returns the blocks holding a position where the
// flags have been set `gate` times in a row (d2, d4, d8: ~0 where the gate is below 2, 4, 8), and
// in block 1 also a run that starts at 46; *rises counts the runs that start in the blocks.
// AMB: a position with another letter (planes tam, qam) counts as identical, which it scores at
// most.  Flags are then set where they may be, so a run may start later than the flags do: every
// block where they have been set often enough is named; blocks whose windows hold another
// letter are left out of *rises and named if any flag is set (with `count`).
template <bool AMB>
SXC_HD inline uint32_t slice_blocks(const BasePlanes* tpl, const BasePlanes* qpl, const uint32_t* tam,
                                    const uint32_t* qam, const Lag& g, int t, uint32_t d2, uint32_t d4, uint32_t d8,
                                    bool count, int* rises) {
  // x[i] bit b: position i of block b differs (words of the planes are offset by two blocks)
  uint32_t x[32];
  uint32_t dirty = 0;  // blocks with another letter in their windows
  {
    const int qj = g.i0 + g.shift;
    const int tb = g.i0 & 31, qb = qj & 31;
    const BasePlanes* tw = tpl + (g.i0 >> 5) + SLICE_BLOCKS * t;
    const BasePlanes* qw = qpl + (qj >> 5) + SLICE_BLOCKS * t;
    BasePlanes t0 = tw[0], q0 = qw[0];
    static_for<0, 32>([&](auto B) {
      constexpr int b = decltype(B)::value;
      const BasePlanes t1 = tw[b + 1], q1 = qw[b + 1];
      x[b] = (funnel32(t1.lo, t0.lo, tb) ^ funnel32(q1.lo, q0.lo, qb)) |
             (funnel32(t1.hi, t0.hi, tb) ^ funnel32(q1.hi, q0.hi, qb));
      t0 = t1;
      q0 = q1;
      if constexpr (AMB) {
        const int at = SLICE_BLOCKS * t + b;
        const uint32_t *ta = tam + (g.i0 >> 5) + at, *qa = qam + (qj >> 5) + at;
        const uint32_t other = funnel32(ta[1], ta[0], tb) | funnel32(qa[1], qa[0], qb);
        x[b] &= ~other;
        dirty |= (other ? 1u : 0u) << b;
      }
      if constexpr (b % 4 == 3) keep_order();
    });
    if (AMB && t == 0) dirty &= ~3u;  // before the lag
    dirty |= (dirty << 1) | (dirty << 2);
  }
  transpose32(x);
  keep_order();
  // c: differences among the 46 positions before the block, plus 4: all 32 of the block before and
  // the last 14 of the one before that.  At most 27 differences <=> bit 5 of the sum is clear.
  uint32_t c[6];
  {
    uint32_t p[6] = {}, q[6] = {}, r[6] = {}, last[6] = {}, first[6] = {}, all[6];
    sum8(x + 18, p);
    keep_order();
    const uint32_t rest[8] = {x[26], x[27], x[28], x[29], x[30], x[31], 0u, 0u};
    sum8(rest, q);
    sum_digits<4>(p, q, last);  // <= 14
    keep_order();
    sum8(x, p);
    sum8(x + 8, q);
    sum_digits<5>(p, q, r);
    keep_order();
    uint32_t two[6] = {x[16] ^ x[17], x[16] & x[17], 0u, 0u, 0u, 0u};
    sum_digits<5>(r, two, first);  // <= 18
    sum_digits<6>(first, last, all);
    uint32_t carry = 0;
    static_for<0, 6>([&](auto I) {
      constexpr int i = decltype(I)::value;
      uint32_t s, cy;
      add3(all[i] << 1, last[i] << 2, carry, s, cy);
      c[i] = s;
      carry = cy;
    });
    uint32_t four = c[2];  // + 4
    c[2] = ~c[2];
    static_for<3, 6>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const uint32_t s = c[i] ^ four;
      four = c[i] & four;
      c[i] = s;
    });
    keep_order();
  }
  // blocks with n = 32 block + i inside the lag: ha up to i = e, hb after it
  const int last = (g.npos - 1) >> 5, e = (g.npos - 1) & 31;
  const int nb = last + 3 - SLICE_BLOCKS * t;
  const uint32_t ha = nb >= 32 ? ~0u : (1u << nb) - 1;
  const uint32_t hb = nb - 1 >= 32 ? ~0u : (1u << (nb - 1)) - 1;
  const uint32_t la = t ? ~3u : ~15u, lb = t ? ~3u : ~7u;  // flags from n = 46; bits 0, 1 have no history
  uint32_t any = 0, wrapped = 0, at46 = 0;
  uint32_t runs = 0, set = 0;
  uint32_t f[40], r2[40], r4[40], r8[40];
  auto gates = [&](auto I) {
    constexpr int i = decltype(I)::value;
    r2[i] = f[i] & ((i >= 1 ? f[i >= 1 ? i - 1 : 0] : 0u) | d2);
    r4[i] = r2[i] & ((i >= 2 ? r2[i >= 2 ? i - 2 : 0] : 0u) | d4);
    r8[i] = r4[i] & ((i >= 4 ? r4[i >= 4 ? i - 4 : 0] : 0u) | d8);
  };
  static_for<0, 32>([&](auto I) {
    constexpr int i = decltype(I)::value;
    // the count moves up where position n differs and n - 46 does not, down for the opposite
    const uint32_t old = i < 14 ? x[(i + 18) & 31] << 2 : x[(i - 14) & 31] << 1;
    uint32_t m = x[i] ^ old;
    static_for<0, 6>([&](auto J) {
      constexpr int j = decltype(J)::value;
      const uint32_t next = m & (c[j] ^ old);
      c[j] ^= m;
      m = next;
    });
    f[i] = ~c[5] & (i <= e ? ha : hb) & (i < 14 ? la : lb);
    gates(I);
    if constexpr (i >= 1) {
      runs += __builtin_popcount(f[i] & ~f[i - 1] & ~7u & ~dirty);
      opaque(runs);  // (one add per count)
    }
    if constexpr (i >= 8) any |= AMB ? r8[i] : r8[i] & ~r8[i - 1];
    if constexpr (AMB) set |= f[i];
    if constexpr (i == 14) at46 = t ? 0u : f[i] & 8u;
    keep_order();
  });
  // the first positions of the next block follow the last of this one
  static_for<32, 40>([&](auto I) {
    constexpr int i = decltype(I)::value;
    f[i] = f[i - 32] >> 1;
    gates(I);
    if constexpr (i == 32) runs += __builtin_popcount(f[i] & ~f[i - 1] & ~3u & ~(dirty >> 1));
    wrapped |= AMB ? r8[i] : r8[i] & ~r8[i - 1];
  });
  *rises = (int)runs;
  any = (any & ~7u) | ((wrapped & ~3u) << 1) | at46;
  if constexpr (AMB) any |= count ? set & dirty & ~7u : 0u;
  return any;
}

// The runs of block k of lag `rank` that were set `gate` times in a row for the first time inside
// the block, found again position by position, and their tails.  AMB: returns the runs that start
// in the block if its windows hold another letter (see slice_blocks).
template <int NB, class Ex>
SXC_HD inline int slice_runs(Ex& ex, char* sm, const ScanArgs& a, const sxc_pair_dev& pr, const uint16_t* cands,
                             int ps, int rank, const Lag& g, int k, int gate, int min_run) {
  using SS = ScanSmem<NB>;
  const BasePlanes* tpl = (const BasePlanes*)(sm + SS::TPL);
  const BasePlanes* qpl = (const BasePlanes*)(sm + SS::QPL);
  auto match = [&](int b) {  // of block b >= -2
    const BasePlanes t = planes_at(tpl, g.i0 + 32 * b), q = planes_at(qpl, g.i0 + g.shift + 32 * b);
    return ~((t.lo ^ q.lo) | (t.hi ^ q.hi));
  };
  const int s = k - 1;  // k >= 1
  // another letter in block b (AMB)
  auto other = [&](int b) {
    if constexpr (!SS::AMB) return 0u;
    return b < 0 ? 0u : bits_at((const uint32_t*)(sm + SS::TAM), g.i0 + 32 * b) |
                            bits_at((const uint32_t*)(sm + SS::QAM), g.i0 + g.shift + 32 * b);
  };
  uint32_t m2 = s < 2 ? 0u : match(s - 2), m1 = s < 1 ? 0u : match(s - 1);
  uint32_t o2 = other(s - 2), o1 = other(s - 1);
  // score of position n by the tables (AMB), and of the window before block b
  auto score_at = [&](int n) {
    return code_score((const unsigned char*)(sm + SS::SCORE), (unsigned char)sm[SS::TCODE + g.i0 + n],
                      (unsigned char)sm[SS::QCODE + g.i0 + g.shift + n]);
  };
  auto window_before = [&](int b) {
    if (!SS::AMB || !(o1 | o2)) return 100 * (popc64(m1) + popc64(m2 >> 18));
    int W = 0;
    for (int n = 32 * b < 46 ? 0 : 32 * b - 46; n < 32 * b; ++n) W += score_at(n);
    return W;
  };
  const uint32_t prev = (32 * s - 1 >= 46 && window_before(s) > SXC_WIN_THRESHOLD) ? 1u : 0u;
  bool dirty = false;  // of the block next_flags has seen last,
  int carried = -1;    // and its last window's score, if so
  // flags of the next block, b (DoOne's positions only: 46 <= n < npos)
  auto next_flags = [&](int b) {
    const uint32_t m0 = match(b), o0 = other(b);
    uint32_t f = 0;
    dirty = (o0 | o1 | o2) != 0;
    if (!dirty) {
      carried = -1;
      const uint32_t old = funnel32(m1, m2, 18);  // m(n - 46)
      // 2-bit group r: m(n) + 1 - m(n - 46)
      const uint32_t one = ~(m0 ^ old), two = m0 & ~old;
      const int C = popc64(m1) + popc64(m2 >> 18);
      uint32_t ub = byte_perm(0u, (uint32_t)(C + 128 - SXC_MIN_MATCHES), 0u);  // half_flags' u, every byte
      f = window_flags(interleave16(byte_perm(two, one, 0x05040100u)),
                       interleave16(byte_perm(two, one, 0x07060302u)), ub);
      if (b < 2) f &= b == 0 ? 0u : 0xFFFFC000u;
      if (g.npos - 32 * b < 32) f &= g.npos > 32 * b ? (1u << (g.npos - 32 * b)) - 1 : 0u;
    } else {
      int W = carried >= 0 ? carried : window_before(b);
      for (int n = 32 * b; n < 32 * b + 32 && n < g.npos; ++n) {
        W += score_at(n);
        if (n >= 46) {
          W -= score_at(n - 46);
          f |= (W > SXC_WIN_THRESHOLD ? 1u : 0u) << (n & 31);
        }
      }
      carried = W;
    }
    m2 = m1;
    m1 = m0;
    o2 = o1;
    o1 = o0;
    return f;
  };
  const uint32_t f0 = next_flags(s);
  const uint64_t f = (uint64_t)f0 | ((uint64_t)next_flags(k) << 32);
  uint64_t rises = f & ~((f << 1) | prev);
  const int starts = SS::AMB && dirty ? popc64(rises >> 32) : 0;
  rises &= 0xFFFFFFFFull << (33 - gate);
  for (;;) {
    // the next run that is long enough or still open: found by all lanes before any takes a tail
    int ns = -1, ne = g.npos;
    bool open = false;
    while (ns < 0 && rises) {
      const int r = __builtin_ctzll(rises);
      rises &= rises - 1;
      const uint64_t clear = ~f & (~0ull << r);
      open = !clear;  // (the last run of the two blocks)
      if (clear) ne = 32 * s + __builtin_ctzll(clear);
      // Too short to be kept (keep_min_run).  A run that starts at 46, where DoOne's test begins,
      // may have been above the threshold before, so the bound does not hold for it.
      ns = 32 * s + r;
      if (clear && ne - ns < min_run && ns != 46) ns = -1;
    }
    if (ns < 0) return starts;
    if (open) {
      ne = g.npos;
      for (int b = k + 1; 32 * b < g.npos; ++b) {
        const uint32_t fb = next_flags(b);
        if (~fb) {
          ne = 32 * b + __builtin_ctz(~fb);
          break;
        }
      }
      if (ne - ns < min_run && ns != 46) return starts;
    }
    drain_run<NB>(ex, sm, a, pr, cands, ps, rank, ns, ne);
  }
}

// Pure A/C/G/T lags [lo, hi).  Score = 100 * [match], and a window sum > 1889 <=> >= 19 matches,
// <=> <= 27 differences.  C(n) = C(n - 1) + m(n) - m(n - 46) with m(< 0) = 0 equals the reference's
// running `match` (analysis/CrossCorr.cc:700-705).  A thread takes a slice of a lag, 32 blocks of
// 32 positions, and transposes their difference words, so that one operation moves the 32 blocks'
// counts by one position each; blocks with a run that may be kept (or any run, where all are
// wanted) go to a queue, whose entries all threads take through slice_runs.
// Vector issue bounds it: a slice takes some 1600 instructions (about 190 for the difference
// words, 260 for the transposition, 130 for the first counts, 30 per position), 55 per block of 32
// positions against 110 to 120 where a thread took one block at a time and 150 more before its
// first, and 32 blocks share one start.  306 M instructions for 8192 strands at N = 8192 take
// 0.507 ms, all of the chip's issue rate: the slices 0.28, the named blocks about 0.2.  One launch, before (a block at a time) and now: 8192 strands at
// N = 8192 0.80 and 0.51 ms, 24000 at 2048 3.59 and 1.46 ms, 40000 at 512 1.19 and 0.64 ms, 1000
// at 32768 1.96 and 0.75 ms.
template <int NB, class Ex>
SXC_HD inline void scan_sliced(Ex& ex, char* sm, const ScanArgs& a, const sxc_pair_dev& pr, const uint16_t* cands,
                               int ps, int lo, int hi, int min_run) {
  using SS = ScanSmem<NB>;
  constexpr int H = SS::N / 2;
  constexpr int SLICES = (SS::WPL - 1 + SLICE_BLOCKS - 1) / SLICE_BLOCKS;
  static_assert(SLICES >= 1 && SLICES <= 32, "slices of a lag");
  constexpr int QCAP = SS::SQCAP;
  static_assert(32 * SLICE_BLOCKS <= QCAP, "32 slices' blocks fit the queue");
  int* misc = (int*)(sm + SS::MISC);
  int* queue = (int*)(sm + SS::QUEUE);
  uint16_t* lags = (uint16_t*)(sm + SS::LAGS);
  int* first = (int*)(sm + SS::RANGE);  // of slice t: its first lag
  int* many = first + 32;               // and how many lags have one
  int* runs = (int*)(sm + SS::RUNS);
  const BasePlanes* tpl = (const BasePlanes*)(sm + SS::TPL);
  const BasePlanes* qpl = (const BasePlanes*)(sm + SS::QPL);
  const uint32_t* tam = (const uint32_t*)(sm + SS::TAM);
  const uint32_t* qam = (const uint32_t*)(sm + SS::QAM);
  const int Lt = misc[SM_LT], Lq = misc[SM_LQ];
  const int gate = scan_gate(min_run);
  const uint32_t d2 = gate >= 2 ? 0u : ~0u, d4 = gate >= 4 ? 0u : ~0u, d8 = gate >= 8 ? 0u : ~0u;
  ex.each([&](int tid) { runs[tid] = 0; });
  for (int c0 = lo; c0 < hi; c0 += SLICE_LAGS) {
    const int nl = (hi - c0 < SLICE_LAGS) ? hi - c0 : SLICE_LAGS;
    ex.each([&](int tid) {
      for (int x = tid; x < nl; x += SCAN_NT) lags[x] = cands[c0 + x];
    });
    ex.sync();
    // A lag has a slice t if npos >= P, which holds for an interval of shifts (npos is concave in
    // the shift), and FindTop's lags ascend.
    ex.each([&](int tid) {
      if (tid >= SLICES) return;
      const int P = 32 * (SLICE_BLOCKS * tid + 1) + 1;
      auto below = [&](int idx) {  // lags before idx
        int u = 0, v = nl;
        while (u < v) {
          const int w = (u + v) >> 1;
          if ((int)lags[w] < idx) {
            u = w + 1;
          } else {
            v = w;
          }
        }
        return u;
      };
      const int x0 = below(H + P - Lt + 1);
      int x1 = below(H + Lq - P + 1);
      if (P > Lq || P > Lt - 1 || x1 < x0) x1 = x0;
      first[tid] = x0;
      many[tid] = x1 - x0;
    });
    ex.sync();
    int total = 0;
    for (int t = 0; t < SLICES; ++t) total += many[t];
    // Blocks queued before the current slices, kept per thread: every thread must see the same
    // count.  Slices whose blocks overflow the queue are scanned again, 32 at a time, whose blocks
    // always fit an empty one; their runs are counted the first time (slices below `counted`).
    int queued = 0, width = SCAN_NT, counted = 0;
    for (int base = 0; base < total;) {
      ex.each([&](int tid) {
        int id = base + tid;
        if (tid >= width || id >= total) return;
        const bool count = id >= counted;
        int t = 0;
        while (id >= many[t]) id -= many[t++];
        id += first[t];
        const Lag g = lag_geometry(lags[id], H, Lq, Lt);
        int rises;
        uint32_t any = slice_blocks<SS::AMB>(tpl, qpl, tam, qam, g, t, d2, d4, d8, a.stats != nullptr, &rises);
        runs[tid] += count ? rises : 0;
        while (any) {
          const int b = __builtin_ctz(any);
          any &= any - 1;
          const int at = ex.atomic_add_shared(&misc[SM_QN], 1);  // (one atomic per wave)
          if (at < QCAP) queue[at] = id | (SLICE_BLOCKS * t + b - 2) << 9;
        }
      });
      ex.sync();
      const int qn = misc[SM_QN];
      ex.sync();  // every thread has read the count
      const bool over = qn > QCAP;
      if (over) {
        if (counted < base + width) counted = base + width;
        width = 32;
      } else {
        base += width;
        if (base >= counted) width = SCAN_NT;
      }
      if (!over && qn <= QCAP / 2 && base < total) {
        queued = qn;
        continue;
      }
      const int n = over ? queued : qn;
      ex.each([&](int tid) {
        for (int x = tid; x < n; x += SCAN_NT) {
          const int id = queue[x] & (SLICE_LAGS - 1), k = queue[x] >> 9;
          runs[tid] +=
              slice_runs<NB>(ex, sm, a, pr, cands, ps, c0 + id, lag_geometry(lags[id], H, Lq, Lt), k, gate, min_run);
        }
      });
      ex.sync();
      ex.each([&](int tid) {
        if (tid == 0) misc[SM_QN] = 0;
      });
      ex.sync();
      queued = 0;
    }
  }
  ex.each([&](int tid) {
    if (a.stats) ex.atomic_add_shared(&misc[SM_RUNS], runs[tid]);
  });
  ex.sync();
}

template <int NB, class Ex>
SXC_HD inline void scan_body(Ex& ex, char* sm, const ScanArgs& a, int blk) {
  using SS = ScanSmem<NB>;
  constexpr int N = SS::N;
  const int split = a.split > 1 ? a.split : 1;
  const int ps = a.list ? a.list[blk / split] : blk / split, part = blk % split;
  const sxc_pair_dev pr = a.pairs[ps / a.strands];
  const int strand = ps % a.strands;
  const sxc_chunk tch = a.tchunks[pr.t_chunk];
  const sxc_chunk qch = a.qchunks[pr.q_chunk];
  // each kernel takes its own kind only, whatever it is launched over
  if (scan_kind(tch.flags, qch.flags) != (SS::SLICED ? SCAN_PURE : SS::HASN ? SCAN_N : SCAN_GENERAL)) return;
  const sxc_tables* tab = a.tab;
  unsigned char* tc = (unsigned char*)(sm + SS::TCODE);
  unsigned char* qc = (unsigned char*)(sm + SS::QCODE);
  double* equal = (double*)(sm + SS::EQUAL);
  double* gcv = (double*)(sm + SS::GC);
  unsigned char* score = (unsigned char*)(sm + SS::SCORE);
  int* misc = (int*)(sm + SS::MISC);
  const unsigned char* ts = a.seq + tch.off;
  const unsigned char* qs = a.seq + qch.off;
  const uint16_t* gcands = a.cands + (size_t)ps * N;
  unsigned char* cls = (unsigned char*)(sm + SS::CLS);
  unsigned char* rc = (unsigned char*)(sm + SS::RC);
  // the general kernel stages the chunk bytes (16-byte aligned in HBM) and the tables in LDS
  ex.each([&](int tid) {
    if constexpr (!SS::PURE) {
      const uint32_t* ts4 = (const uint32_t*)ts;
      const uint32_t* qs4 = (const uint32_t*)qs;
      uint32_t* tc4 = (uint32_t*)tc;
      uint32_t* qc4 = (uint32_t*)qc;
      for (int i = tid; i < (tch.len + 3) / 4; i += SCAN_NT) tc4[i] = ts4[i];
      for (int i = tid; i < (qch.len + 3) / 4; i += SCAN_NT) qc4[i] = qs4[i];
      for (int i = tid; i < SXC_NCLASS * SXC_NCLASS; i += SCAN_NT) {
        equal[i] = (&tab->equal[0][0])[i];
        score[i] = (&tab->score[0][0])[i];
      }
      for (int i = tid; i < SXC_NCLASS; i += SCAN_NT) gcv[i] = tab->gc[i];
      if (tid < 5 * 32) ((int*)(sm + SS::RUNS))[tid] = 0;
      for (int i = tid; i < 128; i += SCAN_NT) {
        cls[i] = tab->cls[i];
        rc[i] = tab->rc[i];
      }
    }
    if (tid == 0) {
      misc[SM_QN] = 0;
      misc[SM_NRB] = 0;
      misc[SM_KEPT] = 0;
      misc[SM_RUNS] = 0;
      misc[SM_NCAND] = a.ncand[ps];
      misc[SM_LT] = tch.len;
      misc[SM_LQ] = qch.len;
    }
  });
  ex.sync();
  const int Lt = tch.len, Lq = qch.len;
  if constexpr (SS::SLICED) {
    // 2-bit codes A=0, C=1, G=2, T=3 from the ASCII letters (read from HBM); complement =
    // code ^ 3.  Strand 1 (DNAVector::ReverseComplement, analysis/DNAVector.cc:482-521) turns the
    // query's planes around.
    BasePlanes* tpl = (BasePlanes*)(sm + SS::TPL);
    BasePlanes* qpl = (BasePlanes*)(sm + SS::QPL);
    ex.each([&](int tid) {
      for (int w = tid; w < SS::PLW; w += SCAN_NT) {
        const BasePlanes none = {0, 0};
        const bool in = w >= 2 && w < 2 + N / 32;
        tpl[w] = in ? planes_of(ts, Lt, w - 2) : none;
        qpl[w] = in ? planes_of(qs, Lq, w - 2) : none;
      }
    });
    ex.sync();
    if (strand) {
      BasePlanes* rpl = (BasePlanes*)(sm + SS::RPL);
      ex.each([&](int tid) {
        for (int w = tid; w < N / 32; w += SCAN_NT) {
          const int p = Lq - 32 - 32 * w;  // first base of the word, reversed
          BasePlanes r = {0, 0};
          if (p > -32) {
            const BasePlanes v = planes_at(qpl, p);
            const uint32_t keep = p >= 0 ? ~0u : (1u << (32 + p)) - 1;
            r.lo = ~reverse_bits(v.lo) & keep;
            r.hi = ~reverse_bits(v.hi) & keep;
          }
          rpl[w] = r;
        }
      });
      ex.sync();
      ex.each([&](int tid) {
        for (int w = tid; w < N / 32; w += SCAN_NT) qpl[w + 2] = rpl[w];
      });
      ex.sync();
    }
  } else if constexpr (SS::PURE) {
    // 2-bit codes A=0, C=1, G=2, T=3 from the ASCII letters (read from HBM); complement =
    // code ^ 3
    uint32_t* tpk = (uint32_t*)(sm + SS::TPK);
    uint32_t* qpk = (uint32_t*)(sm + SS::QPK);
    ex.each([&](int tid) {
      for (int w = tid; w < SS::PKW; w += SCAN_NT) {
        uint32_t vt = 0, vq = 0, nt = 0, nq = 0;
        for (int b = 0; b < 16; ++b) {
          const int i = 16 * w + b;
          if (i < Lt) {
            const unsigned x = ts[i];
            vt |= (((x >> 1) ^ (x >> 2)) & 3u) << (2 * b);
            nt |= (x == 'N' ? 1u : 0u) << (2 * b);
          }
          if (i < Lq) {
            // DNAVector::ReverseComplement for strand 1 (analysis/DNAVector.cc:482-521);
            // the complement of N is N
            const unsigned x = strand ? qs[Lq - 1 - i] : qs[i];
            vq |= ((((x >> 1) ^ (x >> 2)) & 3u) ^ (strand ? 3u : 0u)) << (2 * b);
            nq |= (x == 'N' ? 1u : 0u) << (2 * b);
          }
        }
        tpk[w] = vt;
        qpk[w] = vq;
        if constexpr (SS::HASN) {
          ((uint32_t*)(sm + SS::TNK))[w] = nt;
          ((uint32_t*)(sm + SS::QNK))[w] = nq;
        }
      }
    });
    ex.sync();
  } else {
    // base codes in place; the reverse complement swaps symmetric positions
    ex.each([&](int tid) {
      for (int i = tid; i < Lt; i += SCAN_NT) {
        const unsigned char c = cls[tc[i] & 127];
        tc[i] = c < SXC_CLASS_ZERO ? c : (unsigned char)(128 | tc[i]);
      }
      if (strand) {
        for (int i = tid; i < (Lq + 1) / 2; i += SCAN_NT) {
          const unsigned char x = qc[i], y = qc[Lq - 1 - i];
          const unsigned char rx = rc[x & 127], ry = rc[y & 127];
          const unsigned char cx = cls[rx & 127], cy = cls[ry & 127];
          qc[i] = cy < SXC_CLASS_ZERO ? cy : (unsigned char)(128 | ry);
          qc[Lq - 1 - i] = cx < SXC_CLASS_ZERO ? cx : (unsigned char)(128 | rx);
        }
      } else {
        for (int i = tid; i < Lq; i += SCAN_NT) {
          const unsigned char c = cls[qc[i] & 127];
          qc[i] = c < SXC_CLASS_ZERO ? c : (unsigned char)(128 | qc[i]);
        }
      }
    });
    ex.sync();
    ex.each([&](int tid) {
      BasePlanes* tpl = (BasePlanes*)(sm + SS::TPL);
      BasePlanes* qpl = (BasePlanes*)(sm + SS::QPL);
      uint32_t* tam = (uint32_t*)(sm + SS::TAM);
      uint32_t* qam = (uint32_t*)(sm + SS::QAM);
      // per thread, two 16-bit counts each: words with another letter of the target and the query; A, C
      // and G, T of the target, of the query
      int sum[5] = {0, 0, 0, 0, 0};
      auto count = [&](const BasePlanes& b, uint32_t other, int left, int side) {
        const uint32_t v = ~other & (left >= 32 ? ~0u : left > 0 ? (1u << left) - 1 : 0u);
        sum[0] += (other != 0) << (16 * side);
        sum[1 + 2 * side] += __builtin_popcount(v & ~b.lo & ~b.hi) + (__builtin_popcount(v & b.lo & ~b.hi) << 16);
        sum[2 + 2 * side] += __builtin_popcount(v & ~b.lo & b.hi) + (__builtin_popcount(v & b.lo & b.hi) << 16);
      };
      for (int w = tid; w < SS::PLW; w += SCAN_NT) {
        BasePlanes t = {0, 0}, q = {0, 0};
        uint32_t to = 0, qo = 0;
        if (w >= 2 && w < 2 + N / 32) {
          t = planes_of_codes(tc, Lt, w - 2, to);
          q = planes_of_codes(qc, Lq, w - 2, qo);
          count(t, to, Lt - 32 * (w - 2), 0);
          count(q, qo, Lq - 32 * (w - 2), 1);
        }
        tpl[w] = t;
        qpl[w] = q;
        tam[w] = to;
        qam[w] = qo;
      }
      // (32 places for each sum: with one, the additions are scans over the lanes, 15 us in all)
      int* part = (int*)(sm + SS::RUNS);
      for (int k = 0; k < 5; ++k) ex.atomic_add_shared(&part[32 * k + (tid & 31)], sum[k]);
    });
    ex.sync();
    ex.each([&](int tid) {
      if (tid >= 5) return;
      const int* part = (const int*)(sm + SS::RUNS) + 32 * tid;
      int n = 0;
      for (int k = 0; k < 32; ++k) n += part[(k + tid) & 31];
      misc[SM_AMB + tid] = n;
    });
    ex.sync();
  }
  const uint16_t* cands = gcands;
  const int ncand = misc[SM_NCAND];
  // this workgroup's share of the lags (all of them unless the scan is split)
  const int lo = (int)((int64_t)ncand * part / split), hi = (int)((int64_t)ncand * (part + 1) / split);
  constexpr int CE = SS::CE;
  const int min_run = a.mode == 0 && !a.ptable ? a.min_run[SS::HASN ? 1 : SS::PURE ? 0 : 2] : 0;
  // Queue entries before the current epoch, kept per thread: every thread must see the same
  // count, and the shared counter may already hold the next epoch's pushes of a faster wave.
  int queued = 0;
  bool sliced = SS::SLICED;
  if constexpr (SS::AMB) sliced = slices_pay(misc, SS::LOG, scan_gate(min_run), split, hi - lo);
  if constexpr (SS::SLICED || SS::AMB)
    if (sliced) scan_sliced<NB>(ex, sm, a, pr, cands, ps, lo, hi, min_run);
  for (int e0 = sliced ? hi : lo; e0 < hi; e0 += CE) {
    const int qstart = queued;
    const int e1 = (e0 + CE < hi) ? e0 + CE : hi;
    if constexpr (SS::BMRUNS) {
      scan_epoch_bitmap<NB>(ex, sm, cands, e0, e1, SS::GSZ, min_run, a.stats != nullptr, [&](int n) {
        drain<NB>(ex, sm, a, pr, cands, ps, n, e0);
        ex.each([&](int tid) {
          if (tid == 0) misc[SM_QN] = 0;
        });
        ex.sync();
      });
      continue;
    }
    const int runs0 = misc[SM_RUNS];  // no thread pushes before the next barrier
    ex.sync();
    scan_epoch_segments<NB>(ex, sm, cands, e0, e1, SS::GSZ, min_run);
    const int qn = misc[SM_QN];
    ex.sync();  // every thread has read the count before any thread pushes again
    queued = qn;
    if (qn > SS::QCAP) {
      // the epoch overflowed the queue: keep what came before it, redo its lags one by one
      drain<NB>(ex, sm, a, pr, cands, ps, qstart, e0);  // (compact queue: empty)
      ex.each([&](int tid) {
        if (tid == 0) misc[SM_RUNS] = runs0;  // its runs are counted again below
      });
      for (int c = e0; c < e1; ++c) {
        ex.each([&](int tid) {
          if (tid == 0) misc[SM_QN] = 0;
        });
        ex.sync();
        scan_epoch_segments<NB>(ex, sm, cands, c, c + 1, SCAN_NT, min_run);
        const int n1 = misc[SM_QN];
        drain<NB>(ex, sm, a, pr, cands, ps, n1, c);
      }
      ex.each([&](int tid) {
        if (tid == 0) misc[SM_QN] = 0;
      });
      ex.sync();
      queued = 0;
    } else if (SS::COMPACT || qn > SS::QCAP / 2 || e1 == hi) {
      drain<NB>(ex, sm, a, pr, cands, ps, qn, e0);
      ex.each([&](int tid) {
        if (tid == 0) misc[SM_QN] = 0;
      });
      ex.sync();
      queued = 0;
    }
  }
  ex.each([&](int tid) {
    if (tid == 0) {
      if (split == 1) {
        a.counts[ps] = misc[SM_KEPT];
        if (a.stats) {
          a.stats[2 * ps] = ncand;
          a.stats[2 * ps + 1] = misc[SM_RUNS];
        }
      } else if (a.stats) {
        if (part == 0) a.stats[2 * ps] = ncand;
        ex.atomic_add_global(&a.stats[2 * ps + 1], misc[SM_RUNS]);
      }
    }
  });
}

}  // namespace sxc
