// sxc_kernels.hip -- gfx950 kernels of the chunk-pair path and their launchers.
//
// Build: hipcc --offload-arch=gfx950 -O3 -ffp-contract=off (FFTReal and the reference's
// double arithmetic are never contracted into FMA; see sxc_fft.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sxc_fft_kernels.h"
#include "sxc_kernels.h"
#include "sxc_pipeline.h"
#include "sxc_scan.h"
#include "sxc_scan_kernels.h"

namespace sxc {

template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_peaks(const float* xc, double cutoff, uint16_t* cands,
                                                     int32_t* ncand) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  peaks_body<NB>(ex, sm, xc, cutoff, cands, ncand);
  if (threadIdx.x == 0) ncand[1] = 0;  // the run count of a scan that follows (it may be split)
}

// Plain-API kernels ----------------------------------------------------------------

// CCSignal::SetSequence: the 4*N encoded signal of one chunk.
template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_encode(EncodeArgs a) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  encode_body<NB>(ex, sm, a, (int)blockIdx.x);
}

// CrossCorrelation::CrossCorrelate of given signals against resident target spectra.
template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_xcorr(XcorrArgs a) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  using SM = Smem<NB>;
  float* lut = (float*)(sm + SM::LUT);
  for (int i = threadIdx.x; i < SXC_LUT_LEN; i += Geo<NB>::NT) lut[i] = a.tab->lut[i];
  __syncthreads();
  const Twiddle tw{lut, a.osc};
  // a workgroup per channel; k_sum_channels adds them
  const int ch = blockIdx.x;
  correlate<NB>(ex, sm, a.tab, tw, SeqView{nullptr, nullptr, 0, 0}, a.spectra, a.qsig, TailRef{nullptr, 0, nullptr},
                nullptr, ch, ch + 1);
  const float* Y = (const float*)(sm + SM::Y);
  for (int p = threadIdx.x; p < Geo<NB>::N; p += Geo<NB>::NT) a.parts[(size_t)ch * Geo<NB>::N + p] = Y[pad(p)];
}

// A split CrossCorrelate's second half (XcorrArgs.parts): xc = 0 + A + C + G + T.
__global__ __launch_bounds__(256) void k_sum_channels(const float* parts, int N, float* xc) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p < N) xc[p] = (((0.f + parts[p]) + parts[N + p]) + parts[2 * N + p]) + parts[3 * N + p];
}

// GetMatchProbabilityEx + PrintMatch identity for given runs (one thread per run).  The sums are
// the reference's, base after base, so a thread is a chain of additions; what they wait for is
// read 16 bases ahead, through tables in LDS, and a workgroup is one wave so that a few hundred
// runs spread over the CUs.  (1600 runs of two 3001-bp chunks: 85 us with every base's four
// dependent reads from memory in the chain.)
__global__ __launch_bounds__(64) void k_prob(ProbArgs a) {
  __shared__ double equal[SXC_NCLASS * SXC_NCLASS], gc[SXC_NCLASS];
  __shared__ unsigned char cls[128];
  const sxc_tables* tab = a.tab;
  for (int i = threadIdx.x; i < SXC_NCLASS * SXC_NCLASS; i += 64) equal[i] = (&tab->equal[0][0])[i];
  for (int i = threadIdx.x; i < SXC_NCLASS; i += 64) gc[i] = tab->gc[i];
  for (int i = threadIdx.x; i < 128; i += 64) cls[i] = tab->cls[i];
  __syncthreads();
  const int k = blockIdx.x * 64 + threadIdx.x;
  if (k >= a.n) return;
  const int32_t* r = a.runs + 3 * k;
  const int st = r[0], sq = r[1], len = r[2];
  const unsigned char *t = a.t + st, *q = a.q + sq;
  double matches = 0, gct = 0, gcq = 0;
  int i = 0;
  for (; i + 16 <= len; i += 16) {
    unsigned char tb[16], qb[16];
    static_for<0, 16>([&](auto K) {
      tb[decltype(K)::value] = t[i + decltype(K)::value];
      qb[decltype(K)::value] = q[i + decltype(K)::value];
    });
    double e[16], gt[16], gq[16];
    static_for<0, 16>([&](auto K) {
      constexpr int x = decltype(K)::value;
      const int ca = cls[tb[x] & 127], cb = cls[qb[x] & 127];
      e[x] = equal[ca * SXC_NCLASS + cb];
      gt[x] = gc[ca];
      gq[x] = gc[cb];
    });
    static_for<0, 16>([&](auto K) {
      matches += e[decltype(K)::value];
      gct += gt[decltype(K)::value];
      gcq += gq[decltype(K)::value];
    });
  }
  for (; i < len; ++i) {
    const int ca = cls[t[i] & 127], cb = cls[q[i] & 127];
    matches += equal[ca * SXC_NCLASS + cb];
    gct += gc[ca];
    gcq += gc[cb];
  }
  const double ident = matches / (double)len;
  const double gc_target = gct / (double)len;
  const double at_target = 1. - gc_target;
  double rr = gcq * gc_target;
  rr += ((double)len - gcq) * at_target;
  const double p = rr / (double)len / 2.;
  const double s = sqrt(p * (1. - p) * (double)len);
  const double m = p * (double)len;
  const double x = (double)len * ident;
  const double cdf = 0.5 * (1. + erf((m - x) / s / 1.414213562));
  a.prob[k] = exp(-(cdf * a.target_size));
  a.ident[k] = ident;
}

// Exclusive scan of per-(pair, strand) kept counts (clipped to cap) -> offsets, total.
// With nflag: total[1] receives the scan's count of records flagged near min_prob, and the
// counter is cleared for the next scan.  One workgroup, bound by latency: each thread sums a
// contiguous share, the shares are scanned by lane shuffles within a wave and across the 16
// waves through LDS.
__global__ __launch_bounds__(1024) void k_scan_counts(const int32_t* counts, int n, int cap, int64_t* offsets,
                                                      int64_t* total, int32_t* max_count, int32_t* nflag) {
  __shared__ int64_t wsum[16];
  __shared__ int wmax[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int per = (n + 1023) / 1024;
  const int b = t * per < n ? t * per : n, e = (b + per < n) ? b + per : n;
  int64_t s = 0;
  int m = 0;
  for (int i = b; i < e; ++i) {
    const int c = counts[i];
    s += c < cap ? c : cap;
    m = c > m ? c : m;
  }
  int64_t inc = s;  // inclusive over the wave's lanes
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t v = __shfl_up(inc, d, 64);
    const int v2 = __shfl_xor(m, d, 64);
    if (lane >= d) inc += v;
    m = v2 > m ? v2 : m;
  }
  if (lane == 63) {
    wsum[wave] = inc;
    wmax[wave] = m;
  }
  __syncthreads();
  int64_t acc = inc - s;
  for (int w = 0; w < wave; ++w) acc += wsum[w];
  if (t == 1023) {
    *total = acc + s;
    int mm = 0;
    for (int w = 0; w < 16; ++w) mm = wmax[w] > mm ? wmax[w] : mm;
    *max_count = mm;
    if (nflag) {
      total[1] = *nflag;
      *nflag = 0;
    }
  }
  for (int i = b; i < e; ++i) {
    offsets[i] = acc;
    const int c = counts[i];
    acc += c < cap ? c : cap;
  }
}

__global__ __launch_bounds__(256) void k_clear_runs(int32_t* stats, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) stats[2 * i + 1] = 0;
}

// Orders each (pair, strand)'s kept records by (lag rank, run start) -- the order
// FilterMatches pushes them -- and packs them at their offsets.
// Records that would land at or beyond out_cap are not written (the host compares the
// total with out_cap and packs again into a larger buffer).
__global__ __launch_bounds__(256) void k_finalize(const sxc_result_dev* slots, const uint64_t* keys,
                                                  const int32_t* counts, const int64_t* offsets, int cap,
                                                  sxc_result_dev* out, int64_t out_cap) {
  const int ps = blockIdx.x;
  const int n = counts[ps] < cap ? counts[ps] : cap;
  const size_t base = (size_t)ps * cap;
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    const uint64_t ke = keys[base + e];
    int rank = 0;
    for (int k = 0; k < n; ++k) rank += keys[base + k] < ke;
    const int64_t at = offsets[ps] + rank;
    if (at < out_cap) out[at] = slots[base + e];
  }
}

// Orders MatchUp runs by (lag rank, run start): rank by counting smaller keys, 1024 of which the
// workgroup reads into LDS at a time (1600 runs: 90 us with every thread reading every key from
// memory).
__global__ __launch_bounds__(64) void k_order_runs(const int32_t* runs, const uint64_t* keys, int n, int32_t* out) {
  __shared__ uint64_t part[1024];
  const int e = blockIdx.x * 64 + threadIdx.x;
  const uint64_t ke = e < n ? keys[e] : 0;
  int rank = 0;
  for (int k0 = 0; k0 < n; k0 += 1024) {
    const int m = n - k0 < 1024 ? n - k0 : 1024;
    __syncthreads();
    for (int k = threadIdx.x; k < m; k += 64) part[k] = keys[k0 + k];
    __syncthreads();
    int k = 0;
    for (; k + 8 <= m; k += 8)
      static_for<0, 8>([&](auto K) { rank += part[k + decltype(K)::value] < ke; });
    for (; k < m; ++k) rank += part[k] < ke;
  }
  if (e >= n) return;
  out[3 * rank] = runs[3 * e];
  out[3 * rank + 1] = runs[3 * e + 1];
  out[3 * rank + 2] = runs[3 * e + 2];
}

// ---------------------------------------------------------------- launchers

hipError_t launch_order_runs(const int32_t* runs, const uint64_t* keys, int n, int32_t* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_order_runs, dim3((n + 63) / 64), dim3(64), 0, s, runs, keys, n, out);
  return hipGetLastError();
}

#define SXC_NB_SWITCH(NB, CALL)      \
  switch (NB) {                      \
    case 9: CALL(9); break;          \
    case 10: CALL(10); break;        \
    case 11: CALL(11); break;        \
    case 12: CALL(12); break;        \
    case 13: CALL(13); break;        \
    case 14: CALL(14); break;        \
    case 15: CALL(15); break;        \
    default: return hipErrorInvalidValue; \
  }

const FftEntry* fft_table_default(int* n) {
  static const FftEntry t[] = {SXC_FFT_ENTRY(9) SXC_FFT_ENTRY(10) SXC_FFT_ENTRY(11) SXC_FFT_ENTRY(12)
                                   SXC_FFT_ENTRY(13) SXC_FFT_ENTRY(14) SXC_FFT_ENTRY(15)};
  *n = (int)(sizeof(t) / sizeof(t[0]));
  return t;
}

const FftEntry* fft_entry(int geo) {
  for (auto tf : {fft_table_default, fft_table_r2, fft_table_s32, fft_table_occ, fft_table_lean}) {
    int n = 0;
    const FftEntry* t = tf(&n);
    for (int i = 0; i < n; ++i)
      if (t[i].geo == geo) return &t[i];
  }
  return nullptr;
}

int fft_geometries(int nb, int* out, int cap) {
  int n = 0;
  for (auto tf : {fft_table_default, fft_table_r2, fft_table_s32, fft_table_occ, fft_table_lean}) {
    int nt = 0;
    const FftEntry* t = tf(&nt);
    for (int i = 0; i < nt; ++i) {
      const int g = t[i].geo;
      if (geo_nb(g) != nb) continue;
      bool dup = false;  // the same geometry under another code
      for (int j = 0; j < n; ++j)
        dup |= geo_sa(out[j]) == geo_sa(g) && geo_km(out[j]) == geo_km(g) && geo_occ(out[j]) == geo_occ(g) &&
               geo_lean(out[j]) == geo_lean(g);
      if (!dup && n < cap) out[n++] = g;
    }
  }
  return n;
}

hipError_t launch_correlate(int geo, const PairArgs& a, int total, hipStream_t s) {
  if (a.parts) return launch_correlate_parts(geo_nb(geo), a, total, s);
  const FftEntry* e = fft_entry(geo);
  return e ? e->correlate(a, total, s) : hipErrorInvalidValue;
}

// Workgroups per (pair, strand) for n of them.  Every workgroup packs both chunks first, so a
// share pays only while compute units are idle.
// Pure A/C/G/T: a share's slices also come in whole waves.  us with 1 / 2 / 4 / 8 / 16 workgroups
// per strand at N = 8192: 2 strands 42 / 34 / 34 / 30 / 29, 32 strands 50 / 36 / 33 / 29 / 30, 128
// strands 50 / 39 / 42 / 39 / 51, 512 strands 68 / 65 / 87 / 97 / 140, 1024 strands 99 / 102 /
// 135 / 175 / 266 (N = 2048 the same within 10%); at N = 32768, with 4 times the lags and
// positions: 32 strands 359 / 196 / 146 / 94 / 81, 128 strands 356 / 203 / 203 / 202 / 203, 512
// strands 501 / 438 / 555 / - / -, 2048 strands 1434 / 1406 / 1965 / - / -.
// With N, lags are taken 8 or 16 at a time: up to 2048 workgroups in all (8 per CU), more than 4 per
// strand only to 102 strands (1 / 2 / 4 / 8 at N = 8192: 96 strands 156 / 95 / 76 / 64, 256 strands 163 /
// 113 / 103 / 117, 400 strands 183 / 141 / 154 / 162, 800 strands 251 / 224 / 242 / 282; at N = 2048 400
// strands 312 / 208 / 180 / 170).  With other letters the same to 320 strands, 2 above them.
// Then no more than pays by the rounds of workgroups that fit the device (scan_resident), as a share
// costs its packing and the middle shares hold the longer diagonals: with other letters at every N,
// with N at 32768 where fewer than 8 of them fit a CU and one per strand is resident at once.  us with
// 1 / 2 / 3 / 4 shares, one other letter in the target and one in 16 bases: N = 512, 800 strands 120 / 200 /
// 200 / 292 and 171 / 183 / 169 / 197; N = 2048, 800 strands 352 / 368 / 326 / 459 and 1242 / 1152 / 1100 /
// 1222; N = 8192, 256 strands 302 / 256 / 233 / 270 and 1307 / 817 / 727 / 657, 320 strands 324 / 269 /
// 256 / 398 and 1340 / 837 / 761 / 1048, 640 strands 347 / 460 / 346 / 605 and 1381 / 1413 / 1371 / 1555;
// N = 16384, 160 strands 623 / 507 / 443 / 744 and 4486 / 2491 / 2378 / 3350; N = 32768, 128 strands 2092 /
// 1471 / 1755 / 2376 and 15393 / 8154 / 11801 / 11592, 256 strands 2092 / 2907 / 3011 / 4739 and 15389 /
// 16005 / 19767 / 22960, 320 strands 4065 / 4220 / 3431 / 5939 and 30355 / 23276 / 23561 / 28650; with N at
// 32768, 160 strands 1550 / 1102 / 872 / 1198, 512 strands 1933 / 2118 / 2399 / 2866.
static int resident_scans(int kind, int nb) {  // workgroups that fit 256 CUs
#define CALL(X) return 256 * (kind == SCAN_N ? scan_resident<(X) | 64>() : scan_resident<X>())
  switch (nb) {
    case 12: CALL(12);
    case 13: CALL(13);
    case 14: CALL(14);
    case 15: CALL(15);
    default: CALL(11);  // (the most waves already)
  }
#undef CALL
}

// At most `most` shares of n strands: the fewest whose rounds on `resident` places, per share, are
// within 10% of the least.
static int shares_by_rounds(int n, int resident, int most) {
  if ((int64_t)n * most <= resident) return most;
  auto rounds = [&](int k) { return ((int64_t)n * k + resident - 1) / resident; };
  int best = 1;
  for (int k = 2; k <= most; ++k)
    if (rounds(k) * best < rounds(best) * k) best = k;
  for (int k = 1; k < best; ++k)
    if (10 * rounds(k) * best <= 11 * rounds(best) * k) return k;
  return best;
}

static int scan_split(int kind, int nb, int n) {
  if (n <= 0) return 1;
  if (kind == SCAN_PURE) return n <= 32 ? 16 : n <= 128 ? 8 : n <= (nb >= 14 ? 2048 : 768) ? 2 : 1;
  const int most = std::max(1, std::min({2048 / n, std::max(kind == SCAN_GENERAL && n > 320 ? 2 : 4, 512 / n), 16}));
  const int resident = resident_scans(kind, nb);
  return kind == SCAN_GENERAL || (nb == 15 && n <= resident) ? shares_by_rounds(n, resident, most) : most;
}

hipError_t launch_scan(int nb, const ScanArgs& a, int total, const ScanKinds& kinds, bool can_split, hipStream_t s) {
  // One launch per kind that occurs.  Shares of a strand add their run counts, so those start at
  // zero (cleared here and not by the pair kernel, which one more store made 3% slower at N = 16384).
  if (kinds.all() * a.strands != total || (kinds.mixed() && !a.list)) return hipErrorInvalidValue;
  int first = 0;
  if (can_split && a.stats)
    for (int k = 0; k < 3; ++k)
      if (kinds.pairs[k] > 0 && scan_split(k, nb, kinds.pairs[k] * a.strands) > 1) {
        hipLaunchKernelGGL(k_clear_runs, dim3((total + 255) / 256), dim3(256), 0, s, a.stats, total);
        break;
      }
  for (int k = 0; k < 3; ++k) {
    if (kinds.pairs[k] <= 0) continue;
    ScanArgs b = a;
    const int n = kinds.pairs[k] * a.strands;
    b.split = can_split ? scan_split(k, nb, n) : 1;
    b.list = a.list ? a.list + first : nullptr;
    first += n;
    // a launch of 2^32 threads or more is not refused: its last workgroups are missing
    if ((int64_t)n * b.split * SCAN_NT >= (int64_t)1 << 32) return hipErrorInvalidValue;
    const hipError_t e = (k == 0 ? launch_scan_pure : k == 1 ? launch_scan_n : launch_scan_general)(nb, b, n * b.split, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_peaks(int nb, const float* xc, double cutoff, uint16_t* cands, int32_t* ncand, hipStream_t s) {
#define CALL(X) hipLaunchKernelGGL(k_peaks<X>, dim3(1), dim3(Geo<X>::NT), 0, s, xc, cutoff, cands, ncand)
  SXC_NB_SWITCH(nb, CALL)
#undef CALL
  return hipGetLastError();
}

hipError_t launch_spectra(int geo, const SpecArgs& a, hipStream_t s) {
  if (a.per_channel) return launch_spectra_parts(geo_nb(geo), a, s);
  const FftEntry* e = fft_entry(geo);
  return e ? e->spectra(a, s) : hipErrorInvalidValue;
}

hipError_t launch_encode(int nb, const EncodeArgs& a, int n, hipStream_t s) {
#define CALL(X) hipLaunchKernelGGL(k_encode<X>, dim3(n), dim3(Geo<X>::NT), 0, s, a)
  SXC_NB_SWITCH(nb, CALL)
#undef CALL
  return hipGetLastError();
}

hipError_t launch_xcorr(int nb, const XcorrArgs& a, hipStream_t s) {
#define CALL(X) hipLaunchKernelGGL(k_xcorr<X>, dim3(4), dim3(Geo<X>::NT), 0, s, a)
  SXC_NB_SWITCH(nb, CALL)
#undef CALL
  hipLaunchKernelGGL(k_sum_channels, dim3((1 << nb) / 256), dim3(256), 0, s, a.parts, 1 << nb, a.xc);
  return hipGetLastError();
}

hipError_t launch_prob(const ProbArgs& a, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_prob, dim3((a.n + 63) / 64), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_count_offsets(const int32_t* counts, int n, int cap, int64_t* offsets, int64_t* total,
                                int32_t* max_count, hipStream_t s, int32_t* nflag) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, s, counts, n, cap, offsets, total, max_count, nflag);
  return hipGetLastError();
}

hipError_t launch_order_records(const int32_t* counts, int n, int cap, const int64_t* offsets,
                                const sxc_result_dev* slots, const uint64_t* keys, sxc_result_dev* out,
                                int64_t out_cap, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_finalize, dim3(n), dim3(256), 0, s, slots, keys, counts, offsets, cap, out, out_cap);
  return hipGetLastError();
}

}  // namespace sxc
