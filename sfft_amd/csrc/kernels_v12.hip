// sFFT v1/v2 kernels for gfx950.
//
//   comb          v2 heavy-hitter prefilter: strided W-point sub-sample, FFT
//                 in LDS, top-2k residues (src/computefourier-1.0-2.0.cc:48-82)
//   comb_merge    sort+dedupe of several comb loops' residues (cf12 492-502)
//   fold_fft      permuted-filter bucketization folded into B buckets, then
//                 the B-point FFT in LDS (cf12 222-275)
//   select        top-2k buckets of each location loop (cf12 278-302)
//   vote          v1 exact-integer location votes (cf12 91-116) without an
//                 n-sized score array (count / scan / write over chunks)
//   estimate      per located frequency, the lower median over loops of
//                 bucket / filter (cf12 340-419)
//
// Signals of a batch are independent; blockIdx encodes (signal, loop) or
// (signal, chunk).  All index arithmetic is exact: for n = 2^p the low 32
// bits of i * a already give (i * a) mod n.
#include <algorithm>
#include <climits>
#include <mutex>
#include <string>

#include "device_common.hpp"
#include "internal.hpp"

namespace sfa {
namespace k {

using namespace sfa::dev;

namespace {

__device__ __forceinline__ int ilog2(int v) { return 31 - __clz(v); }

inline int pow2_ceil_int(int v)
{
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

__device__ __forceinline__ int64_t loop_offset(int l, int Lloc, int Bl, int Be)
{
  return (int64_t)min(l, Lloc) * Bl + (int64_t)max(0, l - Lloc) * Be;
}

inline int64_t loop_offset_host(int l, int Lloc, int Bl, int Be)
{
  return (int64_t)std::min(l, Lloc) * Bl + (int64_t)std::max(0, l - Lloc) * Be;
}

// Levels of a selection above the LDS size: threads, entries picked per
// chunk at most, entries per chunk, and of the last level.
constexpr int kTopThreads = 512, kTopMax = 4096, kTopChunk = 4096, kTopLast = 16384;

// ---------------------------------------------------------------- comb
// Comb loop c of signal s by one workgroup of TB threads.  LDS: W double2 at
// smem64, kTopScratch ints at sh.
template <int TB>
__device__ __forceinline__ void comb_block(const V12Launch &a, int s, int c, double2 *smem64,
                                           int *sh)
{
  const int cl = a.comb_loops;
  const int stride = 2 * a.L + max(cl, 1);
  const int off = a.params[(int64_t)s * stride + 2 * a.L + c];
  const int W = a.W, logW = ilog2(W);
  const int sigma = a.n / W;
  const double2 *x = a.x[s];
  slot_fft_fill(smem64, logW, [&](int i) { return x[(int64_t)off + (int64_t)i * sigma]; });
  slot_fft(smem64, logW, a.tw64, a.tw_nmax / W);
  // |.|^2 into the same LDS, as doubles (staged through registers: W is at
  // most kMaxLdsComb)
  constexpr int kPer = (kMaxLdsComb + TB - 1) / TB;
  double v[kPer];
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    const int i = threadIdx.x + q * TB;
    if (i < W) {
      const double2 z = smem64[fft_slot<double2>(i, logW)];
      v[q] = z.x * z.x + z.y * z.y;
    }
  }
  __syncthreads();
  double *mag = reinterpret_cast<double *>(smem64);
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    const int i = threadIdx.x + q * TB;
    if (i < W) mag[i] = v[q];
  }
  __syncthreads();
  int *out = a.approved + ((int64_t)s * cl + c) * a.num;
  block_top_num(mag, W, a.num, out, sh);
  if (cl == 1 && threadIdx.x == 0) {
    a.num_comb[s] = a.num;
    a.count[s] = (int64_t)a.num * (a.n / W);
  }
}

// Combs in a launch of their own (beside the fold on a second stream):
// kBlock threads for batches; more for a few signals, whose comb is on the
// latency path.
template <int TB>
__global__ void __launch_bounds__(TB) k_comb(V12Launch a)
{
  extern __shared__ double2 smem64[];
  __shared__ int sh[kTopScratch];
  comb_block<TB>(a, blockIdx.x / a.comb_loops, blockIdx.x % a.comb_loops, smem64, sh);
}

// Selections above the LDS size, in levels: block (t, chunk) takes `chunk`
// entries of row t's list (the first level: every index of the row) and
// writes the num largest of them, by block_top_num's rule, in list order, to
// its place of the next list.  An entry in the row's num largest is in its
// chunk's, and the lists stay in index order, so the last level (one chunk)
// picks what one selection over the whole row would, ties included.  One
// 256-thread workgroup over a whole row took 660 us for 100 of 131,072; two
// levels (chunks of 4096, then 3200 candidates) take 28 us.
struct TopLevel {
  const double *mag;    // rows of `row` powers; null: |xs64|^2 of the v1 loops
  int64_t row;
  const int *list;      // entries per row: list_len (null on the first level)
  int list_len, chunk, chunks;
  int num;
  int *out;             // per row: out_stride entries, num per chunk
  int64_t out_stride;
  bool comb_last;       // last level of a single comb loop: counts too
};

__global__ void __launch_bounds__(kTopThreads) k_top_level(V12Launch a, TopLevel v)
{
  extern __shared__ double lds_mag[];
  __shared__ int sh[kTopScratch];
  __shared__ int pick[kTopMax];
  const int t = (int)(blockIdx.x / (unsigned)v.chunks), ch = (int)(blockIdx.x % (unsigned)v.chunks);
  const int e0 = ch * v.chunk, len = min(v.chunk, v.list_len - e0);
  const int *list = v.list ? v.list + (int64_t)t * v.list_len + e0 : nullptr;
  const double *mag = v.mag ? v.mag + t * v.row : nullptr;
  const double2 *z = a.xs64 + (int64_t)(t / a.Lloc) * a.xs + (int64_t)(t % a.Lloc) * a.B_loc;
  for (int i = threadIdx.x; i < len; i += blockDim.x) {
    const int e = list ? list[i] : e0 + i;
    if (mag) {
      lds_mag[i] = mag[e];
    } else {
      const double2 y = z[e];
      lds_mag[i] = y.x * y.x + y.y * y.y;
    }
  }
  __syncthreads();
  int *out = v.out + (int64_t)t * v.out_stride + (int64_t)ch * v.num;
  const int take = min(v.num, len);
  if (len > v.num) block_top_num(lds_mag, len, v.num, pick, sh);
  __syncthreads();
  for (int i = threadIdx.x; i < take; i += blockDim.x) {
    const int p = len > v.num ? pick[i] : i;
    out[i] = list ? list[p] : e0 + p;
  }
  if (v.comb_last && threadIdx.x == 0) {
    a.num_comb[t] = a.num;
    a.count[t] = (int64_t)a.num * (a.n / a.W);
  }
}

// Several comb loops: union of residues, ascending (bitmap over W in LDS).
__global__ void __launch_bounds__(kBlock) k_comb_merge(V12Launch a)
{
  extern __shared__ unsigned bits[];
  __shared__ int sh[16];
  const int s = blockIdx.x;
  const int W = a.W, words = (W + 31) / 32;
  const int tot = a.comb_loops * a.num;
  int *ap = a.approved + (int64_t)s * tot;
  for (int i = threadIdx.x; i < words; i += blockDim.x) bits[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < tot; i += blockDim.x) {
    const int r = ap[i];
    atomicOr(&bits[r >> 5], 1u << (r & 31));
  }
  __syncthreads();
  const int C = (words + blockDim.x - 1) / blockDim.x;
  const int lo = threadIdx.x * C, hi = min(words, lo + C);
  int cnt = 0;
  for (int wd = lo; wd < hi; wd++) cnt += __popc(bits[wd]);
  int total;
  int pos = block_exclusive_scan(cnt, sh, total);
  // write after everyone has read the unmerged lists
  __syncthreads();
  for (int wd = lo; wd < hi; wd++) {
    unsigned b = bits[wd];
    while (b) {
      const int bit = __ffs(b) - 1;
      ap[pos++] = wd * 32 + bit;
      b &= b - 1;
    }
  }
  if (threadIdx.x == 0) {
    a.num_comb[s] = total;
    a.count[s] = (int64_t)total * (a.n / W);
    if (a.count_host) a.count_host[s] = a.count[s];
  }
}

// ---------------------------------------------------------------- fold + FFT
// One block per (signal, loop).  Each thread owns buckets m = tid + q*T and
// sums, in ascending tap order like the reference, x[(i*ai) mod n]*tap[i]
// over the taps i = m + r*B < w.  LDS: B double2.  FP64 only (the FP32
// form folds in k_fold_sorted).
constexpr int kQ = 8;  // buckets per thread in flight (independent gathers)

__global__ void __launch_bounds__(kBlock) k_fold_fft64(V12Launch a, int l0, int nl)
{
  extern __shared__ double2 smem64[];
  const int s = blockIdx.x / nl, l = l0 + blockIdx.x % nl;
  const bool isloc = l < a.Lloc;
  const int B = isloc ? a.B_loc : a.B_est;
  const int w = isloc ? a.w_loc : a.w_est;
  const double2 *__restrict__ taps = isloc ? a.taps_loc : a.taps_est;
  const int stride = 2 * a.L + max(a.comb_loops, 1);
  const unsigned ai = (unsigned)a.params[(int64_t)s * stride + a.L + l];
  const double2 *__restrict__ x = a.x[s];
  const unsigned mask = (unsigned)a.n - 1;
  const int logB = ilog2(B);
  const int T = blockDim.x;
  const int R = (w + B - 1) / B;
  for (int mb = threadIdx.x; mb < B; mb += T * kQ) {
    double2 acc[kQ];
#pragma unroll
    for (int q = 0; q < kQ; q++) acc[q] = make_double2(0.0, 0.0);
    for (int r = 0; r < R; r++) {
      double2 xv[kQ], tv[kQ];
#pragma unroll
      for (int q = 0; q < kQ; q++) {
        const int m = mb + q * T;
        const int i = m + r * B;
        if (m < B && i < w) {
          xv[q] = x[((unsigned)i * ai) & mask];
          tv[q] = taps[i];
        }
      }
#pragma unroll
      for (int q = 0; q < kQ; q++) {
        const int m = mb + q * T;
        const int i = m + r * B;
        if (m < B && i < w) {
          const double re = xv[q].x * tv[q].x - xv[q].y * tv[q].y;
          const double im = xv[q].x * tv[q].y + xv[q].y * tv[q].x;
          acc[q].x = acc[q].x + re;
          acc[q].y = acc[q].y + im;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; q++) {
      const int m = mb + q * T;
      if (m < B) smem64[fft_slot<double2>(bitrev(m, logB), logB)] = acc[q];
    }
  }
  slot_fft(smem64, logB, a.tw64, a.tw_nmax / B);
  double2 *out = a.xs64 + (int64_t)s * a.xs +
                 loop_offset(l, a.Lloc, a.B_loc, a.B_est);
  for (int j = threadIdx.x; j < B; j += T) out[j] = smem64[fft_slot<double2>(j, logB)];
}

// ---------------------------------------------------------------- sorted fold
// Bucket sums with the gathers in address order.  Loop l adds x[p] * tap[i]
// into bucket b = i mod B for the taps i = b + kB < w at p = i*ai mod n;
// p mod B = b*ai mod B, so bucket b only ever reads residue class
// r = b*ai mod B, and b = r*a mod B (a*ai = 1 mod n).  Viewing the signal as
// n/B rows of B samples (p = r + t*B), a workgroup takes the buckets of
// f.res consecutive residues in every loop of the part, one (residue, loop)
// pair per thread, and is the only reader of those residues' lines.  It
// sorts its pairs' taps by row (a counting sort in LDS) and walks the sorted
// list: neighbouring lanes read the same or the next row, so a 128-byte line
// is requested once, whichever loops' taps meet in it, and every load of the
// walk is independent of the others.  The products replace the taps in LDS,
// and each pair's thread adds its own in the form's fixed order:
//   FP64  ascending tap order, as the reference does;
//   FP32  chunk by chunk of 2^seg_log rows, in ascending tap order within a
//         chunk, with compensated (2Sum) sums, the chunks' sums added in
//         chunk order.
//
// Bound by HBM on batches: the 850,060 gathers of a signal (n = 2^22, k = 64)
// touch 422,076 lines, 13.83 GB per 256 signals, read in 2.76 ms (5.0 TB/s;
// a large copy reaches 4.7).  Before, with the gathers of a 256-row chunk in
// flight at a time in tap order, 3.72 ms; the FP64 form, one wave per 64
// buckets in tap order, took 1.03 ms per 64 signals against 0.80 ms.  One
// signal is bound by the phases' latency: 19 us against 36 us (FP32), 17 us
// against 24 us (FP64, n = 2^22, k = 100).
constexpr int kMaxTaps = 32;           // taps per pair: 5 bits of a list entry
constexpr int kFoldThreads = 512;      // and pairs per workgroup at most
constexpr int kWalkAhead = 8;          // gathers in flight per thread
constexpr int kSortAhead = 8;          // sort steps and tap loads in flight per thread
constexpr int kPackLog = 3, kPackChunks = 1 << kPackLog;  // tap counts in one 64-bit word
constexpr size_t kFoldLds = 150 * 1024;  // dynamic LDS of a workgroup at most

// Loops [l0, l0 + nl) of one bucket count and precision.
struct FoldPart {
  int fp32;
  int l0, nl;
  int B, logB;
  int res, log_res;      // residues per workgroup
  int groups;            // B / res
  int tR;                // LDS stride of a pair's taps (max ceil(w/B), odd)
  unsigned inv_tR;       // idx / tR = idx * inv_tR >> 20 for idx below kFoldThreads * tR
  int nbins, bin_shift;  // sort bins of 2^bin_shift rows
  int seg_log;           // FP32: rows per chunk 2^seg_log
  int order_at;          // the sorted list, then FP32 the taps' order: in words of LDS
};

struct FoldParts {
  FoldPart p[2];
  int groups;  // workgroups per signal, all parts
  // the workgroups past S * groups clear the dense outputs, zero_blocks per
  // signal (the estimates are written later on the stream): a launch less,
  // and the stores run beside the gathers
  int zero_blocks;
  // the first workgroups run the combs of the batch's signals (S x comb
  // loops, 0 when they have a launch of their own)
  int combs;
};

// sum + cmp gains v, compensated (2Sum)
__device__ __forceinline__ void add2(float2 &sum, float2 &cmp, float2 v)
{
  float t = sum.x + v.x, bp = t - sum.x;
  cmp.x += (sum.x - (t - bp)) + (v.x - bp);
  sum.x = t;
  t = sum.y + v.y;
  bp = t - sum.y;
  cmp.y += (sum.y - (t - bp)) + (v.y - bp);
  sum.y = t;
}

// Group g of the part's residues in signal s.
template <bool FP32>
__device__ __forceinline__ void fold_group(const V12Launch &a, const FoldPart &f, int s, int g,
                                           double2 *smem64, int *sh)
{
  using T2 = typename std::conditional<FP32, float2, double2>::type;
  constexpr int T = kFoldThreads;
  const int tid = threadIdx.x;
  const int npairs = f.res * f.nl;
  T2 *slots = reinterpret_cast<T2 *>(smem64);
  int *bins = reinterpret_cast<int *>(smem64);  // until the list is built
  uint2 *pp = reinterpret_cast<uint2 *>(smem64 + (npairs * f.tR * sizeof(T2) + 15) / 16);
  int *tap_at = reinterpret_cast<int *>(pp + npairs);
  uint16_t *list = reinterpret_cast<uint16_t *>(tap_at + npairs);
  const int B = f.B, logB = f.logB;
  const unsigned mask = (unsigned)a.n - 1, rmask = ((unsigned)a.n >> logB) - 1;
  const int *prm = a.params + (int64_t)s * (2 * a.L + max(a.comb_loops, 1));
  const bool has = tid < npairs;
  const int l = f.l0 + (has ? tid >> f.log_res : 0);
  const unsigned av = (unsigned)prm[l], ai = (unsigned)prm[a.L + l];
  const unsigned res = (unsigned)(g * f.res + (tid & (f.res - 1)));
  const int b = (int)((res * av) & (unsigned)(B - 1));
  const int w = l < a.Lloc ? a.w_loc : a.w_est;
  const int R = (has && b < w) ? (w - b + B - 1) / B : 0;
  const unsigned p0 = ((unsigned)b * ai) & mask, step = ((unsigned)B * ai) & mask;
  const unsigned row0 = p0 >> logB, srow = step >> logB;  // row of tap k: row0 + k srow
  if (has) {
    // the pair's first sample and stride, and its run of taps (bit 31: of
    // the location filter)
    pp[tid] = make_uint2(p0, step);
    tap_at[tid] = b * (l < a.Lloc ? a.tR_loc : a.tR_est) | (l < a.Lloc ? INT_MIN : 0);
  }
  for (int i = tid; i < f.nbins; i += T) bins[i] = 0;
  __syncthreads();
  for (int k = 0; k < R; k++)
    atomicAdd(&bins[((row0 + (unsigned)k * srow) & rmask) >> f.bin_shift], 1);
  __syncthreads();
  int total;
  {
    const int C = (f.nbins + T - 1) / T;
    const int lo = min(f.nbins, tid * C), hi = min(f.nbins, lo + C);
    int sum = 0;
    for (int i = lo; i < hi; i++) sum += bins[i];
    int run = block_exclusive_scan(sum, sh, total);
    for (int i = lo; i < hi; i++) {
      const int v = bins[i];
      bins[i] = run;
      run += v;
    }
  }
  __syncthreads();
  for (int k0 = 0; k0 < R; k0 += kSortAhead) {
    int at[kSortAhead];
#pragma unroll
    for (int u = 0; u < kSortAhead; u++)
      if (k0 + u < R)
        at[u] = atomicAdd(&bins[((row0 + (unsigned)(k0 + u) * srow) & rmask) >> f.bin_shift], 1);
#pragma unroll
    for (int u = 0; u < kSortAhead; u++)
      if (k0 + u < R) list[at[u]] = (uint16_t)(tid << 5 | (k0 + u));
  }
  __syncthreads();
  const double2 *__restrict__ x = a.x[s];
  double2 xv[kWalkAhead];
  int at[kWalkAhead];
  auto gather = [&](int j0) {
#pragma unroll
    for (int u = 0; u < kWalkAhead; u++) {
      const int j = j0 + u * T;
      at[u] = -1;
      if (j < total) {
        const unsigned e = list[j];
        const int pr = (int)(e >> 5), k = (int)(e & 31);
        const uint2 q = pp[pr];
        xv[u] = x[(q.x + (unsigned)k * q.y) & mask];
        at[u] = pr * f.tR + k;
      }
    }
  };
  gather(tid);  // in flight while the taps are staged
  // the taps, by bucket, in coalesced runs
  {
    const T2 *tl, *te;
    if constexpr (FP32) {
      tl = a.tapsT_loc32;
      te = a.tapsT_est32;
    } else {
      tl = a.tapsT_loc;
      te = a.tapsT_est;
    }
    const int cnt = npairs * f.tR;
    for (int i0 = tid; i0 < cnt; i0 += kSortAhead * T) {
      T2 t[kSortAhead];
#pragma unroll
      for (int u = 0; u < kSortAhead; u++) {
        const int idx = min(i0 + u * T, cnt - 1);
        const int pr = (int)(((unsigned)idx * f.inv_tR) >> 20), k = idx - pr * f.tR;
        const int ta = tap_at[pr];
        const T2 *tp = ta < 0 ? tl : te;
        t[u] = tp[(ta & INT_MAX) + min(k, (ta < 0 ? a.tR_loc : a.tR_est) - 1)];
      }
#pragma unroll
      for (int u = 0; u < kSortAhead; u++) slots[min(i0 + u * T, cnt - 1)] = t[u];
    }
  }
  __syncthreads();
  for (int j0 = tid;;) {
#pragma unroll
    for (int u = 0; u < kWalkAhead; u++) {
      if (at[u] < 0) continue;
      const T2 t = slots[at[u]];
      if constexpr (FP32) {
        slots[at[u]] = cmul(make_float2((float)xv[u].x, (float)xv[u].y), t);
      } else {
        slots[at[u]] = make_double2(xv[u].x * t.x - xv[u].y * t.y, xv[u].x * t.y + xv[u].y * t.x);
      }
    }
    j0 += kWalkAhead * T;
    if (j0 >= total) break;
    gather(j0);
  }
  __syncthreads();
  if (!has) return;
  const T2 *mine = slots + tid * f.tR;
  const int64_t out = (int64_t)s * a.xs + loop_offset(l, a.Lloc, a.B_loc, a.B_est) + b;
  if constexpr (FP32) {
    // the taps in summation order, a byte each, where the list was: stable
    // counting sorts by the chunk, kPackLog bits at a time, the counts and
    // the places (their exclusive byte-wise prefix sum) in 64-bit words
    const int tR4 = (f.tR + 3) & ~3;
    uint8_t *order = reinterpret_cast<uint8_t *>(
        reinterpret_cast<uint32_t *>(smem64) + f.order_at) + tid * tR4;
    uint8_t *from = order + npairs * tR4;  // second list, for several passes
    for (int sft = 0; sft == 0 || (rmask >> f.seg_log) >> sft; sft += kPackLog) {
      auto bits = [&](unsigned k) {
        return 8 * (int)((((row0 + k * srow) & rmask) >> (f.seg_log + sft)) & (kPackChunks - 1));
      };
      uint64_t place = 0;
      for (int k = 0; k < R; k++) place += 1ull << bits(k);
      place *= 0x0101010101010100ull;
      if (sft) {
        uint8_t *t = order;
        order = from;
        from = t;
      }
      for (int i = 0; i < R; i++) {
        const unsigned k = sft ? from[i] : (unsigned)i;
        const int c8 = bits(k);
        order[(place >> c8) & 255] = (uint8_t)k;
        place += 1ull << c8;
      }
    }
    float2 tot = make_float2(0.f, 0.f), sum = tot, cmp = tot;
    unsigned chunk = ~0u;
    for (int i0 = 0; i0 < R; i0 += 4) {
      // four taps' products and chunks at a time
      const unsigned four = *reinterpret_cast<const unsigned *>(order + i0);
      float2 v[4];
      unsigned c[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const unsigned k = min((four >> (8 * u)) & 255u, (unsigned)(R - 1));  // past R: unused
        v[u] = mine[k];
        c[u] = ((row0 + k * srow) & rmask) >> f.seg_log;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (i0 + u >= R) break;
        if (c[u] != chunk) {
          tot = make_float2(tot.x + (sum.x + cmp.x), tot.y + (sum.y + cmp.y));
          sum = cmp = make_float2(0.f, 0.f);
          chunk = c[u];
        }
        add2(sum, cmp, v[u]);
      }
    }
    tot = make_float2(tot.x + (sum.x + cmp.x), tot.y + (sum.y + cmp.y));
    a.xs32[out] = tot;
  } else {
    double2 acc = make_double2(0.0, 0.0);
    for (int k = 0; k < R; k++) {
      acc.x = acc.x + mine[k].x;
      acc.y = acc.y + mine[k].y;
    }
    a.xs64[out] = acc;
  }
}

// grid: f.combs, S x f.groups, S x f.zero_blocks
__global__ void __launch_bounds__(kFoldThreads) k_fold_sorted(V12Launch a, FoldParts f)
{
  extern __shared__ double2 smem64[];
  __shared__ int sh[16];
  unsigned blk = blockIdx.x;
  if (blk < (unsigned)f.combs) {
    comb_block<kFoldThreads>(a, (int)blk / a.comb_loops, (int)blk % a.comb_loops, smem64,
                             reinterpret_cast<int *>(smem64 + a.W));
    return;
  }
  blk -= (unsigned)f.combs;
  if (blk >= (unsigned)(a.S * f.groups)) {
    const unsigned z = blk - (unsigned)(a.S * f.groups);
    double2 *out = a.o_dense[z / (unsigned)f.zero_blocks];
    if (!out) return;  // not wanted on the device
    const int64_t step = (int64_t)f.zero_blocks * kFoldThreads;
    for (int64_t i = (int64_t)(z % (unsigned)f.zero_blocks) * kFoldThreads + threadIdx.x; i < a.n;
         i += step)
      out[i] = make_double2(0.0, 0.0);
    return;
  }
  const int s = (int)(blk / (unsigned)f.groups);
  int g = (int)(blk % (unsigned)f.groups);
  FoldPart p = f.p[0];
  if (g >= p.groups) {
    g -= p.groups;
    p = f.p[1];
  }
  // workgroups dispatched one after another take residues four groups apart
  // (a rotation of g by two bits): with neighbours side by side in a row
  // the same reads took longer (256 x n = 2^22 FP32 step 3.72 against 3.48
  // ms, 64 signals FP64 1.10 against 1.02 ms, 8 x 2^24 2.92 against 2.87;
  // one to six bits, bit reversal and a signal per XCD gave 3.42-3.73,
  // 1.03-1.19 and 2.86-3.01, none better on all three)
  const int lg = p.logB - p.log_res;
  if (lg > 2) g = ((g << 2) | (g >> (lg - 2))) & (p.groups - 1);
  if (p.fp32) fold_group<true>(a, p, s, g, smem64, sh);
  else fold_group<false>(a, p, s, g, smem64, sh);
}

// ---------------------------------------------------------------- v1 votes
constexpr int kFftPer = 8;  // points per thread of k_bucket_fft_v1 at most

// One block per (signal, location loop): top-num buckets by |.|^2.
// LDS: B doubles.  v1 location loops are always FP64 (xs64): their top-2k
// choice is made among leakage-level bucket powers FP32 cannot resolve.
template <bool GLOBAL>
__global__ void __launch_bounds__(kBlock) k_select(V12Launch a)
{
  extern __shared__ double lds_mag[];
  __shared__ int sh[kTopScratch];
  // above the LDS size the magnitudes go to mag_buf
  double *mag = GLOBAL ? a.mag_buf + (int64_t)blockIdx.x * a.B_loc : lds_mag;
  const int s = blockIdx.x / a.Lloc, l = blockIdx.x % a.Lloc;
  const int B = a.B_loc;
  const int64_t base = (int64_t)s * a.xs + (int64_t)l * a.B_loc;
  const double2 *xs = a.xs64 + base;
  for (int i = threadIdx.x; i < B; i += blockDim.x) {
    const double2 z = xs[i];
    mag[i] = z.x * z.x + z.y * z.y;
  }
  if (GLOBAL) __threadfence_block();
  __syncthreads();
  block_top_num(mag, B, a.num, a.J + ((int64_t)s * a.Lloc + l) * a.num, sh);
}

// v1: the bucket FFTs of every loop in one launch, a location loop's block
// going on to select its top-num buckets from LDS (as k_select, whose launch
// and reads this saves; the location and estimation loops were two
// launches).  One signal, n = 2^20, k = 50: 17 us against 6 + 6 + 13.
// LDS: the largest loop's points.
__global__ void __launch_bounds__(1024) k_bucket_fft_v1(V12Launch a)
{
  extern __shared__ double2 smem64[];
  __shared__ int sh[kTopScratch];
  const int s = blockIdx.x / a.L, l = blockIdx.x % a.L;
  const bool isloc = l < a.Lloc;
  const int B = isloc ? a.B_loc : a.B_est, logB = ilog2(B), T = blockDim.x;
  const int64_t at = (int64_t)s * a.xs + loop_offset(l, a.Lloc, a.B_loc, a.B_est);
  if (!isloc && a.fp32) {
    float2 *buf = reinterpret_cast<float2 *>(smem64), *io = a.xs32 + at;
    slot_fft_fill(buf, logB, [&](int m) { return io[m]; });
    slot_fft(buf, logB, a.tw32, a.tw_nmax / B);
    for (int m = threadIdx.x; m < B; m += T) io[m] = buf[fft_slot<float2>(m, logB)];
    return;
  }
  double2 *io = a.xs64 + at;
  slot_fft_fill(smem64, logB, [&](int m) { return io[m]; });
  slot_fft(smem64, logB, a.tw64, a.tw_nmax / B);
  if (!isloc) {
    for (int m = threadIdx.x; m < B; m += T) io[m] = smem64[fft_slot<double2>(m, logB)];
    return;
  }
  double v[kFftPer];
#pragma unroll
  for (int q = 0; q < kFftPer; q++) {
    const int i = threadIdx.x + q * T;
    if (i < B) {
      const double2 z = smem64[fft_slot<double2>(i, logB)];
      io[i] = z;
      v[q] = z.x * z.x + z.y * z.y;
    }
  }
  __syncthreads();
  double *mag = reinterpret_cast<double *>(smem64);
#pragma unroll
  for (int q = 0; q < kFftPer; q++)
    if (threadIdx.x + q * T < B) mag[threadIdx.x + q * T] = v[q];
  __syncthreads();
  block_top_num(mag, B, a.num, a.J + ((int64_t)s * a.Lloc + l) * a.num, sh);
}

// A frequency f is a hit when, in at least thr of the location loops, its
// permuted position p = f*ai mod n lies in the range
// [ceil((J-1/2) n/B), ceil((J+1/2) n/B)) of a selected bucket J
// (src/computefourier-1.0-2.0.cc:91-116).  Candidates are enumerated from the
// ranges of loops 0..Lloc-thr (candidate c: loop c / (num*m), then selected
// bucket, then offset in the range); a candidate is counted only from the
// first such loop that selects it, so every hit appears once.  The candidate
// list of a signal is cut into chunks of kVoteChunk, one block each:
// k_vote_count counts each chunk's hits, k_vote_write writes the hits in
// candidate order.  LDS: Lloc * B bits of selected-bucket flags
constexpr int kVoteChunk = 8 * kBlock;
static_assert(kVoteChunk == 2048, "vote_chunks() assumes chunks of 2048 candidates");

// Both kernels evaluate a thread's eight candidates together, so that their
// dependent reads overlap.
struct VoteCtx {
  const int *prm, *J;
  const unsigned *selbits;
  int64_t total, per_loop;
  unsigned mask;
  int words, half, logm;
};

__device__ VoteCtx vote_setup(const V12Launch &a, int s, unsigned *selbits)
{
  VoteCtx v;
  const int B = a.B_loc, Lloc = a.Lloc, num = a.num, n = a.n;
  v.words = (B + 31) / 32;
  v.prm = a.params + (int64_t)s * (2 * a.L + max(a.comb_loops, 1));
  v.mask = (unsigned)n - 1;
  v.logm = ilog2(n) - ilog2(B);
  v.half = (1 << v.logm) / 2;
  v.per_loop = (int64_t)num << v.logm;
  v.total = (int64_t)max(Lloc - a.thr + 1, 0) * v.per_loop;
  v.J = a.J + (int64_t)s * Lloc * num;
  v.selbits = selbits;
  for (int i = threadIdx.x; i < Lloc * v.words; i += blockDim.x) selbits[i] = 0;
  __syncthreads();
  for (int l = 0; l < Lloc; l++)
    for (int i = threadIdx.x; i < num; i += blockDim.x) {
      const int b = v.J[l * num + i];
      atomicOr(&selbits[l * v.words + (b >> 5)], 1u << (b & 31));
    }
  __syncthreads();
  return v;
}

// Candidates ch kVoteChunk + i kBlock + threadIdx.x, i < 8: bit i of the
// result says whether it is a hit, loc[i] its frequency.
constexpr int kVotePer = kVoteChunk / kBlock;

__device__ __forceinline__ unsigned vote_keep(const V12Launch &a, const VoteCtx &v, int ch,
                                              unsigned (&loc)[kVotePer])
{
  int l0[kVotePer], score[kVotePer];
  unsigned at[kVotePer], keep = 0, earlier = 0;
#pragma unroll
  for (int i = 0; i < kVotePer; i++) {
    const int64_t c = (int64_t)ch * kVoteChunk + i * kBlock + threadIdx.x;
    keep |= (c < v.total ? 1u : 0u) << i;
    int64_t r = c < v.total ? c : 0;
    int l = 0;
    while (r >= v.per_loop) {  // few loops to start from
      r -= v.per_loop;
      l++;
    }
    l0[i] = l;
    const int jb = v.J[(int64_t)l * a.num + (int)(r >> v.logm)];
    at[i] = (((unsigned)jb << v.logm) - (unsigned)v.half +
             ((unsigned)r & ((1u << v.logm) - 1)) + (unsigned)a.n) & v.mask;
  }
#pragma unroll
  for (int i = 0; i < kVotePer; i++) {
    loc[i] = (at[i] * (unsigned)v.prm[l0[i]]) & v.mask;  // original frequency
    score[i] = 0;
  }
  for (int l = 0; l < a.Lloc; l++) {
    const unsigned ai = (unsigned)v.prm[a.L + l];
#pragma unroll
    for (int i = 0; i < kVotePer; i++) {
      const unsigned bk = ((((loc[i] * ai) & v.mask) + (unsigned)v.half) & v.mask) >> v.logm;
      const int sel = (v.selbits[l * v.words + (bk >> 5)] >> (bk & 31)) & 1;
      score[i] += sel;
      earlier |= (unsigned)((l < l0[i]) & sel) << i;
    }
  }
  unsigned hit = 0;
#pragma unroll
  for (int i = 0; i < kVotePer; i++) hit |= (score[i] >= a.thr ? 1u : 0u) << i;
  return hit & keep & ~earlier;
}

// grid: S x chunks
__global__ void __launch_bounds__(kBlock) k_vote_count(V12Launch a, int chunks)
{
  extern __shared__ unsigned selbits[];
  __shared__ int sh[16];
  const int s = blockIdx.x / chunks, ch = blockIdx.x % chunks;
  const VoteCtx v = vote_setup(a, s, selbits);
  unsigned loc[kVotePer];
  int tot;
  (void)block_exclusive_scan(__popc(vote_keep(a, v, ch, loc)), sh, tot);
  if (threadIdx.x == 0) a.vote_cnt[blockIdx.x] = tot;
}

// grid: S x chunks.  A chunk's hits follow those of the signal's chunks
// before it, whose counts the block sums itself (a scan kernel between the
// two cost a launch); the last chunk writes the located count (at most
// hits_cap).
__global__ void __launch_bounds__(kBlock) k_vote_write(V12Launch a, int chunks)
{
  extern __shared__ unsigned selbits[];
  constexpr int NW = kBlock / 64;
  __shared__ int64_t s_base[NW];
  __shared__ int s_cnt[kVotePer * NW];
  const int s = blockIdx.x / chunks, ch = blockIdx.x % chunks;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int64_t before = 0;
  for (int c = threadIdx.x; c < ch; c += kBlock) before += a.vote_cnt[(int64_t)s * chunks + c];
  const VoteCtx v = vote_setup(a, s, selbits);
  unsigned loc[kVotePer];
  const unsigned keep = vote_keep(a, v, ch, loc);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
  if (lane == 0) s_base[wid] = before;
#pragma unroll
  for (int i = 0; i < kVotePer; i++) {
    const uint64_t b = __ballot((keep >> i) & 1);
    if (lane == 0) s_cnt[i * NW + wid] = __popcll(b);
  }
  __syncthreads();
  int64_t base = 0;
#pragma unroll
  for (int w = 0; w < NW; w++) base += s_base[w];
  int *hits = a.hits + (int64_t)s * a.hits_cap;
#pragma unroll
  for (int i = 0; i < kVotePer; i++) {
    const uint64_t b = __ballot((keep >> i) & 1);
#pragma unroll
    for (int w = 0; w < NW; w++) {
      if (w == wid && ((keep >> i) & 1)) {
        const int64_t pos = base + __popcll(b & ((1ull << lane) - 1));
        if (pos < a.hits_cap) hits[pos] = (int)loc[i];
      }
      base += s_cnt[i * NW + w];
    }
  }
  if (ch == chunks - 1 && threadIdx.x == 0) {
    a.count[s] = min(base, a.hits_cap);
    if (a.count_host) a.count_host[s] = min(base, a.hits_cap);
  }
}

// ---------------------------------------------------------------- v2 votes (diagnostic)
// The v2 location votes (src/computefourier-1.0-2.0.cc:125-184), which never
// change the output (every frequency they append is already in the comb
// prefill), counted for parity tests.  The reference walks, for location
// loop l and selected bucket J, the positions of the range
// [ceil((J-1/2) n/B), ceil((J+1/2) n/B)) in the classes of the comb residues,
// adds one to score[h] of the frequency h = position * a mod n and appends h
// when its score reaches thr.  Those frequencies are the located set
// {j W + c}; a frequency's score after loop l is the number of loops <= l
// whose selected buckets hold h * ai mod n.  One thread per located
// frequency (prefill order) writes its append key -- (loop where the score
// reaches thr, rank of that bucket in J, offset of the position in the
// range), the order of the reference's appends -- or -1.
__global__ void __launch_bounds__(kBlock) k_comb_vote_keys(V12Launch a, int64_t chunks,
                                                          int64_t *keys, int64_t stride)
{
  extern __shared__ unsigned selbits[];
  const int s = (int)(blockIdx.x / chunks);
  const int64_t t = (blockIdx.x % chunks) * kBlock + threadIdx.x;
  const int B = a.B_loc, Lloc = a.Lloc, num = a.num;
  const int words = (B + 31) / 32;
  const int *J = a.J + (int64_t)s * Lloc * num;
  for (int i = threadIdx.x; i < Lloc * words; i += blockDim.x) selbits[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < Lloc * num; i += blockDim.x) {
    const int l = i / num, b = J[i];
    atomicOr(&selbits[l * words + (b >> 5)], 1u << (b & 31));
  }
  __syncthreads();
  const int nc = a.num_comb[s];
  const int64_t located = (int64_t)nc * (a.n / a.W);
  if (t >= a.est_cap) return;
  if (t >= located) {  // capacity past the located set (several comb loops)
    keys[(int64_t)s * stride + 2 * t] = -1;
    keys[(int64_t)s * stride + 2 * t + 1] = -1;
    return;
  }
  const int *prm = a.params + (int64_t)s * (2 * a.L + max(a.comb_loops, 1));
  const unsigned mask = (unsigned)a.n - 1;
  const int m = a.n / B, half = m / 2, logm = ilog2(m);
  const unsigned h = (unsigned)(t / nc) * (unsigned)a.W +
                     (unsigned)a.approved[(int64_t)s * a.comb_loops * num + t % nc];
  int64_t key = -1;
  int score = 0;
  for (int l = 0; l < Lloc && key < 0; l++) {
    const unsigned p = (h * (unsigned)prm[a.L + l]) & mask;
    const unsigned bk = ((p + (unsigned)half) & mask) >> logm;
    const unsigned *sb = selbits + l * words;
    if (!((sb[bk >> 5] >> (bk & 31)) & 1)) continue;
    if (++score < a.thr) continue;
    int rank = __popc(sb[bk >> 5] & ((1u << (bk & 31)) - 1));
    for (unsigned wd = 0; wd < (bk >> 5); wd++) rank += __popc(sb[wd]);
    const unsigned low = (bk * (unsigned)m - (unsigned)half + (unsigned)a.n) & mask;
    key = (int64_t)l << 48 | (int64_t)rank << 28 | (int64_t)((p - low) & mask);
  }
  keys[(int64_t)s * stride + 2 * t] = key;
  keys[(int64_t)s * stride + 2 * t + 1] = (int64_t)h;
}

// ---------------------------------------------------------------- estimate
// Per located frequency h and loop l: the bucket h hashes to, divided by the
// filter response at h's offset from the bucket centre (a half-bucket tie
// rounds down, cf12 371-378); then the lower median (rank (L-1)/2) of the
// real and imaginary parts separately (cf12 406-413).
//
// Blocks are mapped so that every block of one signal lands on the same XCD
// (workgroups are dispatched round-robin over the 8 XCDs): the signal's
// buckets then stay in that XCD's L2 while its located set is estimated.
constexpr int kXcds = 8;

__device__ __forceinline__ bool xcd_block(int64_t b, int S, int64_t per_signal,
                                          int &s, int64_t &c)
{
  if (S < kXcds) {  // too few signals to give each XCD its own: spread them
    s = (int)(b / per_signal);
    c = b % per_signal;
    return s < S;
  }
  const int x = (int)(b % kXcds);
  const int64_t q = b / kXcds;
  s = x + kXcds * (int)(q / per_signal);
  c = q % per_signal;
  return s < S;
}

__host__ __device__ inline int64_t xcd_grid(int S, int64_t per_signal)
{
  return S < kXcds ? (int64_t)S * per_signal
                   : (int64_t)((S + kXcds - 1) / kXcds) * kXcds * per_signal;
}

__host__ __device__ constexpr int pow2_at_least(int v)
{
  return v <= 1 ? 1 : 2 * pow2_at_least((v + 1) / 2);
}

// Ascending sort of v[0..LMAX) with Batcher's odd-even merge network on the
// next power of two; comparators that touch a slot >= LMAX compare with an
// implicit +inf and are dropped at compile time.
template <int LMAX>
__device__ __forceinline__ void sort_net(double (&v)[LMAX])
{
  constexpr int N = pow2_at_least(LMAX);
#pragma unroll
  for (int p = 1; p < N; p <<= 1) {
#pragma unroll
    for (int k = p; k >= 1; k >>= 1) {
#pragma unroll
      for (int j = k % p; j + k < N; j += 2 * k) {
#pragma unroll
        for (int i = 0; i < k; i++) {
          const int lo = i + j, hi = i + j + k;
          if (hi < LMAX && i < N - j - k && lo / (2 * p) == hi / (2 * p)) {
            const double x = fmin(v[lo], v[hi]), y = fmax(v[lo], v[hi]);
            v[lo] = x;
            v[hi] = y;
          }
        }
      }
    }
  }
}

// Ascending sort of v[O..O+10) with a 29-comparator 10-input network
// (every 0-1 input checked).
template <int LMAX, int O>
__device__ __forceinline__ void sort10(double (&v)[LMAX])
{
  constexpr int net[29][2] = {{4, 9}, {3, 8}, {2, 7}, {1, 6}, {0, 5}, {1, 4}, {6, 9}, {0, 3},
                              {5, 8}, {0, 2}, {3, 6}, {7, 9}, {0, 1}, {2, 4}, {5, 7}, {8, 9},
                              {1, 2}, {4, 6}, {7, 8}, {3, 5}, {2, 5}, {6, 8}, {1, 3}, {4, 7},
                              {2, 3}, {6, 7}, {3, 4}, {5, 6}, {4, 5}};
#pragma unroll
  for (int c = 0; c < 29; c++) {
    const int lo = O + net[c][0], hi = O + net[c][1];
    const double x = fmin(v[lo], v[hi]), y = fmax(v[lo], v[hi]);
    v[lo] = x;
    v[hi] = y;
  }
}

// Lower median (rank 9) of 20 values: with both halves sorted, the 10th
// smallest of their union is max_i min(A[i], B[9-i]).
template <int LMAX>
__device__ __forceinline__ double median20(double (&v)[LMAX])
{
  sort10<LMAX, 0>(v);
  sort10<LMAX, 10>(v);
  double m = fmin(v[0], v[19]);
#pragma unroll
  for (int i = 1; i < 10; i++) m = fmax(m, fmin(v[i], v[19 - i]));
  return m;
}

// Lower median (rank (L-1)/2) of v[0..L), slots past L holding +inf.
template <int LMAX>
__device__ __forceinline__ double lower_median1(double (&v)[LMAX], int L)
{
  if constexpr (LMAX == 20) {
    if (L == 20) return median20<LMAX>(v);
  }
  sort_net<LMAX>(v);
  const int rank = (L - 1) / 2;
  double m = v[0];
#pragma unroll
  for (int l = 1; l < LMAX; l++)
    if (l == rank) m = v[l];
  return m;
}

template <int LMAX>
__device__ __forceinline__ double2 lower_median(double (&vr)[LMAX], double (&vi)[LMAX],
                                                int L)
{
  const double re = lower_median1<LMAX>(vr, L);
  return make_double2(re, lower_median1<LMAX>(vi, L));
}

__device__ __forceinline__ double2 load_bucket(const V12Launch &a, bool fp32, bool isloc,
                                               int64_t idx)
{
  if (fp32 && !(a.loc64 && isloc)) {
    const float2 u = a.xs32[idx];
    return make_double2((double)u.x, (double)u.y);
  }
  return a.xs64[idx];
}

// load_bucket without a branch between the precisions (two 8-byte words
// wherever they lie), so that several can be in flight.
template <bool FP32>
__device__ __forceinline__ double2 raw_bucket(const V12Launch &a, bool isloc, int64_t idx)
{
  if constexpr (!FP32) {
    return a.xs64[idx];
  } else {
    const bool wide = a.loc64 && isloc;
    const double *p = wide ? reinterpret_cast<const double *>(a.xs64 + idx)
                           : reinterpret_cast<const double *>(a.xs32 + idx);
    const double w0 = p[0], w1 = p[wide ? 1 : 0];
    const float fx = __int_as_float(__double2loint(w0)), fy = __int_as_float(__double2hiint(w0));
    return wide ? make_double2(w0, w1) : make_double2((double)fx, (double)fy);
  }
}

// bucket / G with the reference's operation order (division by |G|^2)
__device__ __forceinline__ void divide_by_filter(double2 U, double2 G, double den,
                                                 bool conj, double &vr, double &vi)
{
  vr = (U.x * G.x + U.y * G.y) / den;
  vi = conj ? (U.x * G.y - U.y * G.x) / den : (U.y * G.x - U.x * G.y) / den;
}

// FP32 form: bucket u times g = G / |G|^2, one complex multiply instead of
// two divisions, each part one product and one fused multiply-add.  sign
// (V12Launch::conj_sign) is 1.0 for the reference's conjugated estimate and
// -1.0 for the other, whose imaginary part is the exact negation; it is a
// launch argument rather than a select on ref_conj, so the negation stays
// one multiplication.  Every FP32 estimation path calls this, so they
// agree bit for bit.
__device__ __forceinline__ void mul_by_inverse(double ux, double uy, double2 g, double sign,
                                               double &vr, double &vi)
{
  vr = fma(ux, g.x, uy * g.y);
  vi = sign * fma(ux, g.y, -(uy * g.x));
}

// Bucket and filter value of frequency h in loop l, computed directly.
__device__ __forceinline__ void hash_direct(const V12Launch &a, int l, unsigned ai,
                                            unsigned h, int &hashed, double2 &G)
{
  const bool isloc = l < a.Lloc;
  const int B = isloc ? a.B_loc : a.B_est;
  const int logm = ilog2(a.n) - ilog2(B), m = 1 << logm;
  const unsigned p = (ai * h) & ((unsigned)a.n - 1);
  hashed = (int)(p >> logm);
  int dist = (int)(p & (unsigned)(m - 1));
  if (dist > m / 2) {
    hashed = (hashed + 1) & (B - 1);
    dist -= m;
  }
  G = (isloc ? a.win_loc : a.win_est)[dist + m / 2];
}

__device__ __forceinline__ void write_result(const V12Launch &a, int s, int64_t t,
                                             unsigned h, double2 val)
{
  if (a.o_freq && t < a.o_cap) {
    int32_t *of = a.o_freq[s];
    double2 *ov = a.o_val[s];
    if (of) of[t] = (int32_t)h;
    if (ov) ov[t] = val;
  }
  if (a.o_dense) {
    double2 *od = a.o_dense[s];
    if (od) od[h] = val;
  }
}

// v2: the located set is h = j*W + c for the comb residues c (in the
// reference's prefill order t = j*num_comb + i).  When W is a multiple of
// m = n/B, every h with the same residue has the same offset from its
// bucket centre and its bucket advances by (ai*W/m) mod B per alias row j,
// so the filter value and base bucket are tabulated per (residue, loop).
// Block tile: kTI residues x kTJ alias rows, kTI*kTJ/256 hits per thread.
constexpr int kTI = 64, kTJ = 16;

template <int LMAX, bool FP32, bool ALLFAST>
__global__ void __launch_bounds__(kBlock) k_estimate_comb(V12Launch a, int tiles_i,
                                                          int tiles_j)
{
  __shared__ int t_hash[kTI * LMAX];
  __shared__ double2 t_g[kTI * LMAX];
  __shared__ double t_den[FP32 ? 1 : kTI * LMAX];
  __shared__ unsigned s_ai[LMAX];
  __shared__ unsigned s_step[LMAX];
  __shared__ unsigned s_mask[LMAX];
  __shared__ int s_off[LMAX];
  int s;
  int64_t c;
  if (!xcd_block(blockIdx.x, a.S, (int64_t)tiles_i * tiles_j, s, c)) return;
  const int ti = (int)(c % tiles_i), tj = (int)(c / tiles_i);
  const int nc = a.num_comb[s];
  const int rows = a.n / a.W;
  if (ti * kTI >= nc || tj * kTJ >= rows) return;
  const int L = a.L;
  const int stride = 2 * L + max(a.comb_loops, 1);
  const int *approved = a.approved + (int64_t)s * a.comb_loops * a.num;
  if (threadIdx.x < L) {
    const int l = threadIdx.x;
    const unsigned ai = (unsigned)a.params[(int64_t)s * stride + L + l];
    const int B = l < a.Lloc ? a.B_loc : a.B_est;
    const int m = a.n / B;
    s_ai[l] = ai;
    s_mask[l] = (unsigned)(B - 1);
    s_off[l] = (int)loop_offset(l, a.Lloc, a.B_loc, a.B_est);
    // 0 marks a loop whose W is not a multiple of m (direct hashing)
    s_step[l] = (a.W % m == 0) ? ((ai * (unsigned)(a.W / m)) & (unsigned)(B - 1)) | 0x80000000u
                               : 0u;
  }
  __syncthreads();
  if (ALLFAST) {
    // every loop tabulated: a lean loop body with per-loop scalars in LDS
    for (int e = threadIdx.x; e < kTI * L; e += blockDim.x) {
      const int l = e / kTI, il = e % kTI;  // consecutive threads: consecutive il
      const int i = ti * kTI + il;
      if (i < nc) {
        int hashed;
        double2 G;
        hash_direct(a, l, s_ai[l], (unsigned)approved[i], hashed, G);
        const double den = G.x * G.x + G.y * G.y;
        t_hash[l * kTI + il] = hashed;
        if (FP32) {
          t_g[l * kTI + il] = make_double2(G.x / den, G.y / den);
        } else {
          t_g[l * kTI + il] = G;
          t_den[l * kTI + il] = den;
        }
      }
    }
    __syncthreads();
    const double2 *xs64 = a.xs64 + (int64_t)s * a.xs;
    const float2 *xs32 = FP32 ? a.xs32 + (int64_t)s * a.xs : nullptr;
    const bool conj = a.ref_conj;
    const double sign = a.conj_sign;
    for (int e = threadIdx.x; e < kTI * kTJ; e += kBlock) {
      // re-read the per-loop scalars from LDS every hit instead of holding
      // 3 x LMAX of them in registers across the loop (occupancy)
      asm volatile("" ::: "memory");
      const int jl = e / kTI;
      const int il = (e + jl) % kTI;  // skew: see below
      const int i = ti * kTI + il;
      const int j = tj * kTJ + jl;
      // hits past the tile's edge run too (clamped indices, nothing
      // written) so that every thread reaches the barriers below
      const bool valid = i < nc && j < rows;
      const int ic = min(i, nc - 1), jc = min(j, rows - 1);
      const unsigned h = (unsigned)jc * (unsigned)a.W + (unsigned)approved[ic];
      double vr[LMAX], vi[LMAX];
#pragma unroll
      for (int l = 0; l < LMAX; l++) {
        if (l < L) {
          const int hashed =
              (int)(((unsigned)t_hash[l * kTI + il] + (unsigned)jc * (s_step[l] & 0x7fffffffu)) &
                    s_mask[l]);
          const double2 g = t_g[l * kTI + il];
          double2 U;
          if (FP32) {
            const float2 u = xs32[s_off[l] + hashed];
            mul_by_inverse((double)u.x, (double)u.y, g, sign, vr[l], vi[l]);
          } else {
            U = xs64[s_off[l] + hashed];
            const double den = t_den[l * kTI + il];
            divide_by_filter(U, g, den, conj, vr[l], vi[l]);
          }
        } else {
          vr[l] = __longlong_as_double(0x7ff0000000000000ll);  // +inf pads
          vi[l] = vr[l];
        }
        // every 4 loops the block's wavefronts meet, so that they read the
        // same loops' bucket arrays together (L1 reuse; measured -7%)
        if (l % 4 == 3) __syncthreads();
      }
      const double2 med = lower_median<LMAX>(vr, vi, L);
      if (valid) write_result(a, s, (int64_t)j * nc + i, h, med);
    }
    return;
  }
  for (int e = threadIdx.x; e < kTI * L; e += blockDim.x) {
    const int l = e / kTI, il = e % kTI;  // consecutive threads: consecutive il
    const int i = ti * kTI + il;
    if (i < nc && (s_step[l] & 0x80000000u)) {
      int hashed;
      double2 G;
      hash_direct(a, l, s_ai[l], (unsigned)approved[i], hashed, G);
      const double den = G.x * G.x + G.y * G.y;
      t_hash[l * kTI + il] = hashed;
      if (FP32) {
        t_g[l * kTI + il] = make_double2(G.x / den, G.y / den);
      } else {
        t_g[l * kTI + il] = G;
        t_den[l * kTI + il] = den;
      }
    }
  }
  __syncthreads();
  const int64_t sbase = (int64_t)s * a.xs;
  // Hit e of the tile: row jl = e / kTI, residue il skewed by the row so that
  // a thread's table entries change from hit to hit (keeps them in LDS rather
  // than hoisted into registers) while a wavefront still writes consecutive
  // output slots.
  for (int e = threadIdx.x; e < kTI * kTJ; e += kBlock) {
    const int jl = e / kTI;
    const int il = (e + jl) % kTI;
    const int i = ti * kTI + il;
    const int j = tj * kTJ + jl;
    if (i >= nc || j >= rows) continue;
    const unsigned h = (unsigned)j * (unsigned)a.W + (unsigned)approved[i];
    double vr[LMAX], vi[LMAX];
#pragma unroll
    for (int l = 0; l < LMAX; l++) {
      if (l < L) {
        const bool isloc = l < a.Lloc;
        const int B = isloc ? a.B_loc : a.B_est;
        const int64_t off = sbase + loop_offset(l, a.Lloc, a.B_loc, a.B_est);
        const unsigned step = s_step[l];
        if (step & 0x80000000u) {
          const int hashed = (t_hash[l * kTI + il] +
                              (int)(((unsigned)j * (step & 0x7fffffffu)) & (unsigned)(B - 1))) &
                             (B - 1);
          const double2 U = load_bucket(a, FP32, isloc, off + hashed);
          const double2 g = t_g[l * kTI + il];
          if (FP32) {
            mul_by_inverse(U.x, U.y, g, a.conj_sign, vr[l], vi[l]);
          } else {
            divide_by_filter(U, g, t_den[l * kTI + il], a.ref_conj, vr[l], vi[l]);
          }
        } else {
          int hashed;
          double2 G;
          hash_direct(a, l, s_ai[l], h, hashed, G);
          const double2 U = load_bucket(a, FP32, isloc, off + hashed);
          divide_by_filter(U, G, G.x * G.x + G.y * G.y, a.ref_conj, vr[l], vi[l]);
        }
      } else {
        vr[l] = __longlong_as_double(0x7ff0000000000000ll);  // +inf pads
        vi[l] = vr[l];
      }
    }
    write_result(a, s, (int64_t)j * nc + i, h, lower_median<LMAX>(vr, vi, L));
  }
}

// ------------------------------------------------------ v2: alias-row layout
// With W a multiple of m = n/B, frequency h = j*W + c of comb residue c
// lies in bucket hashed0(c) + j*ai*d (mod B) of a loop, d = W/m, for its
// alias rows j < rows = n/W = B/d.  Stored at position r*rows + (q * u^-1
// mod rows) for bucket b = r + d*q (u = ai mod rows, odd), the buckets of
// rows j, j+1, ... of one residue are adjacent: a wavefront of 64 rows reads
// 512 contiguous bytes instead of 64 scattered lines.  The products and the
// median are the same as in k_estimate_comb, so the results are identical.

// inverse of odd a modulo 2^32 (Newton's iteration from a*a = 1 mod 8)
__device__ __forceinline__ unsigned inv_odd(unsigned a)
{
  unsigned x = a;
#pragma unroll
  for (int i = 0; i < 4; i++) x *= 2u - a * x;
  return x;
}

// Per (signal, residue, loop): where the residue's bucket row lies and what
// its buckets are multiplied or divided by.  Written once per batch; the
// workgroups of k_estimate_rows copy their residues'
// entries to LDS (computing them there cost every 64 rows' workgroup the
// hashing and the quotients again).
struct RowEntry32 {
  double gx, gy;    // G / |G|^2
  unsigned off, q;  // byte offsets: loop l's row r; the residue's place in it
};
struct RowEntry64 {
  double gx, gy;    // G
  double den, inv;  // |G|^2 and its reciprocal
  unsigned off, q;  // as above; bit 31 of q: not to be divided by inv
};

// Entry t = (signal, residue slot, loop).
template <bool FP32>
__device__ __forceinline__ void rows_entry(const V12Launch &a, int64_t t)
{
  using Entry = typename std::conditional<FP32, RowEntry32, RowEntry64>::type;
  constexpr unsigned kElt = FP32 ? sizeof(float2) : sizeof(double2);
  const int L = a.L, cap = a.comb_loops * a.num;
  if (t >= (int64_t)a.S * cap * L) return;
  const int l = (int)(t % L);
  const int64_t si = t / L;
  const int s = (int)(si / cap), i = (int)(si % cap);
  if (i >= a.num_comb[s]) return;
  const unsigned ai =
      (unsigned)a.params[(int64_t)s * (2 * L + max(a.comb_loops, 1)) + L + l];
  int hashed;
  double2 G;
  hash_direct(a, l, ai, (unsigned)a.approved[si], hashed, G);
  const int rows = a.n / a.W;
  const int B = l < a.Lloc ? a.B_loc : a.B_est;
  const int d = B / rows;
  const unsigned uinv = inv_odd(ai) & (unsigned)(rows - 1);
  const double den = G.x * G.x + G.y * G.y;
  Entry e;
  e.off = (unsigned)(loop_offset(l, a.Lloc, a.B_loc, a.B_est) + (hashed % d) * rows) * kElt;
  e.q = (((unsigned)(hashed / d) * uinv) & (unsigned)(rows - 1)) * kElt;
  if constexpr (FP32) {
    e.gx = G.x / den;
    e.gy = G.y / den;
  } else {
    e.gx = G.x;
    e.gy = G.y;
    e.den = den;
    e.inv = 1.0 / den;
    const bool near1 = den >= 0x1p-100 && den <= 0x1p100 &&
                       (G.x == 0.0 || fabs(G.x) >= 0x1p-100) &&
                       (G.y == 0.0 || fabs(G.y) >= 0x1p-100);
    if (!near1) e.q |= 0x80000000u;
  }
  reinterpret_cast<Entry *>(a.rows_tab)[t] = e;
}

// The entries in a launch of their own, after a comb on the second stream.
template <bool FP32>
__global__ void __launch_bounds__(kBlock) k_rows_table(V12Launch a)
{
  rows_entry<FP32>(a, (int64_t)blockIdx.x * kBlock + threadIdx.x);
}

// Zero or of a magnitude whose quotients by a filter power near one neither
// overflow nor lose bits to underflow on the way (false for infinities and
// NaN): the FP64 estimate divides such buckets by a tabulated reciprocal.
__device__ __forceinline__ bool plain_value(double v)
{
  const double m = fabs(v);
  return m == 0.0 || (m >= 0x1p-700 && m <= 0x1p700);
}

// Bucket FFTs of loops [l0, l0 + nl), written in the alias-row layout.
// FP64: rows_odd[s L + l] says whether any bucket is not a plain value.
// The workgroups past the transforms write the estimation entries, one a
// thread, when the comb is done by now (a launch of their own cost a single
// signal 4 us).
template <bool FP32>
__global__ void __launch_bounds__(1024) k_bucket_fft_rows(V12Launch a, int l0, int nl)
{
  using T2 = typename std::conditional<FP32, float2, double2>::type;
  extern __shared__ char rraw[];
  T2 *rbuf = reinterpret_cast<T2 *>(rraw);
  if (blockIdx.x >= (unsigned)(a.S * nl)) {
    rows_entry<FP32>(a, (int64_t)(blockIdx.x - (unsigned)(a.S * nl)) * blockDim.x + threadIdx.x);
    return;
  }
  const int s = blockIdx.x / nl, l = l0 + blockIdx.x % nl;
  const int B = l < a.Lloc ? a.B_loc : a.B_est;
  const int logB = ilog2(B);
  const int rows = a.n / a.W, d = B / rows;
  const int stride = 2 * a.L + max(a.comb_loops, 1);
  const unsigned ai = (unsigned)a.params[(int64_t)s * stride + a.L + l];
  const unsigned uinv = inv_odd(ai) & (unsigned)(rows - 1);
  T2 *io;
  if constexpr (FP32) io = a.xs32; else io = a.xs64;
  io += (int64_t)s * a.xs + loop_offset(l, a.Lloc, a.B_loc, a.B_est);
  slot_fft_fill(rbuf, logB, [&](int m) { return io[m]; });
  if constexpr (FP32) slot_fft(rbuf, logB, a.tw32, a.tw_nmax / B);
  else slot_fft(rbuf, logB, a.tw64, a.tw_nmax / B);
  int odd = 0;
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    const int r = b % d, q = b / d;
    const T2 z = rbuf[fft_slot<T2>(b, logB)];
    if (!FP32) odd |= !plain_value(z.x) | !plain_value(z.y);
    io[r * rows + (int)(((unsigned)q * uinv) & (unsigned)(rows - 1))] = z;
  }
  if (!FP32) {
    odd = __syncthreads_or(odd);
    if (threadIdx.x == 0) a.rows_odd[(int64_t)s * a.L + l] = odd;
  }
}

// Residues per tile of k_estimate_rows (RI / 4 per wavefront): 16 for
// batches, 4 when a batch gives too few tiles to fill the chip.
constexpr int kRI = 16, kRIsmall = 4;

// RN(a / den) from inv = RN(1 / den): q0 is within 1.5 ulp of the quotient,
// its residual is exact to 2^-53 of itself, and where the quotient lies next
// to a rounding midpoint q0 is half an ulp away, so the corrected sum lies
// on the quotient's side of the midpoint (Markstein).  Holds while nothing
// over- or underflows: see plain_value.  The residual is formed negated and
// multiplied by -inv: for a = -0 the product is then -0, which leaves q0 = -0
// as it is, where a - den q0 = +0 would turn it into +0 (the same
// instructions; the signs are operand modifiers).
__device__ __forceinline__ double div_by(double a, double den, double inv)
{
  const double q0 = a * inv;
  return fma(fma(den, q0, -a), -inv, q0);
}

// v, negated where flip is the sign bit (exact; an integer operation)
__device__ __forceinline__ double flip_sign(double v, unsigned flip)
{
  return __hiloint2double(__double2hiint(v) ^ (int)flip, __double2loint(v));
}

// Bucket of entry e at byte jm of the alias rows: a row starts on a multiple
// of its length, so the place within it is or-ed on.
template <typename T2, typename Entry>
__device__ __forceinline__ T2 row_bucket(const char *xs, const Entry &e, unsigned jm,
                                         unsigned row_mask)
{
  return *reinterpret_cast<const T2 *>(xs + (((e.q + jm) & row_mask) | e.off));
}

// Median value of one residue at the byte offset jm of its alias row; tab:
// the residue's L entries in LDS, xs: the signal's buckets.
template <int LMAX, bool FULL>
__device__ __forceinline__ double2 rows_median(const char *xs, const RowEntry32 *tab, unsigned jm,
                                               unsigned row_mask, int L, unsigned flip, bool)
{
  double vr[LMAX], vi[LMAX];
#pragma unroll
  for (int l = 0; l < LMAX; l++) {
    if (FULL || l < L) {
      const RowEntry32 e = tab[l];
      const float2 u = row_bucket<float2>(xs, e, jm, row_mask);
      const double ux = (double)u.x, uy = (double)u.y;
      vr[l] = fma(ux, e.gx, uy * e.gy);  // as mul_by_inverse
      vi[l] = flip_sign(fma(ux, e.gy, -(uy * e.gx)), flip);
    } else {
      vr[l] = __longlong_as_double(0x7ff0000000000000ll);  // +inf pads
      vi[l] = vr[l];
    }
  }
  return lower_median<LMAX>(vr, vi, FULL ? LMAX : L);
}

// The imaginary numerator of divide_by_filter: u.x gy - u.y gx, or with flip
// (the unconjugated estimate) u.y gx - u.x gy, the same difference of
// products with their signs flipped (a flipped result would turn a zero
// difference's +0 into -0).
__device__ __forceinline__ double imag_part(double2 u, const RowEntry64 &e, unsigned flip)
{
  return flip_sign(u.x, flip) * e.gy - flip_sign(u.y, flip) * e.gx;
}

// FP64: the reference's operation order (cf12 383-398); odd: with divisions,
// one part and one quotient at a time (rare, so with few registers).
template <int LMAX, bool FULL>
__device__ __forceinline__ double2 rows_median(const char *xs, const RowEntry64 *tab, unsigned jm,
                                               unsigned row_mask, int L, unsigned flip, bool odd)
{
  if (!odd) {
    double vr[LMAX], vi[LMAX];
#pragma unroll
    for (int l = 0; l < LMAX; l++) {
      if (FULL || l < L) {
        const RowEntry64 e = tab[l];
        const double2 u = row_bucket<double2>(xs, e, jm, row_mask);
        vr[l] = div_by(u.x * e.gx + u.y * e.gy, e.den, e.inv);
        vi[l] = div_by(imag_part(u, e, flip), e.den, e.inv);
      } else {
        vr[l] = __longlong_as_double(0x7ff0000000000000ll);
        vi[l] = vr[l];
      }
    }
    return lower_median<LMAX>(vr, vi, FULL ? LMAX : L);
  }
  double part[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    double v[LMAX];
#pragma unroll
    for (int l = 0; l < LMAX; l++) {
      if (FULL || l < L) {
        const RowEntry64 e = tab[l];
        const double2 u = row_bucket<double2>(xs, e, jm, row_mask);
        v[l] = (c == 0 ? u.x * e.gx + u.y * e.gy : imag_part(u, e, flip)) / e.den;
      } else {
        v[l] = __longlong_as_double(0x7ff0000000000000ll);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    part[c] = lower_median1<LMAX>(v, FULL ? LMAX : L);
  }
  return make_double2(part[0], part[1]);
}

// FULL: L == LMAX, so the loop over loops has no branch and the compiler
// issues all bucket loads of a frequency before the first wait.
template <int LMAX, bool FULL, bool FP32, int RI>
__global__ void __launch_bounds__(kBlock) k_estimate_rows(V12Launch a, int tiles_i, int tiles_j)
{
  using T2 = typename std::conditional<FP32, float2, double2>::type;
  using Entry = typename std::conditional<FP32, RowEntry32, RowEntry64>::type;
  __shared__ double2 stage[64 * (RI + 1)];  // [row][residue], padded
  __shared__ Entry tab[RI * LMAX];
  __shared__ int s_odd;
  int s;
  int64_t c;
  if (!xcd_block(blockIdx.x, a.S, (int64_t)tiles_i * tiles_j, s, c)) return;
  const int ti = (int)(c % tiles_i), tj = (int)(c / tiles_i);
  const int nc = a.num_comb[s];
  const int rows = a.n / a.W;
  if (ti * RI >= nc) return;
  const int L = a.L;
  const int cap = a.comb_loops * a.num;
  const int *approved = a.approved + (int64_t)s * cap;
  {
    // the tile's entries, contiguous in the table, copied as 8-byte words
    const int cnt = min(RI, nc - ti * RI) * L * (int)(sizeof(Entry) / 8);
    const uint64_t *src = reinterpret_cast<const uint64_t *>(
        reinterpret_cast<const Entry *>(a.rows_tab) + ((int64_t)s * cap + ti * RI) * L);
    uint64_t *dst = reinterpret_cast<uint64_t *>(tab);
    int odd = 0;
    for (int e = threadIdx.x; e < cnt; e += blockDim.x) {
      const uint64_t w = src[e];
      dst[e] = w;
      if (!FP32 && e % (int)(sizeof(Entry) / 8) == (int)(sizeof(Entry) / 8) - 1)
        odd |= (int)(w >> 63);
    }
    if (!FP32) {
      if ((int)threadIdx.x < L) odd |= a.rows_odd[(int64_t)s * L + threadIdx.x];
      if (threadIdx.x == 0) s_odd = 0;
      __syncthreads();
      if (odd) s_odd = 1;
    }
    __syncthreads();
  }
  const T2 *xsig;
  if constexpr (FP32) xsig = a.xs32 + (int64_t)s * a.xs;
  else xsig = a.xs64 + (int64_t)s * a.xs;
  const char *xs = reinterpret_cast<const char *>(xsig);
  const bool odd = !FP32 && s_odd;
  const unsigned flip = a.ref_conj ? 0u : 0x80000000u;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned row_mask = (unsigned)(rows - 1) * (unsigned)sizeof(T2);
  const unsigned jm = (unsigned)(tj * 64 + lane) * (unsigned)sizeof(T2);  // an alias row a lane
  for (int q = 0; q < RI / 4; q++) {
    asm volatile("" ::: "memory");
    const int il = wid * (RI / 4) + q;  // one residue per wavefront
    if (ti * RI + il >= nc) break;      // wave-uniform; no barrier inside
    stage[lane * (RI + 1) + il] =
        rows_median<LMAX, FULL>(xs, tab + il * L, jm, row_mask, L, flip, odd);
  }
  __syncthreads();
  // row by row: RI consecutive output slots per row
  for (int e = threadIdx.x; e < 64 * RI; e += blockDim.x) {
    const int jr = e / RI, il = e % RI;
    const int i = ti * RI + il, jj = tj * 64 + jr;
    if (i < nc && jj < rows)
      write_result(a, s, (int64_t)jj * nc + i, (unsigned)jj * (unsigned)a.W + (unsigned)approved[i],
                   stage[jr * (RI + 1) + il]);
  }
}

// v1: one thread per hit of the vote list.  Few hits, so bound by the reads'
// latency: kHitAhead loops' reads are issued together.
constexpr int kHitAhead = 4;  // divides every median network's size
template <int LMAX, bool FP32>
__global__ void __launch_bounds__(kBlock) k_estimate_hits(V12Launch a, int64_t chunks)
{
  __shared__ unsigned s_ai[LMAX];
  int s;
  int64_t c;
  if (!xcd_block(blockIdx.x, a.S, chunks, s, c)) return;
  const int L = a.L;
  const int stride = 2 * L + max(a.comb_loops, 1);
  if (threadIdx.x < L)
    s_ai[threadIdx.x] = (unsigned)a.params[(int64_t)s * stride + L + threadIdx.x];
  __syncthreads();
  const int64_t t = c * blockDim.x + threadIdx.x;
  if (t >= a.count[s]) return;
  const unsigned h = (unsigned)a.hits[(int64_t)s * a.hits_cap + t];
  const int64_t sbase = (int64_t)s * a.xs;
  double vr[LMAX], vi[LMAX];
#pragma unroll
  for (int l0 = 0; l0 < LMAX; l0 += kHitAhead) {
    // buckets and filter values of kHitAhead loops in flight (past L: the
    // last loop's again, unused)
    double2 U[kHitAhead], G[kHitAhead];
#pragma unroll
    for (int u = 0; u < kHitAhead; u++) {
      const int l = min(l0 + u, L - 1);
      const bool isloc = l < a.Lloc;
      int hashed;
      hash_direct(a, l, s_ai[l], h, hashed, G[u]);
      U[u] = raw_bucket<FP32>(a, isloc,
                              sbase + loop_offset(l, a.Lloc, a.B_loc, a.B_est) + hashed);
    }
#pragma unroll
    for (int u = 0; u < kHitAhead; u++) {
      const int l = l0 + u;
      if (l < L) {
        divide_by_filter(U[u], G[u], G[u].x * G[u].x + G[u].y * G[u].y, a.ref_conj, vr[l], vi[l]);
      } else {
        vr[l] = __longlong_as_double(0x7ff0000000000000ll);
        vi[l] = vr[l];
      }
    }
  }
  write_result(a, s, t, h, lower_median<LMAX>(vr, vi, L));
}

__global__ void k_zero(double2 *out, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t j = i; j < n; j += stride) out[j] = make_double2(0.0, 0.0);
}

// Kernels whose dynamic LDS can exceed the default 64 KiB opt in to the
// device maximum (once per kernel; see raise_lds_limit).
template <typename K>
void allow_lds(K kernel, size_t bytes)
{
  if (bytes > 65536) raise_lds_limit(reinterpret_cast<const void *>(kernel));
}

int launched(const char *what)
{
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return -1;
  }
  return 0;
}

int launch_failed(const char *what)
{
  const hipError_t e = hipGetLastError();
  set_error(std::string(what) + ": " + (e != hipSuccess ? hipGetErrorString(e)
                                                         : "invalid transform shape"));
  return -1;
}

}  // namespace

// ---------------------------------------------------------------- scratch
// Device memory of the allocation-free exec (sfft_exec_sparse_noalloc): the
// workspace of one signal is carved from it instead of allocated.  Every GPU
// the library runs on holds its own copy for the life of the process.  In
// host code `scratch` is only a stand-in for the symbol: its device address
// comes from hipGetSymbolAddress, once per device, and only that address is
// passed to kernels and copies.
static __device__ __align__(256) char scratch[kNoAllocScratch];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch[kMaxDevices] = {};
bool g_scratch_done[kMaxDevices] = {};
}  // namespace

int noalloc_setup()
{
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("noalloc set-up: no current device");
    return -1;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_done[dev]) return 0;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    set_error(std::string("noalloc set-up: hipGetSymbolAddress: ") + hipGetErrorString(e));
    return -1;
  }
  g_scratch[dev] = ptr;
  g_scratch_done[dev] = true;
  return 0;
}

void *noalloc_scratch(int dev)
{
  if (dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch[dev];
}

// The a.num largest of each of `rows` rows of `len` entries (powers at mag,
// null: the v1 loops' |xs64|^2) into out, a.num per row; lists: 2 len ints of
// scratch per row.  Returns launches or -1.
static int top_levels(const V12Launch &a, hipStream_t st, const double *mag, int len, int rows,
                      int *lists, int *out, bool comb_last)
{
  TopLevel v;
  v.mag = mag;
  v.row = len;
  v.list = nullptr;
  v.num = a.num;
  int *next = lists, *other = lists + (int64_t)rows * len;
  if (a.num > kTopMax) {
    set_error("selection of more than 4096 entries above the LDS size");
    return -1;
  }
  for (int launches = 1;; launches++) {
    v.list_len = len;
    const bool last = len <= kTopLast;
    // every level at least halves the list: num is at most half a chunk
    v.chunk = last ? len : std::max(kTopChunk, 2 * pow2_ceil_int(a.num));
    v.chunks = (len + v.chunk - 1) / v.chunk;
    v.out = last ? out : next;
    const int left = (v.chunks - 1) * v.num + std::min(v.num, len - (v.chunks - 1) * v.chunk);
    v.out_stride = last ? v.num : left;
    v.comb_last = last && comb_last;
    const size_t lds = (size_t)v.chunk * sizeof(double);
    allow_lds(k_top_level, lds + kTopMax * sizeof(int));  // with its static picks
    hipLaunchKernelGGL(k_top_level, dim3((unsigned)(rows * v.chunks)), dim3(kTopThreads), lds, st,
                       a, v);
    if (launched("top_level") != 0) return -1;
    if (last) return launches;
    v.list = next;
    std::swap(next, other);
    len = left;
  }
}

// Below this many comb transforms per batch they run with kCombWide threads.
constexpr int kFewCombs = 64, kCombWide = 1024;

static int comb_merge(const V12Launch &a, hipStream_t st);

int comb(const V12Launch &a, hipStream_t st)
{
  int launches = 1;
  if (a.W <= kMaxLdsComb) {
    const size_t lds = (size_t)a.W * sizeof(double2);
    if (a.S * a.comb_loops < kFewCombs) {
      allow_lds(k_comb<kCombWide>, lds);
      hipLaunchKernelGGL(k_comb<kCombWide>, dim3(a.S * a.comb_loops), dim3(kCombWide), lds, st,
                         a);
    } else {
      allow_lds(k_comb<kBlock>, lds);
      hipLaunchKernelGGL(k_comb<kBlock>, dim3(a.S * a.comb_loops), dim3(kBlock), lds, st, a);
    }
    if (launched("comb") != 0) return -1;
  } else {
    if (comb_power(a, st) != 0) {
      set_error("comb FFT launch failed");
      return -1;
    }
    int *lists = reinterpret_cast<int *>(a.comb_buf);  // the transforms are done
    const int levels = top_levels(a, st, a.mag_buf, a.W, a.S * a.comb_loops, lists, a.approved,
                                  a.comb_loops == 1);
    if (levels < 0) return -1;
    launches = 2 + levels;
  }
  if (a.comb_loops == 1) return launches;
  return comb_merge(a, st) == 0 ? launches + 1 : -1;
}

size_t rows_entry_bytes(bool fp32) { return fp32 ? sizeof(RowEntry32) : sizeof(RowEntry64); }

static int64_t rows_entries(const V12Launch &a)
{
  return (int64_t)a.S * a.comb_loops * a.num * a.L;
}

int rows_table(const V12Launch &a, hipStream_t st)
{
  if (!a.rows_layout) return 0;
  const dim3 grid((unsigned)((rows_entries(a) + kBlock - 1) / kBlock));
  if (a.fp32) hipLaunchKernelGGL(k_rows_table<true>, grid, dim3(kBlock), 0, st, a);
  else hipLaunchKernelGGL(k_rows_table<false>, grid, dim3(kBlock), 0, st, a);
  return launched("rows_table") == 0 ? 1 : -1;
}

// The part of loops [l0, l0 + nl) with `res` residues per workgroup and its
// LDS; false when the loops do not fit the kernel's limits.
static bool fold_part(const V12Launch &a, bool fp32, int l0, int nl, int B, int res, FoldPart &f,
                      size_t &lds)
{
  const size_t elt = fp32 ? sizeof(float2) : sizeof(double2);
  f.fp32 = fp32;
  f.l0 = l0;
  f.nl = nl;
  f.B = B;
  f.logB = 31 - __builtin_clz((unsigned)B);
  f.res = std::min(res, B);
  f.log_res = 31 - __builtin_clz((unsigned)f.res);
  f.groups = B / f.res;
  const int rows = a.n / B;
  const int seg = std::min(rows, a.seg_rows);
  f.seg_log = 31 - __builtin_clz((unsigned)seg);
  f.tR = 0;
  if (l0 < a.Lloc) f.tR = std::max(f.tR, a.tR_loc);
  if (l0 + nl > a.Lloc) f.tR = std::max(f.tR, a.tR_est);
  if (f.tR > kMaxTaps) return false;
  f.tR |= 1;
  f.inv_tR = (1u << 20) / (unsigned)f.tR + 1;
  const size_t npairs = (size_t)f.res * nl;
  const size_t slots = (npairs * f.tR * elt + 15) / 16 * 16;
  f.nbins = rows;
  f.bin_shift = 0;
  while (f.nbins > 2048 || f.nbins * sizeof(int) > slots) {  // the bins use the slots' LDS
    f.nbins >>= 1;
    f.bin_shift++;
  }
  lds = slots + npairs * (sizeof(uint2) + sizeof(int));
  f.order_at = (int)(lds / 4);
  const size_t list = (npairs * f.tR * sizeof(uint16_t) + 3) / 4 * 4;
  const size_t order = npairs * ((f.tR + 3) & ~3) * ((rows >> f.seg_log) > kPackChunks ? 2 : 1);
  lds += fp32 ? std::max(list, order) : list;
  return npairs <= kFoldThreads && lds <= kFoldLds;
}

// The sorted fold of loops [0, n64) in FP64 (from loop `from` on) and
// [n64, L) in FP32, and its LDS.  False when the loops do not fit.
static bool fold_parts(const V12Launch &a, int from, int n64, FoldParts &f, size_t &lds)
{
  // 16 residues (256 contiguous bytes of a row) read HBM 5-10 % faster than
  // 8 on batches (with the groups in their natural order: FP32 256 x n =
  // 2^22, k = 64: 3.20 against 3.56 ms beside the estimation; FP64 64
  // signals: 0.81 against 0.86 ms); a launch of few workgroups is faster
  // spread over twice as many (one signal: 19.0 against 20.8 us), and a
  // workgroup's LDS does not hold 16 residues of many FP64 loops
  f = FoldParts{};
  lds = 0;
  int np = 0;
  auto add = [&](bool fp32, int l0, int l1) {
    if (l1 <= l0) return true;
    const int B = l0 < a.Lloc ? a.B_loc : a.B_est;
    size_t need = 0;
    const bool wide = (int64_t)a.S * B >= 16 * 512 &&
                      fold_part(a, fp32, l0, l1 - l0, B, 16, f.p[np], need);
    if (!wide && !fold_part(a, fp32, l0, l1 - l0, B, 8, f.p[np], need)) return false;
    lds = std::max(lds, need);
    f.groups += f.p[np].groups;
    np++;
    return true;
  };
  // where the bucket count or precision changes (with both, they change at
  // the same loop: n64 is 0, Lloc or L)
  const int cut = a.B_loc == a.B_est ? n64 : a.Lloc;
  return add(n64 == 0, from, cut) && add(cut >= n64, std::max(cut, from), a.L);
}

// Loops in FP64 of a batch: the first ones.
static int fp64_loops(const V12Launch &a)
{
  return !a.fp32 ? a.L : (a.loc64 ? a.Lloc : 0);
}

static size_t comb_lds(const V12Launch &a)
{
  return (size_t)a.W * sizeof(double2) + kTopScratch * sizeof(int);
}

bool fuse_comb(const V12Launch &a)
{
  // in the fold's launch the comb costs no second stream and no events; its
  // LDS is every workgroup's of the launch, so it has to leave room for two
  // on a CU, or the launch has to be small
  if (a.comb_loops == 0 || a.W > kMaxLdsComb || a.fold_mode == 0) return false;
  FoldParts f;
  size_t lds;
  if (!fold_parts(a, 0, fp64_loops(a), f, lds)) return false;
  const size_t need = comb_lds(a);
  return need <= std::max(lds, (size_t)79 * 1024) ||
         (need <= kFoldLds && (int64_t)a.S * (f.groups + a.comb_loops) <= 256);
}

static int comb_merge(const V12Launch &a, hipStream_t st)
{
  const size_t lb = (size_t)((a.W + 31) / 32) * 4;
  hipLaunchKernelGGL(k_comb_merge, dim3(a.S), dim3(kBlock), lb, st, a);
  return launched("comb_merge");
}

static int fold_sorted(const V12Launch &a, hipStream_t st, int from, int n64)
{
  FoldParts f;
  size_t lds = 0;
  if (!fold_parts(a, from, n64, f, lds)) {
    set_error("fold: more than 32 taps per bucket");
    return -1;
  }
  f.zero_blocks = a.zero_dense ? (int)std::min<int64_t>(512, (a.n + 4095) / 4096) : 0;
  f.combs = a.comb_fused ? a.S * a.comb_loops : 0;
  if (f.combs) lds = std::max(lds, comb_lds(a));
  const int64_t blocks = f.combs + (int64_t)a.S * (f.groups + f.zero_blocks);
  if (blocks == 0) return 0;
  allow_lds(k_fold_sorted, lds);
  hipLaunchKernelGGL(k_fold_sorted, dim3((unsigned)blocks), dim3(kFoldThreads), lds, st, a, f);
  if (launched("fold_sorted") != 0) return -1;
  if (!f.combs || a.comb_loops == 1) return 1;
  return comb_merge(a, st) == 0 ? 2 : -1;
}

// Whether the bucket FFTs of a v1 batch select the top buckets too.
static bool v1_fft_select(const V12Launch &a)
{
  return a.comb_loops == 0 && a.fold_mode >= 1 && a.B_loc <= kMaxLdsFft64 &&
         a.B_est <= kMaxLdsFft64;
}

int fold_fft(const V12Launch &a, hipStream_t st, int part)
{
  // loops [0, n64) in FP64, [n64, L) in FP32 (with the FFTs in part 1
  // whatever the schedule)
  const int n64 = fp64_loops(a);
  const int B64 = n64 == 0 ? 0 : (n64 > a.Lloc ? max(a.B_loc, a.B_est) : a.B_loc);
  int launches = 0;
  if (part == 0) {
    int from = 0;  // first loop of the sorted fold
    if (n64 > 0 && a.fold_mode == 0) {
      allow_lds(k_fold_fft64, (size_t)B64 * sizeof(double2));
      hipLaunchKernelGGL(k_fold_fft64, dim3(a.S * n64), dim3(kBlock),
                         (size_t)B64 * sizeof(double2), st, a, 0, n64);
      if (launched("fold_fft64") != 0) return -1;
      launches++;
      from = n64;
    }
    const int rc = fold_sorted(a, st, from, n64);
    return rc < 0 ? -1 : launches + rc;
  }
  // part 1: the bucket FFTs of every loop not fused into its fold
  if (a.rows_layout) {
    // v2: every loop in one precision, written in the alias-row layout
    const int Bm = max(a.B_loc, a.B_est), T = fft_threads(Bm);
    const int64_t entries = a.comb_fused ? rows_entries(a) : 0;
    const dim3 grid((unsigned)((int64_t)a.S * a.L + (entries + T - 1) / T));
    if (a.fp32) {
      allow_lds(k_bucket_fft_rows<true>, (size_t)Bm * sizeof(float2));
      hipLaunchKernelGGL(k_bucket_fft_rows<true>, grid, dim3(T), (size_t)Bm * sizeof(float2), st,
                         a, 0, a.L);
    } else {
      allow_lds(k_bucket_fft_rows<false>, (size_t)Bm * sizeof(double2));
      hipLaunchKernelGGL(k_bucket_fft_rows<false>, grid, dim3(T), (size_t)Bm * sizeof(double2), st,
                         a, 0, a.L);
    }
    if (launched("bucket_fft_rows") != 0) return -1;
    return 1;
  }
  if (v1_fft_select(a)) {
    const size_t lds = std::max((size_t)a.B_loc * sizeof(double2),
                                (size_t)a.B_est * (a.fp32 ? sizeof(float2) : sizeof(double2)));
    // few signals: every thread the selection can use
    const int T = a.S * a.Lloc < 256 ? 1024 : std::max(256, fft_threads(max(a.B_loc, a.B_est)));
    allow_lds(k_bucket_fft_v1, lds);
    hipLaunchKernelGGL(k_bucket_fft_v1, dim3(a.S * a.L), dim3(T), lds, st, a);
    return launched("bucket_fft_v1") == 0 ? 1 : -1;
  }
  // the location and estimation loops as batches of one bucket count and
  // precision: in LDS up to the LDS size, else radix-2 runs plus columns;
  // FP64 loops fused into their fold (schedule 0) are done
  const int f0 = a.fold_mode == 0 ? n64 : 0;  // first loop still to transform
  int groups[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  int ng = 0;
  auto add_run = [&](int l0, int l1) {
    // split [l0, l1) at Lloc (bucket counts) and n64 (precision)
    int cuts[4] = {l0, std::min(std::max(a.Lloc, l0), l1), std::min(std::max(n64, l0), l1), l1};
    std::sort(cuts, cuts + 4);
    for (int c = 0; c < 3; c++)
      if (cuts[c + 1] > cuts[c]) {
        groups[ng][0] = cuts[c];
        groups[ng][1] = cuts[c + 1];
        groups[ng][2] = cuts[c] < a.Lloc ? a.B_loc : a.B_est;
        ng++;
      }
  };
  add_run(f0, a.L);
  for (int gi = 0; gi < ng; gi++) {
    int l0 = groups[gi][0], l1 = groups[gi][1];
    const int B = groups[gi][2];
    // merge with the next run when bucket count and precision agree
    while (gi + 1 < ng && groups[gi + 1][2] == B && (groups[gi + 1][0] < n64) == (l0 < n64)) {
      l1 = groups[++gi][1];
    }
    const int64_t off = loop_offset_host(l0, a.Lloc, a.B_loc, a.B_est);
    const int rc = l0 < n64
                       ? radix2_fft64(a.xs64 + off, a.tmp64 ? a.tmp64 + off : nullptr, B,
                                      a.S, l1 - l0, a.xs, B, a.tw64, a.tw_nmax, st)
                       : radix2_fft32(a.xs32 + off, a.tmp32 ? a.tmp32 + off : nullptr, B,
                                      a.S, l1 - l0, a.xs, B, a.tw32, a.tw_nmax, st);
    if (rc < 0) return launch_failed("bucket FFT");
    launches += rc;
  }
  return launches;
}

// The top buckets of every location loop: in LDS up to its size, above it
// in levels; more picks than a level takes, over the HBM array.  Returns
// launches or -1.
static int select_loops(const V12Launch &a, hipStream_t st)
{
  if (a.B_loc <= kMaxLdsSelect) {
    allow_lds(k_select<false>, (size_t)a.B_loc * sizeof(double));
    hipLaunchKernelGGL(k_select<false>, dim3(a.S * a.Lloc), dim3(kBlock),
                       (size_t)a.B_loc * sizeof(double), st, a);
  } else if (a.num <= kTopMax) {
    return top_levels(a, st, nullptr, a.B_loc, a.S * a.Lloc, a.cand_buf, a.J, false);
  } else {
    hipLaunchKernelGGL(k_select<true>, dim3(a.S * a.Lloc), dim3(kBlock), 0, st, a);
  }
  return launched("select") == 0 ? 1 : -1;
}

int select_vote_v1(const V12Launch &a, hipStream_t st)
{
  const int selects = v1_fft_select(a) ? 0 : select_loops(a, st);
  if (selects < 0) return -1;
  const size_t lb = (size_t)a.Lloc * ((a.B_loc + 31) / 32) * 4;
  const int chunks = vote_chunks(a.n, a.B_loc, a.num, a.Lloc, a.thr);
  const dim3 grid((unsigned)((int64_t)a.S * chunks));
  hipLaunchKernelGGL(k_vote_count, grid, dim3(kBlock), lb, st, a, chunks);
  if (launched("vote_count") != 0) return -1;
  hipLaunchKernelGGL(k_vote_write, grid, dim3(kBlock), lb, st, a, chunks);
  return launched("vote_write") == 0 ? selects + 2 : -1;
}

int comb_vote_keys(const V12Launch &a, int64_t *keys, int64_t stride, hipStream_t st)
{
  const int selects = select_loops(a, st);
  if (selects < 0) return -1;
  const int64_t chunks = (a.est_cap + kBlock - 1) / kBlock;
  const size_t lb = (size_t)a.Lloc * ((a.B_loc + 31) / 32) * 4;
  allow_lds(k_comb_vote_keys, lb);
  hipLaunchKernelGGL(k_comb_vote_keys, dim3((unsigned)((int64_t)a.S * chunks)), dim3(kBlock), lb,
                     st, a, chunks, keys, stride);
  return launched("comb_vote_keys") == 0 ? selects + 1 : -1;
}

// Blocks that keep every CU busy with several wavefronts.
constexpr int64_t kFillBlocks = 1024;

template <int LMAX, int RI>
void launch_rows(const V12Launch &a, hipStream_t st, int tiles_j)
{
  const int tiles_i = (a.comb_loops * a.num + RI - 1) / RI;
  const dim3 grid((unsigned)xcd_grid(a.S, (int64_t)tiles_i * tiles_j));
  if (a.fp32) {
    if (a.L == LMAX)
      hipLaunchKernelGGL((k_estimate_rows<LMAX, true, true, RI>), grid, dim3(kBlock), 0, st, a,
                         tiles_i, tiles_j);
    else
      hipLaunchKernelGGL((k_estimate_rows<LMAX, false, true, RI>), grid, dim3(kBlock), 0, st, a,
                         tiles_i, tiles_j);
  } else {
    if (a.L == LMAX)
      hipLaunchKernelGGL((k_estimate_rows<LMAX, true, false, RI>), grid, dim3(kBlock), 0, st, a,
                         tiles_i, tiles_j);
    else
      hipLaunchKernelGGL((k_estimate_rows<LMAX, false, false, RI>), grid, dim3(kBlock), 0, st,
                         a, tiles_i, tiles_j);
  }
}

template <int LMAX>
void launch_estimate(const V12Launch &a, hipStream_t st)
{
  if (a.comb_loops > 0 && a.rows_layout) {
    const int tiles_j = (a.n / a.W + 63) / 64;
    const int64_t big = (int64_t)a.S * ((a.comb_loops * a.num + kRI - 1) / kRI) * tiles_j;
    if (big >= kFillBlocks) launch_rows<LMAX, kRI>(a, st, tiles_j);
    else launch_rows<LMAX, kRIsmall>(a, st, tiles_j);
  } else if (a.comb_loops > 0) {
    const int tiles_i = (a.comb_loops * a.num + kTI - 1) / kTI;
    const int tiles_j = (a.n / a.W + kTJ - 1) / kTJ;
    const dim3 grid((unsigned)xcd_grid(a.S, (int64_t)tiles_i * tiles_j));
    const bool allfast = a.W % (a.n / a.B_loc) == 0 && a.W % (a.n / a.B_est) == 0;
    if (a.fp32) {
      if (allfast)
        hipLaunchKernelGGL((k_estimate_comb<LMAX, true, true>), grid, dim3(kBlock), 0, st, a,
                           tiles_i, tiles_j);
      else
        hipLaunchKernelGGL((k_estimate_comb<LMAX, true, false>), grid, dim3(kBlock), 0, st,
                           a, tiles_i, tiles_j);
    } else {
      if (allfast)
        hipLaunchKernelGGL((k_estimate_comb<LMAX, false, true>), grid, dim3(kBlock), 0, st,
                           a, tiles_i, tiles_j);
      else
        hipLaunchKernelGGL((k_estimate_comb<LMAX, false, false>), grid, dim3(kBlock), 0, st,
                           a, tiles_i, tiles_j);
    }
  } else {
    const int64_t chunks = (a.est_cap + kBlock - 1) / kBlock;
    const dim3 grid((unsigned)xcd_grid(a.S, chunks));
    if (a.fp32)
      hipLaunchKernelGGL((k_estimate_hits<LMAX, true>), grid, dim3(kBlock), 0, st, a, chunks);
    else
      hipLaunchKernelGGL((k_estimate_hits<LMAX, false>), grid, dim3(kBlock), 0, st, a, chunks);
  }
}

int estimate(const V12Launch &a, hipStream_t st)
{
  // the smallest median network that holds the loops
  if (a.L <= 8) launch_estimate<8>(a, st);
  else if (a.L <= 12) launch_estimate<12>(a, st);
  else if (a.L <= 16) launch_estimate<16>(a, st);
  else if (a.L <= 20) launch_estimate<20>(a, st);
  else if (a.L <= 24) launch_estimate<24>(a, st);
  else launch_estimate<32>(a, st);
  return launched("estimate");
}

int zero_dense(double2 *out, int64_t n, hipStream_t st)
{
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, st, out, n);
  return launched("zero_dense");
}

}  // namespace k
}  // namespace sfa
