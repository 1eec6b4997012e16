// Device helpers shared by the sFFT kernels: complex arithmetic, an
// in-LDS radix-2 FFT, block scans and the top-num selection with the
// reference's tie rule.  Compiled with -ffp-contract=off, so every FP64
// product and sum below is rounded on its own, as in the reference's SSE2
// code.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sfa {
namespace dev {

constexpr int kBlock = 256;

__device__ __forceinline__ double2 cadd(double2 a, double2 b)
{
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b)
{
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b)
{
  return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b)
{
  return make_float2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
  return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}

__device__ __forceinline__ unsigned bitrev(unsigned v, int bits)
{
  return bits == 0 ? 0u : (__brev(v) >> (32 - bits));
}

// Stages s .. s+R-1 of an in-place radix-2 DIT FFT over N points in LDS, in
// registers: with h = 2^(s-1), the 2^R points i0 + m*h (m < 2^R) of a group
// only meet each other in those stages, so one thread loads them, applies the
// stages' butterflies in order (the same cmul / add / sub on the same
// twiddles as one stage per pass) and stores them.  Ends with a barrier.
template <typename T2, int R>
__device__ __forceinline__ void lds_fft_pass(T2 *buf, int N, int s, const T2 *__restrict__ tw,
                                             int tws)
{
  constexpr int M = 1 << R;
  const int h = 1 << (s - 1);
  const int groups = N >> R;
  for (int g = threadIdx.x; g < groups; g += blockDim.x) {
    const int j = g & (h - 1);
    const int i0 = ((g >> (s - 1)) << (s - 1 + R)) + j;  // group block * (h << R) + j
    T2 v[M];
#pragma unroll
    for (int m = 0; m < M; m++) v[m] = buf[i0 + m * h];
#pragma unroll
    for (int r = 0; r < R; r++) {
      // stage s + r: half-size H = h << r; the lower point i0 + m*h sits at
      // j + (m mod 2^r) * h within its butterfly block
      const int tstride = (N >> (s + r)) * tws;
#pragma unroll
      for (int m = 0; m < M; m++) {
        if (m & (1 << r)) continue;
        const int m1 = m + (1 << r);
        const T2 w = tw[(j + (m & ((1 << r) - 1)) * h) * tstride];
        const T2 u = v[m];
        const T2 t = cmul(v[m1], w);
        v[m] = cadd(u, t);
        v[m1] = csub(u, t);
      }
    }
#pragma unroll
    for (int m = 0; m < M; m++) buf[i0 + m * h] = v[m];
  }
  __syncthreads();
}

// In-place radix-2 decimation-in-time FFT of N = 2^logN points held in LDS in
// bit-reversed order; output in natural order.  tw[j * tws] = e^{-2 pi i j/N}
// where tws = Nmax / N for a table built for Nmax.  Three stages per LDS pass
// (lds_fft_pass); every butterfly is the radix-2 one, so results are those of
// one stage per pass, bit for bit.  Ends with a barrier.
template <typename T2>
__device__ void lds_fft(T2 *buf, int logN, const T2 *__restrict__ tw, int tws)
{
  const int N = 1 << logN;
  int s = 1;
  for (; logN - s + 1 >= 3; s += 3) lds_fft_pass<T2, 3>(buf, N, s, tw, tws);
  if (logN - s + 1 == 2) lds_fft_pass<T2, 2>(buf, N, s, tw, tws);
  else if (logN - s + 1 == 1) lds_fft_pass<T2, 1>(buf, N, s, tw, tws);
}

// Where point i of an N-point transform in LDS lies.  The passes below read
// points 1, 8, 64, ... apart, and the bit-reversed input arrives 2^(logN-6)
// apart; laid out by i, each of these puts the lanes of a read on a few
// banks.  Xor-ing higher bits into the low ones (a linear map, so
// fft_slot(i + j) = fft_slot(i) ^ fft_slot(j) for i, j without common bits)
// spreads all of them over the banks.  The bucket FFTs of 20 loops of 4096
// FP64 points went from 20 to 12 us (with one group of eight points a thread
// instead of two), of 8 x 20 loops of 16,384 FP32 points from 81 to 60 us.
// k_v3_run keeps lds_fft: built on this one it once ended a run with an
// illegal access (n = 2^22, k = 500) whose cause is not known.  A host build
// of both forms with bounds checks stays in bounds and gives the oracle's
// bits, also from corrupted buckets, and the variant's assembly shows no
// fault; it stays out all the same.
template <typename T2>
__device__ __forceinline__ unsigned fft_slot(unsigned i, int logN)
{
  constexpr int kLog = sizeof(T2) == 16 ? 4 : 5;  // log2 of the points in a row of banks
  unsigned p = i ^ ((i >> 3) & 7u) ^ (((i >> 6) & 3u) << 3);
  if (logN >= 10) {
    const unsigned t = i >> (logN - kLog);  // rotated: clear of the bits above
    p ^= (t << 1 | t >> (kLog - 1)) & ((1u << kLog) - 1);
  }
  return p;
}

// Stages s .. s+R-1 of an in-place radix-2 DIT FFT over N points in LDS, in
// registers: with h = 2^(s-1), the 2^R points i0 + m*h (m < 2^R) of a group
// only meet each other in those stages, so one thread loads them, applies the
// stages' butterflies in order (the same cmul / add / sub on the same
// twiddles as one stage per pass) and stores them.  cnt transforms, N points
// apart.  Starts with a barrier, before which the first group's twiddles are
// on their way.
template <typename T2, int R>
__device__ __forceinline__ void slot_fft_pass(T2 *buf, int logN, int s, const T2 *__restrict__ tw,
                                             int tws, int cnt)
{
  constexpr int M = 1 << R;
  const int N = 1 << logN, h = 1 << (s - 1);
  const int groups = cnt << (logN - R);
  // twiddles of a group: stage s + r needs 2^r, w[2^r - 1 + q], for the
  // lower points at j + q h within their butterfly block
  auto twiddles = [&](int g, T2 (&w)[M - 1]) {
    const int j = g & (h - 1);
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int q = 0; q < (1 << r); q++)
        w[(1 << r) - 1 + q] = tw[(j + q * h) * ((N >> (s + r)) * tws)];
  };
  T2 w[M - 1];
  int g = threadIdx.x;
  if (g < groups) twiddles(g, w);
  __syncthreads();
  for (; g < groups;) {
    const int gi = g & ((N >> R) - 1);  // the group within its transform
    const int j = gi & (h - 1);
    const int i0 = ((gi >> (s - 1)) << (s - 1 + R)) + j;  // group block * (h << R) + j
    T2 *const at = buf + ((g >> (logN - R)) << logN);
    const unsigned p0 = fft_slot<T2>((unsigned)i0, logN);
    T2 v[M];
#pragma unroll
    for (int m = 0; m < M; m++) v[m] = at[p0 ^ fft_slot<T2>((unsigned)(m * h), logN)];
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int m = 0; m < M; m++) {
        if (m & (1 << r)) continue;
        const int m1 = m + (1 << r);
        const T2 u = v[m];
        const T2 t = cmul(v[m1], w[(1 << r) - 1 + (m & ((1 << r) - 1))]);
        v[m] = cadd(u, t);
        v[m1] = csub(u, t);
      }
    }
#pragma unroll
    for (int m = 0; m < M; m++) at[p0 ^ fft_slot<T2>((unsigned)(m * h), logN)] = v[m];
    g += blockDim.x;
    if (g < groups) twiddles(g, w);
  }
}

// lds_fft of cnt runs of N = 2^logN points, with point i of the bit-reversed
// input and of the natural-order output at fft_slot(i) of its run.  tw[j * tws] = e^{-2 pi i j/N} where tws =
// Nmax / N for a table built for Nmax.  Three stages per LDS pass
// (slot_fft_pass); every butterfly is the radix-2 one, so results are those of
// one stage per pass, bit for bit.  Starts and ends with a barrier.
template <typename T2>
__device__ __forceinline__ void slot_fft(T2 *buf, int logN, const T2 *__restrict__ tw, int tws,
                                         int cnt = 1)
{
  int s = 1;
  for (; logN - s + 1 >= 3; s += 3) slot_fft_pass<T2, 3>(buf, logN, s, tw, tws, cnt);
  if (logN - s + 1 == 2) slot_fft_pass<T2, 2>(buf, logN, s, tw, tws, cnt);
  else if (logN - s + 1 == 1) slot_fft_pass<T2, 1>(buf, logN, s, tw, tws, cnt);
  __syncthreads();
}

// The input of slot_fft: point i from src(i), kFillAhead loads in flight.
constexpr int kFillAhead = 8;
template <typename T2, typename F>
__device__ __forceinline__ void slot_fft_fill(T2 *buf, int logN, F src)
{
  const int N = 1 << logN, T = blockDim.x;
  for (int i0 = threadIdx.x; i0 < N; i0 += kFillAhead * T) {
    T2 v[kFillAhead];
#pragma unroll
    for (int u = 0; u < kFillAhead; u++) v[u] = src(min(i0 + u * T, N - 1));
#pragma unroll
    for (int u = 0; u < kFillAhead; u++)  // past the end: point N - 1 again, same value
      buf[fft_slot<T2>(bitrev((unsigned)min(i0 + u * T, N - 1), logN), logN)] = v[u];
  }
}

// Threads for one N-point transform in LDS: one group of eight points each.
__host__ __device__ inline int fft_threads(int N) { return N / 8 < 64 ? 64 : N / 8 > 1024 ? 1024 : N / 8; }

// Exclusive prefix sum over the block (blockDim.x a multiple of 64);
// tmp holds >= 16 ints of LDS.  Contains barriers.
__device__ __forceinline__ int block_exclusive_scan(int v, int *tmp, int &total)
{
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) tmp[wid] = x;
  __syncthreads();
  int off = 0, tot = 0;
  for (int q = 0; q < nw; q++) {
    const int t = tmp[q];
    off += (q < wid) ? t : 0;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

// Indices of the num largest of mag[0..N) (in LDS), written ascending to out
// -- the rule of src/utils.cc:130-158: cutoff = (num+1)-th largest value;
// every index with mag > cutoff, then indices with mag == cutoff in index
// order until num are taken; output sorted.  mag values are >= +0, so their
// IEEE bit patterns order like the values.  Requires N >= num + 1.
// The cutoff is found by byte-wise radix selection from the top byte; once
// at most 128 keys share the selected prefix, their exact rank is computed
// directly.  The top byte (seven exponent bits) takes few values, so its
// histogram is counted once per value and wave, not by 64 atomics on one
// word; the picked indices are compacted by wave ballots over contiguous
// shares (a contiguous run per thread put a wave's reads on one bank).
// With both, the comb kernel of one signal (4096 points, 1024 threads) went
// from 28 to 25 us.
// Uses kTopScratch ints of LDS at sh.  Contains barriers, none after the
// last writes of out.
constexpr int kTopScratch = 2 * 256 + 32;
__device__ void block_top_num(const double *mag, int N, int num, int *out,
                              int *sh)
{
  int *misc = sh + 512;    // 32
  const int T = blockDim.x, tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6, nw = T >> 6;
  // rank of the cutoff in ascending order among the keys matching prefix
  int rank = N - num - 1;
  uint64_t prefix = 0, hi_mask = 0;
  uint64_t cut = 0;
  bool direct = false;
  for (int pass = 7; pass >= 0; --pass) {
    const int shift = pass * 8;
    // two histograms in turn, cleared in pairs
    int *hist = sh + 256 * (pass & 1);
    if (pass & 1) {
      for (int d = tid; d < 512; d += T) sh[d] = 0;
      __syncthreads();
    }
    if (pass == 7) {
      for (int i0 = wid * 64; i0 < N; i0 += T) {
        const int i = i0 + lane;
        const int d = i < N ? (int)((uint64_t)__double_as_longlong(mag[i]) >> 56) : -1;
        uint64_t left = __ballot(d >= 0);
        while (left) {  // wave-uniform
          const int d0 = __shfl(d, __ffsll((unsigned long long)left) - 1, 64);
          const uint64_t same = __ballot(d == d0);
          if (lane == 0) atomicAdd(&hist[d0], __popcll(same));
          left &= ~same;
        }
      }
    } else {
      for (int i = tid; i < N; i += T) {
        const uint64_t key = (uint64_t)__double_as_longlong(mag[i]);
        if ((key & hi_mask) == prefix) atomicAdd(&hist[(key >> shift) & 255], 1);
      }
    }
    __syncthreads();
    if (tid < 64) {
      // lane l holds bins 4l..4l+3; the bin holding rank is in the first
      // lane whose inclusive count exceeds rank
      int h[4], sum = 0;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        h[q] = hist[4 * tid + q];
        sum += h[q];
      }
      int incl = sum;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (tid >= o) incl += y;
      }
      const unsigned long long ball = __ballot(rank < incl);
      if (tid == __ffsll(ball) - 1) {
        int cum = incl - sum, q = 0;
        while (q < 3 && rank >= cum + h[q]) cum += h[q++];
        misc[0] = 4 * tid + q;
        misc[1] = rank - cum;
        misc[2] = h[q];
        misc[3] = 0;
      }
    }
    __syncthreads();
    prefix |= (uint64_t)misc[0] << shift;
    hi_mask |= 255ull << shift;
    rank = misc[1];
    const int cand = misc[2];
    __syncthreads();  // misc and hist are rewritten below
    if (pass > 0 && cand <= 128) {
      // the rank-th smallest of the cand keys matching prefix: the key with
      // (#keys < it) <= rank < (#keys <= it)
      // the 128 keys as low words in hist[0..128), high words in hist[128..256)
      unsigned *klo = reinterpret_cast<unsigned *>(hist), *khi = klo + 128;
      for (int i = tid; i < N; i += T) {
        const uint64_t key = (uint64_t)__double_as_longlong(mag[i]);
        if ((key & hi_mask) == prefix) {
          const int slot = atomicAdd(&misc[3], 1);
          klo[slot] = (unsigned)key;
          khi[slot] = (unsigned)(key >> 32);
        }
      }
      __syncthreads();
      if (tid < cand) {
        const uint64_t kj = (uint64_t)klo[tid] | (uint64_t)khi[tid] << 32;
        int lt = 0, le = 0;
        for (int q = 0; q < cand; q++) {
          const uint64_t kq = (uint64_t)klo[q] | (uint64_t)khi[q] << 32;
          lt += kq < kj;
          le += kq <= kj;
        }
        if (lt <= rank && rank < le) {  // every such thread holds the same key
          misc[4] = (int)(unsigned)(kj & 0xffffffffu);
          misc[5] = (int)(unsigned)(kj >> 32);
        }
      }
      __syncthreads();
      cut = (uint64_t)(unsigned)misc[4] | (uint64_t)(unsigned)misc[5] << 32;
      __syncthreads();
      direct = true;
      break;
    }
  }
  if (!direct) cut = prefix;
  // a contiguous share per wave, 64 keys a step, so that ballots rank the
  // picked keys in index order
  const int share = ((N + nw - 1) / nw + 63) & ~63;
  const int lo = min(N, wid * share), hi = min(N, lo + share);
  int ngt = 0, neq = 0;
  for (int i0 = lo; i0 < hi; i0 += 64) {
    const bool in = i0 + lane < hi;
    const uint64_t key = in ? (uint64_t)__double_as_longlong(mag[i0 + lane]) : 0;
    ngt += __popcll(__ballot(in && key > cut));
    neq += __popcll(__ballot(in && key == cut));
  }
  __syncthreads();  // misc is still being read above
  if (lane == 0) {
    misc[wid] = ngt;
    misc[16 + wid] = neq;
  }
  __syncthreads();
  int tot_gt = 0, gt_before = 0, eq_before = 0;
  for (int q = 0; q < nw; q++) {
    tot_gt += misc[q];
    gt_before += q < wid ? misc[q] : 0;
    eq_before += q < wid ? misc[16 + q] : 0;
  }
  const int need = num - tot_gt;  // ties to take, lowest indices first
  int pos = gt_before + min(eq_before, need);
  const uint64_t below = (1ull << lane) - 1;
  for (int i0 = lo; i0 < hi; i0 += 64) {
    const bool in = i0 + lane < hi;
    const uint64_t key = in ? (uint64_t)__double_as_longlong(mag[i0 + lane]) : 0;
    const uint64_t eq = __ballot(in && key == cut);
    const bool take =
        in && (key > cut || (key == cut && eq_before + __popcll(eq & below) < need));
    const uint64_t tk = __ballot(take);
    if (take) out[pos + __popcll(tk & below)] = i0 + lane;
    pos += __popcll(tk);
    eq_before += __popcll(eq);
  }
}

}  // namespace dev
}  // namespace sfa
