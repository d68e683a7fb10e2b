// aak_kernels.hip -- dense stage of the AAK waveform on CDNA4 (gfx950).
//
//   k_rates        spline evaluation of (e, v, M, S) on the dense grid with the
//                  block's knot coefficients staged in LDS, then the three
//                  phase rates from the PN frequency maps (AAK.cc:233-253)
//   fold kernels   the Adams-Bashforth phase folds (AAK.cc:244-293) computed in
//                  parallel but reproducing the sequential FP64 rounding bit for
//                  bit: inside one binade every value is an integer multiple of
//                  the same ulp, so sums of the rounded steps are exact: FP64
//                  scans in the single pass (k_fold_resolve), int64 prefix sums
//                  in the three-pass form; binade crossings and values near
//                  zero are replayed serially in FP64, exact ties by parity
//   k_modesum      harmonic sum with Bessel amplitudes, Doppler phases, LISA
//                  response and Planck taper (AAK.cc:409-547): per block of 1024
//                  or 256 samples the amplitudes are Taylor-expanded in e
//                  (k_modesum_setup); 256-sample blocks where that does not
//                  apply are summed per sample (k_modesum_direct)
//   k_weighted_dot PSD-weighted inner products of a rocFFT spectrum (lengths
//                  the fused FFT of aak_fft.hip does not take), k_dot_final
//                  the last reduction of either form (AAK_manager.cu:352-446)
//
// Compiled with -ffp-contract=off: every expression that feeds the phases
// must round exactly like the reference CPU build.
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>

#include <algorithm>
#include <mutex>

#include "aak_dense.hpp"
#include "aak_math.hpp"

namespace aak {

// ------------------------------------------------------------------ rates
constexpr int kRatesThreads = kRatesBlock;
constexpr int kRatesSlots = 1024;  // workgroups that run at once: 4 per CU
constexpr int kStageCap = 256;  // knot intervals staged in LDS per block (else direct evaluation)

__device__ inline int knot_search(const double *x, int lo, int hi, double t) {
  // largest k in [lo, hi-1] with x[k] <= t (hi is exclusive upper knot)
  while (hi > lo + 1) {
    const int m = (hi + lo) >> 1;
    if (x[m] > t) hi = m;
    else lo = m;
  }
  return lo;
}

__device__ inline double sample_time(const DenseParams &P, int i) {
  if (i == 0) return P.t_first;
  if (i == P.N) return P.t_last;
  return (double)(i - P.i0) * P.dt;
}

// Spline values (e, v, M, S) of one sample straight from the knot table.
__device__ inline void spline_sample(const DenseParams &P, const double *tab, double t, double *y) {
  const KnotGrid &g = P.grid;
  const int K = g.K;
  const double *head = tab + (size_t)kTableArrays * K;
  if (g.flat && t >= knot_time(g, head, K - 1)) {
    // past the table: flat intervals, whose cubic is y[K-1] + 0
#pragma unroll
    for (int a = 0; a < 4; a++) y[a] = tab[(size_t)a * K + K - 1] + 0.0;
    return;
  }
  const int k = knot_index(g, head, t);
  const double x0 = knot_time(g, head, k), x1 = knot_time(g, head, k + 1);
  const double dl = t - x0;
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const double *ya = tab + (size_t)a * K, *ca = tab + (size_t)(4 + a) * K;
    double b, d;
    spline_interval(x0, x1, ya[k], ya[k + 1], ca[k], ca[k + 1], &b, &d);
    y[a] = ya[k] + dl * (b + dl * (ca[k] + dl * d));
  }
}

// Several quotients by one divisor: its reciprocal is refined once, then each
// quotient takes a product, its exact residual and the correction, as the
// compiler's division does for operands that it need not scale.  Same bits as
// a / b while |a|, |b| and |a / b| lie within [2^-600, 2^600] (plain).
struct SharedDivisor {
  double b, y;
  __device__ explicit SharedDivisor(double d) : b(d) {
    y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    y = fma(fma(-d, y, 1.0), y, y);
  }
  __device__ double operator()(double a) const {
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
  }
};
// |x| within [2^-99, 2^100): products of up to six such factors stay plain.
struct PlainRange {
  unsigned lo = 0xffffffffu, hi = 0;
  __device__ void add(double x) {
    const unsigned u = (unsigned)__double2hiint(x) & 0x7fffffffu;
    lo = min(lo, u);
    hi = max(hi, u);
  }
  __device__ bool plain() const { return lo >= (1023u - 99u) << 20 && hi < (1023u + 100u) << 20; }
};

// Last sample evaluated.  Likelihoods read the rates up to the last folded step
// and e and the amplitude below the end of the signal (<= last_fold + 1), all
// within whole blocks; past that a source that plunged needs nothing (single
// waveforms keep every sample for the phase output and the dense arrays).
__host__ __device__ inline int rates_last(const DenseParams &P) {
  const long long end = ((long long)(P.last_fold + 1) / kRatesBlock + 1) * kRatesBlock - 1;
  return P.full_dense || end > P.N ? P.N : (int)end;
}

// Workgroup b: the samples [256 per b, 256 per (b + 1)), `per` of them to a thread.
// Bound by the vector unit: about 400 FP64 operations per sample, 26 us of issue
// at N = 2^21 (memory, 84 MB written, is 17 us).  Each saves work per sample:
// several samples per thread share the workgroup's set-up (knot intervals) and
// the terms in cos(iota) alone; quotients by one divisor share its reciprocal,
// 12 divisions for the price of 7.  With 128 registers four workgroups fit a
// CU, so the grid is cut into at most 1024 equal parts (a 1025th would run
// alone after them), more only where the knots in LDS or 64 samples per thread
// limit a part.  At N = 2^21 the stage, with the guard, takes 51 us: 60 with
// one sample per thread and separate divisions, 53 with 4 per thread in 2050
// workgroups, 72 with five workgroups per CU (96 registers, spills).  Below
// 2^18 samples each thread takes one, as before: 20 us at 2^17 either way, 24
// with 4.
__global__ __launch_bounds__(kRatesThreads, 4) void k_rates(DenseParams P, DenseBuffers B, int per) {
  __shared__ double s_x[kStageCap + 1];
  __shared__ double s_c[16][kStageCap];
  __shared__ int s_lo, s_cnt;
  const int tid = threadIdx.x;
  // the guard's segment words and ticket start cleared for each waveform
  if (blockIdx.x == 0 && tid <= kGuardGrid) B.guard_work[tid] = (tid < kGuardGrid) ? -2 : 0;
  const int last = rates_last(P), i_lo = blockIdx.x * kRatesThreads * per;
  // the last workgroup takes what a division of [0, last) leaves
  const int i_hi = blockIdx.x + 1 == gridDim.x ? last : i_lo + kRatesThreads * per - 1;
  const KnotGrid &g = P.grid;
  const int K = g.K;
  const double *tab = B.knots;
  const double *head = tab + (size_t)kTableArrays * K;
  if (tid == 0) {
    const int klo = knot_index(g, head, sample_time(P, i_lo));
    const int khi = knot_index(g, head, sample_time(P, i_hi));
    s_lo = klo;
    s_cnt = khi - klo + 1;
  }
  __syncthreads();
  const int klo = s_lo, cnt = s_cnt;
  const bool staged = (cnt <= kStageCap);
  if (staged) {
    // one interval per thread: knot time and the cubic of each array
    for (int j = tid; j < cnt; j += kRatesThreads) {
      const int k = klo + j;
      const double x0 = knot_time(g, head, k), x1 = knot_time(g, head, k + 1);
      s_x[j] = x0;
      if (j == cnt - 1) s_x[cnt] = x1;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const double *ya = tab + (size_t)a * K, *ca = tab + (size_t)(4 + a) * K;
        double b, d;
        spline_interval(x0, x1, ya[k], ya[k + 1], ca[k], ca[k + 1], &b, &d);
        s_c[4 * a][j] = ya[k];
        s_c[4 * a + 1][j] = b;
        s_c[4 * a + 2][j] = ca[k];
        s_c[4 * a + 3][j] = d;
      }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int i = i_lo + tid; i <= i_hi; i += kRatesThreads) {
    const double t = sample_time(P, i);
    double y[4];
    if (g.flat && t >= knot_time(g, head, K - 1)) {
#pragma unroll
      for (int a = 0; a < 4; a++) y[a] = tab[(size_t)a * K + K - 1] + 0.0;
    } else if (staged) {
      const int k = knot_search(s_x, 0, cnt, t);
      const double dl = t - s_x[k];
#pragma unroll
      for (int a = 0; a < 4; a++)
        y[a] = s_c[4 * a][k] + dl * (s_c[4 * a + 1][k] + dl * (s_c[4 * a + 2][k] + dl * s_c[4 * a + 3][k]));
    } else {
      spline_sample(P, tab, t, y);
    }
    const double e = y[0], v = y[1], M = y[2], S = y[3];
    B.e[i] = e;
    if (P.full_dense) {
      B.v[i] = v;
      B.M[i] = M;
      B.S[i] = S;
    }
    const double Y = P.coslam;
    double T = PN::dtdm_num(v, e, Y, S), R = PN::drdm_num(v, e, Y, S), Th = PN::dthetadm_num(v, e, Y, S),
           Ph = PN::dphidm_num(v, e, Y, S);
    const double v2 = v * v, v4 = v2 * v2;
    double dR, dphi, dTh, Oph;  // (Th - R) / T / M, R / T / M, (Ph - Th) / T / M, Ph / T / M
    PlainRange g1;
    g1.add(v4);
    g1.add(T);
    g1.add(R);
    g1.add(Th);
    g1.add(Ph);
    g1.add(M);
    bool plain = g1.plain();
    if (plain) {
      T = SharedDivisor(256. * v4)(T);
      const SharedDivisor d16(16. * v);
      R = d16(R);
      Th = d16(Th);
      Ph = d16(Ph);
      const double a = Th - R, b = Ph - Th;
      PlainRange g2;
      g2.add(a);
      g2.add(b);
      plain = g2.plain();
      const SharedDivisor dT(T), dM(M);
      dR = dM(dT(a));
      dphi = dM(dT(R));
      dTh = dM(dT(b));
      Oph = dM(dT(Ph));
    } else {
      T /= 256. * v4;
      R /= 16. * v;
      Th /= 16. * v;
      Ph /= 16. * v;
    }
    if (!plain) {
      dR = (Th - R) / T / M;
      dphi = R / T / M;
      dTh = (Ph - Th) / T / M;
      Oph = Ph / T / M;
    }
    const double phidot = dphi;
    B.rate[0][i] = dR;
    B.rate[1][i] = phidot;
    B.rate[2][i] = dTh;
    // amplitude of the mode sum (AAK.cc:481), with OmegaPhi of the prograde case
    // from the maps already evaluated here; x^(2/3) as cbrt(x)^2 (within a few
    // ulp of pow: the amplitude scales the waveform and feeds no phase)
    const double Om = (Y > 0) ? Oph : PN::omega_phi(v, e, Y, S, M);
    const double cr = cbrt(Om * P.Mphys * kMsunSec);
    B.amp[i] = (cr * cr) * P.zeta;
    if (i == 0) B.nu0[0] = R / T / (2. * kPi * M);
    // the reference's test is Phidot <= 0 (AAK.cc:254): a NaN rate is kept as it is
    if (i > P.i0 && i <= P.guard_last && phidot <= 0.) {
      atomicAdd(&B.flags[0], 1);
      atomicMax(&B.flags[5], 0x7fffffff - i);  // the first such sample, for the guard
    }
    // a non-positive rate at t = 0 has no earlier value to take: the waveform is
    // rejected (flags[3]; the likelihood of such a template reads NaN)
    if (i == P.i0 && phidot <= 0.) B.flags[3] = 1;
  }
}

void launch_rates(const DenseParams &P, const DenseBuffers &B, hipStream_t s) {
  const long long last = rates_last(P), slots = (long long)kRatesThreads * kRatesSlots;
  // no more samples than LDS holds knots for (fast sources have a knot every few
  // samples, beyond it every sample searches the table): with a knot per 10
  // samples the stage takes 50 us at N = 2^21, 72 without this limit (60 with
  // one sample per thread); with one per 3.5 samples 51, 71 (56)
  const double rows = (kStageCap - 8) * P.grid.dt_large / (kRatesThreads * P.dt);
  const int most = rows < 1.0 ? 1 : rows < 64.0 ? (int)rows : 64;
  const int per = (int)std::min((long long)most, std::max(1LL, (last + slots - 1) / slots));
  const int nb = (int)std::max(1LL, (last + kRatesThreads * per - 1) / (kRatesThreads * per));
  hipLaunchKernelGGL(k_rates, dim3(nb), dim3(kRatesThreads), 0, s, P, B, per);
}

// Non-positive radial rates take the previous (already corrected) value
// (AAK.cc:254): sample i in (i0, guard_last] with Phidot <= 0 gets the rate of
// the last sample j in (i0, i] whose rate is not <= 0 (a NaN rate counts as
// such a sample and is kept, as the reference's test leaves it), or of i0 if
// there is none.  Every sample before the first non-positive one (recorded
// by k_rates) is such a sample, so only [first, guard_last] is walked, split
// into kGuardGrid segments.  Each workgroup takes a ticket, finds its
// segment's last good index and publishes it at once; its carry is the
// maximum over the segments before it, which never wait on anything, so the
// waits are short and cannot form a cycle.  The fix then runs in chunks of
// kGuardThreads x kGuardPer with an inclusive max-scan of the last good index
// over the threads.  Good samples are never written, so a replaced sample
// reads a final value.  The kernel returns at once when k_rates counted no
// such sample, so it is always enqueued and needs no host round trip.
constexpr int kGuardThreads = 1024;

// Look-back words of the single-pass fold (k_fold_resolve), kLW per block and
// phase, reset by k_guard for every waveform: the action of a block on one
// grid and its grid key, the exact end value, the approximate sum and L1 norm
// of the block's increments and their inclusive prefixes; then, of a block
// with a crossing action, its grid keys, its representative start and the
// four ends (CrossAction).  "Not yet", "failed", "no action" and "crossing"
// are signalling-NaN patterns that arithmetic never produces and no run total
// or key can equal.
constexpr int kLwAct = 0, kLwKey = 2, kLwIncl = 3, kLwAggS = 4, kLwAggL = 5, kLwIncS = 6, kLwIncL = 7;
constexpr int kLwXKey = 8, kLwXBase = 9, kLwXEnd = 10;  // ends: words 10..13
constexpr long long kLookEmpty = 0x7FF4A5A5A5A5A5A5LL;
constexpr long long kLookFail = 0x7FF4A5A5A5A5A5A6LL;
constexpr long long kLookNone = 0x7FF4A5A5A5A5A5A7LL;
constexpr long long kLookCross = 0x7FF4A5A5A5A5A5A8LL;
constexpr int kGuardPer = 32;  // consecutive samples per thread and chunk
constexpr int kGuardSpinCap = 1 << 22;

__device__ inline bool phidot_ok(double r) { return !(r <= 0.); }

__global__ __launch_bounds__(kGuardThreads) void k_guard(DenseParams P, DenseBuffers B, FoldReset R) {
  {
    // the fold's look-back words, replay marks and tickets for this waveform
    const int gt = blockIdx.x * blockDim.x + threadIdx.x, gs = gridDim.x * blockDim.x;
    for (int k = gt; k < R.nwords; k += gs) R.words[k] = kLookEmpty;
    if (R.status && gt < 6) R.status[gt] = R.force == 1 ? 1 : 0;
    if (R.ctr && gt < 2 * 3 * kLookCtrStride) R.ctr[gt] = 0;
  }
  if (P.guard_last <= P.i0 || B.flags[0] == 0) return;
  __shared__ int s_w[kGuardThreads / 64];
  __shared__ int s_t, s_carry;
  double *r = B.rate[1];
  int *gw = B.guard_work;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_t = atomicAdd(gw + kGuardGrid, 1);
  __syncthreads();
  const int t = s_t;
  const int first = 0x7fffffff - B.flags[5];
  const int n = P.guard_last - first + 1;
  const int per = ((n + kGuardGrid - 1) / kGuardGrid + kGuardThreads - 1) / kGuardThreads * kGuardThreads;
  const int lo = first + t * per, hi = min(P.guard_last, lo + per - 1);
  // the segment's last good index, published at once
  int last = -1;
  for (int i = lo + tid; i <= hi; i += kGuardThreads)
    if (phidot_ok(r[i])) last = i;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) last = max(last, __shfl_xor(last, o, 64));
  if (lane == 0) s_w[wave] = last;
  __syncthreads();
  if (wave == 0) {
    int agg = -1;
    for (int w = 0; w < kGuardThreads / 64; w++) agg = max(agg, s_w[w]);
    if (lane == 0) __hip_atomic_store(gw + t, agg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // carry: the last good index of the segments before this one
    int c = first - 1;
    bool late = false;
    if (lane < t) {
      int v, spins = 0;
      while ((v = __hip_atomic_load(gw + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == -2) {
        if (++spins > kGuardSpinCap) {
          late = true;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
      if (!late) c = max(c, v);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c = max(c, __shfl_xor(c, o, 64));
    const bool any_late = __ballot(late) != 0;
    if (lane == 0) {
      s_carry = c;
      if (any_late) B.flags[3] = 1;  // a wait past the cap rejects the waveform
    }
  }
  __syncthreads();
  int carry = s_carry;
  for (int base = lo; base <= hi; base += kGuardThreads * kGuardPer) {
    const int i0 = base + tid * kGuardPer;
    double v[kGuardPer];
    int lst = -1;
#pragma unroll
    for (int q = 0; q < kGuardPer; q++) {
      const int i = i0 + q;
      v[q] = (i <= hi) ? r[i] : 1.0;
      if (i <= hi && phidot_ok(v[q])) lst = i;
    }
    // inclusive max-scan of the last good index over the threads
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(lst, o, 64);
      if (lane >= o) lst = max(lst, u);
    }
    if (lane == 63) s_w[wave] = lst;
    __syncthreads();
    int before = carry, chunk = carry;
    for (int w = 0; w < kGuardThreads / 64; w++) {
      const int x = s_w[w];
      if (w < wave) before = max(before, x);
      chunk = max(chunk, x);
    }
    // last good index before this thread's samples; its value is read only
    // when the thread's first sample needs it, later ones come from registers
    int src = max(before, __shfl_up(lst, 1, 64));
    if (lane == 0) src = before;
    double srcv = (i0 <= hi && !phidot_ok(v[0])) ? r[src] : 0.0;
#pragma unroll
    for (int q = 0; q < kGuardPer; q++) {
      const int i = i0 + q;
      if (i <= hi) {
        if (phidot_ok(v[q])) srcv = v[q];
        else r[i] = srcv;
      }
    }
    carry = chunk;
    __syncthreads();
  }
}

void launch_phidot_guard(const DenseParams &P, const DenseBuffers &B, const FoldReset &R, hipStream_t s) {
  if (P.guard_last <= P.i0 && R.nwords == 0 && !R.status && !R.ctr) return;
  hipLaunchKernelGGL(k_guard, dim3(kGuardGrid), dim3(kGuardThreads), 0, s, P, B, R);
}

// ------------------------------------------------------------------ folds
__device__ inline double fold_incr(const double *rate, int i0, int dir, int s, double dt) {
  const int i = i0 + dir * s;
  const double r = rate[i];
  const double rm = (s == 0) ? r : rate[i - dir];
  const double d = (1.5 * r - .5 * rm) * dt;
  return dir > 0 ? d : -d;
}

__device__ inline int out_index(const FoldArgs &A, int s) { return A.i0 + A.dir * (s + 1); }

// A block's increments are read with consecutive lanes on consecutive steps
// (coalesced) and staged in LDS; each lane then takes its run of
// kFoldPerThread consecutive steps from LDS.  One pad double per run keeps
// both access patterns free of bank conflicts.
static_assert(kFoldPerThread == 16, "fold_lds_index assumes runs of 16");
constexpr int kFoldLds = kFoldBlock + kFoldBlock / kFoldPerThread;
static_assert(kFoldLds >= 4096, "the serial replay stages 4096 steps in the staging array");
__device__ inline int fold_lds_index(int l) { return l + (l >> 4); }

// Every load is issued before the first use.  An interior block (all its
// steps in range, none of them step 0) reads at fixed offsets from one base
// pointer per lane; other blocks clamp: steps past the end read the last
// step's rates (in bounds) and stage 0.  DIR is the fold direction (A.dir).
template <int DIR>
__device__ inline void stage_increments(const FoldArgs &A, int p, int b, double *sd) {
  const double *rate = A.rate[p];
  double r[kFoldPerThread], rm[kFoldPerThread];
  if (b > 0 && (b + 1) * kFoldBlock <= A.nsteps) {
    const double *rp = rate + (A.i0 + DIR * (b * kFoldBlock + (int)threadIdx.x));
#pragma unroll
    for (int q = 0; q < kFoldPerThread; q++) {
      r[q] = rp[DIR * q * kFoldThreads];
      rm[q] = rp[DIR * q * kFoldThreads - DIR];
    }
  } else {
#pragma unroll
    for (int q = 0; q < kFoldPerThread; q++) {
      const int s = min(b * kFoldBlock + (int)threadIdx.x + q * kFoldThreads, A.nsteps - 1);
      const int i = A.i0 + DIR * s;
      r[q] = rate[i];
      rm[q] = rate[s == 0 ? i : i - DIR];
    }
  }
#pragma unroll
  for (int q = 0; q < kFoldPerThread; q++) {
    const int l = threadIdx.x + q * kFoldThreads;
    const double d = (1.5 * r[q] - .5 * rm[q]) * A.dt;
    sd[fold_lds_index(l)] = (b * kFoldBlock + l < A.nsteps) ? (DIR > 0 ? d : -d) : 0.0;
  }
  __syncthreads();
}

// Block-wide exclusive scans over kFoldThreads lanes: inclusive shuffle scan
// inside each 64-lane wave, wave totals through LDS.  `sh` needs
// kFoldThreads / 64 entries.  Integer scans are exact; the double scan is an
// approximation consumer (the fold's binade prediction) whose error the
// bound E covers.
template <class T>
__device__ inline T wave_incl_sum(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

template <class T>
__device__ inline T block_excl_sum(T v, T *sh, T *total) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const T incl = wave_incl_sum(v);
  if (lane == 63) sh[wave] = incl;
  __syncthreads();
  T before = T(0), tot = T(0);
#pragma unroll
  for (int w = 0; w < kFoldThreads / 64; w++) {
    const T x = sh[w];
    if (w < wave) before += x;
    tot += x;
  }
  if (total) *total = tot;
  __syncthreads();
  return before + incl - v;
}

// Segmented inclusive scan of (flag, value) pairs over the block, lanes in
// order: a set flag starts a new segment.  Returns the inclusive value of the
// lane's segment prefix; shv/shf need kFoldThreads / 64 entries.
__device__ inline long long block_seg_incl(long long v, int f, long long *shv, int *shf) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const long long uv = __shfl_up(v, o, 64);
    const int uf = __shfl_up(f, o, 64);
    if (lane >= o && !f) {
      v += uv;
      f |= uf;
    }
  }
  if (lane == 63) {
    shv[wave] = v;
    shf[wave] = f;
  }
  __syncthreads();
  if (!f) {
    // carry in from the earlier waves, back to the nearest segment start
    for (int w = wave - 1; w >= 0; w--) {
      v += shv[w];
      if (shf[w]) break;
    }
  }
  __syncthreads();
  return v;
}

// approximate block sums and prefix ranges
template <int DIR>
__global__ __launch_bounds__(kFoldThreads) void k_fold_sums(FoldArgs A, FoldWork W) {
  __shared__ double sh[2 * (kFoldThreads / 64)];
  __shared__ double sd[kFoldLds];
  const int p = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  const int base = b * kFoldBlock + tid * kFoldPerThread;
  stage_increments<DIR>(A, p, b, sd);
  double run = 0.0, mn = 0.0, mx = 0.0;
  for (int j = 0; j < kFoldPerThread; j++) {
    const int s = base + j;
    if (s < A.nsteps) {
      run += sd[fold_lds_index(tid * kFoldPerThread + j)];
      mn = fmin(mn, run);
      mx = fmax(mx, run);
    }
  }
  double tot;
  const double off = block_excl_sum(run, sh, &tot);
  double lmn = off + mn, lmx = off + mx;
  for (int o = 32; o > 0; o >>= 1) {
    lmn = fmin(lmn, __shfl_xor(lmn, o, 64));
    lmx = fmax(lmx, __shfl_xor(lmx, o, 64));
  }
  if ((tid & 63) == 0) {
    sh[tid >> 6] = lmn;
    sh[kFoldThreads / 64 + (tid >> 6)] = lmx;
  }
  __syncthreads();
  if (tid == 0) {
    double bmn = sh[0], bmx = sh[kFoldThreads / 64];
    for (int w = 1; w < kFoldThreads / 64; w++) {
      bmn = fmin(bmn, sh[w]);
      bmx = fmax(bmx, sh[kFoldThreads / 64 + w]);
    }
    W.bsum[p * A.nblk + b] = tot;
    W.bmin[p * A.nblk + b] = bmn;
    W.bmax[p * A.nblk + b] = bmx;
  }
}

// approximate block start values and the error bound E
__global__ __launch_bounds__(1024) void k_fold_plan(FoldArgs A, FoldWork W) {
  __shared__ double s_w[16], s_m[16];
  const int p = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (A.nblk + 1023) / 1024;
  double loc = 0.0;
  for (int j = 0; j < per; j++) {
    const int b = tid * per + j;
    if (b < A.nblk) loc += W.bsum[p * A.nblk + b];
  }
  // exclusive prefix of loc over the threads: shuffles inside each wave, then
  // the wave totals (approximate starts: the bound E covers their rounding)
  double incl = loc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  double before = 0.0;
  for (int w = 0; w < wave; w++) before += s_w[w];
  const double up = __shfl_up(incl, 1, 64);
  double run = A.x0[p] + (before + (lane > 0 ? up : 0.0));
  double amax = fabs(A.x0[p]);
  for (int j = 0; j < per; j++) {
    const int b = tid * per + j;
    if (b < A.nblk) {
      W.xstart[p * A.nblk + b] = run;
      amax = fmax(amax, fmax(fabs(run + W.bmin[p * A.nblk + b]), fabs(run + W.bmax[p * A.nblk + b])));
      run += W.bsum[p * A.nblk + b];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, 64));
  if (lane == 0) s_m[wave] = amax;
  __syncthreads();
  if (tid == 0) {
    double m = s_m[0];
    for (int w = 1; w < 16; w++) m = fmax(m, s_m[w]);
    int ex = 0;
    frexp(m > 0.0 ? m : 1.0, &ex);
    W.E[p] = ((double)A.nsteps + 2.0 * kFoldBlock) * ldexp(1.0, ex - 52);
    W.status[p] = W.force_replay == 1 ? 1 : 0;
  }
}

__device__ inline int binade_key(double a, double E) {
  const double aa = fabs(a);
  const double lo = aa - E, hi = aa + E;
  if (!(lo > 0.0)) return -1;
  int klo, khi;
  frexp(lo, &klo);
  frexp(hi, &khi);
  if (klo != khi) return -1;
  return (klo + 4096) * 2 + (a > 0.0 ? 1 : 0);
}

// Fallback: plain serial replay of one phase's whole fold, by one workgroup
// with buf (bufn doubles of LDS) as staging; used when the item bookkeeping
// overflowed or a check failed (correct for any input).
__device__ void fold_serial_replay(const FoldArgs &A, const FoldWork &W, int p, double *buf, int bufn) {
  if (threadIdx.x == 0) atomicAdd(W.fallbacks, 1);
  double x = A.x0[p];
  if (threadIdx.x == 0) A.out[p][A.i0] = x;
  for (int base = 0; base < A.nsteps; base += bufn) {
    const int n = min(bufn, A.nsteps - base);
    for (int j = threadIdx.x; j < n; j += blockDim.x) buf[j] = fold_incr(A.rate[p], A.i0, A.dir, base + j, A.dt);
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int j = 0; j < n; j++) {
        x = x + buf[j];
        buf[j] = x;
      }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += blockDim.x) A.out[p][out_index(A, base + j)] = buf[j];
    __syncthreads();
  }
}

// Classify steps, build the block's item list (PLAN) or write the exact
// fold values of run steps (WRITE, after the chain resolved the run starts).
template <bool WRITE, int DIR>
__global__ __launch_bounds__(kFoldThreads, WRITE ? 3 : 4) void k_fold_local(FoldArgs A, FoldWork W) {
  __shared__ double shd[kFoldThreads / 64];
  __shared__ long long shl[2 * (kFoldThreads / 64)];
  __shared__ int shi[kFoldThreads];
  __shared__ int shf[kFoldThreads / 64];
  __shared__ double sd[kFoldLds];
  const int p = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  if (W.status[p]) {
    // the write pass of a phase the chain could not resolve: its first
    // workgroup replays the fold serially
    if (WRITE && b == 0) fold_serial_replay(A, W, p, sd, 4096);
    return;
  }
  const int base = b * kFoldBlock + tid * kFoldPerThread;
  const double E = W.E[p];
  stage_increments<DIR>(A, p, b, sd);
  double d[kFoldPerThread];
  double tsum = 0.0;
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) {
    d[j] = sd[fold_lds_index(tid * kFoldPerThread + j)];
    tsum += d[j];
  }
  double dummy;
  double a0 = W.xstart[p * A.nblk + b] + block_excl_sum(tsum, shd, &dummy);
  // keys: >= 0 binade grid, -1 exact replay, -2 beyond the end
  int key[kFoldPerThread];
  long long r[kFoldPerThread];
  int tie_mask = 0, head_mask = 0;
  int prev_key = -3;
  // key of the previous lane's last step, for head detection across lanes
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) {
    const int s = base + j;
    if (s >= A.nsteps) {
      key[j] = -2;
      r[j] = 0;
      continue;
    }
    const double a1 = a0 + d[j];
    const int k0 = binade_key(a0, E);
    const int k1 = binade_key(a1, E);
    if (k0 >= 0 && k0 == k1) {
      key[j] = k0;
      const int kexp = (k0 >> 1) - 4096;
      const double f = ldexp(d[j], 53 - kexp);
      const double fl = floor(f);
      const double fr = f - fl;
      long long ri = (long long)fl;
      if (fr > 0.5) ri += 1;
      else if (fr == 0.5) tie_mask |= (1 << j);
      r[j] = ri;
    } else {
      key[j] = -1;
      r[j] = 0;
    }
    a0 = a1;
  }
  // head flags need the previous lane's last key
  shi[tid] = key[kFoldPerThread - 1];
  __syncthreads();
  prev_key = (tid > 0) ? shi[tid - 1] : -3;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) {
    const int kprev = (j == 0) ? prev_key : key[j - 1];
    const bool h = (key[j] != -2) && (key[j] == -1 || kprev == -1 || kprev == -3 || key[j] != kprev);
    if (h) head_mask |= (1 << j);
  }
  // does the next lane start a new item (or lie beyond the end)?
  shi[tid] = ((head_mask & 1) || key[0] == -2) ? 1 : 0;
  __syncthreads();
  const bool next_starts = (tid + 1 < kFoldThreads) ? (shi[tid + 1] != 0) : true;
  __syncthreads();
  // segmented carry of r across lanes: summary (has_head, tail_sum)
  long long tail = 0;
  int has_head = 0;
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) {
    if (head_mask & (1 << j)) {
      has_head = 1;
      tail = 0;
    }
    tail += r[j];
  }
  // carry into the lane: the segmented inclusive scan of the previous lane
  const long long seg_incl = block_seg_incl(tail, has_head, shl, shf);
  long long carry = __shfl_up(seg_incl, 1, 64);
  if ((tid & 63) == 63) shl[kFoldThreads / 64 + (tid >> 6)] = seg_incl;  // for the next wave's lane 0
  __syncthreads();
  if ((tid & 63) == 0) carry = (tid > 0) ? shl[kFoldThreads / 64 + (tid >> 6) - 1] : 0;
  __syncthreads();
  // item and tie numbering
  const int nh = __popc(head_mask);
  int nheads_tot;
  const int item_base = block_excl_sum(nh, shi, &nheads_tot);
  const int nt = __popc(tie_mask);
  int nties_tot;
  const int tie_base = block_excl_sum(nt, shi, &nties_tot);
  if (!WRITE && tid == 0) {
    W.nitems[p * A.nblk + b] = nheads_tot;
    W.nties[p * A.nblk + b] = nties_tot;
    if (nheads_tot > kFoldMaxItems || nties_tot > kFoldMaxTies) atomicExch(&W.status[p], 1);
  }
  if (nheads_tot > kFoldMaxItems || nties_tot > kFoldMaxTies) return;
  FoldItem *items = W.items + ((size_t)p * A.nblk + b) * kFoldMaxItems;
  FoldTie *ties = W.ties + ((size_t)p * A.nblk + b) * kFoldMaxTies;
  long long P = carry;
  int item = item_base - 1, tcount = tie_base;
  int c_item = -1, c_k = 0, c_tf = 0;  // WRITE: the item of the current run
  long long c_m = 0;
  double outv[kFoldPerThread];  // WRITE: values of the run steps, NaN elsewhere
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) outv[j] = __builtin_nan("");
#pragma unroll
  for (int j = 0; j < kFoldPerThread; j++) {
    if (key[j] == -2) break;
    const int sl = tid * kFoldPerThread + j;
    if (head_mask & (1 << j)) {
      item++;
      P = 0;
      if (!WRITE) {
        items[item].kind = (key[j] == -1) ? 1 : 0;
        items[item].k = (key[j] >= 0) ? (key[j] >> 1) - 4096 : 0;
        items[item].sgn = (key[j] >= 0) ? ((key[j] & 1) ? 1 : -1) : 0;
        items[item].first = sl;
        items[item].tie_first = tcount;
        items[item].d = d[j];
      }
    }
    P += r[j];
    const bool last_of_run =
        (key[j] >= 0) && ((j + 1 < kFoldPerThread) ? (((head_mask >> (j + 1)) & 1) || key[j + 1] == -2) : next_starts);
    if (tie_mask & (1 << j)) {
      if (!WRITE) {
        ties[tcount].step = sl;
        ties[tcount].P = P;
        ties[tcount].up = 0;
      }
      tcount++;
    }
    if (!WRITE) {
      // the run total is the inclusive prefix at the run's last step
      if (last_of_run) items[item].R = P;
    } else if (key[j] >= 0) {
      if (item != c_item) {
        c_item = item;
        c_m = items[item].m_start;
        c_k = items[item].k;
        c_tf = items[item].tie_first;
      }
      long long ups = 0;
      for (int q = c_tf; q < tcount; q++) ups += ties[q].up;
      const long long m = c_m + P + ups;
      outv[j] = ldexp((double)m, c_k - 53);
    }
  }
  if (WRITE) {
    // coalesced stores of the run steps; single steps were written by the chain
#pragma unroll
    for (int j = 0; j < kFoldPerThread; j++) sd[fold_lds_index(tid * kFoldPerThread + j)] = outv[j];
    __syncthreads();
    // step s goes to A.i0 + DIR (s + 1)
    double *op = A.out[p] + (A.i0 + DIR * (b * kFoldBlock + tid + 1));
#pragma unroll
    for (int q = 0; q < kFoldPerThread; q++) {
      const int s = b * kFoldBlock + tid + q * kFoldThreads;
      const double v = sd[fold_lds_index(tid + q * kFoldThreads)];
      if (s < A.nsteps && !__builtin_isnan(v)) op[DIR * q * kFoldThreads] = v;
    }
  }
}

// Exact start of every run, resolution of the exact ties, FP64 replay of the
// single steps near binade boundaries.  The item and tie lists of all blocks
// are gathered into LDS; consecutive runs on one binade grid without ties
// form a segment whose total is a segmented int64 scan, so the one serial
// lane only visits segment heads (binade changes, ties, single steps), each
// packed beforehand into one walk record; the run starts inside a segment
// are then filled in parallel, one item per lane, and re-checked against
// their binade.  Lists too long for LDS take a serial walk over global
// memory with the same arithmetic.
constexpr int kChainThreads = 256;
constexpr int kChainMaxBlocks = 2048;
constexpr int kChainMaxItems = 1152;
constexpr int kChainMaxTies = 512;

// One item (run or single step) in walk order; returns false on a failed
// binade check.  ties: the item's ties, nt of them.
template <class ItemRef, class TiePtr>
__device__ inline bool chain_item(const FoldArgs &A, int p, int b, ItemRef I, TiePtr ties, int nt, double &x,
                                  long long extra_R) {
  if (I.kind == 1) {
    x = x + I.d;
    A.out[p][out_index(A, b * kFoldBlock + I.first)] = x;
    return true;
  }
  int kx;
  frexp(x, &kx);
  if (kx != I.k || (x > 0.0 ? 1 : -1) != I.sgn) return false;
  const long long m = (long long)ldexp(x, 53 - I.k);
  I.m_start = m;
  long long ups = 0;
  for (int q = 0; q < nt; q++) {
    const long long val = m + ties[q].P + ups;
    const int up = (int)(val & 1LL);
    ties[q].up = up;
    ups += up;
  }
  const long long mend = m + I.R + extra_R + ups;
  const long long am = mend < 0 ? -mend : mend;
  if (am < (1LL << 52) || am >= (1LL << 53)) return false;
  x = ldexp((double)mend, I.k - 53);
  return true;
}

static_assert(kChainThreads == kFoldThreads, "the chain uses the fold's block scans");

// One serial step of the chain's walk: a segment head (run or single step).
struct ChainHead {
  union {
    long long R;  // kind 0: total of the segment's runs (ties rounded down)
    double d;     // kind 1: the step's increment
  };
  int out;        // kind 1: output index of the step
  short k, tie_first, nt;
  signed char kind, sgn;
};

// Exclusive prefix of the per-thread chunk sums of v[0..n) (chunks of
// ceil(n / kChainThreads) consecutive entries), written in place; returns the
// total.  One wave-level scan and one block barrier pair.
__device__ inline int chain_excl_scan(int *v, int n, int *sh) {
  const int tid = threadIdx.x;
  const int per = (n + kChainThreads - 1) / kChainThreads;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  int sum = 0;
  for (int j = lo; j < hi; j++) sum += v[j];
  int total;
  int run = block_excl_sum(sum, sh, &total);
  for (int j = lo; j < hi; j++) {
    const int c = v[j];
    v[j] = run;
    run += c;
  }
  __syncthreads();
  return total;
}

__global__ __launch_bounds__(kChainThreads) void k_fold_chain(FoldArgs A, FoldWork W) {
  __shared__ int s_io[kChainMaxBlocks + 1], s_to[kChainMaxBlocks + 1];
  __shared__ int s_tmp[kChainThreads / 64];
  __shared__ long long s_ltmp[2 * (kChainThreads / 64)];
  __shared__ int s_ftmp[kChainThreads / 64];
  __shared__ FoldItem s_items[kChainMaxItems];
  __shared__ FoldTie s_ties[kChainMaxTies];
  __shared__ long long s_pref[kChainMaxItems];  // exclusive R prefix inside the segment
  __shared__ int s_head[kChainMaxItems];        // head flags
  __shared__ int s_seg[kChainMaxItems];         // item -> block (gather), then item -> segment
  __shared__ int s_hlist[kChainMaxItems];       // segment -> head item
  __shared__ long long s_mh[kChainMaxItems];    // segment -> exact start of the head run
  __shared__ ChainHead s_hinfo[kChainMaxItems];
  __shared__ int s_nheads, s_ok;
  const int p = blockIdx.x;
  const int tid = threadIdx.x;
  if (W.status[p]) return;
  const int nblk = A.nblk;
  const int *gni = W.nitems + p * nblk, *gnt = W.nties + p * nblk;
  FoldItem *gitems = W.items + (size_t)p * nblk * kFoldMaxItems;
  FoldTie *gties = W.ties + (size_t)p * nblk * kFoldMaxTies;
  bool fits = nblk <= kChainMaxBlocks;
  int TI = 0, TT = 0;
  if (fits) {
    for (int b = tid; b < nblk; b += kChainThreads) {
      s_io[b] = gni[b];
      s_to[b] = gnt[b];
    }
    __syncthreads();
    TI = chain_excl_scan(s_io, nblk, s_tmp);
    TT = chain_excl_scan(s_to, nblk, s_tmp);
    fits = TI <= kChainMaxItems && TT <= kChainMaxTies;
  }
  if (!fits) {
    if (tid != 0) return;
    double x = A.x0[p];
    A.out[p][A.i0] = x;
    for (int b = 0; b < nblk; b++) {
      FoldItem *it = gitems + (size_t)b * kFoldMaxItems;
      FoldTie *tb = gties + (size_t)b * kFoldMaxTies;
      const int ni = gni[b], nt = gnt[b];
      for (int q = 0; q < ni; q++) {
        const int t0 = it[q].tie_first, t1 = (q + 1 < ni) ? it[q + 1].tie_first : nt;
        if (!chain_item<FoldItem &>(A, p, b, it[q], tb + t0, t1 - t0, x, 0)) {
          W.status[p] = 1;
          return;
        }
      }
    }
    return;
  }
  if (tid == 0) {
    s_io[nblk] = TI;
    s_to[nblk] = TT;
  }
  __syncthreads();
  // block of every item (LDS only), and the ties of every block
  for (int b = tid; b < nblk; b += kChainThreads) {
    const int io = s_io[b], ni = s_io[b + 1] - io;
    for (int j = 0; j < ni; j++) s_seg[io + j] = b;
    const int to = s_to[b], nt = s_to[b + 1] - to;
    for (int j = 0; j < nt; j++) s_ties[to + j] = gties[(size_t)b * kFoldMaxTies + j];
  }
  __syncthreads();
  // gather: independent loads, items get their block and a block-global tie offset
  for (int i = tid; i < TI; i += kChainThreads) {
    const int b = s_seg[i];
    FoldItem it = gitems[(size_t)b * kFoldMaxItems + (i - s_io[b])];
    it.blk = b;
    it.tie_first += s_to[b];
    s_items[i] = it;
  }
  __syncthreads();
  // tie count of item i: up to the next item's first tie, or the block's end
  auto nties_of = [&](int i) {
    const FoldItem &I = s_items[i];
    const int end = (i + 1 < TI && s_items[i + 1].blk == I.blk) ? s_items[i + 1].tie_first : s_to[I.blk + 1];
    return end - I.tie_first;
  };
  // segment heads: single steps, items with ties and their successors,
  // changes of binade or sign
  for (int i = tid; i < TI; i += kChainThreads) {
    const FoldItem &I = s_items[i];
    int h = 1;
    if (i > 0) {
      const FoldItem &Q = s_items[i - 1];
      h = (I.kind != 0 || Q.kind != 0 || nties_of(i) > 0 || nties_of(i - 1) > 0 || I.k != Q.k || I.sgn != Q.sgn) ? 1 : 0;
    }
    s_head[i] = h;
  }
  __syncthreads();
  const int per = (TI + kChainThreads - 1) / kChainThreads;
  const int lo = min(TI, tid * per), hi = min(TI, lo + per);
  {
    // segmented exclusive scan of R over items: chunk summaries, then lanes
    long long tail = 0;
    int has = 0, cnt = 0;
    for (int j = lo; j < hi; j++) {
      if (s_head[j]) {
        has = 1;
        tail = 0;
        cnt++;
      }
      tail += s_items[j].kind == 0 ? s_items[j].R : 0;
    }
    const long long incl = block_seg_incl(tail, has, s_ltmp, s_ftmp);
    long long carry = __shfl_up(incl, 1, 64);
    if ((tid & 63) == 63) s_ltmp[kChainThreads / 64 + (tid >> 6)] = incl;
    __syncthreads();
    if ((tid & 63) == 0) carry = (tid > 0) ? s_ltmp[kChainThreads / 64 + (tid >> 6) - 1] : 0;
    int nheads;
    int pos = block_excl_sum(cnt, s_tmp, &nheads);
    long long run = carry;
    for (int j = lo; j < hi; j++) {
      if (s_head[j]) {
        run = 0;
        s_hlist[pos++] = j;
      }
      s_pref[j] = run;
      s_seg[j] = pos - 1;
      run += s_items[j].kind == 0 ? s_items[j].R : 0;
    }
    if (tid == 0) s_nheads = nheads;
  }
  __syncthreads();
  const int nh = s_nheads;
  // one walk record per segment
  for (int q = tid; q < nh; q += kChainThreads) {
    const int h = s_hlist[q];
    const int last = ((q + 1 < nh) ? s_hlist[q + 1] : TI) - 1;
    const FoldItem &I = s_items[h];
    ChainHead H;
    H.kind = (signed char)I.kind;
    H.sgn = (signed char)I.sgn;
    H.k = (short)I.k;
    H.tie_first = (short)I.tie_first;
    H.nt = (short)nties_of(h);
    if (I.kind == 1) {
      H.d = I.d;
      H.out = out_index(A, I.blk * kFoldBlock + I.first);
    } else {
      H.R = (last > h) ? s_pref[last] + s_items[last].R : I.R;
      H.out = 0;
    }
    s_hinfo[q] = H;
  }
  __syncthreads();
  // serial walk over the segment heads; the next record is read ahead
  if (tid == 0) {
    double x = A.x0[p];
    A.out[p][A.i0] = x;
    int ok = 1;
    ChainHead Hn = s_hinfo[0];
    for (int q = 0; q < nh; q++) {
      const ChainHead H = Hn;
      if (q + 1 < nh) Hn = s_hinfo[q + 1];
      if (H.kind == 1) {
        x = x + H.d;
        A.out[p][H.out] = x;
        s_mh[q] = 0;
        continue;
      }
      int kx;
      frexp(x, &kx);
      if (kx != H.k || (x > 0.0 ? 1 : -1) != H.sgn) {
        ok = 0;
        break;
      }
      const long long m = (long long)ldexp(x, 53 - H.k);
      s_mh[q] = m;
      long long ups = 0;
      for (int t = 0; t < H.nt; t++) {
        FoldTie &T = s_ties[H.tie_first + t];
        const int up = (int)((m + T.P + ups) & 1LL);
        T.up = up;
        ups += up;
      }
      const long long mend = m + H.R + ups;
      const long long am = mend < 0 ? -mend : mend;
      if (am < (1LL << 52) || am >= (1LL << 53)) {
        ok = 0;
        break;
      }
      x = ldexp((double)mend, H.k - 53);
    }
    s_ok = ok;
    if (!ok) W.status[p] = 1;
  }
  __syncthreads();
  if (!s_ok) return;
  // exact start of every run, re-checked against its binade
  int bad = 0;
  for (int i = tid; i < TI; i += kChainThreads) {
    const int q = s_seg[i];
    long long m = s_mh[q];
    if (i > s_hlist[q]) {
      m += s_pref[i];
      const long long am = m < 0 ? -m : m;
      if (am < (1LL << 52) || am >= (1LL << 53)) bad = 1;
    }
    s_items[i].m_start = m;
  }
  if (bad) W.status[p] = 1;
  __syncthreads();
  for (int i = tid; i < TI; i += kChainThreads) {
    const int b = s_items[i].blk;
    gitems[(size_t)b * kFoldMaxItems + (i - s_io[b])].m_start = s_items[i].m_start;
  }
  for (int b = tid; b < nblk; b += kChainThreads) {
    const int to = s_to[b], nt = s_to[b + 1] - to;
    for (int j = 0; j < nt; j++) gties[(size_t)b * kFoldMaxTies + j].up = s_ties[to + j].up;
  }
}

// Single-pass alternative to k_fold_local<false> + k_fold_chain +
// k_fold_local<true>: each workgroup rounds the increments of its block on
// the block's grid and obtains the exact value before its first step by a
// decoupled look-back over the blocks before it (Merrill and Garland,
// "Single-pass Parallel Prefix Scan with Decoupled Look-back", 2016), with
// the exact fold as the operator:
// - a block whose values lie on one binade grid for certain acts on the value
//   before it as m -> m + R (m the value in units of its binade's ulp), so
//   consecutive such blocks on one grid compose by adding their totals; it
//   publishes R and its grid key as soon as it has its approximate start;
// - a block that crosses into the next binade once, or holds exact ties, acts
//   on the value before it through that value's last two bits (CrossAction):
//   it publishes the ends of four representative starts, and later blocks
//   apply it themselves;
// - every block publishes its exact end value.
// Each published value is one 64-bit word written and polled with relaxed
// device-scope atomics, so no fence orders it against anything else; "not
// yet" and "failed" are signalling-NaN patterns arithmetic never produces.
// The look-back reads 64 predecessors at a time with one wave, adds the
// totals of the nearest run of blocks on one grid, sets each crossing block it
// meets aside and stops at the first block with an exact end value, from
// which it applies them forward; it waits only on blocks that are neither
// (the first one, and those whose binade the approximate values leave open).
// Every block checks its own start and end against its binades as the chain
// does, so a result that passes is the chain's result bit for bit; a failed
// check, too many serial units or a wait longer than kLookSpinCap polls marks
// the phase, which k_fold_replay then replays serially.
// Blocks take tickets from their phase's counter in the order they start, so
// every block a workgroup waits on has started before it and waits only on
// earlier blocks itself: the waits cannot form a cycle.
constexpr int kLookSpinCap = 1 << 18;

__device__ inline long long look_load(const long long *v) {
  return __hip_atomic_load(v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void look_store(long long *v, long long x) {
  __hip_atomic_store(v, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a value every lane holds, kept in scalar registers
__device__ inline double uniform_double(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffLL));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// a 64-bit value of lane q, read by every lane of the wave
__device__ inline long long lane_read64(long long v, int q) {
  const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffLL), q);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), q);
  return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// binade key of an exact value, as binade_key with E = 0 (-1 for 0, inf, NaN)
__device__ inline int exact_key(double x) {
  if (!(fabs(x) > 0.0) || !(fabs(x) < __builtin_inf())) return -1;
  int kx;
  frexp(x, &kx);
  return (kx + 4096) * 2 + (x > 0.0 ? 1 : 0);
}

// Action of a block whose steps are runs on grid kin, one certain step into
// the next binade up or down, and runs on grid kout.  Moving the start by 4
// units of kin's ulp keeps every parity on the way (ties round alike) and
// moves the end by 2, 4 or 8 units of kout's ulp (one binade up, none, one
// down), so the ends of four consecutive starts m0 .. m0 + 3 (m0 a multiple
// of 4) give the end of any other start on grid kin.
struct CrossAction {
  int kin, kout;     // binade keys; kin < 0: none
  long long m0;
  long long end[4];
};

// Look-back state of block j: 2 end value known (or failed; v its bits), 1 on
// one grid with its action published (v the total, key the grid), 3 crossing
// with its action published, 0 none of these (yet).
struct LookState {
  int st;
  long long v;
};
__device__ inline LookState look_state(const long long *lw, int j, int &key) {
  const long long *w = lw + (size_t)j * kLW;
  const long long iw = look_load(w + kLwIncl);  // all loads in flight at once
  const long long aw = look_load(w + kLwAct), kw = look_load(w + kLwKey);
  key = -1;
  if (iw != kLookEmpty) return {2, iw};
  if (aw == kLookCross) return {3, 0};
  if (aw != kLookEmpty && aw != kLookNone && kw != kLookEmpty) {
    key = (int)kw;
    return {1, aw};
  }
  return {0, 0};
}

// The action of crossing block j (state 3).  Its words are stored before the
// state's, but unordered with it: each is polled until it is there.
__device__ inline bool cross_load(const long long *lw, int j, CrossAction &c) {
  const long long *w = lw + (size_t)j * kLW;
  for (int spins = 0; spins <= kLookSpinCap; spins++) {
    const long long k = look_load(w + kLwXKey);
    c.m0 = look_load(w + kLwXBase);
    bool have = k != kLookEmpty && c.m0 != kLookEmpty;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      c.end[r] = look_load(w + kLwXEnd + r);
      have = have && c.end[r] != kLookEmpty;
    }
    if (have) {
      c.kin = (int)(k & 0xffffff);
      c.kout = (int)(k >> 24);
      return true;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

// The end of a crossing block that starts at x; false when x is not on its grid.
__device__ inline bool cross_apply(const CrossAction &c, double &x) {
  if (exact_key(x) != c.kin) return false;
  const int ki = (c.kin >> 1) - 4096, ko = (c.kout >> 1) - 4096;
  const long long m = (long long)ldexp(x, 53 - ki);
  const int r = (int)(m & 3);
  const long long q = (m - c.m0 - r) >> 2;  // exact
  const long long e = r == 0 ? c.end[0] : r == 1 ? c.end[1] : r == 2 ? c.end[2] : c.end[3];
  const long long n = e + q * (ko > ki ? 2 : ko == ki ? 4 : 8);
  const long long an = n < 0 ? -n : n;
  if (an < (1LL << 52) || an >= (1LL << 53)) return false;
  x = ldexp((double)n, ko - 53);
  return true;
}

// The value before a block from an exact end value w and the blocks combined
// after it (key K, total c; K < 0: none).
__device__ inline bool look_finish(long long w, int K, long long c, double &x_out) {
  if (w == kLookFail) return false;
  double x = __longlong_as_double(w);
  if (K >= 0) {
    if (exact_key(x) != K) return false;
    const int k = (K >> 1) - 4096;
    const long long m = (long long)ldexp(x, 53 - k) + c;
    const long long am = m < 0 ? -m : m;
    if (am < (1LL << 52) || am >= (1LL << 53)) return false;
    x = ldexp((double)m, k - 53);
  }
  x_out = x;
  return true;
}

// One phase of one fold direction: its arrays picked once, at the top of the
// kernel, so that they stay in scalar registers.
struct FoldPhase {
  const double *rate;
  double *out;
  double x0, dt;
  int i0, nsteps;
};

// Crossing blocks met by one look-back, nearest first, each with the blocks
// on one grid combined after it.  A waveform's phase crosses a binade about
// 20 times, most of them inside block 0, which no block looks past; a block
// beyond the stack's end is waited for.
constexpr int kLookStack = 32;
struct LookPending {
  long long c;
  int K, j;
};

// Wave 0: exact value before block b's first step.  Returns false when the
// phase failed (a failed predecessor, a failed binade check, a wait past the
// cap).  `pend`: kLookStack entries of LDS.
__device__ inline bool fold_look_back(const FoldPhase &F, const long long *lw, int b, LookPending *pend,
                                      double &x_out) {
  const int lane = threadIdx.x & 63;
  int j = b - 1;     // nearest block of the window
  int K = -1;        // grid key of the combined blocks
  long long c = 0;   // their total
  int spins = 0, np = 0;
  // the end value w of a block, through the combined blocks and those set aside
  auto finish = [&](long long w) {
    if (!look_finish(w, K, c, x_out)) return false;
    while (np > 0) {
      np--;
      const LookPending &q = pend[np];
      CrossAction ca;
      if (!cross_load(lw, q.j, ca) || !cross_apply(ca, x_out)) return false;
      if (!look_finish(__double_as_longlong(x_out), q.K, q.c, x_out)) return false;
    }
    return true;
  };
  for (;;) {
    const int jb = j - lane;
    // block -1 stands for the start value x0
    LookState S = {2, __double_as_longlong(F.x0)};
    int key = -1;
    if (jb >= 0) S = look_state(lw, jb, key);
    int start = 0;  // lanes before it are combined or set aside
    for (;;) {
      const int s0 = __shfl(S.st, start, 64);
      const int k0 = __shfl(key, start, 64);
      const int Kc = (K >= 0) ? K : (s0 == 1 ? k0 : -2);
      const bool ext = S.st == 1 && key == Kc && key >= 0;
      const unsigned long long mask = ~(__ballot(ext) >> start);
      const int s = min(64, mask ? start + __builtin_ctzll(mask) : 64);
      if (s > start) {
        long long v = (lane >= start && lane < s) ? S.v : 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        c += v;
        K = Kc;
      }
      if (s == 64) {
        j -= 64;
        break;
      }
      const int js = j - s, ss = __shfl(S.st, s, 64);
      if (ss == 2) return finish(__shfl(S.v, s, 64));
      if (ss == 3 && np < kLookStack) {
        if (lane == 0) pend[np] = LookPending{c, K, js};
        __builtin_amdgcn_wave_barrier();
        np++;
        K = -1;
        c = 0;
        start = s + 1;
        if (start < 64) continue;
        j -= 64;
        break;
      }
      // not yet published, or on another grid: wait for a change of state; an
      // end value is used at once, a newly published action is combined by the
      // next window, which starts at that block
      LookState T;
      int tk;
      do {
        if (++spins > kLookSpinCap) return false;
        __builtin_amdgcn_s_sleep(1);
        T = look_state(lw, js, tk);
      } while (T.st == ss);
      if (T.st == 2) return finish(T.v);
      j = js;
      break;
    }
  }
}

// Wave 0: the approximate value before block b (S) and |x0| plus the L1 norm
// of the increments before it (L), from the sums every block publishes right
// after loading its rates; the nearest block with published prefixes ends
// the walk back.  The blocks waited on publish their sums without waiting
// themselves, so the waits are short.  Returns false after a wait past the
// cap.
__device__ inline bool approx_look_back(const FoldPhase &F, const long long *lw, int b, double &S, double &L) {
  const int lane = threadIdx.x & 63;
  int j = b - 1;
  double s = 0.0, l = 0.0;
  int spins = 0;
  for (;;) {
    const int jb = j - lane;
    int st = 2;  // block -1 stands for the start value
    double vs = F.x0, vl = fabs(F.x0);
    if (jb >= 0) {
      const long long *w = lw + (size_t)jb * kLW;
      const long long is = look_load(w + kLwIncS), il = look_load(w + kLwIncL);
      const long long as = look_load(w + kLwAggS), al = look_load(w + kLwAggL);
      if (is != kLookEmpty && il != kLookEmpty) {
        vs = __longlong_as_double(is);
        vl = __longlong_as_double(il);
      } else if (as != kLookEmpty && al != kLookEmpty) {
        st = 1;
        vs = __longlong_as_double(as);
        vl = __longlong_as_double(al);
      } else {
        st = 0;
      }
    }
    const unsigned long long m2 = __ballot(st == 2), m0 = __ballot(st == 0);
    const int f2 = m2 ? __builtin_ctzll(m2) : 64, f0 = m0 ? __builtin_ctzll(m0) : 64;
    // lanes before the first unpublished block, or through the nearest prefix
    const int upto = (f0 < f2) ? f0 : (f2 < 64 ? f2 + 1 : 64);
    double ts = (lane < upto) ? vs : 0.0, tl = (lane < upto) ? vl : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ts += __shfl_xor(ts, o, 64);
      tl += __shfl_xor(tl, o, 64);
    }
    s += ts;
    l += tl;
    if (f0 < f2) {
      j -= f0;
      for (;;) {
        if (++spins > kLookSpinCap) return false;
        __builtin_amdgcn_s_sleep(1);
        const long long *w = lw + (size_t)j * kLW;
        const long long as = look_load(w + kLwAggS), al = look_load(w + kLwAggL);
        if (as != kLookEmpty && al != kLookEmpty) break;
      }
      continue;
    }
    if (f2 < 64) {
      S = s;
      L = l;
      return true;
    }
    j -= 64;
  }
}

// Inclusive sum over the wave, lanes in order, by data-parallel moves (shifts
// inside rows of 16 lanes, then two row broadcasts).
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double wave_scan(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr 1
  v = dpp_add<0x112, 0xf>(v);  // row_shr 2
  v = dpp_add<0x114, 0xf>(v);  // row_shr 4
  v = dpp_add<0x118, 0xf>(v);  // row_shr 8
  v = dpp_add<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  return v;
}
__device__ inline double lane_readd(double v, int q) { return __longlong_as_double(lane_read64(__double_as_longlong(v), q)); }

// A block's steps in units of 64: register q of wave w holds unit 4 q + w, one
// step per lane, so loads, stores and scans all run along the lanes.
constexpr int kFoldUnits = kFoldBlock / 64;
constexpr int kFoldSerial = 24;  // units of one block that may be replayed step by step
constexpr int kFoldBatch = 4;     // steps per lane whose loads are in flight together
static_assert(kFoldUnits == 64, "one lane per unit");

// Place of step `off` of a block among its 4096 array elements, lowest index first.
template <int DIR>
__device__ inline unsigned fold_elem(unsigned off) { return DIR > 0 ? off : kFoldBlock - 1 - off; }

// The increments of block b, through a buffer descriptor of its elements (one
// offset register for all loads); steps past the end read the last step's
// rates (in bounds).
template <int DIR>
__device__ inline void load_increments(const FoldPhase &F, int b, double *d) {
  const int ib = F.i0 + DIR * b * kFoldBlock;
  const unsigned n = (unsigned)min(kFoldBlock, F.nsteps - b * kFoldBlock);
  const double *base = F.rate + (DIR > 0 ? ib : ib - (kFoldBlock - 1));
  const double *prev = b > 0 ? base - DIR : base;  // the rate of the step before; step 0 takes its own
  const int shift = b > 0 ? 0 : -8 * DIR;
  typedef int v2i __attribute__((ext_vector_type(2)));
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, kFoldBlock * 8, 0x00020000);
  const auto rp = __builtin_amdgcn_make_buffer_rsrc((void *)prev, 0, kFoldBlock * 8, 0x00020000);
  unsigned tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // offsets are cheaper formed again than kept
#pragma unroll
  for (int h = 0; h < kFoldPerThread; h += kFoldBatch) {
    double r[kFoldBatch], rm[kFoldBatch];
#pragma unroll
    for (int q = 0; q < kFoldBatch; q++) {
      const int e = 8 * (int)fold_elem<DIR>(min(tid + (h + q) * kFoldThreads, n - 1));
      r[q] = __builtin_bit_cast(double, (v2i)__builtin_amdgcn_raw_buffer_load_b64(rb, e, 0, 0));
      // step 0 of the fold reads out of the descriptor's range (0) and is set below
      rm[q] = __builtin_bit_cast(double, (v2i)__builtin_amdgcn_raw_buffer_load_b64(rp, e + shift, 0, 0));
    }
#pragma unroll
    for (int q = 0; q < kFoldBatch; q++) {
      if (h + q == 0 && b == 0 && tid == 0) rm[q] = r[q];
      const double v = (1.5 * r[q] - .5 * rm[q]) * F.dt;
      d[h + q] = (tid + (h + q) * kFoldThreads < n) ? (DIR > 0 ? v : -v) : 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Grid of the values on the way from a through increments of sum s and L1 norm
// l, each known to within E, where that is certain: the values lie between
// a - (l - s) / 2 and a + (l + s) / 2.  The frexp exponent, or -5000; also
// -5000 where an increment may pass a quarter of the binade (the rounding by
// 1.5 2^52 u needs |d| <= 2^51 u).
__device__ inline int sure_exponent(double a, double s, double l, double E) {
  double lo = a - 0.5 * (l - s), hi = a + 0.5 * (l + s);
  if (a < 0.0) {
    const double t = lo;
    lo = -hi;
    hi = -t;
  }
  lo -= E;
  hi += E;
  if (!(lo > 0.0) || !(hi < 1e300)) return -5000;
  int k, kh;
  frexp(lo, &k);
  frexp(hi, &kh);
  return k == kh && l < ldexp(0.25, k) ? k : -5000;
}

// LDS of one workgroup of the single-pass fold.
struct FoldShared {
  double red[2 * (kFoldThreads / 64)];
  double xs, E, x;
  int t, ok, nserial, unsure;
  double sum[kFoldUnits], l1[kFoldUnits];  // per unit: approximate sum and L1 norm; rounded total in sum
  double xu[kFoldUnits];                   // exact start of each unit
  int slot[kFoldUnits];                    // row of ser holding the unit's increments; -1 on one grid, -2 with ties
  double adj[kFoldUnits][2];               // of a unit with ties, by parity of its start: what they add to its total
  unsigned long long flip[kFoldUnits][2];  // and the ties that round the other way
  unsigned long long up[kFoldUnits];       // ties whose other neighbour lies above
  double ser[kFoldSerial][64];
  double park[kFoldPerThread][64];
  LookPending pend[kLookStack];
};

// Walk of wave 0 over its block's units from x (EXACT: the same in every lane;
// otherwise one start per lane).  Lane u holds unit u: its grid exponent,
// rounded total and serial row.  A run of units on one grid is one add of
// exact sums; a serial unit is replayed step by step.  EXACT: xu receives the
// exact start of the lane's unit and the serial units' values are written.
template <bool EXACT, int DIR>
__device__ inline bool fold_walk(const FoldPhase &F, FoldShared &S, int b, int k, int slot, double R,
                                 double &x, double &xu) {
  const int lane = threadIdx.x & 63;
  const unsigned long long serial = __ballot(slot >= 0), tied = __ballot(slot == -2);
  bool good = true;
  int pos = 0;
  while (pos < kFoldUnits) {
    const unsigned long long rest = serial >> pos;
    if (rest & 1) {
      // a chain of dependent adds, the next increments loaded ahead; EXACT: one
      // lane walks and leaves each value in its increment's place
      double *ser = S.ser[__builtin_amdgcn_readlane(slot, pos)];
      if (!EXACT || lane == 0) {
        double v[4], w[4];
        auto chain = [&](int h, double *c) {
#pragma unroll
          for (int s = 0; s < 4; s++) c[s] = x = x + c[s];
          if (EXACT)
#pragma unroll
            for (int s = 0; s < 4; s++) ser[h + s] = c[s];
        };
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = ser[s];
#pragma unroll 1
        for (int h = 0; h < 64; h += 8) {
#pragma unroll
          for (int s = 0; s < 4; s++) w[s] = ser[h + 4 + s];
          __builtin_amdgcn_sched_barrier(0);
          chain(h, v);
#pragma unroll
          for (int s = 0; s < 4; s++) v[s] = ser[((h + 8) & 63) + s];
          __builtin_amdgcn_sched_barrier(0);
          chain(h + 4, w);
        }
      }
      if (EXACT) {
        x = uniform_double(x);
        __builtin_amdgcn_wave_barrier();
        const int s = b * kFoldBlock + pos * 64 + lane;
        if (s < F.nsteps) F.out[F.i0 + DIR * (s + 1)] = ser[lane];
      }
      pos++;
      continue;
    }
    const int kk = __builtin_amdgcn_readlane(k, pos);
    const int key = (kk + 4096) * 2 + (x > 0.0 ? 1 : 0);
    if ((tied >> pos) & 1) {
      // exact ties: the total by the parity of the start
      good = good && exact_key(x) == key;
      if (EXACT && lane == pos) xu = x;
      x = x + (lane_readd(R, pos) + S.adj[pos][(long long)ldexp(x, 53 - kk) & 1]);
      good = good && exact_key(x) == key;
      pos++;
      continue;
    }
    const unsigned long long stop = rest | (tied >> pos);
    const int end = stop ? pos + __builtin_ctzll(stop) : kFoldUnits;
    const bool in = lane >= pos && lane < end;
    good = good && __ballot(in && k != kk) == 0 && exact_key(x) == key;
    const double incl = wave_scan(in ? R : 0.0);
    if (EXACT && in) xu = x + (incl - R);
    x = x + lane_readd(incl, 63);
    good = good && exact_key(x) == key;
    pos = end;
  }
  return good;
}

// The kernel is bound by latency: a block loads, waits for the approximate
// sums of those before it, rounds, and waits for its exact start.  So what
// counts is that all blocks of a 2^21-sample waveform run at once (1536
// workgroups; six per CU) and that no block is late.  A block on one grid u
// (all but about 20 per phase) rounds each step with one add and one subtract
// of 1.5 2^52 u, and every sum of the rounded steps is a multiple of u below
// 2^53 u, so plain FP64 scans are exact; its steps stay in registers, one
// per lane, from load to store.  Other blocks test each unit of 64 steps in
// the same way and replay the few units that hold a crossing or a tie.
// Classifying every step into item lists staged in LDS (39 KB, four
// workgroups per CU, a second wave of them) took 78 us per waveform at
// N = 2^21, this form 61 us.
template <int DIR>
__global__ __launch_bounds__(kFoldThreads, 6) void k_fold_resolve(FoldArgs A, FoldWork W) {
  __shared__ FoldShared S;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = blockIdx.y;
  const FoldPhase F = {A.rate[p], A.out[p], A.x0[p], A.dt, A.i0, A.nsteps};
  int *status = W.status + p;
  unsigned *ctr = W.look_ctr + p * kLookCtrStride;
  long long *lw = W.look + (size_t)p * A.nblk * kLW;
  if (tid == 0) {
    S.t = (int)atomicAdd(ctr, 1u);
    S.nserial = 0;
    S.unsure = 0;
    // entry: a phase already marked (the replay hook) skips to the end
    S.ok = __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
  }
  __syncthreads();
  const int b = __builtin_amdgcn_readfirstlane(S.t);
  long long *mw = lw + (size_t)b * kLW;  // this block's words
  double d[kFoldPerThread];
  load_increments<DIR>(F, b, d);
  // the block's approximate sum and L1 norm, published at once for the
  // approximate look-back of the blocks after it
  double tsum = 0.0, tl1 = 0.0;
#pragma unroll
  for (int q = 0; q < kFoldPerThread; q++) {
    tsum += d[q];
    tl1 += fabs(d[q]);
  }
  tsum = wave_scan(tsum);
  tl1 = wave_scan(tl1);
  if (lane == 63) {
    S.red[wave] = tsum;
    S.red[kFoldThreads / 64 + wave] = tl1;
  }
  __syncthreads();
  double bsum = 0.0, bl1 = 0.0;
#pragma unroll
  for (int w = 0; w < kFoldThreads / 64; w++) {
    bsum += S.red[w];
    bl1 += S.red[kFoldThreads / 64 + w];
  }
  // approximate start of the block, and the bound E on the distance between
  // approximate and exact values in it: every value up to the block's end,
  // either way, is at most U = |x0| + the L1 norm so far in magnitude, so
  // each of at most nsteps + 2 kFoldBlock roundings on either path is at most
  // half an ulp of U
  if (wave == 0) {
    if (lane == 0) {
      look_store(mw + kLwAggL, __double_as_longlong(bl1));
      look_store(mw + kLwAggS, __double_as_longlong(bsum));
    }
    double s = F.x0, L = fabs(F.x0);
    const bool aok = (b == 0) || approx_look_back(F, lw, b, s, L);
    if (lane == 0) {
      look_store(mw + kLwIncL, __double_as_longlong(L + bl1));
      look_store(mw + kLwIncS, __double_as_longlong(s + bsum));
      const double U = (L + bl1) * (1.0 + 0x1p-24);
      int ex = 0;
      frexp(U > 0.0 ? U : 1.0, &ex);
      S.xs = s;
      S.E = ((double)F.nsteps + 2.0 * kFoldBlock) * ldexp(1.0, ex - 52);
      if (!aok) S.ok = 0;
    }
  }
  __syncthreads();
  const double E = uniform_double(S.E), xs = uniform_double(S.xs);
  bool ok = __builtin_amdgcn_readfirstlane(S.ok) != 0;
  const int kb = ok ? __builtin_amdgcn_readfirstlane(sure_exponent(xs, uniform_double(bsum), uniform_double(bl1), E)) : -5000;
  bool on_grid = kb > -5000;
  // The loops over the units are rolled and rotate the units through d[0]: the
  // kernel is short enough for instruction fetch to count.
  // Wave 0 leaves its steps in LDS while it looks back, so that the look-back's
  // registers come on top of none of them (80 in all: six workgroups per CU).
  auto park = [&]() {
#pragma unroll
    for (int q = 0; q < kFoldPerThread; q++) S.park[q][lane] = d[q];
  };
  auto unpark = [&]() {
#pragma unroll
    for (int q = 0; q < kFoldPerThread; q++) d[q] = S.park[q][lane];
  };
  auto rotate = [&](double last) {
#pragma unroll
    for (int q = 0; q + 1 < kFoldPerThread; q++) d[q] = d[q + 1];
    d[kFoldPerThread - 1] = last;
  };
  if (on_grid) {
    const double C = ldexp(1.5, kb - 1), half = ldexp(0.5, kb - 53);
    int tie = 0;
#pragma unroll 1
    for (int q = 0; q < kFoldPerThread; q++) {
      const double v = (d[0] + C) - C;
      tie |= fabs(d[0] - v) == half;
      const double sc = wave_scan(v);
      if (lane == 63) S.sum[4 * q + wave] = sc;
      rotate(sc);
    }
    on_grid = __syncthreads_or(tie) == 0;
    if (!on_grid) load_increments<DIR>(F, b, d);
  }
  const int ib = F.i0 + DIR * b * kFoldBlock;
  double *op = F.out + (DIR > 0 ? ib + 1 : ib - kFoldBlock);  // element 0 of the block
  const unsigned n = (unsigned)min(kFoldBlock, F.nsteps - b * kFoldBlock);
  unsigned off0 = tid;
  asm volatile("" : "+v"(off0));
  if (on_grid) {
    const double R = S.sum[lane], incl = wave_scan(R);
    const double tot = lane_readd(incl, 63);
    if (wave == 0) {
      park();
      const int key = (kb + 4096) * 2 + (xs > 0.0 ? 1 : 0);
      if (lane == 0) {
        look_store(mw + kLwKey, (long long)key);
        look_store(mw + kLwAct, (long long)ldexp(tot, 53 - kb));
      }
      double x = 0.0;
      bool wok = b == 0 ? (x = F.x0, true) : fold_look_back(F, lw, b, S.pend, x);
      if (W.force_replay == 2 && b == A.nblk / 2) wok = false;  // test hook
      wok = wok && exact_key(x) == key && exact_key(x + tot) == key;
      if (lane == 0) {
        if (!wok) __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        look_store(mw + kLwIncl, wok ? __double_as_longlong(x + tot) : kLookFail);
        if (wok && b == 0) F.out[F.i0] = x;
        S.x = x;
        S.ok = wok ? 1 : 0;
      }
      unpark();
    }
    __syncthreads();
    if (!S.ok) return;
    const double xu = S.x + (incl - R);  // exact start of unit `lane`
#pragma unroll 1
    for (int q = 0; q < kFoldPerThread; q++, rotate(d[0]))
      if (off0 + q * kFoldThreads < n)
        op[fold_elem<DIR>(off0 + q * kFoldThreads)] = lane_readd(xu, 4 * q + wave) + d[0];
    return;
  }
  // a block with a crossing, ties or values near zero: unit by unit
  int k = -5000, slot = -1;
  double R = 0.0;
  if (ok) {
#pragma unroll 1
    for (int q = 0; q < kFoldPerThread; q++) {
      const double s = wave_scan(d[0]);
      const unsigned long long neg = __ballot(d[0] < 0.0), fin = __ballot(d[0] == d[0]);
      const double l = (fin == ~0ULL && (neg == 0 || neg == ~0ULL)) ? fabs(s) : wave_scan(fabs(d[0]));
      if (lane == 63) {
        S.sum[4 * q + wave] = s;
        S.l1[4 * q + wave] = l;
      }
      rotate(d[0]);
    }
    __syncthreads();
    const double us = S.sum[lane], ul = S.l1[lane];
    const double au = xs + (wave_scan(us) - us);  // approximate start of unit `lane`
    k = sure_exponent(au, us, ul, E);
    const int kin = sure_exponent(xs, 0.0, 0.0, E);
    __syncthreads();
#pragma unroll 1
    for (int q = 0; q < kFoldPerThread; q++) {
      const int u = 4 * q + wave, ku = __builtin_amdgcn_readlane(k, u);
      const double du = d[0], C = ldexp(1.5, ku - 1), v = (du + C) - C;
      double res = du;
      if (ku > -5000) {
        res = wave_scan(v);
        const unsigned long long ties = __ballot(fabs(du - v) == ldexp(0.5, ku - 53));
        if (ties) {
          // v is the even multiple; a tie rounds to the other one when the
          // value before it is odd, which also turns every later parity
          const unsigned long long odd = __ballot((long long)ldexp(res - v, 53 - ku) & 1);
          const unsigned long long up = __ballot(v < du) & ties;
          if (lane < 2) {
            unsigned long long flip = 0, par = lane;
            int add = 0;
            for (unsigned long long t = ties; t; t &= t - 1) {
              const int i = __builtin_ctzll(t);
              if ((par ^ (odd >> i)) & 1) {
                flip |= 1ULL << i;
                add += (up >> i) & 1 ? 1 : -1;
                par ^= 1;
              }
            }
            S.flip[u][lane] = flip;
            S.adj[u][lane] = ldexp((double)add, ku - 53);
          }
          if (lane == 0) S.up[u] = up;
        }
        if (lane == 63) {
          S.sum[u] = res;
          S.slot[u] = ties ? -2 : -1;
        }
      } else {
        // steps whose binade is open, or two binades up, leave no action to publish
        const int ks = sure_exponent(lane_readd(au, u) + wave_scan(du), 0.0, 0.0, E);
        const bool sure = kin > -5000 && ks > -5000 && ks <= kin + 1;
        int row = 0;
        if (lane == 0) {
          row = atomicAdd(&S.nserial, 1);
          S.slot[u] = row;
        }
        row = __builtin_amdgcn_readfirstlane(row);
        if (__ballot(sure) != ~0ULL && lane == 0) S.unsure = 1;
        if (row < kFoldSerial) S.ser[row][lane] = du;
      }
      rotate(res);
    }
    __syncthreads();
    R = S.sum[lane];
    slot = S.slot[lane];
    if (slot >= 0) k = -5000;
    ok = S.nserial <= kFoldSerial;
  }
  if (wave == 0) {
    park();
    const int kin = sure_exponent(xs, 0.0, 0.0, E);
    bool pub = ok && b > 0 && !S.unsure && kin > -5000 && __ballot(k > kin + 1) == 0;
    if (pub) {
      // four consecutive starts about the approximate one, lanes 0..3 (and
      // again in every four lanes)
      const long long m0 = (long long)ldexp(xs, 53 - kin) & ~3LL;
      double y = ldexp((double)(m0 + (lane & 3)), kin - 53), unused;
      const bool good = fold_walk<false, DIR>(F, S, b, k, slot, R, y, unused);
      const int kout = exact_key(y), kd = (kout >> 1) - (kin + 4096);
      const bool same = kout >= 0 && kd >= -1 && kd <= 1 && (kout & 1) == (xs > 0.0 ? 1 : 0) &&
                        kout == __builtin_amdgcn_readfirstlane(kout);
      pub = __ballot(good && same) == ~0ULL;
      if (pub) {
        if (lane < 4) look_store(mw + kLwXEnd + lane, (long long)ldexp(y, 53 - ((kout >> 1) - 4096)));
        if (lane == 0) {
          look_store(mw + kLwXBase, m0);
          look_store(mw + kLwXKey, ((long long)kout << 24) | ((kin + 4096) * 2 + (xs > 0.0 ? 1 : 0)));
        }
      }
    }
    if (lane == 0) look_store(mw + kLwAct, pub ? kLookCross : kLookNone);
    double x = 0.0, xu = 0.0;
    bool wok = ok && (b == 0 ? (x = F.x0, true) : fold_look_back(F, lw, b, S.pend, x));
    if (W.force_replay == 2 && b == A.nblk / 2) wok = false;  // test hook
    if (wok) {
      if (b == 0 && lane == 0) F.out[F.i0] = x;
      wok = fold_walk<true, DIR>(F, S, b, k, slot, R, x, xu);
      if (!(x == x)) wok = false;  // a NaN phase takes the serial replay
    }
    if (lane == 0) {
      if (!wok) __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      look_store(mw + kLwIncl, wok ? __double_as_longlong(x) : kLookFail);
      S.ok = wok ? 1 : 0;
    }
    S.xu[lane] = xu;
    unpark();
  }
  __syncthreads();
  if (!S.ok) return;
#pragma unroll 1
  for (int q = 0; q < kFoldPerThread; q++, rotate(d[0])) {
    const int u = 4 * q + wave;
    const int sl = S.slot[u];
    if (sl < 0 && off0 + q * kFoldThreads < n) {
      double v = d[0];
      if (sl == -2) {
        const int ku = __builtin_amdgcn_readlane(k, u);
        const unsigned long long f = S.flip[u][(long long)ldexp(S.xu[u], 53 - ku) & 1] & (~0ULL >> (63 - lane)), up = S.up[u];
        v = v + ldexp((double)((int)__popcll(f & up) - (int)__popcll(f & ~up)), ku - 53);
      }
      op[fold_elem<DIR>(off0 + q * kFoldThreads)] = S.xu[u] + v;
    }
  }
}

// serial replay of the phases whose single-pass fold failed
__global__ __launch_bounds__(kFoldThreads) void k_fold_replay(FoldArgs A, FoldWork W) {
  __shared__ double sd[kFoldLds];
  if (W.status[blockIdx.x]) fold_serial_replay(A, W, blockIdx.x, sd, 4096);
}

int fold_exact(const DenseParams &P, const DenseBuffers &B, const FoldWork &W, int nblk_cap, int dir, int nsteps,
               int mode, FoldArgs *defer_replay, hipStream_t s) {
  if (nsteps <= 0) return 0;
  FoldArgs A;
  for (int p = 0; p < 3; p++) {
    A.rate[p] = B.rate[p];
    A.out[p] = B.phase[p];
    A.x0[p] = P.x0[p];
  }
  A.i0 = P.i0;
  A.dir = dir;
  A.nsteps = nsteps;
  A.dt = P.dt;
  A.nblk = (nsteps + kFoldBlock - 1) / kFoldBlock;
  if (A.nblk > nblk_cap) return -1;
  if (mode == 0) {
    if (dir > 0) hipLaunchKernelGGL(k_fold_resolve<1>, dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
    else hipLaunchKernelGGL(k_fold_resolve<-1>, dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
    // the replay check can ride on the next launch that does not read the
    // phases (the mode-sum setup); otherwise it is a launch of its own
    if (defer_replay) *defer_replay = A;
    else hipLaunchKernelGGL(k_fold_replay, dim3(3), dim3(kFoldThreads), 0, s, A, W);
    return 0;
  }
  if (dir > 0) hipLaunchKernelGGL(k_fold_sums<1>, dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  else hipLaunchKernelGGL(k_fold_sums<-1>, dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  hipLaunchKernelGGL(k_fold_plan, dim3(3), dim3(1024), 0, s, A, W);
  if (dir > 0) hipLaunchKernelGGL((k_fold_local<false, 1>), dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  else hipLaunchKernelGGL((k_fold_local<false, -1>), dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  hipLaunchKernelGGL(k_fold_chain, dim3(3), dim3(kChainThreads), 0, s, A, W);
  if (dir > 0) hipLaunchKernelGGL((k_fold_local<true, 1>), dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  else hipLaunchKernelGGL((k_fold_local<true, -1>), dim3(A.nblk, 3), dim3(kFoldThreads), 0, s, A, W);
  return 0;
}

// per-waveform counters (non-positive Phidot samples, fold fallbacks); a
// kernel rather than a memset so the sequence can be captured in a graph
__global__ void k_clear_flags(int *flags) {
  if (threadIdx.x < 8) flags[threadIdx.x] = 0;
}

void launch_clear_flags(const DenseBuffers &B, hipStream_t s) {
  hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(64), 0, s, B.flags);
}

// Phases and frequencies per sample (AAKPhase.cc:338-346): t, Phi, Phi+gamma,
// Phi+gamma+alpha, Phidot, Phidot+gammadot, Phidot+gammadot+alphadot, e.
__global__ void k_phase_out(DenseParams P, DenseBuffers B, double *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int N = P.N;
  if (i >= N) return;
  const double gim = B.phase[0][i], Phi = B.phase[1][i], alp = B.phase[2][i];
  const double gd = B.rate[0][i], Pd = B.rate[1][i], ad = B.rate[2][i];
  out[i] = sample_time(P, i);
  out[(size_t)N + i] = Phi;
  out[2 * (size_t)N + i] = Phi + gim;
  out[3 * (size_t)N + i] = Phi + gim + alp;
  out[4 * (size_t)N + i] = Pd;
  out[5 * (size_t)N + i] = Pd + gd;
  out[6 * (size_t)N + i] = Pd + gd + ad;
  out[7 * (size_t)N + i] = B.e[i];
}

void launch_phase_out(const DenseParams &P, const DenseBuffers &B, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_phase_out, dim3((P.N + 255) / 256), dim3(256), 0, s, P, B, out);
}

// phases after the plunge buffer stay at their plunge values (AAK.cc:265-269)
__global__ void k_fold_fill(DenseParams P, DenseBuffers B) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + P.last_fold + 2;
  if (i > P.N) return;
  for (int p = 0; p < 3; p++) B.phase[p][i] = B.phase[p][P.ip];
}

void launch_fold_fill(const DenseParams &P, const DenseBuffers &B, hipStream_t s) {
  // only the dense arrays and the phase output read phases past the last
  // folded step; the mode sum of a likelihood stops at the end of the taper
  if (!P.full_dense) return;
  const int n = P.N - (P.last_fold + 2) + 1;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fold_fill, dim3((n + 255) / 256), dim3(256), 0, s, P, B);
}

// ------------------------------------------------------------------ mode sum
// J_{n-2..n+2}(x) by Miller's backward recurrence normalised with
// J_0 + 2 sum J_2k = 1 (A&S 9.12); n = 1 returns (-J_1, J_0, J_1, J_2, J_3).
__device__ inline void bessel_five(int n, double x, double *J) {
  if (x == 0.0) {
    for (int q = 0; q < 5; q++) J[q] = (n - 2 + q == 0) ? 1.0 : 0.0;
    if (n == 1) { J[0] = 0.0; J[1] = 1.0; J[2] = 0.0; J[3] = 0.0; J[4] = 0.0; }
    return;
  }
  const int nmax = n + 2;
  const int nmin = (n >= 2) ? n - 2 : 0;
  int top = nmax + 40 + (int)x;
  top += (top & 1);
  const double inv = 1.0 / x;
  double jp1 = 0.0, j = 1.0e-280, sum = 0.0;
  double w0 = 0, w1 = 0, w2 = 0, w3 = 0, w4 = 0;
  for (int k = top; k >= 1; k--) {
    const int q = k - nmin;
    if (q == 0) w0 = j;
    else if (q == 1) w1 = j;
    else if (q == 2) w2 = j;
    else if (q == 3) w3 = j;
    else if (q == 4) w4 = j;
    if ((k & 1) == 0) sum += 2.0 * j;
    const double jm1 = fma((2.0 * k) * inv, j, -jp1);
    jp1 = j;
    j = jm1;
    if (fabs(j) > 1.0e250) {
      j *= 1.0e-250; jp1 *= 1.0e-250; sum *= 1.0e-250;
      w0 *= 1.0e-250; w1 *= 1.0e-250; w2 *= 1.0e-250; w3 *= 1.0e-250; w4 *= 1.0e-250;
    }
  }
  if (nmin == 0) w0 = j;
  sum += j;
  const double norm = 1.0 / sum;
  if (n == 1) {
    J[1] = w0 * norm; J[2] = w1 * norm; J[3] = w2 * norm; J[4] = w3 * norm; J[0] = -J[2];
  } else {
    J[0] = w0 * norm; J[1] = w1 * norm; J[2] = w2 * norm; J[3] = w3 * norm; J[4] = w4 * norm;
  }
}

// Per-sample part of the mode sum (AAK.cc:425-481): everything that does not
// depend on the harmonic, folded into the weights of a_n, b_n, c_n in h_I and
// h_II, so that h = Amp * sum_n [cos(nPhi)(alpha_n W_a + gamma_n W_c) +
// sin(nPhi) beta_n W_b] with a_n = Amp alpha_n cos(nPhi) etc. (AAK.cc:493-504).
struct SampleGeom {
  double e, Phi, nu, gimdot, Amp, ti, cosorbphs;
  double W[6];  // a, b, c weights of h_I, then of h_II
};

__device__ inline double affine_sc(const double *c, double sa, double ca) { return c[0] + c[1] * sa + c[2] * ca; }

// The harmonic-independent quantities need only be accurate (they set
// amplitudes and the Doppler term), except the orientation angle's argument
// 2 (gamma + beta), which is rounded as in the reference; the sample time and
// the dense arrays are read as they are.
__device__ inline void sample_geometry(const DenseParams &P, const DenseBuffers &B, int i, SampleGeom &G) {
#pragma clang fp contract(fast)
  const double ti = sample_time(P, i);
  const double e = B.e[i];
  const double gim = B.phase[0][i], alp = B.phase[2][i];
  G.ti = ti;
  G.e = e;
  G.Phi = B.phase[1][i];
  G.gimdot = B.rate[0][i];
  G.nu = (i == 0) ? B.nu0[0] : B.rate[1][i] * (0.5 / kPi);
  const double coslam = P.coslam;
  const double cosqS = P.cosqS, sinqS = P.sinqS, cosqK = P.cosqK, sinqK = P.sinqK;
  const double halfsqrt3 = P.halfsqrt3;
  double sa, ca;
  sincos(alp, &sa, &ca);
  // orientation of L (AAK.cc:425-433)
  const double cosqL = affine_sc(P.g_cosqL, sa, ca);
  const double sinqL = sqrt(1. - cosqL * cosqL);
  const double phiLup = affine_sc(P.g_phiLup, sa, ca), phiLdown = affine_sc(P.g_phiLdown, sa, ca);
  // cos(phiL - phiS) with phiL = atan2(phiLup, phiLdown) (atan2(0, 0) = 0)
  const double rL2 = phiLup * phiLup + phiLdown * phiLdown;
  const double irL = rL2 > 0. ? rsqrt(rL2) : 0.;
  const double cphiL = rL2 > 0. ? phiLdown * irL : 1., sphiL = phiLup * irL;
  const double Ldotn = cosqL * cosqS + sinqL * sinqS * (cphiL * P.cos_phS + sphiL * P.sin_phS);
  const double Ldotn2 = Ldotn * Ldotn;
  const double betaup = -P.Sdotn + coslam * Ldotn;
  const double betadown = affine_sc(P.g_betadown, sa, ca);
  const double beta = atan2(betaup, betadown);
  // the reference's rounded argument 2 (gamma + beta) of the orientation angle
  const double gb = gim + beta;
  const double gam = 2. * gb;
  double sin2gam, cos2gam;
  sincos(gam, &sin2gam, &cos2gam);
  double cosorbphs = 0.0, FplusI, FcrosI, FplusII, FcrosII, h3;
  if (P.mich) {
    // LISA orbit phase; the shifted angles by angle subtraction from one sincos
    const double orbphs = 2. * kPi * ti / kYear;
    double so, co;
    sincos(orbphs, &so, &co);
    cosorbphs = co * P.cos_phS + so * P.sin_phS;             // cos(orbphs - phiS)
    const double sinorbphs = so * P.cos_phS - co * P.sin_phS;  // sin(orbphs - phiS)
    const double cosorbK = co * P.cos_phK + so * P.sin_phK;    // cos(orbphs - phiK)
    const double cosq = .5 * cosqS - halfsqrt3 * sinqS * cosorbphs;
    // phiw = orbphs + atan2(Yw, Xw): double angles by (X^2 - Y^2, 2XY) / (X^2 + Y^2)
    const double Yw = halfsqrt3 * cosqS + .5 * sinqS * cosorbphs, Xw = sinqS * sinorbphs;
    const double rw = Xw * Xw + Yw * Yw;
    const double irw = rw > 0. ? 1. / rw : 0.;
    const double c2w = rw > 0. ? (Xw * Xw - Yw * Yw) * irw : 1., s2w = 2. * Xw * Yw * irw;
    const double c2o = co * co - so * so, s2o = 2. * so * co;
    const double cos2phi = c2o * c2w - s2o * s2w, sin2phi = s2o * c2w + c2o * s2w;
    const double psiup = .5 * cosqK - halfsqrt3 * sinqK * cosorbK - cosq * P.psi_c0;
    const double psidown = P.psi_c1 - halfsqrt3 * co * P.psi_c2 - halfsqrt3 * so * P.psi_c3;
    const double rp = psiup * psiup + psidown * psidown;
    const double irp = rp > 0. ? 1. / rp : 0.;
    const double cos2psi = rp > 0. ? (psidown * psidown - psiup * psiup) * irp : 1.;
    const double sin2psi = 2. * psidown * psiup * irp;
    const double cosq1 = .5 * (1. + cosq * cosq);
    FplusI = cosq1 * cos2phi * cos2psi - cosq * sin2phi * sin2psi;
    FcrosI = cosq1 * cos2phi * sin2psi + cosq * sin2phi * cos2psi;
    FplusII = cosq1 * sin2phi * cos2psi + cosq * cos2phi * sin2psi;
    FcrosII = cosq1 * sin2phi * sin2psi - cosq * cos2phi * cos2psi;
    h3 = halfsqrt3;
  } else {
    FplusI = P.ldc_c2psi;
    FcrosI = -P.ldc_s2psi;
    FplusII = P.ldc_s2psi;
    FcrosII = P.ldc_c2psi;
    h3 = 1.0;
  }
  G.cosorbphs = cosorbphs;
  G.Amp = B.amp[i];
  // rotation to the wave frame (KSParMap.cc:532-574): cos(rot) = (nxL).(nxS) / N,
  // sin(rot) = (L.(nxS) - S.(nxL)) / N, N = |nxL| |nxS|, all affine or quadratic
  // in (sin alpha, cos alpha)
  const double cn = affine_sc(P.g_rc, sa, ca), sn = affine_sc(P.g_rs, sa, ca);
  const double *q2 = P.g_nxL2;
  const double nxL2 = q2[0] + q2[1] * (sa * sa) + q2[2] * (ca * ca) + q2[3] * sa + q2[4] * ca + q2[5] * (sa * ca);
  const double iN2 = 1. / (nxL2 * P.nxS2);
  const double rot0 = 2. * (cn * cn) * iN2 - 1., rot1 = cn * sn * iN2;
  // h = Ap0 X + Ac0 Y per channel, with Ap0, Ac0 linear in (a, b, c)
  const double XI = h3 * (FplusI * rot0 - FcrosI * rot1), YI = h3 * (FplusI * rot1 + FcrosI * rot0);
  const double XII = h3 * (FplusII * rot0 - FcrosII * rot1), YII = h3 * (FplusII * rot1 + FcrosII * rot0);
  const double pa = -(1. + Ldotn2) * cos2gam, pb = (1. + Ldotn2) * sin2gam, pc = 1. - Ldotn2;
  const double qa = 2. * Ldotn * sin2gam, qb = 2. * Ldotn * cos2gam;
  G.W[0] = pa * XI + qa * YI;
  G.W[1] = pb * XI + qb * YI;
  G.W[2] = pc * XI;
  G.W[3] = pa * XII + qa * YII;
  G.W[4] = pb * XII + qb * YII;
  G.W[5] = pc * XII;
}

// Angle reduced to [-pi, pi] in FP64, returned in FP32 (the reduction error,
// ~k 2.4e-16 rad, is far below FP32 resolution).
__device__ inline float reduce_2pi_f(double x) {
  const double k = rint(x * (1.0 / (2.0 * kPi)));
  return (float)fma(-k, 6.283185307179586, x);
}

// Hardware sine/cosine (v_sin_f32, v_cos_f32; absolute error ~1e-6 for
// |x| <= 4 pi): the response factors they feed set amplitudes, where such
// errors are far below the FP32 harmonic sum's own.
__device__ inline void sincos_hw(float x, float *s, float *c) {
  *s = __sinf(x);
  *c = __cosf(x);
}

// The mixed form's per-sample geometry: the same response as sample_geometry,
// rebuilt in FP32 from unit vectors after the large angles (gamma, alpha, the
// orbital phase) are reduced mod 2 pi in FP64.  With P = cos g E1 + sin g E2,
// Q = L x P (E1, E2 the orbital-plane pair of GeomF32), the harmonic-n
// quadrupole is -a_n (PP - QQ) - b_n (PQ + QP) + c_n (PP + QQ), and a
// channel with (transverse-traceless) response tensor R reads it as R : H.
// For LISA, R = sqrt 3 Lambda(D) with D = (x x - y y)/2 (channel I) or
// (x y + y x)/2 (channel II) on the cartwheel's arm frame (x, y) at orbital
// phase 2 pi t / yr, and Lambda the TT projection about n:
// E Lambda(D) E' = eps D eps' + (eps . eps') (n D n) / 2, eps = E - (n.E) n.
// Without LISA, R = pp - qq and pq + qp on the sky basis.  Nothing here
// divides by a quantity that can vanish, so orientations where the reference's
// angles are ill-conditioned (n along L or S, the source near the detector's
// normal) cost no accuracy.  The phase, its rates, e, t and the amplitude are
// read as they are.
__device__ inline void sample_geometry_mixed(const DenseParams &P, const DenseBuffers &B, int i, SampleGeom &G) {
#pragma clang fp contract(fast)
  const GeomF32 &F = P.gf;
  const double ti = sample_time(P, i);
  G.ti = ti;
  G.e = B.e[i];
  G.Phi = B.phase[1][i];
  G.gimdot = B.rate[0][i];
  G.nu = (i == 0) ? B.nu0[0] : B.rate[1][i] * (0.5 / kPi);
  G.Amp = B.amp[i];
  const float gim = reduce_2pi_f(B.phase[0][i]), alp = reduce_2pi_f(B.phase[2][i]);
  float sa, ca, s2g, c2g;
  sincos_hw(alp, &sa, &ca);
  sincos_hw(2.f * gim, &s2g, &c2g);
  float E1[3], E2[3];
  for (int k = 0; k < 3; k++) {
    E1[k] = F.e1c[k] + F.e1s[k] * sa + F.e1k[k] * ca;
    E2[k] = F.e2s[k] * sa + F.e2k[k] * ca;
  }
  // r[ch][0..2] = E1 R E1, E2 R E2, E1 R E2 of each channel
  float r[2][3];
  float cosorbphs = 0.f;
  if (P.mich) {
    float so, co;
    sincos_hw(reduce_2pi_f(2. * kPi * ti / kYear), &so, &co);
    cosorbphs = co * F.cos_phS + so * F.sin_phS;
    const float h3 = 0.8660254037844386f;
    const float x[3] = {0.5f * so * co, -(co * co + 0.5f * so * so), -h3 * so};
    const float y[3] = {so * so + 0.5f * co * co, -0.5f * so * co, h3 * co};
    auto dot3 = [](const float *a, const float *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; };
    const float nx = dot3(F.n, x), ny = dot3(F.n, y), n1 = dot3(F.n, E1), n2 = dot3(F.n, E2);
    const float x1 = dot3(E1, x) - n1 * nx, y1 = dot3(E1, y) - n1 * ny;
    const float x2 = dot3(E2, x) - n2 * nx, y2 = dot3(E2, y) - n2 * ny;
    const float g11 = 1.f - n1 * n1, g22 = 1.f - n2 * n2, g12 = -n1 * n2;
    const float tI = 0.5f * (nx * nx - ny * ny), tII = nx * ny;
    const float s3 = 1.7320508075688772f;
    r[0][0] = s3 * (0.5f * (x1 * x1 - y1 * y1) + 0.5f * g11 * tI);
    r[0][1] = s3 * (0.5f * (x2 * x2 - y2 * y2) + 0.5f * g22 * tI);
    r[0][2] = s3 * (0.5f * (x1 * x2 - y1 * y2) + 0.5f * g12 * tI);
    r[1][0] = s3 * (x1 * y1 + 0.5f * g11 * tII);
    r[1][1] = s3 * (x2 * y2 + 0.5f * g22 * tII);
    r[1][2] = s3 * (0.5f * (x1 * y2 + y1 * x2) + 0.5f * g12 * tII);
  } else {
    const float p1 = F.p[0] * E1[0] + F.p[1] * E1[1] + F.p[2] * E1[2];
    const float q1 = F.q[0] * E1[0] + F.q[1] * E1[1] + F.q[2] * E1[2];
    const float p2 = F.p[0] * E2[0] + F.p[1] * E2[1] + F.p[2] * E2[2];
    const float q2 = F.q[0] * E2[0] + F.q[1] * E2[1] + F.q[2] * E2[2];
    r[0][0] = p1 * p1 - q1 * q1;
    r[0][1] = p2 * p2 - q2 * q2;
    r[0][2] = p1 * p2 - q1 * q2;
    r[1][0] = 2.f * p1 * q1;
    r[1][1] = 2.f * p2 * q2;
    r[1][2] = p1 * q2 + q1 * p2;
  }
  G.cosorbphs = cosorbphs;
  for (int ch = 0; ch < 2; ch++) {
    const float dlt = r[ch][0] - r[ch][1], two12 = 2.f * r[ch][2];
    G.W[3 * ch + 0] = -(c2g * dlt + s2g * two12);
    G.W[3 * ch + 1] = -(c2g * two12 - s2g * dlt);
    G.W[3 * ch + 2] = r[ch][0] + r[ch][1];
  }
}

// Planck taper between plunge and zero time (AAK.cc:535-547)
__device__ inline double taper(const DenseParams &P, int i, double ti) {
  if (i <= P.ip) return 1.0;
  const double tp = P.t_plunge, tz = P.t_zero;
  return exp((tp - tz) / (ti - tp) + (tp - tz) / (ti - tz)) + 1.;
}

// Doppler-shifted harmonic phase exactly as the reference rounds it.
__device__ inline double harmonic_phase(const DenseParams &P, const SampleGeom &G, double nn, double gdpi) {
  if (P.mich) {
    const double fn = nn * G.nu + gdpi;
    const double Doppler = 2. * kPi * fn * kAUsec * P.sinqS * G.cosorbphs;
    return nn * G.Phi + Doppler;
  }
  return nn * G.Phi;
}

// ------------------------------------------------------------------ Taylor form
// Inside one block of samples e varies by a few 1e-5: the amplitude factors
// alpha_n, beta_n, gamma_n are expanded in delta = e - e_ref once per block
// (k_modesum_setup) and evaluated per sample by Horner (k_modesum).  The order
// p is the smallest with remainder bound 7 n (n delta)^{p+1}/(p+1)! <= 1e-17
// (1e-9 for the FP32 harmonic loop of the mixed form).
// Blocks where no order up to kTaylorMax qualifies, or where the Bessel series
// is not used (e > kSeriesMaxE, more than kTaylorModes harmonics), are summed
// per sample by k_modesum_direct.
constexpr int kMsThreads = 256;
constexpr int kTaylorModes = 128;
// Samples per expansion block: 256 << exp_shift (host-set, default 2 in the
// mixed form and in FP64 from 2^18 signal samples on, else 0).  One expansion serves
// 1024 samples while the setup work falls fourfold and the mean order rises
// little (mixed, over the production prior: from 2.0 to 2.5); blocks that need
// more than order 8 are expanded per 256 samples.
__host__ __device__ inline int exp_shift(const DenseParams &P) { return P.xshift; }
constexpr int kSetupThreads = 64;
// doubles reserved per block in B.ms_coef per harmonic (orders up to kTaylorMax)
constexpr int kCoefStride = 3 * (kTaylorMax + 1);

// Uniform, read-only data through the scalar path: the coefficients of a block
// are the same for all its lanes, so they are fetched with scalar loads into
// SGPRs and feed the FMAs directly.
typedef const __attribute__((address_space(4))) double *cdptr;
typedef const __attribute__((address_space(4))) float *cfptr;
typedef const __attribute__((address_space(4))) int *ciptr;

// B.ms_p[blk]: the Taylor order of 256-sample block blk, or -1 for the
// per-sample path; B.ms_slot[blk]: the slot of its expansion (coefficients
// and e_ref).
__device__ inline int block_order(const DenseBuffers &B, int blk) { return ((ciptr)B.ms_p)[blk]; }
__device__ inline int block_slot(const DenseBuffers &B, int blk) { return ((ciptr)B.ms_slot)[blk]; }

template <int PO, bool MIXED>
__device__ void setup_harmonics(const DenseParams &P, const DenseBuffers &B, int blk, double eref, const double *sq,
                                double *sJ) {
  constexpr int NC = 3 * (PO + 1);
  for (int n = threadIdx.x + 1; n <= P.nmodes; n += kSetupThreads) {
    // series length: the bound for orders n+1, n+2 covers the higher orders
    bessel_run<kSetupThreads>(n, PO, eref, B.bessel_c, B.bessel_lgf, P.bterms[n], sJ);
    const size_t base = (size_t)blk * P.nmodes * kCoefStride;
    // each coefficient is stored as soon as it is formed
    if (MIXED)
      taylor_amplitudes_p<PO, kSetupThreads>(
          n, eref, sq, sJ, CoefStore<PO, float>{reinterpret_cast<float *>(B.ms_coef + base) + (size_t)(n - 1) * NC});
    else
      taylor_amplitudes_p<PO, kSetupThreads>(n, eref, sq, sJ, CoefStore<PO, double>{B.ms_coef + base + (size_t)(n - 1) * NC});
  }
}

// Range of e over samples [i0, i0 + len) below n_end, reduced over the wave
// (every lane holds it); lo > hi when the range holds no signal sample.
__device__ inline void e_range(const DenseBuffers &B, int i0, int len, int n_end, double &lo, double &hi) {
  lo = 1e300;
  hi = -1e300;
  // eight loads in flight per lane before the first use
  constexpr int kU = 8;
  for (int q0 = threadIdx.x; q0 < len; q0 += kU * kSetupThreads) {
    double v[kU];
    bool in[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int q = q0 + u * kSetupThreads, i = i0 + q;
      in[u] = q < len && i < n_end;
      v[u] = in[u] ? B.e[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kU; u++)
      if (in[u]) {
        lo = fmin(lo, v[u]);
        hi = fmax(hi, v[u]);
      }
  }
  for (int o = 1; o < 64; o <<= 1) {
    lo = fmin(lo, __shfl_xor(lo, o));
    hi = fmax(hi, __shfl_xor(hi, o));
  }
}

// The expansion of one slot at order p about eref (one harmonic per lane).
template <bool MIXED>
__device__ inline void setup_slot(const DenseParams &P, const DenseBuffers &B, int slot, int p, double eref,
                                  double *sJ) {
  double sq[kTaylorMax + 1];
  taylor_sqrt1me2(eref, p, sq);
  switch (p) {
    case 0: setup_harmonics<0, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 1: setup_harmonics<1, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 2: setup_harmonics<2, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 3: setup_harmonics<3, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 4: setup_harmonics<4, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 5: setup_harmonics<5, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 6: setup_harmonics<6, MIXED>(P, B, slot, eref, sq, sJ); break;
    case 7: setup_harmonics<7, MIXED>(P, B, slot, eref, sq, sJ); break;
    default: setup_harmonics<8, MIXED>(P, B, slot, eref, sq, sJ); break;
  }
}

// Block setup, 2^xs waves per expansion block of 256 << xs samples, the first
// waves of all blocks before the second ones.  Each finds the range of e over
// the block's signal samples, the order p and e_ref (every lane derives the same
// values from a butterfly reduction); the first wave then expands, one harmonic
// per lane.  The Bessel run of a lane is staged in LDS (dynamic orders) and the
// expansion is formed in registers.  An expansion block of more than 256
// samples that no order up to kTaylorMax serves (fast evolution near a
// plunge) is expanded per 256 samples (slot ne + blk; flags[4] counts such
// blocks), one by each of its waves, which otherwise end with their look at the
// range.  A launch behind the setup that walked a list of such blocks took 5 us
// with an empty list (setup and sum, mixed, N = 2^21: 101 against 98 us) and 12
// to 18 more with 14 to 58 of them (FP64: 127 and 198 against 115 and 182).
// Other failures (no Bessel series: e > kSeriesMaxE, more than kTaylorModes
// harmonics; 256 samples beyond order kTaylorMax) list the 256-sample blocks for
// the per-sample path.  A block with no signal sample gets p = 0 and no
// coefficients.
template <bool MIXED>
__global__ __launch_bounds__(kSetupThreads) void k_modesum_setup(DenseParams P, DenseBuffers B, FoldArgs FA,
                                                                 FoldWork FW, int ne) {
  __shared__ double s_J[kTaylorOrders][kSetupThreads];
  const int xs = exp_shift(P), span = kMsThreads << xs, sub = 1 << xs;
  // the waves of a block lie a multiple of 8 workgroups apart: one XCD, whose
  // L2 then holds the block's e (17 against 66 MB read, 98 against 102 us)
  const int stride = (ne + 7) & ~7;
  const int lane = threadIdx.x, part = blockIdx.x / stride, eb = blockIdx.x % stride;
  if (part >= sub) {
    // workgroups past the expansion blocks': the serial replay of a phase
    // whose single-pass fold failed (the setup reads e only)
    const int p = blockIdx.x - stride * sub;
    if (FW.status[p]) fold_serial_replay(FA, FW, p, &s_J[0][0], kTaylorOrders * kSetupThreads);
    return;
  }
  if (eb >= ne) return;
  const int n_end = min(P.N, P.ip + P.ib);
  const int nb = (P.N + 2 + kMsThreads - 1) / kMsThreads;
  double lo, hi;
  e_range(B, eb * span, span, n_end, lo, hi);
  const double tol = MIXED ? kTaylorTolFp32 : kTaylorTolFp64;
  bool any = lo <= hi;
  const bool series = P.bessel_series && P.nmodes <= kTaylorModes && hi <= P.e_series;
  int p = -1, slot = eb, first = eb * sub, end = min(nb, first + sub);
  double eref = 0.0;
  if (!any) {
    p = 0;
  } else if (series) {
    eref = 0.5 * (lo + hi);
    p = taylor_order(P.nmodes, 0.5 * (hi - lo), tol);
  }
  if (p < 0 && series && sub > 1) {
    if (part == 0 && lane == 0) atomicAdd(&B.flags[4], 1);
    first += part;
    if (first >= nb) return;
    end = first + 1;
    slot = ne + first;
    e_range(B, first * kMsThreads, kMsThreads, n_end, lo, hi);
    any = lo <= hi;
    p = 0;
    eref = 0.0;
    if (any) {
      eref = 0.5 * (lo + hi);
      p = taylor_order(P.nmodes, 0.5 * (hi - lo), tol);
    }
  } else if (part > 0) {
    return;
  }
  if (lane == 0) {
    B.ms_eref[slot] = eref;
    for (int blk = first; blk < end; blk++) {
      B.ms_p[blk] = p;
      B.ms_slot[blk] = slot;
      if (p < 0) B.ms_list[atomicAdd(&B.flags[2], 1)] = blk;
    }
  }
  if (p < 0 || !any) return;
  setup_slot<MIXED>(P, B, slot, p, eref, &s_J[0][lane]);
}

int modesum_blocks(const DenseParams &P) { return (P.N + 2 + kMsThreads - 1) / kMsThreads; }
static int expansion_blocks(const DenseParams &P) {
  const int span = kMsThreads << exp_shift(P);
  return (P.N + 2 + span - 1) / span;
}
int modesum_slots(const DenseParams &P) { return expansion_blocks(P) + modesum_blocks(P); }

// Per-sample phase factors shared by both harmonic loops: u = exp(i (Phi + dA))
// with Phi reduced mod 2 pi (Cody-Waite, three parts of 2 pi) and q0 = exp(i dB),
// where the Doppler term of harmonic n is n dA + dB; q_n = q0 u^n by rotation.
struct PhaseSeed {
  double ur, ui, qr, qi, dA, dB;
};

template <bool MIXED>
__device__ inline void phase_seed(const DenseParams &P, const SampleGeom &G, PhaseSeed &S) {
  const double kq = rint(G.Phi * (1.0 / (2.0 * kPi)));
  double phr = fma(-kq, 6.283185307179586, G.Phi);
  phr = fma(-kq, 2.4492935982947064e-16, phr);
  phr = fma(-kq, -5.989539619436679e-33, phr);
  S.dA = 0.0;
  S.dB = 0.0;
  if (P.mich) {
    const double proj = kAUsec * P.sinqS * G.cosorbphs;
    S.dA = 2. * kPi * G.nu * proj;
    S.dB = 2. * G.gimdot * proj;
  }
  if (MIXED) {
    // the seeds of the FP32 loop.  u: sincosf of the FP32 angle, corrected to
    // first order by the angle's FP32 remainder (|remainder| <= 1.2e-7, so
    // the dropped second-order term is below 1e-14).  dB is a small angle (the
    // Doppler shift of the periapsis precession), so FP32 keeps its rotation
    // to ~6e-8.
    const double th = phr + S.dA;
    const float thf = (float)th, tl = (float)(th - (double)thf);
    float su, cu;
    sincosf(thf, &su, &cu);
    S.ui = fmaf(cu, tl, su);
    S.ur = fmaf(-su, tl, cu);
    float qi, qr;
    sincosf((float)S.dB, &qi, &qr);
    S.qi = qi;
    S.qr = qr;
  } else {
    sincos(phr + S.dA, &S.ui, &S.ur);
    sincos(S.dB, &S.qi, &S.qr);
  }
}

// FP64 harmonic loop at Taylor order PO.  The response factors are the same
// for every harmonic, so only the three sums
//   Sa = sum cos(s_n) alpha_n, Sg = sum cos(s_n) gamma_n, Sb = sum sin(s_n) beta_n
// are needed; with alpha_n = sum_j a_nj d^j (and likewise for beta, gamma)
// they are accumulated per power, Sa_j = sum_n cos(s_n) a_nj, one FMA with a
// scalar operand per coefficient, and combined with d^j after the loop.  The
// rotation gives exp(i theta), theta = n Phi + Doppler_n; the reference's
// argument is its rounded s_n = rn(rn(n Phi) + Doppler_n), which differs from
// theta by a few ulp of s_n (~1e-9 rad late in a year-long inspiral).
// E = theta - s_n = fma(n, Phi, -s_n) + Doppler_n, accurate to the rounding of
// Doppler_n (~1e-14 rad), and exp(i s_n) = exp(i theta) (1 - i E) to second
// order in E.
template <int PO>
__device__ inline void harmonics_fp64(int nmodes, cdptr cf, double Phi, double d, const PhaseSeed &S, double *sum) {
  constexpr int NC = 3 * (PO + 1);
  double qr = S.qr, qi = S.qi;
  double Sa[PO + 1], Sb[PO + 1], Sg[PO + 1];
#pragma unroll
  for (int j = 0; j <= PO; j++) Sa[j] = Sb[j] = Sg[j] = 0.0;
  const double ur = S.ur, ui = S.ui;
#pragma unroll 2
  for (int nn = 1; nn <= nmodes; nn++, cf += NC) {
    const double tr = fma(qr, ur, -(qi * ui));
    qi = fma(qr, ui, qi * ur);
    qr = tr;
    const double dn = (double)nn;
    const double D = fma(dn, S.dA, S.dB);
    const double s_ = dn * Phi + D;  // not contracted: rn(rn(n Phi) + D)
    const double E = fma(dn, Phi, -s_) + D;
    const double cnp = fma(E, qi, qr), snp = fma(-E, qr, qi);
#pragma unroll
    for (int j = 0; j <= PO; j++) {
      Sa[j] = fma(cnp, cf[j], Sa[j]);
      Sb[j] = fma(snp, cf[PO + 1 + j], Sb[j]);
      Sg[j] = fma(cnp, cf[2 * (PO + 1) + j], Sg[j]);
    }
  }
  double a = Sa[PO], b = Sb[PO], g = Sg[PO];
#pragma unroll
  for (int j = PO - 1; j >= 0; j--) {
    a = fma(a, d, Sa[j]);
    b = fma(b, d, Sb[j]);
    g = fma(g, d, Sg[j]);
  }
  sum[0] = a;
  sum[1] = b;
  sum[2] = g;
}

// FP32 harmonic loop (mixed precision): rotation and the per-power sums in
// FP32 from FP64-reduced phase factors; no argument correction.
template <int PO>
__device__ inline void harmonics_fp32(int nmodes, cfptr cf, float d, const PhaseSeed &S, double *sum) {
  constexpr int NC = 3 * (PO + 1);
  float qr = (float)S.qr, qi = (float)S.qi;
  float Sa[PO + 1], Sb[PO + 1], Sg[PO + 1];
#pragma unroll
  for (int j = 0; j <= PO; j++) Sa[j] = Sb[j] = Sg[j] = 0.f;
  const float ur = (float)S.ur, ui = (float)S.ui;
#pragma unroll 2
  for (int nn = 1; nn <= nmodes; nn++, cf += NC) {
    const float tr = fmaf(qr, ur, -(qi * ui));
    qi = fmaf(qr, ui, qi * ur);
    qr = tr;
#pragma unroll
    for (int j = 0; j <= PO; j++) {
      Sa[j] = fmaf(qr, cf[j], Sa[j]);
      Sb[j] = fmaf(qi, cf[PO + 1 + j], Sb[j]);
      Sg[j] = fmaf(qr, cf[2 * (PO + 1) + j], Sg[j]);
    }
  }
  float a = Sa[PO], b = Sb[PO], g = Sg[PO];
#pragma unroll
  for (int j = PO - 1; j >= 0; j--) {
    a = fmaf(a, d, Sa[j]);
    b = fmaf(b, d, Sb[j]);
    g = fmaf(g, d, Sg[j]);
  }
  sum[0] = a;
  sum[1] = b;
  sum[2] = g;
}

// Samples past the signal (or the two padding slots) get time and zeros.
__device__ inline bool modesum_tail(const DenseParams &P, const DenseBuffers &B, int i, int n_end) {
  double *hI = B.h, *hII = B.h2;
  if (i >= P.N) {
    B.t[i] = 0.0;
    hI[i] = 0.0;
    hII[i] = 0.0;
    return true;
  }
  if (i >= n_end) {
    B.t[i] = sample_time(P, i);
    hI[i] = 0.0;
    hII[i] = 0.0;
    return true;
  }
  return false;
}

// Taylor-form mode sum for blocks with B.ms_p >= 0.  MIXED: the harmonic loop
// runs in FP32 (phases, their reduction mod 2 pi, the block expansions and the
// final scaling stay FP64).
template <bool MIXED>
__device__ inline void modesum_block(const DenseParams &P, const DenseBuffers &B, int blk) {
  const int p = block_order(B, blk);
  if (p < 0) return;  // k_modesum_direct sums this block
  const int slot = block_slot(B, blk);
  const int i = blk * kMsThreads + threadIdx.x;
  if (i >= P.N + 2) return;
  const int n_end = min(P.N, P.ip + P.ib);  // samples [0, n_end) carry the signal
  if (modesum_tail(P, B, i, n_end)) return;
  SampleGeom G;
  if (MIXED) sample_geometry_mixed(P, B, i, G);
  else sample_geometry(P, B, i, G);
  B.t[i] = G.ti;
  PhaseSeed S;
  phase_seed<MIXED>(P, G, S);
  const double d = G.e - B.ms_eref[slot];
  const size_t base = (size_t)slot * P.nmodes * kCoefStride;
  double sum[3];
  if (MIXED) {
    cfptr cf = (cfptr)(B.ms_coef + base);
    const float fd = (float)d;
    switch (p) {
      case 0: harmonics_fp32<0>(P.nmodes, cf, fd, S, sum); break;
      case 1: harmonics_fp32<1>(P.nmodes, cf, fd, S, sum); break;
      case 2: harmonics_fp32<2>(P.nmodes, cf, fd, S, sum); break;
      case 3: harmonics_fp32<3>(P.nmodes, cf, fd, S, sum); break;
      case 4: harmonics_fp32<4>(P.nmodes, cf, fd, S, sum); break;
      case 5: harmonics_fp32<5>(P.nmodes, cf, fd, S, sum); break;
      case 6: harmonics_fp32<6>(P.nmodes, cf, fd, S, sum); break;
      case 7: harmonics_fp32<7>(P.nmodes, cf, fd, S, sum); break;
      default: harmonics_fp32<8>(P.nmodes, cf, fd, S, sum); break;
    }
  } else {
    cdptr cf = (cdptr)(B.ms_coef + base);
    switch (p) {
      case 0: harmonics_fp64<0>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 1: harmonics_fp64<1>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 2: harmonics_fp64<2>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 3: harmonics_fp64<3>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 4: harmonics_fp64<4>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 5: harmonics_fp64<5>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 6: harmonics_fp64<6>(P.nmodes, cf, G.Phi, d, S, sum); break;
      case 7: harmonics_fp64<7>(P.nmodes, cf, G.Phi, d, S, sum); break;
      default: harmonics_fp64<8>(P.nmodes, cf, G.Phi, d, S, sum); break;
    }
  }
  const double accI = G.W[0] * sum[0] + G.W[1] * sum[1] + G.W[2] * sum[2];
  const double accII = G.W[3] * sum[0] + G.W[4] * sum[1] + G.W[5] * sum[2];
  const double sc = (i <= P.ip) ? G.Amp : G.Amp / taper(P, i, G.ti);
  B.h[i] = sc * accI;
  B.h2[i] = sc * accII;
}

// One workgroup per 256-sample block, XCD-aware: workgroups are dispatched in
// index order and dealt to the 8 XCDs round-robin (workgroup g runs on XCD
// g % 8), so g is mapped to the block that puts the 2^xs sample blocks of one
// expansion block on one XCD (their Taylor coefficients are fetched into one
// L2) while the blocks in flight at any moment stay one contiguous stretch of
// the waveform, spread over every XCD (no XCD idles past a plunge).  Blocks
// beyond the last whole group of 8 << xs keep their index.
template <bool MIXED>
__global__ __launch_bounds__(kMsThreads) void k_modesum(DenseParams P, DenseBuffers B, int nb) {
  const int xs = exp_shift(P), g = blockIdx.x;
  const int full = nb / (8 << xs) * (8 << xs);
  int blk = g;
  if (g < full) {
    const int x = g & 7, r = g >> 3;
    blk = ((((r >> xs) << 3) | x) << xs) | (r & ((1 << xs) - 1));
  }
  modesum_block<MIXED>(P, B, blk);
}

// Per-sample mode sum for the 256-sample blocks listed by k_modesum_setup (B.ms_p < 0):
// eight lanes per sample, each summing every eighth harmonic (the per-harmonic
// Bessel and phase evaluation is the long part), partial sums combined by
// shuffles.  A fixed grid walks the list, 32 samples per workgroup.
constexpr int kDirectGroups = 8;
constexpr int kDirectSamples = kMsThreads / kDirectGroups;
constexpr int kDirectGrid = 1024;

__device__ inline void modesum_direct_part(const DenseParams &P, const DenseBuffers &B, const SampleGeom &G, int g,
                                           double *hI, double *hII) {
  const double e = G.e, sq1me2 = sqrt(1 - e * e), gdpi = G.gimdot / kPi;
  double accI = 0.0, accII = 0.0, J[5];
  for (int nn = 1 + g; nn <= P.nmodes; nn += kDirectGroups) {
    const double nPhi = harmonic_phase(P, G, (double)nn, gdpi);
    if (P.bessel_series && e <= P.e_series)
      bessel_five_series(nn, e, B.bessel_c, B.bessel_lgf, P.bterms[nn], P.bterms[0], J);
    else
      bessel_five(nn, nn * e, J);
    double snp, cnp;
    sincos(nPhi, &snp, &cnp);
    const double al = -nn * (J[0] - 2. * e * J[1] + 2. / nn * J[2] + 2. * e * J[3] - J[4]);
    const double be = -nn * sq1me2 * (J[0] - 2. * J[2] + J[4]);
    const double ga = 2. * J[2];
    accI += cnp * (al * G.W[0] + ga * G.W[2]) + snp * (be * G.W[1]);
    accII += cnp * (al * G.W[3] + ga * G.W[5]) + snp * (be * G.W[4]);
  }
  *hI = accI;
  *hII = accII;
}

__global__ __launch_bounds__(kMsThreads) void k_modesum_direct(DenseParams P, DenseBuffers B) {
  const int count = B.flags[2];
  const int span = kMsThreads;           // samples per listed block
  const int per = span / kDirectSamples;  // workgroup passes per listed block
  const int units = count * per;
  const int g = threadIdx.x % kDirectGroups, sl = threadIdx.x / kDirectGroups;
  const int n_end = min(P.N, P.ip + P.ib);
  for (int u = blockIdx.x; u < units; u += gridDim.x) {
    const int blk = B.ms_list[u / per];
    const int i = blk * span + (u % per) * kDirectSamples + sl;
    // every lane takes part in the shuffles below; inactive ones add zeros
    bool work = i < P.N + 2;
    if (work && g == 0) work = !modesum_tail(P, B, i, n_end);
    else if (work) work = (i < P.N && i < n_end);
    double accI = 0.0, accII = 0.0;
    SampleGeom G;
    if (work) {
      sample_geometry(P, B, i, G);
      modesum_direct_part(P, B, G, g, &accI, &accII);
    }
#pragma unroll
    for (int o = 1; o < kDirectGroups; o <<= 1) {
      accI += __shfl_xor(accI, o, 64);
      accII += __shfl_xor(accII, o, 64);
    }
    if (work && g == 0) {
      B.t[i] = G.ti;
      const double sc = (i <= P.ip) ? G.Amp : G.Amp / taper(P, i, G.ti);
      B.h[i] = sc * accI;
      B.h2[i] = sc * accII;
    }
  }
}

// Setup (every wave of an expansion block, and the replay of a deferred fold),
// the sum, and the blocks left to the per-sample path.
void launch_modesum(const DenseParams &P, const DenseBuffers &B, const FoldArgs *replay, const FoldWork *fw,
                    hipStream_t s) {
  const int nb = modesum_blocks(P), ne = expansion_blocks(P);
  const FoldArgs FA = replay ? *replay : FoldArgs{};
  const FoldWork FW = fw ? *fw : FoldWork{};
  const int ng = (((ne + 7) & ~7) << exp_shift(P)) + (replay ? 3 : 0);
  if (P.mixed) {
    hipLaunchKernelGGL(k_modesum_setup<true>, dim3(ng), dim3(kSetupThreads), 0, s, P, B, FA, FW, ne);
    hipLaunchKernelGGL(k_modesum<true>, dim3(nb), dim3(kMsThreads), 0, s, P, B, nb);
  } else {
    hipLaunchKernelGGL(k_modesum_setup<false>, dim3(ng), dim3(kSetupThreads), 0, s, P, B, FA, FW, ne);
    hipLaunchKernelGGL(k_modesum<false>, dim3(nb), dim3(kMsThreads), 0, s, P, B, nb);
  }
  hipLaunchKernelGGL(k_modesum_direct, dim3(kDirectGrid), dim3(kMsThreads), 0, s, P, B);
}

// ------------------------------------------------------------------ likelihood
// <h w, d> and <h w, h w> over two channels; the weighted spectrum is written
// back (the reference leaves h~ w in its FFT buffer).
constexpr int kDotThreads = 256;
constexpr int kDotBlocks = 1024;

__global__ __launch_bounds__(kDotThreads) void k_weighted_dot(const double2 *hf, const double2 *data, const double *w,
                                                              int nbins, double2 *hw_out, double *partials) {
  __shared__ double s_dh[kDotThreads], s_hh[kDotThreads];
  double dh = 0.0, hh = 0.0;
  const int total = 2 * nbins;
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < total; q += gridDim.x * blockDim.x) {
    const double2 h = hf[q];
    const double ww = w[q];
    const double2 x = make_double2(h.x * ww, h.y * ww);
    const double2 dd = data[q];
    dh += x.x * dd.x + x.y * dd.y;
    hh += x.x * x.x + x.y * x.y;
    if (hw_out) hw_out[q] = x;
  }
  s_dh[threadIdx.x] = dh;
  s_hh[threadIdx.x] = hh;
  __syncthreads();
  for (int o = kDotThreads / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s_dh[threadIdx.x] += s_dh[threadIdx.x + o];
      s_hh[threadIdx.x] += s_hh[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = s_dh[0];
    partials[2 * blockIdx.x + 1] = s_hh[0];
  }
}

// out = 4 x (sum of the partial pairs); NaN when the waveform was rejected
// on the device (flags[3], a non-positive radial rate at t = 0)
// flags: the waveform's flags (flags[3]: rejected on the device, the result
// is NaN) or null; clear: flags to zero once read (the lane's, so that its
// next waveform starts from zeros without a clearing launch) or null.
__global__ __launch_bounds__(kDotThreads) void k_dot_final(const double *partials, int nparts, double *out,
                                                           const int *flags, int *clear) {
  __shared__ double s_dh[kDotThreads], s_hh[kDotThreads];
  double dh = 0.0, hh = 0.0;
  // four pairs in flight per lane before the first add; the adds keep the
  // order of one pair per step
  constexpr int kU = 4;
  for (int q0 = threadIdx.x; q0 < nparts; q0 += kU * kDotThreads) {
    double2 v[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int q = q0 + u * kDotThreads;
      v[u] = (q < nparts) ? reinterpret_cast<const double2 *>(partials)[q] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < kU; u++)
      if (q0 + u * kDotThreads < nparts) {
        dh += v[u].x;
        hh += v[u].y;
      }
  }
  s_dh[threadIdx.x] = dh;
  s_hh[threadIdx.x] = hh;
  __syncthreads();
  for (int o = kDotThreads / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s_dh[threadIdx.x] += s_dh[threadIdx.x + o];
      s_hh[threadIdx.x] += s_hh[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const bool bad = flags && flags[3] != 0;
    out[0] = bad ? __builtin_nan("") : 4.0 * s_dh[0];
    out[1] = bad ? __builtin_nan("") : 4.0 * s_hh[0];
  }
  __syncthreads();
  if (clear && threadIdx.x < 8) clear[threadIdx.x] = 0;
}

void launch_dot_final(const double *partials, int nparts, double *out, const int *flags, int *clear, hipStream_t s) {
  hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(kDotThreads), 0, s, partials, nparts, out, flags, clear);
}

void launch_weighted_dot(const double2 *hf, const double2 *data, const double *w, int nbins, double2 *hw_out,
                         double *partials, double *out, const int *flags, int *clear, hipStream_t s) {
  const int need = (2 * nbins + kDotThreads - 1) / kDotThreads;
  const int nb = need < kDotBlocks ? need : kDotBlocks;
  hipLaunchKernelGGL(k_weighted_dot, dim3(nb), dim3(kDotThreads), 0, s, hf, data, w, nbins, hw_out, partials);
  hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(kDotThreads), 0, s, partials, nb, out, flags, clear);
}

}  // namespace aak
