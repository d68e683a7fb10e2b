// aak_fft.hip -- noise-weighted inner products of a real waveform pair on
// CDNA4 (gfx950): a real FFT of length N = 2M fused with the PSD weighting and
// the two reductions <h w, d w> and <h w, h w> (AAK_manager.cu:352-446 and
// kernel.cu:557-567 semantics: one-sided spectrum, DC and Nyquist bins with
// full weight).
//
// The M-point complex FFT of z_m = h_2m + i h_2m+1 runs in four-step form with
// M = R C, m = a C + b, k = k1 + R k2:
//   pass 1 (k_fft_cols):  R-point FFTs down the columns b, times W_M^(b k1);
//   pass 2 (k_fft_rows):  C-point FFTs along the rows k1.
// Row k1 and row R - k1 hold Z_k and Z_(M-k) for every k of either row, so the
// second pass also forms the real spectrum H_k = E_k + W_N^k O_k,
// E_k = (Z_k + conj Z_(M-k)) / 2, O_k = (Z_k - conj Z_(M-k)) / 2i, weights it
// and accumulates the two sums; the spectrum is written only on request.  The
// weighted data and weights are stored once, at input time, in that pass's
// order (row k1, then k2), so every read is contiguous.  HBM traffic per
// likelihood is about 2 x (16 + 16 + 16 + 16 + 8) MB at N = 2^21.
//
// Each FFT is a Stockham autosort transform of radix-16 stages (a radix-8,
// -4 or -2 stage finishes lengths that are not powers of 16) on registers,
// exchanging through LDS between stages; LDS rows carry one pad element per 16
// so that the stride-16 writes of the first stage spread over all banks.
// Twiddles come from tables computed on the host in extended precision.
#include <hip/hip_runtime.h>

#include "aak_fft.hpp"

namespace aak {

__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cmul_mi(double2 a) { return make_double2(a.y, -a.x); }  // a * (-i)

// cos(pi/8), sin(pi/8), sqrt(1/2)
constexpr double kC8 = 0.92387953251128675613;
constexpr double kS8 = 0.38268343236508977173;
constexpr double kR2 = 0.70710678118654752440;
constexpr double kS3 = 0.86602540378443864676;  // sin(2 pi / 3)
constexpr double kC20 = 0.93969262078590838405, kS20 = 0.34202014332566873304;  // cos, sin of 20 degrees,
constexpr double kC40 = 0.76604444311897803520, kS40 = 0.64278760968653932632;  // 40 and
constexpr double kC80 = 0.17364817766693034885, kS80 = 0.98480775301220805937;  // 80

__device__ __forceinline__ void dft4(double2 &a0, double2 &a1, double2 &a2, double2 &a3) {
  const double2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = cmul_mi(csub(a1, a3));
  a0 = cadd(t0, t2);
  a1 = cadd(t1, t3);
  a2 = csub(t0, t2);
  a3 = csub(t1, t3);
}

__device__ __forceinline__ void dft3(double2 &a0, double2 &a1, double2 &a2) {
  const double2 t = cadd(a1, a2), u = cmul_mi(csub(a1, a2));
  const double2 c = make_double2(a0.x - 0.5 * t.x, a0.y - 0.5 * t.y);
  a0 = cadd(a0, t);
  a1 = make_double2(c.x + kS3 * u.x, c.y + kS3 * u.y);
  a2 = make_double2(c.x - kS3 * u.x, c.y - kS3 * u.y);
}

// Forward DFT of RS points, v in natural order, o out in natural order.
template <int RS>
__device__ __forceinline__ void dft(double2 *v, double2 *o) {
  if constexpr (RS == 2) {
    o[0] = cadd(v[0], v[1]);
    o[1] = csub(v[0], v[1]);
  } else if constexpr (RS == 9) {
    // n = 3 n1 + n2, k = k1 + 3 k2
#pragma unroll
    for (int n2 = 0; n2 < 3; n2++) dft3(v[n2], v[3 + n2], v[6 + n2]);
    // v[n2 + 3 k1] *= W9^(n2 k1)
    v[4] = cmul(v[4], make_double2(kC40, -kS40));
    v[5] = cmul(v[5], make_double2(kC80, -kS80));
    v[7] = cmul(v[7], make_double2(kC80, -kS80));
    v[8] = cmul(v[8], make_double2(-kC20, -kS20));
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++) dft3(v[3 * k1], v[3 * k1 + 1], v[3 * k1 + 2]);
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++)
#pragma unroll
      for (int k2 = 0; k2 < 3; k2++) o[k1 + 3 * k2] = v[3 * k1 + k2];
  } else if constexpr (RS == 12) {
    // n = 4 n1 + n2, k = k1 + 3 k2
#pragma unroll
    for (int n2 = 0; n2 < 4; n2++) dft3(v[n2], v[4 + n2], v[8 + n2]);
    // v[n2 + 4 k1] *= W12^(n2 k1)
    v[5] = cmul(v[5], make_double2(kS3, -0.5));
    v[6] = cmul(v[6], make_double2(0.5, -kS3));
    v[7] = cmul_mi(v[7]);
    v[9] = cmul(v[9], make_double2(0.5, -kS3));
    v[10] = cmul(v[10], make_double2(-0.5, -kS3));
    v[11] = make_double2(-v[11].x, -v[11].y);
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++) dft4(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++)
#pragma unroll
      for (int k2 = 0; k2 < 4; k2++) o[k1 + 3 * k2] = v[4 * k1 + k2];
  } else if constexpr (RS == 4) {
    dft4(v[0], v[1], v[2], v[3]);
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = v[r];
  } else if constexpr (RS == 8) {
    // n = 2 n1 + n2, k = k1 + 4 k2
    dft4(v[0], v[2], v[4], v[6]);
    dft4(v[1], v[3], v[5], v[7]);
    v[3] = cmul(v[3], make_double2(kR2, -kR2));
    v[5] = cmul_mi(v[5]);
    v[7] = cmul(v[7], make_double2(-kR2, -kR2));
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) {
      o[k1] = cadd(v[2 * k1], v[2 * k1 + 1]);
      o[k1 + 4] = csub(v[2 * k1], v[2 * k1 + 1]);
    }
  } else {
    static_assert(RS == 16, "radix 2, 4, 8, 9, 12 or 16");
    // n = 4 n1 + n2, k = k1 + 4 k2
#pragma unroll
    for (int n2 = 0; n2 < 4; n2++) dft4(v[n2], v[4 + n2], v[8 + n2], v[12 + n2]);
    // v[n2 + 4 k1] *= W16^(n2 k1)
    v[5] = cmul(v[5], make_double2(kC8, -kS8));
    v[9] = cmul(v[9], make_double2(kR2, -kR2));
    v[13] = cmul(v[13], make_double2(kS8, -kC8));
    v[6] = cmul(v[6], make_double2(kR2, -kR2));
    v[10] = cmul_mi(v[10]);
    v[14] = cmul(v[14], make_double2(-kR2, -kR2));
    v[7] = cmul(v[7], make_double2(kS8, -kC8));
    v[11] = cmul(v[11], make_double2(-kR2, -kR2));
    v[15] = cmul(v[15], make_double2(-kC8, kS8));
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) dft4(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
      for (int k2 = 0; k2 < 4; k2++) o[k1 + 4 * k2] = v[4 * k1 + k2];
  }
}

constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x / 2); }
// radix of the stage that faces `rem` remaining points: a factor of 9 or 3 first,
// then 16 while that leaves a power of 16 or at least 4 behind, then 8, 4 or 2
constexpr int stage_radix(int rem) {
  return rem % 9 == 0                               ? 9
         : rem % 3 == 0                             ? 12
         : (ilog2(rem) >= 4 && ilog2(rem) != 5)     ? 16
         : ilog2(rem) == 5                          ? 8
                                                    : rem;
}

__device__ inline int pad(int i) { return i + (i >> 4); }

// The stages are forced inline: shared by many kernels they would become calls,
// which cost the two passes 5 us of 66 per inner product at N = 2^21.
// One Stockham stage of radix RS on L points held in x (LDS, padded), NT threads.
// MUL (first stage only): the points are read as conj(x f), f in global memory.
template <int L, int NT, int NS, int RS, bool MUL = false>
__device__ __forceinline__ void fft_stage(double2 *x, int t, const double2 *tw, const double2 *f = nullptr) {
  constexpr int NB = L / RS;
  constexpr int PER = (NB + NT - 1) / NT;
  double2 o[PER][RS];
#pragma unroll
  for (int u = 0; u < PER; u++) {
    const int j = t + u * NT;
    if (NB % NT == 0 || j < NB) {
      const int jm = (unsigned)j % NS;
      double2 v[RS];
#pragma unroll
      for (int r = 0; r < RS; r++) v[r] = x[pad(j + r * NB)];
      if constexpr (MUL) {
#pragma unroll
        for (int r = 0; r < RS; r++) {
          const double2 m = cmul(v[r], f[j + r * NB]);
          v[r] = make_double2(m.x, -m.y);
        }
      }
      if constexpr (NS > 1) {
#pragma unroll
        for (int r = 1; r < RS; r++) v[r] = cmul(v[r], tw[r * jm * (L / (RS * NS))]);
      }
      dft<RS>(v, o[u]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; u++) {
    const int j = t + u * NT;
    if (NB % NT == 0 || j < NB) {
      const int d = (unsigned)j / NS * NS * RS + (unsigned)j % NS;
#pragma unroll
      for (int r = 0; r < RS; r++) x[pad(d + r * NS)] = o[u][r];
    }
  }
  __syncthreads();
}

template <int L, int NT, int NS>
__device__ __forceinline__ void fft_stages(double2 *x, int t, const double2 *tw) {
  if constexpr (NS < L) {
    constexpr int RS = stage_radix(L / NS);
    fft_stage<L, NT, NS, RS>(x, t, tw);
    fft_stages<L, NT, NS * RS>(x, t, tw);
  }
}

// Whole L-point FFT of conj(x f).
template <int L, int NT>
__device__ __forceinline__ void fft_conj_product(double2 *x, int t, const double2 *tw, const double2 *f) {
  constexpr int RS = stage_radix(L);
  fft_stage<L, NT, 1, RS, true>(x, t, tw, f);
  fft_stages<L, NT, RS>(x, t, tw);
}

// The points of a thread's first-stage butterflies, straight from global memory
// (a caller requests them before what it needs only after the FFT: loads return
// in order; at N = 2^18 the second pass takes 12.0 us so, 15.4 with them last):
// butterfly j reads src[j + r L / RS], contiguous across the threads for each r.
template <int L, int NT>
struct FirstPoints {
  static constexpr int RS = stage_radix(L), NB = L / RS, PER = (NB + NT - 1) / NT;
  double2 v[PER][RS];
  __device__ __forceinline__ void load(const double2 *src, int t) {
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int j = t + u * NT;
      if (NB % NT == 0 || j < NB) {
#pragma unroll
        for (int r = 0; r < RS; r++) v[u][r] = src[j + r * NB];
      }
    }
  }
};

// Whole L-point FFT from the points of the first stage (no twiddles).
template <int L, int NT>
__device__ __forceinline__ void fft_first(FirstPoints<L, NT> &p, double2 *x, int t, const double2 *tw) {
  constexpr int RS = FirstPoints<L, NT>::RS, NB = FirstPoints<L, NT>::NB;
#pragma unroll
  for (int u = 0; u < FirstPoints<L, NT>::PER; u++) {
    const int j = t + u * NT;
    if (NB % NT == 0 || j < NB) {
      double2 o[RS];
      dft<RS>(p.v[u], o);
#pragma unroll
      for (int r = 0; r < RS; r++) x[pad(j * RS + r)] = o[r];
    }
  }
  __syncthreads();
  fft_stages<L, NT, RS>(x, t, tw);
}

template <int L, int NT>
__device__ __forceinline__ void fft_first_global(const double2 *src, double2 *x, int t, const double2 *tw) {
  FirstPoints<L, NT> p;
  p.load(src, t);
  fft_first<L, NT>(p, x, t, tw);
}

__device__ inline double2 tw2(const double2 *hi, const double2 *lo, long long e) {
  return cmul(hi[e >> 10], lo[e & 1023]);
}

// ---------------------------------------------------------------- pass 1
// columns per workgroup: 8 (one 128-byte line per row) up to 512-point
// columns, 4 beyond (two workgroups per CU at 1024 points); the workgroups
// of the two halves of a line are placed on one XCD (col_group)
template <int LR>
constexpr int col_cols() { return LR <= 512 ? 8 : 4; }
// LDS stride of a column: padded length, plus one so the columns of a row
// start on different banks
template <int LR>
constexpr int col_stride() { return LR + LR / 16 + 1; }
// threads per column or row: one butterfly each in the first stage (16, 12 or 9
// points), in whole waves
template <int L>
constexpr int fft_threads() { return L <= 1024 ? 64 : L % 3 == 0 ? L / stage_radix(L) : L / 16; }

// Channel and column group of a workgroup.  Workgroups are dealt round-robin to
// the 8 XCDs in launch order; groups 2q and 2q + 1 of half a 128-byte line
// per row are paired on one XCD, launched 8 apart, so each line is fetched
// into one L2 once.
template <int CC>
__device__ inline void col_group(int &ch, int &grp) {
  ch = blockIdx.y;
  grp = blockIdx.x;
  if (CC < 8) {
    const int L = blockIdx.y * gridDim.x + blockIdx.x, total = gridDim.x * gridDim.y;
    if ((total & 15) == 0) {
      const int xcd = L & 7, r = L >> 3;
      const int g = ((((r >> 1) << 3) | xcd) << 1) | (r & 1);
      ch = g / gridDim.x;
      grp = g % gridDim.x;
    }
  }
}

template <int LR>
__global__ __launch_bounds__(col_cols<LR>() * fft_threads<LR>()) void k_fft_cols(FftArgs F, const double *h0,
                                                                                  const double *h1, double2 *Y) {
  constexpr int CC = col_cols<LR>(), CS = col_stride<LR>(), NT = fft_threads<LR>();
  __shared__ double2 s[CC * CS];
  int ch, grp;
  col_group<CC>(ch, grp);
  const int b0 = grp * CC, tid = threadIdx.x;
  constexpr int PT = (LR + NT - 1) / NT;  // elements per thread in the staging loops
  constexpr bool kFull = LR % NT == 0;
  const double2 *z = reinterpret_cast<const double2 *>(ch ? h1 : h0);
  {
    // every load in flight before the first LDS store
    double2 v[PT];
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      if (kFull || idx < CC * LR) v[q] = z[(size_t)(idx / CC) * F.C + b0 + idx % CC];
    }
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      if (kFull || idx < CC * LR) s[(idx % CC) * CS + pad(idx / CC)] = v[q];
    }
  }
  __syncthreads();
  fft_stages<LR, NT, 1>(s + (tid / NT) * CS, tid % NT, F.twR);
  double2 *Yc = Y + (size_t)ch * F.M;
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const int idx = tid + q * CC * NT;
    const int k1 = idx / CC, c = idx % CC, b = b0 + c;
    if (kFull || idx < CC * LR)
      Yc[(size_t)k1 * F.C + b] = cmul(s[c * CS + pad(k1)], tw2(F.twMhi, F.twMlo, (long long)b * k1));
  }
}

// ---------------------------------------------------------------- pass 2
// One workgroup per row pair, half of it per row: block 0 takes rows 0 and R/2
// (each its own mirror), block p > 0 rows p and R - p.
constexpr int kFinalLanes = 256;       // lanes of the final reduction's order
constexpr int kFinalSpinCap = 1 << 20;  // polls of one missing pair before it reads as NaN

constexpr int kFinalMaxPer = 8;         // pairs per lane: F.R <= 2048

__device__ inline long long final_peek(const double *p) {
  return __hip_atomic_load(reinterpret_cast<const long long *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The value of a published word, first read as v (polled again while it still
// reads kFinalEmpty); the word is returned to kFinalEmpty.
__device__ inline double final_take(double *p, long long v) {
  long long *w = reinterpret_cast<long long *>(p);
  int spins = 0;
  while (v == kFinalEmpty) {
    if (++spins > kFinalSpinCap) {
      v = 0x7FF8000000000000LL;
      break;
    }
    __builtin_amdgcn_s_sleep(1);
    v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __hip_atomic_store(w, kFinalEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __longlong_as_double(v);
}

__device__ inline void final_put(double *p, double x) {
  __hip_atomic_store(reinterpret_cast<long long *>(p), __double_as_longlong(x), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_fft_final_reset(double *partials, int nwords) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += gridDim.x * blockDim.x)
    reinterpret_cast<long long *>(partials)[i] = kFinalEmpty;
}

// The final reduction, run by one workgroup of BS threads with LDS scratch
// sd (2 kFinalLanes doubles): collects the R published pairs and sums them in
// the order of k_dot_final.
template <int BS>
__device__ void final_collect(int R, double *partials, const FftFinal &fin, double *sd) {
  const int tid = threadIdx.x;
  double *sh = sd + kFinalLanes;
  // every word of the thread's lanes is requested before the first is used
  constexpr int kVL = (kFinalLanes + BS - 1) / BS;  // lanes per thread
  long long w[kVL][2 * kFinalMaxPer];
#pragma unroll
  for (int v = 0; v < kVL; v++)
#pragma unroll
    for (int k = 0; k < kFinalMaxPer; k++) {
      const int q = tid + v * BS + k * kFinalLanes;
      if (tid + v * BS < kFinalLanes && q < R) {
        w[v][2 * k] = final_peek(partials + 2 * q);
        w[v][2 * k + 1] = final_peek(partials + 2 * q + 1);
      }
    }
#pragma unroll
  for (int v = 0; v < kVL; v++) {
    const int t = tid + v * BS;
    if (t >= kFinalLanes) break;
    double pd = 0.0, ph = 0.0;
#pragma unroll
    for (int k = 0; k < kFinalMaxPer; k++) {
      const int q = t + k * kFinalLanes;
      if (q < R) {
        pd += final_take(partials + 2 * q, w[v][2 * k]);
        ph += final_take(partials + 2 * q + 1, w[v][2 * k + 1]);
      }
    }
    sd[t] = pd;
    sh[t] = ph;
  }
  __syncthreads();
  for (int o = kFinalLanes / 2; o > 0; o >>= 1) {
    for (int t = tid; t < o; t += BS) {
      sd[t] += sd[t + o];
      sh[t] += sh[t + o];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const bool bad = fin.flags && fin.flags[3] != 0;
    fin.out[0] = bad ? __builtin_nan("") : 4.0 * sd[0];
    fin.out[1] = bad ? __builtin_nan("") : 4.0 * sh[0];
  }
  __syncthreads();
  if (fin.clear && tid < 8) fin.clear[tid] = 0;
}

template <int LC, bool FINAL>
__global__ __launch_bounds__(2 * fft_threads<LC>()) void k_fft_rows(FftArgs F, const double2 *Y, double *partials,
                                                                    double2 *hw_out, FftFinal fin) {
  constexpr int RSD = LC + LC / 16, NT = fft_threads<LC>();
  __shared__ double2 s[2 * RSD];
  __shared__ double s_red[2 * NT / 64][2];
  const int ch = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x;
  if (FINAL && blk == F.R / 2) {
    // the extra column of workgroups: (R/2, 1), dispatched after every row
    // workgroup, collects their pairs, so each pair it waits for is on its
    // way; (R/2, 0) has nothing to do.  LDS of the FFT serves as scratch where
    // it is large enough.
    constexpr bool kReuse = 4 * RSD >= 2 * kFinalLanes;
    __shared__ double s_fin[kReuse ? 1 : 2 * kFinalLanes];
    if (ch == 1) final_collect<2 * NT>(F.R, partials, fin, kReuse ? reinterpret_cast<double *>(s) : s_fin);
    return;
  }
  const int half = tid / NT;
  const int A = blk, B = blk == 0 ? F.R / 2 : F.R - blk;
  const double2 *Yc = Y + (size_t)ch * F.M;
  const double2 *Dp = F.Dp[ch];
  const double *wp = F.wp[ch];
  // the FFT's points, then this thread's weighted data and weights, whose
  // latency hides behind the FFT (loads return in order, so the points come
  // first); k2 = tid + q 2NT in rows A and B
  FirstPoints<LC, NT> points;
  points.load(Yc + (size_t)(half ? B : A) * F.C, tid % NT);
  constexpr int KP = (LC + 2 * NT - 1) / (2 * NT);
  constexpr bool kFull = LC % (2 * NT) == 0;
  double2 dA[KP], dB[KP];
  double wA[KP], wB[KP];
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k2 = min(tid + q * 2 * NT, LC - 1);
    dA[q] = Dp[A * LC + k2];
    wA[q] = wp[A * LC + k2];
    dB[q] = Dp[B * LC + k2];
    wB[q] = wp[B * LC + k2];
  }
  fft_first<LC, NT>(points, s + half * RSD, tid % NT, F.twC);
  const double2 *sA = s, *sB = s + RSD;
  double2 *hw = hw_out ? hw_out + (size_t)ch * (F.M + 1) : nullptr;
  double dh = 0.0, hh = 0.0;
  // W_N^(row + R k2) = W_N^row W_N^(R k2)
  const double2 WrA = tw2(F.twNhi, F.twNlo, A), WrB = tw2(F.twNhi, F.twNlo, B);
  // H_k from Z_k and conj(Z_(M-k)), k = row + R k2, weighted and summed
  auto emit = [&](long long k, double2 W, double2 zk, double2 zm, double2 d, double w) {
    const double2 zmc = make_double2(zm.x, -zm.y);
    const double2 E = make_double2(0.5 * (zk.x + zmc.x), 0.5 * (zk.y + zmc.y));
    const double2 dz = make_double2(zk.x - zmc.x, zk.y - zmc.y);
    const double2 O = make_double2(0.5 * dz.y, -0.5 * dz.x);
    const double2 WO = cmul(W, O);
    const double2 x = make_double2((E.x + WO.x) * w, (E.y + WO.y) * w);
    dh += x.x * d.x + x.y * d.y;
    hh += x.x * x.x + x.y * x.y;
    if (hw) hw[k] = x;
  };
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k2 = tid + q * 2 * NT;
    if (kFull || k2 < LC) {
      const double2 t = F.twNr[k2];
      const long long kA = A + (long long)F.R * k2, kB = B + (long long)F.R * k2;
      if (blk == 0) {
        // row 0 (Z_(M-k) in row 0 itself) and row R/2 (its own mirror)
        if (k2 == 0) {
          // H_0 = E_0 + O_0 and H_M = E_0 - O_0, both real
          const double2 z0 = sA[0];
          const double wm = wp[F.M];
          const double2 dm = Dp[F.M];
          const double2 x0 = make_double2((z0.x + z0.y) * wA[q], 0.0), xm = make_double2((z0.x - z0.y) * wm, 0.0);
          dh += x0.x * dA[q].x + x0.y * dA[q].y + xm.x * dm.x + xm.y * dm.y;
          hh += x0.x * x0.x + xm.x * xm.x;
          if (hw) {
            hw[0] = x0;
            hw[F.M] = xm;
          }
        } else {
          emit(kA, t, sA[pad(k2)], sA[pad(LC - k2)], dA[q], wA[q]);
        }
        emit(kB, cmul(WrB, t), sB[pad(k2)], sB[pad(LC - 1 - k2)], dB[q], wB[q]);
      } else {
        emit(kA, cmul(WrA, t), sA[pad(k2)], sB[pad(LC - 1 - k2)], dA[q], wA[q]);
        emit(kB, cmul(WrB, t), sB[pad(k2)], sA[pad(LC - 1 - k2)], dB[q], wB[q]);
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    dh += __shfl_xor(dh, o, 64);
    hh += __shfl_xor(hh, o, 64);
  }
  if ((tid & 63) == 0) {
    s_red[tid >> 6][0] = dh;
    s_red[tid >> 6][1] = hh;
  }
  __syncthreads();
  if (tid == 0) {
    double a = 0.0, b = 0.0;
    for (int w = 0; w < 2 * NT / 64; w++) {
      a += s_red[w][0];
      b += s_red[w][1];
    }
    const int q = ch * (F.R / 2) + blk;
    if (FINAL) {
      final_put(partials + 2 * q, a);
      final_put(partials + 2 * q + 1, b);
    } else {
      partials[2 * q] = a;
      partials[2 * q + 1] = b;
    }
  }
}

// ------------------------------------------- data and weights in bin order
// H_k from Z_k and Z_(M-k) (E + W O, W = W_N^k), weighted, and its two sums.
__device__ __forceinline__ void add_bin(double2 W, double2 zk, double2 zm, double2 d, double w, double &dh,
                                        double &hh) {
  const double2 E = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
  const double2 O = make_double2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
  const double2 WO = cmul(W, O);
  const double2 x = make_double2((E.x + WO.x) * w, (E.y + WO.y) * w);
  dh += x.x * d.x + x.y * d.y;
  hh += x.x * x.x + x.y * x.y;
}
// Bins 0 and M, both real: H_0 = E_0 + O_0, H_M = E_0 - O_0.  The products with
// the zero imaginary parts stay: they pass on data that are not finite.
__device__ __forceinline__ void add_ends(double2 z0, double2 d0, double w0, double2 dm, double wm, double &dh,
                                         double &hh) {
  const double x0 = (z0.x + z0.y) * w0, xm = (z0.x - z0.y) * wm;
  dh += x0 * d0.x + 0.0 * d0.y + xm * dm.x + 0.0 * dm.y;
  hh += x0 * x0 + xm * xm;
}

// The workgroup's sums; valid in thread 0.
template <int THREADS>
__device__ __forceinline__ void block_sums(double &dh, double &hh) {
  __shared__ double s_red[THREADS / 64][2];
  for (int o = 32; o > 0; o >>= 1) {
    dh += __shfl_xor(dh, o, 64);
    hh += __shfl_xor(hh, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s_red[threadIdx.x >> 6][0] = dh;
    s_red[threadIdx.x >> 6][1] = hh;
  }
  __syncthreads();
  dh = hh = 0.0;
  for (int w = 0; w < THREADS / 64; w++) {
    dh += s_red[w][0];
    hh += s_red[w][1];
  }
}

// Pass 2 for data and weights that a caller holds in bin order, k = k1 + R k2:
// four neighbouring row pairs per workgroup, so that a step in k2 reads 64
// bytes of data and 32 of weights per row group; the two workgroups that share
// a 128-byte line run on one XCD.  Reading them so costs less than bringing
// them into the row order first: 32 us at N = 2^21 where the row-ordered pass
// takes 21 and the two transposes before it took 24.
constexpr int kNatRows = 4;
template <int LC>
__global__ __launch_bounds__(2 * kNatRows * fft_threads<LC>()) void k_fft_rows_natural(FftArgs F, const double2 *Y,
                                                                                       double *partials) {
  constexpr int G = kNatRows, NT = fft_threads<LC>(), BS = 2 * G * NT, RSD = LC + LC / 16 + 1;
  __shared__ double2 s[2 * G * RSD];
  int ch, grp;
  col_group<G>(ch, grp);
  const int tid = threadIdx.x, r = tid % G, blk = grp * G + r;
  const int A = blk, B = blk == 0 ? F.R / 2 : F.R - blk;
  const double2 *Dp = F.Dp[ch];
  const double *wp = F.wp[ch];
  // the row of the wave's FFT (A rows first, then B rows), requested before the
  // data: loads return in order, and the FFT waits for its points only
  const int row = tid / NT, rb = grp * G + row % G;
  const int k1 = row < G ? rb : (rb == 0 ? F.R / 2 : F.R - rb);
  FirstPoints<LC, NT> points;
  points.load(Y + (size_t)ch * F.M + (size_t)k1 * F.C, tid % NT);
  // this thread's data and weights: rows A and B at k2 = (tid + q BS) / G
  constexpr int KP = (G * LC + BS - 1) / BS;
  constexpr bool kFull = G * LC % BS == 0;
  double2 dA[KP], dB[KP];
  double wA[KP], wB[KP];
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k2 = min((tid + q * BS) / G, LC - 1);
    dA[q] = Dp[A + F.R * k2];
    wA[q] = wp[A + F.R * k2];
    dB[q] = Dp[B + F.R * k2];
    wB[q] = wp[B + F.R * k2];
  }
  fft_first<LC, NT>(points, s + row * RSD, tid % NT, F.twC);
  const double2 *sA = s + r * RSD, *sB = s + (G + r) * RSD;
  const double2 WrA = tw2(F.twNhi, F.twNlo, A), WrB = tw2(F.twNhi, F.twNlo, B);
  double dh = 0.0, hh = 0.0;
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k2 = (tid + q * BS) / G;
    if (kFull || k2 < LC) {
      const double2 t = F.twNr[k2];
      if (blk == 0) {
        if (k2 == 0) add_ends(sA[0], dA[q], wA[q], Dp[F.M], wp[F.M], dh, hh);
        else add_bin(t, sA[pad(k2)], sA[pad(LC - k2)], dA[q], wA[q], dh, hh);
        add_bin(cmul(WrB, t), sB[pad(k2)], sB[pad(LC - 1 - k2)], dB[q], wB[q], dh, hh);
      } else {
        add_bin(cmul(WrA, t), sA[pad(k2)], sB[pad(LC - 1 - k2)], dA[q], wA[q], dh, hh);
        add_bin(cmul(WrB, t), sB[pad(k2)], sA[pad(LC - 1 - k2)], dB[q], wB[q], dh, hh);
      }
    }
  }
  block_sums<BS>(dh, hh);
  if (tid == 0) {
    const int q = ch * (F.R / (2 * G)) + grp;
    partials[2 * q] = dh;
    partials[2 * q + 1] = hh;
  }
}

// Short series (M <= 4096): the whole inner product in one workgroup and one
// launch, half of the threads per channel (R = 1, C = M; data and weights in
// bin order).  Bound by latency: 9 us at N = 4096 (10 with the launch), where
// five launches of the general form took 22.
template <int M>
__global__ __launch_bounds__(2 * fft_threads<M>()) void k_fft_small(FftArgs F, const double *h0, const double *h1,
                                                                    double *out) {
  constexpr int NT = fft_threads<M>(), RSD = M + M / 16, KP = (M / 2 + NT - 1) / NT;
  __shared__ double2 s[2 * RSD];
  const int ch = threadIdx.x / NT, t = threadIdx.x % NT;
  const double2 *Dp = F.Dp[ch];
  const double *wp = F.wp[ch];
  FirstPoints<M, NT> points;
  points.load(reinterpret_cast<const double2 *>(ch ? h1 : h0), t);
  // bins k and M - k of this thread, k = t + q NT < M / 2
  double2 dk[KP], dm[KP];
  double wk[KP], wm[KP];
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k = min(t + q * NT, M / 2 - 1);
    dk[q] = Dp[k];
    wk[q] = wp[k];
    dm[q] = Dp[M - k];
    wm[q] = wp[M - k];
  }
  const double2 dc = Dp[M / 2];
  const double wc = wp[M / 2];
  double2 *x = s + ch * RSD;
  fft_first<M, NT>(points, x, t, F.twC);
  double dh = 0.0, hh = 0.0;
#pragma unroll
  for (int q = 0; q < KP; q++) {
    const int k = t + q * NT;
    if (k < M / 2) {
      if (k == 0) {
        add_ends(x[0], dk[q], wk[q], dm[q], wm[q], dh, hh);
        add_bin(tw2(F.twNhi, F.twNlo, M / 2), x[pad(M / 2)], x[pad(M / 2)], dc, wc, dh, hh);
      } else {
        const double2 zk = x[pad(k)], zm = x[pad(M - k)];
        add_bin(tw2(F.twNhi, F.twNlo, k), zk, zm, dk[q], wk[q], dh, hh);
        add_bin(tw2(F.twNhi, F.twNlo, M - k), zm, zk, dm[q], wm[q], dh, hh);
      }
    }
  }
  block_sums<2 * NT>(dh, hh);
  if (threadIdx.x == 0) {
    out[0] = 4.0 * dh;
    out[1] = 4.0 * hh;
  }
}

// ---------------------------------------------------------------- other lengths
// The M-point transform of a length N = 2M that the passes above do not take,
// as Bluestein's convolution (L. Bluestein, 1970): with c_m = exp(-i pi m^2 / M),
//   Z_k = c_k sum_m (z_m c_m) conj(c_(k-m)),
// a cyclic convolution of length L >= 2M - 1 with a fixed filter, whose
// transform F is formed once per handle.  L = R C with R from 2^a, C from 2^a,
// 3 2^a and 9 2^a, at most half longer than it must be from N = 514 on and a
// third from 1538 on.
// Both transforms of the convolution run in the four-step form above, and what
// lies between them stays in LDS:
//   k_chirp_cols   columns b of z_m c_m (zero from M on), times W_L^(b k1);
//   k_chirp_rows   rows k1: forward FFT, times F, inverse FFT, times
//                  W_L^(-b k1), in place;
//   k_chirp_back   columns b back to m = a C + b < M, times c_m;
//   k_chirp_dot    the real spectrum from Z_k and Z_(M-k), weighting, both sums.
// Inverse transforms are conjugated forward ones; F carries their 1/L.
// At N = 2103840 (1024 x 2304) the four kernels move 0.48 GB and take 53 + 69 +
// 40 + 14 us, 196 us per likelihood with the final sum, where the library's
// transform took 781 us in twelve kernels.  Factors 9 and 12 as one stage each
// and one row per workgroup (four of 256 threads per CU share the LDS) matter
// most to the rows: 111 us with radices 16, 16, 3, 3 and two rows per workgroup.
// A 1536 x 1536 split took 84 + 91 + 76 us: 104 KB of LDS for 4 columns leaves
// one workgroup per CU.  Against 80-bit transforms the spectrum's error is
// 6e-16 (relative L2), the library's 1.1e-15.
__device__ inline double2 conjd(double2 a) { return make_double2(a.x, -a.y); }

__global__ void k_chirp_table(double2 *c, int M) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  // m^2 mod 2M in integers: the angle is exact before its one rounding
  const long long q = ((long long)m * m) % (2LL * M);
  double sn, cs;
  sincospi((double)q / (double)M, &sn, &cs);
  c[m] = make_double2(cs, -sn);
}

// FILTER: the columns of the filter conj(c_|m|) instead of a channel.
template <int LR, bool FILTER>
__global__ __launch_bounds__(col_cols<LR>() * fft_threads<LR>()) void k_chirp_cols(ChirpArgs F, const double *h0,
                                                                                   const double *h1, double2 *Y) {
  constexpr int CC = col_cols<LR>(), CS = col_stride<LR>(), NT = fft_threads<LR>();
  __shared__ double2 s[CC * CS];
  int ch, grp;
  col_group<CC>(ch, grp);
  const int b0 = grp * CC, tid = threadIdx.x;
  constexpr int PT = (LR + NT - 1) / NT;
  const double2 *z = reinterpret_cast<const double2 *>(ch ? h1 : h0);
  {
    double2 v[PT], c[PT];
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      const int m = (idx / CC) * F.C + b0 + idx % CC;
      v[q] = c[q] = make_double2(0.0, 0.0);
      if (idx < CC * LR) {
        if (FILTER) {
          const int j = m < F.M ? m : F.L - m;
          if (j < F.M) c[q] = F.chirp[j];
        } else if (m < F.M) {
          v[q] = z[m];
          c[q] = F.chirp[m];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      if (idx < CC * LR) s[(idx % CC) * CS + pad(idx / CC)] = FILTER ? conjd(c[q]) : cmul(v[q], c[q]);
    }
  }
  __syncthreads();
  fft_stages<LR, NT, 1>(s + (tid / NT) * CS, tid % NT, F.twR);
  double2 *Yc = Y + (size_t)ch * F.L;
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const int idx = tid + q * CC * NT;
    const int k1 = idx / CC, c = idx % CC, b = b0 + c;
    if (idx < CC * LR)
      Yc[(size_t)k1 * F.C + b] = cmul(s[c * CS + pad(k1)], tw2(F.twLhi, F.twLlo, (long long)b * k1));
  }
}

// One row per workgroup.  FILTER: the filter's transform (with the 1/L) goes to
// Fo in the order of the rows.
template <int LC, bool FILTER>
__global__ __launch_bounds__(fft_threads<LC>()) void k_chirp_rows(ChirpArgs F, double2 *Y, double2 *Fo) {
  constexpr int NT = fft_threads<LC>(), PT = (LC + NT - 1) / NT;
  __shared__ double2 x[LC + LC / 16];
  const int ch = blockIdx.y, t = threadIdx.x, k1 = blockIdx.x;
  double2 *row = Y + (size_t)ch * F.L + (size_t)k1 * F.C;
  fft_first_global<LC, NT>(row, x, t, F.twC);
  const size_t f0 = (size_t)k1 * F.C;
  if (FILTER) {
    const double inv = 1.0 / (double)F.L;
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int k2 = t + q * NT;
      if (k2 < LC) Fo[f0 + k2] = make_double2(x[pad(k2)].x * inv, x[pad(k2)].y * inv);
    }
    return;
  }
  fft_conj_product<LC, NT>(x, t, F.twC, F.filter + f0);
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const int b = t + q * NT;
    if (b < LC) row[b] = conjd(cmul(x[pad(b)], tw2(F.twLhi, F.twLlo, (long long)b * k1)));
  }
}

template <int LR>
__global__ __launch_bounds__(col_cols<LR>() * fft_threads<LR>()) void k_chirp_back(ChirpArgs F, const double2 *Y,
                                                                                   double2 *Z) {
  constexpr int CC = col_cols<LR>(), CS = col_stride<LR>(), NT = fft_threads<LR>();
  __shared__ double2 s[CC * CS];
  int ch, grp;
  col_group<CC>(ch, grp);
  const int b0 = grp * CC, tid = threadIdx.x;
  constexpr int PT = (LR + NT - 1) / NT;
  const double2 *Yc = Y + (size_t)ch * F.L;
  double2 *Zc = Z + (size_t)ch * F.M;
  {
    double2 v[PT];
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      v[q] = make_double2(0.0, 0.0);
      if (idx < CC * LR) v[q] = Yc[(size_t)(idx / CC) * F.C + b0 + idx % CC];
    }
#pragma unroll
    for (int q = 0; q < PT; q++) {
      const int idx = tid + q * CC * NT;
      if (idx < CC * LR) s[(idx % CC) * CS + pad(idx / CC)] = conjd(v[q]);
    }
  }
  __syncthreads();
  fft_stages<LR, NT, 1>(s + (tid / NT) * CS, tid % NT, F.twR);
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const int idx = tid + q * CC * NT;
    const int m = (idx / CC) * F.C + b0 + idx % CC;
    if (idx < CC * LR && m < F.M) Zc[m] = cmul(conjd(s[(idx % CC) * CS + pad(idx / CC)]), F.chirp[m]);
  }
}

// H_k and H_(M-k) of one pair (k <= M/2) from Z_k and Z_(M-k), weighted and
// summed over both channels.
constexpr int kPairThreads = 256, kPairBlocks = 1024;
__global__ __launch_bounds__(kPairThreads) void k_chirp_dot(ChirpArgs F, const double2 *Z, const double2 *data,
                                                            const double *w, double2 *hw_out, double *partials) {
  __shared__ double s_red[kPairThreads / 64][2];
  const int M = F.M, nb = M + 1, half = M / 2 + 1, tid = threadIdx.x;
  double dh = 0.0, hh = 0.0;
  for (int q = blockIdx.x * kPairThreads + tid; q < 2 * half; q += gridDim.x * kPairThreads) {
    const int ch = q >= half, k = q - ch * half, j = M - k;
    const double2 *Zc = Z + (size_t)ch * M;
    const double2 *dc = data + (size_t)ch * nb;
    const double *wc = w + (size_t)ch * nb;
    double2 *hc = hw_out ? hw_out + (size_t)ch * nb : nullptr;
    const double2 zk = Zc[k], zm = k == 0 ? zk : Zc[j];
    const double2 dk = dc[k], dj = dc[j];
    const double wk = wc[k], wj = wc[j];
    const double2 E = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
    const double2 O = make_double2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
    const double2 WO = cmul(tw2(F.twNhi, F.twNlo, k), O);
    // H_k = E + W O, H_(M-k) = conj(E - W O)
    const double2 a = make_double2((E.x + WO.x) * wk, (E.y + WO.y) * wk);
    const double2 b = make_double2((E.x - WO.x) * wj, -(E.y - WO.y) * wj);
    dh += a.x * dk.x + a.y * dk.y;
    hh += a.x * a.x + a.y * a.y;
    if (hc) hc[k] = a;
    if (j != k) {
      dh += b.x * dj.x + b.y * dj.y;
      hh += b.x * b.x + b.y * b.y;
      if (hc) hc[j] = b;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    dh += __shfl_xor(dh, o, 64);
    hh += __shfl_xor(hh, o, 64);
  }
  if ((tid & 63) == 0) {
    s_red[tid >> 6][0] = dh;
    s_red[tid >> 6][1] = hh;
  }
  __syncthreads();
  if (tid == 0) {
    for (int v = 1; v < kPairThreads / 64; v++) {
      dh += s_red[v][0];
      hh += s_red[v][1];
    }
    partials[2 * blockIdx.x] = dh;
    partials[2 * blockIdx.x + 1] = hh;
  }
}

// ---------------------------------------------------------------- launch
template <int LR>
static void launch_cols(const FftArgs &F, const double *h0, const double *h1, double2 *Y, hipStream_t s) {
  hipLaunchKernelGGL(k_fft_cols<LR>, dim3(F.C / col_cols<LR>(), 2), dim3(col_cols<LR>() * fft_threads<LR>()), 0, s, F,
                     h0, h1, Y);
}

template <int LC>
static void launch_rows(const FftArgs &F, const double2 *Y, double *partials, double2 *hw, const FftFinal *fin,
                        hipStream_t s) {
  if (fin)
    hipLaunchKernelGGL((k_fft_rows<LC, true>), dim3(F.R / 2 + 1, 2), dim3(2 * fft_threads<LC>()), 0, s, F, Y,
                       partials, nullptr, *fin);
  else
    hipLaunchKernelGGL((k_fft_rows<LC, false>), dim3(F.R / 2, 2), dim3(2 * fft_threads<LC>()), 0, s, F, Y, partials,
                       hw, FftFinal{});
}

bool fft_supported(int N, int *R, int *C) {
  if (N < 256 || (N & (N - 1))) return false;
  int m = 0;
  while ((1 << m) < N / 2) m++;
  if (m < 7 || m > 22) return false;
  *R = 1 << ((m + 1) / 2);
  *C = (N / 2) / *R;
  return true;
}

int fft_partials(const FftArgs &F) { return F.R; }

// Table layout: W_R | W_C | W_M lo | W_M hi | W_N lo | W_N hi | W_N^(R k2).
static void table_offsets(const FftArgs &F, size_t o[8]) {
  const size_t nhi = (size_t)F.M / 1024 + 2;
  o[0] = 0;
  o[1] = o[0] + F.R;
  o[2] = o[1] + F.C;
  o[3] = o[2] + 1024;
  o[4] = o[3] + nhi;
  o[5] = o[4] + 1024;
  o[6] = o[5] + nhi;
  o[7] = o[6] + F.C;
}

size_t fft_table_size(const FftArgs &F) {
  size_t o[8];
  table_offsets(F, o);
  return o[7];
}

void fft_fill_tables(const FftArgs &F, double2 *tw) {
  // W_L^e = exp(-2 pi i e / L), computed in extended precision
  auto root = [](long long e, long long L) {
    const long double pi = 3.141592653589793238462643383279502884L;
    const long double a = -2.0L * pi * (long double)(e % L) / (long double)L;
    return make_double2((double)cosl(a), (double)sinl(a));
  };
  size_t o[8];
  table_offsets(F, o);
  const int nhi = (int)(o[4] - o[3]);
  for (int e = 0; e < F.R; e++) tw[o[0] + e] = root(e, F.R);
  for (int e = 0; e < F.C; e++) tw[o[1] + e] = root(e, F.C);
  for (int e = 0; e < 1024; e++) {
    tw[o[2] + e] = root(e, F.M);
    tw[o[4] + e] = root(e, F.N);
  }
  for (int e = 0; e < nhi; e++) {
    tw[o[3] + e] = root(1024LL * e, F.M);
    tw[o[5] + e] = root(1024LL * e, F.N);
  }
  for (int e = 0; e < F.C; e++) tw[o[6] + e] = root((long long)F.R * e, F.N);
}

void fft_bind_tables(FftArgs *F, const double2 *tw) {
  size_t o[8];
  table_offsets(*F, o);
  F->twR = tw + o[0];
  F->twC = tw + o[1];
  F->twMlo = tw + o[2];
  F->twMhi = tw + o[3];
  F->twNlo = tw + o[4];
  F->twNhi = tw + o[5];
  F->twNr = tw + o[6];
}

void launch_fft_pass1(const FftArgs &F, const double *h0, const double *h1, double2 *Y, hipStream_t s) {
  switch (F.R) {
    case 16: launch_cols<16>(F, h0, h1, Y, s); break;
    case 32: launch_cols<32>(F, h0, h1, Y, s); break;
    case 64: launch_cols<64>(F, h0, h1, Y, s); break;
    case 128: launch_cols<128>(F, h0, h1, Y, s); break;
    case 256: launch_cols<256>(F, h0, h1, Y, s); break;
    case 512: launch_cols<512>(F, h0, h1, Y, s); break;
    case 1024: launch_cols<1024>(F, h0, h1, Y, s); break;
    default: launch_cols<2048>(F, h0, h1, Y, s); break;
  }
}

static void launch_pass2(const FftArgs &F, const double2 *Y, double *partials, double2 *hw_out, const FftFinal *fin,
                         hipStream_t s) {
  switch (F.C) {
    case 8: launch_rows<8>(F, Y, partials, hw_out, fin, s); break;
    case 16: launch_rows<16>(F, Y, partials, hw_out, fin, s); break;
    case 32: launch_rows<32>(F, Y, partials, hw_out, fin, s); break;
    case 64: launch_rows<64>(F, Y, partials, hw_out, fin, s); break;
    case 128: launch_rows<128>(F, Y, partials, hw_out, fin, s); break;
    case 256: launch_rows<256>(F, Y, partials, hw_out, fin, s); break;
    case 512: launch_rows<512>(F, Y, partials, hw_out, fin, s); break;
    case 1024: launch_rows<1024>(F, Y, partials, hw_out, fin, s); break;
    default: launch_rows<2048>(F, Y, partials, hw_out, fin, s); break;
  }
}

void launch_fft_pass2(const FftArgs &F, const double2 *Y, double *partials, double2 *hw_out, hipStream_t s) {
  launch_pass2(F, Y, partials, hw_out, nullptr, s);
}

void launch_fft_pass2_final(const FftArgs &F, const double2 *Y, double *partials, const FftFinal &fin, hipStream_t s) {
  launch_pass2(F, Y, partials, nullptr, &fin, s);
}

void launch_fft_final_reset(double *partials, int npairs, hipStream_t s) {
  hipLaunchKernelGGL(k_fft_final_reset, dim3(8), dim3(256), 0, s, partials, 2 * npairs);
}

// ------------------------------------------- data and weights in bin order
template <int LC>
static void launch_natural(const FftArgs &F, const double2 *Y, double *partials, hipStream_t s) {
  hipLaunchKernelGGL(k_fft_rows_natural<LC>, dim3(F.R / (2 * kNatRows), 2), dim3(2 * kNatRows * fft_threads<LC>()), 0,
                     s, F, Y, partials);
}

int fft_natural_partials(const FftArgs &F) { return F.R / kNatRows; }

void launch_fft_pass2_natural(const FftArgs &F, const double2 *Y, double *partials, hipStream_t s) {
  switch (F.C) {
    case 64: launch_natural<64>(F, Y, partials, s); break;
    case 128: launch_natural<128>(F, Y, partials, s); break;
    case 256: launch_natural<256>(F, Y, partials, s); break;
    case 512: launch_natural<512>(F, Y, partials, s); break;
    default: launch_natural<1024>(F, Y, partials, s); break;
  }
}

template <int M>
static void launch_small(const FftArgs &F, const double *h0, const double *h1, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_fft_small<M>, dim3(1), dim3(2 * fft_threads<M>()), 0, s, F, h0, h1, out);
}

bool launch_fft_small(const FftArgs &F, const double *h0, const double *h1, double *out, hipStream_t s) {
  switch (F.M) {
    case 128: launch_small<128>(F, h0, h1, out, s); break;
    case 256: launch_small<256>(F, h0, h1, out, s); break;
    case 512: launch_small<512>(F, h0, h1, out, s); break;
    case 1024: launch_small<1024>(F, h0, h1, out, s); break;
    case 2048: launch_small<2048>(F, h0, h1, out, s); break;
    case 4096: launch_small<4096>(F, h0, h1, out, s); break;
    default: return false;
  }
  return true;
}

// ---------------------------------------------------------------- other lengths
// Columns of 2^a points, rows of 2^a, 3 2^a or 9 2^a.
static const int kChirpRows[] = {16,  32,  48,  64,  96,  128, 144,  192,  256, 288,
                                 384, 512, 576, 768, 1024, 1152, 1536, 2048, 2304};

// Lengths whose half is a product of primes up to 17 stay with the library's
// mixed-radix transforms, which need no convolution for them: at N = 2000000 they
// take 106 us against 183 of the convolution, at 250000 39 against 46, at 4000
// 22 against 29; with the factor 17 119 against 198 at N = 2228224, 131 against
// 202 at 2263040, 41 against 53 at 278528, 28 against 32 at 8704.  With a factor
// from 19 on the library runs a convolution too, and this one is faster (N =
// 2490368 = 19 2^17: 242 us against 787, 2103840: 196 against 781, 1048578: 107
// against 384, 65538: 37 against 56, 4002: 29 against 44, 1002: 23 against 30,
// 74: 25 against 27) but for the shortest (38 to 62: 26 against 23).
bool chirp_supported(int N, int *R, int *C) {
  if (N < 64 || (N & 1)) return false;
  int rest = N / 2;
  for (int q : {2, 3, 5, 7, 11, 13, 17})
    while (rest % q == 0) rest /= q;
  if (rest == 1) return false;
  const long long need = (long long)N - 1;  // 2M - 1
  long long best = 0;
  for (int r = 16; r <= 2048; r *= 2)
    for (int c : kChirpRows) {
      // the shortest product; columns no longer than rows leave two workgroups
      // per CU (1024-point columns); only 2048 x 1536 has no such form
      const long long l = (long long)r * c;
      if (l < need || (c < r && c != 1536)) continue;
      if (best == 0 || l < best || (l == best && r > *R)) {
        best = l;
        *R = r;
        *C = c;
      }
    }
  return best != 0;
}

int chirp_partials(const ChirpArgs &F) {
  const int need = (2 * (F.M / 2 + 1) + kPairThreads - 1) / kPairThreads;
  return need < kPairBlocks ? need : kPairBlocks;
}

// Table layout: W_R | W_C | W_L lo | W_L hi | W_N lo | W_N hi, then the chirp
// and the filter's transform, which the device forms.
static void chirp_offsets(const ChirpArgs &F, size_t o[9]) {
  o[0] = 0;
  o[1] = o[0] + F.R;
  o[2] = o[1] + F.C;
  o[3] = o[2] + 1024;
  o[4] = o[3] + (size_t)F.L / 1024 + 2;
  o[5] = o[4] + 1024;
  o[6] = o[5] + (size_t)F.M / 1024 + 2;
  o[7] = o[6] + F.M;
  o[8] = o[7] + F.L;
}

size_t chirp_table_size(const ChirpArgs &F) {
  size_t o[9];
  chirp_offsets(F, o);
  return o[8];
}

size_t chirp_host_tables(const ChirpArgs &F, double2 *tw) {
  size_t o[9];
  chirp_offsets(F, o);
  if (!tw) return o[6];
  auto root = [](long long e, long long L) {
    const long double pi = 3.141592653589793238462643383279502884L;
    const long double a = -2.0L * pi * (long double)(e % L) / (long double)L;
    return make_double2((double)cosl(a), (double)sinl(a));
  };
  for (int e = 0; e < F.R; e++) tw[o[0] + e] = root(e, F.R);
  for (int e = 0; e < F.C; e++) tw[o[1] + e] = root(e, F.C);
  for (int e = 0; e < 1024; e++) {
    tw[o[2] + e] = root(e, F.L);
    tw[o[4] + e] = root(e, F.N);
  }
  for (size_t e = 0; e < o[4] - o[3]; e++) tw[o[3] + e] = root(1024LL * e, F.L);
  for (size_t e = 0; e < o[6] - o[5]; e++) tw[o[5] + e] = root(1024LL * e, F.N);
  return o[6];
}

void chirp_bind_tables(ChirpArgs *F, double2 *tw) {
  size_t o[9];
  chirp_offsets(*F, o);
  F->twR = tw + o[0];
  F->twC = tw + o[1];
  F->twLlo = tw + o[2];
  F->twLhi = tw + o[3];
  F->twNlo = tw + o[4];
  F->twNhi = tw + o[5];
  F->chirp = tw + o[6];
  F->filter = tw + o[7];
}

namespace {
struct ChirpCall {
  const ChirpArgs &F;
  const double *h0, *h1;
  double2 *Y, *Z, *Fo;
  hipStream_t s;
};
template <int S>
void chirp_cols(const ChirpCall &c, bool filter) {
  const dim3 grid(c.F.C / col_cols<S>(), filter ? 1 : 2), block(col_cols<S>() * fft_threads<S>());
  if (filter) hipLaunchKernelGGL((k_chirp_cols<S, true>), grid, block, 0, c.s, c.F, nullptr, nullptr, c.Y);
  else hipLaunchKernelGGL((k_chirp_cols<S, false>), grid, block, 0, c.s, c.F, c.h0, c.h1, c.Y);
}
template <int S>
void chirp_rows(const ChirpCall &c, bool filter) {
  const dim3 grid(c.F.R, filter ? 1 : 2), block(fft_threads<S>());
  if (filter) hipLaunchKernelGGL((k_chirp_rows<S, true>), grid, block, 0, c.s, c.F, c.Y, c.Fo);
  else hipLaunchKernelGGL((k_chirp_rows<S, false>), grid, block, 0, c.s, c.F, c.Y, nullptr);
}
template <int S>
void chirp_back(const ChirpCall &c) {
  hipLaunchKernelGGL(k_chirp_back<S>, dim3(c.F.C / col_cols<S>(), 2), dim3(col_cols<S>() * fft_threads<S>()), 0, c.s,
                     c.F, c.Y, c.Z);
}
#define CHIRP_POW2(fn, ...)                     \
    case 16: fn<16>(__VA_ARGS__); break;        \
    case 32: fn<32>(__VA_ARGS__); break;        \
    case 64: fn<64>(__VA_ARGS__); break;        \
    case 128: fn<128>(__VA_ARGS__); break;      \
    case 256: fn<256>(__VA_ARGS__); break;      \
    case 512: fn<512>(__VA_ARGS__); break;      \
    case 1024: fn<1024>(__VA_ARGS__); break;
void chirp_cols_of(const ChirpCall &c, bool filter) {
  switch (c.F.R) {
    CHIRP_POW2(chirp_cols, c, filter)
    default: chirp_cols<2048>(c, filter); break;
  }
}
void chirp_back_of(const ChirpCall &c) {
  switch (c.F.R) {
    CHIRP_POW2(chirp_back, c)
    default: chirp_back<2048>(c); break;
  }
}
void chirp_rows_of(const ChirpCall &c, bool filter) {
  switch (c.F.C) {
    CHIRP_POW2(chirp_rows, c, filter)
    case 48: chirp_rows<48>(c, filter); break;
    case 96: chirp_rows<96>(c, filter); break;
    case 144: chirp_rows<144>(c, filter); break;
    case 192: chirp_rows<192>(c, filter); break;
    case 288: chirp_rows<288>(c, filter); break;
    case 384: chirp_rows<384>(c, filter); break;
    case 576: chirp_rows<576>(c, filter); break;
    case 768: chirp_rows<768>(c, filter); break;
    case 1152: chirp_rows<1152>(c, filter); break;
    case 1536: chirp_rows<1536>(c, filter); break;
    case 2304: chirp_rows<2304>(c, filter); break;
    default: chirp_rows<2048>(c, filter); break;
  }
}
#undef CHIRP_POW2
}  // namespace

void launch_chirp_init(const ChirpArgs &F, double2 *tw, double2 *Y, hipStream_t s) {
  size_t o[9];
  chirp_offsets(F, o);
  hipLaunchKernelGGL(k_chirp_table, dim3((F.M + 255) / 256), dim3(256), 0, s, tw + o[6], F.M);
  const ChirpCall c = {F, nullptr, nullptr, Y, nullptr, tw + o[7], s};
  chirp_cols_of(c, true);
  chirp_rows_of(c, true);
}

void launch_chirp_fft(const ChirpArgs &F, const double *h0, const double *h1, double2 *Y, double2 *Z, hipStream_t s) {
  const ChirpCall c = {F, h0, h1, Y, Z, nullptr, s};
  chirp_cols_of(c, false);
  chirp_rows_of(c, false);
  chirp_back_of(c);
}

void launch_chirp_dot(const ChirpArgs &F, const double2 *Z, const double2 *data, const double *w, double2 *hw_out,
                      double *partials, hipStream_t s) {
  hipLaunchKernelGGL(k_chirp_dot, dim3(chirp_partials(F)), dim3(kPairThreads), 0, s, F, Z, data, w, hw_out, partials);
}

}  // namespace aak
