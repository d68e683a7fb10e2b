// aak_fft.hpp -- fused real FFT + noise-weighted inner products (aak_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace aak {

// N = 2M real samples per channel, M = R C (powers of two).  Tables: W_R^e,
// W_C^e (e < R, C), W_M^e = twMhi[e >> 10] twMlo[e & 1023] for e < M and
// W_N^k = twNhi[k >> 10] twNlo[k & 1023] for k <= M, twNr[k2] = W_N^(R k2) for
// k2 < C.  Dp, wp: weighted data and
// weights of each channel in the order of the second pass, position
// k1 * C + k2 for bin k = k1 + R k2 (k < M), position M for the Nyquist bin.
struct FftArgs {
  int N, M, R, C;
  const double2 *twR, *twC, *twMlo, *twMhi, *twNlo, *twNhi, *twNr;
  const double2 *Dp[2];
  const double *wp[2];
};

// Lengths handled (powers of two, 2^8 <= N <= 2^23) and their R, C.
bool fft_supported(int N, int *R, int *C);
// Partial-sum pairs written by launch_fft_pass2.
int fft_partials(const FftArgs &F);
// Twiddle tables of F's lengths: their size (double2 entries), their values
// (host memory, extended-precision roots) and the table pointers of F bound
// to a device copy.
size_t fft_table_size(const FftArgs &F);
void fft_fill_tables(const FftArgs &F, double2 *tw);
void fft_bind_tables(FftArgs *F, const double2 *tw);
// Channels h0 and h1 (16-byte aligned).  Pass 1 writes the 2M-complex scratch Y;
// pass 2 writes fft_partials(F) pairs (sum of <h w, d w>, sum of |h w|^2) to
// partials and, if hw_out is not null, the weighted spectra h~ w ([2][M+1],
// natural order).
void launch_fft_pass1(const FftArgs &F, const double *h0, const double *h1, double2 *Y, hipStream_t s);
void launch_fft_pass2(const FftArgs &F, const double2 *Y, double *partials, double2 *hw_out, hipStream_t s);

// Pass 2 with the final reduction folded in: each row workgroup publishes its
// pair in `partials` (words that read kFinalEmpty until written); one extra
// workgroup, dispatched after all of them, collects the pairs and sums them
// in the order of the separate final reduction (k_dot_final: 256 lanes, lane t adds pairs t, t + 256, ...
// in turn, then a halving tree), writes out[0..1] = 4 x the sums (NaN when
// flags[3] is set), zeroes clear[0..7] (flags and clear may be null) and
// returns every word to kFinalEmpty.  A pair that never arrives within the
// spin cap reads as NaN.  launch_fft_final_reset brings a new buffer to that
// state.
struct FftFinal {
  double *out;
  const int *flags;
  int *clear;
};
constexpr long long kFinalEmpty = 0x7FF4A5A5A5A5A5B1LL;  // a signalling NaN: no arithmetic result
void launch_fft_pass2_final(const FftArgs &F, const double2 *Y, double *partials, const FftFinal &fin, hipStream_t s);
void launch_fft_final_reset(double *partials, int npairs, hipStream_t s);

// Data and weights in bin order (Dp, wp of M + 1 bins each).  Pass 2 for C from
// 64 to 1024: fft_natural_partials(F) pairs.
int fft_natural_partials(const FftArgs &F);
void launch_fft_pass2_natural(const FftArgs &F, const double2 *Y, double *partials, hipStream_t s);
// The whole inner product of a short series, M from 128 to 4096 with R = 1 and
// C = M: out[0..1] = 4 x the sums.  False: another M.
bool launch_fft_small(const FftArgs &F, const double *h0, const double *h1, double *out, hipStream_t s);

// Lengths N = 2M whose half has a prime factor above 17: the M-point transform as a cyclic
// convolution of length L = R C >= 2M - 1 (Bluestein), R from 2^a, C from 2^a,
// 3 2^a and 9 2^a.
// Tables as in FftArgs (W_L in place of W_M); chirp: exp(-i pi m^2 / M), m < M;
// filter: the convolution filter's transform over L, position k1 C + k2.
struct ChirpArgs {
  int N, M, L, R, C;
  const double2 *twR, *twC, *twLlo, *twLhi, *twNlo, *twNhi, *chirp, *filter;
};
// Lengths handled (even, from 64 to 4718590, N/2 with a prime factor above 17)
// and the smallest R C for them.
bool chirp_supported(int N, int *R, int *C);
int chirp_partials(const ChirpArgs &F);
// Size of the tables (double2 entries); the part the host fills (its size, and
// its values when tw is given: the rest is formed by launch_chirp_init, which
// uses L entries of Y); the pointers of F bound to a device copy.
size_t chirp_table_size(const ChirpArgs &F);
size_t chirp_host_tables(const ChirpArgs &F, double2 *tw);
void chirp_bind_tables(ChirpArgs *F, double2 *tw);
void launch_chirp_init(const ChirpArgs &F, double2 *tw, double2 *Y, hipStream_t s);
// Channels h0 and h1 (16-byte aligned) to their M-point transforms Z ([2][M]),
// with 2L entries of scratch Y.
void launch_chirp_fft(const ChirpArgs &F, const double *h0, const double *h1, double2 *Y, double2 *Z, hipStream_t s);
// chirp_partials(F) pairs (sum of <h w, d w>, sum of |h w|^2) and, if hw_out is
// not null, the weighted spectra ([2][M+1]); data and weights in natural order.
void launch_chirp_dot(const ChirpArgs &F, const double2 *Z, const double2 *data, const double *w, double2 *hw_out,
                      double *partials, hipStream_t s);

}  // namespace aak
