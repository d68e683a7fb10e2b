// aak_noalloc.hip -- the noise-weighted inner product on caller-owned device
// buffers, with no device allocation: aak_inner_product_noalloc.
//
// Short series take one kernel (k_fft_small), longer ones the first pass of the
// likelihood stage's four-step FFT, a second pass that reads the caller's data
// and weights in bin order, and the final reduction.  Their scratch -- the
// four-step intermediate, the twiddle tables and the partial sums -- lives in
// one file-scope device array, `scratch`, of kScratchBytes per GPU, held from
// module load to the end of the process.  Its device address is taken once per
// device with hipGetSymbolAddress and used for every kernel argument; the
// array's name itself is never handed to a kernel.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <string>

#include "aak_dense.hpp"
#include "aak_fft.hpp"

namespace aak {
int set_last_error(int code, const std::string &msg);
}

using namespace aak;

namespace {

// Largest length served: N = 2^21 (M = 2^20 complex points, R = C = 1024).
constexpr int kMaxN = 1 << 21;
constexpr size_t kMaxM = (size_t)kMaxN / 2;
constexpr size_t kAlign = 256;

constexpr size_t align_up(size_t b) { return (b + kAlign - 1) / kAlign * kAlign; }

// Regions for the largest length; smaller lengths use prefixes of each.
constexpr size_t kBytesY = align_up(sizeof(double2) * 2 * kMaxM);        // four-step intermediate, 2 channels
constexpr size_t kBytesTw = align_up(sizeof(double2) * 16384);           // twiddle tables (at most 10254 entries)
constexpr size_t kBytesP = align_up(sizeof(double) * 2 * 2048);          // partial-sum pairs (R <= 2048)
constexpr size_t kOffY = 0, kOffTw = kOffY + kBytesY, kOffP = kOffTw + kBytesTw,
                 kScratchBytes = kOffP + kBytesP;  // ~32 MiB
constexpr int kSmallM = 4096;  // points up to which one workgroup takes the whole product

__device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char *g_scratch[kMaxDevices] = {};  // device address of `scratch`, per device
int g_table_n[kMaxDevices] = {};             // length whose twiddles the device's scratch holds

int fail(int code, const std::string &msg) { return set_last_error(code, msg); }

}  // namespace

extern "C" int aak_inner_product_noalloc(const double *hI, const double *hII, const double *hI_f,
                                         const double *hII_f, const double *ASDinv1, const double *ASDinv2,
                                         int length, double *like_out, void *stream) {
  FftArgs F{};
  int R = 0, C = 0;
  if (!fft_supported(length, &R, &C) || length > kMaxN)
    return fail(-2, "inner_product_noalloc: length must be a power of two in [2^8, 2^21], got " +
                        std::to_string(length));
  if (!hI || !hII || !hI_f || !hII_f || !ASDinv1 || !ASDinv2 || !like_out)
    return fail(-2, "inner_product_noalloc: null pointer");
  const uintptr_t mis = (uintptr_t)hI | (uintptr_t)hII | (uintptr_t)hI_f | (uintptr_t)hII_f;
  if (mis & 15) return fail(-2, "inner_product_noalloc: series and spectra must be 16-byte aligned");
  F.N = length;
  F.M = length / 2;
  const bool small = F.M <= kSmallM;
  F.R = small ? 1 : R;
  F.C = small ? F.M : C;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(-100, std::string("HIP: ") + hipGetErrorString(e) + " at hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) return fail(-2, "inner_product_noalloc: device index out of range");
  unsigned char *base = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_scratch[dev]) {
      void *p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p)
        return fail(-100, std::string("HIP: ") + hipGetErrorString(e) + " at hipGetSymbolAddress(scratch)");
      g_scratch[dev] = static_cast<unsigned char *>(p);
    }
    base = g_scratch[dev];
    double2 *tw = reinterpret_cast<double2 *>(base + kOffTw);
    if (g_table_n[dev] != length) {
      // the tables of a new length: filled in a static host array (under the
      // lock) and copied; the call waits for the copy.  Later calls of this
      // length copy nothing and only enqueue kernels
      static double2 host[kBytesTw / sizeof(double2)];
      const size_t n = fft_table_size(F);
      if (n > kBytesTw / sizeof(double2)) return fail(-2, "inner_product_noalloc: twiddle tables too large");
      fft_fill_tables(F, host);
      e = hipMemcpyAsync(tw, host, sizeof(double2) * n, hipMemcpyHostToDevice, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e != hipSuccess) {
        g_table_n[dev] = 0;
        return fail(-100, std::string("HIP: ") + hipGetErrorString(e) + " uploading the FFT tables");
      }
      g_table_n[dev] = length;
    }
    fft_bind_tables(&F, tw);
  }
  double2 *Y = reinterpret_cast<double2 *>(base + kOffY);
  double *partials = reinterpret_cast<double *>(base + kOffP);
  F.Dp[0] = reinterpret_cast<const double2 *>(hI_f);
  F.Dp[1] = reinterpret_cast<const double2 *>(hII_f);
  F.wp[0] = ASDinv1;
  F.wp[1] = ASDinv2;
  // per call with its wait: N = 256 15 us in one launch (27 in five), 8192 25.5
  // (30.4), where one workgroup's LDS ends; 2^14 27 us in three launches (31),
  // 2^21 64 (73)
  if (small) {
    launch_fft_small(F, hI, hII, like_out, s);
  } else {
    launch_fft_pass1(F, hI, hII, Y, s);
    launch_fft_pass2_natural(F, Y, partials, s);
    launch_dot_final(partials, fft_natural_partials(F), like_out, nullptr, nullptr, s);
  }
  e = hipGetLastError();
  if (e != hipSuccess) return fail(-100, std::string("HIP: ") + hipGetErrorString(e) + " launching the inner product");
  return 0;
}
