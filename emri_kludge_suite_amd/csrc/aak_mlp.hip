// aak_mlp.hip -- learned start point for the frequency map (KSParMap.cc:397-440):
// a 4-128-128-128-3 network with GELU activations, BF16 weights and FP32
// accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16), with its
// training kernels (one for forward, backward and weight-gradient partials,
// one for their sum and Adam) and batched inference.
//
// The network maps the normalised features of a trajectory point
// (a, 1/sqrt(p), e, cos iota) to the standardised corrections
// (v_map - 1/sqrt(p), M_map/M - 1, s_map - a); the host turns them into the
// start point of a Newton polish of the map (aak_freqmap.hpp).
//
// Rounding points (the CPU gradient reference reproduces them): weight
// matrices in BF16, biases FP32; the inputs of every matrix-core product in
// BF16 (activations A1..A3, the output gradient dY and the back-propagated
// dZ3, dZ2); everything else FP32.  Layer 1 (K = 4) and the products with
// K = 3 or an output width of 3 on the weight-gradient side run on the VALU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../include/gpuAAK.h"
#include "aak_mlp.hpp"

namespace aak {
int set_last_error(int code, const std::string &msg);
}

using namespace aak;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int H = kMlpHidden;  // 128
constexpr int LDW = H + 8;     // LDS row stride (bf16): 272 B, conflict-free 16-byte fragment reads
constexpr int TILE = 64;       // rows per workgroup of the inference kernel
constexpr int GROWS = 32;      // rows per tile of the gradient kernel: the K of one matrix instruction
constexpr int LDT = GROWS + 8; // its transposed tiles' row stride (80 B, conflict-free 16-byte reads)
constexpr int kGradGroups = 256;  // most workgroups (and partial gradients) of the gradient kernel
constexpr int kThreads = 256;

int fail(int code, const std::string &msg) { return set_last_error(code, msg); }

#define MLPCHK(x)                                                                                     \
  do {                                                                                                \
    hipError_t e_ = (x);                                                                              \
    if (e_ != hipSuccess) return fail(-100, std::string("HIP: ") + hipGetErrorString(e_) + " at " #x); \
  } while (0)

__device__ __forceinline__ uint16_t bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// GELU, tanh form, and its derivative
__device__ __forceinline__ float gelu(float z) {
  const float c = 0.7978845608028654f;
  return 0.5f * z * (1.0f + tanhf(c * (z + 0.044715f * z * z * z)));
}
__device__ __forceinline__ float gelu_and_grad(float z, float *grad) {
  const float c = 0.7978845608028654f;
  const float t = tanhf(c * (z + 0.044715f * z * z * z));
  *grad = 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * c * (1.0f + 3.0f * 0.044715f * z * z);
  return 0.5f * z * (1.0f + t);
}

__device__ __forceinline__ bf16x8 load8(const uint16_t *p) {
  const uint4 v = *reinterpret_cast<const uint4 *>(p);
  return __builtin_bit_cast(bf16x8, v);
}

// Parameter offsets (floats) in the flat vector: W1[4][128] b1 W2[128][128]
// b2 W3[128][128] b3 W4[128][3] b4[3]; W[k][n] is input k to output n.
constexpr int oW1 = 0, oB1 = oW1 + 4 * H, oW2 = oB1 + H, oB2 = oW2 + H * H, oW3 = oB2 + H, oB3 = oW3 + H * H,
              oW4 = oB3 + H, oB4 = oW4 + 3 * H, kNP = oB4 + 3;
static_assert(kNP == kMlpParams, "parameter count");

// Stage W (H x H, k-major bf16 in global) into LDS, transposed (row n holds
// input k contiguous) when `trans`, natural (row k holds n) otherwise.
__device__ void stage_hxh(uint16_t *lds, const uint16_t *W, bool trans) {
  for (int q = threadIdx.x; q < H * H / 8; q += kThreads) {
    const int k = q / (H / 8), n0 = (q % (H / 8)) * 8;
    const uint4 v = *reinterpret_cast<const uint4 *>(W + k * H + n0);
    const uint16_t *e = reinterpret_cast<const uint16_t *>(&v);
    if (trans) {
      for (int j = 0; j < 8; j++) lds[(n0 + j) * LDW + k] = e[j];
    } else {
      *reinterpret_cast<uint4 *>(lds + k * LDW + n0) = v;
    }
  }
}

// One 16-row x 128-column product per wave: acc[t] (columns 16t..16t+15,
// C layout: lane holds rows 4(l/16)+i of column l%16) += act[16 rows][K] x B,
// B fragments from `wl` (row = output column, K contiguous).
__device__ __forceinline__ void wave_gemm_128(floatx4 acc[8], const uint16_t *act, const uint16_t *wl, int K) {
  const int l = threadIdx.x & 63;
  for (int k0 = 0; k0 < K; k0 += 32) {
    const bf16x8 a = load8(act + (l & 15) * LDW + k0 + 8 * (l >> 4));
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const bf16x8 b = load8(wl + (16 * t + (l & 15)) * LDW + k0 + 8 * (l >> 4));
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[t], 0, 0, 0);
    }
  }
}

// ---------------------------------------------------------------- inference
// Rows [blockIdx.x * 64, +64) of X to Y.
__global__ __launch_bounds__(kThreads) void k_mlp_forward(const float *__restrict__ X, int n,
                                                          const float *__restrict__ P, const uint16_t *__restrict__ Pb,
                                                          float *__restrict__ Y) {
  __shared__ __align__(16) uint16_t wl[H * LDW];
  __shared__ __align__(16) uint16_t act[TILE * LDW];
  __shared__ float xs[TILE][4];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row0 = blockIdx.x * TILE;
  for (int q = threadIdx.x; q < TILE * 4; q += kThreads) {
    const int r = q >> 2, k = q & 3, gr = row0 + r;
    xs[r][k] = gr < n ? X[(size_t)gr * 4 + k] : 0.f;
  }
  __syncthreads();
  // layer 1 on the VALU: lane (row l%16 of the wave, columns 32 (l/16) + j)
  {
    const int r = 16 * w + (l & 15);
    const float x0 = xs[r][0], x1 = xs[r][1], x2 = xs[r][2], x3 = xs[r][3];
    for (int j = 0; j < 32; j++) {
      const int c = 32 * (l >> 4) + j;
      float z = P[oB1 + c];
      z = fmaf(x0, bf16_to_f32(Pb[oW1 + c]), z);
      z = fmaf(x1, bf16_to_f32(Pb[oW1 + H + c]), z);
      z = fmaf(x2, bf16_to_f32(Pb[oW1 + 2 * H + c]), z);
      z = fmaf(x3, bf16_to_f32(Pb[oW1 + 3 * H + c]), z);
      act[r * LDW + c] = bf16_bits(gelu(z));
    }
  }
  // layers 2 and 3 on the matrix cores
  for (int layer = 0; layer < 2; layer++) {
    __syncthreads();
    stage_hxh(wl, Pb + (layer ? oW3 : oW2), true);
    __syncthreads();
    floatx4 acc[8];
    for (int t = 0; t < 8; t++) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    wave_gemm_128(acc, act + 16 * w * LDW, wl, H);
    __syncthreads();
    const float *bias = P + (layer ? oB3 : oB2);
    for (int t = 0; t < 8; t++) {
      const int c = 16 * t + (l & 15);
      for (int i = 0; i < 4; i++) {
        const int r = 16 * w + 4 * (l >> 4) + i;
        const float z = acc[t][i] + bias[c];
        act[r * LDW + c] = bf16_bits(gelu(z));
      }
    }
  }
  // layer 4: output width 3, padded to 16 columns
  __syncthreads();
  for (int q = threadIdx.x; q < 16 * H; q += kThreads) {
    const int j = q / H, k = q % H;
    wl[j * LDW + k] = j < 3 ? Pb[oW4 + k * 3 + j] : (uint16_t)0;
  }
  __syncthreads();
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < H; k0 += 32) {
    const bf16x8 a = load8(act + (16 * w + (l & 15)) * LDW + k0 + 8 * (l >> 4));
    const bf16x8 b = load8(wl + (l & 15) * LDW + k0 + 8 * (l >> 4));
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
  const int j = l & 15;
  if (j < 3) {
    for (int i = 0; i < 4; i++) {
      const int gr = row0 + 16 * w + 4 * (l >> 4) + i;
      if (gr < n) Y[(size_t)gr * 3 + j] = acc[i] + P[oB4 + j];
    }
  }
}

// ---------------------------------------------------------------- gradient
// Forward, loss, backward chain and weight gradients of tiles of 32 rows; row r
// of the batch is row idx[r] of X/T (idx null: identity).  A workgroup takes
// tiles blockIdx.x, + gridDim.x, ... and writes one partial gradient and one
// partial of the squared error.
//   waves        wave w: rows 16 (w & 1), output columns 32 (w >> 1)
//   products     weights as B fragments straight from L2 (Wt the transposed
//                copies for the forward direction), the next layer's loaded while
//                this one's activations are formed;
//                activations and dZ through LDS, once per direction
//   registers    gelu'(Z1..Z3) of the wave's 16 x 32 elements stay there; dW2,
//                dW3 (K = the tile's 32 rows: one matrix instruction per
//                16 x 16 block) and the VALU sums of dW1, dW4 and the biases
//                accumulate over the workgroup's tiles
// Bound by the latency of the chain of seven products and barriers, about
// 19 us for one tile, and by the 137 KB of each partial: the work itself is
// 0.8 GFLOP at 4096 rows.  There it takes 30 us, where separate forward,
// backward and weight-gradient kernels took 280: those passed Z1..Z3 and
// dZ1..dZ3 through memory, 12 MB, and the last ran 32 workgroups that walked
// 128 rows one after another.  At 16384 rows: 43 us with up to 256 workgroups
// (one per CU), 64 with up to 128.
constexpr int CB = 2;              // 16-column blocks of a wave
constexpr int kGradThreads = 512;  // eight waves: two per SIMD
typedef bf16x8 Frags[CB][4];       // [16-column block][32-deep K step]
__device__ __forceinline__ void load_frags(Frags f, const uint16_t *W, int l, int col0) {
#pragma unroll
  for (int t = 0; t < CB; t++)
#pragma unroll
    for (int k = 0; k < 4; k++) f[t][k] = load8(W + (col0 + 16 * t + (l & 15)) * H + 32 * k + 8 * (l >> 4));
}
// acc[t] = (16 rows of act) x (the wave's column blocks, f)
__device__ __forceinline__ void frag_gemm(floatx4 acc[CB], const uint16_t *act, const Frags f, int l) {
#pragma unroll
  for (int t = 0; t < CB; t++) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const bf16x8 a = load8(act + (l & 15) * LDW + 32 * k + 8 * (l >> 4));
#pragma unroll
    for (int t = 0; t < CB; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, f[t][k], acc[t], 0, 0, 0);
  }
}
// dW[t] += A^T dZ over the tile's rows: block row w of wave w
__device__ __forceinline__ void grad_gemm(floatx4 acc[8], const uint16_t *at, const uint16_t *dt, int l, int w) {
  const bf16x8 a = load8(at + (16 * w + (l & 15)) * LDT + 8 * (l >> 4));
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const bf16x8 d = load8(dt + (16 * t + (l & 15)) * LDT + 8 * (l >> 4));
    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, d, acc[t], 0, 0, 0);
  }
}
// Four rows r..r+3 of one column, rounded: row-major and transposed.
__device__ __forceinline__ void put4(uint16_t *rm, uint16_t *tp, int r, int c, const float v[4]) {
  uint16_t b[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    b[i] = bf16_bits(v[i]);
    if (rm) rm[(r + i) * LDW + c] = b[i];
  }
  if (tp)
    *reinterpret_cast<uint2 *>(tp + c * LDT + r) =
        make_uint2(b[0] | ((uint32_t)b[1] << 16), b[2] | ((uint32_t)b[3] << 16));
}

__global__ __launch_bounds__(kGradThreads) void k_mlp_gradient(const float *__restrict__ X, const float *__restrict__ T,
                                                              const int *__restrict__ idx, int n,
                                                              const float *__restrict__ P,
                                                              const uint16_t *__restrict__ Pb,
                                                              const uint16_t *__restrict__ Wt, float *__restrict__ part,
                                                              float *__restrict__ loss_part, float dscale) {
  __shared__ __align__(16) uint16_t rows[5][GROWS * LDW];  // A1, A2, A3, dZ3, dZ2
  __shared__ __align__(16) uint16_t cols[4][H * LDT];      // A1, A2, dZ3, dZ2 transposed
  __shared__ float sm[7][H];                    // W1, b1, b2, b3
  __shared__ __align__(16) uint16_t w4t[16 * LDW];  // W4 transposed, outputs past 3 zero
  __shared__ __align__(16) uint16_t w4n[H * 8];     // W4, zeros past 3
  __shared__ float xs[GROWS][4], ts[GROWS][4];
  __shared__ float dy[8][16][4];  // each wave's rows of dY
  __shared__ float red[2][10][H];
  __shared__ float red4[2][4];
  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  const int rg = 16 * (w & 1), col0 = 16 * CB * (w >> 1), lc = l & 15, lr = rg + 4 * (l >> 4);
  const int tiles = (n + GROWS - 1) / GROWS;

  // the small parameters: W1 and the biases as floats, W4 for either direction
  for (int q = tid; q < 4 * H; q += kGradThreads) sm[q / H][q % H] = bf16_to_f32(Pb[oW1 + q]);
  for (int q = tid; q < 3 * H; q += kGradThreads) {
    const int c = q % H, j = q / H;
    sm[4 + j][c] = P[(j == 0 ? oB1 : j == 1 ? oB2 : oB3) + c];
    const uint16_t v = Pb[oW4 + 3 * c + j];
    w4t[j * LDW + c] = v;
    w4n[c * 8 + j] = v;
  }
  for (int q = tid; q < 13 * H; q += kGradThreads) w4t[(3 + q / H) * LDW + q % H] = 0;
  for (int q = tid; q < 5 * H; q += kGradThreads) w4n[(q % H) * 8 + 3 + q / H] = 0;
  const float b4 = lc < 3 ? P[oB4 + lc] : 0.f;

  floatx4 dw2[8], dw3[8];
  float dw1[CB][4], dw4[CB][3], db1[CB], db2[CB], db3[CB], db4 = 0.f, se = 0.f;
#pragma unroll
  for (int t = 0; t < 8; t++) dw2[t] = dw3[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < CB; t++) {
    db1[t] = db2[t] = db3[t] = 0.f;
    for (int k = 0; k < 4; k++) dw1[t][k] = 0.f;
    for (int j = 0; j < 3; j++) dw4[t][j] = 0.f;
  }

#pragma unroll 1
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int row0 = tile * GROWS;
    // opaque offset: keeps the weights' fragments (128 registers) from being
    // hoisted out of the tile loop, into scratch
    int o = 0;
    asm volatile("" : "+s"(o));
    Frags f;
    load_frags(f, Wt + o, l, col0);
    if (tid < GROWS * 4) {
      const int r = tid >> 2, k = tid & 3, gr = row0 + r;
      xs[r][k] = gr < n ? X[(size_t)(idx ? idx[gr] : gr) * 4 + k] : 0.f;
    } else if (tid - GROWS * 4 < GROWS * 3) {
      const int q = tid - GROWS * 4, r = q / 3, j = q % 3, gr = row0 + r;
      ts[r][j] = gr < n ? T[(size_t)(idx ? idx[gr] : gr) * 3 + j] : 0.f;
    }
    __syncthreads();
    float in[4];  // 1 for the rows below n
#pragma unroll
    for (int i = 0; i < 4; i++) in[i] = row0 + lr + i < n ? 1.f : 0.f;
    float g1[CB][4], g2[CB][4], g3[CB][4];
    // layer 1 on the VALU
#pragma unroll
    for (int t = 0; t < CB; t++) {
      const int c = col0 + 16 * t + lc;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float *x = xs[lr + i];
        float z = sm[4][c];
        z = fmaf(x[0], sm[0][c], z);
        z = fmaf(x[1], sm[1][c], z);
        z = fmaf(x[2], sm[2][c], z);
        z = fmaf(x[3], sm[3][c], z);
        v[i] = gelu_and_grad(z, &g1[t][i]);
      }
      put4(rows[0], cols[0], lr, c, v);
    }
    __syncthreads();
    floatx4 acc[CB];
    frag_gemm(acc, rows[0] + rg * LDW, f, l);
    load_frags(f, Wt + o + H * H, l, col0);
#pragma unroll
    for (int t = 0; t < CB; t++) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = gelu_and_grad(acc[t][i] + sm[5][col0 + 16 * t + lc], &g2[t][i]);
      put4(rows[1], cols[1], lr, col0 + 16 * t + lc, v);
    }
    __syncthreads();
    frag_gemm(acc, rows[1] + rg * LDW, f, l);
    load_frags(f, Pb + o + oW3, l, col0);
#pragma unroll
    for (int t = 0; t < CB; t++) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = gelu_and_grad(acc[t][i] + sm[6][col0 + 16 * t + lc], &g3[t][i]);
      put4(rows[2], nullptr, lr, col0 + 16 * t + lc, v);
    }
    __syncthreads();
    // layer 4 and the loss, by all four waves of the rows
    {
      floatx4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const bf16x8 a = load8(rows[2] + (rg + lc) * LDW + 32 * k + 8 * (l >> 4));
        y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, load8(w4t + lc * LDW + 32 * k + 8 * (l >> 4)), y, 0, 0, 0);
      }
      if (lc < 3) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float d = row0 + lr + i < n ? y[i] + b4 - ts[lr + i][lc] : 0.f;
          se += d * d;
          db4 += dscale * d;
          dy[w][4 * (l >> 4) + i][lc] = dscale * d;
        }
      }
    }
    __syncthreads();
    // dA3 = dY W4^T (K padded from 3); dZ = dA * gelu'(Z)
    {
      uint16_t u[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (l < 16)
        for (int q = 0; q < 3; q++) u[q] = bf16_bits(dy[w][lc][q]);
      bf16x8 a;
      __builtin_memcpy(&a, u, 16);
#pragma unroll
      for (int t = 0; t < CB; t++) {
        // lanes past 15 face the zeros of dY's K = 8..31
        const bf16x8 b = load8(w4n + (col0 + 16 * t + lc) * 8);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < CB; t++) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        v[i] = in[i] != 0.f ? acc[t][i] * g3[t][i] : 0.f;
        db3[t] += v[i];
        const float a3 = bf16_to_f32(rows[2][(lr + i) * LDW + col0 + 16 * t + lc]);
        const float *d = dy[w][4 * (l >> 4) + i];
#pragma unroll
        for (int j = 0; j < 3; j++) dw4[t][j] = fmaf(a3, d[j], dw4[t][j]);
      }
      put4(rows[3], cols[2], lr, col0 + 16 * t + lc, v);
    }
    __syncthreads();
    frag_gemm(acc, rows[3] + rg * LDW, f, l);
    load_frags(f, Pb + o + oW2, l, col0);
#pragma unroll
    for (int t = 0; t < CB; t++) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        v[i] = in[i] != 0.f ? acc[t][i] * g2[t][i] : 0.f;
        db2[t] += v[i];
      }
      put4(rows[4], cols[3], lr, col0 + 16 * t + lc, v);
    }
    __syncthreads();
    frag_gemm(acc, rows[4] + rg * LDW, f, l);
#pragma unroll
    for (int t = 0; t < CB; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float d = in[i] != 0.f ? acc[t][i] * g1[t][i] : 0.f;
        db1[t] += d;
#pragma unroll
        for (int k = 0; k < 4; k++) dw1[t][k] = fmaf(xs[lr + i][k], d, dw1[t][k]);
      }
    grad_gemm(dw3, cols[1], cols[2], l, w);
    grad_gemm(dw2, cols[0], cols[3], l, w);
    __syncthreads();  // the next tile overwrites
  }

  float *out = part + (size_t)blockIdx.x * kNP;
#pragma unroll
  for (int t = 0; t < 8; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int q = (16 * w + 4 * (l >> 4) + i) * H + 16 * t + lc;
      out[oW2 + q] = dw2[t][i];
      out[oW3 + q] = dw3[t][i];
    }
  // the VALU sums: over a column's lanes, then the two row groups.  Sum s:
  // 0..3 dW1, 4..6 dW4, 7..9 the biases 1..3
  auto rowsum = [](float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
  };
#pragma unroll
  for (int t = 0; t < CB; t++)
#pragma unroll
    for (int s = 0; s < 10; s++) {
      const float x = rowsum(s < 4 ? dw1[t][s] : s < 7 ? dw4[t][s - 4] : s == 7 ? db1[t] : s == 8 ? db2[t] : db3[t]);
      if (l < 16) red[w & 1][s][col0 + 16 * t + lc] = x;
    }
  se = rowsum(se);
  db4 = rowsum(db4);
  if (w < 2 && l < 3) red4[w][l] = db4;
  se += __shfl_xor(se, 1);  // lanes 0..2 hold the sums, the rest 0
  se += __shfl_xor(se, 2);
  if (w < 2 && l == 0) red4[w][3] = se;
  __syncthreads();
  for (int q = tid; q < 10 * H; q += kGradThreads) {
    const int s = q / H, c = q % H;
    const int o = s < 4 ? oW1 + s * H + c : s < 7 ? oW4 + 3 * c + s - 4 : s == 7 ? oB1 + c : s == 8 ? oB2 + c : oB3 + c;
    out[o] = red[0][s][c] + red[1][s][c];
  }
  if (tid < 3) out[oB4 + tid] = red4[0][tid] + red4[1][tid];
  if (tid == 3) loss_part[blockIdx.x] = red4[0][3] + red4[1][3];
}

// ----------------------------------------------------------------- Adam
// g = sum of the partials (four slices of them per parameter, 64 parameters per
// workgroup, so that many loads are in flight); with step > 0 an Adam step on
// the FP32 master copy, whose BF16 copies are refreshed; with step == 0 only g
// is written.
__device__ __forceinline__ void put_bf16(int p, float x, uint16_t *Pb, uint16_t *Wt) {
  const uint16_t b = bf16_bits(x);
  Pb[p] = b;
  const int q2 = p - oW2, q3 = p - oW3;
  if (q2 >= 0 && q2 < H * H) Wt[(q2 % H) * H + q2 / H] = b;
  if (q3 >= 0 && q3 < H * H) Wt[H * H + (q3 % H) * H + q3 / H] = b;
}

__global__ __launch_bounds__(kThreads) void k_mlp_adam(int nparts, const float *__restrict__ part,
                                                       float *__restrict__ grad, float *__restrict__ P,
                                                       uint16_t *__restrict__ Pb, uint16_t *__restrict__ Wt,
                                                       float *__restrict__ m1, float *__restrict__ m2, int step,
                                                       float lr, float b1, float b2, float eps) {
  __shared__ float sum[4][64];
  const int j = threadIdx.x & 63, slice = threadIdx.x >> 6, p = blockIdx.x * 64 + j;
  float g = 0.f;
  if (p < kNP) {
#pragma unroll 8
    for (int c = slice; c < nparts; c += 4) g += part[(size_t)c * kNP + p];
  }
  sum[slice][j] = g;
  __syncthreads();
  if (slice || p >= kNP) return;
  g = (sum[0][j] + sum[1][j]) + (sum[2][j] + sum[3][j]);
  grad[p] = g;
  if (step <= 0) return;
  const float a = b1 * m1[p] + (1.f - b1) * g, v = b2 * m2[p] + (1.f - b2) * g * g;
  m1[p] = a;
  m2[p] = v;
  const float ah = a / (1.f - powf(b1, (float)step)), vh = v / (1.f - powf(b2, (float)step));
  const float x = P[p] - lr * ah / (sqrtf(vh) + eps);
  P[p] = x;
  put_bf16(p, x, Pb, Wt);
}

__global__ void k_mlp_round(const float *__restrict__ P, uint16_t *__restrict__ Pb, uint16_t *__restrict__ Wt) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p < kNP) put_bf16(p, P[p], Pb, Wt);
}

}  // namespace

// ------------------------------------------------------------------ host
struct aak_mlp_s {
  float *P = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
  uint16_t *Pb = nullptr;
  uint16_t *Wt = nullptr;  // W2, W3 in BF16, transposed (row n holds input k)
  int step = 0;
  float norm[kMlpNorm] = {};  // feature centres/scales and target means/scales
  hipStream_t s = nullptr;
  int dev = 0;  // device the model lives on (callers may be other host threads)
  // training / gradient scratch (grown on demand)
  int cap = 0;
  float *X = nullptr, *T = nullptr, *loss = nullptr, *part = nullptr;
  int *idx = nullptr;
  int data_n = 0;
  float *pin = nullptr;  // pinned: X | T of up to kPinRows rows, gradient, loss partials
  bool no_pin = false;   // test hook: as if pinned memory were not to be had
  // inference scratch
  std::mutex mu;
  int icap = 0;
  float *iX = nullptr, *iY = nullptr;
  std::vector<float> hx, hy;
};


namespace aak {

static void free_scratch(aak_mlp_s *m) {
  void *ps[] = {m->X, m->T, m->loss, m->part, m->idx};
  for (void *p : ps)
    if (p) (void)hipFree(p);
  m->X = m->T = m->loss = m->part = nullptr;
  m->idx = nullptr;
  m->cap = 0;
  m->data_n = 0;
}

// Rows up to which a gradient call passes its data through pinned memory, read
// and written by the kernels themselves: 56 us a call at 4096 rows against 90
// with two uploads and two downloads, 46 against 121 at 64, 83 against 120 at
// 16384.  Longer calls upload, so the buffer stays at 0.6 MB.
constexpr int kPinRows = 16384;

// The model's pinned buffer, formed on first use; null where it cannot be had
// (the call then uploads).
static float *pinned_buffer(aak_mlp_s *m) {
  if (m->no_pin) return nullptr;
  if (!m->pin && hipHostMalloc((void **)&m->pin, sizeof(float) * (7 * (size_t)kPinRows + kNP + kGradGroups),
                               hipHostMallocDefault) != hipSuccess) {
    m->pin = nullptr;
    (void)hipGetLastError();
  }
  return m->pin;
}

static int grad_groups(int B) { return std::min(kGradGroups, (B + GROWS - 1) / GROWS); }

// Scratch for batches of up to B rows over a data set of `data` rows.
static int grow_scratch(aak_mlp_s *m, int B, int data) {
  const int groups = grad_groups(B);
  if (groups > m->cap) {
    void *ps[] = {m->loss, m->part};
    for (void *p : ps)
      if (p) (void)hipFree(p);
    m->loss = m->part = nullptr;
    m->cap = 0;
    MLPCHK(hipMalloc(&m->loss, sizeof(float) * groups));
    MLPCHK(hipMalloc(&m->part, sizeof(float) * (size_t)groups * kNP));
    m->cap = groups;
  }
  if (data > m->data_n) {
    if (m->X) (void)hipFree(m->X);
    if (m->T) (void)hipFree(m->T);
    if (m->idx) (void)hipFree(m->idx);
    MLPCHK(hipMalloc(&m->X, sizeof(float) * 4 * (size_t)data));
    MLPCHK(hipMalloc(&m->T, sizeof(float) * 3 * (size_t)data));
    MLPCHK(hipMalloc(&m->idx, sizeof(int) * (size_t)data));
    m->data_n = data;
  }
  return 0;
}

// One forward + backward over rows idx[0 .. B) of X, T (idx null: the first B);
// with `update` an Adam step.
static void launch_step(aak_mlp_s *m, const float *X, const float *T, const int *idx, int B, float lr, bool update,
                        float *grad, float *loss) {
  const int groups = grad_groups(B);
  const float dscale = 2.f / (3.f * (float)B);
  hipLaunchKernelGGL(k_mlp_gradient, dim3(groups), dim3(kGradThreads), 0, m->s, X, T, idx, B, m->P, m->Pb, m->Wt,
                     m->part, loss, dscale);
  if (update) m->step++;
  hipLaunchKernelGGL(k_mlp_adam, dim3((kNP + 63) / 64), dim3(kThreads), 0, m->s, groups, m->part, grad, m->P, m->Pb,
                     m->Wt, m->m1, m->m2, update ? m->step : 0, lr, 0.9f, 0.999f, 1e-8f);
}

// launch_step over the uploaded data.  loss_sum (optional) gets the squared error.
static int train_step(aak_mlp_s *m, const int *idx, int B, float lr, bool update, double *loss_sum) {
  const int groups = grad_groups(B);
  launch_step(m, m->X, m->T, idx, B, lr, update, m->grad, m->loss);
  MLPCHK(hipGetLastError());
  if (loss_sum) {
    std::vector<float> lp(groups);
    MLPCHK(hipMemcpyAsync(lp.data(), m->loss, sizeof(float) * groups, hipMemcpyDeviceToHost, m->s));
    MLPCHK(hipStreamSynchronize(m->s));
    double s = 0.0;
    for (float x : lp) s += x;
    *loss_sum = s;
  }
  return 0;
}

// Normalised features of (a, p, e, iota) and the corrections of a map
// (v_map, M_map/M, s_map) -- see the file comment.
static void features(const aak_mlp_s *m, const double *pt, float *x) {
  const double a = pt[0], p = pt[1], e = pt[2], ci = cos(pt[3]);
  const double f[4] = {a, 1.0 / sqrt(p), e, ci};
  for (int k = 0; k < 4; k++) x[k] = (float)((f[k] - m->norm[k]) / m->norm[4 + k]);
}

int mlp_infer(aak_mlp_s *m, const double *pts, int n, double *maps) {
  if (n <= 0) return 0;
  std::lock_guard<std::mutex> lk(m->mu);
  MLPCHK(hipSetDevice(m->dev));
  if (n > m->icap) {
    if (m->iX) (void)hipFree(m->iX);
    if (m->iY) (void)hipFree(m->iY);
    m->iX = m->iY = nullptr;
    m->icap = 0;
    MLPCHK(hipMalloc(&m->iX, sizeof(float) * 4 * (size_t)n));
    MLPCHK(hipMalloc(&m->iY, sizeof(float) * 3 * (size_t)n));
    m->icap = n;
  }
  m->hx.resize(4 * (size_t)n);
  m->hy.resize(3 * (size_t)n);
  for (int i = 0; i < n; i++) features(m, pts + 4 * (size_t)i, m->hx.data() + 4 * (size_t)i);
  MLPCHK(hipMemcpyAsync(m->iX, m->hx.data(), sizeof(float) * 4 * (size_t)n, hipMemcpyHostToDevice, m->s));
  hipLaunchKernelGGL(k_mlp_forward, dim3((n + TILE - 1) / TILE), dim3(kThreads), 0, m->s, m->iX, n, m->P, m->Pb,
                     m->iY);
  MLPCHK(hipGetLastError());
  MLPCHK(hipMemcpyAsync(m->hy.data(), m->iY, sizeof(float) * 3 * (size_t)n, hipMemcpyDeviceToHost, m->s));
  MLPCHK(hipStreamSynchronize(m->s));
  for (int i = 0; i < n; i++) {
    const double *pt = pts + 4 * (size_t)i;
    const float *y = m->hy.data() + 3 * (size_t)i;
    const double c[3] = {m->norm[8] + m->norm[11] * (double)y[0], m->norm[9] + m->norm[12] * (double)y[1],
                         m->norm[10] + m->norm[13] * (double)y[2]};
    maps[3 * (size_t)i + 0] = 1.0 / sqrt(pt[1]) + c[0];
    maps[3 * (size_t)i + 1] = 1.0 + c[1];
    maps[3 * (size_t)i + 2] = pt[0] + c[2];
  }
  return 0;
}

}  // namespace aak

// ------------------------------------------------------------------ C ABI
extern "C" {

int aak_mlp_create(int seed, aak_mlp *out) {
  if (!out) return fail(-2, "null model pointer");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(-100, "no HIP device");
  aak_mlp_s *m = new aak_mlp_s();
  if (hipGetDevice(&m->dev) != hipSuccess) m->dev = 0;
  auto bail = [&](int rc) {
    aak_mlp_destroy(m);
    return rc;
  };
  if (hipStreamCreateWithFlags(&m->s, hipStreamNonBlocking) != hipSuccess) return bail(fail(-100, "stream"));
  float *bufs[4];
  for (int k = 0; k < 4; k++)
    if (hipMalloc(&bufs[k], sizeof(float) * kNP) != hipSuccess) {
      for (int j = 0; j < k; j++) (void)hipFree(bufs[j]);
      return bail(fail(-100, "device allocation of the parameters failed"));
    }
  m->P = bufs[0];
  m->m1 = bufs[1];
  m->m2 = bufs[2];
  m->grad = bufs[3];
  if (hipMalloc(&m->Pb, sizeof(uint16_t) * kNP) != hipSuccess ||
      hipMalloc(&m->Wt, sizeof(uint16_t) * 2 * H * H) != hipSuccess)
    return bail(fail(-100, "device allocation failed"));
  // He-style initialisation; identity normalisation until the trainer sets it
  std::mt19937_64 rng((uint64_t)seed);
  std::vector<float> p(kNP, 0.f);
  auto fill = [&](int off, int fan_in, int count) {
    std::normal_distribution<float> d(0.f, sqrtf(2.f / (float)fan_in));
    for (int i = 0; i < count; i++) p[off + i] = d(rng);
  };
  fill(oW1, 4, 4 * H);
  fill(oW2, H, H * H);
  fill(oW3, H, H * H);
  fill(oW4, H, 3 * H);
  for (int k = 0; k < 4; k++) m->norm[4 + k] = 1.f;
  for (int k = 0; k < 3; k++) m->norm[11 + k] = 1.f;
  const int rc = aak_mlp_set_params(m, p.data(), nullptr);
  if (rc) return bail(rc);
  std::vector<float> zero(kNP, 0.f);
  if (hipMemcpy(m->m1, zero.data(), sizeof(float) * kNP, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(m->m2, zero.data(), sizeof(float) * kNP, hipMemcpyHostToDevice) != hipSuccess)
    return bail(fail(-100, "upload failed"));
  *out = m;
  return 0;
}

int aak_mlp_destroy(aak_mlp m) {
  if (!m) return fail(-1, "null model");
  if (m->s) (void)hipStreamSynchronize(m->s);
  free_scratch(m);
  if (m->pin) (void)hipHostFree(m->pin);
  void *ps[] = {m->P, m->m1, m->m2, m->grad, m->Pb, m->Wt, m->iX, m->iY};
  for (void *p : ps)
    if (p) (void)hipFree(p);
  if (m->s) (void)hipStreamDestroy(m->s);
  delete m;
  return 0;
}

int aak_mlp_set_params(aak_mlp m, const float *params, const float *norm) {
  if (!m || !params) return fail(-2, "null argument");
  MLPCHK(hipMemcpyAsync(m->P, params, sizeof(float) * kNP, hipMemcpyHostToDevice, m->s));
  hipLaunchKernelGGL(k_mlp_round, dim3((kNP + kThreads - 1) / kThreads), dim3(kThreads), 0, m->s, m->P, m->Pb, m->Wt);
  MLPCHK(hipGetLastError());
  MLPCHK(hipStreamSynchronize(m->s));
  if (norm) std::memcpy(m->norm, norm, sizeof(m->norm));
  m->step = 0;
  return 0;
}

int aak_mlp_get_params(aak_mlp m, float *params, float *norm) {
  if (!m) return fail(-1, "null model");
  if (params) {
    MLPCHK(hipMemcpyAsync(params, m->P, sizeof(float) * kNP, hipMemcpyDeviceToHost, m->s));
    MLPCHK(hipStreamSynchronize(m->s));
  }
  if (norm) std::memcpy(norm, m->norm, sizeof(m->norm));
  return kNP;
}

int aak_mlp_forward(aak_mlp m, const float *X, int n, float *Y) {
  if (!m || !X || !Y || n < 0) return fail(-2, "bad argument");
  if (n == 0) return 0;
  std::lock_guard<std::mutex> lk(m->mu);
  MLPCHK(hipSetDevice(m->dev));
  if (n > m->icap) {
    if (m->iX) (void)hipFree(m->iX);
    if (m->iY) (void)hipFree(m->iY);
    m->iX = m->iY = nullptr;
    m->icap = 0;
    MLPCHK(hipMalloc(&m->iX, sizeof(float) * 4 * (size_t)n));
    MLPCHK(hipMalloc(&m->iY, sizeof(float) * 3 * (size_t)n));
    m->icap = n;
  }
  MLPCHK(hipMemcpyAsync(m->iX, X, sizeof(float) * 4 * (size_t)n, hipMemcpyHostToDevice, m->s));
  hipLaunchKernelGGL(k_mlp_forward, dim3((n + TILE - 1) / TILE), dim3(kThreads), 0, m->s, m->iX, n, m->P, m->Pb,
                     m->iY);
  MLPCHK(hipGetLastError());
  MLPCHK(hipMemcpyAsync(Y, m->iY, sizeof(float) * 3 * (size_t)n, hipMemcpyDeviceToHost, m->s));
  MLPCHK(hipStreamSynchronize(m->s));
  return 0;
}

int aak_mlp_gradient(aak_mlp m, const float *X, const float *T, int n, float *grad, double *loss) {
  if (!m || !X || !T || !grad || n <= 0) return fail(-2, "bad argument");
  MLPCHK(hipSetDevice(m->dev));
  if (n <= kPinRows && pinned_buffer(m)) {
    // the kernels read the rows from pinned host memory, each once, and leave
    // the gradient there
    int rc = grow_scratch(m, n, 0);
    if (rc) return rc;
    float *pX = m->pin, *pT = pX + 4 * (size_t)kPinRows, *pG = pT + 3 * (size_t)kPinRows, *pL = pG + kNP;
    std::memcpy(pX, X, sizeof(float) * 4 * (size_t)n);
    std::memcpy(pT, T, sizeof(float) * 3 * (size_t)n);
    launch_step(m, pX, pT, nullptr, n, 0.f, false, pG, pL);
    MLPCHK(hipGetLastError());
    MLPCHK(hipStreamSynchronize(m->s));
    std::memcpy(grad, pG, sizeof(float) * kNP);
    double ls = 0.0;
    for (int g = 0; g < grad_groups(n); g++) ls += pL[g];
    if (loss) *loss = ls / (3.0 * n);
    return 0;
  }
  int rc = grow_scratch(m, n, n);
  if (rc) return rc;
  MLPCHK(hipMemcpyAsync(m->X, X, sizeof(float) * 4 * (size_t)n, hipMemcpyHostToDevice, m->s));
  MLPCHK(hipMemcpyAsync(m->T, T, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice, m->s));
  double ls = 0.0;
  rc = train_step(m, nullptr, n, 0.f, false, &ls);
  if (rc) return rc;
  MLPCHK(hipMemcpyAsync(grad, m->grad, sizeof(float) * kNP, hipMemcpyDeviceToHost, m->s));
  MLPCHK(hipStreamSynchronize(m->s));
  if (loss) *loss = ls / (3.0 * n);
  return 0;
}

int aak_test_mlp_no_pinned(aak_mlp m, int on) {
  if (!m) return fail(-1, "null model");
  m->no_pin = on != 0;
  return 0;
}

int aak_mlp_train(aak_mlp m, const float *X, const float *T, int n, int epochs, int batch, float lr0, float lr1,
                  int seed, double *loss_per_epoch) {
  if (!m || !X || !T || n <= 0 || epochs <= 0 || batch <= 0 || batch > n) return fail(-2, "bad argument");
  MLPCHK(hipSetDevice(m->dev));
  int rc = grow_scratch(m, batch, n);
  if (rc) return rc;
  MLPCHK(hipMemcpyAsync(m->X, X, sizeof(float) * 4 * (size_t)n, hipMemcpyHostToDevice, m->s));
  MLPCHK(hipMemcpyAsync(m->T, T, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice, m->s));
  std::mt19937_64 rng((uint64_t)seed);
  std::vector<int> id(n);
  for (int i = 0; i < n; i++) id[i] = i;
  const int steps_per_epoch = n / batch;
  const long long total = (long long)epochs * steps_per_epoch;
  long long done = 0;
  for (int ep = 0; ep < epochs; ep++) {
    std::shuffle(id.begin(), id.end(), rng);
    MLPCHK(hipMemcpyAsync(m->idx, id.data(), sizeof(int) * (size_t)n, hipMemcpyHostToDevice, m->s));
    // the index upload must finish before `id` is reshuffled
    MLPCHK(hipStreamSynchronize(m->s));
    double ep_loss = 0.0;
    for (int st = 0; st < steps_per_epoch; st++, done++) {
      // cosine decay from lr0 to lr1
      const double f = 0.5 * (1.0 + cos(M_PI * (double)done / (double)total));
      const float lr = (float)(lr1 + (lr0 - lr1) * f);
      double ls = 0.0;
      rc = train_step(m, m->idx + (size_t)st * batch, batch, lr, true, (st == steps_per_epoch - 1) ? &ls : nullptr);
      if (rc) return rc;
      ep_loss = ls / (3.0 * batch);
    }
    if (loss_per_epoch) loss_per_epoch[ep] = ep_loss;
  }
  MLPCHK(hipStreamSynchronize(m->s));
  return 0;
}

int aak_mlp_set_norm(aak_mlp m, const float *norm) {
  if (!m || !norm) return fail(-2, "null argument");
  std::memcpy(m->norm, norm, sizeof(m->norm));
  return 0;
}

int aak_mlp_predict_maps(aak_mlp m, const double *pts, int n, double *maps) {
  if (!m || (n > 0 && (!pts || !maps)) || n < 0) return fail(-2, "bad argument");
  return mlp_infer(m, pts, n, maps);
}

}  // extern "C"
