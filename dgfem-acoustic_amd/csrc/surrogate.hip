// Source-to-receiver surrogate: a Fourier-feature MLP trained and queried on the GPU with this
// file's kernels (BF16 MFMA GEMMs with FP32 accumulation, fused bias/activation epilogues, loss,
// bias reduction, Adam). No reference counterpart: the reference has no learned component.
//
// Network: x in [0,1]^in (normalised source and receiver coordinates)
//   z = [sin(2 pi B x), cos(2 pi B x)]                      B: F x in, fixed, N(0, sigma^2)
//   h_1 = silu(W_1 z + b_1), h_l = silu(W_l h_{l-1} + b_l)  width w, l = 1..depth
//   y = W_o h_depth + b_o                                   out samples
// GEMM operands are BF16 (weights keep an FP32 master copy), accumulation is FP32; activations
// are rounded to BF16 once, where they become the next GEMM's operand.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/dgk_surrogate.h"
#include "handover.hpp"

// Scratch of the allocation-free forward pass (dgs_forward_noalloc): one copy per GPU, held until
// the process ends. Host code never uses this name as an address; it uses the per-device pointer
// that hipGetSymbolAddress returns (dgs::scratch_base).
static __device__ __align__(256) unsigned char scratch[16u << 20];

namespace dgs {

constexpr size_t kScratchBytes = 16u << 20;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Error : std::runtime_error {
  dgs_status st;
  Error(dgs_status s, const std::string& m) : std::runtime_error(m), st(s) {}
};

#define DGS_HIP(x)                                                                              \
  do {                                                                                          \
    hipError_t e_ = (x);                                                                        \
    if (e_ != hipSuccess) throw ::dgs::Error(DGS_ERR_DEVICE, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);  // round to nearest even (finite)
}
__device__ inline float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ inline float silu(float x) { return x * sigm(x); }
__device__ inline float dsilu(float x) {
  const float s = sigm(x);
  return s * (1.0f + x * (1.0f - s));
}

enum { EPI_STORE = 0, EPI_BIAS_ACT = 1, EPI_BIAS = 2, EPI_DACT = 3 };

struct GemmArgs {
  int M, N, K;
  int mrows;          // rows of the result that are stored (<= M)
  const uint16_t* A;  // k-contiguous: element (m, k) at A[m*lda + k]; m-contiguous: A[k*lda + m]
  int64_t lda;
  const uint16_t* B;  // k-contiguous: element (k, n) at B[n*ldb + k]; n-contiguous: B[k*ldb + n]
  int64_t ldb;
  const float* bias;  // [N]
  float* pre;         // [M][ldc] pre-activation (written by BIAS_ACT when given, read by DACT)
  uint16_t* outb;     // [M][ldc] BF16 result
  float* outf;        // [M][ldc] FP32 result
  int ldc;
};

// All products run on v_mfma_f32_16x16x32_bf16 with K ascending in steps of 32 from a zero
// accumulator, so a result does not depend on the tile that computes it. Operand lane layout (probed
// on gfx950): A lane l holds A[l%16][8(l/16)+i], B lane l holds B[8(l/16)+i][l%16]; accumulator
// register j of lane l is C[4(l/16)+j][l%16]. Operands are staged in LDS k-contiguous ([row][k]), so
// that each lane's fragment is one 16-byte read. Shapes: M, N, K multiples of 64 (checked on the
// host), operands 16-byte aligned with lda and ldb multiples of 64.
__device__ __forceinline__ f32x4 mma(const uint16_t* a, const uint16_t* b, f32x4 c) {
  const bf16x8 va = __builtin_bit_cast(bf16x8, *(const u32x4*)a), vb = __builtin_bit_cast(bf16x8, *(const u32x4*)b);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, va, c, 0, 0, 0);
}

// The B fragment goes in as the matrix core's row operand, so that a lane's four results are four
// consecutive columns of one row of C: one 8- or 16-byte access instead of four scattered ones.
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // caller's memory: 4-byte aligned
template <int EPI>
__device__ __forceinline__ void gemm_store(const GemmArgs& g, int row, int col, f32x4 v) {
  if (row >= g.mrows || col >= g.N) return;
  const int64_t o = (int64_t)row * g.ldc + col;
  if (EPI == EPI_STORE) {
    *(f32x4*)(g.outf + o) = v;
  } else if (EPI == EPI_BIAS) {
    *(f32x4a4*)(g.outf + o) = v + *(const f32x4*)(g.bias + col);
  } else {
    float r[4];
    if (EPI == EPI_BIAS_ACT) {
      const f32x4 p = v + *(const f32x4*)(g.bias + col);
      if (g.pre) *(f32x4*)(g.pre + o) = p;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = silu(p[i]);
    } else {
      const f32x4 p = *(const f32x4*)(g.pre + o);
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = v[i] * dsilu(p[i]);
    }
    *(u32x2*)(g.outb + o) = u32x2{f2bf(r[0]) | (uint32_t)f2bf(r[1]) << 16, f2bf(r[2]) | (uint32_t)f2bf(r[3]) << 16};
  }
}

// Small tile: a 32x32 piece of C per workgroup, each of 4 waves a 16x16 quarter. A network layer of a
// few hundred rows has only tens of 64x64 tiles for 256 CUs and is bound by memory latency, so the
// tile is small and K goes through LDS in chunks of 256 (or its remainder, a multiple of 64), the next
// two chunks' global loads in flight: one or two round trips cover a layer. 256 x 512 x 512: 10.1 ->
// 4.1 us forward against 64x64 tiles loaded 32 k at a time without prefetch.
// AT / BT: the operand is m- / n-contiguous in memory; a thread then loads 8 k-rows of 4 values and
// transposes them in registers.
constexpr int kSmall = 32, kChunk = 256, kSmallLd = kChunk + 8;
struct Staged {
  u32x4 v[4];
};
template <bool T>
__device__ __forceinline__ void stage_load(const uint16_t* X, int64_t ld, int r0, int k0, int kc, Staged& s) {
  const int tid = threadIdx.x;
  if (!T) {
    const uint16_t* p = X + (int64_t)(r0 + (tid >> 3)) * ld + k0 + (tid & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (64 * i < kc) s.v[i] = *(const u32x4*)(p + 64 * i);
  } else if ((tid >> 3) * 8 < kc) {
    const uint16_t* p = X + (int64_t)(k0 + (tid >> 3) * 8) * ld + r0 + (tid & 7) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x2 a = *(const u32x2*)(p + (2 * i) * ld), b = *(const u32x2*)(p + (2 * i + 1) * ld);
      s.v[i] = u32x4{a.x, a.y, b.x, b.y};  // k-rows 2i and 2i+1, values 0..3 of each
    }
  }
}
template <bool T>
__device__ __forceinline__ void stage_store(uint16_t* lds, int kc, const Staged& s) {
  const int tid = threadIdx.x;
  if (!T) {
    uint16_t* p = lds + (tid >> 3) * kSmallLd + (tid & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (64 * i < kc) *(u32x4*)(p + 64 * i) = s.v[i];
  } else if ((tid >> 3) * 8 < kc) {
    uint16_t* p = lds + (tid & 7) * 4 * kSmallLd + (tid >> 3) * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // row j of the block: k-rows 0..7
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = j < 2 ? s.v[i].x : s.v[i].y, hi = j < 2 ? s.v[i].z : s.v[i].w;
        w[i] = j & 1 ? (lo >> 16) | (hi & 0xffff0000u) : (lo & 0xffffu) | (hi << 16);
      }
      *(u32x4*)(p + j * kSmallLd) = u32x4{w[0], w[1], w[2], w[3]};
    }
  }
}

template <bool AT, bool BT, int EPI>
__device__ __forceinline__ void gemm_small(const GemmArgs& g, int bx, int by, uint16_t* sA, uint16_t* sB) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = by * kSmall, n0 = bx * kSmall;
  const int wr = (wave >> 1) * 16, wc = (wave & 1) * 16;
  const uint16_t* fa = sA + (wr + (lane & 15)) * kSmallLd + 8 * (lane >> 4);
  const uint16_t* fb = sB + (wc + (lane & 15)) * kSmallLd + 8 * (lane >> 4);
  f32x4 acc{0, 0, 0, 0};
  Staged ra[2], rb[2];
  auto load = [&](int k0, Staged& a, Staged& b) {
    if (k0 >= g.K) return;
    const int kc = min(kChunk, g.K - k0);
    stage_load<AT>(g.A, g.lda, m0, k0, kc, a);
    stage_load<BT>(g.B, g.ldb, n0, k0, kc, b);
  };
  auto chunk = [&](int k0, Staged& a, Staged& b) {
    if (k0 >= g.K) return;
    const int kc = min(kChunk, g.K - k0);
    stage_store<AT>(sA, kc, a);
    stage_store<BT>(sB, kc, b);
    __syncthreads();
    load(k0 + 2 * kChunk, a, b);
    if (kc == kChunk) {
#pragma unroll
      for (int k = 0; k < kChunk; k += 32) acc = mma(fa + k, fb + k, acc);
    } else {
      for (int k = 0; k < kc; k += 32) acc = mma(fa + k, fb + k, acc);
    }
    __syncthreads();
  };
  load(0, ra[0], rb[0]);
  load(kChunk, ra[1], rb[1]);
  for (int k0 = 0; k0 < g.K; k0 += 2 * kChunk) {
    chunk(k0, ra[0], rb[0]);
    chunk(k0 + kChunk, ra[1], rb[1]);
  }
  gemm_store<EPI>(g, m0 + wr + (lane & 15), n0 + wc + 4 * (lane >> 4), acc);
}

template <bool AT, bool BT, int EPI>
__global__ __launch_bounds__(256) void k_gemm_small(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t sA[kSmall * kSmallLd], sB[kSmall * kSmallLd];
  gemm_small<AT, BT, EPI>(g, blockIdx.x, blockIdx.y, sA, sB);
}

// Large tile: BT x BT of C per workgroup (64 or 128), each of 4 waves a quarter, both operands
// k-contiguous; K advances 64 per step through two LDS buffers with the next step's global loads in
// registers. For layers with enough tiles to fill the chip, where the small tile would read every
// operand value from L2 BT/32 times as often. Rows beyond M (N) repeat the last and are not stored.
template <int BT, int EPI>
__global__ __launch_bounds__(256) void k_gemm_large(GemmArgs g) {
  constexpr int LD = 72, W = BT / 2, F = W / 16, NL = BT / 32;
  __shared__ __attribute__((aligned(16))) uint16_t sA[2][BT * LD], sB[2][BT * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // workgroup b runs on XCD b % 8: all column tiles of a row panel go to one XCD, whose L2 then
  // fetches the panel once instead of all eight
  const int cols = (g.N + BT - 1) / BT, t = blockIdx.x / 8;
  const int m0 = (t / cols * 8 + blockIdx.x % 8) * BT, n0 = t % cols * BT;
  if (m0 >= g.M) return;
  const int wr = (wave >> 1) * W, wc = (wave & 1) * W;
  f32x4 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0, 0, 0, 0};
  const int lr = tid >> 3, lk = (tid & 7) * 8;
  const uint16_t *pa[NL], *pb[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    pa[i] = g.A + (int64_t)min(m0 + lr + 32 * i, g.M - 1) * g.lda + lk;
    pb[i] = g.B + (int64_t)min(n0 + lr + 32 * i, g.N - 1) * g.ldb + lk;
  }
  u32x4 ra[NL], rb[NL];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      ra[i] = *(const u32x4*)(pa[i] + k0);
      rb[i] = *(const u32x4*)(pb[i] + k0);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      *(u32x4*)&sA[buf][(lr + 32 * i) * LD + lk] = ra[i];
      *(u32x4*)&sB[buf][(lr + 32 * i) * LD + lk] = rb[i];
    }
  };
  load(0);
  store(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < g.K; k0 += 64, buf ^= 1) {
    if (k0 + 64 < g.K) load(k0 + 64);
#pragma unroll
    for (int k = 0; k < 64; k += 32) {
      bf16x8 a[F], b[F];
#pragma unroll
      for (int i = 0; i < F; ++i) {
        const int o = (16 * i + (lane & 15)) * LD + k + 8 * (lane >> 4);
        a[i] = __builtin_bit_cast(bf16x8, *(const u32x4*)&sA[buf][wr * LD + o]);
        b[i] = __builtin_bit_cast(bf16x8, *(const u32x4*)&sB[buf][wc * LD + o]);
      }
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    }
    if (k0 + 64 < g.K) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
      gemm_store<EPI>(g, m0 + wr + 16 * i + (lane & 15), n0 + wc + 16 * j + 4 * (lane >> 4), acc[i][j]);
}

// z[r][f] = sin(2 pi B_f . x_r), z[r][F + f] = cos(2 pi B_f . x_r), rounded to BF16.
// Row r is taken from row idx[r] (when given) or min(r, m - 1) of x, and kept in row r of `keep` (when
// given).
__global__ void k_features(int n, int m, int in, int F, const int* __restrict__ idx, const float* __restrict__ x,
                           const float* __restrict__ Bm, uint16_t* __restrict__ z, float* __restrict__ keep) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= (int64_t)n * F) return;
  const int r = (int)(i / F), f = (int)(i % F);
  const int64_t xr = idx ? idx[r] : min(r, m - 1);
  float a = 0;
  for (int d = 0; d < in; ++d) a += Bm[f * in + d] * x[xr * in + d];
  a *= 6.283185307179586f;
  z[(int64_t)r * 2 * F + f] = f2bf(sinf(a));
  z[(int64_t)r * 2 * F + F + f] = f2bf(cosf(a));
  if (keep)
    for (int d = f; d < in; d += F) keep[(int64_t)r * in + d] = x[xr * in + d];
}

// Relative squared error per sample: loss_r = w_r sum_j (y - t)^2, w_r = 1 / (n |t_r|^2);
// dY = 2 w_r (y - t) rounded to BF16. One workgroup per sample row. With idx, row r's target and
// weight are row idx[r] of the resident set, the weight divided by the batch size so that the
// minibatch loss is the mean of W_r |y_r - t_r|^2.
__global__ __launch_bounds__(256) void k_loss(int N, const float* __restrict__ y, const float* __restrict__ t,
                                              const float* __restrict__ w, const int* __restrict__ idx,
                                              uint16_t* __restrict__ dy, float* __restrict__ loss_row) {
  __shared__ float red[256];
  const int r = blockIdx.x;
  const int64_t tr = idx ? idx[r] : r;
  const float wr = idx ? w[tr] / (float)(int)gridDim.x : w[tr];
  float s = 0;
#pragma unroll 8
  for (int j = threadIdx.x; j < N; j += 256) {
    const int64_t o = (int64_t)r * N + j;
    const float d = y[o] - t[tr * N + j];
    s += d * d;
    dy[o] = f2bf(2.0f * wr * d);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss_row[r] = wr * red[0];
}

// db[n] = sum_m d[m][n] over BF16 rows, 64 columns per workgroup, m ascending. The sum is one serial
// chain per column; what it waited for was a dependent memory round trip every few rows (31 us at 256
// x 512), so 256 rows at a time come in coalesced 16-byte loads through LDS (s: 256 * 64 values).
constexpr int kSumCols = 64, kSumRows = 256;
__device__ __forceinline__ void colsum(int M, int N, const uint16_t* __restrict__ d, float* __restrict__ db, int n0,
                                       uint16_t* s) {
  const int tid = threadIdx.x;
  float sum = 0;
  for (int m0 = 0; m0 < M; m0 += kSumRows) {
    u32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int m = m0 + 32 * i + (tid >> 3);
      if (m < M) v[i] = *(const u32x4*)(d + (int64_t)m * N + n0 + (tid & 7) * 8);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (m0 + 32 * i + (tid >> 3) < M) *(u32x4*)(s + (32 * i + (tid >> 3)) * kSumCols + (tid & 7) * 8) = v[i];
    __syncthreads();
    if (tid < kSumCols) {
      const int rows = min(kSumRows, M - m0);
#pragma unroll 16
      for (int m = 0; m < rows; ++m) sum += bf2f(s[m * kSumCols + tid]);
    }
  }
  if (tid < kSumCols) db[n0 + tid] = sum;
}

// Backward pass of one layer in one launch: the workgroups take the tiles of dX = (d W) silu'(pre)
// (nx of them, none for the first layer), of dW = d^T x, and the bias gradient's column groups.
__global__ __launch_bounds__(256) void k_backward(GemmArgs dx, int nx, GemmArgs dw, int rows, float* db) {
  __shared__ __attribute__((aligned(16))) uint16_t sh[2 * kSmall * kSmallLd];
  static_assert(2 * kSmall * kSmallLd >= kSumRows * kSumCols, "the column sums share the tiles' LDS");
  const int b = blockIdx.x;
  const int ns = dw.M / kSumCols;  // the serial sums start first
  if (b < ns) {
    colsum(rows, dw.M, dw.A, db, b * kSumCols, sh);
  } else if (b < ns + nx) {
    const int t = b - ns, cols = dx.N / kSmall;
    gemm_small<false, true, EPI_DACT>(dx, t % cols, t / cols, sh, sh + kSmall * kSmallLd);
  } else {
    const int t = b - ns - nx, cols = dw.N / kSmall;
    gemm_small<true, true, EPI_STORE>(dw, t % cols, t / cols, sh, sh + kSmall * kSmallLd);
  }
}

// sum of n values into out[0] (one workgroup)
__global__ __launch_bounds__(256) void k_sum(int n, const float* __restrict__ v, float* __restrict__ out) {
  __shared__ float red[256];
  float s = 0;
  for (int i = threadIdx.x; i < n; i += 256) s += v[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// Adam with bias correction; refreshes the BF16 copy of the weights. Four parameters per thread (the
// parameter count is a multiple of 64).
__global__ void k_adam(int64_t n4, f32x4* __restrict__ p, u32x2* __restrict__ pb, const f32x4* __restrict__ g,
                       f32x4* __restrict__ m, f32x4* __restrict__ v, float lr, float b1, float b2, float c1, float c2,
                       float eps) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    const f32x4 gi = g[i];
    f32x4 mi = m[i], vi = v[i], w = p[i];
    uint32_t h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // one fixed order of rounding, whatever the compiler would contract
      mi[k] = fmaf(1 - b1, gi[k], b1 * mi[k]);
      vi[k] = fmaf(gi[k], (1 - b2) * gi[k], b2 * vi[k]);
      w[k] = w[k] - lr * (mi[k] / c1) / (sqrtf(vi[k] / c2) + eps);
      h[k] = f2bf(w[k]);
    }
    m[i] = mi;
    v[i] = vi;
    p[i] = w;
    pb[i] = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
  }
}

__global__ void k_tobf(int64_t n, const float* __restrict__ p, uint16_t* __restrict__ pb) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    pb[i] = f2bf(p[i]);
}

}  // namespace

// ------------------------------------------------------------------------------- the network
struct Net {
  dgs_config cfg{};
  int device = 0;                  // HIP device the network lives on
  int L = 0;                       // weight layers (depth hidden + output)
  std::vector<int> din, dout;      // per layer
  std::vector<int64_t> woff, boff; // offsets into the flat parameter vector
  int64_t nparam = 0;
  hipStream_t s = nullptr;
  float* P = nullptr;   // FP32 master parameters [W_1 b_1 ... W_L b_L]
  uint16_t* Pb = nullptr;  // BF16 copy (only the W parts are read)
  float* G = nullptr;   // gradients, same layout
  float* Am = nullptr;  // Adam moments
  float* Av = nullptr;
  float* Bm = nullptr;  // Fourier matrix F x in
  int64_t adam_t = 0;
  // per-batch buffers (max_batch rows)
  float *x = nullptr, *t = nullptr, *w = nullptr, *y = nullptr, *loss_row = nullptr;  // x: the last pass's rows
  uint16_t* z = nullptr;
  std::vector<uint16_t*> h;  // BF16 activations of hidden layers
  std::vector<float*> pre;   // FP32 pre-activations of hidden layers
  uint16_t *dA = nullptr, *dB = nullptr;  // ping-pong BF16 gradients of pre-activations
  // resident training set
  float *X = nullptr, *T = nullptr, *W = nullptr;
  int64_t ndata = 0;
  std::vector<void*> allocs;
  std::string err;
  dgk::SlabUser slabs;

  template <typename U>
  U* alloc(size_t n) {
    void* p = nullptr;
    DGS_HIP(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(U)));
    allocs.push_back(p);
    return (U*)p;
  }
  ~Net() {
    for (void* p : allocs) (void)hipFree(p);
    if (s) (void)hipStreamDestroy(s);
  }
};

namespace {

thread_local std::string g_err;

template <class F>
dgs_status guarded(Net* n, F&& f) {
  try {
    f();
    return DGS_OK;
  } catch (const Error& e) {
    g_err = e.what();
    if (n) n->err = e.what();
    return e.st;
  } catch (const std::exception& e) {
    g_err = e.what();
    if (n) n->err = e.what();
    return DGS_ERR_INVALID;
  }
}

void check_gemm(const GemmArgs& g) {
  if (g.M % 64 || g.N % 64 || g.K % 64 || g.M <= 0 || g.N <= 0 || g.K <= 0)
    throw Error(DGS_ERR_INVALID, "GEMM shape must be multiples of 64");
}

// C = A B with both operands k-contiguous (the forward pass): the 128-wide tile where there are two
// workgroups of it per CU (256 of them), the 64-wide one from one and a half per CU on, else the 32-wide.
// With fewer, a larger tile's workgroups stand alone on their CUs and wait for memory at every K step. us
// per layer with the 32 / 64 / 128 tile: 2560 x 512 x 512 (320 tiles of 64) 8.5 / 9.4 / 17.6, 3072 (384)
// 9.5 / 9.6 / 17.7, 4096 (512) 11.3 / 10.0 / 18.0; 12288 x 512 x 512 (384 tiles of 128) 28 / 23.1 / 23.8,
// 16384 (512) 37 / 28.5 / 25.4, 20480 (640, the last wave of them a quarter full) 45 / 34.9 / 38.7, 8192 x 1024 x
// 1024 (512) 60 / 40.9 / 33.3.
constexpr int kTiles128 = 512, kTiles64 = 384;
template <int EPI>
void gemm(Net& n, GemmArgs g) {
  check_gemm(g);
  auto rows = [&](int t) { return (g.M + t - 1) / t; };
  auto cols = [&](int t) { return (g.N + t - 1) / t; };
  auto tiles = [&](int t) { return (int64_t)rows(t) * cols(t); };
  auto grid = [&](int t) { return dim3((rows(t) + 7) / 8 * 8 * cols(t)); };  // row panels in eights, one per XCD
  if (tiles(128) >= kTiles128) hipLaunchKernelGGL((k_gemm_large<128, EPI>), grid(128), dim3(256), 0, n.s, g);
  else if (tiles(64) >= kTiles64) hipLaunchKernelGGL((k_gemm_large<64, EPI>), grid(64), dim3(256), 0, n.s, g);
  else
    hipLaunchKernelGGL((k_gemm_small<false, false, EPI>), dim3(cols(kSmall), rows(kSmall)), dim3(256), 0, n.s, g);
  DGS_HIP(hipGetLastError());
}

// Device buffers of one forward pass: inputs x [m][in] (padded to whole tiles with copies of the
// last row, or rows idx[r] of x), features z, per hidden layer l the BF16 activations h(l) and (for
// a backward pass) FP32 pre-activations pre(l), output y [m][out].
struct Pass {
  const float* x;
  int m;                       // rows of x and y
  const int* idx = nullptr;
  float* keep = nullptr;       // the rows of the pass stay here (Net::x, what dgs_forward_timed runs on)
  uint16_t* z;
  uint16_t* h[2];  // hidden layer l writes h[l % 2] (when not per layer)
  const std::vector<uint16_t*>* hl = nullptr;  // per-layer buffers (training keeps them for backward)
  const std::vector<float*>* prel = nullptr;
  float* y;
};

// Device address of `scratch` on device dev, looked up once per device with that device current.
std::mutex g_scratch_mu;
unsigned char* g_scratch[64] = {};
unsigned char* scratch_base(int dev) {
  if (dev < 0 || dev >= 64) throw Error(DGS_ERR_INVALID, "device ordinal out of range for the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[dev]) {
    int cur = 0;
    DGS_HIP(hipGetDevice(&cur));
    if (cur != dev) DGS_HIP(hipSetDevice(dev));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    DGS_HIP(e);
    g_scratch[dev] = (unsigned char*)p;
  }
  return g_scratch[dev];
}

size_t aligned256(size_t bytes) { return (bytes + 255) / 256 * 256; }

// Layout of one forward pass of mp rows in the scratch array (256-byte aligned pieces: features, two
// layers' activations and, with own_y, the outputs, which otherwise go to the caller's memory; inputs stay
// there); returns the bytes needed.
size_t scratch_layout(const Net& n, int mp, bool own_y, unsigned char* base, Pass* b) {
  const dgs_config& k = n.cfg;
  const size_t z = aligned256((size_t)mp * 2 * k.n_freq * sizeof(uint16_t));
  const size_t h = aligned256((size_t)mp * k.width * sizeof(uint16_t));
  if (base) {
    b->z = (uint16_t*)base;
    b->h[0] = (uint16_t*)(base + z);
    b->h[1] = (uint16_t*)(base + z + h);
    if (own_y) b->y = (float*)(base + z + 2 * h);
  }
  return z + 2 * h + (own_y ? aligned256((size_t)mp * k.out_dim * sizeof(float)) : 0);
}

// The networks the allocation-free pass takes, wherever y lies: those of which 64 rows of inputs,
// features, activations, FP32 pre-activations and outputs fit the scratch array. More than a pass keeps
// there: the limit is the entry point's, the same for every y.
bool scratch_takes(const Net& n) {
  const dgs_config& k = n.cfg;
  const size_t f = sizeof(float);
  return aligned256(64 * (size_t)k.in_dim * f) + scratch_layout(n, 64, true, nullptr, nullptr) +
             aligned256(64 * (size_t)k.width * f) <=
         kScratchBytes;
}

// Whether kernels on device dev write p as their own memory: not host memory, which they may have no
// mapping of, nor another GPU's, which they may have no access to.
bool own_memory(const void* p, int dev) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();  // memory that the runtime does not know
    return false;
  }
  return at.type == hipMemoryTypeDevice && at.device == dev;
}

void check_batch(const Net& n, int rows) {
  if (rows <= 0 || rows > n.cfg.max_batch || rows % 64)
    throw Error(DGS_ERR_INVALID, "batch rows must be a positive multiple of 64 up to max_batch");
}

// forward pass of `rows` rows (a multiple of 64)
void forward(Net& n, int rows, const Pass& b) {
  const int F = n.cfg.n_freq, in = n.cfg.in_dim;
  const int64_t tot = (int64_t)rows * F;
  hipLaunchKernelGGL(k_features, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, n.s, rows, b.m, in, F, b.idx, b.x,
                     n.Bm, b.z, b.keep);
  DGS_HIP(hipGetLastError());
  const uint16_t* a = b.z;
  for (int l = 0; l < n.L; ++l) {
    GemmArgs g{};
    g.M = g.mrows = rows;
    g.N = n.dout[l];
    g.K = n.din[l];
    g.A = a;
    g.lda = n.din[l];
    g.B = n.Pb + n.woff[l];
    g.ldb = n.din[l];
    g.bias = n.P + n.boff[l];
    g.ldc = n.dout[l];
    if (l + 1 < n.L) {
      g.pre = b.prel ? (*b.prel)[l] : nullptr;
      g.outb = b.hl ? (*b.hl)[l] : b.h[l % 2];
      gemm<EPI_BIAS_ACT>(n, g);
      a = g.outb;
    } else {
      g.outf = b.y;
      g.mrows = b.m;
      gemm<EPI_BIAS>(n, g);
    }
  }
}

// forward pass of `rows` rows in n.x (or rows idx[r] of the resident set); output in n.y
void forward(Net& n, int rows, const int* idx = nullptr) {
  Pass b{};
  b.x = idx ? n.X : n.x;
  b.m = rows;
  b.idx = idx;
  if (idx) b.keep = n.x;
  b.z = n.z;
  b.hl = &n.h;
  b.prel = &n.pre;
  b.y = n.y;
  forward(n, rows, b);
}

// loss and gradients of the rows in (n.x, n.t, n.w) or of rows idx[r] of the resident set;
// loss_row filled; gradients in n.G
void backward(Net& n, int rows, const int* idx = nullptr) {
  const int No = n.cfg.out_dim;
  hipLaunchKernelGGL(k_loss, dim3(rows), dim3(256), 0, n.s, No, n.y, idx ? n.T : n.t, idx ? n.W : n.w, idx, n.dA,
                     n.loss_row);
  DGS_HIP(hipGetLastError());
  uint16_t* d = n.dA;  // gradient of layer l's pre-activation, [rows][dout[l]]
  uint16_t* d2 = n.dB;
  for (int l = n.L - 1; l >= 0; --l) {
    // dW_l = d^T xin
    GemmArgs w{};
    w.M = w.mrows = n.dout[l];
    w.N = n.din[l];
    w.K = rows;
    w.A = d;
    w.lda = n.dout[l];
    w.B = l ? n.h[l - 1] : n.z;
    w.ldb = n.din[l];
    w.outf = n.G + n.woff[l];
    w.ldc = n.din[l];
    check_gemm(w);
    const int nw = (w.M / kSmall) * (w.N / kSmall);
    // d_{l-1} = (d W_l) * silu'(pre_{l-1})
    GemmArgs x{};
    int nx = 0;
    if (l) {
      x.M = x.mrows = rows;
      x.N = n.din[l];
      x.K = n.dout[l];
      x.A = d;
      x.lda = n.dout[l];
      x.B = n.Pb + n.woff[l];
      x.ldb = n.din[l];
      x.pre = n.pre[l - 1];
      x.outb = d2;
      x.ldc = n.din[l];
      check_gemm(x);
      nx = (x.M / kSmall) * (x.N / kSmall);
    }
    hipLaunchKernelGGL(k_backward, dim3(nx + nw + n.dout[l] / kSumCols), dim3(256), 0, n.s, x, nx, w, rows,
                       n.G + n.boff[l]);
    DGS_HIP(hipGetLastError());
    std::swap(d, d2);
  }
}

void upload_rows(Net& n, int rows, const float* x, const float* t, const float* w) {
  DGS_HIP(hipMemcpyAsync(n.x, x, (size_t)rows * n.cfg.in_dim * sizeof(float), hipMemcpyHostToDevice, n.s));
  if (t) DGS_HIP(hipMemcpyAsync(n.t, t, (size_t)rows * n.cfg.out_dim * sizeof(float), hipMemcpyHostToDevice, n.s));
  if (w) DGS_HIP(hipMemcpyAsync(n.w, w, (size_t)rows * sizeof(float), hipMemcpyHostToDevice, n.s));
}

void refresh_bf16(Net& n) {
  hipLaunchKernelGGL(k_tobf, dim3(1024), dim3(256), 0, n.s, n.nparam, n.P, n.Pb);
  DGS_HIP(hipGetLastError());
}

void create_impl(Net& n, const dgs_config* c) {
  if (!c) throw Error(DGS_ERR_INVALID, "NULL config");
  n.cfg = *c;
  const dgs_config& k = n.cfg;
  if (k.in_dim < 1 || k.in_dim > 64 || k.n_freq < 32 || k.n_freq % 32 || k.width < 64 || k.width % 64 ||
      k.depth < 1 || k.out_dim < 64 || k.out_dim % 64 || k.max_batch < 64 || k.max_batch % 64)
    throw Error(DGS_ERR_INVALID, "unsupported network shape (width, out_dim, max_batch multiples of 64, n_freq of 32)");
  n.L = k.depth + 1;
  DGS_HIP(hipGetDevice(&n.device));
  (void)scratch_base(n.device);  // the allocation-free forward pass's scratch address on this device
  for (int l = 0; l < n.L; ++l) {
    n.din.push_back(l ? k.width : 2 * k.n_freq);
    n.dout.push_back(l + 1 < n.L ? k.width : k.out_dim);
  }
  for (int l = 0; l < n.L; ++l) {
    n.woff.push_back(n.nparam);
    n.nparam += (int64_t)n.din[l] * n.dout[l];
    n.boff.push_back(n.nparam);
    n.nparam += n.dout[l];
  }
  DGS_HIP(hipStreamCreateWithFlags(&n.s, hipStreamNonBlocking));
  n.P = n.alloc<float>(n.nparam);
  n.Pb = n.alloc<uint16_t>(n.nparam);
  n.G = n.alloc<float>(n.nparam);
  n.Am = n.alloc<float>(n.nparam);
  n.Av = n.alloc<float>(n.nparam);
  n.Bm = n.alloc<float>((size_t)k.n_freq * k.in_dim);
  const int mb = k.max_batch;
  n.x = n.alloc<float>((size_t)mb * k.in_dim);
  n.t = n.alloc<float>((size_t)mb * k.out_dim);
  n.w = n.alloc<float>(mb);
  n.y = n.alloc<float>((size_t)mb * k.out_dim);
  n.loss_row = n.alloc<float>(mb);
  n.z = n.alloc<uint16_t>((size_t)mb * 2 * k.n_freq);
  for (int l = 0; l + 1 < n.L; ++l) {
    n.h.push_back(n.alloc<uint16_t>((size_t)mb * k.width));
    n.pre.push_back(n.alloc<float>((size_t)mb * k.width));
  }
  const int dmax = std::max(k.width, k.out_dim);
  n.dA = n.alloc<uint16_t>((size_t)mb * dmax);
  n.dB = n.alloc<uint16_t>((size_t)mb * dmax);
  // initial parameters: He-normal weights, zero biases; Fourier matrix N(0, sigma^2)
  std::mt19937_64 rng(k.seed);
  std::normal_distribution<double> nd(0.0, 1.0);
  std::vector<float> hp(n.nparam, 0.0f);
  for (int l = 0; l < n.L; ++l) {
    const double sd = std::sqrt(2.0 / n.din[l]) * (l + 1 < n.L ? 1.0 : 0.5);
    for (int64_t i = 0; i < (int64_t)n.din[l] * n.dout[l]; ++i) hp[n.woff[l] + i] = (float)(sd * nd(rng));
  }
  std::vector<float> hb((size_t)k.n_freq * k.in_dim);
  for (auto& v : hb) v = (float)(k.freq_sigma * nd(rng));
  DGS_HIP(hipMemcpy(n.P, hp.data(), hp.size() * sizeof(float), hipMemcpyHostToDevice));
  DGS_HIP(hipMemcpy(n.Bm, hb.data(), hb.size() * sizeof(float), hipMemcpyHostToDevice));
  DGS_HIP(hipMemset(n.x, 0, (size_t)mb * k.in_dim * sizeof(float)));
  DGS_HIP(hipMemset(n.Am, 0, n.nparam * sizeof(float)));
  DGS_HIP(hipMemset(n.Av, 0, n.nparam * sizeof(float)));
  DGS_HIP(hipMemset(n.G, 0, n.nparam * sizeof(float)));
  refresh_bf16(n);
  DGS_HIP(hipStreamSynchronize(n.s));
}

}  // namespace
}  // namespace dgs

using dgs::Net;

extern "C" {

struct dgs_net : Net {};

dgs_status dgs_create(const dgs_config* cfg, dgs_net** out) {
  if (!out) return DGS_ERR_INVALID;
  *out = nullptr;
  dgs_net* n = new dgs_net();
  dgs_status st = dgs::guarded(n, [&] { dgs::create_impl(*n, cfg); });
  if (st != DGS_OK) {
    delete n;
    return st;
  }
  *out = n;
  return DGS_OK;
}

dgs_status dgs_destroy(dgs_net* n) {
  delete n;
  return DGS_OK;
}

const char* dgs_last_error(const dgs_net* n) { return n ? n->err.c_str() : dgs::g_err.c_str(); }

int64_t dgs_num_params(const dgs_net* n) { return n ? n->nparam : 0; }

dgs_status dgs_get_params(dgs_net* n, float* params, float* fourier) {
  if (!n) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    DGS_HIP(hipStreamSynchronize(n->s));
    if (params) DGS_HIP(hipMemcpy(params, n->P, n->nparam * sizeof(float), hipMemcpyDeviceToHost));
    if (fourier)
      DGS_HIP(hipMemcpy(fourier, n->Bm, (size_t)n->cfg.n_freq * n->cfg.in_dim * sizeof(float), hipMemcpyDeviceToHost));
  });
}

dgs_status dgs_set_params(dgs_net* n, const float* params, const float* fourier) {
  if (!n) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    DGS_HIP(hipStreamSynchronize(n->s));
    if (params) DGS_HIP(hipMemcpy(n->P, params, n->nparam * sizeof(float), hipMemcpyHostToDevice));
    if (fourier)
      DGS_HIP(hipMemcpy(n->Bm, fourier, (size_t)n->cfg.n_freq * n->cfg.in_dim * sizeof(float), hipMemcpyHostToDevice));
    dgs::refresh_bf16(*n);
    DGS_HIP(hipMemset(n->Am, 0, n->nparam * sizeof(float)));
    DGS_HIP(hipMemset(n->Av, 0, n->nparam * sizeof(float)));
    n->adam_t = 0;
    DGS_HIP(hipStreamSynchronize(n->s));
  });
}

dgs_status dgs_forward(dgs_net* n, int rows, const float* x, float* y) {
  if (!n || rows < 0 || (rows && (!x || !y))) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    const int mb = n->cfg.max_batch, in = n->cfg.in_dim, No = n->cfg.out_dim;
    // few rows: the kernels read the inputs and write the outputs in a page-locked slab themselves (half
    // of it each), without copy commands. us with copies / without, 2048 outputs: 16 rows 139 / 47, 64 rows
    // 105 / 64, 128 rows 138 / 96, 192 rows (1.5 MB) 127 / 124, 256 (2 MB) 149 / 150, 384 187 / 210. More
    // outputs are downloaded, through the whole slab when its inputs have been read.
    constexpr size_t half = dgk::Slabs::kSlabBytes / 2, most = (size_t)2 << 20;
    static_assert(most <= half, "inputs and outputs of a pass in one slab");
    dgk::Slab slab(n->s);
    for (int r0 = 0; r0 < rows; r0 += mb) {
      const int m = std::min(mb, rows - r0);
      const int mp = (m + 63) / 64 * 64;  // whole 64-row tiles, padded with copies of the last row
      const size_t xbytes = (size_t)m * in * sizeof(float), ybytes = (size_t)m * No * sizeof(float);
      dgs::Pass b{};
      b.m = m;
      b.z = n->z;
      b.hl = &n->h;
      b.prel = &n->pre;
      b.y = n->y;
      if (xbytes <= half && slab.data()) {
        memcpy(slab.data(), x + (size_t)r0 * in, xbytes);
        b.x = (const float*)slab.data();
        b.keep = n->x;
      } else {
        DGS_HIP(hipMemcpyAsync(n->x, x + (size_t)r0 * in, xbytes, hipMemcpyHostToDevice, n->s));
        b.x = n->x;
      }
      const bool direct = ybytes <= most && slab.data();
      if (direct) b.y = (float*)(slab.data() + half);
      dgs::forward(*n, mp, b);
      float* to = y + (size_t)r0 * No;
      if (direct) {
        DGS_HIP(hipStreamSynchronize(n->s));
        memcpy(to, b.y, ybytes);
      } else {
        DGS_HIP(dgk::download({{(const char*)n->y, (char*)to, ybytes}}, n->s, slab));
      }
    }
  });
}

dgs_status dgs_forward_noalloc(dgs_net* n, int rows, const float* x, float* y) {
  if (!n || rows < 0 || (rows && (!x || !y))) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    const int in = n->cfg.in_dim, No = n->cfg.out_dim;
    dgs::Pass b{};
    if (!dgs::scratch_takes(*n))
      throw dgs::Error(DGS_ERR_INVALID, "network too wide for the 16 MiB forward scratch (64 rows do not fit)");
    const bool own_y = rows > 0 && !dgs::own_memory(y, n->device);
    // rows per pass: the largest multiple of 64 whose buffers fit the scratch array
    const int mb = 64 * (int)(dgs::kScratchBytes / dgs::scratch_layout(*n, 64, own_y, nullptr, nullptr));
    unsigned char* base = dgs::scratch_base(n->device);
    for (int r0 = 0; r0 < rows; r0 += mb) {
      const int m = std::min(mb, rows - r0);
      const int mp = (m + 63) / 64 * 64;  // whole 64-row tiles, padded with copies of the last row
      b.x = x + (size_t)r0 * in;
      b.m = m;
      b.y = y + (size_t)r0 * No;
      dgs::scratch_layout(*n, mp, own_y, base, &b);
      dgs::forward(*n, mp, b);
      if (own_y)
        DGS_HIP(hipMemcpyAsync(y + (size_t)r0 * No, b.y, (size_t)m * No * sizeof(float), hipMemcpyDefault, n->s));
    }
    DGS_HIP(hipStreamSynchronize(n->s));
  });
}

dgs_status dgs_forward_timed(dgs_net* n, int rows, int reps, double* ms_per_rep) {
  if (!n || reps < 1 || !ms_per_rep) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    dgs::check_batch(*n, rows);
    hipEvent_t a, b;
    DGS_HIP(hipEventCreate(&a));
    DGS_HIP(hipEventCreate(&b));
    DGS_HIP(hipEventRecord(a, n->s));
    for (int i = 0; i < reps; ++i) dgs::forward(*n, rows);
    DGS_HIP(hipEventRecord(b, n->s));
    DGS_HIP(hipEventSynchronize(b));
    float ms = 0;
    DGS_HIP(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *ms_per_rep = ms / reps;
  });
}

dgs_status dgs_gradients(dgs_net* n, int rows, const float* x, const float* t, const float* w, float* grad,
                         double* loss) {
  if (!n || !x || !t || !w) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    dgs::check_batch(*n, rows);
    dgs::upload_rows(*n, rows, x, t, w);
    dgs::forward(*n, rows);
    dgs::backward(*n, rows);
    std::vector<float> lr(rows);
    DGS_HIP(hipMemcpyAsync(lr.data(), n->loss_row, rows * sizeof(float), hipMemcpyDeviceToHost, n->s));
    if (grad) DGS_HIP(hipMemcpyAsync(grad, n->G, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->s));
    DGS_HIP(hipStreamSynchronize(n->s));
    if (loss) {
      double s = 0;
      for (float v : lr) s += v;
      *loss = s;
    }
  });
}

dgs_status dgs_set_data(dgs_net* n, int64_t rows, const float* x, const float* t, const float* w) {
  if (!n || rows < 1 || !x || !t || !w) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    DGS_HIP(hipStreamSynchronize(n->s));
    for (void* p : {(void*)n->X, (void*)n->T, (void*)n->W}) {
      if (!p) continue;
      auto it = std::find(n->allocs.begin(), n->allocs.end(), p);
      if (it != n->allocs.end()) n->allocs.erase(it);
      DGS_HIP(hipFree(p));
    }
    n->X = n->alloc<float>((size_t)rows * n->cfg.in_dim);
    n->T = n->alloc<float>((size_t)rows * n->cfg.out_dim);
    n->W = n->alloc<float>(rows);
    DGS_HIP(hipMemcpy(n->X, x, (size_t)rows * n->cfg.in_dim * sizeof(float), hipMemcpyHostToDevice));
    DGS_HIP(hipMemcpy(n->T, t, (size_t)rows * n->cfg.out_dim * sizeof(float), hipMemcpyHostToDevice));
    DGS_HIP(hipMemcpy(n->W, w, rows * sizeof(float), hipMemcpyHostToDevice));
    n->ndata = rows;
  });
}

dgs_status dgs_train(dgs_net* n, int steps, int batch, float lr, uint64_t seed, float* losses) {
  if (!n || steps < 0) return DGS_ERR_INVALID;
  return dgs::guarded(n, [&] {
    dgs::check_batch(*n, batch);
    if (!n->ndata) throw dgs::Error(DGS_ERR_INVALID, "no training data (dgs_set_data)");
    if (steps == 0) return;
    // minibatch indices: each epoch is a seeded permutation of the rows
    std::mt19937_64 rng(seed);
    std::vector<int> idx((size_t)steps * batch), perm(n->ndata);
    for (int64_t i = 0; i < n->ndata; ++i) perm[i] = (int)i;
    size_t pos = perm.size();
    for (auto& v : idx) {
      if (pos == perm.size()) {
        std::shuffle(perm.begin(), perm.end(), rng);
        pos = 0;
      }
      v = perm[pos++];
    }
    int* didx = nullptr;
    float* dloss = nullptr;
    DGS_HIP(hipMalloc(&didx, idx.size() * sizeof(int)));
    DGS_HIP(hipMalloc(&dloss, steps * sizeof(float)));
    try {
      DGS_HIP(hipMemcpyAsync(didx, idx.data(), idx.size() * sizeof(int), hipMemcpyHostToDevice, n->s));
      const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
      for (int it = 0; it < steps; ++it) {
        const int* bi = didx + (size_t)it * batch;
        dgs::forward(*n, batch, bi);
        dgs::backward(*n, batch, bi);
        hipLaunchKernelGGL(dgs::k_sum, dim3(1), dim3(256), 0, n->s, batch, n->loss_row, dloss + it);
        ++n->adam_t;
        const float c1 = 1.0f - std::pow(b1, (float)n->adam_t), c2 = 1.0f - std::pow(b2, (float)n->adam_t);
        hipLaunchKernelGGL(dgs::k_adam, dim3(2048), dim3(256), 0, n->s, n->nparam / 4, (dgs::f32x4*)n->P,
                           (dgs::u32x2*)n->Pb, (const dgs::f32x4*)n->G, (dgs::f32x4*)n->Am, (dgs::f32x4*)n->Av, lr, b1,
                           b2, c1, c2, eps);
        DGS_HIP(hipGetLastError());
      }
      if (losses) DGS_HIP(hipMemcpyAsync(losses, dloss, steps * sizeof(float), hipMemcpyDeviceToHost, n->s));
      DGS_HIP(hipStreamSynchronize(n->s));
    } catch (...) {
      (void)hipFree(didx);
      (void)hipFree(dloss);
      throw;
    }
    DGS_HIP(hipFree(didx));
    DGS_HIP(hipFree(dloss));
  });
}

}  // extern "C"
