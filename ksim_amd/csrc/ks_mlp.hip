// MLP forward and backward on the gfx950 matrix cores: fused GEMM + bias + activation kernels per layer (mlp_layer_kernel: bf16 on
// v_mfma_f32_32x32x16_bf16, 8 consecutive k per lane; cut_layer_kernel: fp32 on the same instruction, every value in three bf16 parts) and
// whole-network kernels.  Output fragment layout (both): lane l, register r -> row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#include "ks_common.h"
#include "ks_cut.h"
#include "ks_philox.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <cstdlib>
#include <vector>

namespace ks {

typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kBM = 128, kBN = 128;  // kBM: the largest row tile

// FAST: the result is rounded to bf16 right away, so the hardware exponential (abs. error ~1e-7 near zero) is
// exact enough; the fp32 path keeps expm1f.
template <int ACT, bool FAST>
__device__ __forceinline__ float activate(float x) {
  if (ACT == KS_ACT_ELU) {
    // exp(x) - 1 >= x everywhere, so ELU is the median of (x, 0, exp(x) - 1): one instruction instead of compare + select
    if (FAST) return __builtin_amdgcn_fmed3f(x, 0.f, __expf(x) - 1.0f);
    return x > 0.f ? x : expm1f(x);
  }
  if (ACT == KS_ACT_RELU) return fmaxf(x, 0.f);
  if (ACT == KS_ACT_TANH) return tanhf(x);
  if (ACT == KS_ACT_GELU) {  // tanh form (jax.nn.gelu's default): 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    // tanh(u) = 1 - 2 / (exp(2u) + 1); the hardware exponential is exact enough when the result is rounded to bf16
    const float t = FAST ? 1.f - 2.f / (__expf(2.f * u) + 1.f) : tanhf(u);
    return 0.5f * x * (1.f + t);
  }
  return x;
}

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }


// First layer: VEC consecutive fp32 inputs of row m starting at column k (zero beyond the real width or batch),
// converted to T and packed into one 16-byte register vector.
template <typename T, int VEC>
__device__ __forceinline__ u32x4 load_first(const float* __restrict__ x, int64_t m, int64_t M, int64_t ldx, int k,
                                            int Kreal) {
  float f[VEC];
  if (m < M && (ldx & 3) == 0 && k + VEC <= Kreal) {  // whole vector inside a 16-byte aligned row: wide loads
    const float4* p4 = reinterpret_cast<const float4*>(x + m * ldx + k);
#pragma unroll
    for (int e = 0; e < VEC / 4; ++e) {
      const float4 t = p4[e];
      f[4 * e] = t.x; f[4 * e + 1] = t.y; f[4 * e + 2] = t.z; f[4 * e + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < VEC; ++e) f[e] = (m < M && k + e < Kreal) ? x[m * ldx + k + e] : 0.f;
  }
  unsigned w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned lo = __builtin_bit_cast(unsigned short, (__bf16)f[2 * e]);
    const unsigned hi = __builtin_bit_cast(unsigned short, (__bf16)f[2 * e + 1]);
    w[e] = lo | (hi << 16);
  }
  return u32x4{w[0], w[1], w[2], w[3]};
}

// T = math/storage type of activations and weights (__bf16).
// FIRST: x is the caller's unpadded fp32 input (row stride ldx = in_dim).
// LAST: y is the caller's unpadded fp32 output (row stride ldy = out_dim).
// BM: rows per workgroup (128, or 64 for small batches so that the grid still covers every CU twice).
// The K loop is software-pipelined: the global loads of slice k+1 are issued into registers before the MFMAs
// of slice k run out of LDS, so HBM/L2 latency overlaps the matrix-core work.
template <typename T, bool FIRST, bool LAST, int ACT, int BM, int BN, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void mlp_layer_kernel(int64_t M, int K /*padded to BK*/, int Kreal, int Nreal,
                                                        const void* __restrict__ xin, int64_t ldx,
                                                        const T* __restrict__ W /*(Np, K)*/,
                                                        const float* __restrict__ bias /*(Np)*/,
                                                        void* __restrict__ yout, int64_t ldy) {
  static_assert(sizeof(T) == 2, "fp32 layers have a kernel of their own");
  constexpr int BK = 64;                 // elements of K per slice
  constexpr int PAD = 8;                 // keeps 16-byte row alignment and spreads LDS banks
  constexpr int VEC = 16 / sizeof(T);    // elements per 16-byte load
  constexpr int NT = 64 * WAVES_M * WAVES_N;    // threads per workgroup
  constexpr int A_VECS = BM * BK / VEC / NT;    // 16-byte loads per thread for the A slice
  constexpr int B_VECS = BN * BK / VEC / NT;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;  // output block of one wavefront
  constexpr int MI = WM / 32, NI = WN / 32;     // 32 x 32 MFMA tiles per wavefront
  static_assert(A_VECS >= 1 && B_VECS >= 1 && MI >= 1 && NI >= 1, "tile too small for the workgroup");
  extern __shared__ __attribute__((aligned(16))) unsigned char mlp_lds[];
  T (*As)[BK + PAD] = reinterpret_cast<T (*)[BK + PAD]>(mlp_lds);
  T (*Bs)[BK + PAD] = reinterpret_cast<T (*)[BK + PAD]>(mlp_lds + sizeof(T) * BM * (BK + PAD));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  // Workgroup l of a launch runs on XCD l % 8, each with its own L2: the column tiles of one row tile go to one XCD, one after the
  // other, so that its rows are fetched once.  Row tiles past the last whole eight follow in plain order.
  // Slices of the reduction (weight gradients) of 512 rows or more: all tiles of a slice, which read the same rows of both operands, go to one
  // XCD (65536 x 512 x 512: 70 -> 62 us).  Shorter ones are over before the rows come round again.
  int64_t m_tile = blockIdx.x;
  int n_tile = blockIdx.y, z = blockIdx.z;
  if (gridDim.z % 8 == 0 && K >= 512 * (int)gridDim.z) {
    const unsigned l = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, tiles = gridDim.x * gridDim.y, q = l >> 3, zq = q / tiles;
    z = (int)(zq * 8 + (l & 7));
    n_tile = (int)((q - zq * tiles) / gridDim.x);
    m_tile = (q - zq * tiles) % gridDim.x;
  } else if (gridDim.y > 1) {
    const int64_t l = (int64_t)blockIdx.y * gridDim.x + blockIdx.x, whole = (int64_t)(gridDim.x & ~7u) * gridDim.y;
    const int64_t q = l < whole ? l >> 3 : l - whole;
    n_tile = (int)(q % gridDim.y);
    m_tile = l < whole ? (q / gridDim.y) * 8 + (l & 7) : (int64_t)(gridDim.x & ~7u) + q / gridDim.y;
  }
  const int64_t m0 = m_tile * BM;
  const int n0 = n_tile * BN;
  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  constexpr int VPR = BK / VEC;  // 16-byte vectors per tile row
  u32x4 ra[A_VECS], rb[B_VECS];
  // global -> registers for the K slice starting at KS_K0 (kept as a macro so the register arrays never have
  // their address taken)
#define KS_FETCH(KS_K0)                                                                                        \
  {                                                                                                            \
    _Pragma("unroll") for (int c = 0; c < A_VECS; ++c) {                                                       \
      const int v = tid + NT * c, row = v / VPR, col = (v % VPR) * VEC;                                        \
      const int64_t m = m0 + row;                                                                              \
      if constexpr (FIRST) {                                                                                   \
        ra[c] = load_first<T, VEC>((const float*)xin, m, M, ldx, (KS_K0) + col, Kreal);                        \
      } else {                                                                                                 \
        ra[c] = (m < M) ? *reinterpret_cast<const u32x4*>((const T*)xin + m * ldx + (KS_K0) + col)             \
                        : u32x4{0u, 0u, 0u, 0u};                                                              \
      }                                                                                                        \
    }                                                                                                          \
    _Pragma("unroll") for (int c = 0; c < B_VECS; ++c) {                                                       \
      const int v = tid + NT * c, row = v / VPR, col = (v % VPR) * VEC;                                        \
      rb[c] = *reinterpret_cast<const u32x4*>(W + (int64_t)(n0 + row) * K + (KS_K0) + col);                    \
    }                                                                                                          \
  }

  // gridDim.z > 1: this workgroup reduces only its slice of K and writes partial sums to its own copy of the
  // output (LAST outputs only; the caller adds the copies up in a fixed order)
  const int kslice = (K / BK + (int)gridDim.z - 1) / (int)gridDim.z * BK;  // whole stages; the last slices may be shorter or empty
  const int kbeg = min(K, z * kslice), kend = min(K, kbeg + kslice);
  KS_FETCH(min(kbeg, K - BK))
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
#pragma unroll
    for (int c = 0; c < A_VECS; ++c) {
      const int v = tid + NT * c, row = v / VPR, col = (v % VPR) * VEC;
      *reinterpret_cast<u32x4*>(&As[row][col]) = ra[c];
    }
#pragma unroll
    for (int c = 0; c < B_VECS; ++c) {
      const int v = tid + NT * c, row = v / VPR, col = (v % VPR) * VEC;
      *reinterpret_cast<u32x4*>(&Bs[row][col]) = rb[c];
    }
    __syncthreads();
    // Next slice in flight while the matrix cores work on this one.  The fetch is unconditional (the last pass
    // re-reads its own slice) so that the register arrays are plain loop-carried values.
    const int kn = k0 + BK < kend ? k0 + BK : k0;
    KS_FETCH(kn)
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      bf16x8 af[MI], bfr[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = *(const bf16x8*)&As[wm * WM + i * 32 + (lane & 31)][kk + (lane >> 5) * 8];
#pragma unroll
      for (int j = 0; j < NI; ++j) bfr[j] = *(const bf16x8*)&Bs[wn * WN + j * 32 + (lane & 31)][kk + (lane >> 5) * 8];
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
#undef KS_FETCH
  // ---- epilogue: bias + activation + store
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int col = n0 + wn * WN + j * 32 + (lane & 31);
      const float b = z == 0 ? bias[col] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm * WM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row >= M) continue;
        const float v = acc[i][j][r] + b;
        if (LAST) {
          if (col < Nreal) ((float*)yout)[(int64_t)z * M * ldy + row * ldy + col] = v;
        } else {
          ((T*)yout)[row * ldy + col] = to_bf16(activate<ACT, true>(v));
        }
      }
    }
}

// ---------------------------------------------------------------- fp32 products on the bf16 matrix instruction (cut_bf16)
template <int MI, int NJ>
__device__ __forceinline__ void mma_bf16(const bf16x8 (&a)[MI], const bf16x8 (&b)[NJ], f32x16 (&acc)[MI][NJ]) {
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
}

// The order of the eight is part of a result's bits: every kernel that multiplies cut values goes through here, 16 k after 16 k.
template <int MI, int NJ>
__device__ __forceinline__ void mma_cut(const bf16x8 (&a)[3][MI], const bf16x8 (&b)[3][NJ], f32x16 (&acc)[MI][NJ], f32x16 (&low)[MI][NJ]) {
  mma_bf16(a[2], b[1], low);
  mma_bf16(a[1], b[2], low);
  mma_bf16(a[2], b[0], low);
  mma_bf16(a[0], b[2], low);
  mma_bf16(a[1], b[1], low);
  mma_bf16(a[1], b[0], low);
  mma_bf16(a[0], b[1], low);
  mma_bf16(a[0], b[0], acc);
}

template <int ACT, int MI>
__device__ __forceinline__ void activate_tiles(f32x16 (&acc)[MI][2]) {
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = activate<ACT, false>(acc[i][j][r]);
}

// Four neighbouring floats at any address of a float: rows of an odd width start at one, and a 16-byte load needs no more than that.  Against
// four loads of a float each: 102400 x 475 -> 128 186 -> 155 us, its weight gradient 155 -> 140 (rows of a multiple of four: 106 and 93; what
// remains is that a row's 128 bytes lie in two cache lines).
struct __attribute__((packed, aligned(4))) Float4Any { float x, y, z, w; };
__device__ __forceinline__ float4 load4_any(const float* p) {
  const Float4Any v = *reinterpret_cast<const Float4Any*>(p);
  return float4{v.x, v.y, v.z, v.w};
}

// fp32 layers: y = act(x W^T + b) on BM x 128 tiles, four wavefronts of BM / 2 x 64 each, operands cut on their way to LDS.  A stage is
// 32 k: thread t cuts the fragment q = t % 4 of rows t / 4 + 64 r, k = 16 (q / 2) + 4 (q % 2) + {0..3, 8..11}, so that four neighbouring
// lanes read 128 bytes of a row in two loads.  A part's fragments lie [q][row] with two spare ones per q: neighbouring lanes write into
// different banks and a matrix instruction's operand is one 16-byte read per lane.  The next stage's rows are requested before the
// products and stay in flight over the barriers.  BM = 128: two workgroups per CU, one cutting while the other multiplies.
//   102400 x 128 -> 512: 163 us on the fp32 instruction, 127 here; 102400 x 512 -> 128: 139, 110 here (122 TFLOP/s; the fp32 instruction's
//   time alone is 87 us), of 53 in matrix instructions and 45 of memory traffic; relative error against 64 bits 2.0e-7 -> 0.64e-7 and
//   4.0e-7 -> 1.2e-7
// Every fp32 kernel of a single layer starts from the bias and adds the products in one order (mma_cut), so a row's numbers do not depend
// on the batch it comes in or the kernel that batch takes.
// x (M, Kreal) with row stride ldx; K: Kreal padded to 32 (W's stride; its padding is zero).  Columns of y past Nreal are not written when y is
// the caller's (LAST); otherwise y is as wide as the padded layer.  gridDim.z > 1 (LAST): slice z of the reduction goes to its own copy
// of the output.
template <int BM, bool VA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BM == 128 ? 2 : 3, BM == 128 ? 2 : 3)))
void cut_layer_kernel(int64_t M, int K, int Kreal, int Nreal, const float* __restrict__ x, int64_t ldx, const float* __restrict__ W,
                      const float* __restrict__ bias, float* __restrict__ y, int64_t ldy, int act) {
  constexpr int LA = BM + 2, LB = 128 + 2, MI = BM / 64, AV = BM / 64;
  __shared__ u32x4 As[3 * 4 * LA], Bs[3 * 4 * LB];  // [part][q][row]
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, c = lane & 31, h = lane >> 5;
  // Workgroup l of a launch runs on XCD l % 8, each with its own L2: the column tiles of one row tile go to one XCD, one after the
  // other, so that its rows are fetched once (102400 x 128 -> 512 reads 64 MB instead of 210).  Row tiles past the last whole eight follow in
  // plain order.
  // Slices of the reduction, 512 rows or more: all tiles of a slice go to one XCD.
  unsigned m_tile = blockIdx.x, n_tile = blockIdx.y;
  int z = blockIdx.z;
  if (gridDim.z % 8 == 0 && K >= 512 * (int)gridDim.z) {
    const unsigned l = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, tiles = gridDim.x * gridDim.y, q = l >> 3, zq = q / tiles;
    z = (int)(zq * 8 + (l & 7));
    n_tile = (q - zq * tiles) / gridDim.x;
    m_tile = (q - zq * tiles) % gridDim.x;
  } else if (gridDim.y > 1) {  // tiles of an output that fits the card's memory: 32 bits
    const unsigned l = blockIdx.y * gridDim.x + blockIdx.x, rows8 = gridDim.x & ~7u, whole = rows8 * gridDim.y;
    const unsigned q = l < whole ? l >> 3 : l - whole, d = q / gridDim.y;
    n_tile = q - d * gridDim.y;
    m_tile = l < whole ? d * 8 + (l & 7) : rows8 + d;
  }
  const int64_t m0 = (int64_t)m_tile * BM;
  const int n0 = (int)n_tile * 128;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * 64;
  f32x16 acc[MI][2], low[MI][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float b = z == 0 ? bias[n0 + wn + 32 * j + c] : 0.f;  // padded to whole tiles
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) { acc[i][j][r] = b; low[i][j][r] = 0.f; }
  }
  const int kslice = (K / 32 + (int)gridDim.z - 1) / (int)gridDim.z * 32;  // whole stages; the last slices may be shorter or empty
  const int kbeg = min(K, z * kslice), stages = min(kslice, K - kbeg) / 32;
  // rows past the batch repeat the last one, their results are dropped
  const int lrow = t >> 2, q = t & 3, lk = kbeg + 16 * (q >> 1) + 4 * (q & 1);
  const float* pa[AV];
#pragma unroll
  for (int r = 0; r < AV; ++r) {
    const int64_t m = m0 + lrow + 64 * r;
    pa[r] = x + (m < M ? m : M - 1) * ldx;
  }
  const float* pb = W + (int64_t)(n0 + lrow) * K + lk;
  const int64_t b64 = (int64_t)64 * K;
  float4 ra[AV][2], rb[2][2];
  auto fetch = [&](int n) __attribute__((always_inline)) {
    const bool inside = kbeg + 32 * (n + 1) <= Kreal;  // the whole stage
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = lk + 32 * n + 8 * u, left = Kreal - k;  // steps of the row still inside the input (VA: a multiple of four)
#pragma unroll
      for (int r = 0; r < AV; ++r) {
        const float* at = pa[r] + k;
        ra[r][u] = float4{0.f, 0.f, 0.f, 0.f};
        if (VA) {
          if (left > 0) ra[r][u] = *reinterpret_cast<const float4*>(at);
        } else if (inside) {
          ra[r][u] = load4_any(at);
        } else {
          if (left > 0) ra[r][u].x = at[0];
          if (left > 1) ra[r][u].y = at[1];
          if (left > 2) ra[r][u].z = at[2];
          if (left > 3) ra[r][u].w = at[3];
        }
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) rb[r][u] = *reinterpret_cast<const float4*>(pb + r * b64 + 32 * n + 8 * u);
    }
  };
  auto cut = [&](const float4 (&f)[2], u32x4* to, int stride) __attribute__((always_inline)) {
    const float v[8] = {f[0].x, f[0].y, f[0].z, f[0].w, f[1].x, f[1].y, f[1].z, f[1].w};
    u32x4 part[3];
    cut_bf16<3>(v, part);
#pragma unroll
    for (int p = 0; p < 3; ++p) to[p * 4 * stride] = part[p];
  };
  if (stages > 0) fetch(0);
  for (int n = 0; n < stages; ++n) {
    if (n > 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // LDS only: the requested rows stay in flight
#pragma unroll
    for (int r = 0; r < AV; ++r) cut(ra[r], As + q * LA + lrow + 64 * r, LA);
#pragma unroll
    for (int r = 0; r < 2; ++r) cut(rb[r], Bs + q * LB + lrow + 64 * r, LB);
    if (n + 1 < stages) fetch(n + 1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 fa[3][MI], fb[3][2];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[p][i] = __builtin_bit_cast(bf16x8, As[(p * 4 + 2 * s + h) * LA + wm + 32 * i + c]);
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[p][j] = __builtin_bit_cast(bf16x8, Bs[(p * 4 + 2 * s + h) * LB + wn + 32 * j + c]);
      }
      mma_cut(fa, fb, acc, low);
    }
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = join_cut(acc[i][j][r], low[i][j][r]);
  switch (act) {
    case KS_ACT_ELU: activate_tiles<KS_ACT_ELU>(acc); break;
    case KS_ACT_RELU: activate_tiles<KS_ACT_RELU>(acc); break;
    case KS_ACT_TANH: activate_tiles<KS_ACT_TANH>(acc); break;
    case KS_ACT_GELU: activate_tiles<KS_ACT_GELU>(acc); break;
    default: break;
  }
  // one row of the tile after the other: uniform steps from one address per lane
  const int64_t row0 = m0 + wm + 4 * h;
  const int col = n0 + wn + c;
  float* out = y + ((int64_t)z * M + row0) * ldy + col;
  const bool on0 = col < Nreal, on1 = col + 32 < Nreal, whole = m0 + BM <= M;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int down = 32 * i + 8 * (r >> 2) + (r & 3);
      const bool on = whole || row0 + down < M;
      float* o = out + down * ldy;
      if (on && on0) o[0] = acc[i][0][r];
      if (on && on1) o[32] = acc[i][1][r];
    }
}

// ---------------------------------------------------------------- fp32 layers over few rows
// A layer of an fp32 network over few rows (sgemm_small_kernel): the whole-network kernel would give 32 rows to one CU, whose matrix rate then takes 80 us
// for three layers of 512.  A wavefront owns a 32 x 32 tile of the layer with both operands straight from memory in registers (weights in
// fragment order, eight groups of 8 k ahead) and the layers are launches of their own: rows x width / 1024 wavefronts over the chip.
// SHARE wavefronts cut the reduction of a narrow output layer as the whole-network kernel's do (same parts, same order of the sum).
// blockIdx.z picks one of two networks over the same rows (actor and critic).
struct SmallLayer {
  const float* x;
  int64_t ldx;
  int Kreal, nk, nt, Nreal, act, vec;
  const u32x4* Wp;
  const float* bp;
  float* y;
  int64_t ldy;
};

// A single fp32 layer over few rows: the same tiles, products of cut values (mma_cut) in cut_layer_kernel's order.  Bound by latency: 4096 x
// 128 -> 40: 11.1 -> 6.9 us.
__global__ __launch_bounds__(256) void cut_small_kernel(int64_t M, SmallLayer p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 31, h = lane >> 5;
  const int j = (int)blockIdx.x * 4 + wave;
  if (j >= p.nt) return;
  const int64_t m0 = (int64_t)blockIdx.y * 32, m = m0 + c < M ? m0 + c : M - 1;  // rows past the batch repeat the last one
  f32x16 acc[1][1], low[1][1];
  const float b = p.bp[32 * j + c];
#pragma unroll
  for (int r = 0; r < 16; ++r) { acc[0][0][r] = b; low[0][0][r] = 0.f; }
  const float* xr = p.x + m * p.ldx;
  const u32x4* wr = p.Wp + (int64_t)j * p.nk * 64 + lane;
  typedef __attribute__((ext_vector_type(4))) float f32x4v;
  const int steps = (p.nk + 1) / 2, last = p.Kreal - 1;  // a step is two groups of 8 k
  constexpr int PF = 4;
  f32x4v xf[PF][2], wf[PF][2];
  // groups past the end and columns past the row's end load something valid and count as zero
  auto request = [&](int u, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int g = 2 * s + e < p.nk ? 2 * s + e : p.nk - 1, k = 8 * g + 4 * h;
      if (p.vec) xf[u][e] = *reinterpret_cast<const f32x4v*>(xr + (k < last - 3 ? k : last - 3));
      else xf[u][e] = f32x4v{xr[k < last ? k : last], xr[k + 1 < last ? k + 1 : last], xr[k + 2 < last ? k + 2 : last], xr[k + 3 < last ? k + 3 : last]};
      wf[u][e] = __builtin_bit_cast(f32x4v, wr[(int64_t)g * 64]);
    }
  };
  auto step = [&](int u, int s) __attribute__((always_inline)) {
    float xv[8], wv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 16 * s + 8 * (e >> 2) + 4 * h + (e & 3);
      xv[e] = k < p.Kreal ? xf[u][e >> 2][e & 3] : 0.f;
      wv[e] = k < p.Kreal ? wf[u][e >> 2][e & 3] : 0.f;
    }
    u32x4 xp[3], wp[3];
    cut_bf16<3>(xv, xp);
    cut_bf16<3>(wv, wp);
    bf16x8 a[3][1], w[3][1];
#pragma unroll
    for (int q = 0; q < 3; ++q) { a[q][0] = __builtin_bit_cast(bf16x8, xp[q]); w[q][0] = __builtin_bit_cast(bf16x8, wp[q]); }
    mma_cut(a, w, acc, low);
  };
#pragma unroll
  for (int u = 0; u < PF; ++u) request(u, u);
  int s = 0;
  for (; s + PF <= steps; s += PF)
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      step(u, s + u);
      request(u, s + u + PF);
    }
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (s + u < steps) step(u, s + u);
  const int col = 32 * j + c;
  if (col >= p.Nreal) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t row = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
    if (row < M) p.y[row * p.ldy + col] = join_cut(acc[0][0][r], low[0][0][r]);
  }
}

template <int SHARE>
__global__ __launch_bounds__(256) void sgemm_small_kernel(int64_t M, SmallLayer p0, SmallLayer p1) {
  constexpr int TPW = 4 / SHARE;  // tiles per workgroup
  __shared__ float red[SHARE > 1 ? 4 : 1][SHARE > 1 ? 1024 : 1];
  const SmallLayer& p = blockIdx.z == 0 ? p0 : p1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 31, h = lane >> 5;
  const int part = wave % SHARE, tile = (int)blockIdx.x * TPW + wave / SHARE;
  const bool on = tile < p.nt;
  const int j = on ? tile : 0;
  const int64_t m0 = (int64_t)blockIdx.y * 32, m = m0 + c < M ? m0 + c : M - 1;  // rows past the batch repeat the last one
  const int per = (p.nk + SHARE - 1) / SHARE, g0 = part * per, g1 = on ? (g0 + per < p.nk ? g0 + per : p.nk) : 0;
  f32x16 acc;
  const float b = part == 0 ? p.bp[32 * j + c] : 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = b;
  const float* xr = p.x + m * p.ldx;
  const u32x4* wr = p.Wp + (int64_t)j * p.nk * 64 + lane;
  typedef __attribute__((ext_vector_type(4))) float f32x4v;
  // groups past the end and columns past the row's end load something valid; the columns count as zero, the groups are not used
  auto load_x = [&](int g) __attribute__((always_inline)) {
    const int k = 8 * g + 4 * h, last = p.Kreal - 1;
    f32x4v v;
    if (p.vec) v = *reinterpret_cast<const f32x4v*>(xr + (k < last - 3 ? k : last - 3));
    else v = f32x4v{xr[k < last ? k : last], xr[k + 1 < last ? k + 1 : last], xr[k + 2 < last ? k + 2 : last], xr[k + 3 < last ? k + 3 : last]};
    return v;
  };
  auto mma = [&](int g, f32x4v xv, f32x4v wv) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(8 * g + 4 * h + e < p.Kreal ? xv[e] : 0.f, wv[e], acc, 0, 0, 0);
  };
  constexpr int PF = 8;
  f32x4v xf[PF], wf[PF];
  if (g0 < g1) {
    const int gl = g1 - 1;
    auto request = [&](int u, int g) __attribute__((always_inline)) {
      g = g < gl ? g : gl;
      xf[u] = load_x(g);
      wf[u] = __builtin_bit_cast(f32x4v, wr[(int64_t)g * 64]);
    };
#pragma unroll
    for (int u = 0; u < PF; ++u) request(u, g0 + u);
    int g = g0;
    for (; g + PF <= g1; g += PF)
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        mma(g + u, xf[u], wf[u]);
        request(u, g + u + PF);
      }
#pragma unroll
    for (int u = 0; u < PF; ++u)
      if (g + u < g1) mma(g + u, xf[u], wf[u]);
  }
  if constexpr (SHARE > 1) {
    if (part > 0)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave][r * 64 + lane] = acc[r];
    __syncthreads();
    if (part > 0) return;
    for (int q = 1; q < SHARE; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += red[wave + q][r * 64 + lane];
  }
  const int col = 32 * j + c;
  if (!on || col >= p.Nreal) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t row = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
    if (row >= M) continue;
    float v = acc[r];
    switch (p.act) {
      case KS_ACT_ELU: v = activate<KS_ACT_ELU, false>(v); break;
      case KS_ACT_RELU: v = activate<KS_ACT_RELU, false>(v); break;
      case KS_ACT_TANH: v = activate<KS_ACT_TANH, false>(v); break;
      case KS_ACT_GELU: v = activate<KS_ACT_GELU, false>(v); break;
      default: break;
    }
    p.y[row * p.ldy + col] = v;
  }
}

// ---------------------------------------------------------------- matrix-core yardstick
// Nothing but 32x32x16 bf16 MFMAs on register operands: eight independent accumulator tiles per wavefront (the fused
// kernel's own count), no loads, no LDS, no epilogue.  What this loop reaches is the most any kernel built on that
// instruction can reach on this part at the clock it sustains under matrix load.  Per workgroup: stamps[2 b] = shader
// clock cycles of the loop, stamps[2 b + 1] = the same interval on the constant 100 MHz counter.
__global__ __launch_bounds__(256) void mfma_yardstick_kernel(int iters, float* __restrict__ out, long long* __restrict__ stamps) {
  f32x16 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
  bf16x8 a, b;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // operands that differ between lanes and are neither zero nor all equal
    const unsigned h = (threadIdx.x * 8u + e + blockIdx.x * 977u) * 2654435761u;
    a[e] = (__bf16)(((float)(h >> 8) / 8388608.0f) - 1.0f);
    b[e] = (__bf16)(((float)((h * 40503u) >> 8) / 8388608.0f) - 1.0f);
  }
  const long long c0 = clock64(), w0 = wall_clock64();
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i], 0, 0, 0);
  }
  const long long c1 = clock64(), w1 = wall_clock64();
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum += acc[i][r];
  out[(int64_t)blockIdx.x * 256 + threadIdx.x] = sum;
  if (stamps && threadIdx.x == 0) {
    stamps[2 * (int64_t)blockIdx.x] = c1 - c0;
    stamps[2 * (int64_t)blockIdx.x + 1] = w1 - w0;
  }
}

// ---------------------------------------------------------------- whole network in one kernel
// A 512-thread workgroup keeps a BM-row tile of activations in LDS for the whole network (bf16, or fp32 in fp32 networks) and walks the
// layers in place; only the network input and output touch HBM.  The product is computed transposed,
// C^T = W * A^T: the weights are the MFMA "A" operand (32 output features x 16 k), the activations the "B"
// operand (16 k x 32 batch rows), so that a lane's accumulators hold 4 consecutive features of one batch row
// and the epilogue writes them back with one 8-byte LDS store.  Wavefront w owns output tiles w and w + 8 and
// all BM rows; its weight fragments stream from global memory (L2-resident, pre-ordered so that a fragment is
// one contiguous 1 KB read) through a register ring kPF steps deep; activation fragments come from LDS.
constexpr int kFusedMaxWidth = 512;
constexpr int kFusedWaves = 8;
// ring depth: 4 steps, 2 for the 64-row tile (two workgroups per CU, 128 registers each)
constexpr int kPF = 4;

struct FusedArgs {
  int64_t M;
  int n_layers, in_dim, out_dim, lda;
  int fk[KS_MAX_LAYERS], fn[KS_MAX_LAYERS];
  const u32x4* Wp[KS_MAX_LAYERS];
  const float* bp[KS_MAX_LAYERS];
  const float* x;
  float* y;
  long long* prof;  // phase time stamps of wavefront 0, written only by -DKS_PROFILE builds
  // training forward: hidden layer l's activations also go to save[l], (M, save_ld[l]) row-major in working precision, for the backward pass
  void* save[KS_MAX_LAYERS];
  int save_ld[KS_MAX_LAYERS];
  int64_t save_rows;  // rows of the saved arrays: M, or the whole tiles' (what the padding rows hold is finite and of no use)
  void* save_in;      // nullable: the network input as well, (save_rows, in_width) in working precision, zero beyond the real inputs
  int in_width;       // 0 without save_in
};

#ifdef KS_PROFILE
#define KS_MLP_STAMP(k) if (a.prof && tid == 0) a.prof[(int64_t)blockIdx.x * 32 + (k)] = wall_clock64();
#define KS_MLP_STAMP2(k) if (a.prof && threadIdx.x == 0) a.prof[(int64_t)blockIdx.x * 32 + (k)] = wall_clock64();
#else
#define KS_MLP_STAMP(k)
#define KS_MLP_STAMP2(k)
#endif

// One fragment step of both operands: 16 k of bf16 in one matrix instruction, or 8 k of fp32 in four (lane half h holds k = 8 step +
// 4 h + e in element e, so instruction e multiplies k = 8 step + e and 8 step + 4 + e); 16 bytes of each operand per lane either way.
// SWAP: the operands change places, so that a lane holds 16 rows of one feature instead of 16 features of one row; the same sums.
template <typename T, bool SWAP = false>
__device__ __forceinline__ f32x16 fused_mma(const u32x4& w, const u32x4& b, f32x16 acc) {
  if constexpr (SWAP) return fused_mma<T, false>(b, w, acc);
  if constexpr (sizeof(T) == 2) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  } else {
    typedef __attribute__((ext_vector_type(4))) float f32x4v;
    const f32x4v wf = __builtin_bit_cast(f32x4v, w), bf = __builtin_bit_cast(f32x4v, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[e], bf[e], acc, 0, 0, 0);
  }
  return acc;
}

// One layer's MFMA work of one wavefront: NT output tiles (weights w[t]) times MI row tiles.  `arow` points at
// this lane's activation fragment of K step 0 (row lane % 32 of the first row tile, k half lane / 32).
// Weight fragments sit in a register ring kPF steps ahead; activation fragments are read one step ahead.
// side: memory traffic of the tile that goes on beside the products, side.even(step) and side.odd(step) in turn.
struct NoSide {
  __device__ __forceinline__ void even(int) {}
  __device__ __forceinline__ void odd(int) {}
};
template <typename T, int NT, int MI, int kPF, bool SWAP = false, typename Side = NoSide>
__device__ __forceinline__ void fused_layer_mma(f32x16 (&acc)[2][MI], const u32x4* __restrict__ w0,
                                                const u32x4* __restrict__ w1, int nk, const T* __restrict__ arow,
                                                int lda, Side&& side = Side{}) {
  static_assert(kPF % 2 == 0, "the activation double buffer relies on an even ring depth");
  constexpr int SK = 32 / (int)sizeof(T);  // k per step
  u32x4 rw[kPF][NT];
#pragma unroll
  for (int u = 0; u < kPF; ++u) {
    const int st = u < nk ? u : nk - 1;
    rw[u][0] = w0[st * 64];
    if (NT > 1) rw[u][NT - 1] = w1[st * 64];
  }
  u32x4 bq[2][MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) bq[0][i] = *(const u32x4*)(arow + i * 32 * lda);
  int s = 0;
  for (; s + kPF <= nk; s += kPF) {
#pragma unroll
    for (int u = 0; u < kPF; ++u) {
      const int step = s + u;
      const int nstep = step + 1 < nk ? step + 1 : step;
#pragma unroll
      for (int i = 0; i < MI; ++i) bq[(u + 1) & 1][i] = *(const u32x4*)(arow + i * 32 * lda + nstep * SK);
      u32x4 wf[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[t] = rw[u][t];
      const int nx = step + kPF < nk ? step + kPF : nk - 1;
      rw[u][0] = w0[nx * 64];
      if (NT > 1) rw[u][NT - 1] = w1[nx * 64];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[t][i] = fused_mma<T, SWAP>(wf[t], bq[u & 1][i], acc[t][i]);
      if (u & 1) side.odd(step);
      else side.even(step);
    }
  }
#pragma unroll
  for (int u = 0; u < kPF - 1; ++u) {
    if (s + u < nk) {
      const int step = s + u;
      const int nstep = step + 1 < nk ? step + 1 : step;
#pragma unroll
      for (int i = 0; i < MI; ++i) bq[(u + 1) & 1][i] = *(const u32x4*)(arow + i * 32 * lda + nstep * SK);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[t][i] = fused_mma<T, SWAP>(rw[u][t], bq[u & 1][i], acc[t][i]);
    }
  }
}

// Accumulator tile layout: lane l, register r -> feature 32 j + 8 (r / 4) + 4 (l / 32) + r % 4 of batch row l % 32.
__device__ __forceinline__ void fused_bias_init(f32x16& acc, const float* __restrict__ bias, int j, int lane) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 b = *reinterpret_cast<const float4*>(bias + j * 32 + 8 * g + 4 * (lane >> 5));
    acc[4 * g] = b.x; acc[4 * g + 1] = b.y; acc[4 * g + 2] = b.z; acc[4 * g + 3] = b.w;
  }
}

// Hidden layer: activation, round to bf16, back into the tile (4 consecutive features = one 8-byte LDS store).
template <int ACT, typename T>
__device__ __forceinline__ void fused_store_hidden(const f32x16& acc, T* __restrict__ act, int lda, int j,
                                                   int row, int lane) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int f0 = j * 32 + 8 * g + 4 * (lane >> 5);
    if constexpr (sizeof(T) == 4) {
      *reinterpret_cast<float4*>(act + row * lda + f0) =
          float4{activate<ACT, false>(acc[4 * g]), activate<ACT, false>(acc[4 * g + 1]), activate<ACT, false>(acc[4 * g + 2]), activate<ACT, false>(acc[4 * g + 3])};
      continue;
    }
    const uint2 packed = {pack_bf16(activate<ACT, true>(acc[4 * g]), activate<ACT, true>(acc[4 * g + 1])),
                          pack_bf16(activate<ACT, true>(acc[4 * g + 2]), activate<ACT, true>(acc[4 * g + 3]))};
    *reinterpret_cast<uint2*>(act + row * lda + f0) = packed;
  }
}

// The first `ld` columns of the finished tile's rows (zeros from column `held` on), 16 bytes per thread and pass, to rows m0.. of dst (M, ld); rows
// from M on are left out.  ld: whole 16-byte pieces, at most one pass of the workgroup.
// A pass every two steps of the K loop that reads the tile next (a tile of n columns is n / 16 steps and n / 32 passes), the rest behind it.  All at
// once before the loop, the stores stood ahead of its weights, which are waited for in order: 65536 rows of 68-512-512-512-20, training forward
// 120 -> 114 us, backward 171 -> 167.
template <typename T, int ROWS>
struct TileRowsOut {
  static constexpr int PC = 16 / (int)sizeof(T);  // entries of a piece
  const T* from = nullptr;
  T* to = nullptr;
  int64_t to_step = 0;
  int from_step = 0, per = 1, left = 0;  // left: rows from this thread's next one on
  bool real = false;
  uint4 v = {0u, 0u, 0u, 0u};

  __device__ __forceinline__ TileRowsOut() {}
  __device__ __forceinline__ TileRowsOut(const T* act, int lda, T* dst, int ld, int held, int64_t m0, int64_t M) {
    const int pieces = ld / PC, r0 = (int)threadIdx.x / pieces, c = ((int)threadIdx.x - r0 * pieces) * PC;
    per = 64 * kFusedWaves / pieces;
    left = r0 < per ? (M - m0 < ROWS ? (int)(M - m0) : ROWS) - r0 : 0;
    real = c < held;
    from = act + r0 * lda + c;
    from_step = per * lda;
    to = dst + (m0 + r0) * ld + c;
    to_step = (int64_t)per * ld;
  }
  __device__ __forceinline__ void even(int) {
    if (left > 0 && real) v = *reinterpret_cast<const uint4*>(from);
  }
  __device__ __forceinline__ void odd(int) {
    if (left > 0) *reinterpret_cast<uint4*>(to) = v;
    from += from_step;
    to += to_step;
    left -= per;
  }
  __device__ __forceinline__ void finish() {
    while (left > 0) {
      even(0);
      odd(0);
    }
  }
};

// Output layer: fp32 rows of the caller's (M, out_dim) matrix.
__device__ __forceinline__ void fused_store_output(const f32x16& acc, float* __restrict__ y, int64_t M, int out_dim,
                                                   int j, int64_t m, int lane) {
  if (m >= M) return;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int f0 = j * 32 + 8 * g + 4 * (lane >> 5);
    float* dst = y + m * out_dim + f0;
    if ((out_dim & 3) == 0 && f0 + 4 <= out_dim) {
      *reinterpret_cast<float4*>(dst) = float4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (f0 + e < out_dim) dst[e] = acc[4 * g + e];
    }
  }
}

// The output of a single layer, which the stores bound: with a lane per feature (SWAP) a store is two runs of 128 bytes, with a lane per row
// 64 pieces of 16 (12288 x 128 -> 384: 13.5 -> 8.3 us, 65536 rows: 44.9 -> 28.3, of 27 at the card's copy rate).  Networks keep a lane per row:
// their outputs are narrow, and the second form of the last layer cost them 1 %.
__device__ __forceinline__ void fused_store_output_swapped(const f32x16& acc, float* __restrict__ y, int64_t M, int out_dim, int j, int64_t m0,
                                                           int lane) {
  const int col = 32 * j + (lane & 31);
  if (col >= out_dim) return;
  const int64_t row0 = m0 + 4 * (lane >> 5);
  float* dst = y + row0 * out_dim + col;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int down = 8 * (r >> 2) + (r & 3);
    if (row0 + down < M) dst[(int64_t)down * out_dim] = acc[r];
  }
}

// How many wavefronts cut the reduction of a narrow fp32 layer of nt <= 2 tiles (their partial tiles, 4 KB each per row tile, have to fit the
// activation tile)
__host__ __device__ inline int fused_share(int nt, int lda) {
  int share = nt == 1 ? 4 : 2;
  while (share > 1 && share * nt * 1024 > 32 * lda) share >>= 1;
  return share;
}

// One layer of the whole-network kernel for one wavefront: MFMA work, barrier, epilogue, barrier.
template <int ACT, typename T, int MI, bool LAST, bool SAVE, bool SWAP = false>
__device__ __forceinline__ void fused_layer(const FusedArgs& a, int l, T* __restrict__ act, int64_t m0, int lane,
                                            int wave, int64_t tile, TileRowsOut<T, MI * 32>& out) {
  const int nk = a.fk[l], nt = a.fn[l], lda = a.lda;
  const T* arow = act + (lane & 31) * lda + (lane >> 5) * (16 / (int)sizeof(T));
  const int row = lane & 31;
  // what the layer before left (or the network input) goes out beside this one's products; smaller tiles share the CU with other workgroups,
  // which do the same, and have no registers for it
  constexpr bool LATER = SAVE && sizeof(T) == 2 && MI == 4;
  if constexpr (SAVE && sizeof(T) == 2 && !LATER) out.finish();
  NoSide none;
  auto& side = [&]() -> auto& {
    if constexpr (LATER) return out;
    else return none;
  }();
  if (sizeof(T) == 4 && MI <= 2 && nt <= 2) {
    // Few tiles in fp32 (an output layer of 21 or 1 columns): one wavefront's 8 k per 256 cycles would leave the others idle for the
    // layer's whole reduction (256 wide: 3.4 us of 25), so 2 or 4 wavefronts cut a tile's reduction and add up through the tile's
    // own LDS, as many as it has room for (4 KB each).
    // The same number for every row tile: a row's sums must not depend on the batch it comes in.
    const int share = fused_share(nt, lda);
    const bool busy = wave < share * nt * MI;
    const int tl = busy ? wave / share : 0, part = busy ? wave % share : 0, j = tl / MI, i = tl % MI;
    const int per = (nk + share - 1) / share, k0 = part * per, kn = busy ? (nk - k0 < per ? nk - k0 : per) : 0;
    f32x16 acc[2][1];
    fused_bias_init(acc[0][0], a.bp[l], j, lane);
    if (part > 0)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.f;
    const u32x4* w0 = a.Wp[l] + ((int64_t)j * nk + k0) * 64 + lane;
    if (kn > 0) fused_layer_mma<T, 1, 1, 2>(acc, w0, w0, kn, arow + i * 32 * lda + k0 * 8, lda);
    __syncthreads();  // every wavefront has read this layer's input; the tile can be overwritten
    float* sc = reinterpret_cast<float*>(act);
    if (share > 1) {
      if (busy && part > 0)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[wave * 1024 + r * 64 + lane] = acc[0][0][r];
      __syncthreads();
      if (busy && part == 0)
        for (int q = 1; q < share; ++q)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[0][0][r] += sc[(wave + q) * 1024 + r * 64 + lane];
      __syncthreads();
    }
    if (busy && part == 0) {
      if (LAST) fused_store_output(acc[0][0], a.y, a.M, a.out_dim, j, m0 + i * 32 + row, lane);
      else fused_store_hidden<ACT, T>(acc[0][0], act, lda, j, i * 32 + row, lane);
    }
  } else if (nt * MI <= kFusedWaves) {  // few tiles: one (feature tile, row tile) pair per wavefront
    const bool busy = wave < nt * MI;
    const int j = busy ? wave / MI : 0, i = busy ? wave % MI : 0;
    f32x16 acc[2][1];
    if (SWAP) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][0][r] = a.bp[l][j * 32 + row];
    } else {
      fused_bias_init(acc[0][0], a.bp[l], j, lane);
    }
    acc[1][0] = acc[0][0];
    const u32x4* w0 = a.Wp[l] + (int64_t)j * nk * 64 + lane;
    if (busy) fused_layer_mma<T, 1, 1, (MI == 2 ? 2 : kPF), SWAP>(acc, w0, w0, nk, arow + i * 32 * lda, lda, side);
    if constexpr (LATER) out.finish();
    KS_MLP_STAMP2(2 + 3 * l)
    __syncthreads();  // every wavefront has read this layer's input; the tile can be overwritten
    KS_MLP_STAMP2(3 + 3 * l)
    if (busy) {
      if (SWAP) fused_store_output_swapped(acc[0][0], a.y, a.M, a.out_dim, j, m0 + i * 32, lane);
      else if (LAST) fused_store_output(acc[0][0], a.y, a.M, a.out_dim, j, m0 + i * 32 + row, lane);
      else fused_store_hidden<ACT, T>(acc[0][0], act, lda, j, i * 32 + row, lane);
    }
  } else {
    const int mine = wave < nt ? (wave + kFusedWaves < nt ? 2 : 1) : 0;
    const int j0 = wave < nt ? wave : 0, j1 = wave + kFusedWaves < nt ? wave + kFusedWaves : j0;
    f32x16 acc[2][MI];
    if (SWAP) {
#pragma unroll
      for (int r = 0; r < 16; ++r) { acc[0][0][r] = a.bp[l][j0 * 32 + row]; acc[1][0][r] = a.bp[l][j1 * 32 + row]; }
    } else {
      fused_bias_init(acc[0][0], a.bp[l], j0, lane);
      fused_bias_init(acc[1][0], a.bp[l], j1, lane);
    }
#pragma unroll
    for (int i = 1; i < MI; ++i) {
      acc[0][i] = acc[0][0];
      acc[1][i] = acc[1][0];
    }
    const u32x4* w0 = a.Wp[l] + (int64_t)j0 * nk * 64 + lane;
    const u32x4* w1 = a.Wp[l] + (int64_t)j1 * nk * 64 + lane;
    if (mine == 2) fused_layer_mma<T, 2, MI, (MI == 2 ? 2 : kPF), SWAP>(acc, w0, w1, nk, arow, lda, side);
    else if (mine == 1) fused_layer_mma<T, 1, MI, (MI == 2 ? 2 : kPF), SWAP>(acc, w0, w0, nk, arow, lda, side);
    if constexpr (LATER) out.finish();
    KS_MLP_STAMP2(2 + 3 * l)
    __syncthreads();
    KS_MLP_STAMP2(3 + 3 * l)
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (t < mine) {
        const int j = t == 0 ? j0 : j1;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          if (SWAP) fused_store_output_swapped(acc[t][i], a.y, a.M, a.out_dim, j, m0 + i * 32, lane);
          else if (LAST) fused_store_output(acc[t][i], a.y, a.M, a.out_dim, j, m0 + i * 32 + row, lane);
          else fused_store_hidden<ACT, T>(acc[t][i], act, lda, j, i * 32 + row, lane);
        }
      }
  }
  __syncthreads();
  KS_MLP_STAMP2(4 + 3 * l)
  // The next layer only reads the tile until every wavefront (this copy included, which sits before that barrier in program order) has passed
  // the next barrier.  Rows are as wide as the backward pass's layers, which is more than the tile's (zeros) where the width is no multiple of 128.
  if constexpr (sizeof(T) == 2) {
    if (SAVE && !LAST) out = TileRowsOut<T, MI * 32>(act, lda, reinterpret_cast<T*>(a.save[l]), a.save_ld[l], nt * 32, m0, a.save_rows);
  } else if (!LAST && a.save[l]) {  // one form for both in fp32, whose code without this is 4 % slower (8192 rows of 71-256-256-256-21: 31.5 -> 32.9 us)
    T* dst = reinterpret_cast<T*>(a.save[l]);
    const int ld = a.save_ld[l], w4 = ld / 4, held = nt * 8;
    for (int idx = threadIdx.x; idx < MI * 32 * w4; idx += 64 * kFusedWaves) {
      const int r = idx / w4, c4 = idx - r * w4;
      if (m0 + r < a.M)
        *reinterpret_cast<uint4*>(dst + (m0 + r) * ld + c4 * 4) =
            c4 < held ? *reinterpret_cast<const uint4*>(act + r * lda + c4 * 4) : uint4{0u, 0u, 0u, 0u};
    }
  }
}

// The network's input rows, one piece of memory, into the tile; zero beyond the batch and from column in_dim to K0.  V: what a thread requests at a
// time, and Q of them before it waits.  bf16 tiles of 64 rows and more (kHeld): the loads stand behind no condition (the index is held back to the
// last one), as behind one they are waited for one by one, and the zeros go in as 16-byte pieces, one of which may hold a row's last columns too:
// hence the barrier.  Tiles of 32 rows are two to five loads a thread, of which most would be repeats, and the barrier costs as much as the entries
// of padding; fp32 networks read beside six matrix instructions a product.  In us, behind conditions -> held back:
//   68-3 x 128-20, 4096 rows 6.87 -> 7.02, 12000 rows 8.78 -> 8.00; 120-3 x 128-20 7.02 -> 7.21 and 8.09 -> 8.37; 71-3 x 256-20, 12000 rows 12.98 -> 14.15;
//   43-3 x 128-20, 12000 rows 7.63 -> 8.19; a pair 68-3 x 256, 64 rows 9.45 -> 9.57; fp32 71-3 x 128-20, 20000 rows 36.4 -> 36.9
//   68-3 x 128-20, 20000 rows 10.28 -> 9.49; 71-3 x 512-20, 20000 rows, four at a time 37.9 -> 39.6, six 37.7; 67-3 x 256-20, 65536 rows 39.6 -> 37.5; 67-2 x 256-20, 524288 rows 242 -> 206; training forward of 65536
//   rows of 67-3 x 128-20 40.5 -> 34.7; worst of a sweep: 55-2 x 256-20, 30000 rows 13.8 -> 14.4
template <typename T, int BM, typename V>
__device__ __forceinline__ void mlp_input_tile(T* __restrict__ act, int lda, const float* __restrict__ src, int rows, int in_dim, int K0) {
  constexpr bool kHeld = sizeof(T) == 2 && BM >= 64;
  constexpr int NTHR = 64 * kFusedWaves, E = sizeof(V) / 4, Q = BM >= 128 ? 8 : kHeld && E == 1 ? 6 : 4, PC = 16 / (int)sizeof(T);
  const int tid = threadIdx.x, total = rows * in_dim / E;
  const V* from = reinterpret_cast<const V*>(src);
  if constexpr (kHeld) {
    if (K0 > in_dim || rows < BM) {
      const int first = in_dim / PC, pieces = K0 / PC - first;
      for (int idx = tid; idx < BM * pieces; idx += NTHR) {
        const int r = idx / pieces;
        *reinterpret_cast<u32x4*>(act + r * lda + (first + idx - r * pieces) * PC) = u32x4{0u, 0u, 0u, 0u};
      }
      for (int idx = rows * first + tid; idx < BM * first; idx += NTHR) {
        const int r = idx / first;
        *reinterpret_cast<u32x4*>(act + r * lda + (idx - r * first) * PC) = u32x4{0u, 0u, 0u, 0u};
      }
      __syncthreads();
    }
  } else {
    const int padw = K0 - in_dim;
    for (int idx = tid; idx < BM * padw; idx += NTHR) {
      const int r = idx / padw, c = idx - r * padw;
      act[r * lda + in_dim + c] = (T)0.0f;
    }
    for (int idx = rows * in_dim + tid; idx < BM * in_dim; idx += NTHR) {
      const int r = idx / in_dim, c = idx - r * in_dim;
      act[r * lda + c] = (T)0.0f;
    }
  }
  for (int base = tid; base < total; base += NTHR * Q) {
    V v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int idx = base + q * NTHR;
      if constexpr (kHeld) v[q] = from[min(idx, total - 1)];
      else v[q] = idx < total ? from[idx] : V{};
    }
    if constexpr (kHeld) {
#pragma unroll
      for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(v[q]));  // keeps the loads out of the conditions below
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int idx = base + q * NTHR;
      if (idx < total) {
        const int r = idx * E / in_dim, c = idx * E - r * in_dim;
        if constexpr (E == 1) act[r * lda + c] = (T)v[q];
        else if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4*>(act + r * lda + c) = v[q];
        else *reinterpret_cast<uint2*>(act + r * lda + c) = uint2{pack_bf16(v[q][0], v[q][1]), pack_bf16(v[q][2], v[q][3])};
      }
    }
  }
}

// SAVE: the training forward of bf16 networks (FusedArgs::save, save_in)
template <int ACT, typename T, int BM, bool SINGLE = false, bool SAVE = false>
__device__ __forceinline__ void mlp_fused_body(const FusedArgs& a, int64_t tile) {
  constexpr int MI = BM / 32;
  constexpr int NTHR = 64 * kFusedWaves;
  extern __shared__ __attribute__((aligned(16))) unsigned char mlp_lds[];
  T* act = reinterpret_cast<T*>(mlp_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t m0 = tile * BM;
  const int lda = a.lda;
  constexpr int SK = 32 / (int)sizeof(T);
  KS_MLP_STAMP(0)
  {  // network input -> tile; zero beyond the batch and in the K padding of the first layer
    const int in_dim = a.in_dim;
    const int K0 = SAVE && a.in_width > a.fk[0] * SK ? a.in_width : a.fk[0] * SK;  // the copy that is kept is padded further
    const int64_t rows_left = a.M - m0;
    const int rows = rows_left < BM ? (int)rows_left : BM;
    const float* src = a.x + m0 * in_dim;
    if ((in_dim & 3) == 0) mlp_input_tile<T, BM, f32x4>(act, lda, src, rows, in_dim, K0);  // rows are 16-byte aligned
    else mlp_input_tile<T, BM, float>(act, lda, src, rows, in_dim, K0);
  }
  __syncthreads();
  KS_MLP_STAMP(1)
  TileRowsOut<T, BM> out;
  if (SAVE && a.save_in) out = TileRowsOut<T, BM>(act, lda, reinterpret_cast<T*>(a.save_in), a.in_width, a.in_width, m0, a.save_rows);  // the tile stays until the first layer's barrier
  if constexpr (!SINGLE)
    for (int l = 0; l + 1 < a.n_layers; ++l) fused_layer<ACT, T, MI, false, SAVE>(a, l, act, m0, lane, wave, tile, out);
  fused_layer<ACT, T, MI, true, SAVE, SINGLE>(a, SINGLE ? 0 : a.n_layers - 1, act, m0, lane, wave, tile, out);
}

// SINGLE: one bf16 layer
template <int ACT, typename T, int BM, bool SINGLE = false, bool SAVE = false>
__global__ __launch_bounds__(64 * kFusedWaves) __attribute__((amdgpu_waves_per_eu(BM <= 64 ? 4 : 2, BM <= 64 ? 4 : 2)))
void mlp_fused_kernel(const FusedArgs a) {
  mlp_fused_body<ACT, T, BM, SINGLE, SAVE>(a, blockIdx.x);
}

// Two networks over the same rows in one launch (actor and critic of a control step): blockIdx.y picks the network, so
// the second network's workgroups fill the CUs next to the first one's instead of waiting for their launch to drain.
template <int ACT, typename T, int BM>
__global__ __launch_bounds__(64 * kFusedWaves) __attribute__((amdgpu_waves_per_eu(BM <= 64 ? 4 : 2, BM <= 64 ? 4 : 2)))
void mlp_fused_pair_kernel(const FusedArgs a, const FusedArgs b, const KsActionSample s) {
  // Workgroup L of the launch runs on XCD L % 8.  XCDs 0-3 take the first network and 4-7 the second, so that an XCD's L2
  // fetches one network's weights, not both (the weights are cold at every control step: the physics launch in between
  // sweeps the L2s).
  const int64_t L = blockIdx.x + (int64_t)blockIdx.y * gridDim.x;
  int net = blockIdx.y;
  int64_t tile = blockIdx.x;
  if (gridDim.x % 4 == 0) {
    net = (int)(L % 8) / 4;
    tile = (L / 8) * 4 + (L % 8) % 4;
  }
  if (net == 0) mlp_fused_body<ACT, T, BM>(a, tile);
  else mlp_fused_body<ACT, T, BM>(b, tile);
  // The actions of the actor's rows, by all wavefronts from the means that the last layer's have just written (the layer ends with a barrier),
  // instead of one more small launch per control step: 8192 K-Bots in two groups 448.9 -> 444.0 us, 64 of them 226.7 -> 225.7, 4096 humanoids
  // 320.1 -> 319.3 (four processes a side in turn on one card, which differed by 0.2 % at most).
  if (net != 0 || !s.action) return;
  const int nu = a.out_dim;
  const int64_t m0 = tile * BM;
  const int n = (int)(a.M - m0 < BM ? a.M - m0 : BM) * nu;
  for (int i = threadIdx.x; i < n; i += 64 * kFusedWaves) {
    const int r = i / nu, u = i - r * nu;
    const int64_t idx = m0 * nu + i;
    s.action[idx] = sampled_action(a.y[idx], s.log_std, s.noise_normal, s.rng, s.clip_max, m0 + r, u, idx);
  }
}

// Two single bf16 layers, e.g. the actor's and the critic's projection of one depth, or the input gradients of both: a few thousand rows of one
// fill the chip for less time than a launch costs (12288 x 128 -> 384: 9.7 us each one after the other, 14.2 both).
template <int BM>
__global__ __launch_bounds__(64 * kFusedWaves) __attribute__((amdgpu_waves_per_eu(BM <= 64 ? 4 : 2, BM <= 64 ? 4 : 2)))
void mlp_single_pair_kernel(const FusedArgs a, const FusedArgs b, unsigned tiles_a) {
  if (blockIdx.x < tiles_a) mlp_fused_body<KS_ACT_NONE, __bf16, BM, true>(a, blockIdx.x);
  else mlp_fused_body<KS_ACT_NONE, __bf16, BM, true>(b, blockIdx.x - tiles_a);
}

// ---------------------------------------------------------------- few rows through a wide bf16 network
// Over a few row tiles the whole-network kernel is bound by how fast a CU takes in weights (66 GB/s whatever is in flight: 1.1 MB of a
// 3 x 512 network are 16 us), so here the 32-wide output tiles of a layer go to as many CUs.  A layer needs the whole of the one before
// it, which is a launch boundary, 3 to 4 us; the first launch makes up for its own by taking the first layer, whose weights are few,
// in every workgroup, and the last hidden layer's launch also runs the output layer in the workgroup that arrives last at a row tile.
// Per output the sums are the whole-network kernel's in the same order, so the results do not depend on the path.
//   68-512-512-512-20: one row 17.6 -> 12.4 us, 256 rows 17.8 -> 13.8; as one of a pair, 64 rows 17.9 -> 12.6
constexpr int kSplitTile = 2 * (kFusedMaxWidth / 32) * 64;  // 16-byte fragments of a 32-row tile of activations: [k step][lane]

// What a launch needs of a network, resolved on the host: the arguments are a scalar load away, and one that depends on another is two.
struct SplitFirst {
  const float* x;
  const u32x4 *w0, *w1;
  const float *b0, *b1;
  u32x4* h;           // activations of every row tile for the next launch, in the order of the matrix operand
  unsigned* arrived;  // per row tile: zeroed here, counted by the last hidden layer's launch
  int M, in_dim, lda, nk0, nt0, nk1, nt1;
};
struct SplitLayer {
  const u32x4 *h, *w;
  const float* b;
  u32x4* h_out;  // null: this is the output layer
  const u32x4* wo;  // the output layer, where it follows in this launch, else null
  const float* bo;
  float* y;
  unsigned* arrived;
  int M, out_dim, nk, nt, nko, nto;
};

__device__ __forceinline__ void device_store8(void* p, uint2 v) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32x4 device_load16(const u32x4* p) {
  const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
  const uint2 lo = __builtin_bit_cast(uint2, __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  const uint2 hi = __builtin_bit_cast(uint2, __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  return u32x4{lo.x, lo.y, hi.x, hi.y};
}

// A finished tile j of 32 features, activated and rounded, as fragments of the next layer's operand.  ACROSS: written past this XCD's L2, for
// a reader inside this launch.
template <int ACT, bool ACROSS>
__device__ __forceinline__ void split_store(const f32x16& acc, u32x4* __restrict__ h, int j, int lane) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const uint2 v = {pack_bf16(activate<ACT, true>(acc[4 * g]), activate<ACT, true>(acc[4 * g + 1])),
                     pack_bf16(activate<ACT, true>(acc[4 * g + 2]), activate<ACT, true>(acc[4 * g + 3]))};
    uint2* to = reinterpret_cast<uint2*>(h + (2 * j + (g >> 1)) * 64 + (lane & 31) + 32 * (g & 1)) + (lane >> 5);
    if (ACROSS) device_store8(to, v);
    else *to = v;
  }
}

constexpr int kSplitSteps = kFusedMaxWidth / 16;  // K steps of the widest layer

__device__ __forceinline__ void split_fetch(u32x4 (&f)[kSplitSteps], const u32x4* __restrict__ src, int nk, int lane) {
#pragma unroll
  for (int u = 0; u < kSplitSteps; ++u) f[u] = src[min(u, nk - 1) * 64 + lane];
}

// 32 rows of the network input, rounded, to the tile: sixteen threads a row, eight values (zero beyond the batch and the row) each and pass
__device__ __forceinline__ void split_stage_input(const SplitFirst& s, __bf16* __restrict__ act, int64_t m0, int tid) {
  const int row = tid >> 4;
  const bool in = m0 + row < s.M;
  const float* src = s.x + (m0 + (in ? row : 0)) * s.in_dim;
  for (int c = (tid & 15) * 8; c < s.nk0 * 16; c += 128) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = src[min(c + e, s.in_dim - 1)];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = in && c + e < s.in_dim ? v[e] : 0.f;
    *reinterpret_cast<u32x4*>(act + row * s.lda + c) = u32x4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
  }
}

template <int ACT>
__device__ __forceinline__ void split_first_body(const SplitFirst& s) {
  extern __shared__ __attribute__((aligned(16))) unsigned char mlp_lds[];
  __bf16* act = reinterpret_cast<__bf16*>(mlp_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = blockIdx.x;
  const int64_t tile = blockIdx.y, m0 = tile * 32;
  if (j >= s.nt1) return;  // the other network of the launch is wider
  const int j0 = min(wave, s.nt0 - 1), j1 = min(wave + kFusedWaves, s.nt0 - 1);
  const u32x4 *w0 = s.w0 + (int64_t)j0 * s.nk0 * 64 + lane, *w1 = s.w0 + (int64_t)j1 * s.nk0 * 64 + lane;
  f32x16 acc0[2][1];
  fused_bias_init(acc0[0][0], s.b0, j0, lane);
  fused_bias_init(acc0[1][0], s.b0, j1, lane);
  split_stage_input(s, act, m0, tid);
  u32x4 w[kSplitSteps];  // this workgroup's tile of the second layer, on its way during the first
  if (wave == 0) split_fetch(w, s.w1 + (int64_t)j * s.nk1 * 64, s.nk1, lane);
  __syncthreads();
  const __bf16* arow = act + (lane & 31) * s.lda + (lane >> 5) * 8;
  fused_layer_mma<__bf16, 2, 1, kPF>(acc0, w0, w1, s.nk0, arow, s.lda);
  __syncthreads();  // every wavefront has read the input; the tile takes the first layer's output
  if (wave < s.nt0) fused_store_hidden<ACT, __bf16>(acc0[0][0], act, s.lda, j0, lane & 31, lane);
  if (wave + kFusedWaves < s.nt0) fused_store_hidden<ACT, __bf16>(acc0[1][0], act, s.lda, j1, lane & 31, lane);
  __syncthreads();
  if (wave != 0) return;
  if (j == 0 && lane == 0) s.arrived[tile] = 0;
  f32x16 acc;
  fused_bias_init(acc, s.b1, j, lane);
#pragma unroll
  for (int u = 0; u < kSplitSteps; ++u)
    if (u < s.nk1) acc = fused_mma<__bf16>(w[u], *reinterpret_cast<const u32x4*>(arow + u * 16), acc);
  split_store<ACT, false>(acc, s.h + tile * kSplitTile, j, lane);
}

// The first two layers: workgroup (j, tile, network) computes output tile j of the second one.
template <int ACT>
__global__ __launch_bounds__(64 * kFusedWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void mlp_split_first_kernel(const SplitFirst p, const SplitFirst q) {
  if (blockIdx.z == 0) split_first_body<ACT>(p);
  else split_first_body<ACT>(q);
}

template <int ACT>
__device__ __forceinline__ void split_layer_body(const SplitLayer& s) {
  const int lane = threadIdx.x, j = blockIdx.x;
  const int64_t tile = blockIdx.y, m = tile * 32 + (lane & 31);
  if (j >= s.nt) return;
  u32x4 w[kSplitSteps], x[kSplitSteps];
  split_fetch(w, s.w + (int64_t)j * s.nk * 64, s.nk, lane);
  split_fetch(x, s.h + tile * kSplitTile, s.nk, lane);
  f32x16 acc;
  fused_bias_init(acc, s.b, j, lane);
#pragma unroll
  for (int u = 0; u < kSplitSteps; ++u)
    if (u < s.nk) acc = fused_mma<__bf16>(w[u], x[u], acc);
  if (!s.h_out) {
    fused_store_output(acc, s.y, s.M, s.out_dim, j, m, lane);
    return;
  }
  u32x4* h = s.h_out + tile * kSplitTile;
  if (!s.wo) {
    split_store<ACT, false>(acc, h, j, lane);
    return;
  }
  split_store<ACT, true>(acc, h, j, lane);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this tile has reached memory
  unsigned before = 0;
  if (lane == 0) before = atomicAdd(s.arrived + tile, 1u);
  if (__builtin_amdgcn_readfirstlane(before) != (unsigned)s.nt - 1u) return;
#pragma unroll
  for (int u = 0; u < kSplitSteps; ++u) x[u] = device_load16(h + min(u, s.nko - 1) * 64 + lane);
  for (int t = 0; t < s.nto; ++t) {
    split_fetch(w, s.wo + (int64_t)t * s.nko * 64, s.nko, lane);
    fused_bias_init(acc, s.bo, t, lane);
#pragma unroll
    for (int u = 0; u < kSplitSteps; ++u)
      if (u < s.nko) acc = fused_mma<__bf16>(w[u], x[u], acc);
    fused_store_output(acc, s.y, s.M, s.out_dim, t, m, lane);
  }
}

// A later layer, a wavefront per output tile; the last hidden layer's launch ends with the output layer.
template <int ACT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mlp_split_layer_kernel(const SplitLayer p, const SplitLayer q) {
  if (blockIdx.z == 0) split_layer_body<ACT>(p);
  else split_layer_body<ACT>(q);
}

// ---------------------------------------------------------------- whole-network backward pass of the hidden layers
// dZ_{l-1} = (dZ_l W_l) * f'(Y_{l-1}) for l = L-1 .. 1 in one launch, a 128-row tile per workgroup that never leaves LDS: the product is the
// forward kernel's K loop over the fragment-ordered transposed weights, its epilogue multiplies by f' of the activations that the training
// forward left, and the finished tile goes out row by row (an operand of the weight gradients below) with its column sums (the bias
// gradient, one partial row per tile).
// Bound by the products (58 us at the rate of a large product) and the tile's way in and out of memory (80 at the copy rate), which a single
// workgroup per CU does one after the other.  65536 rows of 68-512-512-512-20: 174 -> 157 us (203 -> 185 just behind other kernels) since
// activations and gradients move as whole rows; as transposes every lane loaded and stored 2 bytes at a time.  167 -> 146 between other kernels
// since no load stands behind a condition: the entry's tile was 32 loads one after the other and a layer's activations three groups.  Column sums over half the rows
// a thread would keep all wavefronts busy with them, but their partial rows cost the final sum more than that gains.
struct FusedBwdArgs {
  int64_t M;
  int n_layers, lda;
  int fk[KS_MAX_LAYERS], fn[KS_MAX_LAYERS];   // the forward kernel's K steps and output tiles per layer
  const u32x4* WtP[KS_MAX_LAYERS];            // l >= 1: W_l^T in fragment order, [input tile][step over outputs][lane] x 16 bytes
  const float* dy;                            // (M, out_dim): gradient of the network output, in the caller's layout
  int out_dim, np_last;                       // np_last: columns of dz[L-1] (the output width padded for the weight-gradient product)
  const __bf16* y[KS_MAX_LAYERS];             // hidden layer l's activations, row-major, as the training forward left them
  __bf16* dz[KS_MAX_LAYERS];                  // out, every layer: dZ_l (whole tiles of rows, width); zero beyond the batch
  float* bias_part[KS_MAX_LAYERS];            // out, every layer: (tiles, width) column sums of dZ_l per tile
};

template <int ACT>
__global__ __launch_bounds__(64 * kFusedWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void mlp_fused_bwd_kernel(const FusedBwdArgs a) {
  constexpr int MI = 4, BM = 128, NTHR = 64 * kFusedWaves;
  extern __shared__ __attribute__((aligned(16))) unsigned char mlp_lds[];
  __bf16* act = reinterpret_cast<__bf16*>(mlp_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t tile = blockIdx.x, m0 = tile * BM;
  const int lda = a.lda, L = a.n_layers;
  {  // the last layer's gradient tile from the caller's fp32 rows, which are one piece of memory; zero in the padding columns and beyond the
     // batch (such rows stay zero through every layer).  Eight entries of a thread are requested at a time.
    const int np = a.np_last, od = a.out_dim;
    for (int idx = tid; idx < BM * (np / 8); idx += NTHR)
      *reinterpret_cast<u32x4*>(act + (idx / (np / 8)) * lda + idx % (np / 8) * 8) = u32x4{0u, 0u, 0u, 0u};
    const int held = (int)(a.M - m0 < BM ? a.M - m0 : BM) * od;  // at least one row
    const float* dy = a.dy + m0 * od;
    __syncthreads();
    for (int first = tid; first < held; first += 8 * NTHR) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = dy[min(first + u * NTHR, held - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(v[u]));  // keeps the loads out of the conditions below
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int at = first + u * NTHR, r = at / od;
        if (at < held) act[r * lda + at - r * od] = (__bf16)v[u];
      }
    }
  }
  __syncthreads();
  // The finished tile's column sums (the bias gradient's share) go out before the next K loop reads the tile, the tile itself beside it
  TileRowsOut<__bf16, BM> out;
  auto tile_out = [&](__bf16* dst, float* bias_part, int width) {
    out = TileRowsOut<__bf16, BM>(act, lda, dst, width, width, m0, m0 + BM);
    if (tid >= width / 2) return;
    f32x2 cs = {0.f, 0.f};
#pragma unroll 32
    for (int r = 0; r < BM; ++r) {
      const bf16x2 v = *reinterpret_cast<const bf16x2*>(act + r * lda + 2 * tid);
      cs[0] += (float)v[0]; cs[1] += (float)v[1];
    }
    float* part = bias_part + tile * width + 2 * tid;
    part[0] = cs[0];
    part[1] = cs[1];
  };
  tile_out(a.dz[L - 1], a.bias_part[L - 1], a.np_last);
  const __bf16* arow = act + (lane & 31) * lda + (lane >> 5) * 8;
  const int row = lane & 31;
  for (int l = L - 1; l >= 1; --l) {
    const int nk = a.fn[l] * 2;  // K steps over layer l's outputs
    const int nt = a.fk[l] / 2;  // 32-wide tiles over layer l - 1's outputs
    const int mine = wave < nt ? (wave + kFusedWaves < nt ? 2 : 1) : 0;
    const int j0 = wave < nt ? wave : 0, j1 = wave + kFusedWaves < nt ? wave + kFusedWaves : j0;
    f32x16 acc[2][MI];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][i][r] = 0.f;
    const u32x4* w0 = a.WtP[l] + (int64_t)j0 * nk * 64 + lane;
    const u32x4* w1 = a.WtP[l] + (int64_t)j1 * nk * 64 + lane;
    if (mine == 2) fused_layer_mma<__bf16, 2, MI, kPF>(acc, w0, w1, nk, arow, lda, out);
    else if (mine == 1) fused_layer_mma<__bf16, 1, MI, kPF>(acc, w0, w0, nk, arow, lda, out);
    out.finish();
    // Y_{l-1} takes dZ_l's place in the tile on its way to the lanes that need it, and every lane leaves dZ_{l-1} where it read Y: whole rows in
    // 16-byte pieces in and out of memory, 8 bytes per lane of the tile.
    const int width = nt * 32, pieces = width / 8, per = NTHR / pieces, yr = tid / pieces, yc = (tid - yr * pieces) * 8;
    // Requested without a condition, the row held back to the last one: behind conditions the loads were waited for in three groups, and each of
    // them for the stores ahead of it.
    const int rows = (int)(a.M - m0 < BM ? a.M - m0 : BM);
    const __bf16* yt = a.y[l - 1] + m0 * width + yc;
    u32x4 yv[16];  // a width of 512: 8 rows a pass
#pragma unroll
    for (int u = 0; u < 16; ++u) yv[u] = *reinterpret_cast<const u32x4*>(yt + min(yr + u * per, rows - 1) * width);
    __syncthreads();  // every wavefront has read dZ_l
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int r = yr + u * per;
      if (yr < per && r < BM) *reinterpret_cast<u32x4*>(act + r * lda + yc) = r < rows ? yv[u] : u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (t < mine) {
        const int j = t == 0 ? j0 : j1;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            uint2* at = reinterpret_cast<uint2*>(act + (i * 32 + row) * lda + j * 32 + 8 * g + 4 * (lane >> 5));
            const uint2 y4 = *at;
            float d[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const unsigned w = e < 2 ? y4.x : y4.y;
              const float yv1 = __builtin_bit_cast(float, (e & 1) ? w & 0xffff0000u : w << 16);
              d[e] = 1.f;
              if (ACT == KS_ACT_ELU) d[e] = yv1 > 0.f ? 1.f : yv1 + 1.f;
              if (ACT == KS_ACT_RELU) d[e] = yv1 > 0.f ? 1.f : 0.f;
              if (ACT == KS_ACT_TANH) d[e] = 1.f - yv1 * yv1;
              d[e] *= acc[t][i][4 * g + e];
            }
            *at = uint2{pack_bf16(d[0], d[1]), pack_bf16(d[2], d[3])};
          }
      }
    __syncthreads();
    tile_out(a.dz[l - 1], a.bias_part[l - 1], width);
  }
  out.finish();
}

// Weight gradients behind it: slice z of C (np, kp) = dZ^T Y over rows [z kslice, (z + 1) kslice) of dZ (lda = np columns) and Y (ldb columns), both
// row-major as the kernels above left them, in whole tiles of 128 rows of which dZ's are zero beyond the batch; 128 x 128 tiles.  Both operands are wanted with their rows as the reduction, which is what the
// transposing LDS read gives: sixteen lanes that point at four rows of sixteen columns receive four rows of one column each.  A row of the tile
// is padded by 64 bytes, so that four rows lie on different banks.
// Eight wavefronts: two groups of four take one half of the slice's rows each, every wavefront a quarter of the tile; the second group hands its
// sums over through LDS at the end, so a slice is one copy of the gradient.  A stage is 32 rows, the next one's pieces are in flight over the
// products and go to the other buffer behind them: one barrier per stage.  The pieces of two stages are on their way at a time.
// 65536 rows, against the products of transposes that this replaces: 512 x 512 63 -> 50 us (34 GFLOP, 28 us at the rate of a large product; 134
// MB of operands, 26), 512 x 128 and 128 x 512 33 and 29 -> 24, and the sum of half as many slices 26 -> 24.  128 x 256 tiles take 48 us and
// leave twice the slices; two workgroups per CU on half the rows each take 52.  Whole gradient of 68-512-512-512-20: 392 -> 336 us.
typedef short s16x4_t __attribute__((ext_vector_type(4)));
constexpr int kCwRows = 32, kCwStride = 2 * 128 + 64 /* bytes */, kCwLds = 2 * 2 * 2 * kCwRows * kCwStride;  // group, buffer, operand

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void chain_wgrad_kernel(int64_t Mp, int np, int ldb, int kp, int kslice, const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                        float* __restrict__ C) {
  constexpr int S = kCwStride, BUF = 2 * kCwRows * S, NP = kCwRows * 16 / 256;  // a stage; 16-byte pieces of an operand's stage per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char mlp_lds[];
  // Workgroup l runs on XCD l % 8: the tiles of one slice, which read the same rows, go to one XCD
  int tile = blockIdx.x, z = blockIdx.y;
  {
    const int l = blockIdx.y * gridDim.x + blockIdx.x, q = l >> 3;
    tile = q % gridDim.x;
    z = (q / gridDim.x) * 8 + (l & 7);
  }
  const int tiles_j = ldb / 128, i0 = tile / tiles_j * 128, j0 = tile % tiles_j * 128;
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), t = threadIdx.x & 255, wave = t >> 6, lane = t & 63;
  const int64_t zbeg = min(Mp, (int64_t)z * kslice), zend = min(Mp, zbeg + kslice);
  const int half = (int)((zend - zbeg) / 2), stages = half / kCwRows;  // an even number of whole stages, the same for both groups
  const int64_t kbeg = zbeg + grp * half;
  unsigned char* buf = mlp_lds + grp * 2 * BUF;
  f32x16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  const int row = t >> 4, piece = t & 15;  // the thread's pieces of a stage: rows `row` and row + 16
  const unsigned oa = row * np + 8 * piece, ob = row * ldb + 8 * piece;
  u32x4 ra[2][NP], rb[2][NP];
  auto fetch = [&](int n, u32x4 (&ra)[NP], u32x4 (&rb)[NP]) __attribute__((always_inline)) {
    const int64_t k0 = kbeg + (int64_t)min(n, stages - 1) * kCwRows;
#pragma unroll
    for (int u = 0; u < NP; ++u) ra[u] = *reinterpret_cast<const u32x4*>(A + (k0 + 16 * u) * np + i0 + oa);
#pragma unroll
    for (int u = 0; u < NP; ++u) rb[u] = *reinterpret_cast<const u32x4*>(B + (k0 + 16 * u) * ldb + j0 + ob);
  };
  auto put = [&](unsigned char* to, const u32x4 (&ra)[NP], const u32x4 (&rb)[NP]) __attribute__((always_inline)) {
    to += row * S + 16 * piece;
#pragma unroll
    for (int u = 0; u < NP; ++u) *reinterpret_cast<u32x4*>(to + 16 * u * S) = ra[u];
#pragma unroll
    for (int u = 0; u < NP; ++u) *reinterpret_cast<u32x4*>(to + (kCwRows + 16 * u) * S) = rb[u];
  };
  // lane's part of a fragment of 32 columns and 16 rows: column lane % 32, rows 8 (lane / 32) + 0..7, four per read
  const int frow = 8 * (lane >> 5) + ((lane & 15) >> 2), fcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  typedef s16x4_t __attribute__((address_space(3))) * lds_quad;
  auto frag = [&](const unsigned char* at) __attribute__((always_inline)) {
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_quad)(at)), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_quad)(at + 4 * S));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * 64;
  if (stages > 0) {
    fetch(0, ra[0], rb[0]);
    fetch(1, ra[1], rb[1]);
    put(buf, ra[0], rb[0]);
  }
  for (int n = 0; n < stages; n += 2)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    fetch(n + u + 2, ra[u], rb[u]);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // LDS only: the requested pieces stay in flight
    const unsigned char* from = buf + u * BUF;
    bf16x8 fa[kCwRows / 16][2], fb[kCwRows / 16][2];
#pragma unroll
    for (int s = 0; s < kCwRows / 16; ++s) {
#pragma unroll
      for (int a = 0; a < 2; ++a) fa[s][a] = frag(from + (16 * s + frow) * S + 2 * (wi + 32 * a + fcol));
#pragma unroll
      for (int b = 0; b < 2; ++b) fb[s][b] = frag(from + (kCwRows + 16 * s + frow) * S + 2 * (wj + 32 * b + fcol));
    }
#pragma unroll
    for (int s = 0; s < kCwRows / 16; ++s)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s][a], fb[s][b], acc[a][b], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    put(buf + (1 - u) * BUF, ra[1 - u], rb[1 - u]);  // the last one's is not read
  }
  // the second group's sums, a row of matrix tiles at a time
  float* mine = reinterpret_cast<float*>(mlp_lds) + t;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    __syncthreads();
    if (grp == 1)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(16 * b + r) * 256] = acc[a][b][r];
    __syncthreads();
    if (grp == 0)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] += mine[(16 * b + r) * 256];
  }
  if (grp == 1) return;
  float* out = C + (int64_t)z * np * kp;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int gj = j0 + wj + 32 * b + (lane & 31);
      if (gj >= kp) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) out[(int64_t)(i0 + wi + 32 * a + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kp + gj] = acc[a][b][r];
    }
}

struct DevMlp {
  int n_layers, activation, dtype;
  int dims[KS_MAX_LAYERS + 1];
  int kpad[KS_MAX_LAYERS];  // padded input width of layer l
  int npad[KS_MAX_LAYERS];  // padded output width of layer l
  void* W[KS_MAX_LAYERS];   // one allocation per layer: W, b and, where there are any, Wp and bp
  float* b[KS_MAX_LAYERS];
  // whole-network and small-batch kernels (every padded width <= kFusedMaxWidth): weights re-ordered into MFMA fragments
  int fused;                    // 1: the whole-network kernel runs this network (the tables below also serve single fp32 layers over few rows)
  int fk[KS_MAX_LAYERS];        // K steps per layer, of 16 (bf16) or 8 (fp32)
  int fn[KS_MAX_LAYERS];        // 32-wide output tiles per layer
  int lda;                      // LDS row stride of the activation tile, in elements
  void* Wp[KS_MAX_LAYERS];      // [tile][k step][lane] x 16 bytes
  float* bp[KS_MAX_LAYERS];     // bias padded to 32 * fn
  // training state (ks_mlp_train_init): fp32 master weights in the padded (npad, kpad) layout, their gradients
  // and Adam moments, and the transposed working copy that the input-gradient GEMM reads
  int train;
  float *mW[KS_MAX_LAYERS], *mb[KS_MAX_LAYERS];
  float *gW[KS_MAX_LAYERS], *gb[KS_MAX_LAYERS];
  float *m1W[KS_MAX_LAYERS], *m2W[KS_MAX_LAYERS], *m1b[KS_MAX_LAYERS], *m2b[KS_MAX_LAYERS];
  void* Wt[KS_MAX_LAYERS];      // (kpad, npad) working-precision transpose
  void* WtP[KS_MAX_LAYERS];     // whole-network kernel only, l >= 1 or a single layer: W_l^T in fragment order, for the input gradients
  int chain_saved;              // the last training forward kept what the whole-network backward pass reads
  int bias_frozen[KS_MAX_LAYERS];  // leading bias entries of the layer that the optimiser leaves alone
  float* zero_bias;             // zeros, as wide as the widest GEMM output
  double* sq_part;              // kSqBlocks partial sums of squares per gradient tensor (weights and biases of every layer)
};


// ---------------------------------------------------------------- training: the small kernels around the GEMMs
// The three matrix products of a layer's backward pass reuse the layer kernels (mlp_layer_kernel, cut_layer_kernel: Y = X W^T):
//   input gradient   dY_prev = dZ W        : X = dZ (M, npad),      "W" = W^T (kpad, npad)
//   weight gradient  dW = dZ^T Y_prev      : X = dZ^T (npad, Mp),   "W" = Y_prev^T (kpad, Mp), fp32 output
// so what is left are transposes, the activation derivative, column sums and the optimiser.
template <typename T>
__device__ __forceinline__ float to_f32(T v) { return (float)v; }
template <typename T>
__device__ __forceinline__ T from_f32(float v) { return (T)v; }

// fp32 (M, n) -> T (M, ld), zero in the padding columns
template <typename T>
__global__ __launch_bounds__(256) void cast_pad_kernel(int64_t M, int n, int ld, const float* __restrict__ src, T* __restrict__ dst) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * ld) return;
  const int64_t m = idx / ld;
  const int c = (int)(idx - m * ld);
  dst[idx] = from_f32<T>(c < n ? src[m * n + c] : 0.f);
}

// T (M, ld) -> fp32 (M, n): the input gradient in the caller's layout; optionally added to what is there, and rows
// flagged in zero_rows come out as zero (an episode boundary stops the gradient)
template <typename T>
__global__ __launch_bounds__(256) void unpad_cast_kernel(int64_t M, int n, int ld, const T* __restrict__ src, float* __restrict__ dst,
                                                         int accumulate, const uint8_t* __restrict__ zero_rows) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * n) return;
  const int64_t m = idx / n;
  const int c = (int)(idx - m * n);
  if (zero_rows && zero_rows[m]) { dst[idx] = 0.f; return; }
  const float v = to_f32(src[m * ld + c]);
  dst[idx] = accumulate ? dst[idx] + v : v;
}

// (M, ld_src) with C meaningful columns -> (Cpad, Mp) transposed, zero outside (C, M).  S is float or T.
template <typename S, typename T>
__global__ __launch_bounds__(256) void transpose_kernel(int64_t M, int C, int64_t ld_src, const S* __restrict__ src, int Cpad, int64_t Mp,
                                                        T* __restrict__ dst) {
  __shared__ float tile[32][33];
  const int64_t m0 = (int64_t)blockIdx.x * 32;
  const int c0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int64_t m = m0 + r;
    const int c = c0 + tx;
    tile[r][tx] = (m < M && c < C) ? (float)src[m * ld_src + c] : 0.f;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int c = c0 + r;
    const int64_t m = m0 + tx;
    if (c < Cpad && m < Mp) dst[(int64_t)c * Mp + m] = from_f32<T>(tile[tx][r]);
  }
}

// y = gelu(z), tanh form, over a whole (M, ld) buffer
template <typename T>
__global__ __launch_bounds__(256) void gelu_forward_kernel(int64_t n, const T* __restrict__ z, T* __restrict__ y) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const float x = to_f32(z[idx]);
  y[idx] = from_f32<T>(0.5f * x * (1.f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x))));
}

// dZ = dY * gelu'(Z) from the stored pre-activation, written over dY
template <typename T>
__global__ __launch_bounds__(256) void gelu_backward_kernel(int64_t n, const T* __restrict__ z, T* __restrict__ dy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const float x = to_f32(z[idx]);
  const float t = tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x));
  const float d = 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * 0.7978845608028654f * (1.f + 3.f * 0.044715f * x * x);
  dy[idx] = from_f32<T>(to_f32(dy[idx]) * d);
}

// dZ = dY * act'(Z), written over dY; act' is expressed through the stored activation output Y.
template <typename T, int ACT>
__global__ __launch_bounds__(256) void act_backward_kernel(int64_t n, const T* __restrict__ y, T* __restrict__ dy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const float yv = to_f32(y[idx]);
  float d = 1.f;
  if (ACT == KS_ACT_ELU) d = yv > 0.f ? 1.f : yv + 1.f;  // elu'(z) = exp(z) = elu(z) + 1 for z <= 0
  if (ACT == KS_ACT_RELU) d = yv > 0.f ? 1.f : 0.f;
  if (ACT == KS_ACT_TANH) d = 1.f - yv * yv;
  dy[idx] = from_f32<T>(to_f32(dy[idx]) * d);
}

// One pass over the gradient that a layer hands down, fusing what the backward step of the layer below needs:
//   dZ = dY * act'(Y) (in place), its transpose (for the weight-gradient product), the transpose of the stored
//   activation Y (the other operand of the weight-gradient product of the layer above) and the column sums of dZ
//   (the bias gradient, as kColsumSlices partial rows that sum_parts_kernel adds in a fixed order).
// A workgroup owns 64 columns and every kColsumSlices-th tile of 64 rows; tiles go through LDS so that both the
// row-major and the transposed accesses are 16-byte vectors.  Needs C % 64 == 0 and Mp % 64 == 0.
template <typename T, int ACT>
__global__ __launch_bounds__(256) void bwd_prep_kernel(int64_t M, int64_t Mp, int C, const T* __restrict__ y, T* __restrict__ dy,
                                                       T* __restrict__ dzT, T* __restrict__ yT, float* __restrict__ part) {
  constexpr int kPad = sizeof(T) == 2 ? 2 : 1;
  constexpr int kVec = 16 / sizeof(T);        // elements per 16-byte vector
  constexpr int kNv = 16 / kVec;              // vectors per thread and tile (16 elements)
  __shared__ T sdz[64][64 + kPad];
  __shared__ T sy[64][64 + kPad];
  const int t = threadIdx.x;
  const int c0 = blockIdx.x * 64;
  const int r = t >> 2, seg = (t & 3) * 16;
  float acc = 0.f;
  for (int64_t tile = blockIdx.y; tile < Mp / 64; tile += gridDim.y) {
    const int64_t m0 = tile * 64, m = m0 + r;
    T vy[16], vd[16];
    if (m < M) {
#pragma unroll
      for (int k = 0; k < kNv; ++k) {
        reinterpret_cast<uint4*>(vy)[k] = reinterpret_cast<const uint4*>(y + m * C + c0 + seg)[k];
        reinterpret_cast<uint4*>(vd)[k] = reinterpret_cast<const uint4*>(dy + m * C + c0 + seg)[k];
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const float yv = to_f32(vy[k]);
        float d = 1.f;
        if (ACT == KS_ACT_ELU) d = yv > 0.f ? 1.f : yv + 1.f;
        if (ACT == KS_ACT_RELU) d = yv > 0.f ? 1.f : 0.f;
        if (ACT == KS_ACT_TANH) d = 1.f - yv * yv;
        vd[k] = from_f32<T>(to_f32(vd[k]) * d);
      }
#pragma unroll
      for (int k = 0; k < kNv; ++k) reinterpret_cast<uint4*>(dy + m * C + c0 + seg)[k] = reinterpret_cast<uint4*>(vd)[k];
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) { vy[k] = from_f32<T>(0.f); vd[k] = from_f32<T>(0.f); }
    }
    __syncthreads();  // the previous tile's readers are done
#pragma unroll
    for (int k = 0; k < 16; ++k) { sdz[r][seg + k] = vd[k]; sy[r][seg + k] = vy[k]; }
    __syncthreads();
    if (t < 64) {
      float s0 = 0.f;
      for (int rr = 0; rr < 64; ++rr) s0 += to_f32(sdz[rr][t]);
      acc += s0;
    }
    // transposed: this thread writes 16 consecutive rows of column c0 + r
    T od[16], oy[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) { od[k] = sdz[seg + k][r]; oy[k] = sy[seg + k][r]; }
#pragma unroll
    for (int k = 0; k < kNv; ++k) {
      reinterpret_cast<uint4*>(dzT + (int64_t)(c0 + r) * Mp + m0 + seg)[k] = reinterpret_cast<uint4*>(od)[k];
      reinterpret_cast<uint4*>(yT + (int64_t)(c0 + r) * Mp + m0 + seg)[k] = reinterpret_cast<uint4*>(oy)[k];
    }
  }
  if (t < 64) part[(int64_t)blockIdx.y * C + c0 + t] = acc;
}

// column sums of a (M, ld) matrix in two deterministic stages: gridDim.y row slices write partial sums, which
// sum_parts_kernel adds up in a fixed order
constexpr int kColsumSlices = 64;
template <typename T>
__global__ __launch_bounds__(256) void colsum_kernel(int64_t M, int ld, const T* __restrict__ a, float* __restrict__ part) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), g = threadIdx.x >> 6;
  float s = 0.f;
  if (c < ld)
    for (int64_t m = (int64_t)blockIdx.y * 4 + g; m < M; m += 4 * (int64_t)gridDim.y) s += to_f32(a[m * ld + c]);
  red[g][threadIdx.x & 63] = s;
  __syncthreads();
  if (g == 0 && c < ld)
    part[(int64_t)blockIdx.y * ld + c] = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

// out[c] = sum over z of part[z][c] for the few columns of a bias gradient: a workgroup of 64 threads per column adds its nz
// partial sums with a fixed tree (one thread walking them one after the other pays nz dependent load latencies)
__global__ __launch_bounds__(64) void sum_parts_tree_kernel(int64_t n, int nz, const float* __restrict__ part, float* __restrict__ out) {
  __shared__ float red[64];
  const int64_t c = blockIdx.x;
  float s = 0.f;
  for (int z = threadIdx.x; z < nz; z += 64) s += part[(int64_t)z * n + c];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 32; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = red[0];
}

// out[i] = sum over z of part[z][i], z ascending
__global__ __launch_bounds__(256) void sum_parts_kernel(int64_t n, int nz, const float* __restrict__ part, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int z0 = 0; z0 < nz; z0 += 8) {  // eight slices' loads in flight, added in slice order
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = z0 + k < nz ? part[(int64_t)(z0 + k) * n + i] : 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (z0 + k < nz) s += v[k];
  }
  out[i] = s;
}

// Every gradient of a network from its partial sums, in one launch (the whole-network backward pass): weight gradient l =
// the sum of its nz[l] row slices, z ascending as in sum_parts_kernel; bias gradient l = the sum over the row tiles of the
// per-tile column sums, in the order of sum_parts_tree_kernel.
// Bound by memory.  Weights (padded to whole matrix tiles) go four to a thread in 16-byte loads.  A workgroup takes sixteen columns of bias sums, a
// row of them 64 bytes: a wavefront per column fetched 64 rows for 4 bytes of each.  68-512-512-512-20
// over 65536 rows: 25 -> 16.7 us (65 MB of slices).
constexpr int kFinishCols = 16;
struct GradFinishArgs {
  int n_layers, tiles;
  int nz[KS_MAX_LAYERS], nb[KS_MAX_LAYERS];
  int64_t nW[KS_MAX_LAYERS];
  int first_w[KS_MAX_LAYERS + 1], first_b[KS_MAX_LAYERS + 1];  // workgroups of the weights, then of the biases, per layer
  const float *wpart[KS_MAX_LAYERS], *bpart[KS_MAX_LAYERS];
  float *gW[KS_MAX_LAYERS], *gb[KS_MAX_LAYERS];
};
__global__ __launch_bounds__(256) void grad_finish_kernel(GradFinishArgs a) {
  __shared__ float lanes[64][kFinishCols + 1];
  const int nbias = a.first_b[a.n_layers], t = threadIdx.x;
  if ((int)blockIdx.x >= nbias) {  // the biases first: their chains are the longer ones
    const int b = blockIdx.x - nbias;
    int l = 0;
    while (l + 1 < a.n_layers && b >= a.first_w[l + 1]) ++l;
    const int64_t i = ((int64_t)(b - a.first_w[l]) * 256 + t) * 4, n = a.nW[l];
    if (i >= n) return;
    float4 s = {0.f, 0.f, 0.f, 0.f};
    const float* part = a.wpart[l] + i;
    const int nz = a.nz[l];
    for (int z0 = 0; z0 < nz; z0 += 8) {  // eight slices' loads in flight, added in slice order
      float4 v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = z0 + k < nz ? *reinterpret_cast<const float4*>(part + (int64_t)(z0 + k) * n) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (z0 + k < nz) { s.x += v[k].x; s.y += v[k].y; s.z += v[k].z; s.w += v[k].w; }
    }
    *reinterpret_cast<float4*>(a.gW[l] + i) = s;
    return;
  }
  const int b = blockIdx.x;
  int l = 0;
  while (l + 1 < a.n_layers && b >= a.first_b[l + 1]) ++l;
  const int n = a.nb[l], c0 = (b - a.first_b[l]) * kFinishCols, c = t % kFinishCols, k0 = t / kFinishCols;
  {  // thread (column c, k0) is lanes k0, k0 + 16, + 32 and + 48 of the column's sum: lane k adds the tiles k, k + 64, ...
    constexpr int Q = 64 * kFinishCols / 256;
    float s[Q] = {};
    if (c0 + c < n) {
      const float* part = a.bpart[l] + c0 + c;
      for (int z0 = 0; z0 < a.tiles; z0 += 128) {  // two rounds of the lanes in flight
        float v[2][Q];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const int z = z0 + 64 * h + k0 + 16 * q;
            v[h][q] = z < a.tiles ? part[(int64_t)z * n] : 0.f;
          }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < Q; ++q) s[q] += v[h][q];
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) lanes[k0 + 16 * q][c] = s[q];
  }
  __syncthreads();
  const int lane = t & 63;
  for (int cc = t >> 6; cc < kFinishCols; cc += 4) {
    float s = lanes[lane][cc];
    for (int w = 32; w > 0; w >>= 1) s += __shfl_down(s, w);  // lane k adds lane k + w: the same tree for every column
    if (lane == 0 && c0 + cc < n) a.gb[l][c0 + cc] = s;
  }
}


// Sum of squares of gradient buffers, NaNs counted as zero (the optimiser zeroes them first), added to *acc in double.
// Every addition happens in a fixed order (a strided pass per lane, a tree over the lanes, then the partial sums one after
// the other), so the clip factor, and with it a whole update, is the same bits on every run.
constexpr int kSqBlocks = 64;
constexpr int kSqTensors = 64;  // gradient tensors per launch
struct SqTensors {
  const float* g[kSqTensors];
  int64_t n[kSqTensors];
  double* part[kSqTensors];  // kSqBlocks of them
};

__device__ __forceinline__ double block_sqsum(const float* __restrict__ g, int64_t n, int first, int stride, double* red) {
  double s = 0.0;
  for (int64_t i = first; i < n; i += stride) {
    const float v = g[i];
    if (v == v) s += (double)v * (double)v;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  return red[0];
}

// grid (kSqBlocks, tensors): part[tensor][block] = this block's share of the tensor
__global__ __launch_bounds__(256) void sqnorm_parts_kernel(SqTensors t) {
  __shared__ double red[256];
  const double v = block_sqsum(t.g[blockIdx.y], t.n[blockIdx.y], (int)(blockIdx.x * 256 + threadIdx.x), kSqBlocks * 256, red);
  if (threadIdx.x == 0) t.part[blockIdx.y][blockIdx.x] = v;
}

// one workgroup: *acc += every network's partial sums, a wavefront per network, the networks in order
constexpr int kSqNets = 32;
struct SqNets {
  double* acc;
  int nets;
  int n[kSqNets];
  const double* part[kSqNets];
};
__global__ __launch_bounds__(1024) void sqnorm_finish_kernel(SqNets t) {
  __shared__ double sum[kSqNets];
  const int lane = threadIdx.x & 63;
  for (int k = threadIdx.x >> 6; k < t.nets; k += 16) {
    double s = 0.0;
    for (int i = lane; i < t.n[k]; i += 64) s += t.part[k][i];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s += __shfl_down(s, d);
    if (lane == 0) sum[k] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = *t.acc;
    for (int k = 0; k < t.nets; ++k) v += sum[k];
    *t.acc = v;
  }
}

// one workgroup over a whole buffer (small tensors that belong to no network: log standard deviations, head parameters)
__global__ __launch_bounds__(256) void sqnorm_kernel(int64_t n, const float* __restrict__ g, double* __restrict__ acc) {
  __shared__ double red[256];
  const double v = block_sqsum(g, n, (int)threadIdx.x, 256, red);
  if (threadIdx.x == 0) *acc += v;
}

// optax.chain(zero_nans, clip_by_global_norm, add_decayed_weights, scale_by_adam, scale(lr), scale(-1)) on one tensor
__global__ __launch_bounds__(256) void adam_kernel(int64_t n, float* __restrict__ p, const float* __restrict__ g,
                                                  float* __restrict__ m1, float* __restrict__ m2, KsAdamParams a,
                                                  const double* __restrict__ sqnorm) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float gv = g[i];
  if (!(gv == gv)) gv = 0.f;                                       // zero_nans
  if (a.max_grad_norm > 0.f && sqnorm) {                           // clip_by_global_norm
    const float norm = (float)sqrt(*sqnorm);
    if (norm > a.max_grad_norm) gv = gv / norm * a.max_grad_norm;
  }
  gv += a.weight_decay * p[i];                                     // add_decayed_weights
  const float nm1 = a.b1 * m1[i] + (1.f - a.b1) * gv;              // scale_by_adam
  const float nm2 = a.b2 * m2[i] + (1.f - a.b2) * gv * gv;
  m1[i] = nm1;
  m2[i] = nm2;
  const float mhat = nm1 / (1.f - powf(a.b1, (float)a.step));
  const float vhat = nm2 / (1.f - powf(a.b2, (float)a.step));
  p[i] -= a.lr * mhat / (sqrtf(vhat) + a.eps);
}

// fp32 master (npad, kpad) -> working copies: W (npad, kpad), W^T (kpad, npad) and, for the whole-network kernel,
// the fragment-ordered copy [tile][k step][lane][8]
template <typename T>
__global__ __launch_bounds__(256) void refresh_kernel(int npad, int kpad, const float* __restrict__ mW, T* __restrict__ W,
                                                      T* __restrict__ Wt, T* __restrict__ Wp, int fk, int fn,
                                                      __bf16* __restrict__ WtP) {
  constexpr int G = 16 / (int)sizeof(T);  // entries of a lane's fragment
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < (int64_t)npad * kpad) {
    const int o = (int)(idx / kpad), i = (int)(idx - (int64_t)o * kpad);
    const float v = mW[idx];
    W[idx] = from_f32<T>(v);
    if (Wt) Wt[(int64_t)i * npad + o] = from_f32<T>(v);
  }
  if (Wp && idx < (int64_t)fn * fk * 64 * G) {
    const int e = (int)(idx % G), lane = (int)((idx / G) & 63);
    const int64_t js = idx / (64 * G);
    const int st = (int)(js % fk), j = (int)(js / fk);
    const int o = j * 32 + (lane & 31), i = st * 2 * G + (lane >> 5) * G + e;
    Wp[idx] = from_f32<T>((o < npad && i < kpad) ? mW[(int64_t)o * kpad + i] : 0.f);
  }
  if (WtP && idx < (int64_t)((fk + 1) / 2) * (2 * fn) * 64 * 8) {  // the transposed roles: tiles over the inputs, 2 fn steps over the outputs
    const int e = (int)(idx & 7), lane = (int)((idx >> 3) & 63);
    const int64_t js = idx >> 9;
    const int st = (int)(js % (2 * fn)), j = (int)(js / (2 * fn));
    const int i = j * 32 + (lane & 31), o = st * 16 + (lane >> 5) * 8 + e;
    WtP[idx] = (__bf16)((o < npad && i < kpad) ? mW[(int64_t)o * kpad + i] : 0.f);
  }
}

// One optimiser step of several networks in one launch: every weight and bias element goes through the chain of adam_kernel, and the
// workgroup that updates a 32 x 32 tile of a master weight also writes the tile's working copies (W, W^T, the fragment-ordered copies), as
// refresh_kernel does; the transposed ones go through LDS, so that all leave in runs of 64 bytes and more.  The biases of a tile's rows ride
// on the first tile of those rows.  Bound by memory for the large networks (28 bytes of state and up to 10 of copies per weight), by its launch for the
// small ones, of which a recurrent policy has a dozen: actor and critic of 3 x 512 in bf16 2 x 13.5 -> 12.9 us, the twelve networks of a GRU
// policy 12 x 6 -> 10 us.
constexpr int kOptLayers = 24;  // layers per launch
struct AdamLayer {
  int npad, kpad, fk, fn, frozen, first_block;
  float *mW, *m1W, *m2W, *mb, *m1b, *m2b;
  const float *gW, *gb;
  void *W, *Wt, *Wp;
  __bf16* WtP;
  float *b, *bp;
};
struct AdamTable {
  int n;
  AdamLayer layer[kOptLayers];
};
struct AdamStep {
  float lr, b1, b2, eps, weight_decay, max_grad_norm, c1, c2;  // c1, c2: 1 - b^step
};

__device__ __forceinline__ float adam_element(float p, float g, float& m1, float& m2, const AdamStep& a, float norm) {
  float gv = g;
  if (!(gv == gv)) gv = 0.f;                                       // zero_nans
  if (a.max_grad_norm > 0.f && norm > a.max_grad_norm) gv = gv / norm * a.max_grad_norm;  // clip_by_global_norm
  gv += a.weight_decay * p;                                        // add_decayed_weights
  m1 = a.b1 * m1 + (1.f - a.b1) * gv;                              // scale_by_adam
  m2 = a.b2 * m2 + (1.f - a.b2) * gv * gv;
  const float mhat = m1 / a.c1;
  const float vhat = m2 / a.c2;
  return p - a.lr * mhat / (sqrtf(vhat) + a.eps);
}

// four neighbouring entries in working precision
template <typename T>
__device__ __forceinline__ void store4(T* to, const float (&v)[4]) {
  if constexpr (sizeof(T) == 2) *reinterpret_cast<uint2*>(to) = uint2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
  else *reinterpret_cast<float4*>(to) = float4{v[0], v[1], v[2], v[3]};
}

template <typename T>
__global__ __launch_bounds__(256) void adam_layers_kernel(AdamTable t, AdamStep a, const double* __restrict__ sqnorm) {
  __shared__ float tr[32][33];
  int l = 0;
  while (l + 1 < t.n && (int)blockIdx.x >= t.layer[l + 1].first_block) ++l;
  const AdamLayer& n = t.layer[l];
  const int tile = (int)blockIdx.x - n.first_block, ti = n.kpad / 32, o0 = tile / ti * 32, i0 = (tile - tile / ti * ti) * 32;
  const float norm = a.max_grad_norm > 0.f && sqnorm ? (float)sqrt(*sqnorm) : 0.f;
  constexpr int G = 16 / (int)sizeof(T);  // entries of a lane's fragment
  const int x = threadIdx.x >> 3, y = (threadIdx.x & 7) * 4;
  {
    const int o = o0 + x, i = i0 + y;
    const int64_t idx = (int64_t)o * n.kpad + i;
    const float4 p4 = *reinterpret_cast<const float4*>(n.mW + idx), g4 = *reinterpret_cast<const float4*>(n.gW + idx);
    float4 m14 = *reinterpret_cast<const float4*>(n.m1W + idx), m24 = *reinterpret_cast<const float4*>(n.m2W + idx);
    float v[4];
    v[0] = adam_element(p4.x, g4.x, m14.x, m24.x, a, norm);
    v[1] = adam_element(p4.y, g4.y, m14.y, m24.y, a, norm);
    v[2] = adam_element(p4.z, g4.z, m14.z, m24.z, a, norm);
    v[3] = adam_element(p4.w, g4.w, m14.w, m24.w, a, norm);
    *reinterpret_cast<float4*>(n.m1W + idx) = m14;
    *reinterpret_cast<float4*>(n.m2W + idx) = m24;
    *reinterpret_cast<float4*>(n.mW + idx) = float4{v[0], v[1], v[2], v[3]};
    store4<T>(reinterpret_cast<T*>(n.W) + idx, v);
    // [tile o / 32][k step i / 2G][lane (o % 32) + 32 ((i % 2G) / G)][i % G], G = 8 (bf16) or 4 (fp32).  The fragment copy is padded to
    // 32 outputs and 2G inputs, the master to the coarser tiles of the per-layer kernel: master entries beyond the fragment copy are padding
    // (zero weights with zero gradients) and have no place in it.
    if (n.Wp && o < n.fn * 32 && i < n.fk * 2 * G)
      store4<T>(reinterpret_cast<T*>(n.Wp) + (((int64_t)(o >> 5) * n.fk + i / (2 * G)) * 64 + (o & 31) + 32 * ((i / G) & 1)) * G + i % G, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) tr[y + e][x] = v[e];
  }
  if (n.Wt || n.WtP) {  // the same for the whole workgroup
    __syncthreads();
    const int i = i0 + x, o = o0 + y;
    const float v[4] = {tr[x][y], tr[x][y + 1], tr[x][y + 2], tr[x][y + 3]};
    if (n.Wt) store4<T>(reinterpret_cast<T*>(n.Wt) + (int64_t)i * n.npad + o, v);
    if (n.WtP && o < n.fn * 32 && i < n.fk * 2 * G)  // the fragment copy with the roles of input and output exchanged
      store4<__bf16>(n.WtP + ((((int64_t)(i >> 5) * (2 * n.fn) + (o >> 4)) * 64 + (i & 31) + 32 * ((o >> 3) & 1)) << 3) + (o & 7), v);
  }
  if (i0 == 0 && threadIdx.x < 32) {
    const int o = o0 + (int)threadIdx.x;
    float v = n.mb[o];
    if (o >= n.frozen) {
      float m1 = n.m1b[o], m2 = n.m2b[o];
      v = adam_element(v, n.gb[o], m1, m2, a, norm);
      n.m1b[o] = m1; n.m2b[o] = m2; n.mb[o] = v;
    }
    n.b[o] = v;
    if (n.bp && o < n.fn * 32) n.bp[o] = v;
  }
}

static inline int round_up(int x, int m) { return (x + m - 1) / m * m; }

static uint16_t f32_to_bf16_rne(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

template <typename T, bool FIRST, bool LAST, int BM, int BN, int WAVES_M, int WAVES_N>
static int launch_layer_tile(int act, hipStream_t s, int64_t M, int npad, int K, int Kreal, int Nreal, const void* x,
                             int64_t ldx, const void* W, const float* b, void* y, int64_t ldy, int ksplit = 1) {
  constexpr int BK = 64, PAD = 8;
  constexpr int lds = (int)sizeof(T) * (BM + BN) * (BK + PAD);
  const dim3 grid((unsigned)((M + BM - 1) / BM), (unsigned)(npad / BN), (unsigned)ksplit);
  const dim3 block(64 * WAVES_M * WAVES_N);
#define KS_LAUNCH(A)                                                                                           \
  {                                                                                                            \
    auto kfn = mlp_layer_kernel<T, FIRST, LAST, A, BM, BN, WAVES_M, WAVES_N>;                                  \
    if (lds > 64 * 1024 &&                                                                                     \
        hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)  \
      return fail(KS_ELAUNCH, "ks_mlp_forward: cannot raise the LDS limit to %d bytes", lds);                  \
    hipLaunchKernelGGL(kfn, grid, block, lds, s, M, K, Kreal, Nreal, x, ldx, (const T*)W, b, y, ldy);          \
  }
  if (LAST) { KS_LAUNCH(KS_ACT_NONE) return KS_OK; }
  switch (act) {
    case KS_ACT_ELU: KS_LAUNCH(KS_ACT_ELU) break;
    case KS_ACT_RELU: KS_LAUNCH(KS_ACT_RELU) break;
    case KS_ACT_TANH: KS_LAUNCH(KS_ACT_TANH) break;
    case KS_ACT_GELU: KS_LAUNCH(KS_ACT_GELU) break;
    default: KS_LAUNCH(KS_ACT_NONE) break;
  }
#undef KS_LAUNCH
  return KS_OK;
}

// fp32 layers.  128-row tiles from one and a half per CU on: fewer leave CUs idle (25600 x 512 -> 128, 200 tiles: 39.7 us of 64-row tiles'
// 34.3; 51200, 400 tiles: 62.2 of 74.2; 16384 x 128 -> 512, 512 tiles: 22.5 of 24.4).
static int launch_layer_f32(int act, hipStream_t s, int64_t M, int npad, int K, int Kreal, int Nreal, const void* x, int64_t ldx, const void* W,
                            const float* b, void* y, int64_t ldy, int ksplit = 1) {
  const bool small = (M + 127) / 128 * (npad / kBN) * ksplit < 400;
  const bool va = ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && Kreal % 4 == 0;
  auto kfn = small ? (va ? cut_layer_kernel<64, true> : cut_layer_kernel<64, false>)
                   : (va ? cut_layer_kernel<128, true> : cut_layer_kernel<128, false>);
  const int bm = small ? 64 : 128;
  hipLaunchKernelGGL(kfn, dim3((unsigned)((M + bm - 1) / bm), (unsigned)(npad / kBN), (unsigned)ksplit), dim3(256), 0, s, M, K, Kreal, Nreal,
                     (const float*)x, ldx, (const float*)W, b, (float*)y, ldy, act);
  return KS_OK;
}

// bf16 tile choice.  Large batches take the whole layer width per workgroup (BN = 512 or 256) so that the activations
// are read from HBM once per layer; small (rollout-sized) batches take 64 x 128 tiles so that the grid still
// covers the 256 CUs more than once.
template <typename T, bool FIRST, bool LAST>
static int launch_layer(int act, hipStream_t s, int64_t M, int npad, int K, int Kreal, int Nreal, const void* x,
                        int64_t ldx, const void* W, const float* b, void* y, int64_t ldy) {
#define KS_ARGS act, s, M, npad, K, Kreal, Nreal, x, ldx, W, b, y, ldy
  if constexpr (sizeof(T) == 4) {
    // between layers the rows are as wide as the padded layer, and so is the reduction
    return launch_layer_f32(LAST ? KS_ACT_NONE : act, s, M, npad, K, FIRST ? Kreal : K, LAST ? Nreal : npad, x, ldx, W, b, y, ldy);
  } else {
    if (M >= 32768 && npad % 512 == 0) return launch_layer_tile<T, FIRST, LAST, 128, 512, 2, 4>(KS_ARGS);
    if (M >= 32768 && npad % 256 == 0) return launch_layer_tile<T, FIRST, LAST, 128, 256, 2, 2>(KS_ARGS);
    if (M * (npad / kBN) <= 128 * 512) return launch_layer_tile<T, FIRST, LAST, 64, 128, 2, 2>(KS_ARGS);
    return launch_layer_tile<T, FIRST, LAST, 128, 128, 2, 2>(KS_ARGS);
  }
#undef KS_ARGS
}

}  // namespace ks

using namespace ks;

struct KsMlp {
  DevMlp m;
  std::vector<float> host_w[KS_MAX_LAYERS], host_b[KS_MAX_LAYERS];  // the caller's fp32 parameters, for ks_mlp_train_init
};

extern "C" int ks_mlp_create(const KsMlpDesc* d, KsMlp** out) {
  if (!d || !out) return fail(KS_EINVAL, "ks_mlp_create: null argument");
  if (d->n_layers < 1 || d->n_layers > KS_MAX_LAYERS) return fail(KS_ELIMIT, "ks_mlp_create: %d layers (1..%d)", d->n_layers, KS_MAX_LAYERS);
  if (d->dtype != KS_MLP_F32 && d->dtype != KS_MLP_BF16) return fail(KS_EINVAL, "ks_mlp_create: unknown dtype");
  if (d->activation < KS_ACT_NONE || d->activation > KS_ACT_GELU) return fail(KS_EINVAL, "ks_mlp_create: unknown activation");
  for (int l = 0; l <= d->n_layers; ++l)
    if (d->dims[l] < 1 || d->dims[l] > 65536) return fail(KS_EINVAL, "ks_mlp_create: bad width %d", d->dims[l]);
  KsMlp* h = new KsMlp();
  DevMlp& m = h->m;
  std::memset(&m, 0, sizeof(m));
  m.n_layers = d->n_layers; m.activation = d->activation; m.dtype = d->dtype;
  const int bk = d->dtype == KS_MLP_BF16 ? 64 : 32;
  const size_t esz = d->dtype == KS_MLP_BF16 ? 2 : 4;
  for (int l = 0; l <= d->n_layers; ++l) m.dims[l] = d->dims[l];
  // Beside the row-major copy of the weights a fragment-ordered one, for the whole-network kernel and the small-batch kernel.  A single fp32 layer
  // over many rows stays with the per-layer kernel (fused = 0): there is nothing to keep on chip between layers, and its output rows leave in
  // longer runs.  fp32 networks with GELU stay with it, too: the backward pass needs their pre-activations, which the whole-network kernel does not
  // keep, and inference has to give the training forward's bits: the ratio of a policy update's first step is exactly one (68-256-256-20, 4096
  // rows: 39 us, 22 on the whole-network kernel).
  bool fusable = d->dtype == KS_MLP_BF16 || d->n_layers == 1 || d->activation != KS_ACT_GELU;
  for (int l = 0; l <= d->n_layers && fusable; ++l)
    if (round_up(d->dims[l], 32) > kFusedMaxWidth) fusable = false;
  const int G = 16 / (int)esz, sk = 2 * G;  // entries of a lane's fragment, k per step
  int kmax = 0;
  for (int l = 0; l < d->n_layers; ++l) {
    if (!d->weights[l] || !d->biases[l]) { ks_mlp_destroy(h); return fail(KS_EINVAL, "ks_mlp_create: layer %d has no weights", l); }
    const int out = d->dims[l + 1], in = d->dims[l];
    h->host_w[l].assign(d->weights[l], d->weights[l] + (size_t)out * in);
    h->host_b[l].assign(d->biases[l], d->biases[l] + out);
    m.npad[l] = round_up(out, kBN);
    // hidden activations are stored with the producer's padded width, so the consumer's K equals it
    m.kpad[l] = l == 0 ? round_up(in, bk) : m.npad[l - 1];
    if (fusable) {
      m.fn[l] = round_up(out, 32) / 32;
      m.fk[l] = (l == 0 ? round_up(in, sk) : m.fn[l - 1] * 32) / sk;
      kmax = m.fk[l] * sk > kmax ? m.fk[l] * sk : kmax;
      if (l + 1 < d->n_layers && m.fn[l] * 32 > kmax) kmax = m.fn[l] * 32;
    }
    // one allocation and one upload per layer: weights, biases and, where there are any, their fragment-ordered copies
    const size_t nw = (size_t)m.npad[l] * m.kpad[l], np = (size_t)m.fn[l] * m.fk[l] * 64 * G;
    auto up = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
    const size_t at_b = up(nw * esz), at_wp = at_b + up((size_t)m.npad[l] * 4), at_bp = at_wp + up(np * esz);
    std::vector<unsigned char> host(at_bp + (size_t)m.fn[l] * 32 * 4, 0);
    for (int o = 0; o < out; ++o) {
      unsigned char* row = host.data() + (size_t)o * m.kpad[l] * esz;
      const float* src = d->weights[l] + (size_t)o * in;
      if (esz == 4) std::memcpy(row, src, (size_t)in * 4);
      else for (int i = 0; i < in; ++i) ((uint16_t*)row)[i] = f32_to_bf16_rne(src[i]);
      if (!fusable) continue;
      // inputs i .. i + G - 1 of output o: [tile o / 32][k step i / sk][lane (o % 32) + 32 ((i % sk) / G)]
      unsigned char* to = host.data() + at_wp + ((size_t)(o >> 5) * m.fk[l] * 64 + (o & 31)) * 16;
      for (int c = 0; c * G < in; ++c)
        std::memcpy(to + ((size_t)(c >> 1) * 64 + 32 * (c & 1)) * 16, row + (size_t)c * 16, (size_t)(in - c * G < G ? in - c * G : G) * esz);
    }
    std::memcpy(host.data() + at_b, d->biases[l], (size_t)out * 4);
    if (fusable) std::memcpy(host.data() + at_bp, d->biases[l], (size_t)out * 4);
    if (hipMalloc(&m.W[l], host.size()) != hipSuccess || hipMemcpy(m.W[l], host.data(), host.size(), hipMemcpyHostToDevice) != hipSuccess) {
      ks_mlp_destroy(h);
      return fail(KS_ELAUNCH, "ks_mlp_create: upload of layer %d failed", l);
    }
    m.b[l] = (float*)((char*)m.W[l] + at_b);
    if (fusable) { m.Wp[l] = (char*)m.W[l] + at_wp; m.bp[l] = (float*)((char*)m.W[l] + at_bp); }
  }
  if (fusable) {
    m.lda = kmax + 16 / (int)esz;  // +16 bytes per row: 16-byte aligned rows that start 4 banks apart
    m.fused = d->dtype == KS_MLP_BF16 || d->n_layers > 1;
  }
  *out = h;
  return KS_OK;
}

namespace ks {
// For the recurrent sequence kernels, which multiply by a one-layer network's weights themselves: the live working-precision
// weight matrix of layer l, (npad, kpad) row-major, and, once ks_mlp_train_init has run, its transpose (kpad, npad).  The
// optimiser step rewrites both in place, so the pointers stay valid for the life of the handle.
int mlp_peek_layer(const KsMlp* h, int l, const void** W, const void** Wt, int* npad, int* kpad, int* dtype) {
  if (!h || l < 0 || l >= h->m.n_layers) return fail(KS_EINVAL, "mlp_peek_layer: no such layer");
  *W = h->m.W[l]; *Wt = h->m.train ? h->m.Wt[l] : nullptr;
  *npad = h->m.npad[l]; *kpad = h->m.kpad[l]; *dtype = h->m.dtype;
  return KS_OK;
}
// fp32 master bias of layer l (training handles), padded to the layer's width; updated in place by the optimiser step
const float* mlp_peek_bias(const KsMlp* h, int l) { return h && h->m.train && l >= 0 && l < h->m.n_layers ? h->m.mb[l] : nullptr; }
}  // namespace ks

extern "C" int ks_mlp_destroy(KsMlp* h) {
  if (!h) return KS_OK;
  for (int l = 0; l < KS_MAX_LAYERS; ++l) {
    if (h->m.W[l]) (void)hipFree(h->m.W[l]);  // the biases and the fragment-ordered copies live behind it
    float* t[] = {h->m.mW[l], h->m.mb[l], h->m.gW[l], h->m.gb[l], h->m.m1W[l], h->m.m2W[l], h->m.m1b[l], h->m.m2b[l]};
    for (float* q : t)
      if (q) (void)hipFree(q);
    if (h->m.Wt[l]) (void)hipFree(h->m.Wt[l]);
  }
  if (h->m.zero_bias) (void)hipFree(h->m.zero_bias);
  if (h->m.sq_part) (void)hipFree(h->m.sq_part);
  delete h;
  return KS_OK;
}

static FusedArgs fused_args(const DevMlp& m, int64_t M, const float* x, float* y) {
  FusedArgs a;
  std::memset(&a, 0, sizeof(a));
  a.M = M; a.n_layers = m.n_layers; a.in_dim = m.dims[0]; a.out_dim = m.dims[m.n_layers]; a.lda = m.lda;
  for (int l = 0; l < m.n_layers; ++l) {
    a.fk[l] = m.fk[l]; a.fn[l] = m.fn[l];
    a.Wp[l] = (const u32x4*)m.Wp[l]; a.bp[l] = m.bp[l];
  }
  a.x = x; a.y = y;
  return a;
}

// A single bf16 layer given by its arguments (no hidden layers, nothing kept), on the row tiles of launch_fused
static int launch_fused_args(const FusedArgs& a, hipStream_t s);

template <typename T, int BM>
static int launch_fused_tile(const DevMlp& m, hipStream_t s, int64_t M, const float* x, float* y, char* const* save,
                             char* save_in = nullptr) {
  FusedArgs a = fused_args(m, M, x, y);
  if (save)
    for (int l = 0; l + 1 < m.n_layers; ++l) {
      a.save[l] = save[l];
      a.save_ld[l] = m.npad[l];
    }
  a.save_rows = M;
  if (save_in) {
    a.save_in = save_in;
    a.save_rows = (M + 127) / 128 * 128;
    a.in_width = round_up(m.kpad[0], kBN);
  }
#ifdef KS_PROFILE
  if (const char* e = getenv("KS_MLP_PROF_PTR")) a.prof = (long long*)strtoull(e, nullptr, 16);
#endif
  const int lds = BM * m.lda * (int)sizeof(T);
  const int64_t blocks = (M + BM - 1) / BM;
  if (blocks > 0x7fffffff) return fail(KS_ELIMIT, "ks_mlp_forward: too many rows");
#define KS_LAUNCH(A)                                                                                           \
  {                                                                                                            \
    auto kfn = sizeof(T) == 2 && save ? mlp_fused_kernel<A, T, BM, false, sizeof(T) == 2> : mlp_fused_kernel<A, T, BM>; \
    if constexpr (sizeof(T) == 2 && BM != 64)                                                                  \
      if (m.n_layers == 1) kfn = mlp_fused_kernel<KS_ACT_NONE, T, BM, true>;                                   \
    if (lds > 64 * 1024 &&                                                                                     \
        hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)  \
      return fail(KS_ELAUNCH, "ks_mlp_forward: cannot raise the LDS limit to %d bytes", lds);                  \
    hipLaunchKernelGGL(kfn, dim3((unsigned)blocks), dim3(64 * kFusedWaves), lds, s, a);                        \
  }
  switch (m.activation) {
    case KS_ACT_ELU: KS_LAUNCH(KS_ACT_ELU) break;
    case KS_ACT_RELU: KS_LAUNCH(KS_ACT_RELU) break;
    case KS_ACT_TANH: KS_LAUNCH(KS_ACT_TANH) break;
    case KS_ACT_GELU: KS_LAUNCH(KS_ACT_GELU) break;
    default: KS_LAUNCH(KS_ACT_NONE) break;
  }
#undef KS_LAUNCH
  return check_launch("ks_mlp_forward");
}

// Row tile: 128 rows amortise each weight fragment over four MFMAs; smaller batches take smaller tiles so that
// the grid still reaches every CU.
static int launch_fused(const DevMlp& m, hipStream_t s, int64_t M, const float* x, float* y, char* const* save = nullptr) {
  if (m.dtype == KS_MLP_F32) {
    // 64 rows share a weight fragment between two row tiles where that still leaves every CU a workgroup (and the tile fits LDS: up to
    // 512 wide); the fp32 matrix rate, not the weights' way from L2, bounds both
    if (M >= 64 * 256) return launch_fused_tile<float, 64>(m, s, M, x, y, save);
    return launch_fused_tile<float, 32>(m, s, M, x, y, save);
  }
#ifdef KS_PROFILE
  if (const char* e = getenv("KS_MLP_BM")) {
    const int bm = atoi(e);
    if (bm == 128) return launch_fused_tile<__bf16, 128>(m, s, M, x, y, save);
    if (bm == 64) return launch_fused_tile<__bf16, 64>(m, s, M, x, y, save);
    if (bm == 32) return launch_fused_tile<__bf16, 32>(m, s, M, x, y, save);
  }
#endif
  if (M >= 128 * 256) return launch_fused_tile<__bf16, 128>(m, s, M, x, y, save);
  // a single layer with a lane per feature: 64 rows of it need more than 128 registers (20000 x 128 -> 384: 16.4 us of 12.1), and narrow ones
  // are better off with a lane per row (20000 x 128 -> 20: 4.7 us of 5.5)
  if (M >= 64 * 256 && (m.n_layers > 1 || m.fn[0] <= 2)) return launch_fused_tile<__bf16, 64>(m, s, M, x, y, save);
  return launch_fused_tile<__bf16, 32>(m, s, M, x, y, save);
}

// The row tile that a single bf16 layer takes in the form with a lane per feature, 0 where it takes another form (launch_fused)
static int single_bm(const DevMlp& m, int64_t M) {
  if (!m.fused || m.dtype != KS_MLP_BF16 || m.n_layers != 1) return 0;
  if (M >= 128 * 256) return 128;
  return M >= 64 * 256 && m.fn[0] <= 2 ? 0 : 32;
}

static int launch_fused_args(const FusedArgs& a, hipStream_t s) {
  const int bm = a.M >= 128 * 256 ? 128 : 32, lds = bm * a.lda * 2;
  auto kfn = bm == 128 ? mlp_fused_kernel<KS_ACT_NONE, __bf16, 128, true> : mlp_fused_kernel<KS_ACT_NONE, __bf16, 32, true>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(KS_ELAUNCH, "ks_mlp_train_backward: cannot raise the LDS limit to %d bytes", lds);
  hipLaunchKernelGGL(kfn, dim3((unsigned)((a.M + bm - 1) / bm)), dim3(64 * kFusedWaves), lds, s, a);
  return KS_OK;
}

// Two of them, of one row tile, in one launch
static int launch_single_pair(const FusedArgs& a, const FusedArgs& b, int bm, hipStream_t s) {
  const int lds = bm * (a.lda > b.lda ? a.lda : b.lda) * 2;
  const int64_t ta = (a.M + bm - 1) / bm, tb = (b.M + bm - 1) / bm;
  if (ta + tb > 0x7fffffff) return fail(KS_ELIMIT, "ks_mlp: too many rows");
  auto kfn = bm == 128 ? mlp_single_pair_kernel<128> : mlp_single_pair_kernel<32>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(KS_ELAUNCH, "ks_mlp: cannot raise the LDS limit to %d bytes", lds);
  hipLaunchKernelGGL(kfn, dim3((unsigned)(ta + tb)), dim3(64 * kFusedWaves), lds, s, a, b, (unsigned)ta);
  return KS_OK;
}

template <typename T, int BM>
static int launch_fused_pair_tile(const DevMlp& m0, const DevMlp& m1, hipStream_t s, int64_t M, const float* x0, float* y0,
                                  const float* x1, float* y1, const KsActionSample& sample) {
  const FusedArgs a = fused_args(m0, M, x0, y0), b = fused_args(m1, M, x1, y1);
  const int lds = BM * (m0.lda > m1.lda ? m0.lda : m1.lda) * (int)sizeof(T);
  const int64_t blocks = (M + BM - 1) / BM;
  if (blocks > 0x7fffffff) return fail(KS_ELIMIT, "ks_mlp_forward_pair: too many rows");
#define KS_LAUNCH(A)                                                                                           \
  {                                                                                                            \
    auto kfn = mlp_fused_pair_kernel<A, T, BM>;                                                                \
    if (lds > 64 * 1024 &&                                                                                     \
        hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)  \
      return fail(KS_ELAUNCH, "ks_mlp_forward_pair: cannot raise the LDS limit to %d bytes", lds);             \
    hipLaunchKernelGGL(kfn, dim3((unsigned)blocks, 2), dim3(64 * kFusedWaves), lds, s, a, b, sample);          \
  }
  switch (m0.activation) {
    case KS_ACT_ELU: KS_LAUNCH(KS_ACT_ELU) break;
    case KS_ACT_RELU: KS_LAUNCH(KS_ACT_RELU) break;
    case KS_ACT_TANH: KS_LAUNCH(KS_ACT_TANH) break;
    case KS_ACT_GELU: KS_LAUNCH(KS_ACT_GELU) break;
    default: KS_LAUNCH(KS_ACT_NONE) break;
  }
#undef KS_LAUNCH
  return check_launch("ks_mlp_forward_pair");
}

// Whether M rows go through the small-batch kernel.  Networks of several layers: up to 2048 rows (one tile per SIMD at 512 wide) where the
// whole-network kernel gives its wavefronts two tiles of a layer (68-512-512-512-20: 83 -> 52 us at 256 rows, 61 at 2048; 256 wide it takes 30
// to this one's 40).  Single layers: up to 1024 tiles, one per SIMD; past that the reuse in the per-layer kernel's larger tiles wins
// (128 -> 512: 8.1 us of 9.0 at 2048 rows, 12.4 of 10.1 at 4096; 475 -> 128: 31 of 27 at 8192 rows, 53 of 30 at 16384; 128 -> 40: 7.0 of 8.2
// at 4096).
constexpr int64_t kSmallRows = 2048;
static bool small_ok(const DevMlp& m, int64_t M) {
  if (m.dtype != KS_MLP_F32 || !m.Wp[0]) return false;
  if (m.n_layers == 1) return (M + 31) / 32 * m.fn[0] <= 1024;
  int wide = 0;
  for (int l = 0; l + 1 < m.n_layers; ++l) wide = m.fn[l] > wide ? m.fn[l] : wide;
  return wide > kFusedWaves && M <= kSmallRows;
}

static int64_t small_ws_floats(const DevMlp& m, int64_t M) {  // two buffers of hidden activations
  int wide = 0;
  for (int l = 0; l + 1 < m.n_layers; ++l) wide = m.fn[l] * 32 > wide ? m.fn[l] * 32 : wide;
  return (M * wide + 63) / 64 * 64;
}

static SmallLayer small_layer(const DevMlp& m, int64_t M, int l, const float* x, float* y, float* ws) {
  const bool last = l == m.n_layers - 1;
  const int64_t half = small_ws_floats(m, M);
  SmallLayer p;
  p.x = l == 0 ? x : ws + (l & 1 ? 0 : half);
  p.Kreal = l == 0 ? m.dims[0] : m.fn[l - 1] * 32;
  p.ldx = p.Kreal;
  p.nk = m.fk[l]; p.nt = m.fn[l];
  p.y = last ? y : ws + (l & 1 ? half : 0);
  p.Nreal = last ? m.dims[l + 1] : m.fn[l] * 32;
  p.ldy = p.Nreal;
  p.act = last ? KS_ACT_NONE : m.activation;
  p.vec = p.ldx % 4 == 0 && ((uintptr_t)p.x & 15) == 0;  // then Kreal is at least 4
  p.Wp = (const u32x4*)m.Wp[l]; p.bp = m.bp[l];
  return p;
}

// one network, or two of the same depth over the same number of rows
static int launch_small(const DevMlp& a, const DevMlp* b, hipStream_t s, int64_t M, const float* xa, float* ya, void* wa, const float* xb,
                        float* yb, void* wb) {
  for (int l = 0; l < a.n_layers; ++l) {
    const SmallLayer p = small_layer(a, M, l, xa, ya, (float*)wa), q = b ? small_layer(*b, M, l, xb, yb, (float*)wb) : p;
    const int nets = b ? 2 : 1, nt = p.nt > q.nt ? p.nt : q.nt;
    // the whole-network kernel cuts narrow layers only where it has layers to itself: a single layer is one wavefront's reduction
    const int sa = a.n_layers > 1 && p.nt <= 2 ? fused_share(p.nt, a.lda) : 1, sb = b ? (q.nt <= 2 ? fused_share(q.nt, b->lda) : 1) : sa;
    auto go = [&](int share, const SmallLayer& u, const SmallLayer& v, int n, int tiles) {
      const dim3 grid((unsigned)((tiles * share + 3) / 4), (unsigned)((M + 31) / 32), (unsigned)n);
      if (a.n_layers == 1) {
        hipLaunchKernelGGL(cut_small_kernel, grid, dim3(256), 0, s, M, u);
        return;
      }
      auto kfn = share == 4 ? sgemm_small_kernel<4> : (share == 2 ? sgemm_small_kernel<2> : sgemm_small_kernel<1>);
      hipLaunchKernelGGL(kfn, grid, dim3(256), 0, s, M, u, v);
    };
    if (sa == sb) go(sa, p, q, nets, nt);
    else { go(sa, p, p, 1, p.nt); go(sb, q, q, 1, q.nt); }
  }
  return check_launch("ks_mlp_forward");
}

// Whether M rows of a bf16 network go through the layer-wise kernels for few rows.  The hidden layers have to be wide enough for their
// weights to be worth the second launch (one row of 68-3 x 384-20: 13.9 -> 11.7 us, 68-2 x 384-20: 9.9 -> 9.0, 3 x 352: 13.1
// -> 12.4, 3 x 288: 11.1 -> 11.4, a layer of 320 columns being 10 tiles), and every row tile repeats the first layer in every workgroup,
// which past 256 rows costs a pair of networks more than it gains (512 rows: 17.9 -> 23).
constexpr int64_t kSplitRows = 256;
constexpr int kSplitTiles = 12;
static bool split_ok(const DevMlp& m, int64_t M) {
  if (m.dtype != KS_MLP_BF16 || !m.fused || m.n_layers < 3 || m.fn[m.n_layers - 1] > 2) return false;
  for (int l = 0; l + 1 < m.n_layers; ++l)
    if (m.fn[l] < kSplitTiles) return false;
  return M <= kSplitRows;
}

static int64_t split_ws_bytes(int64_t M) {
  const int64_t tiles = (M + 31) / 32;
  return tiles * (2 * kSplitTile * 16 + 4) + 256;
}

// where the launches of a call keep their activations: two buffers, then the counters
static u32x4* split_buffer(void* ws, int64_t M, int k) {
  return reinterpret_cast<u32x4*>(((uintptr_t)ws + 15) & ~(uintptr_t)15) + k * ((M + 31) / 32) * kSplitTile;
}

static SplitFirst split_first(const DevMlp& m, int64_t M, const float* x, void* ws) {
  return {x, (const u32x4*)m.Wp[0], (const u32x4*)m.Wp[1], m.bp[0], m.bp[1], split_buffer(ws, M, 0), reinterpret_cast<unsigned*>(split_buffer(ws, M, 2)),
          (int)M, m.dims[0], m.lda, m.fk[0], m.fn[0], m.fk[1], m.fn[1]};
}

static SplitLayer split_layer(const DevMlp& m, int64_t M, int l, float* y, void* ws) {
  const int out = m.n_layers - 1;
  const bool ends = l + 1 == out;
  return {split_buffer(ws, M, l & 1), (const u32x4*)m.Wp[l], m.bp[l], l == out ? nullptr : split_buffer(ws, M, (l & 1) ^ 1),
          ends ? (const u32x4*)m.Wp[out] : nullptr, m.bp[out], y, reinterpret_cast<unsigned*>(split_buffer(ws, M, 2)),
          (int)M, m.dims[m.n_layers], m.fk[l], m.fn[l], m.fk[out], m.fn[out]};
}

// one network, or two of the same depth and activation over the same number of rows
static int launch_split(const DevMlp& a, const DevMlp* b, hipStream_t s, int64_t M, const float* xa, float* ya, void* wa, const float* xb,
                        float* yb, void* wb) {
  const SplitFirst p = split_first(a, M, xa, wa), q = b ? split_first(*b, M, xb, wb) : p;
  const unsigned tiles = (unsigned)((M + 31) / 32), nets = b ? 2 : 1;
  auto wide = [&](int l) { return (unsigned)(b && b->fn[l] > a.fn[l] ? b->fn[l] : a.fn[l]); };
  const int lds = 32 * (b && b->lda > a.lda ? b->lda : a.lda) * 2;
#define KS_LAUNCH(A)                                                                                                                     \
  {                                                                                                                                      \
    hipLaunchKernelGGL(mlp_split_first_kernel<A>, dim3(wide(1), tiles, nets), dim3(64 * kFusedWaves), lds, s, p, q);                     \
    for (int l = 2; l == 2 || l + 1 < a.n_layers; ++l) {                                                                                 \
      const SplitLayer u = split_layer(a, M, l, ya, wa), v = b ? split_layer(*b, M, l, yb, wb) : u;                                      \
      hipLaunchKernelGGL(mlp_split_layer_kernel<A>, dim3(wide(l), tiles, nets), dim3(64), 0, s, u, v);                                   \
    }                                                                                                                                    \
  }
  switch (a.activation) {
    case KS_ACT_ELU: KS_LAUNCH(KS_ACT_ELU) break;
    case KS_ACT_RELU: KS_LAUNCH(KS_ACT_RELU) break;
    case KS_ACT_TANH: KS_LAUNCH(KS_ACT_TANH) break;
    case KS_ACT_GELU: KS_LAUNCH(KS_ACT_GELU) break;
    default: KS_LAUNCH(KS_ACT_NONE) break;
  }
#undef KS_LAUNCH
  return check_launch("ks_mlp_forward");
}

// Whether two pieces of memory share a float
struct Span {
  const float* p;
  int64_t n;
};
static bool meet(Span a, Span b) { return a.p && b.p && (uintptr_t)a.p < (uintptr_t)(b.p + b.n) && (uintptr_t)b.p < (uintptr_t)(a.p + a.n); }

// `sample`: what the launch also makes of the first network's output where the two share one; its `action` is NULL on return then
static int forward_pair(const KsMlp* h0, const KsMlp* h1, ks_stream_t stream, int64_t M, const float* x0, float* y0, const float* x1, float* y1,
                        void* workspace0, void* workspace1, KsActionSample& sample) {
  if (!h0 || !h1) return fail(KS_EINVAL, "ks_mlp_forward_pair: null handle");
  if (M < 0) return fail(KS_EINVAL, "ks_mlp_forward_pair: negative row count");
  if (M == 0) return KS_OK;
  if (!x0 || !y0 || !x1 || !y1) return fail(KS_EINVAL, "ks_mlp_forward_pair: null pointer");
  if (y0 == y1) return fail(KS_EINVAL, "ks_mlp_forward_pair: the two outputs must differ");
  hipStream_t s = (hipStream_t)stream;
  const Span in0 = {x0, M * h0->m.dims[0]}, in1 = {x1, M * h1->m.dims[0]}, out0 = {y0, M * h0->m.dims[h0->m.n_layers]},
             out1 = {y1, M * h1->m.dims[h1->m.n_layers]};
  if (meet(out0, in1) || meet(out1, in0) || meet(out0, out1)) {  // e.g. the second reads what the first writes: one after the other
    const int rc = ks_mlp_forward(h0, stream, M, x0, y0, workspace0);
    return rc != KS_OK ? rc : ks_mlp_forward(h1, stream, M, x1, y1, workspace1);
  }
  if (small_ok(h0->m, M) && small_ok(h1->m, M) && h0->m.n_layers == h1->m.n_layers && h0->m.n_layers > 1 && workspace0 && workspace1 &&
      workspace0 != workspace1)
    return launch_small(h0->m, &h1->m, s, M, x0, y0, workspace0, x1, y1, workspace1);
  if (split_ok(h0->m, M) && split_ok(h1->m, M) && h0->m.n_layers == h1->m.n_layers && h0->m.activation == h1->m.activation && workspace0 &&
      workspace1 && workspace0 != workspace1)
    return launch_split(h0->m, &h1->m, s, M, x0, y0, workspace0, x1, y1, workspace1);
  // single layers
  if (const int bm = single_bm(h0->m, M); bm && bm == single_bm(h1->m, M)) {
    const int rc = launch_single_pair(fused_args(h0->m, M, x0, y0), fused_args(h1->m, M, x1, y1), bm, s);
    return rc != KS_OK ? rc : check_launch("ks_mlp_forward_pair");
  }
  // one launch when both networks run as whole-network kernels with the same activation and row tile; else one each
  if (h0->m.fused && h1->m.fused && h0->m.activation == h1->m.activation && h0->m.dtype == h1->m.dtype && M < 64 * 256) {
    KsActionSample with = sample;
    // actions over rows that another workgroup has yet to read or write, and deviations or noise that the networks write, wait for both networks
    const Span act = {sample.action, out0.n}, noise = {sample.noise_normal, out0.n}, dev = {sample.log_std, h0->m.dims[h0->m.n_layers]};
    bool apart = act.p != out0.p && meet(act, out0);
    for (const Span& x : {in0, in1, out1}) apart |= meet(act, x);
    for (const Span& y : {out0, out1}) apart |= meet(noise, y) || meet(dev, y);
    (apart ? with : sample).action = nullptr;
    if (h0->m.dtype == KS_MLP_F32) return launch_fused_pair_tile<float, 32>(h0->m, h1->m, s, M, x0, y0, x1, y1, with);
    return launch_fused_pair_tile<__bf16, 32>(h0->m, h1->m, s, M, x0, y0, x1, y1, with);
  }
  const int rc = ks_mlp_forward(h0, stream, M, x0, y0, workspace0);
  if (rc != KS_OK) return rc;
  return ks_mlp_forward(h1, stream, M, x1, y1, workspace1);
}

extern "C" int ks_mlp_forward_pair(const KsMlp* h0, const KsMlp* h1, ks_stream_t stream, int64_t M, const float* x0,
                                   float* y0, const float* x1, float* y1, void* workspace0, void* workspace1) {
  KsActionSample none = {};
  return forward_pair(h0, h1, stream, M, x0, y0, x1, y1, workspace0, workspace1, none);
}

extern "C" int ks_mlp_forward_pair_sample(const KsMlp* actor, const KsMlp* critic, ks_stream_t stream, int64_t M, const float* x0, float* y0,
                                          const float* x1, float* y1, void* workspace0, void* workspace1, const KsActionSample* sample) {
  if (!sample || (M > 0 && !sample->action)) return fail(KS_EINVAL, "ks_mlp_forward_pair_sample: null pointer");
  KsActionSample left = *sample;
  const int rc = forward_pair(actor, critic, stream, M, x0, y0, x1, y1, workspace0, workspace1, left);
  if (rc != KS_OK || M <= 0 || !left.action) return rc;
  return ks_sample_action(stream, M, actor->m.dims[actor->m.n_layers], y0, left.log_std, left.noise_normal, left.rng, left.clip_max, left.action);
}

extern "C" int ks_mfma_yardstick(ks_stream_t stream, int32_t workgroups, int32_t iters, float* out, int64_t* stamps) {
  if (workgroups < 1 || iters < 1) return fail(KS_EINVAL, "ks_mfma_yardstick: workgroups and iterations must be positive");
  if (!out) return fail(KS_EINVAL, "ks_mfma_yardstick: null output");
  hipLaunchKernelGGL(mfma_yardstick_kernel, dim3((unsigned)workgroups), dim3(256), 0, (hipStream_t)stream, iters, out,
                     reinterpret_cast<long long*>(stamps));
  return check_launch("ks_mfma_yardstick");
}

// Enough for M rows and for any smaller batch: a caller sizes one buffer for its largest batch.  Batches too large for the small-batch
// kernel need nothing themselves, but the smaller ones do.
extern "C" int64_t ks_mlp_workspace_bytes(const KsMlp* h, int64_t M) {
  if (!h || M < 0) return 0;
  const int64_t few = M < kSmallRows ? M : kSmallRows;
  if (h->m.n_layers > 1 && small_ok(h->m, few)) return 2 * 4 * small_ws_floats(h->m, few);
  if (split_ok(h->m, 1)) return split_ws_bytes(M < kSplitRows ? M : kSplitRows);
  if (h->m.fused) return 0;
  int widest = 0;
  for (int l = 0; l + 1 < h->m.n_layers; ++l) widest = h->m.npad[l] > widest ? h->m.npad[l] : widest;
  const int64_t esz = h->m.dtype == KS_MLP_BF16 ? 2 : 4;
  return 2 * M * widest * esz + 256;
}

extern "C" int ks_mlp_forward(const KsMlp* h, ks_stream_t stream, int64_t M, const float* x, float* y, void* workspace) {
  if (!h) return fail(KS_EINVAL, "ks_mlp_forward: null handle");
  if (M < 0) return fail(KS_EINVAL, "ks_mlp_forward: negative row count");
  if (M == 0) return KS_OK;
  if (!x || !y) return fail(KS_EINVAL, "ks_mlp_forward: null pointer");
  const DevMlp& m = h->m;
  if (small_ok(m, M) && (m.n_layers == 1 || workspace)) return launch_small(m, nullptr, (hipStream_t)stream, M, x, y, workspace, nullptr, nullptr, nullptr);
  if (split_ok(m, M) && workspace) return launch_split(m, nullptr, (hipStream_t)stream, M, x, y, workspace, nullptr, nullptr, nullptr);
  if (m.fused) return launch_fused(m, (hipStream_t)stream, M, x, y);
  if (m.n_layers > 1 && !workspace) return fail(KS_EINVAL, "ks_mlp_forward: workspace required");
  if ((M + kBM - 1) / kBM > 0x7fffffff) return fail(KS_ELIMIT, "ks_mlp_forward: too many rows");
  const int64_t esz = m.dtype == KS_MLP_BF16 ? 2 : 4;
  int widest = 0;
  for (int l = 0; l + 1 < m.n_layers; ++l) widest = m.npad[l] > widest ? m.npad[l] : widest;
  char* buf[2] = {(char*)workspace, (char*)workspace + ((M * widest * esz + 255) / 256) * 256};
  const void* in = x;
  int64_t ldin = m.dims[0];
  hipStream_t s = (hipStream_t)stream;
  for (int l = 0; l < m.n_layers; ++l) {
    const bool first = l == 0, last = l == m.n_layers - 1;
    void* outp = last ? (void*)y : (void*)buf[l & 1];
    const int64_t ldo = last ? m.dims[l + 1] : m.npad[l];
#define KS_GO(T)                                                                                                      \
  if (first && last) rc = launch_layer<T, true, true>(m.activation, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo); \
  else if (first) rc = launch_layer<T, true, false>(m.activation, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);   \
  else if (last) rc = launch_layer<T, false, true>(m.activation, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);    \
  else rc = launch_layer<T, false, false>(m.activation, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);
    int rc = KS_OK;
    if (m.dtype == KS_MLP_BF16) { KS_GO(__bf16) } else { KS_GO(float) }
#undef KS_GO
    if (rc != KS_OK) return rc;
    in = outp;
    ldin = ldo;
  }
  return check_launch("ks_mlp_forward");
}

// ---------------------------------------------------------------------------------------------
// training entry points
// ---------------------------------------------------------------------------------------------
static int widest_pad(const DevMlp& m) {
  int w = 0;
  for (int l = 0; l < m.n_layers; ++l) {
    w = m.npad[l] > w ? m.npad[l] : w;
    w = round_up(m.kpad[l], kBN) > w ? round_up(m.kpad[l], kBN) : w;
  }
  return w;
}

template <typename T>
static void refresh_layers(DevMlp& m, hipStream_t s);

extern "C" int ks_mlp_train_init(KsMlp* h) {
  if (!h) return fail(KS_EINVAL, "ks_mlp_train_init: null handle");
  DevMlp& m = h->m;
  if (m.train) return KS_OK;
  // a failure part way leaves nothing behind: what was allocated so far is released and the handle stays untrained
  auto give_up = [&](const char* what) {
    for (int l = 0; l < KS_MAX_LAYERS; ++l) {
      float** t[] = {&m.mW[l], &m.mb[l], &m.gW[l], &m.gb[l], &m.m1W[l], &m.m2W[l], &m.m1b[l], &m.m2b[l]};
      for (float** q : t) {
        if (*q) (void)hipFree(*q);
        *q = nullptr;
      }
      if (m.Wt[l]) (void)hipFree(m.Wt[l]);
      m.Wt[l] = nullptr;
      m.WtP[l] = nullptr;
    }
    if (m.zero_bias) (void)hipFree(m.zero_bias);
    if (m.sq_part) (void)hipFree(m.sq_part);
    m.zero_bias = nullptr;
    m.sq_part = nullptr;
    m.train = 0;
    return fail(KS_ELAUNCH, "ks_mlp_train_init: %s failed", what);
  };
  const size_t esz = m.dtype == KS_MLP_BF16 ? 2 : 4;
  for (int l = 0; l < m.n_layers; ++l) {
    const size_t n = (size_t)m.npad[l] * m.kpad[l], nb = m.npad[l];
    std::vector<float> w(n, 0.f), b(nb, 0.f);
    for (int o = 0; o < m.dims[l + 1]; ++o) {
      for (int i = 0; i < m.dims[l]; ++i) w[(size_t)o * m.kpad[l] + i] = h->host_w[l][(size_t)o * m.dims[l] + i];
      b[o] = h->host_b[l][o];
    }
    float** wbufs[] = {&m.mW[l], &m.gW[l], &m.m1W[l], &m.m2W[l]};
    float** bbufs[] = {&m.mb[l], &m.gb[l], &m.m1b[l], &m.m2b[l]};
    for (float** q : wbufs)
      if (hipMalloc((void**)q, n * 4) != hipSuccess || hipMemset(*q, 0, n * 4) != hipSuccess) return give_up("allocation");
    for (float** q : bbufs)
      if (hipMalloc((void**)q, nb * 4) != hipSuccess || hipMemset(*q, 0, nb * 4) != hipSuccess) return give_up("allocation");
    if (hipMemcpy(m.mW[l], w.data(), n * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m.mb[l], b.data(), nb * 4, hipMemcpyHostToDevice) != hipSuccess)
      return give_up("upload");
    // the first layer's transpose is padded to whole output tiles of the input-gradient product; the padding stays zero
    const size_t nt = l == 0 ? (size_t)round_up(m.kpad[0], kBN) * m.npad[0] : n;
    size_t np = 0;
    if (m.fused && esz == 2 && (l >= 1 || m.n_layers == 1))  // bf16: (fk / 2, rounded up) tiles of inputs x (2 fn) steps over outputs
      np = (size_t)((m.fk[l] + 1) / 2) * (2 * m.fn[l]) * 512 * 2;
    const size_t ntb = (nt * esz + 255) / 256 * 256;
    if (hipMalloc(&m.Wt[l], ntb + np) != hipSuccess || hipMemset(m.Wt[l], 0, ntb + np) != hipSuccess) return give_up("allocation");
    if (np) m.WtP[l] = (char*)m.Wt[l] + ntb;  // freed with Wt
  }
  const int wz = widest_pad(m);
  if (hipMalloc((void**)&m.zero_bias, (size_t)wz * 4) != hipSuccess || hipMemset(m.zero_bias, 0, (size_t)wz * 4) != hipSuccess)
    return give_up("allocation");
  if (hipMalloc((void**)&m.sq_part, sizeof(double) * kSqBlocks * 2 * KS_MAX_LAYERS) != hipSuccess)
    return give_up("allocation");
  m.train = 1;
  // working copies (among them the transposes, which did not exist yet) from the master weights
  if (m.dtype == KS_MLP_BF16) refresh_layers<__bf16>(m, (hipStream_t)0);
  else refresh_layers<float>(m, (hipStream_t)0);
  if (hipStreamSynchronize((hipStream_t)0) != hipSuccess) return give_up("refresh");
  return KS_OK;
}

template <typename T>
static void refresh_layers(DevMlp& m, hipStream_t s) {
  for (int l = 0; l < m.n_layers; ++l) {
    const int64_t n = (int64_t)m.npad[l] * m.kpad[l];
    const int64_t np = m.Wp[l] ? (int64_t)m.fn[l] * m.fk[l] * 512 : 0;
    const int64_t tot = n > np ? n : np;
    hipLaunchKernelGGL(refresh_kernel<T>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, m.npad[l], m.kpad[l], m.mW[l],
                       (T*)m.W[l], (T*)m.Wt[l], (T*)m.Wp[l], m.fk[l], m.fn[l], (__bf16*)m.WtP[l]);
    (void)hipMemcpyAsync(m.b[l], m.mb[l], (size_t)m.npad[l] * 4, hipMemcpyDeviceToDevice, s);
    if (m.bp[l]) (void)hipMemcpyAsync(m.bp[l], m.mb[l], (size_t)m.fn[l] * 32 * 4, hipMemcpyDeviceToDevice, s);
  }
}

constexpr int kDwSplit = 32;  // slices the weight-gradient reduction over the rows is cut into
// Slices of the whole-network backward pass's weight gradients (chain_wgrad_kernel): a workgroup per CU, at most 64 slices (every slice is a copy
// of the gradient to write and to add up: 65536 x 512 x 512 with 32 instead of 16, 52 us instead of 50 and 27 instead of 24 for the sums) of 512
// rows or more.
static int chain_dw_slices(int np, int kp128, int64_t Mp) {
  int ks = 8;
  while (ks < 64 && ks * (np / 128) * (kp128 / 128) < 256 && Mp >= 1024 * (int64_t)ks) ks *= 2;
  return ks;
}
// Slices of the row reduction of a single layer's weight gradient (wgrad_kernel, 128 x 128 tiles): a workgroup per CU (its registers
// admit no second one), a slice of at least three stages per group, below which the start and the slice sum cost as much as the
// products; a multiple of eight, for the XCD mapping, once there are that many.
static int wgrad_slices(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  int64_t slices = (256 + tiles - 1) / tiles;
  if (slices > K / 192) slices = K / 192;
  if (slices >= 8) slices = slices / 8 * 8;
  return slices > 1 ? (int)slices : 1;
}
constexpr int kDiscMaxSlices = 64;  // most slices of a weight-gradient product of the discriminator (sgemm_kernel)

// workspace: hidden activations of every layer, two (M, widest) gradient buffers, two transposes (widest, Mp)
struct TrainWs {
  char* act[KS_MAX_LAYERS];
  char* pre[KS_MAX_LAYERS];  // pre-activations of the hidden layers, kept only for GELU (not recoverable from its output)
  char *d0, *d1, *t0, *t1, *t2;
  float* part;  // partial sums of the split reductions
  int64_t Mp;
  // whole-network backward pass (chain_ok): the network input as the kernels multiply it, (M, its width in whole 128), per layer dZ in whole
  // 128-row tiles and one row of bias partial sums per tile
  char *in, *dz[KS_MAX_LAYERS];
  float *bpart[KS_MAX_LAYERS], *wpart[KS_MAX_LAYERS];  // wpart: the row slices of each layer's weight-gradient product
  int64_t Mp128;
};

// Whether a batch of M rows goes through the whole-network backward pass: bf16 networks that run the whole-network forward
// kernel on 128-row tiles, with hidden layers wide enough that every wavefront owns whole feature tiles of all four row tiles
// (the accumulator-order copy of the activations is laid out for that split).
static bool chain_ok(const DevMlp& m, int64_t M) {
  if (!m.fused || m.dtype != KS_MLP_BF16 || m.activation == KS_ACT_GELU || m.n_layers < 2 || M < 128 * 256) return false;
  for (int l = 0; l + 1 < m.n_layers; ++l)
    if (m.npad[l] != m.fn[l] * 32 || m.fn[l] * 4 <= kFusedWaves || !m.WtP[l + 1]) return false;
  // the kept input and the output gradient are cut from the LDS tile at their padded widths
  if (round_up(m.kpad[0], kBN) + 8 > m.lda || m.npad[m.n_layers - 1] + 8 > m.lda) return false;
  return true;
}
static int64_t carve_train(const DevMlp& m, int64_t M, char* base, TrainWs* ws) {
  const int64_t esz = m.dtype == KS_MLP_BF16 ? 2 : 4;
  const int64_t Mp = (M + 63) / 64 * 64;
  const int wz = widest_pad(m);
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += (bytes + 255) / 256 * 256;
    return p;
  };
  TrainWs w;
  std::memset(&w, 0, sizeof(w));
  const int64_t rows = chain_ok(m, M) ? (M + 127) / 128 * 128 : M;  // the whole-network backward pass reads whole tiles
  for (int l = 0; l + 1 < m.n_layers; ++l) w.act[l] = take(rows * m.npad[l] * esz);
  if (m.activation == KS_ACT_GELU)
    for (int l = 0; l + 1 < m.n_layers; ++l) w.pre[l] = take(M * m.npad[l] * esz);
  w.d0 = take(M * wz * esz);
  w.d1 = take(M * wz * esz);
  w.t0 = take((int64_t)wz * Mp * esz);
  w.t1 = take((int64_t)wz * Mp * esz);
  w.t2 = take((int64_t)wz * Mp * esz);
  int64_t maxw = 0;
  for (int l = 0; l < m.n_layers; ++l) maxw = (int64_t)m.npad[l] * m.kpad[l] > maxw ? (int64_t)m.npad[l] * m.kpad[l] : maxw;
  int64_t nparts = kDwSplit * maxw > (int64_t)4 * kColsumSlices * wz ? kDwSplit * maxw : (int64_t)4 * kColsumSlices * wz;
  if (m.n_layers == 1)  // the one-pass weight and bias gradient of a single layer: slices of both
    nparts = (int64_t)wgrad_slices(m.dims[1], m.dims[0], M) * m.dims[1] * (m.dims[0] + 1);
  w.part = (float*)take(nparts * 4);
  w.Mp = Mp;
  w.Mp128 = (M + 127) / 128 * 128;
  if (chain_ok(m, M)) {
    const int64_t tiles = w.Mp128 / 128;
    for (int l = 0; l < m.n_layers; ++l) {
      w.dz[l] = take((int64_t)m.npad[l] * w.Mp128 * esz);
      w.bpart[l] = (float*)take(tiles * m.npad[l] * 4);
      w.wpart[l] = (float*)take((int64_t)chain_dw_slices(m.npad[l], round_up(m.kpad[l], kBN), w.Mp128) * m.npad[l] * m.kpad[l] * 4);
    }
    w.in = take((int64_t)round_up(m.kpad[0], kBN) * w.Mp128 * esz);
  }
  if (ws) *ws = w;
  return off;
}

extern "C" int64_t ks_mlp_train_workspace_bytes(const KsMlp* h, int64_t M) {
  if (!h || M < 0) return 0;
  return carve_train(h->m, M, nullptr, nullptr) + 256;
}

template <typename T>
static int train_forward(DevMlp& m, hipStream_t s, int64_t M, const float* x, float* y, const TrainWs& ws) {
  // networks that fit the whole-network kernel run it, with every hidden layer's activations written out for the backward
  // pass as well, in rows of the width that pass expects (its padding is in units of 128, the kernel's of 32)
  bool whole = m.fused && m.activation != KS_ACT_GELU;
  if (sizeof(T) == 2)  // bf16 networks of other widths take the per-layer kernel
    for (int l = 0; whole && l + 1 < m.n_layers; ++l) whole = m.npad[l] == m.fn[l] * 32;
  m.chain_saved = 0;
  if (whole && chain_ok(m, M)) {
    m.chain_saved = 1;
    return launch_fused_tile<__bf16, 128>(m, s, M, x, y, ws.act, ws.in);
  }
  if (whole) return launch_fused(m, s, M, x, y, ws.act);
  const void* in = x;
  int64_t ldin = m.dims[0];
  for (int l = 0; l < m.n_layers; ++l) {
    const bool first = l == 0, last = l == m.n_layers - 1;
    const bool split_act = !last && m.activation == KS_ACT_GELU;  // keep the pre-activation, then apply GELU
    void* outp = last ? (void*)y : (split_act ? (void*)ws.pre[l] : (void*)ws.act[l]);
    const int64_t ldo = last ? m.dims[l + 1] : m.npad[l];
    const int act_l = split_act ? KS_ACT_NONE : m.activation;
    int rc;
    if (first && last) rc = launch_layer<T, true, true>(act_l, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);
    else if (first) rc = launch_layer<T, true, false>(act_l, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);
    else if (last) rc = launch_layer<T, false, true>(act_l, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);
    else rc = launch_layer<T, false, false>(act_l, s, M, m.npad[l], m.kpad[l], m.dims[l], m.dims[l + 1], in, ldin, m.W[l], m.b[l], outp, ldo);
    if (rc != KS_OK) return rc;
    if (split_act) {
      const int64_t n = M * m.npad[l];
      hipLaunchKernelGGL(gelu_forward_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, (const T*)ws.pre[l], (T*)ws.act[l]);
      outp = ws.act[l];
    }
    in = outp;
    ldin = ldo;
  }
  return KS_OK;
}

extern "C" int ks_mlp_train_forward(KsMlp* h, ks_stream_t stream, int64_t M, const float* x, float* y, void* workspace) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_train_forward: call ks_mlp_train_init first");
  if (M <= 0 || !x || !y || !workspace) return fail(KS_EINVAL, "ks_mlp_train_forward: bad argument");
  if ((M + kBM - 1) / kBM > 0x7fffffff) return fail(KS_ELIMIT, "ks_mlp_train_forward: too many rows");
  TrainWs ws;
  carve_train(h->m, M, (char*)workspace, &ws);
  const int rc = h->m.dtype == KS_MLP_BF16 ? train_forward<__bf16>(h->m, (hipStream_t)stream, M, x, y, ws)
                                           : train_forward<float>(h->m, (hipStream_t)stream, M, x, y, ws);
  return rc != KS_OK ? rc : check_launch("ks_mlp_train_forward");
}

static int chain_wgrad(hipStream_t s, int slices, int64_t Mp, int np, int ldb, int kp, const __bf16* dz, const __bf16* y, float* part) {
  const int64_t kslice = ((Mp + slices - 1) / slices + 4 * kCwRows - 1) / (4 * kCwRows) * (4 * kCwRows);  // slices past the last row add zeros
  if (hipFuncSetAttribute((const void*)chain_wgrad_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kCwLds) != hipSuccess)
    return fail(KS_ELAUNCH, "ks_mlp_train_backward: cannot raise the LDS limit to %d bytes", kCwLds);
  hipLaunchKernelGGL(chain_wgrad_kernel, dim3((unsigned)((np / 128) * (ldb / 128)), (unsigned)slices), dim3(512), kCwLds, s, Mp, np, ldb, kp, (int)kslice,
                     dz, y, part);
  return KS_OK;
}

// The backward pass of a network whose forward kept what it reads (chain_ok): every layer's gradient in one launch of mlp_fused_bwd_kernel,
// then one weight-gradient product per layer.
static int train_backward_chain(DevMlp& m, hipStream_t s, int64_t M, const float* dy, const TrainWs& ws) {
  const int L = m.n_layers;
  const int64_t Mp = ws.Mp128, tiles = Mp / 128;
  const int npl = m.npad[L - 1];
  {
    FusedBwdArgs a;
    std::memset(&a, 0, sizeof(a));
    a.M = M; a.n_layers = L; a.lda = m.lda;
    a.dy = dy; a.out_dim = m.dims[L]; a.np_last = npl;
    for (int l = 0; l < L; ++l) {
      a.fk[l] = m.fk[l]; a.fn[l] = m.fn[l];
      a.WtP[l] = (const u32x4*)m.WtP[l];
      if (l + 1 < L) a.y[l] = (const __bf16*)ws.act[l];
      a.dz[l] = (__bf16*)ws.dz[l];
      a.bias_part[l] = ws.bpart[l];
    }
    const int lds = 128 * m.lda * 2;
#define KS_LAUNCH(A)                                                                                           \
  {                                                                                                            \
    auto kfn = mlp_fused_bwd_kernel<A>;                                                                        \
    if (lds > 64 * 1024 &&                                                                                     \
        hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)  \
      return fail(KS_ELAUNCH, "ks_mlp_train_backward: cannot raise the LDS limit to %d bytes", lds);           \
    hipLaunchKernelGGL(kfn, dim3((unsigned)tiles), dim3(64 * kFusedWaves), lds, s, a);                         \
  }
    switch (m.activation) {
      case KS_ACT_ELU: KS_LAUNCH(KS_ACT_ELU) break;
      case KS_ACT_RELU: KS_LAUNCH(KS_ACT_RELU) break;
      case KS_ACT_TANH: KS_LAUNCH(KS_ACT_TANH) break;
      default: KS_LAUNCH(KS_ACT_NONE) break;
    }
#undef KS_LAUNCH
  }
  GradFinishArgs g;
  std::memset(&g, 0, sizeof(g));
  g.n_layers = L; g.tiles = (int)tiles;
  int wblocks = 0, bblocks = 0;
  for (int l = L - 1; l >= 0; --l) {
    const int np = m.npad[l], kp = m.kpad[l], kp128 = round_up(kp, kBN);
    const int slices = chain_dw_slices(np, kp128, Mp);
    const int rc = chain_wgrad(s, slices, Mp, np, kp128, kp, (const __bf16*)ws.dz[l], l > 0 ? (const __bf16*)ws.act[l - 1] : (const __bf16*)ws.in, ws.wpart[l]);
    if (rc != KS_OK) return rc;
    g.nz[l] = slices; g.nW[l] = (int64_t)np * kp; g.nb[l] = np;
    g.wpart[l] = ws.wpart[l]; g.bpart[l] = ws.bpart[l]; g.gW[l] = m.gW[l]; g.gb[l] = m.gb[l];
  }
  for (int l = 0; l < L; ++l) {
    g.first_w[l] = wblocks; g.first_b[l] = bblocks;
    wblocks += (int)((g.nW[l] + 1023) / 1024);
    bblocks += (g.nb[l] + kFinishCols - 1) / kFinishCols;
  }
  g.first_w[L] = wblocks; g.first_b[L] = bblocks;
  hipLaunchKernelGGL(grad_finish_kernel, dim3((unsigned)(wblocks + bblocks)), dim3(256), 0, s, g);
  return KS_OK;
}

template <int PARTS>
static int wgrad(hipStream_t s, int64_t M, int N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                 int64_t ldc, float* part, float* colsum);

// dX = dZ W of a single bf16 layer as a layer over the transposed fragments
static FusedArgs single_dx_args(const DevMlp& m, int64_t M, const float* dy, float* dx) {
  FusedArgs a;
  std::memset(&a, 0, sizeof(a));
  a.M = M; a.n_layers = 1; a.in_dim = m.dims[1]; a.out_dim = m.dims[0]; a.lda = 32 * m.fn[0] + 8;
  a.fk[0] = 2 * m.fn[0]; a.fn[0] = (m.fk[0] + 1) / 2;
  a.Wp[0] = (const u32x4*)m.WtP[0]; a.bp[0] = m.zero_bias;
  a.x = dy; a.y = dx;
  return a;
}

// Backward pass of a single layer (the projections of the recurrent cells and their networks, over all the (step, env) rows of a
// trajectory slice): no activation to pass through, so the caller's gradient and input are the operands of both products as they are.
template <typename T>
static int train_backward_single(DevMlp& m, hipStream_t s, int64_t M, const float* x, int64_t ldx, const float* dy, const TrainWs& ws, float* dx,
                                 bool want_w, bool accumulate_dx, const uint8_t* zero_rows) {
  const int np = m.npad[0], in = m.dims[0], out = m.dims[1], kp128 = round_up(m.kpad[0], kBN);
  const bool plain = !accumulate_dx && !zero_rows;
  if (dx && sizeof(T) == 2 && plain && m.WtP[0]) {
    // dX = dZ W: the whole-network kernel over the transposed fragments
    const int rc = launch_fused_args(single_dx_args(m, M, dy, dx), s);
    if (rc != KS_OK) return rc;
  } else if (dx) {
    int rc;
    T* tmp = (T*)ws.d1;
    if constexpr (sizeof(T) == 4) {
      rc = launch_layer_f32(KS_ACT_NONE, s, M, kp128, np, out, plain ? in : kp128, dy, out, m.Wt[0], m.zero_bias, plain ? dx : tmp,
                            plain ? in : kp128);
    } else {
      const int64_t n = M * np;
      hipLaunchKernelGGL(cast_pad_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, M, out, np, dy, (T*)ws.d0);
      rc = launch_layer<T, false, false>(KS_ACT_NONE, s, M, kp128, np, np, kp128, ws.d0, np, m.Wt[0], m.zero_bias, tmp, kp128);
    }
    if (rc != KS_OK) return rc;
    if (sizeof(T) == 2 || !plain) {
      const int64_t n = M * in;
      hipLaunchKernelGGL(unpad_cast_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, M, in, kp128, (const T*)tmp, dx,
                         accumulate_dx ? 1 : 0, zero_rows);
    }
  }
  if (!want_w) return KS_OK;
  return wgrad<sizeof(T) == 2 ? 1 : 3>(s, out, in, M, dy, out, x, ldx, m.gW[0], m.kpad[0], ws.part, m.gb[0]);
}

template <typename T>
static int train_backward(DevMlp& m, hipStream_t s, int64_t M, const float* x, const float* dy, const TrainWs& ws,
                          float* dx = nullptr, bool want_w = true, bool accumulate_dx = false, const uint8_t* zero_rows = nullptr) {
  const int L = m.n_layers;
  const int64_t Mp = ws.Mp;
  if (L == 1) return train_backward_single<T>(m, s, M, x, m.dims[0], dy, ws, dx, want_w, accumulate_dx, zero_rows);
  if constexpr (sizeof(T) == 2) if (m.chain_saved && want_w && !dx) return train_backward_chain(m, s, M, dy, ws);
  T* dz = (T*)ws.d0;
  T* dnext = (T*)ws.d1;
  {  // the output gradient in working precision, padded to the last layer's width
    const int64_t n = M * m.npad[L - 1];
    hipLaunchKernelGGL(cast_pad_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, M, m.dims[L], m.npad[L - 1], dy, dz);
  }
  // The layer-l step needs dZ_l (row-major, for the input gradient), dZ_l^T and Y_{l-1}^T (for the weight gradient) and
  // the column sums of dZ_l.  For hidden layers of a width that is a multiple of 64 one fused pass (bwd_prep_kernel)
  // turns the input gradient of the layer above into all four; otherwise separate kernels do.
  T* dzT = (T*)ws.t0;    // dZ_l^T
  T* dzT_next = (T*)ws.t2;
  bool have_dzT = false, have_bias = false;
  for (int l = L - 1; l >= 0; --l) {
    const int np = m.npad[l], kp = m.kpad[l], kp128 = round_up(kp, kBN);
    if (l == 0 && dx) {  // gradient with respect to the network input
      // an fp32 network whose input width needs no padding: the product writes the caller's buffer itself
      const bool direct = sizeof(T) == 4 && m.dims[0] == kp128 && !accumulate_dx && !zero_rows;
      const int rc0 = launch_layer<T, false, false>(KS_ACT_NONE, s, M, kp128, np, np, kp128, dz, np, m.Wt[0], m.zero_bias,
                                                    direct ? (T*)dx : dnext, kp128);
      if (rc0 != KS_OK) return rc0;
      if (!direct) {
        const int64_t n = M * m.dims[0];
        hipLaunchKernelGGL(unpad_cast_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, M, m.dims[0], kp128, (const T*)dnext, dx,
                           accumulate_dx ? 1 : 0, zero_rows);
      }
    }
    if (!want_w && l == 0) break;
    if (want_w && !have_bias) {
      const int nz = M >= 32768 ? 4 * kColsumSlices : kColsumSlices;  // narrow layers: more row slices fill the chip
      hipLaunchKernelGGL(colsum_kernel<T>, dim3((unsigned)((np + 63) / 64), nz), dim3(256), 0, s, M, np, dz, ws.part);
      hipLaunchKernelGGL(sum_parts_tree_kernel, dim3((unsigned)np), dim3(64), 0, s, (int64_t)np, nz, ws.part, m.gb[l]);
    }
    if (want_w && !have_dzT)
      hipLaunchKernelGGL((transpose_kernel<T, T>), dim3((unsigned)((Mp + 31) / 32), (unsigned)((np + 31) / 32)), dim3(256), 0, s, M, np,
                         (int64_t)np, dz, np, Mp, dzT);
    have_dzT = have_bias = false;
    bool have_yT = false;
    int rc;
    if (l > 0) {
      // input gradient, then through the activation of the layer below
      rc = launch_layer<T, false, false>(KS_ACT_NONE, s, M, kp, np, np, kp, dz, np, m.Wt[l], m.zero_bias, dnext, kp);
      if (rc != KS_OK) return rc;
      const bool fused = want_w && m.activation != KS_ACT_GELU && kp % 64 == 0 && kp == kp128 && kp == m.npad[l - 1];
      if (fused) {
#define KS_PREP(A) hipLaunchKernelGGL((bwd_prep_kernel<T, A>), dim3((unsigned)(kp / 64), kColsumSlices), dim3(256), 0, s, M, Mp, kp, \
                                      (const T*)ws.act[l - 1], dnext, dzT_next, (T*)ws.t1, ws.part)
        switch (m.activation) {
          case KS_ACT_ELU: KS_PREP(KS_ACT_ELU); break;
          case KS_ACT_RELU: KS_PREP(KS_ACT_RELU); break;
          case KS_ACT_TANH: KS_PREP(KS_ACT_TANH); break;
          default: KS_PREP(KS_ACT_NONE); break;
        }
#undef KS_PREP
        hipLaunchKernelGGL(sum_parts_tree_kernel, dim3((unsigned)kp), dim3(64), 0, s, (int64_t)kp, kColsumSlices, ws.part, m.gb[l - 1]);
        have_yT = have_dzT = have_bias = true;
      } else {
        const int64_t n = M * kp;
#define KS_ACTB(A) hipLaunchKernelGGL((act_backward_kernel<T, A>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, (const T*)ws.act[l - 1], dnext)
        switch (m.activation) {
          case KS_ACT_ELU: KS_ACTB(KS_ACT_ELU); break;
          case KS_ACT_RELU: KS_ACTB(KS_ACT_RELU); break;
          case KS_ACT_TANH: KS_ACTB(KS_ACT_TANH); break;
          case KS_ACT_GELU:
            hipLaunchKernelGGL(gelu_backward_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, (const T*)ws.pre[l - 1], dnext);
            break;
          default: break;
        }
#undef KS_ACTB
      }
    }
    if (!want_w) {
      T* tmp = dz; dz = dnext; dnext = tmp;
      continue;
    }
    // weight gradient: dZ^T (np, Mp) times Y_prev^T (kp128, Mp)^T
    if (!have_yT) {
      if (l == 0)
        hipLaunchKernelGGL((transpose_kernel<float, T>), dim3((unsigned)((Mp + 31) / 32), (unsigned)((kp128 + 31) / 32)), dim3(256), 0, s, M,
                           m.dims[0], (int64_t)m.dims[0], x, kp128, Mp, (T*)ws.t1);
      else
        hipLaunchKernelGGL((transpose_kernel<T, T>), dim3((unsigned)((Mp + 31) / 32), (unsigned)((kp128 + 31) / 32)), dim3(256), 0, s, M,
                           m.npad[l - 1], (int64_t)m.npad[l - 1], (const T*)ws.act[l - 1], kp128, Mp, (T*)ws.t1);
    }
    // the reduction runs over the rows: cut it into slices so that the grid covers the chip, then add the slices up
    // wide layers over many rows: 128 x 128 output tiles halve the operand traffic per flop, twice the slices keep the grid
    const bool wide = Mp >= 32768 && np % 128 == 0;
    int ksplit = wide ? kDwSplit : kDwSplit / 2;
    while (ksplit > 1 && Mp / 64 < ksplit) ksplit >>= 1;
    if constexpr (sizeof(T) == 4)
      rc = launch_layer_f32(KS_ACT_NONE, s, np, kp128, (int)Mp, (int)Mp, kp, dzT, Mp, ws.t1, m.zero_bias,
                            ksplit > 1 ? (void*)ws.part : (void*)m.gW[l], kp, ksplit);
    else if (wide)
      rc = launch_layer_tile<T, false, true, 128, 128, 2, 2>(KS_ACT_NONE, s, np, kp128, (int)Mp, (int)Mp, kp, dzT, Mp, ws.t1,
                                                              m.zero_bias, ksplit > 1 ? (void*)ws.part : (void*)m.gW[l], kp, ksplit);
    else
      rc = launch_layer_tile<T, false, true, 64, 128, 2, 2>(KS_ACT_NONE, s, np, kp128, (int)Mp, (int)Mp, kp, dzT, Mp, ws.t1,
                                                             m.zero_bias, ksplit > 1 ? (void*)ws.part : (void*)m.gW[l], kp, ksplit);
    if (rc != KS_OK) return rc;
    if (ksplit > 1) {
      const int64_t n = (int64_t)np * kp;
      hipLaunchKernelGGL(sum_parts_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, ksplit, ws.part, m.gW[l]);
    }
    if (l == 0) break;
    T* tmp = dz; dz = dnext; dnext = tmp;
    tmp = dzT; dzT = dzT_next; dzT_next = tmp;
  }
  return KS_OK;
}

extern "C" int ks_mlp_train_backward(KsMlp* h, ks_stream_t stream, int64_t M, const float* x, const float* dy, void* workspace) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_train_backward: call ks_mlp_train_init first");
  if (M <= 0 || !x || !dy || !workspace) return fail(KS_EINVAL, "ks_mlp_train_backward: bad argument");
  if (M > (1 << 30)) return fail(KS_ELIMIT, "ks_mlp_train_backward: too many rows");
  TrainWs ws;
  carve_train(h->m, M, (char*)workspace, &ws);
  const int rc = h->m.dtype == KS_MLP_BF16 ? train_backward<__bf16>(h->m, (hipStream_t)stream, M, x, dy, ws)
                                           : train_backward<float>(h->m, (hipStream_t)stream, M, x, dy, ws);
  return rc != KS_OK ? rc : check_launch("ks_mlp_train_backward");
}

// The hidden projections' gradient: their input is a block of columns of what the recurrence kept per step, and copying it out first was a pass
// of its own (102400 x 128: 21 us beside a product of 92; the product takes as long on the strided rows).
extern "C" int ks_mlp_layer_weight_grad(KsMlp* h, ks_stream_t stream, int64_t M, const float* x, int64_t ldx, const float* dy, void* workspace) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_layer_weight_grad: call ks_mlp_train_init first");
  if (h->m.n_layers != 1) return fail(KS_EINVAL, "ks_mlp_layer_weight_grad: the network has %d layers, not one", h->m.n_layers);
  if (M <= 0 || !x || !dy || !workspace || ldx < h->m.dims[0]) return fail(KS_EINVAL, "ks_mlp_layer_weight_grad: bad argument");
  if (M > (1 << 30)) return fail(KS_ELIMIT, "ks_mlp_layer_weight_grad: too many rows");
  TrainWs ws;
  carve_train(h->m, M, (char*)workspace, &ws);
  const int rc = h->m.dtype == KS_MLP_BF16 ? train_backward_single<__bf16>(h->m, (hipStream_t)stream, M, x, ldx, dy, ws, nullptr, true, false, nullptr)
                                           : train_backward_single<float>(h->m, (hipStream_t)stream, M, x, ldx, dy, ws, nullptr, true, false, nullptr);
  return rc != KS_OK ? rc : check_launch("ks_mlp_layer_weight_grad");
}

extern "C" int ks_mlp_train_backward_dx(KsMlp* h, ks_stream_t stream, int64_t M, const float* x, const float* dy, float* dx,
                                        int32_t weight_gradients, int32_t accumulate_dx, const uint8_t* zero_rows, void* workspace) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_train_backward_dx: call ks_mlp_train_init first");
  if (M <= 0 || !dy || !dx || !workspace || (weight_gradients && !x)) return fail(KS_EINVAL, "ks_mlp_train_backward_dx: bad argument");
  if (M > (1 << 30)) return fail(KS_ELIMIT, "ks_mlp_train_backward_dx: too many rows");
  TrainWs ws;
  carve_train(h->m, M, (char*)workspace, &ws);
  const bool w = weight_gradients != 0, acc = accumulate_dx != 0;
  const int rc = h->m.dtype == KS_MLP_BF16 ? train_backward<__bf16>(h->m, (hipStream_t)stream, M, x, dy, ws, dx, w, acc, zero_rows)
                                           : train_backward<float>(h->m, (hipStream_t)stream, M, x, dy, ws, dx, w, acc, zero_rows);
  return rc != KS_OK ? rc : check_launch("ks_mlp_train_backward_dx");
}

extern "C" int ks_mlp_freeze_bias_prefix(KsMlp* h, int32_t layer, int32_t count) {
  if (!h) return fail(KS_EINVAL, "ks_mlp_freeze_bias_prefix: null handle");
  if (layer < 0 || layer >= h->m.n_layers || count < 0 || count > h->m.dims[layer + 1])
    return fail(KS_EINVAL, "ks_mlp_freeze_bias_prefix: layer %d, count %d out of range", layer, count);
  h->m.bias_frozen[layer] = count;
  return KS_OK;
}

extern "C" int ks_grad_sqnorm(ks_stream_t stream, int64_t n, const float* g, double* acc) {
  if (n < 0 || !acc || (n > 0 && !g)) return fail(KS_EINVAL, "ks_grad_sqnorm: bad argument");
  if (n == 0) return KS_OK;
  hipLaunchKernelGGL(sqnorm_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, n, g, acc);
  return check_launch("ks_grad_sqnorm");
}

extern "C" int ks_mlps_grad_sqnorm(const KsMlp* const* nets, int32_t count, ks_stream_t stream, double* acc) {
  if (count < 0 || (count > 0 && !nets) || !acc) return fail(KS_EINVAL, "ks_mlps_grad_sqnorm: bad argument");
  for (int k = 0; k < count; ++k)
    if (!nets[k] || !nets[k]->m.train) return fail(KS_EINVAL, "ks_mlps_grad_sqnorm: network %d: call ks_mlp_train_init first", k);
  for (int k = 0; k < count;) {  // as many networks at a time as the tables hold
    SqTensors t;
    SqNets f;
    f.nets = 0; f.acc = acc;
    int nt = 0;
    for (; k < count && f.nets < kSqNets && nt + 2 * nets[k]->m.n_layers <= kSqTensors; ++k) {
      const DevMlp& m = nets[k]->m;
      const int first = nt;
      auto add = [&](const float* g, int64_t n) { t.g[nt] = g; t.n[nt] = n; t.part[nt] = m.sq_part + (nt - first) * kSqBlocks; ++nt; };
      for (int l = 0; l < m.n_layers; ++l) {
        add(m.gW[l], (int64_t)m.npad[l] * m.kpad[l]);
        const int fz = m.bias_frozen[l];
        if (m.npad[l] > fz) add(m.gb[l] + fz, (int64_t)m.npad[l] - fz);
      }
      f.n[f.nets] = (nt - first) * kSqBlocks;
      f.part[f.nets++] = m.sq_part;
    }
    hipLaunchKernelGGL(sqnorm_parts_kernel, dim3(kSqBlocks, (unsigned)nt), dim3(256), 0, (hipStream_t)stream, t);
    hipLaunchKernelGGL(sqnorm_finish_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, f);
  }
  return check_launch("ks_mlps_grad_sqnorm");
}

extern "C" int ks_mlp_grad_sqnorm(const KsMlp* h, ks_stream_t stream, double* acc) {
  if (!h || !h->m.train || !acc) return fail(KS_EINVAL, "ks_mlp_grad_sqnorm: bad argument");
  return ks_mlps_grad_sqnorm(&h, 1, stream, acc);
}

static int check_adam(const KsAdamParams* p, const char* who) {
  if (!p) return fail(KS_EINVAL, "%s: null parameters", who);
  if (p->step < 1) return fail(KS_EINVAL, "%s: step starts at 1", who);
  if (!(p->b1 >= 0.f && p->b1 < 1.f && p->b2 >= 0.f && p->b2 < 1.f)) return fail(KS_EINVAL, "%s: betas must be in [0, 1)", who);
  return KS_OK;
}

extern "C" int ks_adam_step(ks_stream_t stream, int64_t n, float* param, const float* grad, float* m1, float* m2,
                            const KsAdamParams* p, const double* sqnorm) {
  const int rc = check_adam(p, "ks_adam_step");
  if (rc != KS_OK) return rc;
  if (n < 0 || (n > 0 && (!param || !grad || !m1 || !m2))) return fail(KS_EINVAL, "ks_adam_step: bad argument");
  if (n == 0) return KS_OK;
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, param, grad, m1, m2, *p, sqnorm);
  return check_launch("ks_adam_step");
}

extern "C" int ks_mlps_adam_step(KsMlp* const* nets, int32_t count, ks_stream_t stream, const KsAdamParams* p, const double* sqnorm) {
  if (count < 0 || (count > 0 && !nets)) return fail(KS_EINVAL, "ks_mlps_adam_step: bad argument");
  for (int k = 0; k < count; ++k)
    if (!nets[k] || !nets[k]->m.train) return fail(KS_EINVAL, "ks_mlps_adam_step: network %d: call ks_mlp_train_init first", k);
  const int rc = check_adam(p, "ks_mlps_adam_step");
  if (rc != KS_OK) return rc;
  const AdamStep a = {p->lr, p->b1, p->b2, p->eps, p->weight_decay, p->max_grad_norm, (float)(1.0 - std::pow((double)p->b1, (double)p->step)),
                      (float)(1.0 - std::pow((double)p->b2, (double)p->step))};
  for (int k = 0; k < count;) {  // networks of one precision, each once, as many as the table holds
    AdamTable t;
    t.n = 0;
    int blocks = 0;
    const int from = k, dtype = nets[k]->m.dtype;
    for (; k < count; ++k) {
      const DevMlp& m = nets[k]->m;
      bool again = false;
      for (int q = from; q < k; ++q) again |= nets[q] == nets[k];
      if (again || m.dtype != dtype || t.n + m.n_layers > kOptLayers) break;
      for (int l = 0; l < m.n_layers; ++l) {
        t.layer[t.n++] = {m.npad[l], m.kpad[l], m.fk[l], m.fn[l], m.bias_frozen[l], blocks, m.mW[l], m.m1W[l], m.m2W[l], m.mb[l], m.m1b[l], m.m2b[l],
                          m.gW[l], m.gb[l], m.W[l], m.Wt[l], m.Wp[l], (__bf16*)m.WtP[l], m.b[l], m.bp[l]};
        blocks += m.npad[l] / 32 * (m.kpad[l] / 32);  // npad: whole tiles of 128; kpad: of 64 (bf16) or 32
      }
    }
    if (dtype == KS_MLP_BF16) hipLaunchKernelGGL(adam_layers_kernel<__bf16>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, t, a, sqnorm);
    else hipLaunchKernelGGL(adam_layers_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, t, a, sqnorm);
  }
  return check_launch("ks_mlps_adam_step");
}

extern "C" int ks_mlp_adam_step(KsMlp* h, ks_stream_t stream, const KsAdamParams* p, const double* sqnorm) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_adam_step: call ks_mlp_train_init first");
  return ks_mlps_adam_step(&h, 1, stream, p, sqnorm);
}

// ---------------------------------------------------------------- discriminator update (ksim/task/amp.py:360-438)
// Gradient of   0.5 sum (D(real) - 1)^2 + 0.5 sum (D(sim) + 1)^2 + coef / 2 * mean_b sum_t |grad_x D(real[b, t])|^2
// with respect to every weight and bias of an MLP D with one output, applied frame by frame.  The last term differentiates
// the network twice.  With z_l = W_l y_{l-1} + b_l, y_l = f(z_l), the input gradient is g = W_1^T d_1 with d_L = 1,
// d_l = f'(z_l) * (W_{l+1}^T d_{l+1}) =: f'(z_l) * a_l.  The gradient of P(g) walks that computation backwards, which is a
// forward sweep through the layers: with v_0 = dP/dg,
//   dP/dW_l += d_l^T v_{l-1},   u_l = v_{l-1} W_l^T,   v_l = u_l * f'(z_l),   r_l = u_l * a_l * f''(z_l),
// and r_l, the part that reaches z_l through f', joins the ordinary backward pass of the squared-error terms as an extra
// gradient of z_l on the real rows.  The discriminator is small next to the policy, so everything here runs in fp32 on the
// master weights, the products on the fp32 matrix-core instruction.
namespace ks {

// first and second derivative of the activation from its output y = f(z)
__device__ __forceinline__ void act_derivatives(int act, float y, float& d1, float& d2) {
  d1 = 1.f; d2 = 0.f;
  if (act == KS_ACT_ELU) { if (y <= 0.f) { d1 = y + 1.f; d2 = y + 1.f; } }  // exp(z) = elu(z) + 1 for z <= 0
  else if (act == KS_ACT_RELU) d1 = y > 0.f ? 1.f : 0.f;
  else if (act == KS_ACT_TANH) { d1 = 1.f - y * y; d2 = -2.f * y * d1; }
}

// Words that workgroups on different XCDs hand each other inside one launch: written through, and read past, the L2 of the writer's and
// reader's XCD.  A device-scope fence does the same for everything at once by writing back and invalidating whole L2s: with one per
// workgroup the weight-gradient products below took 41 us instead of 9.5 (and 18.8 with one uncut slice).
__device__ __forceinline__ void device_store(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float device_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// What becomes of an entry of the product, at (i, j) of the output and of the arrays beside it (all with the output's stride):
enum { kEpiStore,    // C (+)= v
       kEpiLayer,    // C = act(v + bias_j): a layer of the forward pass
       kEpiDelta,    // C = v, C2 = f'(Y) v: a_l and d_l of the input gradient's chain
       kEpiPenalty,  // C = scale v, and the tile's sum of v^2 to sums[tile]: the penalty's gradient and value
       kEpiTangent,  // C = f'(Y) v, C2 = f''(Y) X v: v_l and r_l of the sweep back through that chain
       kEpiDz,       // C = f'(Y) v (+ X on the first x_rows rows): the ordinary backward pass
       kEpiTop,      // C = act(v + bias_j) =: y and, on the first x_rows rows, C2 = X_j, C3 = f'(y) X_j: the last hidden layer, whose input
                     // gradient starts from the output layer's one row of weights X
       kEpiOut };    // the output layer, N = 1: C = v + bias - target, the gradient of the squared error (target 1 on the first x_rows rows, where
                     // C2 = 1 too, and -1 on the others)
struct SgemmArgs {
  int M, N, K;
  const float *A, *A2;  // A2: rows (or, stored (k, i), reduction steps) from a_split on come from this second array
  int64_t lda;
  int a_split;
  const float *B, *B2, *B3;  // stored (k, j): reduction steps from b_split on come from the second array, from b_split2 on from the third
  int64_t ldb;
  int b_split, b_split2;
  float* C;
  int64_t ldc;
  int kslice;
  int epi, act, accumulate;
  const float *bias, *Y, *X;
  int x_rows;
  float *C2, *C3;
  float scale;
  double* sums;
  float* colsum;        // sum_k A(i, k) over the steps k >= cs_from, per row i of the output, never accumulated
  int cs_from;
  unsigned* zero;       // the first workgroup clears `zeros` counters for the launches that follow
  int zeros;
  // reduction cut into gridDim.z slices: slice z leaves its tile in part[z] (tile-major, column sums behind the 1024 entries) and the last
  // workgroup to arrive at a tile adds the slices up in slice order.  counters: one zero per tile, zero again afterwards.
  float* part;
  unsigned* counters;
};
constexpr int kTilePart = 1024 + 32;

// C(i, j) (+)= sum_k A(i, k) B(k, j) in fp32 on the matrix cores, for the discriminator's batches of a thousand rows or so: a
// 32 x 32 tile per workgroup, whose wavefronts cut the reduction between them, each straight from memory into registers (a chunk
// of 32 steps' loads in flight under the previous chunk's 16 v_mfma_f32_32x32x2_f32), and add their tiles up in LDS.  A product of
// 1024 x 256 x 256 is then 256 workgroups and one memory latency plus 0.9 us of matrix work; 64 x 64 tiles with the whole
// reduction behind one barrier per 16 steps left it on 64 CUs for 22 us.
// A_KC: A is stored (i, k) with k contiguous, otherwise (k, i); B_KC: B is stored (j, k) with k contiguous, otherwise (k, j).
// A lane of half h feeds steps k = 8 (s / 4) + 4 h + s % 4 of a chunk, so that k-contiguous rows are read 16 bytes at a time.
// The reduction steps of a (k, .) operand may come from up to three arrays one after the other, from steps 0, at1 and at2 on.
struct SgemmRows {
  const float *p0, *p1, *p2;
  int at1, at2;
  __device__ __forceinline__ const float* row(int k, int64_t ld) const {
    return k < at1 ? p0 + (int64_t)k * ld : (k < at2 ? p1 + (int64_t)(k - at1) * ld : p2 + (int64_t)(k - at2) * ld);
  }
  __device__ __forceinline__ bool together(int k0) const {  // steps k0 .. k0 + 31 lie in one array
    return k0 + 32 <= at1 || (k0 >= at1 && k0 + 32 <= at2) || k0 >= at2;
  }
};

template <bool KC>
__device__ __forceinline__ void sgemm_fetch(float (&v)[16], const SgemmRows& r, int64_t ld, int k0, int kend, int h, bool wide) {
  if (k0 + 32 <= kend && (KC || r.together(k0))) {  // a whole chunk of one array: no checks per load
    if (KC) {
      const float* q = r.p0 + k0 + 4 * h;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (wide) {
          const float4 t = *reinterpret_cast<const float4*>(q + 8 * s);
          v[4 * s] = t.x; v[4 * s + 1] = t.y; v[4 * s + 2] = t.z; v[4 * s + 3] = t.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * s + e] = q[8 * s + e];
        }
      }
    } else {
      const float* q = r.row(k0, ld) + 4 * h * ld;
#pragma unroll
      for (int s = 0; s < 16; ++s) v[s] = q[(8 * (s >> 2) + (s & 3)) * ld];
    }
    return;
  }
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int k = k0 + 8 * (s >> 2) + 4 * h + (s & 3);
    float x = 0.f;
    if (k < kend) x = KC ? r.p0[k] : *r.row(k, ld);
    v[s] = x;
  }
}

// workgroup (bx, by, bz) of a grid (gx, gy, gz): row tile, column tile and slice of the reduction
template <bool A_KC, bool B_KC, int WAVES>
__device__ __forceinline__ void sgemm_tile(const SgemmArgs& g, int bx, int by, int bz, int gx, int gy, int gz) {
  constexpr int RW = WAVES > 8 ? 8 : WAVES;  // tiles held in LDS at a time
  __shared__ float red[RW][1024];
  __shared__ float cred[WAVES][64];
  __shared__ double sred[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 31, h = lane >> 5;
  const int i0 = bx * 32, j0 = by * 32;
  const int zbeg = bz * g.kslice, zend = min(g.K, zbeg + g.kslice);
  const int per = ((zend - zbeg + WAVES - 1) / WAVES + 7) / 8 * 8;
  const int kbeg = zbeg + wave * per, kend = min(zend, kbeg + per);
  // rows and columns past the matrix repeat the last one; their results are not stored
  const int ia = min(i0 + c, g.M - 1), jb = min(j0 + c, g.N - 1);
  SgemmRows ra = {}, rb = {};
  if (A_KC) ra.p0 = ia < g.a_split ? g.A + (int64_t)ia * g.lda : g.A2 + (int64_t)(ia - g.a_split) * g.lda;
  else ra = {g.A + ia, g.A2 + ia, g.A2 + ia, g.a_split, 0x7fffffff};
  if (B_KC) rb.p0 = g.B + (int64_t)jb * g.ldb;
  else rb = {g.B + jb, g.B2 + jb, g.B3 + jb, g.b_split, g.b_split2};
  if (g.zero && bx == 0 && by == 0 && bz == 0)
    for (int x = threadIdx.x; x < g.zeros; x += 64 * WAVES) g.zero[x] = 0;
  const bool wa = A_KC && g.lda % 4 == 0 && (((uintptr_t)g.A | (uintptr_t)g.A2) & 15) == 0;  // kbeg is a multiple of 8
  const bool wb = B_KC && g.ldb % 4 == 0 && ((uintptr_t)g.B & 15) == 0;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  float cs = 0.f;
  float a[16], b[16];
  if (kbeg < kend) {
    sgemm_fetch<A_KC>(a, ra, g.lda, kbeg, kend, h, wa);
    sgemm_fetch<B_KC>(b, rb, g.ldb, kbeg, kend, h, wb);
  }
  for (int k0 = kbeg; k0 < kend; k0 += 32) {
    float a1[16], b1[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) a1[s] = b1[s] = 0.f;
    if (k0 + 32 < kend) {
      sgemm_fetch<A_KC>(a1, ra, g.lda, k0 + 32, kend, h, wa);
      sgemm_fetch<B_KC>(b1, rb, g.ldb, k0 + 32, kend, h, wb);
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], acc, 0, 0, 0);
      cs += k0 + 8 * (s >> 2) + 4 * h + (s & 3) >= g.cs_from ? a[s] : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) { a[s] = a1[s]; b[s] = b1[s]; }
  }
  cred[wave][lane] = cs;
  if (WAVES > RW) {  // the upper half's tiles first, added by the lower half
    if (wave >= RW)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave - RW][(8 * (r >> 2) + 4 * h + (r & 3)) * 32 + c] = acc[r];
    __syncthreads();
    if (wave < RW)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += red[wave][(8 * (r >> 2) + 4 * h + (r & 3)) * 32 + c];
    __syncthreads();
  }
  if (wave < RW)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][(8 * (r >> 2) + 4 * h + (r & 3)) * 32 + c] = acc[r];
  __syncthreads();
  const bool sliced = gz > 1, want_cs = g.colsum && by == 0;
  const int tile = by * gx + bx, tiles = gx * gy;
  float csum = 0.f;
  if (want_cs && threadIdx.x < 32)
    for (int w = 0; w < WAVES; ++w) csum += cred[w][threadIdx.x] + cred[w][threadIdx.x + 32];
  if (sliced) {
    float* mine = g.part + ((int64_t)bz * tiles + tile) * kTilePart;
    for (int x = threadIdx.x; x < 1024; x += 64 * WAVES) {
      float v = 0.f;
      for (int w = 0; w < RW; ++w) v += red[w][x];
      device_store(mine + x, v);
    }
    if (want_cs && threadIdx.x < 32) device_store(mine + 1024 + threadIdx.x, csum);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's part has reached memory
    __syncthreads();
    __shared__ unsigned last;
    if (threadIdx.x == 0) last = atomicAdd(&g.counters[tile], 1u) == (unsigned)gz - 1u;
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0) g.counters[tile] = 0;
    for (int x = threadIdx.x; x < kTilePart; x += 64 * WAVES) {
      float v = 0.f;
      for (int z = 0; z < gz; ++z) v += device_load(g.part + ((int64_t)z * tiles + tile) * kTilePart + x);
      if (x < 1024) red[0][x] = v;
      else csum = v;  // x = 1024 + thread: the tile is a whole number of passes
    }
    __syncthreads();
  }
  if (want_cs && threadIdx.x < 32 && i0 + (int)threadIdx.x < g.M) g.colsum[i0 + threadIdx.x] = csum;
  double sq = 0.0;
#pragma unroll
  for (int x = threadIdx.x; x < 1024; x += 64 * WAVES) {
    const int il = x >> 5, jl = x & 31, i = i0 + il, j = j0 + jl;
    float v = 0.f;
    for (int w = 0; w < (sliced ? 1 : RW); ++w) v += red[w][x];
    if (i >= g.M || j >= g.N) continue;
    const int64_t o = (int64_t)i * g.ldc + j;
    float d1 = 1.f, d2 = 0.f;
    if (g.epi == kEpiDelta || g.epi == kEpiTangent || g.epi == kEpiDz) act_derivatives(g.act, g.Y[o], d1, d2);
    switch (g.epi) {
      case kEpiLayer:
        v += g.bias[j];
        if (g.act == KS_ACT_ELU) v = v > 0.f ? v : expm1f(v);
        else if (g.act == KS_ACT_RELU) v = fmaxf(v, 0.f);
        else if (g.act == KS_ACT_TANH) v = tanhf(v);
        g.C[o] = v;
        break;
      case kEpiTop:
        v += g.bias[j];
        if (g.act == KS_ACT_ELU) v = v > 0.f ? v : expm1f(v);
        else if (g.act == KS_ACT_RELU) v = fmaxf(v, 0.f);
        else if (g.act == KS_ACT_TANH) v = tanhf(v);
        g.C[o] = v;
        if (i < g.x_rows) {
          act_derivatives(g.act, v, d1, d2);
          g.C2[o] = g.X[j];
          g.C3[o] = d1 * g.X[j];
        }
        break;
      case kEpiOut:
        g.C[o] = v + g.bias[j] - (i < g.x_rows ? 1.f : -1.f);
        if (i < g.x_rows) g.C2[o] = 1.f;
        break;
      case kEpiDelta: g.C[o] = v; g.C2[o] = d1 * v; break;
      case kEpiPenalty: g.C[o] = g.scale * v; sq += (double)v * v; break;
      case kEpiTangent: g.C2[o] = v * g.X[o] * d2; g.C[o] = v * d1; break;
      case kEpiDz: v *= d1; if (i < g.x_rows) v += g.X[o]; g.C[o] = v; break;
      default: g.C[o] = g.accumulate ? g.C[o] + v : v;
    }
  }
  if (g.sums) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) sq += __shfl_down(sq, d);
    if (lane == 0) sred[wave] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < WAVES; ++w) t += sred[w];
      g.sums[(int64_t)by * gx + bx] = t;
    }
  }
}

template <bool A_KC, bool B_KC, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void sgemm_kernel(SgemmArgs g) {  // rows on x: y admits 65536 tiles only
  sgemm_tile<A_KC, B_KC, WAVES>(g, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.x, gridDim.y, gridDim.z);
}

// The discriminator's loss terms: half the squared errors of the real and of the simulated rows (the output gradient is the error itself), and
// the penalty, factor times the sum of its tiles' sums of squares, all in a fixed order.  One workgroup of 1024 threads.
struct DiscLosses {
  int64_t n_real, n, tiles;
  const float* err;
  const double* sums;
  double factor;
  float* losses;
};
__device__ __forceinline__ void disc_losses(const DiscLosses& d) {
  __shared__ double sh[3][1024];
  double a = 0.0, b = 0.0, c = 0.0;
  for (int64_t i = threadIdx.x; i < d.n; i += 1024) {
    const float e = d.err[i];
    if (i < d.n_real) a += 0.5 * (double)e * e; else b += 0.5 * (double)e * e;
  }
  for (int64_t i = threadIdx.x; i < d.tiles; i += 1024) c += d.sums[i];
  sh[0][threadIdx.x] = a; sh[1][threadIdx.x] = b; sh[2][threadIdx.x] = c;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int k = 0; k < 3; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) { d.losses[0] = (float)sh[0][0]; d.losses[1] = (float)sh[1][0]; d.losses[2] = (float)(d.factor * sh[2][0]); }
}

// Every weight and bias gradient of the discriminator in one launch, the penalty's share and the ordinary one as one reduction over both
// passes' rows; the first workgroup adds up the losses.  They were six launches of 9.5 us, each too small to fill the chip.
struct SgemmGroup {
  int n;
  int first[KS_MAX_LAYERS + 1];  // workgroups [first[l], first[l + 1]) behind the first one belong to product l
  int slices[KS_MAX_LAYERS];
  SgemmArgs g[KS_MAX_LAYERS];
};
__global__ __launch_bounds__(1024) void disc_wgrad_kernel(SgemmGroup t, DiscLosses d) {
  if (blockIdx.x == 0) {
    disc_losses(d);
    return;
  }
  const int b = blockIdx.x - 1;
  int l = 0;
  while (l + 1 < t.n && b >= t.first[l + 1]) ++l;
  const SgemmArgs& g = t.g[l];
  const int gx = (g.M + 31) / 32, gy = (g.N + 31) / 32, at = b - t.first[l], tile = at % (gx * gy);
  sgemm_tile<false, false, 16>(g, tile % gx, tile / gx, at / (gx * gy), gx, gy, t.slices[l]);
}

// Everything of the discriminator's gradient that stays inside a frame, in one launch: the forward pass, the input gradient's chain and the sweep
// back through it on the real rows, the ordinary backward pass.  A workgroup takes 16 rows through all of it, the operand of the next product in
// LDS, 16 columns of a product to a wavefront on v_mfma_f32_16x16x4_f32, the weights straight from L2.  Arrays that a later phase reads by entry
// (y, a, r) are read by the thread that wrote them.
// Few frames are bound by the chain of products itself (63 us for 2 x 1024 frames of 71-256-256-1, of which the matrix instructions are 17), where
// a launch per product (sgemm_kernel) added a launch, its gap and a trip of the operands through memory to each.  The whole gradient of
// 71-256-256-1, launches per product -> this: 2 x 32 frames 78 -> 66 us, 2 x 1024 101 -> 81, 2 x 12288 538 -> 382, 2 x 131072 5575 -> 3982;
// 71-128-128-1 67 -> 36, 73 -> 46, 243 -> 181, 2298 -> 1897; 60-256-1 44 -> 24, 50 -> 31, 194 -> 112, 1907 -> 1130.
// Requesting a product's first weights before the stores of the one before it was slower (63 -> 68 us).
struct DiscRowsArgs {
  int L, act, penalty, lda, zeros, tiles_real;
  int64_t R, M;
  float scale;
  const float *real, *sim;
  int dims[KS_MAX_LAYERS + 1], ld[KS_MAX_LAYERS];
  const float *W[KS_MAX_LAYERS], *b[KS_MAX_LAYERS];
  float *y[KS_MAX_LAYERS], *a[KS_MAX_LAYERS], *d[KS_MAX_LAYERS], *r[KS_MAX_LAYERS], *v[KS_MAX_LAYERS], *dz[KS_MAX_LAYERS];
  float *g, *ones;
  double* sums;  // one sum of squares per tile of real rows
  unsigned* zero;
};
constexpr int kDrRows = 16, kDrWaves = 16;

// Columns j0 .. j0 + 15 of op (16 rows, K) times W^T (KC: W stored (j, k)) or W (stored (k, j)); op: this lane's row at its first k, zeros from K to
// the next multiple of 16.  A lane of quarter h feeds k = 16 s + 4 h + e to instruction e of step s; four steps' weights are in flight under four
// steps' products.  Columns from N on repeat the last one.
// Four sums of at most sixteen products each, added up every four steps: error against 64 bits, root mean square in units of 2^-24 of the result,
// K = 64 / 128 / 256 1.4 / 1.5 / 1.6, where two sums over the whole reduction gave 1.8 / 2.4 / 3.3 and sgemm_kernel's four wavefronts 1.4 / 1.9 / 2.5.
// The whole gradient of 2 x 1024 frames against two sums: 71-256-256-1 80.2 -> 80.8 us, 71-128-128-1 44.8 -> 46.2; folded only every eight steps 83.
template <bool KC>
__device__ __forceinline__ f32x4 disc_product(const float* __restrict__ op, const float* __restrict__ W, int ld, int K, int N, int j0, int lane) {
  const int j = min(j0 + (lane & 15), N - 1), h = lane >> 4, nk = (K + 15) / 16;
  float w[16], next[16];
  const unsigned own = KC ? (unsigned)(j * ld + 4 * h) : (unsigned)(4 * h * ld + j);  // beside an address that the whole wavefront shares
  auto fetch = [&](float (&t)[16], int s0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k0 = 16 * min(s0 + s, nk - 1);
      if (KC) {
        const float4 x = *reinterpret_cast<const float4*>(W + k0 + own);
        t[4 * s] = x.x; t[4 * s + 1] = x.y; t[4 * s + 2] = x.z; t[4 * s + 3] = x.w;
      } else if (k0 + 16 <= K) {
#pragma unroll
        for (int e = 0; e < 4; ++e) t[4 * s + e] = (W + (int64_t)(k0 + e) * ld)[own];
      } else {  // the reduction ends inside the step: zeros past it, as the operand's (a repeated row that holds an infinity would make them NaN)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = k0 + 4 * h + e;
          const float x = W[(int64_t)min(k, K - 1) * ld + j];
          t[4 * s + e] = k < K ? x : 0.f;
        }
      }
    }
  };
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  fetch(w, 0);
  for (int s0 = 0; s0 < nk; s0 += 4) {
    if (s0 + 4 < nk) fetch(next, s0 + 4);
    f32x4 part[4] = {};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (s0 + s < nk) {
        const float4 x = *reinterpret_cast<const float4*>(op + 16 * (s0 + s));
        part[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, w[4 * s], part[0], 0, 0, 0);
        part[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, w[4 * s + 1], part[1], 0, 0, 0);
        part[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, w[4 * s + 2], part[2], 0, 0, 0);
        part[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, w[4 * s + 3], part[3], 0, 0, 0);
      }
#pragma unroll
    for (int s = 0; s < 16; ++s) w[s] = next[s];
    sum += (part[0] + part[1]) + (part[2] + part[3]);
  }
  return sum;
}

__global__ __launch_bounds__(64 * kDrWaves) void disc_rows_kernel(const DiscRowsArgs a) {
  extern __shared__ __align__(16) float disc_rows_lds[];
  __shared__ float err[kDrRows];
  __shared__ double sred[kDrWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, h = lane >> 4, L = a.L, lda = a.lda;
  const bool real = (int)blockIdx.x < a.tiles_real, pen = real && a.penalty;
  const int64_t row0 = real ? (int64_t)blockIdx.x * kDrRows : a.R + (int64_t)((int)blockIdx.x - a.tiles_real) * kDrRows;
  const int64_t left = (real ? a.R : a.M) - row0;
  const int rows = left < kDrRows ? (int)left : kDrRows;
  float *cur = disc_rows_lds, *nxt = cur + kDrRows * lda, *top = nxt + kDrRows * lda;
  const int at = c * lda + 4 * h;  // this lane's operand
  if (blockIdx.x == 0)
    for (int x = tid; x < a.zeros; x += 64 * kDrWaves) a.zero[x] = 0;
  {
    const int K = a.dims[0], w16 = (K + 15) / 16 * 16;
    const float* x = real ? a.real + row0 * K : a.sim + (row0 - a.R) * K;
    for (int e = tid; e < kDrRows * w16; e += 64 * kDrWaves) {
      const int i = e / w16, k = e - i * w16;
      cur[i * lda + k] = i < rows && k < K ? x[i * K + k] : 0.f;
    }
  }
  __syncthreads();
  auto turn = [&]() {
    __syncthreads();  // the next operand is whole; the one before it can be overwritten
    float* t = cur;
    cur = nxt;
    nxt = t;
  };
  // own entries (4 h + r, j) of a row-major array of width N, zero where there is none
  auto own = [&](const float* p, int N, int j, float (&v)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = j < N && 4 * h + r < rows ? p[(row0 + 4 * h + r) * N + j] : 0.f;
  };

  for (int l = 0; l + 1 < L; ++l) {
    const int N = a.dims[l + 1];
    const bool opens = pen && l == L - 2;
    for (int j0 = 16 * wave; j0 < N; j0 += 16 * kDrWaves) {
      const f32x4 z = disc_product<true>(cur + at, a.W[l], a.ld[l], a.dims[l], N, j0, lane);
      const int j = j0 + c;
      const float bias = j < N ? a.b[l][j] : 0.f, x = opens && j < N ? a.W[L - 1][j] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * h + r;
        const bool held = j < N && i < rows;
        float y = z[r] + bias, d1, d2;
        if (a.act == KS_ACT_ELU) y = y > 0.f ? y : expm1f(y);
        else if (a.act == KS_ACT_RELU) y = fmaxf(y, 0.f);
        else if (a.act == KS_ACT_TANH) y = tanhf(y);
        nxt[i * lda + j] = j < N ? y : 0.f;
        const int64_t o = (row0 + i) * N + j;
        if (held) a.y[l][o] = y;
        if (!opens) continue;
        act_derivatives(a.act, y, d1, d2);
        const float dd = d1 * x;
        top[i * lda + j] = j < N ? dd : 0.f;
        if (held) { a.a[l][o] = x; a.d[l][o] = dd; }
      }
    }
    turn();
  }
  {  // the output layer, a row to a wavefront
    float s = 0.f;
    for (int k = lane; k < a.dims[L - 1]; k += 64) s += cur[wave * lda + k] * a.W[L - 1][k];
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w);
    if (lane == 0) {
      const float e = s + a.b[L - 1][0] - (real ? 1.f : -1.f);
      err[wave] = e;
      if (wave < rows) {
        a.dz[L - 1][row0 + wave] = e;
        if (real) a.ones[row0 + wave] = 1.f;
      }
    }
  }
  __syncthreads();

  if (pen) {
    float* t = cur;  // the chain starts from the d that the last hidden layer left
    cur = top;
    top = t;
    for (int l = L - 2; l > 0; --l) {
      const int N = a.dims[l];
      for (int j0 = 16 * wave; j0 < N; j0 += 16 * kDrWaves) {
        const int j = j0 + c;
        float y[4], d1, d2;
        own(a.y[l - 1], N, j, y);
        const f32x4 z = disc_product<false>(cur + at, a.W[l], a.ld[l], a.dims[l + 1], N, j0, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 4 * h + r;
          act_derivatives(a.act, y[r], d1, d2);
          const float dd = d1 * z[r];
          nxt[i * lda + j] = j < N ? dd : 0.f;
          if (j < N && i < rows) { a.a[l - 1][(row0 + i) * N + j] = z[r]; a.d[l - 1][(row0 + i) * N + j] = dd; }
        }
      }
      turn();
    }
    double sq = 0.0;
    {
      const int N = a.dims[0];
      for (int j0 = 16 * wave; j0 < N; j0 += 16 * kDrWaves) {
        const f32x4 z = disc_product<false>(cur + at, a.W[0], a.ld[0], a.dims[1], N, j0, lane);
        const int j = j0 + c;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 4 * h + r;
          const float gg = a.scale * z[r];
          nxt[i * lda + j] = j < N ? gg : 0.f;
          if (j < N && i < rows) {
            a.g[(row0 + i) * N + j] = gg;
            sq += (double)z[r] * z[r];
          }
        }
      }
    }
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) sq += __shfl_down(sq, w);
    if (lane == 0) sred[wave] = sq;
    turn();
    if (tid == 0) {
      double s = 0.0;
      for (int w = 0; w < kDrWaves; ++w) s += sred[w];
      a.sums[blockIdx.x] = s;
    }
    for (int l = 1; l < L; ++l) {
      const int N = a.dims[l];
      for (int j0 = 16 * wave; j0 < N; j0 += 16 * kDrWaves) {
        const int j = j0 + c;
        float y[4], x[4], d1, d2;
        own(a.y[l - 1], N, j, y);
        own(a.a[l - 1], N, j, x);
        const f32x4 z = disc_product<true>(cur + at, a.W[l - 1], a.ld[l - 1], a.dims[l - 1], N, j0, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 4 * h + r;
          act_derivatives(a.act, y[r], d1, d2);
          const float vv = z[r] * d1;
          nxt[i * lda + j] = j < N ? vv : 0.f;
          if (j < N && i < rows) { a.r[l - 1][(row0 + i) * N + j] = z[r] * x[r] * d2; a.v[l - 1][(row0 + i) * N + j] = vv; }
        }
      }
      turn();
    }
  }

  for (int l = L; l > 1; --l) {  // gradient of z_{l-1}
    const int N = a.dims[l - 1];
    for (int j0 = 16 * wave; j0 < N; j0 += 16 * kDrWaves) {
      const int j = j0 + c;
      float y[4], x[4] = {0.f, 0.f, 0.f, 0.f}, d1, d2;
      own(a.y[l - 2], N, j, y);
      if (pen) own(a.r[l - 2], N, j, x);
      f32x4 z;
      if (l == L) {
        const float w = j < N ? a.W[L - 1][j] : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = err[4 * h + r] * w;
      } else {
        z = disc_product<false>(cur + at, a.W[l - 1], a.ld[l - 1], a.dims[l], N, j0, lane);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * h + r;
        act_derivatives(a.act, y[r], d1, d2);
        const float dd = z[r] * d1 + x[r];
        nxt[i * lda + j] = j < N ? dd : 0.f;
        if (j < N && i < rows) a.dz[l - 2][(row0 + i) * N + j] = dd;
      }
    }
    turn();
  }
}

// The weight and bias gradient of a single layer over many rows, C(i, j) = sum_k A(k, i) B(k, j) with both operands fp32 and stored
// (k, .), on the bf16 matrix instruction.  PARTS = 1: operands rounded to bf16, what a bf16 network's products take.  PARTS = 3: fp32, every
// value cut in three (cut_bf16, mma_cut).
// A 128 x 128 tile per workgroup of two groups of four wavefronts; each group takes half of the slice's rows in stages of 32 and each of
// its wavefronts a 64 x 64 block.  The groups take turns: while one multiplies out of its LDS buffer the other cuts the stage it has in
// registers, writes it to its own and requests the next, so a SIMD has one wavefront of matrix work and one of vector work at any time.
// A thread holds 8 rows x 4 columns of a stage, and a fragment is 8 rows of one column: 16-byte loads and 16-byte LDS writes.  Column
// 4 l + e of the tile goes to slot 32 e + l, so that neighbouring lanes write neighbouring fragments; a matrix tile is then every fourth
// column.
// `colsum` also receives sum_k A(k, i), the bias gradient, from the fp32 values in the loaders' registers.
// The k range is cut into slices of kslice; with more than one slice, slice z writes its partial product (M, N) densely to
// C + z * M * N and its column sums to colsum + z * M, and sum_slices_kernel adds them up in a fixed order.
// A launch takes the products of several layers, whose workgroups follow one another: each by itself cuts a few thousand rows into as many
// slices as there are CUs and is over in two launches of a few microseconds (twelve layers of a GRU actor and critic, 12288 rows: 24 launches,
// 194 us -> two, 135 us; a seventh of the slices for each of the twelve: the same, at that many rows the operands' way in sets the pace).
// Bound by the matrix instructions (eight per product of 16 rows, 64 us at the first size below) and the cuts beside them; the operands
// take 44 us at the card's copy rate.  The predecessor multiplied on the fp32 instruction, whose time alone is 87 us there.
//   102400 x 512 x 128, fp32: 122 -> 93 us (110 -> 145 TFLOP/s); relative error against 64 bits 7.3e-7 -> 1.9e-7
//   12288 x 384 x 128, bf16: 44 us in five launches (cast, two transposes, product, column sums) -> 11.4
// EDGE: a width is no multiple of four.
constexpr int kTnKB = 32;  // rows of a stage
__host__ __device__ constexpr int tn_buf(int parts) { return parts * (kTnKB / 8) * 256; }  // one group's LDS buffer, in 16-byte fragments

struct WgradJob {
  int M, N, K, kslice, tiles, slices;
  const float *A, *B;
  int64_t lda, ldb, ldc;
  float *C, *colsum;        // the gradients
  float *part, *colpart;    // partial products and column sums, where there is more than one slice
  unsigned first, first_sum;  // the job's first workgroup in wgrad_kernel and in sum_slices_kernel
};
// Twelve: two networks of two recurrent layers.  A table of 36 changes nothing up to three layers and gives 1 to 2 % of an update at five (LSTM, 12800
// rows: 2643 -> 2588 us).
constexpr int kWgradJobs = 12;
// A layer by itself has kernels of its own (JOBS = 1): the search for a workgroup's job and its place in it are two or three loads and a division one
// after the other (bf16, 12288 rows of 128 -> 384: 15.2 us, 16.0 through the search; of 128 -> 1: 10.9 and 11.3).
template <int JOBS>
struct WgradTable {
  int n;
  WgradJob job[JOBS];
};
template <int JOBS>
__device__ __forceinline__ const WgradJob& wgrad_find(const WgradTable<JOBS>& table, unsigned WgradJob::*first) {
  int which = 0;
  if constexpr (JOBS > 1)
    while (which + 1 < table.n && blockIdx.x >= table.job[which + 1].*first) ++which;
  return table.job[which];
}

template <int PARTS, bool EDGE, int JOBS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void wgrad_kernel(const WgradTable<JOBS> table) {
  extern __shared__ __attribute__((aligned(16))) u32x4 tn_lds[];  // [group][part][8 rows][slot: 128 of A, 128 of B]
  const WgradJob& job = wgrad_find(table, &WgradJob::first);
  const int M = job.M, N = job.N, K = job.K, kslice = job.kslice, tiles = JOBS > 1 ? job.tiles : gridDim.x, slices = JOBS > 1 ? job.slices : gridDim.y;
  const int lb = JOBS > 1 ? (int)(blockIdx.x - job.first) : (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (JOBS > 1 && lb >= tiles * slices) return;  // the workgroups that fill up the job's last eight
  const float *__restrict__ A = job.A, *__restrict__ B = job.B;
  const int64_t lda = job.lda, ldb = job.ldb, ldc = job.ldc;
  const bool sliced = slices > 1;
  float *__restrict__ C = sliced ? job.part : job.C, *__restrict__ colsum = sliced ? job.colpart : job.colsum;
  // Workgroup l runs on XCD l % 8: the tiles of one slice, which read the same rows, go to one XCD one after the other
  int tile = blockIdx.x, z = blockIdx.y;
  if constexpr (JOBS > 1) {
    tile = lb % tiles;
    z = lb / tiles;
  }
  if (slices % 8 == 0) {
    const int q = lb >> 3;
    tile = q % tiles;
    z = (q / tiles) * 8 + (lb & 7);
  }
  const int tiles_n = (N + 127) / 128;
  const int grp = threadIdx.x >> 8, t = threadIdx.x & 255, i0 = tile / tiles_n * 128, j0 = tile % tiles_n * 128;
  const int zbeg = min(K, z * kslice), zend = min(K, zbeg + kslice);
  const int half = ((zend - zbeg + 2 * kTnKB - 1) / (2 * kTnKB)) * kTnKB;  // rows per group, in whole stages; the same number for both
  const int kbeg = min(zend, zbeg + grp * half), kend = min(zend, kbeg + half), stages = half / kTnKB;
  const int wave = t >> 6, lane = t & 63, c = lane & 31, h = lane >> 5;
  const int ea = (wave >> 1) * 2, eb = (wave & 1) * 2;  // first of the wavefront's two matrix tiles of either operand
  f32x16 acc[2][2], low[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = low[a][b][r] = 0.f;
  // threads 0-127 of a group load A, the others B: rows 8 kg + r, columns 4 l + e; columns past the matrix repeat its last ones, whose
  // products are not stored
  const bool isb = t >= 128;
  const int kg = (t & 127) >> 5, l = t & 31;
  const int width = isb ? N : M, c0 = (isb ? j0 : i0) + 4 * l;
  const int64_t ld = isb ? ldb : lda;
  const float* src = (isb ? B : A) + (int64_t)(kbeg + 8 * kg) * ld;
  // four columns that reach over the matrix's edge (EDGE; at most one lane of a tile's row) are loaded one by one
  const bool edge = EDGE && c0 < width + (width < 4 ? 128 : 0) && c0 + 4 > width;
  const int first = max(0, min(c0, width - 4));
  float4 v[8];
  float4 cs = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int n) __attribute__((always_inline)) {
    const int k0 = kbeg + kTnKB * n + 8 * kg;
    const float* q = src + (int64_t)n * kTnKB * ld;
    const bool full = kbeg + kTnKB * (n + 1) <= kend;  // otherwise the group's last rows, and zeros beyond them
    if (edge) {
      const int a0 = min(c0, width - 1), a1 = min(c0 + 1, width - 1), a2 = min(c0 + 2, width - 1), a3 = min(c0 + 3, width - 1);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float* p = q + r * ld;
        v[r] = float4{0.f, 0.f, 0.f, 0.f};
        if (full || k0 + r < kend) v[r] = float4{p[a0], p[a1], p[a2], p[a3]};
      }
    } else if (full) {
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = load4_any(q + r * ld + first);
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        v[r] = float4{0.f, 0.f, 0.f, 0.f};
        if (k0 + r < kend) v[r] = load4_any(q + r * ld + first);
      }
    }
  };
  u32x4* buf = tn_lds + grp * tn_buf(PARTS);
  auto put = [&]() __attribute__((always_inline)) {
    if (!isb)
#pragma unroll
      for (int r = 0; r < 8; ++r) { cs.x += v[r].x; cs.y += v[r].y; cs.z += v[r].z; cs.w += v[r].w; }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float f[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = e == 0 ? v[r].x : e == 1 ? v[r].y : e == 2 ? v[r].z : v[r].w;
      u32x4 part[PARTS];
      cut_bf16<PARTS>(f, part);
#pragma unroll
      for (int p = 0; p < PARTS; ++p) buf[(p * (kTnKB / 8) + kg) * 256 + (isb ? 128 : 0) + 32 * e + l] = part[p];
    }
  };
  auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < kTnKB / 16; ++s) {
      bf16x8 fa[PARTS][2], fb[PARTS][2];
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const u32x4* at_k = buf + (p * (kTnKB / 8) + 2 * s + h) * 256 + c;
          fa[p][q] = __builtin_bit_cast(bf16x8, at_k[32 * (ea + q)]);
          fb[p][q] = __builtin_bit_cast(bf16x8, at_k[128 + 32 * (eb + q)]);
        }
      if constexpr (PARTS == 3) mma_cut(fa, fb, acc, low);
      else mma_bf16(fa[0], fb[0], acc);
    }
  };
  if (stages > 0) fetch(0);
  for (int p = 0; p <= 2 * stages; ++p) {
    const int n = (p - grp) >> 1;
    if (((p ^ grp) & 1) == 0) {
      if (n < stages) {
        put();
        if (n + 1 < stages) fetch(n + 1);
      }
    } else if (p > grp) {
      multiply();
    }
    // LDS only: the requested rows stay in flight over it
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  if constexpr (PARTS == 3)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = join_cut(acc[a][b][r], low[a][b][r]);
  // the second group hands its tile over in two halves through the buffers, which are free now
  float* mine = reinterpret_cast<float*>(tn_lds) + t;
  for (int a = 0; a < 2; ++a) {
    if (grp == 1) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(16 * b + r) * 256] = a == 0 ? acc[0][b][r] : acc[1][b][r];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if (a == 0) acc[0][b][r] += mine[(16 * b + r) * 256];
          else acc[1][b][r] += mine[(16 * b + r) * 256];
        }
    }
    __syncthreads();
  }
  if (colsum && j0 == 0) {
    float* sums = reinterpret_cast<float*>(tn_lds);  // [group][8 rows][128]
    if (!isb) *reinterpret_cast<float4*>(sums + (grp * 4 + kg) * 128 + 4 * l) = cs;
    __syncthreads();
    if (threadIdx.x < 128 && i0 + (int)threadIdx.x < M) {
      float s = 0.f;
      for (int r = 0; r < 8; ++r) s += sums[r * 128 + threadIdx.x];
      colsum[(sliced ? (int64_t)z * M : 0) + i0 + threadIdx.x] = s;
    }
  }
  if (grp == 1) return;
  float* out = sliced ? C + (int64_t)z * M * N : C;
  const int64_t ldo = sliced ? N : ldc;
  const int gj = j0 + 4 * c + eb;
  const bool pair = ldo % 2 == 0 && ((uintptr_t)out & 7) == 0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int gi = i0 + 4 * (8 * (r >> 2) + 4 * h + (r & 3)) + ea + a;
      if (gi >= M || gj >= N) continue;
      float* o = out + (int64_t)gi * ldo + gj;
      if (pair && gj + 1 < N) {
        *reinterpret_cast<float2*>(o) = float2{acc[a][0][r], acc[a][1][r]};
      } else {
        o[0] = acc[a][0][r];
        if (gj + 1 < N) o[1] = acc[a][1][r];
      }
    }
}

// C = the sum of nz slices of (M, N), and colsum = the sum of nz rows of M behind it in the same launch.  A workgroup takes 64 entries,
// a quarter of the slices to each wavefront with 16 loads in flight, then adds the four in order.
template <int JOBS>
__global__ __launch_bounds__(256) void sum_slices_kernel(const WgradTable<JOBS> table) {
  __shared__ float sh[256];
  const WgradJob& job = wgrad_find(table, &WgradJob::first_sum);
  const int M = job.M, N = job.N, nz = job.slices;
  const float *__restrict__ part = job.part, *__restrict__ colpart = job.colpart;
  float *__restrict__ C = job.C, *__restrict__ colsum = job.colsum;
  const int64_t ldc = job.ldc;
  const int64_t mn = (int64_t)M * N, wblocks = (mn + 63) / 64, block = blockIdx.x - job.first_sum;
  const bool col = block >= wblocks;
  const int64_t n = col ? M : mn, idx = (block - (col ? wblocks : 0)) * 64 + (threadIdx.x & 63);
  const float* src = col ? colpart : part;
  const int w = threadIdx.x >> 6, per = (nz + 3) / 4, zb = w * per, ze = min(nz, zb + per);
  float s = 0.f;
  if (idx < n)
    for (int z0 = zb; z0 < ze; z0 += 16) {
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = z0 + k < ze ? src[(int64_t)(z0 + k) * n + idx] : 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) s += v[k];
    }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (w > 0 || idx >= n) return;
  s = sh[threadIdx.x] + sh[threadIdx.x + 64] + sh[threadIdx.x + 128] + sh[threadIdx.x + 192];
  if (col) { colsum[idx] = s; return; }
  const int i = (int)(idx / N), j = (int)(idx - (int64_t)i * N);
  C[(int64_t)i * ldc + j] = s;
}

}  // namespace ks

struct DiscWs {
  float* y[KS_MAX_LAYERS];      // hidden outputs, all rows
  float* a[KS_MAX_LAYERS];      // real rows: W_{l+1}^T d_{l+1}
  float* d[KS_MAX_LAYERS];      // real rows: d_l
  float* r[KS_MAX_LAYERS];      // real rows: extra gradient of z_l
  float* v[KS_MAX_LAYERS];      // real rows: v_l of the sweep back, l = 1 .. L - 1
  float* dz[KS_MAX_LAYERS];     // all rows: gradient of z_l, l = 1 .. L at [l - 1]
  float *g, *ones, *part;
  unsigned* counters;
  double* sums;                 // one sum of squares per tile of the input gradient
};

static int64_t disc_penalty_tiles(const DevMlp& m, int64_t R) { return ((R + 31) / 32) * ((m.dims[0] + 31) / 32); }

// Floats of a row in disc_rows_kernel's LDS, 0 where the launches per product are to run: a linear network has no chain, and of networks wider than
// 320 only a few fit three operands of 16 rows into the 64 KiB that a launch has without asking (336 would; 320 is what was measured).  A second pass of the
// wavefronts over 257 columns and more costs less than the products' launches (71-272-272-1, launches -> chain, 2 x 32 / 1024 / 131072 frames: 88 -> 78,
// 127 -> 95, 8079 -> 5548 us; 71-320-320-1 93 -> 86, 150 -> 109, 9285 -> 5612).
// A hidden layer occupies a wavefront per 16 of its columns; where that leaves most of the sixteen idle, the launches per product win once the rows
// fill the chip, the sooner the narrower the widest hidden layer is and the fewer products there are, whatever the input's width.  Time of the chain over
// that of the launches at M rows in all, 20, 71 and 300 inputs, one and two hidden layers, with the penalty | without:
//   16 and 32 wide: M = 8192 0.56 to 0.70 | 0.68 to 0.91, 16384 0.80 to 0.90 | 0.92 to 1.16, 24576 0.89 to 1.01 | 1.11 to 1.18, 262144 1.16 to 1.53 | 1.41 to 1.74
//   48 wide: 16384 0.71 to 0.85 | 0.83 to 0.99, 65536 0.83 to 0.98 | one layer 1.02 to 1.09, two 0.90 to 0.98, 262144 0.89 to 1.08 | 0.97 to 1.16
//   64 wide, one layer: 16384 0.76 to 0.84 | 0.91 to 0.97, 65536 0.84 to 0.97 | 0.99 to 1.07, 262144 0.87 to 1.10 | 1.04 to 1.13
//   64 wide, two layers: 0.42 to 0.96 | 0.49 to 1.00 up to 262144 rows; 80 wide and wider 0.48 to 0.96 | 0.53 to 1.01
// (before a product's sums were folded every 64 columns, which adds up to 0.03 to the narrow ones: 20-65-1 at 262144 1.03 | 0.92, 20-16-1 at
// 24576 1.03, the others at the last rows of the rule below 0.79 to 1.00).
static int disc_rows_lda(const DevMlp& m, int64_t M, bool penalty) {
  int w = 0, hidden = 0;
  for (int l = 0; l < m.n_layers; ++l) {
    w = std::max(w, round_up(m.dims[l], 16));
    if (l > 0) hidden = std::max(hidden, m.dims[l]);
  }
  const bool deep = m.n_layers > 2;
  const int64_t most = hidden > 64 || (hidden > 48 && deep) ? M : hidden > 32 ? (penalty || deep ? 65536 : 16384) : (penalty ? 24576 : 8192);
  return m.n_layers > 1 && w <= 320 && M <= most ? w + 4 : 0;
}

static int64_t carve_disc(const DevMlp& m, int64_t R, int64_t M, char* base, DiscWs* ws) {
  int64_t off = 0;
  auto take = [&](int64_t floats) {
    char* p = base ? base + off : nullptr;
    off += (floats * 4 + 255) / 256 * 256;
    return (float*)p;
  };
  DiscWs w;
  std::memset(&w, 0, sizeof(w));
  for (int l = 0; l < m.n_layers; ++l) w.dz[l] = take(M * m.dims[l + 1]);
  for (int l = 0; l + 1 < m.n_layers; ++l) {
    w.v[l] = take(R * m.dims[l + 1]);
    w.y[l] = take(M * m.dims[l + 1]);
    w.a[l] = take(R * m.dims[l + 1]);
    w.d[l] = take(R * m.dims[l + 1]);
    w.r[l] = take(R * m.dims[l + 1]);
  }
  w.g = take(R * m.dims[0]);
  w.ones = take(R);
  w.sums = (double*)take(2 * std::max(disc_penalty_tiles(m, R), (R + ks::kDrRows - 1) / ks::kDrRows));
  w.part = take((int64_t)m.n_layers * 512 * kTilePart);  // a sliced product has at most 512 (slice, tile) pairs
  w.counters = (unsigned*)take((int64_t)m.n_layers * 512);
  if (ws) *ws = w;
  return off;
}

static void sgemm_finish_args(SgemmArgs& g) {
  if (!g.A2) { g.A2 = g.A; g.a_split = 0x7fffffff; }
  if (!g.B2) { g.B2 = g.B; g.b_split = 0x7fffffff; }
  if (!g.B3) { g.B3 = g.B2; g.b_split2 = 0x7fffffff; }
}

// One product over activations, whose reduction is a layer's width: four wavefronts share it.
template <bool B_KC>
static void sgemm_go(hipStream_t s, SgemmArgs g) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return;
  sgemm_finish_args(g);
  g.kslice = (g.K + 15) / 16 * 16;
  hipLaunchKernelGGL((sgemm_kernel<true, B_KC, 4>), dim3((unsigned)((g.M + 31) / 32), (unsigned)((g.N + 31) / 32)), dim3(256), 0, s, g);
}

// Slices for the products of a group, whose reductions over the same K rows all get as many: the fewest rounds of workgroups over the CUs (one of
// 1024 threads at a time each), weighed against the rows left to a wavefront.  A workgroup takes about 8 us beside its products, 32 rows of its
// sixteen wavefronts 1.7; a slice keeps the 512 rows that give every wavefront a chunk of loads.  (1024 + 1024 frames, 71-256-256-1: 96 tiles
// in two slices 19 us; sliced one by one, 384 workgroups, they took 29.)
static int group_slices(int tiles, int widest, int64_t K) {
  int best = 1;
  double least = 0.0;
  for (int s = 1; s <= kDiscMaxSlices && (s == 1 || (K >= 512ll * s && widest * s <= 512)); ++s) {
    const double t = ((tiles * s + 256) / 256) * (8.0 + 1.7 * (double)((K + 512ll * s - 1) / (512ll * s)));  // one more for the losses
    if (s == 1 || t < least) { least = t; best = s; }
  }
  return best;
}

static int group_blocks(SgemmGroup& t) {
  int tiles = 0, widest = 0;
  for (int k = 0; k < t.n; ++k) {
    const int n = ((t.g[k].M + 31) / 32) * ((t.g[k].N + 31) / 32);
    tiles += n;
    widest = n > widest ? n : widest;
  }
  int blocks = 0;
  for (int k = 0; k < t.n; ++k) {
    SgemmArgs& g = t.g[k];
    sgemm_finish_args(g);
    const int want = group_slices(tiles, widest, g.K);
    g.kslice = (((g.K + want - 1) / want) + 15) / 16 * 16;
    t.slices[k] = (g.K + g.kslice - 1) / g.kslice;
    t.first[k] = blocks;
    blocks += ((g.M + 31) / 32) * ((g.N + 31) / 32) * t.slices[k];
  }
  return blocks;
}

// C (M, N) = A^T B over K rows with the column sums of A beside it, on 128 x 128 tiles: the weight and bias gradient of a single layer.
static WgradJob wgrad_job(int64_t M, int N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc, float* part,
                          float* colsum) {
  WgradJob j;
  j.M = (int)M; j.N = N; j.K = (int)K; j.A = A; j.lda = lda; j.B = B; j.ldb = ldb; j.C = C; j.ldc = ldc; j.colsum = colsum; j.part = part;
  j.tiles = (int)(((M + 127) / 128) * ((N + 127) / 128));
  j.slices = wgrad_slices(M, N, K);  // the layer's own number, so that a gradient does not depend on what it shares the launch with
  j.kslice = (int)(((K + j.slices - 1) / j.slices + 2 * kTnKB - 1) / (2 * kTnKB)) * 2 * kTnKB;  // slices past the last row add zeros
  j.colpart = part + (int64_t)j.slices * M * N;
  j.first = j.first_sum = 0;
  return j;
}

// Several of them, of one kind: a launch for the products and one for the sums of their slices
template <int PARTS, int JOBS>
static int launch_wgrads(hipStream_t s, const WgradTable<JOBS>& t, dim3 grid, unsigned sums, bool edge) {
  constexpr int lds = 2 * tn_buf(PARTS) * 16;
  auto kfn = edge ? wgrad_kernel<PARTS, true, JOBS> : wgrad_kernel<PARTS, false, JOBS>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(KS_ELAUNCH, "ks_mlp_train_backward: cannot raise the LDS limit to %d bytes", lds);
  hipLaunchKernelGGL(kfn, grid, dim3(512), lds, s, t);
  if (sums) hipLaunchKernelGGL(sum_slices_kernel<JOBS>, dim3(sums), dim3(256), 0, s, t);
  return KS_OK;
}

template <int PARTS, int JOBS>
static int wgrads(hipStream_t s, WgradTable<JOBS>& t) {
  unsigned blocks = 0, sums = 0;
  bool edge = false;
  for (int k = 0; k < t.n; ++k) {
    WgradJob& j = t.job[k];
    edge |= j.M % 4 || j.N % 4;
    j.first = blocks;
    blocks += (unsigned)round_up(j.tiles * j.slices, 8);  // the next job's slices stay on the XCDs they are meant for
    j.first_sum = sums;
    if (j.slices > 1) sums += (unsigned)(((int64_t)j.M * j.N + 63) / 64 + (j.M + 63) / 64);
  }
  if (t.n > 1) return launch_wgrads<PARTS>(s, t, dim3(blocks), sums, edge);
  const WgradTable<1> one = {1, {t.job[0]}};
  return launch_wgrads<PARTS>(s, one, dim3((unsigned)one.job[0].tiles, (unsigned)one.job[0].slices), sums, edge);
}

template <int PARTS>
static int wgrad(hipStream_t s, int64_t M, int N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                 int64_t ldc, float* part, float* colsum) {
  WgradTable<1> t;
  t.n = 1;
  t.job[0] = wgrad_job(M, N, K, A, lda, B, ldb, C, ldc, part, colsum);
  return wgrads<PARTS>(s, t);
}

// ---------------------------------------------------------------------------------------------
// backward pass of several single layers, e.g. all projections of a recurrent actor and critic
// ---------------------------------------------------------------------------------------------
// The gradient of the network input by a single layer of bf16: the whole-network kernel over the transposed fragments
static bool single_dx_ok(const DevMlp& m) { return m.dtype == KS_MLP_BF16 && m.WtP[0]; }

static int64_t wgrad_part_floats(const DevMlp& m, int64_t M) { return (int64_t)wgrad_slices(m.dims[1], m.dims[0], M) * m.dims[1] * (m.dims[0] + 1); }

static int check_layer_backward(const KsLayerBackward& q) {
  if (!q.mlp || !q.mlp->m.train) return fail(KS_EINVAL, "ks_mlps_layer_backward: call ks_mlp_train_init first");
  if (q.mlp->m.n_layers != 1) return fail(KS_EINVAL, "ks_mlps_layer_backward: the network has %d layers, not one", q.mlp->m.n_layers);
  if (q.M <= 0 || !q.dy || (!q.x && !q.dx) || (q.x && q.ldx < q.mlp->m.dims[0])) return fail(KS_EINVAL, "ks_mlps_layer_backward: bad argument");
  if (q.M > (1 << 30)) return fail(KS_ELIMIT, "ks_mlps_layer_backward: too many rows");
  return KS_OK;
}

extern "C" int64_t ks_mlps_layer_backward_workspace_bytes(int32_t n, const KsLayerBackward* q) {
  int64_t parts = 0, most = 0;
  for (int k = 0; q && k < n; ++k) {
    if (!q[k].mlp || q[k].M < 0) return 0;
    const DevMlp& m = q[k].mlp->m;
    if (q[k].x) parts += (wgrad_part_floats(m, q[k].M) * 4 + 255) / 256 * 256;
    if (q[k].dx && m.dtype == KS_MLP_BF16 && !single_dx_ok(m)) most = std::max(most, carve_train(m, q[k].M, nullptr, nullptr));
  }
  return std::max(parts, most) + 256;
}

extern "C" int ks_mlps_layer_backward(int32_t n, const KsLayerBackward* q, ks_stream_t stream, void* workspace) {
  if (n < 0 || (n > 0 && (!q || !workspace))) return fail(KS_EINVAL, "ks_mlps_layer_backward: bad argument");
  for (int k = 0; k < n; ++k)
    if (const int rc = check_layer_backward(q[k])) return rc;
  // entries that need one another's results, or write one gradient, by themselves in their order
  bool apart = true;
  for (int k = 0; k < n; ++k) {
    const Span dx = {q[k].dx, q[k].M * q[k].mlp->m.dims[0]};
    for (int j = 0; j < n; ++j) {
      if (j == k) continue;
      const int in = q[j].mlp->m.dims[0];
      apart &= !(meet(dx, {q[j].x, (q[j].M - 1) * q[j].ldx + in}) || meet(dx, {q[j].dy, q[j].M * q[j].mlp->m.dims[1]}) || meet(dx, {q[j].dx, q[j].M * in}) ||
                 (q[j].mlp == q[k].mlp && q[j].x && q[k].x));
    }
  }
  if (!apart) {
    for (int k = 0; k < n; ++k)
      if (const int rc = ks_mlps_layer_backward(1, q + k, stream, workspace)) return rc;
    return KS_OK;
  }
  hipStream_t s = (hipStream_t)stream;
  // input gradients: those of bf16 layers two to a launch, each with the next one that has its row tile
  FusedArgs held;
  int held_bm = 0;
  for (int k = 0; k < n; ++k) {
    if (!q[k].dx) continue;
    DevMlp& m = q[k].mlp->m;
    int rc = KS_OK;
    if (single_dx_ok(m)) {
      const FusedArgs a = single_dx_args(m, q[k].M, q[k].dy, q[k].dx);
      const int bm = a.M >= 128 * 256 ? 128 : 32;
      if (held_bm == bm) {
        rc = launch_single_pair(held, a, bm, s);
        held_bm = 0;
      } else {
        if (held_bm) rc = launch_fused_args(held, s);
        held = a;
        held_bm = bm;
      }
    } else if (m.dtype == KS_MLP_BF16) {
      TrainWs ws;
      carve_train(m, q[k].M, (char*)workspace, &ws);
      rc = train_backward_single<__bf16>(m, s, q[k].M, nullptr, 0, q[k].dy, ws, q[k].dx, false, false, nullptr);
    } else {
      rc = train_backward_single<float>(m, s, q[k].M, nullptr, 0, q[k].dy, TrainWs{}, q[k].dx, false, false, nullptr);  // writes dx itself: no workspace
    }
    if (rc != KS_OK) return rc;
  }
  if (held_bm)
    if (const int rc = launch_fused_args(held, s)) return rc;
  // weight gradients, those of a precision together
  char* part = (char*)workspace;
  for (int bf16 = 0; bf16 < 2; ++bf16) {
    WgradTable<kWgradJobs> t;
    t.n = 0;
    for (int k = 0; k <= n; ++k) {
      if (t.n == kWgradJobs || (k == n && t.n > 0)) {
        const int rc = bf16 ? wgrads<1>(s, t) : wgrads<3>(s, t);
        if (rc != KS_OK) return rc;
        t.n = 0;
      }
      if (k == n || !q[k].x || (q[k].mlp->m.dtype == KS_MLP_BF16) != (bf16 != 0)) continue;
      DevMlp& m = q[k].mlp->m;
      t.job[t.n++] = wgrad_job(m.dims[1], m.dims[0], q[k].M, q[k].dy, m.dims[1], q[k].x, q[k].ldx, m.gW[0], m.kpad[0], (float*)part, m.gb[0]);
      part += (wgrad_part_floats(m, q[k].M) * 4 + 255) / 256 * 256;
    }
  }
  return check_launch("ks_mlps_layer_backward");
}

extern "C" int64_t ks_mlp_disc_workspace_bytes(const KsMlp* h, int64_t n_real, int64_t n_sim) {
  if (!h || n_real < 0 || n_sim < 0) return 0;
  return carve_disc(h->m, n_real, n_real + n_sim, nullptr, nullptr) + 256;
}

extern "C" int ks_mlp_disc_loss_grad(KsMlp* h, ks_stream_t stream, int64_t n_real, const float* real, int64_t n_sim, const float* sim,
                                     float grad_penalty_coef, int64_t n_motions, float* losses, void* workspace) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_disc_loss_grad: call ks_mlp_train_init first");
  DevMlp& m = h->m;
  const int L = m.n_layers, act = m.activation;
  const int64_t R = n_real, M = n_real + n_sim;
  if (m.dims[L] != 1) return fail(KS_EINVAL, "ks_mlp_disc_loss_grad: the discriminator must have one output, not %d", m.dims[L]);
  if (act == KS_ACT_GELU) return fail(KS_EINVAL, "ks_mlp_disc_loss_grad: GELU is not supported here (ELU, ReLU, tanh or none)");
  if (n_real < 0 || n_sim < 0 || M <= 0 || (n_real > 0 && !real) || (n_sim > 0 && !sim) || !losses || !workspace)
    return fail(KS_EINVAL, "ks_mlp_disc_loss_grad: bad argument");
  if (M > 4000000) return fail(KS_ELIMIT, "ks_mlp_disc_loss_grad: %lld rows exceed the limit of 4000000", (long long)M);
  const bool penalty = grad_penalty_coef != 0.f && R > 0;
  if (penalty && (n_motions <= 0 || n_real % n_motions != 0))
    return fail(KS_EINVAL, "ks_mlp_disc_loss_grad: %lld real frames do not divide into %lld motions", (long long)n_real, (long long)n_motions);
  hipStream_t s = (hipStream_t)stream;
  DiscWs ws;
  carve_disc(m, R, M, (char*)workspace, &ws);
  SgemmArgs z = {};  // fields left out below are zero
  DiscLosses losses_of = {R, M, 0, ws.dz[L - 1], ws.sums, penalty ? 0.5 * (double)grad_penalty_coef * (double)(1.f / (float)n_motions) : 0.0, losses};
  const float penalty_scale = penalty ? grad_penalty_coef * (1.f / (float)n_motions) : 0.f;
  const int lda = disc_rows_lda(m, M, penalty);
  if (lda) {
    DiscRowsArgs a;
    std::memset(&a, 0, sizeof(a));
    a.L = L; a.act = act; a.penalty = penalty; a.lda = lda; a.zeros = 512 * L; a.zero = ws.counters;
    a.R = R; a.M = M; a.scale = penalty_scale; a.real = real; a.sim = sim; a.g = ws.g; a.ones = ws.ones; a.sums = ws.sums;
    a.tiles_real = (int)((R + kDrRows - 1) / kDrRows);
    for (int l = 0; l < L; ++l) {
      a.dims[l] = m.dims[l]; a.ld[l] = m.kpad[l]; a.W[l] = m.mW[l]; a.b[l] = m.mb[l]; a.y[l] = ws.y[l]; a.a[l] = ws.a[l];
      a.d[l] = ws.d[l]; a.r[l] = ws.r[l]; a.v[l] = ws.v[l]; a.dz[l] = ws.dz[l];
    }
    a.dims[L] = 1;
    if (penalty) losses_of.tiles = a.tiles_real;
    const int tiles = a.tiles_real + (int)((n_sim + kDrRows - 1) / kDrRows);
    hipLaunchKernelGGL(disc_rows_kernel, dim3((unsigned)tiles), dim3(64 * kDrWaves), 3 * kDrRows * lda * sizeof(float), s, a);
  } else {
    // forward over the real rows, then the simulated ones; the last hidden layer also opens the input gradient's chain (a, d of its output), the
    // output layer leaves the gradient of the squared errors
    for (int l = 0; l < L; ++l) {
      SgemmArgs g = z;
      g.M = (int)M; g.N = m.dims[l + 1]; g.K = m.dims[l];
      if (l > 0) g.A = ws.y[l - 1];
      else if (R == 0 || n_sim == 0) g.A = R ? real : sim;
      else { g.A = real; g.A2 = sim; g.a_split = (int)R; }
      g.lda = g.K; g.B = m.mW[l]; g.ldb = m.kpad[l];
      g.ldc = g.N; g.bias = m.mb[l]; g.act = act; g.x_rows = (int)R;
      if (l == 0) { g.zero = ws.counters; g.zeros = 512 * L; }
      if (l == L - 1) { g.epi = kEpiOut; g.C = ws.dz[l]; g.C2 = ws.ones; }
      else if (l == L - 2 && penalty) { g.epi = kEpiTop; g.C = ws.y[l]; g.X = m.mW[L - 1]; g.C2 = ws.a[l]; g.C3 = ws.d[l]; }
      else { g.epi = kEpiLayer; g.C = ws.y[l]; }
      sgemm_go<true>(s, g);
    }
    if (penalty) {
      // input gradient on the real rows: d_L = 1, d_{L-1} from the forward pass, down to g = d_1 W_1, which leaves its tiles as the penalty's
      // gradient
      for (int l = L > 1 ? L - 2 : 0; l >= 0; --l) {  // hidden layer l (its output is y[l - 1]); l = 0: the input
        SgemmArgs g = z;
        g.M = (int)R; g.N = m.dims[l]; g.K = m.dims[l + 1];
        g.A = l + 1 == L ? ws.ones : ws.d[l]; g.lda = g.K; g.B = m.mW[l]; g.ldb = m.kpad[l]; g.ldc = g.N; g.act = act;
        if (l > 0) { g.C = ws.a[l - 1]; g.C2 = ws.d[l - 1]; g.Y = ws.y[l - 1]; g.epi = kEpiDelta; }
        else { g.C = ws.g; g.epi = kEpiPenalty; g.scale = penalty_scale; g.sums = ws.sums; }
        sgemm_go<false>(s, g);
      }
      losses_of.tiles = disc_penalty_tiles(m, R);
      for (int l = 1; l < L; ++l) {  // the sweep back through that computation, first layer to last
        SgemmArgs g = z;
        g.M = (int)R; g.N = m.dims[l]; g.K = m.dims[l - 1];
        g.A = l == 1 ? ws.g : ws.v[l - 2]; g.lda = g.K; g.B = m.mW[l - 1]; g.ldb = m.kpad[l - 1];
        g.C = ws.v[l - 1]; g.C2 = ws.r[l - 1]; g.ldc = g.N; g.Y = ws.y[l - 1]; g.X = ws.a[l - 1]; g.act = act; g.epi = kEpiTangent;
        sgemm_go<true>(s, g);
      }
    }

    // ordinary backward pass of the squared-error terms over all rows, with r_l added on the real rows
    for (int l = L; l > 1; --l) {
      SgemmArgs g = z;
      g.M = (int)M; g.N = m.dims[l - 1]; g.K = m.dims[l]; g.A = ws.dz[l - 1]; g.lda = g.K; g.B = m.mW[l - 1]; g.ldb = m.kpad[l - 1];
      g.C = ws.dz[l - 2]; g.ldc = g.N; g.Y = ws.y[l - 2]; g.X = ws.r[l - 2]; g.x_rows = penalty ? (int)R : 0; g.act = act; g.epi = kEpiDz;
      sgemm_go<false>(s, g);
    }
  }

  // weight gradients: d_l^T v_{l-1} over the real rows, where there is a penalty, then dz_l^T y_{l-1} over all rows; the bias gradients are the
  // column sums of dz that ride along
  SgemmGroup t;
  t.n = 0;
  const int P = penalty ? (int)R : 0;
  for (int l = 1; l <= L; ++l) {
    SgemmArgs g = z;
    g.M = m.dims[l]; g.N = m.dims[l - 1]; g.K = P + (int)M; g.lda = g.M; g.ldb = g.N;
    const float *y0 = l > 1 ? ws.y[l - 2] : (R ? real : sim), *y1 = l == 1 && R && n_sim ? sim : nullptr;  // the rows' inputs, in one or two arrays
    if (penalty) {
      g.A = l == L ? ws.ones : ws.d[l - 1]; g.A2 = ws.dz[l - 1]; g.a_split = P;
      g.B = l == 1 ? ws.g : ws.v[l - 2]; g.B2 = y0; g.b_split = P;
      g.B3 = y1; g.b_split2 = P + (int)R;
    } else {
      g.A = ws.dz[l - 1]; g.B = y0; g.B2 = y1; g.b_split = (int)R;
    }
    g.C = m.gW[l - 1]; g.ldc = m.kpad[l - 1]; g.colsum = m.gb[l - 1]; g.cs_from = P;
    g.part = ws.part + (int64_t)(l - 1) * 512 * kTilePart; g.counters = ws.counters + (l - 1) * 512;
    t.g[t.n++] = g;
  }
  const int blocks = group_blocks(t);
  hipLaunchKernelGGL(disc_wgrad_kernel, dim3((unsigned)blocks + 1), dim3(1024), 0, s, t, losses_of);
  return check_launch("ks_mlp_disc_loss_grad");
}

// strided copy of the meaningful (out, in) block of a padded (npad, kpad) matrix
__global__ __launch_bounds__(256) void unpad_kernel(int rows, int cols, int ld, const float* __restrict__ src, float* __restrict__ dst) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)rows * cols) return;
  const int r = (int)(idx / cols), c = (int)(idx - (int64_t)r * cols);
  dst[idx] = src[(int64_t)r * ld + c];
}

extern "C" int ks_mlp_get_params(const KsMlp* h, ks_stream_t stream, int32_t l, float* weight, float* bias, int32_t gradients) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_get_params: call ks_mlp_train_init first");
  const DevMlp& m = h->m;
  if (l < 0 || l >= m.n_layers) return fail(KS_EINVAL, "ks_mlp_get_params: layer %d out of range", l);
  const int out = m.dims[l + 1], in = m.dims[l];
  if (weight)
    hipLaunchKernelGGL(unpad_kernel, dim3((unsigned)(((int64_t)out * in + 255) / 256)), dim3(256), 0, (hipStream_t)stream, out, in,
                       m.kpad[l], gradients ? m.gW[l] : m.mW[l], weight);
  if (bias)
    hipLaunchKernelGGL(unpad_kernel, dim3((unsigned)((out + 255) / 256)), dim3(256), 0, (hipStream_t)stream, 1, out, out,
                       gradients ? m.gb[l] : m.mb[l], bias);
  return check_launch("ks_mlp_get_params");
}

// Every weight and bias of a network in one launch, entry 2 l / 2 l + 1 = weight / bias of layer l.
struct UnpadArgs {
  int n;
  int first_block[2 * KS_MAX_LAYERS + 1];
  int rows[2 * KS_MAX_LAYERS], cols[2 * KS_MAX_LAYERS], ld[2 * KS_MAX_LAYERS];
  const float* src[2 * KS_MAX_LAYERS];
  float* dst[2 * KS_MAX_LAYERS];
};
__global__ __launch_bounds__(256) void unpad_net_kernel(UnpadArgs a) {
  int e = 0;
  while (e + 1 < a.n && (int)blockIdx.x >= a.first_block[e + 1]) ++e;
  const int64_t total = (int64_t)a.rows[e] * a.cols[e];
  const int64_t idx = ((int64_t)blockIdx.x - a.first_block[e]) * 256 + threadIdx.x;
  if (idx >= total) return;
  const int r = (int)(idx / a.cols[e]), c = (int)(idx - (int64_t)r * a.cols[e]);
  a.dst[e][idx] = a.src[e][(int64_t)r * a.ld[e] + c];
}

extern "C" int64_t ks_mlp_param_floats(const KsMlp* h, int32_t layer) {
  if (!h || layer < 0 || layer > h->m.n_layers) return -1;
  int64_t off = 0;
  for (int l = 0; l < layer; ++l)
    off += ((int64_t)h->m.dims[l] * h->m.dims[l + 1] + 3) / 4 * 4 + ((int64_t)h->m.dims[l + 1] + 3) / 4 * 4;
  return off;
}

extern "C" int ks_mlps_copy_params_from(const KsMlp* const* nets, int32_t count, ks_stream_t stream, float* const* weights, float* const* biases,
                                        const int32_t* bias_first, int32_t gradients) {
  if (count < 0 || (count > 0 && (!nets || !weights || !biases))) return fail(KS_EINVAL, "ks_mlp_copy_params: null pointer");
  int at = 0;  // layer in the tables
  for (int k = 0; k < count; ++k) {
    if (!nets[k] || !nets[k]->m.train) return fail(KS_EINVAL, "ks_mlp_copy_params: call ks_mlp_train_init first");
    for (int l = 0; l < nets[k]->m.n_layers; ++l, ++at) {
      if (!weights[at] || !biases[at]) return fail(KS_EINVAL, "ks_mlp_copy_params: layer %d has no destination", l);
      if (bias_first && (bias_first[at] < 0 || bias_first[at] >= nets[k]->m.dims[l + 1]))
        return fail(KS_EINVAL, "ks_mlp_copy_params: layer %d has no bias %d", l, (int)bias_first[at]);
    }
  }
  at = 0;
  for (int k = 0; k < count;) {  // as many networks at a time as the table holds
    UnpadArgs a;
    a.n = 0;
    int blocks = 0;
    for (; k < count && a.n + 2 * nets[k]->m.n_layers <= 2 * KS_MAX_LAYERS; ++k) {
      const DevMlp& m = nets[k]->m;
      for (int l = 0; l < m.n_layers; ++l, ++at) {
        const int o = m.dims[l + 1], i = m.dims[l], w = a.n, b = a.n + 1;
        a.rows[w] = o; a.cols[w] = i; a.ld[w] = m.kpad[l]; a.src[w] = gradients ? m.gW[l] : m.mW[l]; a.dst[w] = weights[at];
        const int f = bias_first ? bias_first[at] : 0, nb = o - f;
        a.rows[b] = 1; a.cols[b] = nb; a.ld[b] = nb; a.src[b] = (gradients ? m.gb[l] : m.mb[l]) + f; a.dst[b] = biases[at];
        a.first_block[w] = blocks; blocks += (int)(((int64_t)o * i + 255) / 256);
        a.first_block[b] = blocks; blocks += (nb + 255) / 256;
        a.n += 2;
      }
    }
    a.first_block[a.n] = blocks;
    hipLaunchKernelGGL(unpad_net_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
  }
  return check_launch("ks_mlp_copy_params");
}

extern "C" int ks_mlps_copy_params(const KsMlp* const* nets, int32_t count, ks_stream_t stream, float* const* weights, float* const* biases,
                                   int32_t gradients) {
  return ks_mlps_copy_params_from(nets, count, stream, weights, biases, nullptr, gradients);
}

extern "C" int ks_mlp_copy_params(const KsMlp* h, ks_stream_t stream, float* const* weights, float* const* biases, int32_t gradients) {
  return ks_mlps_copy_params(&h, 1, stream, weights, biases, gradients);
}

// packed one after the other, each starting at a multiple of four floats
extern "C" int ks_mlp_get_all_params(const KsMlp* h, ks_stream_t stream, float* out, int32_t gradients) {
  if (!h || !h->m.train) return fail(KS_EINVAL, "ks_mlp_get_all_params: call ks_mlp_train_init first");
  if (!out) return fail(KS_EINVAL, "ks_mlp_get_all_params: null pointer");
  float *weights[KS_MAX_LAYERS], *biases[KS_MAX_LAYERS];
  for (int l = 0; l < h->m.n_layers; ++l) {
    weights[l] = out + ks_mlp_param_floats(h, l);
    biases[l] = weights[l] + ((int64_t)h->m.dims[l] * h->m.dims[l + 1] + 3) / 4 * 4;
  }
  return ks_mlp_copy_params(h, stream, weights, biases, gradients);
}
