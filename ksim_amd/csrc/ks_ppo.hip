// GAE / returns scan, advantage normalisation, PPO loss and reward/termination
// reduction for gfx950.  Streaming, HBM-bound kernels: every array is read or
// written exactly once per launch, with 64 consecutive elements per wavefront.
#include "ks_common.h"
#include <atomic>
#include <mutex>

namespace ks {

static thread_local char g_err[256] = "";
char* err_buf() { return g_err; }

// ---------------------------------------------------------------------------------------------
// Deterministic two-stage reductions (no atomics): stage 1 writes one partial per block,
// stage 2 re-reads the <= 1024 partials in a fixed order.
// ---------------------------------------------------------------------------------------------
constexpr int kMaxPartials = 1024;

__device__ inline double wave_sum(double x) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) x += __shfl_down(x, s);
  return x;
}

// Sum over a 256-thread block; result valid in thread 0.
__device__ inline double block_sum(double x, double* lds4) {
  x = wave_sum(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = x;
  __syncthreads();
  return lds4[0] + lds4[1] + lds4[2] + lds4[3];
}

// Sum and sum of squares over a block of WAVES wavefronts into partial[block] and partial[kMaxPartials + block].
template <int WAVES>
__device__ inline void block_moments(double s, double ss, double* __restrict__ partial) {
  __shared__ double lds[2][WAVES];
  s = wave_sum(s);
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) { lds[0][threadIdx.x >> 6] = s; lds[1][threadIdx.x >> 6] = ss; }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    for (int w = 0; w < WAVES; ++w) t += lds[threadIdx.x][w];
    partial[threadIdx.x * kMaxPartials + blockIdx.x] = t;
  }
}


// ---------------------------------------------------------------------------------------------
// GAE, (B, T) layout.  One wavefront per env row.  The recurrences R_t = r'_t + g m_t R_{t+1} and
// A_t = d_t + g l m_t A_{t+1} (ksim/task/ppo.py:66-75) are compositions of affine maps x -> d + c x, which are
// associative.  Lanes hold time in DESCENDING order (lane i of a 64-step chunk holds t = chunk_end - i), so the
// reverse scan over time is a forward scan over lanes: four DPP row_shr steps inside 16-lane rows, then
// row_bcast:15 and row_bcast:31 to chain the rows; no LDS traffic.  Chunks are chained from the end of the row
// through a wave-uniform carry read from lane 63.
// ---------------------------------------------------------------------------------------------
template <int kCtrl, int kRowMask>
__device__ __forceinline__ float dpp_take(float old, float x) {  // lanes without a valid source keep `old`
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, x),
                                                                kCtrl, kRowMask, 0xf, false));
}

// one scan step: (c, d) <- (c, d) o (c, d)[source lane]; identity where there is no source
template <int kCtrl, int kRowMask>
__device__ __forceinline__ void scan_step(float& c, float& d) {
  const float pc = dpp_take<kCtrl, kRowMask>(1.0f, c);
  const float pd = dpp_take<kCtrl, kRowMask>(0.0f, d);
  d = d + c * pd;
  c = c * pc;
}

// over groups of N lanes: the steps that would cross a group's boundary are left out
template <int N>
__device__ __forceinline__ void affine_scan(float& c, float& d) {
  scan_step<0x111, 0xf>(c, d);  // row_shr:1
  scan_step<0x112, 0xf>(c, d);  // row_shr:2
  scan_step<0x114, 0xf>(c, d);  // row_shr:4
  scan_step<0x118, 0xf>(c, d);  // row_shr:8
  if (N >= 32) scan_step<0x142, 0xa>(c, d);  // row_bcast:15 -> rows 1 and 3
  if (N >= 64) scan_step<0x143, 0xc>(c, d);  // row_bcast:31 -> rows 2 and 3
}

__device__ __forceinline__ float lane63(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

constexpr int kGaeMaxChunks = 4;  // rows of up to 256 steps keep every load in flight at once

// MOMENTS: the block also leaves the sum and the sum of squares of its advantages in `partial` (the first half of their
// normalisation, which would otherwise read them again in a launch of its own); then a block of 8 wavefronts walks several rows,
// so that at most kMaxPartials blocks cover the batch.
// LPR: lanes per row.  Rows of up to 32 (16) steps share a wavefront two (four) at a time: a trajectory of 24 or 32 steps would leave
// half of the lanes and of the loads in flight unused (16384 x 32 with moments: 13.0 -> 6.9 us).
template <bool MOMENTS, int LPR>
__global__ __launch_bounds__(MOMENTS ? 512 : 256) void gae_bt_kernel(
    int64_t B, int64_t T, const float* __restrict__ values, const float* __restrict__ rewards,
    const uint8_t* __restrict__ dones, const uint8_t* __restrict__ successes, float gamma, float lam,
    int mc, float* __restrict__ gae, float* __restrict__ returns, float* __restrict__ targets, double* __restrict__ partial) {
  constexpr int RPW = 64 / LPR, CH = LPR == 64 ? kGaeMaxChunks : 1;
  const int lane = threadIdx.x & (LPR - 1);
  double msum = 0.0, msq = 0.0;
  const int64_t rows_per_pass = (int64_t)(blockDim.x >> 6) * RPW;
  for (int64_t r0 = (int64_t)blockIdx.x * rows_per_pass + (threadIdx.x >> 6) * RPW; r0 < B; r0 += (int64_t)gridDim.x * rows_per_pass) {
    const int64_t row = r0 + (threadIdx.x & 63) / LPR;
    const bool row_ok = RPW == 1 || row < B;
    const int64_t base = (row_ok ? row : B - 1) * T;
    const float v_last = values[base + T - 1];  // bootstrap = last value repeated, ppo.py:79
    const float gl = gamma * lam;
    const float omg = 1.0f - gamma;
    float carry_r = 0.f, carry_a = 0.f, v_after = v_last;  // v_after: value at the first step after the chunk
    const int64_t nchunk = LPR == 64 ? (T + 63) >> 6 : 1;
    for (int64_t c0 = nchunk - 1; c0 >= 0; c0 -= CH) {
      // issue the loads of up to CH chunks before any of them is scanned
      float v[CH], r[CH];
      uint8_t dn[CH], sc[CH];
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        const int64_t c = c0 - k;
        const int64_t t = c * LPR + LPR - 1 - lane;  // descending time across lanes
        const bool valid = c >= 0 && t < T && row_ok;
        v[k] = valid ? values[base + t] : 0.f;
        r[k] = valid ? rewards[base + t] : 0.f;
        dn[k] = valid ? dones[base + t] : (uint8_t)0;
        sc[k] = (valid && successes) ? successes[base + t] : (uint8_t)0;
      }
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        const int64_t c = c0 - k;
        if (c < 0) break;
        const int64_t t = c * LPR + LPR - 1 - lane;
        const bool valid = t < T && row_ok;
        // V(s_{t+1}) sits one lane down; lane 0 takes the first value after the chunk (wave_shr:1 keeps `old` there), and a row's
        // last step, which is the first of its lanes in use, takes the bootstrap
        float v_up = dpp_take<0x138, 0xf>(v_after, v[k]);
        if (t + 1 >= T) v_up = v_last;
        const float mask = dn[k] ? 0.f : 1.f;
        const float rb = omg * r[k] + gamma * v[k] * (sc[k] ? 1.f : 0.f);  // ppo.py:82-83
        const float delta = rb + gamma * v_up * mask - v[k];                // ppo.py:86
        float c_r = valid ? gamma * mask : 1.f, d_r = valid ? rb : 0.f;
        float c_a = valid ? gl * mask : 1.f, d_a = valid ? delta : 0.f;
        affine_scan<LPR>(c_r, d_r);
        affine_scan<LPR>(c_a, d_a);
        const float R = d_r + c_r * carry_r;
        const float A = d_a + c_a * carry_a;
        if (valid) {
          if (gae) gae[base + t] = A;
          if (returns) returns[base + t] = R;
          if (targets) targets[base + t] = mc ? R : A + v[k];  // ppo.py:107
          if (MOMENTS) { msum += (double)A; msq += (double)A * (double)A; }
        }
        if (LPR == 64) {
          carry_r = lane63(R);
          carry_a = lane63(A);
          v_after = lane63(v[k]);
        }
      }
    }
  }
  if constexpr (MOMENTS) block_moments<8>(msum, msq, partial);
}

// GAE, (T, N) layout.  A workgroup owns 32 consecutive envs and walks back in time in chunks of 32 steps: all 256
// threads load the chunk's (32 steps x 32 envs) tiles into LDS (128-byte rows, every load independent of the
// recurrence), the first 32 threads run the recurrence out of LDS, one env each, and all threads write the results
// back.  With one lane per env doing its own loads, 8192 envs would be 128 wavefronts with one dependent stream of
// loads each; here every CU has eight times as many loads in flight and N / 32 workgroups spread over the chip.
constexpr int kTnEnvs = 32, kTnSteps = 32;
template <bool MOMENTS>  // as in gae_bt_kernel
__global__ __launch_bounds__(256) void gae_tn_kernel(
    int64_t T, int64_t N, const float* __restrict__ values, const float* __restrict__ rewards,
    const uint8_t* __restrict__ dones, const uint8_t* __restrict__ successes, float gamma, float lam,
    int mc, float* __restrict__ gae, float* __restrict__ returns, float* __restrict__ targets, int64_t tiles, double* __restrict__ partial) {
  __shared__ float sv[kTnSteps][kTnEnvs], sr[kTnSteps][kTnEnvs], oa[kTnSteps][kTnEnvs], orr[kTnSteps][kTnEnvs];
  __shared__ uint8_t sd[kTnSteps][kTnEnvs], ss[kTnSteps][kTnEnvs];
  const int tx = threadIdx.x & (kTnEnvs - 1), ty = threadIdx.x / kTnEnvs;
  // Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Four neighbouring tiles share every 128-byte
  // line of the byte arrays, so neighbouring tiles go to one XCD: workgroup b takes tile (b % 8) * (grid / 8) + b / 8.
  double msum = 0.0, msq = 0.0;
  for (int64_t b = blockIdx.x; b < tiles; b += gridDim.x) {
  int64_t tile = b;
  if (tiles % 8 == 0) tile = (b % 8) * (tiles / 8) + b / 8;
  const int64_t e = tile * kTnEnvs + tx;
  const bool in = e < N;
  const float gl = gamma * lam, omg = 1.0f - gamma;
  float R = 0.f, A = 0.f, v_up = 0.f;
  for (int64_t t1 = T; t1 > 0; t1 -= kTnSteps) {
    const int64_t t0 = t1 > kTnSteps ? t1 - kTnSteps : 0;
    const int n = (int)(t1 - t0);
    for (int k = ty; k < n; k += 256 / kTnEnvs) {
      const int64_t i = (t0 + k) * N + e;
      sv[k][tx] = in ? values[i] : 0.f;
      sr[k][tx] = in ? rewards[i] : 0.f;
      sd[k][tx] = in ? dones[i] : (uint8_t)0;
      ss[k][tx] = (in && successes) ? successes[i] : (uint8_t)0;
    }
    __syncthreads();
    if (threadIdx.x < kTnEnvs) {
      if (t1 == T) v_up = sv[n - 1][tx];
      for (int k = n - 1; k >= 0; --k) {
        const float v = sv[k][tx], r = sr[k][tx];
        const float mask = sd[k][tx] ? 0.f : 1.f;
        const float sc = ss[k][tx] ? 1.f : 0.f;
        const float rb = omg * r + gamma * v * sc;
        const float delta = rb + gamma * v_up * mask - v;
        R = rb + gamma * mask * R;
        A = delta + gl * mask * A;
        oa[k][tx] = A;
        orr[k][tx] = R;
        v_up = v;
      }
    }
    __syncthreads();
    if (in)
      for (int k = ty; k < n; k += 256 / kTnEnvs) {
        const int64_t i = (t0 + k) * N + e;
        const float a = oa[k][tx], rr = orr[k][tx];
        if (gae) gae[i] = a;
        if (returns) returns[i] = rr;
        if (targets) targets[i] = mc ? rr : a + sv[k][tx];
        if (MOMENTS) { msum += (double)a; msq += (double)a * (double)a; }
      }
    __syncthreads();
  }
  }
  if constexpr (MOMENTS) block_moments<4>(msum, msq, partial);
}

__global__ __launch_bounds__(256) void moments_kernel(int64_t n, const float* __restrict__ x,
                                                       double* __restrict__ partial) {
  __shared__ double lds[4];
  double s = 0.0, ss = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double v = x[i];
    s += v;
    ss += v * v;
  }
  s = block_sum(s, lds);
  ss = block_sum(ss, lds);
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = s;
    partial[kMaxPartials + blockIdx.x] = ss;
  }
}

__global__ __launch_bounds__(256) void normalize_kernel(int64_t n, int nparts, const float* __restrict__ x,
                                                         const double* __restrict__ partial,
                                                         float* __restrict__ out) {
  __shared__ double lds[4];
  __shared__ float s_mean, s_inv;
  double s = 0.0, ss = 0.0;
  for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
    s += partial[i];
    ss += partial[kMaxPartials + i];
  }
  s = block_sum(s, lds);
  ss = block_sum(ss, lds);
  if (threadIdx.x == 0) {
    const double mean = s / (double)n;
    double var = ss / (double)n - mean * mean;
    if (var < 0.0) var = 0.0;
    double sd = sqrt(var);
    if (sd < 1e-6) sd = 1e-6;  // ppo.py:118
    s_mean = (float)mean;
    s_inv = (float)(1.0 / sd);
  }
  __syncthreads();
  const float mean = s_mean, inv = s_inv;
  const int64_t n4 = (((uintptr_t)x | (uintptr_t)out) & 15) == 0 ? n / 4 : 0;  // whole 16-byte groups; the rest one by one
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = i0; i < n4; i += step) {
    float4 v = reinterpret_cast<const float4*>(x)[i];
    v.x = (v.x - mean) * inv; v.y = (v.y - mean) * inv; v.z = (v.z - mean) * inv; v.w = (v.w - mean) * inv;
    reinterpret_cast<float4*>(out)[i] = v;
  }
  for (int64_t i = 4 * n4 + i0; i < n; i += step) out[i] = (x[i] - mean) * inv;
}

// the adaptive-KL factor: a device scalar when the caller keeps it there, otherwise the host's number
__device__ __forceinline__ float kl_scale_of(const KsPpoLossParams& p) { return p.kl_scale_device ? *p.kl_scale_device : p.kl_scale; }

// ---------------------------------------------------------------------------------------------
// A sum over the whole grid in the launch that makes its parts: every block leaves its part beside a check word, and the last block waits for them and adds
// them up in order.  A part is whole when part ^ check is this launch's tag, so the two stores need no order, whatever the workspace held before
// (tags are 64 bits and no two launches' are alike; a graph's replays share theirs, hence the zeros that the last block leaves).  Nothing waits for the
// last block, so the others always come to their end; it gives up with a NaN after twenty seconds, for a workspace that two calls write at once.
// The loss, its sum in a launch of its own -> here: 250 x 24 elements of 17 actions with their advantages 37.8 -> 34.9 us a call (the host's time for the
// launch), 16384 x 32 of 20 actions 48.1 -> 46.5 (3.9 us and a gap, of which the wait for the last parts stays).
// ---------------------------------------------------------------------------------------------
struct GridSum {
  unsigned long long* slots;  // gridDim.x parts, then as many check words from kMaxPartials on
  unsigned long long tag;
};
static GridSum grid_sum(void* workspace) {
  static std::atomic<unsigned long long> launches{0};
  unsigned long long x = (launches.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9e3779b97f4a7c15ull;  // splitmix64 (Steele, Lea and Flood, 2014)
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return {(unsigned long long*)workspace, x ^ (x >> 31)};
}
__device__ __forceinline__ void store_shared(unsigned long long* p, unsigned long long v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned long long load_shared(const unsigned long long* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// `part`: the block's sum in thread 0 of 256.  Whether this is the last block, in whose thread 0 `total` is the whole sum afterwards.
__device__ __forceinline__ bool grid_total(const GridSum& g, double part, double* lds4, double& total) {
  if (threadIdx.x == 0) {
    const unsigned long long bits = __builtin_bit_cast(unsigned long long, part);
    store_shared(g.slots + blockIdx.x, bits);
    store_shared(g.slots + kMaxPartials + blockIdx.x, bits ^ g.tag);
  }
  if (blockIdx.x != gridDim.x - 1) return false;
  constexpr unsigned long long kPatience = 2000000000ull;  // of the 100 MHz counter
  const unsigned long long start = wall_clock64();
  double s = 0.0;
#pragma unroll 1
  for (unsigned i = threadIdx.x; i < gridDim.x; i += blockDim.x) {
    unsigned long long bits, check;
#pragma unroll 1
    for (;;) {
      bits = load_shared(g.slots + i);
      check = load_shared(g.slots + kMaxPartials + i);
      if ((bits ^ check) == g.tag) break;
      if (wall_clock64() - start > kPatience) {
        bits = 0x7ff8000000000000ull;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    store_shared(g.slots + i, 0);
    store_shared(g.slots + kMaxPartials + i, 0);
    s += __builtin_bit_cast(double, bits);
  }
  total = block_sum(s, lds4);
  return true;
}

// ---------------------------------------------------------------------------------------------
// PPO loss (ppo.py:207-246), one lane per (b, t) element.
// ---------------------------------------------------------------------------------------------
struct PpoLossIO {
  const float *adv, *tgt, *lp_on, *v_on, *lp_off, *v_off, *ent;
  float *policy, *value, *kl, *entropy;
};

// The four terms of element i from its log ratio and entropy sum; returns their sum.
__device__ __forceinline__ float ppo_loss_terms(const PpoLossIO& io, const KsPpoLossParams& p, float kl_scale, int64_t i, float log_ratio,
                                                float es) {
  const float lr = fminf(fmaxf(log_ratio, -p.log_clip_value), p.log_clip_value);
  const float ratio = expf(lr);
  const float cr = fminf(fmaxf(ratio, 1.f - p.clip_param), 1.f + p.clip_param);
  const float ad = io.adv[i];
  const float policy = -fminf(ratio * ad, cr * ad);
  const float von = io.v_on[i], voff = io.v_off[i], tg = io.tgt[i];
  float vobj;
  if (p.use_clipped_value_loss) {
    const float vc = von + fminf(fmaxf(voff - von, -p.clip_param), p.clip_param);
    const float ce = vc - tg, er = voff - tg;
    vobj = 0.5f * fmaxf(er * er, ce * ce);
  } else {
    const float er = tg - voff;
    vobj = 0.5f * er * er;
  }
  const float value = vobj * p.value_loss_coef;
  const float klv = -log_ratio * p.kl_coef * kl_scale;  // the sum of on - off is the log ratio negated, to the bit
  const float entv = io.ent ? -es * p.entropy_coef : 0.f;
  if (io.policy) io.policy[i] = policy;
  if (io.value) io.value[i] = value;
  if (io.kl) io.kl[i] = klv;
  if (io.entropy && io.ent) io.entropy[i] = entv;
  return policy + value + klv + entv;
}

// Elements whose A actions a lane can read where they lie: A = 1, and the widths whose rows are too long to stage.
__global__ __launch_bounds__(256) void ppo_loss_kernel(int64_t n, int A, KsPpoLossParams p, PpoLossIO io, GridSum sum, float* __restrict__ mean) {
  __shared__ double lds[4];
  double acc = 0.0;
  const float kl_scale = kl_scale_of(p);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    float log_ratio = 0.f, es = 0.f;
    const float* a_on = io.lp_on + i * A;
    const float* a_off = io.lp_off + i * A;
    for (int a = 0; a < A; ++a) log_ratio += a_off[a] - a_on[a];
    if (io.ent) {
      const float* e = io.ent + i * A;
      for (int a = 0; a < A; ++a) es += e[a];
    }
    acc += (double)ppo_loss_terms(io, p, kl_scale, i, log_ratio, es);
  }
  if (!mean) return;
  acc = block_sum(acc, lds);
  double total;
  if (grid_total(sum, acc, lds, total) && threadIdx.x == 0) mean[0] = (float)(total / (double)n);
}

// The A log-probabilities of an element are contiguous: lanes that walk an element each touch 64 lines per load and miss the
// vector L1 on most of them (16384 x 32 elements, A = 20: 137 us, 1.0 TB/s).  Here a wavefront copies the contiguous 64 A floats of
// its 64 elements with one 16-byte load per lane and array at a time, all of them in flight, leaves off - on and the entropies in
// LDS with an odd row stride, and sums every element's row in order from there: bound by the bytes (31 us at that size).
constexpr int kLossMaxA = 31;  // four wavefronts' tiles within 64 KB of LDS

__global__ __launch_bounds__(256) void ppo_loss_rows_kernel(int64_t n, int A, int wave_floats, KsPpoLossParams p, PpoLossIO io, GridSum sum,
                                                            float* __restrict__ mean) {
  extern __shared__ float loss_lds[];
  __shared__ double lds[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int LD = A | 1;
  float* sd = loss_lds + wave * wave_floats;
  float* se = sd + 64 * LD;
  const float kl_scale = kl_scale_of(p);
  const unsigned inv_a = 0xffffffffu / (unsigned)A + 1u;  // x / A = mulhi(x, inv_a) for x < 64 * 32 < 2^16
  double acc = 0.0;
  const int64_t tiles = (n + 63) / 64;
  for (int64_t tile = (int64_t)blockIdx.x * 4 + wave; tile < tiles; tile += (int64_t)gridDim.x * 4) {
    const int64_t i0 = tile * 64;
    const int rows = (int)(n - i0 < 64 ? n - i0 : 64);
    const int cnt = rows * A;  // i0 * A is a multiple of 64: the span starts on a 16-byte boundary of its array
    const float* on = io.lp_on + i0 * A;
    const float* off = io.lp_off + i0 * A;
    const float* en = io.ent ? io.ent + i0 * A : nullptr;
    auto put = [&](float* dst, int x, float v) {
      const int r = (int)__umulhi((unsigned)x, inv_a);
      dst[r * LD + (x - r * A)] = v;
    };
    if (rows == 64) {
#pragma unroll 2
      for (int x = 4 * lane; x < cnt; x += 256) {
        const float4 f = *reinterpret_cast<const float4*>(off + x), g = *reinterpret_cast<const float4*>(on + x);
        float4 h = {0.f, 0.f, 0.f, 0.f};
        if (en) h = *reinterpret_cast<const float4*>(en + x);
        put(sd, x, f.x - g.x); put(sd, x + 1, f.y - g.y); put(sd, x + 2, f.z - g.z); put(sd, x + 3, f.w - g.w);
        if (en) { put(se, x, h.x); put(se, x + 1, h.y); put(se, x + 2, h.z); put(se, x + 3, h.w); }
      }
    } else {
      for (int x = lane; x < cnt; x += 64) {
        put(sd, x, off[x] - on[x]);
        if (en) put(se, x, en[x]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wavefront's own LDS tile: no other wavefront touches it
    __builtin_amdgcn_wave_barrier();
    if (lane < rows) {
      float log_ratio = 0.f, es = 0.f;
      for (int a = 0; a < A; ++a) log_ratio += sd[lane * LD + a];
      if (en) for (int a = 0; a < A; ++a) es += se[lane * LD + a];
      acc += (double)ppo_loss_terms(io, p, kl_scale, i0 + lane, log_ratio, es);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (!mean) return;
  acc = block_sum(acc, lds);
  double total;
  if (grid_total(sum, acc, lds, total) && threadIdx.x == 0) mean[0] = (float)(total / (double)n);
}

// ---------------------------------------------------------------------------------------------
// Reward total (rl.py:219-239) and done/success (rl.py:1049-1050).
// ---------------------------------------------------------------------------------------------
struct RewardScales {
  float s[KS_MAX_REWARD_TERMS];
};

__global__ __launch_bounds__(256) void reward_total_kernel(
    int64_t n, int K, const float* __restrict__ comps, RewardScales sc, int use_min, float cmin, int use_max,
    float cmax, float* __restrict__ total, int k, const int8_t* __restrict__ terms, uint8_t* __restrict__ done,
    uint8_t* __restrict__ success) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (total) {
    float t = 0.f;
    for (int j = 0; j < K; ++j) {
      const float term = comps[(int64_t)j * n + i] * sc.s[j];
      t = (j == 0) ? term : t + term;  // insertion-order sum, rl.py:235
    }
    if (use_min) t = fmaxf(t, cmin);
    if (use_max) t = fminf(t, cmax);
    total[i] = t;
  }
  if (k > 0) {
    bool d = false, s = true;
    for (int j = 0; j < k; ++j) {
      const int8_t t = terms[(int64_t)j * n + i];
      d |= t != 0;
      s &= t != -1;
    }
    if (done) done[i] = d ? 1 : 0;
    if (success) success[i] = (s && d) ? 1 : 0;
  }
}

__global__ __launch_bounds__(256) void copy_f32_kernel(int64_t n, const float* __restrict__ src, float* __restrict__ dst) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) dst[i] = src[i];
}

static inline int grid_for(int64_t n, int block, int cap) {
  int64_t g = (n + block - 1) / block;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return (int)g;
}

// ---------------------------------------------------------------- a minibatch's columns of every array of a trajectory
// dst[o][j] = src[o][index[j]] for pieces of `inner` bytes, several arrays per launch: the env columns of a minibatch.  An array goes in words
// as wide as its pieces and pointers allow, four words in flight per thread.  Bound by memory for
// the observations and by the launch for the small arrays: the thirteen arrays of a K-Bot minibatch (512 of 1024 envs x 100 steps, 230 MB both
// ways) 130 us in thirteen launches -> 75, the eight of 2048 envs x 32 steps with 68 observations 55 -> 28.
struct GatherArray {
  const char* src;
  char* dst;
  uint32_t words, inner;  // words in all, words per piece
  uint32_t log_bytes;     // of a word: 0 .. 4
  uint32_t first_block;
};
struct GatherTable {
  GatherArray a[KS_GATHER_ARRAYS];
  int n;
};
constexpr int kGatherWords = 1024;  // per workgroup

template <typename T>
__device__ __forceinline__ void gather_words(const GatherArray& a, int64_t columns, uint32_t picked, const int64_t* __restrict__ index) {
  const T* src = reinterpret_cast<const T*>(a.src);
  T* dst = reinterpret_cast<T*>(a.dst);
  const uint32_t base = (blockIdx.x - a.first_block) * kGatherWords + threadIdx.x;
  T v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t w = min(base + 256 * k, a.words - 1), piece = w / a.inner, c = w - piece * a.inner, o = piece / picked;
    const int64_t at = index[piece - o * picked];
    v[k] = src[((int64_t)o * columns + min(max(at, (int64_t)0), columns - 1)) * a.inner + c];  // an index outside the array stays inside it
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (base + 256 * k < a.words) dst[base + 256 * k] = v[k];
}

__global__ __launch_bounds__(256) void gather_columns_kernel(GatherTable t, int64_t columns, uint32_t picked, const int64_t* __restrict__ index) {
  int e = 0;
  while (e + 1 < t.n && blockIdx.x >= t.a[e + 1].first_block) ++e;
  const GatherArray& a = t.a[e];
  switch (a.log_bytes) {
    case 4: gather_words<uint4>(a, columns, picked, index); break;
    case 3: gather_words<uint2>(a, columns, picked, index); break;
    case 2: gather_words<uint32_t>(a, columns, picked, index); break;
    case 1: gather_words<uint16_t>(a, columns, picked, index); break;
    default: gather_words<uint8_t>(a, columns, picked, index);
  }
}

// ---------------------------------------------------------------- the two batches of a discriminator step
// A window of frames from each drawn clip, wrapping round at its end, and the frames of each drawn env, both batches in one launch.  What was drawn
// comes with the launch's arguments, so nothing is uploaded first: two uploads and two gathers were four launches of a few microseconds, for which
// the host needed 45 of a step's 140 us (32 + 32 sequences of 32 frames of 71).
struct WindowTable {
  int32_t clip[KS_WINDOWS], start[KS_WINDOWS], env[KS_WINDOWS];
};

// blockIdx.x: a sequence of the real batch, then of the simulated one; a sequence is one run of `floats` floats that starts anywhere in its clip
__global__ __launch_bounds__(256) void gather_windows_kernel(const WindowTable t, int batch, uint32_t floats, uint32_t row, uint32_t clip_floats,
                                                             const float* __restrict__ motions, const float* __restrict__ sim,
                                                             float* __restrict__ real_out, float* __restrict__ sim_out) {
  const bool real = (int)blockIdx.x < batch;
  const int k = real ? (int)blockIdx.x : (int)blockIdx.x - batch;
  const float* src = real ? motions + (int64_t)t.clip[k] * clip_floats : sim + (int64_t)t.env[k] * floats;
  const uint32_t first = real ? (uint32_t)t.start[k] * row : 0u, wrap = real ? clip_floats : floats;
  float* dst = (real ? real_out : sim_out) + (int64_t)k * floats;
  const uint32_t base = blockIdx.y * 2048u + threadIdx.x;
  float v[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const uint32_t e = min(base + 256u * u, floats - 1) + first;
    v[u] = src[e < wrap ? e : e % wrap];
  }
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (base + 256u * u < floats) dst[base + 256u * u] = v[u];
}

}  // namespace ks

using namespace ks;

extern "C" int ks_gather_windows(ks_stream_t stream, int32_t batch, int64_t window_t, int64_t frame, int64_t clips, int64_t clip_t, int64_t envs,
                                 const float* motions, const float* sim, const int64_t* clip, const int64_t* start, const int64_t* env,
                                 float* real_out, float* sim_out) {
  if (batch < 1 || batch > KS_WINDOWS) return fail(KS_ELIMIT, "ks_gather_windows: %d sequences, of 1 to %d", batch, KS_WINDOWS);
  if (window_t < 1 || frame < 1 || clips < 1 || clip_t < 1 || envs < 1) return fail(KS_EINVAL, "ks_gather_windows: bad size");
  if (!motions || !sim || !clip || !start || !env || !real_out || !sim_out) return fail(KS_EINVAL, "ks_gather_windows: null pointer");
  // 32-bit positions inside a sequence: the last one lies below clip_t + window_t frames
  if (clip_t > 0x7fffffff || window_t > 0x7fffffff || frame > 0x7fffffff || (clip_t + window_t) * frame > 0x7fffffff - 2048)
    return fail(KS_ELIMIT, "ks_gather_windows: clips or windows too long");
  const int64_t floats = window_t * frame;
  if (floats > KS_WINDOW_FLOATS) return fail(KS_ELIMIT, "ks_gather_windows: windows too long");  // a block per 2048 floats on the grid's y axis
  WindowTable t;
  for (int k = 0; k < batch; ++k) {
    if (clip[k] < 0 || clip[k] >= clips || start[k] < 0 || start[k] >= clip_t || env[k] < 0 || env[k] >= envs || clips > 0x7fffffff || envs > 0x7fffffff)
      return fail(KS_EINVAL, "ks_gather_windows: sequence %d lies outside its array", k);
    t.clip[k] = (int32_t)clip[k];
    t.start[k] = (int32_t)start[k];
    t.env[k] = (int32_t)env[k];
  }
  hipLaunchKernelGGL(gather_windows_kernel, dim3(2u * (unsigned)batch, (unsigned)((floats + 2047) / 2048)), dim3(256), 0, (hipStream_t)stream, t, batch,
                     (uint32_t)floats, (uint32_t)frame, (uint32_t)(clip_t * frame), motions, sim, real_out, sim_out);
  return check_launch("ks_gather_windows");
}

extern "C" const char* ks_version(void) { return "ksim_hip 0.1 (gfx950)"; }
extern "C" const char* ks_last_error(void) { return ks::err_buf(); }
extern "C" int64_t ks_abi_sizeof(int32_t which) {
  switch (which) {
    case 0: return sizeof(KsPpoLossParams);
    case 1: return sizeof(KsModelDesc);
    case 2: return sizeof(KsStepIO);
    case 3: return sizeof(KsTermsDesc);
    case 4: return sizeof(KsObserveIO);
    case 5: return sizeof(KsTerminateIO);
    case 6: return sizeof(KsMlpDesc);
    case 7: return sizeof(KsRewardIO);
    case 8: return sizeof(KsObsElem);
    case 9: return sizeof(KsTermDesc);
    case 10: return sizeof(KsRewardDesc);
    case 11: return sizeof(KsRng);
    case 12: return sizeof(KsAdamParams);
    case 13: return sizeof(KsEventDesc);
    case 14: return sizeof(KsRewardScanIO);
    case 15: return sizeof(KsRewardScanDesc);
    case 16: return sizeof(KsGruDesc);
    case 17: return sizeof(KsLstmDesc);
    case 18: return sizeof(KsGaussianHead);
    case 19: return sizeof(KsCommandIO);
    case 20: return sizeof(KsMixtureHead);
    case 21: return sizeof(KsNoiseStage);
    case 22: return sizeof(KsRandomVar);
    case 23: return sizeof(KsActionSample);
    case 24: return sizeof(KsLayerBackward);
    case 25: return sizeof(KsGatherArray);
    case 26: return sizeof(KsSequence);
    default: return -1;
  }
}

static int check_gae_args(int64_t n0, int64_t n1, const float* v, const float* r, const uint8_t* d) {
  if (n0 < 0 || n1 < 0) return fail(KS_EINVAL, "ks_gae: negative size");
  if (n0 > 0 && n1 > 0 && (!v || !r || !d)) return fail(KS_EINVAL, "ks_gae: null input");
  if (n0 > (int64_t)1 << 40 || n1 > (int64_t)1 << 40) return fail(KS_ELIMIT, "ks_gae: size too large");
  return KS_OK;
}

extern "C" int ks_gae_bt(ks_stream_t stream, int64_t B, int64_t T, const float* values, const float* rewards,
                         const uint8_t* dones, const uint8_t* successes, float gamma, float lam,
                         int monte_carlo_returns, float* gae, float* returns, float* targets) {
  if (int rc = check_gae_args(B, T, values, rewards, dones)) return rc;
  if (B == 0 || T == 0) return KS_OK;
  const int rows_per_block = 4 * (T <= 16 ? 4 : (T <= 32 ? 2 : 1));
  const int64_t grid = (B + rows_per_block - 1) / rows_per_block;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_gae_bt: B too large");
  auto kfn = T <= 16 ? gae_bt_kernel<false, 16> : (T <= 32 ? gae_bt_kernel<false, 32> : gae_bt_kernel<false, 64>);
  hipLaunchKernelGGL(kfn, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, B, T, values, rewards,
                     dones, successes, gamma, lam, monte_carlo_returns, gae, returns, targets, nullptr);
  return check_launch("ks_gae_bt");
}

extern "C" int ks_gae_tn(ks_stream_t stream, int64_t T, int64_t N, const float* values, const float* rewards,
                         const uint8_t* dones, const uint8_t* successes, float gamma, float lam,
                         int monte_carlo_returns, float* gae, float* returns, float* targets) {
  if (int rc = check_gae_args(T, N, values, rewards, dones)) return rc;
  if (N == 0 || T == 0) return KS_OK;
  const int64_t grid = (N + kTnEnvs - 1) / kTnEnvs;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_gae_tn: N too large");
  hipLaunchKernelGGL(gae_tn_kernel<false>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, T, N, values, rewards,
                     dones, successes, gamma, lam, monte_carlo_returns, gae, returns, targets, grid, nullptr);
  return check_launch("ks_gae_tn");
}

extern "C" int ks_gae_normalized(ks_stream_t stream, int time_major, int64_t n0, int64_t n1, const float* values, const float* rewards,
                                 const uint8_t* dones, const uint8_t* successes, float gamma, float lam, int monte_carlo_returns,
                                 float* gae, float* returns, float* targets, float* advantages, void* workspace) {
  if (int rc = check_gae_args(n0, n1, values, rewards, dones)) return rc;
  if (n0 == 0 || n1 == 0) return KS_OK;
  if (!gae || !advantages || !workspace) return fail(KS_EINVAL, "ks_gae_normalized: null pointer");
  const int64_t n = n0 * n1;
  double* partial = (double*)workspace;
  int g;
  if (time_major) {
    const int64_t tiles = (n1 + kTnEnvs - 1) / kTnEnvs;
    g = (int)(tiles < kMaxPartials ? tiles : kMaxPartials);
    hipLaunchKernelGGL(gae_tn_kernel<true>, dim3(g), dim3(256), 0, (hipStream_t)stream, n0, n1, values, rewards, dones, successes, gamma, lam,
                       monte_carlo_returns, gae, returns, targets, tiles, partial);
  } else {
    g = grid_for(n0, 8 * (n1 <= 16 ? 4 : (n1 <= 32 ? 2 : 1)), kMaxPartials);
    auto kfn = n1 <= 16 ? gae_bt_kernel<true, 16> : (n1 <= 32 ? gae_bt_kernel<true, 32> : gae_bt_kernel<true, 64>);
    hipLaunchKernelGGL(kfn, dim3(g), dim3(512), 0, (hipStream_t)stream, n0, n1, values, rewards, dones, successes, gamma, lam,
                       monte_carlo_returns, gae, returns, targets, partial);
  }
  hipLaunchKernelGGL(normalize_kernel, dim3(grid_for(n, 1024, 1024)), dim3(256), 0, (hipStream_t)stream, n, g, gae, partial, advantages);
  return check_launch("ks_gae_normalized");
}

extern "C" int ks_normalize_advantages(ks_stream_t stream, int64_t n, const float* gae, float* advantages,
                                       void* workspace) {
  if (n < 0) return fail(KS_EINVAL, "ks_normalize_advantages: negative size");
  if (n == 0) return KS_OK;
  if (!gae || !advantages || !workspace) return fail(KS_EINVAL, "ks_normalize_advantages: null pointer");
  const int g = grid_for(n, 256 * 4, kMaxPartials);
  double* partial = (double*)workspace;
  hipLaunchKernelGGL(moments_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, n, gae, partial);
  hipLaunchKernelGGL(normalize_kernel, dim3(grid_for(n, 1024, 1024)), dim3(256), 0, (hipStream_t)stream, n, g, gae,
                     partial, advantages);
  return check_launch("ks_normalize_advantages");
}

// ---------------------------------------------------------------------------------------------
// ks_normalize_advantages without a workspace argument: the block partials live in a file-scope device array.
// The array's name is only a host-side handle; its device address is looked up once per device with
// hipGetSymbolAddress (each GPU holds its own copy) and that pointer is what the kernels receive.
// ---------------------------------------------------------------------------------------------
namespace ks {
static __device__ __align__(256) unsigned char scratch[KS_REDUCE_WORKSPACE_BYTES];
constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices] = {};
static std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device.
static int scratch_on_current_device(const char* who, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(KS_ELAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(KS_ELIMIT, "%s: device %d beyond the %d this library keeps scratch for", who, dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(KS_ELAUNCH, "%s: hipGetSymbolAddress: %s", who, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return KS_OK;
}
}  // namespace ks

extern "C" int ks_normalize_advantages_static(ks_stream_t stream, int64_t n, const float* gae, float* advantages) {
  if (n < 0) return fail(KS_EINVAL, "ks_normalize_advantages_static: negative size");
  if (n > KS_NORMALIZE_STATIC_MAX_N)
    return fail(KS_ELIMIT, "ks_normalize_advantages_static: n = %lld beyond the maximum of %lld elements", (long long)n,
                (long long)KS_NORMALIZE_STATIC_MAX_N);
  if (n == 0) return KS_OK;
  if (!gae || !advantages) return fail(KS_EINVAL, "ks_normalize_advantages_static: null pointer");
  void* ptr = nullptr;
  if (int rc = scratch_on_current_device("ks_normalize_advantages_static", &ptr)) return rc;
  double* partial = (double*)ptr;
  // every partial that stage 2 reads is written by stage 1 of the same call, so nothing has to be cleared
  const int g = grid_for(n, 256 * 4, kMaxPartials);
  hipLaunchKernelGGL(moments_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, n, gae, partial);
  hipLaunchKernelGGL(normalize_kernel, dim3(grid_for(n, 1024, 1024)), dim3(256), 0, (hipStream_t)stream, n, g, gae,
                     partial, advantages);
  return check_launch("ks_normalize_advantages_static");
}

extern "C" int ks_ppo_loss(ks_stream_t stream, int64_t n, int32_t A, const KsPpoLossParams* params,
                           const float* advantages, const float* value_targets, const float* on_log_probs,
                           const float* on_values, const float* off_log_probs, const float* off_values,
                           const float* off_entropy, float* policy_loss, float* value_loss, float* kl_loss,
                           float* entropy_loss, float* loss_out, void* workspace) {
  if (n < 0 || A < 1) return fail(KS_EINVAL, "ks_ppo_loss: bad size n=%lld A=%d", (long long)n, A);
  if (!params) return fail(KS_EINVAL, "ks_ppo_loss: null params");
  if (n == 0) return KS_OK;
  if (!advantages || !value_targets || !on_log_probs || !on_values || !off_log_probs || !off_values || !workspace)
    return fail(KS_EINVAL, "ks_ppo_loss: null pointer");
  const int g = grid_for(n, 256, kMaxPartials);
  const GridSum sum = grid_sum(workspace);
  const PpoLossIO io = {advantages, value_targets, on_log_probs, on_values, off_log_probs, off_values, off_entropy,
                        policy_loss, value_loss, kl_loss, entropy_loss};
  const bool aligned = (((uintptr_t)on_log_probs | (uintptr_t)off_log_probs | (uintptr_t)off_entropy) & 15) == 0;
  if (A > 1 && A <= kLossMaxA && aligned) {
    const int wave_floats = 64 * (A | 1) * (off_entropy ? 2 : 1);
    hipLaunchKernelGGL(ppo_loss_rows_kernel, dim3(g), dim3(256), 4 * wave_floats * (int)sizeof(float), (hipStream_t)stream, n, (int)A, wave_floats,
                       *params, io, sum, loss_out);
  } else {
    hipLaunchKernelGGL(ppo_loss_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, n, (int)A, *params, io, sum, loss_out);
  }
  return check_launch("ks_ppo_loss");
}

extern "C" int ks_reward_total(ks_stream_t stream, int64_t n, int32_t K, const float* components,
                               const float* scales, int32_t use_clip_min, float clip_min, int32_t use_clip_max,
                               float clip_max, float* total, int32_t k, const int8_t* terminations, uint8_t* done,
                               uint8_t* success) {
  if (n < 0 || K < 0 || k < 0) return fail(KS_EINVAL, "ks_reward_total: negative size");
  if (K > KS_MAX_REWARD_TERMS || k > KS_MAX_REWARD_TERMS)
    return fail(KS_ELIMIT, "ks_reward_total: more than %d terms", KS_MAX_REWARD_TERMS);
  if (n == 0) return KS_OK;
  if (total && (K == 0 || !components || !scales)) return fail(KS_EINVAL, "ks_reward_total: total needs K>0 components");
  if (k > 0 && !terminations) return fail(KS_EINVAL, "ks_reward_total: null terminations");
  RewardScales sc{};
  for (int j = 0; j < K && scales; ++j) sc.s[j] = scales[j];
  const int64_t grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_reward_total: n too large");
  hipLaunchKernelGGL(reward_total_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, n, (int)K,
                     components, sc, use_clip_min, clip_min, use_clip_max, clip_max, total, (int)k, terminations, done,
                     success);
  return check_launch("ks_reward_total");
}

extern "C" int ks_copy_f32(ks_stream_t stream, int64_t n, const float* src, float* dst) {
  if (n < 0) return fail(KS_EINVAL, "ks_copy_f32: negative size");
  if (n == 0) return KS_OK;
  if (!src || !dst) return fail(KS_EINVAL, "ks_copy_f32: null pointer");
  hipLaunchKernelGGL(copy_f32_kernel, dim3(grid_for(n, 256, 65536)), dim3(256), 0, (hipStream_t)stream, n, src, dst);
  return check_launch("ks_copy_f32");
}

// ---------------------------------------------------------------------------------------------
// Gaussian policy head and the gradient of the PPO objective
// ---------------------------------------------------------------------------------------------
namespace ks {

constexpr float kHalfLog2Pi = 0.91893853320467274178f;

__global__ __launch_bounds__(256) void gaussian_log_prob_kernel(int64_t n, int nu, const float* __restrict__ mean,
                                                               const float* __restrict__ log_std,
                                                               const float* __restrict__ action, float* __restrict__ lp,
                                                               float* __restrict__ ent) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const int a = (int)(idx % nu);
  const float ls = log_std[a];
  const float z = (action[idx] - mean[idx]) * __expf(-ls);
  lp[idx] = -0.5f * z * z - ls - kHalfLog2Pi;
  if (ent) ent[idx] = 0.5f + kHalfLog2Pi + ls;
}

// What the three gradient kernels below share: the gradient of the mean objective with respect to one action's log-density, from
// the row's log ratio, and with respect to the value.
__device__ __forceinline__ float surrogate_grad(const KsPpoLossParams& p, float kl_scale, float logr, float A, float inv_m) {
  const bool log_inside = logr > -p.log_clip_value && logr < p.log_clip_value;
  const float ratio = __expf(fminf(fmaxf(logr, -p.log_clip_value), p.log_clip_value));
  const float lo = 1.f - p.clip_param, hi = 1.f + p.clip_param;
  const float s1 = ratio * A, s2 = fminf(fmaxf(ratio, lo), hi) * A;
  // d(-min(s1, s2)) / d(log ratio); inside the clip range both surrogates coincide
  const bool ratio_inside = ratio > lo && ratio < hi;
  const float g_logr = log_inside && (s1 < s2 || ratio_inside) ? -A * ratio : 0.f;
  return (g_logr - p.kl_coef * kl_scale) * inv_m;  // kl term: (on_lp - lp) * kl_coef * kl_scale per action
}

__device__ __forceinline__ float value_grad(const KsPpoLossParams& p, float vv, float vo, float t, float inv_m) {
  float gv;
  if (p.use_clipped_value_loss) {
    const float dvv = vv - vo;
    const float vc = vo + fminf(fmaxf(dvv, -p.clip_param), p.clip_param);
    const float e = vv - t, ec = vc - t;
    if (e * e >= ec * ec) gv = e;
    else gv = (dvv > -p.clip_param && dvv < p.clip_param) ? ec : 0.f;
  } else {
    gv = vv - t;
  }
  return p.value_loss_coef * gv * inv_m;
}

// The gradient kernels give every (row, action) pair a thread: a workgroup takes whole rows, the pairs leave their log-density
// differences in LDS, one thread per row adds them in action order and turns the sum into the row's gradient factor, and the pairs
// finish with it.  With one thread per row the lanes walked rows 80-2000 bytes apart, twice, and a batch of 12288 rows was 96
// wavefronts (mixture of 10, 17 actions: 610 us, most of it private-memory traffic of the run-time-indexed component arrays).
struct PpoGradIO {
  const float *action, *on_lp, *adv, *tgt, *on_v, *v;
  float* d_value;
};

// What a thread needs of its row (thread r takes row row0 + r; a thread without one reads the last), requested ahead of the pairs' work.
struct PpoRow {
  float adv, v, on_v, tgt;
};
__device__ __forceinline__ PpoRow row_fetch(const PpoGradIO& io, int64_t M, int64_t row0, int rows) {
  const int64_t m = min(row0 + min((int)threadIdx.x, rows - 1), M - 1);
  return {io.adv[m], io.v[m], io.on_v[m], io.tgt[m]};
}

// sel[r] <- gradient factor of row row0 + r from the per-pair differences el[r * nu + a]; also writes the rows' value gradients.
// Barriers on both sides; every thread of the workgroup calls it, which has at least as many threads as rows.
__device__ __forceinline__ void row_factors(const PpoRow& in, float* __restrict__ d_value, const KsPpoLossParams& p, float kl_scale, float inv_m, int64_t M,
                                            int64_t row0, int rows, int nu, const float* el, float* sel) {
  __syncthreads();
  const int r = threadIdx.x;
  if (r < rows && row0 + r < M) {
    float logr = 0.f;
    for (int a = 0; a < nu; ++a) logr += el[r * nu + a];
    sel[r] = surrogate_grad(p, kl_scale, logr, in.adv, inv_m);
    d_value[row0 + r] = value_grad(p, in.v, in.on_v, in.tgt, inv_m);
  }
  __syncthreads();
}

// Gaussian with one log deviation per action.  The log-std gradient of a thread's action is accumulated in its register over the
// workgroup's rows (blockDim.x / nu whole rows at a time, so a thread keeps its action), then over the threads in a fixed order:
// block partials, then ppo_grad_finish_kernel, so the result does not depend on scheduling.  1024 threads: at most 256 workgroups
// (the partials' buffer) still keep 16 wavefronts per CU in flight (65536 rows x 20 actions: 36 -> 19 us).  The next rows' pairs are
// requested as soon as these are used up and the row's own values ahead of the pairs': a workgroup walks its rows a launch's width apart, five
// times there, and waited for memory twice each time (14.4 -> 11.2 us).  At the last stop nothing more is requested, as the barrier waits for it
// (12288 rows 7.0, 6.7 requesting the last rows again, 6.5; 1000 rows of one action 15.2, 15.8, 15.3).
__global__ __launch_bounds__(1024) void ppo_loss_grad_kernel(int64_t M, int nu, KsPpoLossParams p, const float* __restrict__ mean,
                                                            const float* __restrict__ log_std, PpoGradIO io, float* __restrict__ d_mean,
                                                            float* __restrict__ partial) {
  __shared__ float el[1024], sel[1024];
  const int rows = 1024 / nu, r = threadIdx.x / nu, a = threadIdx.x - r * nu;
  const bool mine = r < rows;
  const float inv_m = 1.0f / (float)M, kl_scale = kl_scale_of(p), g_ent = -p.entropy_coef * inv_m;
  const float ls = mine ? log_std[a] : 0.f, is = __expf(-ls);
  float dls = 0.f, f_action, f_mean, f_on_lp;
  auto fetch = [&](int64_t row0) __attribute__((always_inline)) {
    const int64_t i = min(row0 * nu + threadIdx.x, M * nu - 1);
    f_action = io.action[i];
    f_mean = mean[i];
    f_on_lp = io.on_lp[i];
  };
  const int64_t first = (int64_t)blockIdx.x * rows, stride = (int64_t)gridDim.x * rows;
  fetch(first);
  PpoRow in = row_fetch(io, M, first, rows);
  for (int64_t row0 = first; row0 < M; row0 += stride) {
    const bool ok = mine && row0 + r < M;
    const int64_t i = row0 * nu + threadIdx.x;  // the pairs of whole rows are contiguous
    const float z = (f_action - f_mean) * is;
    if (ok) el[threadIdx.x] = (-0.5f * z * z - ls - kHalfLog2Pi) - f_on_lp;
    const bool more = row0 + stride < M;
    if (more) fetch(row0 + stride);
    row_factors(in, io.d_value, p, kl_scale, inv_m, M, row0, rows, nu, el, sel);
    if (more) in = row_fetch(io, M, row0 + stride, rows);
    if (ok) {
      const float g_lp = sel[r];
      d_mean[i] = g_lp * z * is;
      dls += g_lp * (z * z - 1.f) + g_ent;
    }
    __syncthreads();  // the next rows reuse el and sel
  }
  el[threadIdx.x] = dls;
  __syncthreads();
  if ((int)threadIdx.x < nu) {
    float s = 0.f;
    for (int k = 0; k < rows; ++k) s += el[k * nu + threadIdx.x];
    partial[(int64_t)blockIdx.x * nu + threadIdx.x] = s;
  }
}

// log N(action; mean, std) and the entropy per action for the mean | raw deviation head
__global__ __launch_bounds__(256) void gaussian_head_log_prob_kernel(int64_t n, int nu, KsGaussianHead hd, const float* __restrict__ raw,
                                                                    const float* __restrict__ action, float* __restrict__ lp,
                                                                    float* __restrict__ ent) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n) return;
  const int64_t m = idx / nu;
  const int a = (int)(idx - m * nu);
  const float mean = raw[m * 2 * nu + a] + (hd.mean_bias ? hd.mean_bias[a] : 0.f);
  const float r = raw[m * 2 * nu + nu + a];
  const float sp = r > 20.f ? r : log1pf(expf(r));
  const float sd = fminf((sp + hd.min_std) * hd.var_scale, hd.max_std);
  const float z = (action[idx] - mean) / sd, ls = logf(sd);
  lp[idx] = -0.5f * z * z - ls - kHalfLog2Pi;
  if (ent) ent[idx] = 0.5f + kHalfLog2Pi + ls;
}

// One (row, action) pair of the mean | raw deviation head: raw (M, 2 nu) = means | raw deviations,
// std = min((softplus(raw_std) + min_std) * var_scale, max_std).
struct HeadPair {
  float z, sd, sig;
  bool capped;

  // the log-density of the pair's action
  __device__ __forceinline__ float eval(const KsGaussianHead& hd, const float* __restrict__ raw, int64_t m, int a, int nu, float action) {
    const float mean = raw[m * 2 * nu + a] + (hd.mean_bias ? hd.mean_bias[a] : 0.f);
    const float x = raw[m * 2 * nu + nu + a];
    const float sp = x > 20.f ? x : log1pf(expf(x));
    const float pre = (sp + hd.min_std) * hd.var_scale;
    capped = pre >= hd.max_std;
    sd = capped ? hd.max_std : pre;
    sig = x > 20.f ? 1.f : 1.f / (1.f + expf(-x));
    z = (action - mean) / sd;
    return -0.5f * z * z - logf(sd) - kHalfLog2Pi;
  }
  __device__ __forceinline__ void grad(const KsGaussianHead& hd, float g_lp, float g_ent, int64_t m, int a, int nu, float* __restrict__ d_raw) const {
    d_raw[m * 2 * nu + a] = g_lp * z / sd;
    // d/d log(std) of the log-density is z^2 - 1 and of the entropy 1; then through the cap, the scale and the softplus
    const float d_ls = g_lp * (z * z - 1.f) + g_ent;
    d_raw[m * 2 * nu + nu + a] = capped ? 0.f : d_ls / sd * hd.var_scale * sig;
  }
};

// One pair of the mixture-of-Gaussians head: raw (M, 3 nu K) = component means, raw deviations and logits per action.  The entropy
// term uses the usual upper bound of a mixture's entropy, sum_k pi_k H_k + H(pi).  The components stay in registers between the two
// halves: KMAX is the compile-time bound of the loops over K.
template <int KMAX>
struct MixturePair {
  float lpi[KMAX], z[KMAX], sd[KMAX], sig[KMAX], lsd[KMAX], lp;
  unsigned mean_clipped, sd_capped;

  __device__ __forceinline__ float eval(const KsMixtureHead& hd, const float* __restrict__ raw, int64_t m, int a, int nu, float action) {
    const int K = hd.num_mixtures;
    const float* rm = raw + m * 3 * nu * K;
    const float bias = hd.mean_bias ? hd.mean_bias[a] : 0.f;
    const float lo = hd.clip_lo ? hd.clip_lo[a] : -INFINITY, hi = hd.clip_hi ? hd.clip_hi[a] : INFINITY;
    mean_clipped = sd_capped = 0;
    float lmax = -INFINITY;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) { lpi[k] = rm[(2 * nu + a) * K + k]; lmax = fmaxf(lmax, lpi[k]); }
    float zs = 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) zs += expf(lpi[k] - lmax);
    const float lse = lmax + logf(zs);  // the logits' normaliser
    float tmax = -INFINITY;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) {
        lpi[k] -= lse;
        const float r0 = rm[a * K + k] + bias;
        const float mean = fminf(fmaxf(r0, lo), hi);
        if (r0 < lo || r0 > hi) mean_clipped |= 1u << k;
        const float y = rm[(nu + a) * K + k];
        const float sp = y > 20.f ? y : log1pf(expf(y));
        const float pre = (sp + hd.min_std) * hd.var_scale;
        if (pre >= hd.max_std) sd_capped |= 1u << k;
        sd[k] = pre >= hd.max_std ? hd.max_std : pre;
        sig[k] = y > 20.f ? 1.f : 1.f / (1.f + expf(-y));
        z[k] = (action - mean) / sd[k];
        lsd[k] = logf(sd[k]);
        tmax = fmaxf(tmax, lpi[k] - 0.5f * z[k] * z[k] - lsd[k] - kHalfLog2Pi);
      }
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) acc += expf(lpi[k] - 0.5f * z[k] * z[k] - lsd[k] - kHalfLog2Pi - tmax);
    lp = tmax + logf(acc);
    return lp;
  }
  __device__ __forceinline__ void grad(const KsMixtureHead& hd, float g_lp, float g_ent, int64_t m, int a, int nu, float* __restrict__ d_raw) const {
    const int K = hd.num_mixtures;
    // entropy bound: sum_k pi_k (h_k - log pi_k), h_k = 1/2 + log sqrt(2 pi) + log sd_k
    float gbar = 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) gbar += expf(lpi[k]) * (0.5f + kHalfLog2Pi + lsd[k] - lpi[k]);
    float* dm = d_raw + m * 3 * nu * K;
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (k < K) {
        const float pi = expf(lpi[k]);
        const float resp = expf(lpi[k] - 0.5f * z[k] * z[k] - lsd[k] - kHalfLog2Pi - lp);  // responsibility of component k
        dm[a * K + k] = (mean_clipped >> k & 1u) ? 0.f : g_lp * resp * z[k] / sd[k];
        const float d_ls = g_lp * resp * (z[k] * z[k] - 1.f) + g_ent * pi;
        dm[(nu + a) * K + k] = (sd_capped >> k & 1u) ? 0.f : d_ls / sd[k] * hd.var_scale * sig[k];
        dm[(2 * nu + a) * K + k] = g_lp * (resp - pi) + g_ent * pi * (0.5f + kHalfLog2Pi + lsd[k] - lpi[k] - gbar);
      }
  }
};

// The gradient with respect to the raw head outputs.  A workgroup takes 256 / nu whole rows; a head of more than 256 actions takes
// a row per workgroup and evaluates its pairs once for the row's sum and again for the gradient.
template <typename Pair, typename Head>
__global__ __launch_bounds__(256) void ppo_loss_grad_pairs_kernel(int64_t M, int nu, KsPpoLossParams p, Head hd, const float* __restrict__ raw,
                                                                 PpoGradIO io, float* __restrict__ d_raw) {
  __shared__ float el[256], sel[256];
  const float inv_m = 1.0f / (float)M, kl_scale = kl_scale_of(p), g_ent = -p.entropy_coef * inv_m;
  Pair pair;
  if (nu <= 256) {
    const int rows = 256 / nu, r = threadIdx.x / nu, a = threadIdx.x - r * nu;
    const int64_t row0 = (int64_t)blockIdx.x * rows, m = row0 + r;
    const bool ok = r < rows && m < M;
    const PpoRow in = row_fetch(io, M, row0, rows);
    if (ok) el[threadIdx.x] = pair.eval(hd, raw, m, a, nu, io.action[m * nu + a]) - io.on_lp[m * nu + a];
    row_factors(in, io.d_value, p, kl_scale, inv_m, M, row0, rows, nu, el, sel);
    if (ok) pair.grad(hd, sel[r], g_ent, m, a, nu, d_raw);
  } else {
    const int64_t m = blockIdx.x;
    const PpoRow in = row_fetch(io, M, m, 1);
    float part = 0.f;
    for (int a = threadIdx.x; a < nu; a += 256) part += pair.eval(hd, raw, m, a, nu, io.action[m * nu + a]) - io.on_lp[m * nu + a];
    el[threadIdx.x] = part;
    row_factors(in, io.d_value, p, kl_scale, inv_m, M, m, 1, 256, el, sel);
    for (int a = threadIdx.x; a < nu; a += 256) {
      pair.eval(hd, raw, m, a, nu, io.action[m * nu + a]);
      pair.grad(hd, sel[0], g_ent, m, a, nu, d_raw);
    }
  }
}

// d_log_std[a] = sum over the blocks' partial sums: one workgroup per action, a fixed tree over up to 256 partials (one
// thread walking them one after the other spends 256 dependent load latencies on it)
__global__ __launch_bounds__(256) void ppo_grad_finish_kernel(int nblocks, int nu, const float* __restrict__ partial, float* __restrict__ d_log_std) {
  __shared__ float red[256];
  const int a = blockIdx.x;
  float s = 0.f;
  for (int b = threadIdx.x; b < nblocks; b += 256) s += partial[(int64_t)b * nu + a];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) d_log_std[a] = red[0];
}

// adaptive KL: partial[b] = sum over the block's strided share of (on_lp - lp), every element of every row
__global__ __launch_bounds__(256) void kl_parts_kernel(int64_t n, const float* __restrict__ on_lp, const float* __restrict__ lp,
                                                       float* __restrict__ partial) {
  __shared__ float red[256];
  float s = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) s += on_lp[i] - lp[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void kl_adapt_kernel(int nblocks, float inv_rows, float kl_coef, float desired,
                                                       const float* __restrict__ partial, float* __restrict__ kl_scale) {
  __shared__ float red[256];
  red[threadIdx.x] = (int)threadIdx.x < nblocks ? partial[threadIdx.x] : 0.f;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float coef = kl_coef * *kl_scale;
    const float kl_mean = red[0] * inv_rows * coef;
    float c = coef;
    if (kl_mean > desired * 1.5f) c = coef * 1.5f;
    if (kl_mean < desired / 1.5f) c = c / 1.5f;
    c = fminf(fmaxf(c, 1e-8f), 1e2f);
    *kl_scale = c / kl_coef;
  }
}

// One-pole low-pass along the time axis of a trajectory, one thread per (env column, joint), walking the T steps in order:
// y_t = y_{t-1} + alpha (x_t + bias - y_{t-1}), y_{t-1} = 0 at the steps flagged fresh (the carry restarts with the
// episode) and y0 before the first step.  Rows are (t, m) with ld floats each; the first nu columns hold the signal, the
// others travel unchanged.  `add` is an observation-dependent part of the bias: add[(t M + m) add_ld + k] joins joint
// add_first + k.
// Bound by the latency of the steps' loads, a few thousand threads each with its own run of T: a group of steps is requested whole, without
// conditions between its loads, ahead of the arithmetic and the stores of the group before it (loads and stores are waited for in order).
// 1024 envs x 100 steps x 20 joints of rows of 40: 64 -> 30 us; the sweep back: 44 -> 18 (20 steps a group: 28 and 17).  A control step of 4096
// envs 5.7 -> 3.4.
constexpr int kLowpassAhead = 10;

template <int kAhead>  // steps of a group; 1 for the control steps of a rollout, which are calls of one step
__global__ __launch_bounds__(256) void lowpass_scan_kernel(int64_t T, int64_t M, int nu, int ld, float alpha,
                                                           const float* __restrict__ x, const float* __restrict__ mean_bias,
                                                           const float* __restrict__ add, int64_t add_ld, int add_first, int add_count,
                                                           const float* __restrict__ y0, const uint8_t* __restrict__ fresh,
                                                           float* __restrict__ y, float* __restrict__ y_last) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * (int64_t)ld) return;
  const int64_t m = idx / ld;
  const int j = (int)(idx - m * ld);
  if (j >= nu) {  // the columns behind the signal (raw deviations of the head): copied when the output is another buffer
    if (x != y)
      for (int64_t t0 = 0; t0 < T; t0 += kAhead) {
        float v[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) v[k] = t0 + k < T ? x[((t0 + k) * M + m) * ld + j] : 0.f;
#pragma unroll
        for (int k = 0; k < kAhead; ++k)
          if (t0 + k < T) y[((t0 + k) * M + m) * ld + j] = v[k];
      }
    return;
  }
  const float b = mean_bias ? mean_bias[j] : 0.f;
  const bool has_add = add && j >= add_first && j < add_first + add_count;
  const float* addp = has_add ? add + (j - add_first) : x + j;  // a joint without a term of its own reads its signal twice
  const int64_t addl = has_add ? add_ld : ld;
  float last = y0 ? y0[m * nu + j] : 0.f;
  struct Steps { float v[kAhead], w[kAhead]; unsigned f[kAhead]; } now, next = {};
  auto fetch = [&](int64_t t0, Steps& s) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int64_t r = (t0 + k < T ? t0 + k : T - 1) * M + m;
      s.v[k] = x[r * ld + j];
      s.w[k] = addp[r * addl];
      s.f[k] = 0u;
    }
    if (fresh)
#pragma unroll
      for (int k = 0; k < kAhead; ++k) s.f[k] = fresh[(t0 + k < T ? t0 + k : T - 1) * M + m];
  };
  fetch(0, now);
  for (int64_t t0 = 0; t0 < T; t0 += kAhead) {
    // in place, the group's own stores come behind these loads, and every thread reads its own entries only
    if (t0 + kAhead < T) fetch(t0 + kAhead, next);
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (t0 + k < T) {
        float v = now.v[k] + b;
        v = has_add ? v + now.w[k] : v;
        if (now.f[k]) last = 0.f;
        last = last + alpha * (v - last);
        y[((t0 + k) * M + m) * ld + j] = last;
      }
    now = next;
  }
  if (y_last) y_last[m * nu + j] = last;
}

// Reverse sweep of the same recursion: with g_t = dL/dy_t on entry, the gradient reaching y_t is
// G_t = g_t + (1 - alpha) G_{t+1} unless step t + 1 is fresh (the carry was cut there), and dL/dx_t = alpha G_t, written in
// place.  d_y0 receives (1 - alpha) G_0 unless step 0 is fresh.
__global__ __launch_bounds__(256) void lowpass_scan_backward_kernel(int64_t T, int64_t M, int nu, int ld, float alpha,
                                                                    const uint8_t* __restrict__ fresh, float* __restrict__ g,
                                                                    float* __restrict__ d_y0) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * (int64_t)nu) return;
  const int64_t m = idx / nu;
  const int j = (int)(idx - m * nu);
  float carry = 0.f;  // (1 - alpha) G_{t+1}, or 0 across an episode start
  constexpr int kAhead = kLowpassAhead;
  struct Steps { float v[kAhead]; unsigned f[kAhead]; } now, next = {};
  auto fetch = [&](int64_t t0, Steps& s) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      s.v[k] = g[((t0 - k >= 0 ? t0 - k : 0) * M + m) * ld + j];
      s.f[k] = 0u;
    }
    if (fresh)
#pragma unroll
      for (int k = 0; k < kAhead; ++k) s.f[k] = fresh[(t0 - k >= 0 ? t0 - k : 0) * M + m];
  };
  fetch(T - 1, now);
  for (int64_t t0 = T - 1; t0 >= 0; t0 -= kAhead) {
    if (t0 - kAhead >= 0) fetch(t0 - kAhead, next);
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (t0 - k >= 0) {
        const float G = now.v[k] + carry;
        g[((t0 - k) * M + m) * ld + j] = alpha * G;
        carry = now.f[k] ? 0.f : (1.f - alpha) * G;
      }
    now = next;
  }
  if (d_y0) d_y0[idx] = carry;
}

// Mirrored rows: mirror[r][j] = sign[j] * x[r][perm[j]], and a copy of the rows in `same` where the caller wants both.  Row r goes
// (r / group) * group rows further down in either output, so that whole groups of rows and of images can alternate in one buffer.
// Bound by memory.  A thread keeps four columns and takes them of kMirrorRows rows, all of them requested at once: the columns' places and signs are
// read once, and what they point at does not wait for them again.  The last four columns of a row overlap the ones before where the width is odd (the
// same values twice).  `span` rows lie side by side in a workgroup; rows of more than 1024 columns take it several times.
//   100 x 512 rows of 475 and their images: 154 us as a permutation and a concatenation, 79 with a column's place
//   read for every row, 64 (4.6 TB/s) here
struct __attribute__((packed, aligned(4))) RowQuad { float v[4]; };  // rows of an odd width start at any float; a 16-byte access needs no more
constexpr int kMirrorRows = 4;
__global__ __launch_bounds__(256) void mirror_rows_kernel(int64_t rows, int n, int quads, int span, int64_t group, const float* __restrict__ x,
                                                          const int* __restrict__ perm, const float* __restrict__ sign, float* __restrict__ same,
                                                          float* __restrict__ mirror) {
  const int r0 = quads > 256 ? 0 : (int)(threadIdx.x / (unsigned)quads), first = (int)threadIdx.x - r0 * quads;
  if (r0 >= span) return;
  const int64_t row0 = (int64_t)blockIdx.x * (span * kMirrorRows), g0 = row0 / group, rest0 = row0 - g0 * group;
  auto out_row = [&](int r) { return row0 + r + (rest0 + r < group ? g0 : g0 + (rest0 + r) / group) * (same ? group : 0); };
  for (int e = first; e < quads; e += 256) {
    const int j = n >= 4 && 4 * e > n - 4 ? n - 4 : 4 * e;
    if (n >= 4) {
      int place[4];
      float sg[4], got[kMirrorRows][4];
      RowQuad own[kMirrorRows];
#pragma unroll
      for (int k = 0; k < 4; ++k) { place[k] = perm[j + k]; sg[k] = sign[j + k]; }
#pragma unroll
      for (int u = 0; u < kMirrorRows; ++u) {
        const float* row = x + min(row0 + r0 + u * span, rows - 1) * n;
        own[u] = *reinterpret_cast<const RowQuad*>(row + j);
#pragma unroll
        for (int k = 0; k < 4; ++k) got[u][k] = row[place[k]];
      }
#pragma unroll
      for (int u = 0; u < kMirrorRows; ++u) {
        const int r = r0 + u * span;
        if (row0 + r >= rows) break;
        const int64_t at = out_row(r) * n + j;
        RowQuad m;
#pragma unroll
        for (int k = 0; k < 4; ++k) m.v[k] = sg[k] * got[u][k];
        if (same) *reinterpret_cast<RowQuad*>(same + at) = own[u];
        *reinterpret_cast<RowQuad*>(mirror + at) = m;
      }
    } else {
      for (int u = 0; u < kMirrorRows; ++u) {
        const int r = r0 + u * span;
        if (row0 + r >= rows) break;
        const float* row = x + (row0 + r) * n;
        const int64_t at = out_row(r) * n;
        for (int k = 0; k < n; ++k) {
          if (same) same[at + k] = row[k];
          mirror[at + k] = sign[k] * row[perm[k]];
        }
      }
    }
  }
}

// One thread per (row, j): diff = y[r][j] - sign[j] ym[r][perm[j]].  perm is a bijection, so the thread owns dym[r][perm[j]].
// The row's loss is summed by the thread of j = 0 over the row, in index order.
__global__ __launch_bounds__(256) void mirror_loss_grad_kernel(int64_t rows, int n, float scale, const float* __restrict__ y,
                                                               const float* __restrict__ ym, const int* __restrict__ perm,
                                                               const float* __restrict__ sign, float* __restrict__ dy,
                                                               float* __restrict__ dym, float* __restrict__ loss) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * n) return;
  const int64_t r = idx / n;
  const int j = (int)(idx - r * n);
  const float c = 2.f * scale / ((float)n * (float)rows);
  const int pj = perm[j];
  const float sj = sign[j];
  const float diff = y[idx] - sj * ym[r * n + pj];
  dy[idx] += c * diff;
  dym[r * n + pj] = -c * sj * diff;
  if (loss && j == 0) {
    float s = 0.f;
    for (int k = 0; k < n; ++k) {
      const float d = y[r * n + k] - sign[k] * ym[r * n + perm[k]];
      s += d * d;
    }
    loss[r] = scale * s / (float)n;
  }
}

}  // namespace ks

static float lowpass_alpha(float ctrl_dt, float cutoff) {  // actions.py:254-255, in float like ks_action_filter
  return ctrl_dt / (1.f / (6.28318530717958647692f * cutoff) + ctrl_dt);
}

extern "C" int ks_lowpass_scan(ks_stream_t stream, int64_t T, int64_t M, int32_t nu, int32_t ld, float ctrl_dt, float cutoff,
                               const float* x, const float* mean_bias, const float* add, int64_t add_ld, int32_t add_first,
                               int32_t add_count, const float* y0, const uint8_t* fresh, float* y, float* y_last) {
  if (T < 0 || M < 0 || nu < 1 || ld < nu) return ks::fail(KS_EINVAL, "ks_lowpass_scan: bad shape (T %lld, M %lld, nu %d, ld %d)", (long long)T, (long long)M, nu, ld);
  if (!(ctrl_dt > 0.f) || !(cutoff > 0.f)) return ks::fail(KS_EINVAL, "ks_lowpass_scan: ctrl_dt and the cutoff frequency must be positive");
  if (T == 0 || M == 0) return KS_OK;
  if (!x || !y) return ks::fail(KS_EINVAL, "ks_lowpass_scan: null pointer");
  if (add && (add_first < 0 || add_count < 1 || add_first + add_count > nu || add_ld < add_count))
    return ks::fail(KS_EINVAL, "ks_lowpass_scan: the additive bias covers joints [%d, %d) of %d with rows of %lld floats", add_first,
                    add_first + add_count, nu, (long long)add_ld);
  const int64_t total = M * ld, grid = (total + 255) / 256;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_lowpass_scan: too many elements");
  hipLaunchKernelGGL(T == 1 ? ks::lowpass_scan_kernel<1> : ks::lowpass_scan_kernel<ks::kLowpassAhead>, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, T, M, nu, ld,
                     lowpass_alpha(ctrl_dt, cutoff), x, mean_bias, add, add_ld, add_first, add_count, y0, fresh, y, y_last);
  return ks::check_launch("ks_lowpass_scan");
}

extern "C" int ks_lowpass_scan_backward(ks_stream_t stream, int64_t T, int64_t M, int32_t nu, int32_t ld, float ctrl_dt, float cutoff,
                                        const uint8_t* fresh, float* g, float* d_y0) {
  if (T < 0 || M < 0 || nu < 1 || ld < nu) return ks::fail(KS_EINVAL, "ks_lowpass_scan_backward: bad shape");
  if (!(ctrl_dt > 0.f) || !(cutoff > 0.f)) return ks::fail(KS_EINVAL, "ks_lowpass_scan_backward: ctrl_dt and the cutoff frequency must be positive");
  if (T == 0 || M == 0) return KS_OK;
  if (!g) return ks::fail(KS_EINVAL, "ks_lowpass_scan_backward: null pointer");
  const int64_t total = M * nu, grid = (total + 255) / 256;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_lowpass_scan_backward: too many elements");
  hipLaunchKernelGGL(ks::lowpass_scan_backward_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, T, M, nu, ld,
                     lowpass_alpha(ctrl_dt, cutoff), fresh, g, d_y0);
  return ks::check_launch("ks_lowpass_scan_backward");
}

static int mirror_rows(const char* who, ks_stream_t stream, int64_t rows, int64_t group, int32_t n, const float* x, const int32_t* perm,
                       const float* sign, float* same, float* mirror) {
  const int quads = n / 4 + (n % 4 != 0), span = quads >= 256 ? 1 : 256 / quads, per = span * ks::kMirrorRows;
  const int64_t grid = (rows + per - 1) / per;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "%s: too many elements", who);
  hipLaunchKernelGGL(ks::mirror_rows_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, rows, n, quads, span, group, x, perm, sign, same,
                     mirror);
  return ks::check_launch(who);
}

extern "C" int ks_signed_permute(ks_stream_t stream, int64_t rows, int32_t n, const float* x, const int32_t* perm, const float* sign,
                                 float* out) {
  if (rows < 0 || n < 1) return ks::fail(KS_EINVAL, "ks_signed_permute: bad shape");
  if (rows == 0) return KS_OK;
  if (!x || !perm || !sign || !out || x == out) return ks::fail(KS_EINVAL, "ks_signed_permute: null pointer, or in place");
  return mirror_rows("ks_signed_permute", stream, rows, rows, n, x, perm, sign, nullptr, out);
}

extern "C" int ks_mirror_pairs(ks_stream_t stream, int64_t groups, int64_t group, int32_t n, const float* x, const int32_t* perm, const float* sign,
                               float* out) {
  if (groups < 0 || group < 0 || n < 1) return ks::fail(KS_EINVAL, "ks_mirror_pairs: bad shape");
  if (groups == 0 || group == 0) return KS_OK;
  if (!x || !perm || !sign || !out || x == out) return ks::fail(KS_EINVAL, "ks_mirror_pairs: null pointer, or in place");
  return mirror_rows("ks_mirror_pairs", stream, groups * group, group, n, x, perm, sign, out, out + group * n);
}

extern "C" int ks_mirror_loss_grad(ks_stream_t stream, int64_t rows, int32_t n, float scale, const float* y, const float* ym,
                                   const int32_t* perm, const float* sign, float* dy, float* dym, float* loss) {
  if (rows < 1 || n < 1) return ks::fail(KS_EINVAL, "ks_mirror_loss_grad: bad shape");
  if (!y || !ym || !perm || !sign || !dy || !dym) return ks::fail(KS_EINVAL, "ks_mirror_loss_grad: null pointer");
  const int64_t total = rows * n, grid = (total + 255) / 256;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_mirror_loss_grad: too many elements");
  hipLaunchKernelGGL(ks::mirror_loss_grad_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, rows, n, scale, y, ym, perm,
                     sign, dy, dym, loss);
  return ks::check_launch("ks_mirror_loss_grad");
}

extern "C" int ks_ppo_adapt_kl(ks_stream_t stream, int64_t rows, int32_t A, const float* on_log_probs, const float* log_probs,
                               float kl_coef, float desired_kl, float* kl_scale, float* workspace) {
  if (rows < 1 || A < 1) return ks::fail(KS_EINVAL, "ks_ppo_adapt_kl: bad shape");
  if (!on_log_probs || !log_probs || !kl_scale || !workspace) return ks::fail(KS_EINVAL, "ks_ppo_adapt_kl: null pointer");
  if (!(kl_coef > 0.f) || !(desired_kl > 0.f)) return ks::fail(KS_EINVAL, "ks_ppo_adapt_kl: kl_coef and desired_kl must be positive");
  const int64_t n = rows * A;
  const int64_t want = (n + 1023) / 1024;
  const int blocks = (int)(want < 256 ? want : 256);
  hipLaunchKernelGGL(ks::kl_parts_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, n, on_log_probs, log_probs, workspace);
  hipLaunchKernelGGL(ks::kl_adapt_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, blocks, 1.f / (float)rows, kl_coef, desired_kl,
                     (const float*)workspace, kl_scale);
  return ks::check_launch("ks_ppo_adapt_kl");
}

extern "C" int ks_gaussian_log_prob(ks_stream_t stream, int64_t M, int32_t nu, const float* mean, const float* log_std,
                                    const float* action, float* log_prob, float* entropy) {
  if (M < 0 || nu < 1) return ks::fail(KS_EINVAL, "ks_gaussian_log_prob: bad shape");
  if (M == 0) return KS_OK;
  if (!mean || !log_std || !action || !log_prob) return ks::fail(KS_EINVAL, "ks_gaussian_log_prob: null pointer");
  const int64_t n = M * nu;
  hipLaunchKernelGGL(ks::gaussian_log_prob_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, nu, mean,
                     log_std, action, log_prob, entropy);
  return ks::check_launch("ks_gaussian_log_prob");
}

extern "C" int ks_ppo_loss_grad(ks_stream_t stream, int64_t M, int32_t nu, const KsPpoLossParams* params, const float* mean,
                                const float* log_std, const float* action, const float* on_log_probs,
                                const float* advantages, const float* value_targets, const float* on_values,
                                const float* values, float* d_mean, float* d_value, float* d_log_std, void* workspace) {
  if (!params) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad: null parameters");
  if (M < 1 || nu < 1 || nu > KS_MAX_ACTIONS) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad: bad shape (1..%d actions)", KS_MAX_ACTIONS);
  if (!mean || !log_std || !action || !on_log_probs || !advantages || !value_targets || !on_values || !values || !d_mean ||
      !d_value || !d_log_std || !workspace)
    return ks::fail(KS_EINVAL, "ks_ppo_loss_grad: null pointer");
  const int64_t want = (M + 1024 / nu - 1) / (1024 / nu);
  const int blocks = (int)(want < KS_PPO_GRAD_BLOCKS ? want : KS_PPO_GRAD_BLOCKS);
  const ks::PpoGradIO io = {action, on_log_probs, advantages, value_targets, on_values, values, d_value};
  hipLaunchKernelGGL(ks::ppo_loss_grad_kernel, dim3(blocks), dim3(1024), 0, (hipStream_t)stream, M, nu, *params, mean, log_std, io, d_mean,
                     (float*)workspace);
  hipLaunchKernelGGL(ks::ppo_grad_finish_kernel, dim3(nu), dim3(256), 0, (hipStream_t)stream, blocks, nu, (const float*)workspace,
                     d_log_std);
  return ks::check_launch("ks_ppo_loss_grad");
}

extern "C" int ks_ppo_loss_grad_head(ks_stream_t stream, int64_t M, int32_t nu, const KsPpoLossParams* params,
                                     const KsGaussianHead* head, const float* raw, const float* action, const float* on_log_probs,
                                     const float* advantages, const float* value_targets, const float* on_values,
                                     const float* values, float* d_raw, float* d_value) {
  if (!params || !head) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_head: null parameters");
  if (M < 1 || nu < 1) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_head: bad shape");
  if (!raw || !action || !on_log_probs || !advantages || !value_targets || !on_values || !values || !d_raw || !d_value)
    return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_head: null pointer");
  if (!(head->max_std > 0.f) || head->min_std < 0.f || !(head->var_scale > 0.f))
    return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_head: bad deviation bounds");
  const int64_t rows = nu <= 256 ? 256 / nu : 1, grid = (M + rows - 1) / rows;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_ppo_loss_grad_head: too many rows");
  const ks::PpoGradIO io = {action, on_log_probs, advantages, value_targets, on_values, values, d_value};
  hipLaunchKernelGGL((ks::ppo_loss_grad_pairs_kernel<ks::HeadPair, KsGaussianHead>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M,
                     nu, *params, *head, raw, io, d_raw);
  return ks::check_launch("ks_ppo_loss_grad_head");
}

extern "C" int ks_gaussian_head_log_prob(ks_stream_t stream, int64_t M, int32_t nu, const KsGaussianHead* head, const float* raw,
                                         const float* action, float* log_prob, float* entropy) {
  if (M < 0 || nu < 1) return ks::fail(KS_EINVAL, "ks_gaussian_head_log_prob: bad shape");
  if (M == 0) return KS_OK;
  if (!head || !raw || !action || !log_prob) return ks::fail(KS_EINVAL, "ks_gaussian_head_log_prob: null pointer");
  if (!(head->max_std > 0.f) || head->min_std < 0.f || !(head->var_scale > 0.f))
    return ks::fail(KS_EINVAL, "ks_gaussian_head_log_prob: bad deviation bounds");
  const int64_t n = M * nu, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_gaussian_head_log_prob: too many elements");
  hipLaunchKernelGGL(ks::gaussian_head_log_prob_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, n, nu, *head, raw, action,
                     log_prob, entropy);
  return ks::check_launch("ks_gaussian_head_log_prob");
}

extern "C" int ks_ppo_loss_grad_mixture(ks_stream_t stream, int64_t M, int32_t nu, const KsPpoLossParams* params,
                                        const KsMixtureHead* head, const float* raw, const float* action, const float* on_log_probs,
                                        const float* advantages, const float* value_targets, const float* on_values,
                                        const float* values, float* d_raw, float* d_value) {
  if (!params || !head) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_mixture: null parameters");
  if (M < 1 || nu < 1) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_mixture: bad shape");
  if (head->num_mixtures < 1 || head->num_mixtures > KS_MAX_MIXTURES)
    return ks::fail(KS_ELIMIT, "ks_ppo_loss_grad_mixture: %d components, 1..%d are built", head->num_mixtures, KS_MAX_MIXTURES);
  if (!raw || !action || !on_log_probs || !advantages || !value_targets || !on_values || !values || !d_raw || !d_value)
    return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_mixture: null pointer");
  if (!(head->max_std > 0.f) || head->min_std < 0.f || !(head->var_scale > 0.f))
    return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_mixture: bad deviation bounds");
  if ((head->clip_lo == nullptr) != (head->clip_hi == nullptr)) return ks::fail(KS_EINVAL, "ks_ppo_loss_grad_mixture: clip_lo and clip_hi come together");
  const int64_t rows = nu <= 256 ? 256 / nu : 1, grid = (M + rows - 1) / rows;
  if (grid > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_ppo_loss_grad_mixture: too many rows");
  const ks::PpoGradIO io = {action, on_log_probs, advantages, value_targets, on_values, values, d_value};
  const int K = head->num_mixtures;  // the loops over the components are unrolled to the next bound
  auto kfn = K <= 5 ? ks::ppo_loss_grad_pairs_kernel<ks::MixturePair<5>, KsMixtureHead>
                    : (K <= 10 ? ks::ppo_loss_grad_pairs_kernel<ks::MixturePair<10>, KsMixtureHead>
                               : ks::ppo_loss_grad_pairs_kernel<ks::MixturePair<KS_MAX_MIXTURES>, KsMixtureHead>);
  hipLaunchKernelGGL(kfn, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, nu, *params, *head, raw, io, d_raw);
  return ks::check_launch("ks_ppo_loss_grad_mixture");
}

extern "C" int ks_gather_columns(ks_stream_t stream, int32_t n, const KsGatherArray* arrays, int64_t columns, int64_t picked, const int64_t* index) {
  if (n < 0 || (n > 0 && !arrays) || columns < 0 || picked < 0) return ks::fail(KS_EINVAL, "ks_gather_columns: bad argument");
  if (n > KS_GATHER_ARRAYS) return ks::fail(KS_ELIMIT, "ks_gather_columns: %d arrays (0..%d)", n, KS_GATHER_ARRAYS);
  if (picked > 0 && (columns == 0 || !index)) return ks::fail(KS_EINVAL, "ks_gather_columns: nothing to pick from");
  if (picked > 0x7fffffff) return ks::fail(KS_ELIMIT, "ks_gather_columns: too many columns");
  ks::GatherTable t;
  t.n = 0;
  int64_t blocks = 0;
  for (int k = 0; k < n; ++k) {
    const KsGatherArray& a = arrays[k];
    if (a.outer < 0 || a.inner < 0) return ks::fail(KS_EINVAL, "ks_gather_columns: array %d: negative size", k);
    if (a.outer == 0 || a.inner == 0 || picked == 0) continue;
    if (!a.src || !a.dst) return ks::fail(KS_EINVAL, "ks_gather_columns: array %d: null pointer", k);
    const uint64_t bits = (uint64_t)(uintptr_t)a.src | (uint64_t)(uintptr_t)a.dst | (uint64_t)a.inner;
    uint32_t lb = 0;
    while (lb < 4 && !(bits >> lb & 1)) ++lb;
    const int64_t inner = a.inner >> lb;
    if (a.outer > 0xffffffffll / inner / picked) return ks::fail(KS_ELIMIT, "ks_gather_columns: array %d is too large", k);
    const int64_t words = a.outer * inner * picked;
    t.a[t.n++] = {(const char*)a.src, (char*)a.dst, (uint32_t)words, (uint32_t)inner, lb, (uint32_t)blocks};
    blocks += (words + ks::kGatherWords - 1) / ks::kGatherWords;
  }
  if (t.n == 0) return KS_OK;
  hipLaunchKernelGGL(ks::gather_columns_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, t, columns, (uint32_t)picked, index);
  return ks::check_launch("ks_gather_columns");
}
