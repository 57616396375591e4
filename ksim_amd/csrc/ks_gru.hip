// GRU and LSTM cells for recurrent policies in the rollout, and the GRU's backward pass through time.  The two gate projections are plain linear
// layers and run through the MLP entry points (matrix cores for bf16); one streaming kernel then combines the gates.
#include "ks_common.h"

#include <type_traits>
#include <vector>

namespace ks {

// gi = W_ih x + b (M, 3H), gh = W_hh h + (0, 0, b_n) (M, 3H), gate order reset | update | candidate:
//   r = sigmoid(gi_r + gh_r), z = sigmoid(gi_z + gh_z), n = tanh(gi_n + r * gh_n), h' = n + z (h - n)
// An env that starts an episode (fresh[m] != 0) takes h = 0; gh was computed from the stored h, so its
// contribution is replaced by the bias part alone, which for zero h is (0, 0, b_n).
__global__ __launch_bounds__(256) void gru_gate_kernel(int64_t M, int H, const float* __restrict__ gi,
                                                       const float* __restrict__ gh, const float* __restrict__ h_in,
                                                       const float* __restrict__ bias_n, const uint8_t* __restrict__ fresh,
                                                       float* __restrict__ h_out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* a = gi + m * 3 * H;
  const float* b = gh + m * 3 * H;
  const float hr = f ? 0.f : b[j], hz = f ? 0.f : b[H + j], hn = f ? bias_n[j] : b[2 * H + j];
  const float h = f ? 0.f : h_in[idx];
  const float r = 1.f / (1.f + expf(-(a[j] + hr)));
  const float z = 1.f / (1.f + expf(-(a[H + j] + hz)));
  const float n = tanhf(a[2 * H + j] + r * hn);
  h_out[idx] = n + z * (h - n);
}

// The same cell for training: also keeps what the backward pass needs, saved (M, 5H) = r | z | n | hn | h, where hn is the
// hidden part of the candidate (what r multiplies) and h the hidden state the cell actually used (zero for a fresh env).
__global__ __launch_bounds__(256) void gru_gate_train_kernel(int64_t M, int H, const float* __restrict__ gi,
                                                             const float* __restrict__ gh, const float* __restrict__ h_in,
                                                             const float* __restrict__ bias_n, const uint8_t* __restrict__ fresh,
                                                             float* __restrict__ h_out, float* __restrict__ saved) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* a = gi + m * 3 * H;
  const float* b = gh + m * 3 * H;
  const float hr = f ? 0.f : b[j], hz = f ? 0.f : b[H + j], hn = f ? bias_n[j] : b[2 * H + j];
  const float h = f ? 0.f : h_in[idx];
  const float r = 1.f / (1.f + expf(-(a[j] + hr)));
  const float z = 1.f / (1.f + expf(-(a[H + j] + hz)));
  const float n = tanhf(a[2 * H + j] + r * hn);
  h_out[idx] = n + z * (h - n);
  float* sv = saved + m * 5 * H;
  sv[j] = r; sv[H + j] = z; sv[2 * H + j] = n; sv[3 * H + j] = hn; sv[4 * H + j] = h;
}

// Backward through the gates of one step.  dh_out is the gradient reaching h' (from the layer above at this step plus
// from the next step).  d_gi (M, 3H) is the gradient of the input projection's output, d_gh (M, 3H) that of the hidden
// projection's output (its n part is also the gradient of bias_n, fresh rows included); dh_in = dh_out * z is the direct
// path to the previous hidden state, zero for a fresh env (the hidden projection adds its share afterwards).
__global__ __launch_bounds__(256) void gru_gate_backward_kernel(int64_t M, int H, const float* __restrict__ dh_out,
                                                                const float* __restrict__ saved, const uint8_t* __restrict__ fresh,
                                                                float* __restrict__ d_gi, float* __restrict__ d_gh,
                                                                float* __restrict__ dh_in) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* sv = saved + m * 5 * H;
  const float r = sv[j], z = sv[H + j], n = sv[2 * H + j], hn = sv[3 * H + j], h = sv[4 * H + j];
  const float d = dh_out[idx];
  const float dn_pre = d * (1.f - z) * (1.f - n * n);
  const float dz_pre = d * (h - n) * z * (1.f - z);
  const float dr_pre = dn_pre * hn * r * (1.f - r);
  float* a = d_gi + m * 3 * H;
  float* b = d_gh + m * 3 * H;
  a[j] = dr_pre; a[H + j] = dz_pre; a[2 * H + j] = dn_pre;
  b[j] = dr_pre; b[H + j] = dz_pre; b[2 * H + j] = dn_pre * r;
  dh_in[idx] = f ? 0.f : d * z;
}

// LSTM: g = W_ih x + W_hh h + b (M, 4H) in gate order input | forget | cell | output:
//   c' = sigmoid(f) c + sigmoid(i) tanh(g),  h' = sigmoid(o) tanh(c').  A fresh env starts from h = c = 0, which
// leaves only the input projection (it carries the whole bias).
__global__ __launch_bounds__(256) void lstm_gate_kernel(int64_t M, int H, const float* __restrict__ gi,
                                                        const float* __restrict__ gh, const float* __restrict__ c_in,
                                                        const uint8_t* __restrict__ fresh, float* __restrict__ h_out,
                                                        float* __restrict__ c_out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* a = gi + m * 4 * H;
  const float* b = gh + m * 4 * H;
  float g[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) g[k] = a[k * H + j] + (f ? 0.f : b[k * H + j]);
  const float c = f ? 0.f : c_in[idx];
  const float si = 1.f / (1.f + expf(-g[0])), sf = 1.f / (1.f + expf(-g[1])), so = 1.f / (1.f + expf(-g[3]));
  const float cn = sf * c + si * tanhf(g[2]);
  c_out[idx] = cn;
  h_out[idx] = so * tanhf(cn);
}

// The LSTM cell for training: saved (M, 7H) = i | f | g | o | tanh(c') | c | h with the gate activations, the cell and
// hidden state the step actually used (zero for a fresh env).
__global__ __launch_bounds__(256) void lstm_gate_train_kernel(int64_t M, int H, const float* __restrict__ gi,
                                                              const float* __restrict__ gh, const float* __restrict__ h_in,
                                                              const float* __restrict__ c_in, const uint8_t* __restrict__ fresh,
                                                              float* __restrict__ h_out, float* __restrict__ c_out,
                                                              float* __restrict__ saved) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* a = gi + m * 4 * H;
  const float* b = gh + m * 4 * H;
  float g[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) g[k] = a[k * H + j] + (f ? 0.f : b[k * H + j]);
  const float c = f ? 0.f : c_in[idx], h = f ? 0.f : h_in[idx];
  const float si = 1.f / (1.f + expf(-g[0])), sf = 1.f / (1.f + expf(-g[1])), so = 1.f / (1.f + expf(-g[3]));
  const float tg = tanhf(g[2]);
  const float cn = sf * c + si * tg;
  const float tc = tanhf(cn);
  c_out[idx] = cn;
  h_out[idx] = so * tc;
  float* sv = saved + m * 7 * H;
  sv[j] = si; sv[H + j] = sf; sv[2 * H + j] = tg; sv[3 * H + j] = so; sv[4 * H + j] = tc; sv[5 * H + j] = c; sv[6 * H + j] = h;
}

// Backward through the gates of one LSTM step: dh_out, dc_out are the gradients reaching h' and c'.  d_g (M, 4H) is the
// gradient of the summed gate pre-activations, hence of both projections' outputs; dc_in = dc f is the gradient of the
// incoming cell state and dh_in starts at zero (the hidden projection adds its share afterwards); both are zero for a fresh env.
__global__ __launch_bounds__(256) void lstm_gate_backward_kernel(int64_t M, int H, const float* __restrict__ dh_out,
                                                                 const float* __restrict__ dc_out, const float* __restrict__ saved,
                                                                 const uint8_t* __restrict__ fresh, float* __restrict__ d_g,
                                                                 float* __restrict__ dh_in, float* __restrict__ dc_in) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * H) return;
  const int64_t m = idx / H;
  const int j = (int)(idx - m * H);
  const bool f = fresh && fresh[m];
  const float* sv = saved + m * 7 * H;
  const float si = sv[j], sf = sv[H + j], tg = sv[2 * H + j], so = sv[3 * H + j], tc = sv[4 * H + j], c = sv[5 * H + j];
  const float dh = dh_out[idx];
  const float dc = dc_out[idx] + dh * so * (1.f - tc * tc);
  float* a = d_g + m * 4 * H;
  a[j] = dc * tg * si * (1.f - si);
  a[H + j] = dc * c * sf * (1.f - sf);
  a[2 * H + j] = dc * si * (1.f - tg * tg);
  a[3 * H + j] = dh * tc * so * (1.f - so);
  dc_in[idx] = f ? 0.f : dc * sf;
  dh_in[idx] = 0.f;
}

// ---------------------------------------------------------------- a whole trajectory of one LSTM layer in one launch
// The step-by-step path costs two GEMM launches and a gate kernel per step, layer and network: a minibatch of 100 control steps
// is thousands of launches of a few microseconds each.  Here a workgroup of eight wavefronts owns 4 rows (envs) for all T
// steps, so that a minibatch of a thousand rows is one workgroup per CU.  The product runs on v_mfma_f32_4x4x1 (sixteen
// independent 4x4 outer products per instruction): block b = lane / 4 of wavefront w is hidden unit 16 w + b, its four B entries
// are that unit's input / forget / cell / output rows of W_hh and the four A entries, the same for every block and therefore
// broadcast from one block, the four rows' hidden state; after K = 128 instructions and a 4 x 4 transpose inside each group of
// four lanes, lane (b, j) holds the four gate pre-activations of its unit for row j.  The wavefront's slice of W_hh stays in
// 128 vector registers per lane for the whole sequence, the hidden state of the 4 rows lives in LDS (double buffered), the
// cell state in a register; a step is 128 MFMAs (the fp32 matrix rate: 4 rows x 512 x 128 multiply-adds per CU), the gate
// arithmetic of one (unit, row) per lane, and one barrier.  fp32 cells of hidden size 128.
typedef __attribute__((ext_vector_type(4))) float f32x4;
// One recurrent layer over a trajectory, as the sequence kernels take it; a launch runs one or two of them (blockIdx.y): the actor's and the
// critic's layer of one depth, which are as many workgroups as a batch has sets of 4 rows and leave half the chip idle below 1024 rows, each by
// itself as long as the other.  Whole updates of an LSTM policy: 64 envs x 100 steps 2670 -> 1760 us, 512 x 60 2570 -> 2030, 2 x 128 x 80 with
// mirror images 4740 -> 3530; with 1024 rows per network nothing changes.
struct Seq {
  int64_t M;
  const float* in;  // forward: the input projections (T, M, gates); backward: dH
  const void* W;    // forward: W_hh; backward: its transpose
  int ldw;
  const float *bias_n, *h0, *c0;
  const uint8_t* fresh;
  float* saved;
  float *out0, *out1;  // forward: hs, cs (LSTM); backward: d_g (LSTM) or d_gi, d_gh (GRU)
  float *dh0, *dc0;
};

constexpr int kSeqRows = 4, kSeqH = 128, kSeqWaves = 8, kSeqPadH = kSeqH + 4;

__device__ __forceinline__ float sigmoid_ks(float x) { return 1.f / (1.f + expf(-x)); }

// 1 / (1 + e^-x) and tanh x = 1 - 2 / (e^2x + 1) on v_exp_f32 and v_rcp_f32; both saturate correctly (e^y = inf gives 0 and -1 + 2 = 1)
__device__ __forceinline__ float seq_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
__device__ __forceinline__ float seq_tanh(float x) { return 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f); }

// Barrier for data that the wavefronts of a workgroup hand each other through LDS only: it waits for this wavefront's LDS
// traffic, not for its global loads and stores.  __syncthreads() would also drain the step's stores (and the loads fetched
// ahead for the next step) before every barrier, a memory round trip per step of the sequence.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The LSTM forward kernel's way in and out of memory: a step's inputs are requested a step ahead of their use.  Where the activations are kept, nine
// results a step leave behind it, one load or store (KS_SEQ_SIDE, a single instruction from a uniform address) after every eight matrix instructions
// of the next.  All together at a step's end they held the CU's wavefronts up at once, and a store or load under a condition makes the compiler wait
// for the step's stores before the next step: loads and stores are counted together and waited for in order.  Hence no conditions (the outputs that
// a launch has are template arguments, rows past the batch repeat the last row and store its values once more, the last step requests its own inputs
// again) and nothing pending where the loop is entered.  Without kept activations a step stores one or two values, and the order imposed on its
// matrix instructions costs more than it gives: loads at its start, stores at its end, the rest as the compiler likes.
// Two layers, everything at the step's end and under conditions -> one after every eight -> as here:
//   1024 rows x 100 steps, kept 372 -> 358 -> 358 us, not kept 302 -> 314 -> 298; 64 x 100, not kept 145 -> 155 -> 136; 512 x 24 with cell states
//   43.9 -> 45.7 -> 41.7; one step (a rollout's call) of 4096 rows 34.6 -> 34.4 -> 33.6, of 64 10.3 -> 10.5 -> 10.3
// What is left is issue and power: 2048 of 3500 cycles of a step are matrix instructions, at 2.0 to 2.2 GHz.  The backward kernel (342 -> 361 us) and
// the GRU's (31 us either way) did not gain from the same order.
__device__ __forceinline__ void seq_loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)
#define KS_SEQ_SIDE(OP)                \
  {                                    \
    __builtin_amdgcn_sched_barrier(0); \
    OP;                                \
    __builtin_amdgcn_sched_barrier(0); \
  }

// where hidden unit u of a row sits in the LDS copy of the state: unit u = 16 q + b is register q of block b (see the forward
// kernel), and a lane reads its block's 8 registers as 8 consecutive floats
__device__ __forceinline__ int seq_slot(int u) { return 8 * (u & 15) + (u >> 4); }

// Transpose of a 4 x 4 block held by four neighbouring lanes (lane j of the group holds a0..a3): out[g] = a_j of lane g.
// Two stages of exchanges within the group (DPP quad permutes) and selects: lanes that differ in the low bit swap what lies off their
// diagonal in the pairs (a0, a1), (a2, a3), then lanes that differ in the high bit in the pairs (0, 2), (1, 3).  (A select by lane index per
// entry became branches: 221 -> 198 us for 100 steps of an LSTM layer.)
template <int CTRL>
__device__ __forceinline__ float quad_perm(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ void quad_swap(float& lo, float& hi, bool upper) {  // the upper lane sends `lo`, the lower one `hi`
  const float got = quad_perm<CTRL>(upper ? lo : hi);
  lo = upper ? got : lo;
  hi = upper ? hi : got;
}
__device__ __forceinline__ void quad_transpose(float a0, float a1, float a2, float a3, int j, float (&out)[4]) {
  const bool odd = (j & 1) != 0, high = (j & 2) != 0;
  quad_swap<0xB1>(a0, a1, odd);   // quad_perm [1,0,3,2]
  quad_swap<0xB1>(a2, a3, odd);
  quad_swap<0x4E>(a0, a2, high);  // quad_perm [2,3,0,1]
  quad_swap<0x4E>(a1, a3, high);
  out[0] = a0; out[1] = a1; out[2] = a2; out[3] = a3;
}

// Sums over the four 16-lane rows of a wavefront, scattered: row q of lanes ends up with the total of v[q], added up as
// (row 0 + row 1) + (row 2 + row 3).  A swap exchanges half of one register with half of the other, which is the whole exchange of a
// stage; through LDS the same sums were eight permutes of a hundred cycles.
__device__ __forceinline__ float rows_reduce_scatter(float v0, float v1, float v2, float v3) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1" : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3));
  float lo = v0 + v1, hi = v2 + v3;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
  return lo + hi;
}

template <bool CELL, bool SAVE>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lstm_seq_forward_kernel(int T, int groups, Seq first, Seq second) {
  constexpr int H = kSeqH;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ gi = s.in;
  const float* __restrict__ W = (const float*)s.W;
  const int ldw = s.ldw;
  const float *h0 = s.h0, *c0 = s.c0;
  const uint8_t* __restrict__ fresh = s.fresh;
  float *hs = s.out0, *cs = s.out1;  // with T = 1, hs / cs may be h0 / c0
  float* __restrict__ saved = s.saved;
  __shared__ __attribute__((aligned(16))) float sh[2][kSeqRows][kSeqPadH];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 3, unit = 16 * wave + (lane >> 2);
  // The weights are the B operand: block b, entry lane % 4: W_hh[gate lane % 4, unit][k].  The hidden state is the A operand and
  // is the same for all sixteen blocks, so it is broadcast from one block per instruction (CBSZ = 4, ABID = k % 16): the four
  // lanes of block k % 16 hold h[row 0..3][k] in register k / 16, i.e. the 512 values of the state sit once in 8 registers of the
  // wavefront instead of once per block.  In LDS the state is stored in that order (row, block, register), two 16-byte reads per
  // lane and step.
  float wa[H];
  {
    const float4* src = reinterpret_cast<const float4*>(W + (int64_t)(j * H + unit) * ldw);
#pragma unroll
    for (int k4 = 0; k4 < H / 4; ++k4) {
      const float4 v = src[k4];
      wa[4 * k4] = v.x; wa[4 * k4 + 1] = v.y; wa[4 * k4 + 2] = v.z; wa[4 * k4 + 3] = v.w;
    }
  }
  // A workgroup takes `groups` sets of 4 rows one after the other with the same registers of weights: a single step over
  // thousands of rows (the rollout's call) would otherwise fetch the 256 KB of W_hh once per 4 rows.
  for (int grp = 0; grp < groups; ++grp) {
  const int64_t r0 = ((int64_t)blockIdx.x * groups + grp) * kSeqRows;
  if (r0 >= M) break;  // the same for every thread of the workgroup
  const unsigned jr = r0 + j < M ? j : (unsigned)(M - 1 - r0);
  const int64_t m = r0 + jr;
  if (grp > 0) __syncthreads();  // the previous set's last read of the state buffers is over
  float c = c0[m * H + unit];
  float hprev = h0[m * H + unit];  // the state this lane's (unit, row) enters the step with
  sh[0][j][seq_slot(unit)] = hprev;
  struct In { float g[4]; unsigned f; } in0 = {}, in1 = {};
  float si = 0.f, sf = 0.f, tg = 0.f, so = 0.f, tc = 0.f, cp = 0.f, hu = 0.f;
  auto load = [&](int t, In& in, int k) __attribute__((always_inline)) {
    const int64_t o = (int64_t)(t < T ? t : T - 1) * M + r0;
    if (k < 4) in.g[k] = (gi + (o * 4 + k) * H)[jr * 4 * H + unit];
    else if (fresh) in.f = (fresh + o)[jr];
  };
  auto store = [&](int t, int k) __attribute__((always_inline)) {
    const int64_t o = (int64_t)t * M + r0;
    if (k == 0) (hs + o * H)[jr * H + unit] = hprev;
    if (CELL && k == 1) (cs + o * H)[jr * H + unit] = c;
    if (SAVE && k >= 2) {
      const float v[7] = {si, sf, tg, so, tc, cp, hu};
      (saved + (o * 7 + k - 2) * H)[jr * 7 * H + unit] = v[k - 2];
    }
  };
#pragma unroll
  for (int k = 0; k < 5; ++k) load(0, in0, k);
  seq_loads_done();
  __syncthreads();
  auto step = [&](int t, auto cur, bool first, const In& in, In& next) __attribute__((always_inline)) {
    if constexpr (!SAVE) {
#pragma unroll
      for (int k = 0; k < 5; ++k) load(t + 1, next, k);
    }
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    float ha[8];
    {
      const float4 a0 = *reinterpret_cast<const float4*>(&sh[cur][j][8 * (lane >> 2)]);
      const float4 a1 = *reinterpret_cast<const float4*>(&sh[cur][j][8 * (lane >> 2) + 4]);
      ha[0] = a0.x; ha[1] = a0.y; ha[2] = a0.z; ha[3] = a0.w; ha[4] = a1.x; ha[5] = a1.y; ha[6] = a1.z; ha[7] = a1.w;
    }
    // k runs 0..127 in order, even k into one accumulator and odd k into the other
#define KS_SEQ_MFMA(K0)                                                                                            \
    acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ha[(K0) >> 4], wa[(K0)], acc0, 4, (K0) & 15, 0);                       \
    acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ha[((K0) + 1) >> 4], wa[(K0) + 1], acc1, 4, ((K0) + 1) & 15, 0);
#define KS_SEQ_MFMA8(N, OP) KS_SEQ_MFMA(8 * N) KS_SEQ_MFMA(8 * N + 2) KS_SEQ_MFMA(8 * N + 4) KS_SEQ_MFMA(8 * N + 6) if constexpr (SAVE) KS_SEQ_SIDE(OP)
#define KS_SEQ_OUT(N) KS_SEQ_MFMA8(N, if (!first) store(t - 1, N))
#define KS_SEQ_IN(N) KS_SEQ_MFMA8(N, load(t + 1, next, 13 - N))
    KS_SEQ_OUT(0) KS_SEQ_OUT(1) KS_SEQ_OUT(2) KS_SEQ_OUT(3) KS_SEQ_OUT(4) KS_SEQ_OUT(5) KS_SEQ_OUT(6) KS_SEQ_OUT(7) KS_SEQ_OUT(8)
    KS_SEQ_IN(9) KS_SEQ_IN(10) KS_SEQ_IN(11) KS_SEQ_IN(12) KS_SEQ_IN(13) KS_SEQ_MFMA8(14, ) KS_SEQ_MFMA8(15, )
#undef KS_SEQ_IN
#undef KS_SEQ_OUT
#undef KS_SEQ_MFMA8
#undef KS_SEQ_MFMA
    // lane (unit, gate lane % 4) now holds that gate for the four rows in its four registers; the gates want the transpose
    // within each group of four lanes: lane (unit, row j) with the four gates
    float pre[4];
    quad_transpose(acc0[0] + acc1[0], acc0[1] + acc1[1], acc0[2] + acc1[2], acc0[3] + acc1[3], j, pre);
    const bool f = in.f != 0;
    cp = f ? 0.f : c;
    hu = f ? 0.f : hprev;
    // the hardware exponential and reciprocal (about 1 ulp each) instead of the library's expf, tanhf and IEEE division: a
    // fifth of the instructions, and the gates are as many instructions per step as the matrix work is cycles
    si = seq_sigmoid(in.g[0] + (f ? 0.f : pre[0]));
    sf = seq_sigmoid(in.g[1] + (f ? 0.f : pre[1]));
    tg = seq_tanh(in.g[2] + (f ? 0.f : pre[2]));
    so = seq_sigmoid(in.g[3] + (f ? 0.f : pre[3]));
    c = sf * cp + si * tg;
    tc = seq_tanh(c);
    hprev = so * tc;
    sh[cur ^ 1][j][seq_slot(unit)] = hprev;
    if constexpr (!SAVE) { store(t, 0); store(t, 1); }
    lds_barrier();  // the new hidden state is complete; the buffer just read is free for the step after next
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  step(0, even, true, in0, in1);
  int t = 1;
  for (; t + 1 < T; t += 2) {
    step(t, odd, false, in1, in0);
    step(t + 1, even, false, in0, in1);
  }
  if (t < T) step(t, odd, false, in1, in0);
  if constexpr (SAVE) {
#pragma unroll
    for (int k = 0; k < 9; ++k) store(T - 1, k);
  }
  }
}

// The reverse sweep of the same layer: dH (T, M, H) is the gradient reaching h_t from the layer above; the gradient through
// W_hh and that of the cell state are carried in registers.  Per step: the gate derivatives from the saved activations
// (lstm_gate_backward_kernel's formulas) into d_g (T, M, 4H) and LDS, then dh_{t-1} = d_g W_hh over the transposed weights.
// Here the sixteen blocks of an MFMA are four quarters of the 4H gate rows (K split four ways: quarter kg = lane / 16 is gate kg) times
// four groups of four units.  The gate gradients are the A operand (entries = the four rows), the same for the four blocks of a quarter and
// broadcast to them from one block per instruction (CBSZ = 2, ABID = k mod 4): a lane fetches 32 of its quarter's 128 gate rows, eight 16-byte
// reads per step.  (Fetched by every block, they were 32 reads per lane, as many cycles of the LDS pipe as the products are of the matrix
// cores.)  A lane accumulates, for its unit, the four rows' partial sums over its quarter; the quarters are added up and scattered over
// the lane rows, which leaves lane l with unit 16 w + l % 16 of row l / 16.
// 1024 rows, 100 steps: 248 -> 169 us, of which the 128 products of two wavefronts per SIMD are 85.
// where the gradient of gate row g H + u of a row sits in LDS: lane (quarter g, block a = u mod 4, row) reads its 32 as consecutive floats;
// the paddings put the sixteen lanes of a quarter on different banks
constexpr int kSeqGateA = 36, kSeqGateRow = 4 * 4 * kSeqGateA + 16;

__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lstm_seq_backward_kernel(int T, Seq first, Seq second) {
  constexpr int H = kSeqH;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ dH = s.in;
  const float* __restrict__ saved = s.saved;
  const uint8_t* __restrict__ fresh = s.fresh;
  const float* __restrict__ Wt = (const float*)s.W;
  const int ldwt = s.ldw;
  float* __restrict__ d_g = s.out0;
  float *dh0 = s.dh0, *dc0 = s.dc0;
  if ((int64_t)blockIdx.x * kSeqRows >= M) return;  // the other layer of the launch has more rows
  __shared__ __attribute__((aligned(16))) float sg[2][kSeqRows * kSeqGateRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane >> 4, blk = (lane >> 2) & 3, i = lane & 3;
  const int unit = 16 * wave + (lane & 15);  // the (unit, row kg) whose gate arithmetic and carried gradients this lane owns
  const int64_t r0 = (int64_t)blockIdx.x * kSeqRows;
  const int64_t m = r0 + kg;
  const bool row_ok = m < M;
  const int64_t mc = row_ok ? m : M - 1;
  // B operand, entry lane % 4 of block (kg, lane / 4 % 4): Wt[unit][gate row 128 kg + s]
  float wa[128];
  {
    const float4* src = reinterpret_cast<const float4*>(Wt + (int64_t)unit * ldwt + 128 * kg);
#pragma unroll
    for (int s4 = 0; s4 < 32; ++s4) {
      const float4 v = src[s4];
      wa[4 * s4] = v.x; wa[4 * s4 + 1] = v.y; wa[4 * s4 + 2] = v.z; wa[4 * s4 + 3] = v.w;
    }
  }
  float dhc = 0.f, dc = 0.f;
  const int put = kg * kSeqGateRow + (unit & 3) * kSeqGateA + (unit >> 2);  // of gate 0; the next gate 4 kSeqGateA on
  const int get = i * kSeqGateRow + (4 * kg + blk) * kSeqGateA;
  // the step's inputs from memory are fetched one step ahead, under the matrix work of the step before
  float nx[7];
  uint8_t fnext = 0;
  {
    const int64_t o = (int64_t)(T - 1) * M + mc;
    const float* sv = saved + o * 7 * H + unit;
#pragma unroll
    for (int k = 0; k < 6; ++k) nx[k] = sv[k * H];
    nx[6] = dH[o * H + unit];
    if (fresh) fnext = fresh[o];
  }
  int cur = 0;
  for (int t = T - 1; t >= 0; --t) {
    const bool f = fnext != 0;
    const float si = nx[0], sf = nx[1], tg = nx[2], so = nx[3], tc = nx[4], cp = nx[5];
    const float dh = nx[6] + dhc;
    if (t > 0) {
      const int64_t o = (int64_t)(t - 1) * M + mc;
      const float* sv = saved + o * 7 * H + unit;
#pragma unroll
      for (int k = 0; k < 6; ++k) nx[k] = sv[k * H];
      nx[6] = dH[o * H + unit];
      if (fresh) fnext = fresh[o];
    }
    const float dct = dc + dh * so * (1.f - tc * tc);
    const float gI = dct * tg * si * (1.f - si), gF = dct * cp * sf * (1.f - sf), gG = dct * si * (1.f - tg * tg),
                gO = dh * tc * so * (1.f - so);
    dc = f ? 0.f : dct * sf;
    float* to = &sg[cur][put];
    to[0] = gI; to[4 * kSeqGateA] = gF; to[8 * kSeqGateA] = gG; to[12 * kSeqGateA] = gO;
    if (row_ok) {
      float* dg = d_g + ((int64_t)t * M + m) * 4 * H + unit;
      dg[0] = gI; dg[H] = gF; dg[2 * H] = gG; dg[3 * H] = gO;
    }
    lds_barrier();  // the gate gradients are complete; the buffer of the step before is free for the step after
    float ga[32];
    {
      const float4* src = reinterpret_cast<const float4*>(&sg[cur][get]);
#pragma unroll
      for (int q4 = 0; q4 < 8; ++q4) {
        const float4 v = src[q4];
        ga[4 * q4] = v.x; ga[4 * q4 + 1] = v.y; ga[4 * q4 + 2] = v.z; ga[4 * q4 + 3] = v.w;
      }
    }
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 32; ++q) {  // k = 4 q .. 4 q + 3 of the quarter, even k into one accumulator and odd k into the other
      acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q], acc0, 2, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 1], acc1, 2, 1, 0);
      acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 2], acc0, 2, 2, 0);
      acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 3], acc1, 2, 3, 0);
    }
    const float mine = rows_reduce_scatter(acc0[0] + acc1[0], acc0[1] + acc1[1], acc0[2] + acc1[2], acc0[3] + acc1[3]);
    dhc = f ? 0.f : mine;
    cur ^= 1;
  }
  if (row_ok) {
    if (dh0) dh0[m * H + unit] = dhc;
    if (dc0) dc0[m * H + unit] = dc;
  }
}

// ---------------------------------------------------------------- a whole trajectory of one GRU layer in one launch
// The layout of the LSTM kernels above: eight wavefronts own 4 rows for all T steps, block b = lane / 4 of wavefront w is hidden
// unit 16 w + b, its B entries are that unit's reset / update / candidate rows of W_hh (the fourth entry is zero), and the four
// rows' state is the A operand broadcast from one block per instruction.  fp32 cells multiply with v_mfma_f32_4x4x1 (128 per step);
// bf16 cells with v_mfma_f32_4x4x4 bf16 (32 per step), for which the state, kept in fp32 in a register of the lane that owns it,
// is rounded to bf16 on its way to LDS, as the per-step products round their input.  Bound by the latency of a step's chain
// (LDS read, products, gates, LDS write, barrier); the per-step launches this replaces were four per step and layer (512 rows,
// 24 steps, bf16: 4 x 24 launches of 3-8 us -> one of 27 us; 30 backward).
typedef __attribute__((ext_vector_type(4))) short s16x4;

__device__ __forceinline__ short bf16_bits(float x) { return __builtin_bit_cast(short, (__bf16)x); }

template <bool BF>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gru_seq_forward_kernel(int T, int groups, Seq first, Seq second) {
  constexpr int H = kSeqH;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ gi = s.in;
  const void* __restrict__ Wv = s.W;
  const int ldw = s.ldw;
  const float* __restrict__ bias_n = s.bias_n;
  const float* h0 = s.h0;
  const uint8_t* __restrict__ fresh = s.fresh;
  float* hs = s.out0;  // with T = 1, hs may be h0
  float* __restrict__ saved = s.saved;
  // fp32: the state in seq_slot order, two 16-byte reads per lane and step.  bf16: in natural order, block b reads units 4 b .. 4 b + 3
  // and 64 + 4 b .. (8 bytes each): the operands of instructions b and 16 + b
  __shared__ __attribute__((aligned(16))) float sh[2][kSeqRows][kSeqPadH];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 3, blk = lane >> 2, unit = 16 * wave + blk;
  constexpr int NW = BF ? 1 : H, NB = BF ? H / 4 : 1;
  float wa[NW];
  s16x4 wb[NB];
  if constexpr (BF) {
    const s16x4* src = reinterpret_cast<const s16x4*>((const short*)Wv + (int64_t)((j < 3 ? j : 0) * H + unit) * ldw);
#pragma unroll
    for (int k4 = 0; k4 < NB; ++k4) {
      const s16x4 v = src[k4];
      wb[k4] = j < 3 ? v : s16x4{0, 0, 0, 0};
    }
  } else {
    const float4* src = reinterpret_cast<const float4*>((const float*)Wv + (int64_t)((j < 3 ? j : 0) * H + unit) * ldw);
#pragma unroll
    for (int k4 = 0; k4 < NW / 4; ++k4) {
      const float4 v = src[k4];
      wa[4 * k4] = j < 3 ? v.x : 0.f; wa[4 * k4 + 1] = j < 3 ? v.y : 0.f; wa[4 * k4 + 2] = j < 3 ? v.z : 0.f; wa[4 * k4 + 3] = j < 3 ? v.w : 0.f;
    }
  }
  const float bn = bias_n[unit];
  for (int grp = 0; grp < groups; ++grp) {  // as in the LSTM kernel: several sets of 4 rows with the same registers of weights
    const int64_t r0 = ((int64_t)blockIdx.x * groups + grp) * kSeqRows;
    if (r0 >= M) break;  // the same for every thread of the workgroup
    const int64_t m = r0 + j;
    const bool row_ok = m < M;
    const int64_t mc = row_ok ? m : M - 1;  // loads of the rows past the batch are clamped, their stores dropped
    if (grp > 0) __syncthreads();
    float hprev = h0[mc * H + unit];
    if constexpr (BF) reinterpret_cast<short*>(&sh[0][j][0])[unit] = bf16_bits(hprev);
    else sh[0][j][seq_slot(unit)] = hprev;
    __syncthreads();
    int cur = 0;
    float gnext[3];
    uint8_t fnext = 0;
#pragma unroll
    for (int g = 0; g < 3; ++g) gnext[g] = gi[mc * 3 * H + g * H + unit];
    if (fresh) fnext = fresh[mc];
    for (int t = 0; t < T; ++t) {
      float gin[3];
#pragma unroll
      for (int g = 0; g < 3; ++g) gin[g] = gnext[g];
      const bool f = fnext != 0;
      if (t + 1 < T) {  // the next step's inputs, fetched under this step's work
        const int64_t tn = (int64_t)(t + 1) * M + mc;
#pragma unroll
        for (int g = 0; g < 3; ++g) gnext[g] = gi[tn * 3 * H + g * H + unit];
        if (fresh) fnext = fresh[tn];
      }
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
      if constexpr (BF) {
        const s16x4* row = reinterpret_cast<const s16x4*>(&sh[cur][j][0]);
        const s16x4 a0 = row[blk], a1 = row[16 + blk];
#define KS_GRU_MFMA(B)                                                                                    \
        acc0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a0, wb[(B)], acc0, 4, (B), 0);                       \
        acc1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a1, wb[16 + (B)], acc1, 4, (B), 0);
#define KS_GRU_MFMA4(B) KS_GRU_MFMA(B) KS_GRU_MFMA((B) + 1) KS_GRU_MFMA((B) + 2) KS_GRU_MFMA((B) + 3)
        KS_GRU_MFMA4(0) KS_GRU_MFMA4(4) KS_GRU_MFMA4(8) KS_GRU_MFMA4(12)
#undef KS_GRU_MFMA4
#undef KS_GRU_MFMA
      } else {
        float ha[8];
        {
          const float4 a0 = *reinterpret_cast<const float4*>(&sh[cur][j][8 * blk]);
          const float4 a1 = *reinterpret_cast<const float4*>(&sh[cur][j][8 * blk + 4]);
          ha[0] = a0.x; ha[1] = a0.y; ha[2] = a0.z; ha[3] = a0.w; ha[4] = a1.x; ha[5] = a1.y; ha[6] = a1.z; ha[7] = a1.w;
        }
#define KS_GRU_MFMA(K0)                                                                                            \
        acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ha[(K0) >> 4], wa[(K0)], acc0, 4, (K0) & 15, 0);                    \
        acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ha[((K0) + 1) >> 4], wa[(K0) + 1], acc1, 4, ((K0) + 1) & 15, 0);
#define KS_GRU_MFMA8(K0) KS_GRU_MFMA(K0) KS_GRU_MFMA((K0) + 2) KS_GRU_MFMA((K0) + 4) KS_GRU_MFMA((K0) + 6)
#define KS_GRU_MFMA32(K0) KS_GRU_MFMA8(K0) KS_GRU_MFMA8((K0) + 8) KS_GRU_MFMA8((K0) + 16) KS_GRU_MFMA8((K0) + 24)
        KS_GRU_MFMA32(0) KS_GRU_MFMA32(32) KS_GRU_MFMA32(64) KS_GRU_MFMA32(96)
#undef KS_GRU_MFMA32
#undef KS_GRU_MFMA8
#undef KS_GRU_MFMA
      }
      float pre[4];
      quad_transpose(acc0[0] + acc1[0], acc0[1] + acc1[1], acc0[2] + acc1[2], acc0[3] + acc1[3], j, pre);
      const float hu = f ? 0.f : hprev;
      const float hn = bn + (f ? 0.f : pre[2]);
      // the library's functions and IEEE division, as in gru_gate_kernel: seq_tanh cancels near zero (1.5e-7 absolute, three digits of 1e-4)
      const float r = sigmoid_ks(gin[0] + (f ? 0.f : pre[0]));
      const float z = sigmoid_ks(gin[1] + (f ? 0.f : pre[1]));
      const float n = tanhf(gin[2] + r * hn);
      hprev = n + z * (hu - n);
      if constexpr (BF) reinterpret_cast<short*>(&sh[cur ^ 1][j][0])[unit] = bf16_bits(hprev);
      else sh[cur ^ 1][j][seq_slot(unit)] = hprev;
      if (row_ok) {
        const int64_t o = (int64_t)t * M + m;
        hs[o * H + unit] = hprev;
        if (saved) {
          float* sv = saved + o * 5 * H + unit;
          sv[0] = r; sv[H] = z; sv[2 * H] = n; sv[3 * H] = hn; sv[4 * H] = hu;
        }
      }
      lds_barrier();
      cur ^= 1;
    }
  }
}

// The reverse sweep (gru_gate_backward_kernel's formulas): dh_{t-1} = dh_t z + d_gh W_hh.  Sixteen blocks = four quarters of the 3H gate
// rows (96 each) times four groups of four units, operands and sums as in the LSTM's sweep; in bf16 a step of four k is one block's entry.
template <bool BF>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gru_seq_backward_kernel(int T, Seq first, Seq second) {
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ dH = s.in;
  const float* __restrict__ saved = s.saved;
  const uint8_t* __restrict__ fresh = s.fresh;
  const void* __restrict__ Wtv = s.W;
  const int ldwt = s.ldw;
  float *__restrict__ d_gi = s.out0, *__restrict__ d_gh = s.out1;
  float* dh0 = s.dh0;
  if ((int64_t)blockIdx.x * kSeqRows >= M) return;  // the other layer of the launch has more rows
  constexpr int H = kSeqH, KQ = 3 * H / 4;  // gate rows per quarter
  typedef typename std::conditional<BF, short, float>::type G;
  // what a lane reads (KQ / 4 consecutive entries), padded so that the sixteen lanes of a quarter hit different banks
  constexpr int LA = BF ? 24 : 28, LR = 16 * LA + (BF ? 64 : 16);
  __shared__ __attribute__((aligned(16))) G sg[2][kSeqRows * LR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane >> 4, blk = (lane >> 2) & 3, i = lane & 3;
  const int unit = 16 * wave + (lane & 15);
  const int64_t m = (int64_t)blockIdx.x * kSeqRows + kg;
  const bool row_ok = m < M;
  const int64_t mc = row_ok ? m : M - 1;
  constexpr int NW = BF ? 1 : KQ, NB = BF ? KQ / 4 : 1;
  float wa[NW];
  s16x4 wb[NB];
  if constexpr (BF) {
    const s16x4* src = reinterpret_cast<const s16x4*>((const short*)Wtv + (int64_t)unit * ldwt + KQ * kg);
#pragma unroll
    for (int s4 = 0; s4 < NB; ++s4) wb[s4] = src[s4];
  } else {
    const float4* src = reinterpret_cast<const float4*>((const float*)Wtv + (int64_t)unit * ldwt + KQ * kg);
#pragma unroll
    for (int s4 = 0; s4 < NW / 4; ++s4) {
      const float4 v = src[s4];
      wa[4 * s4] = v.x; wa[4 * s4 + 1] = v.y; wa[4 * s4 + 2] = v.z; wa[4 * s4 + 3] = v.w;
    }
  }
  // where gate row g H + unit of this lane's row goes: quarter, block (fp32: k mod 4; bf16: k / 4 mod 4) and place among the block's entries
  int put[3];
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    const int row = g * H + unit, q = row / KQ, k = row - q * KQ;
    put[g] = kg * LR + (BF ? (4 * q + ((k >> 2) & 3)) * LA + (k >> 4) * 4 + (k & 3) : (4 * q + (k & 3)) * LA + (k >> 2));
  }
  const int get = i * LR + (4 * kg + blk) * LA;
  float dhc = 0.f;
  float nx[6];
  uint8_t fnext = 0;
  {
    const int64_t o = (int64_t)(T - 1) * M + mc;
    const float* sv = saved + o * 5 * H + unit;
#pragma unroll
    for (int k = 0; k < 5; ++k) nx[k] = sv[k * H];
    nx[5] = dH[o * H + unit];
    if (fresh) fnext = fresh[o];
  }
  int cur = 0;
  for (int t = T - 1; t >= 0; --t) {
    const bool f = fnext != 0;
    const float r = nx[0], z = nx[1], n = nx[2], hn = nx[3], h = nx[4];
    const float d = nx[5] + dhc;
    if (t > 0) {
      const int64_t o = (int64_t)(t - 1) * M + mc;
      const float* sv = saved + o * 5 * H + unit;
#pragma unroll
      for (int k = 0; k < 5; ++k) nx[k] = sv[k * H];
      nx[5] = dH[o * H + unit];
      if (fresh) fnext = fresh[o];
    }
    const float gN = d * (1.f - z) * (1.f - n * n);
    const float gZ = d * (h - n) * z * (1.f - z);
    const float gR = gN * hn * r * (1.f - r);
    const float gNh = gN * r;
    if constexpr (BF) {
      sg[cur][put[0]] = bf16_bits(gR); sg[cur][put[1]] = bf16_bits(gZ); sg[cur][put[2]] = bf16_bits(gNh);
    } else {
      sg[cur][put[0]] = gR; sg[cur][put[1]] = gZ; sg[cur][put[2]] = gNh;
    }
    if (row_ok) {
      const int64_t o = ((int64_t)t * M + m) * 3 * H + unit;
      d_gi[o] = gR; d_gi[o + H] = gZ; d_gi[o + 2 * H] = gN;
      d_gh[o] = gR; d_gh[o + H] = gZ; d_gh[o + 2 * H] = gNh;
    }
    lds_barrier();
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    if constexpr (BF) {
      s16x4 ga[6];
      const s16x4* src = reinterpret_cast<const s16x4*>(&sg[cur][get]);
#pragma unroll
      for (int q = 0; q < 6; ++q) ga[q] = src[q];
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        acc0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ga[q], wb[4 * q], acc0, 2, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ga[q], wb[4 * q + 1], acc1, 2, 1, 0);
        acc0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ga[q], wb[4 * q + 2], acc0, 2, 2, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ga[q], wb[4 * q + 3], acc1, 2, 3, 0);
      }
    } else {
      float ga[24];
      const float4* src = reinterpret_cast<const float4*>(&sg[cur][get]);
#pragma unroll
      for (int q4 = 0; q4 < 6; ++q4) {
        const float4 v = src[q4];
        ga[4 * q4] = v.x; ga[4 * q4 + 1] = v.y; ga[4 * q4 + 2] = v.z; ga[4 * q4 + 3] = v.w;
      }
#pragma unroll
      for (int q = 0; q < 24; ++q) {
        acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q], acc0, 2, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 1], acc1, 2, 1, 0);
        acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 2], acc0, 2, 2, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(ga[q], wa[4 * q + 3], acc1, 2, 3, 0);
      }
    }
    const float mine = rows_reduce_scatter(acc0[0] + acc1[0], acc0[1] + acc1[1], acc0[2] + acc1[2], acc0[3] + acc1[3]);
    dhc = f ? 0.f : d * z + mine;
    cur ^= 1;
  }
  if (row_ok && dh0) dh0[m * H + unit] = dhc;
}

}  // namespace ks

using namespace ks;

struct KsGru {
  int I, H;
  KsMlp *proj_i, *proj_h;
  float* bias_n;        // device (H), as given at creation
  const float* bias_nt; // training handles: the same entries of the hidden projection's bias, which the optimiser updates in place
  const float* bn() const { return bias_nt ? bias_nt : bias_n; }
};

extern "C" int ks_gru_create(const KsGruDesc* d, KsGru** out) {
  if (!d || !out) return fail(KS_EINVAL, "ks_gru_create: null argument");
  if (d->input_size < 1 || d->hidden_size < 1 || d->hidden_size > 21845) return fail(KS_EINVAL, "ks_gru_create: bad sizes %d -> %d", d->input_size, d->hidden_size);
  if (!d->weight_ih || !d->weight_hh) return fail(KS_EINVAL, "ks_gru_create: weights are required");
  const int H = d->hidden_size, I = d->input_size;
  std::vector<float> zero(3 * (size_t)H, 0.f), bh(3 * (size_t)H, 0.f);
  if (d->bias_n) for (int j = 0; j < H; ++j) bh[2 * (size_t)H + j] = d->bias_n[j];
  KsGru* g = new KsGru{I, H, nullptr, nullptr, nullptr, nullptr};
  KsMlpDesc md = {};
  md.n_layers = 1; md.activation = KS_ACT_NONE; md.dtype = d->dtype;
  md.dims[0] = I; md.dims[1] = 3 * H; md.weights[0] = d->weight_ih; md.biases[0] = d->bias ? d->bias : zero.data();
  int rc = ks_mlp_create(&md, &g->proj_i);
  if (rc == KS_OK) {
    md.dims[0] = H; md.weights[0] = d->weight_hh; md.biases[0] = bh.data();
    rc = ks_mlp_create(&md, &g->proj_h);
  }
  if (rc == KS_OK && (hipMalloc((void**)&g->bias_n, H * 4) != hipSuccess ||
                      hipMemcpy(g->bias_n, bh.data() + 2 * (size_t)H, H * 4, hipMemcpyHostToDevice) != hipSuccess))
    rc = fail(KS_ELAUNCH, "ks_gru_create: upload failed");
  if (rc != KS_OK) { ks_gru_destroy(g); return rc; }
  *out = g;
  return KS_OK;
}

extern "C" int ks_gru_destroy(KsGru* g) {
  if (!g) return KS_OK;
  ks_mlp_destroy(g->proj_i);
  ks_mlp_destroy(g->proj_h);
  if (g->bias_n) (void)hipFree(g->bias_n);
  delete g;
  return KS_OK;
}

static int64_t up256(int64_t n) { return (n + 255) / 256 * 256; }

// whether the one-launch sequence kernels cover this cell: hidden size 128, either precision
static bool gru_seq_weights(const KsGru* g, const void** W, int* ldw, const void** Wt, int* ldwt, bool* bf16) {
  int np = 0, kp = 0, dt = 0;
  *W = *Wt = nullptr;
  if (!g || g->H != kSeqH || mlp_peek_layer(g->proj_h, 0, W, Wt, &np, &kp, &dt) != KS_OK) return false;
  if (np != 3 * kSeqH || kp < kSeqH || (kp & 7)) return false;
  *ldw = kp; *ldwt = np; *bf16 = dt == KS_MLP_BF16;
  return *W != nullptr;
}

// sets of 4 rows per workgroup of the sequence kernels: one while there is at most one set per CU (long sequences want every CU),
// more when a short call covers so many rows that re-reading the weights per set would dominate it
static int seq_groups(int64_t T, int64_t sets) {
  int groups = 1;
  if (T * 8 <= 64) while (groups < 8 && sets > (int64_t)256 * groups) groups *= 2;
  return groups;
}

extern "C" int ks_gru_sequence_supported(const KsGru* g) {
  const void *W, *Wt;
  int a, b;
  bool bf;
  return gru_seq_weights(g, &W, &a, &Wt, &b, &bf) ? 1 : 0;
}

// the checks and launch of `n` layers over T steps (0 rows: nothing to do); `fill` checks a layer's operands and adds its weights
template <typename Fill, typename Launch>
static int run_sequences(const char* who, int32_t n, int64_t T, const KsSequence* q, Fill fill, Launch launch) {
  if (n < 1 || n > 2 || !q) return fail(KS_EINVAL, "%s: one or two sequences", who);
  Seq s[2];
  int m = 0;
  int64_t rows = 0;
  for (int k = 0; k < n; ++k) {
    if (!q[k].cell || !q[k].in || !q[k].out0) return fail(KS_EINVAL, "%s: null argument", who);
    if (T < 0 || q[k].M < 0) return fail(KS_EINVAL, "%s: negative size", who);
    if (T == 0 || q[k].M == 0) continue;
    s[m] = {q[k].M, q[k].in, nullptr, 0, nullptr, q[k].h0, q[k].c0, q[k].fresh, q[k].saved, q[k].out0, q[k].out1, q[k].dh0, q[k].dc0};
    const int rc = fill(q[k], s[m]);
    if (rc != KS_OK) return rc;
    rows = s[m].M > rows ? s[m].M : rows;
    ++m;
  }
  if (m == 0) return KS_OK;
  if ((rows + kSeqRows - 1) / kSeqRows > 0x7fffffff || T > 0x7fffffff) return fail(KS_ELIMIT, "%s: too many rows or steps", who);
  if (m == 1) s[1] = s[0];
  launch(s, m, (rows + kSeqRows - 1) / kSeqRows);
  return check_launch(who);
}

extern "C" int ks_gru_sequences_forward(ks_stream_t stream, int32_t n, int64_t T, const KsSequence* q) {
  const char* who = "ks_gru_sequence_forward";
  bool bf[2] = {};
  int m = 0;
  auto fill = [&](const KsSequence& c, Seq& s) -> int {
    const KsGru* g = (const KsGru*)c.cell;
    if (!c.h0) return fail(KS_EINVAL, "%s: null argument", who);
    const void* Wt;
    int ldwt;
    if (!gru_seq_weights(g, &s.W, &s.ldw, &Wt, &ldwt, &bf[m++])) return fail(KS_EINVAL, "%s: needs a cell of hidden size %d", who, kSeqH);
    if (T > 1 && c.out0 == c.h0) return fail(KS_EINVAL, "%s: the output may alias the initial state only for T = 1", who);
    if (m == 2 && bf[0] != bf[1]) return fail(KS_EINVAL, "%s: two layers of one precision", who);
    s.bias_n = g->bn();
    return KS_OK;
  };
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) {
    const int groups = seq_groups(T, sets);
    hipLaunchKernelGGL(bf[0] ? gru_seq_forward_kernel<true> : gru_seq_forward_kernel<false>, dim3((unsigned)((sets + groups - 1) / groups), (unsigned)count),
                       dim3(64 * kSeqWaves), 0, (hipStream_t)stream, (int)T, groups, s[0], s[1]);
  });
}

extern "C" int ks_gru_sequences_backward(ks_stream_t stream, int32_t n, int64_t T, const KsSequence* q) {
  const char* who = "ks_gru_sequence_backward";
  bool bf[2] = {};
  int m = 0;
  auto fill = [&](const KsSequence& c, Seq& s) -> int {
    const void* W;
    int ldw;
    if (!c.saved || !c.out1) return fail(KS_EINVAL, "%s: null argument", who);
    if (!gru_seq_weights((const KsGru*)c.cell, &W, &ldw, &s.W, &s.ldw, &bf[m++])) return fail(KS_EINVAL, "%s: needs a cell of hidden size %d", who, kSeqH);
    if (!s.W) return fail(KS_EINVAL, "%s: ks_gru_train_init has not run", who);
    if (m == 2 && bf[0] != bf[1]) return fail(KS_EINVAL, "%s: two layers of one precision", who);
    return KS_OK;
  };
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) {
    hipLaunchKernelGGL(bf[0] ? gru_seq_backward_kernel<true> : gru_seq_backward_kernel<false>, dim3((unsigned)sets, (unsigned)count), dim3(64 * kSeqWaves), 0,
                       (hipStream_t)stream, (int)T, s[0], s[1]);
  });
}

extern "C" int ks_gru_sequence_forward(const KsGru* g, ks_stream_t stream, int64_t T, int64_t M, const float* gi, const float* h0,
                                       const uint8_t* fresh, float* hs, float* saved) {
  const KsSequence q = {g, M, gi, h0, nullptr, fresh, saved, hs, nullptr, nullptr, nullptr};
  return ks_gru_sequences_forward(stream, 1, T, &q);
}

extern "C" int ks_gru_sequence_backward(const KsGru* g, ks_stream_t stream, int64_t T, int64_t M, const float* dH, const float* saved,
                                        const uint8_t* fresh, float* d_gi, float* d_gh, float* dh0) {
  const KsSequence q = {g, M, dH, nullptr, nullptr, fresh, const_cast<float*>(saved), d_gi, d_gh, dh0, nullptr};
  return ks_gru_sequences_backward(stream, 1, T, &q);
}

extern "C" int64_t ks_gru_workspace_bytes(const KsGru* g, int64_t M) {
  if (!g || M < 0) return -1;
  const int64_t gates = up256(M * 3 * g->H * 4);
  return 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M)) + up256(ks_mlp_workspace_bytes(g->proj_h, M));
}

extern "C" int ks_gru_forward(const KsGru* g, ks_stream_t stream, int64_t M, const float* x, const float* h_in,
                              const uint8_t* fresh, float* h_out, void* workspace) {
  if (!g || !x || !h_in || !h_out) return fail(KS_EINVAL, "ks_gru_forward: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_gru_forward: negative row count");
  if (M == 0) return KS_OK;
  if (!workspace) return fail(KS_EINVAL, "ks_gru_forward: workspace is required");
  const int64_t gates = up256(M * 3 * g->H * 4);
  char* w = (char*)workspace;
  float* gi = (float*)w;
  float* gh = (float*)(w + gates);
  void* wi = w + 2 * gates;
  void* wh = w + 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M));
  int rc = ks_mlp_forward(g->proj_i, stream, M, x, gi, wi);
  if (rc != KS_OK) return rc;
  // one step of the sequence kernel where it applies: a rollout's steps and the replay of its trajectory then give the same bits
  if (ks_gru_sequence_supported(g)) return ks_gru_sequence_forward(g, stream, 1, M, gi, h_in, fresh, h_out, nullptr);
  rc = ks_mlp_forward(g->proj_h, stream, M, h_in, gh, wh);
  if (rc != KS_OK) return rc;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_gru_forward: too many elements");
  hipLaunchKernelGGL(gru_gate_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, gi, gh, h_in,
                     g->bn(), fresh, h_out);
  return check_launch("ks_gru_forward");
}

extern "C" int ks_gru_train_init(KsGru* g) {
  if (!g) return fail(KS_EINVAL, "ks_gru_train_init: null handle");
  int rc = ks_mlp_train_init(g->proj_i);
  if (rc == KS_OK) rc = ks_mlp_train_init(g->proj_h);
  // the hidden projection's bias is (0, 0, b_n): only its candidate part is a parameter of the cell
  if (rc == KS_OK) rc = ks_mlp_freeze_bias_prefix(g->proj_h, 0, 2 * g->H);
  if (rc == KS_OK) g->bias_nt = mlp_peek_bias(g->proj_h, 0) + 2 * g->H;
  return rc;
}

extern "C" int ks_gru_projections(KsGru* g, KsMlp** input_projection, KsMlp** hidden_projection) {
  if (!g || !input_projection || !hidden_projection) return fail(KS_EINVAL, "ks_gru_projections: null argument");
  *input_projection = g->proj_i;
  *hidden_projection = g->proj_h;
  return KS_OK;
}

extern "C" int ks_gru_grad_sqnorm(const KsGru* g, ks_stream_t stream, double* acc) {
  if (!g || !acc) return fail(KS_EINVAL, "ks_gru_grad_sqnorm: null argument");
  const KsMlp* nets[] = {g->proj_i, g->proj_h};
  return ks_mlps_grad_sqnorm(nets, 2, stream, acc);
}

extern "C" int ks_gru_adam_step(KsGru* g, ks_stream_t stream, const KsAdamParams* params, const double* sqnorm) {
  if (!g || !g->bias_nt) return fail(KS_EINVAL, "ks_gru_adam_step: call ks_gru_train_init first");
  KsMlp* nets[] = {g->proj_i, g->proj_h};
  return ks_mlps_adam_step(nets, 2, stream, params, sqnorm);
}

extern "C" int ks_gru_train_forward(const KsGru* g, ks_stream_t stream, int64_t M, const float* x, const float* h_in,
                                    const uint8_t* fresh, float* h_out, float* saved, void* workspace) {
  if (!g || !x || !h_in || !h_out || !saved) return fail(KS_EINVAL, "ks_gru_train_forward: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_gru_train_forward: negative row count");
  if (M == 0) return KS_OK;
  if (!workspace) return fail(KS_EINVAL, "ks_gru_train_forward: workspace is required");
  const int64_t gates = up256(M * 3 * g->H * 4);
  char* w = (char*)workspace;
  float* gi = (float*)w;
  float* gh = (float*)(w + gates);
  void* wi = w + 2 * gates;
  void* wh = w + 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M));
  int rc = ks_mlp_forward(g->proj_i, stream, M, x, gi, wi);
  if (rc != KS_OK) return rc;
  // one step of the sequence kernel where it applies: a rollout's steps and the replay of its trajectory then give the same bits
  if (ks_gru_sequence_supported(g)) return ks_gru_sequence_forward(g, stream, 1, M, gi, h_in, fresh, h_out, saved);
  rc = ks_mlp_forward(g->proj_h, stream, M, h_in, gh, wh);
  if (rc != KS_OK) return rc;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_gru_train_forward: too many elements");
  hipLaunchKernelGGL(gru_gate_train_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, gi, gh, h_in,
                     g->bn(), fresh, h_out, saved);
  return check_launch("ks_gru_train_forward");
}

extern "C" int64_t ks_gru_backward_workspace_bytes(const KsGru* g, int64_t M) {
  if (!g || M < 0) return -1;
  return ks_mlp_train_workspace_bytes(g->proj_h, M);
}

extern "C" int ks_gru_backward_step(KsGru* g, ks_stream_t stream, int64_t M, const float* dh_out, const float* saved,
                                    const uint8_t* fresh, float* d_gi, float* d_gh, float* dh_in, void* workspace) {
  if (!g || !dh_out || !saved || !d_gi || !d_gh || !dh_in || !workspace) return fail(KS_EINVAL, "ks_gru_backward_step: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_gru_backward_step: negative row count");
  if (M == 0) return KS_OK;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_gru_backward_step: too many elements");
  hipLaunchKernelGGL(gru_gate_backward_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, dh_out, saved, fresh,
                     d_gi, d_gh, dh_in);
  int rc = check_launch("ks_gru_backward_step");
  if (rc != KS_OK) return rc;
  // dh_in += d_gh W_hh, except across an episode boundary
  return ks_mlp_train_backward_dx(g->proj_h, stream, M, nullptr, d_gh, dh_in, 0, 1, fresh, workspace);
}

struct KsLstm {
  int I, H;
  KsMlp *proj_i, *proj_h;
};

extern "C" int ks_lstm_create(const KsLstmDesc* d, KsLstm** out) {
  if (!d || !out) return fail(KS_EINVAL, "ks_lstm_create: null argument");
  if (d->input_size < 1 || d->hidden_size < 1 || d->hidden_size > 16384) return fail(KS_EINVAL, "ks_lstm_create: bad sizes %d -> %d", d->input_size, d->hidden_size);
  if (!d->weight_ih || !d->weight_hh) return fail(KS_EINVAL, "ks_lstm_create: weights are required");
  const int H = d->hidden_size, I = d->input_size;
  std::vector<float> zero(4 * (size_t)H, 0.f);
  KsLstm* g = new KsLstm{I, H, nullptr, nullptr};
  KsMlpDesc md = {};
  md.n_layers = 1; md.activation = KS_ACT_NONE; md.dtype = d->dtype;
  md.dims[0] = I; md.dims[1] = 4 * H; md.weights[0] = d->weight_ih; md.biases[0] = d->bias ? d->bias : zero.data();
  int rc = ks_mlp_create(&md, &g->proj_i);
  if (rc == KS_OK) {
    md.dims[0] = H; md.weights[0] = d->weight_hh; md.biases[0] = zero.data();
    rc = ks_mlp_create(&md, &g->proj_h);
  }
  if (rc != KS_OK) { ks_lstm_destroy(g); return rc; }
  *out = g;
  return KS_OK;
}

extern "C" int ks_lstm_destroy(KsLstm* g) {
  if (!g) return KS_OK;
  ks_mlp_destroy(g->proj_i);
  ks_mlp_destroy(g->proj_h);
  delete g;
  return KS_OK;
}

extern "C" int64_t ks_lstm_workspace_bytes(const KsLstm* g, int64_t M) {
  if (!g || M < 0) return -1;
  const int64_t gates = up256(M * 4 * g->H * 4);
  return 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M)) + up256(ks_mlp_workspace_bytes(g->proj_h, M));
}

extern "C" int ks_lstm_forward(const KsLstm* g, ks_stream_t stream, int64_t M, const float* x, const float* h_in,
                               const float* c_in, const uint8_t* fresh, float* h_out, float* c_out, void* workspace) {
  if (!g || !x || !h_in || !c_in || !h_out || !c_out) return fail(KS_EINVAL, "ks_lstm_forward: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_lstm_forward: negative row count");
  if (M == 0) return KS_OK;
  if (!workspace) return fail(KS_EINVAL, "ks_lstm_forward: workspace is required");
  const int64_t gates = up256(M * 4 * g->H * 4);
  char* w = (char*)workspace;
  float* gi = (float*)w;
  float* gh = (float*)(w + gates);
  void* wi = w + 2 * gates;
  void* wh = w + 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M));
  int rc = ks_mlp_forward(g->proj_i, stream, M, x, gi, wi);
  if (rc != KS_OK) return rc;
  // one step of the sequence kernel where it applies: a rollout's steps and the replay of its trajectory then give the same bits
  if (ks_lstm_sequence_supported(g)) return ks_lstm_sequence_forward(g, stream, 1, M, gi, h_in, c_in, fresh, h_out, c_out, nullptr);
  rc = ks_mlp_forward(g->proj_h, stream, M, h_in, gh, wh);
  if (rc != KS_OK) return rc;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_lstm_forward: too many elements");
  hipLaunchKernelGGL(lstm_gate_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, gi, gh, c_in, fresh,
                     h_out, c_out);
  return check_launch("ks_lstm_forward");
}

// whether the one-launch sequence kernels cover this cell: fp32, hidden size 128
static bool lstm_seq_weights(const KsLstm* g, const float** W, int* ldw, const float** Wt, int* ldwt) {
  const void *w = nullptr, *wt = nullptr;
  int np = 0, kp = 0, dt = 0;
  if (!g || g->H != kSeqH) return false;
  if (mlp_peek_layer(g->proj_h, 0, &w, &wt, &np, &kp, &dt) != KS_OK) return false;
  if (dt != KS_MLP_F32 || np != 4 * kSeqH || kp < kSeqH || (kp & 3)) return false;
  *W = (const float*)w; *ldw = kp;
  *Wt = (const float*)wt; *ldwt = np;
  return w != nullptr;
}

extern "C" int ks_lstm_sequence_supported(const KsLstm* g) {
  const float *W, *Wt;
  int a, b;
  return lstm_seq_weights(g, &W, &a, &Wt, &b) ? 1 : 0;
}

extern "C" int ks_lstm_sequences_forward(ks_stream_t stream, int32_t n, int64_t T, const KsSequence* q) {
  const char* who = "ks_lstm_sequence_forward";
  auto fill = [&](const KsSequence& c, Seq& s) -> int {
    const float *W, *Wt;
    int ldwt;
    if (!c.h0 || !c.c0) return fail(KS_EINVAL, "%s: null argument", who);
    if (!lstm_seq_weights((const KsLstm*)c.cell, &W, &s.ldw, &Wt, &ldwt)) return fail(KS_EINVAL, "%s: needs an fp32 cell of hidden size %d", who, kSeqH);
    if (T > 1 && (c.out0 == c.h0 || (c.out1 && c.out1 == c.c0))) return fail(KS_EINVAL, "%s: outputs may alias the initial state only for T = 1", who);
    s.W = W;
    return KS_OK;
  };
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) {
    const int groups = seq_groups(T, sets);
    const dim3 grid((unsigned)((sets + groups - 1) / groups), (unsigned)count);
    auto run = [&](dim3 grid, const Seq& first, const Seq& second) {
      const bool cell = first.out1 != nullptr, save = first.saved != nullptr;
      hipLaunchKernelGGL(cell ? (save ? lstm_seq_forward_kernel<true, true> : lstm_seq_forward_kernel<true, false>)
                              : (save ? lstm_seq_forward_kernel<false, true> : lstm_seq_forward_kernel<false, false>),
                         grid, dim3(64 * kSeqWaves), 0, (hipStream_t)stream, (int)T, groups, first, second);
    };
    if (count == 2 && (!s[0].out1 != !s[1].out1 || !s[0].saved != !s[1].saved)) {  // a kernel writes the same outputs for both of its layers
      run(dim3(grid.x), s[0], s[0]);
      run(dim3(grid.x), s[1], s[1]);
    } else {
      run(grid, s[0], s[1]);
    }
  });
}

extern "C" int ks_lstm_sequences_backward(ks_stream_t stream, int32_t n, int64_t T, const KsSequence* q) {
  const char* who = "ks_lstm_sequence_backward";
  auto fill = [&](const KsSequence& c, Seq& s) -> int {
    const float *W, *Wt;
    int ldw;
    if (!c.saved) return fail(KS_EINVAL, "%s: null argument", who);
    if (!lstm_seq_weights((const KsLstm*)c.cell, &W, &ldw, &Wt, &s.ldw)) return fail(KS_EINVAL, "%s: needs an fp32 cell of hidden size %d", who, kSeqH);
    if (!Wt) return fail(KS_EINVAL, "%s: ks_lstm_train_init has not run", who);
    s.W = Wt;
    return KS_OK;
  };
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) {
    hipLaunchKernelGGL(lstm_seq_backward_kernel, dim3((unsigned)sets, (unsigned)count), dim3(64 * kSeqWaves), 0, (hipStream_t)stream, (int)T, s[0], s[1]);
  });
}

extern "C" int ks_lstm_sequence_forward(const KsLstm* g, ks_stream_t stream, int64_t T, int64_t M, const float* gi, const float* h0,
                                        const float* c0, const uint8_t* fresh, float* hs, float* cs, float* saved) {
  const KsSequence q = {g, M, gi, h0, c0, fresh, saved, hs, cs, nullptr, nullptr};
  return ks_lstm_sequences_forward(stream, 1, T, &q);
}

extern "C" int ks_lstm_sequence_backward(const KsLstm* g, ks_stream_t stream, int64_t T, int64_t M, const float* dH, const float* saved,
                                         const uint8_t* fresh, float* d_g, float* dh0, float* dc0) {
  const KsSequence q = {g, M, dH, nullptr, nullptr, fresh, const_cast<float*>(saved), d_g, nullptr, dh0, dc0};
  return ks_lstm_sequences_backward(stream, 1, T, &q);
}

extern "C" int ks_lstm_train_init(KsLstm* g) {
  if (!g) return fail(KS_EINVAL, "ks_lstm_train_init: null handle");
  int rc = ks_mlp_train_init(g->proj_i);
  if (rc == KS_OK) rc = ks_mlp_train_init(g->proj_h);
  // the cell has one bias, carried by the input projection: the hidden projection's stays zero
  if (rc == KS_OK) rc = ks_mlp_freeze_bias_prefix(g->proj_h, 0, 4 * g->H);
  return rc;
}

extern "C" int ks_lstm_projections(KsLstm* g, KsMlp** input_projection, KsMlp** hidden_projection) {
  if (!g || !input_projection || !hidden_projection) return fail(KS_EINVAL, "ks_lstm_projections: null argument");
  *input_projection = g->proj_i;
  *hidden_projection = g->proj_h;
  return KS_OK;
}

extern "C" int ks_lstm_train_forward(const KsLstm* g, ks_stream_t stream, int64_t M, const float* x, const float* h_in,
                                     const float* c_in, const uint8_t* fresh, float* h_out, float* c_out, float* saved,
                                     void* workspace) {
  if (!g || !x || !h_in || !c_in || !h_out || !c_out || !saved) return fail(KS_EINVAL, "ks_lstm_train_forward: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_lstm_train_forward: negative row count");
  if (M == 0) return KS_OK;
  if (!workspace) return fail(KS_EINVAL, "ks_lstm_train_forward: workspace is required");
  const int64_t gates = up256(M * 4 * g->H * 4);
  char* w = (char*)workspace;
  float* gi = (float*)w;
  float* gh = (float*)(w + gates);
  void* wi = w + 2 * gates;
  void* wh = w + 2 * gates + up256(ks_mlp_workspace_bytes(g->proj_i, M));
  int rc = ks_mlp_forward(g->proj_i, stream, M, x, gi, wi);
  if (rc != KS_OK) return rc;
  if (ks_lstm_sequence_supported(g)) return ks_lstm_sequence_forward(g, stream, 1, M, gi, h_in, c_in, fresh, h_out, c_out, saved);
  rc = ks_mlp_forward(g->proj_h, stream, M, h_in, gh, wh);
  if (rc != KS_OK) return rc;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_lstm_train_forward: too many elements");
  hipLaunchKernelGGL(lstm_gate_train_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, gi, gh, h_in, c_in,
                     fresh, h_out, c_out, saved);
  return check_launch("ks_lstm_train_forward");
}

extern "C" int64_t ks_lstm_backward_workspace_bytes(const KsLstm* g, int64_t M) {
  if (!g || M < 0) return -1;
  return ks_mlp_train_workspace_bytes(g->proj_h, M);
}

extern "C" int ks_lstm_backward_step(KsLstm* g, ks_stream_t stream, int64_t M, const float* dh_out, const float* dc_out,
                                     const float* saved, const uint8_t* fresh, float* d_g, float* dh_in, float* dc_in,
                                     void* workspace) {
  if (!g || !dh_out || !dc_out || !saved || !d_g || !dh_in || !dc_in || !workspace) return fail(KS_EINVAL, "ks_lstm_backward_step: null argument");
  if (M < 0) return fail(KS_EINVAL, "ks_lstm_backward_step: negative row count");
  if (M == 0) return KS_OK;
  const int64_t n = M * g->H, grid = (n + 255) / 256;
  if (grid > 0x7fffffff) return fail(KS_ELIMIT, "ks_lstm_backward_step: too many elements");
  hipLaunchKernelGGL(lstm_gate_backward_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, M, g->H, dh_out, dc_out,
                     saved, fresh, d_g, dh_in, dc_in);
  const int rc = check_launch("ks_lstm_backward_step");
  if (rc != KS_OK) return rc;
  // dh_in = d_g W_hh, except across an episode boundary
  return ks_mlp_train_backward_dx(g->proj_h, stream, M, nullptr, d_g, dh_in, 0, 1, fresh, workspace);
}

extern "C" int ks_lstm_grad_sqnorm(const KsLstm* g, ks_stream_t stream, double* acc) {
  if (!g || !acc) return fail(KS_EINVAL, "ks_lstm_grad_sqnorm: null argument");
  const KsMlp* nets[] = {g->proj_i, g->proj_h};
  return ks_mlps_grad_sqnorm(nets, 2, stream, acc);
}

extern "C" int ks_lstm_adam_step(KsLstm* g, ks_stream_t stream, const KsAdamParams* params, const double* sqnorm) {
  if (!g) return fail(KS_EINVAL, "ks_lstm_adam_step: null handle");
  KsMlp* nets[] = {g->proj_i, g->proj_h};
  return ks_mlps_adam_step(nets, 2, stream, params, sqnorm);
}
