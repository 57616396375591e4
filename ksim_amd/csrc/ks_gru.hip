// GRU and LSTM cells for recurrent policies in the rollout, and the GRU's backward pass through time.  The two gate projections are plain linear
// layers and run through the MLP entry points (matrix cores for bf16); one streaming kernel then combines the gates.
#include "ks_common.h"
#include "ks_cut.h"

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

// What the gate gradients of an LSTM step take from its activations alone: factors of the gradient that reaches the cell state (the hidden state for the
// output gate), and what of the latter reaches the former.
struct LstmSlopes {
  float i, f, g, o, cell, keep;
  __device__ __forceinline__ void make(float si, float sf, float tg, float so, float tc, float c) {
    i = tg * si * (1.f - si);
    f = c * sf * (1.f - sf);
    g = si * (1.f - tg * tg);
    o = tc * so * (1.f - so);
    cell = so * (1.f - tc * tc);
    keep = sf;
  }
  // gate gradients i | f | g | o from those reaching h' and c'; returns that of the cell state
  __device__ __forceinline__ float gates(float dh, float dc, float (&out)[4]) const {
    const float dct = fmaf(dh, cell, dc);
    out[0] = dct * i; out[1] = dct * f; out[2] = dct * g; out[3] = dh * o;
    return dct;
  }
};

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
  LstmSlopes slope;
  slope.make(sv[j], sv[H + j], sv[2 * H + j], sv[3 * H + j], sv[4 * H + j], sv[5 * H + j]);
  float gate[4];
  const float dct = slope.gates(dh_out[idx], dc_out[idx], gate);
  float* a = d_g + m * 4 * H;
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k * H + j] = gate[k];
  dc_in[idx] = f ? 0.f : dct * slope.keep;
  dh_in[idx] = 0.f;
}

// ---------------------------------------------------------------- a whole trajectory of one LSTM layer in one launch
// The step-by-step path costs two GEMM launches and a gate kernel per step, layer and network: a minibatch of 100 control steps
// is thousands of launches of a few microseconds each.  Here a workgroup of eight wavefronts owns 4 or 8 rows (envs) for all T
// steps, so that a minibatch of a thousand rows is one workgroup per CU.  A wavefront's 16 units keep their slice of W_hh for the whole sequence, cut
// in three bf16 parts (ks_cut.h): two parts in registers, the third in LDS.  A step is the products of the cut state with it (CutTile), the gate
// arithmetic of one or two (unit, row) per lane, and one barrier.  fp32 cells of hidden size 128.
// On v_mfma_f32_4x4x1, four rows a workgroup, a step's products took 2048 cycles for four rows; cut they take 1536 for four and 2560 for eight, and
// a sum rounds no more (the state after 100 steps is 1.8e-7 from 64 bits as it was, the gate gradients 1.6e-7, of 1.8e-7).  Two layers (blockIdx.y), 100 steps, us:
//   rows a layer:                     64         360 (60 steps)   1024
//   forward, activations kept     154 -> 134   112 -> 103       400 -> 340
//   forward, not kept             135 -> 132                    327 -> 268
//   backward                      139 -> 118    99 -> 94        348 -> 296
// 24 steps of 512 rows, every CU at work once: 53 -> 50, not kept 44.7 -> 46.7 (the weights' cut), backward 54 -> 52.
// With activations kept, 1024 rows move 1.2 GB, 240 us at the rate of a large copy.  What is left: issue, since only two vector instructions hide under
// a 16-cycle matrix instruction (eight rows 5100 cycles a step, of which products 2560), the state's way through LDS at the head of a step (400), and the
// clock, which falls to 1.9 GHz with every CU at work.  Also built: two sets of four rows half a step apart, one's gates between the other's products
// (not kept 300 us: nothing more hides, and four rows need 1.2 times the products); the backward product split over the gate rows instead
// of over the units of dh (175 us of 119 for 64 rows: eight times the tiles' ends, and partial sums to add); all weights requested before the first is cut (the
// same); a copy of the steps for operands that cannot overflow, without the check for it (64 rows 129, not kept 126, 1024 rows kept 378: the copies' registers).
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

// tanh x = 1 - 2 / (e^2x + 1) on v_exp_f32 and v_rcp_f32; it saturates correctly (e^y = inf gives 1, e^y = 0 gives -1)
__device__ __forceinline__ float seq_tanh(float x) { return 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f); }

// Barrier for data that the wavefronts of a workgroup hand each other through LDS only: it waits for this wavefront's LDS
// traffic, not for its global loads and stores.  __syncthreads() would also drain the step's stores (and the loads fetched
// ahead for the next step) before every barrier, a memory round trip per step of the sequence.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The LSTM kernels' way in and out of memory: a step's inputs are requested a step ahead of their use, and where the activations are kept, the nine
// results a step leave between the matrix instructions of the next: together at a step's end they hold the CU's wavefronts up at once.  A store or load
// under a condition makes the compiler wait for the step's stores before the next step (loads and stores are counted together and waited for in order).
// Hence no conditions: the outputs that a launch has are template arguments, rows past the batch repeat the last row and store its values once more, the
// last step requests its own inputs again, and nothing is pending where the loop is entered.
__device__ __forceinline__ void seq_loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)
// GRU: where hidden unit u of a row sits in the LDS copy of the state: unit u = 16 q + b is register q of block b (see the forward
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

constexpr int kLstmStateLd = kSeqH + 8;  // 16-bit entries of a row of the state; the padding puts neighbouring rows on different banks
constexpr int lstm_forward_lds(int rows) { return kSeqWaves * 16 * 64 * 16 + 2 * 3 * rows * kLstmStateLd * 2; }

constexpr float kLog2e = 1.44269504f;
constexpr int kStepRows = 16;
typedef f32x4 f32x4_any __attribute__((aligned(4)));  // a state lies where the caller has it: one load all the same

// holds a value, and with it the arithmetic that follows, to its place between two matrix instructions
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }

// A 16-column tile of the product of R rows with fp32 weights, both cut in three (cut_bf16).  The parts are rows of the A operand, which has sixteen:
//   R = 8: rows 0..7 and 8..15 of `a` are first and second parts, of `b` third and again first parts: five instructions per 32 k.
//   R = 4: rows 0..3, 4..7, 8..11, 12..15 of `a` are first, second, third and again first parts, `b` is `a` without the latter two: three instructions per 32 k.
// Eight of the nine products, all but the one of the third parts, below 2^-32 of the result.  With s(i, j) the sum of the products of the state's part i with
// the weights' part j in order of k, and s(i, 12) of both smaller parts' together, an entry is s(0, 0) + ((s(0, 12) + (s(2, 0) + s(2, 1))) + (s(1, 0) + s(1, 12))):
// the largest products by themselves, so that a sum of one term, or of one among zeros, is rounded once.  Its bits do not depend on R, nor on other rows.
//   SPLIT: s(i, 12) is s(i, 1) + s(i, 2), so that with R = 4 the product of the third parts is left out at the end and `b` is not needed: for a single tile over
//   a long reduction, where masking `a` costs more than the additions.
// Without the state's third times the weights' second parts, and with the smaller products in the sum of the largest, eight rows took four instructions per 32 k (1024
// rows 240 us instead of 268, kept 325 instead of 340, backward 280 instead of 296), but a single product was up to 3.5 times 2^-24 off, instead of once.
template <int R, bool SPLIT>
struct CutTile {
  static constexpr int kSteps = R == 8 ? 5 : 3;  // matrix instructions per 32 k
  f32x4 a0, a1, a2, b0, b1;                      // the sums over `a` and `b` by the weights' parts; without SPLIT a1 has those of a2 as well
  __device__ __forceinline__ void clear() { a0 = a1 = a2 = b0 = b1 = f32x4{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ void add(int step, bf16x8 a, bf16x8 b, bf16x8 w0, bf16x8 w1, bf16x8 w2) {
    f32x4& to = SPLIT ? a2 : a1;
    if (step == 0) a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w0, a0, 0, 0, 0);
    if (step == kSteps / 2) a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w1, a1, 0, 0, 0);
    if (step == kSteps - 1) to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(R == 8 || SPLIT ? a : b, w2, to, 0, 0, 0);
    if (R == 8 && step == 1) b0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, w0, b0, 0, 0, 0);
    if (R == 8 && step == 3) b1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, w1, b1, 0, 0, 0);
  }
  // which of a lane's sums count, as factors (0 or 1): R = 8 lanes 32..63 and 0..31, R = 4 lane rows 1 to 3 and 0 to 2; `kept` R = 4's lane rows 0 and 1
  struct Lanes {
    float upper, lower, kept;
    __device__ __forceinline__ explicit Lanes(int lane) : upper(lane >= 4 * R ? 1.f : 0.f), lower(lane < (R == 8 ? 32 : 48) ? 1.f : 0.f), kept(lane < 32 ? 1.f : 0.f) {}
  };
  // In kRows pieces, which stand between matrix instructions: lane l gets column l % 16 of rows seq_row<R>(l) + q in out[q].  `t` carries values from one
  // piece to the next.  The swaps' operands come out of vector instructions, never straight out of a matrix instruction: nothing inserts that one's wait
  // states into the asm.  (The builtins give the same result twice where both are used.)
  static constexpr int kRows = R == 8 ? 8 : 4;
  __device__ __forceinline__ void rows(int piece, Lanes& lanes, float (&t)[4], float (&out)[R / 4]) const {
    constexpr int kEach = R == 8 ? 1 : 2, kSwap = 4 / kEach;
    if (piece < kSwap) {
      pin(lanes.upper);
      pin(lanes.lower);
#pragma unroll
      for (int i = kEach * piece; i < kEach * piece + kEach; ++i) {
        if constexpr (R == 8) t[i] = fmaf(b0[i] + b1[i], lanes.lower, fmaf(a0[i], lanes.upper, SPLIT ? a1[i] + a2[i] : a1[i]));
        else if constexpr (!SPLIT) t[i] = fmaf(a1[i], lanes.lower, a0[i] * lanes.upper);
        else t[i] = lanes.lower != 0.f ? fmaf(a0[i], lanes.upper, fmaf(a2[i], lanes.kept, a1[i])) : a0[i];  // whose infinities have to arrive as such
      }
    }
    if constexpr (R == 8) {
      if (piece == kSwap)
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]));
      if (piece == kSwap + 1) t[0] += t[2], t[1] += t[3];
      if (piece == kSwap + 2) {  // the first parts' sums of the lane's rows
        const bool upper = (threadIdx.x & 32) != 0;
        t[2] = upper ? b0[2] : a0[0], t[3] = upper ? b0[3] : a0[1];
      }
      if (piece == kSwap + 3) out[0] = t[2] + t[0], out[1] = t[3] + t[1];
    } else {
      if (piece == kSwap)  // register i of lane row q changes places with register q of lane row i
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1\n\t"
                     "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1"
                     : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]));
      if (piece == kSwap + 1) out[0] = t[3] + ((t[0] + t[2]) + t[1]);
    }
  }
  // for the lane's rows, from the sums of `a`'s rows over a matrix instruction (its wait states included), those of the first parts
  static __device__ __forceinline__ void first_rows(const f32x4& sum, float (&p)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = sum[i];
    asm volatile("s_nop 15\n\ts_nop 15\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
    if (R == 4) asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(p[0]), "+v"(p[1]));
  }
};
template <int R>
__device__ __forceinline__ int seq_row(int lane) { return R == 8 ? 4 * ((lane >> 4) & 1) + 2 * (lane >> 5) : lane >> 4; }
// the operands' rows (CutTile) out of R first, R second and R third parts
template <int R>
__device__ __forceinline__ bf16x8 get_a(const unsigned short* rows, int ld, int lane, int k) {
  const int row = lane & 15;
  return *reinterpret_cast<const bf16x8*>(rows + (R == 8 || row < 12 ? row : row - 12) * ld + k);
}
template <int R>
__device__ __forceinline__ bf16x8 get_b(const unsigned short* rows, int ld, int lane, int k, bf16x8 a) {
  const int row = lane & 15;
  if constexpr (R == 8) return *reinterpret_cast<const bf16x8*>(rows + (row < 8 ? 16 + row : row - 8) * ld + k);
  else return (row & 8) ? bf16x8{} : a;
}
// the entry `bytes` after base[entries], whose address is the same for every lane
template <typename T>
__device__ __forceinline__ T& at(T* base, int64_t entries, unsigned bytes) {
  typedef typename std::conditional<std::is_const<T>::value, const char, char>::type Byte;
  return *reinterpret_cast<T*>(reinterpret_cast<Byte*>(base + entries) + bytes);
}

template <int R, bool CELL, bool SAVE>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lstm_seq_forward_kernel(int T, int groups, Seq first, Seq second) {
  constexpr int H = kSeqH, KB = H / 32, V = R / 4;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ gi = s.in;
  const float* __restrict__ W = (const float*)s.W;
  const int ldw = s.ldw;
  const float *h0 = s.h0, *c0 = s.c0;
  // without episode starts a byte of the inputs is read in the flag's place and masked away
  const uint8_t* __restrict__ fresh = s.fresh ? s.fresh : (const uint8_t*)s.in;
  const unsigned fresh_mask = s.fresh ? 0xffu : 0u;
  float *hs = s.out0, *cs = s.out1;
  float* __restrict__ saved = s.saved;
  if ((int64_t)blockIdx.x * groups * R >= M) return;  // the other layer of the launch has more rows
  extern __shared__ __attribute__((aligned(16))) unsigned char seq_lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int unit = 16 * wave + (lane & 15), row = seq_row<R>(lane), kq = 8 * (lane >> 4);
  u32x4* w2 = reinterpret_cast<u32x4*>(seq_lds) + wave * 16 * 64 + lane;  // fragment (tile, k block) 64 entries on
  typedef unsigned short State[3 * R][kLstmStateLd];
  State* sh = reinterpret_cast<State*>(seq_lds + kSeqWaves * 16 * 64 * 16);  // of even and odd steps
  // The tiles of a wavefront are its 16 units' forget, cell, input and output gates, in this order: all but the last one's arithmetic finds
  // matrix instructions to stand between.  B operand: column lane % 16 is the unit, rows k = 32 kb + 8 (lane / 16) + 0..7.
  constexpr int kGate[4] = {1, 2, 0, 3};
  bf16x8 w0[4][KB], w1[4][KB];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const float* src = W + (int64_t)(kGate[n] * H + unit) * ldw + kq;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const float4 lo = *reinterpret_cast<const float4*>(src + 32 * kb), hi = *reinterpret_cast<const float4*>(src + 32 * kb + 4);
      const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      u32x4 part[3];
      cut_bf16<3>(v, part);
      w0[n][kb] = __builtin_bit_cast(bf16x8, part[0]);
      w1[n][kb] = __builtin_bit_cast(bf16x8, part[1]);
      w2[(n * KB + kb) * 64] = part[2];
    }
  }
  // A workgroup takes `groups` sets of R rows one after the other with the same registers of weights: a few steps over
  // thousands of rows would otherwise fetch and cut the 256 KB of W_hh once per set (two layers, 4096 rows x 2 steps 51.5 us of 38, 8192 x 8 215 of 179).
  for (int grp = 0; grp < groups; ++grp) {
  const int64_t r0 = ((int64_t)blockIdx.x * groups + grp) * R;
  if (r0 >= M) break;  // the same for every thread of the workgroup
  // the lane's rows and their bytes into a step's states, inputs and kept activations; rows past the batch repeat the last one and store its values once more
  unsigned jr[V], oh[V], og[V], ov[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    jr[q] = r0 + row + q < M ? row + q : (unsigned)(M - 1 - r0);
    oh[q] = (jr[q] * H + unit) * 4;
    og[q] = (jr[q] * 4 * H + unit) * 4;
    ov[q] = (jr[q] * 7 * H + unit) * 4;
  }
  if (grp > 0) __syncthreads();  // the previous set's last read of the state buffers is over
  // c, h: the states this lane's (unit, rows) leave a step with, g: its inputs by gate, requested a step ahead, v: its activations i | f | g | o | tanh(c')
  // and the states it started from, which are zero in an episode's first step
  float c[V], h[V], g[V][4], v[V][7];
  unsigned flag[V];
  auto load = [&](int t, int gate, int q) __attribute__((always_inline)) {
    const int64_t o = (int64_t)(t < T ? t : T - 1) * M + r0;
    if (gate < 4) g[q][gate] = at(gi, (o * 4 + gate) * H, og[q]);
    else flag[q] = at(fresh, o, jr[q]);
  };
  auto store = [&](int t, int k, int q) __attribute__((always_inline)) {
    const int64_t o = (int64_t)t * M + r0;
    if (k == 0) at(hs, o * H, oh[q]) = h[q];
    if (CELL && k == 1) at(cs, o * H, oh[q]) = c[q];
    if (SAVE && k >= 2) at(saved, (o * 7 + k - 2) * H, ov[q]) = v[q][k - 2];
  };
  float hn[V], cn[V];  // the states the next step starts from
  auto begin = [&](int to) __attribute__((always_inline)) {
    unsigned part[3];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const bool f = (flag[q] & fresh_mask) != 0;
      hn[q] = f ? 0.f : h[q];
      cn[q] = f ? 0.f : c[q];
    }
    cut_pair(hn[0], hn[V - 1], part);
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = 0; q < V; ++q) sh[to][p * R + row + q][unit] = (unsigned short)(part[p] >> (16 * q));
  };
#pragma unroll
  for (int q = 0; q < V; ++q) {
    c[q] = at(c0, r0 * H, oh[q]);
    h[q] = at(h0, r0 * H, oh[q]);
#pragma unroll
    for (int gate = 0; gate < 5; ++gate) load(0, gate, q);
  }
  begin(0);
  seq_loads_done();
  __syncthreads();
  typedef CutTile<R, false> Tile;
  typename Tile::Lanes lanes(lane);
  float x[V] = {}, t4[4] = {}, bad = 0.f;
  auto activate = [](int gate, float x) {
    x = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * (gate == 2 ? 2.f * kLog2e : -kLog2e)) + 1.f);
    return gate == 2 ? fmaf(-2.f, x, 1.f) : x;
  };
  // A tile's gate, in pieces of a few instructions (`x` carries the value from one to the next): activation(x) of the hardware exponential and
  // reciprocal (about 1 ulp each) instead of the library's expf, tanhf and IEEE division, a fifth of the instructions.
  constexpr int kAct = R == 8 ? 8 : 5;
  auto act = [&](int gate, int piece) __attribute__((always_inline)) {
    auto add_input = [&](int q) { x[q] = g[q][gate] + x[q]; };
    auto scale = [&](int q) { x[q] *= gate == 2 ? 2.f * kLog2e : -kLog2e; };
    auto check = [&](int q) { bad = fmaf(x[q], 0.f, bad); };  // NaN once a preactivation is not finite
    auto power = [&](int q) { x[q] = __builtin_amdgcn_exp2f(x[q]); };
    auto invert = [&](int q) { x[q] = __builtin_amdgcn_rcpf(x[q]); };
    auto finish = [&](int q) { v[q][gate] = gate == 2 ? fmaf(-2.f, x[q], 1.f) : x[q]; };
    if constexpr (R == 8) {
      if (piece == 0) add_input(0), add_input(1);
      if (piece == 1) scale(0), scale(1);
      if (piece == 2 || piece == 3) check(piece - 2), power(piece - 2);
      if (piece == 4) x[0] += 1.f, x[1] += 1.f;
      if (piece == 5 || piece == 6) invert(piece - 5);
      if (piece == 7) finish(0), finish(1);
    } else {
      if (piece == 0) add_input(0);
      if (piece == 1) check(0), scale(0);
      if (piece == 2) power(0);
      if (piece == 3) x[0] += 1.f, invert(0);
      if (piece == 4) finish(0);
    }
  };
  auto cells = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < V; ++q) c[q] = fmaf(v[q][1], v[q][5], v[q][0] * v[q][2]);
  };
  auto leave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < V; ++q) {
      v[q][4] = seq_tanh(c[q]);
      h[q] = v[q][3] * v[q][4];
    }
  };
  // Step t's gates whose sums of the first parts' products are not finite: those decide, the other parts of an infinity are NaN.
  auto first_parts = [&](int t, int from) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      f32x4 sum = {};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(get_a<R>(&sh[from][0][0], kLstmStateLd, lane, 32 * kb + kq), w0[n][kb], sum, 0, 0, 0);
      float p[4];
      Tile::first_rows(sum, p);
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const int64_t o = (int64_t)t * M + r0;
        const bool starts = (at(fresh, o, jr[q]) & fresh_mask) != 0;  // an episode's first step has no product, whatever the weights are
        const float gate = activate(kGate[n], at(gi, (o * 4 + kGate[n]) * H, og[q]) + (starts ? 0.f : p[q]));
        v[q][kGate[n]] = fabsf(p[q]) < __builtin_inff() ? v[q][kGate[n]] : gate;
      }
    }
    cells();
  };
  auto step = [&](int t, auto from, bool first) __attribute__((always_inline)) {
    constexpr int B = R == 8 ? 2 : KB;  // eight rows read `b` again for each tile
    bf16x8 a[KB], b[B];
    auto load_b = [&](int kb) __attribute__((always_inline)) { b[kb % B] = get_b<R>(&sh[from][0][0], kLstmStateLd, lane, 32 * kb + kq, a[kb]); };
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) a[kb] = get_a<R>(&sh[from][0][0], kLstmStateLd, lane, 32 * kb + kq);
#pragma unroll
    for (int kb = 0; kb < B; ++kb) load_b(kb);
    u32x4 ring[2] = {w2[0], w2[64]};
    Tile tile, done;
    constexpr int S = Tile::kSteps, N = KB * S;  // matrix instructions per 32 k and per tile
    constexpr int R0 = 2, A0 = R0 + Tile::kRows, L0 = A0 + kAct;
    static_assert(L0 + V <= N && 9 * V <= 2 * N, "");
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      if (n > 0) done = tile;
      tile.clear();
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int kb = i / S, slot = n * KB + kb;
        tile.add(i % S, a[kb], b[kb % B], w0[n][kb], w1[n][kb], __builtin_bit_cast(bf16x8, ring[slot % 2]));
        if (i % S == S - 1 && slot + 2 < 4 * KB) {
          ring[slot % 2] = w2[(slot + 2) * 64];
          if (B < KB) load_b((kb + B) % KB);
        }
        // between the matrix instructions: under the first tile the last step's results leave; under the next ones the gate of the tile before
        __builtin_amdgcn_sched_barrier(0);
        if (n == 0) {
          if (SAVE && !first) {
#pragma unroll
            for (int k = 9 * V * i / N; k < 9 * V * (i + 1) / N; ++k) store(t - 1, k / V, k % V);
          }
          if (i == N - 1) {
#pragma unroll
            for (int q = 0; q < V; ++q) {
              load(t + 1, 4, q);
              v[q][5] = cn[q];
              v[q][6] = hn[q];
            }
          }
        } else {
          const int gate = kGate[n - 1];
          if (i >= R0 && i < L0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) pin(t4[k]);
#pragma unroll
            for (int q = 0; q < V; ++q) pin(x[q]);
              if (i < A0) done.rows(i - R0, lanes, t4, x);
            else act(gate, i - A0);
          }
          if (i >= L0 && i < L0 + V) load(t + 1, gate, i - L0);
          if (n == 3 && i == N - 1) cells();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // what has no more matrix instructions to stand between: tanh of the cell state and the output gate
#pragma unroll
    for (int k = 0; k < Tile::kRows; ++k) tile.rows(k, lanes, t4, x);
#pragma unroll
    for (int k = 0; k < kAct; ++k) act(3, k);
    leave();
    if (__builtin_expect(__any(!(bad == 0.f)), 0)) {
      bad = 0.f;
      first_parts(t, from);
      leave();
    }
    begin(1 - decltype(from)::value);
#pragma unroll
    for (int q = 0; q < V; ++q) load(t + 1, 3, q);
    if constexpr (!SAVE) {
#pragma unroll
      for (int k = 0; k < 2 * V; ++k) store(t, k / V, k % V);
    }
    lds_barrier();  // the new state is complete; the buffer just read is free for the step after next
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  step(0, even, true);
  int t = 1;
  for (; t + 1 < T; t += 2) {
    step(t, odd, false);
    step(t + 1, even, false);
  }
  if (t < T) step(t, odd, false);
  if constexpr (SAVE) {
#pragma unroll
    for (int k = 0; k < 9 * V; ++k) store(T - 1, k / V, k % V);
  }
  }
}

// A single step (a rollout's call: T = 1, hs / cs may be h0 / c0), to the same bits: with no next step to keep the weights for, a workgroup takes sixteen
// rows, whose three parts are an A operand each, and streams W_hh through its wavefronts, cut on the way.  It asks for neither the registers nor the
// LDS that would keep a CU to itself.  Two layers, through the sequence kernels -> here: 4096 rows 34.6 -> 22.1 us, 1000 20.2 -> 11.6, 64 10.3 -> 10.7;
// a rollout's control step of 4096 robots, whose physics runs beside the critic's layers, 421 -> 400.
template <bool CELL, bool SAVE>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(4, 4))) void lstm_step_kernel(Seq first, Seq second) {
  constexpr int H = kSeqH, KB = H / 32, R = kStepRows;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M, r0 = (int64_t)blockIdx.x * R;
  if (r0 >= M) return;  // the other layer of the launch has more rows
  const float *W = (const float*)s.W, *gi = s.in;
  const int ldw = s.ldw;
  __shared__ __attribute__((aligned(16))) unsigned short sh[3][R][kLstmStateLd];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int unit = 16 * wave + (lane & 15), kq = 8 * (lane >> 4);
  // the tiles are the unit's gates in the order below, their weights fetched a tile (four blocks of 32 k) ahead
  constexpr int kGate[4] = {1, 2, 0, 3};
  float4 w[KB][2];
  auto fetch = [&](int slot) __attribute__((always_inline)) {
    const float* src = W + (int64_t)(kGate[slot / KB] * H + unit) * ldw + 32 * (slot % KB) + kq;
    w[slot % KB][0] = *reinterpret_cast<const float4*>(src);
    w[slot % KB][1] = *reinterpret_cast<const float4*>(src + 4);
  };
#pragma unroll
  for (int slot = 0; slot < KB; ++slot) fetch(slot);
  {
    const int row = threadIdx.x >> 5, k = 4 * (threadIdx.x & 31);
    const int64_t m = r0 + row < M ? r0 + row : M - 1;
    f32x4 h = *reinterpret_cast<const f32x4_any*>(s.h0 + m * H + k);
    if (s.fresh && s.fresh[m]) h = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned lo[3], hi[3];
    cut_pair(h[0], h[1], lo);
    cut_pair(h[2], h[3], hi);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(&sh[p][row][k]) = uint2{lo[p], hi[p]};
  }
  // this lane's unit in rows 4 (lane / 16) + 0..3; rows past the batch repeat the last one and store its values once more
  const int64_t rows_left = M - r0;
  unsigned row[4];
  float c[4], h[4];
  int live = 0;  // bit i: row i goes on with an episode, whose first step has no product, whatever the weights are
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    row[i] = 4 * (lane >> 4) + i;
    if (row[i] >= rows_left) row[i] = (unsigned)(rows_left - 1);
    const bool f = s.fresh && s.fresh[r0 + row[i]];
    live |= f ? 0 : 1 << i;
    c[i] = f ? 0.f : at(s.c0, r0 * H, (row[i] * H + unit) * 4);
    if (SAVE) h[i] = f ? 0.f : at(s.h0, r0 * H, (row[i] * H + unit) * 4);
  }
  asm volatile("" : "+v"(live));  // as selects on four flags it became branches: 34.7 us of 21.6 for 4096 rows
  float g[2][4];
  auto inputs = [&](int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) g[n % 2][i] = at(gi, (r0 * 4 + kGate[n]) * H, (row[i] * 4 * H + unit) * 4);
  };
  inputs(0);
  __syncthreads();  // all states are read: from here on the outputs may be written over them
  auto mma = [](bf16x8 x, u32x4 y, f32x4& acc) __attribute__((always_inline)) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8, y), acc, 0, 0, 0);
  };
  float v[4][4];  // by gate
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int gate = kGate[n];
    float pre[4];
    if (n + 1 < 4) inputs(n + 1);
    f32x4 first[3] = {}, low[3] = {};  // by the state's parts: CutTile's products in its order
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int slot = n * KB + kb;
      const float4 lo = w[kb][0], hi = w[kb][1];
      if (slot + KB < 4 * KB) fetch(slot + KB);
      bf16x8 a[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8*>(&sh[p][lane & 15][32 * kb + kq]);
      const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      u32x4 part[3];
      cut_bf16<3>(x, part);
#pragma unroll
      for (int p = 0; p < 3; ++p) mma(a[p], part[0], first[p]);
#pragma unroll
      for (int p = 0; p < 3; ++p) mma(a[p], part[1], low[p]);
      mma(a[0], part[2], low[0]);
      mma(a[1], part[2], low[1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)  // the first parts decide where their sum is not finite, as in the sequence kernel
      pre[i] = join_cut(first[0][i], (low[0][i] + (first[2][i] + low[2][i])) + (first[1][i] + low[1][i]));
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // the arithmetic of the sequence kernel's pieces
      float x = g[n % 2][i] + __builtin_bit_cast(float, __builtin_bit_cast(int, pre[i]) & ((int)((unsigned)live << (31 - i)) >> 31));
      x *= gate == 2 ? 2.f * kLog2e : -kLog2e;
      x = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
      v[gate][i] = gate == 2 ? fmaf(-2.f, x, 1.f) : x;
    }
    __builtin_amdgcn_sched_barrier(0);  // a tile after the other: interleaved they spill (4096 rows 23.1 us of 21.6)
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float cn = fmaf(v[1][i], c[i], v[0][i] * v[2][i]), tc = seq_tanh(cn);
    at(s.out0, r0 * H, (row[i] * H + unit) * 4) = v[3][i] * tc;
    if (CELL) at(s.out1, r0 * H, (row[i] * H + unit) * 4) = cn;
    if (SAVE) {
      const float out[7] = {v[0][i], v[1][i], v[2][i], v[3][i], tc, c[i], h[i]};
#pragma unroll
      for (int k = 0; k < 7; ++k) at(s.saved, (r0 * 7 + k) * H, (row[i] * 7 * H + unit) * 4) = out[k];
    }
  }
}

// The reverse sweep of the same layer: dH (T, M, H) is the gradient reaching h_t from the layer above; the gradient through
// W_hh and that of the cell state are carried in registers.  Per step: the gate derivatives from the saved activations
// (lstm_gate_backward_kernel's formulas) into d_g (T, M, 4H) and, cut in three, into LDS, then dh_{t-1} = d_g W_hh over the transposed weights: a
// wavefront's tile is its 16 units, over all 4H gate rows.  The weights' third parts lie in registers for third_regs of the sixteen k blocks and in LDS
// for the others; eight rows, which have more sums, leave as few there as LDS allows and read the gate gradients a block less ahead.
constexpr int kLstmGateLd = 4 * kSeqH + 8;
constexpr int third_regs(int rows) { return rows == 8 ? 3 : 4; }
constexpr int lstm_backward_lds(int rows) { return kSeqWaves * (16 - third_regs(rows)) * 64 * 16 + 2 * 3 * rows * kLstmGateLd * 2; }

template <int R>
__global__ __launch_bounds__(64 * kSeqWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void lstm_seq_backward_kernel(int T, Seq first, Seq second) {
  constexpr int H = kSeqH, V = R / 4, KB = 4 * H / 32, kThirdRegs = third_regs(R), kAhead = R == 8 ? 2 : 3;
  const Seq s = blockIdx.y == 0 ? first : second;
  const int64_t M = s.M;
  const float* __restrict__ dH = s.in;
  const float* __restrict__ saved = s.saved;
  const uint8_t* __restrict__ fresh = s.fresh ? s.fresh : (const uint8_t*)s.in;  // as in the forward kernel
  const unsigned fresh_mask = s.fresh ? 0xffu : 0u;
  const float* __restrict__ Wt = (const float*)s.W;
  const int ldwt = s.ldw;
  float* __restrict__ d_g = s.out0;
  float *dh0 = s.dh0, *dc0 = s.dc0;
  const int64_t r0 = (int64_t)blockIdx.x * R;
  if (r0 >= M) return;  // the other layer of the launch has more rows
  extern __shared__ __attribute__((aligned(16))) unsigned char seq_lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int unit = 16 * wave + (lane & 15), row = seq_row<R>(lane), kq = 8 * (lane >> 4);  // the (unit, rows) whose gates this lane owns
  typename CutTile<R, true>::Lanes lanes(lane);
  u32x4* w2 = reinterpret_cast<u32x4*>(seq_lds) + wave * (16 - kThirdRegs) * 64 + lane;  // k block kThirdRegs and on
  typedef unsigned short Gates[3 * R][kLstmGateLd];
  Gates* sg = reinterpret_cast<Gates*>(seq_lds + kSeqWaves * (16 - kThirdRegs) * 64 * 16);  // of even and odd steps
  // the lane's rows and their bytes into a step's states, gates and kept activations; rows past the batch repeat the last one and store its values once more
  unsigned jr[V], oh[V], og[V], ov[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    jr[q] = r0 + row + q < M ? row + q : (unsigned)(M - 1 - r0);
    oh[q] = (jr[q] * H + unit) * 4;
    og[q] = (jr[q] * 4 * H + unit) * 4;
    ov[q] = (jr[q] * 7 * H + unit) * 4;
  }
  // B operand: column lane % 16 is the unit, rows the gate rows 32 kb + 8 (lane / 16) + 0..7
  bf16x8 w0[KB], w1[KB], w2r[kThirdRegs];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const float* src = Wt + (int64_t)unit * ldwt + 32 * kb + kq;
    const float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    u32x4 part[3];
    cut_bf16<3>(v, part);
    w0[kb] = __builtin_bit_cast(bf16x8, part[0]);
    w1[kb] = __builtin_bit_cast(bf16x8, part[1]);
    if (kb < kThirdRegs) w2r[kb < kThirdRegs ? kb : 0] = __builtin_bit_cast(bf16x8, part[2]);
    else w2[(kb - kThirdRegs) * 64] = part[2];
  }
  float dhc[V], dc[V];
  // a step's inputs i | f | g | o | tanh(c') | c | dH, requested under the products of the step before
  float in[V][7];
  unsigned flag[V];
  auto load = [&](int t, int k, int q) __attribute__((always_inline)) {
    const int64_t o = (int64_t)(t > 0 ? t : 0) * M + r0;
    if (k < 6) in[q][k] = at(saved, (o * 7 + k) * H, ov[q]);
    else if (k == 6) in[q][k] = at(dH, o * H, oh[q]);
    else flag[q] = at(fresh, o, jr[q]);
  };
#pragma unroll
  for (int q = 0; q < V; ++q) {
    dhc[q] = dc[q] = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) load(T - 1, k, q);
  }
  float t4[4] = {};
  auto step = [&](int t, auto cur) __attribute__((always_inline)) {
    bool f[V];
    float gate[V][4];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      f[q] = (flag[q] & fresh_mask) != 0;
      LstmSlopes slope;
      slope.make(in[q][0], in[q][1], in[q][2], in[q][3], in[q][4], in[q][5]);
      const float dct = slope.gates(in[q][6] + dhc[q], dc[q], gate[q]);
      dc[q] = f[q] ? 0.f : dct * slope.keep;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned part[3];
      cut_pair(gate[0][g], gate[V - 1][g], part);
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < V; ++q) sg[cur][p * R + row + q][g * H + unit] = (unsigned short)(part[p] >> (16 * q));
    }
    lds_barrier();  // the gate gradients are complete; the buffer of the step before is free for the step after
    constexpr int D = kAhead + 1;
    bf16x8 a[D], b[D];
    auto load_ab = [&](int kb) __attribute__((always_inline)) {
      a[kb % D] = get_a<R>(&sg[cur][0][0], kLstmGateLd, lane, 32 * kb + kq);
      if constexpr (R == 8) b[kb % D] = get_b<R>(&sg[cur][0][0], kLstmGateLd, lane, 32 * kb + kq, a[kb % D]);
    };
#pragma unroll
    for (int kb = 0; kb < kAhead; ++kb) load_ab(kb);
    CutTile<R, true> tile;
    tile.clear();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (kb + kAhead < KB) load_ab(kb + kAhead);
#pragma unroll
      for (int i = 0; i < CutTile<R, true>::kSteps; ++i)
        tile.add(i, a[kb % D], b[kb % D], w0[kb], w1[kb],
                 kb < kThirdRegs ? w2r[kb < kThirdRegs ? kb : 0] : __builtin_bit_cast(bf16x8, w2[(kb - (kb < kThirdRegs ? kb : kThirdRegs)) * 64]));
      // between the products the step's gate gradients leave and the inputs of the next come
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < V; ++q) {
        if (kb < 8) load(t - 1, kb, q);
        else if (kb < 12) at(d_g, (((int64_t)t * M + r0) * 4 + kb - 8) * H, og[q]) = gate[q][kb - 8];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    float x[V];
#pragma unroll
    for (int k = 0; k < CutTile<R, true>::kRows; ++k) tile.rows(k, lanes, t4, x);
#pragma unroll
    for (int q = 0; q < V; ++q) {  // the first parts decide, entry by entry
      const float first = t4[R == 8 ? 2 + q : 3];
      x[q] = fabsf(first) < __builtin_inff() ? x[q] : first;
    }
#pragma unroll
    for (int q = 0; q < V; ++q) dhc[q] = f[q] ? 0.f : x[q];
  };
  int t = T - 1;
  for (; t >= 1; t -= 2) {
    step(t, std::integral_constant<int, 0>{});
    step(t - 1, std::integral_constant<int, 1>{});
  }
  if (t == 0) step(0, std::integral_constant<int, 0>{});
#pragma unroll
  for (int q = 0; q < V; ++q) {
    if (dh0) at(dh0, r0 * H, oh[q]) = dhc[q];
    if (dc0) at(dc0, r0 * H, oh[q]) = dc[q];
  }
}

// ---------------------------------------------------------------- a whole trajectory of one GRU layer in one launch
// As for the LSTM, eight wavefronts own 4 rows for all T steps: block b = lane / 4 of wavefront w is hidden
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
  for (int grp = 0; grp < groups; ++grp) {  // several sets of 4 rows with the same registers of weights
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
// rows (96 each) times four groups of four units, in bf16 a step of four k is one
// block's entry.  The gate gradients are the A operand (entries = the four rows), the same for the four blocks of a quarter and broadcast to them from one
// block per instruction (CBSZ = 2, ABID = k mod 4); a lane's partial sums over its quarter are added up and scattered over the lane rows.
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
  const int rc = launch(s, m, (rows + kSeqRows - 1) / kSeqRows);
  return rc != KS_OK ? rc : check_launch(who);
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
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) -> int {
    const int groups = seq_groups(T, sets);
    hipLaunchKernelGGL(bf[0] ? gru_seq_forward_kernel<true> : gru_seq_forward_kernel<false>, dim3((unsigned)((sets + groups - 1) / groups), (unsigned)count),
                       dim3(64 * kSeqWaves), 0, (hipStream_t)stream, (int)T, groups, s[0], s[1]);
    return KS_OK;
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
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) -> int {
    hipLaunchKernelGGL(bf[0] ? gru_seq_backward_kernel<true> : gru_seq_backward_kernel<false>, dim3((unsigned)sets, (unsigned)count), dim3(64 * kSeqWaves), 0,
                       (hipStream_t)stream, (int)T, s[0], s[1]);
    return KS_OK;
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

// Rows per workgroup: 8 once sets of 4 are more than the CUs, which hold one workgroup each.
static bool lstm_wide(int count, const Seq& a, const Seq& b) {
  return (a.M + 3) / 4 + (count > 1 ? (b.M + 3) / 4 : 0) > 256;
}

template <typename... P, typename... A>
static int launch_lstm(const char* who, void (*fn)(P...), dim3 grid, int lds, ks_stream_t stream, A... args) {
  if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(KS_ELAUNCH, "%s: cannot reserve %d bytes of LDS", who, lds);
  hipLaunchKernelGGL(fn, grid, dim3(64 * kSeqWaves), lds, (hipStream_t)stream, args...);
  return KS_OK;
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
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) -> int {
    auto run = [&](int count, const Seq& first, const Seq& second) -> int {
      const bool cell = first.out1 != nullptr, save = first.saved != nullptr;
      if (T == 1) {
        const int64_t most = first.M > second.M ? first.M : second.M;
        hipLaunchKernelGGL(cell ? (save ? lstm_step_kernel<true, true> : lstm_step_kernel<true, false>)
                                : (save ? lstm_step_kernel<false, true> : lstm_step_kernel<false, false>),
                           dim3((unsigned)((most + kStepRows - 1) / kStepRows), (unsigned)count), dim3(64 * kSeqWaves), 0, (hipStream_t)stream, first, second);
        return KS_OK;
      }
      const bool wide = lstm_wide(count, first, second);
      const int rows = wide ? 8 : 4, groups = wide ? (seq_groups(T, sets) + 1) / 2 : seq_groups(T, sets);
      auto fn = wide ? (cell ? (save ? lstm_seq_forward_kernel<8, true, true> : lstm_seq_forward_kernel<8, true, false>)
                            : (save ? lstm_seq_forward_kernel<8, false, true> : lstm_seq_forward_kernel<8, false, false>))
                    : (cell ? (save ? lstm_seq_forward_kernel<4, true, true> : lstm_seq_forward_kernel<4, true, false>)
                            : (save ? lstm_seq_forward_kernel<4, false, true> : lstm_seq_forward_kernel<4, false, false>));
      const int64_t M = first.M > second.M ? first.M : second.M;
      return launch_lstm(who, fn, dim3((unsigned)((M + rows * groups - 1) / (rows * groups)), (unsigned)count), lstm_forward_lds(rows), stream, (int)T, groups,
                         first, second);
    };
    if (count == 2 && (!s[0].out1 != !s[1].out1 || !s[0].saved != !s[1].saved)) {  // a kernel writes the same outputs for both of its layers
      const int rc = run(1, s[0], s[0]);
      return rc != KS_OK ? rc : run(1, s[1], s[1]);
    }
    return run(count, s[0], s[1]);
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
  return run_sequences(who, n, T, q, fill, [&](const Seq* s, int count, int64_t sets) -> int {
    const bool wide = lstm_wide(count, s[0], s[1]);
    return launch_lstm(who, wide ? lstm_seq_backward_kernel<8> : lstm_seq_backward_kernel<4>, dim3((unsigned)(wide ? (sets + 1) / 2 : sets), (unsigned)count),
                       lstm_backward_lds(wide ? 8 : 4), stream, (int)T, s[0], s[1]);
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
