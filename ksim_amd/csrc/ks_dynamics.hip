// Fused control-step kernel: S physics substeps of one env per wavefront.
//
// One 64-lane wavefront owns one env (64-thread workgroups, so a workgroup barrier is a wave barrier).
// Where the data lives:
//   registers  the mass matrix / Newton Hessian as a 32x32 matrix-core accumulator tile while it is assembled and
//              factored, then row i of the factor for the substitutions; the lane's own body / dof / sphere
//              constants; all per-dof and per-row solver vectors
//   LDS        state (qpos, qvel, warm start, torques), body poses, com-based inertias and motion axes,
//              a staging copy of M and of J (column access), one broadcast vector
//   HBM        touched once at the start and once at the end of the control step
// Cross-lane traffic is v_readlane broadcasts (pivots, triangular solves), DPP reductions and LDS
// broadcasts; the rank updates of the Hessian and of its factorisation run as 32x32x2 fp32 MFMAs; every
// branch on solver progress is wave-uniform, so a converged env stops iterating.
// Phases of one substep: kinematics along ancestor chains -> centre of mass -> com-based inertias / motion
// axes -> composite inertias -> mass matrix -> velocities + RNE bias along ancestor chains -> smooth forces ->
// sphere/plane contacts, pyramidal rows -> Cholesky of M -> Newton with exact line search -> semi-implicit Euler.
// The arithmetic follows the MuJoCo model that ksim/engine.py:257 invokes through mjx.step.
#include "ks_common.h"
#include "ks_model.h"
#include "ks_philox.h"
#include "ks_step_args.h"

#include <cmath>
#include <cstddef>
#include <cstring>

namespace ks {

typedef __attribute__((ext_vector_type(16))) float f32x16;

// Hand-over through LDS between lanes of the workgroup's one wavefront.  The LDS pipeline serves a wavefront's accesses in the order
// they were issued, so a read behind a write needs no wait: this only keeps the compiler from moving accesses across the line.
// (__syncthreads() would drain the wavefront's LDS and memory traffic at two dozen places of a substep.)
#define KS_SYNC() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); }
#ifndef KS_STEP_WAVES
#define KS_STEP_WAVES 4  // wavefronts per SIMD the register allocation aims at
#endif
// Phase timers for kernel tuning: compiled in only with -DKS_PROFILE, which reuses the dbg_M buffer for cycle counts.
#ifdef KS_PROFILE
#define KS_TICK(k) { const long long t_now = clock64(); prof[k] += (float)(t_now - t_last); t_last = t_now; }
#else
#define KS_TICK(k)
#endif
// A phase boundary of the step kernel.  The part of the LDS layout that depends on the model's sizes is rebuilt from an offset
// the compiler cannot see through: its array addresses are then a few scalar additions at the start of each phase instead of
// values that stay live from the top of the kernel, where they do not fit the scalar registers and every use reads its address
// back out of a vector register lane.
#define KS_PHASE(k) { KS_TICK(k) int off_ = 0; asm volatile("" : "+s"(off_)); l = carve<NP>(lds_raw, lds_raw + off_, nb, nq, nv, nu, ns); }
// Register rows (mass matrix, Hessian, Jacobian) are padded from nv to a compile-time width NP, one kernel
// instantiation per width: the padding rows are unit rows and the padding columns zero, so the factorisation,
// the triangular solves and the row products run without any bound checks.
__host__ __device__ inline int padded_nv(int nv) { return nv <= 8 ? 8 : nv <= 16 ? 16 : nv <= 24 ? 24 : nv <= 28 ? 28 : 32; }
// Row stride of M and J in LDS, a constant of the instantiation: rows are 16-byte aligned (read with ds_read_b128, one row per
// lane) and the stride in 16-byte units is odd, which spreads 16 consecutive rows over all 64 banks.
__host__ __device__ constexpr int stride_of(int np) { return (np / 4) % 2 ? np : np + 4; }

struct Lds {
  // at the same place for every model of an instantiation
  float *vbuf, *qvel, *warm, *drow, *M;
  // behind them, sized by the model
  float *qpos, *tau;
  float *xpos, *xquat;
  float *cinert, *crb, *cdof, *buf, *cvel, *cfrc, *fsub;
  float *xanchor, *xaxis;  // joint anchors and axes: dead once the motion axes are built, so they share buf and fsub
  float* J;
  float *con_off, *con_D, *con_kip;
  int *con_body, *sub_end;
  unsigned* con_mask;
};

__host__ __device__ inline int up4(int n) { return (n + 3) & ~3; }

__host__ __device__ inline int lds_floats(int nb, int nq, int nv, int nu, int ns) {
  const int np = padded_nv(nv), js = stride_of(np);
  int n = 0;
  n += 32 + 32 + 32 + 64 + np * js;                                  // vbuf qvel warm drow M
  n += up4(nq) + up4(nu);                                            // qpos tau
  n += up4(nb * 3) + up4(nb * 4);                                    // xpos xquat
  n += up4(nv * 6) + up4(nb * 6);                                    // cdof cvel
  const int scratch = 2 * up4(nb * 10) + up4(nv * 6) + 2 * up4(nb * 6);  // cinert crb buf fsub cfrc
  const int jsz = up4(4 * ns * js + 32);                             // J overlays that scratch once it is dead
  n += scratch > jsz ? scratch : jsz;
  n += up4(ns * 3) + 4 * up4(ns) + up4(nb);                          // con_off con_D con_kip con_body con_mask sub_end
  return n + 8;
}

template <int NP>
__device__ __forceinline__ Lds carve(float* base, float* p, int nb, int nq, int nv, int nu, int ns) {
  constexpr int js = stride_of(NP);
  Lds l;
  l.vbuf = base; l.qvel = base + 32; l.warm = base + 64; l.drow = base + 96; l.M = base + 160;
  p += 160 + NP * js;
  auto take = [&](int n) {
    float* r = p;
    p += up4(n);
    return r;
  };
  l.qpos = take(nq); l.tau = take(nu);
  l.xpos = take(nb * 3); l.xquat = take(nb * 4);
  l.cdof = take(nv * 6); l.cvel = take(nb * 6);
  {
    float* first = p;
    l.cinert = take(nb * 10); l.crb = take(nb * 10); l.buf = take(nv * 6);
    l.fsub = take(nb * 6); l.cfrc = take(nb * 6);
    l.xanchor = l.buf; l.xaxis = l.fsub;
    float* end = p;
    l.J = first;  // written only after the bias forces are out of fsub
    float* jend = first + up4(4 * ns * js + 32);
    p = end > jend ? end : jend;
  }
  l.con_off = take(ns * 3); l.con_D = take(ns); l.con_kip = take(ns);
  l.con_body = reinterpret_cast<int*>(take(ns));
  l.con_mask = reinterpret_cast<unsigned*>(take(ns));
  l.sub_end = reinterpret_cast<int*>(take(nb));
  return l;
}

// NP consecutive floats from a 16-byte aligned LDS address
template <int NP>
__device__ __forceinline__ void load_row(const float* p, float (&v)[NP]) {
  const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int k = 0; k < NP / 4; ++k) {
    const float4 t = q[k];
    v[4 * k] = t.x; v[4 * k + 1] = t.y; v[4 * k + 2] = t.z; v[4 * k + 3] = t.w;
  }
}


// Right-looking Cholesky of a symmetric matrix of up to 32 rows with the rank-1 updates on the matrix cores.
// The matrix sits in the accumulator layout of the 32x32x2 fp32 MFMA: lane c + 32 h holds, in register
// 4 g + e, the entry (row 8 g + 4 h + e, column c).  A step takes the two columns j, j + 1, whose rows lie in neighbouring registers of one
// lane half: row j is scaled by its pivot's reciprocal root, its share is taken off row j + 1 by one multiply-add, that row is scaled, and the
// two go to one MFMA as both operands, -l l^T, one in each lane half (the instruction's two k), which updates every entry right of and below
// them at once; row j + 1, already up to date, is left out of the left operand.  The instruction holds a SIMD's vector issue for 64 cycles
// whether its second k is used or not (fp32 MFMAs and vector instructions take turns), and with one column per step that was a fifth of the
// kernel: 8192 mixed robots 507 -> 474 us per control step, 4096 humanoids 356 -> 338.  (Here and below the two figures of a pair are from one
// card in turn; cards differ by up to 4 %, so pairs do not continue one another.)
// Column j below the diagonal and row j right of it are left as they were when the pivot was reached, L[k][j] * L[j][j] (the scaled row
// goes into the MFMA only): read down a lane, that is what both substitutions take in their square-root-free form (back_steps),
// once the upper lane half has handed its 16 registers to the lower one.  On return, in lane i < NP:
//   R[j], j < i : L[i][j] * L[j][j]              R[k], k > i : L[k][i] * L[i][i]              myinv = 1 / L[i][i]
// `nv` (wave-uniform) is the real size: the steps of the padded columns, which would multiply zeros, are branched over
// (only steps past the next smaller instantiation's size carry the test).
constexpr int padded_from(int np) { return np > 28 ? 28 : (np > 24 ? 24 : (np > 16 ? 16 : (np > 8 ? 8 : 0))); }

// one lane half of x below, the same half of y above
__device__ __forceinline__ float halves(float x, float y, int half) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y), false, false);
  return __builtin_bit_cast(float, half ? r[1] : r[0]);
}

// Lanes first .. first + count - 1, known at compile time, as the condition of a select: one scalar instruction, which costs the vector issue
// nothing, instead of a compare (4.5 cycles of it).  `site` is a zero the compiler cannot see through, one per call of a solver: shared between
// the call sites the masks would be sixty-odd scalar register pairs that live across the solver and are read back from spill lanes.
// 4096 humanoids 336 -> 329 us per control step, 8192 mixed robots 491 -> 486, 64 robots 235 -> 233 (volatile instead of `site`: 329, 487, 235).
__device__ __forceinline__ bool in_lanes(int first, int count, int site) {
  unsigned long long mask;
  asm("s_bfm_b64 %0, %1, %2" : "=s"(mask) : "i"(count), "i"(first), "s"(site));
  return __builtin_amdgcn_inverse_ballot_w64(mask);
}

template <int NP>
__device__ __forceinline__ void chol_tile(f32x16& T, float (&R)[NP], float& myinv, int nv) {
  int site = 0;
  asm volatile("" : "+s"(site));
  myinv = 1.f;
  // a pivot below 1e-30 (or not a number) counts as 1e-30: the reciprocal root is capped instead of the pivot floored,
  // which is the same number and one instruction less on the chain
  auto inv_root = [](float pivot) { return fminf(__builtin_amdgcn_rsqf(pivot), 1e15f); };
#pragma unroll
  for (int j = 0; j < NP; j += 2) {
    if (j >= padded_from(NP) && j >= nv) continue;  // padded columns: unit pivots, nothing below or right of them
    const int hj = (j >> 2) & 1, rho = 4 * (j >> 3) + (j & 3), own = j + 32 * hj;
    const float inv0 = inv_root(lane_bcast(T[rho], own));
    myinv = in_lanes(j, 1, site) ? inv0 : myinv;
    const bool right0 = in_lanes(own + 1, 31 - j, site);
    float a0 = right0 ? T[rho] : 0.f;  // beside the reciprocal root, not behind it
    a0 *= inv0;
    const float v = T[rho + 1] - a0 * lane_bcast(a0, own + 1);
    T[rho + 1] = v;
    const float inv1 = inv_root(lane_bcast(v, own + 1));
    myinv = in_lanes(j + 1, 1, site) ? inv1 : myinv;
    const bool right1 = in_lanes(own + 2, 30 - j, site);
    float a1 = right1 ? v : 0.f;
    a1 *= inv1;
    // the last real columns have nothing right of or below them
    if (j + 2 < NP && !(j + 2 >= padded_from(NP) && j + 2 >= nv)) {
      const float b = halves(a0, a1, hj), na = in_lanes(j + 1, 1, site) ? 0.f : -b;
      T = __builtin_amdgcn_mfma_f32_32x32x2f32(na, b, T, 0, 0, 0);
    }
  }
  asm volatile("s_nop 15\n\ts_nop 3" : "+v"(T));  // the substitutions' assembly takes these registers as vector instructions leave them
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int jlo = 8 * g + e, jhi = 8 * g + 4 + e;
      if (jlo < NP) R[jlo] = T[4 * g + e];
      if (jhi < NP) R[jhi] = __shfl_xor(T[4 * g + e], 32);
    }
}

// Mass matrix (LDS, NP rows: beyond nv unit rows and zero columns) into the accumulator layout.  What the tile holds outside
// NP x NP is a copy of entries inside it, which the factorisation writes but never reads, except that column 31 is the right-hand
// side `rhs` (32 floats in LDS) where the matrix leaves room for it (chol_solve).
template <int NP>
__device__ __forceinline__ void load_mtile(f32x16& T, const float* __restrict__ M, const float* __restrict__ rhs, int lane) {
  const int c = lane & 31, half = lane >> 5;
  const float* row = M + min(c, NP - 1) * stride_of(NP);
  if (NP < 32) row = c == 31 ? rhs : row;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 v = *reinterpret_cast<const float4*>(row + min(8 * g + 4 * half, NP - 4));
    T[4 * g] = v.x; T[4 * g + 1] = v.y; T[4 * g + 2] = v.z; T[4 * g + 3] = v.w;
  }
}

template <int NP>
__device__ __forceinline__ bool padded_out(int k, int nv) { return k >= padded_from(NP) && k >= nv; }  // such unknowns are zero and couple to nothing

// A substitution step: w_i += w_K c_i in the COUNT lanes from FIRST on, lane K being in their row of 16.  `v_fmac` takes lane K of its row through
// DPP, which wants two wait states behind the write of any of its registers (s_nop 1); the mask is one scalar instruction.  Broadcast to
// all 32 rows through a scalar register, the step was a lane read, two wait states and the multiply-add, for every column one after the
// other; now the chains are 16 columns at most, and what one row of lanes takes off the other are products side by side (row_products).  With the
// rows kept unscaled (two selects per pair of columns less) a wavefront alone factors and solves M in 4570 cycles instead of 4970, and 4096
// humanoids' control step has 76.5 M vector instructions instead of 79 M: rollout steps of 64 and of 1024 K-Bots, of 4096 humanoids and of an
// LSTM policy 1.1, 1.3, 1.3 and 1.0 % faster.  Error against 64 bits over 6000 random states, as shares of the largest
// entry, the rotations by quaternions (qrot) included: of qacc_smooth, rms, 0.71e-6 -> 0.70e-6 (kbot_scale_model) and 1.69e-6 -> 1.70e-6 (humanoid_model with joint limits), of qacc, the
// median env's largest, 2.6e-6 -> 2.2e-6 and 4.1e-6 -> 3.7e-6.
template <int K, int FIRST, int COUNT>
__device__ __forceinline__ void row_step(float& w, float c) {
  unsigned long long mask;
  asm("s_bfm_b64 %1, %4, %3\n\tv_cndmask_b32_e64 %2, 0, %2, %1\n\ts_nop 1\n\tv_fmac_f32_dpp %0, %0, %2 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(w), "=&s"(mask), "+v"(c) : "i"(FIRST), "i"(COUNT), "i"(K % 16));
}
// columns K down to LO + 1 of the backward substitution, K up to HI - 1 of the forward one, within a row of 16 lanes: with w_i = y_i / L[i][i]
// a step is w_i -= (R[k] / L[i][i]^2) w_k (m = -1 / L[i][i]^2)
template <int NP, int K, int LO>
__device__ __forceinline__ void back_steps(const float (&R)[NP], float m, float& w, int nv) {
  if constexpr (K > LO) {
    if (!padded_out<NP>(K, nv)) row_step<K, LO, K - LO>(w, R[K] * m);
    back_steps<NP, K - 1, LO>(R, m, w, nv);
  }
}
template <int NP, int K, int HI>
__device__ __forceinline__ void forward_steps(const float (&R)[NP], float m, float& w, int nv) {
  if constexpr (K < HI) {
    if (!padded_out<NP>(K, nv)) row_step<K, K + 1, HI - K>(w, R[K] * m);
    forward_steps<NP, K + 1, HI>(R, m, w, nv);
  }
}
// sum over K < END, a multiple of four of them, of R[K] x_K, x_K in lane K % 16 of each row of 16
#define KS_ROW_PRODUCT(OP, T, R, LANE) OP " %" #T ", %4, %" #R " row_newbcast:%" #LANE " row_mask:0xf bank_mask:0xf\n\t"
#define KS_ROW_PRODUCTS(OP) "s_nop 1\n\t" KS_ROW_PRODUCT(OP, 0, 5, 9) KS_ROW_PRODUCT(OP, 1, 6, 10) KS_ROW_PRODUCT(OP, 2, 7, 11) KS_ROW_PRODUCT(OP, 3, 8, 12)
template <int NP, int K, int END>
__device__ __forceinline__ void row_products_from(const float (&R)[NP], float x, float (&t)[4]) {
  if constexpr (K < END) {
    asm(KS_ROW_PRODUCTS("v_fmac_f32_dpp") : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3])
        : "v"(x), "v"(R[K]), "v"(R[K + 1]), "v"(R[K + 2]), "v"(R[K + 3]), "i"(K % 16), "i"(K % 16 + 1), "i"(K % 16 + 2), "i"(K % 16 + 3));
    row_products_from<NP, K + 4, END>(R, x, t);
  }
}
template <int NP, int K, int END>
__device__ __forceinline__ float row_products(const float (&R)[NP], float x) {
  float t[4];
  asm(KS_ROW_PRODUCTS("v_mul_f32_dpp") : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3])
      : "v"(x), "v"(R[K]), "v"(R[K + 1]), "v"(R[K + 2]), "v"(R[K + 3]), "i"(K % 16), "i"(K % 16 + 1), "i"(K % 16 + 2), "i"(K % 16 + 3));
  row_products_from<NP, K + 4, END>(R, x, t);
  return (t[0] + t[1]) + (t[2] + t[3]);
}

// lanes 0..15 of x in lanes 0..15 and 16..31 of `lower`, lanes 16..31 in both of `upper` (assembly: the builtin's two results come out the same)
__device__ __forceinline__ void lane_rows(float x, float& lower, float& upper) {
  lower = upper = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lower), "+v"(upper));
}

// L^T x = y, lane i holding w_i = y_i / L[i][i] and returning x_i.  Of more than 16 rows the upper lane row comes first; what it takes off the
// lower one are products without a chain.
template <int NP>
__device__ __forceinline__ float back_substitute(const float (&R)[NP], float myinv, float w, int nv) {
  const float m = -myinv * myinv;
  if constexpr (NP > 16) {
    back_steps<NP, NP - 1, 16>(R, m, w, nv);
    float upper, lower;
    lane_rows(w, lower, upper);
    const float below = fmaf(row_products<NP, 16, NP>(R, upper), m, w);
    w = in_lanes(0, 16, 0) ? below : w;
  }
  back_steps<NP, (NP > 16 ? 15 : NP - 1), 0>(R, m, w, nv);
  return w;
}

// x = (L L^T)^-1 b, lane i holding b_i and returning x_i
template <int NP>
__device__ __forceinline__ float solve_regs(const float (&R)[NP], float myinv, float b, int nv) {
  const float m = -myinv * myinv;
  float w = b * myinv * myinv;
  forward_steps<NP, 0, (NP > 16 ? 15 : NP - 1)>(R, m, w, nv);
  if constexpr (NP > 16) {
    float upper, lower;
    lane_rows(w, lower, upper);
    const float above = fmaf(row_products<NP, 0, 16>(R, lower), m, w);
    w = in_lanes(16, 16, 0) ? above : w;
    forward_steps<NP, 16, NP - 1>(R, m, w, nv);
  }
  return back_substitute<NP>(R, myinv, w, nv);
}

// Factors the tile and returns x = (L L^T)^-1 b, lane i holding b_i (zero beyond nv).  A matrix of fewer than 32 columns carries b
// along as column 31 of its tile (load_mtile): the rank-1 updates of the factorisation then are the forward substitution too, and what
// is left of it is to hand y = L^-1 b, times L[i][i], which the two lanes of that column hold, to the lanes of its rows, through LDS (`vbuf`,
// 32 floats).
template <int NP>
__device__ __forceinline__ float chol_solve(f32x16& T, float (&R)[NP], float& myinv, int lane, float b, int nv, float* vbuf) {
  chol_tile<NP>(T, R, myinv, nv);
  if constexpr (NP == 32) {
    return solve_regs<NP>(R, myinv, b, nv);
  } else {
    asm volatile("" : "+v"(lane));
    KS_SYNC();
    if ((lane & 31) == 31) {
      float4* dst = reinterpret_cast<float4*>(vbuf) + (lane >> 5);
#pragma unroll
      for (int g = 0; g < 4; ++g) dst[2 * g] = {T[4 * g], T[4 * g + 1], T[4 * g + 2], T[4 * g + 3]};
    }
    KS_SYNC();
    const float y = vbuf[lane & 31];  // times L[i][i]
    KS_SYNC();
    return back_substitute<NP>(R, myinv, y * myinv * myinv, nv);
  }
}

// dot product of an LDS row (per-lane address, 16-byte aligned) with a broadcast register vector
template <int NP>
__device__ __forceinline__ float row_dot(const float* row, const float (&vv)[NP]) {
  const float4* q = reinterpret_cast<const float4*>(row);
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int k = 0; k < NP / 4; ++k) {  // two chains of fused multiply-adds, one instruction per product
    const float4 t = q[k];
    s0 = fmaf(t.x, vv[4 * k], s0);
    s1 = fmaf(t.y, vv[4 * k + 1], s1);
    s0 = fmaf(t.z, vv[4 * k + 2], s0);
    s1 = fmaf(t.w, vv[4 * k + 3], s1);
  }
  return s0 + s1;
}

// Per-lane constants of one substep, as stored in DevModel::lane_rec (64 dwords, filled by ks_model_create):
// lane L's body (L < nb), dof (L < nv), contact sphere (L < ns) and its share of the (i, ancestor j) dof pairs.
// Lanes beyond a range carry the entries of index 0 (or -1 / zero where the kernel tests for that).
constexpr int kPairSets = (kMaxPairs + 63) / 64;

struct LaneRec {
  int b_jtype, b_qadr, b_dofadr, b_depth;
  float b_q0, b_mass, d_stiffness;  // d_stiffness: spring of the hinge whose dof this lane holds
  float d_damping;
  float b_pos[3], d_armature, b_jaxis[3], d_gear, b_jpos[3], d_lo;
  float b_quat[4], b_iquat[4];
  int d_body, d_act, d_jtype, d_k;
  float d_hi;
  int s_body;
  float s_invw;
  unsigned s_mask;
  int pk[kPairSets];
  // the body's ancestors from the tree root down to itself, 16 bits each: body | first dof << 5 | hinge << 10 | free joint << 11
  unsigned b_chain[kMaxDepth / 2];
  // rows that live on the dof's own lane: hinge limit (range, inverse weight, address of the joint angle) and dry
  // friction (level and the constant stiffness 1 / R of its row)
  int d_limited, d_qadr;
  float d_rlo, d_rhi, d_invw, d_floss, d_frD;
  int pad[7];
};
static_assert(sizeof(LaneRec) == sizeof(DevModel::lane_rec) / 64, "LaneRec must fill the record");
static_assert(kMaxB <= 32 && kMaxV <= 32 && kMaxDepth % 2 == 0, "a link of b_chain holds 5 + 5 bits");
constexpr int kRecPieces = sizeof(LaneRec) / 16;
// ... and what the env itself may bring beside them
struct LaneIn {
  LaneRec rec;
  V3 ipos, inertia, sph_pos;  // of the lane's body and contact sphere
  float mass_scale, damping_scale, armature_scale, sph_radius;
};
// one field of a lane's record
#define KS_REC(m, lane, field) (__builtin_bit_cast(decltype(LaneRec::field), (m).lane_rec[offsetof(LaneRec, field) / 16][lane][offsetof(LaneRec, field) / 4 % 4]))

struct LsPoint {
  float alpha, cost, d0, d1;
};

// wave_sum of three or four values side by side: their steps fill each other's waits, and the two last ones leave the rows they do not reach as they
// are instead of adding a zero to them (a move and an addition each).  The first step is the compiler's, as in wave_sum: where a value is a product
// it goes into that addition unrounded, which a sum that begins in the assembly loses (qacc in the last bits).  A substep takes seven such sets.
// Against one sum after the other, in turn on one card: control step of 64 robots 231.9 -> 228.4 us, 8192 mixed robots 482 -> 478, 4096 humanoids
// 328.9 -> 326.8, the same bits (spread of a side 0.1 to 0.4 %).
// The compiler does not look into the assembly for hazards.  Covered here: a DPP read needs two instructions behind the write of its register (s_nop 1
// ahead of the first step, the other values' steps between two of its own) and a lane read one behind it (s_nop 0).  Not covered: values that come
// straight from a matrix instruction, and a vector write of the lane mask (v_cmpx) just ahead.
#define KS_SUM_STEP(CTRL) "v_add_f32_dpp %0, %0, %0 " CTRL "\n\tv_add_f32_dpp %1, %1, %1 " CTRL "\n\tv_add_f32_dpp %2, %2, %2 " CTRL "\n\t"
#define KS_SUM_STEP4(CTRL) KS_SUM_STEP(CTRL) "v_add_f32_dpp %3, %3, %3 " CTRL "\n\t"
#define KS_ROW "row_mask:0xf bank_mask:0xf bound_ctrl:1"
#define KS_SUM_STEPS(STEP) "s_nop 1\n\t" STEP("row_shr:2 " KS_ROW) STEP("row_shr:4 " KS_ROW) STEP("row_shr:8 " KS_ROW) \
    STEP("row_bcast:15 row_mask:0xa bank_mask:0xf") STEP("row_bcast:31 row_mask:0xc bank_mask:0xf") "s_nop 0"
__device__ __forceinline__ void wave_sums(float& x, float& y, float& z) {
  x += dpp_shift<0x111, 0xf>(x); y += dpp_shift<0x111, 0xf>(y); z += dpp_shift<0x111, 0xf>(z);
  asm(KS_SUM_STEPS(KS_SUM_STEP) : "+v"(x), "+v"(y), "+v"(z));
  x = lane_bcast(x, 63); y = lane_bcast(y, 63); z = lane_bcast(z, 63);
}
__device__ __forceinline__ void wave_sums(float& x, float& y, float& z, float& w) {
  x += dpp_shift<0x111, 0xf>(x); y += dpp_shift<0x111, 0xf>(y); z += dpp_shift<0x111, 0xf>(z); w += dpp_shift<0x111, 0xf>(w);
  asm(KS_SUM_STEPS(KS_SUM_STEP4) : "+v"(x), "+v"(y), "+v"(z), "+v"(w));
  x = lane_bcast(x, 63); y = lane_bcast(y, 63); z = lane_bcast(z, 63); w = lane_bcast(w, 63);
}

// constraint impedance d(|pos|) of a solimp whose parameters are already clamped
__device__ __forceinline__ float impedance_of(float pos, float dmin, float dmax, float width_inv, float mid, float power, float imp_a,
                                              float imp_b) {
  const float ix = fabsf(pos) * width_inv;
  // x^power: the default power of 2 (and 1) without the general power function
  const float ox = 1.f - ix;
  const float px = power == 2.f ? ix * ix : (power == 1.f ? ix : powf(ix, power));
  const float po = power == 2.f ? ox * ox : (power == 1.f ? ox : powf(ox, power));
  const float ia = imp_a * px;
  const float ib = 1.f - imp_b * po;
  const float iy = ix < mid ? ia : ib;
  float imp = dmin + iy * (dmax - dmin);
  imp = fminf(fmaxf(imp, dmin), dmax);
  if (ix > 1.f) imp = dmax;
  return imp;
}
// of the contact rows, and of the rows of joint limits and dry friction
__device__ __forceinline__ float impedance(const ModelHead& m, float pos) {
  return impedance_of(pos, m.dmin, m.dmax, m.width_inv, m.mid, m.power, m.imp_a, m.imp_b);
}
__device__ __forceinline__ float impedance_dof(const ModelHead& m, float pos) {
  return impedance_of(pos, m.dr_dmin, m.dr_dmax, m.dr_width_inv, m.dr_mid, m.dr_power, m.dr_imp_a, m.dr_imp_b);
}

// The rows a dof lane carries itself: the violated limit of its hinge (J = lim_s e_j, lim_s = +-1, 0 when none) and its
// dry friction (J = e_j, force clipped at +-fr_fl, 0 when none).  All zero on lanes that hold no dof.
struct DofRows {
  float lim_s, lim_aref, lim_D, fr_fl, fr_aref, fr_D, fr_rf;  // fr_rf = fr_fl / fr_D, where the friction force saturates
};

// Cost of the lane's rows at acceleration qa; their force on the dof, their Hessian diagonal and which of them are in
// their quadratic zone (bit 0 limit, bit 1 friction).
__device__ __forceinline__ float dofrow_eval(const DofRows& r, float qa, float& force, float& hdiag, int& zone) {
  float cost = 0.f;
  force = 0.f; hdiag = 0.f; zone = 0;
  const float xl = r.lim_s * qa - r.lim_aref;
  if (r.lim_s != 0.f && xl < 0.f) {
    cost = 0.5f * r.lim_D * xl * xl; force = -r.lim_D * xl * r.lim_s; hdiag = r.lim_D; zone = 1;
  }
  if (r.fr_fl > 0.f) {
    const float xf = qa - r.fr_aref, rf = r.fr_rf;
    if (xf <= -rf) { cost += r.fr_fl * (-0.5f * rf - xf); force += r.fr_fl; }
    else if (xf >= rf) { cost += r.fr_fl * (-0.5f * rf + xf); force -= r.fr_fl; }
    else { cost += 0.5f * r.fr_D * xf * xf; force -= r.fr_D * xf; hdiag += r.fr_D; zone |= 2; }
  }
  return cost;
}

// Coefficients of the rows' cost along qa + alpha s, in the zones the rows are in at that alpha.
__device__ __forceinline__ void dofrow_quad(const DofRows& r, float qa, float sdir, float alpha, float& t0, float& t1,
                                            float& t2) {
  t0 = 0.f; t1 = 0.f; t2 = 0.f;
  const float x0 = r.lim_s * qa - r.lim_aref, jv = r.lim_s * sdir;
  if (r.lim_s != 0.f && x0 + alpha * jv < 0.f) {
    t0 = 0.5f * x0 * x0 * r.lim_D; t1 = jv * x0 * r.lim_D; t2 = 0.5f * jv * jv * r.lim_D;
  }
  if (r.fr_fl > 0.f) {
    const float f0 = qa - r.fr_aref, rf = r.fr_rf, x = f0 + alpha * sdir;
    if (x <= -rf) { t0 += r.fr_fl * (-0.5f * rf - f0); t1 -= r.fr_fl * sdir; }
    else if (x >= rf) { t0 += r.fr_fl * (-0.5f * rf + f0); t1 += r.fr_fl * sdir; }
    else { t0 += 0.5f * f0 * f0 * r.fr_D; t1 += sdir * f0 * r.fr_D; t2 += 0.5f * sdir * sdir * r.fr_D; }
  }
}

__device__ __forceinline__ bool in_bracket(const LsPoint& x, const LsPoint& y) {
  return ((x.d0 < y.d0) && (y.d0 < 0.f)) || ((x.d0 > y.d0) && (y.d0 > 0.f));
}

// ---------------------------------------------------------------- line search over contact rows (at most 32 of them)
// Three step lengths are evaluated at once: the 16-lane groups 0, 1, 2 hold copies of the rows (rows 16..31 as a second set in
// the same lanes) and take one step length each, so the sums of the constant, linear and quadratic coefficients are three
// independent DPP reductions within the groups, and cost, slope and the Newton estimate of the next step length are formed
// for all three points by the same instructions.  What comes out is read into scalar registers as bit patterns, and the
// bracket is kept there: comparisons of slopes are integer comparisons of sign and magnitude on the scalar unit, which
// neither occupies the vector issue port nor puts its latency behind vector compares.  The search is the longest part of the
// wavefronts that a launch ends with (up to eight iterations of it per Newton step): evaluating the points one after the other
// and bracketing on the vector unit, it was 34 % of their time.
struct LsBits {  // a point of the search: step length, cost, slope, Newton estimate of the next step length
  int alpha, cost, d0, next;
};

__device__ __forceinline__ float bits_f(int b) { return __builtin_bit_cast(float, b); }
__device__ __forceinline__ int lane_bits(float x, int lane) { return __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane); }

__device__ __forceinline__ float line_search_rows(int iterations, int nefc, int lane, float Jaref, float jv, float D, float g0, float g1,
                                                  float g2, float gtol) {
  const int grp = lane >> 4, r = lane & 15;
  const bool two = nefc > 16;  // wave-uniform
  const float j1 = __shfl(Jaref, r), v1 = __shfl(jv, r), D1 = __shfl(D, r);
  const float a0 = 0.5f * j1 * j1 * D1, a1 = v1 * j1 * D1, a2 = 0.5f * v1 * v1 * D1;
  float j2 = 0.f, v2 = 0.f, b0 = 0.f, b1 = 0.f, b2 = 0.f;
  if (two) {
    j2 = __shfl(Jaref, 16 + r); v2 = __shfl(jv, 16 + r);
    const float D2 = __shfl(D, 16 + r);
    b0 = 0.5f * j2 * j2 * D2; b1 = v2 * j2 * D2; b2 = 0.5f * v2 * v2 * D2;
  }
  float al, cost, slope, next;  // of the lane's group, in its lane 15
  auto eval = [&](float step) {
    al = step;
    const bool on1 = j1 + al * v1 < 0.f;  // rows beyond nefc carry zeros
    float x0 = on1 ? a0 : 0.f, x1 = on1 ? a1 : 0.f, x2 = on1 ? a2 : 0.f;
    if (two) {
      const bool on2 = j2 + al * v2 < 0.f;
      x0 += on2 ? b0 : 0.f; x1 += on2 ? b1 : 0.f; x2 += on2 ? b2 : 0.f;
    }
    x0 += dpp_shift<0x111, 0xf>(x0); x1 += dpp_shift<0x111, 0xf>(x1); x2 += dpp_shift<0x111, 0xf>(x2);
    asm("s_nop 1\n\t" KS_SUM_STEP("row_shr:2 " KS_ROW) KS_SUM_STEP("row_shr:4 " KS_ROW) KS_SUM_STEP("row_shr:8 " KS_ROW) : "+v"(x0), "+v"(x1), "+v"(x2));
    // lane 15 of each group holds the group's totals; the other lanes carry numbers nobody reads
    const float q0 = g0 + x0, q1 = g1 + x1, q2 = g2 + x2;
    cost = al * al * q2 + al * q1 + q0;
    const float d0 = 2.f * al * q2 + q1, d1 = 2.f * q2 + (q2 == 0.f ? 1e-15f : 0.f);
    // Newton estimate of the step length: d0 / d1 by reciprocal and product (1 ulp), a tenth of a division's instructions
    next = al - d0 * __builtin_amdgcn_rcpf(d1);
    slope = d0 == d0 ? d0 : 0.f;  // a NaN takes part in no bracket
  };
  auto fetch = [&](LsBits& p, int at) { p = {lane_bits(al, at), lane_bits(cost, at), lane_bits(slope, at), lane_bits(next, at)}; };
  LsBits p0, lo, hi;
  eval(0.f);
  fetch(p0, 15);
  eval(bits_f(p0.next));
  if (bits_f(lane_bits(slope, 15)) < bits_f(p0.d0)) { fetch(lo, 15); hi = p0; } else { fetch(hi, 15); lo = p0; }
  const unsigned tol = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, fmaxf(gtol, 0.f)));  // bits of a number >= 0 order like the number
  for (int it = 0; it < iterations; ++it) {
    const unsigned ml = (unsigned)lo.d0 & 0x7fffffffu, mh = (unsigned)hi.d0 & 0x7fffffffu;
    if ((lo.d0 < 0) & (ml != 0u) & (ml < tol)) break;  // the slope at lo is negative and within the tolerance
    if ((hi.d0 > 0) & (mh < tol)) break;               // that at hi positive and within it
    eval(grp == 0 ? bits_f(lo.next) : (grp == 1 ? bits_f(hi.next) : 0.5f * (bits_f(lo.alpha) + bits_f(hi.alpha))));
    const int s0 = lane_bits(slope, 15), s1 = lane_bits(slope, 31), s2 = lane_bits(slope, 47);
    // Each end of the bracket moves to the candidate whose slope has its sign and is the nearest to zero, if one is nearer than its
    // own (and not zero).  Magnitude - 1 as an unsigned number puts a zero slope last; a tie goes to the candidate asked first.
    const unsigned m0 = ((unsigned)s0 & 0x7fffffffu) - 1u, m1 = ((unsigned)s1 & 0x7fffffffu) - 1u, m2 = ((unsigned)s2 & 0x7fffffffu) - 1u;
    const unsigned own_l = ml ? ml - 1u : 0u, own_h = mh ? mh - 1u : 0u;
    const unsigned l0 = (s0 ^ lo.d0) < 0 ? ~0u : m0, l1 = (s1 ^ lo.d0) < 0 ? ~0u : m1, l2 = (s2 ^ lo.d0) < 0 ? ~0u : m2;
    const unsigned h0 = (s0 ^ hi.d0) < 0 ? ~0u : m0, h1 = (s1 ^ hi.d0) < 0 ? ~0u : m1, h2 = (s2 ^ hi.d0) < 0 ? ~0u : m2;
    const unsigned bl = min(l0, min(l1, l2)), bh = min(h0, min(h1, h2));
    const bool move_l = bl < own_l, move_h = bh < own_h;
    if (!(move_l | move_h)) break;
    if (move_l) fetch(lo, bl == l0 ? 15 : (bl == l2 ? 47 : 31));  // asked in the order lo's estimate, middle, hi's estimate
    if (move_h) fetch(hi, bh == h1 ? 31 : (bh == h2 ? 47 : 15));  // hi's estimate, middle, lo's
  }
  const float cl = bits_f(lo.cost), ch = bits_f(hi.cost), c0 = bits_f(p0.cost);
  const bool improved = (cl < c0) || (ch < c0);
  return improved ? (cl < ch ? bits_f(lo.alpha) : bits_f(hi.alpha)) : 0.f;
}

// sum of one component over a contiguous subtree range of an array with `w` floats per body; four reads in flight at a time
// (the root's range is every body: read by read it is twenty LDS latencies in a row)
__device__ __forceinline__ float range_sum(const float* base, int w, int b, int e) {
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  const float* p = base + w * b;
  int left = e - b;
  for (; left >= 4; left -= 4, p += 4 * w) {
    const float x0 = p[0], x1 = p[w], x2 = p[2 * w], x3 = p[3 * w];
    s0 += x0; s1 += x1; s2 += x2; s3 += x3;
  }
  if (left > 0) {
    const float x0 = p[0], x1 = p[left > 1 ? w : 0], x2 = p[left > 2 ? 2 * w : 0];
    s0 += x0;
    s1 += left > 1 ? x1 : 0.f;
    s2 += left > 2 ? x2 : 0.f;
  }
  return (s0 + s1) + (s2 + s3);
}

// ------------------------------------------------------------------------------------------- the fused kernel
// FWD = true is the forward-only variant (derived fields + warm start of a given state, no actuation, no
// integration) that replaces the mjx.forward of a reset.
template <bool FWD, int NP, bool DR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KS_STEP_WAVES, KS_STEP_WAVES)))
void step_kernel(StepArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds_raw[];
  const DevModel& m = *a.model;
  const ModelHead& mh = a.head;
  const int lane = threadIdx.x;
  // heaviest envs first when an order is given (ks_work_order, which also keeps neighbouring envs on one XCD); without
  // one, workgroup b takes env (b % 8) (N / 8) + b / 8 for the same reason
  int64_t env = blockIdx.x;
  if (a.env_order) env = a.env_order[blockIdx.x];
  else if (a.N % 8 == 0) env = (int64_t)(blockIdx.x % 8) * (a.N / 8) + blockIdx.x / 8;
  if (a.env_mask && !a.env_mask[env]) return;  // wave-uniform
  int work = 0;  // wave-uniform cost estimate of this control step
  const int nb = mh.nb, nq = mh.nq, nv = mh.nv, nu = mh.nu, ns = mh.ns;
  constexpr int nvs = stride_of(NP), js = nvs;
  Lds l = carve<NP>(lds_raw, lds_raw, nb, nq, nv, nu, ns);
  const int rq = mh.root_free ? 7 : 0;
  const int rv = rq ? 6 : 0;

  for (int i = lane; i < nq; i += 64) l.qpos[i] = a.qpos[env * nq + i];
  if (lane < 32) l.qvel[lane] = lane < nv ? a.qvel[env * nv + lane] : 0.f;
  if (lane < nv) l.warm[lane] = a.qacc_warmstart ? a.qacc_warmstart[env * nv + lane] : 0.f;
  // The mass matrix: a substep writes the entries that couple dofs of one chain, the same ones every time; everything else is
  // written here, once per launch (zero, and one on the diagonal of the padding rows).
  for (int i = lane; i < NP * nvs / 4; i += 64) reinterpret_cast<float4*>(l.M)[i] = {0.f, 0.f, 0.f, 0.f};
  KS_SYNC();
  if (lane >= nv && lane < NP) l.M[lane * nvs + lane] = 1.f;
  for (int i = lane; i < nu; i += 64) l.tau[i] = a.ctrl_in ? a.ctrl_in[env * nu + i] : 0.f;
  for (int i = lane; i < nb; i += 64) l.sub_end[i] = m.body_subtree_end[i];
  if (lane == 0) {  // world body
    for (int k = 0; k < 3; ++k) l.xpos[k] = 0.f;
    l.xquat[0] = 1.f; l.xquat[1] = l.xquat[2] = l.xquat[3] = 0.f;
    for (int k = 0; k < 6; ++k) l.cvel[k] = 0.f;
  }
  const float mu = a.friction ? a.friction[env] : mh.friction;
  const float latency = a.latency ? a.latency[env] : 0.f;
  const float scale = 1.0f / (mh.meaninertia * (float)(nv > 1 ? nv : 1));
  KS_SYNC();
#ifdef KS_PROFILE
  float prof[16];
  for (int k = 0; k < 16; ++k) prof[k] = 0.f;
  long long t_last = clock64();
#endif

  const int nsub = FWD ? 1 : a.substeps;
  int act_wait = 0;  // substeps until the next actuator update
  // An env that the termination pass has just reset still owes the forward pass of its reset (engine.py:213: derived
  // quantities and the warm start of the new episode, from the reset state with zero controls).  With `fresh` given the
  // step does it itself, as a pass `sub = -1` that neither actuates nor integrates, instead of a masked launch of the
  // forward-only kernel between the termination pass and this step.
  const bool fresh_env = !FWD && a.fresh && a.fresh[env];  // wave-uniform
  // The arguments, and the sizes and LDS offsets that follow from them, are taken afresh in each substep and in the
  // write-back: `s_load`s through the scalar cache and a little scalar arithmetic.  Taken once, the ~60 pointers, sizes and
  // offsets stay live across the solver, which leaves SGPRs for a third of them: the rest lay in VGPR lanes (194
  // `v_writelane`s and ~280 `v_readlane`s, all of them VALU work, and two VGPRs of a file that is full; now 38 of the former; three
  // VGPRs of the 28-dof instance spill, 768 B of scratch an env and step).  4096 humanoid envs: 82.4 M -> 79.1 M VALU
  // instructions a launch, 253.3 -> 246.6 us; the pointers alone, without sizes and offsets, 248.1 us.
  const auto arguments = []() -> const StepArgs& {
    typedef const __attribute__((address_space(4))) StepArgs* ArgsPtr;
    ArgsPtr p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();  // the kernel's one parameter lies at its start
    asm volatile("" : "+s"(p));
    return *(const StepArgs*)p;
  };
  const auto load_lane = [env](const StepArgs& a, LaneIn& in) __attribute__((always_inline)) {
    const DevModel& m = *a.model;
    const int nb = a.head.nb, nv = a.head.nv, ns = a.head.ns;
    int lane = threadIdx.x;
    asm volatile("" : "+v"(lane));
    uint4* dst = reinterpret_cast<uint4*>(&in.rec);
#pragma unroll
    for (int k = 0; k < kRecPieces; ++k) dst[k] = *reinterpret_cast<const uint4*>(m.lane_rec[k][lane]);
    // the row of an optional operand: this env's, or row 0 of what stands in for it
    auto row_of = [&](unsigned bit) -> int64_t { return (a.given & bit) ? env : 0; };
    const int bl = lane < nb ? lane : 0, dl = lane < nv ? lane : 0, sl = lane < ns ? lane : 0;
    in.ipos = ld3(a.body_ipos + (row_of(kOptIpos) * nb + bl) * 3);
    in.inertia = ld3(a.body_inertia + (row_of(kOptInertia) * nb + bl) * 3);
    in.mass_scale = a.mass_scale[row_of(kOptMass) * nb + bl];
    in.damping_scale = a.damping_scale[row_of(kOptDamping) * nv + dl];
    in.armature_scale = a.armature_scale[row_of(kOptArmature) * nv + dl];
    in.sph_pos = ld3(a.sph_pos + (row_of(kOptSphere) * ns + sl) * 3);
    in.sph_radius = a.sph_radius[row_of(kOptSphere) * ns + sl];
  };
  LaneIn in;
  load_lane(arguments(), in);
  for (int sub = fresh_env ? -1 : 0; sub < nsub; ++sub) {
    const StepArgs& a = arguments();
    const DevModel& m = *a.model;
    const ModelHead& mh = a.head;
    const int nb = mh.nb, nq = mh.nq, nv = mh.nv, nu = mh.nu, ns = mh.ns;
    Lds l = carve<NP>(lds_raw, lds_raw, nb, nq, nv, nu, ns);
    const int rq = mh.root_free ? 7 : 0;
    const int rv = rq ? 6 : 0;
    // One word says which operands are given and which outputs wanted.  It is asked all over the substep; a pointer compared with zero
    // where it is needed is a scalar load that the wavefront waits for, a dozen of them a substep.  With the solver's limits taken
    // together as well (below), and the line search's sums side by side in assembly: control steps of 64 and of 1024 K-Bots and of an LSTM
    // policy's 0.4 % faster, of 4096 humanoids' the same.
    unsigned given = a.given;
    asm volatile("" : "+s"(given));  // here, not where it is used
    const bool fwd = FWD || sub < 0;
    // The lane id is re-materialised per substep so that per-lane LDS addresses are recomputed inside the loop
    // instead of being hoisted out of it into ~130 long-lived registers (which would halve the occupancy).
    int lane_v = threadIdx.x;
    asm volatile("" : "+v"(lane_v));
    const int lane = lane_v;
    // ---- the lane's constants, as the end of the last substep has requested them
    const bool is_body = lane > 0 && lane < nb;
    const bool is_dof = lane < nv;
    const bool is_sph = lane < ns;
    const LaneRec& rec = in.rec;
    // the row of an optional operand: this env's, or row 0 of what stands in for it
    auto row_of = [&](unsigned bit) -> int64_t { return (given & bit) ? env : 0; };
    const int b_jtype = rec.b_jtype, b_qadr = rec.b_qadr, b_dofadr = rec.b_dofadr, b_depth = rec.b_depth;
    const V3 b_pos = {rec.b_pos[0], rec.b_pos[1], rec.b_pos[2]};
    const V3 b_ipos = in.ipos, b_inertia = in.inertia;
    const V3 b_jaxis = {rec.b_jaxis[0], rec.b_jaxis[1], rec.b_jaxis[2]}, b_jpos = {rec.b_jpos[0], rec.b_jpos[1], rec.b_jpos[2]};
    const Quat b_quat = {rec.b_quat[0], rec.b_quat[1], rec.b_quat[2], rec.b_quat[3]};
    const Quat b_iquat = {rec.b_iquat[0], rec.b_iquat[1], rec.b_iquat[2], rec.b_iquat[3]};
    const float b_q0 = rec.b_q0;
    const float b_mass = is_body ? rec.b_mass * in.mass_scale : 0.f;
    const int d_body = rec.d_body, d_act = rec.d_act, d_jtype = rec.d_jtype, d_k = rec.d_k;
    const float d_damping = rec.d_damping * in.damping_scale;
    const float d_armature = rec.d_armature * in.armature_scale;
    const float d_gear = rec.d_gear, d_lo = rec.d_lo, d_hi = rec.d_hi;
    const int s_body = rec.s_body;
    const V3 s_pos = in.sph_pos;
    const float s_rad = in.sph_radius;
    const float s_invw = rec.s_invw;
    const unsigned s_mask = rec.s_mask;
    unsigned chain[kMaxDepth / 2];
#pragma unroll
    for (int k = 0; k < kMaxDepth / 2; ++k) chain[k] = rec.b_chain[k];
    int pk[kPairSets];
#pragma unroll
    for (int k = 0; k < kPairSets; ++k) pk[k] = rec.pk[k];

    // ---- actuators (ksim/engine.py:287-320, ksim/actuators.py:198-217)
    const bool actuate = !fwd && act_wait == 0;
    if (!fwd) act_wait = (act_wait == 0 ? a.actuator_period : act_wait) - 1;
    if (actuate && lane < nu) {
      const int u = lane;
      // the actuator inputs of this control step are read again at every actuator update (they stay in the caches):
      // held in registers they would be live across the solver of every substep
      const bool posvel = a.actuator_type == KS_ACT_POSITION_VELOCITY;
      const int na = posvel ? 2 * nu : nu;  // width of the action vector
      const int64_t ea = env * na + lane, srow = (int64_t)sub * a.N + env;
      const int64_t noise_a = ((given & kOptActionNoise) ? srow : 0) * na + u, noise_t = ((given & kOptTorqueNoise) ? srow : 0) * nu + u;
      const float u_last = a.last_ctrl[ea], u_act = a.action[ea];
      const int64_t drop_at = row_of(kOptDrop) * na + u;
      const bool u_drop = a.drop[drop_at] != 0;
      const float u_kp = a.kp[lane] * a.kp_scale[row_of(kOptKp)];
      const float u_kd = a.kd[lane] * a.kd_scale[row_of(kOptKd)];
      const float u_lim = a.ctrl_clip[lane] * a.torque_limit_scale[row_of(kOptLimit)];
      const float u_zero = a.zero_offset[row_of(kOptZero) * nu + u];
      const float u_abias = a.action_bias[row_of(kOptActionBias) * nu + u], u_tbias = a.torque_bias[row_of(kOptTorqueBias) * nu + u];
      const float u_anoise = a.action_noise[noise_a], u_tnoise = a.torque_noise[noise_t];
      float prct = (float)sub - latency;
      prct = fminf(fmaxf(prct, 0.f), 1.f);
      const float c = u_drop ? u_last : u_last * (1.0f - prct) + u_act * prct;
      float t;
      if (a.actuator_type == KS_ACT_TORQUE) {
        t = c + u_tnoise;
      } else {
        float target_vel = 0.f;
        if (posvel) {  // the velocity targets ride in the second half of the action vector
          const float v_last = a.last_ctrl[ea + nu], v_act = a.action[ea + nu];
          const bool v_drop = a.drop[drop_at + nu] != 0;
          target_vel = (v_drop ? v_last : v_last * (1.0f - prct) + v_act * prct) + a.action_noise[noise_a + nu];
        }
        const float target = c * a.action_scale + u_anoise + u_abias;
        const float q = l.qpos[rq + u] - u_zero;
        t = u_kp * (target - q) + u_kd * (target_vel - l.qvel[rv + u]);
        t = t + u_tnoise + u_tbias;
        t = fminf(fmaxf(t, -u_lim), u_lim);
      }
      l.tau[u] = t;
    }

    // ---- events (ksim/engine.py:322-333, ksim/events.py): impulses on the root velocity when an interval runs out
    if (!fwd && (given & kHasEvents)) {
      const uint64_t ev_step = a.event_rng.step + (a.event_rng.step_base ? *a.event_rng.step_base : 0ull);
#pragma nounroll
      for (int e = 0; e < a.n_events; ++e) {  // a rolled loop: nothing of the event records is kept across the substeps
        if (a.events[e].kind != KS_EVENT_FORCE_PUSH) {
          const KsEventDesc ev = a.events[e];
          // the timer stays in memory between substeps (lane 0 owns it) so that it costs no register over the solver
          float* tleft = a.event_state + (int64_t)e * a.N + env;
          float left = lane_bcast(lane == 0 ? *tleft : 0.f, 0) - mh.dt;
          if (left <= 0.f) {  // wave-uniform
            float u0, u1, u2;
            if (a.event_uniform) {
              const float* u = a.event_uniform + (((int64_t)sub * a.N + env) * a.n_events + e) * KS_EVENT_DRAWS;
              u0 = u[0]; u1 = u[1]; u2 = u[2];
            } else {
              const Philox4 r = draw(a.event_rng.seed, ev_step, kRngEvent, (uint64_t)env, (uint32_t)(sub * KS_MAX_EVENTS + e));
              u0 = u01(r.x); u1 = u01(r.y); u2 = u01(r.z);
            }
            if (lane == 0) {
              if (ev.kind == KS_EVENT_LINEAR_PUSH) {
                const float th = 6.28318530717958647692f * u0, mag = (ev.lo + u1 * (ev.hi - ev.lo)) * ev.mag * ev.level_scale;
                l.qvel[0] += cosf(th) * mag;
                l.qvel[1] += sinf(th) * mag;
              } else if (ev.kind == KS_EVENT_ANGULAR_PUSH) {
                const float mag = (ev.lo + u1 * (ev.hi - ev.lo)) * ev.mag;
                l.qvel[5] += (u0 < 0.5f ? -mag : mag) * ev.level_scale;
              } else if (ev.kind == KS_EVENT_JUMP) {
                const float h = (ev.lo + u0 * (ev.hi - ev.lo)) * ev.level_scale;
                for (int k = 0; k < 3; ++k) l.qvel[k] += sqrtf(2.f * -mh.gravity[k] * h);
              }
            }
            left = ev.interval_lo + u2 * (ev.interval_hi - ev.interval_lo);
          }
          if (lane == 0) *tleft = left;
        }
      }
      KS_SYNC();
    }

    KS_PHASE(0)
    // ---- kinematics.  Every body first writes its pose relative to its parent (joint rotation included) to
    // LDS, then composes the poses along its own chain of ancestors from the root down: max_depth short
    // steps shared by all bodies instead of one full pass per tree level.
    V3 xipos = {0.f, 0.f, 0.f};
    Mat3 ximat;
#pragma unroll
    for (int k = 0; k < 9; ++k) ximat.m[k] = 0.f;
    float* lpose = l.cinert;  // 7 floats per body; the inertia scratch is not in use yet
    if (is_body) {
      V3 tl;
      Quat ql;
      if (b_jtype == kJntFree) {
        tl = ld3(l.qpos + b_qadr);
        ql = qnormalize({l.qpos[b_qadr + 3], l.qpos[b_qadr + 4], l.qpos[b_qadr + 5], l.qpos[b_qadr + 6]});
      } else {
        tl = b_pos;
        ql = b_quat;
        if (b_jtype == kJntHinge) {
          float hs, hc;
          sincosf(0.5f * (l.qpos[b_qadr] - b_q0), &hs, &hc);
          const Quat jr = {hc, b_jaxis.x * hs, b_jaxis.y * hs, b_jaxis.z * hs};
          // rotation about the joint anchor: p + R_b (a - R_j a) with a the anchor in the body frame
          const V3 arm = qrot(jr, V3{-b_jpos.x, -b_jpos.y, -b_jpos.z}, b_jpos);
          tl = qrot(b_quat, arm, b_pos);
          ql = qmul(b_quat, jr);
        }
      }
      st3(lpose + 7 * lane, tl);
      lpose[7 * lane + 3] = ql.w; lpose[7 * lane + 4] = ql.x; lpose[7 * lane + 5] = ql.y; lpose[7 * lane + 6] = ql.z;
    }
    KS_SYNC();
    {
      V3 pos = {0.f, 0.f, 0.f};
      Quat quat = {1.f, 0.f, 0.f, 0.f};
      // two links per step: both poses are on their way from LDS before the first is needed
      unsigned ch[kMaxDepth / 2];
#pragma unroll
      for (int k = 0; k < kMaxDepth / 2; ++k) ch[k] = chain[k];
      for (int k = 0; k < mh.max_depth; k += 2) {
        const float* p0 = lpose + 7 * (int)(ch[0] & 31u);
        const float* p1 = lpose + 7 * (int)((ch[0] >> 16) & 31u);
        const V3 t0 = ld3(p0), t1 = ld3(p1);
        const Quat q0 = {p0[3], p0[4], p0[5], p0[6]}, q1 = {p1[3], p1[4], p1[5], p1[6]};
        if (k < b_depth) {
          pos = qrot(quat, t0, pos);
          quat = qmul(quat, q0);
        }
        if (k + 1 < b_depth) {
          pos = qrot(quat, t1, pos);
          quat = qmul(quat, q1);
        }
#pragma unroll
        for (int i = 0; i + 1 < kMaxDepth / 2; ++i) ch[i] = ch[i + 1];
      }
      if (is_body) {
        quat = qnormalize(quat);
        const Mat3 R = q2mat(quat);
        V3 anchor = pos, axis = {0.f, 0.f, 1.f};
        if (b_jtype == kJntHinge) {
          anchor = pos + mul(R, b_jpos);
          axis = mul(R, b_jaxis);
        }
        st3(l.xpos + 3 * lane, pos);
        l.xquat[4 * lane] = quat.w; l.xquat[4 * lane + 1] = quat.x; l.xquat[4 * lane + 2] = quat.y; l.xquat[4 * lane + 3] = quat.z;
        st3(l.xanchor + 3 * lane, anchor);
        st3(l.xaxis + 3 * lane, axis);
        xipos = pos + mul(R, b_ipos);
        ximat = q2mat(qnormalize(qmul(quat, b_iquat)));
      }
    }
    KS_SYNC();

    KS_PHASE(1)
    // ---- centre of mass of the tree (wave-uniform), com-based inertias and motion axes
    float mt = b_mass;
    V3 com = xipos * b_mass;
    wave_sums(mt, com.x, com.y, com.z);
    com = com * (mt > 1e-15f ? 1.0f / mt : 0.f);
    if (lane == 0) {  // world body entries of the per-substep scratch (the scratch is reused by J later)
      for (int k = 0; k < 10; ++k) l.cinert[k] = 0.f;
      for (int k = 0; k < 6; ++k) l.cfrc[k] = 0.f;
    }
    float ci[10];
    {
      const float* R = ximat.m;
      const float I0 = b_inertia.x, I1 = b_inertia.y, I2 = b_inertia.z;
      const V3 d = xipos - com;
      const float d2 = dot(d, d);
      ci[0] = R[0] * I0 * R[0] + R[1] * I1 * R[1] + R[2] * I2 * R[2] + b_mass * (d2 - d.x * d.x);
      ci[1] = R[3] * I0 * R[3] + R[4] * I1 * R[4] + R[5] * I2 * R[5] + b_mass * (d2 - d.y * d.y);
      ci[2] = R[6] * I0 * R[6] + R[7] * I1 * R[7] + R[8] * I2 * R[8] + b_mass * (d2 - d.z * d.z);
      ci[3] = R[0] * I0 * R[3] + R[1] * I1 * R[4] + R[2] * I2 * R[5] - b_mass * d.x * d.y;
      ci[4] = R[0] * I0 * R[6] + R[1] * I1 * R[7] + R[2] * I2 * R[8] - b_mass * d.x * d.z;
      ci[5] = R[3] * I0 * R[6] + R[4] * I1 * R[7] + R[5] * I2 * R[8] - b_mass * d.y * d.z;
      ci[6] = b_mass * d.x; ci[7] = b_mass * d.y; ci[8] = b_mass * d.z;
      ci[9] = b_mass;
      if (is_body) {
#pragma unroll
        for (int k = 0; k < 10; ++k) l.cinert[10 * lane + k] = ci[k];
        if ((given & kOutCinert) && sub == nsub - 1) {  // the LDS copy is scratch that the constraint rows reuse: export it here
#pragma unroll
          for (int k = 0; k < 10; ++k) a.cinert[((int64_t)env * nb + lane) * 10 + k] = ci[k];
        }
      }
      if ((given & kOutCinert) && sub == nsub - 1 && lane == 0)
        for (int k = 0; k < 10; ++k) a.cinert[(int64_t)env * nb * 10 + k] = 0.f;  // world body
    }
    Sp my_cdof = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
    if (is_dof) {
      const V3 off = com - ld3(l.xanchor + 3 * d_body);
      if (d_jtype == kJntFree) {
        if (d_k < 3) {
          my_cdof.l = {d_k == 0 ? 1.f : 0.f, d_k == 1 ? 1.f : 0.f, d_k == 2 ? 1.f : 0.f};
        } else {
          const V3 ax = qrot({l.xquat[4 * d_body], l.xquat[4 * d_body + 1], l.xquat[4 * d_body + 2], l.xquat[4 * d_body + 3]},
                             V3{d_k == 3 ? 1.f : 0.f, d_k == 4 ? 1.f : 0.f, d_k == 5 ? 1.f : 0.f}, V3{0.f, 0.f, 0.f});
          my_cdof = {ax, cross(ax, off)};
        }
      } else {
        const V3 ax = ld3(l.xaxis + 3 * d_body);
        my_cdof = {ax, cross(ax, off)};
      }
      st6(l.cdof + 6 * lane, my_cdof);
    }
    KS_SYNC();

    KS_PHASE(2)
    // ---- composite inertias (subtree = contiguous body range) and the mass matrix
    for (int idx = lane; idx < nb * 10; idx += 64) {
      const int b = idx * 205 >> 11, k = idx - 10 * b;  // idx / 10 below 1024
      l.crb[idx] = b > 0 ? range_sum(l.cinert + k, 10, b, l.sub_end[b]) : 0.f;
    }
    KS_SYNC();
    if (is_dof) {
      const Sp f = inert_mul(l.crb + 10 * d_body, my_cdof);
      st6(l.buf + 6 * lane, f);
      l.M[lane * nvs + lane] = dot(my_cdof, f) + d_armature;
    }
    KS_SYNC();
#pragma unroll
    for (int k0 = 0; k0 < kPairSets; k0 += 4) {  // four sets of 64 pairs: all their reads before the first write
      if (64 * k0 >= mh.npairs) break;
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int p = max(pk[k0 + k], 0);
        v[k] = dot(ld6(l.cdof + 6 * (p & 0xff)), ld6(l.buf + 6 * (p >> 8)));
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (pk[k0 + k] >= 0) {
          const int i = pk[k0 + k] >> 8, j = pk[k0 + k] & 0xff;
          l.M[i * nvs + j] = v[k];
          l.M[j * nvs + i] = v[k];
        }
    }

    KS_PHASE(3)
    // ---- body velocities and bias accelerations: the motion axes are all expressed in one frame, so every
    // body accumulates them over the dofs of its own ancestor chain, root first (no pass per tree level)
    {
      Sp v = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
      Sp acc = {{0.f, 0.f, 0.f}, {-mh.gravity[0], -mh.gravity[1], -mh.gravity[2]}};
      auto hinge = [&](const Sp& cd, float qd) {
        acc = acc + cross_motion(v, cd) * qd;
        v = v + cd * qd;
      };
      auto link = [&](unsigned e, const Sp& cd0, float qd0) {  // cd0, qd0: axis and velocity of the link's first dof
        if (e & (1u << 10)) {
          hinge(cd0, qd0);
        } else if (e & (1u << 11)) {
          const int da = (int)((e >> 5) & 31u);
          // the translations' axes are the world's, and the three rotations act on one velocity, so their sum does
          v.l = v.l + V3{qd0, l.qvel[da + 1], l.qvel[da + 2]};
          const Sp dv = ld6(l.cdof + 6 * (da + 3)) * l.qvel[da + 3] + ld6(l.cdof + 6 * (da + 4)) * l.qvel[da + 4] +
                        ld6(l.cdof + 6 * (da + 5)) * l.qvel[da + 5];
          acc = acc + cross_motion(v, dv);
          v = v + dv;
        }
      };
      for (int k = 0; k < mh.max_depth; k += 2) {
        const unsigned e0 = chain[0] & 0xffffu, e1 = chain[0] >> 16;
        const int d0 = (int)((e0 >> 5) & 31u), d1 = (int)((e1 >> 5) & 31u);
        const Sp c0 = ld6(l.cdof + 6 * d0), c1 = ld6(l.cdof + 6 * d1);
        const float v0 = l.qvel[d0], v1 = l.qvel[d1];
        if (k < b_depth) link(e0, c0, v0);
        if (k + 1 < b_depth) link(e1, c1, v1);
#pragma unroll
        for (int i = 0; i + 1 < kMaxDepth / 2; ++i) chain[i] = chain[i + 1];
      }
      Sp cf = inert_mul(ci, acc) + cross_force(v, inert_mul(ci, v));
      // ---- force pushes (ksim/events.py:240-365): a wrench held on one body enters the Newton-Euler pass as an
      // external force on that body, so the subtree sums and the projection on the motion axes below turn it into
      // the generalised force J^T f.  Lane 0 owns the state in memory; the other lanes get it by broadcast.
      if (!fwd && (given & kHasForceEvents)) {
        const uint64_t ev_step = a.event_rng.step + (a.event_rng.step_base ? *a.event_rng.step_base : 0ull);
        Sp ext = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
#pragma nounroll
        for (int e = 0; e < a.n_events; ++e) {
          if (a.events[e].kind != KS_EVENT_FORCE_PUSH) continue;
          const KsEventDesc ev = a.events[e];
          float* st = a.event_force + ((int64_t)e * a.N + env) * KS_EVENT_FORCE_STATE;
          float* tleft = a.event_state + (int64_t)e * a.N + env;
          float s7[7];
#pragma unroll
          for (int k = 0; k < 7; ++k) s7[k] = lane_bcast(lane == 0 ? st[k] : 0.f, 0);
          float dur = s7[0] - mh.dt, left = lane_bcast(lane == 0 ? *tleft : 0.f, 0) - mh.dt;
#pragma unroll
          for (int k = 0; k < 6; ++k) s7[1 + k] *= ev.level_scale;   // events.py:296: the carried wrench itself is rescaled
          const bool on = dur > 0.f && lane == ev.body;                // events.py:297-299, 302-307
          const V3 f = {s7[1] * ev.level_scale, s7[2] * ev.level_scale, s7[3] * ev.level_scale};
          const V3 tq = {s7[4] * ev.level_scale, s7[5] * ev.level_scale, s7[6] * ev.level_scale};
          const V3 mom = tq + cross(xipos - com, f);                    // moment about the centre of mass of the tree
          ext = {{on ? mom.x : 0.f, on ? mom.y : 0.f, on ? mom.z : 0.f}, {on ? f.x : 0.f, on ? f.y : 0.f, on ? f.z : 0.f}};
          if (left <= 0.f) {  // wave-uniform: a new wrench (events.py:320-358)
            float u[10];
            if (a.event_uniform) {
              const float* up = a.event_uniform + (((int64_t)sub * a.N + env) * a.n_events + e) * KS_EVENT_DRAWS;
#pragma unroll
              for (int k = 0; k < 10; ++k) u[k] = up[k];
            } else {
#pragma unroll
              for (int q = 0; q < 3; ++q) {
                const Philox4 r = draw(a.event_rng.seed, ev_step, kRngEvent, (uint64_t)env, (uint32_t)((sub * KS_MAX_EVENTS + e) * 4 + 1 + q));
                u[4 * q] = u01(r.x); u[4 * q + 1] = u01(r.y);
                if (q < 2) { u[4 * q + 2] = u01(r.z); u[4 * q + 3] = u01(r.w); }
              }
            }
            const V3 d0 = {2.f * u[0] - 1.f, 2.f * u[1] - 1.f, 2.f * u[2] - 1.f}, d1 = {2.f * u[4] - 1.f, 2.f * u[5] - 1.f, 2.f * u[6] - 1.f};
            const float sc = ev.lo + u[3] * (ev.hi - ev.lo);
            const float kf = sc * ev.mag / sqrtf(dot(d0, d0)), kt = sc * ev.mag2 / sqrtf(dot(d1, d1));
            const int which = min(2, (int)(3.f * u[7]));
            const float wf = which == 1 ? 0.f : kf, wt = which == 0 ? 0.f : kt;
            s7[1] = d0.x * wf; s7[2] = d0.y * wf; s7[3] = d0.z * wf;
            s7[4] = d1.x * wt; s7[5] = d1.y * wt; s7[6] = d1.z * wt;
            left = ev.interval_lo + u[8] * (ev.interval_hi - ev.interval_lo);
            dur = ev.duration_lo + u[9] * (ev.duration_hi - ev.duration_lo);
          }
          if (lane == 0) {
            *tleft = left;
            st[0] = dur;
#pragma unroll
            for (int k = 1; k < 7; ++k) st[k] = s7[k];
          }
        }
        cf = {cf.a - ext.a, cf.l - ext.l};
      }
      if (is_body) {
        st6(l.cvel + 6 * lane, v);
        st6(l.cfrc + 6 * lane, cf);
      }
    }
    KS_SYNC();
    for (int idx = lane; idx < nb * 6; idx += 64) {
      const int b = idx * 171 >> 10, k = idx - 6 * b;  // idx / 6 below 500
      l.fsub[idx] = b > 0 ? range_sum(l.cfrc + k, 6, b, l.sub_end[b]) : 0.f;
    }
    KS_SYNC();

    KS_PHASE(4)
    // ---- mass-matrix row into registers; smooth forces: passive - bias + actuator
    const float* Mrow = l.M + (is_dof ? lane : 0) * nvs;
    float qfs = 0.f, my_qvel = 0.f;
    if (is_dof) {
      my_qvel = l.qvel[lane];
      const float bias = dot(my_cdof, ld6(l.fsub + 6 * d_body));
      float f = -d_damping * my_qvel - bias;
      if (rec.d_stiffness != 0.f) f -= rec.d_stiffness * (l.qpos[rec.d_qadr] - m.qpos0[rec.d_qadr]);  // joint spring about qpos0
      if (d_act >= 0) f += d_gear * fminf(fmaxf(l.tau[d_act], d_lo), d_hi);
      qfs = f;
      if (given & kOutBias) a.dbg_bias[env * nv + lane] = bias;
#ifndef KS_PROFILE
      if (given & kOutM) for (int j = 0; j < nv; ++j) a.dbg_M[env * nv * nv + lane * nv + j] = l.M[lane * nvs + j];
#endif
    }

    KS_PHASE(5)
    // ---- contacts: sphere vs plane z = 0, compacted to the penetrating ones
    float dist = 1.f;
    V3 cpos = {0.f, 0.f, 0.f};
    if (is_sph) {
      const V3 c = qrot({l.xquat[4 * s_body], l.xquat[4 * s_body + 1], l.xquat[4 * s_body + 2], l.xquat[4 * s_body + 3]}, s_pos, ld3(l.xpos + 3 * s_body));
      dist = c.z - s_rad;
      cpos = {c.x, c.y, c.z - s_rad - 0.5f * dist};
      if (given & kOutDist) a.contact_dist[env * ns + lane] = dist;
    }
    const bool touching = is_sph && (dist < 0.f);
    const unsigned long long cmask = __ballot(touching);
    const int ncon = __popcll(cmask);
    const bool frictionless = mh.frictionless != 0;
    const int nefc = frictionless ? ncon : 4 * ncon;
    // A launch ends with its slowest wavefront, and an env with many contacts runs several times longer than an airborne
    // one: waves with more constraint rows get a higher issue priority on their SIMD, which shortens exactly those.
    if (nefc >= 20) __builtin_amdgcn_s_setprio(3);
    else if (nefc >= 12) __builtin_amdgcn_s_setprio(2);
    else if (nefc > 0) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    if (touching) {
      const int c = __popcll(cmask & ((1ull << lane) - 1ull));
      l.con_body[c] = s_body;
      l.con_mask[c] = s_mask;
      st3(l.con_off + 3 * c, cpos - com);
      const float invweight = frictionless ? s_invw : (s_invw + mu * mu * s_invw) * 2.f * mu * mu * mh.impratio_inv;
      const float imp = impedance(mh, dist);
      const float Rr = fmaxf(invweight * (1.f - imp) * __builtin_amdgcn_rcpf(imp), 1e-15f);  // imp lies in [1e-4, 1)
      l.con_D[c] = __builtin_amdgcn_rcpf(Rr);
      l.con_kip[c] = mh.con_k * imp * dist;
    }
    KS_SYNC();

    KS_PHASE(6)
    // ---- Cholesky of M and the unconstrained acceleration (registers only)
    float R[NP];
    float myinv, qas_all;
    {
      f32x16 T;
      if (lane < 32) l.vbuf[lane] = qfs;
      KS_SYNC();
      load_mtile<NP>(T, l.M, l.vbuf, lane);
      qas_all = chol_solve<NP>(T, R, myinv, lane, qfs, nv, l.vbuf);
    }
    const float qas = is_dof ? qas_all : 0.f;  // lanes that hold no row carry meaningless numbers
    if ((given & kOutSmooth) && is_dof) a.dbg_qacc_smooth[env * nv + lane] = qas;

    KS_PHASE(7)
    float qacc = qas;
    float Mqacc = qfs;  // M qacc = smooth + constraint force: what the implicit integration step solves against
    int niter = 0;
    // ---- rows on the dof lanes (models with joint limits or dry friction only).  Their Jacobians are unit vectors, so
    // nothing of them is stored: lane j derives J a - aref of its rows from its own qacc wherever the solver needs it.
    DofRows dr = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int ndr = 0;
    if (DR) {
      int lane_r = threadIdx.x;
      asm volatile("" : "+v"(lane_r));
      if (is_dof) {
        if (KS_REC(m, lane_r, d_limited)) {
          const float q = l.qpos[KS_REC(m, lane_r, d_qadr)];
          const float dlo = q - KS_REC(m, lane_r, d_rlo), dhi = KS_REC(m, lane_r, d_rhi) - q;
          const float pos = fminf(dlo, dhi);
          if (pos < 0.f) {  // the nearer side, once violated
            dr.lim_s = dlo < dhi ? 1.f : -1.f;
            const float imp = impedance_dof(mh, pos);
            dr.lim_D = 1.f / fmaxf(KS_REC(m, lane_r, d_invw) * (1.f - imp) / imp, 1e-15f);
            dr.lim_aref = -mh.dr_b * dr.lim_s * my_qvel - mh.dr_k * imp * pos;
          }
        }
        dr.fr_fl = a.frictionloss ? ((KS_REC(m, lane_r, d_jtype) == kJntHinge) ? a.frictionloss[env * nv + lane] : 0.f) : KS_REC(m, lane_r, d_floss);
        dr.fr_D = KS_REC(m, lane_r, d_frD);
        dr.fr_rf = dr.fr_fl / dr.fr_D;
        dr.fr_aref = -mh.dr_b * my_qvel;
      }
      ndr = __popcll(__ballot(dr.lim_s != 0.f)) + __popcll(__ballot(dr.fr_fl > 0.f));
    }
    if (nefc > 0 || (DR && ndr > 0)) {
      // ---- constraint rows.  Lane j builds column j of J: the motion axis of dof j is one LDS read away, so a contact
      // costs the lane one cross product and its four pyramid edges, written to LDS row-wise (consecutive lanes,
      // consecutive addresses).  The row lanes then take their reference acceleration from a row product with qvel.
      const bool is_row = lane < nefc;
      float aref = 0.f, D = 0.f;
      {
        const bool col = lane < NP;  // the padding columns are written too (zeros): the row products read NP floats
        const Sp cd = ld6(l.cdof + 6 * (is_dof ? lane : 0));
        float* Jc = l.J + (col ? lane : 0);
        for (int k = 0; k < ncon; ++k) {  // wave-uniform
          const V3 off = ld3(l.con_off + 3 * k);
          const bool on = is_dof && ((l.con_mask[k] >> lane) & 1u);
          const V3 jac = cd.l + cross(cd.a, off);
          if (frictionless) {
            if (col) Jc[k * js] = on ? jac.z : 0.f;
          } else if (col) {  // rows of a contact: z + mu y, z - mu y, z - mu x, z + mu x
            Jc[(4 * k) * js] = on ? jac.z + mu * jac.y : 0.f;
            Jc[(4 * k + 1) * js] = on ? jac.z - mu * jac.y : 0.f;
            Jc[(4 * k + 2) * js] = on ? jac.z - mu * jac.x : 0.f;
            Jc[(4 * k + 3) * js] = on ? jac.z + mu * jac.x : 0.f;
          }
        }
        if (frictionless && col)  // whole blocks of four rows are read back below: the tail of the last block is zero
          for (int r = nefc; r < ((nefc + 3) & ~3); ++r) Jc[r * js] = 0.f;
        KS_SYNC();
        if (is_row) {
          const int c = frictionless ? lane : lane >> 2;
          float vv[NP];
          load_row<NP>(l.qvel, vv);
          const float vel = row_dot<NP>(l.J + lane * js, vv);
          aref = -mh.con_b * vel - l.con_kip[c];
          D = l.con_D[c];
        }
      }
      const float warm = is_dof ? l.warm[lane] : 0.f;
      KS_SYNC();
      KS_PHASE(8)
      // cost of the warm start and of the unconstrained acceleration; start from the cheaper one
      float Ma_w = 0.f, Ma_s = 0.f, Jar_w = 0.f, Jar_s = 0.f;
      {
        float vv[NP];
        if (lane < 32) l.vbuf[lane] = warm;
        KS_SYNC();
        load_row<NP>(l.vbuf, vv);
        if (is_dof) Ma_w = row_dot<NP>(Mrow, vv);
        if (is_row) Jar_w = row_dot<NP>(l.J + (is_row ? lane : 0) * js, vv) - aref;
        KS_SYNC();
        if (lane < 32) l.vbuf[lane] = qas;
        KS_SYNC();
        load_row<NP>(l.vbuf, vv);
        if (is_dof) Ma_s = row_dot<NP>(Mrow, vv);
        if (is_row) Jar_s = row_dot<NP>(l.J + (is_row ? lane : 0) * js, vv) - aref;
      }
      float drc_w = 0.f, drc_s = 0.f;
      if (DR) {
        float f_, h_;
        int z_;
        drc_w = dofrow_eval(dr, warm, f_, h_, z_);
        drc_s = dofrow_eval(dr, qas, f_, h_, z_);
      }
      float rows_w = ((is_row && Jar_w < 0.f) ? 0.5f * D * Jar_w * Jar_w : 0.f) + drc_w, gauss_w = is_dof ? (Ma_w - qfs) * (warm - qas) : 0.f;
      float cost_s = ((is_row && Jar_s < 0.f) ? 0.5f * D * Jar_s * Jar_s : 0.f) + drc_s;
      wave_sums(rows_w, gauss_w, cost_s);
      const float cost_w = rows_w + 0.5f * gauss_w;
      const bool use_warm = cost_w < cost_s;
      qacc = use_warm ? warm : qas;
      float Ma = use_warm ? Ma_w : Ma_s;
      float Jaref = use_warm ? Jar_w : Jar_s;
      float cost = use_warm ? cost_w : cost_s;
      float prev_cost = INFINITY;
      bool first = true;
      KS_PHASE(9)
      unsigned long long am_factored = 0ull;  // active set that R currently factors
      unsigned long long amd_factored = 0ull; // and the quadratic zones of the dof-lane rows
      bool have_factor = false;               // none yet: R holds the factor of M
      while (true) {
        // ---- constraint update: active set, forces, cost
        const bool active = is_row && (Jaref < 0.f);
        const float force = active ? -D * Jaref : 0.f;
        unsigned long long am = __ballot(active);
        float qfc = 0.f;
        if (nefc <= 32) {
          // J^T f with the rows split between the lane halves: the forces go through LDS (one 16-byte broadcast read per
          // block of four rows), lane j of half h sums the blocks 2 i + h of column j, and the halves meet at the end.
          if (lane < 32) l.vbuf[lane] = force;  // zero beyond the rows and on the inactive ones
          KS_SYNC();
          const int jc = (lane & 31) < nv ? (lane & 31) : 0, hh = lane >> 5;
          const int nblk = (nefc + 3) >> 2;
          for (int b0 = 0; b0 < nblk; b0 += 4) {  // two blocks per half, read together
            const bool ok0 = b0 + hh < nblk, ok1 = b0 + 2 + hh < nblk;
            const int k0 = ok0 ? b0 + hh : 0, k1 = ok1 ? b0 + 2 + hh : 0;
            const float4 f0 = *reinterpret_cast<const float4*>(l.vbuf + 4 * k0), f1 = *reinterpret_cast<const float4*>(l.vbuf + 4 * k1);
            const float *J0 = l.J + (4 * k0) * js + jc, *J1 = l.J + (4 * k1) * js + jc;
            const float s0 = (J0[0] * f0.x + J0[js] * f0.y) + (J0[2 * js] * f0.z + J0[3 * js] * f0.w);
            const float s1 = (J1[0] * f1.x + J1[js] * f1.y) + (J1[2 * js] * f1.z + J1[3 * js] * f1.w);
            qfc += ok0 ? s0 : 0.f;
            qfc += ok1 ? s1 : 0.f;
          }
          qfc += __shfl_xor(qfc, 32);
        } else {
          for (unsigned long long t = am; t; t &= t - 1) {
            const int r = __builtin_ctzll(t);
            qfc += l.J[r * js + (lane < nv ? lane : 0)] * lane_bcast(force, r);
          }
        }
        float dr_cost = 0.f, dr_force = 0.f, dr_h = 0.f;
        unsigned long long amd = 0ull;
        if (DR) {
          int zone;
          dr_cost = dofrow_eval(dr, qacc, dr_force, dr_h, zone);
          qfc += dr_force;
          amd = (__ballot(zone & 1) & 0xffffffffull) | (__ballot(zone & 2) << 32);
        }
        if (!is_dof) qfc = 0.f;
        // ---- gradient; stop before paying for another Hessian when the solver is done
        const float grad = is_dof ? Ma - qfs - qfc : 0.f;
        float gauss = is_dof ? (Ma - qfs) * (qacc - qas) : 0.f, row_cost = (active ? 0.5f * D * Jaref * Jaref : 0.f) + dr_cost, grad2 = grad * grad;
        wave_sums(gauss, row_cost, grad2);
        gauss *= 0.5f;
        if (!first) {
          prev_cost = cost;
          cost = row_cost + gauss;
        }
        first = false;
        const float improvement = scale * (prev_cost - cost);
        const float gradient = scale * __builtin_amdgcn_sqrtf(grad2);
        int iterations = mh.iterations, ls_iterations = mh.ls_iterations;  // together, as `given`
        float tolerance = mh.tolerance, ls_tolerance = mh.ls_tolerance, meaninertia = mh.meaninertia;
        asm volatile("" : "+s"(iterations), "+s"(ls_iterations), "+s"(tolerance), "+s"(ls_tolerance), "+s"(meaninertia));
        bool done = niter >= iterations;
        done |= improvement < tolerance;
        done |= gradient < tolerance;
        if (done && !(iterations == 1 && niter == 0)) break;
        KS_PHASE(10)
        // ---- Newton direction: H = M + J^T diag(D active) J.  The rank-nefc term runs on the matrix cores: one
        // 32x32x2 fp32 MFMA per pair of constraint rows, operands straight from the LDS copy of J (lane = column,
        // lane half = row of the pair).  The accumulator tile holds, in lane c, rows {8g + 4 (lane / 32) + e} of
        // column c, which by symmetry is row c: the upper lane half hands its 16 entries to the lower one and
        // lane i < 32 ends up with row i of H in registers, as the factorisation wants it.
        // H depends on the iterate only through the active set: while that stays the same (the usual case once the
        // solver closes in) the factor of the previous iteration is still the factor of H and is kept.
        float step_all;
        if (!have_factor || am != am_factored || (DR && amd != amd_factored)) {
          l.drow[lane] = active ? D : 0.f;
          if (lane < 32) l.vbuf[lane] = grad;
          KS_SYNC();
          f32x16 hc;
          load_mtile<NP>(hc, l.M, l.vbuf, lane);
          const int col = lane & 31, half = lane >> 5;
          const bool col_ok = NP == 32 || col < NP;
          // the operands of four products at a time are fetched before the first of them (a row past the last counts as zero)
          for (int r0 = 0; r0 < nefc; r0 += 8) {
            float jr[4], dj[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int r = r0 + 2 * i + half;
              const bool row_ok = r < nefc;
              const int rc = row_ok ? r : 0;
              const float x = l.J[rc * js + (col_ok ? col : 0)], d = l.drow[rc];
              jr[i] = (col_ok && row_ok) ? x : 0.f;
              dj[i] = d * jr[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (r0 + 2 * i < nefc) hc = __builtin_amdgcn_mfma_f32_32x32x2f32(dj[i], jr[i], hc, 0, 0, 0);
          }
          if (DR) {  // unit-vector rows add their stiffness to the diagonal
            const float hd = __shfl(dr_h, col);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
              for (int e = 0; e < 4; ++e) hc[4 * g + e] += (8 * g + 4 * half + e == col) ? hd : 0.f;
          }
          KS_PHASE(11)
          step_all = chol_solve<NP>(hc, R, myinv, lane, grad, nv, l.vbuf);
          am_factored = am;
          amd_factored = amd;
          have_factor = true;
        } else {
          step_all = solve_regs<NP>(R, myinv, grad, nv);
        }
        const float search = is_dof ? -step_all : 0.f;
        KS_PHASE(12)
        // ---- exact line search along `search`
        float mv = 0.f, jv = 0.f;
        {
          float vv[NP];
          KS_SYNC();
          if (lane < 32) l.vbuf[lane] = search;
          KS_SYNC();
          load_row<NP>(l.vbuf, vv);
          if (is_dof) mv = row_dot<NP>(Mrow, vv);
          if (is_row) jv = row_dot<NP>(l.J + (is_row ? lane : 0) * js, vv);
        }
        float search2 = search * search, g1 = is_dof ? search * (Ma - qfs) : 0.f, g2 = is_dof ? search * mv : 0.f;
        wave_sums(search2, g1, g2);
        g2 *= 0.5f;
        const float smag = __builtin_amdgcn_sqrtf(search2) * meaninertia * (float)(nv > 1 ? nv : 1);
        const float gtol = tolerance * ls_tolerance * smag;
        const float g0 = gauss;
        float alpha;
        if (nefc <= 32 && !(DR && ndr > 0)) {
          alpha = line_search_rows(ls_iterations, nefc, lane, Jaref, jv, D, g0, g1, g2, gtol);
        } else {
          const float q0r = 0.5f * Jaref * Jaref * D, q1r = jv * Jaref * D, q2r = 0.5f * jv * jv * D;
          // With at most 16 constraint rows the three sums of a cost evaluation share one reduction: the 16-lane
          // groups 0, 1, 2 hold copies of the rows with the constant, linear and quadratic coefficient, and one
          // DPP reduction within the groups yields all three totals.
          // Rows 16..31 ride along as a second copy in the same lanes, so up to 32 rows need no more reduction steps.
          const bool packed = DR && nefc <= 32, two = nefc > 16;
          float pk_j = 0.f, pk_jv = 0.f, pk_q = 0.f, pk_j2 = 0.f, pk_jv2 = 0.f, pk_q2 = 0.f;
          const int grp = lane >> 4;
          if (packed) {
            const int r = lane & 15;
            pk_j = __shfl(Jaref, r);
            pk_jv = __shfl(jv, r);
            const float c0 = __shfl(q0r, r), c1 = __shfl(q1r, r), c2 = __shfl(q2r, r);
            pk_q = grp == 0 ? c0 : (grp == 1 ? c1 : (grp == 2 ? c2 : 0.f));
            if (two) {
              pk_j2 = __shfl(Jaref, 16 + r);
              pk_jv2 = __shfl(jv, 16 + r);
              const float e0 = __shfl(q0r, 16 + r), e1 = __shfl(q1r, 16 + r), e2 = __shfl(q2r, 16 + r);
              pk_q2 = grp == 0 ? e0 : (grp == 1 ? e1 : (grp == 2 ? e2 : 0.f));
            }
          }
          auto point = [&](float alpha) {
            float q0, q1, q2;
            if (packed) {
              float x = (pk_j + alpha * pk_jv < 0.f) ? pk_q : 0.f;  // rows beyond nefc carry zeros
              if (two) x += (pk_j2 + alpha * pk_jv2 < 0.f) ? pk_q2 : 0.f;
              if (DR && ndr > 0) {
                // The rows on the dof lanes join the same reduction.  Lane j < 32 holds the three coefficients of its own rows:
                // the constant one belongs in group 0, the linear one in group 1, so each lane keeps the one of its own group
                // and swaps the other with the lane 16 away; the quadratic ones go to the upper lane half (groups 2 and 3).
                float t0, t1, t2;
                dofrow_quad(dr, qacc, search, alpha, t0, t1, t2);
                const float got = __shfl_xor(grp == 0 ? t1 : t0, 16);
                const float up = __shfl(t2, lane & 31);
                x += grp == 0 ? t0 + got : (grp == 1 ? t1 + got : up);
              }
              x += dpp_shift<0x111, 0xf>(x);
              x += dpp_shift<0x112, 0xf>(x);
              x += dpp_shift<0x114, 0xf>(x);
              x += dpp_shift<0x118, 0xf>(x);  // lane 15 of each 16-lane group holds the group's total
              q0 = g0 + lane_bcast(x, 15);
              q1 = g1 + lane_bcast(x, 31);
              q2 = g2 + lane_bcast(x, 47) + (DR ? lane_bcast(x, 63) : 0.f);
            } else {
              const bool on = is_row && (Jaref + alpha * jv < 0.f);
              q0 = g0 + wave_sum(on ? q0r : 0.f);
              q1 = g1 + wave_sum(on ? q1r : 0.f);
              q2 = g2 + wave_sum(on ? q2r : 0.f);
            }
            if (DR && ndr > 0 && !packed) {
              float t0, t1, t2;
              dofrow_quad(dr, qacc, search, alpha, t0, t1, t2);
              q0 += wave_sum(t0);
              q1 += wave_sum(t1);
              q2 += wave_sum(t2);
            }
            LsPoint p;
            p.alpha = alpha;
            p.cost = alpha * alpha * q2 + alpha * q1 + q0;
            p.d0 = 2.f * alpha * q2 + q1;
            p.d1 = 2.f * q2 + (q2 == 0.f ? 1e-15f : 0.f);
            return p;
          };
          const LsPoint p0 = point(0.f);
          // Newton estimates of the step length: d0 / d1 by reciprocal and product (1 ulp), a tenth of an IEEE division's instructions
          auto newton_alpha = [](const LsPoint& x) { return x.alpha - x.d0 * __builtin_amdgcn_rcpf(x.d1); };
          LsPoint lo = point(newton_alpha(p0));
          LsPoint hi;
          if (lo.d0 < p0.d0) { hi = p0; } else { hi = lo; lo = p0; }
          bool swap = true;
          int it = 0;
          while (true) {
            bool ls_done = it >= ls_iterations;
            ls_done |= !swap;
            ls_done |= (lo.d0 < 0.f) && (lo.d0 > -gtol);
            ls_done |= (hi.d0 > 0.f) && (hi.d0 < gtol);
            if (ls_done) break;
            const LsPoint lo_next = point(newton_alpha(lo));
            const LsPoint hi_next = point(newton_alpha(hi));
            const LsPoint mid = point(0.5f * (lo.alpha + hi.alpha));
            LsPoint nlo = lo, nhi = hi;
            const bool s1 = in_bracket(nlo, lo_next); if (s1) nlo = lo_next;
            const bool s2 = in_bracket(nlo, mid);     if (s2) nlo = mid;
            const bool s3 = in_bracket(nlo, hi_next); if (s3) nlo = hi_next;
            const bool t1 = in_bracket(nhi, hi_next); if (t1) nhi = hi_next;
            const bool t2 = in_bracket(nhi, mid);     if (t2) nhi = mid;
            const bool t3 = in_bracket(nhi, lo_next); if (t3) nhi = lo_next;
            lo = nlo; hi = nhi;
            swap = s1 | s2 | s3 | t1 | t2 | t3;
            ++it;
          }
          const bool improved = (lo.cost < p0.cost) || (hi.cost < p0.cost);
          alpha = lo.cost < hi.cost ? lo.alpha : hi.alpha;
          if (!improved) alpha = 0.f;
        }
        qacc += alpha * search;
        Ma += alpha * mv;
        Jaref += alpha * jv;
        ++niter;
        KS_PHASE(13)
      }
      Mqacc = Ma;
      // ---- Cartesian contact forces on the bodies (mjData.cfrc_ext), only when asked for: a pyramid row with force f
      // pushes along normal +- mu tangent (rows of a contact: z + mu y, z - mu y, z - mu x, z + mu x)
      if ((given & kOutCfrc) && sub == nsub - 1) {
        const float f = (is_row && Jaref < 0.f) ? -D * Jaref : 0.f;
        const int q = lane & 3;
        float fx = 0.f, fy = 0.f, fz = f;
        if (!frictionless) {
          fx = q == 3 ? mu * f : (q == 2 ? -mu * f : 0.f);
          fy = q == 0 ? mu * f : (q == 1 ? -mu * f : 0.f);
          fx += __shfl_xor(fx, 1); fy += __shfl_xor(fy, 1); fz += __shfl_xor(fz, 1);
          fx += __shfl_xor(fx, 2); fy += __shfl_xor(fy, 2); fz += __shfl_xor(fz, 2);
        }
        KS_SYNC();  // the line search is done with drow
        const int cc = frictionless ? lane : lane >> 2;
        if (is_row && (frictionless || q == 0)) { l.drow[3 * cc] = fx; l.drow[3 * cc + 1] = fy; l.drow[3 * cc + 2] = fz; }
        KS_SYNC();
        if (lane < nb) {
          Sp w = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
          for (int k = 0; k < ncon; ++k)
            if (l.con_body[k] == lane) {
              const V3 F = ld3(l.drow + 3 * k);
              w.a = w.a + cross(ld3(l.con_off + 3 * k), F);
              w.l = w.l + F;
            }
          float* dst = a.cfrc_ext + ((int64_t)env * nb + lane) * 6;
          dst[0] = w.a.x; dst[1] = w.a.y; dst[2] = w.a.z; dst[3] = w.l.x; dst[4] = w.l.y; dst[5] = w.l.z;
        }
      }
    } else if ((given & kOutCfrc) && sub == nsub - 1) {
      for (int i = lane; i < nb * 6; i += 64) a.cfrc_ext[(int64_t)env * nb * 6 + i] = 0.f;
    }
    work += (1 + niter) * (16 + nefc + ndr);
    if (sub == nsub - 1) {  // outputs of the last substep go out here: nothing of them stays live to the end
      if ((given & kOutQacc) && lane < nv) a.qacc[env * nv + lane] = qacc;
      if ((given & kOutNiter) && lane == 0) a.solver_niter[env] = niter;
      if ((given & kOutNefc) && lane == 0) a.nefc[env] = nefc + ndr;
    }
    KS_SYNC();
    if (is_dof) l.warm[lane] = qacc;

    KS_PHASE(14)
    // Behind the solver, whose register rows set the occupancy: for the next substep, and what the integration needs of it.
    // Requested at the top of a substep, and three fields of it once more here, a wavefront waited twice: 64 robots' control
    // step 0.8 %, 1024 K-Bots' and 4096 humanoids' 0.3 % slower.  The actuator's inputs requested here as well cost more
    // (16 spilled registers) than they save, 2.5 %, and so did reading the joint's addresses from LDS instead, 1.1 %.
    load_lane(a, in);
    // ---- semi-implicit Euler
    if (!fwd) {
      int lane_e = threadIdx.x;
      asm volatile("" : "+v"(lane_e));
      const int b_jtype = in.rec.b_jtype, b_qadr = in.rec.b_qadr, b_dofadr = in.rec.b_dofadr;
      const float d_damping = in.rec.d_damping * in.damping_scale;
      const float my_qvel = lane_e < nv ? l.qvel[lane_e] : 0.f;
      float qacc_int = qacc;
      if (mh.eulerdamp) {
        // implicit in the joint damping: (M + dt diag(damping)) a = M qacc.  For torque motors, whose force does
        // not depend on velocity, this is MuJoCo's implicitfast step; qacc itself (warm start, output) is unchanged.
        f32x16 T;
        const float b = is_dof ? Mqacc : 0.f;
        if (lane < 32) l.vbuf[lane] = b;
        KS_SYNC();
        load_mtile<NP>(T, l.M, l.vbuf, lane);
        const int c = lane & 31, half = lane >> 5;
        const float hd = mh.dt * __shfl(is_dof ? d_damping : 0.f, c);
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) T[4 * g + e] += (8 * g + 4 * half + e == c) ? hd : 0.f;  // lanes of column 31: dof 31 or none
        float R2[NP];
        float inv2;
        const float sol = chol_solve<NP>(T, R2, inv2, lane, b, nv, l.vbuf);
        qacc_int = is_dof ? sol : 0.f;
      }
      if (is_dof) l.qvel[lane] = my_qvel + mh.dt * qacc_int;
      KS_SYNC();
      if (is_body) {
        const int qa = b_qadr, da = b_dofadr;
        if (b_jtype == kJntFree) {
          const V3 p = ld3(l.qpos + qa), v = ld3(l.qvel + da), w = ld3(l.qvel + da + 3);
          Quat q = {l.qpos[qa + 3], l.qpos[qa + 4], l.qpos[qa + 5], l.qpos[qa + 6]};
          // the turn by |w| dt about w, whose half angle is h = |w| dt / 2, from x = h^2: sin(h) / |w| and cos(h) as their series,
          // whose first terms left out are below 2^-30 for h <= 1/2.  Root, sine, cosine and division are a long chain for one lane:
          // this stage of a wavefront alone 2720 -> 2320 cycles, rollout steps of 1024 K-Bots and of an LSTM policy 0.3 and 0.5 %
          // faster.  Largest error against 64 bits, 2^-24: sin(h) / |w| 2.66 -> 1.36, cos(h) 0.98 -> 0.92 (|w| to 199 / s).
          const float half_dt = 0.5f * mh.dt, w2 = dot(w, w), x = w2 * half_dt * half_dt;
          if (x <= 0.25f) {
            const float s = half_dt * fmaf(x, fmaf(x, fmaf(x, fmaf(x, 1.f / 362880, -1.f / 5040), 1.f / 120), -1.f / 6), 1.f);
            const float c = fmaf(x, fmaf(x, fmaf(x, fmaf(x, fmaf(x, -1.f / 3628800, 1.f / 40320), -1.f / 720), 1.f / 24), -0.5f), 1.f);
            q = qmul(q, {c, w.x * s, w.y * s, w.z * s});
          } else if (const float n = sqrtf(w2); n > 1e-15f) {
            const float h = n * half_dt, s = sinf(h) / n;
            q = qmul(q, {cosf(h), w.x * s, w.y * s, w.z * s});
          }
          q = qnormalize(q);
          st3(l.qpos + qa, p + v * mh.dt);
          l.qpos[qa + 3] = q.w; l.qpos[qa + 4] = q.x; l.qpos[qa + 5] = q.y; l.qpos[qa + 6] = q.z;
        } else if (b_jtype == kJntHinge) {
          l.qpos[qa] += mh.dt * l.qvel[da];
        }
      }
    }
    KS_SYNC();
  }

  KS_PHASE(15)
#ifdef KS_PROFILE
  if (a.dbg_M && lane == 0) for (int k = 0; k < 16; ++k) a.dbg_M[env * nv * nv + k] = prof[k];
#endif
  // ---- write back
  {
    const StepArgs& a = arguments();
    const ModelHead& mh = a.head;
    if (!FWD) {
      for (int i = lane; i < nq; i += 64) a.qpos[env * nq + i] = l.qpos[i];
      if (lane < nv) a.qvel[env * nv + lane] = l.qvel[lane];
      if (a.work && lane == 0) a.work[env] = work;
      if (a.time && lane == 0) {  // dt added once per substep in fp32, like the reference's accumulation
        float time = a.time[env];
        for (int k = 0; k < nsub; ++k) time += mh.dt;
        a.time[env] = time;
      }
      if (a.last_ctrl) {
        const int na = a.actuator_type == KS_ACT_POSITION_VELOCITY ? 2 * nu : nu;
        for (int i = lane; i < na; i += 64) a.last_ctrl[env * na + i] = a.action[env * na + i];
      }
    }
    if (a.qacc_warmstart && lane < nv) a.qacc_warmstart[env * nv + lane] = l.warm[lane];
    if (a.ctrl_out) for (int i = lane; i < nu; i += 64) a.ctrl_out[env * nu + i] = l.tau[i];
    if (a.xpos) for (int i = lane; i < nb * 3; i += 64) a.xpos[env * nb * 3 + i] = l.xpos[i];
    if (a.xquat) for (int i = lane; i < nb * 4; i += 64) a.xquat[env * nb * 4 + i] = l.xquat[i];
    if (a.cvel) for (int i = lane; i < nb * 6; i += 64) a.cvel[env * nb * 6 + i] = l.cvel[i];
    if (a.traj_ctrl) for (int i = lane; i < nu; i += 64) a.traj_ctrl[env * nu + i] = l.tau[i];
    if (a.traj_xpos) for (int i = lane; i < nb * 3; i += 64) a.traj_xpos[env * nb * 3 + i] = l.xpos[i];
    if (a.traj_xquat) for (int i = lane; i < nb * 4; i += 64) a.traj_xquat[env * nb * 4 + i] = l.xquat[i];
  }
}

}  // namespace ks

using namespace ks;

// ---------------------------------------------------------------------------------------------
// C ABI: model upload and the step / forward entry points
// ---------------------------------------------------------------------------------------------
struct KsModel {
  DevModel host;
  DevModel* dev;
  int device;
};

extern "C" int ks_model_create(const KsModelDesc* d, KsModel** out) {
  if (!d || !out) return fail(KS_EINVAL, "ks_model_create: null argument");
  if (d->nb < 1 || d->nb > kMaxB || d->nq < 0 || d->nq > kMaxQ || d->nv < 0 || d->nv > kMaxV || d->nu < 0 ||
      d->nu > kMaxU || d->ns < 0 || d->ns > kMaxS)
    return fail(KS_ELIMIT, "ks_model_create: sizes nb=%d nq=%d nv=%d nu=%d ns=%d exceed %d/%d/%d/%d/%d", d->nb, d->nq,
                d->nv, d->nu, d->ns, kMaxB, kMaxQ, kMaxV, kMaxU, kMaxS);
  if (d->nv > 64 || 4 * d->ns > 64) return fail(KS_ELIMIT, "ks_model_create: more than 64 dofs or constraint rows");
  if (d->condim != 0 && d->condim != 1 && d->condim != 3) return fail(KS_EINVAL, "ks_model_create: condim %d (1 or 3)", d->condim);
  if (!(d->dt > 0.0)) return fail(KS_EINVAL, "ks_model_create: dt must be positive");
  KsModel* km = new KsModel();
  DevModel& m = km->host;
  std::memset(&m, 0, sizeof(m));
  m.nb = d->nb; m.nq = d->nq; m.nv = d->nv; m.nu = d->nu; m.ns = d->ns;
  m.iterations = d->iterations; m.ls_iterations = d->ls_iterations; m.eulerdamp = d->eulerdamp;
  m.frictionless = d->condim == 1 ? 1 : 0;
  m.dt = (float)d->dt;
  for (int k = 0; k < 3; ++k) m.gravity[k] = (float)d->gravity[k];
  m.tolerance = (float)d->tolerance; m.ls_tolerance = (float)d->ls_tolerance;
  m.meaninertia = (float)d->meaninertia; m.friction = (float)d->friction; m.impratio_inv = (float)(1.0 / d->impratio);
  {  // solref / solimp -> (k, b) and clamped impedance parameters, for the contact rows and for the dof-lane rows
    auto convert = [&](const double* solref, const double* solimp, float* out /*k b dmin dmax 1/width mid power imp_a imp_b*/) {
      double timeconst = solref[0], dampratio = solref[1];
      double dmin = solimp[0], dmax = solimp[1], width = solimp[2], mid = solimp[3], power = solimp[4];
      if (timeconst < 2 * d->dt) timeconst = 2 * d->dt;
      auto clampd = [](double x, double lo, double hi) { return x < lo ? lo : (x > hi ? hi : x); };
      dmin = clampd(dmin, 1e-4, 0.9999); dmax = clampd(dmax, 1e-4, 0.9999);
      width = width < 1e-15 ? 1e-15 : width; mid = clampd(mid, 1e-4, 0.9999); power = power < 1 ? 1 : power;
      double k = 1.0 / (dmax * dmax * timeconst * timeconst * dampratio * dampratio), b = 2.0 / (dmax * timeconst);
      if (solref[0] <= 0) k = -solref[0] / (dmax * dmax);
      if (solref[1] <= 0) b = -solref[1] / dmax;
      out[0] = (float)k; out[1] = (float)b; out[2] = (float)dmin; out[3] = (float)dmax; out[4] = (float)(1.0 / width);
      out[5] = (float)mid; out[6] = (float)power;
      out[7] = (float)(1.0 / std::pow(mid, power - 1.0)); out[8] = (float)(1.0 / std::pow(1.0 - mid, power - 1.0));
    };
    float c[9];
    convert(d->solref, d->solimp, c);
    m.con_k = c[0]; m.con_b = c[1]; m.dmin = c[2]; m.dmax = c[3]; m.width_inv = c[4]; m.mid = c[5]; m.power = c[6]; m.imp_a = c[7]; m.imp_b = c[8];
    bool own = false;
    for (int k = 0; k < 2; ++k) own |= d->dof_solref[k] != 0.0;
    for (int k = 0; k < 5; ++k) own |= d->dof_solimp[k] != 0.0;
    if (own) convert(d->dof_solref, d->dof_solimp, c);
    m.dr_k = c[0]; m.dr_b = c[1]; m.dr_dmin = c[2]; m.dr_dmax = c[3]; m.dr_width_inv = c[4]; m.dr_mid = c[5]; m.dr_power = c[6];
    m.dr_imp_a = c[7]; m.dr_imp_b = c[8];
  }
  for (int b = 0; b < d->nb; ++b) {
    m.body_parent[b] = d->body_parent[b]; m.body_jtype[b] = d->body_jtype[b]; m.body_qadr[b] = d->body_qadr[b];
    m.body_dofadr[b] = d->body_dofadr[b]; m.body_subtree_end[b] = d->body_subtree_end[b];
    if (b > 0 && (d->body_parent[b] < 0 || d->body_parent[b] >= b)) { delete km; return fail(KS_EINVAL, "ks_model_create: body %d has parent %d (must precede it)", b, d->body_parent[b]); }
    if (d->body_subtree_end[b] <= b || d->body_subtree_end[b] > d->nb) { delete km; return fail(KS_EINVAL, "ks_model_create: bad subtree_end for body %d", b); }
    if (b > 0 && d->body_jtype[b] != kJntFree && d->body_jtype[b] != kJntHinge) { delete km; return fail(KS_EINVAL, "ks_model_create: body %d needs a free or hinge joint", b); }
    if (b > 0) {  // the joint's coordinates and dofs must lie inside qpos / qvel: the kernel and the tables below index with them
      const int nqj = d->body_jtype[b] == kJntFree ? 7 : 1, nvj = d->body_jtype[b] == kJntFree ? 6 : 1;
      if (d->body_qadr[b] < 0 || d->body_qadr[b] + nqj > d->nq || d->body_dofadr[b] < 0 || d->body_dofadr[b] + nvj > d->nv) {
        delete km;
        return fail(KS_EINVAL, "ks_model_create: body %d has qpos address %d and dof address %d outside nq=%d / nv=%d", b,
                    d->body_qadr[b], d->body_dofadr[b], d->nq, d->nv);
      }
    }
    for (int k = 0; k < 3; ++k) {
      m.body_pos[b][k] = (float)d->body_pos[b][k]; m.body_ipos[b][k] = (float)d->body_ipos[b][k];
      m.body_inertia[b][k] = (float)d->body_inertia[b][k]; m.jnt_axis[b][k] = (float)d->jnt_axis[b][k];
      m.jnt_pos[b][k] = (float)d->jnt_pos[b][k];
    }
    for (int k = 0; k < 4; ++k) { m.body_quat[b][k] = (float)d->body_quat[b][k]; m.body_iquat[b][k] = (float)d->body_iquat[b][k]; }
    m.body_mass[b] = (float)d->body_mass[b];
    m.body_invweight0[b] = (float)d->body_invweight0[b];
    int n = 0;  // links from the root down to b
    for (int c = b; c > 0; c = d->body_parent[c]) ++n;
    if (n > kMaxDepth) { delete km; return fail(KS_ELIMIT, "ks_model_create: tree deeper than %d", kMaxDepth); }
    m.body_depth[b] = n;
    if (n > m.max_depth) m.max_depth = n;
  }
  m.root_free = d->nb > 1 && m.body_jtype[1] == kJntFree;
  for (int q = 0; q < d->nq; ++q) m.qpos0[q] = (float)d->qpos0[q];
  for (int j = 0; j < d->nv; ++j) {
    m.dof_body[j] = d->dof_body[j]; m.dof_parent[j] = d->dof_parent[j]; m.dof_act[j] = -1;
    m.dof_damping[j] = (float)d->dof_damping[j]; m.dof_armature[j] = (float)d->dof_armature[j];
    if (d->dof_parent[j] >= j || d->dof_body[j] < 1 || d->dof_body[j] >= d->nb) { delete km; return fail(KS_EINVAL, "ks_model_create: bad dof %d", j); }
  }
  for (int b = 1; b < d->nb; ++b) {
    if (!d->jnt_limited[b]) continue;
    if (d->body_jtype[b] != kJntHinge) { delete km; return fail(KS_EINVAL, "ks_model_create: body %d: only hinges can be limited", b); }
    if (!(d->jnt_range[b][0] < d->jnt_range[b][1])) { delete km; return fail(KS_EINVAL, "ks_model_create: body %d: empty joint range", b); }
    if (!(d->dof_invweight0[d->body_dofadr[b]] > 0.0)) { delete km; return fail(KS_EINVAL, "ks_model_create: body %d: a limited joint needs dof_invweight0 > 0", b); }
    m.dofrows = 1;
  }
  m.invw_ok = 1;
  for (int j = 0; j < d->nv; ++j)
    if (d->body_jtype[d->dof_body[j]] == kJntHinge && !(d->dof_invweight0[j] > 0.0)) m.invw_ok = 0;
  for (int j = 0; j < d->nv; ++j) {
    if (d->dof_frictionloss[j] == 0.0) continue;
    if (!(d->dof_frictionloss[j] > 0.0) || d->body_jtype[d->dof_body[j]] != kJntHinge) { delete km; return fail(KS_EINVAL, "ks_model_create: dof %d: frictionloss must be positive and on a hinge", j); }
    if (!(d->dof_invweight0[j] > 0.0)) { delete km; return fail(KS_EINVAL, "ks_model_create: dof %d: dry friction needs dof_invweight0 > 0", j); }
    m.dofrows = 1;
    ++m.nfriction;
  }
  for (int u = 0; u < d->nu; ++u) {
    const int j = d->act_dof[u];
    if (j < 0 || j >= d->nv) { delete km; return fail(KS_EINVAL, "ks_model_create: actuator %d drives dof %d", u, j); }
    if (m.dof_act[j] >= 0) { delete km; return fail(KS_EINVAL, "ks_model_create: dof %d has two actuators", j); }
    m.dof_act[j] = u; m.act_dof[u] = j; m.act_gear[u] = (float)d->act_gear[u];
    m.act_lo[u] = (float)d->act_lo[u]; m.act_hi[u] = (float)d->act_hi[u];
  }
  for (int s = 0; s < d->ns; ++s) {
    if (d->sph_body[s] < 1 || d->sph_body[s] >= d->nb) { delete km; return fail(KS_EINVAL, "ks_model_create: sphere %d on body %d", s, d->sph_body[s]); }
    m.sph_body[s] = d->sph_body[s]; m.sph_radius[s] = (float)d->sph_radius[s];
    for (int k = 0; k < 3; ++k) m.sph_pos[s][k] = (float)d->sph_pos[s][k];
  }
  // dof masks and (i, ancestor j) pairs
  int np = 0;
  for (int i = 0; i < d->nv; ++i)
    for (int j = d->dof_parent[i]; j >= 0; j = d->dof_parent[j]) {
      m.pair_i[np] = (short)i; m.pair_j[np] = (short)j; ++np;
    }
  m.npairs = np;
  for (int b = 1; b < d->nb; ++b) {
    unsigned mask = 0;
    for (int j = 0; j < d->nv; ++j) {
      for (int c = b; c > 0; c = d->body_parent[c])
        if (c == d->dof_body[j]) { mask |= 1u << j; break; }
    }
    m.body_dofmask[b] = mask;
  }
  for (int L = 0; L < 64; ++L) {
    m.ones[L] = 1.f;
    LaneRec r;
    std::memset(&r, 0, sizeof(r));
    const bool is_body = L > 0 && L < d->nb;
    const int bl = is_body ? L : 0;
    r.b_jtype = m.body_jtype[bl]; r.b_qadr = m.body_qadr[bl]; r.b_dofadr = m.body_dofadr[bl];
    r.b_depth = is_body ? m.body_depth[bl] : -1;
    for (int c = bl, k = r.b_depth - 1; c > 0; c = d->body_parent[c], --k) {
      const unsigned link = (unsigned)c | (unsigned)m.body_dofadr[c] << 5 | (m.body_jtype[c] == kJntHinge ? 1u << 10 : 0u) |
                            (m.body_jtype[c] == kJntFree ? 1u << 11 : 0u);
      r.b_chain[k / 2] |= link << (16 * (k & 1));
    }
    r.b_q0 = (is_body && r.b_jtype == kJntHinge) ? m.qpos0[r.b_qadr] : 0.f;
    r.b_mass = m.body_mass[bl];
    for (int k = 0; k < 3; ++k) {
      r.b_pos[k] = m.body_pos[bl][k];
      r.b_jaxis[k] = m.jnt_axis[bl][k]; r.b_jpos[k] = m.jnt_pos[bl][k];
    }
    for (int k = 0; k < 4; ++k) { r.b_quat[k] = m.body_quat[bl][k]; r.b_iquat[k] = m.body_iquat[bl][k]; }
    const bool is_dof = L < d->nv;
    const int dl = is_dof ? L : 0;
    r.d_body = d->nv > 0 ? m.dof_body[dl] : 0;
    r.d_act = is_dof ? m.dof_act[dl] : -1;
    r.d_jtype = m.body_jtype[r.d_body];
    r.d_k = dl - m.body_dofadr[r.d_body];
    r.d_damping = m.dof_damping[dl]; r.d_armature = m.dof_armature[dl];
    r.d_stiffness = 0.f;
    const int ua = r.d_act >= 0 ? r.d_act : 0;
    r.d_gear = m.act_gear[ua]; r.d_lo = m.act_lo[ua]; r.d_hi = m.act_hi[ua];
    r.d_limited = 0; r.d_qadr = 0; r.d_rlo = 0.f; r.d_rhi = 0.f; r.d_invw = 0.f; r.d_floss = 0.f; r.d_frD = 0.f;
    if (is_dof && r.d_jtype == kJntHinge) {
      r.d_limited = d->jnt_limited[r.d_body] != 0;
      r.d_qadr = m.body_qadr[r.d_body];
      r.d_stiffness = (float)d->dof_stiffness[dl];
      r.d_rlo = (float)d->jnt_range[r.d_body][0]; r.d_rhi = (float)d->jnt_range[r.d_body][1];
      r.d_invw = (float)d->dof_invweight0[dl];
      r.d_floss = (float)d->dof_frictionloss[dl];
      const double imp0 = m.dr_dmin;  // impedance at pos = 0
      r.d_frD = (float)(1.0 / std::max(d->dof_invweight0[dl] * (1.0 - imp0) / imp0, 1e-15));
    }
    const int sl = L < d->ns ? L : 0;
    r.s_body = m.sph_body[sl]; r.s_invw = m.body_invweight0[r.s_body];
    r.s_mask = m.body_dofmask[r.s_body];
    for (int k = 0; k < kPairSets; ++k) {
      const int p = L + 64 * k;
      r.pk[k] = p < m.npairs ? ((int)m.pair_i[p] << 8) | (int)m.pair_j[p] : -1;
    }
    for (int k = 0; k < kRecPieces; ++k) std::memcpy(m.lane_rec[k][L], (const char*)&r + 16 * k, 16);
  }
  if (hipGetDevice(&km->device) != hipSuccess) { delete km; return fail(KS_ELAUNCH, "ks_model_create: no HIP device"); }
  if (hipMalloc((void**)&km->dev, sizeof(DevModel)) != hipSuccess) { delete km; return fail(KS_ELAUNCH, "ks_model_create: hipMalloc failed"); }
  if (hipMemcpy(km->dev, &m, sizeof(DevModel), hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(km->dev); delete km; return fail(KS_ELAUNCH, "ks_model_create: upload failed");
  }
  *out = km;
  return KS_OK;
}

extern "C" int ks_model_destroy(KsModel* m) {
  if (!m) return KS_OK;
  (void)hipFree(m->dev);
  delete m;
  return KS_OK;
}

extern "C" int ks_model_lds_bytes(const KsModel* m) {
  if (!m) return 0;
  return lds_floats(m->host.nb, m->host.nq, m->host.nv, m->host.nu, m->host.ns) * 4;
}

static int launch_step(const KsModel* km, ks_stream_t stream, const KsStepIO* io, bool forward_only) {
  if (!km || !io) return fail(KS_EINVAL, "ks_step: null argument");
  const DevModel& m = km->host;
  if (io->N < 0) return fail(KS_EINVAL, "ks_step: negative env count");
  if (io->N == 0) return KS_OK;
  if (io->N > 0x7fffffff) return fail(KS_ELIMIT, "ks_step: too many envs");
  if (!io->qpos || !io->qvel) return fail(KS_EINVAL, "ks_step: qpos and qvel are required");
  StepArgs a;
  std::memset(&a, 0, sizeof(a));
  a.model = km->dev;
  a.head = m;
  a.N = io->N;
  a.qpos = io->qpos; a.qvel = io->qvel; a.qacc_warmstart = io->qacc_warmstart; a.time = io->time;
  a.friction = io->friction; a.mass_scale = io->mass_scale; a.env_mask = io->env_mask; a.fresh = io->fresh;
  a.qacc = io->qacc; a.ctrl_out = io->ctrl_out; a.xpos = io->xpos; a.xquat = io->xquat; a.cvel = io->cvel;
  a.traj_ctrl = io->traj_ctrl; a.traj_xpos = io->traj_xpos; a.traj_xquat = io->traj_xquat;
  a.solver_niter = io->solver_niter; a.nefc = io->nefc;
  a.dbg_M = io->dbg_M; a.dbg_bias = io->dbg_bias; a.dbg_qacc_smooth = io->dbg_qacc_smooth;
  a.contact_dist = io->contact_dist; a.cinert = io->cinert; a.cfrc_ext = io->cfrc_ext;
  a.armature_scale = io->armature_scale; a.damping_scale = io->damping_scale;
  a.frictionloss = io->frictionloss; a.body_ipos = io->body_ipos; a.body_inertia = io->body_inertia;
  a.sph_pos = io->sph_pos; a.sph_radius = io->sph_radius;
  if ((io->sph_pos == nullptr) != (io->sph_radius == nullptr)) return fail(KS_EINVAL, "ks_step: sph_pos and sph_radius come together");
  if (io->frictionloss && !m.invw_ok) return fail(KS_EINVAL, "ks_step: per-env frictionloss needs dof_invweight0 > 0 on every hinge");
  a.env_order = forward_only ? nullptr : io->env_order; a.work = io->work;
  a.ctrl_in = io->ctrl_in;
  if (!forward_only) {
    if (io->substeps < 1 || io->substeps > 64) return fail(KS_EINVAL, "ks_step: substeps must be in 1..64");
    if (io->actuator_period < 1) return fail(KS_EINVAL, "ks_step: actuator_period must be >= 1");
    if (m.nu > 0 && (!io->action || !io->last_ctrl)) return fail(KS_EINVAL, "ks_step: action and last_ctrl are required");
    if (io->actuator_type < KS_ACT_TORQUE || io->actuator_type > KS_ACT_POSITION_VELOCITY)
      return fail(KS_EINVAL, "ks_step: unknown actuator type %d", io->actuator_type);
    if (io->actuator_type != KS_ACT_TORQUE && m.nu > 0 && (!io->kp || !io->kd || !io->ctrl_clip))
      return fail(KS_EINVAL, "ks_step: position actuators need kp, kd and ctrl_clip");
    if (io->actuator_type != KS_ACT_TORQUE && m.nu + (m.body_jtype[1] == kJntFree ? 7 : 0) > m.nq)
      return fail(KS_EINVAL, "ks_step: position actuators assume one actuator per joint after the root");
    a.substeps = io->substeps; a.actuator_period = io->actuator_period; a.actuator_type = io->actuator_type;
    a.action = io->action; a.last_ctrl = io->last_ctrl; a.latency = io->latency; a.zero_offset = io->zero_offset;
    a.drop = io->drop; a.kp = io->kp; a.kd = io->kd; a.ctrl_clip = io->ctrl_clip;
    a.kp_scale = io->kp_scale; a.kd_scale = io->kd_scale; a.torque_limit_scale = io->torque_limit_scale;
    a.action_scale = io->action_scale;
    a.action_noise = io->action_noise; a.torque_noise = io->torque_noise; a.action_bias = io->action_bias;
    a.torque_bias = io->torque_bias;
    if (io->n_events < 0 || io->n_events > KS_MAX_EVENTS) return fail(KS_ELIMIT, "ks_step: %d events (0..%d)", io->n_events, KS_MAX_EVENTS);
    if (io->n_events > 0) {
      if (!io->event_state) return fail(KS_EINVAL, "ks_step: events need event_state");
      for (int e = 0; e < io->n_events; ++e) {
        const KsEventDesc& ev = io->events[e];
        if (ev.kind < KS_EVENT_LINEAR_PUSH || ev.kind > KS_EVENT_FORCE_PUSH)
          return fail(KS_EINVAL, "ks_step: event %d: unknown kind %d", e, ev.kind);
        if (ev.kind == KS_EVENT_FORCE_PUSH) {
          if (ev.body < 1 || ev.body >= m.nb) return fail(KS_EINVAL, "ks_step: event %d: body %d outside 1..%d", e, ev.body, m.nb - 1);
          if (!io->event_force) return fail(KS_EINVAL, "ks_step: a force push needs event_force");
          ++a.n_force_events;
        } else if (m.nv < 6 || m.body_jtype[1] != kJntFree) {
          return fail(KS_EINVAL, "ks_step: velocity events push a floating base");
        }
      }
      a.event_force = io->event_force;
      a.n_events = io->n_events;
      for (int e = 0; e < io->n_events; ++e) a.events[e] = io->events[e];
      a.event_state = io->event_state; a.event_uniform = io->event_uniform; a.event_rng = io->event_rng;
    }
  }
  // stand-ins for the operands that were not given
  const DevModel* dm = km->dev;
  auto stand_in = [&](const float*& p, unsigned bit, const float* other) { if (p) a.given |= bit; else p = other; };
  stand_in(a.mass_scale, kOptMass, dm->ones); stand_in(a.damping_scale, kOptDamping, dm->ones); stand_in(a.armature_scale, kOptArmature, dm->ones);
  stand_in(a.body_ipos, kOptIpos, &dm->body_ipos[0][0]); stand_in(a.body_inertia, kOptInertia, &dm->body_inertia[0][0]);
  stand_in(a.sph_pos, kOptSphere, &dm->sph_pos[0][0]); stand_in(a.sph_radius, kOptSphere, dm->sph_radius);
  stand_in(a.kp_scale, kOptKp, dm->ones); stand_in(a.kd_scale, kOptKd, dm->ones); stand_in(a.torque_limit_scale, kOptLimit, dm->ones);
  stand_in(a.zero_offset, kOptZero, dm->zeros); stand_in(a.action_bias, kOptActionBias, dm->zeros);
  stand_in(a.torque_bias, kOptTorqueBias, dm->zeros); stand_in(a.action_noise, kOptActionNoise, dm->zeros);
  stand_in(a.torque_noise, kOptTorqueNoise, dm->zeros);
  stand_in(a.kp, 0u, dm->zeros); stand_in(a.kd, 0u, dm->zeros); stand_in(a.ctrl_clip, 0u, dm->zeros);  // torque actuators
  if (a.drop) a.given |= kOptDrop; else a.drop = reinterpret_cast<const uint8_t*>(dm->zeros);
  a.given |= (a.cinert ? kOutCinert : 0u) | (a.dbg_bias ? kOutBias : 0u) | (a.dbg_M ? kOutM : 0u) | (a.contact_dist ? kOutDist : 0u) |
             (a.dbg_qacc_smooth ? kOutSmooth : 0u) | (a.cfrc_ext ? kOutCfrc : 0u) | (a.qacc ? kOutQacc : 0u) | (a.solver_niter ? kOutNiter : 0u) |
             (a.nefc ? kOutNefc : 0u) | (a.n_events > 0 ? kHasEvents : 0u) | (a.n_force_events > 0 ? kHasForceEvents : 0u);
  const int bytes = lds_floats(m.nb, m.nq, m.nv, m.nu, m.ns) * 4;
  if (bytes > 160 * 1024) return fail(KS_ELIMIT, "ks_step: model needs %d bytes of LDS", bytes);
  void (*fn)(StepArgs) = nullptr;
  switch (padded_nv(m.nv)) {
#define KS_CASE(W)                                                                                       \
  case W:                                                                                                \
    fn = (m.dofrows || io->frictionloss) ? (forward_only ? step_kernel<true, W, true> : step_kernel<false, W, true>)           \
                   : (forward_only ? step_kernel<true, W, false> : step_kernel<false, W, false>);        \
    break;
    KS_CASE(8) KS_CASE(16) KS_CASE(24) KS_CASE(28) KS_CASE(32)
#undef KS_CASE
    default: return fail(KS_ELIMIT, "ks_step: no kernel for %d dofs", m.nv);
  }
  if (bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(KS_ELAUNCH, "ks_step: cannot raise the LDS limit: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)io->N), dim3(64), bytes, (hipStream_t)stream, a);
  return check_launch("ks_step");
}

extern "C" int ks_step(const KsModel* model, ks_stream_t stream, const KsStepIO* io) {
  return launch_step(model, stream, io, false);
}

extern "C" int ks_forward(const KsModel* model, ks_stream_t stream, const KsStepIO* io) {
  return launch_step(model, stream, io, true);
}

namespace ks {
constexpr int kWorkBuckets = 512, kWorkShift = 2, kWorkThreads = 256;  // buckets of four work units
constexpr int kXcds = 8;  // workgroup b of a launch runs on XCD b % 8, each XCD with an L2 of its own
__device__ __forceinline__ int work_bucket(int w) { return min(max(w, 0) >> kWorkShift, kWorkBuckets - 1); }
// Counting sort of envs by descending work in one workgroup: histogram, suffix sums, scatter.
// With gridDim.x == 8 (N a multiple of 8) workgroup r sorts the envs of region r = [r N / 8, (r + 1) N / 8) and writes them
// to order[r], order[r + 8], ...: the step kernel's workgroup b = r + 8 k then runs on XCD r and finds there only envs of
// region r.  The state rows of neighbouring envs share 128-byte lines (an env's qpos row is 108 bytes); kept inside one XCD
// such a line is fetched into, and written back from, one L2 instead of two.
// Four wavefronts and 4 KB of LDS: in a rollout on several streams this launch has to find room on a CU that another group's
// physics launch fills, and a small workgroup finds it as soon as one wavefront per SIMD has left.
__global__ __launch_bounds__(kWorkThreads) void work_order_kernel(int64_t N, const int32_t* __restrict__ work, int32_t* __restrict__ order) {
  __shared__ int hist[kWorkBuckets];
  __shared__ int scan[kWorkBuckets];
  const int t = threadIdx.x;
  const int regions = gridDim.x, region = blockIdx.x;
  const int64_t n = N / regions, first = region * n;
  for (int b = t; b < kWorkBuckets; b += kWorkThreads) hist[b] = 0;
  __syncthreads();
  for (int64_t i = t; i < n; i += kWorkThreads) atomicAdd(&hist[work_bucket(work[first + i])], 1);
  __syncthreads();
  // inclusive suffix sums (heaviest bucket first) by doubling
  for (int b = t; b < kWorkBuckets; b += kWorkThreads) scan[b] = hist[b];
  __syncthreads();
  for (int off = 1; off < kWorkBuckets; off <<= 1) {
    int v[kWorkBuckets / kWorkThreads];
    for (int k = 0; k < kWorkBuckets / kWorkThreads; ++k) {
      const int b = t + kWorkThreads * k;
      v[k] = scan[b] + (b + off < kWorkBuckets ? scan[b + off] : 0);
    }
    __syncthreads();
    for (int k = 0; k < kWorkBuckets / kWorkThreads; ++k) scan[t + kWorkThreads * k] = v[k];
    __syncthreads();
  }
  // bucket b starts after all heavier buckets: scan[b] - hist[b]
  for (int b = t; b < kWorkBuckets; b += kWorkThreads) hist[b] = scan[b] - hist[b];
  __syncthreads();
  for (int64_t i = t; i < n; i += kWorkThreads) {
    const int pos = atomicAdd(&hist[work_bucket(work[first + i])], 1);
    order[(int64_t)pos * regions + region] = (int32_t)(first + i);
  }
}
}  // namespace ks

extern "C" int ks_work_order(ks_stream_t stream, int64_t N, const int32_t* work, int32_t* order) {
  using namespace ks;
  if (N < 0 || N > 0x7fffffff) return fail(KS_EINVAL, "ks_work_order: bad env count");
  if (N == 0) return KS_OK;
  if (!work || !order) return fail(KS_EINVAL, "ks_work_order: null argument");
  const int regions = (N % kXcds == 0 && N >= 64 * kXcds) ? kXcds : 1;
  hipLaunchKernelGGL(work_order_kernel, dim3(regions), dim3(kWorkThreads), 0, (hipStream_t)stream, N, work, order);
  return check_launch("ks_work_order");
}
