// Kernel argument block of the fused control-step kernel (device pointers, passed by value).
#pragma once
#include <stdint.h>

#include "../../include/ksim_hip.h"
#include "ks_model.h"

namespace ks {

// Operands that a call may leave out.  Their pointers are never null in the kernel: what is not given points at ones, zeros or the
// model's own values, and its bit in StepArgs::given is clear, which takes the env out of the index.  The loads of a substep are then
// straight-line code with one latency between them, where a branch around each was a round trip of its own.
enum StepOptional : unsigned {
  kOptMass = 1u << 0, kOptDamping = 1u << 1, kOptArmature = 1u << 2, kOptIpos = 1u << 3, kOptInertia = 1u << 4, kOptSphere = 1u << 5,
  kOptKp = 1u << 6, kOptKd = 1u << 7, kOptLimit = 1u << 8, kOptZero = 1u << 9, kOptDrop = 1u << 10, kOptActionBias = 1u << 11,
  kOptTorqueBias = 1u << 12, kOptActionNoise = 1u << 13, kOptTorqueNoise = 1u << 14,
  // what else a substep asks about: outputs that are wanted, and events
  kOutCinert = 1u << 15, kOutBias = 1u << 16, kOutM = 1u << 17, kOutDist = 1u << 18, kOutSmooth = 1u << 19, kOutCfrc = 1u << 20,
  kOutQacc = 1u << 21, kOutNiter = 1u << 22, kOutNefc = 1u << 23, kHasEvents = 1u << 24, kHasForceEvents = 1u << 25,
};

struct StepArgs {
  const DevModel* model;
  ModelHead head;
  unsigned given;
  int64_t N;
  int substeps, actuator_period, actuator_type;
  float action_scale;
  float *qpos, *qvel, *qacc_warmstart, *time, *last_ctrl;
  const float *action, *ctrl_in, *latency, *zero_offset;
  const uint8_t* drop;
  const float *kp, *kd, *ctrl_clip, *kp_scale, *kd_scale, *torque_limit_scale;
  const float *action_bias, *torque_bias, *action_noise, *torque_noise;
  const float *friction, *mass_scale;
  const uint8_t* env_mask;
  const uint8_t* fresh;
  float *qacc, *ctrl_out, *xpos, *xquat, *cvel, *traj_ctrl, *traj_xpos, *traj_xquat;
  int32_t *solver_niter, *nefc;
  float *dbg_M, *dbg_bias, *dbg_qacc_smooth, *contact_dist, *cinert, *cfrc_ext;
  const float *armature_scale, *damping_scale;
  const float *frictionloss, *body_ipos, *body_inertia, *sph_pos, *sph_radius;
  const int32_t* env_order;
  int32_t* work;
  int n_events;
  KsEventDesc events[KS_MAX_EVENTS];
  float* event_state;
  const float* event_uniform;
  KsRng event_rng;
  float* event_force;
  int n_force_events;
};

}  // namespace ks
