"""GAE / PPO-loss host interface with the reference's names and argument meaning.

Mirrors ksim/task/ppo.py: ``compute_ppo_inputs`` (54-121), ``clipped_value_loss``
(124-135 — folded into the loss kernel), ``compute_ppo_loss`` (149-246),
``PPOInputs`` / ``PPOVariables`` (ppo.py:30-47 in the reference).  Arrays are torch
CUDA tensors of shape (B, T) (log-probs (B, T, A)); the arithmetic runs in the HIP
kernels of libksimhip.so.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Mapping

import torch

from . import _lib


@dataclass
class PPOInputs:
    advantages_bt: torch.Tensor
    value_targets_bt: torch.Tensor
    gae_bt: torch.Tensor
    returns_bt: torch.Tensor


@dataclass
class PPOVariables:
    log_probs: torch.Tensor
    values: torch.Tensor
    entropy: torch.Tensor | None = None
    aux_losses: Mapping[str, torch.Tensor] | None = None


def _as_bytes(x: torch.Tensor) -> torch.Tensor:
    if x.dtype == torch.bool:
        return x.view(torch.uint8)
    if x.dtype in (torch.uint8, torch.int8):
        return x
    raise _lib.KsError(f"dones/successes must be bool or 1-byte integers, got {x.dtype}")


def _workspace(device) -> torch.Tensor:
    return torch.empty(_lib.KS_REDUCE_WORKSPACE_BYTES, dtype=torch.uint8, device=device)


def compute_ppo_inputs(
    values_bt: torch.Tensor,
    rewards_bt: torch.Tensor,
    dones_bt: torch.Tensor,
    successes_bt: torch.Tensor | None,
    decay_gamma: float,
    gae_lambda: float,
    normalize_advantages: bool = False,
    monte_carlo_returns: bool = False,
    *,
    time_major: bool = False,
) -> PPOInputs:
    """GAE and returns. ``time_major=True`` takes (T, N) arrays (the rollout buffer's layout)."""
    lib = _lib.load()
    dones = _as_bytes(dones_bt)
    succ = None if successes_bt is None else _as_bytes(successes_bt)
    _lib.require_cuda(values_bt, rewards_bt, dtype=torch.float32)
    _lib.require_cuda(dones, succ)
    if values_bt.dim() != 2 or rewards_bt.shape != values_bt.shape or dones.shape != values_bt.shape:
        raise _lib.KsError("values, rewards and dones must share one 2-D shape")
    if succ is not None and succ.shape != values_bt.shape:
        raise _lib.KsError("successes must have the shape of values")
    stream, addr = _lib.current_stream(), _lib.addr
    gae, ret, tgt = torch.empty_like(values_bt), torch.empty_like(values_bt), torch.empty_like(values_bt)
    adv = gae
    if normalize_advantages:
        adv, ws = torch.empty_like(values_bt), _workspace(values_bt.device)
        _lib.check(lib.ks_gae_normalized(stream, time_major, *values_bt.shape, addr(values_bt), addr(rewards_bt), addr(dones), addr(succ),
                                         decay_gamma, gae_lambda, int(monte_carlo_returns), addr(gae), addr(ret), addr(tgt), addr(adv),
                                         addr(ws)))
    else:
        fn = lib.ks_gae_tn if time_major else lib.ks_gae_bt
        _lib.check(fn(stream, *values_bt.shape, addr(values_bt), addr(rewards_bt), addr(dones), addr(succ), decay_gamma, gae_lambda,
                      int(monte_carlo_returns), addr(gae), addr(ret), addr(tgt)))
    return PPOInputs(advantages_bt=adv, value_targets_bt=tgt, gae_bt=gae, returns_bt=ret)


def compute_ppo_loss(
    ppo_inputs: PPOInputs,
    on_policy_variables: PPOVariables,
    off_policy_variables: PPOVariables,
    *,
    clip_param: float = 0.2,
    value_loss_coef: float = 0.5,
    entropy_coef: float = 0.008,
    kl_coef: float = 1e-3,
    log_clip_value: float = 5.0,
    use_clipped_value_loss: bool = True,
    kl_scale: float = 1.0,
) -> dict[str, torch.Tensor]:
    """Per-element loss terms (B, T) plus ``"total"`` = mean over (B, T) of their sum (ppo.py:485-486)."""
    lib = _lib.load()
    on, off = on_policy_variables, off_policy_variables
    if on.log_probs.dim() != 3 or off.log_probs.shape != on.log_probs.shape:
        raise _lib.KsError("log_probs must be rank 3 (B, T, A) and match")
    if on.values.dim() != 2 or off.values.dim() != 2 or ppo_inputs.advantages_bt.dim() != 2:
        raise _lib.KsError("values and advantages must be rank 2 (B, T)")
    B, T, A = on.log_probs.shape
    for x in (on.values, off.values, ppo_inputs.advantages_bt, ppo_inputs.value_targets_bt):
        if tuple(x.shape) != (B, T):
            raise _lib.KsError("shape prefix mismatch between log_probs, values and ppo inputs")
    _lib.require_cuda(on.log_probs, on.values, off.log_probs, off.values, off.entropy, ppo_inputs.advantages_bt,
                      ppo_inputs.value_targets_bt, dtype=torch.float32)
    dev = on.values.device
    names = ("policy", "value", "kl") if off.entropy is None else ("policy", "value", "kl", "entropy")
    out = {k: torch.empty_like(on.values) for k in names}
    total = torch.empty((), dtype=torch.float32, device=dev)
    params = _lib.KsPpoLossParams(clip_param, value_loss_coef, entropy_coef, kl_coef, log_clip_value, kl_scale,
                                  int(use_clipped_value_loss))
    ws, addr = _workspace(dev), _lib.addr
    _lib.check(
        lib.ks_ppo_loss(_lib.current_stream(), B * T, A, params, addr(ppo_inputs.advantages_bt), addr(ppo_inputs.value_targets_bt),
                        addr(on.log_probs), addr(on.values), addr(off.log_probs), addr(off.values), addr(off.entropy), addr(out["policy"]),
                        addr(out["value"]), addr(out["kl"]), addr(out.get("entropy")), addr(total), addr(ws))
    )
    if off.aux_losses is not None:  # ppo.py:242-244 — user terms pass through and join the mean
        aux_sum = None
        for name, term in off.aux_losses.items():
            out[name] = term
            aux_sum = term if aux_sum is None else aux_sum + term
        total = total + aux_sum.mean()
    out["total"] = total
    return out
