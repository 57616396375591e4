"""Host side of the AMP discriminator update (ksim/task/amp.py:441-545): batches of reference and simulated motions, the
loss gradient (`ks_mlp_disc_loss_grad`), the optimiser step, `disc_num_passes` times per policy update.

The discriminator is an `MLP` with one output that scores each frame of a motion, so a motion (T, F) gets logits (T,) as
`AMPTask.call_discriminator` asks (amp.py:257-268).  The AMP reward from those logits is `ksim_amd.rewards.AMPReward`.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from . import _lib
from . import _lib_terms as T
from .mlp import MLP


@dataclass
class AMPConfig:  # the discriminator's part of ksim/task/amp.py:62-95
    amp_reference_batch_size: int = 32
    disc_num_passes: int = 1
    amp_grad_penalty_coef: float = 10.0
    learning_rate: float = 3e-4
    adam_b1: float = 0.9
    adam_b2: float = 0.999
    adam_eps: float = 1e-8
    weight_decay: float = 0.0
    max_grad_norm: float | None = None


def loop_slice(clip: torch.Tensor, start: int, window_t: int) -> torch.Tensor:
    """A window of `window_t` frames from `start`, wrapping round when the clip is shorter (amp.py:53-58)."""
    idx = (torch.arange(window_t, device=clip.device) + int(start)) % clip.shape[0]
    return clip[idx]


def _on_device(rows: torch.Tensor, device: torch.device) -> torch.Tensor:
    """Indices drawn on the host, where the motions are: in one copy that nothing waits for (a copy from pageable memory would hold the host until
    the GPU has caught up)."""
    if device.type == "cuda":
        rows = torch.empty(rows.shape, dtype=torch.int64, pin_memory=True).copy_(rows).to(device, non_blocking=True)
    return rows


def _draw_clips(n: int, t_clip: int, batch_b: int, generator: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    return torch.randint(0, n, (batch_b,), generator=generator), torch.randint(0, t_clip, (batch_b,), generator=generator)


def _draw_envs(num_envs: int, batch_b: int, generator: torch.Generator) -> torch.Tensor:
    """All envs in the order drawn; the first `batch_b` are the batch's."""
    if num_envs % batch_b != 0:
        raise ValueError(f"amp_reference_batch_size ({batch_b}) must divide batch_size ({num_envs}).")
    return torch.randperm(num_envs, generator=generator)


def _windows(motions: torch.Tensor, window_t: int, clip_idx: torch.Tensor, starts: torch.Tensor) -> torch.Tensor:
    t_clip, batch_b = motions.shape[1], clip_idx.shape[0]
    # every window of the batch in one gather: frame (start + t) mod T_clip of the drawn clip, as loop_slice takes them
    frames = (starts[:, None] + torch.arange(window_t)[None, :]) % t_clip
    if motions.is_contiguous():
        rows = _on_device((clip_idx[:, None] * t_clip + frames).view(-1), motions.device)
        return motions.view(motions.shape[0] * t_clip, *motions.shape[2:]).index_select(0, rows).view(batch_b, window_t, *motions.shape[2:])
    # strided or expanded clips: indexed where they are (a flat view of them would be a copy of every clip)
    both = _on_device(torch.stack([clip_idx[:, None].expand_as(frames), frames]), motions.device)
    return motions[both[0], both[1]]


def _sequences(sim_motions: torch.Tensor, envs: torch.Tensor) -> torch.Tensor:
    return sim_motions.index_select(0, _on_device(envs, sim_motions.device))


def make_real_batch(motions: torch.Tensor, window_t: int, batch_b: int, generator: torch.Generator) -> torch.Tensor:
    """`batch_b` windows from reference clips (N, T_clip, F): a clip drawn uniformly, then a uniform start in it
    (amp.py:570-625; the draws come from `generator`, not from jax's key splitting)."""
    return _windows(motions, window_t, *_draw_clips(motions.shape[0], motions.shape[1], batch_b, generator))


def make_sim_batch(sim_motions: torch.Tensor, batch_b: int, generator: torch.Generator) -> torch.Tensor:
    """`batch_b` distinct envs of the rollout's motions (num_envs, T, F) (amp.py:627-652)."""
    return _sequences(sim_motions, _draw_envs(sim_motions.shape[0], batch_b, generator)[:batch_b])


def _batches(motions: torch.Tensor, sim_motions: torch.Tensor, batch_b: int, generator: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    """`make_real_batch` and `make_sim_batch` of one step, in one launch where both are plain fp32 arrays of frames on one GPU and what was drawn
    is in host memory, where the launcher reads it (a default device and a generator of its kind draw elsewhere).  Not while the stream is captured:
    a graph would replay one step's draws for ever, and the functions of the single batches refuse that."""
    shape, (num_envs, window_t) = motions.shape, sim_motions.shape[:2]
    clip_idx, starts = _draw_clips(shape[0], shape[1], batch_b, generator)
    envs = _draw_envs(num_envs, batch_b, generator)
    plain = (1 <= batch_b <= T.KS_WINDOWS and len(shape) == sim_motions.dim() == 3 and shape[2] == sim_motions.shape[2]
             and motions.dtype == sim_motions.dtype == torch.float32 and motions.is_cuda and motions.device == sim_motions.device
             and motions.is_contiguous() and sim_motions.is_contiguous() and motions.numel() > 0 and sim_motions.numel() > 0
             and (shape[1] + window_t) * shape[2] <= T.KS_WINDOW_FLOATS
             and motions.device.index == torch._C._cuda_getDevice() and clip_idx.is_cpu and starts.is_cpu and envs.is_cpu
             and not torch._C._cuda_isCurrentStreamCapturing())
    if not plain:
        return _windows(motions, window_t, clip_idx, starts), _sequences(sim_motions, envs[:batch_b])
    n, t_clip, frame = shape
    real, sim = (torch.empty((batch_b, window_t, frame), dtype=torch.float32, device=motions.device) for _ in range(2))
    _lib.check(_lib.load().ks_gather_windows(_lib.current_stream(), batch_b, window_t, frame, n, t_clip, num_envs, motions.data_ptr(), sim_motions.data_ptr(),
                                             clip_idx.data_ptr(), starts.data_ptr(), envs.data_ptr(), real.data_ptr(), sim.data_ptr()))
    return real, sim


class DiscriminatorUpdate:
    """Owns the discriminator's optimiser state; `step` is one pass of amp.py:486-527, `update` all of them."""

    def __init__(self, disc: MLP, cfg: AMPConfig):
        if disc.out_dim != 1:
            raise _lib.KsError(f"the discriminator scores a frame with one number, not {disc.out_dim}")
        self.disc, self.cfg, self.count = disc, cfg, 0
        disc.train_init()
        self._acc = torch.zeros(1, dtype=torch.float64, device="cuda")

    def loss_grad(self, real: torch.Tensor, sim: torch.Tensor) -> torch.Tensor:
        """Gradients into the discriminator's buffers; returns the (real, simulated, penalty) loss terms, on the device."""
        return self.disc.disc_loss_grad(real, sim, self.cfg.amp_grad_penalty_coef)

    def step(self, real: torch.Tensor, sim: torch.Tensor) -> dict[str, torch.Tensor]:
        losses = self.loss_grad(real, sim)
        sq = None
        if self.cfg.max_grad_norm is not None:
            self._acc.zero_()
            self.disc.grad_sqnorm(self._acc)
            sq = self._acc
        self.count += 1
        c = self.cfg
        self.disc.adam_step(T.KsAdamParams(c.learning_rate, c.adam_b1, c.adam_b2, c.adam_eps, c.weight_decay,
                                           0.0 if c.max_grad_norm is None else c.max_grad_norm, self.count), sq)
        return {"disc_loss": losses.sum(), "disc_real_loss": losses[0], "disc_sim_loss": losses[1], "disc_gp_loss": losses[2]}

    def update(self, motions: torch.Tensor, sim_motions: torch.Tensor, generator: torch.Generator) -> dict[str, torch.Tensor]:
        """`disc_num_passes` steps, each on fresh batches; the metrics are averaged over the passes (amp.py:529-536)."""
        sums: dict[str, torch.Tensor] = {}
        for _ in range(self.cfg.disc_num_passes):
            for k, v in self.step(*_batches(motions, sim_motions, self.cfg.amp_reference_batch_size, generator)).items():
                sums[k] = v if k not in sums else sums[k] + v
        return sums if self.cfg.disc_num_passes == 1 else {k: v / self.cfg.disc_num_passes for k, v in sums.items()}
