"""MLP forward on the matrix cores (policy / critic / discriminator networks of the rollout path).

The reference leaves the network to the task (``sample_action``, ksim/task/rl.py:892-926); the configs here
use plain MLP stacks.  Weights are given as (out, in) fp32 arrays, like the reference's linear layers.
"""
from __future__ import annotations

import ctypes
from typing import Sequence

import numpy as np
import torch

from . import _lib
from . import _lib_terms as T

_ACT = {None: T.ACT_NONE, "none": T.ACT_NONE, "elu": T.ACT_ELU, "relu": T.ACT_RELU, "tanh": T.ACT_TANH,
        "gelu": T.ACT_GELU}


class MLP:
    def __init__(self, weights: Sequence, biases: Sequence, activation: str = "elu", dtype: str = "bf16"):
        lib = _lib.load()
        if len(weights) != len(biases) or not weights:
            raise _lib.KsError("one bias per weight matrix is required")
        if dtype not in ("bf16", "f32"):
            raise _lib.KsError("dtype must be 'bf16' or 'f32'")
        torch.zeros(1, device="cuda")  # make sure a HIP context exists before the library allocates
        ws = [np.ascontiguousarray(w.detach().cpu().numpy() if isinstance(w, torch.Tensor) else w, dtype=np.float32)
              for w in weights]
        bs = [np.ascontiguousarray(b.detach().cpu().numpy() if isinstance(b, torch.Tensor) else b, dtype=np.float32)
              for b in biases]
        dims = [ws[0].shape[1]]
        for w, b in zip(ws, bs):
            if w.ndim != 2 or w.shape[1] != dims[-1] or b.shape != (w.shape[0],):
                raise _lib.KsError("weight / bias shapes do not chain")
            dims.append(w.shape[0])
        d = T.KsMlpDesc()
        d.n_layers, d.activation = len(ws), _ACT[activation]
        d.dtype = T.MLP_BF16 if dtype == "bf16" else T.MLP_F32
        for i, v in enumerate(dims):
            d.dims[i] = v
        for i, (w, b) in enumerate(zip(ws, bs)):
            d.weights[i] = w.ctypes.data
            d.biases[i] = b.ctypes.data
        self.dims, self.dtype, self.activation = dims, dtype, activation
        self._lib = lib
        self._handle = ctypes.c_void_p()
        _lib.check(lib.ks_mlp_create(ctypes.byref(d), ctypes.byref(self._handle)))

    @property
    def in_dim(self) -> int:
        return self.dims[0]

    @property
    def out_dim(self) -> int:
        return self.dims[-1]

    def flops_per_row(self) -> int:
        return 2 * sum(a * b for a, b in zip(self.dims[:-1], self.dims[1:]))

    def workspace(self, M: int, device) -> torch.Tensor | None:
        """Scratch of one call on `M` rows, None where the call needs none.  It belongs to the call: taken from torch's allocator on the
        current stream and given back there when the launches are queued.  Calls on other streams, in other threads and in other captured
        graphs never share it, and a replayed graph finds it in the graph's own memory."""
        need = int(self._lib.ks_mlp_workspace_bytes(self._handle, M))
        return torch.empty(need, dtype=torch.uint8, device=device) if need else None

    def __call__(self, x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
        _lib.require_cuda(x, dtype=torch.float32)
        if x.dim() != 2 or x.shape[1] != self.in_dim:
            raise _lib.KsError(f"expected input (M, {self.in_dim}), got {tuple(x.shape)}")
        M = x.shape[0]
        if out is None:
            out = torch.empty((M, self.out_dim), dtype=torch.float32, device=x.device)
        else:
            _lib.require_cuda(out, dtype=torch.float32)
            if tuple(out.shape) != (M, self.out_dim):
                raise _lib.KsError("output has the wrong shape")
        ws = self.workspace(M, x.device)
        _lib.check(self._lib.ks_mlp_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(out),
                                            _lib.addr(ws)))
        return out

    def forward_pair(self, x: torch.Tensor, out: torch.Tensor, other: "MLP", x_other: torch.Tensor,
                     out_other: torch.Tensor, sample: "T.KsActionSample | None" = None) -> None:
        """This network on ``x`` and ``other`` on ``x_other`` (same row count), in one launch when the library can; with ``sample``
        (`env_terms.action_sample`) also the actions of this network's output."""
        M = x.shape[0]
        for net, a, o in ((self, x, out), (other, x_other, out_other)):
            _lib.require_cuda(a, dtype=torch.float32)
            _lib.require_cuda(o, dtype=torch.float32)
            if tuple(a.shape) != (M, net.in_dim) or tuple(o.shape) != (M, net.out_dim):
                raise _lib.KsError(f"expected input (M, {net.in_dim}) and output (M, {net.out_dim})")
        ws, ws_other = self.workspace(M, x.device), other.workspace(M, x.device)  # both held until both are launched
        args = (self._handle, other._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(out), _lib.addr(x_other), _lib.addr(out_other),
                _lib.addr(ws), _lib.addr(ws_other))
        _lib.check(self._lib.ks_mlp_forward_pair(*args) if sample is None else self._lib.ks_mlp_forward_pair_sample(*args, ctypes.byref(sample)))

    # ------------------------------------------------------------------ training (ksim/task/ppo.py:495-565)
    def train_init(self) -> None:
        """fp32 master weights, gradients and Adam moments beside the working copies."""
        _lib.check(self._lib.ks_mlp_train_init(self._handle))
        self._training = True

    def _train_ws(self, M: int, device) -> torch.Tensor:
        need = int(self._lib.ks_mlp_train_workspace_bytes(self._handle, M))
        ws = getattr(self, "_tws", None)
        if ws is None or ws.numel() < need or ws.device != torch.device(device):
            ws = torch.empty(need, dtype=torch.uint8, device=device)
            self._tws = ws
        return ws

    def train_forward(self, x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
        """Forward pass that keeps the hidden activations for `backward` (same rows, called next)."""
        _lib.require_cuda(x, dtype=torch.float32)
        if x.dim() != 2 or x.shape[1] != self.in_dim:
            raise _lib.KsError(f"expected input (M, {self.in_dim}), got {tuple(x.shape)}")
        M = x.shape[0]
        if out is None:
            out = torch.empty((M, self.out_dim), dtype=torch.float32, device=x.device)
        _lib.check(self._lib.ks_mlp_train_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(out),
                                                  _lib.addr(self._train_ws(M, x.device))))
        return out

    def backward(self, x: torch.Tensor, dy: torch.Tensor) -> None:
        """Gradients of sum(dy * net(x)) into the handle; `x` is the input of the preceding `train_forward`."""
        _lib.require_cuda(x, dy, dtype=torch.float32)
        if tuple(dy.shape) != (x.shape[0], self.out_dim):
            raise _lib.KsError("dy must have the shape of the network output")
        _lib.check(self._lib.ks_mlp_train_backward(self._handle, _lib.current_stream(), x.shape[0], _lib.addr(x),
                                                   _lib.addr(dy), _lib.addr(self._train_ws(x.shape[0], x.device))))

    def backward_dx(self, x: torch.Tensor | None, dy: torch.Tensor, dx: torch.Tensor, *, weight_gradients: bool = True,
                    accumulate: bool = False, zero_rows: torch.Tensor | None = None) -> torch.Tensor:
        """`backward` that also writes (or adds) the gradient with respect to the network input into `dx`; without
        `weight_gradients` only that.  Rows flagged in `zero_rows` (uint8) get a zero input gradient."""
        _lib.require_cuda(x, dy, dx, dtype=torch.float32)
        M = dy.shape[0]
        if tuple(dy.shape) != (M, self.out_dim) or tuple(dx.shape) != (M, self.in_dim) or (x is not None and tuple(x.shape) != (M, self.in_dim)):
            raise _lib.KsError("x and dx must be (M, in), dy (M, out)")
        if x is None and weight_gradients:
            raise _lib.KsError("the weight gradients need the input")
        if zero_rows is not None:
            _lib.require_cuda(zero_rows, dtype=torch.uint8)
            if tuple(zero_rows.shape) != (M,):
                raise _lib.KsError("zero_rows must be (M,) uint8")
        _lib.check(self._lib.ks_mlp_train_backward_dx(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(dy),
                                                      _lib.addr(dx), int(weight_gradients), int(accumulate),
                                                      _lib.addr(zero_rows), _lib.addr(self._train_ws(M, dy.device))))
        return dx

    def layer_weight_grad(self, x: torch.Tensor, dy: torch.Tensor) -> None:
        """`backward` of a network of one layer whose input rows are a block of columns of wider rows: x (M, in), its columns side by side."""
        _lib.require_cuda(dy, dtype=torch.float32)
        if not x.is_cuda or x.dtype != torch.float32 or x.dim() != 2 or x.shape[1] != self.in_dim or x.stride(1) != 1 or x.stride(0) < self.in_dim:
            raise _lib.KsError(f"expected fp32 rows of {self.in_dim} on the GPU, columns side by side")
        if tuple(dy.shape) != (x.shape[0], self.out_dim):
            raise _lib.KsError("dy must have the shape of the network output")
        _lib.check(self._lib.ks_mlp_layer_weight_grad(self._handle, _lib.current_stream(), x.shape[0], x.data_ptr(), x.stride(0), dy.data_ptr(),
                                                      _lib.addr(self._train_ws(x.shape[0], x.device))))

    def disc_loss_grad(self, real: torch.Tensor, sim: torch.Tensor, grad_penalty_coef: float) -> torch.Tensor:
        """Gradient of the AMP discriminator loss (ksim/task/amp.py:360-438) into the handle: real (B, T, in) reference
        motions, sim (B2, T2, in) simulated ones; returns the (real, simulated, penalty) terms of the loss, on the device."""
        _lib.require_cuda(real, sim, dtype=torch.float32)
        if real.dim() != 3 or sim.dim() != 3 or real.shape[2] != self.in_dim or sim.shape[2] != self.in_dim:
            raise _lib.KsError(f"motions must be (B, T, {self.in_dim}), got {tuple(real.shape)} and {tuple(sim.shape)}")
        n_real, n_sim = real.shape[0] * real.shape[1], sim.shape[0] * sim.shape[1]
        need = int(self._lib.ks_mlp_disc_workspace_bytes(self._handle, n_real, n_sim))
        ws = getattr(self, "_dws", None)
        if ws is None or ws.numel() < need or ws.device != real.device:
            ws = torch.empty(need, dtype=torch.uint8, device=real.device)
            self._dws = ws
        losses = torch.empty(3, dtype=torch.float32, device=real.device)
        _lib.check(self._lib.ks_mlp_disc_loss_grad(self._handle, _lib.current_stream(), n_real, _lib.addr(real), n_sim, _lib.addr(sim),
                                                   float(grad_penalty_coef), max(real.shape[0], 1), _lib.addr(losses), _lib.addr(ws)))
        return losses

    @classmethod
    def _borrow(cls, lib, handle, dims, dtype: str) -> "MLP":
        """A view of a network that another object owns (the projections inside a GRU cell): never destroyed here."""
        self = cls.__new__(cls)
        self._lib, self._handle, self.dims, self.dtype, self.activation = lib, handle, list(dims), dtype, "none"
        self._borrowed = True
        return self

    def networks(self) -> list["MLP"]:
        """The networks whose parameters an optimiser step over this one updates."""
        return [self]

    def grad_sqnorm(self, acc: torch.Tensor) -> None:
        _lib.require_cuda(acc, dtype=torch.float64)
        _lib.check(self._lib.ks_mlp_grad_sqnorm(self._handle, _lib.current_stream(), _lib.addr(acc)))

    def adam_step(self, params: "T.KsAdamParams", sqnorm: torch.Tensor | None) -> None:
        _lib.check(self._lib.ks_mlp_adam_step(self._handle, _lib.current_stream(), ctypes.byref(params), _lib.addr(sqnorm)))

    def parameters(self, gradients: bool = False) -> list[tuple[torch.Tensor, torch.Tensor]]:
        """[(weight (out, in), bias (out))] copies of the fp32 master parameters, or of their gradients."""
        return copy_parameters([self], gradients)[0]

    def close(self) -> None:
        if getattr(self, "_borrowed", False):
            return
        if self._handle:
            self._lib.ks_mlp_destroy(self._handle)
            self._handle = ctypes.c_void_p()

    def __del__(self):  # pragma: no cover
        try:
            self.close()
        except Exception:
            pass


def _handles(nets: Sequence[MLP]):
    return (ctypes.c_void_p * len(nets))(*[net._handle for net in nets])


def copy_parameters(nets: Sequence[MLP], gradients: bool = False) -> list[list[tuple[torch.Tensor, torch.Tensor]]]:
    """`MLP.parameters` of several networks, in one launch."""
    empty, f32, dev = torch.empty, torch.float32, torch.device("cuda", torch._C._cuda_getDevice())
    out = [[(empty((o, i), dtype=f32, device=dev), empty((o,), dtype=f32, device=dev)) for i, o in zip(net.dims[:-1], net.dims[1:])] for net in nets]
    table = ctypes.c_void_p * sum(map(len, out))
    _lib.check(_lib.load().ks_mlps_copy_params(_handles(nets), len(nets), _lib.current_stream(), table(*[w.data_ptr() for net in out for w, _ in net]),
                                               table(*[b.data_ptr() for net in out for _, b in net]), int(gradients)))
    return out


def grad_sqnorm(nets: Sequence[MLP], acc: torch.Tensor) -> None:
    """Adds the squared gradient norm over all of `nets` to `acc`."""
    _lib.require_cuda(acc, dtype=torch.float64)
    _lib.check(_lib.load().ks_mlps_grad_sqnorm(_handles(nets), len(nets), _lib.current_stream(), _lib.addr(acc)))


def adam_step(nets: Sequence[MLP], params: "T.KsAdamParams", sqnorm: torch.Tensor | None) -> None:
    """One optimiser step of all of `nets`; `sqnorm` is the squared gradient norm over everything optimised together."""
    _lib.check(_lib.load().ks_mlps_adam_step(_handles(nets), len(nets), _lib.current_stream(), ctypes.byref(params), _lib.addr(sqnorm)))


def random_mlp(dims: Sequence[int], seed: int, activation: str = "elu", dtype: str = "bf16"):
    """Random-init network: W ~ N(0, 1/fan_in), b = 0. Returns (MLP, weights, biases)."""
    rng = np.random.default_rng(seed)
    ws = [rng.normal(scale=1.0 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [np.zeros(o, dtype=np.float32) for o in dims[1:]]
    return MLP(ws, bs, activation=activation, dtype=dtype), ws, bs
