"""Recurrent policy / critic networks for the rollout, and the backward pass through time of the GRU stack.

The shipped examples build their actor and critic as an input projection, a stack of GRU cells and an output MLP
(examples/walking.py:40-208); the carry `(depth, N, hidden)` travels with the env state and is zeroed for envs that
start an episode (ksim/task/rl.py:1072-1080).  Weights use the (out, in) layout and gate order (reset | update |
candidate) of the reference's cells.
"""
from __future__ import annotations

import ctypes
from typing import Sequence

import numpy as np
import torch

from . import _lib
from . import _lib_terms as T
from . import mlp as mlp_mod
from .mlp import MLP


# (step, env) rows that `RecurrentNetwork.forward_sequence` takes through the layers at a time: a layer keeps its input, its projected input and
# its states of that many, 0.5 GB for an LSTM of hidden size 128, whatever the length of the rollout
SEQUENCE_ROWS = 131072


# (step, env) rows up to which `RecurrentNetwork.backward` puts all weight gradients into one launch at its end; us of an update at the end and layer
# by layer: LSTM 1536 rows 922 and 932, 12800 1260 and 1282, 32768 1902 and 1974, 51200 2993 and 2936; GRU in bf16 12288 855 and 864, 32768 1450 and
# 1450, 65536 2696 and 2716; GRU in fp32 16384 1221 and 1204
LATER_ROWS = 32768


def _f32(a) -> np.ndarray:
    return np.ascontiguousarray(a.detach().cpu().numpy() if isinstance(a, torch.Tensor) else a, dtype=np.float32)


class SequenceCall:
    """The recurrence of one layer over a trajectory, ready to launch; holds what the launch reads and writes."""

    def __init__(self, entry: str, dtype: str, steps: int, rows: int, handle, x, h0, c0, fresh, saved, out0, out1):
        self.key, self.steps, self.rows, self.handle = (entry, dtype, steps), steps, rows, handle
        self.tensors = (x, h0, c0, fresh, saved, out0, out1)

    def record(self) -> "T.KsSequence":
        return T.KsSequence(self.handle.value, self.rows, *map(_lib.addr, self.tensors), None, None)


def run_sequences(calls: Sequence[SequenceCall]) -> None:
    """Launches the calls: two of one kind, precision and length (a layer of the actor and one of the critic) together, which keeps a chip busy
    that either of them fills halfway; others one after the other."""
    lib, stream = _lib.load(), _lib.current_stream()
    calls = list(calls)
    while calls:
        n = 2 if len(calls) > 1 and calls[0].key == calls[1].key else 1
        _lib.check(getattr(lib, calls[0].key[0])(stream, n, calls[0].steps, (T.KsSequence * n)(*(c.record() for c in calls[:n]))))
        del calls[:n]


class LayerForward:
    """A single layer over rows x (M, in), ready to launch; `out` (M, out) holds the result then."""

    def __init__(self, net: MLP, x: torch.Tensor, out: torch.Tensor | None = None):
        self.net, self.x = net, x
        self.out = torch.empty((x.shape[0], net.out_dim), dtype=torch.float32, device=x.device) if out is None else out


class LayerBackward:
    """The backward pass of a single layer from the gradient dy (M, out) of its output, ready to launch: weight and bias gradient into its
    handle where the input x (M, in; a block of columns of wider rows, if need be) is given, gradient of the input into `dx` where that is."""

    def __init__(self, net: MLP, dy: torch.Tensor, x: torch.Tensor | None = None, dx: torch.Tensor | None = None):
        M = dy.shape[0]
        _lib.require_cuda(dy, dx, dtype=torch.float32)
        # of a contiguous input the strides say nothing where it has one row or one column
        ldx = 0 if x is None else net.in_dim if x.is_contiguous() else x.stride(0)
        if (tuple(dy.shape) != (M, net.out_dim) or (dx is not None and tuple(dx.shape) != (M, net.in_dim))
                or (x is not None and (tuple(x.shape) != (M, net.in_dim) or x.dtype != torch.float32 or not x.is_cuda
                                       or not (x.is_contiguous() or x.stride(1) == 1) or ldx < net.in_dim))):
            raise _lib.KsError("dy must be (M, out), dx and x (M, in) fp32 rows on the GPU, the columns of x side by side")
        self.net, self.dy, self.x, self.dx, self.ldx = net, dy, x, dx, ldx

    def record(self) -> "T.KsLayerBackward":
        return T.KsLayerBackward(self.net._handle.value, self.dy.shape[0], _lib.addr(self.x), self.ldx, _lib.addr(self.dy), _lib.addr(self.dx))


def run_layers(calls: Sequence[LayerForward]) -> None:
    """Launches single layers, two over as many rows each in one launch where the library can (`ks_mlp_forward_pair`)."""
    calls = list(calls)
    while calls:
        a = calls.pop(0)
        if calls and calls[0].x.shape[0] == a.x.shape[0]:
            b = calls.pop(0)
            a.net.forward_pair(a.x, a.out, b.net, b.x, b.out)
        else:
            a.net(a.x, out=a.out)


def run_layers_backward(calls: Sequence[LayerBackward]) -> None:
    """Launches the backward passes of single layers, together where the library can."""
    lib, table = _lib.load(), (T.KsLayerBackward * len(calls))(*(c.record() for c in calls))
    ws = torch.empty(int(lib.ks_mlps_layer_backward_workspace_bytes(len(calls), table)), dtype=torch.uint8, device=calls[0].dy.device)
    _lib.check(lib.ks_mlps_layer_backward(len(calls), table, _lib.current_stream(), _lib.addr(ws)))


def _listed(calls) -> list:
    return calls if isinstance(calls, list) else [calls]


def run_calls(calls) -> None:
    """Launches what the passes of several networks have ready, calls of a kind together."""
    for kind, run in ((LayerForward, run_layers), (SequenceCall, run_sequences), (LayerBackward, run_layers_backward)):
        some = [c for c in calls if isinstance(c, kind)]
        if some:
            run(some)


def lockstep(*passes):
    """Runs generators that yield calls (`SequenceCall`, `LayerForward`, lists of `LayerBackward`) side by side, launching what they yield
    together; returns their results."""
    results, live = [None] * len(passes), list(range(len(passes)))
    while live:
        calls = []
        for k in tuple(live):
            try:
                calls += _listed(next(passes[k]))
            except StopIteration as stop:
                results[k] = stop.value
                live.remove(k)
        run_calls(calls)
    return results


def _layer(net: MLP, x: torch.Tensor, out: torch.Tensor | None = None):
    """A network's forward pass inside a pass over a trajectory: single bf16 layers, which rows of a trajectory hardly fill the chip with, are left
    to `lockstep`, which puts those of two networks into one launch."""
    if len(net.dims) == 2 and net.dtype == "bf16":
        call = LayerForward(net, x, out)
        yield call
        return call.out
    return net(x, out=out)


class GRUCell:
    """h' = GRU(x, h) for N envs at once (`ks_gru_forward`)."""

    def __init__(self, weight_ih, weight_hh, bias=None, bias_n=None, dtype: str = "bf16"):
        lib = _lib.load()
        if dtype not in ("bf16", "f32"):
            raise _lib.KsError("dtype must be 'bf16' or 'f32'")
        wi, wh = _f32(weight_ih), _f32(weight_hh)
        H = wh.shape[1] if wh.ndim == 2 else -1
        if wi.ndim != 2 or wh.shape != (3 * H, H) or wi.shape[0] != 3 * H:
            raise _lib.KsError("weight_ih must be (3H, input) and weight_hh (3H, H)")
        b = None if bias is None else _f32(bias)
        bn = None if bias_n is None else _f32(bias_n)
        if (b is not None and b.shape != (3 * H,)) or (bn is not None and bn.shape != (H,)):
            raise _lib.KsError("bias must be (3H) and bias_n (H)")
        torch.zeros(1, device="cuda")
        d = T.KsGruDesc()
        d.input_size, d.hidden_size = wi.shape[1], H
        d.dtype = T.MLP_BF16 if dtype == "bf16" else T.MLP_F32
        d.weight_ih, d.weight_hh = wi.ctypes.data, wh.ctypes.data
        d.bias = None if b is None else b.ctypes.data
        d.bias_n = None if bn is None else bn.ctypes.data
        self.input_size, self.hidden_size, self.dtype = int(wi.shape[1]), int(H), dtype
        self._lib = lib
        self._handle = ctypes.c_void_p()
        _lib.check(lib.ks_gru_create(ctypes.byref(d), ctypes.byref(self._handle)))
        self._proj: MLP | None = None

    def workspace(self, M: int, device) -> torch.Tensor:
        """Scratch of one call, as `MLP.workspace`."""
        return torch.empty(int(self._lib.ks_gru_workspace_bytes(self._handle, M)), dtype=torch.uint8, device=device)

    def __call__(self, x: torch.Tensor, h: torch.Tensor, fresh: torch.Tensor | None = None,
                 out: torch.Tensor | None = None) -> torch.Tensor:
        _lib.require_cuda(x, dtype=torch.float32)
        _lib.require_cuda(h, dtype=torch.float32)
        M = x.shape[0]
        if tuple(x.shape) != (M, self.input_size) or tuple(h.shape) != (M, self.hidden_size):
            raise _lib.KsError(f"expected x (M, {self.input_size}) and h (M, {self.hidden_size})")
        if fresh is not None:
            _lib.require_cuda(fresh, dtype=torch.uint8)
            if tuple(fresh.shape) != (M,):
                raise _lib.KsError("fresh must be (M,) uint8")
        if out is None:
            out = torch.empty_like(h)
        else:
            _lib.require_cuda(out, dtype=torch.float32)
            if tuple(out.shape) != tuple(h.shape):
                raise _lib.KsError("output has the wrong shape")
        ws = self.workspace(M, x.device)
        _lib.check(self._lib.ks_gru_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(h),
                                            _lib.addr(fresh), _lib.addr(out), _lib.addr(ws)))
        return out

    # ------------------------------------------------------------------ training (ksim/task/ppo.py:572-694)
    def train_init(self) -> None:
        """fp32 master weights, gradients and Adam moments of both projections; afterwards `proj_i` / `proj_h` expose them."""
        _lib.check(self._lib.ks_gru_train_init(self._handle))
        pi, ph = ctypes.c_void_p(), ctypes.c_void_p()
        _lib.check(self._lib.ks_gru_projections(self._handle, ctypes.byref(pi), ctypes.byref(ph)))
        H = self.hidden_size
        self.proj_i = MLP._borrow(self._lib, pi, (self.input_size, 3 * H), self.dtype)
        self.proj_h = MLP._borrow(self._lib, ph, (H, 3 * H), self.dtype)
        self._bws: torch.Tensor | None = None

    def train_forward(self, x, h, fresh, out, saved) -> torch.Tensor:
        """`__call__` that also fills `saved` (M, 5H) = r | z | n | hn | h for `backward_step`."""
        _lib.require_cuda(x, h, out, saved, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        M, H = x.shape[0], self.hidden_size
        if tuple(x.shape) != (M, self.input_size) or tuple(h.shape) != (M, H) or tuple(out.shape) != (M, H) or tuple(saved.shape) != (M, 5 * H):
            raise _lib.KsError("expected x (M, input), h and out (M, H), saved (M, 5H)")
        ws = self.workspace(M, x.device)
        _lib.check(self._lib.ks_gru_train_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(h), _lib.addr(fresh),
                                                  _lib.addr(out), _lib.addr(saved), _lib.addr(ws)))
        return out

    @property
    def sequence_supported(self) -> bool:
        """Whether this cell has the one-launch-per-trajectory kernels (`ks_gru_sequence_forward / _backward`)."""
        return bool(self._lib.ks_gru_sequence_supported(self._handle))

    def _input_projection(self) -> MLP:
        """W_ih x + b of this cell as a network of one layer; there from the start, trained or not."""
        if self._proj is None:
            pi, ph = ctypes.c_void_p(), ctypes.c_void_p()
            _lib.check(self._lib.ks_gru_projections(self._handle, ctypes.byref(pi), ctypes.byref(ph)))
            self._proj = MLP._borrow(self._lib, pi, (self.input_size, 3 * self.hidden_size), self.dtype)
        return self._proj

    def sequence_call(self, x, h0, fresh, hs, saved, gi=None) -> "SequenceCall":
        """`sequence_forward` up to the recurrence itself, whose launch the caller makes (`run_sequences`); `gi`: the projected input (T M, 3H),
        where the caller has it."""
        _lib.require_cuda(x, h0, hs, saved, gi, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        Tn, M, H = x.shape[0], x.shape[1], self.hidden_size
        if (tuple(x.shape) != (Tn, M, self.input_size) or tuple(h0.shape) != (M, H) or tuple(hs.shape) != (Tn, M, H)
                or (saved is not None and tuple(saved.shape) != (Tn, M, 5 * H)) or tuple(fresh.shape) != (Tn, M)
                or (gi is not None and tuple(gi.shape) != (Tn * M, 3 * H))):
            raise _lib.KsError("expected x (T, M, input), h0 (M, H), hs (T, M, H), saved (T, M, 5H), fresh (T, M), gi (T M, 3H)")
        if gi is None:
            gi = self._input_projection()(x.reshape(Tn * M, self.input_size))
        return SequenceCall("ks_gru_sequences_forward", self.dtype, Tn, M, self._handle, gi, h0, None, fresh, saved, hs, None)

    def sequence_forward(self, x, h0, fresh, hs, saved) -> None:
        """The layer over a whole trajectory: x (T, M, input) -> hs (T, M, H) and `saved` (T, M, 5H; None where no backward
        pass follows), from the carry h0; the input projection is one product over all T M rows, the recurrence one launch."""
        run_sequences([self.sequence_call(x, h0, fresh, hs, saved)])

    def sequence_backward_call(self, dH, saved, fresh, d_gi, d_gh) -> "SequenceCall":
        """`sequence_backward`, checked; the caller makes the launch (`run_sequences`)."""
        _lib.require_cuda(dH, saved, d_gi, d_gh, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        Tn, M, H = dH.shape[0], dH.shape[1], self.hidden_size
        if (tuple(dH.shape) != (Tn, M, H) or tuple(saved.shape) != (Tn, M, 5 * H) or tuple(d_gi.shape) != (Tn, M, 3 * H)
                or tuple(d_gh.shape) != (Tn, M, 3 * H) or tuple(fresh.shape) != (Tn, M)):
            raise _lib.KsError("expected dH (T, M, H), saved (T, M, 5H), d_gi and d_gh (T, M, 3H), fresh (T, M)")
        return SequenceCall("ks_gru_sequences_backward", self.dtype, Tn, M, self._handle, dH, None, None, fresh, saved, d_gi, d_gh)

    def sequence_backward(self, dH, saved, fresh, d_gi, d_gh) -> None:
        """The reverse sweep over the trajectory: dH (T, M, H), the gradient reaching every h_t from above, -> d_gi, d_gh (T, M, 3H)."""
        run_sequences([self.sequence_backward_call(dH, saved, fresh, d_gi, d_gh)])

    def backward_step(self, dh_out, saved, fresh, d_gi, d_gh, dh_in) -> None:
        """One step of the backward pass through time: dh_out (M, H) -> d_gi, d_gh (M, 3H) and dh_in (M, H)."""
        _lib.require_cuda(dh_out, saved, d_gi, d_gh, dh_in, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        M, H = dh_out.shape[0], self.hidden_size
        if (tuple(dh_out.shape) != (M, H) or tuple(saved.shape) != (M, 5 * H) or tuple(d_gi.shape) != (M, 3 * H)
                or tuple(d_gh.shape) != (M, 3 * H) or tuple(dh_in.shape) != (M, H)):
            raise _lib.KsError("expected dh_out, dh_in (M, H), saved (M, 5H), d_gi, d_gh (M, 3H)")
        need = int(self._lib.ks_gru_backward_workspace_bytes(self._handle, M))
        if self._bws is None or self._bws.numel() < need or self._bws.device != dh_out.device:
            self._bws = torch.empty(need, dtype=torch.uint8, device=dh_out.device)
        _lib.check(self._lib.ks_gru_backward_step(self._handle, _lib.current_stream(), M, _lib.addr(dh_out), _lib.addr(saved),
                                                  _lib.addr(fresh), _lib.addr(d_gi), _lib.addr(d_gh), _lib.addr(dh_in), _lib.addr(self._bws)))

    def grad_sqnorm(self, acc: torch.Tensor) -> None:
        _lib.check(self._lib.ks_gru_grad_sqnorm(self._handle, _lib.current_stream(), _lib.addr(acc)))

    def adam_step(self, params, sqnorm) -> None:
        _lib.check(self._lib.ks_gru_adam_step(self._handle, _lib.current_stream(), ctypes.byref(params), _lib.addr(sqnorm)))

    def parameters(self, gradients: bool = False) -> dict:
        """Copies of weight_ih, weight_hh, bias (3H) and bias_n (H), or of their gradients."""
        H, empty, f32, dev = self.hidden_size, torch.empty, torch.float32, torch.device("cuda", torch._C._cuda_getDevice())
        wi, wh = empty((3 * H, self.input_size), dtype=f32, device=dev), empty((3 * H, H), dtype=f32, device=dev)
        bi, bn = empty((3 * H,), dtype=f32, device=dev), empty((H,), dtype=f32, device=dev)
        pair = ctypes.c_void_p * 2  # of the hidden projection's bias only the new gate's entries hold anything
        _lib.check(self._lib.ks_mlps_copy_params_from(pair(self.proj_i._handle, self.proj_h._handle), 2, _lib.current_stream(),
                                                      pair(wi.data_ptr(), wh.data_ptr()), pair(bi.data_ptr(), bn.data_ptr()),
                                                      (ctypes.c_int32 * 2)(0, 2 * H), int(gradients)))
        return dict(weight_ih=wi, weight_hh=wh, bias=bi, bias_n=bn)

    def __del__(self):
        h = getattr(self, "_handle", None)
        if h:
            self._lib.ks_gru_destroy(h)
            self._handle = None


class LSTMCell:
    """(h', c') = LSTM(x, (h, c)) for N envs at once (`ks_lstm_forward`); gate rows ordered input | forget | cell | output."""

    def __init__(self, weight_ih, weight_hh, bias=None, dtype: str = "bf16"):
        lib = _lib.load()
        if dtype not in ("bf16", "f32"):
            raise _lib.KsError("dtype must be 'bf16' or 'f32'")
        wi, wh = _f32(weight_ih), _f32(weight_hh)
        H = wh.shape[1] if wh.ndim == 2 else -1
        if wi.ndim != 2 or wh.shape != (4 * H, H) or wi.shape[0] != 4 * H:
            raise _lib.KsError("weight_ih must be (4H, input) and weight_hh (4H, H)")
        b = None if bias is None else _f32(bias)
        if b is not None and b.shape != (4 * H,):
            raise _lib.KsError("bias must be (4H)")
        torch.zeros(1, device="cuda")
        d = T.KsLstmDesc()
        d.input_size, d.hidden_size = wi.shape[1], H
        d.dtype = T.MLP_BF16 if dtype == "bf16" else T.MLP_F32
        d.weight_ih, d.weight_hh = wi.ctypes.data, wh.ctypes.data
        d.bias = None if b is None else b.ctypes.data
        self.input_size, self.hidden_size, self.dtype = int(wi.shape[1]), int(H), dtype
        self._lib = lib
        self._handle = ctypes.c_void_p()
        _lib.check(lib.ks_lstm_create(ctypes.byref(d), ctypes.byref(self._handle)))
        self._proj: MLP | None = None

    def workspace(self, M: int, device) -> torch.Tensor:
        """Scratch of one call, as `MLP.workspace`."""
        return torch.empty(int(self._lib.ks_lstm_workspace_bytes(self._handle, M)), dtype=torch.uint8, device=device)

    def __call__(self, x: torch.Tensor, h: torch.Tensor, c: torch.Tensor, fresh: torch.Tensor | None = None,
                 out: tuple | None = None) -> tuple[torch.Tensor, torch.Tensor]:
        for t in (x, h, c):
            _lib.require_cuda(t, dtype=torch.float32)
        M = x.shape[0]
        if tuple(x.shape) != (M, self.input_size) or tuple(h.shape) != (M, self.hidden_size) or tuple(c.shape) != tuple(h.shape):
            raise _lib.KsError(f"expected x (M, {self.input_size}) and h, c (M, {self.hidden_size})")
        if fresh is not None:
            _lib.require_cuda(fresh, dtype=torch.uint8)
            if tuple(fresh.shape) != (M,):
                raise _lib.KsError("fresh must be (M,) uint8")
        ho, co = (torch.empty_like(h), torch.empty_like(c)) if out is None else out
        for t in (ho, co):
            _lib.require_cuda(t, dtype=torch.float32)
            if tuple(t.shape) != tuple(h.shape):
                raise _lib.KsError("output has the wrong shape")
        ws = self.workspace(M, x.device)
        _lib.check(self._lib.ks_lstm_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(h), _lib.addr(c),
                                             _lib.addr(fresh), _lib.addr(ho), _lib.addr(co), _lib.addr(ws)))
        return ho, co

    # ------------------------------------------------------------------ training (ksim/task/ppo.py:572-694)
    def train_init(self) -> None:
        _lib.check(self._lib.ks_lstm_train_init(self._handle))
        pi, ph = ctypes.c_void_p(), ctypes.c_void_p()
        _lib.check(self._lib.ks_lstm_projections(self._handle, ctypes.byref(pi), ctypes.byref(ph)))
        H = self.hidden_size
        self.proj_i = MLP._borrow(self._lib, pi, (self.input_size, 4 * H), self.dtype)
        self.proj_h = MLP._borrow(self._lib, ph, (H, 4 * H), self.dtype)
        self._bws: torch.Tensor | None = None

    def train_forward(self, x, h, c, fresh, h_out, c_out, saved) -> None:
        """`__call__` that also fills `saved` (M, 7H) = i | f | g | o | tanh(c') | c | h for `backward_step`."""
        _lib.require_cuda(x, h, c, h_out, c_out, saved, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        M, H = x.shape[0], self.hidden_size
        if tuple(x.shape) != (M, self.input_size) or any(tuple(t.shape) != (M, H) for t in (h, c, h_out, c_out)) or tuple(saved.shape) != (M, 7 * H):
            raise _lib.KsError("expected x (M, input), h, c and outputs (M, H), saved (M, 7H)")
        ws = self.workspace(M, x.device)
        _lib.check(self._lib.ks_lstm_train_forward(self._handle, _lib.current_stream(), M, _lib.addr(x), _lib.addr(h), _lib.addr(c),
                                                   _lib.addr(fresh), _lib.addr(h_out), _lib.addr(c_out), _lib.addr(saved), _lib.addr(ws)))

    @property
    def sequence_supported(self) -> bool:
        """Whether this cell has the one-launch-per-trajectory kernels (`ks_lstm_sequence_forward / _backward`)."""
        return bool(self._lib.ks_lstm_sequence_supported(self._handle))

    def _input_projection(self) -> MLP:
        """W_ih x + b of this cell as a network of one layer; there from the start, trained or not."""
        if self._proj is None:
            pi, ph = ctypes.c_void_p(), ctypes.c_void_p()
            _lib.check(self._lib.ks_lstm_projections(self._handle, ctypes.byref(pi), ctypes.byref(ph)))
            self._proj = MLP._borrow(self._lib, pi, (self.input_size, 4 * self.hidden_size), self.dtype)
        return self._proj

    def sequence_call(self, x, h0, c0, fresh, hs, cs, saved, gi=None) -> "SequenceCall":
        """`sequence_forward` up to the recurrence itself, whose launch the caller makes (`run_sequences`); `gi`: the projected input (T M, 4H),
        where the caller has it."""
        _lib.require_cuda(x, h0, c0, hs, cs, saved, gi, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        Tn, M, H = x.shape[0], x.shape[1], self.hidden_size
        if (tuple(x.shape) != (Tn, M, self.input_size) or any(tuple(t.shape) != (M, H) for t in (h0, c0))
                or any(t is not None and tuple(t.shape) != (Tn, M, H) for t in (hs, cs))
                or (saved is not None and tuple(saved.shape) != (Tn, M, 7 * H)) or tuple(fresh.shape) != (Tn, M)
                or (gi is not None and tuple(gi.shape) != (Tn * M, 4 * H))):
            raise _lib.KsError("expected x (T, M, input), h0, c0 (M, H), hs, cs (T, M, H), saved (T, M, 7H), fresh (T, M), gi (T M, 4H)")
        if gi is None:
            gi = self._input_projection()(x.reshape(Tn * M, self.input_size))
        return SequenceCall("ks_lstm_sequences_forward", self.dtype, Tn, M, self._handle, gi, h0, c0, fresh, saved, hs, cs)

    def sequence_forward(self, x, h0, c0, fresh, hs, cs, saved) -> None:
        """The layer over a whole trajectory: x (T, M, input) -> hs, cs (T, M, H) and `saved` (T, M, 7H), from the carry
        (h0, c0); the input projection is one product over all T M rows, the recurrence one launch.  `cs` and `saved` may be
        None where no backward pass follows."""
        run_sequences([self.sequence_call(x, h0, c0, fresh, hs, cs, saved)])

    def sequence_backward_call(self, dH, saved, fresh, d_g) -> "SequenceCall":
        """`sequence_backward`, checked; the caller makes the launch (`run_sequences`)."""
        _lib.require_cuda(dH, saved, d_g, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        Tn, M, H = dH.shape[0], dH.shape[1], self.hidden_size
        if (tuple(dH.shape) != (Tn, M, H) or tuple(saved.shape) != (Tn, M, 7 * H) or tuple(d_g.shape) != (Tn, M, 4 * H)
                or tuple(fresh.shape) != (Tn, M)):
            raise _lib.KsError("expected dH (T, M, H), saved (T, M, 7H), d_g (T, M, 4H), fresh (T, M)")
        return SequenceCall("ks_lstm_sequences_backward", self.dtype, Tn, M, self._handle, dH, None, None, fresh, saved, d_g, None)

    def sequence_backward(self, dH, saved, fresh, d_g) -> None:
        """The reverse sweep over the trajectory: dH (T, M, H), the gradient reaching every h_t from above, -> d_g (T, M, 4H)."""
        run_sequences([self.sequence_backward_call(dH, saved, fresh, d_g)])

    def backward_step(self, dh_out, dc_out, saved, fresh, d_g, dh_in, dc_in) -> None:
        """One step of the backward pass through time: (dh_out, dc_out) -> d_g (M, 4H), dh_in, dc_in (M, H)."""
        _lib.require_cuda(dh_out, dc_out, saved, d_g, dh_in, dc_in, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        M, H = dh_out.shape[0], self.hidden_size
        if (any(tuple(t.shape) != (M, H) for t in (dh_out, dc_out, dh_in, dc_in)) or tuple(saved.shape) != (M, 7 * H)
                or tuple(d_g.shape) != (M, 4 * H)):
            raise _lib.KsError("expected gradients of the states (M, H), saved (M, 7H), d_g (M, 4H)")
        need = int(self._lib.ks_lstm_backward_workspace_bytes(self._handle, M))
        if self._bws is None or self._bws.numel() < need or self._bws.device != dh_out.device:
            self._bws = torch.empty(need, dtype=torch.uint8, device=dh_out.device)
        _lib.check(self._lib.ks_lstm_backward_step(self._handle, _lib.current_stream(), M, _lib.addr(dh_out), _lib.addr(dc_out),
                                                   _lib.addr(saved), _lib.addr(fresh), _lib.addr(d_g), _lib.addr(dh_in),
                                                   _lib.addr(dc_in), _lib.addr(self._bws)))

    def grad_sqnorm(self, acc: torch.Tensor) -> None:
        _lib.check(self._lib.ks_lstm_grad_sqnorm(self._handle, _lib.current_stream(), _lib.addr(acc)))

    def adam_step(self, params, sqnorm) -> None:
        _lib.check(self._lib.ks_lstm_adam_step(self._handle, _lib.current_stream(), ctypes.byref(params), _lib.addr(sqnorm)))

    def parameters(self, gradients: bool = False) -> dict:
        """Copies of weight_ih, weight_hh and bias (4H), or of their gradients."""
        ((wi, bi),), ((wh, _),) = mlp_mod.copy_parameters((self.proj_i, self.proj_h), gradients)
        return dict(weight_ih=wi, weight_hh=wh, bias=bi)

    def __del__(self):
        h = getattr(self, "_handle", None)
        if h:
            self._lib.ks_lstm_destroy(h)
            self._handle = None


class RecurrentNetwork:
    """input projection -> GRU or LSTM stack -> output MLP (examples/walking.py:124-150, 198-208;
    examples/kbot/train.py:903-915).  The carry is (depth, N, hidden) for GRU layers and (depth, 2, N, hidden), hidden
    state then cell state, for LSTM layers, like the arrays the reference stacks."""

    def __init__(self, input_proj: tuple, cells: Sequence[GRUCell], output_proj: MLP, dtype: str = "bf16"):
        w, b = input_proj
        self.input_proj = MLP([w], [b], activation="none", dtype=dtype)
        self.cells, self.output_proj = tuple(cells), output_proj
        H = self.input_proj.out_dim
        if any(c.input_size != H or c.hidden_size != H for c in self.cells) or output_proj.in_dim != H:
            raise _lib.KsError("the projection, the cells and the output network must share one hidden size")
        if len({type(c) for c in self.cells}) > 1:
            raise _lib.KsError("the recurrent layers must all be of one kind")
        self.lstm = bool(self.cells) and isinstance(self.cells[0], LSTMCell)
        self.hidden_size, self.depth = H, len(self.cells)
        self.in_dim, self.out_dim = self.input_proj.in_dim, output_proj.out_dim

    def initial_carry(self, num_envs: int, device="cuda") -> torch.Tensor:
        shape = (self.depth, 2, num_envs, self.hidden_size) if self.lstm else (self.depth, num_envs, self.hidden_size)
        return torch.zeros(*shape, dtype=torch.float32, device=device)

    def __call__(self, obs: torch.Tensor, carry: torch.Tensor, fresh: torch.Tensor | None = None,
                 out: torch.Tensor | None = None) -> torch.Tensor:
        """One control step for every env: `carry` is advanced in place."""
        N = obs.shape[0]
        want = (self.depth, 2, N, self.hidden_size) if self.lstm else (self.depth, N, self.hidden_size)
        if tuple(carry.shape) != want:
            raise _lib.KsError(f"carry must be {want}")
        x = self.input_proj(obs)
        for i, cell in enumerate(self.cells):  # the layer's new hidden state is also the next layer's input
            if self.lstm:
                x, _ = cell(x, carry[i, 0], carry[i, 1], fresh, out=(carry[i, 0], carry[i, 1]))
            else:
                x = cell(x, carry[i], fresh, out=carry[i])
        return self.output_proj(x, out=out)

    def forward_sequence(self, obs: torch.Tensor, carry0: torch.Tensor, fresh: torch.Tensor) -> torch.Tensor:
        """`forward_sequence_pass` by itself."""
        return lockstep(self.forward_sequence_pass(obs, carry0, fresh))[0]

    def forward_sequence_pass(self, obs: torch.Tensor, carry0: torch.Tensor, fresh: torch.Tensor):
        """The network over a trajectory without keeping anything for a backward pass: obs (T, M, in), carry0 the carry of the
        first step (left as it is), fresh (T, M) uint8 -> (T, M, out).  The same numbers as T calls, one control step each.  Long
        trajectories go through in stretches of `SEQUENCE_ROWS` rows, whole steps, each from the carry the last one left."""
        T_, M, H = obs.shape[0], obs.shape[1], self.hidden_size
        want = (self.depth, 2, M, H) if self.lstm else (self.depth, M, H)
        if tuple(obs.shape) != (T_, M, self.in_dim) or tuple(carry0.shape) != want or tuple(fresh.shape) != (T_, M):
            raise _lib.KsError(f"expected obs (T, M, in), carry0 {want}, fresh (T, M)")
        if not all(c.sequence_supported for c in self.cells):
            carry = carry0.clone()
            out = torch.empty(T_, M, self.out_dim, dtype=torch.float32, device=obs.device)
            for t in range(T_):
                self(obs[t], carry, fresh=fresh[t], out=out[t])
            return out
        out = torch.empty(T_, M, self.out_dim, dtype=torch.float32, device=obs.device)
        fresh = fresh.contiguous()
        steps = max(1, SEQUENCE_ROWS // max(M, 1))
        carry = [carry0[i].unbind(0) if self.lstm else (carry0[i],) for i in range(self.depth)]  # per layer (h, c) or (h,)
        for t0 in range(0, T_, steps):
            n = min(steps, T_ - t0)
            x = (yield from _layer(self.input_proj, obs[t0:t0 + n].contiguous().view(n * M, self.in_dim))).view(n, M, H)
            for i, cell in enumerate(self.cells):
                states = [torch.empty(n, M, H, dtype=torch.float32, device=obs.device)]
                if self.lstm:  # the cell state only where another stretch starts from it
                    states.append(torch.empty_like(states[0]) if t0 + n < T_ else None)
                # the projected rows, as large as four states, are gone before the next layer's come
                yield cell.sequence_call(x, *carry[i], fresh[t0:t0 + n], *states, None, (yield from _layer(cell._input_projection(), x.view(n * M, H))))
                x = states[0]
                if t0 + n < T_:
                    carry[i] = tuple(s[-1].clone() for s in states)
            yield from _layer(self.output_proj, x.view(n * M, H), out[t0:t0 + n].view(n * M, self.out_dim))
        return out

    # ------------------------------------------------------------------ training: backward pass through time
    def train_init(self) -> None:
        self.input_proj.train_init()
        for c in self.cells:
            c.train_init()
        self.output_proj.train_init()

    def train_forward(self, obs: torch.Tensor, carry0: torch.Tensor, fresh: torch.Tensor) -> torch.Tensor:
        """`train_forward_pass` by itself."""
        return lockstep(self.train_forward_pass(obs, carry0, fresh))[0]

    def train_forward_pass(self, obs: torch.Tensor, carry0: torch.Tensor, fresh: torch.Tensor):
        """The network over a trajectory, obs (T, M, in), starting from carry0 (the rollout's carry layout); envs flagged
        in fresh (T, M) uint8 start an episode at that step (their carry is zero there).  Returns (T, M, out) and keeps
        what `backward` needs.  This is the scan over time inside the loss of PPOTask._single_step
        (ksim/task/ppo.py:572-694)."""
        T_, M = obs.shape[0], obs.shape[1]
        H, dev = self.hidden_size, obs.device
        _lib.require_cuda(obs, carry0, dtype=torch.float32)
        _lib.require_cuda(fresh, dtype=torch.uint8)
        want = (self.depth, 2, M, H) if self.lstm else (self.depth, M, H)
        if tuple(obs.shape) != (T_, M, self.in_dim) or tuple(carry0.shape) != want or tuple(fresh.shape) != (T_, M):
            raise _lib.KsError(f"expected obs (T, M, in), carry0 {want}, fresh (T, M)")
        obs = obs.contiguous()
        x = (yield from _layer(self.input_proj, obs.view(T_ * M, self.in_dim))).view(T_, M, H)
        xs, saved = [], []
        for i, cell in enumerate(self.cells):
            hs = torch.empty(T_, M, H, dtype=torch.float32, device=dev)
            sv = torch.empty(T_, M, (7 if self.lstm else 5) * H, dtype=torch.float32, device=dev)
            if self.lstm and getattr(cell, "proj_i", None) is not None and cell.sequence_supported:
                yield cell.sequence_call(x, carry0[i, 0], carry0[i, 1], fresh, hs, None, sv, (yield from _layer(cell.proj_i, x.view(T_ * M, H))))
            elif self.lstm:
                cs = torch.empty(T_, M, H, dtype=torch.float32, device=dev)
                for t in range(T_):
                    h0, c0 = (carry0[i, 0], carry0[i, 1]) if t == 0 else (hs[t - 1], cs[t - 1])
                    cell.train_forward(x[t], h0, c0, fresh[t], hs[t], cs[t], sv[t])
            elif getattr(cell, "proj_i", None) is not None and cell.sequence_supported:
                yield cell.sequence_call(x, carry0[i], fresh, hs, sv, (yield from _layer(cell.proj_i, x.view(T_ * M, H))))
            else:
                for t in range(T_):
                    cell.train_forward(x[t], carry0[i] if t == 0 else hs[t - 1], fresh[t], hs[t], sv[t])
            xs.append(x)
            saved.append(sv)
            x = hs
        # a single layer keeps nothing for its backward pass; what the training forward refuses (no rows, no train_init) is left to it
        if len(self.output_proj.dims) == 2 and self.output_proj.dtype == "bf16" and T_ * M > 0 and getattr(self.output_proj, "_training", False):
            out = yield from _layer(self.output_proj, x.view(T_ * M, H))
        else:
            out = self.output_proj.train_forward(x.view(T_ * M, H))
        out = out.view(T_, M, self.out_dim)
        self._tape = dict(obs=obs, xs=xs, saved=saved, top=x, fresh=fresh.contiguous(), T=T_, M=M)
        return out

    def backward(self, d_out: torch.Tensor) -> None:
        """`backward_pass` by itself."""
        lockstep(self.backward_pass(d_out))

    def backward_pass(self, d_out: torch.Tensor):
        """Gradients of sum(d_out * output) with respect to every parameter, into the handles (the jax.grad through the
        scan).  Per layer, top to bottom: a sweep over the steps, last to first, that carries the gradient of the
        recurrent state, then one pass over all (step, env) rows for the weight gradients and the gradient of the layer's
        inputs."""
        tp = self._tape
        T_, M, H = tp["T"], tp["M"], self.hidden_size
        G = 4 if self.lstm else 3
        dev = d_out.device
        _lib.require_cuda(d_out, dtype=torch.float32)
        if tuple(d_out.shape) != (T_, M, self.out_dim):
            raise _lib.KsError("d_out must have the shape of the output")
        dH = torch.empty(T_, M, H, dtype=torch.float32, device=dev)
        # Few rows: the weight gradients of all layers wait for the last of them and share a launch.  Many rows fill the chip layer by layer, and
        # the gate gradients, which the weight gradients read, are as large as all that the forward pass keeps.
        later: list[LayerBackward] | None = [] if T_ * M <= LATER_ROWS else None

        def layer(net, x, dy, dx=None):  # calls of a layer's backward pass that are due now
            if later is None:
                return [LayerBackward(net, dy, x, dx)]
            later.append(LayerBackward(net, dy, x))
            return [] if dx is None else [LayerBackward(net, dy, None, dx)]

        top, d_top = tp["top"].view(T_ * M, H), d_out.contiguous().view(T_ * M, self.out_dim)
        if len(self.output_proj.dims) == 2:
            yield layer(self.output_proj, top, d_top, dH.view(T_ * M, H))
        else:
            self.output_proj.backward_dx(top, d_top, dH.view(T_ * M, H))
        for i in range(self.depth - 1, -1, -1):
            cell, sv = self.cells[i], tp["saved"][i]
            d_gi = torch.empty(T_, M, G * H, dtype=torch.float32, device=dev)
            d_gh = d_gi if self.lstm else torch.empty(T_, M, G * H, dtype=torch.float32, device=dev)
            fused = cell.sequence_supported
            if fused and self.lstm:
                yield cell.sequence_backward_call(dH, sv, tp["fresh"], d_gi)
            elif fused:
                yield cell.sequence_backward_call(dH, sv, tp["fresh"], d_gi, d_gh)
            else:
                carry = torch.zeros(2, M, H, dtype=torch.float32, device=dev)   # gradient of the hidden state, ping-pong
                ccarry = torch.zeros(2, M, H, dtype=torch.float32, device=dev)  # and of the cell state (LSTM)
            for t in range(T_ - 1, -1, -1) if not fused else ():
                dH[t] += carry[t & 1]
                if self.lstm:
                    cell.backward_step(dH[t], ccarry[t & 1], sv[t], tp["fresh"][t], d_gi[t], carry[(t + 1) & 1], ccarry[(t + 1) & 1])
                else:
                    cell.backward_step(dH[t], sv[t], tp["fresh"][t], d_gi[t], d_gh[t], carry[(t + 1) & 1])
            h_used = sv.view(T_ * M, sv.shape[2])[:, (6 if self.lstm else 4) * H:]
            dX = torch.empty(T_, M, H, dtype=torch.float32, device=dev)
            yield (layer(cell.proj_h, h_used, d_gh.view(T_ * M, G * H))
                   + layer(cell.proj_i, tp["xs"][i].reshape(T_ * M, H), d_gi.view(T_ * M, G * H), dX.view(T_ * M, H)))
            dH = dX
        yield (later or []) + [LayerBackward(self.input_proj, dH.view(T_ * M, H), tp["obs"].view(T_ * M, self.in_dim))]

    def networks(self) -> list[MLP]:
        """Every network whose parameters an optimiser step updates: the projections and both products of every cell."""
        if any(getattr(c, "proj_i", None) is None for c in self.cells):
            raise _lib.KsError("call train_init first")
        return [self.input_proj, *(p for c in self.cells for p in (c.proj_i, c.proj_h)), self.output_proj]

    def grad_sqnorm(self, acc: torch.Tensor) -> None:
        mlp_mod.grad_sqnorm(self.networks(), acc)

    def adam_step(self, params, sqnorm) -> None:
        mlp_mod.adam_step(self.networks(), params, sqnorm)
