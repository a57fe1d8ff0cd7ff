"""Stacked LSTM on top of the single-layer core: layer l's outputs are layer l+1's inputs, and in the backward
pass layer l+1's input gradient is layer l's upstream gradient.  The reference is single-layer only
(flashlstm_v2/python/flashlstm/streaming_lstm.py:380-430); this is the thin layer loop a multi-layer workload
needs, with everything resident on the GPU in fp16 between layers."""
import ctypes
import math
from typing import List, Optional, Sequence, Tuple

import torch

from .core import F16, F32, LstmCore, _dtype_code, _ptr


def _pointers(tensors):
    """A C array of the device addresses of `tensors` (None: a null pointer)."""
    return (ctypes.c_void_p * len(tensors))(*[_ptr(t) for t in tensors])


def _layer_states(states, shape, name):
    """Per-layer states -- a (L,B,H) tensor, a sequence of (B,H) tensors or None -- as one contiguous (L,B,H) tensor.  Layers
    of a sequence may be None (zeros)."""
    if states is None:
        return None
    if not torch.is_tensor(states):
        states = list(states)
        if len(states) != shape[0]:
            raise ValueError(f"{name} must have one entry per layer")
        like = next((t for t in states if t is not None), None)
        if like is None:
            return None
        states = torch.stack([torch.zeros_like(like) if t is None else t for t in states])
    if not states.is_cuda or tuple(states.shape) != shape:
        raise ValueError(f"{name} must hold CUDA tensors of shape {shape[1:]}, one per layer")
    return states.contiguous()


class LstmStack:
    """num_layers LSTM layers of equal hidden size; layer 0 takes `input_size` features."""

    def __init__(self, batch: int, input_size: int, hidden_size: int, num_layers: int):
        if num_layers < 1:
            raise ValueError("num_layers must be >= 1")
        self.B, self.I, self.H, self.L = int(batch), int(input_size), int(hidden_size), int(num_layers)
        self.layers: List[LstmCore] = [LstmCore(self.B, self.I if l == 0 else self.H, self.H) for l in range(self.L)]
        self._lib = self.layers[0].lib
        self._inputs: List = []
        self.last_loss_scale = 1.0

    def close(self) -> None:
        for layer in self.layers:
            layer.close()
        self._inputs = []

    def _plans(self):
        """The layers' plans as a C array, read anew for every call: a layer that has been closed is a null pointer, which
        the library refuses."""
        return (ctypes.c_void_p * self.L)(*[layer._h for layer in self.layers])

    def pack(self, params: Sequence[Tuple]) -> None:
        """params[l] = (w_ih, w_hh, b_ih, b_hh) of layer l (fp32 CUDA tensors, torch.nn.LSTM layout)."""
        if len(params) != self.L:
            raise ValueError(f"expected parameters for {self.L} layers")
        for layer, (w_ih, w_hh, b_ih, b_hh) in zip(self.layers, params):
            layer.pack(w_ih, w_hh, b_ih, b_hh)

    def forward(self, x, h0: Optional[Sequence] = None, c0: Optional[Sequence] = None):
        """x (T,B,I) fp16 on the GPU -> (y of the top layer (T,B,H) fp16, [hy per layer], [cy per layer])."""
        y, hy, cy = self._forward(x, h0, c0)
        return y, list(hy.unbind(0)), list(cy.unbind(0))

    def _forward(self, x, h0, c0):
        """forward() with the final states as (L,B,H) tensors: one library call for the whole stack, one wait."""
        if x.dtype != torch.float16:
            raise ValueError("x must be fp16 (activations travel between layers in fp16)")
        if not x.is_cuda or x.dim() != 3 or x.shape[1] != self.B or x.shape[2] != self.I:
            raise ValueError(f"x must be a CUDA tensor of shape (T, {self.B}, {self.I})")
        x = x.contiguous()
        T, shape = x.shape[0], (self.L, self.B, self.H)
        h0, c0 = _layer_states(h0, shape, "h0"), _layer_states(c0, shape, "c0")
        if h0 is not None and c0 is not None and h0.dtype != c0.dtype:
            raise ValueError("h0 and c0 must share a dtype")
        state = h0 if h0 is not None else c0
        ys = [torch.empty((T, self.B, self.H), device=x.device, dtype=torch.float16) for _ in range(self.L)]
        hy = torch.empty(shape, device=x.device, dtype=torch.float16)
        cy = torch.empty_like(hy)
        rc = self._lib.flstm_stack_forward(self._plans(), self.L, T, x.data_ptr(), F16, _ptr(h0), _ptr(c0),
                                           F16 if state is None else _dtype_code(state), _pointers(ys), F16, hy.data_ptr(),
                                           cy.data_ptr(), LstmCore._stream())
        if rc != 0:
            raise RuntimeError(f"flstm_stack_forward failed with status {rc}")
        self._inputs = [x] + ys[:-1]
        return ys[-1], hy, cy

    def backward(self, dy_top, *, loss_scale="auto", d_hn: Optional[Sequence] = None,
                 d_cn: Optional[Sequence] = None, want_dx: bool = True, dy_factor: float = 1.0):
        """dy_top (T,B,H): gradient wrt the top layer's outputs, times 1 / dy_factor: the gradient is dy_factor * dy_top
        (a loss that averages over many elements has a gradient of the form tiny_constant * tensor_of_order_one; handing
        the two over apart keeps the tensor in fp16 range and saves the fp32 passes that would form their product).  loss_scale (a power of two) multiplies it before
        it is rounded to fp16 and stays on every inter-layer gradient, so that small gradients survive the fp16
        hand-over between layers; it is divided out of everything returned.  "auto" (the default) picks the power
        of two that brings the largest |dy_top| to about 64: far enough from the fp16 maximum (65504) for the
        gradients to grow a thousandfold on the way down, and far enough from the smallest normal fp16 number
        (6e-5) for them to shrink a few hundredfold per layer (the mean-squared-error gradient of a 4096 x 128 x
        2048 output is ~2e-9 per element: with a scale of 2^12 the bottom layer of a 4-layer stack loses all of
        its gradient).  The scale used is kept in self.last_loss_scale.
        Returns (dx of layer 0 (fp32 when a loss scale is in use) or None, [(dW_ih, dW_hh, db) per layer], [dh0 per layer], [dc0 per layer])."""
        return self._backward(dy_top, loss_scale, d_hn, d_cn, want_dx, dy_factor)[:4]

    def _backward(self, dy_top, loss_scale, d_hn, d_cn, want_dx, dy_factor=1.0, dx_dtype=None, both_biases=False):
        """backward(), one library call for the whole stack with one wait.  dx_dtype: of layer 0's dx (None: as backward()
        documents); both_biases: a fifth result, the bias gradients again in tensors of their own (for bias_hh)."""
        if not self._inputs:
            raise RuntimeError("backward needs a forward pass first")
        T, B, H, dev = self._inputs[0].shape[0], self.B, self.H, dy_top.device
        if tuple(dy_top.shape) != (T, B, H):
            raise ValueError(f"dy must have shape ({T}, {B}, {H})")
        dy_top = dy_top.contiguous()
        if dy_top.dtype not in (torch.float16, torch.float32):
            dy_top = dy_top.float()
        dy_code, stream = _dtype_code(dy_top), LstmCore._stream()
        if isinstance(loss_scale, str):
            if loss_scale != "auto":
                raise ValueError("loss_scale must be a positive number or 'auto'")
            amax = ctypes.c_float()
            rc = self._lib.flstm_core_absmax(self.layers[0]._h, dy_top.data_ptr(), dy_code, dy_top.numel(), ctypes.byref(amax), stream)
            if rc != 0:
                raise RuntimeError(f"flstm_core_absmax failed with status {rc}")
            amax = amax.value * abs(float(dy_factor))
            S = 2.0 ** min(60, max(-14, math.floor(math.log2(64.0 / amax)))) if 0.0 < amax < float("inf") else 1.0
        else:
            S = float(loss_scale) if loss_scale and loss_scale > 0 else 1.0
        self.last_loss_scale = S
        if dx_dtype is None:
            dx_dtype = torch.float16 if S == 1.0 else torch.float32   # fp32: the unscaled values may lie below the fp16 range
        ins = [self._inputs[l].shape[2] for l in range(self.L)]
        f32 = lambda *shape: torch.empty(shape, device=dev, dtype=torch.float32)
        dxs = [torch.empty((T, B, ins[l]), device=dev, dtype=torch.float16 if l > 0 else dx_dtype) if l > 0 or want_dx else None
               for l in range(self.L)]
        dW_ih, dW_hh = [f32(4 * H, ins[l]) for l in range(self.L)], [f32(4 * H, H) for _ in range(self.L)]
        db = [f32(4 * H) for _ in range(self.L)]
        db2 = [f32(4 * H) for _ in range(self.L)] if both_biases else None
        dh0, dc0 = f32(self.L, B, H), f32(self.L, B, H)
        states = []
        for grads, name in ((d_hn, "d_hn"), (d_cn, "d_cn")):
            grads = None if grads is None else [None if g is None else g.float().contiguous() for g in grads]
            if grads is not None and (len(grads) != self.L or any(g is not None and tuple(g.shape) != (B, H) for g in grads)):
                raise ValueError(f"{name} must hold one tensor of shape ({B}, {H}) (or None) per layer")
            states.append(grads)
        for layer in self.layers:   # (a layer used on its own with accumulate_into has left it on, which a stack's pass refuses)
            layer.set_option("accumulate_grads", 0)
        rc = self._lib.flstm_stack_backward(
            self._plans(), self.L, T, _pointers(self._inputs), F16, dy_top.data_ptr(), dy_code, S * float(dy_factor),
            None if states[0] is None else _pointers(states[0]), None if states[1] is None else _pointers(states[1]), F32, S,
            _pointers(dxs), F16 if dxs[0] is None else _dtype_code(dxs[0]), _pointers(dW_ih), _pointers(dW_hh), _pointers(db),
            None if db2 is None else _pointers(db2), _pointers(list(dh0.unbind(0))), _pointers(list(dc0.unbind(0))), stream)
        if rc != 0:
            raise RuntimeError(f"flstm_stack_backward failed with status {rc}")
        return dxs[0], list(zip(dW_ih, dW_hh, db)), list(dh0.unbind(0)), list(dc0.unbind(0)), db2, dh0, dc0

    def backward_mse(self, y_top, target, **kwargs):
        """backward() for the loss mean((y_top - target)^2) over all elements: its gradient 2 / N * (y_top - target) is
        handed over as the fp16 difference and the factor 2 / N (see dy_factor).  y_top: what forward() returned."""
        if y_top.dtype != torch.float16 or target.dtype != torch.float16:
            return self.backward((y_top.float() - target.float()), dy_factor=2.0 / y_top.numel(), **kwargs)
        return self.backward(torch.sub(y_top, target), dy_factor=2.0 / y_top.numel(), **kwargs)


class _StackFunction(torch.autograd.Function):
    """Autograd node around LstmStack: inputs (x, h0 (L,B,H) or None, c0 or None, 4 * L parameters)."""

    @staticmethod
    def forward(ctx, module, x, h0, c0, y_dtype, loss_scale, *params):
        L = module.num_layers
        stack = module._stack_for(x.shape[1])
        with torch.no_grad():
            stream = LstmCore._stream()
            for l, layer in enumerate(stack.layers):
                layer._pack_enqueue(*params[4 * l:4 * l + 4], stream)
            y, hy, cy = stack._forward(x, None if h0 is None else h0.half(), None if c0 is None else c0.half())
            if y_dtype != y.dtype:
                y = y.to(y_dtype)
        module._generation += 1
        ctx.module, ctx.stack, ctx.generation, ctx.loss_scale = module, stack, module._generation, loss_scale
        ctx.has_state = (h0 is not None, c0 is not None)
        ctx.x_dtype = x.dtype
        ctx.set_materialize_grads(False)   # (a gradient nobody has stays None instead of becoming a tensor of zeros)
        return y, hy, cy

    @staticmethod
    def backward(ctx, dy, dhn, dcn):
        if ctx.generation != ctx.module._generation:
            raise RuntimeError("StackedLSTM keeps the caches of its most recent forward pass only: call backward "
                               "before the next forward pass of the same module")
        stack = ctx.stack
        if dy is None:
            x = stack._inputs[0]
            dy = torch.zeros((x.shape[0], stack.B, stack.H), device=x.device, dtype=torch.float16)
        dx, grads, _, _, db_hh, dh0, dc0 = stack._backward(dy, ctx.loss_scale, dhn, dcn, ctx.needs_input_grad[1],
                                                           dx_dtype=ctx.x_dtype, both_biases=True)
        flat = []
        for (dW_ih, dW_hh, db), db2 in zip(grads, db_hh):
            flat += [dW_ih, dW_hh, db, db2]
        gh0 = dh0.half() if ctx.has_state[0] and ctx.needs_input_grad[2] else None
        gc0 = dc0.half() if ctx.has_state[1] and ctx.needs_input_grad[3] else None
        return (None, dx, gh0, gc0, None, None, *flat)


class StackedLSTM(torch.nn.Module):
    """Multi-layer LSTM as an nn.Module with autograd, on the device-resident core: the training surface for a
    stacked workload.  The reference's module is single-layer and host-streaming
    (flashlstm_v2/python/flashlstm/streaming_lstm.py:380-430, mirrored by flashlstm.StreamingLSTM); this one keeps
    every sequence on the GPU.  Parameters carry torch.nn.LSTM's names (weight_ih_l0, weight_hh_l0, bias_ih_l0,
    bias_hh_l0, ...), layout and initialisation (U(-1/sqrt(H), 1/sqrt(H)), fp32, on the GPU), so a state_dict moves
    between the two.

    forward(x, (h0, c0)=None) -> (y, (h_n, c_n)):  x (T,B,I) fp16 CUDA; h0 / c0 (L,B,H) fp16 or None (zeros);
    y (T,B,H) in `output_dtype` (fp16, or fp32 for losses whose gradient per element lies below the fp16 range: the
    gradient arrives in y's dtype); h_n, c_n (L,B,H) fp16.  Differentiable in x, h0, c0 and all parameters.  Inside,
    gradients pass from layer to layer in fp16 under a power-of-two loss scale (`loss_scale`, default "auto").
    The module keeps the caches of its MOST RECENT forward pass only; backward must run before the next forward."""

    def __init__(self, input_size: int, hidden_size: int, num_layers: int = 1, *, output_dtype=torch.float16,
                 loss_scale="auto", device="cuda"):
        super().__init__()
        if num_layers < 1:
            raise ValueError("num_layers must be >= 1")
        self.input_size, self.hidden_size, self.num_layers = int(input_size), int(hidden_size), int(num_layers)
        self.output_dtype, self.loss_scale = output_dtype, loss_scale
        H = self.hidden_size
        for l in range(self.num_layers):
            I = self.input_size if l == 0 else H
            for name, shape in ((f"weight_ih_l{l}", (4 * H, I)), (f"weight_hh_l{l}", (4 * H, H)),
                                (f"bias_ih_l{l}", (4 * H,)), (f"bias_hh_l{l}", (4 * H,))):
                self.register_parameter(name, torch.nn.Parameter(torch.empty(shape, device=device, dtype=torch.float32)))
        self.reset_parameters()
        self._stacks = {}       # batch size -> LstmStack
        self._generation = 0

    def reset_parameters(self) -> None:
        k = 1.0 / self.hidden_size ** 0.5
        for p in self.parameters():     # same order as torch.nn.LSTM.reset_parameters
            torch.nn.init.uniform_(p, -k, k)

    def _stack_for(self, batch: int) -> LstmStack:
        st = self._stacks.get(batch)
        if st is None:
            for old in self._stacks.values():   # one batch size at a time: the caches are large
                old.close()
            self._stacks = {}
            st = self._stacks[batch] = LstmStack(batch, self.input_size, self.hidden_size, self.num_layers)
        return st

    def forward(self, x, state=None):
        if not x.is_cuda or x.dtype != torch.float16 or x.dim() != 3 or x.shape[2] != self.input_size:
            raise ValueError(f"x must be a CUDA float16 tensor of shape (T, B, {self.input_size})")
        h0 = c0 = None
        if state is not None:
            h0, c0 = state
            for name, t in (("h0", h0), ("c0", c0)):
                if t is not None and (not t.is_cuda or tuple(t.shape) != (self.num_layers, x.shape[1], self.hidden_size)):
                    raise ValueError(f"{name} must be a CUDA tensor of shape ({self.num_layers}, {x.shape[1]}, {self.hidden_size})")
        params = [getattr(self, f"{n}_l{l}") for l in range(self.num_layers) for n in ("weight_ih", "weight_hh", "bias_ih", "bias_hh")]
        y, h_n, c_n = _StackFunction.apply(self, x.contiguous(), h0, c0, self.output_dtype, self.loss_scale, *params)
        return y, (h_n, c_n)

    def release(self) -> None:
        """Frees the device caches (plans are rebuilt on the next forward pass)."""
        for st in self._stacks.values():
            st.close()
        self._stacks = {}
