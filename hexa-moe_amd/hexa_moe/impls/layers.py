"""Autograd functions of the cascaded MoE (reference: hexa_moe_cuda/hexa_moe/impls/layers.py).

FusedMoE_Shared_CudaCore is the MoE FFN of one depth in data-centric mode on one GPU: the ten steps
of the paper's formula table, each an expert-specific operator of libhexa_moe_hip.so:

    forward   1  y1 = ESMM(x, W1, b1)            3  y = ESMM(act(y1), W2, b2), summed over the slots
    backward  4  db2 = ESS(dy)                    5  dW2 = ESTMM(act(y1), dy)     6  dy2 = ESMM(dy, W2^T)
              7  dy1 = dy2 * act'(y1)             8  db1 = ESS(dy1)               9  dW1 = ESTMM(dy1, x)
              10 dx = ESMM(dy1, W1^T), summed over the slots

The bodies are autograd nodes in C++ (csrc/torch_ops.cpp) over the C ABI's depth calls.  Against the reference
(layers.py:99-277, 280-474) on the same math:
  * weights are read in their parameter layout ([E,h,d_in], [E,h,d_out]); nothing is concatenated,
    permuted or copied per call (layers.py:119-122, 307-309, 412, 438 copy every expert weight);
  * results are written in their final type; no fp32 staging buffers, zero-fills or cast kernels
    (layers.py:230-231, 260, 275);
  * the routing lists are built once per depth on the device, without .item() (layers.py:238), and the
    same metadata serves all six matmuls, both ESS calls and the backward;
  * gradients are returned for the Parameters that were passed in (the reference passes `.data`, so
    its expert gradients are dropped: cascaded_moe.py:553-559);
  * the activation is evaluated once (fused, or as a part of the autograd graph between the two layers), not a second
    time in the backward (layers.py:281-283, 407), so stochastic activations (dropout) use one mask.
"""
from typing import Any

import torch
import torch.nn.functional as F

from .. import _native
from . import losses


def is_plain_gelu(fn) -> bool:
    """True for activations known to be the exact (erf) GELU, which the kernels fuse."""
    return fn is F.gelu or getattr(fn, "hexa_fused", None) == "gelu"


def fused_gelu(x):
    """Marker activation: pass `activation_fn=fused_gelu` to get the fused GELU epilogue."""
    return F.gelu(x)


fused_gelu.hexa_fused = "gelu"


class MLP_Implement:
    """Dense FFN depth (reference: layers.py:25-95): y = act(x fc1_w^T + b1) fc2_w + b2 with
    fc1_w [h, d_in], fc2_w [h, d_out].  Plain differentiable PyTorch (rocBLAS GEMMs); on one GPU the
    reference's gradient all-reduces are the identity."""

    @staticmethod
    def apply(config: Any, tokens_input, fc1_w, fc2_w, fc1_bias, fc2_bias):
        dt = tokens_input.dtype
        hid = F.linear(tokens_input, fc1_w.to(dt), fc1_bias.to(dt) if fc1_bias is not None else None)
        out = config.activation_fn(hid) @ fc2_w.to(dt)
        if fc2_bias is not None:
            out = out + fc2_bias.to(dt)
        return out


class RoutePool:
    """Routing-metadata buffers shared across the MoE depths: one int32 device buffer per depth, allocated on first
    use and reused by every later step.  A buffer that a pending backward will read is left alone and a new one takes
    its slot.  A copy of the pool starts empty."""

    def __init__(self):
        self._core = None

    @property
    def core(self):
        if self._core is None:
            self._core = _native.load().RoutePool()
        return self._core

    @property
    def _slots(self):
        return self.core.slots

    def clear(self):
        self.core.clear()

    def __getstate__(self):
        return {}

    def __setstate__(self, state):
        self._core = None


def _need_gpu(x):
    if not x.is_cuda:
        raise RuntimeError("hexa_moe: the MoE FFN runs on the GPU only (no CPU fallback); move the module "
                           "and its input to a HIP device")


class _OneOperation(torch.autograd.Function):
    """`call(*tensors)`, a tensor or a tuple of them, as one operation of a torch.jit trace.  The kernels write through raw
    pointers, so of a call's own tensor operations a trace would keep allocations that nothing fills."""

    @staticmethod
    def forward(ctx, call, *tensors):
        state = torch._C._get_tracing_state()
        torch._C._set_tracing_state(None)
        try:
            with torch.set_grad_enabled(any(ctx.needs_input_grad)):
                ctx.inputs = [t if t is None else t.detach().requires_grad_(need) for t, need in zip(tensors, ctx.needs_input_grad[1:])]
                ctx.outputs = call(*ctx.inputs)
            results = [o.detach() for o in ((ctx.outputs,) if torch.is_tensor(ctx.outputs) else ctx.outputs)]
        finally:
            torch._C._set_tracing_state(state)
        ctx.set_materialize_grads(False)
        results = [o.detach() for o in results]     # (the tracer expects to have seen what becomes the operation's result)
        return results[0] if torch.is_tensor(ctx.outputs) else tuple(results)

    @staticmethod
    def backward(ctx, *grads):
        outputs = (ctx.outputs,) if torch.is_tensor(ctx.outputs) else ctx.outputs
        inputs = [t for t in ctx.inputs if t is not None and t.requires_grad]
        outputs, grads = zip(*[(o, g) for o, g in zip(outputs, grads) if g is not None])
        found = iter(torch.autograd.grad(outputs, inputs, grads, allow_unused=True))
        return (None, *(next(found) if t is not None and t.requires_grad else None for t in ctx.inputs))


def _traceable(call, *tensors):
    return call(*tensors) if torch._C._get_tracing_state() is None else _OneOperation.apply(call, *tensors)


def _two_halves(native, config, stage, routing, x, wg, fc1_w, fc2_w, fc1_bias, fc2_bias, chosen, dtype=None):
    """A depth whose activation is the caller's: it is evaluated once, between the two halves, as an ordinary part of
    the autograd graph.  Returns (y, l_aux, idx)."""
    y1, l_aux, idx, handle = native.depth_in(config.route_pool.core, stage, x, wg, fc1_w, fc1_bias, chosen, fc2_w, routing, dtype)
    y2 = config.activation_fn(y1)
    if y2.dtype != y1.dtype:
        y2 = y2.to(y1.dtype)
    return native.depth_out(handle, y2, fc2_w, fc2_bias), l_aux, idx


class FusedMoE_Shared_CudaCore:
    """The MoE FFN of one depth for a routing decision that the caller made (config.routing_, a [T,k] tensor, or the
    reference's config.indices_, a list of k vectors)."""

    @staticmethod
    def apply(config: Any, tokens_input, fc1_w, fc2_w, fc1_bias, fc2_bias):
        x = tokens_input
        _need_gpu(x)
        indices = getattr(config, "routing_", None)
        if indices is None:
            indices = config.indices_
        chosen = indices if torch.is_tensor(indices) else torch.stack([i.reshape(-1) for i in indices], dim=1)
        native = _native.load()
        routing = native.Routing(chosen.shape[1], int(config.num_global_experts))
        stage = config.stage

        def call(x, chosen, fc1_w, fc2_w, fc1_bias, fc2_bias):
            if is_plain_gelu(config.activation_fn):
                return native.depth(config.route_pool.core, stage, x, None, fc1_w, fc2_w, fc1_bias, fc2_bias, chosen, routing, [], [], None)[0]
            return _two_halves(native, config, stage, routing, x, None, fc1_w, fc2_w, fc1_bias, fc2_bias, chosen)[0]

        return _traceable(call, x, chosen, fc1_w, fc2_w, fc1_bias, fc2_bias)


class FusedMoEDepth:
    """One MoE depth -- gate projection, softmax + top-k + auxiliary loss, the routing segment pass and the MoE FFN --
    as one library call per direction (two with an activation that the kernels do not fuse), the gate path's share of
    dx added inside the expert path's slot sum (reference: impls/cascaded_moe.py:508-568 and impls/layers.py:99-474)."""

    events = None   # optional {"fwd": [torch.cuda.Event, ...], "bwd": [...]} recorded around the major kernels

    @staticmethod
    def apply(config: Any, opts: Any, tokens_input, wg, fc1_w, fc2_w, fc1_bias, fc2_bias, dtype=None):
        """opts: (top_k, noise scale, whether the loss is GShard's, sigma).  dtype: the type the depth runs in where that is
        not the tokens'; y then comes in it or in the tokens'.  Returns (y, l_aux); the decision is left in config.routing_."""
        top_k, noise_scale, is_gshard, sigma = opts
        native = _native.load()
        routing = native.Routing(top_k, config.num_global_experts, noise_scale, sigma, is_gshard)
        stage = config.stage

        def call(tokens_input, wg, fc1_w, fc2_w, fc1_bias, fc2_bias):
            if is_plain_gelu(config.activation_fn):
                fwd = bwd = ()
                if FusedMoEDepth.events:
                    fwd, bwd = ([0 if e is None else e.cuda_event for e in FusedMoEDepth.events[d] or ()] for d in ("fwd", "bwd"))
                y, l_aux, idx = native.depth(config.route_pool.core, stage, tokens_input, wg, fc1_w, fc2_w, fc1_bias, fc2_bias, None,
                                             routing, fwd, bwd, dtype)
            else:
                y, l_aux, idx = _two_halves(native, config, stage, routing, tokens_input, wg, fc1_w, fc2_w, fc1_bias, fc2_bias, None, dtype)
            config.routing_ = idx
            return y, l_aux

        return _traceable(call, tokens_input, wg, fc1_w, fc2_w, fc1_bias, fc2_bias)


def topk_and_loss(scores, top_k, loss_fn=losses.gshard_loss):
    """Top-k expert choice as one [T,k] int64 tensor (what the routing pass reads directly) and the
    auxiliary loss."""
    top_k = min(int(top_k), int(scores.size(1)))
    topk_indices = torch.topk(scores, top_k, dim=1).indices
    l_loss = loss_fn(scores, topk_indices) if loss_fn is not None else None
    return topk_indices, l_loss


def simplified_extract_critical(scores, top_k, loss_fn=losses.gshard_loss):
    """Same contract as the reference's helper (layers.py:476-484): the k index vectors and the loss."""
    topk_indices, l_loss = topk_and_loss(scores, top_k, loss_fn)
    return [col.reshape(-1) for col in topk_indices.unbind(dim=1)], l_loss
