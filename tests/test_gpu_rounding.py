"""Where a result is rounded to 16 bits: contractions that are no multiple of 32, and fp32 master weights used for fewer than
32 rows an expert, keep the fp32 product up to the activation and up to the sum it joins, and take erf from the library."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _sweep(dtype):
    """Every value of the type between -5.6 and -2, where GELU is what is left of 1 + erf: an error of erf shows in it whole."""
    v = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dtype).double()
    return v[(v > -5.6) & (v < -2.0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_takes_erf(dev, dtype):
    """y1 = v exactly (one non-zero product).  Bounds: rounding of the result, and of erf near -1 in fp32 -- 2 units of 2^-24
    for erff, one for 1 + erf, times |v| / 2 for GELU and 1 / 2 for GELU', whose second term has a few roundings of its own.
    (With the polynomial erf of the kernels for aligned sizes, 6e-7, GELU of a sixth of the bf16 values lies outside.)"""
    from hexa_moe import _lib, ops
    v = _sweep(dtype)
    T, d_in, d_out = v.numel(), 8, 8
    x = torch.zeros(T, d_in, dtype=dtype)
    x[:, 0] = v.to(dtype)
    w = torch.zeros(1, d_out, d_in, dtype=dtype)
    w[0, :, 0] = 1.0
    route = ops.route_build(torch.zeros(T, 1, dtype=torch.int64, device=dev), 1)
    y1, y2 = ops.esmm(x.to(dev), w.to(dev), None, route, False, _lib.HEXA_W_OUT_IN, gelu=True)
    assert torch.equal(y1[0, :, 0].double().cpu(), v)
    unit = 2.0 ** -24
    rounding, tiny = (1.01 * 2.0 ** -8, 2.0 ** -134) if dtype == torch.bfloat16 else (1.01 * 2.0 ** -11, 2.0 ** -25)
    tail = 0.5 * torch.erfc(-v / math.sqrt(2.0))                       # Phi(v)
    want = v * tail
    bound = rounding * want.abs() + tiny + 0.5 * v.abs() * 3 * unit
    assert ((y2[0].double().cpu() - want[:, None]).abs() <= bound[:, None]).all()
    dy = torch.zeros(T, d_in, dtype=dtype)
    dy[:, 0] = 1.0
    dy1 = ops.esmm(dy.to(dev), w.to(dev), None, route, False, _lib.HEXA_W_OUT_IN, gelu_bwd_of=y1)
    second = v * torch.exp(-0.5 * v * v) / math.sqrt(2.0 * math.pi)
    want = tail + second
    bound = rounding * want.abs() + tiny + 0.5 * 3 * unit + 32 * unit * second.abs()
    assert ((dy1[0].double().cpu() - want[:, None]).abs() <= bound[:, None]).all()


class _Layer:
    """A layer without biases, its input and dy, and what it gives with every product in 64 bits and rounded where the general
    kernels round: y1, GELU of the fp32 y1 (an activation of the caller's, and contractions that are multiples of 32 without masters: of
    the rounded one), dy1 likewise, and each slot's sum."""

    def __init__(self, dev, dtype, T, d, h, E, k, masters, act):
        from hexa_moe import moe as hmoe
        self.dtype, self.dev, self.k = dtype, dev, k
        self.fused = act == "gelu" and (masters or d % 32 != 0)     # GELU of the fp32 product
        g = torch.Generator().manual_seed(T + d + h + k)
        m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                              mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, mlp_fc1_bias=False, mlp_fc2_bias=False,
                              activation_fn=torch.nn.functional.gelu if act == "gelu" else lambda t: torch.nn.functional.gelu(t))
        for n, p in m.named_parameters():
            p.data = (torch.rand(p.shape, generator=g) * 2 - 1) * 0.3
            if not n.startswith("gates") and not masters:
                p.data = p.data.to(dtype)
        self.m = m.to(dev)
        self.x, self.dy = (torch.randn(T, d, generator=g).to(dtype) for _ in range(2))

    def run(self, dy, aux):
        x = self.x.to(self.dev).requires_grad_(True)
        with torch.autocast("cuda", dtype=self.dtype):
            y, l_aux = self.m(0, x)
        assert y.dtype == self.dtype
        torch.autograd.backward([y, l_aux], [dy.to(self.dev), torch.full_like(l_aux, aux)])
        return y.detach().cpu(), x.grad.cpu()

    def want(self, gate_dx, slot_by_slot):
        """(y, dx), the slots' products and the gate's share of dx (gate_dx) added before they are rounded; with slot_by_slot
        rounded as each joins."""
        rounded = lambda t: t.to(self.dtype).double()      # noqa: E731
        route = self.m.dispatch_params.routing_.long().cpu()
        w1, w2 = (rounded(p[0].detach().cpu()) for p in (self.m.batched_fc1_w, self.m.batched_fc2_w))
        phi = lambda v: 0.5 * torch.erfc(-v / math.sqrt(2.0))     # noqa: E731
        y = dx = None
        if gate_dx is not None:
            dx = gate_dx.double()
        for s in range(self.k):
            e = route[:, s]
            p1 = torch.bmm(w1[e], self.x.double()[:, :, None])[:, :, 0]
            y1 = rounded(p1)
            y2 = rounded(p1 * phi(p1) if self.fused else y1 * phi(y1))
            q = torch.bmm(self.dy.double()[:, None], w2[e].transpose(1, 2).contiguous())[:, 0]
            grad = phi(y1) + y1 * torch.exp(-0.5 * y1 * y1) / math.sqrt(2.0 * math.pi)
            dy1 = rounded((q if self.fused else rounded(q)) * grad)
            p2, r = torch.bmm(y2[:, None], w2[e])[:, 0], torch.bmm(dy1[:, None], w1[e])[:, 0]
            y, dx = p2 if y is None else y + p2, r if dx is None else dx + r
            if slot_by_slot:
                y, dx = rounded(y), rounded(dx)
        return y.to(self.dtype), dx.to(self.dtype)


def _check(layer, fused, gate, slot_by_slot=False):
    """As good as every value is the one expected.  fp32 sums differ from 64 bits by some 2^-22, which moves a value over a
    rounding boundary of bf16 once in thousands, and one element of y1 or dy1 that was moved so moves a few of its row's: below
    1 % in all.  One more rounding on the way changes a fifth of the values and more."""
    from hexa_moe import _lib
    lib = _lib.load()
    _lib.check(lib.hexa_set_option(b"backward_fused", fused), "hexa_set_option")
    try:
        gate_dx = layer.run(torch.zeros_like(layer.dy), 50.0)[1] if gate else None
        y, dx = layer.run(layer.dy, 50.0 if gate else 0.0)
    finally:
        _lib.check(lib.hexa_set_option(b"backward_fused", 0), "hexa_set_option")
    for name, got, want in zip(("y", "dx"), (y, dx), layer.want(gate_dx, slot_by_slot)):
        differ = (got != want).double().mean().item()
        assert differ < 0.03, (name, differ)


@pytest.mark.parametrize("fused", [0, 2])     # shared launches, one launch per product
@pytest.mark.parametrize("d,h", [(64, 128), (72, 264)])
def test_masters_used_for_few_rows(dev, fused, d, h):
    layer = _Layer(dev, torch.bfloat16, 60, d, h, 8, 1, True, "gelu")
    _check(layer, fused, False)


@pytest.mark.parametrize("fused", [0, 2])
@pytest.mark.parametrize("masters,d,h,act", [(False, 72, 264, "gelu"), (False, 64, 136, "gelu"), (False, 64, 264, "own"), (True, 64, 128, "gelu")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_share_of_one_slot(dev, dtype, masters, d, h, act, fused):
    """dx = the gate's share as it is stored + the fp32 product, rounded once (hidden sizes that are no multiple of 32, and
    masters used for few rows)."""
    _check(_Layer(dev, dtype, 60, d, h, 8, 1, masters, act), fused, True)


def test_accumulated_product_of_a_ragged_contraction(dev):
    """out += x . w where the contraction is no multiple of 32: the fp32 product joins what is there (328 is long enough for the
    pipelined kernel, which would round it first)."""
    from hexa_moe import _lib, ops
    T, d_in, d_out, E = 500, 328, 136, 4
    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(1, T, d_in, generator=g).to(torch.bfloat16), (torch.randn(E, d_in, d_out, generator=g) / d_in ** 0.5).to(torch.bfloat16)
    old = torch.randn(T, d_out, generator=g).to(torch.bfloat16)
    routing = torch.randint(0, E, (T, 1), generator=g)
    out = ops.esmm(x.to(dev), w.to(dev), None, ops.route_build(routing.to(dev), E), True, _lib.HEXA_W_IN_OUT, out=old.clone().to(dev), accumulate=True)
    product = torch.bmm(x[0].double()[:, None], w.double()[routing[:, 0]])[:, 0]
    differ = (out.cpu() != (old.double() + product).to(torch.bfloat16)).double().mean().item()
    assert differ < 0.01, differ


@pytest.mark.parametrize("fused", [0, 2])
@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("masters,d,h,k,act", [(True, 64, 128, 2, "gelu"), (True, 64, 128, 2, "own"), (True, 520, 264, 3, "gelu"),
                                               (True, 72, 136, 2, "own"), (False, 72, 136, 2, "gelu"), (False, 64, 264, 3, "own")])
def test_slots(dev, masters, d, h, k, act, gate, fused):
    """Masters used for few rows: the slots' fp32 products are added and rounded once.  Hidden sizes that are no multiple of 32:
    each joins the rounded sum of those before it."""
    _check(_Layer(dev, torch.bfloat16, 60, d, h, 12, k, masters, act), fused, gate, slot_by_slot=not masters)


@pytest.mark.parametrize("bad", [-1, 6])
def test_slots_without_an_expert(dev, bad):
    """Ids of no expert: the (token, slot) adds nothing, and a token without any slot gets zeros."""
    from types import SimpleNamespace

    from hexa_moe.impls import layers
    T, d, h, E, k = 70, 64, 96, 6, 2
    g = torch.Generator().manual_seed(5)
    x = torch.randn(T, d, generator=g).to(torch.bfloat16).to(dev).requires_grad_(True)
    w1, w2 = ((torch.randn(E, h, d, generator=g) / 8).to(dev).requires_grad_(True) for _ in range(2))
    dy = torch.randn(T, d, generator=g).to(torch.bfloat16).to(dev)
    routing = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    routing[::3, 0] = bad
    routing[::4, 1] = bad
    config = SimpleNamespace(num_global_experts=E, routing_=routing.to(dev), activation_fn=torch.nn.functional.gelu, stage=0,
                             route_pool=layers.RoutePool())
    y = layers.FusedMoE_Shared_CudaCore.apply(config, x, w1, w2, None, None)
    y.backward(dy)
    xr = x.detach().double().cpu().requires_grad_(True)
    r1, r2 = (w.detach().to(torch.bfloat16).double().cpu() for w in (w1, w2))
    want = torch.zeros(T, d, dtype=torch.float64)
    for s in range(k):
        for e in range(E):
            rows = (routing[:, s] == e).nonzero()[:, 0]
            want = want.index_add(0, rows, torch.nn.functional.gelu(xr[rows] @ r1[e].t()) @ r2[e])
    want.backward(dy.double().cpu())
    for got, ref in ((y, want), (x.grad, xr.grad)):
        got, ref = got.detach().double().cpu(), ref.detach()
        assert (got - ref).norm() <= 6.8e-3 * ref.norm()      # roundings as in test_gpu_backward_fused.py
        none = (routing == bad).all(1)
        assert none.any() and (got[none] == 0).all()
