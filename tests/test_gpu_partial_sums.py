"""Partial results that a second pass adds: the gate's dwg, one for every four chunks of 64 tokens, and the parts of large fp32 weight
gradients, four values a thread."""
import pytest
import torch

from _util import TOL, assert_close, gen, make_routing
from oracle import hexa_oracle as O

pytestmark = pytest.mark.gpu


# tokens: a chunk and four of them, one less and one more; dims and experts: ends of 128 columns and 32 experts
@pytest.mark.parametrize("T", [1, 63, 65, 192, 255, 256, 257, 512, 1030])
@pytest.mark.parametrize("d,E", [(8, 1), (136, 33), (120, 65), (256, 32)])
def test_gate_dwg(dev, T, d, E):
    from hexa_moe import ops
    g = gen(T + d)
    x, wg, dl = torch.randn(T, d, generator=g).bfloat16(), torch.randn(E, d, generator=g), torch.randn(T, E, generator=g)
    print(f"gate dwg: T={T} d={d} E={E}", flush=True)
    dx, dwg = ops.gate_backward(dl.to(dev), x.to(dev), wg.to(dev))
    torch.cuda.synchronize()
    # fp32 sums of up to 1030 products of order 1: 2^-24 times the root of their number at most, against the largest value
    assert_close(dwg, dl.double().t() @ x.double(), 2e-6, "gate dwg")
    assert_close(dx, dl.double() @ wg.double(), 2 ** -8, "gate dx")
    for need_dx in (True, False):
        assert torch.equal(ops.gate_backward(dl.to(dev), x.to(dev), wg.to(dev), need_dx=need_dx)[1], dwg)


# results just below and above the size from which four values a thread are added; two and eight parts
@pytest.mark.parametrize("T,E,k,d_in,d_out", [(2200, 2, 1, 508, 512), (2200, 2, 1, 512, 516), (6000, 3, 1, 1028, 256), (5000, 4, 2, 512, 260)])
def test_fp32_weight_gradient_parts(dev, T, E, k, d_in, d_out):
    from hexa_moe import ops
    print(f"fp32 parts: T={T} E={E} k={k} {d_in} -> {d_out}, {ops.estmm32_slots(T, k, E, d_out, d_in)} slots", flush=True)
    assert ops.estmm32_slots(T, k, E, d_out, d_in) > 0
    routing = make_routing(T, E, k, seed=T)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    g = gen(d_out)
    x, dy = torch.randn(T, d_in, generator=g), torch.randn(k, T, d_out, generator=g)
    want = O.estmm(dy.double(), x.double(), token_ids, offsets, True, E)
    got = ops.estmm(dy.to(dev), x.to(dev), route, True, False)
    torch.cuda.synchronize()
    assert_close(got, want, TOL[torch.float32], "estmm")
    assert_close(ops.estmm(dy.to(dev), x.to(dev), route, True, False, out=torch.ones_like(got), accumulate=True), want + 1, TOL[torch.float32], "estmm +=")
