"""Partial results that a second pass adds: the gate's dwg, one for every four chunks of 64 tokens, and the parts of large fp32 weight
gradients, four values a thread; the fp32 bias gradient by column sums of the tiles of dy1."""
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


# 128 x 128 tiles (the rule asks for 180 of them and 100 tokens an expert): columns that end inside a tile and inside a wavefront's 32, lists
# of no, few and many rows, two slots; one size on the 64 x 64 tiles, whose bias gradient is a pass of its own
@pytest.mark.parametrize("T,E,k,d_in,d_out,skew", [(3000, 4, 1, 64, 1028, None), (2100, 7, 2, 36, 788, "zipf"), (5000, 3, 1, 132, 640, "one"),
                                                      (3000, 4, 1, 64, 512, None)])
def test_fp32_bias_gradient_beside_dy1(dev, T, E, k, d_in, d_out, skew):
    from hexa_moe import _lib, ops
    print(f"fp32 column sums: T={T} E={E} k={k} {d_in} -> {d_out} {skew}", flush=True)
    routing = make_routing(T, E, k, seed=T, skew=skew, empty=2 if skew == "zipf" else 0)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    g = gen(d_in)
    x, W, y1 = torch.randn(T, d_in, generator=g), torch.randn(E, d_out, d_in, generator=g) / d_in ** 0.5, torch.randn(k, T, d_out, generator=g)
    t = y1.double()
    want = O.esmm(x.double(), W.transpose(1, 2).double(), None, token_ids, offsets, False) * \
        (0.5 * (1 + torch.erf(t / 2 ** 0.5)) + t * torch.exp(-0.5 * t * t) / (2 * torch.pi) ** 0.5)
    got, db = ops.esmm_gelu_bwd_ess(x.to(dev), W.to(dev), route, _lib.HEXA_W_OUT_IN, y1.to(dev))
    torch.cuda.synchronize()
    assert_close(got, want, TOL[torch.float32], "dy1")
    sums = O.ess(got.double().cpu(), token_ids, offsets, True, E)
    assert_close(db, sums, TOL[torch.float32], "db")
    assert torch.equal(db.cpu()[sums.abs().sum(1) == 0], sums[sums.abs().sum(1) == 0].float())       # no rows: zeros
    assert torch.equal(db, ops.esmm_gelu_bwd_ess(x.to(dev), W.to(dev), route, _lib.HEXA_W_OUT_IN, y1.to(dev))[1])


# Lists of 160 and more tiles, values with a mean: what a chain of partial sums would lose.  Both orders of additions modelled on the CPU give
# 0.7 (20000 rows a list) and 0.7 (65536) of the pass's error; groups of tiles in a chain 1.3 and 2.4.
@pytest.mark.parametrize("T,E,k", [(65536, 1, 1), (20000, 2, 2)])
def test_fp32_bias_gradient_of_long_lists(dev, T, E, k):
    """No less exact than a pass over the stored rows."""
    from hexa_moe import _lib, ops
    print(f"fp32 column sums: T={T} E={E} k={k}", flush=True)
    routing = make_routing(T, E, k, seed=1, skew="one")
    route = ops.route_build(routing.to(dev), E)
    g = gen(T)
    x, W = torch.randn(T, 32, generator=g).to(dev), (torch.randn(E, 512, 32, generator=g) / 32 ** 0.5).to(dev)
    x[:, 0], W[:, :, 0] = 1.0, 0.1
    dy1, db = ops.esmm_gelu_bwd_ess(x, W, route, _lib.HEXA_W_OUT_IN, torch.full((k, T, 512), 10.0, device=dev))     # GELU'(10) = 1
    by_pass = ops.ess(dy1, route, True)
    torch.cuda.synchronize()
    want = torch.zeros(E, 512, dtype=torch.float64, device=dev)
    for s in range(k):
        want.index_add_(0, routing[:, s].to(dev), dy1[s].double())
    err = lambda v: ((v.double() - want).norm() / want.norm()).item()      # noqa: E731
    assert err(db) <= 1.1 * err(by_pass), (err(db), err(by_pass))
