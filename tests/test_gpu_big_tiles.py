"""The ESMM kernel with 256x256 tiles (an expert's lists of all slots in one row sequence): ends of tiles, of stages of 64 contraction
indices and of runs of four row tiles, empty experts, one expert with every row, and the values outside the tables of GELU and GELU'."""
import math

import pytest
import torch

from _util import TOL, assert_close, make_linear, make_routing
from oracle import hexa_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16]
# tokens, experts, slots, in, out, skew: one row; one tile and one more row or column; five row tiles of one expert; several tiles
# per workgroup; contraction ends inside a stage; a single partial stage behind three
SIZES = [(1, 3, 1, 256, 256, None), (257, 2, 1, 256, 264, "one"), (513, 7, 2, 320, 520, "zipf"), (1281, 1, 1, 264, 248, None),
         (5000, 5, 3, 200, 2056, None), (9000, 4, 1, 1024, 2048, "zipf")]


@pytest.fixture
def big(dev):
    from hexa_moe import _lib
    lib = _lib.load()

    def only(fn, tile=15, pipe=0):                      # (15: an error where the 256x256 kernel does not run)
        _lib.check(lib.hexa_set_option(b"tile", tile), "hexa_set_option")
        _lib.check(lib.hexa_set_option(b"pipe", pipe), "hexa_set_option")
        try:
            out = fn()
            torch.cuda.synchronize()
            return out
        finally:
            _lib.check(lib.hexa_set_option(b"tile", 0), "hexa_set_option")
            _lib.check(lib.hexa_set_option(b"pipe", 0), "hexa_set_option")
    return only


def test_sizes_it_does_not_cover_are_refused(dev, big):
    """What the other tests here stand on: a forced kernel that does not run is an error."""
    from hexa_moe import _lib, ops
    route = ops.route_build(make_routing(64, 2, 1, seed=0).to(dev), 2)
    x, W, _ = make_linear(64, 128, 256, 2, 1, seed=0, dtype=torch.bfloat16, m2s=False)     # (two stages of contraction indices)
    with pytest.raises(RuntimeError, match="256x256"):
        big(lambda: ops.esmm(x.to(dev), W.to(dev), None, route, False, _lib.HEXA_W_IN_OUT))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,E,k,d_in,d_out,skew", SIZES)
def test_products(dev, big, T, E, k, d_in, d_out, skew, dtype):
    from hexa_moe import _lib, ops
    print(f"big tiles: T={T} E={E} k={k} {d_in} -> {d_out} {skew} {dtype}", flush=True)
    routing = make_routing(T, E, min(k, E), seed=T, skew=skew, empty=2 if skew == "zipf" else 0)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    for m2s in (False, True):
        x, W, b = make_linear(T, d_in, d_out, E, k, seed=d_out, dtype=dtype, m2s=m2s)
        want = O.esmm(x.float(), W.float(), b.float(), token_ids, offsets, m2s)
        for layout, w in ((_lib.HEXA_W_IN_OUT, W), (_lib.HEXA_W_OUT_IN, W.transpose(1, 2).contiguous())):
            for bias in (b, b.float()):
                got = big(lambda: ops.esmm(x.to(dev), w.to(dev), bias.to(dev), route, m2s, layout))
                assert_close(got, want, TOL[dtype], f"esmm m2s={m2s} layout={layout} bias {bias.dtype}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,E,k,d_in,d_out,skew", [(700, 2, 1, 320, 264, None), (2000, 5, 2, 256, 768, "zipf"), (300, 3, 1, 4096, 256, "one"),
                                                      (9000, 4, 2, 224, 2312, "zipf")])
def test_activations(dev, big, T, E, k, d_in, d_out, skew, dtype):
    """Bit for bit the values of the 128x128 kernels, which take the same sums in the same order: also for arguments outside the
    activation's table (zeros, tiny and large values, infinities, NaN), alone in a lane's piece or in all of it."""
    from hexa_moe import _lib, ops
    print(f"big activations: T={T} E={E} k={k} {d_in} -> {d_out} {skew} {dtype}", flush=True)
    routing = make_routing(T, E, k, seed=T, skew=skew)
    route = ops.route_build(routing.to(dev), E)
    x, W, _ = make_linear(T, d_in, d_out, E, k, seed=d_out, dtype=dtype, m2s=False)
    x[::7] *= 100
    x[5::11] = 0
    x[3::50] *= 1e-6
    y1 = torch.randn((k, T, d_out), generator=torch.Generator().manual_seed(1)).to(dtype)
    y1[:, ::5] *= 1e-4
    y1[:, 2::9] = 0
    y1[0, 3, :5], y1[0, 4, 64:72], y1[0, 6, 7], y1[:, 7::13] = math.inf, math.nan, -math.inf, y1[:, 7::13] * 50
    x, w, y1 = x.to(dev), W.transpose(1, 2).contiguous().to(dev), y1.to(dev)
    bits = lambda t: t.view(torch.int16)                     # noqa: E731
    calls = [lambda: ops.esmm(x, w, None, route, False, _lib.HEXA_W_OUT_IN, gelu=True),
             lambda: (ops.esmm(x, w, None, route, False, _lib.HEXA_W_OUT_IN, gelu_bwd_of=y1),),
             lambda: (ops.esmm_gelu_bwd_ess(x, w, route, _lib.HEXA_W_OUT_IN, y1)[0],)]        # the instances with column sums
    for call in calls:
        for got, want in zip(big(call), big(call, tile=0)):
            nan = torch.isnan(want)
            assert torch.equal(torch.isnan(got), nan)
            assert torch.equal(bits(got)[~nan], bits(want)[~nan])
    y1 = y1.nan_to_num(1.0, 2.0, -2.0)
    dx, db = big(lambda: ops.esmm_gelu_bwd_ess(x, w, route, _lib.HEXA_W_OUT_IN, y1))
    assert torch.equal(bits(dx), bits(big(lambda: ops.esmm_gelu_bwd_ess(x, w, route, _lib.HEXA_W_OUT_IN, y1), tile=0)[0]))
    offsets, ids = route.offsets.cpu(), route.token_ids.cpu()
    for e in range(E):
        rows = torch.cat([dx[s][ids[s, offsets[s, e]:offsets[s, e + 1]].long().to(dev)] for s in range(k)]).double()
        # fp32 sums of n terms in any order: at most n - 1 roundings of a partial sum of at most the terms' magnitudes
        bound = 2 ** -24 * len(rows) * rows.abs().sum(0) + 1e-30
        assert ((db[e].double() - rows.sum(0)).abs() <= bound).all(), e


@pytest.mark.parametrize("dtype", DTYPES)
def test_rule_and_the_layer_around_it(dev, big, dtype):
    """A layer whose four ESMM calls the rule sends to the 256x256 kernel by itself (GELU, sum over slots, GELU' with column sums that
    are folded later, slot sum with the gate's share), against the pipelined kernel: the same sums in the same order but for the
    column sums."""
    import torch.nn.functional as F
    from hexa_moe import moe as hmoe, ops, _lib
    T, d, h, E, k = 14000, 2048, 4096, 4, 2
    print(f"big tiles by rule: T={T} E={E} k={k} {d} -> {h} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    with torch.device(dev):
        m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                              mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, mlp_fc1_bias=True, mlp_fc2_bias=True,
                              activation_fn=F.gelu)
    for n, p in m.named_parameters():
        p.data = (torch.rand(p.shape, generator=g, device=dev) * 2 - 1) * (0.05 if "gates" in n else 0.02)
        p.data = p.data if "gates" in n else p.data.to(dtype)
    x, dy = torch.randn(T, d, generator=g, device=dev).to(dtype), torch.randn(T, d, generator=g, device=dev).to(dtype)

    def step():
        m.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        y, l_aux = m(0, xi)
        torch.autograd.backward([y, l_aux], [dy, torch.full((), 3.0, device=dev)])
        return {"y": y.detach(), "dx": xi.grad, **{n: p.grad for n, p in m.named_parameters()}}

    rule, pipe = big(step, tile=0), big(step, tile=0, pipe=1)
    for n in rule:
        a, b = rule[n].double(), pipe[n].double()
        if n.startswith("batched_fc1_bias"):
            # fp32 sums of some 7000 terms in two orders, rounded once each
            assert (a - b).norm() <= (1e-5 + 2.0 ** (-7 if dtype == torch.bfloat16 else -10)) * b.norm(), n
        else:
            assert torch.equal(rule[n], pipe[n]), n
    # which kernel the rule took shows in the order of the column sums, which the kernels group differently
    idx = torch.topk(torch.randn(T, E, generator=g, device=dev), k, 1).indices
    route = ops.route_build(idx, E)
    w = m.batched_fc2_w[0].detach()
    w = w if tuple(w.shape) == (E, h, d) else w.transpose(1, 2).contiguous()
    y1 = torch.randn(k, T, h, generator=g, device=dev).to(dtype)
    db = [big(lambda: ops.esmm_gelu_bwd_ess(dy, w, route, _lib.HEXA_W_OUT_IN, y1)[1], **o) for o in ({"tile": 0}, {}, {"tile": 0, "pipe": 1})]
    assert torch.equal(db[0], db[1]) and not torch.equal(db[0], db[2])
