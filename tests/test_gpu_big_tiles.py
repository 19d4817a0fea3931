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

    def only(fn, tile=14):
        _lib.check(lib.hexa_set_option(b"tile", tile), "hexa_set_option")
        try:
            out = fn()
            torch.cuda.synchronize()
            return out
        finally:
            _lib.check(lib.hexa_set_option(b"tile", 0), "hexa_set_option")
    return only


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
@pytest.mark.parametrize("T,E,k,d_in,d_out,skew", [(700, 2, 1, 320, 264, None), (2000, 5, 2, 256, 768, "zipf"), (300, 3, 1, 4096, 256, "one")])
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
             lambda: (ops.esmm(x, w, None, route, False, _lib.HEXA_W_OUT_IN, gelu_bwd_of=y1),)]
    for call in calls:
        for got, want in zip(big(call), big(call, tile=0)):
            nan = torch.isnan(want)
            assert torch.equal(torch.isnan(got), nan)
            assert torch.equal(bits(got)[~nan], bits(want)[~nan])
    y1 = y1.nan_to_num(1.0, 2.0, -2.0)
    dx, db = big(lambda: ops.esmm_gelu_bwd_ess(x, w, route, _lib.HEXA_W_OUT_IN, y1))
    offsets, ids = route.offsets.cpu(), route.token_ids.cpu()
    for e in range(E):
        rows = torch.cat([dx[s][ids[s, offsets[s, e]:offsets[s, e + 1]].long().to(dev)] for s in range(k)]).double()
        # fp32 sums of n terms in any order: at most n - 1 roundings of a partial sum of at most the terms' magnitudes
        bound = 2 ** -24 * len(rows) * rows.abs().sum(0) + 1e-30
        assert ((db[e].double() - rows.sum(0)).abs() <= bound).all(), e
