"""The fp32 kernels' split into bf16 terms: as exact as fp32 sums on both tile sizes, and values that cannot be split (infinities,
NaN, magnitudes whose terms overflow or fall below the smallest normal bf16) multiplied as they are."""
import math

import pytest
import torch

from _util import make_linear, make_routing
from oracle import hexa_oracle as O

pytestmark = pytest.mark.gpu

# tokens, experts, slots, in, out: 128 x 128 tiles in ESMM / in ESTMM / cut lists, 64 x 64 tiles, ragged everything
SIZES = [(3100, 8, 2, 132, 1100), (600, 8, 1, 1028, 1032), (2500, 2, 1, 1284, 1284), (777, 4, 2, 100, 196), (37, 3, 1, 4, 260)]


def change(kind, x):
    if kind in ("inf", "nan", "3.4e38"):
        x.view(-1)[x.numel() // 3] = float(kind)
        x.view(-1)[-1] = -float(kind)
    elif kind == "zeros":
        x.zero_()
    elif kind != "normal":
        x.mul_(float(kind))
    return x


@pytest.mark.parametrize("kind", ["normal", "1e-30", "1e-36", "1e25", "3.4e38", "inf", "nan", "zeros"])
@pytest.mark.parametrize("T,E,k,d_in,d_out", SIZES)
def test_split(dev, T, E, k, d_in, d_out, kind):
    from hexa_moe import _lib, ops
    print(f"fp32 split: T={T} E={E} k={k} {d_in} -> {d_out} {kind}", flush=True)
    routing = make_routing(T, E, k, seed=T)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    x, W, b = make_linear(T, d_in, d_out, E, k, seed=d_out, dtype=torch.float32, m2s=False)
    x = change(kind, x)
    b.zero_()
    dy = torch.randn((k, T, d_out), generator=torch.Generator().manual_seed(1))

    def compare(got, want, terms, what):
        got, fits = got.cpu().double(), want.abs() <= 3.4e38
        assert torch.equal(torch.isnan(got), torch.isnan(want)), what
        inf = torch.isinf(want)
        assert torch.equal(got[inf], want[inf]), what
        # a sum of n products is rounded 6 n / 16 times (twice per product on the fp32 pipe) while it grows: random roundings of
        # 2^-24 / sqrt(3) and a partial sum of sqrt(1/2) the last one give sqrt(n) / 4 (sqrt(n / 3)) of 2^-24; where one value
        # makes the result, of the order of one rounding
        err, ref = (got - want)[fits].norm().item(), want[fits].norm().item()
        least = 2 ** -149 * math.sqrt(want.numel() * terms)      # (roundings of denormal sums)
        assert err <= (1 + math.sqrt(terms)) * 2 ** -24 * ref + least, (what, err / max(ref, 1e-300))

    want = O.esmm(x.double(), W.double(), b.double(), token_ids, offsets, False)
    for layout, w in ((_lib.HEXA_W_IN_OUT, W), (_lib.HEXA_W_OUT_IN, W.transpose(1, 2).contiguous())):
        compare(ops.esmm(x.to(dev), w.to(dev), b.to(dev), route, False, layout), want, d_in, f"esmm layout {layout}")
    want = O.estmm(dy.double(), x.double(), token_ids, offsets, True, E)
    compare(ops.estmm(dy.to(dev), x.to(dev), route, True, False), want, T * k / E, "estmm")


@pytest.mark.parametrize("scale", [1e-31, 1e-33, 1e-35, 1e-36, 1e-37, 1e-40])
@pytest.mark.parametrize("T,E,k,d_in,d_out", SIZES)
def test_small_beside_ordinary(dev, T, E, k, d_in, d_out, scale):
    """Single columns and single contraction indices of small values among ordinary ones, each result column (and row) by itself:
    as exact as if all of the operand were as small."""
    from hexa_moe import _lib, ops
    print(f"fp32 split: T={T} E={E} k={k} {d_in} -> {d_out} {scale} beside 1", flush=True)
    routing = make_routing(T, E, k, seed=T)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    x, W, b = make_linear(T, d_in, d_out, E, k, seed=d_out, dtype=torch.float32, m2s=False)
    b.zero_()
    few = sorted({0, d_in // 2 + 1, d_in - 1})              # contraction indices (columns of dw) and result columns (rows of dw)
    x[:, few] *= scale
    W[:, :, 1] *= scale
    W[:, [i for i in range(d_in) if i not in few], 0] = 0     # (one result column of the small tokens' values alone)
    W[:, :, -2] *= scale

    def compare(got, want, terms, dims, what):
        """Norms over dims: see test_split for the bound."""
        err, ref = ((got.cpu().double() - want).norm(dim=dims), want.norm(dim=dims))
        least = 2 ** -149 * math.sqrt(want.numel() / ref.numel() * terms)
        worst = (err / ((1 + math.sqrt(terms)) * 2 ** -24 * ref + least)).max().item()
        assert worst <= 1, (what, worst)

    want = O.esmm(x.double(), W.double(), b.double(), token_ids, offsets, False)
    for layout, w in ((_lib.HEXA_W_IN_OUT, W), (_lib.HEXA_W_OUT_IN, W.transpose(1, 2).contiguous())):
        compare(ops.esmm(x.to(dev), w.to(dev), b.to(dev), route, False, layout), want, d_in, (0, 1), f"esmm layout {layout}")
    dy = torch.randn((k, T, d_out), generator=torch.Generator().manual_seed(1))
    dy[..., 1] *= scale
    dy[..., -2] *= scale
    want = O.estmm(dy.double(), x.double(), token_ids, offsets, True, E)
    got = ops.estmm(dy.to(dev), x.to(dev), route, True, False).cpu()
    rows, cols = [o for o in range(d_out) if o not in (1, d_out - 2)], [i for i in range(d_in) if i not in few]
    compare(got[:, rows], want[:, rows], T * k / E, (0, 1), "estmm columns")
    if cols:
        compare(got[..., cols], want[..., cols], T * k / E, (0, 2), "estmm rows")


@pytest.mark.parametrize("T,E,k,d_in,d_out", SIZES)
def test_small_products(dev, T, E, k, d_in, d_out):
    """Ordinary terms whose products reach below the smallest normal number (2^-126): sums of about 2^-120 keep their bits."""
    from hexa_moe import _lib, ops
    print(f"fp32 split: T={T} E={E} k={k} {d_in} -> {d_out} products of 1e-36", flush=True)
    routing = make_routing(T, E, k, seed=T)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    x, W, b = make_linear(T, d_in, d_out, E, k, seed=d_out, dtype=torch.float32, m2s=False)
    dy = torch.randn((k, T, d_out), generator=torch.Generator().manual_seed(1))
    for t in (x, W, dy):
        t *= 1e-18
    b.zero_()
    for got, want, terms in ((ops.esmm(x.to(dev), W.to(dev), b.to(dev), route, False, _lib.HEXA_W_IN_OUT),
                              O.esmm(x.double(), W.double(), b.double(), token_ids, offsets, False), d_in),
                             (ops.estmm(dy.to(dev), x.to(dev), route, True, False), O.estmm(dy.double(), x.double(), token_ids, offsets, True, E), T * k / E)):
        # (every addition of a term's 16 products rounds to 2^-149 at the least: 6 n / 16 of them)
        err, ref = (got.cpu().double() - want).norm().item(), want.norm().item()
        assert err <= (1 + math.sqrt(terms)) * (2 ** -24 * ref + 2 ** -149 * math.sqrt(want.numel())), err / ref
