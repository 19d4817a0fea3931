"""The persistent ESTMM kernel: lists that end inside a step of 32, empty lists and experts, more blocks than workgroups, blocks over the
result's edge, lists cut into parts, no plan.  Its sums are those of the one-block kernel in the same order: equal bit for bit."""
import pytest
import torch

from _util import TOL, assert_close, make_routing
from oracle import hexa_oracle as O

pytestmark = pytest.mark.gpu

# tokens, experts, slots, m, n, skew: one row; lists around 32; several rounds of workgroups without and with a plan; lists cut into
# parts beside empty ones; more experts than a workgroup sorts; one expert; three slots and two rounds
SIZES = [(1, 3, 1, 8, 8, None), (65, 2, 2, 136, 120, None), (700, 40, 1, 264, 1160, None), (9000, 33, 1, 392, 1500 // 8 * 8, "zipf"),
         (4000, 6, 2, 256, 640, "zipf"), (600, 300, 1, 128, 136, None), (2049, 1, 1, 128, 384, None), (6000, 7, 3, 520, 1544, "zipf")]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,k,m,n,skew", SIZES)
def test_estmm_flow(dev, T, E, k, m, n, skew, dtype):
    from hexa_moe import _lib, ops
    lib = _lib.load()
    print(f"estmm flow: T={T} E={E} k={k} {m} x {n} {skew} {dtype}", flush=True)
    routing = make_routing(T, E, k, seed=T, skew=skew, empty=2 if skew else 0)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    g = torch.Generator().manual_seed(m)
    a, b = torch.randn(k, T, m, generator=g).to(dtype), torch.randn(T, n, generator=g).to(dtype)
    for wide_first in (True, False):                         # the per-slot operand's dimension is the result's first or second
        dy, x, per = (a, b, (True, False)) if wide_first else (b, a, (False, True))
        dy, x = dy.to(dev), x.to(dev)
        for out in (dtype, torch.float32):
            got = {}
            for tile in (8, 15):                             # (15: an error where the persistent kernel does not run)
                _lib.check(lib.hexa_set_option(b"tile", tile), "hexa_set_option")
                try:
                    dw = ops.estmm(dy, x, route, *per, out_dtype=out)
                    got[tile] = dw, ops.estmm(dy, x, route, *per, out=dw.clone(), accumulate=True)
                    torch.cuda.synchronize()
                finally:
                    _lib.check(lib.hexa_set_option(b"tile", 0), "hexa_set_option")
            for want, have in zip(got[8], got[15]):
                assert torch.equal(have, want), (wide_first, out)
            if T * m * n < 2e9:
                want = O.estmm(dy.cpu().float(), x.cpu().float(), token_ids, offsets, wide_first, E)
                assert_close(got[15][0], want, TOL[dtype], f"{wide_first} {out}")


@pytest.mark.parametrize("wide_first", [True, False])
def test_many_blocks_in_one_dimension(dev, wide_first):
    """Block numbers of 32768 and more take the sign bit of the word that holds a block's row and column.  (The operands in fp32
    give the reference: 32 products a result, each exact in fp32, summed in some order.)"""
    from hexa_moe import ops
    T, few, many = 32, 8, 32768 * 128 + 8
    print(f"estmm flow: {many} {'rows' if wide_first else 'columns'} of the result", flush=True)
    route = ops.route_build(torch.zeros((T, 1), dtype=torch.int64, device=dev), 1)
    g = torch.Generator(device=dev).manual_seed(1)
    a, b = (torch.randn(T, n, generator=g, device=dev, dtype=torch.bfloat16) for n in (few, many))
    if wide_first:
        a, b = b, a
    got = ops.estmm(a[None], b, route, True, False)[0]
    want = torch.matmul(a.float().t().contiguous(), b.float())
    bound = 2 ** -24 * T * torch.matmul(a.float().abs().t().contiguous(), b.float().abs())
    assert ((got - want).abs() <= 2 * bound).all()
