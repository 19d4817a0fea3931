"""Ids outside [0, E) in a routing decision add nothing to a sum over slots, whatever the memory of the scratch held."""
import pytest
import torch

from _util import gen, uniform

pytestmark = pytest.mark.gpu

BOUND = {torch.float32: 1e-6, torch.bfloat16: 4e-3, torch.float16: 5e-4}   # 16 bits: each slot's product and the sum are rounded


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _poison(dev, *sizes):
    """Leaves NaN in what the allocator hands out next for tensors of these sizes (bytes)."""
    held = [torch.full((n // 4,), float("nan"), device=dev) for n in sizes for _ in range(3)]
    del held


def _decision(T, E, k, seed, first=True):
    """[T, k] with about a sixth of the ids no expert's, among them all of the first and the last token's."""
    g = gen(seed)
    ids = torch.randint(0, E, (T, k), generator=g)
    off = torch.rand(T, k, generator=g) < 1 / 6
    off[0] = off[T - 1] = True
    if not first:
        off[:, 0] = False
    return torch.where(off, torch.where(torch.rand(T, k, generator=g) < 0.5, -1, E + 2), ids), off


def _expected(x, W, bias, ids, off, start):
    """fp64: the slots' products summed over the (token, slot) pairs that have an expert."""
    out = start.double().clone()
    for s in range(ids.shape[1]):
        for e in range(W.shape[0]):
            rows = ((ids[:, s] == e) & ~off[:, s]).nonzero()[:, 0]
            out[rows] += x[s, rows].double() @ W[e].double() + bias[e].double()
    return out


@pytest.mark.parametrize("dtype", list(BOUND))
@pytest.mark.parametrize("accumulate", [True, False])
@pytest.mark.parametrize("T,k,E,d_in,d_out", [
    (130, 2, 3, 64, 8),            # rows shorter than a wavefront's piece
    (257, 3, 5, 32, 136),
    (4100, 2, 8, 128, 512),        # several row tiles per expert, rows as wide as a wavefront's piece
    (2049, 4, 4, 64, 1032),        # wider than it
    (300, 3, 4, 40, 72)])          # 16 bits: a contraction of 40 adds slot by slot
def test_sum_over_slots_takes_the_listed_rows(dev, dtype, accumulate, T, k, E, d_in, d_out):
    from hexa_moe import _lib, ops
    # (slot by slot and without earlier contents, the sum starts from the first slot's row, which has to be there)
    by_slot = dtype != torch.float32 and d_in % 32 != 0
    ids, off = _decision(T, E, k, 7 * T + k, first=accumulate or not by_slot)
    g = gen(T)
    x, W = torch.randn(k, T, d_in, generator=g).to(dtype), uniform((E, d_in, d_out), d_in ** -0.5, g).to(dtype)
    bias = uniform((E, d_out), 0.5, g).to(dtype)
    start = torch.randn(T, d_out, generator=g).to(dtype) if accumulate else torch.zeros(T, d_out, dtype=dtype)
    route = ops.route_build(ids.to(dev), E)
    xd, Wd, bd = x.to(dev), W.to(dev), bias.to(dev)
    out = start.to(dev) if accumulate else None
    size = T * d_out * x.element_size()
    _poison(dev, size, (k - 1) * size)
    y = ops.esmm(xd, Wd, bd, route, True, _lib.HEXA_W_IN_OUT, out=out, accumulate=accumulate)
    want = _expected(x, W, bias, ids, off, start)
    got = y.double().cpu()
    assert torch.isfinite(got).all()
    assert float((got - want).norm() / want.norm()) < BOUND[dtype]
    none = off.all(1)
    assert torch.equal(y.cpu()[none], start[none])
