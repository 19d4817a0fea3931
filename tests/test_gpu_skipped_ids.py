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


@pytest.mark.parametrize("dtype", list(BOUND))
@pytest.mark.parametrize("T,k,E", [(1, 2, 2), (70, 1, 3), (130, 2, 3), (1500, 3, 70)])
def test_the_reference_operators_take_lists_with_unassigned_ends(dev, dtype, T, k, E):
    """TOKEN_COUNT and TOKEN_ASSIGN into lists of num_tokens entries, then the matmul operators on them."""
    import hexa_moe_cuda as ext
    d_in, d_out, full = 32, 64, dtype == torch.float32
    ids, off = _decision(T, E, k, T + E)
    if T > 1:
        off[1], ids[1] = False, 0
    g = gen(T + 1)
    x, W = torch.randn(k, T, d_in, generator=g).to(dtype), uniform((E, d_in, d_out), d_in ** -0.5, g).to(dtype)
    bias, start = uniform((E, d_out), 0.5, g).to(dtype), torch.randn(T, d_out, generator=g).to(dtype)
    tok = torch.full((k * T,), -1, dtype=torch.int32, device=dev)
    exp = torch.full((k * T,), -1, dtype=torch.int32, device=dev)
    cum = torch.arange(0, (k + 1) * T, T, dtype=torch.int32, device=dev)
    for s in range(k):
        r = ids[:, s].to(torch.int32).contiguous().to(dev)
        count, offsets = torch.zeros(E, dtype=torch.int32, device=dev), torch.zeros(E + 1, dtype=torch.int32, device=dev)
        ext.TOKEN_COUNT(count, offsets, r, T, E)
        ext.TOKEN_ASSIGN(tok[s * T:(s + 1) * T], exp[s * T:(s + 1) * T], offsets, r, T, E)
    y = start.to(dev)
    _poison(dev, (k - 1) * T * d_out * x.element_size() or 4)
    ext.ESMM_TENSOR_CORE(y, x.to(dev), W.to(dev), bias.to(dev), tok, exp, cum, full, full, full, True, T, k, d_in, d_out, E)
    want = _expected(x, W, bias, ids, off, start)
    assert float((y.double().cpu() - want).norm() / want.norm()) < BOUND[dtype]
    # the gradients of a layer d_out -> d_in with weights W: j_y [k,T,d_in], x [T,d_out]
    j_x, j_w, j_b = start.to(dev), torch.zeros(E, d_in, d_out, dtype=dtype, device=dev), torch.zeros(E, d_in, dtype=dtype, device=dev)
    rows = torch.randn(T, d_out, generator=g).to(dtype)
    ext.FUSED_GRAD(j_b, j_x, j_w, x.to(dev), W.to(dev), rows.to(dev), tok, exp, cum, full, full, True, T, k, d_out, d_in, E)
    want = _expected(x, W, torch.zeros_like(bias), ids, off, start)
    assert float((j_x.double().cpu() - want).norm() / want.norm()) < BOUND[dtype]
    for e in range(E):
        at = [((ids[:, s] == e) & ~off[:, s]).nonzero()[:, 0] for s in range(k)]
        dw = sum(x[s, a].double().t() @ rows[a].double() for s, a in enumerate(at))
        db = sum(x[s, a].double().sum(0) for s, a in enumerate(at))
        assert float((j_w[e].double().cpu() - dw).norm()) <= BOUND[dtype] * float(dw.norm()) + 1e-30
        assert float((j_b[e].double().cpu() - db).norm()) <= BOUND[dtype] * float(db.norm()) + 1e-30
