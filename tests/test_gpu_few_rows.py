"""Lists that end anywhere inside a row tile, in the kernels that copy and multiply only the blocks of 32 rows that hold something or
that take a tile's rows block by block: the pipelined ESMM and the ESMM of the shared backward launches."""
import pytest
import torch
import torch.nn.functional as F

from _util import TOL, assert_close, gen
from oracle import hexa_oracle as O

pytestmark = pytest.mark.gpu

# rows of every expert: none, one, the ends of 32-row blocks and of 128-row tiles, tiles of one to four blocks behind full ones
ROWS = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128, 129, 160, 161, 0, 300, 226]
E = len(ROWS)


def _lists(seed):
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(ROWS))
    return ids[torch.randperm(len(ids), generator=gen(seed))]


@pytest.fixture
def knobs():
    from hexa_moe import _lib
    lib, used = _lib.load(), set()

    def set_(**cfg):
        for name, value in cfg.items():
            used.add(name)
            _lib.check(lib.hexa_set_option(name.encode(), value), "hexa_set_option")
    yield set_
    for name in used:
        _lib.check(lib.hexa_set_option(name.encode(), 0), "hexa_set_option")


# whole stages and a contraction that ends inside one; 9 and 3 column tiles, the last of 8 columns (workgroups of two tiles and of one)
@pytest.mark.parametrize("d_in,d_out", [(256, 1032), (200, 1032), (256, 264)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_pipelined_esmm(dev, knobs, dtype, k, d_in, d_out):
    """Against fp64, and bit for bit against the one-tile kernel, which multiplies all rows of every tile (column sums: up to the order of a
    tile's rows).  Then NaN in the rows of the longest list: what a workgroup's earlier tile left in LDS is not multiplied, so
    every other list's results stay as they were."""
    from hexa_moe import _lib, ops
    print(f"few rows: pipelined ESMM {d_in} -> {d_out} k={k} {dtype}", flush=True)
    first = _lists(d_in)
    T = len(first)
    routing = torch.stack([(first + s) % E for s in range(k)], 1)
    _, offsets, token_ids = O.route_build(routing, E)
    route = ops.route_build(routing.to(dev), E)
    g = gen(d_out)
    x = torch.randn(T, d_in, generator=g).to(dtype)
    W = (torch.randn(E, d_in, d_out, generator=g) / d_in ** 0.5).to(dtype)
    b = torch.randn(E, d_out, generator=g).to(dtype)
    Wt, back = W.transpose(1, 2).contiguous().to(dev), torch.randn(k, T, d_out, generator=g).to(dtype).to(dev)

    def results(x, back):
        y1, y2 = ops.esmm(x, Wt, b.to(dev), route, False, _lib.HEXA_W_OUT_IN, gelu=True)
        dy1, db = ops.esmm_gelu_bwd_ess(x, Wt, route, _lib.HEXA_W_OUT_IN, back)
        dx = ops.esmm(back, Wt, None, route, True, _lib.HEXA_W_IN_OUT)
        torch.cuda.synchronize()
        return {"y1": y1, "dx": dx, "y2": y2, "dy1": dy1, "db": db}

    knobs(pipe=2)
    alone = results(x.to(dev), back)
    knobs(pipe=1)
    got = results(x.to(dev), back)
    want = O.esmm(x.double(), W.double(), b.double(), token_ids, offsets, False)
    assert_close(got["y1"], want, TOL[dtype], "y1")
    assert_close(got["y2"], F.gelu(want), TOL[dtype], "y2")
    assert_close(got["dx"], O.esmm(back.double().cpu(), W.transpose(1, 2).double(), None, token_ids, offsets, True), TOL[dtype], "dx")
    for n in got:
        # (contractions that are no multiple of 32: the one-tile kernel activates the fp32 product, and adds it to the other slot's)
        exact = {"y1": True, "dx": k == 1, "y2": d_in % 32 == 0, "dy1": d_in % 32 == 0, "db": False}[n]
        if exact:
            assert torch.equal(got[n], alone[n]), n
        else:
            assert_close(got[n], alone[n], TOL[dtype], n)

    most = ROWS.index(max(ROWS))
    x[first == most] = float("nan")
    bad = back.clone()
    bad[:, (first == most).to(dev)] = float("nan")
    nan = results(x.to(dev), bad)
    rest = (first != most).to(dev)
    for n in ("y1", "y2", "dy1"):
        assert torch.equal(nan[n][:, rest], got[n][:, rest]) and bool(nan[n][:, ~rest].isnan().all()), n
    assert torch.equal(nan["dx"][rest], got["dx"][rest])
    others = [e for e in range(E) if all((e - s) % E != most for s in range(k))]
    assert torch.equal(nan["db"][others], got["db"][others])


# (64, 192): whole stages in both launches; (264, 520): the launches whose epilogue takes the fp32 product, column tiles that end early
@pytest.mark.parametrize("d,h", [(64, 192), (264, 520)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("T", [65, 260, 1030, sum(ROWS)])       # 2, 5, 17 and 26 chunks of the gate's backward: every remainder of four
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_shared_backward_launches(dev, knobs, dtype, T, k, d, h):
    """Against launches of their own: the same sums in the same order (dwg: one partial result per chunk here, one per four chunks there)."""
    from hexa_moe import moe as hmoe
    print(f"few rows: shared launches T={T} k={k} {d} -> {h} {dtype}", flush=True)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0], mlp_ratio=h / d,
                          num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu).to(dev)
    g = gen(T + d)
    for name, p in m.named_parameters():
        p.data = ((torch.rand(p.shape, generator=g) * 2 - 1) * 0.1).to(torch.float32 if name.startswith("gates") else dtype).to(dev)
    m.gates[0].wg.weight.data = torch.eye(E, d, device=dev)
    first = _lists(T)[:T]
    x = torch.randn(T, d, generator=g)
    x[:, :E] = 0.1 * x[:, :E].clamp(-2, 2)
    for s in range(k):
        x[torch.arange(T), (first + s) % E] = 4.0 - 2 * s
    x, dy = x.to(dtype).to(dev), torch.randn(T, d, generator=g).to(dtype).to(dev)
    res = []
    for fused in (1, 2):
        knobs(backward_fused=fused)
        m.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        y, l_aux = m(0, xi)
        torch.autograd.backward([y, l_aux], [dy, torch.full((), 3.0, device=dev)])
        torch.cuda.synchronize()
        assert torch.equal(m.dispatch_params.routing_.cpu().long(), torch.stack([(first + s) % E for s in range(k)], 1))
        res.append((xi.grad, {n: p.grad.clone() for n, p in m.named_parameters()}))
    (dx1, g1), (dx2, g2) = res
    assert_close(dx1, dx2, 1e-2, "dx")                 # (with one slot the gate's share is added elsewhere)
    for n in g1:
        if "fc1_bias" in n:                            # the column sums of two kernels group a tile's rows differently
            assert_close(g1[n], g2[n], 1e-2, n)
        else:
            assert torch.equal(g1[n], g2[n]), n
