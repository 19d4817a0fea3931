"""What the MoE depth refuses before anything reaches a kernel: operands that are not on the tokens' GPU, and operands that
hold less than would be read."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

T, D, H, E, K = 96, 64, 128, 4, 2
ACTS = {"gelu": F.gelu, "lambda": lambda t: F.gelu(t)}


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _operands(dev):
    g = torch.Generator().manual_seed(0)
    n = lambda *s: (torch.randn(*s, generator=g) * 0.2).to(torch.bfloat16).to(dev)      # noqa: E731
    return {"x": n(T, D), "wg": n(E, D).float(), "w1": n(E, H, D), "w2": n(E, H, D), "b1": n(E, H), "b2": n(E, D),
            "chosen": torch.randint(0, E, (T, K), generator=g).to(dev)}


def _run(o, act, gated):
    from hexa_moe.impls.layers import FusedMoE_Shared_CudaCore, FusedMoEDepth, RoutePool
    cfg = SimpleNamespace(num_global_experts=E, stage=0, route_pool=RoutePool(), activation_fn=ACTS[act], indices_=None, routing_=o["chosen"])
    rest = (o["w1"], o["w2"], o["b1"], o["b2"])
    if gated:
        return FusedMoEDepth.apply(cfg, (K, 0.0, True, 0.0), o["x"], o["wg"], *rest)[0]
    return FusedMoE_Shared_CudaCore.apply(cfg, o["x"], *rest)


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("gated,name", [(g, n) for g in (False, True) for n in ("w1", "w2", "b1", "b2", "wg" if g else "chosen")])
def test_operands_on_the_cpu_are_refused(dev, act, gated, name):
    o = _operands(dev)
    good = _run(o, act, gated)
    o[name] = o[name].cpu()
    with pytest.raises(RuntimeError, match="must be on the tokens' device"):
        _run(o, act, gated)
    o[name] = o[name].to(dev)
    assert torch.equal(_run(o, act, gated), good)


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("name,cut", [("w1", lambda t: t[:-1]), ("w1", lambda t: t[:, :-8]), ("w1", lambda t: t[..., :-8]),
                                      ("w2", lambda t: t[:-1]), ("w2", lambda t: t[:, :-8]), ("w2", lambda t: t[0]),
                                      ("b1", lambda t: t[:-1]), ("b2", lambda t: t[:, :-1]),
                                      ("chosen", lambda t: t[:-1]), ("chosen", lambda t: torch.cat([t, t])), ("x", lambda t: t[:-1]),
                                      ("x", lambda t: t[:, :-8]), ("x", lambda t: t.view(2, T // 2, D))])
def test_operands_of_other_sizes_are_refused(dev, act, name, cut):
    o = _operands(dev)
    o[name] = cut(o[name])
    with pytest.raises(RuntimeError, match="hexa_moe"):
        _run(o, act, False)


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("name,cut", [("wg", lambda t: t[:-1]), ("wg", lambda t: t[:, :-8]), ("x", lambda t: t.view(2, T // 2, D)),
                                      ("w1", lambda t: t[:-1])])
def test_operands_of_other_sizes_are_refused_with_a_gate(dev, act, name, cut):
    o = _operands(dev)
    o[name] = cut(o[name])
    with pytest.raises(RuntimeError, match="hexa_moe"):
        _run(o, act, True)


@pytest.mark.parametrize("change", [lambda t: t[:, :-1], lambda t: t[..., :-8], lambda t: t[0], lambda t: t.cpu()])
def test_what_an_activation_returns_is_checked(dev, change, monkeypatch):
    o = _operands(dev)
    monkeypatch.setitem(ACTS, "odd", lambda t: change(F.gelu(t)))
    with pytest.raises(RuntimeError, match="hexa_moe"):
        _run(o, "odd", False)


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.int16, torch.uint8, torch.bool])
def test_a_decision_in_another_type_is_refused(dev, act, dtype):
    o = _operands(dev)
    o["chosen"] = o["chosen"].to(dtype)
    with pytest.raises(TypeError, match="int32 or int64"):
        _run(o, act, False)


@pytest.mark.parametrize("act", list(ACTS))
def test_a_decision_is_read_in_its_own_type_and_strides(dev, act):
    """Top-1, with ids that are no expert's: an int64 id whose low 32 bits name an expert is not that expert's."""
    def run(chosen):
        o = _operands(dev)
        o["chosen"] = chosen
        ws = [o[n].requires_grad_(True) for n in ("w1", "w2", "b1", "b2")]
        y = _run(o, act, False)
        y.backward(o["x"])
        return [y.detach()[kept]] + [w.grad for w in ws]

    ids = _operands(dev)["chosen"][:, :1].clone()
    kept = torch.ones(T, dtype=torch.bool, device=dev)
    kept[[3, 4, T - 1]] = False
    low = torch.where(kept[:, None], ids, torch.full_like(ids, -1)).to(torch.int32)
    want = run(low)
    high = torch.where(kept[:, None], ids, ids + (1 << 32))
    wide = torch.full((2, T + 1), 99, dtype=torch.int64, device=dev)
    wide[1, :T] = high[:, 0]
    for chosen in (high, wide[1:, :T].t(), low.expand(T, 4)[:, 2:3]):
        for a, b in zip(run(chosen), want):
            assert torch.equal(a, b)
