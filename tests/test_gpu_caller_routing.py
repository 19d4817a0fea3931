"""Routing decisions of the caller's that no gate makes: no tokens, more slots than experts, more experts than the router
or a weight gradient's work plan takes."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from _util import gen, uniform

pytestmark = pytest.mark.gpu

ACTS = {"gelu": F.gelu, "lambda": lambda t: F.gelu(t)}
BOUND = {torch.float32: 2e-6, torch.bfloat16: 1e-2}     # 16 bits: y1, act(y1), each slot's product and the sum are rounded


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _layer(T, E, k, d, h, dtype, master, seed, dev):
    g = gen(seed)
    o = {"x": torch.randn(T, d, generator=g).to(dtype), "w1": uniform((E, h, d), d ** -0.5, g), "w2": uniform((E, h, d), h ** -0.5, g),
         "b1": uniform((E, h), 0.3, g), "b2": uniform((E, d), 0.3, g)}
    o = {n: (t.to(dtype) if n != "x" and not master else t).to(dev).requires_grad_(True) for n, t in o.items()}
    return o, torch.randint(0, E, (T, k), generator=g).to(dev)


def _run(o, chosen, E, act):
    from hexa_moe.impls.layers import FusedMoE_Shared_CudaCore, RoutePool
    cfg = SimpleNamespace(num_global_experts=E, stage=0, route_pool=RoutePool(), activation_fn=ACTS[act], routing_=chosen, indices_=None)
    return FusedMoE_Shared_CudaCore.apply(cfg, o["x"], o["w1"], o["w2"], o["b1"], o["b2"])


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("dtype,master", [(torch.float32, True), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("k", [1, 2])
def test_no_tokens(dev, act, dtype, master, k):
    o, chosen = _layer(0, 3, k, 16, 32, dtype, master, 1, dev)
    y = _run(o, chosen, 3, act)
    assert y.shape == (0, 16) and y.dtype == dtype
    y.backward(torch.empty_like(y))
    for n, t in o.items():
        assert t.grad.shape == t.shape and t.grad.dtype == t.dtype and not t.grad.any(), n


@pytest.mark.parametrize("act", list(ACTS))
def test_no_tokens_through_a_gate_outside_the_fused_router(dev, act):
    from hexa_moe import moe as hmoe
    # (the GShard loss divides by the number of tokens and raises)
    m = hmoe.MoE_Cascaded({"type": "cosine_top", "k": 1, "gate_noise": 1.0}, [16], [0], 4, 1, mlp_ratio=2, activation_fn=ACTS[act],
                          is_gshard_loss=False).to(dev)
    x = torch.empty(0, 16, device=dev, requires_grad=True)
    y, _ = m(0, x)
    y.sum().backward()
    assert y.shape == (0, 16) and x.grad.shape == (0, 16) and not m.batched_fc1_w[0].grad.any() and not m.batched_fc2_bias[0].grad.any()


def _expected(o, chosen, dtype):
    """(y, its gradients for dy = 1) in fp64 from the weights rounded to the tokens' type."""
    v = {n: t.detach().to(dtype if n in ("x", "w1", "w2") else t.dtype).double().requires_grad_(True) for n, t in o.items()}
    y = torch.zeros(chosen.shape[0], v["w2"].shape[2], dtype=torch.float64, device=chosen.device)
    for s in range(chosen.shape[1]):
        e = chosen[:, s].long()
        y1 = (v["w1"][e] @ v["x"].unsqueeze(2)).squeeze(2) + v["b1"][e]
        y = y + (F.gelu(y1).unsqueeze(1) @ v["w2"][e]).squeeze(1) + v["b2"][e]
    y.sum().backward()
    return y.detach(), {n: t.grad for n, t in v.items()}


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("dtype,master", [(torch.float32, True), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("T,E,k", [(40, 1, 2), (200, 2, 3), (33, 3, 11)])
def test_more_slots_than_experts(dev, act, dtype, master, T, E, k):
    o, chosen = _layer(T, E, k, 32, 64, dtype, master, T, dev)
    y = _run(o, chosen, E, act)
    y.backward(torch.ones_like(y))
    want, grads = _expected(o, chosen, dtype)
    assert float((y.double() - want).norm() / want.norm()) < BOUND[dtype]
    for n, t in o.items():
        assert float((t.grad.double() - grads[n]).norm() / grads[n].norm()) < BOUND[dtype], n


@pytest.mark.parametrize("act", list(ACTS))
def test_more_experts_than_a_plan_orders(dev, act):
    """Inference has no weight gradients and needs no plan; a 16-bit backward refuses, as hexa_estmm_plan does."""
    o, chosen = _layer(96, 4100, 2, 16, 32, torch.bfloat16, False, 3, dev)
    with torch.no_grad():
        y = _run(o, chosen, 4100, act)
    want, _ = _expected(o, chosen, torch.bfloat16)
    assert float((y.double() - want).norm() / want.norm()) < BOUND[torch.bfloat16]
    y = _run(o, chosen, 4100, act)
    with pytest.raises(RuntimeError, match="4096 experts"):
        y.backward(torch.ones_like(y))
