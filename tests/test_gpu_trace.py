"""A module under torch.jit.trace: every MoE depth is one operation of the trace and gives what it gives eagerly, also for
inputs the trace has not seen, in the forward and the backward."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


class _Model(torch.nn.Module):
    def __init__(self, act, k, fused_depth):
        super().__init__()
        from hexa_moe import moe as hmoe
        torch.manual_seed(0)
        self.m = hmoe.MoE_Cascaded({"type": "top", "k": k, "fp32_gate": True, "gate_noise": 0.0}, [64, 64], [0, 1], 4, 2, mlp_ratio=2, activation_fn=act)
        self.m.fused_depth = fused_depth
        for p in self.m.parameters():
            torch.nn.init.uniform_(p.data, -0.2, 0.2)

    def forward(self, x):
        y, l0 = self.m(0, x)
        y, l1 = self.m(1, y + x)
        return y, l0 + l1


def _step(f, model, x):
    model.zero_grad(set_to_none=True)
    x = x.clone().requires_grad_(True)
    y, aux = f(x)
    (y.square().mean() + aux).backward()
    return [y.detach(), aux.detach(), x.grad] + [p.grad for p in model.parameters()]


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("act", [F.gelu, lambda t: F.gelu(t)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("fused_depth", [True, False])
def test_traced_module_matches_eager(act, k, fused_depth):
    model = _Model(act, k, fused_depth).cuda()
    x, other = torch.randn(2, 96, 64, device="cuda").unbind(0)
    traced = torch.jit.trace(model, (x,), check_trace=False)
    for t in (x, other, other):
        junk = [torch.full((n,), float("nan"), device="cuda") for n in (96 * 64, 96 * 128, 2 * 96 * 128) for _ in range(6)]
        del junk
        with torch.no_grad():
            for a, b in zip(traced(t), model(t)):
                assert torch.equal(a, b)
        for a, b in zip(_step(traced, model, t), _step(model, model, t)):
            assert (a is None) == (b is None) and (a is None or torch.equal(a, b))
