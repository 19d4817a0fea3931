"""The MoE depth has no forward-mode derivative, and says so instead of returning a result without its tangent."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

E, H, D, T = 2, 16, 8, 4
SHAPES = {"x": (T, D), "wg": (E, D), "w1": (E, H, D), "w2": (E, H, D), "b1": (E, H), "b2": (E, D)}


@pytest.mark.parametrize("half,dual", [(h, d) for h in (False, True) for d in SHAPES if not (h and d in ("w2", "b2"))])
def test_dual_operands_are_refused(half, dual):
    """(looked at before the device, so CPU tensors do)"""
    from hexa_moe import _native
    n = _native.load()
    with fwAD.dual_level():
        o = {k: torch.zeros(*s) for k, s in SHAPES.items()}
        o[dual] = fwAD.make_dual(o[dual], torch.ones_like(o[dual]))
        r = n.Routing(1, E)
        with pytest.raises(NotImplementedError, match="forward-mode"):
            if half:
                n.depth_in(n.RoutePool(), 0, o["x"], o["wg"], o["w1"], o["b1"], None, o["w2"], r, None)
            else:
                n.depth(n.RoutePool(), 0, o["x"], o["wg"], o["w1"], o["w2"], o["b1"], o["b2"], None, r, [], [], None)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [F.gelu, lambda t: F.gelu(t)])
@pytest.mark.parametrize("dual", ["x", "batched_fc1_w", "batched_fc2_w", "batched_fc2_bias", "batched_fc1_bias"])
def test_module_refuses_dual_operands(act, dual):
    from hexa_moe import moe as hmoe
    m = hmoe.MoE_Cascaded({"type": "top", "k": 1, "fp32_gate": True, "gate_noise": 0.0}, [D], [0], E, 1, mlp_ratio=2, activation_fn=act).cuda()
    x = torch.randn(T, D, device="cuda")
    with fwAD.dual_level():
        if dual == "x":
            x = fwAD.make_dual(x, torch.ones_like(x))
        else:
            plist = getattr(m, dual)
            p = plist[0]
            del plist._parameters["0"]
            setattr(plist, "0", fwAD.make_dual(p.detach(), torch.ones_like(p)))
        with pytest.raises(NotImplementedError, match="forward-mode"):
            m(0, x)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [F.gelu, lambda t: F.gelu(t)])
@pytest.mark.parametrize("transform", ["grad", "vmap", "jvp"])
def test_function_transforms_are_refused(act, transform):
    from hexa_moe import moe as hmoe
    m = hmoe.MoE_Cascaded({"type": "top", "k": 1, "fp32_gate": True, "gate_noise": 0.0}, [D], [0], E, 1, mlp_ratio=2, activation_fn=act).cuda()
    x = torch.randn(T, D, device="cuda")
    f = lambda t: m(0, t)[0]      # noqa: E731
    with pytest.raises((RuntimeError, NotImplementedError)):
        if transform == "grad":
            torch.func.grad(lambda t: f(t).sum())(x)
        elif transform == "vmap":
            torch.func.vmap(f)(x.expand(3, T, D))
        else:
            torch.func.jvp(f, (x,), (torch.ones_like(x),))
