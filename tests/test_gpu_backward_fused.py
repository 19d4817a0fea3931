"""The backward whose independent products share launches (library option "backward_fused"), against the one-launch-per-
product form: the same sums in the same order, so every gradient but dx (whose gate share is added elsewhere with one
slot) is the same to the bit."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,h,E,k,bias,act", [(1, 64, 128, 3, 1, True, "gelu"), (130, 72, 144, 5, 2, True, "gelu"), (700, 264, 520, 13, 3, False, "gelu"),
                                                (2048, 128, 256, 4, 2, True, "own"), (1500, 136, 400, 2, 1, True, "own")])
def test_shared_launches_equal_separate_ones(dev, dtype, T, d, h, E, k, bias, act):
    from hexa_moe import _lib, moe as hmoe
    print(f"shared launches: T={T} d={d} h={h} E={E} k={k} {act} {dtype}", flush=True)
    lib = _lib.load()
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, mlp_fc1_bias=bias, mlp_fc2_bias=bias,
                          activation_fn=F.gelu if act == "gelu" else lambda t: F.gelu(t)).to(dev).to(dtype)
    g = torch.Generator().manual_seed(T)
    for p in m.parameters():
        p.data = ((torch.rand(p.shape, generator=g) * 2 - 1) * 0.1).to(p.dtype).to(dev)
    m.gates[0].wg.weight.data = m.gates[0].wg.weight.data.float()
    x = torch.randn(T, d, generator=g).to(dtype).to(dev)
    dy = torch.randn(T, d, generator=g).to(dtype).to(dev)
    res = []
    try:
        for fused in (1, 2):
            _lib.check(lib.hexa_set_option(b"backward_fused", fused), "hexa_set_option")
            m.zero_grad(set_to_none=True)
            xi = x.clone().requires_grad_(True)
            y, l_aux = m(0, xi)
            torch.autograd.backward([y, l_aux], [dy, torch.full((), 3.0, device=dev)])
            torch.cuda.synchronize()
            res.append((xi.grad.float(), {n: p.grad.clone() for n, p in m.named_parameters()}))
    finally:
        _lib.check(lib.hexa_set_option(b"backward_fused", 0), "hexa_set_option")
    (dx1, g1), (dx2, g2) = res
    for n in g1:
        same = torch.equal(g1[n], g2[n])
        assert same or "fc1_bias" in n, n       # the column sums of two kernels group a tile's rows differently
        assert (g1[n].float() - g2[n].float()).norm() <= 1e-2 * g2[n].float().norm(), n
    assert (dx1 - dx2).norm() <= 1e-2 * dx2.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,h,E,k,bias,act", [(130, 72, 144, 5, 2, True, "gelu"), (700, 264, 520, 13, 3, False, "gelu"),
                                                (2048, 128, 256, 4, 2, True, "own"), (1500, 136, 400, 2, 1, True, "own")])
def test_shared_launches_against_fp64(dev, dtype, T, d, h, E, k, bias, act):
    """y1, act(y1), dy1 and the result are each rounded once (rms of a rounding: 2^-7 / sqrt(12) = 2.3e-3 of the value's power of
    two in bf16, an eighth of it in fp16); four of them in a chain, and half as much again."""
    from _util import layer_fp64, rel_err
    from hexa_moe import moe as hmoe
    print(f"shared launches, fp64: T={T} d={d} h={h} E={E} k={k} {act} {dtype}", flush=True)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, mlp_fc1_bias=bias, mlp_fc2_bias=bias,
                          activation_fn=F.gelu if act == "gelu" else lambda t: F.gelu(t)).to(dev).to(dtype)
    g = torch.Generator().manual_seed(T)
    for p in m.parameters():
        p.data = ((torch.rand(p.shape, generator=g) * 2 - 1) * 0.1).to(p.dtype).to(dev)
    wg = m.gates[0].wg.weight
    wg.data = wg.data.float()
    x = torch.randn(T, d, generator=g).to(dtype).to(dev).requires_grad_(True)
    dy = torch.randn(T, d, generator=g).to(dtype).to(dev)
    y, l_aux = m(0, x)
    torch.autograd.backward([y, l_aux], [dy, torch.full((), 3.0, device=dev)])
    params = [wg, m.batched_fc1_w[0], m.batched_fc2_w[0], m.batched_fc1_bias[0] if bias else None, m.batched_fc2_bias[0] if bias else None]
    y_ref, aux_ref, grads = layer_fp64(x, m.dispatch_params.routing_, *params, dy, 3.0)
    assert abs(l_aux.item() - aux_ref.item()) <= 1e-5 * abs(aux_ref.item())
    most = 6.8e-3 if dtype == torch.bfloat16 else 8.5e-4
    names = ("y", "dx", "dwg", "dW1", "dW2", "db1", "db2")
    errs = {n: rel_err(a.grad if n != "y" else a, b)[0] for n, a, b in zip(names, [y, x] + params, [y_ref] + grads) if b is not None}
    assert all(e <= most for e in errs.values()), errs
