"""fp32 tokens under 16-bit autocast are rounded inside the gate's launch and a top-1 result leaves the second layer as fp32:
the same layer fed with tokens rounded beforehand gives the same decisions, results and gradients."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["gelu", "lambda"])
@pytest.mark.parametrize("T,d,E,k,offset", [
    (2304, 384, 32, 1, 0),     # the pipelined kernel stores y
    (4608, 768, 32, 1, 0),     # between one and two tiles per CU: the one-tile kernel does
    (65, 264, 5, 1, 0), (1, 64, 4, 1, 0), (130, 40, 6, 1, 0),   # ragged rows, pieces and experts
    (300, 64, 300, 1, 0),      # a gate in a launch of its own: tokens rounded in front of it
    (500, 128, 8, 2, 0),       # two slots: y leaves in the 16-bit type
    (500, 128, 8, 1, 1),       # tokens that start at no multiple of 16 bytes
])
def test_rounded_on_the_way(dev, dtype, act, T, d, E, k, offset):
    from hexa_moe import moe as hmoe
    torch.manual_seed(3)
    fn = F.gelu if act == "gelu" else lambda t: F.gelu(t)      # noqa: E731
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          num_global_experts=E, total_depth=1, data_centric=True, activation_fn=fn)
    for p in m.parameters():
        torch.nn.init.uniform_(p.data, -0.08, 0.08)
    m = m.to(dev)
    full = torch.randn(T * d + offset, device=dev)[offset:].view(T, d).detach()
    dy = torch.randn(T, d, device=dev).to(dtype)

    def run(x):
        x = x.detach().requires_grad_(True)
        with torch.autocast("cuda", dtype=dtype):
            y, l_aux = m(0, x)
        torch.autograd.backward([y, l_aux], [dy.to(y.dtype), torch.ones_like(l_aux)])
        grads = [p.grad for p in m.parameters()]
        for p in m.parameters():
            p.grad = None
        return y.detach(), l_aux.detach(), x.grad, m.dispatch_params.routing_, grads

    y, l_aux, dx, routing, grads = run(full)
    y16, l_aux16, dx16, routing16, grads16 = run(full.to(dtype))
    assert y.dtype == torch.float32 and dx.dtype == torch.float32 and y16.dtype == dtype
    assert torch.equal(routing, routing16) and torch.equal(l_aux, l_aux16)
    assert torch.equal(dx, dx16.float())
    for a, b in zip(grads, grads16):
        assert torch.equal(a, b)
    # rounded like y16, or not rounded at all: within the rounding of a 16-bit value (fp16: of its subnormals)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((y - y16.float()).abs() <= ulp * y16.float().abs() + 2.0 ** -24).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,E,k", [(2304, 384, 32, 1), (65, 264, 5, 1), (500, 128, 8, 2)])
def test_against_fp64(dev, dtype, T, d, E, k):
    """The layer in 64 bits for the tokens and weights as they are rounded.  Four roundings in a chain, as in
    test_gpu_backward_fused.py."""
    from _util import layer_fp64, rel_err
    from hexa_moe import moe as hmoe
    torch.manual_seed(4)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu)
    for p in m.parameters():
        torch.nn.init.uniform_(p.data, -0.08, 0.08)
    m = m.to(dev)
    x = torch.randn(T, d, device=dev).requires_grad_(True)
    with torch.autocast("cuda", dtype=dtype):
        y, l_aux = m(0, x)
    dy = torch.randn(T, d, device=dev).to(dtype)
    torch.autograd.backward([y, l_aux], [dy.to(y.dtype), torch.ones_like(l_aux)])
    params = [m.gates[0].wg.weight, m.batched_fc1_w[0], m.batched_fc2_w[0], m.batched_fc1_bias[0], m.batched_fc2_bias[0]]
    w = [params[0], params[1].to(dtype), params[2].to(dtype), *params[3:]]
    y_ref, aux_ref, grads = layer_fp64(x.to(dtype), m.dispatch_params.routing_, *w, dy, 1.0)
    assert abs(l_aux.item() - aux_ref.item()) <= 1e-5 * abs(aux_ref.item())
    most = 6.8e-3 if dtype == torch.bfloat16 else 8.5e-4
    names = ("y", "dx", "dwg", "dW1", "dW2", "db1", "db2")
    errs = {n: rel_err(a.grad if n != "y" else a, b)[0] for n, a, b in zip(names, [y, x] + params, [y_ref] + grads)}
    assert all(e <= most for e in errs.values()), errs


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,h,E,aux", [
    (9216, 384, 1536, 32, True), (9216, 384, 1536, 32, False),     # shared launches; without the gate's share nothing else passes over dx
    (100, 384, 1536, 32, True), (301, 264, 1000, 5, True),         # the gate's share first and dx onto it
    (3700, 768, 3072, 8, True), (3700, 768, 3072, 8, False),       # separate launches
    (1, 8, 16, 4, True), (33, 40, 264, 6, False),
])
def test_dx_leaves_as_fp32(dev, dtype, T, d, h, E, aux):
    """The pass that finishes dx widens it: what it stores is the 16-bit value, and what tokens rounded beforehand get."""
    from hexa_moe import moe as hmoe
    print(f"dx as fp32: T={T} {d} -> {h} E={E} aux={aux} {dtype}", flush=True)
    torch.manual_seed(5)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": 1, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu).to(dev)
    for p in m.parameters():
        torch.nn.init.uniform_(p.data, -0.08, 0.08)
    full, dy = torch.randn(T, d, device=dev), torch.randn(T, d, device=dev).to(dtype)
    got = []
    for x in (full, full.to(dtype)):
        x = x.detach().requires_grad_(True)
        with torch.autocast("cuda", dtype=dtype):
            y, l_aux = m(0, x)
        torch.autograd.backward([y, l_aux] if aux else [y], [dy.to(y.dtype), torch.ones_like(l_aux)] if aux else [dy.to(y.dtype)])
        torch.cuda.synchronize()
        got.append(x.grad)
    assert got[0].dtype == torch.float32 and torch.equal(got[0], got[0].to(dtype).float()) and torch.equal(got[0], got[1].float())
