"""The gate's projection inside the router's launch, over the model dimensions where its trips end (a trip is six chunks of 16 columns of
each quarter, and a quarter may be a chunk shorter than the first), and weights that start anywhere."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# 8 to 384 columns are one trip of one to six chunks, 392 two (the second of one chunk for some quarters and none for others), 1160 four.  Up to 16 experts
# have no trips (rounded tokens: where columns and experts are few): a quarter of no, one, an even and an odd number of chunks, a last chunk of one piece
DIMS = [8, 16, 24, 40, 64, 72, 104, 128, 136, 192, 200, 256, 264, 320, 384, 392, 448, 512, 520, 768, 776, 1024, 1160]


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32", "autocast"])
@pytest.mark.parametrize("E,k,loss,T", [(7, 2, "gshard", 197), (16, 2, "importance", 129), (17, 1, "gshard", 70), (33, 1, "importance", 130), (64, 3, "importance", 65)])
def test_equal_to_the_gate_alone(dev, dtype, E, k, loss, T):
    """Routing, scores (through l_aux and the gate's gradient) and y are bit for bit those of the gate in a launch of its own."""
    from hexa_moe import _lib, moe as hmoe
    lib = _lib.load()
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16}.get(dtype, torch.float32)
    for d in DIMS:
        print(f"gate trips: T={T} d={d} E={E} k={k} {dtype} {loss}", flush=True)
        torch.manual_seed(d)
        m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 1.0 if loss == "importance" else 0.0, "fp32_gate": True}, model_dim_list=[d],
                              moe_idx_list=[0], mlp_ratio=1, num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu,
                              is_gshard_loss=loss == "gshard").to(dev).train()
        for name, p in m.named_parameters():
            torch.nn.init.uniform_(p.data, -0.5, 0.5)
            if not name.startswith("gates"):
                p.data = p.data.to(dt)
        x = torch.randn(T, d, device=dev).to(dt).requires_grad_(True)
        res = []
        try:
            for alone in (0, 2):
                _lib.check(lib.hexa_set_option(b"gate_router", alone), "hexa_set_option")
                m.zero_grad(set_to_none=True)
                x.grad = None
                torch.manual_seed(3)
                with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == "autocast"):
                    y, l_aux = m(0, x)
                torch.autograd.backward([y, l_aux], [torch.ones_like(y), torch.ones_like(l_aux)])
                torch.cuda.synchronize()
                res.append((m.dispatch_params.routing_.clone(), y.detach(), l_aux.detach(), m.gates[0].wg.weight.grad.clone()))
        finally:
            _lib.check(lib.hexa_set_option(b"gate_router", 0), "hexa_set_option")
        for name, a, b in zip(("routing", "y", "l_aux", "dwg"), *res):
            assert torch.equal(a, b), (name, d)


@pytest.mark.parametrize("dtype", ["bf16", "fp32", "autocast"])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_gate_weights_inside_a_larger_buffer(dev, dtype, offset):
    """Values that start `offset` floats behind a 16-byte boundary give what a tensor of their own gives."""
    from hexa_moe import moe as hmoe
    T, d, E = 300, 136, 9
    print(f"gate weights {offset} floats into a buffer, {dtype}", flush=True)
    torch.manual_seed(offset)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": 2, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0], mlp_ratio=1,
                          num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu, is_gshard_loss=True).to(dev).train()
    if dtype == "bf16":
        for name, p in m.named_parameters():
            if not name.startswith("gates"):
                p.data = p.data.bfloat16()
    wg = m.gates[0].wg.weight
    own = torch.randn(E, d, device=dev)
    buffer = torch.empty(E * d + 4, device=dev)
    x = torch.randn(T, d, device=dev).to(torch.bfloat16 if dtype == "bf16" else torch.float32).requires_grad_(True)
    res = []
    for place in (own, buffer[offset:offset + E * d].view(E, d).copy_(own)):
        wg.data = place
        assert wg.data_ptr() % 16 == (4 * offset if place is not own else 0)
        m.zero_grad(set_to_none=True)
        x.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == "autocast"):
            y, l_aux = m(0, x)
        torch.autograd.backward([y, l_aux], [torch.ones_like(y), torch.ones_like(l_aux)])
        torch.cuda.synchronize()
        res.append((m.dispatch_params.routing_.clone(), y.detach(), l_aux.detach(), x.grad.clone(), wg.grad.clone()))
    for name, a, b in zip(("routing", "y", "l_aux", "dx", "dwg"), *res):
        assert torch.equal(a, b), name
