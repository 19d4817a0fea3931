"""The gate's projection inside the router's launch, over the model dimensions where its trips end: a trip is six chunks of 16 columns of
each quarter, and a quarter may be a chunk shorter than the first."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# 8 to 384 columns are one trip of one to six chunks, 392 two (the second of one chunk for some quarters and none for others), 1160 four
DIMS = [8, 16, 24, 40, 64, 72, 104, 128, 136, 192, 200, 256, 264, 320, 384, 392, 448, 512, 520, 768, 776, 1024, 1160]


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32", "autocast"])
@pytest.mark.parametrize("E,k,loss,T", [(7, 2, "gshard", 197), (33, 1, "importance", 130), (64, 3, "importance", 65)])
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
