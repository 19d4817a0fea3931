"""A forward that no backward follows leaves y1 out; y and the auxiliary loss are bit for bit those of the forward that stores it."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# tokens, dim, hidden, experts, top_k: the pipelined kernel (one tile and several per workgroup, contraction and columns that end inside
# a tile), the one-tile kernel (short contraction; the unrounded product), the 256x256 kernel (full and partial tiles), fp32
@pytest.mark.parametrize("T,d,h,E,k,dtype,tile", [
    (144, 384, 1536, 32, 1, "bf16", 0), (5000, 320, 1288, 4, 2, "fp16", 0), (2000, 264, 1056, 13, 3, "fp16", 0), (300, 64, 136, 5, 1, "bf16", 0),
    (120, 384, 768, 32, 2, "autocast", 0), (3000, 256, 1032, 3, 1, "autocast", 0), (9000, 320, 776, 4, 2, "bf16", 15), (9000, 256, 1024, 4, 1, "fp16", 15),
    (513, 128, 520, 8, 2, "fp32", 0)])
def test_same_results_without_y1(dev, T, d, h, E, k, dtype, tile):
    from hexa_moe import _lib
    from hexa_moe import moe as hmoe
    print(f"forward only: T={T} {d} -> {h} E={E} k={k} {dtype} tile={tile}", flush=True)
    torch.manual_seed(T)
    m = hmoe.MoE_Cascaded(gate_type={"type": "top", "k": k, "gate_noise": 0.0, "fp32_gate": True}, model_dim_list=[d], moe_idx_list=[0],
                          mlp_ratio=h / d, num_global_experts=E, total_depth=1, data_centric=True, activation_fn=F.gelu, is_gshard_loss=True).to(dev)
    for name, p in m.named_parameters():
        torch.nn.init.uniform_(p.data, -0.1, 0.1)
        if not name.startswith("gates"):
            p.data = p.data.to({"bf16": torch.bfloat16, "fp16": torch.float16}.get(dtype, torch.float32))
    m.eval()
    x = torch.randn(T, d, device=dev).to({"bf16": torch.bfloat16, "fp16": torch.float16}.get(dtype, torch.float32))
    lib = _lib.load()
    _lib.check(lib.hexa_set_option(b"tile", tile), "hexa_set_option")
    try:
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == "autocast"):
            want, want_aux = m(0, x)
            with torch.no_grad():
                for _ in range(2):
                    got, aux = m(0, x)
                    torch.cuda.synchronize()
                    assert torch.equal(got, want) and torch.equal(aux, want_aux)
    finally:
        _lib.check(lib.hexa_set_option(b"tile", 0), "hexa_set_option")
