"""A forward that no backward follows leaves y1 out; y and the auxiliary loss are bit for bit those of the forward that stores it."""
import ctypes

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


# the same sizes and kernels, through the C ABI's option: an element type instead of autocast
@pytest.mark.parametrize("T,d,h,E,k,dtype,tile", [
    (144, 384, 1536, 32, 1, "bf16", 0), (5000, 320, 1288, 4, 2, "fp16", 0), (2000, 264, 1056, 13, 3, "fp16", 0), (300, 64, 136, 5, 1, "bf16", 0),
    (120, 384, 768, 32, 2, "bf16", 0), (3000, 256, 1032, 3, 1, "bf16", 0), (9000, 320, 776, 4, 2, "bf16", 15), (9000, 256, 1024, 4, 1, "fp16", 15),
    (513, 128, 520, 8, 2, "fp32", 0), (3000, 128, 520, 4, 2, "fp32", 0)])
def test_y1_stays_unwritten(dev, T, d, h, E, k, dtype, tile):
    """Every kernel that these sizes run leaves y1 as it was; y2 and y are those of the call that stores it."""
    from hexa_moe import _lib, ops
    from _util import gen, make_routing
    print(f"y1 unwritten: T={T} {d} -> {h} E={E} k={k} {dtype} tile={tile}", flush=True)
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[dtype]
    g, lib, p = gen(T), _lib.load(), ops._ptr
    new = lambda *s: (torch.rand(*s, generator=g) - 0.5).to(dt).to(dev)     # noqa: E731
    x, w1, b1, w2, b2 = new(T, d), new(E, h, d), new(E, h), new(E, h, d), new(E, d)
    idx = make_routing(T, E, k, seed=E).int().to(dev)
    plan = ops.DepthPlan(T, k, E, d, h, d, *[dt] * 8, 0, 0.0, 0.0)
    res = []
    _lib.check(lib.hexa_set_option(b"tile", tile), "hexa_set_option")
    try:
        for no_y1 in (0, 1):
            o = _lib.DepthOpts(ctypes.sizeof(_lib.DepthOpts), 0, 0, 0, 1, no_y1, 0)
            n = ctypes.c_int64()
            _lib.check(lib.hexa_moe_depth_part_ws_bytes(ctypes.byref(plan.desc), ctypes.byref(o), ctypes.byref(n), None), "ws_bytes")
            ws = torch.empty(n.value, dtype=torch.uint8, device=dev)
            blob = torch.empty(ops.route_blob_ints(T, k, E), dtype=torch.int32, device=dev)
            y1, y2, y = torch.full((k, T, h), -77.0, dtype=dt, device=dev), torch.empty(k, T, h, dtype=dt, device=dev), torch.empty(T, d, dtype=dt, device=dev)
            _lib.check(lib.hexa_moe_depth_part_forward(ctypes.byref(plan.desc), ctypes.byref(o), p(x), None, None, p(w1), p(b1), p(w2), p(b2), None, None, p(idx),
                                                       None, None, p(blob), None, p(y1), p(y2), p(y), p(ws), n.value, None, 0, ops._stream()), "forward")
            torch.cuda.synchronize()
            res.append((y1, y2, y))
    finally:
        _lib.check(lib.hexa_set_option(b"tile", 0), "hexa_set_option")
    (y1, y2, y), (none, y2_alone, y_alone) = res
    assert bool((none == -77.0).all()) and not bool((y1 == -77.0).any())
    assert torch.equal(y2, y2_alone) and torch.equal(y, y_alone)
