"""A MoE depth through the tensor-level wrappers of the C ABI's depth calls (ops.DepthPlan, moe_depth_forward / _backward),
and in parts, against the module."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

T, D, H, E = 300, 64, 128, 5


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


class _Depth:
    """Module and buffers of one depth; bias and gate as the C ABI takes them."""

    def __init__(self, dev, dtype, k):
        from hexa_moe import _lib, moe as hmoe, ops
        torch.manual_seed(k)
        self.k, self.dtype, self.dev = k, dtype, dev
        m = hmoe.MoE_Cascaded({"type": "top", "k": k, "fp32_gate": True, "gate_noise": 0.0}, [D], [0], E, 1, mlp_ratio=H / D, activation_fn=F.gelu)
        for n, p in m.named_parameters():
            torch.nn.init.uniform_(p.data, -0.3, 0.3)
            p.data = p.data.to(dev, torch.float32 if n.startswith("gates") else dtype)
        self.m, self.x, self.dy = m, torch.randn(T, D, device=dev).to(dtype), torch.randn(T, D, device=dev).to(dtype)
        x = self.x.clone().requires_grad_(True)
        y, aux = m(0, x)
        torch.autograd.backward([y, aux], [self.dy, torch.ones_like(aux)])
        self.want = {"y": y.detach(), "l_aux": aux.detach(), "dx": x.grad, "dwg": m.gates[0].wg.weight.grad, "dw1": m.batched_fc1_w[0].grad,
                     "db1": m.batched_fc1_bias[0].grad, "dw2": m.batched_fc2_w[0].grad, "db2": m.batched_fc2_bias[0].grad}
        new = lambda *s, t=dtype: torch.empty(*s, dtype=t, device=dev)      # noqa: E731
        f32 = torch.float32
        self.w = {n: p.detach().contiguous() for n, p in zip(("wg", "w1", "w2", "b1", "b2"), (
            m.gates[0].wg.weight, m.batched_fc1_w[0], m.batched_fc2_w[0], m.batched_fc1_bias[0], m.batched_fc2_bias[0]))}
        self.plan = ops.DepthPlan(T, k, E, D, H, D, dtype, dtype, dtype, dtype, dtype, dtype, dtype, dtype, 0, 0.0, 0.0)
        self.logits, self.scores, self.stats = new(T, E, t=f32), new(T, E, t=f32), new(2 * E + 1, t=f32)
        self.idx, self.estmm_plan = new(T, k, t=torch.int32), new(_lib.estmm_plan_ints(E), t=torch.int32)
        self.blob = new(ops.route_blob_ints(T, k, E), t=torch.int32)
        self.y1, self.y2, self.y, self.dy1 = new(k, T, H), new(k, T, H), new(T, D), new(k, T, H)
        self.g_aux = torch.ones((), device=dev)
        self.grads = {"dx": new(T, D), "dwg": new(E, D, t=f32), "dw1": new(E, H, D), "db1": new(E, H), "dw2": new(E, H, D), "db2": new(E, D)}

    def forward(self):
        from hexa_moe import ops
        w = self.w
        ops.moe_depth_forward(self.plan, self.x, w["wg"], None, w["w1"], w["b1"], w["w2"], w["b2"], self.logits, self.scores, self.idx, None,
                              self.stats, self.blob, self.estmm_plan, self.y1, self.y2, self.y,
                              torch.empty(self.plan.fwd_bytes, dtype=torch.uint8, device=self.dev))

    def same(self, names):
        for n in names:
            assert torch.equal(self.grads[n] if n in self.grads else self.y, self.want[n]), n


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [1, 2])
def test_wrappers_give_what_the_module_gives(dev, dtype, k):
    from hexa_moe import ops
    d = _Depth(dev, dtype, k)
    d.forward()
    ops.moe_depth_backward(d.plan, d.dy, d.g_aux, d.x, d.w["wg"], d.w["w1"], d.w["w2"], d.scores, d.idx, None, d.stats, d.blob, d.estmm_plan,
                           d.y1, d.y2, d.grads["dx"], d.grads["dwg"], d.grads["dw1"], d.grads["db1"], d.grads["dw2"], d.grads["db2"], d.dy1,
                           torch.empty(d.plan.bwd_bytes, dtype=torch.uint8, device=dev))
    d.same(("y", "dx", "dwg", "dw1", "db1", "dw2", "db2"))
    assert float(d.stats[-1]) == float(d.want["l_aux"])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("gated", [True, False])
def test_parts_stay_inside_the_scratch_they_ask_for(dev, dtype, k, gated):
    """Every part with exactly the bytes it asks for, in front of memory that has to stay as it is."""
    from hexa_moe import _lib, ops
    lib, d, p = _lib.load(), _Depth(dev, dtype, k), ops._ptr
    d.forward()
    want = {n: t.clone() for n, t in (("y", d.y), ("y1", d.y1), ("y2", d.y2))}
    GUARD = 1 << 16

    def run(part, backward, *args):
        o = _lib.DepthOpts(ctypes.sizeof(_lib.DepthOpts), part, 0, 0, int(not gated))
        sizes = [ctypes.c_int64(), ctypes.c_int64()]
        _lib.check(lib.hexa_moe_depth_part_ws_bytes(ctypes.byref(d.plan.desc), ctypes.byref(o), *[ctypes.byref(s) for s in sizes]), "ws_bytes")
        n = sizes[backward].value
        ws = torch.full((n + GUARD,), 0xA5, dtype=torch.uint8, device=dev)
        fn = lib.hexa_moe_depth_part_backward if backward else lib.hexa_moe_depth_part_forward
        _lib.check(fn(ctypes.byref(d.plan.desc), ctypes.byref(o), *args, p(ws), n, None, 0, ops._stream()), "part")
        assert bool((ws[n:] == 0xA5).all()), f"part {part} wrote behind its scratch"

    w, g = d.w, d.grads
    wg = w["wg"] if gated else None
    for t in (d.y, d.y1, d.y2, d.scores, d.stats):
        t.fill_(float("nan"))
    run(1, 0, p(d.x), p(wg), None, None, None, None, None, p(d.logits), p(d.scores), p(d.idx), None, p(d.stats), p(d.blob), p(d.estmm_plan), None, None, None)
    run(2, 0, p(d.x), None, None, p(w["w1"]), p(w["b1"]), None, None, None, None, None, None, None, p(d.blob), None, p(d.y1), None, None)
    assert torch.equal(d.y1, want["y1"])
    d.y2.copy_(want["y2"])
    run(4, 0, None, None, None, None, None, p(w["w2"]), p(w["b2"]), None, None, None, None, None, p(d.blob), None, None, p(d.y2), p(d.y))
    assert torch.equal(d.y, want["y"])
    run(4, 1, p(d.dy), None, None, None, None, p(w["w2"]), None, None, None, None, p(d.blob), p(d.estmm_plan), None, p(d.y2), None, None, None, None,
        p(g["dw2"]), p(g["db2"]), p(d.dy1))
    d.same(("dw2", "db2"))
    # the activation's derivative between the halves, as the caller would have it
    y1 = d.y1.clone().requires_grad_(True)
    F.gelu(y1).backward(d.dy1)
    d.dy1.copy_(y1.grad)
    run(2, 1, None, p(d.g_aux) if gated else None, p(d.x), p(wg), p(w["w1"]), None, p(d.scores), p(d.idx), None, p(d.stats), p(d.blob), p(d.estmm_plan),
        None, None, p(g["dx"]), p(g["dwg"]) if gated else None, p(g["dw1"]), p(g["db1"]), None, None, p(d.dy1))
    bound = 1e-5 if dtype == torch.float32 else 1e-2       # GELU' of a dy2 rounded in between
    for n in ("dw1", "db1") + (("dx", "dwg") if gated else ()):
        assert float((g[n].double() - d.want[n].double()).norm()) <= bound * float(d.want[n].double().norm()), n
