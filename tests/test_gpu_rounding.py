"""Where a result is rounded to 16 bits: contractions that are no multiple of 32, and fp32 master weights used for fewer than
32 rows an expert, keep the fp32 product up to the activation and up to the sum it joins, and take erf from the library."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _sweep(dtype):
    """Every value of the type between -5.6 and -2, where GELU is what is left of 1 + erf: an error of erf shows in it whole."""
    v = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dtype).double()
    return v[(v > -5.6) & (v < -2.0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_takes_erf(dev, dtype):
    """y1 = v exactly (one non-zero product).  Bounds: rounding of the result, and of erf near -1 in fp32 -- 2 units of 2^-24
    for erff, one for 1 + erf, times |v| / 2 for GELU and 1 / 2 for GELU', whose second term has a few roundings of its own.
    (With the polynomial erf of the kernels for aligned sizes, 6e-7, GELU of a sixth of the bf16 values lies outside.)"""
    from hexa_moe import _lib, ops
    v = _sweep(dtype)
    T, d_in, d_out = v.numel(), 8, 8
    x = torch.zeros(T, d_in, dtype=dtype)
    x[:, 0] = v.to(dtype)
    w = torch.zeros(1, d_out, d_in, dtype=dtype)
    w[0, :, 0] = 1.0
    route = ops.route_build(torch.zeros(T, 1, dtype=torch.int64, device=dev), 1)
    y1, y2 = ops.esmm(x.to(dev), w.to(dev), None, route, False, _lib.HEXA_W_OUT_IN, gelu=True)
    assert torch.equal(y1[0, :, 0].double().cpu(), v)
    unit = 2.0 ** -24
    rounding, tiny = (1.01 * 2.0 ** -8, 2.0 ** -134) if dtype == torch.bfloat16 else (1.01 * 2.0 ** -11, 2.0 ** -25)
    tail = 0.5 * torch.erfc(-v / math.sqrt(2.0))                       # Phi(v)
    want = v * tail
    bound = rounding * want.abs() + tiny + 0.5 * v.abs() * 3 * unit
    assert ((y2[0].double().cpu() - want[:, None]).abs() <= bound[:, None]).all()
    dy = torch.zeros(T, d_in, dtype=dtype)
    dy[:, 0] = 1.0
    dy1 = ops.esmm(dy.to(dev), w.to(dev), None, route, False, _lib.HEXA_W_OUT_IN, gelu_bwd_of=y1)
    second = v * torch.exp(-0.5 * v * v) / math.sqrt(2.0 * math.pi)
    want = tail + second
    bound = rounding * want.abs() + tiny + 0.5 * 3 * unit + 32 * unit * second.abs()
    assert ((dy1[0].double().cpu() - want[:, None]).abs() <= bound[:, None]).all()
