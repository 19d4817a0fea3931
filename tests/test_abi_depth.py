"""The C ABI's depth descriptor is what version 9 says it is, whatever lies behind it; options travel apart from it."""
import ctypes

import pytest

SIZES = (256, 2, 8, 64, 128, 64)
TYPES = (2, 2, 0, 0, 0, 0, 0, 0)


def _desc(reserved=0):
    from hexa_moe import _lib
    return _lib.DepthDesc(*SIZES, *TYPES, 0, 0.0, 0.0, reserved)


def _bytes(fn, *args):
    from hexa_moe import _lib
    f, b = ctypes.c_int64(), ctypes.c_int64()
    rc = getattr(_lib.load(), fn)(*args, ctypes.byref(f), ctypes.byref(b))
    return rc, f.value, b.value


def test_descriptor_of_version_9():
    from hexa_moe import _lib
    assert ctypes.sizeof(_lib.DepthDesc) == 72
    want = _bytes("hexa_moe_depth_ws_bytes", ctypes.byref(_desc()))
    assert want[0] == 0 and want[1] > 0 and want[2] > 0
    # a caller's struct ends with `reserved`, which nobody had to clear, and is followed by whatever it is followed by
    for fill in (0x01, 0x7f, 0xff):
        memory = (ctypes.c_ubyte * 256)(*[fill] * 256)
        ctypes.memmove(memory, bytes(_desc(reserved=int.from_bytes(bytes([fill] * 4), "little", signed=True))), 72)
        assert _bytes("hexa_moe_depth_ws_bytes", ctypes.cast(memory, ctypes.POINTER(_lib.DepthDesc))) == want


def test_options():
    from hexa_moe import _lib
    d, size = _desc(), ctypes.sizeof(_lib.DepthOpts)
    whole = _bytes("hexa_moe_depth_ws_bytes", ctypes.byref(d))
    ask = lambda *o: _bytes("hexa_moe_depth_part_ws_bytes", ctypes.byref(d), ctypes.byref(_lib.DepthOpts(*o)))      # noqa: E731
    assert _bytes("hexa_moe_depth_part_ws_bytes", ctypes.byref(d), None) == whole
    assert ask(size) == whole
    assert ask(8, 7, 1, 1) == whole         # a caller that knows `part` only: what follows it is not looked at
    assert ask(size, 7, 1, 0)[0] == -2      # wide_y is for top-1
    assert ask(size, -1)[0] == -1
    assert ask(size, 8)[0] == -1            # no such part
    for n in (0, 3, size + 4):
        assert ask(n)[0] == -1


@pytest.mark.parametrize("fn", ["hexa_moe_depth_part_ws_bytes", "hexa_moe_depth_ws_bytes"])
def test_null_descriptor(fn):
    assert _bytes(fn, *([None] * (2 if "part" in fn else 1)))[0] == -1


@pytest.mark.parametrize("no_gate", [0, 1])
@pytest.mark.parametrize("act_dt", [0, 2])
def test_a_part_takes_its_own_scratch(no_gate, act_dt):
    """The backward's pieces: the first layer's half has the gate's and the column sums', each half its weight gradient's."""
    from hexa_moe import _lib
    T, k, E, d, h, size = 32768, 2, 64, 1024, 4096, 2 if act_dt else 4
    desc = _lib.DepthDesc(T, k, E, d, h, d, act_dt, act_dt, *[0] * 6, 0, 0.0, 0.0, 0)
    ask = lambda part: _bytes("hexa_moe_depth_part_ws_bytes", ctypes.byref(desc),      # noqa: E731
                              ctypes.byref(_lib.DepthOpts(ctypes.sizeof(_lib.DepthOpts), part, 0, 0, no_gate)))
    fwd, bwd = zip(*[ask(p)[1:] for p in (1, 2, 4, 7)])
    slots = (k - 1) * T * d * size
    assert fwd[1] <= 256 and fwd[2] == slots and fwd[3] == fwd[2] + (fwd[0] if not no_gate else 0)
    if no_gate:
        assert fwd[0] <= 256
    plan = -(-(4 * E + 32) * 4 // 256) * 256
    assert bwd[1] + bwd[2] - plan == bwd[3]
    ess, partial = 8 * E * d * 4, 128 << 20      # of the weight gradient's scratch at most
    assert bwd[2] <= plan + ess + partial
    colsum = k * (T // 128 + E) * h * 4
    gate = T * E * 4 + T * d * size + (T // 64 + 1) * E * d * 4
    assert bwd[1] <= plan + colsum + partial + slots + (0 if no_gate else gate)


@pytest.mark.parametrize("act_dt,careful", [(0, 1), (2, 0), (2, 1)])
def test_scratch_of_slots_that_are_added_unrounded(act_dt, careful):
    """16-bit tokens with the option: one fp32 result a slot; otherwise a result of the tokens' type for each slot but the first."""
    from hexa_moe import _lib
    T, k, E, d, h = 512, 3, 64, 256, 512
    desc = _lib.DepthDesc(T, k, E, d, h, d, act_dt, act_dt, *[0] * 6, 0, 0.0, 0.0, 0)
    ask = lambda c: _bytes("hexa_moe_depth_part_ws_bytes", ctypes.byref(desc),      # noqa: E731
                           ctypes.byref(_lib.DepthOpts(ctypes.sizeof(_lib.DepthOpts), 7, 0, c, 0)))
    (rc, fwd, bwd), (rc0, fwd0, bwd0) = ask(careful), ask(0)
    more = T * d * (k * 4 - (k - 1) * 2) if careful and act_dt else 0
    assert rc == rc0 == 0 and (fwd - fwd0, bwd - bwd0) == (more, more)


def test_fp32_dx_takes_a_16_bit_one_in_scratch():
    """Top-1, 16-bit tokens, whole 16-byte pieces; anything else is refused and not ignored."""
    from hexa_moe import _lib
    size = ctypes.sizeof(_lib.DepthOpts)

    def ask(T, k, d, act_dt, part=7):
        desc = _lib.DepthDesc(T, k, 8, d, 64, d, act_dt, act_dt, *[0] * 6, 0, 0.0, 0.0, 0)
        return [_bytes("hexa_moe_depth_part_ws_bytes", ctypes.byref(desc), ctypes.byref(_lib.DepthOpts(size, part, 0, 0, 0, 0, wide))) for wide in (0, 1)]

    for part in (1, 2, 3, 4, 7):
        plain, wide = ask(256, 1, 64, 2, part)
        assert wide[:2] == plain[:2] and wide[2] == plain[2] + (256 * 64 * 2 if part & 2 else 0)
    for args in ((256, 2, 64, 2), (256, 1, 64, 0), (3, 1, 4, 2)):
        plain, wide = ask(*args)
        assert plain[0] == 0 and wide[0] == -2


@pytest.mark.parametrize("offset,refused", [(0, False), (16, False), (4, True), (8, True), (15, True)])
def test_fp32_dx_is_16_byte_aligned(offset, refused):
    """It is stored 16 bytes at a time.  (No pointer is read: the workspace is said to be empty, which is looked at next.)"""
    from hexa_moe import _lib
    lib = _lib.load()
    desc, opts = _lib.DepthDesc(256, 1, 8, 64, 64, 64, 2, 2, *[0] * 6, 0, 0.0, 0.0, 0), _lib.DepthOpts(ctypes.sizeof(_lib.DepthOpts), 2, 0, 0, 1, 0, 1)
    any_ = ctypes.c_void_p(4096)
    rc = lib.hexa_moe_depth_part_backward(ctypes.byref(desc), ctypes.byref(opts), any_, None, any_, None, any_, any_, None, None, None, None, any_, None,
                                          any_, any_, ctypes.c_void_p(4096 + offset), None, None, None, None, None, any_, any_, 0, None, 0, None)
    assert rc == -1
    assert (b"aligned" in lib.hexa_last_error()) == refused, lib.hexa_last_error()
