"""Inline-assembly stores of more than 8 bytes and the wait states behind them; asynchronous copies and the waits in front of the barriers
that publish them."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "hexa-moe_amd" / "csrc"


def test_wide_stores_are_followed_by_wait_states():
    """gfx950 reads a wide store's data for two wait states after its issue: a vector instruction that overwrites the registers
    must not follow closer.  The compiler sees to that for stores of its own only."""
    found = 0
    for path in sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.h"))):
        for text in re.findall(r'asm[^;"]*"([^"]*)"', path.read_text()):
            for store in re.finditer(r"(global|flat|buffer)_store_(dwordx[34]|b96|b128)", text):
                found += 1
                assert re.match(r"[^\\]*\\n\\ts_nop [1-9]", text[store.end():]), (path.name, text)
    assert found >= 4


def test_copies_are_awaited_before_the_barrier_behind_them():
    """A barrier does not wait for asynchronous copies into LDS.  In the gate's kernel, which issues them and reads them in one block, a
    wait of its own stands between."""
    text = re.sub(r"//[^\n]*", "", (CSRC / "router.hip").read_text())
    copies = list(re.finditer(r"\bdma16\(|global_load_lds\(", text))
    assert copies
    for c in copies:
        barrier = re.compile(r"__syncthreads\(\)|barrier_nofence\(\)").search(text, c.end())
        assert barrier and "wait_vmcnt<0>()" in text[c.end():barrier.start()], text[c.start():barrier.start()]
