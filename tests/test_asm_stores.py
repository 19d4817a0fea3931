"""Inline-assembly stores of more than 8 bytes and the wait states behind them."""
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
