"""Rules that the kernels' sources keep and that no run on a GPU reliably shows when they are broken."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "kafka_llm_service_amd" / "ops" / "csrc"

#: loads that a kernel's own loop waits for by count, asm statement by asm statement: (file, function)
COUNTED = {("attention.hip", "asm_load16"), ("attention.hip", "asm_load4")}


def asm_statements(src: str):
    """(where it starts, its text up to the closing parenthesis) of every inline-asm statement."""
    for m in re.finditer(r"asm volatile\(", src):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = src[i]
            if c == '"' and src[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += {"(": 1, ")": -1}.get(c, 0)
            i += 1
        yield m.start(), src[m.start():i]


@pytest.mark.parametrize("path", sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")), ids=lambda p: p.name)
def test_asm_loads_wait_in_their_own_statement(path):
    """The compiler takes an asm statement's outputs as written at its end: it may copy, spill or reuse the registers of a load
    that is still on its way. So a statement that loads into registers also waits (LDS-DMA has no register to write)."""
    src = path.read_text()
    for start, text in asm_statements(src):
        load = re.search(r"\b(?:global|flat|buffer|scratch)_load_(?!lds)\w+ %\d|\bds_read\w* %\d|\bs_load\w* %\d", text)
        if load and "s_waitcnt" not in text[load.start():]:
            owner = re.findall(r"(\w+)\([^()]*\) \{", src[:start])
            assert (path.name, owner[-1] if owner else "") in COUNTED, (path.name, text)
