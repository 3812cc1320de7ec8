"""What the compiler does not do for inline assembly, held against the HIP sources."""

from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "pyre_amd" / "csrc"


def test_loads_into_lds_wait_for_m0():
    """A load that goes straight into LDS takes its place there from m0 and needs a wait state behind a scalar write of it: the
    compiler puts one behind its own writes, but none between the instructions of an inline block."""
    blocks = [(f.name, text) for f in sorted(CSRC.glob("*.h*")) for text in re.findall(r'asm volatile\("([^"]*)"', f.read_text())]
    loads = [(name, text) for name, text in blocks if "_lds_" in text]
    assert len(loads) >= 6
    for name, text in loads:
        lines = [x.strip() for x in text.split("\\n\\t")]
        at = next(i for i, x in enumerate(lines) if "_lds_" in x)
        writes = [i for i, x in enumerate(lines[:at]) if re.match(r"s_\w+ m0\b", x)]
        assert writes, (name, text)  # m0 is written where it is used
        assert any(x.startswith("s_nop") for x in lines[writes[-1] + 1:at]), (name, text)
