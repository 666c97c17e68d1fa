"""The name that a plan reports for a kernel is the name of the function it
launches, which a trace shows: every entry of the kernel tables."""
from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "cmtj_amd" / "csrc"


def test_entries_name_the_function_they_launch():
    pairs = []
    for f in sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip")):
        text = f.read_text().replace("\\\n", " ")
        pairs += [(f.name, *p) for p in re.findall(r'&\s*(?:cmtj::)?(k_\w+)<[^"]*?"(k_\w+)<', text)]
    assert len(pairs) >= 20
    assert [p for p in pairs if p[1] != p[2]] == []
