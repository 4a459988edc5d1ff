"""Buffer accesses of the HIP sources, read on the CPU: none carries a step in its scalar
offset.  Rows past S are zeroed by the range check of a load's buffer resource; the check is
documented for the per-lane and immediate offsets only, so a step in the scalar offset could
read memory behind the tensor."""

from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "tiledattention_amd" / "csrc"
# builtin -> index of its scalar-offset argument
ACCESSES = {
    "__builtin_amdgcn_raw_ptr_buffer_load_lds": 4,
    "__builtin_amdgcn_raw_buffer_load_b128": 2,
    "__builtin_amdgcn_raw_buffer_load_b32": 2,
    "__builtin_amdgcn_raw_buffer_store_b128": 3,
    "__builtin_amdgcn_raw_buffer_store_b32": 3,
}


def _calls(text, name):
    """The top-level arguments of every call of ``name``."""
    for m in re.finditer(re.escape(name) + r"\(", text):
        depth, args, cur = 1, [], ""
        for ch in text[m.end():]:
            depth += ch in "([{"
            depth -= ch in ")]}"
            if depth == 0:
                break
            if ch == "," and depth == 1:
                args.append(cur.strip())
                cur = ""
            else:
                cur += ch
        yield args + [cur.strip()]


def test_scalar_offset_is_zero():
    seen = 0
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        text = re.sub(r"//[^\n]*", "", path.read_text())
        for name, index in ACCESSES.items():
            for args in _calls(text, name):
                assert args[index] == "0", f"{path.name}: {name} scalar offset {args[index]}"
                seen += 1
        others = set(re.findall(r"__builtin_amdgcn_(?:raw|struct)\w*buffer\w*", text)) - set(ACCESSES)
        assert not others, (path.name, others)
    assert seen >= 12
