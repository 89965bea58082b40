"""Where the kernels' buffer accesses put their position.  The range check of a raw
buffer load or store covers the offset in the vector operand and leaves out the
scalar one, so a request that may run past its buffer has to carry its whole
position in the vector operand.  Read from the sources (no GPU needed)."""
import os
import re

import pytest

import qlib

FILES = ["k_attn.hip", "k_fattn.hip", "k_gemv_f32.hip"]


def arguments(text, at):
    """The arguments of the call whose parenthesis opens at text[at]."""
    depth, args, start = 0, [], at + 1
    for i in range(at, len(text)):
        if text[i] in "([{":
            depth += 1
        elif text[i] in ")]}":
            depth -= 1
            if depth == 0:
                return args + [text[start:i].strip()]
        elif text[i] == "," and depth == 1:
            args.append(text[start:i].strip())
            start = i + 1
    raise AssertionError("unbalanced call")


@pytest.mark.parametrize("name", FILES)
def test_buffer_positions_are_range_checked(name):
    text = re.sub(r"//.*", "", open(os.path.join(qlib.PKG, "csrc", name)).read())
    calls = [arguments(text, m.end() - 1) for m in re.finditer(r"__builtin_amdgcn_raw_buffer_\w+\(", text)]
    assert calls
    for args in calls:
        assert args[-2] == "0", f"{name}: scalar offset {args[-2]!r} in a call of {args}"
