"""Cross-lane reads of the device code stand where every lane of the group or
wave is active: not behind `&&`, `||` or `?:`, where a lane whose condition
is false is off, and a read of it gives zero.  (A template parameter as the
condition is the same for all lanes.  read_lane reads lanes that are off.)"""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "meerkat_amd",
                    "csrc")
SHUFFLE = re.compile(r"\b(group_read|__shfl\w*|ballot|__ballot|__builtin_amdgcn_ds_\w*permute)\s*\(")
UNIFORM = re.compile(r"\bMAP\s*(&&|\?)")


def behind_a_condition(text):
    """Statements of `text` with a cross-lane read after a short circuit."""
    text = re.sub(r"//[^\n]*", "", text)
    found = []
    for st in re.split(r"[;{}]", UNIFORM.sub("MAP +", text)):
        for m in SHUFFLE.finditer(st):
            # operators of the expression that the read belongs to
            if re.search(r"&&|\|\||\?", st[:m.start()]):
                # `if (a && b) x = read(...)`: the read is not in the condition
                head = re.match(r"\s*(else\s+)?(if|for|while)\s*\(", st)
                if head:
                    depth, i = 1, head.end()
                    while depth and i < len(st):
                        depth += {"(": 1, ")": -1}.get(st[i], 0)
                        i += 1
                    if i <= m.start() and not re.search(r"&&|\|\||\?", st[i:m.start()]):
                        continue
                found.append(" ".join(st.split()))
    return found


def test_the_check_itself():
    assert behind_a_condition("t |= a && i < gl && group_read(b, i) == b;")
    assert behind_a_condition("x = p ? __shfl(v, 3, 64) : 0;")
    assert not behind_a_condition("const uint32_t o = group_read(b, i); t |= a && o == b;")
    assert not behind_a_condition("w = MAP ? __shfl_down(v, 1, 64) : 0u; // a && ballot(x)")


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))),
                         ids=os.path.basename)
def test_no_cross_lane_read_behind_a_condition(path):
    with open(path) as f:
        assert behind_a_condition(f.read()) == []
