"""The header's list of versions names the entry points that came after 210, and the version moved with the last of them."""
import os
import re

from fsa_hip import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_new_entry_points_are_in_the_list():
    text = open(os.path.join(ROOT, "include", "fsa_hip.h")).read()
    history = re.search(r"/\* Library version.*?\*/", text, flags=re.S).group(0)
    last = [int(v) for v in re.findall(r"^ \*   (\d+):", history, flags=re.M)][-1]
    assert _lib.load().fsa_version() == last >= 230
    named = [re.compile(n.replace("*", ".*") + "$") for n in re.findall(r"fsa_[a-z0-9_]+\*?", history)]
    new = [n for n in _lib.SIGNATURES if "direct" in n or "tiles" in n or "layer" in n or n == "fsa_matmul"]
    older = {"fsa_build_tiles", "fsa_max_tiles"}
    for n in set(new) - older:
        assert any(p.match(n) for p in named), n
