"""CPU: every object's rule in the Makefile names all headers of this repository that its source includes, so that none is left as it was when one of them changes."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-candle_amd", "csrc")


def includes(path, seen):
    for name in re.findall(r'^#include "([^"]+)"', open(path).read(), re.M):
        at = os.path.normpath(os.path.join(os.path.dirname(path), name))
        if at not in seen:
            seen.add(at)
            includes(at, seen)
    return seen


def test_rules_name_their_headers():
    rules = re.findall(r"^(\w+)\.o: (.+)$", open(os.path.join(CSRC, "Makefile")).read(), re.M)
    assert len(rules) > 15
    for name, names in rules:
        names = [os.path.normpath(os.path.join(CSRC, n)) for n in names.split()]
        missing = includes(names[0], set()) - set(names)
        assert not missing, (name, sorted(os.path.basename(m) for m in missing))
