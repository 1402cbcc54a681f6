"""Every object of the kernel library names the headers that its source includes, straight or by way of others, among its prerequisites: an
edit of a header leaves no object of the same library behind."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm_simple_amd", "csrc")


def included(path, seen):
    for name in re.findall(r'#include "([^"]+)"', open(path).read()):
        header = os.path.normpath(os.path.join(os.path.dirname(path), name))
        if header not in seen:
            seen.add(header)
            included(header, seen)
    return seen


def rules():
    text = open(os.path.join(CSRC, "Makefile")).read().replace("\\\n", " ")
    found = {}
    for targets, needs in re.findall(r"^(\S+\.o(?: \S+\.o)*): (?!HIPFLAGS)(.*)$", text, re.M):
        for target in targets.split():
            found.setdefault(target, []).extend(needs.split())
    return found


@pytest.mark.parametrize("target", sorted(rules()))
def test_prerequisites(target):
    needs = rules()[target]
    assert len(needs) == len(set(needs)), needs
    source = next(n for n in needs if n.endswith(".hip"))
    assert included(os.path.join(CSRC, source), set()) <= {os.path.normpath(os.path.join(CSRC, n)) for n in needs}
