"""A function of the device code that takes restrict pointers holds no work-group barrier: inside it the compiler may take the
barrier for one that cannot touch what those pointers reach, and move their reads and writes past it."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "c0ven_amd", "csrc")
BARRIER = re.compile(r"\b(unit_barrier|__syncthreads|__builtin_amdgcn_s_barrier)\s*\(")


def closing(text, at, opening, close):
    """The index past the bracket that closes the one at `at`."""
    depth = 0
    for i in range(at, len(text)):
        depth += (text[i] == opening) - (text[i] == close)
        if depth == 0:
            return i + 1
    raise AssertionError("unbalanced")


def restrict_functions(text):
    """(line, body) of each function or lambda with a restrict parameter."""
    text = re.sub(r"//[^\n]*", lambda m: " " * len(m.group()), text)
    seen = set()
    for m in re.finditer(r"__restrict__", text):
        depth, i = 0, m.start()  # back to the parameter list's opening bracket
        while depth >= 0:
            i -= 1
            depth += (text[i] == ")") - (text[i] == "(")
        if i in seen:
            continue
        seen.add(i)
        body = text.index("{", closing(text, i, "(", ")"))
        yield text.count("\n", 0, i) + 1, text[body:closing(text, body, "{", "}")]


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))),
                         ids=os.path.basename)
def test_no_barrier_under_restrict(path):
    with open(path) as f:
        text = f.read()
    for line, body in restrict_functions(text):
        assert not BARRIER.search(body), "%s:%d" % (os.path.basename(path), line)


def test_the_check_finds_one():
    text = "auto f = [&](const int *__restrict__ a, int b) { if (b) { unit_barrier(); } return a[0]; };"
    [(line, body)] = restrict_functions(text)
    assert line == 1 and BARRIER.search(body)
