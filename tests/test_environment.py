"""The library reads its environment variables while a context, an ensemble or
an adjoint is created and never afterwards: a variable changed later, by
another thread perhaps, neither changes nor races with a run.

Read off the sources: every getenv stands in a function named *_create, or in
one that only such functions (and each other) call.
"""
import os
import re

from conftest import ROOT

CSRC = os.path.join(ROOT, "fdmap_github_amd", "csrc")


def functions():
    """(name, body) of every function at file or namespace level"""
    out = []
    for f in sorted(os.listdir(CSRC)):
        if f.endswith((".hip", ".hpp")):
            text = open(os.path.join(CSRC, f)).read()
            text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
            for m in re.finditer(r"^[A-Za-z_][^\n;{}#]*?(\w+)\([^;{}]*\)\s*\{\n(.*?)^\}", text, flags=re.S | re.M):
                out.append((m.group(1), m.group(2)))
    return out


def test_environment_is_read_at_creation():
    funcs = functions()
    assert sum(b.count("getenv(") for _, b in funcs) == sum(
        re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, f)).read()).count("getenv(")
        for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp")))
    readers = {n for n, b in funcs if "getenv(" in b}
    assert "fdm_create" in readers
    todo, seen = set(readers), set()
    while todo:
        r = todo.pop()
        seen.add(r)
        if r.endswith("_create"):
            continue
        callers = {n for n, b in funcs if n != r and re.search(rf"\b{r}\(", b)}
        # an entry point other than a creation has no callers here
        assert callers, f"{r} reaches getenv"
        todo |= callers - seen
