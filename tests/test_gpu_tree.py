"""GPU parity of the tree parser (parse_keys_tree, parse_tree, link_tiles) with the C restatement, at
the sizes where its tiles (256 key positions per wavefront, 4 per lane) and the groups of 64 tiles
end, on nesting that runs through many tiles, in both its forms (entries as rows, entries looped
over), and that the grammars and token streams it does not take go to the element-level kernels."""
import itertools
import os

import numpy as np
import pytest

from conftest import GRAMMARS
from tree_tables import form

pytestmark = pytest.mark.gpu

HEAD = "params {\n  lookback = 1.\n  lookahead = 1.\n}\nignore = /\\s/.\n"
LOOPS = HEAD + 'S -> "a" "b" S "c" "d" "e" "f" | "x".\n'
ELEMENTS = HEAD + 'S -> "a" S "b" "c" "d" "e" "f" "g" "h" "i" "j" "k" | "x".\n'


def _bundle(name):
    from alpacc_amd.gen.tables import generate
    if name == "loops":
        return generate(LOOPS)
    if name == "elements":
        return generate(ELEMENTS)
    return generate(os.path.join(GRAMMARS, name + ".alp"))


def _doc(name, tokens):
    """A flat document of about `tokens` tokens."""
    if name == "json":
        return ("[" + ",".join(["7"] * max(1, (tokens - 1) // 2)) + "]").encode()
    if name == "sexp":
        return ("(" + " ".join(["a"] * max(0, tokens - 2)) + ")").encode()
    if name == "arithmetic":
        return "+".join(["a"] * max(1, (tokens + 1) // 2)).encode()
    depth = max(0, (tokens - 1) // (7 if name == "loops" else 11))
    tail = "cdef" if name == "loops" else "bcdefghijk"
    return (("ab" if name == "loops" else "a") * depth + "x" + tail * depth).encode()


def _nested(name, depth):
    if name == "json":
        return ("[" * depth + "1" + "]" * depth).encode()
    if name == "sexp":
        return ("(" * depth + "a" + ") b" * (depth - 1) + ")").encode()
    if name == "arithmetic":
        return ("(" * depth + "a" + ")*b" * depth).encode()
    return _doc(name, 7 * depth)


def _tree(r):
    if r is None:
        return None
    return tuple(np.asarray(x).reshape(-1) for x in r)


def _same(got, want):
    if got is None or want is None:
        return got is None and want is None
    return all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("name", ["json", "sexp", "arithmetic", "loops", "elements"])
def test_tile_edges(name):
    from alpacc_amd.runtime import Context
    from oracle.c import coracle
    b = _bundle(name)
    assert form(b.parser) == {"loops": "loops", "elements": "elements"}.get(name, "rows")
    orc = coracle.Oracle(b)
    docs = []
    for positions in (3, 4, 5, 8, 255, 256, 257, 260, 511, 512, 513, 1024, 1025, 16383, 16384, 16385,
                      16640, 32768, 40000):
        docs += [_doc(name, positions - 2 + d) for d in (0, 1)]
    docs += [_nested(name, d) for d in (2, 63, 64, 65, 300, 9000)]
    docs += [docs[-1][:-1], docs[-1] + docs[-1][-1:], docs[20][:len(docs[20]) // 2] + docs[20]]
    ctx = Context(b)
    try:
        ctx.profile(True)
        want = [_tree(orc.parse(d)) for d in docs]
        assert sum(w is not None for w in want) >= 20
        for i, d in enumerate(docs):
            assert _same(_tree(ctx.parse_int(d)), want[i]), (name, i, len(d))
        stages = {k for k, v in ctx.read_profile().items() if v[1]}
        assert ("parse_expand" if name == "elements" else "parse_tree") in stages, stages
        got = ctx.parse_int_batch(docs)
        for i in range(len(docs)):
            assert _same(_tree(got[i]), want[i]), (name, i, "batch")
    finally:
        ctx.close()


@pytest.mark.parametrize("name,max_len", [("llp01", 5), ("sexp", 4)])
def test_end_terminals_among_tokens(name, max_len):
    """Token streams that hold the start or end terminal: verdicts and nodes of the C restatement,
    by the element-level kernels."""
    from alpacc_amd.runtime import Context
    from oracle.c import coracle
    b = _bundle(name)
    orc = coracle.Oracle(b)
    px = b.parser
    ctx = Context(b)
    try:
        ctx.profile(True)
        accepted = 0
        for n in range(1, max_len + 1):
            for c in itertools.product(range(px.num_terminals), repeat=n):
                ends = px.start_terminal in c or px.end_terminal in c
                if not ends:
                    continue
                kinds = np.array(c, dtype=np.uint32)
                t = np.arange(n, dtype=np.uint32)
                want = _tree(orc.parse_tokens(kinds, t.astype(np.int64), t.astype(np.int64) + 1))
                got = _tree(ctx.parse_tokens(kinds, t, t + 1))
                assert (got is None) == (want is None), c
                if want is not None:
                    assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2]), c
                    accepted += 1
        if accepted:
            assert ctx.read_profile()["parse_tree"][1] == 0
    finally:
        ctx.close()
