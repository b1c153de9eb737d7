"""Documents on both sides of every size at which a call takes other kernels, against the C
restatement: the one-workgroup lexer, the start states a lex_emit workgroup finds itself, the look-back
groups, the fused key scan and tree link, the one-workgroup tile scan, and the batched call's
document limits. Each size runs with few tokens and with one token per byte (where a fresh context's
estimate of the position tiles is four times too small), twice on one context."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20
DENSE = {"json": (b"[", b"7,", b"7]"), "sexp": (b"(", b"()", b")")}


def _dense(g, n):
    head, body, tail = DENSE[g]
    d = head + body * ((n - len(head) - len(tail)) // len(body)) + tail
    return d + b" " * (n - len(d))


def _sparse(g, n):
    from alpacc_amd import datagen
    d = getattr(datagen, g + "_doc")(n - n // 64 - 8, seed=n).tobytes()[:n]
    return d + b" " * (n - len(d))


def _rows(r):
    return None if r is None else [np.asarray(x).reshape(-1) for x in r]


def _same(got, want, what):
    got, want = _rows(got), _rows(want)
    assert (got is None) == (want is None), what
    for a, b in zip(got or [], want or []):
        assert np.array_equal(a, b), what


@pytest.fixture(scope="module")
def bundles():
    from alpacc_amd.gen.tables import generate
    from oracle.c import coracle
    out = {}
    for g in ("json", "sexp"):
        b = generate(os.path.join(GRAMMARS, g + ".alp"))
        out[g] = (b, coracle.Oracle(b))
    return out


@pytest.mark.parametrize("g", ["json", "sexp"])
@pytest.mark.parametrize("edge", [8 * KIB, 16 * KIB, 32 * KIB, 64 * KIB, 2 * MIB, 8 * MIB, 16 * MIB])
def test_single_document(bundles, g, edge):
    from alpacc_amd.runtime import Context
    b, orc = bundles[g]
    around = (-2, -1, 0, 1) if edge < MIB else (0, 1)
    for make in (_sparse, _dense):
        ctx = Context(b)
        try:
            for d in (make(g, edge + i) for i in around):
                assert len(d) - edge in around
                tokens, tree = orc.lex(d), orc.parse(d)
                assert tree is not None
                for call in range(2 if edge < MIB else 1):
                    what = (g, make.__name__, len(d), call)
                    print(*what, flush=True)
                    _same(ctx.parse_int(d), tree, what)
                    _same(ctx.lex_int(d), tokens, what)
        finally:
            ctx.close()


@pytest.mark.parametrize("g", ["json", "sexp"])
@pytest.mark.parametrize("sizes", [
    [40] * 1023, [40] * 1024, [40] * 1025,               # descriptors read in place or copied
    [256 * KIB, 9], [9, 256 * KIB + 1],                  # tile map by pb_setup or pb_tile_docs
    [512 * KIB, 9], [9, 512 * KIB + 1, 9],               # one scan chunk per document or more
    [8 * MIB - 64, 9], [2 * MIB + 1] * 4 + [9],          # one workgroup's tile scan or three kernels
], ids=lambda s: f"{len(s)}x{max(s)}")
def test_batch(bundles, g, sizes):
    from alpacc_amd.runtime import Context
    b, orc = bundles[g]
    for make in (_sparse, _dense):
        docs = [make(g, n) if n > 100 else _dense(g, n) for n in sizes]
        docs[len(docs) // 2] = docs[len(docs) // 2][:-2] + b"))"  # rejected (sexp: unbalanced)
        want = {d: (orc.lex(d), orc.parse(d)) for d in set(docs)}
        ctx = Context(b)
        try:
            for call in range(2):
                print(g, make.__name__, len(docs), max(sizes), call, flush=True)
                lex, tree = ctx.lex_int_batch(docs), ctx.parse_int_batch(docs)
                for i, d in enumerate(docs):
                    _same(lex[i], want[d][0], (i, call))
                    _same(tree[i], want[d][1], (i, call))
        finally:
            ctx.close()
