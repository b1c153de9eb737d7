"""Both verdicts at the sizes at which a call takes other kernels: rejected single documents there (by
the lexer, for a missing pair, by their depth, by a bracket), and batches whose large documents are
accepted while a small one of its own is rejected. One scan chunk of the batched lexer is 1024 wave
tiles, 2 MiB."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS
from test_gpu_launch_edges import KIB, MIB, _dense, _same, _sparse

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bundles():
    from alpacc_amd.gen.tables import generate
    from oracle.c import coracle
    out = {}
    for g in ("json", "sexp"):
        b = generate(os.path.join(GRAMMARS, g + ".alp"))
        out[g] = (b, coracle.Oracle(b))
    return out


def _rejected(g, d):
    """Documents of d's length, each rejected at another place."""
    body = d.rstrip(b" ")
    pad = b" " * (len(d) - len(body))
    out = {"lexer, first byte": b"\x01" + d[1:], "lexer, last byte": d[:-1] + b"\x01",
           "depth, last bracket gone": body[:-1] + b" " + pad}
    if g == "json":
        wrong = {b"]": b"}", b"}": b"]"}[body[-1:]]
        out["bracket"] = body[:-1] + wrong + pad
        out["pair"] = body[:-1] + b":" + pad
    else:
        k = body.rindex(b"(")
        out["depth, below zero"] = body[:k] + b")" + body[k + 1:] + pad
    return out


@pytest.mark.parametrize("g", ["json", "sexp"])
@pytest.mark.parametrize("edge", [8 * KIB, 16 * KIB, 32 * KIB, 64 * KIB, 2 * MIB, 16 * MIB])
def test_rejected_single_documents(bundles, g, edge):
    from alpacc_amd.runtime import Context
    b, orc = bundles[g]
    ctx = Context(b)
    try:
        for make in (_sparse, _dense):
            for d in (make(g, edge), make(g, edge + 1)):
                rejected = 0
                for where, x in _rejected(g, d).items():
                    want = orc.parse(x)
                    print(g, make.__name__, len(x), where, want is None, flush=True)
                    rejected += want is None
                    _same(ctx.parse_int(x), want, (g, len(x), where))
                    _same(ctx.lex_int(x), orc.lex(x), (g, len(x), where))
                assert rejected >= 3
                _same(ctx.parse_int(d), orc.parse(d), (g, len(d)))
    finally:
        ctx.close()


@pytest.mark.parametrize("g", ["json", "sexp"])
@pytest.mark.parametrize("sizes", [
    [40] * 1023, [40] * 1024, [40] * 1025, [256 * KIB, 9], [9, 256 * KIB + 1], [2 * MIB, 9],
    [9, 2 * MIB + 1, 9], [2 * MIB + 1, 2 * MIB]], ids=lambda s: f"{len(s)}x{max(s)}")
def test_accepted_large_documents_in_batches(bundles, g, sizes):
    from alpacc_amd.runtime import Context
    b, orc = bundles[g]
    bad = b"[1,2" if g == "json" else b"(a b"
    for make in (_sparse, _dense):
        docs = [make(g, n) if n > 100 else _dense(g, n) for n in sizes]
        want = {d: (orc.lex(d), orc.parse(d)) for d in {*docs, bad}}
        assert all(want[d][1] is not None for d in docs) and want[bad][1] is None
        docs.insert(len(docs) // 2, bad)
        ctx = Context(b)
        try:
            for call in range(2):
                print(g, make.__name__, len(docs), max(sizes), call, flush=True)
                lex, tree = ctx.lex_int_batch(docs), ctx.parse_int_batch(docs)
                assert sum(t is None for t in tree) == 1
                for i, d in enumerate(docs):
                    _same(lex[i], want[d][0], (i, call))
                    _same(tree[i], want[d][1], (i, call))
        finally:
            ctx.close()


@pytest.mark.parametrize("g", ["json", "sexp"])
def test_graph_replay_with_lengths_exchanged(bundles, g):
    """Batches of the same lengths in another order have the same plan: a replayed graph takes the
    descriptors of the call."""
    from alpacc_amd.runtime import Context
    b, orc = bundles[g]
    sizes = [9_000, 300, 40_000, 2_100, 700]
    docs = [_sparse(g, n) for n in sizes]
    want = {d: orc.parse(d) for d in docs}
    assert all(w is not None for w in want.values())
    ctx = Context(b)
    try:
        ctx.set_tuning(graph_mode=2)
        for call in range(8):
            order = np.random.default_rng(call).permutation(len(docs))
            batch = [docs[int(i)] for i in order]
            for t, d in zip(ctx.parse_int_batch(batch), batch):
                _same(t, want[d], call)
        assert ctx.tuning()["graph_launches"] == 8
        assert ctx.tuning()["graph_captures"] < 8
    finally:
        ctx.close()
