"""A document that closes more brackets than it opens, between others in a batch: the others' results
are those of the C restatement, and matching the brackets does not search the documents before it."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", ["json", "sexp"])
def test_closing_brackets_end_at_their_document(g):
    from alpacc_amd import datagen
    from alpacc_amd.gen.tables import generate
    from alpacc_amd.runtime import Context
    from oracle.c import coracle
    b = generate(os.path.join(GRAMMARS, g + ".alp"))
    orc = coracle.Oracle(b)
    op, cl = (b"[", b"]") if g == "json" else (b"(", b")")
    n = 1 << 20
    small = [getattr(datagen, g + "_doc")(k, seed=k).tobytes() for k in (300, 5_000, 90_000)]
    deep = op * 700 + (b"1" if g == "json" else b"") + cl * 700
    closing = [cl * n, op * 900 + cl * (n // 2)]
    want = {d: orc.parse(d) for d in small + [deep]}
    assert all(w is not None for w in want.values())
    assert all(orc.parse(d[:4096]) is None for d in closing)

    def run(ctx, docs):
        ctx.profile(True)
        got = ctx.parse_int_batch(docs)
        for d, t in zip(docs, got):
            assert (t is None) == (d not in want)
            for x, y in zip(t or (), want.get(d) or ()):
                assert np.array_equal(np.asarray(x).reshape(-1), np.asarray(y).reshape(-1))
        return ctx.read_profile()["link_tiles"][0]

    ctx = Context(b)
    try:
        mixed = [small[0], closing[0], small[1], deep, closing[1], small[2], deep]
        ordinary = getattr(datagen, g + "_doc")(n, seed=1).tobytes()
        want[ordinary] = orc.parse(ordinary)
        even = [ordinary if d in closing else d for d in mixed]
        times = [min(run(ctx, docs) for _ in range(3)) for docs in (even, mixed)]
        print(g, times)
        # searched through the documents before, the closing brackets take 24 ms per MiB here, against
        # 0.01 ms of the ordinary documents and 0.02 now
        assert times[1] < 20 * times[0] + 1.0
    finally:
        ctx.close()
