"""Host arrays that a call returns are the caller's: at the sizes where downloads change their way
(staging, lent pinned blocks, sliced copies) they equal the C restatement's, keep their values through
later calls and after the context is closed, and blocks beyond the lending bound are copies."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu


def _tree(r):
    return tuple(np.asarray(x).reshape(-1).copy() for x in r)


@pytest.mark.parametrize("total", [64 << 20, 1 << 20, 0])
def test_arrays_stay_the_callers(total, monkeypatch):
    from alpacc_amd import datagen, runtime
    from alpacc_amd.gen.tables import generate
    from oracle.c import coracle
    monkeypatch.setattr(runtime, "LEASE_TOTAL", total)
    b = generate(os.path.join(GRAMMARS, "sexp.alp"))
    orc = coracle.Oracle(b)
    ctx = runtime.Context(b)
    kept = []
    try:
        # 7.7 bytes of tree per input byte: 1 KB .. 30 MB of arrays
        for i, n in enumerate((100, 17_000, 17_100, 40_000, 140_000, 600_000, 2_200_000, 4_000_000)):
            doc = datagen.sexp_doc(n, seed=n)
            kept.append((ctx.parse_int(doc), _tree(orc.parse(doc))))
            if i % 3 == 2:  # some results are dropped: their blocks are lent again
                got, want = kept.pop(0)
                assert all(np.array_equal(g.reshape(-1), w) for g, w in zip(got, want))
                del got
        assert ctx._lent.allocated <= total
        batch = [datagen.sexp_doc(n, seed=n + 1) for n in (50, 9_000, 90_000)]
        kept += [(t, _tree(orc.parse(d))) for t, d in zip(ctx.parse_int_batch(batch), batch)]
    finally:
        ctx.close()
    for got, want in kept:
        for g, w in zip(got, want):
            assert np.array_equal(g.reshape(-1), w)
            g[...] = 0  # writable, and nobody else's
