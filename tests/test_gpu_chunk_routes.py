"""The chunked lexer's two ways to its input, chunks laid end to end (shorter than 4096 bytes) and
loads that map to the original string: both sides of that size, documents that start anywhere in a
16-byte word, chunk ends at every place of a lane's 32 bytes, against the C restatement."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["arithmetic", "sexp", "json"])
def case(request):
    from alpacc_amd import datagen
    from alpacc_amd.gen.tables import generate
    from alpacc_amd.runtime import Context, DeviceBuffer
    from oracle.c import coracle
    g = request.param
    b = generate(os.path.join(GRAMMARS, g + ".alp"))
    gen = {"json": datagen.json_doc, "arithmetic": datagen.arith_doc, "sexp": datagen.sexp_doc}[g]
    ctx = Context(b)
    yield g, gen, ctx, coracle.Oracle(b), DeviceBuffer
    ctx.close()


def _lex(ctx, DeviceBuffer, doc, chunk, offset):
    n = len(doc)
    cap = n + -(-n // min(chunk, n)) + 1
    bufs = [DeviceBuffer(n + 64, ctx.lib)] + [DeviceBuffer(k * cap, ctx.lib) for k in (4, 8, 8)]
    # other documents' bytes around it
    bufs[0].upload(np.frombuffer(doc[-offset:] + doc + doc[:16] if offset else doc + doc[:16],
                                 dtype=np.uint8))
    rc, nt = ctx.lex_chunked_device(bufs[0].ptr + offset, n, chunk, bufs[1].ptr, bufs[2].ptr,
                                    bufs[3].ptr, cap)
    launches = ctx.lib.alpacc_last_launch_count(ctx.handle)
    out = None if rc != 1 else [b.download(dt, nt) for b, dt in
                                zip(bufs[1:], (np.uint32, np.uint64, np.uint64))]
    for b in bufs:
        b.free()
    return out, launches


def test_both_sides_of_the_rule(case):
    g, gen, ctx, orc, buf = case
    accepted = 0
    for n in (12_301, 70_001, 600_000):
        doc = gen(n, seed=n).tobytes()
        for k, chunk in enumerate((1, 31, 32, 33, 63, 1000, 2047, 4095, 4096, 4097, 4127, 4128, 8191,
                                   11_111, n - 1, n, 1 << 24)):
            offset = (k * 5 + n) % 16
            print(g, n, chunk, offset, flush=True)
            want = orc.lex(doc, chunk=chunk, wide=True)
            got, launches = _lex(ctx, buf, doc, chunk, offset)
            assert (got is None) == (want is None), (n, chunk, offset)
            for x, y in zip(got or (), want or ()):
                assert np.array_equal(x, np.asarray(y)), (n, chunk, offset)
            accepted += got is not None
            # the copy of short chunks, lex_reduce, lex_emit, the chunks' last tokens; a document of
            # one chunk is never laid out
            assert launches == (4 if chunk < 4096 and chunk < n else 3), (n, chunk)
    assert accepted >= 6


def test_every_place_in_a_lane(case):
    g, gen, ctx, orc, buf = case
    doc = gen(9_000, seed=5).tobytes()
    for k in range(34):
        chunk, offset = 4096 + k, k % 16
        want = orc.lex(doc, chunk=chunk, wide=True)
        got, _ = _lex(ctx, buf, doc, chunk, offset)
        assert (got is None) == (want is None), (chunk, offset)
        for x, y in zip(got or (), want or ()):
            assert np.array_equal(x, np.asarray(y)), (chunk, offset)
