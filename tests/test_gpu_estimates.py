"""What a context learns from its calls (how many open ends and key positions to expect) does not
follow it to other calls: a small deeply nested document does not make a later large flat one allocate
more than a new context does, and a dense one does not move later sparse ones off their kernels for
good."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _bundle(g):
    from alpacc_amd.gen.tables import generate
    return generate(os.path.join(GRAMMARS, g + ".alp"))


class _Device:
    """A document on the device with room for its tree."""

    def __init__(self, ctx, docs):
        from alpacc_amd.runtime import DeviceBuffer
        data = np.frombuffer(b"".join(docs), dtype=np.uint8)
        self.ctx, self.n = ctx, data.shape[0]
        self.lengths = np.array([len(d) for d in docs], dtype=np.uint64)
        self.offsets = np.concatenate([[0], np.cumsum(self.lengths)[:-1]]).astype(np.uint64)
        self.cap = 4 * self.n + 4096
        self.bufs = [DeviceBuffer(k * self.cap, ctx.lib) for k in (1, 4, 4, 8)]
        self.bufs[0].upload(data)

    def parse(self):
        rc, count = self.ctx.parse_device(self.bufs[0].ptr, self.n, *(b.ptr for b in self.bufs[1:]),
                                          self.cap)
        assert rc == 1 and count
        return self.ctx.lib.alpacc_last_launch_count(self.ctx.handle)

    def parse_batch(self):
        rc, total, res = self.ctx.parse_batch_device(self.bufs[0].ptr, self.offsets, self.lengths,
                                                     *(b.ptr for b in self.bufs[1:]), self.cap)
        assert rc == 1 and (res["status"] == 1).all()
        return self.ctx.lib.alpacc_last_launch_count(self.ctx.handle)


def _held(bundle, calls, tune=None):
    """Device bytes of a context after calls [(batched, documents)]."""
    from alpacc_amd.runtime import Context
    ctx = Context(bundle)
    try:
        for batched, docs in calls:
            d = _Device(ctx, docs)
            d.parse_batch() if batched else d.parse()
            if tune:
                ctx.set_tuning(**tune)
        return int(ctx.lib.alpacc_device_bytes(ctx.handle))
    finally:
        ctx.close()


@pytest.mark.parametrize("tune", [None, {"lex_blocks_per_cu": 2}], ids=["", "tuned"])
@pytest.mark.parametrize("batched", [False, True], ids=["single", "batch"])
def test_nested_request_then_large_document(batched, tune):
    from alpacc_amd import datagen
    b = _bundle("json")
    deep = b"[" * 300 + b"1" + b"]" * 299 + b"]"
    flat = datagen.json_doc(16 * MIB, seed=3).tobytes()
    new = _held(b, [(batched, [flat])])
    after = _held(b, [(batched, [deep]), (batched, [deep, deep] if batched else [deep]),
                      (batched, [flat])], tune)
    assert after <= new + MIB, (new, after)


def test_exact_need_is_kept():
    """A call that needed more than its estimate does not run again the next time."""
    from alpacc_amd.runtime import Context
    b = _bundle("json")
    docs = [b"[" * k + b"1" + b"]" * k for k in (300, 40_000)]
    ctx = Context(b)
    try:
        for d in docs:
            dev = _Device(ctx, [d])
            first, second = dev.parse(), dev.parse()
            assert first > second, len(d)  # the tree kernels ran twice
            assert dev.parse() == second
        assert _Device(ctx, docs).parse_batch() == _Device(ctx, docs).parse_batch()
        assert ctx.tuning()["brackets_per_kib"] > 256
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [4000, 16_000, 60_000])
def test_dense_document_then_sparse_ones(n):
    from alpacc_amd import datagen
    from alpacc_amd.runtime import Context
    b = _bundle("json")
    dense = b"[" + b"7," * 200_000 + b"7]"
    sparse = datagen.json_doc(n, seed=4).tobytes()
    ctx = Context(b)
    try:
        new = _Device(ctx, [sparse]).parse()
    finally:
        ctx.close()
    ctx = Context(b)
    try:
        d = _Device(ctx, [dense])
        d.parse(), d.parse()
        s = _Device(ctx, [sparse])
        counts = [s.parse() for _ in range(12)]
        assert counts[-1] == new, (new, counts)
    finally:
        ctx.close()
