"""The memory that host results are made of: ordinary private memory at every size (a forked child has
it, and nothing but the program writes to it), of each array its own where results are small, and blocks
that are used again only when no array views them, from whichever thread the last one goes."""
import gc
import os
import re
import threading

import numpy as np
import pytest

from conftest import GRAMMARS


def _flags(addr):
    """The kernel's flags of the mapping that holds addr."""
    inside = False
    with open("/proc/self/smaps") as f:
        for line in f:
            m = re.match(r"([0-9a-f]+)-([0-9a-f]+) ", line)
            if m:
                inside = int(m[1], 16) <= addr < int(m[2], 16)
            elif inside and line.startswith("VmFlags:"):
                return set(line.split()[1:])
    raise AssertionError("no such mapping")


@pytest.mark.gpu
def test_results_are_ordinary_memory():
    from alpacc_amd import datagen
    from alpacc_amd.gen.tables import generate
    from alpacc_amd.runtime import Context
    ctx = Context(generate(os.path.join(GRAMMARS, "json.alp")))
    try:
        for n in (300, 20_000, 60_000, 250_000, 500_000, 2_000_000, 8_000_000):
            doc = datagen.json_doc(n, seed=n)
            for r in (ctx.parse_int(doc), ctx.lex_int(doc), ctx.parse_int(doc, chunk_size=1 << 24),
                      ctx.parse_int_batch([doc, doc])[1]):
                for x in r:
                    # shared (sh), device memory (io, pf), not copied to a child (dc, wf)
                    assert not _flags(x.ctypes.data) & {"sh", "io", "pf", "dc", "wf"}, n
    finally:
        ctx.close()


def test_blocks_are_bounded_and_used_again(monkeypatch):
    from alpacc_amd import runtime
    monkeypatch.setattr(runtime, "LEASE_TOTAL", 4 << 20)
    pool = runtime.BlockPool()
    a = pool.empty(200_000)
    at = a.ctypes.data
    part = a[1000:1016].view(np.uint32)
    a[:] = 7
    del a
    gc.collect()
    b = pool.empty(200_000)
    assert b.ctypes.data != at and (part == 0x07070707).all()  # the slice keeps the block
    b[:] = 9
    assert (part == 0x07070707).all()
    del part
    gc.collect()
    assert pool.empty(150_000).ctypes.data == at
    many = [pool.empty(500_000) for _ in range(20)]
    assert pool.allocated <= 4 << 20
    assert len({x.ctypes.data for x in many}) == 20
    assert pool.empty(1000).nbytes == 1000 and pool.empty(0).nbytes == 0
    held = pool.empty(300_000)
    held[:] = 3
    pool.close()
    assert (held == 3).all()
    del many, held
    gc.collect()


def test_blocks_come_back_from_other_threads():
    from alpacc_amd import runtime
    pool = runtime.BlockPool()
    errors = []

    def owner(x, tag):
        if not (x == tag).all():
            errors.append(tag)
        x[:] = 0

    for i in range(200):
        threads = []
        for k in range(4):
            x = pool.empty(130_000 + 1000 * k)
            x[:] = (4 * i + k) % 251
            threads.append(threading.Thread(target=owner, args=(x, (4 * i + k) % 251)))
            del x
        for t in threads:
            t.start()
        if i % 2:
            for t in threads:
                t.join()
        threads.clear()
    assert not errors
    assert pool.allocated <= runtime.LEASE_TOTAL
