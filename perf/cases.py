"""Performance cases: what a program that uses this framework has it do.

A program generates a grammar's tables once, opens a Context on them and keeps it. It then lexes or
parses documents that are already in device memory (``lex_device``, ``parse_device``,
``lex_chunked_device``, ``parse_batch_device``), or hands over a document as host bytes and takes
the tree as host arrays (``parse_int``). The grammars are the three that ship with the framework and
have a document generator: json, arithmetic, sexp. Sizes run from one small request to the 256 MiB
document of the headline benchmark; documents and batches are ragged and start where the previous
one ends.

Every output is a whole number (token kinds, positions, node words, parents, verdicts).
"""
from __future__ import annotations

import functools
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from alpacc_amd import datagen
from alpacc_amd.gen.tables import generate
from alpacc_amd.runtime import REFERENCE_CHUNK, Context

HERE = os.path.dirname(os.path.abspath(__file__))
GRAMMARS = os.path.join(os.path.dirname(HERE), "alpacc_amd", "grammars")

DOC = {"json": datagen.json_doc, "arithmetic": datagen.arith_doc, "sexp": datagen.sexp_doc}
# tokens and tree nodes per input byte of the generated documents (they settle from 16 KiB up)
TOKENS = {"json": 0.1506, "arithmetic": 0.379, "sexp": 0.1675}
NODES = {"json": 0.3132, "arithmetic": 1.021, "sexp": 0.4806}
# output nodes (or tokens) a program makes room for, per input byte
ROOM = {"json": 0.5, "arithmetic": 1.25, "sexp": 0.625}

# documents joined to one: before, between and after them
SHELL = {"json": (b"[", b",", b"]"), "sexp": (b"(", b" ", b")"), "arithmetic": (b"", b"+", b"")}

BLOCK = 8 << 20  # large documents are lists of blocks of this size, generated side by side


def listed():
    return [
        # one small request: the whole call is launches and waits
        {"name": "parse_json_2k", "kind": "parse", "grammar": "json", "bytes": 2003},
        # a web page's worth of JSON
        {"name": "parse_json_64k", "kind": "parse", "grammar": "json", "bytes": 65537},
        # an ordinary file
        {"name": "parse_json_1m", "kind": "parse", "grammar": "json", "bytes": 1048579},
        # a large file: the reference's chunk size, in one piece
        {"name": "parse_json_16m", "kind": "parse", "grammar": "json", "bytes": 16777216},
        # the headline benchmark's document
        {"name": "parse_json_256m", "kind": "parse", "grammar": "json", "bytes": 268435456},
        # program text rather than data: short tokens, a node for every byte
        {"name": "parse_arith_1m", "kind": "parse", "grammar": "arithmetic", "bytes": 1048576},
        # the lexer alone, on one small request and on a whole dump
        {"name": "lex_json_4k", "kind": "lex", "grammar": "json", "bytes": 4099},
        {"name": "lex_json_256m", "kind": "lex", "grammar": "json", "bytes": 268435456},
        # the reference's lexer entry as generated: its loop over 16 MiB chunks, 64-bit spans
        {"name": "lex_json_chunked_48m", "kind": "chunked", "grammar": "json", "bytes": 50331651},
        # a server's batch of small requests, sizes spread over their logarithm
        {"name": "batch_json_requests", "kind": "batch", "grammar": "json", "docs": 200,
         "low": 256, "high": 65536},
        # a corpus in one call: log-normal document sizes around 64 KiB, up to 16 MiB
        {"name": "batch_sexp_256m", "kind": "corpus", "grammar": "sexp", "docs": 512,
         "bytes": 268435456},
        # host bytes in, host arrays out
        {"name": "host_json_256k", "kind": "host", "grammar": "json", "bytes": 262147},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    grammar = rng.choice(["json", "json", "sexp", "arithmetic"])
    kind = rng.choice(["parse", "parse", "parse", "lex", "chunked", "batch", "corpus", "host"])
    # an arithmetic document has three times the nodes of a JSON document of its size
    top = (64 << 20) if grammar == "arithmetic" else (256 << 20)
    case = {"kind": kind, "grammar": grammar}
    if kind in ("parse", "lex"):
        case["bytes"] = spread(500, top)
    elif kind == "chunked":
        case["bytes"] = spread(1 << 20, 96 << 20)
    elif kind == "batch":
        case["docs"] = spread(2, 2000)
        case["low"] = spread(128, 2048)
        case["high"] = spread(4096, 65536)
    elif kind == "corpus":
        case["docs"] = spread(16, 512)
        case["bytes"] = case["docs"] * spread(96 << 10, min(512 << 10, top // case["docs"]))
    else:
        case["bytes"] = spread(500, 4 << 20)
    return case


def _sizes(case):
    """Document sizes of a batch; they belong to the case, not to the seed of its contents."""
    if case["kind"] == "corpus":
        return datagen.sexp_batch_sizes(count=case["docs"], total=case["bytes"])
    rng = np.random.Generator(np.random.PCG64(case["docs"]))
    lo, hi = math.log(case["low"]), math.log(case["high"])
    return np.exp(rng.uniform(lo, hi, case["docs"])).astype(np.int64)


def _bytes(case):
    if case["kind"] in ("batch", "corpus"):
        return int(_sizes(case).sum())
    return case["bytes"]


@functools.lru_cache(maxsize=None)
def _context(grammar):
    return Context(generate(os.path.join(GRAMMARS, grammar + ".alp")))


@functools.lru_cache(maxsize=None)
def _pool():
    return ThreadPoolExecutor(max_workers=16)


def _many(grammar, sizes, seeds):
    """Documents of the given sizes, one after the other, in one array."""
    ends = np.cumsum(sizes)
    out = np.empty(int(ends[-1]), dtype=np.uint8)
    jobs = [_pool().submit(DOC[grammar], int(n), int(s), out[int(e) - int(n):int(e)])
            for n, s, e in zip(sizes, seeds, ends)]
    for j in jobs:
        j.result()
    return out


def _document(grammar, n, seed):
    """One document of n bytes."""
    if n < 2 * BLOCK:
        return DOC[grammar](n, seed)
    head, sep, tail = SHELL[grammar]
    count = n // BLOCK
    room = n - len(head) - len(tail) - len(sep) * (count - 1)
    sizes = np.full(count, room // count)
    sizes[-1] += room - int(sizes.sum())
    blocks = _many(grammar, sizes, [seed * 1000003 + i for i in range(count)])
    out = np.empty(n, dtype=np.uint8)
    at = len(head)
    out[:at] = np.frombuffer(head, dtype=np.uint8)
    src = 0
    for i, k in enumerate(int(s) for s in sizes):
        if i:
            out[at:at + len(sep)] = np.frombuffer(sep, dtype=np.uint8)
            at += len(sep)
        out[at:at + k] = blocks[src:src + k]
        at += k
        src += k
    out[at:] = np.frombuffer(tail, dtype=np.uint8)
    return out


def _shuffled(grammar, n, seed):
    """One document of n bytes: eight blocks that belong to the case, in an order that the seed
    decides, so that a program's arrays of its tree have the same length for every seed."""
    head, sep, tail = SHELL[grammar]
    room = n - len(head) - len(tail) - 7 * len(sep)
    blocks = [DOC[grammar](room // 8 + (room % 8 if i == 7 else 0), 100 + i) for i in range(8)]
    order = np.random.Generator(np.random.PCG64(seed)).permutation(8)
    return head + sep.join(blocks[i].tobytes() for i in order) + tail


def _room(count, dtype=torch.int32):
    """Room for a result, filled with zeros: a call writes as many entries as it counts."""
    return torch.zeros(count, dtype=dtype, device="cuda")


def prepare(case, seed):
    grammar, kind = case["grammar"], case["kind"]
    state = {"kind": kind, "ctx": _context(grammar)}
    if kind == "host":
        state["doc"] = _shuffled(grammar, case["bytes"], seed)
        return state
    if kind in ("batch", "corpus"):
        sizes = _sizes(case)
        doc = _many(grammar, sizes, [seed * 1000003 + i for i in range(len(sizes))])
        state["lengths"] = sizes.astype(np.uint64)
        state["offsets"] = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.uint64)
    else:
        doc = _document(grammar, case["bytes"], seed)
    n = len(doc)
    state["n"] = n
    state["doc"] = torch.from_numpy(doc).cuda()
    if kind == "lex":
        state["cap"] = n
        state["kinds"], state["starts"], state["ends"] = _room(n), _room(n), _room(n)
    elif kind == "chunked":
        state["cap"] = cap = n + n // REFERENCE_CHUNK + 1
        state["kinds"] = _room(cap)
        state["starts"], state["ends"] = _room(cap, torch.int64), _room(cap, torch.int64)
    else:
        state["cap"] = cap = int(ROOM[grammar] * n) + 4096
        state["parent"], state["node"], state["span"] = _room(cap), _room(cap), _room(2 * cap)
    return state


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "host":
        tree = ctx.parse_int(state["doc"])
        if tree is None:
            return {"status": 0}
        return {"status": 1, "parent": tree[0], "node": tree[1], "span": tree[2]}
    doc, n, cap = state["doc"].data_ptr(), state["n"], state["cap"]
    if kind in ("lex", "chunked"):
        kinds, starts, ends = state["kinds"], state["starts"], state["ends"]
        if kind == "lex":
            status, count = ctx.lex_device(doc, n, kinds.data_ptr(), starts.data_ptr(),
                                           ends.data_ptr(), cap)
        else:
            status, count = ctx.lex_chunked_device(doc, n, REFERENCE_CHUNK, kinds.data_ptr(),
                                                   starts.data_ptr(), ends.data_ptr(), cap)
        return {"status": status, "count": count, "kinds": kinds, "starts": starts, "ends": ends}
    parent, node, span = state["parent"], state["node"], state["span"]
    tree = {"parent": parent, "node": node, "span": span}
    if kind == "parse":
        status, count = ctx.parse_device(doc, n, parent.data_ptr(), node.data_ptr(),
                                         span.data_ptr(), cap)
        return {"status": status, "count": count, **tree}
    status, count, docs = ctx.parse_batch_device(doc, state["offsets"], state["lengths"],
                                                 parent.data_ptr(), node.data_ptr(),
                                                 span.data_ptr(), cap)
    return {"status": status, "count": count, "verdicts": docs["status"].copy(),
            "first": docs["offset"].astype(np.int64), "nodes": docs["count"].astype(np.int64),
            **tree}


def work(case):
    """The document in, and out: a kind and two positions per token, or a parent, a node word and
    two positions per tree node. The work is look-ups and whole-number scans, about two per byte."""
    n, grammar = _bytes(case), case["grammar"]
    if case["kind"] == "lex":
        out = 12 * TOKENS[grammar] * n
    elif case["kind"] == "chunked":
        out = 20 * TOKENS[grammar] * n
    else:
        out = 16 * NODES[grammar] * n
    return {"bytes": int(n + out), "flops": 2 * n}


def exact(case, seed):
    """No output is a rounded number: they are compared for equality."""
    return None
