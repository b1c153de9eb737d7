"""The rule that sends a grammar to the tree parser, on the CPU: for every shipped grammar and every
random one whose entries it takes, parents found with one stack of symbol owners (what the tree
parser computes) equal the parents of the C restatement (previous smaller-or-equal s,
parser.fut:286-296), and both reject the same token streams."""
import os

import numpy as np
import pytest

from conftest import GRAMMARS
from lookahead_grammar import QK, sentence as pg_sentence, source
from random_grammar import corrupt, sentence
from test_fuzz_grammars import kept_grammars
from tree_tables import entries, form, key_entries, parents


def _check(b, docs):
    from oracle.c import coracle
    orc = coracle.Oracle(b)
    accepted = 0
    for d in docs:
        toks = orc.lex(d)
        if toks is None or not b.parser.pair_index.shape[0]:
            continue
        want = orc.parse(d)
        got = parents(b.parser, np.asarray(toks[0]).tolist())
        assert (got is None) == (want is None), d
        if want is not None:
            assert got == np.asarray(want[0]).tolist(), d
            accepted += 1
    return accepted


def test_shipped_grammars():
    from alpacc_amd import datagen
    from alpacc_amd.gen.tables import generate
    gens = {"json": datagen.json_doc, "sexp": datagen.sexp_doc, "arithmetic": datagen.arith_doc}
    for g, gen in gens.items():
        b = generate(os.path.join(GRAMMARS, g + ".alp"))
        assert form(b.parser) == "rows"
        docs = [gen(n, seed=n).tobytes() for n in (40, 1000, 9000)]
        docs += [datagen.flip_bytes(gen(900, seed=s), seed=s).tobytes() for s in range(6)]
        assert _check(b, docs) >= 3
    for g in ("llp01", "paper_grammar", "list"):
        assert form(generate(os.path.join(GRAMMARS, g + ".alp")).parser) == "rows"


@pytest.mark.parametrize("part", range(4))
def test_random_grammars(part):
    forms = {}
    for seed, q, k, b, prods in kept_grammars(40)[part::4]:
        f = form(b.parser)
        forms[f] = forms.get(f, 0) + 1
        if f == "elements":
            continue
        docs = []
        for target in (1, 4, 16, 200):
            d = sentence(prods, seed * 100 + target, target)
            docs += [d, corrupt(d, seed + target)]
        _check(b, docs)
    print(part, forms)
    assert forms.get("rows", 0) + forms.get("loops", 0) > 0


def test_lookahead_grammars():
    from alpacc_amd.gen.tables import generate
    for q, k in QK:
        b = generate(source(q, k))
        if form(b.parser) != "elements":
            docs = [pg_sentence(n, seed=n) for n in (1, 30, 2000)]
            assert _check(b, docs) > 0 or not b.parser.pair_index.shape[0]


def test_end_entries_stand_at_the_ends():
    """Entries that push unowned or pop unfilled symbols are found at the first and last position
    only (the table's keys carry the start and end terminals there)."""
    from alpacc_amd import datagen
    from alpacc_amd.gen.tables import generate
    from oracle.c import coracle
    b = generate(os.path.join(GRAMMARS, "json.alp"))
    kinds = np.asarray(coracle.Oracle(b).lex(datagen.json_doc(5000, seed=3))[0]).tolist()
    kind = [entries(b.parser)[e][4] for e in key_entries(b.parser, kinds)]
    assert kind[0] == 1 and kind[-1] == 2 and not any(kind[1:-1])
