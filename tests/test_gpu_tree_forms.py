"""The tree parser with tables of more than 255 pair entries, whose entry ids are 16 bits wide: both
its forms (entries as rows, entries looped over), workgroups of four and of two wavefronts, 32-bit and
64-bit spans, alone and in a batch, against the C restatement. A nonterminal for every letter and an
alternative for every letter in each make as many entries as pairs of letters."""
import numpy as np
import pytest

from tree_tables import form

pytestmark = pytest.mark.gpu

HEAD = "params {\n  lookback = 1.\n  lookahead = 1.\n}\nignore = /\\s/.\n"
LETTERS = "abcdefghijklmnopqrstuvwxyz"


def _grammar(m, tail):
    """S -> c Nc !, Nc -> d Nd tail | . for all letters c, d: the letters, a dot, the tails, a mark."""
    end = " ".join(f'"{t}"' for t in tail)
    rules = ["S -> " + " | ".join(f'"{c}" N{c} "!"' for c in LETTERS[:m]) + ".\n"]
    rules += [f"N{c} -> " + " | ".join(f'"{d}" N{d} {end}' for d in LETTERS[:m]) + ' | ".".\n'
              for c in LETTERS[:m]]
    return HEAD + "".join(rules)


def _doc(m, tail, n, seed):
    rng = np.random.default_rng(seed)
    letters = "".join(LETTERS[int(i)] for i in rng.integers(0, m, n))
    return (letters + "." + tail * (n - 1) + "!").encode()


def _same(got, want, what):
    assert (got is None) == (want is None), what
    for x, y in zip(got or (), want or ()):
        assert np.array_equal(np.asarray(x).reshape(-1), np.asarray(y).reshape(-1)), what


@pytest.mark.parametrize("m,tail,want_form", [
    (17, "", "rows"), (17, "-+", "rows"), (26, "", "rows"), (17, "-+*/", "loops"),
    (20, "-+*/=", "loops"), (17, "-+*/=<>^&", "elements")],
    ids=lambda v: str(v) if v != "" else "none")
def test_wide_entry_ids(m, tail, want_form):
    from alpacc_amd.gen.tables import generate
    from alpacc_amd.runtime import Context
    from oracle.c import coracle
    b = generate(_grammar(m, tail), name=f"letters{m}")
    assert np.asarray(b.parser.pair_entry).reshape(-1, 4).shape[0] > 255
    assert form(b.parser) == want_form
    orc = coracle.Oracle(b)
    docs = [_doc(m, tail, n, n) for n in (1, 2, 50, 63, 64, 65, 252, 253, 254, 255, 1000, 4000, 70_000)]
    docs += [docs[-1][:-2] + b"!", docs[-2] + b"!", docs[-3].replace(b".", b"..", 1), docs[6][:100]]
    if len(tail) > 1:  # a symbol exchanged far from the one it belongs to
        swapped = bytearray(docs[-5])
        swapped[-3], swapped[-4] = swapped[-4], swapped[-3]
        docs.append(bytes(swapped))
    want = [orc.parse(d) for d in docs]
    assert sum(w is not None for w in want) == 13
    ctx = Context(b)
    try:
        ctx.profile(True)
        for i, d in enumerate(docs):
            print(m, repr(tail), i, len(d), flush=True)
            _same(ctx.parse_int(d), want[i], i)
            _same(ctx.parse_int(d, chunk_size=1 << 24), want[i], (i, "64-bit spans"))
        for i, got in enumerate(ctx.parse_int_batch(docs)):
            _same(got, want[i], (i, "batch"))
        ran = ctx.read_profile()
        assert (ran["parse_tree"][1] > 0) == (want_form != "elements")
        assert (ran["parse_expand"][1] > 0) == (want_form == "elements")
    finally:
        ctx.close()
