"""The autotuner times the searches' launch choices only for grammars that run the searches."""
import os

import pytest

from conftest import GRAMMARS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", ["json", "elements"])
def test_only_choices_that_run(g):
    from alpacc_amd import autotune, datagen
    from alpacc_amd.gen.tables import generate
    from test_gpu_tree import ELEMENTS
    if g == "json":
        b = generate(os.path.join(GRAMMARS, "json.alp"))
        docs = [datagen.json_doc(n, seed=n) for n in (500, 20_000, 60_000)]
    else:
        b = generate(ELEMENTS)
        docs = [b"a" * n + b"x" + b"bcdefghijk" * n for n in (20, 800, 2_000)]
    rec = autotune.tune(b, docs, reps=1, save_result=False)
    tried = {name for t in rec["tried"] for name in t}
    assert {"lexer_tables_in_lds", "lex_blocks_per_cu", "keys_blocks_per_cu"} <= tried
    assert bool(set(autotune.SEARCHES) & tried) == (g == "elements")
    if g == "json":
        assert all(rec["params"][k] == autotune.DEFAULTS[k] for k in autotune.SEARCHES)
