"""The node records of parse_tree are stored as words, by every entry as many as the largest entry
has, and then get their parents as half-words. What the compiler is told about these stores, read in
the device code as the front end emits it (before any optimisation): the half-word stores may meet
word stores (they carry the type that aliases everything), and the rounds of record stores are
fenced, since a round overwrites what other lanes stored in the round before."""
import os
import re
import subprocess

import pytest

from alpacc_amd import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: body} of the parse_tree instances, and the metadata nodes {id: text}."""
    out = str(tmp_path_factory.mktemp("ir") / "device.ll")
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-shared")]
    subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-Xclang", "-disable-llvm-passes",
                    "-emit-llvm", "-S", "-I", os.path.join(build.ROOT, "include"), build.SRC, "-o",
                    out], check=True, capture_output=True)
    text = open(out).read()
    bodies = {m[1]: m[2] for m in re.finditer(
        r"^define [^\n]*@(\w*parse_tree\w*)\([^\n]*\{\n(.*?)^\}", text, re.M | re.S)}
    helpers = {m[1]: m[2] for m in re.finditer(
        r"^define [^\n]*@(\w*ft_set_parent\w*)\([^\n]*\{\n(.*?)^\}", text, re.M | re.S)}
    meta = dict(re.findall(r"^!(\d+) = (.*)$", text, re.M))
    assert len(bodies) >= 12
    return bodies, helpers, meta


def _access_type(meta, tag):
    base = re.match(r"!\{!\d+, !(\d+), ", meta[tag])[1]
    return re.match(r'!\{!"([^"]+)"', meta[base])[1]


def test_parent_halves_alias_the_records(kernels):
    bodies, helpers, meta = kernels
    stores = re.findall(r"store i16 [^\n]*!tbaa !(\d+)", "\n".join([*bodies.values(),
                                                                   *helpers.values()]))
    assert stores
    assert {_access_type(meta, t) for t in stores} == {"omnipotent char"}


def test_record_rounds_are_fenced(kernels):
    bodies, _, _ = kernels
    # every instance that takes entries as rows has one more fence than its twin that loops over them
    # (template arguments <span type, batched, entry ids, rows, linking>)
    syncs = {}
    for name, body in bodies.items():
        *kind, rows, link = re.search(r"parse_treeI(\w)Lb(\d)E(\w)Lb(\d)ELb(\d)E", name).groups()
        if link == "0":
            syncs[(*kind, rows)] = len(re.findall(r"call [^\n]*wave_lds_sync", body))
    assert len(syncs) >= 12
    for *kind, rows in list(syncs):
        if rows == "1":
            assert syncs[(*kind, "1")] == syncs[(*kind, "0")] + 1, kind
