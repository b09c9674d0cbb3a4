"""The operation counts that the roofline figures use are those of the code that runs."""
import json
import os
import re

import pytest

import bench
from pelelm_amd.mechanisms import hipgen
from pelelm_amd.mechanisms import mechanism as M


@pytest.mark.parametrize("name", ["LiDryer", "drm19", "dodecane53", "dodecane56", "heptane88"])
def test_emitted_counts_are_of_the_emitted_code(name):
    mech = M.load(name)
    with open(os.path.join(M.HERE, f"{name}_ops.json")) as f:
        doc = json.load(f)
    assert doc["emitted"] == hipgen.emitted_counts(mech)
    with open(os.path.join(M.HERE, "..", "csrc", "mech", f"{name}.inc")) as f:
        code = f.read()
    # exponentials and logarithms of the rates as they stand in the file: one per species
    # (the loop's) and the others written out
    wdot = re.sub("//.*", "", code[code.index(" void wdot("):code.index("T_LOW")])
    written = sum(len(re.findall(rf"\b{t}\(", wdot)) for t in ("exp", "log10", "log", "pow", "sqrt"))
    assert doc["emitted"]["wdot"]["transcendentals"] == written - 1 + mech.nspec
    fixed, per_iter, trans = bench.rhs_ops(name)
    assert trans == doc["emitted"]["wdot"]["transcendentals"] + 1
    # an iteration of HY2T evaluates two polynomials, whatever the number of species
    assert per_iter == bench.rhs_ops("LiDryer")[1]
    assert fixed < 2 * (doc["emitted"]["wdot"]["flops"] + doc["emitted"]["gibbs"]["flops"])
