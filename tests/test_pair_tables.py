"""The quadratic form of the jump sums (lmc_pairs.cpp, no GPU): its tables, summed over the
non-reference sites and pairs of random environments, equal the sums over every cluster, for every
reference element, in either order of a pair, sparse and over the list of all pairs."""
import os
import subprocess

import pytest

from latticemontecarlo_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "latticemontecarlo_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pairs") / "pair_check")
    src = [os.path.join(ROOT, "tests", "cpp", "pair_check.cpp")]
    src += [os.path.join(CSRC, f) for f in ("lmc_pairs.cpp", "lmc_tables.cpp", "lmc_model.cpp")]
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + CSRC, *src, "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("kind", ["E0", "Quartic"])
@pytest.mark.parametrize("els", [["Al"], ["Al", "Zn"], ["Al", "Mg", "Zn"], ["Al", "Cu", "Mg", "Zn"],
                                 ["Al", "Cu", "Mg", "Sn", "Zn"]])
def test_quadratic_form_equals_cluster_sums(program, tmp_path, els, kind):
    path = str(tmp_path / "c.json")
    synth.write_coefficients(path, els, kind, seed=5, randomize_norm=True, n_rows=2)
    out = subprocess.run([program, path, {"E0": "1", "Quartic": "2"}[kind], *els], check=True,
                         capture_output=True, text=True).stdout
    # each side adds at most 1 228 terms, four times the sum of magnitudes in the differences of
    # a pair's four values: 4 * 1228 * 2^-53 relative to the sum of magnitudes
    assert float(out) < 4 * 1228 * 2.0 ** -53
