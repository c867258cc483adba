"""What a jump evaluation checks of the occupancy that it is given: species codes past the model's at any
site that it reads, the vacancy's own among them, and the environment rows of jump samples."""
import numpy as np
import pytest

from conftest import random_alloc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


def _setup(coeffs, n=8):
    import latticemontecarlo_amd as L
    path, els = coeffs["e0_3n"]
    model = L.Model(path, els, L.E0)
    occ = random_alloc(n, model.species, 0.05, seed=3)
    vac = int(np.flatnonzero(occ == model.species.index("X"))[0])
    return L, model, occ, vac, n


@pytest.mark.parametrize("where", ["own", "neighbour", "environment", "far"])
def test_species_codes_past_the_model_are_reported(torch, coeffs, where):
    from latticemontecarlo_amd import capi
    L, model, occ, vac, n = _setup(coeffs)
    batch = L.ReplicaBatch([n], [occ])
    near = L.fcc_neighbors(n, vac, 1)
    env = {int(s) for b in near for s in L.jump_environment(n, vac, int(b))} | {vac}
    site = {"own": vac, "neighbour": int(near[5]), "environment": max(env - {vac} - {int(b) for b in near}),
            "far": min(set(range(4 * n ** 3)) - env)}[where]
    batch.occ[site] = 200
    L.eval_jumps(model, batch, [vac])
    torch.cuda.synchronize()
    if where == "far":
        model.check_errors()
    else:
        with pytest.raises(capi.LmcError):
            model.check_errors()
    model.check_errors()  # reported once


def test_sample_rows_hold_the_species_of_every_slot(torch, coeffs):
    """Also at the vacancy's own slot, where a caller may have left an atom."""
    L, model, occ, vac, n = _setup(coeffs)
    for code in (model.species.index("X"), model.species.index("Zn")):
        occ[vac] = code
        batch = L.ReplicaBatch([n], [occ])
        env = L.jump_samples(model, batch, [vac])[0].cpu().numpy()
        for row, b in zip(env, L.fcc_neighbors(n, vac, 1)):
            assert row[:60].tolist() == [int(occ[s]) for s in L.jump_environment(n, vac, int(b))]
            assert not row[60:].any()
