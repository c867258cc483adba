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


@pytest.mark.parametrize("many", [1, 40, 0, 1000])
@pytest.mark.parametrize("name,kind", [("e0_3n", 1), ("q_4", 2)])
def test_shared_and_single_wave_sums_match_oracle(torch, coeffs, name, kind, many):
    """One workgroup to each vacancy up to the number of CUs (0 here), eight vacancies to a workgroup above;
    contents below and above both limits of the sparse sums, and an invalid vacancy among the others."""
    import latticemontecarlo_amd as L
    import oracle as O
    from latticemontecarlo_amd import capi
    path, els = coeffs[name]
    R = many or torch.cuda.get_device_properties(0).multi_processor_count
    model, n = L.Model(path, els, kind), 5
    x = model.species.index("X")
    occs = [random_alloc(n, model.species, (0.02, 0.06, 0.08, 0.10, 0.2)[r % 5], seed=500 + r) for r in range(R)]
    vac = np.array([int(np.flatnonzero(o == x)[0]) for o in occs])
    print(f"{R} vacancies, {name}", flush=True)
    got = [v.cpu().numpy().reshape(R, 12) for v in L.eval_jumps(model, L.ReplicaBatch([n] * R, occs), vac)]
    model.check_errors()
    lat = O.Lattice(n)
    om = O.Model(lat, path, els, kind)
    for r in sorted({*range(min(R, 10)), *range(max(R - 5, 0), R)}):
        for j, b in enumerate(sorted(int(b) for b in lat.neighbors(int(vac[r]), 1))):
            ea, de = om.barrier_de(occs[r], int(vac[r]), b)
            assert got[0][r, j] == b
            assert abs(got[1][r, j] - ea) <= 1e-9 and abs(got[2][r, j] - de) <= 1e-9, (r, j)
    bad = vac.copy()
    bad[R // 2] = 4 * n ** 3
    other = [v.cpu().numpy().reshape(R, 12) for v in L.eval_jumps(model, L.ReplicaBatch([n] * R, occs), bad)]
    with pytest.raises(capi.LmcError):
        model.check_errors()
    keep = np.arange(R) != R // 2
    assert all(np.array_equal(g[keep], o[keep]) for g, o in zip(got, other))
