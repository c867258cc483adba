"""Batches with more replicas than the chip has CUs, stepped by one wave per replica: several replicas of
unequal boxes, solvents and solute contents share a workgroup and its tables (those of its first
replica's solvent). A sample of replicas from both ends and the middle of workgroups is replayed by the
oracle, as are the atoms' jumps; first-order and chain steps, both barrier models, value tables in LDS
(ternary E0) and partly in global memory (quaternary Quartic), environments past the sparse limit."""
import numpy as np
import pytest

from conftest import random_alloc
from test_config_gpu import _replay, _start_atoms

pytestmark = pytest.mark.gpu

TOL_E = 1e-9


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


def _batch(species, R):
    """Boxes of 4 to 7 cells; every fifth replica is Mg-based, every seventh concentrated."""
    sizes = [4 + r % 4 for r in range(R)]
    occs = []
    for r, n in enumerate(sizes):
        occ = random_alloc(n, species, 0.25 if r % 7 == 3 else 0.02 + 0.01 * (r % 5), seed=9000 + r)
        if r % 5 == 2:
            al, mg = species.index("Al"), species.index("Mg")
            occ = np.where(occ == al, mg, np.where(occ == mg, al, occ)).astype(np.uint8)
        occs.append(occ)
    return sizes, occs


def _time_bound(om, lat, species, occ, vac, sel, time, tt, T):
    """Relative rounding of a chain trajectory's time beyond 1e-12. A step's time divides by the sum of
    p_ki (1 - p_ik) (KineticMcChainOmpi.cpp:93-151), whose terms are rounded to a few 2^-53 of p_ki: relative to
    a sum that makes the step A times as long as the first-order residence time, some 2^-53 A. Sixteen
    covers its dozen additions and the rounding of the rates."""
    occ, x, worst, before = occ.copy(), species.index("X"), 0.0, 0.0
    for s, t in zip(sel, time):
        beta = 1 / 8.617333262145e-5 / (np.interp(before, *tt) if tt else T)
        total = sum(np.exp(-om.barrier_de(occ, vac, int(b))[0] * beta) for b in lat.neighbors(vac, 1))
        worst = max(worst, abs(t - before) * total * 1e13)
        occ[vac], occ[s] = occ[s], x
        vac, before = int(s), t
    return 16 * 2.0 ** -53 * worst


@pytest.mark.parametrize("name,kind,chain,full", [
    ("e0_3n", 1, False, False), ("e0_3n", 1, False, True), ("q_4", 2, False, True), ("q_3n", 2, False, False),
    ("e0_3n", 1, True, False), ("q_4", 2, True, True), ("e0_4n", 1, True, True),
])
def test_large_batches_match_oracle(torch, coeffs, tmp_path, name, kind, chain, full):
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = coeffs[name]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    R = 2 * cus + 37
    model = L.Model(path, els, kind)
    sizes, occs = _batch(model.species, R)
    temps = np.linspace(450.0, 750.0, R)
    steps, seed = 24 if chain else 80, 31
    opts = dict(rate_corrector=True, solute_disp=True) if full else {}
    tt = (np.array([0.0, 1e-9, 1e-6]), np.array([800.0, 600.0, 400.0])) if full else None
    print(f"{R} replicas, {name} chain={chain} full={full}", flush=True)
    drv = (L.KineticMcChain if chain else L.KineticMcFirst)(model, None, sizes, occs, temps, seed,
                                                            maximum_steps=10 ** 9, **opts)
    sample = sorted({0, 1, 2, 3, 17, 23, R // 2, R // 2 + 1, R // 2 + 2, R - 3, R - 2, R - 1})
    if full:
        drv.set_schedule(*tt)
        drv.set_trace(steps)
        drv.set_log(10, capacity=200)
        atoms = [_start_atoms(n, 1, seed=r) for r, n in enumerate(sizes)]
        drv.set_atoms([a[0][0] for a in atoms], [a[1][0] for a in atoms])
    drv.run(steps // 3)
    drv.run(steps - steps // 3)
    model.check_errors()
    st, occ = drv.state(), drv.occupancy()
    tr = drv.trace() if full else None
    now = drv.atoms() if full else None
    assert np.all(st["steps"] == steps)
    for r in sample:
        lat = O.Lattice(sizes[r])
        om = O.Model(lat, path, els, kind)  # the trajectory refers to it
        k = O.Kmc(om, None, lat, occs[r], temps[r], seed, replica=r, tt=tt, chain=chain, **opts)
        want = k.run(steps, trace=True)
        ost = k.state()
        assert int(st["vacancy"][r]) == ost["vacancy"], f"replica {r}"
        assert np.array_equal(occ[r], k.occupancy()) and np.array_equal(st["disp"][r], ost["disp"])
        start = int(np.flatnonzero(occs[r] == model.species.index("X"))[0])
        rtol = 1e-12 + (_time_bound(om, lat, model.species, occs[r], start, want["sel"], want["time"], tt, temps[r])
                        if chain else 0.0)
        np.testing.assert_allclose(st["time"][r], ost["time"], rtol=rtol)
        assert abs(st["energy"][r] - ost["energy"]) <= TOL_E * steps
        if not full:
            continue
        np.testing.assert_allclose(st["com"][r], ost["com"], rtol=0, atol=1e-9)
        np.testing.assert_allclose(st["temperature"][r], ost["temperature"], rtol=1e-12)
        assert np.array_equal(tr["sel"][r], want["sel"].astype(np.int64))
        np.testing.assert_allclose(tr["ea"][r], want["ea"], rtol=0, atol=TOL_E)
        np.testing.assert_allclose(tr["de"][r], want["de"], rtol=0, atol=TOL_E)
        np.testing.assert_allclose(tr["time"][r], want["time"], rtol=rtol)
        hops = np.concatenate([[start], tr["sel"][r]])
        ra, rs = _replay(sizes[r], atoms[r][0][0], atoms[r][1][0], zip(hops[:-1], hops[1:]))
        assert np.array_equal(now[0][r], ra) and np.array_equal(now[1][r], rs)
    if full:
        files = [str(tmp_path / f"{r}.txt") if r in sample else None for r in range(R)]
        drv.write_log(files)
        for r in sample:
            head, *lines = [x.split("\t") for x in open(files[r]).read().strip().split("\n")]
            energy = np.concatenate([[0.0], np.cumsum(tr["de"][r])])
            assert [int(x[0]) for x in lines] == list(range(steps))  # every step below 99
            for s, x in enumerate(lines):
                assert float(x[head.index("energy")]) == pytest.approx(energy[s], rel=1e-4, abs=1e-9)


@pytest.mark.parametrize("name,kind", [("e0_4n", 1), ("q_3n", 2), ("q_4", 2)])
def test_chain_teams_that_share_a_cu(torch, coeffs, name, kind):
    """Two teams of a CU have half of its LDS each, so that less of the value tables is there than for the same
    replicas in a smaller batch: none of a quaternary model's, where that has all (E0) or part (Quartic)."""
    import latticemontecarlo_amd as L
    path, els = coeffs[name]
    model = L.Model(path, els, kind)
    R = torch.cuda.get_device_properties(0).multi_processor_count + 44
    sizes, occs = _batch(model.species, R)
    print(f"{R} chain replicas, {name}", flush=True)
    got = []
    for many in (R, 40):
        drv = L.KineticMcChain(model, None, sizes[:many], occs[:many], 650.0, 7, maximum_steps=10 ** 9)
        drv.run(12)
        model.check_errors()
        got.append(drv.state())
    assert np.array_equal(got[0]["vacancy"][:40], got[1]["vacancy"])
    assert np.array_equal(got[0]["disp"][:40], got[1]["disp"])
    np.testing.assert_allclose(got[0]["energy"][:40], got[1]["energy"], rtol=0, atol=TOL_E)


@pytest.mark.parametrize("R", [5, 300])
def test_formulations_are_different_kernels(torch, coeffs, R):
    """1 is one wave per replica and 2 four at every batch size: both follow the same trajectory, and the
    autotuner reports both times and keeps one of the two."""
    import latticemontecarlo_amd as L
    path, els = coeffs["e0_3n"]
    model = L.Model(path, els, L.E0)
    sizes, occs = _batch(model.species, R)
    got = []
    for form in (0, 1, 2):
        drv = L.KineticMcFirst(model, None, sizes, occs, 600.0, 5, maximum_steps=10 ** 9)
        drv.set_formulation(form)
        drv.run(100)
        got.append(drv.state())
    for other in got[1:]:
        assert np.array_equal(got[0]["vacancy"], other["vacancy"]) and np.array_equal(got[0]["disp"], other["disp"])
        np.testing.assert_allclose(other["time"], got[0]["time"], rtol=1e-12)
    # 0 stands for one of them; the two add the energies' terms in different orders
    one, four = (g["energy"].tolist() for g in got[1:])
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert got[0]["energy"].tolist() == (four if R <= cus else one)
    assert one != four
    tune = drv.autotune(steps=40)
    assert tune["formulation"] in (1, 2) and tune["ms_solvent"] > 0 and tune["ms_wide"] > 0
    assert tune["ms_dense"] == (tune["ms_wide"] if R <= cus else tune["ms_solvent"])


def test_captured_launches_keep_their_lds(torch, coeffs):
    """A captured launch with much dynamic LDS, replayed after launches of the same kernel with less."""
    import latticemontecarlo_amd as L
    path, els = coeffs["e0_3n"]
    model = L.Model(path, els, L.E0)

    def driver(R):
        sizes, occs = _batch(model.species, R)
        d = L.KineticMcFirst(model, None, sizes, occs, 600.0, 5, maximum_steps=10 ** 9)
        d.set_formulation(1)
        return d
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    large, small, want = driver(8 * cus), driver(1), driver(8 * cus)  # eight replicas in a workgroup, and one
    large.build_graph(20, 2)
    for _ in range(3):
        small.run(20)
        large.run_graph(20, 2)
        small.state()
        for _ in range(2):
            want.run(20)
        a, b = large.state(), want.state()
        assert np.array_equal(a["vacancy"], b["vacancy"]) and np.array_equal(a["time"], b["time"])
        assert np.array_equal(a["energy"], b["energy"])
