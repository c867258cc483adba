"""Serial canonical trials where trials tried side by side meet: boxes of 256 sites at high temperature
(nearly every round has an accepted trial that a later one read), a box with one solute (pairs found
after the first 63 and 127 attempts), equal shares (every first attempt wins), runs cut into launches of
1, 7 and more trials, and annealing schedules whose windows, triggers and cooldowns are shorter than a
round. Trajectories are the sequential oracle's."""
import numpy as np
import pytest

from conftest import random_alloc

pytestmark = pytest.mark.gpu
TOL_E = 1e-9


def _occ(n, species, frac, seed):
    if frac is None:  # one solute
        occ = np.full(4 * n ** 3, species.index("Al"), np.uint8)
        occ[seed % len(occ)] = species.index("Mg")
        return occ
    return random_alloc(n, species, frac, seed=seed, vacancy=False)


@pytest.mark.parametrize("lds", [True, False])
@pytest.mark.parametrize("fracs", [(0.3, 0.5, 0.02), (None, 0.01, None)])
def test_side_by_side_trials(coeffs, fracs, lds):
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = coeffs["e0_3n"]
    sizes, chunks, seed = [4, 4, 6], [1, 7, 200, 16, 3], 11
    gp = L.Model(path, els, L.PAIRSITE)
    occs = [_occ(n, gp.species, f, 31 + r) for r, (n, f) in enumerate(zip(sizes, fracs))]
    total = sum(chunks)
    ge = L.Model(path, els, L.ENERGY)
    drv = L.CanonicalMc(gp, ge, sizes, occs, 3000.0, 900.0, seed, maximum_steps=total)
    drv.set_lds_occupancy(lds)
    drv.set_trace(total)
    for k in chunks:
        drv.run(k)
    gst, gtr, gocc = drv.state(), drv.trace(), drv.occupancy()
    gp.check_errors()
    for r, n in enumerate(sizes):
        lat = O.Lattice(n)
        op, oe = O.Model(lat, path, els, O.PAIRSITE), O.Model(lat, path, els, O.ENERGY)
        c = O.Cmc(op, oe, lat, occs[r], 3000.0, 900.0, seed, replica=r)
        tr = c.run(total, total, trace=True)
        assert np.array_equal(gtr["p"][r], tr["p"]) and np.array_equal(gtr["q"][r], tr["q"])
        np.testing.assert_allclose(gtr["de"][r], tr["de"], rtol=0, atol=TOL_E)
        assert np.array_equal(gtr["acc"][r], tr["acc"])
        assert np.array_equal(gocc[r], c.occupancy())
        st = c.state()
        assert int(gst["accepted"][r]) == st["accepted"]
        assert abs(gst["energy"][r] - st["energy"]) <= TOL_E * total


@pytest.mark.parametrize("steps, T0", [(60, 3000.0), (400, 900.0), (9000, 300.0)])
def test_short_annealing_windows(coeffs, steps, T0):
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = coeffs["e0_3n"]
    n, R, seed = 4, 3, 5
    gp = L.Model(path, els, L.PAIRSITE)
    occs = [random_alloc(n, gp.species, 0.02 + 0.1 * r, seed=60 + r, vacancy=False) for r in range(R)]
    drv = L.SimulatedAnnealing(gp, None, [n] * R, occs, T0, seed, maximum_steps=steps)
    drv.set_trace(steps)
    drv.run(steps // 3)
    drv.run(steps - steps // 3)
    gst, gtr, ga = drv.state(), drv.trace(), drv.annealing_state()
    lat = O.Lattice(n)
    op = O.Model(lat, path, els, O.PAIRSITE)
    for r in range(R):
        c = O.Cmc(op, None, lat, occs[r], T0, T0, seed, replica=r, anneal=True)
        tr = c.run(steps, steps, trace=True)
        st, oa = c.state(), c.anneal_state()
        assert np.array_equal(gtr["p"][r], tr["p"]) and np.array_equal(gtr["acc"][r], tr["acc"])
        assert int(gst["accepted"][r]) == st["accepted"]
        assert ga["temperature"][r] == pytest.approx(oa["temperature"], rel=1e-12)
        assert abs(ga["lowest"][r] - oa["lowest"]) <= TOL_E * steps
        assert int(ga["reheats"][r]) == oa["reheats"]


@pytest.mark.parametrize("K, lds", [(64, True), (64, False), (3, True)])
def test_rounds_over_compositions(coeffs, K, lds):
    """Rounds where the most frequent species is not the first, where nothing is rare (every site of an
    environment has terms), where pairs are found late, and where the swapped sites are neighbours."""
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = coeffs["e0_4n"]
    sizes, chunks, seed = [4, 5, 6, 12], [1, 70, 5, 150], 23
    gp, ge = L.Model(path, els, L.PAIRSITE), L.Model(path, els, L.ENERGY)
    shares = [(0.25, 0.25, 0.25, 0.25), (0.05, 0.1, 0.8, 0.05), (0.98, 0.0, 0.0, 0.02), (0.1, 0.5, 0.1, 0.3)]
    codes = [gp.species.index(e) for e in els]
    rng = np.random.default_rng(3)
    occs = [rng.choice(codes, 4 * n ** 3, p=w).astype(np.uint8) for n, w in zip(sizes, shares)]
    total = sum(chunks)
    drv = L.CanonicalMc(gp, ge, sizes, occs, 2500.0, 700.0, seed, maximum_steps=total)
    drv.set_lds_occupancy(lds)
    drv.set_parallel_trials(K)
    drv.set_trace(total)
    for k in chunks:
        drv.run(k)
    gst, gtr, gocc = drv.state(), drv.trace(), drv.occupancy()
    gp.check_errors()
    for r, n in enumerate(sizes):
        lat = O.Lattice(n)
        op, oe = O.Model(lat, path, els, O.PAIRSITE), O.Model(lat, path, els, O.ENERGY)
        c = O.Cmc(op, oe, lat, occs[r], 2500.0, 700.0, seed, replica=r)
        tr = c.run_omp(total, total, K, trace=True)
        ran = int(gst["steps"][r])
        assert ran == c.state()["steps"]
        assert np.array_equal(gtr["p"][r][:ran], tr["p"][:ran]) and np.array_equal(gtr["q"][r][:ran], tr["q"][:ran])
        np.testing.assert_allclose(gtr["de"][r][:ran], tr["de"][:ran], rtol=0, atol=TOL_E)
        assert np.array_equal(gtr["acc"][r][:ran], tr["acc"][:ran])
        assert np.array_equal(gocc[r], c.occupancy())
