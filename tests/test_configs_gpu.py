"""The benchmark workloads, run on the GPU through the C ABI and checked against the oracle:

* the single-replica 10^3-cell KMC (4000 sites, Al/Mg/Zn 3840/80/80, T = 500 K) for 2000 steps
  with the E0 and the Quartic barrier models, bit-exact event choice;
* the batched 1024 x 20^3-cell workload replayed from a HIP graph, eight sampled replicas
  replayed by the oracle;
* uneven-size batches (8, 11, 13 and 16 cells in one batch) for the three first-order kernel
  shapes and the chain shape, and canonical MC on 30^3-cell replicas at Al/Mg/Zn 90/5/5 under
  the linear 800 -> 300 K ramp;
* the surrogate's 12 x 1024-row inference batch: full fallback equals the plain path, energies
  stay exact with the specified fallback rule;
* 50^3-cell quaternary replicas (Al/Cu/Mg/Zn 94/2/2/2, T = 450 K);
* the early stop of KineticMcFirstAbstract::IsEscaped (KineticMcAbstract.cpp:192-223).

Bars as in the other parity tests: ids, event choice and occupancy bit-exact, energies within
1e-9 eV, time within 1e-12 relative.
"""
import numpy as np
import pytest

from conftest import QUATERNARY, TERNARY
from test_gpu_parity import TOL_E, _compare_kmc, _run_kmc_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


@pytest.fixture(scope="module")
def bench_coeffs(tmp_path_factory):
    """The workloads' synthetic coefficient files (reference JSON schema)."""
    from latticemontecarlo_amd import synth
    d = tmp_path_factory.mktemp("bench_coeffs")
    out = {}
    for name, els, kind in [("e0", TERNARY, "E0"), ("quartic", TERNARY, "Quartic"),
                            ("e0_q", QUATERNARY, "E0")]:
        p = str(d / f"{name}.json")
        synth.write_coefficients(p, els, kind, seed=2024)
        out[name] = (p, els)
    return out


def _alloy(n, species, counts, seed, vacancy=True):
    from latticemontecarlo_amd import synth
    return synth.random_occupancy(n, species, counts, seed=seed, vacancy=vacancy)


@pytest.mark.parametrize("model,kind", [("e0", 1), ("quartic", 2)])
def test_single_replica_10_cells_2000_steps(torch, bench_coeffs, model, kind):
    """10^3 cells, Al/Mg/Zn 3840/80/80 placed by a seeded shuffle, one vacancy, T = 500 K."""
    species = ["Al", "Mg", "X", "Zn"]
    occ = _alloy(10, species, {"Mg": 80, "Zn": 80}, seed=1)
    steps = 2000
    print(f"single replica 10^3 cells {model} {steps} steps", flush=True)
    gst, gtr, gocc, refs = _run_kmc_pair(bench_coeffs, model, kind, 10, 1, steps, 500.0, form=0,
                                         occs=[occ])
    _compare_kmc(gst, gtr, gocc, refs, steps)


def test_batched_1024_replicas_20_cells_graph(torch, bench_coeffs):
    """1024 replicas of 20^3 cells (Mg, Zn 1-5 at.% each, T 400-700 K) advanced by a replayed
    HIP graph; eight replicas spread over the batch are replayed by the oracle."""
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = bench_coeffs["e0"]
    gb = L.Model(path, els, L.E0)
    ge = L.Model(path, els, L.ENERGY)
    R, n, seed = 1024, 20, 2024
    rng = np.random.default_rng(seed)
    N = 4 * n ** 3
    occs, temps = [], []
    for r in range(R):
        xm, xz = rng.uniform(0.01, 0.05, 2)
        occs.append(_alloy(n, gb.species, {"Mg": round(xm * N), "Zn": round(xz * N)},
                           seed=seed * 100003 + r))
        temps.append(rng.uniform(400.0, 700.0))
    drv = L.KineticMcFirst(gb, ge, [n] * R, occs, np.array(temps), seed, maximum_steps=10 ** 12)
    drv.set_formulation(0)
    print("batched 1024 x 20^3: graph of 3 x 100 steps", flush=True)
    drv.build_graph(100, 3)
    drv.run_graph(100, 3)
    st, occ_now = drv.state(), drv.occupancy()
    gb.check_errors()
    assert np.all(st["steps"] == 300)
    lat = O.Lattice(n)
    ob, oe = O.Model(lat, path, els, O.E0), O.Model(lat, path, els, O.ENERGY)
    for r in np.linspace(0, R - 1, 8).astype(int):
        k = O.Kmc(ob, oe, lat, occs[r], temps[r], seed, replica=int(r))
        k.run(300)
        ost = k.state()
        assert int(st["vacancy"][r]) == ost["vacancy"], f"replica {r}"
        assert np.array_equal(occ_now[r], k.occupancy()), f"replica {r}"
        assert np.array_equal(st["disp"][r], ost["disp"])
        np.testing.assert_allclose(st["time"][r], ost["time"], rtol=1e-12)
        assert abs(st["energy"][r] - ost["energy"]) <= TOL_E * 300
        assert abs(st["abs_energy"][r] - ost["abs_energy"]) <= TOL_E * (300 + abs(ost["abs_energy"]))


def test_surrogate_12x1024_rows_full_fallback_and_exact_energies(torch, bench_coeffs):
    """The surrogate inference batch of 12 x 1024 event rows per step (1024 replicas of 20^3
    cells): with every event falling back, the trajectory is the plain path's (selections and
    occupancies equal, barriers within 1e-9 eV); with the specified fallback rule, the tracked
    energies stay those of the cluster expansion of the final configurations."""
    import latticemontecarlo_amd as L
    path, els = bench_coeffs["e0"]
    gb = L.Model(path, els, L.E0)
    ge = L.Model(path, els, L.ENERGY)
    R, n, seed, steps = 1024, 20, 2025, 60
    rng = np.random.default_rng(seed)
    N = 4 * n ** 3
    occs, temps = [], []
    for r in range(R):
        xm, xz = rng.uniform(0.01, 0.05, 2)
        occs.append(_alloy(n, gb.species, {"Mg": round(xm * N), "Zn": round(xz * N)},
                           seed=seed * 100003 + r))
        temps.append(rng.uniform(400.0, 700.0))
    temps = np.array(temps)
    sur = L.Surrogate(gb, n_members=4, seed=4)
    print("surrogate 1024 x 20^3: full fallback against plain", flush=True)
    a = L.KineticMcFirst(gb, ge, [n] * R, occs, temps, seed, maximum_steps=10 ** 12)
    b = L.KineticMcFirst(gb, ge, [n] * R, occs, temps, seed, maximum_steps=10 ** 12)
    a.set_formulation(0)
    b.set_surrogate(sur, threshold=-1.0)
    a.set_trace(steps)
    b.set_trace(steps)
    a.run(steps)
    b.run(steps)
    gb.check_errors()
    ta, tb = a.trace(), b.trace()
    assert np.array_equal(ta["sel"], tb["sel"])
    np.testing.assert_allclose(tb["ea"], ta["ea"], rtol=0, atol=1e-9)
    np.testing.assert_allclose(tb["de"], ta["de"], rtol=0, atol=1e-9)
    for x, y in zip(a.occupancy(), b.occupancy()):
        assert np.array_equal(x, y)
    st = b.surrogate_stats()
    assert st["events"] == 12 * R * steps and st["fallbacks"] == st["events"]
    del a, b
    # trained surrogate, specified rule: energies tracked through served steps stay exact
    print("surrogate 1024 x 20^3: trained, energies", flush=True)
    s_drv = L.KineticMcFirst(gb, None, [n] * R, occs, temps, seed + 1, maximum_steps=10 ** 12)
    E, K, D = [], [], []
    for _ in range(6):
        s_drv.run(8)
        e, k, d = s_drv.samples()
        E.append(e)
        K.append(k)
        D.append(d)
    env, ek, de = L.augment(torch.cat(E), torch.cat(K), torch.cat(D))
    del s_drv
    sur.train(env, ek, de, epochs=8, batch=4096, lr=3e-3, seed=1)
    c = L.KineticMcFirst(gb, ge, [n] * R, occs, temps, seed, maximum_steps=10 ** 12)
    c.set_surrogate(sur)
    c.run(steps)
    gb.check_errors()
    st = c.state()
    final = c.occupancy()
    e_final = L.total_energy(ge, L.ReplicaBatch([n] * R, final)).cpu().numpy()
    np.testing.assert_allclose(st["abs_energy"], e_final, rtol=0,
                               atol=TOL_E * steps + 1e-12 * np.abs(e_final).max())
    s2 = c.surrogate_stats()
    print(f"served {s2['events'] - s2['fallbacks']} of {s2['events']} events", flush=True)
    assert s2["events"] == 12 * R * steps and s2["fallbacks"] < s2["events"]


@pytest.mark.parametrize("form", [0, 1, 2, 3])
def test_uneven_size_batch_matches_oracle(torch, coeffs, form):
    """Replicas of 8, 11, 13 and 16 cells (and 9 twice) in one batch: per-replica offsets and box
    sizes with one wave per replica (1), four (0, 2) and in chain steps (3)."""
    sizes = [8, 11, 13, 16, 9, 9]
    steps = 100 if form == 3 else 300
    print(f"uneven sizes {sizes} form {form}", flush=True)
    gst, gtr, gocc, refs = _run_kmc_pair(coeffs, "e0_3n", 1, sizes, len(sizes), steps,
                                         np.linspace(450.0, 700.0, len(sizes)), form=form)
    _compare_kmc(gst, gtr, gocc, refs, steps)


def test_uneven_size_quartic_batch_matches_oracle(torch, coeffs):
    sizes = [7, 12, 10, 5]
    steps = 250
    print(f"uneven sizes {sizes} quartic", flush=True)
    gst, gtr, gocc, refs = _run_kmc_pair(coeffs, "q_3n", 2, sizes, len(sizes), steps, 600.0,
                                         form=0, rate_corrector=True, solute_disp=True)
    _compare_kmc(gst, gtr, gocc, refs, steps)


def test_canonical_mc_30_cells_ramp(torch, bench_coeffs):
    """CanonicalMc on 30^3-cell replicas (108000 sites) at Al/Mg/Zn 90/5/5, T linear 800 -> 300 K
    over the run's trials, occupancy in LDS."""
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = bench_coeffs["e0"]
    n, R, trials = 30, 3, 3000
    N = 4 * n ** 3
    gp = L.Model(path, els, L.PAIRSITE)
    occs = [_alloy(n, gp.species, {"Mg": round(0.05 * N), "Zn": round(0.05 * N)}, seed=11 * 7 + r,
                   vacancy=False) for r in range(R)]
    seed = 2024
    print(f"canonical MC {R} x {n}^3, {trials} trials", flush=True)
    drv = L.CanonicalMc(gp, None, [n] * R, occs, 800.0, 300.0, seed, maximum_steps=trials)
    drv.set_trace(trials)
    drv.run(trials)
    gtr, gst, gocc = drv.trace(), drv.state(), drv.occupancy()
    lat = O.Lattice(n)
    op = O.Model(lat, path, els, O.PAIRSITE)
    for r in range(R):
        c = O.Cmc(op, None, lat, occs[r], 800.0, 300.0, seed, replica=r)
        tr = c.run(trials, trials, trace=True)
        assert np.array_equal(gtr["p"][r], tr["p"]) and np.array_equal(gtr["q"][r], tr["q"])
        assert np.array_equal(gtr["acc"][r], tr["acc"])
        np.testing.assert_allclose(gtr["de"][r], tr["de"], rtol=0, atol=TOL_E)
        assert np.array_equal(gocc[r], c.occupancy())
        assert int(gst["accepted"][r]) == c.state()["accepted"]


def _site_id(n, X, Y, Z):
    """x-major lattice id of the site at (X, Y, Z) in a/2 units (X + Y + Z even)."""
    return X * 2 * n * n + Y * n + Z // 2


def _window(occ_big, n, m, corner):
    """The occupancy of the m^3-cell box whose site (x, y, z) is the n^3-cell box's site
    corner + (x, y, z) (no wrap: the window lies inside the big box)."""
    X0, Y0, Z0 = corner
    x, y, z = np.meshgrid(np.arange(2 * m), np.arange(2 * m), np.arange(2 * m), indexing="ij")
    on = (x + y + z) % 2 == 0
    x, y, z = x[on], y[on], z[on]
    out = np.zeros(4 * m ** 3, np.uint8)
    out[_site_id(m, x, y, z)] = occ_big[_site_id(n, x + X0, y + Y0, z + Z0)]
    return out


def test_quaternary_50_cells(torch, bench_coeffs):
    """Two 50^3-cell replicas (500000 sites) of Al/Cu/Mg/Zn 94/2/2/2 at 450 K, 150 steps.

    The oracle restates the reference's tolerance geometry, which cannot build a 50^3-cell box:
    its fractional shell gap 1/(4 n^2) reaches the 1e-4 comparison tolerance at n = 50, and the
    orbit construction then runs past the feature vector. Each big replica is therefore checked
    against the oracle on a 20^3-cell box holding the same local configuration around the
    vacancy: while the vacancy stays 4 a/2 steps inside that window, no environment site wraps
    in either box, the 12 neighbours sort alike, and both trajectories must agree jump for jump.
    """
    import latticemontecarlo_amd as L
    import oracle as O
    path, els = bench_coeffs["e0_q"]
    species = ["Al", "Cu", "Mg", "X", "Zn"]
    n, m, steps, seed = 50, 20, 150, 2024
    N = 4 * n ** 3
    c = round(0.02 * N)
    x = species.index("X")
    vac_xyz = [(50, 51, 49), (37, 60, 55)]
    occs = []
    for r, (X, Y, Z) in enumerate(vac_xyz):
        occ = _alloy(n, species, {"Cu": c, "Mg": c, "Zn": c}, seed=seed * 100003 + r)
        v, w = int(np.flatnonzero(occ == x)[0]), _site_id(n, X, Y, Z)
        occ[v], occ[w] = occ[w], x
        occs.append(occ)
    gb = L.Model(path, els, L.E0)
    print(f"quaternary 2 x {n}^3, {steps} steps", flush=True)
    drv = L.KineticMcFirst(gb, None, [n] * 2, occs, 450.0, seed, maximum_steps=10 ** 9)
    drv.set_formulation(2)
    drv.set_trace(steps)
    drv.run(steps)
    gtr, gst, gocc = drv.trace(), drv.state(), drv.occupancy()
    gb.check_errors()
    lat = O.Lattice(m)
    ob = O.Model(lat, path, els, O.E0)
    for r, (X, Y, Z) in enumerate(vac_xyz):
        corner = (X - m, Y - m, Z - m)
        small = _window(occs[r], n, m, corner)
        k = O.Kmc(ob, None, lat, small, 450.0, seed, replica=r)
        tr = k.run(steps, trace=True)
        # the oracle's path stays inside the window's wrap-free core
        path_xyz = np.array([lat.position(int(s)) * 2 * m for s in tr["sel"]]).round().astype(int)
        assert np.abs(path_xyz - m).max() <= m - 4, "the test's seeds keep the vacancy in the window"
        big_sel = _site_id(n, path_xyz[:, 0] + corner[0], path_xyz[:, 1] + corner[1],
                           path_xyz[:, 2] + corner[2])
        assert np.array_equal(gtr["sel"][r], big_sel), f"replica {r}"
        np.testing.assert_allclose(gtr["ea"][r], tr["ea"], rtol=0, atol=TOL_E)
        np.testing.assert_allclose(gtr["de"][r], tr["de"], rtol=0, atol=TOL_E)
        np.testing.assert_allclose(gtr["time"][r], tr["time"], rtol=1e-12)
        assert np.array_equal(_window(gocc[r], n, m, corner), k.occupancy())
        assert int(gst["steps"][r]) == steps


def _escape_start(n, species, seed):
    """A dilute alloy whose vacancy starts with three Mg atoms among its first neighbours, so
    that it escapes (all 1-3NN sites solvent) only after some steps."""
    import oracle as O
    occ = _alloy(n, species, {"Mg": 4 * n ** 3 // 100, "Zn": 4 * n ** 3 // 100}, seed=seed)
    x = species.index("X")
    v = int(np.flatnonzero(occ == x)[0])
    nb = O.Lattice(n).neighbors(v, 1)
    mg = species.index("Mg")
    for s in nb[:3]:
        occ[s] = mg
    return occ


@pytest.mark.parametrize("form", [0, 1, 2, 3])
def test_early_stop_matches_oracle(torch, coeffs, form):
    """early_stop: the step that finds every 1-3NN site of the vacancy solvent sets steps to
    maximum_steps + 1, still applies its jump, and the replica stops (KineticMcAbstract.cpp:
    140-190, 192-223). Steps, time, energy, occupancy and the trace up to the stop match."""
    path, els = coeffs["e0_3n"]
    import latticemontecarlo_amd as L
    species = L.Model(path, els, L.E0).species
    n, R, steps, maxs = 6, 5, 400, 10 ** 6
    occs = [_escape_start(n, species, 40 + r) for r in range(R)]
    print(f"early stop form {form}", flush=True)
    gst, gtr, gocc, refs, esc = _run_kmc_pair(coeffs, "e0_3n", 1, n, R, steps,
                                              np.linspace(450.0, 650.0, R), form=form,
                                              maximum_steps=maxs, occs=occs, early_stop=True,
                                              escape_info=True)
    escaped = 0
    for r, (st, tr, occ) in enumerate(refs):
        assert int(gst["escaped"][r]) == int(st["escaped"]), f"replica {r}"
        assert int(gst["steps"][r]) == st["steps"]
        if st["escaped"]:
            escaped += 1
            assert st["steps"] == maxs + 2
        ran = int(np.count_nonzero(gtr["sel"][r] >= 0))
        assert ran == int(np.count_nonzero(tr["time"])), f"replica {r}"
        assert ran >= 1 and (st["escaped"] or ran == steps)
        assert np.array_equal(gtr["sel"][r][:ran], tr["sel"][:ran].astype(np.int64))
        assert np.all(gtr["sel"][r][ran:] == -1)
        np.testing.assert_allclose(gtr["ea"][r][:ran], tr["ea"][:ran], rtol=0, atol=TOL_E)
        np.testing.assert_allclose(gtr["time"][r][:ran], tr["time"][:ran], rtol=1e-12)
        assert np.array_equal(gocc[r], occ)
        assert int(gst["vacancy"][r]) == st["vacancy"]
        np.testing.assert_allclose(gst["time"][r], st["time"], rtol=1e-12)
        assert abs(gst["energy"][r] - st["energy"]) <= TOL_E * steps
        if st["escaped"]:  # the escape check's moment: before the last step's jump
            v0 = int(np.flatnonzero(occs[r] == species.index("X"))[0])
            assert int(esc["step"][r]) == ran - 1
            assert int(esc["site_before"][r]) == (int(tr["sel"][ran - 2]) if ran > 1 else v0)
            t_before = tr["time"][ran - 2] if ran > 1 else 0.0
            np.testing.assert_allclose(esc["t_exit"][r], t_before, rtol=1e-12)
        else:
            assert int(esc["site_before"][r]) == -1
    assert escaped >= 3, "the start configurations are built to escape within the run"


@pytest.mark.parametrize("name,kind,record", [("e0_3n", 1, False), ("q_3n", 2, True)])
def test_occupancy_window_long_trajectories(torch, coeffs, name, kind, record):
    """1500 steps on boxes of 8, 9 and 12 cells, in which the vacancy crosses the box many times; with atom
    tracking and the log compiled in (record) or not."""
    import latticemontecarlo_amd as L
    sizes = [8, 8, 9, 12]
    steps = 1500
    opts = {}
    print(f"window {name} record={record}", flush=True)
    if not record:
        gst, gtr, gocc, refs = _run_kmc_pair(coeffs, name, kind, sizes, len(sizes), steps,
                                             np.array([450.0, 700.0, 550.0, 600.0]), form=0)
        _compare_kmc(gst, gtr, gocc, refs, steps)
        return
    import oracle as O
    path, els = coeffs[name]
    gb = L.Model(path, els, kind)
    species = gb.species
    from conftest import random_alloc
    occs = [random_alloc(n, species, 0.06, seed=800 + r) for r, n in enumerate(sizes)]
    drv = L.KineticMcFirst(gb, None, sizes, occs, 600.0, 77, maximum_steps=10 ** 9)
    drv.set_formulation(0)
    l2a = [np.arange(4 * n ** 3) for n in sizes]
    drv.set_atoms(l2a)
    drv.set_log(50, capacity=1000)
    drv.set_trace(steps)
    drv.run(steps)
    gtr, gocc = drv.trace(), drv.occupancy()
    for r, n in enumerate(sizes):
        lat = O.Lattice(n)
        ob = O.Model(lat, path, els, kind)
        k = O.Kmc(ob, None, lat, occs[r], 600.0, 77, replica=r)
        tr = k.run(steps, trace=True)
        assert np.array_equal(gtr["sel"][r], tr["sel"].astype(np.int64)), f"replica {r}"
        np.testing.assert_allclose(gtr["ea"][r], tr["ea"], rtol=0, atol=TOL_E)
        assert np.array_equal(gocc[r], k.occupancy())
