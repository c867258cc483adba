"""The energy of a small batch's trajectories, bit for bit: every jump's change is the sum over the state
clusters in list order (84 running sums of every 84th cluster; the four sums 21 apart added two and
two, then the 21 results one after another), and the energy is their sum in step order. A trajectory
whose changes cancel leaves nothing but the rounding of these sums, which another order would not
reproduce."""
import json

import numpy as np
import pytest

from conftest import random_alloc

pytestmark = pytest.mark.gpu

NORM = (256, 1536, 768, 3072, 2048, 3072, 6144, 6144)


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


class Ordered:
    def __init__(self, path, model):
        theta = json.load(open(path))["Base"]["theta"]
        self.weight = {(int(lab), tuple(int(c) for c in codes)): theta[i] / NORM[int(lab)]
                       for i, (lab, codes) in enumerate(model.eci_keys())}
        self.x = model.species.index("X")

    def de(self, n, occ, v, nb):
        """Energy change of the vacancy's jump v -> nb in occ."""
        import latticemontecarlo_amd as L
        rows = [[int(x) for x in row] for row in L.jump_state_clusters(n, v, nb)]
        mig = int(occ[nb])
        values = []
        for end, other, sign in ((v, nb, 1), (nb, v, -1)):
            for lab, *sites in rows:
                if end not in sites or other in sites:
                    continue
                rest = [int(occ[s]) for s in sites if s >= 0 and s != end]
                w = [self.weight[(lab, tuple(sorted(rest + [c])))] for c in (mig, self.x)]
                values.append(sign * (w[0] - w[1]))
        assert len(values) == 452
        a = np.zeros((6, 4, 21))
        a.reshape(-1)[:452] = values
        sums = np.zeros((4, 21))
        for batch in a:
            sums = sums + batch
        lanes = (sums[0] + sums[1]) + (sums[2] + sums[3])
        total = 0.0
        for p in lanes:
            total += float(p)
        return total


@pytest.mark.parametrize("form", [0, 2, 3])
@pytest.mark.parametrize("name,kind,sizes,solute,full", [
    ("e0_3n", 1, [7], 0.0, False),       # pure solvent: every change is zero but for its rounding
    ("q_3n", 2, [8], 0.01, True),        # log and atoms, the Quartic model
    ("e0_4n", 1, [6, 9, 7], 0.06, False),
    ("e0_4n", 1, [6, 5], 0.2, True),     # environments past the sparse limit
])
def test_energies_are_the_ordered_cluster_sums(torch, coeffs, tmp_path, name, kind, sizes, solute, full, form):
    import latticemontecarlo_amd as L
    path, els = coeffs[name]
    model = L.Model(path, els, kind)
    occs = [random_alloc(n, model.species, solute, seed=40 + n) for n in sizes]
    R, steps = len(sizes), 40
    drv = L.KineticMcFirst(model, None, sizes, occs, 600.0, 11, maximum_steps=10 ** 6)
    drv.set_formulation(form)
    drv.set_trace(steps)
    if full:
        drv.set_atoms([np.arange(4 * n ** 3) for n in sizes])
        drv.set_log(10, capacity=1000)
    drv.run(1)
    drv.run(steps - 1)
    st, tr = drv.state(), drv.trace()
    exact = Ordered(path, model)
    for r, n in enumerate(sizes):
        occ = occs[r].copy()
        v = int(np.flatnonzero(occ == exact.x)[0])
        energy, before, want = 0.0, [], []
        for s in range(steps):
            nb = int(tr["sel"][r, s])
            mig = occ[nb]
            if form == 3:  # the reverse of the jump nb -> v after the jump
                occ[v], occ[nb] = mig, exact.x
                want.append(-exact.de(n, occ, nb, v))
            else:
                want.append(exact.de(n, occ, v, nb))
                occ[v], occ[nb] = mig, exact.x
            before.append(energy)
            energy += want[-1]
            v = nb
        assert v == int(st["vacancy"][r])
        assert tr["de"][r].tolist() == want, f"replica {r}"
        assert float(st["energy"][r]) == energy and float(st["abs_energy"][r]) == energy
        if solute == 0.0:
            assert max(map(abs, want)) < 1e-13
        if full and r == 0:
            files = [None] * R
            files[r] = str(tmp_path / "log.txt")
            drv.write_log(files)
            head, *lines = [x.split("\t") for x in open(files[r]).read().strip().split("\n")]
            assert len(lines) == steps
            for x in lines:  # printed with fewer digits
                s = int(x[0])
                assert float(x[head.index("energy")]) == pytest.approx(before[s], rel=1e-4, abs=1e-9)
                assert float(x[head.index("dE")]) == pytest.approx(want[s], rel=1e-4, abs=1e-9)
