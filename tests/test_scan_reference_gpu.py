"""Scans of frames with another base metal: the sums run about the species that the caller names, whose
tables are formed at its first scan, also while the caller's stream is being captured. Against the oracle."""
import numpy as np
import pytest

from conftest import random_alloc
from test_exit_time import _oracle_scan

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("name,kind,base,solute", [("e0_3n", 1, "Mg", 0.08), ("e0_3n", 1, "Zn", 0.08),
                                                   ("q_4", 2, "Mg", 0.08), ("q_4", 2, "Cu", 0.25)])
def test_scan_of_another_base_metal(torch, coeffs, name, kind, base, solute, captured):
    import latticemontecarlo_amd as L
    import oracle as O
    from latticemontecarlo_amd import capi
    path, els = coeffs[name]
    n = 6
    gm = L.Model(path, els, kind)
    sp = gm.species
    occ = random_alloc(n, sp, solute, seed=72)
    al, code = sp.index("Al"), sp.index(base)
    occ = np.where(occ == al, code, np.where(occ == code, al, occ)).astype(np.uint8)
    vac = int(np.flatnonzero(occ == sp.index("X"))[0])
    sites = [vac] + [int(s) for s in np.random.default_rng(6).choice(4 * n ** 3, 11, replace=False)]
    d = torch.from_numpy(occ).cuda()
    L.api.vacancy_scan(gm, d, n, vac, al, sites)  # the model's tables, about its default species
    K = len(sites)
    s = torch.tensor(sites).cuda()
    nb = torch.zeros((K, 12), dtype=torch.int64, device="cuda")
    ea, de = (torch.zeros((K, 12), dtype=torch.float64, device="cuda") for _ in range(2))

    def scan(stream):
        capi.check(capi.lib().lmc_vacancy_scan(gm.h, capi.dptr(d), n, vac, code, capi.dptr(s), K, capi.dptr(nb),
                                               capi.dptr(ea), capi.dptr(de), capi.stream_ptr(stream)))

    print(f"scan about {base}: {name} n={n} sites={K} captured={captured}", flush=True)
    torch.cuda.synchronize()
    if captured:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            scan(torch.cuda.current_stream())
        assert not nb.any()
        graph.replay()
    else:
        scan(None)
    torch.cuda.synchronize()
    gm.check_errors()
    om = O.Model(O.Lattice(n), path, els, kind)
    ref = _oracle_scan(om, occ, vac, code, sp.index("X"), sites, n)
    nb, ea, de = nb.cpu().numpy(), ea.cpu().numpy(), de.cpu().numpy()
    for i, rows in enumerate(ref):
        for j, (rnb, rea, rde) in enumerate(rows):
            assert nb[i, j] == rnb
            assert abs(ea[i, j] - rea) <= 1e-9 and abs(de[i, j] - rde) <= 1e-9, (i, j)
