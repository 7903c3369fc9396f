"""Stable dt of lists larger than one pass of the reduction's grid (more than
2048 blocks of 256 cells) and of lists of a few cells: the fastest cell in the
first, last or a middle cell of any patch decides, bit for bit as the oracle."""
import numpy as np
import pytest

from hamers_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", [0, 1, 2, 3])
@pytest.mark.parametrize("ns", [[(1100, 700), (5, 3), (63, 65)], [(1, 1), (3, 2)]], ids=["large", "tiny"])
def test_fastest_cell_anywhere(ns, where):
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, PatchData
    from hamers_amd.reconstructor import computeSpectralRadiusesAndStableDtOnPatches

    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    rng = np.random.default_rng(where)
    g, dx = 4, (0.01, 0.02)
    Qs = []
    for i, n in enumerate(ns):
        shp = (n[1] + 2 * g, n[0] + 2 * g)
        rho, vel = 0.5 + rng.random(shp), [rng.normal(size=shp) for _ in range(2)]
        if where < 3 and i == (0 if where < 2 else len(ns) - 1):
            j, k = ((0, 0), (n[1] - 1, n[0] - 1), (n[1] // 2, n[0] // 2))[where]
            vel[where % 2][g + j, g + k] = 30.0
        Qs.append(W.conservative_from_primitive_single(rho, vel, 0.2 + rng.random(shp), 1.4))
    rec = ConvectiveFluxReconstructor("dt", 2, "SINGLE_SPECIES", "WCNS6_LD_HLLC_HLL", species_gamma=(1.4,), species_R=(1.0,))
    prm = O.Params(dim=2, scheme=1)
    refs = [O.spectral_radiuses_and_dt(prm, Q, n, g, dx) for Q, n in zip(Qs, ns)]
    pds = [PatchData(n, (g, g), dx, torch.from_numpy(Q).to("cuda:0"),
                     [torch.empty(O.face_shape(4, n, a), dtype=torch.float64, device="cuda:0") for a in range(2)], None)
           for Q, n in zip(Qs, ns)]
    got = computeSpectralRadiusesAndStableDtOnPatches(rec, pds)
    print(f"{ns} where {where}: {got}", flush=True)
    assert got == [max(r[a] for r in refs) for a in range(2)] + [min(r[2] for r in refs), O.level_dt(refs)]
