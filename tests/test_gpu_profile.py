"""Stage timing (hm_profile_enable): the launches it counts are those the call
makes without it.  A batched single-species call takes both flux stages in one
launch with 4- or 8-row tiles and in two with 24-row ones, the multi-species
models in one, and two under the persistent schedule; a small per-patch call
has the flux alone.  Outputs are the same bits with the timing on and off."""
import sys

import numpy as np
import pytest

from hamers_amd import workloads as W

pytestmark = pytest.mark.gpu


def _patches(torch, rec, Qi, n, dx, count):
    from hamers_amd import PatchData
    from oracle import oracle as O

    Q = torch.from_numpy(W.fill_periodic(Qi, 4)).to("cuda:0")
    out = []
    for _ in range(count):
        F = [torch.zeros(O.face_shape(rec.num_eqn, n, a), dtype=torch.float64, device="cuda:0") for a in range(len(n))]
        S = torch.zeros((rec.num_eqn,) + tuple(reversed(n)), dtype=torch.float64, device="cuda:0")
        out.append(PatchData(n, (4,) * len(n), dx, Q, F, S))
    return out


def _flux(pds):
    return [f.cpu().numpy() for pd in pds for f in pd.F]


def _check(torch, rec, pds, call, launches):
    call()
    torch.cuda.synchronize()
    plain = _flux(pds)
    rec.enable_profiling(True)
    call()
    prof = rec.read_profile()
    rec.enable_profiling(False)
    print({k: v for k, v in prof.items()}, flush=True)
    assert tuple(prof[s][1] for s in rec.STAGES) == launches
    assert all((ms > 0.0) == (n > 0) for ms, n in prof.values())
    assert all(np.array_equal(a, b) for a, b in zip(plain, _flux(pds)))


@pytest.mark.parametrize("rows,launches", [(4, (1, 0, 1, 0, 0)), (8, (1, 0, 1, 0, 0)), (24, (1, 0, 1, 1, 0))])
@pytest.mark.parametrize("dim", [2, 3])
def test_single_species_batch(dim, rows, launches):
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, PatchList
    from hamers_amd.reconstructor import set_schedule

    Qi, n, dx = W.density_wave_convergence(16, dim=dim)
    print(f"case: {dim}D, tiles of {rows} rows", flush=True)
    sys.stdout.flush()
    rec = ConvectiveFluxReconstructor("profile", dim, "SINGLE_SPECIES", "WCNS6_LD_HLLC_HLL")
    pds = _patches(torch, rec, Qi, n, dx, 3)
    plist = PatchList(pds, rec.num_arrays)
    set_schedule(rec, plist, {"tile_rows": rows, "xcd_remap": 1, "order": 0})
    _check(torch, rec, pds, lambda: rec.computeConvectiveFluxAndSourceOnPatches(plist, 0.0, 1e-3), launches)


@pytest.mark.parametrize("persistent,launches", [(0, (1, 0, 1, 0, 1)), (1, (1, 0, 1, 1, 1))])
def test_five_equation_batch(persistent, launches):
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, PatchList
    from hamers_amd.reconstructor import set_schedule

    Qi, n, dx = W.interface_advection_convergence(8, dim=3)
    print(f"case: five-equation, persistent {persistent}", flush=True)
    rec = ConvectiveFluxReconstructor("profile", 3, "FIVE_EQN_ALLAIRE", "WCNS5_JS_HLLC_HLL", num_species=2,
                                      species_gamma=(1.6, 1.4), species_R=(1.0, 1.0))
    pds = _patches(torch, rec, Qi, n, dx, 2)
    plist = PatchList(pds, rec.num_arrays)
    set_schedule(rec, plist, {"tile_rows": 4, "xcd_remap": 1, "order": 0, "persistent": persistent})
    _check(torch, rec, pds, lambda: rec.computeConvectiveFluxAndSourceOnPatches(plist, 0.0, 1e-3), launches)


def test_small_patch():
    import torch

    from hamers_amd import ConvectiveFluxReconstructor

    Qi, n, dx = W.density_wave_convergence(16, dim=2)
    print("case: one 16^2 patch", flush=True)
    rec = ConvectiveFluxReconstructor("profile", 2, "SINGLE_SPECIES", "WCNS5_JS_HLLC_HLL")
    pds = _patches(torch, rec, Qi, n, dx, 1)
    _check(torch, rec, pds, lambda: rec.computeConvectiveFluxAndSourceOnPatch(pds[0], 0.0, 1e-3), (0, 0, 1, 0, 0))
