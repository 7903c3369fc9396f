"""Tiles of the fused multi-species flux: the block-uniform column arithmetic
(the kernel's multiplications in place of divisions) visits every midpoint face
and writes every output face once for all small extents (on the CPU), and
patches whose tiles wrap over several rows, hold single columns or end part
filled equal the oracle (on the GPU)."""
import numpy as np
import pytest

from hamers_amd import workloads as W
from oracle import oracle as O


def _shape(nA):
    """mtile_shape of hm_kernels.hpp."""
    nt = (nA + 1 + 61) // 62
    R = (nA + 1 + nt - 1) // nt + 2
    return R, 256 // R, nt


def _mul(d):
    return (65536 + d - 1) // d


def test_small_divisions_are_exact():
    x = np.arange(256)
    for d in range(1, 257):
        assert np.array_equal((x * _mul(d)) >> 16, x // d), d
    # column wrap: cu < nU + W < 256 with nU < W <= 85
    for nU in range(1, 85):
        x = np.arange(nU + 85)
        assert np.array_equal((x * _mul(nU)) >> 16, x // nU), nU


@pytest.mark.parametrize("axis", [0, 1])
def test_tiles_cover_every_face_once(axis):
    lane = np.arange(256)
    for nA in (1, 2, 7, 8, 61, 62, 64, 123, 124, 125, 200):
        R, Wd, nt = _shape(nA)
        assert R * Wd <= 256
        for nU, nV in ((1, 1), (1, 9), (3, 5), (8, 8), (Wd, 2), (Wd + 1, 3), (200, 1)):
            first = (lane * _mul(R if axis == 0 else Wd)) >> 16
            rest = lane - first * (R if axis == 0 else Wd)
            w, r = (first, rest) if axis == 0 else (rest, first)
            out = np.zeros((nU * nV, nA + 1), dtype=int)
            mid = np.zeros((nU * nV, nA + 3), dtype=int)
            tiles = nt * -(-nU * nV // Wd)
            for tile in range(tiles):
                tw, tA = tile // nt, tile % nt
                j = tA * (R - 2) + r
                t0 = tw * Wd
                v0 = t0 // nU
                cu = t0 - v0 * nU + w
                if nU >= Wd:
                    over = cu >= nU
                    tv, cu = v0 + over, cu - over * nU
                else:
                    q = (cu * _mul(nU)) >> 16
                    tv, cu = v0 + q, cu - q * nU
                inside = (lane < R * Wd) & (j < nA + 3) & (tv < nV)
                col = tv * nU + cu
                mid[col[inside], j[inside]] += 1
                writes = inside & (r >= 1) & (r <= R - 2) & (j <= nA + 1)
                np.add.at(out, (col[writes], j[writes] - 1), 1)
            assert np.all(out == 1), (nA, nU, nV)
            assert np.all(mid >= 1), (nA, nU, nV)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", [1, 0], ids=["WCNS6_LD", "WCNS5_JS"])
@pytest.mark.parametrize("model", ["FIVE_EQN_ALLAIRE", "FOUR_EQN_CONSERVATIVE"])
@pytest.mark.parametrize("n", [(3, 2, 70), (130, 1, 5), (1, 1, 9), (64, 65, 2), (5, 63, 4)])
def test_tile_shapes_against_oracle(n, model, scheme):
    """Same bits as the oracle, batched and per patch (ghost width 5, so the caller's box differs from the scratch box)."""
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, PatchData

    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    five, g, gamma = model == "FIVE_EQN_ALLAIRE", 5, (1.4, 1.67)
    rng = np.random.default_rng(sum(n))
    shp = tuple(v + 2 * g for v in reversed(n))
    z, y, x = np.meshgrid(*[np.linspace(0, 1, s) for s in shp], indexing="ij")
    Z1 = 0.5 + 0.45 * np.sin(2 * np.pi * (x + y + z)) * rng.uniform(0.9, 1, shp)
    vel = [0.3 * np.sin(2 * np.pi * (y + b * z)) + 0.1 * rng.uniform(-1, 1, shp) for b in range(3)]
    p = 1.0 + 0.5 * rng.uniform(0, 1, shp) + (x > 0.5)
    if five:
        Q = W.conservative_from_primitive_five([Z1, 0.3 * (1 - Z1)], vel, p, [Z1, 1 - Z1], gamma)
    else:
        Q = W.conservative_from_primitive_four([Z1, 0.3 * (1 - Z1)], vel, p, gamma, (1.0, 2.0))
    dx, dt = tuple(1.0 / v for v in n), 1e-3
    rec = ConvectiveFluxReconstructor("tiles", 3, model, "WCNS6_LD_HLLC_HLL" if scheme else "WCNS5_JS_HLLC_HLL",
                                      num_species=2, species_gamma=gamma, species_R=(1.0, 1.0 if five else 2.0))
    prm = O.Params(dim=3, model=O.FIVE_EQN_ALLAIRE if five else O.FOUR_EQN_CONSERVATIVE, num_species=2, scheme=scheme,
                   gamma=list(gamma), R=[1.0, 1.0 if five else 2.0])
    Fr, Sr = O.rhs_patch(prm, Q, n, g, dx, dt)
    for batched in (False, True):
        F = [torch.full(O.face_shape(rec.num_eqn, n, a), np.nan, dtype=torch.float64, device="cuda:0") for a in range(3)]
        S = torch.zeros((rec.num_eqn,) + tuple(reversed(n)), dtype=torch.float64, device="cuda:0")
        pd = PatchData(n, (g,) * 3, dx, torch.from_numpy(Q).to("cuda:0"), F, S)
        if batched:
            rec.computeConvectiveFluxAndSourceOnPatches([pd], 0.0, dt)
        else:
            rec.computeConvectiveFluxAndSourceOnPatch(pd, 0.0, dt)
        torch.cuda.synchronize()
        print(f"{model} {n} scheme {scheme} batched {batched}", flush=True)
        for a in range(3):
            assert np.array_equal(F[a].cpu().numpy(), Fr[a]), a
        assert np.array_equal(S.cpu().numpy(), Sr)
