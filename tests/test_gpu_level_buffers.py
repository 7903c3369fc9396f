"""A level's stage buffers: steps of a level whose patches leave ghost cells
uncovered (an L-shaped union, one patch alone, patches two cells wide) keep the
caller's values there in every stage, steps through a hierarchy (which keeps
the start state) and on their own agree, and one-stage, two-stage and
three-stage tableaux give the oracle's steps of the ghosted domain."""
import numpy as np
import pytest

from hamers_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TABLEAUX = {"euler": (((1.0,),), ((1.0,),)),
            "heun": (((1.0,), (1.0, 0.0)), ((1.0,), (0.5, 0.5))),
            "ssp3": (((1.0,), (0.75, 0.25), (1 / 3, 0.0, 2 / 3)), ((1.0,), (0.0, 0.25), (0.0, 0.0, 2 / 3)))}


def _domain(n, g, seed):
    rng = np.random.default_rng(seed)
    shp = (n[1] + 2 * g, n[0] + 2 * g)
    y, x = np.meshgrid(*[np.arange(s) / s for s in shp], indexing="ij")
    rho = 1.0 + 0.3 * np.sin(2 * np.pi * (x + y)) + 0.02 * rng.random(shp)
    vel = [0.4 * np.cos(2 * np.pi * y), 0.3 * np.sin(2 * np.pi * x)]
    return W.conservative_from_primitive_single(rho, vel, 1.0 + 0.2 * rng.random(shp), 1.4)


@pytest.mark.parametrize("tableau", sorted(TABLEAUX))
@pytest.mark.parametrize("boxes", [[((0, 0), (20, 12)), ((0, 12), (9, 14))], [((3, 2), (17, 11))], [((0, 0), (2, 30)), ((2, 0), (13, 30))]],
                         ids=["ell", "lone", "thin"])
def test_uncovered_ghosts_keep_their_values(boxes, tableau):
    """Against the oracle on each patch's ghost box: same-level ghosts from the stage state, the others constant in time."""
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, Level

    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    n, g = (32, 32), 4
    dx, dt = (1 / 32, 1 / 32), 2e-3
    whole = _domain(n, g, 5)
    rec = ConvectiveFluxReconstructor("buf", 2, "SINGLE_SPECIES", "WCNS6_LD_HLLC_HLL", species_gamma=(1.4,))
    al, be = TABLEAUX[tableau]
    lvl = Level(rec, boxes, ((0, 0), n), (0, 0), dx)
    lvl.set_rk_coefficients(al, be)

    class View:
        def __init__(self, ptr, shape):
            self.owner = lvl
            self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (ptr, False), "version": 3}

    cut = lambda A, lo, m: A[:, lo[1]:lo[1] + m[1] + 2 * g, lo[0]:lo[0] + m[0] + 2 * g]  # noqa: E731
    for i, (lo, m) in enumerate(boxes):
        ptr, gg = lvl.patch_array(i)
        assert gg == g
        t = torch.as_tensor(View(ptr, (4, m[1] + 2 * g, m[0] + 2 * g)), device="cuda:0")
        t.copy_(torch.from_numpy(np.ascontiguousarray(cut(whole, lo, m))))
    prm = O.Params(dim=2, scheme=1)
    state = whole.copy()
    for step in range(2):
        U, L = [state], []
        for a, b in zip(al, be):
            src = U[-1]
            Ls = {}
            for lo, m in boxes:
                F, S = O.rhs_patch(prm, np.ascontiguousarray(cut(src, lo, m)), m, g, dx, dt)
                t = -(F[0][:, :, 1:] - F[0][:, :, :-1]) / dx[0] - (F[1][:, 1:] - F[1][:, :-1]) / dx[1]
                Ls[lo] = t + S
            L.append(Ls)
            new = state.copy()  # cells no patch holds keep the caller's values
            for lo, m in boxes:
                q = np.zeros((4, m[1], m[0]))
                inner = np.s_[:, g + lo[1]:g + lo[1] + m[1], g + lo[0]:g + lo[0] + m[0]]
                for k in range(len(a)):
                    if a[k]:
                        q = q + a[k] * U[k][inner]
                    if b[k]:
                        q = q + b[k] * L[k][lo]
                new[inner] = q
            U.append(new)
        state = U[-1]
        lvl.advance(dt, 1, use_graph=bool(step))
    torch.cuda.synchronize()
    for i, (lo, m) in enumerate(boxes):
        want = state[:, g + lo[1]:g + lo[1] + m[1], g + lo[0]:g + lo[0] + m[0]]
        got = lvl.read_patch(i)
        print(f"{tableau} patch {i}: max diff {np.abs(got - want).max():.3e}", flush=True)
        assert np.array_equal(got, want)


def test_levels_of_a_hierarchy_step_alone_as_before():
    """A coarse level keeps its start state in a hierarchy; on its own it steps as a level that never was in one."""
    import torch

    from hamers_amd import ConvectiveFluxReconstructor, Hierarchy, Level

    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    n, dx, dt = (48, 40), (1 / 48, 1 / 40), 2e-3
    rec = ConvectiveFluxReconstructor("buf", 2, "SINGLE_SPECIES", "WCNS5_JS_HLLC_HLL", species_gamma=(1.4,))
    boxes = [((0, 0), (24, 40)), ((24, 0), (24, 40))]
    Q = _domain(n, 0, 9)
    out = []
    for used in (False, True):
        C = Level(rec, boxes, ((0, 0), n), (1, 1), dx)
        C.write_global(Q)
        if used:
            F = Level(rec, [((24, 24), (32, 32))], ((0, 0), (96, 80)), (1, 1), tuple(v / 2 for v in dx))
            F.write_patch(0, np.repeat(np.repeat(Q[:, 12:28, 12:28], 2, axis=1), 2, axis=2))
            H = Hierarchy(C, F)
            H.advance(dt, 1)
            C.write_global(Q)
        C.advance(dt, 2, use_graph=True)
        torch.cuda.synchronize()
        out.append(C.read_global(Q.shape))
    assert np.array_equal(out[0], out[1])
