"""Operators on geometry arrays that are not a brick's, against the oracle on the same arrays.

Tolerance as in the parity tests: tendency relative max-norm <= 1e-12 (FAST mode on these generic states too)."""
import numpy as np
import pytest

from gpu_cases import Case, relmax

pytestmark = pytest.mark.gpu

TENDENCY_TOL = 1e-12


def _tendency_error(case, precision, box=None):
    """The product's tendency on case.grid's arrays against the oracle's on the same ones."""
    import atum_hip as A
    import atum_hip._lib as L
    d, g, o = case.dg, case.grid, case.ogrid
    dg = A.DGSEM(law=d.law, grid=g, volume_form=d.volume_form, surface_numericalflux=d.surface_numericalflux,
                 directions=d.directions, auxstate=case.aux, precision=precision)
    assert box is None or L.lib.atm_dg_box_elements(dg.h) == box
    for name in ("g", "MJ", "MJI", "faceMJ", "normal"):
        getattr(o, name)[...] = getattr(g, name)  # in place: the oracle's operator points there
    qf, dqf = dg.fieldarray(case.q), dg.fieldarray()
    dg(dqf, qf, 0.0, increment=False)
    dg.ctx.sync()
    return relmax(dqf.numpy(), case.odg.tendency(case.q))


@pytest.mark.parametrize("precision", ["reference", "fast"])
@pytest.mark.parametrize("dim,form,sflux", [(2, "ec", "roe"), (3, "ec", "rusanov"), (2, "weak", "rusanov")])
@pytest.mark.parametrize("scaled", ["MJ", "g", "faceMJ"])
def test_face_jacobians_of_their_own(scaled, dim, form, sflux, precision):
    """Rectangular elements whose face Jacobians are not their Jacobians times the metric: what a face adds is
    scaled by faceMJ MJI, whatever the metric."""
    c = Case("euler", dim, 3, 3, form=form, sflux=sflux, seed=60 + dim)
    g = c.grid
    for name, f in {"MJ": (("MJ", 2.0), ("MJI", 0.5)), "g": (("g", 2.0),), "faceMJ": (("faceMJ", 0.5),)}[scaled]:
        setattr(g, name, getattr(g, name) * f)
    assert _tendency_error(c, precision) <= TENDENCY_TOL


def _shear(grid):
    """The brick's elements turned and sheared, their Jacobians varying within each: contravariant metric, Jacobians
    and normals as such elements have them."""
    dim = grid.dim
    S = np.eye(dim)
    if dim > 1:
        c, s = np.cos(0.3), np.sin(0.3)
        S[:2, :2] = [[c, -s], [s, c]]
        S[-1, 0] += 0.4
    inv, det = np.linalg.inv(S), np.linalg.det(S)
    x = grid.points
    vary = 1 + 0.1 * np.sin(x.sum(axis=0) / np.ptp(x) + np.arange(grid.Ntot) % grid.Np)
    g = grid.g.reshape(dim, dim, -1)  # [c, a]: plane a + dim c
    grid.g = np.einsum("bax,bc->cax", g, inv).reshape(dim * dim, -1) / vary
    grid.MJ = grid.MJ * det * vary
    grid.MJI = 1 / grid.MJ
    n = inv.T @ grid.normal
    size = np.sqrt((n * n).sum(axis=0))
    grid.normal = n / size
    grid.faceMJ = grid.faceMJ * det * size


GRAVITY = dict(gravity_domain=True, bc="reflect")
GENERAL = [("advection", 1, "weak", "rusanov", {}), ("advection", 2, "weak", "rusanov", {}),
           ("euler", 1, "weak", "rusanov", {}), ("euler", 3, "weak", "rusanov", {}),
           ("shallow_water", 2, "weak", "rusanov", {}),
           ("euler_gravity", 3, "weak", "rusanov", dict(GRAVITY, periodic=(False,) * 3, source="coriolis", omega=1e-2)),
           ("linear_euler_gravity", 3, "weak", "rusanov",
            dict(GRAVITY, periodic=(True, True, False), directions=(3,), ordering="stacked")),
           ("euler", 1, "ec", "roe", {}), ("euler", 2, "ec", "rusanov", {}), ("euler", 3, "ec", "roe", {}),
           ("euler_gravity", 2, "ec", "roe", dict(GRAVITY, periodic=(True, False))),
           ("euler_gravity", 3, "ec", "rusanov", dict(GRAVITY, periodic=(False,) * 3)),
           ("euler_gravity", 3, "ec", "roe", dict(GRAVITY, periodic=(True, False, False)))]


@pytest.mark.parametrize("N", [1, 2, 4, 7])
@pytest.mark.parametrize("law,dim,form,sflux,kw", GENERAL, ids=[f"{c[0]}{c[1]}d-{c[2]}-{c[3]}" for c in GENERAL])
def test_turned_and_sheared_elements(law, dim, form, sflux, kw, N):
    """The kernels of elements that are no boxes, against the oracle."""
    c = Case(law, dim, N, [3, 2, 2][:dim], form=form, sflux=sflux, seed=70 + N, **kw)
    _shear(c.grid)
    for precision in ("reference",) if form == "weak" else ("reference", "fast"):
        assert _tendency_error(c, precision, box=0) <= TENDENCY_TOL, precision


@pytest.mark.parametrize("law,dim,form,sflux,precision", [("shallow_water", 2, "weak", "rusanov", "reference"),
                                                          ("euler", 2, "ec", "rusanov", "fast"),
                                                          ("euler", 3, "ec", "roe", "fast"),
                                                          ("euler", 2, "ec", "roe", "reference")])
def test_turned_and_sheared_elements_in_a_batch(law, dim, form, sflux, precision):
    """Members of several degrees whose elements are no boxes beside one whose are, batched: the bits of each alone."""
    import atum_hip as A
    import atum_hip._lib as L
    dgs, q0 = [], []
    for N, boxes in ((3, False), (5, False), (1, False), (7, False), (3, True)):
        c = Case(law, dim, N, 2, form=form, sflux=sflux, seed=80 + N)
        if not boxes:
            _shear(c.grid)
        dgs.append(A.DGSEM(law=c.dg.law, grid=c.grid, volume_form=c.dg.volume_form,
                           surface_numericalflux=c.dg.surface_numericalflux, precision=precision))
        assert L.lib.atm_dg_box_elements(dgs[-1].h) == boxes
        q0.append(c.q)
    dts = [1e-4 * (i + 1) for i in range(len(dgs))]
    qs = [dg.fieldarray(q) for dg, q in zip(dgs, q0)]
    A.LSRKEnsemble(dgs, qs, dts).run(3)
    for dg, q, start, dt in zip(dgs, qs, q0, dts):
        alone = dg.fieldarray(start)
        A.LSRK54(dg, alone, dt).run(alone, 3)
        dg.ctx.sync()
        assert np.isfinite(alone.numpy()).all() and np.abs(alone.numpy() - start).max() > 0
        np.testing.assert_array_equal(q.numpy(), alone.numpy())
