"""Operators on geometry arrays that are not a brick's, against the oracle on the same arrays.

Tolerance as in the parity tests: tendency relative max-norm <= 1e-12 (FAST mode on these generic states too)."""
import numpy as np
import pytest

from gpu_cases import Case, relmax

pytestmark = pytest.mark.gpu

TENDENCY_TOL = 1e-12


def _tendency_error(case, precision):
    """The product's tendency on case.grid's arrays against the oracle's on the same ones."""
    import atum_hip as A
    d, g, o = case.dg, case.grid, case.ogrid
    dg = A.DGSEM(law=d.law, grid=g, volume_form=d.volume_form, surface_numericalflux=d.surface_numericalflux,
                 directions=d.directions, auxstate=case.aux, precision=precision)
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
