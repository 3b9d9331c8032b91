"""Creating an operator beside work that is queued on the device."""
import time

import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["box", "last element not a box"])
def test_creation_does_not_wait_for_queued_work(kind):
    """An operator made from geometry arrays does not wait for what its context's stream still has to do."""
    import atum_hip as A

    def bubble(K):
        v = P.julia_range(0.0, 2000.0, K + 1)
        grid = A.brickgrid(A.LobattoCell(4, 3), (v, v, v), (False,) * 3)
        law = A.EulerGravityLaw(3, grav=9.81, problem=A.Problem(boundary="reflect"))
        if kind != "box":
            grid.MJI = grid.MJI.copy()
            grid.MJI[-1] = np.nextafter(grid.MJI[-1], np.inf)
        aux = law.auxiliary(grid.points)
        return lambda: A.DGSEM(law=law, grid=grid, volume_form=A.FluxDifferencingForm(A.EntropyConservativeFlux()),
                               surface_numericalflux=A.RoeFlux(), auxstate=aux), grid
    make, grid = bubble(12)
    small, _ = bubble(3)
    small()
    dg = make()
    q = dg.fieldarray(P.rising_bubble(grid.points))
    run = A.LSRK54(dg, q, 1e-9)
    run.run(q, 2)
    dg.ctx.sync()
    run.run(q, 1000)  # some tenths of a second on the device
    t0 = time.perf_counter()
    beside = small()  # (kept: giving it back waits)
    t1 = time.perf_counter()
    dg.ctx.sync()
    t2 = time.perf_counter()
    del beside
    assert t2 - t0 > 0.1
    assert t1 - t0 < 0.5 * (t2 - t0)
