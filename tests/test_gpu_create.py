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
    run.run(q, 3000)  # half a second on the device
    t0 = time.perf_counter()
    beside = small()  # (kept: giving it back waits)
    t1 = time.perf_counter()
    dg.ctx.sync()
    t2 = time.perf_counter()
    del beside
    assert t2 - t0 > 0.1
    assert t1 - t0 < 0.5 * (t2 - t0)


def test_boxes_are_found_in_meshes_of_more_elements_than_workgroups():
    """The look-over's workgroups take several elements each past 65536: the records of all are right, and an
    element late in the mesh that is no box is seen."""
    import atum_hip as A
    import atum_hip._lib as L
    rng = np.random.default_rng(3)
    coords = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.7, 1.3, k))]) for k in (263, 251)]
    grid = A.brickgrid(A.LobattoCell(1, 2), coords, (True, False))
    assert grid.K > 65536
    q0 = rng.uniform(1, 2, (1, grid.Ntot))

    def make(geometry="host"):
        return A.DGSEM(law=A.AdvectionLaw(2, (1.0, -0.4), problem=A.Problem(boundary="zero_inflow")), grid=grid,
                       surface_numericalflux=A.RusanovFlux(), geometry=geometry)
    out = []
    for dg in (make(), make("device")):
        assert L.lib.atm_dg_box_elements(dg.h) == 1
        q, dq = dg.fieldarray(q0), dg.fieldarray()
        dg(dq, q, 0.0, increment=False)
        dg.ctx.sync()
        out.append(dq.numpy())
    np.testing.assert_array_equal(out[0], out[1])
    for name, at in (("MJ", -3), ("faceMJ", -5)):
        kept = getattr(grid, name)
        setattr(grid, name, kept.copy())
        getattr(grid, name)[at] = np.nextafter(kept[at], np.inf)
        assert L.lib.atm_dg_box_elements(make().h) == 0, name
        setattr(grid, name, kept)
