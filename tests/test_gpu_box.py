"""Box elements: operators whose elements are all axis-aligned boxes run kernels on a compact
geometry; any other element keeps the general ones.  The general kernels are reached here with the
last node's MJI one ulp off, which is no box's, so both forms compute on otherwise equal geometry."""
import numpy as np
import pytest

import problems as P
from gpu_cases import _flux, make_state

pytestmark = pytest.mark.gpu


def pair(law, dim, N, Kd, form="weak", sflux="rusanov", bc="copy", periodic=True, directions=None,
         ordering="cartesian", precision="reference", source=None, seed=0, geometry="host", level=False):
    """(box operator, general operator, state); uneven coordinates, so that every box differs."""
    import atum_hip as A
    rng = np.random.default_rng(seed)
    size = 2000.0 if "gravity" in law else 2.0
    coords = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.7, 1.3, k))]) * size / k for k in Kd]
    per = (periodic,) * dim if isinstance(periodic, bool) else periodic
    states = rng.uniform(1, 2, (2 * dim, dim + 2))
    states[:, -1] += 8  # positive pressure
    prob = A.Problem(boundary=bc, source=source, omega=1e-2, bc_states=states if bc == "prescribed" else None)
    u = (1.0, -0.4, 0.7)[:dim]

    def build(off):
        g = A.brickgrid(A.LobattoCell(N, dim), coords, per, ordering)
        if off:
            g.MJI = g.MJI.copy()
            g.MJI[-1] = np.nextafter(g.MJI[-1], np.inf)
        if law == "advection":
            alaw = A.AdvectionLaw(dim, u, problem=prob)
        elif law == "euler":
            alaw = A.EulerLaw(dim, problem=prob)
        elif law == "shallow_water":
            alaw = A.ShallowWaterLaw(dim, grav=9.81, problem=prob)
        else:
            prob.referencestate = lambda x: P.isothermal_reference(x)
            alaw = A.EulerGravityLaw(dim, problem=prob, pde_level_balance=level)
            if law == "linear_euler_gravity":
                alaw = A.LinearEulerGravityLaw(alaw)
        vf = A.WeakForm() if form == "weak" else A.FluxDifferencingForm(_flux(A, form))
        return A.DGSEM(law=alaw, grid=g, volume_form=vf, surface_numericalflux=_flux(A, sflux),
                       directions=directions, precision=precision, geometry="host" if off else geometry)

    box, general = build(False), build(True)
    q = make_state(law, box.grid.points, rng, box.auxstate)
    if "gravity" in law and law != "linear_euler_gravity":
        q = make_state("euler_gravity", box.grid.points, rng, box.auxstate)
    return box, general, q


def device_bytes(dg):
    import atum_hip._lib as L
    return L.lib.atm_dg_device_bytes(dg.h)


def tendencies(box, general, q0):
    out = []
    for dg in (box, general):
        q = dg.fieldarray(q0)
        dq = dg.fieldarray(np.cos(np.arange(q0.size)).reshape(q0.shape))
        dg(dq, q, 0.0, increment=True)
        dg.ctx.sync()
        out.append(dq.numpy())
    return out


WEAK = [("advection", 1, (7,), {}), ("advection", 2, (5, 3), dict(bc="zero_inflow", periodic=(True, False))),
        ("advection", 3, (3, 2, 4), {}), ("euler", 1, (9,), dict(bc="prescribed", periodic=False)),
        ("euler", 2, (4, 5), dict(bc="reflect", periodic=(False, True))), ("euler", 3, (3, 2, 3), {}),
        ("euler_gravity", 2, (3, 4), dict(bc="reflect", periodic=(True, False))),
        ("euler_gravity", 3, (2, 3, 2), dict(bc="reflect", periodic=False, source="coriolis")),
        ("euler_gravity", 3, (2, 2, 3), dict(bc="copy", periodic=(True, True, False), level=True)),
        ("linear_euler_gravity", 2, (3, 4), dict(bc="reflect", periodic=(True, False), directions=(2,),
                                                 ordering="stacked")),
        ("linear_euler_gravity", 3, (2, 3, 4), dict(bc="reflect", periodic=(True, True, False), directions=(3,),
                                                    ordering="stacked")),
        ("shallow_water", 1, (6,), {}), ("shallow_water", 2, (5, 4), {}), ("shallow_water", 2, (1, 1), {}),
        ("shallow_water", 3, (2, 3, 2), {}), ("advection", 2, (3, 4), dict(directions=(2,)))]


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("law,dim,Kd,kw", WEAK, ids=[f"{c[0]}{c[1]}d{i}" for i, c in enumerate(WEAK)])
def test_weak_box_kernels_equal_the_general_ones(law, dim, Kd, kw, N):
    """The same operations in the same order on the same numbers: every value equal (the last node is left
    out: its MJI differs)."""
    box, general, q0 = pair(law, dim, N, Kd, seed=N, **kw)
    assert device_bytes(box) > device_bytes(general)  # the compact geometry was found here, and not there
    a, b = tendencies(box, general, q0)
    np.testing.assert_array_equal(a[:, :-1], b[:, :-1])


@pytest.mark.parametrize("dim,Kd", [(1, (6,)), (2, (4, 3)), (3, (2, 3, 2))])
def test_weak_box_kernels_without_pressure(dim, Kd):
    """A sound speed of zero: the root of the box kernels is that of the general ones there too."""
    box, general, q0 = pair("euler", dim, 3, Kd, seed=5)
    rho = 2.0 ** np.random.default_rng(1).integers(-2, 3, q0[0].shape)
    q0[0], q0[1:-1], q0[-1] = rho, rho, dim * rho / 2  # velocity 1, all energy kinetic
    a, b = tendencies(box, general, q0)
    assert np.isfinite(a).all()
    np.testing.assert_array_equal(a[:, :-1], b[:, :-1])


@pytest.mark.parametrize("dim,Kd", [(1, (5,)), (2, (4, 3)), (3, (3, 2, 2))])
def test_device_built_and_host_built_boxes_agree(dim, Kd):
    import atum_hip as A
    hb, _, q0 = pair("euler", dim, 4, Kd, seed=3)
    db, _, _ = pair("euler", dim, 4, Kd, seed=3, geometry="device")
    outs = []
    for dg in (hb, db):
        q = dg.fieldarray(q0)
        A.LSRK54(dg, q, 1e-3).run(q, 3)
        dg.ctx.sync()
        outs.append(q.numpy())
    np.testing.assert_array_equal(outs[0], outs[1])


FAST = [("euler", 2, (4, 3), dict(bc="prescribed", periodic=False)), ("euler", 2, (3, 5), {}),
        ("euler", 3, (2, 3, 2), dict(bc="reflect", periodic=(False, True, False))),
        ("euler_gravity", 2, (3, 4), dict(bc="reflect", periodic=(True, False), level=True)),
        ("euler_gravity", 3, (2, 2, 3), dict(bc="reflect", periodic=False, source="coriolis")),
        ("euler_gravity", 3, (3, 2, 2), dict(bc="copy", periodic=(True, False, False), ordering="stacked"))]


FD = FAST + [("euler", 1, (7,), dict(bc="prescribed", periodic=False)),
             ("euler_gravity", 1, (5,), dict(bc="reflect", periodic=False))]


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("sflux", ["roe", "rusanov"])
@pytest.mark.parametrize("law,dim,Kd,kw", FD, ids=[f"{c[0]}{c[1]}d{i}" for i, c in enumerate(FD)])
def test_reference_order_box_kernels_against_the_general_ones(law, dim, Kd, kw, sflux, N):
    """The same order of the sums with another form of the logarithmic means: each form is within 1e-12
    of the oracle's tendency (relative max-norm, tests/test_gpu_parity.py)."""
    box, general, q0 = pair(law, dim, N, Kd, form="ec", sflux=sflux, seed=20 + N, **kw)
    assert device_bytes(box) > device_bytes(general)
    a, b = tendencies(box, general, q0)
    assert np.abs(a - b).max() <= 2e-12 * np.abs(b).max()


# 2-D elements of N = 7 and 3-D ones of N = 3 take a workgroup each: 256 of them, and one more; 512, and one more
DEALT = FAST + [("euler", 2, (16, 16), {}), ("euler", 2, (257, 1), {}),
                ("euler_gravity", 3, (8, 8, 4), dict(bc="reflect", periodic=False)),
                ("euler_gravity", 3, (257, 1, 1), dict(bc="reflect", periodic=False)),
                ("euler_gravity", 3, (8, 8, 8), dict(bc="reflect", periodic=False)),
                ("euler_gravity", 3, (513, 1, 1), dict(bc="reflect", periodic=False))]


@pytest.mark.parametrize("N", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("sflux", ["roe", "rusanov"])
@pytest.mark.parametrize("law,dim,Kd,kw", DEALT, ids=[f"{c[0]}{c[1]}d{i}" for i, c in enumerate(DEALT)])
def test_reference_order_pairs_dealt_out_over_threads(law, dim, Kd, kw, sflux, N):
    """A small mesh's kernel, which deals a line's pairs out, in one-, two- and three-element workgroups against
    the batched one, which does not: the same operations in the same order, so the same bits."""
    import atum_hip as A
    box, _, q0 = pair(law, dim, N, Kd, form="ec", sflux=sflux, seed=30 + N, **kw)
    q = box.fieldarray(q0)
    A.LSRKEnsemble([box], [q], [1e-4]).run(2)
    box.ctx.sync()
    want = q.numpy()
    assert np.isfinite(want).all() and np.abs(want - q0).max() > 0
    default = box.epw
    for epw in (default, 1, 2, 3):
        if epw != default and epw not in box.epw_candidates():
            continue
        box.epw = epw
        q = box.fieldarray(q0)
        A.LSRK54(box, q, 1e-4).run(q, 2)
        box.ctx.sync()
        np.testing.assert_array_equal(q.numpy(), want)


# N = 7 in 2-D and N = 3 in 3-D take a wave each: the most workgroups whose work is dealt out by role, and one more
ROLES = FAST + [("euler", 2, (48, 32), {}), ("euler", 2, (1537, 1), {}),
                ("euler_gravity", 3, (8, 8, 8), dict(bc="reflect", periodic=False)),
                ("euler_gravity", 3, (513, 1, 1), dict(bc="reflect", periodic=False))]


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("sflux", ["roe", "rusanov"])
@pytest.mark.parametrize("law,dim,Kd,kw", ROLES, ids=[f"{c[0]}{c[1]}d{i}" for i, c in enumerate(ROLES)])
def test_fast_elements_dealt_out_by_role(law, dim, Kd, kw, sflux, N):
    """A small mesh's kernel, which deals the directions and faces out, in one-, two- and three-element
    workgroups against the batched one, which does not: the same operations in the same order, so the same bits."""
    import atum_hip as A
    box, _, q0 = pair(law, dim, N, Kd, form="ec", sflux=sflux, precision="fast", seed=40 + N, **kw)
    q = box.fieldarray(q0)
    A.LSRKEnsemble([box], [q], [1e-4]).run(2)
    box.ctx.sync()
    want = q.numpy()
    assert np.isfinite(want).all() and np.abs(want - q0).max() > 0
    default = box.epw
    for epw in (default, 1, 2, 3):
        if epw != default and epw not in box.epw_candidates():
            continue
        box.epw = epw
        q = box.fieldarray(q0)
        A.LSRK54(box, q, 1e-4).run(q, 2)
        box.ctx.sync()
        np.testing.assert_array_equal(q.numpy(), want)


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("sflux", ["roe", "rusanov"])
@pytest.mark.parametrize("law,dim,Kd,kw", FAST, ids=[f"{c[0]}{c[1]}d{i}" for i, c in enumerate(FAST)])
def test_fast_box_kernels_against_the_general_ones(law, dim, Kd, kw, sflux, N):
    """Another order of the same sums: each form is within 1e-12 of the oracle's tendency (relative
    max-norm, tests/test_gpu_fast.py), so they are within 2e-12 of each other."""
    box, general, q0 = pair(law, dim, N, Kd, form="ec", sflux=sflux, precision="fast", seed=10 + N, **kw)
    assert device_bytes(box) > device_bytes(general)
    a, b = tendencies(box, general, q0)
    assert np.abs(a - b).max() <= 2e-12 * np.abs(b).max()


@pytest.mark.parametrize("explicit", [True, False])
@pytest.mark.parametrize("split,paper", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("law,dim,N", [("advection", 2, 4), ("euler_gravity", 2, 3), ("euler_gravity", 3, 3)])
def test_ark_step_with_sums_in_the_implicit_kernel(law, dim, N, split, paper, explicit):
    """One ARK23 step whose implicit operator is on box elements (its kernel adds the stages' tendencies up)
    against the general operators (a pass for each sum): the same operations in the same order, so equal in
    the columns that the last node's other MJI cannot reach in three tendencies."""
    import atum_hip as A
    K = (11, 4) if dim == 2 else (11, 2, 4)
    lin_law = law if law == "advection" else "linear_euler_gravity"
    kw = dict(bc="zero_inflow" if law == "advection" else "reflect", periodic=(True,) * (dim - 1) + (False,),
              ordering="stacked", seed=5)
    lb, lg, q0 = pair(lin_law, dim, N, K, directions=(dim,), **kw)
    eb, eg, q0 = pair(law, dim, N, K, **kw)
    out = []
    for lin, ex in ((lb, eb), (lg, eg)):
        q = lin.fieldarray(q0)
        A.ARK23(ex if explicit else None, lin, q, 1e-3, split_rhs=split, paperversion=paper).run(q, 1)
        lin.ctx.sync()
        out.append(q.numpy().reshape(q0.shape[0], lin.grid.K, -1))
    # stacked elements: the first dimension's index of element e is (e // K[-1]) % K[0]
    x = (np.arange(lb.grid.K) // K[-1]) % K[0]
    far = (x >= 3) & (x <= 6)
    assert np.isfinite(out[0]).all()
    # (unsplit without an explicit operator the explicit part is minus the implicit one: nothing moves)
    assert (np.abs(out[0] - q0.reshape(out[0].shape)).max() > 0) == (explicit or split)
    np.testing.assert_array_equal(out[0][:, far], out[1][:, far])


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("precision,dim,sflux", [("fast", 2, "roe"), ("fast", 3, "rusanov"), ("fast", 3, "roe"),
                                                 ("reference", 3, "roe"), ("reference", 3, "rusanov"),
                                                 ("reference", 2, "roe")])
def test_ark_stage_in_one_launch(precision, dim, sflux, N):
    """Both tendencies of a stage in one launch against two launches (an element order set on the explicit
    operator, the mesh's own, takes them apart): the same numbers."""
    import atum_hip as A
    K = (3, 4) if dim == 2 else (3, 2, 4)
    kw = dict(bc="reflect", periodic=(True,) * (dim - 1) + (False,), ordering="stacked", seed=N)
    lin, _, q0 = pair("linear_euler_gravity", dim, N, K, directions=(dim,), **kw)
    ex, _, q0 = pair("euler_gravity", dim, N, K, form="ec", sflux=sflux, precision=precision, **kw)
    out = []
    for order in (None, np.arange(lin.grid.K)):
        ex.set_schedule(order)
        q = lin.fieldarray(q0)
        A.ARK23(ex, lin, q, 1e-3, split_rhs=False).run(q, 2)
        lin.ctx.sync()
        out.append(q.numpy())
    assert np.isfinite(out[0]).all() and np.abs(out[0] - q0).max() > 0
    np.testing.assert_array_equal(out[0], out[1])
