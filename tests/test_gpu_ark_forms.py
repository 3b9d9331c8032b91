"""Which form a stage of ARK23 takes: the form of one launch stores no explicit tendency (the start of the workspace)."""
import numpy as np
import pytest

from test_gpu_box import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,dim,one", [("fast", 2, True), ("fast", 3, True), ("reference", 3, True),
                                               ("reference", 2, False)])
def test_stage_form(precision, dim, one):
    import atum_hip as A
    K = (3, 4) if dim == 2 else (3, 2, 4)
    kw = dict(bc="reflect", periodic=(True,) * (dim - 1) + (False,), ordering="stacked", seed=3)
    lin, _, q0 = pair("linear_euler_gravity", dim, 3, K, directions=(dim,), **kw)
    ex, general, q0 = pair("euler_gravity", dim, 3, K, form="ec", sflux="roe", precision=precision, **kw)
    for op, order, want in ((ex, None, one), (ex, np.arange(lin.grid.K), False), (general, None, False)):
        op.set_schedule(order)
        q = lin.fieldarray(q0)
        ark = A.ARK23(op, lin, q, 1e-3, split_rhs=False)
        ark.work.fill_(-7.0)
        ark.run(q, 1)
        lin.ctx.sync()
        explicit = ark.work.numpy().ravel()[:q0.size]
        assert np.all(explicit == -7.0) == want
        assert np.isfinite(q.numpy()).all()
