"""Box and general operators of one configuration are tuned apart: their kernels differ."""
import pytest

from test_gpu_box import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,sflux,precision", [("weak", "rusanov", "reference"), ("ec", "roe", "fast")])
def test_a_cached_shape_is_of_the_same_kernels(form, sflux, precision):
    import atum_hip._lib as L
    from atum_hip.tuning import TuneCache, autotune, autotune_batch
    box, general, q0 = pair("euler", 2, 3, (4, 4), form=form, sflux=sflux, precision=precision)
    assert (L.lib.atm_dg_box_elements(box.h), L.lib.atm_dg_box_elements(general.h)) == (1, 0)
    cache = TuneCache()
    shape = next(e for e in general.epw_candidates() if e in box.epw_candidates())
    cache.put(general, shape)
    assert autotune(general, q0, reps=2, cache=cache) == (shape, {})
    best, times = autotune(box, q0, reps=2, cache=cache)
    assert times and cache.get(box) == best and cache.get(general) == shape
    # a batch's launch groups are those of the tuning
    assert len(autotune_batch([box, general], [q0, q0], [1e-6, 1e-6])) == 2
