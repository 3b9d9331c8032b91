"""Requests that are on the device together because one of them outlasts the submission of all the others."""
import numpy as np
import pytest

from gpu_cases import relmax
from serve_requests import make_stream, oracle_result

pytestmark = pytest.mark.gpu

STATE_TOL = 1e-10  # states, relative max-norm (tests/test_gpu_parity.py)


def _overlapping(reqs, steps):
    """All arrive at once, behind a small request of `steps` steps: hundreds of ticks, where building and
    submitting a request takes about a millisecond."""
    import dataclasses
    first = next(r for r in reqs if r.kind == "vortex")
    reqs = [dataclasses.replace(r, arrival=0.0) for r in reqs]
    return [dataclasses.replace(first, rid=len(reqs), steps=steps, arrival=-1.0)] + reqs


def test_overlapping_results_equal_alone():
    import atum_hip as A
    reqs = _overlapping(make_stream(duration=0.3, rate=60.0, seed=5, steps=(3, 17), vortex_k=(2, 6), sw_k=(2, 6),
                                    imex_kh=(2, 3), imex_kv=3, nrange=(2, 5)), 4000)
    assert len(reqs) >= 9 and {r.kind for r in reqs} == {"vortex", "sw", "imex"}
    server = A.Server(chunk=4)
    stats = server.run(reqs)
    server.close()
    assert stats.completed == len(reqs) and stats.max_active >= 2
    cache = {}
    for r in reqs:
        assert np.array_equal(r.result, A.run_alone(r, cache)), (r.rid, r.kind)


def test_overlapping_results_against_oracle():
    import atum_hip as A
    reqs = make_stream(duration=0.25, rate=60.0, seed=22, steps=(20, 100), vortex_k=(2, 5), sw_k=(2, 5),
                       imex_kh=(2, 3), imex_kv=3, nrange=(3, 7))
    assert {r.kind for r in reqs} == {"vortex", "sw", "imex"}
    reqs = _overlapping(reqs, 4000)
    server = A.Server(chunk=8)
    stats = server.run(reqs)
    server.close()
    assert stats.completed == len(reqs) and stats.max_active >= 2
    for r in reqs[1:]:  # the first one's many steps are the other test's
        assert relmax(r.result, oracle_result(r)) <= STATE_TOL, (r.rid, r.kind, r.key)
